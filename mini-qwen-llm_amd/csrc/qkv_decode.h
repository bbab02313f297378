// Device code of the split-K decode kernels (see qkv_decode.hip for the design).
#pragma once

#include <type_traits>
#include <utility>

#include "mqk_device.h"
#include "mqk_kernels.h"

namespace mqk {

using DecKernel = void (*)(ProblemArgs, WeightArgs, EpilogueArgs, int, float*, uint32_t*, int);
// Kernels of one block of up to 16 * mb rows (mb 1, 2, 4; the split's k range at most 16
// tiles for int4 and for mb 4, 32 otherwise), of one block with longer splits (up to 32
// tiles; mb 4 only for 16-bit weights), and of several 64-row blocks whose longest split has nk tiles (1 .. 13).
DecKernel decode_kernel_bf16(int mb);
DecKernel decode_kernel_w4(int mb);
DecKernel decode_kernel_f16(int mb);
DecKernel decode_long_kernel_bf16();
DecKernel decode_long_kernel_w4(int mb);
DecKernel decode_long_kernel_f16();
DecKernel decode_multi_kernel_bf16(int nk);
DecKernel decode_multi_kernel_w4(int nk);

namespace {

constexpr int kDecRows = 64;            // token rows per block (one block per call when T <= 64)
constexpr int kDecMaxBlocks = 16;       // most 64-row blocks one launch streams the weights for
constexpr int kDecThreads = 512;        // 8 waves; wave w owns columns [16w, 16w+16) of the head
constexpr int kDecWaves = kDecThreads / 64;
constexpr int kDecMaxNK = 16;           // k tiles of one x slice in LDS (64-wide tiles)
// Longest k range of a split in a launch of one block: two x slices, staged
// one after the other (wider models, e.g. hidden 5120 with 56 heads, then keep
// one workgroup per CU with 4 splits of 20 tiles instead of 5 splits over two
// rounds).
constexpr int kDecLongMaxNK = 2 * kDecMaxNK;
constexpr int kDecLookahead = 6;        // weight tiles in flight per wave (64-row blocks)
constexpr int kDecLookaheadSmall = 16;  // ... 16- and 32-row blocks, which leave the registers for it
// Longest k range (in 64-wide tiles) of a split in a launch of several blocks:
// beyond it the held weights and the finisher no longer fit the 256 VGPRs of a
// wave without spilling, and such launches run one block each.
constexpr int kDecMultiMaxNK = 13;
constexpr int kDecKc = kDecMaxNK * kBK;     // LDS row length of the x slice (bf16), 2 KB
constexpr int kMaxHeads = kDecodeMaxHeads;
constexpr int kCounterBytes = int(kDecodeCounterBytes);
constexpr int kTileFloats = kDecRows * kHeadDim;
constexpr int kPitch = kHeadDim + 4;    // fp32 pitch of the finisher's LDS head tile
constexpr int kDecMaxSpins = 1 << 14;   // default polls (s_sleep 2 apart, ~1 ms) before a wait is handed off

static_assert(kDecRows * kDecKc * 2 > 160 * 1024 / 2, "x slice must keep one workgroup per CU");
static_assert(kDecRows * 8 == kDecThreads, "one 16-byte x chunk per thread per k tile");
static_assert(kDecRows * kPitch * 4 <= kDecRows * kDecKc * 2, "the head tile aliases the x slice");
static_assert(kDecWaves * 16 == kHeadDim, "one 16-column group per wave");

// x slice layout in LDS: tile-major, [k tile t][row 0..63][8 chunks of 16 B]
// (8 KB per 64-wide k tile); chunk c of row r is stored in slot c ^ ((r >> 1) & 7),
// so the 16 rows one quarter-wave reads (8 even rows in one half of the banks, 8
// odd rows in the other) hit 16 different bank groups.  (Blocks of 16 * MB rows: MB
// quarters of that per tile.)
template <int MB>
__device__ __forceinline__ int dec_lds_off(int t, int row, int chunk) {
  return t * (16 * MB * 64) + row * 64 + ((chunk ^ ((row >> 1) & 7)) << 3);  // in 16-bit elements
}

__device__ __forceinline__ int xcc_id() {
  return __builtin_amdgcn_s_getreg((20) | (0 << 6) | ((4 - 1) << 11));  // hwreg(HW_REG_XCC_ID, 0, 4)
}

// k-tile range [kt0, kt0 + nk) of split s of S over nkt tiles (balanced).
__device__ __forceinline__ void split_range(int s, int S, int nkt, int& kt0, int& nk) {
  kt0 = int((int64_t(s) * nkt) / S);
  nk = int((int64_t(s + 1) * nkt) / S) - kt0;
}

// A block has MB (1, 2 or 4) row blocks of 16 token rows.  k tile t of its x slice is
// staged by 2 * MB direct L2 -> LDS loads of 8 rows each (1 KB, contiguous in LDS):
// wave w loads rows [8 (w % (2 MB)), +8) of every tile t with t % (4 / MB) ==
// w / (2 MB); lane L takes row + L/8 and LDS slot L % 8, i.e. global chunk
// (L % 8) ^ ((row >> 1) & 7).  Rows >= M re-read row M-1; those LDS rows only feed
// output rows that are never stored.
template <int MB>
struct XStage {
  static constexpr int kRows = 16 * MB;
  static constexpr int kTileBytes = kRows * 128;
  static constexpr int kStep = 4 / MB;  // tiles between the ones a wave loads
  const uint16_t* src;                  // this lane's chunk of the wave's first tile
  uint32_t dst;                         // LDS byte address of the wave's first 1 KB
  int first;                            // the wave's first tile

  __device__ __forceinline__ XStage(const ProblemArgs& p, int64_t kbeg, uint32_t xs_lds, int r0) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int part = MB == 4 ? wave : wave % (2 * MB);  // (8 waves)
    first = MB == 4 ? 0 : wave / (2 * MB);
    const int row = part * 8 + (lane >> 3);
    const int gq = (lane & 7) ^ ((row >> 1) & 7);
    const int grow = r0 + row < int(p.M) ? r0 + row : int(p.M) - 1;
    src = p.x + int64_t(grow) * p.K + kbeg + first * kBK + gq * 8;
    dst = xs_lds + uint32_t(first * kTileBytes + part * 1024);
  }
  // the wave's i-th tile, first + kStep * i, if it is below nk
  template <int I>
  __device__ __forceinline__ void one(int nk) const {
    if (MB == 4 || first + kStep * I < nk) dma16_at<I * kStep * kBK * 2>(src, dst + uint32_t(I * kStep * kTileBytes));
  }
  template <int... I>
  __device__ __forceinline__ void some(int nk, std::integer_sequence<int, I...>) const {
    (one<I>(nk), ...);
  }
  // tiles 0 .. NK-1: one address per lane, the tiles' steps as instruction offsets
  template <int NK>
  __device__ __forceinline__ void all() const {
    some(NK, std::make_integer_sequence<int, (NK + kStep - 1) / kStep>{});
  }
  // tiles 0 .. nk-1 (nk at run time)
  __device__ __forceinline__ void range(int nk) const {
    for (int t = first; t < nk; t += kStep)
      dma16(src + (t - first) * kBK, dst + uint32_t((t - first) * kTileBytes));
  }
};

// 16x16x32 operand layout: lane (c, g) = (lane & 15, lane >> 4) holds column c
// of the wave's 16 (B) / row c of a 16-row block (A) and 8 k values; inside a
// 64-wide k tile, block kk (0, 1) of 32 and lane group g give k = kk*32 + g*8.
// acc[mb][j] = C[mb*16 + 4g + j][16*wave + c].
template <class E, int MB>
__device__ __forceinline__ void mma_tile(const uint16_t* xs, int t, const u32x4_t (&b)[2], f32x4_t (&acc)[MB]) {
  const int lane = threadIdx.x & 63;
  const int c16 = lane & 15, g4 = lane >> 4;
  u32x4_t a[2][MB];  // all activation fragments of the tile in flight before the first MFMA
#pragma unroll
  for (int kk = 0; kk < 2; ++kk)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
      a[kk][mb] = *reinterpret_cast<const u32x4_t*>(xs + dec_lds_off<MB>(t, mb * 16 + c16, kk * 4 + g4));
#pragma unroll
  for (int kk = 0; kk < 2; ++kk)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[mb] = E::mfma(a[kk][mb], b[kk], acc[mb]);
}

template <int MB>
__device__ __forceinline__ void zero_acc(f32x4_t (&acc)[MB]) {
#pragma unroll
  for (int i = 0; i < MB; ++i) acc[i] = f32x4_t{};
}

// 8 consecutive bf16 (16 bytes, 16-byte aligned: the launcher checks gamma / cos / sin).
__device__ __forceinline__ u32x4_t load8_bf16(const uint16_t* ptr) { return *reinterpret_cast<const u32x4_t*>(ptr); }

// Element i (0..7) of 8 packed 16-bit elements, as float.
template <class E>
__device__ __forceinline__ float elem_lane(const u32x4_t& v, int i) {
  const uint32_t wd = i < 2 ? v.x : (i < 4 ? v.y : (i < 6 ? v.z : v.w));
  return E::to_f32((i & 1) ? wd >> 16 : wd & 0xFFFFu);
}

// Weight fragment load: non-temporal, so the weight stream does not evict the
// split partials and the x slice from the L2.
__device__ __forceinline__ u32x4_t wload(const uint16_t* ptr) {
  return load_global_nt(reinterpret_cast<const u32x4_t*>(ptr));
}

struct Int4Col {  // this lane's column of an int4 projection
  const int32_t* qw;
  const uint16_t* sc;
  const int32_t* qz;
  int64_t n;      // columns of the projection
  int64_t col;
  int group;
  bool fp16;
};

__device__ __forceinline__ Int4Col int4_col(const WeightArgs& w, int proj, int64_t col) {
  const int64_t n = proj == 0 ? w.n_cols[0] : (proj == 1 ? w.n_cols[1] : w.n_cols[2]);
  return Int4Col{pick3_uniform(proj, w.qw[0], w.qw[1], w.qw[2]),
                 static_cast<const uint16_t*>(pick3_uniform(proj, w.sc[0], w.sc[1], w.sc[2])),
                 pick3_uniform(proj, w.qz[0], w.qz[1], w.qz[2]), n, col,
                 w.group, w.scale_fp16 != 0};
}

__device__ __forceinline__ void dequant_tile(const Int4Col& ic, const uint32_t (&q)[2], uint32_t sraw, uint32_t zw,
                                             u32x4_t (&b)[2]) {
  const float scale = ic.fp16 ? f16_to_f32(sraw) : bf16_to_f32(sraw);
  const float zero = float((zw >> ((ic.col % 8) * 4)) & 0xFu);
  b[0] = dequant_int4x8(q[0], zero, scale);
  b[1] = dequant_int4x8(q[1], zero, scale);
}

// The same partial with a run-time k-range and one tile's loads at a time: the
// arithmetic (per-tile dequant, MFMA order) is identical to run_split, so
// its result is bit-identical.  Used by the recompute path only.
template <class E, bool INT4, int MB>
__device__ void partial_any(const ProblemArgs& p, const WeightArgs& w, int proj, int hh, int kt0, int nk,
                            const uint16_t* xs, uint32_t xs_lds, f32x4_t (&acc)[MB], int r0) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int c16 = lane & 15, g4 = lane >> 4;
  const int64_t kbeg = int64_t(kt0) * kBK;
  const int64_t col = int64_t(hh) * kHeadDim + wave * 16 + c16;
  zero_acc(acc);
  XStage<MB>(p, kbeg, xs_lds, r0).range(nk);
  wait_vm<0>();
  barrier();
  for (int t = 0; t < nk; ++t) {
    const int64_t k0 = kbeg + int64_t(t) * kBK;
    u32x4_t b[2];
    if constexpr (!INT4) {
      const uint16_t* wp = pick3_uniform(proj, w.w[0], w.w[1], w.w[2]) + col * p.K + k0 + g4 * 8;
      b[0] = load_global(reinterpret_cast<const u32x4_t*>(wp));
      b[1] = load_global(reinterpret_cast<const u32x4_t*>(wp + 32));
    } else {
      const Int4Col ic = int4_col(w, proj, col);
      const int64_t grp = k0 / ic.group;
      const uint32_t q[2] = {uint32_t(load_global(ic.qw + (k0 / 8 + g4) * ic.n + col)),
                             uint32_t(load_global(ic.qw + (k0 / 8 + 4 + g4) * ic.n + col))};
      dequant_tile(ic, q, load_global(ic.sc + grp * ic.n + col),
                   uint32_t(load_global(ic.qz + grp * (ic.n / 8) + col / 8)), b);
    }
    mma_tile<E, MB>(xs, t, b, acc);
  }
}

// partial_any over a range longer than one x slice: slices of kDecMaxNK tiles,
// each staged once every wave is done with the previous one, the tiles
// accumulated in order into one sum (the arithmetic of the two-slice split).
// (A function of its own rather than a loop in partial_any: that keeps the code
// of the one-slice kernels, C3's among them, exactly as it was.)
template <class E, bool INT4, int MB>
__device__ void partial_any_long(const ProblemArgs& p, const WeightArgs& w, int proj, int hh, int kt0, int nk,
                                 const uint16_t* xs, uint32_t xs_lds, f32x4_t (&acc)[MB], int r0) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int c16 = lane & 15, g4 = lane >> 4;
  const int64_t col = int64_t(hh) * kHeadDim + wave * 16 + c16;
  zero_acc(acc);
  for (int c0 = 0; c0 < nk; c0 += kDecMaxNK) {
    const int cn = nk - c0 < kDecMaxNK ? nk - c0 : kDecMaxNK;
    const int64_t kbeg = int64_t(kt0 + c0) * kBK;
    if (c0 > 0) barrier();  // every wave is done with the previous slice
    XStage<MB>(p, kbeg, xs_lds, r0).range(cn);
    wait_vm<0>();
    barrier();
    for (int t = 0; t < cn; ++t) {
      const int64_t k0 = kbeg + int64_t(t) * kBK;
      u32x4_t b[2];
      if constexpr (!INT4) {
        const uint16_t* wp = pick3_uniform(proj, w.w[0], w.w[1], w.w[2]) + col * p.K + k0 + g4 * 8;
        b[0] = load_global(reinterpret_cast<const u32x4_t*>(wp));
        b[1] = load_global(reinterpret_cast<const u32x4_t*>(wp + 32));
      } else {
        const Int4Col ic = int4_col(w, proj, col);
        const int64_t grp = k0 / ic.group;
        const uint32_t q[2] = {uint32_t(load_global(ic.qw + (k0 / 8 + g4) * ic.n + col)),
                               uint32_t(load_global(ic.qw + (k0 / 8 + 4 + g4) * ic.n + col))};
        dequant_tile(ic, q, load_global(ic.sc + grp * ic.n + col),
                   uint32_t(load_global(ic.qz + grp * (ic.n / 8) + col / 8)), b);
      }
      mma_tile<E, MB>(xs, t, b, acc);
    }
  }
}

// What a workgroup works on: split `split` of head (128-column tile) `head`,
// projection `proj` / head `hh` inside it, for the launch's `nblk` 64-row blocks.
struct DecWork {
  int head, split, splits, proj, hh, nblk;
  uint32_t inc;  // this split's arrival increment (its XCD, and the forced flag for tests)
  int max_spins;  // polls of a designated finisher's final wait before it hands the block off
  int H;                  // heads of the projection (row stride of its output, in heads)
  const uint16_t* gamma;  // QK-Norm weights of the projection (Q or K)
  uint16_t* out;          // q / k / v (may be null: cache only)
};

// Arrival counter of a (head, block), one atomic add per split: bits 0-4 count
// the splits that have published (at most 16), bits 5-12 sum their XCDs x and
// bits 13-22 sum x * x, bits 23-27 count splits forced onto the recompute path
// (tests), and bit 30 marks a block whose designated finisher gave up waiting
// for the others (see run_split).  The splits of a head are dispatched to one
// XCD (workgroups go round-robin over the XCDs, from a starting XCD that
// depends on the hardware queue), so their partials meet in one L2; the last
// arrival checks that they did: n * sum(x^2) == sum(x)^2 exactly when all n
// values of x are equal.
constexpr uint32_t kAbandoned = 1u << 30;
constexpr uint32_t kForcedUnit = 1u << 23;
__device__ __forceinline__ uint32_t arrival_inc(int x, bool forced) {
  return 1u + (uint32_t(x) << 5) + (uint32_t(x * x) << 13) + (forced ? kForcedUnit : 0u);
}
__device__ __forceinline__ bool all_arrived(uint32_t v, int splits) { return (v & 0x1Fu) == uint32_t(splits); }
// some split ran on another XCD than the others (or was forced to recompute)
__device__ __forceinline__ bool any_foreign(uint32_t v, int splits) {
  v = __builtin_amdgcn_readfirstlane(v);  // (the same in every lane: scalar arithmetic)
  const uint32_t sx = (v >> 5) & 0xFFu, sxx = (v >> 13) & 0x3FFu;
  return ((v >> 23) & 0x1Fu) != 0 || uint32_t(splits) * sxx != sx * sx;
}

// Finishes 64-row block `blk` of the workgroup's head: sums every split's partial
// in split order (RECOMPUTE: recomputes them all), applies RMSNorm + RoPE (Q/K),
// stores the bf16 rows and resets the block's arrival counter.  prow / cslot:
// RoPE-table offset and paged-cache slot of this thread's row of the block.
template <class E, bool INT4, int MB, bool MULTI, bool RECOMPUTE, bool LONG = false>
__device__ __forceinline__ void finish_block(const ProblemArgs& p, const WeightArgs& w, const EpilogueArgs& e,
                                             const DecWork& d, int blk, const f32x4_t (&acc)[MB], int64_t prow,
                                             int64_t cslot, uint16_t* xs, float* __restrict__ part,
                                             uint32_t* __restrict__ counters) {
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int n_tiles = p.n_tiles;
  const int M = int(p.M);
  const uint32_t xs_lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(xs));
  float* tile = reinterpret_cast<float*>(xs);  // the finisher's head tile aliases the x slice
  uint32_t* counter = counters + blk * n_tiles + d.head;
  if (RECOMPUTE && tid == 0)  // statistics: heads finished on the recompute path
    __hip_atomic_fetch_add(counters + kDecodeRecomputeWord, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

  // thread -> row r = tid / 8, c = tid % 8 of the head tile: columns [8c, 8c+8)
  // and [64+8c, 64+8c+8), so every RoPE pair (d, d+64) is thread-local.  Its
  // gamma / cos / sin operands are loaded under the partial reads; its RoPE row
  // was read when the block started, so no dependent load stalls the finisher.
  const int r = tid >> 3;
  const int c = tid & 7;
  const int hd = e.head_dim;
  const PairRuns pr = pair_runs(c, hd);  // (head_dim 64: two heads per block, see pair_runs)
  constexpr int kRows = 16 * MB;
  const int rr = blk * kRows + r;  // this thread's row of the launch
  const bool row_in = (MB == 4 || r < kRows) && rr < M;
  const bool qk = e.qkv == 1 && d.proj != 2;  // (qkv 2: q and k stored as projected)
  f32x4_t sum[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) sum[mb] = f32x4_t{};
  if constexpr (!RECOMPUTE) {
    // The other splits' fragments of this wave are pulled into LDS with direct
    // L2 -> LDS loads (a CU fetches faster that way than into VGPRs), up to 16 / MB
    // splits per batch in the x slice's space, which no wave reads any more; each
    // wave reads back only the 4 KB regions it loaded itself, so its own vmcnt
    // wait is the only synchronisation.  Summation is in split order.  In a
    // launch of several blocks the finisher reads its own partial back as well:
    // its registers then hold the weights of the later blocks instead.
    const char* frag = reinterpret_cast<const char*>(part) +
                       (((int64_t(blk) * n_tiles + d.head) * kDecWaves + wave) * MB * 64) * sizeof(f32x4_t);
    const int64_t split_stride = int64_t(d.nblk) * n_tiles * (kRows * kHeadDim) * sizeof(float);
    constexpr int kSlots = 16 / MB;         // splits per batch
    constexpr int kSlotBytes = MB * 1024;   // one wave's fragments of a split
    const uint32_t slot0 = xs_lds + uint32_t(wave * kSlotBytes);
    const char* slot0_ptr = reinterpret_cast<const char*>(xs) + wave * kSlotBytes;
    int slot = 0, first = 0;
#pragma unroll 1
    for (int q = 0; q < d.splits; ++q) {
      if (MULTI || q != d.split) {  // (MULTI: this split's partial too, see below)
        const char* src = frag + q * split_stride + lane * 16;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          dma16(src + mb * 1024, slot0 + uint32_t(slot * kDecWaves * kSlotBytes + mb * 1024));
        ++slot;
      }
      if (slot == kSlots || q == d.splits - 1) {  // the slots filled, or the last split: add in split order
        wait_vm<0>();
        int u_slot = 0;
#pragma unroll 1
        for (int u = first; u <= q; ++u) {
          if (!MULTI && u == d.split) {
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) sum[mb] += acc[mb];
          } else {
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
              sum[mb] += *reinterpret_cast<const f32x4_t*>(slot0_ptr + u_slot * kDecWaves * kSlotBytes + mb * 1024 +
                                                           lane * 16);
            ++u_slot;
          }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // reads done before the next batch overwrites
        slot = 0;
        first = q + 1;
      }
    }
  } else {
    // Some split ran on another XCD: its partial may not be visible through this
    // L2.  Recompute every split here (same arithmetic, same order).
    const int nkt = int(p.K / kBK);
    for (int s = 0; s < d.splits; ++s) {
      int s_kt0, s_nk;
      split_range(s, d.splits, nkt, s_kt0, s_nk);
      __syncthreads();  // every wave is done with the x slice of the previous split
      f32x4_t part_s[MB];
      if constexpr (LONG) partial_any_long<E, INT4, MB>(p, w, d.proj, d.hh, s_kt0, s_nk, xs, xs_lds, part_s, blk * kRows);
      else partial_any<E, INT4, MB>(p, w, d.proj, d.hh, s_kt0, s_nk, xs, xs_lds, part_s, blk * kRows);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) sum[mb] += part_s[mb];
    }
  }

  // (loaded only now: during the partial sums the registers hold the weights of later blocks)
  u32x4_t g_lo{}, g_hi{}, c_lo{}, c_hi{}, s_lo{}, s_hi{};
  if (qk && row_in) {
    const uint16_t* gamma = d.gamma;
    g_lo = load8_bf16(gamma + pr.dim_lo);
    g_hi = load8_bf16(gamma + pr.dim_hi);
    c_lo = load8_bf16(e.cos + prow + pr.dim_lo);
    c_hi = load8_bf16(e.cos + prow + pr.dim_hi);
    s_lo = load8_bf16(e.sin + prow + pr.dim_lo);
    s_hi = load8_bf16(e.sin + prow + pr.dim_hi);
  }

  // ---- head tile to LDS (fp32 [16 MB][kPitch]); the x slice is no longer read ----------
  __syncthreads();
  {
    const int c16 = lane & 15, g4 = lane >> 4;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int j = 0; j < 4; ++j) tile[(mb * 16 + g4 * 4 + j) * kPitch + wave * 16 + c16] = sum[mb][j];
  }
  __syncthreads();

  if (MB < 4 && r >= kRows) return;  // (whole waves; the counter is reset by thread 0)
  float lo[8], hi[8];
  {
    const float* src = tile + r * kPitch;
    const f32x4_t a0 = *reinterpret_cast<const f32x4_t*>(src + pr.col_lo);
    const f32x4_t a1 = *reinterpret_cast<const f32x4_t*>(src + pr.col_lo + 4);
    const f32x4_t b0 = *reinterpret_cast<const f32x4_t*>(src + pr.col_hi);
    const f32x4_t b1 = *reinterpret_cast<const f32x4_t*>(src + pr.col_hi + 4);
    lo[0] = a0.x; lo[1] = a0.y; lo[2] = a0.z; lo[3] = a0.w;
    lo[4] = a1.x; lo[5] = a1.y; lo[6] = a1.z; lo[7] = a1.w;
    hi[0] = b0.x; hi[1] = b0.y; hi[2] = b0.z; hi[3] = b0.w;
    hi[4] = b1.x; hi[5] = b1.y; hi[6] = b1.z; hi[7] = b1.w;
  }
  if (qk) {
    // RMSNorm over the head (fused_qkv_rope.py:98-100), then rotate-half RoPE
    // (:102-118).  Every fused multiply-add is explicit and nothing else is
    // contracted, so each instantiation of this code (the finish from partials
    // and the recompute finish) rounds identically.
#pragma clang fp contract(off)
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) ss = __builtin_fmaf(hi[i], hi[i], __builtin_fmaf(lo[i], lo[i], ss));
    ss = head_sum(ss, hd);
    const float rms = head_rms(ss, e.eps, hd);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float x1n = lo[i] * rms * elem_lane<E>(g_lo, i);
      const float x2n = hi[i] * rms * elem_lane<E>(g_hi, i);
      const float t1 = __builtin_fmaf(x1n, elem_lane<E>(c_lo, i), -(x2n * elem_lane<E>(s_lo, i)));
      const float t2 = __builtin_fmaf(x2n, elem_lane<E>(c_hi, i), x1n * elem_lane<E>(s_hi, i));
      lo[i] = t1;
      hi[i] = t2;
    }
  }
  if (row_in) {
    u32x4_t o1, o2;
    o1.x = E::pack2(lo[0], lo[1]);
    o1.y = E::pack2(lo[2], lo[3]);
    o1.z = E::pack2(lo[4], lo[5]);
    o1.w = E::pack2(lo[6], lo[7]);
    o2.x = E::pack2(hi[0], hi[1]);
    o2.y = E::pack2(hi[2], hi[3]);
    o2.z = E::pack2(hi[4], hi[5]);
    o2.w = E::pack2(hi[6], hi[7]);
    if (e.qkv) {
      const int H = d.H;
      uint16_t* base = d.out;
      if (base) {
        uint16_t* dst = base + (int64_t(rr) * H + d.hh) * kHeadDim;
        *reinterpret_cast<u32x4_t*>(dst + pr.col_lo) = o1;
        *reinterpret_cast<u32x4_t*>(dst + pr.col_hi) = o2;
      }
      if (cslot >= 0) {
        uint16_t* crow = paged_row(e, cslot, d.proj, d.hh);
        *reinterpret_cast<u32x4_t*>(crow + pr.col_lo) = o1;
        *reinterpret_cast<u32x4_t*>(crow + pr.col_hi) = o2;
      }
    } else {  // plain GEMM output [M, N] (whole 128-column tiles: N % 128 == 0)
      uint16_t* dst = e.out + int64_t(rr) * e.N + int64_t(d.head) * kHeadDim;
      *reinterpret_cast<u32x4_t*>(dst + pr.col_lo) = o1;
      *reinterpret_cast<u32x4_t*>(dst + pr.col_hi) = o2;
    }
  }
  if (tid == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The weights of a wave's 16 columns over its split of NK k tiles as bf16 MFMA
// fragments, held in registers (int4 weights dequantised once, in block 0).
template <int NK>
struct HeldWeights {
  u32x4_t b[NK][2];
};

// Block 0: streams the wave's weight slice from HBM into registers (16-bit weights: each
// tile's two fragments are requested about kDecLookahead tiles ahead of its
// MFMAs, after the x slice, so early tiles land early; int4: the packed words
// with their scales and zeros) and multiplies each 64-wide k tile as soon as it
// has landed.
template <class E, bool INT4, int MB, int NK>
__device__ __forceinline__ void first_block(const ProblemArgs& p, const WeightArgs& w, const DecWork& d,
                                            int kt0, uint16_t* xs, HeldWeights<NK>& hw, f32x4_t (&acc)[MB]) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int c16 = lane & 15, g4 = lane >> 4;
  const uint32_t xs_lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(xs));
  const int64_t kbeg = int64_t(kt0) * kBK;
  const int64_t col = int64_t(d.hh) * kHeadDim + wave * 16 + c16;
  constexpr int kAhead = MB == 4 ? kDecLookahead : kDecLookaheadSmall;
  constexpr int kLook = NK < kAhead ? NK : kAhead;
  if constexpr (!INT4) {
    const uint16_t* wp = pick3_uniform(d.proj, w.w[0], w.w[1], w.w[2]) + col * p.K + kbeg + g4 * 8;
    XStage<MB>(p, kbeg, xs_lds, 0).template all<NK>();
#pragma unroll
    for (int t = 0; t < kLook; ++t)
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) hw.b[t][kk] = wload(wp + t * kBK + kk * 32);
    wait_vm<2 * kLook>();  // the x slice has landed (older than the weight loads) ...
    barrier();             // ... in every wave
#pragma unroll
    for (int t = 0; t < NK; ++t) {
      if (t + kLook < NK) {
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) hw.b[t + kLook][kk] = wload(wp + (t + kLook) * kBK + kk * 32);
        // (left free, the compiler sank these loads below the next tiles' MFMAs until
        // three or four were in flight instead of 2 * kLook: hidden 4096, 32 / 8 heads,
        // T = 64 19.6 -> 19.0 us in a replayed graph)
        asm volatile("" ::: "memory");
      }
      mma_tile<E, MB>(xs, t, hw.b[t], acc);
    }
  } else {
    // int4 weights are 4x smaller: load them with their scales and zeros, then
    // the x slice, and wait for everything
    const Int4Col ic = int4_col(w, d.proj, col);
    uint32_t q4[NK][2], sraw[NK], zw[NK];
#pragma unroll
    for (int t = 0; t < NK; ++t) {
      const int64_t k0 = kbeg + int64_t(t) * kBK;
      const int64_t grp = k0 / ic.group;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) q4[t][kk] = uint32_t(load_global(ic.qw + (k0 / 8 + kk * 4 + g4) * ic.n + col));
      sraw[t] = load_global(ic.sc + grp * ic.n + col);
      zw[t] = uint32_t(load_global(ic.qz + grp * (ic.n / 8) + col / 8));
    }
    XStage<MB>(p, kbeg, xs_lds, 0).template all<NK>();
    wait_vm<0>();
    barrier();
#pragma unroll
    for (int t = 0; t < NK; ++t) {
      dequant_tile(ic, q4[t], sraw[t], zw[t], hw.b[t]);
      mma_tile<E, MB>(xs, t, hw.b[t], acc);
    }
  }
}

// Tiles per barrier when a later block consumes its x slice: the MFMAs of a
// group start once its tiles have landed, under the loads of the next groups.
constexpr int kDecGroup = 4;

// A later block at row r0: stages its x slice (NK direct loads per thread, in
// tile order) and multiplies it by the held weights, group by group as the tiles
// land.  After the first group's wait and barrier -- when every memory operation
// each thread issued before the call (e.g. a partial's stores) has completed --
// it calls after_first_wait() in every thread.
template <int NK, class F>
__device__ __forceinline__ void later_block(const ProblemArgs& p, int64_t kbeg, int r0, uint16_t* xs,
                                            const HeldWeights<NK>& hw, f32x4_t (&acc)[4], F&& after_first_wait) {
  const uint32_t xs_lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(xs));
  XStage<4>(p, kbeg, xs_lds, r0).template all<NK>();
#pragma unroll
  for (int g0 = 0; g0 < NK; g0 += kDecGroup) {
    const int g1 = g0 + kDecGroup < NK ? g0 + kDecGroup : NK;
    wait_vm_n(NK - g1);  // (the loads of the later groups may stay in flight)
    barrier();
    if (g0 == 0) after_first_wait();
#pragma unroll
    for (int t = g0; t < g1; ++t) mma_tile<Bf16, 4>(xs, t, hw.b[t], acc);
  }
}

// This wave's fp32 partial of block `blk` to part[split][blk][head][wave][mb][lane]
// (fragment order, 16-byte stores; not waited for here).
template <int MB>
__device__ __forceinline__ void publish_partial(const ProblemArgs& p, const DecWork& d, int blk,
                                                const f32x4_t (&acc)[MB], float* __restrict__ part) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  f32x4_t* mine = reinterpret_cast<f32x4_t*>(part) +
                  (((int64_t(d.split) * d.nblk + blk) * p.n_tiles + d.head) * kDecWaves + wave) * MB * 64 + lane;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) mine[mb * 64] = acc[mb];
}

__device__ __forceinline__ uint32_t arrive(uint32_t* counter, const DecWork& d) {
  return __hip_atomic_fetch_add(counter, d.inc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + d.inc;
}

// RoPE-table offset and paged-cache slot of this thread's row (tid / 8) of block b.
template <int MB>
__device__ __forceinline__ void block_rows(const EpilogueArgs& e, const DecWork& d, int M, int b, int64_t& prow,
                                           int64_t& cslot) {
  const int r = threadIdx.x >> 3;
  const int rr = b * 16 * MB + r;
  const bool in = (MB == 4 || r < 16 * MB) && rr < M;
  prow = (e.qkv == 1 && d.proj != 2 && in) ? rope_row(e, rr) * e.head_dim : 0;
  cslot = (e.qkv && d.proj != 0 && in) ? paged_slot(e, rr) : -1;
}

// The end of a one-block split: publishes its partial; the last split to arrive
// finishes the head (from the partials, or by recomputation when some split ran
// on another XCD).
template <class E, bool INT4, int MB, bool LONG>
__device__ __forceinline__ void combine_single(const ProblemArgs& p, const WeightArgs& w, const EpilogueArgs& e,
                                               const DecWork& d, const f32x4_t (&acc)[MB], int64_t prow, int64_t cslot,
                                               uint16_t* xs, uint32_t* arrival, float* __restrict__ part,
                                               uint32_t* __restrict__ counters) {
  publish_partial<MB>(p, d, 0, acc, part);
  __builtin_amdgcn_s_waitcnt(0);  // this thread's stores have reached the L2
  __syncthreads();                // ... and every thread's
  if (threadIdx.x == 0) arrival[0] = arrive(counters + d.head, d);
  __syncthreads();
  const uint32_t seen = arrival[0];
  if (!all_arrived(seen, d.splits)) return;
  if (any_foreign(seen, d.splits)) finish_block<E, INT4, MB, false, true, LONG>(p, w, e, d, 0, acc, prow, cslot, xs, part, counters);
  else finish_block<E, INT4, MB, false, false, LONG>(p, w, e, d, 0, acc, prow, cslot, xs, part, counters);
}

// Several 64-row blocks.  Block 0 streams the weights into registers; each later
// block stages its rows' x slice in the same LDS and multiplies it by the held
// weights, so the weights are read from HBM once per launch.
//
// Block b is finished by its designated split b % splits.  (Were the last split
// to arrive to finish it, the slowest split would finish every block and fall
// further behind each time.)  A block's arrival is counted one block later: the
// staging of the next block already waits for all outstanding memory operations,
// the partial's stores included, so the counter increment needs no wait of its
// own and its latency hides under the next block's MFMAs.  The designated split
// finishes a block when it arrives last; otherwise it notes the block and checks
// its counter again, without waiting, at its next blocks, and waits for what is
// still open after its last block.  That wait is bounded: on time-out the block is
// marked kAbandoned and its last split to arrive finishes it instead, so no
// workgroup waits on one that cannot start before it exits.  Blocks whose splits
// did not all run on the XCD the grid assumes are recomputed after the block
// loop, when the held weights no longer need their registers.
template <bool INT4, int NK>
__device__ __forceinline__ void run_split_multi(const ProblemArgs& p, const WeightArgs& w, const EpilogueArgs& e,
                                                const DecWork& d, int kt0, uint16_t* xs, uint32_t* arrival,
                                                float* __restrict__ part, uint32_t* __restrict__ counters) {
  const uint32_t xs_lds = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(xs));
  const int64_t kbeg = int64_t(kt0) * kBK;
  const int M = int(p.M);
  const int nblk = d.nblk;
  const int n_tiles = p.n_tiles;
  const bool tid0 = threadIdx.x == 0;
  const f32x4_t no_acc[4] = {};
  uint32_t deferred = 0;  // blocks to finish by recomputation after the loop
  uint32_t pending = 0;   // designated blocks noted, not yet finished
  HeldWeights<NK> hw;

  // Finish block b (counter value v, every split arrived), or defer it.
  auto finish_or_defer = [&](int b, uint32_t v) {
    if (any_foreign(v, d.splits)) {
      deferred |= 1u << b;
    } else {
      int64_t b_prow, b_cslot;
      block_rows<4>(e, d, M, b, b_prow, b_cslot);
      finish_block<Bf16, INT4, 4, true, false>(p, w, e, d, b, no_acc, b_prow, b_cslot, xs, part, counters);
    }
  };
  // The counter value of block b after this split's arrival (seen) and the value
  // of the oldest noted block read at the same time (probed, probe_blk >= 0):
  // finish what this split is due to finish.
  auto decide = [&](int b, uint32_t seen, int probe_blk, uint32_t probed) {
    const bool mine = b % d.splits == d.split;
    if (all_arrived(seen, d.splits) && (mine || (seen & kAbandoned))) finish_or_defer(b, seen);
    else if (mine) pending |= 1u << b;
    if (probe_blk >= 0 && probe_blk != b && all_arrived(probed, d.splits)) {
      pending &= ~(1u << probe_blk);
      finish_or_defer(probe_blk, probed);
    }
  };

  // (block 0 ahead of the loop: inside it, what the finish of another iteration may
  // still have in flight made the compiler wait for every weight load before the first
  // MFMA: hidden 4096, 32 / 8 heads, T = 128 27.4 -> 25.9 us, T = 300 32.7 -> 32.2)
  {
    f32x4_t acc[4];
    zero_acc(acc);
    first_block<Bf16, INT4, 4, NK>(p, w, d, kt0, xs, hw, acc);
    publish_partial<4>(p, d, 0, acc, part);
  }
#pragma unroll 1
  for (int blk = 1; blk < nblk; ++blk) {
    f32x4_t acc[4];
    zero_acc(acc);
    // this block's x slice in the same LDS once every wave is done with it (the
    // previous block's MFMAs or a finish).
    // Once its first tiles have landed, so have the previous block's partial
    // stores (issued earlier): then that block's arrival is counted and the
    // counter of the oldest noted block read; both values are used after this
    // block's MFMAs.
    barrier();
    const int probe_blk = pending != 0 ? __builtin_ctz(pending) : -1;
    uint32_t seen = 0, probed = 0;
    later_block<NK>(p, kbeg, blk * kDecRows, xs, hw, acc, [&]() {
      if (tid0) {
        seen = arrive(counters + (blk - 1) * n_tiles + d.head, d);
        if (probe_blk >= 0)
          probed = __hip_atomic_load(counters + probe_blk * n_tiles + d.head, __ATOMIC_RELAXED,
                                     __HIP_MEMORY_SCOPE_AGENT);
      }
    });
    publish_partial<4>(p, d, blk, acc, part);
    if (tid0) {
      arrival[0] = seen;
      arrival[1] = probed;
    }
    __syncthreads();
    seen = arrival[0];
    probed = arrival[1];
    __syncthreads();  // (arrival is rewritten by the next block)
    decide(blk - 1, seen, probe_blk, probed);
  }
  // the last block's arrival
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (tid0) arrival[0] = arrive(counters + (nblk - 1) * n_tiles + d.head, d);
  __syncthreads();
  const uint32_t last_seen = arrival[0];
  __syncthreads();
  decide(nblk - 1, last_seen, -1, 0);

  // the noted blocks still open
#pragma unroll 1
  while (pending != 0) {
    const int b = __builtin_ctz(pending);
    pending &= pending - 1u;
    uint32_t* counter = counters + b * n_tiles + d.head;
    if (tid0) {
      uint32_t v = __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      for (int spin = 0; !all_arrived(v, d.splits) && spin < d.max_spins; ++spin) {
        __builtin_amdgcn_s_sleep(2);
        v = __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      // give up: the last split to arrive sees kAbandoned and finishes the block;
      // if every split arrived meanwhile, the fetch-or returns a full count
      if (!all_arrived(v, d.splits))
        v = __hip_atomic_fetch_or(counter, kAbandoned, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      arrival[0] = v;
    }
    __syncthreads();
    const uint32_t v = arrival[0];
    __syncthreads();
    if (all_arrived(v, d.splits)) finish_or_defer(b, v);
  }
#pragma unroll 1
  for (int b = 0; b < nblk; ++b) {
    if (!(deferred >> b & 1u)) continue;
    int64_t b_prow, b_cslot;
    block_rows<4>(e, d, M, b, b_prow, b_cslot);
    __syncthreads();  // every wave is done with the LDS
    finish_block<Bf16, INT4, 4, true, true>(p, w, e, d, b, no_acc, b_prow, b_cslot, xs, part, counters);
  }
}

// The workgroup's split: grid position -> (head, split), XCD check, k range.
template <int ROWS>  // rows of a block
__device__ __forceinline__ DecWork dec_work(const ProblemArgs& p, const EpilogueArgs& e, int splits,
                                            int ctl, int& kt0, int& nk) {
  const int bid = blockIdx.x;
  const int xcds = p.xcds;
  const int q = bid / xcds;
  DecWork d;
  d.split = q % splits;
  d.head = (q / splits) * xcds + bid % xcds;
  d.splits = splits;
  d.nblk = int((p.M + ROWS - 1) / ROWS);
  split_head(d.head, e.Hq, e.Hkv, d.proj, d.hh);
  d.H = d.proj == 0 ? e.Hq : e.Hkv;
  d.gamma = pick3_uniform(d.proj, e.q_gamma, e.k_gamma, e.k_gamma);
  d.out = pick3_uniform(d.proj, e.q, e.k, e.v);
  // (XCC_ID is the physical XCD; a partition of the GPU holds xcds of them)
  d.inc = arrival_inc(xcc_id() % xcds, (ctl & 1) != 0);
  d.max_spins = ctl >> 1;
  split_range(d.split, splits, int(p.K / kBK), kt0, nk);
  return d;
}

// One block of up to 16 * MB rows (T <= 64: decode steps, tails).  MB = 4 and int4 weights:
// splits of at most kDecMaxNK tiles (decode_long_body runs longer ones); 16-bit weights
// with MB = 1 and 2: up to kDecLongMaxNK, whose x slice (64 or 128 KB) the LDS holds at
// once.  Each tile
// count's stream is its own unrolled code; what follows it is shared.
//
// Why the smaller blocks: at T <= 16 a 64-row block stages, multiplies, publishes and
// reads back four times the rows the call has.  Measured on MI355X (one call):
// hidden 4096, 32 / 8 heads T = 8 18.1 -> 15.6 us, T = 24 18.2 -> 16.6 us; hidden 1024,
// 16 / 8 heads T = 1 9.9 -> 8.4 us; int4 hidden 4096 T = 8 16.4 -> 12.8 us.  What is left
// at T <= 16 is the weight stream (50 MB at 5.1 TB/s: 9.9 us) and ~5 us of launch,
// first loads and the two cross-workgroup steps.
template <class E, bool INT4, int MB>
__device__ __forceinline__ void decode_body(const ProblemArgs& p, const WeightArgs& w, const EpilogueArgs& e, int splits,
                                            float* __restrict__ part, uint32_t* __restrict__ counters, int ctl) {
  // (sized for 64 rows whatever MB: more than half of the LDS keeps one workgroup per CU)
  __shared__ __attribute__((aligned(16))) uint16_t xs[kDecRows * kDecKc];
  __shared__ uint32_t arrival[2];
  if ((blockIdx.x / p.xcds / splits) * p.xcds + blockIdx.x % p.xcds >= p.n_tiles) return;  // padding
  int kt0, nk;
  const DecWork d = dec_work<16 * MB>(p, e, splits, ctl, kt0, nk);
  int64_t prow, cslot;  // read now: a positions[] load here is off every critical path
  block_rows<MB>(e, d, int(p.M), 0, prow, cslot);
  f32x4_t acc[MB];
  zero_acc<MB>(acc);
#define MQK_DEC_CASE(n)                                       \
  case n: {                                                   \
    HeldWeights<n> hw;                                        \
    first_block<E, INT4, MB, n>(p, w, d, kt0, xs, hw, acc);   \
    break;                                                    \
  }
#define MQK_DEC_CASES_16                                              \
  MQK_DEC_CASE(1) MQK_DEC_CASE(2) MQK_DEC_CASE(3) MQK_DEC_CASE(4)     \
  MQK_DEC_CASE(5) MQK_DEC_CASE(6) MQK_DEC_CASE(7) MQK_DEC_CASE(8)     \
  MQK_DEC_CASE(9) MQK_DEC_CASE(10) MQK_DEC_CASE(11) MQK_DEC_CASE(12)  \
  MQK_DEC_CASE(13) MQK_DEC_CASE(14) MQK_DEC_CASE(15) MQK_DEC_CASE(16)
  if constexpr (MB == 4 || INT4) {
    switch (nk) {
      MQK_DEC_CASES_16
      default: return;  // the launcher guarantees 1 <= nk <= kDecMaxNK
    }
  } else {
    switch (nk) {
      MQK_DEC_CASES_16
      MQK_DEC_CASE(17) MQK_DEC_CASE(18) MQK_DEC_CASE(19) MQK_DEC_CASE(20)
      MQK_DEC_CASE(21) MQK_DEC_CASE(22) MQK_DEC_CASE(23) MQK_DEC_CASE(24)
      MQK_DEC_CASE(25) MQK_DEC_CASE(26) MQK_DEC_CASE(27) MQK_DEC_CASE(28)
      MQK_DEC_CASE(29) MQK_DEC_CASE(30) MQK_DEC_CASE(31) MQK_DEC_CASE(32)
      default: return;  // ... 1 <= nk <= kDecLongMaxNK
    }
  }
#undef MQK_DEC_CASES_16
#undef MQK_DEC_CASE
  combine_single<E, INT4, MB, false>(p, w, e, d, acc, prow, cslot, xs, arrival, part, counters);
}

// One block whose splits are longer than one x slice (or, int4, than the packed words
// one slice can keep in registers)
// (kDecMaxNK < nk <= kDecLongMaxNK for the longest): two slices, the second staged
// once every wave is done with the first, its tiles accumulated after the first's,
// so the order of the sums is that of one slice.  16-bit weights: a first slice of
// kDecMaxNK tiles; int4: two halves (a 16-tile first slice keeps too many packed
// words live and spills).  (Balanced ranges: a launch whose longest split exceeds one
// slice has splits of at least kDecMaxNK tiles.)
template <class E, bool INT4, int MB>
__device__ __forceinline__ void decode_long_body(const ProblemArgs& p, const WeightArgs& w, const EpilogueArgs& e,
                                                 int splits, float* __restrict__ part, uint32_t* __restrict__ counters,
                                                 int ctl) {
  __shared__ __attribute__((aligned(16))) uint16_t xs[kDecRows * kDecKc];
  __shared__ uint32_t arrival[2];
  if ((blockIdx.x / p.xcds / splits) * p.xcds + blockIdx.x % p.xcds >= p.n_tiles) return;  // padding
  int kt0, nk;
  const DecWork d = dec_work<16 * MB>(p, e, splits, ctl, kt0, nk);
  int64_t prow, cslot;
  block_rows<MB>(e, d, int(p.M), 0, prow, cslot);
  f32x4_t acc[MB];
  zero_acc<MB>(acc);
  const int n1 = INT4 ? (nk + 1) / 2 : kDecMaxNK;
#define MQK_DEC_SLICE(n)                                             \
  case n: {                                                          \
    HeldWeights<n> hw;                                               \
    first_block<E, INT4, MB, n>(p, w, d, kt0 + from, xs, hw, acc);   \
    break;                                                           \
  }
#define MQK_DEC_SLICES_8_16                                                              \
  MQK_DEC_SLICE(8) MQK_DEC_SLICE(9) MQK_DEC_SLICE(10) MQK_DEC_SLICE(11) MQK_DEC_SLICE(12) \
  MQK_DEC_SLICE(13) MQK_DEC_SLICE(14) MQK_DEC_SLICE(15) MQK_DEC_SLICE(16)
  if constexpr (INT4) {
#pragma unroll 1
    for (int s = 0; s < 2; ++s) {  // (nk 16 .. 32: halves of 8 .. 16)
      const int from = s ? n1 : 0, n = s ? nk - n1 : n1;
      if (s) __syncthreads();  // every wave is done with the first x slice
      switch (n) {
        MQK_DEC_SLICES_8_16
        default: return;
      }
    }
  } else {
    {
      HeldWeights<kDecMaxNK> hw;
      first_block<E, INT4, MB, kDecMaxNK>(p, w, d, kt0, xs, hw, acc);
    }
    __syncthreads();
    const int from = n1;
    switch (nk - n1) {
      case 0: break;
      MQK_DEC_SLICE(1) MQK_DEC_SLICE(2) MQK_DEC_SLICE(3) MQK_DEC_SLICE(4)
      MQK_DEC_SLICE(5) MQK_DEC_SLICE(6) MQK_DEC_SLICE(7)
      MQK_DEC_SLICES_8_16
      default: return;  // the launcher guarantees kDecMaxNK <= nk <= kDecLongMaxNK
    }
  }
#undef MQK_DEC_SLICES_8_16
#undef MQK_DEC_SLICE
  combine_single<E, INT4, MB, true>(p, w, e, d, acc, prow, cslot, xs, arrival, part, counters);
}

// Several 64-row blocks, the weights held in registers across them.  Its splits
// cover NKC or NKC - 1 k tiles (balanced ranges), and each NKC is its own kernel
// so that the register allocation of the held weights fits the actual k range.
template <bool INT4, int NKC>
__device__ __forceinline__ void decode_multi_body(const ProblemArgs& p, const WeightArgs& w, const EpilogueArgs& e,
                                                  int splits, float* __restrict__ part, uint32_t* __restrict__ counters,
                                                  int ctl) {
  __shared__ __attribute__((aligned(16))) uint16_t xs[kDecRows * kDecKc];
  __shared__ uint32_t arrival[2];
  if ((blockIdx.x / p.xcds / splits) * p.xcds + blockIdx.x % p.xcds >= p.n_tiles) return;  // padding
  int kt0, nk;
  const DecWork d = dec_work<kDecRows>(p, e, splits, ctl, kt0, nk);
  if (nk == NKC) run_split_multi<INT4, NKC>(p, w, e, d, kt0, xs, arrival, part, counters);
  else if constexpr (NKC > 1) run_split_multi<INT4, NKC - 1>(p, w, e, d, kt0, xs, arrival, part, counters);
}

}  // namespace
}  // namespace mqk
