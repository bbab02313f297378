// The fused front for fp32 (and fp16) callers: x, weights, norm weights and
// RoPE tables in that type, q / k / v out in it.  The reference op accepts such
// tensors too (mini_qwen/kernels/fused_qkv_rope.py:130-195; the fp32 layer of the
// reference's CPU-runnable configuration), but its Triton kernel rounds every Q /
// K output to bf16 before storing it into the fp32 / fp16 buffer (:117-120), and
// with fp16 tensors its GEMM output is rounded to fp16 before the norm.  This
// kernel keeps the fp32 projection, norm and RoPE and rounds once, to the output
// type: it computes the op's fp32 composition (the unfused reference path,
// attention.py:102-109) to fp32 / fp16 precision, not the fused reference's bits.
//
// fp32: one workgroup of eight waves computes 16 * MB token rows x one head (128
// columns), a wave 16 columns of every row, on the fp32 matrix core (products and sums
// in fp32).  fp16 callers whose hidden size or tables the 16-bit tile kernels do not
// take run f16_f32_qkv_kernel, further down.  In both the accumulators then go through
// LDS so that eight threads hold a row's 128 dims (each the RoPE pairs d, d+64 for eight
// d), apply RMSNorm and RoPE in fp32, and store.
#include <type_traits>

#include "mqk_device.h"
#include "mqk_kernels.h"

namespace mqk {
namespace {

constexpr int kEpiPitch = kHeadDim + 4;  // LDS row pitch of the accumulator tile

// Element i of a norm weight or RoPE table of type T, as fp32.
template <class T>
__device__ __forceinline__ float elem(const void* p, int64_t i) {
  return float(static_cast<const T*>(p)[i]);
}
// 8 values stored as 8 consecutive elements
template <class T>
__device__ __forceinline__ void store8(void* dst, const float (&v)[8], int i0) {
  if constexpr (sizeof(T) == 4) {
    float* d = static_cast<float*>(dst);
    *reinterpret_cast<f32x4_t*>(d) = f32x4_t{v[i0], v[i0 + 1], v[i0 + 2], v[i0 + 3]};
    *reinterpret_cast<f32x4_t*>(d + 4) = f32x4_t{v[i0 + 4], v[i0 + 5], v[i0 + 6], v[i0 + 7]};
  } else {
    typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
    h8_t h;
#pragma unroll
    for (int i = 0; i < 8; ++i) h[i] = _Float16(v[i0 + i]);
    *static_cast<h8_t*>(dst) = h;
  }
}

// Norm, RoPE and store of the accumulator tile ep [rows][kEpiPitch], of token rows
// row0 + r: thread tid has row r = tid / 8, dims d = 8c .. 8c+7 and 64 + 8c ..
// (c = tid % 8).  Waves whose rows are past the tile's leave whole.
template <class T, int ROWS>
__device__ __forceinline__ void finish_rows(const F32Args& a, const float* ep, int proj, int hh, int64_t row0) {
  const int r = int(threadIdx.x) >> 3, c = int(threadIdx.x) & 7;
  if (r >= ROWS) return;
  const int64_t t = row0 + r;
  const int hd = a.head_dim;
  const PairRuns pr = pair_runs(c, hd);  // (head_dim 64: two heads per block)
  float lo[8], hi[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    lo[i] = ep[r * kEpiPitch + pr.col_lo + i];
    hi[i] = ep[r * kEpiPitch + pr.col_hi + i];
  }
  if (proj < 2) {
    // (every lane of the row's lane group takes part in the sum; rows past M are copies of row M - 1, or zeros)
    const float ss = head_sum(run_sumsq(lo, hi), hd);
    const float rms = head_rms(ss, a.eps, hd);
    if (t < a.M) {
      const void* g = proj == 0 ? a.q_gamma : a.k_gamma;
      const int64_t prow = rope_row(a, t) * hd;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
#pragma clang fp contract(off)
        const int d = pr.dim_lo + i, d2 = pr.dim_hi + i;
        const float x1n = lo[i] * rms * elem<T>(g, d);
        const float x2n = hi[i] * rms * elem<T>(g, d2);
        lo[i] = __builtin_fmaf(x1n, elem<T>(a.cos, prow + d), -(x2n * elem<T>(a.sin, prow + d)));
        hi[i] = __builtin_fmaf(x2n, elem<T>(a.cos, prow + d2), x1n * elem<T>(a.sin, prow + d2));
      }
    }
  }
  if (t < a.M) {
    const int H = proj == 0 ? a.Hq : a.Hkv;
    T* dst = static_cast<T*>(pick3_uniform(proj, a.q, a.k, a.v)) + (t * H + hh) * kHeadDim;
    store8<T>(dst + pr.col_lo, lo, 0);
    store8<T>(dst + pr.col_hi, hi, 0);
  }
}

// The fp32 kernel (tiles of 32 rows and more; 16-row tiles: F32Narrow).  Its bound at
// T = 128, hidden 1024, 16 / 8 heads is the fp32 matrix
// core (6.8 us at 256 operations a clock and CU); the weights, 16 MB, take 3.3 us.  So
// nothing is allowed between the MFMAs but their operands:
//   * a weight element is used by one wave only, so weights go from the L2 to registers,
//     16 bytes (4 k) a lane, two stages ahead of their MFMAs;
//   * x, which all eight waves read, goes L2 -> LDS directly (dma16) into a ring of three
//     stages, with one barrier per stage: stage s + 2 overwrites the slot of s - 1, which
//     every wave has left when it arrives at the barrier of s.
// k order: in a group of 16 k, lane (c, g) = (lane & 15, lane >> 4) holds k = 4g .. 4g+3
// of its x row / weight row c, and MFMA i of the group takes element i of both.
// LDS stage: panels [row][64 floats] of 16 chunks of 16 bytes, chunk c of row r in slot
// c ^ (r & 15): the 16 rows that a quarter-wave reads are 16 different slots.
// Measured on MI355X (replayed graph; before: both operands through registers into LDS,
// 32 k ahead): hidden 1024, 16 / 8 heads T = 256 28.1 -> 23.4 us; T = 512 44.9 -> 39.8;
// hidden 2048, 32 / 4 heads T = 300 83.6 -> 71.0; T = 1024 189.7 -> 178.4 (120 TFLOP/s; a
// large fp32 matrix product reaches 131).
template <int MB>
struct F32Tile {
  static constexpr int kRows = 16 * MB;
  static constexpr int kStageK = 64;  // k per stage
  static constexpr int kQuads = kStageK / 16;         // weight loads per lane and stage
  static constexpr int kStageBytes = kRows * kStageK * 4;
  static constexpr int kLoads = kStageBytes / 1024;   // dma16 per stage, over the 8 waves
  static constexpr int kDma = (kLoads + 7) / 8;       // ... of each wave (the last ones twice if it is not whole)
  static constexpr int kEpiBytes = kRows * kEpiPitch * 4;
  static constexpr int kLdsBytes = 3 * kStageBytes > kEpiBytes ? 3 * kStageBytes : kEpiBytes;
};
constexpr int kF32Threads = 512;

template <int MB>
struct F32Stream {
  using Tile = F32Tile<MB>;
  static constexpr int kQuads = Tile::kQuads;
  static constexpr int kLdsBytes = Tile::kLdsBytes;
  const float* xsrc[Tile::kDma];  // this lane's chunk of each of its rows, k 0
  int xk[Tile::kDma];             // ... its k within a stage
  uint32_t xdst[Tile::kDma];      // LDS byte address of each load in slot 0
  const float* wp;                // this lane's weight row, k 4g
  const float* xs;
  int K;
  f32x4_t w[3][kQuads];
  f32x4_t acc[MB];

  __device__ __forceinline__ F32Stream(const F32Args& a, const float* W, int64_t row0, const float* lds)
      : xs(lds), K(int(a.K)) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
#pragma unroll
    for (int j = 0; j < Tile::kDma; ++j) {
      int i = wave + 8 * j;
      if (Tile::kLoads % 8 != 0 && i >= Tile::kLoads) i = Tile::kLoads - 1;
      const int flat = i * 4 + (lane >> 4), row = flat % Tile::kRows, panel = flat / Tile::kRows;
      // rows past M re-read row M - 1: they feed output rows that are not stored
      const int64_t grow = row0 + row < a.M ? row0 + row : a.M - 1;
      xsrc[j] = static_cast<const float*>(a.x) + grow * a.K;
      xk[j] = panel * 64 + ((lane & 15) ^ (row & 15)) * 4;
      xdst[j] = base + uint32_t(i * 1024);
    }
    wp = W + int64_t(wave * 16 + (lane & 15)) * a.K + (lane >> 4) * 4;
#pragma unroll
    for (auto& v : acc) v = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  // Stage s in slot and registers J: its x, and its weights of group q (k past K re-reads
  // the row's last chunk / group; those products are not formed).
  template <int J>
  __device__ __forceinline__ void load_x(int s) {
#pragma unroll
    for (int j = 0; j < Tile::kDma; ++j) {
      int k = s * Tile::kStageK + xk[j];
      k = k < K ? k : K - 4;
      dma16(xsrc[j] + k, xdst[j] + uint32_t(J * Tile::kStageBytes));
    }
  }
  template <int J>
  __device__ __forceinline__ void load_w(int s, int q) {
    int k = s * Tile::kStageK + 16 * q;
    k = k < K ? k : K - 16;
    w[J][q] = load_global(reinterpret_cast<const f32x4_t*>(wp + k));
    asm volatile("" ::: "memory");  // (the waits count these loads; none may move past here)
  }
  template <int J>
  __device__ __forceinline__ void issue(int s) {
    load_x<J>(s);
#pragma unroll
    for (int q = 0; q < kQuads; ++q) load_w<J>(s, q);
  }
  template <int J>
  __device__ __forceinline__ void read_x(int q, f32x4_t (&x)[MB]) const {
    const int lane = threadIdx.x & 63, c16 = lane & 15, g4 = lane >> 4;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
      x[mb] = *reinterpret_cast<const f32x4_t*>(xs + J * (Tile::kStageBytes / 4) + (q / 4) * (Tile::kRows * 64) +
                                                (mb * 16 + c16) * 64 + (((q % 4) * 4 + g4) ^ c16) * 4);
  }
  // The groups of the stage in slot J, with MORE the loads of stage s + 2 among them (in
  // one run ahead of the MFMAs they keep the matrix cores waiting for the address unit:
  // T = 256, hidden 1024 26.3 -> 23.3 us).
  template <int J, bool MORE, bool LAST>
  __device__ __forceinline__ void multiply(int s, int groups) {
    constexpr int kNext = (J + 2) % 3;
    if (MORE) load_x<kNext>(s + 2);
    f32x4_t x[2][MB];  // the next group's x under this group's MFMAs
    read_x<J>(0, x[0]);
#pragma unroll
    for (int q = 0; q < kQuads; ++q) {
      if (LAST && q >= groups) break;
      if (MORE) load_w<kNext>(s + 2, q);
      if (q + 1 < kQuads) read_x<J>(q + 1, x[(q + 1) & 1]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
          f32x4_t& c = acc[mb];
          c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[q & 1][mb][i], w[J][q][i], c, 0, 0, 0);
        }
      // (left free, the compiler reads the whole stage first: too many registers for two
      // workgroups per CU)
      __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (no read of this slot in flight at the next barrier)
  }
  // Stage s with stage s + 2 put under way.  Issued after the x of s: the weights of s
  // and all of s + 1.
  template <int J, bool MORE>
  __device__ __forceinline__ void step(int s) {
    wait_vm<2 * kQuads + Tile::kDma>();
    barrier();
    multiply<J, MORE, false>(s, kQuads);
  }
  template <int J>
  __device__ __forceinline__ void last(int s) {
    wait_vm<0>();
    barrier();
    multiply<J, false, true>(s, (K - s * Tile::kStageK + 15) / 16);
  }
  __device__ __forceinline__ void run() {
    const int n = (K + Tile::kStageK - 1) / Tile::kStageK;
    if (n == 1) {
      issue<1>(0);
    } else {
      // (slots so that the last two stages are always in 0 and 1: the loads that each
      // wait counts are then the same on every path)
      int s = (n - 2) % 3;
      if (s == 0) {
        issue<0>(0);
        issue<1>(1);
      } else if (s == 1) {
        issue<2>(0);
        issue<0>(1);
        step<2, true>(0);
      } else {
        issue<1>(0);
        issue<2>(1);
        step<1, true>(0);
        step<2, true>(1);
      }
#pragma unroll 1
      for (; s < n - 2; s += 3) {
        step<0, true>(s);
        step<1, true>(s + 1);
        step<2, true>(s + 2);
      }
      step<0, false>(s);
    }
    last<1>(n - 1);
  }
};

// dma16 of the 16 bytes at uniform base `from` + `off` bytes.
__device__ __forceinline__ void dma16_from(const void* from, uint32_t off, uint32_t lds_base) {
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %1\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %2, %3\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved)
      : "s"(__builtin_amdgcn_readfirstlane(lds_base)), "v"(off), "s"(from)
      : "memory");
}

// 16-row tiles: a weight element serves one MFMA only, and a wave's register load of 16
// weight rows x 64 bytes occupies the CU's load path for ~64 clocks (13.8 us for the 512
// KB of 128 columns at hidden 1024, whatever the number of rows: above the 8.2 us of the
// MFMAs).  So here the weights too go to LDS, as loads of 4 rows x 256 bytes, each wave's
// 16 columns to a ring of its own that needs no barrier; x comes in units of four stages
// with one barrier each, and the first reads of a stage are issued under the last MFMAs
// of the one before.  Measured as above: T = 128, hidden 1024, 16 / 8 heads 22.4 -> 16.4 us.
struct F32Narrow {
  static constexpr int kStageK = 64;
  static constexpr int kPanel = 16 * kStageK;  // floats of 16 rows of one stage (4 KB)
  static constexpr int kXStages = 4;           // stages per unit of x
  static constexpr int kXRing = 3, kWRing = 3;
  static constexpr int kXFloats = kXRing * kXStages * kPanel;
  static constexpr int kLdsBytes = (kXFloats + kWRing * 8 * kPanel) * 4;
  const float* xb;        // (uniform) x row row0, and this wave's first weight row
  const float* wb;
  uint32_t xo[2], wo[4];  // this lane's byte offset from there to its row of each load
  int xk[2], wk[4];       // ... and its k in the load's 64
  uint32_t base;
  const float* lds;
  int K, n, wave, lane;
  f32x4_t acc[2], x[2], w[2];

  __device__ __forceinline__ F32Narrow(const F32Args& a, const float* W, int64_t row0, const float* lds_)
      : lds(lds_), K(int(a.K)), n(int((a.K + kStageK - 1) / kStageK)),
        wave(__builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6)), lane(int(threadIdx.x) & 63) {
    base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
    const int r4 = lane >> 4, slot = lane & 15;
    xb = static_cast<const float*>(a.x) + row0 * a.K;
    wb = W + int64_t(wave * 16) * a.K;
#pragma unroll
    for (int j = 0; j < 2; ++j) {  // load i = 2 wave + j of a unit: panel i / 4, rows 4 (i % 4) ..
      const int row = (2 * wave + j) % 4 * 4 + r4;
      // rows past M re-read row M - 1: they feed output rows that are not stored
      xk[j] = (slot ^ row) * 4;
      xo[j] = (uint32_t(row0 + row < a.M ? row : int(a.M - 1 - row0)) * uint32_t(K) + uint32_t(xk[j])) * 4;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      wk[j] = (slot ^ (j * 4 + r4)) * 4;
      wo[j] = (uint32_t(j * 4 + r4) * uint32_t(K) + uint32_t(wk[j])) * 4;
    }
    acc[0] = acc[1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  // 64 k of 4 rows from k0 (k past K re-reads the row's last chunk; those products are
  // not formed).  Uniform base and a lane offset that stays: with a 64-bit address per lane
  // and load, the address arithmetic held up the MFMAs (T = 128, hidden 1024 18.6 us
  // against 16.4).
  template <bool WHOLE>
  __device__ __forceinline__ void load(const float* from, uint32_t off, int k, int k0, uint32_t dst) const {
    if (!WHOLE && k0 + kStageK > K) {
      const int in_row = k0 + k < K ? k0 + k : K - 4;
      dma16_from(from, off + uint32_t(in_row - k) * 4, dst);
    } else {
      dma16_from(from + k0, off, dst);
    }
  }
  __device__ __forceinline__ void load_x(int u) const {
#pragma unroll
    for (int j = 0; j < 2; ++j)
      load<false>(xb, xo[j], xk[j], u * kXStages * kStageK + (2 * wave + j) / 4 * kStageK,
                  base + uint32_t((u % kXRing * kXStages * kPanel) * 4 + (2 * wave + j) * 1024));
  }
  template <bool WHOLE = false>
  __device__ __forceinline__ void load_w(int s, int j) const {
    load<WHOLE>(wb, wo[j], wk[j], s * kStageK,
                base + uint32_t((kXFloats + (s % kWRing * 8 + wave) * kPanel) * 4 + j * 1024));
  }
  __device__ __forceinline__ void read(int s, int q) {
    const int c16 = lane & 15, g4 = lane >> 4;
    const int at = c16 * 64 + ((q * 4 + g4) ^ c16) * 4;
    x[q & 1] = *reinterpret_cast<const f32x4_t*>(lds + (s / kXStages % kXRing * kXStages + s % kXStages) * kPanel + at);
    w[q & 1] = *reinterpret_cast<const f32x4_t*>(lds + kXFloats + (s % kWRing * 8 + wave) * kPanel + at);
  }
  __device__ __forceinline__ void mfmas(int q) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      acc[q & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[q & 1][i], w[q & 1][i], acc[q & 1], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  }
  // Until stage s has landed with LATER of this wave's loads under way.  A stage that
  // begins a unit of x waits for every wave's part of it; arriving there, a wave has no
  // read of the unit before in flight, whose slot the loads after the barrier overwrite.
  template <int LATER>
  __device__ __forceinline__ void landed(int s) const {
    wait_vm<LATER>();
    if (s % kXStages == 0) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      barrier();
    }
  }
  // Stage s with the loads of stage s + 2 (into the slot of s - 1, whose reads the MFMAs
  // above have waited for) and, every fourth stage, of x two units on among its MFMAs.
  template <bool WHOLE>
  __device__ __forceinline__ void stage(int s) {
    const bool more_x = s % kXStages == 0 && s + 2 * kXStages < n;
    if (more_x) load_x(s / kXStages + 2);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      load_w<WHOLE>(s + 2, q);
      if (q < 3) {
        read(s, q + 1);
      } else {
        if (more_x) {
          landed<6>(s + 1);
        } else {
          landed<4>(s + 1);
        }
        read(s + 1, 0);
      }
      mfmas(q);
    }
  }
  __device__ __forceinline__ void run() {
    load_x(0);
    if (n > kXStages) load_x(1);
#pragma unroll
    for (int j = 0; j < 4; ++j) load_w(0, j);
    if (n == 1) {
      landed<0>(0);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) load_w(1, j);
      landed<4>(0);
    }
    read(0, 0);
    int s = 0;
    const int whole = K / kStageK;
#pragma unroll 1
    for (; s + 2 < whole; ++s) stage<true>(s);
    if (s + 2 < n) {
      stage<false>(s);
      ++s;
    }
    if (s + 2 == n) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (q < 3) {
          read(s, q + 1);
        } else {
          landed<0>(s + 1);
          read(s + 1, 0);
        }
        mfmas(q);
      }
      ++s;
    }
    const int groups = (K - s * kStageK + 15) / 16;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (q >= groups) break;
      if (q < 3) read(s, q + 1);
      mfmas(q);
    }
  }
};

template <int MB>
__global__ void __launch_bounds__(kF32Threads, MB == 1 ? 2 : 4) f32_qkv_kernel(F32Args a, int xcds) {
  using Stream = std::conditional_t<MB == 1, F32Narrow, F32Stream<MB>>;
  constexpr int kRows = 16 * MB;
  __shared__ __attribute__((aligned(16))) float lds[Stream::kLdsBytes / 4];
  const int n_rt = int((a.M + kRows - 1) / kRows);
  const int tile = xcd_tile_id(int(blockIdx.x), int(gridDim.x), xcds);
  const int rt = tile % n_rt;
  const int h = tile / n_rt;
  int proj, hh;
  split_head(h, a.Hq, a.Hkv, proj, hh);
  const float* W = static_cast<const float*>(pick3_uniform(proj, a.w[0], a.w[1], a.w[2])) + int64_t(hh) * kHeadDim * a.K;
  const int64_t row0 = int64_t(rt) * kRows;
  Stream st(a, W, row0, lds);
  st.run();
  __syncthreads();  // every wave is done with the ring
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if constexpr (MB == 1) st.acc[0] += st.acc[1];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      lds[(mb * 16 + 4 * (lane >> 4) + j) * kEpiPitch + 16 * wave + (lane & 15)] = st.acc[mb][j];
  __syncthreads();
  finish_rows<float, kRows>(a, lds, proj, hh, row0);
}

// The fp16 kernel: four waves, ROWS (32, or 16 when 32-row tiles would leave CUs idle) x
// 128 columns, a wave 32 columns; k tiles of 32 staged in LDS (row pitch kHPitch halves:
// 8-byte reads free of bank conflicts), the next tile's loads in registers under the
// current tile's MFMAs, on the fp16 matrix cores (exact products, fp32 sums).  It takes
// hidden sizes that are no multiple of 64 and tables that are not 16-byte aligned; the
// 16-bit tile kernels run the rest, about three times as fast.
constexpr int kKT = kF32BK;
constexpr int kHPitch = kKT + 4;
constexpr int kThreads = 256;
static_assert(kHeadDim * kHPitch * 2 <= 32 * kEpiPitch * 4, "the accumulator tile reuses the weight tile's LDS");

template <int ROWS>
__global__ void __launch_bounds__(kThreads) f16_f32_qkv_kernel(F32Args a, int xcds) {
  static_assert(ROWS == 16 || ROWS == 32, "row tile");
  typedef _Float16 T;
  typedef _Float16 h4_t __attribute__((ext_vector_type(4)));
  __shared__ __attribute__((aligned(16))) T xh[ROWS * kHPitch];
  __shared__ __attribute__((aligned(16))) float ep[32 * kEpiPitch];  // the weight tile, then the accumulator tile
  T* wh = reinterpret_cast<T*>(ep);
  const int n_rt = int((a.M + ROWS - 1) / ROWS);
  const int tile = xcd_tile_id(int(blockIdx.x), int(gridDim.x), xcds);
  const int rt = tile % n_rt;
  const int h = tile / n_rt;
  int proj, hh;
  split_head(h, a.Hq, a.Hkv, proj, hh);
  const T* W = static_cast<const T*>(a.w[proj]) + int64_t(hh) * kHeadDim * a.K;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t row0 = int64_t(rt) * ROWS;

  // staging: thread tid loads 4 consecutive k of x row (tid / 8) (threads of
  // rows < ROWS) and of weight rows (tid / 8) + 32 j, j = 0..3
  const int sr = tid >> 3, sk = (tid & 7) * 4;
  const bool x_row = sr < ROWS;
  const bool x_in = x_row && row0 + sr < a.M;
  const T* xp = static_cast<const T*>(a.x) + (x_in ? (row0 + sr) * a.K : 0) + sk;
  const T* wp = W + int64_t(sr) * a.K + sk;
  h4_t xr4, wr4[4];
  auto hload = [&](int64_t k0) {
    xr4 = x_in ? *reinterpret_cast<const h4_t*>(xp + k0) : h4_t{};
#pragma unroll
    for (int j = 0; j < 4; ++j) wr4[j] = *reinterpret_cast<const h4_t*>(wp + int64_t(32 * j) * a.K + k0);
  };
  auto hstage = [&]() {
    if (x_row) *reinterpret_cast<h4_t*>(xh + sr * kHPitch + sk) = xr4;
#pragma unroll
    for (int j = 0; j < 4; ++j) *reinterpret_cast<h4_t*>(wh + (sr + 32 * j) * kHPitch + sk) = wr4[j];
  };
  if constexpr (ROWS == 32) {
    f32x16_t acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
    // lane l: x row (l & 31), weight row 32 * wave + (l & 31), k 4 (l >> 5) .. +4 of each 8
    const _Float16* xa = xh + (lane & 31) * kHPitch + 4 * (lane >> 5);
    const _Float16* wb = wh + (32 * wave + (lane & 31)) * kHPitch + 4 * (lane >> 5);
    hload(0);
    for (int64_t k0 = 0; k0 < a.K; k0 += kKT) {
      hstage();
      __syncthreads();
      if (k0 + kKT < a.K) hload(k0 + kKT);
#pragma unroll
      for (int kk = 0; kk < kKT / 8; ++kk)
        acc = __builtin_amdgcn_mfma_f32_32x32x8f16(*reinterpret_cast<const h4_t*>(xa + 8 * kk),
                                                    *reinterpret_cast<const h4_t*>(wb + 8 * kk), acc, 0, 0, 0);
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
      ep[(8 * (i >> 2) + 4 * (lane >> 5) + (i & 3)) * kEpiPitch + 32 * wave + (lane & 31)] = acc[i];
  } else {
    f32x4_t acc[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // lane l: x row (l & 15), weight rows 32 * wave + 16 b + (l & 15), k 4 (l >> 4) .. +4 of each 16
    const _Float16* xa = xh + (lane & 15) * kHPitch + 4 * (lane >> 4);
    const _Float16* wb = wh + (32 * wave + (lane & 15)) * kHPitch + 4 * (lane >> 4);
    hload(0);
    for (int64_t k0 = 0; k0 < a.K; k0 += kKT) {
      hstage();
      __syncthreads();
      if (k0 + kKT < a.K) hload(k0 + kKT);
#pragma unroll
      for (int kk = 0; kk < kKT / 16; ++kk)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          acc[b] = __builtin_amdgcn_mfma_f32_16x16x16f16(
              *reinterpret_cast<const h4_t*>(xa + 16 * kk),
              *reinterpret_cast<const h4_t*>(wb + 16 * b * kHPitch + 16 * kk), acc[b], 0, 0, 0);
      __syncthreads();
    }
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        ep[(4 * (lane >> 4) + j) * kEpiPitch + 32 * wave + 16 * b + (lane & 15)] = acc[b][j];
  }
  __syncthreads();
  finish_rows<T, ROWS>(a, ep, proj, hh, row0);
}

// Token rows per workgroup: the least time of the busiest CU, the larger tile when two
// are equal (it reads the weights fewer times).  One tile of 16, 32, 48, 64 rows took 21,
// 34.5, 51, 66 us at hidden 2048 beyond the launch (and half of that at 1024): their
// ratios are kCost.  Counting rows alone put 16-row tiles at T = 700, 32 / 4 heads: 164
// us, 64-row tiles 141.
int f32_tile_rows(int64_t M, int64_t K, int64_t heads, int cus) {
  constexpr int kCost[4] = {21, 33, 49, 64};
  // (16-row tiles: byte offsets of 16 rows in 32 bits)
  const int first = K < (int64_t(1) << 26) ? 1 : 2;
  int rows = 0;
  int64_t least = 0;
  for (int mb = first; mb <= 4; ++mb) {
    const int64_t tiles = (M + 16 * mb - 1) / (16 * mb) * heads;
    const int64_t cost = (tiles + cus - 1) / cus * kCost[mb - 1];
    if (rows == 0 || cost <= least) {
      least = cost;
      rows = 16 * mb;
    }
  }
  return rows;
}

}  // namespace

hipError_t launch_f32_qkv(const F32Args& a, bool half, int cus, int xcds, hipStream_t stream) {
  const int64_t heads = a.Hq + 2 * a.Hkv;
  auto blocks = [&](int rows) { return (a.M + rows - 1) / rows * heads; };
  int rows;
  if (half) {
    rows = blocks(32) < cus ? 16 : 32;
  } else {
    rows = f32_tile_rows(a.M, a.K, heads, cus);
  }
  if (a.K % kF32BK != 0 || a.K > (int64_t(1) << 30) || blocks(rows) <= 0 || blocks(rows) > (int64_t(1) << 31) - 1)
    return hipErrorInvalidValue;
  using Kernel = void (*)(F32Args, int);
  const Kernel k = half ? (rows == 16 ? f16_f32_qkv_kernel<16> : f16_f32_qkv_kernel<32>)
                        : (rows == 16   ? f32_qkv_kernel<1>
                           : rows == 32 ? f32_qkv_kernel<2>
                           : rows == 48 ? f32_qkv_kernel<3>
                                        : f32_qkv_kernel<4>);
  hipLaunchKernelGGL(k, dim3(unsigned(blocks(rows))), dim3(half ? kThreads : kF32Threads), 0, stream, a, xcds);
  return hipGetLastError();
}

}  // namespace mqk
