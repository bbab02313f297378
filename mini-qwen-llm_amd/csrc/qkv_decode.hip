// Split-K projection for small token counts (decode steps, T <= 64, and up to
// sixteen 64-row blocks per launch at mid T) with the per-head norm + RoPE
// applied once the split partial sums of a block are combined.
//
// At decode the op is weight-read bound: Qwen3-8B's 50 MB of projection
// weights against 64 tokens.  Measured on MI355X: one CU sustains only a few
// tens of GB/s of reads, so every CU must stream its share of the weights;
// splitting a head's columns (instead of K) would re-read the activations from
// L2 per workgroup, which measured 3-4x slower than the weight stream itself;
// and two workgroups sharing a CU finish twice as late as one alone.  Hence:
//   * one 512-thread workgroup per CU (its activation slice in LDS is larger
//     than half the LDS, so the hardware cannot co-schedule two);
//   * each head is split along K into S = floor(CUs per XCD / heads per XCD)
//     k-ranges, and the grid maps all splits of head h to XCD h % 8
//     (workgroup b runs on XCD b % 8), so every XCD gets the same number of
//     workgroups, at most one per CU;
//   * inside a workgroup, wave w owns columns [16w, 16w+16) of the head over
//     the split's whole k-range, for all 64 token rows (v_mfma_f32_16x16x32_bf16,
//     4 row blocks, so each weight fragment feeds 4 MFMAs and no reduction
//     between waves is needed).  The activation slice is staged once in LDS
//     with direct L2 -> LDS loads; the wave's weight slice streams HBM -> VGPR,
//     all of it issued up front, and each 64-wide k tile is multiplied as soon
//     as its fragments land.
// Combining the splits: each workgroup writes its fp32 partial tile [64 x 128]
// (in MFMA fragment order, 16-byte stores) with plain stores, which stay in (or are written back from) the L2 of its
// XCD, and bumps the head's arrival counter; the workgroup that arrives last
// reads the other partials with plain loads -- all of them were written
// through the same L2 -- adds them in split order, applies RMSNorm over the
// head (fused_qkv_rope.py:98-100) and rotate-half RoPE (:102-118), writes
// bf16 q/k (or v unchanged) and resets the counter for the next call.
// Device-coherent (sc1) accesses measured ~0.5 TB/s and an agent-scope fence
// pair (L2 writeback + invalidate) ~2x the whole op, so neither is used.
//
// Each workgroup checks the XCD it actually runs on (hardware register
// XCC_ID).  If any split of a head ran elsewhere, its partial may sit in a
// different L2, so the last workgroup instead recomputes every split of the
// head itself, with the same per-split arithmetic and summation order: slower,
// bit-identical, and correct whatever the dispatch order.
#include "qkv_decode.h"

namespace mqk {
namespace {

template <int MB>
__global__ void __launch_bounds__(kDecThreads, 1)
decode_kernel(ProblemArgs p, WeightArgs w, EpilogueArgs e, int splits, float* __restrict__ part,
              uint32_t* __restrict__ counters, int ctl) {
  decode_body<Bf16, false, MB>(p, w, e, splits, part, counters, ctl);
}

__global__ void __launch_bounds__(kDecThreads, 1)
decode_long_kernel(ProblemArgs p, WeightArgs w, EpilogueArgs e, int splits, float* __restrict__ part,
                   uint32_t* __restrict__ counters, int ctl) {
  decode_long_body<Bf16, false, 4>(p, w, e, splits, part, counters, ctl);
}

}  // namespace

DecKernel decode_kernel_bf16(int mb) { return mb == 1 ? decode_kernel<1> : (mb == 2 ? decode_kernel<2> : decode_kernel<4>); }
DecKernel decode_long_kernel_bf16() { return decode_long_kernel; }

int g_decode_force_recompute = 0;
int g_decode_max_spins = kDecMaxSpins;

int decode_splits_for(int64_t M, int64_t K, int n_tiles, int requested, int cus, int xcds) {
  (void)M;
  const int nkt = int(K / kBK);
  if (nkt < 1) return 0;
  const int max_nk = kDecLongMaxNK;  // (both weight formats: splits of up to two x slices)
  const int min_splits = (nkt + max_nk - 1) / max_nk;  // bound on a split's k-range
  int s = requested;
  if (s <= 0) {
    // one workgroup per CU: (heads per XCD) x splits <= CUs per XCD
    xcds = xcds < 1 ? 1 : xcds;
    const int heads_per_xcd = (n_tiles + xcds - 1) / xcds;
    s = (cus / xcds) / heads_per_xcd;
    // at least four k tiles per split: with little to stream per split, the
    // finisher's partial reads cost more than the extra CUs save (measured at
    // hidden 1024: 9.2-10 us with four splits against 10.6-11.4 us with eight)
    if (s > nkt / 4) s = nkt / 4;
    if (s < min_splits) s = min_splits;
  }
  if (s < min_splits || s > nkt || s > kDecMaxNK) return 0;
  return s;
}

size_t decode_counter_bytes() { return size_t(kCounterBytes); }

size_t decode_workspace_bytes(int n_tiles, int splits, int blocks) {
  return size_t(kCounterBytes) + size_t(splits) * blocks * n_tiles * kTileFloats * sizeof(float);
}

int decode_max_blocks(int n_tiles, int64_t K, int splits) {
  if (splits < 1 || (K / kBK + splits - 1) / splits > kDecMultiMaxNK) return 1;
  const int by_counters = kMaxHeads / (n_tiles < 1 ? 1 : n_tiles);
  return by_counters < kDecMaxBlocks ? by_counters : kDecMaxBlocks;
}

hipError_t launch_decode(int int4, const ProblemArgs& p, const WeightArgs& w, const EpilogueArgs& e,
                         int splits, void* workspace, hipStream_t stream) {
  const int nkt = int(p.K / kBK);
  const int blocks = int((p.M + kDecRows - 1) / kDecRows);  // 64-row blocks of this launch
  // (p.xcds <= 8: the arrival counter's XCD sums hold x < 8)
  if (splits < 1 || splits > kDecMaxNK || splits > nkt || p.xcds > 8 ||
      (nkt + splits - 1) / splits > (blocks > 1 ? kDecMultiMaxNK : kDecLongMaxNK) ||
      p.n_tiles > kMaxHeads || blocks < 1 || blocks > decode_max_blocks(p.n_tiles, p.K, splits) || p.xcds < 1)
    return hipErrorInvalidValue;
  uint32_t* counters = static_cast<uint32_t*>(workspace);
  float* part = reinterpret_cast<float*>(static_cast<char*>(workspace) + kCounterBytes);
  const dim3 grid(((p.n_tiles + p.xcds - 1) / p.xcds) * p.xcds * splits);
  // ctl: bit 0 forces the recompute path, the rest is the final wait's poll limit
  const int fr = (g_decode_force_recompute ? 1 : 0) | (g_decode_max_spins << 1);
  auto a16 = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0; };
  if (e.qkv && !(a16(e.q_gamma) && a16(e.k_gamma) && a16(e.cos) && a16(e.sin))) return hipErrorInvalidValue;
  if (!e.qkv && (e.N % kHeadDim != 0 || !a16(e.out) || int64_t(p.n_tiles) * kHeadDim != e.N))
    return hipErrorInvalidValue;
  if (p.in_gamma || (p.half && (int4 || blocks > 1))) return hipErrorInvalidValue;  // (x normalised ahead; no such form)
  const int nkc = (nkt + splits - 1) / splits;  // longest k range of a split, in tiles
  const int mb = p.M <= 16 ? 1 : (p.M <= 32 ? 2 : 4);  // 16-row blocks a one-block launch works on
  DecKernel kernel = nullptr;
  if (blocks > 1) kernel = int4 ? decode_multi_kernel_w4(nkc) : decode_multi_kernel_bf16(nkc);
  else if ((mb == 4 || int4) && nkc > kDecMaxNK)
    kernel = int4 ? decode_long_kernel_w4(mb) : (p.half ? decode_long_kernel_f16() : decode_long_kernel_bf16());
  else kernel = int4 ? decode_kernel_w4(mb) : (p.half ? decode_kernel_f16(mb) : decode_kernel_bf16(mb));
  if (!kernel) return hipErrorInvalidValue;
  hipLaunchKernelGGL(kernel, grid, dim3(kDecThreads), 0, stream, p, w, e, splits, part, counters, fr);
  return hipGetLastError();
}

}  // namespace mqk
