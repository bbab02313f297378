// Pre-pass of the fused input RMSNorm: the per-token scale
// rsqrt(mean(x^2) + eps) of the decoder's input_layernorm
// (mini_qwen/model/layers/rms_norm.py:15-17), and the rows it normalises.
//
// Where the workspace has room (the sizes its query gives), the pre-pass writes
// the normalised rows bf16(gamma * bf16(x * scale)) there and the projection
// reads them as its x.  A row is read once and written once, while a projection
// kernel that normalises what it stages does so once per column tile, in the
// critical path of every stage: measured on MI355X (hidden 4096, 32 / 8 heads,
// one call, without -> with the rows written ahead) T = 24 25.3 -> 22.4 us, T = 777
// 71.8 -> 58.8 us, T = 4096 220 -> 194 us; int4 weights T = 777 238 -> 81 us, T = 4096
// 356 -> 280 us (the plain call: 18.2 / 52.1 / 180 and 75 / 267 us; T = 24 has since
// become 20.3 us with the decode kernel's 32-row blocks).  A workspace without room for
// the rows (or more than kNormAheadMaxBytes of them) gets the scales only, and the tile
// kernels apply them as they stage their x tiles (input_norm8): the same bits from the
// same tiles.
//
// One wave per token row, bound by latency at decode sizes and by the copy at large
// T: 16-byte loads, up to 4096 or 8192 of a row's elements and their gammas in flight
// and held (HELD = 8 or 16 chunks per lane; longer rows are read again for the second
// pass, from the L2), fp32 sum of squares, 64-lane butterfly.  Rows get a workgroup each
// until there are enough of them to fill the CUs with four per workgroup.
#include "mqk_device.h"
#include "mqk_kernels.h"

namespace mqk {
namespace {

// out null: the scale only; else the normalised row (gamma then non-null).
template <int HELD>  // 16-byte chunks per lane held in registers
__global__ void __launch_bounds__(256)
row_scale_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ gamma, int64_t M, int64_t K, float eps,
                 float* __restrict__ scale, uint16_t* __restrict__ out) {
  const int64_t row = int64_t(blockIdx.x) * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (row >= M) return;
  const int lane = threadIdx.x & 63;
  const u32x4_t* src = reinterpret_cast<const u32x4_t*>(x + row * K);
  const int chunks = int(K / 8);
  constexpr int kStep = 64 * HELD;  // chunks per pass over a row
  u32x4_t v[HELD], g[HELD];
  auto load = [&](const u32x4_t* from, int c0, u32x4_t (&to)[HELD]) {
#pragma unroll
    for (int i = 0; i < HELD; ++i) {
      const int c = c0 + i * 64 + lane;
      to[i] = c < chunks ? from[c] : u32x4_t{0, 0, 0, 0};
    }
  };
  const u32x4_t* gsrc = reinterpret_cast<const u32x4_t*>(gamma);
  float ss = 0.f;
  for (int c0 = 0; c0 < chunks; c0 += kStep) {
    load(src, c0, v);
    if (out && c0 == 0) load(gsrc, 0, g);  // (under the sum and the butterfly)
#pragma unroll
    for (int i = 0; i < HELD; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float a = bf16_to_f32(v[i][j] & 0xFFFFu), b = bf16_to_f32(v[i][j] >> 16);
        ss += a * a + b * b;
      }
  }
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) ss += __shfl_xor(ss, m);
  const float sc = rsqrtf(ss / float(K) + eps);
  if (!out) {
    if (lane == 0) scale[row] = sc;
    return;
  }
  u32x4_t* dst = reinterpret_cast<u32x4_t*>(out + row * K);
  for (int c0 = 0; c0 < chunks; c0 += kStep) {
    if (chunks > kStep) {
      load(src, c0, v);
      if (c0 > 0) load(gsrc, c0, g);
    }
#pragma unroll
    for (int i = 0; i < HELD; ++i) {
      const int c = c0 + i * 64 + lane;
      if (c < chunks) dst[c] = input_norm8(v[i], sc, g[i]);
    }
  }
}

}  // namespace

hipError_t launch_row_scale(const uint16_t* x, const uint16_t* gamma, int64_t M, int64_t K, float eps, float* scale,
                            uint16_t* out, hipStream_t stream) {
  if (M <= 0) return hipSuccess;
  const int rows = M > 1024 ? 4 : 1;  // rows (waves) per workgroup
  const dim3 grid(unsigned((M + rows - 1) / rows)), block(unsigned(rows * 64));
  if (K <= 4096)
    hipLaunchKernelGGL(row_scale_kernel<8>, grid, block, 0, stream, x, gamma, M, K, eps, scale, out);
  else
    hipLaunchKernelGGL(row_scale_kernel<16>, grid, block, 0, stream, x, gamma, M, K, eps, scale, out);
  return hipGetLastError();
}

}  // namespace mqk
