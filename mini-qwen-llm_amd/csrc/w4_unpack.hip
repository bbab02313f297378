// int4 projection weights -> the bf16 nn.Linear layout, for calls that reuse them
// over many token rows.
//
// The int4 tile kernel dequantises a weight once per row tile it multiplies, on the
// vector units, inside the stage loop that feeds the matrix cores: its stage costs
// ~1.9 us (256 x 256 tiles) however few tiles run, against ~1.4 us of the bf16 loop.
// With enough rows it is cheaper to dequantise every weight once, into the
// workspace, and run the bf16 plan on it.  The value is the one the tile kernels
// multiply, (q - z) * s exact in fp32 and rounded once to bf16 (dequant_int4x8), and
// the sums run in the same order.  Measured on MI355X, whole call (hidden 4096, 32 / 8
// heads): T = 1536 135 -> 104 us, T = 4096 267 -> 201 us, T = 8214 423 -> 366 us; this kernel
// takes 13.4 us of that, for 12.6 MB of reads and 50 MB of writes (4.7 TB/s; a copy
// reaches 5.1).
//
// A workgroup turns 64 columns x 64 packed words (512 k): words come in along the
// columns (256-byte runs), go through LDS (pitch 65: no bank conflicts either way)
// and leave along k, 1 KB of one weight row per wave store.
#include "mqk_device.h"
#include "mqk_kernels.h"

namespace mqk {
namespace {

constexpr int kCols = 64;    // columns of a workgroup
constexpr int kWords = 64;   // packed words (8 k each) of a workgroup
constexpr int kMaxGroups = kWords * 8 / 64 + 1;  // quantisation groups (multiples of 64 k) it can touch

__global__ void __launch_bounds__(256)
w4_unpack_kernel(WeightArgs w, int64_t K, uint16_t* __restrict__ out) {
  __shared__ uint32_t words[kWords][kCols + 1];
  __shared__ float scale[kMaxGroups][kCols], zero[kMaxGroups][kCols];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t row0 = int64_t(blockIdx.x) * kCols;  // first row of `out` (column of the three projections)
  int proj = 0;
  int64_t c0 = row0;
  if (c0 >= w.n_cols[0]) {
    c0 -= w.n_cols[0];
    proj = 1;
    if (c0 >= w.n_cols[1]) {
      c0 -= w.n_cols[1];
      proj = 2;
    }
  }
  const int64_t N = proj == 0 ? w.n_cols[0] : (proj == 1 ? w.n_cols[1] : w.n_cols[2]);
  const int32_t* qw = pick3_uniform<const int32_t>(proj, w.qw[0], w.qw[1], w.qw[2]);
  const int32_t* qz = pick3_uniform<const int32_t>(proj, w.qz[0], w.qz[1], w.qz[2]);
  const uint16_t* sc = pick3_uniform<const uint16_t>(proj, static_cast<const uint16_t*>(w.sc[0]),
                                             static_cast<const uint16_t*>(w.sc[1]), static_cast<const uint16_t*>(w.sc[2]));
  const int64_t j0 = int64_t(blockIdx.y) * kWords;
  const int nj = int(K / 8 - j0 < kWords ? K / 8 - j0 : kWords);
  const int64_t g0 = j0 * 8 / w.group;
  const int ng = int(((j0 + nj) * 8 - 1) / w.group - g0) + 1;
  uint32_t r[kWords / 4];  // all of this thread's words in flight at once
#pragma unroll
  for (int i = 0; i < kWords / 4; ++i) {
    const int j = wave + 4 * i;
    r[i] = j < nj ? uint32_t(load_global(qw + (j0 + j) * N + c0 + lane)) : 0u;
  }
#pragma unroll
  for (int i = 0; i < kWords / 4; ++i) words[wave + 4 * i][lane] = r[i];
  for (int g = wave; g < ng; g += 4) {
    const int64_t col = c0 + lane;
    const uint32_t sraw = load_global(sc + (g0 + g) * N + col);
    const uint32_t zw = uint32_t(load_global(qz + (g0 + g) * (N / 8) + col / 8));
    scale[g][lane] = w.scale_fp16 ? f16_to_f32(sraw) : bf16_to_f32(sraw);
    zero[g][lane] = float((zw >> ((col % 8) * 4)) & 0xFu);
  }
  __syncthreads();
  if (lane >= nj) return;
  const int g = int((j0 + lane) * 8 / w.group - g0);
  u32x4_t* dst = reinterpret_cast<u32x4_t*>(out + row0 * K) + j0 + lane;
#pragma unroll 4
  for (int n = wave * (kCols / 4); n < (wave + 1) * (kCols / 4); ++n)
    dst[int64_t(n) * (K / 8)] = dequant_int4x8(words[lane][n], zero[g][n], scale[g][n]);
}

}  // namespace

hipError_t launch_w4_unpack(const WeightArgs& w, int n_tiles, int64_t K, uint16_t* out, hipStream_t stream) {
  const int64_t blocks = (K / 8 + kWords - 1) / kWords;
  if (n_tiles < 1 || K < 64 || K % 64 != 0 || blocks > 65535 || w.group < 64 || w.group % 64 != 0 ||
      w.n_cols[0] + w.n_cols[1] + w.n_cols[2] != int64_t(n_tiles) * kHeadDim || w.n_cols[0] % kHeadDim != 0 ||
      w.n_cols[1] % kHeadDim != 0)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(w4_unpack_kernel, dim3(unsigned(n_tiles * (kHeadDim / kCols)), unsigned(blocks)), dim3(256), 0,
                     stream, w, K, out);
  return hipGetLastError();
}

}  // namespace mqk
