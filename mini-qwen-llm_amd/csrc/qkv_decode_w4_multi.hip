// Split-K decode kernels, int4 weights, several 64-row blocks.
#include "qkv_decode.h"

namespace mqk {
namespace {

template <int NKC>
__global__ void __launch_bounds__(kDecThreads, 1)
decode_multi_kernel(ProblemArgs p, WeightArgs w, EpilogueArgs e, int splits, float* __restrict__ part,
                    uint32_t* __restrict__ counters, int ctl) {
  decode_multi_body<true, NKC>(p, w, e, splits, part, counters, ctl);
}

}  // namespace

DecKernel decode_multi_kernel_w4(int nk) {
  // (the kernel of NKC tiles also runs splits of NKC - 1: one tile takes the one of two)
  static const DecKernel k[kDecMultiMaxNK + 1] = {
      nullptr,
      decode_multi_kernel<2>, decode_multi_kernel<2>, decode_multi_kernel<3>,  decode_multi_kernel<4>,
      decode_multi_kernel<5>, decode_multi_kernel<6>, decode_multi_kernel<7>,  decode_multi_kernel<8>,
      decode_multi_kernel<9>, decode_multi_kernel<10>, decode_multi_kernel<11>, decode_multi_kernel<12>,
      decode_multi_kernel<13>};
  return nk >= 1 && nk <= kDecMultiMaxNK ? k[nk] : nullptr;
}

}  // namespace mqk
