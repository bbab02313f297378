// Split-K decode kernels, int4 weights, one block of rows.
#include "qkv_decode.h"

namespace mqk {
namespace {

template <int MB>
__global__ void __launch_bounds__(kDecThreads, 1)
decode_kernel(ProblemArgs p, WeightArgs w, EpilogueArgs e, int splits, float* __restrict__ part,
              uint32_t* __restrict__ counters, int ctl) {
  decode_body<Bf16, true, MB>(p, w, e, splits, part, counters, ctl);
}

template <int MB>
__global__ void __launch_bounds__(kDecThreads, 1)
decode_long_kernel(ProblemArgs p, WeightArgs w, EpilogueArgs e, int splits, float* __restrict__ part,
                   uint32_t* __restrict__ counters, int ctl) {
  decode_long_body<Bf16, true, MB>(p, w, e, splits, part, counters, ctl);
}

}  // namespace

DecKernel decode_kernel_w4(int mb) { return mb == 1 ? decode_kernel<1> : (mb == 2 ? decode_kernel<2> : decode_kernel<4>); }
DecKernel decode_long_kernel_w4(int mb) {
  return mb == 1 ? decode_long_kernel<1> : (mb == 2 ? decode_long_kernel<2> : decode_long_kernel<4>);
}

}  // namespace mqk
