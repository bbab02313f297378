// Split-K decode kernels, fp16 tensors, one block of rows.
#include "qkv_decode.h"

namespace mqk {
namespace {

template <int MB>
__global__ void __launch_bounds__(kDecThreads, 1)
decode_f16_kernel(ProblemArgs p, WeightArgs w, EpilogueArgs e, int splits, float* __restrict__ part,
                  uint32_t* __restrict__ counters, int ctl) {
  decode_body<Fp16, false, MB>(p, w, e, splits, part, counters, ctl);
}

__global__ void __launch_bounds__(kDecThreads, 1)
decode_long_f16_kernel(ProblemArgs p, WeightArgs w, EpilogueArgs e, int splits, float* __restrict__ part,
                       uint32_t* __restrict__ counters, int ctl) {
  decode_long_body<Fp16, false, 4>(p, w, e, splits, part, counters, ctl);
}

}  // namespace

DecKernel decode_kernel_f16(int mb) { return mb == 1 ? decode_f16_kernel<1> : (mb == 2 ? decode_f16_kernel<2> : decode_f16_kernel<4>); }
DecKernel decode_long_kernel_f16() { return decode_long_f16_kernel; }

}  // namespace mqk
