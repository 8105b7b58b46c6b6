// The fused 1-D step under the reference kernels' AL rule (A8_AL_KERNEL_RULE) for
// 16-bit parameters (bf16, fp16).
#include "a8_update1d_kern.cuh"

namespace a8 {

int launch_any_kernel_rule_16bit(int dtype, int sr, int vbits, int mode, const Desc1D& one, const Desc1D* table,
                                 int ntab, int64_t nwg, const Hyper1D& h, hipStream_t st) {
  return launch_rule<1, false>(dtype, sr, vbits, mode, one, table, ntab, nwg, h, st);
}

hipError_t update1d_kh_upload_qmap(const float* q8, const float* q4) { return upload_qmap_tu(q8, q4); }

}  // namespace a8
