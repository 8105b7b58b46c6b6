// The fused 1-D step for 16-bit parameters (bf16, fp16) under the default AL rule:
// these instantiations of a8_update1d_kern.cuh in a translation unit of their own,
// so that they compile in parallel with the 32- and 64-bit ones.
#include "a8_update1d_kern.cuh"

namespace a8 {

int launch_any_16bit(int dtype, int sr, int vbits, int mode, const Desc1D& one, const Desc1D* table,
                     int ntab, int64_t nwg, const Hyper1D& h, hipStream_t st) {
  return launch_rule<0, false>(dtype, sr, vbits, mode, one, table, ntab, nwg, h, st);
}

hipError_t update1d_h_upload_qmap(const float* q8, const float* q4) { return upload_qmap_tu(q8, q4); }

}  // namespace a8
