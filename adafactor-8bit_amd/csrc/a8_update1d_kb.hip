// The fused 1-D step for bf16 parameters under the reference kernels' AL rule (A8_AL_KERNEL_RULE): these instantiations of
// a8_update1d_kern.cuh in a translation unit of their own, so that they compile in
// parallel with the others.
#include "a8_update1d_kern.cuh"

namespace a8 {

A8_UNIT(launch_1d_kb) { return launch_rule<1, 1>(dtype, sr, vbits, mode, one, table, ntab, nwg, h, st); }

hipError_t update1d_kb_upload_qmap(const float* q8, const float* q4) { return upload_qmap_tu(q8, q4); }

}  // namespace a8
