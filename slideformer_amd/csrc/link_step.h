// The update launch of the streaming pipeline's direct path: kernels that read
// and write page-locked host memory over the host link.
#ifndef SLIDEFORMER_AMD_LINK_STEP_H
#define SLIDEFORMER_AMD_LINK_STEP_H

#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/layer_adam.h"

namespace la_link {

// la_adamw_step's update on arrays of which any may be in page-locked host
// memory.  The caller has checked every array's placement and that the dtype
// triple is registered; the pointers' own alignment is checked here.
// `link_read`: bytes per element that the kernel reads from host memory.
__attribute__((visibility("hidden"))) int step(const la_scalars_t& sc, int p_dtype, void* p, int g_dtype,
                                               const void* g, int s_dtype, void* m, void* v, uint64_t n,
                                               uint16_t* p_bf16_out, const float* clip_coef, unsigned link_read,
                                               hipStream_t stream);

}  // namespace la_link

#endif  // SLIDEFORMER_AMD_LINK_STEP_H
