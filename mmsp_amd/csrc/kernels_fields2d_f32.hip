// kernels_fields2d_f32.hip -- the FP32 form of the 2-D four-step field strips.
#include "fields2d_launch.hpp"

namespace mmspx {

int launch_fields2d_f32(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk,
                        int nsteps)
{
	return launch_fields2d_prec<MMSPX_F32>(g, p, a, b, st, chunk, nsteps);
}

}  // namespace mmspx
