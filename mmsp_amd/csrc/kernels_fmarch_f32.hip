// kernels_fmarch_f32.hip -- the 3-D field march, FP32 grain growth.
#include "fmarch_launch.hpp"

namespace mmspx {

int launch_fmarch_f32_gg(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, const TuneChoice& t,
                        int nsteps)
{
	return launch_fmarch_prec<MMSPX_F32, 1>(g, p, a, b, st, t, nsteps);
}

}  // namespace mmspx
