// kernels_fmarch_f32_zener.hip -- the 3-D field march, FP32 Zener pinning.
#include "fmarch_launch.hpp"

namespace mmspx {

int launch_fmarch_f32_zener(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, const TuneChoice& t,
                        int nsteps)
{
	return launch_fmarch_prec<MMSPX_F32, 3>(g, p, a, b, st, t, nsteps);
}

}  // namespace mmspx
