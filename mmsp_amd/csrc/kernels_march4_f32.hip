// kernels_march4_f32.hip -- the FP32 form of the 3-D four-level march.
#include "march4_launch.hpp"

namespace mmspx {

int launch_march4_f32(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, const TuneChoice& t,
                      int nsteps)
{
	return launch_march4_prec<MMSPX_F32>(g, p, a, b, st, t, nsteps);
}

}  // namespace mmspx
