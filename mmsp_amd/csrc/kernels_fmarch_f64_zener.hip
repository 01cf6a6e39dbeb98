// kernels_fmarch_f64_zener.hip -- the 3-D field march, FP64 Zener pinning.
#include "fmarch_launch.hpp"

namespace mmspx {

int launch_fmarch_f64_zener(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, const TuneChoice& t,
                        int nsteps)
{
	return launch_fmarch_prec<MMSPX_F64, 3>(g, p, a, b, st, t, nsteps);
}

}  // namespace mmspx
