// kernels_fused_gg_f64.hip -- the tiled kernels of grain growth and Zener pinning, FP64 form.
#include "fused_launch.hpp"

namespace mmspx {

int launch_fused_gg_f64(MMSPX_FUSED_ARGS)
{
	(void)prec;
	return launch_fused_gg<MMSPX_F64>(g, p, a, b, st, t, nsteps, aux);
}

}  // namespace mmspx
