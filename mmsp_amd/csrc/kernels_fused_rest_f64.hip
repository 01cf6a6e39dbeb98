// kernels_fused_rest_f64.hip -- the tiled kernels of Ostwald ripening and multi-phase grain growth, FP64 form.
#include "fused_launch.hpp"

namespace mmspx {

int launch_fused_rest_f64(MMSPX_FUSED_ARGS)
{
	(void)prec;
	return launch_fused_rest<MMSPX_F64>(g, p, a, b, st, t, nsteps, aux);
}

}  // namespace mmspx
