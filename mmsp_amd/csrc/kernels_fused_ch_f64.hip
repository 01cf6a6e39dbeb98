// kernels_fused_ch_f64.hip -- the tiled kernels of Cahn-Hilliard and model B, FP64 form.
#include "fused_launch.hpp"

namespace mmspx {

int launch_fused_ch_f64(MMSPX_FUSED_ARGS)
{
	(void)prec;
	return launch_fused_ch<MMSPX_F64>(g, p, a, b, st, t, nsteps, aux);
}

}  // namespace mmspx
