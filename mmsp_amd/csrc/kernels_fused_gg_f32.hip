// kernels_fused_gg_f32.hip -- the tiled kernels of grain growth and Zener pinning, the float forms.
#include "fused_launch.hpp"

namespace mmspx {

int launch_fused_gg_f32(MMSPX_FUSED_ARGS)
{
	return prec == MMSPX_F32 ? launch_fused_gg<MMSPX_F32>(g, p, a, b, st, t, nsteps, aux)
	                         : launch_fused_gg<MMSPX_F32REF>(g, p, a, b, st, t, nsteps, aux);
}

}  // namespace mmspx
