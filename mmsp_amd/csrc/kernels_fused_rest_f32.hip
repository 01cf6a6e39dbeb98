// kernels_fused_rest_f32.hip -- the tiled kernels of Ostwald ripening and multi-phase grain growth, the float forms.
#include "fused_launch.hpp"

namespace mmspx {

int launch_fused_rest_f32(MMSPX_FUSED_ARGS)
{
	return prec == MMSPX_F32 ? launch_fused_rest<MMSPX_F32>(g, p, a, b, st, t, nsteps, aux)
	                         : launch_fused_rest<MMSPX_F32REF>(g, p, a, b, st, t, nsteps, aux);
}

}  // namespace mmspx
