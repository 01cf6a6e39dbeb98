// fused.hpp -- what the choice of the tiled kernels (kernels_fused.hip) and their
// launches (fused_launch.hpp) share.
#pragma once

#include "core.hpp"

namespace mmspx {

inline bool all_periodic(const Geom& g)
{
	for (int k = 0; k < g.dim; k++)
		if (g.b0[k] != MMSPX_PERIODIC || g.b1[k] != MMSPX_PERIODIC) return false;
	return true;
}

inline bool gg_q_compiled(int q) { return q == 2 || q == 4 || q == 8 || q == 16 || q == 32; }

// every axis periodic on both sides or on neither (the fused Cahn-Hilliard
// bodies map the non-periodic sides; an axis periodic on one side only takes
// the two-pass kernels)
inline bool axes_uniform(const Geom& g)
{
	for (int k = 0; k < g.dim; k++)
		if ((g.b0[k] == MMSPX_PERIODIC) != (g.b1[k] == MMSPX_PERIODIC)) return false;
	return true;
}

// the Cahn-Hilliard bodies that map non-periodic sides: the register queues
// (3-D and the 2-D row strips) and the 2-D wave strips
inline bool ch_body_maps_edges(const Geom& g, const TuneChoice& t)
{
	if (g.dim == 3) return t.opt == 1 || t.opt == 2 || t.opt == 3;
	return t.tz == kChWaveOut || t.opt == 1;
}

// field counts of the 3-D march for grain growth and Zener pinning
inline bool march_q_compiled(int q) { return q == 2 || q == 4 || q == 8; }

// The launches, a translation unit for each family of models and precision: the
// runtime loads a translation unit's kernels at the first use of one of them. All
// in one took 27 to 32 ms, also where a call needed one for its last step; now 1
// (Allen-Cahn), 3 (Cahn-Hilliard) and 8 ms (grain growth).
#define MMSPX_FUSED_ARGS                                                                                                  \
	const Geom &g, int prec, const ModelParams &p, const void *a, void *b, hipStream_t st, const TuneChoice &t, int nsteps, \
	    void *aux
int launch_fused_ac_f64(MMSPX_FUSED_ARGS);
int launch_fused_ac_f32(MMSPX_FUSED_ARGS);  // and the reference's float form, as the others
int launch_fused_ch_f64(MMSPX_FUSED_ARGS);
int launch_fused_ch_f32(MMSPX_FUSED_ARGS);
int launch_fused_gg_f64(MMSPX_FUSED_ARGS);
int launch_fused_gg_f32(MMSPX_FUSED_ARGS);
int launch_fused_rest_f64(MMSPX_FUSED_ARGS);
int launch_fused_rest_f32(MMSPX_FUSED_ARGS);

}  // namespace mmspx
