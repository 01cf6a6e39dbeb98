// kernels_steps2d.hip -- launches of the 2-D multi-step wave strips
// (steps2d.hpp): Allen-Cahn and Cahn-Hilliard, tile bodies 13 (eight levels
// per pass) and 14 (four).
#include <algorithm>
#include <cmath>

#include "steps2d.hpp"

namespace mmspx {

// One wave per (strip, chunk) item, four waves per workgroup; items run
// strip-fastest and an XCD takes a contiguous run of them, so neighbouring
// strips of the same rows share their halo columns in one L2. The item is
// made wave-uniform so that the march's row bookkeeping runs on the scalar unit.
template <int PREC, int MODEL, int L, bool EDGES, int UNIT, bool FULL>
__global__ void __launch_bounds__(256) steps2d_k(const typename Form<PREC>::S* __restrict__ a,
                                                 typename Form<PREC>::S* __restrict__ b, Geom g, ModelParams p,
                                                 int chunk_len, int strips, int nitems, int levels)
{
	int tile = blockIdx.x;
	if ((gridDim.x & 7) == 0) tile = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
	const int item = __builtin_amdgcn_readfirstlane(tile * 4 + (int)(threadIdx.x >> 6));
	if (item >= nitems) return;  // a whole wave; the waves share nothing
	const int s = item % strips, chunk = item / strips;
	const int xb = chunk * chunk_len;
	steps2d<PREC, MODEL, L, EDGES, UNIT, FULL>(a, b, g, p, s * (64 - 2 * L), xb, min(xb + chunk_len, g.n[0]), levels);
}

template <int PREC, int MODEL, int L, bool EDGES, int UNIT, bool FULL>
static int launch_body(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk,
                       int levels)
{
	using S = typename Form<PREC>::S;
	const int strips = (g.n[1] + 63 - 2 * L) / (64 - 2 * L);
	const int nitems = strips * ((g.n[0] + chunk - 1) / chunk);
	const int blocks = ((nitems + 3) / 4 + 7) / 8 * 8;
	hipLaunchKernelGGL((steps2d_k<PREC, MODEL, L, EDGES, UNIT, FULL>), dim3(blocks), dim3(256), 0, st, (const S*)a, (S*)b,
	                   g, p, chunk, strips, nitems, levels);
	MMSPX_HIP(hipGetLastError());
	return 0;
}

template <int PREC, int MODEL, bool EDGES, int UNIT>
static int launch_unit(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk,
                       int levels)
{
	// whole passes: every level in straight-line code; a last pass of fewer
	// steps branches over the levels past its last one
	if (levels == 8) return launch_body<PREC, MODEL, 8, EDGES, UNIT, true>(g, p, a, b, st, chunk, levels);
	if (levels == 4) return launch_body<PREC, MODEL, 4, EDGES, UNIT, true>(g, p, a, b, st, chunk, levels);
	return launch_body<PREC, MODEL, 8, EDGES, 0, false>(g, p, a, b, st, chunk, levels);
}

template <int PREC, int MODEL>
static int launch_model(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk,
                        int levels)
{
	int unit = g.w[0] == 1.0 && g.w[1] == 1.0 && g.wf[0] == 1.0f && g.wf[1] == 1.0f;
	if (unit && (MODEL == S2_CH_DW ? p.kappa == 1.0 && p.kappaf == 1.0f : unit_coefficients(p))) unit = 2;
	bool edges = false;
	for (int k = 0; k < 2; k++) edges |= g.b0[k] != MMSPX_PERIODIC || g.b1[k] != MMSPX_PERIODIC;
	if (edges)
		return unit == 2 ? launch_unit<PREC, MODEL, true, 2>(g, p, a, b, st, chunk, levels)
		       : unit    ? launch_unit<PREC, MODEL, true, 1>(g, p, a, b, st, chunk, levels)
		                 : launch_unit<PREC, MODEL, true, 0>(g, p, a, b, st, chunk, levels);
	return unit == 2 ? launch_unit<PREC, MODEL, false, 2>(g, p, a, b, st, chunk, levels)
	       : unit    ? launch_unit<PREC, MODEL, false, 1>(g, p, a, b, st, chunk, levels)
	                 : launch_unit<PREC, MODEL, false, 0>(g, p, a, b, st, chunk, levels);
}

template <int PREC>
static int launch_prec(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk,
                       int levels)
{
	switch (p.model) {
	case MMSPX_AC: return launch_model<PREC, S2_AC>(g, p, a, b, st, chunk, levels);
	case MMSPX_CH: return launch_model<PREC, S2_CH>(g, p, a, b, st, chunk, levels);
	case MMSPX_CH_DW: return launch_model<PREC, S2_CH_DW>(g, p, a, b, st, chunk, levels);
	}
	return fail(MMSPX_EUNSUPPORTED, "the multi-step wave strips run Allen-Cahn and Cahn-Hilliard");
}

bool steps2d_supported(const Geom& g, int prec, int model)
{
	// the reference's float form is bound by its conversions: the one-step
	// strips and temporal blocks stay faster (1024^2 Cahn-Hilliard 5.7 us per
	// step against 5.9, Allen-Cahn 3.2 against 3.6)
	if (prec != MMSPX_F64 && prec != MMSPX_F32) return false;
	if (g.dim != 2 || (model != MMSPX_AC && model != MMSPX_CH && model != MMSPX_CH_DW)) return false;
	// a level's halo stands for the neighbouring nodes only where both sides wrap or neither does
	for (int k = 0; k < 2; k++)
		if ((g.b0[k] == MMSPX_PERIODIC) != (g.b1[k] == MMSPX_PERIODIC)) return false;
	return true;
}

int steps2d_max_steps(int model, int body) { return (body == 13 ? 8 : 4) / (model == MMSPX_AC ? 1 : 2); }

// Body and rows per wave by a cost model. A pass takes T0 (launch, first loads,
// last stores) plus a wave's time: its level-rows, L per row it writes and
// L(L-1) in the triangle it starts with, at `level` microseconds each for a
// wave alone on its SIMD (about 5.4 cycles an instruction), times what sharing
// a SIMD among n waves costs, 0.28 + share * n (their instructions fill each
// other's latencies, more so in float); moving the grid at 5 TB/s overlaps all
// but a quarter of the shorter of the two. Waves at a non-periodic edge take
// longer and set the time of a launch that fills the chip about once. Fitted
// to a sweep of 2 to 64 rows and both bodies on sides 128 to 4096: mostly
// within 10 % of the best measured. Against the one-step strips and temporal
// blocks it replaces (us per step, periodic, FP64): Allen-Cahn 512^2 1.46 ->
// 1.02, 4096^2 36.2 -> 14.6, double-well Cahn-Hilliard 256^2 3.20 -> 1.21,
// 1024^2 6.00 -> 2.83, 4096^2 43.5 -> 21.4; FP32 1024^2 2.18 -> 1.36 and 4.69
// -> 2.19; walls, FP64 407 x 756: Allen-Cahn 3.66 -> 1.69, Cahn-Hilliard
// 4.17 -> 2.83. It was faster at every size tried, 17 x 49 to 4096^2.
TuneChoice steps2d_choice_many(const Geom* const* g, int count, int prec, int model)
{
	constexpr double kT0 = 2.5, kSimds = 1024, kBytesPerUs = 5e6;
	const bool f64 = prec == MMSPX_F64;
	const double level = model == MMSPX_AC ? (f64 ? 0.054 : 0.040) : model == MMSPX_CH_DW ? (f64 ? 0.0375 : 0.033)
	                                                                                     : (f64 ? 0.044 : 0.034);
	const double share = model == MMSPX_AC ? (f64 ? 0.72 : 0.56) : model == MMSPX_CH_DW ? (f64 ? 0.64 : 0.47)
	                                                                                    : (f64 ? 0.68 : 0.50);
	bool edges = false;
	double nodes = 0.0;
	for (int m = 0; m < count; m++) {
		for (int k = 0; k < 2; k++) edges |= g[m]->b0[k] != MMSPX_PERIODIC;
		nodes += g[m]->nodes;
	}
	const double move = 2.0 * nodes * (f64 ? 8 : 4) / kBytesPerUs;
	TuneChoice out{2, 1, kSteps8Cols, 8, 13};
	double best = 1e300;
	for (int body = 13; body <= 14; body++) {
		const int L = body == 13 ? 8 : 4, cols = 64 - 2 * L;
		for (int c = 2; c <= 64; c += count > 1 && c >= 8 ? 4 : 1) {
			double waves = 0.0;
			for (int m = 0; m < count; m++)
				waves += (double)((g[m]->n[1] + cols - 1) / cols) * ((g[m]->n[0] + c - 1) / c);
			double n = waves / kSimds;
			n = n <= 4.0 ? std::ceil(n) : n + 0.5;
			const double wave = level * (edges ? 1.0 + 0.045 * L : 1.0) * L * (c + L - 1) * std::max(1.0, 0.28 + share * n);
			const double cost = (kT0 + std::max(wave, move) + 0.25 * std::min(wave, move)) / L;
			if (cost < best) {
				best = cost;
				out = TuneChoice{2, 1, cols, c, body};
			}
		}
	}
	return out;
}

bool steps2d_choice(const Geom& g, int prec, int model, TuneChoice* out)
{
	if (!steps2d_supported(g, prec, model)) return false;
	const Geom* one = &g;
	*out = steps2d_choice_many(&one, 1, prec, model);
	return true;
}

int launch_steps2d(const Geom& g, int prec, const ModelParams& p, const void* a, void* b, hipStream_t st, int body,
                   int chunk, int nsteps)
{
	if (!steps2d_supported(g, prec, p.model))
		return fail(MMSPX_EUNSUPPORTED, "the multi-step wave strips take 2-D Allen-Cahn and Cahn-Hilliard grids in "
		                                "the MMSPX_F64 and MMSPX_F32 forms, axes periodic on both sides or on neither");
	if (chunk < 1 || nsteps < 1 || nsteps > steps2d_max_steps(p.model, body))
		return fail(MMSPX_EINVAL, "more steps than a pass of the multi-step wave strips takes");
	const int levels = nsteps * (p.model == MMSPX_AC ? 1 : 2);
	switch (prec) {
	case MMSPX_F64: return launch_prec<MMSPX_F64>(g, p, a, b, st, chunk, levels);
	case MMSPX_F32: return launch_prec<MMSPX_F32>(g, p, a, b, st, chunk, levels);
	}
	return fail(MMSPX_EINVAL, "unknown precision");
}

}  // namespace mmspx
