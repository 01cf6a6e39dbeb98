// fmarch_launch.hpp -- launches of the 3-D field march (fmarch.hpp), one
// translation unit per precision.
#pragma once

#include "fmarch.hpp"

namespace mmspx {

// One workgroup per (tile, chunk), XCD-contiguous runs as the other marches.
template <int PREC, int Q, int KIND, int R, int L, int LEVELS, bool UNIT>
__global__ void __launch_bounds__(1024) fmarch_k(const typename Form<PREC>::S* __restrict__ a,
                                                 typename Form<PREC>::S* __restrict__ b, Geom g, ModelParams p,
                                                 int chunk_len, int tiles_y, int tiles_z, int ntiles)
{
	constexpr int TY = 16 / Q * R - 2 * (L - 1), TZ = 64 - 2 * L;
	int tile = blockIdx.x;
	if ((gridDim.x & 7) == 0) tile = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
	if (tile >= ntiles) return;
	const int tz = tile % tiles_z;
	const int t2 = tile / tiles_z;
	const int ty = t2 % tiles_y;
	const int xb = t2 / tiles_y * chunk_len;
	fmarch<PREC, Q, KIND, R, L, LEVELS, UNIT>(a, b, g, p, ty * TY, tz * TZ, xb, min(xb + chunk_len, g.n[0]));
}

template <int PREC, int Q, int KIND, int R, int L, int LEVELS, bool UNIT>
static int launch_fmarch_body(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	using S = typename Form<PREC>::S;
	constexpr int TY = 16 / Q * R - 2 * (L - 1), TZ = 64 - 2 * L;
	const int tiles_y = (g.n[1] + TY - 1) / TY;
	const int tiles_z = (g.n[2] + TZ - 1) / TZ;
	const int ntiles = tiles_y * tiles_z * ((g.n[0] + chunk - 1) / chunk);
	hipLaunchKernelGGL((fmarch_k<PREC, Q, KIND, R, L, LEVELS, UNIT>), dim3((ntiles + 7) / 8 * 8), dim3(1024), 0, st,
	                   (const S*)a, (S*)b, g, p, chunk, tiles_y, tiles_z, ntiles);
	MMSPX_HIP(hipGetLastError());
	return 0;
}

// whole passes, and a last one of fewer steps (which multiplies by unit weights
// too); OWN: the number of those that has a tile of its own
template <int PREC, int Q, int R, int L, int KIND, int OWN = 0>
static int launch_fmarch_steps(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk,
                               int nsteps)
{
	if (nsteps == L) {
		bool unit = true;
		for (int k = 0; k < 3; k++) unit = unit && g.w[k] == 1.0 && g.wf[k] == 1.0f;
		return unit ? launch_fmarch_body<PREC, Q, KIND, R, L, L, true>(g, p, a, b, st, chunk)
		            : launch_fmarch_body<PREC, Q, KIND, R, L, L, false>(g, p, a, b, st, chunk);
	}
	if (nsteps == 1) return launch_fmarch_body<PREC, Q, KIND, R, L, 1, false>(g, p, a, b, st, chunk);
	if constexpr (L > 2 && OWN != 2) {
		if (nsteps == 2) return launch_fmarch_body<PREC, Q, KIND, R, L, 2, false>(g, p, a, b, st, chunk);
	}
	if constexpr (L > 3 && OWN != 3) {
		if (nsteps == 3) return launch_fmarch_body<PREC, Q, KIND, R, L, 3, false>(g, p, a, b, st, chunk);
	}
	return fail(MMSPX_EINVAL, "more steps than a pass of the field march takes");
}

template <int PREC, int KIND>
static int launch_fmarch_prec(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st,
                              const TuneChoice& t, int nsteps)
{
	// rows per wave R and steps per pass L; the tile is 16/Q*R - 2(L-1) x 64 - 2L
	auto is = [&](int q, int r, int l) {
		return g.fields == q && t.ty == 16 / q * r - 2 * (l - 1) && t.tz == 64 - 2 * l;
	};
	if constexpr (PREC == MMSPX_F32) {
		if (is(8, 8, 3)) return launch_fmarch_steps<PREC, 8, 8, 3, KIND, 2>(g, p, a, b, st, t.chunk, nsteps);
		if (is(8, 12, 2)) return launch_fmarch_steps<PREC, 8, 12, 2, KIND>(g, p, a, b, st, t.chunk, nsteps);
		if (is(4, 6, 4)) return launch_fmarch_steps<PREC, 4, 6, 4, KIND, 3>(g, p, a, b, st, t.chunk, nsteps);
		if (is(4, 8, 3)) return launch_fmarch_steps<PREC, 4, 8, 3, KIND>(g, p, a, b, st, t.chunk, nsteps);
		if (is(2, 4, 4)) return launch_fmarch_steps<PREC, 2, 4, 4, KIND>(g, p, a, b, st, t.chunk, nsteps);
	} else {
		if (is(8, 5, 2)) return launch_fmarch_steps<PREC, 8, 5, 2, KIND>(g, p, a, b, st, t.chunk, nsteps);
		if (is(8, 6, 2)) return launch_fmarch_steps<PREC, 8, 6, 2, KIND>(g, p, a, b, st, t.chunk, nsteps);
		if (is(4, 6, 2)) return launch_fmarch_steps<PREC, 4, 6, 2, KIND>(g, p, a, b, st, t.chunk, nsteps);
		if (is(4, 4, 3)) return launch_fmarch_steps<PREC, 4, 4, 3, KIND, 2>(g, p, a, b, st, t.chunk, nsteps);
		if (is(2, 3, 4)) return launch_fmarch_steps<PREC, 2, 3, 4, KIND, 3>(g, p, a, b, st, t.chunk, nsteps);
		if (is(2, 4, 3)) return launch_fmarch_steps<PREC, 2, 4, 3, KIND>(g, p, a, b, st, t.chunk, nsteps);
	}
	return fail(MMSPX_EINVAL, "no field march compiled for this tile and field count");
}

}  // namespace mmspx
