// march4_launch.hpp -- launches of the 3-D four-level march (march4.hpp), one
// translation unit per precision.
#pragma once

#include <type_traits>

#include "wmarch4.hpp"

namespace mmspx {

// One workgroup per (tile, chunk), XCD-contiguous runs as the other marches.
template <int PREC, int MODEL, int TY, int TZ, int NT, int LEVELS, int UNIT>
__global__ void __launch_bounds__(NT) march4_k(const typename Form<PREC>::S* __restrict__ a,
                                               typename Form<PREC>::S* __restrict__ b, Geom g, ModelParams p,
                                               int chunk_len, int tiles_y, int tiles_z, int ntiles)
{
	int tile = blockIdx.x;
	if ((gridDim.x & 7) == 0) tile = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
	if (tile >= ntiles) return;
	const int tz = tile % tiles_z;
	const int t2 = tile / tiles_z;
	const int ty = t2 % tiles_y;
	const int xb = t2 / tiles_y * chunk_len;
	march4<PREC, MODEL, TY, TZ, NT, LEVELS, UNIT>(a, b, g, p, ty * TY, tz * TZ, xb, min(xb + chunk_len, g.n[0]));
}

template <int PREC, int MODEL, int TY, int TZ, int NT, int LEVELS, int UNIT>
static int launch_march4_body(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	using S = typename Form<PREC>::S;
	const int tiles_y = (g.n[1] + TY - 1) / TY;
	const int tiles_z = (g.n[2] + TZ - 1) / TZ;
	const int ntiles = tiles_y * tiles_z * ((g.n[0] + chunk - 1) / chunk);
	hipLaunchKernelGGL((march4_k<PREC, MODEL, TY, TZ, NT, LEVELS, UNIT>), dim3((ntiles + 7) / 8 * 8), dim3(NT), 0, st,
	                   (const S*)a, (S*)b, g, p, chunk, tiles_y, tiles_z, ntiles);
	MMSPX_HIP(hipGetLastError());
	return 0;
}

template <int PREC, int MODEL, int NW, int R, int LEVELS, int UNIT>
__global__ void __launch_bounds__(64 * NW) wmarch4_k(const typename Form<PREC>::S* __restrict__ a,
                                                     typename Form<PREC>::S* __restrict__ b, Geom g, ModelParams p,
                                                     int chunk_len, int tiles_y, int tiles_z, int ntiles)
{
	int tile = blockIdx.x;
	if ((gridDim.x & 7) == 0) tile = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
	if (tile >= ntiles) return;
	const int tz = tile % tiles_z;
	const int t2 = tile / tiles_z;
	const int ty = t2 % tiles_y;
	const int xb = t2 / tiles_y * chunk_len;
	wmarch4<PREC, MODEL, NW, R, LEVELS, UNIT>(a, b, g, p, ty * (NW * R - 6), tz * 56, xb, min(xb + chunk_len, g.n[0]));
}

template <int PREC, int MODEL, int NW, int R, int LEVELS, int UNIT>
static int launch_wmarch4_body(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	using S = typename Form<PREC>::S;
	constexpr int TY = NW * R - 6, TZ = 56;
	const int tiles_y = (g.n[1] + TY - 1) / TY;
	const int tiles_z = (g.n[2] + TZ - 1) / TZ;
	const int ntiles = tiles_y * tiles_z * ((g.n[0] + chunk - 1) / chunk);
	// a last pass of fewer steps multiplies by unit weights too
	hipLaunchKernelGGL((wmarch4_k<PREC, MODEL, NW, R, LEVELS, LEVELS == 4 ? UNIT : 0>), dim3((ntiles + 7) / 8 * 8),
	                   dim3(64 * NW), 0, st, (const S*)a, (S*)b, g, p, chunk, tiles_y, tiles_z, ntiles);
	MMSPX_HIP(hipGetLastError());
	return 0;
}

template <int PREC, int MODEL, int LEVELS, int UNIT>
static int launch_march4_tile(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st,
                              const TuneChoice& t)
{
	if (t.ty == 26 && t.tz == 52) return launch_march4_body<PREC, MODEL, 26, 52, 512, LEVELS, UNIT>(g, p, a, b, st, t.chunk);
	if (t.ty == 32 && t.tz == 32) return launch_march4_body<PREC, MODEL, 32, 32, 384, LEVELS, UNIT>(g, p, a, b, st, t.chunk);
	if (t.ty == 16 && t.tz == 32) return launch_march4_body<PREC, MODEL, 16, 32, 256, LEVELS, UNIT>(g, p, a, b, st, t.chunk);
	if (t.ty == 16 && t.tz == 16) return launch_march4_body<PREC, MODEL, 16, 16, 128, LEVELS, UNIT>(g, p, a, b, st, t.chunk);
	// a wave's lanes along axis 2
	if (t.ty == 26 && t.tz == 56) return launch_wmarch4_body<PREC, MODEL, 16, 2, LEVELS, UNIT>(g, p, a, b, st, t.chunk);
	if constexpr (PREC == MMSPX_F64) {
		if (t.ty == 42 && t.tz == 56) return launch_wmarch4_body<PREC, MODEL, 12, 4, LEVELS, UNIT>(g, p, a, b, st, t.chunk);
	} else {
		if (t.ty == 30 && t.tz == 56) return launch_wmarch4_body<PREC, MODEL, 12, 3, LEVELS, UNIT>(g, p, a, b, st, t.chunk);
	}
	// a wide tile: 16 x 64 in double (the registers of 32 x 64 do not fit), 32 x 64 in float
	if constexpr (PREC == MMSPX_F64) {
		if (t.ty == 16 && t.tz == 64) return launch_march4_body<PREC, MODEL, 16, 64, 448, LEVELS, UNIT>(g, p, a, b, st, t.chunk);
	} else {
		if (t.ty == 32 && t.tz == 64) return launch_march4_body<PREC, MODEL, 32, 64, 704, LEVELS, UNIT>(g, p, a, b, st, t.chunk);
	}
	return fail(MMSPX_EINVAL, "no four-level march compiled for this tile");
}

template <int PREC, int MODEL>
static int launch_march4_model(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st,
                               const TuneChoice& t, int nsteps)
{
	bool weights = true;
	for (int k = 0; k < 3; k++) weights = weights && g.w[k] == 1.0 && g.wf[k] == 1.0f;
	int unit = weights;
	if (MODEL == S2_CH) unit = weights && p.K == 1.0 && p.Kf == 1.0f;
	if (MODEL == S2_CH_DW) unit = weights && p.kappa == 1.0 && p.kappaf == 1.0f;
	if (MODEL != S2_CH_DW && unit && unit_coefficients(p)) unit = 2;
	const int levels = nsteps * (MODEL == S2_AC ? 1 : 2);
	// fewer than four levels: a last pass of fewer steps
	auto run = [&](auto lv) {
		constexpr int L = decltype(lv)::value;
		if constexpr (MODEL != S2_CH_DW) {
			if (unit == 2) return launch_march4_tile<PREC, MODEL, L, 2>(g, p, a, b, st, t);
		}
		return unit ? launch_march4_tile<PREC, MODEL, L, 1>(g, p, a, b, st, t)
		            : launch_march4_tile<PREC, MODEL, L, 0>(g, p, a, b, st, t);
	};
	if (levels == 4) return run(std::integral_constant<int, 4>{});
	if (levels == 2) return run(std::integral_constant<int, 2>{});
	if constexpr (MODEL == S2_AC) {
		if (levels == 1) return run(std::integral_constant<int, 1>{});
		if (levels == 3) return run(std::integral_constant<int, 3>{});
	}
	return fail(MMSPX_EINVAL, "more steps than a pass of the four-level march takes");
}

template <int PREC>
static int launch_march4_prec(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st,
                              const TuneChoice& t, int nsteps)
{
	switch (p.model) {
	case MMSPX_AC: return launch_march4_model<PREC, S2_AC>(g, p, a, b, st, t, nsteps);
	case MMSPX_CH: return launch_march4_model<PREC, S2_CH>(g, p, a, b, st, t, nsteps);
	case MMSPX_CH_DW: return launch_march4_model<PREC, S2_CH_DW>(g, p, a, b, st, t, nsteps);
	}
	return fail(MMSPX_EUNSUPPORTED, "the four-level march runs Allen-Cahn and Cahn-Hilliard");
}

}  // namespace mmspx
