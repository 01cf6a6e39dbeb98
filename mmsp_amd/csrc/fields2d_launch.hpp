// fields2d_launch.hpp -- launches of the 2-D four-step field strips
// (fields2d.hpp), one translation unit per precision.
#pragma once

#include "fields2d.hpp"

namespace mmspx {

// One workgroup of W waves per (strip, chunk) item, strip-fastest, an XCD
// taking a contiguous run of items (neighbouring strips share halo columns in
// its L2).
template <int PREC, int Q, int KIND, int W, bool UNIT, bool FULL>
__global__ void __launch_bounds__(64 * W, PREC == MMSPX_F32 ? 5 : 1) fields2d_k(const typename Form<PREC>::S* __restrict__ a,
                                                     typename Form<PREC>::S* __restrict__ b, Geom g, ModelParams p,
                                                     int chunk_len, int strips, int nitems, int steps)
{
	int item = blockIdx.x;
	if ((gridDim.x & 7) == 0) item = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
	if (item >= nitems) return;
	const int s = item % strips;
	const int xb = item / strips * chunk_len;
	fields2d<PREC, Q, KIND, W, UNIT, FULL>(a, b, g, p, s * kSteps4Cols, xb, min(xb + chunk_len, g.n[0]), steps);
}

template <int PREC, int Q, int KIND, int W>
static int launch_fields2d_body(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk,
                                int nsteps)
{
	using S = typename Form<PREC>::S;
	const int strips = (g.n[1] + kSteps4Cols - 1) / kSteps4Cols;
	const int nitems = strips * ((g.n[0] + chunk - 1) / chunk);
	const dim3 grid((nitems + 7) / 8 * 8), block(64 * W);
	// whole passes: every level in straight-line code; a last pass of fewer
	// steps branches over the levels past its last one
	if (nsteps < kFieldsSteps)
		hipLaunchKernelGGL((fields2d_k<PREC, Q, KIND, W, false, false>), grid, block, 0, st, (const S*)a, (S*)b, g, p, chunk,
		                   strips, nitems, nsteps);
	else if (g.w[0] == 1.0 && g.w[1] == 1.0 && g.wf[0] == 1.0f && g.wf[1] == 1.0f)
		hipLaunchKernelGGL((fields2d_k<PREC, Q, KIND, W, true, true>), grid, block, 0, st, (const S*)a, (S*)b, g, p, chunk, strips,
		                   nitems, nsteps);
	else
		hipLaunchKernelGGL((fields2d_k<PREC, Q, KIND, W, false, true>), grid, block, 0, st, (const S*)a, (S*)b, g, p, chunk, strips,
		                   nitems, nsteps);
	MMSPX_HIP(hipGetLastError());
	return 0;
}

template <int PREC, int KIND>
static int launch_fields2d_kind(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk,
                                int nsteps)
{
	switch (g.fields) {
	case 2: return launch_fields2d_body<PREC, 2, KIND, 1>(g, p, a, b, st, chunk, nsteps);
	case 4: return launch_fields2d_body<PREC, 4, KIND, 1>(g, p, a, b, st, chunk, nsteps);
	case 8: return launch_fields2d_body<PREC, 8, KIND, 4>(g, p, a, b, st, chunk, nsteps);
	case 16: return launch_fields2d_body<PREC, 16, KIND, 8>(g, p, a, b, st, chunk, nsteps);
	case 32:
		if constexpr (PREC == MMSPX_F32 || KIND == 1)
			return launch_fields2d_body<PREC, 32, KIND, 16>(g, p, a, b, st, chunk, nsteps);
	}
	return fail(MMSPX_EUNSUPPORTED, "the four-step field strips take 2, 4, 8, 16 or 32 fields");
}

template <int PREC>
static int launch_fields2d_prec(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk,
                                int nsteps)
{
	return p.model == MMSPX_ZENER ? launch_fields2d_kind<PREC, 3>(g, p, a, b, st, chunk, nsteps)
	                              : launch_fields2d_kind<PREC, 1>(g, p, a, b, st, chunk, nsteps);
}

}  // namespace mmspx
