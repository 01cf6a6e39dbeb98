// kernels_gga2d.hip -- launches of the 2-D multi-phase grain growth strips (gga2d.hpp).
#include "gga2d.hpp"

namespace mmspx {

// One wave per (strip, chunk) item, four waves per workgroup, strip-fastest; an
// XCD takes a contiguous run of items (neighbouring strips share halo columns
// in its L2). The item is wave-uniform, so rows are the scalar unit's.
template <int PREC, int Q, bool UNIT>
__global__ void __launch_bounds__(256, 4) gga2d_k(const typename Form<PREC>::S* __restrict__ a,
                                               typename Form<PREC>::S* __restrict__ b, Geom g, ModelParams p,
                                               int chunk_len, int strips, int nitems)
{
	__shared__ typename Form<PREC>::S slots[Q > 4 ? 8 * 256 : 1];
	int tile = blockIdx.x;
	if ((gridDim.x & 7) == 0) tile = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
	const int item = __builtin_amdgcn_readfirstlane(tile * 4 + (int)(threadIdx.x >> 6));
	if (item >= nitems) return;  // a whole wave; the waves share nothing
	const int s = item % strips, chunk = item / strips;
	const int xb = chunk * chunk_len;
	gga2d<PREC, Q, UNIT>(a, b, g, p, s * kGgaCols, xb, min(xb + chunk_len, g.n[0]), slots + (Q > 4 ? threadIdx.x : 0));
}

template <int PREC, int Q>
static int launch_gga2d_q(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	using S = typename Form<PREC>::S;
	const int strips = (g.n[1] + kGgaCols - 1) / kGgaCols;
	const int nitems = strips * ((g.n[0] + chunk - 1) / chunk);
	const dim3 grid(((nitems + 3) / 4 + 7) / 8 * 8), block(256);
	if (g.w[0] == 1.0 && g.w[1] == 1.0 && g.wf[0] == 1.0f && g.wf[1] == 1.0f)
		hipLaunchKernelGGL((gga2d_k<PREC, Q, true>), grid, block, 0, st, (const S*)a, (S*)b, g, p, chunk, strips, nitems);
	else
		hipLaunchKernelGGL((gga2d_k<PREC, Q, false>), grid, block, 0, st, (const S*)a, (S*)b, g, p, chunk, strips, nitems);
	MMSPX_HIP(hipGetLastError());
	return 0;
}

template <int PREC>
static int launch_gga2d_prec(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	switch (g.fields) {
	case 2: return launch_gga2d_q<PREC, 2>(g, p, a, b, st, chunk);
	case 4: return launch_gga2d_q<PREC, 4>(g, p, a, b, st, chunk);
	case 8: return launch_gga2d_q<PREC, 8>(g, p, a, b, st, chunk);
	}
	return fail(MMSPX_EUNSUPPORTED, "multi-phase wave strips take 2, 4 or 8 fields in the MMSPX_F64 and MMSPX_F32 forms");
}

int launch_gga2d(const Geom& g, int prec, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	if (prec == MMSPX_F64) return launch_gga2d_prec<MMSPX_F64>(g, p, a, b, st, chunk);
	if (prec == MMSPX_F32) return launch_gga2d_prec<MMSPX_F32>(g, p, a, b, st, chunk);
	return fail(MMSPX_EUNSUPPORTED, "multi-phase wave strips take 2, 4 or 8 fields in the MMSPX_F64 and MMSPX_F32 forms");
}

}  // namespace mmspx
