// kernels_batch_steps.hip -- batched and served grids on the multi-step
// kernels: 2-D members by the multi-step wave strips (steps2d.hpp), one wave
// per item, 3-D members by the four-level march (march4.hpp), one workgroup
// per item. A pass takes the steps the single-grid kernels take, so a launch
// per step becomes one per 2 to 8 steps. Member tables are read once into
// scalar registers; items run in list order, dealt so that an XCD takes a
// contiguous run of them.
#include <type_traits>

#include "batch.hpp"
#include "march4.hpp"
#include "steps2d.hpp"

namespace mmspx {

__device__ __forceinline__ int dealt_block()
{
	return (gridDim.x & 7) == 0 ? (int)((blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3)) : (int)blockIdx.x;
}

// A member's buffer as global memory. (Picked by comparison: indexing the pair
// by a variable put the whole member record, 488 bytes a lane, into scratch
// memory, written by every wave, and made all accesses flat: a four-step pass
// over 32 Allen-Cahn grids of 112 to 621 squared in FP32 took 43.7 us, 17.4 this
// way; the march over a 125^3 FP32 Cahn-Hilliard grid among others 43.2, 20.7.)
template <typename S>
__device__ __forceinline__ S* member_buf(const BMember& m, int k)
{
	return (S*)(GlobalT<S>*)(uintptr_t)(k ? m.buf[1] : m.buf[0]);
}

template <int PREC, int MODEL, int L, bool EDGES, bool FULL>
__global__ void __launch_bounds__(256) steps2d_batch(const BMember* __restrict__ mem, const BItem* __restrict__ items,
                                                     int nitems, int parity, int levels)
{
	using S = typename Form<PREC>::S;
	const int it = __builtin_amdgcn_readfirstlane(dealt_block() * 4 + (int)(threadIdx.x >> 6));
	if (it >= nitems) return;  // a whole wave; the waves share nothing
	const BItem w = items[it];
	const BMember m = mem[w.m];
	const int src = (parity + m.phase) & 1;
	steps2d<PREC, MODEL, L, EDGES, 0, FULL>(member_buf<S>(m, src), member_buf<S>(m, src ^ 1), m.g, m.p, w.z0, w.xb, w.xe,
	                                            levels);
}

template <int PREC, int MODEL, int TY, int TZ, int NT, int LEVELS>
__global__ void __launch_bounds__(NT) march4_batch(const BMember* __restrict__ mem, const BItem* __restrict__ items,
                                                   int nitems, int parity)
{
	using S = typename Form<PREC>::S;
	const int it = dealt_block();
	if (it >= nitems) return;  // the whole workgroup
	const BItem w = items[it];
	const BMember m = mem[w.m];
	const int src = (parity + m.phase) & 1;
	march4<PREC, MODEL, TY, TZ, NT, LEVELS, 0>(member_buf<S>(m, src), member_buf<S>(m, src ^ 1), m.g, m.p, w.y0, w.z0, w.xb,
	                                               w.xe);
}

template <int PREC, int MODEL, int L, bool EDGES>
static void strips(const BMember* mem, const BItem* items, int n, int parity, hipStream_t st, int levels)
{
	const dim3 grid(((n + 3) / 4 + 7) / 8 * 8);
	if (levels == L)
		hipLaunchKernelGGL((steps2d_batch<PREC, MODEL, L, EDGES, true>), grid, dim3(256), 0, st, mem, items, n, parity,
		                   levels);
	else
		hipLaunchKernelGGL((steps2d_batch<PREC, MODEL, L, EDGES, false>), grid, dim3(256), 0, st, mem, items, n, parity,
		                   levels);
}

template <int PREC, int MODEL>
static void strips_of(const BatchTile& t, const BMember* mem, const BItem* items, int n, int parity, hipStream_t st,
                      int nsteps)
{
	const int levels = nsteps * (MODEL == S2_AC ? 1 : 2);
	// Cahn-Hilliard members are periodic
	if constexpr (MODEL == S2_AC) {
		if (t.edges)
			return t.lv == 8 ? strips<PREC, MODEL, 8, true>(mem, items, n, parity, st, levels)
			                 : strips<PREC, MODEL, 4, true>(mem, items, n, parity, st, levels);
	}
	return t.lv == 8 ? strips<PREC, MODEL, 8, false>(mem, items, n, parity, st, levels)
	                 : strips<PREC, MODEL, 4, false>(mem, items, n, parity, st, levels);
}

template <int PREC>
static int strips_prec(int model, const BatchTile& t, const BMember* mem, const BItem* items, int n, int parity,
                       hipStream_t st, int nsteps)
{
	switch (model) {
	case MMSPX_AC: strips_of<PREC, S2_AC>(t, mem, items, n, parity, st, nsteps); return 0;
	case MMSPX_CH: strips_of<PREC, S2_CH>(t, mem, items, n, parity, st, nsteps); return 0;
	case MMSPX_CH_DW: strips_of<PREC, S2_CH_DW>(t, mem, items, n, parity, st, nsteps); return 0;
	}
	return fail(MMSPX_EUNSUPPORTED, "the multi-step wave strips run Allen-Cahn and Cahn-Hilliard");
}

int launch_batch_steps2d(int model, int prec, const BatchTile& t, const BMember* mem, const BItem* items, int n,
                         int parity, hipStream_t st, int nsteps)
{
	if (prec == MMSPX_F64) return strips_prec<MMSPX_F64>(model, t, mem, items, n, parity, st, nsteps);
	if (prec == MMSPX_F32) return strips_prec<MMSPX_F32>(model, t, mem, items, n, parity, st, nsteps);
	return fail(MMSPX_EUNSUPPORTED, "the multi-step wave strips run the MMSPX_F64 and MMSPX_F32 forms");
}

template <int PREC, int MODEL, int TY, int TZ, int NT>
static void march_tile(const BMember* mem, const BItem* items, int n, int parity, hipStream_t st, int nsteps)
{
	const dim3 grid((n + 7) / 8 * 8);
	if (nsteps == 2)
		hipLaunchKernelGGL((march4_batch<PREC, MODEL, TY, TZ, NT, 4>), grid, dim3(NT), 0, st, mem, items, n, parity);
	else
		hipLaunchKernelGGL((march4_batch<PREC, MODEL, TY, TZ, NT, 2>), grid, dim3(NT), 0, st, mem, items, n, parity);
}

template <int PREC, int MODEL>
static int march_model(const BatchTile& t, const BMember* mem, const BItem* items, int n, int parity, hipStream_t st,
                       int nsteps)
{
	if (t.y3 == 26 && t.z3 == 52) return march_tile<PREC, MODEL, 26, 52, 512>(mem, items, n, parity, st, nsteps), 0;
	if (t.y3 == 32 && t.z3 == 32) return march_tile<PREC, MODEL, 32, 32, 384>(mem, items, n, parity, st, nsteps), 0;
	if (t.y3 == 16 && t.z3 == 32) return march_tile<PREC, MODEL, 16, 32, 256>(mem, items, n, parity, st, nsteps), 0;
	if (t.y3 == 16 && t.z3 == 16) return march_tile<PREC, MODEL, 16, 16, 128>(mem, items, n, parity, st, nsteps), 0;
	if constexpr (PREC == MMSPX_F64) {
		if (t.y3 == 16 && t.z3 == 64) return march_tile<PREC, MODEL, 16, 64, 448>(mem, items, n, parity, st, nsteps), 0;
	} else {
		if (t.y3 == 32 && t.z3 == 64) return march_tile<PREC, MODEL, 32, 64, 704>(mem, items, n, parity, st, nsteps), 0;
	}
	return fail(MMSPX_EINVAL, "no four-level march compiled for this tile");
}

int launch_batch_march4(int model, int prec, const BatchTile& t, const BMember* mem, const BItem* items, int n,
                        int parity, hipStream_t st, int nsteps)
{
	if (prec == MMSPX_F64)
		return model == MMSPX_CH_DW ? march_model<MMSPX_F64, S2_CH_DW>(t, mem, items, n, parity, st, nsteps)
		                            : march_model<MMSPX_F64, S2_CH>(t, mem, items, n, parity, st, nsteps);
	if (prec == MMSPX_F32)
		return model == MMSPX_CH_DW ? march_model<MMSPX_F32, S2_CH_DW>(t, mem, items, n, parity, st, nsteps)
		                            : march_model<MMSPX_F32, S2_CH>(t, mem, items, n, parity, st, nsteps);
	return fail(MMSPX_EUNSUPPORTED, "the four-level march runs the MMSPX_F64 and MMSPX_F32 forms");
}

}  // namespace mmspx
