// fused_launch.hpp -- tiled kernels for single grids: fused single-pass
// Cahn-Hilliard (2-D/3-D, periodic) and marching-strip Allen-Cahn and grain
// growth (2-D, any boundary condition). Tile bodies live in tiles.hpp.
//
// Cahn-Hilliard: the reference takes two full sweeps per step
// (cahn-hilliard.cpp:69-76): mu into a temporary grid, then c + dt*M*lap(mu).
// Unfused, that moves 40 bytes per FP64 cell-update through HBM (c in, mu out,
// mu in, c in, c' out); the fused tile moves the compulsory 16 (c in, c' out)
// and recomputes mu on a one-cell halo from the same wrapped values, so the
// result is bitwise that of the two-pass form. Only periodic boundaries take
// it; other boundaries keep the two-pass kernels, where mu at a mapped
// neighbour is mu of the mapped node exactly as in the reference.
//
// Workgroup ids are remapped so that the workgroups one XCD receives (ids are
// dealt round-robin over the 8 XCDs) form a contiguous run of tiles with the
// axis-0 chunk slowest: an XCD sweeps whole planes of one chunk, so halo reads
// of neighbouring tiles hit its own L2.
#pragma once

#include <algorithm>

#include "fused.hpp"
#include "tiles.hpp"

namespace mmspx {

__device__ __forceinline__ int xcd_tile(int ntiles)
{
	int tile = blockIdx.x;
	if ((gridDim.x & 7) == 0) tile = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
	return tile < ntiles ? tile : -1;
}

// BODY 0: LDS rings, 1: register queues; MU as mu_of (0 polynomial, 1 double
// well, 2 polynomial plus noise)
template <int PREC, int MU, int DIM, int TY, int TZ, int NT, int BODY>
__global__ void __launch_bounds__(NT) ch_fused(const typename Form<PREC>::S* __restrict__ a,
                                               typename Form<PREC>::S* __restrict__ b, Geom g, ModelParams p,
                                               int chunk_len, int tiles_y, int tiles_z, int ntiles)
{
	const int tile = xcd_tile(ntiles);
	if (tile < 0) return;
	const int tz = tile % tiles_z;
	const int t2 = tile / tiles_z;
	const int ty = t2 % tiles_y;
	const int chunk = t2 / tiles_y;
	const int xb = chunk * chunk_len;
	const int xe = min(xb + chunk_len, g.n[0]);
	if constexpr (BODY == 1)
		ch_tile_rq<PREC, MU, DIM, TY, TZ, NT>(a, b, g, p, ty * TY, tz * TZ, xb, xe);
	else
		ch_tile<PREC, MU, DIM, TY, TZ, NT>(a, b, g, p, ty * TY, tz * TZ, xb, xe);
}

// Two steps per pass (3-D, periodic, deterministic chemical potentials).
// FP32 on 32 x 32 tiles asks for six waves per SIMD (80 VGPRs, no spill), so
// two 768-thread workgroups share a CU.
template <int PREC, int MU, int TY, int TZ, int NT, bool PHI2, bool UNIT>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu((PREC != MMSPX_F64 && TZ == 32) ? 6 : 1)))
ch_fused2(const typename Form<PREC>::S* __restrict__ a,
                                                typename Form<PREC>::S* __restrict__ b, Geom g, ModelParams p,
                                                int chunk_len, int tiles_y, int tiles_z, int ntiles)
{
	const int tile = xcd_tile(ntiles);
	if (tile < 0) return;
	const int tz = tile % tiles_z;
	const int t2 = tile / tiles_z;
	const int ty = t2 % tiles_y;
	const int chunk = t2 / tiles_y;
	const int xb = chunk * chunk_len;
	const int xe = min(xb + chunk_len, g.n[0]);
	ch_tile_rq2<PREC, MU, TY, TZ, NT, PHI2, UNIT>(a, b, g, p, ty * TY, tz * TZ, xb, xe);
}

// 3-D plane march (Allen-Cahn, model A, grain growth, Zener pinning): one
// workgroup per (tile, chunk), XCD-contiguous runs as the Cahn-Hilliard tiles.
template <int PREC, int Q, int KIND, int TY, int TZ, int NT>
__global__ void __launch_bounds__(NT) march3d_k(const typename Form<PREC>::S* __restrict__ a,
                                                typename Form<PREC>::S* __restrict__ b, Geom g, ModelParams p,
                                                int chunk_len, int tiles_y, int tiles_z, int ntiles,
                                                const typename Form<PREC>::S* __restrict__ cin,
                                                typename Form<PREC>::S* __restrict__ wout)
{
	const int tile = xcd_tile(ntiles);
	if (tile < 0) return;
	const int tz = tile % tiles_z;
	const int t2 = tile / tiles_z;
	const int ty = t2 % tiles_y;
	const int chunk = t2 / tiles_y;
	const int xb = chunk * chunk_len;
	march3d<PREC, Q, KIND, TY, TZ, NT>(a, b, g, p, ty * TY, tz * TZ, xb, min(xb + chunk_len, g.n[0]), cin, wout);
}

// The plane march two steps per pass (periodic Allen-Cahn, grain growth,
// Zener pinning): one workgroup per (tile, chunk), as march3d_k.
template <int PREC, int Q, int KIND, int TY, int TZ, int NT>
__global__ void __launch_bounds__(NT) march3d2_k(const typename Form<PREC>::S* __restrict__ a,
                                                 typename Form<PREC>::S* __restrict__ b, Geom g, ModelParams p,
                                                 int chunk_len, int tiles_y, int tiles_z, int ntiles)
{
	const int tile = xcd_tile(ntiles);
	if (tile < 0) return;
	const int tz = tile % tiles_z;
	const int t2 = tile / tiles_z;
	const int ty = t2 % tiles_y;
	const int chunk = t2 / tiles_y;
	const int xb = chunk * chunk_len;
	march3d2<PREC, Q, KIND, TY, TZ, NT>(a, b, g, p, ty * TY, tz * TZ, xb, min(xb + chunk_len, g.n[0]));
}

// 3-D Ostwald ripening in one pass (periodic): one workgroup per (tile, chunk).
template <int PREC, int Q, int TY, int TZ, int NT>
__global__ void __launch_bounds__(NT) march3d_ow_k(const typename Form<PREC>::S* __restrict__ a,
                                                   typename Form<PREC>::S* __restrict__ b, Geom g, ModelParams p,
                                                   int chunk_len, int tiles_y, int tiles_z, int ntiles)
{
	const int tile = xcd_tile(ntiles);
	if (tile < 0) return;
	const int tz = tile % tiles_z;
	const int t2 = tile / tiles_z;
	const int ty = t2 % tiles_y;
	const int chunk = t2 / tiles_y;
	const int xb = chunk * chunk_len;
	march3d_ow<PREC, Q, TY, TZ, NT>(a, b, g, p, ty * TY, tz * TZ, xb, min(xb + chunk_len, g.n[0]));
}

template <int PREC, int TZ>
__global__ void __launch_bounds__(TZ) ac_tiled(const typename Form<PREC>::S* __restrict__ a,
                                               typename Form<PREC>::S* __restrict__ b, Geom g, ModelParams p,
                                               int chunk_len, int strips, int ntiles)
{
	const int tile = xcd_tile(ntiles);
	if (tile < 0) return;
	const int s = tile % strips, chunk = tile / strips;
	const int xb = chunk * chunk_len;
	ac_strip<PREC, TZ>(a, b, g, p, s * TZ, xb, min(xb + chunk_len, g.n[0]));
}

template <int PREC, int Q, int TZ>
__global__ void __launch_bounds__(TZ) gg_tiled(const typename Form<PREC>::S* __restrict__ a,
                                               typename Form<PREC>::S* __restrict__ b, Geom g, ModelParams p,
                                               int chunk_len, int strips, int ntiles)
{
	const int tile = xcd_tile(ntiles);
	if (tile < 0) return;
	const int s = tile % strips, chunk = tile / strips;
	const int xb = chunk * chunk_len;
	gg_strip<PREC, Q, TZ>(a, b, g, p, s * TZ, xb, min(xb + chunk_len, g.n[0]));
}

template <int PREC, int Q, int TX, int TC, int NT>
__global__ void __launch_bounds__(NT) gg_tile2d(const typename Form<PREC>::S* __restrict__ a,
                                                typename Form<PREC>::S* __restrict__ b, Geom g, ModelParams p, int tiles_c,
                                                int ntiles)
{
	const int tile = xcd_tile(ntiles);
	if (tile < 0) return;
	const int tc = tile % tiles_c, tr = tile / tiles_c;
	gg_tile<PREC, Q, TX, TC, NT>(a, b, g, p, tr * TX, tc * TC);
}

// Wave strips (2-D Allen-Cahn and grain growth): one wave per (strip, chunk)
// item, four waves per workgroup, strips kWaveCols columns wide. Items run
// strip-fastest, so a workgroup's waves and an XCD's run of workgroups cover
// neighbouring strips of the same rows (shared halo columns in one L2).
template <int PREC, int Q, int KIND>
__global__ void __launch_bounds__(256) wave_strips(const typename Form<PREC>::S* __restrict__ a,
                                                   typename Form<PREC>::S* __restrict__ b, Geom g, ModelParams p,
                                                   int chunk_len, int strips, int nitems, int ntiles)
{
	const int tile = xcd_tile(ntiles);
	if (tile < 0) return;
	const int item = tile * 4 + (int)(threadIdx.x >> 6);
	if (item >= nitems) return;  // a whole wave; the waves share nothing
	const int s = item % strips, chunk = item / strips;
	const int xb = chunk * chunk_len;
	strip_wave<PREC, Q, KIND>(a, b, g, p, s * kWaveCols, xb, min(xb + chunk_len, g.n[0]));
}

// Split wave strips (2-D grain growth, Zener pinning): one workgroup of W
// waves per (strip, chunk) item, each wave holding Q/W of the fields. Items
// run strip-fastest, as the wave strips.
template <int PREC, int Q, int KIND, int W>
__global__ void __launch_bounds__(64 * W) wave_strips_split(const typename Form<PREC>::S* __restrict__ a,
                                                            typename Form<PREC>::S* __restrict__ b, Geom g,
                                                            ModelParams p, int chunk_len, int strips, int nitems)
{
	const int item = xcd_tile(nitems);
	if (item < 0) return;  // the whole workgroup
	const int s = item % strips, chunk = item / strips;
	const int xb = chunk * chunk_len;
	strip_wave_split<PREC, Q, KIND, W>(a, b, g, p, s * kWaveCols, xb, min(xb + chunk_len, g.n[0]));
}

// Two steps per pass on the split strips (periodic): one workgroup of W
// waves per (strip of kChWaveOut columns, chunk), strip-fastest.
template <int PREC, int Q, int KIND, int W>
__global__ void __launch_bounds__(64 * W) wave_strips_split2(const typename Form<PREC>::S* __restrict__ a,
                                                             typename Form<PREC>::S* __restrict__ b, Geom g,
                                                             ModelParams p, int chunk_len, int strips, int nitems)
{
	const int item = xcd_tile(nitems);
	if (item < 0) return;  // the whole workgroup
	const int s = item % strips, chunk = item / strips;
	const int xb = chunk * chunk_len;
	strip_wave_split2<PREC, Q, KIND, W>(a, b, g, p, s * kChWaveOut, xb, min(xb + chunk_len, g.n[0]));
}

// Temporal blocks (2-D periodic Allen-Cahn): one workgroup per TX x kTbCols
// tile, `steps` (<= kTbMaxSteps) steps per launch.
template <int PREC, int TX, int NT>
__global__ void __launch_bounds__(NT) ac_tblocks(const typename Form<PREC>::S* __restrict__ a,
                                                 typename Form<PREC>::S* __restrict__ b, Geom g, ModelParams p,
                                                 int tiles_y, int ntiles, int steps)
{
	const int tile = xcd_tile(ntiles);
	if (tile < 0) return;
	const int ty = tile % tiles_y, tx = tile / tiles_y;
	ac_tblock<PREC, TX, kTbMaxSteps, NT>(a, b, g, p, tx * TX, ty * kTbCols, steps);
}

// Cahn-Hilliard wave strips (2-D periodic): one wave per (strip, chunk) item,
// four waves per workgroup, kChWaveOut columns per strip; odd chunks march
// downward.
template <int PREC, int MU>
__global__ void __launch_bounds__(256) ch_waves(const typename Form<PREC>::S* __restrict__ a,
                                                typename Form<PREC>::S* __restrict__ b, Geom g, ModelParams p,
                                                int chunk_len, int strips, int nitems, int ntiles)
{
	const int tile = xcd_tile(ntiles);
	if (tile < 0) return;
	const int item = tile * 4 + (int)(threadIdx.x >> 6);
	if (item >= nitems) return;  // a whole wave; the waves share nothing
	const int s = item % strips, chunk = item / strips;
	const int xb = chunk * chunk_len;
	ch_wave<PREC, MU>(a, b, g, p, s * kChWaveOut, xb, min(xb + chunk_len, g.n[0]), chunk & 1);
}

// Ostwald ripening wave strips (2-D periodic), laid out as the Cahn-Hilliard
// ones (all rows march upward)
template <int PREC, int Q>
__global__ void __launch_bounds__(256) ow_waves(const typename Form<PREC>::S* __restrict__ a,
                                                typename Form<PREC>::S* __restrict__ b, Geom g, ModelParams p,
                                                int chunk_len, int strips, int nitems, int ntiles)
{
	const int tile = xcd_tile(ntiles);
	if (tile < 0) return;
	const int item = tile * 4 + (int)(threadIdx.x >> 6);
	if (item >= nitems) return;  // a whole wave; the waves share nothing
	const int s = item % strips, chunk = item / strips;
	const int xb = chunk * chunk_len;
	ow_wave<PREC, Q>(a, b, g, p, s * kChWaveOut, xb, min(xb + chunk_len, g.n[0]));
}

template <int PREC, int MU, int DIM, int TY, int TZ, int NT, int BODY>
static int launch_ch_body(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	using S = typename Form<PREC>::S;
	const int nx = g.n[0];
	const int ny = DIM == 3 ? g.n[1] : 1;
	const int nz = DIM == 3 ? g.n[2] : g.n[1];
	const int tiles_y = (ny + TY - 1) / TY;
	const int tiles_z = (nz + TZ - 1) / TZ;
	const int chunks = (nx + chunk - 1) / chunk;
	const int ntiles = tiles_y * tiles_z * chunks;
	// round the grid up to a multiple of 8 so the XCD remap applies; extra ids exit
	const int blocks = (ntiles + 7) / 8 * 8;
	hipLaunchKernelGGL((ch_fused<PREC, MU, DIM, TY, TZ, NT, BODY>), dim3(blocks), dim3(NT), 0, st, (const S*)a, (S*)b, g,
	                   p, chunk, tiles_y, tiles_z, ntiles);
	MMSPX_HIP(hipGetLastError());
	return 0;
}

// The grid weights and the gradient coefficient are all exactly 1 (dx = 1,
// kappa or K = 1): the two-step bodies then leave out the multiplications by them.
static bool unit_weights(const Geom& g, const ModelParams& p, int mu)
{
	for (int k = 0; k < 3; k++)
		if (g.w[k] != 1.0 || g.wf[k] != 1.0f) return false;
	return mu == 1 ? (p.kappa == 1.0 && p.kappaf == 1.0f) : (p.K == 1.0 && p.Kf == 1.0f);
}

template <int PREC, int MU, int TY, int TZ, int NT, bool PHI2>
static int launch_ch2_body(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	using S = typename Form<PREC>::S;
	const int tiles_y = (g.n[1] + TY - 1) / TY;
	const int tiles_z = (g.n[2] + TZ - 1) / TZ;
	const int chunks = (g.n[0] + chunk - 1) / chunk;
	const int ntiles = tiles_y * tiles_z * chunks;
	const int blocks = (ntiles + 7) / 8 * 8;
	if (unit_weights(g, p, MU))
		hipLaunchKernelGGL((ch_fused2<PREC, MU, TY, TZ, NT, PHI2, true>), dim3(blocks), dim3(NT), 0, st, (const S*)a,
		                   (S*)b, g, p, chunk, tiles_y, tiles_z, ntiles);
	else
		hipLaunchKernelGGL((ch_fused2<PREC, MU, TY, TZ, NT, PHI2, false>), dim3(blocks), dim3(NT), 0, st, (const S*)a,
		                   (S*)b, g, p, chunk, tiles_y, tiles_z, ntiles);
	MMSPX_HIP(hipGetLastError());
	return 0;
}

// opt 1 selects the register-queue body (opt 2 and 3, register queues with
// more threads per tile, are dispatched in launch_ch_prec)
template <int PREC, int MU, int DIM, int TY, int TZ, int NT>
static int launch_ch(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk, int opt)
{
	if (opt == 1) return launch_ch_body<PREC, MU, DIM, TY, TZ, NT, 1>(g, p, a, b, st, chunk);
	return launch_ch_body<PREC, MU, DIM, TY, TZ, NT, 0>(g, p, a, b, st, chunk);
}

template <int PREC, int Q, int KIND, int TY, int TZ, int NT>
static int launch_march_body(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk,
                             const void* cin = nullptr, void* wout = nullptr)
{
	using S = typename Form<PREC>::S;
	const int tiles_y = (g.n[1] + TY - 1) / TY;
	const int tiles_z = (g.n[2] + TZ - 1) / TZ;
	const int chunks = (g.n[0] + chunk - 1) / chunk;
	const int ntiles = tiles_y * tiles_z * chunks;
	const int blocks = (ntiles + 7) / 8 * 8;
	hipLaunchKernelGGL((march3d_k<PREC, Q, KIND, TY, TZ, NT>), dim3(blocks), dim3(NT), 0, st, (const S*)a, (S*)b, g,
	                   p, chunk, tiles_y, tiles_z, ntiles, (const S*)cin, (S*)wout);
	MMSPX_HIP(hipGetLastError());
	return 0;
}

// 3-D Ostwald ripening: the two passes as plane marches (8 x 64 or 16 x 32
// tiles, 2, 3 or 4 fields); w goes through `aux` (one scalar plane per node)
template <int PREC>
static int launch_ow3d(const Geom& g, const ModelParams& p, const void* a, void* b, void* aux, hipStream_t st,
                       const TuneChoice& t)
{
	const int chunk = t.chunk > 0 ? t.chunk : 32;
	if (t.opt != 8) return fail(MMSPX_EINVAL, "3-D Ostwald ripening runs tile body 8");
	if (!aux) return fail(MMSPX_EINVAL, "3-D Ostwald ripening needs a scalar plane for w");
	const bool t864 = t.ty == 8 && t.tz == 64, t1632 = t.ty == 16 && t.tz == 32;
	if (!t864 && !t1632) return fail(MMSPX_EINVAL, "no 3-D march compiled for this tile");
	int rc;
	switch (g.fields) {
	case 2:
		rc = t864 ? launch_march_body<PREC, 2, 5, 8, 64, 512>(g, p, a, b, st, chunk, nullptr, aux)
		          : launch_march_body<PREC, 2, 5, 16, 32, 512>(g, p, a, b, st, chunk, nullptr, aux);
		break;
	case 3:
		rc = t864 ? launch_march_body<PREC, 3, 5, 8, 64, 512>(g, p, a, b, st, chunk, nullptr, aux)
		          : launch_march_body<PREC, 3, 5, 16, 32, 512>(g, p, a, b, st, chunk, nullptr, aux);
		break;
	case 4:
		rc = t864 ? launch_march_body<PREC, 4, 5, 8, 64, 512>(g, p, a, b, st, chunk, nullptr, aux)
		          : launch_march_body<PREC, 4, 5, 16, 32, 512>(g, p, a, b, st, chunk, nullptr, aux);
		break;
	default: return fail(MMSPX_EUNSUPPORTED, "the 3-D Ostwald march takes 2, 3 or 4 fields");
	}
	if (rc) return rc;
	return t864 ? launch_march_body<PREC, 1, 6, 8, 64, 256>(g, p, aux, b, st, chunk, a, nullptr)
	            : launch_march_body<PREC, 1, 6, 16, 32, 256>(g, p, aux, b, st, chunk, a, nullptr);
}

// 3-D Ostwald ripening in one pass (tile body 12, periodic): 2, 3 or 4
// fields on 8 x 64 tiles (704 threads) or 16 x 32 (640), one point of the
// tile and its halo per thread
template <int PREC, int Q, int TY, int TZ, int NT>
static int launch_ow1_body(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	using S = typename Form<PREC>::S;
	const int tiles_y = (g.n[1] + TY - 1) / TY;
	const int tiles_z = (g.n[2] + TZ - 1) / TZ;
	const int chunks = (g.n[0] + chunk - 1) / chunk;
	const int ntiles = tiles_y * tiles_z * chunks;
	const int blocks = (ntiles + 7) / 8 * 8;
	hipLaunchKernelGGL((march3d_ow_k<PREC, Q, TY, TZ, NT>), dim3(blocks), dim3(NT), 0, st, (const S*)a, (S*)b, g, p,
	                   chunk, tiles_y, tiles_z, ntiles);
	MMSPX_HIP(hipGetLastError());
	return 0;
}

template <int PREC, int Q>
static int launch_ow1_q(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st,
                        const TuneChoice& t, int chunk)
{
	if (t.ty == 8 && t.tz == 64) return launch_ow1_body<PREC, Q, 8, 64, 704>(g, p, a, b, st, chunk);
	if (t.ty == 16 && t.tz == 32) return launch_ow1_body<PREC, Q, 16, 32, 640>(g, p, a, b, st, chunk);
	return fail(MMSPX_EINVAL, "no one-pass 3-D Ostwald march compiled for this tile");
}

template <int PREC>
static int launch_ow1(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, const TuneChoice& t)
{
	const int chunk = t.chunk > 0 ? t.chunk : 32;
	if (!all_periodic(g)) return fail(MMSPX_EUNSUPPORTED, "the one-pass 3-D Ostwald march needs periodic boundaries");
	switch (g.fields) {
	case 2: return launch_ow1_q<PREC, 2>(g, p, a, b, st, t, chunk);
	case 3: return launch_ow1_q<PREC, 3>(g, p, a, b, st, t, chunk);
	case 4: return launch_ow1_q<PREC, 4>(g, p, a, b, st, t, chunk);
	}
	return fail(MMSPX_EUNSUPPORTED, "the 3-D Ostwald march takes 2, 3 or 4 fields");
}

// tile body 8 on 3-D grids: Allen-Cahn on 8, 16 or 32 x 64 and 16 x 32 tiles;
// the vector models (2, 4 or 8 fields) on 8 x 64 and 16 x 32 tiles, one node
// per thread
template <int PREC, int KIND>
static int launch_march(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st,
                        const TuneChoice& t)
{
	const int chunk = t.chunk > 0 ? t.chunk : 32;
	if (t.opt != 8) return fail(MMSPX_EINVAL, "3-D Allen-Cahn, grain growth, Zener pinning and multi-phase grain growth run tile body 8");
	if constexpr (KIND == 0 || KIND == 2) {
		if (t.ty == 8 && t.tz == 64) return launch_march_body<PREC, 1, KIND, 8, 64, 256>(g, p, a, b, st, chunk);
		if (t.ty == 16 && t.tz == 64) return launch_march_body<PREC, 1, KIND, 16, 64, 256>(g, p, a, b, st, chunk);
		if (t.ty == 32 && t.tz == 64) return launch_march_body<PREC, 1, KIND, 32, 64, 512>(g, p, a, b, st, chunk);
		if (t.ty == 16 && t.tz == 32) return launch_march_body<PREC, 1, KIND, 16, 32, 256>(g, p, a, b, st, chunk);
	} else {
		const bool t864 = t.ty == 8 && t.tz == 64, t1632 = t.ty == 16 && t.tz == 32;
		switch (g.fields) {
		case 2:
			if (t864) return launch_march_body<PREC, 2, KIND, 8, 64, 512>(g, p, a, b, st, chunk);
			if (t1632) return launch_march_body<PREC, 2, KIND, 16, 32, 512>(g, p, a, b, st, chunk);
			break;
		case 4:
			if (t864) return launch_march_body<PREC, 4, KIND, 8, 64, 512>(g, p, a, b, st, chunk);
			if (t1632) return launch_march_body<PREC, 4, KIND, 16, 32, 512>(g, p, a, b, st, chunk);
			break;
		case 8:
			if (t864) return launch_march_body<PREC, 8, KIND, 8, 64, 512>(g, p, a, b, st, chunk);
			if (t1632) return launch_march_body<PREC, 8, KIND, 16, 32, 512>(g, p, a, b, st, chunk);
			break;
		default: return fail(MMSPX_EUNSUPPORTED, "the 3-D march takes 2, 4 or 8 fields");
		}
	}
	return fail(MMSPX_EINVAL, "no 3-D march compiled for this tile");
}

// Tile body 12 on periodic 3-D grids: the plane march two steps per pass.
// The threads own the tile and its one-cell halo, one point each for the
// vector models (8 x 64 tiles on 704 threads, 16 x 32 on 640, 8 x 32 on
// 384), two or three for Allen-Cahn (16 x 32 on 320, 16 x 64 on 640, 32 x 64
// on 768). LDS: the phi^n plane with a two-cell halo and the phi^{n+1} plane
// on the owned points, both double-buffered, Q fields each.
template <int PREC, int Q, int KIND, int TY, int TZ, int NT>
static int launch_march2_body(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	using S = typename Form<PREC>::S;
	constexpr size_t lds = (size_t)2 * Q * ((TY + 4) * (TZ + 4) + (TY + 2) * (TZ + 2)) * sizeof(S);
	if constexpr (lds > (size_t)160 * 1024) {
		return fail(MMSPX_EINVAL, "the planes of this tile and field count do not fit the LDS");
	} else {
		const int tiles_y = (g.n[1] + TY - 1) / TY;
		const int tiles_z = (g.n[2] + TZ - 1) / TZ;
		const int chunks = (g.n[0] + chunk - 1) / chunk;
		const int ntiles = tiles_y * tiles_z * chunks;
		const int blocks = (ntiles + 7) / 8 * 8;
		hipLaunchKernelGGL((march3d2_k<PREC, Q, KIND, TY, TZ, NT>), dim3(blocks), dim3(NT), 0, st, (const S*)a,
		                   (S*)b, g, p, chunk, tiles_y, tiles_z, ntiles);
		MMSPX_HIP(hipGetLastError());
		return 0;
	}
}

template <int PREC, int Q, int KIND>
static int launch_march2_q(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st,
                           const TuneChoice& t, int chunk)
{
	if (t.ty == 8 && t.tz == 64) return launch_march2_body<PREC, Q, KIND, 8, 64, 704>(g, p, a, b, st, chunk);
	if (t.ty == 16 && t.tz == 32) return launch_march2_body<PREC, Q, KIND, 16, 32, 640>(g, p, a, b, st, chunk);
	if (t.ty == 8 && t.tz == 32) return launch_march2_body<PREC, Q, KIND, 8, 32, 384>(g, p, a, b, st, chunk);
	return fail(MMSPX_EINVAL, "no two-step 3-D march compiled for this tile");
}

template <int PREC, int KIND>
static int launch_march2(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st,
                         const TuneChoice& t, int nsteps)
{
	const int chunk = t.chunk > 0 ? t.chunk : 32;
	if (!all_periodic(g)) return fail(MMSPX_EUNSUPPORTED, "tile body 12 (two steps per pass) needs periodic boundaries");
	if (PREC == MMSPX_F32REF) return fail(MMSPX_EUNSUPPORTED, "tile body 12 runs the MMSPX_F64 and MMSPX_F32 forms");
	if (nsteps == 1) {
		// an odd last step: the one-step march
		const TuneChoice t1{2, KIND == 0 ? 16 : 8, KIND == 0 ? 32 : 64, chunk, 8};
		return launch_march<PREC, KIND>(g, p, a, b, st, t1);
	}
	if (nsteps != 2) return fail(MMSPX_EINVAL, "tile body 12 takes one or two steps per pass");
	if constexpr (PREC == MMSPX_F32REF) {
		return fail(MMSPX_EUNSUPPORTED, "tile body 12 runs the MMSPX_F64 and MMSPX_F32 forms");
	} else if constexpr (KIND == 0) {
		if (t.ty == 16 && t.tz == 32) return launch_march2_body<PREC, 1, 0, 16, 32, 320>(g, p, a, b, st, chunk);
		if (t.ty == 16 && t.tz == 64) return launch_march2_body<PREC, 1, 0, 16, 64, 640>(g, p, a, b, st, chunk);
		if (t.ty == 32 && t.tz == 64) return launch_march2_body<PREC, 1, 0, 32, 64, 768>(g, p, a, b, st, chunk);
		return fail(MMSPX_EINVAL, "no two-step 3-D march compiled for this tile");
	} else {
		switch (g.fields) {
		case 2: return launch_march2_q<PREC, 2, KIND>(g, p, a, b, st, t, chunk);
		case 4: return launch_march2_q<PREC, 4, KIND>(g, p, a, b, st, t, chunk);
		case 8: return launch_march2_q<PREC, 8, KIND>(g, p, a, b, st, t, chunk);
		}
		return fail(MMSPX_EUNSUPPORTED, "the two-step 3-D march takes 2, 4 or 8 fields");
	}
}

template <int PREC, int MU>
static int launch_ch_waves(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	using S = typename Form<PREC>::S;
	const int strips = (g.n[1] + kChWaveOut - 1) / kChWaveOut;
	const int nitems = strips * ((g.n[0] + chunk - 1) / chunk);
	const int ntiles = (nitems + 3) / 4;
	const int blocks = (ntiles + 7) / 8 * 8;
	hipLaunchKernelGGL((ch_waves<PREC, MU>), dim3(blocks), dim3(256), 0, st, (const S*)a, (S*)b, g, p, chunk, strips,
	                   nitems, ntiles);
	MMSPX_HIP(hipGetLastError());
	return 0;
}

template <int PREC, int MU>
static int launch_ch_prec(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st,
                          const TuneChoice& t, int nsteps)
{
	const int chunk = t.chunk > 0 ? t.chunk : 32;
	if (!all_periodic(g) && !ch_body_maps_edges(g, t))
		return fail(MMSPX_EUNSUPPORTED, "non-periodic boundaries run the register-queue bodies (1, 2, 3) or the "
		                                "2-D wave strips");
	if (g.dim == 3 && (t.opt == 6 || t.opt == 7)) {
		// two steps per pass: body 6 on 32 x 64 tiles (896 threads; the c^n plane
		// double-buffered in FP32, single in FP64 where the LDS would not hold
		// two), body 7 on 32 x 32 tiles (768 threads, every plane
		// double-buffered); an odd last step runs the one-step register queues
		if constexpr (MU == 2) {
			return fail(MMSPX_EUNSUPPORTED, "the two-step bodies take the deterministic chemical potentials");
		} else {
			if (nsteps == 1)
				return launch_ch_body<PREC, MU, 3, 32, 64, 768, 1>(g, p, a, b, st, PREC == MMSPX_F64 ? 32 : 16);
			if (nsteps != 2) return fail(MMSPX_EINVAL, "the two-step bodies take one or two steps per pass");
			if (t.opt == 6) {
				if (t.ty != 32 || t.tz != 64) return fail(MMSPX_EINVAL, "tile body 6 runs 32 x 64 tiles");
				return launch_ch2_body<PREC, MU, 32, 64, 896, PREC != MMSPX_F64>(g, p, a, b, st, chunk);
			}
			if (t.ty != 32 || t.tz != 32) return fail(MMSPX_EINVAL, "tile body 7 runs 32 x 32 tiles");
			return launch_ch2_body<PREC, MU, 32, 32, 768, true>(g, p, a, b, st, chunk);
		}
	}
	if (g.dim == 3 && t.ty == 32 && t.tz == 32) return fail(MMSPX_EINVAL, "32 x 32 tiles run tile body 7");
	if (g.dim == 3 && (t.opt == 2 || t.opt == 3)) {
		// register queues on 32 x 64 tiles with 768 or 1024 threads (fewer own points each)
		if (t.ty != 32 || t.tz != 64) return fail(MMSPX_EINVAL, "tile bodies 2 and 3 run 32 x 64 tiles");
		if (t.opt == 3) return launch_ch_body<PREC, MU, 3, 32, 64, 1024, 1>(g, p, a, b, st, chunk);
		return launch_ch_body<PREC, MU, 3, 32, 64, 768, 1>(g, p, a, b, st, chunk);
	}
	if (g.dim == 3) {
		if (t.ty == 16 && t.tz == 64) return launch_ch<PREC, MU, 3, 16, 64, 256>(g, p, a, b, st, chunk, t.opt);
		if (t.ty == 32 && t.tz == 64) return launch_ch<PREC, MU, 3, 32, 64, 512>(g, p, a, b, st, chunk, t.opt);
		if (t.ty == 8 && t.tz == 32) return launch_ch<PREC, MU, 3, 8, 32, 256>(g, p, a, b, st, chunk, t.opt);
		if (t.ty == 4 && t.tz == 128) return launch_ch<PREC, MU, 3, 4, 128, 256>(g, p, a, b, st, chunk, t.opt);
		return launch_ch<PREC, MU, 3, 8, 64, 256>(g, p, a, b, st, chunk, t.opt);
	}
	if (t.tz == kChWaveOut) return launch_ch_waves<PREC, MU>(g, p, a, b, st, chunk);
	if (t.tz == 64) return launch_ch<PREC, MU, 2, 1, 64, 64>(g, p, a, b, st, chunk, t.opt);
	if (t.tz == 128) return launch_ch<PREC, MU, 2, 1, 128, 128>(g, p, a, b, st, chunk, t.opt);
	return launch_ch<PREC, MU, 2, 1, 256, 256>(g, p, a, b, st, chunk, t.opt);
}

template <int PREC, int TZ>
static int launch_ac(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	using S = typename Form<PREC>::S;
	const int strips = (g.n[1] + TZ - 1) / TZ;
	const int ntiles = strips * ((g.n[0] + chunk - 1) / chunk);
	const int blocks = (ntiles + 7) / 8 * 8;
	hipLaunchKernelGGL((ac_tiled<PREC, TZ>), dim3(blocks), dim3(TZ), 0, st, (const S*)a, (S*)b, g, p, chunk, strips,
	                   ntiles);
	MMSPX_HIP(hipGetLastError());
	return 0;
}

template <int PREC, int Q, int TZ>
static int launch_gg_q(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	using S = typename Form<PREC>::S;
	const int strips = (g.n[1] + TZ - 1) / TZ;
	const int ntiles = strips * ((g.n[0] + chunk - 1) / chunk);
	const int blocks = (ntiles + 7) / 8 * 8;
	hipLaunchKernelGGL((gg_tiled<PREC, Q, TZ>), dim3(blocks), dim3(TZ), 0, st, (const S*)a, (S*)b, g, p, chunk, strips,
	                   ntiles);
	MMSPX_HIP(hipGetLastError());
	return 0;
}

template <int PREC, int Q, int TX>
static int launch_gg_tile_q(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st)
{
	using S = typename Form<PREC>::S;
	constexpr int TC = 64, NT = 256;
	const int tiles_c = (g.n[1] + TC - 1) / TC;
	const int ntiles = tiles_c * ((g.n[0] + TX - 1) / TX);
	const int blocks = (ntiles + 7) / 8 * 8;
	hipLaunchKernelGGL((gg_tile2d<PREC, Q, TX, TC, NT>), dim3(blocks), dim3(NT), 0, st, (const S*)a, (S*)b, g, p,
	                   tiles_c, ntiles);
	MMSPX_HIP(hipGetLastError());
	return 0;
}

template <int PREC, int TX>
static int launch_gg_tile(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st)
{
	switch (g.fields) {
	case 2: return launch_gg_tile_q<PREC, 2, TX>(g, p, a, b, st);
	case 4: return launch_gg_tile_q<PREC, 4, TX>(g, p, a, b, st);
	case 8: return launch_gg_tile_q<PREC, 8, TX>(g, p, a, b, st);
	case 16: return launch_gg_tile_q<PREC, 16, TX>(g, p, a, b, st);
	case 32: return launch_gg_tile_q<PREC, 32, TX>(g, p, a, b, st);
	}
	return fail(MMSPX_EUNSUPPORTED, "no tiled grain-growth kernel for this field count");
}

template <int PREC, int TZ>
static int launch_gg_tz(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	switch (g.fields) {
	case 2: return launch_gg_q<PREC, 2, TZ>(g, p, a, b, st, chunk);
	case 4: return launch_gg_q<PREC, 4, TZ>(g, p, a, b, st, chunk);
	case 8: return launch_gg_q<PREC, 8, TZ>(g, p, a, b, st, chunk);
	case 16: return launch_gg_q<PREC, 16, TZ>(g, p, a, b, st, chunk);
	case 32: return launch_gg_q<PREC, 32, TZ>(g, p, a, b, st, chunk);
	}
	return fail(MMSPX_EUNSUPPORTED, "no tiled grain-growth kernel for this field count");
}

template <int PREC, int TX>
static int launch_tb(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int steps)
{
	using S = typename Form<PREC>::S;
	const int tiles_y = (g.n[1] + kTbCols - 1) / kTbCols;
	const int ntiles = tiles_y * ((g.n[0] + TX - 1) / TX);
	const int blocks = (ntiles + 7) / 8 * 8;
	// 8-row blocks on 8 waves, 16- and 32-row blocks on 16 (a wave takes 3
	// of the 24, 32 or 48 region rows per step): 512^2 FP64 with 32 rows 1.48
	// us per step on 1024 threads against 2.50 on 256
	constexpr int NT = TX == 8 ? 512 : 1024;
	hipLaunchKernelGGL((ac_tblocks<PREC, TX, NT>), dim3(blocks), dim3(NT), 0, st, (const S*)a, (S*)b, g, p, tiles_y,
	                   ntiles, steps);
	MMSPX_HIP(hipGetLastError());
	return 0;
}

template <int PREC, int Q, int KIND>
static int launch_wave_q(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	using S = typename Form<PREC>::S;
	const int strips = (g.n[1] + kWaveCols - 1) / kWaveCols;
	const int nitems = strips * ((g.n[0] + chunk - 1) / chunk);
	const int ntiles = (nitems + 3) / 4;
	const int blocks = (ntiles + 7) / 8 * 8;
	hipLaunchKernelGGL((wave_strips<PREC, Q, KIND>), dim3(blocks), dim3(256), 0, st, (const S*)a, (S*)b, g, p, chunk,
	                   strips, nitems, ntiles);
	MMSPX_HIP(hipGetLastError());
	return 0;
}

// Grain growth and Zener pinning: the wave strips keep four rows of every field in registers: compiled for up
// to 128 bytes of field values per cell (FP32 up to 32 fields, FP64 up to 16).
template <int PREC>
static int launch_wave(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	constexpr bool wide = sizeof(typename Form<PREC>::S) == 4;
	if (p.model == MMSPX_ZENER) {
		if constexpr (PREC != MMSPX_F32REF) {
			switch (g.fields) {
			case 2: return launch_wave_q<PREC, 2, 3>(g, p, a, b, st, chunk);
			case 4: return launch_wave_q<PREC, 4, 3>(g, p, a, b, st, chunk);
			case 8: return launch_wave_q<PREC, 8, 3>(g, p, a, b, st, chunk);
			case 16: return launch_wave_q<PREC, 16, 3>(g, p, a, b, st, chunk);
			case 32:
				if constexpr (wide) return launch_wave_q<PREC, 32, 3>(g, p, a, b, st, chunk);
				break;
			}
		}
		return fail(MMSPX_EUNSUPPORTED, "no wave-strip kernel for this field count and precision");
	}
	switch (g.fields) {
	case 2: return launch_wave_q<PREC, 2, 1>(g, p, a, b, st, chunk);
	case 4: return launch_wave_q<PREC, 4, 1>(g, p, a, b, st, chunk);
	case 8: return launch_wave_q<PREC, 8, 1>(g, p, a, b, st, chunk);
	case 16: return launch_wave_q<PREC, 16, 1>(g, p, a, b, st, chunk);
	case 32:
		if constexpr (wide) return launch_wave_q<PREC, 32, 1>(g, p, a, b, st, chunk);
		break;
	}
	return fail(MMSPX_EUNSUPPORTED, "no wave-strip kernel for this field count and precision");
}

template <int PREC, int Q, int KIND, int W>
static int launch_split_q(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	using S = typename Form<PREC>::S;
	const int strips = (g.n[1] + kWaveCols - 1) / kWaveCols;
	const int nitems = strips * ((g.n[0] + chunk - 1) / chunk);
	const int blocks = (nitems + 7) / 8 * 8;
	hipLaunchKernelGGL((wave_strips_split<PREC, Q, KIND, W>), dim3(blocks), dim3(64 * W), 0, st, (const S*)a, (S*)b, g,
	                   p, chunk, strips, nitems);
	MMSPX_HIP(hipGetLastError());
	return 0;
}

template <int PREC, int KIND, int W>
static int launch_split_w(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	switch (g.fields) {
	case 8: return launch_split_q<PREC, 8, KIND, W>(g, p, a, b, st, chunk);
	case 16: return launch_split_q<PREC, 16, KIND, W>(g, p, a, b, st, chunk);
	case 32: return launch_split_q<PREC, 32, KIND, W>(g, p, a, b, st, chunk);
	}
	return fail(MMSPX_EUNSUPPORTED, "split wave strips take 8, 16 or 32 fields");
}

// The split strips: grain growth and Zener pinning with 8, 16 or 32 fields
// on W = 2 (body 4) or 4 (body 5) waves per strip
template <int PREC>
static int launch_split(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk,
                        int waves)
{
	if (p.model == MMSPX_ZENER) {
		if constexpr (PREC != MMSPX_F32REF)
			return waves == 4 ? launch_split_w<PREC, 3, 4>(g, p, a, b, st, chunk)
			                  : launch_split_w<PREC, 3, 2>(g, p, a, b, st, chunk);
		return fail(MMSPX_EUNSUPPORTED, "Zener pinning runs the MMSPX_F64 and MMSPX_F32 forms");
	}
	return waves == 4 ? launch_split_w<PREC, 1, 4>(g, p, a, b, st, chunk)
	                  : launch_split_w<PREC, 1, 2>(g, p, a, b, st, chunk);
}

template <int PREC, int Q, int KIND, int W>
static int launch_split2_q(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	using S = typename Form<PREC>::S;
	const int strips = (g.n[1] + kChWaveOut - 1) / kChWaveOut;
	const int nitems = strips * ((g.n[0] + chunk - 1) / chunk);
	const int blocks = (nitems + 7) / 8 * 8;
	hipLaunchKernelGGL((wave_strips_split2<PREC, Q, KIND, W>), dim3(blocks), dim3(64 * W), 0, st, (const S*)a, (S*)b,
	                   g, p, chunk, strips, nitems);
	MMSPX_HIP(hipGetLastError());
	return 0;
}

template <int PREC, int KIND, int W>
static int launch_split2_w(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	if constexpr (W == 1) {
		// one wave holds every field: 2, 4 or 8 of them
		switch (g.fields) {
		case 2: return launch_split2_q<PREC, 2, KIND, 1>(g, p, a, b, st, chunk);
		case 4: return launch_split2_q<PREC, 4, KIND, 1>(g, p, a, b, st, chunk);
		case 8: return launch_split2_q<PREC, 8, KIND, 1>(g, p, a, b, st, chunk);
		}
		return fail(MMSPX_EUNSUPPORTED, "the one-wave two-step strips take 2, 4 or 8 fields");
	} else {
		switch (g.fields) {
		case 8: return launch_split2_q<PREC, 8, KIND, W>(g, p, a, b, st, chunk);
		case 16: return launch_split2_q<PREC, 16, KIND, W>(g, p, a, b, st, chunk);
		case 32: return launch_split2_q<PREC, 32, KIND, W>(g, p, a, b, st, chunk);
		}
		return fail(MMSPX_EUNSUPPORTED, "split wave strips take 8, 16 or 32 fields");
	}
}

// Grain growth and Zener pinning, periodic 2-D: two steps per pass on the
// split strips, W = 2 (body 9) or 4 (body 10) waves per strip for 8, 16 or
// 32 fields, one wave (body 11) for 2, 4 or 8; a single step (an odd last
// one) runs the one-step split strips (W = 2, 4) or wave strips (W = 1)
template <int PREC>
static int launch_split2(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk,
                         int waves, int nsteps)
{
	if (!all_periodic(g)) return fail(MMSPX_EUNSUPPORTED, "the two-step split strips need periodic boundaries");
	if (nsteps == 1)
		return waves == 1 ? launch_wave<PREC>(g, p, a, b, st, chunk) : launch_split<PREC>(g, p, a, b, st, chunk, waves);
	if (nsteps != 2) return fail(MMSPX_EINVAL, "the two-step split strips take one or two steps per pass");
	const bool zener = p.model == MMSPX_ZENER;
	if constexpr (PREC == MMSPX_F32REF) {
		if (zener) return fail(MMSPX_EUNSUPPORTED, "Zener pinning runs the MMSPX_F64 and MMSPX_F32 forms");
		return waves == 1 ? launch_split2_w<PREC, 1, 1>(g, p, a, b, st, chunk)
		     : waves == 4 ? launch_split2_w<PREC, 1, 4>(g, p, a, b, st, chunk)
		                  : launch_split2_w<PREC, 1, 2>(g, p, a, b, st, chunk);
	} else {
		if (waves == 1)
			return zener ? launch_split2_w<PREC, 3, 1>(g, p, a, b, st, chunk) : launch_split2_w<PREC, 1, 1>(g, p, a, b, st, chunk);
		if (waves == 4)
			return zener ? launch_split2_w<PREC, 3, 4>(g, p, a, b, st, chunk) : launch_split2_w<PREC, 1, 4>(g, p, a, b, st, chunk);
		return zener ? launch_split2_w<PREC, 3, 2>(g, p, a, b, st, chunk) : launch_split2_w<PREC, 1, 2>(g, p, a, b, st, chunk);
	}
}

template <int PREC, int Q>
static int launch_ow_q(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	using S = typename Form<PREC>::S;
	const int strips = (g.n[1] + kChWaveOut - 1) / kChWaveOut;
	const int nitems = strips * ((g.n[0] + chunk - 1) / chunk);
	const int ntiles = (nitems + 3) / 4;
	const int blocks = (ntiles + 7) / 8 * 8;
	hipLaunchKernelGGL((ow_waves<PREC, Q>), dim3(blocks), dim3(256), 0, st, (const S*)a, (S*)b, g, p, chunk, strips,
	                   nitems, ntiles);
	MMSPX_HIP(hipGetLastError());
	return 0;
}

template <int PREC>
static int launch_ow(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk)
{
	if constexpr (PREC != MMSPX_F32REF) {
		switch (g.fields) {
		case 2: return launch_ow_q<PREC, 2>(g, p, a, b, st, chunk);
		case 3: return launch_ow_q<PREC, 3>(g, p, a, b, st, chunk);
		case 4: return launch_ow_q<PREC, 4>(g, p, a, b, st, chunk);
		case 5: return launch_ow_q<PREC, 5>(g, p, a, b, st, chunk);
		case 6: return launch_ow_q<PREC, 6>(g, p, a, b, st, chunk);
		case 7: return launch_ow_q<PREC, 7>(g, p, a, b, st, chunk);
		case 8: return launch_ow_q<PREC, 8>(g, p, a, b, st, chunk);
		}
	}
	return fail(MMSPX_EUNSUPPORTED, "Ostwald wave strips take 2 to 8 fields in the MMSPX_F64 and MMSPX_F32 forms");
}

// Allen-Cahn and model A
template <int PREC>
static int launch_fused_ac(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st,
                           const TuneChoice& t, int nsteps, void* aux)
{
	[[maybe_unused]] const int chunk = t.chunk > 0 ? t.chunk : 32;
	switch (p.model) {
	case MMSPX_AC_NOISE:
		if (g.dim == 3) return launch_march<PREC, 2>(g, p, a, b, st, t);
		// model A: wave strips only (the noise is drawn per node and step)
		if (t.opt == 2 && t.ty == 1 && t.tz == kWaveCols) return launch_wave_q<PREC, 1, 2>(g, p, a, b, st, chunk);
		return fail(MMSPX_EUNSUPPORTED, "Allen-Cahn with noise runs the wave strips (1 x 64, body 2) or the generic kernel");
	case MMSPX_AC:
		if (g.dim == 3) return t.opt == 12 ? launch_march2<PREC, 0>(g, p, a, b, st, t, nsteps)
		                                   : launch_march<PREC, 0>(g, p, a, b, st, t);
		if (t.tz == kTbCols) {
			if (!all_periodic(g)) return fail(MMSPX_EUNSUPPORTED, "temporal blocks need periodic boundaries");
			if (nsteps < 1 || nsteps > kTbMaxSteps) return fail(MMSPX_EINVAL, "temporal blocks take 1..8 steps per pass");
			if (t.ty == 8) return launch_tb<PREC, 8>(g, p, a, b, st, nsteps);
			return t.ty == 32 ? launch_tb<PREC, 32>(g, p, a, b, st, nsteps) : launch_tb<PREC, 16>(g, p, a, b, st, nsteps);
		}
		if (t.opt == 2 && t.ty == 1 && t.tz == kWaveCols) return launch_wave_q<PREC, 1, 0>(g, p, a, b, st, chunk);
		if (t.tz == 64) return launch_ac<PREC, 64>(g, p, a, b, st, chunk);
		if (t.tz == 128) return launch_ac<PREC, 128>(g, p, a, b, st, chunk);
		return launch_ac<PREC, 256>(g, p, a, b, st, chunk);
	}
	return fail(MMSPX_EINVAL, "unknown model");
}

// Cahn-Hilliard and model B
template <int PREC>
static int launch_fused_ch(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st,
                           const TuneChoice& t, int nsteps, void* aux)
{
	[[maybe_unused]] const int chunk = t.chunk > 0 ? t.chunk : 32;
	switch (p.model) {
	case MMSPX_CH: return launch_ch_prec<PREC, 0>(g, p, a, b, st, t, nsteps);
	case MMSPX_CH_DW: return launch_ch_prec<PREC, 1>(g, p, a, b, st, t, nsteps);
	case MMSPX_CH_NOISE: return launch_ch_prec<PREC, 2>(g, p, a, b, st, t, nsteps);
	}
	return fail(MMSPX_EINVAL, "unknown model");
}

// Grain growth and Zener pinning
template <int PREC>
static int launch_fused_gg(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st,
                           const TuneChoice& t, int nsteps, void* aux)
{
	[[maybe_unused]] const int chunk = t.chunk > 0 ? t.chunk : 32;
	switch (p.model) {
	case MMSPX_ZENER:
		if (g.dim == 3) return t.opt == 12 ? launch_march2<PREC, 3>(g, p, a, b, st, t, nsteps)
		                                   : launch_march<PREC, 3>(g, p, a, b, st, t);
		if (t.opt >= 9 && t.opt <= 11 && t.ty == 1 && t.tz == kChWaveOut)
			return launch_split2<PREC>(g, p, a, b, st, chunk, t.opt == 11 ? 1 : t.opt == 10 ? 4 : 2, nsteps);
		if ((t.opt == 4 || t.opt == 5) && t.ty == 1 && t.tz == kWaveCols)
			return launch_split<PREC>(g, p, a, b, st, chunk, t.opt == 5 ? 4 : 2);
		if (t.opt == 2 && t.ty == 1 && t.tz == kWaveCols) return launch_wave<PREC>(g, p, a, b, st, chunk);
		return fail(MMSPX_EUNSUPPORTED, "Zener pinning runs the wave strips (1 x 64, body 2) or the generic kernel");
	case MMSPX_GG:
		if (g.dim == 3) return t.opt == 12 ? launch_march2<PREC, 1>(g, p, a, b, st, t, nsteps)
		                                   : launch_march<PREC, 1>(g, p, a, b, st, t);
		if (t.opt >= 9 && t.opt <= 11 && t.ty == 1 && t.tz == kChWaveOut)
			return launch_split2<PREC>(g, p, a, b, st, chunk, t.opt == 11 ? 1 : t.opt == 10 ? 4 : 2, nsteps);
		// ty > 1: 2-D tiles of ty (8 or 16) rows x 64 columns; body 2 with 64
		// columns: wave strips; otherwise LDS-row marching strips
		if ((t.opt == 4 || t.opt == 5) && t.ty == 1 && t.tz == kWaveCols)
			return launch_split<PREC>(g, p, a, b, st, chunk, t.opt == 5 ? 4 : 2);
		if (t.opt == 2 && t.ty == 1 && t.tz == kWaveCols) return launch_wave<PREC>(g, p, a, b, st, chunk);
		if (t.ty > 1) return t.ty == 16 ? launch_gg_tile<PREC, 16>(g, p, a, b, st) : launch_gg_tile<PREC, 8>(g, p, a, b, st);
		if (t.tz == 64) return launch_gg_tz<PREC, 64>(g, p, a, b, st, chunk);
		if (t.tz == 256 && PREC != MMSPX_F64) return launch_gg_tz<PREC, 256>(g, p, a, b, st, chunk);
		return launch_gg_tz<PREC, 128>(g, p, a, b, st, chunk);
	}
	return fail(MMSPX_EINVAL, "unknown model");
}

// Ostwald ripening and multi-phase grain growth
template <int PREC>
static int launch_fused_rest(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st,
                           const TuneChoice& t, int nsteps, void* aux)
{
	[[maybe_unused]] const int chunk = t.chunk > 0 ? t.chunk : 32;
	switch (p.model) {
	case MMSPX_OSTWALD:
		if (g.dim == 3) {
			if constexpr (PREC == MMSPX_F32REF) return fail(MMSPX_EUNSUPPORTED, "no 3-D march for this form");
			else return t.opt == 12 ? launch_ow1<PREC>(g, p, a, b, st, t) : launch_ow3d<PREC>(g, p, a, b, aux, st, t);
		}
		if (g.dim == 2 && t.ty == 1 && t.tz == kChWaveOut) {
			if (!all_periodic(g)) return fail(MMSPX_EUNSUPPORTED, "Ostwald wave strips need periodic boundaries");
			return launch_ow<PREC>(g, p, a, b, st, chunk);
		}
		return fail(MMSPX_EUNSUPPORTED, "Ostwald ripening runs the wave strips (1 x 60) or the generic kernels");
	case MMSPX_GG_ANISO:
		if (g.dim == 3) {
			if constexpr (PREC == MMSPX_F32REF) return fail(MMSPX_EUNSUPPORTED, "no 3-D march for this form");
			else return launch_march<PREC, 4>(g, p, a, b, st, t);
		}
		if (t.opt == 2 && t.ty == 1 && t.tz == kWaveCols) return launch_gga2d(g, PREC, p, a, b, st, chunk);
		return fail(MMSPX_EUNSUPPORTED, "multi-phase grain growth runs the wave strips (1 x 64, body 2) or the generic kernel");
	}
	return fail(MMSPX_EINVAL, "unknown model");
}

}  // namespace mmspx
