// kernels_fused.hip -- the tiled kernels for single grids (fused_launch.hpp): which
// of them, and of the multi-step kernels, a grid and a call take, and the dispatch.
#include <algorithm>
#include <cstring>

#include "fused.hpp"

namespace mmspx {

bool fused_supported(const Geom& g, int prec, int model)
{
	(void)prec;
	if (g.dim == 3) {
		if (model == MMSPX_AC || model == MMSPX_AC_NOISE) return true;
		if (model == MMSPX_GG) return march_q_compiled(g.fields);
		if (model == MMSPX_ZENER || model == MMSPX_GG_ANISO) return march_q_compiled(g.fields) && prec != MMSPX_F32REF;
		if (model == MMSPX_OSTWALD) return g.fields >= 2 && g.fields <= 4 && prec != MMSPX_F32REF;
	}
	switch (model) {
	case MMSPX_CH:
	case MMSPX_CH_DW:
	case MMSPX_CH_NOISE: return g.dim >= 2 && axes_uniform(g);
	case MMSPX_AC:
	case MMSPX_AC_NOISE: return g.dim == 2;
	case MMSPX_GG: return g.dim == 2 && gg_q_compiled(g.fields);
	// Ostwald ripening: the wave strips for 2 to 8 fields on periodic grids
	case MMSPX_OSTWALD:
		return g.dim == 2 && all_periodic(g) && g.fields >= 2 && g.fields <= 8 && prec != MMSPX_F32REF;
	// multi-phase grain growth: the wave strips for 2, 4 and 8 fields (the
	// per-node arrays of more fields would not fit the registers)
	case MMSPX_GG_ANISO:
		return g.dim == 2 && (g.fields == 2 || g.fields == 4 || g.fields == 8) && prec != MMSPX_F32REF;
	// Zener pinning: the wave strips, where their registers hold the fields
	case MMSPX_ZENER:
		return g.dim == 2 && gg_q_compiled(g.fields) && prec != MMSPX_F32REF && (g.fields < 32 || prec != MMSPX_F64);
	}
	return false;
}

// Periodic 3-D Cahn-Hilliard with a deterministic chemical potential: two
// steps per pass on 32 x 32 tiles (768 threads) or, in FP32, 32 x 64 tiles
// (896 threads), whichever the cost model below favours. A workgroup's time
// grows with its planes (chunk + 6: three halo planes of the two steps on
// each side are recomputed) times the R3 points each thread owns; a launch
// takes as many such rounds as its workgroups fill the 256 CUs. One
// workgroup fits a CU, except FP32 on 32 x 32 tiles (80 VGPRs, 44 KB of LDS:
// two per CU), where a launch of more than 256 workgroups takes rounds of
// 512, each 1.7 times as long (the two share the CU; fitted to the FP32
// sweep, which the model then matches at every side). The chunk with the
// least rounds x time wins (ties: the longer chunk).
// Against a sweep of every chunk on cubes of side 48 to 256 (us per step):
// the model picks the measured best in FP64 at every side (128^3: 8-plane
// chunks, 10.8 against 22.9 for the former 8 x 32 LDS-ring default; 192^3:
// 32, 25.8 against 41.5; 224^3: 48, 37.8 against 59.7; 256^3: 64, 50.5) and
// in FP32 (128^3 32 x 32 tiles with 8-plane chunks 8.8 against 18.8; 192^3
// 32 x 64 with 16, 16.9 against 34.0; 224^3 32 x 32 with 24, 25.9 against
// 47.1; 256^3 32 x 64 with 32, 29.6).
static TuneChoice two_step_choice(const Geom& g, int prec)
{
	constexpr int kCUs = 256;
	static const int chunks[] = {6, 8, 12, 16, 24, 32, 48, 64};
	TuneChoice best{2, 32, 32, 64, 7};
	double best_cost = 1e300;
	for (int body = 7; body >= 6; body--) {
		if (body == 6 && prec != MMSPX_F32) continue;  // FP64 32 x 64 tiles spill
		const int ty = 32, tz = body == 7 ? 32 : 64, nt = body == 7 ? 768 : 896;
		const double own = (double)(ty + 6) * (tz + 6) / nt;  // R3 points per thread
		const bool two_per_cu = body == 7 && prec == MMSPX_F32;
		const int64_t tiles = (int64_t)((g.n[1] + ty - 1) / ty) * ((g.n[2] + tz - 1) / tz);
		for (int c : chunks) {
			const int64_t wgs = tiles * ((g.n[0] + c - 1) / c);
			const double rounds = (two_per_cu && wgs > kCUs) ? 1.7 * (double)((wgs + 2 * kCUs - 1) / (2 * kCUs))
			                                                 : (double)((wgs + kCUs - 1) / kCUs);
			const double cost = rounds * (c + 6) * own;
			if (cost <= best_cost) {
				best_cost = cost;
				best = TuneChoice{2, ty, tz, c, body};
			}
		}
	}
	return best;
}

// Periodic 3-D grain growth and Zener pinning (2 or 4 fields; 8 in FP32 from
// 2^22 nodes): the plane march two steps per pass (body 12) where its 64-node
// tile rows fit the last axis (padding at most an eighth of it): 8 x 64 tiles
// (one node and its halo per thread, 704 threads), 64-plane chunks halved
// until a launch has 256 workgroups per CU that fit (two for 2 fields, one
// otherwise by registers): 256^3 x 2 FP64 81.0 us per step against 117.0 for
// the one-step march, x 4 FP64 178.6 (239.6), x 4 FP32 111.8 (125.2), x 8 FP32
// 222.0 (253.3); Zener x 2 FP32 34.7 (54.8), x 4 107.0 (122.4); 192^3 x 8 FP32
// 109.1 (125.6); 128^3 x 2 FP32 8.6 (12.2), x 4 FP64 24.6 (27.4); 64^3 x 4
// FP32 5.6 (7.1). 128^3 x 8 FP32 gains nothing (29.5 against 28.6), and 8 FP64
// fields fit the LDS on 8 x 32 tiles only (256^3: 488.5 against 481.0): those
// stay on the one-step march.
// Allen-Cahn (the last two steps of a call, pass_choice): 16 x 64 or 32 x 64
// tiles and the chunk from the cost model of two_step_choice: rounds x (chunk +
// 3 planes) x owned points per thread (16 x 64: 1188 on 640 threads, two
// workgroups per CU in rounds of 512 each 1.7 times as long; 32 x 64: 2244 on
// 768, one per CU).
static bool march2_choice(const Geom& g, int prec, int model, TuneChoice* out)
{
	constexpr int kCUs = 256;
	if (!all_periodic(g) || (prec != MMSPX_F64 && prec != MMSPX_F32)) return false;
	if (model != MMSPX_AC && model != MMSPX_GG && model != MMSPX_ZENER) return false;
	const int nz = g.n[2], pad = (nz + 63) / 64 * 64 - nz;
	if (pad * 8 > nz) return false;
	if (model == MMSPX_AC) {
		double best_cost = 1e300;
		for (int ty : {16, 32}) {
			const double own = ty == 16 ? 1188.0 / 640 : 2244.0 / 768;
			const int64_t tiles = (int64_t)((g.n[1] + ty - 1) / ty) * ((nz + 63) / 64);
			for (int c : {4, 8, 16, 32, 64}) {
				const int64_t wgs = tiles * ((g.n[0] + c - 1) / c);
				const double rounds = (ty == 16 && wgs > kCUs) ? 1.7 * (double)((wgs + 2 * kCUs - 1) / (2 * kCUs))
				                                               : (double)((wgs + kCUs - 1) / kCUs);
				const double cost = rounds * (c + 3) * own;
				if (cost < best_cost) {
					best_cost = cost;
					*out = TuneChoice{2, ty, 64, c, 12};
				}
			}
		}
		return true;
	}
	const int q = g.fields;
	if (!(q == 2 || q == 4 || (q == 8 && prec == MMSPX_F32 && g.nodes >= ((int64_t)1 << 22)))) return false;
	const int per_cu = q == 2 ? 2 : 1;
	const int64_t tiles = (int64_t)((g.n[1] + 7) / 8) * ((nz + 63) / 64);
	int chunk = 64;
	while (chunk > 4 && tiles * ((g.n[0] + chunk - 1) / chunk) < (int64_t)kCUs * per_cu) chunk /= 2;
	*out = TuneChoice{2, 8, 64, chunk, 12};
	return true;
}

static TuneChoice search_default(const Geom& g, int prec, int model)
{
	TuneChoice t;
	if (steps2d_choice(g, prec, model, &t)) return t;
	if (fields2d_choice(g, prec, model, &t)) return t;
	if (fmarch_choice(g, prec, model, &t)) return t;
	if (march4_choice(g, prec, model, &t)) return t;
	return one_step_choice(g, prec, model);
}

// The search looks at up to 434 tiles and chunks (8 us on a host core for 3-D
// Allen-Cahn and Cahn-Hilliard, 1 us in 2-D), in front of every call: one step
// of 64^3 Allen-Cahn took 10.2 us, host-bound, and takes 5.8. So a thread keeps
// its last eight answers, by what they depend on (the extents, boundaries,
// fields, form and model; nothing of a state or its buffers).
TuneChoice default_choice(const Geom& g, int prec, int model)
{
	struct Plan {
		int key[13];
		TuneChoice t;
	};
	thread_local Plan plans[8];
	thread_local int count = 0, next = 0;
	const int key[13] = {g.dim,   g.n[0],  g.n[1],  g.n[2],  g.b0[0],  g.b0[1], g.b0[2],
	                     g.b1[0], g.b1[1], g.b1[2], g.fields, prec,    model};
	for (int k = 0; k < count; k++)
		if (std::memcmp(plans[k].key, key, sizeof key) == 0) return plans[k].t;
	Plan& p = plans[next];
	std::memcpy(p.key, key, sizeof key);
	p.t = search_default(g, prec, model);
	next = (next + 1) % 8;
	count = std::max(count, next == 0 ? 8 : next);
	return p.t;
}

// A multi-step pass cut short forms fewer levels on tiles made for all of them,
// so the steps left over at a call's end, and calls of fewer steps than a pass,
// go to a one- or two-step kernel where that takes less (us a call, cut pass and
// this):
// - 2-D periodic Allen-Cahn up to 2^20 nodes: temporal blocks, which take up to
//   eight steps in one launch: FP64 128^2 6 steps 8.6 and 6.0, 512^2 14.0 and 9.1
//   for 7, 1024^2 9.6 and 7.9 for one; four are a whole pass of four levels.
//   From 1300^2 the strips are faster throughout (one step 9.8 and 11.8).
// - one step of 2-D Allen-Cahn between walls, and two between 2^20 and 2^23
//   nodes: the wave strips (FP64 1024^2 8.7 and 5.6; FP32 2048^2 15.7 and 8.9,
//   two steps 19.5 and 17.1; two at 700^2 7.1 and 8.6, at 4096^2 42 and 45).
// - one step of 2-D Cahn-Hilliard: its wave strips (1024^2 FP64 8.4 and 6.5,
//   FP32 7.3 and 5.7; 2048^2 FP32 14.6 and 10.1).
// - one or two steps of 2-D grain growth and Zener pinning from 2^21 values (nodes
//   x fields): the split strips (512^2 x 32 FP32 one 21.2 and 16.4, two 29.3 and
//   22.9). Below, their rows a wave are a longer serial march than the cut pass
//   (at the end of a call of 48 steps: 64^2 x 32 FP32 one 6.2 and 12.8 us, 309 x
//   73 x 2 FP64 3.5 and 7.1).
// - one step of 3-D Allen-Cahn from 2^18 nodes: the plane march (FP64 256^3 69 and
//   45; FP32 41 and 24; below, after 48 steps, 48^3 FP64 4.8 and 5.8), in FP32 up
//   to 2^20 nodes on 16 x 32 tiles (64^3 5.8 against 7.0 on that march's own
//   default, 64 x 128 x 128 6.4 against 7.4); two, from 2^20 nodes: that march two
//   steps per pass where it fits (256^3 FP64 73 and 60, FP32 42 and 35).
// - one step of 3-D Cahn-Hilliard: march4_last_step_choice.
// - one step of 3-D grain growth and Zener pinning: the plane march (192^3 x 8
//   FP32 157 and 120, 256^3 x 8 392 and 243, 96^3 x 4 16.4 and 11.9), but for 8
//   fields in FP64 where its 64-node tile rows would be padded by more than an
//   eighth (150 x 203 x 97 130 and 152, 96^3 34 and 39).
TuneChoice pass_choice(const Geom& g, int prec, int model, const TuneChoice& full, int left)
{
	if (full.opt < 13 || full.opt > 17) return full;
	const int64_t nodes = g.nodes;
	if (g.dim == 2 && model == MMSPX_AC && all_periodic(g)) {
		const bool blocks = left < kTbMaxSteps && left != 4 && nodes <= ((int64_t)1 << 20);
		return blocks ? one_step_choice(g, prec, model) : full;
	}
	if (left >= fused_steps_per_launch(model, full)) return full;
	TuneChoice t = full;
	switch (full.opt) {
	case 13:
	case 14:
		if (left == 1 || (left == 2 && model == MMSPX_AC && nodes >= ((int64_t)1 << 20) && nodes < ((int64_t)1 << 23)))
			t = one_step_choice(g, prec, model);
		break;
	case 15:
		if (model == MMSPX_AC) {
			if (left == 1 && nodes >= ((int64_t)1 << 18))
				t = prec == MMSPX_F32 && nodes <= ((int64_t)1 << 20) ? TuneChoice{2, 16, 32, 4, 8} : one_step_choice(g, prec, model);
			else if (left == 2 && nodes >= ((int64_t)1 << 20) && !march2_choice(g, prec, model, &t)) t = full;
		} else if (!march4_last_step_choice(g, prec, full, &t)) {
			t = full;
		}
		break;
	case 16:
		if (left <= 2 && nodes * g.fields >= ((int64_t)1 << 21)) t = one_step_choice(g, prec, model);
		break;
	case 17: {
		const int pad = (g.n[2] + 63) / 64 * 64 - g.n[2];
		if (left == 1 && !(g.fields == 8 && prec == MMSPX_F64 && pad * 8 > g.n[2])) t = one_step_choice(g, prec, model);
		break;
	}
	}
	return t.variant == 2 ? t : full;
}

// The defaults where no multi-step kernel runs (the reference's float form, noise,
// other boundaries, other field counts, Ostwald ripening, multi-phase grain
// growth) and, by pass_choice, of a call's last steps. From sweeps of the
// candidates below on MI355X (the figures quoted are microseconds per step from
// those sweeps).
TuneChoice one_step_choice(const Geom& g, int prec, int model)
{
	if (!fused_supported(g, prec, model)) return TuneChoice{1, 0, 0, 0, 0};
	const int64_t nodes = g.nodes;
	// 3-D Allen-Cahn, model A, grain growth, Zener pinning and multi-phase
	// grain growth: the plane march.
	// 256^3 sweep (us per step): Allen-Cahn FP64 16 x 32 tiles with 32-plane
	// chunks 44.5 (6.0 TB/s; 8 x 64 45.0, 32 x 64 46.5, one thread per node
	// 93.5), FP32 32 x 64 with 16-plane chunks 24.6 (16 x 64 24.8; 32-plane
	// chunks 31.7); grain growth 8 fields 8 x 64 with 64-plane chunks, FP32
	// 252 (16 x 32 275, one thread per node 430), FP64 484 (935); Zener 4
	// fields FP32 122 (211). Chunks are halved until the launch has 512
	// workgroups (two per CU) or more.
	// Multi-phase grain growth is bound by its per-node arithmetic, not by
	// bytes: one-hot grains with 8 fields, 128^3 FP64 200 us per step on 8 x
	// 64 tiles with 16-plane chunks (256 workgroups; 206 with 8-plane chunks,
	// 374 with 32) against 253 for one thread per node, FP32 87 against 155;
	// at 64^3 one thread per node wins (41.5 against 54.1), so the march
	// starts at 2^21 nodes, with 16-plane chunks halved to no less than 8
	// until the launch has 256 workgroups.
	if (g.dim == 3 && model == MMSPX_GG_ANISO) {
		if (nodes < ((int64_t)1 << 21)) return TuneChoice{1, 0, 0, 0, 0};
		const int64_t tiles = (int64_t)((g.n[1] + 7) / 8) * ((g.n[2] + 63) / 64);
		int chunk = 16;
		while (chunk > 8 && tiles * ((g.n[0] + chunk - 1) / chunk) < 256) chunk /= 2;
		return TuneChoice{2, 8, 64, chunk, 8};
	}
	// Ostwald ripening: the two passes as marches, 8 x 64 tiles with 32-plane
	// chunks halved (to no less than 4) until a launch has 1024 workgroups:
	// 256^3 x 2 fields FP64 215 us per step against 340 for the generic
	// passes (FP32 121.5 against 172.6), 128^3 x 4 FP64 with 4-plane chunks
	// 40.4 against 57.4; below 2^20 nodes the generic passes win (the
	// example's 128 x 64 x 16 grid: 8.4 against 12.9)
	// Periodic with 2 fields and 64-node tile rows that pad the last axis by at
	// most an eighth: the one-pass march (body 12, w kept in LDS), 8 x 64
	// tiles with 64-plane chunks halved until a launch has 512 workgroups
	// (two per CU): 256^3 FP64 156.8 us per step against 213.7 for the two
	// marches, FP32 75.1 against 121.6; 128^3 FP64 24.0 against 28.7. With 3
	// or 4 fields its registers leave one workgroup per CU in FP64 (192^3 x 3
	// FP64 134.0 against 125.6; 128^3 x 4 FP64 40.0 against 40.3), so those
	// stay on the two marches.
	if (g.dim == 3 && model == MMSPX_OSTWALD) {
		if (nodes < ((int64_t)1 << 20)) return TuneChoice{1, 0, 0, 0, 0};
		const int64_t tiles = (int64_t)((g.n[1] + 7) / 8) * ((g.n[2] + 63) / 64);
		const int pad = (g.n[2] + 63) / 64 * 64 - g.n[2];
		if (g.fields == 2 && all_periodic(g) && (prec == MMSPX_F64 || prec == MMSPX_F32) && pad * 8 <= g.n[2]) {
			int c = 64;
			while (c > 4 && tiles * ((g.n[0] + c - 1) / c) < 512) c /= 2;
			return TuneChoice{2, 8, 64, c, 12};
		}
		int chunk = 32;
		while (chunk > 4 && tiles * ((g.n[0] + chunk - 1) / chunk) < 1024) chunk /= 2;
		return TuneChoice{2, 8, 64, chunk, 8};
	}
	TuneChoice two;
	if (g.dim == 3 && model != MMSPX_AC && march2_choice(g, prec, model, &two)) return two;
	if (g.dim == 3 && (model == MMSPX_AC || model == MMSPX_AC_NOISE || model == MMSPX_GG || model == MMSPX_ZENER)) {
		const bool scalar = model == MMSPX_AC || model == MMSPX_AC_NOISE;
		const int ty = scalar ? (prec == MMSPX_F64 ? 16 : 32) : 8;
		const int tz = scalar ? (prec == MMSPX_F64 ? 32 : 64) : 64;
		int chunk = scalar ? (prec == MMSPX_F64 ? 32 : 16) : 64;
		const int64_t tiles = (int64_t)((g.n[1] + ty - 1) / ty) * ((g.n[2] + tz - 1) / tz);
		while (chunk > 4 && tiles * ((g.n[0] + chunk - 1) / chunk) < 512) chunk /= 2;
		return TuneChoice{2, ty, tz, chunk, 8};
	}
	// Allen-Cahn, in the reference's float form and for the last steps of a call
	// (pass_choice): periodic grids take temporal blocks of 48 columns and 8
	// steps per pass (512^2: 2.05 us per step in FP64 against 4.58 us for one
	// thread per node). Block heights from a sweep of 8, 16, 32 rows (on 512,
	// 1024, 1024 threads) x 4, 8 steps, sides 256 to 4096: 16 rows up to 2^16
	// nodes (256^2 FP64 1.10 us, FP32 0.97), 32 rows above (512^2 FP64 1.48
	// against 1.57 with 16 rows and 1.69 with 8, FP32 1.26; 1024^2 3.09 and
	// 2.22; 2048^2 10.6 against 13.6 with 16 rows, FP32 6.95 against 9.41;
	// 4096^2 36.7 and 24.6 against 47.4 and 33.5).
	// Other boundaries and model A: the wave strips, 4-row chunks below 2^21
	// nodes, 8 below 2^23, 16 above (Neumann FP64: 1024^2 5.5 us per step
	// against 8.6 for one thread per node, 2048^2 12.6 against 16.5, 4096^2
	// 43.3 against 61.1; model A FP64 1024^2 7.7 us, 4096^2 60.8)
	const int wave_chunk = nodes < ((int64_t)1 << 21) ? 4 : nodes < ((int64_t)1 << 23) ? 8 : 16;
	const int tb_rows = nodes <= ((int64_t)1 << 16) ? 16 : 32;
	if (model == MMSPX_AC)
		return all_periodic(g) ? TuneChoice{2, tb_rows, kTbCols, 8, 3} : TuneChoice{2, 1, kWaveCols, wave_chunk, 2};
	if (model == MMSPX_AC_NOISE) return TuneChoice{2, 1, kWaveCols, wave_chunk, 2};
	// multi-phase grain growth (one-hot grains, 8 fields): 2-row chunks below
	// 2^21 nodes (1024^2 FP64 28.5 us per step against 32.0 with 4 rows, 33.3
	// with 8 and 77.3 for one thread per node; 512^2 12.2, 13.7 and 17.6), 8
	// rows above (2048^2 FP64 132 us, FP32 53.4: within 6 % of the best of 2..16)
	if (model == MMSPX_GG_ANISO) return TuneChoice{2, 1, kWaveCols, nodes < ((int64_t)1 << 21) ? 2 : 8, 2};
	// Ostwald ripening (4 fields): with the row rings, 4-row chunks below 2^21
	// nodes (1024^2 FP64 17.0 us per step against 18.0 with 8 rows; the
	// generic two passes: 28 us), 8 above (2048^2 FP64 51.1 against 52.2, FP32
	// 27.2 against 28.5)
	if (model == MMSPX_OSTWALD) return TuneChoice{2, 1, kChWaveOut, nodes < ((int64_t)1 << 21) ? 4 : 8, 0};
	// Grain growth and Zener pinning with 8, 16 or 32 fields: the split strips.
	// Below 2^21 nodes four waves per strip (a quarter of the fields each)
	// with 8-row chunks in FP32 and 16 in FP64; above, two waves with 64-row
	// chunks. Measured per step: 2048^2 x 32 FP32 233.7 us against 248.2 for
	// the wave strips (32-row chunks) and 388 for one thread per node; 2048^2
	// x 32 FP64 459.5 against 835.9 for the 8 x 64 tile; 2048^2 x 16 Zener
	// FP32 115.4 against 118.3; 512^2 x 32 FP32 15.7 against 20.3 on two
	// waves; 512^2 x 8 FP32 7.9 against 9.4 for one thread per node; 1024^2 x
	// 16 FP64 47.1 against 82.0.
	// Periodic grids take the split strips two steps per pass on four waves
	// (body 10): 2048^2 x 32 FP32 149.6 us per step with 16-row chunks
	// against 241.2 for the one-step split strips, FP64 275.0 with 32-row
	// chunks against 465.6; 2048^2 x 16 Zener FP32 73.0 against 117.3;
	// 1024^2 x 32 FP32 30.7 with 8-row chunks against 49.6; 512^2 x 8 FP32 5.0
	// against 8.1; 1024^2 x 8 FP64 15.8 against 24.7 (two waves: 1-8 % slower).
	if ((model == MMSPX_GG || model == MMSPX_ZENER) && (g.fields == 8 || g.fields == 16 || g.fields == 32)) {
		if (all_periodic(g))
			return TuneChoice{2, 1, kChWaveOut, nodes < ((int64_t)1 << 21) ? 8 : prec == MMSPX_F64 ? 32 : 16, 10};
		if (nodes < ((int64_t)1 << 21)) return TuneChoice{2, 1, kWaveCols, prec == MMSPX_F64 ? 16 : 8, 5};
		return TuneChoice{2, 1, kWaveCols, 64, 4};
	}
	// Grain growth and Zener pinning with 2 or 4 fields: the wave strips,
	// 4-row chunks below 2^21 nodes, 16 above (2 and 4 fields, 512^2 .. 4096^2,
	// FP32 and FP64: 1.4 to 1.9 times faster than one thread per node; 1024^2
	// x 4 FP32 8.0 us against 12.0, 4096^2 x 4 FP64 219.7 against 354.1)
	// Periodic: two steps per pass on one wave per strip (body 11), 8-row
	// chunks below 2^21 nodes and 16 above (2048^2 x 2 FP64 13.8 us per step
	// against 22.2 for the wave strips, 2048^2 x 4 FP32 14.4 against 23.0,
	// 1024^2 x 4 FP64 9.7 against 14.1, 512^2 x 2 FP64 3.2 against 4.6; Zener
	// 2048^2 x 4 FP32 13.5 against 22.5)
	if ((model == MMSPX_GG || model == MMSPX_ZENER) && all_periodic(g))
		return TuneChoice{2, 1, kChWaveOut, nodes < ((int64_t)1 << 21) ? 8 : 16, 11};
	if (model == MMSPX_GG || model == MMSPX_ZENER)
		return TuneChoice{2, 1, kWaveCols, nodes < ((int64_t)1 << 21) ? 4 : 16, 2};
	// 2-D Cahn-Hilliard: wave strips (1024^2 FP64 6.8 us per step against 13.5
	// us for the LDS row strips; 4096^2 FP64 42.4 us against 69 us). Chunks
	// from a sweep of 3..32 rows with the row ring: 3 below 2^17 nodes (256^2
	// FP64 3.0 us against 3.2 with 4 rows), 4 below 2^21 (1024^2 6.8, FP32
	// 5.2), then 16 in FP64 (2048^2 15.6 against 16.5 with 8; 4096^2 42.4) and
	// 8 in FP32 below 2^23 (2048^2 11.3 against 11.5), 16 above (4096^2 30.7)
	if (g.dim == 2) {
		const int c = nodes < ((int64_t)1 << 17)                          ? 3
		              : nodes < ((int64_t)1 << 21)                        ? 4
		              : nodes < ((int64_t)1 << 23) && prec != MMSPX_F64 ? 8
		                                                                  : 16;
		return TuneChoice{2, 1, kChWaveOut, c, 0};
	}
	// other boundaries than periodic: the register queues (8 x 32 tiles on
	// 256 threads below 2^24 nodes, 32 x 64 on 768 above)
	if (!all_periodic(g))
		return nodes < (int64_t)16 * 64 * 32 * 512 ? TuneChoice{2, 8, 32, 16, 1}
		                                            : TuneChoice{2, 32, 64, prec == MMSPX_F64 ? 32 : 16, 2};
	if (model != MMSPX_CH_NOISE && (prec == MMSPX_F64 || prec == MMSPX_F32)) return two_step_choice(g, prec);
	if (nodes < (int64_t)16 * 64 * 32 * 512) return TuneChoice{2, 8, 32, 16, 0};
	// 256^3: register queues on 32 x 64 tiles with 768 threads. FP64 with
	// 32-plane chunks, one workgroup per CU (52.3 us per step, against 53.0
	// with 512 or 1024 threads, 55.9 with 16-plane chunks, 54.4 for 16 x 64
	// tiles with 24-plane chunks, 64-75 us for chunks of 12, 20 and 24 that
	// leave CUs with uneven work); FP32 with 16-plane chunks, two per CU
	// (31.3 us, against 31.7 with 512 threads, 35.0 with 32-plane chunks)
	// model B (noise, FP64): 32-plane chunks on 1024 threads (95.9 us against
	// 97.6 with 768 in one sweep, 92.6 against 91.6 in another: the two are
	// within the noise; 16-plane chunks take 99-107 us)
	if (model == MMSPX_CH_NOISE && prec == MMSPX_F64) return TuneChoice{2, 32, 64, 32, 3};
	return TuneChoice{2, 32, 64, prec == MMSPX_F64 ? 32 : 16, 2};
}

bool multi_step_body_runs(const Geom& g, int prec, int model, int body)
{
	switch (body) {
	case 13:
	case 14: return steps2d_supported(g, prec, model);
	case 15: return march4_supported(g, prec, model);
	case 16: return fields2d_supported(g, prec, model);
	case 17: return fmarch_supported(g, prec, model);
	}
	return true;
}

bool tile_known(const Geom& g, const TuneChoice& t)
{
	if (t.chunk < 2 || t.chunk > 4096) return false;
	if (g.dim == 3 && t.opt == 17)
		return fmarch_tile_known(MMSPX_F64, g.fields, t.ty, t.tz) || fmarch_tile_known(MMSPX_F32, g.fields, t.ty, t.tz);
	if (g.dim == 3 && t.opt == 15)
		return march4_tile_known(MMSPX_F64, t.ty, t.tz) || march4_tile_known(MMSPX_F32, t.ty, t.tz);
	if (g.dim == 3)
		return (t.ty == 8 && t.tz == 64) || (t.ty == 16 && t.tz == 64) || (t.ty == 32 && t.tz == 64) ||
		       (t.ty == 8 && t.tz == 32) || (t.ty == 4 && t.tz == 128) || (t.ty == 32 && t.tz == 32) ||
		       (t.ty == 16 && t.tz == 32);
	if (g.dim == 2 && (t.opt == 13 || t.opt == 14 || t.opt == 16))
		return t.ty == 1 && t.tz == (t.opt == 13 ? kSteps8Cols : kSteps4Cols);
	if (g.dim == 2)
		return (t.ty == 1 && (t.tz == 64 || t.tz == 128 || t.tz == 256 || t.tz == kChWaveOut)) ||
		       ((t.ty == 8 || t.ty == 16 || t.ty == 32) && t.tz == kTbCols && t.chunk <= kTbMaxSteps) ||
		       (t.opt == 1 && (t.ty == 8 || t.ty == 16) && t.tz == 64);
	return false;
}

int tile_candidates(const Geom& g, int prec, int model, TuneChoice* out, int max)
{
	int n = 0;
	auto add = [&](int ty, int tz, int chunk, int opt) {
		if (n < max) out[n++] = TuneChoice{2, ty, tz, chunk, opt};
	};
	const bool ch = ch_family(model);
	// the default itself (its tile and chunk come from a cost model, not from the
	// lists below), so that tuning never ends on a slower one
	const TuneChoice def = default_choice(g, prec, model);
	if (def.variant == 2) add(def.ty, def.tz, def.chunk, def.opt);
	// Allen-Cahn and Cahn-Hilliard, 3-D periodic: the four-level march
	n += march4_candidates(g, prec, model, out + n, max - n);
	// grain growth and Zener pinning, periodic: several steps per pass
	n += fmarch_candidates(g, prec, model, out + n, max - n);
	if (fields2d_supported(g, prec, model))
		for (int c : {8, 16, 32, 64, 128}) add(1, kSteps4Cols, c, 16);
	if (g.dim == 2 && model == MMSPX_OSTWALD) {
		for (int c : {4, 8, 16, 32, 64}) add(1, kChWaveOut, c, 0);
		return n;
	}
	if (g.dim == 2 && model == MMSPX_GG_ANISO) {
		for (int c : {2, 4, 8, 16, 32}) add(1, kWaveCols, c, 2);
		return n;
	}
	const bool split = (model == MMSPX_GG || model == MMSPX_ZENER) && (g.fields == 8 || g.fields == 16 || g.fields == 32);
	if (g.dim == 2 && (model == MMSPX_AC_NOISE || model == MMSPX_ZENER)) {
		// model A and Zener pinning: wave strips, and the split strips
		for (int c : {8, 12, 16, 24, 32}) add(1, kWaveCols, c, 2);
		if (split)
			for (int c : {8, 16, 32, 64})
				for (int body = 4; body <= 5; body++) add(1, kWaveCols, c, body);
		if (split && model == MMSPX_ZENER && all_periodic(g))
			for (int c : {8, 16, 32, 64})
				for (int body = 9; body <= 10; body++) add(1, kChWaveOut, c, body);
		if (model == MMSPX_ZENER && (g.fields == 2 || g.fields == 4 || g.fields == 8) && all_periodic(g))
			for (int c : {8, 16, 32, 64}) add(1, kChWaveOut, c, 11);
		return n;
	}
	if (g.dim == 3 && !ch) {
		// the plane march: Allen-Cahn on four tiles, the vector models on two
		const bool scalar = model == MMSPX_AC || model == MMSPX_AC_NOISE;
		for (int c : {16, 32, 64}) {
			add(8, 64, c, 8);
			add(16, 32, c, 8);
			if (scalar) {
				add(16, 64, c, 8);
				add(32, 64, c, 8);
			}
		}
		// two steps per pass on periodic grids (Allen-Cahn, grain growth,
		// Zener pinning; the 8-field FP64 planes fit the LDS on 8 x 32 only)
		// (Ostwald ripening: the one-pass march)
		const bool two = all_periodic(g) && model != MMSPX_AC_NOISE && model != MMSPX_GG_ANISO &&
		                 (prec == MMSPX_F64 || prec == MMSPX_F32);
		if (two)
			for (int c : {8, 16, 32, 64}) {
				if (scalar) {
					add(16, 64, c, 12);
					add(32, 64, c, 12);
				} else if (g.fields == 8 && prec == MMSPX_F64) {
					add(8, 32, c, 12);
				} else {
					add(8, 64, c, 12);
					add(16, 32, c, 12);
				}
			}
		return n;
	}
	const bool edges = !all_periodic(g);  // Cahn-Hilliard: the bodies that map non-periodic sides
	if (g.dim == 3) {
		const int tiles[4][2] = {{16, 64}, {8, 64}, {8, 32}, {4, 128}};
		for (auto& t : tiles)
			for (int c : {16, 32, 64})
				for (int opt = edges ? 1 : 0; opt < 2; opt++) add(t[0], t[1], c, opt);
		// 32 x 64: register queues only (the LDS rings would leave one
		// workgroup per CU), on 512 and 768 threads
		for (int c : {12, 16, 22, 32})
			for (int body = 1; body <= 3; body++) add(32, 64, c, body);
		for (int c : {20, 22, 24}) add(16, 64, c, 1);
		// two steps per pass (deterministic chemical potentials, periodic grids)
		if ((model == MMSPX_CH || model == MMSPX_CH_DW) && !edges)
			for (int c : {6, 8, 12, 16, 24, 32, 48, 64}) {
				add(32, 64, c, 6);
				add(32, 32, c, 7);
			}
	} else if (g.dim == 2) {
		// LDS-row strips (Cahn-Hilliard: both tile bodies; non-periodic: the register queues)
		for (int tz : {64, 128, 256})
			for (int c : {16, 32, 64, 128})
				for (int opt = (ch && edges) ? 1 : 0; opt < (ch ? 2 : 1); opt++) add(1, tz, c, opt);
		// Cahn-Hilliard wave strips
		if (ch)
			for (int c : {8, 16, 32, 64}) add(1, kChWaveOut, c, 0);
		// grain growth: 2-D tiles
		if (model == MMSPX_GG && g.fields > 1) {
			add(8, 64, 8, 1);
			add(16, 64, 16, 1);
		}
		// Allen-Cahn and grain growth: wave strips, where compiled
		const bool wave = model == MMSPX_AC || (model == MMSPX_GG && (g.fields < 32 || prec != MMSPX_F64));
		if (wave)
			for (int c : {8, 12, 16, 24, 32}) add(1, kWaveCols, c, 2);
		if (split)
			for (int c : {8, 16, 32, 64})
				for (int body = 4; body <= 5; body++) add(1, kWaveCols, c, body);
		// periodic: the split strips two steps per pass (one wave for 2, 4, 8 fields)
		if (split && all_periodic(g))
			for (int c : {8, 16, 32, 64})
				for (int body = 9; body <= 10; body++) add(1, kChWaveOut, c, body);
		if ((model == MMSPX_GG || model == MMSPX_ZENER) && (g.fields == 2 || g.fields == 4 || g.fields == 8) &&
		    all_periodic(g))
			for (int c : {8, 16, 32, 64}) add(1, kChWaveOut, c, 11);
		// Allen-Cahn and Cahn-Hilliard: several steps per pass in registers
		if (steps2d_supported(g, prec, model))
			for (int c : {4, 8, 16, 32, 64}) {
				add(1, kSteps8Cols, c, 13);
				add(1, kSteps4Cols, c, 14);
			}
		// periodic Allen-Cahn: temporal blocks (chunk = steps per pass)
		if (model == MMSPX_AC && all_periodic(g))
			for (int tx : {8, 16, 32})
				for (int k : {4, 8}) add(tx, kTbCols, k, 3);
	}
	return n;
}

bool fused_needs_plane(const Geom& g, int model, const TuneChoice& t)
{
	return model == MMSPX_OSTWALD && g.dim == 3 && t.opt != 12;
}

int fused_steps_per_launch(int model, const TuneChoice& t)
{
	if ((model == MMSPX_AC || model == MMSPX_CH || model == MMSPX_CH_DW) && (t.opt == 13 || t.opt == 14))
		return steps2d_max_steps(model, t.opt);
	if ((model == MMSPX_AC || model == MMSPX_CH || model == MMSPX_CH_DW) && t.opt == 15) return march4_max_steps(model);
	if ((model == MMSPX_GG || model == MMSPX_ZENER) && t.opt == 16) return kFieldsSteps;
	if ((model == MMSPX_GG || model == MMSPX_ZENER) && t.opt == 17) return fmarch_steps(t);
	if (model == MMSPX_AC && t.tz == kTbCols) return std::max(1, std::min(t.chunk, kTbMaxSteps));
	if ((model == MMSPX_CH || model == MMSPX_CH_DW) && (t.opt == 6 || t.opt == 7)) return 2;
	if ((model == MMSPX_GG || model == MMSPX_ZENER) && t.opt >= 9 && t.opt <= 11) return 2;
	if ((model == MMSPX_AC || model == MMSPX_GG || model == MMSPX_ZENER) && t.opt == 12) return 2;
	return 1;
}

int launch_fused_step(const Geom& g, int prec, const ModelParams& p, const void* a, void* b, hipStream_t st,
                      const TuneChoice& t, int nsteps, int64_t* launches, void* aux)
{
	if (prec != MMSPX_F64 && prec != MMSPX_F32 && prec != MMSPX_F32REF) return fail(MMSPX_EINVAL, "unknown precision");
	const int chunk = t.chunk > 0 ? t.chunk : 32;
	const bool f64 = prec == MMSPX_F64;
	int rc;
	if (g.dim == 2 && (t.opt == 13 || t.opt == 14)) rc = launch_steps2d(g, prec, p, a, b, st, t.opt, chunk, nsteps);
	else if (g.dim == 2 && t.opt == 16) rc = launch_fields2d(g, prec, p, a, b, st, chunk, nsteps);
	else if (g.dim == 3 && t.opt == 17) rc = launch_fmarch(g, prec, p, a, b, st, t, nsteps);
	else if (g.dim == 3 && t.opt == 15) rc = launch_march4(g, prec, p, a, b, st, t, nsteps);
	else if (ac_family(p.model)) rc = (f64 ? launch_fused_ac_f64 : launch_fused_ac_f32)(g, prec, p, a, b, st, t, nsteps, aux);
	else if (ch_family(p.model)) rc = (f64 ? launch_fused_ch_f64 : launch_fused_ch_f32)(g, prec, p, a, b, st, t, nsteps, aux);
	else if (p.model == MMSPX_GG || p.model == MMSPX_ZENER)
		rc = (f64 ? launch_fused_gg_f64 : launch_fused_gg_f32)(g, prec, p, a, b, st, t, nsteps, aux);
	else rc = (f64 ? launch_fused_rest_f64 : launch_fused_rest_f32)(g, prec, p, a, b, st, t, nsteps, aux);
	if (rc == 0) *launches += 1;
	return rc;
}

}  // namespace mmspx
