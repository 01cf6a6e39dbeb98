// kernels_march4.hip -- the 3-D four-level march (march4.hpp): its FP64 form,
// dispatch and tile choice (tile body 15).
#include <algorithm>

#include "march4_launch.hpp"

namespace mmspx {

int launch_march4_f32(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, const TuneChoice& t,
                      int nsteps);

bool march4_supported(const Geom& g, int prec, int model)
{
	if (g.dim != 3 || (prec != MMSPX_F64 && prec != MMSPX_F32)) return false;
	if (model != MMSPX_AC && model != MMSPX_CH && model != MMSPX_CH_DW) return false;
	// byte offsets inside a plane are 32 bits
	if ((int64_t)g.n[1] * g.n[2] >= (int64_t)1 << 28) return false;
	for (int k = 0; k < 3; k++)
		if (g.b0[k] != MMSPX_PERIODIC || g.b1[k] != MMSPX_PERIODIC) return false;
	return true;
}

int march4_max_steps(int model) { return model == MMSPX_AC ? 4 : 2; }

// the last two have a wave's lanes along axis 2 (wmarch4.hpp)
static const int kTiles[2][7][2] = {{{26, 52}, {16, 64}, {32, 32}, {16, 32}, {16, 16}, {26, 56}, {42, 56}},
                                    {{32, 64}, {26, 52}, {32, 32}, {16, 32}, {16, 16}, {26, 56}, {30, 56}}};

bool march4_tile_known(int prec, int ty, int tz)
{
	for (auto& t : kTiles[prec == MMSPX_F64 ? 0 : 1])
		if (t[0] == ty && t[1] == tz) return true;
	return false;
}

// Tile and chunk by a cost model: a workgroup of a chunk of c planes takes
// c + 6 iterations (the march starts three planes early and ends three late);
// tau is the time of one iteration when 1, 2, .. workgroups share a CU
// (microseconds, Cahn-Hilliard; the last entry is how many fit), a launch
// takes full rounds of 256 CUs and one of what is left. Fitted to sweeps of
// chunks of 3 to 64 planes on 18 grids from 32^3 to 320^3, odd ones among
// them; it picks the best measured or within 5 % of it. Against the one- and
// two-step marches and register queues before (us per step): Allen-Cahn FP64
// 64^3 4.4 -> 3.3, 150 x 203 x 97 17.4 -> 6.8, 256^3 31.6 -> 23.7; FP32 150 x
// 203 x 97 12.2 -> 4.8, 256^3 19.0 -> 13.3; Cahn-Hilliard FP64 64^3 8.0 ->
// 5.6, 128^3 10.4 -> 9.6, 150 x 203 x 97 19.3 -> 10.6, 256^3 46.4 -> 38.6;
// FP32 150 x 203 x 97 13.9 -> 8.0, 256^3 29.1 -> 22.3. The tiles with lanes
// along axis 2 are the fastest from about 96^3 on; Allen-Cahn in FP32, where
// they save least, takes them as 9 % slower (192^3 26 x 56 tiles 8.0 us, 32 x
// 64 7.2; Cahn-Hilliard 13.0 and 13.1).
// us of one launch: `wgs` workgroups of c + 6 iterations, ta[n-1] us each with n to a CU
static double march_time(int64_t wgs, int c, const double* ta)
{
	int cap = 0;
	while (cap < 6 && ta[cap] > 0.0) cap++;
	const int64_t round = 256 * cap, rest = wgs % round;
	return (c + 6) * ((double)(wgs / round) * ta[cap - 1] + (rest ? ta[(int)((rest + 255) / 256) - 1] : 0.0));
}

static int64_t march_wgs(const Geom& g, int ty, int tz, int c)
{
	return (int64_t)((g.n[1] + ty - 1) / ty) * ((g.n[2] + tz - 1) / tz) * ((g.n[0] + c - 1) / c);
}

static const double tau[2][7][6] = {
    {{1.45}, {1.36}, {1.36}, {1.00, 1.51}, {0.92, 1.10, 1.30, 1.51}, {1.30}, {1.94}},
    {{1.31}, {1.08, 1.64}, {1.05, 1.41}, {0.79, 1.00, 1.26, 1.52}, {0.77, 0.86, 0.96, 1.06, 1.16, 1.26}, {0.97, 1.39}, {1.10, 1.62}}};

// the chunk of least time on tile k; us receives that time
static TuneChoice march_best_chunk(const Geom* const* g, int count, int prec, int model, int k, double* us)
{
	const int f = prec == MMSPX_F64 ? 0 : 1, ty = kTiles[f][k][0], tz = kTiles[f][k][1];
	TuneChoice out{2, ty, tz, 8, 15};
	*us = 1e300;
	for (int c = 3; c <= 64; c += count > 1 && c >= 8 ? 4 : 1) {
		int64_t wgs = 0;
		for (int m = 0; m < count; m++) wgs += march_wgs(*g[m], ty, tz, c);
		const double t = march_time(wgs, c, tau[f][k]) * (k >= 5 && f == 1 && model == MMSPX_AC ? 1.09 : 1.0);
		if (t < *us) {
			*us = t;
			out.chunk = c;
		}
	}
	return out;
}

static TuneChoice march_best(const Geom* const* g, int count, int prec, int model, int tiles)
{
	TuneChoice out{};
	double us = 1e300;
	for (int k = 0; k < tiles; k++) {
		double t;
		const TuneChoice c = march_best_chunk(g, count, prec, model, k, &t);
		if (t < us) {
			us = t;
			out = c;
		}
	}
	return out;
}

// every tile with the model's chunk, half of it and twice it
int march4_candidates(const Geom& g, int prec, int model, TuneChoice* out, int max)
{
	int n = 0;
	if (!march4_supported(g, prec, model)) return 0;
	const Geom* one = &g;
	for (int k = 0; k < 7; k++) {
		double us;
		const TuneChoice t = march_best_chunk(&one, 1, prec, model, k, &us);
		for (int c : {t.chunk / 2, t.chunk, 2 * t.chunk})
			if (c >= 2 && n < max) out[n++] = TuneChoice{2, t.ty, t.tz, c, 15};
	}
	return n;
}

TuneChoice march4_choice_many(const Geom* const* g, int count, int prec)
{
	return march_best(g, count, prec, MMSPX_CH, 5);  // the tiles the batch kernels are built for
}

bool march4_choice(const Geom& g, int prec, int model, TuneChoice* out)
{
	if (!march4_supported(g, prec, model)) return false;
	const Geom* one = &g;
	*out = march_best(&one, 1, prec, model, 7);
	return true;
}

int launch_march4(const Geom& g, int prec, const ModelParams& p, const void* a, void* b, hipStream_t st,
                  const TuneChoice& t, int nsteps)
{
	if (!march4_supported(g, prec, p.model))
		return fail(MMSPX_EUNSUPPORTED, "the four-level march takes periodic 3-D Allen-Cahn and Cahn-Hilliard grids in "
		                                "the MMSPX_F64 and MMSPX_F32 forms");
	if (t.chunk < 1 || nsteps < 1) return fail(MMSPX_EINVAL, "bad chunk or step count");
	return prec == MMSPX_F64 ? launch_march4_prec<MMSPX_F64>(g, p, a, b, st, t, nsteps)
	                         : launch_march4_f32(g, p, a, b, st, t, nsteps);
}

// A last single Cahn-Hilliard step: the march's short pass (two of its levels;
// 0.84 of a whole pass in FP64, 0.92 in FP32) or body 2, the register queues on
// 32 x 64 tiles, which run in rounds of one workgroup a CU in FP64, of two in
// FP32. us, short pass and body 2: FP64 192^3 33 and 48, 224^3 43 and 51, 240^3
// 54 and 53, 256^3 66 and 59, 320^3 131 and 145; FP32 176^3 22 and 21, 192^3 25
// and 22, 224^3 30 and 32, 256^3 44 and 36, 320^3 77 and 65.
bool march4_last_step_choice(const Geom& g, int prec, const TuneChoice& full, TuneChoice* out)
{
	const int f = prec == MMSPX_F64 ? 0 : 1;
	int k = 0;
	while (k < 6 && !(kTiles[f][k][0] == full.ty && kTiles[f][k][1] == full.tz)) k++;
	const double march = (f ? 0.92 : 0.84) * march_time(march_wgs(g, full.ty, full.tz, full.chunk), full.chunk, tau[f][k]);
	*out = TuneChoice{2, 32, 64, f ? 16 : 32, 2};
	// fitted to the figures above: a round of w workgroups
	auto round_us = [&](double w) {
		return w <= 0.0 ? 0.0 : f == 0 ? 47.0 + 12.5 * w / 256.0 : w <= 256.0 ? 21.0 + 1.5 * w / 256.0 : 22.0 + 14.0 * w / 512.0;
	};
	const int64_t wgs = march_wgs(g, out->ty, out->tz, out->chunk), full_round = f ? 512 : 256;
	const double queues = (double)(wgs / full_round) * round_us((double)full_round) + round_us((double)(wgs % full_round));
	return queues < march;
}

// The body mmspx_get_tile reports for a default the four-level march runs: the
// pass it takes the place of (7 and 12 several steps per pass, 8 the plane
// march, which Allen-Cahn reports where 64-node tile rows would pad the last
// axis by more than an eighth).
int march4_reported_body(const Geom& g, int model)
{
	if (model != MMSPX_AC) return 7;
	const int pad = (g.n[2] + 63) / 64 * 64 - g.n[2];
	return pad * 8 <= g.n[2] ? 12 : 8;
}

}  // namespace mmspx
