// kernels_fmarch.hip -- the 3-D field march (fmarch.hpp): dispatch and tile
// choice (tile body 17).
#include <algorithm>

#include "core.hpp"

namespace mmspx {

int launch_fmarch_f32_gg(const Geom&, const ModelParams&, const void*, void*, hipStream_t, const TuneChoice&, int);
int launch_fmarch_f32_zener(const Geom&, const ModelParams&, const void*, void*, hipStream_t, const TuneChoice&, int);
int launch_fmarch_f64_gg(const Geom&, const ModelParams&, const void*, void*, hipStream_t, const TuneChoice&, int);
int launch_fmarch_f64_zener(const Geom&, const ModelParams&, const void*, void*, hipStream_t, const TuneChoice&, int);

bool fmarch_supported(const Geom& g, int prec, int model)
{
	if (g.dim != 3 || (prec != MMSPX_F64 && prec != MMSPX_F32)) return false;
	if (model != MMSPX_GG && model != MMSPX_ZENER) return false;
	if (g.fields != 2 && g.fields != 4 && g.fields != 8) return false;
	// row starts inside a plane are 32 bits
	if ((int64_t)g.n[1] * g.n[2] >= (int64_t)1 << 28) return false;
	for (int k = 0; k < 3; k++)
		if (g.b0[k] != MMSPX_PERIODIC || g.b1[k] != MMSPX_PERIODIC) return false;
	return true;
}

// Tiles with their cost: a pass takes t0 plus, for every round of 256
// workgroups (one fills a CU), `plane` microseconds for each of the chunk's
// planes and the 2 (L - 1) its march starts and ends with; or, where that is
// longer, what the planes it reads and writes take at `tbs` TB/s.
struct FieldTile {
	int prec, fields, ty, tz;
	double t0, plane, tbs;
};
static const FieldTile kFieldTiles[] = {
    {MMSPX_F32, 8, 12, 58, 2.3, 3.66, 4.0}, {MMSPX_F32, 8, 22, 60, 0.6, 4.47, 4.6}, {MMSPX_F32, 4, 18, 56, 0.4, 3.67, 2.9},
    {MMSPX_F32, 4, 28, 58, 2.4, 3.80, 3.8}, {MMSPX_F32, 2, 26, 56, 1.6, 2.65, 2.7}, {MMSPX_F64, 8, 8, 60, 1.3, 3.19, 5.4},
    {MMSPX_F64, 8, 10, 60, 1.1, 3.88, 5.1}, {MMSPX_F64, 4, 22, 60, 0.8, 3.91, 5.1}, {MMSPX_F64, 4, 12, 58, 2.3, 3.38, 4.1},
    {MMSPX_F64, 2, 18, 56, 1.6, 3.21, 3.1}, {MMSPX_F64, 2, 28, 58, 2.1, 3.49, 4.0}};

bool fmarch_tile_known(int prec, int fields, int ty, int tz)
{
	for (const FieldTile& t : kFieldTiles)
		if (t.prec == prec && t.fields == fields && t.ty == ty && t.tz == tz) return true;
	return false;
}

TuneChoice fmarch_any_tile(int prec, int fields, int chunk)
{
	for (const FieldTile& t : kFieldTiles)
		if (t.prec == prec && t.fields == fields) return TuneChoice{2, t.ty, t.tz, chunk, 17};
	return TuneChoice{1, 0, 0, 0, 0};
}

// us per step of the one- and two-step plane marches (bodies 8 and 12) on 8 x
// 64 tiles: a launch's floor and a rate per node of the padded grid
static double plane_march_us(const Geom& g, int prec, int body)
{
	struct {
		int prec, fields, body;
		double t0, node;
	} static const table[] = {{MMSPX_F32, 8, 12, 0.0, 12.8}, {MMSPX_F32, 8, 8, 7.8, 11.2}, {MMSPX_F32, 4, 12, 4.4, 5.5},
	                          {MMSPX_F32, 4, 8, 5.9, 5.7},   {MMSPX_F32, 2, 12, 3.6, 2.5}, {MMSPX_F32, 2, 8, 5.3, 4.2},
	                          {MMSPX_F64, 8, 12, 9.8, 27.2}, {MMSPX_F64, 8, 8, 9.8, 27.2}, {MMSPX_F64, 4, 12, 6.3, 10.1},
	                          {MMSPX_F64, 4, 8, 7.2, 10.6},  {MMSPX_F64, 2, 12, 4.2, 4.6}, {MMSPX_F64, 2, 8, 5.5, 5.4}};
	const double nodes = (double)g.n[0] * ((g.n[1] + 7) / 8 * 8) * ((g.n[2] + 63) / 64 * 64);
	for (auto& t : table)
		if (t.prec == prec && t.fields == g.fields && t.body == body) return t.t0 + t.node * nodes * 1e-6;
	return 0.0;
}

// us of a pass on tile t with its best chunk
static double best_pass(const Geom& g, const FieldTile& t, TuneChoice* out)
{
	const int L = (64 - t.tz) / 2;
	const double node_bytes = (double)t.fields * (t.prec == MMSPX_F64 ? 8 : 4);
	const double plane_bytes = ((t.ty + 2 * L) * 64.0 + (double)t.ty * t.tz) * node_bytes;
	const int64_t tiles = (int64_t)((g.n[1] + t.ty - 1) / t.ty) * ((g.n[2] + t.tz - 1) / t.tz);
	double best = 1e300;
	auto take = [&](int c) {
		const int64_t wgs = tiles * ((g.n[0] + c - 1) / c);
		const int planes = c + 2 * (L - 1);
		const double work = t.plane * planes * (double)((wgs + 255) / 256);
		const double move = plane_bytes * planes * (double)wgs / (t.tbs * 1e6);
		const double us = t.t0 + std::max(work, move);
		if (us < best) {
			best = us;
			*out = TuneChoice{2, t.ty, t.tz, c, 17};
		}
	};
	for (int c = 3; c <= 16; c++) take(c);
	for (int n = 1; n <= 32; n++) {
		const int c = (g.n[0] + n - 1) / n;
		if (c > 16 && c <= 512) take(c);
	}
	return best;
}

// Tile and chunk by the cost above, where that is 7 % less than the plane
// marches take (both fitted to a sweep of 12 grids from 40 x 24 x 128 to 256^3,
// within 10 %). us per step, plane march and this: 256^3 x 8 FP32 212 and 167,
// FP64 451 and 337; x 4 FP32 106 and 81; 192^3 x 8 FP32 107 and 69; 150 x 203 x
// 97 x 8 FP32 60 and 32, FP64 152 and 71, x 2 FP32 22 and 11; 96^3 x 8 FP64 40
// and 23. The plane marches keep grids that fill their tiles while the launch
// is short or has few fields: 64^3 x 4 FP32 5.7 and 9.3, 128^3 x 4 14.6 and
// 16.9, 128^3 x 2 FP64 12.2 and 15.8.
bool fmarch_choice(const Geom& g, int prec, int model, TuneChoice* out)
{
	if (!fmarch_supported(g, prec, model)) return false;
	double best = 1e300;
	for (const FieldTile& t : kFieldTiles) {
		if (t.prec != prec || t.fields != g.fields) continue;
		TuneChoice c;
		const double us = best_pass(g, t, &c) / fmarch_steps(c);
		if (us < best) {
			best = us;
			*out = c;
		}
	}
	return best < 0.93 * plane_march_us(g, prec, one_step_choice(g, prec, model).opt == 12 ? 12 : 8);
}

int fmarch_candidates(const Geom& g, int prec, int model, TuneChoice* out, int max)
{
	int n = 0;
	if (!fmarch_supported(g, prec, model)) return 0;
	for (const FieldTile& t : kFieldTiles)
		if (t.prec == prec && t.fields == g.fields) {
			TuneChoice best;
			best_pass(g, t, &best);
			for (int c : {best.chunk, 4, 8, 16, 32, 64})
				if (n < max) out[n++] = TuneChoice{2, t.ty, t.tz, c, 17};
		}
	return n;
}

int launch_fmarch(const Geom& g, int prec, const ModelParams& p, const void* a, void* b, hipStream_t st,
                  const TuneChoice& tile, int nsteps)
{
	if (!fmarch_supported(g, prec, p.model))
		return fail(MMSPX_EUNSUPPORTED, "the field march takes periodic 3-D grain growth and Zener pinning with 2, 4 or 8 "
		                                "fields in the MMSPX_F64 and MMSPX_F32 forms");
	if (tile.chunk < 1 || nsteps < 1) return fail(MMSPX_EINVAL, "bad chunk or step count");
	// a last pass of fewer steps: the tile made for that many, if there is one
	// (two steps of 256^3 x 8 FP32: 457 us on the three-step tile, 369 on its own)
	TuneChoice t = tile;
	if (nsteps < fmarch_steps(tile))
		for (const FieldTile& o : kFieldTiles)
			if (o.prec == prec && o.fields == g.fields && (64 - o.tz) / 2 == nsteps) {
				best_pass(g, o, &t);
				break;
			}
	if (prec == MMSPX_F64)
		return p.model == MMSPX_ZENER ? launch_fmarch_f64_zener(g, p, a, b, st, t, nsteps)
		                              : launch_fmarch_f64_gg(g, p, a, b, st, t, nsteps);
	return p.model == MMSPX_ZENER ? launch_fmarch_f32_zener(g, p, a, b, st, t, nsteps)
	                              : launch_fmarch_f32_gg(g, p, a, b, st, t, nsteps);
}

}  // namespace mmspx
