// kernels_fields2d.hip -- the FP64 form of the 2-D four-step field strips,
// tile body 16, and what both precisions share.
#include <algorithm>
#include <cmath>

#include "fields2d_launch.hpp"

namespace mmspx {

int launch_fields2d_f32(const Geom& g, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk,
                        int nsteps);

bool fields2d_supported(const Geom& g, int prec, int model)
{
	if (prec != MMSPX_F64 && prec != MMSPX_F32) return false;
	if (g.dim != 2 || (model != MMSPX_GG && model != MMSPX_ZENER)) return false;
	for (int k = 0; k < 2; k++)
		if (g.b0[k] != MMSPX_PERIODIC || g.b1[k] != MMSPX_PERIODIC) return false;
	// Zener pinning in double has no tiled kernel for 32 fields (fused_supported)
	if (g.fields == 32 && prec == MMSPX_F64 && model == MMSPX_ZENER) return false;
	return g.fields == 2 || g.fields == 4 || g.fields == 8 || g.fields == 16 || g.fields == 32;
}

// Rows per workgroup by a cost model. A pass takes T0 plus a workgroup's rows
// (chunk and five for the rows its march starts with) at `row` microseconds
// each, times what n waves on a SIMD cost, max(1, a + b n); a launch of more
// workgroups than `resident` per CU runs in rounds (0: the wave slots are not
// the limit, n is simply what the launch has). Moving the grid at 5 TB/s
// (times `move`, which takes in the halo) overlaps all but a quarter of the
// shorter of the two. Fitted per field count and precision to a sweep of 2 to
// 158 rows on sides 128 to 2048: the model picks the measured best in most
// cells, always within 6 %. Against the two-step split strips it replaces (us
// per step): 2048^2 x 32 FP32 140 -> 82.5, FP64 259 -> 180; 1024^2 x 32 FP32
// 31.5 -> 22.8; 2048^2 x 16 FP32 71.7 -> 42.2; 512^2 x 8 FP32 4.4 -> 3.6, FP64
// 6.2 -> 5.7; 2048^2 x 4 FP32 15.0 -> 11.4; 128^2 x 2 FP32 1.9 -> 1.1. It was
// faster at every size and field count of the sweep.
bool fields2d_choice(const Geom& g, int prec, int model, TuneChoice* out)
{
	if (!fields2d_supported(g, prec, model)) return false;
	struct Cost {
		int fields, waves, resident[2];
		double t0[2], row[2], a[2], b[2], move[2];
	};
	// [0] FP32, [1] FP64
	static const Cost table[] = {
	    {2, 1, {0, 0}, {2.31, 2.25}, {0.33, 0.45}, {0.39, 0.29}, {0.48, 0.65}, {1.4, 1.3}},
	    {4, 1, {0, 0}, {2.25, 2.14}, {0.55, 0.82}, {0.37, 0.19}, {0.57, 0.76}, {1.3, 1.0}},
	    {8, 4, {0, 0}, {3.1, 3.6}, {0.54, 0.69}, {0.45, 0.25}, {0.37, 0.59}, {0.4, 0.45}},
	    {16, 8, {4, 2}, {3.7, 4.1}, {0.68, 1.02}, {0.55, 0.34}, {0.22, 0.33}, {0.46, 0.47}},
	    {32, 16, {2, 0}, {4.4, 5.3}, {1.11, 0.69}, {-0.24, -0.31}, {0.226, 0.695}, {0.1, 0.66}},
	};
	const Cost* k = table;
	while (k->fields != g.fields) k++;
	const int f = prec == MMSPX_F64 ? 1 : 0;
	const double strips = (g.n[1] + kSteps4Cols - 1) / kSteps4Cols, cus = 256.0;
	const double move = 2.0 * (double)g.nodes * g.fields * (f ? 8 : 4) / 5e6 * k->move[f];
	const double per = std::max(k->waves / 4.0, 0.25);  // waves per SIMD a workgroup on every CU adds
	auto row = [&](double n) { return n > 0.0 ? k->row[f] * std::max(1.0, k->a[f] + k->b[f] * n) : 0.0; };
	auto cost = [&](int c) {
		const double items = strips * ((g.n[0] + c - 1) / c);
		double r;
		if (k->resident[f] > 0) {
			const double whole = std::floor(items / (cus * k->resident[f]));
			r = whole * row(k->resident[f] * per) + row(std::ceil((items - whole * cus * k->resident[f]) / cus) * per);
		} else {
			const double n = items * k->waves / (4.0 * cus);
			const double up = k->waves < 4 ? std::ceil(n) : std::ceil(items / cus) * per;
			r = row(up > 6.0 ? n + 0.5 * std::max(1.0, per) : up);
		}
		const double t = (c + 5) * r;
		return k->t0[f] + std::max(t, move) + 0.25 * std::min(t, move);
	};
	int best = 2;
	double least = cost(2);
	auto take = [&](int c) {
		const double v = cost(c);
		if (v < least) {
			least = v;
			best = c;
		}
	};
	for (int c = 3; c <= 16; c++) take(c);
	// longer ones that split the rows evenly
	for (int n = 1; n <= 64; n++) {
		const int c = (g.n[0] + n - 1) / n;
		if (c > 16 && c <= 512) take(c);
	}
	*out = TuneChoice{2, 1, kSteps4Cols, best, 16};
	return true;
}

int launch_fields2d(const Geom& g, int prec, const ModelParams& p, const void* a, void* b, hipStream_t st, int chunk,
                    int nsteps)
{
	if (!fields2d_supported(g, prec, p.model))
		return fail(MMSPX_EUNSUPPORTED, "the four-step field strips take periodic 2-D grain growth and Zener pinning with "
		                                "2, 4, 8, 16 or 32 fields in the MMSPX_F64 and MMSPX_F32 forms");
	if (chunk < 1 || nsteps < 1 || nsteps > kFieldsSteps)
		return fail(MMSPX_EINVAL, "more steps than a pass of the four-step field strips takes");
	return prec == MMSPX_F64 ? launch_fields2d_prec<MMSPX_F64>(g, p, a, b, st, chunk, nsteps)
	                         : launch_fields2d_f32(g, p, a, b, st, chunk, nsteps);
}

}  // namespace mmspx
