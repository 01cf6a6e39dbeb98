// gga2d.hpp -- 2-D multi-phase grain growth (grain_growth/anisotropic/phase_field/
// graingrowth.cpp:108-188), wave strips: one wave per (strip, chunk), any boundary.
//
// Lane l holds column c0 - 1 + l of all Q fields, columns outside the grid the
// node check_boundary maps them to, and lanes 1 .. 62 are written; axis-1
// neighbours move by DPP wave shifts, axis-0 neighbours are a window of three row
// slots whose roles rotate; row x+2 is loaded into row x-1's once that is used.
//
// Bound by vector instructions, so what a node does not need is kept off them.
// Which lanes have a field present is one 64-bit scalar mask per field and row,
// from one comparison as the row arrives; a node's own set is the scalar or of
// the row's mask, the rows' beside it and the mask shifted by a lane either way.
// A node with at most 4 of 8 fields present (nearly all) packs them in ascending
// order through a column of LDS slots of its own and takes the 4-slot rates: the
// same additions in the same order as the full loops, which skip absent fields.
// 1024^2 x 8 FP64: 36.0 us per step with the sets and the packing done by
// comparisons and selects in the lanes (920 vector instructions a node), 28.5
// this way, 4.7 TB/s of the 134 MB a step moves; FP32 20.4; 4 fields FP64 18.4.
#pragma once

#include "steps2d.hpp"

namespace mmspx {

constexpr int kGgaCols = 62;

template <int PREC, int Q, bool UNIT>
__device__ __forceinline__ void gga2d(const typename Form<PREC>::S* __restrict__ a, typename Form<PREC>::S* __restrict__ b,
                                      const Geom& g, const ModelParams& p, int c0, int xb, int xe,
                                      typename Form<PREC>::S* slots)
{
	using F = Form<PREC>;
	using S = typename F::S;
	constexpr int K = 4, ST = 256;  // packed slots, threads of a workgroup
	const int lane = threadIdx.x & 63;
	const int nx = g.n[0], ny = g.n[1];
	const size_t N = (size_t)nx * ny;
	const int c = c0 - 1 + lane;
	const unsigned cm = (unsigned)edge_map(c, ny, g.b0[1], g.b1[1]);
	const bool out = lane >= 1 && lane < 63 && c < ny;
	const unsigned co = out ? (unsigned)c : 0u;
	using Mask = unsigned long long;
	S w[3][Q];
	Mask mlo[Q], my[Q], mhi[Q];  // lanes whose field is positive in rows x-1, x, x+1
	auto load_row = [&](int x, S (&v)[Q]) {
		const S* r = a + (size_t)edge_map(min(x, xe), nx, g.b0[0], g.b1[0]) * ny;
#pragma unroll
		for (int f = 0; f < Q; f++) v[f] = (r + f * N)[cm];
	};
	auto mark = [&](const S (&v)[Q], Mask (&m)[Q]) {
#pragma unroll
		for (int f = 0; f < Q; f++) m[f] = __ballot(v[f] > S(0));
	};
	load_row(xb - 1, w[0]);
	load_row(xb, w[1]);
	load_row(xb + 1, w[2]);
	mark(w[0], mlo);
	mark(w[1], my);
	auto row = [&](int x, S (&lo)[Q], const S (&y)[Q], const S (&hi)[Q]) {
		mark(hi, mhi);
		S phi[Q], lap[Q];
		bool in[Q];
		int n = 0;
#pragma unroll
		for (int f = 0; f < Q; f++) {
			phi[f] = y[f];
			lap[f] = lap2<PREC, UNIT, false>(g, hi[f], lo[f], shift_next(y[f]), shift_prev(y[f]), y[f]);
			in[f] = __builtin_amdgcn_inverse_ballot_w64(mlo[f] | my[f] | mhi[f] | my[f] << 1 | my[f] >> 1);
			mlo[f] = my[f];
			my[f] = mhi[f];
		}
		if (x + 1 < xe) load_row(x + 2, lo);  // row x+2 takes x-1's slot
		if constexpr (Q > K) {
			S* at = slots;
#pragma unroll
			for (int f = 0; f < Q; f++) {
				if (in[f] && n < K) {
					at[0] = phi[f];
					at[K * ST] = lap[f];
				}
				n += in[f] ? 1 : 0;
				at += in[f] ? ST : 0;
			}
		} else {
#pragma unroll
			for (int f = 0; f < Q; f++) n += in[f] ? 1 : 0;
		}
		if (n >= 2) {
			S dp[Q];
			auto full = [&]() {
				uint32_t act = 0;
#pragma unroll
				for (int f = 0; f < Q; f++) act |= in[f] ? 1u << f : 0u;
				gga_rates<PREC, Q>(phi, lap, act, p, dp);
			};
			if constexpr (Q > K) {
				if (n <= K) {
					S cphi[K], clap[K], cdp[K];
#pragma unroll
					for (int s = 0; s < K; s++) {
						cphi[s] = slots[s * ST];
						clap[s] = slots[(K + s) * ST];
					}
					gga_rates4<PREC>(cphi, clap, n, p, cdp);
#pragma unroll
					for (int s = 0; s < K; s++) slots[s * ST] = cdp[s];
					S* at = slots;
#pragma unroll
					for (int f = 0; f < Q; f++) {
						dp[f] = 0;
						if (in[f]) {
							dp[f] = at[0];
							at += ST;
						}
					}
				} else {
					full();
				}
			} else {
				full();
			}
			gga_project<PREC, Q>(phi, dp, (S)n, Q, p);
		}
		if (out) {
			S* r = b + (size_t)x * ny;
#pragma unroll
			for (int f = 0; f < Q; f++) (r + f * N)[co] = phi[f];
		}
	};
	// one copy of the body (the 8-field rates are large) and copies of the slots
#pragma unroll 1
	for (int x = xb; x < xe; x++) {
		row(x, w[0], w[1], w[2]);
#pragma unroll
		for (int f = 0; f < Q; f++) {
			const S next = w[0][f];
			w[0][f] = w[1][f];
			w[1][f] = w[2][f];
			w[2][f] = next;
		}
	}
}

}  // namespace mmspx
