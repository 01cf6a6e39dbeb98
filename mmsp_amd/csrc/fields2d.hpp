// fields2d.hpp -- 2-D grain growth and Zener pinning, four explicit steps per
// pass in registers: W waves per (strip of columns, chunk of rows), Q/W fields
// each.
//
// The layout of the multi-step wave strips (steps2d.hpp): lane l holds column
// c0 - 4 + l of every level (phi^n .. phi^{n+4}), level s is right on lanes s
// .. 63 - s, 56 columns are written; at iteration t row t of level 0 has
// arrived and level s forms its row t - s; column neighbours move by DPP wave
// shifts, row neighbours sit in registers whose roles rotate over a six-row
// unrolled march. Wave h holds fields h*Q/W .. (h+1)*Q/W - 1.
//
// The update needs sum_j phi_j^2 over all fields in field order
// (graingrowth.cpp:91-97). The rows whose sums iteration t + 1 needs (the
// newest row of levels 0..3) are complete at the end of iteration t: every
// wave publishes its squares to LDS and the waves then sum one level each, so
// a row takes two barriers however many waves and levels there are, and one
// LDS read per square. With one wave (W = 1) the sums stay in registers.
//
// A four-step pass over 2048^2 x 32 FP32 takes 330 us, of which moving the grid
// once takes 240 and vector work (about 18 instructions per field, node and
// step at 2.3 cycles, 4.4 where a shift is folded in) about 200 beside it, on
// 64/56 of the columns. Two fields per wave, so that many
// waves meet the latencies of a row: 2048^2 x 32 FP32 85.4 us with four,
// 512^2 x 8 FP32 4.3 against 3.6; four where one wave then holds all of them
// and needs no exchange (2048^2 x 4 FP32 11.4 us, 12.4 on two waves).
//
// Every value is the one-step kernels' for that node and step, from the same
// operands in the same order (KIND 3 holds field 0, zener.cpp:117-135), so a
// pass gives the bits of single steps. Periodic grids.
#pragma once

#include "steps2d.hpp"

namespace mmspx {

// `steps` <= 4 of them (four where FULL). UNIT: both grid weights are exactly 1.
template <int PREC, int Q, int KIND, int W, bool UNIT, bool FULL>
__device__ __forceinline__ void fields2d(const typename Form<PREC>::S* __restrict__ a,
                                         typename Form<PREC>::S* __restrict__ b, const Geom& g, const ModelParams& p,
                                         int c0, int xb, int xe, int steps)
{
	using F = Form<PREC>;
	using S = typename F::S;
	using Sum = typename F::Sum;
	constexpr int L = kFieldsSteps, H = Q / W, U = 6;
	static_assert(Q % W == 0, "the strips hold Q/W fields per wave");
	__shared__ Sum sq[W > 1 ? L : 1][W > 1 ? Q : 1][64], tot[W > 1 ? L : 1][64];
	const int nl = FULL ? L : steps;
	const int lane = threadIdx.x & 63;
	const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
	const int f0 = wv * H;
	const int nx = g.n[0], ny = g.n[1];
	const size_t N = (size_t)nx * ny;
	const int c = c0 - L + lane;
	const unsigned cm = (unsigned)wrap(c, ny);
	const bool out = lane >= L && lane < 64 - L && c < ny;
	const unsigned co = out ? (unsigned)c : 0u;
	const int base = xb - nl;  // level 0's row at iteration 0
	const int tend = xe - xb + 2 * nl;
	const S* __restrict__ af = a + (size_t)f0 * N;
	S* __restrict__ bf = b + (size_t)f0 * N;
	// level 0's rows arrive in order, three in flight; rows past the last one
	// the chunk reads load that row again
	int tl = 0, wr = wrap(base, nx);
	auto ld = [&](S* w) {
		const S* __restrict__ r = af + (size_t)wr * ny;
#pragma unroll
		for (int j = 0; j < H; j++) w[j] = (r + j * N)[cm];
		if (++tl < tend) wr = wr + 1 == nx ? 0 : wr + 1;
	};

	S l0[U][H];         // level 0, row t in slot t % 6
	S lv[L - 1][3][H];  // level s >= 1 in lv[s - 1], row r in slot r % 3
#pragma unroll
	for (int s = 0; s < L - 1; s++)
#pragma unroll
		for (int k = 0; k < 3; k++)
#pragma unroll
			for (int j = 0; j < H; j++) lv[s][k][j] = 0;
	auto at = [&](int s, int r, int j) -> S& { return s == 0 ? l0[r % U][j] : lv[s - 1][r % 3][j]; };
	// level s at iteration t (t6 = t mod 6, known at compile time): row t - s
	// from rows t-s-1 .. t-s+1 of level s - 1 and that row's sum
	auto level = [&](int s, int t, int t6, Sum sum) {
		const int r = t6 + 36 - s;
		S v[H];
		S* __restrict__ dst = bf + (size_t)(base + t - s) * ny;
#pragma unroll
		for (int j = 0; j < H; j++) {
			const S y = at(s - 1, r, j);
			const typename F::L lap =
			    lap2<PREC, UNIT, false>(g, at(s - 1, r + 1, j), at(s - 1, r - 1, j), shift_next(y), shift_prev(y), y);
			v[j] = (KIND == 3 && f0 + j == 0) ? y : F::gg(y, sum, lap, p);
			if (s < L) at(s, r, j) = v[j];
		}
		if (s == nl && out) {
#pragma unroll
			for (int j = 0; j < H; j++) (dst + j * N)[co] = v[j];
		}
	};
	auto iter = [&](int t, int t6) {
		ld(l0[(t6 + 3) % U]);
		Sum sum[L];
#pragma unroll
		for (int s = 0; s < L; s++) {
			if constexpr (W > 1) {
				sum[s] = tot[s][lane];
			} else {
				sum[s] = 0;
#pragma unroll
				for (int j = 0; j < H; j++) {
					const Sum v = at(s, t6 + 36 - 1 - s, j);
					sum[s] += v * v;
				}
			}
		}
#pragma unroll
		for (int s = 1; s <= L; s++)
			if (s <= nl && 2 * s <= t) level(s, t, t6, sum[s - 1]);
		if constexpr (W > 1) {
#pragma unroll
			for (int s = 0; s < L; s++)
				if (s < nl)
#pragma unroll
					for (int j = 0; j < H; j++) {
						const Sum v = at(s, t6 + 36 - s, j);
						sq[s][f0 + j][lane] = v * v;
					}
			__syncthreads();
			for (int s = wv; s < nl; s += W) {
				Sum acc = 0;
#pragma unroll
				for (int q = 0; q < Q; q++) acc += sq[s][q][lane];
				tot[s][lane] = acc;
			}
			__syncthreads();
		}
	};
	ld(l0[0]);
	ld(l0[1]);
	ld(l0[2]);
#pragma unroll
	for (int k = 3; k < U; k++)
#pragma unroll
		for (int j = 0; j < H; j++) l0[k][j] = 0;
	for (int t = 0;; t += U) {
#pragma unroll
		for (int u = 0; u < U; u++) {
			if (t + u >= tend) return;
			iter(t + u, u);
		}
	}
}

}  // namespace mmspx
