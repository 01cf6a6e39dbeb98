// march4.hpp -- 3-D periodic Cahn-Hilliard (two explicit steps per pass) and
// Allen-Cahn (four) as one plane march over four LEVELS, each a radius-1
// stencil of the one before: mu^n, c^{n+1}, mu^{n+1}, c^{n+2}
// (cahn-hilliard.cpp:69-76, twice), or phi^{n+1} .. phi^{n+4}
// (allen-cahn.cpp:68-71, four times). One pass reads and writes the grid once.
//
// A workgroup takes a TY x TZ tile of the (axis 1, axis 2) plane over planes
// [xb, xe). Each thread owns a 2 x 2 block of points of the tile and its
// three-cell halo (region R3). The iteration at plane P forms level 1 at P,
// level 2 at P-1, level 3 at P-2 and level 4 at P-3, which it writes. Axis-0
// neighbours are the thread's own values at the planes before and after, in
// registers whose roles rotate over a six-plane unrolled march (three slots a
// level; level 0's next plane is loaded into the oldest slot once that is used); in-plane
// neighbours inside the block are registers too, and the block's eight outer
// ones come from LDS, where every level's plane is published once. What bounds
// the march is LDS traffic and VALU work side by side: a point and level costs
// three LDS words this way (one written, two read) where a thread that owns
// scattered points pays five, and one address per plane serves the block. The
// planes are double-buffered, so one barrier per iteration orders everything,
// and all of an iteration's LDS reads are of planes finished before it, so
// they can be in flight together.
//
// Every value is the one-step kernels' for that node and step (the halo
// recomputes what the neighbouring tile computes), so the bits are theirs.
// Points past the levels' regions are formed from whatever lies beside them in
// the planes and never reach a written node; all LDS reads stay inside the
// array, with the level-0 planes, which are never read outside, at its ends.
#pragma once

#include "steps2d.hpp"

namespace mmspx {

// The three-axis laplacian (see lap2).
template <int PREC, bool UNIT, bool ZERO>
__device__ __forceinline__ typename Form<PREC>::L lap3(const Geom& g, typename Form<PREC>::S xh,
                                                       typename Form<PREC>::S xl, typename Form<PREC>::S yh,
                                                       typename Form<PREC>::S yl, typename Form<PREC>::S zh,
                                                       typename Form<PREC>::S zl, typename Form<PREC>::S y)
{
	using S = typename Form<PREC>::S;
	auto term = [&](S h, S l) -> S {
		if constexpr (PREC == MMSPX_F64) return __builtin_fma(-2.0, y, h) + l;
		else return __builtin_fmaf(-2.0f, y, h) + l;
	};
	S tx = term(xh, xl), ty = term(yh, yl), tz = term(zh, zl);
	if constexpr (!UNIT) {
		tx = (PREC == MMSPX_F64 ? (S)g.w[0] : (S)g.wf[0]) * tx;
		ty = (PREC == MMSPX_F64 ? (S)g.w[1] : (S)g.wf[1]) * ty;
		tz = (PREC == MMSPX_F64 ? (S)g.w[2] : (S)g.wf[2]) * tz;
	}
	return ((ZERO ? S(0) + tx : tx) + ty) + tz;
}

// Row pitch (elements) of an LDS plane of `cols` columns read by `bz` lanes a
// block row: a wave's next block row (two rows down) should start in the bank
// where the one before ended, so that its contiguous runs do not overlap (FP32:
// 150 x 203 x 97 Cahn-Hilliard 11.8 -> 10.7 us per step on 16 x 16 tiles, 256^3
// 23.9 -> 23.5; in double it changed nothing)
constexpr int lds_pitch(int cols, int bz, int elem)
{
	if (elem == 8) return cols;
	int best = cols, miss = 1 << 20;
	for (int w = cols; w < cols + 32; w += 2) {
		const int words = elem / 4, d = ((2 * w - bz) * words % 64 + 64) % 64;
		const int m = (d < 64 - d ? d : 64 - d) * 8 + (w - cols);
		if (m < miss) {
			miss = m;
			best = w;
		}
	}
	return best;
}

// LEVELS < 4: a last pass of fewer steps, level LEVELS is written. UNIT 1: every
// grid weight is 1 and, for Cahn-Hilliard, so is the gradient coefficient, 2: so
// is every coefficient (the multiplications by them are left out; the bits are
// the same).
template <int PREC, int MODEL, int TY, int TZ, int NT, int LEVELS, int UNIT>
__device__ __forceinline__ void march4(const typename Form<PREC>::S* __restrict__ a,
                                       typename Form<PREC>::S* __restrict__ b, const Geom& g, const ModelParams& p,
                                       int y0, int z0, int xb, int xe)
{
	using F = Form<PREC>;
	using S = typename F::S;
	static_assert(TY % 2 == 0 && TZ % 2 == 0, "the region divides into 2 x 2 blocks");
	constexpr int P4Y = TY + 8, P4Z = TZ + 8;  // level 0 (four-cell halo)
	constexpr int R3Y = TY + 6, R3Z = TZ + 6;  // level 1: the threads' blocks
	constexpr int R2Y = TY + 4, R2Z = TZ + 4;  // level 2
	constexpr int R1Y = TY + 2, R1Z = TZ + 2;  // level 3
	constexpr int BY = R3Y / 2, BZ = R3Z / 2;
	constexpr int PW = lds_pitch(P4Z, BZ, sizeof(S)), W1 = lds_pitch(R3Z, BZ, sizeof(S));
	constexpr int W2 = lds_pitch(R2Z, BZ, sizeof(S)), W3 = lds_pitch(R1Z, BZ, sizeof(S));
	constexpr int N0 = P4Y * PW, N1 = R3Y * W1, N2 = R2Y * W2, N3 = R1Y * W3;
	static_assert(BY * BZ <= NT, "one block per thread");
	constexpr int RN = P4Y * P4Z - R3Y * R3Z;  // level 0's points outside R3 (a one-cell ring)
	constexpr int MR = (RN + NT - 1) / NT;
	// level 0 first and last; reads up to three rows before level 3's and
	// one row after level 1's planes land in their neighbours
	constexpr int O3 = N0, O2 = O3 + 2 * N3, O1 = O2 + 2 * N2, O0 = O1 + 2 * N1;
	static_assert(3 * W3 + 3 <= N0 && 2 * W1 + 2 <= N0, "stray reads stay inside the array");
	__shared__ S lds[O0 + N0];

	const int nx = g.n[0], ny = g.n[1], nz = g.n[2];
	const int64_t plane = (int64_t)ny * nz;
	const int t = threadIdx.x;
	// spare threads repeat the last block: the same values to the same places
	const int e = min(t, BY * BZ - 1);
	const int r0 = e / BZ * 2, c0 = e % BZ * 2;  // the block's first point in R3
	// a plane's row holds its even columns, then its odd ones, so a wave's accesses
	// are contiguous; j: the block's pair of columns. Even / odd column of the
	// pair, or of the pair beside it, at these indices of the planes' first row
	const int j0 = c0 / 2;
	const int q0 = (r0 + 1) * PW + j0, q1 = r0 * W1 + j0, q2 = (r0 - 1) * W2 + j0 - 1, q3 = (r0 - 2) * W3 + j0 - 1;
	unsigned off[4];
	bool w2[4], w3[4], out[4];  // the point belongs to level 2's, level 3's region; is written
#pragma unroll
	for (int k = 0; k < 4; k++) {
		const int r = r0 + (k >> 1), c = c0 + (k & 1), y = y0 - 3 + r, z = z0 - 3 + c;
		off[k] = (unsigned)(wrap(y, ny) * nz + wrap(z, nz)) * (unsigned)sizeof(S);
		w2[k] = r >= 1 && r <= R2Y && c >= 1 && c <= R2Z;
		w3[k] = r >= 2 && r < R1Y + 2 && c >= 2 && c < R1Z + 2;
		out[k] = r >= 3 && r < TY + 3 && c >= 3 && c < TZ + 3 && y < ny && z < nz;
	}
	unsigned roff[MR];
	int rq[MR];
#pragma unroll
	for (int j = 0; j < MR; j++) {
		const int u = t + j * NT;
		roff[j] = 0;
		rq[j] = 0;
		if (u < RN) {
			int pr, pc;
			if (u < P4Z) {
				pr = 0;
				pc = u;
			} else if (u < 2 * P4Z) {
				pr = P4Y - 1;
				pc = u - P4Z;
			} else {
				pr = 1 + (u - 2 * P4Z) / 2;
				pc = (u & 1) ? P4Z - 1 : 0;
			}
			roff[j] = (unsigned)(wrap(y0 - 4 + pr, ny) * nz + wrap(z0 - 4 + pc, nz)) * (unsigned)sizeof(S);
			rq[j] = pr * PW + (pc & 1) * (PW / 2) + pc / 2;
		}
	}
	// planes arrive in order and wrap; a plane's address is scalar, the point's
	// byte offset in it 32 bits
	auto at = [](const S* base, unsigned o) -> const S& { return *(const S*)((const char*)base + o); };
	int wx = wrap(xb - 4, nx);
	auto src_next = [&]() {
		const S* s = a + (int64_t)wx * plane;
		wx = wx + 1 == nx ? 0 : wx + 1;
		return s;
	};

	S f[3][4];                       // level 0 at P-1, P, P+1: plane i in slot i % 3
	S v1[3][4], v2[3][4], v3[3][4];  // levels 1..3
	S rg[2][MR];
#pragma unroll
	for (int k = 0; k < 4; k++)
#pragma unroll
		for (int s = 0; s < 3; s++) v1[s][k] = v2[s][k] = v3[s][k] = 0;
	const S* ring_src = nullptr;
#pragma unroll
	for (int s = 0; s < 3; s++) {
		ring_src = src_next();
#pragma unroll
		for (int k = 0; k < 4; k++) f[s][k] = at(ring_src, off[k]);
		if (s == 1)
#pragma unroll
			for (int j = 0; j < MR; j++) rg[0][j] = at(ring_src, roff[j]);
	}
	__syncthreads();  // the previous tile of a persistent loop may still read the planes

	// one level at the block: in-plane neighbours from plane q (row pitch W),
	// values h, m, l at the planes after, at and before; r0 receives the laplacians
	// `odd` planes (level 0 and 2) have the block's first column in the odd half
	auto laps = [&](const S* __restrict__ q, int W, bool odd, const S (&h)[4], const S (&m)[4], const S (&l)[4],
	                typename F::L (&o)[4]) {
		// columns c0 (A), c0 + 1 (B), c0 - 1 (L), c0 + 2 (R) of the plane
		const int A = odd ? W / 2 : 0, B = odd ? 1 : W / 2, Lc = odd ? 0 : W / 2 - 1, Rc = odd ? W / 2 + 1 : 1;
		const S u0 = q[A - W], u1 = q[B - W], d0 = q[A + 2 * W], d1 = q[B + 2 * W];
		const S l0 = q[Lc], l1 = q[Lc + W], h0 = q[Rc], h1 = q[Rc + W];
		o[0] = lap3<PREC, UNIT != 0, MODEL == S2_CH>(g, h[0], l[0], m[2], u0, m[1], l0, m[0]);
		o[1] = lap3<PREC, UNIT != 0, MODEL == S2_CH>(g, h[1], l[1], m[3], u1, h0, m[0], m[1]);
		o[2] = lap3<PREC, UNIT != 0, MODEL == S2_CH>(g, h[2], l[2], d0, m[0], m[3], l1, m[2]);
		o[3] = lap3<PREC, UNIT != 0, MODEL == S2_CH>(g, h[3], l[3], d1, m[1], h1, m[2], m[3]);
	};
	auto mu = [&](S c, typename F::L lap) -> S {
		if constexpr (MODEL == S2_CH_DW && UNIT) return F::mu_dw1(c, lap);
		else if constexpr (MODEL == S2_CH_DW) return F::mu_dw(c, lap, p);
		else if constexpr (UNIT == 2) return mu_unit<PREC>(c, lap);
		else if constexpr (UNIT == 1) return F::mu_poly1(c, lap, p);
		else return F::mu_poly(c, lap, p);
	};
	auto odd = [&](S y, typename F::L lap) -> S {
		if constexpr (MODEL == S2_AC) return UNIT == 2 ? ac_unit<PREC>(y, lap, p) : F::ac(y, lap, p);
		else return mu(y, lap);
	};
	auto even = [&](S y, typename F::L lap, S c) -> S {
		if constexpr (MODEL == S2_AC) return UNIT == 2 ? ac_unit<PREC>(y, lap, p) : F::ac(y, lap, p);
		else return F::ch(c, lap, p);
	};

	// the iteration at plane P = xb - 3 + i; j = i mod 6 is known at compile
	// time, depth the levels whose first plane has been reached
	auto iter = [&](int i, int j, int depth) {
		const int P = xb - 3 + i;
		S(&fm)[4] = f[j % 3];
		S(&fc)[4] = f[(j + 1) % 3];
		S(&fp)[4] = f[(j + 2) % 3];
#pragma unroll
		for (int m = 0; m < MR; m++) rg[(j + 1) & 1][m] = at(ring_src, roff[m]);
		// plane P+2 takes P-1's slot once P-1 has been used
		auto load = [&]() {
			ring_src = src_next();
#pragma unroll
			for (int k = 0; k < 4; k++) fm[k] = at(ring_src, off[k]);
		};
		S* __restrict__ l0 = lds + ((j & 1) ? O0 : 0);
		S* __restrict__ l1w = lds + O1 + ((j & 1) ? N1 : 0);
		const S* __restrict__ l1r = lds + O1 + ((j & 1) ? 0 : N1);
		S* __restrict__ l2w = lds + O2 + ((j & 1) ? N2 : 0);
		const S* __restrict__ l2r = lds + O2 + ((j & 1) ? 0 : N2);
		S* __restrict__ l3w = lds + O3 + ((j & 1) ? N3 : 0);
		const S* __restrict__ l3r = lds + O3 + ((j & 1) ? 0 : N3);
		l0[q0 + PW / 2] = fc[0];
		l0[q0 + 1] = fc[1];
		l0[q0 + PW + PW / 2] = fc[2];
		l0[q0 + PW + 1] = fc[3];
#pragma unroll
		for (int m = 0; m < MR; m++)
			if (t + m * NT < RN) l0[rq[m]] = rg[j & 1][m];
		__syncthreads();
		typename F::L lp[4];
		// the written level, at plane x
		auto write = [&](int x, auto value) {
			if (LEVELS < 4 && (x < xb || x >= xe)) return;
			S* dst = b + (int64_t)x * plane;
#pragma unroll
			for (int k = 0; k < 4; k++)
				if (out[k]) *(S*)((char*)dst + off[k]) = value(k);
		};
		// level 1 at P
		S(&a1)[4] = v1[j % 3];
		S(&b1)[4] = v1[(j + 2) % 3];  // P-1
		S(&c1)[4] = v1[(j + 1) % 3];  // P-2
		laps(l0 + q0, PW, true, fp, fc, fm, lp);
		if constexpr (LEVELS == 1) {
			write(P, [&](int k) { return odd(fc[k], lp[k]); });
			load();
			return;
		}
#pragma unroll
		for (int k = 0; k < 4; k++) a1[k] = odd(fc[k], lp[k]);
		l1w[q1] = a1[0];
		l1w[q1 + W1 / 2] = a1[1];
		l1w[q1 + W1] = a1[2];
		l1w[q1 + W1 + W1 / 2] = a1[3];
		if (depth < 2) {
			load();
			return;
		}
		// level 2 at P-1: level 1 at P, P-1, P-2, level 0 at P-1
		S(&a2)[4] = v2[j % 3];
		S(&b2)[4] = v2[(j + 2) % 3];
		S(&c2)[4] = v2[(j + 1) % 3];
		laps(l1r + q1, W1, false, a1, b1, c1, lp);
		if constexpr (LEVELS == 2) {
			write(P - 1, [&](int k) { return even(b1[k], lp[k], fm[k]); });
			load();
			return;
		}
#pragma unroll
		for (int k = 0; k < 4; k++) {
			a2[k] = even(b1[k], lp[k], fm[k]);
			if (w2[k]) l2w[q2 + (k >> 1) * W2 + ((k & 1) ? 1 : W2 / 2)] = a2[k];
		}
		load();
		if (depth < 3) return;
		// level 3 at P-2
		S(&a3)[4] = v3[j % 3];
		S(&b3)[4] = v3[(j + 2) % 3];
		S(&c3)[4] = v3[(j + 1) % 3];
		laps(l2r + q2, W2, true, a2, b2, c2, lp);
		if constexpr (LEVELS == 3) {
			write(P - 2, [&](int k) { return odd(b2[k], lp[k]); });
			return;
		}
#pragma unroll
		for (int k = 0; k < 4; k++) {
			a3[k] = odd(b2[k], lp[k]);
			if (w3[k]) l3w[q3 + (k >> 1) * W3 + ((k & 1) ? W3 / 2 : 0)] = a3[k];
		}
		if (depth < 4) return;
		// level 4 at P-3
		laps(l3r + q3, W3, false, a3, b3, c3, lp);
		write(P - 3, [&](int k) { return even(b3[k], lp[k], c2[k]); });
	};
	// level s starts at iteration 2 (s - 1)
#pragma unroll
	for (int i = 0; i < 6; i++) iter(i, i, 1 + i / 2);
	const int n = xe - xb + 2 + LEVELS;  // level LEVELS reaches plane xe - 1 in the last iteration
	for (int i = 6;; i += 6) {
#pragma unroll
		for (int u = 0; u < 6; u++) {
			if (i + u >= n) return;
			iter(i + u, u, 4);
		}
	}
}

}  // namespace mmspx
