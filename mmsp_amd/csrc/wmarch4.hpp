// wmarch4.hpp -- the four-level march of march4.hpp (3-D periodic Cahn-Hilliard
// and Allen-Cahn, the same levels and the same bits) with a wave's lanes along
// axis 2.
//
// A workgroup of NW waves takes a (NW*R - 6) x 56 tile of the (axis 1, axis 2)
// plane. Lane l of every wave holds column z0 - 4 + l of every level (level s is
// right on lanes s .. 63 - s, 56 columns are written), wave h rows h*R ..
// h*R + R - 1 of the tile and its three-row halo. Axis-2 neighbours move by DPP
// wave shifts, axis-0 neighbours and the rows of the same wave are registers,
// and only a wave's first and last row go through LDS: two words written and two
// read per R points and level, where a 2 x 2 block of march4.hpp moves twelve
// for four. One barrier per plane.
//
// In double that march was bound by LDS and vector work side by side (256^3
// Cahn-Hilliard 42 us per step: 22 and 20). Here vector work is 73 % of the
// time at the rates the instructions reach (4.3 cycles for a double add or a
// shift), the rest waits at the barrier; 16 waves of two rows, the most a
// workgroup holds, or 12 of four where the grid gives each enough planes. Whole
// calls at 256^3 FP64, us per step: Cahn-Hilliard 38.0, Allen-Cahn 25.1 where
// every coefficient is one and 27.1 otherwise; 320^3 Cahn-Hilliard 70.6. Tried
// at 256^3 in a loop of their own, Cahn-Hilliard and Allen-Cahn: 8 waves of four
// rows 7 and 5 % slower, a column pair per lane (half the shifts) 12 and 8 %,
// levels two planes apart, so that none waits for another, 4 %.
#pragma once

#include "march4.hpp"

namespace mmspx {

// The three-axis laplacian (see lap2), axis-2 neighbours from the lanes beside.
template <int PREC, bool UNIT, bool ZERO>
__device__ __forceinline__ typename Form<PREC>::L wlap3(const Geom& g, typename Form<PREC>::S xh,
                                                        typename Form<PREC>::S xl, typename Form<PREC>::S yh,
                                                        typename Form<PREC>::S yl, typename Form<PREC>::S y)
{
	using S = typename Form<PREC>::S;
	S tx, ty, tz;
	if constexpr (PREC == MMSPX_F64) {
		tx = __builtin_fma(-2.0, y, xh) + xl;
		ty = __builtin_fma(-2.0, y, yh) + yl;
		tz = __builtin_fma(-2.0, y, shift_next(y)) + shift_prev(y);
	} else {
		tx = __builtin_fmaf(-2.0f, y, xh) + xl;
		ty = __builtin_fmaf(-2.0f, y, yh) + yl;
		tz = (shift_next(y) - 2.0f * y) + shift_prev(y);  // the shifts fold into the subtract and the add
	}
	if constexpr (!UNIT) {
		tx = (PREC == MMSPX_F64 ? (S)g.w[0] : (S)g.wf[0]) * tx;
		ty = (PREC == MMSPX_F64 ? (S)g.w[1] : (S)g.wf[1]) * ty;
		tz = (PREC == MMSPX_F64 ? (S)g.w[2] : (S)g.wf[2]) * tz;
	}
	return ((ZERO ? S(0) + tx : tx) + ty) + tz;
}

template <int PREC, int MODEL, int NW, int R, int LEVELS, int UNIT>
__device__ __forceinline__ void wmarch4(const typename Form<PREC>::S* __restrict__ a,
                                        typename Form<PREC>::S* __restrict__ b, const Geom& g, const ModelParams& p,
                                        int y0, int z0, int xb, int xe)
{
	using F = Form<PREC>;
	using S = typename F::S;
	constexpr int TY = NW * R - 6;
	__shared__ S edge[4][2][2][NW + 1][64];

	const int nx = g.n[0], ny = g.n[1], nz = g.n[2];
	const int64_t plane = (int64_t)ny * nz;
	const int lane = threadIdx.x & 63;
	const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
	const int z = z0 - 4 + lane;
	// a row's address is scalar, the lane's byte offset in it 32 bits
	const unsigned zc = (unsigned)wrap(z, nz) * (unsigned)sizeof(S);
	auto uniform = [](int v) { return (unsigned)__builtin_amdgcn_readfirstlane(v); };
	const bool zout = lane >= 4 && lane < 60 && z < nz;
	// the wave's rows of the tile and its three-row halo, wave-uniform
	const int r0 = wv * R;
	unsigned row[R];
#pragma unroll
	for (int k = 0; k < R; k++) {
		const int r = r0 + k, y = y0 - 3 + r;
		row[k] = uniform(wrap(y, ny)) * (unsigned)nz;
	}
	// the rows that are written: 3 <= r < TY + 3 and y < ny
	const int klo = 3 - r0, khi = min(TY + 3, ny - y0 + 3) - r0;
	const bool first = wv == 0, last = wv == NW - 1;
	const unsigned rrow = uniform(wrap(first ? y0 - 4 : y0 + TY + 3, ny)) * (unsigned)nz;
	int wx = (int)uniform(wrap(xb - 4, nx));
	auto src_next = [&]() {
		const S* s = a + (int64_t)wx * plane;
		wx = wx + 1 == nx ? 0 : wx + 1;
		return s;
	};

	S f[3][R];                       // level 0 at P-1, P, P+1: plane i in slot i % 3
	S v1[3][R], v2[3][R], v3[3][R];  // levels 1..3
	S rg[2];
	rg[0] = rg[1] = 0;
#pragma unroll
	for (int k = 0; k < R; k++)
#pragma unroll
		for (int s = 0; s < 3; s++) v1[s][k] = v2[s][k] = v3[s][k] = 0;
	unsigned o = zc;
	const S* ring_src = nullptr;
#pragma unroll
	for (int s = 0; s < 3; s++) {
		ring_src = src_next();
#pragma unroll
		for (int k = 0; k < R; k++) f[s][k] = load_at(ring_src + row[k], o);
		if (s == 1 && (first || last)) rg[0] = load_at(ring_src + rrow, o);
	}

	auto publish = [&](int level, int buf, const S (&v)[R]) {
		edge[level][buf][0][wv + 1][lane] = v[R - 1];
		edge[level][buf][1][wv][lane] = v[0];
	};
	// one level: values h, m, l at the planes after, at and before
	S up[4], dn[4];
	auto fetch = [&](int level, int buf) {
		up[level] = edge[level][buf][0][wv][lane];
		dn[level] = edge[level][buf][1][wv + 1][lane];
	};
	auto form = [&](int level, const S (&h)[R], const S (&m)[R], const S (&l)[R], auto value) {
#pragma unroll
		for (int k = 0; k < R; k++) {
			const S yl = k > 0 ? m[k > 0 ? k - 1 : 0] : up[level], yh = k < R - 1 ? m[k < R - 1 ? k + 1 : 0] : dn[level];
			value(k, wlap3<PREC, UNIT != 0, MODEL == S2_CH>(g, h[k], l[k], yh, yl, m[k]));
		}
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
		S(&fm)[R] = f[j % 3];
		S(&fc)[R] = f[(j + 1) % 3];
		S(&fp)[R] = f[(j + 2) % 3];
		if (first || last) {
			keep_value(o);
			rg[(j + 1) & 1] = load_at(ring_src + rrow, o);
		}
		auto load = [&]() {
			ring_src = src_next();
			keep_value(o);
#pragma unroll
			for (int k = 0; k < R; k++) fm[k] = load_at(ring_src + row[k], o);
		};
		const int w = j & 1, r = w ^ 1;
		publish(0, w, fc);
		if (first) edge[0][w][0][0][lane] = rg[j & 1];
		if (last) edge[0][w][1][NW][lane] = rg[j & 1];
		__syncthreads();
		// every row beside this iteration reads is of a plane finished before it
		fetch(0, w);
		if (depth > 1) fetch(1, r);
		if (depth > 2) fetch(2, r);
		if (depth > 3) fetch(3, r);
		// the written level's row k, at plane x
		auto write = [&](int x, int k, S v) {
			if (LEVELS < 4 && (x < xb || x >= xe)) return;
			keep_value(v);
			if (k >= klo && k < khi)
				if (zout) {
					keep_value(o);
					store_at(b + (int64_t)x * plane + row[k], o, v);
				}
		};
		S(&a1)[R] = v1[j % 3];
		S(&b1)[R] = v1[(j + 2) % 3];  // P-1
		S(&c1)[R] = v1[(j + 1) % 3];  // P-2
		if constexpr (LEVELS == 1) {
			form(0, fp, fc, fm, [&](int k, typename F::L lap) { write(P, k, odd(fc[k], lap)); });
			load();
			return;
		}
		form(0, fp, fc, fm, [&](int k, typename F::L lap) { a1[k] = odd(fc[k], lap); });
		publish(1, w, a1);
		if (depth < 2) {
			load();
			return;
		}
		S(&a2)[R] = v2[j % 3];
		S(&b2)[R] = v2[(j + 2) % 3];
		S(&c2)[R] = v2[(j + 1) % 3];
		if constexpr (LEVELS == 2) {
			form(1, a1, b1, c1, [&](int k, typename F::L lap) { write(P - 1, k, even(b1[k], lap, fm[k])); });
			load();
			return;
		}
		form(1, a1, b1, c1, [&](int k, typename F::L lap) { a2[k] = even(b1[k], lap, fm[k]); });
		publish(2, w, a2);
		load();
		if (depth < 3) return;
		S(&a3)[R] = v3[j % 3];
		S(&b3)[R] = v3[(j + 2) % 3];
		S(&c3)[R] = v3[(j + 1) % 3];
		if constexpr (LEVELS == 3) {
			form(2, a2, b2, c2, [&](int k, typename F::L lap) { write(P - 2, k, odd(b2[k], lap)); });
			return;
		}
		form(2, a2, b2, c2, [&](int k, typename F::L lap) { a3[k] = odd(b2[k], lap); });
		publish(3, w, a3);
		if (depth < 4) return;
		form(3, a3, b3, c3, [&](int k, typename F::L lap) { write(P - 3, k, even(b3[k], lap, c2[k])); });
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
