// steps2d.hpp -- 2-D Allen-Cahn and Cahn-Hilliard, several explicit steps per
// pass in registers: one wave per (strip of columns, chunk of rows).
//
// A pass is a chain of LEVELS, each a radius-1 stencil of the one before:
// Allen-Cahn (allen-cahn.cpp:68-71) has one level per step (phi^{n+1} from
// phi^n); Cahn-Hilliard (cahn-hilliard.cpp:69-76) has two (mu^n from c^n, then
// c^{n+1} from mu^n and c^n). Lane l of the wave holds column c0 - L + l of
// every level (L = LEVELS) and level s is right on lanes s .. 63 - s, so the
// wave writes 64 - 2L columns; column neighbours move by DPP wave shifts, row
// neighbours sit in registers. The wave marches down the rows: at iteration t
// row t of level 0 has arrived and level s forms its row t - s, each from the
// three newest rows of the level before. Three row slots per level whose roles
// rotate over a six-row unrolled march, so nothing is copied; level 0 has six,
// three of them in flight. No LDS, no barriers, and what a level would have
// written to memory stays in registers.
//
// Every value is the one-step kernels' for that node and step, formed from
// the same operands in the same order (the halo recomputes what the
// neighbouring strip or chunk computes), so a pass gives the bits of single
// steps. Boundaries: an axis is periodic on both sides or on neither. Periodic:
// lanes and rows past the edge hold the wrapped nodes. Otherwise a level's
// boundary node takes check_boundary's neighbour (MMSP.utility.cpp:42-57) of
// that same level: itself (Neumann, Dirichlet) or its inner neighbour
// (mirror); what lies outside is formed but never read. Only waves that reach
// such an edge run the bodies with those selects (EX for rows, EZ for
// columns: eight more instructions a level in double for each).
#pragma once

#include "tiles.hpp"

namespace mmspx {

// wave shifts whose end lanes (0, resp. 63) receive zero: those lanes are
// outside every level's valid lanes, and with no value to keep the shift needs
// no copy of its source first (and in float folds into the add that uses it)
__device__ __forceinline__ int shift_prev(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x138, 0xf, 0xf, true); }
__device__ __forceinline__ int shift_next(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x130, 0xf, 0xf, true); }
__device__ __forceinline__ float shift_prev(float v) { return __builtin_bit_cast(float, shift_prev(__builtin_bit_cast(int, v))); }
__device__ __forceinline__ float shift_next(float v) { return __builtin_bit_cast(float, shift_next(__builtin_bit_cast(int, v))); }
__device__ __forceinline__ double shift_prev(double v)
{
	const int2 s = __builtin_bit_cast(int2, v);
	return __builtin_bit_cast(double, make_int2(shift_prev(s.x), shift_prev(s.y)));
}
__device__ __forceinline__ double shift_next(double v)
{
	const int2 s = __builtin_bit_cast(int2, v);
	return __builtin_bit_cast(double, make_int2(shift_next(s.x), shift_next(s.y)));
}

// Keeps a store's value computed where it stands (not moved under the store's
// condition, which would split the march into a branch per row and the lane
// shifts from the arithmetic they fold into).
template <typename T>
__device__ __forceinline__ void keep_value(T& v)
{
	asm volatile("" : "+v"(v));
}
// A row's start, the same for every lane, in scalar registers: accesses at a
// lane's byte offset from it take the offset from one vector register (and not a
// 64-bit vector sum per row, some of them kept through the march).
template <typename T>
using GlobalT = __attribute__((address_space(1))) T;
template <typename T>
__device__ __forceinline__ GlobalT<T>* scalar_row(T* p)
{
	GlobalT<T>* q = (GlobalT<T>*)p;
	asm volatile("" : "+s"(q));
	return q;
}
template <typename T>
__device__ __forceinline__ T load_at(const T* row, unsigned byte)
{
	return *(const GlobalT<T>*)((const GlobalT<char>*)scalar_row(row) + byte);
}
template <typename T>
__device__ __forceinline__ void store_at(T* row, unsigned byte, T v)
{
	*(GlobalT<T>*)((GlobalT<char>*)scalar_row(row) + byte) = v;
}

enum { S2_AC = 0, S2_CH = 1, S2_CH_DW = 2 };

// The two-axis laplacian of y in the reference's order. yh - 2y is one fma:
// 2y is exact, so it rounds as the subtraction does. The reference adds the
// first axis to zero, which changes only a -0.0 to +0.0; ZERO keeps that add.
// It can be left out where the sign of a zero laplacian cannot reach the
// result: a zero axis term is -0.0 only at a node whose value is +0.0, where
// Allen-Cahn's +0 - (+-0) is +0 and the double well's mu is +0 - (+-0) = +0;
// and a lap mu of -0.0 needs a mu of +0.0, which no node with c = -0.0 has
// beside neighbours with mu = -0.0, so c + (+-0) is the same.
template <int PREC, bool UNIT, bool ZERO>
__device__ __forceinline__ typename Form<PREC>::L lap2(const Geom& g, typename Form<PREC>::S xh,
                                                       typename Form<PREC>::S xl, typename Form<PREC>::S zh,
                                                       typename Form<PREC>::S zl, typename Form<PREC>::S y)
{
	using S = typename Form<PREC>::S;
	S tx, tz;
	if constexpr (PREC == MMSPX_F64) {
		tx = __builtin_fma(-2.0, y, xh) + xl;
		tz = __builtin_fma(-2.0, y, zh) + zl;
	} else {
		// the shifted neighbours fold into the subtract and the add
		tx = __builtin_fmaf(-2.0f, y, xh) + xl;
		tz = (zh - 2.0f * y) + zl;
	}
	if constexpr (!UNIT) {
		tx = (PREC == MMSPX_F64 ? (S)g.w[0] : (S)g.wf[0]) * tx;
		tz = (PREC == MMSPX_F64 ? (S)g.w[1] : (S)g.wf[1]) * tz;
	}
	return (ZERO ? S(0) + tx : tx) + tz;
}

// The updates with every coefficient one (r = u = K = 1: nr is -1), where the
// multiplications by them are exact and are left out: three of Allen-Cahn's 22
// double operations (1000 steps of 512^2 1275 -> 1205 us, 256^3 27.7 -> 25.0 us
// per step, the reference chemical potential on 333 x 517 walls 490 -> 472).
template <int PREC>
__device__ __forceinline__ typename Form<PREC>::S cube(typename Form<PREC>::S y)
{
	if constexpr (PREC == MMSPX_F64) return cube_cr(y);
	else return y * y * y;
}
template <int PREC>
__device__ __forceinline__ typename Form<PREC>::S mu_unit(typename Form<PREC>::S c, typename Form<PREC>::L lap)
{
	return (-c + cube<PREC>(c)) - lap;
}
template <int PREC>
__device__ __forceinline__ typename Form<PREC>::S ac_unit(typename Form<PREC>::S y, typename Form<PREC>::L lap,
                                                          const ModelParams& p)
{
	return y - (PREC == MMSPX_F64 ? (typename Form<PREC>::S)p.dtM : (typename Form<PREC>::S)p.dtMf) * mu_unit<PREC>(y, lap);
}
static inline bool unit_coefficients(const ModelParams& p)
{
	return p.nr == -1.0 && p.u == 1.0 && p.K == 1.0 && p.nrf == -1.0f && p.uf == 1.0f && p.Kf == 1.0f;
}

// One pass over columns [c0, c0 + 64 - 2L) and rows [xb, xe): `levels` <= L
// levels (L where FULL). UNIT 1: both grid weights are exactly 1, 2: and every
// coefficient (their multiplications are left out; the bits are the same).
template <int PREC, int MODEL, int L, bool EX, bool EZ, int UNIT, bool FULL>
__device__ __forceinline__ void steps2d_body(const typename Form<PREC>::S* __restrict__ a,
                                        typename Form<PREC>::S* __restrict__ b, const Geom& g, const ModelParams& p,
                                        int c0, int xb, int xe, int levels)
{
	using F = Form<PREC>;
	using S = typename F::S;
	constexpr int U = 6;  // rows per turn of the unrolled march (level 0's slots)
	const int lane = threadIdx.x & 63;
	const int nx = g.n[0], ny = g.n[1];
	const int nl = FULL ? L : levels;
	const int c = c0 - L + lane;
	const unsigned cm = (unsigned)tile_map(c, ny, g.b0[1], g.b1[1]);
	const bool out = lane >= L && lane < 64 - L && c < ny;
	const bool zlo = EZ && c == 0, zhi = EZ && c == ny - 1;
	const bool zlm = g.b0[1] == MMSPX_MIRROR, zhm = g.b1[1] == MMSPX_MIRROR;
	const int base = xb - nl;   // level 0's row at iteration 0
	const int tend = xe - xb + 2 * nl;
	// level 0's rows arrive in order; rows past the last one the chunk reads
	// load that row again, rows outside a non-periodic axis (never read) the
	// edge row. Row bookkeeping is scalar: every lane has the same rows.
	int tl = 0, raw = base, wr = wrap(base, nx);
	auto ld = [&]() {
		const int row = EX ? min(max(raw, 0), nx - 1) : wr;
		const S v = (a + (size_t)row * ny)[cm];
		if (++tl < tend) {
			raw++;
			wr = wr + 1 == nx ? 0 : wr + 1;
		}
		return v;
	};

	S l0[U];       // level 0, row t in slot t % 6
	S lv[L][3];    // level s >= 1 in lv[s - 1], row r in slot r % 3
#pragma unroll
	for (int s = 0; s < L; s++) lv[s][0] = lv[s][1] = lv[s][2] = 0;
	// level s at iteration t (t6 = t mod 6, known at compile time)
	auto at = [&](int s, int r) -> S { return s == 0 ? l0[r % U] : lv[s - 1][r % 3]; };
	auto level = [&](int s, int t, int t6) {
		// rows r-1, r, r+1 of level s-1, r = t - s (t6 + 12 - s keeps the slot index positive)
		const int r = t6 + 12 * 3 - s;
		const S y = at(s - 1, r);
		S xl = at(s - 1, r - 1), xh = at(s - 1, r + 1);
		S zl = shift_prev(y), zh = shift_next(y);
		const int x = base + t - s;
		if constexpr (EX) edge_mu(xl, xh, y, x, nx, g.b0[0], g.b1[0]);
		if constexpr (EZ) {
			const S ol = zl, oh = zh;
			if (zlo) zl = zlm ? oh : y;
			if (zhi) zh = zhm ? ol : y;
		}
		const typename F::L lap = lap2<PREC, UNIT != 0, MODEL == S2_CH>(g, xh, xl, zh, zl, y);
		S v;
		if constexpr (MODEL == S2_AC) v = UNIT == 2 ? ac_unit<PREC>(y, lap, p) : F::ac(y, lap, p);
		else if (s & 1)
			v = MODEL == S2_CH_DW ? (UNIT == 2 ? F::mu_dw1(y, lap) : F::mu_dw(y, lap, p))
			                      : (UNIT == 2 ? mu_unit<PREC>(y, lap) : F::mu_poly(y, lap, p));
		else v = F::ch(at(s - 2, r), lap, p);
		lv[s - 1][r % 3] = v;
		if (FULL ? s == L : s == nl) {
			if (out) (b + (size_t)x * ny)[c] = v;
		}
	};
	l0[0] = ld();
	l0[1] = ld();
	l0[2] = ld();
	l0[3] = l0[4] = l0[5] = 0;
	if constexpr (FULL) {
		// the first 2L iterations: level s starts at iteration 2s
#pragma unroll
		for (int t = 0; t < 2 * L; t++) {
			l0[(t + 3) % U] = ld();
#pragma unroll
			for (int s = 1; s <= L; s++)
				if (2 * s <= t) level(s, t, t % U);
		}
		for (int t = 2 * L;; t += U) {
#pragma unroll
			for (int u = 0; u < U; u++) {
				if (t + u >= tend) return;
				const int t6 = (2 * L + u) % U;
				l0[(t6 + 3) % U] = ld();
#pragma unroll
				for (int s = 1; s <= L; s++) level(s, t + u, t6);
			}
		}
	} else {
		for (int t = 0;; t += U) {
#pragma unroll
			for (int u = 0; u < U; u++) {
				if (t + u >= tend) return;
				l0[(u + 3) % U] = ld();
#pragma unroll
				for (int s = 1; s <= L; s++)
					if (s <= nl && 2 * s <= t + u) level(s, t + u, u);
			}
		}
	}
}

template <int PREC, int MODEL, int L, bool EDGES, int UNIT, bool FULL>
__device__ __forceinline__ void steps2d(const typename Form<PREC>::S* __restrict__ a,
                                        typename Form<PREC>::S* __restrict__ b, const Geom& g, const ModelParams& p,
                                        int c0, int xb, int xe, int levels)
{
	if constexpr (EDGES) {
		// the rows and columns a level forms stay inside the grid, or wrap
		const bool ex = g.b0[0] != MMSPX_PERIODIC && (xb < L || xe + L > g.n[0]);
		const bool ez = g.b0[1] != MMSPX_PERIODIC && (c0 < L || c0 - L + 64 > g.n[1]);
		if (ez && g.b0[0] != MMSPX_PERIODIC) {
			steps2d_body<PREC, MODEL, L, true, true, UNIT, FULL>(a, b, g, p, c0, xb, xe, levels);
			return;
		}
		if (ez) {
			steps2d_body<PREC, MODEL, L, false, true, UNIT, FULL>(a, b, g, p, c0, xb, xe, levels);
			return;
		}
		if (ex) {
			steps2d_body<PREC, MODEL, L, true, false, UNIT, FULL>(a, b, g, p, c0, xb, xe, levels);
			return;
		}
	}
	steps2d_body<PREC, MODEL, L, false, false, UNIT, FULL>(a, b, g, p, c0, xb, xe, levels);
}

}  // namespace mmspx
