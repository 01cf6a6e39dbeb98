// fmarch.hpp -- 3-D periodic grain growth and Zener pinning, L explicit steps
// per pass: a plane march with a wave's lanes along axis 2 and one field per
// wave.
//
// A workgroup of 16 waves takes a tile of 16/Q * R - 2 (L - 1) rows and 64 - 2 L
// columns of the (axis 1, axis 2) plane and all Q fields: wave h holds R rows
// (of the tile and its halo) of field h % Q. Levels as in wmarch4.hpp: level s
// is phi^{n+s}, the iteration at plane P forms level s at plane P - s + 1, lane
// l holds column z0 - L + l, axis-2 neighbours move by DPP wave shifts, axis-0
// neighbours and the wave's own rows are registers (three slots a level, roles
// rotating over a three-plane unrolled march). What a point needs from other
// waves, sum_j phi_j^2 (graingrowth.cpp:91-97) and the rows beside the wave's,
// goes through LDS: at the end of an iteration every wave publishes the planes
// the next one is centred on, all waves then sum squares in field order, one
// row each in turn, and fetch the rows beside theirs; two barriers a plane.
//
// Every value is the one-step kernels' for that node and step, from the same
// operands in the same order (KIND 3 holds field 0, zener.cpp:117-135), so a
// pass gives the bits of single steps.
//
// Bound by the exchange and vector work together: 256^3 x 8 FP32 in three-step
// passes of 500 us moves 2.4 TB/s, vector work (2.4e8 instructions a launch) is
// about 46 % of the time at 2.4 cycles each, and the waves wait 38 % of theirs at
// the two barriers; no bank conflicts. R and L
// are what 128 registers a lane hold (6 to 12 values a row). Stores go under
// one condition a row and all addresses are a scalar row start plus one lane
// offset: left to itself the compiler kept a 64-bit address per row in vector
// registers and moved each row's arithmetic under its store's condition (8 rows
// x 3 steps then spilled 89 registers).
#pragma once

#include "steps2d.hpp"

namespace mmspx {

template <int PREC, int Q, int KIND, int R, int L, int LEVELS, bool UNIT>
__device__ __forceinline__ void fmarch(const typename Form<PREC>::S* __restrict__ a,
                                       typename Form<PREC>::S* __restrict__ b, const Geom& g, const ModelParams& p,
                                       int y0, int z0, int xb, int xe)
{
	using F = Form<PREC>;
	using S = typename F::S;
	using Sum = typename F::Sum;
	constexpr int NW = 16, G = NW / Q, RY = G * R, H = L - 1, TY = RY - 2 * H;
	static_assert(G >= 2 && TY > 0, "two or more row groups");
	__shared__ S vals[LEVELS][Q][RY][64];
	__shared__ Sum tot[LEVELS][RY][64];

	const int nx = g.n[0], ny = g.n[1], nz = g.n[2];
	const int64_t plane = (int64_t)ny * nz;
	const size_t N = (size_t)nx * plane;
	const int lane = threadIdx.x & 63;
	const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
	const int q = wv % Q, grp = wv / Q, r0 = grp * R;
	const int z = z0 - L + lane;
	// a row's address is scalar, the lane's byte offset in it 32 bits
	const unsigned zc = (unsigned)wrap(z, nz) * (unsigned)sizeof(S);
	auto uniform = [](int v) { return (unsigned)__builtin_amdgcn_readfirstlane(v); };
	const bool zout = lane >= L && lane < 64 - L && z < nz;
	unsigned row[R];
#pragma unroll
	for (int k = 0; k < R; k++) {
		const int r = r0 + k, y = y0 - H + r;
		row[k] = uniform(wrap(y, ny)) * (unsigned)nz;
	}
	// the rows that are written: H <= r < TY + H and y < ny
	const int klo = H - r0, khi = min(TY + H, ny - y0 + H) - r0;
	const bool first = grp == 0, last = grp == G - 1;
	const unsigned rrow = uniform(wrap(first ? y0 - L : y0 + TY + H, ny)) * (unsigned)nz;
	const S* __restrict__ af = a + (size_t)q * N;
	S* __restrict__ bf = b + (size_t)q * N;
	int wx = (int)uniform(wrap(xb - L, nx));
	S rgc = 0, rgn = 0;  // the ring row at planes P+1, P+2
	unsigned o = zc;
	auto load = [&](S (&v)[R]) {
		const S* s = af + (int64_t)wx * plane;
		wx = wx + 1 == nx ? 0 : wx + 1;
		rgc = rgn;
		keep_value(o);
#pragma unroll
		for (int k = 0; k < R; k++) v[k] = load_at(s + row[k], o);
		if (first || last) {
			keep_value(o);
			rgn = load_at(s + rrow, o);
		}
	};

	S f[3][R];          // level 0 at P-1, P, P+1: plane i in slot i % 3
	S v[L][3][R];       // level s >= 1 in v[s]: what iteration i formed in slot i % 3
	S up[L], dn[L];     // rows beside the wave's
#pragma unroll
	for (int s = 1; s < LEVELS; s++)
#pragma unroll
		for (int k = 0; k < R; k++) v[s][0][k] = v[s][1][k] = v[s][2][k] = 0;

	// the planes the next iteration's levels are centred on: their fields to
	// LDS, the sums of squares in field order, the rows beside the wave's
	auto exchange = [&](const S (&c)[R], int j) {
#pragma unroll
		for (int k = 0; k < R; k++) vals[0][q][r0 + k][lane] = c[k];
#pragma unroll
		for (int s = 1; s < LEVELS; s++)
#pragma unroll
			for (int k = 0; k < R; k++) vals[s][q][r0 + k][lane] = v[s][j][k];
		__syncthreads();
#pragma unroll
		for (int s = 0; s < LEVELS; s++) {
			up[s] = s == 0 ? rgc : S(0);
			dn[s] = s == 0 ? rgc : S(0);
			if (!first) up[s] = vals[s][q][r0 - 1][lane];
			if (!last) dn[s] = vals[s][q][r0 + R][lane];
		}
#pragma unroll
		for (int s = 0; s < LEVELS; s++)
#pragma unroll 1
			for (int r = wv; r < RY; r += NW) {
				Sum acc = 0;
#pragma unroll
				for (int i = 0; i < Q; i++) {
					const Sum u = vals[s][i][r][lane];
					acc += u * u;
				}
				tot[s][r][lane] = acc;
			}
		__syncthreads();
	};
	// level s + 1 from level s: values h, m, l at the planes after, at and before
	auto form = [&](int s, const S (&h)[R], const S (&m)[R], const S (&l)[R], auto value) {
#pragma unroll
		for (int k = 0; k < R; k++) {
			const S y = m[k];
			if (KIND == 3 && q == 0) {
				value(k, y);  // the particles keep their values
				continue;
			}
			const S yl = k > 0 ? m[k > 0 ? k - 1 : 0] : up[s], yh = k < R - 1 ? m[k < R - 1 ? k + 1 : 0] : dn[s];
			S tx, ty, tz;
			if constexpr (PREC == MMSPX_F64) {
				tx = __builtin_fma(-2.0, y, h[k]) + l[k];
				ty = __builtin_fma(-2.0, y, yh) + yl;
				tz = __builtin_fma(-2.0, y, shift_next(y)) + shift_prev(y);
			} else {
				tx = __builtin_fmaf(-2.0f, y, h[k]) + l[k];
				ty = __builtin_fmaf(-2.0f, y, yh) + yl;
				tz = (shift_next(y) - 2.0f * y) + shift_prev(y);
			}
			if constexpr (!UNIT) {
				tx = (PREC == MMSPX_F64 ? (S)g.w[0] : (S)g.wf[0]) * tx;
				ty = (PREC == MMSPX_F64 ? (S)g.w[1] : (S)g.wf[1]) * ty;
				tz = (PREC == MMSPX_F64 ? (S)g.w[2] : (S)g.wf[2]) * tz;
			}
			const typename F::L lap = (tx + ty) + tz;
			value(k, F::gg(y, tot[s][r0 + k][lane], lap, p));
		}
	};
	// the iteration at plane P = xb - H + i; j = i mod 3 is known at compile
	// time, depth the levels whose first plane has been reached
	auto iter = [&](int i, int j, int depth) {
		const int P = xb - H + i;
		S(&fm)[R] = f[j % 3];
		S(&fc)[R] = f[(j + 1) % 3];
		S(&fp)[R] = f[(j + 2) % 3];
		auto write = [&](int x, int k, S val) {
			if (LEVELS < L && (x < xb || x >= xe)) return;
			keep_value(val);
			if (k >= klo && k < khi)
				if (zout) {
					keep_value(o);
					store_at(bf + (int64_t)x * plane + row[k], o, val);
				}
		};
#pragma unroll
		for (int s = 1; s <= LEVELS; s++) {
			if (s > depth) break;
			auto value = [&](int k, S val) {
				if (s == LEVELS) write(P - (s - 1), k, val);
				else v[s][j][k] = val;
			};
			if (s == 1) form(0, fp, fc, fm, value);
			else form(s - 1, v[s - 1][j], v[s - 1][(j + 2) % 3], v[s - 1][(j + 1) % 3], value);
			if (s == 1) load(fm);  // plane P+2 takes P-1's slot
		}
		exchange(fp, j);
	};
	load(f[0]);
	load(f[1]);
	load(f[2]);
	exchange(f[1], 0);  // rgc is the ring row of the first centre plane, xb - L + 1
	const int n = xe - xb + H + LEVELS - 1;
#pragma unroll
	for (int i = 0; i < 2 * H; i++) iter(i, i % 3, 1 + i / 2);
	for (int i = 2 * H;; i += 3) {
#pragma unroll
		for (int u = 0; u < 3; u++) {
			if (i + u >= n) return;
			iter(i + u, (2 * H + u) % 3, L);
		}
	}
}

}  // namespace mmspx
