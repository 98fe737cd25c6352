// Passes over one FP64 statevector and its tangent (gfx950): a tile of 2^K amplitudes is loaded into
// LDS, all gates of a pass are applied there and the tile is written back.
//
// A gate alone moves its arrays once (an HVP at 18 qubits: 16 MB forward, 24 MB reverse, 5 and 11 us
// per launch from the last-level cache, 51 gates 0.89 ms); a pass moves them once for up to 18 gates
// (4 passes; 0.34 ms, with host copies taken out 0.31 and the outer products on the matrix cores 0.29).
// The reverse pass starts at the pass's last state and takes the gates back with G^-1, so that a
// state is kept per pass instead of per gate.  Two threads of a wave own a quad of amplitudes per
// gate, two rows of every product each: vector FMAs have the rate of the FP64 matrix products here,
// and the quad needs no operand layout.  The outer products are matrix products over 16 quads, their
// operands read again from LDS: as vector products and lane exchanges they took 255 of 563 vector
// instructions per wave and gate (20 qubits: 930 us against 890, 10 qubits 139 against 130).
#pragma once

#include "rqc_tile_kernels.hpp"

namespace rqc {

constexpr int kStateK = 10;        // tile qubits: 16 KB per array; 256 tiles at 18 qubits
constexpr int kStateThreads = 512; // two per quad
constexpr int kStateArray = 16 << kStateK;

struct StateGate
{
	int pi, pj;     // tile bits of the gate's wires
	int index;      // circuit gate, the place of its sums
	int first;      // the circuit's first: the tangent before it is zero
};
struct alignas(16) StateOp
{
	zc g[16], z[16], ginv[16], w[16];   // w = G^-1 Z G^-1
	StateGate gate;
};
constexpr int kStateMats = 64;     // matrix entries of an op
// LDS: the arrays, two gates' matrices and (reverse) two gates' sums of each wave, both in turn
constexpr int state_lds_bytes(bool rev)
{
	return (rev ? 4 : 2) * kStateArray + 2 * kStateMats * 16 + (rev ? 2 * kStateThreads * 8 : 0);
}

// index bits of the tile bits 0 .. K - 1, then those of the tile number's bits
struct StateTile
{
	int K, L;
	int bit[32];
};

__device__ __forceinline__ unsigned state_slot(unsigned e) { return (e ^ ((e >> 4) & 15) ^ ((e >> 8) & 15)) * 16; }

__device__ __forceinline__ long state_deposit(const int* bit, int n, unsigned x)
{
	long r = 0;
	for (int t = 0; t < n; t++) { r |= (long)((x >> t) & 1) << bit[t]; }
	return r;
}

// the value of lane n of each 16 lanes
template <int N> __device__ __forceinline__ double row_value(double v)
{
	return __longlong_as_double(__builtin_amdgcn_mov_dpp(__double_as_longlong(v), 0x150 + N, 0xf, 0xf, true));
}
// the value of lane + N (mod 16) of each 16 lanes
template <int N> __device__ __forceinline__ double row_rotate(double v)
{
	const long b = __double_as_longlong(v);
	const unsigned lo = __builtin_amdgcn_mov_dpp((int)(b & 0xffffffff), 0x120 + N, 0xf, 0xf, true),
		hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), 0x120 + N, 0xf, 0xf, true);
	return __longlong_as_double((long)(((unsigned long)hi << 32) | lo));
}
__device__ __forceinline__ zc of_lane(zc v, int n)
{
	// (n is a constant after unrolling)
	switch (n) {
#define RQC_LANE(N) case N: return {row_value<N>(v.x), row_value<N>(v.y)};
	RQC_LANE(0) RQC_LANE(1) RQC_LANE(2) RQC_LANE(3) RQC_LANE(4) RQC_LANE(5) RQC_LANE(6) RQC_LANE(7)
	RQC_LANE(8) RQC_LANE(9) RQC_LANE(10) RQC_LANE(11) RQC_LANE(12) RQC_LANE(13) RQC_LANE(14)
	default: return {row_value<15>(v.x), row_value<15>(v.y)};
#undef RQC_LANE
	}
}

// s = a b or s += a b
__device__ __forceinline__ void mac_first(zc& s, zc a, zc b, bool first)
{
	if (first) { s = zc{fma(-a.y, b.y, a.x * b.x), fma(a.y, b.x, a.x * b.y)}; }
	else { cmac(s, a, b); }
}

// Forward (REV = false): (a, da) -> (oa, oda) through the pass's gates; da null: zero tangent.
// Reverse: (a, da) the pass's last state and tangent, (f, df) the adjoint and its tangent after the
// pass, replaced by those before it in (of, odf) unless null; sums of gate `index` and tile t at
// part[(index gridDim.x + t) kWidth].
//
// At 18 qubits a CU has one tile, two waves per SIMD, and a gate takes 1.4 us forward and 3.1 us
// reverse: bound by the chain of LDS reads, products and the barrier.  The gates' matrices come
// through LDS, loaded a gate ahead, an entry per lane and broadcast inside 16 lanes: from scalar
// loads, each waiting for the cache, a gate took 2.8 and 5.7 us, and with one thread per quad 2.0
// and 4.4; four threads per quad (16 waves) gave nothing at 18 qubits and lost 20 % at 20.
template <bool REV>
__global__ __launch_bounds__(kStateThreads, 2) void k_state_pass(const StateOp* __restrict__ ops, int nops, StateTile T,
	const zc* a, const zc* da, const zc* f, const zc* df, zc* oa, zc* oda, zc* __restrict__ part)
{
	extern __shared__ __align__(16) char lds_raw[];
	constexpr int A = kStateArray;
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nt = blockDim.x;
	// the thread's half of the rows and its quad: a wave owns 32 quads, so that its reads of a quad
	// precede its writes without a barrier
	const int h = lane >> 5, quad = 32 * wave + (lane & 31);
	// (tiles of fewer than 8 qubits: zeros up to a quad per lane)
	const unsigned ne = 1u << T.K, nz = max(ne, 256u);
	const long base = state_deposit(T.bit + T.K, T.L - T.K, blockIdx.x), mine = base | state_deposit(T.bit, T.K, tid);
	for (unsigned n = 0; n < nz; n += nt) {
		const bool in = tid + n < ne;
		const long off = in ? mine | state_deposit(T.bit, T.K, n) : base;
		const unsigned p = state_slot(tid + n);
		auto put = [&](unsigned at, const zc* v) { lds_store_cxd(p + at, in && v != nullptr ? v[off] : zc{0, 0}); };
		put(0, a);
		put(A, da);
		if (REV) {
			put(2 * A, f);
			put(3 * A, df);
		}
	}
	constexpr int M = (REV ? 4 : 2) * A;
	double* sums = reinterpret_cast<double*>(lds_raw + M + 2 * kStateMats * 16);
	auto op = [&](int j) { return ops + (REV ? nops - 1 - j : j); };
	auto matrices = [&](int j) { return reinterpret_cast<const zc*>(op(j))[tid]; };
	auto put = [&](int j, zc v) { lds_store_cxd(M + (j & 1) * (kStateMats * 16) + tid * 16, v); };
	StateGate next = op(0)->gate;
	if (tid < kStateMats) { put(0, matrices(0)); }
	int stored = -1;
	auto store = [&](int j) {
		if (stored >= 0 && tid < 2 * kWidth) {
			// double tid of the sums: matrix, row, column, part (lane 16 row + 8 matrix + 4 part + column)
			const int i = 16 * ((tid >> 3) & 3) + 8 * (tid >> 5) + 4 * (tid & 1) + ((tid >> 1) & 3);
			double s = 0;
			for (int w = 0; w < nt / 64; w++) { s += sums[(j & 1) * kStateThreads + w * 64 + i]; }
			reinterpret_cast<double*>(part + ((long)stored * gridDim.x + blockIdx.x) * kWidth)[tid] = s;
		}
	};
#pragma unroll 1
	for (int j = 0; j < nops; j++) {
		const StateGate o = next;
		zc ahead = {0, 0};
		if (j + 1 < nops) {
			next = op(j + 1)->gate;
			if (tid < kStateMats) { ahead = matrices(j + 1); }
		}
		__syncthreads();
		if (REV) { store(j - 1); }
		const unsigned b = state_slot((unsigned)quad_base(quad, min(o.pi, o.pj), max(o.pi, o.pj)));
		const unsigned si = state_slot(1u << o.pi), sj = state_slot(1u << o.pj);
		const unsigned m = M + (j & 1) * (kStateMats * 16);
		// G, Z, G^-1 and G^-1 Z G^-1, an entry per lane of 16: (2 h + r, c) or, for the transposed
		// products, (r, 2 h + c) at lane 4 r + c
		const unsigned by_row = m + ((lane + 8 * h) & 15) * 16, by_col = m + ((lane & 12) + ((lane + 2 * h) & 3)) * 16;
		const zc mg = lds_load_cxd(REV ? by_col : by_row), mz = lds_load_cxd((REV ? by_col : by_row) + 256);
		const unsigned at[4] = {b, b ^ sj, b ^ si, b ^ si ^ sj};
		const unsigned to[2] = {b ^ (si & -(unsigned)h), b ^ sj ^ (si & -(unsigned)h)};
		zc x[4], dx[4], y[2], dy[2];
#pragma unroll
		for (int k = 0; k < 4; k++) {
			x[k] = lds_load_cxd(at[k]);
			dx[k] = lds_load_cxd(at[k] + A);
		}
		auto put_before = [&]() {
#pragma unroll
			for (int k = 0; k < 2; k++) {
				lds_store_cxd(to[k], y[k]);
				lds_store_cxd(to[k] + A, dy[k]);
			}
		};
		if constexpr (!REV) {
#pragma unroll
			for (int r = 0; r < 2; r++) {
#pragma unroll
				for (int c = 0; c < 4; c++) {
					const zc g = of_lane(mg, 4 * r + c);
					mac_first(y[r], g, x[c], c == 0);
					mac_first(dy[r], g, dx[c], c == 0);
					cmac(dy[r], of_lane(mz, 4 * r + c), x[c]);
				}
			}
			put_before();
		} else {
			const zc mi = lds_load_cxd(by_row + 512), mw = lds_load_cxd(by_row + 768);
			zc fx[4], dfx[4], u[2], du[2];
#pragma unroll
			for (int k = 0; k < 4; k++) {
				fx[k] = lds_load_cxd(at[k] + 2 * A);
				dfx[k] = lds_load_cxd(at[k] + 3 * A);
			}
			// the outer products' operands (4 x 4 x 4 matrix products over 16 quads): amplitude lane & 3 of quad
			// 4 ((lane >> 2) & 3) + (lane >> 4)
			const int lo = min(o.pi, o.pj), hi = max(o.pi, o.pj);
			const unsigned mb = state_slot((unsigned)quad_base(32 * wave + (lane & 12) + (lane >> 4), lo, hi)) ^
				(sj & -(unsigned)(lane & 1)) ^ (si & -(unsigned)((lane >> 1) & 1));
			const unsigned mo[2] = {mb, mb ^ state_slot((unsigned)quad_base(16, lo, hi))};
			GateOperands<double, 2> oa, os;
			auto operand = [&](unsigned at) {
				const zc v = lds_load_cxd(at), d = lds_load_cxd(at + A);
				return double4_t{v.x, v.y, d.x, d.y};
			};
			for (int n = 0; n < 2; n++) { oa.acc[n] = operand(mo[n] + 2 * A); }
			// before the gate: G^-1 x and its tangent G^-1 dx - G^-1 Z G^-1 x
			const bool dzero = o.first != 0;
#pragma unroll
			for (int r = 0; r < 2; r++) {
				zc t;
#pragma unroll
				for (int c = 0; c < 4; c++) {
					const zc gi = of_lane(mi, 4 * r + c);
					mac_first(y[r], gi, x[c], c == 0);
					mac_first(dy[r], gi, dx[c], c == 0);
					mac_first(t, of_lane(mw, 4 * r + c), x[c], c == 0);
				}
				dy[r] = dzero ? zc{0, 0} : dy[r] - t;
			}
			put_before();
			__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
			for (int n = 0; n < 2; n++) { os.acc[n] = operand(mo[n]); }
			// the adjoint before the gate: G^T f, its tangent G^T df + Z^T f
#pragma unroll
			for (int c = 0; c < 2; c++) {
#pragma unroll
				for (int r = 0; r < 4; r++) {
					const zc g = of_lane(mg, 4 * r + c);
					mac_first(u[c], g, fx[r], r == 0);
					mac_first(du[c], g, dfx[r], r == 0);
					cmac(du[c], of_lane(mz, 4 * r + c), fx[r]);
				}
			}
#pragma unroll
			for (int k = 0; k < 2; k++) {
				lds_store_cxd(to[k] + 2 * A, u[k]);
				lds_store_cxd(to[k] + 3 * A, du[k]);
			}
			double4_t c = {0, 0, 0, 0};
			outer44<2>(os, oa, c);
			for (int n = 0; n < 4; n++) {
				c[n] += row_rotate<8>(c[n]);
				c[n] += row_rotate<4>(c[n]);
			}
			sums[(j & 1) * kStateThreads + tid] = (lane & 8) ? ((lane & 4) ? c[3] : c[2]) : ((lane & 4) ? c[1] : c[0]);
			stored = o.index;
		}
		if (tid < kStateMats) { put(j + 1, ahead); }
	}
	__syncthreads();
	if (REV) { store(nops - 1); }
	if (oa != nullptr) {
		for (unsigned n = 0; tid + n < ne; n += nt) {
			const long off = mine | state_deposit(T.bit, T.K, n);
			const unsigned p = state_slot(tid + n) + (REV ? 2 * A : 0);
			oa[off] = lds_load_cxd(p);
			oda[off] = lds_load_cxd(p + A);
		}
	}
}

}  // namespace rqc
