// Cyclic-product sweeps (gfx950): the array M = W_{<=m} U^dagger W_{>m} and, for Hessian-vector
// products, its derivative dM, multiplied by gates from both sides (see rqc_cyc_plan.hpp for the
// method and the layouts).
//
// A tile is 2^K row bits by 2^K column bits of the array.  A workgroup loads it into LDS, applies
// its launch's gate products there and writes it back in the next launch's bit order.  One product
// M <- A M B runs on 4 x 4 blocks (the row quad of A's gate by the column quad of B's) with both
// factors applied in registers: the block is the first operand of the right product, whose result
// lands in the layout of the second operand of the left product, so that a pair of gates costs one
// LDS read and one write.
//
// Bounds and figures (FP64, L = 14, depth 9, against the column sweeps on the same card): HVP 63.8 ms
// (112.9), its launches 41 and 44 TFLOP/s issued where the products alone run at 52 (matrix product
// peak 72) and the transfers alone at 4.2 to 5.0 TB/s (stream copy 6.3): the products and the
// transfers overlap, both at about 4/5 of a tile's time.  L = 12, depth 7 gradient 1.03 ms (3.55),
// bound by LDS writes (a 16-byte write takes 13 cycles per wave, a read 5.5) and transfers.
#pragma once

#include "rqc_tile_kernels.hpp"
#include "rqc_cyc_plan.hpp"

namespace rqc {

// the launch's jobs and their arrays (M, dM)
struct CycArgs
{
	CycJob job[2];
	const void* in[2][2];
	void* out[2][2];
};

// a product's descriptor (CycOp): 12 directions, the matrices, barrier, record
typedef int cyc_op_t __attribute__((ext_vector_type(16)));
static_assert(sizeof(CycOp) == sizeof(cyc_op_t), "descriptor size");

template <int K, bool DUAL> constexpr int cyc_state_bytes() { return (DUAL ? 32 : 16) << (2 * K); }
constexpr int cyc_mats_per_op(bool dual) { return dual ? 4 : 2; }
template <int K, bool DUAL> constexpr int cyc_lds_bytes()
{
	return cyc_state_bytes<K, DUAL>() + kCycOps * cyc_mats_per_op(DUAL) * 256;
}

// the pointer's counterpart in copy i of its region
template <typename P>
__device__ __forceinline__ P* copy_of(P* p, long stride, int i)
{
	typedef typename std::conditional<std::is_const<P>::value, const char, char>::type byte;
	return reinterpret_cast<P*>(reinterpret_cast<byte*>(p) + stride * i);
}

// XOR of the terms selected by the bits of x (masks, so that the terms' loads are unconditional)
template <typename T>
__device__ __forceinline__ T cyc_select(const T* terms, int n, long x)
{
	T r = 0;
	for (int t = 0; t < n; t++) { r ^= terms[t] & -(T)((x >> t) & 1); }
	return r;
}

// the value of lane `l` of a wave
__device__ __forceinline__ long lane_value(long v, int l)
{
	const unsigned lo = __builtin_amdgcn_readlane((int)(v & 0xffffffff), l), hi = __builtin_amdgcn_readlane((int)(v >> 32), l);
	return (long)(((unsigned long)hi << 32) | lo);
}

// OUT (compile-time, so that the stores' place among the loads is known): the fill then waits for
// the next tile's loads alone, not for the stores issued after them (one counter, in order).
template <int K, bool DUAL, typename TS, bool OUT, int LW = 2 * (K - 4)>
__global__ __launch_bounds__(64 << LW, LW >= 2 * (K - 4) ? 4 : 2) void k_cyc_sweep(const CycArgs A, const cx<double>* __restrict__ mats,
	zc* __restrict__ part, long nparts, zc* __restrict__ trace, long stride, const int* skip)
{
	if (skipped(skip)) { return; }
	// evaluation blockIdx.z of several of one plan, `stride` bytes apart (tables, parts and arrays; U shared)
	mats = copy_of(mats, stride, blockIdx.z);
	part = copy_of(part, stride, blockIdx.z);
	trace = copy_of(trace, stride, blockIdx.z);
	extern __shared__ __align__(16) char lds_raw[];
	constexpr int LT = 6 + LW, NT = 1 << LT, NW = NT / 64;
	constexpr int LE = 2 * K - LT, NE = 1 << LE;   // elements per thread (the highest index bits)
	constexpr int NG = 1 << (2 * K - 6 - LW);      // groups of 64 elements per wave and product
	constexpr int DOFF = 4096;                     // LDS bytes from an element of M to that of dM
	constexpr int MB = cyc_state_bytes<K, DUAL>(); // LDS bytes of the gate matrices
	constexpr int NM = DUAL ? 2 : 1;
	typedef TS vec2 __attribute__((ext_vector_type(2)));
	const CycJob& J = A.job[blockIdx.y];
	const long ntiles = 1L << J.ngen;
	if ((long)blockIdx.x >= ntiles) { return; }
	const int tid = threadIdx.x, lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int flags = J.flags;
	const long in_stride = (flags & kCycReadU) ? 0 : stride;
	const vec2* in0 = copy_of(static_cast<const vec2*>(A.in[blockIdx.y][0]), in_stride, blockIdx.z);
	const vec2* in1 = copy_of(static_cast<const vec2*>(A.in[blockIdx.y][1]), in_stride, blockIdx.z);
	const lds_d2* inU = static_cast<const lds_d2*>(A.in[blockIdx.y][0]);
	vec2* out0 = copy_of(static_cast<vec2*>(A.out[blockIdx.y][0]), stride, blockIdx.z);
	vec2* out1 = copy_of(static_cast<vec2*>(A.out[blockIdx.y][1]), stride, blockIdx.z);

	// the gate matrices of the products: left factors transposed, right ones as they are, so that
	// a lane's operand entry is at 4 (lane >> 4) + (lane & 3) in both
	for (int e = tid; e < J.nops * 2 * NM * 16; e += NT) {
		const int t = e & 15, w = (e >> 4) % NM, side = (e / (16 * NM)) & 1, j = e / (32 * NM);
		const int m = side ? J.op[j].mb : J.op[j].ma;
		if (m >= 0) {
			const int pos = side ? t : 4 * (t & 3) + (t >> 2);
			lds_store_cxd(MB + (e - t + pos) * 16, mats[((long)m + w) * 16 + t]);
		}
	}
	// the thread's terms of a load and of a store (NE elements each: the highest index bits)
	const int ip = cyc_select(J.ipos, LT, tid), op = cyc_select(J.opos, LT, tid);
	const long io = cyc_select(J.ioff, LT, tid), oo = cyc_select(J.ooff, LT, tid);
	// (M = U^dagger, dM = 0 at the first launch: U is FP64 in either storage)
	constexpr bool WIDE = sizeof(TS) == 8;
	vec2 pm[NE], pd[NE];
	lds_d2 pu[WIDE ? 1 : NE];
	const bool read_u = flags & kCycReadU;
	const double usign = read_u ? -1.0 : 1.0;
	// A workgroup's tiles are blockIdx.x + n gridDim.x, the grid a power of two: from n to n + 1 the
	// index bits up to the lowest zero bit of n change, so lane t holds the XOR of the terms of the
	// t + 1 lowest bits of n (one lane read per tile and no memory)
	const int lgrid = 31 - __builtin_clz(gridDim.x);
	long ibase = cyc_select(J.tin, J.ngen, blockIdx.x), obase = cyc_select(J.tout, J.ngen, blockIdx.x);
	long istep = 0, ostep = 0;
	for (int t = lgrid; t < J.ngen; t++) {
		const long on = -(long)(t - lgrid <= lane);
		istep ^= J.tin[t] & on;
		ostep ^= J.tout[t] & on;
	}
	auto load = [&]() {
#pragma unroll
		for (int k = 0; k < NE; k++) {
			const long off = ibase ^ io ^ cyc_select(J.ioff + LT, LE, k);
			if constexpr (WIDE) { pm[k] = in0[off]; }
			else if (read_u) { pu[k] = inU[off]; }
			else { pm[k] = in0[off]; }
			if constexpr (DUAL) { pd[k] = read_u ? vec2{0, 0} : in1[off]; }
		}
	};
	auto fill = [&]() {
#pragma unroll
		for (int k = 0; k < NE; k++) {
			const unsigned p = (unsigned)(ip ^ cyc_select(J.ipos + LT, LE, k));
			if constexpr (WIDE) {
				lds_store_cxd(p, cx<double>{pm[k].x, usign * pm[k].y});
			} else {
				const lds_d2 v = read_u ? pu[k] : lds_d2{(double)pm[k].x, (double)pm[k].y};
				lds_store_cxd(p, cx<double>{v.x, usign * v.y});
			}
			if constexpr (DUAL) { lds_store_cxd(p + DOFF, cx<double>{(double)pd[k].x, (double)pd[k].y}); }
		}
	};
	// lane index bits of the operand layouts: l & 3, (l >> 2) & 3, l >> 4
	int lm[6];
#pragma unroll
	for (int t = 0; t < 6; t++) { lm[t] = -((lane >> t) & 1); }
	const int fi = (4 * (lane >> 4) + (lane & 3)) * 16;

	long tile = blockIdx.x;
	load();
	fill();
	__syncthreads();
	for (int n = 1; ; n++) {
		const long next = tile + gridDim.x;
		const int bit = __builtin_ctz(n);
		if (next < ntiles) {
			ibase ^= lane_value(istep, bit);
			load();
		}
		// whether row and column agree in every bit outside the tile, and the tile's place among those
		const long pair = tile >> J.nd;
		const bool diag = (((pair ^ (pair >> 1)) & 0x5555555555555555L) & ((1L << (J.ngen - J.nd)) - 1)) == 0;
#pragma unroll 1
		for (int j = 0; j < J.nops; j++) {
			// (the whole descriptor in one scalar load)
			const cyc_op_t q = reinterpret_cast<const cyc_op_t*>(J.op)[j];
			if (q[14] & 1) { __syncthreads(); }
			const bool ha = q[12] >= 0, hb = q[13] >= 0;
			int wb = 0;
			bool dw = true;   // the wave's elements: row and column agree in the wave bits
			int di = 0, rg = 0;
#pragma unroll
			for (int t = 0; t < K - 4; t++) {
				// (a column bit that is a group bit of the wave's: the record's group has it equal)
				const int r = (wave >> (2 * t)) & 1, c = (2 * t + 1 < LW) ? (wave >> (2 * t + 1)) & 1 : 0;
				wb ^= (q[8 + 2 * t] & -r) ^ (q[9 + 2 * t] & -c);
				if (2 * t + 1 < LW) { dw = dw && r == c; }
				else { rg = q[9 + 2 * t] & -r; }
				di |= r << t;
			}
			const int blk = (lm[2] & q[4]) ^ (lm[3] & q[5]) ^ wb;
			// the element a lane reads (row quad index l & 3, column l >> 4) and writes (the reverse)
			const int la = blk ^ (lm[0] & q[0]) ^ (lm[1] & q[1]) ^ (lm[4] & q[2]) ^ (lm[5] & q[3]);
			const int sa = blk ^ (lm[4] & q[0]) ^ (lm[5] & q[1]) ^ (lm[0] & q[2]) ^ (lm[1] & q[3]);
			const int ld = hb ? la : sa;
			// the wave's groups
			int gd[NG];
#pragma unroll
			for (int g = 0; g < NG; g++) { gd[g] = ((g & 1) ? q[6] : 0) ^ ((g & 2) ? q[7] : 0) ^ ((g & 4) ? q[8 + LW] : 0); }
			if (q[15] >= 0 && diag && dw) {
				// the gate's partial trace: the sum of the blocks with equal row and column bits, four of
				// them the wave's
				auto comb = [&](int m) { return (q[4] & -(m & 1)) ^ (q[5] & -((m >> 1) & 1)) ^ (q[6] & -((m >> 2) & 1)) ^ (q[7] & -((m >> 3) & 1)); };
				const int ra = wb ^ rg ^ (lm[2] & comb(q[14] >> 8)) ^ (lm[3] & comb(q[14] >> 12)) ^ (lm[0] & q[0]) ^ (lm[1] & q[1]) ^
					(lm[4] & q[2]) ^ (lm[5] & q[3]);
				cx<double> v[NM];
#pragma unroll
				for (int s = 0; s < NM; s++) {
					v[s] = lds_load_cxd((unsigned)ra + s * DOFF);
					v[s].x += __shfl_xor(v[s].x, 4);
					v[s].y += __shfl_xor(v[s].y, 4);
					v[s].x += __shfl_xor(v[s].x, 8);
					v[s].y += __shfl_xor(v[s].y, 8);
				}
				if ((lane & 12) == 0) {
					long t = tile & ((1L << J.nd) - 1);
					for (int i = 0; i < (J.ngen - J.nd) / 2; i++) { t |= ((pair >> (2 * i)) & 1) << (J.nd + i); }
					zc* d = part + ((long)q[15] * nparts + ((t << (K - 4)) | di)) * (16 * NM);
#pragma unroll
					for (int s = 0; s < NM; s++) { d[16 * s + 4 * (lane & 3) + (lane >> 4)] = v[s]; }
				}
			}
			const unsigned mj = MB + j * (2 * NM * 256) + fi;
			auto frag = [&](unsigned at) {
				const cx<double> x = lds_load_cxd(at);
				if constexpr (DUAL) {
					const cx<double> y = lds_load_cxd(at + 256);
					return Frag44{x.x, x.y, y.x, y.y, x.x + x.y, x.y - x.x, y.x + y.y, y.y - y.x};
				} else {
					return Frag44{x.x, x.y, 0.0, 0.0, x.x + x.y, x.y - x.x, 0.0, 0.0};
				}
			};
			// dual: (M, dM) of two groups per step; plain: M of four groups
			constexpr int NST = NG / (DUAL ? 2 : 4);
			auto run = [&](auto hac, auto hbc) {
				constexpr bool HA = decltype(hac)::value, HB = decltype(hbc)::value;
				GateOperands<double, 2> o[NST];
				auto load_step = [&](int s) {
#pragma unroll
					for (int n = 0; n < 2; n++) {
						if constexpr (DUAL) {
							o[s].x[n] = lds_load_cxd((unsigned)(ld ^ gd[2 * s + n]));
							o[s].y[n] = lds_load_cxd((unsigned)(ld ^ gd[2 * s + n]) + DOFF);
						} else {
							o[s].x[n] = lds_load_cxd((unsigned)(ld ^ gd[4 * s + 2 * n]));
							o[s].y[n] = lds_load_cxd((unsigned)(ld ^ gd[4 * s + 2 * n + 1]));
						}
					}
				};
				load_step(0);
				const Frag44 fb = HB ? frag(mj + NM * 256) : Frag44{};
				const Frag44 fa = HA ? frag(mj) : Frag44{};
#pragma unroll
				for (int s = 0; s < NST; s++) {
					// the next step's operands load in the shadow of this one's products (the steps'
					// elements are disjoint)
					if (s + 1 < NST) { load_step(s + 1); }
					__builtin_amdgcn_sched_barrier(0);
					__builtin_amdgcn_s_setprio(1);
					if constexpr (HB) {
						if constexpr (DUAL) { gate_mfma44_t<2>(fb, o[s]); }
						else { gate_mfma44_pair_t<2>(fb, o[s]); }
					}
					if constexpr (HA && HB) {
#pragma unroll
						for (int n = 0; n < 2; n++) {
							o[s].x[n] = cx<double>{o[s].acc[n][0], o[s].acc[n][1]};
							o[s].y[n] = cx<double>{o[s].acc[n][2], o[s].acc[n][3]};
						}
					}
					if constexpr (HA) {
						if constexpr (DUAL) { gate_mfma44<2>(fa, o[s]); }
						else { gate_mfma44_pair<2>(fa, o[s]); }
					}
					__builtin_amdgcn_s_setprio(0);
#pragma unroll
					for (int n = 0; n < 2; n++) {
						const cx<double> x = {o[s].acc[n][0], o[s].acc[n][1]}, y = {o[s].acc[n][2], o[s].acc[n][3]};
						if constexpr (DUAL) {
							lds_store_cxd((unsigned)(sa ^ gd[2 * s + n]), x);
							lds_store_cxd((unsigned)(sa ^ gd[2 * s + n]) + DOFF, y);
						} else {
							lds_store_cxd((unsigned)(sa ^ gd[4 * s + 2 * n]), x);
							lds_store_cxd((unsigned)(sa ^ gd[4 * s + 2 * n + 1]), y);
						}
					}
				}
			};
			if (ha && hb) { run(std::true_type{}, std::true_type{}); }
			else if (ha) { run(std::true_type{}, std::false_type{}); }
			else if (hb) { run(std::false_type{}, std::true_type{}); }
		}
		__syncthreads();
		if (!OUT && (flags & kCycTrace)) {
			// the elements whose row and column agree in every bit
			zc s = {0, 0};
#pragma unroll
			for (int k = 0; k < NE; k++) {
				const cx<double> v = lds_load_cxd((unsigned)(op ^ cyc_select(J.opos + LT, LE, k)));
				if ((obase ^ oo ^ cyc_select(J.ooff + LT, LE, k)) == 0) { s += v; }
			}
#pragma unroll
			for (int o = 32; o > 0; o >>= 1) {
				s.x += __shfl_xor(s.x, o);
				s.y += __shfl_xor(s.y, o);
			}
			if (lane == 0) { trace[tile * NW + wave] = s; }
		}
		if constexpr (OUT) {
			const long base = obase ^ oo;
#pragma unroll
			for (int k = 0; k < NE; k++) {
				const unsigned p = (unsigned)(op ^ cyc_select(J.opos + LT, LE, k));
				const long off = base ^ cyc_select(J.ooff + LT, LE, k);
				const cx<double> m = lds_load_cxd(p);
				out0[off] = vec2{(TS)m.x, (TS)m.y};
				if constexpr (DUAL) {
					const cx<double> d = lds_load_cxd(p + DOFF);
					out1[off] = vec2{(TS)d.x, (TS)d.y};
				}
			}
		}
		if (next >= ntiles) { break; }
		__syncthreads();
		fill();
		__syncthreads();
		tile = next;
		obase ^= lane_value(ostep, bit);
	}
}

// Sum of a gate's recorded partial traces R = Tr_rest M, dR = Tr_rest dM in a fixed order (one
// workgroup per execution slot), decoded to its gradient and HVP sums.  Recorded after the gate
// (M = G E): Tr_rest E = G^-1 R and its derivative G^-1 dR + W R, W = -G^-1 Z G^-1; before it
// (M = E G): R G^-1 and dR G^-1 + R W.  The gradient of f = -Tr(G E) by G[r][c] is -E[c][r].
// order: circuit gate of the slot and its side.  Slot fslot writes f = -Tr M: the slot recorded first,
// whose M has seen the forward products alone (the first gate's has been conjugated all the way back:
// 6 qubits, 9 layers, |f| about 1: root mean square error of f 1.15e-15 there, 0.61e-15 here).
template <bool DUAL>
__global__ __launch_bounds__(256) void k_cyc_reduce(const zc* __restrict__ part, long nparts, const int* __restrict__ order,
	const zc* __restrict__ rmats, zc* __restrict__ acc, int fslot, long stride, const int* skip)
{
	if (skipped(skip)) { return; }
	part = copy_of(part, stride, blockIdx.y);
	rmats = copy_of(rmats, stride, blockIdx.y);
	acc = copy_of(acc, stride, blockIdx.y);
	constexpr int NE = DUAL ? 32 : 16, NS = 256 / NE;
	__shared__ zc red[NS][NE];
	const int x = blockIdx.x, e = threadIdx.x & (NE - 1), p0 = threadIdx.x / NE;
	const zc* p = part + (long)x * nparts * NE + e;
	zc s = {0, 0};
#pragma unroll 4
	for (long i = p0; i < nparts; i += NS) { s += p[i * NE]; }
	red[p0][e] = s;
	__syncthreads();
	if (threadIdx.x < NE) {
		for (int i = 1; i < NS; i++) { s += red[i][e]; }
		red[0][e] = s;
	}
	__syncthreads();
	const zc* R = red[0];
	if (x == fslot && threadIdx.x == 0) {
		const zc t = R[0] + R[5] + R[10] + R[15];
		acc[0] = zc{-t.x, -t.y};
	}
	if (threadIdx.x < 32) {
		// rmats: G^-T and W^T
		const zc* Q = rmats + 32L * x;
		const zc* WT = Q + 16;
		const int h = threadIdx.x >> 4, c = (threadIdx.x >> 2) & 3, r = threadIdx.x & 3;   // entry (r, c) of E
		const bool up = order[2 * x + 1] != 0;
		zc v = {0, 0};
		if (h == 0 || DUAL) {
			for (int k = 0; k < 4; k++) {
				if (up) {
					cmac(v, R[16 * h + 4 * r + k], Q[4 * c + k]);
					if (h) { cmac(v, R[4 * r + k], WT[4 * c + k]); }
				} else {
					cmac(v, Q[4 * k + r], R[16 * h + 4 * k + c]);
					if (h) { cmac(v, WT[4 * k + r], R[4 * k + c]); }
				}
			}
		}
		acc[1 + 32L * order[2 * x] + 16 * h + 4 * c + r] = zc{-v.x, -v.y};
	}
}

// Tables of the HVPs along the unit directions E_rc on every gate of one group (the columns of a
// Hessian): column c0 + blockIdx.y (group (c0 + y) / 16, entry (c0 + y) mod 16), at tab + y stride
// bytes, from the table of the circuit without directions.  One thread per 4x4 entry of a slot:
// Z = E_rc, W = -G^-1 E_rc G^-1 = -(column r of G^-1) (row c of it), zero for the other groups' gates.
__global__ __launch_bounds__(kBlock) void k_cyc_unit_tables(const char* __restrict__ base, char* __restrict__ tab, long stride,
	long bytes, long rmats_off, long order_off, int G, int per, int c0)
{
	char* t = tab + stride * blockIdx.y;
	const long first = (long)blockIdx.x * kBlock + threadIdx.x, step = (long)gridDim.x * kBlock;
	const int col = c0 + blockIdx.y, group = col >> 4, r = (col >> 2) & 3, c = col & 3;
	const int* order = reinterpret_cast<const int*>(base + order_off);
	const zc* mats = reinterpret_cast<const zc*>(base);
	const long nm = (long)G * kMats * 16, nr = (long)G * 32, r0 = rmats_off / (long)sizeof(zc);
	for (long i = first; i < bytes / (long)sizeof(zc); i += step) {
		zc v = reinterpret_cast<const zc*>(base)[i];
		const bool in_m = i < nm, in_r = i >= r0 && i < r0 + nr;
		if (in_m || in_r) {
			const long k = in_m ? i : i - r0;
			const int x = (int)(in_m ? k / (16 * kMats) : k / 32), w = (int)((k >> 4) % (in_m ? kMats : 2)), e = (int)(k & 15);
			if (order[2 * x] / per == group) {
				const zc* gi = mats + ((long)x * kMats + kMatGinv) * 16;
				const int a = e >> 2, b = e & 3;
				auto wm = [&](int i2, int j2) { return -(gi[4 * i2 + r] * gi[4 * c + j2]); };
				const zc one = {1, 0}, zero = {0, 0};
				if (in_r) { if (w == 1) { v = wm(b, a); } }
				else if (w == kMatZ) { v = (a == r && b == c) ? one : zero; }
				else if (w == kMatZT) { v = (b == r && a == c) ? one : zero; }
				else if (w == kMatW) { v = wm(a, b); }
			}
		}
		reinterpret_cast<zc*>(t)[i] = v;
	}
}

// f = -sum of the trace parts, in a fixed order
__global__ __launch_bounds__(kBlock) void k_cyc_trace(const zc* __restrict__ part, long n, zc* __restrict__ acc, const int* skip)
{
	if (skipped(skip)) { return; }
	zc s = {0, 0};
#pragma unroll 4
	for (long i = threadIdx.x; i < n; i += kBlock) { s += part[i]; }
	zc r[1] = {s};
	__shared__ zc res[1];
	block_sum_store<1>(r, res);
	__syncthreads();
	if (threadIdx.x == 0) { acc[0] = zc{-res[0].x, -res[0].y}; }
}

}  // namespace rqc
