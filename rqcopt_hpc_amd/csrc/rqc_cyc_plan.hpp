// Host planning of the cyclic-product sweeps (rqc_cyc_kernels.hpp).
//
// The target of a circuit W = W_G ... W_1 is f = -Tr(U^dagger W).  With
//   M_k = W_{<=k} U^dagger W_{>k}       (k gates on the left, the rest on the right)
// every M_k has the trace of U^dagger W, and gate k's environment E_k = W_{<k} U^dagger W_{>k}
// follows from M_k = G_k E_k = G_k M_{k-1} G_k^{-1}, so the partial trace of M_k over the qubits
// outside the gate holds the gate's whole gradient, and that of its derivative dM_k along the
// directions the gate's Hessian-vector product.  One N x N array (two with directions) is swept:
//   forward     M_m = W_{<=m} U^dagger W_{>m}: the first m passes multiply from the left (row bits),
//               the others from the right (column bits), one of each per launch
//   conjugation from M_m downwards M_{k-1} = G_k^{-1} M_k G_k and upwards M_k = G_k M_{k-1} G_k^{-1}
//               (two jobs per launch), recording every gate's partial trace on the way
// No state is checkpointed and nothing is summed over N^2 terms: a partial trace reads the
// elements whose row and column agree outside the gate.  Per amplitude and gate a forward product
// costs 9 block products per 64 elements of (M, dM) and a conjugation 18, against 9 and 30 of the
// column sweeps (recovery, adjoint and outer products), and two arrays move instead of four.  That also bounds what the last passes
// need: the elements whose row and column agree outside the qubits that the remaining passes
// touch (the "free" qubits), 1 / 2^(L-K) of the array for the last pass.
//
// The array is a vector over 2 L index bits (row bit of qubit bit b: id L + b, column bit: id b).
// A launch's tile fixes all bits but K row bits and K column bits.  Each launch writes the array
// in the bit order the next one reads best: the next tile's bits lowest (a tile is one contiguous
// run of 4^K elements), and lowest among them bits that this launch's tile shares, so that its
// stores cover runs as well.
#pragma once

#include <algorithm>
#include <array>
#include <cstdint>
#include <vector>

#include "rqc_pass_search.hpp"

namespace rqc {

constexpr int kCycOps = 8;     // most two-sided gate products of a launch's job
constexpr int kCycBits = 12;   // most tile bits
constexpr int kCycGens = 20;   // most index bits outside a tile (with aligned row and column bits as one)

enum { kCycReadU = 1, kCycNoOut = 2, kCycTrace = 4 };

// One product M <- A M B on a 4 x 4 block per (row quad, column quad); A acts on the two row bits,
// B on the two column bits (-1: absent).  dir: LDS byte offsets of the directions of the lane's
// element: row quad bits lo, hi, column quad bits lo, hi, block bits x, y, group bits, wave bits.
struct alignas(64) CycOp
{
	int dir[kCycBits];
	int ma, mb;     // matrix of the pass's table (the tangent matrix follows it), -1: none
	int barrier;    // bit 0: the waves own other elements than at the previous product; bits 8-11, 12-15:
	                // the combinations of x, y and the group bits that keep row and column bits equal
	int rec;        // execution slot whose partial trace is recorded from the operands, -1: none
};

struct CycJob
{
	int nops, ngen, nd, flags;     // nd: index bits shared by row and column (the first of the ngen)
	CycOp op[kCycOps];
	int ipos[kCycBits], opos[kCycBits];     // LDS byte offset of bit t of a load's / store's index
	long ioff[kCycBits], ooff[kCycBits];    // its element offset in memory (kCycTrace: ooff, tout mark
	long tin[kCycGens], tout[kCycGens];     // the qubits whose row and column differ by that bit)
};

struct CycLaunch
{
	int njobs = 0;
	bool reverse = false;
	CycJob job[2];
	int in[2] = {-1, -1}, out[2] = {-1, -1};   // array pairs (-1: U, or no output)
	double gate_sides[2] = {0, 0};             // one-sided gate products per tile
};

struct CycPass
{
	std::vector<int> slots;   // execution slots of its gates, in order
	std::vector<int> q;       // its K qubit bits, ascending
};

struct CycPlan
{
	int L = 0, K = 0, nbuf = 0;
	std::vector<CycLaunch> launches;
	std::vector<int> up;      // per slot: recorded before (1, upward) or after (0, downward) its gate
	int fslot = 0;            // the slot recorded first, from M_m itself, whose trace gives f
	long ntrace = 0;          // tiles of the tracing launch (target evaluations)
};

// parts of a gate's partial trace: diagonal tiles times diagonal waves
inline long cyc_parts(int L, int K) { return (1L << (L - K)) << (K - 4); }

// LDS byte offset of tile position p (both arrays of a dual sweep in blocks of 256 elements, so
// that the second array is a constant instruction offset away)
inline int cyc_lds_byte(int p, bool dual) { return dual ? ((p >> 8) << 13) | ((p & 255) << 4) : p << 4; }

namespace cyc_detail {

struct SideOp
{
	int a = -1, ma = 0, b = -1, mb = 0, rec = -1;   // slots and table matrices of the two factors
};

// colours of a step's row and column bits by qubit bit
struct Colouring
{
	std::vector<int> r, c;   // indexed by qubit bit, 0 outside the tile
	int beta(int id, int L) const { return id >= L ? r[id - L] : c[id] << 2; }
};

struct Step
{
	std::vector<int> rows, cols;   // qubit bits of the tile, ascending
	std::vector<SideOp> ops;
	Colouring col;
	unsigned fout = 0;             // free qubits of its output
	bool conj = false;
	int flags = 0;
};

// three colours (1, 2, 3) such that the two bits of every listed gate differ, evenly used: two
// colours are two independent vectors of GF(2)^2, the bank term of the bit
inline std::vector<int> colours(const std::vector<int>& q, const std::vector<std::pair<int, int>>& edges)
{
	const int n = (int)q.size();
	std::vector<std::vector<int>> nb(n);
	auto at = [&](int b) { return (int)(std::find(q.begin(), q.end(), b) - q.begin()); };
	for (auto& e : edges) { nb[at(e.first)].push_back(at(e.second)); nb[at(e.second)].push_back(at(e.first)); }
	std::vector<int> order(n), col(n, 0);
	for (int i = 0; i < n; i++) { order[i] = i; }
	std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return nb[x].size() > nb[y].size(); });
	int used[4] = {0, 0, 0, 0};
	for (int i : order) {
		int best = 0;
		for (int c = 1; c <= 3; c++) {
			bool taken = false;
			for (int u : nb[i]) { taken |= (col[u] == c); }
			if (!taken && (best == 0 || used[c] < used[best])) { best = c; }
		}
		if (best == 0) {
			for (int c = 1; c <= 3; c++) { if (best == 0 || used[c] < used[best]) { best = c; } }
		}
		col[i] = best;
		used[best]++;
	}
	return col;
}

// The span of vectors of GF(2)^4 as a bit set of its 16 elements (1: the zero vector alone)
inline unsigned span_add(unsigned span, int v)
{
	if ((span >> v) & 1) { return span; }
	unsigned t = span;
	if (v & 1) { t = ((t & 0x5555) << 1) | ((t >> 1) & 0x5555); }
	if (v & 2) { t = ((t & 0x3333) << 2) | ((t >> 2) & 0x3333); }
	if (v & 4) { t = ((t & 0x0f0f) << 4) | ((t >> 4) & 0x0f0f); }
	if (v & 8) { t = ((t & 0x00ff) << 8) | ((t >> 8) & 0x00ff); }
	return span | t;
}
inline int span_rank(unsigned span) { return __builtin_ctz((unsigned)__builtin_popcount(span)); }

// Bank conflicts of 16-byte LDS accesses by the XOR-linear slots d0 .. d5 of the lane index bits
// (measured): a read's 16-lane phases are the lanes with one parity of bits 2, 3, 4 (lane bit 5
// apart), free of conflicts iff d0, d1, d2 + d3, d2 + d4 are independent mod 16 slots (the read's
// rank, 4); a write takes 8 consecutive lanes at half the rate, at full speed iff d0, d1, d2 have
// rank 2 mod 8 slots.
inline int cyc_write_rank(int d0, int d1, int d2) { return std::min(2, span_rank(span_add(span_add(span_add(1, d0 & 7), d1 & 7), d2 & 7))); }

// the combination of four independent vectors of GF(2)^4 that gives v
inline int cyc_combination(const int* basis, int v)
{
	for (int m = 0; m < 16; m++) {
		int s = 0;
		for (int t = 0; t < 4; t++) { if ((m >> t) & 1) { s ^= basis[t]; } }
		if (s == v) { return m; }
	}
	return 0;
}

}  // namespace cyc_detail

// Passes of the circuit (gate k on qubit bits bi[k], bj[k]), at most gmax gates each.  Among the plans
// with the fewest passes found the search takes the one whose successive passes share qubits best (two
// shared qubits are the four index bits of a 256-byte run that both launches move whole) and whose first
// pass holds the lowest qubit bits (runs of U's rows).  Qubits that a pass does not need are filled up
// with its neighbours'.
inline std::vector<CycPass> plan_cyc_passes(int L, const std::vector<int>& bi, const std::vector<int>& bj, int K, int gmax)
{
	PassSearch S{L, K, gmax, {}, false, true};
	for (size_t k = 0; k < bi.size(); k++) { S.gm.push_back((1u << bi[k]) | (1u << bj[k])); }
	const std::vector<FoundPass> plan = search_passes(S, [&](unsigned last, unsigned u) {
		if (last == 0) {
			int run = 0;
			while (run < 3 && ((u >> run) & 1)) { run++; }
			return std::max(0, 3 - run - (K - __builtin_popcount(u)));
		}
		const int ov = __builtin_popcount(last & u) + 2 * K - __builtin_popcount(last) - __builtin_popcount(u);
		return ov >= 2 ? 0 : ov == 1 ? 2 : 5;
	});
	// fill the passes' sets up to K qubits: the neighbours' first (and the lowest bits for the first)
	const int P = (int)plan.size();
	std::vector<unsigned> q;
	for (const FoundPass& p : plan) { q.push_back(p.used); }
	for (int p = 0; p < P; p++) {
		auto fill = [&](unsigned from) {
			for (int b = 0; b < L && __builtin_popcount(q[p]) < K; b++) { if ((from >> b) & 1) { q[p] |= 1u << b; } }
		};
		const unsigned a = p > 0 ? q[p - 1] : 7u, b = p + 1 < P ? q[p + 1] : 0u;
		fill(a & b);
		if (p > 0 && __builtin_popcount(q[p] & a) >= 2) { fill(b); }
		fill(a);
		fill(b);
		fill((L >= 32) ? ~0u : (1u << L) - 1);
	}
	std::vector<CycPass> out;
	for (int p = 0; p < P; p++) {
		CycPass c;
		c.slots = plan[p].gates;
		for (int b = 0; b < L; b++) { if ((q[p] >> b) & 1) { c.q.push_back(b); } }
		out.push_back(c);
	}
	return out;
}

inline unsigned cyc_qubits(const std::vector<int>& q)
{
	unsigned m = 0;
	for (int b : q) { m |= 1u << b; }
	return m;
}

// passes multiplied from the left: the split with the least work, by the conjugation work that the
// shrinking free sets leave
inline int cyc_split(int L, int K, const std::vector<CycPass>& passes, bool target_only)
{
	const int P = (int)passes.size();
	if (target_only) { return (P + 1) / 2; }
	// the work of every pass on either side: log2 of its tiles counts the bits outside the tile, and
	// a qubit that is not free and outside the tile's rows and columns once
	std::vector<double> left(P + 1, 0), right(P + 1, 0);   // of the first n, of the last n passes
	for (int side = 0; side < 2; side++) {
		unsigned f = 0;
		for (int i = 0; i < P; i++) {
			const CycPass& p = passes[side == 0 ? i : P - 1 - i];
			const unsigned q = cyc_qubits(p.q);
			const int gens = (L - __builtin_popcount(q)) + __builtin_popcount(f & ~q);
			(side == 0 ? left : right)[i + 1] = (side == 0 ? left : right)[i] +
				((double)p.slots.size() + 4.0) * (double)(1UL << gens);
			f |= q;
		}
	}
	int m = 0;
	double best = -1;
	for (int s = 0; s <= P; s++) {
		double w = left[s];
		w += right[P - s];
		w += std::max(s, P - s) * 2.0 * (double)(1UL << (2 * (L - K)));
		if (best < 0 || w < best) { best = w; m = s; }
	}
	return m;
}

// array pairs (one array without directions) of P passes split at m: the forward launches use two in
// turn, and see the jobs' arrays in make_cyc_plan
inline int cyc_arrays(int P, int m, bool target_only)
{
	const int F = std::max(m, P - m), longer = F, shorter = P - F;
	if (target_only) { return std::min(F - 1, 2); }
	return shorter >= 2 ? 4 : longer >= 3 ? 3 : longer == 2 ? 2 : 1;
}

// least arrays of any circuit of G gates (before its passes are known)
inline int cyc_least_arrays(int G, bool target_only)
{
	const int P = (G + kCycOps - 1) / kCycOps;
	return target_only ? cyc_arrays(P, (P + 1) / 2, true) : P <= 2 ? 1 : P == 3 ? 2 : 3;
}

// bi, bj: qubit bits of slot x's wires (the more significant gate index first); m: cyc_split's; with
// target only, the forward launches run to the end and the last one sums the trace
inline CycPlan make_cyc_plan(int L, int K, const std::vector<CycPass>& passes, int m, const std::vector<int>& bi,
	const std::vector<int>& bj, bool target_only, bool dual, int matG, int matGinv)
{
	using namespace cyc_detail;
	const int P = (int)passes.size();
	CycPlan plan;
	plan.L = L;
	plan.K = K;
	plan.up.assign(bi.size(), 0);
	auto qmask = [](const std::vector<int>& q) { return cyc_qubits(q); };
	// steps
	std::vector<Step> fwd, down, up;
	const int F = std::max(m, P - m);
	for (int i = 0; i < F; i++) {
		// the longer side starts first; both end at the split
		const int li = i - (F - m), ri = i - (F - (P - m));
		Step s;
		const CycPass* lp = (li >= 0) ? &passes[li] : nullptr;
		const CycPass* rp = (ri >= 0) ? &passes[P - 1 - ri] : nullptr;
		s.rows = (lp != nullptr ? lp : rp)->q;
		s.cols = (rp != nullptr ? rp : lp)->q;
		const size_t nl = lp != nullptr ? lp->slots.size() : 0, nr = rp != nullptr ? rp->slots.size() : 0;
		for (size_t k = 0; k < std::max(nl, nr); k++) {
			SideOp o;
			if (k < nl) { o.a = lp->slots[k]; o.ma = matG; }
			if (k < nr) { o.b = rp->slots[nr - 1 - k]; o.mb = matG; }   // M G: the last gate first
			s.ops.push_back(o);
		}
		fwd.push_back(s);
	}
	if (F > 1 && m != P - m) {
		// the first launch multiplies from one side: the other side's bits are free to suit U's rows
		// (a right pass alone) and the next launch
		std::vector<int>& side = (m < P - m) ? fwd[0].rows : fwd[0].cols;
		std::vector<int> pick = (m < P - m) ? std::vector<int>{0, 1, 2} : std::vector<int>{};
		for (int b : (m < P - m) ? fwd[1].rows : fwd[1].cols) {
			if ((int)pick.size() < K && std::find(pick.begin(), pick.end(), b) == pick.end()) { pick.push_back(b); }
		}
		std::sort(pick.begin(), pick.end());
		side = pick;
	}
	auto conj_step = [&](const CycPass& p, bool upward, bool last) {
		Step s;
		s.conj = true;
		s.rows = s.cols = p.q;
		const size_t n = p.slots.size();
		for (size_t k = 0; k < n; k++) {
			const int x = upward ? p.slots[k] : p.slots[n - 1 - k];
			SideOp o;
			o.rec = x;
			if (!(last && k + 1 == n)) {
				o.a = o.b = x;
				o.ma = upward ? matG : matGinv;
				o.mb = upward ? matGinv : matG;
			}
			plan.up[x] = upward ? 1 : 0;
			s.ops.push_back(o);
		}
		if (last) { s.flags |= kCycNoOut; }
		return s;
	};
	unsigned fmid = 0;
	if (!target_only) {
		for (int p = m - 1; p >= 0; p--) { down.push_back(conj_step(passes[p], false, p == 0)); }
		for (int p = m; p < P; p++) { up.push_back(conj_step(passes[p], true, p == P - 1)); }
		plan.fslot = (!down.empty() ? down : up)[0].ops[0].rec;
		for (auto* side : {&down, &up}) {
			unsigned f = 0;
			for (int i = (int)side->size() - 1; i >= 0; i--) {
				(*side)[i].fout = f;
				f |= qmask((*side)[i].rows);
			}
			fmid |= f;
		}
	}
	{
		unsigned f = fmid;
		for (int i = F - 1; i >= 0; i--) {
			fwd[i].fout = f;
			f |= qmask(fwd[i].rows) | qmask(fwd[i].cols);
		}
		fwd[0].flags |= kCycReadU;
		if (target_only) { fwd[F - 1].flags |= kCycNoOut | kCycTrace; }
	}
	auto tile_ids = [&](const Step& s) {
		std::vector<char> t(2 * (size_t)L, 0);
		for (int b : s.rows) { t[L + b] = 1; }
		for (int b : s.cols) { t[b] = 1; }
		return t;
	};
	for (auto* steps : {&fwd, &down, &up}) {
		for (Step& s : *steps) {
			s.col.r.assign(L, 0);
			s.col.c.assign(L, 0);
			std::vector<std::pair<int, int>> er, ec;
			for (const SideOp& o : s.ops) {
				const int ra = o.a >= 0 ? o.a : s.conj ? o.rec : -1, cb = o.b >= 0 ? o.b : s.conj ? o.rec : -1;
				if (ra >= 0) { er.emplace_back(bi[ra], bj[ra]); }
				if (cb >= 0) { ec.emplace_back(bi[cb], bj[cb]); }
			}
			const auto cr = colours(s.rows, er), cc = colours(s.cols, ec);
			for (size_t i = 0; i < s.rows.size(); i++) { s.col.r[s.rows[i]] = cr[i]; }
			for (size_t i = 0; i < s.cols.size(); i++) { s.col.c[s.cols[i]] = cc[i]; }
		}
	}
	// memory bit order (id -> position) that step s leaves for its successors (the first primary)
	auto next_layout = [&](const Step& s, const std::vector<const Step*>& succ, const std::vector<int>& pin) {
		const auto ts = tile_ids(s);
		std::vector<std::vector<char>> tn;
		for (auto* n : succ) { tn.push_back(tile_ids(*n)); }
		std::vector<int> common, mid, rest, order;
		for (int id = 0; id < 2 * L; id++) {
			bool in_all = ts[id];
			for (auto& t : tn) { in_all = in_all && t[id]; }
			(in_all ? common : tn[0][id] ? mid : rest).push_back(id);
		}
		auto by_pin = [&](int x, int y) { return pin[x] < pin[y]; };
		for (auto* v : {&common, &mid, &rest}) { std::sort(v->begin(), v->end(), by_pin); }
		// the lowest five: stores of s read LDS, and loads of its successors write it, by these bits
		if (common.size() >= 4) {
			const std::vector<int>& five = common.size() >= 5 ? common : mid;
			int best = -1;
			std::array<int, 5> pick = {};
			const int n = std::min<int>((int)common.size(), 8), n5 = (int)std::min<size_t>(five.size(), 8);
			// bank terms of the candidates in the tile of s (a fifth bit outside it has none) and in its successors'
			int cs[8], c5[8], cn[2][8];
			for (int i = 0; i < n; i++) {
				cs[i] = s.col.beta(common[i], L);
				for (size_t k = 0; k < succ.size(); k++) { cn[k][i] = succ[k]->col.beta(common[i], L); }
			}
			for (int i = 0; i < n5; i++) { c5[i] = s.col.beta(five[i], L); }
			// score: 8 times the stores' read rank and 2 times the loads' write rank, 100 more if both are full
			// (the search ends there); a branch that cannot gain is left out
			auto most = [](int rank, int w) { return rank >= 4 ? 32 + 2 * w + (w == 2 ? 100 : 0) : 8 * rank + 2 * w; };
			for (int a = 0; a < n && best < 100; a++) for (int b = 0; b < n && best < 100; b++) {
				if (a == b) { continue; }
				const unsigned ab = span_add(span_add(1, cs[a]), cs[b]);
				if (most(span_rank(ab) + 2, 2) <= best) { continue; }
				for (int c = 0; c < n && best < 100; c++) {
					if (c == a || c == b) { continue; }
					int w = 2;
					for (size_t k = 0; k < succ.size(); k++) { w = std::min(w, cyc_write_rank(cn[k][a], cn[k][b], cn[k][c])); }
					if (most(span_rank(ab) + 2, w) <= best) { continue; }
					for (int d = 0; d < n && best < 100; d++) {
						if (d == a || d == b || d == c) { continue; }
						const unsigned abd = span_add(ab, cs[c] ^ cs[d]);
						if (most(span_rank(abd) + 1, w) <= best) { continue; }
						for (int e = 0; e < n5; e++) {
							if (&five == &common && (e == a || e == b || e == c || e == d)) { continue; }
							const int sc = most(span_rank(span_add(abd, cs[c] ^ c5[e])), w);
							if (sc > best) { best = sc; pick = {common[a], common[b], common[c], common[d], five[e]}; }
						}
					}
				}
			}
			auto first = [&](std::vector<int>& v, int from, int to) {
				std::vector<int> o(pick.begin() + from, pick.begin() + to);
				for (int id : v) { if (std::find(o.begin(), o.end(), id) == o.end()) { o.push_back(id); } }
				v = o;
			};
			if (&five == &common) { first(common, 0, 5); }
			else { first(common, 0, 4); first(mid, 4, 5); }
		}
		for (auto* v : {&common, &mid, &rest}) { order.insert(order.end(), v->begin(), v->end()); }
		std::vector<int> pos(2 * (size_t)L);
		for (int i = 0; i < 2 * L; i++) { pos[order[i]] = i; }
		return pos;
	};
	const int nb = 2 * K;
	auto build_job = [&](const Step& s, const std::vector<int>& pin, const std::vector<int>& pout, double* sides) {
		CycJob J = {};
		const Colouring& col = s.col;
		J.flags = s.flags;
		J.nops = (int)s.ops.size();
		// tile positions: the four lowest from bits with independent bank terms (the map is then
		// one-to-one), the bank term of the others folded in
		std::vector<int> ids;
		auto add2 = [&](const std::vector<int>& q, const std::vector<int>& c, int off) {
			size_t a = 0, b = 1;
			for (b = 1; b < q.size() && c[q[b]] == c[q[a]]; b++) { }
			ids.push_back(off + q[a]);
			ids.push_back(off + q[b]);
		};
		add2(s.rows, col.r, L);
		add2(s.cols, col.c, 0);
		for (int b : s.rows) { if (std::find(ids.begin(), ids.end(), L + b) == ids.end()) { ids.push_back(L + b); } }
		for (int b : s.cols) { if (std::find(ids.begin(), ids.end(), b) == ids.end()) { ids.push_back(b); } }
		std::vector<int> byte(2 * (size_t)L, 0);
		for (int t = 0; t < nb; t++) {
			byte[ids[t]] = cyc_lds_byte((t < 4 ? 0 : 1 << t) ^ col.beta(ids[t], L), dual);
		}
		// loads and stores run over the tile in memory order
		std::vector<int> oi = ids, oo = ids;
		std::sort(oi.begin(), oi.end(), [&](int x, int y) { return pin[x] < pin[y]; });
		std::sort(oo.begin(), oo.end(), [&](int x, int y) { return pout[x] < pout[y]; });
		const bool trace = s.flags & kCycTrace;
		auto outoff = [&](int id) { return trace ? 1L << (id % L) : 1L << pout[id]; };
		for (int t = 0; t < nb; t++) {
			J.ipos[t] = byte[oi[t]];
			J.ioff[t] = 1L << pin[oi[t]];
			J.opos[t] = byte[oo[t]];
			J.ooff[t] = outoff(oo[t]);
		}
		// bits outside the tile
		const unsigned rm = qmask(s.rows), cm = qmask(s.cols);
		std::vector<std::array<int, 2>> single, pairs;   // (id, -1), or row and column bit together
		for (int b = 0; b < L; b++) {
			const bool ir = rm >> b & 1, ic = cm >> b & 1;
			if (ir && ic) { continue; }
			if (!ir && !ic && !(s.fout >> b & 1)) { pairs.push_back({L + b, b}); continue; }
			if (!ir) { single.push_back({L + b, -1}); }
			if (!ic) { single.push_back({b, -1}); }
		}
		J.nd = (int)pairs.size();
		for (auto* v : {&pairs, &single}) {
			for (auto& g : *v) {
				long ti = 1L << pin[g[0]], to = outoff(g[0]);
				if (g[1] >= 0) { ti ^= 1L << pin[g[1]]; to ^= outoff(g[1]); }
				J.tin[J.ngen] = ti;
				J.tout[J.ngen++] = to;
			}
		}
		// products
		struct Choice { int cl, ch, rl, rh; int ur[2], uc[2]; int x, y, score; int g[2]; };
		// the block directions x, y among four bits (row and column bits of two qubits, bank terms b[0 .. 3])
		// whose reads and writes have the fewest bank conflicts: read s0, s1, x + y, x + t, write w0, w1, x;
		// kept by the terms, since few sets of them occur
		struct Blocks { uint64_t key; int x, y, score; };
		std::array<Blocks, 128> known;
		for (Blocks& k : known) { k.key = 0; }
		auto blocks = [&](const int* b, int s0, int s1, int t, int w0, int w1) {
			const uint64_t key = 1ull << 40 | (uint64_t)s0 << 36 | (uint64_t)s1 << 32 | (uint64_t)t << 28 | (uint64_t)w0 << 24 |
				(uint64_t)w1 << 20 | (uint64_t)(b[0] | b[1] << 4 | b[2] << 8 | b[3] << 12);
			Blocks& r = known[(key * 0x9e3779b97f4a7c15ull) >> 57];
			if (r.key == key) { return r; }
			r = Blocks{key, 0, 0, -1};
			int v[16];
			for (int m = 0; m < 16; m++) { v[m] = (m & 1 ? b[0] : 0) ^ (m & 2 ? b[1] : 0) ^ (m & 4 ? b[2] : 0) ^ (m & 8 ? b[3] : 0); }
			const unsigned base = span_add(span_add(1, s0), s1);
			for (int x = 1; x < 16 && r.score < 36; x++) {
				const int w = 2 * cyc_write_rank(w0, w1, v[x]);
				const unsigned sx = span_add(base, v[x] ^ t);
				if (8 * std::min(4, span_rank(sx) + 1) + w <= r.score) { continue; }
				for (int y = 1; y < 16 && r.score < 36; y++) {
					if (y == x) { continue; }
					const int sc = 8 * span_rank(span_add(sx, v[x] ^ v[y])) + w;
					if (sc > r.score) { r.score = sc; r.x = x; r.y = y; }
				}
			}
			return r;
		};
		const int half = K - 4;   // row bits (and column bits) that number the waves
		auto row_slot = [&](const SideOp& o) { return o.a >= 0 ? o.a : s.conj ? o.rec : -1; };
		auto col_slot = [&](const SideOp& o) { return o.b >= 0 ? o.b : s.conj ? o.rec : -1; };
		auto gate = [&](int x) { return x >= 0 ? (1u << bi[x]) | (1u << bj[x]) : 0u; };
		// the bits of one side with the wave bits w taken out, a gate's (x) first: lo, hi, then the block's
		auto side = [&](int x, unsigned q, const std::vector<int>& c, unsigned w, int& lo, int& hi, int* u) {
			int left[4], n = 0;
			for (unsigned m = q & ~w; m != 0; m &= m - 1) { left[n++] = __builtin_ctz(m); }
			if (x >= 0) {
				lo = bj[x];
				hi = bi[x];
			} else {
				// no gate on this side: any two bits, the colours differing in both pairs
				lo = left[0];
				for (int a = 1; a < 4; a++) {
					hi = left[a];
					const int r0 = left[a == 1 ? 2 : 1], r1 = left[a == 3 ? 2 : 3];
					if (c[lo] != c[hi] && c[r0] != c[r1]) { break; }
				}
			}
			int k = 0;
			for (int i = 0; i < 4; i++) { if (left[i] != lo && left[i] != hi) { u[k++] = left[i]; } }
		};
		// the op's layout with wave bits (rows wr, columns wc) that avoid its gates
		auto fit = [&](const SideOp& o, unsigned wr, unsigned wc, Choice& out) {
			side(row_slot(o), rm, col.r, wr, out.rl, out.rh, out.ur);
			side(col_slot(o), cm, col.c, wc, out.cl, out.ch, out.uc);
			const int b[4] = {col.r[out.ur[0]], col.c[out.uc[0]] << 2, col.r[out.ur[1]], col.c[out.uc[1]] << 2};
			const int rl = col.r[out.rl], rh = col.r[out.rh], cl = col.c[out.cl] << 2, ch = col.c[out.ch] << 2;
			const bool right = o.b >= 0 || (o.a < 0 && o.rec >= 0);
			const Blocks k = right ? blocks(b, rl, rh, cl, cl, ch) : blocks(b, cl, ch, rl, cl, ch);
			out.x = k.x;
			out.y = k.y;
			out.score = k.score;
			return k.score == 36;
		};
		// sets of wave bits, and from product j on the products that they avoid the gates of
		auto subsets = [&](const std::vector<int>& q) {
			std::vector<unsigned> r;
			for (size_t a = 0; a < q.size(); a++) {
				if (half == 1) { r.push_back(1u << q[a]); }
				else { for (size_t b = a + 1; b < q.size(); b++) { r.push_back((1u << q[a]) | (1u << q[b])); } }
			}
			return r;
		};
		const auto wrs = subsets(s.rows), wcs = subsets(s.cols);
		unsigned wr = 0, wc = 0;
		bool have = false;
		for (size_t j = 0; j < s.ops.size(); j++) {
			const SideOp& o = s.ops[j];
			Choice ch;
			const bool keep = have && !(gate(row_slot(o)) & wr) && !(gate(col_slot(o)) & wc) && fit(o, wr, wc, ch);
			if (!keep) {
				// the wave bits that serve the most products from here on
				const int left = (int)(s.ops.size() - j);
				auto reach = [&](const std::vector<unsigned>& ws, auto slot) {
					std::vector<int> n(ws.size(), 0);
					for (size_t i = 0; i < ws.size(); i++) {
						while (n[i] < left && !(gate(slot(s.ops[j + n[i]])) & ws[i])) { n[i]++; }
					}
					return n;
				};
				const std::vector<int> nr = reach(wrs, row_slot), nc = reach(wcs, col_slot);
				int best = -1000;
				for (size_t a = 0; a < wrs.size() && best < left; a++) {
					for (size_t b = s.conj ? a : 0; b < (s.conj ? a + 1 : wcs.size()) && best < left; b++) {
						const int most = std::min(nr[a], nc[b]);
						if (most == 0 || most <= best) { continue; }
						Choice t;
						int run = 1;
						if (!fit(o, wrs[a], wcs[b], t)) { run = t.score - 36; }
						else { while (run < most && fit(s.ops[j + run], wrs[a], wcs[b], t)) { run++; } }
						if (run > best) { best = run; wr = wrs[a]; wc = wcs[b]; }
					}
				}
				fit(o, wr, wc, ch);
			}
			// the group bits complete x and y (mod the span): the first two single bits that do
			{
				unsigned span = span_add(span_add(1, ch.x), ch.y);
				int n = 0;
				for (int t : {1, 3, 0, 2}) {
					if (n < 2 && !((span >> (1 << t)) & 1)) {
						span = span_add(span, 1 << t);
						ch.g[n++] = t;
					}
				}
			}
			CycOp& q = J.op[j];
			q.barrier = (j > 0 && !keep) ? 1 : 0;
			have = true;
			q.rec = o.rec;
			q.ma = o.a >= 0 ? o.ma + 6 * o.a : -1;
			q.mb = o.b >= 0 ? o.mb + 6 * o.b : -1;
			const int bits[4] = {L + ch.ur[0], ch.uc[0], L + ch.ur[1], ch.uc[1]};
			auto at = [&](int mask) {
				int v = 0;
				for (int t = 0; t < 4; t++) { if ((mask >> t) & 1) { v ^= byte[bits[t]]; } }
				return v;
			};
			const int d[8] = {byte[L + ch.rl], byte[L + ch.rh], byte[ch.cl], byte[ch.ch], at(ch.x), at(ch.y), byte[bits[ch.g[0]]],
				byte[bits[ch.g[1]]]};
			for (int i = 0; i < 8; i++) { q.dir[i] = d[i]; }
			unsigned r = wr, c = wc;
			for (int i = 0; i < half; i++, r &= r - 1, c &= c - 1) {
				q.dir[8 + 2 * i] = byte[L + __builtin_ctz(r)];
				q.dir[9 + 2 * i] = byte[__builtin_ctz(c)];
			}
			// the blocks with equal row and column bits, as combinations of the block and group
			// directions (x, y, g0, g1: four bits each)
			if (o.rec >= 0) {
				const int basis[4] = {ch.x, ch.y, 1 << ch.g[0], 1 << ch.g[1]};
				q.barrier |= (cyc_combination(basis, 3) << 8) | (cyc_combination(basis, 12) << 12);
			}
			if (sides != nullptr) { *sides += (o.a >= 0) + (o.b >= 0); }
		}
		return J;
	};
	// launches: array pairs 0, 1 forward in turn
	std::vector<int> lay(2 * (size_t)L);
	for (int b = 0; b < L; b++) { lay[L + b] = b; lay[b] = L + b; }   // M = U^dagger: row bits of M are U's columns
	int cur = -1, used = 0;
	auto use = [&](int b) { used = std::max(used, b + 1); return b; };
	for (int i = 0; i < F; i++) {
		CycLaunch ln;
		ln.njobs = 1;
		std::vector<const Step*> succ;
		if (i + 1 < F) { succ.push_back(&fwd[i + 1]); }
		else {
			if (!down.empty()) { succ.push_back(&down[0]); }
			if (!up.empty()) { succ.push_back(&up[0]); }
		}
		const std::vector<int> out = succ.empty() ? lay : next_layout(fwd[i], succ, lay);
		ln.job[0] = build_job(fwd[i], lay, out, &ln.gate_sides[0]);
		ln.in[0] = cur;
		ln.out[0] = (fwd[i].flags & kCycNoOut) ? -1 : use(cur == 0 ? 1 : 0);
		cur = ln.out[0];
		lay = out;
		plan.launches.push_back(ln);
		if (fwd[i].flags & kCycTrace) { plan.ntrace = 1L << ln.job[0].ngen; }
	}
	// both directions end in the same launch (a launch's jobs all write, or none does): the longer
	// one starts first, in turn into the pair that M_m is not in and pair 2, the shorter one into
	// pair 3 and, once it has read M_m, into M_m's
	const size_t nc = std::max(down.size(), up.size());
	struct Side { const std::vector<Step>* s; std::vector<int> lay; int cur, first, second; };
	const int other = cur == 0 ? 1 : 0;
	Side sides[2] = {{&down, lay, cur, other, 2}, {&up, lay, cur, 3, cur}};
	if (up.size() > down.size()) { std::swap(sides[0].s, sides[1].s); }
	for (size_t i = 0; i < nc; i++) {
		CycLaunch ln;
		ln.reverse = true;
		for (Side& sd : sides) {
			const size_t n = sd.s->size();
			if (i + n < nc) { continue; }
			const size_t k = i + n - nc;
			const int j = ln.njobs++;
			const Step& s = (*sd.s)[k];
			const std::vector<int> out = (k + 1 < n) ? next_layout(s, {&(*sd.s)[k + 1]}, sd.lay) : sd.lay;
			ln.job[j] = build_job(s, sd.lay, out, &ln.gate_sides[j]);
			ln.in[j] = sd.cur;
			ln.out[j] = (s.flags & kCycNoOut) ? -1 : use(k % 2 == 0 ? sd.first : sd.second);
			sd.cur = ln.out[j];
			sd.lay = out;
		}
		plan.launches.push_back(ln);
	}
	plan.nbuf = used;
	return plan;
}

}  // namespace rqc
