// Search of a circuit's passes (host): sets of at most K qubits in turn, each taking ready gates.
//
// Gates on disjoint wires commute, so a pass may take any gate whose predecessors on its two wires are
// done, as long as its wires lie in the pass's set.  Candidates for a set: every window of K consecutive
// wires (cyclic) and the wires of the ready gates in circuit order; a candidate takes its ready gates in
// circuit order, at most gmax.  A beam search keeps, after each pass, the states with the most gates
// done (then the least penalty, then the earlier state and candidate); the first level that finishes
// has the fewest passes found.
//
// The search runs on the first evaluation of a structure, next to evaluations of 50 us at 6 qubits and
// 500 us at 12, so states are bit sets, passes are shared through their parents, and a candidate's gates
// are found by closing wires: 10 qubits, 9 layers 0.28 ms (12 qubits 0.46), against 1.26 ms (2.6) with
// copied states and a test of every gate's predecessors.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

namespace rqc {

struct PassSearch
{
	int L, K, gmax;
	std::vector<unsigned> gm;   // qubit bits of every gate, in circuit order
	bool descending;            // the windows start at the highest qubit bit
	bool by_set;                // states that took another set last are kept apart (the penalty depends on it)
};

struct FoundPass
{
	std::vector<int> gates;
	unsigned used;   // the qubit bits of its gates
};

// penalty(last, used): what a pass on the qubits `used` costs after one on `last` (0: the first one)
template <typename Penalty>
std::vector<FoundPass> search_passes(const PassSearch& S, const Penalty& penalty)
{
	const int L = S.L, K = S.K, G = (int)S.gm.size();
	const unsigned* gm = S.gm.data();
	const size_t W = ((size_t)G + 63) / 64, width = (G <= 256) ? 32 : (G <= 2048) ? 4 : 1;
	const unsigned all = (L >= 32) ? ~0u : (1u << L) - 1;
	// passes taken, with the pass before
	struct Taken { int prev; unsigned used; int first, n; };
	std::vector<Taken> taken;
	std::vector<int> gates;   // of all passes taken
	struct State { int taken, ndone, from, pen; uint64_t hash; };   // gates before `from` are done
	std::vector<State> beam(1, State{-1, 0, 0, 0, 0}), next;
	std::vector<uint64_t> done(W, 0), next_done;
	std::vector<unsigned> windows;
	if (K >= L) { windows.push_back(all); }
	else {
		for (int s = 0; s < L; s++) {
			unsigned m = 0;
			for (int t = 0; t < K; t++) { m |= 1u << (S.descending ? L - 1 - (s + t) % L : (s + t) % L); }
			windows.push_back(m);
		}
	}
	auto gate_hash = [](int k) {   // (splitmix64)
		uint64_t z = (uint64_t)(k + 1) * 0x9e3779b97f4a7c15ull;
		z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
		z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
		return z ^ (z >> 31);
	};
	// the next gate of a state that is not done, from k on
	auto undone = [&](const uint64_t* d, int k) {
		while (k < G) {
			const uint64_t w = ~d[k >> 6] >> (k & 63);
			if (w != 0) { return std::min(G, k + __builtin_ctzll(w)); }
			k = (k | 63) + 1;
		}
		return G;
	};
	std::vector<int> order, table;
	int best = -1, best_pen = 0;   // the plan's last pass
	std::vector<int> lst;
	while (!beam.empty() && best < 0) {
		next.clear();
		next_done.clear();
		// hash table of `next` (open addressing)
		size_t slots = 64;
		while (slots < 2 * beam.size() * (windows.size() + 1)) { slots *= 2; }
		table.assign(slots, -1);
		for (size_t b = 0; b < beam.size(); b++) {
			const State st = beam[b];
			const uint64_t* d = done.data() + b * W;
			const unsigned last = st.taken >= 0 ? taken[st.taken].used : 0;
			// the wires of the ready gates in circuit order (ready gates are disjoint: no other fits
			// once fewer than two places are left)
			unsigned ready = 0, seen = 0;
			if (K < L) {
				for (int k = undone(d, st.from); k < G && seen != all && __builtin_popcount(ready) < K - 1; k = undone(d, k + 1)) {
					if ((gm[k] & seen) == 0) { ready |= gm[k]; }
					seen |= gm[k];
				}
			}
			for (size_t c = 0; c < windows.size() + (K < L ? 1 : 0); c++) {
				// a gate is taken if its wires are open: in the set, and no earlier gate on them left out
				unsigned open = c < windows.size() ? windows[c] : ready, used = 0;
				uint64_t hash = st.hash;
				lst.clear();
				for (int k = undone(d, st.from); k < G && open != 0 && (int)lst.size() < S.gmax; k = undone(d, k + 1)) {
					if ((gm[k] & ~open) == 0) {
						lst.push_back(k);
						used |= gm[k];
						hash ^= gate_hash(k);
					} else { open &= ~gm[k]; }
				}
				if (lst.empty()) { continue; }
				State t{-1, st.ndone + (int)lst.size(), st.from, st.pen + penalty(last, used), hash};
				auto take = [&]() {
					taken.push_back(Taken{st.taken, used, (int)gates.size(), (int)lst.size()});
					gates.insert(gates.end(), lst.begin(), lst.end());
					return (int)taken.size() - 1;
				};
				if (t.ndone == G) {
					if (best < 0 || t.pen < best_pen) {
						best = take();
						best_pen = t.pen;
					}
					continue;
				}
				const size_t at = next_done.size();
				next_done.insert(next_done.end(), d, d + W);
				for (int k : lst) { next_done[at + (k >> 6)] |= 1ull << (k & 63); }
				t.from = undone(next_done.data() + at, st.from);
				// a state with the same gates done (and the same last set) that costs no more is in `next`
				bool dup = false;
				size_t s = hash & (slots - 1);
				for (; table[s] >= 0 && !dup; s = (s + 1) & (slots - 1)) {
					const State& o = next[table[s]];
					dup = o.hash == hash && o.ndone == t.ndone && o.pen <= t.pen && (!S.by_set || taken[o.taken].used == used) &&
						std::equal(next_done.begin() + at, next_done.end(), next_done.begin() + (size_t)table[s] * W);
				}
				if (dup) {
					next_done.resize(at);
					continue;
				}
				table[s] = (int)next.size();
				t.taken = take();
				next.push_back(t);
			}
		}
		if (best >= 0) { break; }
		order.resize(next.size());
		for (size_t i = 0; i < order.size(); i++) { order[i] = (int)i; }
		std::stable_sort(order.begin(), order.end(), [&](int x, int y) {
			const State &a = next[x], &b = next[y];
			return a.ndone != b.ndone ? a.ndone > b.ndone : a.pen < b.pen;
		});
		if (order.size() > width) { order.resize(width); }
		beam.clear();
		done.clear();
		for (int i : order) {
			beam.push_back(next[i]);
			done.insert(done.end(), next_done.begin() + (size_t)i * W, next_done.begin() + ((size_t)i + 1) * W);
		}
	}
	std::vector<FoundPass> out;
	for (int t = best; t >= 0; t = taken[t].prev) {
		const Taken& p = taken[t];
		out.push_back(FoundPass{std::vector<int>(gates.begin() + p.first, gates.begin() + p.first + p.n), p.used});
	}
	std::reverse(out.begin(), out.end());
	return out;
}

}  // namespace rqc
