"""Host planning (headers without device code, compiled here with g++): the cache of plans, the search of a
circuit's passes and the plans of the cyclic-product sweeps."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rqcopt_hpc_amd", "csrc")


def _build(folder, source):
    src, exe = folder / "check.cpp", folder / "check"
    src.write_text(source)
    subprocess.check_call(["g++", "-std=c++17", "-O3", "-Wall", "-Werror", "-pthread", "-I", CSRC, str(src), "-o", str(exe)])
    return str(exe)


def _run(exe, *args):
    return subprocess.run([exe] + [str(a) for a in args], text=True, capture_output=True, timeout=120)


CACHE = r"""
#include <chrono>
#include <cstdio>
#include <future>
#include <thread>
#include "rqc_plan_cache.hpp"
using namespace std::chrono_literals;
int main()
{
	rqc::PlanCache<int> cache;
	auto plan = [](int v) { return [v] { return std::make_shared<const int>(v); }; };
	cache.get({1}, plan(10));
	// a thread plans another structure, and finishes only when told to
	std::promise<void> begun, go;
	std::thread slow([&] {
		cache.get({2}, [&] {
			begun.set_value();
			go.get_future().wait_for(20s);
			return std::make_shared<const int>(20);
		});
	});
	begun.get_future().wait();
	auto hit = std::async(std::launch::async, [&] { return *cache.get({1}, plan(-1)); });
	const bool served = hit.wait_for(5s) == std::future_status::ready;
	// and one that makes the same plan first keeps it
	auto twin = std::async(std::launch::async, [&] { return *cache.get({2}, plan(21)); });
	const bool made = twin.wait_for(5s) == std::future_status::ready;
	go.set_value();
	slow.join();
	const int got = hit.get();
	printf("%d %d %d %d\n", (int)served, got, (int)made, *cache.get({2}, plan(-1)));
	twin.get();
	// the last 64 are kept, the ones used last
	for (int k = 100; k < 163; k++) { cache.get({k}, plan(k)); }
	const int two = *cache.get({2}, plan(-2)), one = *cache.get({1}, plan(-2));
	printf("%d %d\n", two, one);
	// few of large circuits (keys of 20000 integers: three), the newest whatever its size
	std::weak_ptr<const int> kept[5];
	for (int k = 0; k < 4; k++) { kept[k] = cache.get(std::vector<int>(20000, k), plan(k)); }
	kept[4] = cache.get(std::vector<int>(100000, 4), plan(4));
	printf("%d%d%d%d%d", kept[0].expired(), kept[1].expired(), kept[2].expired(), kept[3].expired(), kept[4].expired());
	for (int k = 0; k < 4; k++) { kept[k] = cache.get(std::vector<int>(20000, k), plan(k)); }
	printf(" %d%d%d%d%d", kept[0].expired(), kept[1].expired(), kept[2].expired(), kept[3].expired(), kept[4].expired());
	cache.clear();
	printf(" %d%d%d%d\n", kept[0].expired(), kept[1].expired(), kept[2].expired(), kept[3].expired());
}
"""


def test_a_thread_that_plans_does_not_keep_others_from_their_plans(tmp_path):
    r = _run(_build(tmp_path, CACHE))
    assert r.returncode == 0, r.stderr
    assert r.stdout.split("\n")[:3] == ["1 10 1 21", "21 -2", "11110 10001 1111"]


PLAN = r"""
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include "rqc_cyc_plan.hpp"
using namespace rqc;
int main(int argc, char** argv)
{
	// L layers: a periodic brickwall; L 0 gates: a random circuit
	const int L = atoi(argv[1]), layers = atoi(argv[2]), ngates = atoi(argv[3]), K = L >= 10 ? 6 : 5;
	std::vector<int> bi, bj;
	for (int i = 0; i < layers; i++) {
		for (int q = 0; q + 1 < L; q += 2) {
			bi.push_back((q + i % 2) % L);
			bj.push_back((q + 1 + i % 2) % L);
		}
	}
	srand(L + ngates);
	for (int k = 0; k < ngates; k++) {
		bi.push_back(rand() % L);
		bj.push_back((bi.back() + 1 + rand() % (L - 1)) % L);
	}
	const int G = (int)bi.size();
	double best = 1e9;
	for (int rep = 0; rep < (G > 500 ? 3 : 20); rep++) {
		const auto t0 = std::chrono::steady_clock::now();
		std::vector<CycPass> passes = plan_cyc_passes(L, bi, bj, K, kCycOps);
		// every gate once, after the gates before it on its wires, in a pass that holds its wires
		std::vector<int> last(L, -1), si, sj;
		std::vector<char> seen(G, 0);
		for (CycPass& p : passes) {
			if ((int)p.q.size() != K || p.slots.empty() || (int)p.slots.size() > kCycOps) { return 1; }
			for (int& k : p.slots) {
				unsigned q = 0;
				for (int b : p.q) { q |= 1u << b; }
				if (seen[k]++ || !((q >> bi[k]) & 1) || !((q >> bj[k]) & 1)) { return 2; }
				for (int b : {bi[k], bj[k]}) {
					if (last[b] > k) { return 3; }
					last[b] = k;
				}
				si.push_back(bi[k]);
				sj.push_back(bj[k]);
				k = (int)si.size() - 1;
			}
		}
		if ((int)si.size() != G) { return 4; }
		for (int kind = 0; kind < 3; kind++) {
			const int split = cyc_split(L, K, passes, kind == 0);
			const CycPlan p = make_cyc_plan(L, K, passes, split, si, sj, kind == 0, kind == 2, 0, 2);
			// the arrays are known before the plan is made, and the least of them before the search
			if (p.nbuf != cyc_arrays((int)passes.size(), split, kind == 0)) { return 5; }
			if (p.nbuf < cyc_least_arrays(G, kind == 0)) { return 6; }
		}
		best = std::min(best, std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count());
	}
	// the host's speed: a sort of 20000 numbers
	double yard = 1e9;
	for (int rep = 0; rep < 20; rep++) {
		std::vector<unsigned> v(20000);
		for (size_t i = 0; i < v.size(); i++) { v[i] = (unsigned)(i * 2654435761u); }
		const auto t0 = std::chrono::steady_clock::now();
		std::sort(v.begin(), v.end());
		yard = std::min(yard, std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count());
		if (v[0] > v[1]) { return 7; }
	}
	printf("%.1f %.1f\n", best, yard);
	return 0;
}
"""


YARD_US = 1000.0   # the program's yardstick where the bounds were measured; they grow with it on slower hosts


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    return _build(tmp_path_factory.mktemp("plan"), PLAN)


# Bounds: a first evaluation's planning (passes once, then the target's, the gradient's and the HVP's plan)
# has to stay below what an evaluation of the sizes takes with its planning, 0.13 ms at 6 qubits and 9
# layers to 2.3 ms at 12 and 9; the bound is that of one target evaluation, three times the 0.1 to 0.7 ms
# measured here.
@pytest.mark.parametrize("L,layers,ngates,us", [(6, 3, 0, 130), (6, 9, 0, 400), (8, 7, 0, 600), (10, 5, 0, 600), (10, 9, 0, 1900),
                                                (12, 9, 0, 2100), (14, 0, 200, 16000), (10, 0, 1000, 30000)])
def test_plans_hold_every_gate_in_order_and_are_quick(plan, L, layers, ngates, us):
    r = _run(plan, L, layers, ngates)
    assert r.returncode == 0, r.returncode
    took, yard = map(float, r.stdout.split())
    assert took < us * max(1, yard / YARD_US)
