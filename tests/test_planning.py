"""Host planning (headers without device code, compiled here with g++): the cache of plans."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rqcopt_hpc_amd", "csrc")


def _run(tmp_path, source):
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(source)
    subprocess.check_call(["g++", "-std=c++17", "-O3", "-Wall", "-Werror", "-pthread", "-I", CSRC, str(src), "-o", str(exe)])
    return subprocess.run([str(exe)], text=True, capture_output=True, timeout=120)


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
}
"""


def test_a_thread_that_plans_does_not_keep_others_from_their_plans(tmp_path):
    r = _run(tmp_path, CACHE)
    assert r.returncode == 0, r.stderr
    assert r.stdout.split("\n")[:2] == ["1 10 1 21", "21 -2"]
