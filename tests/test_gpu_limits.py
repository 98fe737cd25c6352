"""Batches, servers and the no-allocation call with little memory: the limits that column sweeps which reduce their sums after
every pass need are accepted, with column blocks as wide, whatever the sweeps share when there is room.

The limits (bytes) and blocks are those of such plans: 2 P + 4 arrays of 2^L x block amplitudes for P
passes, a pass's partial sums and the tables.  Results of the narrow blocks are the single evaluation's
up to the order of FP64 sums of 2^L columns: within 1e-12.
"""
import numpy as np
import pytest

import rqcopt_hpc_amd as R
from helpers import brickwall_perms, haar_unitary, reldiff

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def restore():
    R.require_gpu()
    R.set_precision(R.PRECISION_FP64)
    R.set_autotune(False)
    yield
    R.set_autotune(True)


def _problem(L, depth):
    rng = np.random.default_rng(5 * L + depth)
    T = R.DeviceTarget.brickwall(np.stack([haar_unitary(rng) for _ in range(2)]), brickwall_perms(L, 2))
    V = np.stack([haar_unitary(rng) for _ in range(depth)])
    D = np.stack([v @ (a - a.conj().T) for v, a in zip(V, rng.standard_normal((depth, 4, 4)))])
    return brickwall_perms(L, depth), T, V, D


def _check(got, want):
    assert abs(got[0] - want[0]) < 1e-12 * max(1, abs(want[0]))
    assert reldiff(got[1], want[1]) < 1e-12 and reldiff(got[2], want[2]) < 1e-12


@pytest.mark.parametrize("L,depth,n,limit,block", [
    (8, 5, 1, 1065484, 8), (8, 5, 3, 12167587, 32), (10, 5, 1, 3562413, 8), (10, 5, 3, 34186515, 32), (10, 9, 1, 8501178, 16),
    (10, 9, 1, 115527019, 256), (10, 9, 3, 12038519, 8), (12, 5, 1, 23885234, 16), (12, 5, 3, 3114902358, 1024)])
def test_batches_fit_their_limits(L, depth, n, limit, block):
    print("qubits", L, "layers", depth, "problems", n, "limit", limit, flush=True)
    P, T, V, D = _problem(L, depth)
    want = R.brickwall_unitary_target_projected_hessian_vector_product(T, V, D, P)
    B = R.Batch([(P, T)] * n, workspace_limit=limit)
    try:
        assert B.stats()["workspace_bytes"] <= limit
        assert min(B.plan(p, R.EVAL_HVP)[0] for p in range(n)) >= block
        f, g, h = B.evaluate([R.EVAL_HVP] * n, [V] * n, [D] * n)
        for p in range(n):
            _check((f[p], g[p], h[p]), want)
    finally:
        B.close()


@pytest.mark.parametrize("L,depth,arena,block", [(8, 5, 2395136, 32), (8, 5, 4047872, 64), (10, 5, 4697856, 16),
                                                 (10, 5, 38323200, 128), (10, 9, 17443328, 32), (12, 5, 44478464, 32)])
def test_requests_fit_their_arena(L, depth, arena, block):
    print("qubits", L, "layers", depth, "arena", arena, flush=True)
    P, T, V, D = _problem(L, depth)
    want = R.brickwall_unitary_target_projected_hessian_vector_product(T, V, D, P)
    srv = R.Server(arena_bytes=arena, max_request_bytes=arena, nslots=2)
    try:
        f, g, h, info = srv.wait(srv.submit(srv.session_brickwall(P, T), R.EVAL_HVP, V, D))
        assert info["block"] >= block and info["workspace_bytes"] <= arena
        _check((f, g, h), want)
    finally:
        srv.close()


@pytest.mark.parametrize("L,depth", [(10, 6), (12, 4), (12, 5), (12, 20)])
def test_the_scratch_takes_the_widest_block_that_fits(L, depth):
    """A column block narrower than the first that is tried: the evaluation runs in half of it, and so on
    (it is refused only where one column does not fit).  Half of the scratch holds the states at least."""
    print("qubits", L, "layers", depth, flush=True)
    P, T, V, D = _problem(L, depth)
    want = R.brickwall_unitary_target_projected_hessian_vector_product(T, V, D, P)
    got = R.brickwall_unitary_target_projected_hvp_noalloc(T, V, D, P)
    B, passes = R.last_column_block(), R.last_sweep()[1]
    assert B == 1 << L or (2 * passes + 4) * B * 16 << L > R.noalloc_scratch_bytes() // 4
    _check(got, want)
