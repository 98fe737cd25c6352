"""Tile shapes and tile autotuning of the column sweeps, which dense targets take when the cyclic-product
sweeps' arrays do not fit (a workspace limit here), and samples and block encodings always.

Every shape is forced through the environment overrides and has to be the one that ran (last_tiles); its
FP64 results match the oracle within 1e-12, mixed precision within its stated bounds: |df| / N <= 1e-6,
gradient and HVP within 1e-4.
"""
import os
import time

import numpy as np
import pytest

import oracle as O
import rqcopt_hpc_amd as R
from helpers import brickwall_perms, crandn, haar_unitary, reldiff

pytestmark = pytest.mark.gpu

TOL = 1e-12
KEYS = ("RQC_TILE_LOGE_FP64", "RQC_TILE_LOGC_FP64", "RQC_TILE_LOGE_FP32", "RQC_TILE_LOGC_FP32", "RQC_FWD_TILE")
L, DEPTH = 10, 5


@pytest.fixture(autouse=True)
def clean():
    R.require_gpu()
    saved = {k: os.environ.pop(k, None) for k in KEYS}
    R.set_precision(R.PRECISION_FP64)
    yield
    for k, v in saved.items():
        os.environ.pop(k, None)
        if v is not None:
            os.environ[k] = v
    R.set_precision(R.PRECISION_FP64)
    R.set_eval_autotune(False)
    R.set_workspace_limit(0)


@pytest.fixture(scope="module")
def problem():
    rng = np.random.default_rng(41)
    U = np.linalg.qr(crandn(rng, (1 << L, 1 << L)))[0]
    V = np.stack([haar_unitary(rng) for _ in range(DEPTH)])
    Z, P = crandn(rng, (DEPTH, 4, 4)), brickwall_perms(L, DEPTH)
    T = R.DeviceTarget.dense(U)
    yield V, Z, P, T, O.brickwall_unitary_target_hvp(O.Ufunc.dense(U), V, Z, P, L)
    T.close()


def _limit():
    """Three quarters of the array that one evaluation sweeps: no cyclic-product sweep, several blocks."""
    R.set_workspace_limit((16 if R.get_precision() == R.PRECISION_FP64 else 8) * 3 << (2 * L - 2))


def _launches():
    return R.profile_query(R.KERNEL_FORWARD)[1]


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_tuning_follows_the_sweeps_that_run(problem, prec):
    """An evaluation on the cyclic-product sweeps has no tile to choose and leaves none behind: under a
    limit the same structure is then tuned (4 candidates, 3 runs each, before the evaluation) once."""
    V, Z, P, T, (f_o, dv_o, hz_o) = problem
    R.set_precision(R.PRECISION_FP64 if prec == "fp64" else R.PRECISION_MIXED)
    R.set_eval_autotune(True, forget=True)
    hvp = lambda: R.brickwall_unitary_target_hessian_vector_product(T, V, Z, P)   # noqa: E731
    R.profile_enable(True)
    try:
        counts = []
        for limited in (False, False, True, True):
            if limited:
                _limit()
            R.profile_reset()
            f, dv, hz = hvp()
            assert (R.last_column_block() < 1 << L) == limited
            counts.append(_launches())
    finally:
        R.profile_enable(False)
        R.profile_reset()
    print(counts, R.last_tiles(), flush=True)
    assert counts[0] == counts[1] and counts[2] >= 5 * counts[3]
    K, logC, gmax = R.last_tiles()
    base = 10 if prec == "fp64" else 11
    assert K + logC in (base, base - 1) and gmax in (8, 6)
    tol = TOL if prec == "fp64" else 1e-4
    assert abs(f - f_o) < (TOL if prec == "fp64" else 1e-6 * (1 << L)) and reldiff(dv, dv_o) < tol and reldiff(hz, hz_o) < tol


def test_batches_without_a_tile_to_choose_are_not_timed():
    """Creating a batch that runs cyclic-product sweeps alone takes about as long with autotuning as
    without it: twice at most, where timing four candidates took ten times.  Least of five, each
    another structure."""
    rng = np.random.default_rng(43)
    targets = {n: R.DeviceTarget.brickwall(np.stack([haar_unitary(rng)]), brickwall_perms(n, 1)) for n in (8, 10)}

    def create(on):
        R.set_autotune(on)
        best = 1e9
        for _ in range(5):
            pr = [(np.stack([rng.permutation(n).astype(np.int32) for _ in range(3)]), targets[n]) for n in (8, 10, 8, 10, 8, 10)]
            t0 = time.perf_counter()
            B = R.Batch(pr)
            best = min(best, time.perf_counter() - t0)
            B.close()
        return best

    try:
        create(False)
        off, on = create(False), create(True)
    finally:
        R.set_autotune(True)
    print(f"without {1e3 * off:.2f} ms, with {1e3 * on:.2f} ms", flush=True)
    assert on < 2 * off


# overrides and the reverse tile (K, logC) that has to run; the forward tile follows RQC_FWD_TILE (twice the
# columns by default, one more row bit "k", the reverse pass's own "0")
FP64_SHAPES = {
    "64x16": ({}, (6, 4)),
    "64x8_fwd_64x16": ({"RQC_TILE_LOGE_FP64": "9"}, (6, 3)),
    "64x8_fwd_128x8": ({"RQC_TILE_LOGE_FP64": "9", "RQC_FWD_TILE": "k"}, (6, 3)),
    "64x8_fwd_same": ({"RQC_TILE_LOGE_FP64": "9", "RQC_FWD_TILE": "0"}, (6, 3)),
    "128x8": ({"RQC_TILE_LOGE_FP64": "10", "RQC_TILE_LOGC_FP64": "3"}, (7, 3)),
}
FP32_SHAPES = {
    "64x32": ({}, (6, 5)),
    "64x16_fwd_64x32": ({"RQC_TILE_LOGE_FP32": "10"}, (6, 4)),
    "64x16_fwd_128x16": ({"RQC_TILE_LOGE_FP32": "10", "RQC_FWD_TILE": "k"}, (6, 4)),
    "64x16_fwd_same": ({"RQC_TILE_LOGE_FP32": "10", "RQC_FWD_TILE": "0"}, (6, 4)),
}


@pytest.mark.parametrize("name", list(FP64_SHAPES))
def test_fp64_column_tiles_match_the_oracle(problem, name):
    V, Z, P, T, (f_o, dv_o, hz_o) = problem
    env, shape = FP64_SHAPES[name]
    os.environ.update(env)
    _limit()
    print("tile", name, flush=True)
    for out in (R.brickwall_unitary_target(T, V, P), R.brickwall_unitary_target_and_gradient(T, V, P),
                R.brickwall_unitary_target_hessian_vector_product(T, V, Z, P)):
        assert R.last_sweep()[0] == R.ENGINE_TILE_PASS and R.last_tiles()[:2] == shape and R.last_column_block() < 1 << L
        out = out if isinstance(out, tuple) else (out,)
        assert abs(out[0] - f_o) < TOL * max(1, abs(f_o))
        for a, b in zip(out[1:], (dv_o, hz_o)):
            assert reldiff(a, b) < TOL


@pytest.mark.parametrize("name", list(FP32_SHAPES))
def test_mixed_column_tiles_within_bounds(problem, name):
    V, Z, P, T, (f_o, dv_o, hz_o) = problem
    env, shape = FP32_SHAPES[name]
    os.environ.update(env)
    R.set_precision(R.PRECISION_MIXED)
    _limit()
    print("tile", name, flush=True)
    f, dv, hz = R.brickwall_unitary_target_hessian_vector_product(T, V, Z, P)
    assert R.last_sweep()[0] == R.ENGINE_TILE_PASS and R.last_tiles()[:2] == shape and R.last_column_block() < 1 << L
    assert abs(f - f_o) / (1 << L) < 1e-6 and reldiff(dv, dv_o) < 1e-4 and reldiff(hz, hz_o) < 1e-4


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_issued_flops_of_a_column_sweep(problem, prec):
    """The counters' formula per amplitude and gate, in column blocks (64 x 16 or 64 x 32 tiles): forward
    96 algorithmic, 72 (FP64) or 128 (FP32) issued; reverse 192, with the recovery and both outer products
    240 or 384 issued.  The first pass leaves out tiles without an identity element: of the 25 gates in at
    least 4 passes, all but 8 count in full."""
    V, Z, P, T, _ = problem
    R.set_precision(R.PRECISION_FP64 if prec == "fp64" else R.PRECISION_MIXED)
    _limit()
    R.profile_enable(True)
    try:
        R.profile_reset()
        R.brickwall_unitary_target_hessian_vector_product(T, V, Z, P)
        fwd, rev = R.profile_query_flops(R.KERNEL_FORWARD), R.profile_query_flops(R.KERNEL_REVERSE)
    finally:
        R.profile_enable(False)
        R.profile_reset()
    assert R.last_column_block() < 1 << L
    work = float(DEPTH * (L // 2)) * (1 << (2 * L))
    issued = (72, 240) if prec == "fp64" else (128, 384)
    for (alg, done), per, i in zip((fwd, rev), (96, 192), issued):
        assert (1 - 8 / 25) * per * work < alg <= per * work * (1 + 1e-12)
        assert abs(done / alg - i / per) < 1e-12
