"""Column sweeps whose passes share reductions of their partial sums, against the per-gate engine.

A column block of 2^b of 2^L columns has 2^(L + b - 10) workgroups and 4 parts each, so that a
reduction takes all passes, up to 128 gates, or (512 workgroups) one pass; 130 gates need a second
one in any case, and several blocks add into the same sums.  Sums of at most 2^20 FP64 products of
magnitude 2^-L, rounded at 2^-53, stay within 1e-12.
"""
import numpy as np
import pytest

import rqcopt_hpc_amd as R
from helpers import crandn, haar_unitary, reldiff

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def restore():
    R.require_gpu()
    R.set_precision(R.PRECISION_FP64)
    yield
    R.set_sweep_engine(R.ENGINE_TILE_PASS)
    R.set_workspace_limit(0)


@pytest.mark.parametrize("L,ngates,block", [(6, 40, 16), (7, 130, 16), (7, 33, 64), (9, 40, 32), (9, 40, 128), (10, 21, 512)])
def test_column_blocks_match_gate_launches(L, ngates, block):
    print("qubits", L, "gates", ngates, "columns", block, flush=True)
    rng = np.random.default_rng(L + ngates)
    g = np.stack([haar_unitary(rng) for _ in range(ngates)])
    z = crandn(rng, (ngates, 4, 4))
    w = np.array([rng.choice(L, 2, replace=False) for _ in range(ngates)], dtype=np.int32)
    T = R.DeviceTarget.dense(crandn(rng, (1 << L, 1 << L)) / (1 << (L // 2)))
    calls = (lambda: R.circuit_unitary_target_and_gradient(T, g, w, L),
             lambda: R.circuit_unitary_target_hessian_vector_product(T, g, z, w, L))
    R.set_sweep_engine(R.ENGINE_PER_GATE)
    want = [c() for c in calls]
    R.set_sweep_engine(R.ENGINE_TILE_PASS)
    for c, b in zip(calls, want):
        # the largest limit with a column block of at most the wanted one, found by halving
        limit = 16 << (2 * L + 6)
        while True:
            R.set_workspace_limit(limit)
            a = c()
            if R.last_column_block() <= block:
                break
            limit //= 2
        assert R.last_sweep()[0] == R.ENGINE_TILE_PASS
        for x, y in zip(a, b):
            assert reldiff(x, y) < 1e-12
