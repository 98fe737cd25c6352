"""Cyclic-product sweeps (rqc_cyc_kernels.hpp): target, gradient and HVP of dense targets against
the oracle and the per-gate engine, at the sizes where plans and tiles change.

5 qubits is the smallest tile, 9 / 10 the change of the tile size, and the gate counts cover one
gate (no conjugation), passes of one gate, full passes of 8 and the next pass's first gate; random
wires give passes with one-sided launches, any wire order and gates that repeat a pair.  FP64 sums
of up to 2^22 products of magnitude 1 / N rounded at 2^-53 stay within 1e-12 of either engine.
"""
import numpy as np
import pytest

import oracle as O
import rqcopt_hpc_amd as R
from helpers import brickwall_perms, crandn, haar_unitary, reldiff

pytestmark = pytest.mark.gpu

TOL = 1e-12


@pytest.fixture(autouse=True)
def fp64():
    R.require_gpu()
    R.set_precision(R.PRECISION_FP64)
    yield
    R.set_precision(R.PRECISION_FP64)
    R.set_sweep_engine(R.ENGINE_TILE_PASS)
    R.set_workspace_limit(0)


def _all(T, g, z, w, L):
    return (R.circuit_unitary_target(T, g, w, L), R.circuit_unitary_target_and_gradient(T, g, w, L),
            R.circuit_unitary_target_hessian_vector_product(T, g, z, w, L))


def _check(a, f, dg, hg):
    assert reldiff(a[0], f) < TOL
    assert reldiff(a[1][0], f) < TOL and reldiff(a[1][1], dg) < TOL
    assert reldiff(a[2][0], f) < TOL and reldiff(a[2][1], dg) < TOL
    if np.max(np.abs(hg)) > 0:
        assert reldiff(a[2][2], hg) < TOL
    else:
        assert np.max(np.abs(a[2][2])) < TOL * np.max(np.abs(dg))


@pytest.mark.parametrize("L,ngates", [(5, 1), (5, 8), (5, 17), (6, 2), (6, 9), (7, 1), (7, 33), (8, 16), (9, 25), (10, 9),
                                      (10, 40), (11, 23)])
def test_random_circuits_match_oracle(L, ngates):
    print("qubits", L, "gates", ngates, flush=True)
    rng = np.random.default_rng(100 * L + ngates)
    g = np.stack([haar_unitary(rng) for _ in range(ngates)])
    z = crandn(rng, (ngates, 4, 4))
    w = np.array([rng.choice(L, 2, replace=False) for _ in range(ngates)], dtype=np.int32)
    U = crandn(rng, (1 << L, 1 << L)) / (1 << (L // 2))
    T = R.DeviceTarget.dense(U)
    a = _all(T, g, z, w, L)
    assert R.last_sweep()[0] == R.ENGINE_TILE_PASS and R.last_column_block() == 1 << L
    if L <= 8:
        _check(a, *O.circuit_unitary_target_hvp(O.Ufunc.dense(U), g, z, w, L))
    R.set_sweep_engine(R.ENGINE_PER_GATE)
    b = _all(T, g, z, w, L)
    _check(a, b[0], b[1][1], b[2][2])


@pytest.mark.parametrize("L,depth", [(6, 1), (10, 4), (12, 2), (12, 5)])
def test_brickwalls_match_the_column_sweeps(L, depth):
    """The same evaluation with and without room for the N x N arrays (column blocks of the tile
    passes), and repeated: bitwise equal."""
    print("qubits", L, "layers", depth, flush=True)
    rng = np.random.default_rng(7 * L + depth)
    V = np.stack([haar_unitary(rng) for _ in range(depth)])
    Z = crandn(rng, (depth, 4, 4))
    P = brickwall_perms(L, depth)
    T = R.DeviceTarget.brickwall(np.stack([haar_unitary(rng) for _ in range(3)]), brickwall_perms(L, 3))
    a = R.brickwall_unitary_target_hessian_vector_product(T, V, Z, P)
    b = R.brickwall_unitary_target_hessian_vector_product(T, V, Z, P)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)
    ft = R.brickwall_unitary_target(T, V, P)
    R.set_workspace_limit(max(1 << 20, (1 << (2 * L)) * 16 // 4))
    c = R.brickwall_unitary_target_hessian_vector_product(T, V, Z, P)
    assert R.last_column_block() < 1 << L or L == 6
    assert reldiff(ft, a[0]) < TOL
    for x, y in zip(a, c):
        assert reldiff(x, y) < TOL


@pytest.mark.parametrize("L,depth", [(6, 1), (6, 4), (8, 2), (10, 2)])
def test_hessian_columns_together_match_single_products(L, depth):
    """The Hessian's columns run as several evaluations per launch (all at once at 6 and 8 qubits, in
    chunks of 16 at 10): each equals the HVP along its unit direction, which runs alone."""
    print("qubits", L, "layers", depth, flush=True)
    rng = np.random.default_rng(13 * L + depth)
    V = np.stack([haar_unitary(rng) for _ in range(depth)])
    P = brickwall_perms(L, depth)
    T = R.DeviceTarget.brickwall(np.stack([haar_unitary(rng) for _ in range(3)]), brickwall_perms(L, 3))
    f, dv, H = R.brickwall_unitary_target_gradient_hessian(T, V, P)
    H = np.asarray(H).reshape(16 * depth, 16 * depth)
    for col in sorted({0, 7, 16 * depth - 1, 8 * depth + 3}):
        Z = np.zeros((depth, 4, 4), complex)
        Z[col // 16, (col % 16) // 4, col % 4] = 1
        f1, dv1, hz = R.brickwall_unitary_target_hessian_vector_product(T, V, Z, P)
        assert reldiff(f, f1) < TOL and reldiff(dv, dv1) < TOL
        assert np.max(np.abs(H[:, col] - hz.reshape(-1))) < TOL * np.max(np.abs(H))


@pytest.mark.parametrize("L,ngates", [(5, 3), (6, 17), (9, 12), (10, 31), (11, 20)])
def test_mixed_precision_rounds_between_launches_only(L, ngates):
    """Mixed precision keeps the arrays between launches in complex FP32 and multiplies in FP64: an
    entry is rounded (2^-24 relative) once per launch, at most about 20 times, so gradients and HVPs
    stay within 2e-6 of FP64 (20 roundings of one sign: 1.2e-6), f within that of sqrt(N)."""
    print("qubits", L, "gates", ngates, flush=True)
    rng = np.random.default_rng(31 * L + ngates)
    g = np.stack([haar_unitary(rng) for _ in range(ngates)])
    z = crandn(rng, (ngates, 4, 4))
    w = np.array([rng.choice(L, 2, replace=False) for _ in range(ngates)], dtype=np.int32)
    U = np.linalg.qr(crandn(rng, (1 << L, 1 << L)))[0]
    T = R.DeviceTarget.dense(U)
    a = _all(T, g, z, w, L)
    R.set_precision(R.PRECISION_MIXED)
    m = _all(T, g, z, w, L)
    assert R.last_sweep()[0] == R.ENGINE_TILE_PASS
    for f in (m[0], m[1][0], m[2][0]):
        assert abs(f - a[0]) < 2e-6 * 2 ** (L / 2)
    assert reldiff(m[1][1], a[1][1]) < 2e-6 and reldiff(m[2][1], a[2][1]) < 2e-6 and reldiff(m[2][2], a[2][2]) < 2e-6


def test_f_of_every_kind_is_as_accurate():
    """f of a gradient or HVP comes from the product before any conjugation, after as many gate products
    as a target evaluation's: their rounding errors (against 80-bit arithmetic) have one distribution.
    The root mean squares of 60 complex errors differ by 9 % (120 values each, 1 / sqrt(240) twice);
    1.35 is four times that above one."""
    L, depth, n = 6, 9, 60
    print("qubits", L, "layers", depth, flush=True)
    N, P = 1 << L, brickwall_perms(L, depth)
    wires = [(int(p[2 * k]), int(p[2 * k + 1])) for p in P for k in range(L // 2)]
    err = []
    for seed in range(n):
        rng = np.random.default_rng([L, depth, seed])
        V = np.stack([haar_unitary(rng) for _ in range(depth)])
        U = np.linalg.qr(crandn(rng, (N, N)))[0]
        W = np.eye(N, dtype=np.clongdouble)
        for g, (a, b) in zip(np.repeat(V, L // 2, 0), wires):
            t = np.moveaxis(W.reshape([2] * L + [N]), (a, b), (0, 1))
            y = np.tensordot(g.astype(np.clongdouble).reshape(2, 2, 2, 2), t, ((2, 3), (0, 1)))
            W = np.moveaxis(y, (0, 1), (a, b)).reshape(N, N)
        f = -(U.astype(np.clongdouble).conj() * W).sum()
        T = R.DeviceTarget.dense(U)
        err.append([abs(np.clongdouble(v) - f) for v in (
            R.brickwall_unitary_target(T, V, P), R.brickwall_unitary_target_and_gradient(T, V, P)[0],
            R.brickwall_unitary_target_hessian_vector_product(T, V, crandn(rng, V.shape), P)[0])])
        T.close()
    target, gradient, hvp = np.sqrt(np.mean(np.array(err, float) ** 2, axis=0))
    print(target, gradient, hvp, flush=True)
    assert gradient < 1.35 * target and hvp < 1.35 * target


@pytest.mark.parametrize("prec", [R.PRECISION_FP64, R.PRECISION_MIXED])
@pytest.mark.parametrize("L,ngates", [(5, 9), (9, 30), (10, 30), (11, 50)])
def test_f_of_gates_that_are_not_unitary(L, ngates, prec):
    """A target evaluation takes any gates onto the cyclic-product sweeps in FP64 (gradients and mixed
    precision go gate by gate), at the change of the tile size too; within 1e-12 (mixed: 2e-6 of the
    norm) of the per-gate engine."""
    print("qubits", L, "gates", ngates, "precision", prec, flush=True)
    rng = np.random.default_rng(11 * L + ngates)
    g = crandn(rng, (ngates, 4, 4)) / 2
    w = np.array([rng.choice(L, 2, replace=False) for _ in range(ngates)], dtype=np.int32)
    T = R.DeviceTarget.dense(crandn(rng, (1 << L, 1 << L)))
    R.set_precision(prec)
    f = R.circuit_unitary_target(T, g, w, L)
    assert R.last_sweep()[0] == (R.ENGINE_TILE_PASS if prec == R.PRECISION_FP64 else R.ENGINE_PER_GATE)
    R.set_precision(R.PRECISION_FP64)
    f64, dg = R.circuit_unitary_target_and_gradient(T, g, w, L)
    assert R.last_sweep()[0] == R.ENGINE_PER_GATE
    R.set_sweep_engine(R.ENGINE_PER_GATE)
    f_o, dg_o = R.circuit_unitary_target_and_gradient(T, g, w, L)
    assert f64 == f_o and np.array_equal(dg, dg_o)
    # (f is a sum of 4^L products that cancel: its terms' norm is that of the gradient with its gate)
    norm = np.linalg.norm(dg_o[0]) * np.linalg.norm(g[0])
    assert abs(f - f_o) < (TOL if prec == R.PRECISION_FP64 else 2e-6) * max(norm, abs(f_o))


def test_six_qubits_one_layer_in_column_blocks():
    """A limit below the arrays at 6 qubits: the column blocks of one pass against the whole array."""
    L, depth = 6, 1
    rng = np.random.default_rng(61)
    V, Z = np.stack([haar_unitary(rng) for _ in range(depth)]), crandn(rng, (depth, 4, 4))
    P = brickwall_perms(L, depth)
    T = R.DeviceTarget.brickwall(np.stack([haar_unitary(rng) for _ in range(3)]), brickwall_perms(L, 3))
    a = R.brickwall_unitary_target_hessian_vector_product(T, V, Z, P)
    assert R.last_column_block() == 1 << L
    R.set_workspace_limit(6 * (16 << (2 * L)) // 4)   # a pass's 6 arrays of 16 columns; the cyclic sweeps need 2 of 64
    c = R.brickwall_unitary_target_hessian_vector_product(T, V, Z, P)
    assert R.last_column_block() < 1 << L and R.last_sweep()[0] == R.ENGINE_TILE_PASS
    for x, y in zip(a, c):
        assert reldiff(x, y) < TOL or np.max(np.abs(y)) == 0
