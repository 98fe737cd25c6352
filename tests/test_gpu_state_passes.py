"""HVP of a statevector in passes over tiles (rqc_state_kernels.hpp) against the launches of one gate
each, and against the oracle where it is small.

2 qubits is less than a wave, 6 to 9 change the threads of a tile, 10 is one whole tile, 11 and more
have several tiles and bits outside the gates' window; 64 gates fill a pass and 65 begin the next.
Both paths round FP64 sums of at most 2^13 terms of norm-1 states over at most 130 gates: 130 gates
times 16 products at 2^-53, 2.3e-13, in norm; within 1e-12.
"""
import ctypes as ct

import numpy as np
import pytest

import oracle as O
import rqcopt_hpc_amd as R
from helpers import crandn, haar_unitary, reldiff

pytestmark = pytest.mark.gpu

TOL = 1e-12


@pytest.fixture(autouse=True)
def engine():
    R.require_gpu()
    yield
    R.set_sweep_engine(R.ENGINE_TILE_PASS)


@pytest.mark.parametrize("L,ngates", [(2, 1), (2, 5), (3, 4), (5, 64), (6, 9), (7, 65), (8, 30), (9, 130), (10, 17), (10, 65),
                                      (11, 1), (11, 40), (12, 66), (13, 25)])
def test_passes_match_gate_launches(L, ngates):
    print("qubits", L, "gates", ngates, flush=True)
    rng = np.random.default_rng(10 * L + ngates)
    g = np.stack([haar_unitary(rng) for _ in range(ngates)])
    z = crandn(rng, (ngates, 4, 4))
    w = np.array([rng.choice(L, 2, replace=False) for _ in range(ngates)], dtype=np.int32)
    psi, phi = (v / np.linalg.norm(v) for v in crandn(rng, (2, 1 << L)))
    a = R.quantum_circuit_gates_hessian_vector_product(g, z, w, psi, phi)
    R.set_sweep_engine(R.ENGINE_PER_GATE)
    b = R.quantum_circuit_gates_hessian_vector_product(g, z, w, psi, phi)
    for x, y in zip(a, b):
        if np.max(np.abs(y)) > 0:
            assert reldiff(x, y) < TOL
        else:
            assert np.max(np.abs(x)) == 0   # one gate: no second derivative
    if L <= 6:
        c = O.quantum_circuit_gates_hvp(g, z, w, psi, phi)
        for x, y in zip(a, c):
            assert reldiff(x, y) < TOL or np.max(np.abs(y)) == 0


@pytest.mark.parametrize("L,ngates,bad", [(4, 5, np.nan), (10, 25, np.inf), (12, 30, np.nan)])
def test_a_direction_that_is_not_finite_spoils_what_depends_on_it_alone(L, ngates, bad):
    """The gradients, and the HVP's entries of gates that no path connects with the direction, stay
    finite: those of the launches of one gate each."""
    print("qubits", L, "gates", ngates, bad, flush=True)
    rng = np.random.default_rng(20 * L + ngates)
    g = np.stack([haar_unitary(rng) for _ in range(ngates)])
    z = crandn(rng, (ngates, 4, 4))
    z[ngates // 2, 1, 2] = bad
    w = np.array([rng.choice(L, 2, replace=False) for _ in range(ngates)], dtype=np.int32)
    psi, phi = (v / np.linalg.norm(v) for v in crandn(rng, (2, 1 << L)))
    a = R.quantum_circuit_gates_hessian_vector_product(g, z, w, psi, phi)
    R.set_sweep_engine(R.ENGINE_PER_GATE)
    b = R.quantum_circuit_gates_hessian_vector_product(g, z, w, psi, phi)
    assert np.isfinite(a[0]).all() and np.isfinite(a[1]).all() and np.isfinite(b[2]).any()
    assert np.array_equal(np.isfinite(a[2]), np.isfinite(b[2]))
    on = np.isfinite(b[2])
    assert reldiff(a[1], b[1]) < TOL and np.max(np.abs(a[2][on] - b[2][on])) < TOL * np.max(np.abs(b[2][on]))


class _DeviceArrays:
    """Complex vectors in device memory, from the HIP runtime that the library has loaded."""

    def __init__(self):
        R.lib()
        with open("/proc/self/maps") as maps:
            self.hip = ct.CDLL(next(m.split()[-1] for m in maps if "libamdhip64" in m))
        self.ptrs = []

    def __enter__(self):
        return self

    def __exit__(self, *_):
        for p in self.ptrs:
            assert self.hip.hipFree(p) == 0

    def put(self, a):
        p = ct.c_void_p()
        assert self.hip.hipMalloc(ct.byref(p), ct.c_size_t(a.nbytes)) == 0
        self.ptrs.append(p)
        assert self.hip.hipMemcpy(p, a.ctypes.data_as(ct.c_void_p), ct.c_size_t(a.nbytes), 1) == 0
        return p

    def get(self, p, like):
        out = np.empty_like(like)
        assert self.hip.hipMemcpy(out.ctypes.data_as(ct.c_void_p), p, ct.c_size_t(out.nbytes), 2) == 0
        return out


def _device_hvp(g, z, w, L, psi, phi, out):
    n = len(g)
    dg, hg = np.empty((n, 4, 4), complex), np.empty((n, 4, 4), complex)
    svs = [R.Statevector(p.value, L) for p in (psi, phi, out)]
    vp = lambda a: a.ctypes.data_as(ct.c_void_p)   # noqa: E731
    r = R.lib().quantum_circuit_gates_hessian_vector_product(vp(g), vp(z), n, vp(w), *(ct.byref(s) for s in svs), vp(dg), vp(hg))
    assert r >= 0
    return dg, hg


@pytest.mark.parametrize("L,ngates", [(4, 6), (10, 40), (10, 80), (12, 30), (16, 45), (18, 60), (20, 70)])
def test_states_on_the_device_and_in_place(L, ngates):
    """Device arrays up to 20 qubits, psi_out apart from psi and the same array (one pass, and several
    that read psi first), against the launches of one gate each; sums of up to 2^20 terms, as above."""
    print("qubits", L, "gates", ngates, flush=True)
    rng = np.random.default_rng(30 * L + ngates)
    g = np.stack([haar_unitary(rng) for _ in range(ngates)])
    z = crandn(rng, (ngates, 4, 4))
    w = np.array([rng.choice(L, 2, replace=False) for _ in range(ngates)], dtype=np.int32)
    psi, phi = (v / np.linalg.norm(v) for v in crandn(rng, (2, 1 << L)))
    with _DeviceArrays() as dev:
        d_psi, d_phi, d_out, d_both, d_ref = (dev.put(v) for v in (psi, phi, np.zeros_like(psi), psi, np.zeros_like(psi)))
        a = _device_hvp(g, z, w, L, d_psi, d_phi, d_out)
        b = _device_hvp(g, z, w, L, d_both, d_phi, d_both)
        R.set_sweep_engine(R.ENGINE_PER_GATE)
        c = _device_hvp(g, z, w, L, d_psi, d_phi, d_ref)
        out, both, ref = (dev.get(p, psi) for p in (d_out, d_both, d_ref))
        assert np.array_equal(dev.get(d_psi, psi), psi) and np.array_equal(dev.get(d_phi, phi), phi)
    assert np.array_equal(both, out) and reldiff(out, ref) < TOL
    for x, y, r in zip(a, b, c):
        assert np.array_equal(x, y) and reldiff(x, r) < TOL
