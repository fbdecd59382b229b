"""The fused blocks' gate walks (block matrices and gate correlations) where they can go
wrong: blocks of one gate, around and beyond the 64 gates staged at a time, every gate
kind, circuits without parameters; costs, gradients, apply_to and derivatives against the
oracle (1e-12 in complex128, 1e-5 in complex64, as for the other fused kernels)."""
import numpy as np
import pytest

from squander_hip import Circuit
from squander_hip import _native as nat
from squander_hip import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,count", [(4, 1), (4, 63), (4, 64), (4, 65), (4, 200), (5, 150), (7, 60)])
def test_long_and_short_blocks(oracle, n, count):
    print(n, count, flush=True)
    gates = W.mixed_gate_circuit(n, count, 100 * n + count)
    if not W.param_count(gates):
        gates = np.asarray([[nat.GATE_U3, 1, -1, 0]], dtype=np.int32)
    P = W.param_count(gates)
    U = W.haar_unitary(1 << n, 5).conj().T.copy()
    ps = W.random_params(P, 6, batch=5)
    ctx = nat.Context(0)
    ctx.set_circuit(n, gates)
    ctx.set_target(U)
    ctx.set_fused_cost(True)
    for prec, tol in ((nat.PREC_F64, 1e-12), (nat.PREC_F32, 1e-5)):
        f, c, g = np.empty(5), np.empty(5), np.empty((5, P))
        ctx.check(ctx._L.sqh_optimization_problem_batch(ctx.h, ps.ctypes.data, 5, prec, c.ctypes.data))
        ctx.check(ctx._L.sqh_optimization_problem_combined_batch(ctx.h, ps.ctypes.data, 5, prec, f.ctypes.data,
                                                                 g.ctypes.data))
        for b in range(5):
            fr, gr = oracle.optimization_problem_combined(gates, U, n, ps[b])
            assert abs(c[b] - fr) < tol and abs(f[b] - fr) < tol
            assert np.abs(g[b] - gr).max() < tol
    D = np.empty((P,) + U.shape, dtype=np.complex128)
    ctx.check(ctx._L.sqh_apply_derivate_to(ctx.h, ps[0].ctypes.data, U.ctypes.data, 1 << n, 1 << n, 1 << n,
                                           D.ctypes.data))
    ref = np.asarray(oracle.apply_derivate_to(gates, ps[0], U))
    assert np.linalg.norm(D - ref) <= 1e-12 * np.linalg.norm(ref)


def test_circuit_without_parameters(oracle):
    gates = np.asarray([[nat.GATE_CNOT, 0, 3, 0], [nat.GATE_CZ, 2, 1, 0], [nat.GATE_CNOT, 4, 2, 0]], dtype=np.int32)
    U = W.haar_unitary(32, 8)
    ctx = nat.Context(0)
    ctx.set_circuit(5, gates)
    ctx.set_target(U)
    ctx.set_fused_cost(True)
    c = np.empty(3)
    ctx.check(ctx._L.sqh_optimization_problem_batch(ctx.h, None, 3, nat.PREC_F64, c.ctypes.data))
    want = oracle.optimization_problem(gates, U, 5, np.zeros(0))
    assert np.abs(c - want).max() < 1e-12
    M = U.copy()
    circ = Circuit.from_gate_array(5, gates)
    circ._context().set_fused_cost(True)
    circ.apply_to(np.zeros(0), M)
    ref = oracle.apply_to(gates, np.zeros(0), U)
    assert np.linalg.norm(M - ref) <= 1e-12 * np.linalg.norm(ref)
