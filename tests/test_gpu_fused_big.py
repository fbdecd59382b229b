"""The store pass with whole columns in a workgroup's LDS (11 to 13 qubits, 14 in
complex64): square corners of its ranges (one column, partial column groups, strided rows
and batches, shared and per-matrix parameters) against the streaming path, one pass per
gate, and the streamed costs against the oracle."""
import numpy as np
import pytest
import torch

from squander_hip import _native as nat
from squander_hip import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,f32", [(11, False), (11, True), (12, False), (12, True), (13, False), (13, True),
                                   (14, True)])
@pytest.mark.parametrize("cols,pad,B", [(1, 0, 1), (3, 2, 2), (17, 0, 4)])
def test_big_store_pass(n, f32, cols, pad, B):
    print(n, f32, cols, pad, B, flush=True)
    gates = np.concatenate([W.mixed_gate_circuit(n, 40, n), [[nat.GATE_CNOT, 0, n - 1, 0]]]).astype(np.int32)
    P, d = W.param_count(gates), 1 << n
    gen = torch.Generator(device="cuda").manual_seed(n)
    dt = torch.complex64 if f32 else torch.complex128
    M = torch.randn((B, d + 1, cols + pad), dtype=torch.complex128, device="cuda", generator=gen).to(dt)
    ps = torch.from_numpy(W.random_params(P, 3, batch=B)).cuda()
    ctx = nat.Context(0)
    ctx.set_circuit(n, gates)
    st, bs = cols + pad, (d + 1) * (cols + pad)
    for pb in (0, P):
        X, Y = M.clone(), M.clone()
        torch.cuda.synchronize()
        ctx.check(ctx._L.sqh_apply_to_dev(ctx.h, ps.data_ptr(), pb, X.data_ptr(), d, cols, st, bs, B, int(f32)))
        ctx.check(ctx._L.sqh_apply_to_stream_dev(ctx.h, ps.data_ptr(), pb, Y.data_ptr(), d, cols, st, bs, B, int(f32)))
        ctx.synchronize()
        # FP64: rounding of some hundred operations; FP32: the streaming pass's own error
        tol = 5e-6 if f32 else 1e-13
        assert torch.linalg.norm(X - Y) <= tol * torch.linalg.norm(Y)
        assert torch.equal(X[:, d], M[:, d]) and torch.equal(X[:, :, cols:], M[:, :, cols:])
        # the pass per block does the same products in the same order: which of the two runs
        # (by batch and columns) does not show in the bits
        Z = M.clone()
        torch.cuda.synchronize()
        ctx.check(ctx._L.sqh_apply_to_fused_dev(ctx.h, ps.data_ptr(), pb, Z.data_ptr(), d, cols, st, bs, B, int(f32)))
        ctx.synchronize()
        assert torch.equal(X, Z)


def test_big_costs(oracle):
    gates = W.mixed_gate_circuit(11, 50, 5)
    P = W.param_count(gates)
    rng = np.random.default_rng(1)
    U = np.linalg.qr(rng.standard_normal((2048, 5)) + 1j * rng.standard_normal((2048, 5)))[0]
    ps = W.random_params(P, 7, batch=3)
    ctx = nat.Context(0)
    ctx.set_circuit(11, gates)
    ctx.set_target(U)
    ctx.set_trace_offset(9)
    for prec, tol in ((nat.PREC_F64, 1e-12), (nat.PREC_F32, 1e-5)):
        c = np.empty(3)
        ctx.check(ctx._L.sqh_optimization_problem_batch(ctx.h, ps.ctypes.data, 3, prec, c.ctypes.data))
        for b in range(3):
            M = oracle.apply_to(gates, ps[b], U)
            want = 1.0 - sum(M[j + 9, j].real for j in range(5)) / 5
            assert abs(c[b] - want) < tol
