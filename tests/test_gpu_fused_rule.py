"""The automatic choice between the fused blocks and the register-tile kernels: on both
sides of every line of the rule (qubits 4 to 10, deep and shallow circuits) costs,
gradients and apply_to agree with the forced paths to rounding, strided rows included,
and do not depend on the batch a vector comes in by more."""
import numpy as np
import pytest
import torch

from squander_hip import _native as nat
from squander_hip import workloads as W

pytestmark = pytest.mark.gpu


def _evaluate(ctx, ps, M, stride, mode):
    ctx.set_fused_cost(mode)
    B, P = ps.shape
    c, f, g = np.empty(B), np.empty(B), np.empty((B, P))
    ctx.check(ctx._L.sqh_optimization_problem_batch(ctx.h, ps.ctypes.data, B, nat.PREC_F64, c.ctypes.data))
    ctx.check(ctx._L.sqh_optimization_problem_combined_batch(ctx.h, ps.ctypes.data, B, nat.PREC_F64, f.ctypes.data,
                                                             g.ctypes.data))
    dp, dM = torch.from_numpy(ps).cuda(), torch.from_numpy(M).cuda()
    torch.cuda.synchronize()
    d, cols = M.shape[1], M.shape[2] - stride
    ctx.check(ctx._L.sqh_apply_to_dev(ctx.h, dp.data_ptr(), P, dM.data_ptr(), d, cols, M.shape[2], d * M.shape[2], B, 0))
    ctx.synchronize()
    return c, f, g, dM.cpu().numpy()


@pytest.mark.parametrize("n", [4, 5, 6, 8, 10])
@pytest.mark.parametrize("layers", [0, 1, 3, 14])
def test_automatic_equals_both_paths(n, layers):
    print(n, layers, flush=True)
    gates = W.ansatz_layers(n, W.alternating_pairs(n, layers))
    d, P, B, cols, pad = 1 << n, W.param_count(gates), 3, (1 << n) - 3, 2
    rng = np.random.default_rng(n)
    U = W.haar_unitary(d, 3)[:, :cols].copy()
    ps = W.random_params(P, 4, batch=B)
    M = rng.standard_normal((B, d, cols + pad)) + 1j * rng.standard_normal((B, d, cols + pad))
    ctx = nat.Context(0)
    ctx.set_circuit(n, gates)
    ctx.set_target(U)
    ctx.set_trace_offset(2)
    c, f, g, R = _evaluate(ctx, ps, M, pad, "auto")
    for mode in (True, False):
        c2, f2, g2, R2 = _evaluate(ctx, ps, M, pad, mode)
        assert np.abs(c - c2).max() < 1e-12 and np.abs(f - f2).max() < 1e-12
        assert np.abs(g - g2).max() < 1e-12
        assert np.linalg.norm(R - R2) <= 1e-12 * np.linalg.norm(R)
        assert np.array_equal(R2[:, :, cols:], M[:, :, cols:])
    one = _evaluate(ctx, ps[1:2].copy(), M[1:2].copy(), pad, "auto")
    assert abs(one[0][0] - c[1]) < 1e-12 and np.abs(one[2][0] - g[1]).max() < 1e-12


def test_derivatives_and_apply_to_are_tuned_apart():
    """The derivatives' pass runs some of the blocks per matrix, apply_to all: a batch of as
    many matrices of the same shape measures its own launch shape."""
    import ctypes
    n, cols = 7, 40
    gates = W.mixed_gate_circuit(n, 40, 7)
    P, d = W.param_count(gates), 1 << n
    ctx = nat.Context(0)
    ctx.set_circuit(n, gates)
    ctx.set_fused_cost(True)

    def tuned_ms():
        t, w, ms = ctypes.c_int(), ctypes.c_int(), ctypes.c_double()
        ctx.check(ctx._L.sqh_get_block_config(ctx.h, 0, 256, 16, 1, ctypes.byref(t), ctypes.byref(w),
                                              ctypes.byref(ms)))
        return ms.value

    tuned_ms()  # the shape asked for here is itself measured once
    p = torch.from_numpy(W.random_params(P, 3)).cuda()
    M = torch.randn((P, d, cols), dtype=torch.complex128, device="cuda")
    D = torch.empty_like(M)
    torch.cuda.synchronize()
    times = [tuned_ms()]
    for _ in range(2):
        ctx.check(ctx._L.sqh_apply_derivate_to_dev(ctx.h, p.data_ptr(), M.data_ptr(), d, cols, cols, D.data_ptr()))
        times.append(tuned_ms())
    for _ in range(2):
        ctx.check(ctx._L.sqh_apply_to_dev(ctx.h, p.data_ptr(), 0, M.data_ptr(), d, cols, cols, d * cols, P, 0))
        times.append(tuned_ms())
    ctx.synchronize()
    assert times[0] < times[1] == times[2] < times[3] == times[4]


@pytest.mark.parametrize("n", [4, 5, 6, 7, 8, 9, 10])
@pytest.mark.parametrize("f32", [False, True])
def test_store_pass_shapes_agree(oracle, n, f32):
    """The store pass at every launch shape (the columns' padding in LDS differs): the same
    bits, odd column counts, and the oracle's matrices."""
    gates = W.mixed_gate_circuit(n, 4 * n, 90 + n)
    P, d, B, cols = W.param_count(gates), 1 << n, 3, min(37, (1 << n) - 1)
    rng = np.random.default_rng(n)
    M = rng.standard_normal((B, d, cols)) + 1j * rng.standard_normal((B, d, cols))
    M = M.astype(np.complex64 if f32 else np.complex128)
    ps = W.random_params(P, 5, batch=B)
    ctx = nat.Context(0)
    ctx.set_circuit(n, gates)
    ctx.set_fused_cost(True)
    dp, first = torch.from_numpy(ps).cuda(), None
    for shape in ((4, 1, 1, 0), (4, 1, 2, 1), (4, 1, 4, 0), (4, 2, 2, 1), (2, 1, 1, 0), (2, 1, 4, 1)):
        if n == 10 and shape[0] == 2 or shape[1] == 2 and n > 8 or n == 9 and shape[1] == 2:
            continue
        ctx.set_fused_cost_config(*shape)
        X = torch.from_numpy(M).cuda()
        torch.cuda.synchronize()
        ctx.check(ctx._L.sqh_apply_to_dev(ctx.h, dp.data_ptr(), P, X.data_ptr(), d, cols, cols, d * cols, B, int(f32)))
        ctx.synchronize()
        X = X.cpu().numpy()
        if first is None:
            first = X
            for b in range(B):
                want = oracle.apply_to(gates, ps[b], M[b].astype(np.complex128))
                assert np.linalg.norm(X[b] - want) <= (1e-5 if f32 else 1e-12) * np.linalg.norm(want)
        assert np.array_equal(X, first), shape


@pytest.mark.parametrize("B", [4096, 4097])
def test_four_qubits_across_the_batch_line(oracle, B):
    """Around the batch beyond which 4-qubit complex64 batches and matrices run the tile
    kernels: complex128 costs and gradients keep their bits, the rest agrees to rounding with a
    small batch and the oracle."""
    gates = W.ansatz_layers(4, W.alternating_pairs(4, 20))
    P = W.param_count(gates)
    U = W.haar_unitary(16, 3)
    ps = W.random_params(P, 4, batch=B)
    ctx = nat.Context(0)
    ctx.set_circuit(4, gates)
    ctx.set_target(U)

    def both(p, prec):
        b = p.shape[0]
        c, f, g = np.empty(b), np.empty(b), np.empty((b, P))
        p = np.ascontiguousarray(p)
        ctx.check(ctx._L.sqh_optimization_problem_batch(ctx.h, p.ctypes.data, b, prec, c.ctypes.data))
        ctx.check(ctx._L.sqh_optimization_problem_combined_batch(ctx.h, p.ctypes.data, b, prec, f.ctypes.data,
                                                                 g.ctypes.data))
        return c, f, g

    few = [0, B // 2, B - 1]
    for prec, tol in ((nat.PREC_F64, 0.0), (nat.PREC_F32, 2e-5)):
        for x, y in zip(both(ps, prec), both(ps[few], prec)):
            assert np.abs(x[few] - y).max() <= tol
    f, g = oracle.optimization_problem_combined(gates, U, 4, ps[B - 1])
    c = both(ps[few], nat.PREC_F64)
    assert abs(c[0][2] - f) < 1e-12 and np.abs(c[2][2] - g).max() < 1e-12
    for dt, tol in ((torch.complex128, 1e-12), (torch.complex64, 1e-5)):
        M = torch.from_numpy(np.broadcast_to(U, (B, 16, 16)).copy()).cuda().to(dt)
        dp = torch.from_numpy(ps).cuda()
        torch.cuda.synchronize()
        ctx.check(ctx._L.sqh_apply_to_dev(ctx.h, dp.data_ptr(), P, M.data_ptr(), 16, 16, 16, 256, B,
                                          int(dt == torch.complex64)))
        ctx.synchronize()
        for b in few:
            want = oracle.apply_to(gates, ps[b], U)
            assert np.linalg.norm(M[b].cpu().numpy() - want) <= tol * np.linalg.norm(want)


@pytest.mark.parametrize("B", [2048, 2049])
@pytest.mark.parametrize("n,m", [(5, 8), (7, 4)])
def test_few_columns_across_the_batch_line(oracle, n, m, B):
    """Around the batch beyond which matrices of few entries run the tile kernels: complex128
    costs keep their bits, the rest agrees to rounding with a small batch and the oracle; so do
    matrices that share one parameter vector."""
    gates = W.ansatz_layers(n, W.alternating_pairs(n, 3 * n))
    d, P = 1 << n, W.param_count(gates)
    U = np.ascontiguousarray(W.haar_unitary(d, 3)[:, :m])
    ps = W.random_params(P, 4, batch=B)
    ctx = nat.Context(0)
    ctx.set_circuit(n, gates)
    ctx.set_target(U)

    def both(p, prec):
        b = p.shape[0]
        c, f, g = np.empty(b), np.empty(b), np.empty((b, P))
        p = np.ascontiguousarray(p)
        ctx.check(ctx._L.sqh_optimization_problem_batch(ctx.h, p.ctypes.data, b, prec, c.ctypes.data))
        ctx.check(ctx._L.sqh_optimization_problem_combined_batch(ctx.h, p.ctypes.data, b, prec, f.ctypes.data,
                                                                 g.ctypes.data))
        return c, f, g

    few = [0, B // 2, B - 1]
    for prec, tol in ((nat.PREC_F64, 1e-12), (nat.PREC_F32, 2e-5)):
        many, small = both(ps, prec), both(ps[few], prec)
        for x, y in zip(many, small):
            assert np.abs(x[few] - y).max() <= tol
        if prec == nat.PREC_F64:
            assert np.array_equal(many[0][few], small[0])
            for i, b in enumerate(few):
                f, g = oracle.optimization_problem_combined(gates, U, n, ps[b])
                assert abs(many[0][b] - f) < 1e-12 and np.abs(many[2][b] - g).max() < 1e-12
    for dt, tol in ((torch.complex128, 1e-12), (torch.complex64, 1e-5)):
        for shared in (False, True):
            M = torch.from_numpy(np.broadcast_to(U, (B, d, m)).copy()).cuda().to(dt)
            dp = torch.from_numpy(ps).cuda()
            torch.cuda.synchronize()
            ctx.check(ctx._L.sqh_apply_to_dev(ctx.h, dp.data_ptr(), 0 if shared else P, M.data_ptr(), d, m, m, d * m, B,
                                              int(dt == torch.complex64)))
            ctx.synchronize()
            for b in few:
                want = oracle.apply_to(gates, ps[0 if shared else b], U)
                assert np.linalg.norm(M[b].cpu().numpy() - want) <= tol * np.linalg.norm(want)
