"""How the fused gradient's correlation sums are split over wavefronts: a vector's cost and
gradient are the same bits in every batch, at every launch shape, next to any companions in
the optimiser's rounds, and agree with the oracle where the split changes form (one column
group per task or many, whole rounds and a rest, partials summed by a workgroup per block
or by a wavefront, batches beyond one launch's scratch)."""
import numpy as np
import pytest

from squander_hip import _native as nat
from squander_hip import decompose_batch, default_options
from squander_hip import workloads as W

pytestmark = pytest.mark.gpu


def combined(ctx, ps, prec):
    B, P = ps.shape
    f, g = np.empty(B), np.empty((B, P))
    ps = np.ascontiguousarray(ps)
    ctx.check(ctx._L.sqh_optimization_problem_combined_batch(ctx.h, ps.ctypes.data, B, prec, f.ctypes.data,
                                                             g.ctypes.data))
    return f, g


# the last batch of each runs at every launch shape
@pytest.mark.parametrize("n,cols,batches", [(8, 256, (1, 63, 64, 96, 171, 512, 523)), (8, 251, (2, 65, 203)),
                                            (7, 128, (1, 513, 1301)), (9, 500, (1, 33, 70)), (10, 1024, (1, 3, 18)),
                                            (6, 61, (1, 100, 2999)), (5, 32, (1, 4101)), (4, 16, (1, 1023, 1027))])
@pytest.mark.parametrize("chain", [True, False])
def test_same_bits_in_every_batch_and_shape(oracle, n, cols, batches, chain):
    gates = W.mixed_gate_circuit(n, 5 * n, n)
    P, most = W.param_count(gates), max(batches)
    U = W.haar_unitary(1 << n, 3)[:, :cols].copy()
    ps = W.random_params(P, 4, batch=most)
    ctx = nat.Context(0)
    ctx.set_circuit(n, gates)
    ctx.set_target(U)
    ctx.set_fused_cost(True)
    ctx.set_fused_cost_chain(chain)
    for prec, tol in ((nat.PREC_F64, 1e-12), (nat.PREC_F32, 1e-5)):
        print(n, cols, chain, prec, flush=True)
        f, g = combined(ctx, ps, prec)
        for b in (0, most // 2, most - 1):
            fo, go = oracle.optimization_problem_combined(gates, U, n, ps[b])
            assert abs(f[b] - fo) < tol and np.abs(g[b] - go).max() < tol
        for B in batches:
            for first in (0, most - B):
                f2, g2 = combined(ctx, ps[first:first + B], prec)
                assert np.array_equal(f2, f[first:first + B]) and np.array_equal(g2, g[first:first + B])
        for shape in ((4, 1), (4, 8), (2, 2), (2, 4)):
            ctx.set_fused_grad_config(*shape)
            f2, g2 = combined(ctx, ps, prec)
            assert np.array_equal(f2, f) and np.array_equal(g2, g), shape
        ctx.set_fused_grad_config(0, 0)


@pytest.mark.parametrize("mixed", [False, True])
def test_rounds_do_not_depend_on_companions(mixed):
    """The optimiser's rounds with few and with many live runs: every run of a large call
    ends where it ends alone."""
    n, runs = 7, 700
    gates = W.ansatz_layers(n, W.alternating_pairs(n, 10))
    P = W.param_count(gates)
    T = np.array([W.haar_unitary(1 << n, 5), W.haar_unitary(1 << n, 6)])
    index = (np.arange(runs) % 2).astype(np.int32)
    x0 = W.random_params(P, 7, batch=runs)
    opts = default_options(n, max_inner_iterations=4, max_outer_iterations=1, engine="rounds", mixed_precision=mixed)
    ctx = nat.Context(0)
    ctx.set_circuit(n, gates)
    ctx.set_fused_cost(True)
    all_of = decompose_batch(ctx, T, index, x0, opts)
    for pick in ([0], [1, 350, 699], list(range(200, 270))):
        some = decompose_batch(ctx, T, index[pick], x0[pick], opts)
        assert np.array_equal(some["f"], all_of["f"][pick]) and np.array_equal(some["x"], all_of["x"][pick])


def test_batch_beyond_one_launch(oracle):
    """600,000 vectors of a one-block circuit (5 GB of block matrices and partials) run in
    parts, automatically through the same kernels as a few."""
    n, B = 4, 600001
    gates = W.ansatz_layers(n, W.alternating_pairs(n, 12))
    P = W.param_count(gates)
    U = W.haar_unitary(16, 8)
    ps = W.random_params(P, 9, batch=B)
    ctx = nat.Context(0)
    ctx.set_circuit(n, gates)
    ctx.set_target(U)
    f, g = combined(ctx, ps, nat.PREC_F64)
    for first in (0, B // 2 - 3, B - 5):
        f2, g2 = combined(ctx, ps[first:first + 5], nat.PREC_F64)
        assert np.array_equal(f2, f[first:first + 5]) and np.array_equal(g2, g[first:first + 5])
    fo, go = oracle.optimization_problem_combined(gates, U, n, ps[B - 1])
    assert abs(f[B - 1] - fo) < 1e-12 and np.abs(g[B - 1] - go).max() < 1e-12
