"""The persistent solver's evaluations with four rows per lane (one circuit of 3 or 4
qubits) where they can go wrong: fewer columns than rows, a trace offset, every gate kind,
around and beyond the 64 op words a wavefront holds, gates on one qubit only, mixed
precision; against the lockstep rounds from the same starts."""
import numpy as np
import pytest

from squander_hip import _native as nat
from squander_hip import decompose_batch, default_options
from squander_hip import workloads as W

pytestmark = pytest.mark.gpu


def both(n, gates, cols, off, mixed, evals):
    P, d = W.param_count(gates), 1 << n
    rng = np.random.default_rng(n * 100 + cols)
    T = np.array([np.linalg.qr(rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d)))[0][:, :cols]
                  for _ in range(5)])
    x0 = W.random_params(P, 3, batch=37)
    index = (np.arange(37) % 5).astype(np.int32)
    out = []
    for engine in ("persistent", "rounds"):
        ctx = nat.Context(0)
        ctx.set_circuit(n, gates)
        ctx.set_trace_offset(off)
        opts = default_options(n, max_inner_iterations=evals, max_outer_iterations=1, engine=engine,
                               mixed_precision=mixed)
        out.append(decompose_batch(ctx, T, index, x0, opts))
        again = decompose_batch(ctx, T, index, x0, opts)  # on the kept buffers
        assert np.array_equal(again["x"], out[-1]["x"]) and np.array_equal(again["f"], out[-1]["f"])
    return out


@pytest.mark.parametrize("n", [3, 4])
@pytest.mark.parametrize("count", [1, 63, 64, 65, 150])
@pytest.mark.parametrize("ragged", [False, True])
def test_against_rounds(n, count, ragged):
    print(n, count, ragged, flush=True)
    gates = W.mixed_gate_circuit(n, count, 10 * n + count)
    gates = np.concatenate([gates, [[nat.GATE_U3, n - 1, -1, W.param_count(gates)]]]).astype(np.int32)
    d = 1 << n
    a, b = both(n, gates, d - 3 if ragged else d, 2 if ragged else 0, False, 2)
    # two evaluations: the sums' rounding (1e-15), at most 1e4 times that after a step
    assert np.abs(a["f"] - b["f"]).max() < 1e-11 and np.abs(a["x"] - b["x"]).max() < 1e-11
    a, b = both(n, gates, d, 0, True, 1)  # the complex64 evaluations
    assert np.abs(a["f"] - b["f"]).max() < 1e-5


@pytest.mark.parametrize("n", [3, 4])
def test_one_qubit_only(n):
    gates = np.asarray([[nat.GATE_U3, n - 1, -1, 0], [nat.GATE_RX, n - 1, -1, 3]], dtype=np.int32)
    a, b = both(n, gates, 1 << n, 0, False, 2)
    assert np.abs(a["f"] - b["f"]).max() < 1e-11 and np.abs(a["x"] - b["x"]).max() < 1e-11


@pytest.mark.parametrize("n", [3, 4])
@pytest.mark.parametrize("kind", ["ansatz", "mixed"])
@pytest.mark.parametrize("mixed_precision", [False, True])
def test_same_bits_as_a_column_per_lane(n, kind, mixed_precision):
    """Problems of their own circuits are evaluated with a column per lane: the same runs
    end at the same bits after the same evaluations, line searches included."""
    from squander_hip import decompose_problems
    gates = (W.ansatz_layers(n, W.alternating_pairs(n, 3 * n)) if kind == "ansatz"
             else W.mixed_gate_circuit(n, 8 * n, 40 + n))
    P, d, runs = W.param_count(gates), 1 << n, 64
    rng = np.random.default_rng(n)
    T = np.array([np.linalg.qr(rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d)))[0] for _ in range(5)])
    x0 = W.random_params(P, 3, batch=runs)
    index = (np.arange(runs) % 5).astype(np.int32)
    opts = default_options(n, max_inner_iterations=9, max_outer_iterations=1, engine="persistent",
                           mixed_precision=mixed_precision)
    ctx = nat.Context(0)
    ctx.set_circuit(n, gates)
    a = decompose_batch(ctx, T, index, x0, opts)
    b = decompose_problems(ctx, [(n, gates, T[index[r]], x0[r]) for r in range(runs)], opts)
    assert np.array_equal(a["evals"], b["evals"]) and np.array_equal(a["f"], b["f"])
    assert np.array_equal(a["x"], np.array(b["x"]))
