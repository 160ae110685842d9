"""The pair network's backward pass takes b2 with all its 24 bits: units whose
pre-activation is the last bits of b2, what is left of it when a product of
two BF16 numbers has cancelled the rest, are active.  dL/db2 is then a sum of
at most 64 counted FP32 rows per target: 1e-5 in relative L2 norm."""
import numpy as np
import pytest

from oracle import mlp_oracle as mo
from test_mlp_gpu import oracle_inputs, random_weights, window_case

pytestmark = pytest.mark.gpu


def last_bits_of_b2(seed=5):
    """(params, signs): every unit's W2 row takes one hidden value c, constant
    over the pairs, times -x, and b2 = c x plus or minus its last bits."""
    rng = np.random.default_rng(seed)
    w = mo.unpack(random_weights(seed))
    c = mo.bf16([1.3])[0]
    W1, W2, b2 = np.zeros((64, 16)), np.zeros((64, 64)), np.zeros(64)
    W1[7, mo.BIAS_FEAT] = c
    signs = np.where(np.arange(64) % 2, 1.0, -1.0)
    for u in range(64):
        while b2[u] == 0.0:
            x = mo.bf16([rng.uniform(0.5, 2.0)])[0]
            b = np.float32(c * x * (1.0 + signs[u] * 2.0 ** -20))
            hi = mo.bf16([b])[0]
            lo = mo.bf16([np.float64(b) - hi])[0]
            if hi + lo == c * x and np.sign(np.float64(b) - c * x) == signs[u]:  # 16 bits are not enough
                W2[u, 7], b2[u] = -x, b
    return mo.pack(W1, W2, b2, w["W3"], w["b3"]), signs


def test_backward_sees_all_of_b2():
    params, signs = last_bits_of_b2()
    ctx, model, w, p = window_case((7, 5, 6), before=3, window=2, seed=9)
    with ctx, model:
        model.set_weights(params)
        _, g = ctx.learn_gradient(model)
        nm = model.norm()
    E, pi, q, nd = oracle_inputs(w, p, nm)
    n = w["pos"].shape[0]
    f = mo.forward(params, E, pi, n, q, nd)
    d_out = 2.0 * (f["out"] - mo.targets_from_window(w["target"], nm.a_scale)) / n
    dH = float(np.float32(nd["agg_scale"])) * (d_out @ mo.unpack(params)["W3"][:, :mo.HID])
    want = np.where(signs > 0, dH[pi].sum(axis=0), 0.0)
    got = g[mo.OFF_B2:mo.OFF_W3]
    assert len(pi) > 0 and np.all(want[signs > 0] != 0)
    assert not np.any(got[signs < 0])
    assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)
