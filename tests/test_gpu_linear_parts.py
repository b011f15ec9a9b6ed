"""Linears over parts of K: the pass that sums the parts four columns at a time, against the one element at a time that a bias off its boundary
takes, bit for bit, and against float64."""
import numpy as np
import pytest

from tests.util import down, rand, up

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("splits", [2, 3, 4, 5])
@pytest.mark.parametrize("m,n,form", [(65, 4, {}), (129, 260, dict(bias=1)), (97, 264, dict(bias=1, act="gelu")), (200, 516, dict(bias=1, residual=1)),
                                      (131, 132, dict(bias=1, bias2=1, act="new_gelu", act_from=66)), (70, 256, dict(bias=1, act="silu", glu=True)),
                                      (140, 512, dict(bias=1, n1=128)), (140, 268, dict(bias=1, n1=130)), (77, 1030, dict(bias=1, act="relu"))])
def test_sum_of_parts(hip, m, n, form, splits):
    from rai_amd import ops as R

    k = 1088
    g = np.random.Generator(np.random.PCG64(m * n + splits))
    x, w = rand(g, (m, k), "bf16"), rand(g, (n, k), "bf16", k ** -0.5)
    wide = {b: rand(g, (n + 1,), "bf16") for b in ("bias", "bias2") if form.get(b)}
    res = rand(g, (m, n), "bf16") if form.get("residual") else None
    kw = {key: form[key] for key in ("act", "act_from", "glu", "n1") if key in form}
    if res is not None:
        kw["residual"] = up(res, "bf16")

    def run(shifted):
        biases = {b: up(v, "bf16").narrow(0, 1, n) if shifted else up(np.ascontiguousarray(v[1:]), "bf16") for b, v in wide.items()}
        out = R.linear_packed(up(x, "bf16"), up(w, "bf16"), k_splits=splits, **biases, **kw)
        return [down(o) for o in (out if isinstance(out, tuple) else (out,))]

    a, b = run(False), run(True)
    assert all(np.array_equal(p, q) for p, q in zip(a, b))
    if "act" in form:
        return   # (their values are other tests')
    want = x.astype(np.float64) @ w.T.astype(np.float64) + sum(v[1:].astype(np.float64) for v in wide.values()) + (0 if res is None else res)
    got = np.concatenate([p.astype(np.float64) for p in a], 1)
    # products exact, k + a few additions of f32 below the sum of magnitudes, one rounding to bf16 (2^-9 of a value's binade)
    size = np.abs(x).astype(np.float64) @ np.abs(w).T.astype(np.float64) + 4
    assert np.all(np.abs(got - want) <= (k + 8) * 2.0 ** -24 * size + 2.0 ** -8 * np.abs(want))
