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


@pytest.mark.parametrize("splits", [2, 5])
@pytest.mark.parametrize("m,n,form", [(77, 1030, {}), (70, 264, dict(act_from=100)), (130, 260, dict(residual=1)), (66, 512, dict(n1=128))])
def test_parts_under_an_activation(hip, m, n, form, splits):
    """Against float64, relu being exact; every row and column, whichever pass sums them."""
    from rai_amd import ops as R

    k = 1088
    g = np.random.Generator(np.random.PCG64(m * n + splits))
    x, w, b = rand(g, (m, k), "bf16"), rand(g, (n, k), "bf16", k ** -0.5), rand(g, (n,), "bf16")
    res = rand(g, (m, n), "bf16") if form.get("residual") else None
    kw = {key: form[key] for key in ("act_from", "n1") if key in form} | ({} if res is None else {"residual": up(res, "bf16")})
    out = R.linear_packed(up(x, "bf16"), up(w, "bf16"), bias=up(b, "bf16"), act="relu", k_splits=splits, **kw)
    got = np.concatenate([down(o).astype(np.float64) for o in (out if isinstance(out, tuple) else (out,))], 1)
    want = x.astype(np.float64) @ w.T.astype(np.float64) + b
    at = form.get("act_from", 0)
    want[:, at:] = np.maximum(want[:, at:], 0)
    want += 0 if res is None else res
    size = np.abs(x).astype(np.float64) @ np.abs(w).T.astype(np.float64) + 4
    assert np.all(np.abs(got - want) <= (k + 8) * 2.0 ** -24 * size + 2.0 ** -8 * np.abs(want))


@pytest.mark.parametrize("rows", [70, 131])
def test_parts_onto_an_f32_stream(hip, rows):
    """[o | down] of a hybrid decoder's prompt, 1984 columns in parts: its outputs and the residual are f32."""
    import ctypes as C

    from oracle import bezadra
    from rai_amd._lib import call
    from tests import bezadra_models as bm
    from tests.test_gpu_bezadra import deep_close

    width, ff = 1024, 1920
    name, parts = C.create_string_buffer(32), C.c_int32()
    call("rai_hip_linear_plan", 0, rows, ff + 64, width, 12 * rows * width * 4, name, 32, C.byref(parts))
    assert parts.value > 1
    cfg = bm.config([bm.attention(heads=1, kv_heads=1, dim=64, vdim=64, ff=ff)], width=width, vocab=600)
    p = bezadra.random_params(cfg, "bf16", 3)
    dec = bm.build(cfg, p, "bf16", max_batch=1, max_context=rows)
    ids = np.random.Generator(np.random.PCG64(rows)).integers(0, 600, (1, rows)).astype(np.uint32)
    deep_close(dec.forward(ids)[0][0], bezadra.Model(cfg, p).logits(ids[0])[-1], "bf16", f"{rows} rows")
    dec.close()
