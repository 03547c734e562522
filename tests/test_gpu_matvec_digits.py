"""The Q4_0 projections' integer dot: every launch form (a quarter and a half of a
row per wavefront, a row's blocks loaded by their lanes, staged rows in one, two
and four groups) at its edges, against the float64 oracle, and inputs whose digits
need care: mixed magnitudes inside a block, subnormals, the largest floats,
infinities and NaN."""
import matvec_cases as mc
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
f32 = np.float32
EPS = 1e-6
# of the row's sum of |products|: the rounded y = x w, four roundings a block
# (the halves, at most three times the products in all, and their sum), 8 + 6 + 3
# additions, and the inverse RMS (26 additions of squares under a root, four
# more operations) with its product; each at most 2^-24
TOL = 40 * 2.0 ** -24


def _bound(x, W, w, n, rows):
    """The largest error: TOL of the sum of |products|, and half a step of the
    input's fixed point a value, the step 2^-30 of the power of two above the
    block's largest |x w|."""
    y = np.abs(x if w is None else x * w).reshape(-1, 32)
    step = np.ldexp(1.0, np.frexp(y.max(1).astype(np.float64))[1] - 30)
    per_code = TOL * y + 0.5 * step[:, None]
    inv = 1.0 if w is None else 1.0 / np.sqrt(np.mean(x.astype(np.float64) ** 2) + EPS)
    out = np.empty(rows)
    for r in range(0, rows, 2048):
        b = W[r * (n // 32) * 18:(r + 2048) * (n // 32) * 18].reshape(-1, n // 32, 18)
        d = np.abs(b[:, :, :2].copy().view(np.float16)[:, :, 0].astype(np.float64))
        code = np.abs(np.concatenate([b[:, :, 2:] & 15, b[:, :, 2:] >> 4], 2).astype(np.int8) - 8)
        out[r:r + 2048] = inv * (d * np.einsum("rbv,bv->rb", code.astype(np.float32), per_code.astype(np.float32))).sum(1)
    return out


def _run(rt, x, W, w, n, rows):
    dx, dW, out = rt.upload(x), rt.upload(W), rt.empty(rows)
    dw = None if w is None else rt.upload(w)
    rt.matvec_q4_0_rms(dx, dW, out, n, rows, dw, EPS)
    rt.sync()
    got = out.download(rows)
    for b in (dx, dW, out, dw):
        if b is not None:
            rt.free(b)
    return got


def _check(ora, got, x, W, w, n, rows):
    exact = ora.matvec_q4_0_rms_f64(x, W, w, n, rows, EPS)[0]
    err = np.abs(got.astype(np.float64) - exact) / np.maximum(_bound(x, W, w, n, rows), 1e-300)
    assert np.max(err) <= 1.0, float(np.max(err))


@pytest.mark.parametrize("n,rows", [
    (32, 1), (64, 2048), (2048, 2047), (2080, 3), (4096, 2045), (32, 2049), (512, 2051), (544, 3000), (992, 2064),
    (1056, 2049), (1568, 4099), (2016, 2050), (2304, 3001), (3104, 2052), (1536, 14336), (1536, 12285), (4096, 28667),
    (1024, 28672),
    # where the form changes: 1024, 2048 and 4096 rows, 16, 32, 64 and 96 blocks a row, 2^16 in all
    (512, 1024), (512, 4097), (480, 4369), (32, 65537), (544, 1024), (544, 1025), (1024, 4096), (1024, 4097), (1056, 1025),
    (2048, 2046), (2080, 1024), (2080, 1027), (3072, 2048), (3104, 1025), (4096, 2047)])
@pytest.mark.parametrize("rms", [True, False])
def test_forms(rt, ora, n, rows, rms):
    r = np.random.default_rng(n + rows)
    x = r.standard_normal(n).astype(f32)
    w = (1.0 + 0.1 * r.standard_normal(n)).astype(f32) if rms else None
    W = mc.random_q4_0(r, rows, n)
    _check(ora, _run(rt, x, W, w, n, rows), x, W, w, n, rows)


@pytest.mark.parametrize("kind", ["mixed", "tiny", "subnormal", "huge", "sparse", "zero"])
@pytest.mark.parametrize("n,rows", [(1536, 40), (576, 2200), (1536, 2600)])
def test_magnitudes(rt, ora, kind, n, rows):
    r = np.random.default_rng(len(kind) + n)
    x = r.standard_normal(n).astype(f32)
    if kind == "mixed":
        x = np.ldexp(x, r.integers(-30, 30, n)).astype(f32)
    elif kind == "tiny":
        x *= f32(1e-30)
    elif kind == "subnormal":
        x = (x * f32(1e-20)) * f32(1e-20)
    elif kind == "huge":
        x *= f32(1e30)
    elif kind == "sparse":
        x[r.random(n) < 0.98] = 0.0
    elif kind == "zero":
        x[:] = 0.0
    W = mc.random_q4_0(r, rows, n)
    got = _run(rt, x, W, None, n, rows)
    exact = ora.matvec_q4_0_rms_f64(x, W, None, n, rows, EPS)[0]
    # a result may round into the subnormals: their spacing is 2^-149
    assert np.all(np.abs(got.astype(np.float64) - exact) <= _bound(x, W, None, n, rows) + 40 * 2.0 ** -149)


@pytest.mark.parametrize("n,rows", [(512, 40), (1536, 40), (3072, 1500), (576, 2200), (1536, 2600)])
def test_largest_value_without_weight(rt, ora, n, rows):
    """Each block's largest value meets code 8 (weight 0), so its step shows in
    the others: at 0.9 of a step above the grid and with codes of their sign,
    a truncation to it would be off by 0.9 of a step a value, past the bound."""
    r = np.random.default_rng(n + 1)
    step = 2.0 ** -13  # of 1e5
    k = r.integers(0, 1 << 13, n) + 0.9
    sign = np.where(r.random(n) < 0.5, -1.0, 1.0)
    x = (sign * k * step).astype(f32).reshape(-1, 32)
    at = r.integers(0, 32, n // 32)
    x[np.arange(n // 32), at] = 1e5
    x = x.reshape(-1)
    code = 8 + np.where(np.sign(x) > 0, 1, -1) * r.integers(0, 8, (rows, n))
    code.reshape(rows, -1, 32)[:, np.arange(n // 32), at] = 8
    W = mc.random_q4_0(r, rows, n).reshape(rows, n // 32, 18)
    code = code.reshape(rows, n // 32, 32)
    W[:, :, 2:] = code[:, :, :16] | (code[:, :, 16:] << 4)
    W = W.reshape(-1)
    _check(ora, _run(rt, x, W, None, n, rows), x, W, None, n, rows)


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("n,rows", [(1536, 40), (576, 2200), (1536, 2600)])
def test_not_finite(rt, value, n, rows):
    r = np.random.default_rng(3)
    x = r.standard_normal(n).astype(f32)
    x[n // 2 + 5] = value
    assert np.isnan(_run(rt, x, mc.random_q4_0(r, rows, n), None, n, rows)).all()
