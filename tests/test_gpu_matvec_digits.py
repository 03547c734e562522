"""The Q4_0 projections' integer dot: every launch form (a quarter of a row per
wavefront, a row's blocks loaded by their lanes, staged rows in one, two and
four groups) at its edges, against the float64 oracle, and inputs whose digits
need care: mixed magnitudes inside a block, subnormals, the largest floats,
infinities and NaN."""
import matvec_cases as mc
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
f32 = np.float32
EPS = 1e-6
# per row: three roundings a block, up to 8 + 6 additions and 4 ulp of the
# inverse RMS, each at most 2^-24 of the sum of |products|
TOL = 22 * 2.0 ** -24


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
    exact, mag = ora.matvec_q4_0_rms_f64(x, W, w, n, rows, EPS)
    err = np.abs(got.astype(np.float64) - exact)
    assert np.all(err <= TOL * mag), float(np.max(err / np.maximum(mag, 1e-300)))


@pytest.mark.parametrize("n,rows", [
    (32, 1), (64, 2048), (2048, 2047), (2080, 3), (4096, 2045), (32, 2049), (512, 2051), (544, 3000), (992, 2064),
    (1056, 2049), (1568, 4099), (2016, 2050), (2304, 3001), (3104, 2052), (1536, 14336), (1536, 12285), (4096, 28667),
    (1024, 28672),
    # where the form changes: 1024, 2048 and 4096 rows, 16, 32, 64 and 96 blocks a row, 2^16 in all
    (512, 1024), (512, 4097), (480, 4369), (32, 65537), (544, 1024), (544, 1025), (1024, 4096), (1024, 4097), (1056, 1025), (2048, 2046),
    (2080, 1024), (2080, 1027), (3072, 2048), (3104, 1025), (4096, 2047)])
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
    exact, mag = ora.matvec_q4_0_rms_f64(x, W, None, n, rows, EPS)
    # a result may round into the subnormals: their spacing is 2^-149
    assert np.all(np.abs(got.astype(np.float64) - exact) <= TOL * mag + 40 * 2.0 ** -149)


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("n,rows", [(1536, 40), (576, 2200), (1536, 2600)])
def test_not_finite(rt, value, n, rows):
    r = np.random.default_rng(3)
    x = r.standard_normal(n).astype(f32)
    x[n // 2 + 5] = value
    assert np.isnan(_run(rt, x, mc.random_q4_0(r, rows, n), None, n, rows)).all()
