"""The row-per-workgroup norm engines (f32; hidden 2049 to 8192, and narrower
rows below the prefill engines): the exact fold bit for bit against the oracle,
the tree sum against the operator tolerance, at the edges of each workgroup
shape and of its segments and windows."""
import cases
import numpy as np
import pytest
from test_gpu_parity import assert_bits, assert_bits_nan_equal
from test_gpu_reduction import assert_rms_tolerance, rms_f64

pytestmark = pytest.mark.gpu

# shapes change at 1024, 2048, 3072, 4096 and 6144; segments are 64 wide, a pass of runs 2048
EDGES = [516, 576, 1020, 1024, 1028, 1088, 1536, 2044, 2048, 2052, 2304, 2556, 2564, 3072, 3076, 4092, 4096, 4100, 5124,
         6144, 6148, 8188, 8192]


@pytest.mark.parametrize("hidden", EDGES)
@pytest.mark.parametrize("mode", ["plain", "residual", "addnorm", "addscale"])
def test_exact_rows(rt, ora, hidden, mode):
    rows = 33
    inp, m = cases.rms_case(rows, hidden, 1e-6, 9000 + hidden, mode)
    inp["x"] = cases.adversarial_rows(rows, hidden, 9100 + hidden)
    assert_bits_nan_equal(f"rms_{mode}", cases.rms_gpu(rt, inp, m), cases.rms_oracle(ora, inp, m))


# rows past the eight-wavefront shapes', and the last and first of each engine
ROWS = [(513, 1028), (512, 2048), (513, 2048), (513, 2052), (513, 3072), (513, 3076), (513, 4096), (768, 4100), (768, 6144),
        (256, 8192), (257, 6148), (257, 8192), (1, 512), (1, 516), (800, 260), (801, 260), (801, 380), (800, 384), (801, 384), (2047, 380), (800, 512), (801, 512),
        (2047, 516), (2047, 1536), (2047, 2048), (2048, 516), (2048, 2048)]


@pytest.mark.parametrize("rows,hidden", ROWS)
@pytest.mark.parametrize("mode", ["residual", "plain", "addnorm"])
def test_exact_rows_many(rt, ora, rows, hidden, mode):
    inp, m = cases.rms_case(rows, hidden, 1e-6, 9600 + rows + hidden, mode)
    inp["x"] = cases.adversarial_rows(rows, hidden, 9700 + hidden)
    assert_bits_nan_equal(f"rms_{mode}", cases.rms_gpu(rt, inp, m), cases.rms_oracle(ora, inp, m))


@pytest.mark.parametrize("rows,hidden", [(33, 576), (33, 1536), (513, 1536), (33, 2560), (513, 2560), (33, 4096),
                                         (513, 4096), (33, 6144), (33, 8192), (257, 8192)])
def test_exact_rows_more_crossings_than_windows(rt, ora, rows, hidden):
    # sums that double (row r: every 1 + r % 9 segments), start late, or run into infinity
    rng = np.random.default_rng(hidden + rows)
    inp, m = cases.rms_case(rows, hidden, 1e-6, 9900 + hidden, "residual")
    x = rng.standard_normal((rows, hidden)).astype(np.float32)
    seg = np.arange(hidden) // 64
    for r in range(rows):
        grow = np.exp2(0.5 * (seg // (1 + r % 9)) - 30.0) if r % 4 else np.exp2(0.0 * seg)
        x[r] *= grow.astype(np.float32)
        if r % 5 == 2:
            x[r, : 64 * int(rng.integers(1, hidden // 64))] = 0.0
        if r % 11 == 7:
            x[r] *= np.float32(2.0 ** 62)  # finite squares whose sum may overflow
    inp["x"] = x.reshape(-1)
    assert_bits_nan_equal("rms_residual", cases.rms_gpu(rt, inp, m), cases.rms_oracle(ora, inp, m))


@pytest.mark.parametrize("rows,hidden", [(1, 4096), (701, 2560), (300, 8192)])
@pytest.mark.parametrize("mode", ["residual", "addscale"])
def test_exact_rows_default_reduction(rt_auto, ora, rows, hidden, mode):
    inp, m = cases.rms_case(rows, hidden, 1e-6, 9200 + rows + hidden, mode)
    assert_bits(f"rms_{mode}", cases.rms_gpu(rt_auto, inp, m), cases.rms_oracle(ora, inp, m))


@pytest.mark.parametrize("hidden", [2052, 3072, 3076, 4096, 4100, 6144, 6148, 8192])
@pytest.mark.parametrize("mode", ["plain", "addnorm"])
def test_tree_rows(rt_auto, ora, hidden, mode):
    rows = 17
    inp, m = cases.rms_case(rows, hidden, 1e-6, 9300 + hidden, mode)
    if mode == "plain":
        inp["x"] = cases.adversarial_rows(rows, hidden, 9400 + hidden)
    got, exp = cases.rms_gpu(rt_auto, inp, m), cases.rms_oracle(ora, inp, m)
    if mode == "addnorm":
        assert_bits("residual_out", got[:1], exp[:1])
    base = inp["x"] if mode == "plain" else exp[0]
    assert_rms_tolerance(mode, got[-1], exp[-1], rms_f64(base, inp["w"], rows, hidden, 1e-6))


def test_in_place(rt, ora):
    rows, h, eps = 9, 4096, 1e-6
    inp, m = cases.rms_case(rows, h, eps, 9500, "residual")
    n_exp, out_exp = ora.rms_norm_residual(inp["x"], inp["w"], inp["res"], rows, h, eps)
    work, state, w = rt.upload(inp["x"]), rt.upload(inp["res"]), rt.upload(inp["w"])
    rt.rms_norm_residual(work, w, state, work, state, rows, h, eps)
    rt.sync()
    assert_bits("aliased", [work.download(rows * h), state.download(rows * h)], [np.asarray(n_exp), np.asarray(out_exp)])


def test_more_rows_than_one_launch(rt, ora):
    """A launch holds fewer than 2^32 threads, 512 a row at this width; the rows
    around 2^23 (137 GB of them, in place) in both orders."""
    from atlas_amd import ATLAS_REDUCTION_SEQUENTIAL, ATLAS_REDUCTION_WIDE, OperatorError

    hidden, rows, eps = 4100, (1 << 23) + 3, 1e-6
    try:
        buf = rt.alloc(4 * hidden * rows)
    except OperatorError as e:
        assert e.kind == "OutOfMemory"
        pytest.skip("needs 137 GB of free device memory")
    try:
        rng = np.random.default_rng(1)
        w = rng.standard_normal(hidden).astype(np.float32)
        dw = rt.upload(w)
        near = [0, (1 << 23) - 2, (1 << 23) - 1, 1 << 23, rows - 1]
        for order in (ATLAS_REDUCTION_SEQUENTIAL, ATLAS_REDUCTION_WIDE):
            x = rng.standard_normal((len(near), hidden)).astype(np.float32)
            for r, v in zip(near, x):
                buf.offset(4 * hidden * r).upload(v)
            rt.set_reduction(order)
            rt.rms_norm(buf, dw, buf, rows, hidden, eps)
            rt.sync()
            got = np.stack([buf.offset(4 * hidden * r).download(hidden) for r in near])
            exp = np.asarray(ora.rms_norm(x.reshape(-1), w, len(near), hidden, eps)).reshape(got.shape)
            # 4100 squares summed in another order: at most 4100 x 2^-24 of the sum, half of it of its scale
            assert np.array_equal(got, exp) if order == ATLAS_REDUCTION_SEQUENTIAL else \
                np.max(np.abs(got - exp) / np.abs(exp)) <= 2 * 4100 * 2.0 ** -24
    finally:
        rt.set_reduction(ATLAS_REDUCTION_SEQUENTIAL)
        rt.free(buf)
