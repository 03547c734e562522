"""The row-per-workgroup norm engines (f32; hidden 2049 to 8192, and narrower
rows between the decode and the prefill engines): the exact fold bit for bit
against the oracle, the tree sum against the operator tolerance, at the edges
of each workgroup shape and of its runs."""
import cases
import numpy as np
import pytest
from test_gpu_parity import assert_bits, assert_bits_nan_equal
from test_gpu_reduction import assert_rms_tolerance, rms_f64

pytestmark = pytest.mark.gpu

# shapes change at 2560, 3072, 4096, 5120 and 6144; runs of 64 S values end at 256 + 64 S k
EDGES = [2052, 2304, 2556, 2560, 2564, 3072, 3076, 4092, 4096, 4100, 5120, 5124, 6144, 6148, 8188, 8192]


@pytest.mark.parametrize("hidden", EDGES)
@pytest.mark.parametrize("mode", ["plain", "residual", "addnorm", "addscale"])
def test_exact_rows(rt, ora, hidden, mode):
    rows = 33
    inp, m = cases.rms_case(rows, hidden, 1e-6, 9000 + hidden, mode)
    inp["x"] = cases.adversarial_rows(rows, hidden, 9100 + hidden)
    assert_bits_nan_equal(f"rms_{mode}", cases.rms_gpu(rt, inp, m), cases.rms_oracle(ora, inp, m))


@pytest.mark.parametrize("rows,hidden", [(768, 4100), (768, 5120), (768, 5124), (768, 6144)])
@pytest.mark.parametrize("mode", ["residual", "plain"])
def test_exact_rows_many(rt, ora, rows, hidden, mode):
    inp, m = cases.rms_case(rows, hidden, 1e-6, 9600 + hidden, mode)
    inp["x"] = cases.adversarial_rows(rows, hidden, 9700 + hidden)
    assert_bits_nan_equal(f"rms_{mode}", cases.rms_gpu(rt, inp, m), cases.rms_oracle(ora, inp, m))


@pytest.mark.parametrize("rows,hidden", [(513, 260), (513, 1024), (513, 1028), (513, 1536), (257, 1540), (257, 2048),
                                         (512, 1536), (256, 2048), (1023, 576), (1024, 260), (2047, 1536), (1024, 1540),
                                         (2047, 2048), (2048, 2048)])
@pytest.mark.parametrize("mode", ["residual", "addnorm"])
def test_exact_rows_between_engines(rt, ora, rows, hidden, mode):
    inp, m = cases.rms_case(rows, hidden, 1e-6, 9800 + rows + hidden, mode)
    inp["x"] = cases.adversarial_rows(rows, hidden, 9900 + hidden)
    assert_bits_nan_equal(f"rms_{mode}", cases.rms_gpu(rt, inp, m), cases.rms_oracle(ora, inp, m))


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
