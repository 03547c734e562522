"""QK-norm + RoPE by units: every register-row count of the token engine, heads
past one wavefront's units (17 and more), and head_dim 64 with two heads per
register row, on heads built to break a reordered fold."""
import cases
import numpy as np
import pytest
from atlas_amd import ATLAS_REDUCTION_SEQUENTIAL, ATLAS_REDUCTION_WIDE, rope_tables_gemma4

pytestmark = pytest.mark.gpu

# (head_dim, q_heads, has_key, tokens): one, two and four rows per wavefront,
# then the whole token (<= 16 units) or nine rows (more), at odd unit counts
SHAPES = [
    (64, 1, False, 3), (64, 4, True, 131), (64, 8, True, 611), (64, 15, True, 1100), (64, 15, True, 1251),
    (64, 9, True, 2051), (64, 16, True, 1180), (64, 24, False, 900), (64, 40, True, 501),
    (128, 4, True, 133), (128, 16, True, 300), (128, 32, True, 333), (128, 24, True, 810), (128, 12, True, 1600),
    (256, 16, True, 7), (256, 32, True, 141), (256, 24, False, 290), (256, 16, True, 420), (256, 17, False, 651),
    (256, 32, True, 340), (256, 7, False, 1000), (256, 8, True, 1223),
    (512, 16, True, 5), (512, 16, True, 110), (512, 24, True, 210), (512, 16, True, 501), (512, 9, True, 850),
    (512, 33, True, 253),
    # one wavefront with a token's few units, and the token count from which it takes up to four or six
    (64, 2, False, 9), (64, 3, True, 1300), (128, 1, False, 5), (128, 1, True, 1200), (128, 5, True, 1207),
    (256, 1, False, 1000), (256, 4, True, 1199), (256, 4, True, 1200), (256, 6, True, 1490), (512, 1, True, 1150),
    (512, 2, True, 1201), (512, 15, True, 131), (512, 6, True, 1210),
]


@pytest.mark.parametrize("head_dim,q_heads,has_key,tokens", SHAPES)
def test_units_bit_exact(rt, ora, head_dim, q_heads, has_key, tokens):
    inp, m = cases.qk_case(tokens, q_heads, head_dim, head_dim // 2, 1e6, 1e-6, 60 + tokens + head_dim, has_key)
    inp["q"] = cases.adversarial_rows(tokens * q_heads, head_dim, 61 + tokens).reshape(-1)
    tables = rope_tables_gemma4(inp["pos"], head_dim // 2, head_dim, 1e6)
    cases.assert_bits_nan_equal("qk", cases.qk_gpu(rt, inp, m, tables), cases.qk_oracle(ora, inp, m))


@pytest.mark.parametrize("head_dim,q_heads,tokens", [(64, 5, 40), (64, 24, 900), (256, 16, 420), (512, 16, 501)])
def test_units_tree_sum(rt, ora, head_dim, q_heads, tokens):
    inp, m = cases.qk_case(tokens, q_heads, head_dim, head_dim // 2, 1e4, 1e-6, 70 + tokens + head_dim)
    tables = rope_tables_gemma4(inp["pos"], head_dim // 2, head_dim, 1e4)
    rt.set_reduction(ATLAS_REDUCTION_WIDE)
    try:
        got = cases.qk_gpu(rt, inp, m, tables)
    finally:
        rt.set_reduction(ATLAS_REDUCTION_SEQUENTIAL)
    # f32 sums of at most 512 squares in another order: 512 x 2^-24 bounds the
    # relative change of a row's sum, half of it that of its scale
    for g, e in zip(got, cases.qk_oracle(ora, inp, m)):
        assert np.linalg.norm(g - e) <= 1e-6 * np.linalg.norm(e)


def test_more_tokens_than_one_launch(rt, ora):
    """A launch holds fewer than 2^26 wavefronts and 18 + 1 heads take two a
    token: the tokens around 2^25 (165 GB of heads, in place)."""
    from atlas_amd import OperatorError

    d, qh, half = 64, 18, 32
    tokens, split = (1 << 25) + 5, ((1 << 26) - 8) // 2
    bufs = []
    try:
        for n in (tokens * qh * d, tokens * d, tokens * half):
            bufs.append(rt.alloc(4 * n))
    except OperatorError as e:
        assert e.kind == "OutOfMemory"
        for b in bufs:
            rt.free(b)
        pytest.skip("needs 168 GB of free device memory")
    q, k, rope = bufs  # cosine and sine share their rows
    try:
        rng = np.random.default_rng(2)
        near = np.array([0, split - 1, split, (1 << 25) - 1, 1 << 25, tokens - 1])
        x = rng.standard_normal((near.size, qh * d), dtype=np.float32)
        y = rng.standard_normal((near.size, d), dtype=np.float32)
        cs = rng.standard_normal((near.size, half), dtype=np.float32)
        w = rng.standard_normal((2, d), dtype=np.float32)
        for i, t in enumerate(near):
            for b, v in ((q, x[i]), (k, y[i]), (rope, cs[i])):
                b.offset(v.nbytes * int(t)).upload(v)
        qw, kw = rt.upload(w[0]), rt.upload(w[1])
        rt.qk_norm_rope(q, k, qw, kw, rope, rope, q, k, tokens, qh, 1, d, half, 1e-6)
        rt.sync()
        eq, ek = ora.qk_norm_rope(x, y, w[0], w[1], cs, cs, near.size, qh, True, d, half, 1e-6)
        for i, t in enumerate(near):
            assert np.array_equal(q.offset(4 * qh * d * int(t)).download(qh * d), eq.reshape(x.shape)[i]), t
            assert np.array_equal(k.offset(4 * d * int(t)).download(d), ek.reshape(y.shape)[i]), t
    finally:
        for b in bufs:
            rt.free(b)
