"""CPU model of the segment-parity fold (rms_row_exact_kernel in
atlas_amd/csrc/norm_row_kernels.hip): the in-order f32 sum of a row's squares,
bit for bit, from segments folded side by side.

Inside a binade a running sum is an integer count of its ulps, and adding a
non-negative value raises it by a whole number of ulps that depends on the sum
only through its parity (a tie rounds to even).  So a segment of 64 values
that does not leave the binade raises every even start by one amount and every
odd start by another: two folds from any even and any odd start near the
estimate give both, and a run of such segments composes as a function of the
first start's parity.  Segments that may cross a power of two (by the
estimate, with a margin) are folded from a window of consecutive starts; the
exact start selects its fold, or the segment is folded in order.

The model is checked against the sequential fold on the rows of the GPU tests;
planted mistakes (one parity for both, the windows' nearest start) must fail."""
import cases
import numpy as np
import pytest
from test_fold_model import _bits, _fold_from, _from_bits, _rows, sequential_fold

f32 = np.float32
u32 = np.uint32
MARGIN = 64


def _fold_bits(start_bits, values):
    with np.errstate(invalid="ignore", over="ignore"):
        return _fold_from(np.array(start_bits, np.int64).astype(u32).view(f32), values).view(u32).astype(np.int64)


def segment_fold_model(sq, window=32, parity=True, exact=True, stats=None):
    n = -(-sq.size // 64)
    seg = np.zeros(64 * n, f32)
    seg[:sq.size] = sq
    seg = seg.reshape(n, 64)
    with np.errstate(invalid="ignore", over="ignore"):
        lanes = seg.reshape(n, 16, 4)
        part = ((lanes[..., 0] + lanes[..., 1]) + (lanes[..., 2] + lanes[..., 3])).astype(f32)
        est = np.concatenate([[f32(0)], np.cumsum(part.sum(1, dtype=f32), dtype=f32)])  # any order would do
    eb = est.view(u32).astype(np.int64)
    sb = _bits(sequential_fold(seg[:4].reshape(-1)))
    k = 4
    while k < n:
        lo, hi = max(eb[k] - MARGIN, 0) >> 23, (eb[k + 1] + MARGIN) >> 23
        inc = None
        if lo == hi:
            start = [eb[k] & ~1, eb[k] | 1]
            end = _fold_bits(start, seg[k])
            if all(s >> 23 == e >> 23 for s, e in zip(start, end)):
                inc = [int(e - s) for s, e in zip(start, end)]
        if inc is not None and sb >> 23 == lo:
            nxt = sb + inc[sb & 1 if parity else 0]
            if nxt >> 23 == lo:
                sb, k = nxt, k + 1
                continue
        if stats is not None:
            stats["special"] = stats.get("special", 0) + 1
        at = sb - (eb[k] - window // 2)
        if not exact:
            at = min(max(at, 0), window - 1)
        if lo != hi and 0 <= at < window:
            sb = int(_fold_bits([(eb[k] - window // 2 + at) & 0xFFFFFFFF], seg[k])[0])
        else:
            if stats is not None:
                stats["in order"] = stats.get("in order", 0) + 1
            sb = int(_fold_bits([sb], seg[k])[0])
        k += 1
    return _from_bits(sb)


def _wide_rows():
    yield from _rows()
    r = np.random.default_rng(78)
    for hidden in (4096, 8192, 2052):
        yield f"gaussian_{hidden}", r.standard_normal((40, hidden)).astype(f32)
        yield f"adversarial_{hidden}", cases.adversarial_rows(48, hidden, 6000 + hidden).reshape(48, hidden)


@pytest.mark.parametrize("window", [64, 32, 4])
def test_model_reproduces_the_sequential_fold(window):
    stats, checked = {}, 0
    for name, x in _wide_rows():
        for row in x[::1 if window == 32 else 4]:
            with np.errstate(over="ignore", invalid="ignore"):
                sq = (row * row).astype(f32)
            want, got = sequential_fold(sq), segment_fold_model(sq, window, stats=stats)
            assert _bits(want) == _bits(got) or (np.isnan(want) and np.isnan(got)), (name, window, want, got)
            checked += 1
    assert checked > 300 and stats["special"] > checked and stats["in order"] > 0


@pytest.mark.parametrize("mistake", [{"parity": False}, {"exact": False, "window": 4}])
def test_planted_mistakes_fail(mistake):
    wrong = 0
    for _, x in _rows():
        for row in x[::3]:
            with np.errstate(over="ignore", invalid="ignore"):
                sq = (row * row).astype(f32)
            want = sequential_fold(sq)
            if np.isfinite(want):
                wrong += _bits(want) != _bits(segment_fold_model(sq, **mistake))
    assert wrong > 0
