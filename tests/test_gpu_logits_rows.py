"""The soft cap + argmax rows that are not a multiple of 4 values or not
16-byte aligned (16-byte accesses at 4-byte alignment), their tails, in place,
and the soft cap's shorter divisions over caps and magnitudes at the edges of
the range that takes them."""
import ctypes

import numpy as np
import pytest
from test_gpu_division import _lib as division_lib

pytestmark = pytest.mark.gpu
f32 = np.float32


def _rows(seed, rows, count, std):
    r = np.random.default_rng(seed)
    x = (r.standard_normal(rows * count) * std).astype(f32).reshape(rows, count)
    for i in range(rows):  # ties on the maximum, the last one at or near the row's end
        x[i, [i % count, max(0, count - 1 - i % 6)]] = f32(9 * std)
        if count > 8:
            x[i, (7 * i + 3) % count] = np.nan
    return x.reshape(-1)


def _same(got, exp):
    return np.array_equal(np.where(np.isnan(got), 0, got).view(np.uint32), np.where(np.isnan(exp), 0, exp).view(np.uint32)) \
        and np.array_equal(np.isnan(got), np.isnan(exp))


@pytest.mark.parametrize("rows,count", [(1, 3), (5, 4), (7, 5), (9, 7), (3, 1023), (3, 1026), (2, 4095), (2, 4099),
                                        (1, 32001), (130, 32001), (85, 50257), (3, 1400005),
                                        # where the launch form changes: 512 values, 2^22 in all, steps
                                        # of 4096 that are 0.6 full
                                        (4, 511), (4, 513), (9000, 509), (8300, 515), (1710, 2457), (1710, 2458),
                                        (1025, 4097), (33, 512), (20, 260), (70000, 5)])
@pytest.mark.parametrize("offset,in_place", [(0, False), (4, False), (12, True)])
def test_rows(rt, ora, rows, count, offset, in_place):
    x = _rows(rows + count, rows, count, 8.0)
    exp_c, exp_s = ora.softcap_argmax_rows(x, rows, count, 30.0)
    src = rt.empty(x.size + 8).offset(offset)
    src.upload(x)
    dst = src if in_place else rt.empty(x.size + 8).offset(offset)
    sel = rt.empty(rows, np.uint32)
    rt.softcap_argmax(src, dst, sel, rows, count, 30.0)
    rt.sync()
    assert _same(dst.download(x.size), exp_c)
    assert np.array_equal(sel.download(rows, np.uint32), exp_s)
    src.upload(x)
    rt.argmax(src, sel, rows, count)
    rt.sync()
    assert np.array_equal(sel.download(rows, np.uint32), ora.softcap_argmax_rows(x, rows, count, 0.0)[1])
    for b in {id(src): src, id(dst): dst}.values():
        b.ptr -= offset
        rt.free(next(o for o in rt._buffers if o.ptr == b.ptr))


# 0x3fffffff has an all-ones significand; 2^-20 and 2^20 bound the plain caps
CAPS = [30.0, 50.0, 1.0, 0.37, float(np.array([0x3FFFFFFF], np.uint32).view(f32)[0]), 3.0, 7.0e5, 2.0 ** -20, 2.0 ** 20,
        2.0 ** -21, 1.5e6, 1e-30, 1e30]


@pytest.mark.parametrize("cap", CAPS)
def test_caps_and_magnitudes(rt, ora, cap):
    r = np.random.default_rng(5)
    mant = (1.0 + r.random((400, 1024))).astype(f32)
    sign = np.where(r.random(mant.shape) < 0.5, -1, 1).astype(f32)
    near = np.ldexp(mant, r.integers(-3, 4, mant.shape)).astype(f32) * f32(cap)  # about the cap: both tanh ranges
    far = np.ldexp(mant, r.integers(-75, 66, mant.shape)).astype(f32)            # across the plain range's edges
    edge = np.tile(np.array([2.0 ** -70, 2.0 ** 60, 1.0], f32), 342)[:1024] * mant[:8]
    with np.errstate(over="ignore"):
        x = np.concatenate([near * sign, far * sign, edge, -edge]).astype(f32).reshape(-1)
    buf, out = rt.upload(x), rt.empty(x.size)
    rt.softcap(buf, out, x.size, cap)
    rt.sync()
    assert _same(out.download(x.size), ora.softcap(x, cap))
    rt.free(buf)
    rt.free(out)


# a wavefront meets the IEEE division through any of its values: exact zeros,
# a mask's -inf or lowest float, infinities, NaN and subnormals beside ordinary
# logits, in rows of one value a thread, of one and of four float4 a thread
SPECIAL = np.array([0.0, -0.0, -np.inf, np.inf, np.finfo(f32).min, np.finfo(f32).max, np.nan, 1e-45, -1e-40, 2.0 ** -71],
                   f32)


@pytest.mark.parametrize("rows,count", [(5, 3), (3, 259), (64, 4096), (1024, 4096), (1031, 4099)])
@pytest.mark.parametrize("std", [1.0, 8.0])
def test_special_values(rt, ora, rows, count, std):
    r = np.random.default_rng(rows + count)
    x = (r.standard_normal((rows, count)) * std).astype(f32)
    for i in range(rows):
        if i % 3 == 1:  # one special value in the row
            x[i, r.integers(count)] = SPECIAL[(i // 3) % len(SPECIAL)]
        elif i % 3 == 2:  # a masked row
            x[i, r.random(count) < 0.5] = SPECIAL[2 + (i // 3) % 3]
    x = x.reshape(-1)
    exp_c, exp_s = ora.softcap_argmax_rows(x, rows, count, 30.0)
    src, dst, sel = rt.upload(x), rt.empty(x.size), rt.empty(rows, np.uint32)
    rt.softcap_argmax(src, dst, sel, rows, count, 30.0)
    rt.sync()
    assert _same(dst.download(x.size), exp_c)
    assert np.array_equal(sel.download(rows, np.uint32), exp_s)
    rt.softcap(src, src, x.size, 30.0)
    rt.sync()
    assert _same(src.download(x.size), exp_c)
    for b in (src, dst, sel):
        rt.free(b)


# a signalling NaN is a value like any other NaN: what its lane holds before it
# still counts, for the argmax and for the choice of the soft cap's steps (one
# float4 a lane, and four, 1024 values apart)
@pytest.mark.parametrize("rows,count,apart", [(2, 3000, (1, 2, 3)), (1100, 4096, (1, 3, 1024, 2049, 3074))])
@pytest.mark.parametrize("first", [25.0, 1e30, np.inf, 1e-45])
def test_signalling_nan(rt, ora, rows, count, apart, first):
    r = np.random.default_rng(count)
    x = r.standard_normal((rows, count)).astype(f32)
    for i in range(rows):
        at = 4 * (i % 250)
        x[i, at] = first
        x[i].view(np.uint32)[at + apart[i % len(apart)]] = 0x7F800001 if i % 2 else 0xFFBFFFFF
    x = x.reshape(-1)
    exp_c, exp_s = ora.softcap_argmax_rows(x, rows, count, 30.0)
    src, dst, sel = rt.upload(x), rt.empty(x.size), rt.empty(rows, np.uint32)
    rt.softcap_argmax(src, dst, sel, rows, count, 30.0)
    rt.sync()
    assert _same(dst.download(x.size), exp_c)
    assert np.array_equal(sel.download(rows, np.uint32), exp_s)
    rt.argmax(src, sel, rows, count)
    rt.sync()
    assert np.array_equal(sel.download(rows, np.uint32), ora.softcap_argmax_rows(x, rows, count, 0.0)[1])
    for b in (src, dst, sel):
        rt.free(b)


def test_in_range_division_is_ieee_on_the_exponential_range():
    # every float from 0.625 to infinity, as test_gpu_division does for the activations
    counts = (ctypes.c_uint64 * 4)()
    assert division_lib().atlas_division_check(3, counts) == 0
    inputs, bad, bad_product, _ = (int(c) for c in counts)
    assert inputs == 0x7F800000 - int(np.array([0.625], f32).view(np.uint32)[0]) + 1
    assert bad == 0, f"{bad} inputs differ from the IEEE division"
    assert bad_product > 1000, bad_product  # planted: no correction step
