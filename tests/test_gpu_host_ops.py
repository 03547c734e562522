"""The host-slice operators over the context's buffers: operands from one value
to past what the context keeps, in changing order, against the formulas of
the operators on the CPU; telemetry and refusals as with a buffer per operand."""
import threading

import numpy as np
import pytest
from atlas_amd import NeuralOps, OperatorError

pytestmark = pytest.mark.gpu

KEPT = 16 << 20  # bytes a context keeps; an add's three operands fill it at n = KEPT / 12


@pytest.fixture(scope="module")
def ops():
    return NeuralOps()


# one value, odd ends, the copy kernel's last size and the next, growth, the
# last that is served from the kept buffers and the first that is not, and back
SIZES = [1, 3, 63, 65, 4097, (1 << 18) - 64, 1 << 18, (1 << 18) + 1, 1 << 19, KEPT // 12 - 64, KEPT // 12, KEPT // 12 + 64,
         (KEPT >> 2) + 1, 5, 1000]


@pytest.mark.parametrize("order", [1, -1])
def test_sizes_in_any_order(ops, order):
    rng = np.random.default_rng(7)
    for n in SIZES[::order]:
        a, b = rng.standard_normal(n, dtype=np.float32), rng.standard_normal(n, dtype=np.float32)
        got, t = ops.add(a, b)
        assert np.array_equal(got.view(np.uint32), (a + b).view(np.uint32)), n
        assert 0.0 <= t.gpu_ms <= t.wall_ms
        got, _ = ops.multiply(a, b)
        assert np.array_equal(got.view(np.uint32), (a * b).view(np.uint32)), n
        got, _ = ops.scalar_multiply(a, 0.3)
        assert np.array_equal(got.view(np.uint32), (a * np.float32(0.3)).view(np.uint32)), n


def test_operands_of_different_sizes(ops):
    rng = np.random.default_rng(8)
    for rows, hidden in [(1, 2), (3, 258), (128, 576), (1, 8192), (700, 1536)]:
        x = rng.standard_normal((rows, hidden), dtype=np.float32)
        angle = rng.standard_normal(hidden // 2).astype(np.float32)
        c, s = np.cos(angle), np.sin(angle)
        got, _ = ops.rope(x.reshape(-1), rows, hidden, c, s)
        exp = np.stack([x[:, 0::2] * c - x[:, 1::2] * s, x[:, 0::2] * s + x[:, 1::2] * c], 2).reshape(-1)
        # two rounded products and a rounded sum, each side: 2 ulps of the larger product
        assert np.max(np.abs(got - exp)) <= 4 * np.finfo(np.float32).eps * np.abs(x).max()
        table = rng.standard_normal((11, hidden), dtype=np.float32)
        ids = rng.integers(0, 11, rows).astype(np.uint32)
        got, _ = ops.embedding(table.reshape(-1), 11, hidden, ids)
        assert np.array_equal(got.view(np.uint32), table[ids].reshape(-1).view(np.uint32))


def test_telemetry_and_refusals():
    ops = NeuralOps()
    x = np.ones(1000, np.float32)
    before = ops.rt.telemetry()
    ops.add(x, x)
    after = ops.rt.telemetry()
    assert after.allocations - before.allocations == 3
    assert after.upload_bytes - before.upload_bytes == 8000
    assert after.readback_bytes - before.readback_bytes == 4000
    assert after.dispatches - before.dispatches == 1 and after.syncs - before.syncs == 1
    assert after.resident_bytes == before.resident_bytes
    assert after.peak_resident_bytes >= before.resident_bytes + 12000
    with pytest.raises(OperatorError):
        ops.add(x, x[:-1])
    ops.rt.graph_begin()
    try:
        with pytest.raises(OperatorError):
            ops.add(x, x)
    finally:
        ops.rt.graph_destroy(ops.rt.graph_end())
    assert np.array_equal(ops.add(x, x)[0], x + x)


def test_threads_on_one_context():
    """Threads that share a context take turns, in the kept buffers and past
    them: each call gets its own result, and the telemetry of all of them adds up."""
    ops = NeuralOps()
    rng = np.random.default_rng(9)
    inputs = [rng.standard_normal(n, dtype=np.float32) for n in (1000, 70001, 300000, 64, KEPT // 4, 2)]
    before = ops.rt.telemetry()
    wrong = []

    def work(x):
        for _ in range(20):
            got = ops.add(x, x)[0]
            if not np.array_equal(got, x + x):
                wrong.append(x.size)

    threads = [threading.Thread(target=work, args=(x,)) for x in inputs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert wrong == []
    after = ops.rt.telemetry()
    calls, values = 20 * len(inputs), 20 * sum(x.size for x in inputs)
    assert after.allocations - before.allocations == 3 * calls
    assert after.dispatches - before.dispatches == calls
    assert after.upload_bytes - before.upload_bytes == 8 * values
    assert after.readback_bytes - before.readback_bytes == 4 * values
    assert after.resident_bytes == before.resident_bytes
    # one call at a time: the largest one's operands, not several calls'
    assert after.peak_resident_bytes == before.resident_bytes + 3 * KEPT
