"""The sums in order on the device (q4hip_check_ordered_sum): the wave's and one lane's against plain float32
additions, bit for bit, over lengths at the edges of the wave's runs and of its minimum, on softmax
values and on values made to fail its assumptions: ties at every addition, sums that sit on a power of two or
cross many, denormals, zeros, one large value among small ones, infinities.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

F = np.float32
WAVE_MIN = 1280                        # kOrderedWaveMin of csrc/kernels.h
LENGTHS = [1, 3, 31, 32, 33, 95, 224, 1279, 1280, 1281, 1283, 1299, 1300, 1301, 1535, 1536, 1537, 1792, 1793, 2049, 2560,
           4095, 4097, 6143, 8192, 8193, 15360]


def _rows(n):
    """(kind, values) of rows of n values; kinds 'softmax' combine on the device, 'not finite' cannot."""
    r = np.random.default_rng(n)
    at = r.integers(0, n, 8)
    for spread in (0.3, 1, 2, 4):
        for _ in range(12):
            yield "softmax", np.exp(r.normal(0, spread, n) - spread)
    for _ in range(8):
        yield "uniform", r.random(n)
        yield "short mantissas", r.integers(0, 64, n) / 64
        yield "shorter", r.integers(0, 4, n) / 4
    yield "ones", np.ones(n)
    yield "zeros", np.zeros(n)
    for p in (20, 23, 24, 25):
        yield "ties", np.concatenate([[2.0 ** p], np.ones(n - 1)])
        yield "half ties", np.concatenate([[2.0 ** p], np.full(n - 1, 0.5)])
        yield "just below a power of two", np.concatenate([[2.0 ** p - 2.0], r.integers(0, 2, n - 1)])
        yield "on a power of two, tiny terms", np.concatenate([[2.0 ** p], r.random(n - 1) * 2.0 ** (p - 26)])
    yield "powers of two", 2.0 ** r.integers(-30, 6, n)
    yield "growing", 1.01 ** np.minimum(np.arange(n), 8000)
    yield "growing fast", 2.0 ** (np.arange(n) % 200 - 100)
    yield "denormals", (r.integers(0, 1 << 20, n).astype(np.int32)).view(F)
    yield "denormals, then values", np.concatenate([(r.integers(0, 1 << 10, n // 2).astype(np.int32)).view(F), r.random(n - n // 2)])
    yield "late start", np.concatenate([np.zeros(n - n // 3), r.random(n // 3)])
    yield "sparse", np.where(r.random(n) < 0.01, r.random(n), 0)
    for i in at:
        yield "one large", np.where(np.arange(n) == i, 3e8, r.random(n))
        yield "one at a power of two", np.where(np.arange(n) == i, 2.0 ** 12, r.random(n))
        yield "not finite", np.where(np.arange(n) == i, np.inf, 1.0)
    yield "not finite", np.full(n, 3e38)


@pytest.mark.parametrize("n", LENGTHS)
def test_sums_in_order(n):
    import q4hip
    print(f"{n} values", flush=True)
    with np.errstate(over="ignore"):
        kinds, v = zip(*[(k, np.asarray(x, F)) for k, x in _rows(n)])
        v = np.stack(v)
        want = np.add.accumulate(v, axis=1, dtype=F)[:, -1]       # one float32 addition per value, in order
    wave, lane, combined = q4hip.check_ordered_sum(v)
    for name, got in (("wave", wave), ("lane", lane)):
        bad = np.flatnonzero(got.view(np.uint32) != want.view(np.uint32))
        assert bad.size == 0, f"{name}: {[(kinds[b], float(got[b]), float(want[b])) for b in bad[:5]]}"
    if n < WAVE_MIN:
        assert not combined.any()
    else:
        soft = np.array([k == "softmax" for k in kinds])
        assert combined[soft].mean() > 0.9, "the combined form is the one that runs"
        assert not combined[[not np.isfinite(w) for w in want]].any()
