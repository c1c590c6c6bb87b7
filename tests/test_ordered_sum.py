"""The wave's sum in order (ordered_sum_wave of csrc/kernels.h), restated in numpy float32 and compared bit
for bit with the plain loop of additions: values near ties, exact powers of two, zeros, denormals, sums
that sit on a power of two, one large value among small ones, infinities.  The kernel itself runs the same kinds of
values in tests/test_gpu_ordered_sum.py.
"""
import numpy as np
import pytest

F = np.float32


def _bits(x):
    return int(np.asarray(x, F).view(np.int32))


def _float(b):
    return np.asarray(b, np.int32).view(F)[()]


def in_order(v, s=F(0)):
    for x in v:
        s = F(s + x)
    return s


def wave_sum(v):
    """(sum, whether the runs were combined) as ordered_sum_wave forms it."""
    T = len(v)
    R = 4 * (((T + 255) >> 8) | 1)
    n = (T + R - 1) // R
    assert n <= 64
    e = np.concatenate([v, np.zeros(R, F)]).astype(F)
    est = [F(sum((F(F(e[l * R + k] + e[l * R + k + 1]) + F(e[l * R + k + 2] + e[l * R + k + 3]))
                  for k in range(0, R, 4)), F(0))) for l in range(n)]
    after = np.cumsum(np.array(est, F), dtype=F)
    f0, f1, E, serial = [], [], [], []
    for l in range(n):
        before = after[l - 1] if l else F(0)
        b0 = _bits(before) & ~1
        c0, c1 = _float(b0), _float(b0 | 1)
        run = e[l * R:(l + 1) * R]
        c0, c1 = in_order(run, c0), in_order(run, c1)
        ex = _bits(before) >> 23
        E.append(ex)
        serial.append(l == 0 or ex <= 0 or any((_bits(x) >> 23) != ex for x in
                                              (F(before * F(1 - 2.0**-16)), F(after[l] * F(1 + 2.0**-16)), c0, c1)))
        f0.append(_bits(c0) - b0)
        f1.append(_bits(c1) - (b0 | 1))
    if not np.isfinite(after[-1]):
        return in_order(v), False
    S, l = 0, 0
    while l < n:
        if serial[l]:
            S = _bits(in_order(e[l * R:(l + 1) * R], _float(S)))
            l += 1
            continue
        g0 = g1 = 0                       # the segment's combined increments, as the scan forms them
        s = l
        while s < n and not serial[s]:
            g0, g1 = g0 + (f1[s] if g0 & 1 else f0[s]), g1 + (f0[s] if g1 & 1 else f1[s])
            s += 1
        if (S >> 23) != E[s - 1]:
            return in_order(v), False
        S += g1 if S & 1 else g0
        if (S >> 23) != E[s - 1]:
            return in_order(v), False
        l = s
    return _float(S), True


def _cases():
    r = np.random.default_rng(5)
    for T in (1, 3, 4, 5, 63, 64, 255, 256, 257, 300, 701, 1026, 2049, 4097):
        yield f"softmax {T}", np.exp(r.normal(0, 2, T) - 6).astype(F)
        yield f"uniform {T}", r.random(T).astype(F)
        yield f"short mantissas {T}", (r.integers(0, 64, T) / 64).astype(F)       # ties at every step
        yield f"ones {T}", np.ones(T, F)
        yield f"tie at each addition {T}", np.concatenate([[F(2.0**24)], np.ones(T - 1, F)]).astype(F)
    yield "zeros", np.zeros(500, F)
    yield "denormals", (r.integers(0, 1 << 20, 900).astype(np.int32)).view(F)
    yield "late start", np.concatenate([np.zeros(600, F), r.random(500).astype(F)])
    yield "one large", np.where(np.arange(1000) == 777, F(3e8), r.random(1000).astype(F)).astype(F)
    yield "squares of a row", (r.normal(0, 1, 224).astype(F) ** 2).astype(F)
    yield "infinite", np.where(np.arange(400) == 99, F(np.inf), F(1)).astype(F)
    yield "overflow", np.full(400, F(3e38))


@pytest.mark.parametrize("name,v", list(_cases()), ids=[c[0] for c in _cases()])
def test_runs_combine_to_the_sum_in_order(name, v):
    with np.errstate(over="ignore"):
        got, combined = wave_sum(v)
        want = in_order(v)
    assert _bits(got) == _bits(want), (name, got, want)


def test_runs_do_combine():
    """The fast form is the one that runs: random sums of the softmax's kind hardly ever fall back."""
    r = np.random.default_rng(6)
    done = [wave_sum(np.exp(r.normal(0, 1, 1026)).astype(F))[1] for _ in range(20)]
    assert sum(done) >= 19
