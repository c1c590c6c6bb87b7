"""The one-(row, head)-per-workgroup attention against the oracle: contexts at the edges of its 64-position
K chunks and of the 64- and 128-position chunks of P.V, in a batch of sequences, a short pass at a
position, and one-token steps past the length from which the softmax sum is formed by the whole wave.
Tokens equal, logits bit for bit.  Its time follows the positions in use, not the size of the context.
"""
import numpy as np
import pytest

import oracle
import synth

pytestmark = pytest.mark.gpu


def _same(lg, lo, what):
    bad = np.flatnonzero(np.ascontiguousarray(lg, np.float32).view(np.uint32) != np.ascontiguousarray(lo, np.float32).view(np.uint32))
    assert bad.size == 0, f"{what}: {bad.size} logits differ, first {bad[:5]}"


def _pair(name, kv, ctx):
    import q4hip
    shape = synth.SHAPES[name]
    t = synth.make_model(shape, 95)
    g = q4hip.Model(shape, ctx=ctx, kv_type=q4hip.KV_F16 if kv == "f16" else q4hip.KV_F32)
    g.load(t)
    g.set_decode_mode(q4hip.DECODE_GRAPH)
    o = oracle.Model(shape, t, ctx=ctx, mt=16, threads=8)
    if kv == "f16":
        o.set_variant(oracle.V_KV_F16)
    return shape, g, o


@pytest.mark.parametrize("kv", ["f32", "f16"])
@pytest.mark.parametrize("name", ["small", "small128"])
def test_chunk_edges(name, kv):
    import q4hip
    shape, g, o = _pair(name, kv, 320)
    lens = [1, 2, 61, 62, 63, 64, 125, 126, 127, 128, 189, 190, 191, 253, 255, 256]
    ps = [synth.prompt_ids(300 + n, n, shape.vocab) for n in lens]
    bt = q4hip.Batch(g, len(lens))
    try:
        print(f"{name} {kv} batch", flush=True)
        first = [bt.prefill(b, ps[b], 0) for b in range(len(lens))]
        out = bt.generate(first, lens, 3)          # contexts of each length + 1 .. + 3
        lg = bt.read_logits()
        for b, n in enumerate(lens):
            want = [o.forward(ps[b], 0)]
            for i in range(3):
                want.append(o.forward([want[-1]], n + i))
            assert first[b] == want[0] and out[:, b].tolist() == want[1:], f"sequence of {n}"
            _same(lg[b], o.logits(), f"sequence of {n}")
        ids = synth.prompt_ids(7, 210, shape.vocab)
        for pos, n in ((0, 2), (2, 62), (64, 5), (69, 61), (130, 80)):
            print(f"{name} {kv} pass of {n} at {pos}", flush=True)
            assert g.forward(ids[pos:pos + n], pos) == o.forward(ids[pos:pos + n], pos), f"pass of {n} at {pos}"
            _same(g.read_logits(), o.logits(), f"pass of {n} at {pos}")
    finally:
        bt.close()
        g.close()
        o.close()


@pytest.mark.parametrize("name,kv", [("small", "f32"), ("small128", "f16")])
def test_sum_by_the_wave(name, kv):
    shape, g, o = _pair(name, kv, 1400)
    try:
        ids = synth.prompt_ids(8, 1276, shape.vocab)
        ng, no = g.forward(ids, 0), o.forward(ids, 0)
        assert ng == no
        for i in range(12):                          # 1277 .. 1288 positions
            print(f"{name} {kv} step {i}", flush=True)
            ng, no = g.forward([ng], 1276 + i), o.forward([no], 1276 + i)
            assert ng == no, f"step {i}"
            _same(g.read_logits(), o.logits(), f"step {i}")
    finally:
        g.close()
        o.close()


def test_steps_across_the_limit_of_fp32_rows():
    """Two heads of 128 fp32 columns in one group: a token, and a batch of a few sequences by its
    longest, takes this kernel up to 512 positions and the list kernels from there (the token in two
    captured steps)."""
    import q4hip
    shape, g, o = _pair("small128", "f32", 1000)
    try:
        ids = synth.prompt_ids(9, 506, shape.vocab)
        want = [o.forward(ids, 0)]
        for i in range(14):
            want.append(o.forward([want[-1]], 506 + i))
        last = o.logits().copy()
        assert g.forward(ids, 0) == want[0]
        for run in range(3):                         # the second and third run replay both graphs
            print(f"generate, run {run}", flush=True)
            assert g.generate(want[0], 506, 14) == want[1:]
            _same(g.read_logits(), last, f"run {run}")
        for i in range(14):
            assert g.forward([want[i]], 506 + i) == want[i + 1], f"token {i}"
        _same(g.read_logits(), last, "token by token")
        lens = [505, 500, 511]                       # 512 (2 steps), then 526, in the middle
        bt = q4hip.Batch(g, 3)
        try:
            ps = [synth.prompt_ids(40 + n, n, shape.vocab) for n in lens]
            first = [bt.prefill(b, ps[b], 0) for b in range(3)]
            a = bt.generate(first, lens, 2)
            c = bt.generate(a[-1], [n + 2 for n in lens], 25)
            lg = bt.read_logits()
        finally:
            bt.close()
        for b, n in enumerate(lens):
            w = [o.forward(ps[b], 0)]
            for i in range(27):
                w.append(o.forward([w[-1]], n + i))
            assert [first[b]] + a[:, b].tolist() + c[:, b].tolist() == w, f"sequence of {n}"
            _same(lg[b], o.logits(), f"sequence of {n}")
    finally:
        g.close()
        o.close()


def test_time_follows_the_positions_not_the_context():
    """36 rows of 14 heads are 504 workgroups: two fit a CU with the shared memory of 36 positions, one with
    that of a 4,400-position context (attention 1.5 times as long).  Best of 9 in turn; 1.25 is half way."""
    import q4hip
    shape = synth.Shape(896, 8, 256, 14, 2, 512)
    t = synth.make_model(shape, 96)
    ids = synth.prompt_ids(5, 36, shape.vocab)
    models = [q4hip.Model(shape, ctx=ctx) for ctx in (512, 4400)]
    best = [1e9, 1e9]
    try:
        for m in models:
            m.load(t)
        for _ in range(9):
            for i, m in enumerate(models):
                best[i] = min(best[i], m.profile_pass(ids, 0)["attention"])
    finally:
        for m in models:
            m.close()
    print(f"attention of 8 layers: {best[0]:.1f} us in 512 positions, {best[1]:.1f} in 4,400", flush=True)
    assert best[1] < 1.25 * best[0]
