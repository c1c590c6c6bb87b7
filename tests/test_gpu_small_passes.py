"""Prompt passes and batches of a few tokens against the oracle: 2 to 16 tokens share one matrix-core
token tile (17: two tiles, the second with one token), and rows that are not whole groups of 4
blocks (hidden 192: 6 blocks) take the vector-ALU kernel instead.  Tokens equal, logits bit for bit.
"""
import numpy as np
import pytest

import oracle
import synth

pytestmark = pytest.mark.gpu

SHAPES = {"small": synth.SHAPES["small"], "small128": synth.SHAPES["small128"],
          "hidden192": synth.Shape(192, 2, 320, 3, 1, 512)}


def _same(lg, lo, what):
    bad = np.flatnonzero(np.ascontiguousarray(lg, np.float32).view(np.uint32) != np.ascontiguousarray(lo, np.float32).view(np.uint32))
    assert bad.size == 0, f"{what}: {bad.size} logits differ, first {bad[:5]}"


@pytest.mark.parametrize("head", [synth.GGML_Q4_0, synth.GGML_Q8_0])
@pytest.mark.parametrize("name", list(SHAPES))
def test_passes_and_batches_of_a_few_tokens(name, head):
    import q4hip
    shape = SHAPES[name]
    t = synth.make_model(shape, 91, head_type=head)
    g = q4hip.Model(shape, ctx=96)
    g.load(t)
    o = oracle.Model(shape, t, ctx=96, mt=16, threads=8)
    try:
        for n in (2, 3, 7, 8, 9, 16, 17):
            print(f"{name} pass of {n}", flush=True)
            ids = synth.prompt_ids(90 + n, n, shape.vocab)
            assert g.forward(ids, 0) == o.forward(ids, 0), f"pass of {n}"
            _same(g.read_logits(), o.logits(), f"pass of {n}")
        for B in (2, 5, 8, 9, 17):
            print(f"{name} batch of {B}", flush=True)
            lens = [1 + (7 * b) % 11 for b in range(B)]
            ps = [synth.prompt_ids(60 + b, n, shape.vocab) for b, n in enumerate(lens)]
            bt = q4hip.Batch(g, B)
            try:
                first = [bt.prefill(b, ps[b], 0) for b in range(B)]
                out = bt.generate(first, lens, 2)
                lg = bt.read_logits()
            finally:
                bt.close()
            for b in range(B):
                want = [o.forward(ps[b], 0)]
                for i in range(2):
                    want.append(o.forward([want[-1]], lens[b] + i))
                assert first[b] == want[0] and out[:, b].tolist() == want[1:], f"batch of {B}, sequence {b}"
                _same(lg[b], o.logits(), f"batch of {B}, sequence {b}")
    finally:
        g.close()
        o.close()


@pytest.mark.parametrize("shape", [synth.Shape(128, 1, 256, 2, 1, 192), synth.Shape(192, 1, 256, 3, 1, 1090),
                                   synth.Shape(2112, 1, 2112, 33, 11, 192)], ids=["vocab192", "vocab1090", "hidden2112"])
def test_q8_head_of_batches(shape):
    """The Q8_0 head for several tokens: an odd number of 64-row tiles (192), rows that end inside one
    (1,090), rows wider than it takes (2,112 values: a launch per sequence), and batches at the edges of the 4,
    8 and 16 tokens of a workgroup."""
    import q4hip
    t = synth.make_model(shape, 93, head_type=synth.GGML_Q8_0)
    g = q4hip.Model(shape, ctx=48)
    g.load(t)
    o = oracle.Model(shape, t, ctx=48, mt=16, threads=8)
    try:
        for B in (1, 2, 4, 5, 8, 9, 16, 17, 33):
            print(f"vocab {shape.vocab} hidden {shape.dim} batch of {B}", flush=True)
            lens = [1 + (5 * b) % 7 for b in range(B)]
            ps = [synth.prompt_ids(20 + b, n, shape.vocab) for b, n in enumerate(lens)]
            bt = q4hip.Batch(g, B)
            try:
                first = [bt.prefill(b, ps[b], 0) for b in range(B)]
                out = bt.generate(first, lens, 1)
                lg = bt.read_logits()
            finally:
                bt.close()
            for b in range(B):
                want = o.forward(ps[b], 0)
                assert first[b] == want, f"batch of {B}, sequence {b}"
                assert out[0, b] == o.forward([want], lens[b]), f"batch of {B}, sequence {b}"
                _same(lg[b], o.logits(), f"batch of {B}, sequence {b}")
    finally:
        g.close()
        o.close()
