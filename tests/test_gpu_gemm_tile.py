"""The 32 x 32 matrix-core tiles of large prompt passes against the oracle: token counts at the edges of the
16-, 32- and 64-token tiles, on shapes wide enough that the projections (hidden 2048: o and down at 256 and
from 385 tokens, with the RoPE epilogue at head_dim 64 and 128 from 449) or the fused gate|up projection (ffn
8192, from 113) take them; the other counts stay on k_gemm_sk.  Tokens equal,
logits bit for bit; a decode step after each pass reads the caches that the pass wrote.
"""
import numpy as np
import pytest

import oracle
import synth

pytestmark = pytest.mark.gpu

CASES = {  # shape (the oracle takes hidden up to ffn), token counts
    "hd64": (synth.Shape(2048, 1, 2048, 32, 4, 512), (256, 321, 336, 337, 353, 369, 384, 400, 417, 449,
                                                           450, 464, 465, 481, 497, 512)),
    "hd128": (synth.Shape(2048, 1, 2048, 16, 2, 512), (256, 330, 352, 384, 385, 449, 481, 500)),
    "gate_up": (synth.Shape(128, 1, 8192, 2, 1, 512), (97, 113, 127, 128, 161, 193, 208, 209, 225, 240, 256, 257)),
}


@pytest.mark.parametrize("kv", ["f32", "f16"])
@pytest.mark.parametrize("name", list(CASES))
def test_edges_of_the_tiles(name, kv):
    import q4hip
    shape, counts = CASES[name]
    t = synth.make_model(shape, 97)
    g = q4hip.Model(shape, ctx=520, kv_type=q4hip.KV_F16 if kv == "f16" else q4hip.KV_F32)
    g.load(t)
    o = oracle.Model(shape, t, ctx=520, mt=16, threads=8)
    if kv == "f16":
        o.set_variant(oracle.V_KV_F16)
    try:
        ids = synth.prompt_ids(98, max(counts), shape.vocab)
        for n in counts:
            print(f"{name} {kv} pass of {n}", flush=True)
            ng, no = g.forward(ids[:n], 0), o.forward(ids[:n], 0)
            assert ng == no, f"pass of {n}"
            for what in ("pass", "step after a pass"):
                a, b = g.read_logits(), o.logits()
                bad = np.flatnonzero(a.view(np.uint32) != np.ascontiguousarray(b, np.float32).view(np.uint32))
                assert bad.size == 0, f"{what} of {n}: {bad.size} logits differ"
                if what == "pass":
                    assert g.forward([ng], n) == o.forward([no], n)
    finally:
        g.close()
        o.close()
