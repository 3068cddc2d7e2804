"""The chunk attention of short rows (k_attn_chunk_short) against the oracle, bit for bit: chunks that
end at, before and after its V tiles (64 positions), its score passes (64 or 128 keys) and its longest
rows (128 to 512 positions), after which the general chunk kernel takes over; both head dims it takes
and both group sizes. The second layer's keys and values carry the first layer's attention at every
position into the logits compared after each chunk."""
import numpy as np
import pytest

from hymt2_amd import lib, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu

ENDS = (2, 17, 63, 64, 65, 80, 127, 128, 129, 144, 191, 193, 255, 256, 257, 300)


def bits(a):
    return np.ascontiguousarray(a, dtype=np.float32).view(np.uint32)


@pytest.mark.parametrize("hdim,grp", [(128, 4), (128, 2), (64, 4), (64, 2)])
def test_short_chunk_attention(backend, hdim, grp):
    heads = 512 // hdim
    shape = synth.ModelShape(n_layer=2, hidden=512, ffn=512, heads=heads, kv_heads=heads // grp, hdim=hdim, vocab=300, ctx=320)
    model = synth.make_model(shape, mode="stq", seed=211 + hdim + grp)
    prompt = synth.rand_prompt(synth.rng(212), ENDS[-1], shape.vocab)
    om = O.OracleModel(model, threads=8)
    fm = lib.FusedModel(backend, model)
    try:
        at = 0
        for end in ENDS:
            got = fm.forward([int(t) for t in prompt[at:end]], at, True)
            for i in range(at, end, 16):
                want = om.forward(prompt[i:min(i + 16, end)], i, want_logits=i + 16 >= end)
            assert np.array_equal(bits(got), bits(want)), f"positions {at}..{end - 1}"
            at = end
    finally:
        fm.close()
