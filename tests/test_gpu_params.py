"""The parameters a prepared model holds on the device (norms, RoPE tables) follow the caller's
buffers: each device loop prepares again, and a changed value of any array takes effect, as does
changing it back; a missing array is refused."""
import numpy as np
import pytest

from hymt2_amd import lib, synth

pytestmark = pytest.mark.gpu

SHAPE = synth.ModelShape(n_layer=2, hidden=512, ffn=512, heads=4, kv_heads=2, hdim=128, vocab=400, ctx=40)


def test_changed_parameters_take_effect(backend):
    model = synth.make_model(SHAPE, mode="stq", seed=231)
    prompt = synth.rand_prompt(synth.rng(232), 20, SHAPE.vocab)
    fm = lib.FusedModel(backend, model)
    try:
        def logits():
            ids, _ = fm.generate_ids(prompt, 4, chunk=8)
            return fm.forward([int(ids[-1])], 23)

        first = logits()
        L = model["layers"]
        for a in (L[0]["attn_norm"], L[1]["ffn_norm"], L[1]["q_norm"], L[0]["k_norm"], model["out_norm"],
                  model["rope_cos"], model["rope_sin"]):
            at = (3, 5) if a.ndim == 2 else 7
            kept = a[at]
            a[at] = kept + np.float32(0.5)
            changed = logits()
            assert not np.array_equal(changed, first)
            fresh = lib.Backend()
            try:  # a context that never held the old value
                other = lib.FusedModel(fresh, model)
                ids, _ = other.generate_ids(prompt, 4, chunk=8)
                assert np.array_equal(other.forward([int(ids[-1])], 23), changed)
                other.close()
            finally:
                fresh.close()
            a[at] = kept
            assert np.array_equal(logits(), first)
    finally:
        fm.close()


def test_missing_parameter_is_refused():
    b = lib.Backend()
    model = synth.make_model(SHAPE, mode="stq", seed=233)
    fm = lib.FusedModel(b, model)
    try:
        fm.layers[1].k_norm = None
        with pytest.raises(RuntimeError):
            fm.generate_ids(synth.rand_prompt(synth.rng(234), 8, SHAPE.vocab), 2)
    finally:
        fm.close()
        b.close()
