"""The parameters a prepared model holds on the device (norms, RoPE tables) follow the caller's
buffers: each device loop prepares again, and a changed value of any array takes effect, as does
changing it back; K/V formed with an old value is not reused; a missing array is refused."""
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


def test_prefix_of_changed_parameters_is_not_reused(backend):
    """K/V formed with a norm, RoPE table or weight that has changed since, in place or behind the same
    handle, is not reused: reuse_prefix gives what a fresh context gives. What the sequence's K/V does
    not depend on leaves it alone, and an unchanged model reuses it."""
    model = synth.make_model(SHAPE, mode="stq", seed=235)
    prompt = synth.rand_prompt(synth.rng(236), 20, SHAPE.vocab)

    def run(fm, reuse):
        ids, st = fm.generate_ids(prompt, 4, chunk=8, reuse_prefix=reuse)
        return fm.forward([int(ids[-1])], 23), st.cached_tokens

    def fresh():
        b = lib.Backend()
        try:
            fm = lib.FusedModel(b, model)
            want, _ = run(fm, False)
            fm.close()
            return want
        finally:
            b.close()

    fm = lib.FusedModel(backend, model)
    try:
        fm.generate_ids(prompt, 4, chunk=8)
        got, cached = run(fm, True)
        assert cached == 19 and np.array_equal(got, fresh())
        L = model["layers"]
        for a in (L[0]["attn_norm"], L[0]["ffn_norm"], L[1]["k_norm"], model["rope_cos"], model["rope_sin"]):
            fm.generate_ids(prompt, 4, chunk=8)
            a[(3, 5) if a.ndim == 2 else 7] += np.float32(0.5)
            got, cached = run(fm, True)
            assert cached == 0 and np.array_equal(got, fresh())
        # a weight released and another uploaded, usually at the same address
        L[0]["wk"] = synth.make_weight(synth.rng(237), L[0]["wk"].type, SHAPE.kvdim, SHAPE.hidden)
        fm.generate_ids(prompt, 4, chunk=8)
        at = fm.handles.index(fm.layers[0].wk)
        backend.release(fm.handles[at])
        fm.handles[at] = backend.upload(L[0]["wk"])
        fm.layers[0].wk = fm.handles[at]
        got, cached = run(fm, True)
        assert cached == 0 and np.array_equal(got, fresh())
        # a weight of no model
        fm.generate_ids(prompt, 4, chunk=8)
        backend.release(backend.upload(L[0]["wk"]))
        assert run(fm, True)[1] == 19
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
