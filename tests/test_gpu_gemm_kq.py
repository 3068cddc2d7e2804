"""The Q4_K / Q6_K GEMM (k_gemm_kq) against the oracle, bit for bit.

Cases sit at the edges of its tiles and splits: token counts around 16-token tiles, the counts
where the split changes and those up to 16 where few or long rows stay on the general matvec, row counts that end inside a 16-row tile, K from one block to past the
largest that is split over wavefronts (33 blocks), and extreme block contents (every scale, min,
code and activation at its largest magnitude, of either sign, where the int8 digits of the scaled
weights and the f16 products of mins and bsums reach their bounds). The sizes at which each form of
the launch is chosen follow kq_shape's rules; SPLITS names the form each of its cases takes."""
import numpy as np
import pytest

from conftest import ROOT  # noqa: F401  (sys.path)
from hymt2_amd import abi, lib, synth
from oracle import oracle as O
from test_gpu_fallbacks import check_model
from test_gpu_kernels import bits, run_matvec

pytestmark = pytest.mark.gpu

BLOCK = {abi.GT_Q4_K: 144, abi.GT_Q6_K: 210}


def raw_weight(g, gt, n, k, extreme):
    """Random block bytes (every code, scale and min value occurs); `extreme`: rows of constant
    largest-magnitude fields. The f16 scales stay finite and of ordinary size."""
    b = g.integers(0, 256, size=(n, k // 256, BLOCK[gt]), dtype=np.uint8)
    if extreme:
        b[0::3] = 0xFF               # Q4_K: q 15, sc 63, mn 63; Q6_K: q 31, sc -1
        b[1::3] = 0x00               # Q6_K: q -32
        if gt == abi.GT_Q6_K:
            b[0::2, :, 192:208] = 0x80  # sc -128
            b[1::2, :, 192:208] = 0x7F  # sc 127
    d = synth.f16_bits(g.uniform(0.001, 0.02, size=(n, k // 256, 2))).view(np.uint8).reshape(n, k // 256, 4)
    if gt == abi.GT_Q4_K:
        b[:, :, 0:4] = d
    else:
        b[:, :, 208:210] = d[:, :, :2]
    return synth.Weight(gt, k, n, b.reshape(n, -1))


@pytest.mark.parametrize("gt", [abi.GT_Q4_K, abi.GT_Q6_K])
@pytest.mark.parametrize("n,k", [(1, 256), (17, 512), (100, 2048), (63, 2304), (64, 3072), (65, 4096), (33, 4352),
                                 (48, 6144), (31, 8192), (40, 8448), (4100, 512), (2200, 256)])
def test_gemm_kq_vs_oracle(backend, gt, n, k):
    g = synth.rng(gt * 13 + n + k)
    for nt in (4, 5, 8, 16, 17, 48, 49, 80, 81, 128):
        extreme = nt in (16, 49, 128)
        w = raw_weight(g, gt, n, k, extreme)
        x = synth.activations(g, nt, k)
        if extreme:
            x[0::2] = np.sign(x[0::2])  # every code 127 or -127
            x[1::4] = 1.0               # and bsums at their largest
        out, xq = run_matvec(backend, w, x)
        assert np.array_equal(bits(out), bits(O.matvec(w, x, xq, nt))), f"nt={nt}"


# 12 to 32 blocks alone: (rows, K, tokens) and the form: token tiles x row tiles a workgroup of each K set
SPLITS = [
    (2048, 3328, 33),   # 2 x 1, four blocks a set, the last set's short (13 of 16); 128 row tiles
    (2000, 5120, 47),   # 2 x 1, six blocks a set (20 of 24), ragged rows
    (2048, 6144, 48),   # 2 x 1, full sets (24 blocks)
    (2041, 6144, 64),   # 2 x 1, four token tiles
    (800, 7168, 81),    # 2 x 1, eight blocks a set (28 of 32), six token tiles
    (2560, 3072, 48),   # 2 x 2, three token tiles
    (2048, 3328, 65),   # 2 x 2, five token tiles
    (2017, 6144, 128),  # 2 x 2, an odd number of row tiles
    (4112, 3840, 17),   # 2 x 2, more row tiles than 256
    (4112, 3072, 33),   # 2 x 1, more workgroups of either form than 256
]


@pytest.mark.parametrize("gt", [abi.GT_Q4_K, abi.GT_Q6_K])
@pytest.mark.parametrize("n,k,nt", SPLITS)
def test_split_contractions(backend, gt, n, k, nt):
    g = synth.rng(gt * 17 + n + k + nt)
    w = raw_weight(g, gt, n, k, False)
    x = synth.activations(g, nt, k)
    out, xq = run_matvec(backend, w, x)
    assert np.array_equal(bits(out), bits(O.matvec(w, x, xq, nt)))


def test_gemm_kq_in_a_model(backend):
    """Mixed q/k (Q4_K) and v (Q6_K) rows in one launch, gate/up pairs with the SwiGLU epilogue and
    residual adds, at the 1.8B layer's dimensions and batches that take every split of each."""
    shape = synth.ModelShape(n_layer=1, hidden=2048, ffn=6144, heads=16, kv_heads=4, hdim=128, vocab=600, ctx=160)
    model = synth.make_model(shape, mode="q4km", seed=171)
    prompt = synth.rand_prompt(synth.rng(172), 150, shape.vocab)
    check_model(backend, model, prompt, 4, batches=(16, 48, 77, 128), chunks=(16, 128))


@pytest.mark.parametrize("mode,odd", [("q4km", None), ("q4km", "up"), ("stq", "v"), ("q2", "down")])
def test_pipelined_prefill_kinds(backend, mode, odd):
    """The pipelined chunked prefill of Q4_K_M weights (3, 9 and 19 chunks, a ragged last one), and
    models one of whose layers has a weight of another kind than its launch takes: `up` unlike its
    gate, `v` unlike q and k, `down` unlike the other layers' (these run one chunk after another).
    Greedy ids of the device loop, and the logits after them reading every layer's K/V."""
    shape = synth.ModelShape(n_layer=3, hidden=2048, ffn=1024, heads=16, kv_heads=4, hdim=128, vocab=500, ctx=320)
    model = synth.make_model(shape, mode=mode, seed=181)
    g = synth.rng(182)
    L = model["layers"][1]
    if odd == "up":
        L["wu"] = synth.make_weight(g, abi.GT_Q6_K, shape.ffn, shape.hidden)
    elif odd == "v":
        L["wv"] = synth.make_weight(g, abi.GT_Q6_K, shape.kvdim, shape.hidden)
    elif odd == "down":
        L["wd"] = synth.make_weight(g, abi.GT_Q4_K, shape.hidden, shape.ffn)
    prompt = synth.rand_prompt(synth.rng(183), 290, shape.vocab)
    want = O.OracleModel(model, threads=16).generate(prompt, 4, batch=16)
    om = O.OracleModel(model, threads=16)
    for i in range(0, len(prompt), 16):
        om.forward(prompt[i:i + 16], i, want_logits=False)
    ref = om.forward(want, len(prompt), want_logits=True)
    fm = lib.FusedModel(backend, model)
    try:
        for chunk in (33, 128, 16):
            ids, _ = fm.generate_device(prompt, 4, chunk=chunk)
            assert np.array_equal(ids, want), f"chunk={chunk}"
            assert np.array_equal(bits(fm.forward(list(ids), len(prompt), True)), bits(ref)), f"chunk={chunk}"
    finally:
        fm.close()
