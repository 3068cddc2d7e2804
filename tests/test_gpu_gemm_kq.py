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
from test_gpu_fallbacks import check_model, oracle_logits
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


# up to 11 blocks alone, more than 4096 rows and more than 80 tokens: K halves of four blocks up to
# eight, whole beyond
WIDE = [(4100, 2048, 81), (4100, 2048, 128), (4100, 1280, 81), (4096, 1024, 96), (4100, 2560, 81)]


@pytest.mark.parametrize("gt", [abi.GT_Q4_K, abi.GT_Q6_K])
@pytest.mark.parametrize("n,k,nt", WIDE)
def test_wide_contractions(backend, gt, n, k, nt):
    """The second K half full (eight blocks), short (five) and empty (four)."""
    g = synth.rng(gt * 19 + n + k + nt)
    w = raw_weight(g, gt, n, k, False)
    x = synth.activations(g, nt, k)
    out, xq = run_matvec(backend, w, x)
    assert np.array_equal(bits(out), bits(O.matvec(w, x, xq, nt)))


@pytest.mark.parametrize("rows,k,nt", [((512, 128, 128), 2048, 48), ((2048, 1024, 1100), 2048, 81), ((1000, 500, 520), 3328, 40),
                                       ((1024, 512, 520), 3328, 100), ((2304, 100, 33), 2304, 96), ((1500, 100, 33), 2304, 64)])
def test_mixed_groups(backend, rows, k, nt):
    """Q4_K and Q6_K jobs of one launch (a per-op group of two Q4_K weights and a Q6_K one) in each form
    of the launch: one token tile split, K halves, two token tiles split with one and with two row tiles,
    two token tiles and one with K whole. Row counts end inside tiles."""
    g = synth.rng(sum(rows) + k + nt)
    ws = [raw_weight(g, gt, n, k, False) for n, gt in zip(rows, (abi.GT_Q4_K, abi.GT_Q4_K, abi.GT_Q6_K))]
    hs = [backend.upload(w) for w in ws]
    try:
        x = synth.activations(g, nt, k)
        xq = O.quantize_q8k(x)
        for w, out in zip(ws, backend.matmul(hs, [w.n for w in ws], xq, nt)):
            assert np.array_equal(bits(out), bits(O.matvec(w, x, xq, nt)))
    finally:
        for h in hs:
            backend.release(h)


@pytest.mark.parametrize("gt,hidden,ffn", [(abi.GT_Q6_K, 2048, 1024), (abi.GT_Q4_K, 2048, 2304), (abi.GT_Q6_K, 2048, 2304),
                                           (abi.GT_Q6_K, 2048, 4352), (abi.GT_Q4_K, 2560, 2304), (abi.GT_Q6_K, 2560, 4352)])
def test_pairs_in_a_model(backend, gt, hidden, ffn):
    """Gate and up of either kind: split over wavefronts at 16 tokens (eight and ten blocks) and at 48
    (eight), K whole at 48 (ten) and, in 1, 2 and 4 token tiles by the row count, at 128. Logits after a
    131-token prompt in batches of each."""
    shape = synth.ModelShape(n_layer=1, hidden=hidden, ffn=ffn, heads=hidden // 128, kv_heads=4, hdim=128, vocab=300, ctx=140)
    model = synth.make_model(shape, mode="q4km", seed=191)
    g = synth.rng(192 + ffn)
    for nm in ("wg", "wu"):
        model["layers"][0][nm] = synth.make_weight(g, gt, ffn, hidden)
    prompt = synth.rand_prompt(synth.rng(193), 131, shape.vocab)
    ref = oracle_logits(model, prompt)
    fm = lib.FusedModel(backend, model)
    try:
        for batch in (16, 48, 128):
            assert np.array_equal(bits(fm.prefill(list(prompt), batch=batch)), bits(ref)), f"batch={batch}"
    finally:
        fm.close()


@pytest.mark.parametrize("gt", [abi.GT_Q4_K, abi.GT_Q6_K])
def test_pipelined_forms(backend, gt):
    """Every weight of one kind, four layers and four chunks of a prompt (the last one short): the
    pipelined launches of one to four chunks in their three forms, pairs and single jobs, against the same
    chunks one after another, whose launches the tests above compare with the oracle. Ids of the device
    loop and logits after them."""
    shape = synth.ModelShape(n_layer=4, hidden=2048, ffn=6144, heads=16, kv_heads=4, hdim=128, vocab=500, ctx=520)
    model = synth.make_model(synth.ModelShape(**{**shape.__dict__, "ffn": 256}), mode="q4km", seed=201)
    model["shape"] = shape
    g = synth.rng(202 + gt)
    dims = dict(wq=(2048, 2048), wk=(512, 2048), wv=(512, 2048), wo=(2048, 2048), wg=(6144, 2048), wu=(6144, 2048), wd=(2048, 6144))
    weights = {nm: raw_weight(g, gt, n, k, False) for nm, (n, k) in dims.items()}
    for L in model["layers"]:
        L.update(weights)
    prompt = synth.rand_prompt(synth.rng(203), 500, shape.vocab)
    fm = lib.FusedModel(backend, model)
    try:
        got = []
        for chunk, depth in ((128, 1), (128, 8), (40, 8), (128, 3)):
            before = backend.prefill_pipeline(depth)
            ids, _ = fm.generate_device(prompt, 4, chunk=chunk)
            got.append((ids, fm.forward([int(ids[-1])], 503, True)))
            backend.prefill_pipeline(before)
        assert np.isfinite(got[0][1]).all()
        for ids, logits in got[1:]:
            assert np.array_equal(ids, got[0][0]) and np.array_equal(bits(logits), bits(got[0][1]))
    finally:
        fm.close()


def test_gemm_kq_in_a_model(backend):
    """Mixed q/k (Q4_K) and v (Q6_K) rows in one launch, Q4_K gate/up pairs with the SwiGLU epilogue and
    residual adds, at the 1.8B layer's dimensions and at batches of one, three, five and eight token tiles."""
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
