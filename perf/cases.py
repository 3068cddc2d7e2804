"""The performance cases: the work a program has this backend do, through its public entry points.

A translation program (the Hy-MT2 host, or a program that drives the backend through
``hymt2_amd.lib``) does four kinds of work, and the cases cover each from its smallest calls to its
largest:

* ``layer``: the seven quantized contractions of one transformer layer for ``nt`` tokens, with the
  Q8_K quantization of their inputs (``Backend.quantize_q8k``, ``Backend.matvec``): one token in
  decode, up to 16 in the host's batches, up to 128 in a prefill chunk, for the three weight mixes
  (STQ1_0, Q2_0C, and Q4_K with Q6_K for v and down).
* ``ffn_in`` and ``head``: the decode step's fused feed-forward input and the LM head.
* ``per_op``: the host's unfused path, ``matmul`` of one weight group on host buffers.
* ``forward`` and ``generate``: whole models, one ``fused_forward`` batch of the host and a whole
  greedy translation on the device; both give logits.

Weights are random blocks of the real formats (Q4_K and Q6_K quantized from N(0, 0.02), the
ternary and 2-bit panels with uniform codes and the benchmark's scale ranges), activations are
N(0, 1). Every output of this backend is defined bit for bit, so the tolerance is exact.
"""
import ctypes
import math

import numpy as np
import torch

from hymt2_amd import abi, lib, synth

QK = 256
SEG = np.array([0, 2, 1, 3])  # panel segment of each 64-weight chunk of a block

TYPES = {
    "stq": dict.fromkeys(("wq", "wk", "wv", "wo", "wg", "wu", "wd"), abi.GT_STQ1_0),
    "q2": dict.fromkeys(("wq", "wk", "wv", "wo", "wg", "wu", "wd"), abi.GT_Q2_0C),
    "q4km": dict(wq=abi.GT_Q4_K, wk=abi.GT_Q4_K, wv=abi.GT_Q6_K, wo=abi.GT_Q4_K, wg=abi.GT_Q4_K,
                 wu=abi.GT_Q4_K, wd=abi.GT_Q6_K),
}
NAMES = ("wq", "wk", "wv", "wo", "wg", "wu", "wd")
GROUPS = {"qkv": ("wq", "wk", "wv"), "gate_up": ("wg", "wu"), "down": ("wd",)}
HEADS = {"f16": abi.GT_F16, "q8_0": abi.GT_Q8_0, "q6k": abi.GT_Q6_K}
# device bytes of 256 weights
BLOCK_BYTES = {abi.GT_STQ1_0: 68, abi.GT_Q2_0C: 68, abi.GT_Q4_K: 144, abi.GT_Q6_K: 210, abi.GT_F16: 512,
               abi.GT_Q8_0: 272}


# ------------------------------------------------------------------------------------- the cases

def listed():
    full = dict(hidden=2048, kv=512, ffn=6144)
    model = dict(layers=32, hidden=2048, ffn=6144, heads=16, kv_heads=4, vocab=120818)
    return [
        # the contractions of one decoded token, one call each: latency and launches
        dict(name="layer stq x1", op="layer", mode="stq", nt=1, **full),
        # the host's largest prompt batch (16 tokens), and a prefill chunk of the device loop
        dict(name="layer q4km x16", op="layer", mode="q4km", nt=16, **full),
        dict(name="layer q2 x128", op="layer", mode="q2", nt=128, **full),
        dict(name="layer q4km x128", op="layer", mode="q4km", nt=128, **full),
        # the decode step's widest kernel, alone: the smallest call
        dict(name="ffn_in stq", op="ffn_in", mode="stq", hidden=2048, ffn=6144),
        # the tied fp16 embedding as LM head: the largest read of a decoded token
        dict(name="head f16", op="head", type="f16", hidden=2048, vocab=120818),
        # one token through the host's unfused path (HYMT2_FUSED=0): host buffers in and out
        dict(name="per_op q4km gate_up x1", op="per_op", mode="q4km", group="gate_up", nt=1, **full),
        # the host's own loop: a decoded token, and a batch of its prompt after three others
        dict(name="host step stq", op="forward", mode="stq", head="f16", nt=1, past=150, **model),
        dict(name="host batch q4km x16", op="forward", mode="q4km", head="q6k", nt=16, past=48, **model),
        # a sentence translated with the ternary model: a short prompt, then decode
        dict(name="sentence stq", op="generate", mode="stq", head="f16", prompt=64, new=48, chunk=64, **model),
        # a page put to the 2-bit model: a long chunked prefill, and the first ids of the answer
        dict(name="page q2", op="generate", mode="q2", head="f16", prompt=1024, new=8, chunk=128, **model),
        # a paragraph translated with the 4-bit model and its quantized head
        dict(name="paragraph q4km", op="generate", mode="q4km", head="q6k", prompt=200, new=24, chunk=128, **model),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choices(("layer", "ffn_in", "head", "per_op", "forward", "generate"), (3, 1, 1, 1, 2, 3))[0]
    mode = rng.choice(("stq", "q2", "q4km"))
    # half of the draws at the 1.8B model's dimensions, half at others
    if rng.random() < 0.5:
        dims = dict(hidden=2048, kv=512, ffn=6144)
    else:
        dims = dict(hidden=512 * rng.randint(1, 5), kv=rng.randint(64, 1024), ffn=512 * rng.randint(2, 14))
    if op == "layer":
        return dict(op=op, mode=mode, nt=_log_int(rng, 1, 128), **dims)
    if op == "ffn_in":
        return dict(op=op, mode=mode, hidden=2048, ffn=_log_int(rng, 1000, 9000))
    if op == "head":
        return dict(op=op, type=rng.choice(("f16", "f16", "q8_0")), hidden=dims["hidden"], vocab=_log_int(rng, 8000, 120818))
    if op == "per_op":
        return dict(op=op, mode=mode, group=rng.choice(sorted(GROUPS)), nt=_log_int(rng, 1, 16), **dims)
    model = dict(layers=rng.randint(2, 12), hidden=2048, ffn=6144, heads=16, kv_heads=4, vocab=_log_int(rng, 4000, 60000))
    head = rng.choice(("f16", "q6k"))
    if op == "forward":
        return dict(op=op, mode=mode, head=head, nt=_log_int(rng, 1, 128), past=rng.randint(0, 300), **model)
    return dict(op=op, mode=mode, head=head, prompt=_log_int(rng, 16, 900), new=_log_int(rng, 2, 48),
                chunk=rng.choice((16, 64, 128)), **model)


# ------------------------------------------------------------------------------------- weights

class Weights:
    """Random blocks of each format, made once a state from its seed; weights are runs of them."""

    def __init__(self, seed):
        self.g = np.random.Generator(np.random.PCG64(seed))
        self.pools = {}

    def _runs(self, key, blocks, count, make):
        """`count` consecutive blocks of a pool of at least `blocks`, from a random place."""
        pool = self.pools.get(key)
        if pool is None or len(pool) < count:
            pool = self.pools[key] = make(max(blocks, count + count // 2))
        at = int(self.g.integers(0, len(pool) - count + 1))
        return pool[at:at + count]

    def _gathered(self, quantize, shape):
        def make(count):
            few = quantize(self.g.normal(0, 0.02, (1024, QK)).astype(np.float32)).reshape(1024, shape)
            return few[self.g.integers(0, 1024, count)]
        return make

    def make(self, gtype, n, k):
        nb = n * (k // QK)
        if gtype in (abi.GT_STQ1_0, abi.GT_Q2_0C):
            stq = gtype == abi.GT_STQ1_0

            def codes(count):
                raw = np.frombuffer(self.g.bytes(count * 64), np.uint8).reshape(count, 64)
                return synth.STQ_CODEBOOK[raw & 31] if stq else raw

            def scales(count):
                lo, hi = (0.005, 0.05) if stq else (0.002, 0.02)
                return self.g.uniform(lo, hi, count).astype(np.float16).astype(np.float32)

            pk = self._runs(("codes", stq), 65536, nb, codes).reshape(n, k // QK, 64)
            if stq:
                ps = self._runs(("scales", stq), 65536, nb, scales).reshape(n, k // QK)
            else:  # one scale per 512 weights
                ps = np.repeat(self._runs(("scales", stq), 65536, nb // 2, scales), 2).reshape(n, k // QK)
            return synth.Weight(gtype, k, n, None, np.ascontiguousarray(pk), np.ascontiguousarray(ps), 0 if stq else 1,
                                1 if stq else 3)
        if gtype == abi.GT_Q4_K:
            data = self._runs("q4k", 65536, nb, self._gathered(synth.quantize_q4_k, 144))
        elif gtype == abi.GT_Q6_K:
            data = self._runs("q6k", 65536, nb, self._gathered(synth.quantize_q6_k, 210))
        elif gtype == abi.GT_F16:
            few = self.g.normal(0, 0.02, 1 << 21).astype(np.float16)
            few = few[:len(few) - 1 - int(self.g.integers(0, 999))]  # rows start at other places of it
            data = np.resize(few, n * k).view(np.uint8)
        elif gtype == abi.GT_Q8_0:
            data = self._runs("q8_0", 4096, nb, self._gathered(synth.quantize_q8_0, 272))
        else:
            raise ValueError(f"no weights of type {gtype}")
        return synth.Weight(gtype, k, n, np.ascontiguousarray(data).reshape(n, -1))


def _dims(case):
    """(rows, columns) of the layer's weights."""
    h, f, kv = case["hidden"], case["ffn"], case["kv"]
    return dict(wq=(h, h), wk=(kv, h), wv=(kv, h), wo=(h, h), wg=(f, h), wu=(f, h), wd=(h, f))


def _model(case, w):
    shape = synth.ModelShape(n_layer=case["layers"], hidden=case["hidden"], ffn=case["ffn"], heads=case["heads"],
                             kv_heads=case["kv_heads"], hdim=128, vocab=case["vocab"], ctx=_positions(case) + 8)
    types, dims = TYPES[case["mode"]], _dims(dict(case, kv=shape.kvdim))
    layers = []
    for _ in range(shape.n_layer):
        layer = {nm: w.g.uniform(0.9, 1.1, n).astype(np.float32)
                 for nm, n in (("attn_norm", shape.hidden), ("ffn_norm", shape.hidden), ("q_norm", 128), ("k_norm", 128))}
        layer.update({nm: w.make(types[nm], *dims[nm]) for nm in NAMES})
        layers.append(layer)
    head = w.make(HEADS[case["head"]], shape.vocab, shape.hidden)
    angle = np.arange(shape.ctx, dtype=np.float64)[:, None] * 10000.0 ** (-np.arange(64) / 64.0)
    return dict(shape=shape, mode=case["mode"], layers=layers, embd=head, outw=head,
                out_norm=w.g.uniform(0.9, 1.1, shape.hidden).astype(np.float32),
                rope_cos=np.cos(angle).astype(np.float32), rope_sin=np.sin(angle).astype(np.float32),
                vocab_out=shape.vocab)


def _positions(case):
    return case["past"] + case["nt"] if case["op"] == "forward" else case["prompt"] + case["new"]


class Held:
    """A backend context with what it holds; released with the state."""

    def __init__(self):
        self.backend = lib.Backend()
        self.model, self.handles = None, []

    def upload(self, weight):
        self.handles.append(self.backend.upload(weight))
        return self.handles[-1]

    def __del__(self):
        if getattr(self, "backend", None) is not None and self.backend.impl:
            if self.model is not None:
                self.model.close()
            for h in self.handles:
                self.backend.release(h)
            self.backend.close()


# ------------------------------------------------------------------------------------- a state

def _inputs(case, w):
    """The activations the contractions read: nt rows of the hidden size, and of the FFN's."""
    nt = case.get("nt", 1)
    return {k: w.g.standard_normal((nt, k), dtype=np.float32) for k in (case["hidden"], case["ffn"])}


def _contractions(case):
    names = GROUPS[case["group"]] if case["op"] == "per_op" else NAMES
    return [(nm, TYPES[case["mode"]][nm], *_dims(case)[nm]) for nm in names]


def prepare(case, seed):
    w = Weights(seed)
    op = case["op"]
    held = Held()
    s = dict(case=case, held=held)
    b = held.backend
    if op in ("layer", "per_op"):
        nt = case["nt"]
        weights = [(nm, held.upload(w.make(t, n, k)), n, k) for nm, t, n, k in _contractions(case)]
        x = {k: torch.from_numpy(v).cuda() for k, v in _inputs(case, w).items()}
        act = {k: torch.zeros(nt * (k // QK) * abi.Q8K_BYTES, dtype=torch.uint8, device="cuda") for k in x}
        if op == "layer":
            s.update(weights=weights, x=x, act=act,
                     out=[torch.zeros((nt, n), dtype=torch.float32, device="cuda") for _, _, n, _ in weights])
        else:  # the host's own Q8_K blocks of the group's input
            k = weights[0][3]
            torch.cuda.synchronize()
            b.quantize_q8k(x[k].data_ptr(), act[k].data_ptr(), k, nt)
            torch.cuda.synchronize()
            s.update(handles=[h for _, h, _, _ in weights], rows=[n for _, _, n, _ in weights], xq=act[k].cpu().numpy())
    elif op == "ffn_in":
        h, f = case["hidden"], case["ffn"]
        t = TYPES[case["mode"]]["wg"]
        s.update(gate=held.upload(w.make(t, f, h)), up=held.upload(w.make(t, f, h)),
                 h=torch.from_numpy(w.g.standard_normal(h, dtype=np.float32)).cuda(),
                 norm=torch.from_numpy(w.g.uniform(0.9, 1.1, h).astype(np.float32)).cuda(),
                 out=torch.zeros(f, dtype=torch.float32, device="cuda"))
    elif op == "head":
        s.update(weight=held.upload(w.make(HEADS[case["type"]], case["vocab"], case["hidden"])),
                 h=torch.from_numpy(w.g.standard_normal(case["hidden"], dtype=np.float32)).cuda(),
                 norm=torch.from_numpy(w.g.uniform(0.9, 1.1, case["hidden"]).astype(np.float32)).cuda(),
                 out=torch.zeros(case["vocab"], dtype=torch.float32, device="cuda"))
    else:
        held.model = lib.FusedModel(b, _model(case, w))
        ids = w.g.integers(3, case["vocab"], _positions(case), dtype=np.int32)
        if op == "forward":
            s.update(ids=[int(t) for t in ids[case["past"]:]])
            if case["past"]:
                held.model.prefill([int(t) for t in ids[:case["past"]]], batch=128)
        else:
            s.update(prompt=ids[:case["prompt"]])
    torch.cuda.synchronize()
    return s


def run(s):
    case, held = s["case"], s["held"]
    b, op = held.backend, case["op"]
    if op == "layer":
        nt = case["nt"]
        for k, x in s["x"].items():
            b.quantize_q8k(x.data_ptr(), s["act"][k].data_ptr(), k, nt)
        for (_, h, _, k), out in zip(s["weights"], s["out"]):
            b.matvec(h, s["act"][k].data_ptr(), out.data_ptr(), nt)
        return s["out"]
    if op == "per_op":
        return b.matmul(s["handles"], s["rows"], s["xq"], case["nt"])
    if op == "ffn_in":
        if b.L.hymt2_hip_ffn_in(b.impl, s["gate"], s["up"], s["h"].data_ptr(), s["norm"].data_ptr(),
                                ctypes.c_float(1e-5), s["out"].data_ptr()) != 0:
            raise RuntimeError(f"ffn_in failed: {b.last_error()}")
        return s["out"]
    if op == "head":
        if b.L.hymt2_hip_head(b.impl, s["weight"], s["h"].data_ptr(), s["norm"].data_ptr(), ctypes.c_float(1e-5),
                              s["out"].data_ptr(), 0, None) != 0:
            raise RuntimeError(f"head failed: {b.last_error()}")
        return s["out"]
    if op == "forward":
        return held.model.forward(s["ids"], case["past"])
    # greedy ids on the device, then the logits that follow the last of them
    ids, _ = held.model.generate_ids(s["prompt"], case["new"], chunk=case["chunk"])
    return dict(ids=ids, logits=held.model.forward([int(ids[-1])], case["prompt"] + case["new"] - 1))


# ------------------------------------------------------------------------------------- the floor

def _weight_bytes(gtype, n, k):
    return n * (k // QK) * BLOCK_BYTES[gtype]


def work(case):
    op = case["op"]
    if op in ("layer", "per_op"):
        parts, nt = _contractions(case), case["nt"]
        w = sum(_weight_bytes(t, n, k) for _, t, n, k in parts)
        out = 4 * nt * sum(n for _, _, n, _ in parts)
        fed = {k for _, _, _, k in parts}
        rows = nt * (sum(4 * k for k in fed) if op == "layer" else sum(k // QK * abi.Q8K_BYTES for k in fed))
        return dict(bytes=w + out + rows, flops=2 * nt * sum(n * k for _, _, n, k in parts))
    if op == "ffn_in":
        h, f, t = case["hidden"], case["ffn"], TYPES[case["mode"]]["wg"]
        return dict(bytes=2 * _weight_bytes(t, f, h) + 8 * h + 4 * f, flops=4 * f * h)
    if op == "head":
        h, v = case["hidden"], case["vocab"]
        return dict(bytes=_weight_bytes(HEADS[case["type"]], v, h) + 8 * h + 4 * v, flops=2 * v * h)
    # whole models: every forward reads all weights once (a prompt in one), each token its own K/V
    dims, types = _dims(dict(case, kv=128 * case["kv_heads"])), TYPES[case["mode"]]
    layer = sum(_weight_bytes(types[nm], *dims[nm]) for nm in NAMES)
    per_token = 2 * case["layers"] * sum(n * k for n, k in dims.values())
    head = _weight_bytes(HEADS[case["head"]], case["vocab"], case["hidden"])
    head_flops = 2 * case["vocab"] * case["hidden"]
    kv_row = case["layers"] * case["kv_heads"] * 128 * 2 * 2  # bytes of one position's K and V
    attn = 4 * case["layers"] * case["heads"] * 128           # operations a position attended to
    last = _positions(case)
    if op == "forward":
        forwards, heads, first, tokens = 1, 1, case["past"], case["nt"]
        kv = kv_row * last
    else:
        forwards, heads, first, tokens = case["new"] + 1, case["new"] + 1, 0, last
        kv = kv_row * (case["prompt"] + sum(range(case["prompt"] + 1, last + 1)))
    attended = (first + last) * tokens / 2
    return dict(bytes=forwards * case["layers"] * layer + heads * head + kv,
                flops=tokens * per_token + heads * head_flops + attn * attended)


def tolerance(case):
    # every output is a fixed sequence of IEEE single operations (or exact integers): the same bits
    return "exact"


# ------------------------------------------------------------------------------------- 64 bits

def _q8k(x):
    """Q8_K of rows x: integers and scales of each 256-element block, as float64 rows d * q."""
    v = x.reshape(-1, QK)
    at = np.abs(v).argmax(1)
    top = v[np.arange(len(v)), at]
    inv = np.where(top == 0, np.float32(0), np.float32(-127) / np.where(top == 0, np.float32(1), top)).astype(x.dtype)
    q = np.clip(np.rint(inv[:, None] * v), -127, 127).astype(np.float64)
    d = np.where(inv == 0, 0, 1 / np.where(inv == 0, 1, inv)).astype(x.dtype).astype(np.float64)
    return (d[:, None] * q).reshape(x.shape)


def _values(w):
    """A weight's values as float64 [n][k]."""
    n, k = w.n, w.k
    if w.type in (abi.GT_STQ1_0, abi.GT_Q2_0C):
        seg = w.pk.reshape(n, k // QK, 4, 1, 16)[:, :, SEG]
        code = (seg >> np.arange(0, 8, 2, dtype=np.uint8).reshape(1, 1, 1, 4, 1)) & 3
        return ((code.astype(np.float64) * 2 ** w.pshift - w.poff).reshape(n, k // QK, QK)
                * w.ps.astype(np.float64)[:, :, None]).reshape(n, k)
    b = w.data.reshape(n * k // QK, -1)
    f16 = lambda a: np.ascontiguousarray(a).view(np.float16).astype(np.float64)  # noqa: E731
    if w.type == abi.GT_F16:
        return w.data.view(np.float16).astype(np.float64).reshape(n, k)
    if w.type == abi.GT_Q8_0:
        b = b.reshape(-1, 34)
        return (f16(b[:, :2]) * np.ascontiguousarray(b[:, 2:]).view(np.int8)).reshape(n, k)
    if w.type == abi.GT_Q4_K:
        s, q = b[:, 4:16], b[:, 16:].reshape(-1, 4, 32)
        scale = np.concatenate([s[:, :4] & 63, (s[:, 8:] & 15) | (s[:, :4] >> 6 << 4)], 1)
        least = np.concatenate([s[:, 4:8] & 63, (s[:, 8:] >> 4) | (s[:, 4:8] >> 6 << 4)], 1)
        q = np.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32)
        return ((f16(b[:, :2]) * scale)[:, :, None] * q - (f16(b[:, 2:4]) * least)[:, :, None]).reshape(n, k)
    ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 1, 32)  # Q6_K
    low = np.concatenate([ql & 15, ql >> 4], 2)
    high = qh >> np.array([0, 2, 4, 6], np.uint8).reshape(1, 1, 4, 1) & 3
    scale = f16(b[:, 208:210]) * np.ascontiguousarray(b[:, 192:208]).view(np.int8)
    return (scale[:, :, None] * ((low | high << 4).astype(np.float64) - 32).reshape(-1, 16, 16)).reshape(n, k)


def _product(w, x):
    """x @ values(w).T in float64, on the GPU in runs of rows."""
    x, out = torch.from_numpy(x).cuda(), []
    per = max(1, (1 << 25) // w.k)
    for r in range(0, w.n, per):
        part = synth.Weight(w.type, w.k, min(per, w.n - r), None if w.data is None else w.data[r:r + per],
                            None if w.pk is None else w.pk[r:r + per], None if w.ps is None else w.ps[r:r + per],
                            w.pshift, w.poff)
        out.append((torch.from_numpy(_values(part)).cuda() @ x.T).T)
    return torch.cat(out, 1).cpu().numpy()


def _normed(h, norm):
    h = h.astype(np.float64)
    return h / np.sqrt((h * h).mean() + float(np.float32(1e-5))) * norm


def exact(case, seed):
    w, op = Weights(seed), case["op"]
    if op in ("layer", "per_op"):
        weights = [w.make(t, n, k) for _, t, n, k in _contractions(case)]
        x = {k: _q8k(v) for k, v in _inputs(case, w).items()}
        return [_product(m, x[m.k]) for m in weights]
    if op == "ffn_in":
        t = TYPES[case["mode"]]["wg"]
        gate, up = w.make(t, case["ffn"], case["hidden"]), w.make(t, case["ffn"], case["hidden"])
        h = w.g.standard_normal(case["hidden"], dtype=np.float32)
        x = _q8k(_normed(h, w.g.uniform(0.9, 1.1, case["hidden"]).astype(np.float32))[None])
        g, u = _product(gate, x)[0], _product(up, x)[0]
        return g / (1 + np.exp(-g)) * u
    if op == "head":
        m = w.make(HEADS[case["type"]], case["vocab"], case["hidden"])
        h = w.g.standard_normal(case["hidden"], dtype=np.float32)
        return _product(m, _normed(h, w.g.uniform(0.9, 1.1, case["hidden"]).astype(np.float32))[None])[0]
    return None  # whole models: minutes in float64
