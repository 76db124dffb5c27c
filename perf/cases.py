"""The work a user of this package has it do, as measurable cases.

Five operations, each through the package's public entry points:

  matmul   y = W x for block-quantized weights (gpu.device_matmul_into): one
           token (decode), 2..8 tokens (several sequences), more (prompts).
           `mats` matrices of the same shape in turn, as a decode step goes
           through a model's layers: with enough of them the weights come from
           memory and not from a cache.
  head     the output head: final norm, projection onto the vocabulary, pick.
  attend   one query against a KV cache (gpu.device_attend).
  layer    one decoder layer: `tokens` sequences with one token each
           (chunk false), or one sequence's chunk of a prompt (chunk true).
  session  a small model through block.DeviceSession: a whole prompt and the
           logits after it, or one decode step.

Weights are drawn so that every value is about N(0, 1 / cols): outputs of a
projection are of the size of its inputs, as in a trained model, and softmax
is neither flat nor one-hot.
"""

from __future__ import annotations

import math

import torch

from molla_amd import block, gpu

KINDS = {"q4_0": gpu.Q_Q4_0, "q4_1": gpu.Q_Q4_1, "q5_0": gpu.Q_Q5_0, "q5_1": gpu.Q_Q5_1, "q8_0": gpu.Q_Q8_0,
         "q4_k": gpu.Q_Q4_K, "q5_k": gpu.Q_Q5_K, "q6_k": gpu.Q_Q6_K}
BLOCK = {"q4_0": (32, 18), "q4_1": (32, 20), "q5_0": (32, 22), "q5_1": (32, 24), "q8_0": (32, 34),
         "q4_k": (256, 144), "q5_k": (256, 176), "q6_k": (256, 210)}
# the kinds of a layer's projections (q and k, v, wo, gate and up, down) as
# quantized files mix them
MIXES = {"q4_k": ("q4_k", "q4_k", "q4_k", "q4_k", "q4_k"),
         "q4_k_m": ("q4_k", "q6_k", "q4_k", "q4_k", "q6_k"),
         "q5_k_m": ("q5_k", "q6_k", "q5_k", "q5_k", "q6_k"),
         "q4_0": ("q4_0",) * 5,
         "q8_0": ("q8_0",) * 5}
PROJECTIONS = ("wq", "wk", "wv", "wo", "gate", "up", "down")
MIX_OF = {"wq": 0, "wk": 0, "wv": 1, "wo": 2, "gate": 3, "up": 3, "down": 4}
EPS = 1e-5
ROPE_BASE = 500000.0


def listed():
    return [
        # the smallest projection in use: one token through a small model's MLP matrix
        dict(name="q8_0 4864x896, 1 token", op="matmul", kind="q8_0", rows=4864, cols=896, tokens=1, mats=1, epi="none"),
        # single-user decode: an 8B model's gate or up, from memory
        dict(name="q4_k 14336x4096, 1 token", op="matmul", kind="q4_k", rows=14336, cols=4096, tokens=1, mats=12,
             epi="none"),
        # four sequences decoding together, 4-bit legacy blocks: the down projection
        dict(name="q4_0 4096x14336, 4 tokens", op="matmul", kind="q4_0", rows=4096, cols=14336, tokens=4, mats=12,
             epi="none"),
        # a 5-bit file at an odd batch: gate behind its up (the gated epilogue)
        dict(name="q5_k 14336x4096, 5 tokens", op="matmul", kind="q5_k", rows=14336, cols=4096, tokens=5, mats=8,
             epi="glu"),
        # a ragged short prompt in 8-bit blocks
        dict(name="q8_0 4096x4096, 75 tokens", op="matmul", kind="q8_0", rows=4096, cols=4096, tokens=75, mats=4,
             epi="none"),
        # a prompt chunk through the largest matrix of a layer
        dict(name="q4_k 14336x4096, 256 tokens", op="matmul", kind="q4_k", rows=14336, cols=4096, tokens=256, mats=4,
             epi="none"),
        # eight sequences' next tokens
        dict(name="head q6_k 128256x4096, 8", op="head", kind="q6_k", rows=128256, cols=4096, tokens=8),
        # one query over a long cache
        dict(name="attend f16 32768", op="attend", form="f16", heads=32, kv_heads=8, head_dim=128, count=32768),
        # an 8B layer's token at position 4096
        dict(name="layer 8B 1 token", op="layer", mix="q4_k", width=4096, hidden=14336, heads=32, kv_heads=8,
             head_dim=128, tokens=1, chunk=False, pos=4096, context=4352, form="f16", paged=False),
        # eight sequences over paged q8_0 caches, mixed kinds
        dict(name="layer 8B 8 paged q8", op="layer", mix="q4_k_m", width=4096, hidden=14336, heads=32, kv_heads=8,
             head_dim=128, tokens=8, chunk=False, pos=6000, context=8192, form="q8", paged=True),
        # a prompt's chunk well into its context
        dict(name="layer 8B chunk 256", op="layer", mix="q4_k_m", width=4096, hidden=14336, heads=32, kv_heads=8,
             head_dim=128, tokens=256, chunk=True, pos=3840, context=4352, form="f16", paged=False),
        # a whole prompt (time to the first token) of two layers and a head, into a q8_0 cache
        dict(name="session prompt 1500 q8", op="session", mode="prompt", mix="q4_k", layers=2, width=4096, hidden=14336,
             heads=32, kv_heads=8, head_dim=128, vocab=32768, batch=1, prompt=1500, context=2048, form="q8"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _step(rng, lo, hi, step):
    return max(lo, _log(rng, lo, hi) // step * step)


def draw(rng):
    op = rng.choice(["matmul", "matmul", "matmul", "head", "attend", "attend", "layer", "layer", "layer", "session"])
    if op == "matmul":
        kind = rng.choice(list(BLOCK))
        tokens = rng.choice([1, rng.randint(2, 8), _log(rng, 9, 512)])
        rows = _log(rng, 256, 16384)
        cols = _step(rng, 256, 14336, 256)
        one = rows * cols * BLOCK[kind][1] // BLOCK[kind][0]
        mats = max(1, min(12 if tokens <= 8 else 4, 400_000_000 // one))
        return dict(op="matmul", kind=kind, rows=rows, cols=cols, tokens=tokens, mats=rng.randint(1, mats),
                    epi=rng.choice(["none", "none", "bias", "glu"]))
    if op == "head":
        return dict(op="head", kind=rng.choice(["q6_k", "q6_k", "q8_0", "q4_k"]), rows=_log(rng, 4096, 128256),
                    cols=_step(rng, 512, 4096, 256), tokens=rng.randint(1, 8))
    if op == "attend":
        kv = rng.choice([1, 2, 4, 8])
        return dict(op="attend", form=rng.choice(["f16", "f16", "q8"]), heads=kv * rng.choice([1, 2, 4, 8]), kv_heads=kv,
                    head_dim=rng.choice([64, 128, 128, 256]), count=_log(rng, 1, 65536))
    size = rng.choice([(1024, 2816, 16, 4, 64), (2048, 5632, 32, 4, 64), (2048, 8192, 16, 8, 128),
                       (4096, 11008, 32, 32, 128), (4096, 14336, 32, 8, 128)])
    width, hidden, heads, kv_heads, head_dim = size
    mix = rng.choice(list(MIXES))
    form = rng.choice(["f16", "f16", "q8"])
    if op == "layer":
        chunk = rng.random() < 0.4
        tokens = _log(rng, 9, 400) if chunk else rng.choice([1, rng.randint(2, 8)])
        pos = _log(rng, 1, 8192 if chunk else 16384) - 1
        context = _log(rng, pos + tokens, 16384 + 512)
        return dict(op="layer", mix=mix, width=width, hidden=hidden, heads=heads, kv_heads=kv_heads, head_dim=head_dim,
                    tokens=tokens, chunk=chunk, pos=pos, context=context, form=form, paged=rng.random() < 0.3)
    mode = rng.choice(["prompt", "step"])
    prompt = _log(rng, 9, 1500) if mode == "prompt" else _log(rng, 1, 4000)
    return dict(op="session", mode=mode, mix=mix, layers=rng.randint(1, 2), width=width, hidden=hidden, heads=heads,
                kv_heads=kv_heads, head_dim=head_dim, vocab=_log(rng, 2048, 32768),
                batch=1 if mode == "prompt" else rng.randint(1, 8), prompt=prompt,
                context=_log(rng, prompt + 1, 4096), form=form)


# ---- inputs ----------------------------------------------------------------
class _Inputs:
    """Draws from one seed, in the order asked."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, *shape, mean=0.0, std=1.0):
        return torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32) * std + mean

    def ints(self, lo, hi, shape):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda", dtype=torch.int32)

    def blob(self, kind, rows, cols):
        """A (rows x cols) tensor's blocks; values of about N(0, 1 / cols)."""
        per, size = BLOCK[kind]
        n = rows * cols // per
        std = 1.0 / math.sqrt(cols)
        # the random bytes are the codes; the scale fields are written over them
        b = torch.randint(-2 ** 31, 2 ** 31 - 1, ((n * size + 3) // 4,), generator=self.g, device="cuda",
                          dtype=torch.int32).view(torch.uint8)[:n * size].reshape(n, size)
        jitter = 0.5 + torch.rand(n, generator=self.g, device="cuda", dtype=torch.float32)

        def half(v):
            return v.to(torch.float16).view(torch.uint8).reshape(-1, 2)

        if kind == "q8_0":
            b[:, :2] = half(jitter * (std / 74))
        elif kind in ("q4_0", "q5_0"):
            b[:, :2] = half(jitter * (std / (4.6 if kind == "q4_0" else 9.2)))
        elif kind in ("q4_1", "q5_1"):
            mid, spread = (7.5, 4.6) if kind == "q4_1" else (15.5, 9.2)
            b[:, :2] = half(jitter * (std / spread))
            b[:, 2:4] = half(jitter * (-mid * std / spread))
        elif kind in ("q4_k", "q5_k"):
            mid, spread = (7.5, 4.6) if kind == "q4_k" else (15.5, 9.2)
            sc = self.ints(24, 64, (n, 8))
            m = (sc + self.ints(-3, 4, (n, 8))).clamp(0, 63)
            b[:, :2] = half(jitter * (std / (44 * spread)))
            b[:, 2:4] = half(jitter * (mid * std / (44 * spread)))
            b[:, 4:8] = ((sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6)).to(torch.uint8)
            b[:, 8:12] = ((m[:, :4] & 63) | ((m[:, 4:] >> 4) << 6)).to(torch.uint8)
            b[:, 12:16] = ((sc[:, 4:] & 15) | ((m[:, 4:] & 15) << 4)).to(torch.uint8)
        else:
            s = self.ints(-64, 64, (n, 16))
            b[:, 192:208] = (s + torch.where(s < 0, -32, 32)).to(torch.int8).view(torch.uint8)
            b[:, 208:210] = half(jitter * (std / (64 * 18.5)))
        return b.reshape(-1)

    def cache(self, form, cells, kv_width):
        """`cells` positions of a cache of either form: (cells, halves a position)."""
        v = self.normal(cells, kv_width)
        if form == "f16":
            return v.half()
        x = v.reshape(cells, kv_width // 32, 32)
        amax = x.abs().amax(-1)
        q = torch.trunc(x * (127.0 / amax)[..., None] + torch.where(x < 0, -0.5, 0.5)).clamp(-127, 127).to(torch.int8)
        row = torch.zeros(cells, gpu.cache_row(gpu.CACHE_Q8, kv_width), dtype=torch.float16, device="cuda")
        row[:, :kv_width // 2] = q.reshape(cells, kv_width).view(torch.float16)
        row[:, kv_width // 2:kv_width // 2 + kv_width // 32] = (amax / 127.0).half()
        return row


def _form(case):
    return gpu.CACHE_Q8 if case["form"] == "q8" else gpu.CACHE_F16


def _shapes(case):
    qw, kvw, w, h = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"], case["width"], case["hidden"]
    return {"wq": (qw, w), "wk": (kvw, w), "wv": (kvw, w), "wo": (w, qw), "gate": (h, w), "up": (h, w), "down": (w, h)}


def _layer_inputs(case, g):
    mix = MIXES[case["mix"]]
    host = {n: (mix[MIX_OF[n]], r, c, g.blob(mix[MIX_OF[n]], r, c)) for n, (r, c) in _shapes(case).items()}
    host["attn_norm"] = g.normal(case["width"], mean=1.0, std=0.1)
    host["ffn_norm"] = g.normal(case["width"], mean=1.0, std=0.1)
    return host


def _spec(case):
    return block.BlockSpec(width=case["width"], hidden=case["hidden"], heads=case["heads"], kv_heads=case["kv_heads"],
                           head_dim=case["head_dim"], rope_dim=case["head_dim"], rope_base=ROPE_BASE, neox=False, eps=EPS)


def _tensor(kind, rows, cols, blob):
    return gpu.Tensor.from_bytes(blob, KINDS[kind], cols, rows)


def _device_layer(case, host, steps):
    ws = {n: _tensor(*host[n]) for n in PROJECTIONS}
    return block.DeviceLayer(_spec(case), host["attn_norm"], host["ffn_norm"], ws, steps)


def _layer_state(case, g):
    """The tensors of a layer case, in the order they are drawn."""
    kvw, t = case["kv_heads"] * case["head_dim"], case["tokens"]
    seqs = 1 if case["chunk"] else t
    host = _layer_inputs(case, g)
    x = g.normal(t, case["width"])
    k, v = (g.cache(case["form"], seqs * case["context"], kvw) for _ in range(2))
    first = case["pos"]
    if case["chunk"]:
        pos = torch.arange(first, first + t, dtype=torch.int32, device="cuda")
    else:  # sequences of unequal length
        pos = (first - (torch.arange(t, device="cuda") * (first // 16))).clamp(min=0).to(torch.int32)
    index = None
    if case["paged"]:  # every sequence's positions in cells of its own, in no order
        order = torch.randperm(seqs * case["context"], generator=g.g, device="cuda")
        index = order.to(torch.int32).reshape(seqs, case["context"]).contiguous()
    return host, x, k, v, pos, index


def prepare(case, seed):
    g = _Inputs(seed)
    ctx = gpu.DeviceContext(0)
    op = case["op"]
    if op in ("matmul", "head"):
        mats = case.get("mats", 1)
        ws = [_tensor(case["kind"], case["rows"], case["cols"], g.blob(case["kind"], case["rows"], case["cols"]))
              for _ in range(mats)]
        x = g.normal(case["tokens"] * case["cols"])
        out = torch.empty(mats * case["tokens"] * case["rows"], device="cuda")
        if op == "head":
            gain = g.normal(case["cols"], mean=1.0, std=0.1)
            return dict(case=case, ctx=ctx, w=ws[0], x=x, gain=gain, xn=torch.empty_like(x), out=out)
        aux = g.normal(case["rows"] * (1 if case["epi"] == "bias" else case["tokens"]))
        epi = {"none": gpu.EPI_NONE, "bias": gpu.EPI_BIAS, "glu": gpu.EPI_GLU}[case["epi"]]
        return dict(case=case, ctx=ctx, ws=ws, x=x, aux=None if case["epi"] == "none" else aux, epi=epi, out=out)
    if op == "attend":
        qw, kvw = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
        q = g.normal(qw)
        k, v = (g.cache(case["form"], case["count"], kvw) for _ in range(2))
        return dict(case=case, ctx=ctx, q=q, k=k, v=v, out=torch.empty(qw, device="cuda"))
    steps = torch.from_numpy(gpu.rope_steps(case["head_dim"], ROPE_BASE)).cuda()
    if op == "layer":
        host, x, k, v, pos, index = _layer_state(case, g)
        layer = _device_layer(case, host, steps)
        work = torch.empty(block.layer_workspace(layer, case["context"], case["tokens"]) + 256, dtype=torch.uint8,
                           device="cuda")
        return dict(case=case, ctx=ctx, layer=layer, x0=x, x=torch.empty_like(x), k=k, v=v, pos=pos, index=index, work=work)
    hosts, emb, gain, head, ids, caches = _session_inputs(case, g)
    layers = [_device_layer(case, h, steps) for h in hosts]
    model = block.DeviceModel(_spec(case), emb, layers, gain, _tensor(*head))
    s = block.DeviceSession(ctx, model, case["batch"], case["context"], cache_form=_form(case))
    for i, (k, v) in enumerate(caches):
        s.k[i].copy_(k.reshape(-1))
        s.v[i].copy_(v.reshape(-1))
    if case["mode"] == "step":
        s.ids.copy_(ids)
        s.pos.fill_(case["prompt"])
        return dict(case=case, s=s)
    return dict(case=case, s=s, ids=ids)


def _session_inputs(case, g):
    hosts = [_layer_inputs(case, g) for _ in range(case["layers"])]
    emb = g.normal(case["vocab"], case["width"])
    gain = g.normal(case["width"], mean=1.0, std=0.1)
    head = ("q6_k", case["vocab"], case["width"], g.blob("q6_k", case["vocab"], case["width"]))
    ids = g.ints(0, case["vocab"], (case["prompt"] if case["mode"] == "prompt" else case["batch"],))
    kvw = case["kv_heads"] * case["head_dim"]
    # a decode step finds its context in the cache; a prompt fills it
    caches = [tuple(g.cache(case["form"], case["batch"] * case["context"], kvw) for _ in range(2))
              for _ in range(case["layers"])]
    return hosts, emb, gain, head, ids, caches


# ---- one pass --------------------------------------------------------------
def run(state):
    case = state["case"]
    op = case["op"]
    if op == "matmul":
        n = case["tokens"] * case["rows"]
        for i, w in enumerate(state["ws"]):
            gpu.device_matmul_into(state["ctx"], w, state["x"], state["out"], case["tokens"], i * n, state["epi"],
                                   state["aux"])
        return state["out"]
    if op == "head":
        gpu.device_rms_norm(state["ctx"], state["xn"], state["x"], state["gain"], EPS, case["tokens"])
        gpu.device_matmul_into(state["ctx"], state["w"], state["xn"], state["out"], case["tokens"])
        return dict(logits=state["out"], pick=gpu.device_argmax_ws(state["ctx"], state["out"], case["rows"], case["tokens"]))
    if op == "attend":
        gpu.device_attend(state["ctx"], state["q"], state["k"], state["v"], case["heads"], case["kv_heads"],
                          case["head_dim"], 1.0 / math.sqrt(case["head_dim"]), case["count"], state["out"], _form(case))
        return state["out"]
    if op == "layer":
        x, k, v = state["x"], state["k"], state["v"]
        x.copy_(state["x0"])  # the layer works in place
        kvw = case["kv_heads"] * case["head_dim"]
        if case["paged"]:
            block.device_layer_paged(state["ctx"], state["layer"], x, k, v, state["index"],
                                     0 if case["chunk"] else case["context"], state["pos"], case["context"],
                                     case["tokens"], state["work"], _form(case))
        else:
            stride = 0 if case["chunk"] else case["context"] * gpu.cache_row(_form(case), kvw)
            block.device_layer(state["ctx"], state["layer"], x, k, v, stride, state["pos"], case["context"],
                               case["tokens"], state["work"], _form(case))
        return dict(x=x, k=_seen(case, k), v=_seen(case, v))
    s = state["s"]
    if case["mode"] == "prompt":
        s.prefill(state["ids"])
        s.finish()
    else:
        s.step()
    return dict(logits=s.logits, x=s.x, k=[_seen(case, k) for k in s.k], v=[_seen(case, v) for v in s.v])


def _seen(case, cache):
    """A cache as numbers: halves, or the bytes of q8_0 rows."""
    return cache if case["form"] == "f16" else cache.view(torch.uint8)


# ---- what a pass cannot do without -----------------------------------------
def _bytes(kind, rows, cols):
    return rows * cols // BLOCK[kind][0] * BLOCK[kind][1]


def _layer_work(case, tokens, lengths, chunk):
    """Bytes and operations of one layer; lengths: the keys each token reads."""
    mix = MIXES[case["mix"]]
    b = sum(_bytes(mix[MIX_OF[n]], r, c) for n, (r, c) in _shapes(case).items())
    f = 2 * tokens * sum(r * c for r, c in _shapes(case).values())
    kvw = case["kv_heads"] * case["head_dim"]
    cell = 2 * kvw if case["form"] == "f16" else kvw + kvw // 16
    b += 2 * cell * (max(lengths) if chunk else sum(lengths)) + 8 * tokens * case["width"]
    f += 4 * case["heads"] * case["head_dim"] * sum(lengths)
    return b, f


def work(case):
    op = case["op"]
    if op in ("matmul", "head"):
        r, c, t, m = case["rows"], case["cols"], case["tokens"], case.get("mats", 1)
        b = m * (_bytes(case["kind"], r, c) + 4 * t * r) + 4 * t * c
        if op == "head":
            b += 4 * c + 4 * t
        elif case["epi"] != "none":
            b += m * 4 * r * (1 if case["epi"] == "bias" else t)
        return dict(bytes=b, flops=2 * m * r * c * t)
    if op == "attend":
        kvw = case["kv_heads"] * case["head_dim"]
        cell = 2 * kvw if case["form"] == "f16" else kvw + kvw // 16
        qw = case["heads"] * case["head_dim"]
        return dict(bytes=2 * cell * case["count"] + 8 * qw, flops=4 * qw * case["count"])
    t = case["tokens"] if op == "layer" else (case["prompt"] if case["mode"] == "prompt" else case["batch"])
    if op == "layer":
        if case["chunk"]:
            lengths = [case["pos"] + i + 1 for i in range(t)]
        else:
            lengths = [max(case["pos"] - i * (case["pos"] // 16), 0) + 1 for i in range(t)]
        b, f = _layer_work(case, t, lengths, case["chunk"])
        return dict(bytes=b, flops=f)
    prompt = case["mode"] == "prompt"
    lengths = list(range(1, t + 1)) if prompt else [case["prompt"] + 1] * t
    b, f = _layer_work(case, t, lengths, prompt)
    b, f = b * case["layers"], f * case["layers"]
    b += _bytes("q6_k", case["vocab"], case["width"]) + 4 * t * case["width"] + 4 * case["batch"] * case["vocab"]
    return dict(bytes=b, flops=f + 2 * case["batch"] * case["vocab"] * case["width"])


def tolerance(case):
    op = case["op"]
    if op in ("matmul", "head", "attend"):
        # 32-bit sums of exact products of 22 or 23 bit activations: 1e-7 to
        # 5e-7 off the 64-bit result; a pick differs where two logits tie
        return {"rel": 2e-6, "max": 4e-5, "differ": 0.01 if op == "head" else 0.0}
    # Through a layer a value of the cache may round the other way: a half's
    # last bit, or a q8_0 quant or factor, and what reads it moves with it
    # (2e-5 and 4e-5 of the result off 64 bits after two layers).
    if case["form"] == "q8":
        return {"rel": 2e-4, "max": 1e-2, "differ": 0.005}
    return {"rel": 1e-4, "max": 4e-3, "differ": 0.0}


# ---- the same in 64 bits ---------------------------------------------------
def _values(kind, rows, cols, blob):
    """The tensor's values, (rows, cols) in float64."""
    per, size = BLOCK[kind]
    b = blob.reshape(-1, size)
    n = b.shape[0]

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()

    def bits(at):  # 32 fifth bits, little-endian
        h = b[:, at:at + 4].to(torch.int32)
        return ((h[:, torch.arange(32, device=b.device) // 8] >> (torch.arange(32, device=b.device) % 8)) & 1) << 4

    if kind == "q8_0":
        v = half(0) * b[:, 2:34].contiguous().view(torch.int8).double()
    elif per == 32:
        at = {"q4_0": 2, "q4_1": 4, "q5_0": 6, "q5_1": 8}[kind]
        q = b[:, at:at + 16].to(torch.int32)
        q = torch.cat([q & 15, q >> 4], 1)
        if kind == "q5_0":
            q = q | bits(2)
        elif kind == "q5_1":
            q = q | bits(4)
        if kind in ("q4_0", "q5_0"):
            v = half(0) * (q - (8 if kind == "q4_0" else 16)).double()
        else:
            v = half(0) * q.double() + half(2)
    elif kind in ("q4_k", "q5_k"):
        s = b[:, 4:16].to(torch.int32)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1)
        m = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        q = b[:, size - 128:].to(torch.int32).reshape(n, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(n, 8, 32)
        if kind == "q5_k":
            h = b[:, 16:48].to(torch.int32).reshape(n, 1, 32)
            q = q | (((h >> torch.arange(8, device=b.device).reshape(1, 8, 1)) & 1) << 4)
        v = (half(0) * sc.double())[..., None] * q.double() - (half(2) * m.double())[..., None]
    else:
        ql, qh = b[:, :128].to(torch.int32).reshape(n, 2, 2, 32), b[:, 128:192].to(torch.int32).reshape(n, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)  # quarters 0..3 of each half
        hi = (qh >> torch.tensor([0, 2, 4, 6], device=b.device, dtype=torch.int32).reshape(1, 1, 4, 1)) & 3
        sc = b[:, 192:208].contiguous().view(torch.int8).double().reshape(n, 2, 4, 2, 1)
        v = half(208).reshape(n, 1, 1, 1, 1) * sc * ((lo | (hi << 4)) - 32).double().reshape(n, 2, 4, 2, 16)
    return v.reshape(rows, cols)


def _times(kind, rows, cols, blob, x):
    """x (tokens, cols) through the tensor, 4096 rows at a time."""
    rb = _bytes(kind, 1, cols)
    return torch.cat([x @ _values(kind, min(4096, rows - r), cols, blob[r * rb:min(rows, r + 4096) * rb]).T.contiguous()
                      for r in range(0, rows, 4096)], 1)


def _norm(x, gain):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * gain.double()


def _attend(q, k, v, live):
    """q (tokens, kv heads, group, d) over k, v (keys, kv heads, d); live (tokens, keys) or None."""
    s = torch.matmul(q.transpose(0, 1).reshape(k.shape[1], -1, q.shape[-1]), k.permute(1, 2, 0).contiguous())
    s = s.reshape(k.shape[1], q.shape[0], q.shape[2], -1) / math.sqrt(q.shape[-1])
    if live is not None:
        s = s.masked_fill(~live[None, :, None, :], -math.inf)
    p = torch.softmax(s, -1)
    o = torch.matmul(p.reshape(k.shape[1], -1, p.shape[-1]), v.permute(1, 0, 2).contiguous())
    return o.reshape(k.shape[1], q.shape[0], q.shape[2], -1).transpose(0, 1)


def _read(form, cache, kv_heads, d):
    """Cache rows as float64 (cells, kv heads, d)."""
    kvw = kv_heads * d
    if form == "f16":
        return cache.double().reshape(-1, kv_heads, d)
    q = cache[:, :kvw // 2].contiguous().view(torch.int8).double().reshape(-1, kvw // 32, 32)
    f = cache[:, kvw // 2:kvw // 2 + kvw // 32].double()
    return (q * f[..., None]).reshape(-1, kv_heads, d)


def _stored(form, x):
    """What a cache gives back for the float64 rows x."""
    if form == "f16":
        return x.half().double()
    y = x.reshape(x.shape[0], -1, 32)
    amax = y.abs().amax(-1, keepdim=True)
    q = torch.trunc(y * (127.0 / amax) + torch.where(y < 0, -0.5, 0.5)).clamp(-127, 127)
    return (q * (amax / 127.0).half().double()).reshape(x.shape)


def _rope(x, pos):
    """Adjacent pairs of x (tokens, heads, d) rotated; the angle is a float32 product."""
    d = x.shape[-1]
    step = torch.exp(-2.0 * torch.arange(d // 2, device=x.device).double() / d * math.log(ROPE_BASE)).float()
    a = (pos.float()[:, None] * step).double()
    c, s = a.cos()[:, None], a.sin()[:, None]
    x0, x1 = x[..., 0::2], x[..., 1::2]
    return torch.stack([x0 * c - x1 * s, x0 * s + x1 * c], -1).reshape(x.shape)


def _exact_layer(case, host, x, k, v, pos, cells, chunk):
    """The layer in 64 bits; k, v (cells, kv heads, d) float64 updated in place;
    cells (sequences, positions): where each position lies."""
    t, h, kvh, d = x.shape[0], case["heads"], case["kv_heads"], case["head_dim"]
    xn = _norm(x, host["attn_norm"])
    q = _rope(_times(*host["wq"], xn).reshape(t, h, d), pos)
    kn = _rope(_times(*host["wk"], xn).reshape(t, kvh, d), pos)
    vn = _times(*host["wv"], xn)
    at = cells[0 if chunk else torch.arange(t, device=x.device), pos.long()]
    k[at] = _stored(case["form"], kn.reshape(t, -1)).reshape(t, kvh, d)
    v[at] = _stored(case["form"], vn).reshape(t, kvh, d)
    q = q.reshape(t, kvh, h // kvh, d)
    if chunk:
        n = int(pos.max()) + 1
        rows = cells[0, :n]
        out = []
        for a in range(0, t, 128):
            live = torch.arange(n, device=x.device)[None] <= pos[a:a + 128, None]
            out.append(_attend(q[a:a + 128], k[rows], v[rows], live))
        o = torch.cat(out)
    else:
        o = torch.cat([_attend(q[i:i + 1], k[cells[i, :int(pos[i]) + 1]], v[cells[i, :int(pos[i]) + 1]], None)
                       for i in range(t)])
    x = x + _times(*host["wo"], o.reshape(t, -1))
    xn = _norm(x, host["ffn_norm"])
    gate = _times(*host["gate"], xn)
    return x + _times(*host["down"], gate * torch.sigmoid(gate) * _times(*host["up"], xn))


def exact(case, seed):
    g = _Inputs(seed)
    op = case["op"]
    if op in ("matmul", "head"):
        blobs = [g.blob(case["kind"], case["rows"], case["cols"]) for _ in range(case.get("mats", 1))]
        x = g.normal(case["tokens"] * case["cols"]).double().reshape(case["tokens"], -1)
        if op == "head":
            x = _norm(x, g.normal(case["cols"], mean=1.0, std=0.1))
            return dict(logits=_times(case["kind"], case["rows"], case["cols"], blobs[0], x).reshape(-1), pick=None)
        aux = g.normal(case["rows"] * (1 if case["epi"] == "bias" else case["tokens"])).double()
        out = []
        for b in blobs:
            y = _times(case["kind"], case["rows"], case["cols"], b, x)
            if case["epi"] == "bias":
                y = y + aux
            elif case["epi"] == "glu":
                y = y * torch.sigmoid(y) * aux.reshape(y.shape)
            out.append(y.reshape(-1))
        return torch.cat(out)
    kvh, d = case["kv_heads"], case["head_dim"]
    if op == "attend":
        q = g.normal(case["heads"] * d).double().reshape(1, kvh, -1, d)
        k, v = (_read(case["form"], g.cache(case["form"], case["count"], kvh * d), kvh, d) for _ in range(2))
        return _attend(q, k, v, None).reshape(-1)
    f16 = case["form"] == "f16"

    def shown(cache, like):
        return cache.reshape(like) if f16 else None

    if op == "layer":
        host, x, k, v, pos, index = _layer_state(case, g)
        shape = k.shape
        k, v = (_read(case["form"], c, kvh, d) for c in (k, v))
        seqs = 1 if case["chunk"] else case["tokens"]
        cells = torch.arange(seqs * case["context"], device="cuda").reshape(seqs, -1) if index is None else index.long()
        y = _exact_layer(case, host, x.double(), k, v, pos, cells, case["chunk"])
        return dict(x=y, k=shown(k, shape), v=shown(v, shape))
    hosts, emb, gain, head, ids, caches = _session_inputs(case, g)
    prompt = case["mode"] == "prompt"
    x = emb[ids.long()].double()
    n = x.shape[0]
    pos = torch.arange(n, device="cuda", dtype=torch.int32) if prompt else torch.full((n,), case["prompt"],
                                                                                      dtype=torch.int32, device="cuda")
    cells = torch.arange(case["batch"] * case["context"], device="cuda").reshape(case["batch"], -1)
    ks, vs = [], []
    for host, (k, v) in zip(hosts, caches):
        shape = k.numel()
        k, v = (_read(case["form"], c, kvh, d) for c in (k, v))
        x = _exact_layer(case, host, x, k, v, pos, cells, prompt)
        ks.append(shown(k, shape))
        vs.append(shown(v, shape))
    if prompt:
        x = x[-1:]
    return dict(logits=_times(*head, _norm(x, gain)).reshape(-1), x=x.reshape(-1), k=ks, v=vs)
