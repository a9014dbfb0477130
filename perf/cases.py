"""The workloads that the speed of this framework is judged by.

Each case is one piece of a transformer program as a user writes it on the public entry points
(``cpm_kernels_amd.torch`` for whole sequences, ``cpm_kernels_amd.kernels`` for the decode step), in
the layouts the framework's own models use: activations fp16 ``(batch, hidden, seq)``, weights fp16
``(1, out, in)`` quantised per output row inside the int8 products, normalisation and softmax over
dim 1.  Sizes are those of ``bench.py`` and the tests (d_model 4096, 64 heads of 64, d_ff 10240,
batches of 8 x 512 and 16 x 1024 tokens, 32 decode sequences, the 500 x 4096 x 7996 product) and
generic ones around them.

Kinds of a case
    decode      one layer of one decode step: hidden state (batch, hidden), int8 weights, fp16 key/value cache
    linear      one product of activations and a weight, forward or forward + backward, int8 or fp16
    ffn         LayerNorm -> product -> gelu -> product -> residual add, forward or forward + backward
    attention   fp16 scores, T5 position bias, mask, softmax, P x V, forward or forward + backward
    layer       a whole encoder layer, forward: LayerNorm, q/k/v, attention, projection, the ffn
    embedding   token embedding, forward + backward
"""
import math

import torch

import cpm_kernels_amd.kernels as ck
import cpm_kernels_amd.torch as ct

HALF = torch.float16
BUCKETS, MAX_DISTANCE, EPS = 32, 128, 1e-5


def listed():
    return [
        # the smallest step: one sequence of a small model, some thirty launches of a few microseconds each
        dict(name="decode_1x1024", kind="decode", batch=1, hidden=1024, heads=16, ff=2560, cache=128, pos=100),
        # a serving batch of the large model in the middle of its cache: weights and cache stream from memory
        dict(name="decode_32x4096", kind="decode", batch=32, hidden=4096, heads=64, ff=10240, cache=1024, pos=700),
        # short prompts through one projection, both operands with the contraction contiguous
        dict(name="linear_int8_512", kind="linear", batch=1, tokens=512, din=4096, dout=4096, rows=True, int8=True, train=False),
        # the same at the size of a full batch, up-projection of the ffn
        dict(name="linear_int8_4096", kind="linear", batch=1, tokens=4096, din=4096, dout=10240, rows=True, int8=True, train=False),
        # an fp16 product whose sizes fit no tile
        dict(name="linear_fp16_ragged", kind="linear", batch=8, tokens=500, din=4096, dout=7996, rows=False, int8=False, train=False),
        # fine-tuning one projection in fp16: both gradients, the weight's summed over the batch
        dict(name="linear_fp16_train", kind="linear", batch=8, tokens=512, din=4096, dout=4096, rows=False, int8=False, train=True),
        # prefill of the ffn block
        dict(name="ffn_8x512", kind="ffn", batch=8, seq=512, hidden=4096, ff=10240, train=False),
        # a training step of it: gradients of the input, both weights and the norm's parameters
        dict(name="ffn_train_8x512", kind="ffn", batch=8, seq=512, hidden=4096, ff=10240, train=True),
        # attention of a batch whose longest sequence has 500 tokens
        dict(name="attention_16x500", kind="attention", batch=16, heads=64, head=64, seq=500, train=False),
        # attention in training, gradient of the position bias among the results
        dict(name="attention_train_4x512", kind="attention", batch=4, heads=64, head=64, seq=512, train=True),
        # prefill of a whole layer of the large model, the largest pass
        dict(name="layer_16x1024", kind="layer", batch=16, seq=1024, hidden=4096, heads=64, ff=10240),
        # the two ends of a training step that are no products: gather of token rows, scatter of their gradients
        dict(name="embedding_train_8x512", kind="embedding", batch=8, seq=512, hidden=4096, vocab=30000),
    ]


def _log(rng, lo, hi, multiple=1):
    return max(1, round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / multiple)) * multiple


def _drawn(rng):
    # (the int8 products take sizes that are multiples of 4, the fp16 ones and the additions even ones)
    kind = rng.choice(["decode", "decode", "linear", "linear", "linear", "ffn", "ffn", "attention", "attention", "layer", "embedding"])
    if kind == "decode":
        heads = _log(rng, 8, 64, 2)
        cache = _log(rng, 32, 2048)
        return dict(kind=kind, batch=_log(rng, 1, 32), hidden=64 * heads, heads=heads, ff=_log(rng, 128 * heads, 256 * heads, 64), cache=cache,
                    pos=rng.randrange(cache // 2, cache))
    if kind == "linear":
        return dict(kind=kind, batch=_log(rng, 1, 16), tokens=_log(rng, 32, 1024, 4), din=_log(rng, 512, 10240, rng.choice([4, 64, 128])),
                    dout=_log(rng, 512, 10240, rng.choice([4, 64, 128])), rows=rng.random() < 0.4, int8=rng.random() < 0.6, train=rng.random() < 0.5)
    if kind == "ffn":
        hidden = _log(rng, 512, 4096, 64)
        return dict(kind=kind, batch=_log(rng, 1, 16), seq=_log(rng, 32, 1024, 4), hidden=hidden, ff=_log(rng, 2 * hidden, 4 * hidden, 64), train=rng.random() < 0.5)
    if kind == "attention":
        return dict(kind=kind, batch=_log(rng, 1, 16), heads=_log(rng, 8, 64), head=rng.choice([64, 64, 64, 80, 128]), seq=_log(rng, 32, 1024, 2),
                    train=rng.random() < 0.5)
    if kind == "layer":
        heads = _log(rng, 8, 64)
        return dict(kind=kind, batch=_log(rng, 1, 16), seq=_log(rng, 32, 1024, 4), hidden=64 * heads, heads=heads, ff=_log(rng, 128 * heads, 256 * heads, 64))
    return dict(kind=kind, batch=_log(rng, 1, 16), seq=_log(rng, 32, 1024), hidden=_log(rng, 512, 4096, 64), vocab=_log(rng, 2000, 50000))


def _cost(case):
    w = work(case)
    return w["bytes"] / 8e12 + w["flops"] / 2.5e15


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        case = _drawn(rng)
        if _cost(case) <= most:
            return case


# ---- inputs -------------------------------------------------------------------------------------

class _Source:
    """Seeded values on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0):
        return torch.randn(shape, generator=self.gen, device="cuda", dtype=torch.float32).mul_(std).add_(mean).half()

    def integers(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=self.gen, device="cuda", dtype=torch.int32)

    def norm(self, hidden):
        ln = ct.LayerNorm(hidden, eps=EPS, bias=True).half().cuda()
        with torch.no_grad():
            ln.weight.copy_(self.normal(hidden, std=0.1, mean=1.0))
            ln.bias.copy_(self.normal(hidden, std=0.1))
        return ln

    def position(self, heads):
        pe = ct.PositionEmbedding(heads, BUCKETS, MAX_DISTANCE, True).half().cuda()
        with torch.no_grad():
            pe.weight.copy_(self.normal(heads, BUCKETS, std=0.02))
        return pe

    def keep(self, batch, seq):
        """(batch, seq * seq) True where a key may be looked at: sequences of half to all of the length, padded."""
        lens = self.integers(seq // 2, seq + 1, batch)
        keys = torch.arange(seq, device="cuda")[None, :, None] < lens[:, None, None].clamp(min=1)
        return keys.expand(batch, seq, seq).reshape(batch, seq * seq).contiguous()


def _decode_state(c, src):
    b, d, h, ff, length = c["batch"], c["hidden"], c["heads"], c["ff"], c["cache"]
    s = {"case": c, "x": src.normal(b, d)}
    for name, rows, cols in (("q", d, d), ("k", d, d), ("v", d, d), ("o", d, d), ("up", ff, d), ("down", d, ff)):
        w = src.normal(rows, cols, std=0.02)
        scale = torch.empty(rows, dtype=HALF, device="cuda")
        q = torch.empty((rows, cols), dtype=torch.int8, device="cuda")
        ck.gemm_quantize(1, rows, cols, w.data_ptr(), scale.data_ptr(), q.data_ptr(), False, torch.cuda.current_stream().cuda_stream)
        s["w_" + name], s["s_" + name] = q, scale
    for i in (1, 2):
        s["gamma%d" % i], s["beta%d" % i] = src.normal(d, std=0.1, mean=1.0), src.normal(d, std=0.1)
    s["table"] = src.normal(h, BUCKETS, std=0.02)
    s["mapping"] = torch.empty(MAX_DISTANCE, dtype=torch.int32, device="cuda")
    ck.position_embedding_init(BUCKETS, MAX_DISTANCE, s["mapping"].data_ptr(), False, torch.cuda.current_stream().cuda_stream)
    s["keys"], s["values"] = src.normal(b * h, length, d // h), src.normal(b * h, length, d // h)
    s["keep"] = (torch.arange(length, device="cuda") <= c["pos"]).repeat(b, 1).contiguous()

    def buffer(*shape, dtype=HALF):
        return torch.empty(shape, dtype=dtype, device="cuda")
    s.update(h1=buffer(b, d), h2=buffer(b, ff), q8=buffer(b, max(d, ff), dtype=torch.int8), sv=buffer(b), qv=buffer(b, d), kv=buffer(b, d), vv=buffer(b, d),
             bias=buffer(h, length), scores=buffer(b, h * length), ctx=buffer(b, d), y=buffer(b, d), out=buffer(b, d))
    return s


def prepare(case, seed):
    c, src = case, _Source(seed)
    kind = c["kind"]
    if kind == "decode":
        return _decode_state(c, src)
    s = {"case": c}
    if kind == "linear":
        s["x"] = src.normal(*((c["batch"], c["tokens"], c["din"]) if c["rows"] else (c["batch"], c["din"], c["tokens"])))
        s["w"] = src.normal(1, c["dout"], c["din"], std=0.02)
        if c["train"]:
            s["grad"] = src.normal(*((c["batch"], c["tokens"], c["dout"]) if c["rows"] else (c["batch"], c["dout"], c["tokens"])), std=0.05)
            s["x"].requires_grad_()
            s["w"].requires_grad_()
    elif kind in ("ffn", "layer"):
        d, ff = c["hidden"], c["ff"]
        s["x"] = src.normal(c["batch"], d, c["seq"])
        s["ln"], s["w1"], s["w2"] = src.norm(d), src.normal(1, ff, d, std=0.02), src.normal(1, d, ff, std=0.02)
        if kind == "layer":
            s["ln_att"], s["pe"], s["keep"] = src.norm(d), src.position(c["heads"]), src.keep(c["batch"], c["seq"])
            s.update({"w" + n: src.normal(1, d, d, std=0.02) for n in "qkvo"})
        elif c["train"]:
            s["grad"] = src.normal(c["batch"], d, c["seq"], std=0.05)
            for n in ("x", "w1", "w2"):
                s[n].requires_grad_()
    elif kind == "attention":
        shape = (c["batch"] * c["heads"], c["head"], c["seq"])
        s["q"], s["k"], s["v"] = (src.normal(*shape) for _ in range(3))
        s["pe"], s["keep"] = src.position(c["heads"]), src.keep(c["batch"], c["seq"])
        if c["train"]:
            s["grad"] = src.normal(*shape, std=0.05)
            for n in "qkv":
                s[n].requires_grad_()
    else:
        s["emb"] = ct.Embedding(c["vocab"], c["hidden"]).cuda()
        with torch.no_grad():
            s["emb"].weight.copy_(src.normal(c["vocab"], c["hidden"], std=0.02))
        # token ids come with the frequencies of a text: few ids often, most of them seldom
        u = torch.rand((c["batch"], c["seq"]), generator=src.gen, device="cuda", dtype=torch.float64)
        s["ids"] = (torch.exp(u * math.log(c["vocab"])).to(torch.int32) - 1).clamp_(0, c["vocab"] - 1)
        s["grad"] = src.normal(c["batch"], c["hidden"], c["seq"], std=0.05)
    return s


# ---- one pass -----------------------------------------------------------------------------------

def _decode(s):
    c = s["case"]
    b, d, h, ff, length = c["batch"], c["hidden"], c["heads"], c["ff"], c["cache"]
    head = d // h
    st = torch.cuda.current_stream().cuda_stream
    p = {k: v.data_ptr() for k, v in s.items() if isinstance(v, torch.Tensor)}

    def quantized(vec, n):
        ck.gemv_calc_scale(b, n, vec, p["sv"], st)
        ck.gemv_round(b, n, vec, p["sv"], p["q8"], st)

    def product(w, rows, cols, out):
        ck.gemv_broadcast_mat_int8(b, rows, cols, p["s_" + w], p["w_" + w], p["sv"], p["q8"], out, st)

    def norm(x, i):
        ck.layernorm_step(b, d, x, p["h1"], EPS, True, st)
        ck.arith_batch_mul_add(b, d, p["h1"], p["gamma%d" % i], p["beta%d" % i], p["h1"], st)
    norm(p["x"], 1)
    quantized(p["h1"], d)
    product("q", d, d, p["qv"])
    product("k", d, d, p["kv"])
    product("v", d, d, p["vv"])
    ck.copy_data_to_kv(b * h, length, head, p["kv"], p["keys"], c["pos"], st)
    ck.copy_data_to_kv(b * h, length, head, p["vv"], p["values"], c["pos"], st)
    ck.arith_global_scale(b * d, p["qv"], head ** -0.5, p["qv"], st)
    ck.gemv_fp16(b * h, length, head, p["keys"], p["qv"], p["scores"], st)
    ck.position_embedding_step(c["pos"], length, BUCKETS, MAX_DISTANCE, h, p["mapping"], p["table"], p["bias"], False, st)
    ck.arith_batch_add_forward(b, h * length, p["scores"], p["bias"], p["scores"], st)
    ck.mask(b, h, length, p["scores"], p["keep"], float("-inf"), p["scores"], st)
    ck.softmax_step_inplace(b * h, length, p["scores"], st)
    ck.gemv_fp16_transpose(b * h, head, length, p["values"], p["scores"], p["ctx"], st)
    quantized(p["ctx"], d)
    product("o", d, d, p["y"])
    ck.arith_element_add(b, d, p["y"], p["x"], p["y"], st)
    norm(p["y"], 2)
    quantized(p["h1"], d)
    product("up", ff, d, p["h2"])
    ck.gelu_inplace_forward(b, ff, p["h2"], st)
    quantized(p["h2"], ff)
    product("down", d, ff, p["out"])
    ck.arith_element_add(b, d, p["out"], p["y"], p["out"], st)
    return s["out"], s["keys"], s["values"]


def _linear(s, x, w):
    if s["case"]["rows"]:
        return ct.bmm(x, False, w, True, int8=s["case"]["int8"])
    return ct.bmm(w, False, x, False, int8=s["case"]["int8"])


def _ffn(s, x):
    up = ct.bmm(s["w1"], False, s["ln"](x), False, int8=True)
    return ct.element_add(ct.bmm(s["w2"], False, ct.gelu(up), False, int8=True), x)


def _attention(q, k, v, s, batch, heads):
    """q, k, v (batch * heads, head, seq) -> the same shape; scores are (.., key, query)."""
    seq = q.size(2)
    scores = ct.bmm(k, True, ct.global_scale(q, q.size(1) ** -0.5), False, int8=False)
    scores = ct.batched_add(scores.view(batch, heads, seq, seq), s["pe"](seq, seq))
    scores = ct.mask(scores.view(batch, heads, seq * seq), s["keep"], float("-inf"))
    return ct.bmm(v, False, ct.softmax(scores.view(batch * heads, seq, seq)), False, int8=False)


def _layer(s, x):
    c = s["case"]
    b, d, seq, h = c["batch"], c["hidden"], c["seq"], c["heads"]
    hidden = s["ln_att"](x)
    q, k, v = (ct.bmm(s["w" + n], False, hidden, False, int8=True).view(b * h, d // h, seq) for n in "qkv")
    ct.global_scale_inplace(q, (d // h) ** -0.5)
    scores = ct.bmm(k, True, q, False, int8=False)
    ct.batched_add_inplace(scores.view(b, h, seq, seq), s["pe"](seq, seq))
    ct.mask_inplace(scores.view(b, h, seq * seq), s["keep"], float("-inf"))
    ct.softmax_inplace(scores)
    ctx = ct.bmm(v, False, scores, False, int8=False).view(b, d, seq)
    return _ffn(s, ct.element_add(ct.bmm(s["wo"], False, ctx, False, int8=True), x))


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "decode":
        return _decode(s)
    if kind == "embedding":
        out = s["emb"](s["ids"])
        return (out.detach(),) + torch.autograd.grad(out, [s["emb"].weight], s["grad"])
    if not c.get("train"):
        with torch.no_grad():
            if kind == "linear":
                return _linear(s, s["x"], s["w"])
            if kind == "ffn":
                return _ffn(s, s["x"])
            if kind == "layer":
                return _layer(s, s["x"])
            return _attention(s["q"], s["k"], s["v"], s, c["batch"], c["heads"])
    if kind == "linear":
        out, leaves = _linear(s, s["x"], s["w"]), [s["x"], s["w"]]
    elif kind == "ffn":
        out, leaves = _ffn(s, s["x"]), [s["x"], s["w1"], s["w2"], s["ln"].weight, s["ln"].bias]
    else:
        out, leaves = _attention(s["q"], s["k"], s["v"], s, c["batch"], c["heads"]), [s["q"], s["k"], s["v"], s["pe"].weight]
    return (out.detach(),) + torch.autograd.grad(out, leaves, s["grad"])


# ---- what a pass cannot do without -----------------------------------------------------------------
# Every entry point is a call of its own whose result the caller holds, so the bytes of a pass are those of its calls: each call's inputs read once and
# its outputs written once.  fp16 values count two bytes, int8 weights and mask bytes one.

def _linear_work(b, m, k, n, train):
    """An activation batch (b, m, k) and one weight (n, k)."""
    nbytes, flops = 2 * (b * m * k + n * k + b * m * n), 2 * b * m * k * n
    if train:       # the output's gradient and both operands in, both gradients out
        nbytes += 2 * (b * m * n + 2 * b * m * k + 2 * n * k)
    return nbytes, flops * (3 if train else 1)


def _attention_work(b, h, dh, s, train):
    qkv, sc = 2 * b * h * dh * s, 2 * b * h * s * s
    forward = 2 * qkv + (2 * qkv + sc) + (2 * sc + 2 * h * s * s) + 2 * h * s * s + (2 * sc + b * s * s) + 2 * sc + (sc + 2 * qkv)
    flops = 4 * b * h * dh * s * s
    if not train:
        return forward, flops
    # P x V: both operands and the output's gradient in, two gradients out; softmax: output and gradient in, one out; mask;
    # the bias summed over the batch and into its buckets; the scores: both operands and the gradient in, two out; the scale
    backward = (3 * qkv + 2 * sc) + 3 * sc + (2 * sc + b * s * s) + (sc + 2 * h * s * s) + 2 * h * s * s + (4 * qkv + sc) + 2 * qkv
    return forward + backward, 3 * flops


def work(case):
    c = case
    kind = c["kind"]
    if kind == "linear":
        nbytes, flops = _linear_work(c["batch"], c["tokens"], c["din"], c["dout"], c["train"])
    elif kind == "attention":
        nbytes, flops = _attention_work(c["batch"], c["heads"], c["head"], c["seq"], c["train"])
    elif kind in ("ffn", "layer"):
        b, seq, d, ff = c["batch"], c["seq"], c["hidden"], c["ff"]
        t, train = b * seq, c.get("train", False)
        parts = [_linear_work(b, seq, d, ff, train), _linear_work(b, seq, ff, d, train)]
        # norm, gelu, residual add; backward: norm 2 in, 1 out, gelu 2 in, 1 out, and the sum of the residual's two gradients
        parts.append((4 * t * d + 4 * t * ff + 6 * t * d + ((6 * t * d + 6 * t * ff + 6 * t * d) if train else 0), 0))
        if kind == "layer":
            parts += [_linear_work(b, seq, d, d, False)] * 4
            parts += [_attention_work(b, c["heads"], d // c["heads"], seq, False), (4 * t * d + 6 * t * d, 0)]
        nbytes, flops = (sum(p[i] for p in parts) for i in (0, 1))
    elif kind == "decode":
        b, d, h, ff, length = c["batch"], c["hidden"], c["heads"], c["ff"], c["cache"]
        weights = 4 * d * d + 2 * d * ff
        cache = 2 * 2 * b * d * length
        scores = 2 * b * h * length
        nbytes = weights + cache + 7 * scores + 2 * b * (30 * d + 6 * ff)
        flops = 2 * b * weights + 4 * b * d * length
    else:
        t, d = c["batch"] * c["seq"], c["hidden"]
        # rows gathered and written; gradient read, the weight's gradient, mostly zeros, written whole
        nbytes, flops = 4 * t * d + 2 * t * d + 2 * c["vocab"] * d + 4 * t, t * d
    return {"bytes": nbytes, "flops": flops}


# Four times the difference between a pass and the same pass with every norm, softmax, gelu, addition and fp16 product computed in float64 and rounded
# once (products of int8 values are exact either way).  Where a normalised or activated tensor is quantised afterwards, a last-bit difference of it moves
# some values by one int8 step, which is what the larger numbers are.

def tolerance(case):
    kind, train = case["kind"], case.get("train", False)
    if kind == "linear":                    # seen: int8 2.1e-4; fp16 1.4e-5, the weight's gradient summed over the batch 3.6e-4
        return {"rel": 1e-3 if case["int8"] else 1.5e-3}
    if kind == "attention":                 # seen: 6.0e-4 (gradient of the position bias), 4.7e-4 (of q and k)
        return {"rel": 2.5e-3}
    if kind == "ffn":                       # seen: 7.6e-3 forward, 9.6e-3 backward
        return {"rel": 4e-2 if train else 3e-2}
    if kind == "layer":                     # seen: 7.7e-3
        return {"rel": 3e-2}
    if kind == "decode":                    # seen: 3.9e-3
        return {"rel": 1.6e-2}
    return {"rel": 8e-4}                    # embedding, seen: 2.0e-4 (the gathered rows are copies)
