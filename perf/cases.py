"""The calls whose speed counts: what a user of this framework has it do, over
the range of sizes it is used at.

The single layers go through the kernel API (spbitnet_amd.kernels and the C ABI
of include/spbitnet_amd.h), the whole model through InferenceEngine and
BatchInferenceEngine.  Sizes are those of the BitNet b1.58 2B-4T shape
(ModelConfig.bitnet_b158_2b4t: hidden 2560, FFN 6912, 20 / 5 heads of 128,
vocabulary 128256, 30 layers) and ragged ones around them.

listed() and draw() give the cases, prepare() what a program holds before the
call, run() one pass, work() what the pass cannot do without, exact() its
result in 64 bits and tolerance() how far another correct implementation at the
same precision would be from it.
"""
from __future__ import annotations

import math

import torch

from spbitnet_amd import _lib
from spbitnet_amd import kernels as K
from spbitnet_amd.model import (PROJECTIONS, BatchInferenceEngine, InferenceEngine, Model,
                                ModelConfig, SparseLinear, TransformerLayer)

DEV = "cuda"
HALF = {"f16": torch.float16, "bf16": torch.bfloat16}


# ---- cases ------------------------------------------------------------------

def listed():
    return [
        # one key / value projection of a decode step: the smallest call, all latency
        dict(name="gemv_640x2560", kind="gemv", rows=640, cols=2560),
        # 80 stacked FFN matrices in one call, 267 MB that no cache holds: weights
        # streamed from HBM once, what a large ternary layer costs
        dict(name="gemv_552960x2560", kind="gemv", rows=552960, cols=2560),
        # one FFN layer of a decode step: absmax, int8 quantisation, product and
        # dequantisation in one call
        dict(name="bitlinear_bf16_2560x6912", kind="bitlinear", rows=2560, cols=6912,
             dtype="bf16"),
        # the reference's own pair of calls (absmax, fused layer) in fp16, on a
        # shape whose columns are no multiple of 128
        dict(name="bitlinear_f16_3002x1900", kind="fused", rows=3002, cols=1900, dtype="f16"),
        # a batch of decoding sequences through one layer
        dict(name="gemm_n21_2560x6912", kind="gemm", rows=2560, cols=6912, n=21),
        # a prompt of 2048 tokens through the stacked gate / up projections
        dict(name="gemm_n2048_13824x2560", kind="gemm", rows=13824, cols=2560, n=2048),
        # the cuSPARSELt drop-in: arbitrary int8 weights pruned to 2:4, 256 tokens
        dict(name="sparse_i8_n256_6912x2560", kind="sparse_i8", rows=6912, cols=2560, n=256),
        # attention of one decode step op by op (scores, softmax, output), fp16 cache
        dict(name="attention_f16_seq2500", kind="attention", heads=20, kv_heads=5, head_dim=128,
             seq=2500, max_seq=4096, dtype="f16"),
        # the LM head of one decode step
        dict(name="head_bf16_128256x2560", kind="head", rows=128256, cols=2560, dtype="bf16"),
        # a short question, one sequence: a 33-token prompt, 40 greedy tokens
        dict(name="decode_b1_p33", kind="engine", layers=30, prompt=33, new=40, max_seq=1024),
        # a long prompt, one sequence: 2048 tokens, then the first answer tokens
        dict(name="prefill_b1_p2048", kind="engine", layers=30, prompt=2048, new=2, max_seq=4096),
        # serving: 32 sequences with prompts of unequal length, decoded together
        dict(name="batch32_p100", kind="batch", layers=30, batch=32, prompt=100, new=32,
             max_seq=1024),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# (rows, cols) of the model's projections, single and stacked
_SHAPES = [(640, 2560), (2560, 2560), (3840, 2560), (6912, 2560), (13824, 2560), (2560, 6912)]


def _shape(rng, lo, hi, step):
    """A projection's shape, or a ragged one: rows of any size, cols a multiple of step."""
    if rng.random() < 0.5:
        return rng.choice(_SHAPES)
    return _log(rng, lo, hi), max(step, _log(rng, 256, 8192) // step * step)


def draw(rng):
    kind = rng.choice(["gemv", "bitlinear", "fused", "gemm", "gemm", "sparse_i8", "attention",
                       "head", "engine", "engine", "batch"])
    dtype = rng.choice(["f16", "bf16"])
    if kind == "gemv":
        rows, cols = _shape(rng, 64, 16000, 128)
        return dict(kind=kind, rows=min(rows * _log(rng, 1, 80), 552960 * 2560 // cols), cols=cols)
    if kind in ("bitlinear", "fused"):
        rows, cols = _shape(rng, 64, 16000, 4)
        return dict(kind=kind, rows=rows, cols=cols, dtype=dtype)
    if kind in ("gemm", "sparse_i8"):
        rows, cols = _shape(rng, 64, 14000, 128 if kind == "gemm" else 16)
        n = min(_log(rng, 1, 4096), max(1, 13824 * 2560 * 2048 // (rows * cols)))
        return dict(kind=kind, rows=rows, cols=cols, n=n)
    if kind == "attention":
        heads, kv = rng.choice([(20, 5), (16, 16), (32, 8), (8, 1)])
        max_seq = rng.choice([1024, 4096, 8192])
        return dict(kind=kind, heads=heads, kv_heads=kv, head_dim=rng.choice([64, 128]),
                    seq=_log(rng, 1, max_seq), max_seq=max_seq, dtype=dtype)
    if kind == "head":
        return dict(kind=kind, rows=_log(rng, 4000, 128256), cols=_log(rng, 512, 2560) // 8 * 8,
                    dtype=dtype)
    layers = _log(rng, 1, 30)
    if kind == "engine":
        prompt = _log(rng, 1, 2048)
        return dict(kind=kind, layers=layers, prompt=prompt, new=rng.randint(1, 12),
                    max_seq=rng.choice([2560, 4096]))
    prompt = _log(rng, 8, 100)
    return dict(kind=kind, layers=layers, batch=rng.randint(2, 32), prompt=prompt,
                new=rng.randint(2, 16), max_seq=rng.choice([256, 1024]))


# ---- inputs -----------------------------------------------------------------

_PAIRS = (0x3, 0x5, 0x6, 0x9, 0xA, 0xC)  # the six bitmaps with two of four columns kept


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)


def _words(parts, bits):
    """[rows][k] small values -> int32 [rows][ceil(k / per)], `bits` bits each, first lowest."""
    per = 32 // bits
    rows, k = parts.shape
    pad = -k % per
    if pad:
        parts = torch.nn.functional.pad(parts, (0, pad))
    parts = parts.view(rows, -1, per)
    out = torch.zeros(parts.shape[:2], dtype=torch.int32, device=parts.device)
    for i in range(per):
        out |= parts[:, :, i].to(torch.int32) << (bits * i)
    return out


def _packed(rows, cols, g):
    """Random 2:4 sparse-ternary weights in the packed format: (meta, values)."""
    lut = torch.tensor(_PAIRS, dtype=torch.uint8, device=DEV)
    meta, values = [], []
    for r0 in range(0, rows, 65536):
        r = min(65536, rows - r0)
        pick = torch.randint(0, 6, (r, cols // 4), dtype=torch.uint8, device=DEV, generator=g)
        meta.append(_words(lut[pick.int()], 4))
        signs = torch.randint(0, 4, (r, cols // 4), dtype=torch.uint8, device=DEV, generator=g)
        values.append(_words(signs, 2))
    return torch.cat(meta), torch.cat(values)


def _dense(meta, values, cols):
    """The dense {-1, 0, +1} matrix, int8, of packed weights."""
    rows, groups = meta.shape[0], cols // 4
    sh = torch.arange(8, device=DEV, dtype=torch.int32) * 4
    nib = ((meta[:, :, None] >> sh) & 15).reshape(rows, -1)[:, :groups]
    sh = torch.arange(16, device=DEV, dtype=torch.int32) * 2
    sg = ((values[:, :, None] >> sh) & 3).reshape(rows, -1)[:, :groups]
    out = torch.zeros((rows, groups, 4), dtype=torch.int8, device=DEV)
    seen = torch.zeros_like(nib)
    for j in range(4):
        kept = (nib >> j) & 1
        sign = (sg >> seen.clamp(max=1)) & 1  # a kept column takes the next sign bit, 1 = -1
        out[:, :, j] = (kept * (1 - 2 * sign)).to(torch.int8)
        seen += kept
    return out.view(rows, cols)


def _int8_rows(n, cols, g):
    """Quantised activations as absmax quantisation leaves them: normal, largest 127."""
    x = torch.randn((n, cols), device=DEV, generator=g)
    return (x * (127.0 / x.abs().amax(1, keepdim=True))).round().clamp(-128, 127).to(torch.int8)


def _config(c):
    m = ModelConfig.bitnet_b158_2b4t(c["max_seq"])
    m.num_hidden_layers = c["layers"]
    return m


def _model(c, seed):
    """A model with the activation scales of a trained one: every projection keeps
    its input's variance, attention scores spread over a few units, each layer adds
    a little to the residual stream, and the head is sure of its next token (so
    that greedy tokens do not hang on the last bit of a logit)."""
    g = _gen(seed)
    cfg = _config(c)
    H, I = cfg.hidden_size, cfg.intermediate_size
    kvd = cfg.num_key_value_heads * cfg.head_dim
    shapes = {"q_proj": (H, H), "k_proj": (kvd, H), "v_proj": (kvd, H), "o_proj": (H, H),
              "gate_proj": (I, H), "up_proj": (I, H), "down_proj": (H, I)}
    added = 0.08 / math.sqrt(2 * cfg.num_hidden_layers)  # std of what a block adds; embedding 0.02
    gamma = {n: 1.0 / math.sqrt(k / 2) for n, (_, k) in shapes.items()}
    gamma["q_proj"] *= 1.5
    gamma["down_proj"] *= added

    def norm(n, scale=1.0):
        return scale * (1 + 0.1 * torch.randn(n, device=DEV, generator=g))

    layers = []
    for _ in range(cfg.num_hidden_layers):
        lin = {}
        for name in PROJECTIONS:
            rows, cols = shapes[name]
            meta, values = _packed(rows, cols, g)
            lin[name] = SparseLinear(meta, values, float(torch.tensor(gamma[name])), rows, cols,
                                     meta.shape[1], values.shape[1])
        layers.append(TransformerLayer(**lin, input_layernorm=norm(H),
                                       post_attention_layernorm=norm(H),
                                       attn_sub_norm=norm(H, added), ffn_sub_norm=norm(I)))
    embed = (0.02 * torch.randn((cfg.vocab_size, H), device=DEV, generator=g)).to(torch.bfloat16)
    return Model(cfg, layers, embed, norm(H), lm_head_weight=embed.roll(7, 0).contiguous())


def _prompts(c, seed):
    """Prompts of c["prompt"] tokens; in a batch, of 0.5 to 1.5 times that many."""
    g = torch.Generator().manual_seed(int(seed) % (1 << 62) + 1)
    if c["kind"] == "engine":
        lens = [c["prompt"]]
    else:
        lens = [max(1, int(c["prompt"] * (0.5 + i / max(1, c["batch"] - 1))))
                for i in range(c["batch"])]
    vocab = _config(c).vocab_size
    return [torch.randint(0, vocab, (n,), generator=g).tolist() for n in lens]


def _inputs(c, seed):
    g = _gen(seed)
    if c["kind"] in ("gemv", "gemm"):
        meta, values = _packed(c["rows"], c["cols"], g)
        return dict(meta=meta, values=values, x=_int8_rows(c.get("n", 1), c["cols"], g))
    if c["kind"] in ("bitlinear", "fused"):
        meta, values = _packed(c["rows"], c["cols"], g)
        x = torch.randn(c["cols"], device=DEV, generator=g).to(HALF[c["dtype"]])
        return dict(meta=meta, values=values, x=x, gamma=1.0 / math.sqrt(c["cols"] / 2))
    if c["kind"] == "sparse_i8":
        w = torch.randint(-127, 128, (c["rows"], c["cols"]), dtype=torch.int8, device=DEV,
                          generator=g)
        return dict(w=w, x=_int8_rows(c["n"], c["cols"], g))
    if c["kind"] == "attention":
        shape = (c["kv_heads"], c["max_seq"], c["head_dim"])
        half = HALF[c["dtype"]]
        q = 1.5 * torch.randn((c["heads"], c["head_dim"]), device=DEV, generator=g)
        return dict(q=q.to(half), k=torch.randn(shape, device=DEV, generator=g).to(half),
                    v=torch.randn(shape, device=DEV, generator=g).to(half))
    half = HALF[c["dtype"]]
    w = torch.randn((c["rows"], c["cols"]), device=DEV, generator=g).mul_(0.02).to(half)
    return dict(w=w, x=torch.randn(c["cols"], device=DEV, generator=g).to(half))


def prepare(case, seed):
    c = case
    if c["kind"] in ("engine", "batch"):
        model = _model(c, seed)
        if c["kind"] == "engine":
            eng = InferenceEngine(model, max_seq=c["max_seq"])
        else:
            eng = BatchInferenceEngine(model, max_seq=c["max_seq"], batch=c["batch"])
        return dict(case=c, engine=eng, prompts=_prompts(c, seed))
    s = _inputs(c, seed)
    s["case"] = c
    if c["kind"] == "gemv":
        s["y"] = torch.empty(c["rows"], dtype=torch.int32, device=DEV)
    elif c["kind"] in ("bitlinear", "fused"):
        s["y"] = torch.empty(c["rows"], dtype=HALF[c["dtype"]], device=DEV)
        s["absmax"] = torch.empty(1, dtype=torch.float32, device=DEV)
        s["workspace"] = torch.empty(K.bitlinear_workspace_size(c["cols"]), dtype=torch.uint8,
                                     device=DEV)
    elif c["kind"] in ("gemm", "sparse_i8"):
        s["y"] = torch.empty((c["n"], c["rows"]), dtype=torch.int32, device=DEV)
        if c["kind"] == "sparse_i8":  # weights pruned and compressed once, as at load time
            s["op"] = K.CuSparseLtGemm(c["rows"], c["cols"], c["n"])
            s["op"].prepare(s["w"])
    elif c["kind"] == "attention":
        s["scores"] = torch.empty((c["heads"], c["max_seq"]), dtype=torch.float32, device=DEV)
        s["y"] = torch.empty((c["heads"], c["head_dim"]), dtype=HALF[c["dtype"]], device=DEV)
    else:
        s["y"] = torch.empty(c["rows"], dtype=torch.float32, device=DEV)
    return s


# ---- one pass ---------------------------------------------------------------

def _call(name, *args):
    _lib.check(getattr(_lib.load(), name)(*args), name)


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "engine":
        tokens = s["engine"].generate(s["prompts"][0], c["new"], stop_at_eos=False)
        # the token after the last one: its whole distribution, for a user's sampler
        logits = s["engine"].forward(tokens[-1])
        return dict(tokens=torch.tensor(tokens), logits=logits)
    if kind == "batch":
        tokens = s["engine"].generate(s["prompts"], c["new"], stop_at_eos=False)
        return dict(tokens=torch.tensor(tokens), logits=s["engine"].last_logits())
    if kind == "gemv":
        K.sparse_ternary_gemv_gpu(s["meta"], s["values"], s["x"], s["y"], c["rows"], c["cols"],
                                  s["meta"].shape[1], s["values"].shape[1])
        return s["y"]
    if kind == "bitlinear":
        K.bitlinear_gpu(s["meta"], s["values"], s["x"], s["y"], s["gamma"], c["rows"], c["cols"],
                        s["meta"].shape[1], s["values"].shape[1], s["workspace"])
        return s["y"]
    if kind == "fused":
        K.absmax_reduce_gpu(s["x"], s["absmax"], c["cols"])
        K.fused_sparse_bitlinear_gpu(s["meta"], s["values"], s["x"], s["y"], s["absmax"],
                                     s["gamma"], c["rows"], c["cols"], s["meta"].shape[1],
                                     s["values"].shape[1])
        return s["y"]
    if kind == "gemm":
        K.sparse_ternary_gemm_gpu(s["meta"], s["values"], s["x"], s["y"], c["rows"], c["cols"],
                                  c["n"], s["meta"].shape[1], s["values"].shape[1])
        return s["y"]
    if kind == "sparse_i8":
        s["op"].execute(s["x"], s["y"])
        return s["y"]
    stream = torch.cuda.current_stream().cuda_stream or None
    t = c["dtype"]
    if kind == "head":
        _call(f"spb_gemv_{t}", s["w"].data_ptr(), s["x"].data_ptr(), s["y"].data_ptr(), c["rows"],
              c["cols"], stream)
        return s["y"]
    nh, nkv, hd, seq = c["heads"], c["kv_heads"], c["head_dim"], c["seq"]
    sc, out = s["scores"].data_ptr(), s["y"].data_ptr()
    _call(f"spb_attention_scores_{t}", s["q"].data_ptr(), s["k"].data_ptr(), sc, nh, nkv, hd,
          c["max_seq"], seq, 1.0 / math.sqrt(hd), stream)
    _call("spb_softmax", sc, nh, c["max_seq"], seq, stream)
    _call(f"spb_attention_output_{t}", sc, s["v"].data_ptr(), out, nh, nkv, hd, c["max_seq"], seq,
          stream)
    return dict(out=s["y"], weights=s["scores"][:, :seq])


# ---- what a pass cannot do without --------------------------------------------

def _packed_bytes(rows, cols):
    return 4 * rows * (-(-cols // 32) + -(-cols // 64))


def work(case):
    c = case
    kind = c["kind"]
    if kind in ("engine", "batch"):
        cfg = _config(c)
        H, I, V, L = cfg.hidden_size, cfg.intermediate_size, cfg.vocab_size, c["layers"]
        params = L * (H * (2 * H + 2 * 640) + 3 * H * I)  # dense count, half of them non-zero
        packed, head = params * 3 // 16, 2 * H * V
        lens = [len(p) for p in _prompts(c, 0)]
        steps = c["new"] + (1 if kind == "engine" else 0)
        kv = L * 2 * 640 * 2  # bytes per position
        flops = bytes_ = 0
        for n in lens:
            flops += params * (n - 1 + steps)
            flops += L * 4 * H * sum(range(1, n + steps))
            flops += 2 * H * V * steps
            bytes_ += kv * (n - 1 + sum(range(n, n + steps)))
        prefill = 1 if max(lens) > 1 else 0
        return dict(bytes=bytes_ + (steps + prefill) * packed + steps * head
                    + 4 * V * len(lens), flops=flops)
    if kind == "attention":
        size = 2 * (2 * c["kv_heads"] * c["seq"] * c["head_dim"]
                    + 2 * c["heads"] * c["head_dim"]) + 4 * c["heads"] * c["seq"]
        return dict(bytes=size, flops=4 * c["heads"] * c["seq"] * c["head_dim"])
    rows, cols, n = c["rows"], c["cols"], c.get("n", 1)
    if kind == "head":
        return dict(bytes=2 * rows * cols + 2 * cols + 4 * rows, flops=2 * rows * cols)
    flops = rows * cols * n  # half of the columns are kept, a multiply and an add each
    if kind == "sparse_i8":
        weights = rows * cols * 5 // 8  # kept int8 values and a 2-bit index each
        return dict(bytes=weights + n * cols + 4 * n * rows, flops=flops)
    if kind in ("bitlinear", "fused"):
        return dict(bytes=_packed_bytes(rows, cols) + 2 * cols + 2 * rows, flops=flops)
    return dict(bytes=_packed_bytes(rows, cols) + n * cols + 4 * n * rows, flops=flops)


def tolerance(case):
    kind = case["kind"]
    if kind in ("gemv", "gemm", "sparse_i8"):
        return "exact"  # int32 sums of int8 products
    # elsewhere about four times the distance from exact() that was measured
    if kind in ("bitlinear", "fused", "attention"):
        # one rounding to 16 bits at the end: 1.6e-3 in bf16, 2.0e-4 in fp16
        return {"rel": 6.4e-3 if case["dtype"] == "bf16" else 8e-4}
    if kind == "head":
        return {"rel": 1e-6}  # float32 sums of 16-bit products, in any order
    # bf16 activations and int8 quantisation in every layer: one rounding moves
    # many quantised values of the layers after it, so the logits are 0.047 to
    # 0.086 from exact().  Another path that rounds at the same places is nearer,
    # and the tokens are sure.
    return {"rel": 0.03, "differ": 0.01}


# ---- the result in 64 bits ----------------------------------------------------

def _product(w8, x):
    """w8 int8 [rows][cols] times x float64 [n][cols] -> [n][rows], in pieces."""
    step = max(1, (1 << 27) // w8.shape[1])
    return torch.cat([x @ w8[r:r + step].double().T for r in range(0, w8.shape[0], step)], 1)


def _quant64(x):
    a = x.abs().amax(-1, keepdim=True)
    return torch.clamp(torch.round(x * (127.0 / a)), -128, 127), a


def _linear64(w8, gamma, x):
    q, a = _quant64(x)
    return _product(w8, q) * (gamma * a / 127.0)


def _rms64(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


class _Model64:
    """The model's forward pass in float64 over dense weights."""

    def __init__(self, model):
        self.m, self.c = model, model.config
        self.dense = [{p: (_dense(getattr(l, p).meta, getattr(l, p).values, getattr(l, p).cols),
                           getattr(l, p).gamma) for p in PROJECTIONS} for l in model.layers]
        self.head = model.lm_head().double()

    def rope(self, v, pos):
        hd = self.c.head_dim
        i = torch.arange(hd // 2, device=DEV, dtype=torch.float64)
        ang = pos.double()[:, None] / torch.pow(float(self.c.rope_theta), 2.0 * i / hd)
        cs, sn = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
        x0, x1 = v[..., 0::2], v[..., 1::2]
        return torch.stack([x0 * cs - x1 * sn, x0 * sn + x1 * cs], -1).flatten(-2)

    def forward(self, tokens, cache):
        """Appends tokens to the cache; the residual stream of each."""
        c, eps = self.c, self.c.rms_norm_eps
        nh, nkv, hd = c.num_attention_heads, c.num_key_value_heads, c.head_dim
        n0 = cache[0][0].shape[0] if cache else 0
        pos = torch.arange(n0, n0 + len(tokens), device=DEV)
        x = self.m.embed_tokens[torch.tensor(tokens, device=DEV)].double()
        for li, (l, d) in enumerate(zip(self.m.layers, self.dense)):
            h = _rms64(x, l.input_layernorm, eps)
            q = self.rope(_linear64(*d["q_proj"], h).view(-1, nh, hd), pos)
            k = self.rope(_linear64(*d["k_proj"], h).view(-1, nkv, hd), pos)
            v = _linear64(*d["v_proj"], h).view(-1, nkv, hd)
            if li < len(cache):
                k, v = torch.cat([cache[li][0], k]), torch.cat([cache[li][1], v])
                cache[li] = (k, v)
            else:
                cache.append((k, v))
            seen = torch.arange(k.shape[0], device=DEV)[None, :] <= pos[:, None]
            out = []
            for head in range(nh):
                kv = head * nkv // nh
                sc = (q[:, head] @ k[:, kv].T) / math.sqrt(hd)
                out.append(torch.softmax(sc.masked_fill(~seen, -math.inf), -1) @ v[:, kv])
            o = _linear64(*d["o_proj"], torch.cat(out, -1))
            x = x + _rms64(o, l.attn_sub_norm, eps)
            h = _rms64(x, l.post_attention_layernorm, eps)
            m = torch.relu(_linear64(*d["gate_proj"], h)) ** 2 * _linear64(*d["up_proj"], h)
            x = x + _linear64(*d["down_proj"], _rms64(m, l.ffn_sub_norm, eps))
        return x

    def logits(self, x):
        return self.head @ _rms64(x, self.m.final_norm, self.c.rms_norm_eps)

    def generate(self, prompt, new):
        """Greedy tokens, the last step's logits and those of the step after it."""
        cache, tokens, logits = [], [], None
        x = self.forward(prompt, cache)[-1]
        for _ in range(new):
            logits = self.logits(x)
            tokens.append(int(logits.argmax()))
            x = self.forward(tokens[-1:], cache)[-1]
        return tokens, logits, self.logits(x)


def exact(case, seed):
    c = case
    kind = c["kind"]
    if kind == "engine":
        tokens, _, after = _Model64(_model(c, seed)).generate(_prompts(c, seed)[0], c["new"])
        return dict(tokens=torch.tensor(tokens), logits=after)
    if kind == "batch":
        if c["layers"] * c["batch"] * (c["new"] + 2) > 5000:
            return None  # about a minute: the sequences run one after another
        m = _Model64(_model(c, seed))
        got = [m.generate(p, c["new"]) for p in _prompts(c, seed)]
        return dict(tokens=torch.tensor([t for t, _, _ in got]),
                    logits=torch.stack([last for _, last, _ in got]))
    s = _inputs(c, seed)
    if kind in ("gemv", "gemm"):
        step = 65536
        y = torch.cat([_product(_dense(s["meta"][r:r + step], s["values"][r:r + step], c["cols"]),
                                s["x"].double()) for r in range(0, c["rows"], step)], 1)
        return y[0] if kind == "gemv" else y
    if kind in ("bitlinear", "fused"):
        w = _dense(s["meta"], s["values"], c["cols"])
        return _linear64(w, s["gamma"], s["x"].double()[None])[0]
    if kind == "sparse_i8":
        # of each four the two largest by magnitude, the later of equals first
        w = s["w"].view(c["rows"], -1, 4)
        rank = w.abs().int() * 4 + torch.arange(4, device=DEV)
        keep = torch.zeros_like(w, dtype=torch.bool).scatter_(2, rank.topk(2, 2).indices, True)
        return _product((w * keep).view(c["rows"], -1), s["x"].double())
    if kind == "head":
        return torch.cat([p.double() @ s["x"].double() for p in s["w"].split(16384)])
    seq, group = c["seq"], c["heads"] // c["kv_heads"]
    k = s["k"][:, :seq].double().repeat_interleave(group, 0)
    v = s["v"][:, :seq].double().repeat_interleave(group, 0)
    sc = (k * s["q"].double()[:, None]).sum(-1) / math.sqrt(c["head_dim"])
    p = torch.softmax(sc, -1)
    return dict(out=(p[..., None] * v).sum(1), weights=p)
