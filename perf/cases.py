"""The work whose speed this framework is judged by: its public calls, over the sizes and options they are used with.

Three groups, each through the Python binding's own calls:

* linear: one projection of a layer on f32 activations (``quantize_q8`` and ``matvec_q`` / ``matmul_q``, or
  ``matvec_ref`` for an unquantized matrix), from one decoded token to a stacked prompt;
* pick: the next token from a final hidden state (Exact Shortlist Head and ``sample``) or from full logits;
* prompt / reply: a ``Decoder``: a prompt from its first token to its logits, and a chat turn on a kept context (its
  tokens, then greedy steps replayed from a HIP graph, as a program that serves one user does).

Weights, activations and shapes follow the repository's benchmark and tests (codes uniform over their range, scales
|N(0, 0.02)| over the code range, activations N(0, 1), a final hidden state N(0, 0.5^2)); the others are generic.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

QK = 32


def _package():
    """The framework's package: quanta.cpp_amd/ is not an importable name, so it is loaded by path."""
    if "quanta_cpp_amd" not in sys.modules:
        where = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "quanta.cpp_amd")
        spec = importlib.util.spec_from_file_location("quanta_cpp_amd", os.path.join(where, "__init__.py"),
                                                      submodule_search_locations=[where])
        module = importlib.util.module_from_spec(spec)
        sys.modules["quanta_cpp_amd"] = module
        spec.loader.exec_module(module)
    import quanta_cpp_amd.qnt as qnt
    return sys.modules["quanta_cpp_amd"], qnt


# ------------------------------------------------------------------------------------------------ the cases

def _linear(name, weights, rows, cols, tokens):
    return {"name": name, "kind": "linear", "weights": weights, "rows": rows, "cols": cols, "tokens": tokens}


# Decoder shapes: the benchmark model's widths, and twice-as-wide heads (head_dim 128) at generic widths.
_SHAPES = {"h64": (896, 14, 2, 64, 4864), "h128": (1536, 12, 2, 128, 8960), "narrow": (256, 4, 1, 64, 512)}


def _decoder(name, kind, **kw):
    c = {"name": name, "kind": kind, "shape": "h64", "layers": 2, "vocab": 4096, "weights": "q4mix", "kv_f32": False,
         "hadamard": False, "stack": 512, "context": 0, "tokens": 32, "steps": 0}
    c.update(kw)
    return c


def listed():
    return [
        # The smallest call: one decoded token through an attention projection.
        _linear("linear_q8_1", "q8", 896, 896, 1),
        # A short user turn through the MLP's gate projection: a ragged handful of 16-token tiles.
        _linear("linear_q4_77", "q4", 4864, 896, 77),
        # A stacked prompt through the MLP's down projection: long rows.
        _linear("linear_q4_512", "q4", 896, 4864, 512),
        # A wide 4-bit projection of a larger model, with a ragged batch of tokens.
        _linear("linear_q4_wide_300", "q4", 4096, 14336, 300),
        # An unquantized model (the exporter's default): one decoded token through an f16 projection.
        _linear("linear_f16_1", "f16", 4864, 896, 1),
        # Chat's next token with the session's default sampler: shortlist head with the history as must ids, then the
        # draw.
        {"name": "pick_shortlist", "kind": "pick", "vocab": 151936, "dim": 896, "top_k": 20, "history": 300,
         "top_p": 0.8},
        # The same draw over full logits (a model without the shortlist tensors).
        {"name": "pick_full", "kind": "sample", "vocab": 151936, "top_k": 20, "history": 300, "top_p": 0.8},
        # The benchmark's whole model: its 512-token prompt, one stack.
        _decoder("prompt_512", "prompt", layers=24, vocab=151936, tokens=512),
        # The benchmark's whole model answering a short turn on a 512-token context.
        _decoder("reply_512", "reply", layers=24, vocab=151936, context=512, tokens=24, steps=32),
        # A long document as the prompt: attention over thousands of rows (two of the layers).
        _decoder("prompt_3000", "prompt", tokens=3000, stack=1024),
        # A turn late in a long conversation.
        _decoder("reply_3500", "reply", context=3500, tokens=17, steps=16),
        # An unquantized model's turn: prompt and steps through its f16 matrices.
        _decoder("reply_f16", "reply", weights="f16", tokens=100, steps=16, context=64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "pick", "sample", "prompt", "prompt", "reply", "reply"])
    if kind == "linear":
        weights = rng.choice(["q8", "q8", "q4", "q4", "q4", "f16", "f32"])
        rows, cols = _log(rng, 128, 16384), 32 * _log(rng, 4, 448)
        tokens = 1 if weights in ("f16", "f32") else rng.choice([1, _log(rng, 2, 1024)])
        return {"kind": kind, "weights": weights, "rows": rows, "cols": cols, "tokens": tokens}
    if kind == "pick":
        return {"kind": kind, "vocab": _log(rng, 4000, 151936), "dim": 64 * _log(rng, 4, 28),
                "top_k": _log(rng, 1, 64), "history": _log(rng, 1, 2000), "top_p": rng.choice([0.8, 1.0])}
    if kind == "sample":
        return {"kind": kind, "vocab": _log(rng, 4000, 151936), "top_k": rng.choice([0, 20, _log(rng, 1, 256)]),
                "history": _log(rng, 1, 2000), "top_p": rng.choice([0.8, 0.95])}
    shape = rng.choice(["h64", "h64", "h128", "narrow"])
    weights = rng.choice(["q4mix", "q4mix", "q4mix", "f16", "f32"])
    kv_f32 = rng.random() < 0.2
    c = _decoder("", kind, shape=shape, layers=rng.choice([1, 2]), vocab=_log(rng, 1000, 8000), weights=weights,
                 kv_f32=kv_f32, hadamard=rng.random() < 0.15, stack=32 * rng.choice([1, 4, 8, 16, 16, 32]))
    del c["name"]
    dense = weights in ("f16", "f32")
    if kind == "prompt":
        c["tokens"] = _log(rng, 1, 200 if dense else 700 if kv_f32 else 2900)
        c["context"] = rng.choice([0, 0, rng.randrange(1, 500)])
    else:
        c["context"], c["tokens"] = _log(rng, 16, 200 if dense else 3800), _log(rng, 1, 64)
        c["steps"] = rng.randrange(4, 25)
    return c


# ------------------------------------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator("cuda").manual_seed(seed)


def _matrix(g, weights, rows, cols):
    """A weight matrix in the .qnt layout of its type, as device bytes: quants, then f16 scales per 32."""
    if weights in ("f16", "f32"):
        w = torch.randn(rows, cols, generator=g, device="cuda") * 0.02
        return (w.half() if weights == "f16" else w).view(torch.uint8).reshape(-1)
    if weights == "q8":
        q = torch.randint(-127, 128, (rows * cols,), generator=g, device="cuda", dtype=torch.int8).view(torch.uint8)
        d = torch.randn(rows * cols // QK, generator=g, device="cuda").abs() * (0.02 / 127)
    else:  # both nibbles of a byte uniform over [-8, 7]; one scale per 128 weights where the row allows it
        q = torch.randint(0, 256, (rows * cols // 2,), generator=g, device="cuda", dtype=torch.uint8)
        group = 4 if cols % 128 == 0 else 1
        d = torch.randn(rows * cols // QK // group, generator=g, device="cuda").abs() * (0.02 / 7)
        d = d.repeat_interleave(group)
    return torch.cat([q, d.half().view(torch.uint8)])


def _plain(buf, weights, rows, cols):
    """The same matrix in 64 bits."""
    if weights in ("f16", "f32"):
        return buf.view(torch.float16 if weights == "f16" else torch.float32).reshape(rows, cols).double()
    nq = rows * cols if weights == "q8" else rows * cols // 2
    d = buf[nq:].view(torch.float16).double()
    if weights == "q8":
        q = buf[:nq].view(torch.int8).double().reshape(-1, QK)
    else:
        b = buf[:nq].reshape(-1, QK // 2)
        q = torch.cat([b & 15, b >> 4], 1).double() - 8
    return (q * d[:, None]).reshape(rows, cols)


def _shortlist_copy(head, V, D):
    """The head's 4-bit copy and its per-block error norms, rounded up to f16 (so that they stay bounds)."""
    packed, scales, errs = [], [], []
    w8, d8 = head[:V * D].view(torch.int8).reshape(-1, QK), head[V * D:].view(torch.float16)
    for at in range(0, w8.shape[0], 1 << 20):
        w = w8[at:at + (1 << 20)].float() * d8[at:at + (1 << 20)].float()[:, None]
        m = w.gather(1, w.abs().argmax(1, keepdim=True))
        d = (m / -8).half()
        df = d.float()
        q = torch.where(df != 0, (w / torch.where(df != 0, df, 1) + 8).round().clamp(0, 15), 8)
        err = ((q - 8).double() * df.double() - w.double()).square().sum(1).sqrt()
        e = err.half()
        e = torch.where(e.double() < err, (e.view(torch.int16) + 1).view(torch.float16), e)  # the next f16 up
        q = q.to(torch.uint8)
        packed.append((q[:, :16] | (q[:, 16:] << 4)).reshape(-1))
        scales.append(d.reshape(-1))
        errs.append(e)
    return (torch.cat([torch.cat(packed), torch.cat(scales).view(torch.uint8)]), torch.cat(errs).view(torch.uint8))


def _model(case, seed):
    """The decoder's tensors on the GPU: name -> (bytes, type, rows, cols); norms near 1, small biases."""
    g = _gen(seed)
    D, H, KV, hd, F = _SHAPES[case["shape"]]
    V, mix = case["vocab"], case["weights"] == "q4mix"
    attn, mlp = ("q8", "q4") if mix else (case["weights"],) * 2
    t = {}

    def vec(name, n, mean, sd):
        t[name] = ((torch.randn(n, generator=g, device="cuda") * sd + mean).view(torch.uint8), "f32", 1, n)

    def mat(name, kind, rows, cols):
        t[name] = (_matrix(g, kind, rows, cols), kind, rows, cols)

    mat("model.embed_tokens.weight", attn, V, D)
    vec("model.norm.weight", D, 1.0, 0.05)
    for l in range(case["layers"]):
        p = "model.layers.%d." % l
        vec(p + "input_layernorm.weight", D, 1.0, 0.05)
        vec(p + "post_attention_layernorm.weight", D, 1.0, 0.05)
        for n, rows in (("q", D), ("k", KV * hd), ("v", KV * hd)):
            mat(p + "self_attn.%s_proj.weight" % n, attn, rows, D)
            vec(p + "self_attn.%s_proj.bias" % n, rows, 0.0, 0.02)
        mat(p + "self_attn.o_proj.weight", attn, D, D)
        mat(p + "mlp.gate_proj.weight", mlp, F, D)
        mat(p + "mlp.up_proj.weight", mlp, F, D)
        mat(p + "mlp.down_proj.weight", mlp, D, F)
    if _shortlisted(case):
        h4, err = _shortlist_copy(t["model.embed_tokens.weight"][0], V, D)
        t["quanta.head_q4"], t["quanta.head_err"] = (h4, "q4", V, D), (err, "f16", V, D // QK)
    return t


def _shortlisted(case):
    """The benchmark's vocabulary goes through the shortlist head; the small ones through the full head."""
    return case["weights"] == "q4mix" and case["vocab"] > 100000


def _ids(case, seed):
    rng = np.random.default_rng(seed)
    return (rng.integers(0, case["vocab"], case["context"]).astype(np.int32),
            rng.integers(0, case["vocab"], case["tokens"]).astype(np.int32))


class _View:
    """A device buffer of the decoder, for torch.as_tensor (which keeps this object, and so the decoder, alive)."""

    def __init__(self, dec, ptr, n):
        self.dec = dec
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f4", "data": (ptr, False), "version": 2}


def prepare(case, seed):
    qh, qnt = _package()
    qh.init(0)
    kind = case["kind"]
    code = {"f32": qh.F32, "f16": qh.F16, "q8": qh.Q8_0, "q4": qh.Q4_0}
    if kind == "linear":
        g = _gen(seed)
        rows, cols, n = case["rows"], case["cols"], case["tokens"]
        W = qh.DeviceTensor(_matrix(g, case["weights"], rows, cols), code[case["weights"]], rows, cols)
        x = torch.randn(n, cols, generator=g, device="cuda")
        out = torch.zeros(n, rows, device="cuda")
        q = torch.zeros(n, cols, device="cuda", dtype=torch.int8)
        d = torch.zeros(n, cols // QK, device="cuda")
        return {"qh": qh, "case": case, "W": W, "x": x, "out": out, "q": q, "d": d}
    if kind in ("pick", "sample"):
        g = _gen(seed)
        V = case["vocab"]
        s = {"qh": qh, "case": case, "rng": torch.full((1,), qh.sampler_state(2 * seed + 1), dtype=torch.int64,
                                                       device="cuda"),
             "params": qh.sampler_params(top_k=case["top_k"], top_p=case["top_p"]),
             "history": torch.randint(0, V, (case["history"],), generator=g, device="cuda", dtype=torch.int32)}
        if kind == "sample":
            s["logits"] = torch.randn(V, generator=g, device="cuda") * 3
            s["ws"] = qh.sample_workspace(V)
            return s
        D = case["dim"]
        h8 = _matrix(g, "q8", V, D)
        h4, err = _shortlist_copy(h8, V, D)
        s["head"] = qh.ShortlistHead(qh.DeviceTensor(h8, qh.Q8_0, V, D), qh.DeviceTensor(h4, qh.Q4_0, V, D),
                                     qh.DeviceTensor(err, qh.F16, V, D // QK), top_k=case["top_k"])
        s["x"] = torch.randn(1, D, generator=g, device="cuda") * 0.5
        s["q"] = torch.zeros(1, D, device="cuda", dtype=torch.int8)
        s["d"] = torch.zeros(1, D // QK, device="cuda")
        return s
    D, H, KV, hd, F = _SHAPES[case["shape"]]
    hp = qnt.HParams(vocab_size=case["vocab"], dim=D, n_layers=case["layers"], n_heads=H, n_kv_heads=KV, head_dim=hd,
                     ffn_dim=F, flags=qnt.FLAG_HADAMARD_DOWN if case["hadamard"] else 0)
    tensors = {n: qnt.TensorRec(code[k], rows, cols, b.cpu().numpy()) for n, (b, k, rows, cols) in
               _model(case, seed).items()}
    dec = qh.Decoder(hp, tensors, ctx_len=4096, kv_f32=case["kv_f32"])
    dec.set_prefill_stack(case["stack"])
    context, turn = _ids(case, seed)
    k = 1 if _shortlisted(case) else 0
    if len(context):
        dec.prefill(context, 0, top_k=k)
    s = {"case": case, "dec": dec, "k": k, "turn": turn,
         "logits": torch.as_tensor(_View(dec, dec.views.logits, case["vocab"]), device="cuda"),
         "hidden": torch.as_tensor(_View(dec, dec.views.hidden, D), device="cuda")}
    if case["steps"]:
        if not len(context):
            dec.prefill(turn, 0, top_k=k)
        dec.begin(case["steps"] + 1, top_k=k)
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            dec.step(top_k=k)
    return s


# ------------------------------------------------------------------------------------------------ one pass

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "linear":
        qh, W = s["qh"], s["W"]
        if case["weights"] in ("f16", "f32"):
            qh.matvec_ref(W, s["x"], out=s["out"])
            return s["out"]
        qh.quantize_q8(s["x"], s["q"], s["d"])
        if case["tokens"] == 1:
            qh.matvec_q(W, s["q"], s["d"], out=s["out"])
        else:
            qh.matmul_q(W, s["q"], s["d"], out=s["out"])
        return s["out"]
    if kind == "sample":
        return {"token": s["qh"].sample(s["logits"], s["params"], s["rng"], history=s["history"], ws=s["ws"]),
                "rng": s["rng"]}
    if kind == "pick":
        qh, head = s["qh"], s["head"]
        qh.quantize_q8(s["x"], s["q"], s["d"])
        head(s["q"], s["d"], must=s["history"])
        token = qh.sample(head.logits, s["params"], s["rng"], history=s["history"], head=head)
        return {"logits": head.logits, "coarse": head.coarse, "token": token, "rng": s["rng"]}
    dec, k = s["dec"], s["k"]
    dec.prefill(s["turn"], case["context"], top_k=k)
    if not case["steps"]:
        return {"logits": s["logits"], "hidden": s["hidden"]}
    dec.begin(case["steps"] + 1, top_k=k)
    for _ in range(case["steps"]):
        s["graph"].replay()
    return {"logits": s["logits"], "hidden": s["hidden"], "tokens": dec.out}


_BYTES = {"f32": 4.0, "f16": 2.0, "q8": 1.0625, "q4": 0.5625}


def work(case):
    kind = case["kind"]
    if kind == "linear":
        rows, cols, n = case["rows"], case["cols"], case["tokens"]
        return {"bytes": rows * cols * _BYTES[case["weights"]] + 4 * n * (rows + cols), "flops": 2 * n * rows * cols}
    if kind == "sample":
        return {"bytes": 4 * case["vocab"] + 4 * case["history"], "flops": 4 * case["vocab"]}
    if kind == "pick":  # the 4-bit screen of every row with its error bounds, scores and bounds out
        V, D = case["vocab"], case["dim"]
        return {"bytes": V * (0.5625 * D + D / 16) + 12 * V, "flops": 2 * V * D}
    D, H, KV, hd, F = _SHAPES[case["shape"]]
    mix = case["weights"] == "q4mix"
    attn, mlp = (_BYTES["q8"], _BYTES["q4"]) if mix else (_BYTES[case["weights"]],) * 2
    n_attn, n_mlp, V = 2 * D * D + 2 * D * KV * hd, 3 * D * F, case["vocab"]
    weights = case["layers"] * (n_attn * attn + n_mlp * mlp)
    head = V * (0.5625 * D + D / 16) if _shortlisted(case) else V * D * attn
    row = 2 * KV * hd * (4 if case["kv_f32"] else 2) * case["layers"]  # the cache bytes of one position
    n, c = case["tokens"], case["context"]
    total = weights + head + 4 * V + row * (c + n)
    flops = 2 * n * case["layers"] * (n_attn + n_mlp) + 4 * case["layers"] * H * hd * n * (c + (n + 1) / 2) + 2 * V * D
    for i in range(case["steps"]):
        total += weights + head + 4 * V + row * (c + n + i + 1)
        flops += 2 * case["layers"] * (n_attn + n_mlp) + 4 * case["layers"] * H * hd * (c + n + i + 1) + 2 * V * D
    return {"bytes": total, "flops": flops}


def tolerance(case):
    """Every call promises the bits of the scalar definition: exact int32 block sums, then one float chain per output in
    block order (and position order in attention), whatever the batch, stack or layout."""
    return "exact"


# ------------------------------------------------------------------------------------------------ the same in 64 bits

def _quantized(x):
    """x rounded to its int8 codes per 32 values, in 64 bits."""
    b = x.double().reshape(-1, QK)
    d = b.abs().amax(1, keepdim=True) / 127
    y = torch.where(d > 0, b / torch.where(d > 0, d, 1), 0)
    t = y.trunc()
    return ((t + torch.where((y - t).abs() >= 0.5, y.sign(), 0)) * d).reshape(x.shape)


def _hadamard(x):
    v = x.reshape(-1, 256)
    h = 1
    while h < 256:
        p = v.reshape(-1, 256 // (2 * h), 2, h)
        v = torch.stack([p[:, :, 0] + p[:, :, 1], p[:, :, 0] - p[:, :, 1]], 2).reshape(-1, 256)
        h *= 2
    return (v / 16).reshape(x.shape)


class _Exact:
    """The decoder in plain torch, 64 bits; the cache keeps the precision it is stored in."""

    def __init__(self, case, seed):
        self.c, self.t = case, _model(case, seed)
        self.w = {}
        self.cache = [None] * case["layers"]

    def mat(self, name):
        if name not in self.w:
            b, kind, rows, cols = self.t[name]
            self.w[name] = _plain(b, kind, rows, cols)
        return self.w[name]

    def linear(self, x, name):
        return (_quantized(x) if self.t[name][1] in ("q8", "q4") else x) @ self.mat(name).T

    def norm(self, x, name):
        return x / (x.square().mean(-1, keepdim=True) + 1e-6).sqrt() * self.mat(name)

    def rope(self, x, pos, hd):
        f = 1e6 ** (-2.0 * torch.arange(hd // 2, device="cuda", dtype=torch.float64) / hd)
        a = pos[:, None, None] * f
        u, v = x[..., :hd // 2], x[..., hd // 2:]
        return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()], -1)

    def stored(self, x):
        return x.float().double() if self.c["kv_f32"] else x.float().half().double()

    def forward(self, ids, pos0):
        D, H, KV, hd, F = _SHAPES[self.c["shape"]]
        n = len(ids)
        pos = torch.arange(pos0, pos0 + n, device="cuda")
        x = self.mat("model.embed_tokens.weight")[torch.as_tensor(np.asarray(ids), device="cuda").long()]
        for l in range(self.c["layers"]):
            p = "model.layers.%d." % l
            h = self.norm(x, p + "input_layernorm.weight")
            q, k, v = (self.linear(h, p + "self_attn.%s_proj.weight" % m) + self.mat(p + "self_attn.%s_proj.bias" % m)
                       for m in "qkv")
            q = self.rope(q.reshape(n, H, hd), pos.double(), hd)
            k = self.stored(self.rope(k.reshape(n, KV, hd), pos.double(), hd))
            v = self.stored(v.reshape(n, KV, hd))
            if self.cache[l] is not None:
                k, v = torch.cat([self.cache[l][0], k]), torch.cat([self.cache[l][1], v])
            self.cache[l] = k, v
            o = torch.empty(n, H, hd, device="cuda", dtype=torch.float64)
            later = torch.arange(len(k), device="cuda")[None] > pos[:, None]
            for j in range(H):
                a = q[:, j] @ k[:, j * KV // H].T.contiguous() / math.sqrt(hd)
                o[:, j] = a.masked_fill(later, -math.inf).softmax(-1) @ v[:, j * KV // H].contiguous()
            x = x + self.linear(o.reshape(n, D), p + "self_attn.o_proj.weight")
            h = self.norm(x, p + "post_attention_layernorm.weight")
            gate = self.linear(h, p + "mlp.gate_proj.weight")
            m = gate / (1 + (-gate).exp()) * self.linear(h, p + "mlp.up_proj.weight")
            if self.c["hadamard"]:
                m = _hadamard(m)
            x = x + self.linear(m, p + "mlp.down_proj.weight")
        hidden = self.norm(x[-1:], "model.norm.weight")
        return hidden[0], self.linear(hidden, "model.embed_tokens.weight")[0]


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        g = _gen(seed)
        W = _plain(_matrix(g, case["weights"], case["rows"], case["cols"]), case["weights"], case["rows"], case["cols"])
        x = torch.randn(case["tokens"], case["cols"], generator=g, device="cuda")
        return (x.double() if case["weights"] in ("f16", "f32") else _quantized(x)) @ W.T
    if kind == "sample":
        return None  # whole numbers
    if kind == "pick":
        g = _gen(seed)
        V, D = case["vocab"], case["dim"]
        torch.randint(0, V, (case["history"],), generator=g, device="cuda", dtype=torch.int32)
        h4, _ = _shortlist_copy(_matrix(g, "q8", V, D), V, D)
        x = _quantized(torch.randn(1, D, generator=g, device="cuda") * 0.5)
        # which logits are finite follows from comparisons of rounded scores: only the screen's scores have a value here
        return {"logits": None, "coarse": (x @ _plain(h4, "q4", V, D).T)[0], "token": None, "rng": None}
    context, turn = _ids(case, seed)
    e = _Exact(case, seed)
    if len(context):
        e.forward(context, 0)
    hidden, logits = e.forward(turn, case["context"])
    for i in range(case["steps"]):
        top = logits.topk(2)
        if float(top.values[0] - top.values[1]) < 0.02 * float(logits.std()):
            return None  # two tokens so close that rounding decides which one the steps go on with
        hidden, logits = e.forward([int(top.indices[0])], case["context"] + len(turn) + i)
    out = {"logits": None if _shortlisted(case) else logits, "hidden": hidden}
    if case["steps"]:
        out["tokens"] = None
    return out
