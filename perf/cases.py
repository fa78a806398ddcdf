"""The calls that a program using this library spends its time in, as measurable cases.

A case names an operation of the public Python surface with its sizes:

  proj  one linear layer per matrix, `layers` matrices of one shape (a decode or prefill pass walks the layers of a
        model, so every matrix is read once per pass); device-resident (`gemv_dev`) or, with `host`, the drop-in
        operator functions that take and return host arrays (`q4k_gemv`, `q8_0_gemv_batch`, ...)
  step  one pass of `tokens` sequences through `layers` transformer blocks, attention itself left out: embedding rows,
        norm + quantisation, Q / K / V, output projection, residual add + norms, gated FFN (a Q4_K_M mix of formats)
  ffn   the dense gated FFN on its own
  head  the greedy LM head: host token in, (row, value) of the largest logit out
  moe   the routed sparse experts of a layer, device-resident or (`host`) with host arrays

Weights are valid blocks whose dequantised values are about N(0, 0.02); tokens are N(0, 1).
"""
import math

import numpy as np
import torch

import runnburn_amd as rnb

# format -> (ggml type id, elements per block, bytes per block, prefix of the host operator functions)
FORMATS = {
    "Q4_0": (2, 32, 18, "q4_0"), "Q4_1": (3, 32, 20, "q4_1"), "Q5_0": (6, 32, 22, "q5_0"), "Q5_1": (7, 32, 24, "q5_1"),
    "Q8_0": (8, 32, 34, "q8_0"), "Q8_1": (9, 32, 36, "q8_1"), "Q2_K": (10, 256, 84, "q2k"), "Q3_K": (11, 256, 110, "q3k"),
    "Q4_K": (12, 256, 144, "q4k"), "Q5_K": (13, 256, 176, "q5k"), "Q6_K": (14, 256, 210, "q6k"),
    "IQ2_XXS": (16, 256, 66, "iq2_xxs"), "IQ3_XXS": (18, 256, 98, "iq3_xxs"), "IQ2_S": (22, 256, 82, "iq2_s"),
    "IQ4_XS": (23, 256, 136, "iq4_xs"),
}
# what is met in earnest, most used first: the K-quants and Q8_0 of published models, then the rest
USED = ["Q4_K"] * 5 + ["Q6_K"] * 4 + ["Q8_0"] * 3 + ["Q5_K"] * 3 + ["Q3_K", "Q2_K", "Q4_0", "Q4_0", "Q5_0", "Q4_1", "Q5_1",
                                                                  "Q8_1", "IQ4_XS", "IQ4_XS", "IQ3_XXS", "IQ2_S", "IQ2_XXS"]
VOCAB = 32000  # rows of the embedding table of a step
EPS = 1e-5


def listed():
    return [
        # the smallest call of the drop-in surface: one token through one small matrix, host array in, host array out
        {"name": "host_gemv_small", "op": "proj", "quant": "Q8_0", "rows": 2048, "cols": 2048, "tokens": 1, "layers": 1, "host": True},
        # decoding one sequence: four blocks of an 8B-class model
        {"name": "step_decode", "op": "step", "layers": 4, "n_embd": 4096, "kv_rows": 1024, "n_ff": 14336, "tokens": 1},
        # decoding a dozen sequences together
        {"name": "step_batch", "op": "step", "layers": 2, "n_embd": 4096, "kv_rows": 1024, "n_ff": 14336, "tokens": 12},
        # the next token of a greedy decode, 128256 x 4096 vocabulary
        {"name": "head_greedy", "op": "head", "quant": "Q6_K", "rows": 128256, "cols": 4096},
        # a short ragged batch (speculative tokens of several sequences) on a 13B-class projection
        {"name": "proj_q5k_short", "op": "proj", "quant": "Q5_K", "rows": 13824, "cols": 5120, "tokens": 21, "layers": 2, "host": False},
        # prefill, the benchmark's GEMM: 512 tokens
        {"name": "proj_q4k_prefill", "op": "proj", "quant": "Q4_K", "rows": 14336, "cols": 4096, "tokens": 512, "layers": 1, "host": False},
        # a long prefill chunk through a whole FFN: the largest call
        {"name": "ffn_prefill", "op": "ffn", "down": "Q6_K", "n_ff": 14336, "n_embd": 4096, "tokens": 2048},
        # a prompt of no round length on 8-bit weights
        {"name": "proj_q8_prefill_ragged", "op": "proj", "quant": "Q8_0", "rows": 4096, "cols": 4096, "tokens": 333, "layers": 2, "host": False},
        # a prompt on importance-quantised weights
        {"name": "proj_iq2s_prefill", "op": "proj", "quant": "IQ2_S", "rows": 14336, "cols": 4096, "tokens": 160, "layers": 1, "host": False},
        # sparse experts: one decoded token, a small batch, a prefill chunk
        {"name": "moe_decode", "op": "moe", "down": "Q6_K", "n_expert": 128, "top_k": 8, "n_ff": 768, "n_embd": 2048, "tokens": 1, "shared": False, "host": False},
        {"name": "moe_batch", "op": "moe", "down": "Q6_K", "n_expert": 128, "top_k": 8, "n_ff": 768, "n_embd": 2048, "tokens": 64, "shared": False, "host": False},
        {"name": "moe_prefill", "op": "moe", "down": "Q6_K", "n_expert": 128, "top_k": 8, "n_ff": 768, "n_embd": 2048, "tokens": 512, "shared": False, "host": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["proj"] * 9 + ["ffn"] * 3 + ["step"] * 3 + ["moe"] * 4 + ["head"] * 1)
    if op == "proj":
        # token counts: decode, a few sequences together, prompts
        tokens = rng.choice([1, _log(rng, 2, 32), _log(rng, 33, 2048)])
        quant = rng.choice(USED)
        rows, cols = _log(rng, 512, 28672), 256 * _log(rng, 4, 64)
        while rows * cols * tokens > 120e9:
            tokens = max(1, tokens // 2)
        per = rows * (cols // FORMATS[quant][1]) * FORMATS[quant][2]
        layers = max(1, min(6, int(96e6 // per))) if tokens <= 32 else 1
        host = rng.random() < 0.25
        return {"op": op, "quant": quant, "rows": rows, "cols": cols, "tokens": tokens, "layers": min(2, layers) if host else layers, "host": host}
    if op == "ffn":
        tokens = rng.choice([1, _log(rng, 2, 32), _log(rng, 33, 2048)])
        return {"op": op, "down": rng.choice(["Q6_K", "Q6_K", "Q4_K", "Q5_K", "Q8_0", "Q5_1"]), "n_ff": 256 * _log(rng, 8, 56),
                "n_embd": 256 * _log(rng, 4, 20), "tokens": tokens}
    if op == "step":
        n_embd = 256 * _log(rng, 8, 20)
        return {"op": op, "layers": rng.choice([1, 2, 3]), "n_embd": n_embd, "kv_rows": rng.choice([256, 512, n_embd // 4, n_embd]),
                "n_ff": 256 * _log(rng, 16, 56), "tokens": rng.choice([1, 1, _log(rng, 2, 32)])}
    if op == "head":
        quant = rng.choice(["Q6_K", "Q8_0"])
        return {"op": op, "quant": quant, "rows": _log(rng, 16000, 128256), "cols": 256 * _log(rng, 8, 16)}
    n_expert, top_k = rng.choice([(8, 2), (16, 2), (32, 4), (64, 8), (128, 8)])
    tokens = rng.choice([1, _log(rng, 2, 32), _log(rng, 33, 512)])
    return {"op": op, "down": rng.choice(["Q6_K", "Q6_K", "Q4_K", "Q5_K"]), "n_expert": n_expert, "top_k": top_k,
            "n_ff": 256 * _log(rng, 2, 8), "n_embd": 256 * _log(rng, 4, 16), "tokens": tokens, "shared": rng.random() < 0.3,
            "host": n_expert <= 16 and rng.random() < 0.5}


# ---- synthetic weights -------------------------------------------------------------------------------------------------

def _lut(fn, g):
    """65536 bytes whose high and low halves of the index drive `fn`; picked uniformly they give fn's distribution."""
    u = (torch.arange(256, device="cuda", dtype=torch.float64) + 0.5) / 256
    z = torch.special.ndtri(u)  # normal quantiles
    return fn(z[:, None].expand(256, 256), z[None, :].expand(256, 256)).reshape(-1).to(torch.uint8)


def _nib(z, mean, sd, top):
    return (mean + sd * z).round().clamp(0, top).to(torch.int32)


class _Blocks:
    """Makes packed blocks of every format on the GPU, chunk by chunk."""

    def __init__(self, g):
        self.g = g
        self.nibbles = _lut(lambda a, b: _nib(a, 7.5, 2.8, 15) | (_nib(b, 7.5, 2.8, 15) << 4), g)
        self.int8 = _lut(lambda a, b: ((a + 0.01 * b) * 42).round().clamp(-127, 127).to(torch.int32) & 255, g)

    def _bytes(self, n, k):
        return torch.randint(0, 256, (n, k), generator=self.g, device="cuda", dtype=torch.uint8)

    def _pick(self, lut, n, k):
        return lut[torch.randint(0, 65536, (n, k), generator=self.g, device="cuda")]

    def _half(self, n, mean, spread=0.3):
        u = torch.rand((n, 1), generator=self.g, device="cuda") * (2 * spread) + (1 - spread)
        return (mean * u).to(torch.float16).view(torch.uint8)

    def _six_bit(self, n):
        """12 bytes that hold eight 6-bit scales and eight 6-bit mins, all between 24 and 63."""
        v = torch.randint(24, 64, (n, 16), generator=self.g, device="cuda", dtype=torch.int32)
        sc, mn = v[:, :8], v[:, 8:]
        out = torch.cat([(sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6), (mn[:, :4] & 63) | ((mn[:, 4:] >> 4) << 6),
                         (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], dim=1)
        return out.to(torch.uint8)

    def _chunk(self, fmt, n):
        nib = lambda k: self._pick(self.nibbles, n, k)  # noqa: E731
        if fmt == "Q8_0":
            parts = [self._half(n, 4.8e-4), self._pick(self.int8, n, 32)]
        elif fmt == "Q8_1":
            parts = [self._half(n, 4.8e-4), self._half(n, 1e-3), self._pick(self.int8, n, 32)]
        elif fmt == "Q4_0":
            parts = [self._half(n, 7e-3), nib(16)]
        elif fmt == "Q4_1":
            parts = [self._half(n, 7e-3), self._half(n, -5.2e-2), nib(16)]
        elif fmt == "Q5_0":
            parts = [self._half(n, 2.2e-3), self._bytes(n, 4), nib(16)]
        elif fmt == "Q5_1":
            parts = [self._half(n, 2.2e-3), self._half(n, -3.4e-2), self._bytes(n, 4), nib(16)]
        elif fmt == "Q2_K":
            sc = torch.randint(5, 16, (n, 16), generator=self.g, device="cuda", dtype=torch.int32)
            mn = torch.randint(5, 16, (n, 16), generator=self.g, device="cuda", dtype=torch.int32)
            parts = [(sc | (mn << 4)).to(torch.uint8), self._bytes(n, 64), self._half(n, 1.8e-3), self._half(n, 2.7e-3)]
        elif fmt == "Q3_K":
            parts = [self._bytes(n, 32), self._bytes(n, 64), self._bytes(n, 12), self._half(n, 5e-4)]
        elif fmt == "Q4_K":
            parts = [self._half(n, 1.6e-4), self._half(n, 1.2e-3), self._six_bit(n), nib(128)]
        elif fmt == "Q5_K":
            parts = [self._half(n, 5e-5), self._half(n, 7.7e-4), self._six_bit(n), self._bytes(n, 32), nib(128)]
        elif fmt == "Q6_K":
            sc = torch.randint(48, 128, (n, 16), generator=self.g, device="cuda", dtype=torch.int32)
            sign = 1 - 2 * torch.randint(0, 2, (n, 16), generator=self.g, device="cuda", dtype=torch.int32)
            parts = [nib(128), self._bytes(n, 64), ((sc * sign) & 255).to(torch.uint8), self._half(n, 1.2e-5)]
        elif fmt == "IQ4_XS":
            parts = [self._half(n, 2.5e-5), self._bytes(n, 2), self._bytes(n, 4), nib(128)]
        else:  # IQ2_XXS, IQ2_S, IQ3_XXS: d, then grid indices, signs and scales, any bytes
            parts = [self._half(n, 8e-4), self._bytes(n, FORMATS[fmt][2] - 2)]
        return torch.cat(parts, dim=1)

    def make(self, fmt, rows, cols, into=None):
        """uint8 [rows * cols / elements * bytes], written into a device tensor when one is given."""
        _, elems, nbytes, _ = FORMATS[fmt]
        n = rows * (cols // elems)
        out = into if into is not None else torch.empty(n * nbytes, dtype=torch.uint8, device="cuda")
        view, step = out.view(n, nbytes), max(1, (1 << 25) // nbytes)
        for a in range(0, n, step):
            m = min(step, n - a)
            view[a:a + m] = self._chunk(fmt, m)
        return out


class _Span:
    """A DeviceBuffer as torch sees it."""

    def __init__(self, buf, shape, typestr):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (buf.ptr, False), "version": 2}


def _view(buf, shape, typestr="<f4"):
    return torch.as_tensor(_Span(buf, tuple(shape), typestr), device="cuda")


class _HostWeights:
    """A host array of packed blocks, resident on the device for as long as this object lives."""

    def __init__(self, array):
        self.array = array
        rnb.prewarm([array])

    def __del__(self):
        try:
            rnb.release(self.array)
        except Exception:  # at interpreter exit
            pass


class _Maker:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)
        self.blocks = _Blocks(self.g)

    def weights(self, fmt, rows, cols):
        buf = rnb.DeviceBuffer(rows * (cols // FORMATS[fmt][1]) * FORMATS[fmt][2])
        self.blocks.make(fmt, rows, cols, _view(buf, (buf.nbytes,), "|u1"))
        return buf

    def host_weights(self, fmt, rows, cols):
        return _HostWeights(self.blocks.make(fmt, rows, cols).cpu().numpy())

    def floats(self, *shape, mean=0.0, sd=1.0):
        return torch.randn(shape, generator=self.g, device="cuda") * sd + mean

    def dev_floats(self, *shape, mean=0.0, sd=1.0):
        buf = rnb.DeviceBuffer(4 * math.prod(shape))
        _view(buf, shape).copy_(self.floats(*shape, mean=mean, sd=sd))
        return buf


def _out(*shape):
    buf = rnb.DeviceBuffer(4 * math.prod(shape))
    view = _view(buf, shape)
    view.zero_()
    return buf, view


def _routes(rng, tokens, n_expert, top_k):
    """A router's choice: some experts are liked more than others; slots sorted by expert for batches, rank order for one
    token, as the two callers pass them."""
    logits = (rng.standard_normal((tokens, n_expert)) + 0.4 * rng.standard_normal(n_expert)).astype(np.float32)
    idx = np.argsort(-logits, axis=1, kind="stable")[:, :top_k]
    sel = np.take_along_axis(logits, idx, axis=1)
    w = np.exp(sel - sel[:, :1])
    w = (w / w.sum(axis=1, keepdims=True)).astype(np.float32)
    return idx.astype(np.uint32), w


# ---- what a program has in hand ------------------------------------------------------------------------------------------

def prepare(case, seed):
    m = _Maker(seed)
    op = case["op"]
    s = {"case": case}
    if op == "proj":
        rows, cols, t = case["rows"], case["cols"], case["tokens"]
        if case["host"]:
            s["w"] = [m.host_weights(case["quant"], rows, cols) for _ in range(case["layers"])]
            s["x"] = [m.floats(t * cols).cpu().numpy() for _ in range(case["layers"])]
            s["fn"] = getattr(rnb, FORMATS[case["quant"]][3] + ("_gemv" if t == 1 else "_gemv_batch"))
        else:
            s["w"] = [m.weights(case["quant"], rows, cols) for _ in range(case["layers"])]
            s["x"] = [m.dev_floats(t, cols) for _ in range(case["layers"])]
            s["out"] = [_out(t, rows) for _ in range(case["layers"])]
    elif op == "ffn":
        n_ff, n_embd, t = case["n_ff"], case["n_embd"], case["tokens"]
        s["gate"], s["up"] = m.weights("Q4_K", n_ff, n_embd), m.weights("Q4_K", n_ff, n_embd)
        s["down"] = m.weights(case["down"], n_embd, n_ff)
        s["x"], s["out"] = m.dev_floats(t, n_embd), _out(t, n_embd)
    elif op == "head":
        s["w"] = m.host_weights(case["quant"], case["rows"], case["cols"])
        s["x"] = m.floats(case["cols"]).cpu().numpy()
    elif op == "step":
        n, kv, n_ff, t = case["n_embd"], case["kv_rows"], case["n_ff"], case["tokens"]
        s["embed"] = m.host_weights("Q4_K", VOCAB, n)
        s["ids"] = torch.randint(0, VOCAB, (t,), generator=m.g, device="cuda").cpu().numpy().astype(np.uint32)
        s["hidden"], s["h"] = rnb.DeviceBuffer(4 * t * n), rnb.DeviceBuffer(4 * t * n)
        norm = lambda: m.dev_floats(n, mean=1.0, sd=0.1)  # noqa: E731
        s["layers"] = []
        for _ in range(case["layers"]):
            s["layers"].append({
                "q": m.weights("Q4_K", n, n), "k": m.weights("Q4_K", kv, n), "v": m.weights("Q6_K", kv, n),
                "o": m.weights("Q4_K", n, n), "gate": m.weights("Q4_K", n_ff, n), "up": m.weights("Q4_K", n_ff, n),
                "down": m.weights("Q6_K", n, n_ff), "attn_norm": norm(), "post_attn": norm(), "ffn_norm": norm(),
                "post_ffn": norm(), "attn": m.dev_floats(t, n), "q_out": _out(t, n), "k_out": _out(t, kv),
                "v_out": _out(t, kv), "o_out": _out(t, n), "f_out": _out(t, n)})
        s["hidden_view"] = _view(s["hidden"], (t, n))
    else:
        e, n_ff, n_embd, t = case["n_expert"], case["n_ff"], case["n_embd"], case["tokens"]
        rng = np.random.default_rng(seed)
        idx, route = _routes(rng, t, e, case["top_k"])
        token = np.repeat(np.arange(t, dtype=np.uint32), case["top_k"])
        expert, route = idx.reshape(-1), route.reshape(-1)
        if t > 1:
            order = np.lexsort((token, expert))
            expert, token, route = expert[order], token[order], route[order]
        if case["shared"]:  # the shared expert is one more slot of every token
            expert = np.concatenate([expert, np.full(t, e, np.uint32)])
            token = np.concatenate([token, np.arange(t, dtype=np.uint32)])
            route = np.concatenate([route, rng.uniform(0.2, 0.9, t).astype(np.float32)])
        s["slots"] = (expert, route, token)
        make = m.host_weights if case["host"] else m.weights
        s["gate"], s["up"] = make("Q4_K", e * n_ff, n_embd), make("Q4_K", e * n_ff, n_embd)
        s["down"] = make(case["down"], e * n_embd, n_ff)
        s["shared"] = None
        if case["shared"]:
            s["shared"] = [make("Q4_K", n_ff, n_embd), make("Q4_K", n_ff, n_embd), make(case["down"], n_embd, n_ff)]
        if case["host"]:
            s["x"] = m.floats(t, n_embd).cpu().numpy()
        else:
            s["x"], s["out"] = m.dev_floats(t, n_embd), _out(t, n_embd)
    torch.cuda.synchronize()  # the library has a stream of its own
    return s


# ---- one pass ------------------------------------------------------------------------------------------------------------

def _step(s, case):
    n, kv, n_ff, t = case["n_embd"], case["kv_rows"], case["n_ff"], case["tokens"]
    q4, q6 = FORMATS["Q4_K"][0], FORMATS["Q6_K"][0]
    rnb.quant_embedding_gather_dev(q4, s["embed"].array, VOCAB, n, s["ids"], s["hidden"])
    outs = []
    for i, l in enumerate(s["layers"]):
        if i == 0:
            rnb.rms_norm_dev(s["hidden"], l["attn_norm"], EPS, t, n, None, quantize=True)
        else:
            before = s["layers"][i - 1]
            rnb.rms_norm_add_rms_norm_quantize_dev(before["f_out"][0], before["post_ffn"], EPS, s["hidden"], l["attn_norm"], EPS, t, n, None)
        rnb.gemv_quantized_dev(q4, l["q"], n, n, t, l["q_out"][0])
        rnb.gemv_quantized_dev(q4, l["k"], kv, n, t, l["k_out"][0])
        rnb.gemv_quantized_dev(q6, l["v"], kv, n, t, l["v_out"][0])
        rnb.gemv_dev(q4, l["o"], n, n, l["attn"], t, l["o_out"][0])
        rnb.rms_norm_add_rms_norm_quantize_dev(l["o_out"][0], l["post_attn"], EPS, s["hidden"], l["ffn_norm"], EPS, t, n, s["h"])
        rnb.dense_q4k_silu_ffn_dev(l["gate"], l["up"], l["down"], q6, n_ff, n, t, s["h"], l["f_out"][0])
        outs += [l[k][1] for k in ("q_out", "k_out", "v_out", "o_out", "f_out")]
    return outs + [s["hidden_view"]]


def run(state):
    s, case = state, state["case"]
    op = case["op"]
    if op == "proj":
        rows, cols = case["rows"], case["cols"]
        if case["host"]:
            return [s["fn"](w.array, rows, cols, x) for w, x in zip(s["w"], s["x"])]
        quant = FORMATS[case["quant"]][0]
        for w, x, out in zip(s["w"], s["x"], s["out"]):
            rnb.gemv_dev(quant, w, rows, cols, x, case["tokens"], out[0])
        return [out[1] for out in s["out"]]
    if op == "ffn":
        rnb.dense_q4k_silu_ffn_dev(s["gate"], s["up"], s["down"], FORMATS[case["down"]][0], case["n_ff"], case["n_embd"],
                                   case["tokens"], s["x"], s["out"][0])
        return s["out"][1]
    if op == "head":
        fn = rnb.q6k_gemv_argmax if case["quant"] == "Q6_K" else rnb.q8_0_gemv_argmax
        return fn(s["w"].array, case["rows"], case["cols"], s["x"])
    if op == "step":
        return _step(s, case)
    expert, route, token = s["slots"]
    down = FORMATS[case["down"]][0]
    if case["host"]:
        shared = [w.array for w in s["shared"]] if s["shared"] else None
        return rnb.qwen35_sparse_experts_selected_base_by_token(s["gate"].array, s["up"].array, s["down"].array, expert, route,
                                                                token, case["tokens"], down, case["n_ff"], case["n_embd"], s["x"],
                                                                shared=shared)
    rnb.moe_sparse_experts_by_token_dev(s["gate"], s["up"], s["down"], case["n_expert"], expert, route, token, case["tokens"],
                                        down, case["n_ff"], case["n_embd"], s["x"], s["out"][0], shared=s["shared"])
    return s["out"][1]


# ---- what a pass cannot do without -----------------------------------------------------------------------------------------

def _matrix(fmt, rows, cols):
    return rows * (cols // FORMATS[fmt][1]) * FORMATS[fmt][2]


def work(case):
    op = case["op"]
    if op == "proj":
        rows, cols, t = case["rows"], case["cols"], case["tokens"]
        return {"bytes": case["layers"] * (_matrix(case["quant"], rows, cols) + 4 * t * (rows + cols)),
                "flops": case["layers"] * 2.0 * t * rows * cols}
    if op == "ffn":
        n_ff, n, t = case["n_ff"], case["n_embd"], case["tokens"]
        return {"bytes": 2 * _matrix("Q4_K", n_ff, n) + _matrix(case["down"], n, n_ff) + 8 * t * n, "flops": 6.0 * t * n_ff * n}
    if op == "head":
        return {"bytes": _matrix(case["quant"], case["rows"], case["cols"]) + 4 * case["cols"], "flops": 2.0 * case["rows"] * case["cols"]}
    if op == "step":
        n, kv, n_ff, t = case["n_embd"], case["kv_rows"], case["n_ff"], case["tokens"]
        weights = (2 * _matrix("Q4_K", n, n) + _matrix("Q4_K", kv, n) + _matrix("Q6_K", kv, n) + 2 * _matrix("Q4_K", n_ff, n)
                   + _matrix("Q6_K", n, n_ff) + 16 * n)
        # per layer: the attention vector in, q / k / v / o / f out; once: the embedding rows in, the hidden state out
        return {"bytes": case["layers"] * (weights + 4 * t * (4 * n + 2 * kv)) + t * (_matrix("Q4_K", 1, n) + 4 * n),
                "flops": case["layers"] * 2.0 * t * n * (2 * n + 2 * kv + 3 * n_ff)}
    e, k, n_ff, n, t = case["n_expert"], case["top_k"], case["n_ff"], case["n_embd"], case["tokens"]
    hit = e * (1 - (1 - k / e) ** t) + (1 if case["shared"] else 0)  # distinct experts expected
    slots = t * (k + (1 if case["shared"] else 0))
    return {"bytes": hit * (2 * _matrix("Q4_K", n_ff, n) + _matrix(case["down"], n, n_ff)) + 8 * t * n + 12 * slots,
            "flops": 6.0 * slots * n_ff * n}


def tolerance(case):
    # Activations are quantised to int8 and multiplied exactly; only the order of the f32 sums over the blocks is free: the
    # one-token kernels against the batch kernels on the same rows differ by rel 2e-7, max 1e-6 (all formats, 1280 - 9728 columns).
    if case["op"] in ("proj", "head"):
        return {"rel": 1e-6, "max": 5e-6}
    # Two stages: a difference in the last place of an intermediate can move its int8 code by one.  Inputs moved by one part
    # in 1e7 move the outputs by rel 3e-4 - 8e-4, max 0.03 where any code moved.
    if case["op"] in ("ffn", "moe"):
        return {"rel": 3e-3, "max": 0.1}
    # A chain of such stages: rel 3e-3, max 0.04 after one block, 0.007 - 0.016, max 0.1 after two to four.
    return {"rel": 0.01, "max": 0.16} if case["layers"] == 1 else {"rel": 0.05, "max": 0.4}
