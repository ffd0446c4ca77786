"""The work that programs built on inferi_amd have it do, as measurable cases.

Every case goes through the package's public entry points (the op API of
LlmContext, BatchedMultiqueryAttention and the Llama2 token loop), with the
weights, caches and handles that such a program keeps made in prepare().
Matrices are GGUF blocks with bell-shaped codes and a standard deviation of
0.02, as a quantizer writes them for trained weights; they are laid out here
field by field, so that exact() can form the same values in 64 bits on its own.

Model cases fix the tokens of every step but the last (forced prompt tokens),
so that a near-tie in the logits does not change the work that follows.  They
have fewer layers than the models their shapes come from, which keeps the
largest matrices (and their sum far above the last-level cache) and the
per-layer work; one is whole.
"""

import ctypes
import math

import numpy as np
import torch

import inferi_amd as I

DEV = "cuda:0"
FMT = {"q4_k": I.Q4_K, "q5_k": I.Q5_K, "q6_k": I.Q6_K, "q8_0": I.Q8_0, "q4_0": I.Q4_0, "f16": I.F16}
KV = {"f16": I.F16, "f32": I.F32}

# hidden, ffn, query heads, KV heads, vocabulary, RoPE base, NeoX pairs with QKV biases
SHAPES = {
    "h896": (896, 4864, 14, 2, 32000, 1e6, True),
    "h1536": (1536, 8960, 12, 2, 32000, 1e6, True),
    "h2048": (2048, 5632, 32, 4, 32000, 1e4, False),
    "h3072": (3072, 8192, 24, 8, 128256, 5e5, False),
    "h4096": (4096, 14336, 32, 8, 128256, 5e5, False),
}


def listed():
    return [
        # one projection of a small model: the shortest call there is, a single launch
        {"name": "gemv_896", "kind": "gemv", "fmt": "q8_0", "rows": 896, "cols": 896},
        # a program that drives a decoder layer op by op, as the reference's op API is used (config 4's widths)
        {"name": "ops_layer_2048", "kind": "ops", "shape": "h2048", "fmt": "q4_k", "kv": "f16", "pos": 300},
        # decode attention on its own at the longest cache of config 3
        {"name": "attention_8192", "kind": "attention", "heads": 32, "kv_heads": 8, "head_size": 128, "kv": "f16",
         "pos": 8191},
        # the chat loop's sampling step over a large vocabulary
        {"name": "sample_topp", "kind": "sample", "n": 128256, "temperature": 0.7, "topp": 0.95},
        # a matrix expanded to f32 at load time (the reference's GGUF reader does it for its CPU path)
        {"name": "dequant_q4_k", "kind": "dequant", "fmt": "q4_k", "rows": 14336, "cols": 4096},
        # one product of a prompt of ragged length in another format
        {"name": "gemm_q8_0_509", "kind": "gemm", "fmt": "q8_0", "rows": 8960, "cols": 1536, "m": 509,
         "accumulate": False},
        # decoding behind a 4096-token prompt (config 5's shape): the headline
        {"name": "decode_4096_ctx4k", "kind": "decode", "shape": "h4096", "layers": 8, "fmt": "q4_k", "head": "q6_k",
         "kv": "f16", "pos": 4103, "steps": 16, "temperature": 0.0},
        # decoding with a small model in whole, early in a conversation (config 4)
        {"name": "decode_2048_whole", "kind": "decode", "shape": "h2048", "layers": 22, "fmt": "q4_k", "head": "q6_k",
         "kv": "f16", "pos": 128, "steps": 16, "temperature": 0.0},
        # a small model in 8 bits with QKV biases and NeoX pairs, the reference's f32 cache, sampled
        {"name": "decode_896_q8_0", "kind": "decode", "shape": "h896", "layers": 12, "fmt": "q8_0", "head": "q8_0",
         "kv": "f32", "pos": 777, "steps": 16, "temperature": 0.7},
        # a chat turn: a short prompt to its first logits
        {"name": "prefill_chat_61", "kind": "prefill", "shape": "h4096", "layers": 4, "fmt": "q4_k", "head": "q6_k",
         "mixed": False, "kv": "f16", "p0": 0, "n": 61},
        # a document added to a conversation, in a file whose value and down matrices are Q6_K
        {"name": "prefill_mixed_1021", "kind": "prefill", "shape": "h3072", "layers": 4, "fmt": "q4_k", "head": "q6_k",
         "mixed": True, "kv": "f16", "p0": 517, "n": 1021},
        # the long prompt of config 5
        {"name": "prefill_4096", "kind": "prefill", "shape": "h4096", "layers": 4, "fmt": "q4_k", "head": "q6_k",
         "mixed": False, "kv": "f16", "p0": 0, "n": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "ops", "attention", "sample", "dequant", "gemm", "decode", "decode", "prefill", "prefill"])
    fmt = rng.choice(["q4_k", "q4_k", "q5_k", "q6_k", "q8_0", "q4_0", "f16"])
    shape = rng.choice(sorted(SHAPES))
    # rows of 896 elements are no whole number of 256-element blocks
    if shape == "h896" and fmt in ("q4_k", "q5_k", "q6_k"):
        fmt = "q8_0"
    kv = rng.choice(["f16", "f16", "f32"])
    if kind == "gemv":
        return {"kind": kind, "fmt": fmt, "rows": _log(rng, 64, 40000), "cols": 256 * _log(rng, 2, 56)}
    if kind == "ops":
        return {"kind": kind, "shape": shape, "fmt": fmt, "kv": kv, "pos": _log(rng, 16, 8000)}
    if kind == "attention":
        kvh = rng.choice([1, 2, 4, 8])
        return {"kind": kind, "heads": kvh * rng.choice([1, 3, 4, 6, 7, 8]), "kv_heads": kvh,
                "head_size": rng.choice([64, 80, 96, 128, 128]), "kv": kv, "pos": _log(rng, 30, 30000)}
    if kind == "sample":
        return {"kind": kind, "n": _log(rng, 2000, 152064), "temperature": round(rng.uniform(0.4, 1.5), 2),
                "topp": rng.choice([0.0, 0.8, 0.9, 0.95, 0.99])}
    if kind == "dequant":
        return {"kind": kind, "fmt": fmt, "rows": _log(rng, 256, 14336), "cols": 256 * _log(rng, 3, 56)}
    if kind == "gemm":
        return {"kind": kind, "fmt": fmt, "rows": _log(rng, 512, 14336), "cols": 256 * _log(rng, 3, 56),
                "m": _log(rng, 8, 2500), "accumulate": rng.random() < 0.5}
    if kind == "decode":
        return {"kind": kind, "shape": shape, "layers": rng.randint(2, 6), "fmt": fmt,
                "head": "q8_0" if shape == "h896" else rng.choice(["q6_k", "q8_0"]), "kv": kv,
                "pos": _log(rng, 20, 12000), "steps": rng.randint(4, 16), "temperature": rng.choice([0.0, 0.0, 0.8])}
    return {"kind": kind, "shape": shape, "layers": rng.randint(2, 4), "fmt": fmt,
            "head": "q8_0" if shape == "h896" else "q6_k", "mixed": fmt == "q4_k" and rng.random() < 0.5, "kv": kv,
            "p0": rng.choice([0, 0, _log(rng, 10, 1500)]), "n": _log(rng, 6, 2600)}


# ---------------------------------------------------------------- inputs --

def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed((seed * 1000003 + stream * 7919 + 12345) % (1 << 62))
    return g


def _randn(shape, g, std=1.0, mean=0.0):
    return torch.randn(shape, generator=g, device=DEV) * std + mean


def _u8(half):
    return half.reshape(-1, 1).view(torch.uint8)


def _codes(nb, qk, g, mean, std, hi):
    return _randn((nb, qk), g, std, mean).round_().clamp_(0, hi).to(torch.uint8)


def _pack_scales(sc, mn):
    """Eight 6-bit scales and mins per block in 12 bytes."""
    lo = torch.cat([sc[:, :4] | (sc[:, 4:] >> 4) << 6, mn[:, :4] | (mn[:, 4:] >> 4) << 6], 1)
    return torch.cat([lo, (sc[:, 4:] & 15) | (mn[:, 4:] & 15) << 4], 1)


def matrix(fmt, rows, cols, g, dense=False):
    """rows x cols weights of standard deviation 0.02: the GGUF blocks (bytes), or with dense their values in f64."""
    if fmt == "f16":
        w = _randn((rows, cols), g, 0.02).half()
        return w.double() if dense else w.view(torch.uint8).reshape(-1)
    qk = 32 if fmt in ("q8_0", "q4_0") else 256
    nb = rows * cols // qk
    vary = 0.8 + 0.4 * torch.rand(nb, generator=g, device=DEV)
    if fmt == "q8_0":
        d = (vary * (0.02 / 40)).half()
        q = _randn((nb, 32), g, 40.0).round_().clamp_(-127, 127).to(torch.int8)
        if dense:
            return (d.double()[:, None] * q.double()).reshape(rows, cols)
        return torch.cat([_u8(d), q.view(torch.uint8)], 1).reshape(-1)
    if fmt == "q4_0":
        d = (vary * (0.02 / 2.7)).half()
        q = _codes(nb, 32, g, 8.0, 2.7, 15)
        if dense:
            return (d.double()[:, None] * (q.double() - 8)).reshape(rows, cols)
        return torch.cat([_u8(d), q[:, :16] | q[:, 16:] << 4], 1).reshape(-1)
    if fmt == "q6_k":
        d = (vary * (0.02 / (96 * 10))).half()
        sc = torch.randint(64, 128, (nb, 16), generator=g, device=DEV, dtype=torch.int16)
        sc = sc * (1 - 2 * torch.randint(0, 2, (nb, 16), generator=g, device=DEV, dtype=torch.int16))
        q = _codes(nb, 256, g, 32.0, 10.0, 63)
        if dense:
            v = (q.double().view(nb, 16, 16) - 32) * sc.double()[:, :, None] * d.double()[:, None, None]
            return v.reshape(rows, cols)
        p = q.view(nb, 2, 4, 32)
        ql = torch.cat([(p[:, :, 0] & 15) | (p[:, :, 2] & 15) << 4, (p[:, :, 1] & 15) | (p[:, :, 3] & 15) << 4], 2)
        qh = p[:, :, 0] >> 4 | (p[:, :, 1] >> 4) << 2 | (p[:, :, 2] >> 4) << 4 | (p[:, :, 3] >> 4) << 6
        return torch.cat([ql.reshape(nb, 128), qh.reshape(nb, 64), sc.to(torch.int8).view(torch.uint8), _u8(d)],
                         1).reshape(-1)
    mid, std, hi = (7.5, 2.7, 15) if fmt == "q4_k" else (15.5, 5.4, 31)
    d = (vary * (0.02 / (48 * std))).half()
    dmin = (d.float() * mid).half()
    sc = torch.randint(33, 63, (nb, 8), generator=g, device=DEV, dtype=torch.uint8)
    mn = sc + torch.randint(0, 2, (nb, 8), generator=g, device=DEV, dtype=torch.uint8)
    q = _codes(nb, 256, g, mid, std, hi)
    if dense:
        v = d.double()[:, None, None] * sc.double()[:, :, None] * q.double().view(nb, 8, 32)
        return (v - (dmin.double()[:, None] * mn.double())[:, :, None]).reshape(rows, cols)
    p = q.view(nb, 4, 2, 32)
    parts = [_u8(d), _u8(dmin), _pack_scales(sc, mn)]
    if fmt == "q5_k":
        qh = torch.zeros((nb, 32), device=DEV, dtype=torch.uint8)
        for j in range(8):
            qh |= (p[:, j // 2, j % 2] >> 4) << j
        parts.append(qh)
    return torch.cat(parts + [((p[:, :, 0] & 15) | (p[:, :, 1] & 15) << 4).reshape(nb, 128)], 1).reshape(-1)


_CTX = None


def context():
    """The program's one context (a device, a stream, the loaded kernels)."""
    global _CTX
    if _CTX is None:
        torch.cuda.init()
        _CTX = I.LlmContext(0)
        # The library's first look-up of a kernel form that a type does not have leaves an error behind in the HIP
        # runtime, which torch raises at its own next launch.  A step of a one-layer model of each type makes those
        # look-ups here, and the error is taken from the runtime.
        cfg = I.Llama2Config(n_layers=1, hidden=256, ffn=512, n_heads=4, n_kv_heads=2, vocab=64, max_pos=16)
        for fmt in FMT.values():
            w, s = I.Llama2Weights.synthetic(_CTX, cfg, 1, fmt, fmt, fmt), I.Llama2State(_CTX, cfg)
            I.Llama2.launch(_CTX, s, w)
            s.close()
            w.close()
        ctypes.CDLL("libamdhip64.so.7").hipGetLastError()
    return _CTX


class _Raw:
    """A device allocation of the library as torch sees it (__cuda_array_interface__); the tensors made of it keep
    the allocation's owner."""

    def __init__(self, ptr, shape, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(shape), "typestr": typestr, "version": 3}


def view(ptr, shape, typestr, owner):
    return torch.as_tensor(_Raw(ptr, shape, typestr, owner), device=DEV)


class Handles:
    """A model's weights and state: freed when neither the case's state nor a tensor on their memory is left."""

    def __init__(self):
        self.w = self.s = None

    def __del__(self):
        if self.s is not None:
            self.s.close()
        if self.w is not None:
            self.w.close()


def _dev_struct(st):
    return torch.from_numpy(np.frombuffer(bytes(st), np.uint8).copy()).to(DEV)


def _kv_rows(shape, kv, g):
    x = _randn(shape, g)
    return x.half() if kv == "f16" else x


class Model:
    """Weights and state of a model case, and their buffers as tensors."""

    def __init__(self, case, seed):
        ctx = self.ctx = context()
        hidden, ffn, heads, kvh, vocab, base, neox = SHAPES[case["shape"]]
        self.first = case["pos"] if case["kind"] == "decode" else case["p0"]
        self.count = case["steps"] if case["kind"] == "decode" else case["n"]
        last = self.first + self.count
        self.cfg = I.Llama2Config(n_layers=case["layers"], hidden=hidden, ffn=ffn, n_heads=heads, n_kv_heads=kvh,
                                  vocab=vocab, max_pos=(last + 64) // 64 * 64, rope_theta=base, rms_eps=1e-5,
                                  kv_dtype=KV[case["kv"]], rope_variant=I.ROPE_NEOX if neox else I.ROPE_ORIGINAL)
        own = Handles()
        self.w = own.w = I.Llama2Weights(ctx, self.cfg)
        for name, fmt, rows, cols, data in tensors(case, seed):
            buf = ctx.alloc(data.numel() * data.element_size())
            view(buf.ptr, (buf.nbytes,), "|u1", own).copy_(data.view(torch.uint8).reshape(-1))
            self.w.set(name, fmt, buf, rows, cols)
        self.s = own.s = I.Llama2State(ctx, self.cfg)
        self.tokens = tokens_of(case, seed)
        kv_type = "<f2" if case["kv"] == "f16" else "<f4"
        self.rows = []
        for l in range(case["layers"]):
            for i, which in enumerate(("key_cache", "value_cache")):
                ptr, _ = self.s.buffer(which, l)
                cache = view(ptr, (self.cfg.max_pos, self.cfg.kv_dim), kv_type, own)
                if self.first:
                    cache[:self.first] = past_rows(case, seed, l, i)
                self.rows.append(cache[self.first:last])
        self.logits = view(self.s.buffer("logits")[0], (vocab,), "<f4", own)
        self.probs = view(self.s.buffer("probs")[0], (vocab,), "<f4", own)
        self.sampled = case.get("temperature", 0.0) != 0.0
        if self.sampled:
            self.s.set_sampler(case["temperature"], 0.95, seed)


def tensors(case, seed, dense=False, only=None):
    """(name, type, rows, cols, data) of a model's tensors, one at a time; data in f64 with dense."""
    hidden, ffn, heads, kvh, vocab, _, bias = SHAPES[case["shape"]]
    kv_dim = hidden // heads * kvh
    f = case["fmt"]
    value = down = "q6_k" if case.get("mixed") else f
    embd = "q8_0" if hidden % 256 else "q4_k"
    todo = [("token_embd.weight", embd, vocab, hidden), ("output.weight", case["head"], vocab, hidden),
            ("output_norm.weight", "norm", 1, hidden)]
    for l in range(case["layers"]):
        b = "blk.%d." % l
        todo += [(b + "attn_norm.weight", "norm", 1, hidden), (b + "attn_q.weight", f, hidden, hidden),
                 (b + "attn_k.weight", f, kv_dim, hidden), (b + "attn_v.weight", value, kv_dim, hidden),
                 (b + "attn_output.weight", f, hidden, hidden), (b + "ffn_norm.weight", "norm", 1, hidden),
                 (b + "ffn_gate.weight", f, ffn, hidden), (b + "ffn_up.weight", f, ffn, hidden),
                 (b + "ffn_down.weight", down, hidden, ffn)]
        if bias:
            todo += [(b + "attn_q.bias", "bias", 1, hidden), (b + "attn_k.bias", "bias", 1, kv_dim),
                     (b + "attn_v.bias", "bias", 1, kv_dim)]
    for i, (name, fmt, rows, cols) in enumerate(todo):
        if only is not None and name != only:
            continue
        g = _gen(seed, i)
        if fmt in ("norm", "bias"):
            v = _randn(cols, g, 0.1, 1.0) if fmt == "norm" else _randn(cols, g, 0.5)
            yield name, I.F32, rows, cols, v.double() if dense else v
        else:
            yield name, FMT[fmt], rows, cols, matrix(fmt, rows, cols, g, dense)


def tokens_of(case, seed):
    n = (case["pos"] + case["steps"]) if case["kind"] == "decode" else (case["p0"] + case["n"])
    return np.random.default_rng(seed).integers(0, SHAPES[case["shape"]][4], n).astype(np.uint32)


def past_rows(case, seed, layer, which):
    """Cache rows of the positions before the case's first."""
    hidden, _, heads, kvh = SHAPES[case["shape"]][:4]
    first = case["pos"] if case["kind"] == "decode" else case["p0"]
    return _kv_rows((first, hidden // heads * kvh), case["kv"], _gen(seed, 100000 + 2 * layer + which))


def _vectors(case, seed):
    """Inputs of the op cases in f32 (or as the op takes them), with dense weights where exact() asks."""
    k = case["kind"]
    if k == "gemv":
        return {"x": _randn(case["cols"], _gen(seed, 2))}
    if k == "gemm":
        x = {"x": _randn((case["m"], case["cols"]), _gen(seed, 2)).half()}
        return {**x, "y": _randn((case["m"], case["rows"]), _gen(seed, 3))} if case["accumulate"] else x
    if k == "sample":
        return {"logits": _randn(case["n"], _gen(seed, 2), 3.0),
                "coin": torch.rand(1, generator=_gen(seed, 3), device=DEV).clamp_(max=0.999)}
    if k == "attention":
        shape = (case["pos"] + 1, case["kv_heads"] * case["head_size"])
        return {"q": _randn(case["heads"] * case["head_size"], _gen(seed, 2)), "k": _kv_rows(shape, case["kv"], _gen(seed, 3)),
                "v": _kv_rows(shape, case["kv"], _gen(seed, 4))}
    hidden, ffn, heads, kvh = SHAPES[case["shape"]][:4]
    shape = (case["pos"] + 1, hidden // heads * kvh)
    return {"x": _randn(hidden, _gen(seed, 2)), "k_cache": _kv_rows(shape, case["kv"], _gen(seed, 3)),
            "v_cache": _kv_rows(shape, case["kv"], _gen(seed, 4)), "n1": _randn(hidden, _gen(seed, 5), 0.1, 1.0),
            "n2": _randn(hidden, _gen(seed, 6), 0.1, 1.0)}


def _ops_mats(case):
    hidden, ffn, heads, kvh = SHAPES[case["shape"]][:4]
    kv_dim = hidden // heads * kvh
    return [("q", hidden, hidden), ("k", kv_dim, hidden), ("v", kv_dim, hidden), ("o", hidden, hidden),
            ("gate", ffn, hidden), ("up", ffn, hidden), ("down", hidden, ffn)]


def prepare(case, seed):
    ctx = context()
    k = case["kind"]
    if k in ("decode", "prefill"):
        st = {"case": case, "m": Model(case, seed)}
        torch.cuda.synchronize()
        return st
    st = {"case": case, "ctx": ctx}
    if k in ("gemv", "gemm", "dequant"):
        st["w"] = matrix(case["fmt"], case["rows"], case["cols"], _gen(seed, 1))
    if k == "dequant":
        st["out"] = torch.empty((case["rows"], case["cols"]), device=DEV)
    else:
        st.update(_vectors(case, seed))
    if k == "gemv":
        st["out"] = torch.empty(case["rows"], device=DEV)
    if k == "gemm":
        st["out"] = torch.empty((case["m"], case["rows"]), device=DEV)
    if k == "sample":
        st["probs"] = torch.empty(case["n"], device=DEV)
        st["index"] = torch.zeros(1, device=DEV, dtype=torch.int32)
    if k in ("attention", "ops"):
        if k == "attention":
            heads, kvh, hs = case["heads"], case["kv_heads"], case["head_size"]
        else:
            hidden, ffn, heads, kvh, _, base, neox = SHAPES[case["shape"]]
            hs = hidden // heads
            st["rms"] = _dev_struct(I.RmsNormConfig(1e-5))
            st["rope"] = _dev_struct(I.RoPEConfig(hs, hs * kvh, case["pos"], base))
            st["variant"] = I.ROPE_NEOX if neox else I.ROPE_ORIGINAL
            for i, (name, rows, cols) in enumerate(_ops_mats(case)):
                st["w_" + name] = matrix(case["fmt"], rows, cols, _gen(seed, 10 + i))
                st["y_" + name] = torch.empty(rows, device=DEV)
            st["xn"] = torch.empty(hidden, device=DEV)
            st["xn2"] = torch.empty(hidden, device=DEV)
        st["params"] = I.AttentionParams(case["pos"] + 1, kvh * hs, heads // kvh, heads, hs, case["pos"])
        st["params_gpu"] = _dev_struct(st["params"])
        st["att"] = torch.empty(heads * hs, device=DEV)
    torch.cuda.synchronize()
    return st


# ------------------------------------------------------------------- run --

def _p(t):
    return t.data_ptr()


def run(state):
    case = state["case"]
    k = case["kind"]
    if k in ("decode", "prefill"):
        m = state["m"]
        m.s.reset(m.tokens, m.first)
        if k == "decode":
            I.Llama2.generate(m.ctx, m.s, m.w, m.count)
        else:
            I.Llama2.prefill(m.ctx, m.s, m.w, m.count - 1)
            I.Llama2.generate(m.ctx, m.s, m.w, 1)
        return {"logits": m.logits, "kv": m.rows, **({"probs": m.probs} if m.sampled else {})}
    ctx = state["ctx"]
    if k == "gemv":
        ctx.matmul_quant_assign(_p(state["out"]), _p(state["w"]), FMT[case["fmt"]], case["rows"], case["cols"],
                                _p(state["x"]))
        return state["out"]
    if k == "gemm":
        if case["accumulate"]:
            # a residual product adds to a stream that was written just before
            ctx.dequant(_p(state["out"]), _p(state["y"]), I.F32, state["y"].numel())
        ctx.gemm_quant(_p(state["out"]), _p(state["w"]), FMT[case["fmt"]], case["rows"], case["cols"], _p(state["x"]),
                       case["m"], case["accumulate"])
        return state["out"]
    if k == "dequant":
        ctx.dequant(_p(state["out"]), _p(state["w"]), FMT[case["fmt"]], case["rows"] * case["cols"])
        return state["out"]
    if k == "sample":
        ctx.sample(_p(state["logits"]), _p(state["probs"]), case["n"], case["temperature"], case["topp"],
                   _p(state["coin"]), _p(state["index"]))
        return [state["probs"], state["index"]]
    if k == "attention":
        I.BatchedMultiqueryAttention.launch(ctx, state["params"], _p(state["params_gpu"]), _p(state["q"]), _p(state["k"]),
                                            _p(state["v"]), KV[case["kv"]], _p(state["att"]))
        return state["att"]
    return _ops_layer(ctx, state)


def _ops_layer(ctx, s):
    """One decoder layer by single ops, in the order of the reference's Llama2::launch."""
    case = s["case"]
    fmt = FMT[case["fmt"]]
    hidden, ffn, heads, kvh = SHAPES[case["shape"]][:4]
    kv_dim = hidden // heads * kvh

    def mul(name, x):
        y = s["y_" + name]
        ctx.matmul_quant_assign(_p(y), _p(s["w_" + name]), fmt, y.numel(), x.numel(), _p(x))
        return y

    ctx.rms_norm_assign(_p(s["rms"]), _p(s["xn"]), _p(s["x"]), _p(s["n1"]), hidden)
    q, k, v = mul("q", s["xn"]), mul("k", s["xn"]), mul("v", s["xn"])
    ctx.rope(s["variant"], _p(s["rope"]), _p(q), hidden, _p(k), kv_dim)
    I.BatchedMultiqueryAttention.launch(ctx, s["params"], _p(s["params_gpu"]), _p(q), _p(s["k_cache"]), _p(s["v_cache"]),
                                        KV[case["kv"]], _p(s["att"]))
    o = mul("o", s["att"])
    ctx.add_assign(_p(o), _p(s["x"]), hidden)
    ctx.rms_norm_assign(_p(s["rms"]), _p(s["xn2"]), _p(o), _p(s["n2"]), hidden)
    g, u = mul("gate", s["xn2"]), mul("up", s["xn2"])
    ctx.silu(_p(g), _p(u), ffn)
    out = mul("down", g)
    ctx.add_assign(_p(out), _p(o), hidden)
    return {"q": q, "k": k, "v": v, "att": s["att"], "o": o, "h": g, "out": out}


# ------------------------------------------------- work and tolerances --

def _size(fmt, rows, cols):
    return rows * (cols * 4 if fmt in ("norm", "bias") else I.row_bytes(FMT[fmt], cols))


def work(case):
    k = case["kind"]
    if k == "gemv":
        r, c = case["rows"], case["cols"]
        return {"bytes": _size(case["fmt"], r, c) + 4 * (r + c), "flops": 2 * r * c}
    if k == "gemm":
        r, c, m = case["rows"], case["cols"], case["m"]
        b = _size(case["fmt"], r, c) + 2 * m * c + 4 * m * r * (2 if case["accumulate"] else 1)
        return {"bytes": b, "flops": 2 * r * c * m}
    if k == "dequant":
        r, c = case["rows"], case["cols"]
        return {"bytes": _size(case["fmt"], r, c) + 4 * r * c, "flops": 2 * r * c}
    if k == "sample":
        return {"bytes": 8 * case["n"], "flops": 4 * case["n"]}
    if k == "attention":
        b, f = _attn_work(case["heads"], case["kv_heads"], case["head_size"], case["kv"], case["pos"] + 1)
        return {"bytes": b + 8 * case["heads"] * case["head_size"], "flops": f}
    hidden, ffn, heads, kvh, vocab, _, bias = SHAPES[case["shape"]]
    hs = hidden // heads
    kv_dim = hs * kvh
    f = case["fmt"]
    value = down = "q6_k" if case.get("mixed") else f
    parts = [(f, hidden, hidden), (f, kv_dim, hidden), (value, kv_dim, hidden), (f, hidden, hidden), (f, ffn, hidden),
             (f, ffn, hidden), (down, hidden, ffn)]
    layer_b = sum(_size(*p) for p in parts) + 8 * hidden + (4 * (hidden + 2 * kv_dim) if bias else 0)
    layer_f = sum(2 * r * c for _, r, c in parts)
    if k == "ops":
        b, fl = _attn_work(heads, kvh, hs, case["kv"], case["pos"] + 1)
        return {"bytes": layer_b + b + 4 * (6 * hidden + 2 * kv_dim + ffn), "flops": layer_f + fl}
    head_b, head_f = _size(case["head"], vocab, hidden) + 4 * vocab, 2 * vocab * hidden
    L = case["layers"]
    esz = 2 if case["kv"] == "f16" else 4

    def step(pos):
        b, fl = _attn_work(heads, kvh, hs, case["kv"], pos + 1)
        return L * (layer_b + b + 2 * esz * kv_dim) + head_b, L * (layer_f + fl) + head_f

    if k == "decode":
        every = [step(case["pos"] + i) for i in range(case["steps"])]
        return {"bytes": sum(b for b, _ in every), "flops": sum(fl for _, fl in every)}
    # the prompt's weights are read once for all of its tokens; the last layer forms logits for the last token alone, so
    # that the other tokens need only its K and V
    n, p0 = case["n"], case["p0"]
    keys = sum(p0 + i + 1 for i in range(n))
    fl = (L - 1) * (n * layer_f + 4 * heads * hs * keys) + 4 * n * kv_dim * hidden + step(p0 + n - 1)[1] - (L - 1) * layer_f
    b = L * (layer_b + 2 * esz * kv_dim * (p0 + 2 * n)) + head_b
    return {"bytes": b, "flops": fl}


def _attn_work(heads, kvh, hs, kv, T):
    return 2 * T * kvh * hs * (2 if kv == "f16" else 4), 4 * T * heads * hs


def tolerance(case):
    k = case["kind"]
    if k == "dequant":
        return "exact"
    if k in ("gemv", "attention", "sample"):
        return {"rel": 4e-6, "max": 4e-5}  # f32 sums (two orders: 5e-7, 2e-6)
    if k == "ops":
        return {"rel": 8e-6, "max": 6e-5}  # f32 sums, through a layer (two orders: 1e-6, 8e-6)
    if k == "gemm":
        return {"rel": 1e-3, "max": 4e-3}  # both operands rounded to f16 (against 64 bits: 2e-4, 1e-3)
    if k == "decode" and case["kv"] == "f32":
        return {"rel": 3e-5, "max": 2e-4}  # f32 sums, through the layers (two orders: 5e-6, 2e-5)
    if k == "decode":
        return {"rel": 4e-4, "max": 4e-3}  # and cache rows in f16, a few of which round the other way (1e-4, 1e-3)
    return {"rel": 7e-3, "max": 4e-2}  # f16 operands, through the layers (against 64 bits: 2e-3, 1e-2)


# ----------------------------------------------------------------- exact --

def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + float(np.float32(1e-5))) * w


def _rope(x, pos, hs, base, neox):
    """x [n, heads * hs] rotated at positions pos [n]; the angles are the op's f32 ones."""
    j = np.arange(hs // 2, dtype=np.float32)
    theta = np.power(np.float64(np.float32(base)), (-(2 * j) / np.float32(hs)).astype(np.float64)).astype(np.float32)
    ang = (pos.float()[:, None] * torch.from_numpy(theta).to(DEV)[None, :]).double()
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    y = x.view(x.shape[0], -1, hs)
    a, b = (y[..., :hs // 2], y[..., hs // 2:]) if neox else (y[..., 0::2], y[..., 1::2])
    u, v = a * c - b * s, a * s + b * c
    return (torch.cat([u, v], -1) if neox else torch.stack([u, v], -1)).reshape(x.shape)


def _attend(q, k, v, heads, kvh, first):
    """Causal attention of q [n, heads * hs] at positions first .. over rows k, v [first + n, kvh * hs]."""
    n, T, hs = q.shape[0], k.shape[0], q.shape[1] // heads
    out = torch.empty_like(q)
    mask = torch.arange(T, device=DEV)[None, :] > torch.arange(first, first + n, device=DEV)[:, None]
    for h in range(heads):
        c = h // (heads // kvh) * hs
        s = (q[:, h * hs:(h + 1) * hs] @ k[:, c:c + hs].t()) / math.sqrt(hs)
        out[:, h * hs:(h + 1) * hs] = torch.softmax(s.masked_fill_(mask, -math.inf), -1) @ v[:, c:c + hs]
    return out


def exact(case, seed):
    k = case["kind"]
    if k == "dequant":
        return matrix(case["fmt"], case["rows"], case["cols"], _gen(seed, 1), True)
    if k in ("gemv", "gemm"):
        x = _vectors(case, seed)
        y = x["x"].double() @ matrix(case["fmt"], case["rows"], case["cols"], _gen(seed, 1), True).t()
        return y + x["y"].double() if case.get("accumulate") else y
    x = _vectors(case, seed) if k not in ("decode", "prefill") else None
    if k == "sample":
        return [torch.softmax(x["logits"].double() / float(np.float32(case["temperature"])), 0), None]
    if k == "attention":
        return _attend(x["q"].double()[None], x["k"].double(), x["v"].double(), case["heads"], case["kv_heads"],
                       case["pos"])[0]
    hidden, ffn, heads, kvh, vocab, base, neox = SHAPES[case["shape"]]
    hs = hidden // heads
    silu = torch.nn.functional.silu
    if k == "ops":
        w = {name: matrix(case["fmt"], r, c, _gen(seed, 10 + i), True) for i, (name, r, c) in enumerate(_ops_mats(case))}
        at = torch.tensor([case["pos"]], device=DEV)
        x0 = x["x"].double()[None]
        xn = _rms(x0, x["n1"].double())
        q, kk = (_rope(xn @ w[n].t(), at, hs, base, neox) for n in "qk")
        v = xn @ w["v"].t()
        att = _attend(q, x["k_cache"].double(), x["v_cache"].double(), heads, kvh, case["pos"])
        o = att @ w["o"].t() + x0
        xn = _rms(o, x["n2"].double())
        h = silu(xn @ w["gate"].t()) * (xn @ w["up"].t())
        out = h @ w["down"].t() + o
        return {"q": q[0], "k": kk[0], "v": v[0], "att": att[0], "o": o[0], "h": h[0], "out": out[0]}

    first = case["pos"] if k == "decode" else case["p0"]
    tok = torch.from_numpy(tokens_of(case, seed)[first:].astype(np.int64)).to(DEV)
    n = tok.numel()
    at = torch.arange(first, first + n, device=DEV)

    def one(name):
        for t in tensors(case, seed, True, name):
            return t[4]
        return 0.0

    x = one("token_embd.weight")[tok]
    rows = []
    for l in range(case["layers"]):
        b = "blk.%d." % l
        xn = _rms(x, one(b + "attn_norm.weight"))
        kk = _rope(xn @ one(b + "attn_k.weight").t() + one(b + "attn_k.bias"), at, hs, base, neox)
        v = xn @ one(b + "attn_v.weight").t() + one(b + "attn_v.bias")
        rows += [kk, v]
        if l + 1 == case["layers"]:  # only the last token's logits are asked for
            x, xn = x[-1:], xn[-1:]
        q = _rope(xn @ one(b + "attn_q.weight").t() + one(b + "attn_q.bias"), at[-x.shape[0]:], hs, base, neox)
        past = [past_rows(case, seed, l, i).double() for i in range(2)]
        att = _attend(q, torch.cat([past[0], kk]), torch.cat([past[1], v]), heads, kvh, first + n - x.shape[0])
        x = x + att @ one(b + "attn_output.weight").t()
        xn = _rms(x, one(b + "ffn_norm.weight"))
        h = silu(xn @ one(b + "ffn_gate.weight").t()) * (xn @ one(b + "ffn_up.weight").t())
        x = x + h @ one(b + "ffn_down.weight").t()
    logits = (_rms(x, one("output_norm.weight")) @ one("output.weight").t())[0]
    out = {"logits": logits, "kv": rows}
    if case.get("temperature", 0.0):
        out["probs"] = torch.softmax(logits / float(np.float32(case["temperature"])), 0)
    return out
