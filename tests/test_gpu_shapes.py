"""GPU parity for the model shapes beyond the common ones, against the oracle:
any number of query heads per KV head (Qwen2-0.5B's 7, Qwen2-1.5B's 6,
Llama-3.2-3B's 3, groups of more than 8 that one workgroup splits), head
sizes that are multiples of 8 up to 128, and positions past 65,536.  The
reference's decode attention takes any kv_mul and head size
(fused_attention.rs:80-92) and sizes the cache to context_length
(transformer.rs:85-104).

Bars: the attention op within 1e-3 of max(|e|, 1) (north_star).  Decode
steps: logits normwise within 1e-3 and elementwise within max(1e-3, the
distance of the f32-order oracle from the f64 one), as test_c5_8b_first_steps
sets it.  Weights are N(0, 0.02), the scale of trained models (at 0.05 and
hidden 3072 the activations grow so that any f32 summation order, the
device's or the f32-order oracle's, lands 1-2.5e-3 from exact in two
layers, and which of the two lands closer is chance).  Prefill
(f16 operands on the matrix cores): as test_c5_prefill_4095_tokens, logits
within 5e-2, KV rows normwise within 2e-2, and layer-0 K/V rows within the
f16 rounding bound."""

import numpy as np
import pytest

import oracle as O
from tests.test_gpu_configs import check_layer0_bound
from tests.test_gpu_model import assert_close, oracle_model, run_steps
from tests.test_gpu_ops import _attn_case

pytestmark = pytest.mark.gpu

# (n_heads, n_kv_heads, head_size): group sizes 7, 6, 7, 3, 5, 12, 32, 64, 10,
# 4, 4, 4, 2, 1 (past 4, the split kernel's workgroups hold up to four heads
# at these lengths) and head sizes 64, 128, 32, 80, 96, 112, 40, 8
SHAPES = [(14, 2, 64), (12, 2, 128), (28, 4, 128), (24, 8, 128), (40, 8, 128), (24, 2, 128), (32, 1, 64),
          (64, 1, 32), (20, 2, 80), (16, 4, 96), (8, 2, 112), (16, 4, 32), (6, 3, 40), (4, 4, 8)]


@pytest.mark.parametrize("kv_f16", [True, False], ids=["f16", "f32"])
@pytest.mark.parametrize("nh,nkv,hs", SHAPES, ids=[f"{a}q{b}kv{c}" for a, b, c in SHAPES])
def test_attention_any_group_and_head_size(ctx, oracle_lib, kv_f16, nh, nkv, hs):
    rng = np.random.default_rng(nh * 1000 + nkv * 10 + hs)
    for pos in (0, 1, 100, 777):
        got, ref = _attn_case(ctx, nh, nkv, hs, 800, pos, kv_f16, rng)
        assert_close(got, ref, what=f"pos={pos}")


@pytest.mark.timeout(300)
@pytest.mark.parametrize("nh,nkv,hs", [(8, 2, 128), (14, 2, 64)])
def test_attention_past_65536_positions(ctx, oracle_lib, nh, nkv, hs):
    """A 131,072-row f16 cache attended at positions past 65,536 (more
    positions than 256 splits of 256 hold): the 1e-3 bar, and normwise within
    1e-4 (q scaled so that the softmax is peaked, not a flat average)."""
    import inferi_amd as I

    L = 131072
    rng = np.random.default_rng(hs)
    kv_dim = nkv * hs
    kc = O.encode_f16(rng.standard_normal((L, kv_dim), np.float32))
    vc = O.encode_f16(rng.standard_normal((L, kv_dim), np.float32))
    dk, dv, do = ctx.upload(kc), ctx.upload(vc), ctx.alloc(nh * hs * 4)
    try:
        for pos in (65535, 65536, 100003, L - 1):
            q = (3.0 * rng.standard_normal(nh * hs)).astype(np.float32)
            p = I.AttentionParams(L, kv_dim, nh // nkv, nh, hs, pos)
            dp = ctx.upload(np.frombuffer(bytes(p), np.uint8))
            I.BatchedMultiqueryAttention.launch(ctx, p, dp, ctx.upload(q), dk, dv, I.F16, do)
            got = do.download(np.float32, nh * hs)
            ref = O.attention(q, kc, vc, nh, nkv, hs, pos, True)
            assert_close(got, ref, what=f"pos={pos}")
            nw = float(np.abs(got.astype(np.float64) - ref).max() / np.abs(ref).max())
            assert nw <= 1e-4, f"pos={pos}: normwise {nw:.3e}"
    finally:
        dk.free()
        dv.free()
        do.free()


@pytest.mark.timeout(300)
def test_decode_steps_past_65536_positions(ctx, oracle_lib):
    """A model whose cache holds 131,072 positions decodes at positions
    65,536 and 131,070 (graph-replayed steps) over planted cache rows, equal
    to the oracle's forward over the same rows."""
    import inferi_amd as I

    cfg = I.Llama2Config(n_layers=2, hidden=256, ffn=512, n_heads=4, n_kv_heads=2, vocab=1000, max_pos=131072,
                         rope_theta=500000.0, rms_eps=1e-5, kv_dtype=I.F16)
    w = I.Llama2Weights.synthetic(ctx, cfg, seed=77, std=0.05)
    s = I.Llama2State(ctx, cfg)
    try:
        m = oracle_model(cfg, w)
        rng = np.random.default_rng(78)
        for layer in range(cfg.n_layers):
            for name, which in (("key_cache", "k"), ("value_cache", "v")):
                rows = O.encode_f16(rng.standard_normal((cfg.max_pos, cfg.kv_dim), np.float32))
                m.set_kv_rows(layer, which, rows)
                ptr, n = s.buffer(name, layer)
                assert n >= rows.nbytes
                ctx._check(I.lib().ifr_upload(ctx.h, ptr, rows.ctypes.data, rows.nbytes))
        for pos, tok in ((65536, 321), (131070, 999)):
            prompt = np.zeros(pos + 2, np.uint32)
            prompt[pos] = tok
            s.reset(prompt, pos)
            I.Llama2.generate(ctx, s, w, 1, use_graph=True)
            got = s.read("logits")
            ref = m.forward(tok, pos)
            assert_close(got, ref, what=f"pos {pos}")
            kv = s.read("key_cache", np.uint16, 1).reshape(cfg.max_pos, cfg.kv_dim)[pos]
            assert_close(O.decode_f16(kv), O.decode_f16(m.kv_cache(1, "k")[pos]), tol=2e-3, what=f"layer 1 k row {pos}")
    finally:
        s.close()
        w.close()


# model shapes: (name, config, matrix / head / embedding type, QKV biases + NeoX)
MODELS = {
    # Qwen2-0.5B: hidden 896, 14 query heads over 2 KV heads of 64
    "qwen2_0.5b": (dict(n_layers=2, hidden=896, ffn=4864, n_heads=14, n_kv_heads=2, vocab=1500,
                        rope_theta=1000000.0, rms_eps=1e-6), "Q8_0", True),
    # Qwen2-1.5B: hidden 1536, 12 over 2 of 128
    "qwen2_1.5b": (dict(n_layers=2, hidden=1536, ffn=8960, n_heads=12, n_kv_heads=2, vocab=1500,
                        rope_theta=1000000.0, rms_eps=1e-6), "Q8_0", True),
    # Llama-3.2-3B: hidden 3072, 24 over 8 of 128
    "llama3.2_3b": (dict(n_layers=2, hidden=3072, ffn=8192, n_heads=24, n_kv_heads=8, vocab=1500,
                         rope_theta=500000.0, rms_eps=1e-5), "Q4_K", False),
    # head size 80, 32 over 8
    "hs80": (dict(n_layers=2, hidden=2560, ffn=6912, n_heads=32, n_kv_heads=8, vocab=1500,
                  rope_theta=10000.0, rms_eps=1e-5), "Q4_K", False),
    # 24 query heads of 32 over 2 KV heads
    "g12_hs32": (dict(n_layers=2, hidden=768, ffn=2048, n_heads=24, n_kv_heads=2, vocab=1500,
                      rope_theta=10000.0, rms_eps=1e-5), "Q8_0", False),
}


def model(ctx, name, max_pos):
    import inferi_amd as I

    c, mat, qwen = MODELS[name]
    cfg = I.Llama2Config(max_pos=max_pos, kv_dtype=I.F16, rope_variant=I.ROPE_NEOX if qwen else I.ROPE_ORIGINAL, **c)
    dt = getattr(I, mat)
    w = I.Llama2Weights.synthetic(ctx, cfg, seed=sum(map(ord, name)), std=0.02, mat_dtype=dt, head_dtype=dt,
                                  embd_dtype=dt, qkv_bias=qwen)
    return cfg, w


def scaled(a, e):
    a = np.asarray(a, np.float64)
    return float((np.abs(a - e) / np.maximum(np.abs(e), 1.0)).max())


@pytest.mark.parametrize("mode", ["fused", "unfused", "graph"])
@pytest.mark.parametrize("name", list(MODELS))
def test_decode_model_shapes(ctx, oracle_lib, name, mode):
    """20 steps (a 5-token prompt, then greedy) against the f64 oracle and the
    f32-order oracle; ids where the margin allows; KV rows of the first and
    last layer."""
    import inferi_amd as I

    n = 20
    cfg, w = model(ctx, name, 48)
    s = I.Llama2State(ctx, cfg)
    try:
        prompt = [3, 999, 41, 0, 512]
        logits, toks = run_steps(ctx, s, w, prompt, n, mode)
        m, m32 = oracle_model(cfg, w), oracle_model(cfg, w)
        worst, worst_floor, ids = 0.0, 0.0, 0
        for pos in range(n):
            ref = m.forward(int(toks[pos]), pos)
            with O.f32_accumulation():
                ref32 = m32.forward(int(toks[pos]), pos)
            floor, err = scaled(ref32, ref), scaled(logits[pos], ref)
            normwise = float(np.abs(logits[pos].astype(np.float64) - ref).max() / np.abs(ref).max())
            worst, worst_floor = max(worst, err), max(worst_floor, floor)
            assert normwise <= 1e-3, f"pos {pos}: normwise {normwise:.3e}"
            assert err <= max(1e-3, floor), f"pos {pos}: scaled error {err:.3e}, f32 floor {floor:.3e}"
            if pos + 1 < len(prompt):
                assert int(toks[pos + 1]) == prompt[pos + 1]
                continue
            top2 = np.partition(ref, -2)[-2:]
            if top2[1] - top2[0] > 2 * np.abs(logits[pos].astype(np.float64) - ref).max():
                assert int(toks[pos + 1]) == O.argmax(ref), f"token at {pos + 1}"
                ids += 1
        for layer in (0, cfg.n_layers - 1):
            for which, key in (("key_cache", "k"), ("value_cache", "v")):
                got = O.decode_f16(s.read(which, np.uint16, layer).reshape(cfg.max_pos, cfg.kv_dim)[:n])
                assert_close(got, O.decode_f16(m.kv_cache(layer, key)[:n]), tol=2e-3, what=f"{which} layer {layer}")
        print(f"{name} {mode}: logits within {worst:.2e} of the f64 oracle (f32-order oracle {worst_floor:.2e}), "
              f"{ids}/{n - len(prompt) + 1} greedy ids compared", flush=True)
        assert ids >= (n - len(prompt) + 1) // 2
    finally:
        s.close()
        w.close()


@pytest.mark.timeout(300)
@pytest.mark.parametrize("tile", [0, 256])
@pytest.mark.parametrize("name", list(MODELS))
def test_prefill_model_shapes(ctx, oracle_lib, name, tile):
    """A 150-token prompt: 149 tokens through ifr_llama2_prefill, then 12
    decode steps, every step's logits and every layer's KV rows against the
    oracle over the same sequence; with the GEMM tiles chosen by shape (32 to
    256 wide here, by the product) and forced to 256 x 256 (stacked QKV
    products with biases and NeoX pairs, odd query groups, rows and tokens past
    the matrix edges)."""
    import inferi_amd as I

    P, N = 150, 12
    cfg, w = model(ctx, name, P + N + 4)
    s = I.Llama2State(ctx, cfg)
    ctx.set_option("pf_tile", tile)
    try:
        prompt = np.random.default_rng(11).integers(0, cfg.vocab, P).tolist()
        s.reset(prompt, 0)
        I.Llama2.prefill(ctx, s, w, P - 1)
        got = []
        for _ in range(N):
            I.Llama2.generate(ctx, s, w, 1, use_graph=True)
            got.append(s.read("logits").copy())
        toks = s.tokens(0, P + N)
        m = oracle_model(cfg, w)
        worst = 0.0
        for pos in range(P + N - 1):
            ref = m.forward(int(toks[pos]), pos)
            if pos >= P - 1:
                g = got[pos - (P - 1)].astype(np.float64)
                e = float((np.abs(g - ref) / np.maximum(np.abs(ref), 1.0)).max())
                worst = max(worst, e)
                assert e <= 5e-2, f"step at pos {pos}: {e:.3e}"
        bound = None if MODELS[name][2] else check_layer0_bound(s, cfg, w, [int(t) for t in toks[: P - 1]])
        for layer in range(cfg.n_layers):
            for which, key in (("key_cache", "k"), ("value_cache", "v")):
                e = O.decode_f16(m.kv_cache(layer, key)[: P + N - 1]).astype(np.float64)
                g = O.decode_f16(s.read(which, np.uint16, layer).reshape(cfg.max_pos, cfg.kv_dim)[: P + N - 1])
                nw = float(np.abs(g - e).max() / np.abs(e).max())
                assert nw <= 2e-2, f"layer {layer} {which}: normwise {nw:.3e}"
        print(f"{name}: prefill {P - 1} + {N} steps, logits within {worst:.2e}, layer-0 K/V at "
              f"{bound if bound is None else round(bound, 3)} of the f16 bound", flush=True)
    finally:
        ctx.set_option("pf_tile", 0)
        s.close()
        w.close()


@pytest.mark.timeout(300)
def test_decode_position_buckets(ctx, oracle_lib):
    """The attention launch is sized for the bucket of 256 positions the host
    expects (the graph is captured again when the position leaves it).  A
    20,000-position cache decoded from position 240 across the 256 and 512
    bucket edges, with the graph and without; then the device position moved
    past the host's bucket behind its back (the split kernel's fallback to
    chunks computed from the position it reads).  Positions up to 511 take
    the one-kernel attention, later ones the split one.  Logits against the
    oracle over the same planted cache rows."""
    import inferi_amd as I

    cfg = I.Llama2Config(n_layers=2, hidden=256, ffn=512, n_heads=4, n_kv_heads=1, vocab=1000, max_pos=20000,
                         rope_theta=10000.0, rms_eps=1e-5, kv_dtype=I.F16)
    w = I.Llama2Weights.synthetic(ctx, cfg, seed=91, std=0.05)
    try:
        m = oracle_model(cfg, w)
        rng = np.random.default_rng(92)
        planted = {}
        for layer in range(cfg.n_layers):
            for which in ("k", "v"):
                planted[layer, which] = O.encode_f16(rng.standard_normal((cfg.max_pos, cfg.kv_dim), np.float32))

        def plant(s):
            for (layer, which), rows in planted.items():
                m.set_kv_rows(layer, which, rows)
                ptr, n = s.buffer("key_cache" if which == "k" else "value_cache", layer)
                ctx._check(I.lib().ifr_upload(ctx.h, ptr, rows.ctypes.data, rows.nbytes))

        p0, n = 240, 300
        toks = rng.integers(0, cfg.vocab, p0 + n + 1).astype(np.uint32)
        for use_graph in (True, False):
            s = I.Llama2State(ctx, cfg)
            try:
                plant(s)
                s.reset(toks, p0)
                got = []
                for _ in range(n):
                    I.Llama2.generate(ctx, s, w, 1, use_graph=use_graph)
                    got.append(s.read("logits").copy())
                for i, pos in enumerate(range(p0, p0 + n)):
                    ref = m.forward(int(toks[pos]), pos)
                    if i % 25 == 0 or pos in (255, 256, 511, 512):
                        assert_close(got[i], ref, what=f"graph={use_graph} pos {pos}")
                # a position the host does not know: 5000 (its bucket ends at 768)
                s.reset(toks, p0 + n)
                ptr, _ = s.buffer("pos")
                jump = np.array([5000], np.uint32)
                ctx._check(I.lib().ifr_upload(ctx.h, ptr, jump.ctypes.data, 4))
                big = np.zeros(5002, np.uint32)
                big[5000] = 77
                tok_ptr, _ = s.buffer("tokens")
                ctx._check(I.lib().ifr_upload(ctx.h, tok_ptr, big.ctypes.data, big.nbytes))
                I.Llama2.generate(ctx, s, w, 1, use_graph=use_graph)
                assert_close(s.read("logits"), m.forward(77, 5000), what=f"graph={use_graph} pos 5000 (fallback)")
            finally:
                s.close()
    finally:
        w.close()


@pytest.mark.parametrize("kv_f16", [True, False], ids=["f16", "f32"])
@pytest.mark.parametrize("nh,nkv,hs", [(7, 1, 16), (6, 2, 48), (14, 2, 64), (10, 2, 80), (8, 8, 112), (40, 8, 128)])
def test_attention_one_kernel_edges(ctx, oracle_lib, kv_f16, nh, nkv, hs):
    """Short contexts at the edges of the one-kernel form's waves and batches,
    with head sizes short of the padding, up to the longest it is taken for
    (1024 positions of up to 64 dims, 512 of up to 128; the split kernel's
    where the shape's line lies lower) and one past it.  The
    outputs are averages of at most 1025 N(0, 1) values in f32: 1e-5 leaves
    twenty times the largest difference two summation orders show."""
    rng = np.random.default_rng(nh * 100 + hs)
    top = 1024 if hs <= 64 else 512
    for T in (2, 31, 32, 33, 129, 256, 257, top - 1, top, top + 1):
        got, ref = _attn_case(ctx, nh, nkv, hs, top + 1, T - 1, kv_f16, rng)
        assert np.abs(got - ref).max() <= 1e-5, f"{T} positions"


def _split_group(n_cu, nh, nkv, hs, T, f16):
    """Query heads per workgroup of the split kernel for T positions, by the
    launch's rule."""
    kv_mul, hsp = nh // nkv, 64 if hs <= 64 else 128
    S = max(1, min(256, -(-T // (8192 // hsp))))
    n8, n4 = -(-kv_mul // 8), -(-kv_mul // 4)
    r4, r8 = -(-nkv * S * n4 // n_cu), -(-nkv * S * n8 // n_cu)
    eight = -(-kv_mul // n8) == 8 or kv_mul == 7
    four = T * nkv * hs * (4 if f16 else 8) < 8000000 and (r4 <= 1 or (f16 and (r4 <= r8 or eight)))
    return -(-kv_mul // (n4 if four else n8))


@pytest.mark.parametrize("kv_f16", [True, False], ids=["f16", "f32"])
@pytest.mark.parametrize("nh,nkv,hs", [(40, 8, 64), (48, 8, 64), (56, 8, 64), (64, 8, 64), (40, 8, 128), (48, 8, 128),
                                       (56, 8, 128), (64, 8, 128), (24, 2, 128), (32, 2, 128), (20, 2, 80), (12, 1, 64)])
def test_attention_split_group_edges(ctx, oracle_lib, kv_f16, nh, nkv, hs):
    """The split kernel with at most four query heads per workgroup and with
    five to eight, on both sides of each context where the launch changes
    between them, for every group size, padded head size and cache type.  The
    outputs are averages of N(0, 1) values: scores of N(0, 1) in f32 are off by
    1e-6 at most, and so, relatively, are their weights and the outputs; 1e-5
    allows ten times that."""
    n_cu = ctx.device_info()[1]
    rng = np.random.default_rng(nh * 100 + hs)
    lo = 65536 // (64 if hs <= 64 else 128) + 1
    gt = {T: _split_group(n_cu, nh, nkv, hs, T, kv_f16) for T in range(lo, 12000)}
    edges = [T for T in range(lo, 11999) if gt[T] != gt[T + 1]][:3]
    assert edges and max(gt[T + d] for T in edges for d in (0, 1)) > 4
    for T in edges:
        for n in (T, T + 1):
            got, ref = _attn_case(ctx, nh, nkv, hs, n, n - 1, kv_f16, rng)
            assert np.abs(got - ref).max() <= 1e-5, f"{n} positions, {gt[n]} heads"


def _one_kernel(nh, nkv, hs, T, f16):
    """Whether T positions run in the one-kernel form, by the launch's rule."""
    kv_mul, elems = nh // nkv, T * (64 if hs <= 64 else 128)
    if hs % 16 or elems > 65536:
        return False
    if elems > 32768:
        return f16 and kv_mul >= 6
    return elems <= 16384 or kv_mul >= 2 or T * nkv * hs < 500000


@pytest.mark.parametrize("kv_f16", [True, False], ids=["f16", "f32"])
@pytest.mark.parametrize("nh,nkv,hs", [(4, 4, 24), (8, 8, 64), (16, 16, 64), (32, 32, 64), (8, 4, 64), (14, 2, 64),
                                       (16, 16, 80), (16, 16, 128), (32, 32, 128), (8, 2, 112), (12, 2, 128)])
def test_attention_one_kernel_lines(ctx, oracle_lib, kv_f16, nh, nkv, hs):
    """Both sides of the line between the one-kernel form and the split one,
    wherever the shape's cache type, sharing and size put it.  The bound as in
    test_attention_one_kernel_edges."""
    rng = np.random.default_rng(nh * 100 + hs)
    edges = [T for T in range(1, 1100) if _one_kernel(nh, nkv, hs, T, kv_f16) != _one_kernel(nh, nkv, hs, T + 1, kv_f16)]
    assert len(edges) == (1 if hs % 16 == 0 else 0)
    for T in edges or [256]:
        for n in (T, T + 1):
            got, ref = _attn_case(ctx, nh, nkv, hs, n, n - 1, kv_f16, rng)
            assert np.abs(got - ref).max() <= 1e-5, f"{n} positions"


@pytest.mark.timeout(300)
@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("p0,n,host_end", [(100, 3, 256), (1270, 20, 1536), (1526, 20, 1792)])
def test_decode_past_the_host_bound(ctx, oracle_lib, use_graph, p0, n, host_end):
    """Steps whose attention takes the one-kernel form (64 dims, up to 256
    positions) and the split one (across the edges of two buckets), each step
    against the oracle over the same planted rows; then the device position
    moved past the host's bound, where the kernels discard the rows they
    loaded before they knew it: one position past, and thousands."""
    import inferi_amd as I

    cfg = I.Llama2Config(n_layers=2, hidden=256, ffn=512, n_heads=4, n_kv_heads=1, vocab=1000, max_pos=8000,
                         rope_theta=10000.0, rms_eps=1e-5, kv_dtype=I.F16)
    w = I.Llama2Weights.synthetic(ctx, cfg, seed=93, std=0.05)
    s = I.Llama2State(ctx, cfg)
    try:
        m = oracle_model(cfg, w)
        rng = np.random.default_rng(p0)
        for layer in range(cfg.n_layers):
            for name, which in (("key_cache", "k"), ("value_cache", "v")):
                rows = O.encode_f16(rng.standard_normal((cfg.max_pos, cfg.kv_dim), np.float32))
                m.set_kv_rows(layer, which, rows)
                ptr, _ = s.buffer(name, layer)
                ctx._check(I.lib().ifr_upload(ctx.h, ptr, rows.ctypes.data, rows.nbytes))
        toks = rng.integers(0, cfg.vocab, cfg.max_pos - 1).astype(np.uint32)
        s.reset(toks, p0)
        for pos in range(p0, p0 + n):
            I.Llama2.generate(ctx, s, w, 1, use_graph=use_graph)
            assert_close(s.read("logits"), m.forward(int(toks[pos]), pos), what=f"pos {pos}")
        for far in (host_end, 5000):  # position host_end is row host_end + 1: one past the bucket's rows
            s.reset(toks, p0 + n)
            ptr, _ = s.buffer("pos")
            jump = np.array([far], np.uint32)
            ctx._check(I.lib().ifr_upload(ctx.h, ptr, jump.ctypes.data, 4))
            I.Llama2.generate(ctx, s, w, 1, use_graph=use_graph)
            assert_close(s.read("logits"), m.forward(int(toks[far]), far), what=f"pos {far}")
    finally:
        s.close()
        w.close()
