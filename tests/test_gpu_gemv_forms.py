"""GPU check that every GEMV form the gemv_grp option selects gives the
default decode step's results bit for bit (same arithmetic, same reduction
orders): logits, tokens, KV-cache rows and the residual stream."""

import numpy as np
import pytest

from tests.test_gpu_model import run_steps

pytestmark = pytest.mark.gpu


def decode(ctx, cfg, w, prompt, n, mode="graph"):
    import inferi_amd as I

    s = I.Llama2State(ctx, cfg)
    try:
        logits, toks = run_steps(ctx, s, w, prompt, n, mode)
        kv = {}
        for layer in range(cfg.n_layers):
            for name in ("key_cache", "value_cache"):
                dt = np.uint16 if cfg.kv_dtype == I.F16 else np.float32
                kv[name, layer] = s.read(name, dt, layer).reshape(cfg.max_pos, cfg.kv_dim)[:n]
        x = s.read("x")
    finally:
        s.close()
    return np.array(logits), toks, kv, x


def assert_same(a, b, what):
    a, b = np.asarray(a), np.asarray(b)
    if not np.array_equal(a.view(np.uint8), b.view(np.uint8)):
        d = np.abs(a.astype(np.float64) - b.astype(np.float64))
        raise AssertionError(f"{what}: not bit-identical (max |diff| {d.max():.3e} at {np.unravel_index(d.argmax(), d.shape)})")


@pytest.mark.parametrize("grp", [0, 2, 4, 12, 16, 31, 33, 63, 64, 97, 128, 160, 225, 256, 481])
def test_gemv_forms_same_results(ctx, grp):
    """The looping body, the one-item forms of O, down, gate/up and the
    head, the head's 256-VGPR form, the four-row one-item forms of gate/up
    (bit 7) and of the plain and QKV GEMVs (bit 8), on the C4 shape."""
    import inferi_amd as I

    cfg = I.Llama2Config(n_layers=4, hidden=2048, ffn=5632, n_heads=32, n_kv_heads=4, vocab=32000, max_pos=32,
                         rope_theta=10000.0, rms_eps=1e-5, kv_dtype=I.F16)
    w = I.Llama2Weights.synthetic(ctx, cfg, seed=1000)
    try:
        prompt = [5, 31999, 7, 1234]
        ref = decode(ctx, cfg, w, prompt, 12)
        ctx.set_option("gemv_grp", grp)
        try:
            got = decode(ctx, cfg, w, prompt, 12)
        finally:
            ctx.set_option("gemv_grp", 225)
        assert_same(got[0], ref[0], "logits")
        assert np.array_equal(got[1], ref[1]), "tokens"
        for k in ref[2]:
            assert_same(got[2][k], ref[2][k], f"{k[0]} layer {k[1]}")
        assert_same(got[3], ref[3], "residual x")
    finally:
        w.close()


@pytest.mark.parametrize("dtype_name,rows,cols", [("Q4_K", 4096, 4096), ("Q4_K", 300, 1024), ("Q6_K", 512, 2048)])
def test_matmul_quant_four_row_form(ctx, dtype_name, rows, cols):
    """gemv_grp bit 8: ifr_matmul_quant_xq takes the four-rows-per-wave one-item
    kernel where the format has one, ifr_matmul_quant (which quantizes its
    input in the kernel) its usual one; both against the default form, bit
    for bit, and against the oracle's f64 GEMV at 1e-3."""
    import inferi_amd as I
    import oracle as O

    dtype = getattr(I, dtype_name)
    rng = np.random.default_rng(rows + cols)
    w = O.quantize(dtype, (rng.standard_normal(rows * cols) * 0.02).astype(np.float32))
    x = rng.standard_normal(cols).astype(np.float32)
    dw, dx, y, xq = ctx.upload(w), ctx.upload(x), ctx.alloc(rows * 4), ctx.alloc(ctx.activation_bytes(cols))
    try:
        ctx.quantize_activation(xq, dx, cols)
        e = O.gemv_quant(dtype, w, rows, cols, x)
        for call, arg in ((ctx.matmul_quant_assign, dx), (ctx.matmul_quant_xq, xq)):
            call(y, dw, dtype, rows, cols, arg)
            ref = y.download(np.float32, rows)
            y.upload(np.full(rows, np.nan, np.float32))
            ctx.set_option("gemv_grp", 225 | 256)
            try:
                call(y, dw, dtype, rows, cols, arg)
            finally:
                ctx.set_option("gemv_grp", 225)
            got = y.download(np.float32, rows)
            assert_same(got, ref, f"{dtype_name} {rows}x{cols}")
            assert np.all(np.abs(got - e) <= 1e-3 * np.maximum(np.abs(e), 1.0))
    finally:
        for b in (dw, dx, y, xq):
            b.free()


@pytest.mark.parametrize("gate,down,hidden,ffn", [
    ("Q8_0", "Q8_0", 1024, 544), ("Q8_0", "Q4_0", 1056, 544), ("Q4_0", "Q5_1", 896, 1056), ("Q4_1", "Q5_0", 32, 96),
    ("Q5_0", "F16", 64, 288), ("Q5_1", "F32", 1024, 32), ("F16", "Q8_0", 992, 320), ("F32", "Q4_1", 288, 1024),
    ("Q5_K", "Q6_K", 4096, 256), ("Q6_K", "Q5_K", 4096, 768), ("Q6_K", "Q8_K", 4352, 512), ("Q8_K", "Q4_K", 512, 1280),
    ("Q4_K", "Q6_K", 2048, 512)])
def test_ffn_f32_hidden_every_type(ctx, gate, down, hidden, ffn):
    """The gate/up form that leaves h in f32 with the down GEMV that quantizes
    it, for each type and for gate and down of different types, at one K step
    (32-element types up to 1024, K-quants up to 4096), just past it (the
    looping form) and with ragged FFN widths: the fused step's logits against
    the one-op-per-kernel step's on the same weights.  Both take x as 22-bit
    codes; they differ in the order of f32 sums only, 1e-5 of the largest
    logit (the bar is ten times that)."""
    import inferi_amd as I

    heads = next(h for h in range(1, 200) if hidden % (8 * h) == 0 and hidden // h <= 128)
    cfg = I.Llama2Config(n_layers=2, hidden=hidden, ffn=ffn, n_heads=heads, n_kv_heads=heads, vocab=256, max_pos=16,
                         rope_theta=10000.0, rms_eps=1e-5, kv_dtype=I.F32)
    mats = {"ffn_gate": getattr(I, gate), "ffn_up": getattr(I, gate), "ffn_down": getattr(I, down)}
    # the other matrices in a type that any width takes
    w = I.Llama2Weights.synthetic(ctx, cfg, seed=hidden + ffn, mat_dtype=I.Q8_0, head_dtype=I.Q8_0, embd_dtype=I.Q8_0,
                                  std=0.05, overrides=mats)
    logits = {}
    try:
        for fused in (True, False):
            s = I.Llama2State(ctx, cfg)
            s.reset([3, 250, 17, 99], 0)
            for _ in range(4):
                I.Llama2.launch(ctx, s, w, fused)
            logits[fused] = s.read("logits").astype(np.float64)
            s.close()
    finally:
        w.close()
    err = np.abs(logits[True] - logits[False]).max() / np.abs(logits[False]).max()
    assert err <= 1e-4, f"{err:.2e}"


@pytest.mark.parametrize("planted", [False, True])
def test_choosing_a_form_leaves_hip_errors_alone(planted):
    """Forms that a type does not have (the grouped and four-row ones but for
    Q4_K, the head's 256-VGPR one but for Q6_K) are not asked of the HIP
    runtime: neither an error of a failed look-up is left to the program's
    next HIP check, nor one taken away that the program itself left (a
    device that does not exist)."""
    import ctypes

    import inferi_amd as I

    ctx = I.LlmContext(0)  # its own: a context looks a kernel up once
    path = next(ln.split()[-1] for ln in open("/proc/self/maps") if "libamdhip64.so" in ln)
    hip = ctypes.CDLL(path)
    cfg = I.Llama2Config(n_layers=1, hidden=256, ffn=512, n_heads=4, n_kv_heads=2, vocab=64, max_pos=8,
                         rope_theta=10000.0, rms_eps=1e-5, kv_dtype=I.F16)
    w = I.Llama2Weights.synthetic(ctx, cfg, seed=1, mat_dtype=I.Q8_0, head_dtype=I.Q8_0, embd_dtype=I.Q8_0)
    s = I.Llama2State(ctx, cfg)
    x, xq, y = ctx.zeros(1024), ctx.alloc(ctx.activation_bytes(256)), ctx.alloc(4096)
    try:
        hip.hipGetLastError()
        if planted:
            assert hip.hipSetDevice(-1) != 0
        ctx.quantize_activation(xq, x, 256)  # what an ordinary call leaves of it
        before = hip.hipPeekAtLastError()
        for grp in (511, 225):
            ctx.set_option("gemv_grp", grp)
            s.reset([1, 2], 0)
            I.Llama2.launch(ctx, s, w)
            ctx.matmul_quant_xq(y, x, I.F32, 1, 256, xq)
            assert hip.hipPeekAtLastError() == before
    finally:
        hip.hipGetLastError()
        s.close()
        w.close()
        for b in (x, xq, y):
            b.free()
        ctx.close()
