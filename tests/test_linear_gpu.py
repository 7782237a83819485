"""GPU parity of the quantised linears (include/ktx_linear.h) against oracle/linear_ref.py, through the C ABI.

Tolerances (floating point path, fp32 accumulation in a different order than the un-vendored CUDA/Triton kernels):
  W4/BF16: |y - ref| <= 2^-7*|ref| + 2e-3*max|ref|  (one bf16 ulp of the output + accumulation-order noise);
           norm-wise relative error <= 1e-3 against exact (q-8)*s math in fp64.
  FP8    : same bound; activations that sit on an e4m3 rounding tie after x/s may quantise one step apart, which the
           norm-wise bound (2e-3) absorbs.
The quantiser is integer work: bit-exact against the reference's own quantize_weights (golden fixture)."""
import os

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from oracle.linear_ref import linear_bf16_ref, linear_fp8_ref, linear_w4_ref, quantize_weights_ref  # noqa: E402

GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "linear_w4_golden.npz")


def native():
    from ktransformers_amd import _native
    return _native


def close(y, ref, rel=1e-3):
    y, ref = y.float().cpu(), ref.float()
    tol = 2.0 ** -7 * ref.abs() + 2e-3 * ref.abs().max()
    bad = (y - ref).abs() > tol
    assert not bad.any(), f"{int(bad.sum())} elements out of tolerance, max diff {(y - ref).abs().max()}"
    assert (y - ref).norm() / ref.norm().clamp_min(1e-30) <= max(rel, 2.0 ** -8), float((y - ref).norm() / ref.norm())


@pytest.mark.parametrize("name", ["a", "b"])
@pytest.mark.parametrize("G", [32, 64, 128])
def test_w4_quantizer_bit_exact_vs_reference_golden(name, G):
    n = native()
    g = np.load(GOLD)
    w = torch.from_numpy(g[f"{name}_w"]).view(torch.bfloat16).cuda()
    N, K = w.shape
    h = n.LinearHandle(K, N, "W4", G, 16)
    h.load_bf16(w)
    q, s = h.debug_get_w4()
    assert np.array_equal(s, g[f"{name}_s{G}"])
    live = np.repeat(g[f"{name}_s{G}"] != 0, G, axis=0)
    assert np.array_equal(q[live], g[f"{name}_q{G}"][live])


SHAPES = [(256, 64), (2048, 576), (2048, 3072), (1536, 200), (7168, 1536), (384, 48)]


# every shape at the group size the models use (64); the other group sizes on two shapes
W4_CASES = [(K, N, T, G) for G in (64, 128, 32) for T in (1, 2, 3, 4, 7, 16, 33, 130) for (K, N) in SHAPES
            if G == 64 or (K, N) in ((256, 64), (2048, 576))]


@pytest.mark.parametrize("K,N,T,G", W4_CASES)
def test_w4_forward(K, N, T, G):
    n = native()
    torch.manual_seed(K + N + T)
    w = (torch.randn(N, K) / 10).to(torch.bfloat16)
    x = (torch.randn(T, K) / 10).to(torch.bfloat16)
    bias = (torch.randn(N) / 10).to(torch.bfloat16) if (T % 2 == 0) else None
    q, s = quantize_weights_ref(w.T.contiguous(), G)
    h = n.LinearHandle(K, N, "W4", G, 256)
    h.load_bf16(w.cuda(), bias.cuda() if bias is not None else None)
    y = h.forward(x.cuda())
    close(y, linear_w4_ref(x, q, s, G, bias))
    if T <= 4:   # the same rows through the general kernel
        n.linear_force_gemm(True)
        try:
            y2 = h.forward(x.cuda())
        finally:
            n.linear_force_gemm(False)
        close(y2, linear_w4_ref(x, q, s, G, bias))
    # pre-quantised upload gives the same tiles
    h2 = n.LinearHandle(K, N, "W4", G, 256)
    h2.load_w4(q.to(torch.uint8).cuda(), s.cuda(), bias.cuda() if bias is not None else None)
    assert torch.equal(h2.forward(x.cuda()), y)


@pytest.mark.parametrize("K,N", SHAPES)
@pytest.mark.parametrize("T", [1, 4, 5, 40])
def test_bf16_forward(K, N, T):
    n = native()
    torch.manual_seed(K + N + T)
    w = (torch.randn(N, K) / 10).to(torch.bfloat16)
    x = (torch.randn(T, K) / 10).to(torch.bfloat16)
    h = n.LinearHandle(K, N, "BF16", 0, 64)
    h.load_bf16(w.cuda())
    close(h.forward(x.cuda()), linear_bf16_ref(x, w), rel=1e-3)


@pytest.mark.parametrize("K,N", [(256, 64), (2048, 576), (7168, 1536), (1536, 200), (384, 48)])
@pytest.mark.parametrize("T", [1, 3, 4, 9, 40])
def test_fp8_forward(K, N, T):
    n = native()
    torch.manual_seed(K + N + T)
    w = (torch.randn(N, K) / 4).to(torch.float8_e4m3fn)
    sc = (torch.rand((N + 127) // 128, K // 128) + 0.5) / 32
    x = (torch.randn(T, K) / 10).to(torch.bfloat16)
    bias = (torch.randn(N) / 10).to(torch.bfloat16) if T == 4 else None
    h = n.LinearHandle(K, N, "FP8", 128, 64)
    h.load_fp8(w.cuda(), sc.cuda(), bias.cuda() if bias is not None else None)
    y = h.forward(x.cuda())
    close(y, linear_fp8_ref(x, w, sc, bias), rel=2e-3)


@pytest.mark.parametrize("K,N,T", [(256, 64, 128), (1536, 200, 300), (2048, 576, 513), (7168, 2112, 2048), (512, 4096, 1000)])
def test_fp8_prompt_gemm_against_the_strip_kernel(K, N, T, monkeypatch):
    """Prompt-sized FP8 calls (T >= 128) run act_quant once + lin_fp8_gemm_kernel (csrc/ktx_linear_fp8gemm.inc): the same four MFMAs
    per 128-block in the same order, the same (dot * a_s) * b_s accumulation and the same output rounding as the strip kernel every
    other test of this file pins to the reference (lin_gemm_kernel<FP8>) — so the two paths must agree bit for bit: ragged T and N
    (partial 128-tiles), bias, the GLU epilogue, the decoder layer's adds, a fused input norm, strided rows; and against
    oracle/linear_ref.py at the file's FP8 bound."""
    n = native()
    torch.manual_seed(K + N + T)
    w = (torch.randn(N, K) / 4).to(torch.float8_e4m3fn)
    sc = (torch.rand((N + 127) // 128, K // 128) + 0.5) / 32
    x = (torch.randn(T, K) / 10).to(torch.bfloat16).cuda()
    bias = (torch.randn(N) / 10).to(torch.bfloat16) if N % 3 == 0 else None
    h = n.LinearHandle(K, N, "FP8", 128, T)
    h.load_fp8(w.cuda(), sc.cuda(), bias.cuda() if bias is not None else None)
    add1 = (torch.randn(T, N) / 10).to(torch.bfloat16).cuda()
    nw = (1 + torch.randn(K) / 10).to(torch.bfloat16).cuda()
    xs = torch.zeros(T, K + 64, dtype=torch.bfloat16, device="cuda")[:, :K]
    xs.copy_(x)
    calls = [dict(), dict(add1=add1), dict(norm=(nw, 1e-6)), dict(add1=add1, add2=add1)]
    if N % 16 == 0 and bias is None:
        calls.append(dict(glu=True))
    # the GEMM at every size (ktx_linear_forward_ws would take most of these), and the strip kernel itself to compare with (dev knob 12 keeps it)
    monkeypatch.setattr(n.LinearHandle, "FP8_GEMM_OUT", (0, 0))
    n.timing_enable(2)
    try:
        h.forward(x)
        labels = [t[0] for t in n.timing_collect()]
    finally:
        n.timing_enable(0)
    assert any("lin_fp8_gemm_kernel" in t for t in labels), labels
    # the default GEMM sums a 128-block in ONE K = 128 MFMA (twice the rate; the hardware's own order inside the block) —
    # within one bf16 ulp of the strip kernel; dev knob 27 = 1 keeps the four K = 32 MFMAs, which ARE the strip kernel's bits
    fast = [h.forward(x, **kw) for kw in calls] + [h.forward(xs)]
    n.check(n.lib.ktx_debug_set(27, 1))
    try:
        got = [h.forward(x, **kw) for kw in calls] + [h.forward(xs)]
    finally:
        n.check(n.lib.ktx_debug_set(27, 0))
    monkeypatch.setenv("KTX_FP8_PROMPT_KERNEL", "1")
    n.check(n.lib.ktx_debug_set(12, 1))
    try:
        want = [h.forward(x, **kw) for kw in calls] + [h.forward(xs)]
    finally:
        n.check(n.lib.ktx_debug_set(12, 0))
    for a, b, f, kw in zip(got, want, fast, calls + [dict(strided=True)]):
        assert a.shape == b.shape and torch.equal(a, b), f"{kw.keys()}: {(a != b).sum().item()} of {a.numel()} outputs differ"
        d = (f.float() - b.float()).abs()
        bound = 2.0 ** -7 * b.float().abs() + 2.0 ** -10 * float(b.float().abs().max())
        assert f.shape == b.shape and bool((d <= bound).all()), f"{kw.keys()}: K = 128 MFMA path beyond one bf16 ulp of the strip kernel"
        assert float((f != b).float().mean()) < 0.02, f"{kw.keys()}: {float((f != b).float().mean()):.4f} of the outputs differ"
    close(got[0], linear_fp8_ref(x.cpu(), w, sc, bias), rel=2e-3)
    close(fast[0], linear_fp8_ref(x.cpu(), w, sc, bias), rel=2e-3)


@pytest.mark.parametrize("K,N,T", [(1024, 64, 128), (2048, 577, 300), (7168, 2112, 300), (7168, 2112, 1000), (16384, 7168, 130)])
def test_fp8_tiles_of_prompts_in_one_mfma_a_block(K, N, T, monkeypatch):
    """The tiles of ktx_linear_forward_ws take a 128-block of an FP8 prompt in one MFMA of K = 128, with KTX_FP8_PROMPT_KERNEL=1 in four of K = 32:
    within one bf16 ulp of each other, few outputs different, and of the oracle at the bound of this file; with a row count the eager bits."""
    n = native()
    torch.manual_seed(K + N + T)
    w = (torch.randn(N, K) / 4).to(torch.float8_e4m3fn)
    sc = (torch.rand((N + 127) // 128, K // 128) + 0.5) / 32
    x = (torch.randn(T, K) / 10).to(torch.bfloat16).cuda()
    h = n.LinearHandle(K, N, "FP8", 128, T)
    h.load_fp8(w.cuda(), sc.cuda())
    n.timing_enable(2)
    try:
        one = h.forward(x)
        labels = [t[0] for t in n.timing_collect()]
    finally:
        n.timing_enable(0)
    assert any("lin_tile_kernel" in t for t in labels), labels
    rows = h.forward(x, bsz_tensor=torch.tensor([T], dtype=torch.int32, device="cuda"))
    assert torch.equal(one, rows)
    monkeypatch.setenv("KTX_FP8_PROMPT_KERNEL", "1")
    four = h.forward(x)
    close(one, linear_fp8_ref(x.cpu(), w, sc, None), rel=2e-3)
    d = (one.float() - four.float()).abs()
    assert bool((d <= 2.0 ** -7 * four.float().abs() + 2.0 ** -10 * float(four.float().abs().max())).all())
    assert float((one != four).float().mean()) < 0.02


@pytest.mark.parametrize("T", [1, 127, 128, 130])
def test_fp8_act_quant_writes_its_rows_only(T):
    """ktx_fp8_act_quant leaves the scales behind its T rows as they are (they may be another call's); the padded form zeroes them up to whole tiles."""
    n = native()
    K, ld = 384, 512
    x = torch.randn(T, K, device="cuda").to(torch.bfloat16)
    q = torch.empty(T, K, dtype=torch.uint8, device="cuda")
    want = (x.float().view(T, K // 128, 128).abs().amax(-1) / 448.0).T
    for fn, zeros in ((n.lib.ktx_fp8_act_quant, T), (n.lib.ktx_fp8_act_quant_padded, (T + 127) // 128 * 128)):
        sT = torch.full((K // 128, ld), 7.0, device="cuda")
        n.check(fn(x.data_ptr(), K, T, K, q.data_ptr(), sT.data_ptr(), ld, torch.cuda.current_stream().cuda_stream))
        torch.testing.assert_close(sT[:, :T], want, rtol=2.0 ** -22, atol=0.0)      # (an ulp: torch may multiply by the reciprocal)
        assert not bool(sT[:, T:zeros].any()) and bool((sT[:, zeros:] == 7.0).all())


@pytest.mark.parametrize("exponent", [-133, -126, -90, -82, -81, 0, 9, 98, 99, 100, 126])   # of a block's largest: subnormal scales, both ends of the reciprocal's range, large ones
def test_fp8_act_quant_rounds_as_a_division(exponent):
    """quant8_fp8 multiplies by the scale's reciprocal and corrects the product once: the bytes of x / s in e4m3, zeros' signs included, for every pair of bf16
    mantissas of an element and of its block's largest magnitude."""
    n = native()
    top = torch.ldexp(torch.arange(128, 256, dtype=torch.float64) / 128, torch.tensor(exponent)).to(torch.bfloat16)   # one block a row
    x = torch.ldexp(torch.arange(128, 256, dtype=torch.float64) / 128, torch.tensor(exponent)).expand(128, 128)
    g = torch.Generator().manual_seed(exponent + 200)
    x = torch.ldexp(x, -torch.randint(1, 12, (8, 128, 128), generator=g)) * (1 - 2 * torch.randint(0, 2, (8, 128, 128), generator=g))   # eight sets of exponents and signs
    x[:, :, 5], x[:, :, 6] = 0.0, -0.0
    x = x.to(torch.bfloat16)
    x[..., 0] = top
    x = x.view(1024, 128)
    amax = x.float().abs().amax(1, keepdim=True)
    s = amax / 448.0
    want = torch.where(s > 0, x.float() / s, torch.zeros(())).to(torch.float8_e4m3fn)
    q, sT = torch.empty((1024, 128), dtype=torch.uint8, device="cuda"), torch.empty((1, 1024), device="cuda")
    xc = x.cuda()
    n.check(n.lib.ktx_fp8_act_quant(xc.data_ptr(), 128, 1024, 128, q.data_ptr(), sT.data_ptr(), 1024, torch.cuda.current_stream().cuda_stream))
    assert torch.equal(sT.cpu().view(-1), s.view(-1))
    assert torch.equal(q.cpu(), want.view(torch.uint8))


@pytest.mark.parametrize("K,N,G", [(2048, 576, 64), (1536, 200, 32), (7168, 2112, 128), (1024, 64, -1), (384, 48, 128)])
def test_w8_format_is_the_bf16_kernel_on_marlins_multiplicand_bit_for_bit(K, N, G):
    """The W8 format (include/ktx_linear.h: KTX_LIN_W8, round 4): one byte per weight in HBM, bf16((q - 128) * s) formed in registers
    in front of the BF16 format's MFMAs — so a W8 handle and a BF16 handle loaded with that very matrix must agree bit for bit, for
    decode rows, small and prompt-sized batches, with bias, fused norm, adds and the GLU epilogue; per-channel scales (G = -1) ride
    as groups of 128.  (The multiplicand itself is pinned to the reference's quantize_weights in tests/test_linear_cpu.py.)"""
    n = native()
    from ktransformers_amd.operators.linear import marlin_multiplicand, marlin_quantize
    torch.manual_seed(K + N + G)
    w = (torch.randn(N, K) / 10).to(torch.bfloat16).cuda()
    g = K if G == -1 else G
    hg = min(g, 128)
    bias = (torch.randn(N) / 10).to(torch.bfloat16).cuda() if N % 3 == 0 else None
    q, sc = marlin_quantize(w, 8, g)
    h8 = n.LinearHandle(K, N, "W8", hg, 512)
    h8.load_w8((q + 128).to(torch.uint8).view(N, K).T.contiguous(), sc.view(N, -1).repeat_interleave(g // hg, dim=1).T.contiguous(), bias)
    hb = n.LinearHandle(K, N, "BF16", 0, 512)
    hb.load_bf16(marlin_multiplicand(w, 8, g).contiguous(), bias)
    assert h8.weight_bytes() < 0.6 * hb.weight_bytes()
    nw = (1 + torch.randn(K) / 10).to(torch.bfloat16).cuda()
    for T in (1, 2, 4, 5, 33, 300):
        x = (torch.randn(T, K) / 10).to(torch.bfloat16).cuda()
        add1 = (torch.randn(T, N) / 10).to(torch.bfloat16).cuda()
        calls = [dict(), dict(norm=(nw, 1e-6)), dict(add1=add1)]
        if N % 16 == 0 and bias is None:
            calls.append(dict(glu=True))
        for kw in calls:
            a, b = h8.forward(x, **kw), hb.forward(x, **kw)
            assert torch.equal(a, b), f"T={T} {list(kw)}: {(a != b).sum().item()} of {a.numel()} outputs differ"


def test_fp8_linears_merge_on_block_boundaries():
    """build_merged_linear for block-fp8 checkpoints (round 4): q_a_proj (1536 rows = 12 whole 128-row scale blocks) | kv_a_proj_with_mqa
    (576 rows: the last block is partial) as ONE operator gives exactly the rows the two operators give, decode and prompt sized; a first
    matrix that does not end on a block boundary is refused (None: the separate operators stay)."""
    from types import SimpleNamespace
    from ktransformers_amd.operators.linear import KLinearFP8, build_merged_linear
    from ktransformers_amd.util.loader import DictLoader
    torch.manual_seed(3)
    K = 1024
    def mk(N):
        return (torch.randn(N, K) / 4).to(torch.float8_e4m3fn), (torch.rand((N + 127) // 128, K // 128) + 0.5) / 32
    (wa, sa), (wb, sb), (wc, sc) = mk(1536), mk(576), mk(200)
    ld = DictLoader({"a.weight": wa, "a.weight_scale_inv": sa, "b.weight": wb, "b.weight_scale_inv": sb, "c.weight": wc, "c.weight_scale_inv": sc})
    ops = {}
    for key, N in (("a", 1536), ("b", 576), ("c", 200)):
        ops[key] = KLinearFP8(key, ld, SimpleNamespace(), torch.nn.Linear(K, N, bias=False, device="meta"), device="cuda")
        ops[key].load()
    merged = build_merged_linear(ops["a"], ["a", "b"], ld, "cuda")
    assert merged is not None and merged[1] == [1536, 576]
    assert build_merged_linear(ops["c"], ["c", "b"], ld, "cuda") is None          # 200 rows: not a block boundary
    for T in (1, 3, 200):
        x = (torch.randn(T, K) / 10).to(torch.bfloat16).cuda()
        y = merged[0].forward(x)
        assert torch.equal(y[:, :1536], ops["a"].forward(x)) and torch.equal(y[:, 1536:], ops["b"].forward(x))


def test_fp8_mlp_runs_gate_and_up_as_one_operator():
    """KDeepseekV3MLP on a block-fp8 checkpoint (round 4): gate_proj and up_proj are loaded as ONE operator over the concatenation
    [gate ; up] (whole 128-row scale blocks; the W4 GLU interleave would split blocks) — the SiLU * up input, and so the block's
    output, must be bit for bit what the separate operators give, with and without the fused input norm, decode and prompt sized."""
    from types import SimpleNamespace
    from ktransformers_amd._native import rmsnorm, silu_mul
    from ktransformers_amd.operators.linear import KLinearFP8, KTransformersLinear
    from ktransformers_amd.operators.mlp import KDeepseekV3MLP
    from ktransformers_amd.util.loader import DictLoader
    torch.manual_seed(5)
    H, I = 1024, 512
    def mk(N, K):
        return (torch.randn(N, K) / 4).to(torch.float8_e4m3fn), (torch.rand((N + 127) // 128, K // 128) + 0.5) / 32
    st = {}
    for nm, (N, K) in (("gate_proj", (I, H)), ("up_proj", (I, H)), ("down_proj", (H, I))):
        w, sc = mk(N, K)
        st[f"mlp.{nm}.weight"], st[f"mlp.{nm}.weight_scale_inv"] = w, sc
    ld, cfg = DictLoader(st), SimpleNamespace()
    class Orig(torch.nn.Module):
        def __init__(self):
            super().__init__()
            for nm, (N, K) in (("gate_proj", (I, H)), ("up_proj", (I, H)), ("down_proj", (H, I))):
                setattr(self, nm, KTransformersLinear(f"mlp.{nm}", ld, cfg, torch.nn.Linear(K, N, bias=False, device="meta"), "cuda",
                                                      "KLinearFP8", "cuda", "KLinearFP8"))
    mlp = KDeepseekV3MLP("mlp", ld, cfg, Orig(), "cuda", "cuda")
    mlp.load()
    assert mlp._gate_up is None and mlp._gate_up_cat is not None and mlp._gate_up_cat._h.N == 2 * I
    ops = {nm: KLinearFP8(f"mlp.{nm}", ld, cfg, torch.nn.Linear(H, I, bias=False, device="meta"), device="cuda") for nm in ("gate_proj", "up_proj")}
    for op in ops.values():
        op.load()
    nw = (1 + torch.randn(H) / 10).to(torch.bfloat16).cuda()
    for T in (1, 3, 130):
        x = (torch.randn(T, H) / 10).to(torch.bfloat16).cuda()
        for norm in (None, (nw, 1e-6)):
            xn = x if norm is None else rmsnorm(x, norm[0], norm[1], native_rounding=True)
            want = silu_mul(torch.cat([ops["gate_proj"].forward(xn), ops["up_proj"].forward(xn)], dim=-1))
            assert torch.equal(mlp.gate_up(x, norm), want), f"T={T} norm={norm is not None}"
            # the whole block: SiLU * up rides in down_proj's prologue on decode-sized calls (glu_in) — same bits as the three launches
            res = (torch.randn(T, H) / 10).to(torch.bfloat16).cuda()
            assert torch.equal(mlp.forward(x, add1=res, norm=norm), mlp.down(want, x.shape, add1=res)), f"T={T} block"


@pytest.mark.parametrize("fmt,K,N", [("FP8", 2048, 7168), ("FP8", 1536, 576), ("W4", 2048, 7168), ("W4", 1408, 2048), ("BF16", 512, 200)])
def test_silu_mul_in_the_prologue_of_a_decode_linear(fmt, K, N):
    """ktx_linear_fusion.glu_in (round 5): x rows are [gate | up] and the block-fp8 decode kernel stages silu(gate) * up itself — the
    same roundings as ktx_silu_mul, so bit for bit the two-launch result, with the epilogue adds, the bsz tensor and for every decode
    row count; a prompt-sized call, and the other formats (their MLPs have the GLU epilogue instead), take the separate launch inside
    LinearHandle.forward — same call, same bits."""
    n = native()
    torch.manual_seed(K + N)
    h = n.LinearHandle(K, N, fmt, 128 if fmt == "FP8" else 64, 64)
    if fmt == "FP8":
        h.load_fp8((torch.randn(N, K) / 4).to(torch.float8_e4m3fn).cuda(), ((torch.rand((N + 127) // 128, K // 128) + 0.5) / 32).cuda())
    else:
        h.load_bf16((torch.randn(N, K) / 10).to(torch.bfloat16).cuda())
    for T in (1, 2, 3, 4, 9):
        gu = (torch.randn(T, 2 * K) * 2).to(torch.bfloat16).cuda()
        a1 = torch.randn(T, N).to(torch.bfloat16).cuda()
        a2 = torch.randn(T, N).to(torch.bfloat16).cuda()
        act = n.silu_mul(gu)
        n.timing_collect()
        n.timing_enable(2)
        try:
            got = h.forward(gu, glu_in=True)
            torch.cuda.synchronize()
            labels = [lab for lab, _, _ in n.timing_collect()]
        finally:
            n.timing_enable(0)
        assert torch.equal(got, h.forward(act)), (fmt, T)
        if fmt == "FP8" and T <= 4:       # one launch, and it is the decode kernel with the prologue
            assert len(labels) == 1 and "silu*up in" in labels[0], labels
        assert torch.equal(h.forward(gu, add1=a1, add2=a2, glu_in=True), h.forward(act, add1=a1, add2=a2)), (fmt, T, "adds")
        if T == 3:
            bsz = torch.tensor([2], dtype=torch.int32, device="cuda")
            got, want = h.forward(gu, bsz, glu_in=True), h.forward(n.silu_mul(gu, bsz)[:T], bsz)
            assert torch.equal(got[:2], want[:2]) and bool((got[2:] == 0).all())
    with pytest.raises(n.KtxError):
        h.forward(torch.zeros(1, 2 * K, dtype=torch.bfloat16, device="cuda"), norm=(torch.ones(K, dtype=torch.bfloat16, device="cuda"), 1e-6), glu_in=True)


def test_bsz_tensor_and_graph_capture():
    n = native()
    torch.manual_seed(0)
    K, N = 2048, 576
    w = (torch.randn(N, K) / 10).to(torch.bfloat16)
    x = (torch.randn(4, K) / 10).to(torch.bfloat16).cuda()
    q, s = quantize_weights_ref(w.T.contiguous(), 64)
    h = n.LinearHandle(K, N, "W4", 64, 16)
    h.load_bf16(w.cuda())
    bsz = torch.tensor([2], dtype=torch.int32, device="cuda")
    out = torch.full((4, N), 7.0, dtype=torch.bfloat16, device="cuda")
    h.forward(x, bsz, out)
    close(out[:2], linear_w4_ref(x[:2].cpu(), q, s, 64))
    assert torch.all(out[2:] == 7.0)
    g = torch.cuda.CUDAGraph()
    y = torch.empty((4, N), dtype=torch.bfloat16, device="cuda")
    s0 = torch.cuda.Stream()
    with torch.cuda.stream(s0):
        h.forward(x, None, y)
        torch.cuda.synchronize()
        with torch.cuda.graph(g, stream=s0):
            h.forward(x, None, y)
    y.zero_()
    g.replay()
    torch.cuda.synchronize()
    close(y, linear_w4_ref(x.cpu(), q, s, 64))


def test_errors_are_loud():
    n = native()
    with pytest.raises(n.KtxError):
        n.LinearHandle(100, 64, "W4", 64, 16)          # in_features % 8
    with pytest.raises(n.KtxError):
        n.LinearHandle(256, 64, "W4", 48, 16)          # group size
    h = n.LinearHandle(256, 64, "W4", 64, 4)
    x = torch.zeros(2, 256, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(n.KtxError):
        h.forward(x)                                    # not loaded
    h.load_bf16(torch.zeros(64, 256, dtype=torch.bfloat16, device="cuda"))
    with pytest.raises(n.KtxError):
        h.forward(torch.zeros(8, 256, dtype=torch.bfloat16, device="cuda"))   # T > max_len
    assert torch.all(h.forward(x) == 0)


@pytest.mark.parametrize("T", [1, 3, 4, 9, 40])
@pytest.mark.parametrize("fmt", ["W4", "BF16"])
def test_fused_norm_glu_and_addends(T, fmt):
    """ktx_linear_forward_fused: RMSNorm prologue, [gate|up] GLU epilogue and two addends equal the unfused sequence
    (same kernels, same roundings) bit for bit."""
    n = native()
    torch.manual_seed(T)
    K, I, N = 512, 256, 384
    x = (torch.randn(T, K)).to(torch.bfloat16).cuda()
    nw = (1 + 0.1 * torch.randn(K)).to(torch.bfloat16).cuda()
    g = (torch.randn(I, K) / 10).to(torch.bfloat16).cuda()
    u = (torch.randn(I, K) / 10).to(torch.bfloat16).cuda()
    hg, hu = n.LinearHandle(K, I, fmt, 64, 64), n.LinearHandle(K, I, fmt, 64, 64)
    hg.load_bf16(g); hu.load_bf16(u)
    inter = torch.stack([g.view(-1, 8, K), u.view(-1, 8, K)], dim=1).reshape(-1, K).contiguous()
    hm = n.LinearHandle(K, 2 * I, fmt, 64, 64)
    hm.load_bf16(inter)
    xn = n.rmsnorm(x, nw, 1e-6, native_rounding=True)
    ref = n.silu_mul(torch.cat([hg.forward(xn), hu.forward(xn)], dim=-1))
    got = hm.forward(x, norm=(nw, 1e-6), glu=True)
    assert got.shape == (T, I)
    # the fused prologue sums the squares in a different order: allow the rare 1-ulp flip of a normalised activation
    assert (got != ref).float().mean() < 0.02 and torch.allclose(got.float(), ref.float(), rtol=2 ** -6, atol=1e-3)
    assert torch.equal(hm.forward(xn, glu=True), ref)
    # addends
    w = (torch.randn(N, I) / 10).to(torch.bfloat16).cuda()
    hd = n.LinearHandle(I, N, fmt, 64, 64)
    hd.load_bf16(w)
    a1 = torch.randn(T, N).to(torch.bfloat16).cuda()
    a2 = torch.randn(T, N).to(torch.bfloat16).cuda()
    y = hd.forward(ref)
    want = a2 + (a1 + y)
    assert torch.equal(hd.forward(ref, add1=a1, add2=a2), want)
    # strided input rows (a slice of a wider buffer)
    wide = torch.zeros(T, I + 64, dtype=torch.bfloat16, device="cuda")
    wide[:, :I] = ref
    assert torch.equal(hd.forward(wide[:, :I]), y)


@pytest.mark.parametrize("K,N,G", [(2048, 576, 64), (7168, 1536, 64), (1536, 200, 64), (2048, 576, 128), (2048, 576, 32)])
@pytest.mark.parametrize("T", [33, 130, 257])
def test_w4_prompt_kernel_with_several_strips_per_wavefront(K, N, G, T):
    """lin_gemm_w4n_kernel (prompt-sized W4, 2 / 4 strips per wavefront, packed-fp32 dequantisation epilogue) performs the
    one-strip kernel's operations element for element: bit-identical outputs, with bias, addends and the GLU epilogue,
    ragged feature counts (N % 64 != 0) and ragged token tiles."""
    n = native()
    torch.manual_seed(K + N + T + G)
    w = (torch.randn(N, K) / 10).to(torch.bfloat16).cuda()
    x = (torch.randn(T, K) / 10).to(torch.bfloat16).cuda()
    bias = (torch.randn(N) / 10).to(torch.bfloat16).cuda()
    a1 = torch.randn(T, N).to(torch.bfloat16).cuda()
    h = n.LinearHandle(K, N, "W4", G, 512)
    h.load_bf16(w, bias)
    hg = None
    if N % 16 == 0:
        hg = n.LinearHandle(K, N, "W4", G, 512)
        hg.load_bf16(w)
    outs = {}
    try:
        for knob in (1, 2, 4):
            n.lib.ktx_debug_set(12, knob)
            outs[knob] = (h.forward(x), h.forward(x, add1=a1), hg.forward(x, glu=True) if hg is not None else None)
    finally:
        n.lib.ktx_debug_set(12, 0)
    q, s = quantize_weights_ref(w.cpu().T.contiguous(), G)
    close(outs[1][0], linear_w4_ref(x.cpu(), q, s, G, bias.cpu()))
    for knob in (2, 4):
        for a, b in zip(outs[1], outs[knob]):
            if a is not None:
                assert torch.equal(a, b), f"strips/wavefront = {knob}: {int((a != b).sum())} of {a.numel()} outputs differ"


@pytest.mark.parametrize("H,T", [(128, 1), (64, 3), (16, 4)])
def test_qb_absorb_and_prep_in_one_launch(H, T):
    """ktx_linear_forward_qb_absorb (q_b_proj with q_a_layernorm, the per-head q-absorb products, RoPE of q_pe and the kv half of
    mla_prep, one launch) against the separate calls it replaces: q_b (fused norm) -> absorb_and_prep.  RoPE, the latent norm and
    the absorb products run the same arithmetic on the same q values; q_b's 12 k-steps are summed as two halves instead of one
    run, so q agrees within fp32 re-association (a bf16 ulp here and there), which the comparison allows for."""
    n = native()
    nope, rope, lora, qlora = 128, 64, 512, 1536
    dev = torch.device("cuda", 0)
    g = torch.Generator().manual_seed(H * 10 + T)
    wqb = (torch.randn((H * (nope + rope), qlora), generator=g) / 20).to(torch.bfloat16).to(dev)
    wuk = (torch.randn((H, lora, nope), generator=g) / 10).to(torch.bfloat16).to(dev)
    qa_full = torch.randn((T, qlora + lora + rope), generator=g).to(torch.bfloat16).to(dev)      # the merged q_a | kv_a GEMV output
    q_a, kv = qa_full[:, :qlora], qa_full[:, qlora:]
    nw = (1 + 0.1 * torch.randn((qlora,), generator=g)).to(torch.bfloat16).to(dev)
    knw = (1 + 0.1 * torch.randn((lora,), generator=g)).to(torch.bfloat16).to(dev)
    pos = torch.tensor([5, 77, 4000, 123456][:T], dtype=torch.int64, device=dev)
    inv_freq = (1.0 / (10000 ** (torch.arange(0, rope, 2).float() / rope))).to(dev)
    qb = n.LinearHandle(qlora, H * (nope + rope), "W4", 64, 8, dev)
    qb.load_bf16(wqb)
    qabs = n.LinearHandle(nope, lora, "BF16", 0, 8, dev, batch=H)
    qabs.load_bf16(wuk)
    assert n.qb_absorb_eligible(qb, qabs, T, H, nope, rope, lora)
    q = qb.forward(q_a, norm=(nw, 1e-6)).reshape(T, H * (nope + rope))
    ref = n.absorb_and_prep(qabs, q, kv, knw, 1e-6, pos, inv_freq, 1.3, H, nope, rope, lora)
    for rep in range(2):
        got = n.qb_absorb_and_prep(qb, qabs, q_a, (nw, 1e-6), kv, knw, 1e-6, pos, inv_freq, 1.3, H, nope, rope, lora)
        torch.cuda.synchronize()
        assert torch.equal(got[2], ref[2]) and torch.equal(got[3], ref[3]), "kv half of mla_prep: same code, same bits"
        for a, b, what in ((got[0], ref[0], "q_nope (absorbed)"), (got[1], ref[1], "q_pe")):
            a, b = a.float(), b.float()
            assert torch.isfinite(a).all()
            rel = float((a - b).norm() / b.norm())
            assert rel < 2e-3, (what, rel)
            assert float((a - b).abs().max()) <= 2e-2 * float(b.abs().max()), what


@pytest.mark.parametrize("K,N,G", [(2048, 576, 64), (7168, 1536, 64), (1536, 208, 128)])
def test_prompt_sized_w4_dequantises_once_and_runs_a_library_gemm(K, N, G, monkeypatch):
    """T >= LinearHandle.PROMPT_MIN_T, where the tiles don't take the call (held off here): the W4 weights are expanded once with Marlin's in-register rounding
    bf16((q - 8) * s) (ktx_linear_dequant_bf16: bit-identical to the torch expression on the reference quantiser's q and s) and a plain library
    GEMM runs on them — against fp64 math on the same rounded weights, against the hand-written W4 GEMM, and with the GLU /
    addend epilogues of the decoder layer."""
    import os
    n = native()
    monkeypatch.setattr(n.LinearHandle, "_w4_prompt_on_tiles", lambda self, T: False)
    torch.manual_seed(K + N)
    T = n.LinearHandle.PROMPT_MIN_T + 40
    w = (torch.randn(N, K) / 10).to(torch.bfloat16).cuda()
    x = (torch.randn(T, K) / 10).to(torch.bfloat16).cuda()
    a1 = torch.randn(T, N).to(torch.bfloat16).cuda()
    a2 = torch.randn(T, N).to(torch.bfloat16).cuda()
    h = n.LinearHandle(K, N, "W4", G, 1024)
    h.load_bf16(w)
    q, s = quantize_weights_ref(w.cpu().T.contiguous(), G)
    wdq = ((q.float() - 8.0) * s.float().repeat_interleave(G, dim=0)).T.contiguous().to(torch.bfloat16)      # [N, K]
    assert torch.equal(h.dequant_bf16().cpu(), wdq)
    y = h.forward(x)
    close(y, linear_w4_ref(x.cpu(), q, s, G, None, round_weights=True), rel=2e-3 ** 1)
    os.environ["KTX_W4_PROMPT_KERNEL"] = "1"
    try:
        y_k = h.forward(x)
        y_k_add = h.forward(x, add1=a1, add2=a2)
    finally:
        os.environ.pop("KTX_W4_PROMPT_KERNEL")
    assert float((y.float() - y_k.float()).norm() / y_k.float().norm()) < 3e-3      # exact-integer weights vs bf16-rounded ones
    y_add = h.forward(x, add1=a1, add2=a2)
    assert float((y_add.float() - y_k_add.float()).norm() / y_k_add.float().norm()) < 3e-3
    assert torch.equal(y_add, a2 + (a1 + y))
    if N % 16 == 0:
        hg = n.LinearHandle(K, N, "W4", G, 1024)
        hg.load_bf16(w)
        got = hg.forward(x, glu=True)
        os.environ["KTX_W4_PROMPT_KERNEL"] = "1"
        try:
            ref = hg.forward(x, glu=True)
        finally:
            os.environ.pop("KTX_W4_PROMPT_KERNEL")
        assert got.shape == ref.shape == (T, N // 2)
        assert float((got.float() - ref.float()).norm() / ref.float().norm()) < 5e-3


@pytest.mark.parametrize("K,N,T,G", [(2048, 576, 1500, 64), (128, 264, 513, 128), (1536, 24, 600, 32), (7168, 264, 520, 64), (7168, 2112, 777, 128), (4096, 1000, 1030, 32)])
def test_w4_prompts_on_tiles_multiply_the_rounded_weights(K, N, T, G, monkeypatch):
    """The tiles with bf16((q - 8) s) formed in registers against the expansion and the GEMM: the same products, so the same bits where K is one chunk (to 16 k-steps, and
    past 1024 rows); with K cut the fp32 sums are added in another order, which moves a result by a bf16 step now and then (fewer than 1 in 100 here: a rounding error of about
    2^-22 of the sums against steps of 2^-8)."""
    n = native()
    torch.manual_seed(K + N + T)
    h = n.LinearHandle(K, N, "W4", G, 2048)
    h.load_bf16((torch.randn(N, K) / 10).to(torch.bfloat16).cuda())
    x = (torch.randn(T, K) / 10).to(torch.bfloat16).cuda()
    a1 = torch.randn(T, N).to(torch.bfloat16).cuda()
    hb = n.LinearHandle(K, N, "W4", G, 2048)
    hb.load_bf16((torch.randn(N, K) / 10).to(torch.bfloat16).cuda(), torch.ones(N, dtype=torch.bfloat16, device="cuda"))
    assert h._w4_prompt_on_tiles(T) and not hb._w4_prompt_on_tiles(T)      # (the GEMM adds a bias before it rounds)
    y, y_add = h.forward(x), h.forward(x, add1=a1)
    assert torch.equal(y_add, a1 + y)
    monkeypatch.setattr(n.LinearHandle, "_w4_prompt_on_tiles", lambda self, T: False)
    want = h.forward(x)
    if K <= 2048 or T > 1024:
        assert torch.equal(y, want)
    else:
        assert float((y != want).float().mean()) < 0.01
        torch.testing.assert_close(y.float(), want.float(), rtol=2.0 ** -7, atol=1e-5)


def w4_prompt_both_ways(K, N, T, G=64, max_len=2048):
    """A W4 handle whose prompts of T rows the tiles take, rows for it, and a function that makes the same call on the expansion and the GEMM."""
    n = native()
    torch.manual_seed(K + N + T)
    h = n.LinearHandle(K, N, "W4", G, max_len)
    h.load_bf16((torch.randn(N, K) / 10).to(torch.bfloat16).cuda())
    assert h._w4_prompt_on_tiles(T)

    def on_the_gemm(*a, **kw):
        h._w4_prompt_on_tiles = lambda T: False
        try:
            return h.forward(*a, **kw)
        finally:
            del h._w4_prompt_on_tiles
    return h, (torch.randn(T, K) / 10).to(torch.bfloat16).cuda(), on_the_gemm


@pytest.mark.parametrize("K,N,T", [(2048, 2112, 600), (1024, 1024, 520)])     # (both sides give the same bits: K is one piece)
def test_a_w4_prompt_fills_any_out(K, N, T):
    """`out` as torch takes it: dense, a column slice of a wider buffer, rows that lie further apart, fp32, transposed, on the host, over the input (N = K); what
    has another number of rows is refused before anything is written."""
    h, x, on_the_gemm = w4_prompt_both_ways(K, N, T)
    want = on_the_gemm(x)
    wide = torch.full((T, 2 * N), 7.0, dtype=torch.bfloat16, device="cuda")
    for out in (torch.empty_like(want), wide[:, :N], wide[:, N:], torch.empty((2 * T, N), dtype=torch.bfloat16, device="cuda")[::2], torch.empty((T, N), device="cuda"),
                torch.empty((N, T), dtype=torch.bfloat16, device="cuda").t(), torch.empty((1, T, N), dtype=torch.bfloat16, device="cuda"), torch.empty((T, N), dtype=torch.bfloat16),
                torch.empty(T * N + 1, dtype=torch.bfloat16, device="cuda")[1:].view(T, N)):
        if out.untyped_storage().data_ptr() == wide.untyped_storage().data_ptr():
            wide.fill_(7.0)
        y = h.forward(x, out=out)
        assert y.data_ptr() == out.data_ptr() and torch.equal(out.view(T, N).to("cuda", torch.bfloat16) if out.is_contiguous() else out.to(torch.bfloat16), want), (out.shape, out.stride(), out.dtype)
        if out.data_ptr() == wide.data_ptr():
            assert bool((wide[:, N:] == 7.0).all())
    assert bool((wide[:, :N] == 7.0).all())
    # (a dense buffer with room for the rows asked for, so that a kernel that looked at its address alone would stay inside it)
    room = torch.zeros((T, N), dtype=torch.bfloat16, device="cuda")
    with pytest.raises(RuntimeError):
        h.forward(x, out=room[:T - 1])
    assert not bool(room.any())
    if K == N:
        both = x.clone()
        h.forward(both, out=both)
        assert torch.equal(both, want)


def test_a_w4_prompt_adds_what_torch_adds():
    """Addends of bf16 rows go into the tiles' epilogue; of another dtype, with strided columns, as (1, T, N), with rows far apart, and in halves behind GLU
    they are added as the GEMM's callers always could."""
    K, N, T = 2048, 2112, 600
    h, x, on_the_gemm = w4_prompt_both_ways(K, N, T)
    a = torch.randn((T, N), device="cuda")
    b = a.to(torch.bfloat16)
    far = torch.randn((T, N + 24), device="cuda").to(torch.bfloat16)[:, 8:8 + N]
    half = torch.randn((T, N // 2), device="cuda").to(torch.bfloat16)
    for kw in (dict(add1=b), dict(add1=a), dict(add1=b, add2=a), dict(add1=b.t().contiguous().t()), dict(add1=b.view(1, T, N), add2=far), dict(add2=far),
               dict(glu=True), dict(glu=True, add1=half), dict(glu=True, add1=half, add2=half.float())):
        want, got = on_the_gemm(x, **kw), h.forward(x, **kw)
        assert got.dtype == want.dtype and torch.equal(got, want), {k: getattr(v, "dtype", v) for k, v in kw.items()}
    want = on_the_gemm(x, add1=b)
    here = torch.cat((b, b))
    assert torch.equal(h.forward(x, add1=here[T:], out=here[T:]), want)                  # the residual in place
    assert torch.equal(h.forward(x, add1=here[:T], out=here[1:T + 1]), want)             # one row further on in the same buffer
    for kw in (dict(add1=b[:T - 1]), dict(add1=b[:, :N - 8]), dict(glu=True, add1=b)):
        with pytest.raises(RuntimeError):
            h.forward(x, **kw)


@pytest.mark.parametrize("fmt,T", [("W4", 600), ("W4", 700), ("W4", 40), ("FP8", 3), ("BF16", 300)])
def test_one_row_expanded_to_many(fmt, T):
    """Inputs and addends of stride 0 are the row that they repeat, on the tiles, the GEMM and the decode kernel."""
    n = native()
    K, N = 2048, 2112
    torch.manual_seed(T)
    h = n.LinearHandle(K, N, fmt, {"W4": 64, "FP8": 128, "BF16": 0}[fmt], 1024)
    w = (torch.randn(N, K) / 10).to(torch.bfloat16).cuda()
    if fmt == "FP8":
        h.load_fp8((w.float() * 4).to(torch.float8_e4m3fn), ((torch.rand((N + 127) // 128, K // 128) + 0.5) / 32).cuda())
    else:
        h.load_bf16(w)
    x, a = (torch.randn(1, K) / 10).to(torch.bfloat16).cuda().expand(T, K), torch.randn(1, N).to(torch.bfloat16).cuda().expand(T, N)
    xc, ac = x.contiguous(), a.contiguous()
    assert torch.equal(h.forward(x), h.forward(xc))
    assert torch.equal(h.forward(x, add1=a, add2=a), h.forward(xc, add1=ac, add2=ac))


@pytest.mark.parametrize("K,N,T,G", [(4096, 4096, 512, 64), (7168, 18440, 520, 128), (7168, 4096, 1000, 32)])     # K cut, another launch adds; K whole, strips and rows absent; K cut in two
def test_w4_prompts_on_tiles_of_128_rows(K, N, T, G):
    """The rounded multiplicand on tiles of 128 rows and 256 features: rows of one power of two give the GEMM's bits (an output is one product), random ones differ in fewer than
    1 in 100 and by a bf16 step (see above), and RMSNorm in front, rows that lie further apart and a dense `out` change nothing."""
    n = native()
    h, x, on_the_gemm = w4_prompt_both_ways(K, N, T, G)
    ones = torch.zeros_like(x)
    ones[torch.arange(T), torch.randint(0, K, (T,))] = (2.0 ** torch.randint(-4, 5, (T,)).float()).to(torch.bfloat16).cuda()
    n.timing_enable(2)
    try:
        y = h.forward(ones)
        labels = [t[0] for t in n.timing_collect()]
    finally:
        n.timing_enable(0)
    assert any(t.startswith("lin_tile_kernel<W4,MT8,NW8,NSW2>") for t in labels), labels
    assert torch.equal(y, on_the_gemm(ones))
    y, want = h.forward(x), on_the_gemm(x)
    assert float((y != want).float().mean()) < 0.01
    torch.testing.assert_close(y.float(), want.float(), rtol=2.0 ** -7, atol=1e-5)
    far = torch.zeros((T, K + 64), dtype=torch.bfloat16, device="cuda")[:, :K]
    far.copy_(x)
    out, nw = torch.empty_like(y), (1 + torch.randn(K) / 10).to(torch.bfloat16).cuda()
    assert torch.equal(h.forward(far), y) and h.forward(x, out=out) is out and torch.equal(out, y)
    assert torch.equal(h.forward(far, norm=(nw, 1e-6)), h.forward(n.rmsnorm(x, nw, 1e-6)))


@pytest.mark.parametrize("K,N,T", [(2048, 272, 520), (7168, 272, 520), (2048, 2112, 600)])      # K in one piece; in pieces that another launch adds
def test_a_w4_prompt_keeps_subnormal_results(K, N, T):
    """Outputs under 2^-126, and sums and GLU products of such, are those of the GEMM and of torch.  A row of x is one power of two, so that an output is one product and
    its bits don't depend on the order of the sums."""
    h, _, on_the_gemm = w4_prompt_both_ways(K, N, T)
    x = torch.zeros((T, K), dtype=torch.bfloat16, device="cuda")
    x[torch.arange(T), torch.randint(0, K, (T,))] = (2.0 ** -torch.randint(40, 132, (T,)).float()).to(torch.bfloat16).cuda()
    a = (torch.randn((T, N), device="cuda") * 2.0 ** -128).to(torch.bfloat16)
    for kw in (dict(), dict(add1=a), dict(add1=a, add2=-a), dict(glu=True)):
        want, got = on_the_gemm(x, **kw), h.forward(x, **kw)
        small = (want != 0) & (want.float().abs() < 2.0 ** -126)
        assert float(small.float().mean()) > 0.005 and torch.equal(got, want)


@pytest.mark.parametrize("G", [32, 64, 128])
@pytest.mark.parametrize("K,N,T", [(2048, 264, 520), (2048, 4096, 512)])      # 64 x 64 tiles, 64 x 128 tiles
def test_w4_prompts_of_any_scale(G, K, N, T):
    """Scales of 0, subnormal, tiny, 2^124 and more, infinite and NaN: the tiles' multiplicand is ktx_linear_dequant_bf16's.  A row of x is one power of two, so that an
    output is one product."""
    n = native()
    g = torch.Generator().manual_seed(G + N)
    q = torch.randint(0, 16, (K, N), generator=g, dtype=torch.uint8)
    special = torch.tensor([0.0, 2.0 ** -133, 2.0 ** -127, -2.0 ** -120, 1.0, -3.0, 2.0 ** 124, 2.0 ** 125, -2.0 ** 126, 3.3e38, float("inf"), float("-inf"), float("nan")]).to(torch.bfloat16)
    s = special[torch.randint(0, 10, (K // G, N), generator=g)]
    s[:, :len(special)] = special          # (an infinite weight makes every output of its column NaN: in these columns, and in the others q - 8 is what s leaves room for)
    room = (3.38e38 / s.float().abs()).clamp(max=8).floor().repeat_interleave(G, dim=0)[:, len(special):]
    q[:, len(special):] = torch.minimum(torch.maximum(q[:, len(special):].float(), 8 - room), 8 + room).clamp(0, 15).to(torch.uint8)
    h = n.LinearHandle(K, N, "W4", G, T)
    h.load_w4(q.cuda(), s.cuda())
    assert h._w4_prompt_on_tiles(T)
    x = torch.zeros((T, K), dtype=torch.bfloat16)
    x[torch.arange(T), torch.randint(0, K, (T,), generator=g)] = 0.25
    y = h.forward(x.cuda())
    h._w4_prompt_on_tiles = lambda T: False
    want = h.forward(x.cuda())
    assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y[~y.isnan()], want[~want.isnan()])
    # (q - 8) s, rounded to bf16, with q - 8 in 64 bits
    w = ((q.double() - 8.0) * s.double().repeat_interleave(G, dim=0)).float().to(torch.bfloat16)
    finite = w.float().isfinite().all(0)
    assert 0.9 < float(finite.float().mean()) < 1 and torch.equal(y.cpu()[:, finite].float(), (x.float() @ w[:, finite].float()).to(torch.bfloat16).float())


# ---- lin_sk_kernel (round 3): the decode GEMV dealt over all CUs ----------------------------------------------------------
# Shapes: DeepSeek-V3 linears (k-steps 56 / 128 / 144 / 12 / 16 -> ring depths 7 / 8 / 6 / 4), a glu pair, ragged N.
SK_SHAPES = [(7168, 2112), (16384, 7168), (18432, 1024), (1536, 3072), (2048, 7168), (7168, 4096), (896, 200), (1408, 512)]


def _knobs(n, **kv):
    class K:
        def __enter__(self):
            for k, v in kv.items():
                n.lib.ktx_debug_set(int(k[1:]), v)

        def __exit__(self, *a):
            for k in kv:
                n.lib.ktx_debug_set(int(k[1:]), 0)
    return K()


@pytest.mark.parametrize("K,N", SK_SHAPES)
@pytest.mark.parametrize("T", [1, 2, 4])
def test_all_cu_decode_gemv_both_deals_against_the_reference_math(K, N, T):
    """The all-CU decode GEMV with whole strips per workgroup (default) and with single groups dealt (knob 17 = 1: strips
    shared between workgroups meet through the fixed-point words) against exact (q - 8) * s math, against round 2's
    lin_dec_kernel (knob 16 = 1), and against itself: the shared-strip path adds integers, so replays are bit-identical
    whatever the arrival order, and the meeting words must be back at zero after every launch."""
    n = native()
    torch.manual_seed(K * 3 + N + T)
    w = (torch.randn(N, K) / 10).to(torch.bfloat16)
    x = (torch.randn(T, K) / 10).to(torch.bfloat16)
    q, s = quantize_weights_ref(w.T.contiguous(), 64)
    ref = linear_w4_ref(x, q, s, 64, None)
    h = n.LinearHandle(K, N, "W4", 64, 16)
    h.load_bf16(w.cuda())
    xg = x.cuda()
    y_strips = h.forward(xg)
    close(y_strips, ref)
    with _knobs(n, k17=1):
        y_groups = [h.forward(xg).clone() for _ in range(4)]
    close(y_groups[0], ref)
    for y in y_groups[1:]:
        assert torch.equal(y, y_groups[0]), "shared strips: replays differ (arrival-order dependence or words not reset)"
    with _knobs(n, k16=1):
        y_old = h.forward(xg)
    close(y_old, ref)
    # the two deals differ only in fp32 association (+ the 2^-32 grid of the meeting words): within one bf16 ulp of each other
    d = (y_strips.float() - y_groups[0].float()).abs()
    assert bool((d <= y_strips.float().abs() * 2.0 ** -7 + 1e-6).all())


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), 3.0e38])
def test_shared_strip_words_do_not_swallow_non_finite_parts(bad):
    """a strip shared between workgroups meets through fixed-point words; a part that is NaN, Inf or
    beyond the words' range used to be clamped into a NUMBER (fminf / fmaxf drop a NaN).  It now travels as a marker no sum of
    in-range parts can reach and the finisher writes NaN: a poisoned input row gives non-finite outputs under BOTH deals, the
    words are back at zero afterwards (a clean row right behind it is exact again)."""
    n = native()
    torch.manual_seed(11)
    K, N = 7168, 2112
    w = (torch.randn(N, K) / 10).to(torch.bfloat16)
    h = n.LinearHandle(K, N, "W4", 64, 16)
    h.load_bf16(w.cuda())
    x = (torch.randn(1, K) / 10).to(torch.bfloat16)
    xb = x.clone()
    xb[0, 5] = bad                      # (3e38 * a weight of ~0.1 over a 1 KiB tile stays finite in fp32 but leaves the words' +-2^18 range)
    q, s = quantize_weights_ref(w.T.contiguous(), 64)
    ref = linear_w4_ref(x, q, s, 64, None)
    for knobs in ({}, {"k17": 1}):
        with _knobs(n, **knobs):
            y_bad = h.forward(xb.cuda())
            y_ok = h.forward(x.cuda())
        assert not bool(torch.isfinite(y_bad.float()).all()), f"deal {knobs or 'whole strips'}: the poisoned row came out finite"
        if knobs:   # every output of the row depends on x[5] (one k-step of every strip): all of them must be flagged
            assert float(torch.isfinite(y_bad.float()).float().mean()) < 0.01
        close(y_ok, ref)


@pytest.mark.parametrize("T", [1, 3])
def test_all_cu_decode_gemv_epilogues(T):
    """Fused RMSNorm prologue, glu, bias and both addends through lin_sk_kernel == the same call through lin_dec_kernel up to
    fp32 association (the arithmetic of the prologue and the epilogues is shared expression by expression)."""
    n = native()
    K, N = 7168, 4096
    torch.manual_seed(5 + T)
    w = (torch.randn(N, K) / 10).to(torch.bfloat16).cuda()
    x = torch.randn(T, K).to(torch.bfloat16).cuda()
    nw = (1 + 0.1 * torch.randn(K)).to(torch.bfloat16).cuda()
    a1 = torch.randn(T, N).to(torch.bfloat16).cuda()
    a2 = torch.randn(T, N).to(torch.bfloat16).cuda()
    bias = torch.randn(N).to(torch.bfloat16).cuda()
    h = n.LinearHandle(K, N, "W4", 64, 16)
    h.load_bf16(w, bias)
    hg = n.LinearHandle(K, N, "W4", 64, 16)
    hg.load_bf16(w)
    for kw, hh in ((dict(norm=(nw, 1e-6), add1=a1, add2=a2), h), (dict(norm=(nw, 1e-6), glu=True), hg), (dict(add1=a1), h)):
        y_new = hh.forward(x, **kw)
        with _knobs(n, k16=1):
            y_old = hh.forward(x, **kw)
        with _knobs(n, k17=1):
            y_grp = hh.forward(x, **kw)
        for y in (y_new, y_grp):
            d = (y.float() - y_old.float()).abs()
            assert bool((d <= y_old.float().abs() * 2.0 ** -6 + 2e-2 * y_old.float().abs().max()).all()), float(d.max())
            assert float((y.float() - y_old.float()).norm() / y_old.float().norm()) < 4e-3


def test_all_cu_decode_gemv_under_a_replayed_graph_and_many_handles():
    """Meeting words, slab arena and launch geometry under graph replay: 12 handles created and destroyed in shuffled order
    (slabs are returned when their last piece goes), a captured chain replayed 20 times gives the same bits every time."""
    n = native()
    torch.manual_seed(3)
    K, N = 2048, 1536
    hs, ws = [], []
    for i in range(12):
        w = (torch.randn(N, K) / 10).to(torch.bfloat16).cuda()
        h = n.LinearHandle(K, N, "W4", 64, 8)
        h.load_bf16(w)
        hs.append(h); ws.append(w)
    for i in (1, 5, 7, 2):
        hs[i].close()
    live = [h for i, h in enumerate(hs) if i not in (1, 5, 7, 2)]
    x = (torch.randn(1, K) / 10).to(torch.bfloat16).cuda()
    ys = [torch.empty(1, N, dtype=torch.bfloat16, device="cuda") for _ in live]
    with _knobs(n, k17=1):
        for h, y in zip(live, ys):
            h.forward(x, out=y)
        torch.cuda.synchronize()
        first = [y.clone() for y in ys]
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            for h, y in zip(live, ys):
                h.forward(x, out=y)
        for _ in range(20):
            for y in ys:
                y.zero_()
            g.replay()
            torch.cuda.synchronize()
            for y, f in zip(ys, first):
                assert torch.equal(y, f)


@pytest.mark.parametrize("act_order", [False, True])
@pytest.mark.parametrize("T", [1, 5, 70])
def test_marlin_8bit_operator_multiplies_with_the_reference_multiplicand(T, act_order):
    """KLinearMarlin(num_bits=8) (linear.py:608-666): Marlin's 8-bit multiplicand bf16((q - 128) * s) — pinned to the reference's
    own quantize_weights in tests/test_linear_cpu.py — now formed in registers from the W8 format (one byte per weight); forward
    against fp64 math on that matrix, at the bound of the BF16 kernels (one bf16 rounding of an fp32-accumulated sum)."""
    from types import SimpleNamespace
    from ktransformers_amd.operators.linear import KLinearMarlin, marlin_multiplicand
    from ktransformers_amd.util.loader import DictLoader
    K, N, G = 2048, 576, 64
    torch.manual_seed(T + 31 * act_order)
    w = (torch.randn(N, K) / 10).to(torch.bfloat16)
    x = (torch.randn(T, K) / 10).to(torch.bfloat16)
    op = KLinearMarlin("k", DictLoader({"k.weight": w}), SimpleNamespace(), torch.nn.Linear(K, N, bias=False, device="meta"),
                       device="cuda", num_bits=8, group_size=G, act_order=act_order)
    op.load()
    assert op._h.fmt == "W8" and N * K <= op._h.weight_bytes() < 1.1 * N * K
    y = op.forward(x.cuda())
    torch.cuda.synchronize()
    close(y.cpu(), linear_bf16_ref(x, marlin_multiplicand(w, 8, G)), rel=1e-3)
    # the 8-bit grid is 16x finer than the 4-bit one
    dense = x.double() @ w.double().T
    assert float((y.cpu().double() - dense).norm() / dense.norm()) < 1e-2


@pytest.mark.parametrize("fmt", ["W4", "FP8", "BF16"])
@pytest.mark.parametrize("K,N,T", [(2048, 576, 5), (7168, 2112, 8), (1536, 3072, 7), (16384, 7168, 8)])
def test_five_to_eight_rows_run_as_four_row_passes_of_the_decode_kernel(fmt, K, N, T):
    """Round 6: a 5..8-row call of an unbatched handle is two launches of the decode GEMV (rows 0-3, rows 4..), so every row carries the
    decode kernel's bits — with the fused RMSNorm, the addends (offset by the pass), the GLU epilogue, strided rows and a device-side row
    count — and stays within the file's bound of the 16-row-strip kernel it replaces (dev knob 3 = 1)."""
    n = native()
    torch.manual_seed(K + N + T)
    w = (torch.randn(N, K) / 10).to(torch.bfloat16).cuda()
    if fmt == "FP8":
        h = n.LinearHandle(K, N, "FP8", 128, 16)
        h.load_fp8((w.float() * 4).to(torch.float8_e4m3fn), ((torch.rand((N + 127) // 128, K // 128) + 0.5) / 32).cuda())
    else:
        h = n.LinearHandle(K, N, fmt, 64 if fmt == "W4" else 0, 16)
        h.load_bf16(w)
    x = (torch.randn(T, K) / 4).to(torch.bfloat16).cuda()
    add1 = (torch.randn(T, N) / 10).to(torch.bfloat16).cuda()
    nw = (1 + torch.randn(K) / 10).to(torch.bfloat16).cuda()
    xs = torch.zeros(T, K + 64, dtype=torch.bfloat16, device="cuda")[:, :K]
    xs.copy_(x)
    assert h.decode_eligible(T) and h.decode_eligible(4)
    calls = [dict(), dict(add1=add1), dict(norm=(nw, 1e-6)), dict(add1=add1, add2=add1), dict(norm=(nw, 1e-6), add1=add1)]
    if N % 16 == 0 and fmt == "W4":
        calls.append(dict(glu=True))

    def rows(kw, a, b):
        kw2 = {k: (v[a:b] if k in ("add1", "add2") else v) for k, v in kw.items()}
        return h.forward(x[a:b].contiguous(), **kw2)

    for kw in calls:
        got = h.forward(x, **kw)
        want = torch.cat([rows(kw, 0, 4), rows(kw, 4, T)], dim=0)
        assert got.shape == want.shape and torch.equal(got, want), f"{fmt} {tuple(kw)}: the passes are not the decode kernel's rows"
    assert torch.equal(h.forward(xs), h.forward(x)), "strided rows"
    bsz = torch.tensor([T - 2], dtype=torch.int32, device="cuda")
    yb = h.forward(x, bsz_tensor=bsz)
    assert torch.equal(yb[: T - 2], h.forward(x)[: T - 2]) and not bool(yb[T - 2:].any()), "device-side row count across the passes"
    fast = [h.forward(x, **kw) for kw in calls[:2]]
    n.check(n.lib.ktx_debug_set(3, 1))
    try:
        assert not h.decode_eligible(T)
        slow = [h.forward(x, **kw) for kw in calls[:2]]
    finally:
        n.check(n.lib.ktx_debug_set(3, 0))
    for a, b in zip(fast, slow):
        close(a, b.cpu())


@pytest.mark.parametrize("fmt", ["W4", "FP8", "BF16"])
@pytest.mark.parametrize("K,N,T", [(128, 17, 9), (384, 200, 33), (2176, 577, 16), (7168, 2112, 65), (2176, 1040, 130), (2048, 4104, 300),
                                   (5248, 577, 16), (2816, 1040, 40), (7168, 1536, 513), (2048, 12288, 520)])
def test_batches_and_short_prompts_on_tiles(fmt, K, N, T):
    """ktx_linear_forward_ws (ktx_linear_tile.inc; BF16 of 256 rows and more, where they fill the chip, the GEMM's 256 x 256 tiles in parts of K):
    ragged rows, features and last k-chunk, split and whole K, bias, addends, GLU, strided and misaligned rows, a device-side row count —
    against the oracle at the file's bound; and, where the tiles take a call, an operator's rows do not depend on what else is in the matrix
    (K is cut by K and T alone)."""
    n = native()
    torch.manual_seed(K + N + T)
    w = (torch.randn(N, K) / 10).to(torch.bfloat16)
    x = (torch.randn(T, K) / 10).to(torch.bfloat16)
    bias = (torch.randn(N) / 10).to(torch.bfloat16)
    w8, sc = (torch.randn(N, K) / 4).to(torch.float8_e4m3fn), (torch.rand((N + 127) // 128, K // 128) + 0.5) / 32

    def handle(rows, b):
        h = n.LinearHandle(K, rows, fmt, {"W4": 64, "FP8": 128, "BF16": 0}[fmt], 1024)
        bb = bias[:rows].cuda() if b else None
        if fmt == "FP8":
            h.load_fp8(w8[:rows].cuda(), sc[: (rows + 127) // 128].cuda(), bb)
        else:
            h.load_bf16(w[:rows].cuda(), bb)
        return h

    ref = (linear_fp8_ref(x, w8, sc) if fmt == "FP8" else linear_bf16_ref(x, w) if fmt == "BF16" else
           linear_w4_ref(x, *quantize_weights_ref(w.T.contiguous(), 64), 64, round_weights=T >= 512)).float()

    h, hb, xc = handle(N, False), handle(N, True), x.cuda()
    y = h.forward(xc)
    close(y, ref, rel=2e-3)
    # the bias is added to the rounded sum (or, in the W4 GEMM, to the sum): a half ulp of either, on top of the half ulp that y carries
    want = y.float() + bias.cuda().float()
    assert bool(((hb.forward(xc).float() - want).abs() <= 2.0 ** -8 * (y.float().abs() + want.abs())).all()), "bias"
    a1, a2 = (torch.randn(T, N).to(torch.bfloat16).cuda() for _ in range(2))
    assert torch.equal(h.forward(xc, add1=a1, add2=a2), a2 + (a1 + y))
    wide = torch.zeros(T, K + 64, dtype=torch.bfloat16, device="cuda")
    wide[:, 8:K + 8] = xc
    assert torch.equal(h.forward(wide[:, 8:K + 8]), y), "strided rows"
    wide[:, 3:K + 3] = xc
    close(h.forward(wide[:, 3:K + 3]), ref, rel=2e-3)
    got = h.forward(xc, bsz_tensor=torch.tensor([T - 3], dtype=torch.int32, device="cuda"))
    exact = linear_w4_ref(x, *quantize_weights_ref(w.T.contiguous(), 64), 64).float() if fmt == "W4" else ref   # (no rounded weights with a row count)
    close(got[: T - 3], exact[: T - 3], rel=2e-3)
    assert not bool(got[T - 3:].any())
    if N % 16 == 0:
        g = y.float().view(T, N // 16, 2, 8)
        s = (g[:, :, 0] / (1 + torch.exp(-g[:, :, 0]))).to(torch.bfloat16).float()
        close(h.forward(xc, glu=True), (s * g[:, :, 1]).reshape(T, N // 2).cpu(), rel=5e-3)
    if N > 256 and T < 512:
        assert torch.equal(handle(256, False).forward(xc), y[:, :256]), "a merged operator's rows"


@pytest.mark.parametrize("G", [32, 64, 128])
@pytest.mark.parametrize("K,N,T,how", [(2048, 577, 513, "odd"), (1024, 1000, 512, "rows"), (7168, 264, 640, "capture"), (2048, 12296, 600, "rows"), (384, 33, 1030, "odd")])
def test_w4_prompts_off_the_gemm_multiply_exact_integers(G, K, N, T, how):
    """512 rows and more that the prompt path doesn't take (out_features % 8 != 0, a device-side row count, stream capture) multiply
    (q - 8) exactly and scale in fp32; only that path's multiplicand is rounded to bf16.  Against 64-bit sums an exact product is off by the
    outputs' rounding alone: uniform in half an ulp, 2^-8 / sqrt(12) = 1.1e-3 of a power of two and 1.66e-3 in the norm over mantissas; the
    rounded multiplicand adds an independent error to every term whose (q - 8) * s doesn't fit bf16: 2.1e-3 and more.  2.0e-3 parts the two."""
    n = native()
    torch.manual_seed(K + N + T + G)
    w = (torch.randn(N, K) / 10).to(torch.bfloat16)
    x = (torch.randn(T, K) / 10).to(torch.bfloat16)
    q, s = quantize_weights_ref(w.T.contiguous(), G)
    want = x.cuda().double() @ ((q.double().cuda() - 8.0) * s.cuda().double().repeat_interleave(G, dim=0))
    h = n.LinearHandle(K, N, "W4", G, T)
    h.load_bf16(w.cuda())
    xc = x.cuda()
    if how == "odd":
        y = h.forward(xc)
    elif how == "rows":
        y = h.forward(xc, bsz_tensor=torch.tensor([T], dtype=torch.int32, device="cuda"))
    else:
        y = torch.empty(T, N, dtype=torch.bfloat16, device="cuda")
        h.forward(xc, out=y)
        eager = y.clone()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            h.forward(xc, out=y)
        for _ in range(3):
            y.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert float((y.double() - want).norm() / want.norm()) < 2.0e-3
        assert float((eager.double() - want).norm() / want.norm()) > 2.0e-3     # (the eager call rounds the weights)
    close(y, want.float().cpu())
    assert float((y.double() - want).norm() / want.norm()) < 2.0e-3


@pytest.mark.parametrize("fmt,group", [("W4", 64), ("W4", 128), ("FP8", 128)])
@pytest.mark.parametrize("K,N,T", [(4096, 12000, 33), (4096, 10244, 64), (16384, 5130, 48),   # 188, 164 and 168 workgroups; whole strips, a part of one, rows absent
                                   (2176, 32768, 33), (2944, 32641, 64), (2944, 32640, 48)])   # 64 x 128 tiles on all CUs, which add the pieces of K themselves; and on one less
def test_tiles_of_64_rows_and_256_features(fmt, group, K, N, T):
    """The 64 x 256 tiles against the 64 x 128 ones (dev knob 32 = 1): the same pieces of K, the same bits."""
    from ktransformers_amd import _native
    g = torch.Generator().manual_seed(K + N + T)
    dev = torch.device("cuda", 0)
    h = _native.LinearHandle(K, N, fmt, group, T, dev)
    if fmt == "FP8":
        h.load_fp8((torch.randn((N, K), generator=g) * 100).clamp_(-448, 448).to(torch.float8_e4m3fn).to(dev), torch.rand((-(-N // 128), K // 128), generator=g).to(dev))
    else:
        h.load_bf16((torch.randn((N, K), generator=g) * K ** -0.5).to(torch.bfloat16).to(dev))
    x = torch.randn((T, K), generator=g).to(torch.bfloat16).to(dev)
    got = []
    try:
        for knob in (1, 0):
            _native.lib.ktx_debug_set(32, knob)
            h._ws_need.clear()
            got.append(h.forward(x).clone())
    finally:
        _native.lib.ktx_debug_set(32, 0)
    assert torch.equal(*got)


@pytest.mark.parametrize("fmt,group", [("W4", 32), ("W4", 64), ("W4", 128), ("FP8", 128), ("BF16", 0)])
@pytest.mark.parametrize("K,N", [(2816, 577), (4096, 12000), (7168, 264)])     # 64 x 64, 64 x 256 (W4, FP8) and 64 x 64 tiles in more pieces of K
def test_tiles_of_48_rows(fmt, group, K, N):
    """33 to 48 rows on tiles of 48: the bits that the same rows have among 49, on tiles of 64 (K is cut by K and T alone, alike up to 256 rows)."""
    from ktransformers_amd import _native
    g = torch.Generator().manual_seed(K + N)
    dev = torch.device("cuda", 0)
    h = _native.LinearHandle(K, N, fmt, group, 64, dev)
    if fmt == "FP8":
        h.load_fp8((torch.randn((N, K), generator=g) * 100).clamp_(-448, 448).to(torch.float8_e4m3fn).to(dev), torch.rand((-(-N // 128), K // 128), generator=g).to(dev))
    else:
        h.load_bf16((torch.randn((N, K), generator=g) * K ** -0.5).to(torch.bfloat16).to(dev))
    x = torch.randn((49, K), generator=g).to(torch.bfloat16).to(dev)
    want = h.forward(x)
    for T in (33, 47, 48):
        assert torch.equal(h.forward(x[:T]), want[:T]), f"{T} rows"


@pytest.mark.parametrize("K,N", [(2816, 8200), (4096, 12000), (2176, 32768)])     # tiles of 48 rows and 64, 256 and 128 features
def test_fp8_prompts_of_33_rows_and_more_take_the_k_128_mfma(K, N):
    """ktx_linear_forward_ws with prompt = 1, which holds past 32 rows: 33 to 48 have the bits that they have among 49, on tiles of 64 rows.  Magnitudes over many
    powers of two, half of them cancelling: 8 results in 100000 show the order of the sums (none does with normal weights)."""
    n = native()
    g = torch.Generator().manual_seed(K + N)
    h = n.LinearHandle(K, N, "FP8", 128, 64)
    w = torch.randn((N, K), generator=g).abs() * torch.exp2(torch.randint(-12, 4, (N, K), generator=g).float())
    x = torch.randn((49, K), generator=g) * torch.exp2(torch.randint(-12, 8, (49, K), generator=g).float())
    x[:, 0::2] = -x[:, 1::2]
    h.load_fp8((w * 100).clamp_(max=448).to(torch.float8_e4m3fn).cuda(), torch.rand((-(-N // 128), K // 128), generator=g).cuda())
    x = x.to(torch.bfloat16).cuda()

    def forward(T, prompt):
        y, need = torch.empty((T, N), dtype=torch.bfloat16, device="cuda"), n.lib.ktx_linear_workspace_bytes(h._h, T, 1)
        ws = torch.empty(need, dtype=torch.uint8, device="cuda")
        n.check(n.lib.ktx_linear_forward_ws(h._h, None, T, x.data_ptr(), y.data_ptr(), None, prompt, ws.data_ptr(), need, n._stream_ptr(x.device)))
        return y
    want, other = forward(49, 1), forward(49, 0)
    for T in (33, 47, 48):
        assert torch.equal(forward(T, 1), want[:T]), f"{T} rows"
        assert torch.equal(forward(T, 0), other[:T]) and not torch.equal(other[:T], want[:T])


@pytest.mark.parametrize("N", [24576, 24584])
def test_bf16_prompts_on_the_gemm_of_decode_tiles(N):
    """520 rows of 2048 -> 24576 (whole strips) and 24584 (half a strip at the end) fill the chip with 256 x 256 tiles over the whole K: the GEMM
    reads the decode tiles and writes y itself.  Against 64-bit sums at the file's bound; into strided rows of a larger buffer; with a bias or a
    row count the same sums go through fp32 to the tiles' epilogue: the same bits as the rounded sums with the bias added."""
    n = native()
    K, T = 2048, 520
    torch.manual_seed(N)
    w, x = (torch.randn(N, K, device="cuda") / 10).to(torch.bfloat16), (torch.randn(T, K, device="cuda") / 10).to(torch.bfloat16)
    bias = (torch.randn(N, device="cuda") / 10).to(torch.bfloat16)
    h, hb = n.LinearHandle(K, N, "BF16", 0, T), n.LinearHandle(K, N, "BF16", 0, T)
    h.load_bf16(w)
    hb.load_bf16(w, bias)
    n.timing_enable(2)
    try:
        y = h.forward(x)
        labels = [t[0] for t in n.timing_collect()]
    finally:
        n.timing_enable(0)
    assert len(labels) == 1 and "gemm256_bf16_nt_kernel<bf16,tiles>" in labels[0], labels
    close(y, (x.double() @ w.double().T).float().cpu())
    wide = torch.zeros(T, K + 64, dtype=torch.bfloat16, device="cuda")
    wide[:, 8:K + 8] = x
    assert torch.equal(h.forward(wide[:, 8:K + 8]), y), "strided rows"
    assert torch.equal(hb.forward(x), (y.float() + bias.float()).to(torch.bfloat16)), "bias"
    got = h.forward(x, bsz_tensor=torch.tensor([T - 3], dtype=torch.int32, device="cuda"))
    assert torch.equal(got[: T - 3], y[: T - 3]) and not bool(got[T - 3:].any())


@pytest.mark.parametrize("fmt,K,N,T,kernel", [
    ("BF16", 2048, 7168, 192, "lin_gemm_kernel"), ("BF16", 1536, 4096, 48, "lin_gemm_kernel"), ("BF16", 7168, 2112, 64, "lin_tile_kernel"),
    ("BF16", 4096, 1000, 1025, "lin_gemm_kernel"), ("BF16", 2048, 12288, 1000, "gemm256_bf16_nt_kernel"),
    ("W8", 2048, 3072, 64, "lin_gemm_kernel"), ("W8", 7168, 2112, 64, "lin_tile_kernel"), ("W8", 7168, 2112, 700, "lin_gemm_kernel"),
    ("W4", 2048, 3072, 16, "lin_gemm"), ("W4", 7168, 2112, 16, "lin_tile_kernel"), ("W4", 1536, 2048, 48, "lin_tile_kernel"),
    ("FP8", 2048, 3072, 16, "lin_gemm_kernel"), ("FP8", 2048, 3072, 48, "lin_tile_kernel"), ("FP8", 5120, 9000, 700, "lin_fp8_gemm_kernel"),
    ("FP8", 7168, 2112, 1500, "lin_fp8_gemm_kernel"), ("FP8", 2048, 3072, 1025, "lin_tile_kernel"),
    ("W4", 2176, 2112, 16, "lin_tile_kernel"), ("W4", 128, 2112, 17, "lin_tile_kernel"), ("FP8", 2176, 2112, 16, "lin_tile_kernel"), ("FP8", 256, 2112, 32, "lin_gemm_kernel"),
    ("FP8", 384, 2112, 32, "lin_tile_kernel"), ("FP8", 128, 2112, 33, "lin_tile_kernel"), ("BF16", 2688, 8192, 16, "lin_tile_kernel"), ("BF16", 2688, 8200, 16, "lin_gemm_kernel"),
    ("BF16", 1664, 2112, 17, "lin_tile_kernel"), ("BF16", 2176, 2112, 32, "lin_gemm_kernel"), ("BF16", 2176, 2112, 33, "lin_tile_kernel"), ("W8", 1664, 2112, 64, "lin_gemm_kernel"),
    ("W8", 2176, 2112, 33, "lin_tile_kernel")])
def test_which_kernel_a_batch_takes(fmt, K, N, T, kernel):
    """Strip kernels, tiles or GEMM, where each was measured faster (lin_tile_wins, lin_gemm_parts, LinearHandle.FP8_GEMM_OUT)."""
    n = native()
    h = n.LinearHandle(K, N, fmt, {"W4": 64, "W8": 64, "FP8": 128, "BF16": 0}[fmt], T)
    if fmt == "FP8":
        h.load_fp8(torch.randn(N, K, device="cuda").to(torch.float8_e4m3fn), torch.ones((N + 127) // 128, K // 128, device="cuda"))
    elif fmt == "W8":
        h.load_w8(torch.randint(0, 256, (K, N), dtype=torch.uint8, device="cuda"), torch.ones(K // 64, N, dtype=torch.bfloat16, device="cuda"))
    else:
        h.load_bf16(torch.randn(N, K, device="cuda").to(torch.bfloat16))
    n.timing_enable(2)
    try:
        h.forward(torch.randn(T, K, device="cuda").to(torch.bfloat16))
        labels = [t[0] for t in n.timing_collect()]
    finally:
        n.timing_enable(0)
    assert any(t.startswith(kernel) for t in labels), labels


def test_a_batch_without_memory_for_scratch_runs_on_the_strip_kernels(monkeypatch):
    """The scratch is a want, not a need: where the allocator has none left the call runs as it does without, on the strip kernels."""
    n = native()
    K, N, T = 7168, 264, 48
    torch.manual_seed(1)
    w, x = (torch.randn(N, K) / 10).to(torch.bfloat16), (torch.randn(T, K) / 10).to(torch.bfloat16)
    h = n.LinearHandle(K, N, "W4", 64, T)
    h.load_bf16(w.cuda())
    real, xc = torch.empty, x.cuda()

    def empty(*a, **kw):
        if kw.get("dtype") is torch.uint8:
            raise torch.cuda.OutOfMemoryError("none left")
        return real(*a, **kw)
    monkeypatch.setattr(torch, "empty", empty)
    n.timing_enable(2)
    try:
        y = h.forward(xc)
        labels = [t[0] for t in n.timing_collect()]
    finally:
        n.timing_enable(0)
        monkeypatch.undo()
    assert len(labels) == 1 and labels[0].startswith("lin_gemm"), labels
    close(y, linear_w4_ref(x, *quantize_weights_ref(w.T.contiguous(), 64), 64))


def test_a_w4_prompt_without_memory_for_scratch_multiplies_the_rounded_weights(monkeypatch):
    """Where the allocator has none left for the tiles' scratch a W4 prompt is the GEMM's, with its multiplicand, not the strip kernels'."""
    K, N, T = 7168, 264, 520
    h, x, on_the_gemm = w4_prompt_both_ways(K, N, T)
    want, nw = on_the_gemm(x), torch.ones(K, dtype=torch.bfloat16, device="cuda")
    want_norm = on_the_gemm(x, norm=(nw, 1e-6))
    assert h._scratch(T, True) and not torch.equal(h.forward(x), want)     # (the tiles cut K: other last bits)
    real = torch.empty

    def empty(*a, **kw):
        if kw.get("dtype") is torch.uint8:
            raise torch.cuda.OutOfMemoryError("none left")
        return real(*a, **kw)
    monkeypatch.setattr(torch, "empty", empty)
    got, got_norm = h.forward(x), h.forward(x, norm=(nw, 1e-6))
    monkeypatch.undo()
    assert torch.equal(got, want) and torch.equal(got_norm, want_norm)


def test_calls_go_to_the_current_stream_of_their_device():
    """The raw accessor of the current stream gives torch's own handle, on the default stream and on others, for devices with and without an index."""
    n = native()
    for st in (torch.cuda.default_stream(), torch.cuda.Stream()):
        with torch.cuda.stream(st):
            for dev in (torch.device("cuda", 0), torch.device("cuda")):
                assert n._stream_ptr(dev) == torch.cuda.current_stream(dev).cuda_stream == st.cuda_stream
