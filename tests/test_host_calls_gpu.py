"""csrc/ktx_host.cpp makes the shortest calls without an interpreter step per argument: the same kernels on the same arguments as _native.py's own way, which keeps every
call that the module does not take."""
import copy
import threading
import time

import numpy as np
import pytest
import torch

import ktransformers_amd._native as n

gpu = pytest.mark.gpu


def test_the_module_leaves_what_it_has_not_checked():
    """No call without plain GPU tensors, of whatever arguments: None, and the caller's own checks speak."""
    if n._host is None:
        pytest.skip("needs the built module")
    x, ids, w = torch.zeros((1, 64), dtype=torch.bfloat16), torch.zeros((1, 2), dtype=torch.int64), torch.zeros((1, 2))
    for args in ((), (1, 64, 64, 0, x), (0, 64, 64, 0, x), (1, 64, 64, 0, None), ("1", 64, 64, 0, x), (1, 64, 64, 0, x, x), (2 ** 70, 64, 64, 0, x)):
        assert n._host.linear(*args) is None
    for args in ((), (1, 64, 0, x, ids, w), (1, 64, 0, x, ids, None), (0, 64, 0, x, ids, w)):
        assert n._host.moe(*args) is None
    assert n._host.mla_prefill(*[x] * 5, 1, 1.0) is None and n._host.mla_prefill(x) is None
    for cfg in (1, None, b"short", n._MlaConfig(16, 512, 64, 64, 1.0, 1, 0)):
        assert n._host.mla_decode(cfg, 1, x, x, x, x, ids, ids, None, ids, None, x) is None
    assert n._host.mla_decode() is None
    with pytest.raises(TypeError):
        n._host.bind(1)


class _Count:
    """The module, counting the calls that it took."""

    def __init__(self, module):
        self.module, self.took = module, 0

    def __getattr__(self, name):
        f = getattr(self.module, name)

        def call(*a):
            y = f(*a)
            self.took += y is not None
            return y
        return call


@pytest.fixture
def both(monkeypatch):
    """f(call): the bits that `call` gives from Python and through the module, which are the same, and whether the module took it."""
    if n._host is None:
        pytest.skip("needs the built module")
    module = n._host

    def run(call):
        monkeypatch.setattr(n, "_host", None)
        want = call()
        count = _Count(module)
        monkeypatch.setattr(n, "_host", count)
        got = call()
        monkeypatch.setattr(n, "_host", module)
        assert got.dtype == want.dtype and got.shape == want.shape and got.stride() == want.stride() and got.device == want.device and not got.requires_grad
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
        return count.took
    return run


def _linear(fmt, K=512, N=272):
    h = n.LinearHandle(K, N, fmt, {"W4": 64, "FP8": 128, "BF16": 0}[fmt], 64, 0)
    g = torch.Generator(device="cuda").manual_seed(3)
    w = torch.randn((N, K), device="cuda", generator=g)
    if fmt == "FP8":
        h.load_fp8((w * 50).to(torch.float8_e4m3fn), torch.rand(((N + 127) // 128, K // 128), device="cuda", generator=g))
    else:
        h.load_bf16(w.to(torch.bfloat16))
    return h, torch.randn((16, K), device="cuda", generator=g).to(torch.bfloat16)


@gpu
@pytest.mark.parametrize("fmt", ["W4", "FP8", "BF16"])
def test_linears(both, fmt):
    h, x = _linear(fmt)
    for rows in (1, 2, 7, 8):
        assert both(lambda: h.forward(x[:rows])) == 1, rows
    assert both(lambda: h.forward(torch.nn.Parameter(x[:2]))) == 1
    with torch.inference_mode():
        assert both(lambda: h.forward(x[:2])) == 1
    wide, two = torch.cat((x, x), dim=1), x[:2]
    for call in (lambda: h.forward(x[:9]), lambda: h.forward(x[:4].view(2, 2, -1)), lambda: h.forward(wide[:3, :512]), lambda: h.forward(x[:1].expand(4, -1)),
                 lambda: h.forward(x[:2], out=torch.empty((2, 272), dtype=torch.bfloat16, device="cuda")), lambda: h.forward(x[:2], add1=torch.ones((2, 272), dtype=torch.bfloat16, device="cuda")),
                 lambda: h.forward(x[:4], bsz_tensor=torch.tensor([4], dtype=torch.int32, device="cuda"))):
        assert both(call) == 0
    for bad in (x[:2].float(), x[:2, :256].contiguous(), x[:2].cpu()):
        with pytest.raises(n.KtxError):
            h.forward(bad)
    assert both(lambda: torch.vmap(lambda v: h.forward(two), out_dims=None)(torch.zeros(3))) == 0   # (a tensor of none of its levels, but what is made inside may be wrapped)
    want = h.forward(x[:3])
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        got = h.forward(x[:3])
    s.synchronize()
    assert torch.equal(got, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        held = h.forward(x[:3])
    for _ in range(3):
        held.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(held, want)
    n.TRACE = []
    try:
        h.forward(x[:3])
        assert [name for name, _ in n.TRACE] == ["ktx_linear_forward"]
    finally:
        n.TRACE = None
    with pytest.raises(Exception):
        torch.vmap(lambda v: h.forward(v))(x[:4].view(2, 2, -1))
    h.close()
    with pytest.raises(n.KtxError):
        h.forward(x[:1])


@gpu
def test_experts(both):
    h = n.MoEHandle(8, 2, 512, 256, 64, "AMXINT4", 0)
    g = torch.Generator(device="cuda").manual_seed(4)
    h.load_bf16(*(torch.randn(s, device="cuda", generator=g).to(torch.bfloat16) * 0.05 for s in ((8, 256, 512), (8, 256, 512), (8, 512, 256))))
    x = torch.randn((48, 512), device="cuda", generator=g).to(torch.bfloat16)
    ids, w = torch.randint(-1, 9, (48, 2), device="cuda", generator=g), torch.rand((48, 2), device="cuda", generator=g)
    for T in (1, 3, 48):
        assert both(lambda: h.forward(x[:T], ids[:T], w[:T])) == 1, T
    assert both(lambda: h.forward(x[:2], ids[:2], w[:2], out=torch.zeros_like(x[:2]))) == 0
    assert both(lambda: h.forward(x[:2], ids[:2], w[:2], out=x[2:4].clone(), incremental=True)) == 0
    for bad in ((x[:2].float(), ids[:2], w[:2]), (x[:2], ids[:2].int(), w[:2]), (x[:2], ids[:2], w[:3]), (x[:2], ids[:2], w[:2].double()), (x[:2, :256].contiguous(), ids[:2], w[:2]),
                (x[:2], ids[:2].cpu(), w[:2])):
        with pytest.raises(n.KtxError):
            h.forward(*bad)
    with pytest.raises(n.KtxError):   # more tokens than the handle holds: the library's own refusal
        h.forward(x.repeat(2, 1), ids.repeat(2, 1), w.repeat(2, 1))
    h.close()
    with pytest.raises(n.KtxError):
        h.forward(x[:1], ids[:1], w[:1])


@gpu
@pytest.mark.parametrize("pages_of_one", [False, True])
def test_latent_attention(both, pages_of_one):
    g = torch.Generator(device="cuda").manual_seed(5)
    rand = lambda *s: torch.randn(s, device="cuda", generator=g).to(torch.bfloat16)   # noqa: E731
    B, H, pages = 3, 16, 6
    q, qp, cache = rand(B, H, 512), rand(B, H, 64), rand(pages, 64, 576)
    i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")   # noqa: E731
    wrapper = n.MLAWrapper(B, pages, use_cuda_graph=False, device="cuda", max_q_tokens=B)
    with pytest.raises(n.KtxError):
        wrapper.run(q, qp, cache[..., :512], cache[..., 512:])

    def run(hint=0, q=q, cache=cache, **kw):
        wrapper.plan(i32(0, 1, 2, 3), i32(0, 2, 4, 6), None if pages_of_one else i32(3, 0, 5, 1, 2, 4), i32(100, 128, 65), i32(3), H, 512, 64, 64, 0.07, max_kv_len=hint, identity_pages=pages_of_one)
        return wrapper.run(q, qp, cache[..., :512], cache[..., 512:], **kw)
    for hint in (0, 128):
        assert both(lambda: run(hint)) == 1
    want, held = run(), copy.deepcopy(wrapper)   # (a copy's run reads the copy's sizes, whatever the first wrapper plans next)
    run(128)
    assert both(lambda: held.run(q, qp, cache[..., :512], cache[..., 512:])) == 1 and torch.equal(held.run(q, qp, cache[..., :512], cache[..., 512:]), want)
    held.cfg.sm_scale = 0.14                     # ... and its present values
    assert both(lambda: held.run(q, qp, cache[..., :512], cache[..., 512:])) == 1 and not torch.equal(held.run(q, qp, cache[..., :512], cache[..., 512:]), want)
    assert both(lambda: run(new_ckv=rand(B, 512) * 0, new_kpe=rand(B, 64) * 0)) == 0
    out, lse = run(return_lse=True)
    assert torch.equal(out, run()) and lse.shape == (B, H)
    for bad in (q.float(), rand(B, H, 1024)[..., ::2], rand(B + 1, H, 512)):
        with pytest.raises(n.KtxError):
            run(q=bad)
    with pytest.raises(n.KtxError):
        run(cache=rand(pages, 65, 576)[:, :64])

    T, kv, pad = 70, 100, 128
    q, kn, kp, v = rand(T, H, 192), rand(H, pad, 128), rand(kv, 576), rand(H, 128, pad)
    assert both(lambda: n.mla_prefill(q[..., :128], q[..., 128:], kn, kp[:, 512:], v, kv, 0.07)) == 1
    assert both(lambda: n.mla_prefill(q[..., :128], q[..., 128:], kn, kp[:, 512:], v, np.int64(kv), np.float32(0.07))) == 0
    for bad in ((q[..., :64], q[..., 128:], kn, kp[:, 512:], v), (q[..., :128], q[..., 128:], kn.transpose(0, 1), kp[:, 512:], v), (q[..., :128].float(), q[..., 128:], kn, kp[:, 512:], v)):
        with pytest.raises((n.KtxError, RuntimeError)):
            n.mla_prefill(*bad, kv, 0.07)


@gpu
def test_other_threads_run_while_a_call_waits_for_memory():
    """A call's memory comes without the interpreter's lock: another thread holds the allocator (it gives cached memory back, which waits for the device) while a third one counts."""
    if n._host is None:
        pytest.skip("needs the built module")
    h, x = _linear("BF16")
    a = torch.randn((4096, 4096), device="cuda").to(torch.bfloat16)
    b = torch.empty_like(a)
    for _ in range(3):
        torch.mm(a, a, out=b)
        h.forward(x[:2])
    torch.cuda.synchronize()
    at = {}

    def give_back():
        at["held"] = time.perf_counter()
        torch.cuda.empty_cache()
        at["given"] = time.perf_counter()

    def call():
        at["called"] = time.perf_counter()
        h.forward(x[:2])
        at["returned"] = time.perf_counter()
    cached = torch.empty(512 << 20, dtype=torch.uint8, device="cuda")
    del cached
    for _ in range(3000):
        torch.mm(a, a, out=b)
    threads = [threading.Thread(target=give_back), threading.Thread(target=call)]
    threads[0].start()
    time.sleep(0.03)
    longest, last = 0.0, time.perf_counter()   # (a thread's start() waits for it)
    threads[1].start()
    while threads[1].is_alive():
        time.sleep(0.001)
        longest, last = max(longest, time.perf_counter() - last), time.perf_counter()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    waited = at["returned"] - at["called"]
    if at["called"] >= at["given"] or waited < 0.1:
        pytest.skip(f"the device was done before the call (the allocator was held for {at['given'] - at['held']:.3f} s, the call took {waited:.3f})")
    assert longest < 0.5 * waited, (longest, waited)
