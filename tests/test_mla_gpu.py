"""MLA paged attention against the reference's own torch oracle, at the shapes and tolerance of the reference's
self-test (archive/ktransformers/operators/flashinfer_wrapper.py:254-395: Hq=128, page 64, kv_len 4023 decode and
2 x (q_len 128, kv_len 512) causal prefill, assert_close rtol=atol=5e-3 in bf16), plus V2-Lite/K2 head counts, ragged
batches, non-identity page tables and the latent-cache append."""
import numpy as np
import pytest
import torch

from oracle.mla_ref import mla_paged_ref

from test_mla_prefill_bound import prefill_operands, prefill_scores, prefill_statement

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def run_case(Hq, page_size, kv_lens, q_lens, seed=0, shuffle_pages=False, max_splits=64, rtol=5e-3):
    from ktransformers_amd._native import MLAWrapper
    g = torch.Generator().manual_seed(seed)
    B = len(kv_lens)
    pages_per = [(n + page_size - 1) // page_size for n in kv_lens]
    max_pages = sum(pages_per) + 3
    kv_buf = torch.randn((max_pages, page_size, 576), generator=g).to(torch.bfloat16)
    T = sum(q_lens)
    q_nope = torch.randn((T, Hq, 512), generator=g).to(torch.bfloat16)
    q_pe = torch.randn((T, Hq, 64), generator=g).to(torch.bfloat16)
    perm = torch.randperm(max_pages, generator=g) if shuffle_pages else torch.arange(max_pages)
    kv_indices = perm[:sum(pages_per)].to(torch.int32)
    kv_indptr = torch.tensor([0] + list(np.cumsum(pages_per)), dtype=torch.int32)
    qo_indptr = torch.tensor([0] + list(np.cumsum(q_lens)), dtype=torch.int32)
    kv_len_arr = torch.tensor(kv_lens, dtype=torch.int32)
    sm_scale = 192 ** (-0.5)
    ref, lse_ref = mla_paged_ref(q_nope, q_pe, kv_buf, qo_indptr, kv_indptr, kv_indices, kv_len_arr, sm_scale)

    w = MLAWrapper(B, max_pages, device=DEV, max_q_tokens=T, max_splits=max_splits)
    kvd = kv_buf.to(DEV)
    ckv, k_pe = torch.split(kvd, [512, 64], dim=-1)
    w.plan(qo_indptr.to(DEV), kv_indptr.to(DEV), kv_indices.to(DEV), kv_len_arr.to(DEV),
           torch.tensor([B], dtype=torch.int32, device=DEV), Hq, 512, 64, page_size, sm_scale, torch.bfloat16, torch.bfloat16)
    out, lse = w.run(q_nope.to(DEV), q_pe.to(DEV), ckv, k_pe, return_lse=True)
    torch.cuda.synchronize()
    torch.testing.assert_close(out.float().cpu(), ref.to(torch.bfloat16).float(), rtol=rtol, atol=5e-3)
    torch.testing.assert_close(lse.cpu(), lse_ref, rtol=2e-3, atol=2e-3)


def test_reference_selftest_decode_shape():
    run_case(128, 64, [4023], [1])


def test_reference_selftest_prefill_shape():
    run_case(128, 64, [512, 512], [128, 128], seed=1)


@pytest.mark.parametrize("Hq", [16, 64, 128])      # V2-Lite, Kimi-K2, V3
@pytest.mark.parametrize("kv_len", [1, 31, 32, 33, 1000])
def test_decode_head_counts_and_ragged_lengths(Hq, kv_len):
    run_case(Hq, 64, [kv_len], [1], seed=kv_len, rtol=5e-3 if kv_len >= 1000 else 2.0 ** -7)


def test_ragged_batch_shuffled_pages_page256():
    # kv_len 5 averages only a handful of unit-variance rows, so |out| reaches ~2 where one bf16 ulp (2^-7 relative)
    # exceeds the reference's 5e-3: allow exactly one ulp there
    run_case(128, 256, [700, 5, 2049], [1, 3, 2], seed=3, shuffle_pages=True, rtol=2.0 ** -7)


@pytest.mark.parametrize("Hq,page,kv_lens,q_lens,max_splits", [
    (64, 64, [1, 63, 64, 65, 128, 129, 500, 31, 32, 33] * 2, [1] * 20, 64),   # ends of 64-token steps and of their halves
    (128, 96, [700, 5, 97, 96, 2049] + [40] * 12, [3, 1, 5, 2, 2] + [1] * 12, 64),   # several query tokens a request, pages of 3 tiles
    (64, 32, [6000] + [1] * 17, [1] * 18, 64),       # one request holds almost all: its splits are capped, its merge takes several rounds
    (64, 32, [3000] + [70] * 19, [1] * 20, 256),
    (128, 64, [300] * 17, [1] * 17, 2),
    (64, 64, [200] * 17, [1] * 17, 1),               # one split: normalised in place
])
def test_batches_that_share_the_workgroups(Hq, page, kv_lens, q_lens, max_splits):
    run_case(Hq, page, kv_lens, q_lens, seed=len(kv_lens), shuffle_pages=True, max_splits=max_splits, rtol=2.0 ** -7)


def test_shared_workgroups_with_append_and_fewer_live_requests():
    """18 requests of which 17 are live, the newest token of each taken from the append buffers: the live rows equal the oracle's on the
    appended cache, which ends up updated; the dead request's pages stay as they were."""
    from ktransformers_amd._native import MLAWrapper
    g = torch.Generator().manual_seed(19)
    Hq, page, B, live = 64, 64, 18, 17
    kv_lens = [130, 64, 1, 65, 128, 700] * 3
    pages_per = [(n + page - 1) // page for n in kv_lens]
    kv_buf = torch.randn((sum(pages_per) + 1, page, 576), generator=g).to(torch.bfloat16)
    q_nope, q_pe = (torch.randn((B, Hq, d), generator=g).to(torch.bfloat16) for d in (512, 64))
    new_ckv, new_kpe = (torch.randn((B, d), generator=g).to(torch.bfloat16) for d in (512, 64))
    kv_indices = torch.randperm(sum(pages_per), generator=g).to(torch.int32)
    kv_indptr = torch.tensor([0] + list(np.cumsum(pages_per)), dtype=torch.int32)
    qo_indptr, kv_len_arr = torch.arange(B + 1, dtype=torch.int32), torch.tensor(kv_lens, dtype=torch.int32)
    want = kv_buf.clone()
    for b in range(live):
        pos = kv_lens[b] - 1
        want[int(kv_indices[int(kv_indptr[b]) + pos // page]), pos % page] = torch.cat([new_ckv[b], new_kpe[b]])
    ref, _ = mla_paged_ref(q_nope, q_pe, want, qo_indptr, kv_indptr, kv_indices, kv_len_arr, 192 ** -0.5)
    w = MLAWrapper(B, kv_buf.shape[0], device=DEV, max_q_tokens=B)
    kvd = kv_buf.to(DEV)
    ckv, k_pe = torch.split(kvd, [512, 64], dim=-1)
    w.plan(qo_indptr.to(DEV), kv_indptr.to(DEV), kv_indices.to(DEV), kv_len_arr.to(DEV),
           torch.tensor([live], dtype=torch.int32, device=DEV), Hq, 512, 64, page, 192 ** -0.5)
    out = w.run(q_nope.to(DEV), q_pe.to(DEV), ckv, k_pe, new_ckv=new_ckv.to(DEV), new_kpe=new_kpe.to(DEV))
    torch.cuda.synchronize()
    # kv_len 1: one bf16 ulp (2^-7) of an |out| past 1 exceeds 5e-3
    torch.testing.assert_close(out[:live].float().cpu(), ref[:live].to(torch.bfloat16).float(), rtol=2.0 ** -7, atol=5e-3)
    assert torch.equal(kvd.cpu(), want)


def decode_batch(Hq, lens, page=64, seed=7):
    """A wrapper planned (with the longest context as its hint) for one token of each request, its run(), and the 64-bit result."""
    from ktransformers_amd._native import MLAWrapper
    g = torch.Generator(device=DEV).manual_seed(seed)
    B, pages = len(lens), [(n + page - 1) // page for n in lens]
    first = [0] + list(np.cumsum(pages))
    table = torch.randperm(first[-1], device=DEV, generator=g).to(torch.int32)
    cache, q_nope, q_pe = (torch.randn(s, device=DEV, generator=g).to(torch.bfloat16) for s in ((first[-1], page, 576), (B, Hq, 512), (B, Hq, 64)))
    w = MLAWrapper(B, first[-1], use_cuda_graph=False, device=DEV, max_q_tokens=B)
    dev = [torch.tensor(a, dtype=torch.int32, device=DEV) for a in (range(B + 1), first, lens, [B])]
    w.plan(dev[0], dev[1], table, dev[2], dev[3], Hq, 512, 64, page, 192 ** -0.5, max_kv_len=max(lens))

    def exact():
        out = []
        for b, n in enumerate(lens):
            rows = cache[table[first[b]:first[b + 1]].long()].view(-1, 576)[:n].double()
            out.append(torch.softmax(torch.cat((q_nope[b], q_pe[b]), dim=1).double() @ rows.T * 192 ** -0.5, dim=1) @ rows[:, :512])
        return torch.stack(out)
    return (lambda: w.run(q_nope, q_pe, cache[:, :, :512], cache[:, :, 512:])), exact


@pytest.mark.parametrize("Hq,lens", [(64, [1000] * 20), (128, [500] * 17 + [130, 64, 1]), (128, [8192, 2100, 5000, 8192, 8000, 7000, 6000, 64]), (64, [64, 33] * 10),
                                     (128, [400] * 31 + [9000]), (128, [100] * 19 + [8000]), (128, [300] * 32)])     # the merge's 4 and 8 split lanes: a token of several rounds; of none
def test_wide_decode_is_off_by_the_rounding_of_its_outputs(Hq, lens):
    """mla_decode_wide_kernel multiplies P as two bf16 (2^-17 of it is lost) and adds in fp32: against 64-bit sums the result is off by what rounding
    the exact result to bf16 is off by, to 1 %."""
    run, exact = decode_batch(Hq, lens)
    want = exact()
    floor = float((want.to(torch.bfloat16).double() - want).norm())
    assert float((run().double() - want).norm()) <= 1.01 * floor


@pytest.mark.parametrize("Hq,lens,ramp", [(128, [32, 33, 64, 65, 96, 97, 128, 129, 160, 161, 31, 1, 512, 700, 1024, 3] * 2, 0.0),   # 1 to 5 tiles a workgroup and more, whole and not
                                          (64, [9000] * 60 + [1, 40, 8999, 9000], 0.0),                                          # more than 64 tiles: the page table again
                                          (128, [2000] * 8 + [4000] * 12, 2.5), (128, [2000] * 8 + [4000] * 12, -2.5),            # scores that grow a tile by less than what rescales the sums ...
                                          (64, [4000] * 20, 7.0), (64, [4000] * 20, 0.4)])                                        # ... by more, and by little for long
def test_wide_decode_tiles_and_growing_scores(Hq, lens, ramp):
    """mla_decode_wide_kernel at the edges of its tiles, and where a head's largest score moves on in every tile of 32 (by `ramp`): off by the rounding of its outputs.  One dim,
    which the scores have no part of, holds 2e36: probabilities past 1 would take its sums out of fp32."""
    from ktransformers_amd import _native as n
    g = torch.Generator(device=DEV).manual_seed(11)
    B, page, pages = len(lens), 64, [(m + 63) // 64 for m in lens]
    first = [0] + [int(v) for v in np.cumsum(pages)]
    table = torch.randperm(first[-1], device=DEV, generator=g).to(torch.int32)
    cache, q_nope, q_pe = (torch.randn(s, device=DEV, generator=g).to(torch.bfloat16) for s in ((first[-1], page, 576), (B, Hq, 512), (B, Hq, 64)))
    scale = 192 ** -0.5
    q_nope[..., 7], cache[..., 7] = 0, 2e36
    if ramp:   # the last rotated dim, which O has no part of: q 16 there, a token's key its tile's share
        q_pe[..., -1] = 16
        for b in range(B):
            at = (torch.arange(pages[b] * 64, device=DEV) // 32 % 64).float() * (ramp / 16 / scale)
            cache[table[first[b]:first[b + 1]].long(), :, -1] = at.view(-1, 64).to(torch.bfloat16)
    w = n.MLAWrapper(B, first[-1], use_cuda_graph=False, device=DEV, max_q_tokens=B)
    dev = [torch.tensor(a, dtype=torch.int32, device=DEV) for a in (range(B + 1), first, lens, [B])]
    w.plan(dev[0], dev[1], table, dev[2], dev[3], Hq, 512, 64, page, scale, max_kv_len=max(lens))
    n.timing_enable(2)
    try:
        out = w.run(q_nope, q_pe, cache[:, :, :512], cache[:, :, 512:])
        assert any("mla_decode_wide_kernel" in t[0] for t in n.timing_collect())
    finally:
        n.timing_enable(0)
    want = []
    for b, m in enumerate(lens):
        rows = cache[table[first[b]:first[b + 1]].long()].view(-1, 576)[:m].double()
        want.append(torch.softmax(torch.cat((q_nope[b], q_pe[b]), dim=1).double() @ rows.T * scale, dim=1) @ rows[:, :512])
    want = torch.stack(want)
    assert bool(((out[..., 7].double() - want[..., 7]).abs() <= 2.0 ** -8 * 1.01 * want[..., 7]).all())
    out, want = (torch.cat((t[..., :7], t[..., 8:]), dim=-1) for t in (out, want))
    floor = float((want.to(torch.bfloat16).double() - want).norm())
    assert float((out.double() - want).norm()) <= 1.01 * floor


@pytest.mark.parametrize("page", [64, 96, 256])   # 96: no power of two, so that a tile's page is divided out
def test_wide_decode_appends_in_long_contexts(page):
    """The appended row's tile comes by its own requests (request_any) into the run of tiles that a workgroup already has in flight: contexts of dozens of tiles a workgroup, lengths that are
    whole tiles, so that only the new row makes the difference, and others.  Results, and the cache afterwards."""
    from ktransformers_amd import _native as n
    lens = [4000, 4032, 3072, 2560, 3999, 4001, 96, 2049, 33, 3584, 1, 4000]
    g = torch.Generator(device=DEV).manual_seed(page)
    B, Hq, pages = len(lens), 128, [(m + page - 1) // page for m in lens]
    first = [0] + [int(v) for v in np.cumsum(pages)]
    table = torch.randperm(first[-1], device=DEV, generator=g).to(torch.int32)
    cache, q_nope, q_pe, new = (torch.randn(s, device=DEV, generator=g).to(torch.bfloat16) for s in ((first[-1], page, 576), (B, Hq, 512), (B, Hq, 64), (B, 576)))
    new *= 3   # (a stale row's score and values are others by much)
    after = cache.clone()
    for b, m in enumerate(lens):
        after[int(table[first[b] + (m - 1) // page]), (m - 1) % page] = new[b]
    w = n.MLAWrapper(B, first[-1], use_cuda_graph=False, device=DEV, max_q_tokens=B)
    dev = [torch.tensor(a, dtype=torch.int32, device=DEV) for a in (range(B + 1), first, lens, [B])]
    w.plan(dev[0], dev[1], table, dev[2], dev[3], Hq, 512, 64, page, 192 ** -0.5, max_kv_len=max(lens))
    n.timing_enable(2)
    try:
        out = w.run(q_nope, q_pe, cache[:, :, :512], cache[:, :, 512:], new_ckv=new[:, :512].contiguous(), new_kpe=new[:, 512:].contiguous())
        assert "mla_decode_wide_kernel" in n.timing_collect()[0][0]
    finally:
        n.timing_enable(0)
    assert torch.equal(cache, after)
    want = []
    for b, m in enumerate(lens):
        rows = after[table[first[b]:first[b + 1]].long()].view(-1, 576)[:m].double()
        want.append(torch.softmax(torch.cat((q_nope[b], q_pe[b]), dim=1).double() @ rows.T * 192 ** -0.5, dim=1) @ rows[:, :512])
    want = torch.stack(want)
    floor = (want.to(torch.bfloat16).double() - want).norm(dim=(1, 2))
    err = (out.double() - want).norm(dim=(1, 2))
    assert bool((err <= 1.02 * floor).all()), (err / floor).tolist()   # (the outputs' rounding, each request by itself; of one token the result is the row)


@pytest.mark.parametrize("lens", [[2000] * 20, [40] * 24])   # several splits a request; one, whose result the kernel stores itself
def test_wide_decode_of_infinite_scores(lens):
    """Scores of -inf weigh nothing, wherever a split begins: every even tile of 32 tokens is -inf to every third head."""
    from ktransformers_amd import _native as n
    g = torch.Generator(device=DEV).manual_seed(5)
    B, Hq, page, m = len(lens), 128, 64, lens[0]
    pages = (m + 63) // 64
    cache, q_nope, q_pe = (torch.randn(s, device=DEV, generator=g).to(torch.bfloat16) for s in ((B * pages, page, 576), (B, Hq, 512), (B, Hq, 64)))
    q_pe[..., -1] = 0
    q_pe[:, ::3, -1] = 3e38
    cache[..., -1] = torch.where(torch.arange(64, device=DEV) < 32, -4.0, 0.0).to(torch.bfloat16)
    w = n.MLAWrapper(B, B * pages, use_cuda_graph=False, device=DEV, max_q_tokens=B)
    dev = [torch.tensor(a, dtype=torch.int32, device=DEV) for a in (range(B + 1), range(0, B * pages + 1, pages), lens, [B])]
    w.plan(dev[0], dev[1], None, dev[2], dev[3], Hq, 512, 64, page, 192 ** -0.5, max_kv_len=m, identity_pages=True)
    n.timing_enable(2)
    try:
        out = w.run(q_nope, q_pe, cache[:, :, :512], cache[:, :, 512:])
        assert "mla_decode_wide_kernel" in n.timing_collect()[0][0]
    finally:
        n.timing_enable(0)
    rows = cache.view(B, pages * 64, 576)[:, :m].double()
    want = torch.matmul(torch.softmax(torch.matmul(torch.cat((q_nope, q_pe), dim=2).double(), rows.transpose(1, 2).contiguous()) * 192 ** -0.5, dim=2), rows[..., :512].contiguous())
    floor = float((want.to(torch.bfloat16).double() - want).norm())
    assert float((out.double() - want).norm()) <= 1.01 * floor


@pytest.mark.parametrize("Hq,lens,wide", [(64, [600] * 20, False), (64, [300] * 24, False), (128, [200] * 16, False), (64, [16384] * 2, False), (128, [2000] * 8, False),
                                          (64, [50] * 20, True), (64, [1000] * 20, True), (128, [1000] * 12, True), (128, [8192] * 8, True), (64, [8192] * 3, True)])
def test_which_decode_kernel_a_batch_takes(Hq, lens, wide):
    """The 64-token kernel where it was measured faster (mla_wide_steps): whole second rounds of the other one's workgroups, deep splits, one step; not
    for short contexts in one round.  Both within the bound of the outputs' rounding and P's."""
    from ktransformers_amd import _native as n
    run, exact = decode_batch(Hq, lens)
    n.timing_enable(2)
    try:
        out = run()
        labels = [t[0] for t in n.timing_collect()]
    finally:
        n.timing_enable(0)
    assert any("mla_decode_wide_kernel" in t for t in labels) == wide, labels
    want = exact()
    assert float((out.double() - want).norm() / want.norm()) < 2.4e-3      # (sqrt(2) of 1.66e-3: outputs and probabilities in bf16)


@pytest.mark.parametrize("Hq,lens,kernel", [(128, [3000] * 4, "mla_decode_kernel<2,4>"), (128, [400] * 5, "mla_decode_kernel<2,4>"), (128, [2000, 500, 777, 1999, 1], "mla_decode_kernel<2,4>"),
                                            (128, [1000] * 6, "mla_decode_kernel<2,4>"), (128, [3000, 900, 2100, 2999, 1500, 800], "mla_decode_kernel<2,4>"), (128, [3584] * 7, "mla_decode_kernel<2,4>"),
                                            (128, [3585] * 7, "mla_decode_wide_kernel"), (128, [4500] * 5, "mla_decode_wide_kernel"), (192, [3000] * 5, "mla_decode_wide_kernel"), (128, [6000, 33, 1500, 6000, 64, 4000, 31], "mla_decode_wide_kernel"),
                                            (64, [7000] * 7, "mla_decode_kernel<2,4>"), (64, [4200] * 8, "mla_decode_wide_kernel"), (64, [3000] * 8, "mla_decode_kernel<4,2>")])
def test_which_decode_kernel_a_few_requests_take(Hq, lens, kernel):
    """5 to 7 requests of 128 heads and more leave the 2x4 shape from splits of 8 tiles on, for the kernel that shares out what they hold; the 64-head kernel from there on at 64 heads too."""
    from ktransformers_amd import _native as n
    run, exact = decode_batch(Hq, lens)
    n.timing_enable(2)
    try:
        out = run()
        labels = [t[0] for t in n.timing_collect()]
    finally:
        n.timing_enable(0)
    assert labels[0].startswith(kernel), labels
    want = exact()
    assert float((out.double() - want).norm() / want.norm()) < 2.4e-3      # (sqrt(2) of 1.66e-3: outputs and probabilities in bf16)


@pytest.mark.parametrize("bytes_of_splits,max_splits,partials", [(31, 256, False), (256, 16, False), (256, 256, True)])
def test_few_requests_without_room_for_shares(bytes_of_splits, max_splits, partials):
    """5 requests of long contexts whose workspace, split limit or way of merging leaves no shares of the batch: the 2x4 shape, as for short ones."""
    from ktransformers_amd import _native as n
    lens, Hq = [4500] * 5, 128
    g = torch.Generator(device=DEV).manual_seed(3)
    q_nope, q_pe, cache = (torch.randn(s, device=DEV, generator=g).to(torch.bfloat16) for s in ((5, Hq, 512), (5, Hq, 64), (71, 64, 576)))
    w = n.MLAWrapper(5, 71 * 5, use_cuda_graph=False, device=DEV, max_q_tokens=5, max_splits=max_splits)
    dev = [torch.tensor(a, dtype=torch.int32, device=DEV) for a in (range(6), range(0, 71 * 6, 71), list(range(71)) * 5, lens, [5])]
    w.plan(*dev, Hq, 512, 64, 64, 192 ** -0.5, max_kv_len=4500)
    if bytes_of_splits < 256:
        w.workspace = w.workspace[:bytes_of_splits * 5 * Hq * 514 * 4 + 20]
    n.timing_enable(2)
    try:
        out = w.run(q_nope, q_pe, cache[:, :, :512], cache[:, :, 512:], partials=partials)
        assert n.timing_collect()[0][0].startswith("mla_decode_kernel<2,4>")
    finally:
        n.timing_enable(0)
    if not partials:
        rows = cache.view(-1, 576)[:4500].double()
        want = torch.softmax(torch.cat((q_nope, q_pe), dim=2).double().view(-1, 576) @ rows.T.contiguous() * 192 ** -0.5, dim=1) @ rows[:, :512].contiguous()
        assert float((out.double().view(-1, 512) - want).norm() / want.norm()) < 2.4e-3      # (sqrt(2) of 1.66e-3: outputs and probabilities in bf16)


def test_single_split_equals_many():
    run_case(16, 64, [3000], [1], seed=4, max_splits=1)


def test_cache_append():
    from ktransformers_amd._native import mla_cache_append
    g = torch.Generator().manual_seed(0)
    cache = torch.zeros((8, 64, 1, 576), dtype=torch.bfloat16, device=DEV)
    T = 5
    ckv = torch.randn((T, 512), generator=g).to(torch.bfloat16).to(DEV)
    kpe = torch.randn((T, 64), generator=g).to(torch.bfloat16).to(DEV)
    pos = torch.tensor([0, 63, 64, 200, 511])
    mla_cache_append(cache, ckv, kpe, (pos // 64).to(DEV), (pos % 64).to(DEV))
    torch.cuda.synchronize()
    want = torch.zeros_like(cache)
    want[pos // 64, pos % 64, 0, :512] = ckv          # StaticCache.update (custom_cache.py:189-195)
    want[pos // 64, pos % 64, 0, 512:] = kpe
    assert torch.equal(cache, want)


def test_decode_with_fused_cache_append():
    """run(new_ckv, new_kpe) == cache_append followed by run, and the cache ends up updated."""
    from ktransformers_amd._native import MLAWrapper
    g = torch.Generator().manual_seed(9)
    Hq, page, B = 16, 64, 3
    kv_lens = [130, 64, 1]                               # position kv_len-1 is the token being appended
    pages_per = [(n + page - 1) // page for n in kv_lens]
    kv_buf = torch.randn((sum(pages_per) + 1, page, 576), generator=g).to(torch.bfloat16)
    q_nope = torch.randn((B, Hq, 512), generator=g).to(torch.bfloat16)
    q_pe = torch.randn((B, Hq, 64), generator=g).to(torch.bfloat16)
    new_ckv = torch.randn((B, 512), generator=g).to(torch.bfloat16)
    new_kpe = torch.randn((B, 64), generator=g).to(torch.bfloat16)
    kv_indices = torch.arange(sum(pages_per), dtype=torch.int32)
    kv_indptr = torch.tensor([0] + list(np.cumsum(pages_per)), dtype=torch.int32)
    qo_indptr = torch.arange(B + 1, dtype=torch.int32)
    kv_len_arr = torch.tensor(kv_lens, dtype=torch.int32)
    ref_buf = kv_buf.clone()
    for b in range(B):
        pos = kv_lens[b] - 1
        pg = int(kv_indices[int(kv_indptr[b]) + pos // page])
        ref_buf[pg, pos % page, :512] = new_ckv[b]
        ref_buf[pg, pos % page, 512:] = new_kpe[b]
    ref, _ = mla_paged_ref(q_nope, q_pe, ref_buf, qo_indptr, kv_indptr, kv_indices, kv_len_arr, 192 ** -0.5)
    w = MLAWrapper(B, kv_buf.shape[0], device=DEV, max_q_tokens=B)
    kvd = kv_buf.to(DEV)
    ckv, k_pe = torch.split(kvd, [512, 64], dim=-1)
    w.plan(qo_indptr.to(DEV), kv_indptr.to(DEV), kv_indices.to(DEV), kv_len_arr.to(DEV),
           torch.tensor([B], dtype=torch.int32, device=DEV), Hq, 512, 64, page, 192 ** -0.5)
    out = w.run(q_nope.to(DEV), q_pe.to(DEV), ckv, k_pe, new_ckv=new_ckv.to(DEV), new_kpe=new_kpe.to(DEV))
    torch.cuda.synchronize()
    torch.testing.assert_close(out.float().cpu(), ref.to(torch.bfloat16).float(), rtol=2.0 ** -7, atol=5e-3)
    assert torch.equal(kvd.cpu(), ref_buf), "the kernel must leave the appended rows in the cache"


def test_decode_at_128k_context():
    """128K-token paged latent cache (151 MB per layer), V3 head count.  The oracle's per-head
    K replication would need 19 GB here, so the same math (scores = q . lat^T, fp32 softmax, P . ckv) is evaluated as two
    plain fp32 matmuls over the latent rows."""
    from ktransformers_amd._native import MLAWrapper
    g = torch.Generator().manual_seed(9)
    Hq, page, n = 128, 64, 131072 - 17
    pages = (n + page - 1) // page
    kv = (torch.randn((pages, page, 576), generator=g)).to(torch.bfloat16)
    qn = torch.randn((1, Hq, 512), generator=g).to(torch.bfloat16)
    qp = torch.randn((1, Hq, 64), generator=g).to(torch.bfloat16)
    sm = 192 ** -0.5
    lat = kv.reshape(-1, 576)[:n].float()
    logits = (torch.cat([qn, qp], -1)[0].float() @ lat.T) * sm
    ref = torch.softmax(logits, -1) @ lat[:, :512]
    w = MLAWrapper(1, pages, device=DEV, max_q_tokens=1, max_splits=1024)
    kvd = kv.to(DEV)
    ckv, k_pe = torch.split(kvd, [512, 64], dim=-1)
    w.plan(None, None, None, torch.tensor([n], dtype=torch.int32, device=DEV), None, Hq, 512, 64, page, sm, max_kv_len=n)
    out = w.run(qn.to(DEV), qp.to(DEV), ckv, k_pe)
    torch.testing.assert_close(out[0].float().cpu(), ref.to(torch.bfloat16).float(), rtol=5e-3, atol=5e-3)


# ---- non-absorbed prompt attention (ktx_mla_prefill) ----------------------------------------------------------------------
@pytest.mark.parametrize("H,T,kv_len", [(4, 130, 130), (3, 70, 201), (16, 128, 128), (2, 257, 1000), (128, 64, 64)])
def test_prefill_expanded_against_fp32_attention(H, T, kv_len):
    """Causal softmax(q k^T) v over qk 192 (128 nope + 64 shared rope) / v 128 in fp32 on the same bf16 operands; the queries are
    the last T keys; the padded key rows are zero as the operator makes them."""
    from ktransformers_amd._native import mla_prefill
    g = torch.Generator().manual_seed(H * 1000 + T + kv_len)
    kv_pad = (kv_len + 63) // 64 * 64
    q = torch.randn((T, H, 192), generator=g).to(torch.bfloat16).to(DEV)
    k_nope = torch.zeros((H, kv_pad, 128), dtype=torch.bfloat16, device=DEV)
    k_nope[:, :kv_len] = torch.randn((H, kv_len, 128), generator=g).to(torch.bfloat16).to(DEV)
    cache = torch.randn((kv_len + 5, 576), generator=g).to(torch.bfloat16).to(DEV)      # k_pe lives in the latent cache rows
    cache[kv_len:] = float("nan")                                                        # rows past the context are never used
    v = torch.zeros((H, kv_pad, 128), dtype=torch.bfloat16, device=DEV)
    v[:, :kv_len] = torch.randn((H, kv_len, 128), generator=g).to(torch.bfloat16).to(DEV)
    sm_scale = 192 ** -0.5
    q_pe = q[:, :, 128:].contiguous()
    out = mla_prefill(q[:, :, :128], q_pe, k_nope, cache[:, 512:], v.transpose(1, 2).contiguous(), kv_len, sm_scale)
    k = torch.cat([k_nope[:, :kv_len].float(), cache[:kv_len, 512:].float()[None].expand(H, -1, -1)], dim=-1)    # [H, kv, 192]
    s = torch.einsum("thd,hkd->htk", q.float(), k) * sm_scale
    pos = torch.arange(T, device=DEV)[:, None] + (kv_len - T)
    s = s.masked_fill(torch.arange(kv_len, device=DEV)[None, :] > pos, float("-inf"))
    ref = torch.einsum("htk,hkd->thd", torch.softmax(s, dim=-1), v[:, :kv_len].float())
    torch.testing.assert_close(out.float(), ref.to(torch.bfloat16).float(), rtol=2.0 ** -7, atol=5e-3)


@pytest.mark.parametrize("offset", [0, 4, 1])   # elements: operands on 16 bytes come by LDS-DMA, others through registers
@pytest.mark.parametrize("H,T,kv_len", [(1, 1, 1), (2, 1, 64), (2, 1, 65), (3, 129, 128 + 129), (8, 33, 320), (2, 256, 4160), (130, 130, 321)])   # the last: more workgroups than CUs
def test_prefill_tiles_of_keys(H, T, kv_len, offset):
    """One key tile, two, odd and even counts of them, against attention in 64 bits, at the bound of its roundings (test_mla_prefill_bound.py: which shows a missing tile)."""
    from ktransformers_amd._native import mla_prefill
    q, k_nope, cache, v = prefill_operands(H, T, kv_len)

    def at_offset(x):
        flat = torch.empty(x.numel() + offset, dtype=torch.bfloat16, device=DEV)
        flat[offset:] = x.reshape(-1).to(DEV)
        return flat[offset:].view(x.shape)

    qd = q.to(DEV)
    out = mla_prefill(qd[:, :, :128], qd[:, :, 128:], at_offset(k_nope), at_offset(cache)[:, 512:], at_offset(v.transpose(1, 2).contiguous()), kv_len, 192 ** -0.5)
    ref, bound = prefill_statement(prefill_scores(q, k_nope, cache, kv_len), v[:, :kv_len].double())
    err = (out.cpu().double() - ref).abs()
    assert bool((err <= bound).all()), f"{int((err > bound).sum())} outputs, up to {float((err / bound).max()):.2f} of the bound"


@pytest.mark.parametrize("nsplit", [0, 2, 3, 5, 16])   # 0: the library's own choice
@pytest.mark.parametrize("H,T,kv_len", [(1, 1, 65), (3, 129, 129), (8, 200, 200), (16, 1, 1030), (8, 130, 321), (3, 300, 700), (16, 64, 4160)])
def test_prefill_keys_shared_by_workgroups(H, T, kv_len, nsplit):
    """A query's keys in pieces (ktx_mla_prefill_ws): fewer tiles than pieces, queries that see none of a piece's keys, heads of no eight, one, two and more tiles a piece, against
    attention in 64 bits at the bound of the roundings (the pieces' sums and weights are in 32 bits); without scratch the call is the unshared one's."""
    from ktransformers_amd import _native as n
    q, k_nope, cache, v = prefill_operands(H, T, kv_len)
    k_nope[:, : kv_len // 2] *= 4   # (the largest scores lie in some pieces)
    qd, args = q.to(DEV), (k_nope.to(DEV), cache.to(DEV)[:, 512:], v.transpose(1, 2).contiguous().to(DEV), kv_len, 192 ** -0.5)
    whole = None
    try:
        n.lib.ktx_debug_set(33, 1)
        whole = n.mla_prefill(qd[:, :, :128], qd[:, :, 128:], *args)
        n.lib.ktx_debug_set(33, nsplit)
        need = n.lib.ktx_mla_prefill_workspace_bytes(T, H, kv_len)
        out = n.mla_prefill(qd[:, :, :128], qd[:, :, 128:], *args)
        again = torch.full_like(out, float("nan"))
        k, kp, vt, kv, scale = args
        n.check(n.lib.ktx_mla_prefill_ws(T, H, kv, k.shape[1], scale, qd.data_ptr(), qd.stride(0), qd.stride(1), qd.data_ptr() + 256, qd.stride(0), qd.stride(1), k.data_ptr(), kp.data_ptr(),
                                         kp.stride(0), vt.data_ptr(), again.data_ptr(), torch.empty(max(need, 1), dtype=torch.uint8, device=DEV).data_ptr(), max(need, 1) - 1,
                                         torch.cuda.current_stream().cuda_stream))
    finally:
        n.lib.ktx_debug_set(33, 0)
    assert torch.equal(again, whole if need else out)
    if nsplit or kv_len <= 200 or kv_len >= 1030:   # (the library's choice: one tile or a few are not worth it, many of few pairs are)
        assert (need > 0) == (nsplit > 1 or (not nsplit and kv_len >= 1030))
    ref, bound = prefill_statement(prefill_scores(q, k_nope, cache, kv_len), v[:, :kv_len].double())
    for got in (whole, out):
        err = (got.cpu().double() - ref).abs()
        assert bool((err <= bound).all()), f"{int((err > bound).sum())} outputs, up to {float((err / bound).max()):.2f} of the bound"


@pytest.mark.parametrize("nsplit", [2, 3, 5, 16])
@pytest.mark.parametrize("what", ["scores", "values", "nan"])
def test_prefill_infinities_shared_or_not(what, nsplit):
    """Infinities and NaN come out of a shared query as out of an unshared one: a query whose visible scores are all -inf (head 0), whose first tile's are (head 1), a later run of
    tiles (head 2); an infinite value, which queries before it multiply with 0; a NaN in a key."""
    from ktransformers_amd import _native as n
    H, T, kv_len = 3, 130, 1030
    q, k_nope, cache, v = prefill_operands(H, T, kv_len)
    q[:, :, 0] = 0
    s = prefill_scores(q, k_nope, cache, kv_len)
    ref, bound = prefill_statement(s, v[:, :kv_len].double())
    if what == "scores":
        q[[7, 100], :, 0] = 3e38
        k_nope[:, :, 0] = 0
        for h, keys in enumerate((slice(None), slice(0, 64), slice(192, 384))):
            k_nope[h, keys, 0] = -4
            s[h, [7, 100], keys] = float("-inf")
        ref, bound = prefill_statement(s, v[:, :kv_len].double())
    elif what == "values":
        v[:, 950, 5], v[:, 64, 9], v[:, 1029, 11] = float("inf"), float("-inf"), float("inf")
    else:
        k_nope[1, 970, 3], v[2, 20, 2] = float("nan"), float("nan")
    qd, args = q.to(DEV), (k_nope.to(DEV), cache.to(DEV)[:, 512:], v.transpose(1, 2).contiguous().to(DEV), kv_len, 192 ** -0.5)
    try:
        n.lib.ktx_debug_set(33, 1)
        whole = n.mla_prefill(qd[:, :, :128], qd[:, :, 128:], *args).cpu().double()
        n.lib.ktx_debug_set(33, nsplit)
        shared = n.mla_prefill(qd[:, :, :128], qd[:, :, 128:], *args).cpu().double()
    finally:
        n.lib.ktx_debug_set(33, 0)
    finite = torch.isfinite(whole)
    assert bool((~finite).any()) and bool(finite.any())
    if what == "scores":
        assert bool(torch.isnan(whole[[7, 100], 0]).all()) and bool(finite[:, 2].all())
    assert torch.equal(torch.isnan(whole), torch.isnan(shared)) and torch.equal(whole[torch.isinf(whole)], shared[torch.isinf(whole)])
    for got in (whole, shared):
        assert bool(((got - ref).abs() <= bound)[finite].all())


@pytest.mark.parametrize("Hq,kv_len,T", [(128, 4023, 1), (64, 700, 1), (128, 33, 1), (64, 5000, 3)])
def test_merge_riding_the_unabsorb_launch(Hq, kv_len, T):
    """ktx_mla_decode_partials + ktx_linear_forward_batched_merge (the KV-split merge inside the launch of the per-head un-absorb
    products) against run() followed by forward_batched: the merged row is rounded to bf16 at the same point; only the fp32
    order of the split sum differs (8 split lanes instead of 16)."""
    from ktransformers_amd import _native as n
    g = torch.Generator().manual_seed(Hq + kv_len)
    page = 64
    pages = (kv_len + page - 1) // page
    kv = torch.randn((pages, page, 576), generator=g).to(torch.bfloat16).to(DEV)
    qn = torch.randn((T, Hq, 512), generator=g).to(torch.bfloat16).to(DEV)
    qp = torch.randn((T, Hq, 64), generator=g).to(torch.bfloat16).to(DEV)
    wuv = (torch.randn((Hq, 128, 512), generator=g) / 16).to(torch.bfloat16).to(DEV)
    oabs = n.LinearHandle(512, 128, "BF16", 0, 8, DEV, batch=Hq)
    oabs.load_bf16(wuv)
    w = n.MLAWrapper(1, pages, device=DEV, max_q_tokens=T)
    ckv, k_pe = torch.split(kv, [512, 64], dim=-1)
    qo = torch.tensor([0, T], dtype=torch.int32, device=DEV)
    w.plan(qo, None, None, torch.tensor([kv_len], dtype=torch.int32, device=DEV), None, Hq, 512, 64, page, 192 ** -0.5,
           max_kv_len=kv_len)
    attn = w.run(qn, qp, ckv, k_pe)
    ref = oabs.forward_batched(attn)
    assert n.lib.ktx_linear_merge_eligible(oabs._h, T, 1, Hq)
    for rep in range(2):
        parts = w.run_partials(qn, qp, ckv, k_pe)
        got = n.merge_and_unabsorb(oabs, parts, T, Hq)
        torch.cuda.synchronize()
        a, b = got.float(), ref.float()
        assert torch.isfinite(a).all()
        assert float((a - b).norm() / b.norm()) < 2e-3
        assert float((a - b).abs().max()) <= 2e-2 * float(b.abs().max())
