"""Prompt attention over expanded keys stated in 64 bits, with the bound of the kernel's own roundings; and that the bound shows a key tile that is missing or stale."""
import pytest
import torch


def prefill_operands(H, T, kv_len):
    """bf16 queries [T][H][192], keys [H][kv_pad][128], cache rows [kv_len][576] (their last 64: the rotated part of the keys) and values [H][kv_pad][128]."""
    g = torch.Generator().manual_seed(H * 1000 + T + kv_len)
    kv_pad = (kv_len + 63) // 64 * 64
    q = torch.randn((T, H, 192), generator=g).to(torch.bfloat16)
    k_nope, v = torch.zeros((2, H, kv_pad, 128), dtype=torch.bfloat16)
    k_nope[:, :kv_len] = torch.randn((H, kv_len, 128), generator=g).to(torch.bfloat16)
    v[:, :kv_len] = torch.randn((H, kv_len, 128), generator=g).to(torch.bfloat16)
    cache = torch.randn((kv_len, 576), generator=g).to(torch.bfloat16)
    return q, k_nope, cache, v


def prefill_scores(q, k_nope, cache, kv_len):
    """Causal scores [H][T][kv_len] in 64 bits; the queries are the last T keys'."""
    T, H = q.shape[:2]
    k = torch.cat([k_nope[:, :kv_len].double(), cache[:, 512:].double()[None].expand(H, -1, -1)], dim=-1)
    s = torch.matmul(q.double().transpose(0, 1), k.transpose(1, 2)) * 192 ** -0.5
    return s.masked_fill(torch.arange(kv_len)[None, :] > torch.arange(T)[:, None] + (kv_len - T), float("-inf"))


def prefill_statement(s, v):
    """(outputs [T][H][128], bound of each): the probabilities enter the product as bf16, 2^-8 of each at most, the output is rounded to bf16, and exponents and sums in
    32 bits are far below (2^-14)."""
    p = torch.softmax(s, dim=-1)
    ref, size = torch.matmul(p, v), torch.matmul(p, v.abs())
    return ref.transpose(0, 1), ((2.0 ** -8 + 2.0 ** -14) * size + 2.0 ** -8 * ref.abs()).transpose(0, 1)


@pytest.mark.parametrize("fault", ["missing", "stale values", "stale keys"])
def test_the_bound_shows_a_wrong_key_tile(fault):
    """Each of 65 key tiles left out, with the tile's values or the tile's scores of the one two before it (the buffers' turn): outputs outside the bound."""
    H, T, kv_len = 2, 256, 4160
    q, k_nope, cache, v = prefill_operands(H, T, kv_len)
    s, v = prefill_scores(q, k_nope, cache, kv_len), v[:, :kv_len].double()
    ref, bound = prefill_statement(s, v)
    for t in range(2, kv_len // 64):
        at, old = slice(t * 64, t * 64 + 64), slice(t * 64 - 128, t * 64 - 64)
        s2, v2 = s.clone(), v.clone()
        if fault == "missing":
            s2[:, :, at] = float("-inf")
        elif fault == "stale values":
            v2[:, at] = v[:, old]
        else:
            s2[:, :, at] = torch.where(torch.isinf(s[:, :, at]), s[:, :, at], s[:, :, old])
        got = prefill_statement(s2, v2)[0]
        assert bool(((got - ref).abs() > bound).any()), t
