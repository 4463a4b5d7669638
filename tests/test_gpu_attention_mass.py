"""attn_sum and the fused KL row losses from the separate mass pass (gw_sparse_attn_mass) against
the oracle: sizes at the edges of its 512-query and 128-key tiles, several chunks of queries,
invalid and repeated positions, key rows that are not finite.

Tolerance: fp32 scores and weights on both sides, summed over heads: a weight's relative error is
that of its exponent, |s - lse| ulps of fp32 (2^-23 * 64 at most here) = 1e-5, and attn_sum <= H.
"""
import pytest
import torch

from geoweave_amd.custom_flash_attn import sparse_index_flash_attn as sifa
from geoweave_amd.custom_indexer.indexer_kl_fused import sparse_attention_kl_loss
from oracle import attention as oatt
from oracle import kl_loss as okl

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _mass_pass(monkeypatch):
    # the mass pass whatever the sizes (the rule sends small calls to the pass that stores the scores)
    monkeypatch.setattr(sifa, "_use_mass", lambda *a: True)


def _case(B, T, S, H, K, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(B, n, H, 64, generator=g).to(dtype) for n in (T, S, S))
    pos = torch.rand(B, T, S, generator=g).topk(K, dim=-1).indices.to(torch.int32)
    return q, k, v, pos


def _attn(q, k, v, pos, layout="bthd"):
    x = [t.cuda() if layout == "bthd" else t.cuda().transpose(1, 2).contiguous() for t in (q, k, v)]
    o, a, lse, _ = sifa._flash_attn_forward(*x, pos.cuda(), softmax_scale=0.125, return_attn=True, q_layout=layout)
    torch.cuda.synchronize()
    return a.cpu()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,T,S,H,K", [(1, 1, 1, 1, 1), (2, 33, 127, 3, 20), (1, 511, 128, 2, 64), (1, 513, 129, 16, 100),
                                       (2, 520, 700, 5, 257), (1, 70, 9000, 2, 1000)])
def test_mass_edges(gpu_device, B, T, S, H, K, dtype):
    print(f"[mass] B={B} T={T} S={S} H={H} K={K} {dtype}", flush=True)
    q, k, v, pos = _case(B, T, S, H, K, dtype, T + S)
    if K > 10:
        pos[:, ::4, K // 2:] = -1
        pos[:, min(T - 1, 7)] = S + 3
    _, ra, _ = oatt.sparse_attention(q.float(), k.float(), v.float(), pos, 0.125)
    for layout in ("bthd", "bhtd"):
        a = _attn(q, k, v, pos, layout)
        assert ((a - ra).abs() <= 1e-5 * ra + 1e-7).all()


def test_mass_in_chunks_with_kl(gpu_device):
    # 60,000 keys: the score matrix's 256 MiB hold 1,024 rows a chunk, so chunks of 1,024, 1,024 and 552.
    print("[mass] chunks, KL", flush=True)
    g = torch.Generator().manual_seed(3)
    B, T, S, H, K = 1, 2600, 60000, 2, 1000
    q, k, v = (torch.randn(B, n, H, 64, generator=g).bfloat16() for n in (T, S, S))
    off = torch.randint(0, S, (B, T, 1), generator=g)
    pos = ((off + torch.arange(K).view(1, 1, K) * 7919) % S).to(torch.int32)
    z = torch.randn(B, T, K, generator=g)
    o, a, loss = sparse_attention_kl_loss(q.cuda(), k.cuda(), v.cuda(), pos.cuda(), z.cuda(), 1e-6, 0.125)
    _, ra, _ = oatt.sparse_attention(q.float(), k.float(), v.float(), pos, 0.125)
    assert ((a.cpu() - ra).abs() <= 1e-5 * ra + 1e-7).all()
    assert abs(float(loss) - float(okl.kl_loss(ra, z, 1e-6))) <= 1e-5


def test_mass_of_repeated_positions_and_nonfinite_keys(gpu_device):
    print("[mass] repeated, non-finite", flush=True)
    q, k, v, pos = _case(2, 60, 300, 3, 40, torch.bfloat16, 17)
    pos[pos == 299] = 5
    pos[0, 20, 3] = pos[0, 20, 0]
    _, ra, _ = oatt.sparse_attention(q.float(), k.float(), v.float(), pos, 0.125)
    k[1, 299], v[1, 299] = float("nan"), float("inf")  # a row that no query selected
    a = _attn(q, k, v, pos)
    assert ((a - ra).abs() <= 1e-5 * ra + 1e-7).all()


@pytest.mark.parametrize("case", ["keys of -inf", "scores beyond fp32", "no valid key"])
def test_mass_of_heads_without_weight(gpu_device, case, monkeypatch):
    # Every selected score of a head is -inf: its lse is -inf, it adds nothing (the gather kernel's
    # result, bit for bit where no other head adds).
    print(f"[mass] {case}", flush=True)
    q, k, v, pos = _case(1, 70, 200, 3, 30, torch.bfloat16, 23)
    q = q.abs() + 1
    if case == "keys of -inf":
        k[:, :, 1] = -float("inf")
    elif case == "scores beyond fp32":
        q, k = q * 1e19, -(k.abs() + 1)
        k[:, :, 1] *= 3e19
        q[:, :, [0, 2]] *= 1e-19
    else:
        pos[:, ::2] = -1
    a = _attn(q, k, v, pos)
    monkeypatch.setattr(sifa, "FORWARD_PATH", "gather")
    g = _attn(q, k, v, pos)
    assert torch.isfinite(g).all() and torch.isfinite(a).all()
    assert ((a - g).abs() <= 1e-5 * g + 1e-7).all()


def test_mass_chunks_across_batch_elements(gpu_device):
    # Three groups of 512 queries an element and 60,000 keys: chunks of two groups, the second of them
    # with the last queries of element 0 and the first of element 1. Then six small elements in one.
    for B, T, S, K in ((3, 1100, 60000, 40), (6, 33, 200, 64)):
        print(f"[mass] {B} elements of {T} queries", flush=True)
        g = torch.Generator().manual_seed(S)
        q, k, v = (torch.randn(B, n, 2, 64, generator=g).bfloat16() for n in (T, S, S))
        pos = ((torch.randint(0, S, (B, T, 1), generator=g) + torch.arange(K).view(1, 1, K) * 7919) % S).to(torch.int32)
        z = torch.randn(B, T, K, generator=g)
        _, a, loss = sparse_attention_kl_loss(q.cuda(), k.cuda(), v.cuda(), pos.cuda(), z.cuda(), 1e-6, 0.125)
        _, ra, _ = oatt.sparse_attention(q.float(), k.float(), v.float(), pos, 0.125)
        assert ((a.cpu() - ra).abs() <= 1e-5 * ra + 1e-7).all()
        assert abs(float(loss) - float(okl.kl_loss(ra, z, 1e-6))) <= 1e-5
