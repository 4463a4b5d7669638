"""Top-k over short key sets (up to 4,096 keys, every key a candidate) read from score rows,
against the candidate-list path, which a forced threshold of -inf still takes: the same
entries in the same order, ties and masked keys included, for every dtype, head count and
kind of mask that the route takes.
"""
import pytest
import torch

from geoweave_amd.custom_indexer import sparse_topk_indexer as sti

pytestmark = pytest.mark.gpu


def _inputs(B, T, S, H, dtype, seed, ties=False):
    g = torch.Generator().manual_seed(seed)
    if ties:  # small integers: many equal scores
        q, k = (torch.randint(-1, 2, (B, n, H, 64), generator=g).to(dtype) for n in (T, S))
        w = torch.randint(-1, 3, (B, S, H), generator=g).to(dtype)
    else:
        q, k = (torch.randn(B, n, H, 64, generator=g).to(dtype) for n in (T, S))
        w = (1 + 0.5 * torch.randn(B, S, H, generator=g)).to(dtype)
    return [x.cuda() for x in (q, k, w)]


def _both(q, k, w, mask, topk, view=None):
    a = sti.indexer_topk_forward(q, k, w, mask, topk, 0.125, view_bias=view)
    b = sti.indexer_topk_forward(q, k, w, mask, topk, 0.125, flags=sti.FLAG_TAU_MINUS_INF, view_bias=view)
    torch.cuda.synchronize()
    return a, b


def _same(a, b):
    assert torch.equal(a[0], b[0])
    assert torch.equal(a[1].view(torch.int32 if a[1].dtype == torch.float32 else torch.int16),
                       b[1].view(torch.int32 if b[1].dtype == torch.float32 else torch.int16))


@pytest.mark.parametrize("ties", [False, True])
@pytest.mark.parametrize("S,topk", [(1, 1), (31, 9), (63, 63), (64, 10), (65, 64), (1536, 1024), (1537, 1024), (2748, 1024),
                                    (3072, 300), (3073, 3073), (4095, 1024), (4096, 1)])
def test_row_edges(gpu_device, S, topk, ties):
    print(f"[rows] S={S} topk={topk} ties={ties}", flush=True)
    q, k, w = _inputs(2, 37, S, 4, torch.bfloat16, S, ties)
    _same(*_both(q, k, w, None, topk))


@pytest.mark.parametrize("dtype,H", [(torch.bfloat16, 1), (torch.float16, 2), (torch.bfloat16, 8), (torch.float16, 4),
                                     (torch.float32, 1), (torch.float32, 2), (torch.float32, 4)])
@pytest.mark.parametrize("T", [1, 300])
def test_row_forms(gpu_device, dtype, H, T):
    print(f"[rows] {dtype} H={H} T={T}", flush=True)
    S = 1100
    for ties in (False, True):
        q, k, w = _inputs(1, T, S, H, dtype, 3 * H + T, ties)
        _same(*_both(q, k, w, None, 200))
        g = torch.Generator().manual_seed(T)
        mask = torch.randn(1, T, S, generator=g)
        mask[..., ::3] = float("-inf")  # 733 keys left
        mask[..., 1::9] = torch.finfo(dtype).min
        _same(*_both(q, k, w, mask.cuda(), 200))
        view = (torch.randint(0, 3, (1, T), generator=g).int().cuda(), torch.randint(0, 4, (1, S), generator=g).int().cuda(),
                torch.randn(1, 3, 4, generator=g).to(dtype).cuda())
        _same(*_both(q, k, w, None, 200, view))


def test_rows_with_too_few_finite_scores_and_nan(gpu_device):
    # The even rows have 50 unmasked keys for a top-k of 100: both paths send them to the exact
    # fallback. The odd rows are selected from, NaN scores among them (from gates and from the mask,
    # of both signs): a positive NaN ranks above every number, a negative one is not a candidate. Their
    # selection is the fallback's, to which the forced threshold of +inf sends every row.
    print("[rows] masked, NaN", flush=True)
    q, k, w = _inputs(1, 40, 700, 4, torch.bfloat16, 9)
    mask = torch.zeros(1, 40, 700)
    mask[:, ::2, 50:] = float("-inf")
    mask = mask.bfloat16().cuda()
    nan, minus = torch.tensor([0x7FC0, -0x40], dtype=torch.int16).view(torch.bfloat16).cuda()
    w[0, 300], w[0, 301] = nan, minus
    mask[:, :, 400], mask[:, :, 401] = nan, minus
    k[0, 5, 0, 0] = float("nan")
    a, b = _both(q, k, w, mask, 100)
    exact = sti.indexer_topk_forward(q, k, w, mask, 100, 0.125, flags=sti.FLAG_TAU_PLUS_INF)
    torch.cuda.synchronize()
    order = [x[0].sort(-1).values for x in (a, b, exact)]
    assert torch.equal(order[0], order[1]) and torch.equal(order[0][:, 1::2], order[2][:, 1::2])
    odd = order[0][:, 1::2]
    assert ((odd == 300).any(-1) & (odd == 400).any(-1)).all()
    assert not ((odd == 301) | (odd == 401)).any()
    # the scores, the two NaN entries aside, are the fallback's too (its fp32 dot products round
    # in another order: one bf16 rounding apart at most)
    top = [x[1].float()[:, 1::2].nan_to_num(nan=0.0).sort(-1).values for x in (a, exact)]
    assert ((top[0] - top[1]).abs() <= 2.0 ** -7 * top[1].abs()).all()
