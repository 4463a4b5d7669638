"""Top-k rows whose scores are NaN, of every sign and payload that counts: each row's selection is
top-k distinct keys, from the score rows (short key sets) and from the candidate lists alike."""
import pytest
import torch

from geoweave_amd.custom_indexer import sparse_topk_indexer as sti

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [0x7FC00000, 0x7FFFFFFF, -0x400000, -1])
@pytest.mark.parametrize("S,flags", [(700, 0), (700, sti.FLAG_TAU_MINUS_INF), (700, sti.FLAG_FORCE_WIDE), (5000, 0)])
@pytest.mark.parametrize("every", [1, 7])
def test_rows_of_nan_scores(gpu_device, every, S, flags, bits):
    print(f"[nan scores] bits={bits} S={S} flags={flags} every={every}", flush=True)
    g = torch.Generator().manual_seed(S)
    q, k = (torch.randn(1, n, 2, 64, generator=g).cuda() for n in (40, S))
    w = (1 + 0.5 * torch.rand(1, S, 2, generator=g)).cuda()
    mask = torch.zeros(1, 40, S, device="cuda")
    mask[:, ::2, ::every] = torch.tensor([bits], dtype=torch.int32).view(torch.float32).cuda()
    plain, plain_scores = sti.indexer_topk_forward(q, k, w, None, 100, 0.125)
    idx, scores = sti.indexer_topk_forward(q, k, w, mask, 100, 0.125, flags=flags)
    torch.cuda.synchronize()
    order = idx.sort(-1).values
    assert order.min() >= 0 and order.max() < S and (order.diff(dim=-1) > 0).all()
    # the rows without a NaN select as without the mask
    assert torch.equal(order[:, 1::2], plain.sort(-1).values[:, 1::2])
    assert torch.equal(scores.sort(-1).values[:, 1::2], plain_scores.sort(-1).values[:, 1::2])


def test_nan_gate_of_all_bits(gpu_device):
    # The pattern that stands for "no gate" inside the kernel, as a gate of the input: a NaN score
    # on every path, not a score of 0.
    print("[nan scores] gate of all bits", flush=True)
    g = torch.Generator().manual_seed(1)
    q, k = (torch.randn(1, n, 2, 64, generator=g).cuda() for n in (40, 700))
    w = -(1 + 0.5 * torch.rand(1, 700, 2, generator=g)).cuda()  # other scores are not above 0
    w[0, ::9] = torch.tensor([-1], dtype=torch.int32).view(torch.float32).cuda()
    rows = sti.indexer_topk_forward(q, k, w, None, 100, 0.125)
    lists = sti.indexer_topk_forward(q, k, w, None, 100, 0.125, flags=sti.FLAG_TAU_MINUS_INF)
    torch.cuda.synchronize()
    assert torch.equal(rows[0], lists[0])
    assert torch.equal(rows[1].view(torch.int32), lists[1].view(torch.int32))
    assert torch.equal(rows[1].isnan(), rows[0] % 9 == 0)
