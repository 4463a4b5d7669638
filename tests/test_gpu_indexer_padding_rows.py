"""Lanes of the indexer's filter past the last query (a workgroup takes 128 or 256 queries) own no
candidate list and write none, also where NaN gates or keys make their scores NaN: the memory
behind the workspace stays as it was, and the other batch elements' lists too."""
import ctypes

import pytest
import torch

from geoweave_amd import _lib
from geoweave_amd.custom_indexer import sparse_topk_indexer as sti

pytestmark = pytest.mark.gpu

GUARD = 32 << 20  # past the list of the last lane: 255 lists of 64 KB


def _launch(q, k, w, topk, flags):
    B, T, H, D = q.shape
    S = k.shape[1]
    lib = _lib.load()
    need = int(lib.gw_indexer_topk_workspace_size(B, T, S, topk))
    ws = torch.full((need + GUARD,), 0x5A, device=q.device, dtype=torch.uint8)
    idx = torch.empty(B, T, topk, device=q.device, dtype=torch.int32)
    scores = torch.empty(B, T, topk, device=q.device, dtype=q.dtype)
    rc = lib.gw_indexer_topk_fwd(_lib.dtype_code(q.dtype, allow_fp32=True), q.data_ptr(), k.data_ptr(), w.data_ptr(), None,
                                 B, T, S, H, D, topk, 0.125, flags, idx.data_ptr(), scores.data_ptr(), ws.data_ptr(), need,
                                 ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    _lib.check(rc, "gw_indexer_topk_fwd")
    torch.cuda.synchronize()
    assert (ws[need:] == 0x5A).all()
    return idx, scores


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("S,flags", [(700, sti.FLAG_TAU_MINUS_INF), (5000, 0)])
@pytest.mark.parametrize("bits", [0x7FC0, 0xFFC0, 0x7F80])  # NaN of both signs, inf: the bf16 pattern, or fp32's upper half
def test_lanes_past_the_last_query_write_nothing(gpu_device, bits, S, flags, dtype):
    print(f"[padding rows] bits={bits:x} S={S} flags={flags} {dtype}", flush=True)
    value = torch.tensor([(bits << 16) - (1 << 32 if bits >> 15 else 0)], dtype=torch.int32).view(torch.float32)
    if dtype == torch.bfloat16:
        value = value.view(torch.bfloat16)[1:]
    value = value.cuda()
    g = torch.Generator().manual_seed(S)
    q, k = (torch.randn(2, n, 2, 64, generator=g).to(dtype).cuda() for n in (60, S))
    w = (1 + 0.5 * torch.rand(2, S, 2, generator=g)).to(dtype).cuda()
    bad = w.clone()
    bad[0, ::5] = value  # the other batch element's selection must not change
    ref_idx, ref_scores = _launch(q, k, w, 100, flags)
    idx, scores = _launch(q, k, bad, 100, flags)
    assert torch.equal(idx[1], ref_idx[1]) and torch.equal(scores[1], ref_scores[1])
    bad = k.clone()
    bad[0, ::7, 1, 3] = value
    idx, scores = _launch(q, bad, w, 100, flags)
    assert torch.equal(idx[1], ref_idx[1]) and torch.equal(scores[1], ref_scores[1])
