"""The projection glue with its outputs cast in the same pass (a 16-bit score dtype), against
the glue followed by torch casts: bit for bit the same, v included."""
import pytest
import torch

from geoweave_amd import dsa_layer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rope", [True, False])
@pytest.mark.parametrize("norms", [True, False])
@pytest.mark.parametrize("src,dst", [(torch.bfloat16, torch.float16), (torch.float16, torch.bfloat16)])
@pytest.mark.parametrize("B,N,H,Hi", [(1, 1, 16, 4), (2, 37, 3, 1), (1, 301, 16, 0)])
def test_cast_in_the_glue(gpu_device, B, N, H, Hi, src, dst, norms, rope):
    print(f"[glue cast] {B}x{N} H={H} Hi={Hi} {src}->{dst} norms={norms} rope={rope}", flush=True)
    g = torch.Generator().manual_seed(N + H)
    lay = dsa_layer.GlueLayout(H, 64, Hi, 64)
    y = torch.randn(B, N, lay.ldy, generator=g)
    if src == torch.bfloat16:
        y[0, 0, lay.v_off:lay.v_off + 64] *= 3e4  # v beyond fp16 once cast
    y = y.to(src).cuda()
    ln = [tuple(torch.randn(64, generator=g).cuda() for _ in range(2)) if norms else (None, None) for _ in range(3)]
    pos = torch.randint(0, 30, (B, N, 2), generator=g).int().cuda() if rope else None
    plain = dsa_layer.dsa_glue_forward(y, lay, *ln, 1e-5, pos, 100.0, 30 if rope else None)
    cast = dsa_layer.dsa_glue_forward(y, lay, *ln, 1e-5, pos, 100.0, 30 if rope else None, out_dtype=dst)
    for a, b in zip(plain, cast):
        if a is None:
            assert b is None
            continue
        assert b.dtype == dst and b.shape == a.shape
        assert torch.equal(a.to(dst).contiguous().view(torch.int16), b.contiguous().view(torch.int16))
