"""GPU parity of the union attention forward (gw_sparse_attn_fwd_union) against the oracle.

Sixteen queries of a head share one list of keys per 256-key tile (at most 8 steps of 32
keys, in two groups of 4), so the sizes here sit at the edges of blocks, tiles, steps and
groups, and the positions range from a few keys per tile to every key of it.

Tolerance: P enters its product as fp16 (relative error 2^-11 per weight), V as fp16 (2^-11;
exact for fp16 inputs up to the scaling), o is rounded to the input type (2^-9 in bf16, 2^-12
in fp16); the 2-norm of independent roundings stays below the sum of the three bounds. lse: an
fp32 sum of fp32 weights (1e-5) over fp32 scores, which both sides sum over 64 products (a
random walk of 64 roundings is 8 ulp a side: 16 ulp = 2^-20 of |lse|, the scores' size).
"""
import contextlib

import pytest
import torch

from geoweave_amd.custom_flash_attn import sparse_index_flash_attn as sifa
from oracle import attention as oatt

pytestmark = pytest.mark.gpu

REL = {torch.bfloat16: 2.0 ** -9 + 2.0 ** -10, torch.float16: 2.0 ** -12 + 2.0 ** -10}


@contextlib.contextmanager
def _path(name):
    old = sifa.FORWARD_PATH
    sifa.FORWARD_PATH = name
    try:
        yield
    finally:
        sifa.FORWARD_PATH = old


def _inputs(B, T, S, H, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(B, n, H, 64, generator=g).to(dtype) for n in (T, S, S)]


def _positions(B, T, S, K, seed, lo=0, hi=None):
    """Distinct positions in [lo, hi) per row."""
    g = torch.Generator().manual_seed(seed)
    hi = S if hi is None else hi
    return (lo + torch.rand(B, T, hi - lo, generator=g).topk(K, dim=-1).indices).to(torch.int32)


def _run(q, k, v, pos, scale=0.125, layout="bthd", path="union"):
    qd, kd, vd, pd = (x.cuda() for x in (q, k, v, pos))
    if layout == "bhtd":
        qd, kd, vd = (x.transpose(1, 2).contiguous() for x in (qd, kd, vd))
    with _path(path):
        o, attn, lse, _ = sifa._flash_attn_forward(qd, kd, vd, pd, softmax_scale=scale, return_attn=False, q_layout=layout)
    torch.cuda.synchronize()
    assert attn is None
    return (o.transpose(1, 2) if layout == "bhtd" else o).float().cpu(), lse.cpu()


def _check(q, k, v, pos, o, lse, scale=0.125):
    ro, _, rl = oatt.sparse_attention(q.float(), k.float(), v.float(), pos, scale)
    assert torch.equal(torch.isinf(lse), torch.isinf(rl))
    ok = torch.isfinite(rl)
    assert ((lse[ok] - rl[ok]).abs() <= 1e-5 + 2.0 ** -20 * rl[ok].abs()).all()
    assert torch.isfinite(o).all()
    assert (o - ro).norm() <= REL[q.dtype] * ro.norm()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,S,K", [(1, 1, 1), (15, 255, 7), (16, 256, 256), (17, 257, 40), (255, 513, 16), (257, 700, 300),
                                   (529, 1025, 64), (40, 5000, 600)])
def test_edges(gpu_device, dtype, T, S, K):
    print(f"[union] T={T} S={S} K={K} {dtype}", flush=True)
    q, k, v = _inputs(2, T, S, 3, dtype, T * 31 + S)
    pos = _positions(2, T, S, K, S)
    _check(q, k, v, pos, *_run(q, k, v, pos))


@pytest.mark.parametrize("lo,width,K", [(0, 256, 100), (256, 256, 9), (512, 200, 128), (100, 300, 64), (768, 32, 5)])
def test_clustered_positions(gpu_device, lo, width, K):
    # Whole tiles listed by the block (both groups of steps), one step, and tiles with none.
    print(f"[union] clustered lo={lo} width={width} K={K}", flush=True)
    q, k, v = _inputs(1, 130, 1100, 2, torch.bfloat16, lo + K)
    pos = _positions(1, 130, 1100, K, K, lo, lo + width)
    _check(q, k, v, pos, *_run(q, k, v, pos))


def test_masked_empty_and_growing_scores(gpu_device):
    # -1 and out-of-range positions, rows without any, and scores that rise along the keys (the
    # reference maximum moves many times).
    print("[union] masked", flush=True)
    q, k, v = _inputs(1, 100, 2000, 2, torch.float16, 5)
    q = q.abs() * 4
    k = (k.abs() * torch.linspace(0.1, 4, 2000).view(1, -1, 1, 1)).to(torch.float16)
    pos = _positions(1, 100, 2000, 90, 6)
    pos[:, ::3, 40:] = -1
    pos[:, 7] = -1
    pos[:, 9, 5:] = 5000
    o, lse = _run(q, k, v, pos)
    _check(q, k, v, pos, o, lse)
    assert (o[:, 7] == 0).all()


def test_repeated_positions_and_nonfinite_rows(gpu_device):
    # Both are computed by the gather kernel inside the call.
    print("[union] repeated, non-finite", flush=True)
    q, k, v = _inputs(2, 70, 900, 2, torch.bfloat16, 11)
    pos = _positions(2, 70, 900, 50, 12, 0, 899)
    pos[0, 33, 1] = pos[0, 33, 0]
    _check(q, k, v, pos, *_run(q, k, v, pos))
    k2, v2 = k.clone(), v.clone()
    k2[1, 899], v2[1, 899] = float("nan"), float("inf")  # a row that no query selected
    _check(q, k, v, pos, *_run(q, k2, v2, pos))


@pytest.mark.parametrize("layout", ["bthd", "bhtd"])
def test_layouts_strides_and_column_scales(gpu_device, layout):
    print(f"[union] {layout}", flush=True)
    q, k, v = _inputs(1, 90, 1300, 4, torch.bfloat16, 21)
    v = (v.float() * torch.logspace(-6, 6, 64)).to(torch.bfloat16)
    pos = _positions(1, 90, 1300, 70, 22)
    o, lse = _run(q, k, v, pos, layout=layout)
    ro, _, _ = oatt.sparse_attention(q.float(), k.float(), v.float(), pos, 0.125)
    col = lambda x: x.reshape(-1, 64).norm(dim=0)  # noqa: E731
    assert (col(o - ro) <= REL[torch.bfloat16] * col(ro)).all()
    if layout == "bthd":  # strided views (v read in place from a wider row), positions with a row stride
        wide = torch.zeros(1, 1300, 4 * 64 * 2, dtype=torch.bfloat16)
        wide[..., 256:] = v.reshape(1, 1300, 256)
        vv = wide.cuda()[..., 256:].view(1, 1300, 4, 64)
        pp = torch.cat([pos, pos], -1).cuda()[..., :70]
        with _path("union"):
            o2, _, lse2, _ = sifa._flash_attn_forward(q.cuda(), k.cuda(), vv, pp, softmax_scale=0.125, return_attn=False)
        assert torch.equal(o2.float().cpu(), o) and torch.equal(lse2.cpu(), lse)


def test_routes(gpu_device, monkeypatch):
    # The rule's own choice gives the bits of the pass it names, and not those of the others.
    cases = [(14, "dense", 16500), (15, "union", 16500), (97, "gather", 16500), (17, "dense", 14 * 64), (18, "union", 14 * 64)]
    for ratio, path, few in cases:
        S, K = ratio * 64, 64
        monkeypatch.setattr(sifa, "UNION_FEW", few)
        print(f"[union] route S={S} K={K} few={few}", flush=True)
        q, k, v = _inputs(1, 64, S, 2, torch.bfloat16, S)
        pos = _positions(1, 64, S, K, S)
        o, lse = _run(q, k, v, pos, path="auto")
        for name in ("dense", "union", "gather"):
            on, ln = _run(q, k, v, pos, path=name)
            assert torch.equal(o, on) == (name == path), (ratio, name)
            assert (o - on).norm() <= 2 * REL[torch.bfloat16] * on.norm() and (lse - ln).abs().max() < 1e-4


@pytest.mark.parametrize("limit,value", [("DENSE_MAX_S", 100), ("DENSE_MAX_T", 16), ("DENSE_MAX_K_ROW_STRIDE", 64)])
def test_calls_beyond_the_dense_limits_stay_with_the_gather(gpu_device, monkeypatch, limit, value):
    # With the dense limits lowered below the call, "auto" gives the gather kernel's bits, not the union's.
    print(f"[union] {limit}", flush=True)
    g = torch.Generator().manual_seed(11)
    q, k, v = (torch.randn(1, n, 2, 64, generator=g).bfloat16().cuda() for n in (40, 640, 640))
    pos = torch.rand(1, 40, 640, generator=g).topk(32, dim=-1).indices.to(torch.int32).cuda()

    def run(path):
        monkeypatch.setattr(sifa, "FORWARD_PATH", path)
        return sifa._flash_attn_forward(q, k, v, pos, softmax_scale=0.125, return_attn=False)[0]

    gather, union = run("gather"), run("union")
    assert torch.equal(run("auto"), union) and not torch.equal(gather, union)
    monkeypatch.setattr(sifa, limit, value)
    assert torch.equal(run("auto"), gather)


def _against_gather(q, k, v, pos, rows):
    """Every (row, head) of the union pass against the gather kernel, and the given rows against the oracle."""
    o, lse = _run(q, k, v, pos)
    og, lg = _run(q, k, v, pos, path="gather")
    rel = REL[q.dtype] + (2.0 ** -9 if q.dtype == torch.bfloat16 else 2.0 ** -12)
    assert (o - og).norm() <= rel * og.norm()
    # a head's 64 values: their errors' norm within 8 times the mean's (a wrong tile, list or row gives O(1))
    assert ((o - og).norm(dim=-1) <= 8 * rel * og.norm(dim=-1) + 1e-6).all()
    ok = torch.isfinite(lg)  # -inf: rows without a valid key
    assert torch.equal(lse[~ok], lg[~ok]) and (lse[ok] - lg[ok]).abs().max() <= 1e-4
    _check(q[:, rows], k, v, pos[:, rows], o[:, rows], lse[:, rows])


# Queries for which the launch takes 9 to 16 waves of one or two 16-query blocks (16 heads, 256 CUs).
SHAPES = {(9, 1): 301, (10, 1): 2330, (11, 1): 2590, (12, 1): 2853, (13, 1): 3100, (14, 1): 3361, (15, 1): 3610,
          (16, 1): 3870, (9, 2): 4130, (10, 2): 4650, (11, 2): 5131, (12, 2): 5650, (13, 2): 6170, (14, 2): 6693,
          (15, 2): 7200, (16, 2): 7727}


@pytest.mark.parametrize("shape", SHAPES)
def test_launch_shapes(gpu_device, shape):
    # Tile 0 holds most keys (more than eight units a block), tiles 1 and 3 a few, tile 2 none, tile 4
    # the ragged end; some rows without valid keys, one with a repeated position in a later block.
    T = SHAPES[shape]
    dtype = torch.float16 if shape[0] % 2 else torch.bfloat16
    print(f"[union] {shape[0]} waves of {shape[1]} blocks, T={T} {dtype}", flush=True)
    S, K = 1033, 40
    q, k, v = _inputs(1, T, S, 16, dtype, T)
    pos = torch.cat([_positions(1, T, S, 28, 1, 0, 256), _positions(1, T, S, 5, 2, 256, 512),
                     _positions(1, T, S, 4, 3, 768, 1024), _positions(1, T, S, 3, 4, 1024, S)], -1)
    pos = pos[..., torch.randperm(K, generator=torch.Generator().manual_seed(5))]
    pos[:, 5::97, :] = -1
    pos[:, 3::11, 20:] = -1
    pos[0, T - 3, 7] = pos[0, T - 3, 6]
    rows = sorted(set(range(0, T, 83)) | set(range(T - 40, T)) | {15, 16, 31, 32})
    _against_gather(q, k, v, pos, rows)


@pytest.mark.parametrize("S", [32769, 34816, 34817, 70000])
def test_long_key_ranges(gpu_device, S):
    # 129 and 136 tiles: the most that one pass over the positions holds; 137 and 274: two and three passes.
    print(f"[union] S={S}", flush=True)
    T, K = 70, 400
    q, k, v = _inputs(1, T, S, 2, torch.bfloat16, S)
    edge = (S + 255) // 256 // (1 + (S > 34816) + (S > 69632)) * 256  # about the first pass's end
    near = _positions(1, T, S, 100, 8, max(0, edge - 700), min(S, edge + 700))
    far = _positions(1, T, S, K - 100, 9, 0, max(0, edge - 700))
    pos = torch.cat([near, far], -1)
    pos[0, 20, 3] = pos[0, 20, 50]  # near the line
    pos[0, 50, 3] = S - 1
    pos[0, 50, 4] = S - 1
    _against_gather(q, k, v, pos, list(range(0, T, 3)))


def test_queries_in_several_launches(gpu_device):
    # 100,000 queries and keys: records of 2.4 GiB, so two launches, of 65,536 and 34,464 queries.
    T, K = 100_000, 1050
    print(f"[union] {T} queries and keys", flush=True)
    q, k, v = _inputs(1, T, T, 2, torch.bfloat16, 31)
    g = torch.Generator().manual_seed(32)
    off = torch.randint(0, T, (1, T, 1), generator=g).cuda()
    pos = ((off + torch.arange(K, device="cuda") * 7919) % T).to(torch.int32)
    pos[0, 65_530, 5] = pos[0, 65_530, 4]  # the gather kernel computes the blocks on both sides of the line
    pos[0, 65_560, 5] = pos[0, 65_560, 4]
    rows = list(range(65_500, 65_580, 5)) + [0, T - 1]
    out = {}
    for path in ("union", "gather"):
        with _path(path):
            o, _, lse, _ = sifa._flash_attn_forward(q.cuda(), k.cuda(), v.cuda(), pos, softmax_scale=0.125, return_attn=False)
        out[path] = o.float(), lse
    (o, lse), (og, lg) = out["union"], out["gather"]
    rel = REL[torch.bfloat16] + 2.0 ** -9
    assert (o - og).norm() <= rel * og.norm()
    assert ((o - og).norm(dim=-1) <= 8 * rel * og.norm(dim=-1) + 1e-6).all()
    assert (lse - lg).abs().max() <= 1e-4
    _check(q[:, rows], k, v, pos[:, rows].cpu(), o[:, rows].cpu(), lse[:, rows].cpu())


def test_captured_in_a_graph(gpu_device):
    # The union pass, and the forward with the separate mass, captured and replayed between eager work.
    print("[union] graph", flush=True)
    for S, K, attn in ((1100, 60, False), (1300, 260, True)):
        q, k, v = (x.cuda() for x in _inputs(1, 300, S, 4, torch.bfloat16, S))
        pos = _positions(1, 300, S, K, S).cuda()
        assert sifa._use_mass(1, 300, S, 4, K) if attn else sifa._use_union(1, 300, S, K, 64, 0.125, False)

        def call():
            return sifa._flash_attn_forward(q, k, v, pos, softmax_scale=0.125, return_attn=attn)[:3]

        eager = call()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            call()
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            captured = call()
        for i in range(4):
            for t in captured:
                if t is not None:
                    t.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert all(a is b is None or torch.equal(a, b) for a, b in zip(eager, captured)), (S, i)
            assert torch.equal(call()[0], eager[0])
