"""The rules that choose between the attention passes, at calls that were timed on both sides."""
import pytest

from geoweave_amd.custom_flash_attn import sparse_index_flash_attn as sifa


# batch, queries, keys, heads, selected keys; times of the forward with attn_sum in us: scores
# stored, scores recomputed by the mass pass.
@pytest.mark.parametrize("call,stored,recomputed", [
    ((8, 300, 300, 16, 128), 66, 101), ((1, 300, 300, 16, 128), 57, 92), ((4, 1374, 1374, 16, 128), 137, 153),
    ((8, 421, 421, 16, 72), 72, 108), ((8, 5632, 5632, 16, 512), 2374, 2544), ((8, 2816, 2816, 4, 256), 281, 328),
    ((1, 5496, 5496, 16, 1024), 559, 368), ((8, 1374, 1374, 16, 1024), 745, 277), ((1, 10992, 10992, 16, 1024), 1308, 1225),
    ((1, 9384, 9384, 16, 1024), 1410, 990), ((2, 9216, 9216, 16, 1024), 1892, 1683), ((1, 1574, 1574, 8, 140), 106, 98),
    ((4, 2048, 10992, 16, 1024), 1019, 949), ((1, 1, 5496, 16, 1024), 251, 172),
])
def test_mass_takes_the_faster_pass(call, stored, recomputed):
    assert sifa._use_mass(*call) == (recomputed < stored)


# batch, queries, keys, heads, selected keys; times of the forward without attn_sum in us: dense, union.
@pytest.mark.parametrize("call,dense,union", [
    ((4, 1024, 16384, 16, 1024), 430, 449), ((3, 8347, 10477, 16, 673), 1175, 1260), ((1, 22128, 22128, 12, 1455), 1698, 1781),
    ((1, 10992, 10992, 16, 1024), 640, 730), ((1, 13739, 13739, 16, 1024), 950, 1020), ((4, 7522, 7522, 16, 529), 997, 1091),
    ((1, 16488, 16488, 16, 1024), 1400, 1360), ((1, 21984, 21984, 16, 1024), 2260, 1830), ((1, 1, 16384, 16, 1024), 313, 131),
    ((8, 3768, 8455, 16, 429), 1156, 1130), ((1, 43968, 43968, 16, 1024), 7400, 4340),
])
def test_union_takes_the_faster_pass(call, dense, union):
    batch, seqlen_q, seqlen_k, _, num_kv = call
    assert sifa._use_union(batch, seqlen_q, seqlen_k, num_kv, 64, 0.125, False) == (union < dense)
