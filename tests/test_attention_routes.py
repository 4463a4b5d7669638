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
