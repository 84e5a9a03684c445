"""LBVH builds whose nodes cross the hierarchy's blocks of leaves (256 or 1024,
by the triangle count) and groups of 64 blocks: byte-exact against the oracle."""
import numpy as np
import pytest

import clear_amd as ca
import oracle as orc
from test_gpu_lbvh import assert_same_as_oracle, random_soup, run_segmented, segmented_soup

pytestmark = pytest.mark.gpu


def line_soup(n):
    """Centres at halving distances, many per step: codes with long common
    prefixes, so chains of nodes as deep as the keys allow."""
    k = np.arange(n)
    s = np.zeros((n, 9), np.float32)
    s[:, 0::3] = (0.5 ** (k * 40 // n))[:, None]
    s[:, 1::3] = ((k % 7) * 0.125)[:, None]
    return s


def zero_soup(n):
    """Boxes with zeros of either sign and a few NaN vertices: which of two
    equal bounds a node keeps depends on the order of its leaves."""
    rng = np.random.default_rng(n)
    s = np.where(rng.random((n, 9)) < 0.5, np.float32(0.0), np.float32(-0.0)).astype(np.float32)
    s[rng.random(n) < 0.3] = 1.0
    s[rng.integers(0, n, 3), rng.integers(0, 9, 3)] = np.nan
    return s


SOUPS = {"random": lambda n: random_soup(n, n, dup=True), "same": lambda n: np.full((n, 9), 0.25, np.float32),
         "line": line_soup, "zeros": zero_soup}


@pytest.mark.parametrize("soup", SOUPS)
@pytest.mark.parametrize("n,bits", [(1024, 10), (1025, 10), (1279, 20), (1280, 20), (1281, 20), (16384, 10),
                                    (16385, 20), (40000, 21)])
def test_block_edges_byte_exact(gpu_ctx, n, bits, soup):
    assert_same_as_oracle(gpu_ctx, SOUPS[soup](n), bits)


@pytest.mark.parametrize("n,bits", [(1 << 19, 10), ((1 << 19) + 1, 10), ((1 << 19) + 1, 20),
                                    (1 << 18, 20), ((1 << 18) + 1, 20)])
def test_block_and_tile_rules_byte_exact(gpu_ctx, n, bits):
    assert_same_as_oracle(gpu_ctx, random_soup(n, 3, dup=True), bits)


@pytest.mark.parametrize("sizes", [[1] * 1500 + [3000] + [2] * 600, [256, 1, 767, 1, 1023, 2048] * 3,
                                   [5, 300000, 7, 300000, 1]])
def test_segmented_scenes_across_blocks(gpu_ctx, sizes):
    soup, offs, soups = segmented_soup(sizes, 11)
    print(f"[lbvh segmented] {len(sizes)} scenes, {int(offs[-1])} triangles", flush=True)
    gi, gl = run_segmented(gpu_ctx, soup, offs)
    for s, one in enumerate(soups):
        a, b = int(offs[s]), int(offs[s + 1])
        o = orc.lbvh_build(*ca.soup_to_mesh(one), 10)
        np.testing.assert_array_equal(gl[a:b], o["leaves"], err_msg=f"leaves of scene {s}")
        if b - a > 1:
            np.testing.assert_array_equal(gi[a - s:b - s - 1], o["inodes"], err_msg=f"nodes of scene {s}")
    assert gpu_ctx.device_status() == 0


@pytest.mark.parametrize("n,bits", [(1 << 19, 10), (1 << 19, 20), (1 << 18, 20)])
def test_memory_reserved_for_more_serves_fewer(gpu_ctx, n, bits):
    """At the end of a small shape's range there are more blocks of leaves or
    sort tiles than just above."""
    import torch

    ctx = ca.Context()
    ca.LBVHBuilder(ctx, n + 1, bits)
    tris = torch.from_numpy(random_soup(n, 9, dup=False)).cuda()
    inodes, leaves = ca.node_buffers(n)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    ca.LBVHBuilder(ctx, 0).perform_soup(tris, n, bits, inodes, leaves)
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] == before
