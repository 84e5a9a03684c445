"""The reference's walk over the traversal layout (many rays) against the walk
over the drop-in nodes (few rays at a time): hits, distances, counts and the
stack's overflow are the same, also for rays and nodes at the edges."""
import numpy as np
import pytest

import clear_amd as ca
from test_gpu_trace_nocounts import cuda, edge_rays, mesh

pytestmark = pytest.mark.gpu

MANY, FEW, FACES = 1 << 14, 9000, 4096  # the layout is used from 2^14 rays and 4096 faces on


def trace(ctx, nodes, n, v, f, rays, counts):
    import torch

    R = rays.shape[1]
    hit = torch.empty(R, dtype=torch.int32, device="cuda")
    t = torch.empty(R, dtype=torch.float32, device="cuda")
    st = torch.zeros(2 * R, dtype=torch.int32, device="cuda") if counts else None
    ca.trace_closest(ctx, *nodes, n, v, f, cuda(rays), R, hit, t, st)
    torch.cuda.synchronize()
    return (hit.cpu().numpy(), t.cpu().numpy(),
            st.cpu().numpy().reshape(-1, 2) if counts else np.zeros((R, 2), np.int32), ctx.device_status())


def compare(ctx, nodes, n, v, f, rays, counts, status=0):
    assert rays.shape[1] >= MANY and n >= FACES and rays.shape[1] >= n // 128
    a = trace(ctx, nodes, n, v, f, rays, counts)
    parts = [trace(ctx, nodes, n, v, f, np.ascontiguousarray(rays[:, k:k + FEW]), counts)
             for k in range(0, rays.shape[1], FEW)]
    for k in range(3):  # a NaN distance (vertices that are not finite) may have either sign
        np.testing.assert_array_equal(a[k], np.concatenate([p[k] for p in parts]))
    assert a[3] == status and np.bitwise_or.reduce([p[3] for p in parts]) == status


@pytest.mark.parametrize("counts", [False, True])
@pytest.mark.parametrize("n,bits", [(FACES, 10), (4999, 10), (60000, 20)])
def test_same_as_over_drop_in_nodes(gpu_ctx, n, bits, counts):
    v, f = mesh(n)
    if n == 4999:
        v[7, 1], v[100, 0], v[400, 2] = np.nan, np.inf, -np.inf
    rays = edge_rays(MANY + 1000 + n % 7, seed=n)
    rays[0, 5], rays[4, 6] = np.nan, np.nan
    rays[3:6, 7] = 0.0
    print(f"[trace reference] n={n} bits={bits} counts={counts}", flush=True)
    tv, tf = cuda(v), cuda(f)
    nodes = ca.node_buffers(n)
    ca.LBVHBuilder(gpu_ctx, n, bits).perform(tv, tf, n, bits, *nodes)
    compare(gpu_ctx, nodes, n, tv, tf, rays, counts)


def comb(levels, miss):
    """A chain of nodes whose left child is a node of two leaves and whose
    right child is the next link: a walk that enters every box puts one more
    entry on its stack per level. Every `miss`-th pair lies off to the side.
    Faces beyond the chain belong to nodes that no walk reaches."""
    rng = np.random.default_rng(levels)
    n = FACES
    soup = rng.random((n, 9)).astype(np.float32)
    for k in range(levels):
        if miss and k % miss == 0:
            soup[2 * k:2 * k + 2, 0::3] += np.float32(50.0)
    tri = soup.reshape(n, 3, 3)
    lo, hi = tri.min(1), tri.max(1)
    leaves = np.zeros((n, 12), np.uint32)
    inodes = np.zeros((n - 1, 12), np.uint32)

    def box(rec, a, b):
        rec[0:3], rec[4:7] = a.astype(np.float32).view(np.uint32), b.astype(np.float32).view(np.uint32)

    for k in range(n):
        box(leaves[k], lo[k], hi[k])
        leaves[k, 8] = k
    for k in range(levels):  # link k is node k, its pair node levels + k
        box(inodes[k], lo[2 * k:2 * levels + 1].min(0), hi[2 * k:2 * levels + 1].max(0))
        last = k + 1 == levels
        inodes[k, 8:11] = [0x100 if last else 0, levels + k, 2 * levels if last else k + 1]
        box(inodes[levels + k], lo[2 * k:2 * k + 2].min(0), hi[2 * k:2 * k + 2].max(0))
        inodes[levels + k, 8:11] = [0x101, 2 * k, 2 * k + 1]
    return soup, inodes, leaves


@pytest.mark.parametrize("levels,miss,status", [(20, 3, 0), (63, 0, 0), (64, 2, 0), (64, 0, 0), (65, 0, 4), (65, 2, 4),
                                                (90, 3, 4)])
def test_stack_slots_are_the_drop_in_walks(gpu_ctx, levels, miss, status):
    soup, inodes, leaves = comb(levels, miss)
    v, f = ca.soup_to_mesh(soup)
    rng = np.random.default_rng(5)
    rays = np.empty((7, MANY), np.float32)
    rays[0:3] = rng.random((3, MANY))
    rays[3:6] = rng.normal(size=(3, MANY))
    rays[6] = np.inf
    print(f"[trace reference] comb of {levels} levels", flush=True)
    compare(gpu_ctx, (cuda(inodes), cuda(leaves)), soup.shape[0], cuda(v), cuda(f), rays, True, status)


@pytest.mark.parametrize("counts", [False, True])
def test_leaves_of_faces_beyond_num_faces(gpu_ctx, counts):
    """Leaves may refer to any face of the caller's array, as for the walk over
    the drop-in nodes: a tree over the last faces of a longer array."""
    n, first = 5000, 3000
    v, f = mesh(first + n)
    sub = np.ascontiguousarray(f[first:])
    tv, tf = cuda(v), cuda(f)
    nodes = ca.node_buffers(n)
    ca.LBVHBuilder(gpu_ctx, n, 10).perform(tv, cuda(sub), n, 10, *nodes)
    leaves = nodes[1].cpu().numpy().view(np.uint32).reshape(-1, 12)
    leaves[:, 8] += first
    nodes = (nodes[0], cuda(leaves))
    print(f"[trace reference] faces beyond numFaces, counts={counts}", flush=True)
    compare(gpu_ctx, nodes, n, tv, tf, edge_rays(MANY + 3, seed=11), counts)


@pytest.mark.parametrize("word", [0xFFFFFFFF, 0xABABABAB, 0x80000000])
def test_leaves_that_no_node_refers_to(gpu_ctx, word):
    """Only the leaves of the tree count, as for the walk over the drop-in
    nodes: the others may hold anything."""
    levels = 20
    soup, inodes, leaves = comb(levels, 0)
    leaves[2 * levels + 1:, 8] = word
    v, f = ca.soup_to_mesh(soup)
    print(f"[trace reference] unused leaves of {word:#x}", flush=True)
    compare(gpu_ctx, (cuda(inodes), cuda(leaves)), soup.shape[0], cuda(v), cuda(f), edge_rays(MANY, seed=12), True)
