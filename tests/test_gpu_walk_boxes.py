"""Walks without per-ray counts against the walks whose box decisions are
defined (the oracle's ordered traversal and the same calls with counts), where
those decisions are close: boxes and rays that meet near the coordinate
planes, far from their record's corner."""
import numpy as np
import pytest

import clear_amd as ca
import oracle as orc
from test_gpu_trace_nocounts import cuda, results, same

pytestmark = pytest.mark.gpu


def aimed(p, d, dist):
    """Rays of directions d that reach the points p after `dist`."""
    d = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays = np.empty((7, len(p)), np.float32)
    rays[0:3], rays[3:6], rays[6] = (p - d * dist[:, None]).T, d.T, np.inf
    return rays


def traced(ctx, v, f, rays, walk):
    """Hits of one of the walks without counts, on the device."""
    import torch

    n, R = len(f), rays.shape[1]
    hit, t = results(R)
    tv, tf, tr = cuda(v), cuda(f), cuda(rays)
    if walk == "midpoint":
        ca.trace_closest_bvh(ctx, cuda(ca.build_midpoint_bvh(v, f)), n, tv, tf, tr, R, hit, t, ordered=True)
    else:
        inodes, leaves = ca.node_buffers(n)
        ca.LBVHBuilder(ctx, n).perform(tv, tf, n, 10, inodes, leaves)
        ca.trace_closest(ctx, inodes, leaves, n, tv, tf, tr, R, hit, t, ordered=walk == "ordered", wide=walk == "wide")
    torch.cuda.synchronize()
    assert ctx.device_status() == 0
    return hit, t


@pytest.mark.parametrize("walk", ["ordered", "wide", "midpoint"])
@pytest.mark.parametrize("extent", [1, 10, 100, 1000])
def test_flat_boxes_far_from_their_records_corner(gpu_ctx, extent, walk):
    """A triangle in the plane x = 0 with corners on the axes, beside one whose
    box starts at -extent: rays from 1e-7 to 1 before the plane, and rays aimed
    at an edge."""
    e, R = float(extent), 20000
    soup = np.array([[-e, -e, -e, 1 - e, 1 - e, -e, -e, 1 - e, 1 - e], [0, 0, 0, 0, 1, 0, 0, 0, 1]], np.float32)
    rng = np.random.default_rng(extent)
    b = rng.random((R, 2))
    b = np.where(b.sum(1, keepdims=True) > 1, 1 - b, b)
    b[R // 2:, 0] *= 1e-3
    dist = np.where(np.arange(R) < R // 2, 10.0 ** rng.uniform(-7, 0, R), rng.uniform(0.05, 0.5, R))
    rays = aimed(np.c_[np.zeros(R), b], rng.normal(size=(R, 3)), dist)
    if extent == 100:
        rays[:6, 0] = [0.152555928, 0.0348040573, 0.32536763, -0.888217509, -0.202636451, -0.412320524]
    v, f = ca.soup_to_mesh(soup)
    o = orc.lbvh_build(v, f, 10)
    h, bt, _ = orc.trace_wide(o["inodes"], o["leaves"], 2, v, f, rays)
    assert (h == 1).mean() > 0.99
    print(f"[walk boxes] flat box, extent {extent}, {walk}", flush=True)
    same(*traced(gpu_ctx, v, f, rays, walk), h, bt)


@pytest.mark.parametrize("walk", ["ordered", "wide", "midpoint"])
def test_grid_geometry_around_the_origin(gpu_ctx, walk):
    """Unit squares in the planes x, y, z = 0 of a scene of extent 64 with
    coinciding copies (ties in t), and rays that start near those planes."""
    rng = np.random.default_rng(3)
    k = rng.integers(-64, 64, size=(1500, 2)).astype(np.float32)
    quads = []
    for axis in range(3):
        c = np.zeros((500, 4, 3), np.float32)
        c[:, :, (axis + 1) % 3] = k[500 * axis:500 * axis + 500, :1] + np.array([0, 1, 1, 0], np.float32)
        c[:, :, (axis + 2) % 3] = k[500 * axis:500 * axis + 500, 1:] + np.array([0, 0, 1, 1], np.float32)
        quads.append(c)
    q = np.concatenate(quads)
    soup = np.concatenate([q[:, [0, 1, 2]].reshape(-1, 9), q[:, [0, 2, 3]].reshape(-1, 9)])
    soup = np.concatenate([soup, soup[::3]])
    R = 20000
    pick = rng.integers(0, len(q), R)
    w = rng.random((R, 2, 1)) * np.where(rng.random((R, 1, 1)) < 0.3, 1e-3, 1.0)
    p = q[pick, 0] + w[:, 0] * (q[pick, 1] - q[pick, 0]) + w[:, 1] * (q[pick, 3] - q[pick, 0])
    rays = aimed(p, rng.normal(size=(R, 3)), 10.0 ** rng.uniform(-7, 1, R))
    v, f = ca.soup_to_mesh(soup)
    o = orc.lbvh_build(v, f, 10)
    h, bt, _ = orc.trace_wide(o["inodes"], o["leaves"], len(f), v, f, rays)
    assert (h != 0xFFFFFFFF).mean() > 0.8
    print(f"[walk boxes] grid, {walk}", flush=True)
    same(*traced(gpu_ctx, v, f, rays, walk), h, bt)


@pytest.mark.parametrize("walk", ["ordered", "wide", "midpoint"])
@pytest.mark.parametrize("bound", [np.inf, 0.0])
def test_hits_at_distance_zero(gpu_ctx, bound, walk):
    """Rays that start on the vertices, edges and faces of a bent sheet: all the
    triangles there are hit at t = 0 and the smallest face index wins, so no
    box with entry 0 may be dropped, also for a ray that ends at 0."""
    m = 24
    x, y = np.meshgrid(np.arange(m + 1), np.arange(m + 1), indexing="ij")
    p = np.stack([x, y, (x * y) % 3], -1).astype(np.float32)
    a, b, c, d = p[:-1, :-1], p[1:, :-1], p[1:, 1:], p[:-1, 1:]
    tri = np.concatenate([np.stack([a, b, c], 2).reshape(-1, 3, 3), np.stack([a, c, d], 2).reshape(-1, 3, 3)])
    rng = np.random.default_rng(8)
    tri = tri[rng.permutation(len(tri))]
    R = 9000
    at, u = rng.integers(0, len(tri), R), np.zeros((R, 3))
    k = np.arange(R) % 3  # a vertex, the middle of an edge, a quarter point of a face
    u[k == 0], u[k == 1], u[k == 2] = [1, 0, 0], [0.5, 0.5, 0], [0.25, 0.5, 0.25]
    rays = aimed((tri[at] * u[:, :, None]).sum(1), rng.normal(size=(R, 3)), np.zeros(R))
    rays[6] = bound
    v, f = ca.soup_to_mesh(tri.reshape(-1, 9))
    h, bt = orc.trace_bruteforce_minid(v, f, rays)
    assert (bt[h != 0xFFFFFFFF] == 0).mean() > 0.5
    print(f"[walk boxes] distance zero, bound {bound}, {walk}", flush=True)
    same(*traced(gpu_ctx, v, f, rays, walk), h, bt)


@pytest.mark.parametrize("walk", ["ordered", "wide"])
@pytest.mark.parametrize("n", [1, 2, 5, 600, 5000])
def test_vertices_that_are_not_finite(gpu_ctx, n, walk):
    """Triangles with vertices that are not finite can be accepted at t = NaN,
    after which nothing else is: hits and distances are those of the 4-wide walk
    with counts, which tests the leaves of a visit nearest first."""
    import torch

    soup = ca.gen_cluster_soup(n, seed=n + 3, num_clusters=4, sigma=0.1, e_min=0.05, e_max=0.2)
    rng = np.random.default_rng(n)
    bad = rng.random((n, 9)) < 0.02
    bad[0, 4] = n < 600
    soup[bad] = rng.choice(np.array([np.nan, np.inf, -np.inf], np.float32), bad.sum())
    v, f = ca.soup_to_mesh(soup)
    rays = ca.gen_random_rays(4099, seed=n)
    R = rays.shape[1]
    tv, tf, tr = cuda(v), cuda(f), cuda(rays)
    inodes, leaves = ca.node_buffers(n)
    ca.LBVHBuilder(gpu_ctx, n).perform(tv, tf, n, 10, inodes, leaves)
    print(f"[walk boxes] vertices not finite, n={n}, {walk}", flush=True)
    a, b = results(R), results(R)
    counts = torch.empty(2 * R, dtype=torch.int32, device="cuda")
    ca.trace_closest(gpu_ctx, inodes, leaves, n, tv, tf, tr, R, *a, counts, wide=True)
    ca.trace_closest(gpu_ctx, inodes, leaves, n, tv, tf, tr, R, *b, ordered=walk == "ordered", wide=walk == "wide")
    torch.cuda.synchronize()
    at, bt = a[1].cpu().numpy(), b[1].cpu().numpy()
    assert n <= 2 or np.isnan(at).any()
    np.testing.assert_array_equal(b[0].cpu().numpy(), a[0].cpu().numpy())
    np.testing.assert_array_equal(bt, at)


def chain(levels):
    """A chain of nodes, each with the next link as one child and a node over
    two pairs of leaves as the other: one entry a level for the binary walk,
    three every other level for the 4-wide one. All boxes overlap."""
    n = 4 * levels + 1
    soup = np.random.default_rng(levels).random((n, 9)).astype(np.float32)
    tri = soup.reshape(n, 3, 3)
    lo, hi = tri.min(1), tri.max(1)
    leaves, inodes = np.zeros((n, 12), np.uint32), np.zeros((n - 1, 12), np.uint32)

    def record(rec, a, b, words):
        rec[0:3], rec[4:7] = lo[a:b].min(0).view(np.uint32), hi[a:b].max(0).view(np.uint32)
        rec[8:8 + len(words)] = words

    for k in range(n):
        record(leaves[k], k, k + 1, [k])
    for k in range(levels):  # link k is node k; its tooth is node levels + 3 k over the next two
        tooth, last = levels + 3 * k, k + 1 == levels
        record(inodes[k], 4 * k, n, [0x100 if last else 0, tooth, n - 1 if last else k + 1])
        record(inodes[tooth], 4 * k, 4 * k + 4, [0, tooth + 1, tooth + 2])
        for m in range(2):
            record(inodes[tooth + 1 + m], 4 * k + 2 * m, 4 * k + 2 * m + 2, [0x101, 4 * k + 2 * m, 4 * k + 2 * m + 1])
    return soup, inodes, leaves


@pytest.mark.parametrize("levels", [20, 45, 62])
def test_deep_trees_within_the_binary_walks_stack(gpu_ctx, levels):
    import torch

    soup, inodes, leaves = chain(levels)
    v, f = ca.soup_to_mesh(soup)
    n, R = len(f), 4096
    rng = np.random.default_rng(6)
    rays = np.empty((7, R), np.float32)
    rays[0:3], rays[3:6], rays[6] = rng.random((3, R)), rng.normal(size=(3, R)), np.inf
    h, bt = orc.trace_bruteforce_minid(v, f, rays)
    tv, tf, tr, ti, tl = (cuda(a) for a in (v, f, rays, inodes, leaves))
    counts = torch.empty(2 * R, dtype=torch.int32, device="cuda")
    print(f"[walk boxes] chain of {levels} levels", flush=True)
    for walk in ({"ordered": True, "stats": counts}, {"ordered": True}):
        hit, t = results(R)
        ca.trace_closest(gpu_ctx, ti, tl, n, tv, tf, tr, R, hit, t, **walk)
        torch.cuda.synchronize()
        assert gpu_ctx.device_status() == 0
        same(hit, t, h, bt)


@pytest.mark.parametrize("child", [0xFFFFFFFF, 0xFFFFFFF0, 299, 100000])
def test_malformed_children_are_flagged_by_the_walks_with_counts(gpu_ctx, child):
    """A node whose left child does not exist: the subtree is missing, the
    binary walk flags it, and both walks return the hits of what is left."""
    import torch

    n, R = 300, 4096
    soup = ca.gen_cluster_soup(n, seed=4, num_clusters=4, sigma=0.1, e_min=0.05, e_max=0.2)
    v, f = ca.soup_to_mesh(soup)
    o = orc.lbvh_build(v, f, 10)
    nodes = np.ascontiguousarray(o["inodes"]).view(np.uint32).reshape(-1, 12).copy()
    at = int(np.flatnonzero((nodes[:, 8] & 0xFF) == 0)[1])
    lost, stack = set(), [int(nodes[at, 9])]
    while stack:
        k = stack.pop()
        for c in range(2):
            if (nodes[k, 8] >> (8 * c)) & 0xFF:
                lost.add(int(np.ascontiguousarray(o["leaves"]).view(np.uint32).reshape(-1, 12)[nodes[k, 9 + c], 8]))
            else:
                stack.append(int(nodes[k, 9 + c]))
    nodes[at, 9] = child
    kept = np.array([k for k in range(n) if k not in lost])
    assert 0 < len(kept) < n
    rays = ca.gen_random_rays(R, seed=9)
    h, bt = orc.trace_bruteforce_minid(v, f[kept], rays)
    h = np.where(h == 0xFFFFFFFF, h, kept[np.minimum(h, len(kept) - 1)].astype(np.uint32))
    tn, tl, tv, tf, tr = (cuda(a) for a in (nodes, o["leaves"], v, f, rays))
    counts = torch.empty(2 * R, dtype=torch.int32, device="cuda")
    for wide, status in ((False, 4), (True, 0)):
        print(f"[walk boxes] malformed child {child:#x}, wide={wide}", flush=True)
        hit, t = results(R)
        ca.trace_closest(gpu_ctx, tn, tl, n, tv, tf, tr, R, hit, t, counts, ordered=not wide, wide=wide)
        torch.cuda.synchronize()
        assert gpu_ctx.device_status() == status
        same(hit, t, h, bt)
