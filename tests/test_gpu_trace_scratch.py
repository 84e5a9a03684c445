"""The memory of clr_trace_closest's walk of many rays: it grows without
touching what captured calls use, without ending captures of other streams,
and calls on several streams may share it. The blocks of the other walks stay
while a captured call refers to them."""
import numpy as np
import pytest

import clear_amd as ca
from test_gpu_trace_nocounts import cuda, mesh, results

pytestmark = pytest.mark.gpu


class Scene:
    def __init__(self, ctx, n, rays, seed):
        v, f = mesh(n)
        self.n, self.R = n, rays
        self.v, self.f, self.rays = cuda(v), cuda(f), cuda(ca.gen_random_rays(rays, seed=seed))
        self.nodes = ca.node_buffers(n)
        ca.LBVHBuilder(ctx, n).perform(self.v, self.f, n, 10, *self.nodes)
        self.hit, self.t = results(rays)

    def trace(self, ctx, stream=None, **walk):
        ca.trace_closest(ctx, *self.nodes, self.n, self.v, self.f, self.rays, self.R, self.hit, self.t, stream=stream,
                         **walk)

    def clear(self):
        self.hit.fill_(-7)
        self.t.fill_(-7.0)

    def out(self):
        import torch

        torch.cuda.synchronize()
        return self.hit.cpu().numpy(), self.t.cpu().numpy()


def equal(a, b):
    np.testing.assert_array_equal(a[0], b[0])
    np.testing.assert_array_equal(a[1], b[1])


@pytest.fixture
def ctx(gpu_ctx):  # a fresh one; the session's brings torch up first
    c = ca.Context(0)
    yield c
    c.close()


def by_parts(ctx, s):
    """The scene's hits from calls of too few rays for the layout."""
    import torch

    hit, t = np.empty(s.R, np.int32), np.empty(s.R, np.float32)
    rays = s.rays.cpu().numpy().view(np.float32).reshape(7, s.R)
    for a in range(0, s.R, 9000):
        part = cuda(rays[:, a:a + 9000])
        h, d = results(min(9000, s.R - a))
        ca.trace_closest(ctx, *s.nodes, s.n, s.v, s.f, part, len(h), h, d)
        torch.cuda.synchronize()
        hit[a:a + 9000], t[a:a + 9000] = h.cpu().numpy(), d.cpu().numpy()
    return hit, t


@pytest.mark.parametrize("larger", ["reference", "ordered", "wide"])
@pytest.mark.parametrize("walk", ["ordered", "wide"])
def test_captured_traces_outlive_larger_ones(ctx, walk, larger):
    import torch

    small, large = Scene(ctx, 5000, 20000, 1), Scene(ctx, 60000, 1 << 17, 2)
    small.trace(ctx, **{walk: True})
    want = small.out()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, capture_error_mode="thread_local"):
        small.trace(ctx, **{walk: True})
    for k in range(3):
        print(f"[trace scratch] {walk}, then {larger}: replay {k}", flush=True)
        large.trace(ctx, **({} if larger == "reference" else {larger: True}))
        small.clear()
        torch.cuda.synchronize()
        g.replay()
        equal(small.out(), want)
    if larger == "reference":
        equal(large.out(), by_parts(ctx, large))
    else:  # the same hits from a context with nothing captured
        got = large.out()
        fresh = ca.Context(0)
        large.trace(fresh, **{larger: True})
        equal(large.out(), got)
        fresh.close()
    assert ctx.device_status() == 0


def test_captured_render_outlives_a_larger_scene(ctx):
    import torch

    W, H, spp, depth = 48, 40, 2, 4
    host, big = ca.HostScene(ca.SCENE_CORNELL, W, H, detail=3), Scene(ctx, 60000, 1 << 15, 7)
    ds = ca.DeviceScene(ctx, host)
    states, pixels = ca.new_image(W, H)

    def frame():
        ca.seed_pixel_states(ctx, W, H, states)
        pixels.zero_()
        ca.render(ctx, ds, spp, depth, states, pixels)

    frame()
    torch.cuda.synchronize()
    want = pixels.cpu().numpy()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, capture_error_mode="thread_local"):
        frame()
    for k in range(3):
        print(f"[trace scratch] render replay {k}", flush=True)
        big.trace(ctx, wide=True)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(pixels.cpu().numpy(), want)
    assert ctx.device_status() == 0


def test_streams_of_one_context(ctx):
    import torch

    scenes = [Scene(ctx, 5000, 1 << 14, 3), Scene(ctx, 30000, 1 << 15, 4), Scene(ctx, 60000, 1 << 16, 5)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in scenes]
    for k in range(4):  # the first round grows the block twice while it is in use
        print(f"[trace scratch] streams, round {k}", flush=True)
        for s in scenes:
            s.clear()
        torch.cuda.synchronize()
        for s, stream in zip(scenes, streams):
            s.trace(ctx, stream=stream)
        for s in scenes:
            equal(s.out(), by_parts(ctx, s))
    assert ctx.device_status() == 0


def test_while_another_stream_is_captured(ctx):
    import torch

    s = Scene(ctx, 5000, 1 << 14, 6)
    want = by_parts(ctx, s)
    s.clear()
    x = torch.zeros(1000, device="cuda")
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    print("[trace scratch] beside a capture", flush=True)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, capture_error_mode="global"):
        x += 1.0
        s.trace(ctx, stream=side)
    for _ in range(3):
        g.replay()
    torch.cuda.synchronize()
    assert (x == 3.0).all()
    equal(s.out(), want)
    assert ctx.device_status() == 0
