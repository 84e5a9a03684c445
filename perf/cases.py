"""The work a user of clear_amd has it do, as cases to be timed and compared.

Six kinds of work, each through the package's public entry points:

  build      one LBVH build from Face records or a triangle soup
             (LBVHBuilder.perform / perform_soup);
  segmented  one LBVH build of many scenes (LBVHBuilder.perform_segmented);
  trace      closest hits of a set of rays against a built LBVH (trace_closest:
             the reference's walk, the ordered walk, the 4-wide walk);
  frame      samples added to an accumulating image (render), optionally with
             the display step after it (post_scaling, post_tone_mapping);
  batch      samples added to the images of many scenes (render_batch);
  step       one inverse-rendering step: a differentiable render and its
             gradients (diff.render_image and its backward).

A context, as a program keeps one, is shared by all cases of the process.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import clear_amd as ca
from clear_amd import diff

DEV = "cuda"
_CTX = None


def _ctx():
    global _CTX
    if _CTX is None:
        _CTX = ca.Context(0)
    return _CTX


# ---- the cases --------------------------------------------------------------


def listed():
    return [
        # The smallest build in real use: a mesh of about 35,000 triangles at
        # 20 bits per axis, the reference's own build and its default bits.
        # Launches and short serial chains count.
        {"name": "build_35k", "kind": "build", "input": "faces", "tris": 35_003, "bits": 20},
        # A detailed scene's mesh (the outdoor scene's size) at the same bits.
        {"name": "build_3m", "kind": "build", "input": "faces", "tris": 3_117_058, "bits": 20},
        # The largest build: 2^24 soup triangles with 30-bit codes.
        {"name": "build_16m", "kind": "build", "input": "soup", "tris": 16_777_216, "bits": 10},
        # Many scenes in one build, from a thousand to half a million triangles.
        {"name": "segmented_64", "kind": "segmented", "scenes": 64, "least": 1_007, "most": 499_388},
        # A small visibility query against a small mesh: latency and set-up count.
        {"name": "trace_pick", "kind": "trace", "walk": "ordered", "tris": 20_480, "rays": 4_099},
        # The drop-in closest hit (the default of trace_closest) on a medium mesh.
        {"name": "trace_reference", "kind": "trace", "walk": "reference", "tris": 1_000_003, "rays": 524_309},
        # The largest query: 2^22 incoherent rays against 2^24 triangles.
        {"name": "trace_wide", "kind": "trace", "walk": "wide", "tris": 16_777_216, "rays": 4_194_304},
        # A whole render: the 3.1 M-triangle outdoor scene at 1080p.
        {"name": "render_1080p", "kind": "frame", "scene": "outdoor", "detail": 1024, "width": 1920, "height": 1080,
         "spp": 32, "depth": 8, "mode": "megakernel", "display": False},
        # One pass of a progressive preview: one sample per pixel of the same
        # scene, then the image scaled and tone-mapped for display. The scene's
        # set-up inside the call counts.
        {"name": "preview_720p", "kind": "frame", "scene": "outdoor", "detail": 1024, "width": 1280, "height": 720,
         "spp": 1, "depth": 8, "mode": "megakernel", "display": True},
        # The queue-driven renderer on the scene with every material kind,
        # textures, alpha cut-outs and an environment.
        {"name": "wavefront_showcase", "kind": "frame", "scene": "showcase", "detail": 0, "width": 640, "height": 360,
         "spp": 16, "depth": 8, "mode": "wavefront", "display": False},
        # Many small scenes lit by area lights, rendered together.
        {"name": "batch_32", "kind": "batch", "scenes": 32, "least": 1_000, "most": 200_000, "size": 128, "spp": 32,
         "depth": 5, "mode": "megakernel"},
        # An inverse-rendering step: forward image and gradients of 64 materials.
        {"name": "step_512", "kind": "step", "width": 512, "height": 512, "spp": 8, "depth": 5},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["build", "segmented", "trace", "frame", "batch", "step"])
    if kind == "build":
        soup = rng.random() < 0.5
        return {"kind": kind, "input": "soup" if soup else "faces", "bits": rng.choice([10, 20]),
                "tris": _log(rng, 1_000, 16_777_216 if soup else 4_000_000)}
    if kind == "segmented":
        most = _log(rng, 2_000, 500_000)
        return {"kind": kind, "scenes": min(_log(rng, 2, 256), 40_000_000 // most), "least": _log(rng, 1_000, 2_000),
                "most": most}
    if kind == "trace":
        walk = rng.choice(["reference", "ordered", "wide"])
        small = walk == "reference"
        return {"kind": kind, "walk": walk, "tris": _log(rng, 1_000, 2_000_000 if small else 16_777_216),
                "rays": _log(rng, 1_000, 600_000 if small else 4_194_304)}
    if kind == "frame":
        scene = rng.choice(["outdoor", "showcase", "cornell"])
        w, h = _log(rng, 96, 1920), _log(rng, 64, 1080)
        return {"kind": kind, "scene": scene, "detail": _log(rng, 128, 1024) if scene == "outdoor" else 0,
                "width": w, "height": h, "spp": min(_log(rng, 1, 32), max(1, 12_000_000 // (w * h))),
                "depth": rng.randint(3, 10), "mode": rng.choice(["megakernel", "wavefront"]),
                "display": rng.random() < 0.5}
    if kind == "batch":
        return {"kind": kind, "scenes": rng.randint(2, 32), "least": 1_000, "most": _log(rng, 2_000, 200_000),
                "size": _log(rng, 48, 160), "spp": _log(rng, 2, 32), "depth": rng.randint(3, 8),
                "mode": rng.choice(["megakernel", "wavefront"])}
    return {"kind": kind, "width": _log(rng, 64, 512), "height": _log(rng, 64, 512), "spp": _log(rng, 2, 8),
            "depth": rng.randint(3, 8)}


# ---- inputs -----------------------------------------------------------------


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _unit(n, g):
    """n directions uniform on the sphere."""
    d = torch.randn(n, 3, device=DEV, generator=g)
    return d / d.norm(dim=1, keepdim=True).clamp_min(1e-12)


def _soup(counts, g):
    """Gaussian-cluster soups (64 clusters of sigma 0.02 in the unit cube per
    scene, edges 1e-3..1e-2), float32 [sum(counts), 9]."""
    n, s = sum(counts), len(counts)
    scene = torch.repeat_interleave(torch.arange(s, device=DEV), torch.tensor(counts, device=DEV))
    centres = torch.rand(s * 64, 3, device=DEV, generator=g)
    c = centres[scene * 64 + torch.randint(64, (n,), device=DEV, generator=g)]
    c += 0.02 * torch.randn(n, 3, device=DEV, generator=g)
    e1 = _unit(n, g) * (1e-3 + 9e-3 * torch.rand(n, 1, device=DEV, generator=g))
    e2 = _unit(n, g) * (1e-3 + 9e-3 * torch.rand(n, 1, device=DEV, generator=g))
    v0 = c - (e1 + e2) / 3
    return torch.cat([v0, v0 + e1, v0 + e2], dim=1).contiguous()


def _mesh(soup):
    """The soup as 16-byte vertices and 56-byte Face records (three vertex
    indices, every other attribute absent)."""
    n = soup.shape[0]
    verts = torch.zeros(3 * n, 4, device=DEV)
    verts[:, :3] = soup.view(3 * n, 3)
    faces = torch.full((n, 14), -1, dtype=torch.int32, device=DEV)
    faces[:, :3] = torch.arange(3 * n, dtype=torch.int32, device=DEV).view(n, 3)
    return verts, faces


def _counts(case):
    """Triangles per scene: geometric from `least` to `most`, in a mixed order."""
    s, lo, hi = case["scenes"], case["least"], case["most"]
    sizes = [int(round(lo * (hi / lo) ** (k / max(s - 1, 1)))) for k in range(s)]
    step = next(k for k in (7, 11, 13, 17, 19, 23) if math.gcd(k, s) == 1)
    return [sizes[(k * step) % s] for k in range(s)]


def _states(pixels, g):
    """xorshift128 states, four nonzero words per pixel."""
    return torch.randint(1, 2**31 - 1, (4 * pixels,), device=DEV, generator=g, dtype=torch.int32)


def prepare(case, seed):
    g, ctx, kind = _gen(seed), _ctx(), case["kind"]
    st = {"case": case}
    if kind == "build":
        n = case["tris"]
        st["soup"] = _soup([n], g)
        if case["input"] == "faces":
            st["verts"], st["faces"] = _mesh(st.pop("soup"))
        st["nodes"] = ca.node_buffers(n)
        st["builder"] = ca.LBVHBuilder(ctx, n, case["bits"])
    elif kind == "segmented":
        counts = _counts(case)
        total = sum(counts)
        st["soup"] = _soup(counts, g)
        st["offsets"] = torch.from_numpy(np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)).to(DEV)
        st["total"] = total
        st["nodes"] = (torch.zeros(max(total - len(counts), 1) * ca.INODE_BYTES, dtype=torch.uint8, device=DEV),
                       torch.zeros(total * ca.LEAF_BYTES, dtype=torch.uint8, device=DEV))
        st["builder"] = ca.LBVHBuilder(ctx, 0, 10)
    elif kind == "trace":
        n, r = case["tris"], case["rays"]
        soup = _soup([n], g)
        st["verts"], st["faces"] = _mesh(soup)
        st["nodes"] = ca.node_buffers(n)
        ca.LBVHBuilder(ctx, n, 10).perform_soup(soup, n, 10, *st["nodes"])
        rays = torch.empty(7, r, device=DEV)
        rays[:3] = torch.rand(3, r, device=DEV, generator=g)
        rays[3:6] = _unit(r, g).t()
        rays[6] = math.inf
        st["rays"] = rays
        st["hit"] = torch.empty(r, dtype=torch.int32, device=DEV)
        st["t"] = torch.empty(r, device=DEV)
    elif kind == "frame":
        w, h = case["width"], case["height"]
        scene = {"outdoor": ca.SCENE_TERRAIN, "showcase": ca.SCENE_SHOWCASE, "cornell": ca.SCENE_CORNELL}[case["scene"]]
        host = ca.HostScene(scene, w, h, detail=case["detail"], seed=seed % 1000 + 1)
        st["scene"] = ca.DeviceScene(ctx, host, bits=20)
        st["states"] = _states(w * h, g)
        st["pixels"] = torch.zeros(4 * w * h, device=DEV)
        if case["display"]:
            st["scaled"] = torch.zeros(4 * w * h, device=DEV)
            st["bgr"] = torch.zeros(ca.bmp_row_bytes(w) * h, dtype=torch.uint8, device=DEV)
    elif kind == "batch":
        s = case["size"]
        hosts = [ca.HostScene(ca.SCENE_CLUSTERS, s, s, seed=(seed * 101 + k) % 100_000 + 1, num_triangles=n)
                 for k, n in enumerate(_counts(case))]
        st["batch"] = ca.SceneBatch(ctx, hosts)
        st["states"] = _states(len(hosts) * s * s, g)
        st["pixels"] = torch.zeros(4 * len(hosts) * s * s, device=DEV)
    else:
        host = ca.HostScene(ca.SCENE_ADJOINT, case["width"], case["height"], seed=seed % 1000 + 1)
        r = diff.DiffRenderer(ctx, host, case["spp"], case["depth"])
        st["renderer"] = r
        st["states"] = _states(r.width * r.height, g)
        hidden = r.params()
        st["target"] = r.render(st["states"])  # what the hidden parameters look like
        st["params"] = [p.clone() for p in hidden]
        st["params"][0].fill_(0.5)
        st["params"][1].fill_(0.3)
        for p in st["params"]:
            p.requires_grad_(True)
    return st


# ---- one pass ---------------------------------------------------------------

_MODE = {"megakernel": ca.RENDER_MEGAKERNEL, "wavefront": ca.RENDER_WAVEFRONT}


def run(st):
    case, ctx = st["case"], _ctx()
    kind = case["kind"]
    if kind == "build":
        if case["input"] == "soup":
            st["builder"].perform_soup(st["soup"], case["tris"], case["bits"], *st["nodes"])
        else:
            st["builder"].perform(st["verts"], st["faces"], case["tris"], case["bits"], *st["nodes"])
        return {"inodes": st["nodes"][0], "leaves": st["nodes"][1]}
    if kind == "segmented":
        st["builder"].perform_segmented(st["soup"], st["offsets"], st["total"], 10, *st["nodes"])
        return {"inodes": st["nodes"][0], "leaves": st["nodes"][1]}
    if kind == "trace":
        ca.trace_closest(ctx, *st["nodes"], case["tris"], st["verts"], st["faces"], st["rays"], case["rays"],
                         st["hit"], st["t"], ordered=case["walk"] == "ordered", wide=case["walk"] == "wide")
        return {"face": st["hit"], "t": st["t"]}
    if kind == "frame":
        ca.render(ctx, st["scene"], case["spp"], case["depth"], st["states"], st["pixels"], mode=_MODE[case["mode"]])
        out = {"pixels": st["pixels"], "states": st["states"]}
        if case["display"]:
            w, h = case["width"], case["height"]
            ca.post_scaling(ctx, w, h, case["spp"], st["pixels"], st["scaled"])
            ca.post_tone_mapping(ctx, w, h, ca.bmp_row_bytes(w), st["scaled"], st["bgr"])
            out["bgr"] = st["bgr"]
        return out
    if kind == "batch":
        ca.render_batch(ctx, st["batch"], case["spp"], case["depth"], st["states"], st["pixels"],
                        mode=_MODE[case["mode"]])
        return {"pixels": st["pixels"], "states": st["states"]}
    image = diff.render_image(*st["params"], st["renderer"], st["states"])
    loss = (image - st["target"]).square().mean()
    grads = torch.autograd.grad(loss, st["params"])
    return {"image": image.detach(), "albedo": grads[0], "roughness": grads[1], "emission": grads[2]}


# ---- what a pass cannot do without ------------------------------------------


def _walk(tris):
    """Flops and bytes of one ray that visits one node a level (two box tests
    of 20 flops, 48 bytes of record) and tests one triangle."""
    levels = math.log2(max(tris, 2))
    return 40 * levels + 51, 48 * levels + 48


def work(case):
    kind = case["kind"]
    if kind in ("build", "segmented"):
        n = case["tris"] if kind == "build" else sum(_counts(case))
        # Triangles in (a face's 12 bytes of indices and three 16-byte
        # vertices, or 36 bytes of soup), two 48-byte records out; about 60
        # operations a triangle (its box, its code, one merge).
        return {"bytes": n * ((60 if case.get("input") == "faces" else 36) + 96), "flops": 60 * n}
    if kind == "trace":
        f, b = _walk(case["tris"])
        # Rays in (28 bytes), hits out (8), and the nodes and triangles that
        # the rays reach, each read once.
        return {"bytes": case["rays"] * 36 + min(case["rays"] * b, case["tris"] * 156), "flops": case["rays"] * f}
    if kind == "step":
        pixels, tris, spp, passes = case["width"] * case["height"], 200_014, case["spp"], 2
    elif kind == "batch":
        pixels, tris, spp, passes = case["scenes"] * case["size"] ** 2, case["most"], case["spp"], 1
    else:
        tris = {"outdoor": 2 * case["detail"] ** 2 + 1_024_000, "showcase": 5_134, "cornell": 20_494}[case["scene"]]
        pixels, spp, passes = case["width"] * case["height"], case["spp"], 1
    # A sample casts at least a camera, a shadow and a bounce ray and shades
    # twice (about 300 operations each); states and pixels go in and out.
    rays = 3 * pixels * spp
    f, b = _walk(tris)
    return {"bytes": passes * (pixels * 64 + min(rays * b, tris * 156)), "flops": passes * (rays * f + 600 * pixels * spp)}


# Builds and traces are defined bit for bit (the reference's nodes; the
# closest (t, face) of the triangle test's own arithmetic). So are a render's
# samples and random states, but an image depends on the order in which its
# samples are added: half the samples in each of two calls instead of one call
# changes it by up to 9.2e-8 (2-norm) and 4.9e-7 (largest), and no state. A
# byte of the displayed image may then round the other way. Gradients are
# summed with atomics: two runs differ by up to 6.9e-7 and 2.0e-6.
def tolerance(case):
    if case["kind"] in ("build", "segmented", "trace"):
        return "exact"
    if case["kind"] == "step":
        return {"rel": 2.8e-6, "max": 8e-6}
    return {"rel": 3.7e-7, "max": 2e-6, "differ": 1e-5 if case.get("display") else 0.0}


def exact(case, seed):
    """Hit distances by brute force over all triangles in 64 bits. Path traced
    images and gradients have no such value in reasonable time, and builds
    return whole records."""
    if case["kind"] != "trace" or case["tris"] * case["rays"] > 2**29:
        return None
    st = prepare(case, seed)
    torch.cuda.synchronize()
    v = st["verts"][:, :3].double().view(-1, 3, 3)
    p0, e1, e2 = v[:, 0], v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]
    rays = st["rays"].double()
    out = []
    chunk = max(1, 2**23 // case["tris"])
    for a in range(0, case["rays"], chunk):
        o, d = rays[:3, a:a + chunk].t(), rays[3:6, a:a + chunk].t()
        p = torch.linalg.cross(d[:, None, :], e2[None])
        det = (e1[None] * p).sum(-1)
        s = o[:, None, :] - p0[None]
        b1 = (s * p).sum(-1) / det
        q = torch.linalg.cross(s, e1[None].expand_as(s))
        b2 = (d[:, None, :] * q).sum(-1) / det
        t = (e2[None] * q).sum(-1) / det
        ok = (det.abs() >= 1e-6) & (b1 >= 0) & (b1 <= 1) & (b2 >= 0) & (b1 + b2 <= 1) & (t >= 0)
        out.append(torch.where(ok, t, math.inf).amin(1))
    return {"face": None, "t": torch.cat(out)}
