// Closest-hit traversal of the LBVH for gfx950.
//
// Replaces rayIntersection (OpenCL_PathTracer/OpenCL/bvh_traversal.cl:182-215)
// with the same visiting order and tests, so hits agree bit for bit
// (k_trace_closest; many rays: k_trace_reference):
//   * pop a node, test its own box (rayAABBIntersection, :160-179) against the
//     current t; for child 0 then child 1: push an internal child, or test the
//     leaf box and then the triangle (Moller-Trumbore, :54-108);
//   * a triangle replaces the hit when tt <= t (ties go to the last tested).
// Layout choices for the hardware: one ray per lane, SoA ray planes read
// coalesced, the 64-entry stack lives in LDS as [depth][lane] (16 KiB per
// wave, conflict-free at equal depth) instead of per-lane scratch, and node /
// vertex records are fetched as 16-B vectors.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <string>

#include "internal.h"
#include "traverse_device.h"

namespace clr {
namespace {

constexpr int kTraceBlock = 64;

template <bool STATS>
__global__ __launch_bounds__(kTraceBlock) void k_trace_closest(
    const clr_lbvh_inode* __restrict__ inodes, const clr_lbvh_leaf* __restrict__ leaves,
    uint32_t n, const clr_float3* __restrict__ verts, const clr_face* __restrict__ faces,
    const float* __restrict__ rays, uint32_t numRays, uint32_t* __restrict__ hitFace,
    float* __restrict__ hitT, uint32_t* __restrict__ stats, uint32_t* __restrict__ status,
    const float4* __restrict__ bvh) {
    __shared__ uint32_t s_stack[dev::kStackDepth * kTraceBlock];
    const uint32_t r = blockIdx.x * kTraceBlock + threadIdx.x;
    if (r >= numRays) return;
    const size_t R = numRays;
    dev::V3 o = {rays[r], rays[R + r], rays[2 * R + r]};
    dev::V3 d = {rays[3 * R + r], rays[4 * R + r], rays[5 * R + r]};
    float t = rays[6 * R + r];
    dev::GeomScene g{inodes, leaves, n, verts, faces};
    g.bvh = bvh;
    dev::TraceStats st{0u, 0u};
    bool over = false;
    uint32_t best = dev::closestHit<STATS>(g, o, d, t, dev::LdsStack{s_stack + threadIdx.x, kTraceBlock},
                                           st, nullptr, nullptr, dev::NoAlpha(), &over);
    if (over) atomicOr(status, kStatusStackOverflow);
    const bool hit = best != kEmpty && !isinf(t);
    hitFace[r] = hit ? best : kEmpty;
    hitT[r] = t;
    if constexpr (STATS) {
        stats[2 * (size_t)r] = st.visits;
        stats[2 * (size_t)r + 1] = st.tests;
    }
}

// Triangle record (see GeomScene) of a face at `o`: p0 | tag, the two edges.
__device__ __forceinline__ void storeTri(const clr_float3* __restrict__ verts, const clr_face& f, uint32_t tag,
                                         float4* __restrict__ o) {
    const dev::V3 p0 = dev::loadV3(verts, f.p0), p1 = dev::loadV3(verts, f.p1), p2 = dev::loadV3(verts, f.p2);
    const dev::V3 e1 = p1 - p0, e2 = p2 - p0;
    o[0] = make_float4(p0.x, p0.y, p0.z, __uint_as_float(tag));
    o[1] = make_float4(e1.x, e1.y, e1.z, 0.0f);
    o[2] = make_float4(e2.x, e2.y, e2.z, 0.0f);
}
// Face i's, tagged with its alpha flag.
__device__ __forceinline__ void storeFace(const clr_float3* __restrict__ verts, const clr_face* __restrict__ faces,
                                          uint32_t i, float4* __restrict__ atris) {
    const clr_face& f = faces[i];
    storeTri(verts, f, f.uv0 != dev::kNone && f.alphaTexPtr != dev::kNone ? 1u : 0u, atris + 3 * (size_t)i);
}

// Traversal layout (see GeomScene): node i gets both children's boxes and
// references (unless anodes is null), face i its triangle record. BY_LEAF
// (ReferenceWalk): leaf children and triangle records by leaf, tagged with the
// face.
template <bool BY_LEAF>
__global__ void k_accel_build(const clr_lbvh_inode* __restrict__ inodes, const clr_lbvh_leaf* __restrict__ leaves,
                              uint32_t n, const clr_float3* __restrict__ verts, const clr_face* __restrict__ faces,
                              float4* __restrict__ anodes, float4* __restrict__ atris) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (anodes && i + 1 < n) {
        const uint4 c = reinterpret_cast<const uint4*>(inodes + i)[2];
        float4 box[2][2];
        uint32_t ref[2];
        for (int k = 0; k < 2; ++k) {
            const bool leaf = ((c.x >> (8 * k)) & 0xFFu) != 0;
            const uint32_t ci = k ? c.z : c.y;
            // Malformed nodes: an empty box, which the walks may still enter
            // (slabEnter admits it), and as its reference a leaf of a face that
            // is not there, which they flag.
            if (leaf ? ci >= n : ci >= n - 1) {
                box[k][0] = make_float4(INFINITY, INFINITY, INFINITY, 0.0f);
                box[k][1] = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.0f);
                ref[k] = dev::kNone;
                continue;
            }
            const float4* p = leaf ? reinterpret_cast<const float4*>(leaves + ci)
                                   : reinterpret_cast<const float4*>(inodes + ci);
            box[k][0] = p[0];
            box[k][1] = p[1];
            ref[k] = !leaf ? ci : (BY_LEAF ? ci : leaves[ci].objIdx) | dev::kLeafRef;
        }
        float4* o = anodes + 4 * (size_t)i;
        o[0] = make_float4(box[0][0].x, box[0][0].y, box[0][0].z, __uint_as_float(ref[0]));
        o[1] = make_float4(box[0][1].x, box[0][1].y, box[0][1].z, __uint_as_float(ref[1]));
        o[2] = make_float4(box[1][0].x, box[1][0].y, box[1][0].z, 0.0f);
        o[3] = make_float4(box[1][1].x, box[1][1].y, box[1][1].z, 0.0f);
    }
    if (i >= n) return;
    if constexpr (BY_LEAF) {
        // A leaf that nothing refers to may hold anything: no face has the bit
        // of leaf references, and its record (no edges) is never hit.
        const uint32_t face = leaves[i].objIdx;
        float4* o = atris + 3 * (size_t)i;
        if (face & dev::kLeafRef) o[0] = o[1] = o[2] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        else storeTri(verts, faces[face], face, o);
    } else {
        storeFace(verts, faces, i, atris);
    }
}

// Traversal layout of a CPU midpoint BVH, indexed by node number: internal
// node i (children[1] != 0xFFFFFFFF) gets both children's boxes, a leaf child
// as its face | kLeafRef, an internal child as its node number; leaf node
// slots stay unused. Faces as in k_accel_build.
__global__ void k_accel_build_bvh(const float4* __restrict__ bvh, uint32_t n, const clr_float3* __restrict__ verts,
                                  const clr_face* __restrict__ faces, float4* __restrict__ anodes,
                                  float4* __restrict__ atris) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t numNodes = 2 * n - 1;
    if (anodes && i < numNodes) {
        const uint2 c = *reinterpret_cast<const uint2*>(bvh + 3 * (size_t)i + 2);
        if (c.y != kEmpty && c.x < numNodes && c.y < numNodes) {
            float4 box[2][2];
            uint32_t ref[2];
            for (int k = 0; k < 2; ++k) {
                const uint32_t ci = k ? c.y : c.x;
                const float4* p = bvh + 3 * (size_t)ci;
                box[k][0] = p[0];
                box[k][1] = p[1];
                const uint2 cc = *reinterpret_cast<const uint2*>(p + 2);
                ref[k] = cc.y == kEmpty ? (cc.x | dev::kLeafRef) : ci;
            }
            float4* o = anodes + 4 * (size_t)i;
            o[0] = make_float4(box[0][0].x, box[0][0].y, box[0][0].z, __uint_as_float(ref[0]));
            o[1] = make_float4(box[0][1].x, box[0][1].y, box[0][1].z, __uint_as_float(ref[1]));
            o[2] = make_float4(box[1][0].x, box[1][0].y, box[1][0].z, 0.0f);
            o[3] = make_float4(box[1][1].x, box[1][1].y, box[1][1].z, 0.0f);
        }
    }
    if (i < n) storeFace(verts, faces, i, atris);
}

// 4-wide records (GeomScene::wnodes) of the LBVH: record i holds the
// children of each internal child of node i, or a leaf child itself, in slot
// order left.left, left.right, right.left, right.right (a leaf child takes
// the first of its two slots; the other stays empty).
struct WideSlots {
    float lo[3][4], hi[3][4];
    uint32_t ref[4];
    __device__ __forceinline__ void clear() {
        for (int c = 0; c < 4; ++c) {
            for (int a = 0; a < 3; ++a) {
                lo[a][c] = INFINITY;
                hi[a][c] = -INFINITY;
            }
            ref[c] = dev::kNone;
        }
    }
    __device__ __forceinline__ void put(int c, float4 l, float4 h, uint32_t r, uint32_t n) {
        if ((r & dev::kLeafRef) && (r & ~dev::kLeafRef) >= n) return;  // a face that is not there
        lo[0][c] = l.x;
        lo[1][c] = l.y;
        lo[2][c] = l.z;
        hi[0][c] = h.x;
        hi[1][c] = h.y;
        hi[2][c] = h.z;
        ref[c] = r;
    }
    __device__ __forceinline__ void store(float4* o) const {
        for (int a = 0; a < 3; ++a) {
            o[a] = make_float4(lo[a][0], lo[a][1], lo[a][2], lo[a][3]);
            o[3 + a] = make_float4(hi[a][0], hi[a][1], hi[a][2], hi[a][3]);
        }
        o[6] = make_float4(__uint_as_float(ref[0]), __uint_as_float(ref[1]), __uint_as_float(ref[2]),
                           __uint_as_float(ref[3]));
        o[7] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
};

__global__ void k_accel_wide(const clr_lbvh_inode* __restrict__ inodes, const clr_lbvh_leaf* __restrict__ leaves,
                             uint32_t n, float4* __restrict__ records) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    WideSlots w;
    w.clear();
    if (n == 1 && i == 0) {  // a tree of one leaf: a record that holds it
        const float4* p = reinterpret_cast<const float4*>(leaves);
        w.put(0, p[0], p[1], leaves[0].objIdx | dev::kLeafRef, n);
        w.store(records);
        return;
    }
    if (i + 1 >= n) return;
    const uint4 c = reinterpret_cast<const uint4*>(inodes + i)[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const bool leaf = ((c.x >> (8 * k)) & 0xFFu) != 0;
        const uint32_t ci = k ? c.z : c.y;
        if (leaf) {
            if (ci >= n) continue;  // malformed nodes leave the slot empty
            const float4* p = reinterpret_cast<const float4*>(leaves + ci);
            w.put(2 * k, p[0], p[1], leaves[ci].objIdx | dev::kLeafRef, n);
            continue;
        }
        if (ci >= n - 1) continue;
        const uint4 cc = reinterpret_cast<const uint4*>(inodes + ci)[2];
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            const bool gl = ((cc.x >> (8 * m)) & 0xFFu) != 0;
            const uint32_t gi = m ? cc.z : cc.y;
            if (gl ? gi >= n : gi >= n - 1) continue;
            const float4* p = gl ? reinterpret_cast<const float4*>(leaves + gi)
                                 : reinterpret_cast<const float4*>(inodes + gi);
            w.put(2 * k + m, p[0], p[1], gl ? (leaves[gi].objIdx | dev::kLeafRef) : gi, n);
        }
    }
    w.store(records + 8 * (size_t)i);
}

// The same records for a CPU midpoint BVH, by node number (leaf node slots
// stay unused).
__global__ void k_accel_wide_bvh(const float4* __restrict__ bvh, uint32_t n, float4* __restrict__ records) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t numNodes = 2 * n - 1;
    if (i >= numNodes) return;
    const uint2 c = *reinterpret_cast<const uint2*>(bvh + 3 * (size_t)i + 2);
    WideSlots w;
    w.clear();
    if (n == 1 && c.y == kEmpty) {  // a tree of one leaf: a record that holds it
        w.put(0, bvh[0], bvh[1], c.x | dev::kLeafRef, n);
        w.store(records);
        return;
    }
    if (c.y == kEmpty || c.x >= numNodes || c.y >= numNodes) return;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const uint32_t ci = k ? c.y : c.x;
        const float4* p = bvh + 3 * (size_t)ci;
        const uint2 cc = *reinterpret_cast<const uint2*>(p + 2);
        if (cc.y == kEmpty) {  // a leaf: its face
            w.put(2 * k, p[0], p[1], cc.x | dev::kLeafRef, n);
            continue;
        }
        if (cc.x >= numNodes || cc.y >= numNodes) continue;  // malformed nodes leave the slots empty
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            const uint32_t gi = m ? cc.y : cc.x;
            const float4* q = bvh + 3 * (size_t)gi;
            const uint2 gc = *reinterpret_cast<const uint2*>(q + 2);
            w.put(2 * k + m, q[0], q[1], gc.y == kEmpty ? (gc.x | dev::kLeafRef) : gi, n);
        }
    }
    w.store(records + 8 * (size_t)i);
}

// Trace with the ordered traversal, grid-stride over the rays with a fixed
// grid (waves per CU x CUs). Each lane walks two rays at once, stepping them in
// turn, so one ray's node fetch is in flight while the other's boxes and
// triangles are tested (the walk is bound by dependent load latency). Each
// walker's stack keeps kOrdHalf slots in LDS ([slot][lane]) and the rest in
// its part of `spill`.
constexpr int kOrdLds = 32;
constexpr int kOrdBlock = 128;
constexpr int kOrdHalf = kOrdLds / 2;

// Walkers w0 and w1 over this lane's rays gid, gid + lanes, ...; done(w, r)
// stores ray r's result.
template <class W, class Done>
__device__ __forceinline__ void traceTwo(W& w0, W& w1, const float* __restrict__ rays, uint32_t numRays, uint32_t gid,
                                         uint32_t lanes, uint32_t* __restrict__ status, const Done& done) {
    const size_t R = numRays;
    bool over = false;
    uint32_t next = gid, r0 = kEmpty, r1 = kEmpty;
    auto start = [&](W& w, uint32_t& r) {
        if (next < numRays) {
            r = next;
            next += lanes;
            const dev::V3 o = {rays[r], rays[R + r], rays[2 * R + r]};
            const dev::V3 d = {rays[3 * R + r], rays[4 * R + r], rays[5 * R + r]};
            w.begin(o, d, rays[6 * R + r]);
        } else {
            r = kEmpty;
        }
    };
    auto finish = [&](const W& w, uint32_t r) {
        if (w.over()) over = true;
        done(w, r);
    };
    start(w0, r0);
    start(w1, r1);
    while (r0 != kEmpty || r1 != kEmpty) {
        if (r0 != kEmpty) {
            if (!w0.done()) w0.step();
            if (w0.done()) {
                finish(w0, r0);
                start(w0, r0);
            }
        }
        if (r1 != kEmpty) {
            if (!w1.done()) w1.step();
            if (w1.done()) {
                finish(w1, r1);
                start(w1, r1);
            }
        }
    }
    if (over) atomicOr(status, kStatusStackOverflow);
}

// The reference's walk over the traversal layout. A wave takes as long as its
// longest rays (thousands of visits where k_trace_closest's rays cross a whole
// scene before they meet anything), so a visit's own latency counts: one ray
// per lane, both children's records requested before their boxes are tested.
// 1,000,003 triangles, 524,309 rays: 8.07 ms with k_trace_closest, 5.61 with two
// rays per lane and no early requests, 4.0 now; with 2,000,000
// triangles and 1,000,000 rays 21.0 and 7.1 (first and last). A third
// request for the stack's top was slower (3.7 -> 4.2 ms): a visit is bound by
// its instructions.
constexpr int kReferencePairs = kOrdHalf;  // stack entries in LDS
template <bool STATS>
__global__ __launch_bounds__(kOrdBlock) void k_trace_reference(
    dev::GeomScene g, const float* __restrict__ rays, uint32_t numRays, uint32_t* __restrict__ hitFace,
    float* __restrict__ hitT, uint32_t* __restrict__ stats, uint32_t* __restrict__ status,
    uint32_t* __restrict__ spill) {
    using S = dev::PairStack<kReferencePairs, dev::kStackDepth>;
    __shared__ uint2 s_stack[kReferencePairs * kOrdBlock];
    const uint32_t gid = blockIdx.x * kOrdBlock + threadIdx.x;
    const uint32_t lanes = gridDim.x * kOrdBlock;
    const S stk{s_stack + threadIdx.x, kOrdBlock, reinterpret_cast<uint2*>(spill) + gid, lanes};
    dev::ReferenceWalk<STATS, S> w(g, stk);
    const size_t R = numRays;
    bool over = false;
    auto start = [&](uint32_t r) {
        const dev::V3 o = {rays[r], rays[R + r], rays[2 * R + r]};
        const dev::V3 d = {rays[3 * R + r], rays[4 * R + r], rays[5 * R + r]};
        w.begin(o, d, rays[6 * R + r]);
    };
    uint32_t r = gid;
    if (r < numRays) start(r);
    while (r < numRays) {
        if (!w.done()) w.step();
        if (w.done()) {
            over |= w.over();
            const bool hit = w.best != kEmpty && !isinf(w.t);
            hitFace[r] = hit ? w.best : kEmpty;
            hitT[r] = w.t;
            if constexpr (STATS) {
                stats[2 * (size_t)r] = w.st.visits;
                stats[2 * (size_t)r + 1] = w.st.tests;
            }
            r = numRays - r > lanes ? r + lanes : numRays;
            if (r < numRays) start(r);
        }
    }
    if (over) atomicOr(status, kStatusStackOverflow);
}

// With counts per ray: the walks whose visits and tests are defined.
template <bool WIDE>
__global__ __launch_bounds__(kOrdBlock) void k_trace_counts(
    dev::GeomScene g, const float* __restrict__ rays, uint32_t numRays, uint32_t* __restrict__ hitFace,
    float* __restrict__ hitT, uint32_t* __restrict__ stats, uint32_t* __restrict__ status,
    uint32_t* __restrict__ spill) {
    __shared__ uint32_t s_stack[kOrdLds * kOrdBlock];
    const uint32_t gid = blockIdx.x * kOrdBlock + threadIdx.x;
    const uint32_t lanes = gridDim.x * kOrdBlock;
    using S = dev::SpillStack<kOrdHalf>;
    const S stk0{s_stack + threadIdx.x, kOrdBlock, spill + gid, lanes};
    const S stk1{s_stack + kOrdHalf * kOrdBlock + threadIdx.x, kOrdBlock,
                 spill + (size_t)(dev::kStackPairs - kOrdHalf) * lanes + gid, lanes};
    using W = std::conditional_t<WIDE, dev::Wide<dev::NoAlpha, S, dev::kStackPairs>,
                                 dev::Ordered<dev::NoAlpha, S, true>>;
    W w0(g, stk0, dev::NoAlpha()), w1(g, stk1, dev::NoAlpha());
    traceTwo(w0, w1, rays, numRays, gid, lanes, status, [&](const W& w, uint32_t r) {
        const bool hit = w.best != kEmpty && !isinf(w.t);
        hitFace[r] = hit ? w.best : kEmpty;
        hitT[r] = w.t;
        stats[2 * (size_t)r] = w.st.visits;
        stats[2 * (size_t)r + 1] = w.st.tests;
    });
}

// Without counts: WideWalk, whatever ordered walk the caller asked for (the
// hit is the same). A level of the binary walk's tree leaves it one entry, a
// record (two levels) leaves up to three here: kTracePairs entries suffice for
// every tree of 64 levels, the depth at which the binary walk's 64 always do.
constexpr int kTracePairs = 96;
__global__ __launch_bounds__(kOrdBlock) void k_trace_wide(
    dev::GeomScene g, const float* __restrict__ rays, uint32_t numRays, uint32_t* __restrict__ hitFace,
    float* __restrict__ hitT, uint32_t* __restrict__ status, uint32_t* __restrict__ spill) {
    constexpr int kPairs = kOrdHalf / 2;
    using S = dev::PairStack<kPairs, kTracePairs>;
    __shared__ uint2 s_stack[2 * kPairs * kOrdBlock];
    const uint32_t gid = blockIdx.x * kOrdBlock + threadIdx.x;
    const uint32_t lanes = gridDim.x * kOrdBlock;
    uint2* sp = reinterpret_cast<uint2*>(spill);
    const S stk0{s_stack + threadIdx.x, kOrdBlock, sp + gid, lanes};
    const S stk1{s_stack + kPairs * kOrdBlock + threadIdx.x, kOrdBlock,
                 sp + (size_t)(S::CAP - kPairs) * lanes + gid, lanes};
    using W = dev::WideWalk<dev::NoAlpha, S>;
    W w0(g, stk0, dev::NoAlpha()), w1(g, stk1, dev::NoAlpha());
    traceTwo(w0, w1, rays, numRays, gid, lanes, status, [&](const W& w, uint32_t r) {
        const bool hit = w.best != kEmpty && !isinf(w.t);
        hitFace[r] = hit ? w.best : kEmpty;
        hitT[r] = w.t;
    });
}

}  // namespace

size_t accelNodeBytes(uint32_t n, bool midpoint) {
    const size_t slots = midpoint ? 2 * (size_t)n - 1 : (size_t)std::max(n, 2u) - 1;
    return (slots * 64 + 255) & ~size_t(255);
}

size_t accelWideBytes(uint32_t n, bool midpoint) { return 2 * accelNodeBytes(n, midpoint); }

void launchAccelWide(const clr_lbvh_inode* inodes, const clr_lbvh_leaf* leaves, const clr_bvh_node* bvh, uint32_t n,
                     float4* wnodes, hipStream_t stream) {
    if (bvh)
        k_accel_wide_bvh<<<(2 * n - 1 + 255) / 256, 256, 0, stream>>>(reinterpret_cast<const float4*>(bvh), n, wnodes);
    else
        k_accel_wide<<<(n + 255) / 256, 256, 0, stream>>>(inodes, leaves, n, wnodes);
}

int buildAccel(clr_ctx* ctx, const clr_scene_dev& sd, AccelKind kind, dev::GeomScene& g, hipStream_t stream) {
    const uint32_t n = sd.numFaces;
    const bool midpoint = sd.bvhNodes != nullptr;
    g = dev::GeomScene{sd.internalNodes, sd.leafNodes, n, sd.vertices, sd.faces};
    g.bvh = reinterpret_cast<const float4*>(sd.bvhNodes);
    if (kind == AccelKind::kNone) return CLR_OK;
    const size_t nodeBytes = kind == AccelKind::kBinary ? accelNodeBytes(n, midpoint) : accelWideBytes(n, midpoint);
    const size_t triBytes = ((size_t)n * 48 + 255) & ~size_t(255);
    // Room for either kind where it can be had, so that after a call of one
    // kind a captured call of the other allocates nothing.
    const size_t need = nodeBytes + triBytes, either = accelWideBytes(n, midpoint) + triBytes;
    if (ctx->accelBytes < need) {
        int rc = hipCheck(ctx, hipDeviceSynchronize(), "accel regrow sync");
        if (!rc) rc = giveUp(ctx, ctx->accel, ctx->accelHeld);
        if (rc) return rc;
        ctx->accel = nullptr;
        ctx->accelBytes = 0;
        for (size_t bytes : {either, need}) {
            if (hipMalloc(&ctx->accel, bytes) == hipSuccess) {
                ctx->accelBytes = bytes;
                break;
            }
            (void)hipGetLastError();
            ctx->accel = nullptr;
        }
        if (!ctx->accel)
            return fail(ctx, CLR_ERR_OUT_OF_MEMORY, "traversal layout of " + std::to_string(need) + " bytes");
    }
    holdIfCapturing(stream, ctx->accelHeld);
    float4* nodes = static_cast<float4*>(ctx->accel);
    float4* tris = reinterpret_cast<float4*>(static_cast<char*>(ctx->accel) + nodeBytes);
    launchAccelBuild(sd.internalNodes, sd.leafNodes, sd.bvhNodes, n, sd.vertices, sd.faces,
                     kind == AccelKind::kBinary ? nodes : nullptr, tris, stream);
    g.atris = tris;
    if (kind == AccelKind::kBinary) {
        g.anodes = nodes;
    } else {
        g.wnodes = nodes;
        launchAccelWide(sd.internalNodes, sd.leafNodes, sd.bvhNodes, n, nodes, stream);
    }
    return hipCheck(ctx, hipGetLastError(), "traversal layout launch");
}

void launchAccelBuild(const clr_lbvh_inode* inodes, const clr_lbvh_leaf* leaves, const clr_bvh_node* bvh,
                      uint32_t n, const clr_float3* vertices, const clr_face* faces, float4* anodes, float4* atris,
                      hipStream_t stream) {
    if (bvh)
        k_accel_build_bvh<<<(2 * n - 1 + 255) / 256, 256, 0, stream>>>(reinterpret_cast<const float4*>(bvh), n,
                                                                        vertices, faces, anodes, atris);
    else
        k_accel_build<false><<<(n + 255) / 256, 256, 0, stream>>>(inodes, leaves, n, vertices, faces, anodes, atris);
}

namespace {
// Grid of the kernels with 128-thread blocks: 16 waves per CU (LDS: 16 KiB per
// block).
int traceGrid(clr_ctx* ctx, uint32_t numRays, uint32_t& grid) {
    int cus = 0;
    int rc = hipCheck(ctx, hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device), "CU count");
    if (rc) return rc;
    grid = std::max(1u, std::min((uint32_t)cus * 8u, (numRays + kOrdBlock - 1) / kOrdBlock));
    return CLR_OK;
}
}  // namespace

int traceOrdered(clr_ctx* ctx, const clr_lbvh_inode* inodes, const clr_lbvh_leaf* leaves, const clr_bvh_node* bvh,
                 uint32_t n, const clr_float3* vertices, const clr_face* faces, const float* rays, uint32_t numRays,
                 uint32_t* hitFace, float* hitT, uint32_t* stats, hipStream_t stream, bool wide) {
    if (numRays == 0) return CLR_OK;
    int rc = ensureStatus(ctx);
    if (rc) return rc;
    uint32_t grid = 0;
    rc = traceGrid(ctx, numRays, grid);
    if (rc) return rc;
    // Of the kernels without and with counts the former takes more spill
    // memory; both find room after either.
    static_assert(2 * kTracePairs >= dev::kStackPairs, "spill covers the counting walks");
    rc = ensureTraceSpill(ctx, (size_t)grid * kOrdBlock * 2 * (2 * kTracePairs - kOrdHalf) * sizeof(uint32_t),
                          stream);
    if (rc) return rc;
    clr_scene_dev sd{};
    sd.vertices = vertices;
    sd.faces = faces;
    sd.internalNodes = inodes;
    sd.leafNodes = leaves;
    sd.numFaces = n;
    sd.bvhNodes = bvh;
    dev::GeomScene g;
    rc = buildAccel(ctx, sd, !stats || wide ? AccelKind::kWide : AccelKind::kBinary, g, stream);
    if (rc) return rc;
    if (!stats)
        k_trace_wide<<<grid, kOrdBlock, 0, stream>>>(g, rays, numRays, hitFace, hitT, ctx->devStatus, ctx->traceSpill);
    else if (wide)
        k_trace_counts<true><<<grid, kOrdBlock, 0, stream>>>(g, rays, numRays, hitFace, hitT, stats, ctx->devStatus,
                                                             ctx->traceSpill);
    else
        k_trace_counts<false><<<grid, kOrdBlock, 0, stream>>>(g, rays, numRays, hitFace, hitT, stats, ctx->devStatus,
                                                              ctx->traceSpill);
    return hipCheck(ctx, hipGetLastError(), "trace launch");
}

// The layout pays for itself from 2^14 rays, 4096 triangles and a ray for every
// 128 triangles on (us over the drop-in nodes / over the layout): 1000 triangles,
// 16384 rays 75 / 74 and 2 triangles 12 / 21; 20,000 triangles, 4096 rays 198 / 217,
// 16384 rays 238 / 234, 100,000 rays 283 / 272; 300,000 triangles, 4096 rays 729 / 740,
// 16384 rays 1224 / 940; 2,000,000 triangles, 16384 rays 3819 / 3342.
constexpr uint32_t kLayoutMinRays = 1u << 14, kLayoutMinFaces = 4096, kLayoutFacesPerRay = 128;

int traceClosest(clr_ctx* ctx, const clr_lbvh_inode* inodes, const clr_lbvh_leaf* leaves, const clr_bvh_node* bvh,
                 uint32_t n, const clr_float3* vertices, const clr_face* faces, const float* rays,
                 uint32_t numRays, uint32_t* hitFace, float* hitT, uint32_t* stats,
                 hipStream_t stream) {
    if (numRays == 0) return CLR_OK;
    int rc = ensureStatus(ctx);
    if (rc) return rc;
    // Enough rays of an LBVH walk over the traversal layout, which needs memory:
    // not while the stream is being captured (a graph would keep its address),
    // and not when there is none.
    if (!bvh && numRays >= kLayoutMinRays && n >= kLayoutMinFaces && numRays >= n / kLayoutFacesPerRay) {
        hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(stream, &capture) != hipSuccess) {
            (void)hipGetLastError();
            capture = hipStreamCaptureStatusActive;
        }
        uint32_t grid = 0;
        rc = traceGrid(ctx, numRays, grid);
        if (rc) return rc;
        const size_t nodeBytes = accelNodeBytes(n, false), triBytes = ((size_t)n * 48 + 255) & ~size_t(255);
        const size_t stackBytes = (size_t)grid * kOrdBlock * (dev::kStackDepth - kReferencePairs) * sizeof(uint2);
        if (capture == hipStreamCaptureStatusNone && ensureClosest(ctx, nodeBytes + triBytes + stackBytes)) {
            // Calls on several streams of the context take turns in the block
            // (the first wait finds nothing recorded and passes).
            rc = hipCheck(ctx, hipStreamWaitEvent(stream, ctx->closestDone, 0), "trace order");
            if (rc) return rc;
            dev::GeomScene g{inodes, leaves, n, vertices, faces};
            char* block = static_cast<char*>(ctx->closest);
            float4* nodes = reinterpret_cast<float4*>(block);
            float4* tris = reinterpret_cast<float4*>(block + nodeBytes);
            uint32_t* spill = reinterpret_cast<uint32_t*>(block + nodeBytes + triBytes);
            k_accel_build<true><<<(n + 255) / 256, 256, 0, stream>>>(inodes, leaves, n, vertices, faces, nodes, tris);
            g.anodes = nodes;
            g.atris = tris;
            if (stats)
                k_trace_reference<true><<<grid, kOrdBlock, 0, stream>>>(g, rays, numRays, hitFace, hitT, stats,
                                                                        ctx->devStatus, spill);
            else
                k_trace_reference<false><<<grid, kOrdBlock, 0, stream>>>(g, rays, numRays, hitFace, hitT, stats,
                                                                         ctx->devStatus, spill);
            rc = hipCheck(ctx, hipGetLastError(), "trace launch");
            return rc ? rc : hipCheck(ctx, hipEventRecord(ctx->closestDone, stream), "trace order");
        }
    }
    const unsigned grid = (numRays + kTraceBlock - 1) / kTraceBlock;
    const float4* b4 = reinterpret_cast<const float4*>(bvh);
    if (stats)
        k_trace_closest<true><<<grid, kTraceBlock, 0, stream>>>(
            inodes, leaves, n, vertices, faces, rays, numRays, hitFace, hitT, stats, ctx->devStatus, b4);
    else
        k_trace_closest<false><<<grid, kTraceBlock, 0, stream>>>(
            inodes, leaves, n, vertices, faces, rays, numRays, hitFace, hitT, stats, ctx->devStatus, b4);
    return hipCheck(ctx, hipGetLastError(), "trace launch");
}

}  // namespace clr
