// Ray tracing of the triangle scene on gfx950: the AVPL shooter and the
// G-buffer producer that feed the gather.
//
// The reference shoots AVPLs on the CPU (AvplShooter::createPath,
// AvplShooter.h:77-142, OpenMP over paths) against a kd-tree
// (KdTreeAccelerator.h:17-59, Scene::IntersectRayScene, Scene.cpp:243-255),
// then copies the AVPLs to the GPU every frame (AvplsGpu, data_gpu.cu:5-52).
// Here the paths run on the GPU and the AVPLs land in HBM where the gather
// reads them.
//
//   scene      triangles in the reference's Triangle layout (p0, p1, p2,
//              normal = normalize(cross(p2 - p0, p1 - p0)), material), one
//              64-byte record per triangle in input order; the leaves are
//              triangle pieces (large triangles split into slabs along their
//              longest axis), and the tree over them is a binned-SAH build
//              on the host at scene creation, collapsed to eight-wide nodes
//              (static geometry: built once, traversed by every path and
//              pixel by eight lanes per ray);
//   intersect  Triangle::intersect in FRONT_FACE mode (Triangle.h): Moller-
//              Trumbore on unnormalised barycentrics with the reference's
//              |det| < EPS = 1e-4 rejection; the closest hit with t > 0
//              (KdTreeAccelerator.cpp:301-320); a hit on an emissive
//              triangle counts as no hit (Scene.cpp:247-252).  The arithmetic
//              follows the reference's operation order in FP32 without
//              contraction (this unit is built with -ffp-contract=off), so a
//              CPU restatement finds the same triangle and distance;
//   shoot      createPath per path: light sample (AreaLight::samplePos),
//              cosine direction (sampleCosCone, Sampler.h:13-35), bounces
//              with Russian roulette 0.8, phong_eval / phong_sample
//              (Brdf.h:9-82) and the EPS offsets.  Random numbers come from a
//              counter-based hash of (seed, path, draw) instead of per-thread
//              mt19937_64 streams; each path's AVPLs are written in order at
//              an offset from an exclusive scan of the per-path counts, so
//              the output is deterministic;
//   gbuffer    one primary ray per pixel (pinhole camera), the closest
//              front-facing triangle, position (x, y, z, 1) and normal
//              (n, material) in the G-buffer layout the gather reads.
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <vector>

#include "arc_internal.hpp"
#include "launch_rules.hpp"

using arc::f3;

struct arc_trace_scene {
    arc_ctx* ctx = nullptr;
    int ntri = 0;
    int nleaf = 0;                    // leaves: triangle pieces (a large triangle is split)
    arc::DevBuf tri;                  // 4 float4 per triangle, input order
    arc::DevBuf nodes;                // the tree's eight-wide nodes, 16 float4 each (wide_nodes)
    int stack = 1;                    // most nodes a traversal keeps pending
    int nnodes = 0;                   // eight-wide nodes
    arc::DevBuf mats;                 // material table, 256 entries
    arc::DevBuf emissive;             // per material: emissive != 0
    int max_depth = 0;                // deepest internal node of the binary tree (root = 1)
    // shooter output
    arc::DevBuf count, stage, path_offset, scan_blocks, out;
};

namespace {

constexpr float kEps = 1e-4f;         // EPS (Defines.h:13)
constexpr float kRr = 0.8f;           // rrProb (AvplShooter.h:78)
constexpr float kTwoPi = 6.28318530718f;          // TWO_PI (Defines.h:5)
constexpr float kOneOverTwoPi = 0.15915494309f;   // ONE_OVER_TWO_PI (Defines.h:7)
constexpr float kOneOverPi = 0.318309886f;
constexpr int kThreads = 256;
constexpr int kMaxPieces = 8;         // most leaves one triangle is split into
constexpr int kTraceStack = 48;       // deepest binary tree taken
constexpr int kScan = 1024;

struct V {
    float x, y, z;
};
__host__ __device__ inline V mk(float x, float y, float z) { return V{x, y, z}; }
__device__ inline V operator+(V a, V b) { return mk(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ inline V operator-(V a, V b) { return mk(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ inline V operator*(float s, V a) { return mk(s * a.x, s * a.y, s * a.z); }
__device__ inline V operator*(V a, V b) { return mk(a.x * b.x, a.y * b.y, a.z * b.z); }
// glm::dot and glm::cross operation order
__device__ inline float dot(V a, V b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ inline V cross(V a, V b) {
    return mk(a.y * b.z - b.y * a.z, a.z * b.x - b.z * a.x, a.x * b.y - b.x * a.y);
}
__device__ inline float length(V a) { return sqrtf(dot(a, a)); }
__device__ inline V normalize(V a) { return (1.0f / length(a)) * a; }
__device__ inline V ld(const f3& a) { return mk(a.x, a.y, a.z); }
__device__ inline V ld(const arc_float3& a) { return mk(a.x, a.y, a.z); }

struct Tri {  // 4 float4 per triangle
    float4 a;  // p0, material index (bits)
    float4 b;  // e1 = p2 - p0 (FRONT_FACE first edge)
    float4 c;  // e2 = p1 - p0
    float4 d;  // unit normal, emissive flag
};

struct SceneDev {
    const float4* tri;               // triangles in input order, 4 float4 each
    const float4* nodes;             // eight-wide nodes, 16 float4 each
    int stack;                       // pending nodes of a traversal, per ray
    const arc_material* mats;        // 256 entries
    const int* emissive;             // 256 entries
};

// Triangle::intersect (Triangle.h), FRONT_FACE: e1 = p2 - p0, e2 = p1 - p0.
__device__ inline bool tri_hit(const Tri& T, V o, V dir, float det_eps, float& dist) {
    const V p0 = mk(T.a.x, T.a.y, T.a.z), e1 = mk(T.b.x, T.b.y, T.b.z), e2 = mk(T.c.x, T.c.y, T.c.z);
    const V p = cross(dir, e2);
    const float det = dot(e1, p);
    if (det < det_eps && det > -det_eps) return false;
    const V t = o - p0;
    const float u = dot(t, p);
    if (u < 0.0f || u > det) return false;
    const V q = cross(t, e1);
    const float v = dot(dir, q);
    if (v < 0.0f || u + v > det) return false;
    dist = 1.f / det * dot(e2, q);
    return true;
}

__device__ inline Tri load_tri(const float4* tri, int s) {
    const float4* r = tri + 4 * (size_t)s;
    return Tri{r[0], r[1], r[2], r[3]};
}

__device__ inline float safe_inv(float w) {
    const float m = fmaxf(fabsf(w), 1e-30f);
    return 1.0f / copysignf(m, w);
}

// Closest front-facing hits with t > 0 (ties: the lower triangle index, as a
// loop over the triangles in order finds it), eight lanes per ray.
//
// A step takes one node of the eight-wide tree: each lane of the ray's group
// tests one child, a triangle piece's triangle at once, and the inner children
// that the ray enters before its closest hit go to the group's stack in LDS,
// nearest on top.  The scenes' triangles overlap densely (a ray leaving a
// surface starts inside hundreds of boxes), so a ray is a long chain of
// dependent node reads, and for the few rays of a late bounce the chain is all
// the time: 0.7 ms a ray where one lane walks a two-wide tree.  An eight-wide
// step replaces about three dependent reads by one of 256 consecutive bytes
// and tests up to eight triangles together.  Where the chip is full (a
// G-buffer) the step's vector instructions bound it, about 110, a third of
// them the triangle test: 1280 x 720 pixels over 100K triangles take 1.40 ms,
// 2.26 with a lane per ray.  The order of the children comes from whole-number
// keys compared across DPP: with ds_bpermute and float compares it was half of
// a step (2.01 ms).
//
// The box tests are conservative in FP32: the exit distance carries a factor
// above the slabs' rounding and the keys', so a box that holds the closest hit
// is never passed over.
constexpr int kGroup = 8;                        // lanes per ray
constexpr int kWave = 64;                        // threads of a block that traces: no wave waits on another
constexpr int kGroups = kWave / kGroup;          // its rays
constexpr int kNoChild = 0x7fffffff;
constexpr float kBoxSlack = 1.000002f;

struct Ray {
    V o, d, inv;
    float det_eps;
    float t;       // closest hit so far, INFINITY for none
    int tri;       // its triangle, -1 for none
    int node, sp;  // the node to take next; pending nodes
    bool on;       // still in the tree
};

__device__ inline void ray_start(Ray& r, V o, V d, float det_eps) {
    r.o = o;
    r.d = d;
    r.inv = mk(safe_inv(d.x), safe_inv(d.y), safe_inv(d.z));
    r.det_eps = det_eps;
    r.t = INFINITY;
    r.tri = -1;
    r.node = 0;
    r.sp = 0;
    r.on = true;
}

// v of lane ^ X, X < 8
template <int X>
__device__ inline int lane_xor(int v) {
    constexpr int kQuad[4] = {0xE4, 0xB1, 0x4E, 0x1B};
    if (X >= 4) v = __builtin_amdgcn_update_dpp(v, v, 0x141, 0xf, 0xf, false);  // lane ^ 7
    constexpr int q = X >= 4 ? X ^ 7 : X;
    return q == 0 ? v : __builtin_amdgcn_update_dpp(v, v, kQuad[q], 0xf, 0xf, false);
}

template <int X>
__device__ inline void closer_of(float& t, int& ti) {  // the closer of this lane's hit and lane ^ X's
    const float ot = __int_as_float(lane_xor<X>(__float_as_int(t)));
    const int oi = lane_xor<X>(ti);
    if (oi >= 0 && (ot < t || (ot == t && oi < ti))) {
        t = ot;
        ti = oi;
    }
}

// One child: a hit of its triangle (t, ti) or the entry of its box as a key:
// the distance's bits, the last three replaced by the lane, so that no two of a
// group are equal; -1 for none.
__device__ inline int child_test(const SceneDev& S, const Ray& r, int node, int lane, float& t, int& ti, int& child) {
    const float4* c = S.nodes + 16 * (size_t)node + 2 * lane;
    const float4 lo = c[0], hi = c[1];
    child = __float_as_int(lo.w);
    const float tx0 = (lo.x - r.o.x) * r.inv.x, tx1 = (hi.x - r.o.x) * r.inv.x;
    const float ty0 = (lo.y - r.o.y) * r.inv.y, ty1 = (hi.y - r.o.y) * r.inv.y;
    const float tz0 = (lo.z - r.o.z) * r.inv.z, tz1 = (hi.z - r.o.z) * r.inv.z;
    const float t0 = fmaxf(fmaxf(fminf(tx0, tx1), fminf(ty0, ty1)), fmaxf(fminf(tz0, tz1), 0.f));
    const float t1 = fminf(fminf(fmaxf(tx0, tx1), fmaxf(ty0, ty1)), fminf(fmaxf(tz0, tz1), r.t));
    if (child == kNoChild || !(t0 <= t1 * kBoxSlack) || t0 == INFINITY) return -1;
    if (child < 0) return (__float_as_int(t0) & 0x7ffffff8) | lane;
    float d;
    if (tri_hit(load_tri(S.tri, child), r.o, r.d, r.det_eps, d) && d > 0.f) {
        t = d;
        ti = child;
    }
    return -1;
}

// Of a group's keys, how many are larger than this lane's.
__device__ inline int keys_after(int key) {
    return (lane_xor<1>(key) > key) + (lane_xor<2>(key) > key) + (lane_xor<3>(key) > key) +
           (lane_xor<4>(key) > key) + (lane_xor<5>(key) > key) + (lane_xor<6>(key) > key) +
           (lane_xor<7>(key) > key);
}

// One node of each ray that is on.  stk: the group's stack of (node, entry
// distance).  All lanes of the wave take part.
__device__ inline void ray_step(const SceneDev& S, Ray& r, int2* stk) {
    const int lane = threadIdx.x & (kGroup - 1);
    float t = INFINITY;
    int child = 0, ti = -1, key = -1;
    if (r.on) key = child_test(S, r, r.node, lane, t, ti, child);
    if (__ballot(ti >= 0)) {  // the group's closest, ties to the lower index
        closer_of<1>(t, ti);
        closer_of<2>(t, ti);
        closer_of<4>(t, ti);
        if (ti >= 0 && (t < r.t || (t == r.t && ti < r.tri))) {
            r.t = t;
            r.tri = ti;
        }
    }
    if (__int_as_float(key) > r.t * kBoxSlack) key = -1;
    // the entered children in order of distance, the nearest last
    const int after = keys_after(key);
    if (key >= 0) stk[r.sp + after] = make_int2(-(child + 1), key);
    const uint64_t in = __ballot(key >= 0);
    const unsigned half = threadIdx.x & 32 ? (unsigned)(in >> 32) : (unsigned)in;
    r.sp += __popc(__builtin_amdgcn_ubfe(half, threadIdx.x & 24, 8));
    __builtin_amdgcn_wave_barrier();  // the group's writes before its lanes read them
    if (r.on) {
        r.on = false;
        while (r.sp > 0) {  // the next pending subtree that can still hold a closer hit
            const int2 e = stk[--r.sp];
            if (__int_as_float(e.y) <= r.t * kBoxSlack) {
                r.node = e.x;
                r.on = true;
                break;
            }
        }
    }
    __builtin_amdgcn_wave_barrier();
}

__device__ inline float wave_value(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ inline V wave_value(V v, int lane) {
    return mk(wave_value(v.x, lane), wave_value(v.y, lane), wave_value(v.z, lane));
}

// The ray of the group that starts at lane `from`, by the whole wave: each
// group takes another pending node.  For the last rays of a wave, whose other
// groups have nothing left to do: the chain of dependent reads shortens by as
// many as the ray has nodes pending.  stk: the wave's stack, the other groups'
// parts included (no ray of theirs is in the tree).  Eight nodes are taken at
// once while their 64 children leave one depth-first descent's room.
__device__ inline void ray_wide(const SceneDev& S, Ray& mine, int from, int2* stk) {
    Ray r;
    r.o = wave_value(mine.o, from);
    r.d = wave_value(mine.d, from);
    r.inv = wave_value(mine.inv, from);
    r.det_eps = mine.det_eps;
    r.t = INFINITY;
    r.tri = -1;
    const int lane = threadIdx.x & (kGroup - 1), grp = threadIdx.x / kGroup;
    const uint64_t higher = ~0ull << (threadIdx.x | (kGroup - 1)) << 1;  // the groups after this one
    if (threadIdx.x == 0) stk[0] = make_int2(0, 0);
    __builtin_amdgcn_wave_barrier();
    int sp = 1;
    while (sp > 0) {
        const int take = sp + kWave <= (kGroups - 1) * S.stack ? min(sp, kGroups) : 1;
        float t = INFINITY;
        int child = 0, ti = -1, key = -1;
        if (grp < take) {
            const int2 e = stk[sp - 1 - grp];
            if (__int_as_float(e.y) <= r.t * kBoxSlack) key = child_test(S, r, e.x, lane, t, ti, child);
        }
        sp -= take;
        __builtin_amdgcn_wave_barrier();  // read before it is written
        if (__ballot(ti >= 0)) {
            closer_of<1>(t, ti);
            closer_of<2>(t, ti);
            closer_of<4>(t, ti);
            for (int g = 0; g < take; ++g) {
                const float ot = wave_value(t, g * kGroup);
                const int oi = __builtin_amdgcn_readlane(ti, g * kGroup);
                if (oi >= 0 && (ot < r.t || (ot == r.t && oi < r.tri))) {
                    r.t = ot;
                    r.tri = oi;
                }
            }
        }
        if (__int_as_float(key) > r.t * kBoxSlack) key = -1;
        const int after = keys_after(key);
        const uint64_t in = __ballot(key >= 0);
        if (key >= 0) stk[sp + after + __popcll(in & higher)] = make_int2(-(child + 1), key);
        sp += __popcll(in);
        __builtin_amdgcn_wave_barrier();
    }
    if ((int)(threadIdx.x & ~(kGroup - 1)) == from) {
        mine.t = r.t;
        mine.tri = r.tri;
        mine.on = false;
    }
}

// The rays of a wave, one per lane, through the tree together: an entry of the
// stack is a node and the rays that enter it, its records are read once for the
// wave as scalars, and each child is tested by all of the node's rays.  For trees
// of a few nodes and many rays (rays_together): there a ray in eight lanes of its
// own spends its steps on nodes that its neighbours visit too, and the blocks are
// eight times as many.  Bound by vector instructions, about 14 per child and 40 per
// triangle.  12 triangles, 5 nodes: 1920x1080 pixels 85 -> 23 us, a million rays 79
// -> 36, two million paths 9.8 -> 2.8 ms.  The tests are those of ray_step, so the
// hits are the same bits.  The pending nodes are at most those of one ray that
// enters every box, which S.stack counts.
__device__ inline void packet_trace(const SceneDev& S, Ray& r, int4* stk) {
    using namespace arc;
    uint64_t m = __ballot(r.on);
    int sp = 0, node = 0;
    while (m) {
        ufloat* c = uptr(S.nodes + 16 * (size_t)node);
        for (int k = 0; k < kGroup; ++k, c += 8) {
            const float4 lo = uload4(c), hi = uload4(c + 4);
            const int child = __float_as_int(lo.w);
            if (child == kNoChild) break;  // the children come first
            const float tx0 = (lo.x - r.o.x) * r.inv.x, tx1 = (hi.x - r.o.x) * r.inv.x;
            const float ty0 = (lo.y - r.o.y) * r.inv.y, ty1 = (hi.y - r.o.y) * r.inv.y;
            const float tz0 = (lo.z - r.o.z) * r.inv.z, tz1 = (hi.z - r.o.z) * r.inv.z;
            const float t0 = fmaxf(fmaxf(fminf(tx0, tx1), fminf(ty0, ty1)), fmaxf(fminf(tz0, tz1), 0.f));
            const float t1 = fminf(fminf(fmaxf(tx0, tx1), fmaxf(ty0, ty1)), fminf(fmaxf(tz0, tz1), r.t));
            const bool in = t0 <= t1 * kBoxSlack && t0 != INFINITY;
            const uint64_t enter = __ballot(in) & m;
            if (!enter) continue;
            if (child < 0) {
                if (threadIdx.x == 0) stk[sp] = make_int4(-(child + 1), (int)(uint32_t)enter, (int)(uint32_t)(enter >> 32), 0);
                ++sp;
                continue;
            }
            ufloat* p = uptr(S.tri + 4 * (size_t)child);
            const Tri T{uload4(p), uload4(p + 4), uload4(p + 8), make_float4(0.f, 0.f, 0.f, 0.f)};
            float d;
            if ((enter >> threadIdx.x & 1) && tri_hit(T, r.o, r.d, r.det_eps, d) && d > 0.f &&
                (d < r.t || (d == r.t && child < r.tri))) {
                r.t = d;
                r.tri = child;
            }
        }
        m = 0;
        if (sp > 0) {
            __builtin_amdgcn_wave_barrier();  // lane 0's writes before the wave's reads
            const int4 e = stk[--sp];
            node = __builtin_amdgcn_readfirstlane(e.x);
            m = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane(e.y) |
                (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane(e.z) << 32;
            __builtin_amdgcn_wave_barrier();
        }
    }
    r.on = false;
}

// Each ray to its end: kLanes lanes of the wave per ray, 8 or 1.
template <int kLanes>
__device__ inline void trace_rays(const SceneDev& S, Ray& r, int4* stacks) {
    if constexpr (kLanes == 1) {
        packet_trace(S, r, stacks);
    } else {
        int2* stk = reinterpret_cast<int2*>(stacks) + (size_t)(threadIdx.x / kGroup) * S.stack;
        while (__ballot(r.on)) ray_step(S, r, stk);
    }
}

// Scene::IntersectRayScene: a hit on an emissive triangle is no hit.
__device__ inline int scene_hit(const SceneDev& S, const Ray& r) {
    if (r.tri < 0) return -1;
    return S.emissive[__float_as_int(S.tri[4 * (size_t)r.tri].w) & 255] ? -1 : r.tri;
}

// ------------------------------------------------------------ sampling --
struct Rng {
    uint64_t seed, base;
    uint32_t k;
    __device__ inline float next() { return arc::hash_uniform(seed, base | (uint64_t)(k++)); }
};

// tangentSpace (Util.h:8-14): columns U, V, n.
__device__ inline void tangent_space(V n, V& U, V& W) {
    const V t = mk(n.y, n.z, -n.x);
    U = normalize(cross(t, n));
    W = normalize(cross(U, n));
}

// sampleCosCone (Sampler.h:13-35) with order `order`.
__device__ inline V sample_cos_cone(V n, float u1, float u2, float order, float& pdf) {
    V U, W;
    tangent_space(n, U, W);
    // cos(theta) = u1^(1 / (order + 1)); for the cosine lobe (order 1) the
    // square root, correctly rounded, and sin(theta) = sqrt(1 - cos^2) stand
    // for the reference's acos / pow / sin / cos (the same values up to
    // rounding, without acos's ill conditioning near theta = 0)
    float ct, st;
    if (order == 1.f) {
        ct = sqrtf(u1);
        st = sqrtf(fmaxf(0.f, 1.f - u1));
    } else {
        const float theta = acosf(powf(u1, 1.0f / (order + 1.0f)));
        ct = cosf(theta);
        st = sinf(theta);
    }
    const float phi = kTwoPi * u2;
    const V s = normalize(mk(st * cosf(phi), st * sinf(phi), ct));
    const float cos_theta = s.z;
    pdf = (order + 1.f) * kOneOverTwoPi * powf(cos_theta, order);
    return normalize(mk(U.x * s.x + W.x * s.y + n.x * s.z, U.y * s.x + W.y * s.y + n.y * s.z,
                        U.z * s.x + W.z * s.y + n.z * s.z));
}

__device__ inline float luminance(V v) { return 0.2126f * v.x + 0.7152f * v.y + 0.0722f * v.z; }
__device__ inline V reflect(V v, V n) { return normalize((2.f * dot(v, n)) * n - v); }

// phong_eval (Brdf.h:9-22)
__device__ inline V phong_eval(V wi, V wo, V n, const arc_material& m) {
    if (dot(wi, n) <= 0.f) return mk(0.f, 0.f, 0.f);
    if (dot(wo, n) <= 0.f) return mk(0.f, 0.f, 0.f);
    V res = mk(0.f, 0.f, 0.f);
    const V spec = ld(m.specular);
    if (length(spec) > 0.f) {
        const V r = reflect(wi, n);
        const float c = fmaxf(0.f, dot(r, wo));
        res = res + (kOneOverTwoPi * (m.exponent + 2.f) * powf(c, m.exponent)) * spec;
    }
    return res + kOneOverPi * ld(m.diffuse);
}

// phong_sample (Brdf.h:54-82): a sampled specular direction only decides
// whether the path ends; the returned direction is always the cosine sample
// about n.
__device__ inline V phong_sample(V wi, V n, const arc_material& m, float s0, float s1, float& pdf) {
    const bool has_diffuse = length(ld(m.diffuse)) > 0.f;
    const bool has_specular = length(ld(m.specular)) > 0.f;
    bool chose_specular = has_specular;
    if (has_diffuse && has_specular) {
        const float alpha = luminance(ld(m.specular)) / (luminance(ld(m.specular)) + luminance(ld(m.diffuse)));
        if (s0 <= alpha) {
            s0 /= alpha;
        } else {
            s0 = (s0 - alpha) / (1.f - alpha);
            chose_specular = false;
        }
    }
    if (chose_specular) {
        const V dir = sample_cos_cone(wi, s0, s1, m.exponent, pdf);
        if (dot(dir, n) <= 0.f) return mk(0.f, 0.f, 0.f);
    }
    return sample_cos_cone(n, s0, s1, 1.f, pdf);
}

struct Light {
    V center, front, s, u;  // quad centre, unit front, unit side axes
    float half_w, half_h, area;
    V radiance;
    int mat;
};

struct AvplOut {
    f3 *pos, *nrm, *dir, *rad, *anti;
    int *mat, *bounce;
};

struct Staged {  // AVPLs in the order they were created; path -1: no AVPL
    AvplOut a;
    int* path;
};

// createPath (AvplShooter.h:77-142), a path per group of kLanes lanes (eight, or
// one where a wave's rays are traced together) from its first ray to its last:
// traced, its AVPL staged, continued or replaced by the next path without
// leaving the kernel.  (With a launch per bounce, the host waits for the count
// of live paths 47 times per 100K paths, and a bounce of a handful of rays takes
// as long as its longest ray: 100K paths over 100K triangles took 33 ms, 2.1
// here.)  With eight lanes a ray, a wave shades when at most a third of its live
// rays are still in the tree, so that few lanes wait for the longest one.  What
// bounds it is the longest path, up to 47 rays one after the other (5.4 ms with
// eight lanes for each ray to the end); so a wave with no more than four paths
// left takes their rays one by one with all its lanes (ray_wide).  Draw order per path as in createPath: light position (2),
// first direction (2), then per bounce roulette (1) and the next direction
// (2).  Writes each path's AVPL count; a final scatter puts every path's AVPLs
// together in path order.  AVPLs past `cap` are counted, not staged.
constexpr int kWideRays = 4;   // most rays of a wave that it takes one by one
constexpr int kSlotGrab = 64;  // staging slots a wave takes with one atomic

template <int kLanes>
__global__ __launch_bounds__(kWave) void k_paths(SceneDev S, Light L, uint64_t seed, int paths, int explicit_direct,
                                                    int* __restrict__ next_path, unsigned* __restrict__ n_staged, int cap,
                                                    int* __restrict__ count, Staged st) {
    extern __shared__ int4 lds[];
    int2* stacks = reinterpret_cast<int2*>(lds);
    const int grp = threadIdx.x / kLanes, lane = threadIdx.x & 63;
    const bool lead = (threadIdx.x & (kLanes - 1)) == 0;
    int2* stk = stacks + (size_t)grp * S.stack;
    int slots = 0, nslots = 0;  // the wave's staging slots
    int path = (int)blockIdx.x * (kWave / kLanes) + grp;
    bool wide = false;          // so few paths are left that the wave traces each ray as a whole
    bool fresh = true, done = false;  // the group starts a path; has none left
    V pos{}, nrm{}, rad0{}, in_dir{}, direction{};
    float pdf0 = 0.f;
    int bounce0 = 0, mat0 = 0;
    Rng rng{seed, 0, 0};
    Ray r{};
    for (;;) {
        const bool shade = !r.on && !done;
        bool made = false, ended = fresh && shade;
        V hit_n{}, hit_pos{}, contrib{}, anti{}, rad{}, next{};
        float pdf = 0.f;
        int mat = 0;
        if (shade && !fresh) {
            const int s = scene_hit(S, r);
            ended = true;
            if (s >= 0) {
                made = true;
                const float cos_theta = dot(nrm, direction);
                // getIncidentRadiance() * cos_theta / pdf, per component
                contrib = mk(rad0.x * cos_theta / pdf0, rad0.y * cos_theta / pdf0, rad0.z * cos_theta / pdf0);
                if (bounce0 > 0) contrib = contrib * phong_eval(-1.f * in_dir, direction, nrm, S.mats[mat0 & 255]);
                const float4* T = S.tri + 4 * (size_t)s;
                hit_n = mk(T[3].x, T[3].y, T[3].z);
                const V hit = r.o + r.t * direction;  // Intersection::setPosition(origin + dist * dir)
                hit_pos = hit - kEps * hit_n;
                mat = __float_as_int(T[0].w);
                anti = contrib;
                if (bounce0 == 0 && explicit_direct) anti = mk(0.f, 0.f, 0.f);
                const bool stop = rng.next() > kRr;  // Russian roulette
                rad = stop ? mk(0.f, 0.f, 0.f) : (1.f / kRr) * contrib;
                if (!stop) {
                    const float s0 = rng.next(), s1 = rng.next();
                    next = phong_sample(-1.f * direction, hit_n, S.mats[mat & 255], s0, s1, pdf);
                    ended = length(next) <= 0.f || pdf < 1e-4f;
                }
            }
        }
        const uint64_t mm = __ballot(made && lead);
        if (mm) {  // staging slots for the AVPLs just made
            const int need = __popcll(mm);
            if (nslots < need) {
                if (lane < nslots && (unsigned)(slots + lane) < (unsigned)cap) st.path[slots + lane] = -1;  // not used
                int got = 0;
                if (lane == 0) got = (int)atomicAdd(n_staged, (unsigned)kSlotGrab);
                slots = __builtin_amdgcn_readfirstlane(got);
                nslots = kSlotGrab;
            }
            const int slot = slots + __popcll(mm & ((1ull << lane) - 1ull));
            if (made && lead && (unsigned)slot < (unsigned)cap) {
                st.a.pos[slot] = f3{hit_pos.x, hit_pos.y, hit_pos.z};
                st.a.nrm[slot] = f3{hit_n.x, hit_n.y, hit_n.z};
                st.a.dir[slot] = f3{direction.x, direction.y, direction.z};
                st.a.rad[slot] = f3{rad.x, rad.y, rad.z};
                st.a.anti[slot] = f3{anti.x, anti.y, anti.z};
                st.a.mat[slot] = mat;
                st.a.bounce[slot] = bounce0 + 1;
                st.path[slot] = path;
            }
            slots += need;
            nslots -= need;
        }
        if (made) {
            ++bounce0;
            pos = hit_pos;
            nrm = hit_n;
            rad0 = rad;
            in_dir = direction;
            direction = next;
            pdf0 = pdf;
            mat0 = mat;
        }
        if (shade && ended && !fresh && lead) count[path] = bounce0;
        const uint64_t me = __ballot(shade && ended && !fresh && lead);
        if (me) {  // the next paths
            int got = 0;
            if (lane == 0) got = atomicAdd(next_path, __popcll(me));
            got = __builtin_amdgcn_readfirstlane(got);
            // the group's leader's place among the wave's leaders
            const int mine = got + __popcll(me & ((1ull << (lane & ~(kLanes - 1))) - 1ull));
            if (shade && ended && !fresh) path = mine;
        }
        if (shade && ended) {
            if (path >= paths) {
                done = true;
            } else {  // AreaLight::samplePos: glm::linearRand over [-1, 1]^2, x then y
                rng = Rng{seed, (uint64_t)path << 24, 0};
                const float sx = -1.f + 2.f * rng.next();
                const float sy = -1.f + 2.f * rng.next();
                pos = L.center + (sx * L.half_w) * L.s + (sy * L.half_h) * L.u;
                const float area_pdf = 1.f / L.area;
                rad0 = (1.f / area_pdf) * L.radiance;  // rad / pdf
                const float u1 = rng.next(), u2 = rng.next();
                direction = sample_cos_cone(L.front, u1, u2, 1.f, pdf0);
                nrm = L.front;
                in_dir = mk(0.f, 0.f, 0.f);
                bounce0 = 0;
                mat0 = L.mat;
            }
            fresh = false;
        }
        if (shade && !done) ray_start(r, pos + kEps * nrm, direction, kEps);
        const uint64_t live = __ballot(!done);
        if (live == 0) break;
        if constexpr (kLanes == 1) {
            packet_trace(S, r, lds);
            continue;
        }
        if (wide) {  // every live ray starts here
            for (uint64_t m = live & 0x0101010101010101ull; m; m &= m - 1) ray_wide(S, r, __builtin_ctzll(m), stacks);
            continue;
        }
        wide = __popcll(live) <= kWideRays * kGroup;
        // trace until at most a third of the live rays are in the tree; to the
        // end before the wave takes its last rays one by one
        for (;;) {
            const uint64_t on = __ballot(r.on);
            if (on == 0 || (!wide && 2 * __popcll(on) <= __popcll(live & ~on))) break;
            ray_step(S, r, stk);
        }
    }
    if (lane < nslots && (unsigned)(slots + lane) < (unsigned)cap) st.path[slots + lane] = -1;
}

// Staged AVPL -> offset[path] + bounce - 1: each path's AVPLs together, in
// path order and bounce order.
__global__ __launch_bounds__(kThreads) void k_path_scatter(Staged st, int n_staged, const int* __restrict__ offsets,
                                                           AvplOut o) {
    const int k = blockIdx.x * kThreads + threadIdx.x;
    if (k >= n_staged) return;
    const int i = st.path[k];
    if (i < 0) return;
    const int dst = offsets[i] + st.a.bounce[k] - 1;
    o.pos[dst] = st.a.pos[k];
    o.nrm[dst] = st.a.nrm[k];
    o.dir[dst] = st.a.dir[k];
    o.rad[dst] = st.a.rad[k];
    o.anti[dst] = st.a.anti[k];
    o.mat[dst] = st.a.mat[k];
    o.bounce[dst] = st.a.bounce[k];
}

// Exclusive scan of n ints: per-block scan (kScan per block), block totals,
// then the totals' scan added back.  out[n] = total.
__global__ __launch_bounds__(kScan) void k_scan_local(const int* __restrict__ in, int n, int* __restrict__ out,
                                                      int* __restrict__ block_sums) {
    __shared__ int sh[kScan];
    const int i = blockIdx.x * kScan + threadIdx.x;
    const int v = i < n ? in[i] : 0;
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int off = 1; off < kScan; off <<= 1) {
        const int a = (int)threadIdx.x >= off ? sh[threadIdx.x - off] : 0;
        __syncthreads();
        sh[threadIdx.x] += a;
        __syncthreads();
    }
    if (i < n) out[i] = sh[threadIdx.x] - v;
    if (threadIdx.x == kScan - 1) block_sums[blockIdx.x] = sh[kScan - 1];
}

__global__ __launch_bounds__(kScan) void k_scan_sums(int* __restrict__ sums, int nb) {
    __shared__ int sh[kScan];
    int run = 0;
    for (int base = 0; base < nb; base += kScan) {
        const int t = base + (int)threadIdx.x;
        const int v = t < nb ? sums[t] : 0;
        sh[threadIdx.x] = v;
        __syncthreads();
        for (int off = 1; off < kScan; off <<= 1) {
            const int a = (int)threadIdx.x >= off ? sh[threadIdx.x - off] : 0;
            __syncthreads();
            sh[threadIdx.x] += a;
            __syncthreads();
        }
        if (t < nb) sums[t] = run + sh[threadIdx.x] - v;
        run += sh[kScan - 1];
        __syncthreads();
    }
    if (threadIdx.x == 0) sums[nb] = run;
}

__global__ __launch_bounds__(kScan) void k_scan_add(int* __restrict__ out, int n, const int* __restrict__ sums,
                                                    int nb) {
    const int i = blockIdx.x * kScan + threadIdx.x;
    if (i < n) out[i] += sums[blockIdx.x];
    if (i == 0) out[n] = sums[nb];
}

// ---------------------------------------------------------- G-buffer --
struct Camera {
    V pos, right, up, fwd;  // right and up scaled by tan(fovy / 2) (and the aspect)
};

template <int kLanes>
__global__ __launch_bounds__(kWave) void k_gbuffer(SceneDev S, Camera cam, int W, int H,
                                                      float4* __restrict__ pos4, float4* __restrict__ nrm4) {
    extern __shared__ int4 lds[];
    // a block's rays are 4 x 2 pixels, or 8 x 8
    constexpr int bx = kLanes == 1 ? 8 : 4, by = kWave / kLanes / bx;
    const int grp = threadIdx.x / kLanes, bw = (W + bx - 1) / bx;
    const int px = (int)(blockIdx.x % bw) * bx + grp % bx, py = (int)(blockIdx.x / bw) * by + grp / bx;
    const bool live = px < W && py < H;
    const int i = py * W + px;
    const float sx = 2.f * ((float)px + 0.5f) / (float)W - 1.f;
    const float sy = 1.f - 2.f * ((float)py + 0.5f) / (float)H;
    const V dir = normalize(cam.fwd + sx * cam.right + sy * cam.up);
    Ray r;
    ray_start(r, cam.pos, dir, 0.f);  // a rasteriser has no |det| floor: any front face counts
    r.on = live;
    trace_rays<kLanes>(S, r, lds);
    if (!live || (threadIdx.x & (kLanes - 1)) != 0) return;
    const int s = r.tri;
    const float t = r.t;
    if (s < 0) {
        pos4[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        nrm4[i] = make_float4(0.f, 0.f, -1.f, 1.f);
        return;
    }
    const float4* T = S.tri + 4 * (size_t)s;
    const V x = cam.pos + t * dir;
    pos4[i] = make_float4(x.x, x.y, x.z, 1.f);
    nrm4[i] = make_float4(T[3].x, T[3].y, T[3].z, (float)__float_as_int(T[0].w));
}

// --------------------------------------------------------------- build --
// Packs the triangles in sorted order and their boxes.
__global__ __launch_bounds__(kThreads) void k_pack_tris(const f3* __restrict__ p0, const f3* __restrict__ p1,
                                                        const f3* __restrict__ p2, const int* __restrict__ mat,
                                                        const int* __restrict__ emis, int n,
                                                        float4* __restrict__ tri) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= n) return;
    const int s = i;
    const V a = ld(p0[i]), b = ld(p1[i]), c = ld(p2[i]);
    V nn = cross(c - a, b - a);  // Triangle::calcNormal
    if (length(nn) > 0.f) nn = normalize(nn);
    const int m = mat[i];
    float4* o = tri + 4 * (size_t)s;
    o[0] = make_float4(a.x, a.y, a.z, __int_as_float(m));
    const V e1 = c - a, e2 = b - a;
    o[1] = make_float4(e1.x, e1.y, e1.z, 0.f);
    o[2] = make_float4(e2.x, e2.y, e2.z, 0.f);
    o[3] = make_float4(nn.x, nn.y, nn.z, (float)emis[m & 255]);
}


// A shot's counters: the first path that no group starts with, no AVPL staged.
__global__ void k_paths_reset(int* __restrict__ counters, int first) {
    counters[0] = first;
    counters[1] = 0;
}

template <int kLanes>
__global__ __launch_bounds__(kWave) void k_intersect(SceneDev S, const f3* __restrict__ org,
                                                     const f3* __restrict__ dir, int n, float* __restrict__ t,
                                                     int* __restrict__ tri_index) {
    extern __shared__ int4 lds[];
    const int grp = threadIdx.x / kLanes, i = blockIdx.x * (kWave / kLanes) + grp;
    const bool live = i < n;
    Ray r;
    ray_start(r, ld(org[live ? i : 0]), ld(dir[live ? i : 0]), kEps);
    r.on = live;
    trace_rays<kLanes>(S, r, lds);
    if (!live || (threadIdx.x & (kLanes - 1)) != 0) return;
    const int s = scene_hit(S, r);
    t[i] = s < 0 ? -1.f : r.t;
    tri_index[i] = s;
}

int blocks(int n) { return (n + kThreads - 1) / kThreads; }

SceneDev scene_dev(arc_trace_scene* sc) {
    return SceneDev{sc->tri.as<float4>(), sc->nodes.as<float4>(), sc->stack, sc->mats.as<arc_material>(),
                    sc->emissive.as<int>()};
}

constexpr int kPathBlocks = 4096;  // waves of k_paths: four per SIMD, what its registers let run at once

size_t stack_bytes(const arc_trace_scene* sc) { return sizeof(int2) * (size_t)kGroups * sc->stack; }

// Binned SAH build over the leaves' boxes (host, once per scene): 16 bins
// of the centroids along the longest axis of their bounds, the split of
// least area x count on either side; a run of equal centroids splits at its
// middle.  Below depth kSahDepth the splits take the median instead, which
// bounds the tree's depth by kSahDepth + log2(leaves) for the traversal's
// stack.  Writes the leaf order (leaf slot -> box index) and the internal
// nodes in the library's BvhNode layout (child >= 0: leaf slot; < 0: internal
// -(k + 1)), with their boxes; node 0 is the root.
constexpr int kSahBins = 16;
constexpr int kSahDepth = 26;

void sah_build(const std::vector<float>& lo, const std::vector<float>& hi, std::vector<int>& order,
               std::vector<arc_bvh_node>& nodes) {
    const int n = (int)(lo.size() / 3);
    order.resize(n);
    for (int i = 0; i < n; ++i) order[i] = i;
    nodes.assign(n > 1 ? n - 1 : 0, arc_bvh_node{});
    if (n < 2) return;
    std::vector<float> cen(3 * (size_t)n);
    for (size_t k = 0; k < cen.size(); ++k) cen[k] = 0.5f * (lo[k] + hi[k]);
    auto area = [](const float* l, const float* h) {
        const float x = h[0] - l[0], y = h[1] - l[1], z = h[2] - l[2];
        return x * y + y * z + z * x;
    };
    struct Task { int b, e, node, depth; };
    std::vector<Task> stack{{0, n, 0, 0}};
    int next = 1;
    while (!stack.empty()) {
        const Task T = stack.back();
        stack.pop_back();
        float bl[3] = {INFINITY, INFINITY, INFINITY}, bh[3] = {-INFINITY, -INFINITY, -INFINITY};
        float cl[3] = {INFINITY, INFINITY, INFINITY}, ch[3] = {-INFINITY, -INFINITY, -INFINITY};
        for (int j = T.b; j < T.e; ++j) {
            const int i = order[j];
            for (int d = 0; d < 3; ++d) {
                bl[d] = std::min(bl[d], lo[3 * i + d]);
                bh[d] = std::max(bh[d], hi[3 * i + d]);
                cl[d] = std::min(cl[d], cen[3 * i + d]);
                ch[d] = std::max(ch[d], cen[3 * i + d]);
            }
        }
        arc_bvh_node& nd = nodes[T.node];
        nd.bbMin = arc_float3{bl[0], bl[1], bl[2]};
        nd.bbMax = arc_float3{bh[0], bh[1], bh[2]};
        nd.visited = 0;
        int a = 0;
        for (int d = 1; d < 3; ++d)
            if (ch[d] - cl[d] > ch[a] - cl[a]) a = d;
        const int count = T.e - T.b;
        int mid = T.b + count / 2;
        bool binned = false;
        const float span = ch[a] - cl[a];
        if (span > 0.f && T.depth < kSahDepth) {
            int bc[kSahBins] = {};
            float bbl[kSahBins][3], bbh[kSahBins][3];
            for (int k = 0; k < kSahBins; ++k)
                for (int d = 0; d < 3; ++d) {
                    bbl[k][d] = INFINITY;
                    bbh[k][d] = -INFINITY;
                }
            const float scale = kSahBins / span;
            auto bin_of = [&](int i) {
                return std::min(kSahBins - 1, (int)((cen[3 * i + a] - cl[a]) * scale));
            };
            for (int j = T.b; j < T.e; ++j) {
                const int i = order[j], k = bin_of(i);
                ++bc[k];
                for (int d = 0; d < 3; ++d) {
                    bbl[k][d] = std::min(bbl[k][d], lo[3 * i + d]);
                    bbh[k][d] = std::max(bbh[k][d], hi[3 * i + d]);
                }
            }
            // sweep: areas of the left prefixes and right suffixes
            float ra[kSahBins];
            int rc[kSahBins];
            float sl[3] = {INFINITY, INFINITY, INFINITY}, sh[3] = {-INFINITY, -INFINITY, -INFINITY};
            int cnt = 0;
            for (int k = kSahBins - 1; k > 0; --k) {
                cnt += bc[k];
                for (int d = 0; d < 3; ++d) {
                    sl[d] = std::min(sl[d], bbl[k][d]);
                    sh[d] = std::max(sh[d], bbh[k][d]);
                }
                ra[k] = cnt ? area(sl, sh) : 0.f;
                rc[k] = cnt;
            }
            float best = INFINITY;
            int split = -1;
            for (int d = 0; d < 3; ++d) {
                sl[d] = INFINITY;
                sh[d] = -INFINITY;
            }
            cnt = 0;
            for (int k = 0; k < kSahBins - 1; ++k) {
                cnt += bc[k];
                for (int d = 0; d < 3; ++d) {
                    sl[d] = std::min(sl[d], bbl[k][d]);
                    sh[d] = std::max(sh[d], bbh[k][d]);
                }
                if (cnt == 0 || rc[k + 1] == 0) continue;
                const float cost = (float)cnt * area(sl, sh) + (float)rc[k + 1] * ra[k + 1];
                if (cost < best) {
                    best = cost;
                    split = k;
                }
            }
            if (split >= 0) {  // both sides hold leaves by construction
                auto it = std::partition(order.begin() + T.b, order.begin() + T.e,
                                         [&](int i) { return bin_of(i) <= split; });
                mid = (int)(it - order.begin());
                binned = mid > T.b && mid < T.e;
            }
        }
        if (!binned) {  // median split (deep subtrees, runs of equal centroids)
            mid = T.b + count / 2;
            std::nth_element(order.begin() + T.b, order.begin() + mid, order.begin() + T.e,
                             [&](int x, int y) { return cen[3 * x + a] < cen[3 * y + a]; });
        }
        const int ranges[2][2] = {{T.b, mid}, {mid, T.e}};
        int child[2];
        for (int c = 0; c < 2; ++c) {
            if (ranges[c][1] - ranges[c][0] == 1) {
                child[c] = ranges[c][0];  // leaf slot
            } else {
                const int k = next++;
                child[c] = -(k + 1);
                stack.push_back({ranges[c][0], ranges[c][1], k, T.depth + 1});
            }
        }
        nd.left = child[0];
        nd.right = child[1];
    }
}

// Depth of the deepest internal node (host, from the node array).
int tree_depth(const std::vector<arc_bvh_node>& nodes) {
    if (nodes.empty()) return 0;
    int best = 0;
    std::vector<std::pair<int, int>> st{{0, 1}};
    while (!st.empty()) {
        auto [k, d] = st.back();
        st.pop_back();
        best = std::max(best, d);
        if (nodes[k].left < 0) st.push_back({-(nodes[k].left + 1), d + 1});
        if (nodes[k].right < 0) st.push_back({-(nodes[k].right + 1), d + 1});
    }
    return best;
}

// The binary tree as eight-wide nodes: from a node's two children, the inner
// child of the largest box is replaced by its own children until there are
// eight or only leaves.  A node is 16 float4: per child (box lo, child) and
// (box hi, 0), child >= 0 a triangle, < 0 the eight-wide node -(child + 1),
// kNoChild none.  The boxes are widened by 1e-5 of the scene's largest
// coordinate, far above the rounding of the triangle test, so no hit at a
// piece's edge is lost.  `stack` receives the most nodes a depth-first
// traversal keeps pending.
void wide_nodes(const std::vector<arc_bvh_node>& nodes, const std::vector<int>& order, const std::vector<float>& plo,
                const std::vector<float>& phi, const std::vector<int>& ptri, std::vector<float4>& wide, int& stack) {
    struct Child { int c; float lo[3], hi[3]; };
    auto child = [&](int c) {
        Child r;
        r.c = c;
        for (int d = 0; d < 3; ++d) {
            if (c >= 0) {
                r.lo[d] = plo[3 * (size_t)order[c] + d];
                r.hi[d] = phi[3 * (size_t)order[c] + d];
            } else {
                const arc_bvh_node& n = nodes[-(c + 1)];
                r.lo[d] = (&n.bbMin.x)[d];
                r.hi[d] = (&n.bbMax.x)[d];
            }
        }
        return r;
    };
    auto area = [](const Child& r) {
        const float x = r.hi[0] - r.lo[0], y = r.hi[1] - r.lo[1], z = r.hi[2] - r.lo[2];
        return x * y + y * z + z * x;
    };
    float far = 0.f;
    for (size_t k = 0; k < plo.size(); ++k) far = std::max({far, std::fabs(plo[k]), std::fabs(phi[k])});
    const float pad = 1e-5f * far;
    struct Task { int node, wide, pending; };  // binary node (-1: a tree of one leaf), its place, nodes pending above it
    std::vector<Task> tasks{{nodes.empty() ? -1 : 0, 0, 0}};
    wide.assign(16, float4{});
    stack = 1;
    while (!tasks.empty()) {
        const Task t = tasks.back();
        tasks.pop_back();
        Child c[8];
        int n = 0;
        if (t.node < 0) {
            c[n++] = child(0);
        } else {
            c[n++] = child(nodes[t.node].left);
            c[n++] = child(nodes[t.node].right);
        }
        while (n < 8) {
            int best = -1;
            for (int k = 0; k < n; ++k)
                if (c[k].c < 0 && (best < 0 || area(c[k]) > area(c[best]))) best = k;
            if (best < 0) break;
            const arc_bvh_node& b = nodes[-(c[best].c + 1)];
            c[best] = child(b.left);
            c[n++] = child(b.right);
        }
        int inner = 0;
        for (int k = 0; k < n; ++k) inner += c[k].c < 0;
        stack = std::max(stack, t.pending + inner);
        for (int k = 0; k < 8; ++k) {
            float4 lo{}, hi{};
            int ref = kNoChild;
            if (k < n) {
                if (c[k].c >= 0) {
                    ref = ptri[order[c[k].c]];
                } else {
                    const int w = (int)(wide.size() / 16);
                    wide.resize(wide.size() + 16);
                    tasks.push_back({-(c[k].c + 1), w, t.pending + inner - 1});
                    ref = -(w + 1);
                }
                lo = make_float4(c[k].lo[0] - pad, c[k].lo[1] - pad, c[k].lo[2] - pad, 0.f);
                hi = make_float4(c[k].hi[0] + pad, c[k].hi[1] + pad, c[k].hi[2] + pad, 0.f);
            }
            std::memcpy(&lo.w, &ref, sizeof(int));
            wide[16 * (size_t)t.wide + 2 * k] = lo;
            wide[16 * (size_t)t.wide + 2 * k + 1] = hi;
        }
    }
}

}  // namespace

extern "C" {

int arc_trace_scene_create(arc_ctx* ctx, const arc_float3* p0, const arc_float3* p1, const arc_float3* p2,
                           const int* material, int ntri, const arc_material* materials, int num_materials,
                           int flags, arc_trace_scene** out) {
    if (!ctx || !out || ntri < 1 || !p0 || !p1 || !p2 || !material || !materials || num_materials < 1 ||
        num_materials > 256)
        return ARC_E_INVALID;
    *out = nullptr;
    arc_trace_scene* sc = new arc_trace_scene();
    sc->ctx = ctx;
    sc->ntri = ntri;
    auto fail = [&](int st) {
        arc_trace_scene_destroy(sc);
        return st;
    };
    // the triangles on the host (the tree is built there)
    const size_t v3 = sizeof(arc_float3) * (size_t)ntri;
    std::vector<arc_float3> h0(ntri), h1(ntri), h2(ntri);
    std::vector<int> hm(ntri);
    hipError_t e = hipSuccess;
    if (flags & ARC_INPUT_HOST) {
        std::copy(p0, p0 + ntri, h0.begin());
        std::copy(p1, p1 + ntri, h1.begin());
        std::copy(p2, p2 + ntri, h2.begin());
        std::copy(material, material + ntri, hm.begin());
    } else {
        e = hipMemcpy(h0.data(), p0, v3, hipMemcpyDeviceToHost);
        if (e == hipSuccess) e = hipMemcpy(h1.data(), p1, v3, hipMemcpyDeviceToHost);
        if (e == hipSuccess) e = hipMemcpy(h2.data(), p2, v3, hipMemcpyDeviceToHost);
        if (e == hipSuccess) e = hipMemcpy(hm.data(), material, sizeof(int) * ntri, hipMemcpyDeviceToHost);
        if (e != hipSuccess) return fail(arc::hip_fail(ctx, e, "arc_trace_scene_create", __FILE__, __LINE__));
    }
    // Leaves are triangle pieces: a triangle larger than the median
    // triangle is split along its box's longest axis into up to kMaxPieces
    // slabs (early split clipping), each piece boxed by the triangle clipped
    // to its slab.  Rays leaving a surface start inside the boxes of every
    // large triangle around them and must open all of them; smaller boxes
    // mean fewer.  The clipping runs in double and the boxes are rounded
    // outward, so a piece's box always holds its part of the triangle.
    std::vector<float> plo, phi;
    std::vector<int> ptri;
    {
        std::vector<double> ext(ntri);
        for (int i = 0; i < ntri; ++i) {
            const double e0 = std::max({h0[i].x, h1[i].x, h2[i].x}) - std::min({h0[i].x, h1[i].x, h2[i].x});
            const double e1 = std::max({h0[i].y, h1[i].y, h2[i].y}) - std::min({h0[i].y, h1[i].y, h2[i].y});
            const double e2 = std::max({h0[i].z, h1[i].z, h2[i].z}) - std::min({h0[i].z, h1[i].z, h2[i].z});
            ext[i] = std::max({e0, e1, e2});
        }
        std::vector<double> sorted = ext;
        std::nth_element(sorted.begin(), sorted.begin() + ntri / 2, sorted.end());
        const double unit = sorted[ntri / 2];
        struct D3 { double v[3]; };
        struct Poly {  // a triangle clipped twice has at most 5 corners; 8 leave room for rounding
            D3 at[8];
            int n = 0;
            void add(const D3& p) { if (n < 8) at[n++] = p; }
        };
        auto clip = [](const Poly& in, int a, double c, bool keep_ge) {
            Poly out;
            for (int k = 0; k < in.n; ++k) {
                const D3& p = in.at[k];
                const D3& q = in.at[k + 1 < in.n ? k + 1 : 0];
                const bool pin = keep_ge ? p.v[a] >= c : p.v[a] <= c;
                const bool qin = keep_ge ? q.v[a] >= c : q.v[a] <= c;
                if (pin) out.add(p);
                if (pin != qin) {
                    const double t = (c - p.v[a]) / (q.v[a] - p.v[a]);
                    D3 r;
                    for (int d = 0; d < 3; ++d) r.v[d] = p.v[d] + t * (q.v[d] - p.v[d]);
                    r.v[a] = c;
                    out.add(r);
                }
            }
            return out;
        };
        auto push = [&](int i, const double lo[3], const double hi[3], double pad) {
            for (int d = 0; d < 3; ++d) {
                plo.push_back(std::nextafter((float)(lo[d] - pad), -INFINITY));
                phi.push_back(std::nextafter((float)(hi[d] + pad), INFINITY));
            }
            ptri.push_back(i);
        };
        for (int i = 0; i < ntri; ++i) {
            const D3 v[3] = {{{h0[i].x, h0[i].y, h0[i].z}}, {{h1[i].x, h1[i].y, h1[i].z}},
                             {{h2[i].x, h2[i].y, h2[i].z}}};
            double blo[3], bhi[3];
            for (int d = 0; d < 3; ++d) {
                blo[d] = std::min({v[0].v[d], v[1].v[d], v[2].v[d]});
                bhi[d] = std::max({v[0].v[d], v[1].v[d], v[2].v[d]});
            }
            const double pad = 1e-6 * ext[i] + 1e-12;
            const int k = unit > 0.0 ? std::min(kMaxPieces, std::max(1, (int)std::ceil(ext[i] / unit))) : 1;
            if (k == 1) {
                push(i, blo, bhi, pad);
                continue;
            }
            int a = 0;
            for (int d = 1; d < 3; ++d)
                if (bhi[d] - blo[d] > bhi[a] - blo[a]) a = d;
            Poly whole;
            for (const D3& p : v) whole.add(p);
            for (int j = 0; j < k; ++j) {
                const double lo_a = blo[a] + (bhi[a] - blo[a]) * j / k;
                const double hi_a = j == k - 1 ? bhi[a] : blo[a] + (bhi[a] - blo[a]) * (j + 1) / k;
                const Poly poly = clip(clip(whole, a, lo_a, true), a, hi_a, false);
                double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
                for (int q = 0; q < poly.n; ++q)
                    for (int d = 0; d < 3; ++d) {
                        lo[d] = std::min(lo[d], poly.at[q].v[d]);
                        hi[d] = std::max(hi[d], poly.at[q].v[d]);
                    }
                if (poly.n == 0)  // rounding only: keep the whole triangle box within the slab
                    for (int d = 0; d < 3; ++d) {
                        lo[d] = blo[d];
                        hi[d] = bhi[d];
                    }
                lo[a] = lo_a;
                hi[a] = hi_a;
                push(i, lo, hi, pad);
            }
        }
    }
    const int np = (int)ptri.size();
    sc->nleaf = np;
    std::vector<arc_material> table(256);
    std::vector<int> emis(256, 0);
    for (int k = 0; k < num_materials; ++k) {
        table[k] = materials[k];
        const arc_float3 em = materials[k].emissive;
        emis[k] = (em.x * em.x + em.y * em.y + em.z * em.z) > 0.f ? 1 : 0;  // glm::length(emissive) > 0
    }
    int st = arc::ensure(ctx, sc->mats, sizeof(arc_material) * 256);
    if (st == ARC_OK) st = arc::ensure(ctx, sc->emissive, sizeof(int) * 256);
    if (st == ARC_OK) st = arc::ensure(ctx, sc->tri, sizeof(float4) * 4 * (size_t)ntri);
    arc::DevBuf staging;
    if (st == ARC_OK) st = arc::ensure(ctx, staging, 3 * v3 + sizeof(int) * (size_t)ntri);
    if (st != ARC_OK) {
        arc::release(staging);
        return fail(st);
    }
    char* base = staging.as<char>();
    f3* d0 = reinterpret_cast<f3*>(base);
    f3* d1 = reinterpret_cast<f3*>(base + v3);
    f3* d2 = reinterpret_cast<f3*>(base + 2 * v3);
    int* dm = reinterpret_cast<int*>(base + 3 * v3);
    e = hipMemcpy(d0, h0.data(), v3, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(d1, h1.data(), v3, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(d2, h2.data(), v3, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dm, hm.data(), sizeof(int) * ntri, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(sc->mats.p, table.data(), sizeof(arc_material) * 256, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(sc->emissive.p, emis.data(), sizeof(int) * 256, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        arc::release(staging);
        return fail(arc::hip_fail(ctx, e, "arc_trace_scene_create", __FILE__, __LINE__));
    }
    // the tree: binned SAH over the pieces' boxes, built once on the host
    std::vector<int> order;
    std::vector<arc_bvh_node> hn;
    sah_build(plo, phi, order, hn);
    hipLaunchKernelGGL(k_pack_tris, dim3(blocks(ntri)), dim3(kThreads), 0, ctx->stream, d0, d1, d2, dm,
                       sc->emissive.as<int>(), ntri, sc->tri.as<float4>());
    if (hipGetLastError() != hipSuccess) st = ARC_E_HIP;
    sc->max_depth = tree_depth(hn);
    if (st == ARC_OK && sc->max_depth >= kTraceStack)
        st = arc::fail(ctx, ARC_E_UNSUPPORTED, "triangle tree deeper than the traversal stack");
    if (st == ARC_OK) {
        std::vector<float4> wide;
        wide_nodes(hn, order, plo, phi, ptri, wide, sc->stack);
        sc->nnodes = (int)(wide.size() / 16);
        st = arc::ensure(ctx, sc->nodes, sizeof(float4) * wide.size());
        if (st == ARC_OK) {
            e = hipMemcpy(sc->nodes.p, wide.data(), sizeof(float4) * wide.size(), hipMemcpyHostToDevice);
            if (e != hipSuccess) st = arc::hip_fail(ctx, e, "arc_trace_scene_create", __FILE__, __LINE__);
        }
    }
    if (st == ARC_OK) {
        e = hipStreamSynchronize(ctx->stream);
        if (e != hipSuccess) st = arc::hip_fail(ctx, e, "arc_trace_scene_create", __FILE__, __LINE__);
    }
    arc::release(staging);
    if (st != ARC_OK) return fail(st);
    *out = sc;
    return ARC_OK;
}

void arc_trace_scene_destroy(arc_trace_scene* sc) {
    if (!sc) return;
    if (sc->ctx && sc->ctx->stream) (void)hipStreamSynchronize(sc->ctx->stream);
    arc::release(sc->tri);
    arc::release(sc->nodes);
    arc::release(sc->mats);
    arc::release(sc->emissive);
    arc::release(sc->count);
    arc::release(sc->stage);
    arc::release(sc->path_offset);
    arc::release(sc->scan_blocks);
    arc::release(sc->out);
    delete sc;
}

int arc_trace_intersect(arc_trace_scene* sc, const arc_float3* org, const arc_float3* dir, int n, float* t,
                        int* tri_index) {
    if (!sc || n < 0 || (n > 0 && (!org || !dir || !t || !tri_index))) return ARC_E_INVALID;
    if (n == 0) return ARC_OK;
    arc_ctx* ctx = sc->ctx;
    const bool together = arc::rays_together(arc::Rays::kAny, n, sc->nnodes);
    const int per = together ? kWave : kGroups;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((n + per - 1) / per), dim3(kWave), stack_bytes(sc), ctx->stream, scene_dev(sc),
                           reinterpret_cast<const f3*>(org), reinterpret_cast<const f3*>(dir), n, t, tri_index);
    };
    if (together) launch(k_intersect<1>);
    else launch(k_intersect<kGroup>);
    ARC_LAUNCHED(ctx);
    return ARC_OK;
}

int arc_trace_shoot(arc_trace_scene* sc, const arc_area_light* light, int num_paths, uint64_t seed, int flags,
                    arc_avpls* out, int* num_indirect) {
    if (!sc || !light || !out || !num_indirect || num_paths < 0) return ARC_E_INVALID;
    arc_ctx* ctx = sc->ctx;
    *num_indirect = 0;
    // light frame (AreaLight::updateWorldTransform: lookAt towards -front)
    const float fl = std::sqrt(light->front.x * light->front.x + light->front.y * light->front.y +
                               light->front.z * light->front.z);
    if (!(fl > 0.f) || !(light->width > 0.f) || !(light->height > 0.f) || light->materialIndex < 0 ||
        light->materialIndex > 255)
        return arc::fail(ctx, ARC_E_INVALID, "area light");
    Light L;
    L.center = mk(light->center.x, light->center.y, light->center.z);
    L.front = mk(light->front.x / fl, light->front.y / fl, light->front.z / fl);
    {
        const float fx = -L.front.x, fy = -L.front.y, fz = -L.front.z;  // lookAt forward
        const float ux = light->up.x, uy = light->up.y, uz = light->up.z;
        float sx = fy * uz - fz * uy, sy = fz * ux - fx * uz, sz = fx * uy - fy * ux;  // cross(f, up)
        const float sl = std::sqrt(sx * sx + sy * sy + sz * sz);
        if (!(sl > 0.f)) return arc::fail(ctx, ARC_E_INVALID, "area light: up parallel to front");
        sx /= sl; sy /= sl; sz /= sl;
        L.s = mk(sx, sy, sz);
        L.u = mk(sy * fz - sz * fy, sz * fx - sx * fz, sx * fy - sy * fx);  // cross(s, f)
    }
    L.half_w = 0.5f * light->width;
    L.half_h = 0.5f * light->height;
    L.area = light->width * light->height;
    L.radiance = mk(light->radiance.x, light->radiance.y, light->radiance.z);
    L.mat = light->materialIndex;
    const int explicit_direct = (flags & ARC_SHOOT_NO_EXPLICIT_DIRECT) ? 0 : 1;
    if (num_paths == 0) return ARC_OK;
    const size_t np = (size_t)num_paths;
    // per-path AVPL counts, and the shot's counters
    ARC_TRY(arc::ensure(ctx, sc->count, sizeof(int) * (np + 2)));
    int* count = sc->count.as<int>();
    int* counters = count + np;
    const SceneDev S = scene_dev(sc);
    auto stage_at = [&](arc::DevBuf& buf, size_t c) {
        char* b = buf.as<char>();
        Staged r;
        r.a.pos = reinterpret_cast<f3*>(b);
        r.a.nrm = r.a.pos + c;
        r.a.dir = r.a.nrm + c;
        r.a.rad = r.a.dir + c;
        r.a.anti = r.a.rad + c;
        r.a.mat = reinterpret_cast<int*>(r.a.anti + c);
        r.a.bounce = r.a.mat + c;
        r.path = r.a.bounce + c;
        return r;
    };
    const size_t slot_bytes = 5 * sizeof(f3) + 3 * sizeof(int);
    const bool together = arc::rays_together(arc::Rays::kPaths, num_paths, sc->nnodes);
    const int per = together ? kWave : kGroups;  // paths of a wave
    const int pblocks = std::min((num_paths + per - 1) / per, kPathBlocks);
    // a path makes 5 AVPLs at most on average (roulette at 0.8), and a wave
    // may leave a grab's rest unused
    size_t cap = std::min(std::max(8 * np + (size_t)kSlotGrab * pblocks, sc->stage.bytes / slot_bytes), (size_t)INT_MAX);
    Staged st{};
    unsigned staged = 0;
    for (;;) {  // a second time when the paths made more AVPLs than that
        ARC_TRY(arc::ensure(ctx, sc->stage, cap * slot_bytes));
        st = stage_at(sc->stage, cap);
        hipLaunchKernelGGL(k_paths_reset, dim3(1), dim3(1), 0, ctx->stream, counters, pblocks * per);
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(pblocks), dim3(kWave), stack_bytes(sc), ctx->stream, S, L, seed, num_paths,
                               explicit_direct, counters, reinterpret_cast<unsigned*>(counters + 1), (int)cap, count, st);
        };
        if (together) launch(k_paths<1>);
        else launch(k_paths<kGroup>);
        ARC_LAUNCHED(ctx);
        ARC_HIP(ctx, hipMemcpyAsync(&staged, counters + 1, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
        ARC_HIP(ctx, hipStreamSynchronize(ctx->stream));
        if ((size_t)staged <= cap) break;
        if (staged > (unsigned)INT_MAX) return arc::fail(ctx, ARC_E_UNSUPPORTED, "too many AVPLs");
        cap = std::min((size_t)staged + (size_t)staged / 8, (size_t)INT_MAX);
    }
    // per-path counts -> offsets -> AVPLs in path order
    const int nb = (num_paths + kScan - 1) / kScan;
    ARC_TRY(arc::ensure(ctx, sc->path_offset, sizeof(int) * (np + 1)));
    ARC_TRY(arc::ensure(ctx, sc->scan_blocks, sizeof(int) * ((size_t)nb + 1)));
    hipLaunchKernelGGL(k_scan_local, dim3(nb), dim3(kScan), 0, ctx->stream, count, num_paths,
                       sc->path_offset.as<int>(), sc->scan_blocks.as<int>());
    hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(kScan), 0, ctx->stream, sc->scan_blocks.as<int>(), nb);
    hipLaunchKernelGGL(k_scan_add, dim3(nb), dim3(kScan), 0, ctx->stream, sc->path_offset.as<int>(), num_paths,
                       sc->scan_blocks.as<int>(), nb);
    ARC_LAUNCHED(ctx);
    int total = 0;
    ARC_HIP(ctx, hipMemcpyAsync(&total, sc->path_offset.as<int>() + num_paths, sizeof(int), hipMemcpyDeviceToHost,
                                ctx->stream));
    ARC_HIP(ctx, hipStreamSynchronize(ctx->stream));
    const size_t v3 = sizeof(f3) * (size_t)std::max(total, 1), vi = sizeof(int) * (size_t)std::max(total, 1);
    ARC_TRY(arc::ensure(ctx, sc->out, 5 * v3 + 2 * vi));
    char* base = sc->out.as<char>();
    AvplOut o{reinterpret_cast<f3*>(base), reinterpret_cast<f3*>(base + v3), reinterpret_cast<f3*>(base + 2 * v3),
              reinterpret_cast<f3*>(base + 3 * v3), reinterpret_cast<f3*>(base + 4 * v3),
              reinterpret_cast<int*>(base + 5 * v3), reinterpret_cast<int*>(base + 5 * v3 + vi)};
    if (staged > 0) {
        hipLaunchKernelGGL(k_path_scatter, dim3(blocks((int)staged)), dim3(kThreads), 0, ctx->stream, st, (int)staged,
                           sc->path_offset.as<int>(), o);
        ARC_LAUNCHED(ctx);
    }
    out->position = reinterpret_cast<const arc_float3*>(o.pos);
    out->normal = reinterpret_cast<const arc_float3*>(o.nrm);
    out->incDirection = reinterpret_cast<const arc_float3*>(o.dir);
    out->incRadiance = reinterpret_cast<const arc_float3*>(o.rad);
    out->antiradiance = reinterpret_cast<const arc_float3*>(o.anti);
    out->materialIndex = o.mat;
    out->bounce = o.bounce;
    out->numAvpls = total;
    *num_indirect = total;
    return ARC_OK;
}

int arc_trace_gbuffer(arc_trace_scene* sc, arc_float3 camPos, arc_float3 forward, arc_float3 up, float fovy,
                      int width, int height, float* pos4, float* nrm4) {
    if (!sc || width <= 0 || height <= 0 || !pos4 || !nrm4 || !(fovy > 0.f) || !(fovy < 3.14159f))
        return ARC_E_INVALID;
    arc_ctx* ctx = sc->ctx;
    // camera basis: R = normalize(up x fwd), U = fwd x R
    const float fl = std::sqrt(forward.x * forward.x + forward.y * forward.y + forward.z * forward.z);
    if (!(fl > 0.f)) return ARC_E_INVALID;
    const float fx = forward.x / fl, fy = forward.y / fl, fz = forward.z / fl;
    float rx = up.y * fz - up.z * fy, ry = up.z * fx - up.x * fz, rz = up.x * fy - up.y * fx;
    const float rl = std::sqrt(rx * rx + ry * ry + rz * rz);
    if (!(rl > 0.f)) return ARC_E_INVALID;
    rx /= rl; ry /= rl; rz /= rl;
    const float ux = fy * rz - fz * ry, uy = fz * rx - fx * rz, uz = fx * ry - fy * rx;
    const float th = std::tan(0.5f * fovy), aspect = (float)width / (float)height;
    Camera cam{mk(camPos.x, camPos.y, camPos.z), mk(rx * th * aspect, ry * th * aspect, rz * th * aspect),
               mk(ux * th, uy * th, uz * th), mk(fx, fy, fz)};
    const bool together = arc::rays_together(arc::Rays::kCamera, (long long)width * height, sc->nnodes);
    const int gblocks = together ? ((width + 7) / 8) * ((height + 7) / 8) : ((width + 3) / 4) * ((height + 1) / 2);
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(gblocks), dim3(kWave), stack_bytes(sc), ctx->stream, scene_dev(sc), cam, width, height,
                           reinterpret_cast<float4*>(pos4), reinterpret_cast<float4*>(nrm4));
    };
    if (together) launch(k_gbuffer<1>);
    else launch(k_gbuffer<kGroup>);
    ARC_LAUNCHED(ctx);
    return ARC_OK;
}

int arc_trace_scene_info(arc_trace_scene* sc, int* num_triangles, int* tree_depth) {
    if (!sc) return ARC_E_INVALID;
    if (num_triangles) *num_triangles = sc->ntri;
    if (tree_depth) *tree_depth = sc->max_depth;
    return ARC_OK;
}

}  // extern "C"
