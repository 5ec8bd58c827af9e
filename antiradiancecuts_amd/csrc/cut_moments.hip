// The moment estimator of the error-bound light cut (ARC_ESTIMATOR_MOMENTS).
//
// The reference sums a kept cluster as its random representative times the
// cluster's radiance (kernel_bvh, cudaGather.cu:416-420; cluster(),
// bvh.cu:726-744).  The centroid estimator of gather_cut.hip replaces the
// representative by the node's centroid; on scenes whose AVPLs carry
// unrelated colours and normals both leave errors of several per cent,
// because a node's clamped cosines and its intensity differ per colour
// channel and the inverse-square falloff is convex over the node.  This
// estimator keeps, per internal node:
//
//   per RGB channel c, over the node's AVPLs j (I_jc = L_jc * diffuse / pi):
//     I_c = sum I_jc,  M_c = sum I_jc n_j,  T_c = sum I_jc n_j n_j^T
//   so that the AVPL-side sum  sum_j I_jc max(0, -n_j . d^)  is taken to
//   second order in spherical harmonics: max(0, t) ~ 3/32 + t/2 + 15/32 t^2
//   (the l <= 2 Legendre terms of the clamped cosine), i.e.
//     A_c(d^) = 3/32 I_c - 1/2 M_c . d^ + 15/32 d^T T_c d^;
//   and, over w_j = (I_jr + I_jg + I_jb) / 3, the node's position mean c and
//   covariance S, from which four points c + L v_k (L L^T = S, v_k the
//   vertices (1,1,1), (1,-1,-1), (-1,1,-1), (-1,-1,1) of a tetrahedron, whose
//   mean is 0 and mean outer product the identity) share the node's mean and
//   covariance: the pixel-side factor max(0, n_p . d) / |d|^3 averaged over
//   them is exact to second order in the node's extent.
//
// The estimate of a node is sum_c max(A_c(d^), 0) * K, with d^ the direction
// from the pixel to c and K the four-point average.  The records hold A_c / 4
// (the average's 1/4, which max(., 0) lets through) with its zz term folded
// into the constant by d^ . d^ = 1:
//   A_c / 4 = a_c + b_c . d^ + (txx - tzz) x^2 + (tyy - tzz) y^2 + 2 txy xy + ...
// with a_c = (3/32 I_c + tzz) / 4, b_c = -M_c / 8 and t = 15/128 T_c; the
// pixel then sums K over the four points without scaling.  Kept nodes of at most
// cutExactCount AVPLs are summed exactly over their leaves instead (their
// sorted leaves are contiguous, crec slots [first, first + count)).
//
// The sums come from FP64 prefix sums over the sorted leaves: a node's sum is
// the difference of two prefix rows at its leaf range (the Karras ranges),
// so no tree climb is needed and the covariance is formed in FP64.
#include <algorithm>
#include <climits>
#include <cmath>

#include "cut_common.hpp"

using namespace arc::cut;
using arc::CutPool;
using arc::CutView;

namespace {

constexpr int kMomTerms = 40;   // FP64 sums per leaf (see leaf_terms)
constexpr int kScanBlock = 256;  // leaves per block of the prefix scan
// float4 per internal node record:
//   0 (c, max_c I_c)             1 (s, first leaf, leaf count, -)
//   2-4 the four points, 12 floats   5-7 (b_c, a_c) per channel
//   8-12 per channel (txx - tzz, tyy - tzz, 0, 2txy, 2txz, 2tyz), 18 floats
constexpr int kMom = 13;
// float4 per internal node of the traversal's record, one 48-byte gather per
// node: (box min, max_c I_c), (box max, first leaf), (left, right, count, -)
constexpr int kTrav = 3;
constexpr int kMomStack = 64;    // per-wave stack of the serial traversal (deeper than any tree: 32 code bits + 25 index bits)

// Terms of leaf i of the sorted order (crec leaf record: r0 = position,
// r1 = unit normal, r2 = I), in four groups of ten:
//   group 0: w, w x, w y, w z, w (xx, yy, zz, xy, xz, yz)   (w = mean of I,
//            x relative to the centre of the root's box: smaller prefix
//            totals, less cancellation in a node's covariance)
//   group 1 + c (channel c): I_c, I_c n (3), I_c (nx nx, ny ny, nz nz,
//   nx ny, nx nz, ny nz).
constexpr int kGroup = 10;
constexpr int kGroups = kMomTerms / kGroup;
static_assert(kGroups * kGroup == kMomTerms, "four groups of ten terms");

__device__ inline void root_centre(const arc_bvh_node* __restrict__ nodes, double* ref) {
    const arc_bvh_node& b = nodes[0];
    ref[0] = 0.5 * ((double)b.bbMin.x + b.bbMax.x);
    ref[1] = 0.5 * ((double)b.bbMin.y + b.bbMax.y);
    ref[2] = 0.5 * ((double)b.bbMin.z + b.bbMax.z);
}

__device__ inline void leaf_terms(const float4* __restrict__ crec, int i, int group, const double* ref, double* t) {
    const float4* r = crec + kCrec * (size_t)i;
    if (group == 0) {
        const float4 r0 = r[0], r2 = r[2];
        const double x = r0.x - ref[0], y = r0.y - ref[1], z = r0.z - ref[2];
        const double w = ((double)r2.x + (double)r2.y + (double)r2.z) * (1.0 / 3.0);
        t[0] = w;
        t[1] = w * x; t[2] = w * y; t[3] = w * z;
        t[4] = w * x * x; t[5] = w * y * y; t[6] = w * z * z;
        t[7] = w * x * y; t[8] = w * x * z; t[9] = w * y * z;
    } else {
        const float4 r1 = r[1], r2 = r[2];
        const double nx = r1.x, ny = r1.y, nz = r1.z;
        const double I = group == 1 ? r2.x : group == 2 ? r2.y : r2.z;
        t[0] = I;
        t[1] = I * nx; t[2] = I * ny; t[3] = I * nz;
        t[4] = I * nx * nx; t[5] = I * ny * ny; t[6] = I * nz * nz;
        t[7] = I * nx * ny; t[8] = I * nx * nz; t[9] = I * ny * nz;
    }
}

// Inclusive prefix sums of one group of terms (blockIdx.y) within each
// block of kScanBlock leaves (pre, leaf-major: 40 doubles per leaf) and the
// block totals (tot, 40 per block).
__global__ __launch_bounds__(kScanBlock) void k_mom_scan(const float4* __restrict__ crec,
                                                         const arc_bvh_node* __restrict__ nodes, int n,
                                                         double* __restrict__ pre, double* __restrict__ tot) {
    __shared__ double wt[kScanBlock / 64][kGroup];
    const int i = blockIdx.x * kScanBlock + threadIdx.x;
    const int group = blockIdx.y;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double v[kGroup];
    if (i < n) {
        double ref[3];
        root_centre(nodes, ref);
        leaf_terms(crec, i, group, ref, v);
    } else {
#pragma unroll
        for (int k = 0; k < kGroup; ++k) v[k] = 0.0;
    }
#pragma unroll
    for (int k = 0; k < kGroup; ++k) {
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const double u = __shfl_up(v[k], off);
            if (lane >= off) v[k] += u;
        }
        if (lane == 63) wt[wave][k] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kGroup; ++k) {
        double add = 0.0;
        for (int w = 0; w < wave; ++w) add += wt[w][k];
        v[k] += add;
    }
    if (i < n) {
        double* o = pre + (size_t)kMomTerms * i + kGroup * group;
#pragma unroll
        for (int k = 0; k < kGroup; ++k) o[k] = v[k];
    }
    if (threadIdx.x == kScanBlock - 1) {
        double* o = tot + (size_t)kMomTerms * blockIdx.x + kGroup * group;
#pragma unroll
        for (int k = 0; k < kGroup; ++k) o[k] = v[k];
    }
}

// Block totals -> exclusive block offsets, one workgroup per term.
__global__ __launch_bounds__(kScanBlock) void k_mom_offsets(double* __restrict__ tot, int nblocks) {
    __shared__ double wt[kScanBlock / 64];
    __shared__ double carry_s;
    const int term = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double carry = 0.0;
    for (int base = 0; base < nblocks; base += kScanBlock) {
        const int j = base + threadIdx.x;
        const double x = j < nblocks ? tot[(size_t)kMomTerms * j + term] : 0.0;
        double v = x;
        for (int off = 1; off < 64; off <<= 1) {
            const double u = __shfl_up(v, off);
            if (lane >= off) v += u;
        }
        if (lane == 63) wt[wave] = v;
        __syncthreads();
        double add = 0.0;
        for (int w = 0; w < wave; ++w) add += wt[w];
        v += add;
        if (j < nblocks) tot[(size_t)kMomTerms * j + term] = carry + v - x;
        if (threadIdx.x == kScanBlock - 1) carry_s = v;
        __syncthreads();  // every lane has read wt and carry_s is written
        carry += carry_s;
        __syncthreads();  // carry_s read before the next chunk writes it
    }
}

// Sums of terms [k0, k0 + kGroup) over sorted leaves [first, last].
__device__ inline void range_group(const double* __restrict__ pre, const double* __restrict__ tot, int first,
                                   int last, int k0, double* S) {
    const double* hi = pre + (size_t)kMomTerms * last + k0;
    const double* th = tot + (size_t)kMomTerms * (last / kScanBlock) + k0;
#pragma unroll
    for (int k = 0; k < kGroup; ++k) S[k] = hi[k] + th[k];
    if (first > 0) {
        const double* lo = pre + (size_t)kMomTerms * (first - 1) + k0;
        const double* tl = tot + (size_t)kMomTerms * ((first - 1) / kScanBlock) + k0;
#pragma unroll
        for (int k = 0; k < kGroup; ++k) S[k] -= lo[k] + tl[k];
    }
}

// One record per internal node from the prefix rows at its leaf range, one
// group of terms at a time (the record's position part, then each channel).
__global__ __launch_bounds__(kScanBlock) void k_mom_nodes(const int* __restrict__ ranges,
                                                          const arc_bvh_node* __restrict__ nodes, int n,
                                                          const double* __restrict__ pre,
                                                          const double* __restrict__ tot, float4* __restrict__ mom,
                                                          float4* __restrict__ trav) {
    const int k = blockIdx.x * kScanBlock + threadIdx.x;
    if (k >= n - 1) return;
    const int first = ranges[2 * k], last = ranges[2 * k + 1];
    float4* o = mom + (size_t)kMom * k;
    double S[kGroup];
    range_group(pre, tot, first, last, 0, S);
    const arc_bvh_node& b = nodes[k];
    const double ex = (double)b.bbMax.x - b.bbMin.x, ey = (double)b.bbMax.y - b.bbMin.y,
                 ez = (double)b.bbMax.z - b.bbMin.z;
    const double s = 0.5 * sqrt(ex * ex + ey * ey + ez * ez);
    double cx, cy, cz, sxx = 0, syy = 0, szz = 0, sxy = 0, sxz = 0, syz = 0;
    if (S[0] > 0.0) {
        double ref[3];
        root_centre(nodes, ref);
        const double iw = 1.0 / S[0];
        const double ux = S[1] * iw, uy = S[2] * iw, uz = S[3] * iw;  // relative to ref
        sxx = fmax(S[4] * iw - ux * ux, 0.0);
        syy = fmax(S[5] * iw - uy * uy, 0.0);
        szz = fmax(S[6] * iw - uz * uz, 0.0);
        sxy = S[7] * iw - ux * uy;
        sxz = S[8] * iw - ux * uz;
        syz = S[9] * iw - uy * uz;
        cx = ref[0] + ux; cy = ref[1] + uy; cz = ref[2] + uz;
    } else {  // no intensity: the estimate is 0 wherever the point is
        cx = 0.5 * ((double)b.bbMin.x + b.bbMax.x);
        cy = 0.5 * ((double)b.bbMin.y + b.bbMax.y);
        cz = 0.5 * ((double)b.bbMin.z + b.bbMax.z);
    }
    // Cholesky factor of the covariance, pivoted: the axis of largest
    // variance first, so that the small and noisy entries of a flat or
    // collinear node (FP64 prefix differences) never divide a large one; a
    // pivot below tol ends its column
    auto var = [&](int i) -> double { return i == 0 ? sxx : i == 1 ? syy : szz; };
    int a0 = 0;
    if (syy > var(a0)) a0 = 1;
    if (szz > var(a0)) a0 = 2;
    int a1 = a0 == 0 ? 1 : 0, a2 = 3 - a0 - a1;
    if (var(a2) > var(a1)) {
        const int t = a1;
        a1 = a2;
        a2 = t;
    }
    auto cov = [&](int i, int j) -> double {  // i != j
        const int m = i + j;  // 1: xy, 2: xz, 3: yz
        return m == 1 ? sxy : m == 2 ? sxz : syz;
    };
    // (a variance below 1e-6 of the trace is prefix-difference noise: with
    // 1e6 leaves a prefix total carries about 1e-16 x 4e4 / W of it)
    const double tol = 1e-6 * (sxx + syy + szz) + 1e-300;
    double L00 = 0, L10 = 0, L20 = 0, L11 = 0, L21 = 0, L22 = 0;
    if (var(a0) > tol) {
        L00 = sqrt(var(a0));
        L10 = cov(a1, a0) / L00;
        L20 = cov(a2, a0) / L00;
        const double p11 = var(a1) - L10 * L10;
        if (p11 > tol) {
            L11 = sqrt(p11);
            L21 = (cov(a2, a1) - L20 * L10) / L11;
        }
        L22 = sqrt(fmax(var(a2) - L20 * L20 - L21 * L21, 0.0));
    }
    const double vs[4][3] = {{1, 1, 1}, {1, -1, -1}, {-1, 1, -1}, {-1, -1, 1}};
    float pts[12];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        // offsets along the pivot order (a0, a1, a2), put back on x, y, z
        const double u0 = L00 * vs[q][0];
        const double u1 = L10 * vs[q][0] + L11 * vs[q][1];
        const double u2 = L20 * vs[q][0] + L21 * vs[q][1] + L22 * vs[q][2];
        const double ox = a0 == 0 ? u0 : a1 == 0 ? u1 : u2;
        const double oy = a0 == 1 ? u0 : a1 == 1 ? u1 : u2;
        const double oz = a0 == 2 ? u0 : a1 == 2 ? u1 : u2;
        pts[3 * q] = (float)(cx + ox);
        pts[3 * q + 1] = (float)(cy + oy);
        pts[3 * q + 2] = (float)(cz + oz);
    }
    o[1] = make_float4((float)s, __int_as_float(first), __int_as_float(last - first + 1), 0.f);
    o[2] = make_float4(pts[0], pts[1], pts[2], pts[3]);
    o[3] = make_float4(pts[4], pts[5], pts[6], pts[7]);
    o[4] = make_float4(pts[8], pts[9], pts[10], pts[11]);
    // per channel: A_c(d^) / 4 = 3/128 I_c + (-1/8 M_c) . d^ + d^T (15/128 T_c) d^,
    // the off-diagonal T terms doubled so that the form is a plain dot
    // product with (dx^2, dy^2, dz^2, dx dy, dx dz, dy dz), and the zz term
    // moved into the constant (dz^2 = 1 - dx^2 - dy^2 for a unit d^)
    float* tf = reinterpret_cast<float*>(o + 8);
    double Ib = 0.0;
#pragma unroll 1
    for (int c = 0; c < 3; ++c) {
        range_group(pre, tot, first, last, kGroup * (1 + c), S);
        Ib = fmax(Ib, S[0]);
        const double f = 0.25 * 0.46875;
        o[5 + c] = make_float4((float)(-0.125 * S[1]), (float)(-0.125 * S[2]), (float)(-0.125 * S[3]),
                               (float)(0.25 * 0.09375 * S[0] + f * S[6]));
        tf[6 * c + 0] = (float)(f * (S[4] - S[6]));
        tf[6 * c + 1] = (float)(f * (S[5] - S[6]));
        tf[6 * c + 2] = 0.f;
        tf[6 * c + 3] = (float)(2.0 * f * S[7]);
        tf[6 * c + 4] = (float)(2.0 * f * S[8]);
        tf[6 * c + 5] = (float)(2.0 * f * S[9]);
    }
    tf[18] = 0.f;
    tf[19] = 0.f;
    o[0] = make_float4((float)cx, (float)cy, (float)cz, (float)Ib);
    float4* t = trav + (size_t)kTrav * k;
    t[0] = make_float4(b.bbMin.x, b.bbMin.y, b.bbMin.z, (float)Ib);
    t[1] = make_float4(b.bbMax.x, b.bbMax.y, b.bbMax.z, __int_as_float(first));
    t[2] = make_float4(__int_as_float(b.left), __int_as_float(b.right), __int_as_float(last - first + 1), 0.f);
}

// Squared distances carry 1e-24 (the first addend of their FMA chain) before
// their reciprocal square root: 1e36 bounds the cube of the result, at a
// point that coincides with the pixel the numerators (a cosine times |d|, or
// |d|^2) are 0, and above 1e-17 the addend is below half an ulp.
constexpr float kDistFloor2 = 1e-24f;

__device__ inline float dist2(float dx, float dy, float dz, float floor2) {
    return fmaf(dz, dz, fmaf(dy, dy, fmaf(dx, dx, floor2)));
}

// max(0, n_p . d) / |d|^3 at point x: the pixel-side cosine over the squared
// distance (cudaGather.cu:45-57, pixel factor), as the cosine n_p . d / |d|
// clamped to [0, 1] (the multiply's output clamp; it is at most 1 to
// rounding) times 1 / |d|^2.
__device__ inline float pixel_g(const PixelF& P, const float4& x) {
    const float dx = x.x - P.px, dy = x.y - P.py, dz = x.z - P.pz;
    const float inv = __builtin_amdgcn_rsqf(dist2(dx, dy, dz, kDistFloor2));
    const float c = __builtin_amdgcn_fmed3f((P.nx * dx + P.ny * dy + P.nz * dz) * inv, 0.f, 1.f);
    return c * (inv * inv);
}

// The node's estimate for the pixel, per channel, added to the pixel's sums.
__device__ inline void add_moments(const PixelF& P, const float4* __restrict__ r, Acc& acc) {
    // Records are read in three groups, each just before its use: fewer of
    // them are live at once in scalar registers.
    auto ld = [&](int i) { return uload4(uptr(r + i)); };
    const float4 m0 = ld(0), p01 = ld(2), p12 = ld(3), p23 = ld(4);
    const float K = pixel_g(P, make_float4(p01.x, p01.y, p01.z, 0.f)) +
                    pixel_g(P, make_float4(p01.w, p12.x, p12.y, 0.f)) +
                    pixel_g(P, make_float4(p12.z, p12.w, p23.x, 0.f)) +
                    pixel_g(P, make_float4(p23.y, p23.z, p23.w, 0.f));
    const float dx = m0.x - P.px, dy = m0.y - P.py, dz = m0.z - P.pz;
    const float inv = __builtin_amdgcn_rsqf(dist2(dx, dy, dz, kDistFloor2));
    const float i2 = inv * inv;
    const float xx = dx * dx, yy = dy * dy, xy = dx * dy, xz = dx * dz, yz = dy * dz;
    const float4 mr = ld(5), mg = ld(6), mb = ld(7);
    const float4 t0 = ld(8), t1 = ld(9), t2 = ld(10), t3 = ld(11), t4 = ld(12);
    // (the zz coefficients t0.z, t2.x and t3.z are 0: folded into the constants)
    const float qr = t0.x * xx + t0.y * yy + t0.w * xy + t1.x * xz + t1.y * yz;
    const float qg = t1.z * xx + t1.w * yy + t2.y * xy + t2.z * xz + t2.w * yz;
    const float qb = t3.x * xx + t3.y * yy + t3.w * xy + t4.x * xz + t4.y * yz;
    const float ar = mr.w + inv * (mr.x * dx + mr.y * dy + mr.z * dz) + i2 * qr;
    const float ag = mg.w + inv * (mg.x * dx + mg.y * dy + mg.z * dz) + i2 * qg;
    const float ab = mb.w + inv * (mb.x * dx + mb.y * dy + mb.z * dz) + i2 * qb;
    acc.s0 += fmaxf(ar, 0.f) * K;
    acc.s1 += fmaxf(ag, 0.f) * K;
    acc.s2 += fmaxf(ab, 0.f) * K;
    ++acc.run;
}

// G of one leaf (an AVPL with a unit normal n_a) for the pixel:
// max(0, n . d) max(0, -n_a . d) / |d|^4 (cudaGather.cu:45-57), from one
// reciprocal of |d|^2.  With unit normals the cosines need no clamp at 1;
// |d|^2 carries 1e-18 (below half an ulp from 1e-11 up), and coincident
// points give 0, as both cosines vanish there.
__device__ inline float leaf_g(const PixelF& P, const float4& r0, const float4& r1) {
    const float dx = r0.x - P.px, dy = r0.y - P.py, dz = r0.z - P.pz;
    const float dd = dist2(dx, dy, dz, 1e-18f);
    const float u1 = fmaxf(P.nx * dx + P.ny * dy + P.nz * dz, 0.f);
    const float u2 = fmaxf(-(r1.x * dx + r1.y * dy + r1.z * dz), 0.f);
    const float r = __builtin_amdgcn_rcpf(dd);
    return (u1 * u2) * (r * r);
}

// The Lightcuts bound of a node for the pixel (node_bound) with one
// transcendental: 1 / dmin^2 as the square of 1 / dmin.  The cosine bound
// min(1, hmax / dmin), 0 where hmax <= 0, is hmax / dmin clamped to [0, 1]
// (the multiply's output clamp).
__device__ inline float node_bound1(const PixelF& P, const arc_bvh_node& b, float ilum, float delta2) {
    const float ex = fmaxf(fmaxf(b.bbMin.x - P.px, P.px - b.bbMax.x), 0.f);
    const float ey = fmaxf(fmaxf(b.bbMin.y - P.py, P.py - b.bbMax.y), 0.f);
    const float ez = fmaxf(fmaxf(b.bbMin.z - P.pz, P.pz - b.bbMax.z), 0.f);
    const float dmin2 = fmaxf(ex * ex + ey * ey + ez * ez, delta2);
    const float hmax = P.nx * (P.nx > 0.f ? b.bbMax.x - P.px : b.bbMin.x - P.px) +
                       P.ny * (P.ny > 0.f ? b.bbMax.y - P.py : b.bbMin.y - P.py) +
                       P.nz * (P.nz > 0.f ? b.bbMax.z - P.pz : b.bbMin.z - P.pz);
    const float ri = __builtin_amdgcn_rsqf(dmin2);
    return ilum * __builtin_amdgcn_fmed3f(hmax * ri, 0.f, 1.f) * (ri * ri);
}

// Inclusive sum over the wave's lanes.
__device__ inline int wave_inclusive_sum(int v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int u = __shfl_up(v, off, 64);
        if (lane >= off) v += u;
    }
    return v;
}

__device__ inline int lane_below(uint64_t m) {  // set bits of m below this lane
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// The leaves of nx exact ranges (first << 7 | (count - 1), contiguous sorted
// leaves), at most `most` of them from the from-th on (a multiple of 64), 64
// at a time, one per lane.  A lane's range among those of the
// batch: the ranges that start inside it mark their first lane in LDS, and a
// lane counts the marks up to its own (14 instructions per 64 leaves, where a
// binary search over the ranges' prefix counts takes 56).  Each lane tests its
// leaf against the tile: an AVPL that faces away from every pixel adds 0 to
// every sum (its cosine max(0, n_a . (p - x_a)) is 0), and about half of the
// leaves do (a surface's AVPLs seen from behind).  tb = (centre, half extent)
// of the tile's box: the largest n_a . (p - x_a) over it is n_a . (c - x_a) +
// |n_a| . e, compared with a margin above FP32 rounding.  stage(facing, r0, r1,
// r2) gets each lane's leaf record and whether it can face some pixel, sum()
// follows: the next 64 records are fetched between them, into the registers that
// stage has read.
template <class Stage, class Sum>
__device__ inline void walk_ranges(const float4* __restrict__ crec, const uint32_t* X, int nx, int from, int most,
                                   int* pfx, unsigned char* mark, const float* tb, Stage stage, Sum sum) {
    const int lane = threadIdx.x & 63;
    const int c0 = lane < nx ? (int)(X[lane] & 127u) + 1 : 0;
    const int c1 = lane + 64 < nx ? (int)(X[lane + 64] & 127u) + 1 : 0;
    int s0 = wave_inclusive_sum(c0);
    const int t0 = __builtin_amdgcn_readlane(s0, 63);
    int s1 = wave_inclusive_sum(c1) + t0;
    const int leaves = __builtin_amdgcn_readlane(s1, 63);
    const int total = leaves - from > most ? from + most : leaves;
    s0 = lane < nx ? s0 - c0 : INT_MAX;       // where the range in X[lane] starts
    s1 = lane + 64 < nx ? s1 - c1 : INT_MAX;  // and the one in X[lane + 64]
    pfx[lane] = s0;  // kept in LDS: registers are short
    pfx[lane + 64] = s1;
    const float scale = fabsf(tb[0]) + fabsf(tb[1]) + fabsf(tb[2]) + tb[3] + tb[4] + tb[5];
    float4 b0 = make_float4(0.f, 0.f, 0.f, 0.f), b1 = b0, b2 = b0;
    int before = __popcll(__ballot(s0 < from)) + __popcll(__ballot(s1 < from));  // ranges that start before the batch
    auto fetch = [&](int base) {
        mark[lane] = 0;
        __builtin_amdgcn_wave_barrier();  // the wave's LDS writes come before its reads of other lanes' slots
        const unsigned at0 = (unsigned)(pfx[lane] - base), at1 = (unsigned)(pfx[lane + 64] - base);
        if (at0 < 64u) mark[at0] = 1;
        if (at1 < 64u) mark[at1] = 1;
        __builtin_amdgcn_wave_barrier();
        const uint64_t m = __ballot(mark[lane] != 0);
        const int g = base + lane;
        if (g < total) {
            const int r = before - 1 + lane_below(m) + (int)((m >> lane) & 1);
            const float4* l = crec + kCrec * (size_t)((int)(X[r] >> 7) + (g - pfx[r]));
            b0 = l[0];
            b1 = l[1];
            b2 = l[2];
        }
        before += __popcll(m);
    };
    fetch(from);
#pragma unroll 1
    for (int base = from; base < total; base += 64) {
        const float dx = tb[0] - b0.x, dy = tb[1] - b0.y, dz = tb[2] - b0.z;
        const float reach = b1.x * dx + b1.y * dy + b1.z * dz + fabsf(b1.x) * tb[3] + fabsf(b1.y) * tb[4] +
                            fabsf(b1.z) * tb[5];
        const float margin = 1e-5f * (scale + fabsf(b0.x) + fabsf(b0.y) + fabsf(b0.z));
        const bool facing = base + lane < total && reach > -margin;
        stage(facing, b0, b1, b2);
        if (base + 64 < total) fetch(base + 64);  // in flight while these are summed
        sum();
    }
}

// ---- the cut ----------------------------------------------------------------
//
// Per 8x8 tile: a node is refined when any of the tile's pixels asks for it;
// kept nodes are summed with the moment estimate, or exactly when they hold
// at most exact_count AVPLs.  criterion: ARC_CRITERION_BOUND (bound >
// threshold) or ARC_CRITERION_EXPANSION (s > opening * d_c, or bound *
// (s / d_c)^2 > threshold).
//
//   k_cut_decide   finds each tile's cut and writes it to a pool of chunks:
//                  kKeep kept nodes, or kKeep exact ranges, which are as many
//                  chunks as they hold times kChunkLeaves leaves;
//   k_cut_eval     sums the chunks, a wave per chunk whatever tile it belongs
//                  to, into 64 x 3 partial sums each;
//   k_cut_serial   the tiles that found the pool full, and all tiles where most
//                  would meet their budget (serial_cut): the depth-first cut of
//                  one node at a time, summed as it goes;
//   k_cut_combine  adds each tile's partial sums in the order of its chunks.
//
// One wave that walked its tile's cut node by node and summed it as it went
// paid a dependent record load and a 64-pixel test per node, and the tile
// with the largest cut set the kernel's time: with 375 tiles on 1024 SIMDs
// (200x120 pixels) that was 1.8 ms.
constexpr int kKeep = 128;
// A small image over a small tree has few range chunks: with 2048 leaves in one
// and 5700 chunks for 8192 waves, some CUs held a full set and others none
// (600x300 pixels, 4000 AVPLs, exact up to 128: 431 us for 120 us of vector
// work, 0.67 ms a frame; 0.59 with 1024 leaves, 0.60 with 512, whose parts scan
// their ranges too often).
constexpr int kChunkLeaves = 1024;
constexpr int kNextCounters = 8, kNextStride = 32;  // the counters of k_cut_eval's chunks, a cache line each
constexpr int kPartBits = 5;        // a range chunk is kKeep ranges of at most 128 leaves: at most 32 parts
constexpr int kDecideStack = 640;   // pending nodes per wave
constexpr int kStackReserve = 64;   // of these for the depth-first descent when the rest is full (tree depth <= 57)
enum ChunkKind { kNodes = 0, kRanges = 1 };

__device__ inline float uniform_f(float v) { return __int_as_float(uniform(__float_as_int(v))); }

// The view of an item of the launch's tile list (kMany), or the only one.
template <bool kMany>
struct Views;
template <>
struct Views<false> {
    CutView one;
    __device__ CutView of(int) const { return one; }
};
template <>
struct Views<true> {
    const CutView* many;
    int n;
    __device__ CutView of(int item) const {
        int lo = 0, hi = n - 1;  // the last view whose tiles start at or before item
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (((uint_*)&many[mid].tile_base)[0] <= item) lo = mid;
            else hi = mid - 1;
        }
        CutView v;
        const ARC_UNIFORM_AS uint32_t* src = (const ARC_UNIFORM_AS uint32_t*)(many + lo);
        uint32_t* dst = reinterpret_cast<uint32_t*>(&v);
#pragma unroll
        for (size_t i = 0; i < sizeof(CutView) / 4; ++i) dst[i] = src[i];
        return v;
    }
};

// The view of an item, read again from the kernel's arguments (its first one is a
// Views): what a tile needs only at its start and end is then not held in
// between, where scalar registers are short and spill.
template <bool kMany>
__device__ inline CutView view_again(int item) {
    auto* args = (const ARC_UNIFORM_AS uint32_t*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(args));
    Views<kMany> w;
    uint32_t* dst = reinterpret_cast<uint32_t*>(&w);
#pragma unroll
    for (size_t i = 0; i < sizeof(w) / 4; ++i) dst[i] = args[i];
    return w.of(item);
}

__device__ inline Threshold view_threshold(const CutView& v) {
    Threshold th;
    th.est = v.th_est;
    th.sum = v.th_sum;
    th.eps = v.th_eps;
    th.floor_frac = v.th_floor;
    th.inv_npix = v.th_inv_npix;
    return th;
}

// Tile t of a view: its tile column and row.  The tile grid is the (2 gx) x
// (2 gy) tiles of gx x gy blocks of 16x16 pixels.
__device__ inline int tiles_wide(int W) { return 2 * ((W + 15) / 16); }

// A pixel as the decisions read it from LDS: (p, threshold), (max(n, 0), -),
// (min(n, 0), -).  A lane outside the image stands at pixel 0 with an infinite
// threshold: it never asks for a node, but a node in front of it is not
// dropped (it adds nothing to the image and counts towards the budget).
constexpr int kPixRec = 3;

// The Lightcuts bound of box (lo, hi) with intensity ilum at pixel record P,
// node_bound1's terms with the box corner per axis taken as
// max(n, 0) (hi - p) + min(n, 0) (lo - p).
__device__ inline float pixel_bound(const float4* P, const float4& lo, const float4& hi, float delta2, float& thr) {
    const float4 p = P[0], np = P[1], nm = P[2];
    thr = p.w;
    const float ax = lo.x - p.x, ay = lo.y - p.y, az = lo.z - p.z;
    const float bx = hi.x - p.x, by = hi.y - p.y, bz = hi.z - p.z;
    const float ex = fmaxf(fmaxf(ax, -bx), 0.f), ey = fmaxf(fmaxf(ay, -by), 0.f), ez = fmaxf(fmaxf(az, -bz), 0.f);
    const float dmin2 = fmaxf(ex * ex + ey * ey + ez * ez, delta2);
    const float hmax = np.x * bx + nm.x * ax + np.y * by + nm.y * ay + np.z * bz + nm.z * az;
    const float ri = __builtin_amdgcn_rsqf(dmin2);
    return lo.w * __builtin_amdgcn_fmed3f(hmax * ri, 0.f, 1.f) * (ri * ri);
}

__device__ inline float wave_fmin(float v) {
    for (int off = 32; off > 0; off >>= 1) v = fminf(v, __shfl_xor(v, off));
    return uniform_f(v);
}
__device__ inline float wave_fmax(float v) {
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
    return uniform_f(v);
}
__device__ inline int wave_isum(int v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return uniform(v);
}

// Whether some AVPL of a kept node can face some pixel of the tile (box
// centre tc, half extent te): the largest n_a . (p - x_a) over the node's
// normal box, its box and the tile's box, by interval products per axis, is
// not below 0 by more than FP32 rounding.  A node that fails adds 0 (its
// estimate would add only the clamped cosine's second-order residue).
__device__ inline bool node_faces(const float* tb, const float4& lo, const float4& hi, const float4& nl,
                                  const float4& nh) {
    float reach = 0.f, scale = 0.f;
    auto axis = [&](float c, float e, float plo, float phi, float nlo, float nhi) {
        const float vlo = (c - e) - phi, vhi = (c + e) - plo;  // p - x over the boxes
        reach += fmaxf(fmaxf(nlo * vlo, nlo * vhi), fmaxf(nhi * vlo, nhi * vhi));
        scale += fabsf(c) + e + fabsf(plo) + fabsf(phi);
    };
    axis(tb[0], tb[3], lo.x, hi.x, nl.x, nh.x);
    axis(tb[1], tb[4], lo.y, hi.y, nl.y, nh.y);
    axis(tb[2], tb[5], lo.z, hi.z, nl.z, nh.z);
    return reach > -1e-5f * scale;
}

// A tile's cost where it is cut serially, in vector instructions: a bound test
// is about 30, an estimate 130, a queued exact leaf 18 (26 a pair for the half
// that face the tile, a few for the rest), and the pixel's own loads and stores.
__device__ inline float tile_cost(int tested, int kept, int leaves) {
    return 300.f + 30.f * (float)tested + 130.f * (float)kept + 18.f * (float)leaves;
}

// The k-th tile of a launch in no order: of one view's a block's four are a 16x16-pixel
// block, neighbouring blocks on one XCD.
template <bool kMany>
__device__ inline int unordered_item(const Views<kMany>& views, int wave, int k) {
    if constexpr (kMany) {
        return k;
    } else {
        const int gx = (views.one.W + 15) / 16, gy = (views.one.H + 15) / 16;
        const int b = xcd_block(blockIdx.x, gx * gy);
        return uniform(((b / gx) * 2 + (wave >> 1)) * 2 * gx + (b % gx) * 2 + (wave & 1));
    }
}

// One wave's working memory of k_cut_decide.
struct DecideLds {
    int stack[kDecideStack];  // pending internal nodes
    int amb[128];             // nodes whose decision needs every pixel
    int keep[kKeep + 64];     // kept nodes, flushed in chunks of kKeep
    uint32_t ex[2 * kKeep];   // exact ranges first << 7 | (count - 1), flushed likewise
    float4 pix[64][kPixRec];
};

// The cut of one tile by one wave, 64 nodes at a time, one per lane.
//
// A lane first decides its node from the tile as a whole and a few of its
// pixels, which settles most nodes with a fraction of the 64-pixel test:
//   refined   when one of the sample pixels asks for it (any pixel may);
//   dropped   when the whole box lies behind every pixel's tangent plane (the
//             height over the planes, by interval products over the tile's
//             positions and normals, is below 0 by more than rounding);
//   kept      when the bound at the tile's nearest point with the interval
//             height is below the tile's smallest threshold, and some sample
//             pixel has the box in front of it.
// The rest are queued, and tested against all 64 pixels (from LDS) once 64 of
// them have come together.  Every decision is the one the pixels' bounds
// give: the tile's tests only settle nodes whose outcome they prove, with a
// margin above FP32 rounding.
//
// Bound by the VALU (about 200 instructions per 64 nodes for the first test,
// 30 per node for those that need every pixel) against 30 per node and a
// dependent load each for one node at a time.
template <bool kMany, bool kExpansion>
__global__ __launch_bounds__(kCutThreads) void k_cut_decide(Views<kMany> views, int nitems, CutPool pool) {
    __shared__ DecideLds lds[kCutThreads / 64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    int item;
    if constexpr (kMany) {
        item = uniform(blockIdx.x * (kCutThreads / 64) + wave);
        if (item >= nitems) return;  // the whole wave: no block barrier below
    } else {  // a block's four tiles are one 16x16-pixel block, neighbouring blocks on one XCD
        item = unordered_item(views, wave, 0);
    }
    const CutView v = views.of(item);
    const int t = item - (kMany ? v.tile_base : 0), tw = tiles_wide(v.W);
    const int x = (t % tw) * 8 + (lane & 7), y = (t / tw) * 8 + (lane >> 3);
    const bool live = x < v.W && y < v.H;
    const uint64_t alive = __ballot(live);
    if (alive == 0) {  // a tile of the 16x16 block outside the image
        if (lane == 0) pool.head[item] = -1;
        return;
    }
    if (kMany && v.budget < arc::kSerialBudget) {  // a view whose tiles are cut serially among others whose are not
        if (lane == 0) {
            pool.head[item] = -1;
            pool.serial[atomicAdd(pool.count + arc::kSerialTiles, 1)] = item;
            pool.evaluated[item] = -1;
        }
        return;
    }
    DecideLds& S = lds[wave];
    const bool outside = !((alive >> 63) & 1);  // some lane is outside the image
    const bool expansion = kExpansion && v.criterion == ARC_CRITERION_EXPANSION;
    const float delta2 = v.delta * v.delta;
    float tb[6], tlo[3], thi[3], nlo[3], nhi[3], thr_min;
    int rep[5];
    {
        const int q = live ? y * v.W + x : 0;
        const PixelF P = load_pixel(v.gpos, v.gnrm, v.galb, v.mats, q);
        const float thr = live ? view_threshold(v).at(q) : INFINITY;
        const float px = P.px, py = P.py, pz = P.pz;
        const float nx = P.nx, ny = P.ny, nz = P.nz;
        S.pix[lane][0] = make_float4(px, py, pz, thr);
        S.pix[lane][1] = make_float4(fmaxf(nx, 0.f), fmaxf(ny, 0.f), fmaxf(nz, 0.f), 0.f);
        S.pix[lane][2] = make_float4(fminf(nx, 0.f), fminf(ny, 0.f), fminf(nz, 0.f), 0.f);
        tlo[0] = wave_fmin(live ? px : INFINITY);
        tlo[1] = wave_fmin(live ? py : INFINITY);
        tlo[2] = wave_fmin(live ? pz : INFINITY);
        thi[0] = wave_fmax(live ? px : -INFINITY);
        thi[1] = wave_fmax(live ? py : -INFINITY);
        thi[2] = wave_fmax(live ? pz : -INFINITY);
        nlo[0] = wave_fmin(live ? nx : INFINITY);
        nlo[1] = wave_fmin(live ? ny : INFINITY);
        nlo[2] = wave_fmin(live ? nz : INFINITY);
        nhi[0] = wave_fmax(live ? nx : -INFINITY);
        nhi[1] = wave_fmax(live ? ny : -INFINITY);
        nhi[2] = wave_fmax(live ? nz : -INFINITY);
        thr_min = wave_fmin(thr);
        const uint64_t least = __ballot(live && thr <= thr_min);
        rep[0] = least ? __ffsll((unsigned long long)least) - 1 : __ffsll((unsigned long long)alive) - 1;
        // the corners; lane 63 also where it is outside the image (as it is whenever any lane is)
        rep[1] = 0;
        rep[2] = (alive >> 7) & 1 ? 7 : rep[0];
        rep[3] = (alive >> 56) & 1 ? 56 : rep[0];
        rep[4] = 63;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            tb[a] = 0.5f * (tlo[a] + thi[a]);
            tb[3 + a] = 0.5f * (thi[a] - tlo[a]);
        }
        if (lane == 0) {
            float* o = pool.tbox + 8 * (size_t)item;
#pragma unroll
            for (int a = 0; a < 6; ++a) o[a] = tb[a];
        }
    }
    __builtin_amdgcn_wave_barrier();  // the wave's pixel records before its reads of other lanes'

    int sp = 0, na = 0, ne = 0, nx = 0;             // wave-uniform queue lengths
    int ntest = 0, nvis = 0, nkeep = 0, nleaf = 0;  // wave-uniform counts
    int lexact = 0;                                 // per lane: AVPLs of the exact ranges this lane found
    int ldone = 0;                                  // per lane: AVPLs of the nodes it decided without refining
    int nbud = 0;                                   // nodes kept because the budget was spent
    int head = -1, last = -1;                       // the tile's chunks
    bool full = false, over = false;                // the pool has no room; the budget is reached

    int spare = 0, nspare = 0;  // chunks taken from the pool and not used yet
    // the next chunk, linked to the tile's: part `part` of the entries in chunk `from` (-1: its own); false: the pool is full
    auto chunk = [&](int kind, int cnt, int from, int part, int& c) {
        if (nspare == 0) {
            nspare = head < 0 ? pool.grab : 2 * pool.grab;
            int got = 0;
            if (lane == 0) got = atomicAdd(pool.count + arc::kTaken, nspare);
            spare = uniform(got);
        }
        c = spare;
        if (c >= pool.cap) return false;
        ++spare;
        --nspare;
        if (lane == 0) {
            pool.meta[c] = make_int4(item, kind | (cnt << 8), -1, ((from < 0 ? c : from) << kPartBits) + part);
            if (last >= 0) pool.meta[last].z = c;
        }
        if (head < 0) head = c;
        last = c;
        return true;
    };
    auto evaluated = [&]() { return nkeep + nleaf + wave_isum(lexact); };
    auto flush_keep = [&](int least) {
        while (ne >= least && ne > 0 && !full) {
            const int m = min(ne, kKeep);
            int c;
            if (!chunk(kNodes, m, -1, 0, c)) {
                full = true;
                return;
            }
            uint32_t* dst = pool.entries + (size_t)c * kKeep;
            if (lane < m) dst[lane] = (uint32_t)S.keep[lane];
            if (lane + 64 < m) dst[lane + 64] = (uint32_t)S.keep[lane + 64];
            const int rest = ne - m;  // < 64
            const int r = lane < rest ? S.keep[m + lane] : 0;
            __builtin_amdgcn_wave_barrier();
            if (lane < rest) S.keep[lane] = r;
            __builtin_amdgcn_wave_barrier();
            ne = rest;
        }
    };
    auto flush_ex = [&](int least) {
        while (nx >= least && nx > 0 && !full) {
            const int m = min(nx, kKeep);
            const uint32_t x0 = lane < m ? S.ex[lane] : 0u, x1 = lane + 64 < m ? S.ex[lane + 64] : 0u;
            int parts = 1;
            {
                const int leaves = (lane < m ? (int)(x0 & 127u) + 1 : 0) + (lane + 64 < m ? (int)(x1 & 127u) + 1 : 0);
                parts = (wave_isum(leaves) + kChunkLeaves - 1) / kChunkLeaves;
            }
            int c = -1, first = -1;
            for (int k = 0; k < parts; ++k) {
                if (!chunk(kRanges, m, first, k, c)) {
                    full = true;
                    return;
                }
                if (k == 0) first = c;
            }
            uint32_t* dst = pool.entries + (size_t)first * kKeep;
            if (lane < m) dst[lane] = x0;
            if (lane + 64 < m) dst[lane + 64] = x1;
            const int rest = nx - m;  // < kKeep
            const uint32_t r0 = lane < rest ? S.ex[m + lane] : 0u, r1 = lane + 64 < rest ? S.ex[m + lane + 64] : 0u;
            __builtin_amdgcn_wave_barrier();
            if (lane < rest) S.ex[lane] = r0;
            if (lane + 64 < rest) S.ex[lane + 64] = r1;
            __builtin_amdgcn_wave_barrier();
            nx = rest;
        }
    };
    // The decided nodes of a batch, one per lane: exact ranges, refined nodes
    // (their leaf children are exact ranges of one), kept nodes.
    auto apply = [&](int k, const float4& r0, const float4& r1, const float4& r2, bool exact, bool refine, bool keep) {
        const int first = __float_as_int(r1.w), l = __float_as_int(r2.x), r = __float_as_int(r2.y),
                  count = __float_as_int(r2.z);
        const uint64_t mx = __ballot(exact), mr = __ballot(refine), mk = __ballot(keep);
        ntest += __popcll(mr) + __popcll(mk);
        nvis += __popcll(mr);
        if (exact) {
            S.ex[nx + lane_below(mx)] = ((uint32_t)first << 7) | (uint32_t)(count - 1);
            lexact += count;
        }
        nx += __popcll(mx);
        if (mr) {
            const bool li = refine && l < 0, ri = refine && r < 0, ll = refine && l >= 0, rl = refine && r >= 0;
            const uint64_t mli = __ballot(li), mri = __ballot(ri), mll = __ballot(ll), mrl = __ballot(rl);
            if (li) S.stack[sp + lane_below(mli)] = -(l + 1);
            sp += __popcll(mli);
            if (ri) S.stack[sp + lane_below(mri)] = -(r + 1);
            sp += __popcll(mri);
            if (ll) S.ex[nx + lane_below(mll)] = (uint32_t)l << 7;
            nx += __popcll(mll);
            if (rl) S.ex[nx + lane_below(mrl)] = (uint32_t)r << 7;
            nx += __popcll(mrl);
            nleaf += __popcll(mll) + __popcll(mrl);
        }
        if (mk) {
            bool faces = false;
            if (keep) faces = node_faces(tb, r0, r1, v.nbox[2 * (size_t)k], v.nbox[2 * (size_t)k + 1]);
            const uint64_t mf = __ballot(faces);
            if (faces) S.keep[ne + lane_below(mf)] = k;
            ne += __popcll(mf);
            nkeep += __popcll(mf);
        }
        __builtin_amdgcn_wave_barrier();  // the queues' writes before other lanes read them
        if (ne >= kKeep || nx >= kKeep) {
            over = evaluated() >= v.budget;
            if (!over) {
                flush_keep(kKeep);
                flush_ex(kKeep);
            }
        }
    };
    // The whole subtree of node k, 64 nodes at a time.  False when the budget
    // is reached inside it or the pool is full.
    auto subtree = [&](int root) {
        const int base = sp;
        if (lane == 0) S.stack[sp] = root;
        ++sp;
        __builtin_amdgcn_wave_barrier();
        bool one = false;  // the stack is full: depth first, the node just queued before any other
        while (!over && !full) {
            const int room = kDecideStack - kStackReserve - sp;
            const bool every = one || (room >= 2 && (na >= 64 || sp == base));  // from every pixel
            if (every && na == 0) break;
            const int m = one ? 1 : every ? min(min(64, na), room / 2) : max(1, min(min(64, sp - base), room));
            const bool on = lane < m;
            const int k = !on ? 0 : every ? S.amb[na - 1 - lane] : S.stack[sp - 1 - lane];
            if (every) na -= m;
            else sp -= m;
            __builtin_amdgcn_wave_barrier();  // read before the slots are written over
            const float4* r = v.trav + (size_t)kTrav * k;
            const float4 r0 = r[0], r1 = r[1], r2 = r[2];
            float s2 = 0.f;
            float4 m0 = make_float4(0.f, 0.f, 0.f, 0.f);
            if (expansion) {
                const float4* mr = v.mom + (size_t)kMom * k;
                m0 = mr[0];
                s2 = mr[1].x * mr[1].x;
            }
            const bool small = __float_as_int(r2.z) <= v.exact_count;
            bool ask = false, front = false, exact, refine, keep, unsure = false;
            if (every) {
                for (int p = 0; p < 64; p += 4) {
        #pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        float thr;
                        const float4* P = S.pix[p + u];
                        const float b = pixel_bound(P, r0, r1, delta2, thr);
                        if (expansion) {
                            const float dx = m0.x - P[0].x, dy = m0.y - P[0].y, dz = m0.z - P[0].z;
                            const float dc2 = dx * dx + dy * dy + dz * dz;
                            ask = ask || (b > 0.f && (s2 > v.open2 * dc2 || b * s2 > thr * dc2));
                        } else {
                            ask = ask || b > thr;
                        }
                        front = front || b > 0.f;
                    }
                    if (!__ballot(on && !(small ? front : ask))) break;  // every node is settled
                }
                exact = on && small && front;
                refine = on && !small && ask;
                keep = on && !small && !ask && front;
                one = false;
            } else {
                float ux = 0.f, scale = 0.f, d2 = 0.f;
                bool outside_front = false;
                auto axis = [&](float lo, float hi, float plo, float phi, float nl, float nh) {
                    const float dlo = lo - phi, dhi = hi - plo;  // box - pixel over the tile
                    ux += fmaxf(fmaxf(nl * dlo, nl * dhi), fmaxf(nh * dlo, nh * dhi));
                    scale += fmaxf(fabsf(dlo), fabsf(dhi));
                    const float e = fmaxf(fmaxf(dlo, plo - hi), 0.f);
                    d2 = fmaf(e, e, d2);
                };
                axis(r0.x, r1.x, tlo[0], thi[0], nlo[0], nhi[0]);
                axis(r0.y, r1.y, tlo[1], thi[1], nlo[1], nhi[1]);
                axis(r0.z, r1.z, tlo[2], thi[2], nlo[2], nhi[2]);
                const float ri = __builtin_amdgcn_rsqf(fmaxf(d2, delta2));
                const float most = r0.w * __builtin_amdgcn_fmed3f((ux + 1e-5f * scale) * ri, 0.f, 1.f) * (ri * ri) * 1.001f;
                bool far = true;  // the expansion criterion's distance tests cannot ask for the node
                float lim = thr_min;
                if (expansion) {
                    const float cx = fmaxf(fmaxf(tlo[0] - m0.x, m0.x - thi[0]), 0.f), cy = fmaxf(fmaxf(tlo[1] - m0.y, m0.y - thi[1]), 0.f),
                                cz = fmaxf(fmaxf(tlo[2] - m0.z, m0.z - thi[2]), 0.f);
                    const float dc2 = (cx * cx + cy * cy + cz * cz) * 0.998f;
                    far = s2 <= v.open2 * dc2;
                    lim = thr_min * dc2;
                }
        #pragma unroll
                for (int j = 0; j < 5; ++j) {
                    float thr;
                    const float4* P = S.pix[rep[j]];
                    const float b = pixel_bound(P, r0, r1, delta2, thr);
                    if (expansion) {
                        const float dx = m0.x - P[0].x, dy = m0.y - P[0].y, dz = m0.z - P[0].z;
                        const float dc2 = dx * dx + dy * dy + dz * dz;
                        ask = ask || (b > 0.f && (s2 > v.open2 * dc2 || b * s2 > thr * dc2));
                    } else {
                        ask = ask || b > thr;
                    }
                    front = front || b > 0.f;
                    outside_front = j == 4 && outside && b > 0.f;
                }
                const bool behind = ux < -1e-5f * scale && !outside_front;
                const bool below = expansion ? far && most * s2 <= lim : most <= lim;
                exact = on && small && front && !behind;
                refine = on && !small && ask;
                keep = on && !small && !ask && front && below && !behind;
                unsure = on && !(exact || refine || keep || behind);
                const uint64_t mu = __ballot(unsure);
                if (unsure) S.amb[na + lane_below(mu)] = k;
                na += __popcll(mu);
                one = room < 2 && mu != 0;
            }
            if (on && !refine && (every || !unsure)) ldone += __float_as_int(r2.z);
            apply(k, r0, r1, r2, exact, refine, keep);
        }
        if (!over && !full) over = evaluated() >= v.budget;
        return !over && !full;
    };
    // Node k alone, from every pixel (one per lane): its children are pushed
    // (a leaf as -(leaf + 1)), unless the budget is spent.
    auto single = [&](int k) {
        const float4* r = v.trav + (size_t)kTrav * k;
        const float4 r0 = r[0], r1 = r[1], r2 = r[2];
        float thr;
        const float b = pixel_bound(S.pix[lane], r0, r1, delta2, thr);
        if (!__ballot(b > 0.f)) return;
        const int count = __float_as_int(r2.z);
        if (count <= v.exact_count) {
            if (lane == 0) {
                S.ex[nx] = ((uint32_t)__float_as_int(r1.w) << 7) | (uint32_t)(count - 1);
                lexact += count;
            }
            ++nx;
            return;
        }
        bool ask = b > thr;
        if (expansion) {
            const float4* mr = v.mom + (size_t)kMom * k;
            const float4 m0 = mr[0], p = S.pix[lane][0];
            const float s2 = mr[1].x * mr[1].x, dx = m0.x - p.x, dy = m0.y - p.y, dz = m0.z - p.z;
            const float dc2 = dx * dx + dy * dy + dz * dz;
            ask = b > 0.f && (s2 > v.open2 * dc2 || b * s2 > thr * dc2);
        }
        ++ntest;
        const bool refine = __ballot(ask) != 0;
        if (refine && evaluated() < v.budget) {
            ++nvis;
            const int l = __float_as_int(r2.x), rr = __float_as_int(r2.y);  // child < 0: internal -(k + 1)
            if (lane == 0) {
                S.stack[sp] = -(rr + 1);
                S.stack[sp + 1] = -(l + 1);
            }
            sp += 2;
            return;
        }
        nbud += refine;
        if (node_faces(tb, r0, r1, v.nbox[2 * (size_t)k], v.nbox[2 * (size_t)k + 1])) {
            if (lane == 0) S.keep[ne] = k;
            ++ne;
            ++nkeep;
        }
    };
    // Depth first over subtrees.  The budget ends a cut in depth-first order:
    // a node that asks to be refined is kept once the nodes before it have
    // used the budget up.  A subtree after which the budget is not reached
    // never meets that, and is cut in any order; one that reaches it is taken
    // back and entered a node at a time, and so is one whose AVPLs, at the
    // share of them that the last such subtree's cut evaluated, would reach
    // it.  Nearly every tile's first subtree, the whole tree, is its last.
    float share = 0.f;
    if (lane == 0) S.stack[0] = 0;  // the root
    __builtin_amdgcn_wave_barrier();
    sp = 1;
    while (sp > 0 && !full) {
        const int k = uniform(S.stack[sp - 1]);
        --sp;
        __builtin_amdgcn_wave_barrier();
        if (k < 0) {  // a leaf
            if (lane == 0) S.ex[nx] = (uint32_t)(-(k + 1)) << 7;
            ++nx;
            ++nleaf;
        } else {
            // the queues are empty unless the budget is spent, so taking a
            // subtree back is taking its chunks back
            const int base = sp, c0 = last, t0 = ntest, v0 = nvis, k0 = nkeep, l0 = nleaf, e0 = lexact;
            const float size = __float_as_int(v.trav[(size_t)kTrav * k + 2].z);
            const bool enter = over || share * size > (float)(v.budget - evaluated());
            ldone = 0;
            if (enter || (!subtree(k) && !full)) {
                if (!enter) {
                    share = (float)(evaluated() - k0 - l0 - wave_isum(e0)) / (float)max(wave_isum(ldone), 1);
                    if (lane == 0) {
                        for (int c = c0 >= 0 ? pool.meta[c0].z : head; c >= 0; c = pool.meta[c].z) pool.meta[c].y = 0;
                        if (c0 >= 0) pool.meta[c0].z = -1;
                    }
                    if (c0 < 0) head = -1;
                    last = c0;
                    sp = base;
                    na = ne = nx = 0;
                    ntest = t0;
                    nvis = v0;
                    nkeep = k0;
                    nleaf = l0;
                    lexact = e0;
                    over = false;
                }
                single(k);
            }
        }
        __builtin_amdgcn_wave_barrier();
        over = evaluated() >= v.budget;
        const int least = over && sp > 0 ? kKeep : 1;
        flush_keep(least);
        flush_ex(least);
    }
    if (lane < nspare && spare + lane < pool.cap) pool.meta[spare + lane] = make_int4(item, 0, -1, 0);
    if (full) {  // hand the tile to k_cut_serial, its chunks to nobody
        if (lane == 0) {
            for (int c = head; c >= 0; c = pool.meta[c].z) pool.meta[c].y = 0;
            pool.head[item] = -1;
            pool.serial[atomicAdd(pool.count + arc::kSerialTiles, 1)] = item;
            atomicAdd(pool.count + arc::kFullTiles, 1);
            pool.evaluated[item] = -1;
        }
        return;
    }
    const int total = evaluated();
    if (lane == 0) {
        pool.head[item] = head;
        pool.evaluated[item] = total;
        pool.tbox[8 * (size_t)item + 6] = tile_cost(ntest, nkeep, total - nkeep);
        if (nbud > 0) atomicAdd(pool.count + arc::kSpentTiles, 1);
        if (v.counters) {
            const unsigned long long n = (unsigned long long)__popcll(alive);
            atomicAdd(&v.counters[C_TESTED], n * ntest);
            atomicAdd(&v.counters[C_VISITED], n * nvis);
            atomicAdd(&v.counters[C_EVALUATED], n * total);
            atomicAdd(&v.counters[C_EXACT], n * (total - nkeep));
            atomicAdd(&v.counters[C_BUDGET], (unsigned long long)nbud);
        }
    }
}

// ---- the chunks' sums ----------------------------------------------------
//
// On gfx950 an FP32 add, multiply or FMA whose operands are vector registers
// (or inline constants) issues every 2.4 cycles per SIMD with four waves or
// more, and every 4.5 with a scalar operand; maxima, compares and selects take
// 4.5 too, a reciprocal 8.4 (measured per instruction).  So the records, one
// for many pixels, are read into vector registers (from LDS, where the read
// costs 8 cycles of the CU per 16 bytes and wave), and to pay for the reads a
// wave takes kSlots records at a time: its lanes are kSlots groups, group r
// holds record r, and each lane kSlots of the tile's 64 pixels (its place in
// the group + kGroupLanes b).  The lanes that share a pixel meet once per
// chunk.  Clamps are output modifiers of multiplies, which cost nothing.
constexpr int kSlots = 2, kGroupLanes = 64 / kSlots;
struct Pixels {  // a lane's pixels
    float px[kSlots], py[kSlots], pz[kSlots], nx[kSlots], ny[kSlots], nz[kSlots];
};

// One wave's working memory of k_cut_eval.
struct EvalLds {
    uint32_t ex[kKeep];  // a chunk's kept nodes or exact ranges
    int pfx[kKeep];      // the ranges' leaves' prefix counts
    unsigned char mark[64];       // where ranges start among 64 leaves
    float sum[kSlots][3][64];     // the lanes' sums of a range chunk
    union {
        struct {
            float4 a[64 + 2 * kSlots];  // (x, y, z, nx) of the leaves that face the tile
            float4 b[64 + 2 * kSlots];  // (ny, nz, Ir, Ig)
            float c[64 + 2 * kSlots];   // Ib
        } leaf;
        float4 pix[2][64];      // the tile's pixels on their way to the lanes
    };
};

// G of a leaf (a unit normal) for a pixel, leaf_g's product as the two cosines
// clamped to [0, 1] by their multiplies (they are at most 1 to rounding) over
// |d|^2.
__device__ inline float leaf_cos2(const Pixels& P, int b, float x, float y, float z, float nx, float ny, float nz) {
    const float dx = x - P.px[b], dy = y - P.py[b], dz = z - P.pz[b];
    const float inv = __builtin_amdgcn_rsqf(dist2(dx, dy, dz, kDistFloor2));
    const float c1 = __builtin_amdgcn_fmed3f((P.nx[b] * dx + P.ny[b] * dy + P.nz[b] * dz) * inv, 0.f, 1.f);
    const float c2 = __builtin_amdgcn_fmed3f((nx * dx + ny * dy + nz * dz) * -inv, 0.f, 1.f);
    return (c1 * c2) * (inv * inv);
}

// n staged leaves, n a multiple of 2 kSlots and at most 64 + kSlots, in a plain
// run of their own, added to S.sum: a chunk's sum is plain runs of at most 34
// terms, 16 or 17 of them added plainly, and compensated per chunk, no worse than
// plain runs of 64 (all of a chunk's 512 terms in one run lost 6e-6 of equal
// terms).  S.sum is in LDS since six more registers here are spills.
__device__ inline void sum_leaves(EvalLds& S, int n, const Pixels& P) {
    float run[kSlots][3] = {};
    const int lane = threadIdx.x & 63;
    const int r = (threadIdx.x & 63) / kGroupLanes;
    const float4 *pa = S.leaf.a + r, *pq = S.leaf.b + r;
    const float* pc = S.leaf.c + r;
    for (int j = 0; j < n; j += 2 * kSlots, pa += 2 * kSlots, pq += 2 * kSlots, pc += 2 * kSlots) {
#pragma unroll
        for (int u = 0; u < 2 * kSlots; u += kSlots) {
            const float4 a = pa[u], q = pq[u];
            const float c = pc[u];
#pragma unroll
            for (int b = 0; b < kSlots; ++b) {
                const float g = leaf_cos2(P, b, a.x, a.y, a.z, a.w, q.x, q.y);
                run[b][0] = fmaf(q.z, g, run[b][0]);
                run[b][1] = fmaf(q.w, g, run[b][1]);
                run[b][2] = fmaf(c, g, run[b][2]);
            }
        }
    }
#pragma unroll
    for (int b = 0; b < kSlots; ++b)
#pragma unroll
        for (int c = 0; c < 3; ++c) S.sum[b][c][lane] += run[b][c];
}

// A chunk's exact ranges: the kChunkLeaves leaves from `from` on that face the tile.
__device__ inline void sum_ranges(const float4* __restrict__ crec, EvalLds& S, int nx, int from, const float* tb,
                                  const Pixels& P) {
    const int lane = threadIdx.x & 63;
    int n = 0;
#pragma unroll
    for (int b = 0; b < kSlots; ++b)
#pragma unroll
        for (int c = 0; c < 3; ++c) S.sum[b][c][lane] = 0.f;
    walk_ranges(crec, S.ex, nx, from, kChunkLeaves, S.pfx, S.mark, tb, [&](bool facing, const float4& r0, const float4& r1, const float4& r2) {
        const uint64_t m = __ballot(facing);
        if (facing) {
            const int j = n + lane_below(m);
            S.leaf.a[j] = make_float4(r0.x, r0.y, r0.z, r1.x);
            S.leaf.b[j] = make_float4(r1.y, r1.z, r2.x, r2.y);
            S.leaf.c[j] = r2.z;
        }
        n += __popcll(m);
        __builtin_amdgcn_wave_barrier();  // before the wave's reads of other lanes' writes
    }, [&]() {
        const int whole = n & ~(2 * kSlots - 1), rest = n - whole;
        sum_leaves(S, whole, P);
        if (rest && whole) {  // the rest waits for the next 64 leaves
            float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
            float c = 0.f;
            if (lane < rest) {
                a = S.leaf.a[whole + lane];
                b = S.leaf.b[whole + lane];
                c = S.leaf.c[whole + lane];
            }
            __builtin_amdgcn_wave_barrier();
            if (lane < rest) {
                S.leaf.a[lane] = a;
                S.leaf.b[lane] = b;
                S.leaf.c[lane] = c;
            }
        }
        __builtin_amdgcn_wave_barrier();
        n = rest;
    });
    if (n) {  // padded with leaves without intensity
        if (lane >= n && lane < 2 * kSlots) {
            S.leaf.a[lane] = S.leaf.a[0];
            S.leaf.b[lane] = make_float4(S.leaf.b[0].x, S.leaf.b[0].y, 0.f, 0.f);
            S.leaf.c[lane] = 0.f;
        }
        __builtin_amdgcn_wave_barrier();
        sum_leaves(S, 2 * kSlots, P);
    }
}

// A wave per chunk, the chunks taken as waves come free: a chunk is at most
// kKeep estimates or kChunkLeaves exact pairs per pixel, so the launch's waves
// end together whichever tiles the cut is large in.
template <bool kMany>
__global__ __launch_bounds__(kCutThreads) __attribute__((amdgpu_waves_per_eu(8))) void k_cut_eval(Views<kMany> views, CutPool pool) {
    __shared__ EvalLds lds[kCutThreads / 64];
    const int wave = uniform(threadIdx.x >> 6), lane = threadIdx.x & 63;
    EvalLds& S = lds[wave];
    const int waves = gridDim.x * (kCutThreads / 64);
    const int n = uniform(min(pool.count[arc::kTaken], pool.cap));
    // A wave starts with the chunk of its number and then takes groups of
    // chunks, a fraction of its share, from one of eight counters: a counter
    // serves about 100 atomics per microsecond (one for all took 230 us for 23K
    // chunks).  A counter's groups stand at changing places among eight: a
    // tile's first chunks are its largest and its last ones not used, and they
    // come in eights.  Where a group is eight chunks, one counter keeps up,
    // and all waves work on neighbouring tiles until the end (250001 AVPLs,
    // 1283x719: 16.0 ms, 16.9 with eight).
    const int group = max(1, min(8, n / (4 * waves)));
    const int counters = group == 8 ? 1 : min(kNextCounters, (int)gridDim.x), k = blockIdx.x % counters;
    int c = blockIdx.x * (kCutThreads / 64) + wave;
    for (int left = c < n ? 1 : 0;; ++c, --left) {
        if (left <= 0) {
            if (n <= waves) break;
            int got = 0;
            if (lane == 0) got = atomicAdd(pool.next + kNextStride * k, 1);
            got = uniform(got);
            c = waves + (got * counters + (k + (int)((unsigned)got * 0x9E3779B1u >> 29)) % counters) * group;
            if (c >= n) break;
            left = min(group, n - c);
        }
        const int4 m = pool.meta[c];
        const int item = uniform(m.x), kind = uniform(m.y) & 255, cnt = uniform(m.y) >> 8;
        if (cnt == 0) continue;  // not used, or its tile is cut serially
        const CutView v = views.of(item);
        const int t = item - (kMany ? v.tile_base : 0), tw = tiles_wide(v.W);
        const uint32_t* e = pool.entries + (size_t)(uniform(m.w) >> kPartBits) * kKeep;
        const uint32_t e0 = lane < cnt ? e[lane] : 0u, e1 = lane + 64 < cnt ? e[lane + 64] : 0u;
        const int x = (t % tw) * 8 + (lane & 7), y = (t / tw) * 8 + (lane >> 3);
        const PixelF F = load_pixel(v.gpos, v.gnrm, v.galb, v.mats, x < v.W && y < v.H ? y * v.W + x : 0);
        float* o = pool.part + (size_t)c * 192 + lane;
        if (kind == kNodes) {
            Acc acc;
            const int half = min(cnt, 64);
            for (int j = 0; j < half; ++j)
                add_moments(F, v.mom + kMom * (size_t)__builtin_amdgcn_readlane(e0, j), acc);
            acc.flush();
            for (int j = 64; j < cnt; ++j)
                add_moments(F, v.mom + kMom * (size_t)__builtin_amdgcn_readlane(e1, j - 64), acc);
            acc.flush();
            o[0] = acc.k[0].s;
            o[64] = acc.k[1].s;
            o[128] = acc.k[2].s;
            continue;
        }
        if (lane < cnt) S.ex[lane] = e0;
        if (lane + 64 < cnt) S.ex[lane + 64] = e1;
        S.pix[0][lane] = make_float4(F.px, F.py, F.pz, F.nx);
        S.pix[1][lane] = make_float4(F.ny, F.nz, 0.f, 0.f);
        __builtin_amdgcn_wave_barrier();
        Pixels P;
#pragma unroll
        for (int b = 0; b < kSlots; ++b) {
            const int k = lane % kGroupLanes + kGroupLanes * b;
            const float4 p = S.pix[0][k], q = S.pix[1][k];
            P.px[b] = p.x; P.py[b] = p.y; P.pz[b] = p.z;
            P.nx[b] = p.w; P.ny[b] = q.x; P.nz[b] = q.y;
        }
        __builtin_amdgcn_wave_barrier();  // read before the leaves are written over them
        ufloat* box = uptr(pool.tbox + 8 * (size_t)item);
        const float tb[6] = {box[0], box[1], box[2], box[3], box[4], box[5]};
        sum_ranges(v.crec, S, cnt, (uniform(m.w) & ((1 << kPartBits) - 1)) * kChunkLeaves, tb, P);
#pragma unroll
        for (int ch = 0; ch < 3; ++ch) {
            float out = 0.f;
#pragma unroll
            for (int b = 0; b < kSlots; ++b) {
                float s = S.sum[b][ch][lane];
#pragma unroll
                for (int off = kGroupLanes; off < 64; off <<= 1) s += __shfl_xor(s, off);
                if (lane / kGroupLanes == b) out = s;  // lane l keeps pixel l
            }
            o[64 * ch] = out;
        }
    }
}

// Each tile's partial sums, in the order its chunks were made.
template <bool kMany>
__global__ __launch_bounds__(kCutThreads) void k_cut_combine(Views<kMany> views, int nitems, CutPool pool) {
    const int lane = threadIdx.x & 63;
    const int item = uniform(blockIdx.x * (kCutThreads / 64) + (threadIdx.x >> 6));
    if (item >= nitems) return;
    if (item == 0 && lane == 0) {
        // what the next frame's pool should hold: the tiles that found it full
        // need as much as the others, as far as is known (the count alone grows
        // by what is asked for until it is full, a quarter per frame)
        const int taken = pool.count[arc::kTaken], rest = max(1, nitems - pool.count[arc::kFullTiles]);
        pool.seen[0] = (int)fminf((float)taken * fminf((float)nitems / (float)rest, 8.f), 1e9f);
        pool.seen[1] = pool.count[arc::kSpentTiles] + (pool.fixed ? pool.count[arc::kFullTiles] : 0);
    }
    const CutView v = views.of(item);
    const int t = item - (kMany ? v.tile_base : 0), tw = tiles_wide(v.W);
    const int x = (t % tw) * 8 + (lane & 7), y = (t / tw) * 8 + (lane >> 3);
    if (!__ballot(x < v.W && y < v.H)) {
        if (lane == 0) pool.cost[item] = 0.f;
        return;
    }
    const int evaluated = uniform(pool.evaluated[item]);
    if (evaluated < 0) return;  // k_cut_serial writes it
    if (lane == 0) pool.cost[item] = pool.tbox[8 * (size_t)item + 6];
    Kahan k[3];
    for (int c = uniform(pool.head[item]); c >= 0;) {
        const float* s = pool.part + (size_t)c * 192 + lane;
        c = uniform(pool.meta[c].z);
        k[0].add(s[0]);
        k[1].add(s[64]);
        k[2].add(s[128]);
    }
    if (x >= v.W || y >= v.H) return;
    const int q = y * v.W + x;
    const PixelF P = load_pixel(v.gpos, v.gnrm, v.galb, v.mats, q);
    v.out_rad[q] = make_float4(k[0].s * P.br, k[1].s * P.bg, k[2].s * P.bb, v.counters ? (float)evaluated : 1.f);
}

// One depth-first cut, a node at a time, summed as it goes.  Kept nodes and exact
// ranges are queued in LDS and summed in passes of their own when a queue fills,
// so the traversal carries no sums across its branches.
//
// Bound by vector and scalar issue and by each node's dependent record load.  With
// the tile's set-up held in registers throughout, arguments read again per node
// and records read in two loads, a budget of 8191 at 1283x719 pixels over 250001
// AVPLs took 9.1 ms a frame; 6.8 here and with the tiles in order.
template <bool kMany>
__device__ __forceinline__ void serial_tile(const CutView& v, float* cost, int item, int* S, int* E,
                                            uint32_t* X, int* pfx, unsigned char* mark, float4 (*stage)[3], float* tb) {
    const int lane = threadIdx.x & 63;
    PixelF P;
    float thr;
    bool live;
    {
        const CutView w = view_again<kMany>(item);
        const int t = item - (kMany ? w.tile_base : 0), tw = tiles_wide(w.W);
        const int x = (t % tw) * 8 + (lane & 7), y = (t / tw) * 8 + (lane >> 3);
        live = x < w.W && y < w.H;
        const int q = live ? y * w.W + x : 0;
        P = load_pixel(w.gpos, w.gnrm, w.galb, w.mats, q);
        thr = live ? view_threshold(w).at(q) : INFINITY;
    }
    // what each node needs stays in registers: left to itself the compiler reads
    // some of it from the arguments again per node, a load's latency each
    const float4 *trav = v.trav, *mom = v.mom, *nbox = v.nbox, *crec = v.crec;
    int exact_count = v.exact_count, budget = v.budget;
    asm volatile("" : "+s"(trav), "+s"(mom), "+s"(exact_count), "+s"(budget));
    const float delta2 = v.delta * v.delta;
    {  // the box of the tile's live pixels, as centre and half extent
        const float lx = wave_fmin(live ? P.px : INFINITY), hx = wave_fmax(live ? P.px : -INFINITY);
        const float ly = wave_fmin(live ? P.py : INFINITY), hy = wave_fmax(live ? P.py : -INFINITY);
        const float lz = wave_fmin(live ? P.pz : INFINITY), hz = wave_fmax(live ? P.pz : -INFINITY);
        if (lane == 0) {
            tb[0] = 0.5f * (lx + hx);
            tb[1] = 0.5f * (ly + hy);
            tb[2] = 0.5f * (lz + hz);
            tb[3] = 0.5f * (hx - lx);
            tb[4] = 0.5f * (hy - ly);
            tb[5] = 0.5f * (hz - lz);
        }
        __builtin_amdgcn_wave_barrier();  // lane 0's writes before the wave's reads
    }
    const bool expansion = v.criterion == ARC_CRITERION_EXPANSION;
    auto load = [](const float4* r) { return uload4(uptr(r)); };
    Acc acc;
    unsigned nvis = 0, nev = 0, nerr = 0, nbud = 0, ntest = 0, nexact = 0;  // wave-uniform
    int ne = 0, nx = 0;                                                     // queued, wave-uniform
    auto flush_est = [&]() {
        if (ne == 0) return;
        // the kept nodes that face the tile, one lane per node, compacted in place
        int kept = 0;
        for (int base = 0; base < ne; base += 64) {
            const int j = base + lane;
            bool facing = false;
            int k = 0;
            if (j < ne) {
                k = E[j];
                const float4* r = trav + (size_t)kTrav * k;
                facing = node_faces(tb, r[0], r[1], nbox[2 * (size_t)k], nbox[2 * (size_t)k + 1]);
            }
            const uint64_t fm = __ballot(facing);
            // every lane has read its entry before any is overwritten (kept <= base)
            __builtin_amdgcn_wave_barrier();
            if (facing) E[kept + lane_below(fm)] = k;
            kept += __popcll(fm);
            __builtin_amdgcn_wave_barrier();
        }
        nev -= (unsigned)(ne - kept);
        for (int j = 0; j < kept; ++j) {
            add_moments(P, mom + kMom * (size_t)uniform(E[j]), acc);
            acc.maybe_flush();
        }
        ne = 0;
    };
    auto drain_exact = [&]() {
        int cnt = 0;  // staged leaves
        if (nx > 0)
            walk_ranges(crec, X, nx, 0, INT_MAX, pfx, mark, tb, [&](bool facing, const float4& r0, const float4& r1, const float4& r2) {
                const uint64_t fm = __ballot(facing);
                if (facing) {
                    const int j = lane_below(fm);
                    stage[j][0] = r0;
                    stage[j][1] = r1;
                    stage[j][2] = r2;
                }
                cnt = __popcll(fm);
                __builtin_amdgcn_wave_barrier();
            }, [&]() {
#pragma unroll 1
                for (int j = 0; j < cnt; ++j) acc.add_run(stage[j][2], leaf_g(P, stage[j][0], stage[j][1]));
                acc.maybe_flush();
                __builtin_amdgcn_wave_barrier();  // read before the next 64 leaves' writes
            });
        nx = 0;
    };
    int sp = 0;
    int node = -1;
    for (;;) {
        bool pop = true;  // take the next node from the stack (not a refined node's left child)
        if (node < 0) {
            const int k = -(node + 1);
            const float4* r = trav + (size_t)kTrav * k;
            const float4 r0 = load(r), r1 = load(r + 1), r2 = load(r + 2);
            arc_bvh_node b;
            b.left = __float_as_int(r2.x);
            b.right = __float_as_int(r2.y);
            int count = __float_as_int(r2.z);
            asm volatile("" : "+s"(b.left), "+s"(b.right), "+s"(count));  // the whole record in one wait
            b.bbMin = arc_float3{r0.x, r0.y, r0.z};
            b.bbMax = arc_float3{r1.x, r1.y, r1.z};
            b.visited = 0;  // not read
            const int first = __float_as_int(r1.w);
            const float bound = node_bound1(P, b, r0.w, delta2);
            if (!__ballot(bound > 0.f)) {
                // behind every pixel's tangent plane: contributes exactly 0
            } else if (count <= exact_count) {
                // small node: its AVPLs exactly (refining it would end in the same sum)
                X[nx++] = ((uint32_t)first << 7) | (uint32_t)(count - 1);
                nexact += count;
            } else {
                bool refine;
                if (expansion) {
                    const float4* m = mom + kMom * (size_t)k;
                    const float4 c = load(m), size = load(m + 1);
                    const float dx = c.x - P.px, dy = c.y - P.py, dz = c.z - P.pz;
                    const float dc2 = dx * dx + dy * dy + dz * dz;
                    const float s2 = size.x * size.x;
                    refine = bound > 0.f && (s2 > v.open2 * dc2 || bound * s2 > thr * dc2);
                } else {
                    refine = bound > thr;
                }
                ++ntest;
                bool keep = true;
                if (__ballot(refine)) {
                    if ((int)(nev + nexact) >= budget) {
                        ++nbud;  // cut budget spent: keep the cluster
                    } else if (sp < kMomStack) {
                        S[sp++] = b.right;
                        node = uniform(b.left);
                        ++nvis;
                        keep = false;
                        pop = false;
                    } else {
                        ++nerr;  // stack full: keep the cluster
                    }
                }
                if (keep) {
                    E[ne++] = k;
                    ++nev;
                }
            }
        } else {
            X[nx++] = (uint32_t)node << 7;  // a leaf: a range of one
            ++nexact;
        }
        if (ne == kKeep) flush_est();
        if (nx == kKeep) drain_exact();
        if (pop) {
            if (sp == 0) break;
            node = uniform(S[--sp]);
        }
    }
    flush_est();
    drain_exact();
    acc.flush();
    const int alive = __popcll(__ballot(live));  // all lanes take part in the ballot
    const CutView w = view_again<kMany>(item);
    if (cost && lane == 0) *cost = tile_cost(ntest, nev, nexact);
    if (w.counters && lane == 0) {
        atomicAdd(&w.counters[C_TESTED], (unsigned long long)ntest * alive);
        atomicAdd(&w.counters[C_VISITED], (unsigned long long)nvis * alive);
        atomicAdd(&w.counters[C_EVALUATED], (unsigned long long)(nev + nexact) * alive);
        atomicAdd(&w.counters[C_EXACT], (unsigned long long)nexact * alive);
        atomicAdd(&w.counters[C_ERRORS], (unsigned long long)nerr);
        atomicAdd(&w.counters[C_BUDGET], (unsigned long long)nbud);
    }
    if (live) {
        const int t = item - (kMany ? w.tile_base : 0), tw = tiles_wide(w.W);
        const int q = ((t / tw) * 8 + (lane >> 3)) * w.W + (t % tw) * 8 + (lane & 7);
        const PixelF L = load_pixel(w.gpos, w.gnrm, w.galb, w.mats, q);  // again: its reflectance is not held meanwhile
        w.out_rad[q] = make_float4(acc.k[0].s * L.br, acc.k[1].s * L.bg, acc.k[2].s * L.bb,
                                   w.counters ? (float)(nev + nexact) : 1.f);
    }
}

// The tiles of pool.serial, more than the launch's waves as these come free; with
// `all`, every tile of the launch, a wave each.
template <bool kMany, int kWaves>
__global__ __launch_bounds__(kCutThreads) __attribute__((amdgpu_waves_per_eu(kWaves))) void k_cut_serial(Views<kMany> views, int nitems, int all,
                                                           CutPool pool) {
    __shared__ int stk[kCutThreads / 64][kMomStack];
    __shared__ int qest[kCutThreads / 64][kKeep];       // internal nodes to estimate
    __shared__ uint32_t qex[kCutThreads / 64][kKeep];   // exact ranges: first << 7 | (count - 1)
    __shared__ int qpfx[kCutThreads / 64][kKeep];       // their leaves' prefix counts
    __shared__ unsigned char qmark[kCutThreads / 64][64];  // where ranges start among 64 leaves
    __shared__ float4 lstage[kCutThreads / 64][64][3];  // leaves that face the tile
    __shared__ float tbox[kCutThreads / 64][8];         // the tile's box: centre, half extent
    const int wave = uniform(threadIdx.x >> 6);
    const int waves = gridDim.x * (kCutThreads / 64);
    const int n = all ? nitems : uniform(pool.count[arc::kSerialTiles]);
    const int id = blockIdx.x * (kCutThreads / 64) + wave;
    const bool queue = n > waves;
    auto next = [&]() {
        int got = 0;
        if ((threadIdx.x & 63) == 0) got = atomicAdd(pool.count + arc::kSerialNext, 1);
        return uniform(got);
    };
    for (int k = queue ? next() : uniform(id); k < n; k = next()) {
        const int item = !all ? uniform(pool.serial[k]) : pool.ordered ? uniform(pool.order[k]) : unordered_item(views, wave, k);
        serial_tile<kMany>(views.of(item), pool.cost ? pool.cost + item : nullptr, item, stk[wave], qest[wave], qex[wave],
                           qpfx[wave], qmark[wave], lstage[wave], tbox[wave]);
        if (!queue) break;
    }
}

// The order of the tiles from their costs in the last cut, heaviest first: the
// costs spread over two orders of magnitude, and a heavy tile started last runs
// alone at the end of the launch (1283x719 pixels, 250001 AVPLs, a budget of
// 8191: 8.4 ms in no order, 6.8 so).  A bucket sort on eight buckets per octave of cost, in one
// workgroup; the order within a bucket is that of the LDS atomics.  A tile's
// result does not depend on the order.
constexpr int kOrderBins = 256;
constexpr int kOrderThreads = 1024;

__device__ inline int order_bin(float c) {
    const int b = (int)(__log2f(fmaxf(c, 1.f)) * 8.f);
    return kOrderBins - 1 - min(max(b, 0), kOrderBins - 1);
}

__global__ __launch_bounds__(kOrderThreads) void k_tile_order(const float* __restrict__ cost, int n,
                                                              int* __restrict__ order) {
    __shared__ int hist[kOrderBins];
    __shared__ int off[kOrderBins];
    for (int i = threadIdx.x; i < kOrderBins; i += kOrderThreads) hist[i] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += kOrderThreads) atomicAdd(&hist[order_bin(cost[i])], 1);
    __syncthreads();
    if (threadIdx.x == 0) {
        int s = 0;
        for (int b = 0; b < kOrderBins; ++b) {
            off[b] = s;
            s += hist[b];
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += kOrderThreads) order[atomicAdd(&off[order_bin(cost[i])], 1)] = i;
}

// A frame's pool: no chunk taken, no tile handed back.
__global__ void k_pool_reset(CutPool p) {
    if (threadIdx.x == 0) {
        for (int k = 0; k < arc::kPoolCounters; ++k) p.count[k] = 0;
    }
    p.next[kNextStride * threadIdx.x] = 0;
}

}  // namespace

namespace arc {

int cut_moments_build(arc_gather* g, arc_bvh* b) {
    arc_ctx* ctx = g->ctx;
    const int n = b->n;
    if (n < 2) return ARC_OK;
    if (!b->has_cut_records || !g->crec.p) return fail(ctx, ARC_E_STATE, "moment records need the cut tree");
    const int nblocks = (n + kScanBlock - 1) / kScanBlock;
    ARC_TRY(ensure(ctx, g->mom, sizeof(float4) * kMom * (size_t)(n - 1)));
    ARC_TRY(ensure(ctx, g->mom_trav, sizeof(float4) * kTrav * (size_t)(n - 1)));
    ARC_TRY(ensure(ctx, g->mom_pre, sizeof(double) * kMomTerms * (size_t)n));
    ARC_TRY(ensure(ctx, g->mom_tot, sizeof(double) * kMomTerms * (size_t)nblocks));
    hipLaunchKernelGGL(k_mom_scan, dim3(nblocks, kGroups), dim3(kScanBlock), 0, ctx->stream, g->crec.as<float4>(),
                       b->nodes.as<arc_bvh_node>(), n,
                       g->mom_pre.as<double>(), g->mom_tot.as<double>());
    hipLaunchKernelGGL(k_mom_offsets, dim3(kMomTerms), dim3(kScanBlock), 0, ctx->stream, g->mom_tot.as<double>(),
                       nblocks);
    hipLaunchKernelGGL(k_mom_nodes, dim3((n - 1 + kScanBlock - 1) / kScanBlock), dim3(kScanBlock), 0, ctx->stream,
                       b->ranges.as<int>(), b->nodes.as<arc_bvh_node>(), n, g->mom_pre.as<double>(),
                       g->mom_tot.as<double>(), g->mom.as<float4>(), g->mom_trav.as<float4>());
    ARC_LAUNCHED(ctx);
    ARC_TRY(ensure(ctx, g->mom_nbox, sizeof(float4) * 2 * (size_t)(n - 1)));
    ARC_TRY(node_normal_boxes(b, g->crec.as<float4>(), g->mom_nbox.as<float4>()));
    g->mom_ready = true;
    return ARC_OK;
}

namespace {

// The chunks a tile can need.  Most frames use 9 to 11 per tile at 4000 to 8000
// AVPLs, 25 at 64000 and 25 to 40 at a million where nodes of up to 64 AVPLs
// are summed exactly; 4 to 11, 43 and 60 to 120 where larger ones are.  (8 + n
// / 64 of them cost the first frame of a 600x300 image with 4000 AVPLs 0.1 ms
// of allocation.)
int default_chunks(int n, int exact_count) {
    return exact_count > 64 ? std::min(96, 12 + n / 1024) : std::min(48, 14 + n / 2048);
}

constexpr int kMinChunks = 16384;  // 21 MB

// Readies `mem` for nitems tiles: the chunks of `per_tile` per tile, or as
// many as the last frame asked for when that was more (read from pinned
// memory that k_cut_combine writes: a frame still running counts at the next
// one).  Nothing grows while the stream is captured; held: the caller keeps
// the memory with the graph.  p.cap is 0 when there is no memory for a pool: the
// tiles are cut serially then, as with `want` 0.
int ready_pool(arc_ctx* ctx, hipStream_t stream, CutPoolMem& mem, int nitems, long long want, bool grow, bool held,
               CutPool& p) {
    p = CutPool{};
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    ARC_HIP(ctx, hipStreamIsCapturing(stream, &capture));
    const bool captured = capture != hipStreamCaptureStatusNone;
    const size_t serial = sizeof(int) * 2 * (size_t)nitems;
    if (captured && mem.serial.bytes < serial) return ARC_OK;  // not run before: nothing is allocated now
    ARC_TRY(ensure(ctx, mem.serial, serial));
    if (mem.tiles != nitems) mem.costs = false;
    mem.tiles = nitems;
    p.cost = mem.serial.as<float>();
    p.order = mem.serial.as<int>() + nitems;
    p.ordered = mem.costs ? 1 : 0;
    mem.costs = true;  // the cut that follows writes them
    if (want == 0) return ARC_OK;
    if (!mem.seen) {
        if (captured) return ARC_OK;
        ARC_HIP(ctx, hipHostMalloc(reinterpret_cast<void**>(&mem.seen), 2 * sizeof(int), hipHostMallocDefault));
        mem.seen[0] = mem.seen[1] = 0;
    }
    if (grow) {
        const int seen = *static_cast<volatile int*>(mem.seen);
        want = std::max(want, (long long)mem.cap);
        if (!captured && seen > want) want = (long long)seen + seen / 4;
    }
    // a small image's tiles can hold 512 chunks each (a budget of 65536): no small pools
    want = std::max(want, std::min((long long)kMinChunks, 512LL * nitems));
    want = std::min(want, (long long)(INT_MAX >> kPartBits));  // a chunk's entries and part share a word (67M: 87 GB)
    // one allocation: a new gather's first frame pays for each
    hipError_t e = hipSuccess;
    const size_t chunk = mem.mem.fit((size_t)want, sizeof(float) * 192 + sizeof(uint32_t) * kKeep + sizeof(int4),
                                     sizeof(int) * ((size_t)11 * nitems + arc::kPoolCounters + kNextStride * (kNextCounters + 1)), grow,
                                     !captured, [&] { e = hipStreamSynchronize(ctx->stream); });
    if (e != hipSuccess) return hip_fail(ctx, e, "hipStreamSynchronize", __FILE__, __LINE__);
    mem.cap = (int)chunk;
    if (chunk == 0) return ARC_OK;
    if (captured && !held) mem.mem.keep();
    const size_t part = sizeof(float) * 192 * chunk, entries = sizeof(uint32_t) * kKeep * chunk, meta = sizeof(int4) * chunk;
    char* at = static_cast<char*>(mem.mem.data());
    float* tbox = reinterpret_cast<float*>(at + part + entries + meta);
    int* head = reinterpret_cast<int*>(tbox + 8 * (size_t)nitems);
    int* counters = head + 3 * (size_t)nitems;
    p.entries = reinterpret_cast<uint32_t*>(at + part);
    p.meta = reinterpret_cast<int4*>(at + part + entries);
    p.part = reinterpret_cast<float*>(at);
    p.tbox = tbox;
    p.head = head;
    p.evaluated = head + nitems;
    p.serial = head + 2 * (size_t)nitems;
    p.count = counters;
    p.next = counters + arc::kPoolCounters + kNextStride;
    p.seen = mem.seen;
    p.cap = (int)chunk;
    p.fixed = !grow || mem.mem.refused();
    p.grab = nitems < 4096 ? 4 : 8;
    return ARC_OK;
}

// Resident waves of k_cut_eval: eight per SIMD.
constexpr int kEvalBlocks = 2048;

// Tiles that leave at most four waves per SIMD: k_cut_serial built for four has
// registers for everything.
constexpr int kFewTiles = 4096;

template <bool kMany>
void launch_cut(hipStream_t stream, const Views<kMany>& views, int nitems, bool expansion, bool serial, const CutPool& p) {
    const int blocks = (nitems + 3) / 4;
    if (serial) {
        if (p.ordered)
            hipLaunchKernelGGL(k_tile_order, dim3(1), dim3(kOrderThreads), 0, stream, p.cost, nitems, p.order);
        if (nitems <= kFewTiles)
            hipLaunchKernelGGL((k_cut_serial<kMany, 4>), dim3(blocks), dim3(kCutThreads), 0, stream, views, nitems, 1, p);
        else
            hipLaunchKernelGGL((k_cut_serial<kMany, 8>), dim3(blocks), dim3(kCutThreads), 0, stream, views, nitems, 1, p);
        return;
    }
    hipLaunchKernelGGL(k_pool_reset, dim3(1), dim3(kNextCounters), 0, stream, p);
    if (expansion)
        hipLaunchKernelGGL((k_cut_decide<kMany, true>), dim3(blocks), dim3(kCutThreads), 0, stream, views, nitems, p);
    else
        hipLaunchKernelGGL((k_cut_decide<kMany, false>), dim3(blocks), dim3(kCutThreads), 0, stream, views, nitems, p);
    hipLaunchKernelGGL(k_cut_eval<kMany>, dim3(std::min(8 * blocks, kEvalBlocks)), dim3(kCutThreads), 0, stream, views, p);
    hipLaunchKernelGGL((k_cut_serial<kMany, 8>), dim3(std::min(blocks, kEvalBlocks)), dim3(kCutThreads), 0, stream, views, nitems, 0, p);
    hipLaunchKernelGGL(k_cut_combine<kMany>, dim3(blocks), dim3(kCutThreads), 0, stream, views, nitems, p);
}

}  // namespace

void* PoolDevice::alloc(size_t bytes) {
    void* p = nullptr;
    if (hipMalloc(&p, bytes) == hipSuccess) return p;
    (void)hipGetLastError();
    return nullptr;
}
void PoolDevice::free(void* p) { (void)hipFree(p); }

// What is free but a sixteenth of the device, left to other objects' buffers.
size_t PoolDevice::room() {
    size_t free = 0, total = 0;
    if (hipMemGetInfo(&free, &total) != hipSuccess) {
        (void)hipGetLastError();
        return SIZE_MAX;
    }
    return free > total / 16 ? free - total / 16 : 0;
}

void release_pool(CutPoolMem& mem) {
    mem.mem.release();
    release(mem.serial);
    if (mem.seen) (void)hipHostFree(mem.seen);
    mem = CutPoolMem{};
}

bool cut_pool_short(arc_gather* g) {
    return g->est_chunks == 0 && g->pool.seen && !g->pool.mem.refused() &&
           *static_cast<volatile int*>(g->pool.seen) > g->pool.cap;
}

int cut_moments(arc_gather* g, arc_bvh* b, const CutEBParams& cp, float4* rad, unsigned long long* counters,
                hipEvent_t mark, CutView* defer) {
    arc_ctx* ctx = g->ctx;
    const int n = b->n;
    if (!g->mom_ready || !g->mom.p || g->mom.bytes < sizeof(float4) * kMom * (size_t)(n - 1))
        return fail(ctx, ARC_E_STATE, "moment estimator: node records not built");
    CutEB t{};
    Threshold th{};
    ARC_TRY(prepare_cut(g, b, cp, t, th));
    const int nitems = 4 * ((g->width + 15) / 16) * ((g->height + 15) / 16);
    const CutView v{g->crec.as<float4>(), g->mom.as<float4>(), g->mom_trav.as<float4>(), g->mom_nbox.as<float4>(),
                    g->gpos, g->gnrm, g->galb, g->mats.as<arc_material>(), th.est, th.sum, th.eps, th.floor_frac,
                    th.inv_npix, g->width, g->height, cp.delta, cp.budget, cp.criterion, cp.opening * cp.opening,
                    cp.exact_count, rad, counters, 0, nitems, n};
    if (defer) {
        *defer = v;
        return ARC_OK;
    }
    // what the last cut of this setting says: how many tiles met their budget, or found a pool full that does not grow
    CutPoolMem& mem = g->pool;
    const CutSetting now{nitems, cp.budget, cp.exact_count, cp.criterion, g->est_chunks, cp.eps, cp.image_floor};
    if (mem.seen && !(mem.last == now)) mem.seen[1] = 0;
    const bool serial = serial_cut(cp.budget, nitems, mem.seen ? static_cast<volatile int*>(mem.seen)[1] : 0,
                                   cp.criterion == ARC_CRITERION_EXPANSION);
    mem.last = now;
    CutPool pool{};
    const long long per_tile = serial ? 0 : g->est_chunks > 0 ? g->est_chunks : default_chunks(n, cp.exact_count);
    ARC_TRY(ready_pool(ctx, ctx->stream, g->pool, nitems, per_tile * nitems, g->est_chunks == 0, g->batch_capture, pool));
    if (mark) ARC_HIP(ctx, hipEventRecord(mark, ctx->stream));
    launch_cut<false>(ctx->stream, Views<false>{v}, nitems, cp.criterion == ARC_CRITERION_EXPANSION, pool.cap == 0, pool);
    ARC_LAUNCHED(ctx);
    return ARC_OK;
}

int cut_moments_views(arc_ctx* ctx, hipStream_t stream, const CutView* host_views, const CutView* views, int nviews,
                      CutPoolMem& mem) {
    if (nviews < 1) return ARC_OK;
    int nitems = 0;
    long long want = 0;
    bool expansion = false;
    for (int i = 0; i < nviews; ++i) {
        nitems += host_views[i].ntiles;
        if (!serial_cut(host_views[i].budget, 0, 0))
            want += (long long)host_views[i].ntiles * default_chunks(host_views[i].n, host_views[i].exact_count);
        expansion = expansion || host_views[i].criterion == ARC_CRITERION_EXPANSION;
    }
    CutPool pool{};
    ARC_TRY(ready_pool(ctx, stream, mem, nitems, want, true, true, pool));
    launch_cut<true>(stream, Views<true>{views, nviews}, nitems, expansion, pool.cap == 0, pool);
    ARC_LAUNCHED(ctx);
    return ARC_OK;
}

}  // namespace arc
