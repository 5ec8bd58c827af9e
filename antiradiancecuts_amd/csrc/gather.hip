// AVPL radiance / antiradiance gather on gfx950 — replaces CudaGather
// (cudaGather.h:25-70, cudaGather.cu:156-1051).
//
// Kernels
//   k_pack        AVPL SoA (AvplsGpuParam) -> 80-byte records: position,
//                 unit normal, raw and unit incident direction, radiance with
//                 the AVPL-side Lambertian BRDF folded in, antiradiance with
//                 the disk normalisation 1/(pi r^2) folded in.
//   k_exact_*     exact gather (kernel_radiance_simple :269-314 and
//                 kernel_antiradiance :446-557 fused), Lambertian (two pixels
//                 per lane) and with specular lobes: 64 records at a time in
//                 LDS, runs summed in FP32 and added to the pixel total with
//                 Kahan compensation; split over AVPL ranges.
//   k_exact_f64   the same sums in FP64 with the reference's formulas (the
//                 reference image for error metrics).
//   k_finalize    sums the splits (Kahan), writes radiance, antiradiance and
//                 result = radiance - antiradiance (kernel_combine :782-803).
//   k_cut_sa      light-cut radiance with the solid-angle criterion
//                 (kernel_bvh :316-444): an 8x8 tile's pixels walk the tree
//                 together.
#include <cmath>
#include <cstring>
#include <vector>

#include "cutnet.hpp"
#include "gather_common.hpp"

using arc::DevBuf;
using arc::f3;
using namespace arc::gm;
using namespace arc::gd;

namespace {

// ------------------------------------------------------------- pack ----
__global__ __launch_bounds__(kThreads) void k_pack(arc::AvplsDev a, const arc_material* __restrict__ mats,
                                                   int general, int model, float inv_pi_r2,
                                                   float4* __restrict__ rec) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    const f3 p = a.pos[i], q = a.nrm[i], w = a.dir[i], L = a.rad[i];
    const f3 A = a.anti ? a.anti[i] : f3{0.f, 0.f, 0.f};
    const int mi = a.mat[i];
    const float nq = 1.0f / sqrtf(q.x * q.x + q.y * q.y + q.z * q.z);
    const float w2 = w.x * w.x + w.y * w.y + w.z * w.z;
    const float nw = w2 > 0.f ? 1.0f / sqrtf(w2) : 0.f;
    float lr = L.x, lg = L.y, lb = L.z;
    if (!general && w2 != 0.f) {  // Lambertian AVPL: f_r = diffuse / pi, constant per AVPL
        const arc_material& m = mats[mat_slot(mi)];
        lr *= kOneOverPi * m.diffuse.x;
        lg *= kOneOverPi * m.diffuse.y;
        lb *= kOneOverPi * m.diffuse.z;
    }
    const float as = model == ARC_ANTIRAD_DISK ? inv_pi_r2 : 1.0f;
    float4* r = rec + (size_t)kRecF4 * i;
    r[0] = make_float4(p.x, p.y, p.z, w.x * nw);
    r[1] = make_float4(q.x * nq, q.y * nq, q.z * nq, w.y * nw);
    r[2] = make_float4(w.x, w.y, w.z, w.z * nw);
    r[3] = make_float4(lr, lg, lb, (float)mi);
    r[4] = make_float4(A.x * as, A.y * as, A.z * as, kGuard * sqrtf(w2));  // guard for |w . n|
}

// ------------------------------------------------------------ exact ----
// part layout: [split][6][npix] = radiance rgb, antiradiance rgb.

// c^e for finite c >= 0 and e > 0, rounded once: log2 by the atanh series of
// (m - 1) / (m + 1) and 2^x by its Taylor series, in double (their errors are
// 1e-10 and 5e-9 relative), which issues at half the single rate: powf, which
// carries its logarithm in pairs of floats, takes about twice as long.
__device__ inline float pow_pos(float c, float e) {
    float m = __builtin_amdgcn_frexp_mantf(c);
    int k = __builtin_amdgcn_frexp_expf(c);
    if (m < 0.70710678f) {
        m += m;
        --k;
    }
    const double den = (double)m + 1.0;
    double r = (double)__builtin_amdgcn_rcpf((float)den);
    r = __builtin_fma(r, __builtin_fma(-den, r, 1.0), r);
    const double f = (double)(m - 1.0f) * r, s = f * f;
    double p = 1.0 / 11.0;
    p = __builtin_fma(p, s, 1.0 / 9.0);
    p = __builtin_fma(p, s, 1.0 / 7.0);
    p = __builtin_fma(p, s, 1.0 / 5.0);
    p = __builtin_fma(p, s, 1.0 / 3.0);
    p = __builtin_fma(p, s, 1.0);
    const double log2 = __builtin_fma(f * p, 2.0 / M_LN2, (double)k);
    const double y = fmin(fmax((double)e * log2, -200.0), 200.0);  // beyond: 0 and infinity in float
    const double n = rint(y), x = (y - n) * M_LN2;
    double q = 1.0 / 5040.0;
    q = __builtin_fma(q, x, 1.0 / 720.0);
    q = __builtin_fma(q, x, 1.0 / 120.0);
    q = __builtin_fma(q, x, 1.0 / 24.0);
    q = __builtin_fma(q, x, 1.0 / 6.0);
    q = __builtin_fma(q, x, 0.5);
    q = __builtin_fma(q, x, 1.0);
    q = __builtin_fma(q, x, 1.0);
    return c == 0.f ? 0.f : (float)ldexp(q, (int)n);
}

// A lobe's value: powf where pow_pos does not hold.
__device__ inline float lobe(float c, float e, bool odd) { return odd ? powf(c, e) : pow_pos(c, e); }
__device__ inline bool odd_lobe(float e, float x, float y, float z) {
    return !(e > 0.f && e < 1e5f && fabsf(x) + fabsf(y) + fabsf(z) < 1e15f);
}

// Materials with specular lobes: a wave stages 64 AVPLs at a time in LDS with
// the mirrored incident direction and the two factors of its material, so that
// a pair's BRDFs (cudaGather.cu:59-68) are a dot product and a power each, and
// the powers are left out for AVPLs without a lobe (a branch of the wave) and
// for waves without a pixel that has one.  The pixel's lobe max(0, reflect(-wi,
// n) . wo) is max(0, wi . m) with m = 2 n (n . wo) - wo, one vector per pixel;
// both mirrored vectors are made in double, since their rounding would be in
// every pair alike, times the exponent.
//
// Bound: vector instructions, half of them the powers.  331x247 pixels, 3001
// AVPLs, every other material glossy: 1.97 ms with the BRDFs written out and
// powf, 0.68 here.
constexpr int kPlain = 32;  // pairs summed plainly before a compensated add

struct GlossyLds {
    float4 a[64], b[64];  // position, normal.x; normal.yz, radiance x diffuse / pi .rg
    float4 c[64], d[64];  // .b, radiance x lobe factor; mirrored direction, exponent
};

template <int MODEL, bool DO_RAD, bool DO_ANTI>
__global__ __launch_bounds__(kThreads) void k_exact_glossy(const float4* __restrict__ rec, arc::AvplsDev raw, int chunk,
                                                           const float4* __restrict__ gpos,
                                                           const float4* __restrict__ gnrm,
                                                           const float4* __restrict__ galb,
                                                           const arc_material* __restrict__ mats, int npix,
                                                           float camx, float camy, float camz, AntiParams ap,
                                                           float* __restrict__ part) {
    using V3 = V<float>;
    __shared__ GlossyLds lds[kThreads / 64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    GlossyLds& S = lds[wave];
    const int first = (blockIdx.x * (kThreads / 64) + wave) * 64;
    if (first >= npix) return;
    const int q = first + lane < npix ? first + lane : 0;
    const PixelF P = load_pixel(gpos, gnrm, galb, mats, q);
    // the pixel's lobe
    const Mat<float> pm = material<float>(mats, P.mat);
    const bool pglossy = length(pm.specular) > 0.f;
    V<double> mirror_d;
    {
        const float4 p4 = gpos[q], n4 = gnrm[q];
        const V<double> n = mk<double>(n4.x, n4.y, n4.z);
        const V<double> wo = normalize(mk<double>(camx, camy, camz) - mk<double>(p4.x, p4.y, p4.z));
        mirror_d = 2.0 * n * dot(n, wo) - wo;
    }
    const V3 mirror = mk((float)mirror_d.x, (float)mirror_d.y, (float)mirror_d.z);
    const V3 pspec = (0.5f * kOneOverPi * (pm.exponent + 2.f)) * pm.specular;
    const bool any_glossy = __ballot(pglossy) != 0;
    const bool podd = __ballot(pglossy && odd_lobe(pm.exponent, mirror.x, mirror.y, mirror.z)) != 0;
    auto pixel_brdf = [&](float cm) {  // cm = wi . mirror
        V3 b = mk(P.br, P.bg, P.bb);
        if (any_glossy) {
            const float l = lobe(fmaxf(0.f, cm), pm.exponent, podd);
            if (pglossy) b = b + l * pspec;
        }
        return b;
    };
    const int a0 = blockIdx.y * chunk, a1 = min(raw.n, a0 + chunk);
    Kahan kr[3], ka[3];
    for (int base = a0; base < a1; base += 64) {
        const int cnt = min(64, a1 - base);
        const int mine = lane < cnt ? base + lane : base;
        const float4* r = rec + (size_t)kRecF4 * mine;
        const float4 r4 = r[4];
        uint64_t has_anti = 0;
        if (DO_ANTI) has_anti = __ballot(lane < cnt && !(r4.x == 0.f && r4.y == 0.f && r4.z == 0.f));
        if (DO_RAD) {
            const float4 r0 = r[0], r1 = r[1], r2 = r[2], r3 = r[3];
            const Mat<float> am = material<float>(mats, (int)r3.w);
            const V3 w = mk(r2.x, r2.y, r2.z), L = mk(r3.x, r3.y, r3.z), an = mk(r1.x, r1.y, r1.z);
            const bool flat = length(w) == 0.f;  // no incident direction: a reflectance of 1
            const bool glossy = !flat && length(am.specular) > 0.f;
            const V<double> rd = reflect(ld3<double>(raw.dir[mine]), ld3<double>(raw.nrm[mine]));
            const V3 refl = mk((float)rd.x, (float)rd.y, (float)rd.z);
            const V3 ld = flat ? L : L * (kOneOverPi * am.diffuse);
            const V3 ls = L * ((0.5f * kOneOverPi * (am.exponent + 2.f)) * am.specular);
            const uint64_t gm = __ballot(glossy);
            const uint64_t om = __ballot(glossy && odd_lobe(am.exponent, refl.x, refl.y, refl.z));
            __builtin_amdgcn_wave_barrier();  // the last run's reads come first
            S.a[lane] = make_float4(r0.x, r0.y, r0.z, an.x);
            S.b[lane] = make_float4(an.y, an.z, ld.x, ld.y);
            S.c[lane] = make_float4(ld.z, ls.x, ls.y, ls.z);
            S.d[lane] = make_float4(refl.x, refl.y, refl.z, am.exponent);
            __builtin_amdgcn_wave_barrier();  // before the reads of other lanes' writes
            for (int from = 0; from < cnt; from += kPlain) {
                float s0 = 0.f, s1 = 0.f, s2 = 0.f;
                for (int j = from; j < min(cnt, from + kPlain); ++j) {
                    const float4 a = S.a[j], b = S.b[j], c = S.c[j];
                    const float dx = a.x - P.px, dy = a.y - P.py, dz = a.z - P.pz;
                    const float dd = dx * dx + dy * dy + dz * dz, inv = __builtin_amdgcn_rsqf(dd);
                    const float c1 = clamp01((P.nx * dx + P.ny * dy + P.nz * dz) * inv);
                    const float c2 = clamp01(-(a.w * dx + b.x * dy + b.y * dz) * inv);
                    const float gg = c1 * c2 * __builtin_amdgcn_rcpf(dd);
                    if (!__ballot(!(gg == 0.f))) continue;  // no pixel of the wave sees it
                    V3 l = mk(b.z, b.w, c.x);
                    if (gm >> j & 1) {
                        const float4 d = S.d[j];
                        const float p = lobe(fmaxf(0.f, -(d.x * dx + d.y * dy + d.z * dz) * inv), d.w, (om >> j & 1) != 0);
                        l.x += c.y * p;
                        l.y += c.z * p;
                        l.z += c.w * p;
                    }
                    const V3 f = pixel_brdf((mirror.x * dx + mirror.y * dy + mirror.z * dz) * inv);
                    s0 += l.x * f.x * gg;
                    s1 += l.y * f.y * gg;
                    s2 += l.z * f.z * gg;
                }
                kr[0].add(s0);
                kr[1].add(s1);
                kr[2].add(s2);
            }
        }
        if (DO_ANTI && has_anti) {
            float s0 = 0.f, s1 = 0.f, s2 = 0.f;
            for (uint64_t m = has_anti; m; m &= m - 1) {
                const int i = base + __builtin_ctzll(m);
                const float4* r = rec + (size_t)kRecF4 * i;
                const float4 r0 = r[0], r1 = r[1], r2 = r[2], A = r[4];
                const float dx = r0.x - P.px, dy = r0.y - P.py, dz = r0.z - P.pz;
                const float dd = dx * dx + dy * dy + dz * dz;
                const float inv = rsq(dd);
                const float cn = P.nx * dx + P.ny * dy + P.nz * dz;
                const float ca = -(r1.x * dx + r1.y * dy + r1.z * dz);
                const float wgt = anti_weight<MODEL>(P, r0, r1, r2, A.w, dx, dy, dz, dd, inv, cn, ca, ap, gpos, gnrm, q, raw, i);
                if (!__ballot(wgt != 0.f)) continue;
                // a pixel accepts a few of thousands, so the cosine's rounding, times
                // the exponent, is not averaged out as in the radiance: in double
                const V<double> d = mk<double>(r0.x, r0.y, r0.z) - mk<double>(P.px, P.py, P.pz);
                const double d2 = dot(d, d), ri = inv;
                const V3 f = pixel_brdf((float)(dot(mirror_d, d) * (ri * (1.5 - 0.5 * d2 * ri * ri))));
                if (wgt != 0.f) {
                    s0 += A.x * (f.x * wgt);
                    s1 += A.y * (f.y * wgt);
                    s2 += A.z * (f.z * wgt);
                }
            }
            ka[0].add(s0);
            ka[1].add(s1);
            ka[2].add(s2);
        }
    }
    if (first + lane >= npix) return;
    float* o = part + (size_t)blockIdx.y * 6 * npix + first + lane;
    if (DO_RAD) { o[0] = kr[0].s; o[(size_t)npix] = kr[1].s; o[2 * (size_t)npix] = kr[2].s; }
    if (DO_ANTI) { o[3 * (size_t)npix] = ka[0].s; o[4 * (size_t)npix] = ka[1].s; o[5 * (size_t)npix] = ka[2].s; }
}

// Lambertian materials: the BRDFs are factors of the record and of the pixel.
//
// A lane sums two pixels.  Each wave stages 64 AVPLs at a time in LDS, those
// with antiradiance in a list of their own, so that the others (two thirds of
// a scene's AVPLs: a path's antiradiance leaves only where it is blocked) pay
// nothing for it, and reads a record for both pixels as vector operands: an
// instruction with a scalar operand issues at half the rate, and read by scalar
// loads the records made every first operation on them one.  A wave needs no
// other wave's lists: no barrier.
//
// Bound: vector instructions, 20 per pair for the radiance and 25 (cone) per
// pair with antiradiance.  256x256 pixels, 4096 AVPLs, cone: 387 us with a
// pixel per lane and scalar loads, 160 here; one pixel per lane 170.
constexpr int kExactSlots = 2;

template <int MODEL>
struct ExactLds {
    float4 a[64], b[64];                  // position and normal.x; normal.yz, radiance.rg
    float c[64];                          // radiance.b
    float4 u[64], v[64], w[MODEL == ARC_ANTIRAD_DISK ? 64 : 1];
    float4 A[64];                         // antiradiance, guard of |w . n|
    int i[64];
};

template <int MODEL, bool DO_RAD, bool DO_ANTI>
__global__ __launch_bounds__(kThreads) void k_exact_lambert(const float4* __restrict__ rec, arc::AvplsDev raw, int chunk,
                                                            const float4* __restrict__ gpos,
                                                            const float4* __restrict__ gnrm,
                                                            const float4* __restrict__ galb,
                                                            const arc_material* __restrict__ mats, int npix,
                                                            AntiParams ap, float* __restrict__ part) {
    __shared__ ExactLds<MODEL> lds[kThreads / 64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    ExactLds<MODEL>& S = lds[wave];
    const int first = (blockIdx.x * (kThreads / 64) + wave) * 64 * kExactSlots;
    if (first >= npix) return;
    PixelF P[kExactSlots];
    int q[kExactSlots];
#pragma unroll
    for (int s = 0; s < kExactSlots; ++s) {
        q[s] = first + 64 * s + lane < npix ? first + 64 * s + lane : 0;
        P[s] = load_pixel(gpos, gnrm, galb, mats, q[s]);
        // a pixel without a normal accepts no pair of the cone model
        if (MODEL == ARC_ANTIRAD_CONE && !(P[s].nx == P[s].nx && P[s].ny == P[s].ny && P[s].nz == P[s].nz))
            P[s].nx = P[s].ny = P[s].nz = 0.f;
    }
    const float edge = fmaxf(kConeEps, ap.cos_half);  // c above both
    const int a0 = blockIdx.y * chunk, a1 = min(raw.n, a0 + chunk);
    Kahan kr[kExactSlots][3], ka[kExactSlots][3];
    for (int base = a0; base < a1; base += 64) {
        const int cnt = min(64, a1 - base);
        int na = 0;
        {
            const bool in = lane < cnt;
            const float4* r = rec + (size_t)kRecF4 * (in ? base + lane : base);
            const float4 r0 = r[0], r1 = r[1], r2 = r[2], r3 = r[3], r4 = r[4];
            __builtin_amdgcn_wave_barrier();  // the last run's reads come first
            if (DO_RAD) {
                S.a[lane] = make_float4(r0.x, r0.y, r0.z, r1.x);
                S.b[lane] = make_float4(r1.y, r1.z, r3.x, r3.y);
                S.c[lane] = r3.z;
            }
            if (DO_ANTI) {
                const bool has = in && !(r4.x == 0.f && r4.y == 0.f && r4.z == 0.f);
                const uint64_t m = __ballot(has);
                if (has) {
                    const int k = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                    // a direction that is no number accepts no pair
                    const bool num = r0.w == r0.w && r1.w == r1.w && r2.w == r2.w;
                    S.u[k] = make_float4(r0.x, r0.y, r0.z, num || MODEL == ARC_ANTIRAD_DISK ? r0.w : 0.f);
                    if (MODEL == ARC_ANTIRAD_DISK) {
                        S.v[k] = make_float4(r1.x, r1.y, r1.z, r1.w);
                        S.w[k] = make_float4(r2.x, r2.y, r2.z, r2.w);
                        S.A[k] = r4;
                    } else {
                        S.v[k] = make_float4(num ? r1.w : 0.f, num ? r2.w : 0.f, r4.x, r4.y);
                        S.A[k].x = r4.z;
                    }
                    S.i[k] = base + lane;
                }
                na = __popcll(m);
            }
            __builtin_amdgcn_wave_barrier();  // before the reads of other lanes' writes
        }
        if (DO_RAD) {
            for (int from = 0; from < cnt; from += kPlain) {
                float sum[kExactSlots][3] = {};
#pragma unroll 2
                for (int j = from; j < min(cnt, from + kPlain); ++j) {
                    const float4 a = S.a[j], b = S.b[j];
                    const float lz = S.c[j];
#pragma unroll
                    for (int s = 0; s < kExactSlots; ++s) {
                        const float dx = a.x - P[s].px, dy = a.y - P[s].py, dz = a.z - P[s].pz;
                        const float inv = __builtin_amdgcn_rsqf(dx * dx + dy * dy + dz * dz);
                        const float cn = P[s].nx * dx + P[s].ny * dy + P[s].nz * dz;
                        const float ca = -(a.w * dx + b.x * dy + b.y * dz);
                        const float c1 = fminf(fmaxf(cn * inv, 0.f), 1.f), c2 = fminf(fmaxf(ca * inv, 0.f), 1.f);
                        const float gg = c1 * c2 * (inv * inv);
                        sum[s][0] += b.z * gg;
                        sum[s][1] += b.w * gg;
                        sum[s][2] += lz * gg;
                    }
                }
#pragma unroll
                for (int s = 0; s < kExactSlots; ++s)
                    for (int c = 0; c < 3; ++c) kr[s][c].add(sum[s][c]);
            }
        }
        if (DO_ANTI && na > 0) {
            float sum[kExactSlots][3] = {};
            for (int j = 0; j < na; ++j) {
                const float4 u = S.u[j], v = S.v[j];
                if constexpr (MODEL == ARC_ANTIRAD_DISK) {
                    const float4 w = S.w[j], A = S.A[j];
                    bool may = false;  // some pixel faces the AVPL's direction
#pragma unroll
                    for (int s = 0; s < kExactSlots; ++s)
                        may = may || w.x * P[s].nx + w.y * P[s].ny + w.z * P[s].nz < A.w;
                    if (!__ballot(may)) continue;
#pragma unroll
                    for (int s = 0; s < kExactSlots; ++s) {
                        const float dx = u.x - P[s].px, dy = u.y - P[s].py, dz = u.z - P[s].pz;
                        const float dd = dx * dx + dy * dy + dz * dz;
                        const float inv = __builtin_amdgcn_rsqf(dd);
                        const float cn = P[s].nx * dx + P[s].ny * dy + P[s].nz * dz;
                        const float ca = -(v.x * dx + v.y * dy + v.z * dz);
                        const float m = anti_weight<MODEL>(P[s], u, v, w, A.w, dx, dy, dz, dd, inv, cn, ca, ap, gpos, gnrm,
                                                           q[s], raw, S.i[j]);
                        sum[s][0] += A.x * m;
                        sum[s][1] += A.y * m;
                        sum[s][2] += A.z * m;
                    }
                } else {
                    const float az = S.A[j].x;
#pragma unroll
                    for (int s = 0; s < kExactSlots; ++s) {
                        const float dx = u.x - P[s].px, dy = u.y - P[s].py, dz = u.z - P[s].pz;
                        const float inv = __builtin_amdgcn_rsqf(dx * dx + dy * dy + dz * dz);
                        const float cn = P[s].nx * dx + P[s].ny * dy + P[s].nz * dz;
                        const float cw = u.w * dx + v.x * dy + v.y * dz;
                        const float cp = cn * inv;
                        // the smaller distance from the thresholds decides (no number if either is none), in FP64 inside the guard band
                        const float least = __builtin_elementwise_minimum(-(cw * inv) - edge, cp - kConeEps);
                        bool in = least > 0.f;
                        if (fabsf(least) <= kGuard)
                            in = cone_accept_f64(gpos[q[s]], gnrm[q[s]], raw.pos[S.i[j]], raw.dir[S.i[j]], ap.cos_half_d);
                        const float m = in ? cp * (inv * inv) : 0.f;
                        sum[s][0] += v.z * m;
                        sum[s][1] += v.w * m;
                        sum[s][2] += az * m;
                    }
                }
            }
#pragma unroll
            for (int s = 0; s < kExactSlots; ++s)
                for (int c = 0; c < 3; ++c) ka[s][c].add(sum[s][c]);
        }
    }
#pragma unroll
    for (int s = 0; s < kExactSlots; ++s) {
        const int pix = first + 64 * s + lane;
        if (pix >= npix) continue;
        float* o = part + (size_t)blockIdx.y * 6 * npix + pix;
        const float b[3] = {P[s].br, P[s].bg, P[s].bb};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            if (DO_RAD) o[c * (size_t)npix] = kr[s][c].s * b[c];
            if (DO_ANTI) o[(3 + c) * (size_t)npix] = ka[s][c].s * b[c];
        }
    }
}

// Sums the splits and writes the float4 targets (kernel_combine semantics:
// result = radiance - antiradiance including w, i.e. 1 - 1 = 0).
// Radiance comes from rad_splits splits of `part`, or from rad_in when
// rad_splits < 0 (the cut kernel wrote it); antiradiance from anti_splits
// splits (0: none).  A pixel's splits are summed by kSlices threads: one chain
// of 313 (48x32 pixels, 5000 AVPLs) took 180 us.
template <int kSlices>
__global__ __launch_bounds__(kThreads) void k_finalize(const float* __restrict__ part, int rad_splits,
                                                       int anti_splits, int npix,
                                                       const float4* __restrict__ rad_in,
                                                       float4* __restrict__ out_rad,
                                                       float4* __restrict__ out_anti,
                                                       float4* __restrict__ out_res) {
    constexpr int kPix = kThreads / kSlices;
    const int pix = blockIdx.x * kPix + threadIdx.x % kPix, slice = threadIdx.x / kPix;
    Kahan k[6];
    if (pix < npix) {
        for (int s = slice; s < rad_splits; s += kSlices)
            for (int c = 0; c < 3; ++c) k[c].add(part[((size_t)s * 6 + c) * npix + pix]);
        for (int s = slice; s < anti_splits; s += kSlices)
            for (int c = 3; c < 6; ++c) k[c].add(part[((size_t)s * 6 + c) * npix + pix]);
    }
    if constexpr (kSlices > 1) {
        __shared__ float sum[kSlices][6][kPix];
        for (int c = 0; c < 6; ++c) sum[slice][c][threadIdx.x % kPix] = k[c].s;
        __syncthreads();
        if (slice > 0) return;
        for (int s = 1; s < kSlices; ++s)
            for (int c = 0; c < 6; ++c) k[c].add(sum[s][c][threadIdx.x]);
    }
    if (pix >= npix) return;
    const float4 rad = rad_splits >= 0 ? make_float4(k[0].s, k[1].s, k[2].s, 1.f) : rad_in[pix];
    const float4 anti = make_float4(k[3].s, k[4].s, k[5].s, 1.f);
    if (rad_splits >= 0 && out_rad) out_rad[pix] = rad;
    if (out_anti) out_anti[pix] = anti;
    if (out_res)
        out_res[pix] = make_float4(rad.x - anti.x, rad.y - anti.y, rad.z - anti.z, rad.w - anti.w);
}

// --------------------------------------------------------- exact f64 ----
template <int MODEL>
__global__ __launch_bounds__(kThreads) void k_exact_f64(arc::AvplsDev a, const float4* __restrict__ gpos,
                                                        const float4* __restrict__ gnrm,
                                                        const float4* __restrict__ galb,
                                                        const arc_material* __restrict__ mats, int npix,
                                                        float camx, float camy, float camz, float radius,
                                                        double cos_half, int chunk,
                                                        double* __restrict__ part) {
    using V3 = V<double>;
    const int pix = blockIdx.x * kThreads + threadIdx.x;
    const bool live = pix < npix;
    const int q = live ? pix : 0;
    const float4 p4 = gpos[q], n4 = gnrm[q];
    const V3 pos = mk<double>(p4.x, p4.y, p4.z), nrm = mk<double>(n4.x, n4.y, n4.z);
    Mat<double> pm = material<double>(mats, (int)n4.w);
    if (galb) pm.diffuse = mk<double>(galb[q].x, galb[q].y, galb[q].z);
    const V3 cam = mk<double>(camx, camy, camz);
    const int a0 = blockIdx.y * chunk, a1 = min(a.n, a0 + chunk);
    V3 R = mk<double>(0, 0, 0), A = mk<double>(0, 0, 0);
    for (int i = a0; i < a1; ++i) {
        const V3 apos = ld3<double>(a.pos[i]), anrm = ld3<double>(a.nrm[i]), aw = ld3<double>(a.dir[i]);
        const Mat<double> am = material<double>(mats, a.mat[i]);
        R = R + radiance(pos, nrm, pm, apos, anrm, aw, ld3<double>(a.rad[i]), am, cam);
        if (a.anti) {
            const V3 Av = ld3<double>(a.anti[i]);
            if (MODEL == ARC_ANTIRAD_DISK)
                A = A + antirad_disk(pos, nrm, pm, apos, anrm, aw, Av, cam, (double)radius);
            else
                A = A + antirad_cone(pos, nrm, pm, apos, aw, Av, cam, cos_half);
        }
    }
    if (!live) return;
    double* o = part + (size_t)blockIdx.y * 6 * npix + pix;
    o[0] = R.x; o[(size_t)npix] = R.y; o[2 * (size_t)npix] = R.z;
    o[3 * (size_t)npix] = A.x; o[4 * (size_t)npix] = A.y; o[5 * (size_t)npix] = A.z;
}

__global__ __launch_bounds__(kThreads) void k_finalize_f64(const double* __restrict__ part, int splits, int npix,
                                                           double* __restrict__ rad3, double* __restrict__ anti3) {
    const int pix = blockIdx.x * kThreads + threadIdx.x;
    if (pix >= npix) return;
    double s[6] = {0, 0, 0, 0, 0, 0};
    for (int k = 0; k < splits; ++k)
        for (int c = 0; c < 6; ++c) s[c] += part[((size_t)k * 6 + c) * npix + pix];
    for (int c = 0; c < 3; ++c) {
        if (rad3) rad3[3 * (size_t)pix + c] = s[c];
        if (anti3) anti3[3 * (size_t)pix + c] = s[3 + c];
    }
}

// ------------------------------------------------------ cut (solid) ----
// Decision arithmetic of kernel_bvh (cudaGather.cu:405-414) in FP32 with IEEE
// division and square root and no fused multiply-add, so every traversal
// decision equals the oracle's REF32 decision.
__device__ inline bool cluster_visible(f3 n, f3 p, f3 bmin, f3 bmax) {
#pragma clang fp contract(off)
    const float ax = bmax.x - p.x, ay = bmax.y - p.y, az = bmax.z - p.z;
    const float sa = 1.0f / sqrtf(ax * ax + ay * ay + az * az);
    const float c1 = n.x * (ax * sa) + n.y * (ay * sa) + n.z * (az * sa);
    const float bx = bmin.x - p.x, by = bmin.y - p.y, bz = bmin.z - p.z;
    const float sb = 1.0f / sqrtf(bx * bx + by * by + bz * bz);
    const float c2 = n.x * (bx * sb) + n.y * (by * sb) + n.z * (bz * sb);
    return (c1 > 0.f) || (c2 > 0.f);
}

__device__ inline bool solid_angle_below(f3 p, f3 rep, f3 bmin, f3 bmax, float thresh) {
#pragma clang fp contract(off)
    const float ex = bmax.x - bmin.x, ey = bmax.y - bmin.y, ez = bmax.z - bmin.z;
    const float radius = 0.5f * sqrtf(ex * ex + ey * ey + ez * ez);
    const float dx = rep.x - p.x, dy = rep.y - p.y, dz = rep.z - p.z;
    const float dist = sqrtf(dx * dx + dy * dy + dz * dz);
    const float omega = (2.0f * kPi) * (1.0f - dist / sqrtf(radius * radius + dist * dist));
    return omega < thresh;
}

struct CutTree {
    const arc_bvh_node* nodes;
    const int* mat;
    const f3* pos;
    const f3* nrm;
    const f3* rad;
    const f3* dir;
    int n;  // leaves
};

// The cut's records: a leaf's (position, 0), (unit normal, 0), (radiance times
// the AVPL's Lambertian reflectance, 0) and an inner node's (box lo, left),
// (box hi, right), (position, far), (unit normal, near), (radiance, 0) of its
// representative.  With squared distance d2 from a pixel to the
// representative, d2 > far is certainly below the threshold, d2 < near
// certainly not (SaBand).
constexpr int kSaLeaf = 3, kSaNode = 5;

// Omega = 2 pi (1 - d / sqrt(r^2 + d^2)) < thresh is d2 > ratio(thresh) r2; its
// FP32 value carries at most 2.3e-6 of rounding (4 ulp of 1 in the quotient),
// so it is certain where the threshold moved by 4e-6 either way gives the same
// answer (far, near: the ratios of the moved thresholds).
struct SaBand {
    float far, near;
};

SaBand sa_band(float thresh) {
    auto ratio = [](double t) {
        const double q = 1.0 - t / (2.0 * M_PI);
        if (q >= 1.0) return (double)INFINITY;
        if (q <= 0.0) return -1.0;
        return q * q / (1.0 - q * q);
    };
    const double lo = ratio((double)thresh - 4e-6), hi = ratio((double)thresh + 4e-6);
    return SaBand{(float)(lo * (1.0 + 2e-6)), (float)(hi * (1.0 - 2e-6))};
}

__global__ __launch_bounds__(kThreads) void k_sa_records(CutTree t, const arc_material* __restrict__ mats, SaBand band,
                                                         float4* __restrict__ rec) {
    const int i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= 2 * t.n - 1) return;
    const V<float> p = ld3<float>(t.pos[i]), nrm = normalize(ld3<float>(t.nrm[i])), w = ld3<float>(t.dir[i]);
    V<float> c = ld3<float>(t.rad[i]);
    if (length(w) != 0.f) c = c * (kOneOverPi * material<float>(mats, t.mat[i]).diffuse);
    float far = 0.f, near = 0.f;
    float4* r = rec + kSaLeaf * (size_t)i;
    if (i >= t.n) {
        const arc_bvh_node b = t.nodes[i - t.n];
        const float ex = b.bbMax.x - b.bbMin.x, ey = b.bbMax.y - b.bbMin.y, ez = b.bbMax.z - b.bbMin.z;
        const float r2 = 0.25f * (ex * ex + ey * ey + ez * ez);
        // below 1e-30 the squares lose their accuracy: neither
        far = band.far * r2 + 1e-30f;
        near = band.near * r2 - 1e-30f;
        r = rec + kSaLeaf * (size_t)t.n + kSaNode * (size_t)(i - t.n);
        r[0] = make_float4(b.bbMin.x, b.bbMin.y, b.bbMin.z, __int_as_float(b.left));
        r[1] = make_float4(b.bbMax.x, b.bbMax.y, b.bbMax.z, __int_as_float(b.right));
        r += 2;
    }
    r[0] = make_float4(p.x, p.y, p.z, far);
    r[1] = make_float4(nrm.x, nrm.y, nrm.z, near);
    r[2] = make_float4(c.x, c.y, c.z, 0.f);
}

// kernel_bvh (cudaGather.cu:375-433): each pixel's depth-first cut, the right
// child first.
//
// A wave walks the union of its 8x8 pixels' cuts: an entry of the stack is a
// node and the set of pixels that reach it, so the records are read by scalar
// loads, the stack is one for the wave, and no lane waits for another's branch.
// Neighbouring pixels' cuts are nearly equal.  A pixel sees the nodes in the
// order of its own traversal, and it is in every entry above which its node
// lies: the stack's height is its own stack's, which may overflow
// (stack_size; the pixel is then an error, as in kernel_bvh).
//
// The decisions are made without square roots and divisions wherever the FP32
// formulas' rounding cannot change them, and by these formulas elsewhere.  A
// corner's test is the sign of n . (corner - p), here n . corner - n . p: both
// carry at most 4 ulp of the terms' absolute sums, against a guard of 1e-6 of
// these sums at the scene's largest coordinates (and 1e-12, below which the
// formula's squares may underflow).
//
// Bound: vector and scalar instructions, about 40 of each per visited node
// (half of them its share of the evaluations), and the reads' latency where
// few waves hide it.  1280x720 pixels over 65536 AVPLs: 3.64 ms where each lane
// walked its own tree with the formulas (a wave then waits for its longest
// lane and runs every branch of each step), 0.95 here; 1.33 with the corners'
// differences taken before the products and the stack in LDS.  Fetching the
// right child's record ahead made it 1.1, and a 160x120 image 5 % faster.
constexpr float kSaGuard = 1e-6f;
constexpr int kSaStack = 64;  // entries: a pixel's stack is at most that high

template <bool GENERAL>
__global__ __launch_bounds__(kThreads) void k_cut_sa(CutTree t, const float4* __restrict__ rec,
                                                     const float4* __restrict__ gpos,
                                                     const float4* __restrict__ gnrm,
                                                     const float4* __restrict__ galb,
                                                     const arc_material* __restrict__ mats, int W, int H,
                                                     float camx, float camy, float camz, float thresh,
                                                     int stack_size, int sentinel,
                                                     float4* __restrict__ out_rad,
                                                     unsigned long long* __restrict__ counters) {
    static_assert(kSaStack == 64, "the stack is a register's lanes");
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int tw = (W + 15) / 16, b = xcd_block(blockIdx.x, tw * ((H + 15) / 16));
    const int x = (b % tw) * 16 + (wave & 1) * 8 + (lane & 7);
    const int y = (b / tw) * 16 + (wave >> 1) * 8 + (lane >> 3);
    const bool live = x < W && y < H;
    const int pix = live ? y * W + x : 0;
    const PixelF P = load_pixel(gpos, gnrm, galb, mats, pix);
    const f3 p = f3{P.px, P.py, P.pz}, nraw = f3of(gnrm[pix]);
    ufloat* const root = uptr(rec + kSaLeaf * (size_t)t.n);
    const float np = nraw.x * p.x + nraw.y * p.y + nraw.z * p.z;
    const float scale = fabsf(nraw.x) * (fabsf(p.x) + fmaxf(fabsf(root[0]), fabsf(root[4]))) +
                        fabsf(nraw.y) * (fabsf(p.y) + fmaxf(fabsf(root[1]), fabsf(root[5]))) +
                        fabsf(nraw.z) * (fabsf(p.z) + fmaxf(fabsf(root[2]), fabsf(root[6])));
    const float guard = kSaGuard * scale + 1e-12f;
    // the guards hold for magnitudes whose squares stay finite and for numbers;
    // a pixel outside them is decided by the formulas throughout
    const float far_out = fabsf(p.x) + fabsf(p.y) + fabsf(p.z) + fabsf(root[0]) + fabsf(root[1]) + fabsf(root[2]) +
                          fabsf(root[4]) + fabsf(root[5]) + fabsf(root[6]);
    const bool plain = far_out < 1e15f && fabsf(nraw.x) + fabsf(nraw.y) + fabsf(nraw.z) < 1e3f;
    const uint64_t odd = __ballot(!plain);
    uint64_t alive = __ballot(live), erred = 0;
    unsigned nvis = 0, neval = 0;
    V<float> R = mk(0.f, 0.f, 0.f);
    // the sum is taken without the Lambertian pixel's reflectance
    auto eval = [&](ufloat* r, int idx, uint64_t m) {
        neval += __popcll(m);
        if (!__builtin_amdgcn_inverse_ballot_w64(m)) return;
        if constexpr (GENERAL) {
            Mat<float> pm = material<float>(mats, P.mat);
            if (galb) pm.diffuse = mk(galb[pix].x, galb[pix].y, galb[pix].z);
            const float4 n4 = gnrm[pix];
            R = R + radiance(mk(P.px, P.py, P.pz), mk(n4.x, n4.y, n4.z), pm, ld3<float>(t.pos[idx]),
                             ld3<float>(t.nrm[idx]), ld3<float>(t.dir[idx]), ld3<float>(t.rad[idx]),
                             material<float>(mats, t.mat[idx]), mk(camx, camy, camz));
        } else {
            const float dx = r[0] - P.px, dy = r[1] - P.py, dz = r[2] - P.pz;
            const float inv = __builtin_amdgcn_rsqf(dx * dx + dy * dy + dz * dz);
            const float c1 = clamp01((P.nx * dx + P.ny * dy + P.nz * dz) * inv);
            const float c2 = clamp01(-(r[4] * dx + r[5] * dy + r[6] * dz) * inv);
            const float gg = (c1 * c2) * (inv * inv);
            R.x += r[8] * gg;
            R.y += r[9] * gg;
            R.z += r[10] * gg;
        }
    };
    // the stack: entry j in lane j
    int snode = 0, slo = 0, shi = 0;
    int sp = 0, node = -1;
    uint64_t m = alive;
    while (m) {
        while (node < 0) {
            const int k = -(node + 1);
            if (k >= t.n - 1) {
                erred |= m;
                alive &= ~m;
                break;
            }
            nvis += __popcll(m);
            ufloat* r = root + 4 * kSaNode * (size_t)k;
            const float r0 = r[0], r1 = r[1], r2 = r[2], r4 = r[4], r5 = r[5], r6 = r[6], r8 = r[8], r9 = r[9],
                        r10 = r[10], far = r[11], near = r[15];
            const int left = __float_as_int(r[3]), right = __float_as_int(r[7]);
            const float sa = __builtin_fmaf(nraw.x, r4, __builtin_fmaf(nraw.y, r5, __builtin_fmaf(nraw.z, r6, -np)));
            const float sb = __builtin_fmaf(nraw.x, r0, __builtin_fmaf(nraw.y, r1, __builtin_fmaf(nraw.z, r2, -np)));
            uint64_t visible = __ballot(sa > guard) | __ballot(sb > guard);
            uint64_t unsure = m & (odd | ~(visible | (__ballot(sa < -guard) & __ballot(sb < -guard))));
            if (unsure) {
                bool v = false;
                if (__builtin_amdgcn_inverse_ballot_w64(unsure)) {
                    // most often the box lies in the pixel's plane, a corner not above it to the last bit
                    const float ax = r4 - p.x, ay = r5 - p.y, az = r6 - p.z, bx = r0 - p.x, by = r1 - p.y, bz = r2 - p.z;
                    const bool ha = sa < -guard || (nraw.x * ax == 0.f && nraw.y * ay == 0.f && nraw.z * az == 0.f &&
                                                    fabsf(ax) + fabsf(ay) + fabsf(az) > 1e-12f);
                    const bool hb = sb < -guard || (nraw.x * bx == 0.f && nraw.y * by == 0.f && nraw.z * bz == 0.f &&
                                                    fabsf(bx) + fabsf(by) + fabsf(bz) > 1e-12f);
                    v = !(plain && ha && hb) && cluster_visible(nraw, p, f3{r0, r1, r2}, f3{r4, r5, r6});
                }
                visible = (visible & ~unsure) | __ballot(v);
            }
            visible &= m;
            const float dx = r8 - p.x, dy = r9 - p.y, dz = r10 - p.z;
            const float d2 = dx * dx + dy * dy + dz * dz;
            uint64_t below = __ballot(d2 > far);
            unsure = visible & (odd | ~(below | __ballot(d2 < near)));
            if (unsure) {
                bool v = false;
                if (__builtin_amdgcn_inverse_ballot_w64(unsure))
                    v = solid_angle_below(p, f3{r8, r9, r10}, f3{r0, r1, r2}, f3{r4, r5, r6}, thresh);
                below = (below & ~unsure) | __ballot(v);
            }
            below &= visible;
            if (below) eval(r + 8, t.n + k, below);
            m = visible & ~below;
            if (!m) break;
            if (sp + 2 >= stack_size) {
                erred |= m;
                alive &= ~m;
                break;
            }
            if (__builtin_amdgcn_inverse_ballot_w64(1ull << sp)) {
                snode = left;
                slo = (int)(uint32_t)m;
                shi = (int)(uint32_t)(m >> 32);
            }
            ++sp;
            node = right;
        }
        if (node >= 0) eval(uptr(rec + kSaLeaf * (size_t)node), node, m);
        do {  // the next entry; pixels that erred are in none any more
            if (sp == 0) {
                m = 0;
                break;
            }
            --sp;
            node = __builtin_amdgcn_readlane(snode, sp);
            m = alive & ((uint64_t)(uint32_t)__builtin_amdgcn_readlane(slo, sp) |
                         (uint64_t)(uint32_t)__builtin_amdgcn_readlane(shi, sp) << 32);
        } while (!m);
    }
    if (live) {
        float4 o = GENERAL ? make_float4(R.x, R.y, R.z, 1.f) : make_float4(R.x * P.br, R.y * P.bg, R.z * P.bb, 1.f);
        if (sentinel && __builtin_amdgcn_inverse_ballot_w64(erred)) o = make_float4(100000.f, 0.f, 100000.f, 1.f);
        out_rad[pix] = o;
    }
    if (counters && lane == 0) {  // one atomic per wave
        atomicAdd(&counters[C_VISITED], (unsigned long long)nvis);
        atomicAdd(&counters[C_EVALUATED], (unsigned long long)neval);
        atomicAdd(&counters[C_ERRORS], (unsigned long long)__popcll(erred));
    }
}

// ------------------------------------------------------------- host ----
inline int blocks(long long n) { return (int)((n + kThreads - 1) / kThreads); }

int pick_splits(int npix, int n_avpl) {
    const int pblocks = blocks(npix);
    int s = (2048 + pblocks - 1) / pblocks;
    s = std::max(1, std::min(s, (n_avpl + 255) / 256));
    return s;
}

// The exact kernels' waves cost alike, so their number should fill the chip
// (two to three blocks of each CU's four are resident) and no more, each split
// being written and read once; a split of less than 32 AVPLs costs more to
// start than it saves.  At least 256 per split left a 64x48 image with 500
// AVPLs at 24 blocks, 138 us; 18 us here.
int exact_splits(const arc_gather* g, int npix, int n_avpl) {
    const int per = g->general ? kThreads : kThreads * kExactSlots, pblocks = (npix + per - 1) / per;
    return std::max(1, std::min(2048 / pblocks, (n_avpl + 31) / 32));
}

template <int MODEL, bool DO_RAD, bool DO_ANTI>
void launch_exact(arc_gather* g, const arc::AvplsDev& a, int chunk, int splits, float3 cam, float radius,
                  double cos_half) {
    const int npix = g->width * g->height;
    if (g->general)
        hipLaunchKernelGGL((k_exact_glossy<MODEL, DO_RAD, DO_ANTI>), dim3(blocks(npix), splits), dim3(kThreads), 0,
                           g->ctx->stream, g->rec.as<float4>(), a, chunk, g->gpos, g->gnrm, g->galb,
                           g->mats.as<arc_material>(), npix, cam.x, cam.y, cam.z, anti_params(radius, cos_half),
                           g->part.as<float>());
    else
        hipLaunchKernelGGL((k_exact_lambert<MODEL, DO_RAD, DO_ANTI>),
                           dim3((npix + kThreads * kExactSlots - 1) / (kThreads * kExactSlots), splits), dim3(kThreads),
                           0, g->ctx->stream, g->rec.as<float4>(), a, chunk, g->gpos, g->gnrm, g->galb,
                           g->mats.as<arc_material>(), npix, anti_params(radius, cos_half), g->part.as<float>());
}

template <bool DO_RAD, bool DO_ANTI>
void dispatch_exact(arc_gather* g, int model, const arc::AvplsDev& a, int chunk, int splits, float3 cam,
                    float radius, double cos_half) {
    if (model == ARC_ANTIRAD_DISK) launch_exact<ARC_ANTIRAD_DISK, DO_RAD, DO_ANTI>(g, a, chunk, splits, cam, radius, cos_half);
    else launch_exact<ARC_ANTIRAD_CONE, DO_RAD, DO_ANTI>(g, a, chunk, splits, cam, radius, cos_half);
}

// Eight threads per pixel where there are splits for them.
void finalize(arc_gather* g, int rad_splits, int anti_splits, int npix, float4* rad, float4* anti, float4* res) {
    auto launch = [&](auto kernel, int slices) {
        const int per = kThreads / slices;
        hipLaunchKernelGGL(kernel, dim3((npix + per - 1) / per), dim3(kThreads), 0, g->ctx->stream, g->part.as<float>(),
                           rad_splits, anti_splits, npix, rad, rad, anti, res);
    };
    if (std::max(rad_splits, anti_splits) > 8) launch(k_finalize<8>, 8);
    else launch(k_finalize<1>, 1);
}

// g->crec for n AVPLs: one size for every cut's records, so that a frame of
// another cut does not move the buffer from under a captured graph.
int ensure_records(arc_gather* g, int n) {
    static_assert(kSaLeaf + kSaNode <= 2 * arc::kCrec, "the solid-angle cut's records fit");
    return arc::ensure(g->ctx, g->crec, sizeof(float4) * 2 * arc::kCrec * (size_t)n);
}

// This frame's LBVH for the error-bound and learned cuts, with their node
// records in g->crec.
int build_cut_tree(arc_gather* g, const arc::AvplsDev& a, bool validate) {
    g->mom_ready = false;
    if (a.n > 1) ARC_TRY(ensure_records(g, a.n));
    return arc::bvh_build_cut(g->bvh, a, validate, g->mats.as<arc_material>(), g->crec.as<float4>());
}

// AVPL pointers on the device, staging host input when asked (AvplsGpu,
// data_gpu.cu:5-52).
int stage_avpls(arc_gather* g, const arc_avpls* in, int flags, arc::AvplsDev& out) {
    arc_ctx* ctx = g->ctx;
    const int n = in->numAvpls;
    out.n = n;
    if (!(flags & ARC_INPUT_HOST)) {
        out.pos = reinterpret_cast<const f3*>(in->position);
        out.nrm = reinterpret_cast<const f3*>(in->normal);
        out.dir = reinterpret_cast<const f3*>(in->incDirection);
        out.rad = reinterpret_cast<const f3*>(in->incRadiance);
        out.anti = reinterpret_cast<const f3*>(in->antiradiance);
        out.mat = in->materialIndex;
        out.bounce = in->bounce;
        return ARC_OK;
    }
    const size_t v3 = sizeof(f3) * (size_t)n, vi = sizeof(int) * (size_t)n;
    ARC_TRY(arc::ensure(ctx, g->stage, 5 * v3 + 2 * vi));
    char* base = g->stage.as<char>();
    const void* src[7] = {in->position, in->normal, in->incDirection, in->incRadiance, in->antiradiance,
                          in->materialIndex, in->bounce};
    const size_t sz[7] = {v3, v3, v3, v3, v3, vi, vi};
    char* dst[7];
    size_t off = 0;
    for (int k = 0; k < 7; ++k) {
        dst[k] = base + off;
        off += sz[k];
        if (src[k]) ARC_HIP(ctx, hipMemcpyAsync(dst[k], src[k], sz[k], hipMemcpyHostToDevice, ctx->stream));
    }
    // the caller may free or reuse its host arrays once the call returns
    ARC_HIP(ctx, hipStreamSynchronize(ctx->stream));
    out.pos = reinterpret_cast<const f3*>(dst[0]);
    out.nrm = reinterpret_cast<const f3*>(dst[1]);
    out.dir = reinterpret_cast<const f3*>(dst[2]);
    out.rad = reinterpret_cast<const f3*>(dst[3]);
    out.anti = in->antiradiance ? reinterpret_cast<const f3*>(dst[4]) : nullptr;
    out.mat = reinterpret_cast<const int*>(dst[5]);
    out.bounce = in->bounce ? reinterpret_cast<const int*>(dst[6]) : nullptr;
    return ARC_OK;
}

int validate_params(arc_gather* g, const arc_avpls* avpls, const arc_gather_params* p) {
    if (!g || !avpls || !p) return ARC_E_INVALID;
    if (!g->gpos || !g->gnrm) return arc::fail(g->ctx, ARC_E_STATE, "no G-buffer bound");
    if (avpls->numAvpls < 0) return arc::fail(g->ctx, ARC_E_INVALID, "numAvpls < 0");
    if (avpls->numAvpls > 0 && (!avpls->position || !avpls->normal || !avpls->incDirection ||
                                !avpls->incRadiance || !avpls->materialIndex))
        return arc::fail(g->ctx, ARC_E_INVALID, "AVPL arrays missing");
    if (p->antiradianceModel != ARC_ANTIRAD_DISK && p->antiradianceModel != ARC_ANTIRAD_CONE)
        return arc::fail(g->ctx, ARC_E_INVALID, "antiradianceModel");
    if (p->stackSize < 2 || p->stackSize > 64) return arc::fail(g->ctx, ARC_E_INVALID, "stackSize out of [2, 64]");
    if (p->antiradianceMode != ARC_ANTI_EXACT && p->antiradianceMode != ARC_ANTI_CLUSTERED)
        return arc::fail(g->ctx, ARC_E_INVALID, "antiradianceMode");
    return ARC_OK;
}

float4* target(DevBuf& internal, float4* user, arc_gather* g, int& status) {
    if (user) return user;
    status = arc::ensure(g->ctx, internal, sizeof(float4) * (size_t)g->width * g->height);
    return internal.as<float4>();
}

}  // namespace

extern "C" {

void arc_gather_params_default(arc_gather_params* p) {
    if (!p) return;
    std::memset(p, 0, sizeof(*p));
    p->useLightCuts = 1;                        // CConfigManager.cpp:15
    p->cutMode = ARC_CUT_SOLID_ANGLE;
    p->clusterRefinementThreshold = (float)(M_PI / 10.0);  // CConfigManager.cpp:37
    p->errorBound = 0.01f;
    p->antiradianceModel = ARC_ANTIRAD_DISK;
    p->antiradianceMode = ARC_ANTI_CLUSTERED;   // useClusteredDeferred = 1, CConfigManager.cpp:16
    p->photonRadiusScale = 2.0f;                // CConfigManager.cpp:26
    p->coneHalfAngle = (float)(M_PI / 18.0);
    p->writeSentinel = 1;
    p->stackSize = 32;                          // STACK_SIZE, cudaGather.cu:19
    p->seed = 5489;
    p->cutEstimateDepth = 6;
    p->cutBudget = 1 << 16;
    p->cutPerTile = 0;
    p->cutCriterion = ARC_CRITERION_ESTIMATE;
    p->cutImageFloor = 1.0f;
    p->cutConfidence = 0.9f;
    p->cutEvalDepth = 0;
    p->cutEstimator = ARC_ESTIMATOR_CENTROID;
    p->cutExactCount = 16;
    p->cutOpening = 0.3f;
}

int arc_gather_create(arc_ctx* ctx, int width, int height, const arc_material* materials, int num_materials,
                      arc_gather** out) {
    if (!ctx || !out || width <= 0 || height <= 0 || !materials || num_materials <= 0 || num_materials > 256)
        return ARC_E_INVALID;
    arc_gather* g = new arc_gather();
    g->ctx = ctx;
    g->width = width;
    g->height = height;
    g->num_mats = num_materials;
    for (int i = 0; i < num_materials; ++i) {
        const arc_float3& s = materials[i].specular;
        if (std::sqrt(s.x * s.x + s.y * s.y + s.z * s.z) > 0.f) g->general = true;
    }
    // zero-padded to kMaxMaterials entries: kernels mask indices into the table
    std::vector<arc_material> table(kMaxMaterials);
    std::memset(table.data(), 0, sizeof(arc_material) * table.size());
    std::memcpy(table.data(), materials, sizeof(arc_material) * (size_t)num_materials);
    int st = arc::ensure(ctx, g->mats, sizeof(arc_material) * table.size());
    if (st == ARC_OK) {
        hipError_t e = hipMemcpy(g->mats.p, table.data(), sizeof(arc_material) * table.size(),
                                 hipMemcpyHostToDevice);
        if (e != hipSuccess) st = arc::hip_fail(ctx, e, "hipMemcpy(materials)", __FILE__, __LINE__);
    }
    if (st == ARC_OK) st = arc::ensure(ctx, g->counters, sizeof(unsigned long long) * C_NUM);
    for (int f = 0; st == ARC_OK && f < arc_gather::kRing; ++f)
        for (int i = 0; st == ARC_OK && i < arc_gather::kMarks; ++i) {
            hipError_t e = hipEventCreate(&g->ev[f][i]);
            if (e != hipSuccess) st = arc::hip_fail(ctx, e, "hipEventCreate", __FILE__, __LINE__);
        }
    if (st == ARC_OK) st = arc_bvh_create(ctx, 0, &g->bvh);
    // the frame's tree is rebuilt beside the antiradiance on the second stream
    if (st == ARC_OK) {
        hipError_t e = hipStreamCreateWithFlags(&g->aux, hipStreamNonBlocking);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&g->fork, hipEventDisableTiming);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&g->join, hipEventDisableTiming);
        if (e != hipSuccess) st = arc::hip_fail(ctx, e, "aux stream", __FILE__, __LINE__);
    }
    if (st != ARC_OK) {
        arc_gather_destroy(g);
        return st;
    }
    *out = g;
    return ARC_OK;
}

void arc_gather_destroy(arc_gather* g) {
    if (!g) return;
    if (g->aux) {
        (void)hipStreamSynchronize(g->aux);
        (void)hipStreamDestroy(g->aux);
    }
    if (g->fork) (void)hipEventDestroy(g->fork);
    if (g->join) (void)hipEventDestroy(g->join);
    for (int f = 0; f < arc_gather::kRing; ++f)
        for (int i = 0; i < arc_gather::kMarks; ++i)
            if (g->ev[f][i]) (void)hipEventDestroy(g->ev[f][i]);
    arc::release(g->mats);
    arc::release(g->int_rad);
    arc::release(g->int_anti);
    arc::release(g->int_res);
    arc::release(g->rec);
    arc::release(g->part);
    arc::release(g->counters);
    arc::release(g->stage);
    arc::release(g->anti_idx);
    arc::release(g->cbox);
    arc::release(g->ccount);
    arc::release(g->clist);
    arc::release(g->crec);
    arc::release(g->mom);
    arc::release(g->mom_pre);
    arc::release(g->mom_tot);
    arc::release(g->mom_nbox);
    arc::release(g->mom_trav);
    arc::release_pool(g->pool);
    arc::release(g->cest);
    arc_bvh_destroy(g->bvh);
    delete g;
}

int arc_gather_set_gbuffer(arc_gather* g, const float* pos4, const float* nrm4, const float* albedo4) {
    if (!g || !pos4 || !nrm4) return ARC_E_INVALID;
    g->gpos = reinterpret_cast<const float4*>(pos4);
    g->gnrm = reinterpret_cast<const float4*>(nrm4);
    g->galb = reinterpret_cast<const float4*>(albedo4);
    return ARC_OK;
}

int arc_gather_set_outputs(arc_gather* g, float* result4, float* radiance4, float* antiradiance4) {
    if (!g) return ARC_E_INVALID;
    g->out_res = reinterpret_cast<float4*>(result4);
    g->out_rad = reinterpret_cast<float4*>(radiance4);
    g->out_anti = reinterpret_cast<float4*>(antiradiance4);
    return ARC_OK;
}

arc_bvh* arc_gather_get_bvh(arc_gather* g) { return (g && g->bvh && g->bvh->n > 0) ? g->bvh : nullptr; }

int arc_gather_copy_cut_records(arc_gather* g, int which, float* host, long long max_float4, long long* count) {
    if (!g || !count || max_float4 < 0 || (max_float4 > 0 && !host)) return ARC_E_INVALID;
    if (which != ARC_RECORDS_CENTROID && which != ARC_RECORDS_MOMENTS) return ARC_E_INVALID;
    arc_ctx* ctx = g->ctx;
    const int n = g->bvh ? g->bvh->n : 0;
    *count = 0;
    if (n < 2 || !g->bvh->has_cut_records) return arc::fail(ctx, ARC_E_STATE, "no error-bound cut frame has run");
    const arc::DevBuf& buf = which == ARC_RECORDS_CENTROID ? g->crec : g->mom;
    const long long avail = which == ARC_RECORDS_CENTROID ? (long long)arc::kCrec * (2LL * n - 1) : 13LL * (n - 1);
    if (!buf.p || buf.bytes < sizeof(float4) * (size_t)avail || (which == ARC_RECORDS_MOMENTS && !g->mom_ready))
        return arc::fail(ctx, ARC_E_STATE, "records of this kind were not built by the last frame");
    *count = avail;
    const long long m = std::min(avail, max_float4);
    if (m > 0) {
        ARC_HIP(ctx, hipStreamSynchronize(ctx->stream));
        ARC_HIP(ctx, hipMemcpy(host, buf.p, sizeof(float4) * (size_t)m, hipMemcpyDeviceToHost));
    }
    return ARC_OK;
}

int arc_gather_run(arc_gather* g, const arc_avpls* avpls, arc_float3 camPos, float sceneExtent,
                   const arc_gather_params* p, int flags, arc_gather_stats* stats) {
    ARC_TRY(validate_params(g, avpls, p));
    arc_ctx* ctx = g->ctx;
    const bool profile = (flags & (ARC_RUN_PROFILE | ARC_RUN_TIMELINE)) != 0;
    const int slot = g->ring_next;
    hipEvent_t* ev = g->ev[slot];
    const bool count = (flags & ARC_RUN_COUNTERS) != 0;
    const int npix = g->width * g->height;
    const int n = avpls->numAvpls;
    const float radius = p->photonRadiusScale * sceneExtent / 100.f;  // cudaGather.cu:949
    const double cos_half = std::cos((double)p->coneHalfAngle);
    const float3 cam = make_float3(camPos.x, camPos.y, camPos.z);
    int st = ARC_OK;
    float4* rad = target(g->int_rad, g->out_rad, g, st);
    ARC_TRY(st);
    float4* res = g->out_res;
    float4* anti = g->out_anti;
    if (stats) std::memset(stats, 0, sizeof(*stats));
    if (count) ARC_HIP(ctx, hipMemsetAsync(g->counters.p, 0, sizeof(unsigned long long) * C_NUM, ctx->stream));
    if (profile) ARC_HIP(ctx, hipEventRecord(ev[0], ctx->stream));

    arc::AvplsDev a{};
    ARC_TRY(stage_avpls(g, avpls, flags, a));
    if (n > 0) {
        ARC_TRY(arc::ensure(ctx, g->rec, sizeof(float4) * kRecF4 * (size_t)n));
        hipLaunchKernelGGL(k_pack, dim3(blocks(n)), dim3(kThreads), 0, ctx->stream, a, g->mats.as<arc_material>(),
                           g->general ? 1 : 0, p->antiradianceModel, 1.0f / (kPi * radius * radius),
                           g->rec.as<float4>());
        ARC_LAUNCHED(ctx);
    }
    if (profile) ARC_HIP(ctx, hipEventRecord(ev[1], ctx->stream));

    const int splits = exact_splits(g, npix, std::max(n, 1));
    const int chunk = (std::max(n, 1) + splits - 1) / splits;
    ARC_TRY(arc::ensure(ctx, g->part, sizeof(float) * 6 * (size_t)splits * npix));
    unsigned long long* counters = count ? g->counters.as<unsigned long long>() : nullptr;

    const bool cut = p->useLightCuts && n > 1;
    const bool clustered = p->antiradianceMode == ARC_ANTI_CLUSTERED && n > 0;
    // the clustered antiradiance of a cut frame needs neither the LBVH nor the
    // radiance: it runs on the gather's second stream meanwhile.  Not while
    // the stream is being captured into a graph (arc_batch_capture): there
    // the frame stays on one stream.
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    ARC_HIP(ctx, hipStreamIsCapturing(ctx->stream, &capture));
    const bool overlap = cut && clustered && capture == hipStreamCaptureStatusNone;
    if (p->useLightCuts && p->cutMode != ARC_CUT_SOLID_ANGLE && p->cutMode != ARC_CUT_ERROR_BOUND &&
        p->cutMode != ARC_CUT_LEARNED)
        return arc::fail(ctx, ARC_E_INVALID, "cutMode");
    const bool moments = p->cutMode != ARC_CUT_SOLID_ANGLE;
    if (p->useLightCuts && moments && g->general)
        return arc::fail(ctx, ARC_E_UNSUPPORTED, "the error-bound and learned cuts need Lambertian materials");
    if (p->useLightCuts && p->cutMode == ARC_CUT_LEARNED && !(g->net && g->net->ready))
        return arc::fail(ctx, ARC_E_STATE, "learned cut without a trained arc_cutnet (arc_gather_set_cutnet)");
    if (p->useLightCuts && p->cutMode == ARC_CUT_LEARNED && !(p->cutConfidence >= 0.5f && p->cutConfidence <= 1.f))
        return arc::fail(ctx, ARC_E_INVALID, "cutConfidence");
    if (p->cutEstimateDepth < 0 || p->cutEstimateDepth > 40) return arc::fail(ctx, ARC_E_INVALID, "cutEstimateDepth");
    if (!(p->cutImageFloor >= 0.f)) return arc::fail(ctx, ARC_E_INVALID, "cutImageFloor");
    if (p->cutEvalDepth < 0 || p->cutEvalDepth > 4) return arc::fail(ctx, ARC_E_INVALID, "cutEvalDepth");
    if (p->cutEstimator != ARC_ESTIMATOR_CENTROID && p->cutEstimator != ARC_ESTIMATOR_MOMENTS)
        return arc::fail(ctx, ARC_E_INVALID, "cutEstimator");
    const bool mom_est = p->useLightCuts && p->cutMode == ARC_CUT_ERROR_BOUND && p->cutEstimator == ARC_ESTIMATOR_MOMENTS;
    if (g->defer_cut && (!mom_est || !cut || profile || stats || count))
        return arc::fail(ctx, ARC_E_INVALID, "a frame whose cut joins a batched launch must be a moment-cut frame "
                                             "without profiling or statistics");
    if (p->cutCriterion != ARC_CRITERION_BOUND && p->cutCriterion != ARC_CRITERION_ESTIMATE &&
        p->cutCriterion != ARC_CRITERION_EXPANSION)
        return arc::fail(ctx, ARC_E_INVALID, "cutCriterion");
    if (mom_est && p->cutCriterion == ARC_CRITERION_ESTIMATE)
        return arc::fail(ctx, ARC_E_INVALID, "the moment estimator takes ARC_CRITERION_BOUND or ARC_CRITERION_EXPANSION");
    if (!mom_est && p->useLightCuts && p->cutMode == ARC_CUT_ERROR_BOUND && p->cutCriterion == ARC_CRITERION_EXPANSION)
        return arc::fail(ctx, ARC_E_INVALID, "ARC_CRITERION_EXPANSION needs the moment estimator");
    if (mom_est && (!p->cutPerTile || p->cutEvalDepth != 0))
        return arc::fail(ctx, ARC_E_INVALID, "the moment estimator runs per 8x8 tile (cutPerTile 1, cutEvalDepth 0)");
    if (p->cutExactCount < 0 || (mom_est && p->cutExactCount > 128))
        return arc::fail(ctx, ARC_E_INVALID, "cutExactCount out of [0, 128]");
    if (!(p->cutOpening > 0.f)) return arc::fail(ctx, ARC_E_INVALID, "cutOpening");
    if (p->cutBudget < 1) return arc::fail(ctx, ARC_E_INVALID, "cutBudget");
    // ---- radiance: light cut over this frame's AvplBvh (cudaGather.cu:854-923) or exact
    int rad_splits = -1, anti_splits = 0;
    if (overlap) {
        ARC_HIP(ctx, hipEventRecord(g->fork, ctx->stream));
        ARC_HIP(ctx, hipStreamWaitEvent(g->aux, g->fork, 0));
        hipStream_t main_stream = ctx->stream;
        ctx->stream = g->aux;  // the antiradiance launches go to the second stream
        const int sa = arc::anti_clustered(g, a, p->antiradianceModel, cam, anti_params(radius, cos_half),
                                           (double)p->coneHalfAngle, sceneExtent, g->part.as<float>(), counters,
                                           profile ? ev[7] : nullptr);
        hipError_t e = hipSuccess;
        if (sa == ARC_OK && profile) e = hipEventRecord(ev[8], g->aux);
        if (sa == ARC_OK && e == hipSuccess) e = hipEventRecord(g->join, g->aux);
        ctx->stream = main_stream;
        ARC_TRY(sa);
        if (e != hipSuccess) return arc::hip_fail(ctx, e, "antiradiance stream", __FILE__, __LINE__);
        anti_splits = 1;
    }
    if (cut) {
        // AvplBvh(avpls, false) per frame (cudaGather.cu:858)
        if (moments)
            ARC_TRY(build_cut_tree(g, a, (flags & ARC_TRUST_INPUT) == 0));
        if (mom_est) ARC_TRY(arc::cut_moments_build(g, g->bvh));
        if (!moments)
            ARC_TRY(arc::bvh_build_avpls(g->bvh, a, nullptr, p->seed, (flags & ARC_TRUST_INPUT) == 0));
        if (profile) ARC_HIP(ctx, hipEventRecord(ev[2], ctx->stream));
        arc_bvh* b = g->bvh;
        if (moments) {
            const arc::CutEBParams cp{p->errorBound, p->cutEstimateDepth, 1e-3f * sceneExtent, p->cutBudget,
                                      p->cutPerTile, p->cutCriterion, p->cutImageFloor, p->cutConfidence,
                                      p->cutEvalDepth, p->cutExactCount, p->cutOpening};
            if (p->cutMode == ARC_CUT_LEARNED)
                ARC_TRY(arc::cut_learned(g, b, cp, rad, counters, profile ? ev[6] : nullptr));
            else if (mom_est)
                ARC_TRY(arc::cut_moments(g, b, cp, rad, counters, profile ? ev[6] : nullptr,
                                         g->defer_cut ? &g->def_view : nullptr));
            else
                ARC_TRY(arc::cut_error_bound(g, b, cp, rad, counters, profile ? ev[6] : nullptr));
        } else {
            if (profile) ARC_HIP(ctx, hipEventRecord(ev[6], ctx->stream));
            CutTree t{b->nodes.as<arc_bvh_node>(), b->nd_mat.as<int>(), b->nd_pos.as<f3>(), b->nd_nrm.as<f3>(),
                      b->nd_rad.as<f3>(), b->nd_dir.as<f3>(), b->n};
            ARC_TRY(ensure_records(g, t.n));
            float4* rec = g->crec.as<float4>();
            hipLaunchKernelGGL(k_sa_records, dim3(blocks(2LL * t.n - 1)), dim3(kThreads), 0, ctx->stream, t,
                               g->mats.as<arc_material>(), sa_band(p->clusterRefinementThreshold), rec);
            const dim3 grid(((g->width + 15) / 16) * ((g->height + 15) / 16));
            auto launch = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, ctx->stream, t, rec, g->gpos, g->gnrm, g->galb,
                                   g->mats.as<arc_material>(), g->width, g->height, cam.x, cam.y, cam.z,
                                   p->clusterRefinementThreshold, p->stackSize, p->writeSentinel, rad, counters);
            };
            if (g->general) launch(k_cut_sa<true>);
            else launch(k_cut_sa<false>);
        }
        ARC_LAUNCHED(ctx);
        if (profile) ARC_HIP(ctx, hipEventRecord(ev[3], ctx->stream));
    } else {
        if (profile) ARC_HIP(ctx, hipEventRecord(ev[2], ctx->stream));
        if (profile) ARC_HIP(ctx, hipEventRecord(ev[6], ctx->stream));
        rad_splits = n > 0 ? splits : 0;
        if (n > 0 && !clustered) {  // one pass sums both (kernel_radiance_simple + kernel_antiradiance)
            dispatch_exact<true, true>(g, p->antiradianceModel, a, chunk, splits, cam, radius, cos_half);
            anti_splits = splits;
        } else if (n > 0) {
            dispatch_exact<true, false>(g, p->antiradianceModel, a, chunk, splits, cam, radius, cos_half);
        }
        ARC_LAUNCHED(ctx);
        if (profile) ARC_HIP(ctx, hipEventRecord(ev[3], ctx->stream));
    }
    // ---- antiradiance: clustered lists (kernel_antiradiance_clusterred) or exact
    if (overlap) {
        ARC_HIP(ctx, hipStreamWaitEvent(ctx->stream, g->join, 0));  // what the radiance did not hide
    } else if (clustered) {
        ARC_TRY(arc::anti_clustered(g, a, p->antiradianceModel, cam, anti_params(radius, cos_half),
                                    (double)p->coneHalfAngle, sceneExtent, g->part.as<float>(), counters,
                                    profile ? ev[7] : nullptr));
        anti_splits = 1;
        if (profile) ARC_HIP(ctx, hipEventRecord(ev[8], ctx->stream));
    } else if (cut && n > 0) {
        if (profile) ARC_HIP(ctx, hipEventRecord(ev[7], ctx->stream));
        dispatch_exact<false, true>(g, p->antiradianceModel, a, chunk, splits, cam, radius, cos_half);
        anti_splits = splits;
        ARC_LAUNCHED(ctx);
        if (profile) ARC_HIP(ctx, hipEventRecord(ev[8], ctx->stream));
    } else if (profile) {
        ARC_HIP(ctx, hipEventRecord(ev[7], ctx->stream));  // summed with the radiance: no pass of its own
        ARC_HIP(ctx, hipEventRecord(ev[8], ctx->stream));
    }
    if (g->defer_cut) {
        // the cut of this frame is launched with other views' (arc_batch);
        // arc::gather_finish combines once it has run
        g->def_rad_splits = rad_splits;
        g->def_anti_splits = anti_splits;
        g->def_rad = rad;
        g->deferred = true;
        return ARC_OK;
    }
    if (profile) ARC_HIP(ctx, hipEventRecord(ev[4], ctx->stream));
    finalize(g, rad_splits, anti_splits, npix, rad, anti, res);
    ARC_LAUNCHED(ctx);
    if (profile) ARC_HIP(ctx, hipEventRecord(ev[5], ctx->stream));
    if (stats) {
        stats->numLeafs = cut ? g->bvh->n : 0;
        if (count) {
            unsigned long long c[C_NUM];
            ARC_HIP(ctx, hipMemcpyAsync(c, g->counters.p, sizeof(c), hipMemcpyDeviceToHost, ctx->stream));
            ARC_HIP(ctx, hipStreamSynchronize(ctx->stream));
            stats->visitedNodes = (long long)c[C_VISITED];
            stats->evaluatedNodes = (long long)c[C_EVALUATED];
            stats->antiVisitedNodes = (long long)c[C_ANTI_VISITED];
            stats->antiEvaluatedNodes = (long long)c[C_ANTI_EVALUATED];
            stats->errorPixels = (long long)c[C_ERRORS];
            stats->budgetHits = (long long)c[C_BUDGET];
            stats->fallbackNodes = (long long)c[C_FALLBACK];
            stats->testedNodes = (long long)c[C_TESTED];
            stats->exactLeaves = (long long)c[C_EXACT];
        }
        if (flags & ARC_RUN_PROFILE) {
            ARC_HIP(ctx, hipEventSynchronize(ev[5]));
            float t[5];
            for (int i = 0; i < 5; ++i) ARC_HIP(ctx, hipEventElapsedTime(&t[i], ev[i], ev[i + 1]));
            stats->msUpload = t[0];
            stats->msBvh = t[1];
            stats->msRadiance = t[2];
            stats->msAntiradiance = t[3];
            stats->msCombine = t[4];
            ARC_HIP(ctx, hipEventElapsedTime(&stats->msTotal, ev[0], ev[5]));
        }
    }
    if (profile) {
        g->ring_next = (slot + 1) % arc_gather::kRing;
        g->ring_count = std::min(g->ring_count + 1, arc_gather::kRing);
    }
    return ARC_OK;
}

}  // extern "C"

namespace arc {

int gather_finish(arc_gather* g) {
    if (!g || !g->deferred) return ARC_E_STATE;
    arc_ctx* ctx = g->ctx;
    const int npix = g->width * g->height;
    finalize(g, g->def_rad_splits, g->def_anti_splits, npix, g->def_rad, g->out_anti, g->out_res);
    ARC_LAUNCHED(ctx);
    g->deferred = false;
    return ARC_OK;
}

}  // namespace arc

extern "C" {

int arc_gather_profile_history(arc_gather* g, int frames, float* out) {
    if (!g || frames < 0 || (frames > 0 && !out)) return ARC_E_INVALID;
    arc_ctx* ctx = g->ctx;
    const int n = std::min(frames, g->ring_count);
    for (int k = 0; k < n; ++k) {
        const int slot = (g->ring_next - n + k + arc_gather::kRing) % arc_gather::kRing;
        hipEvent_t* ev = g->ev[slot];
        ARC_HIP(ctx, hipEventSynchronize(ev[5]));
        for (int i = 0; i < 5; ++i) ARC_HIP(ctx, hipEventElapsedTime(&out[6 * k + i], ev[i], ev[i + 1]));
        ARC_HIP(ctx, hipEventElapsedTime(&out[6 * k + 5], ev[0], ev[5]));
    }
    return n;
}

arc_ctx* arc_gather_ctx(arc_gather* g) { return g ? g->ctx : nullptr; }

int arc_gather_kernel_history(arc_gather* g, int frames, float* out) {
    if (!g || frames < 0 || (frames > 0 && !out)) return ARC_E_INVALID;
    arc_ctx* ctx = g->ctx;
    const int n = std::min(frames, g->ring_count);
    for (int k = 0; k < n; ++k) {
        const int slot = (g->ring_next - n + k + arc_gather::kRing) % arc_gather::kRing;
        hipEvent_t* ev = g->ev[slot];
        ARC_HIP(ctx, hipEventSynchronize(ev[5]));
        ARC_HIP(ctx, hipEventElapsedTime(&out[2 * k + 0], ev[6], ev[3]));
        ARC_HIP(ctx, hipEventElapsedTime(&out[2 * k + 1], ev[7], ev[8]));
    }
    return n;
}

int arc_gather_kernel_spans(arc_gather* g, int frames, float* out) {
    if (!g || frames < 0 || (frames > 0 && !out)) return ARC_E_INVALID;
    arc_ctx* ctx = g->ctx;
    const int n = std::min(frames, g->ring_count);
    for (int k = 0; k < n; ++k) {
        const int slot = (g->ring_next - n + k + arc_gather::kRing) % arc_gather::kRing;
        hipEvent_t* ev = g->ev[slot];
        ARC_HIP(ctx, hipEventSynchronize(ev[5]));
        ARC_HIP(ctx, hipEventElapsedTime(&out[4 * k + 0], ev[0], ev[6]));
        ARC_HIP(ctx, hipEventElapsedTime(&out[4 * k + 1], ev[0], ev[3]));
        ARC_HIP(ctx, hipEventElapsedTime(&out[4 * k + 2], ev[0], ev[7]));
        ARC_HIP(ctx, hipEventElapsedTime(&out[4 * k + 3], ev[0], ev[8]));
    }
    return n;
}

int arc_gather_set_cutnet(arc_gather* g, arc_cutnet* net) {
    if (!g) return ARC_E_INVALID;
    if (net && net->ctx->device != g->ctx->device)
        return arc::fail(g->ctx, ARC_E_INVALID, "cutnet on another device");
    g->net = net;
    return ARC_OK;
}

int arc_gather_set_estimate_pool(arc_gather* g, int chunks_per_tile) {
    if (!g) return ARC_E_INVALID;
    if (chunks_per_tile < 0 || chunks_per_tile > 256)
        return arc::fail(g->ctx, ARC_E_INVALID, "estimate pool: 0..256 chunks per tile");
    g->est_chunks = chunks_per_tile;
    g->pool.mem.retry();  // the device may have the memory by now that it refused
    g->pool.last = arc::CutSetting{};
    return ARC_OK;
}

int arc_gather_set_launch_shape(arc_gather* g, int cut_stack, int anti_chunk) {
    if (!g) return ARC_E_INVALID;
    if (cut_stack != 64 && cut_stack != 96 && cut_stack != 128)
        return arc::fail(g->ctx, ARC_E_INVALID, "launch shape: cut_stack is 64, 96 or 128");
    if (anti_chunk != 768 && anti_chunk != 1536 && anti_chunk != 3072)
        return arc::fail(g->ctx, ARC_E_INVALID, "launch shape: anti_chunk is 768, 1536 or 3072");
    g->anti_chunk = anti_chunk;
    return ARC_OK;
}

int arc_gather_cut_samples(arc_gather* g, const arc_avpls* avpls, arc_float3 camPos, float sceneExtent,
                           const arc_gather_params* p, int flags, float* X, float* y, int capacity, uint64_t seed,
                           float keep, int* count) {
    (void)camPos;
    ARC_TRY(validate_params(g, avpls, p));
    arc_ctx* ctx = g->ctx;
    if (!X || !y || capacity < 0 || !count || !(keep > 0.f && keep <= 1.f)) return ARC_E_INVALID;
    if (g->general) return arc::fail(ctx, ARC_E_UNSUPPORTED, "the learned cut needs Lambertian materials");
    if (p->cutEstimateDepth < 0 || p->cutEstimateDepth > 40) return arc::fail(ctx, ARC_E_INVALID, "cutEstimateDepth");
    if (!(p->cutImageFloor >= 0.f)) return arc::fail(ctx, ARC_E_INVALID, "cutImageFloor");
    if (p->cutEvalDepth < 0 || p->cutEvalDepth > 4) return arc::fail(ctx, ARC_E_INVALID, "cutEvalDepth");
    *count = 0;
    const int n = avpls->numAvpls;
    if (n < 2) return ARC_OK;
    arc::AvplsDev a{};
    ARC_TRY(stage_avpls(g, avpls, flags, a));
    ARC_TRY(build_cut_tree(g, a, (flags & ARC_TRUST_INPUT) == 0));
    ARC_TRY(arc::ensure(ctx, g->counters, sizeof(unsigned long long) * C_NUM));
    int* dcount = reinterpret_cast<int*>(g->counters.p);
    ARC_HIP(ctx, hipMemsetAsync(dcount, 0, sizeof(int), ctx->stream));
    const arc::CutEBParams cp{p->errorBound, p->cutEstimateDepth, 1e-3f * sceneExtent, p->cutBudget,
                              1, p->cutCriterion, p->cutImageFloor, p->cutConfidence, 0};
    ARC_TRY(arc::cut_samples(g, g->bvh, cp, X, y, capacity, seed, keep, dcount));
    ARC_HIP(ctx, hipMemcpyAsync(count, dcount, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
    ARC_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return ARC_OK;
}

int arc_gather_exact_f64(arc_gather* g, const arc_avpls* avpls, arc_float3 camPos, float sceneExtent,
                         const arc_gather_params* p, int flags, double* radiance3, double* antiradiance3) {
    ARC_TRY(validate_params(g, avpls, p));
    arc_ctx* ctx = g->ctx;
    const int npix = g->width * g->height;
    const int n = avpls->numAvpls;
    const float radius = p->photonRadiusScale * sceneExtent / 100.f;
    const double cos_half = std::cos((double)p->coneHalfAngle);
    arc::AvplsDev a{};
    ARC_TRY(stage_avpls(g, avpls, flags, a));
    const int splits = pick_splits(npix, std::max(n, 1));
    const int chunk = (std::max(n, 1) + splits - 1) / splits;
    ARC_TRY(arc::ensure(ctx, g->part, sizeof(double) * 6 * (size_t)splits * npix));
    if (n > 0) {
        if (p->antiradianceModel == ARC_ANTIRAD_DISK)
            hipLaunchKernelGGL(k_exact_f64<ARC_ANTIRAD_DISK>, dim3(blocks(npix), splits), dim3(kThreads), 0,
                               ctx->stream, a, g->gpos, g->gnrm, g->galb, g->mats.as<arc_material>(), npix,
                               camPos.x, camPos.y, camPos.z, radius, cos_half, chunk, g->part.as<double>());
        else
            hipLaunchKernelGGL(k_exact_f64<ARC_ANTIRAD_CONE>, dim3(blocks(npix), splits), dim3(kThreads), 0,
                               ctx->stream, a, g->gpos, g->gnrm, g->galb, g->mats.as<arc_material>(), npix,
                               camPos.x, camPos.y, camPos.z, radius, cos_half, chunk, g->part.as<double>());
        ARC_LAUNCHED(ctx);
    }
    hipLaunchKernelGGL(k_finalize_f64, dim3(blocks(npix)), dim3(kThreads), 0, ctx->stream, g->part.as<double>(),
                       n > 0 ? splits : 0, npix, radiance3, antiradiance3);
    ARC_LAUNCHED(ctx);
    return ARC_OK;
}

}  // extern "C"
