// Generalised-winding-number dipole sums on CDNA4.
//
//   direct:  all-pairs sums, one query per lane, sources streamed through
//            the scalar cache (wave-uniform loads → SGPR operands), per-tile
//            partial sums folded with Kahan compensation.
//   tree:    Barnes-Hut over an octree built with octreeDWG's split rule;
//            a wave walks the union of its 64 lanes' traversals with one
//            wave-uniform stack in LDS (node, lane mask), so every node and
//            source load is wave-uniform and each lane still takes exactly
//            the reference's per-query term set.  Few points, and points with
//            little in common, walk alone, with 8 or 64 lanes each.
//
// Terms (reference semantics, d = p − q, r = |d|):
//   plain     A(d·n) / (4π r³ + 1e-8)                         fast_winding_number.cpp:182-184
//   screened  (σρ+1) A(d·n) / (e^{σρ} 4π ρ³ + 1e-7), ρ = max(s, r), r > 1e-10
//                                                             TurboLibiGWN.cu:544-585
// Both are evaluated with numerator and denominator divided by 4π (A·n is
// pre-scaled by 1/(4π) when sources are packed), which is the same value.
#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>
#include <vector>

#include "gwn.h"
#include "scan.h"

namespace dwg {

// ---------------------------------------------------------------------------
// per-pair terms
// ---------------------------------------------------------------------------
// max of two non-negative floats on their bit patterns (the integer order is
// the float order there): one instruction, no NaN quieting of the operands
__device__ __forceinline__ float max_nonneg(float a, float b) {
    return __uint_as_float(max(__float_as_uint(a), __float_as_uint(b)));
}

// The tree walk's point and dipole terms in two factors, t = x · inv, from
// d, r² = |d|² and s²: ρ² = max(r², s²), ρ = √ρ², ρ³ = ρ²·ρ (ROOT:
// ρ·ρ·ρ); the screened guard r > 1e-10 as r² > 1e-20
template <bool SCREENED, bool ROOT = false>
__device__ __forceinline__ float tree_term_split(float dx, float dy, float dz, float r2, float s2, const float4 b,
                                                 float sigma, float sigma_l2e, float& inv, bool& ok) {
    const float dot = __builtin_fmaf(dz, b.z, __builtin_fmaf(dy, b.y, dx * b.x));
    if constexpr (!SCREENED) {
        const float r = fast_sqrt(r2);
        inv = fast_rcp(__builtin_fmaf(r2, r, kEpsPlain * kInv4Pi));
        ok = true;
        return dot;
    } else {
        const float rho2 = max_nonneg(r2, s2);
        const float rho = fast_sqrt(rho2);
        const float rho3 = (ROOT ? rho * rho : rho2) * rho;
        inv = fast_rcp(__builtin_fmaf(fast_exp2(sigma_l2e * rho), rho3, kEpsScreened * kInv4Pi));
        ok = r2 > 1e-20f;
        return __builtin_fmaf(sigma, rho, 1.0f) * dot;
    }
}

// tree_term_split where r² is known to be above s² and the guard
template <bool SCREENED>
__device__ __forceinline__ float bare_term_split(float dx, float dy, float dz, const float4 b, float sigma,
                                                 float sigma_l2e, float& inv) {
    const float r2 = dist2(dx, dy, dz);
    const float dot = __builtin_fmaf(dz, b.z, __builtin_fmaf(dy, b.y, dx * b.x));
    const float r = fast_sqrt(r2);
    if constexpr (!SCREENED) {
        inv = fast_rcp(__builtin_fmaf(r2, r, kEpsPlain * kInv4Pi));
        return dot;
    } else {
        inv = fast_rcp(__builtin_fmaf(fast_exp2(sigma_l2e * r), r2 * r, kEpsScreened * kInv4Pi));
        return __builtin_fmaf(sigma, r, 1.0f) * dot;
    }
}

// part + x·inv with the product rounded first (no fusing), as the walk's
// selected sum rounds it: a term is the same by either path
__device__ __forceinline__ float add_rounded(float part, float x, float inv) {
#pragma clang fp contract(off)
    const float t = x * inv;
    return part + t;
}

// max(r², s²), and s² where r² is no number (an s² never is): the median with ∞,
// which is the least of the numbers among three.  (Of a constant ∞ the compiler makes
// a maximum, and one more instruction that quiets a signalling NaN of s².)
__device__ __forceinline__ float screened_r2(float r2, float s2) {
    float inf;
    asm("v_mov_b32 %0, 0x7f800000" : "=v"(inf));
    return __builtin_amdgcn_fmed3f(r2, s2, inf);
}

// The direct sums' point term as such factors, a = (p, ·), b = (A·n/4π, s²);
// 0 at the guard and where the distance is no number, by the factor x alone, as
// the other is always one.  With the product left to the sum's multiply-add it
// takes 21 instructions screened (24 with ρ = max(r, s), ρ·ρ·ρ and a selected sum:
// 10,000 sources at 2M queries 13.6 → 11.9 ms, the chip's whole issue rate).
// ROOT: ρ³ as ρ·ρ·ρ, one more, for compensated sums, whose error is the factors':
// the root's bias, which ρ²·ρ has once and e^{σρ}, 1 + σρ and ρ·ρ·ρ together, in
// part cancels the reciprocal's (RMS error of 200,000 sources 6.5e-8 → 5.5e-8,
// 292 → 322 µs at 2,000 queries; 10,000 at 2M 11.55 → 12.15 ms).
template <bool SCREENED, bool ROOT>
__device__ __forceinline__ float gwn_term_split(float qx, float qy, float qz, const float4 a, const float4 b,
                                                float sigma, float sigma_l2e, float& inv) {
    const float dx = a.x - qx, dy = a.y - qy, dz = a.z - qz;
    const float r2 = dist2(dx, dy, dz);
    bool ok;
    if constexpr (!SCREENED) return tree_term_split<false>(dx, dy, dz, r2, 0.f, b, sigma, sigma_l2e, inv, ok);
    const float x = tree_term_split<true, ROOT>(dx, dy, dz, screened_r2(r2, b.w), 0.f, b, sigma, sigma_l2e, inv, ok);
    return r2 > 1e-20f ? x : 0.f;
}

// DWG_NEAR_FP64: a screened point term inside its source's screening radius
// (r < s, so ρ = s) in FP64, from the float source a = (p, s), b = A·n/4π
// and query q; 0 unless r > 1e-10 (TurboLibiGWN.cu:544-585)
__device__ __forceinline__ double near_term64(const float4 a, const float4 b, float qx, float qy, float qz,
                                              float sigma) {
    const double dx = double(a.x) - double(qx), dy = double(a.y) - double(qy), dz = double(a.z) - double(qz);
    const double r2 = dx * dx + dy * dy + dz * dz;
    if (!(r2 > 1e-20)) return 0.0;
    const double rho = a.w, sg = sigma;
    const double dot = dx * double(b.x) + dy * double(b.y) + dz * double(b.z);
    const double den = exp(sg * rho) * (rho * rho * rho) + 1e-7 / (4.0 * 3.14159265358979323846);
    return (sg * rho + 1.0) * dot / den;
}

// the split of a screened point term between the FP32 sum and the FP64 one:
// near (r < s, r > 1e-10) goes to FP64
__device__ __forceinline__ bool near_field(float r2, float s) { return r2 < s * s && r2 > 1e-20f; }

// a term and its gradient w.r.t. q from the offset d = p − q (b pre-scaled
// by 1/4π, ε' = ε/4π):
//   plain     w = (d·b)/D, D = r³ + ε';  ∇w = −b/D + 3 r (d·b) d / D²
//   screened  w = g(ρ)(d·b), g = (1 + σρ)/D, D = e^{σρ}ρ³ + ε', ρ = max(r, s),
//             0 unless r > 1e-10;  ∇w = −g b − (d·b) g'(ρ) d / r for r ≥ s
//             (∂ρ/∂q = −d/r), −g b for r < s;
//             g' = (σε' − e^{σρ}ρ²(σ²ρ² + 3σρ + 3)) / D²  (no cancellation)
// as the factors dot = d·b, g and c of w = g·dot, ∇w = c·d − g·b, with s2 the
// squared screening radius (200,000 sources at 2,000 queries 540 → 501 µs with
// selects on two factors instead of four results.  Of that ρ·ρ takes 8, as ρ² in its
// place adds 8 % to the RMS error of ∇w, and ρ^-1 as the root's reciprocal 5 %;
// ρ = ρ²·ρ^-1 would save 5 % of the time for an error of w 8 to 13 % above the
// root's).  A component c·d − g·b is formed before it joins its sum: its two products
// joined one by one, 6 % faster, round twice at the sum's size (half of 2,000
// queries next to one of 20,000 sources: RMS error of ∇w 11 % and maximum 37 % more).
// A screened term at the guard, or whose distance is no number, has only zeros
// (d may still be no number).
template <bool SCREENED>
__device__ __forceinline__ void gwn_term_grad(float dx, float dy, float dz, float s2, const float4 b, float sigma,
                                              float sigma_l2e, float& dot, float& g, float& c) {
    const float r2 = dist2(dx, dy, dz);
    dot = __builtin_fmaf(dz, b.z, __builtin_fmaf(dy, b.y, dx * b.x));
    if constexpr (!SCREENED) {
        const float r = fast_sqrt(r2);
        g = fast_rcp(__builtin_fmaf(r2, r, kEpsPlain * kInv4Pi));
        c = 3.0f * r * (dot * g) * g;
    } else {
        const bool ok = r2 > 1e-20f;
        dot = ok ? dot : 0.0f;
        const float rho2 = screened_r2(r2, s2);
        const float rho = fast_sqrt(rho2), irho = fast_rsq(rho2);
        const float er2 = fast_exp2(sigma_l2e * rho) * (rho * rho);
        const float eps = kEpsScreened * kInv4Pi;
        const float inv = fast_rcp(__builtin_fmaf(er2, rho, eps));
        const float sr = sigma * rho;
        g = ok ? __builtin_fmaf(sigma, rho, 1.0f) * inv : 0.0f;
        const float gp = __builtin_fmaf(er2, __builtin_fmaf(sr, sr + 3.0f, 3.0f), -(sigma * eps));  // −g' D²
        // inside (ρ = s) nothing depends on q through ρ
        c = ok && !(s2 > r2) ? (dot * irho) * (gp * inv) * inv : 0.0f;
    }
}

// a component c·d − g·b of the gradient, of whose products one is rounded before
// they meet.  Plain: the smaller, g·b (c·d next to a source is up to three times
// as large).  Screened: c·d, as 0 · d is 0 by this multiplication, also for a d
// that is no number (plain terms have no zeros to keep, and the compiler unrolls
// a loop with the instruction written out less)
template <bool SCREENED>
__device__ __forceinline__ float grad_component(float c, float d, float g, float b) {
    if constexpr (!SCREENED) return __builtin_fmaf(c, d, -(g * b));
    float cd;
    asm("v_mul_legacy_f32 %0, %1, %2" : "=v"(cd) : "v"(c), "v"(d));
    return __builtin_fmaf(-g, b, cd);
}

// ---------------------------------------------------------------------------
// source packing: (x, y, z, s) and (A·n/4π, s²)
// ---------------------------------------------------------------------------
// the screening radius of every sum: 0 for s ≤ 0 or NaN (ρ = max(s, r) = r), and a
// finite one kept to where its square is finite
__device__ __forceinline__ float screening_radius(float s) {
    return s > 0.f ? (s < INFINITY ? fminf(s, 1.84467429e19f) : s) : 0.f;
}

__global__ void pack_sources_kernel(const float* __restrict__ pts, const float* __restrict__ nrm,
                                    const float* __restrict__ area, const float* __restrict__ radii,
                                    const int* __restrict__ perm, int64_t n, int use_radii,
                                    float4* __restrict__ sa, float4* __restrict__ sb,
                                    Double3* __restrict__ an64) {
    int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t p = perm ? perm[i] : i;
    const float A = area ? area[p] : 2e-6f;
    const float s = use_radii ? screening_radius(radii[p]) : kScreenDefault;
    if (sa) sa[i] = make_float4(pts[3 * p], pts[3 * p + 1], pts[3 * p + 2], s);
    const float nx = nrm[3 * p], ny = nrm[3 * p + 1], nz = nrm[3 * p + 2];
    sb[i] = make_float4(A * nx * kInv4Pi, A * ny * kInv4Pi, A * nz * kInv4Pi, s * s);
    if (an64) an64[i] = Double3(double(A) * nx, double(A) * ny, double(A) * nz);
}

// ---------------------------------------------------------------------------
// direct all-pairs kernel
// ---------------------------------------------------------------------------
constexpr int kDirectThreads = 256;
constexpr int kDirectTile = 64;

// the sources [j0, j1) summed at q: the FP32 sum is sum − comp, and near the
// FP64 sum of the terms inside the screening radius (DWG_NEAR_FP64)
template <bool SCREENED, bool KAHAN, bool NEAR64>
__device__ __forceinline__ void direct_value(const float4* __restrict__ sa, const float4* __restrict__ sb, int64_t j0,
                                             int64_t j1, float qx, float qy, float qz, float sigma, float& sum,
                                             float& comp, double& near) {
    const float sl2e = sigma * kLog2e;
    sum = comp = 0.f;
    near = 0.0;
    auto add = [&](float& part, const float4 a, const float4 b) {
        float inv;
        float x = gwn_term_split<SCREENED, KAHAN>(qx, qy, qz, a, b, sigma, sl2e, inv);
        if constexpr (NEAR64) {
            const float dx = a.x - qx, dy = a.y - qy, dz = a.z - qz;
            const bool nr = near_field(dist2(dx, dy, dz), a.w);
            if (__builtin_amdgcn_ballot_w64(nr)) {
                if (nr) near += near_term64(a, b, qx, qy, qz, sigma);
            }
            x = nr ? 0.f : x;
        }
        part = __builtin_fmaf(x, inv, part);
    };
    for (; j0 + kDirectTile <= j1; j0 += kDirectTile) {
        float part = 0.f;
#pragma unroll 8
        for (int j = 0; j < kDirectTile; ++j) add(part, sa[j0 + j], sb[j0 + j]);
        if (KAHAN) kahan_add(sum, comp, part); else sum += part;
    }
    float part = 0.f;
    for (int64_t j = j0; j < j1; ++j) add(part, sa[j], sb[j]);
    if (KAHAN) kahan_add(sum, comp, part); else sum += part;
}

// the sources [j0, j1) summed at q, value and gradient: s − c for each.  UNROLL
// terms of a tile at a time: 2, and 1 for plain sums that are not split (857 sources at
// 1M queries, plain: 489 µs by 1, 518 by 2, 528 by 4; 3,000 at 300,000 671, 667 and
// 641, screened 1,073, 1,030 and 1,111; 200,000 at 2,000, split, 342, 318 and 333,
// screened, with a multiplication less, 499, 490 and 520)
template <bool SCREENED, bool KAHAN, int UNROLL>
__device__ __forceinline__ void direct_grad(const float4* __restrict__ sa, const float4* __restrict__ sb, int64_t j0,
                                            int64_t j1, float qx, float qy, float qz, float sigma, float (&s)[4],
                                            float (&c)[4]) {
    const float sl2e = sigma * kLog2e;
#pragma unroll
    for (int k = 0; k < 4; ++k) s[k] = c[k] = 0.f;
    float p[4];
    auto term = [&](const float4 a, const float4 b) {
        const float dx = a.x - qx, dy = a.y - qy, dz = a.z - qz;
        float dot, g, c;
        gwn_term_grad<SCREENED>(dx, dy, dz, b.w, b, sigma, sl2e, dot, g, c);
        p[0] = __builtin_fmaf(g, dot, p[0]);
        p[1] += grad_component<SCREENED>(c, dx, g, b.x);
        p[2] += grad_component<SCREENED>(c, dy, g, b.y);
        p[3] += grad_component<SCREENED>(c, dz, g, b.z);
    };
    auto fold = [&]() {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (KAHAN) kahan_add(s[k], c[k], p[k]); else s[k] += p[k];
            p[k] = 0.f;
        }
    };
#pragma unroll
    for (int k = 0; k < 4; ++k) p[k] = 0.f;
    for (; j0 + kDirectTile <= j1; j0 += kDirectTile) {
#pragma unroll UNROLL
        for (int j = 0; j < kDirectTile; ++j) term(sa[j0 + j], sb[j0 + j]);
        fold();
    }
    if (j0 < j1) {
        for (int64_t j = j0; j < j1; ++j) term(sa[j], sb[j]);
        fold();
    }
}

template <bool SCREENED, bool KAHAN, bool NEAR64 = false>
__global__ __launch_bounds__(kDirectThreads) void gwn_direct_kernel(
    const float4* __restrict__ sa, const float4* __restrict__ sb, int64_t n, const float* __restrict__ q,
    int64_t nq, float sigma, float* __restrict__ out) {
    const int64_t i = int64_t(blockIdx.x) * kDirectThreads + threadIdx.x;
    const bool valid = i < nq;
    const float qx = valid ? q[3 * i] : 0.f, qy = valid ? q[3 * i + 1] : 0.f, qz = valid ? q[3 * i + 2] : 0.f;
    float sum, comp;
    double near;
    direct_value<SCREENED, KAHAN, NEAR64>(sa, sb, 0, n, qx, qy, qz, sigma, sum, comp, near);
    if (valid) out[i] = NEAR64 ? float(double(sum - comp) + near) : sum - comp;
}

template <bool SCREENED, bool KAHAN>
__global__ __launch_bounds__(kDirectThreads) void gwn_direct_grad_kernel(
    const float4* __restrict__ sa, const float4* __restrict__ sb, int64_t n, const float* __restrict__ q,
    int64_t nq, float sigma, float* __restrict__ out_w, float* __restrict__ out_g) {
    const int64_t i = int64_t(blockIdx.x) * kDirectThreads + threadIdx.x;
    const bool valid = i < nq;
    const float qx = valid ? q[3 * i] : 0.f, qy = valid ? q[3 * i + 1] : 0.f, qz = valid ? q[3 * i + 2] : 0.f;
    float s[4], c[4];
    direct_grad<SCREENED, KAHAN, SCREENED ? 2 : 1>(sa, sb, 0, n, qx, qy, qz, sigma, s, c);
    if (valid) {
        out_w[i] = s[0] - c[0];
        out_g[3 * i] = s[1] - c[1];
        out_g[3 * i + 1] = s[2] - c[2];
        out_g[3 * i + 2] = s[3] - c[3];
    }
}

// Few queries over many sources leave most of the chip idle (2,000 queries
// are 32 waves for 1,024 SIMDs), so the sources are split: one wave takes 64
// queries (blockIdx.x) and one run of sources (blockIdx.y) and writes its
// sums in FP64 (the Kahan pair and the FP64 near field without a rounding),
// direct_fold_kernel adds the runs in FP64 in a fixed order and rounds once:
// no less exact than one chain.  VALU-bound like the unsplit kernels once
// every SIMD has a few waves.
template <bool SCREENED, bool KAHAN, bool NEAR64>
__global__ __launch_bounds__(64) void gwn_direct_split_kernel(const float4* __restrict__ sa,
                                                              const float4* __restrict__ sb, int64_t n, int64_t run,
                                                              const float* __restrict__ q, int64_t nq, float sigma,
                                                              double* __restrict__ part) {
    const int64_t i = int64_t(blockIdx.x) * 64 + threadIdx.x;
    const bool valid = i < nq;
    const float qx = valid ? q[3 * i] : 0.f, qy = valid ? q[3 * i + 1] : 0.f, qz = valid ? q[3 * i + 2] : 0.f;
    const int64_t j0 = int64_t(blockIdx.y) * run, j1 = j0 + run < n ? j0 + run : n;
    float sum, comp;
    double near;
    direct_value<SCREENED, KAHAN, NEAR64>(sa, sb, j0, j1, qx, qy, qz, sigma, sum, comp, near);
    if (valid) part[int64_t(blockIdx.y) * nq + i] = (double(sum) - double(comp)) + near;
}

template <bool SCREENED, bool KAHAN>
__global__ __launch_bounds__(64) void gwn_direct_grad_split_kernel(const float4* __restrict__ sa,
                                                                   const float4* __restrict__ sb, int64_t n,
                                                                   int64_t run, const float* __restrict__ q,
                                                                   int64_t nq, float sigma,
                                                                   double* __restrict__ part) {
    const int64_t i = int64_t(blockIdx.x) * 64 + threadIdx.x;
    const bool valid = i < nq;
    const float qx = valid ? q[3 * i] : 0.f, qy = valid ? q[3 * i + 1] : 0.f, qz = valid ? q[3 * i + 2] : 0.f;
    const int64_t j0 = int64_t(blockIdx.y) * run, j1 = j0 + run < n ? j0 + run : n;
    float s[4], c[4];
    direct_grad<SCREENED, KAHAN, 2>(sa, sb, j0, j1, qx, qy, qz, sigma, s, c);
    if (valid) {
        double* o = part + int64_t(blockIdx.y) * 4 * nq;
#pragma unroll
        for (int k = 0; k < 4; ++k) o[k * nq + i] = double(s[k]) - double(c[k]);
    }
}

// out = Σ over the splits of part[split][value]: kFoldValues values and
// kFoldRows rows of splits a block, the rows added in order.  Values
// [0, nq) are w, then ∇w by component (nv = 4·nq with a gradient)
constexpr int kFoldValues = 32, kFoldRows = 8;
__global__ __launch_bounds__(kFoldValues * kFoldRows) void direct_fold_kernel(const double* __restrict__ part,
                                                                              int splits, int64_t nq, int64_t nv,
                                                                              float* __restrict__ out_w,
                                                                              float* __restrict__ out_g) {
    __shared__ double lds[kFoldRows][kFoldValues];
    const int c = threadIdx.x % kFoldValues, r = threadIdx.x / kFoldValues;
    const int64_t v = int64_t(blockIdx.x) * kFoldValues + c;
    double s = 0;
    if (v < nv)
        for (int k = r; k < splits; k += kFoldRows) s += part[int64_t(k) * nv + v];
    lds[r][c] = s;
    __syncthreads();
    if (r != 0 || v >= nv) return;
#pragma unroll
    for (int k = 1; k < kFoldRows; ++k) s += lds[k][c];
    if (v < nq) out_w[v] = float(s);
    else out_g[3 * (v % nq) + (v / nq - 1)] = float(s);
}

static void check_direct_args(int64_t n, int64_t nq, const float* radii, uint32_t flags, const float*) {
    DWG_REQUIRE(n >= 0 && nq >= 0, "negative size");
    DWG_REQUIRE(!(flags & DWG_USE_RADII) || radii, "DWG_USE_RADII needs radii");
}

// The source runs a direct sum of nq queries over n sources is split into.
// One wave takes 64 queries; below kDirectWaves waves the chip's 1,024 SIMDs
// hold too few to hide their latencies, and the sources are split until there
// are that many.  A run has at least kDirectMinRun sources, under which the
// second launch costs more than the split saves, and the partial sums fit in
// kDirectPartials doubles.  Depends on the sizes only, so both entry points
// sum alike.
constexpr int64_t kDirectWaves = 4096, kDirectMinRun = 2 * kDirectTile, kDirectMaxSplits = 1024;
constexpr int64_t kDirectPartials = int64_t(1) << 20;

static int64_t direct_splits(int64_t n, int64_t nq, int values) {
    const int64_t waves = (nq + 63) / 64;
    int64_t s = std::min({kDirectWaves / waves, n / kDirectMinRun, kDirectMaxSplits, kDirectPartials / (values * nq)});
    if (s < 2) return 1;
    const int64_t run = ((n + s - 1) / s + kDirectTile - 1) / kDirectTile * kDirectTile;  // whole tiles
    return (n + run - 1) / run;
}

// packs the n sources into sa/sb (room for n + 1 each) and runs the direct
// kernel; `part`: room for kDirectPartials doubles when the sums are split;
// `profile` off records no events (the allocation-free entry point)
static void direct_sums(dwg_ctx* ctx, float4* sa, float4* sb, double* part, const float* pts, const float* nrm,
                        const float* area, const float* radii, int64_t n, const float* q, int64_t nq, float sigma,
                        uint32_t flags, float* out_w, float* out_g, bool profile) {
    if (n > 0) {
        ProfileScope ps(profile ? ctx : nullptr, "pack_sources");
        hipLaunchKernelGGL(pack_sources_kernel, dim3(grid_for(n, 256)), dim3(256), 0, ctx->stream, pts, nrm, area,
                           radii, nullptr, n, (flags & DWG_USE_RADII) ? 1 : 0, sa, sb, nullptr);
        check_launch();
    }
    const bool kahan = flags & DWG_KAHAN, scr = flags & DWG_SCREENED, near64 = scr && (flags & DWG_NEAR_FP64) && !out_g;
    ProfileScope ps(profile ? ctx : nullptr,
                    out_g ? "gwn_direct_grad" : (scr ? "gwn_direct_screened" : "gwn_direct_plain"));
    const int values = out_g ? 4 : 1;
    const int64_t splits = direct_splits(n, nq, values);
    // LAUNCH(screened, kahan) over the two flags
#define DWG_DIRECT_BY_FLAGS(LAUNCH)         \
    do {                                    \
        if (scr && kahan) LAUNCH(true, true);    \
        else if (scr) LAUNCH(true, false);       \
        else if (kahan) LAUNCH(false, true);     \
        else LAUNCH(false, false);               \
    } while (0)
    if (splits > 1) {
        const int64_t run = ((n + splits - 1) / splits + kDirectTile - 1) / kDirectTile * kDirectTile;
        dim3 grid(grid_for(nq, 64), unsigned(splits)), block(64);
#define DWG_SPLIT_GRAD(S, K) \
    hipLaunchKernelGGL((gwn_direct_grad_split_kernel<S, K>), grid, block, 0, ctx->stream, sa, sb, n, run, q, nq, sigma, part)
#define DWG_SPLIT_VALUE(S, K) \
    hipLaunchKernelGGL((gwn_direct_split_kernel<S, K, false>), grid, block, 0, ctx->stream, sa, sb, n, run, q, nq, sigma, part)
#define DWG_SPLIT_NEAR(S, K) \
    hipLaunchKernelGGL((gwn_direct_split_kernel<true, K, true>), grid, block, 0, ctx->stream, sa, sb, n, run, q, nq, sigma, part)
        if (out_g) DWG_DIRECT_BY_FLAGS(DWG_SPLIT_GRAD);
        else if (near64) DWG_DIRECT_BY_FLAGS(DWG_SPLIT_NEAR);
        else DWG_DIRECT_BY_FLAGS(DWG_SPLIT_VALUE);
#undef DWG_SPLIT_GRAD
#undef DWG_SPLIT_VALUE
#undef DWG_SPLIT_NEAR
        check_launch();
        hipLaunchKernelGGL(direct_fold_kernel, dim3(grid_for(values * nq, kFoldValues)), dim3(kFoldValues * kFoldRows),
                           0, ctx->stream, part, int(splits), nq, values * nq, out_w, out_g);
        check_launch();
        return;
    }
    dim3 grid(grid_for(nq, kDirectThreads)), block(kDirectThreads);
#define DWG_DIRECT_GRAD(S, K) \
    hipLaunchKernelGGL((gwn_direct_grad_kernel<S, K>), grid, block, 0, ctx->stream, sa, sb, n, q, nq, sigma, out_w, out_g)
#define DWG_DIRECT_VALUE(S, K) \
    hipLaunchKernelGGL((gwn_direct_kernel<S, K>), grid, block, 0, ctx->stream, sa, sb, n, q, nq, sigma, out_w)
#define DWG_DIRECT_NEAR(S, K) \
    hipLaunchKernelGGL((gwn_direct_kernel<true, K, true>), grid, block, 0, ctx->stream, sa, sb, n, q, nq, sigma, out_w)
    if (out_g) DWG_DIRECT_BY_FLAGS(DWG_DIRECT_GRAD);
    else if (near64) DWG_DIRECT_BY_FLAGS(DWG_DIRECT_NEAR);
    else DWG_DIRECT_BY_FLAGS(DWG_DIRECT_VALUE);
#undef DWG_DIRECT_GRAD
#undef DWG_DIRECT_VALUE
#undef DWG_DIRECT_NEAR
#undef DWG_DIRECT_BY_FLAGS
    check_launch();
}

void gwn_direct(dwg_ctx* ctx, const float* pts, const float* nrm, const float* area, const float* radii, int64_t n,
                const float* q, int64_t nq, float sigma, uint32_t flags, float* out_w, float* out_g) {
    check_direct_args(n, nq, radii, flags, out_g);
    if (nq == 0) return;
    // one array: the partial sums (also where this call does not split: one of the
    // same sources that does may be recorded into a graph next, and can allocate
    // nothing), then the packed sources, each from a line of its own on (the scalar
    // loads' lines: 200,000 sources at 2,000 queries 8 % slower where they straddle)
    const size_t parts = sizeof(double) * kDirectPartials, packed = (sizeof(float4) * size_t(n + 1) + 255) & ~size_t(255);
    char* mem = static_cast<char*>(ctx->buf("direct", parts + 2 * packed));
    double* part = reinterpret_cast<double*>(mem);
    float4 *sa = reinterpret_cast<float4*>(mem + parts), *sb = reinterpret_cast<float4*>(mem + parts + packed);
    direct_sums(ctx, sa, sb, part, pts, nrm, area, radii, n, q, nq, sigma, flags, out_w, out_g, true);
}

// ---------------------------------------------------------------------------
// allocation-free direct sums: the packed sources live in a fixed device
// array instead of the context's growable buffers
// ---------------------------------------------------------------------------
// sa of source i at scratch[i], sb at scratch[kNoAllocSources + 1 + i], then
// the partial sums of a split call (8 + 8 MiB on every device the library
// runs on, held until the process ends)
static __device__ __align__(256) float4 scratch[2 * (kNoAllocSources + 1) + kDirectPartials * sizeof(double) / sizeof(float4)];

namespace {
std::mutex g_scratch_mu;
std::vector<float4*> g_scratch_ptr;  // device address of `scratch` per device ordinal
}  // namespace

void noalloc_init(int device) {
    // the symbol's address differs per device: look it up with that device
    // current, once, and keep it (host code never uses the symbol itself)
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (device < 0) throw Error(DWG_ERR_ARG, "bad device ordinal");
    if (size_t(device) < g_scratch_ptr.size() && g_scratch_ptr[size_t(device)]) return;
    int cur = -1;
    DWG_HIP_CHECK(hipGetDevice(&cur));
    DWG_REQUIRE(cur == device, "noalloc_init: the device must be current");
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
        throw Error(DWG_ERR_HIP, std::string("hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(e));
    if (g_scratch_ptr.size() <= size_t(device)) g_scratch_ptr.resize(size_t(device) + 1, nullptr);
    g_scratch_ptr[size_t(device)] = static_cast<float4*>(p);
}

void gwn_direct_noalloc(dwg_ctx* ctx, const float* pts, const float* nrm, const float* area, const float* radii,
                        int64_t n, const float* q, int64_t nq, float sigma, uint32_t flags, float* out_w,
                        float* out_g) {
    check_direct_args(n, nq, radii, flags, out_g);
    if (n > kNoAllocSources)
        throw Error(DWG_ERR_ARG, "dwg_gwn_direct_noalloc: " + std::to_string(n) + " sources exceed its limit of " +
                                     std::to_string(kNoAllocSources) + " (use dwg_gwn_direct)");
    if (nq == 0) return;
    float4* base = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_scratch_mu);
        if (size_t(ctx->device) < g_scratch_ptr.size()) base = g_scratch_ptr[size_t(ctx->device)];
    }
    if (!base) throw Error(DWG_ERR_STATE, "allocation-free scratch of this device was not set up");
    direct_sums(ctx, base, base + (kNoAllocSources + 1), reinterpret_cast<double*>(base + 2 * (kNoAllocSources + 1)), pts, nrm, area, radii, n, q, nq, sigma, flags, out_w, out_g,
                false);
}

}  // namespace dwg

// ---------------------------------------------------------------------------
// device octree
// ---------------------------------------------------------------------------
dwg_octree::~dwg_octree() {
    for (void* p : {(void*)info, (void*)kid, (void*)cm_r, (void*)cm_lo, (void*)ec, (void*)sa, (void*)sb, (void*)perm,
                    (void*)an64, (void*)cell, (void*)cm64, (void*)payload, (void*)radius})
        dwg::dev_free(p);
}

namespace dwg {

// A leaf with one point is walked like a far dipole: its traversal record
// holds the point (x, y, z), its payload the point's (A·n/4π, s²) and a zero
// residual, so the walk reads the same words for both and evaluates the
// same term, ρ² = max(r², s²) (an internal node's s² is the default
// screening radius's)
constexpr float kDipoleS2 = kScreenDefault * kScreenDefault;

__device__ __forceinline__ void write_point_leaf(int64_t i, const float4 a, const float4 b, float4* __restrict__ cm_r,
                                                 float4* __restrict__ payload) {
    payload[2 * i] = make_float4(b.x, b.y, b.z, a.w * a.w);
    payload[2 * i + 1] = make_float4(0.f, 0.f, 0.f, bare_floor(a.w * a.w, 0.f));
    cm_r[i].x = a.x;
    cm_r[i].y = a.y;
    cm_r[i].z = a.z;
}

// EC/4π per node (FP64 prefix-sum difference, one rounding), into ec and the node
// payload: words 0-3 of an internal node (EC/4π, s²); a leaf with one point carries
// that point's term instead (write_point_leaf)
__global__ void node_ec_kernel(const int4* __restrict__ info, const Double3* __restrict__ scan, int64_t m,
                               const float4* __restrict__ sa, const float4* __restrict__ sb,
                               float4* __restrict__ ec, float4* __restrict__ payload, float4* __restrict__ cm_r) {
    int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= m) return;
    const int4 nf = info[i];
    const Double3 s = scan[nf.z] - scan[nf.y];
    const float x = float(s.x * double(kInv4Pi)), y = float(s.y * double(kInv4Pi)), z = float(s.z * double(kInv4Pi));
    ec[i] = make_float4(x, y, z, 0.f);
    if (nf.x >= 0) {
        payload[2 * i] = make_float4(x, y, z, kDipoleS2);
    } else if (nf.z - nf.y == 1) {
        write_point_leaf(i, sa[nf.y], sb[nf.y], cm_r, payload);
    }
}

// the sources in tree order for new normals, areas and radii; their positions
// are there
__global__ void repack_sources_kernel(const float* __restrict__ nrm, const float* __restrict__ area,
                                      const float* __restrict__ radii, const int* __restrict__ perm, int64_t n,
                                      float4* __restrict__ sa, float4* __restrict__ sb, Double3* __restrict__ an64) {
    int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t p = perm[i];
    const float A = area ? area[p] : 2e-6f;
    sa[i].w = radii ? screening_radius(radii[p]) : kScreenDefault;
    const float nx = nrm[3 * p], ny = nrm[3 * p + 1], nz = nrm[3 * p + 2];
    sb[i] = make_float4(A * nx * kInv4Pi, A * ny * kInv4Pi, A * nz * kInv4Pi, 0.f);
    an64[i] = Double3(double(A) * nx, double(A) * ny, double(A) * nz);
}

void octree_update(dwg_ctx* ctx, dwg_octree* T, const float* nrm, const float* area, const float* radii) {
    const int64_t n = T->n_points, m = T->n_nodes;
    {
        ProfileScope ps(ctx, "octree_pack");
        hipLaunchKernelGGL(repack_sources_kernel, dim3(grid_for(n, 256)), dim3(256), 0, ctx->stream, nrm, area, radii,
                           T->perm, n, T->sa, T->sb, T->an64);
        check_launch();
    }
    {
        ProfileScope ps(ctx, "octree_ec_scan");
        exclusive_scan<Double3>(ctx, T->an64, n);
    }
    ProfileScope ps(ctx, "octree_ec");
    hipLaunchKernelGGL(node_ec_kernel, dim3(grid_for(m, 256)), dim3(256), 0, ctx->stream, T->info, T->an64, m, T->sa,
                       T->sb, T->ec, T->payload, T->cm_r);
    check_launch();
    T->payload_bf16 = false;
    T->updated = true;
}

// the point terms of one-point leaves live in their payload too
__global__ void leaf_payload_kernel(const int4* __restrict__ info, int64_t m, const float4* __restrict__ sa,
                                    const float4* __restrict__ sb, float4* __restrict__ payload,
                                    float4* __restrict__ cm_r) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= m) return;
    const int4 nf = info[i];
    if (nf.x < 0 && nf.z - nf.y == 1) write_point_leaf(i, sa[nf.y], sb[nf.y], cm_r, payload);
}

void octree_set_point_areas(dwg_ctx* ctx, dwg_octree* T, const float* nrm, const float* area) {
    DWG_REQUIRE(T->updated, "octree has no moments yet: call dwg_octree_update first");
    const int64_t n = T->n_points, m = T->n_nodes;
    ProfileScope ps(ctx, "octree_pack");
    hipLaunchKernelGGL(pack_sources_kernel, dim3(grid_for(n, 256)), dim3(256), 0, ctx->stream, nullptr, nrm, area,
                       nullptr, T->perm, n, 0, nullptr, T->sb, nullptr);
    check_launch();
    hipLaunchKernelGGL(leaf_payload_kernel, dim3(grid_for(m, 256)), dim3(256), 0, ctx->stream, T->info, m, T->sa,
                       T->sb, T->payload, T->cm_r);
    check_launch();
}

// ---------------------------------------------------------------------------
// Barnes-Hut traversal, one wave per brick of grid points (kGridParts per
// lane) or per 64 explicit queries
// ---------------------------------------------------------------------------
constexpr int kTreeThreads = 64;
constexpr int kTreeWaves = kTreeThreads / 64;
constexpr int kMaxTreeLevel = 21;
// stack entries a walk of a tree of max_level levels needs at most: 7 left
// over per level and the 8 children of the deepest node opened
__host__ __device__ constexpr int tree_stack_entries(int max_level) { return 7 * max_level + 8; }
constexpr int kStack = tree_stack_entries(kMaxTreeLevel);  // the shared gradient walk's fixed stack
// grid walks: each lane evaluates kGridParts points, one in each 4×4×4 part
// of a brick of kPartsX × kPartsY × kPartsZ parts (parts that differ in z
// share a child's x and y products)
constexpr int kPartsX = 2, kPartsY = 1, kPartsZ = 2;
constexpr int kGridParts = kPartsX * kPartsY * kPartsZ;
// the kernels' GRID of bricks of 2 × 2 × 1 parts, for grids of at most 4 points
// along z, which would leave half of the others empty (over 3,000 sources 500×500×1
// 94 → 69 µs, 2,000×2,000×1 1,033 → 559)
constexpr int kFlatParts = kGridParts + 1;
constexpr int kPointPts = 1;  // explicit queries per lane

struct TreeArgs {
    const int4* __restrict__ info;
    const int2* __restrict__ kid;
    const float4* __restrict__ cm_r;
    const float* __restrict__ payload;  // 8 words per node (see dwg_octree::payload)
    const float4* __restrict__ sa;
    const float4* __restrict__ sb;
};

// Wave-uniform reads of node records go through the scalar data cache: a
// pointer into the constant address space makes each such load an s_load
// (one copy into SGPRs).  Through a generic pointer the compiler emits a
// vector load, which returns 64 copies of the same bytes through the
// vector memory path.
typedef int NativeInt2 __attribute__((ext_vector_type(2)));
typedef float NativeFloat4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int2 scalar_load(const int2* p, int64_t i) {
    const NativeInt2 v = ((const __attribute__((address_space(4))) NativeInt2*)p)[i];
    return make_int2(v.x, v.y);
}

typedef int NativeInt4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ int4 scalar_load(const int4* p, int64_t i) {
    const NativeInt4 v = ((const __attribute__((address_space(4))) NativeInt4*)p)[i];
    return make_int4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ float4 scalar_load(const float4* p, int64_t i) {
    const NativeFloat4 v = ((const __attribute__((address_space(4))) NativeFloat4*)p)[i];
    return make_float4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ float bf16_round(float f) {
    uint32_t u = __float_as_uint(f);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return __uint_as_float(u & 0xFFFF0000u);
}

// The order in which explicit queries share walks: order[slot] where the
// sampled extent of their runs (query_order) is over `limit`, else the
// caller's own
struct QueryOrder {
    const int* order;
    const unsigned int* extent;  // nullptr: the caller's order
    unsigned int limit;
    __device__ __forceinline__ bool sorted() const { return extent && *extent > limit; }
    __device__ __forceinline__ int64_t query(int64_t slot) const { return sorted() ? int64_t(order[slot]) : slot; }
};

struct QueryArgs {
    const float* q;          // explicit points
    QueryOrder order;        // and their order
    const int* self_perm;    // the tree's own points in tree order, results to out[perm[slot]]
    bool grid;               // implicit grid (q and self_perm unused)
    int64_t nq;
    float ox, oy, oz, h;
    int rx, ry, rz;
    int parts;       // 4×4×4 parts of a brick (grid walks): kGridParts or 1
    bool flat;       // the kGridParts parts are kFlatParts' (grid walks)
    int bx, by, bz;  // bricks per axis
    int64_t n_bricks;
    int stack;  // walk stack entries (tree_stack_entries of the tree's depth)
};


template <bool SCREENED, bool COUNT, bool BF16, int GRID, bool NEAR64 = false>
__global__ __launch_bounds__(kTreeThreads) void gwn_tree_kernel(TreeArgs T, QueryArgs Q, float beta, float sigma,
                                                                 uint32_t flags, float* __restrict__ out,
                                                                 int64_t* __restrict__ terms_out) {
    // grid walks: each lane evaluates kGridParts points (one per 4×4×4 part
    // of the brick), so that a pop, its loads and its pushes serve them all
    constexpr int H = GRID == kFlatParts ? kGridParts : GRID ? GRID : kPointPts;
    constexpr int PX = GRID >= kGridParts ? kPartsX : 1,
                  PY = GRID == kFlatParts ? kPartsZ : GRID == kGridParts ? kPartsY : 1,
                  PZ = GRID == kGridParts ? kPartsZ : 1;
    static_assert(kTreeWaves == 1, "one wave per block: the stack lives in the block's dynamic LDS");
    // the stack: Q.stack entries of (record, H lane masks), in dynamic LDS
    // sized by the tree's depth (a shallow tree leaves room for more blocks)
    extern __shared__ uint64_t s_dyn[];
    int2* s_node_w = reinterpret_cast<int2*>(s_dyn);
    uint64_t* s_mask_w = s_dyn + Q.stack;
    __shared__ float4 s_pay[kTreeWaves][16];  // the 8 children's payloads of the node being opened
    __shared__ float4 s_cmr[kTreeWaves][16];  // and their (CM, w) records (twice)
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t blk = xcd_block(blockIdx.x, gridDim.x);
    const int64_t wid = blk * kTreeWaves + wave;
    int64_t qi[H];
    bool valid[H];
    float qx[H], qy[H], qz[H];
    int bxi = 0, byi = 0, bzi = 0;  // the wave's brick (grid walks)
    if (!GRID) {
        // H consecutive runs of 64 queries
#pragma unroll
        for (int h = 0; h < H; ++h) {
            qi[h] = (wid * H + h) * 64 + lane;
            valid[h] = qi[h] < Q.nq;
            if (Q.self_perm) {  // consecutive tree slots: spatially coherent waves
                const float4 a = valid[h] ? T.sa[qi[h]] : make_float4(0.f, 0.f, 0.f, 0.f);
                qx[h] = a.x;
                qy[h] = a.y;
                qz[h] = a.z;
                qi[h] = valid[h] ? int64_t(Q.self_perm[qi[h]]) : 0;
            } else {
                if (valid[h]) qi[h] = Q.order.query(qi[h]);
                qx[h] = valid[h] ? Q.q[3 * qi[h]] : 0.f;
                qy[h] = valid[h] ? Q.q[3 * qi[h] + 1] : 0.f;
                qz[h] = valid[h] ? Q.q[3 * qi[h] + 2] : 0.f;
            }
        }
    } else {
        // brick of kPartsX × kPartsY × kPartsZ parts of 4 × 4 × 4 points
        const int64_t br = wid;
        bxi = int(br % Q.bx);
        byi = int((br / Q.bx) % Q.by);
        bzi = int(br / (int64_t(Q.bx) * Q.by));
#pragma unroll
        for (int h = 0; h < H; ++h) {
            const int x = (bxi * PX + h % PX) * 4 + (lane & 3);
            const int y = (byi * PY + (h / PX) % PY) * 4 + ((lane >> 2) & 3);
            const int z = (bzi * PZ + h / (PX * PY)) * 4 + (lane >> 4);
            valid[h] = br < Q.n_bricks && x < Q.rx && y < Q.ry && z < Q.rz;
            qi[h] = int64_t(x) + int64_t(Q.rx) * (int64_t(y) + int64_t(Q.ry) * z);
            qx[h] = __builtin_fmaf(float(x), Q.h, Q.ox);
            qy[h] = __builtin_fmaf(float(y), Q.h, Q.oy);
            qz[h] = __builtin_fmaf(float(z), Q.h, Q.oz);
        }
    }
    uint64_t all[H];
    bool any = false, every = true;  // every: each part has points
#pragma unroll
    for (int h = 0; h < H; ++h) {
        all[h] = __builtin_amdgcn_ballot_w64(valid[h]);
        any = any || all[h] != 0;
        every = every && all[h] != 0;
    }
    if (!any) return;
    const float sl2e = sigma * kLog2e;
    float sum[H], comp[H];
    int64_t nterms[H];
    double near[H];  // DWG_NEAR_FP64: point terms inside the screening radius, in FP64
#pragma unroll
    for (int h = 0; h < H; ++h) {
        sum[h] = comp[h] = 0.f;
        nterms[h] = 0;
        near[h] = 0.0;
    }
    const bool kahan = flags & DWG_KAHAN;

    auto point_term = [&](const float4 a, const float4 b, bool on, float part, int h) {
        const float dx = a.x - qx[h], dy = a.y - qy[h], dz = a.z - qz[h];
        const float r2 = dist2(dx, dy, dz);
        if constexpr (NEAR64) {
            const bool nr = on && near_field(r2, a.w);
            if (__builtin_amdgcn_ballot_w64(nr)) {  // rare: lanes next to a source
                if (nr) near[h] += near_term64(a, b, qx[h], qy[h], qz[h], sigma);
            }
            on = on && !nr;
        }
        float inv;
        bool ok;
        const float x = tree_term_split<SCREENED>(dx, dy, dz, r2, a.w * a.w, b, sigma, sl2e, inv, ok);
        if (BF16) return __builtin_fmaf((on && ok) ? x : 0.f, inv, part);  // last product fused into the sum
        return part + ((on && ok) ? x * inv : 0.f);
    };
    // (with compensation only the lanes that opened the node, as adding a zero
    // would move bits between the sum and its compensation, and a point's value
    // must not depend on the points it shares the wave with)
    auto add = [&](float part, int h, uint64_t m) {
        if (!kahan) {
            sum[h] += part;
        } else if (__builtin_amdgcn_inverse_ballot_w64(m)) {
            kahan_add(sum[h], comp[h], part);
        }
    };
    // a leaf of several points, summed point by point for the parts whose
    // lanes opened it
    auto leaf_sum = [&](int b, int e, const uint64_t* m) {
        float part[H];
#pragma unroll
        for (int h = 0; h < H; ++h) part[h] = 0.f;
        for (int j = b; j < e; ++j) {
            const float4 pa = scalar_load(T.sa, j), pb = scalar_load(T.sb, j);
#pragma unroll
            for (int h = 0; h < H; ++h)
                if (H == 1 || m[h]) part[h] = point_term(pa, pb, __builtin_amdgcn_inverse_ballot_w64(m[h]), part[h], h);
        }
#pragma unroll
        for (int h = 0; h < H; ++h) {
            if (COUNT && __builtin_amdgcn_inverse_ballot_w64(m[h])) nterms[h] += e - b;
            if (H == 1 || m[h]) add(part[h], h, m[h]);
        }
    };

    // the bounding box of the brick's points, from its corners' indices (the
    // coordinates grow with the index)
    constexpr bool BOX = GRID && !COUNT && !NEAR64;
    float blx = 0.f, bly = 0.f, blz = 0.f, bhx = 0.f, bhy = 0.f, bhz = 0.f;
    if (BOX) {
        const int x0 = bxi * PX * 4, y0 = byi * PY * 4, z0 = bzi * PZ * 4;
        blx = __builtin_fmaf(float(x0), Q.h, Q.ox);
        bly = __builtin_fmaf(float(y0), Q.h, Q.oy);
        blz = __builtin_fmaf(float(z0), Q.h, Q.oz);
        bhx = __builtin_fmaf(float(x0 + 4 * PX - 1), Q.h, Q.ox);
        bhy = __builtin_fmaf(float(y0 + 4 * PY - 1), Q.h, Q.oy);
        bhz = __builtin_fmaf(float(z0 + 4 * PZ - 1), Q.h, Q.oz);
    }

    // the stack holds (traversal record of a node to open, lanes that open
    // it, per part): an internal node's first child, or a leaf's
    // (−count, begin).  In a grid walk the record's top bit says that every
    // lane opens the node: its masks are then neither written nor read back (not
    // where a part lies beyond the grid, whose terms would be computed for nobody)
    constexpr int kAllLanes = BOX ? int(0x80000000u) : 0;
    int sp = 0;
    const int4 root = scalar_load(T.info, 0);
    if (root.x < 0) {
        leaf_sum(root.y, root.z, all);
    } else {
        s_node_w[0] = make_int2(root.x, every ? kAllLanes : 0);
        if (!BOX || !every) {
#pragma unroll
            for (int h = 0; h < H; ++h) s_mask_w[h] = all[h];
        }
        sp = 1;
    }
    while (sp > 0) {
        --sp;
        const int2 top = s_node_w[sp];
        const int fc = uniform(top.x), ty = uniform(top.y);
        const bool full = BOX && ty < 0;
        uint64_t mask[H];
#pragma unroll
        for (int h = 0; h < H; ++h) mask[h] = all[h];
        if (!full) {
#pragma unroll
            for (int h = 0; h < H; ++h) mask[h] = uniform64(s_mask_w[sp * H + h]);
        }
        if (fc < 0) {  // a leaf of several points: summed point by point
            const int b = ty & ~kAllLanes;
            leaf_sum(b, b - fc, mask);
            continue;
        }
        float part[H];
#pragma unroll
        for (int h = 0; h < H; ++h) part[h] = 0.f;
        // the 8 children are contiguous: their records come in one batch of
        // scalar loads, their payloads in one coalesced vector load (word
        // 8c + w of child c in lane 8c + w), so a node costs one memory
        // round trip however many of its children are far or leaves
        int2 nks[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) nks[c] = scalar_load(T.kid, fc + c);
        // payload word 8c + w of child c: loaded by lane 8c + w, and (CM, w)
        // word 4c + w by lanes 4c + w and 32 + 4c + w (a second copy keeps the
        // store unconditional); both read back by the whole wave from LDS at
        // uniform addresses (broadcasts).  Records in LDS instead of SGPRs
        // leave the stack pointer room in the scalar registers
        const float pw = T.payload[int64_t(fc) * 8 + lane];
        const float cw = reinterpret_cast<const float*>(T.cm_r)[int64_t(fc) * 4 + (lane & 31)];
        reinterpret_cast<float*>(s_pay[wave])[lane] = pw;
        reinterpret_cast<float*>(s_cmr[wave])[lane] = cw;
        __builtin_amdgcn_wave_barrier();
        // Children whose far test has one outcome for the whole brick, from its
        // box: child c in lanes c, c + 8, ...  The distances are computed like
        // a lane's own r² and every step is monotone, so dmin² ≤ r² ≤ dmax²
        // holds as rounded and the outcome is each lane's own.  A far child
        // then needs no test and no mask and, beyond its bare floor, neither
        // the guard nor the screening maximum, and its four parts share more
        // of the offsets' products: 57 VALU for 256 terms instead of 68.  The
        // walk is bound by VALU issue: 14,414 → 12,650 VALU per brick and 12.85
        // → 12.33 ms for a 512³ grid over 1M sources, BF16 (75% of the terms
        // take this way).  Classifying the four parts one by one finds more
        // such pairs but costs more branches than it saves (13.4 ms)
        uint32_t far_all = 0, near_all = 0;
        if (BOX && full) {
            const float4 cr = s_cmr[wave][lane & 7];
            const float thr = fmaxf(cr.w, s_pay[wave][2 * (lane & 7) + 1].w);
            const float ax = blx - cr.x, bx = cr.x - bhx, ay = bly - cr.y, by = cr.y - bhy, az = blz - cr.z,
                        bz = cr.z - bhz;
            const float nx = fmaxf(fmaxf(ax, bx), 0.f), ny = fmaxf(fmaxf(ay, by), 0.f), nz = fmaxf(fmaxf(az, bz), 0.f);
            const float fx = fmaxf(fabsf(ax), fabsf(bx)), fy = fmaxf(fabsf(ay), fabsf(by)),
                        fz = fmaxf(fabsf(az), fabsf(bz));
            far_all = uint32_t(__builtin_amdgcn_ballot_w64(dist2(nx, ny, nz) > thr));
            near_all = uint32_t(__builtin_amdgcn_ballot_w64(!(dist2(fx, fy, fz) > cr.w)));
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int2 nk = nks[c];
            if (nk.x == 0) continue;  // empty
            if (BOX && ((far_all >> c) & 1u)) {
                const float4 cr = s_cmr[wave][c], e4 = s_pay[wave][2 * c];
                const float4 lo = BF16 ? make_float4(0.f, 0.f, 0.f, 0.f) : s_pay[wave][2 * c + 1];
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    float dx = cr.x - qx[h], dy = cr.y - qy[h], dz = cr.z - qz[h];
                    if (!BF16) {
                        dx += lo.x;
                        dy += lo.y;
                        dz += lo.z;
                    }
                    float inv;
                    const float x = bare_term_split<SCREENED>(dx, dy, dz, e4, sigma, sl2e, inv);
                    part[h] = BF16 ? __builtin_fmaf(x, inv, part[h]) : add_rounded(part[h], x, inv);
                }
                continue;
            }
            if (BOX && ((near_all >> c) & 1u)) {
                if (nk.x != -1) {
                    s_node_w[sp] = make_int2(nk.x, nk.y | kAllLanes);
                    ++sp;
                }
                continue;
            }
            // one test and one term for every kind of child: an internal
            // node is far when d² > (β·R)² (cm_r.w), a one-point leaf's
            // record makes the test its term's guard, a leaf of several
            // points is never far (∞) and is opened like an internal node
            const float4 cr = s_cmr[wave][c];
            uint64_t nm[H];
            bool push = false;
#pragma unroll
            for (int h = 0; h < H; ++h) {
                nm[h] = 0;
                if (H > 1 && !mask[h]) continue;  // no lane of this part opened the node
                const bool act = __builtin_amdgcn_inverse_ballot_w64(mask[h]);
                const float dx = cr.x - qx[h], dy = cr.y - qy[h], dz = cr.z - qz[h];
                const float r2 = dist2(dx, dy, dz);
                bool far = r2 > cr.w;
                if constexpr (NEAR64) {
                    // point terms inside the screening radius go to the FP64 sum
                    if (nk.x == -1) {
                        const bool nr = act && far && r2 < s_pay[wave][2 * c].w;
                        if (__builtin_amdgcn_ballot_w64(nr)) {  // rare: lanes next to a source
                            if (nr)
                                near[h] += near_term64(scalar_load(T.sa, nk.y), scalar_load(T.sb, nk.y), qx[h], qy[h],
                                                       qz[h], sigma);
                        }
                        far = far && !nr;
                    }
                }
                // lane masks straight from the compare: far for the lanes that
                // opened this node, near ones open the child
                const uint64_t farm = __builtin_amdgcn_ballot_w64(far);
                if (mask[h] & farm) {
                    const float4 e4 = s_pay[wave][2 * c];
                    if (BF16) {
                        // BF16 moments carry a relative error of 2^-9, far above
                        // the rounding of the centre: d = CM_f − q and its |d|²
                        // from the far test serve as they are, and the term's
                        // last product is fused into the sum.  r > 1e-10 holds
                        // for every far node here (far radius floor) and is the
                        // far test of a point.  The lanes that take the term are
                        // selected by the exec mask (mask & farm), not by a
                        // select on the result: one VALU instruction less per term
                        if (__builtin_amdgcn_inverse_ballot_w64(mask[h] & farm)) {
                            float inv;
                            bool ok;
                            const float x = tree_term_split<SCREENED>(dx, dy, dz, r2, e4.w, e4, sigma, sl2e, inv, ok);
                            part[h] = __builtin_fmaf(x, inv, part[h]);
                        }
                    } else {
                        // d = (CM_f − q) + δ: the first difference is exact for
                        // nearby values, so d carries a single rounding (δ = 0
                        // for a point)
                        const float4 lo = s_pay[wave][2 * c + 1];
                        const float ex = dx + lo.x, ey = dy + lo.y, ez = dz + lo.z;
                        float inv;
                        bool ok;
                        const float x =
                            tree_term_split<SCREENED>(ex, ey, ez, dist2(ex, ey, ez), e4.w, e4, sigma, sl2e, inv, ok);
                        // the plain dipole has no r > 1e-10 guard in the reference either
                        part[h] += ((act && far && ok) ? x * inv : 0.f);
                    }
                }
                if (COUNT && act && (far || nk.x == -1)) nterms[h] += 1;
                nm[h] = mask[h] & ~farm;
                push = push || nm[h] != 0;
            }
            if (push && nk.x != -1) {
                // every lane writes the same entry: no divergent branch, so
                // the stack pointer stays in a scalar register
                s_node_w[sp] = nk;  // top bit clear: the masks follow
#pragma unroll
                for (int h = 0; h < H; ++h) s_mask_w[sp * H + h] = nm[h];
                ++sp;
            }
        }
        if (full && kahan) {  // every lane with a point opened it: no masks to go by
#pragma unroll
            for (int h = 0; h < H; ++h) kahan_add(sum[h], comp[h], part[h]);
        } else {
#pragma unroll
            for (int h = 0; h < H; ++h)
                if (H == 1 || mask[h]) add(part[h], h, mask[h]);
        }
    }
#pragma unroll
    for (int h = 0; h < H; ++h) {
        if (valid[h]) {
            if (out) out[qi[h]] = NEAR64 ? float(double(sum[h] - comp[h]) + near[h]) : sum[h] - comp[h];
            if (COUNT) terms_out[qi[h]] = nterms[h];
        }
    }
}

// Barnes-Hut sums at explicit query points, and (GRAD; new, the reference has
// no gradient) their gradient.  The points come in the caller's order, so 64
// consecutive ones need not have anything in common, and one walk for the
// union of their traversals opens many times the nodes each needs.  Here L
// lanes walk for one query alone: lane 8g + c of them tests child c of the
// g-th node from the top of the query's stack, so L / 8 nodes are opened a
// step.  Each query takes exactly its own term set (the far test of
// gwn_tree_kernel; far dipoles at (CM_f − q) + residual, without the residual
// for BF16 moments); a lane sums its terms in FP64 and the lanes are added in
// a fixed order.
// Bound by the L2 reads of the node records (56 B a child, about 20 KB a
// query) and, for few queries, by the latency of a step (records, then
// payloads): few queries take 64 lanes each, many 8.
// A query's stack holds first-child indices (leaves of several points: the
// complement of the leaf's own index) and never overflows: opening a node
// leaves at most 7 entries more than it took, a step takes several nodes only
// while at most kWalkDeep entries wait, and above what that leaves there is
// room for a depth-first descent.
constexpr int kWalkWaves = 4, kWalkDeep = 64;
__host__ __device__ constexpr int walk_stack_entries(int max_level, int lanes) {
    return tree_stack_entries(max_level) + (lanes > 8 ? kWalkDeep + 7 * (lanes / 8) : 0);
}

template <bool SCREENED, bool BF16, bool GRAD, int L>
__global__ __launch_bounds__(kWalkWaves * 64) void gwn_walk_kernel(TreeArgs T, const float* __restrict__ q, int64_t nq,
                                                                    int stack, float sigma, float* __restrict__ out_w,
                                                                    float* __restrict__ out_g) {
    constexpr int kQueries = 64 / L, kNodes = L / 8;
    extern __shared__ int s_stacks[];  // kWalkWaves × kQueries stacks of `stack` entries
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int sub = lane / L, sl = lane % L, g = sl >> 3, c = lane & 7;
    int* ent = s_stacks + (wave * kQueries + sub) * stack;
    const int64_t qi = (int64_t(blockIdx.x) * kWalkWaves + wave) * kQueries + sub;
    const bool valid = qi < nq;
    if (!__builtin_amdgcn_ballot_w64(valid)) return;
    const float qx = valid ? q[3 * qi] : 0.f, qy = valid ? q[3 * qi + 1] : 0.f, qz = valid ? q[3 * qi + 2] : 0.f;
    const float sl2e = sigma * kLog2e;
    double sum[GRAD ? 4 : 1];
#pragma unroll
    for (int k = 0; k < (GRAD ? 4 : 1); ++k) sum[k] = 0.0;
    auto add = [&](float dx, float dy, float dz, float s2, const float4 b) {
        if constexpr (GRAD) {
            float dot, g, c;
            gwn_term_grad<SCREENED>(dx, dy, dz, s2, b, sigma, sl2e, dot, g, c);
            sum[0] += double(g * dot);
            sum[1] += double(grad_component<SCREENED>(c, dx, g, b.x));
            sum[2] += double(grad_component<SCREENED>(c, dy, g, b.y));
            sum[3] += double(grad_component<SCREENED>(c, dz, g, b.z));
        } else {
            float inv;
            bool ok;
            const float x = tree_term_split<SCREENED>(dx, dy, dz, dist2(dx, dy, dz), s2, b, sigma, sl2e, inv, ok);
            sum[0] += double(ok ? x * inv : 0.f);
        }
    };
    // the points of a leaf, 8 lanes of the query a step
    auto leaf = [&](int b, int e) {
        for (int j = b + c; j < e; j += 8) {
            const float4 pa = T.sa[j];
            add(pa.x - qx, pa.y - qy, pa.z - qz, pa.w * pa.w, T.sb[j]);
        }
    };
    const int4 root = T.info[0];
    int sp = 0;
    if (root.x < 0) {
        if (valid && g == 0) leaf(root.y, root.z);
    } else if (valid) {
        ent[0] = root.x;
        sp = 1;
    }
    __builtin_amdgcn_wave_barrier();
    while (__builtin_amdgcn_ballot_w64(sp > 0)) {
        const int nb = min(sp, sp <= kWalkDeep ? kNodes : 1);
        const bool on = g < nb;
        const int top = on ? ent[sp - 1 - g] : 0;
        sp -= nb;
        bool push = false;
        int next = 0;
        if (on && top < 0) {
            const int2 lf = T.kid[~top];
            leaf(lf.y, lf.y - lf.x);
        } else if (on) {
            const int64_t ch = int64_t(top) + c;
            const int2 nk = T.kid[ch];
            const float4 cr = T.cm_r[ch];
            if (nk.x != 0) {
                const float dx = cr.x - qx, dy = cr.y - qy, dz = cr.z - qz;
                // an internal node is far when d² > (β·R)² (cm_r.w), a one-point
                // leaf's record makes the test its term's guard, a leaf of
                // several points is never far (∞)
                if (dist2(dx, dy, dz) > cr.w) {
                    const float4* pay = reinterpret_cast<const float4*>(T.payload) + 2 * ch;
                    const float4 e4 = pay[0];
                    const float4 lo = BF16 ? make_float4(0.f, 0.f, 0.f, 0.f) : pay[1];
                    add(dx + lo.x, dy + lo.y, dz + lo.z, e4.w, e4);
                } else if (nk.x != -1) {
                    push = true;
                    next = nk.x > 0 ? nk.x : ~int(ch);
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
        const uint64_t pm = __builtin_amdgcn_ballot_w64(push) >> (sub * L);  // bit sl: this query's lane
        const uint64_t mine = L == 64 ? pm : pm & ((1ull << (L & 63)) - 1ull);
        if (push) ent[sp + __builtin_popcountll(mine & ((1ull << sl) - 1ull))] = next;
        sp += __builtin_popcountll(mine);
        __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int off = 1; off < L; off <<= 1)
#pragma unroll
        for (int k = 0; k < (GRAD ? 4 : 1); ++k) sum[k] += __shfl_xor(sum[k], off, 64);
    if (valid && sl == 0) {
        out_w[qi] = float(sum[0]);
        if constexpr (GRAD) {
            if (out_g) {
                out_g[3 * qi] = float(sum[1]);
                out_g[3 * qi + 1] = float(sum[2]);
                out_g[3 * qi + 2] = float(sum[3]);
            }
        }
    }
}

// The sums at the tree's own points (Q.self_perm) or at the points of a grid,
// 8 lanes a point as gwn_walk_kernel walks, but with each point's terms summed exactly as a lane of the shared walk sums
// them: the 8 children's terms of an opened node are computed side by side and
// added from child 0 to child 7, node by node in the same depth-first order, so
// the values are the shared walk's bit for bit.  For clouds and grids whose
// shared walks (up to 64 points a wave) leave most of the chip idle: bound by
// the latency of a node's records along one point's walk.
template <int CTRL>
__device__ __forceinline__ float dpp_row(float v) {  // lanes without a source keep v
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), CTRL, 0xF, 0xF, false));
}

template <bool SCREENED, bool BF16>
__global__ __launch_bounds__(kWalkWaves * 64) void gwn_ordered_walk_kernel(TreeArgs T, QueryArgs Q, float sigma,
                                                                            uint32_t flags,
                                                                            float* __restrict__ out) {
    extern __shared__ int s_stacks[];  // kWalkWaves × 8 stacks of `stack` entries
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, sub = lane >> 3, c = lane & 7;
    int* ent = s_stacks + (wave * 8 + sub) * Q.stack;
    const int64_t blk = xcd_block(blockIdx.x, gridDim.x);
    const int64_t slot = (blk * kWalkWaves + wave) * 8 + sub;
    const bool valid = slot < Q.nq;
    if (!__builtin_amdgcn_ballot_w64(valid)) return;
    float qx = 0.f, qy = 0.f, qz = 0.f;
    if (Q.grid) {
        qx = __builtin_fmaf(float(int(slot % Q.rx)), Q.h, Q.ox);
        qy = __builtin_fmaf(float(int(slot / Q.rx % Q.ry)), Q.h, Q.oy);
        qz = __builtin_fmaf(float(int(slot / (int64_t(Q.rx) * Q.ry))), Q.h, Q.oz);
    } else if (valid) {
        const float4 a = T.sa[slot];
        qx = a.x;
        qy = a.y;
        qz = a.z;
    }
    const float sl2e = sigma * kLog2e;
    const bool kahan = flags & DWG_KAHAN;
    float sum = 0.f, comp = 0.f;  // in lane 7 of the point
    // the terms x·inv of lanes 0 .. 7 added to `part` in that order (rounded
    // product by product, or fused, as the shared walk's sums are); the total
    // in lane 7.  Lanes without a term pass the sum on
    auto ordered = [&](float part, bool on, float x, float inv) {
        float t;
        {
#pragma clang fp contract(off)
            t = x * inv;
        }
        auto with = [&](float p) { return !on ? p : BF16 ? __builtin_fmaf(x, inv, p) : p + t; };
        float v = with(part);  // right in lane 0
#pragma unroll
        for (int k = 1; k < 8; ++k) {
            const float before = dpp_row<0x111>(v);  // row_shr 1: lane k takes lane k − 1
            v = c == k ? with(before) : v;
        }
        return v;
    };
    auto fold = [&](float part, bool on) {
        if (!on) return;
        if (kahan) kahan_add(sum, comp, part); else sum += part;
    };
    // a leaf of several points, 8 a step, for the points of the wave that
    // opened one (b .. e; an empty range for the others)
    auto leaf = [&](int b, int e, bool on) {
        float part = 0.f;
        for (int j0 = 0; __builtin_amdgcn_ballot_w64(on && b + j0 < e); j0 += 8) {
            const int j = b + j0 + c;
            const bool have = on && j < e;
            float inv = 0.f, x = 0.f;
            bool ok = false;
            if (have) {
                const float4 pa = T.sa[j];
                const float dx = pa.x - qx, dy = pa.y - qy, dz = pa.z - qz;
                x = tree_term_split<SCREENED>(dx, dy, dz, dist2(dx, dy, dz), pa.w * pa.w, T.sb[j], sigma, sl2e, inv, ok);
            }
            // (a guarded term adds a zero in the shared walk, which leaves the sum)
            const float v = ordered(part, have && ok, x, inv);
            part = __shfl(v, lane | 7, 64);
        }
        fold(part, on);
    };
    const int4 root = T.info[0];
    int sp = 0;
    if (root.x < 0) {
        leaf(root.y, root.z, valid);
    } else if (valid) {
        ent[0] = root.x;
        sp = 1;
    }
    __builtin_amdgcn_wave_barrier();
    while (__builtin_amdgcn_ballot_w64(sp > 0)) {
        const bool on = sp > 0;
        const int top = on ? ent[sp - 1] : 0;
        if (on) --sp;
        const bool node = on && top >= 0;
        bool push = false, term = false;
        int next = 0;
        float x = 0.f, inv = 0.f;
        if (node) {
            const int64_t ch = int64_t(top) + c;
            const int2 nk = T.kid[ch];
            const float4 cr = T.cm_r[ch];
            const float4* pay = reinterpret_cast<const float4*>(T.payload) + 2 * ch;
            const float4 e4 = pay[0];
            const float4 lo = BF16 ? make_float4(0.f, 0.f, 0.f, 0.f) : pay[1];
            const float dx = cr.x - qx, dy = cr.y - qy, dz = cr.z - qz;
            const float r2 = dist2(dx, dy, dz);
            if (nk.x != 0 && r2 > cr.w) {
                bool ok;
                if (BF16) {
                    x = tree_term_split<SCREENED>(dx, dy, dz, r2, e4.w, e4, sigma, sl2e, inv, ok);
                    term = true;
                } else {
                    const float ex = dx + lo.x, ey = dy + lo.y, ez = dz + lo.z;
                    x = tree_term_split<SCREENED>(ex, ey, ez, dist2(ex, ey, ez), e4.w, e4, sigma, sl2e, inv, ok);
                    term = ok;
                }
            } else if (nk.x != 0 && nk.x != -1) {
                push = true;
                next = nk.x > 0 ? nk.x : ~int(ch);
            }
        }
        __builtin_amdgcn_wave_barrier();
        const uint32_t mine = uint32_t(__builtin_amdgcn_ballot_w64(push) >> (8 * sub)) & 0xFFu;
        if (push) ent[sp + __builtin_popcount(mine & ((1u << c) - 1u))] = next;
        sp += __builtin_popcount(mine);
        __builtin_amdgcn_wave_barrier();
        fold(ordered(0.f, term, x, inv), node);
        if (__builtin_amdgcn_ballot_w64(on && top < 0)) {
            int2 lf = make_int2(0, 0);
            if (on && top < 0) lf = T.kid[~top];
            leaf(lf.y, lf.y - lf.x, on && top < 0);
        }
    }
    if (valid && c == 7) out[Q.grid ? slot : int64_t(Q.self_perm[slot])] = sum - comp;
}

// Which walk explicit queries take.  Alone (gwn_walk_kernel), 64 lanes a query
// below kWalkFew, where the waves do not fill the chip (1,000 of 100k sources:
// 17 µs, with 8 lanes 48, shared 1,190), else 8 (32,000: 57 and 75 against
// 1,380 µs; 100,000 with gradient: 0.17 against 2.5 ms).  From share_from on 64 to
// a shared walk, in spatial order: the node records are then read once for 64
// queries, which for 1M queries on the surface takes half the time, while unordered
// ones (2M: 12.8 ms shared, 3.3 ms alone) are put in order first.
constexpr int64_t kWalkFew = 40000;

// A launch of shared walks lasts as long as its longest, which grow with the
// tree, and lone walks cost the same for each query: sharing pays from a number of
// queries on that grows with the sources.  Of queries in order and unordered
// ones, near a surface, alone and shared (µs): 3,000 sources 150,000 70, 76 and 77,
// 97; 200,000 88, 99 and 75, 104.  400,000 sources 200,000 246, 363 and 352, 378;
// 300,000 336, 482 and 359, 368.  With gradient 3,000 sources 200,000 101, 113 and
// 115, 150; 300,000 144, 160 and 132, 165.  30,000 sources 300,000 251, 289 and 276,
// 340; 500,000 395, 467 and 322, 400.  1M sources 500,000 700, 962 and 920, 975;
// 800,000 1,089, 1,479 and 1,156, 1,238
static int64_t share_from(const dwg_octree* T, bool grad) {
    if (T->n_nodes == 1) return 0;  // a leaf has no walk to be alone on
    const double n = double(T->n_points);
    return int64_t(grad ? 62000.0 * std::pow(n, 1.0 / 6.0) : 82000.0 * std::pow(n, 1.0 / 12.0));
}

// The order: a counting sort by the Morton code of a 64³ grid over the tree's
// cube.  Queries that come in order already are left as they are, which a
// sample of runs of 64 decides: they come unsorted when such runs extend, on
// average, over four times the side that 64 of nq uniform points fill (in Morton
// order they extend over 1.9 to 2.4 times, the rows of a grid 14 times).  (32³ and 128³
// cells: 300,000 points over 400,000 sources 417 and 427 µs against 394 with 64³,
// 1M points 690 and 611 against 602.)  Queries in order pay for the launches that
// find it out, which are four for that reason: 8 to 10 µs (200,000 over 3,000 sources 66
// → 75, 800,000 over 400,000 446 → 455; with six launches 84 and 464).  The extent of
// each wave's own queries would cost them nothing, but then unordered ones could
// only walk alone
constexpr int kOrderBits = 6, kOrderBuckets = 1 << (3 * kOrderBits);
constexpr int kOrderSamples = 256;  // runs, one a block of the first launch
constexpr int kOrderThreads = 256;
static_assert(kOrderSamples == kOrderThreads, "a block adds up the samples, one a thread");

// Sources below which a walk is too short to put queries in order for: 300,000 and
// 1M unordered ones as they come 45 and 101 µs over 100 sources, 73 and 168 over 200,
// 111 and 260 over 400; in order 66 and 132, 72 and 142, 78 and 154
constexpr int64_t kOrderSources = 200;

// 12 B of scratch a query, and up to so many queries at a time: more are taken in
// equal parts, so that the scratch a context keeps for this stays below 204 MB
// and a query's number in 32 bits
constexpr int64_t kOrderMost = int64_t(1) << 24;

struct OrderCells {
    uint32_t count[kOrderBuckets];  // queries of a bucket
    uint32_t start[kOrderBuckets];  // queries before a bucket
    uint32_t sample[kOrderSamples]; // extent of a run relative to the cube, times its part near it, in 2^-16
    uint32_t extent;                // their sum
};
constexpr int kOrderZero = kOrderBuckets / kOrderSamples;  // counts that a block of the first launch clears

__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) v = fminf(v, __shfl_xor(v, off, 64));
    return v;
}

__global__ __launch_bounds__(kOrderThreads) void order_sample_kernel(const float* __restrict__ q, int64_t nq,
                                                                     const double4* __restrict__ cell,
                                                                     OrderCells* __restrict__ C) {
    for (int k = threadIdx.x; k < kOrderZero; k += kOrderThreads) C->count[blockIdx.x * kOrderZero + k] = 0;
    if (threadIdx.x >= 64) return;
    const int64_t i = int64_t(blockIdx.x) * (nq / 64) / kOrderSamples * 64 + threadIdx.x;  // nq ≥ 64
    const double4 c = cell[0];
    const float w = float(c.w), x[3] = {q[3 * i], q[3 * i + 1], q[3 * i + 2]};
    // (half the cube's width off it a point's walk is short in any company: such points
    // have no extent, and a run counts by its other points)
    const bool near = fmaxf(fmaxf(fabsf(x[0] - float(c.x)), fabsf(x[1] - float(c.y))), fabsf(x[2] - float(c.z))) <= w;
    const float part = float(__builtin_popcountll(__builtin_amdgcn_ballot_w64(near))) * (1.f / 64.f);
    float e = 0.f;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const float v = near ? x[d] : NAN;  // left out of the least
        e = fmaxf(e, -wave_min(-v) - wave_min(v));
    }
    if (threadIdx.x == 0) C->sample[blockIdx.x] = uint32_t(65536.f * fminf(fmaxf(e / w * part, 0.f), 1.f));
}

__device__ __forceinline__ int order_bucket(const float* __restrict__ q, int64_t i, const double4 c) {
    const float inv = float(double(1 << kOrderBits) / c.w);
    const float lo[3] = {float(c.x - 0.5 * c.w), float(c.y - 0.5 * c.w), float(c.z - 0.5 * c.w)};
    int m = 0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        // (a NaN, also of a cube of no width, becomes 0)
        const int v = int(fminf(fmaxf((q[3 * i + d] - lo[d]) * inv, 0.f), float((1 << kOrderBits) - 1)));
#pragma unroll
        for (int b = 0; b < kOrderBits; ++b) m |= ((v >> b) & 1) << (3 * b + d);
    }
    return m;
}

// the sum of v over the block's NT threads
template <int NT>
__device__ __forceinline__ uint32_t block_sum(uint32_t v) {
    __shared__ uint32_t s_wave[NT / 64];
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) v += uint32_t(__shfl_xor(int(v), off, 64));
    if ((threadIdx.x & 63) == 0) s_wave[threadIdx.x >> 6] = v;
    __syncthreads();
    v = 0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) v += s_wave[w];
    return v;
}

// the lanes whose bucket is this lane's (−1: none)
__device__ __forceinline__ uint64_t same_bucket(int b) {
    uint64_t m = __builtin_amdgcn_ballot_w64(b >= 0);
#pragma unroll
    for (int k = 0; k < 3 * kOrderBits; ++k) {
        const uint64_t ones = __builtin_amdgcn_ballot_w64((b >> k) & 1);
        m &= (b >> k) & 1 ? ones : ~ones;
    }
    return m;
}

// (bucket, place in it) of every query: the scatter then needs no atomics.  The
// lanes of a wave in one bucket take their places with one atomic add, as many
// queries may lie in one (equal ones, or all beyond one corner of the cube: 300,000
// took 0.78 ms one by one)
__global__ __launch_bounds__(kOrderThreads) void order_count_kernel(const float* __restrict__ q, int64_t nq,
                                                                    const double4* __restrict__ cell, unsigned limit,
                                                                    OrderCells* __restrict__ C,
                                                                    int2* __restrict__ place) {
    const uint32_t extent = block_sum<kOrderThreads>(C->sample[threadIdx.x]);
    if (blockIdx.x == 0 && threadIdx.x == 0) C->extent = extent;
    if (extent <= limit) return;
    const double4 root = cell[0];
    const int lane = threadIdx.x & 63;
    for (int64_t i0 = int64_t(blockIdx.x) * kOrderThreads; i0 < nq; i0 += int64_t(gridDim.x) * kOrderThreads) {
        const int64_t i = i0 + threadIdx.x;
        const int b = i < nq ? order_bucket(q, i, root) : -1;
        const uint64_t same = same_bucket(b);
        const int first = b >= 0 ? __builtin_ctzll(same) : lane;
        uint32_t at = 0;
        if (b >= 0 && lane == first) at = atomicAdd(&C->count[b], uint32_t(__builtin_popcountll(same)));
        at = uint32_t(__shfl(int(at), first, 64)) + uint32_t(__builtin_popcountll(same & ((1ull << lane) - 1ull)));
        if (i < nq) place[i] = make_int2(b, int(at));
    }
}

// The buckets' starts: a block takes a tile of them, four a thread, and adds up all
// counts before its own, 1 MB at most and from L2, in place of a launch that does
constexpr int kStartThreads = 1024, kStartTile = 4 * kStartThreads;
__global__ __launch_bounds__(kStartThreads) void order_start_kernel(QueryOrder O, OrderCells* __restrict__ C) {
    if (!O.sorted()) return;
    const uint4* count = reinterpret_cast<const uint4*>(C->count);
    const int tile = blockIdx.x * kStartThreads;  // in fours
    uint32_t before = 0;
#pragma unroll 8
    for (int k = threadIdx.x; k < tile; k += kStartThreads) {
        const uint4 c = count[k];
        before += (c.x + c.y) + (c.z + c.w);
    }
    before = block_sum<kStartThreads>(before);
    const uint4 c = count[tile + threadIdx.x];
    const uint32_t sum = (c.x + c.y) + (c.z + c.w);
    __shared__ uint32_t s_scan[kStartThreads / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t incl = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = uint32_t(__shfl_up(int(incl), off, 64));
        incl += lane >= off ? y : 0;
    }
    if (lane == 63) s_scan[wave] = incl;
    __syncthreads();
    uint32_t at = before + incl - sum;
#pragma unroll
    for (int w = 0; w < kStartThreads / 64; ++w) at += w < wave ? s_scan[w] : 0;
    reinterpret_cast<uint4*>(C->start)[tile + threadIdx.x] = make_uint4(at, at + c.x, at + c.x + c.y, at + c.x + c.y + c.z);
}

__global__ __launch_bounds__(kOrderThreads) void order_scatter_kernel(const int2* __restrict__ place, int64_t nq,
                                                                      QueryOrder O, const OrderCells* __restrict__ C,
                                                                      int* __restrict__ order) {
    if (!O.sorted()) return;
    for (int64_t i = int64_t(blockIdx.x) * kOrderThreads + threadIdx.x; i < nq;
         i += int64_t(gridDim.x) * kOrderThreads) {
        const int2 b = place[i];
        order[C->start[b.x] + b.y] = int(i);
    }
}

// the queries of one launch that shares walks
static int64_t order_part(int64_t nq) {
    const int64_t parts = (nq + kOrderMost - 1) / kOrderMost;
    return ((nq + parts - 1) / parts + 63) / 64 * 64;
}

// Whether queries that share walks are looked at for an order.  A call that is
// recorded into a graph takes them as they come: the scratch of an order could not
// be allocated, or given back by a later call while the graph still used it
static bool may_order(const dwg_ctx* ctx, const dwg_octree* T) {
    if (T->n_points < kOrderSources || T->n_nodes == 1) return false;
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(ctx->stream, &st) == hipSuccess) return st == hipStreamCaptureStatusNone;
    (void)hipGetLastError();
    return false;
}

// the caller's order where there is no memory for another
static QueryOrder query_order(dwg_ctx* ctx, const dwg_octree* T, const float* q, int64_t nq) {
    OrderCells* C = nullptr;
    int2* place = nullptr;
    int* order = nullptr;
    try {
        C = static_cast<OrderCells*>(ctx->buf("order_cells", sizeof(OrderCells)));
        place = static_cast<int2*>(ctx->buf("order_place", sizeof(int2) * size_t(nq)));
        order = static_cast<int*>(ctx->buf("order", sizeof(int) * size_t(nq)));
    } catch (const Error&) {
        (void)hipGetLastError();
        return QueryOrder{};
    }
    ProfileScope ps(ctx, "gwn_query_order");
    const QueryOrder O{order, &C->extent, unsigned(65536.f * 4.f * std::cbrt(64.f / float(nq)) * float(kOrderSamples))};
    hipLaunchKernelGGL(order_sample_kernel, dim3(kOrderSamples), dim3(kOrderThreads), 0, ctx->stream, q, nq, T->cell, C);
    check_launch();
    const unsigned blocks = std::min(grid_for(nq, kOrderThreads), 1024u);
    hipLaunchKernelGGL(order_count_kernel, dim3(blocks), dim3(kOrderThreads), 0, ctx->stream, q, nq, T->cell, O.limit, C,
                       place);
    check_launch();
    hipLaunchKernelGGL(order_start_kernel, dim3(kOrderBuckets / kStartTile), dim3(kStartThreads), 0, ctx->stream, O, C);
    check_launch();
    hipLaunchKernelGGL(order_scatter_kernel, dim3(blocks), dim3(kOrderThreads), 0, ctx->stream, place, nq, O, C, order);
    check_launch();
    return O;
}

template <bool GRAD>
static void launch_walk(dwg_ctx* ctx, const dwg_octree* T, const float* q, int64_t nq, float sigma, uint32_t flags,
                        float* out_w, float* out_g) {
    const TreeArgs A{T->info, T->kid, T->cm_r, reinterpret_cast<const float*>(T->payload), T->sa, T->sb};
    const int lanes = nq < kWalkFew ? 64 : 8;
    const int stack = walk_stack_entries(std::max(T->max_level, 1), lanes);
    const int64_t per = int64_t(kWalkWaves) * (64 / lanes);
    const size_t lds = sizeof(int) * size_t(stack) * size_t(per);
    dim3 grid(grid_for(nq, int(per))), block(kWalkWaves * 64);
#define DWG_WALK(S, B)                                                                                                  \
    do {                                                                                                                \
        if (lanes == 64)                                                                                                \
            hipLaunchKernelGGL((gwn_walk_kernel<S, B, GRAD, 64>), grid, block, lds, ctx->stream, A, q, nq, stack, sigma, \
                               out_w, out_g);                                                                           \
        else                                                                                                            \
            hipLaunchKernelGGL((gwn_walk_kernel<S, B, GRAD, 8>), grid, block, lds, ctx->stream, A, q, nq, stack, sigma, \
                               out_w, out_g);                                                                           \
    } while (0)
    const bool scr = flags & DWG_SCREENED;
    bool done = false;
    if constexpr (!GRAD) {
        if (flags & DWG_FAR_BF16) {
            if (scr) DWG_WALK(true, true);
            else DWG_WALK(false, true);
            done = true;
        }
    }
    if (!done) {
        if (scr) DWG_WALK(true, false);
        else DWG_WALK(false, false);
    }
#undef DWG_WALK
    check_launch();
}

// Value and gradient at many query points: the shared walk and far test of
// gwn_tree_kernel (FP32 path: far dipoles at (CM_f − q) + residual), each
// lane accumulating w and ∇w of its own term set.
template <bool SCREENED>
__global__ __launch_bounds__(kTreeThreads) void gwn_tree_grad_kernel(TreeArgs T, const float* __restrict__ q,
                                                                      int64_t nq, QueryOrder order, float sigma,
                                                                      float* __restrict__ out_w,
                                                                      float* __restrict__ out_g) {
    __shared__ int s_node[kTreeWaves][kStack];
    __shared__ uint64_t s_mask[kTreeWaves][kStack];
    __shared__ float4 s_pay[kTreeWaves][16];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t slot = (int64_t(blockIdx.x) * kTreeWaves + wave) * 64 + lane;
    const bool valid = slot < nq;
    const int64_t qi = valid ? order.query(slot) : slot;
    const float qx = valid ? q[3 * qi] : 0.f, qy = valid ? q[3 * qi + 1] : 0.f, qz = valid ? q[3 * qi + 2] : 0.f;
    const uint64_t all = __builtin_amdgcn_ballot_w64(valid);
    if (all == 0) return;
    const float sl2e = sigma * kLog2e;
    // the terms of one opened node sum into `part`, which folds into `acc`
    // with Kahan compensation: the gradient's near terms are large and
    // cancel, so plain FP32 accumulation over many nodes would lose digits
    float acc[4] = {0.f, 0.f, 0.f, 0.f}, comp[4] = {0.f, 0.f, 0.f, 0.f}, part[4] = {0.f, 0.f, 0.f, 0.f};
    auto add = [&](float dx, float dy, float dz, float s2, const float4 b, bool on) {
        float dot, g, c;
        gwn_term_grad<SCREENED>(dx, dy, dz, s2, b, sigma, sl2e, dot, g, c);
        g = on ? g : 0.f;
        c = on ? c : 0.f;
        part[0] = __builtin_fmaf(g, dot, part[0]);
        part[1] += grad_component<SCREENED>(c, dx, g, b.x);
        part[2] += grad_component<SCREENED>(c, dy, g, b.y);
        part[3] += grad_component<SCREENED>(c, dz, g, b.z);
    };
    // (for the lanes that took part: adding a zero would move bits between the
    // sum and its compensation)
    auto fold = [&](bool on) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (on) kahan_add(acc[k], comp[k], part[k]);
            part[k] = 0.f;
        }
    };
    auto leaf = [&](int b, int e, bool on) {
        for (int j = b; j < e; ++j) {
            const float4 a = scalar_load(T.sa, j);
            add(a.x - qx, a.y - qy, a.z - qz, a.w * a.w, scalar_load(T.sb, j), on);
        }
    };
    int sp = 0;
    const int4 root = T.info[0];
    if (root.x < 0) {
        leaf(root.y, root.z, valid);
        fold(valid);
    } else {
        if (lane == 0) {
            s_node[wave][0] = root.x;
            s_mask[wave][0] = all;
        }
        sp = 1;
    }
    while (sp > 0) {
        --sp;
        const int fc = uniform(s_node[wave][sp]);
        const uint64_t mask = uniform64(s_mask[wave][sp]);
        const bool act = (mask >> lane) & 1;
        reinterpret_cast<float*>(s_pay[wave])[lane] = T.payload[int64_t(fc) * 8 + lane];
        __builtin_amdgcn_wave_barrier();
        for (int c = 0; c < 8; ++c) {
            const int2 nk = scalar_load(T.kid, fc + c);
            if (nk.x == 0) continue;
            if (nk.x < 0) {
                leaf(nk.y, nk.y - nk.x, act);
                continue;
            }
            const float4 cr = scalar_load(T.cm_r, fc + c);
            const float dx = cr.x - qx, dy = cr.y - qy, dz = cr.z - qz;
            const bool far = dist2(dx, dy, dz) > cr.w;
            const uint64_t farm = __builtin_amdgcn_ballot_w64(far);
            if (mask & farm) {
                const float4 lo = s_pay[wave][2 * c + 1];
                add(dx + lo.x, dy + lo.y, dz + lo.z, kDipoleS2, s_pay[wave][2 * c], act && far);
            }
            const uint64_t nm = mask & ~farm;
            if (nm) {
                if (lane == 0) {
                    s_node[wave][sp] = nk.x;
                    s_mask[wave][sp] = nm;
                }
                ++sp;
            }
        }
        fold(act);
        __builtin_amdgcn_wave_barrier();
    }
    if (valid) {
        out_w[qi] = acc[0] - comp[0];
        if (out_g) {
            out_g[3 * qi] = acc[1] - comp[1];
            out_g[3 * qi + 1] = acc[2] - comp[2];
            out_g[3 * qi + 2] = acc[3] - comp[3];
        }
    }
}

static QueryArgs make_points(const float* q, int64_t nq) {
    QueryArgs Q{};
    Q.q = q;
    Q.nq = nq;
    return Q;
}

static QueryArgs make_self(const dwg_octree* T) {
    QueryArgs Q{};
    Q.self_perm = T->perm;
    Q.nq = T->n_points;
    return Q;
}

// Grids of few whole bricks leave the chip short of waves, and the launch lasts
// as long as its longest walks: they take one 4×4×4 part a wave, whose walk
// opens fewer nodes and lasts a quarter as long.  The longer the walks, the
// more bricks it takes to hide the longest: whole ones win from about
// 420 · ∛n on (800 sources: 96³ 100 µs whole and 95 in parts, 112³ 125 and 131;
// 30,000: 144³ 467 and 462, 160³ 560 and 594; 400,000: 160³ 1,011 and 849, 192³
// 1,270 and 1,220, 256³ 1,776 and 2,204).  The values are the same: each point
// takes its own terms in the same order
constexpr double kWholeBricks = 420.0;

// And below kGridAlone points (kGridAloneDense where the sources are a third of
// them or more, as then a part's walks have little in common), or kSelfAlone of
// the tree's own, 8 lanes walk for each point (gwn_ordered_walk_kernel):
// 33×29×31 over 2,000 sources 181 µs by whole bricks, 77 by parts, 33 alone;
// 48³ over 2,000 66 by either; 64³ over 10,000 101 and 151, over 100,000 253 and
// 216; 80³ over 1M 531 and 449.  Own points: 30,000 208 → 52 µs, 200,000 350 →
// 270, 1M 0.91 and 1.56 ms
constexpr int64_t kGridAlone = 131072, kGridAloneDense = 524288, kSelfAlone = 250000;

// `whole_bricks`: for the walks that take no others
static QueryArgs make_grid(const dwg_octree* T, const dwg_grid* g, bool whole_bricks) {
    QueryArgs Q{};
    Q.grid = true;
    Q.ox = g->origin[0];
    Q.oy = g->origin[1];
    Q.oz = g->origin[2];
    Q.h = g->h;
    Q.rx = g->res[0];
    Q.ry = g->res[1];
    Q.rz = g->res[2];
    auto bricks = [&](int parts, int px, int py, int pz) {
        Q.parts = parts;
        Q.bx = (Q.rx + 4 * px - 1) / (4 * px);
        Q.by = (Q.ry + 4 * py - 1) / (4 * py);
        Q.bz = (Q.rz + 4 * pz - 1) / (4 * pz);
        Q.n_bricks = int64_t(Q.bx) * Q.by * Q.bz;
    };
    Q.flat = Q.rz <= 4;
    if (Q.flat) bricks(kGridParts, kPartsX, kPartsZ, kPartsY);
    else bricks(kGridParts, kPartsX, kPartsY, kPartsZ);
    // (also at most 4 points along x, of which whole bricks leave half empty: 4×700×700
    // over 3,000 sources 143 µs whole, 117 in parts, 3×1,500×1,500 over 100,000 BF16
    // 453 and 417)
    auto in_parts = [&]() {
        return (Q.rx <= 4 && T->n_nodes > 1) || double(Q.n_bricks) < kWholeBricks * std::cbrt(double(T->n_points));
    };
    if (!whole_bricks && in_parts()) bricks(1, 1, 1, 1);
    Q.nq = int64_t(Q.rx) * Q.ry * Q.rz;
    return Q;
}

// cm_r.w = (β·R)² for the traversal's far test d² > (β·R)², with the
// rounding sequence float(β·R) then its square (the order the oracle uses),
// clamped below by `floor`.  A leaf with one point gets `point_guard`, so
// that the far test is the point term's own guard (r² > 1e-20 screened,
// none plain: −1); a leaf with several points ∞, so that it is always
// opened and its points summed one by one
__global__ void far_radius_kernel(const int2* __restrict__ kid, const float* __restrict__ r, int64_t m, float beta,
                                  float floor, float point_guard, float4* __restrict__ cm_r) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= m) return;
    const int k = kid[i].x;
    const float br = beta * r[i];
    cm_r[i].w = k == -1 ? point_guard : k < -1 ? INFINITY : fmaxf(br * br, floor);
}

// Far-radius floor of the mixed-precision walk: with d² > 4e-20 every far
// node has r = |d| > 2e-10, so the screened term's r > 1e-10 guard always
// holds there and the walk drops it.  Only a node whose points all lie within
// 1e-10 of each other (duplicates) has (β·R)² below the floor; it is opened
// instead, and its points' own guarded terms give the same sum.
constexpr float kFarFloorBf16 = 4e-20f;

// Far-field moments in the payload of every internal node: EC/4π in FP32,
// or rounded to BF16 (to nearest even, kept in FP32 words) for BF16
// evaluations
__global__ void payload_precision_kernel(const int2* __restrict__ kid, const float4* __restrict__ ec, int64_t m,
                                         int bf16, float4* __restrict__ payload) {
    const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= m || kid[i].x <= 0) return;
    const float4 e = ec[i];
    payload[2 * i] = bf16 ? make_float4(bf16_round(e.x), bf16_round(e.y), bf16_round(e.z), kDipoleS2)
                          : make_float4(e.x, e.y, e.z, kDipoleS2);
}

static void launch_tree(dwg_ctx* ctx, const dwg_octree* Tc, const QueryArgs& Q, float beta, float sigma,
                        uint32_t flags, float* out, int64_t* terms, bool count) {
    DWG_REQUIRE(Tc && Tc->updated, "octree has no moments yet: call dwg_octree_update first");
    DWG_REQUIRE(Tc->max_level <= kMaxTreeLevel, "octree deeper than the traversal stack");
    auto* T = const_cast<dwg_octree*>(Tc);  // the far radii follow β; the tree itself is unchanged
    const bool want_bf16 = (flags & DWG_FAR_BF16) && !count;
    const float floor = want_bf16 ? kFarFloorBf16 : 0.f;
    const float guard = (flags & DWG_SCREENED) ? 1e-20f : -1.f;
    if (!(T->far_beta == beta) || T->far_floor != floor || T->far_guard != guard) {
        hipLaunchKernelGGL(far_radius_kernel, dim3(grid_for(T->n_nodes, 256)), dim3(256), 0, ctx->stream, T->kid,
                           T->radius, T->n_nodes, beta, floor, guard, T->cm_r);
        check_launch();
        T->far_beta = beta;
        T->far_floor = floor;
        T->far_guard = guard;
    }
    if (T->payload_bf16 != want_bf16) {
        hipLaunchKernelGGL(payload_precision_kernel, dim3(grid_for(T->n_nodes, 256)), dim3(256), 0, ctx->stream, T->kid,
                           T->ec, T->n_nodes, int(want_bf16), T->payload);
        check_launch();
        T->payload_bf16 = want_bf16;
    }
    const bool near64 = (flags & DWG_SCREENED) && (flags & DWG_NEAR_FP64);
    if (Q.q && !count && !near64 && Q.nq < share_from(T, false)) {
        if (Q.nq == 0) return;
        ProfileScope ps(ctx, (flags & DWG_SCREENED) ? "gwn_tree_screened" : "gwn_tree_plain");
        launch_walk<false>(ctx, T, Q.q, Q.nq, sigma, flags, out, nullptr);
        return;
    }
    // (a tree that is one leaf has no walk to be alone on)
    const bool alone = T->n_nodes > 1 &&
                       (Q.grid ? Q.nq < kGridAlone || (Q.nq < kGridAloneDense && 3 * T->n_points >= Q.nq)
                               : Q.self_perm && Q.nq < kSelfAlone);
    if (alone && !count && !near64) {
        const bool scr = flags & DWG_SCREENED, bf = flags & DWG_FAR_BF16;
        const TreeArgs A{T->info, T->kid, T->cm_r, reinterpret_cast<const float*>(T->payload), T->sa, T->sb};
        QueryArgs Qs = Q;
        Qs.stack = tree_stack_entries(std::max(T->max_level, 1));
        dim3 grid(grid_for(Q.nq, kWalkWaves * 8)), block(kWalkWaves * 64);
        const size_t lds = sizeof(int) * size_t(Qs.stack) * kWalkWaves * 8;
        ProfileScope ps(ctx, Q.grid ? (scr ? "gwn_tree_grid_screened" : "gwn_tree_grid_plain")
                                    : (scr ? "gwn_tree_screened" : "gwn_tree_plain"));
#define DWG_ORDERED(S, B) \
    hipLaunchKernelGGL((gwn_ordered_walk_kernel<S, B>), grid, block, lds, ctx->stream, A, Qs, sigma, flags, out)
        if (scr && bf) DWG_ORDERED(true, true);
        else if (scr) DWG_ORDERED(true, false);
        else if (bf) DWG_ORDERED(false, true);
        else DWG_ORDERED(false, false);
#undef DWG_ORDERED
        check_launch();
        return;
    }
    TreeArgs A{T->info, T->kid, T->cm_r, reinterpret_cast<const float*>(T->payload), T->sa, T->sb};
    const bool scr = flags & DWG_SCREENED, bf = flags & DWG_FAR_BF16;
    const char* name = count ? "gwn_tree_terms" : (!Q.grid ? (scr ? "gwn_tree_screened" : "gwn_tree_plain")
                                                           : (scr ? "gwn_tree_grid_screened" : "gwn_tree_grid_plain"));
    // explicit points are put in order first, a part of them at a time
    const bool in_order = Q.q && Q.nq >= share_from(T, false) && may_order(ctx, T);
    const int64_t part = in_order ? order_part(Q.nq) : Q.nq;
    for (int64_t first = 0; first < Q.nq; first += part) {
        QueryArgs Qs = Q;
        float* o = out ? out + first : nullptr;
        int64_t* t = terms ? terms + first : nullptr;
        if (in_order) {
            Qs.q = Q.q + 3 * first;
            Qs.nq = std::min(part, Q.nq - first);
            Qs.order = query_order(ctx, T, Qs.q, Qs.nq);
        }
        const int64_t waves = Q.grid ? Q.n_bricks : (Qs.nq + 64 * kPointPts - 1) / (64 * kPointPts);
        dim3 grid(grid_for(waves, kTreeWaves)), block(kTreeThreads);
        // the walk's stack: one record and one lane mask per part for each entry
        Qs.stack = tree_stack_entries(std::max(T->max_level, 1));
        const size_t lds = sizeof(uint64_t) * size_t(Qs.stack) * size_t(1 + (Q.grid ? Q.parts : kPointPts));
        ProfileScope ps(ctx, name);
#define DWG_TREE_LAUNCH(S, C, B, G, N) \
    hipLaunchKernelGGL((gwn_tree_kernel<S, C, B, G, N>), grid, block, lds, ctx->stream, A, Qs, beta, sigma, flags, o, t)
#define DWG_TREE_LAUNCH_Q(S, C, B, N)                \
    do {                                             \
        if (!Q.grid)                                 \
            DWG_TREE_LAUNCH(S, C, B, 0, N);          \
        else if (Q.flat)                             \
            DWG_TREE_LAUNCH(S, C, B, kFlatParts, N); \
        else                                         \
            DWG_TREE_LAUNCH(S, C, B, kGridParts, N); \
    } while (0)
// (the counting and the FP64 near-field walks take whole bricks only)
#define DWG_TREE_LAUNCH_P(S, B)                 \
    do {                                        \
        if (Q.grid && Q.parts == 1)             \
            DWG_TREE_LAUNCH(S, false, B, 1, false); \
        else                                    \
            DWG_TREE_LAUNCH_Q(S, false, B, false);  \
    } while (0)
        if (count) DWG_TREE_LAUNCH_Q(false, true, false, false);
        else if (near64 && bf) DWG_TREE_LAUNCH_Q(true, false, true, true);
        else if (near64) DWG_TREE_LAUNCH_Q(true, false, false, true);
        else if (scr && bf) DWG_TREE_LAUNCH_P(true, true);
        else if (scr) DWG_TREE_LAUNCH_P(true, false);
        else if (bf) DWG_TREE_LAUNCH_P(false, true);
        else DWG_TREE_LAUNCH_P(false, false);
#undef DWG_TREE_LAUNCH_P
#undef DWG_TREE_LAUNCH_Q
#undef DWG_TREE_LAUNCH
        check_launch();
    }
}

void gwn_tree(dwg_ctx* ctx, const dwg_octree* T, const float* q, int64_t nq, float beta, float sigma, uint32_t flags,
              float* out) {
    DWG_REQUIRE(nq >= 0 && (q || nq == 0), "bad query array");
    launch_tree(ctx, T, make_points(q, nq), beta, sigma, flags, out, nullptr, false);
}

void gwn_tree_self(dwg_ctx* ctx, const dwg_octree* T, float beta, float sigma, uint32_t flags, float* out) {
    DWG_REQUIRE(T, "null octree");
    launch_tree(ctx, T, make_self(T), beta, sigma, flags, out, nullptr, false);
}

void gwn_tree_grid(dwg_ctx* ctx, const dwg_octree* T, const dwg_grid* g, float beta, float sigma, uint32_t flags,
                   float* out) {
    DWG_REQUIRE(T, "null octree");
    DWG_REQUIRE(g && g->res[0] > 0 && g->res[1] > 0 && g->res[2] > 0 && g->h > 0, "bad grid");
    launch_tree(ctx, T, make_grid(T, g, (flags & DWG_SCREENED) && (flags & DWG_NEAR_FP64)), beta, sigma, flags, out,
                nullptr, false);
}

void gwn_tree_grad(dwg_ctx* ctx, const dwg_octree* Tc, const float* q, int64_t nq, float beta, float sigma,
                   uint32_t flags, float* out_w, float* out_g) {
    DWG_REQUIRE(Tc && Tc->updated, "octree has no moments yet: call dwg_octree_update first");
    DWG_REQUIRE(Tc->max_level <= kMaxTreeLevel, "octree deeper than the traversal stack");
    DWG_REQUIRE(nq >= 0 && (q || nq == 0) && (out_w || nq == 0), "bad query or output array");
    auto* T = const_cast<dwg_octree*>(Tc);  // far radii follow β and the payload precision; the tree is unchanged
    const float guard = (flags & DWG_SCREENED) ? 1e-20f : -1.f;
    if (!(T->far_beta == beta) || T->far_floor != 0.f || T->far_guard != guard) {
        hipLaunchKernelGGL(far_radius_kernel, dim3(grid_for(T->n_nodes, 256)), dim3(256), 0, ctx->stream, T->kid,
                           T->radius, T->n_nodes, beta, 0.f, guard, T->cm_r);
        check_launch();
        T->far_beta = beta;
        T->far_floor = 0.f;
        T->far_guard = guard;
    }
    if (T->payload_bf16) {
        hipLaunchKernelGGL(payload_precision_kernel, dim3(grid_for(T->n_nodes, 256)), dim3(256), 0, ctx->stream, T->kid,
                           T->ec, T->n_nodes, 0, T->payload);
        check_launch();
        T->payload_bf16 = false;
    }
    if (nq == 0) return;
    if (nq < share_from(T, true)) {
        ProfileScope ps(ctx, "gwn_tree_grad");
        launch_walk<true>(ctx, T, q, nq, sigma, flags, out_w, out_g);
        return;
    }
    TreeArgs A{T->info, T->kid, T->cm_r, reinterpret_cast<const float*>(T->payload), T->sa, T->sb};
    const bool in_order = may_order(ctx, T);
    const int64_t part = in_order ? order_part(nq) : nq;
    for (int64_t first = 0; first < nq; first += part) {
        const int64_t n = std::min(part, nq - first);
        const float* qs = q + 3 * first;
        float *w = out_w + first, *g = out_g ? out_g + 3 * first : nullptr;
        const QueryOrder order = in_order ? query_order(ctx, T, qs, n) : QueryOrder{};
        dim3 grid(grid_for((n + 63) / 64, kTreeWaves)), block(kTreeThreads);
        ProfileScope ps(ctx, "gwn_tree_grad");
        if (flags & DWG_SCREENED)
            hipLaunchKernelGGL(gwn_tree_grad_kernel<true>, grid, block, 0, ctx->stream, A, qs, n, order, sigma, w, g);
        else
            hipLaunchKernelGGL(gwn_tree_grad_kernel<false>, grid, block, 0, ctx->stream, A, qs, n, order, sigma, w, g);
        check_launch();
    }
}

void gwn_tree_terms(dwg_ctx* ctx, const dwg_octree* T, const float* q, int64_t nq, float beta, int64_t* terms) {
    launch_tree(ctx, T, make_points(q, nq), beta, 0.f, 0, nullptr, terms, true);
}

__global__ void sum_i64_kernel(const int64_t* __restrict__ v, int64_t n, unsigned long long* __restrict__ out) {
    __shared__ unsigned long long lds[256];
    unsigned long long s = 0;
    for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n; i += int64_t(gridDim.x) * 256) s += v[i];
    lds[threadIdx.x] = s;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if (threadIdx.x < off) lds[threadIdx.x] += lds[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(out, lds[0]);
}

int64_t gwn_tree_grid_terms(dwg_ctx* ctx, const dwg_octree* T, const dwg_grid* g, float beta) {
    QueryArgs Q = make_grid(T, g, true);
    int64_t* terms = static_cast<int64_t*>(ctx->buf("grid_terms", sizeof(int64_t) * (Q.nq + 1)));
    unsigned long long* tot = reinterpret_cast<unsigned long long*>(terms + Q.nq);
    fill_u32(ctx, tot, 0, 2);
    launch_tree(ctx, T, Q, beta, 0.f, 0, nullptr, terms, true);
    hipLaunchKernelGGL(sum_i64_kernel, dim3(1024), dim3(256), 0, ctx->stream, terms, Q.nq, tot);
    check_launch();
    return int64_t(read_scalar<unsigned long long>(ctx, tot));
}

}  // namespace dwg
