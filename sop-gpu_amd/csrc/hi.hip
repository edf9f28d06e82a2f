// hi.hip -- hydrodynamic interactions: the Rotne-Prager-Yamakawa tensor with
// the TEA (truncated expansion) integrator and the exact Cholesky path.
//
// Reference: src/Integrators/bdhitea_kernel.cu (integrateTea_prepare :33-65,
// integrateTea_RPY :67-87, integrateCholesky_D :89-152,
// integrateCholesky_decompose :154-190, integrateTea_epsilon :212-249,
// integrateTea_force :252-300, integrateCholesky_L :303-361,
// integrateTea_kernel[_unlisted] :364-515) and src/Integrators/bdhitea.cu
// (TeaUpdater::update :133-176).
//
// The per-step preparation (noise into rforce, forces into mforce) is done by
// k_step for HI jobs; these kernels do the rest.  Neighbour coordinates come
// from the step-start buffer, so no kernel reads what it writes.
//
// The exact path factorises the RPY matrix (3N x 3N, padded to a multiple
// of 64 with an identity block) by a blocked Cholesky over outer panels of
// kCholPanel columns, each factored by 64-column steps (k_chol_step), one
// launch per step over the 64-row blocks from the step's diagonal down:
//   the previous step's column block is solved against the inverse of its
//   diagonal block (X = B Li^T on MFMA) and emitted in FP32, and into the
//   panel copy that the updates read (FP32, or split-BF16 pairs hi = bf16(x),
//   lo = bf16(x - hi));
//   the step's column block is updated by the panel's columns to its left on
//   MFMA -- split-BF16 with three products (hi*hi + hi*lo + lo*hi, FP32
//   accumulate) or FP32 -- with the K range split over the workgroup's
//   wavefronts;
//   the diagonal workgroup factors its block (FP64 in the FP32 mode, FP32 in
//   the split-BF16 mode; 16-column passes in registers, rank-16 updates and
//   the inverse's off-diagonal blocks on MFMA) and forms the inverse the
//   next step solves with.
// Wide MFMA kernels then update the next panel's columns and, on a second
// stream beside the next panel's steps, the rest of the trailing matrix.
#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>
#include <mutex>
#include <string>

#include "../../include/sopgpu.h"
#include "devmath.h"
#include "hi.h"
#include "hostutil.h"
#include "jobdesc.h"

namespace sop {

typedef short bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));

struct F6 {
    float xx, xy, xz, yy, yz, zz;
};

// D_ij / D_ii for a normalised separation with its length in w.
__device__ __forceinline__ F6 rpy(const float4 dr, float a) {
    F6 d;
    // the correctly rounded quotients of the reference's expressions; where
    // the operands lie in div_rn_fast's range (ra in (2, 2^59]: every
    // numerator below is then in [2^-60, 1) and every divisor in (2, 2^59]),
    // by the short division, else by the IEEE one -- the same bits
    float ra = div_rn_fast(dr.w, a);
    if (!(div_fast_numerator(dr.w) && a >= kDivFastMinB && a <= kDivFastMaxB)) ra = div_ieee(dr.w, a);
    float crr, cii;
    if (ra > 2.f) {
        constexpr float two_thirds = 2.f / 3.f;
        float q0 = div_rn_fast(0.75f, ra), q1 = div_rn_fast(2.f, ra), q3 = div_rn_fast(two_thirds, ra);
        float q2 = div_rn_fast(q1, ra), q4 = div_rn_fast(q3, ra);
        if (!(ra <= 0x1p59f)) {
            q0 = div_ieee(0.75f, ra);
            q1 = div_ieee(2.f, ra);
            q2 = div_ieee(q1, ra);
            q3 = div_ieee(two_thirds, ra);
            q4 = div_ieee(q3, ra);
        }
        crr = q0 * (1.f - q2);
        cii = q0 * (1.f + q4);
    } else {
        crr = 3.f * ra / 32.f;
        cii = 1.f - 9.f * ra / 32.f;
    }
    d.xx = dr.x * dr.x * crr + cii;
    d.xy = dr.x * dr.y * crr;
    d.xz = dr.x * dr.z * crr;
    d.yy = dr.y * dr.y * crr + cii;
    d.yz = dr.y * dr.z * crr;
    d.zz = dr.z * dr.z * crr + cii;
    return d;
}

// b - a, normalised, length in w
__device__ __forceinline__ float4 unit_sep(const float4 a, const float4 b) {
    float4 dr = b;
    dr.x -= a.x;
    dr.y -= a.y;
    dr.z -= a.z;
    dr.w = sqrtf(dr.x * dr.x + dr.y * dr.y + dr.z * dr.z);
    // correctly rounded quotients: the short division where w and the
    // components lie in its range (w in [2^-60, 2^60], each component 0 or
    // of magnitude at least 2^-60; at most w), else the IEEE one
    const float x = dr.x, y = dr.y, z = dr.z, w = dr.w;
    dr.x = div_rn_fast(x, w);
    dr.y = div_rn_fast(y, w);
    dr.z = div_rn_fast(z, w);
    const bool fast = w >= kDivFastMinA && w <= kDivFastMaxA && div_fast_numerator(fabsf(x)) &&
                      div_fast_numerator(fabsf(y)) && div_fast_numerator(fabsf(z));
    if (!fast) {
        dr.x = div_ieee(x, w);
        dr.y = div_ieee(y, w);
        dr.z = div_ieee(z, w);
    }
    return dr;
}

// rpy(unit_sep(..)) for the separation (x, y, z) of squared length d2, in
// about half the operations, where pair_short_ok holds: every quotient and the
// square root correctly rounded by the short sequences (one reciprocal per
// divisor; 2/ra is twice the rounded 1/ra), so the same bits.  ya = RN(1/a).
// The close form (ra <= 2) is evaluated only where some lane needs it.
__device__ __forceinline__ bool pair_short_ok(float x, float y, float z, float d2) {
    return (fminf(fminf(fabsf(x), fabsf(y)), fabsf(z)) >= 0x1p-32f) & (d2 <= kDivFastMaxB);
}
// a: w / a stays within the short division's range for every w = sqrt(d2) above
__device__ __forceinline__ bool pair_short_radius(float a) { return a >= 0x1p-20f && a <= 0x1p20f; }
__device__ __forceinline__ F6 rpy_short(float x, float y, float z, float d2, float a, float ya) {
    constexpr float two_thirds = 2.f / 3.f;
    const float w = sqrt_rn_fast(d2);
    const float yw = recip_rn_fast(w);
    x = quot_rn_fast(x, w, yw);
    y = quot_rn_fast(y, w, yw);
    z = quot_rn_fast(z, w, yw);
    const float ra = quot_rn_fast(w, a, ya);
    const float yr = recip_rn_fast(ra);
    const float q0 = quot_rn_fast(0.75f, ra, yr), q2 = quot_rn_fast(2.f * yr, ra, yr);
    const float q4 = quot_rn_fast(quot_rn_fast(two_thirds, ra, yr), ra, yr);
    float crr = q0 * (1.f - q2);
    float cii = q0 * (1.f + q4);
    if (__builtin_amdgcn_ballot_w64(!(ra > 2.f))) {
        asm volatile("");  // a branch, not a select: few chunks hold a close pair
        crr = ra > 2.f ? crr : 3.f * ra / 32.f;
        cii = ra > 2.f ? cii : 1.f - 9.f * ra / 32.f;
    }
    F6 d;
    d.xx = x * x * crr + cii;
    d.xy = x * y * crr;
    d.xz = x * z * crr;
    d.yy = y * y * crr + cii;
    d.yz = y * z * crr;
    d.zz = z * z * crr + cii;
    return d;
}

__device__ __forceinline__ int wave_of() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

// tile loop shared with kernels.hip's layout (64-bead tiles, 4 per block)
#define FOR_TILES(ntiles)                                                 \
    const int lane = threadIdx.x & 63;                                    \
    for (int t = blockIdx.x * 4 + wave_of(); t < (ntiles); t += gridDim.x * 4)

__device__ __forceinline__ void hi_finish(const DevJob& J, int d, long long s, float fx, float fy, float fz,
                                          float4 coord) {
    if ((J.flags & JF_PULLING) && J.bflag[d] == 1) {
        fx = 0.0f; fy = 0.0f; fz = 0.0f;
    }
    const float m = J.hOverZeta;
    const float dx = m * fx, dy = m * fy, dz = m * fz;
    coord.x += dx;
    coord.y += dy;
    coord.z += dz;
    J.coord[(s + 1) & 1][d] = coord;
    const bool reset = (s % J.stride == 0) && (s % J.nav == 0);
    const float T0 = reset ? 0.0f : J.T[d];
    J.T[d] = T0 + J.tempNorm * (dx * dx + dy * dy + dz * dz);
}

// ---------------------------------------------------------------------------
// TEA
// ---------------------------------------------------------------------------
__device__ __forceinline__ void eps_add(const float4 c1, const float4 c2, float a, float4& sum) {
    const float4 dr = unit_sep(c1, c2);
    const F6 d = rpy(dr, a);
    float4 p;
    p.w = d.xx + 2 * d.xy + 2 * d.xz + d.yy + 2 * d.yz + d.zz;
    p.x = d.xx * d.xx + d.xy * d.xy + d.xz * d.xz;
    p.y = d.xy * d.xy + d.yy * d.yy + d.yz * d.yz;
    p.z = d.xz * d.xz + d.yz * d.yz + d.zz * d.zz;
    sum.x += p.x;
    sum.y += p.y;
    sum.z += p.z;
    sum.w += p.w;
}

// The all-pairs HI sums (epsilon, TEA step, exact D.F): workgroups of B beads,
// B wavefronts, 64 / B workgroups per 64-bead tile, taking the partners in
// chunks of C.  hi_config chooses (B, C) by the beads of the launch.  Measured
// on TEA runs, us per step of the whole run, with (4, 256) / (8, 256) /
// (16, 256) / (8, 128):
//   4,096 beads of one chain          72 / 68 / 66 / 70
//   9,558 beads of nine chains        58 / 56 / 71 / 51
// One workgroup per CU (16 wavefronts hide the latencies): the largest B that
// still gives every CU one, 256 partners between barriers.  More beads than 16
// per CU: small workgroups, several on a CU, whose last round leaves less of
// the chip idle.
struct HiConfig {
    int beads, chunk;
};
static HiConfig hi_config(long long beads) {
    constexpr int kCus = 256;
    if (beads <= 4 * kCus) return {4, 256};
    if (beads <= 8 * kCus) return {8, 256};
    if (beads <= 16 * kCus) return {16, 256};
    return {8, 128};
}

// Ordered all-pairs sums of a workgroup's B beads.  Each chunk of C
// partners: wavefront w forms the NC components of the terms of beads
// dbase + 2 (w % (B/2)) and the next one with one half of the chunk (a partner
// per lane, its data loaded once for both beads) into an LDS buffer, and
// after the chunk's barrier lanes B c + b of wavefront 0 add component c of
// bead dbase + b in partner order, four terms per LDS read, while the other
// wavefronts already form the next chunk into the second buffer.  Terms that
// the sequential loop skips (the bead itself, partners past n) are -0.0f,
// which leaves every sum unchanged (x + -0 = x for every x), so each sum is
// the same sequence of additions as the reference's bead-by-bead loop.
// `acc` enters as the summing lane's starting value and leaves as its sum.
// `pair` holds the two beads' data: pair.load(j) reads a partner's,
// pair.sep(k, s, ..) its separation from bead k, pair.term(k, s, D, v) fills
// the terms from the RPY block, and pair.general(k, s) gives the block where
// the short evaluation is not admitted.
// Bound by VALU issue: per pair about 90 instructions with the short square
// root and shared reciprocals (150 before: the general square root, range
// checks per quotient and a reciprocal per quotient).
template <int B, int C, int NC, typename Pair>
__device__ __forceinline__ void hi_ordered_sums(float (*buf)[NC][B][C + 4], int n, const int (&b)[2], Pair pair,
                                                float& acc) {
    const int lane = threadIdx.x & 63, w = wave_of();
    const int sc = lane / B, sb = lane % B;
    const int row = 2 * (w % (B / 2)), half = w / (B / 2);
    const float a = pair.a, ya = 1.0f / a;
    const bool radius = pair_short_radius(a);
    int c = 0;
    for (int base = 0; base < n; base += C, ++c) {
        float(*tb)[B][C + 4] = buf[c & 1];
#pragma unroll
        for (int u = 0; u < C / 128; ++u) {
            const int at = half * (C / 2) + 64 * u, j0 = base + at, j = j0 + lane;
            const auto src = pair.load(min(j, n - 1));
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                // the chunk's 64 partners hold the bead itself or pass n
                const bool edge = j0 + 64 > n || (b[k] >= j0 && b[k] < j0 + 64);
                const bool valid = j < n && j != b[k];
                float x, y, z, v[NC];
                pair.sep(k, src, x, y, z);
                const float d2 = x * x + y * y + z * z;
                const bool ok = radius & pair_short_ok(x, y, z, d2);
                pair.term(k, src, rpy_short(x, y, z, d2, a, ya), v);
                const bool bad = edge ? valid & !ok : !ok;
                if (__builtin_amdgcn_ballot_w64(bad)) {
                    if (bad) pair.term(k, src, pair.general(k, src), v);
                }
#pragma unroll
                for (int q = 0; q < NC; ++q) tb[q][row + k][at + lane] = v[q];
                if (edge && !valid) {
#pragma unroll
                    for (int q = 0; q < NC; ++q) tb[q][row + k][at + lane] = -0.f;
                }
            }
        }
        __syncthreads();
        if (w == 0 && sc < NC) {
            const float4* __restrict__ r4 = reinterpret_cast<const float4*>(&tb[sc][sb][0]);
#pragma unroll 8
            for (int k = 0; k < C / 4; ++k) {
                const float4 q = r4[k];
                acc += q.x;
                acc += q.y;
                acc += q.z;
                acc += q.w;
            }
        }
    }
}

// The two beads (clamped to the last one) of wavefront w and their pairs.
struct HiPairBase {
    const float4* __restrict__ cur;
    float4 c[2];
    float a;
    __device__ __forceinline__ void sep(int k, const float4 r, float& x, float& y, float& z) const {
        x = r.x - c[k].x;
        y = r.y - c[k].y;
        z = r.z - c[k].z;
    }
};
__device__ __forceinline__ float4 ld4(const float4* p, int j) {
    typedef float v4 __attribute__((ext_vector_type(4)));
    const v4 v = *reinterpret_cast<const __attribute__((address_space(1))) v4*>(
        reinterpret_cast<const __attribute__((address_space(1))) char*>(
            (const __attribute__((address_space(1))) float4*)p) +
        ((unsigned)j << 4));
    return make_float4(v.x, v.y, v.z, v.w);
}
// epsilon: the sums of the RPY block's squares and of its entries
struct HiPairEps : HiPairBase {
    __device__ __forceinline__ float4 load(int j) const { return ld4(cur, j); }
    __device__ __forceinline__ F6 general(int k, const float4 r) const { return rpy(unit_sep(c[k], r), a); }
    __device__ __forceinline__ void term(int, const float4, const F6 d, float (&v)[4]) const {
        v[3] = d.xx + 2 * d.xy + 2 * d.xz + d.yy + 2 * d.yz + d.zz;
        v[0] = d.xx * d.xx + d.xy * d.xy + d.xz * d.xz;
        v[1] = d.xy * d.xy + d.yy * d.yy + d.yz * d.yz;
        v[2] = d.xz * d.xz + d.yz * d.yz + d.zz * d.zz;
    }
};
// D F of the exact path
struct HiPairD : HiPairBase {
    const float4* __restrict__ mforce;
    struct Src {
        float4 r, f;
    };
    __device__ __forceinline__ Src load(int j) const { return Src{ld4(cur, j), ld4(mforce, j)}; }
    __device__ __forceinline__ void sep(int k, const Src& s, float& x, float& y, float& z) const {
        HiPairBase::sep(k, s.r, x, y, z);
    }
    __device__ __forceinline__ F6 general(int k, const Src& s) const { return rpy(unit_sep(c[k], s.r), a); }
    __device__ __forceinline__ void term(int, const Src& s, const F6 D, float (&v)[3]) const {
        v[0] = D.xx * s.f.x + D.xy * s.f.y + D.xz * s.f.z;
        v[1] = D.xy * s.f.x + D.yy * s.f.y + D.yz * s.f.z;
        v[2] = D.xz * s.f.x + D.yz * s.f.y + D.zz * s.f.z;
    }
};
// the TEA step: D (F_j + C_i rho_j)
struct HiPairTea : HiPairBase {
    const float4* __restrict__ mforce;
    const float4* __restrict__ rforce;
    float ci[2][3];
    struct Src {
        float4 r, f, g;
    };
    __device__ __forceinline__ Src load(int j) const { return Src{ld4(cur, j), ld4(mforce, j), ld4(rforce, j)}; }
    __device__ __forceinline__ void sep(int k, const Src& s, float& x, float& y, float& z) const {
        HiPairBase::sep(k, s.r, x, y, z);
    }
    __device__ __forceinline__ F6 general(int k, const Src& s) const { return rpy(unit_sep(c[k], s.r), a); }
    __device__ __forceinline__ void term(int k, const Src& s, const F6 D, float (&v)[3]) const {
        const float gx = s.f.x + s.g.x * ci[k][0], gy = s.f.y + s.g.y * ci[k][1], gz = s.f.z + s.g.z * ci[k][2];
        v[0] = D.xx * gx + D.xy * gy + D.xz * gz;
        v[1] = D.xy * gx + D.yy * gy + D.yz * gz;
        v[2] = D.xz * gx + D.yz * gy + D.zz * gz;
    }
};
// the beads of this wavefront, of the workgroup's B from dbase
template <int B>
__device__ __forceinline__ void hi_beads(int dbase, int n, int (&b)[2]) {
    const int row = 2 * (wave_of() % (B / 2));
    b[0] = min(dbase + row, n - 1);
    b[1] = min(dbase + row + 1, n - 1);
}

// Per-bead sums of the TEA epsilon (bdhitea_kernel.cu:212-249): without
// lists, the ordered chunk sums of hi_ordered_sums (the same bits as the
// bead-by-bead loop); with lists, wavefront 0 of the tile's first
// workgroup walks bead i's lists.
template <int B, int C>
__global__ __launch_bounds__(64 * B) void k_hi_eps(const DevJob* __restrict__ jobs, const DevJobState* __restrict__ st,
                                                 const int2* __restrict__ tiles, int ntiles) {
    __shared__ __attribute__((aligned(16))) float eterm[2][4][B][C + 4];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int2 td = tiles[blockIdx.x / (64 / B)];
    const int q = blockIdx.x % (64 / B);
    const DevJob& J = jobs[td.x];
    if (!(J.flags & JF_HI) || (J.flags & JF_HI_EXACT)) return;
    const long long s = st[td.x].step;
    if (!(s < J.end_step && s % J.stride == 0 && s % J.hi_eps_freq == 0)) return;
    const bool listed = (J.flags & JF_HI_LISTED) != 0;
    const int n = J.n;
    const float4* __restrict__ cur = J.coord[s & 1];
    const float a = J.hi_a;
    if (listed) {  // lane = bead of the 64-bead tile
        const int d = td.y + lane;
        if (q != 0 || w != 0 || d >= n) return;
        const float4 c = cur[d];
        float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int k = 0; k < J.cov_cnt[d]; ++k) eps_add(c, cur[J.cov_j[(size_t)k * n + d]], a, sum);
        for (int k = 0; k < J.nat_cnt[d]; ++k) eps_add(c, cur[J.nat_j[(size_t)k * n + d]], a, sum);
        for (int k = 0; k < J.pair_cnt[d]; ++k)
            eps_add(c, cur[list_at(J.pair_j, J.idx16, (size_t)k * J.pair_ld + d)], a, sum);
        J.ci[d] = sum;
        J.eps[d] = sum.w;
        return;
    }
    // unlisted: lanes B c + b of wavefront 0 sum component c of bead dbase + b
    const int dbase = td.y + B * q;
    int bb[2];
    hi_beads<B>(dbase, n, bb);
    HiPairEps pair;
    pair.cur = cur;
    pair.a = a;
    pair.c[0] = ld4(cur, bb[0]);
    pair.c[1] = ld4(cur, bb[1]);
    float acc = 0.f;
    hi_ordered_sums<B, C, 4>(eterm, n, bb, pair, acc);
    // component c of bead dbase + b is in lane B c + b of wavefront 0
    const float sy = __shfl(acc, lane + B), sz = __shfl(acc, lane + 2 * B), sw = __shfl(acc, (lane + 3 * B) & 63);
    if (w == 0 && lane < B && dbase + lane < n) {
        J.ci[dbase + lane] = make_float4(acc, sy, sz, sw);
        J.eps[dbase + lane] = sw;
    }
}

// TeaUpdater::update (bdhitea.cu:133-176): epsilon and beta' in FP64, one
// 256-thread workgroup per job.  The reference adds the per-bead values in
// bead order into a double.  Where the values' exponents span few enough bits
// that every partial sum, in any order, is a multiple of the smallest value's
// last place below 2^53 of them, each addition is exact and the order does
// not matter: the workgroup adds them in parallel (4,096 values: 56 -> 8 us,
// the chain of dependent additions).  Otherwise (values apart by more than
// about 2^18, infinities, NaN) wavefront 0 adds them one by one, staged in
// LDS kBetaChunk at a time.
constexpr int kBetaThreads = 256;
__global__ __launch_bounds__(kBetaThreads) void k_hi_beta(const DevJob* __restrict__ jobs,
                                                          DevJobState* __restrict__ st, int njobs) {
    const int jb = blockIdx.x, t = threadIdx.x, lane = t & 63;
    if (jb >= njobs) return;
    const DevJob& J = jobs[jb];
    if (!(J.flags & JF_HI) || (J.flags & JF_HI_EXACT)) return;
    DevJobState& S = st[jb];
    const long long s = S.step;
    if (!(s < J.end_step && s % J.stride == 0 && s % J.hi_eps_freq == 0)) return;
    const int N = J.n;
    constexpr int kBetaChunk = 4096;
    __shared__ __attribute__((aligned(16))) float chunk[kBetaChunk];
    __shared__ double psum[kBetaThreads / 64];
    __shared__ int pmax[kBetaThreads / 64], pmin[kBetaThreads / 64];
    // biased exponents: the largest of all values, the smallest of the nonzero
    double part = 0.0;
    int emax = 0, emin = 255;
#pragma unroll 4
    for (int i = t; i < N; i += kBetaThreads) {
        const float v = J.eps[i];
        const int e = (int)((__float_as_uint(v) >> 23) & 0xffu);
        part += (double)v;
        emax = max(emax, e);
        if (v != 0.0f) emin = min(emin, max(e, 1));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        part += __shfl_xor(part, o);
        emax = max(emax, __shfl_xor(emax, o));
        emin = min(emin, __shfl_xor(emin, o));
    }
    if (lane == 0) {
        psum[t >> 6] = part;
        pmax[t >> 6] = emax;
        pmin[t >> 6] = emin;
    }
    __syncthreads();
    double epsilon = 0.0;
    for (int k = 0; k < kBetaThreads / 64; ++k) {
        epsilon += psum[k];
        emax = max(emax, pmax[k]);
        emin = min(emin, pmin[k]);
    }
    if (t >= 64) return;
    // |partial sum| < N 2^(emax+1), a multiple of 2^(emin-23)
    const int bits = 32 - __builtin_clz((unsigned)N) + emax + 1 - (emin - 23);
    if (emax == 255 || (emax > 0 && bits > 53)) {
        epsilon = 0.0;
        for (int base = 0; base < N; base += kBetaChunk) {
            float v[kBetaChunk / 64];
#pragma unroll
            for (int u = 0; u < kBetaChunk / 64; ++u) {
                const int i = base + 64 * u + lane;
                v[u] = i < N ? J.eps[i] : 0.f;
            }
#pragma unroll
            for (int u = 0; u < kBetaChunk / 64; ++u) chunk[64 * u + lane] = v[u];
            wave_lds_order();
            const int m = min(kBetaChunk, N - base);
            const float4* __restrict__ c4 = reinterpret_cast<const float4*>(chunk);
            int k = 0;
            for (; k + 4 <= m; k += 4) {
                const float4 q = c4[k >> 2];
                epsilon += (double)q.x;
                epsilon += (double)q.y;
                epsilon += (double)q.z;
                epsilon += (double)q.w;
            }
            for (; k < m; ++k) epsilon += (double)chunk[k];
            wave_lds_order();
        }
    }
    if (lane != 0) return;  // the sum is uniform; one lane updates the state
    if (N > 1) epsilon /= 3. * N * (3. * N - 3.);
    if (epsilon > 1.0) {
        if (J.hi_capricious) S.overflow |= 4;
        epsilon = 1.0;
    }
    if (epsilon > J.hi_epsmax) S.overflow |= 4;
    const double a = (3. * N - 1.) * epsilon * epsilon - (3. * N - 2.) * epsilon;
    if (fabs(a) < 1e-7) {
        S.beta = .5f;
        if (J.hi_capricious && J.hi_a > 0.0f) S.overflow |= 8;
    } else {
        S.beta = (float)((1. - sqrt(1. - a)) / a);
    }
    S.eps_traj = epsilon;
}

__device__ __forceinline__ void tea_force(const float4 c1, const float4 c2, const float4 mf, const float4 rf,
                                          const float ci0, const float ci1, const float ci2, float a, float& fx,
                                          float& fy, float& fz) {
    const float4 dr = unit_sep(c1, c2);
    float gx = mf.x, gy = mf.y, gz = mf.z;
    gx += rf.x * ci0;
    gy += rf.y * ci1;
    gz += rf.z * ci2;
    const F6 D = rpy(dr, a);
    fx += D.xx * gx + D.xy * gy + D.xz * gz;
    fy += D.xy * gx + D.yy * gy + D.yz * gz;
    fz += D.xz * gx + D.yz * gy + D.zz * gz;
}

// The TEA step (bdhitea_kernel.cu:364-515).  Unlisted: the terms are
// added in partner order, the order of the reference's sequential loop, by
// hi_ordered_sums.  Listed: wavefront 0 of the tile's first workgroup walks
// the lists.
template <int B, int C>
__global__ __launch_bounds__(64 * B) void k_hi_tea(const DevJob* __restrict__ jobs, const DevJobState* __restrict__ st,
                                                 const int2* __restrict__ tiles, int ntiles, int kstep) {
    __shared__ __attribute__((aligned(16))) float tterm[2][3][B][C + 4];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int2 td = tiles[blockIdx.x / (64 / B)];
    const int q = blockIdx.x % (64 / B);
    const DevJob& J = jobs[td.x];
    if (!(J.flags & JF_HI) || (J.flags & JF_HI_EXACT)) return;
    const DevJobState& S = st[td.x];
    const long long s = S.step + kstep;
    if (s >= J.end_step) return;
    const bool listed = (J.flags & JF_HI_LISTED) != 0;
    const int n = J.n;
    const float4* __restrict__ cur = J.coord[s & 1];
    const float a = J.hi_a;
    if (listed) {  // lane = bead of the 64-bead tile
        const int d = td.y + lane;
        if (q != 0 || w != 0 || d >= n) return;
        float4 cs = J.ci[d];
        const float4 f0 = J.mforce[d];
        const float4 df = J.rforce[d];
        const float beta = S.beta;
        cs.w = beta * beta;
        float ci0 = 1.f / sqrtf(1.f + cs.w * cs.x);
        float ci1 = 1.f / sqrtf(1.f + cs.w * cs.y);
        float ci2 = 1.f / sqrtf(1.f + cs.w * cs.z);
        const float4 coord = cur[d];
        float fx = f0.x, fy = f0.y, fz = f0.z, tx, ty, tz;
        fx += df.x * ci0;
        fy += df.y * ci1;
        fz += df.z * ci2;
        ci0 *= beta;
        ci1 *= beta;
        ci2 *= beta;
        for (int k = 0; k < J.cov_cnt[d]; ++k) {
            const int i = J.cov_j[(size_t)k * n + d];
            tx = 0.f; ty = 0.f; tz = 0.f;
            tea_force(coord, cur[i], J.mforce[i], J.rforce[i], ci0, ci1, ci2, a, tx, ty, tz);
            fx += tx; fy += ty; fz += tz;
        }
        for (int k = 0; k < J.nat_cnt[d]; ++k) {
            const int i = J.nat_j[(size_t)k * n + d];
            tx = 0.f; ty = 0.f; tz = 0.f;
            tea_force(coord, cur[i], J.mforce[i], J.rforce[i], ci0, ci1, ci2, a, tx, ty, tz);
            fx += tx; fy += ty; fz += tz;
        }
        for (int k = 0; k < J.pair_cnt[d]; ++k) {
            const int i = list_at(J.pair_j, J.idx16, (size_t)k * J.pair_ld + d);
            tx = 0.f; ty = 0.f; tz = 0.f;
            tea_force(coord, cur[i], J.mforce[i], J.rforce[i], ci0, ci1, ci2, a, tx, ty, tz);
            fx += tx; fy += ty; fz += tz;
        }
        hi_finish(J, d, s, fx, fy, fz, coord);
        return;
    }
    // unlisted: the wavefront's two beads with their ci (uniform over the
    // wavefront); lanes B c + b of wavefront 0 sum component c of bead dbase + b
    // from its starting value
    const int dbase = td.y + B * q, ds = dbase + lane % B;
    int bd[2];
    hi_beads<B>(dbase, n, bd);
    HiPairTea pair;
    pair.cur = cur;
    pair.mforce = J.mforce;
    pair.rforce = J.rforce;
    pair.a = a;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const float4 cs = ld4(J.ci, bd[k]);
        const float bb = S.beta * S.beta;
        pair.ci[k][0] = 1.f / sqrtf(1.f + bb * cs.x) * S.beta;
        pair.ci[k][1] = 1.f / sqrtf(1.f + bb * cs.y) * S.beta;
        pair.ci[k][2] = 1.f / sqrtf(1.f + bb * cs.z) * S.beta;
        pair.c[k] = ld4(cur, bd[k]);
    }
    float acc = 0.f;
    if (w == 0 && lane < 3 * B && ds < n) {  // the bead's starting value, component lane / B
        const float4 cs = J.ci[ds], f0 = J.mforce[ds], df = J.rforce[ds];
        const float bb = S.beta * S.beta;
        const int k = lane / B;
        const float cc = k == 0 ? cs.x : (k == 1 ? cs.y : cs.z);
        const float f = k == 0 ? f0.x : (k == 1 ? f0.y : f0.z), g = k == 0 ? df.x : (k == 1 ? df.y : df.z);
        acc = f;
        acc += g * (1.f / sqrtf(1.f + bb * cc));
    }
    hi_ordered_sums<B, C, 3>(tterm, n, bd, pair, acc);
    const float sy = __shfl(acc, lane + B), sz = __shfl(acc, lane + 2 * B);
    if (w == 0 && lane < B && ds < n) hi_finish(J, ds, s, acc, sy, sz, cur[ds]);
}

// ---------------------------------------------------------------------------
// exact path
// ---------------------------------------------------------------------------

// F_i + sum_j D_ij F_j into fdf, summed in bead order (hi_ordered_sums), for
// the (single) exact-HI job of the launch: the terms D_ij F_j are the three
// row sums, written exactly as the sequential loop writes them, so every sum
// is the same bits as the bead-by-bead loop.
template <int B, int C>
__global__ __launch_bounds__(64 * B) void k_chol_D(const DevJob* __restrict__ jobs, const DevJobState* __restrict__ st,
                                                 const int2* __restrict__ tiles, int ntiles, int kstep) {
    __shared__ __attribute__((aligned(16))) float dterm[2][3][B][C + 4];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int2 td = tiles[blockIdx.x / (64 / B)];
    const DevJob& J = jobs[td.x];
    if (!(J.flags & JF_HI_EXACT)) return;  // one job per launch: uniform
    const long long s = st[td.x].step + kstep;
    if (s >= J.end_step) return;
    const int n = J.n;
    const int dbase = td.y + B * (blockIdx.x % (64 / B)), ds = dbase + lane % B;
    const float4* __restrict__ cur = J.coord[s & 1];
    int bd[2];
    hi_beads<B>(dbase, n, bd);
    HiPairD pair;
    pair.cur = cur;
    pair.mforce = J.mforce;
    pair.a = J.hi_a;
    pair.c[0] = ld4(cur, bd[0]);
    pair.c[1] = ld4(cur, bd[1]);
    float acc = 0.f;
    if (w == 0 && lane < 3 * B && ds < n) {
        const float4 f0 = J.mforce[ds];
        acc = lane < B ? f0.x : (lane < 2 * B ? f0.y : f0.z);
    }
    hi_ordered_sums<B, C, 3>(dterm, n, bd, pair, acc);
    const float sy = __shfl(acc, lane + B), sz = __shfl(acc, lane + 2 * B);
    if (w == 0 && lane < B && ds < n) J.fdf[ds] = make_float4(acc, sy, sz, 0.0f);
}

// D/D_ii lower block triangle into M on refactorisation steps: block
// (blockIdx.x, blockIdx.y) of 64x64 bead pairs (i in tile x, d in tile y,
// d <= i), identity 3x3 blocks on the diagonal; the same RPY blocks k_chol_D
// sums, written row by row (consecutive threads: consecutive d).
__global__ __launch_bounds__(256) void k_chol_build(const DevJob* __restrict__ jobs, const DevJobState* __restrict__ st,
                                                    const int2* __restrict__ tiles, int kstep) {
    if (blockIdx.y > blockIdx.x) return;
    const int2 ti = tiles[blockIdx.x], tdd = tiles[blockIdx.y];
    const DevJob& J = jobs[ti.x];
    const long long s = st[ti.x].step + kstep;
    const int n = J.n;
    const float4* __restrict__ cur = J.coord[s & 1];
    const size_t ld = J.chol_ld;
    float* __restrict__ M = J.chol_M;
    const float a = J.hi_a;
    const int dl = threadIdx.x & 63;
    const int d = tdd.y + dl;
    if (d >= n) return;
    const float4 c = cur[d];
    for (int il = threadIdx.x >> 6; il < 64; il += 4) {
        const int i = ti.y + il;
        if (i >= n || i < d) continue;
        const size_t r = 3 * (size_t)i, col = 3 * (size_t)d;
        float* m0 = M + r * ld + col;
        if (i == d) {
            for (int p = 0; p < 3; ++p)
                for (int q = 0; q < 3; ++q) m0[p * ld + q] = p == q ? 1.f : 0.f;
            continue;
        }
        const F6 D = rpy(unit_sep(c, cur[i]), a);
        m0[0] = D.xx; m0[1] = D.xy; m0[2] = D.xz;
        m0 += ld;
        m0[0] = D.xy; m0[1] = D.yy; m0[2] = D.yz;
        m0 += ld;
        m0[0] = D.xz; m0[1] = D.yz; m0[2] = D.zz;
    }
}

// Noise sum_j B_ij rforce_j for i's three rows, one wavefront per bead, then
// the Euler step.  faithful: each 3x3 block applied as the symmetric matrix
// of its lower triangle, as integrateCholesky_L reads it
// (bdhitea_kernel.cu:322-337); otherwise the factor itself.
__global__ __launch_bounds__(256) void k_chol_L(const DevJob* __restrict__ jobs, const DevJobState* __restrict__ st,
                                                const int2* __restrict__ tiles, int ntiles, int kstep) {
    const int lane = threadIdx.x & 63;
    // wavefront gw: bead (gw % 64) of tile gw / 64
    for (int gw = blockIdx.x * 4 + wave_of(); gw < ntiles * 64; gw += gridDim.x * 4) {
        const int2 td = tiles[gw >> 6];
        const DevJob& J = jobs[td.x];
        if (!(J.flags & JF_HI_EXACT)) continue;
        const long long s = st[td.x].step + kstep;
        if (s >= J.end_step) continue;
        const int n = J.n;
        const int d = td.y + (gw & 63);
        if (d >= n) continue;
        const size_t ld = J.chol_ld;
        const float* __restrict__ M = J.chol_M;
        const float* __restrict__ g = reinterpret_cast<const float*>(J.rforce);
        const bool faithful = (J.flags & JF_HI_FAITHFUL) != 0;
        const int r = 3 * d;
        float a0 = 0.f, a1 = 0.f, a2 = 0.f;
        // unrolled so that several columns' loads are in flight per lane; each
        // lane still adds its columns in order
#pragma unroll 4
        for (int c = lane; c < r + 3; c += 64) {
            const int blk = c / 3, b = c - 3 * blk;
            const float gc = g[4 * blk + b];
            float b0, b1, b2;
            if (faithful) {
                const int c0 = 3 * blk;
                // B[a][c0+b] = L[r+max(a,b)][c0+min(a,b)]
                b0 = M[(size_t)(r + b) * ld + c0];
                b1 = M[(size_t)(r + (b > 1 ? b : 1)) * ld + c0 + (b < 1 ? b : 1)];
                b2 = M[(size_t)(r + 2) * ld + c0 + b];
                if (blk == d) {  // inside the diagonal block only the lower part exists
                    b0 = M[(size_t)(r + b) * ld + c0];
                }
            } else {
                b0 = c <= r ? M[(size_t)r * ld + c] : 0.f;
                b1 = c <= r + 1 ? M[(size_t)(r + 1) * ld + c] : 0.f;
                b2 = M[(size_t)(r + 2) * ld + c];
            }
            a0 += b0 * gc;
            a1 += b1 * gc;
            a2 += b2 * gc;
        }
        // fixed-order tree reduction across the wavefront
        for (int off = 32; off > 0; off >>= 1) {
            a0 += __shfl_xor(a0, off);
            a1 += __shfl_xor(a1, off);
            a2 += __shfl_xor(a2, off);
        }
        if (lane == 0) {
            const float4 f = J.fdf[d];
            hi_finish(J, d, s, f.x + a0, f.y + a1, f.z + a2, J.coord[s & 1][d]);
        }
    }
}

// ---- blocked Cholesky -------------------------------------------------------
static constexpr int NB = 64;    // inner block: diagonal factor, panel solve
static constexpr int NB2 = kCholPanel;  // outer panel: depth of the trailing update

// The panel copy that the updates read: for every 32 columns of a panel and
// every row one 128-byte record (a cache line), the rows of a chunk one after
// another -- 32 floats (FP32), or 32 bf16 hi parts followed by the 32 lo
// parts (split-BF16).  A wavefront that reads 16 rows of a chunk reads 2 KB on
// end; from rows a kilobyte or a matrix row apart the same operands came from
// a few L2 channels at a quarter of the rate (an update of 960 columns: 19 us).
__device__ __forceinline__ size_t panel_rec(size_t mp, int chunk, size_t row) {
    return ((size_t)chunk * mp + row) * kCholRecord;
}

__device__ __forceinline__ unsigned short f2bf(float x) {  // round to nearest even
    unsigned int u = __float_as_uint(x);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}
__device__ __forceinline__ float bf2f(unsigned short h) { return __uint_as_float(((unsigned int)h) << 16); }

// The diagonal machinery below (factor and inverse of a 64x64 block, the
// panel solve with the inverse) runs in the scalar type R: FP64 for the FP32
// factorisation, FP32 for the split-BF16 one (whose trailing updates carry
// errors near 1e-6 relative; an FP32 diagonal adds ~1e-7, and halves the
// cost of the serial pivot chain and of the inverse's MFMA work).
template <int MODE>
using CholReal = typename std::conditional<MODE == SOP_CHOL_BF16X3, float, double>::type;
template <typename R>
using R4 = typename std::conditional<std::is_same<R, double>::value, f64x4, f32x4>::type;

// A lane's value from another lane of the wavefront (uniform lane index).
__device__ __forceinline__ double readlane_r(double v, int lane) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, lane);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ float readlane_r(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// 1/sqrt(p): the hardware estimate refined by one Newton step (y <- y (3 -
// p y^2) / 2).  FP64: estimate error below 2^-22, after the step near 2^-44
// -- far below the FP32 rounding of the factor it feeds; FP32: within an
// ulp or two of the FP32 value.
__device__ __forceinline__ double rsqrt_r(double p) {
    const double y = __builtin_amdgcn_rsq(p);
    return y * fma(-0.5 * p * y, y, 1.5);
}
__device__ __forceinline__ float rsqrt_r(float p) {
    const float y = __builtin_amdgcn_rsqf(p);
    return y * fmaf(-0.5f * p * y, y, 1.5f);
}

// acc += A B on the 16x16x4 MFMA of R.  Lane layout of both: A[i=l%16][k=l/16],
// B[k=l/16][j=l%16]; D row drow(l/16, v), column l%16 in register v: FP64
// interleaves the rows (l/16 + 4v), FP32 blocks them (4(l/16) + v).
__device__ __forceinline__ f64x4 mfma16(double a, double b, f64x4 acc) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16(float a, float b, f32x4 acc) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0);
}
template <typename R>
__device__ __forceinline__ int drow(int lk, int v) {
    return std::is_same<R, double>::value ? lk + 4 * v : 4 * lk + v;
}

// Four columns (4B .. 4B+3) of the diagonal factorisation, run by one
// wavefront on registers: lanes 0..15 hold the rows of the 16x16 diagonal
// sub-block, lanes 16..63 the rows below it.  The 4x4 block on the diagonal
// is read into every lane (readlane) and factored there, so that one pivot
// waits for a reciprocal square root and two multiply-adds and not for a
// round trip through the columns; then each lane substitutes its row's four
// values, and the columns to the right take the four products, with L[c][k]
// read from lane c.  The same operations, in the same order, as one column
// after another (four passes: 8 -> 4 us of a 64x64 block in FP32).  For lanes
// below the sub-block this is the forward substitution of the panel solve, so
// both run as one pass.  Lanes 0..15 accumulate scratch above their diagonal,
// which is never written back.  y[4B + k] receives 1/L[4B+k][4B+k] (uniform).
template <int B, typename R>
__device__ __forceinline__ void chol16_step(R (&v)[16], R (&y)[16]) {
    constexpr int J = 4 * B;
    R d[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int k = 0; k <= i; ++k) d[i][k] = readlane_r(v[J + k], J + i);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        y[J + k] = rsqrt_r(d[k][k]);
#pragma unroll
        for (int i = k + 1; i < 4; ++i) d[i][k] *= y[J + k];
#pragma unroll
        for (int i = k + 1; i < 4; ++i)
#pragma unroll
            for (int q = k + 1; q <= i; ++q) d[i][q] = fma(-d[i][k], d[q][k], d[i][q]);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
#pragma unroll
        for (int q = 0; q < k; ++q) v[J + k] = fma(-v[J + q], d[k][q], v[J + k]);
        v[J + k] *= y[J + k];  // lane J+k: L[J+k][J+k] = p / sqrt(p)
    }
    if constexpr (B + 1 < 4) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            // all of a column's L[c][k] read before they are used: read and
            // used one by one, each product would wait for its own read
            R lc[12];
#pragma unroll
            for (int c = J + 4; c < 16; ++c) lc[c - 4] = readlane_r(v[J + k], c);
#pragma unroll
            for (int c = J + 4; c < 16; ++c) asm volatile("" : "+s"(lc[c - 4]));
#pragma unroll
            for (int c = J + 4; c < 16; ++c) v[c] = fma(-v[J + k], lc[c - 4], v[c]);
        }
        chol16_step<B + 1>(v, y);
    }
}

static constexpr int kCholThreads = 512;  // a step's workgroup: eight wavefronts, two per SIMD
static constexpr int LDS_ROW = NB + 1;  // row stride of the block being factored
// Row stride of the transposed blocks (Li^T): 16-byte rows, and the four row
// groups of an MFMA operand, four rows apart (load_solve_rows), read in
// distinct bank ranges, in either type.
static constexpr int LDT = NB + 4;

// Column block K of the 64x64 block s (rows 16K..63), factored in registers
// by wavefront 0: lane r holds row 16K + r (lanes 0..15 the diagonal sub-block,
// the others the rows below, forward-substituted in the same pass; lanes past
// row 63 keep zeros).  Wavefront 1 runs the same pass with the rows of the
// identity in lanes 16..31: forward-substituted, e_i becomes row i of the
// transposed inverse of the sub-block, so the inverse comes with the factor
// (a substitution of its own took longer than the pass).  pass_load reads the
// registers; a barrier later, pass_store follows the factorisation.  Lanes
// 0..15 write their scratch above the diagonal back, where nothing reads it.
template <typename R>
__device__ __forceinline__ void pass_load(const R (*s)[LDS_ROW], R (&v)[16], int K) {
    const int r = threadIdx.x & 63, w = wave_of();
    const int q0 = 16 * K;
    const bool row = r < (w == 0 ? NB - q0 : 16);
#pragma unroll
    for (int c = 0; c < 16; ++c) {
        const R e = s[row ? q0 + r : q0][q0 + c];
        v[c] = row && (r >= 16 || c <= r) ? e : w != 0 && r - 16 == c ? R(1) : R(0);
    }
}
template <typename R>
__device__ __forceinline__ void pass_store(R (*s)[LDS_ROW], R* __restrict__ LiT, const R (&v)[16], int K) {
    const int r = threadIdx.x & 63, w = wave_of();
    const int q0 = 16 * K;
    if (w == 0) {
        if (r < NB - q0) {
#pragma unroll
            for (int c = 0; c < 16; ++c) s[q0 + r][q0 + c] = v[c];
        }
    } else if (r >= 16 && r < 32) {
#pragma unroll
        for (int c = 0; c < 16; ++c) LiT[(q0 + r - 16) * LDT + q0 + c] = v[c];
    }
}

// C_IJ -= L_IK L_JK^T for the 16x16 tile (I, J) of s on MFMA, one wavefront.
template <typename R>
__device__ __forceinline__ void rank16_tile(R (*s)[LDS_ROW], int I, int J, int K) {
    const int l = threadIdx.x & 63, lr = l & 15, lk = l >> 4;
    R4<R> acc;
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[v] = s[16 * I + drow<R>(lk, v)][16 * J + lr];
#pragma unroll
    for (int k0 = 0; k0 < 16; k0 += 4)
        acc = mfma16(-s[16 * I + lr][16 * K + k0 + lk], s[16 * J + lr][16 * K + k0 + lk], acc);
#pragma unroll
    for (int v = 0; v < 4; ++v) s[16 * I + drow<R>(lk, v)][16 * J + lr] = acc[v];
}

// Off-diagonal 16x16 block (I, J) of the inverse, J < I, on MFMA by one
// wavefront, in two halves: T = sum_{J<=K<I} L_IK Li_KJ into the
// wavefront's LDS tile (needs the rows J..I-1 of the inverse), then
// Li_IJ = -Li_II T (needs Li_II).
template <typename R>
__device__ __forceinline__ void inv_sum16(const R (*s)[LDS_ROW], const R* __restrict__ LiT, R (*T)[17], int I,
                                          int J) {
    const int l = threadIdx.x & 63, lr = l & 15, lk = l >> 4;
    R4<R> acc = {R(0), R(0), R(0), R(0)};
    for (int k0 = 0; k0 < 16 * (I - J); k0 += 4)
        acc = mfma16(s[16 * I + lr][16 * J + k0 + lk], LiT[(16 * J + lr) * LDT + 16 * J + k0 + lk], acc);
#pragma unroll
    for (int v = 0; v < 4; ++v) T[drow<R>(lk, v)][lr] = acc[v];
}
template <typename R>
__device__ __forceinline__ void inv_apply16(R* __restrict__ LiT, const R (*T)[17], int I, int J) {
    const int l = threadIdx.x & 63, lr = l & 15, lk = l >> 4;
    R4<R> li = {R(0), R(0), R(0), R(0)};
#pragma unroll
    for (int k0 = 0; k0 < 16; k0 += 4) li = mfma16(-LiT[(16 * I + k0 + lk) * LDT + 16 * I + lr], T[k0 + lk][lr], li);
#pragma unroll
    for (int v = 0; v < 4; ++v) LiT[(16 * J + lr) * LDT + 16 * I + drow<R>(lk, v)] = li[v];
}

// Factor the 64x64 block s (lower triangle, row-major) in place and form
// the inverse of the factor, transposed, in LiT (zero above its diagonal),
// with the workgroup's eight wavefronts, in a round per 16-column block K:
// the previous block's rank-16 update of the tiles right of it, a tile per
// wavefront, beside the products that complete row K-1 of the inverse; then
// the factorisation of block K with its diagonal block's inverse (wavefronts 0
// and 1, see pass_load), beside the sums of row K's blocks left of the
// diagonal.  So the inverse trails the factor by one product.
template <typename R>
__device__ __forceinline__ void potrf_inv64(R (*s)[LDS_ROW], R* __restrict__ LiT, R (*T)[16][17]) {
    const int w = wave_of();
    for (int e = threadIdx.x; e < NB * LDT; e += kCholThreads) LiT[e] = R(0);
#pragma unroll 1
    for (int K = 0; K < NB / 16; ++K) {  // one copy of the code: its first pass fetches it
        if (K > 0) {
            // tiles (I, J), K <= J <= I, from the last: (3,3), (3,2), (2,2),
            // (3,1), (2,1), (1,1)
            if (w < (4 - K) * (5 - K) / 2)
                rank16_tile(s, (0x123233 >> (4 * w)) & 15, (0x111223 >> (4 * w)) & 15, K - 1);
            else if (w >= 6 && w - 6 < K - 1)  // row K-1 of the inverse, left of its diagonal
                inv_apply16(LiT, T[w - 6], K - 1, w - 6);
            __syncthreads();
        }
        R v[16];
        if (w < 2) pass_load(s, v, K);
        __syncthreads();
        if (w < 2) {
            R y[16];
            chol16_step<0>(v, y);
            pass_store(s, LiT, v, K);
        } else if (w - 2 < K) {
            inv_sum16(s, LiT, T[w - 2], K, w - 2);
        }
        __syncthreads();
    }
    constexpr int RL = NB / 16 - 1;  // the inverse's last row
    if (w < RL) inv_apply16(LiT, T[w], RL, w);
    __syncthreads();
}

// M[row][col] -= v over the lower triangle, rows and columns below mp, for N
// elements of a lane.  All loads are issued, from clamped addresses, before
// the first store: each behind its own condition, they ran one memory round
// trip after another (64 of them took 25 of a 128x128 tile's 40 us, 128 took
// 80 of a 256x256 tile's 118).
template <int N>
__device__ __forceinline__ void sub_store(float* __restrict__ M, size_t ld, int mp, const int (&row)[N],
                                          const int (&col)[N], const float (&v)[N]) {
    float c[N];
#pragma unroll
    for (int q = 0; q < N; ++q) c[q] = M[(size_t)min(row[q], mp - 1) * ld + min(col[q], mp - 1)];
#pragma unroll
    for (int q = 0; q < N; ++q) c[q] -= v[q];
#pragma unroll
    for (int q = 0; q < N; ++q)
        if (row[q] < mp && col[q] < mp && col[q] <= row[q]) M[(size_t)row[q] * ld + col[q]] = c[q];
}

// Update after an outer panel: C -= P_r P_c^T over the panel copy's kw columns
// for one TM x TN tile of the lower triangle (rows from r0, columns from c0;
// rows at or beyond mp are computed from a clamped row and not written), by
// WM x WN wavefronts of 64 rows each.  Per 32-column chunk the tile's row and
// column records (128 bytes a row, panel_rec) are staged in LDS -- 144 bytes
// apart, so that the 16 rows of an MFMA operand fall in distinct banks -- and
// multiplied from there: split-BF16 hi hi + hi lo + lo hi on 16x16x32 MFMA,
// FP32 on 16x16x4.  Two LDS buffers and D chunks in registers: while chunk k
// is multiplied, chunk k+1 is written to the other buffer and chunks k+2 ..
// k+1+D are on their way; one barrier per chunk.  Bound by the operands: a CU's
// vector loads bring 37 GB/s from L2 or beyond, a 256x256 tile's 1 MB 28 us,
// its split-BF16 products 23 us (one buffer, two barriers and the next chunk
// only took 59 us).
static constexpr int kLdsRec = kCholRecord + 16;
template <int MODE, int TM, int TN, int WM, int WN, int D>
__device__ __forceinline__ void update_tile(float* __restrict__ M, size_t ld, int mp, int kw,
                                            const char* __restrict__ pan, int r0, int c0, char* __restrict__ lds) {
    constexpr int TH = 64 * WM * WN, BUF = (TM + TN) * kLdsRec;
    constexpr int UN = (TM + TN) * (kCholRecord / 16) / TH;  // 16-byte units per thread and chunk
    constexpr int NI = TM / WM / 16, NJ = TN / WN / 16;      // 16x16 tiles per wavefront
    static_assert(UN * TH * 16 == (TM + TN) * kCholRecord, "the threads divide a chunk evenly");
    using V = typename std::conditional<MODE == SOP_CHOL_BF16X3, bf16x8, f32x4>::type;
    const int tid = threadIdx.x, l = tid & 63, w = wave_of(), wr = (w / WN) * (TM / WM), wc = (w % WN) * (TN / WN);
    const int lr = l & 15, lk = l >> 4;
    // the thread's units: row (of the row, then the column operand) and 16-byte unit
    unsigned src[UN], dst[UN];
#pragma unroll
    for (int i = 0; i < UN; ++i) {
        const int e = tid + TH * i, r = e / 8, u = e % 8;
        const int g = min(r < TM ? r0 + r : c0 + r - TM, mp - 1);
        src[i] = (unsigned)g * kCholRecord + 16 * u;
        dst[i] = r * kLdsRec + 16 * u;
    }
    typedef const __attribute__((address_space(1))) char* gptr;
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    const int nch = kw / 32;
    u32x4 v[D][UN];
    auto fetch = [&](u32x4 (&x)[UN], int k) {
        const gptr p = (gptr)pan + (size_t)min(k, nch - 1) * mp * kCholRecord;
#pragma unroll
        for (int i = 0; i < UN; ++i) x[i] = *reinterpret_cast<const __attribute__((address_space(1))) u32x4*>(p + src[i]);
    };
    auto stash = [&](const u32x4 (&x)[UN], int buf) {
#pragma unroll
        for (int i = 0; i < UN; ++i) *reinterpret_cast<u32x4*>(lds + buf * BUF + dst[i]) = x[i];
    };
    f32x4 acc[NI][NJ];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    fetch(v[0], 0);
    stash(v[0], 0);
#pragma unroll
    for (int d = 0; d < D; ++d) fetch(v[d], 1 + d);
    __syncthreads();
    auto at = [&](int buf, int r, int half) {
        return *reinterpret_cast<const V*>(lds + buf * BUF + r * kLdsRec + (kCholRecord / 2) * half + 16 * lk);
    };
    auto chunk = [&](int k, u32x4 (&x)[UN]) {
        stash(x, (k + 1) & 1);
        fetch(x, k + 1 + D);
        __builtin_amdgcn_sched_barrier(0);
        const int buf = k & 1;
        V a0[NI], a1[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            a0[i] = at(buf, wr + 16 * i + lr, 0);
            a1[i] = at(buf, wr + 16 * i + lr, 1);
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const V b0 = at(buf, TM + wc + 16 * j + lr, 0), b1 = at(buf, TM + wc + 16 * j + lr, 1);
            if constexpr (MODE == SOP_CHOL_BF16X3) {
#pragma unroll
                for (int i = 0; i < NI; ++i)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0[i], b0, acc[i][j], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < NI; ++i)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0[i], b1, acc[i][j], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < NI; ++i)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[i], b0, acc[i][j], 0, 0, 0);
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int i = 0; i < NI; ++i)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[i][c], b0[c], acc[i][j], 0, 0, 0);
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int i = 0; i < NI; ++i)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1[i][c], b1[c], acc[i][j], 0, 0, 0);
            }
        }
        __syncthreads();
    };
    // kw is a multiple of 64: an even number of chunks.  The narrow tiles
    // (registers to spare) sum kPart columns at a time and add the parts: one
    // chain of 512 FP32 additions left the FP32 factor's error 8 to 30 % above
    // that of the shorter chains of a step's wavefronts, in parts it is below
    // (order 4,001: 1.29e-6, 1.22e-6 and 1.11e-6 of the factor's norm)
    constexpr bool kParts = NI * NJ <= 8;
    constexpr int kPart = 128;
    f32x4 sum[NI][NJ];
    for (int k = 0; k < nch; k += 2) {
        chunk(k, v[0]);
        chunk(k + 1, v[D - 1]);
        if (kParts && ((k + 2) % (kPart / 32) == 0 || k + 2 == nch)) {
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    sum[i][j] = k + 2 > kPart / 32 ? sum[i][j] + acc[i][j] : acc[i][j];
                    acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
        }
    }
    if constexpr (kParts) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[i][j] = sum[i][j];
    }
    // C -= acc: D rows 4(l/16) + q, column l%16 of each 16x16 tile
    constexpr int NB_ = 32;  // elements of a lane at a time
#pragma unroll
    for (int h = 0; h < NI * NJ * 4; h += NB_) {
        int row[NB_], col[NB_];
        float x[NB_];
#pragma unroll
        for (int e = 0; e < NB_; ++e) {
            const int t = (h + e) / 4, i = t / NJ, j = t % NJ, q = e % 4;
            row[e] = r0 + wr + 16 * i + 4 * lk + q;
            col[e] = c0 + wc + 16 * j + lr;
            x[e] = acc[i][j][q];
        }
        sub_store(M, ld, mp, row, col, x);
    }
}

// Regions [s, mp) x [s, mp): 256x256 tiles by eight wavefronts, one workgroup
// per CU, numbered over the lower triangle row by row and dealt to the XCDs in
// contiguous ranges (workgroup i runs on XCD i % 8), so the tiles an XCD holds
// at once share their row panels in its L2.
static constexpr int BT = 256;
constexpr int kXcds = 8;
template <int MODE>
__global__ __launch_bounds__(512) void k_update_big(float* __restrict__ M, size_t ld, int s, int mp, int kw, int ntr,
                                                    const char* __restrict__ pan) {
    __shared__ __attribute__((aligned(16))) char lds[2 * 2 * BT * kLdsRec];
    const int ntile = ntr * (ntr + 1) / 2, per = (ntile + kXcds - 1) / kXcds;
    const int t = (int)(blockIdx.x % kXcds) * per + (int)(blockIdx.x / kXcds);
    if ((int)(blockIdx.x / kXcds) >= per || t >= ntile) return;
    int bi = (int)((sqrtf(8.0f * (float)t + 1.0f) - 1.0f) * 0.5f);
    while (bi * (bi + 1) / 2 > t) --bi;
    while ((bi + 1) * (bi + 2) / 2 <= t) ++bi;
    const int bj = t - bi * (bi + 1) / 2;
    update_tile<MODE, BT, BT, 4, 2, 1>(M, ld, mp, kw, pan, s + BT * bi, s + BT * bj, lds);
}

// Tile (blockIdx.x, blockIdx.y) of the lower triangle from row and column s
// on: TM x TN tiles by four wavefronts.
template <int MODE, int TM, int TN>
__global__ __launch_bounds__(256, 2) void k_update(float* __restrict__ M, size_t ld, int s, int mp, int kw,
                                                   const char* __restrict__ pan) {
    __shared__ __attribute__((aligned(16))) char lds[2 * (TM + TN) * kLdsRec];
    const int r0 = s + (int)blockIdx.x * TM, c0 = s + (int)blockIdx.y * TN;
    if (c0 >= r0 + TM || c0 >= mp) return;  // wholly above the diagonal, or past the last column
    update_tile<MODE, TM, TN, 2, 2, 2>(M, ld, mp, kw, pan, r0, c0, lds);
}

// ---- the factorisation by fused 64-column steps -----------------------------
// Within an outer panel (columns c0 .. c0+kw-1, nb = kw/64 column blocks),
// step j (0 <= j <= nb) is one launch over the 64-row blocks g >= c0/64 + j
// (workgroup x serves g = c0/64 + j + x; d = c0/64 + j is the step's
// diagonal block):
//  (1) for j >= 1, each row block's solve against column block j-1:
//      X_g = B_g Li^T with B_g the block as the previous step left it and
//      Li^T the inverse of L_{j-1,j-1} (accumulated in CholReal), written to M
//      and to the panel copy;
//  (2) for j < nb, column block j of each row block minus the products of
//      this panel's columns 0 .. 64j-1, on MFMA:
//      B_g = A_gj - sum_k X_gk X_dk^T.  Workgroup 0 (g = d) factors B in
//      CholReal into L_jj and its inverse; the others store B for step j+1.
// Every workgroup forms X_d for (2) itself (the diagonal row block's solve,
// the same arithmetic as workgroup 0's), so no workgroup waits for another.
// Lookahead: the diagonal workgroup's chain (solve, update, factor, inverse)
// is the step's critical path, so the long part of its update -- every
// column left of j-1 -- is formed one step early: while step j-1 runs, one
// extra workgroup solves row block d for column block j-2 itself and forms
// P = A_dd - sum_{k < j-1} X_dk X_dk^T into a step buffer; step j's
// diagonal workgroup then only subtracts X_d,j-1 X_d,j-1^T (64 columns)
// before it factors.  The panel's first step has no such block and forms
// the whole sum.
// A finished panel's update of the next panel's columns runs between the two
// panels' steps, that of the rest of the trailing matrix on the second stream
// beside the next panel's steps, both by the wide MFMA kernels.  (Folded into
// the next panel's steps, the former made each of them read 128 KB of panel
// columns per row block again: at the 37 GB/s a CU's vector loads reach, the
// row blocks took 20-26 us a step and not the diagonal workgroup's 14.)
static constexpr int XS = NB + 4;  // row stride of the FP32 X blocks in LDS (16-byte rows)

struct CholStep {
    float* M;
    size_t ld;
    int mp;
    int c0, kw;                      // this outer panel
    int j;                           // step 0 .. nb
    const void* li_in;               // Li^T of column block j-1 (64 x 64 CholReal, row a = column a of Li)
    void* li_out;                    // Li^T of column block j
    const float* b_in;               // B of column block j-1, mp x 64 by row
    float* b_out;                    // B of column block j
    const float* p_in;               // the diagonal block's P formed by the previous step (j >= 1)
    float* p_out;                    // the next diagonal block's P (when look)
    int look;                        // 1: an extra workgroup forms P for step j+1
    char* pan;                       // this panel's copy (panel_rec)
};

// The 64 values of B a lane feeds the solve's MFMAs, four 16-byte loads: in
// step 4m + i of the sum over t, lane group l/16 takes t = 16m + 4(l/16) + i
// (B[16(w%4) + l%16][t]; B is 64 x 64 FP32, rows r0.. of a row-major mp x 64
// buffer).
__device__ __forceinline__ void load_solve_rows(const float* __restrict__ b, size_t r0, float4 (&bv)[4]) {
    const int l = threadIdx.x & 63, w = wave_of() & 3;
    const float* __restrict__ row = b + (r0 + 16 * w + (l & 15)) * NB + 4 * (l >> 4);
#pragma unroll
    for (int m = 0; m < 4; ++m) bv[m] = *reinterpret_cast<const float4*>(row + 16 * m);
}

// X = B Li^T for one 64x64 block on MFMA in CholReal (B from
// load_solve_rows, LiT[t*LDT + c] = Li[c][t], zero for t > c), to Xs (LDS,
// row stride XS) and, when `out`, to M (rows r0.., columns col0..) and the
// panel copy (columns pcol0.. of the panel).  Wavefront w forms rows 16(w%4) .. +15 of the
// output blocks jb (columns 16jb..) in JBS (a bit each); block jb sums
// t < 16(jb+1) only, where Li^T is not zero.
template <int MODE, int JBS>
__device__ __forceinline__ void solve_block(const float4 (&bv)[4], const CholReal<MODE>* __restrict__ LiT,
                                            float* __restrict__ Xs, bool out, float* __restrict__ M, size_t ld,
                                            size_t mp, size_t r0, size_t col0, char* __restrict__ pan,
                                            int pcol0) {
    using R = CholReal<MODE>;
    const int l = threadIdx.x & 63, w = wave_of() & 3, lr = l & 15, lk = l >> 4;
    R4<R> acc[4];
#pragma unroll
    for (int jb = 0; jb < 4; ++jb) acc[jb] = R4<R>{R(0), R(0), R(0), R(0)};
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const float av[4] = {bv[m].x, bv[m].y, bv[m].z, bv[m].w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int jb = 0; jb < 4; ++jb)
                if (((JBS >> jb) & 1) && m <= jb)
                    acc[jb] = mfma16((R)av[i], LiT[(16 * m + 4 * lk + i) * LDT + 16 * jb + lr], acc[jb]);
    }
#pragma unroll
    for (int jb = 0; jb < 4; ++jb)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            if (!((JBS >> jb) & 1)) continue;
            const int row = 16 * w + drow<R>(lk, v), c = 16 * jb + lr;
            const float x = (float)acc[jb][v];
            Xs[row * XS + c] = x;
            if (!out) continue;
            M[(r0 + row) * ld + col0 + c] = x;
            char* const rec = pan + panel_rec(mp, (pcol0 + 16 * jb) / 32, r0 + row);
            const int e = 16 * (jb & 1) + lr;
            if constexpr (MODE == SOP_CHOL_BF16X3) {
                const unsigned short h = f2bf(x);
                reinterpret_cast<unsigned short*>(rec)[e] = h;
                reinterpret_cast<unsigned short*>(rec)[32 + e] = f2bf(x - bf2f(h));
            } else {
                reinterpret_cast<float*>(rec)[e] = x;
            }
        }
}

// acc += X_g X_d^T over this wavefront's share of the panel's columns left of
// column block j-1, 64(j-1) of them.  Wavefront w forms the half
// h = w/4 of the 64x64 block (rows 0..63, columns 32h .. 32h+31: 4x2 MFMA
// tiles) from the 32-column chunks w%4, w%4 + 4, .., the next chunk's operands
// in flight while one is multiplied.
template <int MODE>
__device__ __forceinline__ void mfma_split(f32x4 (&acc)[4][2], const CholStep& a, size_t rg, size_t rd) {
    const int l = threadIdx.x & 63, w = wave_of(), kq = w & 3, h = w >> 2, lr = l & 15, lk = l >> 4;
    const int n = (a.j >= 2 ? NB * (a.j - 1) : 0) / 32;
    typedef const __attribute__((address_space(1))) char* gptr;
    // byte offsets of the lane's rows within a chunk (128 bytes a row: 32 bits
    // hold 33 million rows); lane group l/16 reads 16 bytes of each half record
    unsigned ao[4], bo[2];
#pragma unroll
    for (int b = 0; b < 4; ++b) ao[b] = (unsigned)(rg + 16 * b + lr) * kCholRecord + 16 * lk;
#pragma unroll
    for (int b = 0; b < 2; ++b) bo[b] = (unsigned)(rd + 32 * h + 16 * b + lr) * kCholRecord + 16 * lk;
    auto chunk = [&](int c) { return (gptr)a.pan + (size_t)c * a.mp * kCholRecord; };
    // the two halves of a record: split-BF16 hi and lo of k = 8(l/16) .. +7;
    // FP32 k = 4(l/16) .. +3 and 16 further on, MFMA step i taking component i
    using V = typename std::conditional<MODE == SOP_CHOL_BF16X3, bf16x8, f32x4>::type;
    auto at = [](gptr p, unsigned off) {
        return *reinterpret_cast<const __attribute__((address_space(1))) V*>(p + off);
    };
    struct Ops {
        V a0[4], a1[4], b0[2], b1[2];
    };
    auto load = [&](Ops& o, int c) {
        const gptr p = chunk(c);
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            o.a0[b] = at(p, ao[b]);
            o.a1[b] = at(p + kCholRecord / 2, ao[b]);
        }
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            o.b0[b] = at(p, bo[b]);
            o.b1[b] = at(p + kCholRecord / 2, bo[b]);
        }
    };
    auto mma = [&](const Ops& o) {
        if constexpr (MODE == SOP_CHOL_BF16X3) {
#pragma unroll
            for (int bi = 0; bi < 4; ++bi)
#pragma unroll
                for (int bj = 0; bj < 2; ++bj)
                    acc[bi][bj] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(o.a0[bi], o.b0[bj], acc[bi][bj], 0, 0, 0);
#pragma unroll
            for (int bi = 0; bi < 4; ++bi)
#pragma unroll
                for (int bj = 0; bj < 2; ++bj)
                    acc[bi][bj] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(o.a0[bi], o.b1[bj], acc[bi][bj], 0, 0, 0);
#pragma unroll
            for (int bi = 0; bi < 4; ++bi)
#pragma unroll
                for (int bj = 0; bj < 2; ++bj)
                    acc[bi][bj] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(o.a1[bi], o.b0[bj], acc[bi][bj], 0, 0, 0);
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int bi = 0; bi < 4; ++bi)
#pragma unroll
                    for (int bj = 0; bj < 2; ++bj)
                        acc[bi][bj] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.a0[bi][i], o.b0[bj][i], acc[bi][bj], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int bi = 0; bi < 4; ++bi)
#pragma unroll
                    for (int bj = 0; bj < 2; ++bj)
                        acc[bi][bj] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.a1[bi][i], o.b1[bj][i], acc[bi][bj], 0, 0, 0);
        }
    };
    // loads without branches (a last chunk again past the end) and held in
    // place: moved or merged by the compiler, the products of one chunk waited
    // for the next one's operands
    if (kq >= n) return;
    Ops o0, o1;
    load(o0, kq);
    for (int c = kq; c < n; c += 8) {
        load(o1, min(c + 4, n - 1));
        __builtin_amdgcn_sched_barrier(0);
        mma(o0);
        __builtin_amdgcn_sched_barrier(0);
        if (c + 4 >= n) break;
        load(o0, min(c + 8, n - 1));
        __builtin_amdgcn_sched_barrier(0);
        mma(o1);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The same over the 64 columns of the X blocks just solved, from LDS; in
// split-BF16 mode each value is split as the panel copy holds it.  Wavefront w
// forms tiles 2(w/4) and the next one of tile row w%4.
template <int MODE>
__device__ __forceinline__ void mfma_lds(f32x4 (&acc)[2], const float* __restrict__ Xg, const float* __restrict__ Xd) {
    const int l = threadIdx.x & 63, w = wave_of() & 3, t0 = 2 * (wave_of() >> 2), lr = l & 15;
    if constexpr (MODE == SOP_CHOL_BF16X3) {
        const int lk = (l >> 4) * 8;
#pragma unroll
        for (int kc = 0; kc < NB; kc += 32) {
            bf16x8 ah, al, bh[2], bl[2];
            const float* a = Xg + (16 * w + lr) * XS + kc + lk;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const unsigned short h = f2bf(a[e]);
                ah[e] = (short)h;
                al[e] = (short)f2bf(a[e] - bf2f(h));
            }
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const float* b = Xd + (16 * (t0 + t) + lr) * XS + kc + lk;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const unsigned short h = f2bf(b[e]);
                    bh[t][e] = (short)h;
                    bl[t][e] = (short)f2bf(b[e] - bf2f(h));
                }
            }
#pragma unroll
            for (int t = 0; t < 2; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh[t], acc[t], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < 2; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl[t], acc[t], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < 2; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh[t], acc[t], 0, 0, 0);
        }
    } else {
        const int lg = l >> 4;  // k = kc+4g .. kc+4g+3
#pragma unroll
        for (int kc = 0; kc < NB; kc += 16) {
            const float4 a = *reinterpret_cast<const float4*>(Xg + (16 * w + lr) * XS + kc + 4 * lg);
            float4 b[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) b[t] = *reinterpret_cast<const float4*>(Xd + (16 * (t0 + t) + lr) * XS + kc + 4 * lg);
#pragma unroll
            for (int t = 0; t < 2; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b[t].x, acc[t], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < 2; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b[t].y, acc[t], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < 2; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b[t].z, acc[t], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < 2; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b[t].w, acc[t], 0, 0, 0);
        }
    }
}

// Eight wavefronts: with four, one per SIMD, the row blocks' long update
// waited for its operands and outlasted the diagonal workgroup's chain (row
// blocks 20-25 us a step, the diagonal 18, while the update still reached over
// the panel before as well, up to 960 columns; now it is at most 384).
template <int MODE>
__global__ __launch_bounds__(kCholThreads) void k_chol_step(CholStep a) {
    using R = CholReal<MODE>;
    // SA: the block factored (R, row stride LDS_ROW), and the partial sums of
    // the update (FP32); LiT: Li^T in, then the new inverse (R, stride LDT),
    // and partial sums; both sized for the larger use
    constexpr int kSA = NB * LDT;  // doubles
    __shared__ __attribute__((aligned(16))) double SA[kSA];
    __shared__ __attribute__((aligned(16))) double LiTraw[kSA];
    __shared__ __attribute__((aligned(16))) float Xg[NB * XS];
    __shared__ __attribute__((aligned(16))) float Xd[NB * XS];
    __shared__ R T[3][16][17];
    R* const LiT = reinterpret_cast<R*>(LiTraw);
    static_assert(NB * LDS_ROW * sizeof(R) <= sizeof(SA), "the factored block fits its buffer");
    static_assert(2 * NB * NB * sizeof(float) <= sizeof(SA), "two wavefronts' partial blocks fit a buffer");
    const int tid = threadIdx.x;
    const int nb = a.kw / NB, j = a.j;
    // workgroup 0: the diagonal block; 1 (when a.look): the lookahead, which
    // serves row block d+1; then the row blocks d+1, d+2, ...
    const bool look = a.look && blockIdx.x == 1;
    const int x = look ? 1 : (int)blockIdx.x - (a.look && blockIdx.x > 1 ? 1 : 0);
    const size_t rd = (size_t)a.c0 + (size_t)NB * j;  // first row of the diagonal block d
    const size_t rg = rd + (size_t)NB * x;             // first row of this workgroup's block g
    const bool update = j < nb;
    const bool diag_p = x == 0 && j >= 1;              // the diagonal block arrives as P
    const bool need_d = update && x != 0 && !look;     // X_d too
    const int l = tid & 63, w = wave_of(), w4 = w & 3, half = w >> 2;
    // the block this workgroup updates: column block j (rows rg), or for the
    // lookahead the next diagonal block (rows and columns rg)
    const size_t cj = look ? rg : rd;
    // every global read first, so their latencies overlap: this row block of
    // column block j (or P), the B rows of the solves, the inverse Li^T.
    // Wavefront w holds tiles t = 2(w/4), 2(w/4)+1 of tile row w%4.
    float mblk[2][4];
    float4 bv[4];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int row = 16 * w4 + 4 * (l >> 4) + q, c = 16 * (2 * half + t) + (l & 15);
            mblk[t][q] = !update ? 0.f : diag_p ? a.p_in[row * NB + c] : a.M[(rg + row) * a.ld + cj + c];
        }
    if (j >= 1) {
        load_solve_rows(a.b_in, need_d && half ? rd : rg, bv);
        {  // Li^T: 16-byte loads, all in flight before the LDS stores
            using V = typename std::conditional<std::is_same<R, double>::value, double2, float4>::type;
            constexpr int EPV = 16 / sizeof(R), NV = NB * NB / (kCholThreads * EPV);
            const V* __restrict__ src = reinterpret_cast<const V*>(a.li_in);
            V lv[NV];
#pragma unroll
            for (int k = 0; k < NV; ++k) lv[k] = src[tid + kCholThreads * k];
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                const int e = EPV * (tid + kCholThreads * k);  // e .. e+EPV-1 in the same row
                *reinterpret_cast<V*>(LiT + (e >> 6) * LDT + (e & 63)) = lv[k];
            }
        }
        __syncthreads();
        const int pcol = NB * (j - 1);  // column block j-1 within the panel
        // with X_d to form as well, half the wavefronts solve each; else the
        // halves share the output blocks (1 + 4 and 2 + 3 sixteenths of work).
        // The lookahead's rows are written by the workgroup that serves them.
        if (need_d) {
            if (half)
                solve_block<MODE, 15>(bv, LiT, Xd, false, a.M, a.ld, a.mp, rd, a.c0 + pcol, a.pan, pcol);
            else
                solve_block<MODE, 15>(bv, LiT, Xg, true, a.M, a.ld, a.mp, rg, a.c0 + pcol, a.pan, pcol);
        } else if (half) {
            solve_block<MODE, 6>(bv, LiT, Xg, !look, a.M, a.ld, a.mp, rg, a.c0 + pcol, a.pan, pcol);
        } else {
            solve_block<MODE, 9>(bv, LiT, Xg, !look, a.M, a.ld, a.mp, rg, a.c0 + pcol, a.pan, pcol);
        }
    }
    if (!update) return;
    __syncthreads();  // X blocks complete; SA and LiT are free
    f32x4 acc[2];
    if (diag_p) {
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    } else {
        // the columns left of j-1, K split over the wavefronts: the partial
        // blocks are summed through LDS in wavefront order
        f32x4 part[4][2];
#pragma unroll
        for (int bi = 0; bi < 4; ++bi)
#pragma unroll
            for (int bj = 0; bj < 2; ++bj) part[bi][bj] = f32x4{0.f, 0.f, 0.f, 0.f};
        mfma_split<MODE>(part, a, rg, cj);
        // partial block of wavefronts (kq, half): half a 64x64 block, tile by
        // tile with a lane's four values together
        auto at = [&](int kq, int tile) {
            float* const buf = kq < 2 ? reinterpret_cast<float*>(SA) : reinterpret_cast<float*>(LiTraw);
            return reinterpret_cast<f32x4*>(buf) + (size_t)((kq & 1) * 2 + half) * 512 + 64 * tile + l;
        };
#pragma unroll
        for (int bi = 0; bi < 4; ++bi)
#pragma unroll
            for (int bj = 0; bj < 2; ++bj) *at(w4, 2 * bi + bj) = part[bi][bj];
        __syncthreads();
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int e = 2 * w4 + t;
            acc[t] = ((*at(0, e) + *at(1, e)) + *at(2, e)) + *at(3, e);
        }
        __syncthreads();  // SA and LiT are reused below
    }
    if (j >= 1) mfma_lds<MODE>(acc, Xg, x == 0 || look ? Xg : Xd);
    R(*S)[LDS_ROW] = reinterpret_cast<R(*)[LDS_ROW]>(SA);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int row = 16 * w4 + 4 * (l >> 4) + q, c = 16 * (2 * half + t) + (l & 15);
            const float b = mblk[t][q] - acc[t][q];
            if (look)
                a.p_out[row * NB + c] = b;
            else if (x == 0)
                S[row][c] = (R)b;
            else
                a.b_out[(rg + row) * NB + c] = b;
        }
    if (x != 0 || look) return;
    __syncthreads();
    potrf_inv64(S, LiT, T);
#pragma unroll
    for (int k = 0; k < NB * NB / kCholThreads; ++k) {
        const int e = tid + kCholThreads * k, r = e / NB, c = e % NB;
        if (c <= r) a.M[(rd + r) * a.ld + rd + c] = (float)S[r][c];
    }
    {  // 16-byte LDS reads, then the stores
        using V = typename std::conditional<std::is_same<R, double>::value, double2, float4>::type;
        constexpr int EPV = 16 / sizeof(R), NV = NB * NB / (kCholThreads * EPV);
        V lv[NV];
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const int e = EPV * (tid + kCholThreads * k);
            lv[k] = *reinterpret_cast<const V*>(LiT + (e >> 6) * LDT + (e & 63));
        }
        V* __restrict__ dst = reinterpret_cast<V*>(a.li_out);
#pragma unroll
        for (int k = 0; k < NV; ++k) dst[tid + kCholThreads * k] = lv[k];
    }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------

// The kernel for (B, C) = cfg over `ntiles` tiles.
#define SOP_HI_LAUNCH(kernel, cfg, ntiles, stream, ...)                                                             \
    do {                                                                                                            \
        const dim3 g((ntiles) * (64 / (cfg).beads)), b(64 * (cfg).beads);                                           \
        if ((cfg).beads == 4) hipLaunchKernelGGL((kernel<4, 256>), g, b, 0, stream, __VA_ARGS__);                   \
        else if ((cfg).beads == 16) hipLaunchKernelGGL((kernel<16, 256>), g, b, 0, stream, __VA_ARGS__);            \
        else if ((cfg).chunk == 256) hipLaunchKernelGGL((kernel<8, 256>), g, b, 0, stream, __VA_ARGS__);            \
        else hipLaunchKernelGGL((kernel<8, 128>), g, b, 0, stream, __VA_ARGS__);                                    \
    } while (0)

hipError_t launch_hi_tea_update(const DevJob* jobs, DevJobState* st, const int2* tiles, int ntiles, int njobs,
                                hipStream_t stream) {
    const HiConfig cfg = hi_config(64ll * ntiles);
    if (ntiles > 0) SOP_HI_LAUNCH(k_hi_eps, cfg, ntiles, stream, jobs, st, tiles, ntiles);
    hipLaunchKernelGGL(k_hi_beta, dim3(njobs), dim3(kBetaThreads), 0, stream, jobs, st, njobs);
    return hipGetLastError();
}

hipError_t launch_hi_tea_step(const DevJob* jobs, const DevJobState* st, const int2* tiles, int ntiles, int kstep,
                              hipStream_t stream) {
    const HiConfig cfg = hi_config(64ll * ntiles);
    if (ntiles > 0) SOP_HI_LAUNCH(k_hi_tea, cfg, ntiles, stream, jobs, st, tiles, ntiles, kstep);
    return hipGetLastError();
}

// The lower triangle's rows from s on, columns [s, s + cols) (cols < 0: all),
// minus the panel copy's kw columns times their transpose.  The next panel's
// columns (cols = 512): 128x64 tiles, which put 3,700 rows on 232 CUs and whose
// sums are taken in parts (update_tile); 128x128 tiles, one sum per element, are
// no faster from 8,000 rows on either (order 12,288 split-BF16 5.33 ms, 5.32 with
// 128x64) and left the factor's error 0.1 % above that of sums in parts.  The
// rest: regions of at least a round of 256x256 tiles take those, smaller ones
// 128x128.
static constexpr int kTrailBigMinTiles = 256;
template <int MODE>
static void trailing_update(float* M, size_t ld, int s, int mp, int cols, int kw, const char* pan,
                            hipStream_t stream) {
    if (s >= mp) return;
    const int nr = (mp - s + 127) / 128;
    const int ntr = (mp - s + BT - 1) / BT, ntile = ntr * (ntr + 1) / 2;
    if (cols >= 0)
        hipLaunchKernelGGL((k_update<MODE, 128, 64>), dim3(nr, cols / 64), dim3(256), 0, stream, M, ld, s, mp, kw, pan);
    else if (ntile >= kTrailBigMinTiles)
        hipLaunchKernelGGL((k_update_big<MODE>), dim3((ntile + kXcds - 1) / kXcds * kXcds), dim3(512), 0, stream, M, ld,
                           s, mp, kw, ntr, pan);
    else
        hipLaunchKernelGGL((k_update<MODE, 128, 128>), dim3(nr, nr), dim3(256), 0, stream, M, ld,
                           s, mp, kw, pan);
}

// Blocked factorisation over outer panels of NB2 columns, each factored by
// fused 64-column steps (k_chol_step).  A panel's update of the next panel's
// columns follows its steps; the rest of the trailing matrix (from the panel
// after the next one on) is updated on `aux`, overlapped with the next panel.
// Panel p's update of the next panel's columns waits for the trailing update
// of panel p-1, which writes them too and reads the copy that panel p+1
// writes.  With aux == nullptr everything runs on `stream`.
hipError_t launch_chol_factor(float* M, size_t ld, int mp, int mode, const CholWork& w, hipStream_t stream,
                              hipStream_t aux, hipEvent_t ev_f, hipEvent_t ev_t2a, hipEvent_t ev_t2b) {
    const bool two = aux != nullptr && ev_f != nullptr && ev_t2a != nullptr && ev_t2b != nullptr;
    hipEvent_t ev_t2[2] = {ev_t2a, ev_t2b};
    bool pending[2] = {false, false};
    hipError_t e = hipSuccess;
    const int nblk = mp / NB;
    float* const pbuf = reinterpret_cast<float*>(w.linv + (size_t)2 * NB * NB);  // after the two inverses
    auto update = [&](int s, int cols, int kw, const char* pan, hipStream_t on) {
        if (mode == SOP_CHOL_F32) trailing_update<SOP_CHOL_F32>(M, ld, s, mp, cols, kw, pan, on);
        else trailing_update<SOP_CHOL_BF16X3>(M, ld, s, mp, cols, kw, pan, on);
    };
    for (int c0 = 0, p = 0; c0 < mp; c0 += NB2, ++p) {
        const int kw = mp - c0 < NB2 ? mp - c0 : NB2, nb = kw / NB;
        char* const pan = w.pan[p & 1];
        for (int j = 0; j <= nb; ++j) {
            const int nwg = nblk - (c0 / NB + j);
            if (nwg <= 0) continue;
            const int look = j + 1 < nb ? 1 : 0;  // a next diagonal block in this panel
            const CholStep a{M, ld, mp, c0, kw, j,
                             w.linv + (size_t)((j + 1) & 1) * NB * NB, w.linv + (size_t)(j & 1) * NB * NB,
                             w.bbuf + (size_t)((j + 1) & 1) * mp * NB, w.bbuf + (size_t)(j & 1) * mp * NB,
                             pbuf + (size_t)(j & 1) * NB * NB, pbuf + (size_t)((j + 1) & 1) * NB * NB, look,
                             pan};
            if (mode == SOP_CHOL_F32)
                hipLaunchKernelGGL(k_chol_step<SOP_CHOL_F32>, dim3(nwg + look), dim3(kCholThreads), 0, stream, a);
            else
                hipLaunchKernelGGL(k_chol_step<SOP_CHOL_BF16X3>, dim3(nwg + look), dim3(kCholThreads), 0, stream, a);
        }
        const int s0 = c0 + kw, s1 = s0 + NB2;  // the next panel, and what follows it
        // the panel before this one updates the next panel's columns on aux,
        // reading the copy that the next panel writes: done with both first
        if (pending[(p + 1) & 1]) {
            if ((e = hipStreamWaitEvent(stream, ev_t2[(p + 1) & 1], 0)) != hipSuccess) return e;
            pending[(p + 1) & 1] = false;
        }
        if (s0 < mp) update(s0, NB2, kw, pan, stream);
        if (s1 < mp && two) {
            if ((e = hipEventRecord(ev_f, stream)) != hipSuccess) return e;
            if ((e = hipStreamWaitEvent(aux, ev_f, 0)) != hipSuccess) return e;
            update(s1, -1, kw, pan, aux);
            if ((e = hipEventRecord(ev_t2[p & 1], aux)) != hipSuccess) return e;
            pending[p & 1] = true;
        } else if (s1 < mp) {
            update(s1, -1, kw, pan, stream);
        }
    }
    for (int q = 0; q < 2; ++q)
        if (pending[q] && (e = hipStreamWaitEvent(stream, ev_t2[q], 0)) != hipSuccess) return e;
    return hipGetLastError();
}

hipError_t launch_chol_step(const DevJob* jobs, const DevJobState* st, const int2* tiles, int ntiles, int kstep,
                            const HiExactWork* w, hipStream_t stream) {
    const HiConfig cfg = hi_config(64ll * ntiles);
    SOP_HI_LAUNCH(k_chol_D, cfg, ntiles, stream, jobs, st, tiles, ntiles, kstep);
    if (w) {
        hipLaunchKernelGGL(k_chol_build, dim3(ntiles, ntiles), dim3(256), 0, stream, jobs, st, tiles, kstep);
        // the factorisation's error covers the event record/wait pairs that
        // order its two streams: report it before the noise reads the factor
        const hipError_t e =
            launch_chol_factor(w->M, w->ld, w->mp, w->mode, w->work, stream, w->aux, w->ev_f, w->ev_t2[0], w->ev_t2[1]);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k_chol_L, dim3(ntiles * 16), dim3(256), 0, stream, jobs, st, tiles, ntiles, kstep);
    return hipGetLastError();
}

}  // namespace sop

// ---------------------------------------------------------------------------
// Factorisation on caller-owned device memory with nothing allocated
// (sop_chol_factor_noalloc): the workspace of launch_chol_factor -- the FP64
// inverses of a panel's diagonal blocks and the two panel copies
// -- sized for matrices up to kNoAllocMaxOrder, lives in one static
// device array that every GPU the library runs on holds until the process
// ends.  Its device address is taken once per device with
// hipGetSymbolAddress; the array's name is never used as an address on the
// host.
// ---------------------------------------------------------------------------
namespace sop {

constexpr int kNoAllocMaxOrder = 12288;  // 3N for N = 4,096 beads
constexpr size_t kNoAllocBBytes = (size_t)2 * kNoAllocMaxOrder * 64 * sizeof(float);  // chol_bbuf_bytes
constexpr size_t kNoAllocPanelBytes = (size_t)kNoAllocMaxOrder * kCholPanel * 4;  // chol_panel_bytes
constexpr size_t kNoAllocScratchBytes = kCholLinvBytes + kNoAllocBBytes + 2 * kNoAllocPanelBytes;  // linv|bbuf|pan0|pan1
static_assert(kCholLinvBytes % 256 == 0 && kNoAllocBBytes % 256 == 0 && kNoAllocPanelBytes % 256 == 0,
              "scratch sections stay 256-byte aligned");

static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
unsigned char* g_scratch_ptr[kMaxDevices] = {};

// The device address of `scratch` on `device` (the current device).
hipError_t scratch_on(int device, unsigned char** out) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (!p) return hipErrorInvalidSymbol;
        g_scratch_ptr[device] = static_cast<unsigned char*>(p);
    }
    *out = g_scratch_ptr[device];
    return hipSuccess;
}

// Rows n..mp-1 of M become the identity padding: zero left of the
// diagonal, one on it (the allocating entry point pads the same way).
__global__ __launch_bounds__(256) void k_chol_pad(float* __restrict__ M, size_t ld, int n, int mp) {
    const int r = n + (int)blockIdx.y;
    const int c = (int)(blockIdx.x * 256 + threadIdx.x);
    if (r >= mp || c > r) return;
    M[(size_t)r * ld + c] = c == r ? 1.0f : 0.0f;
}

}  // namespace

}  // namespace sop

extern "C" int sop_chol_factor_noalloc(int device, int n, float* M, unsigned long long ld, int mode, void* stream) {
    using namespace sop;
    if (n <= 0 || !M) return fail(SOP_E_ARG, "cholesky (no allocation): bad arguments");
    if (n > kNoAllocMaxOrder)
        return fail(SOP_E_ARG, "cholesky (no allocation): order " + std::to_string(n) + " exceeds the maximum " +
                                   std::to_string(kNoAllocMaxOrder));
    if (mode != SOP_CHOL_BF16X3 && mode != SOP_CHOL_F32) return fail(SOP_E_ARG, "cholesky (no allocation): unknown mode");
    const int mp = (n + 63) / 64 * 64;
    if (ld < (unsigned long long)mp)
        return fail(SOP_E_ARG, "cholesky (no allocation): leading dimension " + std::to_string(ld) +
                                   " is below the padded order " + std::to_string(mp));
    if (ld % 4 != 0 || reinterpret_cast<uintptr_t>(M) % 16 != 0)
        return fail(SOP_E_ARG, "cholesky (no allocation): rows must start on 16-byte boundaries "
                               "(M 16-byte aligned, leading dimension a multiple of 4)");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return fail(SOP_E_HIP, "no HIP device available");
    if (device < 0 || device >= ndev || device >= kMaxDevices) return fail(SOP_E_ARG, "device index out of range");
    if (hipSetDevice(device) != hipSuccess) return fail(SOP_E_HIP, "hipSetDevice failed");
    unsigned char* base = nullptr;
    hipError_t e = scratch_on(device, &base);
    if (e != hipSuccess)
        return fail(SOP_E_HIP, std::string("cholesky (no allocation): scratch address: ") + hipGetErrorString(e));
    // the workspace of an order-mp factorisation, carved from the front of each section
    CholWork w{};
    w.linv = reinterpret_cast<double*>(base);
    w.bbuf = reinterpret_cast<float*>(base + kCholLinvBytes);
    w.pan[0] = reinterpret_cast<char*>(base + kCholLinvBytes + kNoAllocBBytes);
    w.pan[1] = w.pan[0] + kNoAllocPanelBytes;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    if (mp > n) hipLaunchKernelGGL(k_chol_pad, dim3((mp + 255) / 256, mp - n), dim3(256), 0, s, M, (size_t)ld, n, mp);
    e = hipGetLastError();
    if (e == hipSuccess) e = launch_chol_factor(M, (size_t)ld, mp, mode, w, s);
    if (e != hipSuccess) return fail(SOP_E_HIP, std::string("cholesky (no allocation): ") + hipGetErrorString(e));
    return 0;
}
