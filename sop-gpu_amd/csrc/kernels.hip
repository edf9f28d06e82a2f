// kernels.hip -- CDNA4 kernels of the SOP Langevin hot path.
//
// k_step, k_step_lds
//              one launch per step for every admitted job: FENE + native
//              LJ 12-6 + repulsive LJ (+ indentation walls) gathered per bead
//              over slot-major lists, then the Hybrid-Taus noise, the
//              fixed/pulled-bead rules and the overdamped Euler update; the
//              LDS variant stages the coordinates of jobs of at most 5,120
//              beads in LDS.  Reference bodies: src/Potentials/covalent_kernel.cu:28-51,
//              native_kernel.cu:27-52, pairs_kernel.cu:33-59,
//              indentation_kernel.cu:71-128, src/Integrators/langevin_kernel.cu:17-58.
// k_step_rows, k_step_rows_one
//              the same step with each bead's force terms spread over the lanes
//              of a wavefront, for launches of too few beads for one per lane;
//              the latter for launches of a single job.
// k_block_rows the steps of a block of small jobs in one launch, a workgroup
//              per job, with the updaters and Verlet lists it begins with.
// k_possible, k_possible_lds, k_possible_boxes, k_possible_cells
//              possible-pairs list: same-job beads j != i, ascending j, with
//              sqrtf(d^2) < threshold, excluding covalent and native partners
//              (src/Updaters/possiblepairlist_kernel.cu:18-71).
// k_sort_rows  row order of the Verlet lists (by list length) and the
//              bonded lists moved into it.
// k_verlet, k_verlet_lds
//              Verlet list: the possible list filtered by sqrtf(d^2) <
//              pairlist_cutoff in stored order (src/Updaters/pairlist_kernel.cu:33-76).
// k_job_update per-job updaters at stride boundaries: indentation tip,
//              force-ramp cantilever, heating schedule
//              (src/Potentials/indentation.cu:414-511, pulling.cu:152-214,
//              src/Integrators/langevin.cu:76-82).
// k_energies   per-bead energies for the output cadence
//              (covalent_kernel.cu:57-77, native_kernel.cu:57-82, pairs_kernel.cu:69-91).
//
// Work is distributed as 64-bead tiles (one wavefront each) that never cross
// a job boundary, so every wavefront reads one job's descriptor through
// scalar loads.  Tiles are assigned to XCDs in contiguous ranges: workgroups
// are dispatched round-robin over the 8 XCDs, so block b runs on XCD b%8, and
// giving XCD x the x-th slice of the tile list keeps each job's coordinates in
// one XCD's L2.
#include "kernels.h"

#include <climits>

#include "devmath.h"

namespace sop {

static constexpr int kTilesPerBlock = 4;  // 256-thread workgroups

__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

struct TileRange {
    int begin, end, step;
};

// Contiguous slice of the tile list for this workgroup's XCD.
__device__ __forceinline__ TileRange xcd_tiles(int ntiles) {
    const int nb = gridDim.x;
    const int nxcd = nb >= 8 ? 8 : 1;
    const int xcd = blockIdx.x % nxcd;
    const int r = blockIdx.x / nxcd;
    const int per_xcd_blocks = nb / nxcd;
    const int slice = (ntiles + nxcd - 1) / nxcd;
    TileRange t;
    t.begin = xcd * slice + r * kTilesPerBlock + wave_id();
    t.end = min((xcd + 1) * slice, ntiles);
    t.step = per_xcd_blocks * kTilesPerBlock;
    return t;
}

// The descriptor's arrays as global-memory pointers.  Through a generic
// pointer the compiler issues flat loads, which are counted with the LDS
// operations as well, so a wait for an LDS read also waits for every
// prefetch in flight; global loads are counted apart from the LDS reads.
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(1))) T* gmem(const T* p) {
    return (const __attribute__((address_space(1))) T*)p;
}
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T* gmem(T* p) {
    return (__attribute__((address_space(1))) T*)p;
}

// Coordinates gathered from global memory with global-address-space loads
// (cin[j]), for the kernels that gather from L2: through a generic pointer
// the gathers are flat loads, which count with the scalar loads too, so a
// wait for a descriptor field also drained every gather in flight.
typedef float f32x4_g __attribute__((ext_vector_type(4)));
typedef float f32x2_g __attribute__((ext_vector_type(2)));
// p[k] of a float2 array in global memory, by a global-address-space load.
__device__ __forceinline__ float2 ldg2(const float2* p, size_t k) {
    const f32x2_g v = ((const __attribute__((address_space(1))) f32x2_g*)p)[k];
    return make_float2(v.x, v.y);
}
struct CoordGlobal {
    const float4* p;
    __device__ __forceinline__ float4 operator[](int j) const {
        const f32x4_g v = ((const __attribute__((address_space(1))) f32x4_g*)p)[j];
        return make_float4(v.x, v.y, v.z, v.w);
    }
};
// The global-gather kernels also read the per-bead counts and the native
// parameters by global-address-space loads; the LDS kernels keep the
// generic loads (the global form costs them registers).
template <typename CP>
constexpr bool kGlobalCoords = std::is_same<CP, CoordGlobal>::value;

// ---------------------------------------------------------------------------
// fused step
// ---------------------------------------------------------------------------

// The scalar factors of the three force terms, shared by every step
// kernel so that each evaluates the same float expressions.
// Repulsive LJ, for d2 < rc2 (pairs_kernel.cu:41-56): the force on the bead
// is (x, y, z) * q; `fast` (the job's a2 and rc2 admit the short division)
// takes div_rn_fast for d2 >= kDivFastMinB.
__device__ __forceinline__ float pair_q(float d2, float a2, float m6, bool fast) {
    float q = div_rn_fast(a2, d2);
    if (!(fast && d2 >= kDivFastMinB)) q = div_ieee(a2, d2);
    q = q * q;
    return m6 * q * q;
}
// FENE (covalent_kernel.cu:36-48): the force is w * (x, y, z).
__device__ __forceinline__ float fene_w(float ks, float R2, float x, float y, float z, float r0) {
    float w = sqrtf(x * x + y * y + z * z);
    w = w - r0;
    return ks * w / ((w + r0) * (1.0f - w * w / R2));
}
// Native LJ 12-6 (native_kernel.cu:36-49), par = (r0^2, -12 eh / r0^2): the
// force is (x, y, z) * q.
__device__ __forceinline__ float native_q(float x, float y, float z, float2 par) {
    float q = par.x / (x * x + y * y + z * z);
    const float p6 = q * q * q;
    return q * (p6 * p6 - p6) * par.y;
}

// Repulsive LJ over a bead's slot-major Verlet entries, in list order.  The
// list words are streamed with non-temporal loads (each is used once per
// step) and fetched one batch of PB ahead: while batch b is computed the
// indices of batch b+1 and the coordinates of batch b are in flight.  PB is
// 8 for gathers from L2 and 6 for gathers from LDS (which keeps the LDS
// kernel within the 64 VGPRs of two workgroups per CU).
// TAILB: the last np % PB entries are loaded as one predicated batch
// instead of one after another (gathers from L2, few wavefronts to hide
// the latency of each).
template <int PB, typename IdxT, bool TAILB = false, typename CP = const float4*>
__device__ __forceinline__ void pair_loop(const __attribute__((address_space(1))) IdxT* __restrict__ pj, int np, int n, CP cin,
                                          const float4 c, float rc2, float a2, float m6, float& fx, float& fy,
                                          float& fz) {
    // every d2 below rc2 and above kDivFastMinB takes the short division
    const bool fast = div_fast_numerator(a2) && rc2 <= kDivFastMaxB;
#define SOP_PAIR(o)                                                  \
    {                                                                \
        const float x = (o).x - c.x, y = (o).y - c.y, z = (o).z - c.z; \
        const float d2 = x * x + y * y + z * z;                      \
        if (d2 < rc2) {                                              \
            const float q = pair_q(d2, a2, m6, fast);                \
            fx += x * q;                                             \
            fy += y * q;                                             \
            fz += z * q;                                             \
        }                                                            \
    }
    int k = 0;
    if (np >= PB) {
        int jn[PB];
#pragma unroll
        for (int u = 0; u < PB; ++u) jn[u] = (int)__builtin_nontemporal_load(pj + (size_t)u * n);
        for (; k + PB <= np; k += PB) {
            float4 o[PB];
#pragma unroll
            for (int u = 0; u < PB; ++u) o[u] = cin[jn[u]];
            if (k + 2 * PB <= np) {
#pragma unroll
                for (int u = 0; u < PB; ++u) jn[u] = (int)__builtin_nontemporal_load(pj + (size_t)(k + PB + u) * n);
            }
#pragma unroll
            for (int u = 0; u < PB; ++u) SOP_PAIR(o[u]);
        }
    }
    if constexpr (TAILB) {
        if (k < np) {
            int jt[PB];
#pragma unroll
            for (int u = 0; u < PB; ++u)
                jt[u] = k + u < np ? (int)__builtin_nontemporal_load(pj + (size_t)(k + u) * n) : 0;
            float4 ot[PB];
#pragma unroll
            for (int u = 0; u < PB; ++u) ot[u] = cin[jt[u]];
#pragma unroll
            for (int u = 0; u < PB; ++u)
                if (k + u < np) SOP_PAIR(ot[u]);
        }
    } else {
        for (; k < np; ++k) {
            const float4 o = cin[(int)__builtin_nontemporal_load(pj + (size_t)k * n)];
            SOP_PAIR(o);
        }
    }
#undef SOP_PAIR
}
// The fixed/pulled rules of the reference's extForces (pulling.cu:108-125,
// langevin_kernel.cu:43-50): a fixed bead's force is zeroed, a pulled bead's
// gets the cantilever force.  The one-byte flag is read for every bead, the
// 16-byte force record only for pulled beads.
template <typename D>
__device__ __forceinline__ void ext_rules_flag(const D& J, int i, int f, float& fx, float& fy, float& fz) {
    if (f == 1) {
        fx = 0.0f; fy = 0.0f; fz = 0.0f;
    } else if (f == 2) {
        const float4 e = J.ext[i];
        fx += e.x; fy += e.y; fz += e.z;
    }
}

// FENE (covalent_kernel.cu:36-48) and native LJ 12-6 (native_kernel.cu:36-49)
// of one bead: nc covalent and nn native partners from slot-major lists of
// slot stride n whose columns for this bead start at cj, cr, nj, npar
// (32- or 16-bit indices; bead order, or row order for sorted rows).
template <typename CJ, typename CR, typename NJ, typename CP>
__device__ __forceinline__ void bonded_terms(const DevJob& J, int nc, int nn, int n, CJ cj, CR cr, NJ nj,
                                             const float2* __restrict__ npar, CP cin,
                                             const float4 c, float& fx, float& fy, float& fz) {
    // FENE (covalent_kernel.cu:36-48)
    {
        for (int k = 0; k < nc; ++k) {
            const int j = cj[(size_t)k * n];
            const float r0 = cr[(size_t)k * n];
            const float4 o = cin[j];
            const float x = o.x - c.x, y = o.y - c.y, z = o.z - c.z;
            const float w = fene_w(J.ks, J.R2, x, y, z, r0);
            fx += w * x;
            fy += w * y;
            fz += w * z;
        }
    }
    // native LJ 12-6 (native_kernel.cu:36-49), gathers four ahead
    {
#define SOP_NAT(o, par)                                                 \
{                                                                   \
    const float x = (o).x - c.x, y = (o).y - c.y, z = (o).z - c.z;     \
    const float q = native_q(x, y, z, par);                         \
    fx += x * q;                                                    \
    fy += y * q;                                                    \
    fz += z * q;                                                    \
}
        int k = 0;
        for (; k + 4 <= nn; k += 4) {
            int jj[4];
            float2 pp[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                jj[u] = nj[(size_t)(k + u) * n];
                pp[u] = kGlobalCoords<CP> ? ldg2(npar, (size_t)(k + u) * n) : npar[(size_t)(k + u) * n];
            }
            float4 o[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) o[u] = cin[jj[u]];
#pragma unroll
            for (int u = 0; u < 4; ++u) SOP_NAT(o[u], pp[u]);
        }
        for (; k < nn; ++k) {
            const float2 par = kGlobalCoords<CP> ? ldg2(npar, (size_t)k * n) : npar[(size_t)k * n];
            const float4 o = cin[nj[(size_t)k * n]];
            SOP_NAT(o, par);
        }
#undef SOP_NAT
    }
}

// The first part of a bead's step, before the repulsive pairs: the extra
// force record, then FENE and native LJ 12-6 (for sorted rows from the
// row-ordered copies -- a wavefront's 64 rows read 64 consecutive words per
// slot -- else in bead order, partner indices 16-bit where the job has a
// 16-bit copy).  i: bead, r: its Verlet row; c = cin[i].
template <bool FO, typename CP>
__device__ __forceinline__ void step_head(const DevJob& J, int i, int r, int n, CP cin, const float4 c, float& fx,
                                          float& fy, float& fz) {
    fx = 0.0f, fy = 0.0f, fz = 0.0f;
    if (J.flags & JF_EXTRA_FORCE) {
        const float4 e = J.fextra[i];
        fx = e.x; fy = e.y; fz = e.z;
        if constexpr (!FO) J.fextra[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    if (J.sort_rows) {
        const int cnt = gmem(J.rb_cnt)[r];
        bonded_terms(J, cnt & 0xffff, cnt >> 16, J.pair_ld, gmem(J.rb_cov_j) + r, gmem(J.rb_cov_r0) + r,
                     gmem(J.rb_nat_j) + r, J.rb_nat_par + r, cin, c, fx, fy, fz);
    } else if (J.nat_j16) {
        bonded_terms(J, kGlobalCoords<CP> ? gmem(J.cov_cnt)[i] : J.cov_cnt[i],
                     kGlobalCoords<CP> ? gmem(J.nat_cnt)[i] : J.nat_cnt[i], n, gmem(J.cov_j16) + i, gmem(J.cov_r0) + i,
                     gmem(J.nat_j16) + i, J.nat_par + i, cin, c, fx, fy, fz);
    } else {
        bonded_terms(J, kGlobalCoords<CP> ? gmem(J.cov_cnt)[i] : J.cov_cnt[i],
                     kGlobalCoords<CP> ? gmem(J.nat_cnt)[i] : J.nat_cnt[i], n, gmem(J.cov_j) + i, gmem(J.cov_r0) + i,
                     gmem(J.nat_j) + i, J.nat_par + i, cin, c, fx, fy, fz);
    }
}

// The per-bead state the tail reads and its noise, formed ahead by a caller
// with latency to hide (which then also writes the RNG state back): the
// Gaussian triple, the temperature accumulator and the fixed/pulled flag.
// A caller that takes several steps says whether one starts a stride (due) and
// gets T and the new coordinates c back.
struct TailPre {
    float3 g;
    float T;
    int flag;
    bool due;
    float4 c;
};

// The rest of a bead's step, after the repulsive pairs: indentation walls,
// then (FO) the forces written to cout, or the noise (of amplitude var), the
// fixed/pulled rules and the Euler update written to `cout` in global memory.  Hydrodynamic
// jobs stop after the forces.  pre: the state loaded ahead (null: loaded
// here).  KEEP: T and the coordinates stay in *pre, nothing is written.
template <bool FO, bool KEEP = false, typename D>
__device__ __forceinline__ void step_tail(const D& J, const DevJobState& S, float var, long long s, int i, const float4 c,
                                          float fx, float fy, float fz, float4* __restrict__ cout,
                                          TailPre* pre = nullptr) {
    // indentation tip and substrate plane (indentation_kernel.cu:71-128)
    if (J.flags & JF_INDENTATION) {
        float4 fin = J.tipF[i];
        float x = c.x - S.tip[0], y = c.y - S.tip[1], z = c.z - S.tip[2];
        const float rr = sqrtf(x * x + y * y + z * z);
        float r2 = rr - J.tipR;
        r2 = 1.0f / r2;
        r2 = r2 * r2;
        float r6 = r2 * r2 * r2;
        float dw = J.tipAp * r6 + J.tipBp;
        dw = dw * r6 / (rr * (rr - J.tipR));
        const float dfx = x * dw, dfy = y * dw, dfz = z * dw;
        fin.x += dfx;
        fin.y += dfy;
        fin.z += dfz;
        if constexpr (!FO) J.tipF[i] = fin;
        x = c.x - S.micaR[0];
        y = c.y - S.micaR[1];
        z = c.z - S.micaR[2];
        float h = x * J.micaN[0] + y * J.micaN[1] + z * J.micaN[2];
        h = 1.0f / h;
        h = h * h;
        r6 = h * h * h;
        float sw = J.surfAp * r6 + J.surfBp;
        sw = sw * r6 * h;
        fx += J.micaN[0] * sw + dfx;
        fy += J.micaN[1] * sw + dfy;
        fz += J.micaN[2] * sw + dfz;
    }
    if constexpr (FO) {
        cout[i] = make_float4(fx, fy, fz, 0.0f);
        return;
    }
    // hydrodynamic jobs: noise and forces for the HI integrator
    // (integrateTea_prepare, bdhitea_kernel.cu:33-65); the update itself
    // runs in hi.hip once every bead's forces are known
    if (J.flags & JF_HI) {
        uint4 rs = pre ? make_uint4(0, 0, 0, 0) : J.rng[i];
        const float3 g = pre ? pre->g : gauss3(rs);
        if (!pre) J.rng[i] = rs;
        J.rforce[i] = make_float4(g.x * var, g.y * var, g.z * var, 0.0f);
        if (J.flags & JF_PULLING) ext_rules_flag(J, i, pre ? pre->flag : (int)J.bflag[i], fx, fy, fz);
        J.mforce[i] = make_float4(fx, fy, fz, 0.0f);
        return;
    }
    // Langevin step (langevin_kernel.cu:24-56)
    if (!(J.flags & JF_MINIMIZATION)) {
        uint4 rs = pre ? make_uint4(0, 0, 0, 0) : J.rng[i];
        const float3 g = pre ? pre->g : gauss3(rs);
        if (!pre) J.rng[i] = rs;
        fx += g.x * var;
        fy += g.y * var;
        fz += g.z * var;
    }
    if (J.flags & JF_PULLING) ext_rules_flag(J, i, pre ? pre->flag : (int)J.bflag[i], fx, fy, fz);
    const float m = J.hOverZeta;
    const float dx = m * fx, dy = m * fy, dz = m * fz;
    float4 cn = c;
    cn.x += dx;
    cn.y += dy;
    cn.z += dz;
    // the temperature accumulator is cleared at updater passes that fall
    // on a multiple of nav (output_manager.cu:124-126)
    const bool reset = (KEEP ? pre->due : s % J.stride == 0) && s % J.nav == 0;
    const float T0 = reset ? 0.0f : (pre ? pre->T : J.T[i]);
    const float T1 = T0 + J.tempNorm * (dx * dx + dy * dy + dz * dz);
    if constexpr (KEEP) {
        pre->T = T1;
        pre->c = cn;
    } else {
        J.T[i] = T1;
        cout[i] = cn;
    }
}

// One bead's step: FENE, native and repulsive terms gathered from `cin`
// (global memory, or the job's coordinates staged in LDS), indentation
// walls, then noise, the fixed/pulled rules and the Euler update, written to
// `cout` in global memory.  Hydrodynamic jobs stop after the forces.
// FO (forces only): the same force terms, written to `cout` (indexed by
// bead) before the noise, with no state changed -- the parity hook of the
// force gather runs the kernel the step runs.
template <int PB, bool FO = false, bool TAILB = false, typename CP = const float4*>
__device__ __forceinline__ void step_bead(const DevJob& J, const DevJobState& S, long long s, int i, int r, int n,
                                          CP cin, float4* __restrict__ cout) {
    const float4 c = cin[i];
    float fx, fy, fz;
    step_head<FO>(J, i, r, n, cin, c, fx, fy, fz);
    // repulsive LJ over the Verlet list (pairs_kernel.cu:41-56)
    const int np = gmem(J.pair_cnt)[r];
    if (J.idx16)
        pair_loop<PB, unsigned short, TAILB>(gmem(static_cast<const unsigned short*>(J.pair_j)) + r, np, J.pair_ld,
                                             cin, c, J.rc2, J.a2, J.m6, fx, fy, fz);
    else
        pair_loop<PB, int, TAILB>(gmem(static_cast<const int*>(J.pair_j)) + r, np, J.pair_ld, cin, c, J.rc2, J.a2,
                                  J.m6, fx, fy, fz);
    step_tail<FO>(J, S, S.var, s, i, c, fx, fy, fz, cout);
}

// FO: forces only, into fout (bead-indexed), for every job of the tiles
// whatever its step (nothing is advanced).
template <bool FO>
__global__ __launch_bounds__(256) void k_step(const DevJob* __restrict__ jobs, const DevJobState* __restrict__ st,
                                              const int2* __restrict__ tiles, int ntiles, int kstep,
                                              float4* __restrict__ fout) {
    const int lane = threadIdx.x & 63;
    const TileRange tr = xcd_tiles(ntiles);
    for (int t = tr.begin; t < tr.end; t += tr.step) {
        const int2 td = tiles[t];
        const DevJob& J = jobs[td.x];
        if (J.lds_step) continue;  // stepped by k_step_lds
        const long long s = st[td.x].step + kstep;
        if (!FO && s >= J.end_step) continue;
        const int r = td.y + lane;  // Verlet row; the lane steps bead perm[r]
        const int n = J.n;
        if (r >= n) continue;
        step_bead<8, FO, true>(J, st[td.x], s, gmem(J.perm)[r], r, n, CoordGlobal{J.coord[s & 1]},
                               FO ? fout : J.coord[(s + 1) & 1]);
    }
}

// The same step for jobs small enough to keep their coordinates in LDS.
// One 1024-thread workgroup per unit; a unit is up to 1024 Verlet rows in
// segments (job, first row, rows, LDS offset): a job's whole 1024-row
// blocks are units of their own, and the rows left over share units with
// other jobs' left-over rows.  The workgroup stages each segment's job
// coordinates in LDS (coalesced), so every neighbour gather of the step
// reads LDS.  Segments start at multiples of 64 threads: no wavefront spans
// two jobs.
// PB: Verlet entries fetched ahead per lane (pair_loop).  With PB <= 6 the
// kernel is built for two 1024-thread workgroups per CU (64 VGPRs), with
// PB = 8 for one (128 VGPRs); two 80 KB LDS stagings fit a CU either way.
template <bool FO, int PB>
__global__ __launch_bounds__(1024, PB <= 6 ? 8 : 4) void k_step_lds(const DevJob* __restrict__ jobs,
                                                                 const DevJobState* __restrict__ st,
                                                                 const int2* __restrict__ units,
                                                                 const int4* __restrict__ segs, int nunits, int kstep,
                                                                 float4* __restrict__ fout) {
    extern __shared__ float4 lds_coord[];
    for (int u = blockIdx.x; u < nunits; u += gridDim.x) {
        const int2 ud = units[u];  // first segment, segments
        __syncthreads();           // the previous unit's gathers are done
        for (int q = 0; q < ud.y; ++q) {
            const int4 sg = segs[ud.x + q];
            const DevJob& J = jobs[sg.x];
            const long long s = st[sg.x].step + kstep;
            if (!FO && s >= J.end_step) continue;
            const float4* __restrict__ g = J.coord[s & 1];
            for (int k = threadIdx.x; k < J.n; k += blockDim.x) lds_coord[sg.w + k] = g[k];
        }
        __syncthreads();
        int t = threadIdx.x;
        for (int q = 0; q < ud.y; ++q) {
            const int4 sg = segs[ud.x + q];
            const int span = (sg.z + 63) & ~63;
            if (t < span) {
                const DevJob& J = jobs[sg.x];
                const long long s = st[sg.x].step + kstep;
                const int r = sg.y + t;  // Verlet row; the thread steps bead perm[r]
                if (t < sg.z && (FO || s < J.end_step))
                    step_bead<PB, FO>(J, st[sg.x], s, J.perm[r], r, J.n, lds_coord + sg.w,
                                      FO ? fout : J.coord[(s + 1) & 1]);
                break;
            }
            t -= span;
        }
    }
}

// The step with each bead's force terms spread over a wavefront, for launches
// whose rows, one per lane, would leave most of the GPU idle or the lanes
// walking their ~150 terms at the latency of one gather after another.
// A wavefront steps R Verlet rows: lane q + R p evaluates, of row q, the terms
// at positions p, p + P, p + 2P ... (P = 64 / R) of a chunk of K = P U terms
// and writes their three components to the wavefront's own LDS rows; lanes
// p < 3 then add component p of row q in stream order -- FENE, native, the
// Verlet entries -- while the next chunk's partners are on their way.
// Positions without a term hold -0.0 (x + (-0.0) is x for every float x), so
// the sums are the one-lane step's, rounded term by term, and the step is
// bit-identical.  Nothing is shared between wavefronts: no barrier, and a
// launch of any number of rows.  Partners are gathered from global memory
// (the coordinates of a job stay in L1/L2), so jobs on either side of the
// LDS limit are stepped by the same launch.  Bound by the latency of its
// dependent reads (tile, record, lists, partners) where rows are few, by those
// and VALU issue (53 % of the cycles at 100,000 rows of a capsid) where many;
// measured at Engine::effective_shape (18,000 beads: 58 us one bead per lane, 16
// us here).
template <int R, bool BLK = false>
struct RowsShape {
    static constexpr int P = 64 / R;              // positions of a row evaluated at a time
    static constexpr int U = R <= 4 || BLK ? 4 : 8;  // terms per lane and chunk
    static constexpr int K = P * U;               // terms of a row per chunk
    // row stride of the LDS rows: the R rows' P consecutive words (writes) and
    // 16-byte reads fall in distinct banks
    static constexpr int KP = K + 64 / R;
};

// p[off bytes on] in global memory: base in scalar registers, a 32-bit offset
// per lane.
template <typename T>
__device__ __forceinline__ T ldg_off(const T* p, unsigned off) {
    return *reinterpret_cast<const __attribute__((address_space(1))) T*>(
        reinterpret_cast<const __attribute__((address_space(1))) char*>(gmem(p)) + off);
}
// Coordinates of bead j (jobs hold far fewer than 2^28 beads).
__device__ __forceinline__ float4 ldg_coord(const float4* p, int j) {
    const f32x4_g v = ldg_off(reinterpret_cast<const f32x4_g*>(p), (unsigned)j << 4);
    return make_float4(v.x, v.y, v.z, v.w);
}

// A FENE (type 0, par.x = r0) or native (type 1) term of a row, fetched ahead
// of its evaluation; type 3: no term at this position.
struct BondedSrc {
    int j, type;
    float2 par;
};
// Term t of the bonded stream (nc FENE, then nn native) of column col of the
// job's bonded lists; i: the row's bead (a partner for positions without a term).
template <typename IdxT>
__device__ __forceinline__ BondedSrc bonded_fetch(const StepDesc& D, int t, int col, int i, int nc, int nn) {
    BondedSrc f;
    f.j = i;
    f.type = 3;
    f.par = make_float2(0.0f, 0.0f);
    if (t < nc) {
        const size_t e = (size_t)t * D.b_ld + col;
        f.type = 0;
        f.j = (int)gmem(static_cast<const IdxT*>(D.cov_j))[e];
        f.par.x = gmem(D.cov_r0)[e];
    } else if (t < nc + nn) {
        const size_t e = (size_t)(t - nc) * D.b_ld + col;
        f.type = 1;
        f.j = (int)gmem(static_cast<const IdxT*>(D.nat_j))[e];
        f.par = ldg2(D.nat_par, e);
    }
    return f;
}

// Adds the first m positions (up to the next multiple of 4) of a row's LDS
// words to acc, in order; 32 at a time with their reads in flight together.
__device__ __forceinline__ void rows_add(const float* __restrict__ t, int m, float& acc) {
    const float4* __restrict__ t4 = reinterpret_cast<const float4*>(t);
    for (; m > 28; m -= 32, t4 += 8) {
        float4 v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = t4[k];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            acc += v[k].x;
            acc += v[k].y;
            acc += v[k].z;
            acc += v[k].w;
        }
    }
    for (; m > 0; m -= 4, ++t4) {
        const float4 v = *t4;
        acc += v.x;
        acc += v.y;
        acc += v.z;
        acc += v.w;
    }
}

// The rows of k_step_rows: R rows of one job by one wavefront, lists of IdxT.
// BLK (k_block_rows): nsteps steps, the coordinates in LDS (two buffers of
// ldc beads from lc, the first filled), a workgroup barrier after each step;
// what a step reads besides them stays in registers.
template <bool FO, int R, typename IdxT, bool BLK = false>
__device__ __forceinline__ void step_rows(const StepDesc& D, const DevJobState& S, float var, long long s, int row0,
                                          float (*term)[R][RowsShape<R, BLK>::KP], float4* __restrict__ fout,
                                          float4* lc = nullptr, int ldc = 0, int nsteps = 1) {
    using Shape = RowsShape<R, BLK>;
    constexpr int P = Shape::P, U = Shape::U, K = Shape::K;
    const int lane = threadIdx.x & 63;
    const int n = D.n;
    const float4* const cin = (s & 1) ? D.coord[1] : D.coord[0];
    // this lane's row (loads from the job's last row where the tile ends
    // early; such lanes have no terms)
    const int q = lane % R, p = lane / R, r = row0 + q, rc = min(r, n - 1);
    // the first chunk's Verlet entries, before the counts are known: slots
    // of the list whether filled or not (the unfilled are not used)
    const IdxT* const pj = static_cast<const IdxT*>(D.pair_j);
    const size_t ld = D.pair_ld;
    const unsigned off = ((unsigned)p * (unsigned)D.pair_ld + (unsigned)rc) * (unsigned)sizeof(IdxT);
    IdxT jn[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int k = min(u * P + p, D.pair_cap - 1);
        jn[u] = gmem(pj)[(size_t)k * ld + rc];
    }
    int np = gmem(D.pair_cnt)[rc];
    int i = rc;
    if (D.perm) i = gmem(D.perm)[rc];
    int nc, nn;
    if (D.b_cnt) {
        const int cnt = gmem(D.b_cnt)[rc];
        nc = cnt & 0xffff;
        nn = cnt >> 16;
    } else {
        nc = gmem(D.cov_cnt)[i];
        nn = gmem(D.nat_cnt)[i];
    }
    const int col = D.b_cnt ? rc : i;
    const float4* lin = lc;  // BLK: the step's coordinates
    auto coord = [&](int j) {
        if constexpr (BLK) return lin[j];
        else return ldg_coord(cin, j);
    };
    float4 c = coord(i);
    const bool noise = !FO && !(D.flags & JF_MINIMIZATION);
    TailPre pre;
    uint4 rng = make_uint4(0, 0, 0, 0);
    if constexpr (!FO) {
        rng = D.rng[i];
        pre.T = gmem(D.T)[i];
        pre.flag = 0;
        if (D.flags & JF_PULLING) pre.flag = (int)gmem(D.bflag)[i];
    }
    float acc = 0.0f;
    if (D.flags & JF_EXTRA_FORCE) {
        float4 e = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (p == 0 && r < n) {
            e = D.fextra[i];
            if constexpr (!FO) D.fextra[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
        const float ex = __shfl(e.x, q), ey = __shfl(e.y, q), ez = __shfl(e.z, q);
        acc = p == 0 ? ex : p == 1 ? ey : ez;
    }
    if (r >= n) nc = nn = np = 0;
    int nbm = nc + nn, npm = np;  // the longest rows (every set of R lanes holds all rows)
#pragma unroll
    for (int o = R / 2; o > 0; o >>= 1) {
        nbm = max(nbm, __shfl_xor(nbm, o));
        npm = max(npm, __shfl_xor(npm, o));
    }
    nbm = __builtin_amdgcn_readfirstlane(nbm);
    npm = __builtin_amdgcn_readfirstlane(npm);
    // partners of the first chunk of pairs, the entries of the second, and
    // the first bonded terms: all on their way during the noise
    // (loads without branches, so that each can be waited for by itself:
    // positions without an entry read slot min(.., npm - 1) of the job's first
    // row and gather the row's own bead)
    float4 o[U];
    auto gather = [&](int b) {
#pragma unroll
        for (int u = 0; u < U; ++u) o[u] = coord(b + u * P + p < np ? (int)jn[u] : i);
    };
    auto fetch = [&](int b) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            jn[u] = ldg_off(pj + (size_t)min(b + u * P, npm - 1) * ld, b + u * P + p < np ? off : 0u);
    };
    constexpr int UB = R <= 4 ? 1 : R / 4;  // bonded terms per lane and chunk: 16 of a row (32 for R = 2)
    BondedSrc f[UB];
    auto bonded = [&](int b) {
#pragma unroll
        for (int u = 0; u < UB; ++u)
            if (b + u * P < nbm) f[u] = bonded_fetch<IdxT>(D, b + u * P + p, col, i, nc, nn);
    };
    bonded(0);
    int phase = BLK ? (int)(s % D.stride) : 0;  // of the step within the stride
    for (int step = 0; step < (BLK ? nsteps : 1); ++step) {
        if (BLK && step > 0) {
            c = coord(i);
            acc = 0.0f;
            if (nbm > P * UB) bonded(0);
            if (npm > K) fetch(0);
        }
        if (npm > 0) gather(0);
        if (npm > K) fetch(K);
        // lanes p = 0 and 1 draw the step's four numbers and form one Box-Muller
        // pair each (gauss3's order; the second's cosine is not used)
        if (noise) {
            const uint32_t u0 = hybrid_taus(rng);
            const uint32_t u1 = hybrid_taus(rng);
            const uint32_t u2 = hybrid_taus(rng);
            const uint32_t u3 = hybrid_taus(rng);
            if (!BLK && p == 0 && r < n) D.rng[i] = rng;
            float sn, cs;
            const float rr = sqrtf(-2.0f * logf_series(uint_to_unit(p == 0 ? u0 : u2)));
            const float th = (float)(6.283185307179586 * (double)uint_to_unit(p == 0 ? u1 : u3));
            sincosf_series(th, sn, cs);
            const float gs = rr * sn;
            pre.g = make_float3(gs, rr * cs, __shfl(gs, (lane + R) & 63));
        }
        // FENE and native terms
        for (int b = 0; b < nbm; b += P * UB) {
            if (b > 0) bonded(b);
            // all the chunk's partners first (positions without a term have the
            // row's own bead), and where both kinds of term occur, both formed
            // side by side: behind a branch each, one waited for the other (350
            // peptides 21.4 -> 21.0 ms; 100,000 beads, 400 steps 27.6 -> 27.2)
            float4 w[UB];
#pragma unroll
            for (int u = 0; u < UB; ++u) w[u] = coord(b + u * P < nbm ? f[u].j : i);
#pragma unroll
            for (int u = 0; u < UB; ++u)
                if (b + u * P < nbm) {
                    const float x = w[u].x - c.x, y = w[u].y - c.y, z = w[u].z - c.z;
                    float v;
                    if (__builtin_amdgcn_ballot_w64(f[u].type == 0)) {
                        const float vf = fene_w(D.ks, D.R2, x, y, z, f[u].par.x);
                        const float vn = native_q(x, y, z, f[u].par);
                        v = f[u].type == 0 ? vf : vn;
                    } else {
                        v = native_q(x, y, z, f[u].par);
                    }
                    const bool ok = f[u].type < 3;
                    term[0][q][u * P + p] = ok ? x * v : -0.0f;
                    term[1][q][u * P + p] = ok ? y * v : -0.0f;
                    term[2][q][u * P + p] = ok ? z * v : -0.0f;
                }
            wave_lds_order();
            if (p < 3) rows_add(&term[p][q][0], min(P * UB, nbm - b), acc);
            wave_lds_order();
        }
        // repulsive pairs: the next chunk's partners and the entries of the one
        // after it are in flight while a chunk is added
        const float rc2 = D.rc2, a2 = D.a2, m6 = D.m6;
        const bool fast = div_fast_numerator(a2) && rc2 <= kDivFastMaxB;
        // term u of the chunk from b into LDS; its factor by the short division,
        // or (SLOW) by whichever the divisor admits
        auto put = [&](int u, bool ok, float x, float y, float z, float w) {
            term[0][q][u * P + p] = ok ? x * w : -0.0f;
            term[1][q][u * P + p] = ok ? y * w : -0.0f;
            term[2][q][u * P + p] = ok ? z * w : -0.0f;
        };
        for (int b = 0; b < npm; b += K) {
            // straight-line code over the chunk's terms, so that their latencies
            // overlap; a divisor outside the short division's range (beads almost
            // on top of each other) sends the chunk through the general one
            bool bad = !fast;
#pragma unroll
            for (int h = 0; h < U; h += 4)
                if (b + h * P < npm) {
#pragma unroll
                    for (int u = h; u < h + 4; ++u) {
                        const float x = o[u].x - c.x, y = o[u].y - c.y, z = o[u].z - c.z;
                        const float d2 = x * x + y * y + z * z;
                        const bool ok = (b + u * P + p < np) & (d2 < rc2);
                        bad = bad | (ok & !(d2 >= kDivFastMinB));
                        float w = div_rn_fast(a2, d2);
                        w = w * w;
                        put(u, ok, x, y, z, m6 * w * w);
                    }
                }
            if (__builtin_amdgcn_ballot_w64(bad)) {
                for (int u = 0; u < U && b + u * P < npm; ++u) {
                    float4 w = o[0];  // the partner of term u (o is indexed by constants only)
#pragma unroll
                    for (int v = 1; v < U; ++v)
                        if (v == u) w = o[v];
                    const float x = w.x - c.x, y = w.y - c.y, z = w.z - c.z;
                    const float d2 = x * x + y * y + z * z;
                    const bool ok = (b + u * P + p < np) & (d2 < rc2);
                    put(u, ok, x, y, z, ok ? pair_q(d2, a2, m6, fast) : 0.0f);
                }
            }
            if (b + K < npm) gather(b + K);
            if (b + 2 * K < npm) fetch(b + 2 * K);
            wave_lds_order();
            if (p < 3) rows_add(&term[p][q][0], min(K, npm - b), acc);
            wave_lds_order();
        }
        const float fy = __shfl(acc, (lane + R) & 63), fz = __shfl(acc, (lane + 2 * R) & 63);
        if constexpr (BLK) {
            if (p == 0 && r < n) {
                pre.due = phase == 0;
                step_tail<false, true>(D, S, var, s + step, i, c, acc, fy, fz, nullptr, &pre);
                lc[((step + 1) & 1) * ldc + i] = pre.c;
                // both buffers are left as one launch per step leaves them
                if (step + 2 >= nsteps) (((s + step) & 1) ? D.coord[0] : D.coord[1])[i] = pre.c;
            }
            __syncthreads();
            lin = lc + ((step + 1) & 1) * ldc;
            if (++phase == D.stride) phase = 0;
        } else if (p == 0 && r < n) {
            float4* const cout = FO ? fout : (s & 1) ? D.coord[0] : D.coord[1];
            step_tail<FO>(D, S, var, s, i, c, acc, fy, fz, cout, FO ? nullptr : &pre);
        }
    }
    if (BLK && p == 0 && r < n) {
        D.T[i] = pre.T;
        if (noise) D.rng[i] = rng;
    }
}

// This wavefront's rows: the tile and the R rows within it.  Grid: one
// wavefront per R rows, four per workgroup; workgroups of one XCD take
// consecutive tiles.
template <int R>
__device__ __forceinline__ int2 rows_of_wave(int w) {
    constexpr int P = RowsShape<R>::P;
    const int nb = gridDim.x, nxcd = nb >= 8 ? 8 : 1;  // the grid is a multiple of 8 from 8 on
    const int gw = ((blockIdx.x % nxcd) * (nb / nxcd) + blockIdx.x / nxcd) * 4 + w;
    return make_int2(gw / P, R * (gw % P));
}

// Rows row0 .. of the job of record D and state S at its step + kstep.
template <bool FO, int R>
__device__ __forceinline__ void step_rows_of(const StepDesc& D, const DevJobState& S, int kstep, int row0,
                                             float (*term)[R][RowsShape<R>::KP], float4* __restrict__ fout) {
    const long long step0 = S.step;
    const float var = S.var;
    // the record's loads are all issued here, not each at its first use
    asm volatile("" ::"s"(D.coord[0]), "s"(D.coord[1]), "s"(D.perm), "s"(D.pair_cnt), "s"(D.pair_j), "s"(D.b_cnt),
                 "s"(D.cov_j), "s"(D.cov_r0), "s"(D.nat_j), "s"(D.nat_par), "s"(D.rng), "s"(D.T), "s"(D.bflag));
    asm volatile("" ::"s"(D.flags), "s"(D.a2), "s"(D.hOverZeta), "s"(D.nav), "s"(D.end_step), "s"(step0), "s"(var));
    const long long s = step0 + kstep;
    if (!FO && s >= D.end_step) return;
    if (row0 >= D.n) return;
    if (D.idx16)
        step_rows<FO, R, unsigned short>(D, S, var, s, row0, term, fout);
    else
        step_rows<FO, R, int>(D, S, var, s, row0, term, fout);
}

// classes: 1 the LDS-step jobs, 2 the others.  FO: forces only, into fout.
template <bool FO, int R>
__global__ __launch_bounds__(256, 4) void k_step_rows(const StepDesc* __restrict__ descs,
                                                      const DevJobState* __restrict__ st,
                                                      const int2* __restrict__ tiles, int ntiles, int kstep,
                                                      int classes, float4* __restrict__ fout) {
    __shared__ __align__(16) float terms[4][3][R][RowsShape<R>::KP];
    const int w = wave_id();
    const int2 at = rows_of_wave<R>(w);
    if (at.x >= ntiles) return;
    const int2 td = tiles[at.x];
    const StepDesc D = descs[td.x];
    if (!(classes & (D.lds_step ? 1 : 2))) return;
    step_rows_of<FO, R>(D, st[td.x], kstep, td.y + at.y, terms[w], fout);
}

// The same for a launch of one job: its record is a kernel argument and its
// tiles are counted, so that the chain of dependent reads that bounds a
// launch of few rows begins two reads later (1,000 beads, 4,000 steps: 36.8 ->
// 34.9 ms; 18,000 beads, 1,000 steps: 19.1 -> 18.7; 100,000 beads, 400 steps:
// 28.0 -> 27.5).
template <bool FO, int R>
__global__ __launch_bounds__(256, 4) void k_step_rows_one(const StepDesc D, const DevJobState* __restrict__ st,
                                                          int kstep, float4* __restrict__ fout) {
    __shared__ __align__(16) float terms[4][3][R][RowsShape<R>::KP];
    const int w = wave_id();
    const int2 at = rows_of_wave<R>(w);
    step_rows_of<FO, R>(D, *st, kstep, 64 * at.x + at.y, terms[w], fout);
}

// ---------------------------------------------------------------------------
// pairlists
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool due(const DevJob& J, long long s, int freq) {
    return s < J.end_step && (s % J.stride == 0) && (s % freq == 0);
}

__device__ __forceinline__ unsigned long long lanes_below(int lane) {
    return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// Possible pairs by the all-pairs scan, one wavefront per 64-bead tile:
// the job's beads are visited in chunks of 64 (one coordinate per lane,
// loaded once), and every bead i of the tile tests the chunk with its own
// coordinates read from the lane holding them.  The order-preserving
// ballot compaction appends the accepted j to bead i's row (bead-major,
// pp_j[i*pp_cap + k]); lane i keeps bead i's running count.  Exclusions
// (the sorted covalent/native partners) become, per chunk, a 64-bit mask
// built by lane i from its own list.  The predicate sqrtf(d^2) < threshold
// is evaluated as d^2 <= pp_d2 (the same set of floats).
__global__ __launch_bounds__(256) void k_possible(const DevJob* __restrict__ jobs, DevJobState* __restrict__ st,
                                                  const int2* __restrict__ tiles, int ntiles, int force,
                                                  int use_boxes, int skip_lds) {
    const int lane = threadIdx.x & 63;
    const TileRange tr = xcd_tiles(ntiles);
    for (int t = tr.begin; t < tr.end; t += tr.step) {
        const int2 td = tiles[t];
        const DevJob& J = jobs[td.x];
        if (use_boxes && J.tile_box) continue;  // built by k_possible_boxes
        if (skip_lds && J.lds_step && J.idx16) continue;  // built by k_possible_lds
        const long long s = st[td.x].step;
        if (!force && !due(J, s, J.pp_freq)) continue;
        const int n = J.n;
        const CoordGlobal cur{J.coord[s & 1]};
        const float d2max = J.pp_d2;
        const int cap = J.pp_cap;
        const int i0 = td.y, nrow = min(64, n - i0);
        const bool own = lane < nrow;  // lane owns bead i0 + lane
        const float4 ci = own ? cur[i0 + lane] : make_float4(0.f, 0.f, 0.f, 0.f);
        const int ne = own ? J.excl_cnt[i0 + lane] : 0;
        int pe = 0;
        int e_next = pe < ne ? J.excl_j[(size_t)pe * n + i0 + lane] : INT_MAX;
        int cnt = 0;  // lane i: entries of bead i0 + i so far
        for (int base = 0; base < n; base += 64) {
            const int j = base + lane;
            const float4 cj = j < n ? cur[j] : make_float4(0.f, 0.f, 0.f, 0.f);
            // this lane's bead: exclusions falling in [base, base + 64)
            unsigned long long ex = 0ull;
            while (e_next < base + 64) {
                ex |= 1ull << (e_next - base);
                ++pe;
                e_next = pe < ne ? J.excl_j[(size_t)pe * n + i0 + lane] : INT_MAX;
            }
            const int exlo = (int)(unsigned)ex, exhi = (int)(unsigned)(ex >> 32);
            for (int b = 0; b < nrow; ++b) {
                // bead b's coordinates, exclusion mask and count: v_readlane with
                // a uniform lane index
                const float xi = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ci.x), b));
                const float yi = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ci.y), b));
                const float zi = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ci.z), b));
                const unsigned long long exb =
                    ((unsigned long long)(unsigned)__builtin_amdgcn_readlane(exhi, b) << 32) |
                    (unsigned)__builtin_amdgcn_readlane(exlo, b);
                const float x = cj.x - xi, y = cj.y - yi, z = cj.z - zi;
                const bool ok = j < n && j != i0 + b && !((exb >> lane) & 1ull) && x * x + y * y + z * z <= d2max;
                const unsigned long long m = __builtin_amdgcn_ballot_w64(ok);
                const int c0 = __builtin_amdgcn_readlane(cnt, b);
                if (ok) {
                    const int pos = c0 + __popcll(m & lanes_below(lane));
                    if (pos < cap) list_put(J.pp_j, J.idx16, (size_t)(i0 + b) * J.pp_ld + pos, j);
                }
                if (lane == b) cnt = c0 + __popcll(m);
            }
        }
        if (own) {
            J.pp_cnt[i0 + lane] = cnt < cap ? cnt : cap;
            if (cnt > cap) atomicOr(&st[td.x].overflow, 1);
        }
    }
}

// Possible pairs of the LDS-step jobs (16-bit entries; the LDS-step bound
// keeps them far below 65,536 beads), over the step kernel's units: the
// workgroup stages the coordinates of each due job in LDS, and wavefront w
// builds the lists of the beads of the unit's rows 64w..64w+63, one bead at
// a time.  The bead is wave-uniform, so its coordinates are one broadcast
// read, its sorted exclusions (and the bead itself) become a 64-bit mask
// per chunk of candidates in scalar registers, and the accepted count is a
// scalar; the candidates j come 64 per chunk from LDS in ascending order.
// The same list in the same order as k_possible.
// Possible-list rows r0 .. r1-1 of job J (r1 > r0) by one wavefront, from
// the job's coordinates `cur` staged in LDS: each row scans the job's beads
// in chunks of 64, ballot-compacts the accepted ones in ascending order, and
// drops the bead's exclusions and itself.  Overflow sets bit 0 of *ovf.
__device__ __forceinline__ void possible_rows(const DevJob& J, const float4* __restrict__ cur, int r0, int r1,
                                              int* ovf) {
    const int lane = threadIdx.x & 63;
    const int n = J.n;
    const float d2max = J.pp_d2;
    const int cap = J.pp_cap, ecap = J.excl_cap;
    const auto ecnt = gmem(J.excl_cnt);
    const auto ej = gmem(J.excl_j);
    const auto pp = gmem(static_cast<unsigned short*>(J.pp_j));
    const auto pcnt = gmem(J.pp_cnt);
    // bead i's exclusion count and its first 64 exclusions (lane k holds
    // the k-th), loaded one bead ahead from clamped addresses
    auto load_ex = [&](int i, int& ne, int& ev) {
        ne = ecnt[i];
        ev = ej[(size_t)min(lane, ecap - 1) * n + i];
    };
    int ne_n, ev_n;
    load_ex(r0, ne_n, ev_n);
    for (int i = r0; i < r1; ++i) {
        const int ne = ne_n;
        int ev = lane < ne ? ev_n : INT_MAX;
        load_ex(min(i + 1, r1 - 1), ne_n, ev_n);
        const float4 ci = cur[i];
        const auto row = pp + (size_t)i * J.pp_ld;
        int eg = 0, pe = 0;  // exclusion group (of 64) and index within it
        int e_next = ne > 0 ? __builtin_amdgcn_readlane(ev, 0) : INT_MAX;
        int self = i;  // the bead itself, until its chunk is passed
        int cnt = 0;
        // One chunk of 64 candidates from `base` with coordinates c; TAIL:
        // the chunk may run past the job's end.  The exclusion mask is
        // formed only for chunks holding an excluded partner or the bead.
        auto chunk = [&](int base, const float4 c, bool tail) {
            const int lim = base + 64;
            const float x = c.x - ci.x, y = c.y - ci.y, z = c.z - ci.z;
            bool acc = x * x + y * y + z * z <= d2max;
            if (tail) acc = acc & (base + lane < n);
            unsigned long long m = __builtin_amdgcn_ballot_w64(acc);
            if (min(e_next, self) < lim) {
                unsigned long long drop = 0ull;
                while (e_next < lim) {
                    drop |= 1ull << (e_next - base);
                    if (++pe == 64) {
                        eg += 64;
                        pe = 0;
                        ev = eg + lane < ne ? ej[(size_t)(eg + lane) * n + i] : INT_MAX;
                    }
                    e_next = eg + pe < ne ? __builtin_amdgcn_readlane(ev, pe) : INT_MAX;
                }
                if (self < lim) {
                    drop |= 1ull << (self - base);
                    self = INT_MAX;
                }
                m &= ~drop;
                acc = acc && !((drop >> lane) & 1ull);
            }
            if (m) {
                if (acc) {
                    const unsigned pos = __builtin_amdgcn_mbcnt_hi(
                        (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, (unsigned)cnt));
                    if ((int)pos < cap)
                        *reinterpret_cast<__attribute__((address_space(1))) unsigned short*>(
                            reinterpret_cast<__attribute__((address_space(1))) char*>(row) + (pos << 1)) =
                            (unsigned short)(base + lane);
                }
                cnt += __popcll(m);
            }
        };
        int b4 = 0;
        for (; b4 + 256 <= n; b4 += 256) {  // four whole chunks, their LDS reads in flight together
            float4 c[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) c[v] = cur[b4 + 64 * v + lane];
#pragma unroll
            for (int v = 0; v < 4; ++v) chunk(b4 + 64 * v, c[v], false);
        }
        if (b4 < n) {  // the last one to four chunks
            float4 c[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) c[v] = cur[min(b4 + 64 * v + lane, n - 1)];
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (b4 + 64 * v < n) chunk(b4 + 64 * v, c[v], true);
        }
        if (lane == 0) {
            pcnt[i] = cnt < cap ? cnt : cap;
            if (cnt > cap) atomicOr(ovf, 1);
        }
    }
}

__device__ __forceinline__ bool possible_lds_wanted(const DevJob& J, long long s, int force, int use_boxes) {
    return J.lds_step && J.idx16 && !(use_boxes && J.tile_box) && (force || due(J, s, J.pp_freq));
}

__global__ __launch_bounds__(1024) void k_possible_lds(const DevJob* __restrict__ jobs, DevJobState* __restrict__ st,
                                                       const int2* __restrict__ units, const int4* __restrict__ segs,
                                                       int nunits, int force, int use_boxes) {
    extern __shared__ float4 lds_coord[];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int u = blockIdx.x; u < nunits; u += gridDim.x) {
        const int2 ud = units[u];  // first segment, segments
        __syncthreads();           // the previous unit's reads are done
        bool any = false;
        for (int q = 0; q < ud.y; ++q) {
            const int4 sg = segs[ud.x + q];
            const DevJob& J = jobs[sg.x];
            const long long s = st[sg.x].step;
            if (!possible_lds_wanted(J, s, force, use_boxes)) continue;
            any = true;
            const float4* __restrict__ g = J.coord[s & 1];
            for (int k = threadIdx.x; k < J.n; k += blockDim.x) lds_coord[sg.w + k] = g[k];
        }
        if (!any) continue;  // the same for every thread of the block
        __syncthreads();
        int t = 64 * w;
        int q = 0;
        int4 sg = make_int4(0, 0, 0, 0);
        for (; q < ud.y; ++q) {  // the segment holding this wavefront's rows
            sg = segs[ud.x + q];
            const int span = (sg.z + 63) & ~63;
            if (t < span) break;
            t -= span;
        }
        if (q == ud.y) continue;
        const DevJob& J = jobs[sg.x];
        if (!possible_lds_wanted(J, st[sg.x].step, force, use_boxes)) continue;
        possible_rows(J, lds_coord + sg.w, sg.y + t, sg.y + min(t + 64, sg.z), &st[sg.x].overflow);
    }
}

// The same lists spread for a few small jobs (the step's split_rows
// shape): four 1024-thread workgroups per 64-row tile, one wavefront per
// row, from the job's coordinates staged in LDS.  Grid: ntiles * 4.
__global__ __launch_bounds__(1024) void k_possible_split(const DevJob* __restrict__ jobs, DevJobState* __restrict__ st,
                                                         const int2* __restrict__ tiles, int ntiles, int force,
                                                         int use_boxes) {
    extern __shared__ float4 lds_coord[];
    const int tile = blockIdx.x >> 2, quarter = blockIdx.x & 3;
    if (tile >= ntiles) return;
    const int2 td = tiles[tile];
    const DevJob& J = jobs[td.x];
    const long long s = st[td.x].step;
    if (!possible_lds_wanted(J, s, force, use_boxes)) return;
    const int n = J.n, row0 = td.y + 16 * quarter;
    if (row0 >= n) return;  // every exit above is uniform over the workgroup
    {
        const float4* __restrict__ g = J.coord[s & 1];
        for (int k = threadIdx.x; k < n; k += 1024) lds_coord[k] = g[k];
    }
    __syncthreads();
    const int i = row0 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (i < n) possible_rows(J, lds_coord, i, i + 1, &st[td.x].overflow);
}

// ---------------------------------------------------------------------------
// possible pairs by bounding boxes (large jobs)
// ---------------------------------------------------------------------------
// The list of k_possible -- the same predicate on the same operands, the
// same ascending-j order -- without the tiles of 64 consecutive beads that no
// bead of a group can reach.  With lo and hi a tile's least and greatest
// coordinates, rounded subtraction, multiplication and addition are monotone,
// so max(lo.x - x, x - hi.x, 0) is at most |r_j.x - x| for each bead j of
// the tile, and the sum of the squares, formed in the order of the predicate,
// at most the predicate's: a tile that fails it holds no accepted bead.

// A tile's box, one wavefront each: J.tile_box[2t] = lo, [2t + 1] = hi.
// A coordinate that is not a number is left out (it is never accepted).
__global__ __launch_bounds__(256) void k_tile_boxes(const DevJob* __restrict__ jobs,
                                                    const DevJobState* __restrict__ st,
                                                    const int2* __restrict__ tiles, int ntiles, int force) {
    const int lane = threadIdx.x & 63;
    const TileRange tr = xcd_tiles(ntiles);
    for (int t = tr.begin; t < tr.end; t += tr.step) {
        const int2 td = tiles[t];
        const DevJob& J = jobs[td.x];
        if (!J.tile_box || J.wide) continue;
        const long long s = st[td.x].step;
        if (!force && !due(J, s, J.pp_freq)) continue;
        const CoordGlobal cur{J.coord[s & 1]};
        float4 lo = cur[min(td.y + lane, J.n - 1)], hi = lo;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            lo.x = fminf(lo.x, __shfl_xor(lo.x, o));
            lo.y = fminf(lo.y, __shfl_xor(lo.y, o));
            lo.z = fminf(lo.z, __shfl_xor(lo.z, o));
            hi.x = fmaxf(hi.x, __shfl_xor(hi.x, o));
            hi.y = fmaxf(hi.y, __shfl_xor(hi.y, o));
            hi.z = fmaxf(hi.z, __shfl_xor(hi.z, o));
        }
        if (lane < 2) J.tile_box[2 * (td.y >> 6) + lane] = lane ? hi : lo;
    }
}

// One wavefront per kBoxBeads consecutive beads.  The boxes are tested 64 at
// a time, one per lane, against each of the beads; the tiles that some bead
// reaches collect in LDS with a mask of those beads, and each such tile's
// coordinates (one contiguous 1 KB load, four tiles ahead) are tested for the
// beads in its mask: ballot, exclusions out, compaction in ascending order.
// What bounds it is the pair tests themselves, ~18 vector instructions per
// bead and near tile.  Four beads a wavefront: 76 us for 18,000 beads of a
// capsid shell (32 A threshold, ~1,000 entries a bead) and 340 us for 100,000;
// eight take 108 and 345 (too few wavefronts for the smaller), two 76 and 380.
// Taking the candidates bead by bead from a cell grid and sorting the accepted
// ones through a bitmap of the job's beads takes 947 and 2,283 us.  Beads in no
// spatial order along the chain make every box span the job: past kWideTiles
// tiles in reach such jobs take the grid (k_possible_cells).
constexpr int kBoxBeads = 4;
constexpr int kBoxAhead = 4;
constexpr int kBoxList = 256;  // collected tiles before they are worked off
constexpr int kBoxSample = 8;  // one group of beads in so many tiles is sampled
__global__ __launch_bounds__(256) void k_possible_boxes(const DevJob* __restrict__ jobs,
                                                        DevJobState* __restrict__ st,
                                                        const int2* __restrict__ tiles, int ntiles, int force) {
    __shared__ unsigned near_tiles[4][kBoxList + 64];  // tile << 8 | beads
    const int lane = threadIdx.x & 63, wv = wave_id();
    volatile unsigned* const list = near_tiles[wv];
    constexpr int kUnits = 64 / kBoxBeads;  // per tile
    const int nunits = kUnits * ntiles;
    const int nb = gridDim.x, nxcd = nb >= 8 ? 8 : 1;
    const int slice = (nunits + nxcd - 1) / nxcd;
    const int xcd = blockIdx.x % nxcd;
    const int hend = min((xcd + 1) * slice, nunits);
    for (int h = xcd * slice + 4 * (int)(blockIdx.x / nxcd) + wv; h < hend; h += 4 * (nb / nxcd)) {
        const int2 td = tiles[h / kUnits];
        const DevJob& J = jobs[td.x];
        if (!J.tile_box || J.wide) continue;
        const long long s = st[td.x].step;
        if (!force && !due(J, s, J.pp_freq)) continue;
        const int n = J.n, nt = (n + 63) >> 6;
        const int i0 = td.y + kBoxBeads * (h % kUnits);
        if (i0 >= n) continue;
        const int nbead = min(kBoxBeads, n - i0);
        const CoordGlobal cur{J.coord[s & 1]}, box{J.tile_box};
        const auto ej = gmem(J.excl_j);
        const float d2max = J.pp_d2;
        const int cap = J.pp_cap, ecap = J.excl_cap, idx16 = J.idx16, ld = J.pp_ld;
        void* const pp = J.pp_j;
        // lanes' beads: coordinates and exclusion counts of i0 + lane % kBoxBeads
        const int il = min(i0 + lane % kBoxBeads, n - 1);
        const float4 rl = cur[il];
        const int nel = gmem(J.excl_cnt)[il];
        float4 lo = box[2 * min(lane, nt - 1)], hi = box[2 * min(lane, nt - 1) + 1];
        int ev[kBoxBeads];  // lane k: the bead's k-th exclusion, -1 past the last
#pragma unroll
        for (int b = 0; b < kBoxBeads; ++b) ev[b] = ej[(size_t)min(lane, ecap - 1) * n + min(i0 + b, n - 1)];
        float px[kBoxBeads], py[kBoxBeads], pz[kBoxBeads];
        int ne[kBoxBeads], cnt[kBoxBeads];
        int most = 0;
#pragma unroll
        for (int b = 0; b < kBoxBeads; ++b) {
            px[b] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(rl.x), b));
            py[b] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(rl.y), b));
            pz[b] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(rl.z), b));
            ne[b] = __builtin_amdgcn_readlane(nel, b);
            ev[b] = lane < ne[b] ? ev[b] : -1;
            cnt[b] = 0;
            most = max(most, ne[b]);
        }
        // candidates of tile e >> 8 (coordinates c) for the beads in e
        auto scan = [&](unsigned e, float4 c) {
            const int base = (int)(e >> 8) << 6;
            if (base + 64 > n && base + lane >= n) c.x = __builtin_nanf("");
#pragma unroll
            for (int b = 0; b < kBoxBeads; ++b) {
                if (!((e >> b) & 1u)) continue;
                const float x = c.x - px[b], y = c.y - py[b], z = c.z - pz[b];
                bool acc = x * x + y * y + z * z <= d2max;
                unsigned long long m = __builtin_amdgcn_ballot_w64(acc);
                unsigned long long hit = __builtin_amdgcn_ballot_w64((unsigned)(ev[b] ^ base) < 64u);
                if (hit | (unsigned long long)(base == td.y) | (unsigned long long)(most > 64)) {
                    unsigned long long drop = base == td.y ? 1ull << (i0 + b - base) : 0ull;
                    while (hit) {
                        const int q = __builtin_ctzll(hit);
                        hit &= hit - 1ull;
                        drop |= 1ull << (__builtin_amdgcn_readlane(ev[b], q) & 63);
                    }
                    for (int g = 64; g < ne[b]; g += 64) {  // exclusions past the 64th
                        const int v = g + lane < ne[b] ? ej[(size_t)(g + lane) * n + i0 + b] : -1;
                        unsigned long long far = __builtin_amdgcn_ballot_w64((unsigned)(v ^ base) < 64u);
                        while (far) {
                            const int q = __builtin_ctzll(far);
                            far &= far - 1ull;
                            drop |= 1ull << (__builtin_amdgcn_readlane(v, q) & 63);
                        }
                    }
                    m &= ~drop;
                    acc = acc && !((drop >> lane) & 1ull);
                }
                if (acc) {
                    const int pos = (int)__builtin_amdgcn_mbcnt_hi(
                        (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, (unsigned)cnt[b]));
                    if (pos < cap) {
                        if (idx16)
                            (gmem(static_cast<unsigned short*>(pp)) + (size_t)(i0 + b) * ld)[pos] =
                                (unsigned short)(base + lane);
                        else
                            (gmem(static_cast<int*>(pp)) + (size_t)(i0 + b) * ld)[pos] = base + lane;
                    }
                }
                cnt[b] += __popcll(m);
            }
        };
        int m = 0, reached = 0;  // collected tiles, and all of them
        for (int c0 = 0; c0 < nt; c0 += 64) {
            const int cn = min(c0 + 64 + lane, nt - 1);
            const float4 lon = box[2 * cn], hin = box[2 * cn + 1];
            unsigned mask = 0u;
#pragma unroll
            for (int b = 0; b < kBoxBeads; ++b) {
                const float x = fmaxf(fmaxf(lo.x - px[b], px[b] - hi.x), 0.0f);
                const float y = fmaxf(fmaxf(lo.y - py[b], py[b] - hi.y), 0.0f);
                const float z = fmaxf(fmaxf(lo.z - pz[b], pz[b] - hi.z), 0.0f);
                mask |= x * x + y * y + z * z <= d2max ? 1u << b : 0u;
            }
            mask &= c0 + lane < nt ? (1u << nbead) - 1u : 0u;
            const unsigned long long some = __builtin_amdgcn_ballot_w64(mask != 0u);
            if (mask)
                list[__builtin_amdgcn_mbcnt_hi((unsigned)(some >> 32),
                                               __builtin_amdgcn_mbcnt_lo((unsigned)some, (unsigned)m))] =
                    (unsigned)(c0 + lane) << 8 | mask;
            m += __popcll(some);
            reached += __popcll(some);
            lo = lon;
            hi = hin;
            if (m == 0 || (m < kBoxList && c0 + 64 < nt)) continue;
            wave_lds_order();
            unsigned e[kBoxAhead];
            float4 c[kBoxAhead];
            auto load = [&](int q) {
#pragma unroll
                for (int u = 0; u < kBoxAhead; ++u) {
                    e[u] = __builtin_amdgcn_readfirstlane(list[min(q + u, m - 1)]);
                    c[u] = cur[min(((int)(e[u] >> 8) << 6) + lane, n - 1)];
                }
            };
            load(0);
            for (int q = 0; q < m; q += kBoxAhead) {
                unsigned eq[kBoxAhead];
                float4 cq[kBoxAhead];
#pragma unroll
                for (int u = 0; u < kBoxAhead; ++u) eq[u] = e[u], cq[u] = c[u];
                load(q + kBoxAhead);
#pragma unroll
                for (int u = 0; u < kBoxAhead; ++u)
                    if (q + u < m) scan(eq[u], cq[u]);
            }
            wave_lds_order();
            m = 0;
        }
        int total = cnt[0];
#pragma unroll
        for (int b = 1; b < kBoxBeads; ++b) total = lane == b ? cnt[b] : total;
        // a sample of the tiles that a group reaches, for the host's choice of the
        // jobs that take the cell grid (Engine::judge_wide)
        if (h % (kBoxSample * kUnits) == 0 && lane == 0) {
            atomicAdd(&st[td.x].near_tiles, (unsigned long long)reached);
            atomicAdd(&st[td.x].near_groups, 1ull);
        }
        if (lane < nbead) {
            J.pp_cnt[i0 + lane] = min(total, cap);
            if (total > cap) atomicOr(&st[td.x].overflow, 1);
        }
    }
}

// ---------------------------------------------------------------------------
// possible pairs by a cell grid (large jobs of beads in no spatial order)
// ---------------------------------------------------------------------------
// The list of k_possible -- the same predicate on the same operands, the
// same ascending-j order -- from the candidates in the 27 cells around the
// bead, for the jobs whose beads lie in no spatial order along the chain
// (J.wide): every box of 64 consecutive beads then spans the job, and
// k_possible_boxes scans all pairs.  Cells are cubes of edge thr*(1+1e-4) +
// 0.01 A + 2^-20 of the job's extent: a pair with sqrtf(d^2) < thr has every
// |coordinate difference| within thr*(1 + 2^-21), and the cell index
// (x - x0) / edge is computed with an error below the margin, so such a pair
// always lies in adjacent cells.  Accepted j are set in a per-wave LDS bitmap
// over the job's beads, the bead's exclusions cleared, and the bitmap read back
// in index order with a wave prefix sum of popcounts.  Bound by the two LDS
// atomics per accepted pair.  Measurements beside kWideTiles.

__device__ __forceinline__ int cell_axis(float x, float org, float inv, int dim) {
    const float q = (x - org) * inv;
    if (!(q >= 0.0f)) return 0;  // below the grid, or NaN
    if (q >= (float)dim) return dim - 1;
    return min((int)q, dim - 1);
}

__device__ __forceinline__ int wave_min(int v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o));
    return v;
}
__device__ __forceinline__ int wave_max(int v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o));
    return v;
}
__device__ __forceinline__ int wave_inclusive_sum(int v, int lane) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(v, o);
        if (lane >= o) v += u;
    }
    return v;
}

// Per job (one 1024-thread block each): bounding box of the coordinates,
// the grid (edge grown until the cell count fits cell_cap), zeroed counts.
__global__ __launch_bounds__(1024) void k_cells_setup(const DevJob* __restrict__ jobs, DevJobState* __restrict__ st,
                                                      int njobs, int force) {
    const int jb = blockIdx.x;
    if (jb >= njobs) return;
    const DevJob& J = jobs[jb];
    if (!J.wide) return;
    DevJobState& S = st[jb];
    const long long s = S.step;
    if (!force && !due(J, s, J.pp_freq)) return;
    const float4* __restrict__ cur = J.coord[s & 1];
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int i = threadIdx.x; i < J.n; i += blockDim.x) {
        const float4 r = cur[i];
        lo[0] = fminf(lo[0], r.x), hi[0] = fmaxf(hi[0], r.x);
        lo[1] = fminf(lo[1], r.y), hi[1] = fmaxf(hi[1], r.y);
        lo[2] = fminf(lo[2], r.z), hi[2] = fmaxf(hi[2], r.z);
    }
    __shared__ float red[6][16];
    __shared__ int dims[4];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        float a = lo[d], b = hi[d];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            a = fminf(a, __shfl_xor(a, o));
            b = fmaxf(b, __shfl_xor(b, o));
        }
        if (lane == 0) {
            red[d][w] = a;
            red[3 + d][w] = b;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const int nw = blockDim.x >> 6;
        float org[3], ext[3];
        for (int d = 0; d < 3; ++d) {
            float a = red[d][0], b = red[3 + d][0];
            for (int k = 1; k < nw; ++k) a = fminf(a, red[d][k]), b = fmaxf(b, red[3 + d][k]);
            org[d] = a;
            ext[d] = b - a;
        }
        int dm[3] = {1, 1, 1};
        const bool finite = isfinite(ext[0]) && isfinite(ext[1]) && isfinite(ext[2]);
        // the last term covers the rounding of x - x0 and of its product
        float edge = J.pp_thr * 1.0001f + 0.01f + 0x1p-20f * fmaxf(fmaxf(ext[0], ext[1]), ext[2]);
        if (finite) {
            for (int it = 0; it < 200; ++it) {
                double cells = 1.0;
                for (int d = 0; d < 3; ++d) cells *= floor((double)ext[d] / edge) + 1.0;
                if (cells <= (double)J.cell_cap) break;
                edge *= 1.1f;
            }
            for (int d = 0; d < 3; ++d) dm[d] = (int)floor((double)ext[d] / edge) + 1;
            if ((long long)dm[0] * dm[1] * dm[2] > J.cell_cap) dm[0] = dm[1] = dm[2] = 1;
        } else {
            org[0] = org[1] = org[2] = 0.0f;
        }
        for (int d = 0; d < 3; ++d) {
            S.cell_org[d] = org[d];
            S.cell_dim[d] = dm[d];
        }
        S.cell_inv = 1.0f / edge;
        dims[0] = dm[0] * dm[1] * dm[2];
    }
    __syncthreads();
    const int nc = dims[0];
    for (int c = threadIdx.x; c < nc; c += blockDim.x) J.cell_cnt[c] = 0;
}

// Each bead's cell and its slot there (the order within a cell is free:
// the bitmap restores index order).
__global__ __launch_bounds__(256) void k_cells_count(const DevJob* __restrict__ jobs, DevJobState* __restrict__ st,
                                                     const int2* __restrict__ tiles, int ntiles, int force) {
    const int lane = threadIdx.x & 63;
    const TileRange tr = xcd_tiles(ntiles);
    for (int t = tr.begin; t < tr.end; t += tr.step) {
        const int2 td = tiles[t];
        const DevJob& J = jobs[td.x];
        if (!J.wide) continue;
        const DevJobState& S = st[td.x];
        const long long s = S.step;
        if (!force && !due(J, s, J.pp_freq)) continue;
        const int i = td.y + lane;
        if (i >= J.n) continue;
        const float4 r = J.coord[s & 1][i];
        const int cx = cell_axis(r.x, S.cell_org[0], S.cell_inv, S.cell_dim[0]);
        const int cy = cell_axis(r.y, S.cell_org[1], S.cell_inv, S.cell_dim[1]);
        const int cz = cell_axis(r.z, S.cell_org[2], S.cell_inv, S.cell_dim[2]);
        const int c = (cz * S.cell_dim[1] + cy) * S.cell_dim[0] + cx;
        J.bead_cell[i] = c;
        J.bead_slot[i] = atomicAdd(&J.cell_cnt[c], 1);
    }
}

// Exclusive scan of the cell counts (one 1024-thread block per job).
__global__ __launch_bounds__(1024) void k_cells_scan(const DevJob* __restrict__ jobs, DevJobState* __restrict__ st,
                                                     int njobs, int force) {
    const int jb = blockIdx.x;
    if (jb >= njobs) return;
    const DevJob& J = jobs[jb];
    if (!J.wide) return;
    const DevJobState& S = st[jb];
    if (!force && !due(J, S.step, J.pp_freq)) return;
    const int nc = S.cell_dim[0] * S.cell_dim[1] * S.cell_dim[2];
    const int per = (nc + blockDim.x - 1) / blockDim.x;
    const int b = threadIdx.x * per, e = min(b + per, nc);
    int sum = 0;
    for (int c = b; c < e; ++c) sum += J.cell_cnt[c];
    __shared__ int part[1024];
    part[threadIdx.x] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        int acc = 0;
        for (int k = 0; k < (int)blockDim.x; ++k) {
            const int v = part[k];
            part[k] = acc;
            acc += v;
        }
    }
    __syncthreads();
    int acc = part[threadIdx.x];
    for (int c = b; c < e; ++c) {
        J.cell_start[c] = acc;
        acc += J.cell_cnt[c];
    }
    if (threadIdx.x == 0) J.cell_start[nc] = J.n;
}

__global__ __launch_bounds__(256) void k_cells_fill(const DevJob* __restrict__ jobs, DevJobState* __restrict__ st,
                                                    const int2* __restrict__ tiles, int ntiles, int force) {
    const int lane = threadIdx.x & 63;
    const TileRange tr = xcd_tiles(ntiles);
    for (int t = tr.begin; t < tr.end; t += tr.step) {
        const int2 td = tiles[t];
        const DevJob& J = jobs[td.x];
        if (!J.wide) continue;
        if (!force && !due(J, st[td.x].step, J.pp_freq)) continue;
        const int i = td.y + lane;
        if (i >= J.n) continue;
        J.cell_beads[J.cell_start[J.bead_cell[i]] + J.bead_slot[i]] = i;
    }
}

// One 64-thread workgroup (one wavefront) per tile; dynamic LDS holds the
// bitmap of ceil(n/64) words for the largest cell-binned job.
// One wavefront per half tile (32 beads), its beads one after another.  A bead's
// candidates (the 3 x 3 rows of three x-adjacent cells, each row one
// contiguous range of cell_beads) are read eight 64-entry chunks at a time,
// all index loads and then all coordinate gathers in flight together; the
// next bead's coordinates and first 64 exclusions are loaded while this one
// is scanned.  Accepted j set bit j of the LDS bitmap bm and bit j / 64 of
// bm2, so the read-back in index order visits only the 64-word blocks of bm
// that hold an entry.
constexpr int kCellChunks = 8;
__global__ __launch_bounds__(64) void k_possible_cells(const DevJob* __restrict__ jobs, DevJobState* __restrict__ st,
                                                       const int2* __restrict__ tiles, int ntiles, int force,
                                                       int cell_words) {
    extern __shared__ unsigned long long bm[];
    unsigned long long* const bm2 = bm + cell_words;  // one bit per word of bm
    const int lane = threadIdx.x;
    const int nb = gridDim.x, nxcd = nb >= 8 ? 8 : 1;
    const int nhalf = 2 * ntiles;  // work units: the two halves of every tile
    const int slice = (nhalf + nxcd - 1) / nxcd;
    const int xcd = blockIdx.x % nxcd;
    const int hend = min((xcd + 1) * slice, nhalf);
    for (int h = xcd * slice + blockIdx.x / nxcd; h < hend; h += nb / nxcd) {
        const int2 td = tiles[h >> 1];
        const DevJob& J = jobs[td.x];
        if (!J.wide) continue;
        const DevJobState& S = st[td.x];
        const long long s = S.step;
        if (!force && !due(J, s, J.pp_freq)) continue;
        const int n = J.n;
        const int i0 = td.y + 32 * (h & 1);
        if (i0 >= n) continue;
        const int nwords = (n + 63) >> 6;
        for (int w = lane; w < nwords; w += 64) bm[w] = 0ull;
        for (int w = lane; w < (nwords + 63) >> 6; w += 64) bm2[w] = 0ull;
        __syncthreads();
        const CoordGlobal cur{J.coord[s & 1]};
        const auto cbeads = gmem(J.cell_beads);
        const auto cstart = gmem(J.cell_start);
        const auto ecnt = gmem(J.excl_cnt);
        const auto ej = gmem(J.excl_j);
        const float d2max = J.pp_d2;
        const int cap = J.pp_cap, ecap = J.excl_cap;
        const int dx = S.cell_dim[0], dy = S.cell_dim[1], dz = S.cell_dim[2];
        const int iend = min(i0 + 32, n);
        float4 r1n = cur[i0];
        int nen = ecnt[i0];
        int evn = ej[(size_t)min(lane, ecap - 1) * n + i0];
        for (int i = i0; i < iend; ++i) {
            const float4 r1 = r1n;
            const int ne = nen, ev = evn;
            if (i + 1 < iend) {
                r1n = cur[i + 1];
                nen = ecnt[i + 1];
                evn = ej[(size_t)min(lane, ecap - 1) * n + i + 1];
            }
            const int cx = cell_axis(r1.x, S.cell_org[0], S.cell_inv, dx);
            const int cy = cell_axis(r1.y, S.cell_org[1], S.cell_inv, dy);
            const int cz = cell_axis(r1.z, S.cell_org[2], S.cell_inv, dz);
            int jlo = INT_MAX, jhi = -1;
            for (int z = max(cz - 1, 0); z <= min(cz + 1, dz - 1); ++z)
                for (int y = max(cy - 1, 0); y <= min(cy + 1, dy - 1); ++y) {
                    const int row = (z * dy + y) * dx;
                    // the cells x-1..x+1 of one row are contiguous in cell_beads
                    const int b = cstart[row + max(cx - 1, 0)];
                    const int e = cstart[row + min(cx + 1, dx - 1) + 1];
                    for (int k0 = b; k0 < e; k0 += 64 * kCellChunks) {
                        int jj[kCellChunks];
#pragma unroll
                        for (int u = 0; u < kCellChunks; ++u) {
                            const int k = k0 + 64 * u + lane;
                            jj[u] = k < e ? cbeads[k] : i;  // past the range: the bead itself, skipped
                        }
                        float4 r2[kCellChunks];
#pragma unroll
                        for (int u = 0; u < kCellChunks; ++u) r2[u] = cur[jj[u]];
#pragma unroll
                        for (int u = 0; u < kCellChunks; ++u) {
                            const int j = jj[u];
                            const float x = r2[u].x - r1.x, y2 = r2[u].y - r1.y, z2 = r2[u].z - r1.z;
                            if (j != i && x * x + y2 * y2 + z2 * z2 <= d2max) {
                                atomicOr(&bm[j >> 6], 1ull << (j & 63));
                                atomicOr(&bm2[j >> 12], 1ull << ((j >> 6) & 63));
                                jlo = min(jlo, j);
                                jhi = max(jhi, j);
                            }
                        }
                    }
                }
            __syncthreads();
            for (int k = lane; k < ne; k += 64) {
                const int e = k < 64 ? ev : ej[(size_t)k * n + i];
                atomicAnd(&bm[e >> 6], ~(1ull << (e & 63)));
            }
            __syncthreads();
            jlo = wave_min(jlo);
            jhi = wave_max(jhi);
            int cnt = 0;
            const size_t rowp = (size_t)i * J.pp_ld;
            if (jhi >= 0) {
                const int wlo = jlo >> 6, whi = jhi >> 6;
                for (int wb = wlo & ~63; wb <= whi; wb += 64) {
                    const unsigned long long m2 = bm2[wb >> 6];
                    if (m2 == 0ull) continue;  // no entry in these 64 words
                    const int w = wb + lane;
                    unsigned long long word = 0ull;
                    if ((m2 >> lane) & 1ull) {
                        word = bm[w];
                        bm[w] = 0ull;
                    }
                    const int pc = __popcll(word);
                    const int incl = wave_inclusive_sum(pc, lane);
                    int pos = cnt + incl - pc;
                    while (word) {
                        const int j = (w << 6) + __builtin_ctzll(word);
                        if (pos < cap) list_put(J.pp_j, J.idx16, rowp + pos, j);
                        ++pos;
                        word &= word - 1ull;
                    }
                    cnt += __shfl(incl, 63);
                    if (lane == 0) bm2[wb >> 6] = 0ull;
                }
            }
            __syncthreads();
            if (lane == 0) {
                J.pp_cnt[i] = cnt < cap ? cnt : cap;
                if (cnt > cap) atomicOr(&st[td.x].overflow, 1);
            }
        }
    }
}

// Verlet list: one 1024-thread workgroup per tile of 64 list rows (the
// beads perm[row]).  Wave w filters the possible lists of the beads of rows
// 4w..4w+3 in stored order with the ballot compaction; the accepted
// entries of the tile collect in LDS rows, and the workgroup then writes
// them out slot-major (pair_j[k*n + row]) so each store covers the 64 rows
// of one slot.  A bead's row is read eight 64-entry
// chunks at a time: all eight index loads, then all eight coordinate
// gathers, are in flight before the first compare.  Entries past the LDS
// row (VerletLds::entries) are rare and stored to their slot directly.
template <typename IdxT>
struct VerletLds;
template <>
struct VerletLds<unsigned short> {  // 256 entries per bead, rows padded by one bank
    static constexpr int entries = 256, stride = 258;
};
template <>
struct VerletLds<int> {
    static constexpr int entries = 255, stride = 256;
};

// w: this wavefront's index among the WAVES wavefronts that build the tile.
// CH: chunks of 64 possible-list entries whose loads are in flight together.
// cur: the job's coordinates (staged in LDS, or a CoordGlobal).
template <typename IdxT, int WAVES, int CH = 8, typename CP = const float4*>
__device__ __forceinline__ void verlet_tile(const DevJob& J, DevJobState& S, CP cur, int i0,
                                            IdxT* __restrict__ rows, int* __restrict__ cnt_s, int w) {
    constexpr int E = VerletLds<IdxT>::entries, RS = VerletLds<IdxT>::stride;
    constexpr int RPW = 64 / WAVES;  // rows per wave
    const int lane = threadIdx.x & 63;
    const int n = J.n;
    const int nrow = min(64, n - i0);
    w = __builtin_amdgcn_readfirstlane(w);
    const int b_lo = RPW * w, b_hi = min(b_lo + RPW, nrow);
    const float d2max = J.pl_d2;  // sqrtf(d2) < pl_cut, exactly
    const int cap = J.pair_cap, ppcap = J.pp_cap, ppld = J.pp_ld;
    const auto pp = gmem(static_cast<const IdxT*>(J.pp_j));
    const auto pj = gmem(static_cast<IdxT*>(J.pair_j));
    // beads of the tile's rows and their possible counts (loads issued
    // unconditionally, from clamped addresses, so that no branch leaves a
    // load pending on one path only)
    const int bl0 = gmem(J.perm)[i0 + min(lane, nrow - 1)];
    const int cl0 = gmem(J.pp_cnt)[bl0];
    const int bl = lane < nrow ? bl0 : 0;
    const int cl = lane < nrow ? cl0 : 0;
    // row b's bead and count (b is wave-uniform: a lane read, not a shuffle)
    auto bead_of = [&](int b) { return __builtin_amdgcn_readlane(bl, b); };
    auto count_of = [&](int b) { return __builtin_amdgcn_readlane(cl, b); };
    // Raw words of 64 CH entries of row b from `base`, loaded without a
    // branch from addresses clamped into the row; the filter replaces the
    // words past the row's count by 0 (a valid bead) and rejects them.
    auto load_idx = [&](int b, int base, int (&j)[CH]) {
        const auto row = pp + (size_t)bead_of(b) * ppld;
#pragma unroll
        for (int u = 0; u < CH; ++u) j[u] = (int)row[(unsigned)min(base + 64 * u + lane, ppcap - 1)];
    };
    // One chunk: gather, compare, and compact the accepted entries in order
    // into the row's LDS entries (or, past them, their slots).  Gathers go
    // out four at a time.
    auto filter = [&](int b, const float4 r1, int npp, int base, int (&j)[CH], int& cnt) {
#pragma unroll
        for (int u = 0; u < CH; ++u) j[u] = base + 64 * u + lane < npp ? j[u] : 0;
#pragma unroll
        for (int h = 0; h < CH; h += 4) {
            float4 c[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) c[u] = cur[j[h + u]];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int k0 = base + 64 * (h + u);
                if (k0 < npp) {
                    const float x = c[u].x - r1.x, y = c[u].y - r1.y, z = c[u].z - r1.z;
                    const bool ok = (k0 + lane < npp) & (x * x + y * y + z * z <= d2max);
                    const unsigned long long m = __builtin_amdgcn_ballot_w64(ok);
                    const int total = cnt + __popcll(m);
                    if (ok) {
                        const int pos = (int)__builtin_amdgcn_mbcnt_hi(
                            (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, (unsigned)cnt));
                        if (total <= E || pos < E) rows[b * RS + pos] = (IdxT)j[h + u];
                        else if (pos < cap) pj[(size_t)pos * J.pair_ld + i0 + b] = (IdxT)j[h + u];
                    }
                    cnt = total;
                }
            }
        }
    };
    // Row b from its first chunk of indices j (loaded ahead); a second chunk
    // is loaded before the first is filtered, further ones as they come.
    auto do_row = [&](int b, int (&j)[CH], const float4 r1) {
        const int npp = count_of(b);
        int cnt = 0;
        int j2[CH];
        const bool two = npp > 64 * CH;
        if (two) load_idx(b, 64 * CH, j2);
        filter(b, r1, npp, 0, j, cnt);
        if (two) {
            filter(b, r1, npp, 64 * CH, j2, cnt);
            for (int base = 128 * CH; base < npp; base += 64 * CH) {
                int j3[CH];
                load_idx(b, base, j3);
                filter(b, r1, npp, base, j3, cnt);
            }
        }
        if (lane == 0) {
            cnt_s[b] = cnt;
            if (cnt > cap) atomicOr(&S.overflow, 2);
        }
    };
    // first chunk and centre of row b (rows past the wave's last load that
    // row's again, unused: no branch)
    auto ahead = [&](int b, int (&j)[CH], float4& r1) {
        b = min(b, b_hi - 1);
        load_idx(b, 0, j);
        r1 = cur[bead_of(b)];
    };
    // The wave's rows as straight-line code (the row loop fully unrolled),
    // a software pipeline two rows deep: while row b is filtered the first
    // chunk of row b+1 is in flight, and row b+2's is issued as soon as row
    // b is done with its registers.  Unrolled, every prefetch has registers
    // of its own and the loads can be waited for one by one.
    if (b_lo >= b_hi) return;
    constexpr int D = RPW < 2 ? 1 : 2;
    int js[D][CH];
    float4 rs[D];
#pragma unroll
    for (int q = 0; q < D; ++q) ahead(b_lo + q, js[q], rs[q]);
#pragma unroll
    for (int q = 0; q < RPW; ++q) {
        const int b = b_lo + q;
        if (b < b_hi) {
            do_row(b, js[q % D], rs[q % D]);
            if (q + D < RPW) ahead(b + D, js[q % D], rs[q % D]);
        }
    }
}

// t: this thread's index among the 64 WAVES threads that store the tile.
template <typename IdxT, int WAVES>
__device__ __forceinline__ void verlet_store(const DevJob& J, int i0, const IdxT* __restrict__ rows,
                                             const int* __restrict__ cnt_s, int t) {
    constexpr int E = VerletLds<IdxT>::entries, RS = VerletLds<IdxT>::stride;
    const int n = J.n, cap = J.pair_cap;
    const int nrow = min(64, n - i0);
    const int b = t & 63, kq = t >> 6;
    const int c = b < nrow ? cnt_s[b] : 0;
    if (b < nrow) {
        if (kq == 0) J.pair_cnt[i0 + b] = c < cap ? c : cap;
    }
    int maxc = min(c, E);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) maxc = max(maxc, __shfl_xor(maxc, o));
    // the four waves' maxima differ only in which beads they saw: all waves
    // see all 64 beads here (b = lane), so maxc is the tile's
    const auto pj = gmem(static_cast<IdxT*>(J.pair_j));
    // a row that outgrew its capacity (flag bit 2 is set) stores only its
    // first cap entries: pair_j holds pair_cap slots
    const int lim = min(c, min(E, cap));
    for (int k = kq; k < maxc; k += WAVES)
        if (k < lim) pj[(size_t)k * J.pair_ld + i0 + b] = rows[b * RS + k];
}

// Re-sorts the rows of each kLdsUnit-row unit of a job by Verlet list
// length (longest first, ties by bead), just before the rebuild that fills
// the rows again, with the lengths of the last rebuild as keys: the 64 rows
// of a wavefront then hold lists of about the same length, so its loop
// over the longest list idles few lanes and reads few padding slots.  Only
// which row and lane serve a bead changes, never the arithmetic, so the
// trajectories are the same bits in any row order.  Bitonic sort in LDS.
// The sort also moves each bead's bonded lists to its new row (the step
// reads them in row order), so it runs at every kSortEvery-th Verlet
// rebuild only: list lengths drift little in between.
__global__ __launch_bounds__(1024) void k_sort_rows(const DevJob* __restrict__ jobs, const DevJobState* __restrict__ st,
                                                    const int2* __restrict__ units, int nunits, int sort_every,
                                                    int force) {
    __shared__ unsigned long long key[kLdsUnit];
    const int t = threadIdx.x;
    for (int u = blockIdx.x; u < nunits; u += gridDim.x) {
        const int2 ud = units[u];
        const DevJob& J = jobs[ud.x];
        if (!J.sort_rows) continue;
        if (!force && !due(J, st[ud.x].step, J.pairs_freq * sort_every)) continue;  // a Verlet rebuild step
        const int m = min(kLdsUnit, J.n - ud.y), r = ud.y + t;
        __syncthreads();  // the previous unit's keys are read
        key[t] = t < m ? ((unsigned long long)(unsigned)(J.pair_cap - J.pair_cnt[r]) << 32) | (unsigned)J.perm[r]
                       : ~0ull;
        __syncthreads();
        for (int k = 2; k <= kLdsUnit; k <<= 1)
            for (int j = k >> 1; j > 0; j >>= 1) {
                const int q = t ^ j;
                if (q > t) {
                    const unsigned long long a = key[t], b = key[q];
                    if ((a > b) == ((t & k) == 0)) {
                        key[t] = b;
                        key[q] = a;
                    }
                }
                __syncthreads();
            }
        if (t < m) {
            // row r now steps bead i: its bonded lists move to row r
            const int i = (int)(unsigned)(key[t] & 0xffffffffull);
            J.perm[r] = i;
            const int n = J.n, ld = J.pair_ld;
            const int nc = J.cov_cnt[i], nn = J.nat_cnt[i];
            J.rb_cnt[r] = nc | (nn << 16);
            for (int k = 0; k < nc; ++k) {
                J.rb_cov_j[(size_t)k * ld + r] = J.cov_j16[(size_t)k * n + i];
                J.rb_cov_r0[(size_t)k * ld + r] = J.cov_r0[(size_t)k * n + i];
            }
            for (int k = 0; k < nn; ++k) {
                J.rb_nat_j[(size_t)k * ld + r] = J.nat_j16[(size_t)k * n + i];
                J.rb_nat_par[(size_t)k * ld + r] = J.nat_par[(size_t)k * n + i];
            }
        }
    }
}

// Wavefronts per 64-row tile of k_verlet (four rows each): sixteen, so that
// the latency of the L2 gathers is hidden by the other wavefronts of the CU.
constexpr int kVerletWaves = 16;
__global__ __launch_bounds__(1024) void k_verlet(const DevJob* __restrict__ jobs, DevJobState* __restrict__ st,
                                                 const int2* __restrict__ tiles, int ntiles, int force, int skip_lds) {
    extern __shared__ __attribute__((aligned(16))) int lds_rows[];  // 64 rows of uint16 or int32 entries
    __shared__ int cnt_s[64];
    const int nb = gridDim.x, nxcd = nb >= 8 ? 8 : 1;
    const int slice = (ntiles + nxcd - 1) / nxcd;
    const int xcd = blockIdx.x % nxcd;
    const int tend = min((xcd + 1) * slice, ntiles);
    for (int t = xcd * slice + blockIdx.x / nxcd; t < tend; t += nb / nxcd) {
        const int2 td = tiles[t];
        const DevJob& J = jobs[td.x];
        DevJobState& S = st[td.x];
        const long long s = S.step;
        if (!force && !due(J, s, J.pairs_freq)) continue;
        if (skip_lds && J.lds_step) continue;  // built by k_verlet_lds
        const CoordGlobal cur{J.coord[s & 1]};
        const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        if (J.idx16)
            verlet_tile<unsigned short, kVerletWaves>(J, S, cur, td.y, reinterpret_cast<unsigned short*>(lds_rows),
                                                      cnt_s, w);
        else
            verlet_tile<int, kVerletWaves>(J, S, cur, td.y, lds_rows, cnt_s, w);
        __syncthreads();
        if (J.idx16)
            verlet_store<unsigned short, kVerletWaves>(J, td.y, reinterpret_cast<const unsigned short*>(lds_rows),
                                                       cnt_s, threadIdx.x);
        else
            verlet_store<int, kVerletWaves>(J, td.y, static_cast<const int*>(lds_rows), cnt_s, threadIdx.x);
        __syncthreads();
    }
}

// The Verlet build of the LDS-step jobs, over the step kernel's units: the
// workgroup stages the coordinates of each job it serves in LDS, so the
// candidate gathers read LDS instead of L2, then builds the unit's rows two
// 64-row tiles at a time (wavefronts 0-7 one tile, 8-15 the other, eight
// rows each) and writes each tile slot-major as k_verlet does.  Same
// lists, same order.
constexpr int kVerletRowsBytes = 64 * VerletLds<unsigned short>::stride * 2;
template <int CH>
__global__ __launch_bounds__(1024) void k_verlet_lds(const DevJob* __restrict__ jobs, DevJobState* __restrict__ st,
                                                     const int2* __restrict__ units, const int4* __restrict__ segs,
                                                     int nunits, int force) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    float4* coords = reinterpret_cast<float4*>(lds_raw + 2 * kVerletRowsBytes);
    __shared__ int cnt_s[2][64];
    const int grp = threadIdx.x >> 9, gt = threadIdx.x & 511;  // tile group, thread in group
    unsigned short* rows = reinterpret_cast<unsigned short*>(lds_raw + grp * kVerletRowsBytes);
    for (int u = blockIdx.x; u < nunits; u += gridDim.x) {
        const int2 ud = units[u];
        __syncthreads();  // the previous unit's reads are done
        for (int q = 0; q < ud.y; ++q) {
            const int4 sg = segs[ud.x + q];
            const DevJob& J = jobs[sg.x];
            const long long s = st[sg.x].step;
            if (!force && !due(J, s, J.pairs_freq)) continue;
            const float4* __restrict__ g = J.coord[s & 1];
            for (int k = threadIdx.x; k < J.n; k += blockDim.x) coords[sg.w + k] = g[k];
        }
        __syncthreads();
        for (int q = 0; q < ud.y; ++q) {
            const int4 sg = segs[ud.x + q];
            const DevJob& J = jobs[sg.x];
            DevJobState& S = st[sg.x];
            if (!force && !due(J, S.step, J.pairs_freq)) continue;
            for (int t0 = 0; t0 < sg.z; t0 += 128) {
                const int i0 = sg.y + t0 + 64 * grp;
                const bool mine = t0 + 64 * grp < sg.z;
                if (mine) verlet_tile<unsigned short, 8, CH>(J, S, coords + sg.w, i0, rows, cnt_s[grp], gt >> 6);
                __syncthreads();
                if (mine) verlet_store<unsigned short, 8>(J, i0, rows, cnt_s[grp], gt);
                __syncthreads();
            }
        }
    }
}

// The Verlet build of the LDS-step jobs spread for a few small jobs (the
// step's split_rows shape): four 1024-thread workgroups per 64-row tile,
// each builds 16 rows, one wavefront per row (the same in-order ballot
// compaction as k_verlet_lds, so the same lists), from the job's
// coordinates staged in LDS.  Grid: ntiles * 4.
__global__ __launch_bounds__(1024) void k_verlet_split(const DevJob* __restrict__ jobs, DevJobState* __restrict__ st,
                                                       const int2* __restrict__ tiles, int ntiles, int force) {
    constexpr int E = VerletLds<unsigned short>::entries, RS = VerletLds<unsigned short>::stride;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    unsigned short* rows = reinterpret_cast<unsigned short*>(lds_raw);
    float4* coords = reinterpret_cast<float4*>(lds_raw + kVerletRowsBytes);
    __shared__ int cnt_s[64];
    const int tile = blockIdx.x >> 2, quarter = blockIdx.x & 3;
    if (tile >= ntiles) return;
    const int2 td = tiles[tile];
    const DevJob& J = jobs[td.x];
    if (!J.lds_step) return;  // built by k_verlet
    DevJobState& S = st[td.x];
    const long long s = S.step;
    if (!force && !due(J, s, J.pairs_freq)) return;
    const int n = J.n, i0 = td.y, nrow = min(64, n - i0);
    if (16 * quarter >= nrow) return;  // every exit above is uniform over the workgroup
    {
        const float4* __restrict__ g = J.coord[s & 1];
        for (int k = threadIdx.x; k < n; k += 1024) coords[k] = g[k];
    }
    __syncthreads();
    const int w = threadIdx.x >> 6;
    verlet_tile<unsigned short, 64, 8>(J, S, coords, i0, rows, cnt_s, 16 * quarter + w);
    __syncthreads();
    // this workgroup's 16 rows: thread (row b, entry lane kq)
    const int b = 16 * quarter + (threadIdx.x & 15), kq = threadIdx.x >> 4;
    if (b < nrow) {
        const int c = cnt_s[b], cap = J.pair_cap;
        if (kq == 0) J.pair_cnt[i0 + b] = c < cap ? c : cap;
        const auto pj = gmem(static_cast<unsigned short*>(J.pair_j));
        const int lim = min(c, min(E, cap));
        for (int k = kq; k < lim; k += 64) pj[(size_t)k * J.pair_ld + i0 + b] = rows[b * RS + k];
    }
}

// ---------------------------------------------------------------------------
// per-job updaters at stride boundaries
// ---------------------------------------------------------------------------
// One wavefront per job.  The reaction on the tip is summed in bead order,
// as the host loop of the reference sums it: the wavefront loads the
// beads' forces kTipChunk at a time (coalesced, all in flight together, and
// clears them), stages their components in LDS, and lane c < 3 adds
// component c bead by bead; the components' sums are then gathered to lane 0.
constexpr int kTipChunk = 512;
__device__ void tip_update(const DevJob& J, DevJobState& S, long long s) {
    __shared__ __align__(16) float comp[3][kTipChunk];
    const int lane = threadIdx.x & 63;
    if (s == J.retraction && lane == 0) S.V = -S.V;
    if (s % J.nav != 0) return;
    float acc = 0.0f;  // lane c < 3: component c
    for (int base = 0; base < J.n; base += kTipChunk) {
        float4 v[kTipChunk / 64];
#pragma unroll
        for (int u = 0; u < kTipChunk / 64; ++u) {
            const int i = base + 64 * u + lane;
            v[u] = i < J.n ? J.tipF[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
#pragma unroll
        for (int u = 0; u < kTipChunk / 64; ++u) {
            const int i = base + 64 * u + lane;
            if (i < J.n) J.tipF[i] = make_float4(0.0f, 0.0f, 0.0f, v[u].w);
            comp[0][64 * u + lane] = v[u].x;
            comp[1][64 * u + lane] = v[u].y;
            comp[2][64 * u + lane] = v[u].z;
        }
        __syncthreads();  // the workgroup is this one wavefront
        const int m = min(kTipChunk, J.n - base);
        if (lane < 3) {
            const float* __restrict__ c = comp[lane];
            int b = 0;
            for (; b + 4 <= m; b += 4) {
                const float4 q = *reinterpret_cast<const float4*>(c + b);
                acc += q.x;
                acc += q.y;
                acc += q.z;
                acc += q.w;
            }
            for (; b < m; ++b) acc += c[b];
        }
        __syncthreads();  // the sums' reads are done before the next chunk's writes
    }
    float f0 = __shfl(acc, 0), f1 = __shfl(acc, 1), f2 = __shfl(acc, 2);
    if (lane != 0) return;
    const float fn = (float)J.nav;
    f0 /= fn;
    f1 /= fn;
    f2 /= fn;
    S.tipFav[0] = f0;
    S.tipFav[1] = f1;
    S.tipFav[2] = f2;
    S.tipFav[3] = sqrtf(f0 * f0 + f1 * f1 + f2 * f2);
    S.dx = (float)(s / J.nav) * S.V;
    if (J.moveSurface) {
        for (int d = 0; d < 3; ++d) S.micaR[d] = J.micaR0[d] + J.dir[d] * S.dx;
    } else {
        for (int d = 0; d < 3; ++d) S.chip[d] = J.chip0[d] + J.dir[d] * S.dx;
    }
    const float dr0 = S.chip[0] - S.tip[0], dr1 = S.chip[1] - S.tip[1], dr2 = S.chip[2] - S.tip[2];
    S.tipDr = sqrtf(dr0 * dr0 + dr1 * dr1 + dr2 * dr2);
    const float df0 = -f0 + dr0 * J.indKs, df1 = -f1 + dr1 * J.indKs, df2 = -f2 + dr2 * J.indKs;
    const float mult = ((J.h * ((float)J.nav)) / (J.tipZeta));
    if (J.fixTrans) {
        const float ct = mult * df0 * J.dir[0] + mult * df1 * J.dir[1] + mult * df2 * J.dir[2];
        for (int d = 0; d < 3; ++d) S.tip[d] += ct * J.dir[d];
    } else {
        S.tip[0] += mult * df0;
        S.tip[1] += mult * df1;
        S.tip[2] += mult * df2;
    }
}

__device__ void pull_update(const DevJob& J, DevJobState& S, long long s) {
    const float xt = J.deltax * (float)(s / J.pullFreq);
    const float4 cn = J.coord[s & 1][J.pulledEnd];
    S.extF[0] = J.k_trans * (S.cant[0] - cn.x);
    S.extF[1] = J.k_trans * (S.cant[1] - cn.y);
    S.extF[2] = J.k_trans * (S.cant[2] - cn.z);
    for (int d = 0; d < 3; ++d) S.cant[d] = J.cant0[d] + xt * J.pullVec[d];
    for (int k = 0; k < J.npulled; ++k) {
        J.ext[J.pulled[k]] = make_float4(S.extF[0], S.extF[1], S.extF[2], 2.0f);
        J.bflag[J.pulled[k]] = 2;
    }
}

// The updaters of one thread's work at step s (mask as k_job_update's).
__device__ void job_update_scalar(const DevJob& J, DevJobState& S, long long s, int mask) {
    if (s >= J.end_step || s % J.stride != 0) return;
    if ((mask & 2) && (J.flags & JF_PULL_UPDATER)) pull_update(J, S, s);
    if ((mask & 4) && (J.flags & JF_HEATING) && s % J.tempFreq == 0) {
        const float temp = J.initialT + (float)(s / J.tempFreq) * J.deltaT;
        S.var = sqrtf(2.0f * temp * J.zeta / J.h);
    }
}

// mask: 1 indentation tip, 2 pulling cantilever, 4 heating schedule.
// One 64-thread workgroup per job; lane 0 does the scalar work.
__global__ __launch_bounds__(64) void k_job_update(const DevJob* __restrict__ jobs, DevJobState* __restrict__ st,
                                                   int njobs, int mask) {
    const int jb = blockIdx.x;
    if (jb >= njobs) return;
    const DevJob& J = jobs[jb];
    DevJobState& S = st[jb];
    const long long s = S.step;
    if (s >= J.end_step || s % J.stride != 0) return;
    if ((mask & 1) && (J.flags & JF_INDENTATION)) tip_update(J, S, s);
    if (threadIdx.x == 0) job_update_scalar(J, S, s, mask);
}

// Verlet lists of the R rows from row0 by one wavefront (k_verlet's filter, in
// the same order), the job's coordinates in LDS: the rows' chunks of 64 possible
// partners are loaded together, and the accepted ones, few, go to their slots
// directly.
template <int R>
__device__ __forceinline__ void verlet_few(const DevJob& J, DevJobState& S, const float4* cur, int row0) {
    const int lane = threadIdx.x & 63, nr = min(R, J.n - row0);
    const int cap = J.pair_cap, ppcap = J.pp_cap, idx16 = J.idx16;
    const float d2max = J.pl_d2;
    const int bl = gmem(J.perm)[row0 + min(lane, nr - 1)];
    const int cl = lane < nr ? gmem(J.pp_cnt)[bl] : 0;
    int most = cl;
#pragma unroll
    for (int o = R / 2; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o));
    most = __builtin_amdgcn_readfirstlane(most);
    int cnt[R];
#pragma unroll
    for (int q = 0; q < R; ++q) cnt[q] = 0;
    for (int base = 0; base < most; base += 64) {
        int j[R];
#pragma unroll
        for (int q = 0; q < R; ++q)
            j[q] = list_at(J.pp_j, idx16,
                           (size_t)__builtin_amdgcn_readlane(bl, q) * J.pp_ld + min(base + lane, ppcap - 1));
#pragma unroll
        for (int q = 0; q < R; ++q) {
            const bool in = base + lane < __builtin_amdgcn_readlane(cl, q);
            const float4 o = cur[in ? j[q] : 0], c = cur[__builtin_amdgcn_readlane(bl, q)];
            const float x = o.x - c.x, y = o.y - c.y, z = o.z - c.z;
            const bool ok = in & (x * x + y * y + z * z <= d2max);
            const unsigned long long m = __builtin_amdgcn_ballot_w64(ok);
            const int pos = (int)__builtin_amdgcn_mbcnt_hi(
                (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, (unsigned)cnt[q]));
            if (ok && pos < cap) list_put(J.pair_j, idx16, (size_t)pos * J.pair_ld + row0 + q, j[q]);
            cnt[q] += __popcll(m);
        }
    }
    int total = cnt[0];
#pragma unroll
    for (int q = 1; q < R; ++q) total = lane == q ? cnt[q] : total;
    if (lane < nr) {
        J.pair_cnt[row0 + lane] = min(total, cap);
        if (total > cap) atomicOr(&S.overflow, 2);
    }
}

// The steps of a block in one launch, for launches of small jobs: one workgroup
// per job, a wavefront per R of its rows (blockDim.x / 64 >= ceil(n / R)), the
// coordinates in LDS and a barrier between steps in the place of a launch.  Of
// k_step_rows' chain only the sums are left: lists and generators stay in
// registers, partners come from LDS.  Bound by the latency of its dependent
// operations: 560 vector instructions a step and wavefront in ~9,000 cycles, at
// one or two wavefronts a SIMD.  ldc: beads of the launch's largest job;
// advance: what the block's last launch adds to the step counters (in the place
// of k_job_advance), 0 for none.  350 peptides of 22 beads, a block of ten
// steps: 37 us, 75 as ten launches of k_step_rows and the gaps between them.
// begin (BLOCK_*): what the block begins with here, in the place of k_job_update
// (but for the tip) and k_verlet_split: 3 us more, for the 12 of the two
// launches.
template <int R>
__global__ __launch_bounds__(1024) void k_block_rows(const DevJob* __restrict__ jobs,
                                                     const StepDesc* __restrict__ descs,
                                                     DevJobState* __restrict__ st, int ldc, int kstep, int nsteps,
                                                     int advance, int begin) {
    using Rows = float[3][R][RowsShape<R, true>::KP];
    extern __shared__ float4 lds_coord[];
    __shared__ float var_s;
    Rows* const terms = reinterpret_cast<Rows*>(lds_coord + 2 * ldc);
    const StepDesc D = descs[blockIdx.x];
    const long long s = st[blockIdx.x].step + kstep;
    float var = st[blockIdx.x].var;
    asm volatile("" ::"s"(D.coord[0]), "s"(D.coord[1]), "s"(D.perm), "s"(D.pair_cnt), "s"(D.pair_j), "s"(D.b_cnt),
                 "s"(D.cov_j), "s"(D.cov_r0), "s"(D.nat_j), "s"(D.nat_par), "s"(D.rng), "s"(D.T), "s"(D.bflag));
    const int steps = (int)min((long long)nsteps, D.end_step - s);
    if (steps <= 0) return;
    const float4* const cin = (s & 1) ? D.coord[1] : D.coord[0];
    for (int i = threadIdx.x; i < D.n; i += blockDim.x) lds_coord[i] = ldg_coord(cin, i);
    const int w = wave_id(), row0 = R * w;
    if (begin & BLOCK_UPDATE) {
        if (threadIdx.x == 0) {
            job_update_scalar(jobs[blockIdx.x], st[blockIdx.x], s, 6);
            var_s = st[blockIdx.x].var;
        }
        __syncthreads();
        var = var_s;
    }
    __syncthreads();
    if ((begin & BLOCK_VERLET) && due(jobs[blockIdx.x], s, jobs[blockIdx.x].pairs_freq)) {
        if (row0 < D.n) verlet_few<R>(jobs[blockIdx.x], st[blockIdx.x], lds_coord, row0);
        __syncthreads();
    }
    if (row0 >= D.n) {  // no rows: the barriers of the others' steps
        for (int k = 0; k < steps; ++k) __syncthreads();
    } else if (D.idx16) {
        step_rows<false, R, unsigned short, true>(D, st[blockIdx.x], var, s, row0, terms[w], nullptr, lds_coord, ldc,
                                                  steps);
    } else {
        step_rows<false, R, int, true>(D, st[blockIdx.x], var, s, row0, terms[w], nullptr, lds_coord, ldc, steps);
    }
    // every wavefront took the step before its first barrier
    if (advance && threadIdx.x == 0) st[blockIdx.x].step = min(s - kstep + advance, D.end_step);
}

__global__ void k_job_advance(const DevJob* __restrict__ jobs, DevJobState* __restrict__ st, int njobs, int nsteps) {
    const int jb = blockIdx.x * blockDim.x + threadIdx.x;
    if (jb >= njobs) return;
    const long long s = st[jb].step + nsteps;
    st[jb].step = s < jobs[jb].end_step ? s : jobs[jb].end_step;
}

// One workgroup; `done` gets `ticket` once every coordinate is in host memory.
__global__ __launch_bounds__(1024) void k_read_coords(const DevJob* __restrict__ job,
                                                      const DevJobState* __restrict__ st, int n,
                                                      float4* __restrict__ host, unsigned* done, unsigned ticket) {
    const float4* const cur = job->coord[st->step & 1];
    for (int i = threadIdx.x; i < n; i += 1024) host[i] = cur[i];
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(done, ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---------------------------------------------------------------------------
// energies (output cadence only)
// ---------------------------------------------------------------------------
// A wavefront takes kEnergyRows Verlet rows, lane q + R p the terms p, p + P,
// ... (P = 64 / R) of row q: four in flight, into LDS, where the row's first
// lane adds them in list order (positions without a term hold -0.0, which
// changes no sum).  FENE terms, few and subtracted in FP64, go round by lane
// reads.  Bound by the gathers' latency where one lane per row walked the
// ~1,000 entries one after another: 134 us for 18,000 beads, 21 here.
constexpr int kEnergyRows = 4;
__global__ __launch_bounds__(256) void k_energies(const DevJob* __restrict__ jobs, const DevJobState* __restrict__ st,
                                                  int job) {
    constexpr int R = kEnergyRows, P = 64 / R, U = 4, K = P * U;
    __shared__ __align__(16) float terms[4][R][K + 4];
    const DevJob& J = jobs[job];
    const int n = J.n, w = wave_id(), row0 = R * (4 * (int)blockIdx.x + w);
    if (row0 >= n) return;
    const int lane = threadIdx.x & 63, q = lane % R, p = lane / R;
    const int r = row0 + q, rc = min(r, n - 1);
    const CoordGlobal cur{J.coord[st[job].step & 1]};
    const int i = gmem(J.perm)[rc];
    const float4 c = cur[i];
    const bool own = r < n;
    const int nc = own ? gmem(J.cov_cnt)[i] : 0, nn = own ? gmem(J.nat_cnt)[i] : 0, np = own ? gmem(J.pair_cnt)[rc] : 0;
    int ncm = nc, nnm = nn, npm = np;  // the longest rows (every set of R lanes holds all rows)
#pragma unroll
    for (int o = R / 2; o > 0; o >>= 1) {
        ncm = max(ncm, __shfl_xor(ncm, o));
        nnm = max(nnm, __shfl_xor(nnm, o));
        npm = max(npm, __shfl_xor(npm, o));
    }
    ncm = __builtin_amdgcn_readfirstlane(ncm);
    nnm = __builtin_amdgcn_readfirstlane(nnm);
    npm = __builtin_amdgcn_readfirstlane(npm);
    float pot = 0.0f;
    for (int b = 0; b < ncm; b += P) {
        double t = 0.0;
        if (b + p < nc) {
            const size_t e = (size_t)(b + p) * n + i;
            const float4 o = cur[gmem(J.cov_j)[e]];
            const float x = o.x - c.x, y = o.y - c.y, z = o.z - c.z;
            float d = sqrtf(x * x + y * y + z * z);
            d = d - gmem(J.cov_r0)[e];
            t = ((double)J.ks / 2.0) * (double)J.R2 * (double)logf_series(1.0f - d * d / (J.R2));
        }
        for (int u = 0; u < min(P, ncm - b); ++u) {
            const double v = __shfl(t, q + R * u);
            if (b + u < nc) pot = (float)((double)pot - v);
        }
    }
    if (own && p == 0) J.energies[i] = pot;
    pot = 0.0f;
    for (int b = 0; b < nnm; b += K) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = b + u * P + p;
            float t = -0.0f;
            if (k < nn) {
                const size_t e = (size_t)k * n + i;
                const float4 o = cur[gmem(J.nat_j)[e]];
                const float2 par = ldg2(J.nat_par, e);
                const float x = o.x - c.x, y = o.y - c.y, z = o.z - c.z;
                const float f = par.x / (x * x + y * y + z * z);
                float p6 = f * f * f;
                const float p12 = p6 * p6;
                p6 = -2.0f * p6;
                const float eh = (float)((double)(-par.y * par.x) / 12.0);
                t = eh * (p6 + p12);
            }
            terms[w][q][u * P + p] = t;
        }
        wave_lds_order();
        if (p == 0) rows_add(terms[w][q], min(K, nnm - b), pot);
        wave_lds_order();
    }
    if (own && p == 0) J.energies[n + i] = pot;
    pot = 0.0f;
    for (int b = 0; b < npm; b += K) {
        float4 o[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // positions past the row's entries gather its own bead
            const int k = b + u * P + p;
            const int j = list_at(J.pair_j, J.idx16, (size_t)min(k, max(np - 1, 0)) * J.pair_ld + rc);
            o[u] = cur[k < np ? j : i];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const float x = o[u].x - c.x, y = o[u].y - c.y, z = o[u].z - c.z;
            const float d2 = x * x + y * y + z * z;
            const float f = J.a2 / d2;
            terms[w][q][u * P + p] = (b + u * P + p < np && d2 < J.rc2) ? J.el * f * f * f : -0.0f;
        }
        wave_lds_order();
        if (p == 0) rows_add(terms[w][q], min(K, npm - b), pot);
        wave_lds_order();
    }
    if (own && p == 0) J.energies[2 * n + i] = pot;
}

// Self-check of div_rn_fast against the IEEE division: every float bit
// pattern b in [lo, hi) (inside the fast range) with each numerator a[k];
// counts the results that differ, and the b whose sqrt_rn_fast or
// recip_rn_fast is not the IEEE square root or reciprocal.
__global__ void k_division_check(unsigned lo, unsigned hi, const float* __restrict__ a, int na,
                                 unsigned long long* __restrict__ bad) {
    unsigned long long mine = 0;
    for (unsigned u = lo + blockIdx.x * blockDim.x + threadIdx.x; u < hi; u += gridDim.x * blockDim.x) {
        const float b = __uint_as_float(u);
        mine += __float_as_uint(sqrt_rn_fast(b)) != __float_as_uint(sqrtf(b)) ? 1ull : 0ull;
        mine += __float_as_uint(recip_rn_fast(b)) != __float_as_uint(1.0f / b) ? 1ull : 0ull;
        for (int k = 0; k < na; ++k)
            mine += __float_as_uint(div_rn_fast(a[k], b)) != __float_as_uint(a[k] / b) ? 1ull : 0ull;
    }
    if (mine) atomicAdd(bad, mine);
}

hipError_t launch_division_check(unsigned lo, unsigned hi, const float* a, int na, unsigned long long* bad,
                                 hipStream_t stream) {
    hipLaunchKernelGGL(k_division_check, dim3(8192), dim3(256), 0, stream, lo, hi, a, na, bad);
    return hipGetLastError();
}

// Advances `count` draws of the Hybrid Taus state of beads [0, n) and
// writes either the raw uint32 outputs or the Gaussian triples.
__global__ void k_rng_probe(uint4* __restrict__ state, int n, int count, int gaussian, float* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint4 s = state[i];
    for (int k = 0; k < count; ++k) {
        if (gaussian) {
            const float3 g = gauss3(s);
            out[((size_t)i * count + k) * 3 + 0] = g.x;
            out[((size_t)i * count + k) * 3 + 1] = g.y;
            out[((size_t)i * count + k) * 3 + 2] = g.z;
        } else {
            const uint32_t u = hybrid_taus(s);
            reinterpret_cast<uint32_t*>(out)[(size_t)i * count + k] = u;
        }
    }
    state[i] = s;
}

// Plain streaming copy (16 B per lane per iteration): the reference point
// for HBM bandwidth and for scaling memory counters.
__global__ __launch_bounds__(256) void k_copy(const float4* __restrict__ src, float4* __restrict__ dst, size_t n) {
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) dst[i] = src[i];
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
hipError_t launch_copy(const float4* src, float4* dst, size_t n, hipStream_t stream) {
    hipLaunchKernelGGL(k_copy, dim3(8192), dim3(256), 0, stream, src, dst, n);
    return hipGetLastError();
}

static int grid_for(int ntiles, int max_blocks) {
    int b = (ntiles + kTilesPerBlock - 1) / kTilesPerBlock;
    if (max_blocks > 0 && b > max_blocks) b = max_blocks;
    if (b >= 8) b = (b + 7) / 8 * 8;  // whole XCD groups
    return b < 1 ? 1 : b;
}

// k_step_rows over every tile for the job classes given (1 LDS-step jobs, 2
// the others), R rows per wavefront.
template <bool FO, int R>
static void launch_rows_of(const StepDesc* one, int classes, const StepDesc* descs, const DevJobState* st,
                           const int2* tiles, int ntiles, int kstep, float4* out, hipStream_t stream) {
    int blocks = (ntiles * (64 / R) + 3) / 4;
    if (blocks >= 8) blocks = (blocks + 7) / 8 * 8;
    if (one)
        hipLaunchKernelGGL((k_step_rows_one<FO, R>), dim3(blocks), dim3(256), 0, stream, *one, st, kstep, out);
    else
        hipLaunchKernelGGL((k_step_rows<FO, R>), dim3(blocks), dim3(256), 0, stream, descs, st, tiles, ntiles, kstep,
                           classes, out);
}
template <bool FO>
static void launch_rows(int R, const StepDesc* one, int classes, const StepDesc* descs, const DevJobState* st,
                        const int2* tiles, int ntiles, int kstep, float4* out, hipStream_t stream) {
    auto* const launch = R == 2   ? launch_rows_of<FO, 2>
                         : R == 4 ? launch_rows_of<FO, 4>
                         : R == 8 ? launch_rows_of<FO, 8>
                                  : launch_rows_of<FO, 16>;
    launch(one, classes, descs, st, tiles, ntiles, kstep, out, stream);
}

hipError_t launch_step(const DevJob* jobs, const StepDesc* descs, const StepDesc* one, const DevJobState* st,
                       const int2* tiles, int ntiles, int any_global,
                       const int2* units, const int4* segs, int nunits, int lds_beads, int kstep, int max_blocks,
                       hipStream_t stream, const StepShape& shape) {
    if (ntiles <= 0) return hipSuccess;
    const int rl = nunits > 0 ? shape.split_rows : 0, rg = any_global ? shape.split_global : 0;
    if (rg)  // with the LDS-step jobs where both classes take the same shape
        launch_rows<false>(rg, one, rl == rg ? 3 : 2, descs, st, tiles, ntiles, kstep, nullptr, stream);
    else if (any_global)
        hipLaunchKernelGGL(k_step<false>, dim3(grid_for(ntiles, max_blocks)), dim3(256), 0, stream, jobs, st, tiles,
                           ntiles, kstep, nullptr);
    if (rl) {
        if (rl != rg) launch_rows<false>(rl, one, 1, descs, st, tiles, ntiles, kstep, nullptr, stream);
    } else if (nunits > 0) {
        const dim3 g(nunits), b(shape.unit_rows);
        const size_t lds = (size_t)lds_beads * sizeof(float4);
        if (shape.pair_batch == 4)
            hipLaunchKernelGGL((k_step_lds<false, 4>), g, b, lds, stream, jobs, st, units, segs, nunits, kstep, nullptr);
        else if (shape.pair_batch == 8)
            hipLaunchKernelGGL((k_step_lds<false, 8>), g, b, lds, stream, jobs, st, units, segs, nunits, kstep, nullptr);
        else
            hipLaunchKernelGGL((k_step_lds<false, 6>), g, b, lds, stream, jobs, st, units, segs, nunits, kstep, nullptr);
    }
    return hipGetLastError();
}

hipError_t launch_block_rows(const DevJob* jobs, const StepDesc* descs, DevJobState* st, int njobs, int beads, int R,
                             int kstep, int nsteps, int advance, int begin, hipStream_t stream) {
    const int waves = (beads + R - 1) / R;
    if (waves > 16 || (R != 8 && R != 16)) return hipErrorInvalidValue;
    const dim3 g(njobs), b(64 * waves);
    auto lds = [&](int kp) { return (size_t)2 * beads * 16 + (size_t)waves * 3 * R * kp * 4; };
    if (R == 8)
        hipLaunchKernelGGL(k_block_rows<8>, g, b, lds(RowsShape<8, true>::KP), stream, jobs, descs, st, beads, kstep,
                           nsteps, advance, begin);
    else
        hipLaunchKernelGGL(k_block_rows<16>, g, b, lds(RowsShape<16, true>::KP), stream, jobs, descs, st, beads, kstep,
                           nsteps, advance, begin);
    return hipGetLastError();
}

hipError_t launch_forces(const DevJob* jobs, const StepDesc* descs, const StepDesc* one, const DevJobState* st,
                         const int2* tiles, int ntiles, int any_global,
                         const int2* units, const int4* segs, int nunits, int lds_beads, float4* out,
                         hipStream_t stream, const StepShape& shape) {
    if (ntiles <= 0) return hipSuccess;
    if (any_global && shape.split_global)
        launch_rows<true>(shape.split_global, one, 2, descs, st, tiles, ntiles, 0, out, stream);
    else if (any_global)
        hipLaunchKernelGGL(k_step<true>, dim3(grid_for(ntiles, 0)), dim3(256), 0, stream, jobs, st, tiles, ntiles, 0,
                           out);
    if (nunits > 0 && shape.split_rows)
        launch_rows<true>(shape.split_rows, one, 1, descs, st, tiles, ntiles, 0, out, stream);
    else if (nunits > 0)
        hipLaunchKernelGGL((k_step_lds<true, 6>), dim3(nunits), dim3(kLdsUnit), (size_t)lds_beads * sizeof(float4),
                           stream, jobs, st, units, segs, nunits, 0, out);
    return hipGetLastError();
}

hipError_t launch_possible(const DevJob* jobs, DevJobState* st, const int2* tiles, int ntiles, int njobs, int boxes,
                           int cell_words, int any_global, const int2* sunits, const int4* segs, int nsunits,
                           int lds_beads, int force, hipStream_t stream, const StepShape& shape) {
    if (ntiles <= 0) return hipSuccess;
    const int use_boxes = boxes != 0;
    if (any_global || nsunits <= 0)
        hipLaunchKernelGGL(k_possible, dim3(grid_for(ntiles, 0)), dim3(256), 0, stream, jobs, st, tiles, ntiles,
                           force, use_boxes, nsunits > 0);
    if (nsunits > 0 && shape.split_rows)
        hipLaunchKernelGGL(k_possible_split, dim3(ntiles * 4), dim3(1024), (size_t)lds_beads * sizeof(float4), stream,
                           jobs, st, tiles, ntiles, force, use_boxes);
    else if (nsunits > 0)
        hipLaunchKernelGGL(k_possible_lds, dim3(nsunits), dim3(kLdsUnit), (size_t)lds_beads * sizeof(float4), stream,
                           jobs, st, sunits, segs, nsunits, force, use_boxes);
    auto of_xcds = [](int blocks) { return blocks >= 8 ? (blocks + 7) / 8 * 8 : blocks; };
    if (boxes & BOXES_NEAR) {
        hipLaunchKernelGGL(k_tile_boxes, dim3(grid_for(ntiles, 0)), dim3(256), 0, stream, jobs, st, tiles, ntiles, force);
        hipLaunchKernelGGL(k_possible_boxes, dim3(of_xcds(64 / kBoxBeads / 4 * ntiles)), dim3(256), 0, stream, jobs, st,
                           tiles, ntiles, force);
    }
    if (boxes & BOXES_WIDE) {
        const dim3 g(grid_for(ntiles, 0)), b(256);
        hipLaunchKernelGGL(k_cells_setup, dim3(njobs), dim3(1024), 0, stream, jobs, st, njobs, force);
        hipLaunchKernelGGL(k_cells_count, g, b, 0, stream, jobs, st, tiles, ntiles, force);
        hipLaunchKernelGGL(k_cells_scan, dim3(njobs), dim3(1024), 0, stream, jobs, st, njobs, force);
        hipLaunchKernelGGL(k_cells_fill, g, b, 0, stream, jobs, st, tiles, ntiles, force);
        // one wavefront per half tile
        hipLaunchKernelGGL(k_possible_cells, dim3(of_xcds(2 * ntiles)), dim3(64),
                           (size_t)(cell_words + (cell_words + 63) / 64) * 8, stream, jobs, st, tiles, ntiles, force,
                           cell_words);
    }
    return hipGetLastError();
}

hipError_t launch_sort_rows(const DevJob* jobs, DevJobState* st, const int2* units, int nunits, int force,
                            hipStream_t stream, const StepShape& shape) {
    if (nunits > 0)
        hipLaunchKernelGGL(k_sort_rows, dim3(nunits), dim3(kLdsUnit), 0, stream, jobs, st, units, nunits,
                           shape.sort_every, force);
    return hipGetLastError();
}

hipError_t launch_verlet(const DevJob* jobs, DevJobState* st, const int2* tiles, int ntiles, int any_idx32,
                         int any_global, const int2* units, int nunits, const int2* sunits, const int4* segs,
                         int nsunits, int lds_beads, int force, hipStream_t stream, const StepShape& shape) {
    if (ntiles <= 0) return hipSuccess;
    if (const hipError_t e = launch_sort_rows(jobs, st, units, nunits, force, stream, shape)) return e;
    int blocks = ntiles;
    if (blocks >= 8) blocks = (blocks + 7) / 8 * 8;
    const size_t lds = any_idx32 ? 64 * VerletLds<int>::stride * sizeof(int)
                                 : 64 * VerletLds<unsigned short>::stride * sizeof(unsigned short);
    if (any_global || nsunits <= 0)
        hipLaunchKernelGGL(k_verlet, dim3(blocks), dim3(64 * kVerletWaves), lds, stream, jobs, st, tiles, ntiles,
                           force, nsunits > 0);
    if (nsunits > 0 && shape.split_rows) {
        const size_t lds = (size_t)kVerletRowsBytes + (size_t)lds_beads * 16;
        hipLaunchKernelGGL(k_verlet_split, dim3(ntiles * 4), dim3(1024), lds, stream, jobs, st, tiles, ntiles, force);
    } else if (nsunits > 0) {
        const size_t lds = 2 * (size_t)kVerletRowsBytes + (size_t)lds_beads * 16;
        if (shape.verlet_chunk == 4)
            hipLaunchKernelGGL(k_verlet_lds<4>, dim3(nsunits), dim3(1024), lds, stream, jobs, st, sunits, segs, nsunits,
                               force);
        else
            hipLaunchKernelGGL(k_verlet_lds<8>, dim3(nsunits), dim3(1024), lds, stream, jobs, st, sunits, segs, nsunits,
                               force);
    }
    return hipGetLastError();
}

hipError_t launch_job_update(const DevJob* jobs, DevJobState* st, int njobs, hipStream_t stream, int mask) {
    if (njobs <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_job_update, dim3(njobs), dim3(64), 0, stream, jobs, st, njobs, mask);
    return hipGetLastError();
}

hipError_t launch_job_advance(const DevJob* jobs, DevJobState* st, int njobs, int nsteps, hipStream_t stream) {
    if (njobs <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_job_advance, dim3((njobs + 63) / 64), dim3(64), 0, stream, jobs, st, njobs, nsteps);
    return hipGetLastError();
}

hipError_t launch_read_coords(const DevJob* job, const DevJobState* st, int n, float4* host, unsigned* done,
                              unsigned ticket, hipStream_t stream) {
    hipLaunchKernelGGL(k_read_coords, dim3(1), dim3(1024), 0, stream, job, st, n, host, done, ticket);
    return hipGetLastError();
}

hipError_t launch_energies(const DevJob* jobs, const DevJobState* st, int job, int n, hipStream_t stream) {
    hipLaunchKernelGGL(k_energies, dim3((n + 4 * kEnergyRows - 1) / (4 * kEnergyRows)), dim3(256), 0, stream, jobs, st, job);
    return hipGetLastError();
}

hipError_t launch_rng_probe(uint4* state, int n, int count, int gaussian, float* out, hipStream_t stream) {
    hipLaunchKernelGGL(k_rng_probe, dim3((n + 255) / 256), dim3(256), 0, stream, state, n, count, gaussian, out);
    return hipGetLastError();
}

const void* step_kernel_symbol() { return reinterpret_cast<const void*>(&k_step<false>); }

}  // namespace sop
