// pth_kernels.hip -- gfx950 kernels of the soft-force path.
//
// Pipeline for one batch of walks (i-groups with their interaction lists):
//   k_spj_table   per superparticle, once per send: {m, q'xx q'yy q'zz q'xy
//                 q'yz q'zx, -eps^2 tr}, q' = 3Q - tr I
//   k_stage_walk  one workgroup per walk: FP64 bounding box of the walk's i
//                 (centre c, half extents, largest r_search), every i as FP32
//                 (x-c, y-c, z-c, rs^2), and the walk's EPJ list gathered
//                 into FP32 records relative to c, split stably into a "near"
//                 region (entries that may lie within max(rs_i, rs_j, r_out)
//                 of some i of the walk) at the front and a "far" region at
//                 the back; records are SoA blocks of 8 {x[8] y[8] z[8] m[8]
//                 rs2[8]}, gaps padded with far massless entries; beside it,
//                 one or more workgroups per walk gather the walk's SPJ list
//                 into 4-float records {x-c y-c z-c table index}
//   k_force       one wave per work item (walk, tile of 64/128/256 i with
//                 1/2/4 i per lane, j-range), one launch per i-per-lane
//                 class: j records are read through the constant address
//                 space (uniform addresses, scalar loads into SGPRs) and used
//                 as SGPR operands by every i of the lane (the VC variant
//                 copies them into VGPRs first; on gfx950 that copy issues at
//                 single rate and costs more than it saves).  Far EPJ blocks
//                 skip the neighbour count and the cutoff (both are known to
//                 be no-ops there).  FP32 pair arithmetic, FP32 partial sums
//                 per chunk, FP64 running sums.
//   k_reduce      fixed-order FP64 sum of the partial results of split walks
//   k_force_plain the plain per-walk form (first kernel of this build): one
//                 workgroup per walk, 64-i tiles, SGPR operands, whole list
//
// Pair formulas (the physics of src/force_gpu_cuda.cu:50-77 and 276-323):
//   EPJ  dx = xj - xi, r2 = |dx|^2 + eps^2, nnb += r2 < max(rs_i,rs_j)^2,
//        rinv = rsqrt(max(r2, r_out^2)), acc += m rinv^3 dx, pot -= m rinv
//   SPJ  dx = xi - xs, r2 = |dx|^2 + eps^2, traceless form
//        rqr = dx.q'.dx - eps^2 tr, meff = m + rqr/(2 r^4),
//        meff3 = (m + 5 rqr/(2 r^4))/r^3,
//        acc += q'.dx/r^5 - meff3 dx, pot -= meff/r
//   (the same quadrupole expansion as the raw-moment form of the CUDA
//   kernel, rearranged as in src/phantomquad_for_p3t_x86.hpp:144-163)
// G multiplies the FP64 sums once at the end.
#include <hip/hip_runtime.h>

#include <climits>
#include <mutex>
#include <type_traits>
#include <unordered_map>

#include "pth_device.h"

namespace pth {

typedef const __attribute__((address_space(4))) float *cfp;
typedef const __attribute__((address_space(4))) int *cip;

__device__ __forceinline__ cfp as_const(const float *p) { return (cfp)(p); }
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// With VC, copies a wave-uniform (SGPR) value into a VGPR, so that the
// arithmetic that uses it has VGPR operands only; otherwise the SGPR value
// is used as an operand directly.
template <bool VC> __device__ __forceinline__ float jv(float s)
{
    if (!VC) return s;
    float v;
    asm("v_mov_b32 %0, %1" : "=v"(v) : "s"(s));
    return v;
}
__device__ __forceinline__ float vcopy(float s) { return jv<true>(s); }

// ---------------------------------------------------------------------------
// staging

__device__ __forceinline__ void put_epj(float *se, long long slot, float x, float y, float z, float m,
                                        float r2)
{
    float *blk = se + (slot >> 3) * 40;
    const int l = (int)(slot & 7);
    blk[l] = x;
    blk[8 + l] = y;
    blk[16 + l] = z;
    blk[24 + l] = m;
    blk[32 + l] = r2;
}

// Staged SPJ record {x-c, y-c, z-c, index of the superparticle's SpjTab
// entry}: only the position depends on the walk.
__device__ __forceinline__ void put_spj(float4 *o, double x, double y, double z, const double (&c)[3], int id)
{
    *o = make_float4((float)(x - c[0]), (float)(y - c[1]), (float)(z - c[2]), __int_as_float(id));
}

// The SPJ table: m, q' = 3Q - tr I (the traceless rearrangement of
// src/phantomquad_for_p3t_x86.hpp:144-163) and -eps^2 tr, from the FP32
// moments in FP64 and rounded once.
__global__ __launch_bounds__(256) void k_spj_table(const SpjDev *__restrict__ spj, long long n, double eps2,
                                                   SpjTab *__restrict__ tab)
{
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const SpjDev p = spj[i];
    const double qxx = p.qxx, qyy = p.qyy, qzz = p.qzz;
    const double tr = qxx + qyy + qzz;
    SpjTab t;
    t.m = p.m;
    t.qxx = (float)(3.0 * qxx - tr);
    t.qyy = (float)(3.0 * qyy - tr);
    t.qzz = (float)(3.0 * qzz - tr);
    t.qxy = (float)(3.0 * (double)p.qxy);
    t.qyz = (float)(3.0 * (double)p.qyz);
    t.qzx = (float)(3.0 * (double)p.qxz);
    t.mtr = (float)(-eps2 * tr);
    tab[i] = t;
}

// bucket of a particle id in the per-walk LDS table (PTH_CO_HASH buckets)
__device__ __forceinline__ unsigned co_hash(long long id)
{
    const unsigned long long u = (unsigned long long)id;
    return ((unsigned)(u ^ (u >> 32)) * 2654435761u) >> 21;
}

struct StageArgs {
    int walk_begin;  // block b < n_walk stages walk walk_begin + b
    // blocks n_walk + p n_walk + v (p < spj_parts) stage part p of the SPJ
    // list of walk walk_begin + v
    int n_walk, spj_parts;
    const EpiDev *epi;
    const WalkDev *walks;
    const long long *es_off, *ss_off;
    const int *id_epj, *id_spj;
    const EpjDev *epj;
    const SpjDev *spj;
    double r_out, eps2;
    double4 *centre;
    int *near_blk;
    float4 *staged_i;
    float *staged_e, *staged_s;
    // changeover mode
    const long long *epi_id;
    const EpjCoDev *epj_co;
    float4 *staged_ic;
    float4 *staged_il;
    float *staged_ec;
    int *walk_err;
    // linear-cutoff mode with double-float near pairs
    int df;
    float *staged_el;
    // monopole superparticles (centre and mass), staged as far EPJ entries
    int mono;
    const EpjDev *spj_mono;
    // persistent force launches: the segment's item counters (zeroed here,
    // before the segment's force launches), or null
    int *counters;
};

// The reduction of a wave's values by op (idempotent: min or max), in lane 63:
// the vector ALU's lane shifts (DPP) instead of 84 LDS permutes (staging of
// the 16,384-particle cluster 47 to 43 us, of 4,096 particles 21 to 17).
template <class F> __device__ __forceinline__ double wave_last(double v, F op)
{
    auto step = [&](auto ctrl, auto rows) {
        const int lo = __double2loint(v), hi = __double2hiint(v);
        v = op(v, __hiloint2double(
                      __builtin_amdgcn_update_dpp(hi, hi, decltype(ctrl)::value, decltype(rows)::value, 0xf, false),
                      __builtin_amdgcn_update_dpp(lo, lo, decltype(ctrl)::value, decltype(rows)::value, 0xf, false)));
    };
    using std::integral_constant;
    step(integral_constant<int, 0x111>(), integral_constant<int, 0xf>());  // row_shr:1
    step(integral_constant<int, 0x112>(), integral_constant<int, 0xf>());  // row_shr:2
    step(integral_constant<int, 0x114>(), integral_constant<int, 0xf>());  // row_shr:4
    step(integral_constant<int, 0x118>(), integral_constant<int, 0xf>());  // row_shr:8
    step(integral_constant<int, 0x142>(), integral_constant<int, 0xa>());  // row_bcast:15 into rows 1, 3
    step(integral_constant<int, 0x143>(), integral_constant<int, 0xc>());  // row_bcast:31 into rows 2, 3
    return v;
}

// SPJ list entries [k_begin, k_end) of walk w: positions relative to the
// centre and table indices, U per thread and pass so that U gathers are in
// flight
template <int U, int WG>
__device__ __forceinline__ void stage_spj(const StageArgs &a, int w, const WalkDev &wk, const double (&c)[3],
                                          int k_begin, int k_end)
{
    float4 *out_s = reinterpret_cast<float4 *>(a.staged_s) + a.ss_off[w];
    const int *ids = a.id_spj + wk.s_off;
    const SpjDev *__restrict__ spj = a.spj;
    const int tid = (int)threadIdx.x;
    for (int k0 = k_begin; k0 < k_end; k0 += WG * U) {
        int id[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k = k0 + WG * u + tid;
            id[u] = k < k_end ? ids[k] : -1;
        }
        double px[U], py[U], pz[U];
#pragma unroll
        for (int u = 0; u < U; u++)
            if (id[u] >= 0) {
                px[u] = spj[id[u]].x;
                py[u] = spj[id[u]].y;
                pz[u] = spj[id[u]].z;
            }
#pragma unroll
        for (int u = 0; u < U; u++)
            if (id[u] >= 0) put_spj(out_s + (k0 + WG * u + tid), px[u], py[u], pz[u], c, id[u]);
    }
}

// CO (changeover mode): every near EPJ also gets its changeover radii and the
// low-order parts of its FP32 relative coordinates staged (per block of 8:
// r_in[8], r_out[8], xlo[8], ylo[8], zlo[8]; x - c = x_hi + x_lo as a
// double-float), every i the low-order parts of its coordinates, and each i
// finds its own EPJ entry
// (same id) among the walk's near entries through an LDS hash table that
// maps the hash of an id to the i's index (the ids themselves are compared
// in place, in global memory); the i's staged slot of that entry and its radii go to
// staged_ic (the force kernel drops the self pair by slot and takes the i's
// changeover radii from there).  walk_err counts i with no such entry.
// EU: EPJ entries per thread and pass of the near/far split, all gathers in
// flight at once, of WG threads per walk.  A pass is a chain of two gathers
// and two barriers (3.5 us): 4 entries where the launch has few walks (its
// latency is exposed), 2 where it has many (fewer registers, so that staging
// waves fit beside the force kernels of other segments)
template <bool CO, int EU, int WG>
__global__ __launch_bounds__(WG) void k_stage_walk(const StageArgs a)
{
    constexpr int NW = WG / 64;
    // the SPJ blocks need only the walk's centre: they run beside the EPJ
    // split, which is sequential within a walk
    const int nw = a.n_walk;
    const bool spj_wg = (int)blockIdx.x >= nw;
    const int w = a.walk_begin + (spj_wg ? ((int)blockIdx.x - nw) % nw : (int)blockIdx.x);
    const WalkDev wk = a.walks[w];
    if (blockIdx.x == 0 && a.counters && threadIdx.x < PLAN_CLASSES * 8) a.counters[threadIdx.x] = 0;
    if (spj_wg && (a.mono || wk.n_s == 0)) return;
    const EpiDev *__restrict__ epi = a.epi;
    const EpjDev *__restrict__ epj = a.epj;
    const int *__restrict__ id_epj = a.id_epj;
    const double r_out = a.r_out;
    float4 *__restrict__ staged_i = a.staged_i;
    float *__restrict__ staged_e = a.staged_e;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    __shared__ double red[NW][7];
    __shared__ int cnt[2 * EU][NW];
    __shared__ int co_idx[CO ? PTH_CO_HASH : 1];
    __shared__ int co_self[CO ? PTH_CO_MAX_NI : 1];
    __shared__ float co_rin[CO ? PTH_CO_MAX_NI : 1], co_rout[CO ? PTH_CO_MAX_NI : 1], co_m[CO ? PTH_CO_MAX_NI : 1];
    const int n_co = (CO && !spj_wg) ? min(wk.n_i, PTH_CO_MAX_NI) : 0;
    if constexpr (CO) {
        if (!spj_wg) {
            for (int k = tid; k < PTH_CO_HASH; k += WG) co_idx[k] = -1;
            __syncthreads();
            for (int k = tid; k < n_co; k += WG) {
                const long long id = a.epi_id[wk.i_off + k];
                unsigned h = co_hash(id);
                // at most PTH_CO_MAX_NI keys in PTH_CO_HASH buckets: a free one exists
                while (atomicCAS(&co_idx[h], -1, k) != -1) h = (h + 1) & (PTH_CO_HASH - 1);
                co_self[k] = -1;
                co_rin[k] = 0.f;
                co_rout[k] = 0.f;
                co_m[k] = 0.f;
            }
            __syncthreads();
        }
    }
    // -- bounding box and largest r_search of the walk's i
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300}, rsm = 0.0;
    for (int k = tid; k < wk.n_i; k += WG) {
        const EpiDev e = epi[wk.i_off + k];
        lo[0] = fmin(lo[0], e.x); hi[0] = fmax(hi[0], e.x);
        lo[1] = fmin(lo[1], e.y); hi[1] = fmax(hi[1], e.y);
        lo[2] = fmin(lo[2], e.z); hi[2] = fmax(hi[2], e.z);
        rsm = fmax(rsm, (double)e.rs);
    }
    for (int d = 0; d < 3; d++) {
        lo[d] = wave_last(lo[d], [](double x, double y) { return fmin(x, y); });
        hi[d] = wave_last(hi[d], [](double x, double y) { return fmax(x, y); });
    }
    rsm = wave_last(rsm, [](double x, double y) { return fmax(x, y); });
    if (lane == 63) {
        for (int d = 0; d < 3; d++) { red[wave][d] = lo[d]; red[wave][3 + d] = hi[d]; }
        red[wave][6] = rsm;
    }
    __syncthreads();
    double c[3], h[3];
    for (int d = 0; d < 3; d++) {
        double l = red[0][d], u = red[0][3 + d];
        for (int v = 1; v < NW; v++) {
            l = fmin(l, red[v][d]);
            u = fmax(u, red[v][3 + d]);
        }
        c[d] = (wk.n_i > 0) ? 0.5 * (l + u) : 0.0;
        h[d] = (wk.n_i > 0) ? 0.5 * (u - l) : 0.0;
    }
    rsm = red[0][6];
    for (int v = 1; v < NW; v++) rsm = fmax(rsm, red[v][6]);
    if (spj_wg) {
        const int part = ((int)blockIdx.x - nw) / nw;
        const int k_begin = (int)((long long)wk.n_s * part / a.spj_parts);
        const int k_end = (int)((long long)wk.n_s * (part + 1) / a.spj_parts);
        // (two in changeover mode: fewer registers, so the staging of the
        // next segment fits beside the changeover force kernels, which are
        // held to 7 waves per SIMD)
        stage_spj<CO ? 2 : 4, WG>(a, w, wk, c, k_begin, k_end);
        return;
    }
    if (tid == 0) a.centre[w] = make_double4(c[0], c[1], c[2], 0.0);
    for (int k = tid; k < wk.n_i; k += WG) {
        const EpiDev e = epi[wk.i_off + k];
        const double rs = (double)e.rs;
        const double dx = e.x - c[0], dy = e.y - c[1], dz = e.z - c[2];
        const float hx = (float)dx, hy = (float)dy, hz = (float)dz;
        staged_i[wk.i_off + k] = make_float4(hx, hy, hz, (float)(rs * rs));
        if (CO || a.df)
            a.staged_il[wk.i_off + k] =
                make_float4((float)(dx - (double)hx), (float)(dy - (double)hy), (float)(dz - (double)hz), 0.f);
    }
    // -- EPJ list: stable split into near (front) and far (back, reversed);
    //    EU entries per thread and pass (entries t0 + 256 u + tid) so that EU
    //    gathers are in flight per thread between the barriers
    const long long base = a.es_off[w];
    const long long cap = a.es_off[w + 1] - base;
    const double hmax = fmax(h[0], fmax(h[1], h[2]));
    int n_near = 0, n_far = 0;
    struct Ent {
        bool valid, nearj;
        float x, y, z, m, r2, xl, yl, zl;
        int jx;
    };
    auto load = [&](int t) {
        Ent q{t < wk.n_e, false, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0};
        if (q.valid) q.jx = id_epj[(long long)wk.e_off + t];
        return q;
    };
    auto classify = [&](Ent &q) {
        if (!q.valid) return;
        const EpjDev e = epj[q.jx];
        const double dx = e.x - c[0], dy = e.y - c[1], dz = e.z - c[2];
        // near: inside the walk's box widened by max(rs_i, rs_j, r_out),
        // with a margin that covers the FP32 rounding of the pair arithmetic
        const double R = fmax(fmax(rsm, (double)e.rs), r_out);
        const double dm = fmax(fabs(dx), fmax(fabs(dy), fabs(dz)));
        const double Rm = R * 1.00001 + 1e-5 * (dm + hmax);
        q.nearj = fabs(dx) <= h[0] + Rm && fabs(dy) <= h[1] + Rm && fabs(dz) <= h[2] + Rm;
        q.x = (float)dx;
        q.y = (float)dy;
        q.z = (float)dz;
        q.xl = (float)(dx - (double)q.x);
        q.yl = (float)(dy - (double)q.y);
        q.zl = (float)(dz - (double)q.z);
        q.m = e.m;
        const double rs = (double)e.rs;
        q.r2 = (float)(rs * rs);
    };
    auto place = [&](const Ent &q, long long slot) {
        put_epj(staged_e, slot, q.x, q.y, q.z, q.m, q.r2);
        if constexpr (!CO) {
            if (a.df && q.nearj) {
                float *blk = a.staged_el + (slot >> 3) * PTH_DF_EXTRA;
                const int l = (int)(slot & 7);
                blk[l] = q.xl;
                blk[8 + l] = q.yl;
                blk[16 + l] = q.zl;
            }
        }
        if constexpr (CO) {
            if (q.nearj) {
                const EpjCoDev co = a.epj_co[q.jx];
                float *blk = a.staged_ec + (slot >> 3) * PTH_CO_EXTRA;
                const int l = (int)(slot & 7);
                blk[l] = co.rin;
                blk[8 + l] = co.rout;
                blk[16 + l] = q.xl;
                blk[24 + l] = q.yl;
                blk[32 + l] = q.zl;
                blk[40 + l] = co_pot_mass(co, q.m);
                // is this the EPJ of one of the walk's i?
                unsigned hb = co_hash(co.id);
                for (;;) {
                    const int k = co_idx[hb];
                    if (k < 0) break;
                    // (the walk's ids are compared in place, not copied to LDS)
                    if (a.epi_id[wk.i_off + k] == co.id) {
                        co_self[k] = (int)slot;
                        co_rin[k] = co.rin;
                        co_rout[k] = co.rout;
                        co_m[k] = co_self_mass(co, q.m);
                        break;
                    }
                    hb = (hb + 1) & (PTH_CO_HASH - 1);
                }
            }
        }
    };
    const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int t0 = 0; t0 < wk.n_e; t0 += WG * EU) {
        Ent q[EU];
#pragma unroll
        for (int u = 0; u < EU; u++) q[u] = load(t0 + WG * u + tid);
#pragma unroll
        for (int u = 0; u < EU; u++) classify(q[u]);
        unsigned long long bn[EU], bf[EU];
#pragma unroll
        for (int u = 0; u < EU; u++) {
            bn[u] = __ballot(q[u].valid && q[u].nearj);
            bf[u] = __ballot(q[u].valid && !q[u].nearj);
        }
        if (lane == 0) {
#pragma unroll
            for (int u = 0; u < EU; u++) {
                cnt[2 * u][wave] = __popcll(bn[u]);
                cnt[2 * u + 1][wave] = __popcll(bf[u]);
            }
        }
        __syncthreads();
        // the entries of part u (t0 + 256 u + tid) follow all of part u - 1's
#pragma unroll
        for (int u = 0; u < EU; u++) {
            int pn = 0, pf = 0, tn = 0, tf = 0;
            for (int v = 0; v < NW; v++) {
                const int cn = cnt[2 * u][v], cf = cnt[2 * u + 1][v];
                if (v < wave) {
                    pn += cn;
                    pf += cf;
                }
                tn += cn;
                tf += cf;
            }
            if (q[u].valid)
                place(q[u], q[u].nearj ? base + n_near + pn + __popcll(bn[u] & below)
                                       : base + cap - 1 - (n_far + pf + __popcll(bf[u] & below)));
            n_near += tn;
            n_far += tf;
        }
        __syncthreads();
    }
    // monopole superparticles: far entries after the EPJ list's far ones (a
    // monopole pair is a far pair: no cutoff, no neighbour count), in list
    // order from the back
    if (a.mono) {
        const int *__restrict__ mid = a.id_spj + wk.s_off;
        for (int k = tid; k < wk.n_s; k += WG) {
            const EpjDev e = a.spj_mono[mid[k]];
            put_epj(staged_e, base + cap - 1 - (n_far + k), (float)(e.x - c[0]), (float)(e.y - c[1]),
                    (float)(e.z - c[2]), e.m, 0.f);
        }
        n_far += wk.n_s;
    }
    // pad the gap between the two regions (far, massless); the padding of the
    // last near block is read by the double-float near loop: zero low parts
    for (long long s = base + n_near + tid; s < base + cap - n_far; s += WG) {
        put_epj(staged_e, s, 1e18f, 1e18f, 1e18f, 0.f, 0.f);
        if (!CO && a.df) {
            float *blk = a.staged_el + (s >> 3) * PTH_DF_EXTRA;
            const int l = (int)(s & 7);
            blk[l] = blk[8 + l] = blk[16 + l] = 0.f;
        }
    }
    if (tid == 0) a.near_blk[w] = (int)((base + ((n_near + 7) & ~7)) >> 3);
    if constexpr (CO) {
        // (the loop above ended with a barrier: co_self is complete)
        int miss = 0;
        for (int k = tid; k < wk.n_i; k += WG) {
            const bool in = k < n_co;
            const int s = in ? co_self[k] : -1;
            a.staged_ic[wk.i_off + k] =
                make_float4(__int_as_float(s), in ? co_rin[k] : 0.f, in ? co_rout[k] : 0.f, in ? co_m[k] : 0.f);
            miss |= (s < 0);
        }
        const int n_miss = __syncthreads_count(miss);
        if (tid == 0) a.walk_err[w] = n_miss;
    }
}

// ---------------------------------------------------------------------------
// force, fused form

struct Consts {
    float eps2, rout2, half, two_half;
};

// EPJ blocks [b_begin, b_end) of a walk's staged list against the lane's i.
// NEAR blocks also count neighbours and apply the cutoff; with DF (near
// blocks in linear-cutoff mode) each separation is taken from double-float
// walk-relative coordinates, (x_j - x_i) + (xlo_j - xlo_i): the FP32 high
// parts of two close particles differ exactly, so the separation keeps FP32
// relative precision however far the pair lies from the walk centre.
// end(b) is called after the sums up to block b are in A.
template <int IPL, int NNB_LE, bool NEAR, bool VC, bool DF = false, class F>
__device__ __forceinline__ void epj_blocks(F &end, cfp se, int b_begin, int b_end, const float (&xi)[IPL],
                                           const float (&yi)[IPL], const float (&zi)[IPL],
                                           const float (&rsi2)[IPL], const Consts &K, double (&A)[IPL][4],
                                           int (&nnb)[IPL], cfp sel = nullptr, const float *xil = nullptr,
                                           const float *yil = nullptr, const float *zil = nullptr)
{
    for (int b0 = b_begin; b0 < b_end; b0 += PTH_FLUSH_BLOCKS) {
        const int b1 = min(b0 + PTH_FLUSH_BLOCKS, b_end);
        float ax[IPL], ay[IPL], az[IPL], p[IPL];
        int nb[IPL];
#pragma unroll
        for (int q = 0; q < IPL; q++) { ax[q] = ay[q] = az[q] = p[q] = 0.f; nb[q] = 0; }
        for (int b = b0; b < b1; b++) {
            const cfp B = se + (size_t)b * 40;
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const float xj = jv<VC>(B[k]), yj = jv<VC>(B[8 + k]), zj = jv<VC>(B[16 + k]);
                const float mj = jv<VC>(B[24 + k]);
                float rj = 0.f;
                if (NEAR) rj = jv<VC>(B[32 + k]);
                float xjl = 0.f, yjl = 0.f, zjl = 0.f;
                if (DF) {
                    const cfp E = sel + (size_t)b * PTH_DF_EXTRA;
                    xjl = E[k];
                    yjl = E[8 + k];
                    zjl = E[16 + k];
                }
#pragma unroll
                for (int q = 0; q < IPL; q++) {
                    float dx = xj - xi[q];
                    float dy = yj - yi[q];
                    float dz = zj - zi[q];
                    if (DF) {
                        dx += xjl - xil[q];
                        dy += yjl - yil[q];
                        dz += zjl - zil[q];
                    }
                    const float r2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, __builtin_fmaf(dx, dx, K.eps2)));
                    float ri;
                    if (NEAR) {
                        // rs^2 >= 0 (or -1 on idle lanes): integer max of the bit patterns
                        const float rs2 = __int_as_float(max(__float_as_int(rsi2[q]), __float_as_int(rj)));
                        if (NNB_LE) nb[q] += (r2 <= rs2) ? 1 : 0;
                        else nb[q] += (r2 < rs2) ? 1 : 0;
                        ri = __builtin_amdgcn_rsqf(__builtin_fmaxf(r2, K.rout2));
                    } else {
                        ri = __builtin_amdgcn_rsqf(r2);
                    }
                    const float mri = mj * ri;
                    const float ri2 = ri * ri;
                    const float mri3 = mri * ri2;
                    ax[q] = __builtin_fmaf(mri3, dx, ax[q]);
                    ay[q] = __builtin_fmaf(mri3, dy, ay[q]);
                    az[q] = __builtin_fmaf(mri3, dz, az[q]);
                    p[q] -= mri;
                }
                // keep each j's VGPR copies next to their use (no hoisting of
                // the whole block's copies, which costs occupancy)
                if (VC) __builtin_amdgcn_sched_barrier(0);
            }
        }
#pragma unroll
        for (int q = 0; q < IPL; q++) {
            A[q][0] += (double)ax[q];
            A[q][1] += (double)ay[q];
            A[q][2] += (double)az[q];
            A[q][3] += (double)p[q];
            nnb[q] += nb[q];
        }
        end(b1);
    }
}

// Changeover weight of one neighbour pair (src/changeover.hpp:294-334 with
// the pair rule of :366-375, i being the first changeover): the Newtonian
// terms weighted by the changeover, f = m (1 - W_acc) / r^3 (acc factor,
// with the j's tree mass m), pg = mp (1 - W_pot) / r (pot_soft) and pt = -mp
// W_pot / r (pot_tot - pot_soft) with its potential mass mp, i.e. what
// src/hard.hpp:1404-1476 leaves for j once the linear-cutoff terms are
// removed (mp = m for a single, the backup mass for a member, 0 for an
// artificial particle).
__device__ __forceinline__ void co_pair(float r2, float mj, float mp, float rin_i, float rout_i, float rin_j,
                                        float rout_j, float &f, float &pg, float &pt)
{
    const float rinv = __builtin_amdgcn_rsqf(r2);
    const float r = r2 * rinv;  // sqrt(r^2 + eps^2), as dr_eps of src/hard.hpp:1420
    const bool use_i = rout_i > rout_j;
    const float rin = use_i ? rin_i : rin_j;
    const float rout = use_i ? rout_i : rout_j;
    const float xr = (r - rin) * __builtin_amdgcn_rcpf(rout - rin);
    const float coff = (rout - rin) * __builtin_amdgcn_rcpf(rout + rin);
    const float x = __builtin_fminf(__builtin_fmaxf(xr, 0.f), 1.f);
    const float x_1 = x - 1.f, x_2 = x_1 * x_1, x_4 = x_2 * x_2;
    const float wacc = x_4 * __builtin_fmaf(
                                 x, __builtin_fmaf(x, __builtin_fmaf(x, __builtin_fmaf(x, 35.f * coff, 20.f), 10.f), 4.f),
                                 1.f);
    const float x2 = x * x, x5 = x2 * x2 * x;
    float wpot = __builtin_fmaf(-coff * x5,
                                __builtin_fmaf(x, __builtin_fmaf(x, __builtin_fmaf(x, 5.f, -20.f), 28.f), -14.f), 1.f);
    if (xr >= 1.f) wpot = (1.f + coff) * r * __builtin_amdgcn_rcpf(rout);
    f = mj * rinv * rinv * rinv * (1.f - wacc);
    const float mpri = mp * rinv;
    pg = mpri * (1.f - wpot);
    pt = -mpri * wpot;
}

// Near EPJ blocks in changeover mode.  Every pair first gets the
// linear-cutoff terms of src/force_gpu_cuda.cu:50-77 (the same instructions
// as epj_blocks), and is tested for being a neighbour pair: r^2 + eps^2 <
// ngb2 max(rs_i, rs_j)^2 + eps^2 with ngb2 = 0.99^2 (getRSearch() = 0.99
// r_search of src/soft_ptcl.hpp:97-101,349-353 on both sides), self excluded
// (by staged slot).  The j of a block of 8 for which some lane of the wave
// has a neighbour pair are revisited (in order) and, on the neighbour pairs
// only, the linear-cutoff terms are replaced by co_pair's; the other j would
// only add zeros there.
// The self pair's -m_i/r_out is removed by the caller (src/hard.hpp:1669-1673
// adds the same term back on the CPU).
// end as in epj_blocks.
template <int IPL, int NNB_LE, class F>
__device__ __forceinline__ void epj_near_co(F &end, cfp se, cfp sec, int b_begin, int b_end, const float (&xi)[IPL],
                                            const float (&yi)[IPL], const float (&zi)[IPL],
                                            const float (&xil)[IPL], const float (&yil)[IPL],
                                            const float (&zil)[IPL], const float (&rsi2)[IPL],
                                            const int (&self)[IPL], const float (&rin_i)[IPL],
                                            const float (&rout_i)[IPL], const Consts &K, float ngb2,
                                            double (&A)[IPL][4], double (&PT)[IPL], int (&nnb)[IPL])
{
    for (int b0 = b_begin; b0 < b_end; b0 += PTH_FLUSH_BLOCKS) {
        const int b1 = min(b0 + PTH_FLUSH_BLOCKS, b_end);
        float ax[IPL], ay[IPL], az[IPL], p[IPL], pt[IPL];
        int nb[IPL];
#pragma unroll
        for (int q = 0; q < IPL; q++) { ax[q] = ay[q] = az[q] = p[q] = pt[q] = 0.f; nb[q] = 0; }
        for (int b = b0; b < b1; b++) {
            const cfp B = se + (size_t)b * 40;
            unsigned hits = 0;  // bit k: some lane has a neighbour pair with j k
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const float xj = B[k], yj = B[8 + k], zj = B[16 + k], mj = B[24 + k], rj = B[32 + k];
                const int sj = b * 8 + k;
                bool hit = false;
#pragma unroll
                for (int q = 0; q < IPL; q++) {
                    const float dx = xj - xi[q];
                    const float dy = yj - yi[q];
                    const float dz = zj - zi[q];
                    const float r2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, __builtin_fmaf(dx, dx, K.eps2)));
                    const float rs2 = __int_as_float(max(__float_as_int(rsi2[q]), __float_as_int(rj)));
                    if (NNB_LE) nb[q] += (r2 <= rs2) ? 1 : 0;
                    else nb[q] += (r2 < rs2) ? 1 : 0;
                    const float ri = __builtin_amdgcn_rsqf(__builtin_fmaxf(r2, K.rout2));
                    const float mri = mj * ri;
                    const float ri2 = ri * ri;
                    const float mri3 = mri * ri2;
                    ax[q] = __builtin_fmaf(mri3, dx, ax[q]);
                    ay[q] = __builtin_fmaf(mri3, dy, ay[q]);
                    az[q] = __builtin_fmaf(mri3, dz, az[q]);
                    p[q] -= mri;
                    hit = ((r2 < __builtin_fmaf(ngb2, rs2, K.eps2)) && sj != self[q]) ? true : hit;
                }
                if (__ballot(hit)) hits |= 1u << k;
            }
            if (hits) {
                // revisit the j with neighbour pairs
                const cfp E = sec + (size_t)b * PTH_CO_EXTRA;
                for (unsigned mk = (unsigned)uniform((int)hits); mk; mk &= mk - 1) {
                    const int k = uniform(__builtin_ctz(mk));
                    const float xj = B[k], yj = B[8 + k], zj = B[16 + k], mj = B[24 + k], rj = B[32 + k];
                    const float rinj = E[k], routj = E[8 + k];
                    const float xjl = E[16 + k], yjl = E[24 + k], zjl = E[32 + k];
                    const float mpj = E[40 + k];
                    const int sj = b * 8 + k;
#pragma unroll
                    for (int q = 0; q < IPL; q++) {
                        const float dx = xj - xi[q];
                        const float dy = yj - yi[q];
                        const float dz = zj - zi[q];
                        const float r2 =
                            __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, __builtin_fmaf(dx, dx, K.eps2)));
                        const float rs2 = __int_as_float(max(__float_as_int(rsi2[q]), __float_as_int(rj)));
                        const bool nbr = (r2 < __builtin_fmaf(ngb2, rs2, K.eps2)) && sj != self[q];
                        // the linear-cutoff terms added above
                        const float ri = __builtin_amdgcn_rsqf(__builtin_fmaxf(r2, K.rout2));
                        const float mri = mj * ri;
                        const float mri3 = mri * (ri * ri);
                        // the pair in double-float relative coordinates: the
                        // high parts are close, so their difference is exact
                        // and the separation keeps full FP32 relative
                        // precision however small it is next to |x - c|
                        const float dxp = dx + (xjl - xil[q]);
                        const float dyp = dy + (yjl - yil[q]);
                        const float dzp = dz + (zjl - zil[q]);
                        const float r2p =
                            __builtin_fmaf(dzp, dzp, __builtin_fmaf(dyp, dyp, __builtin_fmaf(dxp, dxp, K.eps2)));
                        float f, pg, ptj;
                        co_pair(r2p, mj, mpj, rin_i[q], rout_i[q], rinj, routj, f, pg, ptj);
                        ax[q] += nbr ? __builtin_fmaf(f, dxp, -mri3 * dx) : 0.f;
                        ay[q] += nbr ? __builtin_fmaf(f, dyp, -mri3 * dy) : 0.f;
                        az[q] += nbr ? __builtin_fmaf(f, dzp, -mri3 * dz) : 0.f;
                        p[q] -= nbr ? pg - mri : 0.f;
                        pt[q] += nbr ? ptj : 0.f;
                    }
                }
            }
        }
#pragma unroll
        for (int q = 0; q < IPL; q++) {
            A[q][0] += (double)ax[q];
            A[q][1] += (double)ay[q];
            A[q][2] += (double)az[q];
            A[q][3] += (double)p[q];
            PT[q] += (double)pt[q];
            nnb[q] += nb[q];
        }
        end(b1);
    }
}

// One staged SPJ record held in registers (SGPRs unless VC).
struct SpjRec {
    float x, y, z, m, qxx, qyy, qzz, qxy, qyz, qzx, mtr;
};

// A staged SPJ position and its table index (scalar loads).
struct SpjPos {
    float x, y, z;
    int id;
};
__device__ __forceinline__ SpjPos spj_pos(cfp ss, int s)
{
    const cfp R = ss + (size_t)s * PTH_SPJ_STAGED;
    return SpjPos{R[0], R[1], R[2], __float_as_int(R[3])};
}

// One SPJ record from wave-uniform addresses: its staged position and its
// table entry, scalar loads used as SGPR operands, or with VC copied into
// VGPRs first.
template <bool VC> __device__ __forceinline__ SpjRec spj_rec(const SpjPos &q, cfp tab)
{
    const cfp T = tab + (size_t)q.id * 8;
    return SpjRec{jv<VC>(q.x), jv<VC>(q.y), jv<VC>(q.z), jv<VC>(T[0]), jv<VC>(T[1]), jv<VC>(T[2]),
                  jv<VC>(T[3]),  jv<VC>(T[4]), jv<VC>(T[5]), jv<VC>(T[6]), jv<VC>(T[7])};
}

// One SPJ record against the lane's i (src/force_gpu_cuda.cu:276-323 in the
// traceless form of src/phantomquad_for_p3t_x86.hpp:144-163)
template <int IPL>
__device__ __forceinline__ void spj_pair(const SpjRec &c, const float (&xi)[IPL], const float (&yi)[IPL],
                                         const float (&zi)[IPL], const Consts &K, float (&ax)[IPL],
                                         float (&ay)[IPL], float (&az)[IPL], float (&p)[IPL])
{
#pragma unroll
    for (int q = 0; q < IPL; q++) {
        const float dx = xi[q] - c.x;
        const float dy = yi[q] - c.y;
        const float dz = zi[q] - c.z;
        const float r2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, __builtin_fmaf(dx, dx, K.eps2)));
        const float ri = __builtin_amdgcn_rsqf(r2);
        const float ri2 = ri * ri;
        const float ri3 = ri * ri2;
        const float ri4 = ri2 * ri2;
        const float ri5 = ri2 * ri3;
        const float qrx = __builtin_fmaf(c.qzx, dz, __builtin_fmaf(c.qxy, dy, c.qxx * dx));
        const float qry = __builtin_fmaf(c.qyz, dz, __builtin_fmaf(c.qxy, dx, c.qyy * dy));
        const float qrz = __builtin_fmaf(c.qyz, dy, __builtin_fmaf(c.qzx, dx, c.qzz * dz));
        const float rqr = __builtin_fmaf(qrz, dz, __builtin_fmaf(qry, dy, __builtin_fmaf(qrx, dx, c.mtr)));
        const float rqr_ri4 = rqr * ri4;
        const float meff = __builtin_fmaf(rqr_ri4, K.half, c.m);
        const float meff3 = __builtin_fmaf(rqr_ri4, K.two_half, c.m) * ri3;
        p[q] = __builtin_fmaf(-meff, ri, p[q]);
        ax[q] = __builtin_fmaf(-meff3, dx, __builtin_fmaf(ri5, qrx, ax[q]));
        ay[q] = __builtin_fmaf(-meff3, dy, __builtin_fmaf(ri5, qry, ay[q]));
        az[q] = __builtin_fmaf(-meff3, dz, __builtin_fmaf(ri5, qrz, az[q]));
    }
}

template <int IPL>
__device__ __forceinline__ void spj_flush(const float (&ax)[IPL], const float (&ay)[IPL], const float (&az)[IPL],
                                          const float (&p)[IPL], double (&A)[IPL][4])
{
#pragma unroll
    for (int q = 0; q < IPL; q++) {
        A[q][0] += (double)ax[q];
        A[q][1] += (double)ay[q];
        A[q][2] += (double)az[q];
        A[q][3] += (double)p[q];
    }
}

// SPJ records [s_begin, s_end): the next record's table entry and the
// position after it are loaded before the current record is used (scalar
// loads in flight during the pair arithmetic instead of a wait at the top of
// every record; the table index comes from the position loaded one record
// earlier).  end(s) is called after the sums up to record s are in A.
template <int IPL, bool VC, class F>
__device__ __forceinline__ void spj_records(F &end, cfp ss, cfp tab, int s_begin, int s_end, const float (&xi)[IPL],
                                            const float (&yi)[IPL], const float (&zi)[IPL], const Consts &K,
                                            double (&A)[IPL][4])
{
    if (s_begin >= s_end) return;
    SpjRec c = spj_rec<VC>(spj_pos(ss, s_begin), tab);
    SpjPos pn = spj_pos(ss, min(s_begin + 1, s_end - 1));
    for (int s0 = s_begin; s0 < s_end; s0 += PTH_FLUSH_SPJ) {
        const int s1 = min(s0 + PTH_FLUSH_SPJ, s_end);
        float ax[IPL], ay[IPL], az[IPL], p[IPL];
#pragma unroll
        for (int q = 0; q < IPL; q++) ax[q] = ay[q] = az[q] = p[q] = 0.f;
        for (int s = s0; s < s1; s++) {
            // the next record and the position after it (the last ones are
            // re-read: stays in bounds)
            const SpjPos pnn = spj_pos(ss, min(s + 2, s_end - 1));
            const SpjRec n = spj_rec<VC>(pn, tab);
            spj_pair<IPL>(c, xi, yi, zi, K, ax, ay, az, p);
            c = n;
            pn = pnn;
        }
        spj_flush<IPL>(ax, ay, az, p, A);
        end(s1);
    }
}

// Arguments of the fused force launches.
struct ForceArgs {
    const Item *items;
    int n_items;
    const Item *items1;  // split launches: the items of 1 i per lane
    // persistent launches: the class's 8 item counters (one per XCD) and the
    // slots of each XCD's run of items
    int *counter;
    int n_run;
    const int *near_blk;
    const float4 *staged_i;
    const float *staged_e, *staged_s;
    const SpjTab *spj_tab;
    const float4 *staged_ic;  // changeover mode
    const float4 *staged_il;  // changeover mode
    const float *staged_ec;   // changeover mode
    const float *staged_el;   // linear mode, double-float near pairs
    float eps2, rout2, ngb2;
    double G;
    double4 *out_accp;
    int *out_nnb;
    double *out_pott;  // changeover mode
    double4 *part_accp;
    int *part_nnb;
    double *part_pott;  // changeover mode
};

__device__ __forceinline__ Item load_item(const Item *items, int idx)
{
    const cip ci = (cip)(items) + (size_t)idx * 8;
    Item it;
    it.walk = ci[0];
    it.i_begin = ci[1];
    it.n_i_ipl = ci[2];
    it.e_blk_begin = ci[3];
    it.e_blk_end = ci[4];
    it.s_begin = ci[5];
    it.s_end = ci[6];
    it.part = ci[7];
    return it;
}

// A work item's j-range falls into four quarters of about equal cost, cut
// where the FP32 partial sums are flushed: each quarter is summed in FP64 by
// itself, and the quarters' sums are added in order.  So one wave that takes
// the quarters in turn and four waves that take one each give the same bits,
// and a launch is free to do either.  A wave that takes all four pays for
// them: force phase of 4,194,304 particles at chunk 1024 37.3 to 37.6 ms,
// changeover 30.3 to 30.65 (3,000,000); of 8,388,608 with 3 i per lane nothing
// in one segment, 0.8 of 89.3 ms pipelined, changeover 1.4 of 95.3.
struct Cut {
    bool in_e;  // among the EPJ blocks (at most their end), or the SPJ records
    int e, s;   // blocks before e and records before s come before the cut
};
__device__ __forceinline__ Cut cut_at(const Item &it, int near_end, int k)
{
    const int nb = it.e_blk_end - it.e_blk_begin, ns = it.s_end - it.s_begin;
    const int m = min(max(near_end, it.e_blk_begin), it.e_blk_end);
    const long long ue = 8ll * nb, u = (ue + 2ll * ns) * k / 4;
    Cut c{k < 4 && u <= ue, it.e_blk_end, it.s_begin};
    // whole flush groups: 8 blocks from the range's begin, or from where its
    // far part begins; 32 records
    if (c.in_e) {
        const int x = min(nb, ((int)(u >> 3) + PTH_FLUSH_BLOCKS / 2) & ~(PTH_FLUSH_BLOCKS - 1));
        c.e = it.e_blk_begin + x;
        if (c.e > m && x < nb)
            c.e = min(m + ((c.e - m + PTH_FLUSH_BLOCKS - 1) & ~(PTH_FLUSH_BLOCKS - 1)), it.e_blk_end);
    } else if (k < 4) {
        c.s += min(ns, ((int)((u - ue) >> 1) + PTH_FLUSH_SPJ / 2) & ~(PTH_FLUSH_SPJ - 1));
    } else {
        c.s = it.s_end;
    }
    return c;
}

// The i of a tile held by one lane (i = i_begin + lane + 64 k).
template <int IPL> struct Tile {
    float x[IPL], y[IPL], z[IPL], rs2[IPL];
    float xl[IPL], yl[IPL], zl[IPL];               // low parts (DF, CO)
    float rin[IPL], rout[IPL], m[IPL];             // CO
    int self[IPL];                                 // CO
};
template <int IPL, bool CO, bool DF>
__device__ __forceinline__ void load_tile(const ForceArgs &a, const Item &it, int lane, Tile<IPL> &t)
{
    const int n_i = item_n_i(it.n_i_ipl);
#pragma unroll
    for (int q = 0; q < IPL; q++) {
        const bool in = lane + 64 * q < n_i;
        float4 v = make_float4(0.f, 0.f, 0.f, -1.f);
        if (in) v = a.staged_i[it.i_begin + lane + 64 * q];
        t.x[q] = v.x;
        t.y[q] = v.y;
        t.z[q] = v.z;
        t.rs2[q] = v.w;
        if constexpr (DF || CO) {
            float4 l = make_float4(0.f, 0.f, 0.f, 0.f);
            if (in) l = a.staged_il[it.i_begin + lane + 64 * q];
            t.xl[q] = l.x;
            t.yl[q] = l.y;
            t.zl[q] = l.z;
        }
        if constexpr (CO) {
            float4 c = make_float4(__int_as_float(-2), 0.f, 0.f, 0.f);
            if (in) c = a.staged_ic[it.i_begin + lane + 64 * q];
            t.self[q] = __float_as_int(c.x);
            t.rin[q] = c.y;
            t.rout[q] = c.z;
            t.m[q] = c.w;
        }
    }
}

// Components of an i's FP64 sums: acc, pot and, in changeover mode, the
// potential still missing from the total.
template <bool CO> constexpr int n_sum = CO ? 5 : 4;

// Adds the tile's sums over EPJ blocks [e0, e_mid) near and [e_mid, e1) far
// and SPJ records [s0, s1) to A, PT and nnb; between the blocks and the
// records, and wherever sums are flushed, end is told how far they go.
template <int IPL, int NNB_LE, bool VC, bool CO, bool DF, class F>
__device__ __forceinline__ void sum_range(F &end, const ForceArgs &a, const Tile<IPL> &t, int e0, int e_mid, int e1,
                                          int s0, int s1, const Consts &K, double (&A)[IPL][4], double (&PT)[IPL],
                                          int (&nnb)[IPL])
{
    const cfp se = as_const(a.staged_e);
    if constexpr (CO) {
        epj_near_co<IPL, NNB_LE>(end, se, as_const(a.staged_ec), e0, e_mid, t.x, t.y, t.z, t.xl, t.yl, t.zl, t.rs2,
                                 t.self, t.rin, t.rout, K, a.ngb2, A, PT, nnb);
    } else if constexpr (DF) {
        epj_blocks<IPL, NNB_LE, true, VC, true>(end, se, e0, e_mid, t.x, t.y, t.z, t.rs2, K, A, nnb,
                                                as_const(a.staged_el), t.xl, t.yl, t.zl);
    } else
        epj_blocks<IPL, NNB_LE, true, VC>(end, se, e0, e_mid, t.x, t.y, t.z, t.rs2, K, A, nnb);
    epj_blocks<IPL, NNB_LE, false, VC>(end, se, e_mid, e1, t.x, t.y, t.z, t.rs2, K, A, nnb);
    end.records(s0);
    spj_records<IPL, VC>(end, as_const(a.staged_s), as_const(reinterpret_cast<const float *>(a.spj_tab)), s0, s1, t.x,
                         t.y, t.z, K, A);
}

// Changeover mode: the self pairs' linear-cutoff potentials -m_i / max(eps,
// r_out) (added in the near loop with these same FP32 operations) are removed
// in the item whose j-range [e0, e_mid) holds the i's own entry, once all its
// sums are made.
template <int IPL>
__device__ __forceinline__ void drop_self(const Tile<IPL> &t, int e0, int e_mid, const Consts &K, double (&A)[IPL][4])
{
#pragma unroll
    for (int q = 0; q < IPL; q++) {
        const int sb = t.self[q] >> 3;
        if (t.self[q] >= 0 && sb >= e0 && sb < e_mid)
            A[q][3] += (double)(t.m[q] * __builtin_amdgcn_rsqf(__builtin_fmaxf(K.eps2, K.rout2)));
    }
}

// Sums of slot q of a tile to the outputs, or to the item's partial slot.
template <bool CO>
__device__ __forceinline__ void store_sums(const ForceArgs &a, const Item &it, int lane, int q, const double (&A)[4],
                                           double PT, int nnb)
{
    const int i = lane + 64 * q;
    if (i >= item_n_i(it.n_i_ipl)) return;
    const double G = a.G;
    if (it.part < 0) {
        a.out_accp[it.i_begin + i] = make_double4(G * A[0], G * A[1], G * A[2], G * A[3]);
        a.out_nnb[it.i_begin + i] = nnb;
        if constexpr (CO) a.out_pott[it.i_begin + i] = G * (A[3] + PT);
    } else {
        const size_t slot = (size_t)(it.part + q) * 64 + lane;
        a.part_accp[slot] = make_double4(A[0], A[1], A[2], A[3]);
        a.part_nnb[slot] = nnb;
        if constexpr (CO) a.part_pott[slot] = A[3] + PT;
    }
}

// Ends the quarters of an item that one wave takes: the sums up to each cut
// go to LDS (T, this wave's n_sum IPL rows of 64; in registers they would
// cost the 2-i kernel a wave per SIMD).  `at` is the next cut among the
// blocks (records, after records()).  Scalar registers are short all through
// the j loops, so the cuts are not held in any: the changeover kernels leave
// them in LDS (C), the others work them out again from the item (3,000,000
// particles in changeover mode, pipelined, 33.57 ms with the item read again
// and 33.15 with the cuts in LDS; 4,194,304 without, force phase 37.6 and 37.85).
template <int IPL, bool CO> struct Quarters {
    static constexpr int NC = n_sum<CO>;
    const ForceArgs &a;
    int idx, k, at;
    bool first;
    double *T;
    int *C;
    double (&A)[IPL][4], (&PT)[IPL];
    __device__ __forceinline__ void start(const Item &it, int near_end)
    {
        if constexpr (CO)
            for (int q = 1; q < 4; q++) {
                const Cut c = cut_at(it, near_end, q);
                C[q] = c.in_e ? c.e : ~c.s;
            }
        next(it.e_blk_begin, false);
    }
    // the next cut after position pos (of the blocks or, with rec, records)
    __device__ __forceinline__ void next(int pos, bool rec)
    {
        if constexpr (CO) {
            at = INT_MAX;
#pragma unroll 1
            for (; k < 4; k++) {
                const int v = uniform(C[k]);
                if ((v >= 0) == rec) {
                    if (!rec) break;  // the cuts left are among the records
                    continue;
                }
                const int c = rec ? ~v : v;
                if (c > pos) {
                    at = c;
                    break;
                }
            }
            return;
        }
        asm volatile("" : "+s"(idx));
        const Item it = load_item(a.items, idx);
        const int near_end = ((cip)(a.near_blk))[it.walk];
        at = INT_MAX;
        for (; k < 4; k++) {
            const Cut c = cut_at(it, near_end, k);
            if (c.in_e == rec) {
                if (!rec) break;
                continue;
            }
            if ((rec ? c.s : c.e) > pos) {
                at = rec ? c.s : c.e;
                break;
            }
        }
    }
    __device__ __forceinline__ void close()
    {
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int q = 0; q < IPL; q++) {
            double *Tq = T + (size_t)(q * NC) * 64 + lane;
#pragma unroll
            for (int c = 0; c < NC; c++) {
                double &v = c < 4 ? A[q][c] : PT[q];
                Tq[c * 64] = first ? v : Tq[c * 64] + v;
                v = 0.0;
            }
        }
        first = false;
    }
    __device__ __forceinline__ void operator()(int pos)
    {
        if (pos < at) return;
        close();
        next(pos, rec_);
    }
    bool rec_ = false;
    // between the blocks and the records: a cut may lie just there
    __device__ __forceinline__ void records(int s0)
    {
        rec_ = true;
        const int k0 = k;
        next(s0, true);
        if (k > k0) close();
    }
    // the item's sums
    __device__ __forceinline__ void finish()
    {
        if (first) return;
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int q = 0; q < IPL; q++) {
            const double *Tq = T + (size_t)(q * NC) * 64 + lane;
#pragma unroll
            for (int c = 0; c < 4; c++) A[q][c] = Tq[c * 64] + A[q][c];
            if constexpr (CO) PT[q] = Tq[4 * 64] + PT[q];
        }
    }
};
struct NoQuarters {
    __device__ __forceinline__ void operator()(int) const {}
    __device__ __forceinline__ void records(int) const {}
};

// One item by one wave.
template <int IPL, int NNB_LE, bool VC, bool CO, bool DF>
__device__ __forceinline__ void run_tile(const ForceArgs &a, int idx, int lane, const Consts &K, double *T, int *C)
{
    Tile<IPL> t;
    double A[IPL][4], PT[IPL];
    int nnb[IPL];
#pragma unroll
    for (int q = 0; q < IPL; q++) {
        nnb[q] = 0;
        A[q][0] = A[q][1] = A[q][2] = A[q][3] = PT[q] = 0.0;
    }
    const Item it = load_item(a.items, idx);
    if (it.walk < 0) return;  // an empty slot
    load_tile<IPL, CO, DF>(a, it, lane, t);
    const int near_end = ((cip)(a.near_blk))[it.walk];
    const int e_mid = min(max(near_end, it.e_blk_begin), it.e_blk_end);
    Quarters<IPL, CO> end{a, idx, 1, 0, true, T, C, A, PT};
    end.start(it, near_end);
    sum_range<IPL, NNB_LE, VC, CO, DF>(end, a, t, it.e_blk_begin, e_mid, it.e_blk_end, it.s_begin, it.s_end, K, A, PT,
                                       nnb);
    end.finish();
    if constexpr (CO) drop_self<IPL>(t, it.e_blk_begin, e_mid, K, A);
#pragma unroll
    for (int q = 0; q < IPL; q++) store_sums<CO>(a, it, lane, q, A[q], PT[q], nnb[q]);
}

// One item by the four waves of a workgroup, a quarter each; wave q then adds
// up the sums of slot q.  All waves of the workgroup call it with the same
// item.
template <int IPL, int NNB_LE, bool CO, bool DF>
__device__ __forceinline__ void run_tile_split(const ForceArgs &a, const Item *items, int idx, int wave, int lane,
                                               const Consts &K, double *T, int *N)
{
    constexpr int NC = n_sum<CO>;
    Tile<IPL> t;
    double A[IPL][4], PT[IPL];
    int nnb[IPL];
#pragma unroll
    for (int q = 0; q < IPL; q++) {
        nnb[q] = 0;
        A[q][0] = A[q][1] = A[q][2] = A[q][3] = PT[q] = 0.0;
    }
    const Item it = load_item(items, idx);
    if (it.walk < 0) return;  // an empty slot
    load_tile<IPL, CO, DF>(a, it, lane, t);
    const int near_end = ((cip)(a.near_blk))[it.walk];
    const int e_mid = min(max(near_end, it.e_blk_begin), it.e_blk_end);
    const Cut c0 = cut_at(it, near_end, wave), c1 = cut_at(it, near_end, wave + 1);
    const int e0 = wave ? c0.e : it.e_blk_begin, s0 = wave ? c0.s : it.s_begin;
    NoQuarters end;
    sum_range<IPL, NNB_LE, false, CO, DF>(end, a, t, e0, min(max(e_mid, e0), c1.e), c1.e, s0, c1.s, K, A, PT, nnb);
#pragma unroll
    for (int q = 0; q < IPL; q++) {
        double *Tq = T + (size_t)((wave * IPL + q) * NC) * 64 + lane;
#pragma unroll
        for (int c = 0; c < 4; c++) Tq[c * 64] = A[q][c];
        if constexpr (CO) Tq[4 * 64] = PT[q];
        N[(wave * IPL + q) * 64 + lane] = nnb[q];
    }
    __syncthreads();
    if (wave >= IPL) return;
    nnb[0] = 0;
#pragma unroll
    for (int w = 0; w < 4; w++) {
        const double *Tq = T + (size_t)((w * IPL + wave) * NC) * 64 + lane;
#pragma unroll
        for (int c = 0; c < 4; c++) A[0][c] = w ? A[0][c] + Tq[c * 64] : Tq[c * 64];
        if constexpr (CO) PT[0] = w ? PT[0] + Tq[4 * 64] : Tq[4 * 64];
        nnb[0] += N[(w * IPL + wave) * 64 + lane];
    }
    if constexpr (CO) {
        // (each lane's i of slot `wave`)
#pragma unroll
        for (int q = 1; q < IPL; q++)
            if (wave == q) {
                t.self[0] = t.self[q];
                t.m[0] = t.m[q];
            }
        const int sb = t.self[0] >> 3;
        if (t.self[0] >= 0 && sb >= it.e_blk_begin && sb < e_mid)
            A[0][3] += (double)(t.m[0] * __builtin_amdgcn_rsqf(__builtin_fmaxf(K.eps2, K.rout2)));
    }
    store_sums<CO>(a, it, lane, wave, A[0], PT[0], nnb[0]);
}

// Work item idx of this class's launch (empty slots have walk < 0).
template <int NNB_LE, int IPL, bool VC, bool CO, bool DF>
__device__ __forceinline__ void force_item(const ForceArgs &a, int idx, double *T, int *C)
{
    const Consts K{jv<VC>(a.eps2), jv<VC>(a.rout2), jv<VC>(0.5f), jv<VC>(2.5f)};
    run_tile<IPL, NNB_LE, VC, CO, DF>(a, idx, threadIdx.x & 63, K, T, C);
}

// One launch per i-per-lane class: items [0, n_items) of this class, one
// per wave; or, persistent (P), one wave per free wave slot: the waves of
// block b (on XCD b % 8, workgroups being handed to the XCDs round robin)
// take the items of that XCD's run from its counter, in plan order (most
// expensive first), until the run is done.
template <int NNB_LE, int IPL, bool VC, bool CO, bool DF, bool P>
__device__ __forceinline__ void force_items(const ForceArgs &a)
{
    __shared__ double sums[4 * IPL * n_sum<CO> * 64];
    __shared__ int cuts[4][4];  // (changeover mode)
    const int wave = uniform((int)threadIdx.x >> 6);
    double *T = sums + (size_t)wave * (IPL * n_sum<CO> * 64);
    int *C = cuts[wave];
    if constexpr (P) {
        const int x = (int)blockIdx.x & 7;
        int *cnt = a.counter + x;
        for (;;) {
            int k = 0;
            if ((threadIdx.x & 63) == 0) k = atomicAdd(cnt, 1);
            k = uniform(k);
            if (k >= a.n_run) break;
            force_item<NNB_LE, IPL, VC, CO, DF>(a, ((k >> 2) * 8 + x) * 4 + (k & 3), T, C);
        }
    } else {
        const int idx = uniform((int)blockIdx.x * 4 + ((int)threadIdx.x >> 6));
        if (idx >= a.n_items) return;
        force_item<NNB_LE, IPL, VC, CO, DF>(a, idx, T, C);
    }
}

template <int NNB_LE, int IPL, bool VC, bool CO, bool DF, bool P = false>
__global__ __launch_bounds__(256) void k_force(const ForceArgs a)
{
    force_items<NNB_LE, IPL, VC, CO, DF, P>(a);
}

// Changeover mode: its extra per-i state and the revisit of neighbour pairs
// leave room for 5 waves per SIMD at 2 i per lane; held to 7 (a few spilled
// registers, on the revisit path) the force phase runs 10% faster.  With 3
// or 4 i per lane the spills would be heavy: no limit there.
template <int NNB_LE, int IPL, bool VC, bool P = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(IPL <= 2 ? 7 : 1))) void k_force_co(const ForceArgs a)
{
    force_items<NNB_LE, IPL, VC, true, false, P>(a);
}

// Small launches: one item per workgroup, a quarter per wave, and the items
// of 2 and of 1 i per lane in one launch (a.items and its n_items slots, then
// the rest of the grid's slots at a.items1).  With few items a wave per item
// leaves the SIMDs with one or two waves that wait for their scalar loads,
// and the launch lasts as long as its longest item: 1,702 items (16,384
// particles) 140 us, 86 us in quarters.  Workgroup b, on XCD b % 8, takes the
// items of that XCD's runs.
template <int NNB_LE, bool CO, bool DF> __device__ __forceinline__ void force_split(const ForceArgs &a)
{
    __shared__ double sums[4 * 2 * n_sum<CO> * 64];
    __shared__ int ngb[4 * 2 * 64];
    const int wave = uniform((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
    const bool two = (int)blockIdx.x < a.n_items;
    const int b = two ? (int)blockIdx.x : (int)blockIdx.x - a.n_items;
    const int idx = ((b >> 5) * 8 + (b & 7)) * 4 + ((b >> 3) & 3);
    const Consts K{a.eps2, a.rout2, 0.5f, 2.5f};
    if (two) run_tile_split<2, NNB_LE, CO, DF>(a, a.items, idx, wave, lane, K, sums, ngb);
    else run_tile_split<1, NNB_LE, CO, DF>(a, a.items1, idx, wave, lane, K, sums, ngb);
}
template <int NNB_LE, bool DF> __global__ __launch_bounds__(256) void k_force_split(const ForceArgs a)
{
    force_split<NNB_LE, false, DF>(a);
}
template <int NNB_LE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(7))) void k_force_split_co(const ForceArgs a)
{
    force_split<NNB_LE, true, false>(a);
}

// ---------------------------------------------------------------------------
// force, plain per-walk form: SGPR operands, one i per lane, whole list

// NEAR blocks count neighbours and apply the cutoff; far blocks (beyond
// max(r_search, r_out) of every i of the walk, and monopole superparticles)
// have neither.
template <int NNB_LE, bool NEAR>
__device__ __forceinline__ void plain_epj(cfp se, int b_begin, int b_end, float xi, float yi, float zi,
                                          float rsi2, float eps2, float rout2, double (&A)[4], int &nnb)
{
    for (int b0 = b_begin; b0 < b_end; b0 += PTH_FLUSH_BLOCKS) {
        const int b1 = min(b0 + PTH_FLUSH_BLOCKS, b_end);
        float ax = 0.f, ay = 0.f, az = 0.f, p = 0.f;
        int nb = 0;
        for (int b = b0; b < b1; b++) {
            const cfp B = se + (size_t)b * 40;
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const float dx = B[k] - xi;
                const float dy = B[8 + k] - yi;
                const float dz = B[16 + k] - zi;
                const float r2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, __builtin_fmaf(dx, dx, eps2)));
                float ri;
                if (NEAR) {
                    const float rs2 = __int_as_float(max(__float_as_int(rsi2), __float_as_int(B[32 + k])));
                    if (NNB_LE) nb += (r2 <= rs2) ? 1 : 0;
                    else nb += (r2 < rs2) ? 1 : 0;
                    ri = __builtin_amdgcn_rsqf(__builtin_fmaxf(r2, rout2));
                } else {
                    ri = __builtin_amdgcn_rsqf(r2);
                }
                const float mri = B[24 + k] * ri;
                const float mri3 = mri * (ri * ri);
                ax = __builtin_fmaf(mri3, dx, ax);
                ay = __builtin_fmaf(mri3, dy, ay);
                az = __builtin_fmaf(mri3, dz, az);
                p -= mri;
            }
        }
        A[0] += (double)ax;
        A[1] += (double)ay;
        A[2] += (double)az;
        A[3] += (double)p;
        nnb += nb;
    }
}

__device__ __forceinline__ void plain_spj(cfp ss, cfp tab, int s_begin, int s_end, float xi, float yi, float zi,
                                          float eps2, double (&A)[4])
{
    for (int s0 = s_begin; s0 < s_end; s0 += PTH_FLUSH_SPJ) {
        const int s1 = min(s0 + PTH_FLUSH_SPJ, s_end);
        float ax = 0.f, ay = 0.f, az = 0.f, p = 0.f;
        for (int s = s0; s < s1; s++) {
            const cfp R = ss + (size_t)s * PTH_SPJ_STAGED;
            // table entry: m, q'xx, q'yy, q'zz, q'xy, q'yz, q'zx, -eps^2 tr
            const cfp T = tab + (size_t)__float_as_int(R[3]) * 8;
            const float dx = xi - R[0], dy = yi - R[1], dz = zi - R[2];
            const float m = T[0];
            const float r2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, __builtin_fmaf(dx, dx, eps2)));
            const float ri = __builtin_amdgcn_rsqf(r2);
            const float ri2 = ri * ri, ri3 = ri * ri2, ri4 = ri2 * ri2, ri5 = ri2 * ri3;
            const float qrx = __builtin_fmaf(T[6], dz, __builtin_fmaf(T[4], dy, T[1] * dx));
            const float qry = __builtin_fmaf(T[5], dz, __builtin_fmaf(T[4], dx, T[2] * dy));
            const float qrz = __builtin_fmaf(T[5], dy, __builtin_fmaf(T[6], dx, T[3] * dz));
            const float rqr = __builtin_fmaf(qrz, dz, __builtin_fmaf(qry, dy, __builtin_fmaf(qrx, dx, T[7])));
            const float rqr_ri4 = rqr * ri4;
            const float meff = __builtin_fmaf(rqr_ri4, 0.5f, m);
            const float meff3 = __builtin_fmaf(rqr_ri4, 2.5f, m) * ri3;
            p = __builtin_fmaf(-meff, ri, p);
            ax = __builtin_fmaf(-meff3, dx, __builtin_fmaf(ri5, qrx, ax));
            ay = __builtin_fmaf(-meff3, dy, __builtin_fmaf(ri5, qry, ay));
            az = __builtin_fmaf(-meff3, dz, __builtin_fmaf(ri5, qrz, az));
        }
        A[0] += (double)ax;
        A[1] += (double)ay;
        A[2] += (double)az;
        A[3] += (double)p;
    }
}

template <int NNB_LE>
__global__ __launch_bounds__(256) void k_force_plain(const WalkDev *__restrict__ walks,
                                                     const int *__restrict__ near_blk,
                                                     const float4 *__restrict__ staged_i,
                                                     const float *__restrict__ staged_e,
                                                     const float *__restrict__ staged_s,
                                                     const SpjTab *__restrict__ spj_tab,
                                                     const long long *__restrict__ es_off,
                                                     const long long *__restrict__ ss_off,
                                                     float eps2, float rout2, double G,
                                                     double4 *__restrict__ out_accp,
                                                     int *__restrict__ out_nnb)
{
    const int w = blockIdx.x;
    const WalkDev wk = walks[w];
    const int wave = uniform((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int n_tiles = (wk.n_i + 63) >> 6;
    const int eb = uniform((int)(es_off[w] >> 3)), ee = uniform((int)(es_off[w + 1] >> 3));
    const int em = min(max(uniform(near_blk[w]), eb), ee);
    // staged SPJ records of the walk (none with monopole superparticles,
    // which are staged as far EPJ entries)
    const int sb = uniform((int)ss_off[w]), se_ = uniform((int)ss_off[w + 1]);
    for (int t = wave; t < n_tiles; t += 4) {
        const int i = 64 * t + lane;
        float4 v = make_float4(0.f, 0.f, 0.f, -1.f);
        if (i < wk.n_i) v = staged_i[wk.i_off + i];
        double A[4] = {0.0, 0.0, 0.0, 0.0};
        int nnb = 0;
        plain_epj<NNB_LE, true>(as_const(staged_e), eb, em, v.x, v.y, v.z, v.w, eps2, rout2, A, nnb);
        plain_epj<NNB_LE, false>(as_const(staged_e), em, ee, v.x, v.y, v.z, v.w, eps2, rout2, A, nnb);
        plain_spj(as_const(staged_s), as_const(reinterpret_cast<const float *>(spj_tab)), sb, se_, v.x, v.y, v.z,
                  eps2, A);
        if (i < wk.n_i) {
            out_accp[wk.i_off + i] = make_double4(G * A[0], G * A[1], G * A[2], G * A[3]);
            out_nnb[wk.i_off + i] = nnb;
        }
    }
}

// One 256-thread workgroup per split tile.
template <bool CO>
__global__ __launch_bounds__(256) void k_reduce(const RItem *__restrict__ ritems,
                                                const double4 *__restrict__ part_accp,
                                                const int *__restrict__ part_nnb,
                                                const double *__restrict__ part_pott, double G,
                                                double4 *__restrict__ out_accp, int *__restrict__ out_nnb,
                                                double *__restrict__ out_pott)
{
    const RItem r = ritems[blockIdx.x];
    const int t = threadIdx.x;
    if (t >= r.n_i) return;
    const int sub = t >> 6, lane = t & 63;
    double ax = 0, ay = 0, az = 0, p = 0, pt = 0;
    int nb = 0;
    for (int k = 0; k < r.n_part; k++) {
        const size_t slot = (size_t)(r.part_first + k * r.ipl + sub) * 64 + lane;
        const double4 a = part_accp[slot];
        ax += a.x;
        ay += a.y;
        az += a.z;
        p += a.w;
        nb += part_nnb[slot];
        if constexpr (CO) pt += part_pott[slot];
    }
    out_accp[r.out + t] = make_double4(G * ax, G * ay, G * az, G * p);
    out_nnb[r.out + t] = nb;
    if constexpr (CO) out_pott[r.out + t] = G * pt;
}

// ---------------------------------------------------------------------------
// Results [i0, i0 + n) packed for the host: consecutive threads write
// consecutive words, so that the stores to host memory leave as whole lines
// (the {ax, ay, az, pot} records are read from L2 at a stride instead).
__global__ __launch_bounds__(256) void k_results(const double4 *__restrict__ accp, const int *__restrict__ nnb,
                                                 const double *__restrict__ pott, long long i0, int n,
                                                 double *__restrict__ dst)
{
    const double *in = reinterpret_cast<const double *>(accp + i0);
    double *pot = dst + 3 * (size_t)n, *pt = pot + n;
    int *nb = reinterpret_cast<int *>(pott ? pt + n : pt);
    const int step = (int)(gridDim.x * 256), t0 = (int)(blockIdx.x * 256 + threadIdx.x);
    for (int k = t0; k < 3 * n; k += step) dst[k] = in[4 * (k / 3) + k % 3];
    for (int k = t0; k < n; k += step) {
        pot[k] = in[4 * (size_t)k + 3];
        if (pott) pt[k] = pott[i0 + k];
        nb[k] = nnb[i0 + k];
    }
}

// ---------------------------------------------------------------------------
// Index lists given as runs of consecutive indices (pth_dispatch), read where
// the host encoded them (pinned memory): workgroup g expands part g / (2
// n_walk) of n_part of the runs of the EPJ list (g % (2 n_walk) < n_walk) or
// of the SPJ list of one walk.  A part is a range of runs, so that it reads
// nothing else over the link; the runs are taken EXPAND_RUNS at a time into
// LDS (first index, position), each entry they cover finds its run by a binary
// search in LDS and is written coalesced.  Bound by the link (1.6 MB of runs
// per 200-walk batch of the 1,048,576-particle cluster; against copying the
// runs together and uploading them first, that cluster's hooks 20.2 to 19.3
// ms).  A list of few runs (at most EXPAND_FEW, 512 bytes for every part to
// read) is shared out by entries instead: there are too few runs to go round,
// and one may hold the whole list.
#define EXPAND_RUNS 1024
#define EXPAND_FEW 64
__global__ __launch_bounds__(256) void k_expand_runs(const WalkDev *__restrict__ walks, int n_walk, int n_part,
                                                     const int *__restrict__ rid_e, const int *__restrict__ rpos_e,
                                                     const int *__restrict__ n_re, const int *__restrict__ rid_s,
                                                     const int *__restrict__ rpos_s, const int *__restrict__ n_rs,
                                                     int *__restrict__ out_e, int *__restrict__ out_s)
{
    __shared__ int l_id[EXPAND_RUNS], l_pos[EXPAND_RUNS + 1];
    const int part = (int)blockIdx.x / (2 * n_walk), g = (int)blockIdx.x % (2 * n_walk);
    const bool sp = g >= n_walk;
    const int w = sp ? g - n_walk : g;
    const WalkDev wk = walks[w];
    const int n = sp ? wk.n_s : wk.n_e, off = sp ? wk.s_off : wk.e_off, nr = sp ? n_rs[w] : n_re[w];
    // a walk's runs lie where its list would
    const int *__restrict__ rid = (sp ? rid_s : rid_e) + off;
    const int *__restrict__ rpos = (sp ? rpos_s : rpos_e) + off;
    int *__restrict__ out = (sp ? out_s : out_e) + off;
    const bool few = nr <= EXPAND_FEW;
    const int r0 = few ? 0 : (int)((long long)nr * part / n_part);
    const int r1 = few ? nr : (int)((long long)nr * (part + 1) / n_part);
    const int q0 = few ? (int)((long long)n * part / n_part) : 0, q1 = few ? (int)((long long)n * (part + 1) / n_part) : n;
    const int tid = (int)threadIdx.x;
    for (int c0 = r0; c0 < r1; c0 += EXPAND_RUNS) {
        const int nc = min(EXPAND_RUNS, r1 - c0);
        for (int k = tid; k <= nc; k += 256) {
            // (entry nc: where the next run begins)
            if (k < nc) l_id[k] = rid[c0 + k];
            l_pos[k] = c0 + k < nr ? rpos[c0 + k] : n;
        }
        __syncthreads();
        const int p1 = min(l_pos[nc], q1);
        for (int k = max(l_pos[0], q0) + tid; k < p1; k += 256) {
            int lo = 0, hi = nc - 1;
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (l_pos[mid] <= k) lo = mid;
                else hi = mid - 1;
            }
            out[k] = l_id[lo] + (k - l_pos[lo]);
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// The work items of a plan whose sizes the host made (make_plan with
// on_device): block b < n_walk writes walk b's items and reduction items,
// block n_walk + g the empty slots behind the runs of segment g.  A run's
// items are in walk order, where the host's planner puts the most expensive
// first: the items of walks of several chunks differ by at most a factor of
// two in cost; those of walks of one chunk may be much cheaper, and of such
// the order saved nothing (4,194,304 particles' force phase 37.86 ms in walk
// order, 37.79 in the host's).
__global__ __launch_bounds__(64) void k_plan(const WalkDev *__restrict__ walks, const WalkPlan *__restrict__ wplan,
                                             int n_walk, const SegPlan *__restrict__ splan,
                                             const long long *__restrict__ es_off,
                                             const long long *__restrict__ ss_off, Item *__restrict__ items,
                                             RItem *__restrict__ ritems)
{
    // slot of item k of run x of a class that begins at slot `begin`
    auto slot = [](int begin, int x, int k) { return begin + ((k >> 2) * 8 + x) * 4 + (k & 3); };
    const int lane = threadIdx.x;
    if ((int)blockIdx.x >= n_walk) {
        const SegPlan &sp = splan[(int)blockIdx.x - n_walk];
        const int x = lane & 7;
        for (int c = 0; c < 2; c++)
            for (int k = sp.run[c][x + 1] - sp.run[c][x] + (lane >> 3); k < sp.slots[c] / 8; k += 8)
                items[slot(sp.begin[c], x, k)] = Item{-1, 0, 0, 0, 0, 0, 0, -1};
        return;
    }
    const int w = (int)blockIdx.x;
    const WalkDev W = walks[w];
    const WalkPlan wp = wplan[w];
    const SegPlan &sp = splan[wp.seg];
    const long long es = es_off[w] >> 3, ss = ss_off[w], nb = (es_off[w + 1] >> 3) - es, ns = ss_off[w + 1] - ss;
    const int n1 = max(0, (W.n_i - 128 * wp.n2 + 63) >> 6), nt = wp.n2 + n1;
    for (int j = lane; j < nt * wp.nch; j += 64) {
        const int t = j / wp.nch, k = j - t * wp.nch;
        const bool two = t < wp.n2;
        const int c = two ? 1 : 0, u = two ? t : t - wp.n2;
        const int begin = two ? 128 * t : 128 * wp.n2 + 64 * u, n = min(two ? 128 : 64, W.n_i - begin);
        Item it;
        it.walk = w;
        it.i_begin = W.i_off + begin;
        it.n_i_ipl = item_pack(n, c + 1);
        int e0, e1, s0, s1;
        chunk_cut(nb, ns, wp.nch, k, e0, s0);
        chunk_cut(nb, ns, wp.nch, k + 1, e1, s1);
        it.e_blk_begin = (int)es + e0;
        it.e_blk_end = (int)es + e1;
        it.s_begin = (int)ss + s0;
        it.s_end = (int)ss + s1;
        const int part_first = wp.part + (two ? 2 * t : 2 * wp.n2 + u) * wp.nch;
        it.part = wp.nch > 1 ? part_first + k * (c + 1) : -1;
        const int idx = wp.item[c] + u * wp.nch + k - sp.first[c];
        int x = 0;
        for (int q = 1; q < 8; q++) x += idx >= sp.run[c][q];
        items[slot(sp.begin[c], x, idx - sp.run[c][x])] = it;
        if (k == 0 && wp.nch > 1) ritems[wp.ritem + t] = RItem{it.i_begin, n, part_first, wp.nch, c + 1, {0, 0, 0}};
    }
}

// ---------------------------------------------------------------------------
// launchers (host)

hipError_t launch_plan(const WalkDev *walks, const WalkPlan *wplan, int n_walk, const SegPlan *splan, int n_seg,
                       const long long *es_off, const long long *ss_off, Item *items, RItem *ritems, hipStream_t st)
{
    hipLaunchKernelGGL(k_plan, dim3((unsigned)(n_walk + n_seg)), dim3(64), 0, st, walks, wplan, n_walk, splan, es_off,
                       ss_off, items, ritems);
    return hipGetLastError();
}

hipError_t launch_spj_table(const SpjDev *spj, long long n, float eps2, SpjTab *tab, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_spj_table, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, spj, n, (double)eps2, tab);
    return hipGetLastError();
}

hipError_t launch_expand_runs(const WalkDev *walks, int n_walk, const int *rid_e, const int *rpos_e, const int *n_re,
                              const int *rid_s, const int *rpos_s, const int *n_rs, int *out_e, int *out_s,
                              hipStream_t st)
{
    if (n_walk <= 0) return hipSuccess;
    // parts per list: a few blocks per CU for a batch of a few hundred walks
    const int n_part = std::max(1, std::min(8, 4096 / (2 * n_walk)));
    hipLaunchKernelGGL(k_expand_runs, dim3(2u * (unsigned)n_walk * (unsigned)n_part), dim3(256), 0, st, walks, n_walk,
                       n_part, rid_e, rpos_e, n_re, rid_s, rpos_s, n_rs, out_e, out_s);
    return hipGetLastError();
}

hipError_t launch_stage(const BatchDev &b, int k, hipStream_t st)
{
    const SegDev &g = b.seg[k];
    if (g.n_walk <= 0) return hipSuccess;
    StageArgs a;
    a.walk_begin = g.walk_begin;
    a.epi = b.epi;
    a.walks = b.walks;
    a.es_off = b.es_off;
    a.ss_off = b.ss_off;
    a.id_epj = b.id_epj;
    a.id_spj = b.id_spj;
    a.epj = b.epj;
    a.spj = b.spj;
    a.r_out = std::sqrt((double)b.rout2);
    a.eps2 = (double)b.eps2;
    a.centre = b.centre;
    a.near_blk = b.near_blk;
    a.staged_i = b.staged_i;
    a.staged_e = b.staged_e;
    a.staged_s = b.staged_s;
    a.epi_id = b.epi_id;
    a.epj_co = b.epj_co;
    a.staged_ic = b.staged_ic;
    a.staged_il = b.staged_il;
    a.staged_ec = b.staged_ec;
    a.walk_err = b.walk_err;
    a.df = b.df;
    a.staged_el = b.staged_el;
    a.mono = b.mono;
    a.spj_mono = reinterpret_cast<const EpjDev *>(b.spj);
    a.counters = b.persistent ? b.counters + k * PLAN_CLASSES * 8 : nullptr;
    // SPJ parts per walk: enough blocks for a few per CU when the launch
    // has few walks (a dispatched batch), one beside each EPJ block otherwise
    a.n_walk = g.n_walk;
    a.spj_parts = b.mono ? 0 : std::max(1, std::min(8, 2048 / g.n_walk));
    const unsigned nblk = (unsigned)g.n_walk * (1u + (unsigned)a.spj_parts);
    // in changeover mode an entry also costs a hash search: 512 threads of 4
    // entries per walk where a launch has few walks (the 131,071-particle hooks
    // 2,566 to 2,466 us); without it a walk's gathers keep its CU busy, and
    // they gain nothing (16,384 particles 43 to 37 us, 40,000 43 to 53)
    if (b.co && g.n_walk <= 512)
        hipLaunchKernelGGL((k_stage_walk<true, 4, 512>), dim3(nblk), dim3(512), 0, st, a);
    else if (b.co) hipLaunchKernelGGL((k_stage_walk<true, 2, 256>), dim3(nblk), dim3(256), 0, st, a);
    else if (g.n_walk <= 2048) hipLaunchKernelGGL((k_stage_walk<false, 4, 256>), dim3(nblk), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((k_stage_walk<false, 2, 256>), dim3(nblk), dim3(256), 0, st, a);
    return hipGetLastError();
}

// 256-thread blocks of kernel f that the current device holds at once
static unsigned fit_blocks(const void *f)
{
    static std::mutex m;
    static std::unordered_map<const void *, int> per_cu;
    static int cus[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    std::lock_guard<std::mutex> lk(m);
    if (!cus[dev] && hipDeviceGetAttribute(&cus[dev], hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return 0;
    auto it = per_cu.find(f);
    if (it == per_cu.end()) {
        int nb = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, f, 256, 0) != hipSuccess) return 0;
        it = per_cu.emplace(f, nb).first;
    }
    return (unsigned)(it->second * cus[dev]);
}

// Whether a batch's force launches take an item per workgroup (and both
// i-per-lane classes at once).  A launch ends with its longest items, and one
// of a few rounds of waves (8,192 slots) is much of it tail: quarters of items
// shorten that.  Against that stand the four loads of a tile's i and a
// barrier, which other segments' launches beside it do not need: they fill the
// tail.  The changeover kernels wait more than they issue and gain longer.
// Decided by the largest segment, for all: with the first, half-size one
// split and the others not, 2,000,000 particles took 22.1 ms, where either
// form alone takes 21.75 and 22.0.  ms per evaluation, a wave against a
// workgroup per item, by items of the largest launch:
//   one segment: 1,641 0.219 and 0.142; 31,000 1.420 and 1.358; 57,000 2.507
//     and 2.495; 79,000 3.45 and 3.47; 124,000 5.38 and 5.50
//   eight on three streams: 24,000 7.83 and 7.59; 35,000 11.11 and 11.10;
//     43,000 13.45 and 13.48; 52,000 15.88 and 16.03; 109,000 33.24 and 33.89
//   changeover, one: 57,000 2.79 and 2.61; 124,000 5.78 and 5.73; 182,000 8.74
//     and 8.77; 392,000 16.7 and 17.1
//   changeover, eight: 35,000 11.86 and 11.38; 72,000 22.03 and 21.49; 147,000
//     45.4 and 44.6
// The kernel holds 1 and 2 i per lane.
constexpr int SPLIT_ITEMS = 65536, SPLIT_ITEMS_SEGMENTS = 40960, SPLIT_ITEMS_CO = 163840;
bool split_launch(const BatchDev &b)
{
    if (b.plain || b.persistent || b.j_vgpr) return false;
    const int limit = b.co ? SPLIT_ITEMS_CO : b.n_seg > 1 ? SPLIT_ITEMS_SEGMENTS : SPLIT_ITEMS;
    for (int k = 0; k < b.n_seg; k++) {
        const SegDev &g = b.seg[k];
        if (g.seg_count[2] + g.seg_count[3] > 0 || g.seg_count[0] + g.seg_count[1] > limit) return false;
    }
    return true;
}

// nblk blocks of one item per wave; persistent (P): as many blocks as the
// device holds, at most nblk, a multiple of 8 so that every XCD's run of
// items has blocks that drain it
template <int NNB, bool VC, bool CO, bool DF, bool P>
static void launch_class(int ipl, unsigned nblk, const ForceArgs &a, hipStream_t st)
{
    auto go = [&](void (*kern)(ForceArgs)) {
        unsigned n = nblk;
        if constexpr (P) n = std::max(8u, std::min(nblk, fit_blocks((const void *)kern)) & ~7u);
        hipLaunchKernelGGL(kern, dim3(n), dim3(256), 0, st, a);
    };
    if constexpr (CO) {
        if (ipl == 1) go(k_force_co<NNB, 1, VC, P>);
        else if (ipl == 2) go(k_force_co<NNB, 2, VC, P>);
        else if (ipl == 3) go(k_force_co<NNB, 3, VC, P>);
        else go(k_force_co<NNB, 4, VC, P>);
    } else {
        if (ipl == 1) go(k_force<NNB, 1, VC, false, DF, P>);
        else if (ipl == 2) go(k_force<NNB, 2, VC, false, DF, P>);
        else if (ipl == 3) go(k_force<NNB, 3, VC, false, DF, P>);
        else go(k_force<NNB, 4, VC, false, DF, P>);
    }
}

template <int NNB, bool VC, bool CO, bool DF>
static void launch_class(bool persistent, int ipl, unsigned nblk, const ForceArgs &a, hipStream_t st)
{
    if (persistent) launch_class<NNB, VC, CO, DF, true>(ipl, nblk, a, st);
    else launch_class<NNB, VC, CO, DF, false>(ipl, nblk, a, st);
}

hipError_t launch_force(const BatchDev &b, int k, hipStream_t st, unsigned classes)
{
    const SegDev &g = b.seg[k];
    if (b.plain) {
        if (b.n_walk <= 0) return hipSuccess;
        if (b.nnb_le)
            hipLaunchKernelGGL(k_force_plain<1>, dim3(b.n_walk), dim3(256), 0, st, b.walks, b.near_blk, b.staged_i,
                               b.staged_e, b.staged_s, b.spj_tab, b.es_off, b.ss_off, b.eps2, b.rout2, b.G,
                               b.out_accp, b.out_nnb);
        else
            hipLaunchKernelGGL(k_force_plain<0>, dim3(b.n_walk), dim3(256), 0, st, b.walks, b.near_blk, b.staged_i,
                               b.staged_e, b.staged_s, b.spj_tab, b.es_off, b.ss_off, b.eps2, b.rout2, b.G,
                               b.out_accp, b.out_nnb);
        return hipGetLastError();
    }
    static const int ipls[PLAN_CLASSES] = {1, 2, 3, 4};
    ForceArgs a{};
    a.near_blk = b.near_blk;
    a.staged_i = b.staged_i;
    a.staged_e = b.staged_e;
    a.staged_s = b.staged_s;
    a.spj_tab = b.spj_tab;
    a.staged_ic = b.staged_ic;
    a.staged_il = b.staged_il;
    a.staged_ec = b.staged_ec;
    a.staged_el = b.staged_el;
    a.eps2 = b.eps2;
    a.rout2 = b.rout2;
    a.ngb2 = b.ngb2;
    a.G = b.G;
    a.out_accp = b.out_accp;
    a.out_nnb = b.out_nnb;
    a.out_pott = b.out_pott;
    a.part_accp = b.part_accp;
    a.part_nnb = b.part_nnb;
    a.part_pott = b.part_pott;
    if (split_launch(b)) {
        if (!(classes & 2u)) return hipSuccess;  // both classes go with the 2-i launch
        a.items = b.items + g.seg_begin[1];
        a.n_items = g.seg_count[1];
        a.items1 = b.items + g.seg_begin[0];
        const dim3 grid((unsigned)(g.seg_count[0] + g.seg_count[1]));
        if (grid.x == 0) return hipSuccess;
        if (b.co) {
            if (b.nnb_le) hipLaunchKernelGGL(k_force_split_co<1>, grid, dim3(256), 0, st, a);
            else hipLaunchKernelGGL(k_force_split_co<0>, grid, dim3(256), 0, st, a);
        } else if (b.df) {
            if (b.nnb_le) hipLaunchKernelGGL((k_force_split<1, true>), grid, dim3(256), 0, st, a);
            else hipLaunchKernelGGL((k_force_split<0, true>), grid, dim3(256), 0, st, a);
        } else {
            if (b.nnb_le) hipLaunchKernelGGL((k_force_split<1, false>), grid, dim3(256), 0, st, a);
            else hipLaunchKernelGGL((k_force_split<0, false>), grid, dim3(256), 0, st, a);
        }
        return hipGetLastError();
    }
    // the longer classes first: the 1-i launch is about one round of waves,
    // and its run-down tail then overlaps the other force stream's work
    // instead of holding back a longer launch behind it on this stream
    for (int c = PLAN_CLASSES - 1; c >= 0; c--) {
        const int n = g.seg_count[c];
        if (n <= 0 || !((classes >> c) & 1u)) continue;
        a.items = b.items + g.seg_begin[c];
        a.n_items = n;
        // (the plan gives every class whole rows of 8 x 4 items, XCD-major)
        a.counter = b.persistent ? b.counters + (k * PLAN_CLASSES + c) * 8 : nullptr;
        a.n_run = n / 8;
        const bool pers = b.persistent != 0;
        const unsigned nblk = (unsigned)((n + 3) / 4);
        // the changeover and double-float near modes always use SGPR operands
        if (b.co) {
            if (b.nnb_le) launch_class<1, false, true, false>(pers, ipls[c], nblk, a, st);
            else launch_class<0, false, true, false>(pers, ipls[c], nblk, a, st);
        } else if (b.df) {
            if (b.nnb_le) launch_class<1, false, false, true>(pers, ipls[c], nblk, a, st);
            else launch_class<0, false, false, true>(pers, ipls[c], nblk, a, st);
        } else if (b.j_vgpr) {
            if (b.nnb_le) launch_class<1, true, false, false, false>(ipls[c], nblk, a, st);
            else launch_class<0, true, false, false, false>(ipls[c], nblk, a, st);
        } else {
            if (b.nnb_le) launch_class<1, false, false, false>(pers, ipls[c], nblk, a, st);
            else launch_class<0, false, false, false>(pers, ipls[c], nblk, a, st);
        }
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_reduce(const BatchDev &b, int k, hipStream_t st)
{
    const SegDev &g = b.seg[k];
    if (b.plain || g.n_ritems <= 0) return hipSuccess;
    const RItem *ri = b.ritems + g.ritem_begin;
    if (b.co)
        hipLaunchKernelGGL(k_reduce<true>, dim3((unsigned)g.n_ritems), dim3(256), 0, st, ri, b.part_accp,
                           b.part_nnb, b.part_pott, b.G, b.out_accp, b.out_nnb, b.out_pott);
    else
        hipLaunchKernelGGL(k_reduce<false>, dim3((unsigned)g.n_ritems), dim3(256), 0, st, ri, b.part_accp,
                           b.part_nnb, b.part_pott, b.G, b.out_accp, b.out_nnb, b.out_pott);
    return hipGetLastError();
}

hipError_t launch_results(const double4 *accp, const int *nnb, const double *pott, long long i0, int n, double *dst,
                          hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    const unsigned nblk = (unsigned)std::min(512, (n + 255) / 256);
    hipLaunchKernelGGL(k_results, dim3(nblk), dim3(256), 0, st, accp, nnb, pott, i0, n, dst);
    return hipGetLastError();
}

hipError_t launch_all(const BatchDev &b, hipStream_t st)
{
    for (int k = 0; k < b.n_seg; k++) {
        hipError_t e;
        if ((e = launch_stage(b, k, st)) || (e = launch_force(b, k, st)) || (e = launch_reduce(b, k, st))) return e;
    }
    return hipSuccess;
}

}  // namespace pth
