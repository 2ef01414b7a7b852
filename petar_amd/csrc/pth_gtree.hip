// pth_gtree.hip -- the octree, its moments, the i-groups and the interaction
// lists built on the device (pth_gtree_* of include/petar_hip.h), with the
// semantics of the host tree (petar_amd/csrc/host/tree.cpp), which stands in
// for FDPS's TreeForForceLong<...>::QuadrupoleWithSymmetrySearch
// (src/petar.hpp:619-623, 2741) and its multi-walk lists
// (src/petar.hpp:894-899):
//   1. bounding cube (FP64 min/max), 63-bit Morton keys, stable radix sort of
//      (key, index);
//   2. nodes of every level at once: a cell that starts at a particle is a
//      node when its parent holds more than n_leaf_limit particles, which a
//      few keys around the particle decide; per-block counts of every level,
//      one scan and a writing pass number the nodes level by level, each
//      level in Morton order (so children follow their parents' order), with
//      one wait for the host (the counts) in the whole build;
//   3. moments bottom-up (mass, centre of mass, raw second moment about it,
//      particle box and box widened by r_search), each node by eight lanes in
//      the host's summation order;
//   4. i-groups: largest cells with at most n_group_limit particles (or
//      leaves), in Morton order (decided and counted with the nodes, as are
//      the neighbour search's tiles of at most 64);
//   5. walk: one wave per group (four of up to WALK_WIDE groups) traverses the
//      tree with a stack in LDS, popping up to 64 (256) nodes at a time; a node
//      is opened when it contains
//      the group, when the group box is closer to its centre of mass than
//      L/theta, or when the boxes overlap with either side widened by
//      r_search; opened leaves go to the group's leaf list, closed nodes to
//      its node list, both in batch order, in regions of the last build's
//      lengths (a first build counts before it writes);
//   6. lists: one workgroup per group puts its nodes and leaves into the host
//      walk's depth-first order (canonical order) and expands the leaves
//      into their particles.
// Every decision is the same FP64 expression as on the host (no FMA
// contraction in this file), so the lists are the host's lists as sets, and
// entry for entry after the canonical ordering.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <chrono>
#include <climits>
#include <cmath>

#include "pth_internal.h"

#pragma clang fp contract(off)

namespace {

constexpr int GT_MAX_LEVEL = 21;
constexpr long long WALK_WIDE = 1024;
constexpr int WALK_STACK = 2048;  // LDS node stack of one walking wave (8 KB: 20 waves per CU;
                                  // 4096 ran the precision workload's walk in 4.1 ms, 2048 and 2560
                                  // in 3.2 ms, 1536 in 4.7 ms, 1024 in 10.3 ms)

struct GNode {
    long long begin, end;
    int level, n_child;
    long long first_child;
};

__device__ __forceinline__ unsigned long long spread3(unsigned long long v)
{
    v &= 0x1fffffull;
    v = (v | v << 32) & 0x1f00000000ffffull;
    v = (v | v << 16) & 0x1f0000ff0000ffull;
    v = (v | v << 8) & 0x100f00f00f00f00full;
    v = (v | v << 4) & 0x10c30c30c30c30c3ull;
    v = (v | v << 2) & 0x1249249249249249ull;
    return v;
}

// per-block min/max of the coordinates, max of r_search (rs may be null) and
// a flag for non-finite values (which fmin/fmax would skip):
// part[block * 8 + {0..2: min, 3..5: max, 6: max rs, 7: 1 if any non-finite}]
__global__ __launch_bounds__(256) void k_bbox(const double *__restrict__ pos, const double *__restrict__ rs,
                                              long long n, double *__restrict__ part)
{
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300}, rmax = 0.0, bad = 0.0;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        for (int d = 0; d < 3; d++) {
            const double x = pos[3 * i + d];
            lo[d] = fmin(lo[d], x);
            hi[d] = fmax(hi[d], x);
            if (!isfinite(x)) bad = 1.0;
        }
        if (rs) {
            rmax = fmax(rmax, rs[i]);
            if (!isfinite(rs[i])) bad = 1.0;
        }
    }
    __shared__ double red[4][8];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int off = 32; off > 0; off >>= 1) {
        for (int d = 0; d < 3; d++) {
            lo[d] = fmin(lo[d], __shfl_xor(lo[d], off, 64));
            hi[d] = fmax(hi[d], __shfl_xor(hi[d], off, 64));
        }
        rmax = fmax(rmax, __shfl_xor(rmax, off, 64));
        bad = fmax(bad, __shfl_xor(bad, off, 64));
    }
    if (lane == 0) {
        for (int d = 0; d < 3; d++) {
            red[wave][d] = lo[d];
            red[wave][3 + d] = hi[d];
        }
        red[wave][6] = rmax;
        red[wave][7] = bad;
    }
    __syncthreads();
    if (threadIdx.x < 8) {
        const int d = threadIdx.x;
        double v = red[0][d];
        for (int w = 1; w < 4; w++) v = (d < 3) ? fmin(v, red[w][d]) : fmax(v, red[w][d]);
        part[blockIdx.x * 8 + d] = v;
    }
}

// What the host reads back from a build: the root cube and the sizes.
struct TreeMeta {
    double root[3], scale, len, rs_max, bad;
    int level_start[GT_MAX_LEVEL + 2];  // first node of each level, then the node count
    int n_group, n_tile;
};

// The root cube from the nb blocks' partial boxes (the host tree's
// expressions).
__global__ __launch_bounds__(1024) void k_root(const double *__restrict__ part, int nb, TreeMeta *__restrict__ meta)
{
    // thread t reduces component t % 8 over the blocks t / 8, t / 8 + 128, ..
    __shared__ double red[128][8];
    const int c = threadIdx.x & 7, row = threadIdx.x >> 3;
    double q = c < 3 ? 1e300 : c < 6 ? -1e300 : 0.0;
    for (int b = row; b < nb; b += 128) q = c < 3 ? fmin(q, part[8 * b + c]) : fmax(q, part[8 * b + c]);
    red[row][c] = q;
    __syncthreads();
    for (int half = 64; half > 0; half >>= 1) {
        if (row < half) red[row][c] = c < 3 ? fmin(red[row][c], red[row + half][c]) : fmax(red[row][c], red[row + half][c]);
        __syncthreads();
    }
    if (threadIdx.x) return;
    const double *v = red[0];
    double len = 0;
    for (int d = 0; d < 3; d++) len = fmax(len, v[3 + d] - v[d]);
    len = (len > 0) ? len * (1.0 + 1e-9) : 1.0;
    for (int d = 0; d < 3; d++) meta->root[d] = 0.5 * (v[d] + v[3 + d]) - 0.5 * len;
    meta->scale = (double)(1u << GT_MAX_LEVEL) / len;
    meta->len = len;
    meta->rs_max = v[6];
    meta->bad = v[7];
}

__global__ __launch_bounds__(256) void k_keys(const double *__restrict__ pos, long long n,
                                              const TreeMeta *__restrict__ meta, unsigned long long *__restrict__ key,
                                              int *__restrict__ idx)
{
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const double scale = meta->scale;
    unsigned long long c[3];
    for (int d = 0; d < 3; d++) {
        const double f = (pos[3 * i + d] - meta->root[d]) * scale;
        long long v = (long long)floor(f);
        v = min(max(v, 0LL), (long long)(1u << GT_MAX_LEVEL) - 1);
        c[d] = (unsigned long long)v;
    }
    key[i] = spread3(c[0]) << 2 | spread3(c[1]) << 1 | spread3(c[2]);
    idx[i] = (int)i;
}

__global__ __launch_bounds__(256) void k_gather(long long n, const int *__restrict__ sidx,
                                                long long *__restrict__ order, const double *__restrict__ pos, const double *__restrict__ mass,
                                                const double *__restrict__ rs, double *__restrict__ spos,
                                                double *__restrict__ smass, double *__restrict__ srs)
{
    const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    const long long i = sidx[k];
    order[k] = i;
    for (int d = 0; d < 3; d++) spos[3 * k + d] = pos[3 * i + d];
    smass[k] = mass[i];
    srs[k] = rs ? rs[i] : 0.0;
}

// ---- nodes ------------------------------------------------------------------
// A cell of level l is a maximal run of equal 3l-bit key prefixes; it is a
// node when its parent holds more than n_leaf particles (level 0: always).
// The cells that start at particle k are those of the levels from
// d = 1 + (levels shared with particle k - 1) on, so the nodes starting at k
// are consecutive levels d .. e: all down to the first with at most n_leaf
// particles, which key k + n_leaf decides, and the one of level d only if
// its parent (which starts before k) is large enough.  So all levels come
// from one pass over the keys, where splitting level by level took three
// launches and a wait for the host each (bound by those: 16,384 particles,
// 9 levels, 550 us for the tree; 176 us now, 1,048,576 particles 1.21 ms and
// 0.56 ms).

// levels on which two keys agree (21: the same key)
__device__ __forceinline__ int common_levels(unsigned long long a, unsigned long long b)
{
    const unsigned long long x = a ^ b;
    return x ? GT_MAX_LEVEL - 1 - (63 - __clzll((long long)x)) / 3 : GT_MAX_LEVEL;
}

// The sorted keys around a block of 256 particles: those up to KEY_HALO away
// in LDS, the others in memory.  The decisions below are chains of some 30
// dependent reads (binary searches), which from memory took 15 us at 16,384
// particles and 43 us at 1,048,576 (10 and 36 so).
constexpr int KEY_HALO = 512;
struct KeyWindow {
    const unsigned long long *__restrict__ key;
    const unsigned long long *lds;  // keys [k0, k0 + n_lds)
    long long k0;
    int n_lds;
    __device__ __forceinline__ unsigned long long operator[](long long k) const
    {
        const long long j = k - k0;
        return j >= 0 && j < n_lds ? lds[j] : key[k];
    }
};

// How many particles of k's cell of level l lie after k and before k (at most
// m of each are looked at).
__device__ void cell_reach(const KeyWindow &key, long long n, long long k, int l, long long m, long long &left,
                           long long &right)
{
    const unsigned long long kk = key[k];
    left = right = 0;
    for (long long hi = min(m, n - 1 - k); right < hi;) {
        const long long mid = (right + hi + 1) >> 1;
        if (common_levels(kk, key[k + mid]) >= l) right = mid;
        else hi = mid - 1;
    }
    for (long long hi = min(m, k); left < hi;) {
        const long long mid = (left + hi + 1) >> 1;
        if (common_levels(kk, key[k - mid]) >= l) left = mid;
        else hi = mid - 1;
    }
}

// The nodes starting at one particle: levels d .. e (none when e < d), and
// the level of the group and of the tile among them (-1: none).
struct Starts {
    int d, e, group, tile;
};
__device__ Starts starts_at(const KeyWindow &key, long long n, long long k, long long n_leaf, long long n_group,
                            long long n_tile)
{
    const unsigned long long kk = key[k];
    Starts s{k > 0 ? common_levels(key[k - 1], kk) + 1 : 0, -1, -1, -1};
    if (s.d > GT_MAX_LEVEL) return s;
    auto shared = [&](long long m) { return k + m < n ? common_levels(kk, key[k + m]) : -1; };
    const int c = shared(n_leaf);
    long long left, right;
    if (c >= s.d || k == 0) s.e = min(GT_MAX_LEVEL, c + 1);
    else {
        // (c == d - 1: the parent reaches n_leaf particles past k)
        bool big = c == s.d - 1;
        if (!big) {
            cell_reach(key, n, k, s.d - 1, n_leaf, left, right);
            big = left + right + 1 > n_leaf;
        }
        if (!big) return s;
        s.e = s.d;
    }
    // the largest cell of at most m particles, or the leaf: the first such
    // level on the way down, unless it is d and its parent is one already
    auto level = [&](long long m) { return min(max(s.d, shared(m) + 1), s.e); };
    s.group = level(n_group);
    s.tile = level(n_tile);
    const bool ask_g = s.group == s.d && s.d > 0, ask_t = s.tile == s.d && s.d > 0;
    if (ask_g || ask_t) {
        cell_reach(key, n, k, s.d - 1, max(ask_g ? n_group : 0, ask_t ? n_tile : 0), left, right);
        if (ask_g && left + right + 1 <= n_group) s.group = -1;
        if (ask_t && left + right + 1 <= n_tile) s.tile = -1;
    }
    return s;
}

// Rows of the per-block counts: nodes of each level, nodes, groups, tiles.
constexpr int ROW_NODES = GT_MAX_LEVEL + 1, ROW_GROUPS = ROW_NODES + 1, ROW_TILES = ROW_NODES + 2,
              N_ROWS = ROW_NODES + 3;

// Counts per block of 256 particles (row-major, entry N_ROWS nblk zeroed so
// that the scan ends with the total); st: the particles' starts, packed.
__global__ __launch_bounds__(256) void k_starts(const unsigned long long *__restrict__ key, long long n, int n_leaf,
                                                int n_group, int n_tile, int nblk, int *__restrict__ cnt,
                                                unsigned *__restrict__ st)
{
    __shared__ int w[N_ROWS][4];
    __shared__ unsigned long long near[256 + 2 * KEY_HALO];
    const long long b0 = (long long)blockIdx.x * 256, k = b0 + threadIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long long w0 = max(b0 - KEY_HALO, 0LL), w1 = min(b0 + 256 + KEY_HALO, n);
    for (int j = threadIdx.x; j < (int)(w1 - w0); j += 256) near[j] = key[w0 + j];
    __syncthreads();
    Starts s{0, -1, -1, -1};
    if (k < n) {
        s = starts_at(KeyWindow{key, near, w0, (int)(w1 - w0)}, n, k, n_leaf, n_group, n_tile);
        st[k] = (unsigned)(s.d | (s.e + 1) << 8 | (s.group + 1) << 16 | (s.tile + 1) << 24);
    }
    const int n_lev = max(s.e - s.d + 1, 0);
    int nodes = 0;
    for (int l = 0; l <= GT_MAX_LEVEL; l++) {
        const int c = __popcll(__ballot(n_lev > 0 && s.d <= l && l <= s.e));
        nodes += c;
        if (lane == 0) w[l][wave] = c;
    }
    const int g = __popcll(__ballot(s.group >= 0)), t = __popcll(__ballot(s.tile >= 0));
    if (lane == 0) {
        w[ROW_NODES][wave] = nodes;
        w[ROW_GROUPS][wave] = g;
        w[ROW_TILES][wave] = t;
    }
    __syncthreads();
    const int r = threadIdx.x;
    if (r < N_ROWS) cnt[(size_t)r * nblk + blockIdx.x] = w[r][0] + w[r][1] + w[r][2] + w[r][3];
    if (blockIdx.x == 0 && r == 0) cnt[(size_t)N_ROWS * nblk] = 0;
}

// Level table and totals from the scanned counts.
__global__ __launch_bounds__(64) void k_tree_sizes(const int *__restrict__ off, int nblk, TreeMeta *__restrict__ meta)
{
    const int r = threadIdx.x;
    if (r <= ROW_NODES) meta->level_start[r] = off[(size_t)r * nblk];
    if (r == 0) {
        const int g0 = off[(size_t)ROW_GROUPS * nblk], t0 = off[(size_t)ROW_TILES * nblk];
        meta->n_group = t0 - g0;
        meta->n_tile = off[(size_t)N_ROWS * nblk] - t0;
    }
}

// Nodes (all but end and n_child), their preorder numbers (a depth-first
// walk's order: by first particle, then level) and the inverse, the groups
// and the tiles in Morton order.
__global__ __launch_bounds__(256) void k_nodes(long long n, int nblk, const int *__restrict__ off,
                                               const unsigned *__restrict__ st, GNode *__restrict__ nodes,
                                               int *__restrict__ pre, int *__restrict__ node_at,
                                               int *__restrict__ groups, int *__restrict__ tiles)
{
    __shared__ int w[N_ROWS][4];
    const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned v = k < n ? st[k] : 0u;
    const int d = (int)(v & 255u), e = (int)(v >> 8 & 255u) - 1, group = (int)(v >> 16 & 255u) - 1,
              tile = (int)(v >> 24) - 1;
    const unsigned long long below = lane ? ~0ull >> (64 - lane) : 0ull;
    // counts of the waves before this one, and the lanes' ranks
    int mine = 0, nodes_before = 0;  // nodes of the lanes before this one
    for (int l = 0; l <= GT_MAX_LEVEL; l++) {
        const unsigned long long b = __ballot(d <= l && l <= e);
        if (lane == 0) w[l][wave] = __popcll(b);
        mine += __popcll(b);
        nodes_before += __popcll(b & below);
    }
    const unsigned long long bg = __ballot(group >= 0), bt = __ballot(tile >= 0);
    if (lane == 0) {
        w[ROW_NODES][wave] = mine;
        w[ROW_GROUPS][wave] = __popcll(bg);
        w[ROW_TILES][wave] = __popcll(bt);
    }
    __syncthreads();
    auto base = [&](int r) {
        int o = off[(size_t)r * nblk + blockIdx.x];
        for (int q = 0; q < 3; q++)
            if (q < wave) o += w[r][q];
        return o;
    };
    const int p0 = base(ROW_NODES) - off[(size_t)ROW_NODES * nblk] + nodes_before;
    int child = -1;
    for (int l = GT_MAX_LEVEL; l >= 0; l--) {
        const bool in = d <= l && l <= e;
        const unsigned long long b = __ballot(in);
        if (b == 0) continue;
        const int at = base(l) + __popcll(b & below);
        if (!in) continue;
        nodes[at] = GNode{k, 0, l, 0, child};
        const int p = p0 + (l - d);
        pre[at] = p;
        node_at[p] = at;
        if (l == group) groups[base(ROW_GROUPS) - off[(size_t)ROW_GROUPS * nblk] + __popcll(bg & below)] = at;
        if (l == tile) tiles[base(ROW_TILES) - off[(size_t)ROW_TILES * nblk] + __popcll(bt & below)] = at;
        child = at;
    }
}

// End and child count of every node: the end by a search of the keys
// (doubling steps from the smallest possible size), the children being the
// nodes of the next level that start before it.
__global__ __launch_bounds__(256) void k_node_ends(GNode *__restrict__ nodes, long long nn, long long n, int n_leaf,
                                                   const unsigned long long *__restrict__ key,
                                                   const int *__restrict__ pre, int2 *__restrict__ range)
{
    const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
    if (k >= nn) return;
    const long long b = nodes[k].begin, fc = nodes[k].first_child;
    const int l = nodes[k].level;
    const unsigned long long kk = key[b];
    long long in = b, step = fc >= 0 ? (long long)n_leaf : 1;  // particle in is in the cell
    long long out = n;                                         // particle out is not
    while (in + step < n) {
        if (common_levels(kk, key[in + step]) < l) {
            out = in + step;
            break;
        }
        in += step;
        step *= 2;
    }
    while (out - in > 1) {
        const long long mid = (in + out) >> 1;
        if (common_levels(kk, key[mid]) >= l) in = mid;
        else out = mid;
    }
    nodes[k].end = out;
    range[pre[k]] = make_int2((int)b, (int)(out - b));
    if (fc < 0) return;
    int c = 1;
    for (int j = 1; j < 8; j++)
        if (fc + j < nn && nodes[fc + j].level == l + 1 && nodes[fc + j].begin < out) c = j + 1;
    nodes[k].n_child = c;
}

// A node's moments and boxes.
struct Moments {
    double M, c[3], bi[6], bo[6];
};
__device__ __forceinline__ void moments_init(Moments &v)
{
    v.M = 0;
    for (int d = 0; d < 3; d++) {
        v.c[d] = 0;
        v.bi[d] = v.bo[d] = 1e300;
        v.bi[3 + d] = v.bo[3 + d] = -1e300;
    }
}
__device__ __forceinline__ void moments_centre(Moments &v)
{
    if (v.M > 0) {
        for (int d = 0; d < 3; d++) v.c[d] /= v.M;
    } else {
        for (int d = 0; d < 3; d++) v.c[d] = 0.5 * (v.bi[d] + v.bi[3 + d]);
    }
}
// What the walks read of a node, in FP32 relative to the root cube's centre:
// the centre of mass and the two boxes, the boxes' bounds pushed outwards by
// walk_margin (more than every rounding involved), the particle range, level,
// child count, first child and preorder number.  52 B per visited node in
// the group walk (A, B, C, F), in loads of 16 B that neighbouring lanes'
// sibling nodes share lines of, against 152 B of FP64 moments: the walk is
// bound by these gathers (1,048,576 particles, 67M visits: 1.32 ms on the
// FP64 moments, 0.37 ms on these; 4,194,304: 4.6 and 1.27 ms).
struct WalkRec {
    float4 *A;  // centre of mass, first particle (int bits)
    float4 *B;  // low corner of the box widened by r_search (joined with the
                // particle box, should an r_search be negative), last particle + 1
    float4 *C;  // its high corner, level << 8 | child count
    float4 *D, *E;  // particle box (tile walks)
    int2 *F;    // first child, preorder number
};
// Above every error of an FP32 coordinate difference inside the root cube
// widened by r_search: each coordinate and difference is off by at most
// 2^-24 (len + 2 rs_max), and at most four of them meet.
__host__ __device__ inline float walk_margin(double len, double rs_max) { return (float)((len + 2.0 * rs_max) * 0x1p-21); }

struct MomentArrays {
    double *mass, *com, *quad, *box_in, *box_out;
    WalkRec rec;
    const TreeMeta *meta;
    const int *pre;
};

// Moments are made by eight lanes per node, which load its children (or eight
// of its particles at a time) side by side, pass them through LDS and each add
// up one component: the host's sums in its order.  A level waits for the one
// below it, so the chain of loads inside a node is what counts: with a thread
// per node, going through its children or particles one after the other, the
// leaves took 17 us and the inner levels 73 at 16,384 particles, 7 and 28 us so
// (1,048,576: the inner levels 100 us, 48 so).
constexpr int KID = 11;  // doubles per lane in LDS (odd, so that lanes' rows start on different banks)

__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
template <int CTRL> __device__ __forceinline__ double lane_swap(double v)
{
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double min8(double v)
{
    v = fmin(v, lane_swap<0xB1>(v));  // quad_perm [1,0,3,2]
    v = fmin(v, lane_swap<0x4E>(v));  // quad_perm [2,3,0,1]
    return fmin(v, lane_swap<0x141>(v));  // row_half_mirror
}
__device__ __forceinline__ double max8(double v)
{
    v = fmax(v, lane_swap<0xB1>(v));
    v = fmax(v, lane_swap<0x4E>(v));
    return fmax(v, lane_swap<0x141>(v));
}
// (by value: a choice among array elements would put the array into scratch)
__device__ __forceinline__ double pick(int j, double a, double b, double c, double d = 0, double e = 0, double f = 0)
{
    const double lo = j == 0 ? a : j == 1 ? b : c, hi = j == 3 ? d : j == 4 ? e : f;
    return j < 3 ? lo : hi;
}

// The eight lanes' boxes and sums (lane d < 3: m x_d, lane 3: m) joined: every
// lane gets the mass, the boxes and the centre of mass.
__device__ __forceinline__ void moments_join(Moments &v, double s, double *rows, int j)
{
#pragma unroll
    for (int d = 0; d < 3; d++) {
        v.bi[d] = min8(v.bi[d]);
        v.bi[3 + d] = max8(v.bi[3 + d]);
        v.bo[d] = min8(v.bo[d]);
        v.bo[3 + d] = max8(v.bo[3 + d]);
    }
    rows[j * KID + 5] = s;
    wave_sync();
    for (int d = 0; d < 3; d++) v.c[d] = rows[d * KID + 5];
    v.M = rows[3 * KID + 5];
    moments_centre(v);
    wave_sync();
}

// Stores of node k's moments, lane j < 6 holding component j of the
// quadrupole in q, and its walk record, a part per lane.
__device__ __forceinline__ void put_moments(const Moments &v, double q, const MomentArrays &o, const GNode &nd,
                                            long long k, int j)
{
    if (j == 7) o.mass[k] = v.M;
    if (j < 3) o.com[3 * k + j] = pick(j, v.c[0], v.c[1], v.c[2]);
    if (j < 6) {
        o.quad[6 * k + j] = q;
        o.box_in[6 * k + j] = pick(j, v.bi[0], v.bi[1], v.bi[2], v.bi[3], v.bi[4], v.bi[5]);
        o.box_out[6 * k + j] = pick(j, v.bo[0], v.bo[1], v.bo[2], v.bo[3], v.bo[4], v.bo[5]);
    }
    const double len = o.meta->len;
    const float m = walk_margin(len, o.meta->rs_max);
    float p[3], ol[3], oh[3], il[3], ih[3];
    for (int d = 0; d < 3; d++) {
        const double c = o.meta->root[d] + 0.5 * len;
        p[d] = (float)(v.c[d] - c);
        ol[d] = (float)(fmin(v.bo[d], v.bi[d]) - c) - m;
        oh[d] = (float)(fmax(v.bo[3 + d], v.bi[3 + d]) - c) + m;
        il[d] = (float)(v.bi[d] - c) - m;
        ih[d] = (float)(v.bi[3 + d] - c) + m;
    }
    const WalkRec &w = o.rec;
    if (j == 0) w.A[k] = make_float4(p[0], p[1], p[2], __int_as_float((int)nd.begin));
    if (j == 1) w.B[k] = make_float4(ol[0], ol[1], ol[2], __int_as_float((int)nd.end));
    if (j == 2) w.C[k] = make_float4(oh[0], oh[1], oh[2], __int_as_float(nd.level << 8 | nd.n_child));
    if (j == 3) w.D[k] = make_float4(il[0], il[1], il[2], 0.f);
    if (j == 4) w.E[k] = make_float4(ih[0], ih[1], ih[2], 0.f);
    if (j == 5) w.F[k] = make_int2((int)nd.first_child, o.pre[k]);
}

// Moments of the leaves.  A lane holds four particles, so that a leaf of at
// most 32 is read once.
__global__ __launch_bounds__(256) void k_leaf_moments(const GNode *__restrict__ nodes, long long nn,
                                                      const double *__restrict__ pos, const double *__restrict__ mass,
                                                      const double *__restrict__ rs, const MomentArrays out)
{
    constexpr int U = 4;
    __shared__ double lds[256 * KID];
    const long long k = (long long)blockIdx.x * 32 + (threadIdx.x >> 3);
    const int j = threadIdx.x & 7;
    if (k >= nn) return;
    const GNode nd = nodes[k];
    if (nd.n_child != 0) return;
    double *rows = lds + (threadIdx.x & ~7) * KID, *row = rows + j * KID;
    Moments v;
    moments_init(v);
    double x[U][3], m[U], s = 0, q = 0;
    const int col = min(j, 3);
    const bool once = nd.end - nd.begin <= 8 * U;
    for (long long i0 = nd.begin; i0 < nd.end; i0 += 8 * U) {
        double r[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const long long i = min(i0 + 8 * u + j, nd.end - 1);
            for (int d = 0; d < 3; d++) x[u][d] = pos[3 * i + d];
            m[u] = mass[i];
            r[u] = rs[i];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int n = (int)min(nd.end - i0 - 8 * u, 8LL);
            if (n <= 0) break;
            for (int d = 0; d < 3; d++) {  // (a lane past the end holds the last particle once more)
                v.bi[d] = fmin(v.bi[d], x[u][d]);
                v.bi[3 + d] = fmax(v.bi[3 + d], x[u][d]);
                v.bo[d] = fmin(v.bo[d], x[u][d] - r[u]);
                v.bo[3 + d] = fmax(v.bo[3 + d], x[u][d] + r[u]);
                row[d] = x[u][d];
            }
            row[3] = 1.0;
            row[4] = m[u];
            wave_sync();
            for (int t = 0; t < n; t++) s += rows[t * KID + 4] * rows[t * KID + col];
            wave_sync();
        }
    }
    moments_join(v, s, rows, j);
    // components xx, yy, zz, xy, xz, yz
    const int a = (0x100210 >> (4 * j)) & 3, b = (0x221210 >> (4 * j)) & 3;
    for (long long i0 = nd.begin; i0 < nd.end; i0 += 8 * U) {
        if (!once) {
#pragma unroll
            for (int u = 0; u < U; u++) {
                const long long i = min(i0 + 8 * u + j, nd.end - 1);
                for (int d = 0; d < 3; d++) x[u][d] = pos[3 * i + d];
                m[u] = mass[i];
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int n = (int)min(nd.end - i0 - 8 * u, 8LL);
            if (n <= 0) break;
            for (int d = 0; d < 3; d++) row[d] = x[u][d] - v.c[d];
            row[4] = m[u];
            wave_sync();
            for (int t = 0; t < n; t++) q += rows[t * KID + 4] * rows[t * KID + a] * rows[t * KID + b];
            wave_sync();
        }
    }
    put_moments(v, q, out, nd, k, j);
}

// Moments of one inner node (its children are done), eight lanes.
__device__ __forceinline__ void inner_moments(const GNode &nd, long long k, const MomentArrays &o, double *rows, int j)
{
    double *row = rows + j * KID;
    const long long c = nd.first_child + min(j, nd.n_child - 1);
    Moments v;
    double m = o.mass[c], x[3], qc[6], s = 0, q = 0;
    for (int d = 0; d < 3; d++) x[d] = o.com[3 * c + d];
    for (int d = 0; d < 6; d++) {
        v.bi[d] = o.box_in[6 * c + d];
        v.bo[d] = o.box_out[6 * c + d];
        qc[d] = o.quad[6 * c + d];
    }
    for (int d = 0; d < 3; d++) {
        v.bi[d] = fmin(1e300, v.bi[d]);
        v.bo[d] = fmin(1e300, v.bo[d]);
        v.bi[3 + d] = fmax(-1e300, v.bi[3 + d]);
        v.bo[3 + d] = fmax(-1e300, v.bo[3 + d]);
        row[d] = x[d];
    }
    row[3] = 1.0;
    row[4] = m;
    wave_sync();
    const int col = min(j, 3);
    for (int t = 0; t < nd.n_child; t++) s += rows[t * KID + 4] * rows[t * KID + col];
    wave_sync();
    moments_join(v, s, rows, j);
    for (int d = 0; d < 3; d++) x[d] -= v.c[d];
    row[5] = qc[0] + m * x[0] * x[0];
    row[6] = qc[1] + m * x[1] * x[1];
    row[7] = qc[2] + m * x[2] * x[2];
    row[8] = qc[3] + m * x[0] * x[1];
    row[9] = qc[4] + m * x[0] * x[2];
    row[10] = qc[5] + m * x[1] * x[2];
    wave_sync();
    for (int t = 0; t < nd.n_child; t++) q += rows[t * KID + 5 + min(j, 5)];
    wave_sync();
    put_moments(v, q, o, nd, k, j);
}

// The inner nodes of one level, [a, b).
__global__ __launch_bounds__(256) void k_inner_moments(const GNode *__restrict__ nodes, long long a, long long b,
                                                       const MomentArrays o)
{
    __shared__ double lds[256 * KID];
    const long long k = a + (long long)blockIdx.x * 32 + (threadIdx.x >> 3);
    if (k >= b) return;
    const GNode nd = nodes[k];
    if (nd.n_child > 0) inner_moments(nd, k, o, lds + (threadIdx.x & ~7) * KID, threadIdx.x & 7);
}

// The inner nodes of the levels top .. 0, a level after the other, by one
// workgroup: its waves share a CU, so that a barrier lets them see the level
// before.
constexpr int TOP_THREADS = 1024;
constexpr int TOP_NODES = 256;  // per level, at most
__global__ __launch_bounds__(TOP_THREADS) void k_top_moments(const GNode *__restrict__ nodes, int top, const MomentArrays o)
{
    __shared__ double lds[TOP_THREADS * KID];
    for (int l = top; l >= 0; l--) {
        const int a = o.meta->level_start[l], b = o.meta->level_start[l + 1];
        for (int k = a + (int)(threadIdx.x >> 3); k < b; k += TOP_THREADS / 8) {
            const GNode nd = nodes[k];
            if (nd.n_child > 0) inner_moments(nd, k, o, lds + (threadIdx.x & ~7) * KID, threadIdx.x & 7);
        }
        __threadfence_block();
        __syncthreads();
    }
}

__global__ __launch_bounds__(64) void k_fill_int(int *__restrict__ p, long long n, int v)
{
    for (long long k = threadIdx.x; k < n; k += 64) p[k] = v;
}

// Exclusive sums of up to three count arrays (block b takes in[b]), n + 1
// entries each; with pad > 0 every count counts as c + c/4 + pad (a region
// for the next build's list).  *zero, if given, is set to 0.
struct Sums {
    const int *in[3];
    long long *out[3];
};
__global__ __launch_bounds__(1024) void k_sums(long long n, const Sums s, int pad, int *__restrict__ zero)
{
    if (zero && blockIdx.x == 0 && threadIdx.x == 0) *zero = 0;
    constexpr int U = 4;
    __shared__ long long ws[16];
    const int *__restrict__ in = s.in[blockIdx.x];
    long long *__restrict__ out = s.out[blockIdx.x];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    long long carry = 0;
    for (long long k0 = 0; k0 < n; k0 += 1024 * U) {
        const long long k = k0 + U * (long long)threadIdx.x;
        long long v[U], sum = 0;
        for (int u = 0; u < U; u++) {
            const int c = k + u < n ? in[k + u] : 0;
            v[u] = (pad > 0 && k + u < n) ? (long long)c + c / 4 + pad : c;
            sum += v[u];
        }
        long long inc = sum;
        for (int off = 1; off < 64; off <<= 1) {
            const long long t = __shfl_up(inc, off, 64);
            if (lane >= off) inc += t;
        }
        if (lane == 63) ws[wave] = inc;
        __syncthreads();
        long long before = carry, total = 0;
        for (int w = 0; w < 16; w++) {
            if (w < wave) before += ws[w];
            total += ws[w];
        }
        before += inc - sum;
        for (int u = 0; u < U; u++) {
            if (k + u < n) out[k + u] = before;
            before += v[u];
        }
        carry += total;
        __syncthreads();
    }
    if (threadIdx.x == 0) out[n] = carry;
}

// What the host reads back from a walk, and (behind it) the groups' records
// {first particle, size, EPJ entries, SPJ entries} for the planner.
struct WalkTotals {
    long long e, s, l;
    int over, pad;
};
__global__ __launch_bounds__(256) void k_group_info(const GNode *__restrict__ nodes, const int *__restrict__ groups,
                                                    long long ng, const int *__restrict__ cnt_e,
                                                    const int *__restrict__ cnt_s, const long long *__restrict__ off_e,
                                                    const long long *__restrict__ off_s,
                                                    const long long *__restrict__ off_l, const int *__restrict__ over,
                                                    WalkTotals *__restrict__ tot, int4 *__restrict__ info)
{
    const long long g = (long long)blockIdx.x * 256 + threadIdx.x;
    if (g == 0) *tot = WalkTotals{off_e[ng], off_s ? off_s[ng] : 0, off_l[ng], *over, 0};
    if (g >= ng) return;
    const GNode G = nodes[groups[g]];
    info[g] = make_int4((int)G.begin, (int)(G.end - G.begin), cnt_e[g], cnt_s ? cnt_s[g] : 0);
}

// resident records from the tree (the conversions of pth_resident_create)
__global__ __launch_bounds__(256) void k_res_particles(long long n, const double *__restrict__ spos,
                                                       const double *__restrict__ smass,
                                                       const double *__restrict__ srs, pth::EpiDev *__restrict__ epi,
                                                       pth::EpjDev *__restrict__ epj)
{
    const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    const double x = spos[3 * k], y = spos[3 * k + 1], z = spos[3 * k + 2];
    const float rs = (float)srs[k];
    pth::EpiDev e;
    e.x = x;
    e.y = y;
    e.z = z;
    e.rs = rs;
    e.pad = 0;
    epi[k] = e;
    pth::EpjDev j;
    j.x = x;
    j.y = y;
    j.z = z;
    j.m = (float)smass[k];
    j.rs = rs;
    epj[k] = j;
}

// The tree's SPJ lists name nodes by preorder number; for everyone else the
// entries become node numbers (level by level) on their way out.  Siblings
// then lie side by side in the superparticle table: numbered by preorder, with
// whole subtrees between them, 4,194,304 particles' staging took 4.09 ms for
// 3.63 and their force 39.7 for 37.8.  A refill copies the lists anyway (53M
// entries 78 us, by name 114); named where they are put in order, they cost
// that kernel 50 us (215 to 268) whoever reads them.  Bound by the gathers.
__global__ __launch_bounds__(256) void k_node_lists(long long n, const int *__restrict__ list,
                                                    const int *__restrict__ node_at, int *__restrict__ out)
{
    const long long k = 4 * ((long long)blockIdx.x * 256 + threadIdx.x);
    if (k + 4 <= n) {
        const int4 v = *reinterpret_cast<const int4 *>(list + k);
        *reinterpret_cast<int4 *>(out + k) = make_int4(node_at[v.x], node_at[v.y], node_at[v.z], node_at[v.w]);
    } else {
        for (long long j = k; j < n; j++) out[j] = node_at[list[j]];
    }
}

__global__ __launch_bounds__(256) void k_res_nodes(long long nn, const double *__restrict__ nmass,
                                                   const double *__restrict__ ncom, const double *__restrict__ nquad,
                                                   pth::SpjDev *__restrict__ spj)
{
    const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
    if (k >= nn) return;
    const double *q = nquad + 6 * k;
    pth::SpjDev r;
    r.x = ncom[3 * k];
    r.y = ncom[3 * k + 1];
    r.z = ncom[3 * k + 2];
    r.m = (float)nmass[k];
    r.qxx = (float)q[0];
    r.qyy = (float)q[1];
    r.qzz = (float)q[2];
    r.qxy = (float)q[3];
    r.qxz = (float)q[4];
    r.qyz = (float)q[5];
    r.pad[0] = r.pad[1] = r.pad[2] = 0.f;
    spj[k] = r;
}

// monopole superparticles: the node's mass at its centre of mass
__global__ __launch_bounds__(256) void k_res_nodes_mono(long long nn, const double *__restrict__ nmass,
                                                        const double *__restrict__ ncom,
                                                        pth::EpjDev *__restrict__ spj)
{
    const long long k = (long long)blockIdx.x * 256 + threadIdx.x;
    if (k >= nn) return;
    pth::EpjDev r;
    r.x = ncom[3 * k];
    r.y = ncom[3 * k + 1];
    r.z = ncom[3 * k + 2];
    r.m = (float)nmass[k];
    r.rs = 0.f;
    spj[k] = r;
}

struct WalkArgs {
    WalkRec rec;
    const double *ncom, *box_in, *box_out;
    const TreeMeta *meta;
    const int *groups;
    long long n_group;
    // tile walks: group g is node groups[g] with the boxes tbox[12 g ..]
    // (particle box, box widened by r_search) instead of the node's own
    const double *tbox;
    double inv_theta2;
    int theta_pos;
    int *cnt_e, *cnt_s, *cnt_l;             // EPJ entries, closed nodes, opened leaves
    // writing pass: group g's region of each raw list; what does not fit is
    // counted, not written, and sets *over
    const long long *off_l, *off_s;
    int *raw_l, *raw_s;  // preorder numbers
    int *over;
};

__device__ __forceinline__ bool overlap6(const double *a, const double *b)
{
    for (int d = 0; d < 3; d++)
        if (a[d] > b[3 + d] || b[d] > a[3 + d]) return false;
    return true;
}

// false only if boxes (lo, hi) and (l, h) do not meet; NaN bounds meet
__device__ __forceinline__ bool meet(const float (&lo)[3], const float (&hi)[3], const float4 &l, const float4 &h)
{
    return !(lo[0] > h.x || l.x > hi[0] || lo[1] > h.y || l.y > hi[1] || lo[2] > h.z || l.z > hi[2]);
}

// One workgroup of NW waves per group at a time.  The opening test
// is decided in FP32 where its bounds, widened by the margin, leave no doubt,
// and otherwise (a node at the edge of the theta sphere, or whose widened box
// meets the group's) by the host's FP64 expressions; a tile walk takes every
// node whose FP32 boxes meet (a superset: its lists are filtered exactly).
template <bool WRITE, bool TILE, int NW>
__global__ __launch_bounds__(64 * NW) void k_walk(const WalkArgs a)
{
    __shared__ int stk[WALK_STACK];
    __shared__ float lim[GT_MAX_LEVEL + 1];  // (L / theta)^2 of each level, NaN where FP32 has too few digits for it
    __shared__ int3 wave_n[NW];              // children, leaves and closed nodes of each wave
    __shared__ int wave_e[NW];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, thread = threadIdx.x;
    const double len = a.meta->len;
    const float mg = walk_margin(len, a.meta->rs_max);
    if (thread <= GT_MAX_LEVEL) {
        const double L = len / (double)(1LL << thread);
        // (near and below FP32's smallest normal number the relative bounds on
        // squares fail; against NaN the test goes to FP64)
        const double T = L * L * a.inv_theta2;
        lim[thread] = T >= 0x1p-100 ? (float)T : NAN;
    }
    const unsigned long long below = lane ? ~0ull >> (64 - lane) : 0ull;
    for (long long g = blockIdx.x; g < a.n_group; g += gridDim.x) {
        const long long gn = a.groups[g];
        const int gb = __float_as_int(a.rec.A[gn].w), ge = __float_as_int(a.rec.B[gn].w);
        const double *bin = TILE ? a.tbox + 12 * g : a.box_in + 6 * gn;
        const double *bout = TILE ? a.tbox + 12 * g + 6 : a.box_out + 6 * gn;
        // the group's boxes: the particle box as it rounds, both pushed out
        float bl[3], bh[3], il[3], ih[3], ol[3], oh[3];
        for (int d = 0; d < 3; d++) {
            const double c = a.meta->root[d] + 0.5 * len;
            bl[d] = (float)(bin[d] - c);
            bh[d] = (float)(bin[3 + d] - c);
            il[d] = bl[d] - mg;
            ih[d] = bh[d] + mg;
            ol[d] = (float)(fmin(bout[d], bin[d]) - c) - mg;
            oh[d] = (float)(fmax(bout[3 + d], bin[3 + d]) - c) + mg;
        }
        int my_e = 0, nl = 0, ns = 0;
        int *ol_raw = nullptr, *os_raw = nullptr;
        long long cap_l = 0, cap_s = 0;
        if (WRITE) {
            ol_raw = a.raw_l + a.off_l[g];
            cap_l = a.off_l[g + 1] - a.off_l[g];
            if (!TILE) {
                os_raw = a.raw_s + a.off_s[g];
                cap_s = a.off_s[g + 1] - a.off_s[g];
            }
        }
        __syncthreads();
        if (thread == 0) stk[0] = 0;
        int size = 1;
        __syncthreads();
        while (size > 0) {
            // pop k nodes (at most 8 pushed per pop): while k > 1 the stack
            // stays below WALK_STACK - 160; past that, nodes are popped one at
            // a time and a descent adds at most 7 entries per level (21
            // levels, 147 < 160), so the stack never overflows
            int k = (WALK_STACK - 160 - size) / 8;
            k = max(1, min(64 * NW, min(k, size)));
            const bool act = thread < k;
            int c = 0;
            if (act) c = stk[size - 1 - thread];
            if (NW == 1) __syncthreads();
            bool open = false;
            int begin = 0, end = 0, kids = 0;
            int2 F = make_int2(-1, 0);
            if (act) {
                const float4 A = a.rec.A[c], B = a.rec.B[c], C = a.rec.C[c];
                F = a.rec.F[c];
                begin = __float_as_int(A.w);
                end = __float_as_int(B.w);
                const int lv = __float_as_int(C.w);
                kids = lv & 255;
                if ((begin <= gb && ge <= end) || !a.theta_pos) open = true;
                else if (TILE) {
                    const float4 D = a.rec.D[c], E = a.rec.E[c];
                    open = meet(ol, oh, D, E) || meet(il, ih, B, C);
                } else {
                    const float p[3] = {A.x, A.y, A.z};
                    float far = 0.f, near = 0.f;  // bounds of the squared distance
                    for (int d = 0; d < 3; d++) {
                        const float e = fmaxf(fmaxf(bl[d] - p[d], p[d] - bh[d]), 0.f);
                        const float ep = e + mg, em = fmaxf(e - mg, 0.f);
                        far = __builtin_fmaf(ep, ep, far);
                        near = __builtin_fmaf(em, em, near);
                    }
                    const float T = lim[lv >> 8];
                    if (far * 1.00001f < T * 0.99999f) open = true;
                    else if (!(near * 0.99999f > T * 1.00001f) || meet(ol, oh, B, C)) {
                        const double L = len / (double)(1LL << (lv >> 8));
                        double s = 0;
                        for (int d = 0; d < 3; d++) {
                            const double q = a.ncom[3 * (long long)c + d];
                            double e = 0;
                            if (q < bin[d]) e = bin[d] - q;
                            else if (q > bin[3 + d]) e = q - bin[3 + d];
                            s += e * e;
                        }
                        open = s < L * L * a.inv_theta2 || overlap6(bout, a.box_in + 6 * (long long)c) ||
                               overlap6(bin, a.box_out + 6 * (long long)c);
                    }
                }
            }
            const bool leaf = open && kids == 0, closed = act && !open;
            const int mc = (open && !leaf) ? kids : 0;
            const unsigned long long ml = __ballot(leaf), ms = TILE ? 0ull : __ballot(closed);
            // exclusive sum of the child counts (0 .. 8) from their bits
            int pc = 0, tc = 0;
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const unsigned long long m = __ballot((mc >> b) & 1);
                pc += __popcll(m & below) << b;
                tc += __popcll(m) << b;
            }
            if (leaf) my_e += end - begin;
            int3 tot = make_int3(tc, __popcll(ml), __popcll(ms)), off = make_int3(0, 0, 0);
            if (NW > 1) {
                if (lane == 0) wave_n[wave] = tot;
                __syncthreads();
                tot = make_int3(0, 0, 0);
#pragma unroll
                for (int w = 0; w < NW; w++) {
                    const int3 n = wave_n[w];
                    if (w == wave) off = tot;
                    tot = make_int3(tot.x + n.x, tot.y + n.y, tot.z + n.z);
                }
            }
            if (WRITE) {
                const int pl = nl + off.y + __popcll(ml & below), ps = ns + off.z + __popcll(ms & below);
                if (leaf && pl < cap_l) ol_raw[pl] = F.y;
                if (!TILE && closed && ps < cap_s) os_raw[ps] = F.y;
            }
            nl += tot.y;
            ns += tot.z;
            size -= k;
            for (int t = 0; t < mc; t++) stk[size + off.x + pc + t] = F.x + (mc - 1 - t);
            size += tot.x;
            __syncthreads();
        }
        for (int off = 32; off > 0; off >>= 1) my_e += __shfl_xor(my_e, off, 64);
        if (NW > 1) {
            if (lane == 0) wave_e[wave] = my_e;
            __syncthreads();
            my_e = 0;
            for (int w = 0; w < NW; w++) my_e += wave_e[w];
        }
        if (thread == 0) {
            a.cnt_e[g] = my_e;
            a.cnt_l[g] = nl;
            if (!TILE) a.cnt_s[g] = ns;
            if (WRITE && (nl > cap_l || ns > cap_s)) atomicOr(a.over, 1);
        }
    }
}

// The final lists from the raw ones, one workgroup per group or tile.  The raw
// entries are preorder numbers, and a depth-first walk's order is their
// ascending order, so a list is put in order without moving it: each entry
// sets a bit of a map of the tree's nodes in LDS (a window of it at a time,
// for trees of more nodes), and the set bits are read off in order.  A
// segmented radix sort moved every particle and node entry through memory
// three times (1,048,576 particles, 34M + 53M entries: 1.9 ms with its keys,
// and 0.17 ms to move the lists to their places; 0.21 ms here.  4,194,304
// particles: 7.9 and 2.0 ms).
struct OrderArgs {
    const int2 *range;  // first particle and size of each node, in preorder
    int n_words;        // of the node map
    int window;         // words of it held in LDS
    long long n_group;
    const int *cnt_l;
    const long long *roff_l, *roff_s, *off_e, *off_s;
    const int *raw_l, *raw_s;
    int *sort_l;  // room for long ordered leaf lists, in raw_l's layout
    int *id_epj, *id_spj;
};

// Inclusive wave sum in the vector ALU's own lane shifts (DPP): six
// dependent adds, where six LDS permutes would each wait for LDS.
__device__ __forceinline__ int wave_inclusive(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1, 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2, 3
    return v;
}

// Sets the bits of the m entries of raw that fall into words [w0, w0 + nw) of
// the map and returns whether this thread set any.  Neighbouring entries are siblings, i.e.
// bits of one word: a thread takes a run of entries (in aligned quads, which
// may hold up to three words before and after the region's entries) and
// joins the bits of a word before its LDS atomic, and the threads of a wave
// are on different words (lane-strided entries met on a few words and waited
// for each other).
template <int WG>
__device__ __forceinline__ int set_bits(const int *__restrict__ raw, int m, int w0, int nw, unsigned *map)
{
    const int lead = (int)((reinterpret_cast<size_t>(raw) >> 2) & 3);
    const int4 *quads = reinterpret_cast<const int4 *>(raw - lead);
    const int nq = (m + lead + 3) >> 2;
    const int q0 = (int)((long long)nq * threadIdx.x / WG), q1 = (int)((long long)nq * (threadIdx.x + 1) / WG);
    int word = -1, any = 0;
    unsigned bits = 0;
    auto flush = [&]() {
        if (word < 0 || word >= nw) return;
        atomicOr(&map[word], bits);
        any = 1;
    };
    for (int q = q0; q < q1; q++) {
        const int4 v4 = quads[q];
        const int v[4] = {v4.x, v4.y, v4.z, v4.w};
        const int k = 4 * q - lead;  // entry of v[0]
#pragma unroll
        for (int u = 0; u < 4; u++) {
            if (k + u < 0 || k + u >= m) continue;
            const int w = (v[u] >> 5) - w0;
            if (w != word) {
                flush();
                word = w;
                bits = 0;
            }
            bits |= 1u << (v[u] & 31);
        }
    }
    flush();
    return any;
}

// The m entries of raw to out in ascending order: an entry's place is the
// number of bits set below its own, i.e. the sum of its chunk of 64 words
// (sums), of its word in the chunk (below) and the bits below in the word.
// So every entry is placed by itself; reading the bits off word by word left
// most lanes idle, the near cells' bits being packed into a few words.  All
// threads of the block call it; map, below and sums hold `window` words.
template <int WG>
__device__ void order_by_map(const int *__restrict__ raw, int m, int n_words, int window, unsigned *map, int *wtot,
                             int *out)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    constexpr int NW = WG / 64, U = 4;
    int *sums = reinterpret_cast<int *>(map + window);
    unsigned short *below = reinterpret_cast<unsigned short *>(sums + (window + 63) / 64);
    int done = 0;
    for (int w0 = 0; w0 < n_words; w0 += window) {
        const int nw = min(window, n_words - w0), nc = (nw + 63) >> 6;
        for (int k = tid; k < nw; k += WG) map[k] = 0u;
        __syncthreads();
        // (a leaf list often leaves a window empty)
        if (!__syncthreads_or(set_bits<WG>(raw, m, w0, nw, map))) continue;
        for (int c = wave; c < nc; c += NW) {
            const int k = c * 64 + lane;
            const int own = k < nw ? __popc(map[k]) : 0, inc = wave_inclusive(own);
            if (k < nw) below[k] = (unsigned short)(inc - own);
            if (lane == 63) sums[c] = inc;
        }
        __syncthreads();
        if (wave == 0) {
            int carry = 0;
            for (int c0 = 0; c0 < nc; c0 += 64) {
                const int own = c0 + lane < nc ? sums[c0 + lane] : 0, inc = wave_inclusive(own);
                if (c0 + lane < nc) sums[c0 + lane] = carry + inc - own;
                carry += __builtin_amdgcn_readlane(inc, 63);
            }
            if (lane == 0) *wtot = carry;
        }
        __syncthreads();
        for (int k0 = tid; k0 < m; k0 += WG * U) {
            int v[U];
#pragma unroll
            for (int u = 0; u < U; u++) v[u] = k0 + u * WG < m ? raw[k0 + u * WG] : -1;
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int q = (v[u] >> 5) - w0;
                if (v[u] < 0 || q < 0 || q >= nw) continue;
                out[done + sums[q >> 6] + below[q] + __popc(map[q] & ((1u << (v[u] & 31)) - 1u))] = v[u];
            }
        }
        done += *wtot;
        __syncthreads();
    }
}
// LDS bytes of a map of `window` words (even) with its sums.
constexpr size_t map_bytes(int window) { return 6 * (size_t)window + 4 * (size_t)((window + 63) / 64); }

// Writes the particles of m leaves (preorder numbers, in order) to out.  All
// threads of the block call it; eight lanes write a leaf.
template <int WG, int RMAX>
__device__ void expand_leaves(const int *leaves, int m, const int2 *__restrict__ range, int *l_begin, int *l_off,
                              int *wsum, int *__restrict__ out)
{
    static_assert(RMAX % WG == 0, "leaves per pass");
    constexpr int PER = RMAX / WG, NW = WG / 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int done = 0;  // entries written
    for (int l0 = 0; l0 < m; l0 += RMAX) {
        const int nl = min(RMAX, m - l0);
        int v[PER], sum = 0;
        for (int u = 0; u < PER; u++) {
            const int k = tid * PER + u;
            v[u] = 0;
            if (k < nl) {
                const int2 q = range[leaves[l0 + k]];
                l_begin[k] = q.x;
                v[u] = q.y;
            }
            sum += v[u];
        }
        const int inc = wave_inclusive(sum);
        if (lane == 63) wsum[wave] = inc;
        __syncthreads();
        int before = inc - sum, total = 0;
        for (int w = 0; w < NW; w++) {
            if (w < wave) before += wsum[w];
            total += wsum[w];
        }
        for (int u = 0; u < PER; u++) {
            l_off[tid * PER + u] = before;
            before += v[u];
        }
        if (tid == WG - 1) l_off[RMAX] = before;
        __syncthreads();
        for (int k = tid >> 3; k < nl; k += WG / 8) {
            const int o = l_off[k], n = l_off[k + 1] - o, p = l_begin[k];
            for (int j = tid & 7; j < n; j += 8) out[done + o + j] = p + j;
        }
        done += total;
        __syncthreads();
    }
}

// Groups: SORT for canonical order, else batch order.
template <int WG, int RMAX, bool SORT> __global__ __launch_bounds__(WG) void k_order(const OrderArgs a)
{
    extern __shared__ unsigned map[];
    __shared__ int l_pre[SORT ? RMAX : 1], l_begin[RMAX], l_off[RMAX + 1], wsum[WG / 64];
    for (long long g = blockIdx.x; g < a.n_group; g += gridDim.x) {
        const int ms = (int)(a.off_s[g + 1] - a.off_s[g]), ml = a.cnt_l[g];
        const int *raw_s = a.raw_s + a.roff_s[g], *leaves = a.raw_l + a.roff_l[g];
        int *out_s = a.id_spj + a.off_s[g];
        if constexpr (SORT) {
            // ordered leaves: in LDS when they fit
            int *sorted = ml <= RMAX ? l_pre : a.sort_l + a.roff_l[g];
            order_by_map<WG>(raw_s, ms, a.n_words, a.window, map, wsum, out_s);
            order_by_map<WG>(leaves, ml, a.n_words, a.window, map, wsum, sorted);
            leaves = sorted;
            __threadfence_block();
            __syncthreads();
        } else {
            for (int k = threadIdx.x; k < ms; k += WG) out_s[k] = raw_s[k];
        }
        expand_leaves<WG, RMAX>(leaves, ml, a.range, l_begin, l_off, wsum, a.id_epj + a.off_e[g]);
    }
}

// Neighbour-search tiles (leaf lists only, a dozen entries each), one wave
// per tile: an entry's rank is the number of smaller ones; lists of more than
// RMAX entries (degenerate trees) go through the map.
template <int RMAX> __global__ __launch_bounds__(64) void k_order_tiles(const OrderArgs a)
{
    extern __shared__ unsigned map[];
    __shared__ __attribute__((aligned(16))) int l_raw[RMAX];
    __shared__ int l_pre[RMAX], l_begin[RMAX], l_off[RMAX + 1], wsum[1];
    static_assert(RMAX % 64 == 0, "leaves per pass");
    const int lane = threadIdx.x;
    for (long long g = blockIdx.x; g < a.n_group; g += gridDim.x) {
        const int m = a.cnt_l[g];
        const int *raw = a.raw_l + a.roff_l[g];
        int *sorted = l_pre;
        if (m <= RMAX) {
            const int m4 = (m + 3) & ~3;
            for (int k = lane; k < m4; k += 64) l_raw[k] = k < m ? raw[k] : INT_MAX;
            __syncthreads();
            for (int k = lane; k < m; k += 64) {
                const int v = l_raw[k];
                int r = 0;
                for (int j = 0; j < m4; j += 4) {
                    const int4 q = *reinterpret_cast<const int4 *>(l_raw + j);
                    r += (q.x < v) + (q.y < v) + (q.z < v) + (q.w < v);
                }
                l_pre[r] = v;
            }
        } else {
            sorted = a.sort_l + a.roff_l[g];
            order_by_map<64>(raw, m, a.n_words, a.window, map, wsum, sorted);
            __threadfence_block();
        }
        __syncthreads();
        expand_leaves<64, RMAX>(sorted, m, a.range, l_begin, l_off, wsum, a.id_epj + a.off_e[g]);
    }
}

// Regions of a one-pass neighbour filter: the last search's count of
// particle i + 1/4 + 4 (cap[n] = 0, so the scan's last entry is the total).
__global__ __launch_bounds__(256) void k_ngb_caps(long long n, const int *__restrict__ cnt, int *__restrict__ cap)
{
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) {
        const int c = max(cnt[i], 0);
        cap[i] = c + c / 4 + 4;
    } else if (i == n) {
        cap[n] = 0;
    }
}

// Particle i's neighbours, written by a padded filter pass at poff[i], moved
// to off[i] (checked on the host to fit the region).
__global__ __launch_bounds__(256) void k_ngb_compact(long long n, const long long *__restrict__ poff,
                                                     const long long *__restrict__ off, const int *__restrict__ src,
                                                     int *__restrict__ dst)
{
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const long long m = off[i + 1] - off[i];
    const int *s = src + poff[i];
    int *d = dst + off[i];
    for (long long k = 0; k < m; k++) d[k] = s[k];
}

// Boxes of the neighbour-search tiles (the largest cells with at most 64
// particles): the cell's particle box and its box widened by r_search,
// pushed outwards by (|v| + rs_max) 2^-40, far above the rounding of any
// coordinate, difference or box bound involved, so a tile walk with these
// boxes opens every leaf holding a neighbour of a tile particle under the
// exact FP64 test (the walk's lists are a superset; k_ngb filters exactly).
__global__ __launch_bounds__(256) void k_tile_boxes(const int *__restrict__ tiles, long long nt,
                                                    const double *__restrict__ box_in,
                                                    const double *__restrict__ box_out, double rs_max,
                                                    double *__restrict__ tbox)
{
    const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
    if (t >= nt) return;
    const long long c = tiles[t];
    const double m = 0x1p-40;
    for (int d = 0; d < 3; d++) {
        const double lo = box_in[6 * c + d], hi = box_in[6 * c + 3 + d];
        const double lo2 = box_out[6 * c + d], hi2 = box_out[6 * c + 3 + d];
        tbox[12 * t + d] = lo - (fabs(lo) + rs_max) * m;
        tbox[12 * t + 3 + d] = hi + (fabs(hi) + rs_max) * m;
        tbox[12 * t + 6 + d] = lo2 - (fabs(lo2) + rs_max) * m;
        tbox[12 * t + 9 + d] = hi2 + (fabs(hi2) + rs_max) * m;
    }
}

// Neighbour search (src/soft_force.hpp:11-34, SearchNeighborEpEpNoSimd) on
// candidate lists that hold every symmetric-search neighbour (the tile walks
// of pth_gtree_neighbors): for every i of a tile the
// list entries j with |x_i - x_j|^2 < max(rs_i, rs_j)^2 in FP64, self
// included.  One wave per tile at a time, lane l holds i = l (a tile of more
// than 64 particles is a leaf of as many, taken 64 at a time); 64 candidates
// at a time are loaded, one per lane, and those that come within R =
// max(rs of the tile, rs_j) of the tile's box go to LDS, in list order, to be
// read as broadcasts by all lanes.  The gap g between box and j (per axis,
// >= 0) bounds every pair's |dx| from below; g2 = gx^2 + gy^2 + gz^2 and the
// pair's r2 are each within 3 ulp of their exact values however they are
// contracted, so g2 > R^2 (1 + 2^-48) implies r2 >= rs^2 as computed below
// and the skip never drops a neighbour.
// What bounds it: the latency of the candidates' gathers and the pair loop.
// A wave that held eight sub-tiles of 64 i (nearly all tiles have one), took
// the boxes of all eight and of every 64 candidates and then tested all of
// the 64 was 655 us at 1,048,576 particles; this 215.
// Counting pass: cnt[input index of i]; writing pass: input indices of the
// neighbours at ngb[off[input index of i]..], in list order.
struct NgbArgs {
    const double *spos, *srs;
    const long long *order;
    const int4 *info;  // per group: first particle, size, n_epj, n_spj
    const long long *off_e;
    const int *id_epj;
    long long n_group;
    int *cnt;
    const long long *off;
    int *ngb;
    // padded writing pass: particle i writes into [off[i], off[i + 1]) at
    // most, stores its exact count, and sets *flag when it did not fit
    int padded;
    int *flag;
};

struct NgbJ {
    double x, y, z, rs;
};

__device__ __forceinline__ double wave_min(double v)
{
    for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, 64));
    return v;
}

__device__ __forceinline__ double wave_max(double v)
{
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}

template <bool WRITE>
__global__ __launch_bounds__(64) void k_ngb(const NgbArgs a)
{
    __shared__ NgbJ sj[64];
    __shared__ int sid[64];
    const int lane = threadIdx.x;
    for (long long g = blockIdx.x; g < a.n_group; g += gridDim.x) {
        const int4 G = a.info[g];
        const long long eb = a.off_e[g], ee = a.off_e[g + 1];
        for (int s0 = 0; s0 < G.y; s0 += 64) {
            const bool act = s0 + lane < G.y;
            double xi = 0, yi = 0, zi = 0, ri = 0;
            long long oi = 0, w = 0;
            int c = 0, cap = INT_MAX;
            if (act) {
                const long long i = (long long)G.x + s0 + lane;
                xi = a.spos[3 * i];
                yi = a.spos[3 * i + 1];
                zi = a.spos[3 * i + 2];
                ri = a.srs[i];
                oi = a.order[i];
                if (WRITE) {
                    w = a.off[oi];
                    if (a.padded) cap = (int)(a.off[oi + 1] - w);
                }
            }
            const double lx = wave_min(act ? xi : 1e300), hx = wave_max(act ? xi : -1e300);
            const double ly = wave_min(act ? yi : 1e300), hy = wave_max(act ? yi : -1e300);
            const double lz = wave_min(act ? zi : 1e300), hz = wave_max(act ? zi : -1e300);
            const double rt = wave_max(act ? ri : 0.0);
            for (long long k0 = eb; k0 < ee; k0 += 64) {
                const long long k = k0 + lane;
                NgbJ J{0, 0, 0, 0};
                bool near = false;
                int j = 0;
                if (k < ee) {
                    j = a.id_epj[k];
                    J = NgbJ{a.spos[3 * (long long)j], a.spos[3 * (long long)j + 1], a.spos[3 * (long long)j + 2],
                             a.srs[j]};
                    const double gx = fmax(0.0, fmax(lx - J.x, J.x - hx));
                    const double gy = fmax(0.0, fmax(ly - J.y, J.y - hy));
                    const double gz = fmax(0.0, fmax(lz - J.z, J.z - hz));
                    const double R = fmax(rt, J.rs);
                    near = !(gx * gx + gy * gy + gz * gz > R * R * (1 + 0x1p-48));
                }
                const unsigned long long found = __ballot(near);
                if (near) {
                    const int p = __popcll(found & ((1ull << lane) - 1));
                    sj[p] = J;
                    if (WRITE) sid[p] = (int)a.order[j];
                }
                __syncthreads();
                const int m = __popcll(found);
                if (act)
                    for (int q = 0; q < m; q++) {
                        const NgbJ Q = sj[q];
                        const double dx = xi - Q.x, dy = yi - Q.y, dz = zi - Q.z;
                        const double r2 = dx * dx + dy * dy + dz * dz;
                        const double rs = (ri < Q.rs) ? Q.rs : ri;
                        if (r2 < rs * rs) {
                            if (WRITE && c < cap) a.ngb[w + c] = sid[q];
                            c++;
                        }
                    }
                __syncthreads();
            }
            if (!WRITE || a.padded) {
                if (act) a.cnt[oi] = c;
                if (WRITE && c > cap) atomicOr(a.flag, 1);
            }
        }
    }
}

}  // namespace

// ---------------------------------------------------------------------------
// host side

// The lists of a walk: counts per group (EPJ entries, closed nodes, opened
// leaves), offsets, the raw lists and their regions, the read-back.  Kept
// from walk to walk: the counts size the next one's regions.
struct WalkLists {
    DevBuf cnt, off, reg, raw_l, raw_s, sort_l, back;
    PinBuf host;  // WalkTotals, then one int4 per group
    long long n = -1, tot_l = 0, tot_s = 0;
    int passes = 0;
    const int4 *info() const { return reinterpret_cast<const int4 *>(host.as<WalkTotals>() + 1); }
    void release()
    {
        for (DevBuf *b : {&cnt, &off, &reg, &raw_l, &raw_s, &sort_l, &back}) b->release();
        host.release();
    }
};

struct pth_gtree {
    pth_ctx *ctx = nullptr;
    long long n = 0, n_node = 0, n_group = 0, n_tile = 0, n_le = 0, n_ls = 0;
    DevBuf order, key, skey, sidx, sidx2, spos, smass, srs, nodes, nmass, ncom, nquad, box_in, box_out, rec, groups,
        id_epj, id_spj, tmp;
    WalkLists walk, tile_walk;  // the group walk, the neighbour search's
    WalkRec walk_rec() const
    {
        float4 *p = rec.as<float4>();
        return WalkRec{p, p + n_node, p + 2 * n_node, p + 3 * n_node, p + 4 * n_node,
                       reinterpret_cast<int2 *>(p + 5 * n_node)};
    }
    // build-time scratch, released when the build ends (or by pth_gtree_free)
    DevBuf dpos, dmass, drs, part, cnt, off, starts;
    // neighbour lists (pth_gtree_neighbors): count per input index, offsets,
    // entries; tiles, tile boxes, candidate lists
    DevBuf ngb_cnt, ngb_off, ngb, tiles, tbox, tl;
    int walk_passes = 0;  // of the last build: 1 (one padded pass) or 2 (count, then write)
    DevBuf meta;             // TreeMeta of the last build
    DevBuf pre, node_at;     // preorder number of each node, and the inverse
    DevBuf range;            // the nodes' particle ranges, in preorder
    void *pinned = nullptr;  // pinned host copy of meta
    hipEvent_t ev_meta = nullptr;  // that copy
    int tile_passes = 0;  // of the last search's tile walk
    // one-pass neighbour filters: regions from the last completed search's
    // per-particle counts (ngb_cnt), valid while ngb_prev_ok
    DevBuf ngb_cap, ngb_poff, ngb_pad, ngb_flag;
    bool ngb_prev_ok = false;
    long long ngb_prev_n = -1, ngb_prev_total = 0;
    int ngb_passes = 0;  // of the last search's filter
    long long n_ngb = -1;  // total entries, -1 before the first search
    long long n_cand = 0;  // candidate pairs of the last search
    float ms_ngb = 0.f;
    void release_scratch()
    {
        DevBuf *s[] = {&dpos, &dmass, &drs, &part, &cnt, &off, &starts};
        for (DevBuf *b : s) b->release();
    }
    std::vector<int4> groups_h;  // per group: first particle, size, n_epj, n_spj
    // the plan of a resident evaluation of the last build's lists, made on
    // the host while the device writes and orders them, and the parameters
    // it was made for
    mutable Plan pre_plan;  // taken over (swapped out) by a refill
    PlanKey pre_key;
    bool pre_ok = false;
    mutable bool pre_valid = false;
    int n_leaf_limit = 20, n_group_limit = 512;
    double theta = 0.3;
    double rs_max = 0.0, root_len = 1.0;  // largest r_search, root cell side
    bool canonical = false;
    bool built = false;
    float ms_build = 0.f, ms_walk = 0.f, ms_order = 0.f;
};

namespace {

#define GT_CHK(call, what)                               \
    do {                                                 \
        hipError_t e_ = (call);                          \
        if (e_ != hipSuccess) return t->ctx->hip_fail(e_, what); \
    } while (0)

constexpr int TILE_LIMIT = 64;  // particles of a neighbour-search tile

inline unsigned blocks(long long n) { return (unsigned)((n + 255) / 256); }

hipError_t ensure_pinned(pth_gtree *t)
{
    if (t->pinned) return hipSuccess;
    const hipError_t e = hipHostMalloc(&t->pinned, sizeof(TreeMeta), hipHostMallocDefault);
    if (e != hipSuccess) t->pinned = nullptr;
    return e ? e : hipEventCreateWithFlags(&t->ev_meta, hipEventDisableTiming);
}

// temp storage for a hipcub call, grown on demand
hipError_t cub_temp(pth_gtree *t, size_t bytes) { return t->tmp.ensure(std::max<size_t>(bytes, 256)); }

}  // namespace

namespace {

// The tree's part of a walk's arguments.
WalkArgs walk_args(pth_gtree *t)
{
    WalkArgs wa{};
    wa.rec = t->walk_rec();
    wa.ncom = t->ncom.as<double>();
    wa.box_in = t->box_in.as<double>();
    wa.box_out = t->box_out.as<double>();
    wa.meta = t->meta.as<TreeMeta>();
    return wa;
}

// The walk of wa's groups: while there are few of them, four waves each (16,384
// particles, 219 groups: 45 us with one wave, whose serial chain of pops
// leaves the chip idle, 29 with four, 29 with eight).
template <bool WRITE, bool TILE> void launch_walk(const WalkArgs &wa, hipStream_t st)
{
    const unsigned wg = (unsigned)std::min<long long>(wa.n_group, 65536);
    if (wa.n_group <= WALK_WIDE)
        hipLaunchKernelGGL((k_walk<WRITE, TILE, 4>), dim3(wg), dim3(256), 0, st, wa);
    else hipLaunchKernelGGL((k_walk<WRITE, TILE, 1>), dim3(wg), dim3(64), 0, st, wa);
}

// Walks the groups of wa into W's raw lists and reads the counts back: one
// writing pass into regions of the last walk's lengths when that was a walk
// of as many groups (and again_ok says its counts still stand), else a
// counting pass; the writing pass that either may still need is walk_finish's.
template <bool TILE> int walk_run(pth_gtree *t, WalkArgs &wa, WalkLists &W, bool again_ok, long long ng)
{
    pth_ctx *ctx = t->ctx;
    hipStream_t st = ctx->stream;
    hipError_t e;
    const bool again = ng > 0 && again_ok && W.n == ng;
    W.n = -1;  // the counts are about to be rewritten
    W.passes = 0;
    const size_t nc = (size_t)ng + 1, bytes = sizeof(WalkTotals) + sizeof(int4) * (size_t)ng;
    if ((e = W.cnt.ensure(sizeof(int) * (3 * nc + 1))) || (e = W.off.ensure(8 * 3 * nc)) ||
        (e = W.reg.ensure(8 * 2 * nc)) || (e = W.back.ensure(bytes)) || (e = W.host.ensure(bytes)))
        return ctx->hip_fail(e, "walk allocation");
    wa.cnt_e = W.cnt.as<int>();
    wa.cnt_s = wa.cnt_e + nc;
    wa.cnt_l = wa.cnt_s + nc;
    wa.over = wa.cnt_l + nc;
    long long *off_e = W.off.as<long long>(), *off_s = off_e + nc, *off_l = off_s + nc;
    long long *reg_l = W.reg.as<long long>(), *reg_s = reg_l + nc;
    if (again) {
        // (a tile has a dozen leaves: 64 spare ones each would be mostly holes)
        const int pad = TILE ? 8 : 64;
        // (the regions' sum: each at most its length + 1/4 + pad)
        auto room = [&](long long n) { return 4 * (size_t)(n + n / 4 + pad * ng + 64); };
        if ((e = W.raw_l.ensure(room(W.tot_l))) || (!TILE && (e = W.raw_s.ensure(room(W.tot_s)))))
            return ctx->hip_fail(e, "raw list allocation");
        const Sums s{{wa.cnt_l, wa.cnt_s, nullptr}, {reg_l, reg_s, nullptr}};
        hipLaunchKernelGGL(k_sums, dim3(TILE ? 1 : 2), dim3(1024), 0, st, ng, s, pad, wa.over);
        wa.off_l = reg_l;
        wa.off_s = reg_s;
        wa.raw_l = W.raw_l.as<int>();
        wa.raw_s = W.raw_s.as<int>();
        launch_walk<true, TILE>(wa, st);
    } else if (ng > 0) {
        launch_walk<false, TILE>(wa, st);
    }
    const Sums s{{wa.cnt_e, wa.cnt_l, wa.cnt_s}, {off_e, off_l, off_s}};
    hipLaunchKernelGGL(k_sums, dim3(TILE ? 2 : 3), dim3(1024), 0, st, ng, s, 0, again ? nullptr : wa.over);
    hipLaunchKernelGGL(k_group_info, dim3(std::max(1u, blocks(ng))), dim3(256), 0, st, t->nodes.as<GNode>(), wa.groups,
                       ng, wa.cnt_e, TILE ? nullptr : wa.cnt_s, off_e, TILE ? nullptr : off_s, off_l, wa.over,
                       W.back.as<WalkTotals>(), reinterpret_cast<int4 *>(W.back.as<WalkTotals>() + 1));
    // (a tile walk's records stay on the device)
    if ((e = hipGetLastError()) ||
        (e = hipMemcpyAsync(W.host.p, W.back.p, TILE ? sizeof(WalkTotals) : bytes, hipMemcpyDeviceToHost, st)) ||
        (e = hipStreamSynchronize(st)))
        return ctx->hip_fail(e, "tree walk");
    const WalkTotals &tot = *W.host.as<WalkTotals>();
    W.tot_l = tot.l;
    W.tot_s = tot.s;
    W.n = ng;
    W.passes = again && !tot.over ? 1 : 2;
    return PTH_OK;
}

// The writing pass, if one is due, and the final lists.
template <bool TILE> int walk_finish(pth_gtree *t, WalkArgs &wa, WalkLists &W, bool canonical, int *id_epj, int *id_spj)
{
    pth_ctx *ctx = t->ctx;
    hipStream_t st = ctx->stream;
    hipError_t e;
    const long long ng = wa.n_group;
    if (ng <= 0) return PTH_OK;
    const size_t nc = (size_t)ng + 1;
    long long *off_e = W.off.as<long long>(), *off_s = off_e + nc, *off_l = off_s + nc;
    if (W.passes == 2) {
        if ((e = W.raw_l.ensure(4 * (size_t)(W.tot_l + 8))) ||
            (!TILE && (e = W.raw_s.ensure(4 * (size_t)(W.tot_s + 8)))))
            return ctx->hip_fail(e, "raw list allocation");
        wa.off_l = off_l;
        wa.off_s = off_s;
        wa.raw_l = W.raw_l.as<int>();
        wa.raw_s = W.raw_s.as<int>();
        launch_walk<true, TILE>(wa, st);
    }
    if ((e = W.sort_l.ensure(W.raw_l.cap))) return ctx->hip_fail(e, "leaf list allocation");
    OrderArgs o{};
    o.range = t->range.as<int2>();
    o.n_words = (int)((t->n_node + 31) / 32);
    o.n_group = ng;
    o.cnt_l = wa.cnt_l;
    o.roff_l = wa.off_l;
    o.roff_s = wa.off_s;
    o.off_e = off_e;
    o.off_s = off_s;
    o.raw_l = wa.raw_l;
    o.raw_s = wa.raw_s;
    o.sort_l = W.sort_l.as<int>();
    o.id_epj = id_epj;
    o.id_spj = id_spj;
    const dim3 grid((unsigned)std::min<long long>(ng, 65536));
    // map windows: 36 KB for a group (three workgroups of 512 per CU; trees of
    // up to 196,608 nodes in one window), 3 KB for a tile
    if constexpr (TILE) {
        o.window = std::min(o.n_words, 512);
        hipLaunchKernelGGL(k_order_tiles<256>, grid, dim3(64), map_bytes(o.window), st, o);
    } else {
        o.window = std::min(o.n_words, 6144);
        if (canonical)
            hipLaunchKernelGGL((k_order<512, 1024, true>), grid, dim3(512), map_bytes(o.window), st, o);
        else hipLaunchKernelGGL((k_order<512, 1024, false>), grid, dim3(512), 0, st, o);
    }
    if ((e = hipGetLastError())) return ctx->hip_fail(e, "list kernels");
    return PTH_OK;
}

// Builds (or rebuilds, reusing t's device memory) the tree of n particles.
// pos / mass / rs are host arrays, or device arrays when on_device.
int gtree_run(pth_gtree *t, long long n, const double *pos, const double *mass, const double *r_search,
              bool on_device)
{
    pth_ctx *ctx = t->ctx;
    const int n_leaf_limit = t->n_leaf_limit, n_group_limit = t->n_group_limit;
    const double theta = t->theta;
    const bool was_built = t->built;  // groups_h then holds the last build's list lengths
    t->built = false;
    t->pre_valid = false;
    t->n_ngb = -1;
    t->n = n;
    t->n_node = t->n_group = t->n_le = t->n_ls = 0;
    const auto t0 = std::chrono::steady_clock::now();
    hipStream_t st = ctx->stream;
    hipError_t e;
    // particles in (unsorted), then sorted copies
    const double *dpos = pos, *dmass = mass, *drs = r_search;
    if (on_device) {
        if (!device_range(pos, 24 * (size_t)n) || !device_range(mass, 8 * (size_t)n) ||
            (r_search && !device_range(r_search, 8 * (size_t)n)))
            return ctx->fail(PTH_ERR_ARG, "pth_gtree: the particle arrays are not device allocations of n entries");
    } else {
        auto up = [&](DevBuf &b, const double *h, size_t cnt) -> hipError_t {
            hipError_t r = b.ensure(sizeof(double) * cnt);
            if (r == hipSuccess) r = hipMemcpyAsync(b.p, h, sizeof(double) * cnt, hipMemcpyHostToDevice, st);
            return r;
        };
        if ((e = up(t->dpos, pos, 3 * (size_t)n)) || (e = up(t->dmass, mass, (size_t)n)) ||
            (r_search && (e = up(t->drs, r_search, (size_t)n))))
            return ctx->hip_fail(e, "pth_gtree: upload");
        dpos = t->dpos.as<double>();
        dmass = t->dmass.as<double>();
        drs = r_search ? t->drs.as<double>() : nullptr;
    }
    // 1. bounding cube
    const int nb = (int)std::min<long long>(1024, (n + 255) / 256);
    DevBuf &part = t->part;
    if ((e = ensure_pinned(t)) || (e = part.ensure(sizeof(double) * 8 * nb)) || (e = t->meta.ensure(sizeof(TreeMeta))))
        return ctx->hip_fail(e, "bbox");
    TreeMeta *meta = t->meta.as<TreeMeta>();
    hipLaunchKernelGGL(k_bbox, dim3(nb), dim3(256), 0, st, dpos, drs, n, part.as<double>());
    hipLaunchKernelGGL(k_root, dim3(1), dim3(1024), 0, st, part.as<double>(), nb, meta);
    // 2. keys, stable sort of (key, index), sorted particles
    if ((e = t->key.ensure(8 * (size_t)n)) || (e = t->skey.ensure(8 * (size_t)n)) ||
        (e = t->sidx.ensure(4 * (size_t)n)) || (e = t->sidx2.ensure(4 * (size_t)n)) ||
        (e = t->order.ensure(8 * (size_t)n)))
        return ctx->hip_fail(e, "key allocation");
    hipLaunchKernelGGL(k_keys, dim3(blocks(n)), dim3(256), 0, st, dpos, n, meta, t->key.as<unsigned long long>(),
                       t->sidx.as<int>());
    size_t tb = 0;
    if ((e = hipcub::DeviceRadixSort::SortPairs(nullptr, tb, t->key.as<unsigned long long>(),
                                                t->skey.as<unsigned long long>(), t->sidx.as<int>(),
                                                t->sidx2.as<int>(), n, 0, 3 * GT_MAX_LEVEL, st)) ||
        (e = cub_temp(t, tb)) ||
        (e = hipcub::DeviceRadixSort::SortPairs(t->tmp.p, tb, t->key.as<unsigned long long>(),
                                                t->skey.as<unsigned long long>(), t->sidx.as<int>(),
                                                t->sidx2.as<int>(), n, 0, 3 * GT_MAX_LEVEL, st)))
        return ctx->hip_fail(e, "key sort");
    if ((e = t->spos.ensure(24 * (size_t)n)) || (e = t->smass.ensure(8 * (size_t)n)) ||
        (e = t->srs.ensure(8 * (size_t)n)))
        return ctx->hip_fail(e, "particle allocation");
    // 3. nodes, groups and tiles: counts, one scan, one wait for the sizes
    const int nblk = (int)blocks(n);
    const unsigned long long *skey = t->skey.as<unsigned long long>();
    const int n_cnt = N_ROWS * nblk + 1;
    if ((e = t->cnt.ensure(sizeof(int) * (size_t)n_cnt)) || (e = t->off.ensure(sizeof(int) * (size_t)n_cnt)) ||
        (e = t->starts.ensure(4 * (size_t)n)))
        return ctx->hip_fail(e, "node counts");
    hipLaunchKernelGGL(k_starts, dim3(nblk), dim3(256), 0, st, skey, n, n_leaf_limit, n_group_limit, TILE_LIMIT, nblk,
                       t->cnt.as<int>(), t->starts.as<unsigned>());
    if ((e = hipcub::DeviceScan::ExclusiveSum(nullptr, tb, t->cnt.as<int>(), t->off.as<int>(), n_cnt, st)) ||
        (e = cub_temp(t, tb)) ||
        (e = hipcub::DeviceScan::ExclusiveSum(t->tmp.p, tb, t->cnt.as<int>(), t->off.as<int>(), n_cnt, st)))
        return ctx->hip_fail(e, "node scan");
    hipLaunchKernelGGL(k_tree_sizes, dim3(1), dim3(64), 0, st, t->off.as<int>(), nblk, meta);
    if ((e = hipMemcpyAsync(t->pinned, meta, sizeof(TreeMeta), hipMemcpyDeviceToHost, st)) ||
        (e = hipEventRecord(t->ev_meta, st)))
        return ctx->hip_fail(e, "tree sizes");
    // (beside the wait)
    hipLaunchKernelGGL(k_gather, dim3(blocks(n)), dim3(256), 0, st, n, t->sidx2.as<int>(), t->order.as<long long>(),
                       dpos, dmass, drs, t->spos.as<double>(), t->smass.as<double>(), t->srs.as<double>());
    if ((e = hipEventSynchronize(t->ev_meta))) return ctx->hip_fail(e, "tree sizes");
    TreeMeta M;
    std::memcpy(&M, t->pinned, sizeof M);
    if (M.bad != 0.0) return ctx->fail(PTH_ERR_ARG, "pth_gtree: non-finite particle positions or r_search");
    const double len = M.len;
    t->rs_max = M.rs_max;
    t->root_len = len;
    const long long nn = M.level_start[GT_MAX_LEVEL + 1];
    t->n_node = nn;
    t->n_group = M.n_group;
    t->n_tile = M.n_tile;
    if ((e = t->nodes.ensure(sizeof(GNode) * nn)) || (e = t->pre.ensure(4 * nn)) || (e = t->node_at.ensure(4 * nn)) ||
        (e = t->range.ensure(8 * nn)) ||
        (e = t->groups.ensure(4 * t->n_group)) || (e = t->tiles.ensure(4 * t->n_tile)))
        return ctx->hip_fail(e, "node allocation");
    hipLaunchKernelGGL(k_nodes, dim3(nblk), dim3(256), 0, st, n, nblk, t->off.as<int>(), t->starts.as<unsigned>(),
                       t->nodes.as<GNode>(), t->pre.as<int>(), t->node_at.as<int>(), t->groups.as<int>(),
                       t->tiles.as<int>());
    hipLaunchKernelGGL(k_node_ends, dim3(blocks(nn)), dim3(256), 0, st, t->nodes.as<GNode>(), nn, n, n_leaf_limit,
                       skey, t->pre.as<int>(), t->range.as<int2>());
    // 4. moments: the leaves, then the inner nodes level by level
    if ((e = t->nmass.ensure(8 * nn)) || (e = t->ncom.ensure(24 * nn)) || (e = t->nquad.ensure(48 * nn)) ||
        (e = t->box_in.ensure(48 * nn)) || (e = t->box_out.ensure(48 * nn)))
        return ctx->hip_fail(e, "moment allocation");
    if ((e = t->rec.ensure((5 * sizeof(float4) + sizeof(int2)) * (size_t)nn))) return ctx->hip_fail(e, "node records");
    const MomentArrays mo{t->nmass.as<double>(), t->ncom.as<double>(), t->nquad.as<double>(), t->box_in.as<double>(),
                          t->box_out.as<double>(), t->walk_rec(), meta, t->pre.as<int>()};
    hipLaunchKernelGGL(k_leaf_moments, dim3((unsigned)((nn + 31) / 32)), dim3(256), 0, st, t->nodes.as<GNode>(), nn,
                       t->spos.as<double>(), t->smass.as<double>(), t->srs.as<double>(), mo);
    for (int l = GT_MAX_LEVEL; l >= 0; l--) {
        // (the deepest level holds leaves only)
        const long long a = M.level_start[l], b = M.level_start[l + 1];
        if (b <= a || b == nn) continue;
        // small levels, from here to the root, go together
        bool small = true;
        for (int q = 0; q <= l; q++) small = small && M.level_start[q + 1] - M.level_start[q] <= TOP_NODES;
        if (small) {
            hipLaunchKernelGGL(k_top_moments, dim3(1), dim3(TOP_THREADS), 0, st, t->nodes.as<GNode>(), l, mo);
            break;
        }
        hipLaunchKernelGGL(k_inner_moments, dim3((unsigned)((b - a + 31) / 32)), dim3(256), 0, st,
                           t->nodes.as<GNode>(), a, b, mo);
    }
    const long long ng = t->n_group;
    const auto t1 = std::chrono::steady_clock::now();
    t->ms_build = std::chrono::duration<float, std::milli>(t1 - t0).count();
    // 5. walk.  With the previous build's list lengths per group at hand (same
    //    number of groups: a rebuild of slowly moving particles), one writing
    //    pass into regions of those lengths + 1/4 + 64 that also counts;
    //    otherwise a counting pass first.  A list that outgrew its region
    //    means a second, exact writing pass.
    WalkArgs wa = walk_args(t);
    wa.groups = t->groups.as<int>();
    wa.n_group = ng;
    wa.inv_theta2 = (theta > 0) ? 1.0 / (theta * theta) : 0.0;
    wa.theta_pos = theta > 0;
    WalkLists &W = t->walk;
    int rc = walk_run<false>(t, wa, W, was_built, ng);
    if (rc != PTH_OK) return rc;
    const WalkTotals tot = *W.host.as<WalkTotals>();
    t->groups_h.assign(W.info(), W.info() + ng);
    if (tot.e > 0x7fffffffLL || tot.s > 0x7fffffffLL)
        return ctx->fail(PTH_ERR_CAPACITY, "pth_gtree_build: lists exceed the int32 range");
    t->n_le = tot.e;
    t->n_ls = tot.s;
    t->walk_passes = ng > 0 ? W.passes : 0;
    const auto t2 = std::chrono::steady_clock::now();
    t->ms_walk = std::chrono::duration<float, std::milli>(t2 - t1).count();
    // 6. the lists, enqueued without waits
    if ((e = t->id_epj.ensure(4 * (size_t)std::max<long long>(tot.e, 1))) ||
        (e = t->id_spj.ensure(4 * (size_t)std::max<long long>(tot.s, 1))))
        return ctx->hip_fail(e, "list allocation");
    rc = walk_finish<false>(t, wa, W, t->canonical, t->id_epj.as<int>(), t->id_spj.as<int>());
    if (rc != PTH_OK) return rc;
    // meanwhile, the plan of a resident evaluation of these lists under the
    // context's parameters (pth_resident_from_gtree / _refill take it over)
    {
        std::vector<int> ni(ng), nje(ng), njs(ng);
        for (long long g = 0; g < ng; g++) {
            ni[g] = t->groups_h[g].y;
            nje[g] = t->groups_h[g].z;
            njs[g] = t->groups_h[g].w;
        }
        const pth_params &par = ctx->par;
        t->pre_key = PlanKey{par.exec_mode, par.chunk_j, par.max_ipl,
                             par.exec_mode == PTH_EXEC_FUSED ? par.segments : 1, par.spj_monopole,
                             seg_pairs(par)};
        t->pre_ok = make_plan((int)ng, ni.data(), nje.data(), njs.data(), t->pre_key.exec_mode, t->pre_key.chunk_j,
                              t->pre_key.max_ipl, t->pre_plan, t->pre_key.n_seg, t->pre_key.mono != 0,
                              t->pre_key.min_seg_pairs, true);
        t->pre_valid = true;
    }
    if ((e = hipGetLastError()) || (e = hipStreamSynchronize(st))) return ctx->hip_fail(e, "tree walk");
    const auto t3 = std::chrono::steady_clock::now();
    t->ms_order = std::chrono::duration<float, std::milli>(t3 - t2).count();
    t->built = true;
    return PTH_OK;
}

// The tree's SPJ lists as node numbers to out (16-byte aligned).
void node_lists(const pth_gtree *t, int *out, hipStream_t st)
{
    if (t->n_ls <= 0) return;
    hipLaunchKernelGGL(k_node_lists, dim3(blocks((t->n_ls + 3) / 4)), dim3(256), 0, st, t->n_ls, t->id_spj.as<int>(),
                       t->node_at.as<int>(), out);
}

// (Re)fills resident r from tree t: plan, buffers, records and lists.
int resident_fill_gtree(pth_resident *r, const pth_gtree *t, const char *who)
{
    pth_ctx *c = r->ctx;
    const std::string w(who);
    if (!t) return c->fail(PTH_ERR_ARG, w + ": null tree");
    if (!t->built) return c->fail(PTH_ERR_STATE, w + ": the last build of the tree failed");
    if (t->ctx->device != c->device) return c->fail(PTH_ERR_ARG, w + ": the tree lives on another device");
    if (t->n_node > 0x7fffffffLL) return c->fail(PTH_ERR_CAPACITY, w + ": node count exceeds the int32 range");
    const long long ng = t->n_group;
    std::vector<int> ni(ng), ne(ng), ns(ng);
    long long next = 0;
    for (long long g = 0; g < ng; g++) {
        if (t->groups_h[g].x != next)
            return c->fail(PTH_ERR_STATE, w + ": the groups do not tile the particles");
        next += t->groups_h[g].y;
        ni[g] = t->groups_h[g].y;
        ne[g] = t->groups_h[g].z;
        ns[g] = t->groups_h[g].w;
    }
    // the plan made during the build, when it was made for this context's
    // parameters (then taken over: a second refill plans again)
    const pth_params &par = c->par;
    const PlanKey key{par.exec_mode, par.chunk_j, par.max_ipl, par.exec_mode == PTH_EXEC_FUSED ? par.segments : 1,
                      par.spj_monopole, seg_pairs(par)};
    const bool take = t->pre_valid && t->pre_key == key;
    const int rc = resident_setup(r, (int)ng, ni.data(), ne.data(), ns.data(), t->n_le, t->n_ls, (int)t->n,
                                  (int)t->n_node, who, take ? &t->pre_plan : nullptr, t->pre_ok);
    if (take) t->pre_valid = false;
    if (rc != PTH_OK) return rc;
    const Plan &P = r->plan;
    const Arena &A = r->A;
    auto bail = [&](hipError_t e, const char *what) { return c->hip_fail(e, what); };
    if (P.ni_tot != t->n) return c->fail(PTH_ERR_STATE, w + ": the groups do not cover the particles");
    hipStream_t st = c->stream;
    hipError_t e;
    char *d = r->arena.as<char>();
    // plan tables from the host (one copy, from pinned memory: nothing waits
    // for it; the caller has waited for the last refill's), lists and records
    // on the device
    const size_t tables = A.ide - A.walks;
    if ((e = r->h_plan.ensure(tables))) return bail(e, "pinned plan");
    copy_tables_to_arena(r->h_plan.as<char>() - A.walks, P, A);
    if ((e = hipMemcpyAsync(d + A.walks, r->h_plan.p, tables, hipMemcpyHostToDevice, st)) ||
        (P.item_bytes() &&
         (e = hipMemcpyAsync(d + A.items, P.items.data(), P.item_bytes(), hipMemcpyHostToDevice, st))) ||
        (P.ritem_bytes() &&
         (e = hipMemcpyAsync(d + A.ritems, P.ritems.data(), P.ritem_bytes(), hipMemcpyHostToDevice, st))))
        return bail(e, "resident upload");
    if (t->n_le && (e = hipMemcpyAsync(d + A.ide, t->id_epj.p, 4 * (size_t)t->n_le, hipMemcpyDeviceToDevice, st)))
        return bail(e, "resident lists");
    node_lists(t, reinterpret_cast<int *>(d + A.ids), st);
    hipLaunchKernelGGL(k_res_particles, dim3(blocks(t->n)), dim3(256), 0, st, t->n, t->spos.as<double>(),
                       t->smass.as<double>(), t->srs.as<double>(), reinterpret_cast<EpiDev *>(d + A.epi),
                       r->epj.as<EpjDev>());
    if (P.mono)
        hipLaunchKernelGGL(k_res_nodes_mono, dim3(blocks(t->n_node)), dim3(256), 0, st, t->n_node,
                           t->nmass.as<double>(), t->ncom.as<double>(), r->spj.as<EpjDev>());
    else
        hipLaunchKernelGGL(k_res_nodes, dim3(blocks(t->n_node)), dim3(256), 0, st, t->n_node, t->nmass.as<double>(),
                           t->ncom.as<double>(), t->nquad.as<double>(), r->spj.as<SpjDev>());
    if ((e = hipGetLastError())) return bail(e, "resident records");
    if ((e = resident_finish(r))) return bail(e, "resident SPJ table");
    // the tree's next build waits for its own context's stream: another one's
    // copies are done before this returns (and those from the plan's own items)
    if ((t->ctx != c || !P.on_device) && (e = hipStreamSynchronize(st))) return bail(e, "resident records");
    return PTH_OK;
}

}  // namespace

extern "C" {

int pth_gtree_build(pth_ctx *ctx, pth_gtree **out, long long n, const double *pos, const double *mass,
                    const double *r_search, int n_leaf_limit, int n_group_limit, double theta, int canonical)
{
    if (!ctx) return PTH_ERR_ARG;
    if (!out) return ctx->fail(PTH_ERR_ARG, "pth_gtree_build: null output");
    *out = nullptr;
    if (n <= 0 || n > 0x7fffffffLL) return ctx->fail(PTH_ERR_ARG, "pth_gtree_build: n outside [1, 2^31)");
    if (!pos || !mass) return ctx->fail(PTH_ERR_ARG, "pth_gtree_build: null particle arrays");
    if (n_leaf_limit < 1 || n_group_limit < 1) return ctx->fail(PTH_ERR_ARG, "pth_gtree_build: limits must be >= 1");
    HIPCHK(ctx, hipSetDevice(ctx->device), "hipSetDevice");
    pth_gtree *t = new pth_gtree;
    t->ctx = ctx;
    t->n_leaf_limit = n_leaf_limit;
    t->n_group_limit = n_group_limit;
    t->theta = theta;
    t->canonical = canonical != 0;
    const int rc = gtree_run(t, n, pos, mass, r_search, false);
    if (rc != PTH_OK) {
        pth_gtree_free(t);
        return rc;
    }
    *out = t;
    return PTH_OK;
}

int pth_gtree_update(pth_gtree *t, long long n, const double *pos, const double *mass, const double *r_search,
                     int on_device)
{
    if (!t) return PTH_ERR_ARG;
    pth_ctx *ctx = t->ctx;
    if (n <= 0 || n > 0x7fffffffLL) return ctx->fail(PTH_ERR_ARG, "pth_gtree_update: n outside [1, 2^31)");
    if (!pos || !mass) return ctx->fail(PTH_ERR_ARG, "pth_gtree_update: null particle arrays");
    HIPCHK(ctx, hipSetDevice(ctx->device), "hipSetDevice");
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream), "hipStreamSynchronize");
    return gtree_run(t, n, pos, mass, r_search, on_device != 0);
}

int pth_gtree_sizes(const pth_gtree *t, long long *n_node, long long *n_group, long long *n_epj_list,
                    long long *n_spj_list)
{
    if (!t) return PTH_ERR_ARG;
    if (!t->built) return t->ctx->fail(PTH_ERR_STATE, "pth_gtree_sizes: the last build failed");
    if (n_node) *n_node = t->n_node;
    if (n_group) *n_group = t->n_group;
    if (n_epj_list) *n_epj_list = t->n_le;
    if (n_spj_list) *n_spj_list = t->n_ls;
    return PTH_OK;
}

int pth_gtree_download(const pth_gtree *t, long long *order, long long *node_begin, long long *node_end,
                       int *node_level, double *node_mass, double *node_com, double *node_quad, long long *epi_begin,
                       int *n_epi, int *n_epj, int *n_spj, int *id_epj, int *id_spj)
{
    if (!t) return PTH_ERR_ARG;
    pth_ctx *c = t->ctx;
    if (!t->built) return c->fail(PTH_ERR_STATE, "pth_gtree_download: the last build failed");
    HIPCHK(c, hipSetDevice(c->device), "hipSetDevice");
    auto d2h = [&](void *h, const DevBuf &b, size_t bytes) -> hipError_t {
        return (h && bytes) ? hipMemcpy(h, b.p, bytes, hipMemcpyDeviceToHost) : hipSuccess;
    };
    const long long nn = t->n_node, ng = t->n_group;
    HIPCHK(c, d2h(order, t->order, 8 * t->n), "download");
    HIPCHK(c, d2h(node_mass, t->nmass, 8 * nn), "download");
    HIPCHK(c, d2h(node_com, t->ncom, 24 * nn), "download");
    HIPCHK(c, d2h(node_quad, t->nquad, 48 * nn), "download");
    HIPCHK(c, d2h(id_epj, t->id_epj, 4 * t->n_le), "download");
    if (id_spj && t->n_ls > 0) {
        // (by way of the walk's raw lists, which the next walk writes anew:
        // they held these entries, so they have room for them)
        const DevBuf &b = t->walk.raw_s;
        if (b.cap < 4 * (size_t)t->n_ls) return c->fail(PTH_ERR_STATE, "pth_gtree_download: no room for the lists");
        node_lists(t, b.as<int>(), c->stream);
        HIPCHK(c, hipGetLastError(), "list kernel");
        HIPCHK(c, hipStreamSynchronize(c->stream), "download");
        HIPCHK(c, d2h(id_spj, b, 4 * t->n_ls), "download");
    }
    std::vector<GNode> nodes(nn);
    HIPCHK(c, d2h(nodes.data(), t->nodes, sizeof(GNode) * nn), "download");
    for (long long k = 0; k < nn; k++) {
        if (node_begin) node_begin[k] = nodes[k].begin;
        if (node_end) node_end[k] = nodes[k].end;
        if (node_level) node_level[k] = nodes[k].level;
    }
    for (long long g = 0; g < ng; g++) {
        const int4 G = t->groups_h[g];
        if (epi_begin) epi_begin[g] = G.x;
        if (n_epi) n_epi[g] = G.y;
        if (n_epj) n_epj[g] = G.z;
        if (n_spj) n_spj[g] = G.w;
    }
    return PTH_OK;
}

int pth_gtree_timing(const pth_gtree *t, float *ms_build, float *ms_walk, float *ms_order)
{
    if (!t) return PTH_ERR_ARG;
    if (ms_build) *ms_build = t->ms_build;
    if (ms_walk) *ms_walk = t->ms_walk;
    if (ms_order) *ms_order = t->ms_order;
    return PTH_OK;
}

int pth_gtree_stats(const pth_gtree *t, int *walk_passes, int *tile_walk_passes, int *filter_passes)
{
    if (!t) return PTH_ERR_ARG;
    if (walk_passes) *walk_passes = t->walk_passes;
    if (tile_walk_passes) *tile_walk_passes = t->tile_passes;
    if (filter_passes) *filter_passes = t->ngb_passes;
    return PTH_OK;
}

int pth_resident_from_gtree(pth_ctx *c, pth_resident **out, const pth_gtree *t)
{
    if (!c) return PTH_ERR_ARG;
    if (!out) return c->fail(PTH_ERR_ARG, "pth_resident_from_gtree: null output");
    *out = nullptr;
    pth_resident *r = new pth_resident;
    r->ctx = c;
    const int rc = resident_fill_gtree(r, t, "pth_resident_from_gtree");
    if (rc != PTH_OK) {
        pth_resident_free(r);
        return rc;
    }
    *out = r;
    return PTH_OK;
}

int pth_resident_refill(pth_resident *r, const pth_gtree *t)
{
    if (!r) return PTH_ERR_ARG;
    HIPCHK(r->ctx, hipSetDevice(r->ctx->device), "hipSetDevice");
    HIPCHK(r->ctx, hipStreamSynchronize(r->ctx->stream), "hipStreamSynchronize");
    return resident_fill_gtree(r, t, "pth_resident_refill");
}

int pth_gtree_neighbors(pth_gtree *t, long long *n_total)
{
    if (!t) return PTH_ERR_ARG;
    pth_ctx *c = t->ctx;
    if (!t->built) return c->fail(PTH_ERR_STATE, "pth_gtree_neighbors: the last build failed");
    HIPCHK(c, hipSetDevice(c->device), "hipSetDevice");
    hipStream_t st = c->stream;
    const auto t0 = std::chrono::steady_clock::now();
    const long long n = t->n;
    size_t tb = 0;
    hipError_t e;
    // 1. candidate lists: one overlap-only walk per tile (the largest cells
    //    with at most 64 particles; theta opening off: inv_theta2 = 0), the
    //    group walk's symmetric r_search tests on widened tile boxes
    const long long nt = t->n_tile;
    HIPCHK(c, t->tbox.ensure(sizeof(double) * 12 * nt), "neighbour buffers");
    hipLaunchKernelGGL(k_tile_boxes, dim3(blocks(nt)), dim3(256), 0, st, t->tiles.as<int>(), nt,
                       t->box_in.as<double>(), t->box_out.as<double>(), t->rs_max, t->tbox.as<double>());
    WalkArgs wa = walk_args(t);
    wa.groups = t->tiles.as<int>();
    wa.n_group = nt;
    wa.tbox = t->tbox.as<double>();
    wa.theta_pos = 1;
    const unsigned wgt = (unsigned)std::min<long long>(nt, 65536);
    // (regions of the last search's lengths when it had as many tiles)
    WalkLists &W = t->tile_walk;
    int rc = walk_run<true>(t, wa, W, true, nt);
    if (rc != PTH_OK) return rc;
    const long long ncand = W.host.as<WalkTotals>()->e;
    if (ncand > 0x7fffffffLL) {
        W.n = -1;
        return c->fail(PTH_ERR_CAPACITY, "pth_gtree_neighbors: candidates exceed the int32 range");
    }
    t->tile_passes = nt > 0 ? W.passes : 0;
    HIPCHK(c, t->tl.ensure(sizeof(int) * std::max<long long>(ncand, 1)), "neighbour buffers");
    // candidates ascending in tree order, so rows come out in that order
    rc = walk_finish<true>(t, wa, W, true, t->tl.as<int>(), nullptr);
    if (rc != PTH_OK) return rc;
    // 2. exact FP64 filter of the candidates.  After a completed search of
    //    as many particles: one writing pass into regions of that search's
    //    counts + 1/4 + 4 that also counts (their total is at most 1.25 times
    //    its total + 4 n, since ngb_cnt holds exactly its counts), then the
    //    move into place, or an exact writing pass if some particle did not
    //    fit.  Otherwise: count, scan, write.
    const long long prev_total = t->ngb_prev_total;
    // (the region scan accumulates in int: its total must stay below 2^31)
    const bool one_pass_ngb = t->ngb_prev_ok && t->ngb_prev_n == n && n > 0 &&
                              prev_total + prev_total / 4 + 4 * n + 64 < 0x7fffffffLL;
    t->ngb_prev_ok = false;  // ngb_cnt is rewritten below
    HIPCHK(c, t->ngb_cnt.ensure(sizeof(int) * (n + 1)), "neighbour buffers");
    HIPCHK(c, t->ngb_off.ensure(sizeof(long long) * (n + 1)), "neighbour buffers");
    NgbArgs na{};
    na.spos = t->spos.as<double>();
    na.srs = t->srs.as<double>();
    na.order = t->order.as<long long>();
    na.info = reinterpret_cast<const int4 *>(W.back.as<WalkTotals>() + 1);
    na.off_e = W.off.as<long long>();
    na.id_epj = t->tl.as<int>();
    na.n_group = nt;
    na.cnt = t->ngb_cnt.as<int>();
    if (one_pass_ngb) {
        const long long bound = prev_total + prev_total / 4 + 4 * n + 64;
        HIPCHK(c, t->ngb_cap.ensure(sizeof(int) * (n + 1)), "neighbour buffers");
        HIPCHK(c, t->ngb_poff.ensure(sizeof(long long) * (n + 1)), "neighbour buffers");
        HIPCHK(c, t->ngb_pad.ensure(sizeof(int) * (size_t)bound), "neighbour buffers");
        HIPCHK(c, t->ngb_flag.ensure(sizeof(int)), "neighbour buffers");
        hipLaunchKernelGGL(k_ngb_caps, dim3(blocks(n + 1)), dim3(256), 0, st, n, t->ngb_cnt.as<int>(),
                           t->ngb_cap.as<int>());
        if ((e = hipcub::DeviceScan::ExclusiveSum(nullptr, tb, t->ngb_cap.as<int>(), t->ngb_poff.as<long long>(),
                                                  (int)(n + 1), st)) ||
            (e = cub_temp(t, tb)) ||
            (e = hipcub::DeviceScan::ExclusiveSum(t->tmp.p, tb, t->ngb_cap.as<int>(), t->ngb_poff.as<long long>(),
                                                  (int)(n + 1), st)))
            return c->hip_fail(e, "neighbour regions");
        hipLaunchKernelGGL(k_fill_int, dim3(1), dim3(64), 0, st, t->ngb_flag.as<int>(), 1, 0);
        na.off = t->ngb_poff.as<long long>();
        na.ngb = t->ngb_pad.as<int>();
        na.padded = 1;
        na.flag = t->ngb_flag.as<int>();
    }
    // the count of entry n stays 0 so the scan's last entry is the total
    hipLaunchKernelGGL(k_fill_int, dim3(1), dim3(64), 0, st, t->ngb_cnt.as<int>() + n, 1, 0);
    if (one_pass_ngb) hipLaunchKernelGGL(k_ngb<true>, dim3(wgt), dim3(64), 0, st, na);
    else hipLaunchKernelGGL(k_ngb<false>, dim3(wgt), dim3(64), 0, st, na);
    if ((e = hipcub::DeviceScan::ExclusiveSum(nullptr, tb, t->ngb_cnt.as<int>(), t->ngb_off.as<long long>(),
                                              (int)(n + 1), st)) ||
        (e = cub_temp(t, tb)) ||
        (e = hipcub::DeviceScan::ExclusiveSum(t->tmp.p, tb, t->ngb_cnt.as<int>(), t->ngb_off.as<long long>(),
                                              (int)(n + 1), st)))
        return c->hip_fail(e, "neighbour scan");
    long long total = 0;
    int over = 0;
    HIPCHK(c, hipMemcpyAsync(&total, t->ngb_off.as<long long>() + n, 8, hipMemcpyDeviceToHost, st), "neighbour total");
    if (one_pass_ngb)
        HIPCHK(c, hipMemcpyAsync(&over, t->ngb_flag.p, sizeof(int), hipMemcpyDeviceToHost, st), "neighbour total");
    HIPCHK(c, hipStreamSynchronize(st), "neighbour count");
    if (total > 0x7fffffffLL) return c->fail(PTH_ERR_CAPACITY, "pth_gtree_neighbors: lists exceed the int32 range");
    HIPCHK(c, t->ngb.ensure(sizeof(int) * std::max<long long>(total, 1)), "neighbour buffers");
    const bool rewrite = !one_pass_ngb || over != 0;
    if (total > 0 && rewrite) {
        na.off = t->ngb_off.as<long long>();
        na.ngb = t->ngb.as<int>();
        na.padded = 0;
        hipLaunchKernelGGL(k_ngb<true>, dim3(wgt), dim3(64), 0, st, na);
    } else if (total > 0) {
        // every particle fits its region (no flag raised)
        hipLaunchKernelGGL(k_ngb_compact, dim3(blocks(n)), dim3(256), 0, st, n, t->ngb_poff.as<long long>(),
                           t->ngb_off.as<long long>(), t->ngb_pad.as<int>(), t->ngb.as<int>());
    }
    HIPCHK(c, hipGetLastError(), "neighbour search");
    HIPCHK(c, hipStreamSynchronize(st), "neighbour search");
    t->ngb_passes = rewrite ? 2 : 1;
    t->ngb_prev_ok = true;
    t->ngb_prev_n = n;
    t->ngb_prev_total = total;
    t->n_ngb = total;
    t->n_cand = ncand;
    t->ms_ngb = std::chrono::duration<float, std::milli>(std::chrono::steady_clock::now() - t0).count();
    if (n_total) *n_total = total;
    return PTH_OK;
}

int pth_gtree_neighbors_download(const pth_gtree *t, int *count, long long *offset, int *ngb, float *ms)
{
    if (!t) return PTH_ERR_ARG;
    pth_ctx *c = t->ctx;
    if (!t->built || t->n_ngb < 0)
        return c->fail(PTH_ERR_STATE, "pth_gtree_neighbors_download: no neighbour search since the last build");
    HIPCHK(c, hipSetDevice(c->device), "hipSetDevice");
    HIPCHK(c, copy_to_host(c->stream, c->rings, {{count, t->ngb_cnt.p, sizeof(int) * (size_t)t->n},
                                                {offset, t->ngb_off.p, sizeof(long long) * (size_t)(t->n + 1)},
                                                {ngb, t->ngb.p, sizeof(int) * (size_t)t->n_ngb}}), "download");
    if (ms) *ms = t->ms_ngb;
    return PTH_OK;
}

void pth_gtree_free(pth_gtree *t)
{
    if (!t) return;
    if (t->ctx && t->ctx->device >= 0) {
        (void)hipSetDevice(t->ctx->device);
        if (t->ctx->stream) (void)hipStreamSynchronize(t->ctx->stream);
    }
    DevBuf *all[] = {&t->order, &t->key, &t->skey, &t->sidx, &t->sidx2, &t->spos, &t->smass, &t->srs, &t->nodes,
                     &t->nmass, &t->ncom, &t->nquad, &t->box_in, &t->box_out, &t->rec, &t->groups, &t->id_epj,
                     &t->id_spj, &t->tmp, &t->ngb_cnt, &t->ngb_off, &t->ngb, &t->tiles, &t->tbox, &t->tl,
                     &t->ngb_cap, &t->ngb_poff, &t->ngb_pad, &t->ngb_flag, &t->meta, &t->pre, &t->node_at, &t->range};
    t->walk.release();
    t->tile_walk.release();
    for (DevBuf *b : all) b->release();
    t->release_scratch();
    if (t->pinned) (void)hipHostFree(t->pinned);
    if (t->ev_meta) (void)hipEventDestroy(t->ev_meta);
    delete t;
}

}  // extern "C"
