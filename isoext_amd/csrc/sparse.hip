// SparseGrid kernels: corner points, crossing-cell filter, and marching cubes
// over per-cell corner values with an exact position weld.
//
// Reference path replaced:
//   SparseGrid::get_points_from_cell_indices  src/grid/sparse.cu:21-36
//   SparseGrid::filter_cell_indices           src/grid/sparse.cu:150-179
//   mc::marching_cubes on a SparseGrid        src/mc/mc.cu:17-68 with the
//     identity get_cells (src/grid/sparse.cu:61-69) and vertex_welding
//     (src/utils.cu:32-59)
//
// Each sparse cell carries its own 8 corner values, so two cells sharing an
// edge may disagree about its vertex; the reference welds by position only.
// Sparse MC therefore welds instances (crossing edges of cells) with equal
// positions (equality on floats), with the representative of a position = the
// smallest (slot, edge) that produces it; vertex ids follow representative
// order and faces follow (slot, LUT slot) order, so output is deterministic.
// Everything after the first pass works on the active cells, compacted in id
// order: the cells a representative can be in lie in two short runs of that
// list (see k_smc_link), which a workgroup stages in LDS.
// Degenerate triangles (two equal corners) are dropped as in
// src/mc/nagae.cu:71; a position is emitted only if a kept triangle uses it.
// The per-vertex representative is exported for the backward pass.

#include <atomic>
#include <mutex>
#include <type_traits>
#include <utility>

#include "common.h"
#include "mc_luts.h"
#include "sparse.h"

namespace iso {

namespace {

constexpr int kB = 256;

static __constant__ uint64_t cSTris[2][256];

__device__ __forceinline__ void cell_xyz(int64_t id, int64_t Y, int64_t Z, int64_t &x, int64_t &y, int64_t &z) {
    const int64_t cz = Z - 1, cy = Y - 1;
    const int64_t r = div_fast(id, cz);
    z = id - r * cz;
    x = div_fast(r, cy);
    y = r - x * cy;
}

// The same with the divisors' reciprocals from the host: for ids of the grid
// with fewer than 2^31 columns and 2^52 cells (in.div), one FP64 product,
// within 1 of the quotient, and a multiply-high division.
__device__ __forceinline__ void cell_xyz(const SparseMcIn &in, int64_t id, int64_t &x, int64_t &y, int64_t &z) {
    const SparseDiv &d = in.div;
    if (d.ncell == 0 || (uint64_t) id >= (uint64_t) d.ncell) {   // past the grid's end too
        cell_xyz(id, in.g.Y, in.g.Z, x, y, z);
        return;
    }
    const int64_t cz = in.g.Z - 1;
    uint32_t r = (uint32_t) ((double) id * d.inv_cz);
    int64_t m = id - (int64_t) r * cz;
    if (m < 0) {
        --r;
        m += cz;
    } else if (m >= cz) {
        ++r;
        m -= cz;
    }
    const uint32_t q = d.cy.div(r);
    x = q;
    y = r - q * (uint32_t) (in.g.Y - 1);
    z = m;
}

__global__ void k_corner_points(const int64_t *ids, int64_t n, SparseGeom g, float *out) {
    int64_t i = (int64_t) blockIdx.x * kB + threadIdx.x;
    if (i >= n) return;
    int64_t x, y, z;
    cell_xyz(ids[i], g.Y, g.Z, x, y, z);
    float c[3][2] = {{grid_coord(x, g.X, g.amin[0], g.amax[0]), grid_coord(x + 1, g.X, g.amin[0], g.amax[0])},
                     {grid_coord(y, g.Y, g.amin[1], g.amax[1]), grid_coord(y + 1, g.Y, g.amin[1], g.amax[1])},
                     {grid_coord(z, g.Z, g.amin[2], g.amax[2]), grid_coord(z + 1, g.Z, g.amin[2], g.amax[2])}};
    float *o = out + 24 * i;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        o[3 * k + 0] = c[0][k >> 2];
        o[3 * k + 1] = c[1][(k >> 1) & 1];
        o[3 * k + 2] = c[2][k & 1];
    }
}

__global__ void k_crossing_flags(const float *values, int64_t n, float level, uint8_t *flags) {
    int64_t i = (int64_t) blockIdx.x * kB + threadIdx.x;
    if (i >= n) return;
    int c = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) c |= inside(values[8 * i + k], level) << k;
    flags[i] = (c != 0 && c != 255) ? 1 : 0;
}

__device__ __forceinline__ int scross(int cs) {
    int st = 0;
#pragma unroll
    for (int e = 0; e < 12; ++e)
        if (((cs >> edge_a(e)) & 1) != ((cs >> edge_b(e)) & 1)) st |= 1 << e;
    return st;
}

// Rank of edge e among the crossing edges st.
__device__ __forceinline__ int edge_rank(int st, int e) { return __popc(st & ((1 << e) - 1)); }

// Inclusive sums of two counters over a workgroup of kB threads; t0 / t1 the
// totals.  sh: 2 * kB / 64 entries.
__device__ __forceinline__ void block_incl2(int &a, int &b, int &t0, int &t1, int *sh) {
    constexpr int NW = kB / 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    a = wave_incl_sum(a);
    b = wave_incl_sum(b);
    if (lane == 63) {
        sh[wave] = a;
        sh[NW + wave] = b;
    }
    __syncthreads();
    t0 = t1 = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        if (w < wave) {
            a += sh[w];
            b += sh[NW + w];
        }
        t0 += sh[w];
        t1 += sh[NW + w];
    }
    __syncthreads();
}

// ---- pass 1: cases --------------------------------------------------------------
// Per cell its case index, with kSpecial set when a vertex of the cell may
// lie within 16 ulps of a grid point: |level - v| of some corner at most
// cand_eps times the corners' range (cand_eps bounds t near 0 or 1 with a 2x
// margin; NaN or infinite corners are special too).  Per kCellBlk cells the
// active cells and their crossing edges.  One read of the values bounds the
// pass (32 B a cell, four cells in flight per lane: 0.17 ms and 5.1 TB/s for
// 25.7 M cells); it is the only one over all cells, the later passes take the
// active ones.
constexpr int kSpecial = 256;
constexpr uint32_t kResSpecial = 1u << 17;
constexpr int kCellBlk = 1024;

__global__ void __launch_bounds__(kB) k_smc_cases(SparseMcIn in, uint16_t *cases, uint2 *bsum) {
    constexpr int U = kCellBlk / kB;
    const int64_t i0 = (int64_t) blockIdx.x * kCellBlk + threadIdx.x;
    float v[U][8];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int64_t i = min(i0 + u * kB, in.n - 1);
#pragma unroll
        for (int k = 0; k < 8; ++k) v[u][k] = __builtin_nontemporal_load(in.values + 8 * i + k);
    }
    int na = 0, ni = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int64_t i = i0 + u * kB;
        int cs = 0;
        float lo = v[u][0], hi = v[u][0], near = INFINITY;
        bool nan = false;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float x = v[u][k];
            cs |= inside(x, in.level) << k;
            lo = fminf(lo, x);
            hi = fmaxf(hi, x);
            near = fminf(near, fabsf(x - in.level));
            nan |= x != x;
        }
        if (i >= in.n) continue;
        const bool act = cs != 0 && cs != 255;
        const float span = hi - lo;
        const bool sp = nan || !(span < INFINITY) || !(near > in.cand_eps * span);
        if (cases) cases[i] = (uint16_t) (cs | (sp ? kSpecial : 0));
        na += act ? 1 : 0;
        ni += act ? __popc(scross(cs)) : 0;
    }
    __shared__ int sh[2 * kB / 64];
    int ta, ti;
    block_incl2(na, ni, ta, ti, sh);
    if (threadIdx.x == 0) bsum[blockIdx.x] = make_uint2((uint32_t) ta, (uint32_t) ti);
}

// ---- exclusive scans of the block sums ---------------------------------------------
// Chunk sums, then each chunk adds the chunks before it (read by every
// workgroup, a few KB) and scans itself: two launches whatever the count.
constexpr int kScanPer = 4, kScanBlk = kB * kScanPer;

__global__ void __launch_bounds__(kB) k_pair_sums(const uint2 *bsum, int64_t n, longlong2 *chunk) {
    int64_t a = 0, b = 0;
#pragma unroll
    for (int u = 0; u < kScanPer; ++u) {
        const int64_t i = (int64_t) blockIdx.x * kScanBlk + u * kB + threadIdx.x;
        const uint2 v = i < n ? bsum[i] : make_uint2(0, 0);
        a += v.x;
        b += v.y;
    }
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_down(a, o);
        b += __shfl_down(b, o);
    }
    __shared__ int64_t sa[kB / 64], sb[kB / 64];
    if ((threadIdx.x & 63) == 0) {
        sa[threadIdx.x >> 6] = a;
        sb[threadIdx.x >> 6] = b;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kB / 64; ++w) {
            a += sa[w];
            b += sb[w];
        }
        chunk[blockIdx.x] = make_longlong2(a, b);
    }
}

// pre (optional): exclusive prefixes (64-bit); tot[0..1]: the totals.
__global__ void __launch_bounds__(kB) k_pair_scan(const uint2 *bsum, int64_t n, const longlong2 *chunk,
                                                  longlong2 *pre, int64_t *tot) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __shared__ int64_t sa[kB / 64], sb[kB / 64];
    // the chunks before this one
    int64_t a = 0, b = 0;
#pragma unroll 4
    for (int64_t c = threadIdx.x; c < (int64_t) blockIdx.x; c += kB) {
        a += chunk[c].x;
        b += chunk[c].y;
    }
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_down(a, o);
        b += __shfl_down(b, o);
    }
    if (lane == 0) {
        sa[wave] = a;
        sb[wave] = b;
    }
    __syncthreads();
    int64_t ba = 0, bb = 0;
#pragma unroll
    for (int w = 0; w < kB / 64; ++w) {
        ba += sa[w];
        bb += sb[w];
    }
    __syncthreads();
    // this chunk: kScanPer consecutive entries a thread (their sums fit 32 bits: at most 12 * kCellBlk each)
    const int64_t i0 = (int64_t) blockIdx.x * kScanBlk + (int64_t) threadIdx.x * kScanPer;
    uint2 v[kScanPer];
    int ta = 0, tb = 0;
#pragma unroll
    for (int u = 0; u < kScanPer; ++u) {
        v[u] = i0 + u < n ? bsum[i0 + u] : make_uint2(0, 0);
        ta += (int) v[u].x;
        tb += (int) v[u].y;
    }
    __shared__ int sh[2 * kB / 64];
    int ia = ta, ib = tb, all_a, all_b;
    block_incl2(ia, ib, all_a, all_b, sh);
    if (pre) {
        int64_t ra = ba + (ia - ta), rb = bb + (ib - tb);
#pragma unroll
        for (int u = 0; u < kScanPer; ++u) {
            if (i0 + u < n) pre[i0 + u] = make_longlong2(ra, rb);
            ra += v[u].x;
            rb += v[u].y;
        }
    }
    if (threadIdx.x == 0 && blockIdx.x == gridDim.x - 1) {
        tot[0] = ba + all_a;
        tot[1] = bb + all_b;
    }
}

// ---- pass 2: the active cells, in id order ----------------------------------------
// info: case (bits 0-7), kSpecial, crossing edges (bits 16-27).
__global__ void __launch_bounds__(kB) k_smc_compact(SparseMcIn in, const uint16_t *cases, const longlong2 *pre,
                                                    SparseMcWork w) {
    constexpr int U = kCellBlk / kB;   // a wave takes 64 * U consecutive cells
    __shared__ uint16_t cross[256];
    __shared__ int sh[2 * kB / 64];
    cross[threadIdx.x] = (uint16_t) scross(threadIdx.x);
    const int64_t ncell = (in.g.X - 1) * (in.g.Y - 1) * (in.g.Z - 1);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t i0 = (int64_t) blockIdx.x * kCellBlk + wave * (64 * U) + lane;
    int cs[U], st[U], na = 0, ni = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) cs[u] = i0 + 64 * u < in.n ? cases[i0 + 64 * u] : 0;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u) {
        st[u] = cross[cs[u] & 255];   // 0 for the cases without a crossing
        na += __popcll(__ballot(st[u] != 0));
        ni += __popc(st[u]);
    }
    ni = wave_incl_sum(ni);
    if (lane == 63) {
        sh[wave] = na;
        sh[kB / 64 + wave] = ni;
    }
    __syncthreads();
    const longlong2 p0 = pre[blockIdx.x];
    int64_t a = p0.x, q = p0.y;
    for (int v = 0; v < wave; ++v) {
        a += sh[v];
        q += sh[kB / 64 + v];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const uint64_t m = __ballot(st[u] != 0);
        const int n = __popc(st[u]), incl = wave_incl_sum(n);
        if (st[u]) {
            const int64_t k = a + __popcll(m & ((1ull << lane) - 1)), i = i0 + 64 * u;
            const int64_t id = in.ids[i];
            w.aid[k] = id;
            w.aslot[k] = (int32_t) i;
            if ((k & (kB - 1)) == 0) w.bid[k / kB] = id;
            // ids are not checked: cells past the grid's end have larger coordinates than cand_eps was made for
            const int c = cs[u] | (id >= ncell ? kSpecial : 0);
            w.ainfo[k] = make_uint2((uint32_t) (q + incl - n), (uint32_t) c | (uint32_t) st[u] << 16);
        }
        a += __popcll(m);
        q += __shfl(incl, 63);
    }
}

__device__ __forceinline__ int64_t lower_id(const int64_t *ids, int64_t lo, int64_t hi, int64_t key) {
    while (lo < hi) {
        const int64_t m = (lo + hi) >> 1;
        if (ids[m] < key) lo = m + 1;
        else hi = m;
    }
    return lo;
}

// ---- pass 3: representatives ---------------------------------------------------------
// Lower neighbours of a cell (the cells that share an edge with it and come
// before it in id order), in id order.
constexpr int kNbOff[9][3] = {{-1, -1, 0}, {-1, 0, -1}, {-1, 0, 0}, {-1, 0, 1}, {-1, 1, 0},
                              {0, -1, -1}, {0, -1, 0},  {0, -1, 1}, {0, 0, -1}};
// Corner c of a cell as a corner of its neighbour k, or -1.
ISO_HD constexpr int nb_corner(int c, int k) {
    int r = 0;
    for (int a = 0; a < 3; ++a) {
        const int b = ((c >> (2 - a)) & 1) - kNbOff[k][a];
        if (b < 0 || b > 1) return -1;
        r |= b << (2 - a);
    }
    return r;
}
ISO_HD constexpr int nb_edge(int e, int k) {
    const int ca = nb_corner(edge_a(e), k), cb = nb_corner(edge_b(e), k);
    if (ca < 0 || cb < 0) return -1;
    for (int i = 0; i < 12; ++i)
        if (edge_a(i) == ca && edge_b(i) == cb) return i;
    return -1;
}

template <int N, typename F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
    static_for_impl<N>(f, std::make_integer_sequence<int, N>{});
}

// The runs of active cells that hold the lower neighbours of link workgroup
// b's cells: win[3b], win[3b + 1] bound the slice before (x - 1, y - 1 ..
// y + 1), win[3b + 2] starts the run in the same slice (y - 1), which ends
// with the workgroup's own cells.
__global__ void __launch_bounds__(64) k_smc_windows(SparseMcIn in, SparseMcWork w, const int64_t *tot) {
    const int64_t na = tot[0], b = (int64_t) blockIdx.x * 64 + threadIdx.x, a0 = b * kB;
    if (a0 >= na) return;
    const int64_t cz = in.g.Z - 1, cy = in.g.Y - 1, a1 = min(a0 + kB, na);
    const int64_t first = w.bid[b], last = w.aid[a1 - 1];
    const int64_t keys[3] = {first - (cy + 1) * cz - 1, last - (cy - 1) * cz + 2, first - cz - 1};
    // by blocks first (their first ids stay in the L2), then inside the block; the three searches step together
    int64_t lo[3], n[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        lo[j] = 0;
        n[j] = b + 1;   // blocks 0 .. b
    }
    auto search = [&](const int64_t *a) {
        while ((n[0] | n[1] | n[2]) != 0) {
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const int64_t h = n[j] >> 1;
                const bool lt = n[j] > 0 && a[lo[j] + h] < keys[j];
                lo[j] += lt ? h + 1 : 0;
                n[j] = lt ? n[j] - h - 1 : h;
            }
        }
    };
    search(w.bid);
#pragma unroll
    for (int j = 0; j < 3; ++j) {   // the answer is in the block before the first one at or above the key, or at its end
        lo[j] = lo[j] > 0 ? (lo[j] - 1) * kB : 0;
        n[j] = min((int64_t) kB, a1 - lo[j]);
    }
    search(w.aid);
    w.win[3 * b] = (int32_t) lo[0];
    w.win[3 * b + 1] = (int32_t) max(lo[0], lo[1]);
    w.win[3 * b + 2] = (int32_t) lo[2];
}

// Cell edge from corner c (its bit along axis a clear) along axis a.
__device__ __forceinline__ int edge_of(int c, int a) {
    const int k = a * 8 + c;
    return k < 16 ? (int) ((0xff57ff13ffffab98ull >> (4 * k)) & 15) : (int) ((0xf6f4f2f0u >> (4 * (k - 16))) & 15);
}

// Position of the vertex cell slot s (origin (x, y, z)) places on its edge e,
// if that edge crosses the level in the cell.
__device__ __forceinline__ bool inst_pos(const SparseMcIn &in, int64_t s, int64_t x, int64_t y, int64_t z, int e,
                                         float &px, float &py, float &pz) {
    const int ca = edge_a(e), cb = edge_b(e);
    const float va = in.values[8 * s + ca], vb = in.values[8 * s + cb];
    if (inside(va, in.level) == inside(vb, in.level)) return false;
    const float t = edge_t(va, vb, in.level);
    px = lerp1(t, grid_coord(x + (ca >> 2), in.g.X, in.g.amin[0], in.g.amax[0]),
               grid_coord(x + (cb >> 2), in.g.X, in.g.amin[0], in.g.amax[0]));
    py = lerp1(t, grid_coord(y + ((ca >> 1) & 1), in.g.Y, in.g.amin[1], in.g.amax[1]),
               grid_coord(y + ((cb >> 1) & 1), in.g.Y, in.g.amin[1], in.g.amax[1]));
    pz = lerp1(t, grid_coord(z + (ca & 1), in.g.Z, in.g.amin[2], in.g.amax[2]),
               grid_coord(z + (cb & 1), in.g.Z, in.g.amin[2], in.g.amax[2]));
    return true;
}

// Whether the vertex of edge e of active cell a lies within 16 ulps of an end
// of its edge: 0 no, 1 the first end, 2 the second.
__device__ __forceinline__ int near_end(const SparseMcIn &in, const SparseMcWork &w, int64_t a, int e) {
    int64_t x, y, z;
    cell_xyz(in, w.aid[a], x, y, z);
    const int64_t s = w.aslot[a];
    const int ca = edge_a(e), cb = edge_b(e), ax = edge_axis(e);
    const int64_t o = ax == 0 ? x : (ax == 1 ? y : z), n = ax == 0 ? in.g.X : (ax == 1 ? in.g.Y : in.g.Z);
    const float amin = in.g.amin[ax], amax = in.g.amax[ax];
    const float ga = grid_coord(o + ((ca >> (2 - ax)) & 1), n, amin, amax),
                gb = grid_coord(o + ((cb >> (2 - ax)) & 1), n, amin, amax);
    const float r = lerp1(edge_t(in.values[8 * s + ca], in.values[8 * s + cb], in.level), ga, gb);
    if (!near_endpoint(r, ga, gb)) return 0;
    const int64_t kr = ordered_key(r), ka = ordered_key(ga), kb = ordered_key(gb);
    return llabs(kr - ka) <= llabs(kr - kb) ? 1 : 2;
}

// By position, the first (active cell, edge) that holds the vertex of edge e
// of active cell a, a vertex within 16 ulps of corner pc of the cell: the edges
// through that grid point in the cells around it, in id order up to this one.
// Each is in one of the four columns whose places in the active list
// k_smc_link left (w.acol), a step or two from there.  Returns the active
// cell * 16 + edge.
__device__ __forceinline__ int64_t rep_at_point(const SparseMcIn &in, const SparseMcWork &w, int64_t a, int e,
                                                int pc) {
    const int64_t cy = in.g.Y - 1, cz = in.g.Z - 1, id = w.aid[a];
    const int4 col = w.acol[a];
    int64_t o[3];
    cell_xyz(in, id, o[0], o[1], o[2]);
    const int64_t n[3] = {in.g.X, in.g.Y, in.g.Z};
    float g[3][3];   // coordinates around the point, by axis
#pragma unroll
    for (int u = 0; u < 3; ++u) {
        const int64_t q = o[u] + ((pc >> (2 - u)) & 1);
#pragma unroll
        for (int k = 0; k < 3; ++k) g[u][k] = grid_coord(q + k - 1, n[u], in.g.amin[u], in.g.amax[u]);
    }
    // position of the vertex on the edge along axis ax that ends (hi) or begins at the point
    auto place = [&](const float *v, int c, int ax, float p[3]) {
        const int bit = 4 >> ax;
        const bool hi = c & bit;   // c: the point as a corner of the cell with values v
        const float va = v[c & ~bit], vb = v[c | bit];
        if (inside(va, in.level) == inside(vb, in.level)) return false;
        const float t = edge_t(va, vb, in.level);
#pragma unroll
        for (int u = 0; u < 3; ++u)
            p[u] = u == ax ? lerp1(t, hi ? g[u][0] : g[u][1], hi ? g[u][1] : g[u][2]) : lerp1(t, g[u][1], g[u][1]);
        return true;
    };
    float pos[3] = {0.f, 0.f, 0.f};
    place(in.values + 8 * (int64_t) w.aslot[a], pc, edge_axis(e), pos);
    for (int d = 7; d >= 0; --d) {   // the point is corner d of the cell looked at
        const int dx = (pc >> 2) - (d >> 2), dy = ((pc >> 1) & 1) - ((d >> 1) & 1), dz = (pc & 1) - (d & 1);
        const int64_t xx = o[0] + dx, yy = o[1] + dy, zz = o[2] + dz;
        if (xx < 0 || yy < 0 || zz < 0 || yy >= cy || zz >= cz) continue;
        const int64_t key = (xx * cy + yy) * cz + zz;
        if (key > id) break;
        // columns (-1, -1) and (-1, 1) from this cell's z on, (-1, 0) and (0, -1) from z - 1 on, its own: itself or
        // the one before it
        int64_t p = a;
        int steps = dz;
        if (dx < 0 || dy < 0) {
            const bool from_z = dx < 0 && dy != 0;
            p = from_z ? (dy < 0 ? col.x : col.z) : (dx < 0 ? col.y : col.w);
            if (!from_z) ++steps;
        }
        if (steps < 0) --p;
        for (; steps > 0 && p < a && w.aid[p] < key; --steps) ++p;
        if (p < 0 || p > a || (p == a ? id : w.aid[p]) != key) continue;
        const float *v = in.values + 8 * (int64_t) w.aslot[p];
        int first = 16;
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
            float q[3];
            const int e2 = edge_of(d & ~(4 >> ax), ax);
            if (place(v, d, ax, q) && q[0] == pos[0] && q[1] == pos[1] && q[2] == pos[2]) first = min(first, e2);
        }
        if (first < (p == a ? e : 16)) return p * 16 + first;
    }
    return a * 16 + e;
}

// One workgroup per kB active cells.  The lower neighbours of its cells lie
// in two runs of the active list (k_smc_windows), staged in LDS (ids and
// slots; a run longer than its space is searched in global memory instead).
// One lane per cell finds its up to nine neighbours with four binary
// searches; for each crossing edge the first neighbour present is the
// representative's cell where it holds the same two end values, for then it
// is the same vertex (all edges' values come in one round of loads, only of
// the rows that are needed: the L1 takes one row a cycle, and 12 of 18 pairs
// of edge and neighbour are never looked at); else the positions decide, and
// the next neighbour is tried.  That is exact for vertices more than 16 ulps
// from both ends of their edge; the others are found by k_smc_special among
// the edges that may be nearer.  Then one lane per crossing edge turns (cell,
// edge) into the representative's instance index, written in order.
// Workgroups go to the XCDs in contiguous eighths: taken in turn, every XCD
// read all rows (2.7 GB instead of 0.84 GB at the 2048^3 band, 9.7 M active
// cells).  Measured there 0.41 ms, with the windows 0.03 and the special edges
// 0.14; one lane per instance over a column table, which they replace, took
// 1.59 ms and its table 0.17.  L1 rows and the chain of loads bound it (20
// wavefronts a CU by LDS).  In LDS the runs' ids are kept relative to the lowest one they can hold, in
// 32 bits, filled up to a power of two.
constexpr int kWin1 = 1024, kWin2 = 512;
struct LinkLds {
    uint32_t id1[kWin1], id2[kWin2];
    int32_t slot1[kWin1], slot2[kWin2];
    int32_t rep[12 * kB];     // representative's active cell
    uint16_t ent[12 * kB];    // own cell (bits 0-7), own edge (8-11), representative's edge (12-15)
    uint8_t plain[kB];        // the cell's faces are all kept
};

__global__ void __launch_bounds__(kB) k_smc_link(SparseMcIn in, SparseMcWork w, const int64_t *tot) {
    __shared__ LinkLds s;
    const int tid = threadIdx.x;
    const int64_t na = tot[0], blk = xcd_item(blockIdx.x, (na + kB - 1) / kB), a0 = blk * kB;
    if (a0 >= na) return;
    const int64_t a1 = min(a0 + kB, na), a = min(a0 + tid, na - 1);
    const bool valid = a0 + tid < na;
    const int64_t cy = in.g.Y - 1, cz = in.g.Z - 1;
    const int64_t first = w.aid[a0], last = w.aid[a1 - 1];
    const int64_t base1 = first - (cy + 1) * cz - 1, base2 = first - cz - 1, end1 = last - (cy - 1) * cz + 2;
    const int64_t id = w.aid[a], slot = w.aslot[a];
    const uint2 info = w.ainfo[a];
    const int64_t b0 = w.ainfo[a0].x;
    const int st = valid ? (int) (info.y >> 16) & 0xfff : 0;
    int64_t x, y, z;
    cell_xyz(in, id, x, y, z);
    const int64_t wlo = w.win[3 * blk], whi = w.win[3 * blk + 1], plo = w.win[3 * blk + 2];
    const int n1 = (int) (whi - wlo), n2 = (int) (a1 - plo);
    const bool lds1 = n1 < kWin1 && end1 - base1 < 0xffffffffll, lds2 = n2 < kWin2 && last - base2 < 0xffffffffll;
    const int p1 = 1 << (32 - __clz(n1)), p2 = 1 << (32 - __clz(n2));   // the power of two above the count
    if (lds1)
        for (int i = tid; i < p1; i += kB) {
            s.id1[i] = i < n1 ? (uint32_t) (w.aid[wlo + i] - base1) : 0xffffffffu;
            if (i < n1) s.slot1[i] = w.aslot[wlo + i];
        }
    if (lds2)
        for (int i = tid; i < p2; i += kB) {
            s.id2[i] = i < n2 ? (uint32_t) (w.aid[plo + i] - base2) : 0xffffffffu;
            if (i < n2) s.slot2[i] = w.aslot[plo + i];
        }
    __syncthreads();

    // neighbours: index in the active list, present bits.  Keys: the first
    // entry of each neighbour column at or above z - 1 (z for the single ones)
    int64_t nbi[9];
    uint32_t have = 0;   // entries found, before the borders
    if (lds2) {
        const uint32_t k = (uint32_t) (id - cz - 1 - base2);
        int q = 0;
        for (int h = p2 >> 1; h > 0; h >>= 1) q += s.id2[q + h - 1] < k ? h : 0;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const bool hit = s.id2[q] == k + d;   // q <= n2 < p2: a filler ends the run
            nbi[5 + d] = plo + q;
            if (hit) have |= 1u << (5 + d);
            q += hit ? 1 : 0;
        }
    } else {
        const int64_t k = id - cz - 1;
        int64_t q = lower_id(w.aid, plo, a1, k);
        for (int d = 0; d < 3; ++d) {
            const bool hit = q < a1 && w.aid[q] == k + d;
            nbi[5 + d] = q;
            if (hit) have |= 1u << (5 + d);
            q += hit ? 1 : 0;
        }
    }
    if (lds1) {
        const uint32_t k = (uint32_t) (id - cy * cz - 1 - base1), kl = k + 1 - (uint32_t) cz, kh = k + 1 + (uint32_t) cz;
        int q = 0, ql = 0, qh = 0;
        for (int h = p1 >> 1; h > 0; h >>= 1) {
            q += s.id1[q + h - 1] < k ? h : 0;
            ql += s.id1[ql + h - 1] < kl ? h : 0;
            qh += s.id1[qh + h - 1] < kh ? h : 0;
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const bool hit = s.id1[q] == k + d;
            nbi[1 + d] = wlo + q;
            if (hit) have |= 1u << (1 + d);
            q += hit ? 1 : 0;
        }
        nbi[0] = wlo + ql;
        nbi[4] = wlo + qh;
        if (s.id1[ql] == kl) have |= 1u << 0;
        if (s.id1[qh] == kh) have |= 1u << 4;
    } else {
        const int64_t k = id - cy * cz - 1;
        int64_t q = lower_id(w.aid, wlo, whi, k);
        for (int d = 0; d < 3; ++d) {
            const bool hit = q < whi && w.aid[q] == k + d;
            nbi[1 + d] = q;
            if (hit) have |= 1u << (1 + d);
            q += hit ? 1 : 0;
        }
        nbi[0] = lower_id(w.aid, wlo, whi, k + 1 - cz);
        nbi[4] = lower_id(w.aid, wlo, whi, k + 1 + cz);
        if (nbi[0] < whi && w.aid[nbi[0]] == k + 1 - cz) have |= 1u << 0;
        if (nbi[4] < whi && w.aid[nbi[4]] == k + 1 + cz) have |= 1u << 4;
    }
    nbi[8] = a - 1;   // a present lower z neighbour is the entry before
    if (a > 0 && w.aid[a - 1] == id - 1) have |= 1u << 8;
    // ids run on past the borders: z - 1 (neighbours 1, 5, 8), z + 1 (3, 7), y - 1 (0, 5-7), y + 1 (4), x - 1 (0-4)
    if (z == 0) have &= ~0x122u;
    if (z + 1 >= cz) have &= ~0x088u;
    if (y == 0) have &= ~0x0e1u;
    if (y + 1 >= cy) have &= ~0x010u;
    if (x == 0) have &= ~0x01fu;

    float cv[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) cv[k] = in.values[8 * slot + k];
    auto row = [&](int k, int64_t i) -> int64_t {   // slot of neighbour k at index i of the list
        return k < 5 ? (lds1 ? s.slot1[i - wlo] : w.aslot[i]) : (lds2 ? s.slot2[i - plo] : w.aslot[i]);
    };
    // end values of each crossing edge in its first neighbour
    float va[12], vb[12];
    static_for<12>([&](auto E) {
        constexpr int e = E;
        va[e] = vb[e] = 0.0f;
        bool done = !((st >> e) & 1);
        static_for<9>([&](auto K) {
            constexpr int k = K;
            if constexpr (nb_edge(e, k) >= 0) {
                constexpr int c0 = nb_corner(edge_a(e), k), c1 = nb_corner(edge_b(e), k);
                if (!done && ((have >> k) & 1)) {
                    const float *v = in.values + 8 * row(k, nbi[k]);
                    va[e] = v[c0];
                    vb[e] = v[c1];
                    done = true;
                }
            }
        });
    });

    uint32_t own = 0, look = 0;   // edges that represent themselves; edges that may lie near a grid point
    const bool beyond = x >= in.g.X - 1;   // past the grid's end: cand_eps does not hold
    int q = (int) (info.x - b0);   // the cell's first instance in the workgroup
    static_for<12>([&](auto E) {
        constexpr int e = E, ax = edge_axis(e);
        if (!((st >> e) & 1)) return;
        const float ea = cv[edge_a(e)], eb = cv[edge_b(e)];
        // written so that NaN and infinite values do
        const float near = fabsf(eb - ea) * in.cand_eps;
        if (beyond || !(fabsf(in.level - ea) > near && fabsf(eb - in.level) > near)) look |= 1u << e;
        int32_t rep = (int32_t) a;
        int re = e;
        bool first = true, done = false;
        static_for<9>([&](auto K) {
            constexpr int k = K, e2 = nb_edge(e, k);
            if constexpr (e2 >= 0) {
                if (!done && ((have >> k) & 1)) {
                    float na_ = va[e], nb_ = vb[e];
                    if (!first) {   // the neighbour before it has another vertex there, or none
                        constexpr int c0 = nb_corner(edge_a(e), k), c1 = nb_corner(edge_b(e), k);
                        const float *v = in.values + 8 * row(k, nbi[k]);
                        na_ = v[c0];
                        nb_ = v[c1];
                    }
                    first = false;
                    done = na_ == ea && nb_ == eb;
                    if (!done && inside(na_, in.level) != inside(nb_, in.level)) {
                        // other values: the same vertex if the interpolation comes to the same position
                        const float t0 = edge_t(ea, eb, in.level), t1 = edge_t(na_, nb_, in.level);
                        done = true;
#pragma unroll
                        for (int u = 0; u < 3; ++u) {
                            const int64_t o = (u == 0 ? x : (u == 1 ? y : z)) + ((edge_a(e) >> (2 - u)) & 1),
                                          n = u == 0 ? in.g.X : (u == 1 ? in.g.Y : in.g.Z);
                            const float p0 = grid_coord(o, n, in.g.amin[u], in.g.amax[u]),
                                        p1 = u == ax ? grid_coord(o + 1, n, in.g.amin[u], in.g.amax[u]) : p0;
                            done = done && lerp1(t0, p0, p1) == lerp1(t1, p0, p1);
                        }
                    }
                    if (done) {
                        rep = (int32_t) nbi[k];
                        re = e2;
                    }
                }
            }
        });
        if (!done) own |= 1u << e;
        s.rep[q] = rep;
        s.ent[q] = (uint16_t) (tid | (e << 8) | (re << 12));
        ++q;
    });
    s.plain[tid] = look == 0;
    __syncthreads();

    const int64_t blast = w.ainfo[a1 - 1].x + (int64_t) __popc((w.ainfo[a1 - 1].y >> 16) & 0xfff);
    const int nq = (int) (blast - b0);
    for (int i = tid; i < nq; i += kB) {
        const int ent = s.ent[i], lc = ent & 255, re = ent >> 12;
        const int64_t ra = s.rep[i];
        const uint2 f = w.ainfo[ra];
        const int32_t r = (int32_t) f.x + edge_rank((int) (f.y >> 16) & 0xfff, re);
        w.rkey[b0 + i] = r;
        // a vertex owned by a special cell counts where a kept face uses it
        if ((f.y & kSpecial) && s.plain[lc]) w.used[r] = 1;
    }
    if (!valid) return;
    const uint64_t tw = cSTris[in.method][info.y & 255];
    w.ares[a] = own | ((1u << (tw & 15)) - 1) << 12 | (info.y & kSpecial ? kResSpecial : 0u);
    w.alook[a] = look;
    if (look) w.acol[a] = make_int4((int) nbi[0], (int) nbi[1], (int) nbi[4], (int) nbi[5]);
}

// The edges whose vertex may lie near a grid point: a workgroup takes `per`
// active cells, lists those edges in LDS, one lane tests each, and one lane
// finds the representative of one that is near by position.  Then the cells
// that had any: faces with two corners at one position are dropped, the kept
// ones mark the vertices they use.
//
// With few such edges it is a chain of dependent loads: many cells a
// workgroup, so that each step of the chain serves many of them at once (per =
// 512: 226 us, 1024: 147, 4096: 138 at 9.7 M active cells, most of it the
// chain).  Where many corners are at the level, it is the work at those edges,
// and it has to fill the chip: 2048 workgroups before any takes more than kB
// cells.  One lane an edge, from the lowest cell around the point to the first
// that matches, with the columns' places from k_smc_link and nine coordinates
// worked out once: eight lanes with a search and all their own coordinates
// each took six times as long.  Fields rounded to a cell: 200^3 (76 k active
// cells, 4096 a workgroup) 2.06 -> 0.05 ms, the 2048^3 band (9.7 M active
// cells, a quarter of the corners at the level) 10.3 -> 1.85 ms.
constexpr int64_t kSpecWgs = 2048;
constexpr int kSpecBlk = 4096, kSpecCells = 1024, kSpecList = 2048;
__global__ void __launch_bounds__(kB) k_smc_special(SparseMcIn in, SparseMcWork w, const int64_t *tot, int per) {
    // room for one more round of kB cells above the marks at which the lists are worked off
    __shared__ uint32_t list[kSpecList + 12 * kB];   // cell's place in cells (bits 0-11), edge (12-15), corner (16-18)
    __shared__ uint16_t cells[kSpecCells + kB];
    __shared__ uint32_t own[kSpecCells + kB];
    __shared__ int nlist, ncells, nslow;
    const int64_t na = tot[0], a0 = (int64_t) blockIdx.x * per;
    if (a0 >= na) return;
    if (threadIdx.x == 0) nlist = ncells = nslow = 0;
    __syncthreads();
    const int nblk = (int) min<int64_t>(per, na - a0);
    for (int c0 = 0; c0 < nblk; c0 += kB) {
        const int c = c0 + threadIdx.x;
        const uint32_t look = c < nblk ? w.alook[a0 + c] : 0u;
        if (look) {
            const int ci = atomicAdd(&ncells, 1);
            own[ci] = w.ares[a0 + c];
            cells[ci] = (uint16_t) c;
            int k = atomicAdd(&nlist, __popc(look));
            for (uint32_t m = look; m; m &= m - 1) list[k++] = (uint32_t) (ci | (__ffs(m) - 1) << 12);
        }
        __syncthreads();
        const int n = nlist, nc = ncells;
        if (c0 + kB < nblk && n <= kSpecList && nc <= kSpecCells) {
            __syncthreads();   // the counts are read before the next round adds to them
            continue;
        }
        // one lane an entry: those near a point are left ...
        for (int i0 = 0; i0 < n; i0 += kB) {
            const int i = i0 + threadIdx.x;
            uint32_t ent = 0;
            int end = 0;
            if (i < n) {
                ent = list[i];
                const int e = ent >> 12;
                end = near_end(in, w, a0 + cells[ent & 4095], e);
                ent |= (uint32_t) (end == 1 ? edge_a(e) : edge_b(e)) << 16;
            }
            __syncthreads();   // the entries of this round are read
            if (end) list[atomicAdd(&nslow, 1)] = ent;   // at most as many as were read
        }
        __syncthreads();
        // ... and one lane looks around each
        for (int i = threadIdx.x; i < nslow; i += kB) {
            const int ci = list[i] & 4095, e = (list[i] >> 12) & 15;
            const int64_t a = a0 + cells[ci], best = rep_at_point(in, w, a, e, list[i] >> 16), ra = best >> 4;
            const int re = (int) best & 15;
            const uint2 f = w.ainfo[a], fr = w.ainfo[ra];
            w.rkey[f.x + edge_rank((int) (f.y >> 16) & 0xfff, e)] =
                (int32_t) fr.x + edge_rank((int) (fr.y >> 16) & 0xfff, re);
            if (ra == a && re == e) atomicOr(&own[ci], 1u << e);
            else atomicAnd(&own[ci], ~(1u << e));
        }
        __threadfence_block();
        __syncthreads();
        for (int ci = threadIdx.x; ci < nc; ci += kB) {
            const int64_t a = a0 + cells[ci];
            const uint2 f = w.ainfo[a];
            const int st = (int) (f.y >> 16) & 0xfff;
            const uint64_t tw = cSTris[in.method][f.y & 255];
            const int nt = (int) (tw & 15);
            uint32_t kept = 0;
            for (int t = 0; t < nt; ++t) {
                const int32_t r0 = w.rkey[f.x + edge_rank(st, (int) ((tw >> (4 + 12 * t)) & 15))];
                const int32_t r1 = w.rkey[f.x + edge_rank(st, (int) ((tw >> (8 + 12 * t)) & 15))];
                const int32_t r2 = w.rkey[f.x + edge_rank(st, (int) ((tw >> (12 + 12 * t)) & 15))];
                if (r0 == r1 || r0 == r2 || r1 == r2) continue;
                kept |= 1u << t;
                w.used[r0] = 1;
                w.used[r1] = 1;
                w.used[r2] = 1;
            }
            w.ares[a] = (own[ci] & ~(31u << 12)) | kept << 12;
        }
        __syncthreads();
        if (threadIdx.x == 0) nlist = ncells = nslow = 0;
        __syncthreads();
    }
}

// Derivatives of a vertex's coordinate along its edge by the edge's end
// values: with t = (L - va) / (vb - va), dP (L - vb) / (vb - va)^2 and
// -dP (L - va) / (vb - va)^2, dP the edge's length.
__device__ __forceinline__ float2 edge_jac(const SparseMcIn &in, int64_t slot, int64_t x, int64_t y, int64_t z,
                                           int e) {
    const float va = in.values[8 * slot + edge_a(e)], vb = in.values[8 * slot + edge_b(e)], d = vb - va;
    if (!(d != 0.0f)) return make_float2(0.0f, 0.0f);
    const int ax = edge_axis(e);
    const int64_t o = ax == 0 ? x : (ax == 1 ? y : z), n = ax == 0 ? in.g.X : (ax == 1 ? in.g.Y : in.g.Z);
    const float amin = in.g.amin[ax], amax = in.g.amax[ax];
    const float dp = grid_coord(o + 1, n, amin, amax) - grid_coord(o, n, amin, amax), inv2 = 1.0f / (d * d);
    return make_float2(dp * (in.level - vb) * inv2, -dp * (in.level - va) * inv2);
}

// ---- pass 4: numbering and output ------------------------------------------------------
// Vertices an active cell emits: its own representatives; a special cell's
// only where a kept face of some cell uses them.
__device__ __forceinline__ uint32_t emitted(const SparseMcWork &w, int64_t a, uint32_t res) {
    uint32_t own = res & 0xfffu;
    if (res & kResSpecial) {
        const uint2 f = w.ainfo[a];
        const int st = (int) (f.y >> 16) & 0xfff;
        for (uint32_t m = own; m; m &= m - 1) {
            const int e = __ffs(m) - 1;
            if (!w.used[f.x + edge_rank(st, e)]) own &= ~(1u << e);
        }
    }
    return own;
}

// Per kB active cells (one wave): vertices and faces.
__global__ void __launch_bounds__(kB) k_smc_sizes(SparseMcWork w, const int64_t *tot, int64_t nblk, uint2 *bsum) {
    constexpr int U = kB / 64;
    const int lane = threadIdx.x & 63;
    const int64_t na = tot[0], blk = (int64_t) blockIdx.x * U + (threadIdx.x >> 6), a0 = blk * kB + lane;
    if (blk >= nblk) return;
    uint32_t res[U];
#pragma unroll
    for (int u = 0; u < U; ++u) res[u] = a0 + 64 * u < na ? w.ares[a0 + 64 * u] : 0u;
    int v = 0, f = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        v += __popc(emitted(w, a0 + 64 * u, res[u]));
        f += __popc((res[u] >> 12) & 31u);
    }
    v = wave_incl_sum(v);
    f = wave_incl_sum(f);
    if (lane == 63) bsum[blk] = make_uint2((uint32_t) v, (uint32_t) f);
}

// Vertices (position and source edge at their ids, the ids also per
// instance).  Bound by the rows it gathers and writes: 1.23 GB in 0.255 ms for
// 9.7 M vertices (4.8 TB/s); one lane a cell, looping over its vertices, took
// 0.34 ms.
__global__ void __launch_bounds__(kB) k_smc_verts(SparseMcIn in, SparseMcWork w, const int64_t *tot,
                                                  const longlong2 *pre, SparseMcOut o) {
    const int64_t na = tot[0], a0 = (int64_t) blockIdx.x * kB, a = a0 + threadIdx.x;
    if (a0 >= na) return;
    const uint32_t res = a < na ? w.ares[a] : 0u;
    const uint32_t own = emitted(w, a, res);
    __shared__ int sh[2 * kB / 64];
    __shared__ uint16_t list[12 * kB];   // cell (bits 0-7), edge
    const int n = __popc(own);
    int v = n, d = 0, tv, td;
    block_incl2(v, d, tv, td, sh);
    int k = v - n;
    for (uint32_t m = own; m; m &= m - 1) list[k++] = (uint16_t) (threadIdx.x | (__ffs(m) - 1) << 8);
    __syncthreads();
    const int64_t v0 = pre[blockIdx.x].x;
    for (int i = threadIdx.x; i < tv; i += kB) {   // one lane a vertex: coalesced writes, no idle lanes
        const int e = list[i] >> 8;
        const int64_t c = a0 + (list[i] & 255), vid = v0 + i, slot = w.aslot[c];
        int64_t x, y, z;
        cell_xyz(in, w.aid[c], x, y, z);
        float px, py, pz;
        inst_pos(in, slot, x, y, z, e, px, py, pz);
        o.v[3 * vid + 0] = px;
        o.v[3 * vid + 1] = py;
        o.v[3 * vid + 2] = pz;
        if (o.vsrc) o.vsrc[vid] = slot * 12 + e;
        if (o.vjac) o.vjac[vid] = edge_jac(in, slot, x, y, z, e);
        const uint2 f = w.ainfo[c];
        w.vid[f.x + edge_rank((int) (f.y >> 16) & 0xfff, e)] = (int32_t) vid;
    }
}

// Faces in (slot, LUT slot) order; the workgroup's instances' vertex ids are
// gathered in order into LDS first.  19.4 M faces in 0.19 ms; with the faces
// put together in LDS too (coalesced stores, half the wavefronts) 0.26 ms.
__global__ void __launch_bounds__(kB) k_smc_faces(SparseMcIn in, SparseMcWork w, const int64_t *tot,
                                                  const longlong2 *pre, SparseMcOut o) {
    __shared__ int32_t vid[12 * kB];
    __shared__ int sh[2 * kB / 64];
    const int64_t na = tot[0], blk = xcd_item(blockIdx.x, (na + kB - 1) / kB), a0 = blk * kB,
                  a = min(a0 + threadIdx.x, na - 1);
    if (a0 >= na) return;
    const int64_t a1 = min(a0 + kB, na);
    const int64_t b0 = w.ainfo[a0].x;
    const uint2 last = w.ainfo[a1 - 1], f = w.ainfo[a];
    const uint32_t kept = a0 + threadIdx.x < na ? (w.ares[a] >> 12) & 31u : 0u;
    const int nq = (int) (last.x - b0) + __popc((last.y >> 16) & 0xfff);
    for (int i = threadIdx.x; i < nq; i += kB) vid[i] = w.vid[w.rkey[b0 + i]];
    const int n = __popc(kept);
    int k = n, d = 0, tf, td;
    block_incl2(k, d, tf, td, sh);   // its barriers also complete vid[]
    const uint64_t tw = cSTris[in.method][f.y & 255];
    const int st = (int) (f.y >> 16) & 0xfff, lb = (int) (f.x - b0);
    int32_t *out = o.f + 3 * (pre[blk].y + k - n);
    for (uint32_t m = kept; m; m &= m - 1) {
        const int t = __ffs(m) - 1;
        out[0] = vid[lb + edge_rank(st, (int) ((tw >> (4 + 12 * t)) & 15))];
        out[1] = vid[lb + edge_rank(st, (int) ((tw >> (8 + 12 * t)) & 15))];
        out[2] = vid[lb + edge_rank(st, (int) ((tw >> (12 + 12 * t)) & 15))];
        out += 3;
    }
}

__global__ void k_fill_u64(unsigned long long *p, int64_t n, unsigned long long v) {
    for (int64_t i = (int64_t) blockIdx.x * kB + threadIdx.x; i < n; i += (int64_t) gridDim.x * kB) p[i] = v;
}

// single-block exclusive scan of int64 block sums; total in *tot
__global__ void k_scan_i64(int64_t *a, int64_t n, int64_t *tot) {
    __shared__ int64_t sh[1024];
    int64_t per = (n + 1023) / 1024;
    int64_t lo = threadIdx.x * per, hi = min(lo + per, n);
    int64_t sum = 0;
    for (int64_t i = lo; i < hi; ++i) sum += a[i];
    sh[threadIdx.x] = sum;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
        int64_t y = threadIdx.x >= (unsigned) o ? sh[threadIdx.x - o] : 0;
        __syncthreads();
        sh[threadIdx.x] += y;
        __syncthreads();
    }
    int64_t run = sh[threadIdx.x] - sum;
    for (int64_t i = lo; i < hi; ++i) {
        int64_t v = a[i];
        a[i] = run;
        run += v;
    }
    if (threadIdx.x == 1023) *tot = sh[1023];
}

// popcount prefix over bitmap words (blocks of 1024 words, then block sums)
__global__ void k_bit_block(const uint32_t *bits, int64_t nw, int64_t *pre, int64_t *bsum) {
    __shared__ int64_t sh[1024];
    int64_t i = (int64_t) blockIdx.x * 1024 + threadIdx.x;
    int64_t v = i < nw ? __popc(bits[i]) : 0;
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
        int64_t y = threadIdx.x >= (unsigned) o ? sh[threadIdx.x - o] : 0;
        __syncthreads();
        sh[threadIdx.x] += y;
        __syncthreads();
    }
    if (i < nw) pre[i] = sh[threadIdx.x] - v;
    if (threadIdx.x == 1023) bsum[blockIdx.x] = sh[1023];
}

__global__ void k_bit_add(int64_t *pre, int64_t nw, const int64_t *bsum) {
    int64_t i = (int64_t) blockIdx.x * 1024 + threadIdx.x;
    if (i < nw) pre[i] += bsum[blockIdx.x];
}

// ---- population: sorted-key set operations (src/grid/sparse.cu:71-121) ----------

// Bitmap of the elements a set operation keeps, one bit per element, written
// a 64-bit wave ballot at a time (element i -> bit i).
__device__ __forceinline__ bool found_sorted(const int64_t *a, int64_t n, int64_t key) {
    int64_t lo = 0, hi = n;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (a[mid] < key) lo = mid + 1;
        else hi = mid;
    }
    return lo < n && a[lo] == key;
}

// union: b (sorted) elements that start a run and are absent from a
// difference: a elements absent from b (sorted)
__global__ void k_setop_flags(const int64_t *a, int64_t na, const int64_t *b, int64_t nb, int difference,
                              unsigned long long *bits) {
    const int64_t n = difference ? na : nb;
    for (int64_t i0 = (int64_t) blockIdx.x * kB; i0 < n; i0 += (int64_t) gridDim.x * kB) {
        const int64_t i = i0 + threadIdx.x;
        bool keep = false;
        if (i < n) {
            if (difference) keep = !found_sorted(b, nb, a[i]);
            else keep = (i == 0 || b[i] != b[i - 1]) && !found_sorted(a, na, b[i]);
        }
        const unsigned long long m = __ballot(keep);
        if ((threadIdx.x & 63) == 0 && i < n) bits[i >> 6] = m;
    }
}

// Kept elements of `src` (bitmap + per-32-bit-word exclusive prefix) to
// consecutive positions of `out`; `slot` (optional) gets the source index.
__global__ void k_setop_compact(const int64_t *src, int64_t n, const uint32_t *bits, const int64_t *pre,
                                int64_t *out, int64_t *slot) {
    for (int64_t i = (int64_t) blockIdx.x * kB + threadIdx.x; i < n; i += (int64_t) gridDim.x * kB) {
        const uint32_t w = bits[i >> 5];
        if (!((w >> (i & 31)) & 1)) continue;
        const int64_t k = pre[i >> 5] + __popc(w & ((1u << (i & 31)) - 1));
        out[k] = src[i];
        if (slot) slot[k] = i;
    }
}

// Merge of two sorted, disjoint arrays: output k takes a[i] or b[k - i], i the
// number of a elements among the first k outputs (merge-path search on the
// diagonal); slot[k] = i when it comes from a, -1 from b.
__global__ void k_merge_disjoint(const int64_t *a, int64_t na, const int64_t *b, const int64_t *nb_p, int64_t *out,
                                 int64_t *slot, int64_t *n_out) {
    const int64_t nb = *nb_p, n = na + nb;
    if (blockIdx.x == 0 && threadIdx.x == 0) *n_out = n;
    for (int64_t k = (int64_t) blockIdx.x * kB + threadIdx.x; k < n; k += (int64_t) gridDim.x * kB) {
        int64_t lo = max((int64_t) 0, k - nb), hi = min(k, na);
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if (a[mid] < b[k - 1 - mid]) lo = mid + 1;
            else hi = mid;
        }
        const int64_t i = lo, j = k - lo;
        const bool from_a = j >= nb || (i < na && a[i] < b[j]);
        out[k] = from_a ? a[i] : b[j];
        if (slot) slot[k] = from_a ? i : -1;
    }
}

// Per-cell values after a set operation: the old row of the cell's source
// slot, or the default value for a new cell.
__global__ void k_gather_rows(const float *old_values, const int64_t *slot, int64_t n, float dflt, float *out) {
    for (int64_t t = (int64_t) blockIdx.x * kB + threadIdx.x; t < 8 * n; t += (int64_t) gridDim.x * kB) {
        const int64_t s = slot[t >> 3];
        out[t] = s >= 0 ? old_values[8 * s + (t & 7)] : dflt;
    }
}

unsigned nb(int64_t n) { return (unsigned) std::max<int64_t>(1, (n + kB - 1) / kB); }
unsigned gs(int64_t n) { return (unsigned) std::max<int64_t>(1, std::min<int64_t>(8192, (n + kB - 1) / kB)); }

}   // namespace

#define ISO_TRY(x)                       \
    do {                                 \
        hipError_t e_ = (x);             \
        if (e_ != hipSuccess) return e_; \
    } while (0)

// Scratch of a set operation on na (or nb) keys: the bitmap, its word prefix,
// the block sums, the compacted b and two counters.
int64_t sparse_setop_scratch_bytes(int64_t na, int64_t nb) {
    const int64_t n = std::max(na, nb), nw64 = n / 64 + 2, nw32 = 2 * nw64;
    return 8 * (nw64 + nw32 + (nw32 + 1023) / 1024 + 8 + nb + 8) + 256;
}

hipError_t sparse_setop(const int64_t *a, int64_t na, const int64_t *b, int64_t nb, bool difference, void *scratch,
                        int64_t *out, int64_t *slot, int64_t *n_out, hipStream_t st) {
    const int64_t n = difference ? na : nb, nw64 = std::max(na, nb) / 64 + 2, nw32 = 2 * nw64;
    char *p = (char *) scratch;
    unsigned long long *bits = (unsigned long long *) p;
    int64_t *pre = (int64_t *) (p + 8 * nw64);
    int64_t *bsum = pre + nw32;
    const int64_t nblk = (nw32 + 1023) / 1024;
    int64_t *tot = bsum + nblk + 8;
    int64_t *bc = tot + 8;   // compacted b (union)
    hipLaunchKernelGGL(k_fill_u64, dim3(gs(nw64)), dim3(kB), 0, st, bits, nw64, 0ull);
    if (n > 0)
        hipLaunchKernelGGL(k_setop_flags, dim3(gs(n)), dim3(kB), 0, st, a, na, b, nb, difference ? 1 : 0, bits);
    hipLaunchKernelGGL(k_bit_block, dim3((unsigned) nblk), dim3(1024), 0, st, (const uint32_t *) bits, nw32, pre, bsum);
    hipLaunchKernelGGL(k_scan_i64, dim3(1), dim3(1024), 0, st, bsum, nblk, tot);
    hipLaunchKernelGGL(k_bit_add, dim3((unsigned) nblk), dim3(1024), 0, st, pre, nw32, bsum);
    if (difference) {
        if (na > 0)
            hipLaunchKernelGGL(k_setop_compact, dim3(gs(na)), dim3(kB), 0, st, a, na, (const uint32_t *) bits, pre,
                               out, slot);
        ISO_TRY(hipMemcpyAsync(n_out, tot, sizeof(int64_t), hipMemcpyDeviceToDevice, st));
    } else {
        if (nb > 0)
            hipLaunchKernelGGL(k_setop_compact, dim3(gs(nb)), dim3(kB), 0, st, b, nb, (const uint32_t *) bits, pre, bc,
                               (int64_t *) nullptr);
        hipLaunchKernelGGL(k_merge_disjoint, dim3(gs(na + nb)), dim3(kB), 0, st, a, na, bc, tot, out, slot, n_out);
    }
    return hipGetLastError();
}

hipError_t sparse_gather_rows(const float *old_values, const int64_t *slot, int64_t n, float dflt, float *out,
                              hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_gather_rows, dim3(gs(8 * n)), dim3(kB), 0, st, old_values, slot, n, dflt, out);
    return hipGetLastError();
}

hipError_t sparse_corner_points(const int64_t *ids, int64_t n, const SparseGeom &g, float *out, hipStream_t st) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_corner_points, dim3(nb(n)), dim3(kB), 0, st, ids, n, g, out);
    return hipGetLastError();
}

hipError_t sparse_crossing_flags(const float *values, int64_t n, float level, uint8_t *flags, hipStream_t st) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_crossing_flags, dim3(nb(n)), dim3(kB), 0, st, values, n, level, flags);
    return hipGetLastError();
}

hipError_t sparse_mc_luts() {
    // once per device (each GPU holds its own copy of the constant table);
    // host threads that call first together wait for one upload
    constexpr int kMaxDevices = 64;
    static std::atomic<bool> done[kMaxDevices];
    static std::mutex mu;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    if (done[dev].load(std::memory_order_acquire)) return hipSuccess;
    std::lock_guard<std::mutex> lock(mu);
    if (done[dev].load(std::memory_order_relaxed)) return hipSuccess;
    uint64_t h[2][256];
    for (int i = 0; i < 256; ++i) {
        h[0][i] = kNagaeTris[i];
        h[1][i] = kLorensenTris[i];
    }
    e = hipMemcpyToSymbol(HIP_SYMBOL(cSTris), h, sizeof(h));
    if (e == hipSuccess) done[dev].store(true, std::memory_order_release);
    return e;
}

namespace {

// Scratch of the cases pass: the block sums, their chunk sums, the totals
// (active cells, instances) and, with_cases, the cases and the block prefixes
// that the compaction reads.
struct CaseScratch {
    int64_t *tot;
    uint2 *bsum;
    longlong2 *chunk, *pre;
    uint16_t *cases;
    size_t bytes;
    CaseScratch(void *base, int64_t n, bool with_cases) {
        const int64_t nblk = (n + kCellBlk - 1) / kCellBlk, nch = (nblk + kScanBlk - 1) / kScanBlk;
        bytes = 0;
        auto take = [&](size_t b) {
            char *r = (char *) base + bytes;
            bytes += (b + 15) & ~size_t(15);
            return r;
        };
        tot = (int64_t *) take(16);
        bsum = (uint2 *) take(8 * (size_t) nblk);
        chunk = (longlong2 *) take(16 * (size_t) nch);
        pre = (longlong2 *) (with_cases ? take(16 * (size_t) nblk) : nullptr);
        cases = (uint16_t *) (with_cases ? take(2 * (size_t) n) : nullptr);
    }
};

void scan_pairs(const uint2 *bsum, int64_t n, longlong2 *chunk, longlong2 *pre, int64_t *tot, hipStream_t st) {
    const unsigned nch = (unsigned) ((n + kScanBlk - 1) / kScanBlk);
    hipLaunchKernelGGL(k_pair_sums, dim3(nch), dim3(kB), 0, st, bsum, n, chunk);
    hipLaunchKernelGGL(k_pair_scan, dim3(nch), dim3(kB), 0, st, bsum, n, (const longlong2 *) chunk, pre, tot);
}

void cases_pass(const SparseMcIn &in, const CaseScratch &c, hipStream_t st) {
    const int64_t nblk = (in.n + kCellBlk - 1) / kCellBlk;
    hipLaunchKernelGGL(k_smc_cases, dim3((unsigned) nblk), dim3(kB), 0, st, in, c.cases, c.bsum);
    scan_pairs(c.bsum, nblk, c.chunk, c.pre, c.tot, st);
}

// Two counters from the device through a small pinned buffer of the calling thread.
hipError_t read2(const int64_t *src, int64_t out[2], hipStream_t st) {
    struct Pinned {
        int64_t *p = nullptr;
        ~Pinned() {
            if (p) (void) hipHostFree(p);
        }
    };
    thread_local Pinned h;
    if (!h.p) ISO_TRY(hipHostMalloc((void **) &h.p, 2 * sizeof(int64_t), 0));
    ISO_TRY(hipMemcpyAsync(h.p, src, 2 * sizeof(int64_t), hipMemcpyDeviceToHost, st));
    ISO_TRY(hipStreamSynchronize(st));
    out[0] = h.p[0];
    out[1] = h.p[1];
    return hipSuccess;
}

// Workspace of a run.
struct RunWork {
    SparseMcWork w;
    uint2 *bsum;             // per workgroup: vertices, faces
    longlong2 *chunk, *pre;  // their chunk sums and prefixes
    int64_t *tot;
    size_t bytes;
    RunWork(void *base, int64_t ninst, int64_t na) {
        const size_t nblk = nb(na), nch = (nblk + kScanBlk - 1) / kScanBlk;
        bytes = 0;
        auto take = [&](size_t n) {
            char *r = (char *) base + bytes;
            bytes += (n + 255) & ~size_t(255);
            return r;
        };
        w.aid = (int64_t *) take(8 * na);
        w.aslot = (int32_t *) take(4 * na);
        w.ainfo = (uint2 *) take(8 * na);
        w.ares = (uint32_t *) take(4 * na);
        w.alook = (uint32_t *) take(4 * na);
        w.acol = (int4 *) take(16 * na);
        w.win = (int32_t *) take(12 * nblk);
        w.bid = (int64_t *) take(8 * nblk);
        w.rkey = (int32_t *) take(4 * ninst);
        w.vid = (int32_t *) take(4 * ninst);
        w.used = (uint8_t *) take(ninst + 16);
        bsum = (uint2 *) take(8 * nblk);
        chunk = (longlong2 *) take(16 * nch);
        pre = (longlong2 *) take(16 * nblk);
        tot = (int64_t *) take(16);
    }
};

size_t mc_work_bytes(int64_t ninst, int64_t na) { return RunWork(nullptr, ninst, na).bytes; }

}   // namespace

size_t sparse_mc_scratch_bytes(int64_t n) { return CaseScratch(nullptr, n, true).bytes; }

hipError_t sparse_mc_cases(const SparseMcIn &in, void *scratch, int64_t &ninst, int64_t &nact, hipStream_t st) {
    ninst = nact = 0;
    if (in.n == 0) return hipSuccess;
    const CaseScratch c(scratch, in.n, true);
    cases_pass(in, c, st);
    ISO_TRY(hipGetLastError());
    int64_t h[2];
    ISO_TRY(read2(c.tot, h, st));
    nact = h[0];
    ninst = h[1];
    return hipSuccess;
}

hipError_t sparse_mc_count(const SparseMcIn &in, int64_t *scratch, int64_t &ninst, hipStream_t st) {
    ninst = 0;
    if (in.n == 0) return hipSuccess;
    const CaseScratch c(scratch, in.n, false);
    cases_pass(in, c, st);
    ISO_TRY(hipGetLastError());
    int64_t h[2];
    ISO_TRY(read2(c.tot, h, st));
    ninst = h[1];
    return hipSuccess;
}

size_t sparse_mc_work_bytes(int64_t n, int64_t ninst) {
    return ((sparse_mc_scratch_bytes(n) + 255) & ~size_t(255)) + mc_work_bytes(ninst, ninst / 3);
}
size_t sparse_mc_run_bytes(int64_t ninst, int64_t nact) { return mc_work_bytes(ninst, nact); }

hipError_t sparse_mc_run(const SparseMcIn &in, const void *scratch, int64_t ninst, int64_t nact, void *work,
                         size_t work_bytes, SparseMcOut &o, int64_t &nv, int64_t &nf, hipStream_t st) {
    nv = nf = 0;
    if (in.n == 0 || ninst == 0) return hipSuccess;
    if (in.n >= (int64_t) INT32_MAX || ninst >= (int64_t) INT32_MAX) return hipErrorInvalidValue;
    if (mc_work_bytes(ninst, nact) > work_bytes) return hipErrorInvalidValue;
    ISO_TRY(sparse_mc_luts());
    const CaseScratch c(const_cast<void *>(scratch), in.n, true);
    const unsigned nblk = nb(nact);
    const RunWork r(work, ninst, nact);
    const SparseMcWork &w = r.w;

    const int64_t ncell = (in.n + kCellBlk - 1) / kCellBlk, nu = (ninst + 15) / 8;
    hipLaunchKernelGGL(k_fill_u64, dim3(gs(nu)), dim3(kB), 0, st, (unsigned long long *) w.used, nu, 0ull);
    hipLaunchKernelGGL(k_smc_compact, dim3((unsigned) ncell), dim3(kB), 0, st, in, (const uint16_t *) c.cases,
                       (const longlong2 *) c.pre, w);
    hipLaunchKernelGGL(k_smc_windows, dim3((nblk + 63) / 64), dim3(64), 0, st, in, w, (const int64_t *) c.tot);
    hipLaunchKernelGGL(k_smc_link, dim3((nblk + 7) / 8 * 8), dim3(kB), 0, st, in, w, (const int64_t *) c.tot);
    const int per = (int) std::min<int64_t>(kSpecBlk, kB * (nact / (kSpecWgs * kB) + 1));
    hipLaunchKernelGGL(k_smc_special, dim3((unsigned) ((nact + per - 1) / per)), dim3(kB), 0, st, in, w,
                       (const int64_t *) c.tot, per);
    hipLaunchKernelGGL(k_smc_sizes, dim3((nblk + kB / 64 - 1) / (kB / 64)), dim3(kB), 0, st, w, (const int64_t *) c.tot,
                       (int64_t) nblk, r.bsum);
    scan_pairs(r.bsum, nblk, r.chunk, r.pre, r.tot, st);
    ISO_TRY(hipGetLastError());
    int64_t h[2];
    ISO_TRY(read2(r.tot, h, st));
    nv = h[0];
    nf = h[1];
    if (nv > o.cap_v || nf > o.cap_f) return hipSuccess;   // caller makes room: sparse_mc_emit, or the run again
    return sparse_mc_emit(in, scratch, ninst, nact, work, work_bytes, o, st);
}

hipError_t sparse_mc_emit(const SparseMcIn &in, const void *scratch, int64_t ninst, int64_t nact, void *work,
                          size_t work_bytes, const SparseMcOut &o, hipStream_t st) {
    if (in.n == 0 || ninst == 0) return hipSuccess;
    if (mc_work_bytes(ninst, nact) > work_bytes) return hipErrorInvalidValue;
    const CaseScratch c(const_cast<void *>(scratch), in.n, true);
    const RunWork r(work, ninst, nact);
    const unsigned nblk = nb(nact);
    hipLaunchKernelGGL(k_smc_verts, dim3(nblk), dim3(kB), 0, st, in, r.w, (const int64_t *) c.tot,
                       (const longlong2 *) r.pre, o);
    hipLaunchKernelGGL(k_smc_faces, dim3((nblk + 7) / 8 * 8), dim3(kB), 0, st, in, r.w, (const int64_t *) c.tot,
                       (const longlong2 *) r.pre, o);
    ISO_TRY(hipGetLastError());
    ISO_TRY(hipStreamSynchronize(st));
    return hipSuccess;
}

hipError_t sparse_mc(const SparseMcIn &in, int64_t ninst, void *work, size_t work_bytes, SparseMcOut &o,
                     int64_t &nv, int64_t &nf, hipStream_t st) {
    nv = nf = 0;
    if (in.n == 0 || ninst == 0) return hipSuccess;
    if (in.n >= (int64_t) INT32_MAX || ninst >= (int64_t) INT32_MAX) return hipErrorInvalidValue;
    const size_t cb = (sparse_mc_scratch_bytes(in.n) + 255) & ~size_t(255);
    if (cb > work_bytes) return hipErrorInvalidValue;
    cases_pass(in, CaseScratch(work, in.n, true), st);
    // an active cell has at least three crossing edges
    return sparse_mc_run(in, work, ninst, ninst / 3, (char *) work + cb, work_bytes - cb, o, nv, nf, st);
}


}   // namespace iso
