// Backward of marching cubes: vertex-position gradients -> grid values.
//
// A vertex on the edge from point a (value va, position Pa) to point b is
// v = (1 - t) Pa + t Pb with t = (L - va) / (vb - va) (src/mc/nagae.cu:55-59).
// Hence dv/dva = (Pb - Pa) (L - vb) / (vb - va)^2 and
//       dv/dvb = -(Pb - Pa) (L - va) / (vb - va)^2.
// A welded vertex takes its position from one representative edge, so its
// gradient goes to that edge's two values.  Accumulation uses float atomics
// (a grid value is shared by up to six edges).

#include "backward.h"
#include "common.h"

namespace iso {

namespace {

constexpr int kB = 256;

__device__ __forceinline__ void edge_grad(const float *g, float va, float vb, float level, const float pa[3],
                                          const float pb[3], float &ga, float &gb) {
    float d = vb - va;
    ga = gb = 0.0f;
    if (!(d != 0.0f)) return;
    float s = g[0] * (pb[0] - pa[0]) + g[1] * (pb[1] - pa[1]) + g[2] * (pb[2] - pa[2]);
    float inv2 = 1.0f / (d * d);
    ga = s * (level - vb) * inv2;
    gb = -s * (level - va) * inv2;
    if (!isfinite(ga)) ga = 0.0f;
    if (!isfinite(gb)) gb = 0.0f;
}

__global__ void k_bwd_dense(const float *grad_v, const int64_t *keys, int64_t nv, const float *values,
                            DenseGeom g, float level, float *grad_values) {
    int64_t i = (int64_t) blockIdx.x * kB + threadIdx.x;
    if (i >= nv) return;
    int64_t key = keys[i];
    const int64_t p = div_fast(key, 3);
    const int axis = (int) (key - 3 * p);
    const int64_t r = div_fast(p, g.Z), z = p - r * g.Z;
    const int64_t x = div_fast(r, g.Y), y = r - x * g.Y;
    int64_t stride = axis == 0 ? g.Y * g.Z : (axis == 1 ? g.Z : 1);
    int64_t q = p + stride;
    float pa[3] = {grid_coord(x, g.X, g.amin[0], g.amax[0]), grid_coord(y, g.Y, g.amin[1], g.amax[1]),
                   grid_coord(z, g.Z, g.amin[2], g.amax[2])};
    float pb[3] = {pa[0], pa[1], pa[2]};
    if (axis == 0) pb[0] = grid_coord(x + 1, g.X, g.amin[0], g.amax[0]);
    if (axis == 1) pb[1] = grid_coord(y + 1, g.Y, g.amin[1], g.amax[1]);
    if (axis == 2) pb[2] = grid_coord(z + 1, g.Z, g.amin[2], g.amax[2]);
    float ga, gb;
    edge_grad(grad_v + 3 * i, values[p], values[q], level, pa, pb, ga, gb);
    if (ga != 0.0f) atomicAdd(&grad_values[p], ga);
    if (gb != 0.0f) atomicAdd(&grad_values[q], gb);
}


__global__ void k_bwd_sparse(const float *grad_v, const int64_t *vsrc, int64_t nv, const float *values,
                             const int64_t *ids, DenseGeom g, float level, float *grad_values) {
    int64_t i = (int64_t) blockIdx.x * kB + threadIdx.x;
    if (i >= nv) return;
    int64_t src = vsrc[i];
    const int64_t slot = div_fast(src, 12);
    const int e = (int) (src - 12 * slot);
    const int64_t id = ids[slot];
    const int64_t cz = g.Z - 1, cy = g.Y - 1;
    const int64_t r = div_fast(id, cz), z = id - r * cz;
    const int64_t x = div_fast(r, cy), y = r - x * cy;
    int ca = edge_a(e), cb = edge_b(e);
    float pa[3] = {grid_coord(x + (ca >> 2), g.X, g.amin[0], g.amax[0]),
                   grid_coord(y + ((ca >> 1) & 1), g.Y, g.amin[1], g.amax[1]),
                   grid_coord(z + (ca & 1), g.Z, g.amin[2], g.amax[2])};
    float pb[3] = {grid_coord(x + (cb >> 2), g.X, g.amin[0], g.amax[0]),
                   grid_coord(y + ((cb >> 1) & 1), g.Y, g.amin[1], g.amax[1]),
                   grid_coord(z + (cb & 1), g.Z, g.amin[2], g.amax[2])};
    float ga, gb;
    edge_grad(grad_v + 3 * i, values[8 * slot + ca], values[8 * slot + cb], level, pa, pb, ga, gb);
    if (ga != 0.0f) atomicAdd(&grad_values[8 * slot + ca], ga);
    if (gb != 0.0f) atomicAdd(&grad_values[8 * slot + cb], gb);
}

// A workgroup owns kRows rows of the gradient: its vertices are one run of
// the ascending vsrc, and a row's vertices (its cell's representatives) are
// consecutive, so the first of them adds up the row in LDS without atomics,
// and every row leaves as one coalesced write.  Bound by that write (32 B a
// cell); with the derivatives from the forward pass the vertices' values and
// ids, scattered over most lines of the grid's arrays, are not read again.
// A scatter by atomics into a cleared array touches nearly every line of it
// three times: 0.66 ms and 0.12 ms for the clearing at 25.7 M cells and 9.7 M
// vertices, against 0.21 ms (1.09 GB, 5.2 TB/s) and 0.03 ms for the runs.
// kRows 1024 (a longer chain per workgroup, half the wavefronts): 0.32 ms.
constexpr int kRows = 512;

// The runs' bounds, left in the first row that each workgroup will write
// (found by one lane each: a search inside the workgroup costs it a chain of
// loads, and a wave-wide one fetched as many lines as the vertices take).
__global__ void __launch_bounds__(64) k_bwd_sparse_runs(const int64_t *vsrc, int64_t nv, int64_t n,
                                                        float *grad_values) {
    const int64_t b = (int64_t) blockIdx.x * 63 + threadIdx.x, s0 = b * kRows;
    int64_t r[2];   // a run ends where the next lane's begins: 63 runs a wave
    r[0] = lower_bound8(vsrc, nv, 12 * s0);
    r[1] = __shfl_down(r[0], 1);
    if (threadIdx.x == 63 || s0 >= n) return;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        grad_values[8 * s0 + k] = __int_as_float((int) (r[k >> 1] >> (32 * (k & 1))));
}

__global__ void __launch_bounds__(kB) k_bwd_sparse_rows(const float *grad_v, const int64_t *vsrc, const float2 *vjac,
                                                        int64_t n, float *grad_values) {
    __shared__ float row[8 * kRows];
    const int64_t s0 = (int64_t) blockIdx.x * kRows;
    const int tid = threadIdx.x;
    uint32_t r4[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) r4[k] = (uint32_t) __float_as_int(grad_values[8 * s0 + k]);
    const int64_t lo = (int64_t) ((uint64_t) r4[1] << 32 | r4[0]), hi = (int64_t) ((uint64_t) r4[3] << 32 | r4[2]);
    for (int k = tid; k < 8 * kRows; k += kB) row[k] = 0.0f;
    __syncthreads();
    for (int64_t i = lo + tid; i < hi; i += kB) {
        int src = (int) (vsrc[i] - 12 * s0);
        const int r = src / 12;
        if (i > lo && (int) (vsrc[i - 1] - 12 * s0) / 12 == r) continue;   // not its row's first
        for (int64_t j = i;;) {
            const int e = src - 12 * r, ax = edge_axis(e);
            const float g[3] = {grad_v[3 * j], grad_v[3 * j + 1], grad_v[3 * j + 2]};
            // the edge is along one axis; a gradient that is not finite anywhere counts for nothing
            const float s = (ax == 0 ? g[0] : (ax == 1 ? g[1] : g[2])) + (0.0f * g[0] + 0.0f * g[1] + 0.0f * g[2]);
            const float2 d = vjac[j];
            const float ga = s * d.x, gb = s * d.y;
            if (isfinite(ga)) row[8 * r + edge_a(e)] += ga;
            if (isfinite(gb)) row[8 * r + edge_b(e)] += gb;
            if (++j >= hi) break;
            src = (int) (vsrc[j] - 12 * s0);
            if (src / 12 != r) break;
        }
    }
    __syncthreads();
    float *out = grad_values + 8 * s0;
    const int m = (int) min<int64_t>(kRows, n - s0) * 8;
    for (int k = tid; k < m; k += kB) __builtin_nontemporal_store(row[k], out + k);
}

}   // namespace

hipError_t mc_backward_dense(const float *grad_v, const int64_t *keys, int64_t nv, const float *values,
                             const DenseGeom &g, float level, float *grad_values, hipStream_t st) {
    if (nv == 0) return hipSuccess;
    hipLaunchKernelGGL(k_bwd_dense, dim3((unsigned) ((nv + kB - 1) / kB)), dim3(kB), 0, st, grad_v, keys, nv, values,
                       g, level, grad_values);
    return hipGetLastError();
}

hipError_t mc_backward_sparse(const float *grad_v, const int64_t *vsrc, int64_t nv, const float *values,
                              const int64_t *ids, const DenseGeom &g, float level, float *grad_values,
                              hipStream_t st) {
    if (nv == 0) return hipSuccess;
    hipLaunchKernelGGL(k_bwd_sparse, dim3((unsigned) ((nv + kB - 1) / kB)), dim3(kB), 0, st, grad_v, vsrc, nv,
                       values, ids, g, level, grad_values);
    return hipGetLastError();
}

hipError_t mc_backward_sparse_rows(const float *grad_v, const int64_t *vsrc, const float2 *vjac, int64_t nv, int64_t n,
                                   float *grad_values, hipStream_t st) {
    const int64_t nblk = (n + kRows - 1) / kRows;
    hipLaunchKernelGGL(k_bwd_sparse_runs, dim3((unsigned) ((nblk + 62) / 63)), dim3(64), 0, st, vsrc, nv, n, grad_values);
    hipLaunchKernelGGL(k_bwd_sparse_rows, dim3((unsigned) nblk), dim3(kB), 0, st, grad_v, vsrc, vjac, n, grad_values);
    return hipGetLastError();
}

}   // namespace iso
