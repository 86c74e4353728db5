#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "common.h"

namespace iso {

struct SparseGeom {
    int64_t X, Y, Z;   // points per axis
    float amin[3], amax[3];
};

// Reciprocals of the cells per axis; ncell = 0: not used.
struct SparseDiv {
    double inv_cz = 0.0;
    UDiv32 cy;
    int64_t ncell = 0;
};

struct SparseMcIn {
    const float *values;   // (n, 8)
    const int64_t *ids;    // (n) dense cell ids
    int64_t n;
    SparseGeom g;
    float level;
    int method;
    float cand_eps;   // bound on t (or 1 - t) of a vertex within 16 ulps of a grid point
    SparseDiv div;
};

// Active cells (in id order) and crossing-edge instances (cell by cell, in
// edge order) of a run.
struct SparseMcWork {
    int64_t *aid;      // per active cell: dense cell id
    int32_t *aslot;    // its slot
    uint2 *ainfo;      // its first instance; case, special flag, crossing edges
    uint32_t *ares;    // edges that represent themselves, kept faces, special flag
    uint32_t *alook;   // edges whose vertex may lie near a grid point
    int4 *acol;        // of those with such an edge: places in the list of columns (-1, -1), (-1, 0), (-1, 1), (0, -1)
    int32_t *win;      // per workgroup: the runs of active cells its cells' lower neighbours are in
    int64_t *bid;      // first id of each workgroup's active cells
    int32_t *rkey;     // per instance: its representative (first instance at its position)
    int32_t *vid;      // vertex id of a representative
    uint8_t *used;     // special cells: the representative is a corner of a kept face
};

struct SparseMcOut {
    float *v;
    int64_t cap_v;
    int32_t *f;
    int64_t cap_f;
    int64_t *vsrc;   // optional: slot * 12 + edge of each output vertex
    float2 *vjac = nullptr;   // optional: derivatives of its coordinate along the edge by the edge's end values
};

hipError_t sparse_corner_points(const int64_t *ids, int64_t n, const SparseGeom &g, float *out, hipStream_t st);
// Sorted-key set operations of the population path: union of sorted unique a
// with sorted b (duplicates allowed), or a minus b.  out (capacity na + nb /
// na) receives the sorted result, slot[k] the index in a of out[k] (-1 for a
// key new from b), *n_out (device) its length.  No host synchronisation.
int64_t sparse_setop_scratch_bytes(int64_t na, int64_t nb);
hipError_t sparse_setop(const int64_t *a, int64_t na, const int64_t *b, int64_t nb, bool difference, void *scratch,
                        int64_t *out, int64_t *slot, int64_t *n_out, hipStream_t st);
// out row k = old_values row slot[k], or dflt where slot[k] < 0 (8 floats a row).
hipError_t sparse_gather_rows(const float *old_values, const int64_t *slot, int64_t n, float dflt, float *out,
                              hipStream_t st);
hipError_t sparse_crossing_flags(const float *values, int64_t n, float level, uint8_t *flags, hipStream_t st);
// Marching cubes in two steps: the cases of all cells (scratch of
// sparse_mc_scratch_bytes(n), kept for the second step; synchronises for the
// counts), then the run (work of sparse_mc_run_bytes; synchronises for the
// mesh sizes).
size_t sparse_mc_scratch_bytes(int64_t n);
size_t sparse_mc_run_bytes(int64_t ninst, int64_t nact);
hipError_t sparse_mc_cases(const SparseMcIn &in, void *scratch, int64_t &ninst, int64_t &nact, hipStream_t st);
hipError_t sparse_mc_run(const SparseMcIn &in, const void *scratch, int64_t ninst, int64_t nact, void *work,
                         size_t work_bytes, SparseMcOut &o, int64_t &nv, int64_t &nf, hipStream_t st);
// Vertices and faces of a run that found too little room for them (nothing in
// between): o has room for the sizes it returned.
hipError_t sparse_mc_emit(const SparseMcIn &in, const void *scratch, int64_t ninst, int64_t nact, void *work,
                          size_t work_bytes, const SparseMcOut &o, hipStream_t st);
// Both steps with nothing kept between the count and the run (the cases are
// found twice): scratch of the count 8 * (n / 256 + 16) bytes.
size_t sparse_mc_work_bytes(int64_t n, int64_t ninst);
hipError_t sparse_mc_count(const SparseMcIn &in, int64_t *scratch, int64_t &ninst, hipStream_t st);
hipError_t sparse_mc(const SparseMcIn &in, int64_t ninst, void *work, size_t work_bytes, SparseMcOut &o,
                     int64_t &nv, int64_t &nf, hipStream_t st);

}   // namespace iso
