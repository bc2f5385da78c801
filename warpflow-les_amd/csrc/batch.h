// Ensemble (batched) execution: many independent cavities of different
// sizes advanced by one launch per operator.
//
// Every field of every member lives in one pool per field name (member m's
// (n0+6)(n1+6)(n2+6) array at element offset off); every multigrid level l
// in one pool per level array (member m's (n_l+2)^3 array at loff[l]).  A
// batched launch covers a list of work items -- (member, block coordinates),
// numbered member after member -- and runs the single-domain kernel body on
// them, so both paths run the same arithmetic.  The passes over whole fields and
// levels launch a workgroup per entry of a table made at creation; the others
// are a grid-stride loop of at most the workgroups the device holds at once,
// which finds an item's member by search, or a workgroup per member.
// A per-member `active` mask (nullable) lets converged members skip the
// projection iterations of the others inside one captured graph.
#pragma once
#include <vector>

#include "wf_common.h"

namespace wf {

constexpr int BATCH_MAX_LEVELS = 8;

// Device view of one member, derived from wf_member by wf_batch_create.
struct MemDev {
  wf_grid g;  // field geometry, 3 ghost layers
  int64_t off;
  double dx, dy, dz, rey, ulid, noise, dt;
  double ls;    // WALE length scale cw * delta
  double rsum;  // 1/dx^2 + 1/dy^2 + 1/dz^2 (the checkdt viscous limit)
  // 1/h, 1/h^2, 1/(24 h), 1/(12 h h) of each axis and 1/dt, formed here so that no
  // workgroup opens with a chain of FP64 divisions
  double r1[3], r2[3], r24[3], ir12[3], rdt;
  uint32_t seed;
  int nlev;
  int ln[BATCH_MAX_LEVELS][3];
  int64_t loff[BATCH_MAX_LEVELS];
  float lc[BATCH_MAX_LEVELS][3];  // 1/h^2 of each level, as the single-domain path forms it
  int64_t coff;  // coarse-operator offset (elements) in the operator pool
  int red0;      // first reduction-partial slot of this member
  int sum0;      // first sum-partial slot of this member
};

constexpr int BATCH_ICH = 4;  // most planes per item of the element passes

// A work-item list: start[m] .. start[m+1]-1 are member m's items.
struct Plan {
  const int* start;
  const int4* item;  // kinds with a tile shape (plan_tile): (member, k tile, j tile, chunk)
  int total;
  int grid;  // workgroups launched by the grid-stride kinds (<= total)
  int ich;   // i-planes per item
};

struct BView {
  const MemDev* mem;
  int nmem;
};

// Member m's part of the outer loop's break test (solver.py:185-197).
__device__ inline void loop_test(int m, double r, double eps, int it, int* __restrict__ active,
                                 int* __restrict__ iters, int* __restrict__ status) {
  iters[m] = it;
  const bool diverged = !(r <= 10.0), leaves = diverged || (r < eps && it > 1);
  if (diverged && !(r < eps && it > 1)) status[m] = 1;
  active[m] = leaves ? 0 : 1;
}

// Largest m with start[m] <= w (start[0] = 0, start[nmem] = total > w).
__device__ inline int member_of(const int* __restrict__ start, int nmem, int w) {
  int lo = 0, hi = nmem;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (start[mid] <= w)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

// Block coordinates of local block q of a 64 x 4 (k, j) x plane launch over
// a box of extent (d0, d1, d2): the box_grid order (x fastest).
__host__ __device__ inline int cells_blocks(int d0, int d1, int d2) {
  return ((d2 + 63) / 64) * ((d1 + 3) / 4) * d0;
}
__device__ inline Blk cells_blk(int q, int d1, int d2) {
  const int nx = (d2 + 63) / 64, ny = (d1 + 3) / 4;
  return Blk{q % nx, (q / nx) % ny, q / (nx * ny)};
}

// Reduction items: 64 x 4 (k, j) tiles x i-chunks of ich planes.
__host__ __device__ inline int red_blocks(int d0, int d1, int d2, int ich) {
  return ((d2 + 63) / 64) * ((d1 + 3) / 4) * ((d0 + ich - 1) / ich);
}

// Work-item counts per member for each kind of batched launch.
enum PlanKind : int {
  PK_CELLS = 0,     // 64x4 tiles x ich planes over the real cells
  PK_RING,          // 64x4 blocks over real cells + 1 ring layer
  PK_RED,           // reduction tiles over the real cells
  PK_CD0,           // convdiff tiles, components u, v, w
  PK_CD1,
  PK_CD2,
  PK_MOM,           // 8 x 32 (j, k) tiles x ich planes over the real cells: the
                    // three-component conv+diff passes
  PK_STREAM,        // the same tiles, other chunks: WALE and calvel3_calmas
  PK_CDE,           // u's edge planes 0 and ni-2: 8 x 32 (j, k) tiles x 2
  PK_XG,            // w's cross-ghost cells of each real plane, 256 per item
  PK_COP,           // 32-row blocks of the coarsest level's operator
  PK_LCELLS0,       // 64x4 tiles over single planes of level l, l = 0 .. 7
  PK_COUNT = PK_LCELLS0 + BATCH_MAX_LEVELS
};

// The workgroup's entry of a plan with a table.  Nothing is searched or divided
// before its loads: the grid-stride form's member search (a chain of six
// dependent loads per 64 x 4 block) took half the time of a light field pass
// (pp -= mean over 12.1 M cells: 75 us with it, 35 without).
__device__ inline int4 plan_item(const Plan& P, int& w) {
  w = xcd_linear(blockIdx.x, gridDim.x);
  return P.item[w];
}
// f(member index, member, block) for every plane of the workgroup's item of a
// 64 x 4 plan over n0(member) planes.
template <class F>
__device__ inline void item_planes(const Plan& P, const BView& V, const int* active, F&& f) {
  int w;
  const int4 it = plan_item(P, w);
  if (active && !active[it.x]) return;  // uniform per workgroup
  const MemDev& M = V.mem[it.x];
  const int i1 = min(it.w * P.ich + P.ich, M.g.ni);
  for (int i = it.w * P.ich; i < i1; ++i) f(it.x, M, Blk{it.y, it.z, i});
}

// How a level of every member relaxes: one workgroup per item (member, block
// coordinates x, y, z) of a table made at creation.
struct BatchRelax {
  const int4* item = nullptr;  // device
  int total = 0;
  bool single = false;  // every member is one block: all sweeps in one launch, in place
  int rjk = 0, ns = 0;  // blocks: rows and columns, sweeps per launch
  int ich = 0;          // > 0: two-sweep launches in chunks of ich planes instead
  double us = 0;        // estimate of a launch
};

// Host side of a batch (defined in batch.hip).
struct Batch {
  int nmem = 0, nlev = 0;
  MemDev* mem_dev = nullptr;        // nmem descriptors (device)
  MemDev* mem_host = nullptr;       // host copy
  Plan plan[PK_COUNT];
  int* plan_mem[PK_COUNT] = {};     // device start arrays
  BatchRelax relax[BATCH_MAX_LEVELS];
  void* bc_fill = nullptr;          // ghost fills of every member (device; bcs.hip)
  int2 *bc_x = nullptr, *bc_yz = nullptr;  // their items: (member, first x line), (member, plane)
  int bc_nx = 0, bc_nyz = 0;
  double* red_part = nullptr;       // 4 * nred reduction partials (device)
  int nred = 0;
  double* sum_part = nullptr;       // nsum sum partials (device)
  int nsum = 0;
  double* scal = nullptr;           // 4 * nmem scalars (device): means, maxima
  int64_t field_elems = 0;
  int64_t level_elems[BATCH_MAX_LEVELS] = {};
  int64_t cop_elems = 0;
  int max_lds_cells[BATCH_MAX_LEVELS] = {};
  BView view() const { return BView{mem_dev, nmem}; }
};

// Convdiff tiles (8 x 32 (j, k) tiles x i-chunks): shared with convdiff.hip.
__host__ __device__ inline int cd_tiles(int d0, int d1, int d2, int ich) {
  return ((d2 + 31) / 32) * ((d1 + 7) / 8) * ((d0 + ich - 1) / ich);
}
// Operator box of component c over n0 x n1 x n2 cells (solver.py:99-110).
__host__ __device__ inline void op_dims(int c, int n0, int n1, int n2, int& d0, int& d1,
                                        int& d2) {
  d0 = n0 - (c == 0);
  d1 = n1 - (c == 1);
  d2 = n2 - (c == 2);
}
// The outer loop's break test of iteration it (> 0) in the projection's fold:
// each member that takes part records iters[m] = it and leaves the loop when
// rmax[m] < eps and it > 1, or, with status[m] = 1, when rmax[m] > 10 or NaN.
// it = 1 starts the loop: every member takes part.
struct BatchTest {
  int it = 0;
  double eps = 0.0;
  int *active = nullptr, *iters = nullptr, *status = nullptr;
};

// Batched launchers, one per source file (argument checks done by the C ABI).
int batch_noise(const Batch& B, double* u, double* v, double* w, hipStream_t s);
int batch_fill_vis(const Batch& B, double* vis, hipStream_t s);
int batch_wale(const Batch& B, const double* u, const double* v, const double* w, double* vis,
               hipStream_t s);
int batch_checkdt(const Batch& B, const double* u, const double* v, const double* w,
                  const double* vis, double* out4, hipStream_t s);
int batch_wale_checkdt(const Batch& B, const double* u, const double* v, const double* w,
                       double* vis, double* out4, hipStream_t s);
int batch_calvel3(const Batch& B, const double* us, const double* vs, const double* ws,
                  const double* p, double* u, double* v, double* w, double alpha,
                  const int* active, hipStream_t s);
int batch_calmas(const Batch& B, const double* u, const double* v, const double* w, double* su,
                 double* rmax, const int* active, hipStream_t s);
int batch_calvel3_calmas(const Batch& B, const double* us, const double* vs, const double* ws,
                         const double* p, double* u, double* v, double* w, double* su,
                         double* rmax, double alpha, float* r32, const int* active,
                         hipStream_t s, const BatchTest& test = BatchTest{});
int batch_add_ring(const Batch& B, double* p, const double* pp, const int* active,
                   hipStream_t s);
int batch_convdiff(const Batch& B, int comp, const double* u, const double* v,
                   const double* w, const double* coo, const double* vis, double* cstar,
                   double alpha, hipStream_t s, double* coo_save = nullptr);
// The three-component conv+diff passes of the two RK stages (convdiff3_save_
// kernel, convdiff3_kernel), u's edge-plane pass and w's cross-ghost copy, for
// every member (convdiff.hip).
int batch_convdiff3(const Batch& B, const double* u, const double* v, const double* w,
                    const double* vis, const double* wpre, double* us, double* vs, double* ws,
                    double* uoo, double* voo, double* woo, double alpha, hipStream_t s);
int batch_convdiff_u_edges(const Batch& B, const double* u, const double* v, const double* w,
                           const double* uoo, const double* vis, double* us, double alpha,
                           hipStream_t s);
int batch_save_cross_ghosts(const Batch& B, const double* w, double* wpre, hipStream_t s);
int batch_bc_fill(const Batch& B, double* f, int which, const int* active, hipStream_t s);
int batch_bc_fill_n(const Batch& B, double* const* f, const int* which, int nf, bool edges,
                    const int* active, hipStream_t s);
int batch_bc_init(Batch& B);
int batch_vcycle(const Batch& B, float* const* phi, float* const* rhs, float* const* tmp,
                 const float* cop, int npre, int npost, int ncoarse, const int* active,
                 hipStream_t s, bool zero0);
int batch_mg_init();
void batch_relax_plan(const MemDev* mem, int nmem, int l, BatchRelax& P,
                      std::vector<int4>& items);
int batch_mg_mixed(const Batch& B, float* const* phi, float* const* rhs, float* const* tmp,
                   const float* cop, const double* su, double* pp, int ncycles, int npre,
                   int npost, int ncoarse, int flags, const int* active, hipStream_t s);
int batch_mg_correct(const Batch& B, float* const* phi, float* const* rhs, float* const* tmp,
                     const float* cop, const double* su, double* pp, double* p, int ncycles,
                     int npre, int npost, int ncoarse, int flags, const int* active,
                     hipStream_t s);

}  // namespace wf
