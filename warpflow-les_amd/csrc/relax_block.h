// Several RBGS sweeps of a level per launch, by overlapping blocks.
//
// On levels of up to a few million cells a plane-streaming sweep per launch is a
// chain of a few dependent plane steps, and six such launches follow each
// other: 7 us each at 32^3, where their bytes take less than one.  Here a workgroup takes a block of RI x rj x rk
// cells (its tile plus 2 ns cells on every side that is not a domain face),
// relaxes it ns times on its own and writes the tile; what the block's outer
// cells lack from beyond it moves one cell inward per half-sweep and never
// reaches the tile.
//
// A thread owns the (j, k) column of the block, or RI planes of it: the odd
// cells' values A and the even cells' values E, RI/2 each, and their right-hand
// sides stay in registers for the whole launch, so an update's i neighbours are
// registers.  Blocks that fit the CUs once take four threads a column: a
// half-sweep is then a chain of two updates instead of eight.
// LDS mirrors the block for the j and k neighbours (four reads and one write
// per update): planes of PL words, rows of rk + 1 words whose first word is
// zero (it ends the row before it too) and a row of zeros at either end, so
// nothing is tested at a domain face -- a neighbour beyond it is a zero, as
// in the sweep kernels.  Of two neighbouring lanes one updates a plane of its
// own colour one further up, and PL is a multiple of 32 words, so the lanes of
// a row read distinct banks.
//
// Every update is the sweep kernels' expression on the same operands, so the
// results are theirs bit for bit.
#pragma once
#include "mg_common.h"

namespace wf {

// c0*W + c0*E + c1*S + c1*N + c2*B + c2*T with the fused multiply-adds that the
// sweep kernels' sums contract to
template <class T>
__device__ inline T nb6(T c0, T c1, T c2, T W, T E, T S, T N, T Bt, T Tp) {
  return fma(c2, Tp, fma(c2, Bt, fma(c1, N, fma(c1, S, fma(c0, W, c0 * E)))));
}

// Tiles of one axis of n cells under blocks of r (r <= n) and a halo of h
// cells: the first and the last block end at the domain.
__host__ __device__ inline int relax_block_tiles(int n, int r, int h) {
  return r >= n ? 1 : 1 + (n - r + r - 2 * h - 1) / (r - 2 * h);
}

// The even cells E[t] of a thread (level planes p0 + 2 t of column (j, k), t < NH)
// plus the interpolation of the coarse iterate pc, prolong_body's sum; a lane or
// a plane that is not there (live, p0 + 2 t >= n0) gets zero.
template <class T, int NH>
__device__ inline void add_prolonged(T* E, const T* __restrict__ pc, const MgDev& d, int p0, int j,
                                     int k, bool live) {
  const int n0c = d.n0 / 2, s1 = d.n2 / 2 + 2;
  const int pcb = (d.n1 / 2 + 2) * s1 * (int)sizeof(T);
  const auto dq = buf_rsrc(pc, 0x7fffffffu);
  // array index of the lower of the two coarse planes, rows and columns
  const int u0 = (p0 + 1) >> 1;
  const uint32_t o =
      (uint32_t)((((j + 1) >> 1) * s1 + ((k + 1) >> 1)) * (int)sizeof(T) + u0 * pcb);
  uint32_t oc[4];
#pragma unroll
  for (int c = 0; c < 4; ++c)
    oc[c] = live ? o + (uint32_t)(((c >> 1) * s1 + (c & 1)) * (int)sizeof(T)) : BUF_DEAD;
  const T wx = p0 & 1 ? T(0.75) : T(0.25), wy = j & 1 ? T(0.75) : T(0.25),
          wz = k & 1 ? T(0.75) : T(0.25);
  T w[8];
#pragma unroll
  for (int c = 0; c < 8; ++c)
    w[c] = (c & 4 ? T(1) - wx : wx) * (c & 2 ? T(1) - wy : wy) * (c & 1 ? T(1) - wz : wz);
  constexpr int GP = NH % 4 == 0 ? 4 : NH % 3 == 0 ? 3 : 2;
  static_assert(NH % GP == 0, "whole groups");
#pragma unroll
  for (int g = 0; g < NH; g += GP) {
    T q[GP + 1][4];
#pragma unroll
    for (int u = 0; u <= GP; ++u)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        q[u][c] = buf_ld<T>(dq, u0 + g + u <= n0c + 1 ? oc[c] : BUF_DEAD, (g + u) * pcb);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < GP; ++u) {
      T acc = T(0);
#pragma unroll
      for (int c = 0; c < 8; ++c) acc = fma(w[c], q[u + (c >> 2)][c & 3], acc);
      const T v = E[g + u] + acc;
      E[g + u] = live && p0 + 2 * (g + u) < d.n0 ? v : T(0);
    }
  }
}

// h: the halo the tiles were cut for, at least 2 ns.  NSEG: threads of a column,
// RI planes each (the block has NSEG RI planes).  PART: the level may have fewer
// planes than the block (one block along i then); the planes past it stay zero
// under a zero reciprocal diagonal, kept per cell.  PRO: the iterate is pin plus
// the interpolation of pc.  pout may be pin where one block is the level: the
// barriers after the loads come before any store.
template <class T, int RI, int NSEG, int PL, bool PART, bool PRO = false>
__device__ inline void relax_block_body(const T* pin, T* pout,
                                        const T* __restrict__ rhs, const MgDev& d, T c0, T c1,
                                        T c2, int ns, int h, int rj, int rk, Blk B,
                                        T* __restrict__ sm, const T* __restrict__ pc = nullptr) {
  constexpr int NH = RI / 2;  // cells per colour and thread
  constexpr int SH = NSEG > 1;  // LDS planes before the block
  static_assert(RI % 2 == 0 && PL % 32 == 0, "whole pairs, whole bank rows");
  const int tid = threadIdx.x;
  const int n0 = d.n0, n1 = d.n1, n2 = d.n2;
  // block origin and the tile it writes, along one axis
  auto axis = [&](int b, int n, int r, int& o, int& lo, int& hi) {
    const int st = r - 2 * h;
    o = max(min(b * st, n - r), 0);
    lo = b == 0 ? 0 : b * st + h;
    hi = o + r >= n ? n : (b + 1) * st + h;
  };
  int oi, oj, ok, ilo, ihi, jlo, jhi, klo, khi;
  axis(B.z, n0, RI * NSEG, oi, ilo, ihi);
  axis(B.y, n1, rj, oj, jlo, jhi);
  axis(B.x, n2, rk, ok, klo, khi);
  // lanes past the block update a zero word on zeros and store nothing
  const bool live = tid < rj * rk * NSEG;
  const int seg = NSEG > 1 && live ? tid / (rj * rk) : 0;
  const int cl = live ? tid - seg * (rj * rk) : 0;
  const int jr = cl / rk, kr = cl - jr * rk;
  const int j = oj + jr, k = ok + kr, so = seg * RI;
  const int f = (oi + j + k + 1) & 1;  // the first odd cell is on plane oi + so + f
  const bool fb = f != 0;

  const int pb = (int)(d.s0 * (int64_t)sizeof(T));
  auto rsrc = [&](const T* a) {
    return buf_rsrc(reinterpret_cast<const char*>(a) + (int64_t)oi * pb, 0x7fffffffu);
  };
  const uint32_t col = (uint32_t)(((j + 1) * (int)d.s1 + k + 1) * (int)sizeof(T) + so * pb);
  const uint32_t offA = live ? col + (uint32_t)((1 + f) * pb) : BUF_DEAD;
  const uint32_t offE = live ? col + (uint32_t)((2 - f) * pb) : BUF_DEAD;
  auto in = [&](int p, uint32_t o) { return !PART || so + p < n0 ? o : BUF_DEAD; };
  T A[NH], E[NH], ra[NH], re[NH];
  {  // the first half-sweep writes every odd cell: only the even ones are read
    const auto dp = pin ? rsrc(pin) : buf_rsrc(rhs, 0u);  // nullptr: an iterate of zeros
    const auto dr = rsrc(rhs);
#pragma unroll
    for (int t = 0; t < NH; ++t) E[t] = buf_ld<T>(dp, in(2 * t + 1 - f, offE), 2 * t * pb);
#pragma unroll
    for (int t = 0; t < NH; ++t) ra[t] = buf_ld<T>(dr, in(2 * t + f, offA), 2 * t * pb);
#pragma unroll
    for (int t = 0; t < NH; ++t) re[t] = buf_ld<T>(dr, in(2 * t + 1 - f, offE), 2 * t * pb);
  }
  // reciprocal diagonals: interior planes, and the planes at the i faces
  T ri = T(0), rf = T(0);
  if (live) {
    ri = T(1) / mg_coef(d, 1, j, k, c0, c1, c2).ap;
    rf = T(1) / mg_coef(d, 0, j, k, c0, c1, c2).ap;
  }
  const bool flo = oi + so == 0, fhi = oi + so + RI >= n0;
  // 1/ap of the odd and even cells: one value but for the first and last cell,
  // or (PART) one per cell
  constexpr int NR = PART ? NH : 3;
  T rpA[NR], rpE[NR];
  if constexpr (PART) {
#pragma unroll
    for (int t = 0; t < NH; ++t) {
      const int pa = so + 2 * t + f, pe = so + 2 * t + 1 - f;
      rpA[t] = pa >= n0 ? T(0) : pa == 0 || pa == n0 - 1 ? rf : ri;
      rpE[t] = pe >= n0 ? T(0) : pe == 0 || pe == n0 - 1 ? rf : ri;
    }
  } else {
    rpA[0] = flo && !fb ? rf : ri;
    rpE[0] = flo && fb ? rf : ri;
    rpA[1] = rpE[1] = ri;
    rpA[2] = fhi && fb ? rf : ri;
    rpE[2] = fhi && !fb ? rf : ri;
  }

  const int pitch = rk + 1;
  const int wc = live ? (jr + 1) * pitch + kr + 1 : 1;  // this column's word
  const int wq = live ? pitch : 0;                      // one row on
  {  // zero words around the block: all of LDS is cleared, the loads above in flight
    using V4 = __attribute__((ext_vector_type(4))) unsigned;
    constexpr int NV = (RI * NSEG + 2 * SH) * PL * (int)sizeof(T) / 16;
    V4* const z = reinterpret_cast<V4*>(sm);
    for (int w = tid; w < NV; w += (int)blockDim.x) z[w] = V4{0u, 0u, 0u, 0u};
  }
  T* const lA = sm + (so + SH + f) * PL + wc;      // LDS words of the odd cells: lA[2 t PL]
  T* const lE = sm + (so + SH + 1 - f) * PL + wc;  // and of the even ones
  if constexpr (PRO) add_prolonged<T, NH>(E, pc, d, oi + so + 1 - f, j, k, live);
  __syncthreads();
#pragma unroll
  for (int t = 0; t < NH; ++t) lE[2 * t * PL] = E[t];
  __syncthreads();

  // One half-sweep: X from its own column's other colour Y (plane before / after:
  // Y[t-1], Y[t] on lanes where up is false, Y[t], Y[t+1] where it is true; from
  // LDS past a segment's end) and the LDS rows.  The reads of G updates are in flight before the previous G
  // are formed; without that the compiler waits for each update's four.
  constexpr int G = sizeof(T) == 4 && NH % 4 == 0 ? 4 : NH % 3 == 0 ? 3 : 2;
  static_assert(NH % G == 0, "whole groups");
  auto half = [&](T* X, const T* Y, const T* rv, T* l, bool up, const T* rp) {
    T nb[2][G][4];
    T ye = T(0);
    if constexpr (NSEG > 1) ye = up ? l[(2 * NH - 1) * PL] : l[-PL];
    auto fetch = [&](int g, int b) {
#pragma unroll
      for (int e = 0; e < G; ++e) {
        const T* q = l + 2 * (g * G + e) * PL;
        nb[b][e][0] = q[-wq];
        nb[b][e][1] = q[wq];
        nb[b][e][2] = q[-1];
        nb[b][e][3] = q[1];
      }
    };
    fetch(0, 0);
#pragma unroll
    for (int g = 0; g < NH / G; ++g) {
      if (g + 1 < NH / G) fetch(g + 1, (g + 1) & 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < G; ++e) {
        const int t = g * G + e;
        const T yb = t > 0 ? Y[t > 0 ? t - 1 : 0] : ye;
        const T ya = t + 1 < NH ? Y[t + 1 < NH ? t + 1 : 0] : ye;
        const T* v = nb[g & 1][e];
        const T sum = nb6(c0, c1, c2, up ? Y[t] : yb, up ? ya : Y[t], v[0], v[1], v[2], v[3]);
        X[t] = (rv[t] - sum) * rp[PART ? t : t == 0 ? 0 : t == NH - 1 ? 2 : 1];
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  for (int s = 0; s < ns; ++s) {
    half(A, E, ra, lA, fb, rpA);
#pragma unroll
    for (int t = 0; t < NH; ++t) lA[2 * t * PL] = A[t];
    __syncthreads();
    half(E, A, re, lE, !fb, rpE);
    if (s + 1 < ns) {
#pragma unroll
      for (int t = 0; t < NH; ++t) lE[2 * t * PL] = E[t];
      __syncthreads();
    }
  }

  // the tile, and its images on the face ring
  const auto dout = rsrc(pout);
  const bool own = live && j >= jlo && j < jhi && k >= klo && k < khi;
  if (!own) return;
  const int a = ilo - oi - so, b = ihi - oi - so;  // planes of the segment to write
  const bool jf = j == 0 || j == n1 - 1, kf = k == 0 || k == n2 - 1;
  const uint32_t sj = j == 0 ? 0u - (uint32_t)((int)d.s1 * (int)sizeof(T))
                             : (uint32_t)((int)d.s1 * (int)sizeof(T));
  const uint32_t sk = k == 0 ? 0u - (uint32_t)sizeof(T) : (uint32_t)sizeof(T);
  auto put = [&](uint32_t by) {
#pragma unroll
    for (int t = 0; t < NH; ++t) {
      const int pa = 2 * t + f, pe = 2 * t + 1 - f;
      buf_st(dout, pa >= a && pa < b ? offA + by : BUF_DEAD, 2 * t * pb, A[t]);
      buf_st(dout, pe >= a && pe < b ? offE + by : BUF_DEAD, 2 * t * pb, E[t]);
    }
  };
  put(0u);
  if (jf) put(sj);
  if (kf) put(sk);
  if (flo) buf_st(dout, col, 0, fb ? E[0] : A[0]);
  if constexpr (PART) {
#pragma unroll
    for (int t = 0; t < NH; ++t) {
      const int pa = 2 * t + f, pe = 2 * t + 1 - f;
      if (so + pa == n0 - 1) buf_st(dout, offA, (2 * t + 1) * pb, A[t]);
      if (so + pe == n0 - 1) buf_st(dout, offE, (2 * t + 1) * pb, E[t]);
    }
  } else if (fhi) {
    buf_st(dout, col, (RI + 1) * pb, fb ? A[NH - 1] : E[NH - 1]);
  }
}

}  // namespace wf
