// V-cycle legs over the levels that one workgroup holds.
//
// At 16^3 cells and below a level's launches take 4 to 10 us each whatever their
// work, and every launch waits for the one before.  Here one workgroup takes a
// leg of the cycle over all such levels: down, each level's sweeps and the
// restriction of its residual, and up, each level's prolongation and sweeps; the
// iterates pass from leg to leg in the levels' arrays.
//
// A level's cells sit in registers as in relax_block.h: a thread owns WG_RI
// planes of a (j, k) column, odd cells A and even cells E with their right-hand
// sides, and LDS mirrors the level (planes of WG_PL words, zero words and planes
// beyond every face) for the neighbours in other columns and segments.  A
// half-sweep is a chain of two updates (0.3 us at 16^3 in FP64; a column per
// thread: eight, 0.45 us).  Six sweeps and a transfer take 8 us at 12^3 and 11 us
// at 16^3, about 7 of them the launch and the first loads; as launches of their
// own the sweeps took 9.7 and the transfer 4.5.
// Levels of more than 1024 such threads stay with the blocks: one CU's vector
// units and LDS ports bound them (24^3 in FP64, 24 planes a thread: 3 us per
// half-sweep, 55 us for a leg whose launches took 30).
//
// Updates, residuals, restriction and prolongation are the level kernels'
// expressions on the same operands in the same order.
#pragma once
#include "relax_block.h"

namespace wf {

constexpr int WG_RI = 4, WG_PL = 320, WG_THREADS = 1024;
__host__ __device__ inline int wg_threads(int n0, int n1, int n2) {
  return n1 * n2 * ((n0 + WG_RI - 1) / WG_RI);
}
inline bool wg_fits(int n0, int n1, int n2) {
  return n0 <= 16 && (n1 + 2) * ((int64_t)n2 + 1) + 1 <= WG_PL &&
         wg_threads(n0, n1, n2) <= WG_THREADS;
}
inline int wg_lds(int n0, int elem) { return ((n0 + WG_RI - 1) / WG_RI * WG_RI + 2) * WG_PL * elem; }

// One level; down: rc = coarse right-hand side, up: pc = coarse iterate.  zero:
// the iterate is zero, unread.  PART: n0 is no multiple of WG_RI (the planes
// past it stay zero under a zero reciprocal diagonal).
template <class T, bool PART, bool UP>
__device__ inline void wg_level(T* __restrict__ phi, const T* __restrict__ rhs, const MgDev& d,
                                T c0, T c1, T c2, int ns, bool zero, const T* __restrict__ pc,
                                T* __restrict__ rc, T* __restrict__ sm) {
  constexpr int RI = WG_RI, PL = WG_PL, NH = RI / 2;
  const int tid = threadIdx.x;
  const int n0 = d.n0, n1 = d.n1, n2 = d.n2, ncol = n1 * n2;
  const int nseg = (n0 + RI - 1) / RI;
  const int seg = tid / ncol;
  const bool live = tid < ncol * nseg;
  const bool work = (tid & ~63) < ncol * nseg;  // waves without a live lane only wait
  const int col = live ? tid - seg * ncol : 0;
  const int j = col / n2, k = col - j * n2, oi = live ? seg * RI : 0;
  const int f = (j + k + 1) & 1;  // the first odd cell is on plane oi + f
  const bool fb = f != 0;
  MgDev dc;
  dc.n0 = n0 / 2;
  dc.n1 = n1 / 2;
  dc.n2 = n2 / 2;
  dc.s1 = dc.n2 + 2;
  dc.s0 = (int64_t)(dc.n1 + 2) * dc.s1;

  const int pb = (int)(d.s0 * (int64_t)sizeof(T));
  const uint32_t cb = (uint32_t)(((j + 1) * (int)d.s1 + k + 1) * (int)sizeof(T) + oi * pb);
  const uint32_t offA = live ? cb + (uint32_t)((1 + f) * pb) : BUF_DEAD;
  const uint32_t offE = live ? cb + (uint32_t)((2 - f) * pb) : BUF_DEAD;
  auto in = [&](int p, uint32_t o) { return !PART || oi + p < n0 ? o : BUF_DEAD; };
  T A[NH], E[NH], ra[NH], re[NH];
  T ri = T(0), rf = T(0), api = T(0), apf = T(0);
  if (work) {
    const auto dp = zero ? buf_rsrc(rhs, 0u) : buf_rsrc(phi, 0x7fffffffu);
    const auto dr = buf_rsrc(rhs, 0x7fffffffu);
#pragma unroll
    for (int t = 0; t < NH; ++t) E[t] = buf_ld<T>(dp, in(2 * t + 1 - f, offE), 2 * t * pb);
#pragma unroll
    for (int t = 0; t < NH; ++t) ra[t] = buf_ld<T>(dr, in(2 * t + f, offA), 2 * t * pb);
#pragma unroll
    for (int t = 0; t < NH; ++t) re[t] = buf_ld<T>(dr, in(2 * t + 1 - f, offE), 2 * t * pb);
    if (live) {
      api = mg_coef(d, 1, j, k, c0, c1, c2).ap;
      apf = mg_coef(d, 0, j, k, c0, c1, c2).ap;
      ri = T(1) / api;
      rf = T(1) / apf;
    }
  }
  // interior or face value of the cell X[t], whose plane is oi + 2 t + g
  const bool flo = oi == 0, fhi = oi + RI >= n0;
  auto pick = [&](int t, int g, T vi, T vf) -> T {
    if constexpr (PART) {
      const int p = oi + 2 * t + g;
      return p >= n0 ? T(0) : p == 0 || p == n0 - 1 ? vf : vi;
    } else {
      return t == 0 ? (flo && g == 0 ? vf : vi) : t == NH - 1 && fhi && g == 1 ? vf : vi;
    }
  };

  const int pitch = n2 + 1;
  const int wc = live ? (j + 1) * pitch + k + 1 : 1;
  const int wq = live ? pitch : 0;
  {
    using V4 = __attribute__((ext_vector_type(4))) unsigned;
    const int nv = (nseg * RI + 2) * PL * (int)sizeof(T) / 16;
    V4* const z = reinterpret_cast<V4*>(sm);
    for (int w = tid; w < nv; w += (int)blockDim.x) z[w] = V4{0u, 0u, 0u, 0u};
  }
  T* const lo = sm + (oi + 1) * PL + wc;
  T* const lA = lo + f * PL;        // LDS words of the odd cells: lA[2 t PL]
  T* const lE = lo + (1 - f) * PL;  // and of the even ones
  if constexpr (UP) {
    if (work) add_prolonged<T, NH>(E, pc, d, oi + 1 - f, j, k, live);
  }
  __syncthreads();
  if (work) {
#pragma unroll
    for (int t = 0; t < NH; ++t) lE[2 * t * PL] = E[t];
  }
  __syncthreads();

  // use(t, sum of the off-diagonal terms of X[t]) for every cell of X's colour: Y[t]
  // and the plane before or after it from the column, ye beyond the segment and
  // the rows from LDS, all read before the first use
  auto sums = [&](const T* Y, const T* l, bool up, auto&& use) {
    const T ye = up ? l[(2 * NH - 1) * PL] : l[-PL];
    T nb[NH][4];
#pragma unroll
    for (int t = 0; t < NH; ++t) {
      const T* q = l + 2 * t * PL;
      nb[t][0] = q[-wq];
      nb[t][1] = q[wq];
      nb[t][2] = q[-1];
      nb[t][3] = q[1];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < NH; ++t) {
      const T yb = t > 0 ? Y[t > 0 ? t - 1 : 0] : ye;
      const T ya = t + 1 < NH ? Y[t + 1 < NH ? t + 1 : 0] : ye;
      use(t, nb6(c0, c1, c2, up ? Y[t] : yb, up ? ya : Y[t], nb[t][0], nb[t][1], nb[t][2],
                 nb[t][3]));
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  for (int s = 0; s < ns; ++s) {
    if (work) {
      sums(E, lA, fb, [&](int t, T sum) { A[t] = (ra[t] - sum) * pick(t, f, ri, rf); });
#pragma unroll
      for (int t = 0; t < NH; ++t) lA[2 * t * PL] = A[t];
    }
    __syncthreads();
    if (work) {
      sums(A, lE, !fb, [&](int t, T sum) { E[t] = (re[t] - sum) * pick(t, 1 - f, ri, rf); });
      if (!UP || s + 1 < ns)
#pragma unroll
        for (int t = 0; t < NH; ++t) lE[2 * t * PL] = E[t];
    }
    if (!UP || s + 1 < ns) __syncthreads();
  }

  if (live) {  // the level, and its images on the face ring
    const auto dout = buf_rsrc(phi, 0x7fffffffu);
    auto put = [&](uint32_t by) {
#pragma unroll
      for (int t = 0; t < NH; ++t) {
        buf_st(dout, in(2 * t + f, offA + by), 2 * t * pb, A[t]);
        buf_st(dout, in(2 * t + 1 - f, offE + by), 2 * t * pb, E[t]);
      }
    };
    put(0u);
    const uint32_t sj = (uint32_t)((int)d.s1 * (int)sizeof(T));
    if (j == 0) put(0u - sj);
    if (j == n1 - 1) put(sj);
    if (k == 0) put(0u - (uint32_t)sizeof(T));
    if (k == n2 - 1) put((uint32_t)sizeof(T));
    if (oi == 0) buf_st(dout, cb, 0, fb ? E[0] : A[0]);
#pragma unroll
    for (int t = 0; t < NH; ++t) {
      if (oi + 2 * t + f == n0 - 1) buf_st(dout, offA, (2 * t + 1) * pb, A[t]);
      if (oi + 2 * t + 1 - f == n0 - 1) buf_st(dout, offE, (2 * t + 1) * pb, E[t]);
    }
  }
  if constexpr (!UP) {  // residuals in place of the right-hand sides, and their sums
    if (work) {
      sums(E, lA, fb,
           [&](int t, T sum) { ra[t] = ra[t] - fma(pick(t, f, api, apf), A[t], sum); });
      sums(A, lE, !fb,
           [&](int t, T sum) { re[t] = re[t] - fma(pick(t, 1 - f, api, apf), E[t], sum); });
    }
    __syncthreads();
    if (work) {
#pragma unroll
      for (int t = 0; t < NH; ++t) {
        lA[2 * t * PL] = ra[t];
        lE[2 * t * PL] = re[t];
      }
    }
    __syncthreads();
    const int nc = dc.n1 * dc.n2;
    for (int q = tid; q < dc.n0 * nc; q += (int)blockDim.x) {
      const int ci = q / nc, r = q - ci * nc, cj = r / dc.n2, ck = r - cj * dc.n2;
      const T* const l = sm + (2 * ci + 1) * PL + (2 * cj + 1) * pitch + 2 * ck + 1;
      T acc = T(0);
#pragma unroll
      for (int c = 0; c < 8; ++c)
        acc = acc + l[(c >> 2) * PL + ((c >> 1) & 1) * pitch + (c & 1)];
      rc[mg_at(dc, ci, cj, ck)] = acc * T(0.125);
    }
  }
}

// The levels of a leg.
constexpr int WG_MAX_LEVELS = 16;
template <class T>
struct WgLevels {
  MgDev d[WG_MAX_LEVELS];
  T* phi[WG_MAX_LEVELS];
  T* rhs[WG_MAX_LEVELS];
  T c[WG_MAX_LEVELS][3];
};

// Down the levels l0 .. l1 (restricting onto level l1 + 1 last), or up them.
template <class T, bool UP>
__global__ void __launch_bounds__(WG_THREADS)
wg_leg_kernel(WgLevels<T> L, int l0, int l1, int ns, bool zero0) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T* const sm = reinterpret_cast<T*>(smem_raw);
  for (int q = 0; q <= l1 - l0; ++q) {
    const int l = UP ? l1 - q : l0 + q;
    const bool zero = !UP && (l > l0 || zero0);
    const T* const pc = UP ? L.phi[l + 1] : nullptr;
    T* const rc = UP ? nullptr : L.rhs[l + 1];
    if (L.d[l].n0 % WG_RI)
      wg_level<T, true, UP>(L.phi[l], L.rhs[l], L.d[l], L.c[l][0], L.c[l][1], L.c[l][2], ns, zero,
                            pc, rc, sm);
    else
      wg_level<T, false, UP>(L.phi[l], L.rhs[l], L.d[l], L.c[l][0], L.c[l][1], L.c[l][2], ns,
                             zero, pc, rc, sm);
    __syncthreads();  // this level's words are read, its arrays written
  }
}

}  // namespace wf
