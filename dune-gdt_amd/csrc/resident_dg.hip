// resident_dg.hip -- Jacobi-PCG solves in one launch for discontinuous spaces of 4 DoFs per element (gfx950, FP64).
//
// The scheme is that of resident.hip: one workgroup per CU keeps its rows on the chip for the whole solve, partials
// and the neighbours' values go through slots that hold a sentinel until they are stored, every wait is bounded.  What
// differs is the layout: a lane holds elements (4 consecutive rows each), not single rows, because the operator is one of
//   element blocks: the 4 x 4 blocks of an element with itself and up to 4 neighbours, 76 doubles, stay in the lane's
//     registers (152 of its 256), so an iteration reads nothing from memory but the halo;
//   matrix-free SWIPDG on a structured grid: per side of an element four weights (all forms, coefficients and lengths
//     multiplied out and added up before the first step) instead of the forms' loop in every step: 80 operations per
//     element where the closed form takes about 300.  A boundary side is an inner one whose neighbour is zero.
// A workgroup's elements are a rectangle of the lattice where there is one (halo: its perimeter), else consecutive.
// The matrix-free solve runs in the unscaled variables (r, z = D^{-1} r, p): neighbours then need z alone, not also their
// D^{-1/2}.  The sums of p.q and of the norms are those of the workgroups in their order: the three kernels
// add the same terms in another order, so a solve agrees with theirs up to round-off and not bit for bit.  One instance that is
// too large changes the elements per lane (matrix-free) or the path (blocks) of its whole batch, and with them the
// rounding of the others.
// Measured (us per iteration, three kernels -> one launch): element blocks 256 x 192 elements 17.7 -> 5.1, matrix-free
// 512 x 512 elements 23.6 -> 8.7.  What bounds an iteration now: the two exchanges (2.4-3.5 us each with 96-256
// workgroups) and the barriers around them.  More than 131 072 elements with their blocks do not fit in the
// registers of 256 CUs, and reading 168 MB of blocks per step instead leaves nothing to gain; matrix-free 262 144 elements.

#include <algorithm>
#include <cmath>

#include "index_math.hpp"
#include "mf_params.hpp"
#include "resident_device.hpp"

namespace hgdt {
namespace {

constexpr int T = RES_LANES, NW = T / 64;
enum { DG_BLOCKS = 0, DG_MATRIX_FREE = 1 };

struct alignas(16) Pair {
  double a, b;
};

// DoF of an element's side along direction o (side 1: reference coordinate 1), m = 0, 1 along the side
constexpr int side_dof(int o, int side, int m)
{
  return o == 0 ? side + 2 * m : 2 * side + m;
}

// 1 / x for x > 0: hardware reciprocal and two Newton steps (correct to round-off)
__device__ __forceinline__ double inverse(double x)
{
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.), r, r);
  return fma(fma(-x, r, 1.), r, r);
}

__device__ __forceinline__ void lds_read4(const double* p, double (&v)[4])
{
  const Pair a = reinterpret_cast<const Pair*>(p)[0], b = reinterpret_cast<const Pair*>(p)[1];
  v[0] = a.a, v[1] = a.b, v[2] = b.a, v[3] = b.b;
}
__device__ __forceinline__ void lds_write4(double* p, const double (&v)[4])
{
  reinterpret_cast<Pair*>(p)[0] = {v[0], v[1]};
  reinterpret_cast<Pair*>(p)[1] = {v[2], v[3]};
}

// the operator of one element in registers
template <int OP>
struct Element;

template <>
struct Element<DG_BLOCKS> {
  double own[16], nb[4][16]; // row-major blocks (own: unit diagonal, not read)
  __device__ __forceinline__ void load(const ResidentParams& P, const MfParams&, const ResidentTask&, int64_t e,
                                       const unsigned (&)[4])
  {
#pragma unroll
    for (int k = 0; k < 16; ++k)
      own[k] = 0.;
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int k = 0; k < 16; ++k)
        nb[s][k] = 0.;
    if (e < 0)
      return;
    const int64_t ne = P.blk_ne;
    const bool sym = P.blk_sym;
#pragma unroll
    for (int k = 0; k < 16; ++k)
      if (k % 5 != 0) {
        const int up = k / 4 > k % 4 ? 4 * (k % 4) + k / 4 : k; // symmetric: the upper triangle is the one in use
        own[k] = P.scaled[int64_t(sym ? up : k) * ne + e];
      }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int32_t f = s < P.blk_mn ? P.blk_nb[int64_t(s) * ne + e] : -1;
      if (f < 0)
        continue;
      if (sym && f < e) { // stored with the neighbour, transposed
        const double* B = P.scaled + int64_t(16 + 16 * P.blk_mir[int64_t(s) * ne + e]) * ne + f;
#pragma unroll
        for (int k = 0; k < 16; ++k)
          nb[s][4 * (k % 4) + k / 4] = B[int64_t(k) * ne];
      } else {
        const double* B = P.scaled + int64_t(16 + 16 * s) * ne + e;
#pragma unroll
        for (int k = 0; k < 16; ++k)
          nb[s][k] = B[int64_t(k) * ne];
      }
    }
  }
  __device__ __forceinline__ void apply(const double* pl, const double (&a)[4], const unsigned (&place)[4],
                                        double (&y)[4]) const
  {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      y[i] = a[i];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j != i)
          y[i] = fma(own[4 * i + j], a[j], y[i]);
#pragma unroll
    for (int s0 = 0; s0 < 4; s0 += 2) {
      double v[2][4];
      lds_read4(pl + 4 * place[s0], v[0]);
      lds_read4(pl + 4 * place[s0 + 1], v[1]);
#pragma unroll
      for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            y[i] = fma(nb[s0 + g][4 * i + j], v[g][j], y[i]);
    }
  }
};

// With D = u(side 1) - u(side 0) of the element along direction o, and per side J = u_inside - u_outside and D of
// the neighbour (coefficients along the side, W = [2 1; 1 2] their mass matrix up to the factor in the weights),
//   F = flux_own D + flux_nb D_nb,   rows of the side: -+ F +- penalty J,   rows of side 1 / 0: -+ symmetry J
template <>
struct Element<DG_MATRIX_FREE> {
  double fo[4], fn[4], so[4], pn[4]; // flux, own and neighbour; symmetrisation; penalty (sides x-, x+, y-, y+)
  double c[2], cm;                   // Laplace along x and y, product
  __device__ __forceinline__ void load(const ResidentParams& P, const MfParams& M, const ResidentTask& K, int64_t e,
                                       const unsigned (&place)[4])
  {
#pragma unroll
    for (int s = 0; s < 4; ++s)
      fo[s] = fn[s] = so[s] = pn[s] = 0.;
    c[0] = c[1] = cm = 0.;
    if (e < 0)
      return;
    const double* R = P.dg_ref + int64_t(K.inst) * M.ref_stride; // h0, h1, 1 / h1, 1 / h0
    const double h[2] = {R[0], R[1]}, ih[2] = {R[3], R[2]};
    const int64_t step[4] = {-1, 1, -int64_t(K.slice0), int64_t(K.slice0)};
    for (int f = 0; f < M.nef; ++f) {
      const double v = M.ef[f].scale * cf(M.ef[f].coef, M.ef[f].value, e);
      if (M.ef[f].kind == EF_LAPLACE)
        c[0] += v * (h[1] * ih[0]) * (1. / 6.), c[1] += v * (h[0] * ih[1]) * (1. / 6.);
      else
        cm += v * (h[0] * h[1]) * (1. / 36.);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int o = s >> 1;
      const double c6 = h[1 - o] * (1. / 6.), ilen = ih[1 - o];
      const bool inner = place[s] != unsigned(P.zero_place);
      const int nf = inner ? M.ncf : M.nbf;
      for (int f = 0; f < nf; ++f) {
        const MfFaceForm& Fm = M.ff[inner ? 0 : 1][f];
        const double sc = Fm.scale, prm = Fm.param;
        const bool coupling = Fm.kind == (inner ? FF_INNER_COUPLING : FF_DIRICHLET_COUPLING);
        double wo = 1., wn = 0., pen = 0.;
        if (inner) {
          const double os = cf(Fm.omega, Fm.ov, e), on = cf(Fm.omega, Fm.ov, e + step[s]);
          const double inv = inverse(os + on);
          wo = on * inv, wn = os * inv, pen = os * on * inv;
        } else if (!coupling) {
          pen = cf(Fm.omega, Fm.ov, e);
        }
        if (coupling) {
          const double ko = wo * cf(Fm.kappa, Fm.kv, e);
          fo[s] += sc * ko, so[s] += sc * prm * ko;
          if (inner)
            fn[s] += sc * (wn * cf(Fm.kappa, Fm.kv, e + step[s]));
        } else {
          pn[s] += sc * (prm * pen) * ilen;
        }
      }
      fo[s] *= c6 * ih[o], fn[s] *= c6 * ih[o], so[s] *= c6 * ih[o], pn[s] *= c6;
    }
  }
  __device__ __forceinline__ void apply(const double* pl, const double (&a)[4], const unsigned (&place)[4],
                                        double (&y)[4]) const
  {
    // product: W along x, then along y
    const double t[4] = {2. * a[0] + a[1], a[0] + 2. * a[1], 2. * a[2] + a[3], a[2] + 2. * a[3]};
    y[0] = cm * (2. * t[0] + t[2]), y[1] = cm * (2. * t[1] + t[3]);
    y[2] = cm * (t[0] + 2. * t[2]), y[3] = cm * (t[1] + 2. * t[3]);
#pragma unroll
    for (int o = 0; o < 2; ++o) {
      double lo[4], hi[4], r0[2], r1[2];
      lds_read4(pl + 4 * place[2 * o], lo);
      lds_read4(pl + 4 * place[2 * o + 1], hi);
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const double a0 = a[side_dof(o, 0, m)], a1 = a[side_dof(o, 1, m)], d = a1 - a0;
        const double jl = lo[side_dof(o, 1, m)] - a0, jh = a1 - hi[side_dof(o, 0, m)];
        const double dl = lo[side_dof(o, 1, m)] - lo[side_dof(o, 0, m)];
        const double dh = hi[side_dof(o, 1, m)] - hi[side_dof(o, 0, m)];
        const double sy = fma(so[2 * o], jl, fma(so[2 * o + 1], jh, -c[o] * d));
        r0[m] = fma(fo[2 * o], d, fma(fn[2 * o], dl, fma(-pn[2 * o], jl, sy)));
        r1[m] = fma(-fo[2 * o + 1], d, fma(-fn[2 * o + 1], dh, fma(pn[2 * o + 1], jh, -sy)));
      }
      y[side_dof(o, 0, 0)] += 2. * r0[0] + r0[1], y[side_dof(o, 0, 1)] += r0[0] + 2. * r0[1];
      y[side_dof(o, 1, 0)] += 2. * r1[0] + r1[1], y[side_dof(o, 1, 1)] += r1[0] + 2. * r1[1];
    }
  }
};

// PCG of the tasks of one workgroup.  Lane t holds the elements t, t + T, ... of the task's list, E of them (those past its
// end: zeros).  In LDS: p of the own elements, of the halo's, and one element of zeros.
template <int OP, int E>
__global__ void __launch_bounds__(T) k_pcg_resident_dg(ResidentParams P, MfParams M)
{
  extern __shared__ __align__(16) double pl[];
  __shared__ double ga[NW], gv[2][NW];
  __shared__ double red1[1][RES_WAVES], red2[2][RES_WAVES];
  __shared__ int failed;
  constexpr bool MF = OP == DG_MATRIX_FREE;
  constexpr int EL = E * T;
  // (element blocks: registers hold the matrix, LDS also the iterate and D^{1/2}, behind p)
  double* const xl = pl + 4 * (P.zero_place + 1);
  double* const sl = xl + 4 * EL;
  // published values lie by DoF, then by element: lanes of neighbouring elements store and read whole lines
  const unsigned ne = unsigned(P.n / 4);
  const int t = threadIdx.x, wave = t >> 6;
  if (t == 0)
    failed = 0;
  const int last = P.task_start[blockIdx.x + 1];
  for (int task = P.task_start[blockIdx.x]; task < last; ++task) {
    const ResidentTask K = P.tasks[task];
    const bool alone = K.team == 1;
    const int nhalo = K.nhalo;
    const int32_t* const helem = P.halo_rows + K.halo0;
    // D^{1/2} of the scaled system, or (matrix-free) D^{-1} of the unscaled one
    double r[E][4], x[MF ? E : 1][4], sc[MF ? E : 1][4];
    unsigned place[E][4], elem[E]; // (elem: bit 30: read by other workgroups)
    Element<OP> A[E];
    __syncthreads(); // the previous task's last reads of LDS
    if (t < 4)
      pl[4 * P.zero_place + t] = 0.;
#pragma unroll
    for (int k = 0; k < E; ++k) {
      const int64_t at_list = int64_t(K.mask) * EL + k * T + t;
      const int32_t id = P.dg_elements[at_list];
      const int64_t e = id < 0 ? -1 : id & 0x3fffffff;
      elem[k] = unsigned(id);
#pragma unroll
      for (int s = 0; s < 4; ++s)
        place[k][s] = P.sell_local[4 * at_list + s];
      double z[4] = {0., 0., 0., 0.}, xk[4] = {0., 0., 0., 0.}, sk[4] = {0., 0., 0., 0.};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int64_t i = 4 * e + j;
        r[k][j] = 0.;
        if (e >= 0) {
          const double ri = P.r[i], xi = P.x[i], sq = P.dsq[i];
          if constexpr (MF) {
            const double dh = P.dh[i];
            r[k][j] = sq * ri, xk[j] = dh * xi, sk[j] = dh * dh, z[j] = dh * ri;
          } else {
            r[k][j] = z[j] = ri, xk[j] = xi, sk[j] = sq;
          }
        }
        if constexpr (MF)
          x[k][j] = xk[j], sc[k][j] = sk[j];
      }
      if constexpr (!MF)
        lds_write4(xl + 4 * (k * T + t), xk), lds_write4(sl + 4 * (k * T + t), sk);
      lds_write4(pl + 4 * (k * T + t), z);
      A[k].load(P, M, K, e, place[k]);
    }
    for (int h = t; h < nhalo; h += T) {
      const int64_t i = 4 * int64_t(helem[h]);
      double z[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        z[j] = MF ? P.dh[i + j] * P.r[i + j] : P.r[i + j];
      lds_write4(pl + 4 * (EL + h), z);
    }
    const double tol2 = P.S[K.inst].tol2;
    double rn[2], rho_prev = 0., beta = 0.;
    {
      // the initial residual's partials
      double v[2] = {0., 0.};
      for (int b = t; b < K.nv; b += T)
        v[0] += P.part2[2 * int64_t(K.v0 + b)], v[1] += P.part2[2 * int64_t(K.v0 + b) + 1];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const double w = wave_sum(v[k]);
        if ((t & 63) == 0)
          red2[k][wave] = w;
      }
      __syncthreads();
      rn[0] = add_run(red2[0], NW), rn[1] = add_run(red2[1], NW);
    }
    int it = 0, begun = 0, state = 0;
    double alpha = 0., pq = 0.;
    unsigned long long halo[4]; // z (blocks: r) of halo element t
    const int h0 = t < nhalo ? helem[t] : 0;
    const int max_iter = int(min(P.max_iter, int64_t(0x7ffffff0)));
    for (;; ++it) {
      // the lane, opaque in every step: the addresses made from it are not kept in registers across steps
      int l = t;
      asm volatile("" : "+v"(l));
      state = uniform((rn[1] <= tol2) ? 1 : (it >= max_iter) ? 2 : 0);
      begun = state ? it : it + 1;
      const double rho = rn[0];
      if (state)
        break;
      // p = z + beta p on the own elements and on the halo
      if (it > 0) {
        beta = rho / rho_prev;
#pragma unroll
        for (int k = 0; k < E; ++k) {
          double p[4];
          lds_read4(pl + 4 * (k * T + l), p);
#pragma unroll
          for (int j = 0; j < 4; ++j)
            p[j] = fma(beta, p[j], MF ? sc[k][j] * r[k][j] : r[k][j]);
          lds_write4(pl + 4 * (k * T + l), p);
        }
        if (!alone) {
          const double* from = P.r_pub[(it & 1) ^ 1];
          for (int h = l; h < nhalo; h += T) {
            int src = h0;
            if (h >= T) { // not asked for yet
              src = helem[h];
#pragma unroll
              for (int j = 0; j < 4; ++j)
                halo[j] = RES_EMPTY;
            }
            Patience wait;
            bool empty;
            do {
              empty = false;
#pragma unroll
              for (int j = 0; j < 4; ++j)
                if (halo[j] == RES_EMPTY)
                  halo[j] = slot_load(at(from, unsigned(j) * ne + unsigned(src)));
#pragma unroll
              for (int j = 0; j < 4; ++j)
                empty = empty || halo[j] == RES_EMPTY;
              if (empty && wait.over(P.gave_up, P.wait_ticks)) {
                failed = 1;
                break;
              }
            } while (empty);
            double p[4];
            lds_read4(pl + 4 * (EL + h), p);
#pragma unroll
            for (int j = 0; j < 4; ++j)
              p[j] = fma(beta, p[j], __longlong_as_double((long long)halo[j]));
            lds_write4(pl + 4 * (EL + h), p);
          }
        }
      }
      rho_prev = rho;
      __syncthreads();
      if (uniform(failed))
        return;
      double q[E][4], dot = 0.;
#pragma unroll
      for (int k = 0; k < E; ++k) {
        double p[4];
        lds_read4(pl + 4 * (k * T + l), p);
        A[k].apply(pl, p, place[k], q[k]);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          dot = fma(p[j], q[k][j], dot);
      }
      dot = wave_sum(dot);
      if ((l & 63) == 0)
        ga[wave] = dot;
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      const int par = it & 1, set = it % 3;
      double tot1[1];
      const double own1[1] = {add_run(ga, NW)};
      if (alone) {
        tot1[0] = own1[0];
      } else {
        if (l == 0) {
          slot_store(P.g1 + (set * P.n_a + K.own_a) * RES_PAD, own1[0]);
          slot_clear(P.g1 + ((it + 2) % 3 * P.n_a + K.own_a) * RES_PAD);
        }
        if (!exchange_sum<1, NW>(P.g1 + (set * P.n_a + K.a0) * RES_PAD, own1, false, K.na, T, red1, &failed, P.gave_up,
                                 P.wait_ticks, tot1))
          return;
      }
      pq = tot1[0];
      if (!uniform(pq > 0.)) { // breakdown: the iterate holds every earlier step
        state = 3;
        break;
      }
      // update of r, what other workgroups read, the partials of the residual norms
      alpha = rho / pq;
      double v[2] = {0., 0.};
#pragma unroll
      for (int k = 0; k < E; ++k) {
        double z[4], s[4];
        if constexpr (MF) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            s[j] = sc[k][j];
        } else {
          lds_read4(sl + 4 * (k * T + l), s);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const double ri = fma(-alpha, q[k][j], r[k][j]), si = s[j] * ri;
          r[k][j] = ri;
          z[j] = MF ? si : ri;
          if constexpr (MF)
            v[0] = fma(ri, si, v[0]), v[1] = fma(ri, ri, v[1]);
          else
            v[0] = fma(ri, ri, v[0]), v[1] = fma(si, si, v[1]);
        }
        if (elem[k] >> 30 == 1u) {
          double* const to = P.r_pub[par];
          unsigned id = elem[k] & 0x3fffffffu;
          asm volatile("" : "+v"(id));
#pragma unroll
          for (int j = 0; j < 4; ++j)
            slot_store(at(to, unsigned(j) * ne + id), z[j]);
        }
      }
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const double w = wave_sum(v[k]);
        if ((l & 63) == 0)
          gv[k][wave] = w;
      }
      __syncthreads();
      const double own2[2] = {add_run(gv[0], NW), add_run(gv[1], NW)};
      if (!alone && l == 0) {
        double* mine = P.g2 + (par * P.n_v + K.own_a) * RES_PAD;
        slot_store(mine, own2[0]), slot_store(mine + 1, own2[1]);
      }
      // in the time the exchange takes: x, the next step's slots and values emptied, and the halo's values asked for
#pragma unroll
      for (int k = 0; k < E; ++k) {
        double p[4];
        lds_read4(pl + 4 * (k * T + l), p);
        if constexpr (MF) {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            x[k][j] = fma(alpha, p[j], x[k][j]);
        } else {
          double xk[4];
          lds_read4(xl + 4 * (k * T + l), xk);
#pragma unroll
          for (int j = 0; j < 4; ++j)
            xk[j] = fma(alpha, p[j], xk[j]);
          lds_write4(xl + 4 * (k * T + l), xk);
        }
      }
      if (alone) {
        rn[0] = own2[0], rn[1] = own2[1];
      } else {
        if (l == 0) {
          double* next = P.g2 + ((par ^ 1) * P.n_v + K.own_a) * RES_PAD;
          slot_clear(next), slot_clear(next + 1);
        }
#pragma unroll
        for (int k = 0; k < E; ++k)
          if (elem[k] >> 30 == 1u) {
            double* const next = P.r_pub[par ^ 1];
            unsigned id = elem[k] & 0x3fffffffu;
            asm volatile("" : "+v"(id));
#pragma unroll
            for (int j = 0; j < 4; ++j)
              slot_clear(at(next, unsigned(j) * ne + id));
          }
        if (l < nhalo) {
          unsigned id = unsigned(h0);
          asm volatile("" : "+v"(id));
#pragma unroll
          for (int j = 0; j < 4; ++j)
            halo[j] = slot_load(at(P.r_pub[par], unsigned(j) * ne + id));
        }
        if (!exchange_sum<2, NW>(P.g2 + (par * P.n_v + K.a0) * RES_PAD, own2, false, K.na, T, red2, &failed, P.gave_up,
                                 P.wait_ticks, rn))
          return;
      }
    }
#pragma unroll
    for (int k = 0; k < E; ++k)
      if (!(elem[k] >> 31))
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int64_t i = 4 * int64_t(elem[k] & 0x3fffffffu) + j;
          P.x_out[i] = MF ? P.dsq[i] * x[MF ? k : 0][j] : xl[4 * (k * T + t) + j];
        }
    if (K.rank == 0 && t == 0) {
      PcgScalars D = P.S[K.inst];
      D.rz = rn[0], D.rr = rn[1], D.beta = beta, D.alpha = alpha, D.alpha_prev = alpha, D.pq = pq;
      D.iters = begun;
      D.done = state;
      D.brk = 0;
      P.result[K.inst] = D;
    }
  }
}

} // namespace

const void* resident_dg_kernel(const ResidentPlan& plan)
{
  auto k = [](auto kernel) { return reinterpret_cast<const void*>(kernel); };
  if (!plan.matrix_free)
    return k(k_pcg_resident_dg<DG_BLOCKS, 1>);
  return plan.slots == 1 ? k(k_pcg_resident_dg<DG_MATRIX_FREE, 1>) : k(k_pcg_resident_dg<DG_MATRIX_FREE, 2>);
}

// split of an n0 x n1 lattice into equal rectangles of at most `most` cells (the last of a row or column may be smaller):
// few, and with few neighbours in other rectangles
static void rectangles(int64_t n0, int64_t n1, int64_t most, int64_t (&w)[2])
{
  double best = 0.;
  for (int64_t g = 1; g <= n0; ++g) {
    const int64_t a = (n0 + g - 1) / g;
    if (a > most || (n0 + a - 1) / a != g)
      continue;
    const int64_t g1 = (n1 + most / a - 1) / (most / a), b = (n1 + g1 - 1) / g1;
    const double cost = double(g * g1) + 0.02 * double((g1 > 1 ? a : 0) + (g > 1 ? b : 0));
    if (best == 0. || cost < best)
      best = cost, w[0] = a, w[1] = b;
  }
}

static bool on_lattice(const Operator& op, int in)
{
  const Space& s = *op.space;
  const Grid& g = *s.grid;
  const int64_t e0 = g.inst_elem[in], ne = g.inst_elem[in + 1] - e0;
  return int(g.lattice.size()) == g.ninst() && g.ref.geom == HGDT_QUAD && g.lattice[in].n[0] * g.lattice[in].n[1] == ne &&
         s.inst_dof[in] == 4 * e0 && s.inst_dof[in + 1] == 4 * (e0 + ne);
}

// workgroups of an instance with `most` elements each
static int team_of(const Operator& op, int in, int64_t most)
{
  const int64_t ne = (op.space->inst_dof[in + 1] - op.space->inst_dof[in]) / 4;
  if (!on_lattice(op, in))
    return int((ne + most - 1) / most);
  const Lattice& L = op.space->grid->lattice[in];
  int64_t w[2] = {1, 1};
  rectangles(L.n[0], L.n[1], most, w);
  return int(((L.n[0] + w[0] - 1) / w[0]) * ((L.n[1] + w[1] - 1) / w[1]));
}

void resident_plan_dg(ResidentPlan& plan, const Operator& op)
{
  plan.usable = false;
  const SolverFormat& F = op.fmt;
  const Space& sp = *op.space;
  const std::vector<int64_t>& row0 = sp.inst_dof;
  const int ninst = int(row0.size()) - 1;
  const bool mf = F.format == HGDT_FORMAT_MATRIX_FREE;
  if (op.n % 4 != 0 || !reached_by_32_bits(op.n) || (mf ? F.mf_kind != MFK_DG_QUAD : F.blk_mn > 4))
    return;
  for (int in = 0; in < ninst; ++in)
    if (row0[in + 1] == row0[in] || row0[in] % 4 != 0 || (mf && !on_lattice(op, in)))
      return;
  // elements per lane: one, unless an instance then has more workgroups than there are CUs (the same for an instance alone
  // and in a batch, where neither has such an instance: the sums, and so the bits, depend on it)
  int slots = 0;
  std::vector<int> teams(ninst);
  for (int s : {1, 2}) {
    for (int in = 0; in < ninst; ++in)
      teams[in] = team_of(op, in, int64_t(s) * T);
    if (resident_schedule(row0, teams, 1., nullptr, nullptr) >= 0.) {
      slots = s;
      break;
    }
    if (!mf)
      break;
  }
  if (slots == 0)
    return;
  const int64_t EL = int64_t(slots) * T;
  std::vector<int32_t> nb; // blocks: neighbours by slot and element
  if (!mf && F.blk_mn > 0) {
    nb.resize(F.d_blk_nb.count);
    F.d_blk_nb.download(nb.data());
  }
  // the workgroups' elements, and of every element its workgroup and its place there
  std::vector<ResidentTask> tasks;
  std::vector<int32_t> elements, group(op.n / 4), local(op.n / 4);
  for (int in = 0; in < ninst; ++in) {
    const int64_t e0 = row0[in] / 4, ne = (row0[in + 1] - row0[in]) / 4;
    const int a0 = int(tasks.size());
    int64_t w[2] = {ne, 1}, n[2] = {ne, 1};
    if (on_lattice(op, in)) {
      n[0] = sp.grid->lattice[in].n[0], n[1] = sp.grid->lattice[in].n[1];
      rectangles(n[0], n[1], EL, w);
    } else {
      w[0] = EL;
    }
    for (int64_t y = 0; y < n[1]; y += w[1])
      for (int64_t x = 0; x < n[0]; x += w[0]) {
        ResidentTask K{};
        K.inst = in, K.rank = int(tasks.size()) - a0, K.a0 = a0, K.own_a = int(tasks.size());
        K.v0 = F.V.inst_block0[in], K.nv = F.V.inst_block0[in + 1] - K.v0;
        K.slice0 = int32_t(n[0]), K.mask = int(tasks.size());
        const size_t first = elements.size();
        for (int64_t j = y; j < std::min(y + w[1], n[1]); ++j)
          for (int64_t i = x; i < std::min(x + w[0], n[0]); ++i) {
            const int64_t e = e0 + j * n[0] + i;
            group[e] = int32_t(tasks.size()), local[e] = int32_t(elements.size() - first);
            elements.push_back(int32_t(e));
          }
        if (int64_t(elements.size() - first) > EL)
          return;
        elements.resize(first + EL, -1);
        tasks.push_back(K);
      }
    for (size_t k = a0; k < tasks.size(); ++k)
      tasks[k].team = tasks[k].na = int(tasks.size()) - a0;
  }
  // neighbours: places in the workgroup's p, halo lists, which elements others read
  const int64_t nt = int64_t(tasks.size()), ne = op.n / 4;
  auto neighbour = [&](int64_t e, const ResidentTask& K, int s) -> int64_t {
    if (!mf)
      return s < F.blk_mn ? nb[int64_t(s) * ne + e] : -1;
    return sp.grid->nb[e * 4 + s];
  };
  std::vector<std::vector<int32_t>> halo(nt);
  parallel_for(nt, [&](int64_t b0, int64_t b1) {
    for (int64_t b = b0; b < b1; ++b) {
      for (int64_t k = 0; k < EL; ++k) {
        const int32_t e = elements[b * EL + k];
        for (int s = 0; e >= 0 && s < 4; ++s) {
          const int64_t f = neighbour(e, tasks[b], s);
          if (f >= 0 && group[f] != b)
            halo[b].push_back(int32_t(f));
        }
      }
      std::sort(halo[b].begin(), halo[b].end());
      halo[b].erase(std::unique(halo[b].begin(), halo[b].end()), halo[b].end());
    }
  });
  std::vector<uint8_t> read(ne, 0);
  std::vector<int32_t> rows;
  int64_t most = 0;
  for (int64_t b = 0; b < nt; ++b) {
    tasks[b].halo0 = int32_t(rows.size()), tasks[b].nhalo = int32_t(halo[b].size());
    most = std::max<int64_t>(most, tasks[b].nhalo);
    for (int32_t f : halo[b])
      read[f] = 1;
    rows.insert(rows.end(), halo[b].begin(), halo[b].end());
  }
  const int64_t lds = (EL + most + 1 + (mf ? 0 : 2 * EL)) * 4 * int64_t(sizeof(double));
  if (lds > RES_LDS || EL + most >= 65536)
    return;
  std::vector<uint16_t> places(size_t(4 * nt * EL));
  parallel_for(nt, [&](int64_t b0, int64_t b1) {
    for (int64_t b = b0; b < b1; ++b)
      for (int64_t k = 0; k < EL; ++k) {
        const int32_t e = elements[b * EL + k];
        for (int s = 0; s < 4; ++s) {
          const int64_t f = e < 0 ? -1 : neighbour(e, tasks[b], s);
          places[4 * (b * EL + k) + s] =
              uint16_t(f < 0             ? EL + most
                       : group[f] == b   ? local[f]
                                         : EL + (std::lower_bound(halo[b].begin(), halo[b].end(), f) - halo[b].begin()));
        }
        if (e >= 0 && read[e])
          elements[b * EL + k] |= 1 << 30;
      }
  });
  if (rows.empty())
    rows.push_back(0);
  plan.elements.upload(elements);
  plan.sell_local.upload(places);
  plan.halo_rows.upload(rows);
  plan.dg = true, plan.matrix_free = mf, plan.sell = plan.far = false;
  plan.lanes = T, plan.slots = slots, plan.zero_place = int(EL + most);
  plan.step = slots == 1 ? 2. : 3.;
  resident_finish(plan, op, tasks, lds, nt, nt);
}

} // namespace hgdt
