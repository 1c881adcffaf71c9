// resident.hip -- Jacobi-PCG solves in one launch, the vectors kept on the chip (gfx950, FP64).
//
// The solver of solver.hip issues three kernels per iteration.  Below some millions of DoFs their time is not the
// bytes: a kernel boundary and the chains of dependent loads behind it (record, partials, rows) cost 5-6 us each,
// and every vector makes a round trip through the caches per kernel.  Here one workgroup per CU keeps its rows of
// r, x and D^{1/2} in registers and of p (with the rows its stencil reaches into) in LDS for the whole solve:
// 256 CUs hold 128 MB of registers and 40 MB of LDS.  Per iteration a workgroup reads the matrix (or keeps that
// in registers too) and its halo of r, and takes part in two exchanges, p.q and the residual norms.
//
// Exchange: every block partial has a slot in global memory that holds a sentinel until its workgroup has
// stored it; every workgroup of the instance reads all slots, again until none holds the sentinel, and adds
// them in block order.  So the values are their own flags: one store and one load between the slowest
// workgroup and all others (2.4-3.5 us with 256 workgroups, 1-1.3 us with 16).  The sets of slots
// rotate, three for p.q and two for the norms: a workgroup empties its slots of the set that comes up next but one (norms:
// next) when it stores to one.  By then every workgroup has read what they held (it has stored to an exchange since),
// and none polls them again before this workgroup has stored to the p.q exchange in between, which it does after
// waiting for its earlier stores (vmcnt 0).  The rows of r that other workgroups read go the same way, through two
// arrays with the sentinel.  Slot accesses are relaxed atomics at agent scope, for which the XCDs' L2
// caches are coherent; as every value is its own flag, no order between different addresses is needed beyond that.
//
// Every value is computed by the operations of the three kernels in their order (row sums, block partials in
// the operator's and the vector partition, sums over the partials), so for the same launch shapes a solve gives the same
// bits on either path, alone or in a batch.  (The default shapes follow the size: of the instance, or of the batch.)
//
// Measured (us per iteration, three kernels -> one launch): Q1 32^2 15 -> 2.3, 128^2 14 -> 4.5, 701x523 18 -> 7.8, 1023^2
// 33 -> 11.8, P1 48^3 x 6 18 -> 7.0, eight of these in a batch 33 -> 9.4, 100^3 x 6 34 -> 19, 128^3 x 6 54 -> 27; SELL: P1
// triangles of a mesh with 160 401 vertices 18 -> 7.0, P2 triangles with 90 201 DoFs 18 -> 7.5; Q1 hexahedra (13 upper
// diagonals, read in every step) 20^3 15.2 -> 6.8, 40^3 16.1 -> 10.3, 63^3 21.7 -> 16.3.
// What bounds an iteration now: small problems two exchanges of 1-2.5 us, the barriers and sums around them; 4096 rows
// per workgroup LDS (13 reads of 8 bytes per row at 128 B per clock: 1.4 us) and registers (a variant that spilled 46 took
// 19 us instead of 11.8 at 1023^2: the scratch of 256 workgroups evicts L2); 128^3 x 6 the memory
// behind the L2 caches (104 MB of matrix and far p read, 17 MB of p written per iteration: 4.3 TB/s, the rate of a copy).
//
// All workgroups of a team must be on the chip together: the host launches at most one per CU and counts the
// CUs of all running launches of the process.  A wait that outlasts its limit (Operator::solve_wait: another process holds
// the CUs, or in a batch a partner is still busy with an earlier instance) sets a flag at which every workgroup ends; the
// caller then solves with the three kernels.

#include <algorithm>
#include <atomic>
#include <cmath>
#include <condition_variable>
#include <cstring>
#include <map>
#include <mutex>

#include "index_math.hpp"
#include "resident_device.hpp"

namespace hgdt {
namespace {

constexpr bool q_in_lds(int slots, int nu, bool far)
{
  return far || slots > 8 || (slots == 8 && nu >= 4);
}

// PCG of the tasks of one workgroup, one after the other.  Lane t holds rows t, t + T, ... of the workgroup,
// one per slot.  Vector blocks have 1 << LG rows per lane: T lanes, or (LG = 0) any number that divides it.  So
// a slot's rows are a constant away from slot 0's and LDS is read at constant offsets.  Rows past the end of the instance
// hold zeros and take part like others.  NU: strict upper slots compiled for (missing ones have zero values).
// KEEP != 0: the matrix rows stay in registers, else they are read every iteration.
// SAME: the operator blocks are the vector blocks; else they have one row per lane (64-row sums combined by threads).
// NU = 0: SELL-64 storage; p of the own rows is followed by the halo, a list of rows, and the entries hold positions
// in that; KEEP: entries of a row that registers hold (at least the widest slice's).
// FAR: the outermost of the NU offsets reaches further than LDS does (planes of a 3-d lattice): its columns, and the
// halo, are read as p from the other workgroups in every step.
template <int T, int S, int LG, bool SAME, int NU, int KEEP, bool FAR = false>
__global__ void __launch_bounds__(T) k_pcg_resident(ResidentParams P)
{
  extern __shared__ double pl[]; // p of the own rows and `reach` rows to either side (0 outside the instance)
  __shared__ double ga[RES_GROUPS], gv[2][RES_GROUPS];
  __shared__ double red1[1][RES_WAVES], red2[2][RES_WAVES];
  __shared__ int failed;
  constexpr int NW = T / 64, ITEMS = 1 << LG, R = S * T;
  constexpr bool SELL = NU == 0;
  // what registers do not hold: q (in LDS), D^{1/2} (read in every step), x (read and written in every step)
  constexpr bool QLDS = q_in_lds(S, NU, FAR), SQMEM = FAR || S > 8 || (S == 8 && !SELL), XMEM = S > 12;
  constexpr int NN = FAR ? NU - 1 : NU; // upper slots whose columns lie in LDS
  constexpr int MU = SELL ? 1 : NU;
  const int t = threadIdx.x, wave = t >> 6;
  const int vwaves = P.v_block >> 6;
  if (t == 0)
    failed = 0;
  const int last = P.task_start[blockIdx.x + 1];
  for (int task = P.task_start[blockIdx.x]; task < last; ++task) {
    const ResidentTask K = P.tasks[task];
    const int64_t n = P.n;
    const int64_t lo = P.inst_row0[K.inst], hi = P.inst_row0[K.inst + 1];
    const int ku = P.s_nu;
    const int64_t* __restrict__ so = P.s_off + int64_t(K.inst) * ku;
    const bool alone = K.team == 1;
    const int rows = K.rows;
    int off[MU];
    int reach = 0; // rows ahead of the own ones in pl
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int64_t o = u < ku ? so[u] : 0; // padding slots: values 0, offset 0
      off[u] = o < hi - lo ? int(o) : 0;
      if (u < NN)
        reach = max(reach, off[u]);
    }
    const int below = int(min(K.row0 - lo, int64_t(reach)));        // rows of the instance below the own ones
    const int above = int(min(hi - K.row0 - rows, int64_t(reach))); // and above, at most `reach`
    const int nhalo = SELL ? K.nhalo : below + above;
    // row of halo entry e, and its place in pl
    const int32_t* const hrow = P.halo_rows + (SELL ? K.halo0 : 0);
    auto halo_row = [&](int e) { return SELL ? int64_t(hrow[e]) : K.row0 - below + (e < below ? e : rows + e); };
    auto halo_place = [&](int e) { return SELL ? R + e : reach - below + (e < below ? e : rows + e); };
    double r[S], x[XMEM ? 1 : S], sq[SQMEM ? 1 : S];
    double au[!SELL && KEEP ? S : 1][MU], al[!SELL && KEEP ? S : 1][MU];
    constexpr int KW = SELL && KEEP ? KEEP : 2; // (even)
    double mv[SELL && KEEP ? S : 1][KW];
    uint32_t mi[SELL && KEEP ? S : 1][KW / 2];
    int width[SELL ? S : 1];
    __syncthreads(); // the previous task's last reads of LDS
    for (int e = t; e < R + 2 * reach; e += T) {
      const int o = e - reach;
      pl[e] = (o >= -below && o < rows + above) ? P.r[K.row0 + o] : 0.;
    }
    if constexpr (SELL)
      for (int e = t; e < nhalo; e += T)
        pl[R + e] = P.r[halo_row(e)];
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int o = t + s * T;
      const int64_t i = K.row0 + o;
      const bool in = o < rows;
      r[s] = in ? P.r[i] : 0.;
      if constexpr (!SQMEM)
        sq[s] = in ? P.dsq[i] : 0.;
      if constexpr (!XMEM)
        x[s] = in ? P.x[i] : 0.;
      else if (in)
        P.x_out[i] = P.x[i];
      if constexpr (SELL) {
        width[s] = 0;
        if constexpr (KEEP != 0)
#pragma unroll
          for (int k = 0; k < KW; ++k)
            mv[s][k] = 0., mi[s][k / 2] = 0u;
        if (uniform((s * NW + wave) * 64) < rows) {
          const int64_t* sp = P.slice_ptr + K.slice0 + s * NW + uniform(wave);
          const int64_t first = sp[0];
          width[s] = int((sp[1] - first) >> 6);
          if constexpr (KEEP != 0)
#pragma unroll
            for (int k = 0; k < KW; ++k)
              if (k < width[s]) {
                mv[s][k] = P.scaled[first + k * 64 + (t & 63)];
                mi[s][k / 2] |= uint32_t(P.sell_local[first + k * 64 + (t & 63)]) << (k % 2 ? 16 : 0);
              }
        }
      }
      if constexpr (!SELL && KEEP)
#pragma unroll
        for (int u = 0; u < NU; ++u) {
          const bool on = in && u < ku && off[u] > 0;
          au[s][u] = (on && i + off[u] < hi) ? P.scaled[int64_t(u) * n + i] : 0.;
          al[s][u] = (on && i - off[u] >= lo) ? P.scaled[int64_t(u) * n + i - off[u]] : 0.;
        }
    }
    const double tol2 = P.S[K.inst].tol2;
    const bool whole = rows == R;
    // FAR: workgroups that hold columns of the own rows
    const int64_t far_reach = FAR ? int64_t(off[NU - 1 > 0 ? NU - 1 : 0]) : 0;
    const int far_first = FAR ? int((max(K.row0 - far_reach, lo) - lo) / R) : 0;
    const int far_last = FAR ? int((min(K.row0 + rows + far_reach, hi) - 1 - lo) / R) : 0;
    const bool single = alone && K.na == 1 && K.nv == 1; // one partial: the sum itself, in every lane
    const int own_na = (rows + P.a_rows - 1) / P.a_rows;
    const int own_nv = (rows + P.v_block * ITEMS - 1) / (P.v_block * ITEMS);
    // own rows [0, pub_lo) and [pub_hi, ...) are read by other workgroups of the team
    // (SELL: the slots in `pub`)
    const uint32_t pub = SELL ? P.publish[int64_t(K.mask) * T + t] : 0u;
    const int pub_lo = K.rank > 0 ? min(reach, rows) : 0, pub_hi = K.rank + 1 < K.team ? rows - reach : R;
    double rn[2], rho_prev = 0., beta = 0.;
    {
      // the initial residual's partials are complete: summed from memory, in the same order
      double v[2] = {0., 0.};
      if (t < P.v_block)
        for (int b = t; b < K.nv; b += P.v_block)
          v[0] += P.part2[2 * int64_t(K.v0 + b)], v[1] += P.part2[2 * int64_t(K.v0 + b) + 1];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const double w = wave_sum(v[k]);
        if ((t & 63) == 0)
          red2[k][wave] = w;
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        rn[k] = 0.;
#pragma unroll
        for (int w = 0; w < NW; ++w)
          rn[k] += red2[k][w];
      }
    }
    int it = 0, begun = 0;
    int state = 0;
    double alpha = 0., pq = 0.;
    unsigned long long halo[RES_HALO]; // rows of r of the halo, entries t, t + T, ...
    int hr[RES_HALO];                  // SELL: which rows these are
    if constexpr (SELL)
#pragma unroll
      for (int k = 0; k < RES_HALO; ++k)
        hr[k] = t + k * T < nhalo ? hrow[t + k * T] : 0;
    const int max_iter = int(min(P.max_iter, int64_t(0x7ffffff0)));
    for (;; ++it) {
      // the lane, opaque in every step: the addresses made from it are not kept in registers across steps
      int l = t;
      asm volatile("" : "+v"(l));
      // direction update: stopping test, p = r + beta p on the own rows and on the halo
      state = uniform((rn[1] <= tol2) ? 1 : (it >= max_iter) ? 2 : 0);
      begun = state ? it : it + 1;
      const double rho = rn[0];
      if (state)
        break;
      double* const pt = pl + reach + l; // p of the lane's row in slot 0
      if (it > 0)
        beta = rho / rho_prev;
      if constexpr (FAR) {
        // p itself goes to the other workgroups: the rows, then (all have arrived) the step's number as this workgroup's
        // flag; the first wave waits for the flags of the workgroups within reach and fetches the halo
        double* const to = P.r_pub[0] + K.row0;
#pragma unroll
        for (int s = 0; s < S; ++s) {
          const double p = it > 0 ? fma(beta, pt[s * T], r[s]) : r[s];
          pt[s * T] = p;
          if (l + s * T < rows)
            __hip_atomic_store(at(to + s * T, unsigned(l)), p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (uniform(wave) == 0) {
          if (l == 0)
            __hip_atomic_store(P.flags + K.rank, it + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          for (int k = far_first + l; k <= far_last; k += 64) {
            Patience wait;
            while (__hip_atomic_load(P.flags + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < it + 1)
              if (wait.over(P.gave_up, P.wait_ticks)) {
                failed = 1;
                break;
              }
          }
          // The rows are read after the flags: this says so to the compiler (the loop has waited for the flags' values, and
          // the other waves come through the barrier below).  All of these are accesses that the XCDs' L2 caches keep
          // coherent, so no cache has to be written back or emptied in between; fences that do so (release and acquire at
          // agent scope) took heat on 128^3 x 6 tetrahedra from 17.9 to 19.7 ms.
          __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
          const double* from = to - below;
          for (int e = l; e < nhalo; e += 64)
            pl[halo_place(e)] = __hip_atomic_load(at(from, unsigned(e < below ? e : rows + e)), __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT);
        }
      } else if (it > 0) {
#pragma unroll
        for (int s = 0; s < S; ++s)
          pt[s * T] = fma(beta, pt[s * T], r[s]);
        if (!alone) {
          const double* from = P.r_pub[(it & 1) ^ 1] + (SELL ? 0 : K.row0 - below);
          for (int e0 = l; e0 < nhalo; e0 += RES_HALO * T) {
            Patience wait;
            const bool later = e0 >= RES_HALO * T; // entries not asked for yet
            unsigned src[RES_HALO];
#pragma unroll
            for (int k = 0; k < RES_HALO; ++k) {
              const int e = e0 + k * T;
              if (later)
                halo[k] = RES_EMPTY;
              if constexpr (SELL)
                src[k] = later ? (e < nhalo ? hrow[e] : 0) : hr[k];
              else
                src[k] = e < below ? e : rows + e;
            }
            bool empty;
            do {
              empty = false;
#pragma unroll
              for (int k = 0; k < RES_HALO; ++k)
                if (e0 + k * T < nhalo && halo[k] == RES_EMPTY)
                  halo[k] = slot_load(at(from, src[k]));
#pragma unroll
              for (int k = 0; k < RES_HALO; ++k)
                empty = empty || (e0 + k * T < nhalo && halo[k] == RES_EMPTY);
              if (empty && wait.over(P.gave_up, P.wait_ticks)) {
                failed = 1;
                break;
              }
            } while (empty);
#pragma unroll
            for (int k = 0; k < RES_HALO; ++k) {
              const int e = e0 + k * T;
              if (e < nhalo) {
                double& pe = pl[halo_place(e)];
                pe = fma(beta, pe, __longlong_as_double((long long)halo[k]));
              }
            }
          }
        }
      }
      rho_prev = rho;
      __syncthreads();
      if (uniform(failed))
        return;
      // q = Ah p, and p.q of the operator blocks: per 64 rows of one slot, or as the vector blocks
      double q[QLDS ? 1 : S], dot = 0.;
      double* const ql = pl + R + 2 * reach + l;
      auto take = [&](int s, double p, double a) { // the product's row of slot s
        if constexpr (QLDS)
          ql[s * T] = a;
        else
          q[s] = a;
        dot = fma(p, a, dot);
        if (!SAME || s % ITEMS == ITEMS - 1) {
          const double w = wave_sum(dot);
          if ((l & 63) == 0)
            ga[(SAME ? s >> LG : s) * NW + wave] = w;
          dot = 0.;
        }
      };
      if constexpr (SELL && KEEP != 0) {
        constexpr int W = 4; // positions read together
#pragma unroll
        for (int s = 0; s < S; ++s) {
          double a = 0.;
#pragma unroll
          for (int k0 = 0; k0 < KW; k0 += W)
            if (k0 < width[s]) {
              double x[W];
#pragma unroll
              for (int k = 0; k < W; ++k)
                x[k] = pl[k % 2 ? mi[s][(k0 + k) / 2] >> 16 : mi[s][(k0 + k) / 2] & 0xffffu];
#pragma unroll
              for (int k = 0; k < W; ++k)
                a = fma(mv[s][k0 + k], x[k], a);
            }
          take(s, pt[s * T], a);
        }
      } else if constexpr (SELL) {
        // a wave's rows of a slot are one slice; the first entries of the next slice are asked for ahead of the sums
        constexpr int W = 8;
        double m[2][W];
        int c[2][W];
        int64_t first[2];
        auto ask = [&](int s) {
          if (width[s] > 0) {
            first[s & 1] = P.slice_ptr[K.slice0 + s * NW + uniform(wave)];
#pragma unroll
            for (int k = 0; k < W; ++k) {
              const unsigned e = unsigned(min(k, width[s] - 1) * 64 + (l & 63));
              c[s & 1][k] = *at(P.sell_local + first[s & 1], e);
              m[s & 1][k] = *at(P.scaled + first[s & 1], e);
            }
          }
        };
        ask(0);
#pragma unroll
        for (int s = 0; s < S; ++s) {
          if (s + 1 < S)
            ask(s + 1);
          double a = 0.;
          if (width[s] > 0) {
            double x[W];
#pragma unroll
            for (int k = 0; k < W; ++k)
              x[k] = pl[c[s & 1][k]];
#pragma unroll
            for (int k = 0; k < W; ++k)
              if (k < width[s])
                a = fma(m[s & 1][k], x[k], a);
            for (int k = W; k < width[s]; ++k) {
              const unsigned e = unsigned(k * 64 + (l & 63));
              a = fma(*at(P.scaled + first[s & 1], e), pl[*at(P.sell_local + first[s & 1], e)], a);
            }
          }
          take(s, pt[s * T], a);
        }
      } else {
      const double *pd[MU], *pu[MU];
#pragma unroll
      for (int u = 0; u < NN; ++u)
        pd[u] = pt - off[u], pu[u] = pt + off[u];
      // FAR: the outermost columns, asked for two slots at a time ahead of the sums
      const double* const pf = P.r_pub[0] + K.row0;
      const int fo = FAR ? off[NU - 1] : 0;
      const int fl = FAR ? int(max(int64_t(fo) - (K.row0 - lo), int64_t(0))) : 0;  // first row with a column below
      const int fu = FAR ? int(min(hi - fo - K.row0, int64_t(rows))) : 0;          // end of the rows with one above
      double xf[2][2][2]; // [pair of slots][slot][below, above]
      auto far_ask = [&](int s0, int b) {
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          const int o = l + (s0 + g) * T;
          xf[b][g][0] = xf[b][g][1] = 0.;
          if (o >= fl && o < rows)
            xf[b][g][0] = __hip_atomic_load(at(pf - fo, unsigned(o)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          if (o < fu)
            xf[b][g][1] = __hip_atomic_load(at(pf + fo, unsigned(o)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      };
      if constexpr (FAR)
        far_ask(0, 0);
      constexpr int G = S < 2 || NU > 4 || (KEEP && S == 8 && NU == 4) ? 1 : 2; // slots whose loads are in flight together
#pragma unroll
      for (int s0 = 0; s0 < S; s0 += G) {
        double ml[G][MU], mu[G][MU], xl[G][MU], xu[G][MU], xc[G];
        constexpr int FB = 2;
        const int fb = (s0 / FB) & 1;
        if constexpr (FAR)
          if (s0 + G < S)
            far_ask(s0 + G, fb ^ 1);
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const int s = s0 + g;
          if constexpr (KEEP) {
#pragma unroll
            for (int u = 0; u < NU; ++u)
              ml[g][u] = al[s][u], mu[g][u] = au[s][u];
          } else if constexpr (FAR) {
            // (entries past either end of the instance are read from the storage's padding, times p = 0)
#pragma unroll
            for (int u = 0; u < NU; ++u) {
              const double* col = P.scaled + int64_t(u) * n + K.row0 + s * T;
              ml[g][u] = *at(col - off[u], unsigned(l));
              mu[g][u] = *at(col, unsigned(l));
            }
          } else {
            const int oc = min(l + s * T, rows - 1);
#pragma unroll
            for (int u = 0; u < NU; ++u) {
              // (rows whose partner lies below the instance read the first valid entry, times p = 0)
              const double* col = P.scaled + int64_t(u < ku ? u : 0) * n + K.row0;
              ml[g][u] = *at(col - min(off[u], below), unsigned(max(oc - max(off[u] - below, 0), 0)));
              mu[g][u] = *at(col, unsigned(oc));
              if (off[u] <= 0)
                ml[g][u] = mu[g][u] = 0.;
            }
          }
#pragma unroll
          for (int u = 0; u < NN; ++u)
            xl[g][u] = pd[u][s * T], xu[g][u] = pu[u][s * T];
          xc[g] = pt[s * T];
        }
        if constexpr (FAR) {
#pragma unroll
          for (int g = 0; g < G; ++g)
            xl[g][NU - 1] = xf[fb][g][0], xu[g][NU - 1] = xf[fb][g][1];
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const int s = s0 + g;
          double a = 0.;
#pragma unroll
          for (int u = NU - 1; u >= 0; --u)
            a = fma(ml[g][u], xl[g][u], a);
          a += xc[g];
#pragma unroll
          for (int u = 0; u < NU; ++u)
            a = fma(mu[g][u], xu[g][u], a);
          if (!KEEP && !whole)
            a = l + s * T < rows ? a : 0.;
          take(s, xc[g], a);
        }
        if constexpr (!KEEP)
          asm volatile("" ::: "memory"); // no more matrix loads in flight than there are registers for
      }
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      const int par = it & 1, set = it % 3;
      double sv[SQMEM ? S : 1];
      if constexpr (SQMEM)
#pragma unroll
        for (int s = 0; s < S; ++s)
          sv[s] = *at(P.dsq + K.row0, unsigned(min(l + s * T, rows - 1)));
      double tot1[1];
      if (single) {
        tot1[0] = add_run(ga, SAME ? vwaves : P.a_rows >> 6);
      } else {
        double own1[1] = {0.};
        if (l < own_na) {
          const int g = SAME ? vwaves : P.a_rows >> 6;
          own1[0] = add_run(ga + l * g, g);
          if (!alone) {
            slot_store(at(P.g1 + (set * P.n_a + K.own_a) * RES_PAD, unsigned(l) * RES_PAD), own1[0]);
            slot_clear(at(P.g1 + ((it + 2) % 3 * P.n_a + K.own_a) * RES_PAD, unsigned(l) * RES_PAD));
          }
        }
        if (!exchange_sum<1, NW>(P.g1 + (set * P.n_a + K.a0) * RES_PAD, own1, alone, K.na, P.v_block, red1, &failed,
                                 P.gave_up, P.wait_ticks, tot1))
          return;
      }
      pq = tot1[0];
      if (!uniform(pq > 0.)) { // breakdown: the iterate holds every earlier step
        state = 3;
        break;
      }
      // update of r, the rows other workgroups read, the partials of the residual norms
      alpha = rho / pq;
      double v[2] = {0., 0.};
      double* const to = P.r_pub[par] + K.row0;
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const double ri = fma(-alpha, QLDS ? ql[s * T] : q[QLDS ? 0 : s], r[s]);
        r[s] = ri;
        if (!FAR && !alone) {
          const int o = l + s * T;
          if (SELL ? (pub >> s) & 1u : o < pub_lo || o >= pub_hi)
            slot_store(at(to, unsigned(o)), ri);
        }
        const double ru = (SQMEM ? sv[SQMEM ? s : 0] : sq[SQMEM ? 0 : s]) * ri;
        v[0] = fma(ri, ri, v[0]), v[1] = fma(ru, ru, v[1]);
        if (s % ITEMS == ITEMS - 1) {
          const double w0 = wave_sum(v[0]), w1 = wave_sum(v[1]);
          if ((l & 63) == 0)
            gv[0][(s >> LG) * NW + wave] = w0, gv[1][(s >> LG) * NW + wave] = w1;
          v[0] = v[1] = 0.;
        }
      }
      __syncthreads();
      double own2[2] = {0., 0.};
      if (single) {
        rn[0] = add_run(gv[0], vwaves), rn[1] = add_run(gv[1], vwaves);
      } else if (l < own_nv) {
        own2[0] = add_run(gv[0] + l * vwaves, vwaves), own2[1] = add_run(gv[1] + l * vwaves, vwaves);
        if (!alone) {
          double* mine = at(P.g2 + (par * P.n_v + K.own_v) * RES_PAD, unsigned(l) * RES_PAD);
          slot_store(mine, own2[0]), slot_store(mine + 1, own2[1]);
        }
      }
      // in the time the exchange takes: x, the next step's slots and rows emptied, and the halo's rows of r asked for
      // (empty where their workgroup is not that far)
      if constexpr (XMEM) {
        double xv[S];
#pragma unroll
        for (int s = 0; s < S; ++s)
          xv[s] = *at(P.x_out + K.row0, unsigned(min(l + s * T, rows - 1)));
#pragma unroll
        for (int s = 0; s < S; ++s)
          if (l + s * T < rows)
            *at(P.x_out + K.row0, unsigned(l + s * T)) = fma(alpha, pt[s * T], xv[s]);
      } else {
#pragma unroll
        for (int s = 0; s < S; ++s)
          x[s] = fma(alpha, pt[s * T], x[s]);
      }
      if (!alone) {
        if (l < own_nv) {
          double* next = at(P.g2 + ((par ^ 1) * P.n_v + K.own_v) * RES_PAD, unsigned(l) * RES_PAD);
          slot_clear(next), slot_clear(next + 1);
        }
        if constexpr (!FAR) {
          double* const next = P.r_pub[par ^ 1] + K.row0;
#pragma unroll
          for (int s = 0; s < S; ++s) {
            const int o = l + s * T;
            if (SELL ? (pub >> s) & 1u : o < pub_lo || o >= pub_hi)
              slot_clear(at(next, unsigned(o)));
          }
        }
      }
      if (!alone && !FAR) {
        const double* from = P.r_pub[par] + (SELL ? 0 : K.row0 - below);
#pragma unroll
        for (int k = 0; k < RES_HALO; ++k) {
          const int e = l + k * T;
          if (e < nhalo)
            halo[k] = slot_load(at(from, unsigned(SELL ? hr[k] : e < below ? e : rows + e)));
        }
      }
      if (!single && !exchange_sum<2, NW>(P.g2 + (par * P.n_v + K.v0) * RES_PAD, own2, alone, K.nv, P.v_block, red2, &failed,
                                          P.gave_up, P.wait_ticks, rn))
        return;
    }
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int o = t + s * T;
      if (!XMEM && o < rows)
        P.x_out[K.row0 + o] = x[XMEM ? 0 : s];
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

// every slot and published row empty
__global__ void __launch_bounds__(256) k_resident_clear(ResidentParams P, int64_t slots)
{
  const double empty = __longlong_as_double((long long)RES_EMPTY);
  constexpr int FLAGS = RES_MAX_GROUPS;
  const int64_t i = xcd_index(max(max(P.n, slots), int64_t(FLAGS)));
  if (i < slots)
    P.g1[i] = empty;
  if (i < P.n)
    P.r_pub[0][i] = empty, P.r_pub[1][i] = empty;
  if (i < FLAGS)
    P.flags[i] = 0;
  if (i == 0)
    *P.gave_up.device = 0;
}

using Kernel = void (*)(ResidentParams);

// compiled variants: vector and operator blocks of 512 lanes with as many rows per lane as there are slots (the
// default shapes); any vector and operator blocks with one row per lane (shapes set by the caller)
template <int NU>
Kernel kernel_for(int slots, int lg, bool same)
{
  if (same)
    switch (slots * 16 + lg) {
      case 16:
        return k_pcg_resident<RES_LANES, 1, 0, true, NU, 1>;
      case 33:
        return k_pcg_resident<RES_LANES, 2, 1, true, NU, 1>;
      case 66:
        return k_pcg_resident<RES_LANES, 4, 2, true, NU, 1>;
      case 131:
        return k_pcg_resident<RES_LANES, 8, 3, true, NU, 1>;
      case 259:
        return k_pcg_resident<RES_LANES, 16, 3, true, NU, 0>;
    }
  if (lg == 0)
    switch (slots) {
      case 1:
        return k_pcg_resident<RES_LANES, 1, 0, false, NU, 1>;
      case 2:
        return k_pcg_resident<RES_LANES, 2, 0, false, NU, 1>;
      case 4:
        return k_pcg_resident<RES_LANES, 4, 0, false, NU, 1>;
      case 8:
        return k_pcg_resident<RES_LANES, 8, 0, false, NU, 1>;
    }
  return nullptr;
}

// up to RES_WIDE strict upper slots (Q1 on hexahedra): the matrix is read in every step
constexpr int RES_WIDE = 13;
Kernel wide_kernel(int slots, int lg, bool same)
{
  if (same)
    switch (slots * 16 + lg) {
      case 16:
        return k_pcg_resident<RES_LANES, 1, 0, true, RES_WIDE, 0>;
      case 33:
        return k_pcg_resident<RES_LANES, 2, 1, true, RES_WIDE, 0>;
      case 66:
        return k_pcg_resident<RES_LANES, 4, 2, true, RES_WIDE, 0>;
    }
  return nullptr;
}

// FAR: blocks of RES_FAR_BLOCK lanes and 4 rows per lane
Kernel far_kernel(int slots)
{
  return slots == 4 ? k_pcg_resident<RES_FAR_BLOCK, 4, 2, true, 3, 1, true>
         : slots == 8 ? k_pcg_resident<RES_FAR_BLOCK, 8, 2, true, 3, 0, true>
                      : k_pcg_resident<RES_FAR_BLOCK, 12, 2, true, 3, 0, true>;
}

// nu < 0: SELL, slices of at most -nu entries per row
Kernel kernel_of(int slots, int lg, bool same, int nu)
{
  if (nu < 0) {
    if (!same || (1 << lg) != slots)
      return nullptr;
    const int w = -nu;
    switch (slots) {
      case 1:
        return w <= 28 ? k_pcg_resident<RES_LANES, 1, 0, true, 0, 28> : k_pcg_resident<RES_LANES, 1, 0, true, 0, 0>;
      case 2:
        return w <= 12 ? k_pcg_resident<RES_LANES, 2, 1, true, 0, 12> : w <= 28 ? k_pcg_resident<RES_LANES, 2, 1, true, 0, 28>
                                                                       : k_pcg_resident<RES_LANES, 2, 1, true, 0, 0>;
      case 4:
        return w <= 12 ? k_pcg_resident<RES_LANES, 4, 2, true, 0, 12> : k_pcg_resident<RES_LANES, 4, 2, true, 0, 0>;
      case 8:
        return k_pcg_resident<RES_LANES, 8, 3, true, 0, 0>;
    }
    return nullptr;
  }
  return nu <= 3 ? kernel_for<3>(slots, lg, same) : nu <= 4 ? kernel_for<4>(slots, lg, same) : wide_kernel(slots, lg, same);
}

// CUs of a device in use by resident launches of this process
class CuBudget {
  std::mutex m_;
  std::condition_variable cv_;
  std::map<int, int> used_;

public:
  static CuBudget& get()
  {
    static CuBudget* b = new CuBudget; // never destroyed: solves may run while the process ends
    return *b;
  }
  void take(int device, int count, int total)
  {
    std::unique_lock<std::mutex> l(m_);
    cv_.wait(l, [&] { return used_[device] + count <= total; });
    used_[device] += count;
  }
  void give(int device, int count)
  {
    std::lock_guard<std::mutex> l(m_);
    used_[device] -= count;
    cv_.notify_all();
  }
};

int device_cus()
{
  int dev = 0, cus = 0;
  HGDT_HIP(hipGetDevice(&dev));
  HGDT_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  return cus;
}

} // namespace

static int64_t team_of(int64_t rows, int slots, int lanes = RES_LANES)
{
  const int64_t R = int64_t(slots) * lanes;
  return (rows + R - 1) / R;
}

// Whether a single instance takes `slots` rows per lane (the smallest are asked first): few workgroups keep the exchanges
// short, few rows the steps between them.  Measured (Q1, us per iteration with 1 / 2 / 4 / 8 rows per lane): 1 089 rows
// 4.5 / 4.2 / 2.7 / 4.3 (one workgroup: no exchange); 4 096 4.2 / 3.9 / 4.3 / 4.4; 16 384 5.0 / 4.4 / 5.0 / 6.2; 65 536 6.4 / 5.3 / 5.3 / 6.7; 131 044 8.0 / 7.9 / 5.7 / 7.1;
// 262 144 - / - / 7.8 / 7.5.  SELL: 160 401 rows of 7 entries - / 8.5 / 7.6 / 13.4, 90 201 of 11 8.6 / 8.0 / 14.8 / 23
// More than 4 upper slots (hexahedra): 1 000 rows 6.6 / 4.6 / 7.5, 2 197 6.8 / 8.1 / 10.9, 19 683 7.1 / 8.4 / 11.0, 35 937
// 9.3 / 9.2 / 11.7, 68 921 12.5 / 10.5 / 12.2, 132 651 - / 14.8 / 13.8 / 20.7, 300 763 - / - / 17.2 / 23.0 (three kernels:
// 13.6, 15.7, 15.7, 15.1, 16.0, 17.9, 25); 8 rows per lane are not compiled.
enum RowKind { ROWS_DIA, ROWS_WIDE, ROWS_SELL };
static bool enough_rows(int64_t rows, int slots, int cus, RowKind kind)
{
  const int64_t w = team_of(rows, slots);
  if (kind == ROWS_WIDE)
    return slots == 1 ? w <= 1 || (w > 2 && w <= cus / 5) : slots == 2 ? w <= cus / 3 : w <= cus;
  if (kind == ROWS_SELL) // (a row costs more: 9 to 20 scattered reads of LDS)
    return slots == 1 ? w <= cus / 16 : slots <= 4 ? w <= cus / 2 : w <= cus;
  return slots == 1 ? w <= 1 : slots == 2 ? w <= (rows <= 4 * RES_LANES ? 1 : cus / 8) : slots == 4 ? w <= cus / 4 : w <= cus;
}

double resident_schedule(const std::vector<int64_t>& row0, const std::vector<int>& teams, double step,
                         std::vector<int>* order, std::vector<std::vector<int>>* groups)
{
  const int cus = device_cus(), ninst = int(teams.size());
  std::vector<int> by_size(ninst);
  for (int i = 0; i < ninst; ++i)
    by_size[i] = i;
  std::stable_sort(by_size.begin(), by_size.end(),
                   [&](int a, int b) { return row0[a + 1] - row0[a] > row0[b + 1] - row0[b]; });
  std::vector<std::pair<double, int>> load(cus); // (time it is free, workgroup)
  for (int w = 0; w < cus; ++w)
    load[w] = {0., w};
  if (groups)
    groups->assign(ninst, {});
  double last = 0.;
  for (int i : by_size) {
    const int team = teams[i];
    if (team > cus || team > RES_MAX_GROUPS)
      return -1.;
    std::partial_sort(load.begin(), load.begin() + team, load.end());
    // iterations grow like the square root of the size (two dimensions)
    const double end = load[team - 1].first +
                       std::sqrt(double(row0[i + 1] - row0[i])) * (step + (team > 1 ? 2.6 + 0.01 * double(team) : 0.));
    for (int k = 0; k < team; ++k) {
      load[k].first = end;
      if (groups)
        (*groups)[i].push_back(load[k].second);
    }
    last = std::max(last, end);
  }
  if (order)
    *order = by_size;
  return last;
}

// us per iteration of one workgroup with 1, 2, 4, 8, 16 rows per lane (measured)
static double step_of(int slots, RowKind kind = ROWS_DIA)
{
  if (kind == ROWS_WIDE)
    return slots == 1 ? 3.3 : slots == 2 ? 4.6 : 7.5;
  return slots == 1 ? 1.8 : slots == 2 ? 2.1 : slots == 4 ? 2.7 : slots == 8 ? 4.3 : 10.;
}

// rows per lane: -1 when no choice of `fits` (LDS, compiled variant) takes all instances
template <class F>
static int choose_slots(const std::vector<int64_t>& row0, RowKind kind, bool given, F fits)
{
  const int cus = device_cus();
  int best = -1;
  double time = 0.;
  for (int s : {1, 2, 4, 8, 16}) {
    if (row0.size() == 2) {
      if (enough_rows(row0[1] - row0[0], s, cus, kind) && fits(s))
        return s;
      continue;
    }
    std::vector<int> teams;
    for (size_t i = 0; i + 1 < row0.size(); ++i)
      teams.push_back(int(std::min<int64_t>(team_of(row0[i + 1] - row0[i], s), 1 << 20)));
    const double t = resident_schedule(row0, teams, step_of(s, kind), nullptr, nullptr);
    if (t >= 0. && (best < 0 || t < time) && fits(s))
      best = s, time = t;
  }
  // row blocks that the caller chose: any number of workgroups that fits
  for (int s : {1, 2, 4, 8, 16})
    if (given && best < 0 && row0.size() == 2 && team_of(row0[1] - row0[0], s) <= cus && fits(s))
      best = s;
  return best;
}

// doubles a stencil reaches to either side of a row
static int64_t reach_of(const std::vector<int64_t>& row0, const std::vector<std::vector<int64_t>>& s_offs)
{
  int64_t reach = 0;
  for (size_t in = 0; in + 1 < row0.size(); ++in)
    for (int64_t o : s_offs[in])
      if (o < row0[in + 1] - row0[in])
        reach = std::max(reach, o);
  return reach;
}

static int64_t lds_of(int slots, int64_t reach, int s_nu)
{
  return (int64_t(slots) * RES_LANES * (q_in_lds(slots, s_nu <= 3 ? 3 : 4, false) ? 2 : 1) + 2 * reach) *
         int64_t(sizeof(double));
}
static int64_t far_lds(int slots, int64_t near)
{
  return (int64_t(slots) * RES_FAR_BLOCK * 2 + 2 * near) * int64_t(sizeof(double));
}

// FAR: one instance of three offsets, the outermost past what LDS holds; rows per lane (0: not this case)
static int far_slots(const std::vector<int64_t>& row0, const std::vector<std::vector<int64_t>>& s_offs, int s_nu)
{
  if (row0.size() != 2 || s_nu != 3 || s_offs[0].size() != 3 || s_offs[0][2] >= row0[1] - row0[0])
    return 0;
  for (int s : {4, 8, 12})
    if (team_of(row0[1], s, RES_FAR_BLOCK) <= device_cus() && far_lds(s, s_offs[0][1]) <= RES_LDS)
      return s;
  return 0;
}

int64_t resident_padding(const std::vector<int64_t>& row0, const std::vector<std::vector<int64_t>>& s_offs, int s_nu)
{
  if (!far_slots(row0, s_offs, s_nu))
    return 0;
  return std::max<int64_t>(s_offs[0].back(), int64_t(12) * RES_FAR_BLOCK);
}

ResidentShape resident_shape_dia(const std::vector<int64_t>& row0, const std::vector<std::vector<int64_t>>& s_offs,
                                 int s_nu)
{
  if (s_nu < 0 || s_nu > RES_WIDE)
    return {};
  const int64_t reach = reach_of(row0, s_offs);
  const int s = choose_slots(row0, s_nu > 4 ? ROWS_WIDE : ROWS_DIA, false, [&](int k) {
    return lds_of(k, reach, s_nu) <= RES_LDS && !(s_nu == 0 && k > 8) && !(s_nu > 4 && k > 4);
  });
  if (s > 0)
    return {RES_LANES, std::min(s, 8)}; // (16 rows per lane: two blocks of 8 each)
  if (far_slots(row0, s_offs, s_nu))
    return {RES_FAR_BLOCK, 4};
  return {};
}

// one workgroup's rows after the other, instance by instance; false when the lanes that add the partials of an
// instance of one workgroup do not hold them all
static bool list_tasks(const Operator& op, int slots, int lanes, std::vector<ResidentTask>& tasks)
{
  const SolverFormat& F = op.fmt;
  const std::vector<int64_t>& row0 = op.space->inst_dof;
  const int64_t R = int64_t(slots) * lanes, va = int64_t(F.A.block) * F.A.items, vv = int64_t(F.V.block) * F.V.items;
  for (size_t in = 0; in + 1 < row0.size(); ++in) {
    const int64_t ni = row0[in + 1] - row0[in];
    const int team = int((ni + R - 1) / R);
    for (int k = 0; k < team; ++k) {
      ResidentTask K{};
      K.row0 = row0[in] + k * R;
      K.rows = int32_t(std::min(R, ni - k * R));
      K.inst = int32_t(in), K.team = team, K.rank = k;
      K.a0 = F.A.inst_block0[in], K.na = F.A.inst_block0[in + 1] - K.a0;
      K.v0 = F.V.inst_block0[in], K.nv = F.V.inst_block0[in + 1] - K.v0;
      K.own_a = K.a0 + int32_t(k * R / va), K.own_v = K.v0 + int32_t(k * R / vv);
      K.mask = int32_t(tasks.size());
      if (ni == 0 || (team == 1 && (K.na > F.V.block || K.nv > F.V.block)))
        return false;
      tasks.push_back(K);
    }
  }
  return true;
}

void resident_finish(ResidentPlan& plan, const Operator& op, const std::vector<ResidentTask>& tasks, int64_t lds,
                     int64_t n_a, int64_t n_v)
{
  std::vector<int> order, teams(op.space->inst_dof.size() - 1, 0);
  std::vector<std::vector<int>> groups;
  for (const auto& K : tasks)
    teams[K.inst] = K.team;
  if (resident_schedule(op.space->inst_dof, teams, plan.step, &order, &groups) < 0.)
    return;
  std::vector<int64_t> first(groups.size(), 0); // first task of every instance
  for (size_t k = tasks.size(); k-- > 0;)
    first[tasks[k].inst] = int64_t(k);
  std::vector<std::vector<ResidentTask>> of;
  for (int i : order)
    for (size_t k = 0; k < groups[i].size(); ++k) {
      if (groups[i][k] >= int(of.size()))
        of.resize(groups[i][k] + 1);
      of[groups[i][k]].push_back(tasks[first[i] + int64_t(k)]);
    }
  // consecutive workgroups on one XCD (hardware deals them round-robin to 8), as neighbours exchange their halos
  plan.workgroups = int(of.size());
  const size_t q = (of.size() + 7) / 8;
  of.resize(8 * q);
  std::vector<std::vector<ResidentTask>> dealt(8 * q);
  for (size_t w = 0; w < 8 * q; ++w)
    dealt[(w % q) * 8 + w / q] = std::move(of[w]);
  of = std::move(dealt);
  std::vector<ResidentTask> list;
  std::vector<int32_t> start{0};
  for (auto& w : of) {
    list.insert(list.end(), w.begin(), w.end());
    start.push_back(int32_t(list.size()));
  }
  plan.grid = int(of.size()), plan.lds = lds;
  plan.tasks.upload(list);
  plan.task_start.upload(start);
  plan.n_a = n_a, plan.n_v = n_v;
  plan.exchanges = std::any_of(teams.begin(), teams.end(), [](int t) { return t > 1; });
  // (the first workgroup has the first rows of the largest instance, so others wait for it if any wait at all)
  start[0] = start[1];
  plan.start_without = std::move(start);
  plan.d_start_without.release();
  plan.cus = device_cus();
  plan.kernel = plan.dg ? resident_dg_kernel(plan)
                        : reinterpret_cast<const void*>(plan.far ? far_kernel(plan.slots)
                                                                 : kernel_of(plan.slots, plan.lg_items, plan.same_blocks,
                                                                             plan.nu));
  HGDT_HIP(hipFuncSetAttribute(plan.kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int(RES_LDS)));
  plan.exchange.allocate(size_t(RES_PAD * (3 * n_a + 2 * n_v)));
  plan.gave_up.upload(std::vector<int>(1 + RES_MAX_GROUPS, 0));
  if (!plan.host_gave_up)
    HGDT_HIP(hipHostMalloc((void**)&plan.host_gave_up, sizeof(int)));
  plan.usable = true;
}

void resident_plan_dia(ResidentPlan& plan, const Operator& op, const std::vector<std::vector<int64_t>>& s_offs,
                       int s_nu)
{
  plan.usable = false;
  const SolverFormat& F = op.fmt;
  const int bv = F.V.block, iv = F.V.items, ba = F.A.block * F.A.items;
  plan.sell = plan.far = plan.dg = false;
  plan.lanes = RES_LANES;
  if (bv == RES_FAR_BLOCK && iv == 4 && F.A.block == bv && F.A.items == iv) {
    const int slots = far_slots(op.space->inst_dof, s_offs, s_nu);
    std::vector<ResidentTask> tasks;
    if (!slots || !list_tasks(op, slots, RES_FAR_BLOCK, tasks))
      return;
    plan.far = true;
    plan.lanes = RES_FAR_BLOCK;
    plan.slots = slots, plan.lg_items = 2, plan.same_blocks = true, plan.nu = s_nu;
    plan.step = step_of(plan.slots);
    resident_finish(plan, op, tasks, far_lds(slots, s_offs[0][1]), F.A.nblocks, F.V.nblocks);
    return;
  }
  const bool same = bv == RES_LANES && F.A.block == bv && F.A.items == iv;
  if (s_nu < 0 || s_nu > RES_WIDE || RES_LANES % bv != 0 || !(same || (F.A.items == 1 && ba <= 1024 && (ba & (ba - 1)) == 0)))
    return;
  const std::vector<int64_t>& row0 = op.space->inst_dof;
  int lg = 0;
  while ((1 << lg) < iv)
    ++lg;
  if (lg > 0 && bv != RES_LANES)
    return;
  const int64_t reach = reach_of(row0, s_offs);
  const int slots = choose_slots(row0, s_nu > 4 ? ROWS_WIDE : ROWS_DIA, true, [&](int k) {
    // (a diagonal matrix holds no slot to stream)
    return (int64_t(k) * RES_LANES) % ba == 0 && kernel_of(k, lg, same, s_nu) && lds_of(k, reach, s_nu) <= RES_LDS &&
           !(s_nu == 0 && k > 8);
  });
  if (slots < 0)
    return;
  std::vector<ResidentTask> tasks;
  if (!list_tasks(op, slots, RES_LANES, tasks))
    return;
  plan.slots = slots, plan.lg_items = lg, plan.same_blocks = same, plan.nu = s_nu;
  plan.step = step_of(plan.slots, s_nu > 4 ? ROWS_WIDE : ROWS_DIA);
  resident_finish(plan, op, tasks, lds_of(slots, reach, s_nu), F.A.nblocks, F.V.nblocks);
}

// Columns of a block of rows that lie outside it, ascending, and the place of each in this list, by a table over the rows
// of an instance (at most what 256 workgroups hold).  All entries listed and sorted, and a search per entry, took 34 ms of
// the first solve of P2 on 300 x 350 x 2 triangles (60 ms with three steps), the tables take 12.
class Halo {
  const Operator& op_;
  std::vector<int32_t> place_; // -1: not in the list
  int64_t lo_ = 0;             // first row of the instance

public:
  std::vector<int32_t> list;
  explicit Halo(const Operator& op)
    : op_(op)
  {
  }
  // rows [r0, r1) of the instance with the rows [lo, hi); false: a column of another instance (a caller's matrix)
  bool of(int64_t r0, int64_t r1, int64_t lo, int64_t hi)
  {
    for (int32_t c : list)
      place_[c - lo_] = -1;
    list.clear();
    lo_ = lo;
    if (int64_t(place_.size()) < hi - lo)
      place_.resize(hi - lo, -1);
    for (int64_t k = op_.row_ptr[r0]; k < op_.row_ptr[r1]; ++k) {
      const int32_t c = op_.cols[k];
      if (c < lo || c >= hi)
        return false;
      if ((c < r0 || c >= r1) && place_[c - lo] < 0)
        place_[c - lo] = 0, list.push_back(c);
    }
    std::sort(list.begin(), list.end());
    for (size_t i = 0; i < list.size(); ++i)
      place_[list[i] - lo] = int32_t(i);
    return true;
  }
  int32_t place(int32_t c) const
  {
    return place_[c - lo_];
  }
};

int resident_items_sell(const Operator& op)
{
  if (!reached_by_32_bits(op.n))
    return 0;
  const std::vector<int64_t>& row0 = op.space->inst_dof;
  const int s = choose_slots(row0, ROWS_SELL, false, [&](int k) {
    if (k > 8)
      return false;
    // p of the own rows and the halo in LDS
    const int64_t R = int64_t(k) * RES_LANES;
    std::vector<std::pair<int64_t, size_t>> blocks; // first row, instance
    for (size_t in = 0; in + 1 < row0.size(); ++in)
      for (int64_t r = row0[in]; r < row0[in + 1]; r += R)
        blocks.push_back({r, in});
    std::atomic<int64_t> most{0};
    parallel_for(int64_t(blocks.size()), [&](int64_t b0, int64_t b1) {
      Halo halo(op);
      for (int64_t b = b0; b < b1; ++b) {
        const int64_t r = blocks[b].first, lo = row0[blocks[b].second], hi = row0[blocks[b].second + 1];
        const int64_t size = halo.of(r, std::min(r + R, hi), lo, hi) ? int64_t(halo.list.size()) : RES_LDS;
        int64_t m = most;
        while (m < size && !most.compare_exchange_weak(m, size))
          ;
      }
    });
    return (R + most) * int64_t(sizeof(double)) <= RES_LDS;
  });
  return std::max(s, 0);
}

void resident_plan_sell(ResidentPlan& plan, const Operator& op)
{
  plan.usable = false;
  const SolverFormat& F = op.fmt;
  const int slots = F.V.items;
  if (F.V.block != RES_LANES || F.A.block != RES_LANES || F.A.items != slots || slots > RES_MAX_SLOTS ||
      !reached_by_32_bits(op.n))
    return;
  int lg = 0;
  while ((1 << lg) < slots)
    ++lg;
  if (!kernel_of(slots, lg, true, -1))
    return;
  std::vector<ResidentTask> tasks;
  if (!list_tasks(op, slots, RES_LANES, tasks))
    return;
  const int64_t R = int64_t(slots) * RES_LANES, nt = int64_t(tasks.size());
  const std::vector<int64_t>& row0 = op.space->inst_dof;
  std::vector<int64_t> slice_ptr(F.nslices + 1);
  F.d_slice_ptr.download(slice_ptr.data());
  int64_t slices = 0;
  for (ResidentTask& K : tasks) {
    K.slice0 = int32_t(slices);
    slices += (K.rows + 63) / 64;
  }
  if (slices != F.nslices)
    return;
  std::vector<std::vector<int32_t>> halo(nt);
  std::vector<uint16_t> local(std::max<size_t>(F.d_sell_vals.count, 1), 0);
  std::atomic<bool> fits{true};
  parallel_for(nt, [&](int64_t b0, int64_t b1) {
    Halo h(op);
    for (int64_t b = b0; b < b1 && fits; ++b) {
      const ResidentTask& K = tasks[b];
      if (!h.of(K.row0, K.row0 + K.rows, row0[K.inst], row0[K.inst + 1]) ||
          (R + int64_t(h.list.size())) * int64_t(sizeof(double)) > RES_LDS) {
        fits = false;
        return;
      }
      halo[b] = h.list;
      for (int o = 0; o < K.rows; ++o) {
        const int64_t i = K.row0 + o;
        const int64_t sl = K.slice0 + o / 64;
        const int64_t w = (slice_ptr[sl + 1] - slice_ptr[sl]) / 64, len = op.row_ptr[i + 1] - op.row_ptr[i];
        for (int64_t k = 0; k < w; ++k) {
          int64_t at = o; // padding: the own row, as the columns of the storage
          if (k < len) {
            const int32_t c = op.cols[op.row_ptr[i] + k];
            at = (c >= K.row0 && c < K.row0 + K.rows) ? c - K.row0 : R + h.place(c);
          }
          local[slice_ptr[sl] + k * 64 + o % 64] = uint16_t(at);
        }
      }
    }
  });
  if (!fits)
    return;
  // the rows that other workgroups read
  std::vector<uint8_t> read(std::max<int64_t>(op.n, 1), 0);
  std::vector<int32_t> rows;
  int64_t most = 0;
  for (int64_t b = 0; b < nt; ++b) {
    tasks[b].halo0 = int32_t(rows.size()), tasks[b].nhalo = int32_t(halo[b].size());
    most = std::max<int64_t>(most, tasks[b].nhalo);
    for (int32_t c : halo[b])
      read[c] = 1;
    rows.insert(rows.end(), halo[b].begin(), halo[b].end());
  }
  std::vector<uint32_t> pub(nt * RES_LANES, 0u);
  parallel_for(nt, [&](int64_t b0, int64_t b1) {
    for (int64_t b = b0; b < b1; ++b)
      for (int o = 0; o < tasks[b].rows; ++o)
        if (read[tasks[b].row0 + o])
          pub[b * RES_LANES + o % RES_LANES] |= 1u << (o / RES_LANES);
  });
  plan.sell_local.upload(local);
  if (rows.empty())
    rows.push_back(0);
  plan.halo_rows.upload(rows);
  plan.publish.upload(pub);
  plan.sell = true, plan.far = plan.dg = false;
  plan.lanes = RES_LANES;
  int64_t widest = 1;
  for (int64_t k = 0; k < F.nslices; ++k)
    widest = std::max(widest, (slice_ptr[k + 1] - slice_ptr[k]) / 64);
  plan.slots = slots, plan.lg_items = lg, plan.same_blocks = true, plan.nu = -int(std::min<int64_t>(widest, 1 << 20));
  plan.step = step_of(plan.slots);
  resident_finish(plan, op, tasks, (R + most) * int64_t(sizeof(double)), F.A.nblocks, F.V.nblocks);
}

ResidentLaunch::ResidentLaunch(ResidentPlan& plan, ResidentParams P, const MfParams& M, hipStream_t stream)
  : stream_(stream)
{
  P.n_a = plan.n_a, P.n_v = plan.n_v;
  P.dg_elements = plan.elements.ptr, P.zero_place = plan.zero_place;
  P.g1 = plan.exchange.ptr;
  P.g2 = plan.exchange.ptr + 3 * P.n_a * RES_PAD;
  P.sell_local = plan.sell_local.ptr, P.halo_rows = plan.halo_rows.ptr, P.publish = plan.publish.ptr;
  P.tasks = plan.tasks.ptr, P.task_start = plan.task_start.ptr;
  P.gave_up = {plan.gave_up.ptr, plan.host_gave_up}, P.flags = plan.gave_up.ptr + 1;
  if (P.wait_ticks == 0 && plan.exchanges) {
    if (!plan.d_start_without.ptr)
      plan.d_start_without.upload(plan.start_without);
    P.task_start = plan.d_start_without.ptr;
  }
  *plan.host_gave_up = 0;
  const int64_t nx = int64_t(plan.exchange.count);
  if (plan.exchanges)
    hipLaunchKernelGGL(k_resident_clear, dim3(xcd_grid(std::max<int64_t>(std::max(P.n, nx), RES_MAX_GROUPS), 256)),
                       dim3(256), 0, stream, P, nx);
  HGDT_HIP(hipGetLastError());
  HGDT_HIP(hipGetDevice(&device_));
  held_ = std::min(plan.grid, plan.cus);
  CuBudget::get().take(device_, held_, plan.cus);
  MfParams Mk = M;
  void* args[2] = {&P, &Mk}; // (the second: discontinuous spaces)
  const hipError_t e =
      hipLaunchKernel(plan.kernel, dim3(unsigned(plan.grid)), dim3(unsigned(plan.lanes)), args, size_t(plan.lds), stream);
  if (e != hipSuccess)
    CuBudget::get().give(device_, held_);
  HGDT_HIP(e);
}

ResidentLaunch::~ResidentLaunch()
{
  (void)hipStreamSynchronize(stream_); // the CUs are given back with none of its workgroups running
  CuBudget::get().give(device_, held_);
}

bool resident_gave_up(ResidentPlan& plan)
{
  if (!__atomic_load_n(plan.host_gave_up, __ATOMIC_ACQUIRE))
    return false;
  plan.skip = 16; // (whoever holds the CUs may do so for a while, and a wait costs seconds)
  return true;
}

} // namespace hgdt
