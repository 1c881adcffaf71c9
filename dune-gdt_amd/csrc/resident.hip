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
// workgroup and all others (2.4-3.5 us with 256 workgroups, 1-1.3 us with 16).  Two sets of slots alternate, by the
// parity of the step: a workgroup puts the sentinel back into its slots of the other set when it stores to one;
// by then every workgroup has read that other set (it stored to the exchange in between afterwards), and none
// polls it again before this workgroup has stored to that exchange, which it does after waiting for its
// earlier stores.  Slots, published rows and polls are relaxed atomics at agent scope (the XCDs' L2 caches
// are coherent for these); a workgroup waits for its published rows (vmcnt 0) before the barrier ahead of the
// store of its partials, so whoever has seen the partials sees the rows.
//
// Every value is computed by the operations of the three kernels in their order (row sums, block partials in
// the operator's and the vector partition, sums over the partials), so a solve gives the same bits on either path,
// alone or in a batch.
//
// All workgroups of a team must be on the chip together: the host launches at most one per CU and counts the
// CUs of all running launches of the process.  A wait that outlasts its limit (another process holds the
// CUs) sets a flag at which every workgroup ends; the caller then solves with the three kernels.

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <map>
#include <mutex>

#include "block_reduce.hpp"
#include "resident.hpp"

namespace hgdt {
namespace {

constexpr int RES_LANES = 512, RES_WAVES = RES_LANES / 64;
constexpr int RES_MAX_SLOTS = 16;
constexpr int RES_GROUPS = RES_WAVES * RES_MAX_SLOTS; // 64-row groups of a workgroup
constexpr int64_t RES_LDS = 150 * 1024;               // dynamic LDS of a workgroup, of 160 KB

// sentinel of the exchange slots: a NaN no sum produces (a NaN sum is stored as the default NaN)
constexpr unsigned long long RES_EMPTY = 0x7ff8dead00000001ull;

__device__ __forceinline__ void slot_store(double* p, double v)
{
  unsigned long long u = (unsigned long long)__double_as_longlong(v);
  if (v != v)
    u = 0x7ff8000000000000ull;
  __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void slot_clear(double* p)
{
  __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), RES_EMPTY, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long slot_load(const double* p)
{
  return __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void publish(double* p, double v)
{
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double published(const double* p)
{
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// waits until the slot holds a value; false when the wait is over its limit or another workgroup gave up
__device__ bool slot_wait(const double* p, int* gave_up, int64_t ticks, unsigned long long& u)
{
  const long long t0 = wall_clock64();
  for (int k = 1;; ++k) {
    __builtin_amdgcn_s_sleep(1);
    u = slot_load(p);
    if (u != RES_EMPTY)
      return true;
    if ((k & 255) == 0 && (__hip_atomic_load(gave_up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ||
                           wall_clock64() - t0 > ticks)) {
      __hip_atomic_store(gave_up, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return false;
    }
  }
}

// element `i` of an array whose base is the same for the whole wave: a 32-bit byte offset per lane
template <class T>
__device__ __forceinline__ T* at(T* base, unsigned i)
{
  return reinterpret_cast<T*>(reinterpret_cast<uintptr_t>(base) + i * unsigned(sizeof(T)));
}

// sums of `count` partials of NV values as Partials::sum adds them (lane t of `block` lanes adds the partials t,
// t + block, ...; then the waves' butterflies; then the waves in order), in every lane.  Partials come from the
// exchange slots, or (one workgroup, at most `block` partials: own) from the lane that computed them.  false:
// gave up.  One barrier; red is not written again before a later barrier.
template <int NV>
__device__ __forceinline__ bool exchange_sum(const double* slots, const double (&own)[NV], bool alone, int count,
                                             int block, double (*red)[RES_WAVES], int* failed, int* gave_up,
                                             int64_t ticks, double (&tot)[NV])
{
  constexpr int U = 4 / NV;
  const int t = threadIdx.x;
#pragma unroll
  for (int k = 0; k < NV; ++k)
    tot[k] = 0.;
  if (alone) {
    if (t < count)
#pragma unroll
      for (int k = 0; k < NV; ++k)
        tot[k] += own[k];
  } else if (t < block) {
    bool ok = true;
    for (int b = t; b < count && ok; b += U * block) {
      unsigned long long u[U][NV];
#pragma unroll
      for (int j = 0; j < U; ++j)
        if (b + j * block < count)
#pragma unroll
          for (int k = 0; k < NV; ++k)
            u[j][k] = slot_load(at(slots, unsigned(b + j * block) * NV + k));
#pragma unroll
      for (int j = 0; j < U; ++j)
        if (b + j * block < count)
#pragma unroll
          for (int k = 0; k < NV; ++k) {
            if (u[j][k] == RES_EMPTY)
              ok = ok && slot_wait(at(slots, unsigned(b + j * block) * NV + k), gave_up, ticks, u[j][k]);
            tot[k] += __longlong_as_double((long long)u[j][k]);
          }
    }
    if (!ok)
      *failed = 1;
  }
  const int nw = block >> 6;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const double w = wave_sum(tot[k]);
    if ((t & 63) == 0)
      red[k][t >> 6] = w;
  }
  __syncthreads();
  if (*failed)
    return false;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    double s = 0.;
    for (int w = 0; w < nw; ++w)
      s += red[k][w];
    tot[k] = s;
  }
  return true;
}

// PCG of the tasks of one workgroup, one after the other.  S rows per lane; lane t holds row j of its layer
// s >> lg (layers of RES_LANES << lg rows, lg the vector blocks' items): the rows of vector block (layer,
// t / v_block), lane t % v_block.  NU: strict upper slots compiled for (missing ones have zero values).  KEEP: the
// matrix rows stay in registers, else they are read every iteration.
template <int S, int NU, bool KEEP>
__global__ void __launch_bounds__(RES_LANES) k_pcg_resident(ResidentParams P)
{
  extern __shared__ double pl[]; // p of the own rows and `reach` rows to either side (0 outside the instance)
  __shared__ double ga[RES_GROUPS], gv[2][RES_GROUPS];
  __shared__ double red1[1][RES_WAVES], red2[2][RES_WAVES];
  __shared__ int failed;
  const int t = threadIdx.x, wave = t >> 6;
  const int lg = P.v_lg_items, items = 1 << lg;
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
    int off[NU];
    int reach = 0;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int64_t o = u < ku ? so[u] : 0; // padding slots: values 0, offset 0
      off[u] = o < hi - lo ? int(o) : 0;
      reach = max(reach, off[u]);
    }
    // row of slot s relative to the own rows: a lane's part and the slot's (the same in all lanes).  The lane's part
    // is made opaque in every step, so that the compiler does not keep S addresses of every array in registers
    int tb = (((t / P.v_block) * P.v_block) << lg) + t % P.v_block;
    auto row = [&](int s) { return (((s >> lg) * RES_LANES) << lg) + (s & (items - 1)) * P.v_block + tb; };
    const int below = int(min(K.row0 - lo, int64_t(reach)));        // rows of the instance below the own ones
    const int above = int(min(hi - K.row0 - rows, int64_t(reach))); // and above, at most `reach`
    double r[S], x[S], sq[S];
    double au[KEEP ? S : 1][NU], al[KEEP ? S : 1][NU];
    __syncthreads(); // the previous task's last reads of LDS
    for (int e = t; e < rows + 2 * reach; e += RES_LANES) {
      const int o = e - reach;
      pl[e] = (o >= -below && o < rows + above) ? P.r[K.row0 + o] : 0.;
    }
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int o = row(s);
      const int64_t i = K.row0 + o;
      const bool in = o < rows;
      r[s] = in ? P.r[i] : 0.;
      x[s] = in ? P.x[i] : 0.;
      sq[s] = in ? P.dsq[i] : 0.;
      if constexpr (KEEP)
#pragma unroll
        for (int u = 0; u < NU; ++u) {
          const bool on = in && u < ku && off[u] > 0;
          au[s][u] = (on && i + off[u] < hi) ? P.scaled[int64_t(u) * n + i] : 0.;
          al[s][u] = (on && i - off[u] >= lo) ? P.scaled[int64_t(u) * n + i - off[u]] : 0.;
        }
    }
    const double tol2 = P.S[K.inst].tol2;
    const int own_na = (rows + P.a_block - 1) / P.a_block;
    const int own_nv = (rows + (P.v_block << lg) - 1) / (P.v_block << lg);
    // own rows [0, pub_lo) and [pub_hi, rows) are read by other workgroups of the team
    const int pub_lo = K.rank > 0 ? reach : 0, pub_hi = K.rank + 1 < K.team ? rows - reach : rows;
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
      for (int k = 0; k < 2; ++k) {
        double s = 0.;
        for (int w = 0; w < vwaves; ++w)
          s += red2[k][w];
        rn[k] = s;
      }
    }
    int it = 0, begun = 0;
    int state = 0;
    double alpha = 0., pq = 0.;
    const int max_iter = int(min(P.max_iter, int64_t(0x7ffffff0)));
    for (;; ++it) {
      asm volatile("" : "+v"(tb));
      // direction update: stopping test, p = r + beta p on the own rows and on the halo
      state = (rn[1] <= tol2) ? 1 : (it >= max_iter) ? 2 : 0;
      begun = state ? it : it + 1;
      const double rho = rn[0];
      if (state)
        break;
      if (it > 0) {
        beta = rho / rho_prev;
        for (int e = t; e < below + above; e += RES_LANES) {
          const int o = e < below ? e - below : rows + e - below;
          pl[reach + o] = fma(beta, pl[reach + o], published(P.r_pub + K.row0 + o));
        }
#pragma unroll
        for (int s = 0; s < S; ++s) {
          const int o = row(s);
          if (o < rows)
            pl[reach + o] = fma(beta, pl[reach + o], r[s]);
        }
      }
      rho_prev = rho;
      __syncthreads();
      // q = Ah p, and p.q of every group of 64 rows
      double q[S];
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const int o = row(s);
        const bool in = o < rows;
        const int oc = min(o, rows - 1);
        const int c = reach + oc;
        double bl[NU], bu[NU];
        if constexpr (!KEEP) {
#pragma unroll
          for (int u = 0; u < NU; ++u) {
            // (rows whose partner lies below the instance read the first valid entry, times p = 0)
            const double* __restrict__ col = P.scaled + int64_t(u < ku ? u : 0) * n + K.row0;
            bl[u] = *at(col - min(off[u], below), unsigned(max(oc - max(off[u] - below, 0), 0)));
            bu[u] = *at(col, unsigned(oc));
          }
        }
        double a = 0.;
#pragma unroll
        for (int u = NU - 1; u >= 0; --u) {
          const double m = KEEP ? al[KEEP ? s : 0][u] : (off[u] > 0 ? bl[u] : 0.);
          a = fma(m, pl[c - off[u]], a);
        }
        const double pi = pl[c];
        a += pi;
#pragma unroll
        for (int u = 0; u < NU; ++u) {
          const double m = KEEP ? au[KEEP ? s : 0][u] : (off[u] > 0 ? bu[u] : 0.);
          a = fma(m, pl[c + off[u]], a);
        }
        q[s] = a;
        const double w = wave_sum(in ? pi * a : 0.);
        if ((t & 63) == 0)
          ga[o >> 6] = w;
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // the slots cleared by the last exchange are empty
      __syncthreads();
      double own1[1] = {0.};
      const int par = it & 1;
      if (t < own_na) {
        const int g = P.a_block >> 6;
        for (int w = 0; w < g; ++w)
          own1[0] += ga[t * g + w];
        if (!alone) {
          slot_clear(at(P.g1 + (par ^ 1) * P.n_a + K.own_a, unsigned(t)));
          slot_store(at(P.g1 + par * P.n_a + K.own_a, unsigned(t)), own1[0]);
        }
      }
      double tot1[1];
      if (!exchange_sum<1>(P.g1 + par * P.n_a + K.a0, own1, alone, K.na, P.v_block, red1, &failed, P.gave_up,
                           P.wait_ticks, tot1))
        return;
      pq = tot1[0];
      if (!(pq > 0.)) { // breakdown: the iterate holds every earlier step
        state = 3;
        break;
      }
      // update: x and r, the partials of the residual norms, the rows other workgroups read
      alpha = rho / pq;
      double v[2] = {0., 0.};
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const int o = row(s);
        if (o < rows) {
          x[s] = fma(alpha, pl[reach + o], x[s]);
          const double ri = fma(-alpha, q[s], r[s]);
          r[s] = ri;
          const double ru = sq[s] * ri;
          v[0] = fma(ri, ri, v[0]), v[1] = fma(ru, ru, v[1]);
          if (!alone && (o < pub_lo || o >= pub_hi))
            publish(at(P.r_pub + K.row0, unsigned(o)), ri);
        }
        if ((s & (items - 1)) == items - 1) {
          const double w0 = wave_sum(v[0]), w1 = wave_sum(v[1]);
          if ((t & 63) == 0)
            gv[0][(s >> lg) * RES_WAVES + wave] = w0, gv[1][(s >> lg) * RES_WAVES + wave] = w1;
          v[0] = v[1] = 0.;
        }
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // the published rows have arrived
      __syncthreads();
      double own2[2] = {0., 0.};
      if (t < own_nv) {
        for (int w = 0; w < vwaves; ++w)
          own2[0] += gv[0][t * vwaves + w], own2[1] += gv[1][t * vwaves + w];
        if (!alone) {
          double* mine = at(P.g2 + 2 * (par * P.n_v + K.own_v), 2u * unsigned(t));
          double* other = at(P.g2 + 2 * ((par ^ 1) * P.n_v + K.own_v), 2u * unsigned(t));
          slot_clear(other), slot_clear(other + 1);
          slot_store(mine, own2[0]), slot_store(mine + 1, own2[1]);
        }
      }
      if (!exchange_sum<2>(P.g2 + 2 * (par * P.n_v + K.v0), own2, alone, K.nv, P.v_block, red2, &failed, P.gave_up,
                           P.wait_ticks, rn))
        return;
    }
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int o = row(s);
      if (o < rows)
        P.x[K.row0 + o] = x[s];
    }
    if (K.rank == 0 && t == 0) {
      PcgScalars* R = P.S + K.inst;
      R->rz = rn[0], R->rr = rn[1], R->beta = beta, R->alpha = alpha, R->alpha_prev = alpha, R->pq = pq;
      R->iters = begun;
      R->done = state;
      R->brk = 0;
    }
  }
}

__global__ void k_resident_clear(int64_t n, double* __restrict__ slots, int* gave_up)
{
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n)
    slots[i] = __longlong_as_double((long long)RES_EMPTY);
  if (i == 0)
    *gave_up = 0;
}

using Kernel = void (*)(ResidentParams);

template <int NU>
Kernel kernel_for(int slots)
{
  switch (slots) {
    case 1:
      return k_pcg_resident<1, NU, true>;
    case 2:
      return k_pcg_resident<2, NU, true>;
    case 4:
      return k_pcg_resident<4, NU, true>;
    case 8:
      return k_pcg_resident<8, NU, true>;
    default:
      return k_pcg_resident<16, NU, false>;
  }
}

Kernel kernel_of(int slots, int nu)
{
  return nu <= 3 ? kernel_for<3>(slots) : kernel_for<4>(slots);
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

void resident_plan_dia(ResidentPlan& plan, const Operator& op, const std::vector<std::vector<int64_t>>& s_offs,
                       int s_nu)
{
  plan.usable = false;
  const SolverFormat& F = op.fmt;
  const int ba = F.A.block, bv = F.V.block, iv = F.V.items;
  if (s_nu < 0 || s_nu > 4 || F.A.items != 1 || ba > 1024 || (ba & (ba - 1)) != 0 || RES_LANES % bv != 0)
    return;
  const std::vector<int64_t>& row0 = op.space->inst_dof;
  const int ninst = int(row0.size()) - 1;
  const int cus = device_cus();
  int64_t largest = 0, reach = 0;
  std::vector<int64_t> reaches(ninst, 0);
  for (int in = 0; in < ninst; ++in) {
    const int64_t ni = row0[in + 1] - row0[in];
    if (ni == 0)
      return;
    largest = std::max(largest, ni);
    for (int64_t o : s_offs[in])
      if (o < ni)
        reaches[in] = std::max(reaches[in], o);
    reach = std::max(reach, reaches[in]);
  }
  // rows per lane: the fewest with which all instances fit on the chip together
  int slots = 0;
  int64_t total = 0, lds = 0;
  for (int s : {1, 2, 4, 8, 16}) {
    if (s % iv)
      continue;
    const int64_t R = int64_t(s) * RES_LANES;
    if (R % ba)
      continue;
    total = 0;
    for (int in = 0; in < ninst; ++in)
      total += (row0[in + 1] - row0[in] + R - 1) / R;
    lds = (std::min(R, largest) + 2 * reach) * int64_t(sizeof(double));
    if (total <= cus && lds <= RES_LDS) {
      slots = s;
      break;
    }
  }
  if (!slots || (s_nu == 0 && slots == RES_MAX_SLOTS)) // (a diagonal matrix holds no slot to stream)
    return;
  const int64_t R = int64_t(slots) * RES_LANES;
  std::vector<ResidentTask> tasks;
  std::vector<int32_t> start;
  for (int in = 0; in < ninst; ++in) {
    const int64_t ni = row0[in + 1] - row0[in];
    const int team = int((ni + R - 1) / R);
    for (int k = 0; k < team; ++k) {
      ResidentTask K{};
      K.row0 = row0[in] + k * R;
      K.rows = int32_t(std::min(R, ni - k * R));
      K.inst = in, K.team = team, K.rank = k;
      K.a0 = F.A.inst_block0[in], K.na = F.A.inst_block0[in + 1] - K.a0;
      K.v0 = F.V.inst_block0[in], K.nv = F.V.inst_block0[in + 1] - K.v0;
      K.own_a = K.a0 + int32_t(k * R / ba), K.own_v = K.v0 + int32_t(k * R / (int64_t(bv) * iv));
      if (team == 1 && (K.na > bv || K.nv > bv)) // the lanes that add the partials do not hold them
        return;
      start.push_back(int32_t(tasks.size()));
      tasks.push_back(K);
    }
  }
  start.push_back(int32_t(tasks.size()));
  plan.slots = slots, plan.nu = s_nu, plan.workgroups = int(start.size()) - 1, plan.lds = lds;
  plan.tasks.upload(tasks);
  plan.task_start.upload(start);
  plan.exchange.allocate(size_t(2 * F.A.nblocks + 4 * F.V.nblocks));
  plan.gave_up.allocate(1);
  if (!plan.host_gave_up)
    HGDT_HIP(hipHostMalloc((void**)&plan.host_gave_up, sizeof(int)));
  plan.usable = true;
}

bool resident_run(ResidentPlan& plan, ResidentParams P, hipStream_t stream, PcgScalars* host_records)
{
  P.g1 = plan.exchange.ptr;
  P.g2 = plan.exchange.ptr + 2 * P.n_a;
  P.tasks = plan.tasks.ptr, P.task_start = plan.task_start.ptr, P.gave_up = plan.gave_up.ptr;
  P.wait_ticks = int64_t(4) * 100000000; // 4 s
  const int64_t nx = int64_t(plan.exchange.count);
  hipLaunchKernelGGL(k_resident_clear, dim3(unsigned((nx + 255) / 256)), dim3(256), 0, stream, nx, plan.exchange.ptr,
                     plan.gave_up.ptr);
  const Kernel k = kernel_of(plan.slots, plan.nu);
  HGDT_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                               int(RES_LDS)));
  int dev = 0;
  HGDT_HIP(hipGetDevice(&dev));
  struct Hold {
    int dev, count;
    ~Hold()
    {
      CuBudget::get().give(dev, count);
    }
  };
  CuBudget::get().take(dev, plan.workgroups, device_cus());
  Hold hold{dev, plan.workgroups};
  hipLaunchKernelGGL(k, dim3(unsigned(plan.workgroups)), dim3(RES_LANES), size_t(plan.lds), stream, P);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess)
    e = hipMemcpyAsync(plan.host_gave_up, plan.gave_up.ptr, sizeof(int), hipMemcpyDeviceToHost, stream);
  if (e == hipSuccess)
    e = hipMemcpyAsync(host_records, P.S, sizeof(PcgScalars) * P.ninst, hipMemcpyDeviceToHost, stream);
  const hipError_t e2 = hipStreamSynchronize(stream); // also after an error: the CUs are given back with none running
  HGDT_HIP(e);
  HGDT_HIP(e2);
  return *plan.host_gave_up == 0;
}

} // namespace hgdt
