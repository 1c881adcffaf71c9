// resident_device.hpp -- what the one-launch solvers share on the device (resident.hip, resident_dg.hip): the exchange of
// block partials through slots that hold a sentinel until they are stored.
#pragma once

#include "block_reduce.hpp"
#include "resident.hpp"

namespace hgdt {
namespace {

constexpr int RES_LANES = RES_BLOCK;  // lanes of a workgroup (FAR: RES_FAR_BLOCK)
constexpr int RES_MAX_SLOTS = 16;
constexpr int RES_HALO = 4; // halo rows a lane asks for while the residual norms are exchanged
constexpr int RES_WAVES = 12;              // of a workgroup, at most
constexpr int RES_GROUPS = 144;            // 64-row groups of a workgroup, at most
constexpr int RES_MAX_GROUPS = 1024;                  // workgroups of an instance, at most (flags)
constexpr int64_t RES_LDS = 150 * 1024;               // dynamic LDS of a workgroup, of 160 KB

// doubles from one workgroup block's slot to the next: packed slots share lines that all poll while they are written
constexpr int RES_PAD = 2;

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
// limit of a wait: over() after each failed look, true when the wait is to end (its limit is reached, or another
// workgroup gave up).  The first looks follow each other at once; later ones sleep and watch the clock.
struct Patience {
  int looks = 0;
  long long since = 0;
  __device__ __forceinline__ bool over(ResidentFlags gave_up, int64_t ticks)
  {
    if (++looks < 256)
      return false;
    __builtin_amdgcn_s_sleep(2);
    if (looks == 256)
      since = wall_clock64();
    if (looks & 255)
      return false;
    if (!__hip_atomic_load(gave_up.device, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) && wall_clock64() - since <= ticks)
      return false;
    __hip_atomic_store(gave_up.device, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(gave_up.host, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    return true;
  }
};

// a value that is the same in all lanes, as a scalar
__device__ __forceinline__ int uniform(int v)
{
  return __builtin_amdgcn_readfirstlane(v);
}

// element `i` of an array whose base is the same for the whole wave: a 32-bit byte offset per lane
template <class T>
__device__ __forceinline__ T* at(T* base, unsigned i)
{
  return reinterpret_cast<T*>(reinterpret_cast<char*>(const_cast<std::remove_const_t<T>*>(base)) + i * unsigned(sizeof(T)));
}

// sums of `count` partials of NV values as Partials::sum adds them (lane t of `block` lanes adds the partials t,
// t + block, ...; then the waves' butterflies; then the waves in order), in every lane.  Partials come from the
// exchange slots, or (one workgroup, at most `block` partials: own) from the lane that computed them.  false:
// gave up.  One barrier; red is not written again before a later barrier.
template <int NV, int NW>
__device__ __forceinline__ bool exchange_sum(const double* slots, const double (&own)[NV], bool alone, int count,
                                             int block, double (*red)[RES_WAVES], int* failed, ResidentFlags gave_up,
                                             int64_t ticks, double (&tot)[NV])
{
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
    for (int b = t; b < count; b += block) {
      unsigned long long u[NV];
      Patience wait;
      while (true) {
        bool empty = false;
#pragma unroll
        for (int k = 0; k < NV; ++k)
          u[k] = slot_load(at(slots, unsigned(b) * RES_PAD + k));
#pragma unroll
        for (int k = 0; k < NV; ++k)
          empty = empty || u[k] == RES_EMPTY;
        if (!empty)
          break;
        if (wait.over(gave_up, ticks)) {
          *failed = 1;
          break;
        }
      }
      if (*failed)
        break;
#pragma unroll
      for (int k = 0; k < NV; ++k)
        tot[k] += __longlong_as_double((long long)u[k]);
    }
  }
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const double w = wave_sum(tot[k]); // (0 in the waves past `block`: added below without a change)
    if ((t & 63) == 0)
      red[k][t >> 6] = w;
  }
  __syncthreads();
  if (uniform(*failed))
    return false;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    double s = 0.;
#pragma unroll
    for (int w = 0; w < NW; ++w)
      s += red[k][w];
    tot[k] = s;
  }
  return true;
}

// g consecutive LDS values added in order (g a power of two up to 16), four loads at a time
__device__ __forceinline__ double add_run(const double* v, int g)
{
  double s = 0.;
  if (g == 1)
    return s + v[0];
  if (g == 2)
    return s + v[0] + v[1];
  for (int w = 0; w < g; w += 4) {
    const double a = v[w], b = v[w + 1], c = v[w + 2], d = v[w + 3];
    s += a, s += b, s += c, s += d;
  }
  return s;
}

} // namespace
} // namespace hgdt
