// resident.hpp -- PCG solves whose vectors stay on the chip (resident.hip).
#pragma once

#include <memory>

#include "hgdt_internal.hpp"

namespace hgdt {

// one instance's share of a workgroup: consecutive rows of the instance, handled by `rank` of its team
struct ResidentTask {
  int64_t row0;          // first own row
  int32_t rows;          // own rows (the last workgroup of a team may have fewer than the others)
  int32_t inst;
  int32_t team, rank;    // workgroups of the instance, and which of them this is
  int32_t a0, na;        // first block of the instance and their number, operator partition
  int32_t v0, nv;        // the same, vector partition
  int32_t own_a, own_v;  // first own block of either partition
};

struct ResidentParams {
  int64_t n;
  int ninst;
  const int64_t* inst_row0;
  // launch shapes whose block partials (and therefore bits) the solve reproduces: operator blocks of a_block
  // rows, vector blocks of v_block lanes and 1 << v_lg_items rows per lane
  int a_block, v_block, v_lg_items;
  // scaled symmetric DIA: strict upper slots
  int s_nu;
  const int64_t* s_off;
  const double* scaled;
  const double* dsq;
  const double* r;     // r of the initial residual (not written: a solve that gives up leaves it to the caller)
  double* x;           // scaled iterate: read at the start, written by the instances that end
  double* r_pub;       // rows of r that other workgroups of the team read
  const double* part2; // partials of the initial residual, 2 per vector block
  double* g1;          // 2 x (operator blocks): partials of p.q, by parity of the step
  double* g2;          // 2 x 2 x (vector blocks): partials of the two residual norms
  int64_t n_a, n_v;    // operator / vector blocks of all instances
  PcgScalars* S;       // record of every instance: tolerance read, result written
  int64_t max_iter;
  const ResidentTask* tasks;
  const int32_t* task_start; // per workgroup
  int* gave_up;        // set when a wait outlasts its limit: every workgroup then ends
  int64_t wait_ticks;  // limit of one wait, in ticks of the 100 MHz counter
};

// launch plan of an operator: kept with its solver data, rebuilt when partitions or storage change
struct ResidentPlan {
  int64_t version = -1; // SolverCache::version the plan was made for
  bool usable = false;
  int slots = 0;        // rows per lane
  int nu = 0;           // strict upper slots the kernel is compiled for
  int workgroups = 0;
  int64_t lds = 0;
  DeviceArray<ResidentTask> tasks;
  DeviceArray<int32_t> task_start;
  DeviceArray<double> exchange; // g1, g2
  DeviceArray<int> gave_up;
  int* host_gave_up = nullptr;
  ~ResidentPlan()
  {
    if (host_gave_up)
      (void)hipHostFree(host_gave_up);
  }
};

// s_offs: the strict upper offsets of every instance's scaled matrix
void resident_plan_dia(ResidentPlan& plan, const Operator& op, const std::vector<std::vector<int64_t>>& s_offs,
                       int s_nu);
// runs the solve; false when it gave up (then nothing but r_pub and the exchange buffers was written for the
// instances without a result: the caller goes on with one launch per kernel).  Waits for the kernel.
bool resident_run(ResidentPlan& plan, ResidentParams P, hipStream_t stream, PcgScalars* host_records);

} // namespace hgdt
