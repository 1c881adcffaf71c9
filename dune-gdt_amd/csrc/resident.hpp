// resident.hpp -- PCG solves whose vectors stay on the chip (resident.hip; discontinuous spaces: resident_dg.hip).
#pragma once

#include <memory>

#include "hgdt_internal.hpp"
#include "mf_params.hpp"

namespace hgdt {

constexpr int RES_BLOCK = 512;     // lanes of a workgroup, and of the row blocks that suit it
constexpr int RES_FAR_BLOCK = 768; // the same for 3-d lattices whose planes do not fit in LDS (12 rows per lane and 3
                                   // waves per SIMD: 256 workgroups hold 2.36 million rows)
// row blocks for a solve in one launch (block 0: it does not fit on the chip)
struct ResidentShape {
  int block = 0, items = 0;
  bool operator!=(const ResidentShape& o) const
  {
    return block != o.block || items != o.items;
  }
};

// one instance's share of a workgroup: consecutive rows of the instance, handled by `rank` of its team
struct ResidentTask {
  int64_t row0;          // first own row
  int32_t rows;          // own rows (the last workgroup of a team may have fewer than the others)
  int32_t inst;
  int32_t team, rank;    // workgroups of the instance, and which of them this is
  int32_t a0, na;        // first block of the instance and their number, operator partition
  int32_t v0, nv;        // the same, vector partition
  int32_t own_a, own_v;  // first own block of either partition
  // SELL: first own slice, and the rows of other workgroups that the own rows meet (entries of halo_rows)
  int32_t slice0, halo0, nhalo;
  int32_t mask; // its block of `publish`
};

// set when a wait outlasts its limit, for the workgroups (every one then ends) and for the host (pinned memory)
struct ResidentFlags {
  int* device;
  int* host;
};

struct ResidentParams {
  int64_t n;
  int zero_place; // discontinuous spaces: place of the zeros in p
  const int64_t* inst_row0;
  // launch shapes whose block partials (and therefore bits) the solve reproduces: vector blocks of v_block lanes and
  // 1 << v_lg_items rows per lane, operator blocks the same or of a_rows lanes with one row each
  int a_rows, v_block;
  // scaled symmetric DIA: strict upper slots
  int s_nu;
  const int64_t* s_off;
  const double* scaled;
  // scaled SELL-64 values in `scaled`; per entry its position in the workgroup's p (own rows, then its halo)
  const int64_t* slice_ptr;
  const uint16_t* sell_local;
  const int32_t* halo_rows;
  const uint32_t* publish; // per workgroup and lane: the slots whose rows other workgroups read
  // discontinuous spaces: elements of a workgroup, in order (-1: none; bit 30: read by other workgroups); the scaled element
  // blocks as the storage has them; reference data of the matrix-free operator
  const int32_t* dg_elements;
  int blk_mn, blk_sym;
  int64_t blk_ne;
  const int32_t* blk_nb;
  const int32_t* blk_mir;
  const double* dg_ref;
  const double* dh;
  const double* dsq;
  const double* r;     // r of the initial residual (not written: a solve that gives up leaves it to the caller)
  const double* x;     // scaled iterate at the start
  double* x_out;       // and at the end (until then the iterate of workgroups that do not hold it in registers)
  double* r_pub[2];    // rows of r that other workgroups of the team read, by parity of the step
  const double* part2; // partials of the initial residual, 2 per vector block
  double* g1;          // 2 x (operator blocks), padded: partials of p.q, by parity of the step
  double* g2;          // behind it, 2 x (vector blocks), padded: partials of the two residual norms
  int64_t n_a, n_v;    // operator / vector blocks of all instances
  const PcgScalars* S; // records of the instances
  PcgScalars* result;  // and their results (pinned host memory)
  int64_t max_iter;
  const ResidentTask* tasks;
  const int32_t* task_start; // per workgroup
  int* flags;          // FAR: per workgroup, the step whose p it has published
  ResidentFlags gave_up;
  int64_t wait_ticks;  // limit of one wait, in ticks of the 100 MHz counter; 0: a launch that exchanges gives up
};

// launch plan of an operator: kept with its solver data, rebuilt when partitions or storage change
struct ResidentPlan {
  int64_t version = -1; // SolverCache::version the plan was made for
  bool usable = false;
  int slots = 0;        // rows per lane
  int lg_items = 0;     // log2 of the vector blocks' rows per lane
  bool same_blocks = false; // operator blocks = vector blocks
  int nu = 0;           // strict upper slots the kernel is compiled for
  int workgroups = 0;   // with rows; the grid is rounded up to the 8 XCDs
  int grid = 0;
  int64_t lds = 0;
  bool sell = false, far = false, dg = false, matrix_free = false; // (dg: slots are elements per lane)
  int lanes = RES_BLOCK;
  double step = 0.;         // estimate of one iteration of a workgroup
  int zero_place = 0;
  int64_t n_a = 0, n_v = 0; // partials of the two exchanges
  DeviceArray<int32_t> elements;
  DeviceArray<uint16_t> sell_local;
  DeviceArray<int32_t> halo_rows;
  DeviceArray<uint32_t> publish;
  DeviceArray<ResidentTask> tasks;
  DeviceArray<int32_t> task_start;
  // the same with no task for the first workgroup, which the others of its instance then wait for (waits of length 0)
  std::vector<int32_t> start_without;
  DeviceArray<int32_t> d_start_without;
  DeviceArray<double> exchange; // g1, g2
  DeviceArray<int> gave_up;    // and the flags of the workgroups behind it
  int* host_gave_up = nullptr;
  bool exchanges = false;      // some instance has more than one workgroup
  const void* kernel = nullptr;
  int cus = 0;
  int skip = 0; // solves that go without the launch after one that gave up
  ~ResidentPlan()
  {
    if (host_gave_up)
      (void)hipHostFree(host_gave_up);
  }
};

// symmetric DIA storage with these strict upper offsets
ResidentShape resident_shape_dia(const std::vector<int64_t>& inst_row0, const std::vector<std::vector<int64_t>>& s_offs,
                                 int s_nu);
// doubles that the solve reads ahead of and past the scaled matrix's diagonals (those ahead must be finite)
int64_t resident_padding(const std::vector<int64_t>& inst_row0, const std::vector<std::vector<int64_t>>& s_offs, int s_nu);
// s_offs: the strict upper offsets of every instance's scaled matrix
void resident_plan_dia(ResidentPlan& plan, const Operator& op, const std::vector<std::vector<int64_t>>& s_offs,
                       int s_nu);
// the same for SELL storage (general meshes): rows per lane, and the plan
int resident_items_sell(const Operator& op);
void resident_plan_sell(ResidentPlan& plan, const Operator& op);
// discontinuous spaces of 4 DoFs per element: element blocks, or matrix-free (whatever the launch shapes are)
void resident_plan_dg(ResidentPlan& plan, const Operator& op);
const void* resident_dg_kernel(const ResidentPlan& plan);
// Instances of a batch in the order of their size, each on the workgroups that are free first, `teams[i]` of them: the
// estimated time until the last one ends, and (order, groups) which instance is next and on which workgroups.  A workgroup
// takes its instances in this order, so the first unfinished one always has all of its workgroups.  step: us per iteration
// of one workgroup.  Negative: an instance does not fit.
double resident_schedule(const std::vector<int64_t>& row0, const std::vector<int>& teams, double step,
                         std::vector<int>* order, std::vector<std::vector<int>>* groups);
// the tasks (instance by instance) in the order in which the workgroups take them; buffers of the exchanges
void resident_finish(ResidentPlan& plan, const Operator& op, const std::vector<ResidentTask>& tasks, int64_t lds,
                     int64_t n_a, int64_t n_v);
// A launch of the solve.  Its CUs are the solve's until this object goes, which waits for the launch (and for what else the
// stream holds by then).
class ResidentLaunch {
  int device_, held_;
  hipStream_t stream_;

public:
  // results: pinned host memory.  What the launch writes besides these: r_pub, x_out and the exchange buffers; after
  // one that gave up the caller goes on with one launch per kernel.  M: the matrix-free operator.
  ResidentLaunch(ResidentPlan& plan, ResidentParams P, const MfParams& M, hipStream_t stream);
  ~ResidentLaunch();
  ResidentLaunch(const ResidentLaunch&) = delete;
  ResidentLaunch& operator=(const ResidentLaunch&) = delete;
};
// the solve of a finished launch gave up
bool resident_gave_up(ResidentPlan& plan);

} // namespace hgdt
