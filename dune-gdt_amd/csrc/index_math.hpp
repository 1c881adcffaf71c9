// index_math.hpp -- rules on sizes that decide how a launch addresses its rows; plain C++, checked on the CPU.
#pragma once

#include <cstdint>

namespace hgdt {

// Workgroups of an operator application over row blocks of block * items rows: `per` workgroups of `lanes` lanes for each
// block, and inv = 2^32 / per rounded up, with which a device divides a workgroup's number by per (0: per = 1).
struct ApplySplit {
  int lanes = 0;
  uint32_t per = 1, inv = 0;
};

// The division through inv is exact below 2^32 / per (per * inv exceeds 2^32 by less than per; per <= 64), and a grid has
// less than 2^32 lanes: beyond either (batches of very many, very small instances) one workgroup takes a whole block.
constexpr ApplySplit apply_split(int block, int items, int64_t nblocks)
{
  const int64_t rows = int64_t(block) * items;
  const int lanes = items > 1 && rows % 256 == 0 ? 256 : block;
  const int64_t per = rows / lanes;
  if (per == 1 || (nblocks + 8) * per > (int64_t(1) << 26) || (nblocks + 8) * rows >= (int64_t(1) << 31))
    return {block, 1, 0};
  return {lanes, uint32_t(per), uint32_t(((uint64_t(1) << 32) + uint64_t(per) - 1) / uint64_t(per))};
}

// One-launch solves of general storage and of discontinuous spaces address the values that workgroups exchange from the
// start of a vector of n doubles with 32-bit byte offsets, as one scalar base and an offset per lane.  Vectors beyond 4 GB
// (batches: no single instance on the chip is that large) take the kernels per iteration.
constexpr bool reached_by_32_bits(int64_t n)
{
  return n <= (int64_t(1) << 32) / int64_t(sizeof(double));
}

} // namespace hgdt
