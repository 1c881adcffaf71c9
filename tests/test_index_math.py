"""Rules on sizes of csrc/index_math.hpp, compiled for the CPU and compared with plain 64-bit arithmetic."""
import os
import subprocess

from conftest import ROOT


def _run(tmp_path, body):
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text('#include "index_math.hpp"\n#include <cstdio>\n#include <initializer_list>\nusing namespace hgdt;\n'
                   "int main() {\n" + body + "\n  return 0;\n}\n")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "dune-gdt_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def test_workgroups_of_an_application(tmp_path):
    """every launch shape: the workgroups of a block cover its rows once, the device's division is exact for every
    workgroup of the largest grid that uses it, and the grid stays below 2^32 lanes"""
    _run(tmp_path, r"""
  for (int block = 64; block <= 1024; block += 64)
    for (int items = 1; items <= 16; items *= 2)
      for (int64_t nb : {int64_t(1), int64_t(7), int64_t(4096), int64_t(1) << 20, (int64_t(1) << 22) - 8,
                         (int64_t(1) << 26) - 8, (int64_t(1) << 28) - 1}) {
        const ApplySplit s = apply_split(block, items, nb);
        bool ok = s.lanes % 64 == 0 && s.lanes <= block * items && s.lanes <= 1024 && s.per >= 1;
        ok = ok && (items > 1 || (s.lanes == block && s.per == 1));
        ok = ok && (s.per == 1 ? s.lanes == block && s.inv == 0 : int64_t(s.lanes) * s.per == int64_t(block) * items);
        ok = ok && (nb + 8) * s.per < (int64_t(1) << 31) && (s.per == 1 || (nb + 8) * s.per * s.lanes < (int64_t(1) << 32));
        if (s.per > 1) {
          const int64_t n = nb * s.per;
          for (int64_t w = 0; w < n; w += (w < 100000 || w > n - 100000 || n < 1000000) ? 1 : 997)
            ok = ok && int64_t((uint64_t(uint32_t(w)) * s.inv) >> 32) == w / s.per;
        }
        if (!ok) {
          std::printf("block %d items %d blocks %lld\n", block, items, (long long)nb);
          return 1;
        }
      }""")


def test_rows_reached_by_32_bit_offsets(tmp_path):
    """the byte offset of a lane's value, computed in 32 bits, is the one in 64 bits for every row of every vector that is
    admitted: 4 n DoFs by element too, up to the last (2^29 rows: 4 GB)"""
    _run(tmp_path, r"""
  int64_t largest = 0;
  for (int64_t n = 4; n <= (int64_t(1) << 32); n += n < 1024 ? 4 : n / 64) {
    for (int64_t m = n - 1; m <= n + 1; ++m)
      if (reached_by_32_bits(m)) {
        largest = m > largest ? m : largest;
        if (int64_t(uint32_t(m - 1) * uint32_t(sizeof(double))) != (m - 1) * int64_t(sizeof(double)))
          return 1;
      }
  }
  const int64_t limit = int64_t(1) << 29;
  if (!reached_by_32_bits(limit) || reached_by_32_bits(limit + 1) || reached_by_32_bits(2 * limit) || largest > limit)
    return 1;
  if (int64_t(uint32_t(limit - 1) * 8u) != (limit - 1) * 8 || int64_t(uint32_t(limit) * 8u) == limit * 8)
    return 1;""")
