"""The rows that a persistent kernel copies in a plan by lines (persist_columns in
clsparse_amd/csrc/persist_plan.hpp, as fill_tile walks them), on the CPU: both
sides at once as CG and BiCGStab copy them, and one side as the two products of the
learned factor do. Every operand of the side's diagonals is then in the tile and
holds the right row, with nothing else written outside the workgroup's own rows; line
ends with fewer columns than the widest offset, with as many, and more columns to copy
than threads."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r'''
#include <cstdio>
#include <vector>
#include "persist_plan.hpp"
static int check(size_t n, int nd, const int32_t* off, size_t vs) {
  const PersistPlan p = persist_plan(n, nd, off, vs, 256);
  if (p.rows == 0 || p.line == 0) { printf("n %zu: no plan by lines\n", n); return 1; }
  const uint32_t T = kPersistThreads, R = p.rows;
  std::vector<int64_t> tile(p.tile_size);
  uint32_t most = 0, least = T;
  for (Side side : {kBoth, kLower, kUpper})
    for (uint32_t w = 0; w < p.wgs; ++w) {
      const uint32_t first = persist_first_row(p, w), live = persist_live_threads(p, w);
      for (auto& t : tile) t = INT64_MIN;
      int bad = 0;
      auto put = [&](uint32_t at, int64_t row) {
        if (at >= p.tile_size) { bad = 1; return; }
        tile[at] = row;
      };
      const PersistColumns column = persist_columns(p, side, live);
      const uint32_t columns = column.count();
      if (columns > most) most = columns;
      if (live < least) least = live;
      for (uint32_t t = 0; t < T; ++t) {
        if (side != kUpper) put(p.own - p.tile_step + t, int64_t(first) - p.line + t);
        if (side != kLower) put(p.own + R * p.tile_step + t, int64_t(first) + int64_t(R) * p.line + t);
        for (uint32_t e = t; e < columns; e += T) {
          const int32_t c = int32_t(column(e));
          if (c >= 0 && uint32_t(c) < live) { printf("copies an own column\n"); return 1; }
          for (uint32_t k = 0; k < R; ++k)
            put(p.own + k * p.tile_step + c, int64_t(first) + int64_t(k) * p.line + c);
        }
      }
      for (uint32_t t = 0; t < live; ++t)
        for (uint32_t k = 0; k < R; ++k) put(p.own + k * p.tile_step + t, int64_t(first) + t + int64_t(k) * p.line);
      if (bad) { printf("copy outside the tile\n"); return 1; }
      for (uint32_t t = 0; t < live; ++t)
        for (uint32_t k = 0; k < R; ++k) {
          const int64_t i = int64_t(first) + t + int64_t(k) * p.line;
          if (i >= int64_t(n)) continue;
          for (int d = 0; d < nd; ++d) {
            if ((side == kLower && off[d] > 0) || (side == kUpper && off[d] < 0)) continue;
            const int64_t j = i + off[d], at = int64_t(p.own) + int64_t(k) * p.tile_step + t + p.delta[d];
            if (at < 0 || at >= int64_t(p.tile_size)) { printf("tile index\n"); return 1; }
            if (j >= 0 && j < int64_t(n) && tile[at] != j) {
              printf("n %zu side %d wg %u row %lld off %d: %lld\n", n, side, w, (long long)i, off[d], (long long)tile[at]);
              return 1;
            }
          }
        }
    }
  printf("n %zu rows %u side %u most columns %u least live %u\n", n, R, p.side, most, least);
  return 0;
}
int main() {
  int bad = 0;
  const int32_t a[] = {-1124, -256, 0, 256, 1124};            // 100 live columns, 256 to copy past them
  const int32_t b[] = {-1280, -256, -3, 0, 3, 256, 1280};     // 256 of each, 768 to copy
  const int32_t c[] = {-1536, -7, 0, 5, 1536};                // whole column tiles
  const int32_t d[] = {-1535, -1, 0, 1, 1535};                // one idle column
  const int32_t e[] = {-16384, -128, -1, 0, 1, 128, 16384};
  const int32_t f[] = {-12345, -110, -1, 0, 1, 110, 12345};
  const int32_t g[] = {-1025, 0, 1025};                       // one live column, nothing beside it
  for (size_t vs : {4, 8}) {
    bad |= check(200003, 5, a, vs);
    bad |= check(200003, 7, b, vs);
    bad |= check(300000, 5, c, vs);
    bad |= check(300001, 5, d, vs);
    bad |= check(size_t(128) * 128 * 128, 7, e, vs);
    bad |= check(1500000, 7, f, vs);
    bad |= check(150000, 3, g, vs);
  }
  printf(bad ? "FAIL\n" : "OK\n");
  return bad;
}
'''


def test_columns_of_a_plan_by_lines(tmp_path):
    src = tmp_path / "columns.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "columns"
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", os.path.join(ROOT, "clsparse_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.strip().endswith("OK"), out.stdout
    assert "most columns 768" in out.stdout and "least live 100" in out.stdout and "least live 1\n" in out.stdout
