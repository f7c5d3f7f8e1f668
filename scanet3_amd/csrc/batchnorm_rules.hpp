// How the per-channel reductions of a batch normalisation are cut into slices, and the workspace that their partial sums take
// (host only).  A workspace is sized once, for the model's batch; a pass may bring fewer rows and must find room in it.
#pragma once
#include "common.hpp"

#include <algorithm>

namespace sn {

// row-walking form: slices of the rows for every 64 columns
inline int bn_row_slices(int compute_units, int64_t rows, int cols) {
  const int64_t col_blocks = ceil_div((int64_t)cols, (int64_t)64);
  int64_t s = ceil_div((int64_t)compute_units * 4, col_blocks);
  const int64_t by_rows = ceil_div(rows, (int64_t)64);  // at least 64 rows (16 per wave) in a slice
  if (s > by_rows) s = by_rows;
  if (s > 1024) s = 1024;
  return s < 1 ? 1 : (int)s;
}

// the float4-stream reductions: whole vectors of channels, at any number of rows (all of a layer's launches, 60 channels and 64 rows: 31.9 us,
// by rows and with two reads 39.6)
inline bool bn_stream_form(int cols) { return cols % 4 == 0 && cols <= 1024; }
// At least one full trip of 8 loads a thread, 16 rows (a slice leaves one row of partial sums, which the finishing kernels read: with 8 rows
// a slice they cost what the reduction saves) and two workgroups a CU.  All of a layer's reductions, 1000 channels: 4096 rows 51.5 us with
// slices of 8 rows and 46.1 so, 40000 rows 186 with four workgroups a CU and 178 so; 600 channels, 40000 rows, as many slices as the row-walking form has
// (64): 174, now 111.
inline int64_t bn_most_stream_slices(int compute_units, int64_t rows, int cols) {
  const int64_t s = std::min<int64_t>(ceil_div(rows * cols / 4, (int64_t)8 * 256), ceil_div(rows, (int64_t)16));
  return std::max<int64_t>(std::min<int64_t>(s, (int64_t)compute_units * 2), 1);
}
struct BnStream {
  int active, slices;  // slices: at most bn_most_stream_slices, every one with rows
  int64_t n4, per4;
};
inline BnStream bn_stream_of(int compute_units, int64_t rows, int cols) {
  BnStream st;
  const int cg = cols / 4;
  st.active = 256 / cg * cg;
  st.n4 = rows * cols / 4;
  st.per4 = ceil_div(ceil_div(st.n4, bn_most_stream_slices(compute_units, rows, cols)), (int64_t)st.active) * st.active;
  st.slices = (int)ceil_div(st.n4, st.per4);
  return st;
}

// The slices that a pass over `rows` rows may leave in the workspace, per channel and sum.  It never falls as the rows
// grow (the number that is left after rounding to whole trips does), so a workspace for the model's batch
// takes every pass.
inline int bn_max_slices(int compute_units, int64_t rows, int cols) {
  int64_t s = bn_row_slices(compute_units, rows, cols);
  if (bn_stream_form(cols)) s = std::max(s, bn_most_stream_slices(compute_units, rows, cols));
  return (int)s;
}

}  // namespace sn
