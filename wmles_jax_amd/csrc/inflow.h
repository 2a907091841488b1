// Form of the synthetic inflow launch (k_inflow) for a row of N2 cells, n_modes Fourier modes and a
// profile table of n_tab rows: host arithmetic only.
#pragma once
#include <stddef.h>

namespace wmx {

struct InflowForm {
  int coop;       // 1: phases evaluated cooperatively in LDS, 2: with the table's y column there too
  int rows;       // row buffers of the means: two in turn (one barrier a mean), or one
  int threads;
  size_t lds;     // bytes
};

// Cooperative where the (cell, mode) table takes at most 56 KB.  64 KB hold, as far as they go and in
// this order, the second row buffer, 512 threads (two cosine chains a SIMD) and the y column; rows
// of 513 cells and more (up to 1024) with a table near the limit keep one buffer.
inline InflowForm inflow_form(int N2, int n_modes, int n_tab) {
  const size_t word = sizeof(double), lds = 64 * 1024;
  const size_t coop = word * ((size_t)(N2 | 1) * n_modes + 2 * (size_t)N2), tab = word * (size_t)n_tab;
  InflowForm f;
  f.coop = coop <= 56 * 1024 ? 1 : 0;
  f.threads = ((N2 + 63) / 64) * 64;
  if (f.coop && f.threads < 256) f.threads = 256;
  auto bytes = [&](int th, int rows) { return word * ((size_t)rows * th + 1) + (f.coop ? coop : 0); };
  f.rows = bytes(f.threads, 2) <= lds ? 2 : 1;
  if (f.coop && f.threads < 512 && bytes(512, 2) <= lds) f.threads = 512;
  if (f.coop && bytes(f.threads, f.rows) + tab <= lds) f.coop = 2;
  f.lds = bytes(f.threads, f.rows) + (f.coop == 2 ? tab : 0);
  return f;
}

}  // namespace wmx
