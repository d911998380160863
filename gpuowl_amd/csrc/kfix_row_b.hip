// Row passes with 16 elements per thread compiled per (W, R): k_rowm<W, R, F0, F1, SPLIT, NT, FUSED>, T = W/F0 threads.
// "rowx<W>r<R>" runs every mode; the fused launches: "rowcp", "rowcn" (complex exchanges, plain or non-temporal
// accesses) and "rowsp", "rowsn" (split exchanges). Gpu::rowFused chooses.
#include "kfixed.h"

#define PASS(NAME, W, R, F0, F1, SPLIT, NT, FUSED) \
  {NAME #W "r" #R, (const void*)&k_rowm<W, R, F0, F1, SPLIT, NT, FUSED>, W / F0}
#define ROW(W, R, F0, F1) \
  PASS("rowx", W, R, F0, F1, false, false, false), PASS("rowcp", W, R, F0, F1, false, false, true), \
  PASS("rowcn", W, R, F0, F1, false, true, true), PASS("rowsp", W, R, F0, F1, true, false, true), \
  PASS("rowsn", W, R, F0, F1, true, true, true)

extern "C" const OwlKernelEntry owl_kernel_table_row_b[] = {
    ROW(256, 8, 2, 8),
    ROW(512, 4, 4, 8),
    ROW(1024, 4, 4, 16),
    {nullptr, nullptr, 0},
};
