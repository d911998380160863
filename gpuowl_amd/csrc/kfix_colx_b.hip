// Column passes compiled per H (2048 <= H < 3072): k_colx<H, T, C0, C1, C2, SPLIT, NT, SQ> with the radices and threads of
// coltab.h. "colx<H>" runs every mode; the squaring alone: "colcp<H>" (complex exchanges, plain accesses),
// "colcn<H>" (complex, non-temporal), and from H = 2304 up "colx<H>m" (split exchanges, plain) and "colsn<H>" (split,
// non-temporal). Gpu::colPass chooses.
#include "kfixed.h"

#define PASS(NAME, H, SPLIT, NT, SQ) \
  {NAME, (const void*)&k_colx<H, colThreadsX(H), colRadices(H).c0, colRadices(H).c1, colRadices(H).c2, SPLIT, NT, SQ>, \
   colThreadsX(H)}
#define COMPLEX(H) \
  PASS("colx" #H, H, false, false, false), PASS("colcp" #H, H, false, false, true), PASS("colcn" #H, H, false, true, true)
#define SPLIT(H) PASS("colx" #H "m", H, true, false, true), PASS("colsn" #H, H, true, true, true)

extern "C" const OwlKernelEntry owl_kernel_table_colx_b[] = {
    COMPLEX(2048),
    COMPLEX(2304),
    SPLIT(2304),
    COMPLEX(2560),
    SPLIT(2560),
    COMPLEX(2816),
    SPLIT(2816),
    {nullptr, nullptr, 0},
};
