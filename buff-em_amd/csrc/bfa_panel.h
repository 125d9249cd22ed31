// bfa_panel.h -- register-resident LU panel (bfa_panel.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <cstddef>
#include <cstdint>

namespace bfa {
#define XP_MAXW 256      // widest panel
#define XP_MAXWG 128     // workgroups of one panel (a lane of a wave reads one or two words)
#define XP_PLANE XP_MAXW
#define XP_NBUF 4        // exchange buffers, by column
#define XP_FSTRIDE 16    // words between two workgroups' flags (a cache line each)

struct XPanel {
  void *A;               // m x w panel, column-major
  int *ipiv;             // w pivots, absolute (local row + piv_off)
  void *data;            // [XP_NBUF][XP_MAXWG candidate rows, row j][4 words][XP_PLANE]
  unsigned long long *flags;   // [XP_NBUF][XP_MAXWG][XP_FSTRIDE]
  int *err;              // [0] a wait gave up, [1] first zero pivot (1-based)
  int64_t lda;
  unsigned seq0;         // this launch's first sequence number (24 bits, w of them used)
  int m, w, piv_off, nwg;
};
size_t xpanel_bytes();
void xpanel_carve(char *mem, XPanel *p);
int xpanel_max_rows(bool f64);
int launch_xpanel(bool f64, XPanel p, hipStream_t st);
}  // namespace bfa
