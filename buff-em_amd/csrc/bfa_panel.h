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
// exchange memory of one panel at a time: bytes, and its division
size_t xpanel_bytes(bool f64);
void xpanel_carve(bool f64, char *mem, XPanel *p);
// tallest panel whose workgroups run at once on the current device (0: none)
int xpanel_max_rows(bool f64);
int launch_xpanel(bool f64, XPanel p, hipStream_t st);

// several complex64 panels in one launch, XPanelProb::p.nwg workgroups each
// from blk0; rows: rows a workgroup, one of xpanel_group_rows' values
struct XPanelProb {
  XPanel p;
  int blk0, pad;
};
// rows a workgroup for panels of at most m rows that fill `total` rows in all,
// and the workgroups that may run at once with it (0: none)
int xpanel_group_rows(int m, int64_t total, int *resident);
// tallest panel of a grouped launch (0: none)
int xpanel_group_max_rows();
void launch_xpanel_g(const XPanelProb *d, int np, int nblk, int rows, hipStream_t st);
}  // namespace bfa

// moves the device's panel sequence numbers forward (tests of their restart);
// returns the next one to be used
extern "C" unsigned bfa_xpanel_seq(unsigned seq);
// rows a workgroup for a panel of m rows where per_cu[v] workgroups of variant v
// (fewest rows first, four of them) run on each of `cus` CUs; 0: none fits
extern "C" int bfa_xpanel_rows(int f64, int m, int cus, const int *per_cu);
