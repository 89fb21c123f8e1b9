// mk_map.h — integer maps from a launch's tile numbers to output tiles, for
// the kernels and for host-side checks (no HIP headers needed).
#pragma once

#ifdef __HIPCC__
#define MK_HD __host__ __device__ __forceinline__
#else
#define MK_HD inline
#endif

namespace mk {

// Run [r0, r1) of row tiles (bm rows each) whose first row lies in the padded
// row range [beg, end) of the expert that holds row tile rt's first row; the
// last expert's run also takes the row tiles past every range.  The counts may
// sum to more rows than the launch has: the run ends with its tiles_m row tiles.
MK_HD void expert_run(int rt, int beg, int end, bool last, int tiles_m, int bm, int& r0, int& r1) {
  const int first = (beg + bm - 1) / bm, past = (end + bm - 1) / bm;
  r0 = first < 0 ? 0 : first > rt ? rt : first;
  r1 = last || past > tiles_m ? tiles_m : past <= rt ? rt + 1 : past;
}

// Tile t of the run [r0, r1), whose tiles are numbered r0 * tiles_n ..
// r1 * tiles_n - 1: column-major.
MK_HD void expert_run_tile(int t, int r0, int r1, int tiles_n, int& tm, int& tn) {
  const int local = t - r0 * tiles_n, nr = r1 - r0;
  tn = local / nr;
  tm = r0 + local % nr;
}

}  // namespace mk
