// mk_map.h — integer maps from a launch's tile numbers to output tiles, for
// the kernels and for host-side checks (no HIP headers needed).
#pragma once

#ifdef __HIPCC__
#define MK_HD __host__ __device__ __forceinline__
#else
#define MK_HD inline
#endif

namespace mk {

// Expert GEMMs split a tail tile along K from this K on.  The parts' exchange
// takes 20 to 30 us: a third of a tile's time at K 7168 (6 experts of 4096
// columns, 48 tiles: 155 us whole, 92 split), more than it saves at 2048 (280
// tiles: 134 us with the 24 of the tail split, 114 on 144 workgroups; 84
// tiles: 40 whole, 51 split).
constexpr int kExpertSplitK = 4096;

// 128 x 512 tiles stream each expert's activation rows half as often per
// weight byte as 128 x 256 tiles, but a handful of row blocks with a long K
// makes too few of them to stream at the chip's rate: us at 512 / 256 columns,
// K 7168, 2 blocks 56 / 43, 6 90 / 75, 9 120 / 116, 13 143 / 148, 32 314 / 362,
// 64 622 / 729.
MK_HD bool few_row_blocks(long long blocks, long long K) { return K >= kExpertSplitK && blocks <= 10; }

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
