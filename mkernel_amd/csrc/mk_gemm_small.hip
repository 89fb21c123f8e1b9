// mk_gemm_small.hip — bf16 GEMM on tiles of 64 x 64 to 128 x 256 (gfx950): for
// problems that leave the chip idle at the persistent kernel's tiles, and for
// those of any size that cost less in rounds of these (mk_plan.h).
//
// The persistent kernel runs 128 x 256 or 256 x 256 tiles, one workgroup per
// CU; a 128 x 2048 x 2048 product is eight such tiles, so eight of 256 CUs
// work and each streams a whole K panel alone.  Here the tile is chosen to
// fill the chip and, where even that leaves CUs idle, each tile's K is cut
// into two to four parts, a workgroup each.
//
// Parts of one tile meet in the workspace.  Every part takes a ticket when
// its sum is done; all but the last write their fp32 sums there and publish a
// header word, the last keeps its own in registers, waits for the headers of
// the parts that came before it and adds all parts in K order, so the result
// does not depend on which came last.  Only workgroups that already run are
// waited for, so any number of workgroups may be queued, on any stream, and
// none needs another to become resident.
//
// Pipeline: both operands go HBM -> LDS by DMA through an S-deep ring of
// 64-deep K stages, one barrier per stage.  A rows are 128 bytes, 16-byte
// unit c of row r at c ^ ((r >> 1) & 7); B rows are N-contiguous and read
// with the transposing LDS read, units swizzled so that the four k-rows of a
// read fall into different banks.
//
// Bound by latency below ~1 GFLOP and by the operand stream through L2 / LDS
// above (a 128 x 128 tile moves 64 bytes per MFMA cycle).  Measured against
// the persistent kernel's 128 x 256 tiles on one MI355X (us): 128x2048x2048
// 31.9 -> 10.0, 1024^3 18.7 -> 6.8, 512x2048x8192 112 -> 31, 2048^3 33 -> 22,
// 2048x2048x8192 115 -> 76, 1920x2816x5600 79.5 -> 69.
#include "mk_device.h"
#include "mk_internal.h"
#include "mk_once.h"
#include "mk_tile.h"

namespace mk {
namespace {

template <int BM_, int BN_, int WM_, int WN_, int S_>
struct SCfg {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, S = S_;
  static constexpr int WAVES = WM * WN, NT = 64 * WAVES;
  static constexpr int WTM = BM / WM, WTN = BN / WN;
  static constexpr int FM = WTM / 32, FN = WTN / 32;
  static constexpr int BK = 64;
  static constexpr uint32_t A_BYTES = BM * BK * 2;
  static constexpr uint32_t BROW = BN * 2;
  static constexpr int B_UPR = BN / 8;  // 16-byte units per B k-row
  static constexpr uint32_t STAGE = A_BYTES + BK * BROW;
  static constexpr uint32_t LDS_BYTES = S * STAGE;
  // what the ring lets run: the compiler, which cannot know a launch's LDS,
  // else saves registers for more waves and serialises the LDS reads of a stage
  // (128x2048x2048 11.0 us so, 10.0 with the limit)
  static constexpr int WAVES_PER_SIMD = 160 * 1024 / LDS_BYTES * WAVES / 4;
  static constexpr int A_INST = A_BYTES / 1024 / WAVES;
  static constexpr int B_INST = BK * BROW / 1024 / WAVES;
  static constexpr int LOADS = A_INST + B_INST;
  static constexpr int UNITS = FM * FN * 4;  // 16-byte accumulator units per thread
  static_assert(WTN % 32 == 0 && WTM % 32 == 0 && FM >= 1 && FN >= 1 && A_INST >= 1 && B_INST >= 1, "tile too small for the wave grid");
  static_assert(LDS_BYTES <= 160 * 1024, "LDS");
};

template <int N, int L>
__device__ __forceinline__ void wait_pending(int pending) {
  if constexpr (N == 0) {
    wait_vm<0>();
  } else {
    if (pending >= N) wait_vm<N * L>();
    else wait_pending<N - 1, L>(pending);
  }
}

// Swizzle of the 16-byte units of B k-row k (see lds_tr4's users): the four
// k-rows one transposing read touches start 64 bytes apart in the banks.
template <int BN>
__device__ __forceinline__ int b_swizzle(int k) {
  return BN == 64 ? 4 * ((k >> 1) & 1) : 4 * (k & 3);
}

template <class C>
__device__ __forceinline__ void part_out(float* dst, f32x16 (&acc)[C::FM][C::FN], int tid) {
  const __amdgpu_buffer_rsrc_t r = make_rsrc(dst, (uint32_t)(C::BM * C::BN * 4));
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        f32x4 v;
#pragma unroll
        for (int b = 0; b < 4; ++b) v[b] = acc[i][j][4 * a + b];
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), r, tid * 16,
                                               ((i * C::FN + j) * 4 + a) * C::NT * 16, 0x10 /* SC1 */);
      }
}

// acc = sum over parts 0 .. n-1 in order; part `own` is acc as it stands, the
// part at order position q sits in slot slot0 + where[q].
template <class C>
__device__ __forceinline__ void parts_in(const float* slot0, const int* where, int n, int own,
                                         f32x16 (&acc)[C::FM][C::FN], int tid) {
  f32x4 s[C::UNITS];
  for (int q = 0; q < n; ++q) {
    if (q == own) {
#pragma unroll
      for (int u = 0; u < C::UNITS; ++u)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const float x = acc[u / (C::FN * 4)][(u / 4) % C::FN][4 * (u % 4) + b];
          s[u][b] = q == 0 ? x : s[u][b] + x;
        }
    } else {
      const int w = __builtin_amdgcn_readfirstlane(where[q]);
      const __amdgpu_buffer_rsrc_t r = make_rsrc(slot0 + (int64_t)w * (C::BM * C::BN), (uint32_t)(C::BM * C::BN * 4));
      f32x4 v[C::UNITS];
#pragma unroll
      for (int u = 0; u < C::UNITS; ++u)
        v[u] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, tid * 16, u * C::NT * 16, 0));
#pragma unroll
      for (int u = 0; u < C::UNITS; ++u)
#pragma unroll
        for (int b = 0; b < 4; ++b) s[u][b] = q == 0 ? v[u][b] : s[u][b] + v[u][b];
    }
  }
#pragma unroll
  for (int u = 0; u < C::UNITS; ++u)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[u / (C::FN * 4)][(u / 4) % C::FN][4 * (u % 4) + b] = s[u][b];
}

// One tile of a 256 x 256 tile's folded rows is stored (write-through): whoever
// stores the last of them publishes its flag.  Relaxed atomics, as in copy_wt's
// protocol: a release per tile (an L2 write-back) made 4096x4096x256 of world 8
// 61 us, 50 without flags.
template <class C>
__device__ __forceinline__ void part_done(const GemmSmallParams& p, int row, int col, int tid) {
  constexpr uint32_t kParts = (256 / C::BM) * (256 / C::BN);
  wait_vmem_all();
  __syncthreads();
  if (tid != 0) return;
  const int f = row / 256 * p.done_cols + col / 256;
  if (__hip_atomic_fetch_add(p.words + f, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != kParts - 1) return;
  __hip_atomic_store(p.words + f, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const uint32_t epoch =
      p.epoch_ptr ? __hip_atomic_load(p.epoch_ptr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : p.epoch;
  __hip_atomic_store(p.done + f, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <class C, bool REDUCE>
__global__ __launch_bounds__(C::NT) __attribute__((amdgpu_waves_per_eu(1, C::WAVES_PER_SIMD)))
void gemm_small_kernel(GemmSmallParams p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / C::WN, wn = wave % C::WN;
  const uint32_t wave_u = __builtin_amdgcn_readfirstlane(wave);
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  // workgroups are dealt round-robin to the 8 XCDs: give each XCD a
  // contiguous run of ids, hence neighbouring tiles, for its L2 (any G: XCD x
  // has one id more than G / 8 while x < G % 8)
  const uint32_t G = gridDim.x, xcd = blockIdx.x & 7;
  const uint32_t id = xcd * (G >> 3) + min(xcd, G & 7) + (blockIdx.x >> 3);
  const uint32_t t = REDUCE ? id : id / p.split, part = REDUCE ? 0 : id - t * p.split;  // a fold's tiles are whole

  const int ml = lane & 31, g = lane >> 5;
  uint32_t a_rd[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
    const int row = wm * C::WTM + ml;
    a_rd[kk] = row * 128 + (((2 * kk + g) ^ ((row >> 1) & 7)) << 4);
  }
  const int grp = lane >> 4, jr = (lane >> 2) & 3, q4 = lane & 3;
  uint32_t b_rd[C::FN];
#pragma unroll
  for (int j = 0; j < C::FN; ++j) {
    const int krow = 8 * (grp >> 1) + jr;
    const int c = 4 * (wn * C::FN + j) + 2 * (grp & 1) + (q4 >> 1);
    b_rd[j] = krow * C::BROW + ((c ^ b_swizzle<C::BN>(krow)) << 4) + (q4 & 1) * 8;
  }
  // LDS unit -> source chunk of this lane's DMA lanes
  int a_row[C::A_INST], a_chk[C::A_INST], b_row[C::B_INST], b_chk[C::B_INST];
#pragma unroll
  for (int i = 0; i < C::A_INST; ++i) {
    a_row[i] = (wave * C::A_INST + i) * 8 + (lane >> 3);
    a_chk[i] = (lane & 7) ^ ((a_row[i] >> 1) & 7);
  }
#pragma unroll
  for (int i = 0; i < C::B_INST; ++i) {
    const int n = (wave * C::B_INST + i) * 64 + lane;
    b_row[i] = n / C::B_UPR;
    b_chk[i] = (n % C::B_UPR) ^ b_swizzle<C::BN>(b_row[i]);
  }

  const uint32_t k0 = REDUCE ? 0 : part * p.nk / p.split;
  const int n = (REDUCE ? p.nk : (int)((part + 1) * p.nk / p.split)) - (int)k0;
  int tm, tn;
  decode_grouped((int)t, p.tiles_m, p.tiles_n, p.group_m, tm, tn);
  // The rows to fold cost more than the others and are neighbours: each
  // eighth of the columns starts its walk over the rows another eighth
  // further on, so that the fold falls on every XCD.
  if (REDUCE) tm = (tm + tn * 8 / p.tiles_n * ((p.tiles_m + 7) / 8)) % p.tiles_m;
  const int m0 = __builtin_amdgcn_readfirstlane(tm * C::BM), n0 = __builtin_amdgcn_readfirstlane(tn * C::BN);
  const u32x4_t rA = make_rsrc_v(p.A + (int64_t)m0 * p.lda, (uint32_t)(C::BM * p.lda * 2));
  const u32x4_t rB = make_rsrc_v(p.B, (uint32_t)(p.K * p.ldb * 2));
  uint32_t a_src[C::A_INST], b_src[C::B_INST];
#pragma unroll
  for (int i = 0; i < C::A_INST; ++i) a_src[i] = (uint32_t)(a_row[i] * p.lda * 2 + a_chk[i] * 16);
#pragma unroll
  for (int i = 0; i < C::B_INST; ++i) b_src[i] = (uint32_t)(b_row[i] * p.ldb * 2 + (n0 + b_chk[i] * 8) * 2);
  // ring slots as byte offsets, stepped (a modulo of the stage number costs
  // more than a DMA's issue when S is not a power of two)
  auto next_slot = [](uint32_t o) { return o + C::STAGE == C::LDS_BYTES ? 0u : o + C::STAGE; };
  uint32_t wr = 0, rd = 0;
  uint32_t ka = k0 * (C::BK * 2), kb = k0 * (uint32_t)(C::BK * p.ldb * 2);
  // a tile whose K holds an odd number of 32-deep steps ends in a half stage
  int half = (p.K & 32) ? p.nk - 1 - (int)k0 : -1;
  auto issue = [&] {
    const uint32_t slot = lds_base + wr;
    if (half == 0) {
      // the half stage: its second 32 K steps read as zeros (offsets past
      // both buffers' ends)
      uint32_t av[C::A_INST], bv[C::B_INST];
#pragma unroll
      for (int i = 0; i < C::A_INST; ++i) av[i] = a_chk[i] < 4 ? a_src[i] : 0x80000000u;
#pragma unroll
      for (int i = 0; i < C::B_INST; ++i) bv[i] = b_row[i] < 32 ? b_src[i] : 0x80000000u;
      dma16_run<C::A_INST>(rA, slot + wave_u * C::A_INST * 1024, av, ka);
      dma16_run<C::B_INST>(rB, slot + C::A_BYTES + wave_u * C::B_INST * 1024, bv, kb);
    } else {
      dma16_run<C::A_INST>(rA, slot + wave_u * C::A_INST * 1024, a_src, ka);
      dma16_run<C::B_INST>(rB, slot + C::A_BYTES + wave_u * C::B_INST * 1024, b_src, kb);
    }
    --half;
    ka += C::BK * 2;
    kb += (uint32_t)(C::BK * p.ldb * 2);
    wr = next_slot(wr);
  };
  f32x16 acc[C::FM][C::FN];
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
  auto compute = [&] {
    const char* sA = smem + rd;
    const char* sB = sA + C::A_BYTES;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      bf16x8 af[C::FM], bf[C::FN];
#pragma unroll
      for (int i = 0; i < C::FM; ++i) af[i] = *reinterpret_cast<const bf16x8*>(sA + a_rd[kk] + i * 32 * 128);
#pragma unroll
      for (int jj = 0; jj < C::FN; ++jj) {
        const bf16x4_t lo = lds_tr4(sB + b_rd[jj] + kk * 16 * C::BROW);
        const bf16x4_t hi = lds_tr4(sB + b_rd[jj] + kk * 16 * C::BROW + 4 * C::BROW);
        bf[jj] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      }
#pragma unroll
      for (int i = 0; i < C::FM; ++i)
#pragma unroll
        for (int jj = 0; jj < C::FN; ++jj)
          acc[i][jj] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bf[jj], af[i], acc[i][jj], 0, 0, 0);
    }
    rd = next_slot(rd);
  };

#pragma unroll
  for (int s = 0; s < C::S - 1; ++s)
    if (s < n) issue();
  // Each barrier says that every wave's share of stage j has landed and that
  // every wave has read stage j - 1, whose slot the next DMA overwrites.
  int j = 0;
  for (; j + C::S - 1 < n; ++j) {
    wait_vm<(C::S - 2) * C::LOADS>();
    __syncthreads();
    issue();
    compute();
  }
  for (; j < n; ++j) {
    wait_pending<C::S - 2, C::LOADS>(n - 1 - j);
    __syncthreads();
    compute();
  }
  __syncthreads();  // the ring is free: the exchange and the store use it
  if (!REDUCE && p.split > 1) {
    const int parts = p.split, w0 = (int)t * parts;  // the tile's first workgroup, whose slots its parts use
    int* sh = reinterpret_cast<int*>(smem);
    uint32_t* ticket = p.words + t;
    uint32_t* head = p.words + p.tiles_m * p.tiles_n + w0;  // one per part but the last
    if (tid == 0) sh[0] = (int)__hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const int tk = __builtin_amdgcn_readfirstlane(sh[0]);
    float* slot0 = p.ws + (int64_t)w0 * (C::BM * C::BN);
    if (tk < parts - 1) {
      part_out<C>(slot0 + (int64_t)tk * (C::BM * C::BN), acc, tid);
      // write-through stores performed at agent scope, then a relaxed flag
      wait_vmem_all();
      __syncthreads();
      if (tid == 0)
        __hip_atomic_store(head + tk, part + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
    if (tid < parts - 1) {
      uint32_t h;
      while ((h = __hip_atomic_load(head + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == 0u)
        __builtin_amdgcn_s_sleep(1);
      sh[1 + (h - 1u)] = tid;
      // every part is in: both words are clear for the next launch
      __hip_atomic_store(head + tid, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (tid == 0) __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    parts_in<C>(slot0, sh + 1, parts, (int)part, acc, tid);
    __syncthreads();  // sh is read: the store reuses the LDS
  }
  if (REDUCE && m0 >= p.rs_own_row0 && m0 < p.rs_own_row0 + p.rs_own_rows) {
    static_assert(!REDUCE || C::WAVES * 32 * (C::WTN * 4 + 16) <= C::LDS_BYTES, "fold rows in LDS");
    reduce_rows<C, 8, true>(p, acc, m0 - p.rs_own_row0 + wm * C::WTM, n0 + wn * C::WTN, smem, wave, lane);
    if (p.done) part_done<C>(p, m0 - p.rs_own_row0, n0, tid);
  } else {
    // with the fold these are the would-be sends: written once, not read here
    store_rows<C, C::FN, REDUCE>(p.C + (int64_t)(m0 + wm * C::WTM) * p.ldc + n0 + wn * C::WTN, p.ldc, acc, smem, wave,
                                 lane);
  }
}

template <class C, bool REDUCE>
hipError_t launch_s(const GemmSmallParams& p, int grid, hipStream_t stream) {
  static PerDeviceFlag attr_set;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (!attr_set.is_set(dev)) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_small_kernel<C, REDUCE>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS_BYTES);
    if (e != hipSuccess) return e;
    attr_set.set(dev);
  }
  hipLaunchKernelGGL((gemm_small_kernel<C, REDUCE>), dim3(grid), dim3(C::NT), C::LDS_BYTES, stream, p);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_gemm_small(const GemmSmallParams& p, const GemmSmallPlan& plan, bool reduce, hipStream_t stream) {
  const int grid = plan.grid;
  switch (plan.tile * 2 + reduce) {
    case 0: return launch_s<SCfg<64, 64, 2, 2, 3>, false>(p, grid, stream);
    case 1: return launch_s<SCfg<64, 64, 2, 2, 3>, true>(p, grid, stream);
    case 2: return launch_s<SCfg<128, 64, 4, 1, 3>, false>(p, grid, stream);
    case 3: return launch_s<SCfg<128, 64, 4, 1, 3>, true>(p, grid, stream);
    case 4: return launch_s<SCfg<128, 128, 4, 2, 4>, false>(p, grid, stream);
    case 5: return launch_s<SCfg<128, 128, 4, 2, 4>, true>(p, grid, stream);
    case 6: return launch_s<SCfg<192, 128, 2, 4, 4>, false>(p, grid, stream);
    case 8: return launch_s<SCfg<128, 256, 2, 4, 3>, false>(p, grid, stream);
    case 9: return launch_s<SCfg<128, 256, 2, 4, 3>, true>(p, grid, stream);
    case 10: return launch_s<SCfg<128, 128, 2, 4, 2>, false>(p, grid, stream);
    case 11: return launch_s<SCfg<128, 128, 2, 4, 2>, true>(p, grid, stream);
    case 13: return launch_s<SCfg<64, 64, 2, 2, 2>, true>(p, grid, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace mk
