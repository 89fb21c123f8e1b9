// mk_tile.h — building blocks of the tiled bf16 GEMM kernels (gfx950): HBM ->
// LDS DMA with hand-counted completion, the transposing LDS read, the grouped
// tile order, the row-major bf16 store of a wave's accumulators and the fold of
// peers' partials into them.
#pragma once
#include "mk_device.h"

namespace mk {

typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t v2u32_t __attribute__((ext_vector_type(2)));

// Grouped ("super-M") order: runs of group_m row tiles are walked
// column-major so concurrently running workgroups share A rows and B columns
// (reference src/ag_gemm.cu:230-253 uses SUPER_M=12 for the same purpose).
__device__ __forceinline__ void decode_grouped(int t, int tiles_m, int tiles_n, int group_m,
                                               int& tm, int& tn) {
  const int group = group_m * tiles_n;
  const int g = t / group;
  const int first = g * group_m;
  const int gm = min(tiles_m - first, group_m);
  const int r = t - g * group;
  tm = first + r % gm;
  tn = r / gm;
}

// ---------------------------------------------------------------------------
// LDS-DMA helpers
// ---------------------------------------------------------------------------

// Raw buffer descriptor (gfx9 word 3) for inline-asm buffer instructions.
__device__ __forceinline__ u32x4_t make_rsrc_v(const void* base, uint32_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  u32x4_t r;
  r[0] = __builtin_amdgcn_readfirstlane((uint32_t)a);
  r[1] = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32) & 0xffffu);
  r[2] = __builtin_amdgcn_readfirstlane(bytes);
  r[3] = 0x00020000u;
  return r;
}

// 16-byte buffer load straight into LDS: lane l's 16 bytes land at
// lds_addr + 16*l.  Issued through inline asm so the compiler does not
// serialise every later LDS read behind it; completion is tracked by hand
// with wait_stage (vmcnt) followed by a workgroup barrier.
// The compiler's hazard pass does not look inside inline asm, so the wait
// states are written here: a VMEM instruction that reads an SGPR written by a
// VALU instruction (v_readlane / v_readfirstlane, e.g. a reloaded SGPR spill)
// needs 5 wait states, and an LDS DMA after an SALU write of M0 needs 1.
// Without them the load can use a stale rsrc / soffset and fetch wrong bytes.
// M0 is listed as clobbered; the compiler reports that it does not preserve
// a reserved register across inline asm, so it must hold nothing live here.
// In the generated code the compiler's own M0 uses (v_writelane lane
// selects in atomic expansions) set M0 immediately before the use, with no
// DMA between.
__device__ __forceinline__ void dma16(u32x4_t r, uint32_t lds_addr, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "s"(lds_addr), "v"(voff), "s"(r), "s"(soff)
               : "memory", "m0");
}

// Two LDS DMAs in one asm statement (nothing can be scheduled between them),
// so the 5-wait-state guard is paid once per pair.
__device__ __forceinline__ void dma16x2(u32x4_t r, uint32_t lds0, uint32_t lds1, uint32_t v0, uint32_t v1,
                                        uint32_t soff) {
  asm volatile(
      "s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %2, %4, %5 offen lds\n\t"
      "s_mov_b32 m0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %3, %4, %5 offen lds"
      :
      : "s"(lds0), "s"(lds1), "v"(v0), "v"(v1), "s"(r), "s"(soff)
      : "memory", "m0");
}

// N DMAs into consecutive 1 KB LDS blocks starting at lds, paired.
template <int N>
__device__ __forceinline__ void dma16_run(u32x4_t r, uint32_t lds, const uint32_t (&voff)[N], uint32_t soff) {
#pragma unroll
  for (int i = 0; i + 1 < N; i += 2) dma16x2(r, lds + i * 1024, lds + (i + 1) * 1024, voff[i], voff[i + 1], soff);
  if constexpr (N % 2) dma16(r, lds + (N - 1) * 1024, voff[N - 1], soff);
}

// s_waitcnt vmcnt(n) (n <= 63), other counters untouched (gfx9 encoding).
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// Wait until at most `pending` of this thread's most recent stages (L DMA
// instructions each) are still in flight, i.e. every older stage has landed.
template <int S, int L>
__device__ __forceinline__ void wait_stage(int pending) {
  static_assert(S <= 7 && (S - 1) * L < 64, "ring too deep for the waitcnt ladder");
  if (pending >= 5 && S > 5) { wait_vm<(S > 5 ? 5 * L : 0)>(); return; }
  if (pending >= 4 && S > 4) { wait_vm<(S > 4 ? 4 * L : 0)>(); return; }
  if (pending >= 3 && S > 3) { wait_vm<(S > 3 ? 3 * L : 0)>(); return; }
  if (pending >= 2 && S > 2) { wait_vm<2 * L>(); return; }
  if (pending >= 1) { wait_vm<L>(); return; }
  wait_vm<0>();
}

__device__ __forceinline__ bf16x4_t lds_tr4(const char* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
      (__attribute__((address_space(3))) bf16x4_t*)((__attribute__((address_space(3))) char*)(p)));
}

// s_waitcnt lgkmcnt(0), other counters untouched (gfx9 encoding).
__device__ __forceinline__ void wait_lgkm_all() { __builtin_amdgcn_s_waitcnt(0xC07F); }

// Row-major store of a wave's WTM x WTN bf16 sub-tile through a private LDS
// region.  The accumulator layout gives each lane 4 consecutive columns of
// one row, so a direct store instruction touches 32 rows with 16 bytes each:
// a 128 KB tile became ~1000 partial-line L2 writes per wave, and the tile
// epilogue took 13 us of a 200 us tile.  Here each 32-row block goes to LDS
// as rows of WTN bf16 (row pitch padded by 16 bytes, so the 8-byte writes of
// the 32 rows spread over the banks), then comes back 16 bytes per lane
// with consecutive lanes along a row: every store instruction writes whole
// WTN*2-byte row segments.  The region is the wave's own, so only this
// wave's LDS ordering matters (lgkmcnt waits); the caller's workgroup
// barrier must precede the next use of the ring.
template <class C, int NJ = C::FN, bool NT = false>
__device__ __forceinline__ void store_rows(uint16_t* base, int64_t ldc, f32x16 (&acc)[C::FM][C::FN], char* smem,
                                           int wave, int lane) {
  constexpr int W = NJ * 32;              // columns stored per row: accumulator blocks j < NJ
  constexpr int PITCH = W * 2 + 16;       // bytes per LDS row
  constexpr int LPR = W * 2 / 16;         // lanes per row (16 bytes each)
  constexpr int RPI = 64 / LPR;           // rows per store instruction
  static_assert(64 % LPR == 0 && 32 % RPI == 0, "store_rows shape");
  // The lane index goes through an empty asm so that nothing derived from
  // it is hoisted above the K loop (it would stay live across the loop and
  // push the loop's operand registers into spills).
  int l = lane;
  asm volatile("" : "+v"(l));
  const int ml = l & 31, kg = l >> 5;
  char* reg = smem + wave * 32 * PITCH;
  const int rr = l / LPR, cc = l % LPR;
#pragma unroll
  for (int i = 0; i < C::FM; ++i) {
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        uint2 w;
        w.x = pack_bf16x2(acc[i][j][4 * a + 0], acc[i][j][4 * a + 1]);
        w.y = pack_bf16x2(acc[i][j][4 * a + 2], acc[i][j][4 * a + 3]);
        *reinterpret_cast<uint2*>(reg + ml * PITCH + (32 * j + 8 * a + 4 * kg) * 2) = w;
      }
    wait_lgkm_all();
#pragma unroll
    for (int r = 0; r < 32 / RPI; ++r) {
      const int row = r * RPI + rr;
      const uint4 v = *reinterpret_cast<const uint4*>(reg + row * PITCH + cc * 16);
      uint4* dst = reinterpret_cast<uint4*>(base + (int64_t)(i * 32 + row) * ldc + cc * 8);
      if constexpr (NT) {
        typedef uint32_t nt_u32x4 __attribute__((ext_vector_type(4)));
        __builtin_nontemporal_store(nt_u32x4{v.x, v.y, v.z, v.w}, reinterpret_cast<nt_u32x4*>(dst));
      } else {
        *dst = v;
      }
    }
    wait_lgkm_all();  // this block's reads are done before the next block's writes
  }
}

// x += 8 columns of n <= G partials, in order, their loads in flight together
// (indices clamped to the last, so no branch splits the loads; the empty asm
// keeps the compiler from moving each load to its adds, one latency after
// another: ReduceScatter 4096x4096x256 of world 16 took 49.5 us so, 37.9 with
// it; groups of 8 for all but the first peers made one peer's fold 5 % slower).
template <int G>
__device__ __forceinline__ void fold_group(const uint16_t* src, int64_t peer_stride, int n, float (&x)[8]) {
  uint4 v[G];
#pragma unroll
  for (int u = 0; u < G; ++u) v[u] = *reinterpret_cast<const uint4*>(src + (int64_t)min(u, n - 1) * peer_stride);
#pragma unroll
  for (int u = 0; u < G; ++u) asm volatile("" : "+v"(v[u].x), "+v"(v[u].y), "+v"(v[u].z), "+v"(v[u].w));
#pragma unroll
  for (int u = 0; u < G; ++u)
    if (u < n) {
      x[0] += bf16_lo(v[u].x); x[1] += bf16_hi(v[u].x);
      x[2] += bf16_lo(v[u].y); x[3] += bf16_hi(v[u].y);
      x[4] += bf16_lo(v[u].z); x[5] += bf16_hi(v[u].z);
      x[6] += bf16_lo(v[u].w); x[7] += bf16_hi(v[u].w);
    }
}

// Reduce epilogue of an owned tile, row-major: each 32-row block of the
// wave's fp32 accumulators goes through the wave's LDS region (rows of WTN
// fp32, pitch padded by 16 bytes) and comes back 8 columns per lane with
// consecutive lanes along a row; the lane then loads the same 8 columns of
// every peer's bf16 partial (16 bytes per peer: whole row segments per
// instruction, kPeers peers' loads in flight, the remainder as one more group),
// adds them in rank order in fp32
// (deterministic, one rounding) and stores 16 bytes of the owned output.
// In the accumulator layout every load and store instruction would touch
// 32 rows with 8 bytes each.  SMALL (the small-tile kernel; the 256-row kernel
// has no registers left for it): the last peers by fold_group, and with p.done
// the output goes out write-through (performed at agent scope once vmcnt says
// it is stored, the protocol of copy_wt), for a flag that needs no L2
// write-back.
template <class C, int kPeers = 4, bool SMALL = false, class P>
__device__ __forceinline__ void reduce_rows(const P& p, f32x16 (&acc)[C::FM][C::FN], int lrow0, int col0,
                                            char* smem, int wave, int lane) {
  constexpr int PITCH = C::WTN * 4 + 16;  // bytes per LDS row (fp32)
  constexpr int LPR = C::WTN / 8;         // lanes per row (8 columns each)
  constexpr int RPI = 64 / LPR;           // rows per instruction
  static_assert(64 % LPR == 0 && 32 % RPI == 0, "reduce_rows shape");
  int l = lane;
  asm volatile("" : "+v"(l));  // keep lane-derived addressing below the K loop
  const int ml = l & 31, kg = l >> 5;
  char* reg = smem + wave * 32 * PITCH;
  const int rr = l / LPR, cc = l % LPR;
  const int64_t peer_stride = (int64_t)p.rs_own_rows * p.ldc;
  const int np = p.rs_npeers;
  // the wave's rows, from its first column on
  const __amdgpu_buffer_rsrc_t out = make_rsrc(
      p.rs_out + (int64_t)__builtin_amdgcn_readfirstlane(lrow0) * p.ldc + __builtin_amdgcn_readfirstlane(col0),
      (uint32_t)(((C::WTM - 1) * p.ldc + C::WTN) * 2));
#pragma unroll
  for (int i = 0; i < C::FM; ++i) {
#pragma unroll
    for (int j = 0; j < C::FN; ++j)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        f32x4 w;
#pragma unroll
        for (int b = 0; b < 4; ++b) w[b] = acc[i][j][4 * a + b];
        *reinterpret_cast<f32x4*>(reg + ml * PITCH + (32 * j + 8 * a + 4 * kg) * 4) = w;
      }
    wait_lgkm_all();
    for (int r = 0; r < 32 / RPI; ++r) {
      const int row = r * RPI + rr;
      const f32x4 lo = *reinterpret_cast<const f32x4*>(reg + row * PITCH + cc * 32);
      const f32x4 hi = *reinterpret_cast<const f32x4*>(reg + row * PITCH + cc * 32 + 16);
      float x[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      const uint16_t* src = p.rs_recv + (int64_t)(lrow0 + i * 32 + row) * p.ldc + col0 + cc * 8;
      int q = 0;
      for (; q + kPeers <= np; q += kPeers) {
        uint4 v[kPeers];
#pragma unroll
        for (int u = 0; u < kPeers; ++u) v[u] = *reinterpret_cast<const uint4*>(src + (q + u) * peer_stride);
#pragma unroll
        for (int u = 0; u < kPeers; ++u) {
          x[0] += bf16_lo(v[u].x); x[1] += bf16_hi(v[u].x);
          x[2] += bf16_lo(v[u].y); x[3] += bf16_hi(v[u].y);
          x[4] += bf16_lo(v[u].z); x[5] += bf16_hi(v[u].z);
          x[6] += bf16_lo(v[u].w); x[7] += bf16_hi(v[u].w);
        }
      }
      if constexpr (SMALL) {
        const uint16_t* rest = src + q * peer_stride;
        if (np - q > 4) fold_group<kPeers>(rest, peer_stride, np - q, x);
        else if (np - q > 1) fold_group<4>(rest, peer_stride, np - q, x);
        else if (np - q == 1) fold_group<1>(rest, peer_stride, 1, x);
      } else if (q < np) {
        // the last np - q peers as one more group in flight (indices
        // clamped to the last peer, so no branch splits the loads)
        uint4 v[kPeers];
#pragma unroll
        for (int u = 0; u < kPeers; ++u)
          v[u] = *reinterpret_cast<const uint4*>(src + (int64_t)min(q + u, np - 1) * peer_stride);
#pragma unroll
        for (int u = 0; u < kPeers; ++u)
          if (q + u < np) {
            x[0] += bf16_lo(v[u].x); x[1] += bf16_hi(v[u].x);
            x[2] += bf16_lo(v[u].y); x[3] += bf16_hi(v[u].y);
            x[4] += bf16_lo(v[u].z); x[5] += bf16_hi(v[u].z);
            x[6] += bf16_lo(v[u].w); x[7] += bf16_hi(v[u].w);
          }
      }
      uint4 o;
      o.x = pack_bf16x2(x[0], x[1]); o.y = pack_bf16x2(x[2], x[3]);
      o.z = pack_bf16x2(x[4], x[5]); o.w = pack_bf16x2(x[6], x[7]);
      if constexpr (SMALL)
        if (p.done) {
          __builtin_amdgcn_raw_buffer_store_b128(u32x4_t{o.x, o.y, o.z, o.w}, out,
                                                 (int)(((i * 32 + row) * p.ldc + cc * 8) * 2), 0, 0x10 /* SC1 */);
          continue;
        }
      typedef uint32_t nt_u32x4 __attribute__((ext_vector_type(4)));
      __builtin_nontemporal_store(nt_u32x4{o.x, o.y, o.z, o.w},
                                  reinterpret_cast<nt_u32x4*>(p.rs_out + (int64_t)(lrow0 + i * 32 + row) * p.ldc +
                                                              col0 + cc * 8));
    }
    wait_lgkm_all();  // this block's reads are done before the next block's writes
  }
}

}  // namespace mk
