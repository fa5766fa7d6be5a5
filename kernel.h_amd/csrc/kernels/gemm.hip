// fp32 GEMM for gfx950 on the matrix cores: C[m,n] = A[m,k] B[k,n],
// row-major, v_mfma_f32_32x32x2f32 (and v_mfma_f32_16x16x4f32 for the
// 64x64-tile pipelines where it measured faster).
//
// Symbol and memref arguments follow the reference template
// (lib/dsl/kernels/gemm.cpp:116-296): A [m,k], B [k,n], C [m,n], rank 2,
// 21 parameters. The reference computes one element per lane with scalar
// FMAs out of an 8 KiB LDS tile (gemm.cpp:265-296). Here:
//
//   * Workgroup = 256 threads (4 wave64s, 2x2; `gemm_wide`: 512, 4x2)
//     computing a BM x BN tile of C; each wave owns its part as WTM x WTN
//     MFMA accumulator blocks. Five such symbols, all correct for every
//     shape; the launcher scores each by its full-occupancy rate times how
//     busy its last round of workgroups would be (kh_tiles.h) and takes the
//     best, unless the launch has at most 256 tiles of 32x64, or fewer
//     than 256 tiles of 64x64 with whole 32x32 tiles and K a multiple of 128
//     (then a `gemm_ksplit*`, at the end of this file, splits K over 8
//     waves instead); a tune cache, when set, overrides the choice:
//       `gemm`        128x256 tiles (64x128 per wave, 128 accumulator registers
//                     per lane), 16-deep K slabs: the least LDS and L2 traffic
//                     per MFMA (8192^3, 4096^3, 8192x8192x256); persistent
//                     workgroups, two per CU, each looping over its tiles;
//       `gemm_mid`    128x128 tiles (64x64 per wave), 32-deep slabs (the
//                     tune cache's; `gemm_wide` outscores it wherever both
//                     fit);
//       `gemm_small`  64x64 tiles on eight waves of 16x16 MFMAs (16x32 per
//                     wave) in the persistent direct-to-LDS ring, two
//                     workgroups per CU, for grids the larger tiles would
//                     fill unevenly (1024^3, 960^3, 1536^3 to 3584^3);
//       `gemm_small_pf2` 64x64 tiles on four waves of 16x16 MFMAs with
//                     two-ahead register prefetch (the tune cache's);
//       `gemm_wide`   128x128 tiles on eight waves of 16x16 MFMAs (32x64
//                     per wave), 32-deep slabs in `gemm`'s persistent
//                     direct-to-LDS ring, one workgroup per CU, where its
//                     tiles fill whole rounds (2048^3, 6144x6144x1024,
//                     2048x2048x8192, 4096x2048x4096, 8192x1024x8192).
//     Registers are capped for two waves per SIMD (two workgroups per CU, as
//     LDS allows), so one workgroup's barrier and slab hand-over overlap the
//     other's MFMAs. `gemm` and `gemm_mid` raise their waves' priority
//     (s_setprio) while they issue MFMAs, so a wave that is feeding the
//     matrix core wins issue over one that is between slabs (+2% each).
//   * K advances in slabs staged through LDS. `gemm` loads its slabs straight
//     into LDS (buffer_load_dwordx4 ... lds) through three stages: slab ks+2
//     is in flight while slab ks is consumed, and the one barrier per slab sits
//     after the slab's first 8-deep chunk, so the next slab's first fragments
//     are read while the rest of this one feeds the MFMAs. Against staging the
//     slab through registers and ds_write (still used by `gemm_mid` and
//     `gemm_small_pf2`) that is +2% at 8192^3: the
//     stores and the wait for them sat between a wave's last MFMA of one slab
//     and its first of the next.
//   * LDS holds A as [m][k] (one ds_read_b128 per lane delivers four k
//     values) and B as [k][n] (a half-wave reads 32 consecutive n with
//     ds_read_b32), both conflict-free: rows padded by 4 floats when slabs are
//     staged through registers; for direct-to-LDS slabs, whose loads write 64
//     float4s contiguously, A's rows are unpadded with their float4s
//     XOR-swizzled and B's rows padded per group a wave loads. The
//     direct-to-LDS symbols' slab loads are unconditional at any alignment and
//     extent: a dwordx4 buffer load needs 4-byte alignment only and is
//     range-checked dword by dword, and what it carries past K is zeroed in
//     the fragments of a tile's last slabs (or, for short K that is a multiple
//     of 4, selected away in the loads). The register-staged ones' are
//     branch-free buffer loads for aligned operands with k, n multiples of 4,
//     whose range checks zero-fill the tails (the guarded per-element form of
//     the generic path made the compiler split every load into branches and
//     dword pieces, which cost 15% of the MFMA rate).
//   * K order inside an MFMA: the instruction sums k over its two lane
//     halves, and any permutation of k applied to both operands gives the
//     same product. Lane half h reads k = 8c + 4h + {0..3}; MFMA step s of
//     chunk c consumes k = 8c + s (half 0) and 8c + 4 + s (half 1).
//   * Tiles are ordered for the 8 XCDs (each with its own L2): consecutive
//     workgroups go round-robin to XCDs, so the launch index is remapped to
//     give every XCD a contiguous range of tiles, grouped 8 tile-rows deep
//     so neighbouring workgroups share A rows and B columns in L2.
//
// Tails in m, n and k are zero-filled on load and guarded on store, so any
// shape is correct; tiles are grid-strided so any grid is correct, including
// the reference's ceil(m/32) x 256 geometry (kernelh_backend.cpp:225).
// Accumulation is fp32 throughout (the MFMA accumulates in fp32).
#include "gemm_tiles.h"

using khg::Tile;
using khg::gemm_entry;
using khg::kThreads;

static_assert(Tile<2, 4, 16, true>::BM == KH_GEMM_BM && Tile<2, 4, 16, true>::BN == KH_GEMM_BN, "launcher tile size");
static_assert(Tile<2, 2, 32, false>::BM == KH_GEMM_MID_BM && Tile<2, 2, 32, false>::BN == KH_GEMM_MID_BN,
              "launcher tile size");
static_assert(Tile<1, 2, 32, true, 4, 2, 16>::BM == KH_GEMM_SMALL_BM &&
                  Tile<1, 2, 32, true, 4, 2, 16>::BN == KH_GEMM_SMALL_BN &&
                  Tile<1, 2, 32, true, 4, 2, 16>::BK == KH_GEMM_SMALL_BK &&
                  Tile<1, 2, 32, true, 4, 2, 16>::NT == KH_GEMM_SMALL_THREADS &&
                  Tile<2, 2, 32, false, 2, 2, 16>::BM == KH_GEMM_SMALL_BM &&
                  Tile<2, 2, 32, false, 2, 2, 16>::BN == KH_GEMM_SMALL_BN,
              "launcher tile size (gemm_small and gemm_small_pf2)");
static_assert(Tile<2, 4, 32, true, 4, 2, 16>::BM == KH_GEMM_WIDE_BM &&
                  Tile<2, 4, 32, true, 4, 2, 16>::BN == KH_GEMM_WIDE_BN &&
                  Tile<2, 4, 32, true, 4, 2, 16>::NT == KH_GEMM_WIDE_THREADS,
              "launcher tile size (gemm_wide)");

// Entry of a symbol whose tile split assumes THREADS one-dimensional
// threads per workgroup: the arguments in one round, then any other launch
// shape refused by writing NaN over C (khg::refuse_launch) instead of
// computing part of each tile.
#define KH_GEMM_ENTRY_CHECK(THREADS)                                                                            \
  const uint32_t gxy = kh::group_size_word(), gz = kh::group_size_z_word();                                   \
  KH_GEMM_ARGS_READY(gxy, gz);                                                                                 \
  if (kh::threads_x_of(gxy) != (THREADS) || kh::threads_y_of(gxy) != 1 || kh::threads_z_of(gz) != 1) {       \
    khg::refuse_launch(KH_PTR(C), C_n0, C_n1, C_s0);                                                           \
    return;                                                                                                    \
  }

// The reference symbol: 128x256 tiles, persistent. Each workgroup loops
// over tiles bid, bid + grid, ... (the launcher gives it min(tiles, two per
// CU) workgroups; any grid is correct) and the three-stage slab ring runs on
// across them, so a tile starts with its first two slabs already fetched.
// Against one tile per workgroup (the previous form of this symbol, same
// box): 8192^3 143.4 vs 142.0, 8192x8192x256 125.4 vs 123.0 TFLOP/s. Writing C
// as float4s (MFMA operands swapped so a lane holds four consecutive
// columns) let the stores overlap the next tile, but its 32-byte row pieces
// doubled the kernel's L2 misses and measured 0.7% slower at 8192^3; C goes
// out as whole 128-byte lines. K <= 16 takes the per-tile pipeline (or the
// generic path).
extern "C" __global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
gemm(KH_MEMREF2(const float, A), KH_MEMREF2(const float, B), KH_MEMREF2(float, C)) {
  KH_GEMM_ENTRY_CHECK(kThreads);
  khg::gemm_entry_flat<2, 4, 16, true>(KH_PTR(A), KH_PTR(B), KH_PTR(C), A_n0, B_n1, A_n1, A_s0, B_s0, C_s0);
}

// Same arguments and results with 128x128 tiles.
extern "C" __global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
gemm_mid(KH_MEMREF2(const float, A), KH_MEMREF2(const float, B), KH_MEMREF2(float, C)) {
  KH_GEMM_ENTRY_CHECK(kThreads);
  gemm_entry<2, 2, 32, true, false>(KH_PTR(A), KH_PTR(B), KH_PTR(C), A_n0, B_n1, A_n1, A_s0, B_s0, C_s0);
}

// Same arguments and results with 64x64 tiles on eight waves (4 x 2, each
// 16x32 as 1x2 blocks of v_mfma_f32_16x16x4f32), 32-deep slabs through
// `gemm`'s persistent direct-to-LDS ring; 49.5 KB of LDS and 83 VGPRs, so
// two workgroups per CU. Kernel trace, interleaved launches, same bits,
// against the 64x64 tiles it replaced (four waves, register-staged
// slabs; and `gemm_small_pf2` where that was the launcher's choice):
// 1024^3 28.2 -> 23.7 us, 1024x1024x512 16.3 -> 13.5-14.9,
// 1024x1024x8192 201.5 -> 160.9, 1536^3 86.8 -> 83.6, 2048x1024x1024 45.0
// -> 41.9, 2560^3-3584^3 within 1.3%. One workgroup per CU: 1536^3 91.0.
// The tile split assumes 512 threads: any other launch is refused by
// writing NaN over C.
extern "C" __global__ void __launch_bounds__(KH_GEMM_SMALL_THREADS) __attribute__((amdgpu_waves_per_eu(2)))
gemm_small(KH_MEMREF2(const float, A), KH_MEMREF2(const float, B), KH_MEMREF2(float, C)) {
  KH_GEMM_ENTRY_CHECK(KH_GEMM_SMALL_THREADS);
  khg::gemm_entry_flat<1, 2, 32, true, 4, 2, 16>(KH_PTR(A), KH_PTR(B), KH_PTR(C), A_n0, B_n1, A_n1, A_s0, B_s0,
                                                 C_s0);
}

// Same arguments and results with 64x64 tiles on v_mfma_f32_16x16x4f32 (each
// wave 32x32 as 2x2 blocks of 16x16), 32-deep slabs prefetched two ahead
// through registers: more loads in flight per CU, for grids of many tiles.
// The tune space found the 16x16 form faster than the same tiles on 32x32
// MFMAs at every shape timed (rotated U[-1,1] inputs, warm clocks): 2048^3
// 121.5 vs 117.0, 3072^3 123.4 vs 114.2, 2048x2048x8192 127.6 vs 108.1,
// 6144x6144x1024 125.0 vs 121.1 TFLOP/s; level at 1536^3. The persistent
// eight-wave `gemm_small` has since matched or beaten it at every shape
// timed, so the launcher no longer picks it; a tune cache can.
extern "C" __global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
gemm_small_pf2(KH_MEMREF2(const float, A), KH_MEMREF2(const float, B), KH_MEMREF2(float, C)) {
  KH_GEMM_ENTRY_CHECK(kThreads);
  khg::gemm_entry_pipe<2, 2, 32, true, khg::kPipePrefetch2, 2, 2, 16>(KH_PTR(A), KH_PTR(B), KH_PTR(C), A_n0, B_n1,
                                                                      A_n1, A_s0, B_s0, C_s0);
}

// Same arguments and results with 128x128 tiles on eight waves (4 x 2,
// each 32x64 as 2x4 blocks of v_mfma_f32_16x16x4f32), 32-deep slabs through
// `gemm`'s persistent three-stage direct-to-LDS ring (99 KB of LDS: one
// workgroup per CU, two waves per SIMD). Kernel trace against the previous
// `gemm_wide` (64x128 tiles, register-staged slabs), variants interleaved
// launch by launch, same bits: 2048^3 145.2 -> 133.9 us, 6144x6144x1024
// 586.5 -> 557.1, 2048x2048x8192 528.8 -> 487.1; and against `gemm_mid` at
// 4096x2048x4096 529.3 -> 496.9, 8192x1024x8192 1018 -> 965. The same tile
// with the waves 2 x 4 (64x32 each) ran 137.6 us at 2048^3, sixteen waves
// 140.5, 64x128 tiles two per CU 137.8, without s_setprio 137.0. The tile
// split assumes 512 threads: any other launch is refused by writing NaN
// over C.
extern "C" __global__ void __launch_bounds__(KH_GEMM_WIDE_THREADS) __attribute__((amdgpu_waves_per_eu(2)))
gemm_wide(KH_MEMREF2(const float, A), KH_MEMREF2(const float, B), KH_MEMREF2(float, C)) {
  KH_GEMM_ENTRY_CHECK(KH_GEMM_WIDE_THREADS);
  khg::gemm_entry_flat<2, 4, 32, true, 4, 2, 16>(KH_PTR(A), KH_PTR(B), KH_PTR(C), A_n0, B_n1, A_n1, A_s0, B_s0,
                                                 C_s0);
}


// Small tiles with K split over the workgroup's waves (8 at the launcher's
// 512 threads; any 64..512 threads, a multiple of 64, are correct), for
// launches whose larger tiles leave most CUs idle: 512^3 has 64 tiles of
// 64x64 for 256 CUs, and 256 tiles of 32x32. Each wave accumulates the
// products of its contiguous K range straight from global memory, without
// LDS; the partial tiles meet in LDS, where every output is summed in the
// fixed order w0 + w1 + ... : the result does not depend on timing.
//
// Every load is an unconditional buffer load, at any alignment and extent
// (ks_any): rows of A past M and rows of B past the wave's K range read 0
// through the range check, columns of B past N are not stored, and A's k past
// the range are zeroed in registers in the range's last batch. An earlier
// form loaded a clamped address and selected 0 for lanes out of range; the
// compiler turned each such pair into a branch around the load with a wait
// where the branches join, so a wave's loads went out one at a time.
//
// What bounds it: a wave has two batches of loads in flight, and a tile's
// time is its K range's batches at that latency, or its bytes of A and B at
// the CU's share of the cache bandwidth. So the tile is chosen to give each
// CU one workgroup (the launcher: the smallest tile with at most
// KH_GEMM_CUS tiles). Events around rotated launches, 8 waves each,
// 16x16 / 32x16 / 32x32 / 32x64 tiles, and the kernel these shapes ran
// before (in us):
//   16x4096x4096     17.6 / 19.3 / 23.9 / 38.4   89.7
//   100x777x555       6.8 /  6.0 /  6.8 /  9.7   21.6
//   2000x128x8192    84.3 / 70.6 / 48.8 / 73.3   187
//   333x1000x2000    41.4 / 28.8 / 25.3 / 22.6   40.8 (64x64 tiles)
//   8192x64x1000     21.1 / 18.9 / 15.5 / 14.6   22.9 (64x64 tiles)
//   20x100x8000      26.1 / 34.2 / 43.9 / 70.5   107
// Sixteen waves per workgroup and twice the loads in flight measured level;
// B in dwordx2 and dwordx4 loads (a lane holding neighbouring columns) 5%
// slower; 64x16 and 64x32 tiles never best.
namespace {

using khg::v16f;
using khg::v4f;
using kh::u32x4_t;
constexpr int kKsTile = KH_GEMM_KSPLIT_BM;
constexpr int kKsMaxWaves = KH_GEMM_KSPLIT_THREADS / 64;
constexpr int kKsFastBatch = 2;  // groups of 8 k loaded ahead per batch in ks_interior
static_assert(KH_GEMM_KSPLIT_BM == 32 && KH_GEMM_KSPLIT_BN == 32, "one 32x32 MFMA accumulator per wave");

// A uniform pointer, forced into scalar registers: its computation may run
// on the vector ALU (the 64-bit multiply of a row index), and a buffer
// resource built from vector registers costs a loop around every load.
template <typename T>
__device__ __forceinline__ T *uniform_ptr(T *p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return reinterpret_cast<T *>(((uint64_t)hi << 32) | lo);
}

// 32x32 tiles for launches whose tiles are all whole: M, N multiples of 32,
// K of 8 * kKsFastBatch * 8, eight waves, and every buffer span below 2^31
// bytes, the largest record count a buffer resource holds (ks_interior_ok).
// One v_mfma_f32_32x32x2f32 accumulator: lane l (r = l % 32, h = l / 32) loads
// the float4 A[m0 + r][k + 4h .. k + 4h + 3] and the four B[k + 4h + i][n0 + r],
// so MFMA i of a group of 8 k sums k + i (lanes 0-31) and k + 4 + i (lanes
// 32-63): every k of the group exactly once. A comes from one offset register
// plus 32 bytes per group (the instruction's immediate) and B from one offset
// register plus a row step in the scalar offset. Batches of 2 groups, two
// sets in flight, measured best (512^3: 6.2 us; 4 groups 6.8, 8 7.7, three
// sets 6.7).
__device__ __forceinline__ bool ks_interior_ok(int bd, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                                               int64_t ldc, const float *A) {
  constexpr int64_t kLim = int64_t(1) << 29;
  static_assert(KH_GEMM_KSPLIT_INTERIOR_K == 64 * kKsFastBatch, "the launcher's K multiple for this path");
  return bd == KH_GEMM_KSPLIT_THREADS && M > 0 && N > 0 && (M & 31) == 0 && (N & 31) == 0 && K > 0 &&
         K % KH_GEMM_KSPLIT_INTERIOR_K == 0 && (lda & 3) == 0 && kh::aligned16(A) && M <= kLim && N <= kLim &&
         31 * lda + K / 8 < kLim && K * ldb < kLim && ldc < kLim && (M >> 5) * (N >> 5) < (int64_t(1) << 31);
}

__device__ __forceinline__ void ks_interior(const float *__restrict__ A, const float *__restrict__ B,
                                            float *__restrict__ C, int M, int N, int K, int lda, int ldb, int ldc,
                                            int nblocks, float *red) {
  constexpr int nw = kKsMaxWaves, NB = kKsFastBatch;
  const int lane = kh::lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kh::kWave);
  const int r = lane & 31, h = lane >> 5;
  const int tiles_n = N / kKsTile, total = (M / kKsTile) * tiles_n;
  const int kc = K / nw, kb = wave * kc, nbat = kc / (8 * NB);
  const uint32_t va = (uint32_t)(4 * (r * lda + 4 * h)), vb = (uint32_t)(4 * (4 * h * ldb + r));
  const uint32_t bstep = (uint32_t)(4 * ldb);
  const uint32_t abytes = (uint32_t)(4 * (31 * lda + kc)), bbytes = (uint32_t)(4 * ((kc - 1) * ldb + kKsTile));
  struct Set {
    float4 a[NB];
    float b[NB][4];
  };
  for (int t = blockIdx.x; t < total; t += nblocks) {
    const int m0 = __builtin_amdgcn_readfirstlane((t / tiles_n) * kKsTile);
    const int n0 = __builtin_amdgcn_readfirstlane((t % tiles_n) * kKsTile);
    const __amdgpu_buffer_rsrc_t ra = kh::span_rsrc(uniform_ptr(A + (int64_t)m0 * lda + kb), abytes);
    const __amdgpu_buffer_rsrc_t rb = kh::span_rsrc(uniform_ptr(B + (int64_t)kb * ldb + n0), bbytes);
    v16f acc = {};
    Set s0, s1;
    auto load = [&](Set &s, int j) {
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const int g = j * NB + i;
        const u32x4_t u = __builtin_amdgcn_raw_buffer_load_b128(ra, va, (uint32_t)(32 * g), 0);
        s.a[i] = make_float4(__uint_as_float(u.x), __uint_as_float(u.y), __uint_as_float(u.z), __uint_as_float(u.w));
#pragma unroll
        for (int q = 0; q < 4; ++q)
          s.b[i][q] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rb, vb, (uint32_t)(8 * g + q) * bstep, 0));
      }
    };
    auto math = [&](const Set &s) {
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(s.a[i].x, s.b[i][0], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(s.a[i].y, s.b[i][1], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(s.a[i].z, s.b[i][2], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(s.a[i].w, s.b[i][3], acc, 0, 0, 0);
      }
    };
    // Two sets in flight: batch j + 1's loads go out before batch j's MFMAs.
    load(s0, 0);
    for (int j = 0; j < nbat; j += 2) {
      if (j + 1 < nbat) load(s1, j + 1);
      math(s0);
      if (j + 2 < nbat) load(s0, j + 2);
      if (j + 1 < nbat) math(s1);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) red[(wave * 16 + i) * kh::kWave + lane] = acc[i];
    kh::lds_barrier();
#pragma unroll
    for (int i = wave; i < 16; i += nw) {
      float s = red[i * kh::kWave + lane];
#pragma unroll
      for (int w = 1; w < nw; ++w) s += red[(16 * w + i) * kh::kWave + lane];
      C[(int64_t)(m0 + 8 * (i >> 2) + 4 * h + (i & 3)) * ldc + n0 + r] = s;
    }
    kh::lds_barrier();
  }
}

// The general form: tiles of TM x TN blocks of v_mfma_f32_16x16x4f32. In a
// batch of 16 k, lane (r = l % 16, g = l / 16) loads the float4
// A[16 i + r][k + 4g ..] of each row block and the four B[k + 4g + s][16 j + r]
// of each column block; MFMA step s sums k + 4g + s over the lane groups.
// NB batches per set of registers, two sets.
template <int TM, int TN, int NB>
struct KsSet {
  float4 a[NB][TM];
  float b[NB][TN][4];
};

__device__ __forceinline__ bool ks_any_ok(int nw, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                                          int64_t ldc) {
  constexpr int64_t kLim = int64_t(1) << 29;  // floats of a 2^31-byte span
  return nw > 0 && M > 0 && N > 0 && K > 0 && lda >= K && ldb >= N && M <= kLim && N <= kLim &&
         64 * lda < kLim && (K / nw + 64) * ldb < kLim && ldc < kLim && ((M + 15) >> 4) * ((N + 15) >> 4) < kLim;
}

template <int TM, int TN, int NB>
__device__ __forceinline__ void ks_any(const float *__restrict__ A, const float *__restrict__ B,
                                       float *__restrict__ C, int M, int N, int K, int64_t lda, int64_t ldb,
                                       int64_t ldc, int nw, int nblocks, float *red) {
  using Set = KsSet<TM, TN, NB>;
  constexpr int R = 4 * TM * TN;  // accumulator registers
  const int lane = kh::lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kh::kWave);
  const int r = lane & 15, g = lane >> 4;
  const int tiles_n = (N + 16 * TN - 1) / (16 * TN), total = ((M + 16 * TM - 1) / (16 * TM)) * tiles_n;
  // The wave's K range: whole batches but for the last wave's.
  const int kc = 16 * ((K + 16 * nw - 1) / (16 * nw)), kb = wave * kc, kn = kc < K - kb ? kc : K - kb;
  uint32_t va[TM], vb[4];
#pragma unroll
  for (int i = 0; i < TM; ++i) va[i] = (uint32_t)(((16 * i + r) * lda + 4 * g) * 4);
#pragma unroll
  for (int s = 0; s < 4; ++s) vb[s] = (uint32_t)(((4 * g + s) * ldb + r) * 4);
  for (int pid = blockIdx.x; pid < total; pid += nblocks) {
    // One tile per workgroup: neighbouring tiles on one XCD (workgroups go to
    // the 8 XCDs round-robin), so that their rows of A and the two halves of
    // a line of B meet in one L2.
    int t = pid;
    if (nblocks == total) {
      const int x = pid & 7, per = total >> 3, extra = total & 7;
      t = x * per + (x < extra ? x : extra) + (pid >> 3);
    }
    const int m0 = __builtin_amdgcn_readfirstlane(t / tiles_n) * 16 * TM;
    const int n0 = __builtin_amdgcn_readfirstlane(t % tiles_n) * 16 * TN;
    const int rows = M - m0 < 16 * TM ? M - m0 : 16 * TM;
    v4f acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = v4f{};
    if (kn > 0 && wave < nw) {
      const __amdgpu_buffer_rsrc_t ra =
          kh::span_rsrc(uniform_ptr(A + m0 * lda + kb), (uint32_t)(((rows - 1) * lda + K - kb) * 4));
      const __amdgpu_buffer_rsrc_t rb =
          kh::span_rsrc(uniform_ptr(B + kb * ldb + n0), (uint32_t)(((kn - 1) * ldb + N - n0) * 4));
      auto load = [&](Set &f, int k0) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < NB; ++u) {
          // In the vector offset: the range check does not cover the scalar one.
          const uint32_t ao = (uint32_t)(k0 + 16 * u) * 4u, bo = (uint32_t)((k0 + 16 * u) * ldb) * 4u;
#pragma unroll
          for (int i = 0; i < TM; ++i) f.a[u][i] = kh::buf_load4(ra, va[i] + ao);
#pragma unroll
          for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int j = 0; j < TN; ++j)
              f.b[u][j][s] =
                  __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rb, vb[s] + bo + 64u * j, 0, 0));
        }
      };
      auto math = [&](Set &f, int k0) __attribute__((always_inline)) {
        if (k0 + 16 * NB > kn) {
#pragma unroll
          for (int u = 0; u < NB; ++u) {
            const int left = kn - k0 - 16 * u - 4 * g;
#pragma unroll
            for (int i = 0; i < TM; ++i)
              f.a[u][i] = make_float4(left > 0 ? f.a[u][i].x : 0.0f, left > 1 ? f.a[u][i].y : 0.0f,
                                      left > 2 ? f.a[u][i].z : 0.0f, left > 3 ? f.a[u][i].w : 0.0f);
          }
        }
#pragma unroll
        for (int u = 0; u < NB; ++u)
#pragma unroll
          for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < TM; ++i) {
              const float4 a = f.a[u][i];
              const float av = s == 0 ? a.x : s == 1 ? a.y : s == 2 ? a.z : a.w;
#pragma unroll
              for (int j = 0; j < TN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, f.b[u][j][s], acc[i][j], 0, 0, 0);
            }
      };
      Set s0, s1;
      load(s0, 0);
      for (int k = 0; k < kn; k += 32 * NB) {
        if (k + 16 * NB < kn) load(s1, k + 16 * NB);
        math(s0, k);
        if (k + 32 * NB < kn) load(s0, k + 32 * NB);
        if (k + 16 * NB < kn) math(s1, k + 16 * NB);
      }
    }
    // Partial tiles into LDS: red[wave][register][lane].
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) red[(wave * R + (i * TN + j) * 4 + q) * kh::kWave + lane] = acc[i][j][q];
    kh::lds_barrier();
    if (wave < nw) {
      for (int x = wave; x < R; x += nw) {
        float s = red[x * kh::kWave + lane];
        for (int w = 1; w < nw; ++w) s += red[(R * w + x) * kh::kWave + lane];
        const int gr = m0 + 16 * (x / (4 * TN)) + 4 * g + (x & 3), gc = n0 + 16 * ((x >> 2) % TN) + r;
        if (gr < M && gc < N) C[gr * ldc + gc] = s;
      }
    }
    kh::lds_barrier();
  }
}

// The same with 64-bit addresses, at any strides and spans: launches ks_any_ok
// turns down (K from 2^23, a wave's share of B past 2^31 bytes, rows that
// overlap), in `gemm_ksplit_16x16` alone, where the launcher sends such products.
// In the other symbols it costs their general form 4-6% (32x64 at 1271x218x3364 34.5
// -> 36.4 us, `gemm_ksplit_deep` at 2000x128x8190 49.3 -> 51.2, 32x16 at 200x400x5000
// 24.5 -> 25.5, its scalars spilling), there nothing (16x4096x4096 17.2). Rows past
// M and columns past N load the last one's, which is in range, and are not
// stored; k past the wave's range only occur in its last partial batch, where
// the loads are clamped and both operands zeroed. So the loop has no conditional
// load, and what bounds it is, as there, two batches in flight per wave:
// 1x1x(2^23 + 64) 21 ms, 4x64x(2^23 + 1) 35, 20x1000x1000000 4.1. An element per
// thread, one load after another, took 519 ms for the first.
typedef float f4_any __attribute__((ext_vector_type(4), aligned(4)));

template <int TM, int TN>
__device__ __forceinline__ void ks_wide(const float *__restrict__ A, const float *__restrict__ B,
                                        float *__restrict__ C, int64_t M, int64_t N, int64_t K, int64_t lda,
                                        int64_t ldb, int64_t ldc, int nw, int64_t nblocks, float *red) {
  using Set = KsSet<TM, TN, 1>;
  constexpr int R = 4 * TM * TN;  // accumulator registers
  const int lane = kh::lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kh::kWave);
  const int r = lane & 15, g = lane >> 4;
  const int64_t tiles_n = (N + 16 * TN - 1) / (16 * TN), total = ((M + 16 * TM - 1) / (16 * TM)) * tiles_n;
  const int64_t kc = 16 * ((K + 16 * nw - 1) / (16 * nw)), kb = wave * kc, ke = kb + kc < K ? kb + kc : K;
  for (int64_t t = blockIdx.x; t < total; t += nblocks) {
    const int64_t m0 = (t / tiles_n) * 16 * TM, n0 = (t % tiles_n) * 16 * TN;
    v4f acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = v4f{};
    if (wave < nw && kb < ke) {
      const float *pa[TM], *pb[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) pa[i] = A + (m0 + 16 * i + r < M ? m0 + 16 * i + r : M - 1) * lda + 4 * g;
#pragma unroll
      for (int j = 0; j < TN; ++j) pb[j] = B + (n0 + 16 * j + r < N ? n0 + 16 * j + r : N - 1) + 4 * g * ldb;
      auto load = [&](Set &f, int64_t k0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const f4_any a = *reinterpret_cast<const f4_any *>(pa[i] + k0);
          f.a[0][i] = make_float4(a.x, a.y, a.z, a.w);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int j = 0; j < TN; ++j) f.b[0][j][s] = pb[j][(k0 + s) * ldb];
      };
      auto math = [&](const Set &f) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int i = 0; i < TM; ++i) {
            const float4 a = f.a[0][i];
            const float av = s == 0 ? a.x : s == 1 ? a.y : s == 2 ? a.z : a.w;
#pragma unroll
            for (int j = 0; j < TN; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, f.b[0][j][s], acc[i][j], 0, 0, 0);
          }
      };
      const int64_t whole = kb + (ke - kb) / 16 * 16;  // whole batches
      Set s0, s1;
      if (kb < whole) load(s0, kb);
      for (int64_t k = kb; k < whole; k += 32) {
        if (k + 16 < whole) load(s1, k + 16);
        math(s0);
        if (k + 32 < whole) load(s0, k + 32);
        if (k + 16 < whole) math(s1);
      }
      if (whole < ke) {
        const int64_t left = ke - whole - 4 * g;  // of this lane's four k
        float *const fa = reinterpret_cast<float *>(s0.a[0]);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int64_t k = s < left ? whole + s : ke - 1 - 4 * g;
#pragma unroll
          for (int i = 0; i < TM; ++i) fa[4 * i + s] = s < left ? pa[i][k] : 0.0f;
#pragma unroll
          for (int j = 0; j < TN; ++j) s0.b[0][j][s] = s < left ? pb[j][k * ldb] : 0.0f;
        }
        math(s0);
      }
    }
    // Partial tiles into LDS, summed in the order of the waves, as in ks_any.
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) red[(wave * R + (i * TN + j) * 4 + q) * kh::kWave + lane] = acc[i][j][q];
    kh::lds_barrier();
    if (wave < nw) {
      for (int x = wave; x < R; x += nw) {
        float s = red[x * kh::kWave + lane];
        for (int w = 1; w < nw; ++w) s += red[(R * w + x) * kh::kWave + lane];
        const int64_t gr = m0 + 16 * (x / (4 * TN)) + 4 * g + (x & 3), gc = n0 + 16 * ((x >> 2) % TN) + r;
        if (gr < M && gc < N) C[gr * ldc + gc] = s;
      }
    }
    kh::lds_barrier();
  }
}

// What is left, blocks of less than a wave among it: an element per thread.
// Summed in runs of 1024 k, so that a long K costs no precision.
__device__ __forceinline__ void ks_plain(const float *__restrict__ A, const float *__restrict__ B,
                                         float *__restrict__ C, int64_t M, int64_t N, int64_t K, int64_t lda,
                                         int64_t ldb, int64_t ldc, int64_t threads, int64_t nblocks) {
  for (int64_t e = (int64_t)blockIdx.x * threads + threadIdx.x; e < M * N; e += nblocks * threads) {
    const float *a = A + (e / N) * lda, *b = B + e % N;
    float total = 0.0f;
    for (int64_t k0 = 0; k0 < K; k0 += 1024) {
      float s = 0.0f;
      for (int64_t k = k0; k < K && k < k0 + 1024; ++k) s = fmaf(a[k], b[k * ldb], s);
      total += s;
    }
    C[(e / N) * ldc + e % N] = total;
  }
}

}  // namespace

// The arguments the K-split kernels use, loaded in one round (KH_ARGS_READY):
// at 512^3 the launch is ~6 us, and every serial round trip to
// kernel-argument memory before the first operand load is part of it.
#define KH_KSPLIT_ARGS()                                                                                       \
  const uint32_t gw = kh::group_size_word(), gz = kh::group_size_z_word(), nb = kh::grid_blocks_x();          \
  KH_ARGS_READY(A_base, A_off, A_n0, A_n1, A_s0, B_base, B_off, B_n1, B_s0, C_base, C_off, C_s0, gw, gz, nb)

#define KH_KSPLIT_ANY(TM, TN, NB, WIDE)                                                                        \
  const int nw = (int)kh::threads_x_of(gw) / kh::kWave; /* a partial last wave takes no k and no output */    \
  if (ks_any_ok(nw, A_n0, B_n1, A_n1, A_s0, B_s0, C_s0))                                                      \
    ks_any<TM, TN, NB>(KH_PTR(A), KH_PTR(B), KH_PTR(C), (int)A_n0, (int)B_n1, (int)A_n1, A_s0, B_s0, C_s0,    \
                       nw, (int)nb, red);                                                                     \
  else if (WIDE && nw > 0)                                                                                    \
    ks_wide<TM, TN>(KH_PTR(A), KH_PTR(B), KH_PTR(C), A_n0, B_n1, A_n1, A_s0, B_s0, C_s0, nw, nb, red);        \
  else                                                                                                        \
    ks_plain(KH_PTR(A), KH_PTR(B), KH_PTR(C), A_n0, B_n1, A_n1, A_s0, B_s0, C_s0, kh::threads_x_of(gw), nb)

// 32x32 tiles: the whole-tile form where it applies, else the general one.
#define KH_KSPLIT_32X32(NB)                                                                                    \
  __shared__ float red[kKsMaxWaves * 16 * 64];                                                                 \
  KH_KSPLIT_ARGS();                                                                                            \
  if (kh::threads_y_of(gw) == 1 && kh::threads_z_of(gz) == 1 &&                                               \
      ks_interior_ok((int)kh::threads_x_of(gw), A_n0, B_n1, A_n1, A_s0, B_s0, C_s0, KH_PTR(A))) {             \
    ks_interior(KH_PTR(A), KH_PTR(B), KH_PTR(C), (int)A_n0, (int)B_n1, (int)A_n1, (int)A_s0, (int)B_s0,       \
                (int)C_s0, (int)nb, red);                                                                    \
    return;                                                                                                   \
  }                                                                                                           \
  KH_KSPLIT_ANY(2, 2, NB, false)

extern "C" __global__ void __launch_bounds__(KH_GEMM_KSPLIT_THREADS)
gemm_ksplit(KH_MEMREF2(const float, A), KH_MEMREF2(const float, B), KH_MEMREF2(float, C)) {
  KH_KSPLIT_32X32(1);
}

// The same with twice the loads in flight in the general form, for long K over
// operands the L2s do not hold (the rule and what it rests on:
// KH_GEMM_KSPLIT_DEEP_FLOATS).
extern "C" __global__ void __launch_bounds__(KH_GEMM_KSPLIT_THREADS)
gemm_ksplit_deep(KH_MEMREF2(const float, A), KH_MEMREF2(const float, B), KH_MEMREF2(float, C)) {
  KH_KSPLIT_32X32(2);
}

// Smaller tiles, for fewer rows or columns, and one larger.
extern "C" __global__ void __launch_bounds__(KH_GEMM_KSPLIT_THREADS)
gemm_ksplit_16x16(KH_MEMREF2(const float, A), KH_MEMREF2(const float, B), KH_MEMREF2(float, C)) {
  __shared__ float red[kKsMaxWaves * 4 * 64];
  KH_KSPLIT_ARGS();
  KH_KSPLIT_ANY(1, 1, 2, true);
}

extern "C" __global__ void __launch_bounds__(KH_GEMM_KSPLIT_THREADS)
gemm_ksplit_32x16(KH_MEMREF2(const float, A), KH_MEMREF2(const float, B), KH_MEMREF2(float, C)) {
  __shared__ float red[kKsMaxWaves * 8 * 64];
  KH_KSPLIT_ARGS();
  KH_KSPLIT_ANY(2, 1, 2, false);
}

extern "C" __global__ void __launch_bounds__(KH_GEMM_KSPLIT_THREADS)
gemm_ksplit_32x64(KH_MEMREF2(const float, A), KH_MEMREF2(const float, B), KH_MEMREF2(float, C)) {
  __shared__ float red[kKsMaxWaves * 32 * 64];
  KH_KSPLIT_ARGS();
  KH_KSPLIT_ANY(2, 4, 1, false);
}
