// Tile constants shared by the gfx950 kernels and the host launcher's
// geometry (khrt_templates.cpp). Plain macros: included by device and host
// translation units alike.
#pragma once

// Elementwise kernels (vecadd, fused_gelu): dwordx4 vectors per thread per
// grid-stride step.
#define KH_EW_UNROLL 4

// Row templates. Rows of at most KH_ROW16_COLS floats take 16 lanes each,
// four to a wave; a workgroup holds rows of up to KH_ROW_BLOCK_MAX floats in
// registers (1024 threads x 16 float4).
#define KH_ROW16_COLS 256
// Launches of no more rows than this give each a wave instead: there are too
// few to fill the chip four at a time, and a row in 16 lanes takes its two or
// four loads and their share of the reductions one after another. Four rows to a
// wave against one: softmax 1000x100 2.72 vs 2.62 us, 1000x252 3.0 vs 2.7, 2500x252
// 3.3 vs 3.2, 4096x252 3.6 vs 3.6, 4096x160 3.2 vs 3.4; layernorm 1000x100 2.94 vs 2.72,
// 2500x100 level, 6144x200 4.32 vs 3.76, 6144x160 3.78 vs 3.64. Between there and 8192
// rows it depends on the width (6500x252 4.61 vs 4.08, 8192x160 3.90 vs 4.00, 8192x224
// 4.16 vs 4.27). Rows of one float4 per lane (up to 64) are level.
#define KH_SOFTMAX_WAVE_ROWS(cols) ((cols) <= 64 ? 0 : (cols) <= 128 ? 1024 : 2048)
#define KH_LAYERNORM_WAVE_ROWS(cols) ((cols) <= 64 ? 0 : (cols) <= 128 ? 1024 : 6144)
// Launches of more rows than this send stores of parts of cache lines through
// the cache (softmax.hip); with fewer there is nothing to merge them with in
// time (softmax 4096x240 3.35 us streamed, 3.7 cached; 9300x240 5.3 and 5.0).
#define KH_ROW16_CACHED_ROWS 8192
#define KH_ROW_BLOCK_MAX 65536

// Scan: workgroup size chosen by the launcher (the kernel accepts 256..1024).
// One wave of each workgroup runs the look-back; every other thread owns
// KH_SCAN_PER_THREAD consecutive elements, so a tile is
// KH_SCAN_PER_THREAD x (threads - 64) elements.
#ifndef KH_SCAN_PER_THREAD
#define KH_SCAN_PER_THREAD 16
#endif
#define KH_SCAN_THREADS 1024
#define KH_SCAN_TILE (KH_SCAN_PER_THREAD * (KH_SCAN_THREADS - 64))
// The launcher's workgroup size up to KH_SCAN_SMALL_N elements: at
// n = 10^6, 89 tiles of 11,264 ran 8.35 us against 66 of 15,360 in
// 8.52 us; at 2 * 10^6 1024 threads were faster (10.1 against 10.6 us).
#define KH_SCAN_SMALL_THREADS 768
#define KH_SCAN_SMALL_N (3 << 19)

// GEMM block tiles (rows of C x columns of C per workgroup of 256 threads).
#define KH_GEMM_BM 128
#define KH_GEMM_BN 256
#define KH_GEMM_MID_BM 128
#define KH_GEMM_MID_BN 128
#define KH_GEMM_SMALL_BM 64
#define KH_GEMM_SMALL_BN 64
#define KH_GEMM_SMALL_BK 32
// `gemm_small` runs eight waves (512 threads), two workgroups per CU.
#define KH_GEMM_SMALL_THREADS 512
// `gemm_wide`: 128x128 tiles on eight waves (512 threads), one workgroup per
// CU, persistent.
#define KH_GEMM_WIDE_BM 128
#define KH_GEMM_WIDE_BN 128
#define KH_GEMM_WIDE_THREADS 512

// The launcher's tile choice (khrt_templates.cpp, heuristic_gemm_symbol):
// for each symbol, score = its measured rate at full occupancy (TFLOP/s,
// MI355X) x the fraction of the last round of workgroups that is busy, and
// take the best. `gemm` and `gemm_mid` run two workgroups per CU, so a round
// is 2 x KH_GEMM_CUS tiles and a half-empty last round costs a full one;
// `gemm_wide` runs one per CU (a round of KH_GEMM_CUS tiles); the 64x64
// tiles (`gemm_small`, persistent, two per CU) are light enough that a
// partial round costs little, so their rounds are counted per CU. Fitted on 20 shapes from 1024^3 to 8192^3 (square,
// skinny, rectangular, deep K) timed with rotated U[-1,1] inputs and warm
// clocks: the choice is the measured best or within 3% of it on all of them.
// `gemm_wide`'s rate was refitted when it became the persistent 128x128
// ring: 3.3% below `gemm` at 4096^3 (both in whole rounds), level with the
// 64x64 tiles at 2560^3. Its round divides `gemm_mid`'s and its rate is
// higher, so it outscores `gemm_mid` at every shape (measured 5-6% faster
// at 4096x2048x4096 and 8192x1024x8192).
#define KH_GEMM_CUS 256
#define KH_GEMM_ROUND_BIG (2 * KH_GEMM_CUS)
#define KH_GEMM_ROUND_MID (2 * KH_GEMM_CUS)
#define KH_GEMM_ROUND_WIDE KH_GEMM_CUS
#define KH_GEMM_ROUND_SMALL KH_GEMM_CUS
#define KH_GEMM_RATE_BIG 142
#define KH_GEMM_RATE_MID 135
#define KH_GEMM_RATE_WIDE 137
#define KH_GEMM_RATE_SMALL 126
// K split over the 8 waves of a 512-thread workgroup, in tiles of 16x16,
// 32x16, 32x32 (`gemm_ksplit`, `gemm_ksplit_deep`) and 32x64. The launcher
// takes the smallest of them with at most KH_GEMM_CUS tiles: more, smaller
// tiles leave each CU several workgroups that read the same operands again
// (100x777x555: 343 tiles of 16x16 6.8 us, 196 of 32x16 6.0), fewer, larger
// ones leave CUs idle (16x4096x4096: 17.6 us in 256 tiles, 23.9 in 128).
// 32x32 tiles are also taken beyond one round where the 64x64 tiles number
// fewer than the CUs and every 32x32 tile is whole with K a multiple of
// KH_GEMM_KSPLIT_INTERIOR_K (the whole-tile form), from
// KH_GEMM_KSPLIT_MIN_K on; the workgroups then loop over their tiles.
// Kernel trace, rotated inputs, against the 64x64 tiles `gemm_small` then
// had: 640^3 11.5 vs 18.0 us, 1024x512x512 10.2 vs 15.2, 256x2048x2048 25.5
// vs 50.3; level at 768x768x256 and 896^3; at 1024x1024x512 slower (17.3 vs
// 15.9). Against the persistent eight-wave `gemm_small`: 768^3 level (18.0
// vs 17.8), 512x512x2048 14.6 vs 40.4; 32x64 against it: 333x1000x2000 22.6
// vs 40.8, 513x511x509 8.6 vs 13.8.
#define KH_GEMM_KSPLIT_BM 32
#define KH_GEMM_KSPLIT_BN 32
#define KH_GEMM_KSPLIT_THREADS 512
#define KH_GEMM_KSPLIT_INTERIOR_K 128
#define KH_GEMM_KSPLIT_MIN_K 256
// `gemm_ksplit_deep` (twice the loads in flight in the form for tiles that are
// not all whole) is taken from this K on, for operands of at least so many
// floats: past what the L2s hold, where each load takes longer. Events around
// rotated launches, gemm_ksplit / gemm_ksplit_deep:
//   300x520x7001      5.7 M floats  46.2 / 49.7    500x500x8191   8.2 M  52.6 / 52.1
//   500x500x9999     10.0           63.4 / 64.2    500x500x12001 12.0    77.5 / 74.6
//   100x2000x9999    21.0           66.8 / 69.0    500x500x16001 16.0   103.8 / 98.5
//   1500x150x16001   26.4            124 / 109     8000x30x5001  40.2    54.8 / 48.3
// Where all are whole the two run the same code.
#define KH_GEMM_KSPLIT_DEEP_K 2048
#define KH_GEMM_KSPLIT_DEEP_FLOATS (1 << 24)

// Attention: query rows per workgroup (4 wavefronts x 32 rows).
#define KH_ATTN_BLOCK_Q 128
// attention_split and attention_split16: 32 and 16 query rows per workgroup,
// the keys split over its 4 waves.
#define KH_ATTN_SPLIT_THREADS 256
