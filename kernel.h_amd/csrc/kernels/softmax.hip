// Row-wise safe softmax for gfx950: y[r,:] = exp(x[r,:] - max) / sum.
//
// Symbol and memref arguments follow the reference template
// (lib/dsl/kernels/softmax.cpp:68-165): x, y rank-2 [rows, cols], 14
// parameters. The reference runs an online max/sum recurrence serially in
// every thread of a row's block (softmax.cpp:121-145), reading the row 256
// times. Here the row is read once with dwordx4 loads into registers,
// reduced (max, then the sum of exponentials) and written once: 8 B of HBM
// traffic per element. What holds a row depends on its width:
//
//   cols <= 256            16 lanes, four rows per wavefront (rows16)
//   cols <= 2048           one wavefront (row_regs; softmax_wave up to 512 and,
//                          with few rows, from 65; the wide symbol past 1024)
//   cols <= 65536          one workgroup (row_block)
//   beyond                 one workgroup in two sweeps (row_stream)
//
// No path asks anything of the row's alignment: a dwordx4 buffer access
// needs 4-byte alignment only and is range-checked dword by dword, so an odd
// width or stride costs a little of the memory system's efficiency and no
// instructions. Rows are grid-strided; blocks that are not whole wavefronts
// give each thread whole rows instead, so every launch is correct, including
// the reference's rows x min(cols, 256) geometry (kernelh_backend.cpp:
// 256-257) at any cols.
//
// exp(x - m) is evaluated as 2^(x*log2e - m*log2e) with one fma on
// v_exp_f32; y = e * (1/s) with an IEEE reciprocal of s.
#include "kh_device.h"
#include "kh_tiles.h"

namespace {

// A lane's first column, 4 i. Opaque, so that the tail comparisons made from
// it stay inside the row loop: hoisted out of it, V x 4 lane masks took more
// scalar registers than there are.
__device__ __forceinline__ int first_col(int i) {
  int c = 4 * i;
  asm volatile("" : "+v"(c));
  return c;
}

// Columns past the end, which a buffer load fills with 0 (or, where four rows
// share a resource, with the next row), replaced by -inf: component k of the
// float4 that starts at column c.
__device__ __forceinline__ float4 mask_tail(float4 v, int c, int cols) {
  const float ninf = -__builtin_inff();
  return make_float4(c < cols ? v.x : ninf, c + 1 < cols ? v.y : ninf, c + 2 < cols ? v.z : ninf,
                     c + 3 < cols ? v.w : ninf);
}

__device__ __forceinline__ float max4(float4 v) { return fmaxf(fmaxf(v.x, v.y), fmaxf(v.z, v.w)); }

// The fma's exponents all carry the rounding of m * log2e, at most
// 2^-25 |m| log2e: a common factor that cancels in the quotient while it is
// small, but overflows for rows of large values (a row masked throughout
// with the type's lowest value). From |m| = 2^16 (a factor of 1.002) on, and
// for infinities, the subtraction is done first. One branch per wave, rarely
// taken.
template <int V>
__device__ __forceinline__ void shift_extreme(float4 (&v)[V], float &m) {
  const bool far = !(fabsf(m) < 65536.0f);
  if (__builtin_expect(__ballot(far) != 0, 0)) {
    const float d = far ? m : 0.0f;
#pragma unroll
    for (int j = 0; j < V; ++j) v[j] = make_float4(v[j].x - d, v[j].y - d, v[j].z - d, v[j].w - d);
    m -= d;
    if (far) m = 0.0f;  // inf - inf
  }
}

// v := exp(v - m); returns the lane's sum.
template <int V>
__device__ __forceinline__ float exp_sum(float4 (&v)[V], float m) {
  shift_extreme<V>(v, m);
  const float mb = -m * kh::kLog2e;
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < V; ++j) {
    v[j].x = kh::exp2_hw(fmaf(v[j].x, kh::kLog2e, mb));
    v[j].y = kh::exp2_hw(fmaf(v[j].y, kh::kLog2e, mb));
    v[j].z = kh::exp2_hw(fmaf(v[j].z, kh::kLog2e, mb));
    v[j].w = kh::exp2_hw(fmaf(v[j].w, kh::kLog2e, mb));
    s += (v[j].x + v[j].y) + (v[j].z + v[j].w);
  }
  return s;
}

__device__ __forceinline__ float4 scale4(float4 v, float f) {
  return make_float4(v.x * f, v.y * f, v.z * f, v.w * f);
}

// Four rows r0..r0+3 per wavefront, 16 lanes each (V float4 per lane, cols <=
// 64 V): the reductions stay inside a 16-lane DPP row, and a wave's load
// instruction covers four rows' worth of memory instead of a quarter of one.
// One resource spans the rows that exist; a lane's float4 past cols would
// store over the next row, so its offset is moved outside the resource, and
// the one float4 that straddles cols goes out as dwords. Against a wave per
// row (a wave of 1 KiB of lanes for a 256-byte row): 32768x64 9.1 -> 5.0 us;
// at 256 columns (32768 rows, 12.5 us, 5.4 TB/s) the two are level.
//
// A row's 256-byte pieces are whole cache lines only where its start and stride
// are. Where they are not, each store leaves parts of lines that the next one
// completes, so from three pieces a row on those go through the cache (PARTS);
// streamed past it they cost the memory system twice: 16384x200 7.3 -> 6.8 us,
// 300000x200 91 -> 86, 300000x255 147 -> 121 (whole lines through it cost 2-5%,
// 300000x160 64 -> 67, and rows of two pieces 4%, 300000x100 43.6 -> 45.2).
template <int V, bool PARTS = false>
__device__ __forceinline__ void softmax_rows16(const float *__restrict__ X, float *__restrict__ Y, int64_t r0,
                                               int64_t rows, int cols, int64_t xs, int64_t ys, int lane) {
  const int nr = rows - r0 < 4 ? (int)(rows - r0) : 4;
  const __amdgpu_buffer_rsrc_t rx = kh::span_rsrc(X + r0 * xs, (uint32_t)((nr - 1) * xs + cols) * 4u);
  const __amdgpu_buffer_rsrc_t ry = kh::span_rsrc(Y + r0 * ys, (uint32_t)((nr - 1) * ys + cols) * 4u);
  const int g = lane >> 4, c = lane & 15;
  const uint32_t xo = (uint32_t)(g * xs) * 4u, yo = (uint32_t)(g * ys) * 4u;
  float4 v[V];
#pragma unroll
  for (int j = 0; j < V; ++j) v[j] = kh::buf_load4_nt(rx, xo + (uint32_t)(c + 16 * j) * 16u);
  float m = -__builtin_inff();
  const int col0 = first_col(c);
#pragma unroll
  for (int j = 0; j < V; ++j) {
    v[j] = mask_tail(v[j], col0 + 64 * j, cols);
    m = fmaxf(m, max4(v[j]));
  }
  m = kh::row16_max(m);
  const float inv = 1.0f / kh::row16_sum(exp_sum<V>(v, m));
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const int col = col0 + 64 * j;
    const uint32_t off = yo + (uint32_t)col * 4u;
    v[j] = scale4(v[j], inv);
    if constexpr (PARTS)
      kh::buf_store4(ry, col + 3 < cols ? off : kh::kOutside, v[j]);
    else
      kh::buf_store4_nt(ry, col + 3 < cols ? off : kh::kOutside, v[j]);
    if ((cols & 3) != 0 && cols / 64 == j) {  // uniform: the float4s that hold the rows' last columns
      const bool last = col < cols && col + 3 >= cols;
      kh::buf_store1(ry, last ? off : kh::kOutside, v[j].x);
      kh::buf_store1(ry, last && col + 1 < cols ? off + 4u : kh::kOutside, v[j].y);
      kh::buf_store1(ry, last && col + 2 < cols ? off + 8u : kh::kOutside, v[j].z);
    }
  }
}

// One row per wavefront. The row moves through buffer resources spanning
// exactly its cols floats: columns past the end read 0 (replaced by -inf
// before the max) and their stores are dropped, so the path has no per-lane
// branches. With SPLIT (a wave's first row in a launch that fits one round,
// four or more float4 per lane) the loads go out in two halves, the second
// once the first has landed, and nothing else is issued until all have
// (kh::kFirstBurst).
template <int V, bool SPLIT = false>
__device__ __forceinline__ void softmax_row_regs(const float *__restrict__ xr, float *__restrict__ yr, int cols,
                                                 int lane) {
  const __amdgpu_buffer_rsrc_t rx = kh::span_rsrc(xr, (uint32_t)cols * 4u);
  const __amdgpu_buffer_rsrc_t ry = kh::span_rsrc(yr, (uint32_t)cols * 4u);
  constexpr int kHalf = V >= 4 ? V / 2 : V;
  float4 v[V];
#pragma unroll
  for (int j = 0; j < V; ++j) {
    v[j] = kh::buf_load4_nt(rx, (uint32_t)(lane + j * kh::kWave) * 16u);
    if (SPLIT && j + 1 == kHalf && kHalf < V) kh::vm_wait<0>();
  }
  if (SPLIT) kh::vm_wait<0>();
  float m = -__builtin_inff();
  const int col0 = first_col(lane);
#pragma unroll
  for (int j = 0; j < V; ++j) {
    v[j] = mask_tail(v[j], col0 + 4 * kh::kWave * j, cols);
    m = fmaxf(m, max4(v[j]));
  }
  m = kh::wave_max(m);
  const float inv = 1.0f / kh::wave_sum(exp_sum<V>(v, m));
#pragma unroll
  for (int j = 0; j < V; ++j) kh::buf_store4_nt(ry, (uint32_t)(lane + j * kh::kWave) * 16u, scale4(v[j], inv));
}

// One row per workgroup of nt threads, V float4 per thread (cols <= 4 V nt).
// The max and the sum each cross the waves through LDS; the maximum is the
// whole row's before any exponential, so that every element's exponent
// carries the same rounding of m * log2e and it cancels in the quotient. As
// many threads as hold the row (more were slower: 512x12000 7.8 us at 384-768
// threads, 10.5 at 1024): one read and one write per element with every load
// of the row in flight, and where the workgroup is small enough a second one
// on the CU to fill its reductions. The
// wave per row that took such rows a float at a time, twice, was bound by
// that one wave's load latency: 256x32001 301.6 -> 14.1 us (4.6 TB/s),
// 2048x6000 66.3 -> 18.9, 16x65536 285 -> 9.5.
template <int V>
__device__ __forceinline__ void softmax_row_block(const float *__restrict__ xr, float *__restrict__ yr, int cols,
                                                  int nt, int lane, int wave, float (&red)[2][kh::kMaxWaves]) {
  const __amdgpu_buffer_rsrc_t rx = kh::span_rsrc(xr, (uint32_t)cols * 4u);
  const __amdgpu_buffer_rsrc_t ry = kh::span_rsrc(yr, (uint32_t)cols * 4u);
  const int tid = threadIdx.x;
  float4 v[V];
#pragma unroll
  for (int j = 0; j < V; ++j) v[j] = kh::buf_load4_nt(rx, (uint32_t)(tid + j * nt) * 16u);
  float m = -__builtin_inff();
  const int col0 = first_col(tid);
#pragma unroll
  for (int j = 0; j < V; ++j) {
    v[j] = mask_tail(v[j], col0 + 4 * nt * j, cols);
    m = fmaxf(m, max4(v[j]));
  }
  m = kh::block_max(m, red[0], nt / kh::kWave, lane, wave);
  const float inv = 1.0f / kh::block_sum(exp_sum<V>(v, m), red[1], nt / kh::kWave, lane, wave);
#pragma unroll
  for (int j = 0; j < V; ++j) kh::buf_store4_nt(ry, (uint32_t)(tid + j * nt) * 16u, scale4(v[j], inv));
}

// Rows past the registers of a workgroup: an online (max, sum) per thread
// over chunks of kStreamV float4, merged across the workgroup, then a second
// sweep that re-reads the row and writes it.
constexpr int kStreamV = 4;
__device__ __forceinline__ void softmax_row_stream(const float *__restrict__ xr, float *__restrict__ yr,
                                                   int64_t cols, int nt, int lane, int wave,
                                                   float (&red)[2][kh::kMaxWaves]) {
  const int tid = threadIdx.x, chunk = 4 * kStreamV * nt;
  const float ninf = -__builtin_inff();
  float m = ninf, s = 0.0f;
  for (int64_t c0 = 0; c0 < cols; c0 += chunk) {
    const int n = cols - c0 < chunk ? (int)(cols - c0) : chunk;
    const __amdgpu_buffer_rsrc_t rx = kh::span_rsrc(xr + c0, (uint32_t)n * 4u);
    float4 v[kStreamV];
#pragma unroll
    for (int j = 0; j < kStreamV; ++j) v[j] = kh::buf_load4(rx, (uint32_t)(tid + j * nt) * 16u);
    float mn = m;
    const int col0 = first_col(tid);
#pragma unroll
    for (int j = 0; j < kStreamV; ++j) {
      v[j] = mask_tail(v[j], col0 + 4 * nt * j, n);
      mn = fmaxf(mn, max4(v[j]));
    }
    const float ref = mn == ninf ? 0.0f : mn;  // nothing but -inf so far: every term is 0
    float t = 0.0f;
#pragma unroll
    for (int j = 0; j < kStreamV; ++j)
      t += (kh::exp2_hw((v[j].x - ref) * kh::kLog2e) + kh::exp2_hw((v[j].y - ref) * kh::kLog2e)) +
           (kh::exp2_hw((v[j].z - ref) * kh::kLog2e) + kh::exp2_hw((v[j].w - ref) * kh::kLog2e));
    s = s * kh::exp2_hw((m - ref) * kh::kLog2e) + t;
    m = mn;
  }
  const float gm = kh::block_max(m, red[0], nt / kh::kWave, lane, wave);
  // Threads that saw no finite element carry m = -inf, s = 0: contribute 0.
  s = s == 0.0f ? 0.0f : s * kh::exp2_hw((m - gm) * kh::kLog2e);
  const float inv = 1.0f / kh::block_sum(s, red[1], nt / kh::kWave, lane, wave);
  for (int64_t c0 = 0; c0 < cols; c0 += chunk) {
    const int n = cols - c0 < chunk ? (int)(cols - c0) : chunk;
    const __amdgpu_buffer_rsrc_t rx = kh::span_rsrc(xr + c0, (uint32_t)n * 4u);
    const __amdgpu_buffer_rsrc_t ry = kh::span_rsrc(yr + c0, (uint32_t)n * 4u);
    float4 v[kStreamV];
#pragma unroll
    for (int j = 0; j < kStreamV; ++j) v[j] = kh::buf_load4(rx, (uint32_t)(tid + j * nt) * 16u);
#pragma unroll
    for (int j = 0; j < kStreamV; ++j)
      kh::buf_store4_nt(ry, (uint32_t)(tid + j * nt) * 16u,
                        make_float4(kh::exp2_hw((v[j].x - gm) * kh::kLog2e) * inv,
                                    kh::exp2_hw((v[j].y - gm) * kh::kLog2e) * inv,
                                    kh::exp2_hw((v[j].z - gm) * kh::kLog2e) * inv,
                                    kh::exp2_hw((v[j].w - gm) * kh::kLog2e) * inv));
  }
}

// Blocks that are not whole wavefronts (the reference's rows x
// min(cols, 256) geometry, kernelh_backend.cpp:256-257, when cols < 256 is
// not a multiple of 64): the wave reductions need 64 active lanes, so each
// thread takes whole rows, serially.
__device__ __forceinline__ void softmax_row_serial(const float *__restrict__ xr, float *__restrict__ yr,
                                                   int64_t cols) {
  float m = -__builtin_inff();
  for (int64_t c = 0; c < cols; ++c) m = fmaxf(m, xr[c]);
  // The maximum is subtracted first, so that rows of any size do (shift_extreme).
  float s = 0.0f;
  for (int64_t c = 0; c < cols; ++c) s += kh::exp2_hw((xr[c] - m) * kh::kLog2e);
  const float inv = 1.0f / s;
  for (int64_t c = 0; c < cols; ++c) yr[c] = kh::exp2_hw((xr[c] - m) * kh::kLog2e) * inv;
}

// Any width in one wavefront, for launches of softmax_wave past what its
// registers hold: an online (max, sum) per lane, merged, then a second sweep.
__device__ __forceinline__ void softmax_row_wave(const float *__restrict__ xr, float *__restrict__ yr, int64_t cols,
                                                 int lane) {
  const float ninf = -__builtin_inff();
  float m = ninf, s = 0.0f;
  for (int64_t c = lane; c < cols; c += kh::kWave) {
    const float x = xr[c], mn = fmaxf(m, x);
    const float ref = mn == ninf ? 0.0f : mn;  // nothing but -inf so far: every term is 0
    s = s * kh::exp2_hw((m - ref) * kh::kLog2e) + kh::exp2_hw((x - ref) * kh::kLog2e);
    m = mn;
  }
  const float gm = kh::wave_max(m);
  s = s == 0.0f ? 0.0f : s * kh::exp2_hw((m - gm) * kh::kLog2e);
  const float inv = 1.0f / kh::wave_sum(s);
  for (int64_t c = lane; c < cols; c += kh::kWave) yr[c] = kh::exp2_hw((xr[c] - gm) * kh::kLog2e) * inv;
}

// Which register paths a symbol compiles in: the kernel's register
// allocation is that of its widest path, so the narrow symbol stays lean
// (more rows in flight per CU).
enum Symbol { kNarrow, kWide, kBlock };

template <Symbol S>
__device__ __forceinline__ void softmax_rows(const float *__restrict__ X, float *__restrict__ Y, int64_t rows,
                                             int64_t cols, int64_t xs, int64_t ys, int bd, int64_t nb,
                                             float (&red)[2][kh::kMaxWaves]) {
  if (bd % kh::kWave != 0) {
    for (int64_t r = (int64_t)blockIdx.x * bd + threadIdx.x; r < rows; r += bd * nb)
      softmax_row_serial(X + r * xs, Y + r * ys, cols);
    return;
  }
  const int lane = kh::lane_id();
  const int waves_per_block = bd / kh::kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kh::kWave);  // uniform: scalar row loop
  const int64_t nwaves = waves_per_block * nb;
  const int64_t w0 = (int64_t)blockIdx.x * waves_per_block + wave;
  const int c = (int)(cols <= KH_ROW_BLOCK_MAX ? cols : KH_ROW_BLOCK_MAX + 1);
  if (S == kNarrow && c <= KH_ROW16_COLS && xs >= cols && ys >= cols && (xs | ys) < (1 << 26)) {
    // One loop per width: with the choice inside one loop a group of rows of up to
    // 64 floats, over in a microsecond, took 4-6% longer (185147x9 15.6 vs 14.2 us).
    const auto each = [&](auto go) __attribute__((always_inline)) {
      for (int64_t r = 4 * w0; r < rows; r += 4 * nwaves) go(r);
    };
    if (c <= 64)
      each([&](int64_t r) __attribute__((always_inline)) { softmax_rows16<1>(X, Y, r, rows, c, xs, ys, lane); });
    else if (c <= 128)
      each([&](int64_t r) __attribute__((always_inline)) { softmax_rows16<2>(X, Y, r, rows, c, xs, ys, lane); });
    else if (rows > KH_ROW16_CACHED_ROWS && kh::shares_lines(Y, ys))
      each([&](int64_t r) __attribute__((always_inline)) { softmax_rows16<4, true>(X, Y, r, rows, c, xs, ys, lane); });
    else
      each([&](int64_t r) __attribute__((always_inline)) { softmax_rows16<4>(X, Y, r, rows, c, xs, ys, lane); });
    return;
  }
  if (S != kBlock && c <= (S == kWide ? 2048 : 1024)) {
    bool split = kh::split_first_burst(bd * nb);  // each wave's first row only
    for (int64_t r = w0; r < rows; r += nwaves) {
      const float *xr = X + r * xs;
      float *yr = Y + r * ys;
      if (S == kNarrow && c <= 512)
        softmax_row_regs<2>(xr, yr, c, lane);
      else if (S == kNarrow)
        split ? softmax_row_regs<4, true>(xr, yr, c, lane) : softmax_row_regs<4>(xr, yr, c, lane);
      else
        split ? softmax_row_regs<8, true>(xr, yr, c, lane) : softmax_row_regs<8>(xr, yr, c, lane);
      split = false;
    }
    return;
  }
  for (int64_t r = blockIdx.x; r < rows; r += nb) {
    const float *xr = X + r * xs;
    float *yr = Y + r * ys;
    if (S != kBlock && c <= 16 * bd)
      softmax_row_block<4>(xr, yr, c, bd, lane, wave, red);
    else if (S == kNarrow && c <= 32 * bd)
      softmax_row_block<8>(xr, yr, c, bd, lane, wave, red);
    else if (S == kBlock && c <= 64 * bd)
      softmax_row_block<16>(xr, yr, c, bd, lane, wave, red);
    else
      softmax_row_stream(xr, yr, cols, bd, lane, wave, red);
  }
}

}  // namespace

#define KH_SOFTMAX_BODY(S)                                                                                    \
  __shared__ float red[2][kh::kMaxWaves];                                                                      \
  const uint32_t gw = kh::group_size_word(), nb = kh::grid_blocks_x();                                         \
  KH_ARGS_READY(x_base, x_off, x_n0, x_n1, x_s0, y_base, y_off, y_s0, gw, nb);                                 \
  softmax_rows<S>(KH_PTR(x), KH_PTR(y), x_n0, x_n1, x_s0, y_s0, (int)kh::threads_x_of(gw), nb, red)

// The reference symbol: rows up to 1024 floats in 16 lanes or a wave, wider
// ones in a workgroup.
extern "C" __global__ void __launch_bounds__(1024)
softmax(KH_MEMREF2(const float, x), KH_MEMREF2(float, y)) {
  KH_SOFTMAX_BODY(kNarrow);
}

// Same arguments and results for rows of 257..512 floats, and for others up to
// 1023 where row_plan says (khrt_templates.cpp): a wave per row and nothing else,
// without LDS. The path is `softmax`'s, instruction for
// instruction, but as one of that symbol's many it took 2-9% longer: 9300x272
// 6.25 -> 5.80 us, 40000x272 16.9 -> 15.8, 16384x300 9.0 -> 8.6, 16384x512 13.2 ->
// 12.8; at 700 and 1024 columns it is 1% slower (40000x1024 53.6 -> 54.3) but where
// a launch just about fills the chip once (8192x640 10.0 -> 8.9).
extern "C" __global__ void __launch_bounds__(256)
softmax_wave(KH_MEMREF2(const float, x), KH_MEMREF2(float, y)) {
  const uint32_t gw = kh::group_size_word(), nb = kh::grid_blocks_x();
  KH_ARGS_READY(x_base, x_off, x_n0, x_n1, x_s0, y_base, y_off, y_s0, gw, nb);
  const float *__restrict__ X = KH_PTR(x);
  float *__restrict__ Y = KH_PTR(y);
  const int bd = (int)kh::threads_x_of(gw);
  const int64_t rows = x_n0, cols = x_n1, step = (int64_t)(bd / kh::kWave) * nb;
  if (bd % kh::kWave != 0) {
    for (int64_t r = (int64_t)blockIdx.x * bd + threadIdx.x; r < rows; r += (int64_t)bd * nb)
      softmax_row_serial(X + r * x_s0, Y + r * y_s0, cols);
    return;
  }
  const int lane = kh::lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kh::kWave);
  bool split = kh::split_first_burst((int64_t)bd * nb);  // each wave's first row only
  for (int64_t r = (int64_t)blockIdx.x * (bd / kh::kWave) + wave; r < rows; r += step) {
    if (cols <= 256)
      softmax_row_regs<1>(X + r * x_s0, Y + r * y_s0, (int)cols, lane);
    else if (cols <= 512)
      softmax_row_regs<2>(X + r * x_s0, Y + r * y_s0, (int)cols, lane);
    else if (cols <= 1024)
      split ? softmax_row_regs<4, true>(X + r * x_s0, Y + r * y_s0, (int)cols, lane)
            : softmax_row_regs<4>(X + r * x_s0, Y + r * y_s0, (int)cols, lane);
    else
      softmax_row_wave(X + r * x_s0, Y + r * y_s0, cols, lane);
    split = false;
  }
}

// Same arguments and results for rows of 1025..4096 floats (the launcher picks
// it there): a wave per row up to 2048, a workgroup of 192 or 256 threads
// past that. Where the line lies, events around rotated launches, wave
// against workgroup: 4096x1500 9.0 vs 10.4 us, 4096x2048 11.6 vs 12.6,
// 4096x3001 18.2 vs 19.0, 1024x3001 6.1 vs 5.3, 16384x4096 94.0 vs 86.6.
extern "C" __global__ void __launch_bounds__(256)
softmax_wide(KH_MEMREF2(const float, x), KH_MEMREF2(float, y)) {
  KH_SOFTMAX_BODY(kWide);
}

// Same arguments and results; one workgroup per row with 16 float4 per
// thread, for rows past what the reference symbol's eight hold, and of a single
// wave for 2049..4096 floats where row_plan says.
extern "C" __global__ void __launch_bounds__(1024)
softmax_block(KH_MEMREF2(const float, x), KH_MEMREF2(float, y)) {
  KH_SOFTMAX_BODY(kBlock);
}
