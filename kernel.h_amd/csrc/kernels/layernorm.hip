// Layernorm over the last dim for gfx950, eps = 1e-5:
//   y = (x - mean) * rsqrt(var + eps) * gamma + beta.
//
// Symbol and memref arguments follow the reference template
// (lib/dsl/kernels/layernorm.cpp:58-153): x [rows, cols], gamma [cols],
// beta [cols], y [rows, cols], 24 parameters. Two-pass statistics as the
// template pins them (mean first, then the mean of squared deviations; no
// Welford), but the row is read from HBM once, into registers, and the second
// pass runs there. Traffic: 8 B per element + 8 B per column (every row
// shares gamma and beta, so HBM sees them once). What holds a row depends on
// its width:
//
//   cols <= 256            16 lanes, four rows per wavefront (rows16)
//   cols <= 2048           one wavefront (rows_regs; layernorm_wave from 65 to 256
//                          with few rows, the wide symbols past 1024), and many
//                          rows of 2689..4095 that share cache lines
//                          (layernorm_wide_parts)
//   cols <= 65536          one workgroup (row_block)
//   beyond                 one workgroup, three sweeps (row_stream)
//
// No path asks anything of alignment: a dwordx4 buffer access needs 4-byte
// alignment only and is range-checked dword by dword. Rows are grid-strided;
// any block is correct, including the reference's rows x 256 geometry
// (kernelh_backend.cpp:290).
#include <type_traits>

#include "kh_device.h"
#include "kh_tiles.h"

namespace {

constexpr float kEps = 1e-5f;

// Columns the narrow symbol stages gamma and beta for in LDS.
constexpr int kStageCols = 1024;

__device__ __forceinline__ float sum4(float4 v) { return (v.x + v.y) + (v.z + v.w); }

// A lane's first column, 4 i. Opaque, so that the tail comparisons made from
// it stay inside the row loop: hoisted out of it, V x 4 lane masks take more
// scalar registers than there are.
__device__ __forceinline__ int first_col(int i) {
  int c = 4 * i;
  asm volatile("" : "+v"(c));
  return c;
}

// v - mean, 0 past the row's end: component k of the float4 at column c.
__device__ __forceinline__ float4 deviation(float4 v, float mean, int c, int cols) {
  return make_float4(c < cols ? v.x - mean : 0.0f, c + 1 < cols ? v.y - mean : 0.0f, c + 2 < cols ? v.z - mean : 0.0f,
                     c + 3 < cols ? v.w - mean : 0.0f);
}

__device__ __forceinline__ float squares4(float4 d) { return (d.x * d.x + d.y * d.y) + (d.z * d.z + d.w * d.w); }

__device__ __forceinline__ float4 affine4(float4 d, float inv, float4 g, float4 b) {
  return make_float4(fmaf(d.x * inv, g.x, b.x), fmaf(d.y * inv, g.y, b.y), fmaf(d.z * inv, g.z, b.z),
                     fmaf(d.w * inv, g.w, b.w));
}

// gamma and beta are not held in registers: that doubled the register
// footprint and halved the number of rows in flight. The narrow symbol copies
// them into Gs/Bs (kStageCols floats each, 0 past cols) once per workgroup,
// after its waves have issued their first row's loads, and the output reads
// them from LDS; wider rows re-read them per row from L2. The LDS copy takes
// 4x fewer L2 requests for the same 64 lines, which every wave on the chip
// asks for at the same time. Measured at 4096x1024 it runs level with the L2
// re-read (7.4-7.8 us) in a quiet sequence, but held 7.4-7.7 us in the first
// launches after a run of long GEMMs, where the L2 re-read took 8.0-8.4 us.
// Every thread of the block reaches the barrier.
__device__ __forceinline__ void stage_affine(const float *__restrict__ G, const float *__restrict__ B, int cols,
                                             int bd, float *Gs, float *Bs) {
  const __amdgpu_buffer_rsrc_t rg = kh::span_rsrc(G, (uint32_t)cols * 4u), rb = kh::span_rsrc(B, (uint32_t)cols * 4u);
  for (int i = threadIdx.x; 4 * i < cols; i += bd) {
    reinterpret_cast<float4 *>(Gs)[i] = kh::buf_load4(rg, 16u * i);
    reinterpret_cast<float4 *>(Bs)[i] = kh::buf_load4(rb, 16u * i);
  }
  kh::lds_barrier();
}

// Four rows per wavefront, 16 lanes each (V float4 per lane, cols <= 64 V):
// the reductions stay inside a 16-lane DPP row, and a wave's load instruction
// covers four rows' worth of memory instead of a quarter of one. One resource
// spans the rows that exist; a lane's float4 past cols would store over the
// next row, so its offset is moved outside the resource, and the one float4
// that straddles cols goes out as dwords. Against a wave per row: 32768x64
// 10.3 -> 5.4 us. From three pieces a row on, stores whose 256-byte pieces are not
// whole cache lines go through the cache (PARTS), where the next completes them:
// 300000x200 93 -> 87 us, 300000x252 121 -> 106. r0, rstep: in rows.
template <int V, bool PARTS = false>
__device__ __forceinline__ void layernorm_rows16(const float *__restrict__ X, const float *__restrict__ G,
                                                 const float *__restrict__ B, float *__restrict__ Y, int64_t rows,
                                                 int cols, int64_t xs, int64_t ys, int64_t r0, int64_t rstep, int bd,
                                                 int lane, float *Gs, float *Bs) {
  const int g = lane >> 4, c = lane & 15;
  const uint32_t xo = (uint32_t)(g * xs) * 4u, yo = (uint32_t)(g * ys) * 4u;
  const float n = (float)cols;
  float4 v[V];
  auto load_rows = [&](int64_t r) __attribute__((always_inline)) {
    const int nr = rows - r < 4 ? (int)(rows - r) : 4;
    const __amdgpu_buffer_rsrc_t rx = kh::span_rsrc(X + r * xs, (uint32_t)((nr - 1) * xs + cols) * 4u);
#pragma unroll
    for (int j = 0; j < V; ++j) v[j] = kh::buf_load4_nt(rx, xo + (uint32_t)(c + 16 * j) * 16u);
  };
  if (r0 < rows) load_rows(r0);
  stage_affine(G, B, cols, bd, Gs, Bs);
  for (int64_t r = r0; r < rows; r += rstep) {
    if (r != r0) load_rows(r);
    const int nr = rows - r < 4 ? (int)(rows - r) : 4;
    const __amdgpu_buffer_rsrc_t ry = kh::span_rsrc(Y + r * ys, (uint32_t)((nr - 1) * ys + cols) * 4u);
    const int col0 = first_col(c);
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < V; ++j) s += sum4(deviation(v[j], 0.0f, col0 + 64 * j, cols));
    const float mean = kh::row16_sum(s) / n;
    float q = 0.0f;
#pragma unroll
    for (int j = 0; j < V; ++j) {
      v[j] = deviation(v[j], mean, col0 + 64 * j, cols);
      q += squares4(v[j]);
    }
    const float inv = __builtin_amdgcn_rsqf(kh::row16_sum(q) / n + kEps);
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const int col = col0 + 64 * j;
      const uint32_t off = yo + (uint32_t)col * 4u;
      const float4 o = affine4(v[j], inv, *reinterpret_cast<const float4 *>(Gs + col),
                               *reinterpret_cast<const float4 *>(Bs + col));
      if constexpr (PARTS)
        kh::buf_store4(ry, col + 3 < cols ? off : kh::kOutside, o);
      else
        kh::buf_store4_nt(ry, col + 3 < cols ? off : kh::kOutside, o);
      if ((cols & 3) != 0 && cols / 64 == j) {  // uniform: the float4s that hold the rows' last columns
        const bool last = col < cols && col + 3 >= cols;
        kh::buf_store1(ry, last ? off : kh::kOutside, o.x);
        kh::buf_store1(ry, last && col + 1 < cols ? off + 4u : kh::kOutside, o.y);
        kh::buf_store1(ry, last && col + 2 < cols ? off + 8u : kh::kOutside, o.z);
      }
    }
  }
}

// One row per wavefront. Rows move through buffer resources spanning exactly
// cols floats: columns past the end read 0 (kept out of the deviations by a
// select) and their stores are dropped, so the path has no per-lane branches.
// For a wave's first staged row, in a launch that fits one round, and four or
// more float4 per lane, the loads go out in two halves, the second once the
// first has landed (kh::kFirstBurst). Without STAGED, gamma and beta are read
// the same way; with it, from LDS (a lane past cols reads a staged slot it
// does not use: every path that stages has 4 V float4 <= kStageCols). With AHEAD
// they are read beside the row instead of after its reductions.
template <int V, bool STAGED, bool AHEAD = false>
__device__ __forceinline__ void layernorm_rows_regs(const float *__restrict__ X, const float *__restrict__ G,
                                                    const float *__restrict__ B, float *__restrict__ Y,
                                                    int64_t rows, int cols, int64_t xs, int64_t ys,
                                                    int64_t r0, int64_t rstep, int bd, int lane, float *Gs,
                                                    float *Bs) {
  static_assert(!STAGED || 4 * V * kh::kWave <= kStageCols, "staged slots cover every lane's columns");
  const float n = (float)cols;
  const uint32_t row_bytes = (uint32_t)cols * 4u;
  constexpr int kHalf = V >= 4 ? V / 2 : V;
  float4 v[V];
  auto load_row = [&](int64_t r, auto split_tag) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rx = kh::span_rsrc(X + r * xs, row_bytes);
#pragma unroll
    for (int j = 0; j < V; ++j) {
      v[j] = kh::buf_load4_nt(rx, (uint32_t)(lane + j * kh::kWave) * 16u);
      if (decltype(split_tag)::value && j + 1 == kHalf && kHalf < V) kh::vm_wait<0>();
    }
  };
  if constexpr (STAGED) {
    // The staging sits outside the row loop, and the path choice is uniform
    // over the launch. The first row's loads go out before the gamma/beta
    // copy, whose LDS writes wait for them as well (issue order).
    if (r0 < rows) {
      if (kh::split_first_burst(rstep * kh::kWave))  // launch threads
        load_row(r0, std::true_type{});
      else
        load_row(r0, std::false_type{});
    }
    stage_affine(G, B, cols, bd, Gs, Bs);
  }
  const __amdgpu_buffer_rsrc_t rg = kh::span_rsrc(G, row_bytes), rb = kh::span_rsrc(B, row_bytes);
  float4 ga[AHEAD ? V : 1], ba[AHEAD ? V : 1];
  for (int64_t r = r0; r < rows; r += rstep) {
    const __amdgpu_buffer_rsrc_t ry = kh::span_rsrc(Y + r * ys, row_bytes);
    if (!STAGED || r != r0) load_row(r, std::false_type{});
    if constexpr (AHEAD) {
#pragma unroll
      for (int j = 0; j < V; ++j) {
        ga[j] = kh::buf_load4(rg, (uint32_t)(lane + j * kh::kWave) * 16u);
        ba[j] = kh::buf_load4(rb, (uint32_t)(lane + j * kh::kWave) * 16u);
      }
    }
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < V; ++j) s += sum4(v[j]);
    const float mean = kh::wave_sum(s) / n;
    const int col0 = first_col(lane);
    float q = 0.0f;
#pragma unroll
    for (int j = 0; j < V; ++j) {
      v[j] = deviation(v[j], mean, col0 + 4 * kh::kWave * j, cols);
      q += squares4(v[j]);
    }
    const float inv = __builtin_amdgcn_rsqf(kh::wave_sum(q) / n + kEps);
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const uint32_t c = (uint32_t)(lane + j * kh::kWave) * 4u;
      float4 g, b;
      if constexpr (STAGED) {
        g = *reinterpret_cast<const float4 *>(Gs + c);
        b = *reinterpret_cast<const float4 *>(Bs + c);
      } else if constexpr (AHEAD) {
        g = ga[j];
        b = ba[j];
      } else {
        g = kh::buf_load4(rg, 4u * c);
        b = kh::buf_load4(rb, 4u * c);
      }
      kh::buf_store4_nt(ry, 4u * c, affine4(v[j], inv, g, b));
    }
  }
}

// One row per workgroup of nt threads, V float4 per thread (cols <= 4 V nt),
// as many threads as hold the row: every load of the row in flight, one read
// and one write per element (gamma and beta come from L2). The wave
// per row that took such rows a float at a time, in three sweeps, was bound
// by that one wave's load latency: 2048x5000 76.6 -> 17.1 us (4.8 TB/s),
// 512x32001 508 -> 26, 1024x3001 35.0 -> 5.4, 16x65536 602 -> 13.4. More
// threads than the row needs were slower (512x12000 8.3 us at 768, 11.2 at
// 1024; 16384x4096 88.5 at 256, 103 at 512).
template <int V>
__device__ __forceinline__ void layernorm_row_block(const float *__restrict__ xr, const float *__restrict__ G,
                                                    const float *__restrict__ B, float *__restrict__ yr, int cols,
                                                    int nt, int lane, int wave, float (&red)[2][kh::kMaxWaves]) {
  const uint32_t row_bytes = (uint32_t)cols * 4u;
  const __amdgpu_buffer_rsrc_t rx = kh::span_rsrc(xr, row_bytes), ry = kh::span_rsrc(yr, row_bytes);
  const __amdgpu_buffer_rsrc_t rg = kh::span_rsrc(G, row_bytes), rb = kh::span_rsrc(B, row_bytes);
  const int tid = threadIdx.x, nw = nt / kh::kWave;
  const float n = (float)cols;
  float4 v[V];
#pragma unroll
  for (int j = 0; j < V; ++j) v[j] = kh::buf_load4_nt(rx, (uint32_t)(tid + j * nt) * 16u);
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < V; ++j) s += sum4(v[j]);
  const float mean = kh::block_sum(s, red[0], nw, lane, wave) / n;
  const int col0 = first_col(tid);
  float q = 0.0f;
#pragma unroll
  for (int j = 0; j < V; ++j) {
    v[j] = deviation(v[j], mean, col0 + 4 * nt * j, cols);
    q += squares4(v[j]);
  }
  const float inv = __builtin_amdgcn_rsqf(kh::block_sum(q, red[1], nw, lane, wave) / n + kEps);
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const uint32_t off = (uint32_t)(tid + j * nt) * 16u;
    kh::buf_store4_nt(ry, off, affine4(v[j], inv, kh::buf_load4(rg, off), kh::buf_load4(rb, off)));
    if (j & 1) __builtin_amdgcn_sched_barrier(0);  // two float4s of gamma and beta in registers at a time
  }
}

// Rows past the registers of a workgroup: the same two-pass statistics and
// the output in three sweeps over chunks of kStreamV float4 per thread.
constexpr int kStreamV = 4;
__device__ __forceinline__ void layernorm_row_stream(const float *__restrict__ xr, const float *__restrict__ G,
                                                     const float *__restrict__ B, float *__restrict__ yr,
                                                     int64_t cols, int nt, int lane, int wave,
                                                     float (&red)[2][kh::kMaxWaves]) {
  const int tid = threadIdx.x, nw = nt / kh::kWave, chunk = 4 * kStreamV * nt;
  const float n = (float)cols;
  float mean = 0.0f, s = 0.0f;
  for (int sweep = 0; sweep < 2; ++sweep) {
    s = 0.0f;
    for (int64_t c0 = 0; c0 < cols; c0 += chunk) {
      const int nc = cols - c0 < chunk ? (int)(cols - c0) : chunk;
      const __amdgpu_buffer_rsrc_t rx = kh::span_rsrc(xr + c0, (uint32_t)nc * 4u);
      float4 v[kStreamV];
#pragma unroll
      for (int j = 0; j < kStreamV; ++j) v[j] = kh::buf_load4(rx, (uint32_t)(tid + j * nt) * 16u);
      const int col0 = first_col(tid);
      float t = 0.0f;
#pragma unroll
      for (int j = 0; j < kStreamV; ++j) {
        const float4 d = deviation(v[j], mean, col0 + 4 * nt * j, nc);
        t += sweep == 0 ? sum4(d) : squares4(d);
      }
      s += t;
    }
    s = kh::block_sum(s, red[sweep], nw, lane, wave) / n;
    if (sweep == 0) mean = s;
  }
  const float inv = __builtin_amdgcn_rsqf(s + kEps);
  for (int64_t c0 = 0; c0 < cols; c0 += chunk) {
    const int nc = cols - c0 < chunk ? (int)(cols - c0) : chunk;
    const uint32_t bytes = (uint32_t)nc * 4u;
    const __amdgpu_buffer_rsrc_t rx = kh::span_rsrc(xr + c0, bytes), ry = kh::span_rsrc(yr + c0, bytes);
    const __amdgpu_buffer_rsrc_t rg = kh::span_rsrc(G + c0, bytes), rb = kh::span_rsrc(B + c0, bytes);
    float4 v[kStreamV];
#pragma unroll
    for (int j = 0; j < kStreamV; ++j) v[j] = kh::buf_load4(rx, (uint32_t)(tid + j * nt) * 16u);
#pragma unroll
    for (int j = 0; j < kStreamV; ++j) {
      const uint32_t off = (uint32_t)(tid + j * nt) * 16u;
      const float4 d = make_float4(v[j].x - mean, v[j].y - mean, v[j].z - mean, v[j].w - mean);
      kh::buf_store4_nt(ry, off, affine4(d, inv, kh::buf_load4(rg, off), kh::buf_load4(rb, off)));
    }
  }
}

// Blocks that are not whole wavefronts (the reference's own layernorm
// launches use 256 threads, but any block size is accepted): the wave
// reductions need 64 active lanes, so each thread takes whole rows,
// serially, with the same two-pass statistics.
__device__ __forceinline__ void layernorm_row_serial(const float *__restrict__ xr, const float *__restrict__ G,
                                                     const float *__restrict__ B, float *__restrict__ yr,
                                                     int64_t cols) {
  float s = 0.0f;
  for (int64_t c = 0; c < cols; ++c) s += xr[c];
  const float mean = s / (float)cols;
  float q = 0.0f;
  for (int64_t c = 0; c < cols; ++c) {
    const float d = xr[c] - mean;
    q += d * d;
  }
  const float inv = __builtin_amdgcn_rsqf(q / (float)cols + kEps);
  for (int64_t c = 0; c < cols; ++c) yr[c] = fmaf((xr[c] - mean) * inv, G[c], B[c]);
}

// Any width in one wavefront, for launches of layernorm_wave past what its
// registers hold: three sweeps, a float per lane at a time.
__device__ __forceinline__ void layernorm_row_wave(const float *__restrict__ xr, const float *__restrict__ G,
                                                   const float *__restrict__ B, float *__restrict__ yr, int64_t cols,
                                                   int lane) {
  float s = 0.0f;
  for (int64_t c = lane; c < cols; c += kh::kWave) s += xr[c];
  const float mean = kh::wave_sum(s) / (float)cols;
  float q = 0.0f;
  for (int64_t c = lane; c < cols; c += kh::kWave) {
    const float d = xr[c] - mean;
    q += d * d;
  }
  const float inv = __builtin_amdgcn_rsqf(kh::wave_sum(q) / (float)cols + kEps);
  for (int64_t c = lane; c < cols; c += kh::kWave) yr[c] = fmaf((xr[c] - mean) * inv, G[c], B[c]);
}

// Which register paths a symbol compiles in: the kernel's register
// allocation is that of its widest path. Gs and Bs hold kStageCols floats
// each in the narrow symbol and are unused (null) in the others.
enum Symbol { kNarrow, kWide, kMany, kBlock };

template <Symbol S>
__device__ __forceinline__ void layernorm_all(const float *__restrict__ X, const float *__restrict__ G,
                                              const float *__restrict__ B, float *__restrict__ Y, int64_t rows,
                                              int64_t cols, int64_t xs, int64_t ys, int bd, int64_t nb,
                                              float (&red)[2][kh::kMaxWaves], float *Gs, float *Bs) {
  if (bd % kh::kWave != 0) {  // uniform over the block: no thread reaches a barrier below
    for (int64_t r = (int64_t)blockIdx.x * bd + threadIdx.x; r < rows; r += bd * nb)
      layernorm_row_serial(X + r * xs, G, B, Y + r * ys, cols);
    return;
  }
  const int lane = kh::lane_id();
  const int waves_per_block = bd / kh::kWave;
  // Uniform per wave (readfirstlane): the row loop and its buffer resources stay scalar.
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kh::kWave);
  const int64_t r0 = (int64_t)blockIdx.x * waves_per_block + wave;
  const int64_t rstep = waves_per_block * nb;
  const int c = (int)(cols <= KH_ROW_BLOCK_MAX ? cols : KH_ROW_BLOCK_MAX + 1);
  static_assert(kStageCols == 4 * 4 * kh::kWave, "the narrow symbol stages every column its widest wave path holds");
  if (S == kNarrow && c <= KH_ROW16_COLS && xs >= cols && ys >= cols && (xs | ys) < (1 << 26)) {
    if (c <= 64)
      layernorm_rows16<1>(X, G, B, Y, rows, c, xs, ys, 4 * r0, 4 * rstep, bd, lane, Gs, Bs);
    else if (c <= 128)
      layernorm_rows16<2>(X, G, B, Y, rows, c, xs, ys, 4 * r0, 4 * rstep, bd, lane, Gs, Bs);
    else if (rows > KH_ROW16_CACHED_ROWS && kh::shares_lines(Y, ys))
      layernorm_rows16<4, true>(X, G, B, Y, rows, c, xs, ys, 4 * r0, 4 * rstep, bd, lane, Gs, Bs);
    else
      layernorm_rows16<4>(X, G, B, Y, rows, c, xs, ys, 4 * r0, 4 * rstep, bd, lane, Gs, Bs);
  } else if (S == kNarrow && c <= 512) {
    layernorm_rows_regs<2, true>(X, G, B, Y, rows, c, xs, ys, r0, rstep, bd, lane, Gs, Bs);
  } else if (S == kNarrow && c <= 1024) {
    layernorm_rows_regs<4, true>(X, G, B, Y, rows, c, xs, ys, r0, rstep, bd, lane, Gs, Bs);
  } else if ((S == kWide || S == kMany) && c <= 2048) {
    layernorm_rows_regs<8, false, S == kWide>(X, G, B, Y, rows, c, xs, ys, r0, rstep, bd, lane, nullptr, nullptr);
  } else {
    for (int64_t r = blockIdx.x; r < rows; r += nb) {
      const float *xr = X + r * xs;
      float *yr = Y + r * ys;
      if (S != kBlock && c <= 16 * bd)
        layernorm_row_block<4>(xr, G, B, yr, c, bd, lane, wave, red);
      else if (S == kNarrow && c <= 32 * bd)
        layernorm_row_block<8>(xr, G, B, yr, c, bd, lane, wave, red);
      else if (S == kBlock && c <= 64 * bd)
        layernorm_row_block<16>(xr, G, B, yr, c, bd, lane, wave, red);
      else
        layernorm_row_stream(xr, G, B, yr, cols, bd, lane, wave, red);
    }
  }
}

}  // namespace

#define KH_LAYERNORM_BODY(S, GS, BS)                                                                           \
  __shared__ float red[2][kh::kMaxWaves];                                                                      \
  const uint32_t gw = kh::group_size_word(), nb = kh::grid_blocks_x();                                         \
  KH_ARGS_READY(x_base, x_off, x_n0, x_n1, x_s0, gamma_base, gamma_off, beta_base, beta_off, y_base, y_off,    \
                y_s0, gw, nb);                                                                                 \
  layernorm_all<S>(KH_PTR(x), KH_PTR(gamma), KH_PTR(beta), KH_PTR(y), x_n0, x_n1, x_s0, y_s0,                  \
                   (int)kh::threads_x_of(gw), nb, red, GS, BS)

// The reference symbol: rows up to 1024 floats in 16 lanes or a wave, wider
// ones in a workgroup.
extern "C" __global__ void __launch_bounds__(1024)
layernorm(KH_MEMREF2(const float, x), KH_MEMREF1(const float, gamma), KH_MEMREF1(const float, beta),
          KH_MEMREF2(float, y)) {
  __shared__ __attribute__((aligned(16))) float Gs[kStageCols];
  __shared__ __attribute__((aligned(16))) float Bs[kStageCols];
  KH_LAYERNORM_BODY(kNarrow, Gs, Bs);
}

namespace {

// Rows of up to 4 V floats per lane in a wave each, and nothing else.
template <int V, bool STAGED>
__device__ __forceinline__ void layernorm_waves(const float *__restrict__ X, const float *__restrict__ G,
                                                const float *__restrict__ B, float *__restrict__ Y, int64_t rows,
                                                int64_t cols, int64_t xs, int64_t ys, int bd, int64_t nb, float *Gs,
                                                float *Bs) {
  if (bd % kh::kWave != 0) {
    for (int64_t r = (int64_t)blockIdx.x * bd + threadIdx.x; r < rows; r += bd * nb)
      layernorm_row_serial(X + r * xs, G, B, Y + r * ys, cols);
    return;
  }
  const int lane = kh::lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kh::kWave);
  const int64_t r0 = (int64_t)blockIdx.x * (bd / kh::kWave) + wave, rstep = (bd / kh::kWave) * nb;
  if (cols <= 4 * V * kh::kWave)
    layernorm_rows_regs<V, STAGED>(X, G, B, Y, rows, (int)cols, xs, ys, r0, rstep, bd, lane, Gs, Bs);
  else
    for (int64_t r = r0; r < rows; r += rstep) layernorm_row_wave(X + r * xs, G, B, Y + r * ys, cols, lane);
}

}  // namespace

#define KH_LAYERNORM_WAVES(V, STAGED, GS, BS)                                                                  \
  const uint32_t gw = kh::group_size_word(), nb = kh::grid_blocks_x();                                         \
  KH_ARGS_READY(x_base, x_off, x_n0, x_n1, x_s0, gamma_base, gamma_off, beta_base, beta_off, y_base, y_off,    \
                y_s0, gw, nb);                                                                                 \
  layernorm_waves<V, STAGED>(KH_PTR(x), KH_PTR(gamma), KH_PTR(beta), KH_PTR(y), x_n0, x_n1, x_s0, y_s0,        \
                             (int)kh::threads_x_of(gw), nb, GS, BS)

// Same arguments and results for rows of 65..256 floats in launches of few rows
// (KH_LAYERNORM_WAVE_ROWS): a wave per row. One more choice in the reference
// symbol cost its other rows 0.1 us.
extern "C" __global__ void __launch_bounds__(256)
layernorm_wave(KH_MEMREF2(const float, x), KH_MEMREF1(const float, gamma), KH_MEMREF1(const float, beta),
               KH_MEMREF2(float, y)) {
  __shared__ __attribute__((aligned(16))) float Gs[4 * kh::kWave];
  __shared__ __attribute__((aligned(16))) float Bs[4 * kh::kWave];
  KH_LAYERNORM_WAVES(1, true, Gs, Bs);
}

// Same arguments and results for many rows of 2689..4095 floats that share cache
// lines (row_plan, khrt_templates.cpp): a wave per row, held to two on a SIMD by
// the registers it is given. Bound by memory, and here the fewer rows a CU has in
// flight the better: 40000x3000 177 us in workgroups at eight rows a CU
// (layernorm_wide_many), 168 at five, 191 in waves at twenty, 163 in waves at eight.
// At 40000x3072, whole lines, the same four take 161, 158, 179 and 160.
extern "C" __global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
layernorm_wide_parts(KH_MEMREF2(const float, x), KH_MEMREF1(const float, gamma), KH_MEMREF1(const float, beta),
                     KH_MEMREF2(float, y)) {
  KH_LAYERNORM_WAVES(16, false, nullptr, nullptr);
}

// Same arguments and results for rows of 1025..4096 floats (the launcher picks
// it there, up to 2048 from four rows a CU on): a wave per row up to 2048, a
// workgroup past that. Events around rotated launches, wave against workgroup:
// 4096x1100 7.4 vs 8.7 us, 4096x2048 10.9 vs 13.0, 1024x2047 4.8 vs 4.6; past 2048
// the wave's 16 float4 and its share of gamma and beta took 242 registers
// (16384x4096 91.4 vs 88.5).
extern "C" __global__ void __launch_bounds__(256)
layernorm_wide_many(KH_MEMREF2(const float, x), KH_MEMREF1(const float, gamma), KH_MEMREF1(const float, beta),
                    KH_MEMREF2(float, y)) {
  KH_LAYERNORM_BODY(kMany, nullptr, nullptr);
}

// The same for rows of 1025..2048 floats in at most four a CU: gamma and beta are
// under way beside the row. With one wave on a SIMD nothing else covers their
// latency after the reductions (in the same workgroups 600x1468 4.09 -> 3.88 us,
// 200x2048 3.91 -> 3.72). It takes 125 registers for 81, so with more rows it loses
// (1100x1468 5.2 vs 5.9).
extern "C" __global__ void __launch_bounds__(256)
layernorm_wide(KH_MEMREF2(const float, x), KH_MEMREF1(const float, gamma), KH_MEMREF1(const float, beta),
               KH_MEMREF2(float, y)) {
  KH_LAYERNORM_BODY(kWide, nullptr, nullptr);
}

// Same arguments and results; one workgroup per row with 16 float4 per
// thread, for rows past what the reference symbol's eight hold.
extern "C" __global__ void __launch_bounds__(1024)
layernorm_block(KH_MEMREF2(const float, x), KH_MEMREF1(const float, gamma), KH_MEMREF1(const float, beta),
                KH_MEMREF2(float, y)) {
  KH_LAYERNORM_BODY(kBlock, nullptr, nullptr);
}
