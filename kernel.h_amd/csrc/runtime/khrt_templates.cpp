// The seven kernel.h templates behind the C-ABI: embedded gfx950 code
// objects, the registry, the launcher-owned geometry and one entry point per
// template.
//
// Replaces the reference's name -> template dispatch (lib/dsl/registry.cpp:
// 23-36, lib/dsl/program.cpp:17-51) and the per-kernel launch code its
// callers repeat (bench/harness/kernelh_backend.cpp:205-436,
// test/unit/e2e_*_test.cpp). The reference callers own grid/block; here the
// launcher owns geometry per kernel (the kernels stay correct under the
// reference's geometry too), while the memref argument lists, symbol names
// and the hipModuleLoadData / hipModuleLaunchKernel path are unchanged.
#include "kernelh/khrt_internal.hpp"
#include "gemm_tune_list.h"
#include "kh_tiles.h"

#include <algorithm>
#include <array>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <fstream>
#include <initializer_list>
#include <map>
#include <mutex>
#include <string>
#include <vector>

// Code objects linked into the library by kh_embed.S (generated at build).
#define KH_DECLARE_CO(name)              \
  extern "C" const unsigned char kh_co_##name[]; \
  extern "C" const unsigned char kh_co_##name##_end[];
KH_DECLARE_CO(vecadd)
KH_DECLARE_CO(fused_gelu)
KH_DECLARE_CO(softmax)
KH_DECLARE_CO(layernorm)
KH_DECLARE_CO(scan)
KH_DECLARE_CO(gemm)
KH_DECLARE_CO(attention)
KH_DECLARE_CO(util)
KH_DECLARE_CO(roofline)
KH_DECLARE_CO(gemm_tune0)
KH_DECLARE_CO(gemm_tune1)
KH_DECLARE_CO(gemm_tune2)
KH_DECLARE_CO(gemm_tune3)
static_assert(KH_GEMM_TUNE_PARTS == 4, "one code object per part of the tune list");

namespace {

struct CodeObject {
  const char *name;
  const unsigned char *begin;
  const unsigned char *end;
};

const CodeObject kCodeObjects[] = {
    {"vecadd", kh_co_vecadd, kh_co_vecadd_end},       {"fused_gelu", kh_co_fused_gelu, kh_co_fused_gelu_end},
    {"softmax", kh_co_softmax, kh_co_softmax_end},    {"layernorm", kh_co_layernorm, kh_co_layernorm_end},
    {"scan", kh_co_scan, kh_co_scan_end},             {"gemm", kh_co_gemm, kh_co_gemm_end},
    {"attention", kh_co_attention, kh_co_attention_end}, {"util", kh_co_util, kh_co_util_end},
    {"roofline", kh_co_roofline, kh_co_roofline_end},
    {"gemm_tune0", kh_co_gemm_tune0, kh_co_gemm_tune0_end},
    {"gemm_tune1", kh_co_gemm_tune1, kh_co_gemm_tune1_end},
    {"gemm_tune2", kh_co_gemm_tune2, kh_co_gemm_tune2_end},
    {"gemm_tune3", kh_co_gemm_tune3, kh_co_gemm_tune3_end},
};

struct KernelResources {
  const char *symbol;
  khrt_kernel_resources r;
};

// Resource notes of every kernel symbol, generated from the code objects.
const KernelResources kResources[] = {
#include "kh_resources.inc"
};

enum Kind { kVecadd, kGemm, kSoftmax, kLayernorm, kScan, kScanTotals, kFusedGelu, kAttention };

struct Template {
  const char *name;  // template name == kernel symbol
  const char *co;    // code object holding the symbol
  Kind kind;         // its index here
};

// Registry order follows the reference's registration (registry.cpp:23-36).
const Template kTemplates[] = {
    {"vecadd", "vecadd", kVecadd},
    {"gemm", "gemm", kGemm},
    {"softmax", "softmax", kSoftmax},
    {"layernorm", "layernorm", kLayernorm},
    {"scan", "scan", kScan},
    {"scan_totals", "scan", kScanTotals},
    {"fused_gelu", "fused_gelu", kFusedGelu},
    {"attention", "attention", kAttention},
};

const CodeObject *find_co(const char *name) {
  for (const auto &c : kCodeObjects) {
    if (std::strcmp(c.name, name) == 0) return &c;
  }
  return nullptr;
}

const Template *find_template(const char *name) {
  if (name == nullptr) return nullptr;
  for (const auto &t : kTemplates) {
    if (std::strcmp(t.name, name) == 0) return &t;
  }
  return nullptr;
}

std::string registered_list() {
  std::string s;
  for (const auto &t : kTemplates) {
    if (!s.empty()) s += ", ";
    s += t.name;
  }
  return s;
}

int unknown_template(const char *name) {
  return khrt::fail(KHRT_E_INVALID, "unknown kernel '" + std::string(name ? name : "(null)") +
                                        "'; registered kernels: " + registered_list());
}

// Per-device module cache: code object name -> loaded module; symbol ->
// function. Loaded once, kept for the process lifetime.
struct LoadedModule {
  int device;
  std::string co;
  void *module;
};
struct LoadedFunction {
  int device;
  std::string symbol;
  void *function;
};
std::mutex g_mu;
std::vector<LoadedModule> g_modules;
std::vector<LoadedFunction> g_functions;

int get_function(const char *co_name, const char *symbol, void **out) {
  if (int rc = khrt::ensure_device()) return rc;
  const int dev = khrt::current_device();
  std::lock_guard<std::mutex> lock(g_mu);
  for (const auto &f : g_functions) {
    if (f.device == dev && f.symbol == symbol) {
      *out = f.function;
      return 0;
    }
  }
  void *module = nullptr;
  for (const auto &m : g_modules) {
    if (m.device == dev && m.co == co_name) module = m.module;
  }
  if (module == nullptr) {
    const CodeObject *co = find_co(co_name);
    if (co == nullptr) return khrt::fail(KHRT_E_INVALID, std::string("no code object '") + co_name + "'");
    const size_t size = static_cast<size_t>(co->end - co->begin);
    if (size < 64) {
      return khrt::fail(KHRT_E_INVALID, std::string("code object '") + co_name + "' is not part of this build");
    }
    if (int rc = khrt_module_load_data(&module, co->begin, size)) return rc;
    g_modules.push_back({dev, co_name, module});
  }
  void *fn = nullptr;
  if (int rc = khrt_module_get_function(&fn, module, symbol)) return rc;
  g_functions.push_back({dev, symbol, fn});
  *out = fn;
  return 0;
}

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// ---------------------------------------------------------------------------
// GEMM candidates: the launcher's own symbols, then the tune space
// (gemm_tune_list.h). Every one takes the template `gemm` arguments and
// computes C = A B for every shape and grid.
enum GemmPipe { kRegs = 1, kDma = 2, kPf2 = 3, kPersistent = 4, kKsplit = 5, kKsplitDeep = 6 };

const char *pipe_name(int pipe) {
  switch (pipe) {
    case kRegs: return "regs";
    case kDma: return "lds-dma";
    case kPf2: return "prefetch2";
    case kPersistent: return "persistent";
    case kKsplit: return "ksplit";
    case kKsplitDeep: return "ksplit-deep";
    default: return "?";
  }
}

struct GemmCandidate {
  const char *symbol;
  const char *co;
  int mfma, wgm, wgn, wtm, wtn, bk, prio, pipe;
  bool product;
  // Persistent symbols: workgroups resident per CU (their LDS and
  // registers), so the launcher's grid is one round of them.
  int per_cu = 2;
  int ks_bm = KH_GEMM_KSPLIT_BM, ks_bn = KH_GEMM_KSPLIT_BN;  // K-split symbols' tiles
  bool ksplit() const { return pipe == kKsplit || pipe == kKsplitDeep; }
  // K-split: each of the 8 waves holds the whole tile for its K range.
  int waves() const { return ksplit() ? KH_GEMM_KSPLIT_THREADS / 64 : wgm * wgn; }
  int bm() const { return ksplit() ? ks_bm : mfma * wtm * wgm; }
  int bn() const { return ksplit() ? ks_bn : mfma * wtn * wgn; }
  // Slabs (K-split: register sets of loads) in flight ahead of the MFMAs.
  int unroll() const { return pipe == kRegs ? 1 : 2; }
};

#define KH_TUNE_CANDIDATE(PART, MF, WGM, WGN, WTM, WTN, BK, PRIO, PIPE, SYM) \
  {#SYM, "gemm_tune" #PART, MF, WGM, WGN, WTM, WTN, BK, PRIO, PIPE, false},
const GemmCandidate kGemmCandidates[] = {
    {"gemm", "gemm", 32, 2, 2, 2, 4, 16, 1, kPersistent, true},
    {"gemm_mid", "gemm", 32, 2, 2, 2, 2, 32, 1, kRegs, true},
    {"gemm_small", "gemm", 16, 4, 2, 1, 2, 32, 1, kPersistent, true},
    {"gemm_small_pf2", "gemm", 16, 2, 2, 2, 2, 32, 1, kPf2, true},
    {"gemm_wide", "gemm", 16, 4, 2, 2, 4, 32, 1, kPersistent, true, 1},
    {"gemm_ksplit", "gemm", 32, 1, 1, 1, 1, 8, 0, kKsplit, true},
    {"gemm_ksplit_deep", "gemm", 32, 1, 1, 1, 1, 8, 0, kKsplitDeep, true},
    {"gemm_ksplit_16x16", "gemm", 16, 1, 1, 1, 1, 16, 0, kKsplit, true, 2, 16, 16},
    {"gemm_ksplit_32x16", "gemm", 16, 1, 1, 2, 1, 16, 0, kKsplit, true, 2, 32, 16},
    {"gemm_ksplit_32x64", "gemm", 16, 1, 1, 2, 4, 16, 0, kKsplit, true, 2, 32, 64},
    KH_GEMM_TUNE_CONFIGS(KH_TUNE_CANDIDATE)};
#undef KH_TUNE_CANDIDATE
constexpr int kGemmCandidateCount = static_cast<int>(sizeof(kGemmCandidates) / sizeof(kGemmCandidates[0]));
static_assert(kGemmCandidateCount == 10 + KH_GEMM_TUNE_COUNT, "candidate table");

const GemmCandidate *find_gemm_candidate(const char *symbol) {
  if (symbol == nullptr) return nullptr;
  for (const auto &c : kGemmCandidates) {
    if (std::strcmp(c.symbol, symbol) == 0) return &c;
  }
  return nullptr;
}

// Grid of a candidate at m x n: one workgroup per tile, except the
// persistent symbols, which get one round of resident workgroups and loop
// (per_cu: two for `gemm` and `gemm_small`, one for `gemm_wide`, whose
// 99 KB of LDS allow no more).
int64_t candidate_grid(const GemmCandidate &c, int64_t m, int64_t n) {
  const int64_t tiles = ceil_div(m, c.bm()) * ceil_div(n, c.bn());
  // The K-split symbols loop over their tiles as well: one workgroup per CU
  // (their registers allow no more) measured better than one per tile
  // beyond a round (768^3 18.0 vs 19.0 us, 512x1024x1024 15.1 vs 15.7).
  if (c.ksplit()) return std::min<int64_t>(tiles, KH_GEMM_CUS);
  if (c.pipe == kPersistent) return std::min<int64_t>(tiles, int64_t(c.per_cu) * KH_GEMM_CUS);
  return tiles;
}

// The tune cache `kernelh tune` writes: one JSON object per line,
// {"key": "<16 hex>", "best": "<symbol>", "csv": "..."}, keyed by FNV-1a 64
// of "gemm|m=..,n=..,k=..|<device token>". The launcher reads it only when a
// path is set (khrt_set_tune_cache, or KHRT_TUNE_CACHE in the environment at
// the first GEMM launch); the file is read once per path.
std::string fnv1a_hex(const std::string &s) {
  uint64_t h = 1469598103934665603ull;
  for (unsigned char ch : s) {
    h ^= ch;
    h *= 1099511628211ull;
  }
  char buf[17];
  std::snprintf(buf, sizeof buf, "%016llx", static_cast<unsigned long long>(h));
  return buf;
}

// Asked once per device (hipGetDeviceProperties is not cheap enough to sit
// on every launch).
std::string device_token() {
  static std::mutex mu;
  static std::map<int, std::string> memo;
  if (khrt::ensure_device() != 0) return "";
  const int dev = khrt::current_device();
  {
    std::lock_guard<std::mutex> lock(mu);
    auto it = memo.find(dev);
    if (it != memo.end()) return it->second;
  }
  khrt_device_info d{};
  if (khrt_get_device_info(&d) != 0) return "";
  const std::string token = std::string(d.name[0] ? d.name : "AMD Instinct MI355X") + " (" + d.arch + ") cu=" +
                            std::to_string(static_cast<long long>(d.cu_count));
  std::lock_guard<std::mutex> lock(mu);
  memo[dev] = token;
  return token;
}

std::string gemm_shape_text(int64_t m, int64_t n, int64_t k) {
  return "m=" + std::to_string(m) + ",n=" + std::to_string(n) + ",k=" + std::to_string(k);
}

struct TuneCache {
  std::mutex mu;
  bool configured = false;  // khrt_set_tune_cache called, or the environment read
  std::string path;
  bool loaded = false;
  std::map<std::string, std::string> best;  // key -> symbol
};
TuneCache g_tune;

void load_tune_cache_locked() {
  g_tune.best.clear();
  g_tune.loaded = true;
  if (g_tune.path.empty()) return;
  std::ifstream f(g_tune.path);
  std::string line;
  const std::string kk = "{\"key\": \"", kb = "\"best\": \"";
  while (std::getline(f, line)) {
    if (line.rfind(kk, 0) != 0) continue;
    const size_t ke = line.find('"', kk.size());
    const size_t b = line.find(kb);
    if (ke == std::string::npos || b == std::string::npos) continue;
    const size_t be = line.find('"', b + kb.size());
    if (be == std::string::npos) continue;
    g_tune.best[line.substr(kk.size(), ke - kk.size())] = line.substr(b + kb.size(), be - b - kb.size());
  }
}

// The tuned candidate for this GEMM shape, or nullptr (no cache, no entry,
// or an entry naming a symbol this build does not have).
const GemmCandidate *tuned_gemm(int64_t m, int64_t n, int64_t k) {
  std::string key;
  {
    std::lock_guard<std::mutex> lock(g_tune.mu);
    if (!g_tune.configured) {
      const char *env = std::getenv("KHRT_TUNE_CACHE");
      g_tune.path = env != nullptr ? env : "";
      g_tune.configured = true;
      g_tune.loaded = false;
    }
    if (g_tune.path.empty()) return nullptr;
    if (!g_tune.loaded) load_tune_cache_locked();
    if (g_tune.best.empty()) return nullptr;
  }
  const std::string dev = device_token();
  if (dev.empty()) return nullptr;
  key = fnv1a_hex("gemm|" + gemm_shape_text(m, n, k) + "|" + dev);
  std::lock_guard<std::mutex> lock(g_tune.mu);
  auto it = g_tune.best.find(key);
  return it == g_tune.best.end() ? nullptr : find_gemm_candidate(it->second.c_str());
}

// GEMM tile choice: the largest tile whose grid still gives every CU work.
// Rate x busy fraction of the last round of workgroups (kh_tiles.h).
double gemm_score(int64_t tiles, int64_t round, double rate) {
  return rate * static_cast<double>(tiles) / static_cast<double>(ceil_div(tiles, round) * round);
}

const char *heuristic_gemm_symbol(int64_t m, int64_t n, int64_t k) {
  // K split (kh_tiles.h): the smallest tile that gives every CU at most one
  // workgroup; of 32x32 tiles also more, where all are whole and the 64x64
  // tiles number fewer than the CUs.
  auto ks_tiles = [&](int64_t bm, int64_t bn) { return ceil_div(m, bm) * ceil_div(n, bn); };
  const bool whole = m % KH_GEMM_KSPLIT_BM == 0 && n % KH_GEMM_KSPLIT_BN == 0 && k % KH_GEMM_KSPLIT_INTERIOR_K == 0;
  const bool deep = k >= KH_GEMM_KSPLIT_DEEP_K &&
                    (whole || static_cast<double>(m + n) * static_cast<double>(k) >= KH_GEMM_KSPLIT_DEEP_FLOATS);
  // Past the K splits' 32-bit offsets (gemm.hip, ks_any_ok at 8 waves) only the 16x16
  // tiles have a form with 64-bit ones.
  const int64_t span = int64_t(1) << 29;  // floats
  const bool far = k >= span / 64 || (k / 8 + 64) * n >= span;
  const char *ks32 = far ? "gemm_ksplit_16x16" : deep ? "gemm_ksplit_deep" : "gemm_ksplit";
  const int64_t tiles64 = ks_tiles(KH_GEMM_SMALL_BM, KH_GEMM_SMALL_BN);
  // Whole 32x32 tiles move 16 k a batch and wave, the smaller tiles 32, so that
  // an odd multiple of 128 leaves each of their waves half a batch of padding.
  // One 32x16 tile per CU against a 32x32 one on half of them, K = 128: 4.0 vs
  // 3.2 us, 384 5.3 vs 4.6, 640 6.3 vs 5.8, 1408 10.4 vs 9.4, 1920 13.2 vs 11.8
  // (256, 512 and 1024 level; 2048 and past it the smaller, 512x256x4096 22.0 vs
  // 23.8). A 16x16 tile wins but at K = 128: 3.3-3.5 vs 2.9-3.2 us (256 3.4 vs 3.9).
  const bool half = whole && k % (2 * KH_GEMM_KSPLIT_INTERIOR_K) != 0;
  if (ks_tiles(16, 16) <= KH_GEMM_CUS) return half && k == KH_GEMM_KSPLIT_INTERIOR_K ? ks32 : "gemm_ksplit_16x16";
  if (ks_tiles(32, 16) <= KH_GEMM_CUS) return far || (half && k < KH_GEMM_KSPLIT_DEEP_K) ? ks32 : "gemm_ksplit_32x16";
  if (ks_tiles(KH_GEMM_KSPLIT_BM, KH_GEMM_KSPLIT_BN) <= KH_GEMM_CUS) return ks32;
  if (tiles64 < KH_GEMM_CUS && whole && k >= KH_GEMM_KSPLIT_MIN_K) return ks32;
  // Past a slab of the 64x64 tiles only: their merge of eight waves' partial
  // tiles costs more than a single slab's products (448x640, K of 1 to 32: 4.5 us
  // against 4.0 in `gemm_small`; K = 33: 4.6 against 4.9).
  if (k > KH_GEMM_SMALL_BK && ks_tiles(32, 64) <= KH_GEMM_CUS) return far ? ks32 : "gemm_ksplit_32x64";
  const double big = gemm_score(ceil_div(m, KH_GEMM_BM) * ceil_div(n, KH_GEMM_BN), KH_GEMM_ROUND_BIG,
                                KH_GEMM_RATE_BIG);
  const double mid = gemm_score(ceil_div(m, KH_GEMM_MID_BM) * ceil_div(n, KH_GEMM_MID_BN), KH_GEMM_ROUND_MID,
                                KH_GEMM_RATE_MID);
  const double wide = gemm_score(ceil_div(m, KH_GEMM_WIDE_BM) * ceil_div(n, KH_GEMM_WIDE_BN), KH_GEMM_ROUND_WIDE,
                                 KH_GEMM_RATE_WIDE);
  const double small = gemm_score(ceil_div(m, KH_GEMM_SMALL_BM) * ceil_div(n, KH_GEMM_SMALL_BN),
                                  KH_GEMM_ROUND_SMALL, KH_GEMM_RATE_SMALL);
  if (big >= mid && big >= wide && big >= small) return "gemm";
  if (mid >= wide && mid > small) return "gemm_mid";
  if (wide > small) return "gemm_wide";
  return "gemm_small";
}

// The launcher's GEMM candidate: the tune cache's choice for this shape when
// one is set and names a candidate, the heuristic's otherwise.
const GemmCandidate &gemm_choice(int64_t m, int64_t n, int64_t k) {
  if (const GemmCandidate *t = tuned_gemm(m, n, k)) return *t;
  return *find_gemm_candidate(heuristic_gemm_symbol(m, n, k));
}

unsigned clamp_grid(int64_t g) { return static_cast<unsigned>(std::max<int64_t>(1, std::min<int64_t>(g, 1 << 20))); }

using Shape = std::map<std::string, int64_t>;

bool need(const Shape &s, const char *key, int64_t &v) {
  auto it = s.find(key);
  if (it == s.end() || it->second <= 0) return false;
  v = it->second;
  return true;
}

// How softmax and layernorm hold a row of `cols` floats (kh_tiles.h): the
// symbol that runs it, the threads of a workgroup and the rows it takes at a
// time.
struct RowPlan {
  const char *symbol;
  unsigned threads;
  int64_t rows_per_block;
};

RowPlan row_plan(bool softmax, int64_t rows, int64_t cols) {
  const char *narrow = softmax ? "softmax" : "layernorm", *wide = softmax ? "softmax_wide" : "layernorm_wide_many",
             *block = softmax ? "softmax_block" : "layernorm_block";
  // Too few rows for four to a wave.
  const bool few = rows <= (softmax ? KH_SOFTMAX_WAVE_ROWS(cols) : KH_LAYERNORM_WAVE_ROWS(cols));
  // Many rows of 193..255 floats whose ends share cache lines: a wave's four rows
  // leave more parts of lines than it pays in one (softmax 40000x200 14.6 us,
  // 14.1 through the cache, 13.3 in a wave each; 300000x252 118, 107, 99; with
  // 16384 rows and fewer 2-7% the other way).
  const bool many_parts = softmax && cols > 192 && cols % 32 != 0 && rows > 16384;
  if (cols <= KH_ROW16_COLS && !few && !many_parts) {
    // Between two and three workgroups of 16 rows per CU the last ones leave CUs
    // idle for longer than half as large ones do (layernorm 8500x256 5.2 vs 4.6 us,
    // 9300x224 5.5 vs 4.7, 12000x256 5.9 vs 5.5; past three within 4% either way).
    if (!softmax && cols > 128 && rows > 2 * 16 * KH_GEMM_CUS && rows < 3 * 16 * KH_GEMM_CUS) return {narrow, 128, 8};
    return {narrow, 256, 16};
  }
  if (softmax && cols <= 512) return {"softmax_wave", 256, 4};
  // Launches that just about fill the chip once, 28 to 34 rows a CU: `softmax` took
  // 7200x640 8.9 us, 8.2 in softmax_wave, 8192x640 10.0 and 8.9, 8192x768 10.9 and 10.0,
  // 8400x900 12.8 and 12.6, 8192x1024 13.4 and 13.4; with fewer rows the two are
  // level (7000x576 7.05 and 7.28), with more `softmax` is 1% faster.
  if (softmax && cols < 1024 && rows > 28 * KH_GEMM_CUS && rows <= 34 * KH_GEMM_CUS) return {"softmax_wave", 256, 4};
  if (cols <= KH_ROW16_COLS) return {"layernorm_wave", 256, 4};
  if (cols <= 1024) return {narrow, 256, 4};
  // layernorm in at most one wave on a SIMD (layernorm_wide; layernorm_wide_many
  // otherwise, as from 1100x1468, 5.2 vs 5.9 us, and 1000x2000, 4.8 vs 5.0): four
  // rows to a workgroup, or one while that gives a CU two at most (200x1468 3.47 vs
  // 3.30 us, 512x2000 4.00 vs 3.64, 512x1100 3.61 vs 3.67, 800x1468 4.08 vs 4.30).
  if (!softmax && cols <= 2048 && rows <= 4 * KH_GEMM_CUS && rows * cols <= 7 << 18) {
    if (rows <= 2 * KH_GEMM_CUS) return {"layernorm_wide", 64, 1};
    return {"layernorm_wide", 256, 4};
  }
  if (cols <= 2048) return {wide, 256, 4};
  if (cols > KH_ROW_BLOCK_MAX) return {block, 1024, 1};
  // softmax of 2049..4096 floats in up to ten rows per CU, once there is enough to
  // move: a wave per row (16 float4 per lane) holds the chip's rows all at once
  // and crosses no barriers; in workgroups of 192 or 256 threads their bursts of
  // loads meet. Workgroup against wave: 1700x2560 8.0 vs 7.1 us, 2048x3328 11.4 vs
  // 9.2, 2048x4096 13.4 vs 11.3, 2560x2304 10.4 vs 9.2, and the other way 1100x2052
  // 5.3 vs 5.9, 1500x2560 6.4 vs 6.7, 1200x2816 6.0 vs 6.1, 3000x4096 18.2 vs 18.7,
  // 8192x2560 28.5 vs 30.5.
  if (softmax && cols <= 4096 && rows <= 10 * KH_GEMM_CUS && (rows * cols >= 15 << 18 || 2 * rows >= 13 * KH_GEMM_CUS))
    return {block, 64, 1};
  // layernorm of many rows that share cache lines keeps fewer of them in flight
  // (layernorm_wide_parts): 40000x2800 157.6 vs 150.4 us, 40000x3000 177.9 vs 163.1,
  // 40000x3676 209 vs 194, 16384x3792 87.9 vs 84.0; 8192x3000 37.0 vs 37.1, 12300x2564
  // 46.3 vs 47.2, and rows of whole lines 16384x3072 67.8 vs 68.5.
  if (!softmax && cols > 2688 && cols <= 4096 && cols % 32 != 0 && rows > 48 * KH_GEMM_CUS)
    return {"layernorm_wide_parts", 256, 4};
  // A workgroup per row, as few whole waves as hold it at 4, 8 or 16 float4
  // per thread: the fewest that need at most 768 threads. At 4 and 8 (at most 64
  // registers) a CU then holds two workgroups or more, and one's loads fill the
  // other's reductions and stores; at 16 (96 and 94 registers, 20 waves on a CU)
  // two up to 640 threads, 40960 columns. Rotated launches, softmax / layernorm:
  // 300x13000 9.5 / 10.5 us at 832 threads, 7.0 / 7.6 at 448; 1024x16000 26.7 / 28.5
  // at 1024, 23.6 / 25.6 at 512; 512x32001 27.7 / 28.7 at 1024, 24.7 / 25.7 at 512. At
  // 768 and below the two splits are within 4% (2000x10000, 4000x12000). With a CU
  // for every row there is no second workgroup, and 16 float4 gain nothing over 8
  // (256x32001: 14.2 us at 1024 threads, 14.4 at 512).
  auto threads = [&](int v) { return static_cast<unsigned>(64 * ceil_div(ceil_div(cols, 4), 64 * v)); };
  if (cols <= 4096) return {wide, threads(4), 1};
  if (threads(4) <= 768) return {narrow, threads(4), 1};
  if (threads(8) <= 768 || (threads(8) <= 1024 && rows <= KH_GEMM_CUS)) return {narrow, threads(8), 1};
  return {block, threads(16), 1};
}

// How attention spreads (batch, heads, seq) over the chip: query rows per
// workgroup, and what a launch of that symbol takes. `resident` workgroups
// share a CU (registers and LDS), so workgroups run in rounds of that many per
// CU; a round of i of them takes step[i - 1] us for each key step of a wave
// and fixed[i - 1] for its start and merge, a launch `start`.
struct AttentionForm {
  const char *symbol;
  int64_t rows, keys, waves;  // query rows; keys per step; waves the keys are split over
  int resident;
  double start, step[3], fixed[3];
};

// Fitted to the three symbols timed at 1193 launches (1 to 4096 slices of 8 to
// 8192 keys): the symbol taken is within 3% of the fastest at 99% of them and
// loses more than 1% to `attention` at four (at most 9%). A model that paid start
// and merge once per launch, and one workgroup per CU, held up to 64 slices
// and was up to 38% slower than `attention` past that: 256x129 37.8 us for
// 29.7-32, 384x128 31.6 for 25.3, 1024x200 181 for 148.
const AttentionForm kAttentionForms[] = {
    {"attention", KH_ATTN_BLOCK_Q, 64, 1, 2, 1.9, {4.0, 8.0}, {3.1, 4.15}},
    {"attention_split", 32, 32, 4, 2, 2.7, {1.45, 3.85}, {5.15, 5.4}},
    {"attention_split16", 16, 32, 4, 3, 2.9, {0.7, 2.0, 3.35}, {3.4, 3.75, 3.4}},
};

double attention_us(const AttentionForm &f, int64_t slices, int64_t seq) {
  const int64_t per_cu = ceil_div(slices * ceil_div(seq, f.rows), KH_GEMM_CUS);
  const int64_t full = per_cu / f.resident, rest = per_cu % f.resident;
  const int64_t steps = ceil_div(seq, f.keys), longest = ceil_div(steps, f.waves);
  // Waves without a last step leave their share to the CU's other workgroups,
  // but not where there are none.
  const double mean = (static_cast<double>(steps) / static_cast<double>(f.waves) + static_cast<double>(longest)) / 2;
  double us = f.start + static_cast<double>(full) * (f.step[f.resident - 1] * mean + f.fixed[f.resident - 1]);
  if (rest > 0) us += f.step[rest - 1] * (full == 0 ? static_cast<double>(longest) : mean) + f.fixed[rest - 1];
  return us;
}

const AttentionForm &attention_form(int64_t batch, int64_t heads, int64_t seq) {
  const AttentionForm &whole = kAttentionForms[0], &split = kAttentionForms[1], &split16 = kAttentionForms[2];
  // Past this the split kernels' 32-bit offsets do not reach.
  if (batch > 65535 || heads > 65535 || seq > (int64_t(1) << 22)) return whole;
  const double us = attention_us(split, batch * heads, seq), us16 = attention_us(split16, batch * heads, seq);
  if (attention_us(whole, batch * heads, seq) <= 1.02 * std::min(us, us16)) return whole;  // level: the fewer
  return us <= us16 ? split : split16;
}

// Extents of a template's shape, in the order its entry point takes them:
// n; rows, cols; m, n, k; batch, heads, seq, head_dim.
using Dims = std::array<int64_t, 4>;

// Dims of a parsed shape, or the error that names what is missing.
int dims_of(const Template &tpl, const Shape &s, Dims &d) {
  const std::string t = tpl.name;
  if (tpl.kind == kVecadd || tpl.kind == kFusedGelu) {
    if (!need(s, "n", d[0])) {
      if (tpl.kind == kFusedGelu && need(s, "rows", d[0]) && need(s, "cols", d[1])) {
        d[0] *= d[1];
      } else {
        return khrt::fail(KHRT_E_INVALID, t + ": shape attribute 'n' is required and must be positive");
      }
    }
  } else if (tpl.kind == kSoftmax || tpl.kind == kLayernorm) {
    if (!need(s, "rows", d[0]) || !need(s, "cols", d[1])) {
      return khrt::fail(KHRT_E_INVALID, t + ": shape attributes 'rows' and 'cols' are required and must be positive");
    }
  } else if (tpl.kind == kScan || tpl.kind == kScanTotals) {
    if (!need(s, "n", d[0])) return khrt::fail(KHRT_E_INVALID, t + ": shape attribute 'n' is required and must be positive");
  } else if (tpl.kind == kGemm) {
    if (!need(s, "m", d[0]) || !need(s, "n", d[1]) || !need(s, "k", d[2])) {
      return khrt::fail(KHRT_E_INVALID, "gemm: shape attributes 'm', 'n' and 'k' are required and must be positive");
    }
  } else {
    if (!need(s, "batch", d[0]) || !need(s, "heads", d[1]) || !need(s, "seq", d[2]) || !need(s, "head_dim", d[3])) {
      return khrt::fail(KHRT_E_INVALID,
                        "attention: shape attributes 'batch', 'heads', 'seq' and 'head_dim' are required and "
                        "must be positive");
    }
  }
  return 0;
}

// What the launcher runs for a template at a shape: the symbol (every symbol
// of a template takes the same arguments and computes the same result), its
// code object and the launch geometry (see each kernel's header comment).
struct Plan {
  const char *symbol;
  const char *co;
  khrt_dim3 grid, block;
};

int make_plan(const Template &tpl, const Dims &d, Plan &p) {
  p = Plan{tpl.name, tpl.co, {1, 1, 1}, {256, 1, 1}};
  switch (tpl.kind) {
    case kVecadd:
    case kFusedGelu:
      p.grid.x = clamp_grid(ceil_div(ceil_div(d[0], 4), 256LL * KH_EW_UNROLL));
      return 0;
    case kSoftmax:
    case kLayernorm: {
      const RowPlan r = row_plan(tpl.kind == kSoftmax, d[0], d[1]);
      p.symbol = r.symbol;
      p.block.x = r.threads;
      p.grid.x = clamp_grid(ceil_div(d[0], r.rows_per_block));
      return 0;
    }
    case kScan:
      p.block.x = d[0] <= KH_SCAN_SMALL_N ? KH_SCAN_SMALL_THREADS : KH_SCAN_THREADS;
      p.grid.x = clamp_grid(ceil_div(d[0], int64_t(KH_SCAN_PER_THREAD) * (p.block.x - 64)));
      return 0;
    case kScanTotals:
      p.grid.x = clamp_grid(std::min<int64_t>(ceil_div(ceil_div(d[0], 256) + 1, 256), 1024));
      return 0;
    case kGemm: {
      const GemmCandidate &c = gemm_choice(d[0], d[1], d[2]);
      p.symbol = c.symbol;
      p.co = c.co;
      p.grid.x = clamp_grid(candidate_grid(c, d[0], d[1]));
      p.block.x = static_cast<unsigned>(64 * c.waves());
      return 0;
    }
    case kAttention: {
      if (d[3] != 64) {
        return khrt::fail(KHRT_E_INVALID, "attention: the kernel is pinned to head_dim = 64 (got head_dim = " +
                                              std::to_string(d[3]) + ")");
      }
      const AttentionForm &a = attention_form(d[0], d[1], d[2]);
      p.symbol = a.symbol;
      p.grid = {static_cast<unsigned>(ceil_div(d[2], a.rows)), static_cast<unsigned>(d[1]),
                static_cast<unsigned>(d[0])};
      return 0;
    }
  }
  return unknown_template(tpl.name);
}

// The plan of a shape given as text.
int plan_of(const char *name, const char *shape, Plan &p) {
  const Template *t = find_template(name);
  if (t == nullptr) return unknown_template(name);
  Shape s;
  std::string why;
  if (!kernelh::parse_shape_text(shape, s, &why)) return khrt::fail(KHRT_E_INVALID, "malformed shape: expected " + why);
  Dims d{};
  if (int rc = dims_of(*t, s, d)) return rc;
  return make_plan(*t, d, p);
}

// Workgroups of `block` threads of `fn` resident on the whole device at
// once (occupancy per CU x CUs), asked once per function; 0 if unknown.
int64_t resident_workgroups(void *fn, unsigned block) {
  struct Entry {
    void *fn;
    unsigned block;
    int64_t resident;
  };
  static std::mutex mu;
  static std::vector<Entry> cache;
  {
    std::lock_guard<std::mutex> lock(mu);
    for (const auto &e : cache) {
      if (e.fn == fn && e.block == block) return e.resident;
    }
  }
  int per_cu = 0;
  khrt_device_limits live;
  int64_t resident = 0;
  if (hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, static_cast<hipFunction_t>(fn),
                                                         static_cast<int>(block), 0) == hipSuccess &&
      per_cu > 0 && khrt_live_limits(&live) == 0 && live.cu_count > 0) {
    resident = int64_t(per_cu) * live.cu_count;
  } else {
    (void)hipGetLastError();
  }
  std::lock_guard<std::mutex> lock(mu);
  cache.push_back({fn, block, resident});
  return resident;
}

// Functions launched before: what a launch of `symbol` with `threads` threads
// on `device` needs besides its arguments. The verifier's other rules (shared
// memory, threads, wave multiple, occupancy) depend on nothing else, and the
// embedded modules stay loaded for the process's life, so once a launch has
// passed it only the grid is left to check. Entries are only ever appended,
// whole, under the mutex; readers see them through the count. A full table
// only means that further functions verify every launch.
struct Ready {
  const char *symbol;
  int device;
  unsigned threads;
  void *fn;
  int64_t resident;  // workgroups on the device at once (scan; 0: not asked)
  int64_t max_grid[3];
};
constexpr int kMaxReady = 512;
Ready g_ready[kMaxReady];
std::atomic<int> g_nready{0};
std::mutex g_ready_mu;

const Ready *find_ready(const char *symbol, int device, unsigned threads) {
  const int n = g_nready.load(std::memory_order_acquire);
  for (int i = 0; i < n; ++i) {
    const Ready &r = g_ready[i];
    if (r.symbol == symbol && r.threads == threads && r.device == device) return &r;
  }
  return nullptr;
}

void add_ready(const Ready &r) {
  std::lock_guard<std::mutex> lock(g_ready_mu);
  const int n = g_nready.load(std::memory_order_relaxed);
  if (n == kMaxReady || find_ready(r.symbol, r.device, r.threads) != nullptr) return;
  g_ready[n] = r;
  g_nready.store(n + 1, std::memory_order_release);
}

// Kernel parameters of a template call on the stack: the memref descriptors
// of LaunchArgs, contiguous row-major with offset 0.
class StackArgs {
 public:
  void add_memref(const void *ptr, std::initializer_list<int64_t> shape) {
    const uint64_t p = static_cast<uint64_t>(reinterpret_cast<uintptr_t>(ptr));
    const size_t rank = shape.size();
    uint64_t *s = slots_ + count_;
    s[0] = s[1] = p;
    s[2] = 0;
    uint64_t stride = 1;
    for (size_t i = rank; i-- > 0;) {
      s[3 + i] = static_cast<uint64_t>(shape.begin()[i]);
      s[3 + rank + i] = stride;
      stride *= static_cast<uint64_t>(shape.begin()[i]);
    }
    count_ += 3 + 2 * rank;
  }
  void **params() {
    for (size_t i = 0; i < count_; ++i) params_[i] = &slots_[i];
    return params_;
  }
  size_t count() const { return count_; }

 private:
  static constexpr size_t kMax = 44;  // attention: four of rank 4
  uint64_t slots_[kMax];
  void *params_[kMax];
  size_t count_ = 0;
};

// Verifies and launches template `kind` at extents `d`.
int launch_template(Kind kind, StackArgs &args, const Dims &d, void *stream) {
  Plan p;
  if (int rc = make_plan(kTemplates[kind], d, p)) return rc;
  if (int rc = khrt::ensure_device()) return rc;
  const int dev = khrt::current_device();
  const Ready *known = find_ready(p.symbol, dev, p.block.x);
  Ready r;
  if (known != nullptr) {
    r = *known;
  } else {
    r = Ready{p.symbol, dev, p.block.x, nullptr, 0, {0, 0, 0}};
    if (int rc = get_function(p.co, p.symbol, &r.fn)) return rc;
    if (kind == kScan) r.resident = resident_workgroups(r.fn, p.block.x);
    khrt_device_limits live;
    if (int rc = khrt_live_limits(&live)) return rc;
    for (int i = 0; i < 3; ++i) r.max_grid[i] = live.max_grid_dim[i];
  }
  if (kind == kScan && r.resident > 0) {
    // The look-back scan is persistent: one resident wave of workgroups
    // loops over tiles, so launch no more workgroups than fit at once, and
    // as many as give every workgroup the same number of tiles (grid.x is
    // the tile count here): 4370 tiles at n = 2^26 run as 18 full rounds of
    // 243 workgroups, not 17 rounds of 256 and an 18th of 18 tiles, during
    // which HBM idles.
    const int64_t tiles = p.grid.x, rounds = ceil_div(tiles, r.resident);
    p.grid.x = static_cast<unsigned>(ceil_div(tiles, rounds));
  }
  if (known != nullptr && p.grid.x <= r.max_grid[0] && p.grid.y <= r.max_grid[1] && p.grid.z <= r.max_grid[2]) {
    return khrt_launch_raw(r.fn, p.grid, p.block, 0, stream, args.params());
  }
  if (int rc = khrt::verified_launch(r.fn, p.grid, p.block, 0, stream, args.params(), args.count())) return rc;
  if (known == nullptr) add_ready(r);
  return 0;
}

int bad(const char *what) { return khrt::fail(KHRT_E_INVALID, what); }

}  // namespace

extern "C" {

int khrt_template_count(void) { return static_cast<int>(sizeof(kTemplates) / sizeof(kTemplates[0])); }

const char *khrt_template_name(int i) {
  if (i < 0 || i >= khrt_template_count()) return nullptr;
  return kTemplates[i].name;
}

int khrt_template_code_object(const char *name, const void **image, size_t *size) {
  if (image == nullptr || size == nullptr) return bad("khrt_template_code_object: null output");
  const Template *t = find_template(name);
  if (t == nullptr) return unknown_template(name);
  const CodeObject *co = find_co(t->co);
  *image = co->begin;
  *size = static_cast<size_t>(co->end - co->begin);
  if (*size < 64) return khrt::fail(KHRT_E_INVALID, std::string("code object for '") + name + "' is not part of this build");
  return 0;
}

int khrt_template_resources(const char *name, khrt_kernel_resources *out) {
  if (out == nullptr) return bad("khrt_template_resources: null output");
  if (name == nullptr) return unknown_template(name);
  for (const auto &r : kResources) {
    if (std::strcmp(r.symbol, name) == 0) {
      *out = r.r;
      return 0;
    }
  }
  return unknown_template(name);
}

int khrt_template_geometry(const char *name, const char *shape, khrt_dim3 *grid, khrt_dim3 *block) {
  if (grid == nullptr || block == nullptr || shape == nullptr) return bad("khrt_template_geometry: null argument");
  Plan p;
  if (int rc = plan_of(name, shape, p)) return rc;
  *grid = p.grid;
  *block = p.block;
  return 0;
}

int khrt_template_launch_symbol(const char *name, const char *shape, char *out, size_t cap) {
  if (shape == nullptr || out == nullptr || cap == 0) return bad("khrt_template_launch_symbol: null argument");
  Plan p;
  if (int rc = plan_of(name, shape, p)) return rc;  // the same shape checks as a launch
  const size_t len = std::strlen(p.symbol);
  if (len + 1 > cap) return bad("khrt_template_launch_symbol: output buffer too small");
  std::memcpy(out, p.symbol, len + 1);
  return 0;
}

int khrt_template_function(const char *name, void **function) {
  if (function == nullptr) return bad("khrt_template_function: null output");
  const Template *t = find_template(name);
  if (t == nullptr) return unknown_template(name);
  return get_function(t->co, t->name, function);
}

int khrt_gemm_candidate_count(void) { return kGemmCandidateCount; }

int khrt_gemm_candidate_get(int i, khrt_gemm_candidate *out) {
  if (out == nullptr) return bad("khrt_gemm_candidate_get: null output");
  if (i < 0 || i >= kGemmCandidateCount) {
    return khrt::fail(KHRT_E_INVALID, "khrt_gemm_candidate_get: index " + std::to_string(i) + " outside [0, " +
                                          std::to_string(kGemmCandidateCount) + ")");
  }
  const GemmCandidate &c = kGemmCandidates[i];
  *out = khrt_gemm_candidate{};
  std::snprintf(out->symbol, sizeof out->symbol, "%s", c.symbol);
  std::snprintf(out->code_object, sizeof out->code_object, "%s", c.co);
  std::snprintf(out->pipeline, sizeof out->pipeline, "%s", pipe_name(c.pipe));
  out->mfma = c.mfma;
  out->waves = c.waves();
  out->wave_grid_m = c.ksplit() ? 1 : c.wgm;
  out->wave_grid_n = c.ksplit() ? 1 : c.wgn;
  out->wave_tile_m = c.ksplit() ? c.bm() : c.mfma * c.wtm;
  out->wave_tile_n = c.ksplit() ? c.bn() : c.mfma * c.wtn;
  out->bm = c.bm();
  out->bn = c.bn();
  out->bk = c.bk;
  out->unroll = c.unroll();
  out->prio = c.prio;
  out->persistent = c.pipe == kPersistent;
  out->k_split = c.ksplit();
  out->product = c.product;
  return 0;
}

int khrt_gemm_candidate_geometry(const char *symbol, int64_t m, int64_t n, int64_t k, khrt_dim3 *grid,
                                 khrt_dim3 *block) {
  (void)k;
  if (grid == nullptr || block == nullptr) return bad("khrt_gemm_candidate_geometry: null output");
  const GemmCandidate *c = find_gemm_candidate(symbol);
  if (c == nullptr) {
    return khrt::fail(KHRT_E_INVALID, std::string("unknown GEMM candidate '") + (symbol ? symbol : "(null)") + "'");
  }
  if (m <= 0 || n <= 0 || k <= 0) return bad("khrt_gemm_candidate_geometry: m, n and k must be positive");
  *grid = khrt_dim3{clamp_grid(candidate_grid(*c, m, n)), 1, 1};
  *block = khrt_dim3{static_cast<unsigned>(64 * c->waves()), 1, 1};
  return 0;
}

int khrt_gemm_candidate_function(const char *symbol, void **function) {
  if (function == nullptr) return bad("khrt_gemm_candidate_function: null output");
  const GemmCandidate *c = find_gemm_candidate(symbol);
  if (c == nullptr) {
    return khrt::fail(KHRT_E_INVALID, std::string("unknown GEMM candidate '") + (symbol ? symbol : "(null)") + "'");
  }
  return get_function(c->co, c->symbol, function);
}

int khrt_set_tune_cache(const char *path) {
  std::lock_guard<std::mutex> lock(g_tune.mu);
  g_tune.configured = true;
  g_tune.path = path != nullptr ? path : "";
  g_tune.loaded = false;
  return 0;
}

int khrt_tune_cache_key(const char *kernel, const char *shape, char *out, size_t cap) {
  if (kernel == nullptr || shape == nullptr || out == nullptr) return bad("khrt_tune_cache_key: null argument");
  if (cap < 17) return bad("khrt_tune_cache_key: output buffer too small (17 bytes needed)");
  const std::string dev = device_token();
  if (dev.empty()) return khrt::fail(KHRT_E_INVALID, "khrt_tune_cache_key: no device");
  const std::string key = fnv1a_hex(std::string(kernel) + "|" + shape + "|" + dev);
  std::memcpy(out, key.c_str(), 17);
  return 0;
}

int khrt_device_token(char *out, size_t cap) {
  if (out == nullptr || cap == 0) return bad("khrt_device_token: null output");
  const std::string dev = device_token();
  if (dev.empty()) return khrt::fail(KHRT_E_INVALID, "khrt_device_token: no device");
  if (dev.size() + 1 > cap) return bad("khrt_device_token: output buffer too small");
  std::memcpy(out, dev.c_str(), dev.size() + 1);
  return 0;
}

int khrt_fill_f32(void *dst, float value, size_t count, void *stream) {
  if (count == 0) return 0;
  if (dst == nullptr) return bad("khrt_fill_f32: null destination");
  void *fn = nullptr;
  if (int rc = get_function("util", "kh_fill_f32", &fn)) return rc;
  khrt::LaunchArgs a;
  a.add_memref(dst, {static_cast<int64_t>(count)});
  a.add_scalar_bytes(&value, sizeof(value));
  const unsigned grid = clamp_grid(ceil_div(static_cast<int64_t>(count), 256 * 4));
  return khrt_launch_raw(fn, khrt_dim3{grid, 1, 1}, khrt_dim3{256, 1, 1}, 0, stream, a.params());
}

int kh_vecadd(const float *a, const float *b, float *c, int64_t n, void *stream) {
  if (n <= 0) return bad("vecadd: n must be positive");
  if (!a || !b || !c) return bad("vecadd: null buffer");
  StackArgs args;
  args.add_memref(a, {n});
  args.add_memref(b, {n});
  args.add_memref(c, {n});
  return launch_template(kVecadd, args, {n}, stream);
}

int kh_fused_gelu(const float *x, float *tmp, float *out, int64_t n, void *stream) {
  if (n <= 0) return bad("fused_gelu: n must be positive");
  if (!x || !out) return bad("fused_gelu: null buffer");
  StackArgs args;
  args.add_memref(x, {n});
  args.add_memref(tmp, {n});
  args.add_memref(out, {n});
  return launch_template(kFusedGelu, args, {n}, stream);
}

int kh_softmax(const float *x, float *y, int64_t rows, int64_t cols, void *stream) {
  if (rows <= 0 || cols <= 0) return bad("softmax: rows and cols must be positive");
  if (!x || !y) return bad("softmax: null buffer");
  StackArgs args;
  args.add_memref(x, {rows, cols});
  args.add_memref(y, {rows, cols});
  return launch_template(kSoftmax, args, {rows, cols}, stream);
}

int kh_layernorm(const float *x, const float *gamma, const float *beta, float *y, int64_t rows, int64_t cols,
                 void *stream) {
  if (rows <= 0 || cols <= 0) return bad("layernorm: rows and cols must be positive");
  if (!x || !gamma || !beta || !y) return bad("layernorm: null buffer");
  StackArgs args;
  args.add_memref(x, {rows, cols});
  args.add_memref(gamma, {cols});
  args.add_memref(beta, {cols});
  args.add_memref(y, {rows, cols});
  return launch_template(kLayernorm, args, {rows, cols}, stream);
}

int kh_scan(const float *x, float *y, float *y_lo, float *totals_hi, float *totals_lo, int64_t n, void *stream) {
  if (n <= 0) return bad("scan: n must be positive");
  if (!x || !y || !totals_hi || !totals_lo) return bad("scan: null buffer");
  // The look-back state (in totals_lo a 32-byte header and 16 bytes of
  // ticket counters, 256 B past it when there is room; in totals_hi 16 B
  // per tile but the last) always fits the reference's T = ceil(n/256)
  // floats of each;
  // the kernel establishes it on first use and keeps it valid across calls.
  const int64_t T = ceil_div(n, 256);
  StackArgs args;
  args.add_memref(x, {n});
  args.add_memref(y, {n});
  args.add_memref(y_lo, {n});
  args.add_memref(totals_hi, {T});
  args.add_memref(totals_lo, {T});
  return launch_template(kScan, args, {n}, stream);
}

int kh_scan_totals(const float *totals_hi, const float *totals_lo, float *off_hi, float *off_lo, float *off_lo2,
                   float *y, float *y_lo, int64_t n, void *stream) {
  if (n <= 0) return bad("scan_totals: n must be positive");
  if (!totals_hi || !totals_lo || !off_hi || !off_lo || !off_lo2 || !y) return bad("scan_totals: null buffer");
  const int64_t T = ceil_div(n, 256);
  StackArgs args;
  args.add_memref(totals_hi, {T});
  args.add_memref(totals_lo, {T});
  args.add_memref(off_hi, {T});
  args.add_memref(off_lo, {T});
  args.add_memref(off_lo2, {T});
  args.add_memref(y, {n});
  args.add_memref(y_lo, {n});
  return launch_template(kScanTotals, args, {n}, stream);
}

int kh_gemm(const float *A, const float *B, float *C, int64_t m, int64_t n, int64_t k, void *stream) {
  if (m <= 0 || n <= 0 || k <= 0) return bad("gemm: m, n and k must be positive");
  if (!A || !B || !C) return bad("gemm: null buffer");
  StackArgs args;
  args.add_memref(A, {m, k});
  args.add_memref(B, {k, n});
  args.add_memref(C, {m, n});
  return launch_template(kGemm, args, {m, n, k}, stream);
}

int kh_attention(const float *Q, const float *K, const float *V, float *O, int64_t batch, int64_t heads, int64_t seq,
                 int64_t head_dim, void *stream) {
  if (batch <= 0 || heads <= 0 || seq <= 0 || head_dim <= 0) return bad("attention: all extents must be positive");
  if (!Q || !K || !V || !O) return bad("attention: null buffer");
  if (heads > 65535 || batch > 65535) return bad("attention: heads and batch must be <= 65535 (grid y/z)");
  StackArgs args;
  args.add_memref(Q, {batch, heads, seq, head_dim});
  args.add_memref(K, {batch, heads, seq, head_dim});
  args.add_memref(V, {batch, heads, seq, head_dim});
  args.add_memref(O, {batch, heads, seq, head_dim});
  return launch_template(kAttention, args, {batch, heads, seq, head_dim}, stream);
}

// Streaming roofline kernels: 32 workgroups of 256 per CU, grid-strided.
static int launch_stream_roofline(const char *symbol, khrt::LaunchArgs &args, void *stream) {
  void *fn = nullptr;
  if (int rc = get_function("roofline", symbol, &fn)) return rc;
  khrt_device_limits live;
  if (int rc = khrt_live_limits(&live)) return rc;
  const unsigned grid = static_cast<unsigned>(std::max<int64_t>(1, live.cu_count) * 32);
  return khrt::verified_launch(fn, khrt_dim3{grid, 1, 1}, khrt_dim3{256, 1, 1}, 0, stream, args.params(), args.count());
}

static bool vec_ok(const void *p, int64_t n) {
  return (reinterpret_cast<uintptr_t>(p) & 15u) == 0 && n > 0 && (n & 3) == 0;
}

int kh_roofline_triad(const float *a, const float *b, float *c, int64_t n, void *stream) {
  if (!a || !b || !c) return bad("roofline_triad: null buffer");
  if (!vec_ok(a, n) || !vec_ok(b, n) || !vec_ok(c, n)) return bad("roofline_triad: n % 4 == 0 and 16-byte alignment required");
  khrt::LaunchArgs args;
  args.add_memref(a, {n});
  args.add_memref(b, {n});
  args.add_memref(c, {n});
  return launch_stream_roofline("roofline_triad", args, stream);
}

int kh_roofline_copy(const float *src, float *dst, int64_t n, void *stream) {
  if (!src || !dst) return bad("roofline_copy: null buffer");
  if (!vec_ok(src, n) || !vec_ok(dst, n)) return bad("roofline_copy: n % 4 == 0 and 16-byte alignment required");
  khrt::LaunchArgs args;
  args.add_memref(src, {n});
  args.add_memref(dst, {n});
  return launch_stream_roofline("roofline_copy", args, stream);
}

int kh_roofline_mfma(float *out, int64_t blocks, int64_t iters, void *stream) {
  if (!out) return bad("roofline_mfma: null buffer");
  if (blocks <= 0 || blocks > (1 << 20) || iters <= 0) return bad("roofline_mfma: blocks in [1, 2^20], iters > 0");
  void *fn = nullptr;
  if (int rc = get_function("roofline", "roofline_mfma", &fn)) return rc;
  khrt::LaunchArgs args;
  args.add_memref(out, {blocks * 256});
  args.add_scalar_bytes(&iters, sizeof(iters));
  return khrt::verified_launch(fn, khrt_dim3{static_cast<unsigned>(blocks), 1, 1}, khrt_dim3{256, 1, 1}, 0, stream,
                               args.params(), args.count());
}

}  // extern "C"
