// zm_api.hip -- host side of libzeromoe_hip.so: the C ABI declared in
// include/zeromoe.h, argument validation, template dispatch and the per-device
// tables.  Everything below launches stream-ordered HIP work.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>

#include "../../include/zeromoe.h"
#include "zm_decode.hpp"
#include "zm_host.hpp"
#include "zm_mmq.hpp"

using namespace zm;

namespace {
thread_local char g_err[512] = "";
std::atomic<uint64_t> g_mmid_launches{0};
}  // namespace

int zm::fail(const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return -1;
}
void zm::count_mmid_launch() { g_mmid_launches.fetch_add(1, std::memory_order_relaxed); }

namespace {

// ------------------------------------------------------------------ per-device state

constexpr int kMaxDevices = 16;

// Device-resident scratch of zm_mul_mat_id_static: one copy per GPU, held until
// the process ends.  Host code never passes `scratch` itself to a kernel (on the
// host the name is only a stand-in): its per-device address comes from
// hipGetSymbolAddress at set-up (DeviceState::scratch).
constexpr size_t kStaticScratchBytes = 16u << 20;
static __device__ __align__(256) uint8_t scratch[kStaticScratchBytes];

struct DeviceState {
  bool ready = false;
  uint64_t *grid = nullptr;   // IQ2_XXS grid, 256 x u64
  uint64_t *signs = nullptr;  // 128 x u64 byte masks of ksigns_iq2xs
  uint64_t *iq4 = nullptr;    // IQ4_XS value table, 16 x i8
  uint64_t *iq3 = nullptr;    // IQ3_XXS grid, 256 x u32
  uint8_t *scratch = nullptr; // this device's address of `scratch`
  uint64_t *trace = nullptr;  // decode-kernel phase timestamps (ZEROMOE_TRACE=1)
  size_t trace_n = 0;
  int n_cu = 0;               // compute units
  int cus() const { return n_cu > 0 ? n_cu : 256; }
  // a dense shared expert runs beside the routed kernels of a multi-kernel
  // layer (SideBranch; default priority, and the fork and join record into a
  // HIP graph like any other stream work)
  hipStream_t side = nullptr;
  hipEvent_t ev_fork = nullptr, ev_join = nullptr;
  std::mutex *fork_mu = nullptr;  // the events are per device: one fork at a time
};
DeviceState g_dev[kMaxDevices];
std::mutex g_mu;

void builtin_grid(uint64_t grid[256]) {
  // the 256 vectors of {1,3,5}^8 with an even digit sum ((v-1)/2 summed) of
  // smallest norm, lexicographic (coordinate 0 most significant) on ties;
  // coordinate bytes 1 -> 0x08, 3 -> 0x19, 5 -> 0x2b
  static const uint8_t bytev[3] = {0x08, 0x19, 0x2b};
  int count = 0;
  for (int norm = 0; norm < 200 && count < 256; ++norm)
    for (int idx = 0; idx < 6561 && count < 256; ++idx) {
      int t = idx, dig[8], sd = 0, nn = 0;
      for (int j = 7; j >= 0; --j) {
        dig[j] = t % 3;
        t /= 3;
      }
      for (int j = 0; j < 8; ++j) {
        sd += dig[j];
        nn += (1 + 2 * dig[j]) * (1 + 2 * dig[j]);
      }
      if ((sd & 1) || nn != norm) continue;
      uint64_t g = 0;
      for (int j = 0; j < 8; ++j) g |= (uint64_t)bytev[dig[j]] << (8 * j);
      grid[count++] = g;
    }
}

// ggml's kvalues_iq4nl (the table IQ4_NL / IQ4_XS index); replaceable with
// zm_set_iq4nl_table
void builtin_iq4nl(int8_t t[16]) {
  static const int8_t v[16] = {-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113};
  for (int i = 0; i < 16; ++i) t[i] = v[i];
}

// stand-in IQ3_XXS grid: the 256 vectors of four 3-bit digits d with
// d0 + 2 d1 + 4 d2 + 8 d3 = 0 mod 16, in increasing order of the digit
// vector read as a base-8 number, digit d stored as the byte 4 + 8 d (62 for
// 7); ggml's own table is loaded with zm_set_iq3xxs_grid
void builtin_iq3_grid(uint32_t g[256]) {
  static const uint8_t lev[8] = {4, 12, 20, 28, 36, 44, 52, 62};
  int n = 0;
  for (int v = 0; v < 4096 && n < 256; ++v) {
    const int d0 = v & 7, d1 = (v >> 3) & 7, d2 = (v >> 6) & 7, d3 = (v >> 9) & 7;
    if ((d0 + 2 * d1 + 4 * d2 + 8 * d3) % 16) continue;
    g[n++] = (uint32_t)lev[d0] | ((uint32_t)lev[d1] << 8) | ((uint32_t)lev[d2] << 16) | ((uint32_t)lev[d3] << 24);
  }
}

int device_state(DeviceState **out) {
  int dev = 0;
  HIP_OK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return fail("device %d out of range", dev);
  std::lock_guard<std::mutex> lk(g_mu);
  DeviceState &d = g_dev[dev];
  if (!d.ready) {
    HIP_OK(hipDeviceGetAttribute(&d.n_cu, hipDeviceAttributeMultiprocessorCount, dev));
    HIP_OK(hipStreamCreateWithFlags(&d.side, hipStreamNonBlocking));
    HIP_OK(hipEventCreateWithFlags(&d.ev_fork, hipEventDisableTiming));
    HIP_OK(hipEventCreateWithFlags(&d.ev_join, hipEventDisableTiming));
    d.fork_mu = new std::mutex();
    uint64_t grid[256], signs[128];
    builtin_grid(grid);
    for (int i = 0; i < 128; ++i) {
      const int s = i | ((__builtin_popcount(i) & 1) << 7);  // ksigns_iq2xs
      uint64_t m = 0;
      for (int j = 0; j < 8; ++j)
        if ((s >> j) & 1) m |= 0xffull << (8 * j);
      signs[i] = m;
    }
    HIP_OK(hipMalloc(&d.grid, sizeof(grid)));
    HIP_OK(hipMalloc(&d.signs, sizeof(signs)));
    HIP_OK(hipMemcpy(d.grid, grid, sizeof(grid), hipMemcpyHostToDevice));
    HIP_OK(hipMemcpy(d.signs, signs, sizeof(signs), hipMemcpyHostToDevice));
    int8_t tab[16];
    builtin_iq4nl(tab);
    HIP_OK(hipMalloc(&d.iq4, 16));
    HIP_OK(hipMemcpy(d.iq4, tab, 16, hipMemcpyHostToDevice));
    uint32_t g3[256];
    builtin_iq3_grid(g3);
    HIP_OK(hipMalloc(&d.iq3, sizeof(g3)));
    HIP_OK(hipMemcpy(d.iq3, g3, sizeof(g3), hipMemcpyHostToDevice));
    void *sp = nullptr;
    HIP_OK(hipGetSymbolAddress(&sp, HIP_SYMBOL(scratch)));
    d.scratch = (uint8_t *)sp;
    d.ready = true;
  }
  *out = &d;
  return 0;
}

// The state of the current device if zm_init (or any first call) has set it
// up; nullptr otherwise.  Allocates nothing.
DeviceState *device_state_if_ready() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lk(g_mu);
  return g_dev[dev].ready ? &g_dev[dev] : nullptr;
}

}  // namespace

int zm::device_grid(const uint64_t **grid) {
  DeviceState *d;
  if (device_state(&d)) return -1;
  *grid = d->grid;
  return 0;
}

int zm::device_table(int type, const uint64_t **table) {
  DeviceState *d;
  if (device_state(&d)) return -1;
  *table = type == T_IQ4_XS ? d->iq4 : (type == T_IQ3_XXS ? d->iq3 : d->grid);
  return 0;
}

namespace {

// ------------------------------------------------------------------ GEMV dispatch

template <int T, int LPR, int ITER, int NP, bool GU>
void launch_gemv_t(dim3 grid, const GemvArgs &a, hipStream_t st) {
  hipLaunchKernelGGL((k_gemv<T, LPR, ITER, NP, GU>), grid, dim3(256), 0, st, a);
}

template <int T, int NP, bool GU>
int launch_gemv_np(int U, dim3 grid, const GemvArgs &a, hipStream_t st) {
  if (U <= 16) launch_gemv_t<T, 16, 1, NP, GU>(grid, a, st);
  else if (U <= 32) launch_gemv_t<T, 32, 1, NP, GU>(grid, a, st);
  else if (U <= 64) launch_gemv_t<T, 64, 1, NP, GU>(grid, a, st);
  else if (U <= 128) launch_gemv_t<T, 64, 2, NP, GU>(grid, a, st);
  else if (U <= 192) launch_gemv_t<T, 64, 3, NP, GU>(grid, a, st);
  else if (U <= 256) launch_gemv_t<T, 64, 4, NP, GU>(grid, a, st);
  else return fail("row of %d blocks exceeds the 64-block limit", U / 4);
  return 0;
}

template <int T, bool GU>
int launch_gemv_type(int np, int U, dim3 grid, const GemvArgs &a, hipStream_t st) {
  if (np >= 4) return launch_gemv_np<T, 4, GU>(U, grid, a, st);
  if (np >= 2) return launch_gemv_np<T, 2, GU>(U, grid, a, st);
  return launch_gemv_np<T, 1, GU>(U, grid, a, st);
}

// true when the environment variable is set to "0" (switches a path off for testing)
bool getenv_flag_off(const char *name) {
  const char *e = getenv(name);
  return e && e[0] == '0';
}

bool type_supported(int t) {
  return t == T_Q2_K || t == T_Q3_K || t == T_Q4_K || t == T_Q5_K || t == T_Q6_K || t == T_IQ2_XXS || t == T_IQ3_XXS ||
         t == T_IQ4_XS;
}

size_t row_bytes(int t, int64_t n) { return (size_t)(n / QK) * block_bytes(t); }

// pairs per bucket chunk held in registers
int pick_np(int n_pairs, int n_experts) {
  const int act = std::max(1, std::min(n_pairs, n_experts));
  const double avg = (double)n_pairs / act;
  return avg >= 3.0 ? 4 : (avg >= 1.5 ? 2 : 1);
}

// rows per workgroup: enough workgroups to cover the chip several times over
int pick_tile(int nrows, int U, int n_groups) {
  const int lpr = U <= 16 ? 16 : (U <= 32 ? 32 : 64);
  const int step = 4 * (64 / lpr);  // rows one workgroup covers per step
  const int target_wgs = 2048;
  const int tiles = std::max(1, target_wgs / std::max(1, n_groups));
  int tile = (nrows + tiles - 1) / tiles;
  tile = ((tile + step - 1) / step) * step;
  return std::max(step, tile);
}

int launch_gemv(int type, bool gateup, int np, const GemvArgs &a0, int n_groups, hipStream_t st) {
  GemvArgs a = a0;
  if ((type == T_IQ4_XS || type == T_IQ3_XXS) && device_table(type, &a.grid)) return -1;
  const int U = a.nb * 4;
  a.tile_rows = pick_tile(a.nrows, U, n_groups);
  dim3 grid((a.nrows + a.tile_rows - 1) / a.tile_rows, n_groups);
  int rc;
  switch (type) {
  case T_Q2_K: rc = gateup ? launch_gemv_type<T_Q2_K, true>(np, U, grid, a, st) : launch_gemv_type<T_Q2_K, false>(np, U, grid, a, st); break;
  case T_Q3_K: rc = gateup ? launch_gemv_type<T_Q3_K, true>(np, U, grid, a, st) : launch_gemv_type<T_Q3_K, false>(np, U, grid, a, st); break;
  case T_Q4_K: rc = gateup ? launch_gemv_type<T_Q4_K, true>(np, U, grid, a, st) : launch_gemv_type<T_Q4_K, false>(np, U, grid, a, st); break;
  case T_Q5_K: rc = gateup ? launch_gemv_type<T_Q5_K, true>(np, U, grid, a, st) : launch_gemv_type<T_Q5_K, false>(np, U, grid, a, st); break;
  case T_Q6_K: rc = gateup ? launch_gemv_type<T_Q6_K, true>(np, U, grid, a, st) : launch_gemv_type<T_Q6_K, false>(np, U, grid, a, st); break;
  case T_IQ3_XXS: rc = gateup ? launch_gemv_type<T_IQ3_XXS, true>(np, U, grid, a, st) : launch_gemv_type<T_IQ3_XXS, false>(np, U, grid, a, st); break;
  case T_IQ4_XS: rc = gateup ? launch_gemv_type<T_IQ4_XS, true>(np, U, grid, a, st) : launch_gemv_type<T_IQ4_XS, false>(np, U, grid, a, st); break;
  case T_IQ2_XXS: rc = gateup ? launch_gemv_type<T_IQ2_XXS, true>(np, U, grid, a, st) : launch_gemv_type<T_IQ2_XXS, false>(np, U, grid, a, st); break;
  default: return fail("unsupported weight type %d", type);
  }
  if (rc) return rc;
  HIP_OK(hipGetLastError());
  return 0;
}

// ------------------------------------------------------------------ grouped MFMA dispatch

// 16-pair tiles per work item, by the pairs per expert: 64-pair items share the
// weight unpacking where buckets are large, 32-pair items take fewer registers
// and less LDS, 16-pair items leave LDS for two blocks of weights per stage (at
// 10 pairs per expert 3% of even loads exceed them and read their weights twice).
// One op, 1536 rows of 4096, 128 experts, us, by pairs per expert, 16- / 32- /
// 64-pair items:
//   even loads, Q4_K    8 115/117/105  12 126/120/110  20 203/134/123  28 231/163/135  32 239/190/142
//   even loads, Q3_K    8 102/114/132  12 112/118/134  20 183/130/141  28 216/157/149  32 245/180/149
//   even loads, Q6_K    8 155/204/199  12 170/201/203  20 270/246/221  28 324/277/242  32 349/329/246
//   skewed, IQ3_XXS     8  89/ 88/ 93  12 112/101/101  20 157/132/124  28 200/155/137  32 221/170/154
// 64-pair items are the faster ones from 20 (Q3_K, IQ2_XXS: 28) pairs on; they add
// all K blocks in one chain, so they are left to where they gain most.
// Where few experts or rows leave CUs idle the items are halved: 64-pair items (8
// waves on 128 rows) below one workgroup per CU, 32-pair items (4 waves on 64)
// below one, or up to two for types whose 32-pair kernels take longest per block.
// 1 expert, 64 pairs, 1536 rows of 4096, 64- / 32- / 16-pair items: Q6_K 65 / 44 /
// 22 us, Q4_K 32 / 21 / 17.  Mean ratio of 16- to 32-pair items over three shapes, by
// workgroups of the latter: Q4_K 96 0.98, 192 1.00, 256 1.01, 512 1.11; Q2_K 0.81,
// 0.90, 0.99, 1.08; Q6_K 0.47, 0.55, 0.70, 0.83; IQ2_XXS 0.68, 0.66, 0.54, 0.64;
// IQ3_XXS 0.69, 0.77, 0.88, 0.96 (32 experts of 28: 1.19).  Of 32- to 64-pair items:
// Q4_K 96 0.76, 192 0.97, 256 1.05; Q6_K 0.81, 0.89, 0.97; Q3_K and IQ2_XXS 0.9, 1.03,
// 1.46, so those types go from 64- to 16-pair items or stay.
int mmq_wgs32(int type, int cus) {  // workgroups of 32-pair items from which they are taken
  if (type == T_Q3_K || type == T_Q6_K || type == T_IQ2_XXS) return 2 * cus + 1;
  return type == T_IQ3_XXS ? 2 * cus : cus;
}
// ZEROMOE_MMQ_TILES=1, 2 or 4 sets the size for every product (tests of each kernel at each shape)
int forced_tiles() {
  const char *e = getenv("ZEROMOE_MMQ_TILES");
  return e && (e[0] == '1' || e[0] == '2' || e[0] == '4') ? e[0] - '0' : 0;
}
int mmq_tiles(double avg_pairs, int groups, int nrows, int wgs32, int cus) {
  if (const int forced = forced_tiles()) return forced;
  int tt = avg_pairs >= 32.0 ? 4 : (avg_pairs >= 10.0 ? 2 : 1);
  auto wgs = [&](int rows, int pairs) {
    return (long)((nrows + rows - 1) / rows) * groups * (long)std::ceil(avg_pairs / pairs);
  };
  const bool few32 = wgs(64, 32) < wgs32;
  if (tt == 4 && wgs(128, 64) < cus && (few32 || wgs32 <= cus)) tt = 2;
  return tt == 2 && few32 ? 1 : tt;
}
// work items of n_pairs pairs over n_experts buckets: at most one partial run
// per bucket besides the full ones
int mmq_max_items(int n_pairs, int n_experts, int tok) {
  return (n_pairs + tok - 1) / tok + std::min(n_pairs, n_experts);
}
// Whether the grouped MFMA kernel takes this product (the caller then
// quantizes the activations to records); the GEMV takes what is left.
//   - rows, activations: 32-bit buffer offsets (of rows signed, of records not);
//   - alignment: blocks of a multiple of 4 bytes are loaded by dwords, the
//     others start on 2 bytes (gate and up alike within a dword);
//   - pairs: with few of them over many experts its workgroups are too few and too
//     long.  One op over 128 experts, GEMV / this, us, by pairs (1536 rows of 4096, Q4_K):
//     8 13.1 / 21.5, 32 28.7 / 30.2, 48 40.5 / 40.5, 64 52.0 / 48.1, 128 97.1 /
//     72.1; (4096 rows of 1536, Q6_K): 8 18.3 / 19.9, 32 45.3 / 44.0, 48 64.9 /
//     57.5, 128 165.2 / 100.8.  Matrices of few blocks need more pairs, those of
//     the grid types most (kernels alone; gate/up then down, 1792 rows of 1024 and
//     1024 of 1792, 40 pairs: IQ3_XXS 21.0 / 27.2, 12.1 / 15.1, Q4_K 20.7 / 19.8,
//     Q6_K 15.5 / 16.3; 1280 of 2560 and 2560 of 1280: IQ3_XXS 46.1 / 39.4,
//     26.2 / 22.2.  Whole layer, 1024 x 1792, 64 pairs: Q4_K 69.7 / 64.5, IQ3_XXS
//     63.2 / 66.8, IQ2_XXS 57.0 / 62.8; 80: 87.5 / 73.3, 78.8 / 72.6, 64.1 / 63.6).
//     With several pairs per expert less is enough, as the GEMV reads the weights
//     once for every 4: 4 per expert and 24 in all, or 16 per expert (Q2_K: 2 and
//     16; codebook types: 8 and 32, 4 and 64, or 24).  GEMV / 16-pair items, us: 1
//     expert, 1536 rows of 4096, 8 / 16 / 39 pairs: Q4_K 13 / 17, 19 / 17, 36 / 17, Q3_K
//     15 / 19, 21 / 19, 40 / 19, IQ3_XXS 13 / 22, 18 / 22, 32 / 22 (24: 22 / 22); 8 experts
//     of 2: Q2_K 16 / 16, of 4: Q4_K 22 / 22, Q2_K 21 / 17, IQ3_XXS 20 / 23; 4096 rows of
//     1536: 17 / 14, 25 / 16, 25 / 14, 22 / 17; 16 experts of 4, IQ3_XXS 27 / 29, 32 / 24.
//     Layers of 64 tokens x 8 of 64 experts, 4 of them resident (H 4096 F 1536, Q4_K),
//     even routing / routing towards those: GEMV 80 / 287, this 44 / 54.
struct MmqLoad {
  int groups;  // experts that may have pairs
  int likely;  // pairs, of those that a slot table skips as many as even routing would have
  int held;    // pairs, of those that a slot table skips half as many (resident experts are the sought ones)
};
bool mmq_enough(const MmqLoad &n, int type, int nrows, int nb) {
  const bool grid = type == T_IQ2_XXS || type == T_IQ3_XXS, codebook = grid || type == T_IQ4_XS;
  const int many = (size_t)nrows * nb >= 10000 ? 40 : (grid ? 80 : 64);
  const long g = n.groups;
  const long per = type == T_Q2_K ? 2 : (codebook && n.held < 64 ? 8 : 4), least = type == T_Q2_K ? 16 : (codebook ? 32 : 24);
  return n.likely >= many || n.held >= (codebook ? 24 : 16) * g || (n.held >= least && n.held >= per * g);
}
// load null: the caller has found the pairs to be enough
bool mmq_applies(int type, const void *w0, const void *w1, size_t w_estride, int nrows, size_t w_rstride,
                 const MmqLoad *load, size_t xq_rows, int nb) {
  if ((load && !mmq_enough(*load, type, nrows, nb)) || getenv_flag_off("ZEROMOE_MMQ")) return false;
  if ((size_t)nrows * w_rstride >= (1ull << 31) - 4 || xq_rows * xrec_row_bytes(nb) > XREC_MAX_BYTES) return false;
  const uintptr_t lo = (uintptr_t)w0 | (w1 ? (uintptr_t)w1 : 0) | w_estride;
  if (lo & (block_bytes(type) % 4 ? 1 : 3)) return false;
  return !w1 || !(((uintptr_t)w0 ^ (uintptr_t)w1) & 3);
}
// tt: 16-pair tiles per item (the list's); items: bound of *a.n_items (or the
// exact count of a dense product); nw = 1: one-wave workgroups (tt == 2 only)
int launch_mmq(int type, bool gateup, int tt, int nw, int items, const GemvArgs &a0, hipStream_t st) {
  GemvArgs a = a0;
  if ((type == T_IQ4_XS || type == T_IQ3_XXS || type == T_IQ2_XXS) && device_table(type, &a.grid)) return -1;
  const unsigned n = (unsigned)items;
  if (!mmq_launch_a(type, gateup, tt, nw, n, a, st) && !mmq_launch_b(type, gateup, tt, nw, n, a, st) &&
      !mmq_launch_c(type, gateup, tt, nw, n, a, st) && !mmq_launch_d(type, gateup, tt, nw, n, a, st))
    return fail("unsupported weight type %d", type);
  HIP_OK(hipGetLastError());
  return 0;
}
// sort the pairs (b), quantize the rows of x, write the rows of skipped routes (a.out): one launch
int launch_prep(PrepArgs a, hipStream_t st, bool sort = true) {
  a.sort_wgs = sort ? 1 : 0;
  const long blocks = (long)a.rows * a.nb;
  a.q_wgs = (int)((blocks + PREP_QBLOCKS - 1) / PREP_QBLOCKS);
  const int f_wgs = a.out ? (a.b.n_pairs + PREP_FPAIRS - 1) / PREP_FPAIRS : 0;
  hipLaunchKernelGGL(k_prep, dim3(a.sort_wgs + a.q_wgs + f_wgs), dim3(1024), 0, st, a);
  HIP_OK(hipGetLastError());
  return 0;
}

// records for the grouped MFMA kernel, value order of `type`
int launch_quant_rec(const float *x, size_t x_rstride, int nb, int rows, uint8_t *y, int type, hipStream_t st) {
  if (rows <= 0) return 0;
  const long blocks = (long)rows * nb;  // 16 per workgroup
  hipLaunchKernelGGL(k_quant_rec, dim3((unsigned)((blocks + 15) / 16)), dim3(256), 0, st, x, x_rstride, nb, rows, y,
                     xrec_row_bytes(nb), mmq_order(type));
  HIP_OK(hipGetLastError());
  return 0;
}
int launch_quant(const float *x, size_t x_rstride, int nb, int rows, uint8_t *y, size_t y_rstride, int planar,
                 hipStream_t st) {
  if (rows <= 0) return 0;
  const long blocks = (long)rows * nb;  // 16 per workgroup
  hipLaunchKernelGGL(k_quant_q8K, dim3((unsigned)((blocks + 15) / 16)), dim3(256), 0, st, x, x_rstride, nb, rows, y,
                     y_rstride, planar);
  HIP_OK(hipGetLastError());
  return 0;
}

// Work on the device's side stream beside the caller's stream `st`.  Whatever
// way the scope of an open branch is left, `st` waits for what it has launched:
// the side stream reads and writes the caller's buffers.
struct SideBranch {
  DeviceState *d;
  hipStream_t st;
  std::unique_lock<std::mutex> lk;
  bool open = false, ended = false;
  SideBranch(DeviceState *dev, hipStream_t s) : d(dev), st(s) {}
  SideBranch(const SideBranch &) = delete;
  int fork() {
    lk = std::unique_lock<std::mutex>(*d->fork_mu);
    HIP_OK(hipEventRecord(d->ev_fork, st));
    HIP_OK(hipStreamWaitEvent(d->side, d->ev_fork, 0));
    open = true;
    return 0;
  }
  // the branch's last launch is made: recorded here, behind it, and not at the join
  // (8 to 14 us of host time per layer call there)
  int end() {
    ended = true;
    HIP_OK(hipEventRecord(d->ev_join, d->side));
    return 0;
  }
  int join() {
    open = false;
    HIP_OK(hipStreamWaitEvent(st, d->ev_join, 0));
    return 0;
  }
  ~SideBranch() {
    if (!open) return;
    char why[sizeof(g_err)];  // the failure that ends the call, not one of this join
    memcpy(why, g_err, sizeof(why));
    if (ended || !end()) (void)join();
    memcpy(g_err, why, sizeof(why));
  }
};

// simple bump allocator over a caller workspace
struct Bump {
  uint8_t *base;
  size_t off = 0;
  template <class P>
  P *take(size_t bytes) {
    off = (off + 255) & ~(size_t)255;
    P *p = reinterpret_cast<P *>(base ? base + off : nullptr);
    off += bytes;
    return p;
  }
};

// what k_router takes
int check_router(const zm_router_spec &spec) {
  if (spec.n_experts <= 0 || spec.n_experts > ROUTER_MAX_E) return fail("zm_router: n_experts out of range");
  if (spec.topk <= 0 || spec.topk > spec.n_experts || spec.topk > 64) return fail("zm_router: bad topk");
  if (spec.n_groups > 64) return fail("zm_router: n_groups > 64");
  if (spec.gating < 0 || spec.gating > 2) return fail("zm_router: bad gating");
  return 0;
}

}  // namespace

// ====================================================================== C ABI

extern "C" {

const char *zm_last_error(void) { return g_err; }
const char *zm_version(void) { return "zeromoe_amd 0.1 (gfx950)"; }

int zm_init(void) {
  DeviceState *d;
  return device_state(&d);
}

void zm_iq2xxs_builtin_grid(uint64_t grid[256]) { builtin_grid(grid); }

int zm_set_iq2xxs_grid(const uint64_t grid[256]) {
  DeviceState *d;
  if (device_state(&d)) return -1;
  HIP_OK(hipMemcpy(d->grid, grid, 256 * sizeof(uint64_t), hipMemcpyHostToDevice));
  return 0;
}

void zm_iq4nl_builtin_table(int8_t table[16]) { builtin_iq4nl(table); }

void zm_iq3xxs_builtin_grid(uint32_t grid[256]) { builtin_iq3_grid(grid); }

int zm_set_iq3xxs_grid(const uint32_t grid[256]) {
  DeviceState *d;
  if (device_state(&d)) return -1;
  HIP_OK(hipMemcpy(d->iq3, grid, 256 * sizeof(uint32_t), hipMemcpyHostToDevice));
  return 0;
}

int zm_set_iq4nl_table(const int8_t table[16]) {
  DeviceState *d;
  if (device_state(&d)) return -1;
  HIP_OK(hipMemcpy(d->iq4, table, 16, hipMemcpyHostToDevice));
  return 0;
}

int zm_mul_mat_id_negative_skip(void) { return 1; }
int zm_mul_mat_id_negative_skip_batched(void) { return 1; }
uint64_t zm_mul_mat_id_launches(void) { return g_mmid_launches.load(std::memory_order_relaxed); }

int zm_quantize_q8_K(const float *x, int64_t rows, int64_t n, void *y, void *stream) {
  if (!x || !y || rows < 0 || n <= 0 || n % QK) return fail("zm_quantize_q8_K: bad arguments");
  return launch_quant(x, (size_t)n, (int)(n / QK), (int)rows, (uint8_t *)y, (size_t)(n / QK) * 292, 0,
                      (hipStream_t)stream);
}

int zm_router(const zm_router_spec *spec, const float *logits, const float *logit_bias, const float *sel_bias,
              const int32_t *route_map, const float *route_mask, int S, int32_t *ids, float *weights,
              void *stream) {
  if (!spec || !logits || !ids || !weights || S < 0) return fail("zm_router: null argument");
  if (check_router(*spec)) return -1;
  if (S == 0) return 0;
  RouterArgs a{logits, logit_bias, sel_bias, route_map, route_mask, spec->n_experts, spec->topk, spec->gating,
               spec->n_groups, spec->n_groups_used, spec->weights_norm, spec->weights_scale, ids, weights};
  hipLaunchKernelGGL(k_router, dim3((S + 3) / 4), dim3(256), 0, (hipStream_t)stream, a, S);
  HIP_OK(hipGetLastError());
  return 0;
}

int zm_bucket(const int32_t *ids, int S, int K, int E, int32_t *counts, int32_t *offs, int32_t *pairs,
              int32_t *active, int32_t *n_active, void *stream) {
  if (!ids || !counts || !offs || !pairs || !active || !n_active) return fail("zm_bucket: null argument");
  if (E <= 0 || E > BUCKET_MAX_E) return fail("zm_bucket: E out of range (1..%d)", BUCKET_MAX_E);
  if (S < 0 || K <= 0) return fail("zm_bucket: bad S/K");
  const BucketArgs a{ids, (size_t)K, K, S * K, E, counts, offs, pairs, active, n_active, nullptr, nullptr, 0};
  hipLaunchKernelGGL(k_bucket, dim3(1), dim3(1024), 0, (hipStream_t)stream, a);
  HIP_OK(hipGetLastError());
  return 0;
}

// ---------------------------------------------------------------- mul_mat_id hook

}  // extern "C"

namespace {

// A validated MUL_MAT_ID shape (see zm_mul_mat_id's rules) and the workspace
// for it: rows of src1, the bucket arrays and the MFMA work list.
struct MmidShape {
  int64_t I, O, E, n_ids, S, ne11, n_pairs, nq;
  int nb;
  size_t ws_bytes;  // holds the records of every token
  size_t ws_least;  // what the shape is accepted with
};

struct MmidWs {
  uint8_t *xq;
  int32_t *idc, *counts, *offs, *pairs, *active, *n_active, *items, *n_items;
};

// rec: src1 as records and a work list (grouped MFMA kernel), else planar rows
// (GEMV); idc: room for a copy of the ids
size_t mmid_carve(const MmidShape &m, bool rec, bool idc, uint8_t *base, MmidWs *out) {
  Bump b{base};
  MmidWs w{};
  w.xq = b.take<uint8_t>((size_t)m.nq * (rec ? xrec_row_bytes(m.nb) : q8_row_bytes(m.nb)));
  if (idc) w.idc = b.take<int32_t>((size_t)m.n_pairs * 4);
  w.counts = b.take<int32_t>((size_t)m.E * 4);
  w.offs = b.take<int32_t>((size_t)(m.E + 1) * 4);
  w.pairs = b.take<int32_t>((size_t)m.n_pairs * 4);
  w.active = b.take<int32_t>((size_t)m.E * 4);
  w.n_active = b.take<int32_t>(4);
  if (rec) {
    w.items = b.take<int32_t>((size_t)mmq_max_items((int)m.n_pairs, (int)m.E, 16) * 4);
    w.n_items = b.take<int32_t>(4);
  }
  if (out) *out = w;
  return b.off + 256;
}

// The size from which a workspace is accepted, whatever the kernels in use
// would like: callers with a workspace of a fixed size (and of the static
// scratch array) keep the shapes they have.  Q8_K rows, a copy of the ids and a
// list of 32-pair items; every layout but that of records fits it, and of
// records at least half the tokens.
size_t mmid_least(const MmidShape &m) {
  MmidWs w;
  Bump b{nullptr, mmid_carve(m, false, true, nullptr, &w) - 256};
  b.take<int32_t>((size_t)mmq_max_items((int)m.n_pairs, (int)m.E, 32) * 4);
  b.take<int32_t>(4);
  return b.off + 256;
}

// The validation rules of the reference hook (kquant_matmul.cu:705-722) plus
// this kernel set's limits; false = decline.
bool mmid_shape(const zm_tensor *w, const zm_tensor *x, const zm_tensor *ids, const zm_tensor *y, MmidShape *m) {
  if (!w || !x || !ids || !y) return false;
  if (!type_supported(w->type) || x->type != T_F32 || y->type != T_F32 || ids->type != T_I32) return false;
  const int64_t I = w->ne[0], O = w->ne[1], E = w->ne[2];
  if (I <= 0 || I % QK || I / QK > 64 || O <= 0 || O > INT32_MAX || E <= 0 || E > BUCKET_MAX_E || w->ne[3] != 1)
    return false;
  if (w->nb[1] != row_bytes(w->type, I) || w->nb[2] < (size_t)O * w->nb[1]) return false;
  const int64_t n_ids = ids->ne[0], S = ids->ne[1];
  if (ids->nb[0] != 4 || n_ids <= 0 || S <= 0 || ids->ne[2] != 1 || ids->ne[3] != 1) return false;
  if (x->nb[0] != 4 || x->ne[0] != I || (x->ne[1] != 1 && x->ne[1] != n_ids) || x->ne[2] != S || x->ne[3] != 1)
    return false;
  if (x->nb[1] % 16 || x->nb[2] % 16 || ((uintptr_t)x->data & 15)) return false;  // float4 row loads
  if (y->nb[0] != 4 || y->ne[0] != O || y->ne[1] != n_ids || y->ne[2] != S || y->ne[3] != 1) return false;
  if (y->nb[1] % 4 || y->nb[2] % 4 || ids->nb[1] % 4) return false;
  const int64_t n_pairs = n_ids * S;
  if (n_pairs > MMQ_MAX_PAIRS) return false;
  m->I = I;
  m->O = O;
  m->E = E;
  m->n_ids = n_ids;
  m->S = S;
  m->ne11 = x->ne[1];
  m->n_pairs = n_pairs;
  m->nq = m->ne11 * S;
  m->nb = (int)(I / QK);
  m->ws_least = mmid_least(*m);
  m->ws_bytes = std::max(mmid_carve(*m, true, false, nullptr, nullptr), m->ws_least);
  return true;
}

// Whether the extents of two F32 / I32 tensors share a byte.
bool tensors_overlap(const zm_tensor *a, const zm_tensor *b) {
  auto end = [](const zm_tensor *t) {
    size_t n = 4;
    for (int i = 0; i < 4; ++i) n += (size_t)(t->ne[i] - 1) * t->nb[i];
    return (uintptr_t)t->data + n;
  };
  return (uintptr_t)a->data < end(b) && (uintptr_t)b->data < end(a);
}

// The op on a workspace of `cap` >= m.ws_least bytes (256-byte aligned);
// launches only, stream-ordered, allocates nothing.  Returns 1 handled / 0 failed.
int mmid_exec(const MmidShape &m, const zm_tensor *w, const zm_tensor *x, const zm_tensor *ids, zm_tensor *y,
              hipStream_t st, uint8_t *ws, size_t cap, const DeviceState *d) {
  const int nb = m.nb;
  const int ne11 = (int)m.ne11;
  const int64_t n_ids = m.n_ids, n_pairs = m.n_pairs, nq = m.nq, E = m.E, O = m.O;
  const int groups = (int)std::min<int64_t>(E, n_pairs);
  const MmqLoad load{groups, (int)n_pairs, (int)n_pairs};
  bool mmq = mmq_applies(w->type, w->data, nullptr, w->nb[2], (int)O, w->nb[1], &load, (size_t)nq, nb);
  // dst may lie over src1 or ids: then both are taken in before a row is written
  const bool apart = !tensors_overlap(y, x) && !tensors_overlap(y, ids);
  if (mmq && mmid_carve(m, true, !apart, nullptr, nullptr) > cap) {
    // records for half the tokens at a time
    if (m.S == 1 || !apart) {
      mmq = false;
    } else {
      const int64_t cut[3] = {0, m.S / 2, m.S};
      for (int i = 0; i < 2; ++i) {
        zm_tensor xh = *x, ih = *ids, yh = *y;
        MmidShape h = m;
        h.S = xh.ne[2] = ih.ne[1] = yh.ne[2] = cut[i + 1] - cut[i];
        h.n_pairs = h.S * n_ids;
        h.nq = h.S * ne11;
        xh.data = (char *)x->data + (size_t)cut[i] * x->nb[2];
        ih.data = (char *)ids->data + (size_t)cut[i] * ids->nb[1];
        yh.data = (char *)y->data + (size_t)cut[i] * y->nb[2];
        if (!mmid_exec(h, w, &xh, &ih, &yh, st, ws, cap, d)) return 0;
      }
      return 1;
    }
  }
  MmidWs b;
  mmid_carve(m, mmq, !apart, ws, &b);
  // 1. src1 rows (token t, row i11) -> Q8_K row t*ne11 + i11; the buckets; skipped / invalid routes
  const size_t xrow = mmq ? xrec_row_bytes(nb) : q8_row_bytes(nb);
  const int tt = mmq ? mmq_tiles((double)n_pairs / groups, groups, (int)O, mmq_wgs32(w->type, d->cus()), d->cus()) : 1;
  PrepArgs p{};
  p.b = BucketArgs{(const int32_t *)ids->data, ids->nb[1] / 4, (int)n_ids, (int)n_pairs, (int)E, b.counts, b.offs,
                   b.pairs, b.active, b.n_active, b.items, b.n_items, mmq ? 16 * tt : 0};
  p.x = (const float *)x->data;
  p.x_tok = x->nb[2] / 4;
  p.x_row = x->nb[1] / 4;
  p.ne11 = ne11;
  p.nb = nb;
  p.rows = (int)nq;
  p.y = b.xq;
  p.y_rstride = xrow;
  p.order = mmq ? mmq_order(w->type) : -1;
  p.out = apart ? (float *)y->data : nullptr;
  p.out_s = y->nb[2] / 4;
  p.out_k = y->nb[1] / 4;
  p.O = (int)O;
  if (launch_prep(p, st)) return 0;
  if (!apart) {
    if (hipMemcpy2DAsync(b.idc, (size_t)n_ids * 4, ids->data, ids->nb[1], (size_t)n_ids * 4, (size_t)m.S,
                         hipMemcpyDeviceToDevice, st) != hipSuccess)
      return 0;
    p.b.ids = b.idc;
    p.b.id_s = (size_t)n_ids;
    p.rows = 0;
    p.out = (float *)y->data;
    if (launch_prep(p, st, false)) return 0;
  }
  // 2. bucketed GEMV or MFMA
  GemvArgs a{};
  a.w0 = (const uint8_t *)w->data;
  a.w_estride = w->nb[2];
  a.w_rstride = w->nb[1];
  a.nrows = (int)O;
  a.nb = nb;
  a.xq = b.xq;
  a.xq_rstride = xrow;
  a.ne11 = ne11;
  a.K = (int)n_ids;
  a.n_active = b.n_active;
  a.active = b.active;
  a.offs = b.offs;
  a.pairs = b.pairs;
  a.out = (float *)y->data;
  a.out_s = y->nb[2] / 4;
  a.out_k = y->nb[1] / 4;
  a.grid = d->grid;
  a.signs = d->signs;
  if (mmq) {
    a.items = b.items;
    a.n_items = b.n_items;
    a.xq_bytes = (uint32_t)((size_t)nq * xrow);
    if (launch_mmq(w->type, false, tt, 4, mmq_max_items((int)n_pairs, (int)E, 16 * tt), a, st)) return 0;
  } else if (launch_gemv(w->type, false, pick_np((int)n_pairs, (int)E), a, groups, st)) {
    return 0;
  }
  return hipPeekAtLastError() == hipSuccess ? 1 : 0;
}

// Caller-owned workspaces bound to (device, stream) by zm_mul_mat_id_set_workspace.
struct WsBinding {
  int dev;
  hipStream_t stream;
  uint8_t *ptr;
  size_t bytes;
};
constexpr int kMaxBindings = 64;
WsBinding g_bind[kMaxBindings];
int g_nbind = 0;
std::mutex g_bind_mu;

}  // namespace

extern "C" {

size_t zm_mul_mat_id_workspace_size(const zm_tensor *src0, const zm_tensor *src1, const zm_tensor *ids,
                                    const zm_tensor *dst) {
  MmidShape m;
  return mmid_shape(src0, src1, ids, dst, &m) ? m.ws_bytes : 0;
}

int zm_mul_mat_id_set_workspace(void *stream, void *workspace, size_t bytes) {
  int dev = 0;
  HIP_OK(hipGetDevice(&dev));
  if (workspace && ((uintptr_t)workspace & 255)) return fail("zm_mul_mat_id_set_workspace: workspace not 256-byte aligned");
  std::lock_guard<std::mutex> lk(g_bind_mu);
  for (int i = 0; i < g_nbind; ++i)
    if (g_bind[i].dev == dev && g_bind[i].stream == (hipStream_t)stream) {
      if (workspace) {
        g_bind[i].ptr = (uint8_t *)workspace;
        g_bind[i].bytes = bytes;
      } else {
        g_bind[i] = g_bind[--g_nbind];
      }
      return 0;
    }
  if (!workspace) return 0;
  if (g_nbind == kMaxBindings) return fail("zm_mul_mat_id_set_workspace: more than %d bound streams", kMaxBindings);
  g_bind[g_nbind++] = WsBinding{dev, (hipStream_t)stream, (uint8_t *)workspace, bytes};
  return 0;
}

int zm_mul_mat_id(const zm_tensor *w, const zm_tensor *x, const zm_tensor *ids, zm_tensor *y, void *stream,
                  int execute) {
  MmidShape m;
  if (!mmid_shape(w, x, ids, y, &m)) return 0;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  uint8_t *ws = nullptr;
  size_t cap = 0;
  {
    // query: the smallest workspace bound on this device must hold the shape
    // (ggml asks with no stream, then executes on one of its streams);
    // execute: the workspace bound to this stream
    std::lock_guard<std::mutex> lk(g_bind_mu);
    bool any = false;
    for (int i = 0; i < g_nbind; ++i) {
      if (g_bind[i].dev != dev) continue;
      if (!execute) {
        cap = any ? std::min(cap, g_bind[i].bytes) : g_bind[i].bytes;
        any = true;
      } else if (g_bind[i].stream == (hipStream_t)stream) {
        cap = g_bind[i].bytes;
        ws = g_bind[i].ptr;
        any = true;
      }
    }
    if (!any || cap < m.ws_least) {
      fail("zm_mul_mat_id: %s (needs %zu bytes, zm_mul_mat_id_workspace_size)",
           any ? "bound workspace too small" : "no workspace bound for this device/stream", m.ws_bytes);
      return 0;
    }
  }
  if (!execute) return 1;
  DeviceState *d;
  if (device_state(&d) || !mmid_exec(m, w, x, ids, y, (hipStream_t)stream, ws, cap, d)) return 0;
  count_mmid_launch();
  return 1;
}

int zm_mul_mat_id_static(const zm_tensor *w, const zm_tensor *x, const zm_tensor *ids, zm_tensor *dst, void *stream,
                         int execute) {
  MmidShape m;
  if (!mmid_shape(w, x, ids, dst, &m)) return 0;
  if (m.ws_least > kStaticScratchBytes) {
    fail("zm_mul_mat_id_static: shape needs %zu bytes of scratch, more than the %zu-byte device array", m.ws_least,
         kStaticScratchBytes);
    return 0;
  }
  if (!execute) return 1;
  DeviceState *d = device_state_if_ready();
  if (!d) {
    fail("zm_mul_mat_id_static: zm_init has not run on this device");
    return 0;
  }
  // every scratch array is written before it is read within the call, so
  // nothing needs clearing between calls
  if (!mmid_exec(m, w, x, ids, dst, (hipStream_t)stream, d->scratch, kStaticScratchBytes, d)) return 0;
  count_mmid_launch();
  return 1;
}

// ---------------------------------------------------------------- debug: block dots

}  // extern "C"

namespace {
// Debug kernel: per super-block integer parts of one weight row against one
// Q8_K row, computed by both decode dot paths -- the 4-lane quarter path of the
// bucketed GEMV and the whole-block unit path of the fused decode kernel.  The
// unit result is written; a disagreement writes INT32_MIN into isum instead.
template <int T>
__global__ void k_block_dots(const uint8_t *w, const uint8_t *xq, int nb, int32_t *isum, int32_t *imin,
                             const uint64_t *grid, const uint64_t *signs) {
  const int lane = threadIdx.x & 63;
  const int gq = blockIdx.x * 64 + lane;  // quarter index
  const int b = gq >> 2, q = gq & 3;
  QInt r{0, 0};
  int ui = 0, um = 0;
  if (b < nb) {
    Q8Slice s;
    WSlice ws;
    load_q8_slice<T>(xq, nb, b, q, s);
    load_w_slice<T>(w + (size_t)b * block_bytes(T), q, ws);
    r = quarter_int<T>(ws, q, s, grid, signs);
    if constexpr (has_unit<T>()) {
      if (q < unit_per_block<T>()) {
        const rsrc_t rw = make_rsrc(w, (uint32_t)(nb * block_bytes(T)));
        Unit<T> u[1];
        load_unit<T>(rw, b * block_bytes(T), q, u[0]);
        int ri[1], rm[1];
        unit_ints<T, 1>(u, q, xblk_planar(xq, nb, b), grid, signs, ri, rm);
        ui = ri[0];
        um = rm[0];
      }
    }
  }
  r.isum = group_sum_i<4>(r.isum);
  r.imin = group_sum_i<4>(r.imin);
  if constexpr (has_unit<T>()) {
    ui = group_sum_i<4>(ui);
    um = group_sum_i<4>(um);
  } else {
    ui = r.isum;  // no whole-block path for this type: the quarter sums are reported
    um = r.imin;
  }
  if (b < nb && q == 0) {
    const bool agree = ui == r.isum && um == r.imin;
    isum[b] = agree ? ui : INT32_MIN;
    imin[b] = um;
  }
}
}  // namespace

extern "C" {

int zm_block_dots(int type, const void *w_row, const float *x, int n, int32_t *isum, int32_t *imin, void *stream) {
  if (!type_supported(type) || n <= 0 || n % QK || !w_row || !x || !isum || !imin)
    return fail("zm_block_dots: bad arguments");
  DeviceState *d;
  if (device_state(&d)) return -1;
  hipStream_t st = (hipStream_t)stream;
  const int nb = n / QK;
  uint8_t *xq = nullptr;
  HIP_OK(hipMallocAsync((void **)&xq, q8_row_bytes(nb), st));
  if (launch_quant(x, (size_t)n, nb, 1, xq, q8_row_bytes(nb), 1, st)) return -1;
  const dim3 g((unsigned)((nb * 4 + 63) / 64));
  const uint8_t *w = (const uint8_t *)w_row;
  switch (type) {
  case T_Q2_K: hipLaunchKernelGGL(k_block_dots<T_Q2_K>, g, dim3(64), 0, st, w, xq, nb, isum, imin, d->grid, d->signs); break;
  case T_Q3_K: hipLaunchKernelGGL(k_block_dots<T_Q3_K>, g, dim3(64), 0, st, w, xq, nb, isum, imin, d->grid, d->signs); break;
  case T_Q4_K: hipLaunchKernelGGL(k_block_dots<T_Q4_K>, g, dim3(64), 0, st, w, xq, nb, isum, imin, d->grid, d->signs); break;
  case T_Q5_K: hipLaunchKernelGGL(k_block_dots<T_Q5_K>, g, dim3(64), 0, st, w, xq, nb, isum, imin, d->grid, d->signs); break;
  case T_Q6_K: hipLaunchKernelGGL(k_block_dots<T_Q6_K>, g, dim3(64), 0, st, w, xq, nb, isum, imin, d->grid, d->signs); break;
  case T_IQ4_XS: hipLaunchKernelGGL(k_block_dots<T_IQ4_XS>, g, dim3(64), 0, st, w, xq, nb, isum, imin, d->iq4, d->signs); break;
  case T_IQ3_XXS: hipLaunchKernelGGL(k_block_dots<T_IQ3_XXS>, g, dim3(64), 0, st, w, xq, nb, isum, imin, d->iq3, d->signs); break;
  default: hipLaunchKernelGGL(k_block_dots<T_IQ2_XXS>, g, dim3(64), 0, st, w, xq, nb, isum, imin, d->grid, d->signs); break;
  }
  HIP_OK(hipGetLastError());
  HIP_OK(hipFreeAsync(xq, st));
  return 0;
}

// ---------------------------------------------------------------- routed layer

}  // extern "C"

namespace {
struct LayerWs {
  float *logits;
  int32_t *ids;
  float *weights;
  uint8_t *xq;
  int32_t *counts, *offs, *pairs, *active, *n_active;
  uint8_t *aq;
  float *y;
  uint8_t *xq_s, *aq_s;
  float *y_s;
  float *act, *act_s, *f_act;
  uint32_t *f_sync;
  int32_t *items, *n_items;  // MFMA work items
};

size_t layer_ws(const zm_moe_layer *L, int S, uint8_t *base, LayerWs *w) {
  const int H = L->H, F = L->F, E = L->router.n_experts, K = L->router.topk, NS = L->n_slots;
  const int nbH = H / QK, nbF = F / QK;
  Bump b{base};
  LayerWs t{};
  t.logits = b.take<float>((size_t)S * E * 4);
  t.ids = b.take<int32_t>((size_t)S * K * 4);
  t.weights = b.take<float>((size_t)S * K * 4);
  t.xq = b.take<uint8_t>((size_t)S * xrec_row_bytes(nbH));  // records; planar rows are smaller
  t.counts = b.take<int32_t>((size_t)NS * 4);
  t.offs = b.take<int32_t>((size_t)(NS + 1) * 4);
  t.pairs = b.take<int32_t>((size_t)S * K * 4);
  t.active = b.take<int32_t>((size_t)NS * 4);
  t.n_active = b.take<int32_t>(4);
  t.items = b.take<int32_t>((size_t)mmq_max_items(S * K, NS, 16) * 4);
  t.n_items = b.take<int32_t>(4);
  t.aq = b.take<uint8_t>((size_t)S * K * xrec_row_bytes(nbF));
  t.y = b.take<float>((size_t)S * K * H * 4);
  const size_t fs = L->F_shared > 0 ? (size_t)L->F_shared : 0;
  if (fs) {
    t.aq_s = b.take<uint8_t>((size_t)S * xrec_row_bytes((int)(fs / QK)));
    t.y_s = b.take<float>((size_t)S * H * 4);
    t.xq_s = reinterpret_cast<uint8_t *>(t.y_s);  // read for the last time before the down product writes y_s
  }
  // act rows of every pair, then the shared rows (one call has them from the
  // multi-kernel path or from the fused decode kernel), and the fused kernel's
  // sync words (zero at allocation, left at zero by every launch)
  t.act = t.f_act = b.take<float>(((size_t)S * K * F + S * fs) * 4);
  if (fs) t.act_s = base ? t.act + (size_t)S * K * F : nullptr;
  t.f_sync = b.take<uint32_t>((size_t)DEC_SYNC_WORDS * 4);
  if (w) *w = t;
  return b.off + 256;
}

int check_layer(const zm_moe_layer *L) {
  if (!L) return fail("null layer");
  if (L->H <= 0 || L->H % QK || L->H / QK > 64) return fail("H must be a multiple of 256, <= 16384");
  if (L->F <= 0 || L->F % QK || L->F / QK > 64) return fail("F must be a multiple of 256, <= 16384");
  if (!type_supported(L->type_gate) || L->type_up != L->type_gate || !type_supported(L->type_down))
    return fail("unsupported expert types (gate and up must share a type)");
  if (L->n_slots <= 0 || L->n_slots > BUCKET_MAX_E) return fail("n_slots out of range");
  if (L->router.n_experts <= 0 || L->router.n_experts > ROUTER_MAX_E) return fail("n_experts out of range");
  if (L->router.topk <= 0 || L->router.topk > 64 || L->router.topk > L->router.n_experts) return fail("bad topk");
  if (!L->route_map && L->n_slots != L->router.n_experts) return fail("n_slots != n_experts without a slot table");
  if (!L->w_gate || !L->w_up || !L->w_down) return fail("null expert weights");
  if (L->F_shared > 0) {
    if (L->F_shared % QK || L->F_shared / QK > 64 || !type_supported(L->type_shared) || !L->ws_gate || !L->ws_up ||
        !L->ws_down)
      return fail("bad shared expert");
  }
  if (L->router_w && L->H % 4) return fail("router GEMV needs H %% 4 == 0");
  return 0;
}
int units_per_block(int t) {
  return t == T_Q3_K || t == T_Q4_K || t == T_Q5_K || t == T_Q6_K || t == T_IQ4_XS || t == T_IQ3_XXS ? 2 : 1;
}

DecFn find_decode(int tg, int td, int ts, int l1, int ir, int is) {
  if (DecFn f = find_decode_a(tg, td, ts, l1, ir, is)) return f;
  return find_decode_b(tg, td, ts, l1, ir, is);
}

bool fused_enabled() {
  const char *e = getenv("ZEROMOE_FUSED_DECODE");
  return !(e && e[0] == '0');
}

// grid of co-resident workgroups for a decode kernel (cached per device and kernel)
int decode_grid(DecFn fn, int *out) {
  static std::mutex mu;
  static struct Ent {
    int dev;
    DecFn fn;
    int grid;
  } cache[64];
  static int n = 0;
  int dev = 0;
  HIP_OK(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(mu);
  for (int i = 0; i < n; ++i)
    if (cache[i].dev == dev && cache[i].fn == fn) {
      *out = cache[i].grid;
      return 0;
    }
  int per_cu = 0, cus = 0;
  HIP_OK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void *>(fn), DEC_THREADS, 0));
  HIP_OK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  const int grid = per_cu * cus;
  if (grid <= 0) return fail("decode kernel does not fit on a CU");
  if (n < 64) cache[n++] = Ent{dev, fn, grid};
  *out = grid;
  return 0;
}

// Returns 0 when launched, 1 when this shape takes the multi-kernel path, -1 on error.
int launch_fused(const zm_moe_layer *L, const float *x, const float *logits, int S, float *out, int32_t *ids,
                 float *wts, const LayerWs &w, const DeviceState *d, hipStream_t st) {
  const int H = L->H, F = L->F, E = L->router.n_experts, K = L->router.topk;
  const int nbH = H / QK, nbF = F / QK;
  const int Fs = L->F_shared > 0 ? L->F_shared : 0;
  const int nbFs = Fs / QK;
  if (!fused_enabled() || S > DEC_MAX_S || S * K > DEC_MAX_PAIRS || E > DEC_MAX_E)
    return 1;
  if (L->type_up != L->type_gate) return 1;
  const int u1 = nbH * units_per_block(L->type_gate);
  if (Fs && nbH * units_per_block(L->type_shared) > 64) return 1;
  // down rows: IQ2_XXS in half blocks (the decode kernel's H2)
  const int ir = (K * nbF * (L->type_down == T_IQ2_XXS ? 2 : units_per_block(L->type_down)) + 31) / 32;
  const int is = Fs ? (nbFs * units_per_block(L->type_shared) + 31) / 32 : 0;
  // lanes per routed gate/up row: 16 or 32, or 16 + 4 for rows of 20 units
  // where the kernel has that layout
  DecFn fn = nullptr;
  if (u1 == 20) fn = find_decode(L->type_gate, L->type_down, Fs ? L->type_shared : 0, 20, ir, is);
  if (!fn) {
    const int l1 = u1 <= 16 ? 16 : (u1 <= 32 ? 32 : 0);
    fn = find_decode(L->type_gate, L->type_down, Fs ? L->type_shared : 0, l1, ir, is);
  }
  if (!fn) return 1;
  int G = 0;
  if (decode_grid(fn, &G)) return -1;
  const long T1 = (long)S * K * F + (long)S * Fs;
  const size_t q8F = q8l_row_bytes(nbF), q8Fs = Fs ? q8l_row_bytes(nbFs) : 0;
  if ((size_t)S * q8l_row_bytes(nbH) > (size_t)DEC_LDS_Q8 || 2 * ((size_t)K * q8F + q8Fs) > (size_t)DEC_LDS_Q8) return 1;
  if (T1 >= (1l << 24) || (long)S * H >= (1l << 24)) return 1;  // float-reciprocal index math
  if ((T1 + QK - 1) / QK > DEC_MAX_ABLK) return 1;                // act block counters
  DecodeArgs a{};
  a.r = RouterArgs{logits, L->logit_bias, L->sel_bias, L->route_map, L->route_mask, E, K, L->router.gating,
                   L->router.n_groups, L->router.n_groups_used, L->router.weights_norm, L->router.weights_scale,
                   ids, wts};
  a.x = x;
  a.out = out;
  a.H = H;
  a.F = F;
  a.K = K;
  a.S = S;
  a.nbH = nbH;
  a.nbF = nbF;
  a.wg = (const uint8_t *)L->w_gate;
  a.wu = (const uint8_t *)L->w_up;
  a.wd = (const uint8_t *)L->w_down;
  a.g_rstride = row_bytes(L->type_gate, H);
  a.g_estride = a.g_rstride * F;
  a.d_rstride = row_bytes(L->type_down, F);
  a.d_estride = a.d_rstride * H;
  a.Fs = Fs;
  a.nbFs = nbFs;
  if (Fs) {
    a.sg = (const uint8_t *)L->ws_gate;
    a.su = (const uint8_t *)L->ws_up;
    a.sd = (const uint8_t *)L->ws_down;
    a.sg_rstride = row_bytes(L->type_shared, H);
    a.sd_rstride = row_bytes(L->type_shared, Fs);
  }
  {
    const size_t NSl = (size_t)L->n_slots;
    const size_t wgb = NSl * a.g_estride, wdb = NSl * a.d_estride;
    const size_t sgb = Fs ? (size_t)Fs * a.sg_rstride : 0, sdb = Fs ? (size_t)H * a.sd_rstride : 0;
    if (wgb >= (1ull << 31) || wdb >= (1ull << 31) || sgb >= (1ull << 31) || sdb >= (1ull << 31)) return 1;
    a.wg_bytes = (uint32_t)wgb;
    a.wd_bytes = (uint32_t)wdb;
    a.sg_bytes = (uint32_t)sgb;
    a.sd_bytes = (uint32_t)sdb;
  }
  a.act = w.f_act;
  a.sync = w.f_sync;
  auto uses = [&](int t) { return L->type_gate == t || L->type_down == t || (Fs && L->type_shared == t); };
  a.grid = uses(T_IQ4_XS) ? d->iq4 : (uses(T_IQ3_XXS) ? d->iq3 : d->grid);
  a.signs = d->signs;
  a.spin_limit = 1 << 23;
  // test hook: force the bounded waits to give up (a negative limit expires
  // every act-block wait on its first poll, whatever the counters show)
  if (const char *sl = getenv("ZEROMOE_SPIN_LIMIT"); sl && sl[0])
    a.spin_limit = atoi(sl);
  if (const char *tr = getenv("ZEROMOE_TRACE"); tr && tr[0] == '1') {
    DeviceState *dm = const_cast<DeviceState *>(d);
    if (dm->trace_n < (size_t)G * 8) {
      if (dm->trace) (void)hipFree(dm->trace);
      HIP_OK(hipMalloc(&dm->trace, (size_t)G * 8 * sizeof(uint64_t)));
      dm->trace_n = (size_t)G * 8;
    }
    HIP_OK(hipMemsetAsync(dm->trace, 0, dm->trace_n * sizeof(uint64_t), st));
    a.trace = dm->trace;
  }
  void *args[] = {&a};
  // A plain launch of exactly the co-resident grid: every workgroup is
  // dispatched at once on an otherwise idle device; the wait in the kernel is
  // bounded, so a device shared with other work degrades to an error status,
  // never a hang.  ZEROMOE_COOP=1 uses a cooperative launch instead.
  const char *coop = getenv("ZEROMOE_COOP");
  if (coop && coop[0] == '1')
    HIP_OK(hipLaunchCooperativeKernel(reinterpret_cast<const void *>(fn), dim3(G), dim3(DEC_THREADS), args, 0, st));
  else
    HIP_OK(hipLaunchKernel(reinterpret_cast<const void *>(fn), dim3(G), dim3(DEC_THREADS), args, 0, st));
  return 0;
}

}  // namespace

extern "C" {

int zm_debug_trace(uint64_t *host, int n) {
  DeviceState *d;
  if (device_state(&d)) return -1;
  if (!d->trace) return 0;
  const int m = std::min<int>(n, (int)d->trace_n);
  HIP_OK(hipDeviceSynchronize());
  HIP_OK(hipMemcpy(host, d->trace, (size_t)m * sizeof(uint64_t), hipMemcpyDeviceToHost));
  return m;
}

int zm_moe_status(const zm_moe_layer *layer, int S, void *workspace, void *stream) {
  if (check_layer(layer) || S <= 0 || !workspace) return -1;
  LayerWs w;
  layer_ws(layer, S, (uint8_t *)workspace, &w);
  uint32_t err = 0;
  HIP_OK(hipMemcpyAsync(&err, w.f_sync + 1, 4, hipMemcpyDeviceToHost, (hipStream_t)stream));
  HIP_OK(hipStreamSynchronize((hipStream_t)stream));
  if (err) {  // an expired wait leaves the arrival counters unknown: start them over
    HIP_OK(hipMemsetAsync(w.f_sync, 0, (size_t)DEC_SYNC_WORDS * 4, (hipStream_t)stream));
    HIP_OK(hipStreamSynchronize((hipStream_t)stream));
  }
  return (int)err;
}

size_t zm_moe_workspace_size(const zm_moe_layer *layer, int S) {
  if (check_layer(layer) || S <= 0) return 0;
  return layer_ws(layer, S, nullptr, nullptr);
}

int zm_moe_forward(const zm_moe_layer *L, const float *x, const float *logits, int S, float *out, int32_t *ids_out,
                   float *weights_out, void *workspace, size_t workspace_size, void *stream) {
  if (check_layer(L)) return -1;
  if (S <= 0 || !x || !out || (!logits && !L->router_w)) return fail("zm_moe_forward: bad arguments");
  if (S > 65535) return fail("S too large");
  static_assert(65535 * 64 <= MMQ_MAX_PAIRS, "S * topk");
  if (!workspace || workspace_size < layer_ws(L, S, nullptr, nullptr)) return fail("workspace too small");
  DeviceState *d;
  if (device_state(&d)) return -1;
  hipStream_t st = (hipStream_t)stream;
  LayerWs w;
  layer_ws(L, S, (uint8_t *)workspace, &w);
  const int H = L->H, F = L->F, E = L->router.n_experts, K = L->router.topk, NS = L->n_slots;
  const int nbH = H / QK, nbF = F / QK;
  int32_t *ids = ids_out ? ids_out : w.ids;
  float *wts = weights_out ? weights_out : w.weights;

  // router
  const float *lg = logits;
  if (L->router_w) {
    // K slices so that ~512 workgroups stream the router weights; the partial
    // sums go through w.y (S*K*H floats, unused until the down projection)
    int KS = 1;
    while (KS < 16 && ((E + 15) / 16) * ((S + 15) / 16) * KS * 2 <= 512 && H % (64 * KS * 2) == 0 &&
           (size_t)KS * 2 * S * E <= (size_t)S * K * H)
      KS *= 2;
    if (S >= 8 && H % 64 == 0) {
      hipLaunchKernelGGL(k_router_gemm, dim3((E + 15) / 16, (S + 15) / 16, KS), dim3(256), 0, st, L->router_w, x, H,
                         E, S, w.y);
      hipLaunchKernelGGL(k_router_sum, dim3((S * E + 255) / 256), dim3(256), 0, st, w.y, S * E, KS, w.logits);
    } else
      hipLaunchKernelGGL(k_router_gemv, dim3(E), dim3(256), 0, st, L->router_w, x, H, E, S, w.logits);
    lg = w.logits;
  }
  {
    const int rc = launch_fused(L, x, lg, S, out, ids, wts, w, d, st);
    if (rc <= 0) return rc;
  }
  if (check_router(L->router)) return -1;  // before the side stream has work
  // activations -> Q8_K rows: records for the grouped MFMA kernel, planar rows for the GEMV
  const size_t g_row = row_bytes(L->type_gate, H), d_row = row_bytes(L->type_down, F);
  const int groups = std::min(NS, S * K);
  const int likely = L->route_map ? (int)((int64_t)S * K * std::min(NS, E) / E) : S * K;
  const MmqLoad load{groups, likely, (int)std::sqrt((double)likely * S * K)};
  const bool mmq_g = mmq_applies(L->type_gate, L->w_gate, L->w_up, g_row * F, F, g_row, &load, (size_t)S, nbH);
  const bool mmq_d =
      mmq_applies(L->type_down, L->w_down, nullptr, d_row * H, H, d_row, &load, (size_t)S * K, nbF);
  auto quant = [&](bool rec, int type, const float *v, int n, int rows, uint8_t *y, hipStream_t q) {
    return rec ? launch_quant_rec(v, (size_t)n, n / QK, rows, y, type, q)
               : launch_quant(v, (size_t)n, n / QK, rows, y, q8_row_bytes(n / QK), 1, q);
  };
  auto qrow = [](bool rec, int nb) { return rec ? xrec_row_bytes(nb) : q8_row_bytes(nb); };
  // shared expert (dense over all tokens) on the side stream: it needs only x,
  // which it quantizes for itself, so that it starts beside the routing and the
  // preparation (after the fp32 router product, where the layer has one); the combine
  // waits for it.  Waiting for the preparation's rows of
  // x instead cost their time wherever the shared expert is the longer branch
  // (with the skipped rows in k_prep spread wider, 13 tokens, Q6_K shared expert
  // of 2048: layer 204 -> 168 us; 64 tokens, Q4_K: 361 -> 349).
  auto launch_shared = [&](hipStream_t ss) -> int {
    const int ts = L->type_shared, Fs = L->F_shared, nbS = Fs / QK;
    const size_t gr = row_bytes(ts, H), dr = row_bytes(ts, Fs);
    // one bucket of S pairs; from 8 tokens on (as the pairs of a bucket, not of a batch)
    const bool mg = S >= 8 && mmq_applies(ts, L->ws_gate, L->ws_up, 0, Fs, gr, nullptr, (size_t)S, nbH);
    const bool md = S >= 8 && mmq_applies(ts, L->ws_down, nullptr, 0, H, dr, nullptr, (size_t)S, nbS);
    if (quant(mg, ts, x, H, S, w.xq_s, ss)) return -1;
    GemvArgs c{};
    c.w0 = (const uint8_t *)L->ws_gate;
    c.w1 = (const uint8_t *)L->ws_up;
    c.w_rstride = gr;
    c.w_estride = 0;
    c.nrows = Fs;
    c.nb = nbH;
    c.xq = w.xq_s;
    c.xq_rstride = qrow(mg, nbH);
    c.xq_bytes = (uint32_t)((size_t)S * c.xq_rstride);
    c.ne11 = 1;
    c.K = 1;
    c.dense_S = S;
    c.out = w.act_s;
    c.out_s = Fs;
    c.out_k = 0;
    c.grid = d->grid;
    c.signs = d->signs;
    const int nps = S >= 4 ? 4 : (S >= 2 ? 2 : 1);
    // one-wave workgroups of 16 rows where 64-row tiles of 32 tokens would leave CUs idle
    const int cus = d->cus();
    auto dense = [&](bool mmq, bool gu, const GemvArgs &v) {
      const bool few = !forced_tiles() && (long)((v.nrows + 63) / 64) * ((S + 31) / 32) < cus;
      const int t = few ? 2 : mmq_tiles((double)S, 1, v.nrows, mmq_wgs32(ts, cus), cus);
      return mmq ? launch_mmq(ts, gu, t, few ? 1 : 4, (S + 16 * t - 1) / (16 * t), v, ss)
                 : launch_gemv(ts, gu, nps, v, 1, ss);
    };
    if (dense(mg, true, c)) return -1;
    if (quant(md, ts, w.act_s, Fs, S, w.aq_s, ss)) return -1;
    GemvArgs e2 = c;
    e2.w0 = (const uint8_t *)L->ws_down;
    e2.w1 = nullptr;
    e2.w_rstride = dr;
    e2.nrows = H;
    e2.nb = nbS;
    e2.xq = w.aq_s;
    e2.xq_rstride = qrow(md, nbS);
    e2.xq_bytes = (uint32_t)((size_t)S * e2.xq_rstride);
    e2.out = w.y_s;
    e2.out_s = H;
    return dense(md, false, e2) ? -1 : 0;
  };
  SideBranch side(d, st);
  if (L->F_shared > 0 && (side.fork() || launch_shared(d->side) || side.end())) return -1;
  if (zm_router(&L->router, lg, L->logit_bias, L->sel_bias, L->route_map, L->route_mask, S, ids, wts, st))
    return -1;
  // one list for both products, cut for rows between theirs (612 layers of few
  // experts or slots against items that are never halved: the smaller 1.19 times as
  // fast, 45 slower by over 5%, the mean 1.18 and 21, the larger 1.16 and 19)
  const int wgs32 = std::max(mmq_wgs32(L->type_gate, d->cus()), mmq_wgs32(L->type_down, d->cus()));
  const int tt = mmq_g || mmq_d ? mmq_tiles((double)(S * K) / groups, groups, (F + H) / 2, wgs32, d->cus()) : 1;
  {
    PrepArgs p{};
    p.b = BucketArgs{ids, (size_t)K, K, S * K, NS, w.counts, w.offs, w.pairs, w.active, w.n_active, w.items,
                     w.n_items, mmq_g || mmq_d ? 16 * tt : 0};
    p.x = x;
    p.x_tok = p.x_row = (size_t)H;
    p.ne11 = 1;
    p.nb = nbH;
    p.rows = S;
    p.y = w.xq;
    p.y_rstride = qrow(mmq_g, nbH);
    p.order = mmq_g ? mmq_order(L->type_gate) : -1;
    // skipped routes (slot table -1) read as zero rows; router ids are always valid otherwise
    p.out = L->route_map ? w.y : nullptr;
    p.out_s = (size_t)K * H;
    p.out_k = (size_t)H;
    p.O = H;
    if (launch_prep(p, st)) return -1;
  }
  // gate/up + SwiGLU
  const int np = pick_np(S * K, NS);
  GemvArgs a{};
  a.w0 = (const uint8_t *)L->w_gate;
  a.w1 = (const uint8_t *)L->w_up;
  a.w_rstride = g_row;
  a.w_estride = g_row * F;
  a.nrows = F;
  a.nb = nbH;
  a.xq = w.xq;
  a.xq_rstride = qrow(mmq_g, nbH);
  a.xq_bytes = (uint32_t)((size_t)S * a.xq_rstride);
  a.ne11 = 1;
  a.K = K;
  a.n_active = w.n_active;
  a.active = w.active;
  a.offs = w.offs;
  a.pairs = w.pairs;
  a.out = w.act;
  a.out_s = (size_t)K * F;
  a.out_k = F;
  a.grid = d->grid;
  a.signs = d->signs;
  const int max_items = mmq_max_items(S * K, NS, 16 * tt);
  a.items = w.items;
  a.n_items = w.n_items;
  if (mmq_g ? launch_mmq(L->type_gate, true, tt, 4, max_items, a, st)
            : launch_gemv(L->type_gate, true, np, a, groups, st))
    return -1;
  // act -> Q8_K
  if (quant(mmq_d, L->type_down, w.act, F, S * K, w.aq, st)) return -1;
  // down
  GemvArgs b = a;
  b.w0 = (const uint8_t *)L->w_down;
  b.w1 = nullptr;
  b.w_rstride = d_row;
  b.w_estride = d_row * H;
  b.nrows = H;
  b.nb = nbF;
  b.xq = w.aq;
  b.xq_rstride = qrow(mmq_d, nbF);
  b.xq_bytes = (uint32_t)((size_t)S * K * b.xq_rstride);
  b.ne11 = K;
  b.out = w.y;
  b.out_s = (size_t)K * H;
  b.out_k = H;
  if (mmq_d ? launch_mmq(L->type_down, false, tt, 4, max_items, b, st)
            : launch_gemv(L->type_down, false, np, b, groups, st))
    return -1;
  if (L->F_shared > 0 && side.join()) return -1;  // the shared expert's y_s
  const float *ys = L->F_shared > 0 ? w.y_s : nullptr;
  if ((uintptr_t)out & 15)
    hipLaunchKernelGGL(k_combine1, dim3((H + 255) / 256, S), dim3(256), 0, st, w.y, wts, ys, H, K, out);
  else
    hipLaunchKernelGGL(k_combine, dim3((H + 1023) / 1024, S), dim3(256), 0, st, w.y, wts, ys, H, K, out);
  HIP_OK(hipGetLastError());
  return 0;
}

}  // extern "C"
