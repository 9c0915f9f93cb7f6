// zm_mmq.hpp -- bucketed MUL_MAT_ID for batches and prefill on int8 MFMA.
//
// Per active expert, out[pair][row] = W_e[row] . q8(x[pair]) for the pairs of
// the expert's bucket (the CSR of /root/reference/core/batched_dispatch_pipeline.cpp:1181-1202),
// gate/up optionally fused with SwiGLU (moe_routed_ggml.hpp:166-191).
//
// Work split.  A work item is a run of up to 16 * TT pairs of one bucket; a
// workgroup takes one item and 16 * NW weight rows, a wave 16 of them.  K runs
// in super-blocks of 256.  Per block a wave unpacks its 16 rows (gate, then up)
// once and dots them with the item's 16-pair tiles on v_mfma_i32_16x16x64_i8
// (or 16x16x32): pairs are the A operand, weight rows the B operand, so a
// lane's four outputs belong to ONE weight row (lane % 16) and the per-row
// scales are per-lane values.  The K loop is instantiated per tile count of the
// item, so it has no branch per tile.
//
// What bounds it, and the layout that follows.  Loading each lane's few bytes
// of its row straight into registers (16 rows per instruction, 8-16 bytes
// each) kept the vector memory unit busy with addresses: without the weight
// loads the Q4_K gate/up product of 512 tokens (4096 x 1536, 128 experts) took
// 204 us instead of 341, and with loads that always hit the cache 295.  So
// weights come in as they lie in memory: a row's block as consecutive 16-byte
// units, 64 units per direct buffer-to-LDS load, into a slot private to the
// wave, and the lanes pick their fields out of LDS.  The slot is read at the
// start of a block and its next block requested at once, so a request has the
// whole block's arithmetic to land.  Activations are staged the same way, one
// 304-byte record per pair and block (two stages, one barrier per stage; a third
// stage gained nothing).  Units per row are odd (padded), and so is a record,
// counted in 16-byte units: 16 rows read 16 different bank groups.
// The one-stage lead is lost in 15 of the 64 instantiations.  Of types whose rows
// start on either half of a dword the two parities' offsets (wo) come to lie in
// scratch memory (32 to 48 bytes a lane; Q6_K down with 32- and 64-pair items and
// gate/up with 32, Q3_K and IQ2_XXS down with 64, IQ3_XXS down with 32, the one-wave
// variants), and Q3_K gate/up with 64-pair items spills 21 registers: what is
// loaded back in the loop is waited for with vmcnt(0), and the requests before it
// with it.
// On the vector units the unpacking and the tile epilogue (about 100 + 25 per
// tile instructions per matrix and block for Q4_K) are the floor at many pairs
// per expert, the weight stream at few.  Kernel times before (weights straight to
// registers, or the GEMV) and now:
//   512 tokens, Q4_K, skewed loads: gate/up 333 -> 238 us, down 164 -> 145
//   333 tokens, even loads: Q2_K gate/up 210 -> 176; Q3_K down 884 (GEMV) -> 136
//   2048 tokens of 2048 x 768: Q5_K gate/up 328 -> 260, Q6_K down 264 -> 214
//   24 tokens: Q4_K gate/up 211 (GEMV) -> 148, 4.8 TB/s; Q6_K down 168 (GEMV) -> 124, 4.2 TB/s
//   130 tokens, IQ3_XXS: 236 -> 113 per product
//
// Activation record of one 256-value block (k_quant_rec): 256 int8 | 16 f16
// sums of 16 values (integers up to 2032: exact) | f32 d | pad.  The int8 of a
// 64-value chunk are ordered so that k-group g of an MFMA operand is 16
// consecutive bytes: natural order for Q2_K / Q3_K, else the 8-byte group g of
// the chunk's first 32 values, then that of its second 32.
//
// Per type (lane = row n = lane % 16, k-group g = lane / 16):
// Q4_K, Q5_K: the 6-bit sub-block scale sc = 8*hi + lo is folded into the
//   weights (nibble * lo and nibble * hi <= 105: int8), two chains over the
//   block give isum = D_lo + 8 D_hi = sum_sb sc * (q . x)_sb exactly; Q5_K's
//   fifth bit is a third chain with the whole scale, + 16 D_5.
// Q2_K: q * sc <= 45, one chain.
// Q3_K: (4 - q') * sc (q' = 0..7 the quant with its high bit, sc = -32..31) lies in
//   -128..124: one byte permute on an 8-entry table of the scale per 4 weights
//   (tables of all 64 scales in LDS), one chain, isum = -D.
// Their mins: imin = sum_sb m * bsum (f16 operands, exact f32 sums) on one
//   v_mfma_f32_16x16x16_f16 (16 cycles; on f32 operands it took 2 to 4 of 32).
//   f += d_x * (d * isum - dmin * imin), ggml's vec_dot combine.
// Q6_K (signed 8-bit scale per 16 weights; 4 * (q - 32) is int8): two
//   v_mfma_i32_16x16x32_i8 per pair of 16-weight sub-blocks (the first alone,
//   then both), scaled per lane on the integer sums.
// IQ2_XXS, IQ3_XXS, IQ4_XS (grid or table values, one scale per 32 weights): one
//   v_mfma_i32_16x16x32_i8 per sub-block, scaled per lane.
#pragma once

#include <algorithm>

#include "zm_kernels.hpp"

namespace zm {

typedef int v4i_t __attribute__((ext_vector_type(4)));
typedef float v4f_t __attribute__((ext_vector_type(4)));
typedef _Float16 v4h_t __attribute__((ext_vector_type(4)));
typedef _Float16 v2h_t __attribute__((ext_vector_type(2)));
typedef unsigned short v2u16_t __attribute__((ext_vector_type(2)));
typedef unsigned v4u_t __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------- buffer-to-LDS loads
//
// Lane L's 16 bytes land at lds + 16 * L (inactive lanes write nothing,
// out-of-range dwords write zeros).  Inline asm: the compiler's wait insertion
// does not track them, so the caller counts them and waits itself.
__device__ __forceinline__ v4u_t dma_rsrc(const void *p, uint32_t bytes) {
  const uint64_t a = (uint64_t)(uintptr_t)p;
  return v4u_t{(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, bytes, 0x00020000u};
}
__device__ __forceinline__ uint32_t lds_addr(const void *p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)p;
}
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // m0 is written by the asm and by nothing else here
__device__ __forceinline__ void dma_lds16(v4u_t rs, uint32_t lds, int vo, int so) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(vo), "s"(rs), "s"(so)
               : "memory", "m0");
}
#pragma clang diagnostic pop
// at most N vector memory operations of this wave outstanding
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
// the same, then the workgroup barrier (this wave's LDS reads are complete)
template <int N>
__device__ __forceinline__ void wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

template <class P, int A>
__device__ __forceinline__ P lds_get(const uint8_t *p) {
  P v;
  __builtin_memcpy(&v, __builtin_assume_aligned(p, A), sizeof(P));
  return v;
}
// N dwords that start 0, 2 or 4 bytes past the dword p: N + 1 aligned dwords and
// one byte permute each (sel: align_sel).  LDS reads at the 2-byte address itself
// are correct but stall: a third of the Q6_K kernel's LDS time.
template <int N>
struct Dwords {
  uint32_t v[N];
};
template <int N, int A>
__device__ __forceinline__ Dwords<N> lds_get_at(const uint8_t *p, uint32_t sel) {
  uint32_t r[N + 1];
  __builtin_memcpy(r, __builtin_assume_aligned(p, A), 4 * N);
  r[N] = lds_get<uint32_t, 4>(p + 4 * N);
  Dwords<N> o;
#pragma unroll
  for (int i = 0; i < N; ++i) o.v[i] = __builtin_amdgcn_perm(r[i + 1], r[i], sel);
  return o;
}
__device__ __forceinline__ uint32_t align_sel(int bytes) { return 0x03020100u + 0x01010101u * (uint32_t)bytes; }

// four packed bytes times a small factor, bytewise (every product < 256: no
// carry crosses a byte): one packed 16-bit multiply
__device__ __forceinline__ uint32_t mul_bytes(uint32_t packed, uint32_t f) {
  const v2u16_t p = __builtin_bit_cast(v2u16_t, packed);
  const v2u16_t m = {(unsigned short)f, (unsigned short)f};
  return __builtin_bit_cast(uint32_t, p * m);
}
// two bytes of w, picked into 16-bit halves by the permute selector, as f16 (1024 + b, less 1024)
__device__ __forceinline__ v2h_t bytes_f16(uint32_t w, uint32_t sel) {
  const uint32_t u = __builtin_amdgcn_perm(0, w, sel) | 0x64006400u;
  return __builtin_bit_cast(v2h_t, u) - v2h_t{(_Float16)1024.f, (_Float16)1024.f};
}

// ---------------------------------------------------------------- activation records

constexpr int XREC = 304;           // bytes of one block's record
constexpr int XUNITS = XREC / 16;   // 19
// records are reached by unsigned 32-bit offsets; one past every buffer's extent
constexpr uint32_t XOOR = 0xfffffff0u;
constexpr size_t XREC_MAX_BYTES = 0xfffff000u;
__host__ __device__ constexpr size_t xrec_row_bytes(int nb) { return (size_t)nb * XREC; }
// value order of a record's int8: 0 natural, 1 the 8-byte groups of the two 32-value halves of a chunk alternating
__host__ __device__ constexpr int mmq_order(int type) { return type == T_Q2_K || type == T_Q3_K ? 0 : 1; }

// 16 values of block b of a record row (the lane's share of quant_block16)
__device__ __forceinline__ void store_rec16(uint8_t *row, int b, const Q8Out16 &o, int l16, int order) {
  uint8_t *r = row + (size_t)b * XREC;
  if (order == 0) {
    *reinterpret_cast<uint4 *>(r + 16 * l16) = o.q;
  } else {  // values 16 * l16 .. +15 are groups 2q, 2q + 1 of half h of chunk c
    const int c = l16 >> 2, h = (l16 >> 1) & 1, q = l16 & 1;
    *reinterpret_cast<uint2 *>(r + 64 * c + 32 * q + 8 * h) = make_uint2(o.q.x, o.q.y);
    *reinterpret_cast<uint2 *>(r + 64 * c + 32 * q + 16 + 8 * h) = make_uint2(o.q.z, o.q.w);
  }
  reinterpret_cast<_Float16 *>(r + 256)[l16] = (_Float16)(float)o.bsum;
  if (l16 == 0) *reinterpret_cast<float *>(r + 288) = o.d;
}
// f32 rows -> records, 16 lanes per block
static __global__ __launch_bounds__(256) void k_quant_rec(const float *__restrict__ x, size_t x_rstride, int nb,
                                                          int rows, uint8_t *__restrict__ y, size_t y_rstride,
                                                          int order) {
  const int l16 = threadIdx.x & 15;
  const int gb = blockIdx.x * 16 + (threadIdx.x >> 4);
  const int row = gb / nb, b = gb % nb;
  if (row >= rows) return;
  float v[16];
  load16(x + (size_t)row * x_rstride + (size_t)b * QK + 16 * l16, v);
  store_rec16(y + (size_t)row * y_rstride, b, quant_block16(v, l16), l16, order);
}

// ---------------------------------------------------------------- preparation
//
// What a bucketed product needs before it, in one launch: workgroup 0 sorts the
// pairs (and cuts the work list), the next q_wgs quantize the rows of src1, the
// rest write the rows of skipped routes (id < 0: zeros, id >= E: NaN;
// patches/ggml/0002...:50-54, kernels/quant/kquant_matmul.cu:660-663).
// Bound by workgroup 0's chain while the others run beside it.  Kernel times, us,
// as launches of their own -> here: hook, 130 tokens: rows 5.0, copy of the ids
// 4.5, buckets 5.5, skipped rows 6.6, work list 4.7 -> 6.8; layer, 512 tokens x 8:
// rows 6.3, buckets 10.2, work list 4.7 -> 12.6; 2048 x 8: buckets 33.3, work list
// 4.7 and the rows 9.0 -> 27.7.
struct PrepArgs {
  BucketArgs b;
  // src1: row r = token r / ne11, slot r % ne11 at x[token * x_tok + slot * x_row]
  const float *x;
  size_t x_tok, x_row;
  int ne11, nb, rows;
  uint8_t *y;
  size_t y_rstride;
  int order;  // record order, or -1: planar rows
  int sort_wgs, q_wgs;  // 1: workgroup 0 sorts, 0: only rows are written
  // output rows of skipped routes (out null: none)
  float *out;
  size_t out_s, out_k;
  int O;
};
constexpr int PREP_QBLOCKS = 64;  // 256-value blocks quantized per workgroup
constexpr int PREP_FPAIRS = 16;   // pairs looked through per workgroup, one per wave

static __global__ __launch_bounds__(1024) void k_prep(PrepArgs a) {
  __shared__ BucketLds l;
  const int wg = (int)blockIdx.x - a.sort_wgs;
  if (wg < 0) {
    bucket_wg(a.b, l);
    return;
  }
  if (wg < a.q_wgs) {
    const int l16 = threadIdx.x & 15;
    const long gb = (long)wg * PREP_QBLOCKS + (threadIdx.x >> 4);
    const int row = (int)(gb / a.nb), b = (int)(gb - (long)row * a.nb);
    if (row >= a.rows) return;
    const int t = row / a.ne11, i = row - t * a.ne11;
    float v[16];
    load16(a.x + (size_t)t * a.x_tok + (size_t)i * a.x_row + (size_t)b * QK + 16 * l16, v);
    const Q8Out16 o = quant_block16(v, l16);
    uint8_t *yr = a.y + (size_t)row * a.y_rstride;
    if (a.order < 0) store_q8_16(yr, a.nb, b, o, l16);
    else store_rec16(yr, b, o, l16, a.order);
    return;
  }
  const int lane = threadIdx.x & 63;
  const int p = (wg - a.q_wgs) * PREP_FPAIRS + (int)(threadIdx.x >> 6);
  if (p >= a.b.n_pairs) return;
  const int s = p / a.b.K, k = p - s * a.b.K;
  const int e = a.b.ids[(size_t)s * a.b.id_s + k];
  if (e >= 0 && e < a.b.E) return;
  const float v = e < 0 ? 0.0f : __int_as_float(0x7fc00000);
  float *o = a.out + (size_t)s * a.out_s + (size_t)k * a.out_k;
  for (int r = lane; r < a.O; r += 64) o[r] = v;
}

// ---------------------------------------------------------------- weight blocks in LDS

// blocks whose bytes are a multiple of 4 start on a dword; the others (2-byte
// types) are staged from the dword at or below their start
template <int T>
constexpr bool mmq_dword() {
  return block_bytes(T) % 4 == 0;
}
// 16-byte units loaded per row and stage of C blocks (an extra 2 bytes where a block starts inside a dword)
template <int T, int C>
constexpr int mmq_load_units() {
  return (C * block_bytes(T) + (mmq_dword<T>() ? 0 : 2) + 15) / 16;
}
// units of a row's slot: odd, so that 16 rows start in 16 different 16-byte bank groups
template <int T, int C>
constexpr int mmq_units() {
  return mmq_load_units<T, C>() | 1;
}

// the fields of one block that a lane needs
template <int T>
struct MmqW;
template <>
struct MmqW<T_Q4_K> {  // d, dmin, scales | the lane's 8 bytes of each 32-byte qs group
  uint4 hdr;
  uint2 qs[4];
};
template <>
struct MmqW<T_Q5_K> {  // d, dmin, scales | the lane's 8 bytes of qh and of each qs group
  uint4 hdr;
  uint2 qh;
  uint2 qs[4];
};
template <>
struct MmqW<T_Q2_K> {  // scales | the lane's 2 x 16 bytes of qs | d, dmin
  uint4 sc;
  uint4 qs[2];
  uint32_t dd;
};
template <>
struct MmqW<T_Q3_K> {  // the lane's 16 bytes of hmask and 2 x 16 of qs | scales | d
  Dwords<4> hm;
  Dwords<4> qs[2];
  Dwords<3> s;
  uint16_t d;
};
template <>
struct MmqW<T_Q6_K> {  // the lane's 4 x 8 bytes of ql, 2 x 8 of qh | scales | d
  Dwords<2> ql[4];
  Dwords<2> qh[2];
  Dwords<4> sc;
  uint16_t d;
};
template <>
struct MmqW<T_IQ2_XXS> {  // d | all 64 bytes of qs (grid-index and sign+scale words per sub-block)
  uint16_t d;
  Dwords<16> q;
};
template <>
struct MmqW<T_IQ3_XXS> {  // d | the lane's 2 grid-index bytes of each sub-block | 8 scale+sign words
  uint16_t d;
  uint16_t gi[8];
  Dwords<8> sas;
};
template <>
struct MmqW<T_IQ4_XS> {  // d, scales_h, scales_l | the lane's 8 qs bytes of each sub-block
  uint2 hdr;
  uint2 qs[8];
};

// p: the dword of the row's slot that holds the block's first byte, al: that byte's place in it (0 or 2; 0 for dword
// types); A: alignment of p
template <int T, int A>
__device__ __forceinline__ void mmq_read_w(const uint8_t *p, int al, int g, MmqW<T> &w) {
  const uint32_t sel = align_sel(al);
  if constexpr (T == T_Q4_K || T == T_Q5_K) {
    constexpr int QS = T == T_Q5_K ? 48 : 16;
    w.hdr = lds_get<uint4, A>(p);
    if constexpr (T == T_Q5_K) w.qh = lds_get<uint2, (A < 8 ? A : 8)>(p + 16 + 8 * g);
#pragma unroll
    for (int i = 0; i < 4; ++i) w.qs[i] = lds_get<uint2, (A < 8 ? A : 8)>(p + QS + 32 * i + 8 * g);
  } else if constexpr (T == T_Q2_K) {
    w.sc = lds_get<uint4, A>(p);
#pragma unroll
    for (int h = 0; h < 2; ++h) w.qs[h] = lds_get<uint4, A>(p + 16 + 32 * h + 16 * (g & 1));
    w.dd = lds_get<uint32_t, 4>(p + 80);
  } else if constexpr (T == T_Q3_K) {
    w.hm = lds_get_at<4, A>(p + 16 * (g & 1), sel);
#pragma unroll
    for (int h = 0; h < 2; ++h) w.qs[h] = lds_get_at<4, A>(p + 32 + 32 * h + 16 * (g & 1), sel);
    w.s = lds_get_at<3, A>(p + 96, sel);
    w.d = lds_get<uint16_t, 2>(p + 108 + al);
  } else if constexpr (T == T_Q6_K) {
#pragma unroll
    for (int i = 0; i < 4; ++i) w.ql[i] = lds_get_at<2, (A < 8 ? A : 8)>(p + 64 * (i >> 1) + 32 * (i & 1) + 8 * g, sel);
#pragma unroll
    for (int h = 0; h < 2; ++h) w.qh[h] = lds_get_at<2, (A < 8 ? A : 8)>(p + 128 + 32 * h + 8 * g, sel);
    w.sc = lds_get_at<4, A>(p + 192, sel);
    w.d = lds_get<uint16_t, 2>(p + 208 + al);
  } else if constexpr (T == T_IQ2_XXS) {
    w.d = lds_get<uint16_t, 2>(p + al);
    w.q = lds_get_at<16, A>(p, align_sel(2 + al));
  } else if constexpr (T == T_IQ3_XXS) {
    w.d = lds_get<uint16_t, 2>(p + al);
#pragma unroll
    for (int i = 0; i < 8; ++i) w.gi[i] = lds_get<uint16_t, 2>(p + al + 2 + 8 * i + 2 * g);
    w.sas = lds_get_at<8, A>(p + 64, align_sel(2 + al));
  } else {
    w.hdr = lds_get<uint2, (A < 8 ? A : 8)>(p);
#pragma unroll
    for (int i = 0; i < 8; ++i) w.qs[i] = lds_get<uint2, (A < 8 ? A : 8)>(p + 8 + 16 * i + 8 * (g & 1));
  }
}

// ---------------------------------------------------------------- B operands

template <int T>
constexpr bool mmq_folded() {  // scales in the weights: whole-block integer chains
  return T == T_Q2_K || T == T_Q3_K || T == T_Q4_K || T == T_Q5_K;
}
template <int T>
constexpr bool mmq_mins() {
  return T == T_Q2_K || T == T_Q4_K || T == T_Q5_K;
}
template <int T>
constexpr int mmq_chains() {
  return T == T_Q5_K ? 3 : (T == T_Q4_K ? 2 : 1);
}

template <int T, bool FOLDED = mmq_folded<T>()>
struct MmqB;
template <int T>
struct MmqB<T, true> {
  v4i_t b[mmq_chains<T>()][4];  // per chain and 64-weight chunk
  v4h_t mn;                     // mins of the 16-sums 4g .. 4g + 3
  float d, dmin;
};
template <int T>
struct MmqB<T, false> {
  static constexpr int NB = T == T_Q6_K ? 16 : 8;  // sub-blocks
  long b[NB];
  int s[NB];
  float d;
};

// tables: Q3_K 64 x 8 bytes (4 - k) * (s - 32); IQ2_XXS / IQ3_XXS grid and sign masks; IQ4_XS values in tab
template <int T>
__device__ __forceinline__ void mmq_unpack(const MmqW<T> &w, int g, const uint64_t *s_tab, const uint64_t *s_signs,
                                           const uint32_t (&tab)[4], MmqB<T> &o) {
  if constexpr (T == T_Q4_K || T == T_Q5_K) {
    const uint32_t u0 = w.hdr.y, u1 = w.hdr.z, u2 = w.hdr.w;
    const uint32_t sc_lo = u0 & 0x3f3f3f3fu, mn_lo = u1 & 0x3f3f3f3fu;
    const uint32_t sc_hi = (u2 & 0x0f0f0f0fu) | (((u0 >> 6) & 0x03030303u) << 4);
    const uint32_t mn_hi = ((u2 >> 4) & 0x0f0f0f0fu) | (((u1 >> 6) & 0x03030303u) << 4);
    o.d = h2f((uint16_t)(w.hdr.x & 0xffffu));
    o.dmin = h2f((uint16_t)(w.hdr.x >> 16));
    // 16-sums 4g .. 4g + 3 belong to sub-blocks 2g (twice), 2g + 1 (twice)
    const uint32_t mw = (g < 2 ? mn_lo : mn_hi) >> (16 * (g & 1));
    const v2h_t h0 = bytes_f16(mw, 0x0c000c00u), h1 = bytes_f16(mw, 0x0c010c01u);
    o.mn = v4h_t{h0[0], h0[1], h1[0], h1[1]};
    // chunk i = qs group i: sub-block 2i in its low nibbles, 2i + 1 in its high
    // nibbles; Q5_K: the fifth bits are bits 2i, 2i + 1 of the lane's qh bytes
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t scw = (i < 2 ? sc_lo : sc_hi) >> (16 * (i & 1));
      const uint32_t s0 = scw & 0xffu, s1 = (scw >> 8) & 0xffu;
      const uint2 q = w.qs[i];
      const uint32_t n0 = q.x & 0x0f0f0f0fu, n1 = q.y & 0x0f0f0f0fu;
      const uint32_t n2 = (q.x >> 4) & 0x0f0f0f0fu, n3 = (q.y >> 4) & 0x0f0f0f0fu;
      o.b[0][i] = v4i_t{(int)mul_bytes(n0, s0 & 7u), (int)mul_bytes(n1, s0 & 7u), (int)mul_bytes(n2, s1 & 7u),
                        (int)mul_bytes(n3, s1 & 7u)};
      o.b[1][i] = v4i_t{(int)mul_bytes(n0, s0 >> 3), (int)mul_bytes(n1, s0 >> 3), (int)mul_bytes(n2, s1 >> 3),
                        (int)mul_bytes(n3, s1 >> 3)};
      if constexpr (T == T_Q5_K) {
        const uint2 h = w.qh;
        o.b[2][i] = v4i_t{(int)mul_bytes((h.x >> (2 * i)) & 0x01010101u, s0),
                          (int)mul_bytes((h.y >> (2 * i)) & 0x01010101u, s0),
                          (int)mul_bytes((h.x >> (2 * i + 1)) & 0x01010101u, s1),
                          (int)mul_bytes((h.y >> (2 * i + 1)) & 0x01010101u, s1)};
      }
    }
  } else if constexpr (T == T_Q2_K) {
    o.d = h2f((uint16_t)(w.dd & 0xffffu));
    o.dmin = h2f((uint16_t)(w.dd >> 16));
    const uint32_t scb[4] = {w.sc.x, w.sc.y, w.sc.z, w.sc.w};
    const uint32_t mw = ((g < 2 ? (g == 0 ? scb[0] : scb[1]) : (g == 2 ? scb[2] : scb[3])) >> 4) & 0x0f0f0f0fu;
    const v2h_t h0 = bytes_f16(mw, 0x0c010c00u), h1 = bytes_f16(mw, 0x0c030c02u);
    o.mn = v4h_t{h0[0], h0[1], h1[0], h1[1]};
    // chunk c = 2h + jp, weights 64c + 16g .. +15: bit-plane 2jp + (g >> 1) of
    // qs bytes 32h + 16(g & 1) .. +15, sub-block 4c + g
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const uint32_t sc = (scb[c] >> (8 * g)) & 15u;
      const uint4 q = w.qs[c >> 1];
      const int sh = 4 * (c & 1) + 2 * (g >> 1);
#pragma unroll
      for (int k = 0; k < 4; ++k) o.b[0][c][k] = (int)mul_bytes((u4_get(q, k) >> sh) & 0x03030303u, sc);
    }
  } else if constexpr (T == T_Q3_K) {
    o.d = -h2f(w.d);  // the chain carries -(q' - 4) * sc
    o.dmin = 0.f;
    const uint32_t a0 = w.s.v[0] >> (8 * g), a1 = w.s.v[1] >> (8 * g), a2 = w.s.v[2] >> (8 * g);
    // chunk c as for Q2_K (sub-block 4c + g); the high bit of plane 4h + j is bit 4h + j of the hmask byte
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const uint32_t lo4 = ((c & 1 ? a1 : a0) >> (4 * (c >> 1))) & 15u;
      const uint64_t t = s_tab[lo4 | (((a2 >> (2 * c)) & 3u) << 4)];
      const int j = 2 * (c & 1) + (g >> 1);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t hm = w.hm.v[k];
        const uint32_t hb = ((c >= 2 ? hm >> 2 : hm << 2) >> j) & 0x04040404u;
        const uint32_t q = ((w.qs[c >> 1].v[k] >> (2 * j)) & 0x03030303u) | hb;
        o.b[0][c][k] = (int)__builtin_amdgcn_perm((uint32_t)(t >> 32), (uint32_t)t, q);
      }
    }
  } else if constexpr (T == T_Q6_K) {
    o.d = 0.25f * h2f(w.d);  // the operand carries 4 * (q - 32)
    const uint32_t (&scb)[4] = w.sc.v;
    const uint32_t keep0 = g < 2 ? 0xffffffffu : 0u;
    uint2 hb[2];
#pragma unroll
    for (int h = 0; h < 2; ++h)  // the upper of the two top bits flipped: q ^ 32
      hb[h] = make_uint2(w.qh[h].v[0] ^ 0xaaaaaaaau, w.qh[h].v[1] ^ 0xaaaaaaaau);
    // pair p = sub-blocks 2p (lane groups 0-1), 2p + 1 (groups 2-3): low (G < 2)
    // or high nibbles of ql bytes 64h + 32(p & 1) + 8g.., top bits 2G of qh bytes
    // 32h + 8g...  The first operand is sub-block 2p alone, the second both:
    // s0 D0 + s1 D1 = (s0 - s1) D0 + s1 (D0 + D1)
#pragma unroll
    for (int p = 0; p < 8; ++p) {
      const int h = p >> 2, G = p & 3;
      const uint2 q = make_uint2(w.ql[2 * h + (p & 1)].v[0], w.ql[2 * h + (p & 1)].v[1]);
      const uint32_t lx = (G < 2 ? q.x << 2 : q.x >> 2) & 0x3c3c3c3cu, ly = (G < 2 ? q.y << 2 : q.y >> 2) & 0x3c3c3c3cu;
      const uint32_t vx = lx | ((hb[h].x << (6 - 2 * G)) & 0xc0c0c0c0u);
      const uint32_t vy = ly | ((hb[h].y << (6 - 2 * G)) & 0xc0c0c0c0u);
      o.b[2 * p] = (long)(((uint64_t)(vy & keep0) << 32) | (vx & keep0));
      o.b[2 * p + 1] = (long)(((uint64_t)vy << 32) | vx);
      const int s1 = (int)(int8_t)(scb[p >> 1] >> (16 * (p & 1) + 8));
      o.s[2 * p] = (int)(int8_t)(scb[p >> 1] >> (16 * (p & 1))) - s1;
      o.s[2 * p + 1] = s1;
    }
  } else if constexpr (T == T_IQ4_XS) {
    // sub-block sb: weights 8g .. 8g + 7 = low (g < 2) or high nibbles of its qs bytes 8(g & 1) .. +7
    o.d = h2f((uint16_t)(w.hdr.x & 0xffffu));
    const int ns = 4 * (g >> 1);
#pragma unroll
    for (int sb = 0; sb < 8; ++sb) {
      const uint32_t v0 = lut16((w.qs[sb].x >> ns) & 0x0f0f0f0fu, tab[0], tab[1], tab[2], tab[3]);
      const uint32_t v1 = lut16((w.qs[sb].y >> ns) & 0x0f0f0f0fu, tab[0], tab[1], tab[2], tab[3]);
      o.b[sb] = (long)(((uint64_t)v1 << 32) | v0);
      o.s[sb] = iq4_scale(w.hdr.x, w.hdr.y, sb);
    }
  } else {
    // lane group g holds the 8-weight group g of every sub-block: grid values with
    // their signs applied; 1/8 (IQ2_XXS) or 1/4 (IQ3_XXS) folded into d
    o.d = (T == T_IQ2_XXS ? 0.125f : 0.25f) * h2f(w.d);
#pragma unroll
    for (int sb = 0; sb < 8; ++sb) {
      uint32_t glo, ghi, aux;
      if constexpr (T == T_IQ2_XXS) {
        const uint32_t aux0 = w.q.v[2 * sb];
        aux = w.q.v[2 * sb + 1];
        const uint64_t gg = s_tab[(aux0 >> (8 * g)) & 0xffu];
        glo = (uint32_t)gg;
        ghi = (uint32_t)(gg >> 32);
      } else {
        aux = w.sas.v[sb];
        const uint32_t *g3 = reinterpret_cast<const uint32_t *>(s_tab);
        glo = g3[w.gi[sb] & 0xffu];
        ghi = g3[w.gi[sb] >> 8];
      }
      const uint64_t mm = s_signs[(aux >> (7 * g)) & 127u];
      const uint32_t v0 = sign_bytes(glo, (uint32_t)mm), v1 = sign_bytes(ghi, (uint32_t)(mm >> 32));
      o.b[sb] = (long)(((uint64_t)v1 << 32) | v0);
      o.s[sb] = 2 * (int)(aux >> 28) + 1;
    }
  }
}

// ---------------------------------------------------------------- the kernel

// TT: 16-pair tiles per item; NW: waves (16 weight rows each); C: K blocks per stage
// Four waves per SIMD are asked for; 12 of the 64 instantiations reach 3 or 2 (LDS:
// two blocks of both matrices per stage; registers: Q5_K and Q6_K gate/up, 131 to
// 152).  Asked for what they reach, the compiler orders those less well (1024 tokens
// of H 2048 F 768, Q5_K: layer 269 -> 271 us), so its remark on them is turned off.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Wpass-failed"
template <int T, bool GATEUP, int TT, int NW, int C>
static __global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW > 1 ? 4 : 2))) void k_mmq(GemvArgs a) {
  constexpr int TOK = 16 * TT;
  constexpr int NM = GATEUP ? 2 : 1;
  // Blocks are added in runs of 8, and the runs in turn: shorter chains, and no
  // larger rounding error than the GEMV's where that would run (relative to 64
  // bits, rows of 7168, one chain / runs of 8 / GEMV: Q4_K 1.13 / 0.89 / 1.07e-7,
  // Q6_K 1.10 / 0.86 / 0.93e-7).  Four tiles keep one chain, as their second sums
  // would cost the fourth wave per SIMD; not for Q3_K (gate/up, 8 waves with 21
  // spilled registers; with 4 waves and none a layer of 512 tokens takes 494 us
  // instead of 413).
  constexpr bool kTwoLevel = TT <= 2 || T == T_Q3_K;
  constexpr int BB = block_bytes(T);
  constexpr int UN = TOK * XUNITS;          // activation units of a block
  constexpr int NI = (UN + 64 * NW - 1) / (64 * NW);
  constexpr int RU = mmq_units<T, C>(), LU = mmq_load_units<T, C>();
  constexpr int NWI = (16 * RU + 63) / 64;  // weight loads per matrix and stage
  constexpr int WB = 16 * RU * 16;          // LDS bytes of one matrix stage of a wave
  // a stage starts on either half of a dword only where its bytes are no multiple of 4
  constexpr bool kParity = (C * BB) % 4 != 0;
  constexpr bool kGrid = T == T_IQ2_XXS || T == T_IQ3_XXS;
  constexpr int NTAB = T == T_IQ2_XXS ? 256 : (T == T_IQ3_XXS ? 128 : (T == T_Q3_K ? 64 : 1));
  // lookup tables first (largest alignment first), so that their addresses fold into the reads' offset field
  __shared__ __attribute__((aligned(kGrid ? 4096 : 16))) uint64_t s_tab[NTAB];
  __shared__ __attribute__((aligned(kGrid ? 2048 : 8))) uint64_t s_signs[kGrid ? 128 : 1];
  __shared__ __attribute__((aligned(16))) uint8_t s_x[2][C][TOK * XREC];
  __shared__ __attribute__((aligned(16))) uint8_t s_w[NW][NM][WB];
  __shared__ uint32_t s_xoff[TOK];  // byte offset of each pair's activation row (XOOR: none)
  __shared__ long s_out[TOK];   // float offset of each pair's output row (-1: none)
  int e, pc, p1;
  const int li = blockIdx.x / a.row_tiles, rt = blockIdx.x - li * a.row_tiles;
  const int item = a.item0 + li;
  if (a.dense_S > 0) {
    e = 0;
    pc = item * TOK;
    p1 = a.dense_S;
    if (pc >= p1) return;
  } else {
    if (item >= *a.n_items) return;
    const int it = a.items[item];
    e = mmq_item_expert(it);
    pc = a.offs[e] + mmq_item_first(it);
    p1 = a.offs[e + 1];
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int row0 = (rt * NW + wave) * 16;
  const int row = row0 + n;
  const int nb = a.nb;
  const int nt = min(TT, (p1 - pc + 15) / 16);
  if (tid < TOK) {
    int pair = -1;
    if (pc + tid < p1) pair = a.dense_S > 0 ? pc + tid : a.pairs[pc + tid];
    const int Kp = a.dense_S > 0 ? 1 : a.K;
    const int tok = pair / Kp, k = pair - tok * Kp;
    s_xoff[tid] = pair >= 0 ? (uint32_t)((tok * a.ne11 + k % a.ne11) * a.xq_rstride) : XOOR;
    s_out[tid] = pair >= 0 ? (long)((size_t)tok * a.out_s + (size_t)k * a.out_k) : -1;
  }
  if constexpr (T == T_Q3_K) {
    if (tid < 64) {
      uint64_t t = 0;
#pragma unroll
      for (int k = 0; k < 8; ++k) t |= (uint64_t)((uint32_t)((4 - k) * (tid - 32)) & 0xffu) << (8 * k);
      s_tab[tid] = t;
    }
  }
  if constexpr (kGrid) {
    for (int i = tid; i < NTAB; i += 64 * NW) s_tab[i] = a.grid[i];
    for (int i = tid; i < 128; i += 64 * NW) s_signs[i] = a.signs[i];
  }
  uint32_t tab[4] = {0, 0, 0, 0};  // IQ4_XS value table, wave-uniform
  if constexpr (T == T_IQ4_XS) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      tab[2 * i] = (uint32_t)a.grid[i];
      tab[2 * i + 1] = (uint32_t)(a.grid[i] >> 32);
    }
  }
  __syncthreads();
  // activation units of this wave: record u / 19, unit u % 19
  uint32_t xo[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int u = (i * NW + wave) * 64 + lane;
    const int t = u / XUNITS, p = u - XUNITS * t;
    const uint32_t o = t < TOK ? s_xoff[t] : XOOR;
    xo[i] = o != XOOR ? o + 16 * p : XOOR;
  }
  const v4u_t rx = dma_rsrc(a.xq, a.xq_bytes);
  // weight units: row u / RU of the wave's 16, unit u % RU.  The resource starts
  // on a dword; of a 2-byte type the even and the odd blocks of a row start on
  // either half of a dword (al), so each parity has its offsets.  Gate and up
  // lie alike within a dword (the host checks).
  const uint8_t *wm[2] = {a.w0 + (size_t)e * a.w_estride, GATEUP ? a.w1 + (size_t)e * a.w_estride : nullptr};
  const int sh = mmq_dword<T>() ? 0 : (int)((uintptr_t)wm[0] & 3);
  const uint32_t wbytes = ((uint32_t)((size_t)a.nrows * a.w_rstride) + sh + 3) & ~3u;
  v4u_t rw[NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) rw[m] = dma_rsrc(wm[m] - sh, wbytes);
  const int al = mmq_dword<T>() ? 0 : (sh + row * (int)a.w_rstride) & 3;
  int wo[kParity ? 2 : 1][NWI];
#pragma unroll
  for (int i = 0; i < NWI; ++i) {
    const int u = i * 64 + lane;
    const int r = u / RU, p = u - RU * r;
    const bool ok = r < 16 && p < LU && row0 + r < a.nrows;
    const int st = sh + (row0 + r) * (int)a.w_rstride;
    wo[0][i] = ok ? (st & ~3) + 16 * p : OOR;
    if constexpr (kParity) wo[1][i] = ok ? ((st + C * BB) & ~3) + 16 * p : OOR;
  }
  auto dma_w = [&](int m, int s) {  // stage s: blocks s * C ..
    const uint32_t base = lds_addr(&s_w[wave][m][0]);
    const int par = kParity ? s & 1 : 0;
    const int so = (s - par) * (C * BB);
#pragma unroll
    for (int i = 0; i < NWI; ++i) {
      if (64 * (i + 1) > 16 * RU && 64 * i + lane >= 16 * RU) continue;
      const int vo = par ? wo[kParity ? 1 : 0][i] : wo[0][i];
      // a stage that is one block and fills its units exactly never reaches past
      // the resource, whose bounds the scalar offset is not part of; the others
      // add it per lane
      if constexpr (16 * LU == BB) dma_lds16(rw[m], base + i * 1024u, vo, so);
      else dma_lds16(rw[m], base + i * 1024u, vo == OOR ? OOR : vo + so, 0);
    }
  };
  const uint8_t *wl = &s_w[wave][0][0] + n * (RU * 16);

  auto body = [&](auto nt_tag) {
    constexpr int NT = decltype(nt_tag)::value;
    constexpr int NC = mmq_chains<T>();
    constexpr int NIT = (NT * 16 * XUNITS + 64 * NW - 1) / (64 * NW);
    constexpr int NIM = (NT * 16 * XUNITS) / (64 * NW);  // of these, issued by every wave
    auto dma_x = [&](int s, int slot) {
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const uint32_t base = lds_addr(&s_x[0][0][0]) + (slot * C + c) * (uint32_t)(TOK * XREC) + wave * 1024u;
        const int so = min(s * C + c, nb - 1) * XREC;
#pragma unroll
        for (int i = 0; i < NIT; ++i) {
          if ((i * NW + NW) * 64 > UN && (i * NW + wave) * 64 + lane >= UN) continue;
          dma_lds16(rx, base + i * NW * 1024u, (int)xo[i], so);
        }
      }
    };
    v4i_t zero = {0, 0, 0, 0};
    asm("" : "+v"(zero));  // one zero operand for the first MFMA of every chain
    float f[NM][NT][4];
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) f[m][t][j] = 0.f;
    float fs[kTwoLevel ? NM : 1][kTwoLevel ? NT : 1][4] = {};  // sums of 8 blocks
    // request order: x(0) W0(0) W1(0), then per stage W0(s + 1), x(s + 1), W1(s + 1)
    const int ns = (nb + C - 1) / C;
    dma_x(0, 0);
    dma_w(0, 0);
    if constexpr (NM == 2) dma_w(1, 0);
    for (int s = 0; s < ns; ++s) {
      wait_barrier<(NM - 1) * NWI>();  // W0(s) and x(s) have landed; younger: W1(s)
      const uint8_t *xs0 = &s_x[0][0][0] + (s & 1) * (C * TOK * XREC);
      const int sn = min(s + 1, ns - 1);  // past the end: the last stage again, never read
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        if (m == 1) wait_vm<NWI + C * NIM>();  // W1(s); younger: W0(s + 1) and x(s + 1)
        MmqW<T> w[C];
        const int al0 = kParity ? al ^ (2 * (s & 1)) : al;
#pragma unroll
        for (int c = 0; c < C; ++c) {
          // block c starts al0 + c * BB bytes into the slot
          const int o = (c * BB) & ~3, r = (c * BB) & 3;
          if (c == 0) mmq_read_w<T, 16>(wl + m * WB, al0, g, w[c]);
          else if (r == 0) mmq_read_w<T, (BB % 16 ? (BB % 8 ? 4 : 8) : 16)>(wl + m * WB + o, al0, g, w[c]);
          else mmq_read_w<T, 4>(wl + m * WB + o + (al0 ? 4 : 0), al0 ^ 2, g, w[c]);
        }
        wait_lds();
        dma_w(m, sn);                                 // the slot has been read
        if (m == 0) dma_x(sn, (s + 1) & 1);           // every wave is past stage s - 1
#pragma unroll
        for (int c = 0; c < C; ++c) {
          if (C > 1 && s * C + c >= nb) break;
          const uint8_t *xs = xs0 + c * (TOK * XREC);
          MmqB<T> B;
          mmq_unpack<T>(w[c], g, s_tab, s_signs, tab, B);
          asm("" : "+v"(B.d));  // a plain f32 from here on
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            const uint8_t *xt = xs + (16 * t + n) * XREC;
            v4i_t xa[4];
#pragma unroll
            for (int h = 0; h < 4; ++h) xa[h] = *reinterpret_cast<const v4i_t *>(xt + 64 * h + 16 * g);
            float xd[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) xd[j] = *reinterpret_cast<const float *>(xs + (16 * t + 4 * g + j) * XREC + 288);
            if constexpr (mmq_folded<T>()) {
              v4i_t D[NC];
#pragma unroll
              for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int k = 0; k < NC; ++k)
                  D[k] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[q], B.b[k][q], q == 0 ? zero : D[k], 0, 0, 0);
              v4f_t mn;
              if constexpr (mmq_mins<T>()) {
                const v4h_t bs = *reinterpret_cast<const v4h_t *>(xt + 256 + 8 * g);
                mn = __builtin_amdgcn_mfma_f32_16x16x16f16(bs, B.mn, __builtin_bit_cast(v4f_t, zero), 0, 0, 0);
              }
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                int is = D[0][j];
                if constexpr (NC > 1) is += 8 * D[NC > 1 ? 1 : 0][j];
                if constexpr (NC > 2) is += 16 * D[NC > 2 ? 2 : 0][j];
                float v;
                if constexpr (mmq_mins<T>()) v = __builtin_fmaf(B.d, (float)is, -(B.dmin * mn[j]));
                else v = B.d * (float)is;
                f[m][t][j] = __builtin_fmaf(xd[j], v, f[m][t][j]);
                asm volatile("" : "+v"(f[m][t][j]));  // as below
              }
            } else {
              int is[4] = {0, 0, 0, 0};
#pragma unroll
              for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int h = 0; h < 2; ++h) {  // half h of chunk k's operand: 32 values
                  const uint2 xh = h ? make_uint2((uint32_t)xa[k][2], (uint32_t)xa[k][3]) : make_uint2((uint32_t)xa[k][0], (uint32_t)xa[k][1]);
                  const long x8 = __builtin_bit_cast(long, xh);
                  constexpr int PS = MmqB<T>::NB / 8;  // sub-blocks per 32 values
#pragma unroll
                  for (int q = 0; q < PS; ++q) {
                    const int sb = (2 * k + h) * PS + q;
                    const v4i_t D = __builtin_amdgcn_mfma_i32_16x16x32_i8(x8, B.b[sb], zero, 0, 0, 0);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                      is[j] = __mul24(B.s[sb], D[j]) + is[j];
                      asm("" : "+v"(is[j]));  // one multiply-add, not two multiplies and an add of three
                    }
                  }
                }
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                f[m][t][j] = __builtin_fmaf(xd[j], B.d * (float)is[j], f[m][t][j]);
                // computed here: left to float, the tile's operands stay live into the next matrix
                asm volatile("" : "+v"(f[m][t][j]));
              }
            }
          }
        }
      }
      if constexpr (kTwoLevel) {
        if ((s + 1) % (8 / C) == 0 || s + 1 == ns) {
#pragma unroll
          for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                fs[m][t][j] += f[m][t][j];
                f[m][t][j] = s + 1 == ns ? fs[m][t][j] : 0.f;
              }
        }
      }
    }
    wait_vm<0>();  // the requests past the last block land before the LDS is given up
    if (row < a.nrows) {
      // the lane holds (pair 16t + 4g + j, row)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const long o = s_out[16 * t + 4 * g + j];
          if (o < 0) continue;
          a.out[o + row] = GATEUP ? silu_f32(f[0][t][j]) * f[NM - 1][t][j] : f[0][t][j];
        }
    }
  };
  if constexpr (TT == 1) {
    body(std::integral_constant<int, 1>{});
  } else if constexpr (TT == 2) {
    if (nt == 1) body(std::integral_constant<int, 1>{});
    else body(std::integral_constant<int, 2>{});
  } else {
    static_assert(TT == 4, "tiles per item");
    if (nt == 1) body(std::integral_constant<int, 1>{});
    else if (nt == 2) body(std::integral_constant<int, 2>{});
    else if (nt == 3) body(std::integral_constant<int, 3>{});
    else body(std::integral_constant<int, 4>{});
  }
}

#pragma clang diagnostic pop

// ---------------------------------------------------------------- launch

// K blocks per stage of 16-pair items: two where a row's block is no whole
// number of 16-byte units, so that fewer 128-byte lines are fetched twice (a
// line shared by two blocks of a row does not always stay in the L2 from one
// stage to the next: 1.48 times the weights from memory for Q6_K).  24 tokens,
// one / two blocks: Q6_K down 160 / 118 us, Q2_K gate/up 108 / 98, IQ3_XXS gate/up
// 178 / 171, but IQ4_XS gate/up 168 / 188, Q4_K 147 / 150.
template <int T>
constexpr int mmq_stage() {
  return T == T_Q4_K || T == T_IQ4_XS ? 1 : 2;
}
// waves per workgroup: 8 with 64-pair items (4 where 8 waves' weights leave LDS
// for one workgroup only: Q5_K gate/up 288 against 304 us), else 4, or 1 where even their 64-row tiles leave CUs
// idle.  512 tokens, Q4_K gate/up: 64-pair items with 8 waves 260 us, with 4
// waves 294, 32-pair items 289; 333 tokens (21 pairs per expert), Q3_K down: 155
// / 170 / 126.
template <int T, bool GU>
void mmq_launch_t(int tt, int nw, unsigned items, const GemvArgs &a0, hipStream_t st) {
  constexpr int NW4 = GU && (T == T_Q5_K || T == T_Q6_K) ? 4 : 8;
  GemvArgs a = a0;
  if (tt == 4) nw = NW4;
  a.row_tiles = (a.nrows + 16 * nw - 1) / (16 * nw);
  // a grid has fewer than 2^32 threads: matrices of millions of rows take several
  const unsigned most = (unsigned)(0xffffffffu / (64u * nw) / (unsigned)a.row_tiles);
  for (unsigned i = 0; i < items; i += most) {
    a.item0 = (int)i;
    const dim3 grid((unsigned)a.row_tiles * std::min(most, items - i));
    if (tt == 4) hipLaunchKernelGGL((k_mmq<T, GU, 4, NW4, 1>), grid, dim3(64 * NW4), 0, st, a);
    else if (nw == 1) hipLaunchKernelGGL((k_mmq<T, GU, 2, 1, 1>), grid, dim3(64), 0, st, a);
    else if (tt == 1) hipLaunchKernelGGL((k_mmq<T, GU, 1, 4, mmq_stage<T>()>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((k_mmq<T, GU, 2, 4, 1>), grid, dim3(256), 0, st, a);
  }
}
template <int T>
void mmq_launch(bool gateup, int tt, int nw, unsigned items, const GemvArgs &a, hipStream_t st) {
  if (gateup) mmq_launch_t<T, true>(tt, nw, items, a, st);
  else mmq_launch_t<T, false>(tt, nw, items, a, st);
}
// per translation unit: false when the type is not instantiated there
bool mmq_launch_a(int type, bool gateup, int tt, int nw, unsigned items, const GemvArgs &a, hipStream_t st);
bool mmq_launch_b(int type, bool gateup, int tt, int nw, unsigned items, const GemvArgs &a, hipStream_t st);
bool mmq_launch_c(int type, bool gateup, int tt, int nw, unsigned items, const GemvArgs &a, hipStream_t st);
bool mmq_launch_d(int type, bool gateup, int tt, int nw, unsigned items, const GemvArgs &a, hipStream_t st);

}  // namespace zm
