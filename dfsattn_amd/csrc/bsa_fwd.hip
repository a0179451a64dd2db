// Block-sparse flash-attention forward for gfx950 (replaces the external
// block_sparse_attn_func called at dfsattn/attention_wan.py:379-386 and
// dfsattn/attention_hyvideo.py:1075-1082).
//
// Each wave computes S^T = K Q^T with v_mfma_f32_32x32x16 (lane column =
// query, registers = keys), so the online-softmax row statistics need one
// exchange between the two lane halves only. P is rounded to f16 (or bf16)
// and multiplied with V^T as O^T += V^T P^T; the register order of the S^T
// accumulator is reused as the token order of the PV operand, which the V^T
// layout matches. K (row-major) and V^T (transposed by the permute kernel)
// tiles are copied straight from global memory into LDS with 16-byte buffer
// loads.
//
// Schedule: one workgroup = one (head, 128-row query block), four waves of 32
// query rows walking the row's kept key blocks; two workgroups per CU, single
// K and V buffers, the K copy of the next block overlapping softmax and PV,
// the V copy overlapping the next QK^T; the other workgroup on the CU fills
// the gaps. With f16 operands the row's reference maximum comes from its first
// block and later blocks skip the maximum (a block is redone only if its P
// overflows); bf16 operands, whose P has 8 bits, keep the running maximum.
// The LDS operand reads run four MFMAs ahead, and the QK phase runs at raised
// wave priority. A row visits its key blocks in order of distance from its own
// block, so neighbouring query blocks fetch shared key blocks together.
//
// LDS rows are 256 bytes; 16-byte chunk c of row r is stored at chunk
// c ^ (r % 16) so the 32 rows read by one MFMA operand fetch hit distinct
// banks.
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include <type_traits>

#include "common.h"
#include "head_range.h"
#include "lds_copy.h"

namespace dfs {
namespace {

struct BsaParams {
  // L: query rows computed, Lk: keys attended (host values; segment 0 of
  // device cu_seqlens replaces them per workgroup); R: operand rows per head;
  // Lo: out / lse rows per head; Qb = ceil(L / 128) sets the grid, Kb =
  // ceil(Lk / 128); csr_qb: CSR rows per head (the mask may have been
  // selected over a longer sequence).
  int H, L, Lk, R, Qb, Kb, Lo, csr_qb;
  float scale_log2;
  int scale_all;  // 1: every head runs in the scaled instance (f16 q * c may reach 2^15)
  int out_kind;  // 0 bf16, 1 f16, 2 f32
  // Optional device arrays: cu_q / cu_k, segment offsets in execution order
  // (segment 0 = [0, cu[1])); exps [3][H], per-head power-of-two exponents
  // of the f16 operands (q_perm, k_perm, v_t hold x * 2^-e).
  const int32_t* cu_q;
  const int32_t* cu_k;
  const int32_t* exps;
  // Optional Q source read in place of q_perm: execution row r < L is input
  // row q_rows[r] of q_src ([H][L][D], f16 when q_src_f16, else bf16), rows
  // past L are zero. Its exponent exps[0][h] is then only a range mark: the
  // values are read unscaled.
  const uint16_t* q_src;
  const int32_t* q_rows;
  int64_t q_sh, q_sl;  // element strides of q_src between heads and between rows
  int q_src_f16;
  // Optional, = exps when nobody has looked at Q's range yet: the common
  // instance sets word h, and the query block's word of q_block_marks [H][Qb],
  // when a row of its Q leaves the f16 range, and leaves the block to the scaled
  // instance, launched behind it. The common instance never reads these words
  // (head_range.h).
  int32_t* q_marks;
  int32_t* q_block_marks;
  // Element strides of out between heads and between rows.
  int64_t o_sh, o_sl;
  // Order and split of the work (see wg_work): query blocks from long_row on
  // are started first, each by long_parts workgroups; of an XCD's other query
  // blocks the first full_rows are one workgroup each and the rest parts.
  int long_row, long_parts, full_rows, parts;
  int chunks;  // contiguous ranges a head's ordinary query blocks are dealt to XCDs in (1, 2, 4 or 8)
  // Partial results of split query blocks: O [slot][128][D] and (m, l)
  // [slot][128][2], fp32, m in log2 units.
  float* part_o;
  float* part_ml;
};

// Start of the D-element Q row of execution row qrow of head h: q_perm's row,
// or the input row it comes from (nullptr for a zero row past L). f16 tells
// whether the row holds f16 (else bf16) values.
template <int D>
__device__ __forceinline__ const uint16_t* q_row_ptr(const uint16_t* __restrict__ q, const BsaParams& p, int h,
                                                     int qrow, bool& f16) {
  if (p.q_src) {
    f16 = p.q_src_f16 != 0;
    if (qrow >= p.L) return nullptr;
    return p.q_src + h * p.q_sh + p.q_rows[qrow] * p.q_sl;
  }
  f16 = true;
  return q + (static_cast<int64_t>(h) * p.R + qrow) * D;
}

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

template <bool F16>
struct MfmaOp;
template <>
struct MfmaOp<false> {
  typedef bf16x8 vec;
  typedef bf16x2 pair;
  static __device__ __forceinline__ f32x16 run(vec a, vec b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  // One v_cvt_pk (round to nearest even) per pair.
  static __device__ __forceinline__ pair pack(float x, float y) {
    return __builtin_convertvector((f32x2){x, y}, pair);
  }
  // acc + x.lo + x.hi in fp32 (v_dot2 with ones).
  static __device__ __forceinline__ float sum2(pair x, float acc) {
    return __builtin_amdgcn_fdot2_f32_bf16(x, (pair){(__bf16)1.0f, (__bf16)1.0f}, acc, false);
  }
};
template <>
struct MfmaOp<true> {
  typedef f16x8 vec;
  typedef f16x2 pair;
  static __device__ __forceinline__ f32x16 run(vec a, vec b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ pair pack(float x, float y) {
    return __builtin_convertvector((f32x2){x, y}, pair);
  }
  static __device__ __forceinline__ float sum2(pair x, float acc) {
    return __builtin_amdgcn_fdot2(x, (pair){(_Float16)1.0f, (_Float16)1.0f}, acc, false);
  }
};

// Value of the other lane half (lane ^ 32) combined with this lane's.
__device__ __forceinline__ float xhalf_max(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xhalf_sum(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Work of one workgroup: a query block of a head, or part `piece` of the
// `pieces` its column list is cut into, whose result goes to partial slot
// `slot`.
struct Work {
  int h, qb, piece, pieces, slot;
};

// Split query blocks come in two lists: the long ones (8 * ceil(heads *
// blocks / 8), when long_parts > 1), then the tails of the XCDs' lists.
__host__ __device__ inline int long_per_head(const BsaParams& p) { return p.Qb - p.long_row; }
__host__ __device__ inline int long_per_xcd(const BsaParams& p) { return (p.H * long_per_head(p) + 7) >> 3; }
__host__ __device__ inline int chunk_blocks(const BsaParams& p) { return (p.long_row + p.chunks - 1) / p.chunks; }
__host__ __device__ inline int blocks_per_xcd(const BsaParams& p) {
  return ((p.H * p.chunks + 7) >> 3) * chunk_blocks(p);
}
__host__ __device__ inline int split_long(const BsaParams& p) { return p.long_parts > 1 ? 8 * long_per_xcd(p) : 0; }
__host__ __device__ inline int split_tail(const BsaParams& p) {
  return p.parts > 1 ? 8 * (blocks_per_xcd(p) - p.full_rows) : 0;
}
// Query block i of XCD x's list of ordinary blocks; false for a padding slot.
__device__ __forceinline__ bool ordinary_block(const BsaParams& p, int x, int i, int& h, int& qb) {
  const int S = chunk_blocks(p), u = i / S;
  const int g = u * 8 + x;  // this XCD's u-th (head, range)
  h = g / p.chunks;
  qb = ((g + h) & (p.chunks - 1)) * S + (i - u * S);
  return h < p.H && qb < p.long_row;
}
__device__ __forceinline__ bool long_block(const BsaParams& p, int g, int& h, int& qb) {
  const int n = long_per_head(p);
  h = g / n;
  qb = p.long_row + (g - h * n);
  return h < p.H;
}

// Work of this workgroup; false for a padding slot. Hardware deals workgroup
// b to XCD b % 8 and each XCD runs its workgroups in increasing b.
//  * Ordinary query blocks: a head's are dealt in `chunks` contiguous ranges,
//    range g of all heads to XCD g % 8, so that an XCD's L2 serves neighbouring
//    query blocks of 8 / chunks heads in flight. Fewer, longer ranges share
//    more key blocks per L2 as long as the K/V of the heads in flight stays in
//    the 256 MB last-level cache (head_chunks in the Python layout module):
//    whole calls in turn, 20,280 tokens x 40 heads 1,769 us with 8 ranges,
//    1,738 with 4, 1,702 with 1; 4,680 x 40: 169 with 8, 155 with 1; 75,600 x 40
//    (38.7 MB a head): 32.24 ms with 8, 31.90 with 4, 32.05 with 2, 32.41 with 1
//    (a card drifts by about 1%). The ranges rotate with the head.
//  * Long query blocks (HunyuanVideo's text rows keep every key block, three
//    times the others at sparsity 0.3) go first: started in their place at the
//    end of their head, the last head's ran on alone after everything else.
//  * Where the workgroups would not fill the chip's slots evenly, the last
//    blocks of every XCD's list (all of them for small problems) are cut into
//    parts along their columns and bsa_combine_kernel adds the parts up.
__device__ __forceinline__ bool wg_work(const BsaParams& p, Work& wk) {
  const int x = blockIdx.x & 7;
  int j = blockIdx.x >> 3;
  const int n_long = long_per_xcd(p) * p.long_parts;
  if (j < n_long) {
    const int g = j / p.long_parts;
    wk.piece = j - g * p.long_parts;
    wk.pieces = p.long_parts;
    wk.slot = (g * 8 + x) * p.long_parts + wk.piece;
    return long_block(p, g * 8 + x, wk.h, wk.qb);
  }
  j -= n_long;
  int i = j;
  wk.piece = 0;
  wk.pieces = 1;
  wk.slot = 0;
  if (j >= p.full_rows && p.parts > 1) {
    const int t = (j - p.full_rows) / p.parts;
    wk.piece = j - p.full_rows - t * p.parts;
    wk.pieces = p.parts;
    wk.slot = split_long(p) * p.long_parts + (t * 8 + x) * p.parts + wk.piece;
    i = p.full_rows + t;
  }
  return ordinary_block(p, x, i, wk.h, wk.qb);
}

// This lane's share of a Q row as it lies in memory (16-byte chunk 2 s + hl
// of every 32); f16 tells its type. Issued before the column list is built:
// the permutation read and the row read then run under it.
template <int D>
__device__ __forceinline__ void load_q_raw(const uint16_t* __restrict__ q, const BsaParams& p, int h, int qrow, int hl,
                                           uint4* raw, bool& f16) {
  const uint4* src = reinterpret_cast<const uint4*>(q_row_ptr<D>(q, p, h, qrow, f16));
#pragma unroll
  for (int s = 0; s < D / 16; ++s) raw[s] = src ? src[2 * s + hl] : make_uint4(0, 0, 0, 0);
}

// Keys >= valid of the block get -inf (only the last block can be partial).
__device__ __forceinline__ void mask_tail(f32x16* s, int valid, int hl) {
#pragma unroll
  for (int kc = 0; kc < 4; ++kc)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      if (kc * 32 + (r >> 2) * 8 + hl * 4 + (r & 3) >= valid) s[kc][r] = -INFINITY;
}

// Whether a finite bf16 value of this lane's share of a Q row reaches 2^15
// times c (an infinity or NaN stays what it is in either instance). Looked at
// here, a reused mask's call is spared the read of Q in the preparation (35 us
// of 190 at 20,280 tokens x 40 heads).
template <int D>
__device__ __forceinline__ bool q_beyond_f16(const uint4* raw, float c) {
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  // Magnitudes order as their bits; the finite ones end at 0x7f7f.
  auto largest = [&](auto&& keep) {
    u16x2 mx = {0, 0};
#pragma unroll
    for (int s = 0; s < D / 16; ++s) {
      const uint32_t w[4] = {raw[s].x, raw[s].y, raw[s].z, raw[s].w};
#pragma unroll
      for (int i = 0; i < 4; ++i)
        mx = __builtin_elementwise_max(mx, keep(__builtin_bit_cast(u16x2, w[i] & 0x7fff7fffu)));
    }
    return bf16_bits_to_f32(max(mx[0], mx[1])) * c;
  };
  if (largest([](u16x2 m) { return m; }) < 32768.f) return false;
  return largest([](u16x2 m) {  // rare: infinities and NaN become 0
    const u16x2 over = __builtin_elementwise_min(__builtin_elementwise_sub_sat(m, (u16x2)(0x7f7f)), (u16x2)(1));
    return __builtin_elementwise_sub_sat(m, over << (u16x2)(15));
  }) >= 32768.f;
}

// f16 Q fragments with c = scale * log2(e) folded in (q * c rounded to f16),
// so that S^T = K (Q c)^T arrives in log2 units. In the SCALED instance the
// per-head exponents of the f16 operands enter c exactly (q_perm holds
// q 2^-eq and k_perm k 2^-ek, so c' = c 2^(eq + ek)), and a row whose q * c'
// would leave the f16 range is stored as q c' 2^-r (r > 0, the smallest
// power of two that fits): its S arrives as S 2^-r and the kernel multiplies
// it by row_scale = 2^r. The common instance runs heads without exponents at
// a scale where |q c| < 2^15 always holds (f16 q_perm values, or Q source
// values of a head inside the f16 range, times c < 0.5; q_beyond_f16 looks
// where that is not known).
template <int D, bool SCALED>
__device__ __forceinline__ void scale_q(const uint4* raw, bool f16, const BsaParams& p, int h, f16x8* qf,
                                        float& row_scale) {
  float c = p.scale_log2;
  // q_perm holds q 2^-eq; a Q source is read unscaled
  if (SCALED && p.exps) c = ldexpf(c, (p.q_src ? 0 : p.exps[h]) + p.exps[p.H + h]);
  float x[D / 16][8];
  float mx = 0.f;
#pragma unroll
  for (int s = 0; s < D / 16; ++s) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      x[s][i] = (f16 ? f16_bits_to_f32(u16_at(raw[s], i)) : bf16_bits_to_f32(u16_at(raw[s], i))) * c;
      if (SCALED) mx = fmaxf(mx, fabsf(x[s][i]));
    }
  }
  float inv = 1.f;
  row_scale = 1.f;
  if (SCALED) {
    mx = xhalf_max(mx);
    // 2^15 bounds |q c'| after the shift, with room below the f16 maximum.
    const int r = mx >= 32768.f ? ilogbf(mx) - 14 : 0;
    inv = ldexpf(1.f, -r);
    row_scale = ldexpf(1.f, r);
  }
#pragma unroll
  for (int s = 0; s < D / 16; ++s)
#pragma unroll
    for (int i = 0; i < 8; ++i) qf[s][i] = static_cast<_Float16>(x[s][i] * inv);
}

// Lazy online softmax on S' = S - m (f16 operands, log2 units), where the
// running reference m enters through the QK MFMA's C input (negm holds -m in
// every element, times qinv = 2^-r for a row whose Q fragments carry 2^-r). On
// a row's first block m becomes the block maximum; later, m moves only when
// some row of the wave sees a block maximum above m + kLazyTau, and O and l
// are rescaled then. The result is the same softmax: numerator and denominator
// share the reference. The kernel calls this only for a row's first block and
// for a block whose P overflowed f16.
constexpr float kLazyTau = 8.0f;
template <int DCH>
__device__ __forceinline__ void softmax_lazy(f32x16* s, bool first, float& m, float& lsum, f32x16* o, f32x16& negm,
                                             float qinv = 1.f) {
  float mx = -INFINITY;
#pragma unroll
  for (int kc = 0; kc < 4; ++kc)
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[kc][r]);
  const float bm = xhalf_max(mx);
  if (first || __any(bm > kLazyTau)) {
    float shift = first ? bm : fmaxf(bm, 0.f);
    if (!(shift > -INFINITY)) shift = 0.f;  // a row with every key masked keeps m
#pragma unroll
    for (int kc = 0; kc < 4; ++kc)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[kc][r] -= shift;
    if (!first) {
      const float alpha = exp2_fast(-shift);
      lsum *= alpha;
#pragma unroll
      for (int i = 0; i < DCH; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[i][r] *= alpha;
    }
    m += shift;
#pragma unroll
    for (int r = 0; r < 16; ++r) negm[r] = -m * qinv;  // rows stored as Q c 2^-r: the C input is -m 2^-r
  }
}

// Scheduling of an MFMA phase: the LDS operand reads run kAhead MFMAs ahead
// of their MFMAs, so each read's latency is covered by the MFMAs before its
// use (the two waves of a SIMD come from independent workgroups and often
// read at the same time).
// Pinned with scheduling-group barriers:
// kAhead reads, then alternately one MFMA and one read, then the last MFMAs.
constexpr int kAhead = 4;
template <int N>
__device__ __forceinline__ void pin_read_ahead_schedule() {
  constexpr int kMfma = 0x008, kDsRead = 0x100;
  __builtin_amdgcn_sched_group_barrier(kDsRead, kAhead, 0);
#pragma unroll
  for (int i = 0; i < N - kAhead; ++i) {
    __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
    __builtin_amdgcn_sched_group_barrier(kDsRead, 1, 0);
  }
  __builtin_amdgcn_sched_group_barrier(kMfma, kAhead, 0);
}

// O^T += V^T P^T from an LDS V^T tile and P held in registers.
template <int D, typename PvOp>
__device__ __forceinline__ void pv_tile_regs(const uint16_t* v_tile, const typename PvOp::vec* pf, f32x16* o, int l32,
                                             int hl) {
  constexpr int DCH = D / 32, N = 8 * DCH;
  uint4 a[N];
#pragma unroll
  for (int i = 0; i < N; ++i) a[i] = lds_chunk<16>(v_tile, (i % DCH) * 32 + l32, (i / DCH) * 2 + hl);
#pragma unroll
  for (int i = 0; i < N; ++i)
    o[i % DCH] = PvOp::run(__builtin_bit_cast(typename PvOp::vec, a[i]), pf[i / DCH], o[i % DCH]);
  pin_read_ahead_schedule<N>();
}

// S^T = init + K Q^T from an LDS K tile, with the read-ahead schedule above.
template <int D, typename QkOp>
__device__ __forceinline__ void qk_tile_ahead(const uint16_t* k_tile, const typename QkOp::vec* qf, int l32, int hl,
                                              f32x16* s, const f32x16& init) {
  constexpr int CPR = D / 8, DS = D / 16, N = 4 * DS;
  uint4 a[N];
#pragma unroll
  for (int i = 0; i < N; ++i) a[i] = lds_chunk<CPR>(k_tile, (i / DS) * 32 + l32, (i % DS) * 2 + hl);
#pragma unroll
  for (int kc = 0; kc < 4; ++kc) s[kc] = init;
#pragma unroll
  for (int i = 0; i < N; ++i)
    s[i / DS] = QkOp::run(__builtin_bit_cast(typename QkOp::vec, a[i]), qf[i % DS], s[i / DS]);
  pin_read_ahead_schedule<N>();
}

// Running maximum of bf16 operands' scores (S = q.k, c = scale * log2(e); m
// in log2 units), with O and l rescaled when some row's maximum moved. Taken
// for every block: a row's largest weights are then 1 exactly or near it, and
// with P rounded to 8 bits they carry most of the error. Against a reference
// from the row's first block, as f16 operands use it, the error against 64
// bits was 2.5 to 9% larger (1.558e-3 -> 1.627e-3 at 8,191 tokens) and O
// overflowed fp32 for |V| a thousand times smaller; a call of 32,760 tokens x
// 12 heads took 1.82 ms that way, 1.95 with the maximum.
template <int DCH>
__device__ __forceinline__ void softmax_max(const f32x16* s, float c, float& m, float& lsum, f32x16* o) {
  float mx = -INFINITY;
#pragma unroll
  for (int kc = 0; kc < 4; ++kc)
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[kc][r]);
  const float mnew = fmaxf(m, xhalf_max(mx) * c);
  if (__any(mnew > m)) {
    const float alpha = exp2_fast(m - mnew);
    lsum *= alpha;
#pragma unroll
    for (int i = 0; i < DCH; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[i][r] *= alpha;
  }
  m = mnew;
}

// P of a whole block as PV operands, added (the rounded values, this lane's
// share of the row) to lsum. LOG2: S' arrives in log2 units relative to m;
// otherwise P = exp2(S c - m).
template <typename PvOp, bool LOG2>
__device__ __forceinline__ void make_p(const f32x16* s, float c, float m, typename PvOp::vec* pf, float& lsum) {
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) {
    const f32x16& src = s[ks >> 1];
    const int r0 = (ks & 1) * 8;
    typename PvOp::pair pr[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float x0 = src[r0 + 2 * j], x1 = src[r0 + 2 * j + 1];
      pr[j] = PvOp::pack(exp2_fast(LOG2 ? x0 : fmaf(x0, c, -m)), exp2_fast(LOG2 ? x1 : fmaf(x1, c, -m)));
      lsum = PvOp::sum2(pr[j], lsum);
    }
    pf[ks] = __builtin_bit_cast(typename PvOp::vec, pr);
  }
}

// O = O^T / l for row qrow, columns d = dc*32 + g*8 + hl*4 + (0..3), times
// 2^ev for a V operand stored as v 2^-ev; rows past L are dropped, rows with
// no kept block give 0.
template <int D>
__device__ __forceinline__ void store_out(const BsaParams& p, int Lq, int ev, void* __restrict__ out,
                                          const int32_t* __restrict__ out_perm, float* __restrict__ lse,
                                          const f32x16* o, float m, float lsum, int h, int qrow, int hl) {
  constexpr int DCH = D / 32;
  const float ltot = xhalf_sum(lsum);
  const float inv = ltot > 0.f ? ldexpf(1.0f / ltot, ev) : 0.f;  // v_t holds v 2^-ev
  if (qrow >= Lq) return;
  const int orow = out_perm ? out_perm[qrow] : qrow;
  const int64_t obase = h * p.o_sh + orow * p.o_sl;
#pragma unroll
  for (int dc = 0; dc < DCH; ++dc)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d0 = dc * 32 + g * 8 + hl * 4;
      const float v0 = o[dc][g * 4 + 0] * inv, v1 = o[dc][g * 4 + 1] * inv;
      const float v2 = o[dc][g * 4 + 2] * inv, v3 = o[dc][g * 4 + 3] * inv;
      if (p.out_kind == DFS_DTYPE_F32) {
        *reinterpret_cast<float4*>(static_cast<float*>(out) + obase + d0) = make_float4(v0, v1, v2, v3);
      } else if (p.out_kind == DFS_DTYPE_BF16) {
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(out) + obase + d0) =
            make_uint2(f32_to_bf16_bits(v0) | (f32_to_bf16_bits(v1) << 16),
                       f32_to_bf16_bits(v2) | (f32_to_bf16_bits(v3) << 16));
      } else {
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(out) + obase + d0) =
            make_uint2(f32_to_f16_bits(v0) | (f32_to_f16_bits(v1) << 16),
                       f32_to_f16_bits(v2) | (f32_to_f16_bits(v3) << 16));
      }
    }
  if (lse && hl == 0)
    lse[static_cast<int64_t>(h) * p.Lo + qrow] = ltot > 0.f ? (m + log2f(ltot)) * 0.69314718055994531f : -INFINITY;
}

// This wave's 32 rows of a part: O, m (log2 units) and l as they are.
template <int D>
__device__ __forceinline__ void store_part(const BsaParams& p, int slot, const f32x16* o, float m, float lsum, int w,
                                           int l32, int hl) {
  const float ltot = xhalf_sum(lsum);
  const int64_t row = static_cast<int64_t>(slot) * 128 + w * 32 + l32;
  float* dst = p.part_o + row * D;
#pragma unroll
  for (int dc = 0; dc < D / 32; ++dc)
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<float4*>(dst + dc * 32 + g * 8 + hl * 4) =
          make_float4(o[dc][g * 4 + 0], o[dc][g * 4 + 1], o[dc][g * 4 + 2], o[dc][g * 4 + 3]);
  if (hl == 0) *reinterpret_cast<float2*>(p.part_ml + row * 2) = make_float2(m, ltot);
}

// Column list of one CSR row into LDS, ordered by distance |c - qb| from the
// row's own block (c = qb first, then qb - 1, qb + 1, qb - 2, ...). The
// workgroups resident on an XCD at one time run neighbouring Hilbert query
// blocks, whose kept columns cluster around their diagonals, so they fetch
// the same key blocks at about the same time (2% fewer L2 misses than
// ascending order with the partner row's shared columns first, 0.4-1.2%
// faster). Columns live in a bitmap at bit 2|c - qb| + (c > qb), compacted in
// bit order. Columns >= Kb (the keys' blocks) are dropped, and all of them
// where skip() of some thread says so (asked last, when its operands have had
// the list's time to arrive). bm: 2 W + 2 words of LDS scratch, W = (2 Kb +
// 31) / 32. Every thread of the NT-thread workgroup calls this; it returns the
// number of columns, the same to all of them, written to cols.
template <int NT, typename Skip>
__device__ int distance_order_cols(int Kb, const int32_t* __restrict__ col_idx, int qb, int beg, int n,
                                   int32_t* cols, uint32_t* bm, int tid, int w, int lane, Skip&& skip) {
  const int W = (2 * Kb + 31) >> 5;
  for (int i = tid; i < W; i += NT) bm[i] = 0u;
  uint32_t* const skipped = bm + 2 * W + 1;
  if (tid == 0) *skipped = 0u;
  block_barrier();
  for (int i = tid; i < n; i += NT) {
    const int c = col_idx[beg + i];
    if (static_cast<unsigned>(c) < static_cast<unsigned>(Kb)) {
      const int b = 2 * (c >= qb ? c - qb : qb - c) + (c > qb ? 1 : 0);
      atomicOr(&bm[b >> 5], 1u << (b & 31));
    }
  }
  block_barrier();
  // First column position of each word into pre[] (one wave scans), then every
  // thread places its own columns.
  uint32_t* const pre = bm + W;
  if (w == 0) {
    const int per = (W + 63) >> 6;
    const int w0 = lane * per;
    int cnt = 0;
    for (int j = 0; j < per && w0 + j < W; ++j) cnt += __popc(bm[w0 + j]);
    int incl = cnt;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int y = __shfl_up(incl, off, 64);
      if (lane >= off) incl += y;
    }
    uint32_t pos = static_cast<uint32_t>(incl - cnt);
    for (int j = 0; j < per && w0 + j < W; ++j) {
      pre[w0 + j] = pos;
      pos += __popc(bm[w0 + j]);
    }
    if (lane == 63) pre[W] = static_cast<uint32_t>(incl);  // this row's count
  }
  block_barrier();
  for (int i = tid; i < n; i += NT) {
    const int c = col_idx[beg + i];
    if (static_cast<unsigned>(c) < static_cast<unsigned>(Kb)) {
      const int b = 2 * (c >= qb ? c - qb : qb - c) + (c > qb ? 1 : 0);
      cols[pre[b >> 5] + __popc(bm[b >> 5] & ((1u << (b & 31)) - 1u))] = c;
    }
  }
  if (skip()) *skipped = 1u;
  block_barrier();
  return *skipped ? 0 : static_cast<int>(pre[W]);
}

#define BSA_KERNEL_ARGS                                                                                \
  const uint16_t *__restrict__ q, const uint16_t *__restrict__ k, const uint16_t *__restrict__ vt,    \
      const int32_t *__restrict__ row_ptr, const int32_t *__restrict__ col_idx, void *__restrict__ out, \
      const int32_t *__restrict__ out_perm, float *__restrict__ lse, BsaParams p_in

// Split schedule: two workgroups per CU, single K and V buffers.
// One (head, 128-row query block) of the split schedule.
// VARLEN: segment 0 of device cu_seqlens sets the rows and keys (a separate
// instance, so the common one keeps the host lengths as kernel arguments).
// SCALED: rows whose q * c' would leave the f16 range carry 2^-r and S is
// multiplied back by 2^r (the rare instance, for heads with exponents).
template <int D, bool QK_F16, bool PV_F16, bool VARLEN, bool SCALED>
__device__ __forceinline__ void bsa_split_block(const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
                                                const uint16_t* __restrict__ vt,
                                                const int32_t* __restrict__ row_ptr,
                                                const int32_t* __restrict__ col_idx, void* __restrict__ out,
                                                const int32_t* __restrict__ out_perm, float* __restrict__ lse,
                                                const BsaParams& p, const Work& wk, uint16_t* k_lds,
                                                uint16_t* v_lds, int32_t* cols) {
  const int h = wk.h, qb = wk.qb;
  constexpr int DCH = D / 32;
  constexpr int K_LOADS = D / 16;  // buffer loads per thread for a K tile
  constexpr int V_LOADS = D / 16;  // ... for a V^T tile (D rows x 256 bytes)
  constexpr uint32_t TILE_BYTES = 128 * D * 2;
  typedef MfmaOp<QK_F16> QkOp;
  typedef MfmaOp<PV_F16> PvOp;
  // Segment 0 of device cu_seqlens: its query rows and keys (offsets are
  // trusted, as by the reference's varlen kernel, and clamped to the call).
  const int Lq = VARLEN ? min(max(p.cu_q[1], 0), p.L) : p.L;
  const int Lk = VARLEN ? min(max(p.cu_k[1], 0), p.Lk) : p.Lk;
  const int Kb = (Lk + 127) >> 7;
  if (qb * 128 >= Lq) return;  // no row of this block is in the segment
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, hl = lane >> 5, l32 = lane & 31;
  const int64_t row = static_cast<int64_t>(h) * p.csr_qb + qb;
  const int beg = row_ptr[row];
  // A row holds at most as many blocks as the mask has columns (capped by the
  // call's own key blocks; columns past the segment's keys are dropped below).
  const int end = beg + min(max(row_ptr[row + 1] - beg, 0), p.Kb);
  const int qrow = qb * 128 + w * 32 + l32;

  f32x16 o[DCH];
#pragma unroll
  for (int i = 0; i < DCH; ++i) o[i] = f32x16{};
  // f16 Q/K: S arrives in log2 units relative to m (lazy softmax); bf16 Q/K:
  // S = q.k and m is the running maximum.
  float m = QK_F16 ? 0.f : -INFINITY, lsum = 0.f;

  if (beg < end) {
    const uint32_t head_bytes = static_cast<uint32_t>(p.R) * D * 2;
    const auto krs = make_rsrc(k + static_cast<int64_t>(h) * p.R * D, head_bytes);
    const auto vrs = make_rsrc(vt + static_cast<int64_t>(h) * p.R * D, head_bytes);
    void* const k_base = k_lds;
    void* const v_base = v_lds;
    const int ws = __builtin_amdgcn_readfirstlane(w);
    const TileCopy<D * 2> kcopy(ws, lane);
    const TileCopy<256> vcopy(ws, lane);
    typename QkOp::vec qf[D / 16];
    float row_scale = 1.f;  // 2^r of a row whose Q fragments carry 2^-r (SCALED)
    bool q_f16;  // the bf16-operand path takes bf16 rows only (q_perm or a bf16 q_src)
    uint4 q_raw[D / 16];
    load_q_raw<D>(q, p, h, qrow, hl, q_raw, q_f16);
    // Column list of this row into LDS (read back with uniform ds_reads).
    // A block with a row of Q beyond the f16 range is left to the scaled
    // instance, whole: its waves agree through the list's barriers.
    auto left_to_scaled = [&] {
      if (!QK_F16 || SCALED || !p.q_marks || !q_beyond_f16<D>(q_raw, p.scale_log2)) return false;
      p.q_marks[h] = 1;  // every writer stores the same marks
      p.q_block_marks[static_cast<int64_t>(h) * p.Qb + qb] = 1;
      return true;
    };
    const int total = __builtin_amdgcn_readfirstlane(
        distance_order_cols<256>(Kb, col_idx, qb, beg, end - beg, cols, reinterpret_cast<uint32_t*>(cols + p.Kb), tid,
                                 w, lane, left_to_scaled));
    // This workgroup's part of the list (all of it for an unsplit block).
    const int t0 = SCALED ? 0 : total * wk.piece / wk.pieces;
    const int n = SCALED ? total : total * (wk.piece + 1) / wk.pieces;
    auto col_at = [&](int t) -> int { return __builtin_amdgcn_readfirstlane(cols[t]); };
    // n == t0: nothing to do for this part, or every kept column lies past
    // this sequence's keys (a shorter key segment), so cols holds nothing to
    // copy; the row stays empty. n is the same for every wave (read from LDS
    // after a barrier).
    int kb = n > t0 ? col_at(t0) : 0;
    if (n > t0) {
      kcopy.template issue<K_LOADS>(krs, kb * TILE_BYTES, k_base, ws);
      vcopy.template issue<V_LOADS>(vrs, kb * TILE_BYTES, v_base, ws);
    }

    // Q fragments, made under the first copies and forced complete here so no
    // wait for them lands in the loop.
    if constexpr (QK_F16)
      scale_q<D, SCALED>(q_raw, q_f16, p, h, qf, row_scale);
    else
#pragma unroll
      for (int s = 0; s < D / 16; ++s) qf[s] = __builtin_bit_cast(typename QkOp::vec, q_raw[s]);
    const float qinv = 1.f / row_scale;
    f32x16 negm = f32x16{};  // -m (times 2^-r) in every element
#pragma unroll
    for (int s = 0; s < D / 16; ++s) asm volatile("" ::"v"(qf[s]));

    for (int t = t0; t < n; ++t) {
      // After the last block the copies reload the current block into the
      // buffers it has just left (in range; nobody reads them again), so every
      // iteration issues the same loads and the vmcnt waits stay fixed.
      const int kb_next = t + 1 < n ? col_at(t + 1) : kb;
      wait_vmcnt<V_LOADS>();  // this wave's K copies have landed
      block_barrier();        // ... and everybody else's
      f32x16 s[4];
      // Raised wave priority for the QK MFMAs: when both waves of a SIMD
      // reach their MFMA phases together, this one runs ahead and the two
      // drift into alternating MFMA and softmax phases (measured 1.6%).
      __builtin_amdgcn_s_setprio(1);
      qk_tile_ahead<D, QkOp>(k_lds, qf, l32, hl, s, negm);
      __builtin_amdgcn_s_setprio(0);
      if constexpr (SCALED) {  // rows whose q c' exceeds the f16 range carry 2^-r
#pragma unroll
        for (int kc = 0; kc < 4; ++kc)
#pragma unroll
          for (int r = 0; r < 16; ++r) s[kc][r] *= row_scale;
      }
      block_barrier();  // K tile fully consumed
      kcopy.template issue<K_LOADS>(krs, kb_next * TILE_BYTES, k_base, ws);
      if ((Lk & 127) != 0 && kb == (Lk >> 7)) {  // the keys' last block is partial
        int valid = Lk & 127;
        asm volatile("" : "+s"(valid));  // compares stay in this (rare) branch
        mask_tail(s, valid, hl);
      }
      typename PvOp::vec pf[8];
      if constexpr (QK_F16) {
        // The row reference m is set from the first block's maximum. Later
        // blocks skip the maximum: P = exp2(S - m) is formed directly and
        // accepted unless it overflows f16 (some S - m >= 16, which turns the
        // block's row sum inf); only then is the block redone with a moved
        // reference. P <= 2^16 keeps f16's 11-bit precision.
        if (t == t0) softmax_lazy<DCH>(s, true, m, lsum, o, negm, qinv);
        float lblk = 0.f;
        make_p<PvOp, true>(s, 1.f, 0.f, pf, lblk);
        if (t > t0 && __any(!(lblk < INFINITY))) {
          softmax_lazy<DCH>(s, false, m, lsum, o, negm, qinv);
          lblk = 0.f;
          make_p<PvOp, true>(s, 1.f, 0.f, pf, lblk);
        }
        lsum += lblk;
      } else {
        softmax_max<DCH>(s, p.scale_log2, m, lsum, o);
        make_p<PvOp, false>(s, p.scale_log2, m, pf, lsum);
      }
      wait_vmcnt<K_LOADS>();  // V copies landed (the next K may be in flight)
      block_barrier();
      pv_tile_regs<D, PvOp>(v_lds, pf, o, l32, hl);
      block_barrier();  // V tile fully consumed
      vcopy.template issue<V_LOADS>(vrs, kb_next * TILE_BYTES, v_base, ws);
      kb = kb_next;
    }
    wait_vmcnt_0();  // the trailing copies have landed before the workgroup's LDS is released
  }
  if (!SCALED && wk.pieces > 1) {
    store_part<D>(p, wk.slot, o, m, lsum, w, l32, hl);
    return;
  }
  store_out<D>(p, VARLEN ? min(max(p.cu_q[1], 0), p.L) : p.L, p.exps ? p.exps[2 * p.H + h] : 0, out, out_perm,
               lse, o, m, lsum, h, qrow, hl);
}

template <int D, bool QK_F16, bool PV_F16, bool VARLEN, bool SCALED>
__global__ void __launch_bounds__(256, 2) bsa_fwd_split_kernel(BSA_KERNEL_ARGS) {
  __shared__ __attribute__((aligned(16))) uint16_t k_lds[128 * D];
  __shared__ __attribute__((aligned(16))) uint16_t v_lds[D * 128];
  extern __shared__ int32_t cols[];  // kept key blocks of this row (dynamic)
  if constexpr (!SCALED) {
    // Common instance: a query block of a head, or a part of one, XCD-aware.
    Work wk;
    if (!wg_work(p_in, wk)) return;
    if (QK_F16 && common_skips(p_in, wk.h)) return;  // the scaled instance's head
    bsa_split_block<D, QK_F16, PV_F16, VARLEN, false>(q, k, vt, row_ptr, col_idx, out, out_perm, lse, p_in, wk, k_lds,
                                                      v_lds, cols);
  } else {
    // Scaled instance: a small grid (x: workgroups per head, y: head) whose
    // workgroups walk the query blocks of the heads that carry exponents
    // (where only Q left the range, those blocks of them) and exit at once for
    // every other head.
    const int h = blockIdx.y;
    if (!head_scaled(p_in, h)) return;
    for (int qb = blockIdx.x; qb < p_in.Qb; qb += gridDim.x) {
      if (!scaled_block(p_in, h, qb)) continue;
      block_barrier();  // the previous block's LDS reads are done
      bsa_split_block<D, QK_F16, PV_F16, VARLEN, true>(q, k, vt, row_ptr, col_idx, out, out_perm, lse, p_in,
                                                       Work{h, qb, 0, 1, 0}, k_lds, v_lds, cols);
    }
  }
}

// Adds up the parts of the split query blocks: O = sum_p 2^(m_p - M) O_p over
// the same sum of l_p, M the largest m_p, then the scaling, rounding and
// unpermute of store_out. One workgroup per 32 query rows, eight threads a
// row. Reads each part once (64 KB of O per part and block at D = 128). Every
// part enters both sums, so the NaN that a NaN or infinite operand leaves in a
// part's l or O reaches the row as in an uncut block; the weight of a part
// without keys (l = 0, O = 0) is 0.
template <int D, bool VARLEN>
__global__ void __launch_bounds__(256) bsa_combine_kernel(void* __restrict__ out, const int32_t* __restrict__ out_perm,
                                                          float* __restrict__ lse, int qk_f16, BsaParams p) {
  constexpr int DPT = D / 8;  // head dims per thread
  const int r = blockIdx.x >> 2;  // split query block
  const int n_long = split_long(p);
  int h, qb, parts, slot;
  if (r < n_long) {
    if (!long_block(p, r, h, qb)) return;
    parts = p.long_parts;
    slot = r * parts;
  } else {
    const int t = r - n_long;
    if (!ordinary_block(p, t & 7, p.full_rows + (t >> 3), h, qb)) return;
    parts = p.parts;
    slot = n_long * p.long_parts + t * parts;
  }
  if (qk_f16 && head_scaled(p, h)) {  // written whole by the scaled instance
    if (p.q_marks && threadIdx.x == 0) p.q_block_marks[static_cast<int64_t>(h) * p.Qb + qb] = 1;
    return;
  }
  const int Lq = VARLEN ? min(max(p.cu_q[1], 0), p.L) : p.L;
  const int in_block = (blockIdx.x & 3) * 32 + (threadIdx.x >> 3);
  const int qrow = qb * 128 + in_block;
  if (qrow >= Lq) return;
  const int d0 = (threadIdx.x & 7) * DPT;
  const int64_t row0 = static_cast<int64_t>(slot) * 128 + in_block;
  float M = -INFINITY;
  for (int i = 0; i < parts; ++i) {
    const float2 ml = *reinterpret_cast<const float2*>(p.part_ml + (row0 + i * 128) * 2);
    if (ml.y != 0.f) M = fmaxf(M, ml.x);
  }
  float acc[DPT] = {}, l = 0.f;
  for (int i = 0; i < parts; ++i) {
    const float2 ml = *reinterpret_cast<const float2*>(p.part_ml + (row0 + i * 128) * 2);
    const float f = ml.y != 0.f ? exp2_fast(ml.x - M) : 0.f;  // 0: a part without keys
    l += ml.y * f;
    const float4* src = reinterpret_cast<const float4*>(p.part_o + (row0 + i * 128) * D + d0);
#pragma unroll
    for (int j = 0; j < DPT / 4; ++j) {
      const float4 v = src[j];
      acc[4 * j + 0] += v.x * f;
      acc[4 * j + 1] += v.y * f;
      acc[4 * j + 2] += v.z * f;
      acc[4 * j + 3] += v.w * f;
    }
  }
  const float inv = l > 0.f ? ldexpf(1.0f / l, p.exps ? p.exps[2 * p.H + h] : 0) : 0.f;
  const int orow = out_perm ? out_perm[qrow] : qrow;
  const int64_t obase = h * p.o_sh + orow * p.o_sl + d0;
#pragma unroll
  for (int j = 0; j < DPT; j += 4) {
    const float v0 = acc[j] * inv, v1 = acc[j + 1] * inv, v2 = acc[j + 2] * inv, v3 = acc[j + 3] * inv;
    if (p.out_kind == DFS_DTYPE_F32)
      *reinterpret_cast<float4*>(static_cast<float*>(out) + obase + j) = make_float4(v0, v1, v2, v3);
    else if (p.out_kind == DFS_DTYPE_BF16)
      *reinterpret_cast<uint2*>(static_cast<uint16_t*>(out) + obase + j) =
          make_uint2(f32_to_bf16_bits(v0) | (f32_to_bf16_bits(v1) << 16),
                     f32_to_bf16_bits(v2) | (f32_to_bf16_bits(v3) << 16));
    else
      *reinterpret_cast<uint2*>(static_cast<uint16_t*>(out) + obase + j) =
          make_uint2(f32_to_f16_bits(v0) | (f32_to_f16_bits(v1) << 16),
                     f32_to_f16_bits(v2) | (f32_to_f16_bits(v3) << 16));
  }
  if (lse && d0 == 0)
    lse[static_cast<int64_t>(h) * p.Lo + qrow] = l > 0.f ? (M + log2f(l)) * 0.69314718055994531f : -INFINITY;
}

struct BsaArgs {
  const uint16_t *q, *k, *vt;
  const int32_t *row_ptr, *col_idx;
  void* out;
  const int32_t* out_perm;
  float* lse;
};

struct SegParams {
  int H, L, R, csr_qb, Lo;
  int out_kind;
  float scale_log2;
  const int32_t* cu_q;  // [n_seq + 1] (device)
  const int32_t* cu_k;
  int n_seq;
  const int32_t* exps;  // optional [3][H]
  const uint16_t* q_src;  // optional Q source (as in BsaParams)
  const int32_t* q_rows;
  int64_t q_sh, q_sl;  // element strides of q_src
  int q_src_f16;
  int64_t o_sh, o_sl;  // element strides of out
};

__device__ __forceinline__ float operand_at(const uint16_t* base, int64_t i, bool f16) {
  return f16 ? f16_bits_to_f32(base[i]) : bf16_bits_to_f32(base[i]);
}

// Maximum and sum over the wave through register moves, the same bits in
// every lane (each step joins a lane with its mirror).
template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, dpp_mov<0xB1>(v));   // quad_perm [1, 0, 3, 2]
  v = fmaxf(v, dpp_mov<0x4E>(v));   // quad_perm [2, 3, 0, 1]
  v = fmaxf(v, dpp_mov<0x141>(v));  // row_half_mirror
  v = fmaxf(v, dpp_mov<0x140>(v));  // row_mirror
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return xhalf_max(fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1])));
}
__device__ __forceinline__ float wave_sum(float v) {
  v += dpp_mov<0xB1>(v);
  v += dpp_mov<0x4E>(v);
  v += dpp_mov<0x141>(v);
  v += dpp_mov<0x140>(v);
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return xhalf_sum(__uint_as_float(a[0]) + __uint_as_float(a[1]));
}

// The rows of a call after segment 0 of cu_seqlens, in fp32. A workgroup takes
// four consecutive rows of one query block, a wave each, and walks their kept
// key blocks 64 keys at a time: the window's K rows and V^T slots go through
// LDS (chunk-swizzled, read by the four waves), one key per lane for the
// scores, an exact running maximum, then P V with each lane owning head dims
// lane and lane + 64. For n_seq == 2 the rows [cq1, cq2) attend keys
// [ck1, ck2) under the same block mask indexed from each segment's own start
// (query block (r - cq1) / 128 selects the CSR row, key block j covers keys
// ck1 + 128 j ..), as the reference's varlen kernel treats the second sequence
// of its batch (attention_hyvideo.py:1054-1082, the mask repeated per sequence
// at :359). Rows outside every query segment are zero (lse -inf). Windows are
// aligned to 64 keys so that a window's V^T slots are one contiguous run of a
// physical 128-key block; keys of a window outside the column's range are
// masked. Sized for short padding segments (a few hundred tokens), where a
// row's chain counts: 15 us for 32 padding rows of 24 heads and 33 for 138.
// Read from global memory, one key or head dim per lane, each load touched 64
// cache lines: 78 us for the 138 with a row per wave, 100 with four (61 for
// the 32).
template <int D, bool QK_F16, bool PV_F16>
__global__ void __launch_bounds__(256) bsa_segment_kernel(const uint16_t* __restrict__ q,
                                                          const uint16_t* __restrict__ k,
                                                          const uint16_t* __restrict__ vt,
                                                          const int32_t* __restrict__ row_ptr,
                                                          const int32_t* __restrict__ col_idx,
                                                          void* __restrict__ out, const int32_t* __restrict__ out_perm,
                                                          float* __restrict__ lse, SegParams p) {
  constexpr int DPL = D / 64;           // head dims per lane in P V
  constexpr int CPR = D / 8;            // 16-byte chunks of a K row
  constexpr int LOADS = 64 * CPR / 256;  // chunks of a K (or V^T) window per thread
  __shared__ u32x4_t kw[64 * CPR];  // chunk c of key r at r * CPR + (c ^ (r % CPR))
  __shared__ u32x4_t vw[D * 8];     // chunk c of head dim d at d * 8 + (c ^ (d / 2 % 8))
  __shared__ __attribute__((aligned(16))) float qs[4][D];   // the row's q (times the scale), per wave
  __shared__ __attribute__((aligned(16))) float ps[4][64];  // the window's P in V^T slot order, per wave
  const int h = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int cq1 = min(max(p.cu_q[1], 0), p.L);
  const int cq2 = p.n_seq == 2 ? min(max(p.cu_q[2], cq1), p.L) : cq1;
  const int ck1 = p.n_seq == 2 ? min(max(p.cu_k[1], 0), p.L) : 0;
  const int ck2 = p.n_seq == 2 ? min(max(p.cu_k[2], ck1), p.L) : 0;
  const int seg_kb = (ck2 - ck1 + 127) >> 7;
  float sq = p.scale_log2, sv = 1.f;
  if (p.exps) {
    sq = ldexpf(sq, (p.q_src ? 0 : p.exps[h]) + p.exps[p.H + h]);  // a Q source is read unscaled
    sv = ldexpf(1.f, p.exps[2 * p.H + h]);
  }
  auto wave_sync = [] {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_wave_barrier();
  };
  const int64_t hq = static_cast<int64_t>(h) * p.R * D;
  const u32x4_t* krows = reinterpret_cast<const u32x4_t*>(k + hq);
  const u32x4_t* vblocks = reinterpret_cast<const u32x4_t*>(vt + hq);
  // Element j of execution row r's query (r < L).
  auto q_at = [&](int r, int j) -> float {
    if (p.q_src)
      return operand_at(p.q_src, h * p.q_sh + p.q_rows[r] * p.q_sl + j, p.q_src_f16 != 0);
    return operand_at(q, hq + static_cast<int64_t>(r) * D + j, QK_F16);
  };

  // Groups of four rows from cq1 on: 4 divides 128, so a group's rows share
  // query block (r0 - cq1) / 128, its columns and its windows.
  for (int r0 = cq1 + 4 * static_cast<int>(blockIdx.x); r0 < p.L; r0 += 4 * static_cast<int>(gridDim.x)) {
    const int r = r0 + w;
    const bool live = r < cq2;  // a row of the second sequence
    float o[DPL] = {}, m = -INFINITY, l = 0.f;
    if (r0 < cq2 && seg_kb > 0) {
#pragma unroll
      for (int j = 0; j < DPL; ++j) qs[w][j * 64 + lane] = live ? q_at(r, j * 64 + lane) * sq : 0.f;
      const int64_t crow = static_cast<int64_t>(h) * p.csr_qb + ((r0 - cq1) >> 7);
      const int beg = row_ptr[crow], end = row_ptr[crow + 1];
      for (int idx = beg; idx < end; ++idx) {  // columns ascend: stop at the segment's last block
        const int cb = __builtin_amdgcn_readfirstlane(col_idx[idx]);
        if (cb >= seg_kb) break;
        if (cb < 0) continue;
        const int k0 = ck1 + cb * 128, k1 = min(k0 + 128, ck2);
        for (int w0 = k0 & ~63; w0 < k1; w0 += 64) {  // w0 + 64 <= R: whole windows lie in the operands
          u32x4_t kr[LOADS], vr[LOADS];  // plain vectors: uint4 copies across the barrier went through scratch
#pragma unroll
          for (int i = 0; i < LOADS; ++i) {
            const int e = i * 256 + tid;
            kr[i] = krows[static_cast<int64_t>(w0) * CPR + e];
            // V^T block w0 / 128: 16 chunks per head dim, this window's 8
            vr[i] = vblocks[(static_cast<int64_t>(w0 >> 7) * D + (e >> 3)) * 16 + ((w0 >> 3) & 8) + (e & 7)];
          }
          __syncthreads();  // the previous window has been read
#pragma unroll
          for (int i = 0; i < LOADS; ++i) {
            const int e = i * 256 + tid, kr_row = e / CPR, d = e >> 3;
            kw[kr_row * CPR + ((e % CPR) ^ (kr_row % CPR))] = kr[i];
            vw[d * 8 + ((e & 7) ^ ((d >> 1) & 7))] = vr[i];
          }
          __syncthreads();
          const int key = w0 + lane;
          const bool valid = key >= k0 && key < k1;
          float s4[4] = {};  // four chains of the dot product
#pragma unroll 2
          for (int c = 0; c < CPR; ++c) {
            const uint4 kv = __builtin_bit_cast(uint4, kw[lane * CPR + (c ^ (lane % CPR))]);
            const float4 qa = *reinterpret_cast<const float4*>(&qs[w][c * 8]);
            const float4 qb = *reinterpret_cast<const float4*>(&qs[w][c * 8 + 4]);
            const float qe[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
#pragma unroll
            for (int e = 0; e < 8; ++e)
              s4[e & 3] += qe[e] * (QK_F16 ? f16_bits_to_f32(u16_at(kv, e)) : bf16_bits_to_f32(u16_at(kv, e)));
          }
          const float si = valid ? (s4[0] + s4[1]) + (s4[2] + s4[3]) : -INFINITY;
          const float mnew = fmaxf(m, wave_max(si));  // finite: the window holds key max(w0, k0) < k1
          const float alpha = exp2_fast(m - mnew);
          const float pk = valid ? exp2_fast(si - mnew) : 0.f;
          l = l * alpha + wave_sum(pk);
#pragma unroll
          for (int j = 0; j < DPL; ++j) o[j] *= alpha;
          m = mnew;
          // slot of window key `lane` in its 16-key group: swap23 (an involution)
          ps[w][(lane & ~15) | (lane & 3) | ((lane & 4) << 1) | ((lane & 8) >> 1)] = pk;
          wave_sync();
#pragma unroll 2
          for (int c = 0; c < 8; ++c) {
            const float4 pa = *reinterpret_cast<const float4*>(&ps[w][c * 8]);
            const float4 pb = *reinterpret_cast<const float4*>(&ps[w][c * 8 + 4]);
            const float pe[8] = {pa.x, pa.y, pa.z, pa.w, pb.x, pb.y, pb.z, pb.w};
#pragma unroll
            for (int j = 0; j < DPL; ++j) {
              const int d = j * 64 + lane;
              const uint4 vc = __builtin_bit_cast(uint4, vw[d * 8 + (c ^ ((d >> 1) & 7))]);
#pragma unroll
              for (int e = 0; e < 8; ++e)
                o[j] += pe[e] * (PV_F16 ? f16_bits_to_f32(u16_at(vc, e)) : bf16_bits_to_f32(u16_at(vc, e)));
            }
          }
          wave_sync();  // ps is read before the next window overwrites it
        }
      }
      wave_sync();  // qs is read before the next row overwrites it
    }
    if (r >= p.L) continue;
    if (!live) l = 0.f;  // scored with q = 0: the row belongs to no sequence (zero, lse -inf)
    const float inv = l > 0.f ? sv / l : 0.f;
    const int orow = out_perm ? out_perm[r] : r;
    const int64_t ob = h * p.o_sh + orow * p.o_sl;
#pragma unroll
    for (int j = 0; j < DPL; ++j) {
      const float v = o[j] * inv;
      const int64_t at = ob + j * 64 + lane;
      if (p.out_kind == DFS_DTYPE_F32)
        static_cast<float*>(out)[at] = v;
      else if (p.out_kind == DFS_DTYPE_BF16)
        static_cast<uint16_t*>(out)[at] = static_cast<uint16_t>(f32_to_bf16_bits(v));
      else
        static_cast<uint16_t*>(out)[at] = static_cast<uint16_t>(f32_to_f16_bits(v));
    }
    if (lse && lane == 0)
      lse[static_cast<int64_t>(h) * p.Lo + r] = l > 0.f ? (m + log2f(l)) * 0.69314718055994531f : -INFINITY;
  }
}

template <int D, bool QK_F16, bool PV_F16, bool VARLEN>
void launch_split_as(const BsaArgs& a, const BsaParams& p, hipStream_t s) {
  const size_t smem = static_cast<size_t>(p.Kb) * sizeof(int32_t) +
                      static_cast<size_t>(2 * ((2 * p.Kb + 31) / 32) + 2) * sizeof(uint32_t);
  if (!p.scale_all) {
    const int per_xcd = long_per_xcd(p) * p.long_parts + p.full_rows + (blocks_per_xcd(p) - p.full_rows) * p.parts;
    bsa_fwd_split_kernel<D, QK_F16, PV_F16, VARLEN, false><<<dim3(static_cast<unsigned>(8 * per_xcd)), 256, smem, s>>>(
        a.q, a.k, a.vt, a.row_ptr, a.col_idx, a.out, a.out_perm, a.lse, p);
    const int split = split_long(p) + split_tail(p);
    if (split > 0)
      bsa_combine_kernel<D, VARLEN><<<dim3(static_cast<unsigned>(4 * split)), 256, 0, s>>>(a.out, a.out_perm, a.lse,
                                                                                          QK_F16 ? 1 : 0, p);
  }
  if constexpr (QK_F16) {
    // Heads with exponents (only when some bf16 input exceeds the f16 range):
    // a workgroup per CU over all heads, but eight a head at least. Or every
    // head (large scales).
    if (p.exps || p.scale_all) {
      const unsigned per_head = static_cast<unsigned>(p.scale_all ? p.Qb : min(p.Qb, max(8, 256 / p.H)));
      bsa_fwd_split_kernel<D, QK_F16, PV_F16, VARLEN, true>
          <<<dim3(per_head, static_cast<unsigned>(p.H)), 256, smem, s>>>(a.q, a.k, a.vt, a.row_ptr, a.col_idx, a.out,
                                                                     a.out_perm, a.lse, p);
    }
  }
}

template <int D, bool QK_F16, bool PV_F16>
void launch_split(const BsaArgs& a, const BsaParams& p, hipStream_t s) {
  if (p.cu_q) return launch_split_as<D, QK_F16, PV_F16, true>(a, p, s);
  launch_split_as<D, QK_F16, PV_F16, false>(a, p, s);
}

template <int D>
void launch_bsa(const BsaArgs& a, const BsaParams& p, bool qk_f16, bool pv_f16, hipStream_t s) {
  if (qk_f16)
    launch_split<D, true, true>(a, p, s);
  else if (pv_f16)
    launch_split<D, false, true>(a, p, s);
  else
    launch_split<D, false, false>(a, p, s);
}

}  // namespace
}  // namespace dfs

namespace dfs {

int bsa_fwd_impl(const char* name, const void* q_perm, const void* k_perm, const void* v_t,
                           const int32_t* row_ptr, const int32_t* col_idx, int64_t heads,
                           int64_t seq_len, int64_t head_dim, int dtype, int pv_dtype, float scale,
                           void* out, int out_dtype, const int32_t* out_perm, float* lse,
                           const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, int64_t n_seq,
                           const int32_t* exps, const void* q_src, const int32_t* q_rows, int q_src_dtype,
                           int64_t out_head_stride, int64_t out_row_stride, int64_t long_row, int64_t long_parts,
                           int64_t full_rows, int64_t parts, int64_t chunks, void* workspace,
                           int64_t workspace_bytes, int32_t* q_marks, int32_t* q_block_marks,
                           const int64_t* q_strides, dfs_stream_t stream) {
  DFS_REQUIRE((q_perm || q_src) && k_perm && v_t && row_ptr && col_idx && out, "%s: NULL operand", name);
  DFS_REQUIRE(!q_src || q_rows, "%s: q_src needs q_rows", name);
  DFS_REQUIRE(!q_src || q_src_dtype == DFS_DTYPE_BF16 || q_src_dtype == DFS_DTYPE_F16,
              "%s: q_src_dtype=%d (supported: bf16, f16)", name, q_src_dtype);
  DFS_REQUIRE(!q_src || dtype == DFS_DTYPE_F16 || q_src_dtype == DFS_DTYPE_BF16,
              "%s: bf16 Q/K operands need a bf16 q_src", name);
  DFS_REQUIRE(head_dim == 64 || head_dim == 128, "%s: head_dim=%lld (supported: 64, 128)", name,
              (long long)head_dim);
  DFS_REQUIRE(dtype == DFS_DTYPE_BF16 || dtype == DFS_DTYPE_F16, "%s: dtype=%d (supported: bf16, f16)",
              name, dtype);
  DFS_REQUIRE(pv_dtype == DFS_DTYPE_BF16 || pv_dtype == DFS_DTYPE_F16,
              "%s: pv_dtype=%d (supported: bf16, f16)", name, pv_dtype);
  DFS_REQUIRE(!(dtype == DFS_DTYPE_F16 && pv_dtype == DFS_DTYPE_BF16),
              "%s: f16 inputs need an f16 PV operand", name);
  DFS_REQUIRE(out_dtype >= 0 && out_dtype <= 2, "%s: out_dtype=%d", name, out_dtype);
  DFS_REQUIRE(heads > 0 && seq_len > 0, "%s: empty problem", name);
  const int64_t qb = (seq_len + kBlock - 1) / kBlock;
  DFS_REQUIRE(heads * qb < (int64_t(1) << 31) && qb * kBlock * head_dim < (int64_t(1) << 31),
              "%s: problem too large for 32-bit indexing", name);
  // LDS: 64 KB of tiles (split schedule) plus the row's column list.
  DFS_REQUIRE(qb <= 8192, "%s: %lld key blocks exceed the LDS column list", name, (long long)qb);
  DFS_REQUIRE(scale > 0.f && isfinite(scale), "%s: scale must be positive and finite", name);
  DFS_REQUIRE(n_seq == 1 || n_seq == 2, "%s: n_seq=%lld (supported: 1 or 2 sequences)", name, (long long)n_seq);
  DFS_REQUIRE((cu_seqlens_q == nullptr) == (cu_seqlens_k == nullptr),
              "%s: pass both cu_seqlens_q and cu_seqlens_k or neither", name);
  DFS_REQUIRE(n_seq == 1 || cu_seqlens_q, "%s: two sequences need cu_seqlens", name);
  BsaArgs a{static_cast<const uint16_t*>(q_perm), static_cast<const uint16_t*>(k_perm),
            static_cast<const uint16_t*>(v_t), row_ptr, col_idx, out, out_perm, lse};
  BsaParams p{};
  p.H = static_cast<int>(heads);
  p.L = p.Lk = static_cast<int>(seq_len);
  p.R = static_cast<int>(qb * kBlock);
  p.Qb = p.Kb = static_cast<int>(qb);
  p.Lo = static_cast<int>(seq_len);
  p.csr_qb = static_cast<int>(qb);
  p.scale_log2 = scale * 1.4426950408889634f;
  // An f16 operand is below 65504 < 2^16, so q * c stays below 2^15 unless
  // c >= 0.5 (a softmax scale >= 0.35); then every head takes the scaled
  // instance, whose rows carry their own powers of two.
  p.scale_all = (dtype == DFS_DTYPE_F16 && p.scale_log2 >= 0.5f) ? 1 : 0;
  p.out_kind = out_dtype;
  p.cu_q = cu_seqlens_q;
  p.cu_k = cu_seqlens_k;
  p.exps = exps;
  DFS_REQUIRE((q_marks == nullptr) == (q_block_marks == nullptr) &&
                  (!q_marks || (q_marks == exps && q_src && q_src_dtype == DFS_DTYPE_BF16)),
              "%s: Q's range is marked by head and block, for a bf16 Q source", name);
  p.q_marks = q_marks;
  p.q_block_marks = q_block_marks;
  p.q_sh = q_strides ? q_strides[0] : seq_len * head_dim;
  p.q_sl = q_strides ? q_strides[1] : head_dim;
  DFS_REQUIRE(p.q_sh >= 0 && p.q_sl >= 0 && p.q_sh % 8 == 0 && p.q_sl % 8 == 0,
              "%s: q strides %lld, %lld must be non-negative multiples of 8 elements", name, (long long)p.q_sh,
              (long long)p.q_sl);
  p.q_src = static_cast<const uint16_t*>(q_src);
  p.q_rows = q_rows;
  p.q_src_f16 = q_src_dtype == DFS_DTYPE_F16 ? 1 : 0;
  DFS_REQUIRE(out_head_stride > 0 && out_row_stride >= head_dim && out_head_stride % 4 == 0 && out_row_stride % 4 == 0,
              "%s: out strides %lld, %lld must be multiples of 4 elements that hold a row", name,
              (long long)out_head_stride, (long long)out_row_stride);
  p.o_sh = out_head_stride;
  p.o_sl = out_row_stride;
  DFS_REQUIRE(long_row >= 0 && long_row <= qb, "%s: long_row=%lld outside [0, %lld]", name, (long long)long_row,
              (long long)qb);
  p.H = static_cast<int>(heads);
  p.long_row = static_cast<int>(long_row);
  DFS_REQUIRE(chunks == 1 || chunks == 2 || chunks == 4 || chunks == 8, "%s: chunks=%lld (supported: 1, 2, 4, 8)",
              name, (long long)chunks);
  p.chunks = static_cast<int>(chunks);
  const int64_t per_xcd = blocks_per_xcd(p);
  DFS_REQUIRE(parts >= 1 && parts <= 64 && long_parts >= 1 && long_parts <= 64, "%s: parts=%lld, %lld outside [1, 64]",
              name, (long long)parts, (long long)long_parts);
  DFS_REQUIRE(full_rows >= 0 && full_rows <= per_xcd, "%s: full_rows=%lld outside [0, %lld]", name,
              (long long)full_rows, (long long)per_xcd);
  p.long_row = static_cast<int>(long_row);
  p.long_parts = static_cast<int>(long_parts);
  p.full_rows = static_cast<int>(parts > 1 ? full_rows : per_xcd);
  p.parts = static_cast<int>(parts);
  if (p.scale_all) {  // every head runs unsplit in the scaled instance
    p.long_parts = p.parts = 1;
    p.full_rows = static_cast<int>(per_xcd);
  }
  const int64_t slots = static_cast<int64_t>(split_long(p)) * p.long_parts + static_cast<int64_t>(split_tail(p)) * p.parts;
  DFS_REQUIRE(slots < (int64_t(1) << 24), "%s: too many parts", name);
  const int64_t need = slots * 128 * (head_dim + 2) * static_cast<int64_t>(sizeof(float));
  DFS_REQUIRE(slots == 0 || (workspace && workspace_bytes >= need), "%s: workspace of %lld bytes, %lld needed", name,
              (long long)(workspace ? workspace_bytes : 0), (long long)need);
  DFS_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 15u) == 0, "%s: workspace must be 16-byte aligned", name);
  p.part_o = static_cast<float*>(workspace);
  p.part_ml = p.part_o + slots * 128 * head_dim;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const bool qk_f16 = dtype == DFS_DTYPE_F16, pv_f16 = pv_dtype == DFS_DTYPE_F16;
  if (head_dim == 128)
    launch_bsa<128>(a, p, qk_f16, pv_f16, s);
  else
    launch_bsa<64>(a, p, qk_f16, pv_f16, s);
  if (cu_seqlens_q) {
    SegParams sp{};
    sp.H = p.H;
    sp.L = p.L;
    sp.R = p.R;
    sp.csr_qb = p.csr_qb;
    sp.Lo = p.Lo;
    sp.out_kind = out_dtype;
    sp.scale_log2 = p.scale_log2;
    sp.cu_q = cu_seqlens_q;
    sp.cu_k = cu_seqlens_k;
    sp.n_seq = static_cast<int>(n_seq);
    sp.exps = exps;
    sp.q_src = p.q_src;
    sp.q_rows = q_rows;
    sp.q_sh = p.q_sh;
    sp.q_sl = p.q_sl;
    sp.q_src_f16 = p.q_src_f16;
    sp.o_sh = p.o_sh;
    sp.o_sl = p.o_sl;
    // Four rows per workgroup for a few hundred rows per head; a workgroup
    // strides over the rows after segment 0.
    const dim3 grid(64, static_cast<unsigned>(heads));
    auto seg = [&](auto kernel) {
      kernel<<<grid, 256, 0, s>>>(a.q, a.k, a.vt, row_ptr, col_idx, out, out_perm, lse, sp);
    };
    if (head_dim == 128)
      qk_f16 ? seg(bsa_segment_kernel<128, true, true>)
             : pv_f16 ? seg(bsa_segment_kernel<128, false, true>) : seg(bsa_segment_kernel<128, false, false>);
    else
      qk_f16 ? seg(bsa_segment_kernel<64, true, true>)
             : pv_f16 ? seg(bsa_segment_kernel<64, false, true>) : seg(bsa_segment_kernel<64, false, false>);
  }
  return check_launch(name);
}

}  // namespace dfs

extern "C" int64_t dfs_bsa_fwd_workspace_size(int64_t heads, int64_t seq_len, int64_t head_dim, int64_t long_row,
                                              int64_t long_parts, int64_t full_rows, int64_t parts,
                                              int64_t chunks) {
  using namespace dfs;
  const int64_t qb = (seq_len + kBlock - 1) / kBlock;
  if (heads <= 0 || seq_len <= 0 || head_dim <= 0 || long_row < 0 || long_row > qb || long_parts < 1 || parts < 1 ||
      full_rows < 0 || heads * qb >= (int64_t(1) << 31) ||
      (chunks != 1 && chunks != 2 && chunks != 4 && chunks != 8))
    return -1;
  BsaParams p{};
  p.H = static_cast<int>(heads);
  p.Qb = static_cast<int>(qb);
  p.long_row = static_cast<int>(long_row);
  p.long_parts = static_cast<int>(long_parts);
  p.parts = static_cast<int>(parts);
  p.chunks = static_cast<int>(chunks);
  const int64_t per_xcd = blocks_per_xcd(p);
  p.full_rows = static_cast<int>(full_rows < per_xcd ? full_rows : per_xcd);
  const int64_t slots = split_long(p) * long_parts + split_tail(p) * parts;
  return slots * 128 * (head_dim + 2) * static_cast<int64_t>(sizeof(float));
}

extern "C" int dfs_bsa_fwd(const void* q_perm, const void* k_perm, const void* v_t,
                           const int32_t* row_ptr, const int32_t* col_idx, int64_t heads,
                           int64_t seq_len, int64_t head_dim, int dtype, int pv_dtype, float scale,
                           void* out, int out_dtype, const int32_t* out_perm, float* lse,
                           const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, int64_t n_seq,
                           const int32_t* exps, const void* q_src, const int32_t* q_rows, int q_src_dtype,
                           dfs_stream_t stream) {
  return dfs::bsa_fwd_impl("dfs_bsa_fwd", q_perm, k_perm, v_t, row_ptr, col_idx, heads, seq_len, head_dim, dtype,
                           pv_dtype, scale, out, out_dtype, out_perm, lse, cu_seqlens_q, cu_seqlens_k, n_seq, exps,
                           q_src, q_rows, q_src_dtype, seq_len * head_dim, head_dim,
                           (seq_len + dfs::kBlock - 1) / dfs::kBlock, 1, 0, 1, 8, nullptr, 0, nullptr, nullptr, nullptr, stream);
}

extern "C" int dfs_bsa_fwd_parts(const void* q_perm, const void* k_perm, const void* v_t, const int32_t* row_ptr,
                                 const int32_t* col_idx, int64_t heads, int64_t seq_len, int64_t head_dim, int dtype,
                                 int pv_dtype, float scale, void* out, int out_dtype, const int32_t* out_perm,
                                 float* lse, const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, int64_t n_seq,
                                 const int32_t* exps, const void* q_src, const int32_t* q_rows, int q_src_dtype,
                                 int64_t out_head_stride, int64_t out_row_stride, int64_t long_row,
                                 int64_t long_parts, int64_t full_rows, int64_t parts, int64_t chunks,
                                 void* workspace, int64_t workspace_bytes, dfs_stream_t stream) {
  return dfs::bsa_fwd_impl("dfs_bsa_fwd_parts", q_perm, k_perm, v_t, row_ptr, col_idx, heads, seq_len, head_dim, dtype,
                           pv_dtype, scale, out, out_dtype, out_perm, lse, cu_seqlens_q, cu_seqlens_k, n_seq, exps,
                           q_src, q_rows, q_src_dtype, out_head_stride, out_row_stride, long_row, long_parts,
                           full_rows, parts, chunks, workspace, workspace_bytes, nullptr, nullptr, nullptr, stream);
}
