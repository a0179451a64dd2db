// One DFS attention call behind one entry point: the preparation, the scoring
// with top-k and the attention enqueued back to back, every intermediate in
// one caller workspace. The launches are those of the single entry points; a
// call of a thousand tokens took 85 us on the host as four of them with a
// dozen allocations in Python, against 35 us of kernels.
#include <algorithm>

#include "common.h"

namespace dfs {

// permute.hip
int prepare_qkv_impl(const void* q, const void* k, const void* v, const int32_t* perm, int64_t heads, int64_t seq_len,
                     int64_t head_dim, int dtype, int64_t video_len, int64_t q_tile_size, int64_t k_tile_size,
                     int operand_dtype, void* q_perm, void* k_perm, void* v_t, uint16_t* q_pool_hi,
                     uint16_t* q_pool_lo, uint16_t* k_pool_hi, uint16_t* k_pool_lo, int32_t* overflow,
                     int32_t* wave_flags, bool skip_q, const int64_t* strides, dfs_stream_t stream);
int64_t prepare_flag_words(int64_t heads, int64_t seq_len, int64_t head_dim, int64_t q_tile, int64_t k_tile);
int prepare_fixup_impl(const void* q, const void* k, const void* v, const int32_t* perm, int64_t heads,
                       int64_t seq_len, int64_t head_dim, void* q_perm, void* k_perm, void* v_t, int32_t* overflow,
                       int32_t* wave_flags, int64_t q_tile_size, int64_t k_tile_size, bool skip_q, int32_t* exps,
                       int32_t* q_block_marks, const int64_t* strides, dfs_stream_t stream);

// bsa_fwd.hip
int bsa_fwd_impl(const char* name, const void* q_perm, const void* k_perm, const void* v_t, const int32_t* row_ptr,
                 const int32_t* col_idx, int64_t heads, int64_t seq_len, int64_t head_dim, int dtype, int pv_dtype,
                 float scale, void* out, int out_dtype, const int32_t* out_perm, float* lse,
                 const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k, int64_t n_seq, const int32_t* exps,
                 const void* q_src, const int32_t* q_rows, int q_src_dtype, int64_t out_head_stride,
                 int64_t out_row_stride, int64_t long_row, int64_t long_parts, int64_t full_rows, int64_t parts,
                 int64_t chunks, void* workspace, int64_t workspace_bytes, int32_t* q_marks, int32_t* q_block_marks,
                 const int64_t* q_strides, dfs_stream_t stream);

namespace {

// Byte offsets of a call's intermediates in its workspace.
struct Regions {
  int64_t k_perm, v_t, exps, flags, marks, q_hi, q_lo, k_hi, k_lo, shared, bytes;
  int64_t score_bytes;  // one-pass scoring workspace (0: the score matrix takes its place)
  int64_t part_bytes;   // partial results of the attention
};

Regions regions(const dfs_call_args& a) {
  Regions r{};
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    const int64_t here = at;
    at += (bytes + 255) / 256 * 256;
    return here;
  };
  const int64_t rows = (a.seq_len + kBlock - 1) / kBlock * kBlock;
  r.k_perm = take(a.heads * rows * a.head_dim * 2);
  r.v_t = take(a.heads * rows * a.head_dim * 2);
  if (a.dtype == DFS_DTYPE_BF16 && a.operand_dtype == DFS_DTYPE_F16) {
    r.exps = take(3 * a.heads * 4);
    r.flags = take(prepare_flag_words(a.heads, a.seq_len, a.head_dim, a.q_tile, a.k_tile) * 4);
    if (!a.select) r.marks = take(a.heads * (rows / kBlock) * 4);  // the attention's marks of Q's blocks
  }
  int64_t shared = 0;
  if (a.select) {
    const int64_t q_tiles = (a.video_len + kBlock - 1) / kBlock * kBlock / a.q_tile, k_tiles = rows / a.k_tile;
    r.q_hi = take(a.heads * q_tiles * a.head_dim * 2);
    r.q_lo = take(a.heads * q_tiles * a.head_dim * 2);
    r.k_hi = take(a.heads * k_tiles * a.head_dim * 2);
    r.k_lo = take(a.heads * k_tiles * a.head_dim * 2);
    // Rows wider than the one-pass form's 16 * head_dim columns, and tile
    // pairs without one, keep their block sums in a score matrix.
    if (a.k_blocks <= 16 * a.head_dim)
      r.score_bytes = std::max<int64_t>(
          0, dfs_block_score_topk_split_size(a.heads, a.q_tile, a.k_tile, a.q_blocks, a.k_blocks));
    shared = r.score_bytes > 0 ? r.score_bytes : a.heads * a.scored_rows * a.k_blocks * 4;
  }
  r.part_bytes = std::max<int64_t>(0, dfs_bsa_fwd_workspace_size(a.heads, a.seq_len, a.head_dim, a.long_row,
                                                                 a.long_parts, a.full_rows, a.parts, a.chunks));
  // The scoring is over when the attention writes its parts: one region.
  r.shared = take(std::max(shared, r.part_bytes));
  r.bytes = at;
  return r;
}

int check_args(const char* name, const dfs_call_args* a) {
  DFS_REQUIRE(a != nullptr, "%s: NULL arguments", name);
  DFS_REQUIRE(a->heads > 0 && a->seq_len > 0 && (a->head_dim == 64 || a->head_dim == 128),
              "%s: heads=%lld seq_len=%lld head_dim=%lld", name, (long long)a->heads, (long long)a->seq_len,
              (long long)a->head_dim);
  DFS_REQUIRE(a->video_len > 0 && a->video_len <= a->seq_len, "%s: need 0 < video_len=%lld <= seq_len", name,
              (long long)a->video_len);
  DFS_REQUIRE(a->q_tile > 0 && kBlock % a->q_tile == 0 && a->k_tile > 0 && kBlock % a->k_tile == 0,
              "%s: q_tile=%lld, k_tile=%lld (each must divide 128)", name, (long long)a->q_tile,
              (long long)a->k_tile);
  const int64_t blocks = (a->seq_len + kBlock - 1) / kBlock;
  DFS_REQUIRE(!a->select || (a->q_blocks == blocks && a->k_blocks == blocks && a->scored_rows >= 0 &&
                             a->scored_rows <= blocks),
              "%s: the policy's blocks (%lld x %lld, %lld scored) do not match %lld", name, (long long)a->q_blocks,
              (long long)a->k_blocks, (long long)a->scored_rows, (long long)blocks);
  DFS_REQUIRE(a->long_row >= 0 && a->long_row <= blocks && a->long_parts >= 1 && a->parts >= 1 && a->full_rows >= 0,
              "%s: long_row=%lld long_parts=%lld full_rows=%lld parts=%lld", name, (long long)a->long_row,
              (long long)a->long_parts, (long long)a->full_rows, (long long)a->parts);
  return 0;
}

}  // namespace
}  // namespace dfs

extern "C" int64_t dfs_call_workspace_size(const dfs_call_args* a) {
  if (dfs::check_args("dfs_call_workspace_size", a)) return -1;
  return dfs::regions(*a).bytes;
}

extern "C" int dfs_call(const dfs_call_args* a, int phases, dfs_stream_t stream) {
  using namespace dfs;
  const char* name = "dfs_call";
  if (int rc = check_args(name, a)) return rc;
  DFS_REQUIRE((phases & ~7) == 0, "%s: phases=%d", name, phases);
  const Regions r = regions(*a);
  DFS_REQUIRE(a->workspace && a->workspace_bytes >= r.bytes && (reinterpret_cast<uintptr_t>(a->workspace) & 15u) == 0,
              "%s: workspace of %lld bytes, %lld needed (16-byte aligned)", name,
              (long long)(a->workspace ? a->workspace_bytes : 0), (long long)r.bytes);
  char* const ws = static_cast<char*>(a->workspace);
  const bool rounds = a->dtype == DFS_DTYPE_BF16 && a->operand_dtype == DFS_DTYPE_F16;
  void *const k_perm = ws + r.k_perm, *const v_t = ws + r.v_t;
  int32_t* const exps = rounds ? reinterpret_cast<int32_t*>(ws + r.exps) : nullptr;
  uint16_t* pool[4] = {};
  if (a->select) {
    const int64_t at[4] = {r.q_hi, r.q_lo, r.k_hi, r.k_lo};
    for (int i = 0; i < 4; ++i) pool[i] = reinterpret_cast<uint16_t*>(ws + at[i]);
  }
  // A call that reuses its mask reads Q in the attention kernel alone, which
  // then also finds the heads and blocks whose Q leaves the f16 range.
  const bool skip_q = !a->select;
  int32_t* const q_marks = skip_q ? exps : nullptr;
  int32_t* const q_block_marks = q_marks ? reinterpret_cast<int32_t*>(ws + r.marks) : nullptr;
  const int64_t strides[6] = {a->q_head_stride, a->q_row_stride, a->k_head_stride,
                              a->k_row_stride,  a->v_head_stride, a->v_row_stride};
  if (phases & DFS_CALL_PREPARE) {
    int32_t* const flags = rounds ? reinterpret_cast<int32_t*>(ws + r.flags) : nullptr;
    if (int rc = prepare_qkv_impl(a->q, a->k, a->v, a->perm, a->heads, a->seq_len, a->head_dim,
                                  static_cast<int>(a->dtype), a->video_len, a->q_tile, a->k_tile,
                                  static_cast<int>(a->operand_dtype), nullptr, k_perm, v_t, pool[0], pool[1], pool[2],
                                  pool[3], nullptr, flags, skip_q, strides, stream))
      return rc;
    if (rounds)
      if (int rc = prepare_fixup_impl(a->q, a->k, a->v, a->perm, a->heads, a->seq_len, a->head_dim, nullptr, k_perm,
                                      v_t, nullptr, flags, a->q_tile, a->k_tile, skip_q, exps, q_block_marks, strides,
                                      stream))
        return rc;
  }
  if ((phases & DFS_CALL_SELECT) && a->select) {
    const bool one_pass = r.score_bytes > 0;
    void* const shared = ws + r.shared;
    if (int rc = dfs_block_score_topk(pool[0], pool[1], pool[2], pool[3], a->heads, a->head_dim, a->q_tile, a->k_tile,
                                      a->q_blocks, a->k_blocks, a->scored_rows, a->n_cand, a->k_pick, a->dense_col,
                                      a->dense_row, a->row_ptr, a->col_idx,
                                      one_pass ? nullptr : static_cast<float*>(shared), nullptr,
                                      one_pass ? shared : nullptr, r.score_bytes, stream))
      return rc;
  }
  if (phases & DFS_CALL_ATTEND)
    return bsa_fwd_impl(name, nullptr, k_perm, v_t, a->row_ptr, a->col_idx, a->heads, a->seq_len, a->head_dim,
                        static_cast<int>(a->operand_dtype), static_cast<int>(a->operand_dtype),
                        static_cast<float>(a->scale), a->out, static_cast<int>(a->out_dtype), a->out_perm, nullptr,
                        a->cu_seqlens_q, a->cu_seqlens_k, a->n_seq, exps, a->q, a->perm, static_cast<int>(a->dtype),
                        a->out_head_stride, a->out_row_stride, a->long_row, a->long_parts, a->full_rows, a->parts, a->chunks,
                        r.part_bytes ? ws + r.shared : nullptr, r.part_bytes, q_marks, q_block_marks, strides, stream);
  return 0;
}
