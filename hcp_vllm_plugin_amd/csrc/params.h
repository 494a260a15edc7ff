// Kernel parameter blocks and launch functions shared between the kernel
// translation units and the extern "C" layer (abi.hip).
#pragma once

#include "common.h"

namespace hcp {

#ifndef HCP_FWD_WAVES
#define HCP_FWD_WAVES 4  // waves per prefill workgroup, 32 query rows each
#endif
constexpr int kFwdThreads = 64 * HCP_FWD_WAVES;
constexpr int kFwdBM = 32 * HCP_FWD_WAVES;  // query rows per prefill workgroup
constexpr int kFwdBN = 64;                  // keys per prefill tile
constexpr int kFwdPagedMinBlock = 16;      // paged prefill: rows a wave reads from one block

// Column width the attention kernels compute a head_dim in: 64, 128 or 256
// (a smaller head_dim, a multiple of 8, is zero-padded to it inside the
// kernels).
__host__ __device__ constexpr int padded_head_dim(int head_dim) {
  return head_dim <= 64 ? 64 : head_dim <= 128 ? 128 : 256;
}

struct FwdParams {
  const void* q;
  int64_t q_stride_tok, q_stride_head;
  void* out;
  int64_t o_stride_tok, o_stride_head;
  float* lse;
  int64_t lse_stride_head;
  const hcp_varlen_entry* entries;  // varlen: device array
  const int32_t* tiles;             // varlen: device (entry, q_block) pairs
  int32_t num_tiles;                // varlen: tiles; else query blocks
  uint64_t kv_base;                 // varlen, paged: added to the entries' k / v addresses
  int32_t num_heads, num_kv_heads, group;
  int32_t head_dim;  // valid elements per row (<= the kernel's width; the tail is padding)
  float scale_log2;
  int32_t window;           // causal only: key j visible iff j > qpos - window (0: none)
  hcp_varlen_entry single;  // non-varlen: the one entry
  // Optional partial state merged into the result (acc_o NULL: none).  Its
  // rows are indexed like out's; acc_prefix says which side of the merge it
  // is (1: prefix, this pass the suffix).  lse may then be NULL.
  const void* acc_o;
  int64_t acc_stride_tok, acc_stride_head;
  const float* acc_lse;
  int64_t acc_lse_stride_head;
  int32_t acc_prefix;
  // KV split (piece_tiles 0: none): a (query block, head) whose keys span more
  // than piece_tiles tiles runs as unit_pieces() workgroups, each writing an
  // fp32 partial (O normalised, LSE) to the workspace, merged by
  // fwd_reduce_kernel.  Single entry: the first whole_tiles blocks in dispatch
  // order stay whole; block t past them, piece i -> slot (t - whole_tiles) *
  // max_pieces + i.  Varlen: `tiles` holds (entry, q_block, piece, slot)
  // records, slot -1 for a whole block, and `units` the blocks that were cut.
  int32_t piece_tiles, max_pieces, whole_tiles;
  float* ws_o;           // [slot][head][kFwdBM * D], in the kernel's lane order
  float* ws_lse;         // [slot][head][kFwdBM]
  const int32_t* units;  // varlen: device (entry, q_block, first slot, pieces) records
  int32_t num_units;
};

// Keys [lo, lo + n) of an entry that the rows of query block qb see: the
// workgroup's key range before it is cut into tiles.
struct UnitKeys {
  int64_t lo, n;
};
__host__ __device__ inline UnitKeys unit_keys(int64_t kv_len, int64_t causal_offset, int64_t qb,
                                              bool causal, int32_t window) {
  UnitKeys u{0, kv_len};
  if (causal) {
    const int64_t first = causal_offset + qb * kFwdBM;  // last key of the block's first row
    if (window > 0 && first - window + 1 > 0)
      u.lo = first - window + 1 < kv_len ? first - window + 1 : kv_len;
    const int64_t end = first + kFwdBM < kv_len ? first + kFwdBM : kv_len;
    u.n = end > u.lo ? end - u.lo : 0;
  }
  return u;
}
__host__ __device__ inline int unit_pieces(int tiles, int piece_tiles) {
  return tiles > piece_tiles ? (tiles + piece_tiles - 1) / piece_tiles : 1;
}
// first tile of piece i of np (never an empty piece while np <= tiles)
__host__ __device__ inline int piece_begin(int tiles, int np, int i) {
  return static_cast<int>(static_cast<int64_t>(tiles) * i / np);
}

struct DecParams {
  const void* q;
  int64_t q_stride_tok, q_stride_head;
  // the launch's splits: one record per split, each naming the next of its
  // workgroup (works), or an entry index and a key range each
  const hcp_decode_work* works;
  const hcp_varlen_entry* entries;
  const hcp_decode_split* splits;
  int32_t num_splits;
  int32_t num_wgs;   // workgroups per KV head and head chunk
  uint64_t kv_base;  // added to the k / v addresses of paged records
  float* ws_o;    // [num_splits, H, D]
  float* ws_lse;  // [num_splits, H]
  int32_t num_heads, num_kv_heads, group;
  int32_t head_chunks;  // ceil(group / 16): workgroups per (split, KV head)
  int32_t head_dim;     // valid elements per row (<= the kernel's width)
  bool keep_nan;  // NaN scores make their row NaN (else their split is left out): picks the kernel
  float scale_log2;
};

struct RedParams {
  const float* ws_o;
  const float* ws_lse;
  const int32_t* seq_partial_start;
  const int32_t* rows;  // output row of each sequence (NULL: its index)
  // decode_paged_kernel's launches: first and last of the num_slots slots of
  // each sequence (first > last: none, by more than 1: its row is left as it
  // is), in place of seq_partial_start
  const int32_t* seq_slots;
  int32_t num_slots;
  int32_t num_seqs;
  void* out;
  int64_t o_stride_tok, o_stride_head;
  float* lse;
  int64_t lse_stride_head;
  int32_t num_heads;
  int32_t head_dim;  // valid elements per row (<= the kernel's width)
  int32_t groups;    // 1, 2 or 4 column groups per (sequence, head), each over a share of the partials
  // optional running accumulator merged in as one more partial (NULL: none)
  const void* acc_o;
  int64_t acc_stride_tok, acc_stride_head;
  const float* acc_lse;
  int64_t acc_lse_stride_head;
};

constexpr int kDecMaxSeqs = HCP_DECODE_PAGED_MAX_SEQS;  // sequences of a launch that partitions itself

// A pure decode batch over a paged cache, read straight from the step's
// metadata: every workgroup works out its own share of the keys.
struct PagedDecParams {
  DecParams d;           // no splits; d.num_wgs workgroups per KV head and chunk
  hcp_kv_segment kv;     // the cache; block_table, start and len are per sequence
  const void* lens;      // [num_seqs] int32 or int64
  bool lens_wide;
  int32_t num_seqs;
  int64_t bt_stride;     // elements between block-table rows
  int64_t max_len;       // keys a block-table row can name
  int32_t window;        // 0: none
  int32_t* seq_slots;    // [2 * num_seqs]: first and last slot of each sequence (0, -1: no keys;
                         // 0, -2: HCP_LEN_NOT_RUN)
};

struct MergeParams {
  void* out;
  int64_t o_stride_tok, o_stride_head;
  float* out_lse;
  int64_t out_lse_stride;
  const void* po;
  int64_t p_stride_tok, p_stride_head;
  const float* plse;
  int64_t p_lse_stride;
  const void* so;
  int64_t s_stride_tok, s_stride_head;
  const float* slse;
  int64_t s_lse_stride;
  int64_t num_tokens;
  int32_t num_heads, head_dim;
  int32_t out_dtype, p_dtype, s_dtype;
};

struct CacheParams {
  const void* key;
  int64_t k_stride_tok, k_stride_head;
  const void* value;
  int64_t v_stride_tok, v_stride_head;
  const void* slots;  // int32 or int64, one per token
  int64_t num_tokens;
  int32_t num_kv_heads;
  int32_t cpr;        // head_dim / 8: 16-byte chunks per row
  int32_t cpr_shift;  // log2(cpr) when cpr is a power of two, else -1
  void* k_cache;
  void* v_cache;
  int64_t stride_block, stride_head, stride_tok;
  int64_t num_slots;  // num_blocks * block_size
  int32_t bs_shift, bs_mask;
};

// Gather of paged KV segments into one contiguous [total, Hkv, D] K and V
// (prefill over caches with blocks shorter than a wave's 16 rows).
struct GatherParams {
  const hcp_varlen_entry* entries;  // device: paged segments
  const int64_t* out_start;         // device: first output token of each entry
  int64_t max_len;                  // longest segment
  int32_t num_entries;
  int32_t num_kv_heads;
  int32_t cpr;        // head_dim / 8: 16-byte chunks per row
  int32_t cpr_shift;  // log2(cpr) when cpr is a power of two, else -1
  int32_t head_dim;
  void* k_out;
  void* v_out;
};

// One step's metadata, to host memory (fetch_metadata_kernel).
struct MetaParams {
  const void* qsl;
  const void* lens;
  const void* bt;  // NULL: zeros
  int64_t qsl_stride, lens_stride, bt_stride;
  bool qsl_wide, lens_wide, bt_wide;  // int64, else int32
  int32_t n;
  int64_t token;
  int64_t* out;  // [3 n + 2]: the token, then the values
  int64_t max_len;
  int64_t* dev;  // [2 n] or NULL: the lengths of a plain decode batch, the lengths
};

// Prefill in D columns (padded_head_dim): the attention kernel and, when p
// carries a KV split, the merge of its partials into out / lse (and acc).
template <int D>
hipError_t launch_fwd_width(const FwdParams& p, int dtype, bool causal, bool paged, bool varlen,
                            hipStream_t st);
template <>
hipError_t launch_fwd_width<64>(const FwdParams&, int, bool, bool, bool, hipStream_t);
template <>
hipError_t launch_fwd_width<128>(const FwdParams&, int, bool, bool, bool, hipStream_t);
template <>
hipError_t launch_fwd_width<256>(const FwdParams&, int, bool, bool, bool, hipStream_t);
inline hipError_t launch_fwd(const FwdParams& p, int head_dim, int dtype, bool causal, bool paged,
                             bool varlen, hipStream_t st) {
  switch (padded_head_dim(head_dim)) {
    case 256: return launch_fwd_width<256>(p, dtype, causal, paged, varlen, st);
    case 128: return launch_fwd_width<128>(p, dtype, causal, paged, varlen, st);
    default: return launch_fwd_width<64>(p, dtype, causal, paged, varlen, st);
  }
}
hipError_t launch_decode(const DecParams& dp, const RedParams& rp, int head_dim,
                         int dtype, hipStream_t st);
hipError_t launch_decode_paged(const PagedDecParams& p, const RedParams& rp, int head_dim,
                               int dtype, hipStream_t st);
hipError_t launch_merge(const MergeParams& p, hipStream_t st);
hipError_t launch_cache_write(const CacheParams& p, bool slots_i64, hipStream_t st);
hipError_t launch_fetch_metadata(const MetaParams& p, hipStream_t st);
hipError_t launch_gather(const GatherParams& p, hipStream_t st);

}  // namespace hcp
