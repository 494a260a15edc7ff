// extern "C" boundary of libhcp_mi355x.so: argument validation, host-side
// planners and kernel launches.  Declarations and their reference citations
// are in include/hcp_mi355x.h.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <functional>
#include <mutex>
#include <new>
#include <numeric>
#include <vector>

#include "params.h"

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int launch_status(hipError_t e, const char* what) {
  if (e == hipSuccess) return HCP_OK;
  return fail(HCP_ELAUNCH, "%s: HIP launch failed: %s", what, hipGetErrorString(e));
}

bool dtype16(int32_t d) { return d == HCP_DTYPE_F16 || d == HCP_DTYPE_BF16; }

int check_heads(int32_t h, int32_t hkv, int32_t d, int32_t dtype, const char* who) {
  if (h <= 0 || hkv <= 0) return fail(HCP_EINVAL, "%s: num_heads/num_kv_heads must be > 0", who);
  if (h % hkv != 0)
    return fail(HCP_EINVAL, "%s: num_heads (%d) not a multiple of num_kv_heads (%d)", who, h, hkv);
  if (d < 8 || d > 256 || d % 8)
    return fail(HCP_EUNSUPPORTED, "%s: head_dim %d not supported (a multiple of 8 up to 256)",
                who, d);
  if (!dtype16(dtype)) return fail(HCP_EUNSUPPORTED, "%s: dtype %d not supported", who, dtype);
  return HCP_OK;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
bool aligned8(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 7) == 0; }

int check_segment(const hcp_kv_segment& s, int32_t hd, const char* who, int idx) {
  if (s.len < 0 || s.start < 0) return fail(HCP_EINVAL, "%s: entry %d: negative kv start/len", who, idx);
  if (s.len > 0 && (s.k_addr == 0 || s.v_addr == 0))
    return fail(HCP_EINVAL, "%s: entry %d: null k/v address", who, idx);
  if ((s.k_addr & 15) || (s.v_addr & 15))
    return fail(HCP_EINVAL, "%s: entry %d: k/v address not 16-byte aligned", who, idx);
  if ((s.stride_tok % 8) || (s.stride_head % 8) || (s.block_table && (s.stride_block % 8)))
    return fail(HCP_EINVAL, "%s: entry %d: kv strides must be multiples of 8 elements", who, idx);
  if (s.block_table) {
    if (s.block_size <= 0 || (s.block_size & (s.block_size - 1)))
      return fail(HCP_EINVAL, "%s: entry %d: block_size %d not a power of two", who, idx,
                  s.block_size);
  }
  (void)hd;
  return HCP_OK;
}

// Optional partial state merged into an attention pass's result.
struct AccArgs {
  const void* o;
  int64_t stride_tok, stride_head;
  const float* lse;
  int64_t lse_stride_head;
  int32_t prefix;
};

int check_acc(const AccArgs& a, const char* who) {
  if (!a.o || !a.lse) return fail(HCP_EINVAL, "%s: null merge partial out/lse", who);
  if (!aligned16(a.o)) return fail(HCP_EINVAL, "%s: merge partial not 16-byte aligned", who);
  if ((a.stride_tok | a.stride_head) % 8)
    return fail(HCP_EINVAL, "%s: merge partial strides must be multiples of 8 elements", who);
  if (a.stride_tok <= 0 || a.stride_tok >= (int64_t{1} << 24))
    return fail(HCP_EUNSUPPORTED, "%s: merge partial token stride must be in (0, 2^24) elements",
                who);
  return HCP_OK;
}

void set_acc(hcp::FwdParams& p, const AccArgs* a) {
  if (!a) return;
  p.acc_o = a->o;
  p.acc_stride_tok = a->stride_tok;
  p.acc_stride_head = a->stride_head;
  p.acc_lse = a->lse;
  p.acc_lse_stride_head = a->lse_stride_head;
  p.acc_prefix = a->prefix != 0;
}

// ---- KV split of a prefill launch ------------------------------------------
constexpr int kNumCus = 256;
// (query block, head, piece) workgroups of a split launch, and the slots of its
// workspace: 135 MB of partials at head_dim 128 (hcp_split_limits)
constexpr int kMaxPieces = 2048;
constexpr int kMaxUnits = 4 * kNumCus;  // (query block, head) pairs of a launch worth cutting
constexpr int kMinPieceTiles = 4;   // a shorter piece is mostly prologue and epilogue

// A query block of a launch: its tiles and how many of the workgroup's four
// waves have query rows.
struct Unit {
  int tiles, waves;
};
// How a launch is cut: blocks of more than `tiles` tiles into pieces, except
// the `whole` longest.
struct Cut {
  int tiles = 0, whole = 0;
};

// Estimated time (us) of a launch over `units` (per head, longest first) cut
// as `c`, or a lower bound of it that is already past `limit`.  The workgroups
// of one XCD (all XCDs get the same mix), longest first, are run through its
// CUs as the hardware runs them: two to a CU (one at head_dim 256), the next
// into the first slot that frees.  Two workgroups on a CU take tile_us per
// tile (128 rows x 64 keys) between them; one alone takes up to 15% longer
// per tile than two (less when few CUs are busy and the clock is higher), and
// two with one wave of rows each run side by side.  Measured / estimated, us:
// 512 x 32768 at 28 / 4 x 128 whole 488 / 495, cut in 2, 4, 9, 16: 320, 257,
// 248, 262 / 298, 265, 247, 286; 512 x 4096 whole 67 / 64, cut in 2, 4, 8: 48,
// 47, 55 / 48, 48, 56; 3001 x 5003 at 14 / 2 x 64 whole 93 / 91, cut in 3: 82 /
// 77, cut in 3 past 18 whole blocks 74 / 75; 600 x 6000 at 16 / 8 x 256 whole
// 168 / 170, cut in 3: 82 / 79.
// `padded`: every cut block has as many slots in the workspace as the longest.
double split_cost(const std::vector<Unit>& units, Cut c, int group, int num_kvh, int dw,
                  bool padded, double limit, bool* hopeless = nullptr) {
  const double tile_us = dw == 64 ? 0.54 : dw == 128 ? 0.97 : 1.75;
  const double first_us = dw == 256 ? 5.0 : 3.0;   // start and end of a first workgroup
  const double start_us = dw == 256 ? 5.0 : 1.0;   // of one that follows
  const double part_us = dw == 64 ? 0.006 : dw == 128 ? 0.012 : 0.04;  // per partial
  const double reduce_us = dw == 256 ? 8.0 : 6.0;  // the second launch
  const int per_cu = dw == 256 ? 1 : 2;
  // by waves with rows: work of a tile relative to a full one, and the time of
  // a workgroup alone on its CU relative to its work
  static constexpr double kWork[5] = {0.5, 0.5, 0.65, 0.85, 1.0};
  static constexpr double kAlone[5] = {1.8, 1.8, 1.55, 1.3, 1.15};
  static_assert(HCP_FWD_WAVES == 4, "measured with four waves to a workgroup");
  // one XCD's share of the workgroups (xcd_remap), or the whole machine
  const bool by_xcd = num_kvh <= hcp::kNumXcd && hcp::kNumXcd % num_kvh == 0;
  const int share = by_xcd ? hcp::kNumXcd / num_kvh : 1;
  const int cus = by_xcd ? kNumCus / hcp::kNumXcd : kNumCus;
  const int64_t per = static_cast<int64_t>(group) * (by_xcd ? 1 : num_kvh);
  auto pieces = [&](size_t u) {
    return c.tiles > 0 && static_cast<int>(u) >= c.whole ? hcp::unit_pieces(units[u].tiles, c.tiles)
                                                         : 1;
  };
  struct Job {
    double work, alone;
  };
  std::vector<Job> jobs;  // workgroups of one head
  int64_t n = 0, parts = 0, most = 1;
  for (size_t u = 0; u < units.size(); ++u) {
    n += pieces(u);
    if (pieces(u) > 1) parts += pieces(u);
    most = std::max<int64_t>(most, pieces(u));
  }
  const int64_t slots = padded ? (static_cast<int64_t>(units.size()) - c.whole) * most : parts;
  if (c.tiles > 0 && std::max(n, slots) * group * num_kvh > kMaxPieces) return 1e30;
  const double busy = std::min(1.0, static_cast<double>(n * per) / (cus * share));
  const double full_alone = 1.0 + 0.3 * std::max(0.0, busy - 0.5);
  const double merge_us =
      parts > 0 ? reduce_us + static_cast<double>(parts) * group * num_kvh * part_us : 0.0;
  double sum = 0;
  for (size_t u = 0; u < units.size(); ++u) {
    const int nt = units[u].tiles, np = pieces(u), w = units[u].waves;
    const double alone = per_cu == 1 ? 1.0 : w == 4 ? full_alone : kAlone[w];
    for (int i = 0; i < np; ++i) {
      const int tiles = hcp::piece_begin(nt, np, i + 1) - hcp::piece_begin(nt, np, i);
      jobs.push_back({tiles * tile_us * kWork[w], alone});
      sum += jobs.back().work + start_us;
    }
  }
  // evenly spread at best: not worth running through when that already loses
  const double even = sum * per / (static_cast<double>(cus) * share) + merge_us;
  if (even >= limit) {
    if (hopeless) *hopeless = true;
    return even;
  }
  std::sort(jobs.begin(), jobs.end(), [](const Job& a, const Job& b) { return a.work > b.work; });
  struct Cu {
    double at = 0;        // time its jobs' work stands at
    Job job[2];
    int n = 0;
    double next() const {  // when its next job ends
      return at + (n == 1 ? job[0].work * job[0].alone : 2 * std::min(job[0].work, job[1].work));
    }
  };
  std::vector<Cu> cu(cus);
  int64_t j = 0;
  const int64_t items = n * per;
  auto give = [&](Cu& x, double extra) {
    x.job[x.n] = jobs[j / per];
    x.job[x.n++].work += extra;
    j += share;
  };
  for (int s = 0; s < per_cu; ++s)
    for (Cu& x : cu)
      if (j < items) give(x, first_us);
  typedef std::pair<double, int> Ev;  // (end of a CU's next job, CU), earliest on top
  std::vector<Ev> heap;
  for (int i = 0; i < cus; ++i)
    if (cu[i].n) heap.push_back({cu[i].next(), i});
  std::make_heap(heap.begin(), heap.end(), std::greater<Ev>());
  double end = 0;
  while (!heap.empty()) {
    std::pop_heap(heap.begin(), heap.end(), std::greater<Ev>());
    Cu& x = cu[heap.back().second];
    end = heap.back().first;
    if (end + merge_us >= limit) break;  // jobs end in order of time: it loses
    if (x.n == 1) {
      x.n = 0;
    } else {
      const double d = std::min(x.job[0].work, x.job[1].work);
      Job left[2];
      int m = 0;
      for (const Job& y : x.job)
        if (y.work - d > 1e-9) left[m++] = {y.work - d, y.alone};
      for (int i = 0; i < m; ++i) x.job[i] = left[i];
      x.n = m;
    }
    x.at = end;
    while (x.n < per_cu && j < items) give(x, start_us);
    if (x.n == 0) {
      heap.pop_back();
    } else {
      heap.back().first = x.next();
      std::push_heap(heap.begin(), heap.end(), std::greater<Ev>());
    }
  }
  return end + merge_us;
}

// The cut of a launch over `units`, longest first; tiles 0 when cutting does
// not pay (8% or more by the estimate, whose error is about that).
Cut choose_cut(const std::vector<Unit>& units, int group, int num_kvh, int dw, bool padded) {
  Cut best;
  const int heads = group * num_kvh;
  // past 4 workgroups per CU the dispatch order alone evens the load out to
  // what the partials of a cut would cost
  if (units.empty() || static_cast<int64_t>(units.size()) * heads > kMaxUnits) return best;
  const int mx = units[0].tiles;
  if (mx < 2 * kMinPieceTiles) return best;
  double t_best = split_cost(units, best, group, num_kvh, dw, padded, 1e30) * 0.92;
  // whole blocks spread evenly as they are: no cut can win
  bool none = false;
  split_cost(units, best, group, num_kvh, dw, padded, t_best, &none);
  if (none) return best;
  for (int rounds = 0; rounds < 4; ++rounds) {
    // rounds > 0: only what is left after `rounds` whole blocks per CU
    Cut c;
    c.whole = kNumCus * rounds / heads;
    if (rounds > 0 && (c.whole == 0 || c.whole >= static_cast<int>(units.size()))) break;
    const int top = units[c.whole].tiles;
    for (int k : {2, 3, 4, 6, 9, 12, 16, 24, 32, 48, 64}) {
      const int tiles = (top + k - 1) / k;
      if (tiles < kMinPieceTiles) break;
      if (tiles == c.tiles) continue;
      c.tiles = tiles;
      bool hopeless = false;
      const double t = split_cost(units, c, group, num_kvh, dw, padded, t_best, &hopeless);
      // more pieces only add to the even share: none of them can win either
      if (hopeless || t > 1e29) break;
      if (t < t_best) {
        t_best = t;
        best = c;
      }
    }
  }
  return best;
}

int unit_waves(const hcp_varlen_entry& e, int64_t qb) {
  const int64_t rows = e.q_len - qb * hcp::kFwdBM;
  return rows >= hcp::kFwdBM ? hcp::kFwdBM / 32 : static_cast<int>((rows + 31) / 32);
}

int unit_tiles(const hcp_varlen_entry& e, int64_t qb, bool causal, int32_t window) {
  const int64_t n = hcp::unit_keys(e.kv.len, e.causal_offset, qb, causal, window).n;
  return static_cast<int>((n + hcp::kFwdBN - 1) / hcp::kFwdBN);
}

// (O, LSE) partials of `slots` query blocks x num_heads, fp32
size_t split_ws_o_bytes(int64_t slots, int32_t num_heads, int32_t head_dim) {
  return static_cast<size_t>(slots) * num_heads * hcp::kFwdBM * hcp::padded_head_dim(head_dim) *
         sizeof(float);
}
size_t split_ws_bytes(int64_t slots, int32_t num_heads, int32_t head_dim) {
  return split_ws_o_bytes(slots, num_heads, head_dim) +
         static_cast<size_t>(slots) * num_heads * hcp::kFwdBM * sizeof(float);
}

// Workspace of a split launch into p; `slots` partials per head.
int set_split(hcp::FwdParams& p, int32_t piece_tiles, int64_t slots, void* ws, size_t bytes,
              const char* who) {
  const size_t need = split_ws_bytes(slots, p.num_heads, p.head_dim);
  if (!ws || bytes < need)
    return fail(HCP_EWORKSPACE, "%s: workspace %zu bytes < %zu needed", who, bytes, need);
  if (!aligned16(ws)) return fail(HCP_EINVAL, "%s: workspace not 16-byte aligned", who);
  p.piece_tiles = piece_tiles;
  p.ws_o = static_cast<float*>(ws);
  p.ws_lse = reinterpret_cast<float*>(static_cast<char*>(ws) +
                                      split_ws_o_bytes(slots, p.num_heads, p.head_dim));
  return HCP_OK;
}

struct SplitArgs {
  int32_t piece_tiles, whole_blocks;
  void* ws;
  size_t bytes;
  const int32_t* units;  // varlen only
  int32_t num_units, num_slots;
};

}  // namespace

extern "C" {

int hcp_abi_version(void) { return HCP_ABI_VERSION; }

const char* hcp_last_error(void) { return g_err; }

static int fwd_lse_impl(const char* who, const void* q, const void* k, const void* v, void* out,
                        float* lse, int64_t tq, int64_t tk, int32_t num_heads,
                        int32_t num_kv_heads, int32_t head_dim, int64_t q_stride_tok,
                        int64_t q_stride_head, int64_t k_stride_tok, int64_t k_stride_head,
                        int64_t v_stride_tok, int64_t v_stride_head, int64_t o_stride_tok,
                        int64_t o_stride_head, int64_t lse_stride_head, float scale,
                        int32_t causal, int64_t causal_offset, int32_t window, int32_t dtype,
                        void* stream, const AccArgs* acc, const SplitArgs* split = nullptr) {
  int rc = check_heads(num_heads, num_kv_heads, head_dim, dtype, who);
  if (rc) return rc;
  if (tq < 0 || tk < 0) return fail(HCP_EINVAL, "%s: negative tq/tk", who);
  if (tq == 0) return HCP_OK;
  if (!q || !out || (!lse && !acc)) return fail(HCP_EINVAL, "%s: null q/out/lse", who);
  if (acc && (rc = check_acc(*acc, who))) return rc;
  if (tk > 0 && (!k || !v)) return fail(HCP_EINVAL, "%s: null k/v", who);
  if (!aligned16(q) || !aligned16(out) || (tk > 0 && (!aligned16(k) || !aligned16(v))))
    return fail(HCP_EINVAL, "%s: q/k/v/out must be 16-byte aligned", who);
  if ((q_stride_tok | q_stride_head | k_stride_tok | k_stride_head | v_stride_tok |
       v_stride_head | o_stride_tok | o_stride_head) % 8)
    return fail(HCP_EINVAL, "%s: strides must be multiples of 8 elements", who);
  if (!(scale > 0.f) || !std::isfinite(scale))
    return fail(HCP_EINVAL, "%s: scale must be finite and > 0", who);
  if (tq > (int64_t)INT32_MAX * 64) return fail(HCP_EINVAL, "%s: tq too large", who);
  // the kernel counts a segment's keys (and its tiles' key offsets) in int32
  if (tk > (int64_t)INT32_MAX - 256) return fail(HCP_EUNSUPPORTED, "%s: tk too large", who);
  if (window < 0) return fail(HCP_EINVAL, "%s: negative window", who);

  hcp::FwdParams p{};
  p.q = q;
  p.q_stride_tok = q_stride_tok;
  p.q_stride_head = q_stride_head;
  p.out = out;
  p.o_stride_tok = o_stride_tok;
  p.o_stride_head = o_stride_head;
  p.lse = lse;
  p.lse_stride_head = lse_stride_head;
  p.num_heads = num_heads;
  p.num_kv_heads = num_kv_heads;
  p.group = num_heads / num_kv_heads;
  p.head_dim = head_dim;
  p.scale_log2 = scale * hcp::kLog2e;
  p.num_tiles = static_cast<int32_t>((tq + hcp::kFwdBM - 1) / hcp::kFwdBM);
  p.single.q_start = 0;
  p.single.q_len = tq;
  p.single.causal_offset = causal ? causal_offset : 0;
  p.window = causal ? window : 0;
  p.single.kv.k_addr = reinterpret_cast<uint64_t>(k);
  p.single.kv.v_addr = reinterpret_cast<uint64_t>(v);
  p.single.kv.stride_tok = k_stride_tok;
  p.single.kv.stride_head = k_stride_head;
  p.single.kv.len = tk;
  if (k_stride_tok != v_stride_tok || k_stride_head != v_stride_head)
    return fail(HCP_EUNSUPPORTED, "%s: k and v must share strides", who);
  // the kernel's tile offsets are 32-bit: 64 rows of a tile span under 2^31
  // bytes (a single key row is never stepped over)
  if (tk > 1 && (k_stride_tok <= 0 || k_stride_tok >= (int64_t{1} << 24)))
    return fail(HCP_EUNSUPPORTED, "%s: k/v token stride must be in (0, 2^24) elements", who);
  set_acc(p, acc);
  if (split) {
    if (split->whole_blocks < 0 || split->whole_blocks >= p.num_tiles)
      return fail(HCP_EINVAL, "%s: whole_blocks %d of %d", who, split->whole_blocks, p.num_tiles);
    // blocks in dispatch order: the last one first under a causal mask
    int mp = 1;
    for (int64_t t = split->whole_blocks; t < p.num_tiles; ++t)
      mp = std::max(mp, hcp::unit_pieces(unit_tiles(p.single, causal ? p.num_tiles - 1 - t : t,
                                                    causal != 0, p.window),
                                         split->piece_tiles));
    const int64_t slots = static_cast<int64_t>(p.num_tiles - split->whole_blocks) * mp;
    if (slots * num_heads * 4 > INT32_MAX)
      return fail(HCP_EINVAL, "%s: too many pieces", who);
    p.whole_tiles = split->whole_blocks;
    p.max_pieces = mp;
    if ((rc = set_split(p, split->piece_tiles, slots, split->ws, split->bytes, who))) return rc;
  }
  hipError_t e = hcp::launch_fwd(p, head_dim, dtype, causal != 0, false, false,
                                 static_cast<hipStream_t>(stream));
  return launch_status(e, who);
}

int hcp_split_limits(int32_t head_dim, int32_t* max_units, int32_t* min_keys, int32_t* max_pieces,
                     size_t* max_workspace) {
  if (head_dim <= 0 || head_dim > 256 || !max_units || !min_keys || !max_pieces || !max_workspace)
    return fail(HCP_EINVAL, "hcp_split_limits: bad arguments");
  *max_units = kMaxUnits;
  *min_keys = (2 * kMinPieceTiles - 1) * hcp::kFwdBN + 1;  // a block of two pieces
  *max_pieces = kMaxPieces;
  *max_workspace = split_ws_bytes(kMaxPieces, 1, head_dim);
  return HCP_OK;
}

int hcp_plan_fwd_split(int64_t tq, int64_t tk, int32_t num_heads, int32_t num_kv_heads,
                       int32_t head_dim, int32_t causal, int64_t causal_offset, int32_t window,
                       int32_t* whole_blocks, size_t* workspace_bytes) try {
  const char* who = "hcp_plan_fwd_split";
  int rc = check_heads(num_heads, num_kv_heads, head_dim, HCP_DTYPE_BF16, who);
  if (rc) return rc;
  if (tq < 0 || tk < 0 || window < 0 || !whole_blocks || !workspace_bytes)
    return fail(HCP_EINVAL, "%s: bad arguments", who);
  *whole_blocks = 0;
  *workspace_bytes = 0;
  const int64_t blocks = tq / hcp::kFwdBM + (tq % hcp::kFwdBM != 0);
  if (tk > (int64_t)INT32_MAX - 256 || blocks > kMaxUnits || blocks * num_heads > kMaxUnits)
    return 0;
  hcp_varlen_entry e{};
  e.q_len = tq;
  e.causal_offset = causal ? causal_offset : 0;
  e.kv.len = tk;
  std::vector<Unit> units;  // in dispatch order (longest first)
  for (int64_t t = 0; t < blocks; ++t) {
    const int64_t qb = causal ? blocks - 1 - t : t;
    units.push_back({unit_tiles(e, qb, causal != 0, causal ? window : 0), unit_waves(e, qb)});
  }
  const Cut c = choose_cut(units, num_heads / num_kv_heads, num_kv_heads,
                           hcp::padded_head_dim(head_dim), true);
  if (c.tiles > 0) {
    int mp = 1;
    for (size_t t = c.whole; t < units.size(); ++t)
      mp = std::max(mp, hcp::unit_pieces(units[t].tiles, c.tiles));
    *whole_blocks = c.whole;
    *workspace_bytes = split_ws_bytes((blocks - c.whole) * mp, num_heads, head_dim);
  }
  return c.tiles;
} catch (const std::bad_alloc&) {
  return fail(HCP_EINVAL, "hcp_plan_fwd_split: out of host memory");
}

int hcp_attn_fwd_lse_split(const void* q, const void* k, const void* v, void* out, float* lse,
                           int64_t tq, int64_t tk, int32_t num_heads, int32_t num_kv_heads,
                           int32_t head_dim, int64_t q_stride_tok, int64_t q_stride_head,
                           int64_t k_stride_tok, int64_t k_stride_head, int64_t v_stride_tok,
                           int64_t v_stride_head, int64_t o_stride_tok, int64_t o_stride_head,
                           int64_t lse_stride_head, float scale, int32_t causal,
                           int64_t causal_offset, int32_t window, const void* acc_out,
                           int64_t acc_stride_tok, int64_t acc_stride_head,
                           const float* acc_lse, int64_t acc_lse_stride_head,
                           int32_t acc_is_prefix, int32_t piece_tiles, int32_t whole_blocks,
                           void* workspace, size_t workspace_bytes, int32_t dtype,
                           void* stream) {
  const char* who = "hcp_attn_fwd_lse_split";
  if (piece_tiles <= 0) return fail(HCP_EINVAL, "%s: piece_tiles must be > 0", who);
  const AccArgs acc{acc_out, acc_stride_tok, acc_stride_head, acc_lse, acc_lse_stride_head,
                    acc_is_prefix};
  const SplitArgs split{piece_tiles, whole_blocks, workspace, workspace_bytes, nullptr, 0, 0};
  return fwd_lse_impl(who, q, k, v, out, lse, tq, tk, num_heads, num_kv_heads, head_dim,
                      q_stride_tok, q_stride_head, k_stride_tok, k_stride_head, v_stride_tok,
                      v_stride_head, o_stride_tok, o_stride_head, lse_stride_head, scale, causal,
                      causal_offset, window, dtype, stream, acc_out || acc_lse ? &acc : nullptr,
                      &split);
}

int hcp_attn_fwd_lse(const void* q, const void* k, const void* v, void* out, float* lse,
                     int64_t tq, int64_t tk, int32_t num_heads, int32_t num_kv_heads,
                     int32_t head_dim, int64_t q_stride_tok, int64_t q_stride_head,
                     int64_t k_stride_tok, int64_t k_stride_head, int64_t v_stride_tok,
                     int64_t v_stride_head, int64_t o_stride_tok, int64_t o_stride_head,
                     int64_t lse_stride_head, float scale, int32_t causal,
                     int64_t causal_offset, int32_t window, int32_t dtype, void* stream) {
  return fwd_lse_impl("hcp_attn_fwd_lse", q, k, v, out, lse, tq, tk, num_heads, num_kv_heads,
                      head_dim, q_stride_tok, q_stride_head, k_stride_tok, k_stride_head,
                      v_stride_tok, v_stride_head, o_stride_tok, o_stride_head, lse_stride_head,
                      scale, causal, causal_offset, window, dtype, stream, nullptr);
}

int hcp_attn_fwd_lse_merge(const void* q, const void* k, const void* v, void* out, float* lse,
                           int64_t tq, int64_t tk, int32_t num_heads, int32_t num_kv_heads,
                           int32_t head_dim, int64_t q_stride_tok, int64_t q_stride_head,
                           int64_t k_stride_tok, int64_t k_stride_head, int64_t v_stride_tok,
                           int64_t v_stride_head, int64_t o_stride_tok, int64_t o_stride_head,
                           int64_t lse_stride_head, float scale, int32_t causal,
                           int64_t causal_offset, int32_t window, const void* acc_out,
                           int64_t acc_stride_tok, int64_t acc_stride_head,
                           const float* acc_lse, int64_t acc_lse_stride_head,
                           int32_t acc_is_prefix, int32_t dtype, void* stream) {
  const AccArgs acc{acc_out, acc_stride_tok, acc_stride_head, acc_lse, acc_lse_stride_head,
                    acc_is_prefix};
  return fwd_lse_impl("hcp_attn_fwd_lse_merge", q, k, v, out, lse, tq, tk, num_heads,
                      num_kv_heads, head_dim, q_stride_tok, q_stride_head, k_stride_tok,
                      k_stride_head, v_stride_tok, v_stride_head, o_stride_tok, o_stride_head,
                      lse_stride_head, scale, causal, causal_offset, window, dtype, stream, &acc);
}

int hcp_varlen_block_m(int32_t head_dim, int32_t dtype) {
  (void)head_dim;
  (void)dtype;
  return hcp::kFwdBM;
}

static int check_prefill_entry(const hcp_varlen_entry& en, const char* who, int32_t i) {
  // the kernel counts a segment's keys (and its tiles' key offsets) in int32
  if (en.kv.len > (int64_t)INT32_MAX - 256)
    return fail(HCP_EUNSUPPORTED, "%s: entry %d: kv len too large", who, i);
  // the prefill kernel reads a wave's 16 rows of a paged tile from one block
  if (en.kv.block_table && (en.kv.stride_tok <= 0 || en.kv.stride_tok >= (int64_t{1} << 24)))
    return fail(HCP_EUNSUPPORTED, "%s: entry %d: paged token stride must be in (0, 2^24)", who, i);
  if (!en.kv.block_table && en.kv.len > 1 &&
      (en.kv.stride_tok <= 0 || en.kv.stride_tok >= (int64_t{1} << 24)))
    return fail(HCP_EUNSUPPORTED, "%s: entry %d: token stride must be in (0, 2^24)", who, i);
  if (en.kv.block_table && (en.kv.stride_block <= 0 || en.kv.stride_block >= (int64_t{1} << 31)))
    return fail(HCP_EUNSUPPORTED, "%s: entry %d: block stride must be in (0, 2^31) elements",
                who, i);
  // the kernel's in-block byte offsets are 32-bit
  if (en.kv.block_table &&
      static_cast<int64_t>(en.kv.block_size) * en.kv.stride_tok * 2 > (int64_t{1} << 32))
    return fail(HCP_EUNSUPPORTED, "%s: entry %d: block_size * token stride spans over 4 GiB",
                who, i);
  if (en.kv.block_table && en.kv.block_size < hcp::kFwdPagedMinBlock)
    return fail(HCP_EUNSUPPORTED, "%s: entry %d: paged prefill needs block_size >= %d, got %d",
                who, i, hcp::kFwdPagedMinBlock, en.kv.block_size);
  return HCP_OK;
}

int hcp_plan_varlen_tiles(const hcp_varlen_entry* entries, int32_t num_entries, int32_t causal,
                          int32_t block_m, int32_t* tiles_out, int32_t cap) {
  const char* who = "hcp_plan_varlen_tiles";
  if (num_entries < 0 || block_m <= 0) return fail(HCP_EINVAL, "%s: bad sizes", who);
  if (num_entries > 0 && !entries) return fail(HCP_EINVAL, "%s: null entries", who);
  struct T {
    int64_t cost;
    int32_t e, qb;
  };
  std::vector<T> v;
  for (int32_t i = 0; i < num_entries; ++i) {
    const hcp_varlen_entry& en = entries[i];
    if (en.q_len < 0 || en.kv.len < 0) return fail(HCP_EINVAL, "%s: entry %d negative", who, i);
    if (int rc = check_prefill_entry(en, who, i)) return rc;
    const int64_t nqb = (en.q_len + block_m - 1) / block_m;
    for (int64_t b = 0; b < nqb; ++b) {
      int64_t keys = en.kv.len;
      if (causal) {
        const int64_t lim = en.causal_offset + (b + 1) * block_m;
        keys = std::max<int64_t>(0, std::min(keys, lim));
      }
      v.push_back({keys, i, static_cast<int32_t>(b)});
    }
  }
  if (static_cast<int64_t>(v.size()) > INT32_MAX) return fail(HCP_EINVAL, "%s: too many tiles", who);
  const int32_t n = static_cast<int32_t>(v.size());
  if (n > cap || (n > 0 && !tiles_out))
    return fail(HCP_EWORKSPACE, "%s: need %d tiles, cap %d", who, n, cap);
  // longest processing time first; ties keep (entry, block) order
  std::stable_sort(v.begin(), v.end(), [](const T& a, const T& b) { return a.cost > b.cost; });
  for (int32_t i = 0; i < n; ++i) {
    tiles_out[2 * i] = v[i].e;
    tiles_out[2 * i + 1] = v[i].qb;
  }
  return n;
}

int hcp_plan_varlen_split(const hcp_varlen_entry* entries, int32_t num_entries, int32_t causal,
                          int32_t window, int32_t num_heads, int32_t num_kv_heads,
                          int32_t head_dim, int32_t* pieces_out, int32_t cap,
                          int32_t* units_out, int32_t* num_units, int32_t* num_slots,
                          int32_t* piece_tiles, size_t* workspace_bytes) try {
  const char* who = "hcp_plan_varlen_split";
  int rc = check_heads(num_heads, num_kv_heads, head_dim, HCP_DTYPE_BF16, who);
  if (rc) return rc;
  if (num_entries < 0 || window < 0 || cap < 0) return fail(HCP_EINVAL, "%s: bad sizes", who);
  if ((num_entries > 0 && !entries) || !num_units || !num_slots || !piece_tiles ||
      !workspace_bytes)
    return fail(HCP_EINVAL, "%s: null pointer", who);
  *num_units = *num_slots = *piece_tiles = 0;
  *workspace_bytes = 0;
  struct U {
    Unit u;
    int32_t e, qb;
  };
  std::vector<U> blocks;
  for (int32_t i = 0; i < num_entries; ++i) {
    const hcp_varlen_entry& en = entries[i];
    if (en.q_len < 0 || en.kv.len < 0) return fail(HCP_EINVAL, "%s: entry %d negative", who, i);
    if ((rc = check_prefill_entry(en, who, i))) return rc;
    const int64_t nqb = en.q_len / hcp::kFwdBM + (en.q_len % hcp::kFwdBM != 0);
    if (nqb > kMaxUnits || (static_cast<int64_t>(blocks.size()) + nqb) * num_heads > kMaxUnits)
      return 0;
    for (int64_t b = 0; b < nqb; ++b)
      blocks.push_back({{unit_tiles(en, b, causal != 0, causal ? window : 0), unit_waves(en, b)},
                        i, static_cast<int32_t>(b)});
  }
  std::stable_sort(blocks.begin(), blocks.end(),
                   [](const U& a, const U& b) { return a.u.tiles > b.u.tiles; });
  std::vector<Unit> units;
  for (const U& b : blocks) units.push_back(b.u);
  const Cut c = choose_cut(units, num_heads / num_kv_heads, num_kv_heads,
                           hcp::padded_head_dim(head_dim), false);
  if (c.tiles == 0) return 0;
  struct P {
    int32_t cost, e, qb, piece, slot;
  };
  std::vector<P> v;
  int32_t slot = 0, nu = 0;
  for (size_t j = 0; j < blocks.size(); ++j) {
    const U& u = blocks[j];
    const int nt = u.u.tiles;
    const int np = static_cast<int>(j) < c.whole ? 1 : hcp::unit_pieces(nt, c.tiles);
    if (static_cast<int64_t>(v.size()) + np > cap || !pieces_out || !units_out)
      return fail(HCP_EWORKSPACE, "%s: piece cap %d exceeded", who, cap);
    if (np == 1) {
      v.push_back({nt, u.e, u.qb, 0, -1});
      continue;
    }
    units_out[4 * nu] = u.e;
    units_out[4 * nu + 1] = u.qb;
    units_out[4 * nu + 2] = slot;
    units_out[4 * nu + 3] = np;
    ++nu;
    for (int i = 0; i < np; ++i)
      v.push_back({hcp::piece_begin(nt, np, i + 1) - hcp::piece_begin(nt, np, i), u.e, u.qb,
                   i, slot++});
  }
  // longest first; among equals the same piece of every block together, so
  // workgroups in flight at once read the same keys
  std::stable_sort(v.begin(), v.end(), [](const P& a, const P& b) {
    return a.cost != b.cost ? a.cost > b.cost : a.piece < b.piece;
  });
  for (size_t i = 0; i < v.size(); ++i) {
    pieces_out[4 * i] = v[i].e;
    pieces_out[4 * i + 1] = v[i].qb;
    pieces_out[4 * i + 2] = v[i].piece;
    pieces_out[4 * i + 3] = v[i].slot;
  }
  *num_units = nu;
  *num_slots = slot;
  *piece_tiles = c.tiles;
  *workspace_bytes = split_ws_bytes(slot, num_heads, head_dim);
  return static_cast<int>(v.size());
} catch (const std::bad_alloc&) {
  return fail(HCP_EINVAL, "hcp_plan_varlen_split: out of host memory");
}

static int fwd_varlen_impl(const char* who, const void* q, int64_t q_stride_tok,
                           int64_t q_stride_head, void* out, int64_t o_stride_tok,
                           int64_t o_stride_head, float* lse, int64_t lse_stride_head,
                           const hcp_varlen_entry* entries, int32_t num_entries,
                           const int32_t* tiles, int32_t num_tiles, int32_t num_heads,
                           int32_t num_kv_heads, int32_t head_dim, float scale, int32_t causal,
                           int32_t window, int32_t paged, int32_t dtype, void* stream,
                           const AccArgs* acc, const SplitArgs* split = nullptr,
                           uint64_t kv_base = 0, bool lse_optional = false) {
  int rc = check_heads(num_heads, num_kv_heads, head_dim, dtype, who);
  if (rc) return rc;
  if (num_entries < 0 || num_tiles < 0) return fail(HCP_EINVAL, "%s: negative counts", who);
  if (num_tiles == 0) return HCP_OK;
  if (!q || !out || (!lse && !acc && !lse_optional) || !entries || !tiles)
    return fail(HCP_EINVAL, "%s: null pointer", who);
  if (acc && (rc = check_acc(*acc, who))) return rc;
  if (!aligned16(q) || !aligned16(out)) return fail(HCP_EINVAL, "%s: q/out not 16-byte aligned", who);
  if ((q_stride_tok | q_stride_head | o_stride_tok | o_stride_head) % 8)
    return fail(HCP_EINVAL, "%s: strides must be multiples of 8 elements", who);
  if (!(scale > 0.f) || !std::isfinite(scale))
    return fail(HCP_EINVAL, "%s: scale must be finite and > 0", who);
  if (window < 0) return fail(HCP_EINVAL, "%s: negative window", who);
  hcp::FwdParams p{};
  p.window = causal ? window : 0;
  p.q = q;
  p.q_stride_tok = q_stride_tok;
  p.q_stride_head = q_stride_head;
  p.out = out;
  p.o_stride_tok = o_stride_tok;
  p.o_stride_head = o_stride_head;
  p.lse = lse;
  p.lse_stride_head = lse_stride_head;
  p.entries = entries;
  p.tiles = tiles;
  p.num_tiles = num_tiles;
  p.kv_base = kv_base;
  p.num_heads = num_heads;
  p.num_kv_heads = num_kv_heads;
  p.group = num_heads / num_kv_heads;
  p.head_dim = head_dim;
  p.scale_log2 = scale * hcp::kLog2e;
  set_acc(p, acc);
  if (split) {
    if (split->num_units < 0 || split->num_slots < 0 || (split->num_units > 0 && !split->units))
      return fail(HCP_EINVAL, "%s: bad split units", who);
    if (static_cast<int64_t>(split->num_units) * num_heads * 4 > INT32_MAX)
      return fail(HCP_EINVAL, "%s: too many split units", who);
    p.units = split->units;
    p.num_units = split->num_units;
    if ((rc = set_split(p, split->piece_tiles, split->num_slots, split->ws, split->bytes, who)))
      return rc;
  }
  hipError_t e = hcp::launch_fwd(p, head_dim, dtype, causal != 0, paged != 0, true,
                                 static_cast<hipStream_t>(stream));
  return launch_status(e, who);
}

int hcp_attn_fwd_varlen(const void* q, int64_t q_stride_tok, int64_t q_stride_head, void* out,
                        int64_t o_stride_tok, int64_t o_stride_head, float* lse,
                        int64_t lse_stride_head, const hcp_varlen_entry* entries,
                        int32_t num_entries, const int32_t* tiles, int32_t num_tiles,
                        int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, float scale,
                        int32_t causal, int32_t window, int32_t paged, int32_t dtype,
                        void* stream) {
  return fwd_varlen_impl("hcp_attn_fwd_varlen", q, q_stride_tok, q_stride_head, out,
                         o_stride_tok, o_stride_head, lse, lse_stride_head, entries, num_entries,
                         tiles, num_tiles, num_heads, num_kv_heads, head_dim, scale, causal,
                         window, paged, dtype, stream, nullptr);
}

int hcp_attn_fwd_varlen_merge(const void* q, int64_t q_stride_tok, int64_t q_stride_head,
                              void* out, int64_t o_stride_tok, int64_t o_stride_head, float* lse,
                              int64_t lse_stride_head, const hcp_varlen_entry* entries,
                              int32_t num_entries, const int32_t* tiles, int32_t num_tiles,
                              int32_t num_heads, int32_t num_kv_heads, int32_t head_dim,
                              float scale, int32_t causal, int32_t window, int32_t paged,
                              const void* acc_out, int64_t acc_stride_tok,
                              int64_t acc_stride_head, const float* acc_lse,
                              int64_t acc_lse_stride_head, int32_t acc_is_prefix, int32_t dtype,
                              void* stream) {
  const AccArgs acc{acc_out, acc_stride_tok, acc_stride_head, acc_lse, acc_lse_stride_head,
                    acc_is_prefix};
  return fwd_varlen_impl("hcp_attn_fwd_varlen_merge", q, q_stride_tok, q_stride_head, out,
                         o_stride_tok, o_stride_head, lse, lse_stride_head, entries, num_entries,
                         tiles, num_tiles, num_heads, num_kv_heads, head_dim, scale, causal,
                         window, paged, dtype, stream, &acc);
}

int hcp_varlen_launch(const hcp_varlen_args* a, void* stream) {
  const char* who = "hcp_varlen_launch";
  if (!a) return fail(HCP_EINVAL, "%s: null arguments", who);
  if (a->piece_tiles < 0) return fail(HCP_EINVAL, "%s: negative piece_tiles", who);
  if (a->kv_base & 15) return fail(HCP_EINVAL, "%s: kv_base not 16-byte aligned", who);
  const AccArgs acc{a->acc_o, a->acc_stride_tok, a->acc_stride_head, a->acc_lse,
                    a->acc_lse_stride_head, a->acc_is_prefix};
  const SplitArgs split{a->piece_tiles, 0, a->workspace, a->workspace_bytes, a->units,
                        a->num_units, a->num_slots};
  return fwd_varlen_impl(who, a->q, a->q_stride_tok, a->q_stride_head, a->out, a->o_stride_tok,
                         a->o_stride_head, a->lse, a->lse_stride_head, a->entries, a->num_entries,
                         a->tiles, a->num_tiles, a->num_heads, a->num_kv_heads, a->head_dim,
                         a->scale, a->causal, a->window, a->paged, a->dtype, stream,
                         a->acc_o || a->acc_lse ? &acc : nullptr,
                         a->piece_tiles > 0 ? &split : nullptr, a->kv_base, true);
}

int hcp_plan_decode_splits(const hcp_varlen_entry* entries, int32_t num_entries,
                           const int32_t* entry_seq, int32_t num_seqs, int32_t causal,
                           int32_t split_tokens, hcp_decode_split* splits_out, int32_t cap,
                           int32_t* seq_partial_start) {
  const char* who = "hcp_plan_decode_splits";
  if (num_entries < 0 || num_seqs < 0 || split_tokens <= 0)
    return fail(HCP_EINVAL, "%s: bad sizes", who);
  if ((num_entries > 0 && (!entries || !entry_seq)) || !seq_partial_start)
    return fail(HCP_EINVAL, "%s: null pointer", who);
  int32_t n = 0;
  int32_t cur = 0;
  seq_partial_start[0] = 0;
  for (int32_t i = 0; i < num_entries; ++i) {
    const int32_t s = entry_seq[i];
    if (s < 0 || s >= num_seqs || s < cur)
      return fail(HCP_EINVAL, "%s: entry %d: sequence %d out of order/range", who, i, s);
    if (entries[i].q_len != 1)
      return fail(HCP_EINVAL, "%s: entry %d: q_len must be 1 for decode", who, i);
    if (entries[i].kv.len < 0 || entries[i].kv.len > INT32_MAX)
      return fail(HCP_EINVAL, "%s: entry %d: kv len out of range", who, i);
    while (cur < s) seq_partial_start[++cur] = n;
    int64_t len = entries[i].kv.len;
    if (causal) len = std::max<int64_t>(0, std::min<int64_t>(len, entries[i].causal_offset + 1));
    // ceil(len / split_tokens) pieces of (nearly) equal size
    const int64_t pieces = (len + split_tokens - 1) / split_tokens;
    const int64_t step = pieces > 0 ? (len + pieces - 1) / pieces : 0;
    for (int64_t b = 0; b < len; b += step) {
      if (n >= cap || !splits_out) return fail(HCP_EWORKSPACE, "%s: split cap %d exceeded", who, cap);
      splits_out[n].entry = i;
      splits_out[n].key_begin = static_cast<int32_t>(b);
      splits_out[n].key_end = static_cast<int32_t>(std::min<int64_t>(len, b + step));
      splits_out[n].slot = n;
      ++n;
    }
  }
  while (cur < num_seqs) seq_partial_start[++cur] = n;
  // dispatch order: longest first, so the last workgroups of the launch are
  // the short splits and the machine drains evenly
  std::stable_sort(splits_out, splits_out + n, [](const hcp_decode_split& a,
                                                  const hcp_decode_split& b) {
    return a.key_end - a.key_begin > b.key_end - b.key_begin;
  });
  return n;
}

int hcp_plan_decode_lists(const hcp_varlen_entry* entries, int32_t num_entries,
                          const int32_t* entry_seq, int32_t num_seqs,
                          int32_t workgroups, int32_t split_tokens, hcp_decode_work* works,
                          int32_t* work_entry, int32_t cap, int32_t* seq_partial_start,
                          int32_t* num_wgs) try {
  const char* who = "hcp_plan_decode_lists";
  if (num_entries < 0 || num_seqs < 0 || workgroups < 0 || split_tokens < 0 ||
      (workgroups > 0) == (split_tokens > 0))
    return fail(HCP_EINVAL, "%s: bad sizes", who);
  if ((num_entries > 0 && (!entries || !entry_seq)) || !seq_partial_start || !num_wgs ||
      (cap > 0 && !works))
    return fail(HCP_EINVAL, "%s: null pointer", who);
  // lengths in chunks of 32 keys, the kernel's step
  auto chunks = [&](int32_t i) { return (entries[i].kv.len + 31) / 32; };
  int64_t total = 0;
  int32_t cur = 0;
  for (int32_t i = 0; i < num_entries; ++i) {
    const int32_t s = entry_seq[i];
    if (s < 0 || s >= num_seqs || s < cur)
      return fail(HCP_EINVAL, "%s: entry %d: sequence %d out of order/range", who, i, s);
    cur = s;
    if (entries[i].q_len != 1)
      return fail(HCP_EINVAL, "%s: entry %d: q_len must be 1 for decode", who, i);
    if (entries[i].kv.len < 0 || entries[i].kv.len > INT32_MAX)
      return fail(HCP_EINVAL, "%s: entry %d: kv len out of range", who, i);
    total += chunks(i);
  }
  // Each split costs its workgroup its start and its end, as long as about 8
  // chunks take; the smallest budget (chunks + splits * kSplitCost) that
  // `wgs` workgroups can hold the batch in is the one to fill them to.  At
  // least two chunks (64 keys) to a workgroup.
  constexpr int64_t kSplitCost = 8;
  const int64_t wgs = std::max<int64_t>(1, std::min<int64_t>(workgroups, (total + 1) / 2));
  // Chunks of an entry with `left` to go that a workgroup with `room` takes:
  // the rest if there is room for it, else whole steps of 4 (one for each of
  // the 4 waves; single chunks in a small share), but none if the room, less
  // the split's own cost, is under 2.
  auto take = [&](int64_t left, int64_t room) -> int64_t {
    room -= kSplitCost;
    if (left <= room) return left;
    const int64_t step = room >= 16 ? 4 : 1;
    const int64_t t = room / step * step;
    return room < 2 ? 0 : t;
  };
  auto fits = [&](int64_t budget) {
    int64_t w = 0, room = budget;
    for (int32_t i = 0; i < num_entries; ++i)
      for (int64_t left = chunks(i); left > 0;) {
        const int64_t t = take(left, room);
        if (t > 0) {
          left -= t;
          room -= t + kSplitCost;
        }
        if (left > 0) {
          room = budget;
          if (++w >= wgs) return false;
        }
      }
    return true;
  };
  int64_t budget = kSplitCost + std::max<int64_t>(2, (total + wgs - 1) / wgs);
  if (split_tokens == 0) {
    int64_t lo = budget, hi = budget + kSplitCost * (num_entries / wgs + 2) + 8;
    while (!fits(hi)) hi += hi / 2;
    while (lo < hi) {
      const int64_t mid = (lo + hi) / 2;
      if (fits(mid)) hi = mid;
      else lo = mid + 1;
    }
    budget = lo;
  }
  struct Piece {
    int32_t entry, begin, end;
    int64_t wg;
  };
  std::vector<Piece> v;
  int64_t w = 0, room = budget;
  cur = 0;
  seq_partial_start[0] = 0;
  for (int32_t i = 0; i < num_entries; ++i) {
    while (cur < entry_seq[i]) seq_partial_start[++cur] = static_cast<int32_t>(v.size());
    const int64_t len = entries[i].kv.len, c = chunks(i);
    if (split_tokens > 0) {
      // pieces of at most split_tokens keys, a workgroup each
      const int64_t np = (len + split_tokens - 1) / split_tokens;
      const int64_t st = np > 0 ? (len + np - 1) / np : 1;
      for (int64_t b = 0; b < len; b += st)
        v.push_back({i, static_cast<int32_t>(b), static_cast<int32_t>(std::min(len, b + st)), w++});
      continue;
    }
    for (int64_t at = 0; at < c;) {
      const int64_t t = take(c - at, room);
      if (t > 0) {
        v.push_back({i, static_cast<int32_t>(at * 32),
                     static_cast<int32_t>(std::min(len, (at + t) * 32)), w});
        at += t;
        room -= t + kSplitCost;
      }
      if (at < c) {
        room = budget;
        ++w;
      }
    }
  }
  while (cur < num_seqs) seq_partial_start[++cur] = static_cast<int32_t>(v.size());
  const int32_t n = static_cast<int32_t>(v.size());
  if (n > cap) return fail(HCP_EWORKSPACE, "%s: %d splits, cap %d", who, n, cap);
  // records: the first split of each workgroup in workgroup order, then the
  // others, each linked from the one before it
  int32_t heads = 0, more = 0;
  for (int32_t j = 0; j < n; ++j) heads += j == 0 || v[j].wg != v[j - 1].wg;
  int32_t h = 0, prev = -1;
  for (int32_t j = 0; j < n; ++j) {
    const Piece& x = v[j];
    const bool head = j == 0 || x.wg != v[j - 1].wg;
    const int32_t at = head ? h++ : heads + more++;
    hcp_decode_work& r = works[at];
    r = hcp_decode_work{};
    if (work_entry) work_entry[at] = x.entry;
    r.e = entries[x.entry];
    r.key_begin = x.begin;
    r.key_end = x.end;
    r.slot = j;
    r.next = -1;
    if (!head) works[prev].next = at;
    prev = at;
  }
  *num_wgs = heads;
  return n;
} catch (const std::bad_alloc&) {
  return fail(HCP_EINVAL, "hcp_plan_decode_lists: out of host memory");
}

size_t hcp_decode_workspace_bytes(int32_t num_splits, int32_t num_heads, int32_t head_dim) {
  if (num_splits <= 0 || num_heads <= 0 || head_dim <= 0) return 0;
  head_dim = hcp::padded_head_dim(head_dim);  // partials keep the kernel's width
  const size_t n = static_cast<size_t>(num_splits) * num_heads;
  const size_t o = n * head_dim * sizeof(float);
  const size_t o_al = (o + 255) & ~static_cast<size_t>(255);
  return o_al + n * sizeof(float);
}

// What hcp_decode_launch can say beyond the plain entry points.
struct DecodeExtra {
  const hcp_decode_work* works = nullptr;
  int32_t num_wgs = 0;
  const int32_t* rows = nullptr;
  uint64_t kv_base = 0;
  bool keep_nan = false;
};

static int decode_impl(const char* who, const void* q, int64_t q_stride_tok,
                       int64_t q_stride_head, const hcp_varlen_entry* entries,
                       int32_t num_entries, const hcp_decode_split* splits, int32_t num_splits,
                       const int32_t* seq_partial_start, int32_t num_seqs, void* workspace,
                       size_t workspace_bytes, void* out, int64_t o_stride_tok,
                       int64_t o_stride_head, float* lse, int64_t lse_stride_head,
                       const void* acc_o, int64_t acc_stride_tok, int64_t acc_stride_head,
                       const float* acc_lse, int64_t acc_lse_stride_head, int32_t num_heads,
                       int32_t num_kv_heads, int32_t head_dim, float scale, int32_t dtype,
                       void* stream, const DecodeExtra& x = DecodeExtra()) {
  int rc = check_heads(num_heads, num_kv_heads, head_dim, dtype, who);
  if (rc) return rc;
  if (num_entries < 0 || num_splits < 0 || num_seqs < 0)
    return fail(HCP_EINVAL, "%s: negative counts", who);
  if (num_seqs == 0) return HCP_OK;
  if (!q || !out || !seq_partial_start || (num_splits > 0 && !x.works && (!entries || !splits)))
    return fail(HCP_EINVAL, "%s: null pointer", who);
  if (!aligned16(q)) return fail(HCP_EINVAL, "%s: q not 16-byte aligned", who);
  if ((q_stride_tok | q_stride_head) % 8)
    return fail(HCP_EINVAL, "%s: q strides must be multiples of 8 elements", who);
  if (!(scale > 0.f) || !std::isfinite(scale))
    return fail(HCP_EINVAL, "%s: scale must be finite and > 0", who);
  const size_t need = hcp_decode_workspace_bytes(num_splits, num_heads, head_dim);
  if (num_splits > 0 && (!workspace || workspace_bytes < need))
    return fail(HCP_EWORKSPACE, "%s: workspace %zu bytes < %zu needed", who, workspace_bytes, need);
  if (workspace && !aligned16(workspace))
    return fail(HCP_EINVAL, "%s: workspace not 16-byte aligned", who);
  const size_t n = static_cast<size_t>(num_splits) * num_heads;
  const size_t o_al = (n * hcp::padded_head_dim(head_dim) * sizeof(float) + 255) &
                      ~static_cast<size_t>(255);
  hcp::DecParams dp{};
  dp.q = q;
  dp.q_stride_tok = q_stride_tok;
  dp.q_stride_head = q_stride_head;
  dp.entries = entries;
  dp.splits = splits;
  dp.num_splits = num_splits;
  dp.works = x.works;
  dp.num_wgs = x.works ? x.num_wgs : num_splits;
  dp.kv_base = x.kv_base;
  dp.keep_nan = x.keep_nan;
  dp.ws_o = static_cast<float*>(workspace);
  dp.ws_lse = reinterpret_cast<float*>(static_cast<char*>(workspace) + o_al);
  dp.num_heads = num_heads;
  dp.num_kv_heads = num_kv_heads;
  dp.group = num_heads / num_kv_heads;
  dp.head_chunks = (dp.group + 15) / 16;
  dp.head_dim = head_dim;
  dp.scale_log2 = scale * hcp::kLog2e;
  hcp::RedParams rp{};
  rp.ws_o = dp.ws_o;
  rp.ws_lse = dp.ws_lse;
  rp.seq_partial_start = seq_partial_start;
  rp.rows = x.rows;
  rp.num_seqs = num_seqs;
  rp.out = out;
  rp.o_stride_tok = o_stride_tok;
  rp.o_stride_head = o_stride_head;
  rp.lse = lse;
  rp.lse_stride_head = lse_stride_head;
  rp.num_heads = num_heads;
  rp.head_dim = head_dim;
  rp.acc_o = acc_o;
  rp.acc_stride_tok = acc_stride_tok;
  rp.acc_stride_head = acc_stride_head;
  rp.acc_lse = acc_lse;
  rp.acc_lse_stride_head = acc_lse_stride_head;
  hipError_t e = hcp::launch_decode(dp, rp, head_dim, dtype, static_cast<hipStream_t>(stream));
  return launch_status(e, who);
}

int hcp_decode_splitkv(const void* q, int64_t q_stride_tok, int64_t q_stride_head,
                       const hcp_varlen_entry* entries, int32_t num_entries,
                       const hcp_decode_split* splits, int32_t num_splits,
                       const int32_t* seq_partial_start, int32_t num_seqs, void* workspace,
                       size_t workspace_bytes, void* out, int64_t o_stride_tok,
                       int64_t o_stride_head, float* lse, int64_t lse_stride_head,
                       int32_t num_heads, int32_t num_kv_heads, int32_t head_dim, float scale,
                       int32_t dtype, void* stream) {
  return decode_impl("hcp_decode_splitkv", q, q_stride_tok, q_stride_head, entries,
                     num_entries, splits, num_splits, seq_partial_start, num_seqs, workspace,
                     workspace_bytes, out, o_stride_tok, o_stride_head, lse, lse_stride_head,
                     nullptr, 0, 0, nullptr, 0, num_heads, num_kv_heads, head_dim, scale,
                     dtype, stream);
}

int hcp_decode_splitkv_acc(const void* q, int64_t q_stride_tok, int64_t q_stride_head,
                           const hcp_varlen_entry* entries, int32_t num_entries,
                           const hcp_decode_split* splits, int32_t num_splits,
                           const int32_t* seq_partial_start, int32_t num_seqs,
                           void* workspace, size_t workspace_bytes, const void* acc_o,
                           int64_t acc_stride_tok, int64_t acc_stride_head,
                           const float* acc_lse, int64_t acc_lse_stride_head, void* out,
                           int64_t o_stride_tok, int64_t o_stride_head, float* lse,
                           int64_t lse_stride_head, int32_t num_heads, int32_t num_kv_heads,
                           int32_t head_dim, float scale, int32_t dtype, void* stream) {
  const char* who = "hcp_decode_splitkv_acc";
  if (!acc_o || !acc_lse) return fail(HCP_EINVAL, "%s: null accumulator", who);
  if (reinterpret_cast<uintptr_t>(acc_o) % 2)
    return fail(HCP_EINVAL, "%s: acc_o not 2-byte aligned", who);
  return decode_impl(who, q, q_stride_tok, q_stride_head, entries, num_entries, splits,
                     num_splits, seq_partial_start, num_seqs, workspace, workspace_bytes, out,
                     o_stride_tok, o_stride_head, lse, lse_stride_head, acc_o, acc_stride_tok,
                     acc_stride_head, acc_lse, acc_lse_stride_head, num_heads, num_kv_heads,
                     head_dim, scale, dtype, stream);
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Allocation-free decode: the split partials live in this file-scope device
// array instead of a caller workspace.  In host code `scratch` names a
// host-side stand-in, not device memory: its per-device address comes from
// hipGetSymbolAddress (once per device, with that device current) and only
// that address is ever passed to a kernel.
// ---------------------------------------------------------------------------
static __device__ __align__(256) char scratch[HCP_NOALLOC_SCRATCH_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device (resolved on the first
// call there).
int scratch_on_current_device(void** out, const char* who) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(HCP_ELAUNCH, "%s: hipGetDevice: %s", who, hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices)
    return fail(HCP_EUNSUPPORTED, "%s: device index %d beyond %d", who, dev, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(HCP_ELAUNCH, "%s: hipGetSymbolAddress(scratch) on device %d: %s", who, dev,
                  hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return HCP_OK;
}

}  // namespace

extern "C" {

int hcp_decode_splitkv_noalloc(const void* q, int64_t q_stride_tok, int64_t q_stride_head,
                               const hcp_varlen_entry* entries, int32_t num_entries,
                               const hcp_decode_split* splits, int32_t num_splits,
                               const int32_t* seq_partial_start, int32_t num_seqs, void* out,
                               int64_t o_stride_tok, int64_t o_stride_head, float* lse,
                               int64_t lse_stride_head, int32_t num_heads, int32_t num_kv_heads,
                               int32_t head_dim, float scale, int32_t dtype, void* stream) {
  const char* who = "hcp_decode_splitkv_noalloc";
  int rc = check_heads(num_heads, num_kv_heads, head_dim, dtype, who);
  if (rc) return rc;
  if (num_splits < 0 || num_seqs < 0) return fail(HCP_EINVAL, "%s: negative counts", who);
  const size_t need = hcp_decode_workspace_bytes(num_splits, num_heads, head_dim);
  if (need > HCP_NOALLOC_SCRATCH_BYTES)
    return fail(HCP_EWORKSPACE,
                "%s: %d splits x %d heads x head_dim %d need %zu bytes of partials; the "
                "library's fixed scratch holds %zu (use hcp_decode_splitkv with a workspace, "
                "or plan fewer splits)",
                who, num_splits, num_heads, head_dim, need,
                static_cast<size_t>(HCP_NOALLOC_SCRATCH_BYTES));
  void* ws = nullptr;
  if (num_splits > 0 && num_seqs > 0 && (rc = scratch_on_current_device(&ws, who))) return rc;
  return decode_impl(who, q, q_stride_tok, q_stride_head, entries, num_entries, splits,
                     num_splits, seq_partial_start, num_seqs, ws, HCP_NOALLOC_SCRATCH_BYTES, out,
                     o_stride_tok, o_stride_head, lse, lse_stride_head, nullptr, 0, 0, nullptr,
                     0, num_heads, num_kv_heads, head_dim, scale, dtype, stream);
}

int hcp_decode_launch(const hcp_decode_args* a, void* stream) {
  const char* who = "hcp_decode_launch";
  if (!a) return fail(HCP_EINVAL, "%s: null arguments", who);
  if (a->num_works < 0 || a->num_wgs < 0 || a->num_wgs > a->num_works ||
      (a->num_works > 0 && (!a->works || a->num_wgs == 0)))
    return fail(HCP_EINVAL, "%s: bad work list", who);
  if (a->kv_base & 15) return fail(HCP_EINVAL, "%s: kv_base not 16-byte aligned", who);
  if ((a->acc_o == nullptr) != (a->acc_lse == nullptr))
    return fail(HCP_EINVAL, "%s: half an accumulator", who);
  if (reinterpret_cast<uintptr_t>(a->acc_o) % 2)
    return fail(HCP_EINVAL, "%s: acc_o not 2-byte aligned", who);
  int rc = check_heads(a->num_heads, a->num_kv_heads, a->head_dim, a->dtype, who);
  if (rc) return rc;
  void* ws = a->workspace;
  size_t bytes = a->workspace_bytes;
  if (a->use_scratch) {
    bytes = HCP_NOALLOC_SCRATCH_BYTES;
    const size_t need = hcp_decode_workspace_bytes(a->num_works, a->num_heads, a->head_dim);
    if (need > bytes)
      return fail(HCP_EWORKSPACE, "%s: %d splits x %d heads x head_dim %d need %zu bytes of "
                  "partials; the library's fixed scratch holds %zu",
                  who, a->num_works, a->num_heads, a->head_dim, need, bytes);
    if (a->num_works > 0 && a->num_seqs > 0 && (rc = scratch_on_current_device(&ws, who)))
      return rc;
  }
  DecodeExtra x;
  x.works = a->works;
  x.num_wgs = a->num_wgs;
  x.rows = a->seq_rows;
  x.kv_base = a->kv_base;
  x.keep_nan = a->keep_nan != 0;
  return decode_impl(who, a->q, a->q_stride_tok, a->q_stride_head, nullptr, 0, nullptr,
                     a->num_works, a->seq_partial_start, a->num_seqs, ws, bytes, a->out,
                     a->o_stride_tok, a->o_stride_head, a->lse, a->lse_stride_head, a->acc_o,
                     a->acc_stride_tok, a->acc_stride_head, a->acc_lse, a->acc_lse_stride_head,
                     a->num_heads, a->num_kv_heads, a->head_dim, a->scale, a->dtype, stream, x);
}

// Workgroups per KV head and head chunk of hcp_decode_paged: one round of the
// machine (a workgroup's chunk buffers take 128 KB of a CU's LDS).
static int32_t paged_wgs(int32_t num_heads, int32_t num_kv_heads) {
  const int32_t chunks = (num_heads / num_kv_heads + 15) / 16;
  return std::max(1, kNumCus / (num_kv_heads * chunks));
}

size_t hcp_decode_paged_workspace(int32_t num_seqs, int32_t num_heads, int32_t num_kv_heads,
                                  int32_t head_dim) {
  if (num_seqs <= 0 || num_heads <= 0 || num_kv_heads <= 0 || num_heads % num_kv_heads ||
      head_dim <= 0)
    return 0;
  const size_t parts =
      hcp_decode_workspace_bytes(num_seqs + paged_wgs(num_heads, num_kv_heads), num_heads, head_dim);
  return ((parts + 15) & ~static_cast<size_t>(15)) + 2 * sizeof(int32_t) * num_seqs;
}

int hcp_decode_paged(const hcp_decode_paged_args* a, void* stream) {
  const char* who = "hcp_decode_paged";
  if (!a) return fail(HCP_EINVAL, "%s: null arguments", who);
  int rc = check_heads(a->num_heads, a->num_kv_heads, a->head_dim, a->dtype, who);
  if (rc) return rc;
  if (a->num_seqs < 0 || a->window < 0 || a->block_table_width <= 0)
    return fail(HCP_EINVAL, "%s: bad sizes", who);
  if (a->num_seqs > HCP_DECODE_PAGED_MAX_SEQS)
    return fail(HCP_EUNSUPPORTED, "%s: more than %d sequences", who, HCP_DECODE_PAGED_MAX_SEQS);
  if (a->num_seqs == 0) return HCP_OK;
  if (!a->q || !a->out || !a->seq_lens || !a->kv.block_table)
    return fail(HCP_EINVAL, "%s: null pointer", who);
  if (a->lens_dtype != HCP_DTYPE_I32 && a->lens_dtype != HCP_DTYPE_I64)
    return fail(HCP_EUNSUPPORTED, "%s: seq_lens dtype %d (int32 or int64)", who, a->lens_dtype);
  if (!aligned16(a->q) || (a->q_stride_tok | a->q_stride_head) % 8)
    return fail(HCP_EINVAL, "%s: q not in 16-byte rows", who);
  if (!(a->scale > 0.f) || !std::isfinite(a->scale))
    return fail(HCP_EINVAL, "%s: scale must be finite and > 0", who);
  hcp_kv_segment kv = a->kv;
  kv.start = 0;
  kv.len = 1;
  if ((rc = check_segment(kv, a->head_dim, who, 0))) return rc;
  // the kernel sums chunks of 32 keys in 32 bits
  if (a->block_table_width > ((int64_t{1} << 34) / kv.block_size) / a->num_seqs ||
      a->block_table_width * kv.block_size > INT32_MAX)
    return fail(HCP_EUNSUPPORTED, "%s: block table names too many keys", who);
  const size_t need =
      hcp_decode_paged_workspace(a->num_seqs, a->num_heads, a->num_kv_heads, a->head_dim);
  if (!a->workspace || a->workspace_bytes < need)
    return fail(HCP_EWORKSPACE, "%s: workspace %zu bytes < %zu needed", who,
                static_cast<size_t>(a->workspace_bytes), need);
  if (!aligned16(a->workspace)) return fail(HCP_EINVAL, "%s: workspace not 16-byte aligned", who);
  hcp::PagedDecParams p{};
  hcp::DecParams& dp = p.d;
  dp.q = a->q;
  dp.q_stride_tok = a->q_stride_tok;
  dp.q_stride_head = a->q_stride_head;
  dp.num_wgs = paged_wgs(a->num_heads, a->num_kv_heads);
  const size_t slots = static_cast<size_t>(a->num_seqs + dp.num_wgs) * a->num_heads;
  const size_t o_al = (slots * hcp::padded_head_dim(a->head_dim) * sizeof(float) + 255) &
                      ~static_cast<size_t>(255);
  char* const ws = static_cast<char*>(a->workspace);
  dp.ws_o = reinterpret_cast<float*>(ws);
  dp.ws_lse = reinterpret_cast<float*>(ws + o_al);
  dp.num_heads = a->num_heads;
  dp.num_kv_heads = a->num_kv_heads;
  dp.group = a->num_heads / a->num_kv_heads;
  dp.head_chunks = (dp.group + 15) / 16;
  dp.head_dim = a->head_dim;
  dp.scale_log2 = a->scale * hcp::kLog2e;
  dp.keep_nan = a->keep_nan != 0;
  p.kv = kv;
  p.lens = a->seq_lens;
  p.lens_wide = a->lens_dtype == HCP_DTYPE_I64;
  p.num_seqs = a->num_seqs;
  p.bt_stride = a->block_table_stride;
  p.max_len = a->block_table_width * kv.block_size;
  p.window = a->window;
  p.seq_slots = reinterpret_cast<int32_t*>(ws + need - 2 * sizeof(int32_t) * a->num_seqs);
  hcp::RedParams rp{};
  rp.ws_o = dp.ws_o;
  rp.ws_lse = dp.ws_lse;
  rp.seq_slots = p.seq_slots;
  rp.num_slots = a->num_seqs + dp.num_wgs;
  rp.num_seqs = a->num_seqs;
  rp.out = a->out;
  rp.o_stride_tok = a->o_stride_tok;
  rp.o_stride_head = a->o_stride_head;
  rp.lse = a->lse;
  rp.lse_stride_head = a->lse_stride_head;
  rp.num_heads = a->num_heads;
  rp.head_dim = a->head_dim;
  return launch_status(hcp::launch_decode_paged(p, rp, a->head_dim, a->dtype,
                                                static_cast<hipStream_t>(stream)),
                       who);
}

int hcp_merge_attn_states(void* out, int64_t o_stride_tok, int64_t o_stride_head,
                          int32_t out_dtype, float* out_lse, int64_t out_lse_stride_head,
                          const void* prefix_out, int64_t p_stride_tok, int64_t p_stride_head,
                          int32_t prefix_dtype, const float* prefix_lse,
                          int64_t p_lse_stride_head, const void* suffix_out,
                          int64_t s_stride_tok, int64_t s_stride_head, int32_t suffix_dtype,
                          const float* suffix_lse, int64_t s_lse_stride_head,
                          int64_t num_tokens, int32_t num_heads, int32_t head_dim,
                          void* stream) {
  const char* who = "hcp_merge_attn_states";
  if (num_tokens < 0 || num_heads <= 0 || head_dim <= 0)
    return fail(HCP_EINVAL, "%s: bad sizes", who);
  if (head_dim % 8) return fail(HCP_EUNSUPPORTED, "%s: head_dim must be a multiple of 8", who);
  for (int32_t d : {out_dtype, prefix_dtype, suffix_dtype})
    if (d != HCP_DTYPE_F16 && d != HCP_DTYPE_BF16 && d != HCP_DTYPE_F32)
      return fail(HCP_EUNSUPPORTED, "%s: dtype %d not supported", who, d);
  if (num_tokens == 0) return HCP_OK;
  if (!out || !prefix_out || !suffix_out || !prefix_lse || !suffix_lse)
    return fail(HCP_EINVAL, "%s: null pointer", who);
  if (!aligned16(out) || !aligned16(prefix_out) || !aligned16(suffix_out))
    return fail(HCP_EINVAL, "%s: o tensors must be 16-byte aligned", who);
  if ((o_stride_tok | o_stride_head | p_stride_tok | p_stride_head | s_stride_tok |
       s_stride_head) % 8)
    return fail(HCP_EINVAL, "%s: strides must be multiples of 8 elements", who);
  if (num_tokens * num_heads * (head_dim / 8) > (int64_t)INT32_MAX * 256)
    return fail(HCP_EINVAL, "%s: too large", who);
  hcp::MergeParams p{};
  p.out = out;
  p.o_stride_tok = o_stride_tok;
  p.o_stride_head = o_stride_head;
  p.out_lse = out_lse;
  p.out_lse_stride = out_lse_stride_head;
  p.po = prefix_out;
  p.p_stride_tok = p_stride_tok;
  p.p_stride_head = p_stride_head;
  p.plse = prefix_lse;
  p.p_lse_stride = p_lse_stride_head;
  p.so = suffix_out;
  p.s_stride_tok = s_stride_tok;
  p.s_stride_head = s_stride_head;
  p.slse = suffix_lse;
  p.s_lse_stride = s_lse_stride_head;
  p.num_tokens = num_tokens;
  p.num_heads = num_heads;
  p.head_dim = head_dim;
  p.out_dtype = out_dtype;
  p.p_dtype = prefix_dtype;
  p.s_dtype = suffix_dtype;
  return launch_status(hcp::launch_merge(p, static_cast<hipStream_t>(stream)), who);
}

int hcp_reshape_and_cache(const void* key, int64_t k_stride_tok, int64_t k_stride_head,
                          const void* value, int64_t v_stride_tok, int64_t v_stride_head,
                          const void* slot_mapping, int32_t slot_dtype, int64_t num_tokens,
                          int32_t num_kv_heads, int32_t head_dim, const hcp_paged_cache* cache,
                          int32_t dtype, void* stream) {
  const char* who = "hcp_reshape_and_cache";
  if (num_tokens < 0 || num_kv_heads <= 0 || head_dim <= 0)
    return fail(HCP_EINVAL, "%s: bad sizes", who);
  if (head_dim % 8)
    return fail(HCP_EUNSUPPORTED, "%s: head_dim %d must be a multiple of 8", who, head_dim);
  if (!dtype16(dtype)) return fail(HCP_EUNSUPPORTED, "%s: dtype %d not supported", who, dtype);
  if (slot_dtype != HCP_DTYPE_I32 && slot_dtype != HCP_DTYPE_I64)
    return fail(HCP_EUNSUPPORTED, "%s: slot dtype %d (int32 or int64)", who, slot_dtype);
  if (!cache) return fail(HCP_EINVAL, "%s: null cache descriptor", who);
  const hcp_paged_cache& c = *cache;
  if (c.block_size <= 0 || (c.block_size & (c.block_size - 1)))
    return fail(HCP_EINVAL, "%s: block_size %d not a power of two", who, c.block_size);
  if (c.num_blocks < 0) return fail(HCP_EINVAL, "%s: negative num_blocks", who);
  if (num_tokens == 0 || c.num_blocks == 0) return HCP_OK;
  if (!key || !value || !slot_mapping || !c.k_addr || !c.v_addr)
    return fail(HCP_EINVAL, "%s: null pointer", who);
  if (!aligned16(key) || !aligned16(value) || (c.k_addr & 15) || (c.v_addr & 15))
    return fail(HCP_EINVAL, "%s: key/value/cache must be 16-byte aligned", who);
  if ((k_stride_tok | k_stride_head | v_stride_tok | v_stride_head | c.stride_block |
       c.stride_head | c.stride_tok) % 8)
    return fail(HCP_EINVAL, "%s: strides must be multiples of 8 elements", who);
  if (num_tokens * num_kv_heads > (int64_t)INT32_MAX * 16)
    return fail(HCP_EINVAL, "%s: too many rows", who);
  hcp::CacheParams p{};
  p.key = key;
  p.k_stride_tok = k_stride_tok;
  p.k_stride_head = k_stride_head;
  p.value = value;
  p.v_stride_tok = v_stride_tok;
  p.v_stride_head = v_stride_head;
  p.slots = slot_mapping;
  p.num_tokens = num_tokens;
  p.num_kv_heads = num_kv_heads;
  p.cpr = head_dim / 8;
  p.cpr_shift = (p.cpr & (p.cpr - 1)) ? -1 : 31 - __builtin_clz(static_cast<unsigned>(p.cpr));
  p.k_cache = reinterpret_cast<void*>(c.k_addr);
  p.v_cache = reinterpret_cast<void*>(c.v_addr);
  p.stride_block = c.stride_block;
  p.stride_head = c.stride_head;
  p.stride_tok = c.stride_tok;
  p.num_slots = c.num_blocks * c.block_size;
  p.bs_shift = 31 - __builtin_clz(static_cast<unsigned>(c.block_size));
  p.bs_mask = c.block_size - 1;
  (void)dtype;  // a 16-bit copy: the bytes are moved as they are
  return launch_status(hcp::launch_cache_write(p, slot_dtype == HCP_DTYPE_I64,
                                               static_cast<hipStream_t>(stream)),
                       who);
}

int hcp_fetch_metadata(const void* query_start_loc, int32_t qsl_dtype, int64_t qsl_stride,
                       const void* seq_lens, int32_t lens_dtype, int64_t lens_stride,
                       const void* block_table, int32_t bt_dtype, int64_t bt_stride, int32_t n,
                       int64_t max_len, int64_t* dev_out, int64_t token, int64_t* host_out,
                       void* stream) {
  const char* who = "hcp_fetch_metadata";
  for (int32_t d : {qsl_dtype, lens_dtype, bt_dtype})
    if (d != HCP_DTYPE_I32 && d != HCP_DTYPE_I64)
      return fail(HCP_EUNSUPPORTED, "%s: index dtype %d (int32 or int64)", who, d);
  if (n < 0) return fail(HCP_EINVAL, "%s: negative n", who);
  if (!query_start_loc || !host_out || (n > 0 && !seq_lens))
    return fail(HCP_EINVAL, "%s: null pointer", who);
  hcp::MetaParams p{};
  p.qsl = query_start_loc;
  p.lens = seq_lens;
  p.bt = block_table;
  p.qsl_stride = qsl_stride;
  p.lens_stride = lens_stride;
  p.bt_stride = bt_stride;
  p.qsl_wide = qsl_dtype == HCP_DTYPE_I64;
  p.lens_wide = lens_dtype == HCP_DTYPE_I64;
  p.bt_wide = bt_dtype == HCP_DTYPE_I64;
  p.n = n;
  p.token = token;
  p.out = host_out;
  p.max_len = max_len;
  p.dev = dev_out;
  return launch_status(hcp::launch_fetch_metadata(p, static_cast<hipStream_t>(stream)), who);
}

int hcp_wait_metadata(const int64_t* host_out, int64_t token, void* stream) {
  const char* who = "hcp_wait_metadata";
  if (!host_out) return fail(HCP_EINVAL, "%s: null pointer", who);
  const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(50);
  for (int i = 0;; ++i) {
    if (__atomic_load_n(host_out, __ATOMIC_ACQUIRE) == token) return HCP_OK;
    if ((i & 1023) == 1023 && std::chrono::steady_clock::now() > until) break;
  }
  // a long queue ahead of the copy, or an error: wait for the stream itself
  const hipError_t e = hipStreamSynchronize(static_cast<hipStream_t>(stream));
  if (e != hipSuccess) return launch_status(e, who);
  if (__atomic_load_n(host_out, __ATOMIC_ACQUIRE) != token)
    return fail(HCP_ELAUNCH, "%s: the copy did not arrive", who);
  return HCP_OK;
}

int hcp_gather_paged_kv(const hcp_varlen_entry* entries, int32_t num_entries,
                        const int64_t* out_start, int64_t max_len, int32_t num_kv_heads,
                        int32_t head_dim, int32_t dtype, void* k_out, void* v_out,
                        void* stream) {
  const char* who = "hcp_gather_paged_kv";
  if (num_entries < 0 || max_len < 0 || num_kv_heads <= 0 || head_dim <= 0)
    return fail(HCP_EINVAL, "%s: bad sizes", who);
  if (head_dim % 8 || head_dim > 256)
    return fail(HCP_EUNSUPPORTED, "%s: head_dim %d not supported (a multiple of 8 up to 256)",
                who, head_dim);
  if (!dtype16(dtype)) return fail(HCP_EUNSUPPORTED, "%s: dtype %d not supported", who, dtype);
  if (num_entries > 65535) return fail(HCP_EINVAL, "%s: more than 65535 entries", who);
  if (num_entries == 0 || max_len == 0) return HCP_OK;
  if (!entries || !out_start || !k_out || !v_out) return fail(HCP_EINVAL, "%s: null pointer", who);
  if (!aligned8(entries) || !aligned8(out_start) || !aligned16(k_out) || !aligned16(v_out))
    return fail(HCP_EINVAL, "%s: misaligned pointer", who);
  // one thread per 16-byte piece of a (token, head) row, 256 per workgroup:
  // the launch's grid.x (and grid.x * 256) must stay within 32 bits
  if (max_len * num_kv_heads * (head_dim / 8) > (int64_t{1} << 32) - 256)
    return fail(HCP_EINVAL, "%s: too many rows (max_len * num_kv_heads * head_dim / 8 >= 2^32)",
                who);
  hcp::GatherParams p{};
  p.entries = entries;
  p.out_start = out_start;
  p.max_len = max_len;
  p.num_entries = num_entries;
  p.num_kv_heads = num_kv_heads;
  p.cpr = head_dim / 8;
  p.cpr_shift = (p.cpr & (p.cpr - 1)) ? -1 : 31 - __builtin_clz(static_cast<unsigned>(p.cpr));
  p.head_dim = head_dim;
  p.k_out = k_out;
  p.v_out = v_out;
  (void)dtype;  // a 16-bit copy: the bytes are moved as they are
  return launch_status(hcp::launch_gather(p, static_cast<hipStream_t>(stream)), who);
}

}  // extern "C"
