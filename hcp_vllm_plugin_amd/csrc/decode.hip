// Split-KV decode for gfx950: one query token per sequence, long KV segments.
//
// The reference decodes with the prefill kernel, grid (H, 1) per request and
// segment (ring_triton_attn.py:179, ring_backend.py:672,820-830): 28
// workgroups on a 256-CU part, 63 of 64 query rows padding, and every query
// head of a GQA group re-reading the same K/V.  Here:
//
//  * kernel 1 (decode_split_kernel): one workgroup per (split, KV head,
//    head chunk).  A split is a key range of one segment (contiguous peer or
//    paged local; the form is per entry, so one launch serves both).  Up to 16
//    query heads of the KV head are the 16 columns of v_mfma_f32_16x16x32, so
//    with G <= 16 each K/V byte is read from HBM once; a larger group runs in
//    ceil(G / 16) chunks of 16 heads, dispatched next to each other so the
//    chunks after the first mostly read the split's K/V from L2.  Each of the 4 waves walks its
//    own 32-key chunks straight from global memory into MFMA operands (no LDS,
//    no barrier in the loop); the next chunk's loads are in flight while the
//    current one is computed.
//      S^T = K Q^T   A = K rows (one key per lane row), B = Q^T; k-step s
//                    covers d = 32s .. 32s+31, so each K load instruction
//                    reads one contiguous 64 B piece of 16 key rows
//      O^T = V^T P^T A = V^T, B = P^T taken from the S^T registers.
//    For V^T each lane loads 8 keys x 8 contiguous d (16 B per key, whole
//    256 B rows per load instruction) and transposes the 8x8 block in
//    registers; MFMA number u then covers d = 8*row + u.  The 4 waves'
//    (m, l, O) are combined through LDS and one fp32 partial (O normalised,
//    LSE natural log) per (split, head) goes to the workspace.
//  * kernel 2 (decode_reduce_kernel): per (sequence, head) merges all
//    partials of the sequence -- every split of its local and peer segments --
//    with the LSE merge of ring_decode.py:46-61, writing out in the model
//    dtype and optionally the merged LSE.
#include "params.h"

namespace hcp {

constexpr int kDecThreads = 256;
constexpr int kDecChunk = 32;  // keys per wave step
// raw buffer descriptor word 3 (32-bit data format, bounds-checked)
constexpr int kBufWord3 = 0x00020000;
// cache policy of the K/V stream: non-temporal (read once per launch)
constexpr int kStreamAux = 2;
#define HCP_LDS_PTR(T) __attribute__((address_space(3))) T*


// LDS of the split kernel, shared by its paged and contiguous instantiations.
// Each wave double-buffers its chunks' K and V rows; D = 256 runs two waves
// per workgroup so the buffers stay within 128 KB.
template <int D>
struct DecShared {
  static constexpr int CHB = kDecChunk * D * 2;  // bytes of a chunk's K (or V) rows
  static constexpr int W = D == 256 ? 2 : 4;     // waves per workgroup
};

// KEEP_NAN: scores that hold a NaN make their row NaN, as in the prefill
// kernels; without it their split is left out.  (A parameter read where the
// partial is stored costs every split 0.1 to 0.3 us.)
template <int D, typename T, bool PAGED, bool KEEP_NAN>
__device__ __forceinline__ void decode_split_body(const DecParams& p, int kvh_in, int chunk_in,
                                                  int sp, const hcp_varlen_entry& e,
                                                  int64_t kb, int64_t ke,
                                                  char (*bufE)[2 * DecShared<D>::CHB],
                                                  char (*bufO)[2 * DecShared<D>::CHB],
                                                  float (*sm_m)[16], float (*sm_l)[16]) {
  using E = Elem<T>;
  using V8 = typename E::vec8;
  constexpr int QSTEPS = D / 32;         // 16x16x32 k-steps over d
  constexpr int NU = D / 16;             // PV MFMAs (d = NU*row + u)
  constexpr int ROWB = D * 2;            // bytes of one key row of one head
  constexpr int CPR = ROWB / 16;         // 16-byte slots per row
  constexpr int CHB = kDecChunk * ROWB;  // bytes of the K (or V) rows of a chunk
  constexpr int NLD = CHB / 1024;        // LDS-DMA instructions per K (or V) chunk
  constexpr int KPI = 1024 / ROWB;       // key rows per DMA instruction
  static_assert(D == 64 || D == 128 || D == 256, "head_dim");
  constexpr int W = DecShared<D>::W;  // waves per workgroup

  // Wave-private chunk buffers [K rows | V rows] (bufE / bufO: even / odd
  // chunks of the wave, distinct objects so the compiler can tell reads of
  // one from the DMA writes into the other).  Row r's 16-byte slot c sits at
  // slot c ^ (r % CPR): both operand reads below are then conflict-free.

  // (opaque: what is derived from it is rebuilt for every split, not held in
  // registers across the workgroup's list)
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform
  const int c16 = lane & 15;
  const int g4 = lane >> 4;
  // the KV head and head chunk are workgroup-uniform: keep every address
  // built from them in SGPRs (buffer descriptors from VGPR values become
  // waterfall loops).  This workgroup's query heads: h0 .. h0 + G - 1.
  const int kvh = __builtin_amdgcn_readfirstlane(kvh_in);
  const int chunk = __builtin_amdgcn_readfirstlane(chunk_in);
  const int G = p.group - 16 * chunk < 16 ? p.group - 16 * chunk : 16;
  const int h0 = kvh * p.group + 16 * chunk;
  KvAddr kva;
  kva.init(e.kv);

  // A row holds dv <= D valid elements (a multiple of 8): the kernel computes
  // in D columns.  Q's tail is zero; a K/V chunk past dv is fetched from the
  // row's first chunk instead (finite values that meet Q's zero columns, or
  // land in output columns that are never stored), so no load leaves the row.
  const int dv = p.head_dim;
  const int cv = dv / 8;  // valid 16-byte chunks of a row
  // Q^T (B operand): column c16 = query head h0 + c16 (zero for c16 >= G);
  // k-step s covers d = 32s .. 32s+31 (lane group g4: 8 of them)
  V8 qf[QSTEPS];
  {
    const bool hv = c16 < G;
    const char* qrow = reinterpret_cast<const char*>(p.q) +
                       (e.q_start * p.q_stride_tok +
                        static_cast<int64_t>(h0 + (hv ? c16 : 0)) * p.q_stride_head) * 2;
#pragma unroll
    for (int s = 0; s < QSTEPS; ++s) {
      u32x4 x = hv && 32 * s + 8 * g4 < dv ? ldg16(qrow + (32 * s + 8 * g4) * 2)
                                           : u32x4{0, 0, 0, 0};
      qf[s] = as_vec8<V8>(x);
    }
  }

  const float c = p.scale_log2;
  float m_run = -INFINITY, l_run = 0.f;
  f32x4 oacc[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) oacc[u] = f32x4{};

  // ---- HBM -> LDS: one chunk (32 keys) of K and V rows ----
  // DMA instruction j writes rows j*KPI .. j*KPI+KPI-1; lane -> (row kr, slot
  // sl), fetching the row's 16-byte piece (sl ^ row % CPR): every
  // instruction reads KPI whole rows (1 KB), streamed past the caches.
  const int kr = lane / CPR, sl = lane % CPR;
  const int64_t rowb_g = kva.stride_tok * 2;
  // (contiguous segments; paged ones are issued by the loop further down)
  auto issue = [&](int64_t k0, HCP_LDS_PTR(char) dst) __attribute__((always_inline)) {
    if constexpr (!PAGED) {
      const int64_t rows = ke - k0;  // >= 1 valid rows in this chunk
      const int nrec = rows >= kDecChunk ? 0x7fffffff
                                         : static_cast<int>((rows - 1) * rowb_g) + 2 * dv;
      const int64_t base = ((kva.start + k0) * kva.stride_tok +
                            static_cast<int64_t>(kvh) * kva.stride_head) * 2;
      const __amdgpu_buffer_rsrc_t rk =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(kva.k + base), 0, nrec, kBufWord3);
      const __amdgpu_buffer_rsrc_t rv =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(kva.v + base), 0, nrec, kBufWord3);
#pragma unroll
      for (int j = 0; j < NLD; ++j) {
        const int row = j * KPI + kr;
        int ch = sl ^ (row % CPR);
        ch = ch < cv ? ch : 0;
        const int off = static_cast<int>(row * rowb_g) + 16 * ch;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rk, reinterpret_cast<HCP_LDS_PTR(void)>(dst + j * 1024), 16, off, 0, 0, kStreamAux);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rv, reinterpret_cast<HCP_LDS_PTR(void)>(dst + CHB + j * 1024), 16, off, 0, 0,
            kStreamAux);
      }
    }
  };

  // ---- one chunk from LDS: S^T = K Q^T, online softmax, O^T += V^T P^T ----
  auto compute = [&](int64_t k0, const HCP_LDS_PTR(char) src) __attribute__((always_inline)) {
    // K rows 16b + c16, d = 32s + 8g4 .. +7: slot (4s + g4) of that row
    f32x4 s0 = f32x4{}, s1 = f32x4{};
#pragma unroll
    for (int s = 0; s < QSTEPS; ++s) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int row = 16 * b + c16;
        const u32x4 kx = *reinterpret_cast<const HCP_LDS_PTR(u32x4)>(
            src + row * ROWB + 16 * ((4 * s + g4) ^ (row % CPR)));
        if (b == 0)
          s0 = E::mfma16(as_vec8<V8>(kx), qf[s], s0);
        else
          s1 = E::mfma16(as_vec8<V8>(kx), qf[s], s1);
      }
    }
    // V rows 16(j>>2) + 4g4 + (j&3), d = NU*c16 .. +NU-1 (NU/2 words)
    constexpr int VW = NU / 2 < 4 ? 4 : NU / 2;
    typedef uint32_t vwords __attribute__((ext_vector_type(VW)));
    vwords vc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int row = 16 * (j >> 2) + 4 * g4 + (j & 3);
      const HCP_LDS_PTR(char) vrow = src + CHB + row * ROWB;
      if constexpr (NU == 16) {
        const u32x4 x0 = *reinterpret_cast<const HCP_LDS_PTR(u32x4)>(
            vrow + 16 * ((2 * c16) ^ (row % CPR)));
        const u32x4 x1 = *reinterpret_cast<const HCP_LDS_PTR(u32x4)>(
            vrow + 16 * ((2 * c16 + 1) ^ (row % CPR)));
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          vc[j][w] = x0[w];
          vc[j][4 + w] = x1[w];
        }
      } else if constexpr (NU == 8) {
        const u32x4 x = *reinterpret_cast<const HCP_LDS_PTR(u32x4)>(vrow + 16 * (c16 ^ (row % CPR)));
#pragma unroll
        for (int w = 0; w < 4; ++w) vc[j][w] = x[w];
      } else {
        const u32x2 x = *reinterpret_cast<const HCP_LDS_PTR(u32x2)>(
            vrow + 16 * ((c16 >> 1) ^ (row % CPR)) + 8 * (c16 & 1));
        vc[j][0] = x[0];
        vc[j][1] = x[1];
        vc[j][2] = 0;
        vc[j][3] = 0;
      }
    }
    if (k0 + kDecChunk > ke) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (k0 + 4 * g4 + r >= ke) s0[r] = -INFINITY;
        if (k0 + 16 + 4 * g4 + r >= ke) s1[r] = -INFINITY;
      }
    }
    float mx = fmaxf(fmaxf(fmaxf(s0[0], s0[1]), fmaxf(s0[2], s0[3])),
                     fmaxf(fmaxf(s1[0], s1[1]), fmaxf(s1[2], s1[3])));
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float m_new = fmaxf(m_run, mx * c);
    const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
    const float alpha = fast_exp2(m_run - m_use);
    float rs = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      s0[r] = fast_exp2(__builtin_fmaf(s0[r], c, -m_use));
      s1[r] = fast_exp2(__builtin_fmaf(s1[r], c, -m_use));
      rs += s0[r] + s1[r];
    }
    l_run = l_run * alpha + rs;
    m_run = m_new;
#pragma unroll
    for (int u = 0; u < NU; ++u) oacc[u] *= alpha;

    // P enters the PV product as two 16-bit terms: the kernel waits on memory,
    // the second product hides.  One rounded term would be exact only for the
    // largest key of each wave's share of a split, so the error would grow with
    // the length of the splits.
    u32x4 pw, rw;
    auto put = [&](int i, float a, float b) __attribute__((always_inline)) {
      uint32_t hi, lo;
      two_terms<T>(a, b, hi, lo);
      pw[i] = hi;
      rw[i] = lo;
    };
    put(0, s0[0], s0[1]);
    put(1, s0[2], s0[3]);
    put(2, s1[0], s1[1]);
    put(3, s1[2], s1[3]);
    const V8 pf = as_vec8<V8>(pw), rf = as_vec8<V8>(rw);

    // 8 keys x NU d in registers -> NU operands of 8 keys each
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int word = u >> 1;
      u32x4 a;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t x = vc[2 * j][word], y = vc[2 * j + 1][word];
        a[j] = (u & 1) ? ((x >> 16) | (y & 0xffff0000u)) : ((x & 0xffffu) | (y << 16));
      }
      oacc[u] = E::mfma16(as_vec8<V8>(a), pf, oacc[u]);
      oacc[u] = E::mfma16(as_vec8<V8>(a), rf, oacc[u]);
    }
  };

  // ---- the wave's chunks wave, wave+W, ...; next chunk's DMA in flight ----
  const int64_t nchunks = (ke - kb + kDecChunk - 1) / kDecChunk;
  HCP_LDS_PTR(char) be = (HCP_LDS_PTR(char))(bufE[wave]);
  HCP_LDS_PTR(char) bo = (HCP_LDS_PTR(char))(bufO[wave]);
  // The next chunk's DMA is issued unconditionally (past the wave's last
  // chunk it re-reads the split's last chunk into the buffer nobody reads):
  // with no branch around it, the wait before each compute is exactly "the
  // previous chunk's loads", not a conservative wait for all of them.  (Rows
  // past the descriptor's range instead, which read as zeros without traffic,
  // measured slower: 16.5 -> 18.6 us at 8 x ~5500 keys of 2 x 64 heads.)
  const int64_t last = nchunks - 1;
  auto next_k0 = [&](int64_t cn) __attribute__((always_inline)) {
    return kb + (cn < last ? cn : last) * kDecChunk;
  };
  // Before a compute, the wave waits until only the 2*NLD loads it just
  // issued (into the other buffer) are outstanding: its own DMA into the
  // buffer it reads has landed.  Buffers are wave-private, so no barrier.
  int64_t ci = wave;
  // Paged segments: the lane's block ids are fetched one chunk ahead of the
  // chunk's DMA, so looking them up never waits on the DMA in flight.  When
  // the cache spans less than 4 GiB from this head's base the DMA is a
  // bounds-checked buffer load over one descriptor for the whole cache (a
  // block id past the cache reads zeros); otherwise a global load with a
  // 64-bit address (a block id past the cache clamped to its last block).
  if constexpr (PAGED) {
    const int64_t blockb = kva.stride_block * 2;
    const uint64_t span = static_cast<uint64_t>(e.kv.num_blocks) * static_cast<uint64_t>(blockb);
    const bool pbuf = e.kv.num_blocks > 0 && span < (uint64_t{1} << 32);
    if (ci < nchunks) {
      const int64_t hb = static_cast<int64_t>(kvh) * kva.stride_head * 2;
      const int nrec =
          __builtin_amdgcn_readfirstlane(pbuf ? static_cast<int>(static_cast<uint32_t>(span)) : 0);
      // the bases are wave-uniform; say so, or the descriptors land in
      // VGPRs and every buffer load becomes a waterfall loop
      auto uniform_ptr = [](const char* ptr) __attribute__((always_inline)) {
        const uint64_t a = reinterpret_cast<uint64_t>(ptr);
        const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a));
        const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a >> 32));
        return reinterpret_cast<char*>((static_cast<uint64_t>(hi) << 32) | lo);
      };
      const __amdgpu_buffer_rsrc_t rk =
          __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(kva.k + hb), 0, nrec, kBufWord3);
      const __amdgpu_buffer_rsrc_t rv =
          __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(kva.v + hb), 0, nrec, kBufWord3);
      const uint32_t id_max = __builtin_amdgcn_readfirstlane(
          e.kv.num_blocks > 0 && e.kv.num_blocks <= 0xffffffffll
              ? static_cast<uint32_t>(e.kv.num_blocks - 1) : 0xffffffffu);
      uint32_t idA[NLD], idB[NLD];
      auto fetch_ids = [&](int64_t k0, uint32_t (&ids)[NLD]) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NLD; ++j) {
          int64_t key = k0 + j * KPI + kr;
          key = key < ke ? key : ke - 1;  // rows past the split: masked
          ids[j] = static_cast<uint32_t>(kva.bt[(kva.start + key) >> kva.bs_shift]);
        }
      };
      // one chunk's DMA; BUF (compile-time) picks the load form
      auto issue_p = [&](auto buf, int64_t k0, const uint32_t (&ids)[NLD], HCP_LDS_PTR(char) dst)
          __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NLD; ++j) {
          const int row = j * KPI + kr;
          int64_t key = k0 + row;
          key = key < ke ? key : ke - 1;
          const int64_t x = kva.start + key;
          int ch = sl ^ (row % CPR);
          ch = ch < cv ? ch : 0;
          const int64_t inb = (x & kva.bs_mask) * rowb_g + 16 * ch;
          if constexpr (decltype(buf)::value) {
            const uint32_t off = ids[j] * static_cast<uint32_t>(blockb) + static_cast<uint32_t>(inb);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rk, reinterpret_cast<HCP_LDS_PTR(void)>(dst + j * 1024), 16,
                static_cast<int>(off), 0, 0, kStreamAux);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rv, reinterpret_cast<HCP_LDS_PTR(void)>(dst + CHB + j * 1024), 16,
                static_cast<int>(off), 0, 0, kStreamAux);
          } else {
            // a block id past the cache is clamped to its last block
            const uint32_t id = ids[j] < id_max ? ids[j] : id_max;
            const int64_t o = static_cast<int64_t>(id) * blockb + hb + inb;
            __builtin_amdgcn_global_load_lds(
                reinterpret_cast<const __attribute__((address_space(1))) void*>(
                    reinterpret_cast<uintptr_t>(kva.k + o)),
                reinterpret_cast<HCP_LDS_PTR(void)>(dst + j * 1024), 16, 0, kStreamAux);
            __builtin_amdgcn_global_load_lds(
                reinterpret_cast<const __attribute__((address_space(1))) void*>(
                    reinterpret_cast<uintptr_t>(kva.v + o)),
                reinterpret_cast<HCP_LDS_PTR(void)>(dst + CHB + j * 1024), 16, 0, kStreamAux);
          }
        }
      };
      // per step: fetch the ids of chunk ci+2W, issue chunk ci+W (its ids
      // fetched a step ago), wait until only those 3*NLD loads are
      // outstanding -- chunk ci has landed -- and compute it
      auto run_loop = [&](auto buf) __attribute__((always_inline)) {
        fetch_ids(kb + ci * kDecChunk, idA);
        fetch_ids(next_k0(ci + W), idB);
        issue_p(buf, kb + ci * kDecChunk, idA, be);
        while (true) {
          fetch_ids(next_k0(ci + 2 * W), idA);
          issue_p(buf, next_k0(ci + W), idB, bo);
          wait_vmcnt<3 * NLD>();
          compute(kb + ci * kDecChunk, be);
          ci += W;
          if (ci >= nchunks) break;
          fetch_ids(next_k0(ci + 2 * W), idB);
          issue_p(buf, next_k0(ci + W), idA, be);
          wait_vmcnt<3 * NLD>();
          compute(kb + ci * kDecChunk, bo);
          ci += W;
          if (ci >= nchunks) break;
        }
      };
      if (pbuf)
        run_loop(std::true_type{});
      else
        run_loop(std::false_type{});
    }
  }
  if (!PAGED && ci < nchunks) {
    issue(kb + ci * kDecChunk, be);
    while (true) {
      issue(next_k0(ci + W), bo);
      wait_vmcnt<2 * NLD>();
      compute(kb + ci * kDecChunk, be);
      ci += W;
      if (ci >= nchunks) break;
      issue(next_k0(ci + W), be);
      wait_vmcnt<2 * NLD>();
      compute(kb + ci * kDecChunk, bo);
      ci += W;
      if (ci >= nchunks) break;
    }
  }

  // ---- combine the W waves (the chunk buffers are reused for O) ----
  // Each wave's last prefetch (issued unconditionally in the loop) may still
  // be writing bufE/bufO, which sm_o overlays: drain it before the barrier.
  wait_vmcnt<0>();
  __syncthreads();
  // rows of D + 4 floats: the 16 heads' 16-byte stores fall on different banks
  float (*sm_o)[16][D + 4] = reinterpret_cast<float (*)[16][D + 4]>(&bufE[0][0]);
  static_assert(sizeof(float) * W * 16 * (D + 4) <= W * 2 * CHB, "combine staging");
  float l_tot = l_run + __shfl_xor(l_run, 16);
  l_tot += __shfl_xor(l_tot, 32);
  if (g4 == 0) {
    sm_m[wave][c16] = m_run;
    sm_l[wave][c16] = l_tot;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int u = 0; u < NU; u += 4)
      *reinterpret_cast<f32x4*>(&sm_o[wave][c16][NU * (4 * g4 + r) + u]) =
          f32x4{oacc[u][r], oacc[u + 1][r], oacc[u + 2][r], oacc[u + 3][r]};
  __syncthreads();

  for (int idx = tid; idx < G * D; idx += 64 * W) {
    const int h = idx / D, d = idx % D;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < W; ++w) M = fmaxf(M, sm_m[w][h]);
    const float Mu = (M == -INFINITY) ? 0.f : M;
    float L = 0.f, O = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float sc = fast_exp2(sm_m[w][h] - Mu);
      L += sm_l[w][h] * sc;
      O += sm_o[w][h][d] * sc;
    }
    const int head = h0 + h;
    const int64_t slot = static_cast<int64_t>(sp) * p.num_heads + head;
    const bool some = KEEP_NAN ? L != 0.f : L > 0.f;
    global_ptr(p.ws_o)[slot * D + d] = some ? O / L : 0.f;
    if (d == 0) global_ptr(p.ws_lse)[slot] = some ? M * kLn2 + __logf(L) : -INFINITY;
  }
}

// The kernel's one argument, by a pointer the compiler cannot see through:
// its loads stay where they are used.
template <typename P>
__device__ __forceinline__ const P& fresh_params() {
  auto k = __builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(k));
  return *(const P*)k;
}

// Paged-ness is a property of each entry (a sequence's peer segment is
// contiguous, its local segment paged), uniform within a workgroup.
//
// A planned launch gives each workgroup a list of records with about the same
// number of keys in all, one round of the machine: sequences of any lengths
// leave no CU idle at the end.  A record carries its entry, so that a split
// starts with one scalar load and not a chain of three.  Split + merge, 28 / 4
// x 128 heads, before (equal splits in up to four rounds) and after: 16 x 1k-8k
// keys 46.6 -> 32.4 us, 32 x 0.5k-8k 75 -> 60.5 us (5.6 TB/s), 64 x 0.5k-2k 40.7
// -> 35 us, 32 x 34k 366 -> 331 us (6.7 TB/s), 33k in one sequence 22.7 -> 20.4
// us; 8 x 2k-9k at 14 / 2 x 64 16.2 -> 13.1 us.  The last three microseconds or
// so of the short ones are the chain of latencies (record, block ids, keys).
template <int D, typename T, bool KEEP_NAN>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * DecShared<D>::W, 64 * DecShared<D>::W),
                          amdgpu_waves_per_eu(1, 1))) void
decode_split_kernel(DecParams p) {
  constexpr int CHB = DecShared<D>::CHB;
  constexpr int W = DecShared<D>::W;
  __shared__ __attribute__((aligned(1024))) char bufE[W][2 * CHB];
  __shared__ __attribute__((aligned(1024))) char bufO[W][2 * CHB];
  __shared__ float sm_m[W][16];
  __shared__ float sm_l[W][16];
  int kvh;
  int64_t item;
  if (!xcd_remap(blockIdx.x, static_cast<int64_t>(p.num_wgs) * p.head_chunks,
                 p.num_kv_heads, &kvh, &item))
    return;
  const int chunk = static_cast<int>(item % p.head_chunks);
  int s = static_cast<int>(item / p.head_chunks);
  while (true) {
    // the parameters are read afresh for every split: held across the list
    // they would be spilled
    const DecParams& p = fresh_params<DecParams>();
    hcp_decode_work w;
    if (p.works != nullptr) {
      w = global_ptr(p.works)[s];
    } else {
      const hcp_decode_split spl = global_ptr(p.splits)[s];
      w.e = global_ptr(p.entries)[spl.entry];
      w.key_begin = spl.key_begin;
      w.key_end = spl.key_end;
      w.slot = spl.slot;  // workspace partial of this split
      w.next = -1;
    }
    if (w.e.kv.block_table != 0) {
      w.e.kv.k_addr += p.kv_base;
      w.e.kv.v_addr += p.kv_base;
      decode_split_body<D, T, true, KEEP_NAN>(p, kvh, chunk, w.slot, w.e, w.key_begin, w.key_end, bufE, bufO,
                                    sm_m, sm_l);
    } else {
      decode_split_body<D, T, false, KEEP_NAN>(p, kvh, chunk, w.slot, w.e, w.key_begin, w.key_end, bufE,
                                     bufO, sm_m, sm_l);
    }
    if (w.next < 0) return;
    s = w.next;
    __syncthreads();  // this split has been combined out of the buffers
  }
}

// Inclusive prefix sum over the wave's lanes, by DPP moves (inside rows of 16
// lanes, then row 0 -> 1 and 2 -> 3, then the lower half into the upper):
// an add each, where six shuffles through LDS take about 100 cycles each.
__device__ __forceinline__ int wave_prefix(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return x;
}

// Length r as the caller gives it.
__device__ __forceinline__ int64_t paged_len(const PagedDecParams& p, int r) {
  return p.lens_wide ? global_ptr(reinterpret_cast<const int64_t*>(p.lens))[r]
                     : global_ptr(reinterpret_cast<const int32_t*>(p.lens))[r];
}

// A pure decode batch without a plan: lengths and block tables come straight
// from the step's metadata on the device, so the host neither waits for them
// nor plans nor uploads.  The keys of all sequences are laid end to end in
// chunks of 32, each sequence with kStart more for what its split costs to
// start, and cut into equal shares, one for every workgroup; a workgroup finds
// its share by a prefix sum over the lengths.  The piece of sequence r in
// workgroup w is slot w + r: along the batch either w or r grows by one from
// piece to piece, so no two pieces share a slot and a sequence's slots are
// consecutive.  Split + merge at 28 / 4 x 128, against a planned launch of the
// same batch: 1 x 2000 keys 11.5 / 9.6 us, 16 x 1k-8k 34.6 / 32.6 us, 32 x 0.5k-8k
// 60.2 / 60.6 us -- the two microseconds of the sums, for the 100 us a
// step that reading the lengths, planning and the upload kept the GPU waiting.
template <int D, typename T, bool KEEP_NAN>
__global__ __attribute__((amdgpu_flat_work_group_size(64 * DecShared<D>::W, 64 * DecShared<D>::W),
                          amdgpu_waves_per_eu(1, 1))) void
decode_paged_kernel(PagedDecParams p_) {
  constexpr int CHB = DecShared<D>::CHB;
  constexpr int W = DecShared<D>::W;
  constexpr int NT = 64 * W;
  constexpr int EPT = kDecMaxSeqs / NT;  // sequences per thread of the prefix sum
  constexpr int kStart = 8;              // a split's start and end, in chunks
  __shared__ __attribute__((aligned(1024))) char bufE[W][2 * CHB];
  __shared__ __attribute__((aligned(1024))) char bufO[W][2 * CHB];
  __shared__ float sm_m[W][16];
  __shared__ float sm_l[W][16];
  __shared__ int sm_len[kDecMaxSeqs], sm_all[kDecMaxSeqs];  // keys seen, in the cache (-1: not run)
  __shared__ int sm_w[2][W];
  __shared__ int sm_cut[4];
  int kvh;
  int64_t item;
  if (!xcd_remap(blockIdx.x, static_cast<int64_t>(p_.d.num_wgs) * p_.d.head_chunks,
                 p_.d.num_kv_heads, &kvh, &item))
    return;
  const int chunk = static_cast<int>(item % p_.d.head_chunks);
  const int wg = static_cast<int>(item / p_.d.head_chunks);
  const int n = p_.num_seqs;
  {
    // ---- prefix sums over the sequences: chunks, sequences with keys ----
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int c[EPT], cs = 0, zs = 0;
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
      const int r = tid * EPT + j;
      const int64_t given = r < n ? paged_len(p_, r) : 0;
      const int all =  // keys that the sequence's query sees; max_len < 2^31
          static_cast<int>(given < 0 ? 0 : given < p_.max_len ? given : p_.max_len);
      const int len = p_.window > 0 && all > p_.window ? p_.window : all;
      if (r < n) {
        sm_all[r] = given == HCP_LEN_NOT_RUN ? -1 : all;
        sm_len[r] = len;
      }
      c[j] = (len >> 5) + ((len & 31) != 0);
      cs += c[j];
      zs += c[j] > 0;
    }
    const int ci = wave_prefix(cs), zi = wave_prefix(zs);
    if (lane == 63) {
      sm_w[0][wave] = ci;
      sm_w[1][wave] = zi;
    }
    if (tid == 0) sm_cut[0] = -1;
    __syncthreads();
    int cb = ci - cs, zb = zi - zs;
    unsigned total = 0, some = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      if (w < wave) {
        cb += sm_w[0][w];
        zb += sm_w[1][w];
      }
      total += sm_w[0][w];
      some += sm_w[1][w];
    }
    // ---- this workgroup's share: at least two chunks (64 keys) ----
    const unsigned most = static_cast<unsigned>(p_.d.num_wgs), half = (total + 1) / 2;
    const unsigned wgs = most < half ? most : half;
    if (static_cast<unsigned>(wg) < wgs) {
      const unsigned share = total / wgs;
      const unsigned start = share < kStart ? share : kStart;
      const unsigned span = total + start * some, q = span / wgs, rem = span - q * wgs;
      // cuts at span * w / wgs; the thread whose sequence holds one says which
      // of its chunks come before it (in steps of 4, one for each wave, where
      // the shares are long)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const unsigned w = wg + i, x = q * w + rem * w / wgs;
        unsigned base = cb + start * zb;
#pragma unroll
        for (int j = 0; j < EPT; ++j) {
          const unsigned next = base + (c[j] > 0 ? c[j] + start : 0u);
          if (x >= base && (x < next || (w == wgs && x == next && c[j] > 0))) {
            unsigned in = x - base > start ? x - base - start : 0u;
            if (share >= 16) in = (in + 2) & ~3u;
            if (w == wgs || in > static_cast<unsigned>(c[j])) in = c[j];
            sm_cut[2 * i] = tid * EPT + j;
            sm_cut[2 * i + 1] = in;
          }
          base = next;
        }
      }
    }
    __syncthreads();
  }
  const int r0 = __builtin_amdgcn_readfirstlane(sm_cut[0]);
  const int o0 = __builtin_amdgcn_readfirstlane(sm_cut[1]);
  const int r1 = r0 < 0 ? -2 : __builtin_amdgcn_readfirstlane(sm_cut[2]);  // -1, -2: no share
  const int o1 = __builtin_amdgcn_readfirstlane(sm_cut[3]);
  for (int r = r0; r <= r1; ++r) {
    const PagedDecParams& p = fresh_params<PagedDecParams>();
    const int len = __builtin_amdgcn_readfirstlane(sm_len[r]);
    const int all = __builtin_amdgcn_readfirstlane(sm_all[r]);
    const int c = (len >> 5) + ((len & 31) != 0);
    const int b = r == r0 ? o0 : 0, e_ = r == r1 ? o1 : c;
    if (b >= e_) continue;
    if (kvh == 0 && chunk == 0 && threadIdx.x == 0) {
      if (b == 0) global_ptr(p.seq_slots)[2 * r] = wg + r;
      if (e_ == c) global_ptr(p.seq_slots)[2 * r + 1] = wg + r;
    }
    hcp_varlen_entry e;
    e.q_start = r;
    e.q_len = 1;
    e.causal_offset = 0;
    e.kv = p.kv;
    e.kv.block_table = p.kv.block_table + static_cast<uint64_t>(r) * p.bt_stride * 4;
    e.kv.start = all - len;  // the last `window` keys
    e.kv.len = len;
    const int64_t ke = static_cast<int64_t>(e_) * 32;
    decode_split_body<D, T, true, KEEP_NAN>(p.d, kvh, chunk, wg + r, e, static_cast<int64_t>(b) * 32,
                                  ke < len ? ke : len, bufE, bufO, sm_m, sm_l);
    __syncthreads();  // this split has been combined out of the buffers
  }
  // the reduce goes by the slots alone: a sequence without keys says so
  if (wg == 0 && kvh == 0 && chunk == 0) {
    const PagedDecParams& p = fresh_params<PagedDecParams>();
    for (int r = threadIdx.x; r < p.num_seqs; r += NT) {
      if (sm_len[r] > 0) continue;
      global_ptr(p.seq_slots)[2 * r] = 0;
      global_ptr(p.seq_slots)[2 * r + 1] = sm_all[r] < 0 ? -2 : -1;
    }
  }
}

// Merge every partial of one (sequence, query head) -- and the running
// accumulator, when given -- into the output row and its LSE.  One workgroup
// of D threads per (sequence, head) column group, thread d owns column d;
// with many partials per sequence (1, 2 or 4 groups) the groups take
// interleaved shares of the partials and are merged through LDS.  Bound by
// latency: a thread issues the LSEs and columns of 16 partials at once, before
// any maximum is known, and keeps a running maximum over batches of 16 (with
// the maximum taken first, split + merge of 1 x 2000 keys took 10.7 us, now
// 9.4).  Merged by the split kernel's last workgroup of each sequence instead,
// 31 to 64 partials took longer than this launch costs.
template <int D, typename T>
__global__ __launch_bounds__(4 * D) void decode_reduce_kernel(RedParams p) {
  constexpr int U = 16;
  __shared__ float sm_m[4], sm_s[4];
  __shared__ float sm_o[4][D];
  const int ng = p.groups;  // column groups; group gi takes partials gi, gi + ng, ...
  const int sh = blockIdx.x;
  const int seq = sh / p.num_heads, head = sh % p.num_heads;
  const int row = p.rows != nullptr ? p.rows[seq] : seq;  // of out, lse and acc
  const int tid = threadIdx.x;
  const int d = tid % D, gi = tid / D;
  int p0, n;
  if (p.seq_slots != nullptr) {
    // kept inside the workspace whatever stands there: a caller that changes
    // the lengths while the split kernel reads them leaves pairs unwritten
    const int first = p.seq_slots[2 * seq], last = p.seq_slots[2 * seq + 1];
    p0 = first < 0 ? 0 : first < p.num_slots ? first : p.num_slots;
    n = (last < -2 ? -2 : last < p.num_slots ? last : p.num_slots - 1) - p0 + 1;
    if (n < 0) return;  // not run
  } else {
    p0 = p.seq_partial_start[seq];
    n = p.seq_partial_start[seq + 1] - p0;
  }
  const int64_t lstep = p.num_heads;
  const float* lcol = p.ws_lse + static_cast<int64_t>(p0) * lstep + head;
  const int64_t ostep = lstep * D;
  const float* ocol = p.ws_o + (static_cast<int64_t>(p0) * lstep + head) * D + d;

  // accumulator first: out / lse may alias acc_o / acc_lse, and every read
  // of them happens before the barrier below, every write after it
  float acc_l = -INFINITY, acc_v = 0.f;
  if (p.acc_lse != nullptr) {
    acc_l = p.acc_lse[static_cast<int64_t>(head) * p.acc_lse_stride_head + row];
    if (acc_l == INFINITY) acc_l = -INFINITY;  // merge_attn_states reads +inf as empty
    const uint16_t* arow = reinterpret_cast<const uint16_t*>(p.acc_o) +
                           row * p.acc_stride_tok + static_cast<int64_t>(head) * p.acc_stride_head;
    acc_v = d < p.head_dim ? Elem<T>::to_float(arow[d]) : 0.f;
  }
  // a weighted sum relative to the running maximum m
  float m = -INFINITY, S = 0.f, O = 0.f;
  auto rebase = [&](float mn) __attribute__((always_inline)) {
    const float sc = m == -INFINITY ? 0.f : __expf(m - mn);
    S *= sc;
    O *= sc;
    m = mn;
  };
  for (int i0 = gi; i0 < n; i0 += U * ng) {
    float l[U], v[U];
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const int i = i0 + j * ng < n ? i0 + j * ng : i0;  // past the last: not summed
      l[j] = lcol[i * lstep];
      v[j] = ocol[i * ostep];
    }
    float mn = m;
#pragma unroll
    for (int j = 0; j < U; ++j) mn = fmaxf(mn, l[j]);
    // (relative to 0 where no partial has keys: their weights are 0, but one
    // with a NaN LSE makes the sums NaN)
    const float ref = mn == -INFINITY ? 0.f : mn;
    rebase(mn);
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const bool in = i0 + j * ng < n;
      const float w = in ? __expf(l[j] - ref) : 0.f;
      S += w;
      O = in ? __builtin_fmaf(w, v[j], O) : O;
    }
  }
  if (ng > 1) {
    if (d == 0) {
      sm_m[gi] = m;
      sm_s[gi] = S;
    }
    sm_o[gi][d] = O;
  }
  __syncthreads();
  if (gi != 0) return;
  for (int g2 = 1; g2 < ng; ++g2) {
    if (sm_s[g2] == 0.f) continue;
    const float mn = fmaxf(m, sm_m[g2]);
    rebase(mn);
    const float w = __expf(sm_m[g2] - mn);
    S = __builtin_fmaf(w, sm_s[g2], S);
    O = __builtin_fmaf(w, sm_o[g2][d], O);
  }
  const bool nan = S != S;  // the partials' own
  if (acc_l != -INFINITY) {
    const float mn = fmaxf(m, acc_l);
    rebase(mn);
    const float w = __expf(acc_l - mn);
    S += w;
    O = __builtin_fmaf(w, acc_v, O);
  }
  const bool any = m != -INFINITY || nan;
  uint16_t* orow = reinterpret_cast<uint16_t*>(p.out) + row * p.o_stride_tok +
                   static_cast<int64_t>(head) * p.o_stride_head;
  if (d < p.head_dim) orow[d] = Elem<T>::from_float(any ? O / S : 0.f);
  if (p.lse != nullptr && d == 0)
    p.lse[static_cast<int64_t>(head) * p.lse_stride_head + row] =
        any && !nan ? m + __logf(S) : -INFINITY;
}

template <int D, typename T>
static hipError_t launch_dec_t(const DecParams& dp, const RedParams& rp, hipStream_t st) {
  const int64_t grid =
      xcd_grid_size(static_cast<int64_t>(dp.num_wgs) * dp.head_chunks, dp.num_kv_heads);
  if (grid > 0) {
    const dim3 g(static_cast<unsigned>(grid)), b(64 * DecShared<D>::W);
    if (dp.keep_nan)
      hipLaunchKernelGGL((decode_split_kernel<D, T, true>), g, b, 0, st, dp);
    else
      hipLaunchKernelGGL((decode_split_kernel<D, T, false>), g, b, 0, st, dp);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
  }
  const int64_t rgrid = static_cast<int64_t>(rp.num_seqs) * rp.num_heads;
  if (rgrid > 0) {
    // more column groups when a sequence has many partials (one long
    // request split over the whole machine): shorter dependent load chains
    RedParams r = rp;
    const int per_seq = rp.num_seqs > 0 ? dp.num_splits / rp.num_seqs : 0;
    r.groups = per_seq >= 48 ? 4 : per_seq >= 24 ? 2 : 1;
    hipLaunchKernelGGL((decode_reduce_kernel<D, T>), dim3(static_cast<unsigned>(rgrid)),
                       dim3(D * r.groups), 0, st, r);
    return hipGetLastError();
  }
  return hipSuccess;
}

hipError_t launch_decode(const DecParams& dp, const RedParams& rp, int head_dim,
                         int dtype, hipStream_t st) {
  if (head_dim > 128)  // 136 .. 256: computed in 256 columns
    return dtype == HCP_DTYPE_BF16 ? launch_dec_t<256, __bf16>(dp, rp, st)
                                   : launch_dec_t<256, _Float16>(dp, rp, st);
  if (head_dim > 64)  // 72 .. 128: computed in 128 columns
    return dtype == HCP_DTYPE_BF16 ? launch_dec_t<128, __bf16>(dp, rp, st)
                                   : launch_dec_t<128, _Float16>(dp, rp, st);
  return dtype == HCP_DTYPE_BF16 ? launch_dec_t<64, __bf16>(dp, rp, st)
                                 : launch_dec_t<64, _Float16>(dp, rp, st);
}

template <int D, typename T>
static hipError_t launch_dec_paged_t(const PagedDecParams& p, const RedParams& rp,
                                     hipStream_t st) {
  const int64_t grid = xcd_grid_size(static_cast<int64_t>(p.d.num_wgs) * p.d.head_chunks,
                                     p.d.num_kv_heads);
  const dim3 g(static_cast<unsigned>(grid)), b(64 * DecShared<D>::W);
  if (p.d.keep_nan)
    hipLaunchKernelGGL((decode_paged_kernel<D, T, true>), g, b, 0, st, p);
  else
    hipLaunchKernelGGL((decode_paged_kernel<D, T, false>), g, b, 0, st, p);
  const hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  RedParams r = rp;
  const int per_seq = (p.d.num_wgs + rp.num_seqs) / rp.num_seqs;
  r.groups = per_seq >= 48 ? 4 : per_seq >= 24 ? 2 : 1;
  hipLaunchKernelGGL((decode_reduce_kernel<D, T>),
                     dim3(static_cast<unsigned>(rp.num_seqs * rp.num_heads)), dim3(D * r.groups),
                     0, st, r);
  return hipGetLastError();
}

hipError_t launch_decode_paged(const PagedDecParams& p, const RedParams& rp, int head_dim,
                               int dtype, hipStream_t st) {
  const bool bf = dtype == HCP_DTYPE_BF16;
  switch (padded_head_dim(head_dim)) {
    case 256:
      return bf ? launch_dec_paged_t<256, __bf16>(p, rp, st)
                : launch_dec_paged_t<256, _Float16>(p, rp, st);
    case 128:
      return bf ? launch_dec_paged_t<128, __bf16>(p, rp, st)
                : launch_dec_paged_t<128, _Float16>(p, rp, st);
    default:
      return bf ? launch_dec_paged_t<64, __bf16>(p, rp, st)
                : launch_dec_paged_t<64, _Float16>(p, rp, st);
  }
}

}  // namespace hcp
