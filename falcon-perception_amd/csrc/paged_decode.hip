// Split-K paged decode attention (one query token per sequence) and its merge.
//
// Replaces the reference's compiled_flex_attn_decode call (attention.py:17,
// model.py:156-162) on the pool views that PagedKVCache.assign returns
// (paged_attention.py:232), and the block-mask conversion that call depends on
// (paged_attention.py:234-333, paged_inference.py:783-826): the kernel reads
// page_table[batch_idx[b], t / P] itself and bounds the context by input_pos[b].
//
// HBM-bound: every cached K and V row of every sequence is read exactly once.
//   grid  = (cache heads, batch, splits); a workgroup of 4 wavefronts owns one
//           (sequence, cache head, token range) and serves all G = Hq / Hc query
//           heads of that cache head from a single read of K and V.  A launch
//           of more than one to four workgroups to a CU (even_cut_line), or of
//           several sequences under a limit much longer than they are
//           (even_cut_pays), runs as (cache
//           heads, chunks) instead: the contexts laid end to end and cut into
//           equal chunks, a workgroup working through the sequences its chunk
//           touches.  With arrival counters (fp_paged_decode_step) few
//           sequences run as (cache heads, pieces), all pieces of one length
//           (merged_pieces).
//   loads = a row (D elements) is covered by TPR = D * elem / 16 lanes holding
//           16 bytes each, so a wavefront load instruction moves 64 / TPR whole
//           rows, contiguous inside a page; U such loads of K and of V are in
//           flight per lane before the arithmetic starts.
//   math  = each lane group keeps its own online-softmax state (m, l, acc) in
//           log2 space; q.k partial sums are combined across the TPR lanes with
//           DPP adds; lane groups, then wavefronts (through LDS), then splits
//           (through the workspace) are combined at the end: by the merge
//           kernel, or by the last workgroup of a (sequence, cache head) to
//           leave its result where the caller keeps arrival counters.
#include "decode_common.h"
#include "paged_decode_mfma.h"

#include <atomic>

#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>
#include <math.h>

#include <type_traits>

namespace {

using namespace fp_decode;

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
// ---- element access: 16 bytes of a row -----------------------------------
// A lane holds 16 bytes of a K or V row as four 32-bit words.  `Q` is the lane's
// share of a query row, `dot` its contribution to q.k, `unpack` the V values as floats.
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

struct F32 {
  using type = float;
  static constexpr int kEpl = 4;
  struct Q { float f[4]; };
  static __device__ __forceinline__ Q load_q(const v4u& r) {
    return Q{{__uint_as_float(r.x), __uint_as_float(r.y), __uint_as_float(r.z), __uint_as_float(r.w)}};
  }
  static __device__ __forceinline__ float dot(const Q& q, const v4u& k) {
    float p = q.f[0] * __uint_as_float(k.x);
    p = fmaf(q.f[1], __uint_as_float(k.y), p);
    p = fmaf(q.f[2], __uint_as_float(k.z), p);
    return fmaf(q.f[3], __uint_as_float(k.w), p);
  }
  static __device__ __forceinline__ void unpack(const v4u& r, float* f) {
    f[0] = __uint_as_float(r.x);
    f[1] = __uint_as_float(r.y);
    f[2] = __uint_as_float(r.z);
    f[3] = __uint_as_float(r.w);
  }
  static __device__ __forceinline__ void store(char* p, float v) { *reinterpret_cast<float*>(p) = v; }
  static __device__ __forceinline__ float round(float v) { return v; }
};
// bf16 / f16: q.k on the packed pairs with v_dot2 (fp32 accumulate), no conversion of K
struct BF16 {
  using type = __hip_bfloat16;
  static constexpr int kEpl = 8;
  struct Q { v4u w; };
  static __device__ __forceinline__ Q load_q(const v4u& r) { return Q{r}; }
  static __device__ __forceinline__ float dot(const Q& q, const v4u& k) {
    float p = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // the words go through scalars: bit_cast applied directly to a vector element reads element 0
      const uint32_t qw = q.w[i], kw = k[i];
      p = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, qw), __builtin_bit_cast(bf16x2_t, kw), p, false);
    }
    return p;
  }
  static __device__ __forceinline__ void unpack(const v4u& r, float* f) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f[2 * i] = __uint_as_float(r[i] << 16);
      f[2 * i + 1] = __uint_as_float(r[i] & 0xffff0000u);
    }
  }
  static __device__ __forceinline__ void store(char* p, float v) {
    *reinterpret_cast<__hip_bfloat16*>(p) = __float2bfloat16(v);
  }
  static __device__ __forceinline__ float round(float v) { return __bfloat162float(__float2bfloat16(v)); }
};
struct F16 {
  using type = __half;
  static constexpr int kEpl = 8;
  struct Q { v4u w; };
  static __device__ __forceinline__ Q load_q(const v4u& r) { return Q{r}; }
  static __device__ __forceinline__ float dot(const Q& q, const v4u& k) {
    float p = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t qw = q.w[i], kw = k[i];
      p = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2_t, qw), __builtin_bit_cast(f16x2_t, kw), p, false);
    }
    return p;
  }
  static __device__ __forceinline__ void unpack(const v4u& r, float* f) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t w = r[i];
      const f16x2_t h = __builtin_bit_cast(f16x2_t, w);
      f[2 * i] = static_cast<float>(h.x);
      f[2 * i + 1] = static_cast<float>(h.y);
    }
  }
  static __device__ __forceinline__ void store(char* p, float v) { *reinterpret_cast<__half*>(p) = __float2half(v); }
  static __device__ __forceinline__ float round(float v) { return __half2float(__float2half(v)); }
};

// K and V are streamed once: non-temporal loads keep them from displacing the caches
__device__ __forceinline__ v4u stream_load(const char* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const v4u*>(p));
}

// One wavefront iteration: U row loads of K and V per lane are already in registers;
// fold them into the lane group's online-softmax state.  kMasked: rows at or past
// `t1` (only in the last iteration of a split) get a score of -inf.
// GK = 1: the G query heads share one K row; GK = G: every query head has its own K row (a cache
// that stores one K head per query head) while V is still shared.
template <typename E, int TPR, int G, int GK, int U, int RPW, bool kMasked>
__device__ __forceinline__ void fold_rows(const v4u (&kreg)[GK][U], const v4u (&vreg)[U], const typename E::Q (&q)[G],
                                          float qscale, int row0, int t1, float (&m)[G], float (&l)[G],
                                          float (&acc)[G][E::kEpl]) {
  constexpr int EPL = E::kEpl;
  float s[G][U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
#pragma unroll
    for (int g = 0; g < G; ++g) s[g][u] = E::dot(q[g], kreg[GK == 1 ? 0 : g][u]);
  }
#pragma unroll
  for (int g = 0; g < G; ++g) {
    row_sum<TPR, U>(s[g]);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float tot = s[g][u] * qscale;
      s[g][u] = (!kMasked || row0 + u * RPW < t1) ? tot : -INFINITY;
    }
  }
#pragma unroll
  for (int g = 0; g < G; ++g) {
    float mx = m[g];
#pragma unroll
    for (int u = 0; u < U; ++u) mx = fmaxf(mx, s[g][u]);
    const float ms = safe_max(mx);
    const float alpha = fast_exp2(m[g] - ms);
    m[g] = mx;
    float ps = 0.f;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      s[g][u] = fast_exp2(s[g][u] - ms);
      ps += s[g][u];
    }
    l[g] = l[g] * alpha + ps;
#pragma unroll
    for (int e = 0; e < EPL; ++e) acc[g][e] *= alpha;
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    float vf[EPL];
    E::unpack(vreg[u], vf);
#pragma unroll
    for (int g = 0; g < G; ++g) {
#pragma unroll
      for (int e = 0; e < EPL; ++e) acc[g][e] = fmaf(s[g][u], vf[e], acc[g][e]);
    }
  }
}

// ---- main kernel ------------------------------------------------------------
// kAligned: the page size is a power of two and a multiple of the rows one
// wavefront iteration covers, so those rows share one page and one base address.
//
// kPerHeadK serves a cache that holds one K head per QUERY head (the reference stores K and V
// expanded to n_heads because the 2D rotary angles differ per head, model.py:112-114) whose V heads
// are n_rep identical copies: a workgroup takes the G = n_rep query heads of one group, reads their G
// K rows and ONE V row (the first copy), i.e. (G + 1) / 2G of the bytes an expanded read costs.
constexpr int decode_loads_in_flight(int G, bool per_head_k) { return per_head_k && G >= 4 ? 4 : 8; }

// Four workgroups per CU instead of three (at most 128 registers) where the kernel fits without spilling:
// one query head per cache head, and two in fp32 (the 16-bit kernels keep twice the elements per lane).  Not for
// the even cut, which runs two workgroups per CU.
template <typename E, int D, int G, bool kPerHeadK, bool kFlat>
constexpr int decode_waves_per_simd() {
  return (!kFlat && !kPerHeadK && (G == 1 || (G == 2 && sizeof(typename E::type) == 4))) ? 4 : 1;
}

template <typename E, int D, int G, bool kDirect, bool kAligned, bool kPerHeadK = false, bool kFlat = false, bool kPieces = false>
__global__ __launch_bounds__(kThreads, (decode_waves_per_simd<E, D, G, kPerHeadK, kFlat>())) void paged_decode_kernel(const DecodeArgs a) {
  constexpr int EPL = E::kEpl;          // elements per lane
  constexpr int TPR = D / EPL;          // lanes per row
  constexpr int RPW = 64 / TPR;         // rows per wavefront load
  constexpr int GK = kPerHeadK ? G : 1; // K rows per token a workgroup reads
  constexpr int U = decode_loads_in_flight(G, kPerHeadK);  // loads of K (per K head) and of V in flight per lane
  constexpr int CH = RPW * U;           // rows per wavefront iteration
  constexpr int ROWB = D * sizeof(typename E::type);
  constexpr bool kMerges = !kDirect && !kFlat && merges_itself(G, D);

  __shared__ int s_pages[kMaxSplitPages];
  __shared__ float s_acc[kWaves][G][D];
  __shared__ float s_ml[kWaves][G][2];
  constexpr int NR = (2 * GK + RPW - 1) / RPW;  // load instructions for the fresh rows, a row to a lane group
  constexpr bool kEarly = !kFlat && !kPieces;
  constexpr bool kFull = kFlat && G * D >= 1024;  // the registers of a row's loop are all taken (fp32, eight heads, D 128)
  __shared__ __attribute__((aligned(1024))) char s_fresh[kEarly ? NR * 1024 : 16];

  // Workgroups are dealt to the 8 XCDs round-robin by linear id.  Heads run fastest:
  // every head of a sequence has the same amount of work, so each XCD gets an equal
  // share of the non-empty workgroups whatever the context lengths are.
  // The workgroup dispatcher deals consecutive workgroups of an XCD to its four shader engines in turn
  // and starts them in order, so with grid y = sequence every split of a sequence would land on the
  // same engine and an engine's load would be the lengths of "its" sequences (12 % apart at 64
  // sequences of 1 k to 4 k tokens).  Rotating the sequences by the split index spreads each sequence
  // over the engines.
  const int hc = blockIdx.x;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int grp = lane / TPR;  // row of this lane inside a wavefront load
  const int col = lane % TPR;  // 16-byte chunk of the row

  // Tokens [t0, t0 + part) of sequence b; a partial result goes to row hq * part_mul + part_add of the
  // workspace.
  auto piece = [&](const int b, const int t0, const int part, const int split, const int64_t part_mul,
                   const int64_t part_add, const int n_pieces, const int raw, const int trow, const int* pre_pages) {
  int L = trow < 0 ? 0 : raw;
  const int* pages_lds = pre_pages ? pre_pages : s_pages;
  // A position at or beyond max_context is outside what the launch was sized for: the context is read
  // up to max_context from the pool, and the fresh row of a fused append is neither folded nor stored
  // (it must not land on the slot of position max_context - 1, which holds a valid row).
  const bool beyond = L > a.max_context;
  if (beyond) L = a.max_context;
  auto lse_at = [&](int hq) -> float& {
    return a.lse[static_cast<int64_t>(b) * a.Hq + hq];
  };
  if (t0 >= L) {
    if ((kDirect || (kMerges && a.arrivals)) && split == 0) {
      // no visible key at all: out = 0, lse = -inf
      for (int i = tid; i < G * D; i += kThreads) {
        const int g = i / D, d = i - g * D;
        E::store(a.out + b * a.os_b + (hc * G + g) * a.os_h + d * sizeof(typename E::type), 0.f);
      }
      if (tid < G) lse_at(hc * G + tid) = -INFINITY;
      if constexpr (kMerges) clear_next_counter(a, b);
    }
    return;
  }
  const int t1 = L < t0 + part ? L : t0 + part;
  // Fused append: the newest token (position L - 1) is not in the pool yet.  The workgroup whose
  // range holds it reads that row from k_new / v_new, folds it in and writes it to its slot; the
  // pool is only read up to L - 2.
  const bool owns_new = a.k_new != nullptr && !beyond && t1 == L;
  const int t1_pool = owns_new ? t1 - 1 : t1;

  // this lane's 16 bytes of the query row of every head of the group
  typename E::Q q[G];
#pragma unroll
  for (int g = 0; g < G; ++g)
    q[g] = E::load_q(*reinterpret_cast<const v4u*>(a.q + b * a.qs_b + (hc * G + g) * a.qs_h + col * 16));

  float m[G], l[G], acc[G][EPL];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    m[g] = -INFINITY;
    l[g] = 0.f;
#pragma unroll
    for (int e = 0; e < EPL; ++e) acc[g][e] = 0.f;
  }

  // cache head of the workgroup's first K row and of its V row; with kPerHeadK the group's K heads
  // follow at head_stride
  const int64_t head_stride = a.n_slots * ROWB;
  const char* kbase = a.pool_k + static_cast<int64_t>(kPerHeadK ? hc * G : hc) * head_stride + col * 16;
  const char* vbase = a.pool_v + static_cast<int64_t>(kPerHeadK ? hc * G : hc) * head_stride + col * 16;

  // GK fresh rows of K, then as many of V: V is written to every copy so that the pool stays what the reference's append leaves (the
  // copies are read by the prefill kernel and by other callers).  Split by split they travel to LDS beside the page ids (kEarly): asked for
  // behind the other rows they are a trip to memory at the end of a short launch's last splits (one sequence of 711 tokens 8.0 -> 7.6 us a
  // layer).  Pieces and chunks of many lengths end one after the other anyway, and are no faster for it (16 sequences of 350 to
  // 4620 tokens 36.7 / 36.9 us, 64 of 1088 to 4096 117.1 / 117.4).
  const int h0 = kPerHeadK ? hc * G : hc;  // first cache head of this workgroup
  const auto fresh_row = [&](int r) {
    return r < GK ? a.k_new + b * a.kn_b + (h0 + r) * a.kn_h : a.v_new + b * a.vn_b + (h0 + r - GK) * a.vn_h;
  };
  const bool takes_new = owns_new && wave == (kEarly ? kWaves - 1 : 0);
  if constexpr (kEarly) {
    if (takes_new) {
#pragma unroll
      for (int j = 0; j < NR; ++j) {
        const int r = grp + j * RPW < 2 * GK ? grp + j * RPW : 2 * GK - 1;
        fp::load_to_lds(fresh_row(r) + col * 16, s_fresh + j * 1024);
      }
    }
  }

  // page ids of the split -> LDS, then the rows
  int64_t blk0;
  {
    int off_unused;
    a.pd.split(t0, blk0, off_unused);
    int64_t blk_last;
    a.pd.split(t1 - 1, blk_last, off_unused);
    const int nblk = pre_pages ? 0 : static_cast<int>(blk_last - blk0) + 1;
    for (int i = tid; i < nblk; i += kThreads) {
      int64_t page = 0;
      if (blk0 + i < a.n_pages) page = a.page_table[static_cast<int64_t>(trow) * a.pt_row_stride + blk0 + i];
      if (page < 0 || page >= a.pool_pages) page = 0;  // not a page of the pool
      s_pages[i] = static_cast<int>(page);
    }
  }
  __syncthreads();
  const int c_end = t1_pool;

#pragma nounroll
  for (int c0 = t0 + wave * CH; c0 < c_end; c0 += kWaves * CH) {
    v4u kreg[GK][U], vreg[U];
    if (kAligned) {
      // the CH rows of this iteration lie in one page: one base, constant offsets
      const int page = pages_lds[(c0 >> a.pd.shift) - static_cast<int>(blk0)];
      const int64_t slot = static_cast<int64_t>(page) * a.pd.page_size + (c0 & (a.pd.page_size - 1)) + grp;
      const char* kp = kbase + slot * ROWB;
      const char* vp = vbase + slot * ROWB;
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int gk = 0; gk < GK; ++gk) kreg[gk][u] = stream_load(kp + gk * head_stride + u * RPW * ROWB);
        vreg[u] = stream_load(vp + u * RPW * ROWB);
      }
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        int t = c0 + u * RPW + grp;
        if (t >= c_end) t = c_end - 1;
        int64_t blk;
        int off;
        a.pd.split(t, blk, off);
        const int64_t slot = static_cast<int64_t>(pages_lds[blk - blk0]) * a.pd.page_size + off;
#pragma unroll
        for (int gk = 0; gk < GK; ++gk) kreg[gk][u] = stream_load(kbase + gk * head_stride + slot * ROWB);
        vreg[u] = stream_load(vbase + slot * ROWB);
      }
    }
    if (c0 + CH <= c_end)
      fold_rows<E, TPR, G, GK, U, RPW, false>(kreg, vreg, q, a.qscale, c0 + grp, c_end, m, l, acc);
    else
      fold_rows<E, TPR, G, GK, U, RPW, true>(kreg, vreg, q, a.qscale, c0 + grp, c_end, m, l, acc);
  }

  if (takes_new) {
    int at = lane;
    if constexpr (kFlat && !kFull) asm volatile("" : "+v"(at));  // here and below: what only the end of a piece needs is not kept in registers from piece to piece
    const int byte = at % TPR * 16;
    // the newest token: one row, held by lane group 0; the other groups' is masked
    v4u kreg[GK][1], vreg[1];
    if constexpr (kEarly) {
      asm volatile("s_waitcnt vmcnt(0)" : : : "memory");  // the fresh rows have landed in LDS
#pragma unroll
      for (int gk = 0; gk < GK; ++gk) kreg[gk][0] = *reinterpret_cast<const v4u*>(s_fresh + gk * ROWB + byte);
      vreg[0] = *reinterpret_cast<const v4u*>(s_fresh + GK * ROWB + byte);
    } else {
#pragma unroll
      for (int gk = 0; gk < GK; ++gk) kreg[gk][0] = *reinterpret_cast<const v4u*>(fresh_row(gk) + byte);
      vreg[0] = *reinterpret_cast<const v4u*>(fresh_row(GK) + byte);
    }
    fold_rows<E, TPR, G, GK, 1, RPW, true>(kreg, vreg, q, a.qscale, t1 - 1 + at / TPR, t1, m, l, acc);
    if (at < TPR) {
      int64_t blk;
      int off;
      a.pd.split(t1 - 1, blk, off);
      const int64_t slot = static_cast<int64_t>(pages_lds[blk - blk0]) * a.pd.page_size + off;
#pragma unroll
      for (int gk = 0; gk < GK; ++gk) {
        __builtin_nontemporal_store(kreg[gk][0], reinterpret_cast<v4u*>(const_cast<char*>(kbase) + gk * head_stride + slot * ROWB));
        v4u vrow = vreg[0];
        if constexpr (kEarly && GK > 1)
          vrow = *reinterpret_cast<const v4u*>(s_fresh + (GK + gk) * ROWB + byte);
        else if constexpr (GK > 1)
          vrow = *reinterpret_cast<const v4u*>(fresh_row(GK + gk) + byte);
        __builtin_nontemporal_store(vrow, reinterpret_cast<v4u*>(const_cast<char*>(vbase) + gk * head_stride + slot * ROWB));
      }
    }
  }

  // combine the lane groups of this wavefront: every state at the common maximum, then the sums.  Each exchange between the lane
  // halves, and between rows of 16 lanes, adds up two elements at once and leaves one of them in either part, so that a lane
  // ends with a part of the elements.  (An exchange through LDS for every element and group was 0.8 us at the end of every piece; 0.2 us so.)
  // Where the loop in front has no register left the exchange through LDS is the better one, which changes the states in place: with
  // the sums beside them the compiler's loop is 3 % slower (64 sequences of 1024 to 4096 tokens, fp32, eight heads on 8, D 128: 358 / 346 us a layer).
  if constexpr (kFull) {
#pragma unroll
    for (int off = TPR; off < 64; off <<= 1) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const float mo = __shfl_xor(m[g], off), lo = __shfl_xor(l[g], off);
        const float mx = fmaxf(m[g], mo), ms = safe_max(mx);
        const float wa = fast_exp2(m[g] - ms), wb = fast_exp2(mo - ms);
        l[g] = l[g] * wa + lo * wb;
#pragma unroll
        for (int e = 0; e < EPL; ++e) acc[g][e] = acc[g][e] * wa + __shfl_xor(acc[g][e], off) * wb;
        m[g] = mx;
      }
    }
    if (lane < TPR) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
#pragma unroll
        for (int e = 0; e < EPL; ++e) s_acc[wave][g][col * EPL + e] = acc[g][e];
        if (lane == 0) {
          s_ml[wave][g][0] = m[g];
          s_ml[wave][g][1] = l[g];
        }
      }
    }
  } else {
    constexpr int N = G * EPL;
    float sum[N];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float mx = m[g];
      if (TPR <= 8) mx = fmaxf(mx, dpp<0x128>(mx));  // row_ror:8
      if (TPR <= 16) mx = max_across_rows(mx);
      if (TPR <= 32) mx = fp::max_across_lane_halves(mx);
      const float w = fast_exp2(m[g] - safe_max(mx));
      m[g] = mx;
      l[g] *= w;
#pragma unroll
      for (int e = 0; e < EPL; ++e) sum[g * EPL + e] = acc[g][e] * w;
    }
    if (TPR <= 8) {
#pragma unroll
      for (int i = 0; i < N; ++i) sum[i] += dpp<0x128>(sum[i]);
#pragma unroll
      for (int g = 0; g < G; ++g) l[g] += dpp<0x128>(l[g]);
    }
    if (TPR <= 32) add_across_halves<N>(sum);
    if (TPR <= 16) add_across_rows<N / 2>(sum);
    constexpr int NL = TPR <= 16 ? N / 4 : TPR <= 32 ? N / 2 : N;  // elements this lane ends with, from `held` on
    int at = lane;
    if constexpr (kFlat) asm volatile("" : "+v"(at));
    const int held = (TPR <= 32 ? (at >> 5) * (N / 2) : 0) + (TPR <= 16 ? (at >> 4 & 1) * (N / 4) : 0);
    static_assert(NL % EPL == 0 || EPL % NL == 0, "either whole heads or a part of one");
    float* const to = &s_acc[wave][held / EPL][at % TPR * EPL + held % EPL];
    if (TPR > 8 || (at & 8) == 0) {
#pragma unroll
      for (int i = 0; i < NL; ++i) to[i / EPL * D + i % EPL] = sum[i];
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (TPR <= 16) l[g] = sum_across_rows(l[g]);
      if (TPR <= 32) l[g] = sum_across_halves(l[g]);
      if (lane == 0) {
        s_ml[wave][g][0] = m[g];
        s_ml[wave][g][1] = l[g];
      }
    }
  }
  __syncthreads();

  // combine the wavefronts; one thread per (head of the group, element)
  const DecodeArgs& e = reread_args();
  const bool merges = kMerges && e.arrivals != nullptr;
  const bool direct = kDirect || (merges && n_pieces == 1);  // the only piece: out and lse instead of a partial result
  for (int i = tid; i < G * D; i += kThreads) {
    const int g = i / D, d = i - g * D;
    float mn = -INFINITY;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) mn = fmaxf(mn, s_ml[w][g][0]);
    const float ms = safe_max(mn);
    float num = 0.f, den = 0.f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const float wgt = fast_exp2(s_ml[w][g][0] - ms);
      num += s_acc[w][g][d] * wgt;
      den += s_ml[w][g][1] * wgt;
    }
    const int hq = hc * G + g;
    if (direct) {
      const float lse_nat = (mn + log2f(den)) * kLn2;
      E::store(e.out + b * e.os_b + hq * e.os_h + d * sizeof(typename E::type), sink_gate<E>(num / den, lse_nat, e.sinks, hq));
      if (d == 0) e.lse[static_cast<int64_t>(b) * e.Hq + hq] = lse_nat;
    } else {
      const int64_t p = hq * part_mul + part_add;
      if (merges) {
        publish(e.ws_acc + p * D + d, num);
        if (d == 0) publish2(e.ws_ml + p * 2, mn, den);
      } else {
        e.ws_acc[p * D + d] = num;
        if (d == 0) {
          e.ws_ml[p * 2] = mn;
          e.ws_ml[p * 2 + 1] = den;
        }
      }
    }
  }
  if constexpr (kMerges) {
    if (merges && split == 0) clear_next_counter(e, b);
    __shared__ int s_last;
    __shared__ __attribute__((aligned(16))) float s_part[4 * 64 * 4];
    if (merges && !direct && last_to_arrive(b, n_pieces, &s_last)) merge_splits<E, D>(b, part_mul, part_add - split, n_pieces, G, s_part);
  }
  };  // piece

  if constexpr (kPieces) {
    walk_pieces<min_part(ROWB)>(a, piece);
  } else if constexpr (!kFlat) {
    walk_split<kMerges>(a, piece);
  } else {
    __shared__ int s_start[kFlatMaxB + 1];
    walk_even_cut<kThreads>(a, s_start, s_pages, piece);
  }
}

// Writes the plan of a step (see kPlanInts): one wavefront per chunk of the even cut repeats the cut the
// main kernel would make and looks the page ids of its pieces up.
__global__ __launch_bounds__(64) void paged_decode_plan_kernel(const DecodeArgs a) {
  __shared__ int s_start[kFlatMaxB + 1];
  flat_starts(a, s_start);
  __syncthreads();
  const int c = blockIdx.x;
  int* rec = a.plan + static_cast<int64_t>(c) * kPlanInts;
  int* pages = rec + kPlanRec;
  const int total = s_start[a.B];
  const int len = flat_chunk_len(total, a.n_chunks);
  const int64_t lo = static_cast<int64_t>(c) * len;
  const int64_t hi = lo + len < total ? lo + len : total;
  const int lane = threadIdx.x;
  const int64_t pool_pages = a.pool_pages;
  int n = 0, page_off = 0;
  bool ok = true;
  if (lo < total) {
    int b = 0;  // first sequence that ends after lo
    {
      int left = 0, right = a.B - 1;
      while (left < right) {
        const int mid = (left + right) >> 1;
        if (s_start[mid + 1] > lo) right = mid; else left = mid + 1;
      }
      b = left;
    }
    for (; b < a.B && s_start[b] < hi; ++b) {
      const int begin = s_start[b], end = s_start[b + 1];
      if (end == begin) continue;
      const int t0 = lo > begin ? static_cast<int>(lo - begin) : 0;
      const int part = static_cast<int>((hi < end ? hi : end) - begin) - t0;
      int64_t L = fp::load_index(a.input_pos, b, a.pos_i64) + 1;
      int64_t trow = a.batch_idx[b];
      const int64_t L_raw = L > INT32_MAX ? INT32_MAX : L < INT32_MIN ? INT32_MIN : L;
      if (trow < 0 || trow >= a.max_batch) {
        trow = -1;
        L = 0;
      }
      if (L > a.max_context) L = a.max_context;
      if (n >= kPlanPieces) {
        ok = false;
        break;
      }
      int nblk = 0;
      if (t0 < L) {  // the pages of tokens t0 .. min(L, t0 + part) - 1, as the main kernel stages them
        const int t1 = L < t0 + part ? L : t0 + part;
        int64_t blk0, blk_last;
        int off_unused;
        a.pd.split(t0, blk0, off_unused);
        a.pd.split(t1 - 1, blk_last, off_unused);
        nblk = static_cast<int>(blk_last - blk0) + 1;
        if (page_off + nblk > kPlanPages) {
          ok = false;
          break;
        }
        for (int i = lane; i < nblk; i += 64) {
          int64_t page = 0;
          if (blk0 + i < a.n_pages) page = a.page_table[static_cast<int64_t>(trow) * a.pt_row_stride + blk0 + i];
          if (page < 0 || page >= pool_pages) page = 0;  // not a page of the pool
          pages[page_off + i] = static_cast<int>(page);
        }
      }
      if (lane == 0) {
        int* r = rec + 4 + 6 * n;
        r[0] = b;
        r[1] = t0;
        r[2] = part;
        r[3] = static_cast<int>(L_raw);
        r[4] = static_cast<int>(trow);
        r[5] = page_off;
      }
      page_off += nblk;
      ++n;
    }
  }
  if (lane == 0) {
    rec[0] = ok ? n : -1;
    rec[1] = a.B;
    rec[2] = a.n_chunks;
    rec[3] = a.max_context;
  }
  if (c == 0) {
    uint32_t hash = 0;
    for (int i = lane; i < a.B; i += 64)
      hash += plan_hash_term(i, fp::load_index(a.input_pos, i, a.pos_i64) + 1, a.batch_idx[i]);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) hash += __shfl_xor(hash, off);
    if (lane == 0) rec[kPlanHashAt] = static_cast<int>(hash);
  }
}

// ---- cross-split merge ------------------------------------------------------
// One batch of kBatch consecutive splits of a partial row, as this lane holds it.
template <int D, int kBatch>
struct SplitBatch {
  float m[kBatch], l[kBatch], acc[kBatch][(D + 63) / 64];
};

// Requests the splits base .. base + kBatch - 1 (those below `limit`) of partial row p0.
template <int D, int kBatch>
__device__ __forceinline__ void load_batch(const DecodeArgs& a, int64_t p0, int base, int limit, int64_t row_stride,
                                           SplitBatch<D, kBatch>& t) {
  constexpr int DPL = (D + 63) / 64;
#pragma unroll
  for (int s = 0; s < kBatch; ++s) {
    const bool on = base + s < limit;
    const int64_t p = p0 + (on ? base + s : 0) * row_stride;
    t.m[s] = on ? a.ws_ml[p * 2] : -INFINITY;
    t.l[s] = on ? a.ws_ml[p * 2 + 1] : 0.f;
#pragma unroll
    for (int j = 0; j < DPL; ++j) {
      const int d = (threadIdx.x & 63) + j * 64;
      t.acc[s][j] = (on && d < D) ? a.ws_acc[p * D + d] : 0.f;
    }
  }
}

// Folds the splits of a batch that lie below ns into the running state (m_run, den, num) of this lane.  A batch
// that was requested before ns was known may hold rows of splits the sequence does not have (whatever the
// workspace held): they are dropped here by selects and never enter the arithmetic.
template <int D, int kBatch>
__device__ __forceinline__ void fold_batch(SplitBatch<D, kBatch>& t, int base, int ns, float& m_run, float& den,
                                           float (&num)[(D + 63) / 64]) {
  constexpr int DPL = (D + 63) / 64;
  float mn = m_run;
#pragma unroll
  for (int s = 0; s < kBatch; ++s) {
    if (base + s >= ns) {
      t.m[s] = -INFINITY;
      t.l[s] = 0.f;
#pragma unroll
      for (int j = 0; j < DPL; ++j) t.acc[s][j] = 0.f;
    }
    mn = fmaxf(mn, t.m[s]);
  }
  const float ms = safe_max(mn);
  const float keep = fast_exp2(m_run - ms);  // 0 while the state is empty
  den *= keep;
#pragma unroll
  for (int j = 0; j < DPL; ++j) num[j] *= keep;
#pragma unroll
  for (int s = 0; s < kBatch; ++s) {
    const float wgt = fast_exp2(t.m[s] - ms);
    den += t.l[s] * wgt;
#pragma unroll
    for (int j = 0; j < DPL; ++j) num[j] += t.acc[s][j] * wgt;
  }
  m_run = mn;
}

// Folds the splits first, first + stride, ... (kBatch consecutive splits each time, below ns) of partial
// row p0 into the running state (m_run, den, num) of this lane; scores are in log2 units.
template <int D, int kBatch>
__device__ __forceinline__ void merge_batches(const DecodeArgs& a, int64_t p0, int first, int stride, int ns, float& m_run,
                                              float& den, float (&num)[(D + 63) / 64], int64_t row_stride = 1) {
  for (int base = first; base < ns; base += stride) {
    SplitBatch<D, kBatch> t;
    load_batch<D, kBatch>(a, p0, base, ns, row_stride, t);
    fold_batch<D, kBatch>(t, base, ns, m_run, den, num);
  }
}

// Normalises, gates and stores one merged row (lane = output elements lane, lane + 64, ...).
template <typename E, int D>
__device__ __forceinline__ void finish_merge(const DecodeArgs& a, int b, int hq, bool any, float mn, float den,
                                             const float (&num)[(D + 63) / 64]) {
  const float lse_nat = any ? (mn + log2f(den)) * kLn2 : -INFINITY;
#pragma unroll
  for (int j = 0; j < (D + 63) / 64; ++j) {
    const int d = (threadIdx.x & 63) + j * 64;
    if (d >= D) continue;
    const float o = any ? num[j] / den : 0.f;
    E::store(a.out + b * a.os_b + hq * a.os_h + d * sizeof(typename E::type), sink_gate<E>(o, lse_nat, a.sinks, hq));
  }
  if ((threadIdx.x & 63) == 0) a.lse[static_cast<int64_t>(b) * a.Hq + hq] = lse_nat;
}

template <typename E, int D>
__global__ __launch_bounds__(64) void paged_decode_merge_kernel(const DecodeArgs a) {
  const int hq = blockIdx.x;
  const int b = blockIdx.y;
  const int64_t p0 = (static_cast<int64_t>(b) * a.Hq + hq) * a.n_splits;

  // The kernel is a chain of memory latencies, so the first kBatch splits are requested together with the
  // sequence's position, by the launch's split count: the partials of splits this sequence does not have
  // are dropped by selects once its length is known and never enter the arithmetic.
  constexpr int kBatch = 8;
  constexpr int DPL = (D + 63) / 64;  // output elements per lane
  int64_t L = fp::load_index(a.input_pos, b, a.pos_i64) + 1;
  const int64_t trow = a.batch_idx[b];
  SplitBatch<D, kBatch> first;
  load_batch<D, kBatch>(a, p0, 0, a.n_splits, 1, first);
  if (trow < 0 || trow >= a.max_batch) L = 0;
  if (L > a.max_context) L = a.max_context;
  const int part = split_part(static_cast<int>(L), a.split_tokens);
  const int ns = L <= 0 ? 0 : static_cast<int>((L + part - 1) / part);

  // The same lane keeps a running (maximum, denominator, numerator) over batches of kBatch splits, every load
  // of a batch requested at once.  The wide variant of this kernel spreads the batches over several wavefronts.
  float m_run = -INFINITY, den = 0.f, num[DPL];
#pragma unroll
  for (int j = 0; j < DPL; ++j) num[j] = 0.f;
  if (ns > 0) fold_batch<D, kBatch>(first, 0, ns, m_run, den, num);
  merge_batches<D, kBatch>(a, p0, kBatch, kBatch, ns, m_run, den, num);
  finish_merge<E, D>(a, b, hq, ns > 0, m_run, den, num);
}

// Cross-split merge after the even cut: sequence b has one partial result per chunk it touches, in
// workspace rows (chunk + b) * Hq + hq.
template <typename E, int D>
__global__ __launch_bounds__(64) void paged_decode_merge_flat_kernel(const DecodeArgs a) {
  constexpr int DPL = (D + 63) / 64;
  const int hq = blockIdx.x;
  const int b = blockIdx.y;
  const int lane = threadIdx.x;
  int before = 0, total = 0, mine = 0;  // rounded lengths: of the sequences before b, of all, of b
  // the plan's launch values and hash, if the split-K pass had a plan: requested with the positions
  int planned[4] = {0, 0, 0, 0};
  if (a.plan) {
    planned[0] = a.plan[1];
    planned[1] = a.plan[2];
    planned[2] = a.plan[3];
    planned[3] = a.plan[kPlanHashAt];
  }
  uint32_t hash = 0;
  for (int i = lane; i < a.B; i += 64) {
    int64_t L = fp::load_index(a.input_pos, i, a.pos_i64) + 1;
    const int64_t trow = a.batch_idx[i];
    hash += plan_hash_term(i, L, trow);
    if (trow < 0 || trow >= a.max_batch || L < 0) L = 0;
    if (L > a.max_context) L = a.max_context;
    const int Lr = (static_cast<int>(L) + 63) & ~63;
    total += Lr;
    if (i < b) before += Lr;
    if (i == b) mine = Lr;
  }
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    total += __shfl_xor(total, off);
    before += __shfl_xor(before, off);
    mine += __shfl_xor(mine, off);
    hash += __shfl_xor(hash, off);
  }
  // the split-K pass followed a plan (same acceptance test as there) that was made from other positions or slots
  const bool stale = a.plan && planned[0] == a.B && planned[1] == a.n_chunks && planned[2] == a.max_context &&
                     static_cast<uint32_t>(planned[3]) != hash;
  const int len = flat_chunk_len(total, a.n_chunks);
  const int c_first = before / len;
  const int ns = mine > 0 ? (before + mine - 1) / len - c_first + 1 : 0;
  float m_run = -INFINITY, den = 0.f, num[DPL];
#pragma unroll
  for (int j = 0; j < DPL; ++j) num[j] = 0.f;
  merge_batches<D, 8>(a, static_cast<int64_t>(c_first + b) * a.Hq + hq, 0, 8, ns, m_run, den, num, a.Hq);
  if (stale) den = __builtin_nanf("");  // every row of out and lse: not a result
  finish_merge<E, D>(a, b, hq, ns > 0 || stale, m_run, den, num);
}

// Cross-split merge for launches with many splits per sequence: kMergeWideWaves wavefronts per
// (sequence, query head) take the batches of splits round-robin and combine their states through LDS.
constexpr int kMergeWideWaves = 8;
constexpr int kMergeWideSplits = 16;  // launches with more splits than this use it

template <typename E, int D>
__global__ __launch_bounds__(kMergeWideWaves * 64) void paged_decode_merge_wide_kernel(const DecodeArgs a) {
  constexpr int kBatch = 8;
  constexpr int DPL = (D + 63) / 64;
  const int hq = blockIdx.x;
  const int b = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int64_t p0 = (static_cast<int64_t>(b) * a.Hq + hq) * a.n_splits;
  __shared__ float s_m[kMergeWideWaves], s_den[kMergeWideWaves], s_num[kMergeWideWaves][DPL * 64];

  // The kernel is a chain of memory latencies: the position of the sequence and this wavefront's first batch of
  // partial rows are requested together (the batch by the launch's split count; what the sequence does not
  // have is dropped once its length is known), the later batches of a launch of more than 64 splits after it.
  int64_t L = fp::load_index(a.input_pos, b, a.pos_i64) + 1;
  const int64_t trow = a.batch_idx[b];
  SplitBatch<D, kBatch> first;
  load_batch<D, kBatch>(a, p0, wave * kBatch, a.n_splits, 1, first);
  if (trow < 0 || trow >= a.max_batch) L = 0;
  if (L > a.max_context) L = a.max_context;
  const int part = split_part(static_cast<int>(L), a.split_tokens);
  const int ns = L <= 0 ? 0 : static_cast<int>((L + part - 1) / part);

  float m_run = -INFINITY, den = 0.f, num[DPL];
#pragma unroll
  for (int j = 0; j < DPL; ++j) num[j] = 0.f;
  if (wave * kBatch < ns) fold_batch<D, kBatch>(first, wave * kBatch, ns, m_run, den, num);
  merge_batches<D, kBatch>(a, p0, (wave + kMergeWideWaves) * kBatch, kMergeWideWaves * kBatch, ns, m_run, den, num);
  if (lane == 0) {
    s_m[wave] = m_run;
    s_den[wave] = den;
  }
#pragma unroll
  for (int j = 0; j < DPL; ++j) s_num[wave][j * 64 + lane] = num[j];
  __syncthreads();
  if (wave != 0) return;
  float mn = -INFINITY;
#pragma unroll
  for (int w = 0; w < kMergeWideWaves; ++w) mn = fmaxf(mn, s_m[w]);
  const float ms = safe_max(mn);
  den = 0.f;
#pragma unroll
  for (int j = 0; j < DPL; ++j) num[j] = 0.f;
#pragma unroll
  for (int w = 0; w < kMergeWideWaves; ++w) {
    const float wgt = fast_exp2(s_m[w] - ms);  // 0 for a wavefront that had no split
    den += s_den[w] * wgt;
#pragma unroll
    for (int j = 0; j < DPL; ++j) num[j] += s_num[w][j * 64 + lane] * wgt;
  }
  finish_merge<E, D>(a, b, hq, ns > 0, mn, den, num);
}

constexpr int kPhasePartial = 1;
constexpr int kPhaseMerge = 2;
constexpr int kPhasePlan = 4;  // alone: write the step's plan instead of launching the passes

int n_splits_for(int max_context, int split_tokens) {
  const int n = (max_context + split_tokens - 1) / split_tokens;
  return n < 1 ? 1 : n;
}

// Split length of a launch that goes split by split.  Largest split (fewest partials to merge, least per-workgroup
// overhead) that still yields enough workgroups when every sequence is at max_context.  Enough is about 2048 (8 per CU)
// for a batch whose sequences alone give every CU two workgroups: their lengths differ, and small pieces even that out.
// A small batch wants larger pieces: from 512 workgroups (4 * B * Hc in between) the pass no longer gets
// faster, and every further split is one more partial result to merge.
int plain_split_tokens(int B, int Hc, int max_context) {
  int64_t target = 4 * static_cast<int64_t>(B) * Hc;
  target = target < 512 ? 512 : target > 2048 ? 2048 : target;
  int split = 2048;
  while (split > 128 && static_cast<int64_t>(B) * Hc * ((max_context + split - 1) / split) < target) split >>= 1;
  return split;
}

// Chunks per cache head of the even cut: two per CU.
int flat_chunks(int Hc) { return 2 * fp::compute_units() / Hc; }

// Whether the even cut can take a launch at all: the lengths fit LDS, the flat axis is int, a chunk's pages fit the table.
bool even_cut_fits(int Hc, int B, int max_context, int page_size) {
  const int64_t tokens = static_cast<int64_t>(B) * (max_context + 64), chunks = flat_chunks(Hc);
  return chunks >= 1 && B <= kFlatMaxB && tokens < (1ll << 30) && (tokens / chunks + 128) / page_size + 2 <= kMaxSplitPages;
}

// Whether a launch on this side of even_cut_line is cut evenly all the same: its splits are long (1024 tokens or more, or eight
// of 512), so that sequences much shorter than max_context leave CUs idle, and the cut makes at most eight pieces of a
// sequence, which the merge pass (one wavefront per row) takes in one batch.  us a layer split by split / cut evenly, 16 q / 8 kv
// heads, D 128: limit 8192, 300 to 3000 tokens, 8, 12, 16 and 24 sequences 22.4 / 19.5, 28.3 / 24.1, 35.4 / 27.1 and 43.2 / 35.8, 4000 to
// 8000 tokens 40.4 / 39.6, 58.9 / 56.8, 69.7 / 69.2 and 107 / 100; limit 4096, 8 sequences of 64 to 300, 100 to 700 and 300 to 1500 tokens
// 12.6 / 9.9, 14.3 / 11.6 and 14.9 / 15.8, 10 of 100 to 3900 25.7 / 22.8; the price is paid close to the limit, 8 sequences of 3500 to
// 4000 tokens 26.6 / 30.4, and by many short sequences with one query head per cache head: limit 8192, 32 rows, 24 of them of 239 to 459
// tokens, 8 heads 16.5 / 16.9 (a single layer, without the step's plan, 20.1 / 22.2), 31 of 149 to 422, 4 heads 12.4 / 12.8; 8 and 16
// of 149 to 422, 16 q / 8 kv heads 12.9 / 10.8 and 14.7 / 13.8, 48 of 300 to 1500, 8 q / 4 kv heads 29.4 / 25.0.  With shorter splits there is no gain: limit 1024, 16 sequences (256 tokens) 15.5 / 17.5; limit 2048, 16
// sequences (four of 512) 29.2 / 31.4.  Nor with more pieces: one sequence of 12000 tokens 17.1 / 23.1, three of 300 to 3000 12.5 / 14.9.
bool even_cut_pays(int Hc, int B, int max_context, int page_size) {
  const int split = plain_split_tokens(B, Hc, max_context);
  const int n = n_splits_for(max_context, split);
  return n > 1 && (split >= 1024 || (split >= 512 && n >= 8)) && flat_chunks(Hc) <= 8 * static_cast<int64_t>(B) &&
         even_cut_fits(Hc, B, max_context, page_size);
}

// Chunks per cache head of the even cut of a launch, 0 where it goes split by split.  The workspace of its splits has a row
// per (chunk + sequence), and a launch of more than `line` workgroups is always cut.
int even_cut_chunks(int Hc, int B, int n_splits, int max_context, int page_size, int line) {
  const int chunks = flat_chunks(Hc);
  if (!even_cut_fits(Hc, B, max_context, page_size) || static_cast<int64_t>(B) * (n_splits - 1) < chunks) return 0;
  return static_cast<int64_t>(Hc) * B * n_splits > line || even_cut_pays(Hc, B, max_context, page_size) ? chunks : 0;
}

// Splits of all sequences together, about, of a launch with arrival counters that goes piece by piece (walk_pieces): two workgroups to a
// CU.  0 where it goes another way.  us a layer split by split or, with its plan, cut evenly / piece by piece:
//                                              16 q / 8 kv, D 128   16 K and shared V heads   D 64, f16    4 x 8 q / 8 kv, D 64   8 heads, D 64, f32
//   limit 8192, 4 of 100 to 700                     11.5 / 8.8            12.8 / 9.3          10.0 / 8.7        8.6 / 7.9             9.3 / 7.3
//   limit 8192, 5 of 3000 to 8000                   28.4 / 23.9           36.4 / 31.4         18.3 / 16.0      18.9 / 15.6           25.2 / 21.9
//   limit 4096, 8 of 300 to 1500                    15.9 / 12.4           18.0 / 13.9         14.5 / 10.9      14.2 / 10.8           13.2 / 10.8
//   limit 8192, 16 of 350 to 4620                   33.4 / 30.3           44.1 / 41.1         22.4 / 19.5      22.1 / 18.3           30.4 / 28.4
//   limit 1024, 48 of 64 to 500                     20.6 / 16.2           25.4 / 20.4         18.5 / 13.0      17.7 / 14.4           17.1 / 14.5
// The price is paid where the lengths are close to the limit and fill the grid split by split anyway: limit 8192, 4 of 8000 26.6 / 27.4,
// 36.3 / 36.5, 17.3 / 18.1, 16.5 / 17.3 and 24.7 / 25.6.  The lines: with fewer workgroup heads x sequences the merge is on fewer
// workgroups than there are rows to hide it behind (8 heads, one of 711 tokens 8.0 / 8.0, two of 300 to 6000 11.6 / 12.1); a grid of up to four splits that the
// CUs hold at once has few idle workgroups (limit 1024, 16 of 900 to 1000 16.9 / 18.1, of 100 to 900 13.2 / 13.4); and with more
// tokens or sequences the remainders, up to B pieces, run behind the others (limit 8192, 24 of 4000 to 8000 96.7 / 99.8, 60 of these 228 / 261; limit 4096, 24 of
// 64 to 4000 41.2 / 37.9, 32 of 300 to 4000 51.1 / 51.3; limit 2048, 32 of 300 to 2000 33.7 / 31.4; limit 1024, 60 of 100 to 1000 31.8 / 31.8
// and in a step of 28 layers 908 / 920 us).  The line at limit 8192 is that of the long ones; shorter sequences would gain on its other side, too (cut evenly /
// piece by piece, a layer of 28: 17 of 64 to 500 14.9 / 11.1, of 300 to 3000 27.0 / 24.8, of 64 to 8000 51.2 / 48.7; 24 of these 15.4 / 12.0, 34.4 / 32.9 and 69.4 / 70.5,
// D 64, f16 13.9 / 10.7 and 23.7 / 21.0; limit 16384, 12 of 64 to 500 11.5 / 9.4).  The step's plan does not know which way its launches go: one that goes piece by piece reads none.
int merged_pieces(int Hc, int B, int n_splits, int max_context, int page_size) {
  const int64_t groups = static_cast<int64_t>(Hc) * B, tokens = static_cast<int64_t>(B) * (max_context + 64), two = 2 * fp::compute_units();
  if (B < 3 || B > 48 || groups < 32 || n_splits < 2 || (n_splits <= 4 && groups * n_splits <= two) || tokens >= 1 << 22 ||
      groups * max_context > (B <= 24 ? 1 << 20 : 1 << 19))
    return 0;
  int64_t pieces = two / Hc;
  if (pieces > kMostPieces * B) pieces = kMostPieces * B;
  if (pieces > static_cast<int64_t>(B) * (n_splits - 1)) pieces = static_cast<int64_t>(B) * (n_splits - 1);  // a row per (piece + sequence)
  if (pieces < 4) return 0;
  const int64_t longest = tokens / pieces * 3 / 2 + 512;  // walk_pieces: (x + 64) * 17 / 16 + 64, four times
  return longest / page_size + 2 <= kMaxSplitPages ? static_cast<int>(pieces) : 0;
}

// Workgroups to a CU beyond which a launch is always cut evenly.  Numbers, so that a kernel that needs fewer registers does not move
// the line: as many as the even-cut kernels' registers let a CU hold when the sweeps at even_cut_pays and merged_pieces were made.  Since
// then a CU holds one more of the 16-bit kernels for a cache of one K head per query head with V in pairs and whole pages, and in fp32 of most with two
// and four heads (at head_dim 64 and two heads a fourth).  Between the two numbers, cut evenly / split by split, us a layer in a graph of the
// plan and four layers (about 1 us of it the plan): bf16, V in pairs, D 128: limit 4096, 8 heads, 5 sequences of 200 to 1600, 400 to
// 4096 and 3500 to 4096 tokens 14.5 / 12.2, 21.7 / 22.2 and 28.1 / 26.7; limit 512, 24 of 25 to 200 and of 50 to 500 12.5 / 11.0 and 17.0 / 15.3; limit
// 8192, 3 of 800 to 8192, 16 and 4 heads 27.9 / 27.9 and 18.1 / 12.4.  fp32 the same 19.7 / 17.1, 29.6 / 35.2 and 44.8 / 45.9; 14.6 / 14.9 and 22.5 /
// 23.4; 43.8 / 47.3 and 23.4 / 17.8.  fp32, four heads: limit 8192, 16 heads, 3 of 400 to 3200 21.0 / 23.1; limit 512, 12 of 50 to 500 20.6 / 18.1.
// fp32, D 64, two heads: limit 512, 8 heads, 30 of 50 to 500 15.3 / 12.5; limit 8192, 4 heads, 7 of 800 to 8192 20.2 / 17.5.  In fp32 at D 128 either side is
// the better one somewhere; in 16 bits and at D 64 split by split mostly is, and a line one higher there would be worth these figures.
template <typename E, int D, int G, bool kPerHeadK>
constexpr int even_cut_line(bool aligned) {
  const bool narrow = sizeof(typename E::type) == 2;
  if (kPerHeadK) return narrow ? (G == 2 && !aligned ? 3 : 2) : (D == 128 && aligned ? 2 : 3);
  return G == 1 ? 4 : G == 2 ? 3 : G == 4 || (D == 64 && aligned) ? 2 : 1;
}

// Launches with four or more query heads per cache head in a 16-bit type run on the matrix cores.  us a layer on the vector
// pipe / on the matrix cores, 8 cache heads, bf16, eight query heads per cache head: one sequence of 711 tokens 15.7 / 11.1, 16 of 100
// to 600 31.7 / 18.8, 64 of 1000 to 4000 204 / 117; four: 12.0 / 10.7, 22.6 / 17.5 and 120 / 112, at head_dim 64 11.9 / 9.5, 17.2 / 14.4
// and 70.2 / 63.0; f16 the same.  With two the vector pipe is not the limit.
template <typename E, int G, bool kPerHeadK>
constexpr bool on_matrix_cores() { return sizeof(typename E::type) == 2 && !kPerHeadK && G >= 4; }

template <typename E, int D, int G, bool kPerHeadK = false>
void launch_decode(const DecodeArgs& a0, int B, int phases, hipStream_t st) {
  DecodeArgs a = a0;
  if (!merges_itself(G, D)) a.arrivals = nullptr;
  dim3 grid(a.Hc, B, a.n_splits);  // a.Hc = workgroups per sequence and split: cache heads, or groups of G heads
  // rows per wavefront iteration: the loads in flight times 64 / (D * elem / 16) rows each
  const int chunk_rows = decode_loads_in_flight(G, kPerHeadK) * 64 / (D * static_cast<int>(sizeof(typename E::type)) / 16);
  const bool aligned = a.pd.shift >= 0 && a.pd.page_size % chunk_rows == 0;
  // the split-K pass, by the kernel that serves this instance
  auto split_k_pass = [&](auto direct, auto flat, auto pieces, dim3 g, const DecodeArgs& args) {
    constexpr bool kDirect = decltype(direct)::value, kFlat = decltype(flat)::value, kPieces = decltype(pieces)::value;
    if constexpr (on_matrix_cores<E, G, kPerHeadK>())
      launch_mfma(args, std::is_same<E, BF16>::value ? FP_DTYPE_BF16 : FP_DTYPE_F16, D, Cut{kDirect, kFlat, kPieces}, g, st);
    else if (aligned)
      hipLaunchKernelGGL((paged_decode_kernel<E, D, G, kDirect, true, kPerHeadK, kFlat, kPieces>), g, dim3(kThreads), 0, st, args);
    else
      hipLaunchKernelGGL((paged_decode_kernel<E, D, G, kDirect, false, kPerHeadK, kFlat, kPieces>), g, dim3(kThreads), 0, st, args);
  };
  if (a.n_splits == 1) {
    // one split covers every context: the partial pass writes out and lse itself
    if (!(phases & kPhasePartial)) return;  // also the plan phase: such a launch has no even cut
    split_k_pass(std::true_type{}, std::false_type{}, std::false_type{}, grid, a);
  } else {
    // Cut evenly: the work of a workgroup then follows from the lengths of the sequences and not from max_context,
    // which an engine sets to the longest sequence it may ever hold (16 padded rows of 350 to 4620 tokens under a
    // limit of 8192, 16 q heads / 8 kv heads with shared V: 57.4 us a layer split by split, one workgroup to a CU,
    // against 38.8 us; even_cut_pays has where it goes which way).  Two chunks
    // per CU, all of the same length, all resident from the start, so that every CU streams the same
    // number of rows (split by split, the CUs end up with loads 25 % apart at 64 sequences of 1 k to
    // 4 k tokens, and workgroups queue behind busy shader engines).  Measured at 64 sequences of 16 q /
    // 8 kv heads, bf16, % of 8 TB/s for the step with 1 / 2 / 3 / 4 chunks per CU and split by split:
    // D 128: 75.5 / 75.4 / 73.8 / 73.1 and 73.0; D 64: 67.2 / 68.3 / 68.1 / 63.7 and 67.1; 32 q heads:
    // 63.9 / 70.6 / 64.2 / 67.9 and 67.2; 16-token pages: 70.0 / 74.4 / 73.9 / 68.9 and 72.6.  fp32 with
    // two chunks per CU: D 128 80.7 against 78.4 split by split, D 64 76.9 against 76.1, 32 q heads 77.4
    // against 73.4 (the even-cut kernels are not held to 128 registers: two workgroups per CU do not need
    // it, and in fp32 it made them spill).  With the step's plan read by every workgroup the same sweep gives, in us per
    // step for 1 / 2 / 3 chunks per CU: D 128 110.4 / 111.3 / 112.2; D 64 61.7 / 61.3 / 62.1; page size 64, 32
    // sequences 89.2 / 90.9 / 90.4: two stays.
    int line;  // matrix cores: two to a CU, but few sequences want the third (640 / 752 / 896 workgroups, 64 q / 8 kv heads,
               // split by split / cut evenly: 15.1 / 17.9, 21.6 / 25.1 and 19.6 / 18.2 us)
    if constexpr (on_matrix_cores<E, G, kPerHeadK>())
      line = 3 * fp::compute_units();
    else
      line = even_cut_line<E, D, G, kPerHeadK>(aligned) * fp::compute_units();
    const int pieces = a.arrivals ? merged_pieces(a.Hc, B, a.n_splits, a.max_context, a.pd.page_size) : 0;
    DecodeArgs ap = a;
    ap.n_chunks = pieces;
    const int n_chunks = pieces > 0 ? 0 : even_cut_chunks(a.Hc, B, a.n_splits, a.max_context, a.pd.page_size, line);
    DecodeArgs af = a;
    af.B = B;
    af.n_chunks = n_chunks;
    if (phases & kPhasePlan) {
      // the plan of a step serves the even cut only; a launch that goes split by split needs none
      if (a.plan && n_chunks > 0) hipLaunchKernelGGL(paged_decode_plan_kernel, dim3(n_chunks), dim3(64), 0, st, af);
      return;
    }
    if (phases & kPhasePartial) {
      if (n_chunks > 0)
        split_k_pass(std::false_type{}, std::true_type{}, std::false_type{}, dim3(a.Hc, n_chunks), af);
      else if (pieces == 0)
        split_k_pass(std::false_type{}, std::false_type{}, std::false_type{}, grid, a);
      else if constexpr (merges_itself(G, D))
        split_k_pass(std::false_type{}, std::false_type{}, std::true_type{}, dim3(a.Hc, pieces + B), ap);
    }
    if ((phases & kPhaseMerge) && (n_chunks > 0 || !a.arrivals)) {
      if (n_chunks > 0)
        hipLaunchKernelGGL((paged_decode_merge_flat_kernel<E, D>), dim3(a.Hq, B), dim3(64), 0, st, af);
      else if (a.n_splits > kMergeWideSplits)
        hipLaunchKernelGGL((paged_decode_merge_wide_kernel<E, D>), dim3(a.Hq, B), dim3(kMergeWideWaves * 64), 0, st, a);
      else
        hipLaunchKernelGGL((paged_decode_merge_kernel<E, D>), dim3(a.Hq, B), dim3(64), 0, st, a);
    }
  }
}

template <typename E, int D>
int dispatch_group(const DecodeArgs& a, int B, int phases, int kv_rep, hipStream_t st) {
  if (kv_rep > 1) {  // a.Hc already counts groups of kv_rep heads
    switch (kv_rep) {
      case 2: launch_decode<E, D, 2, true>(a, B, phases, st); return FP_OK;
      case 4: launch_decode<E, D, 4, true>(a, B, phases, st); return FP_OK;
      default: return fp::fail(FP_ERR_UNSUPPORTED, "fp_paged_decode: kv_rep = %d (supported: 1, 2, 4)", kv_rep);
    }
  }
  switch (a.Hq / a.Hc) {
    case 1: launch_decode<E, D, 1>(a, B, phases, st); return FP_OK;
    case 2: launch_decode<E, D, 2>(a, B, phases, st); return FP_OK;
    case 4: launch_decode<E, D, 4>(a, B, phases, st); return FP_OK;
    case 8: launch_decode<E, D, 8>(a, B, phases, st); return FP_OK;
    default: return fp::fail(FP_ERR_UNSUPPORTED, "fp_paged_decode: Hq/Hc = %d (supported: 1, 2, 4, 8)", a.Hq / a.Hc);
  }
}

template <typename E>
int dispatch_dim(const DecodeArgs& a, int B, int D, int phases, int kv_rep, hipStream_t st) {
  switch (D) {
    case 64: return dispatch_group<E, 64>(a, B, phases, kv_rep, st);
    case 128: return dispatch_group<E, 128>(a, B, phases, kv_rep, st);
    default: return fp::fail(FP_ERR_UNSUPPORTED, "fp_paged_decode: head_dim %d (supported: 64, 128)", D);
  }
}

int default_split_tokens(int B, int Hc, int max_context, int page_size) {
  int split = plain_split_tokens(B, Hc, max_context);
  if (even_cut_pays(Hc, B, max_context, page_size))  // the workspace has B rows per split: enough of them for the cut
    while (split > 64 && static_cast<int64_t>(B) * (n_splits_for(max_context, split) - 1) < flat_chunks(Hc)) split >>= 1;
  while (split / page_size + 2 > kMaxSplitPages) split >>= 1;
  return split < 64 ? 64 : split;
}

}  // namespace

extern "C" int32_t fp_paged_decode_default_split(int32_t B, int32_t Hc, int32_t max_context, int32_t page_size) {
  if (B <= 0 || Hc <= 0 || max_context < 0 || page_size <= 0)
    return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode_default_split: bad dimension");
  return default_split_tokens(B, Hc, max_context, page_size);
}

extern "C" int32_t fp_paged_decode_step_pieces(int32_t B, int32_t Hq, int32_t Hc, int32_t kv_rep, int32_t D, int32_t max_context,
                                               int32_t page_size, int32_t split_tokens) {
  if (B <= 0 || Hc <= 0 || Hq < Hc || kv_rep <= 0 || D <= 0 || max_context < 0 || page_size <= 0 || split_tokens < 0)
    return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode_step_pieces: bad dimension");
  if (Hq % Hc || (kv_rep > 1 && (Hc != Hq || Hq % kv_rep)) || split_tokens % 64)  // as the launch itself asks
    return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode_step_pieces: Hq = %d, Hc = %d, kv_rep = %d, split_tokens = %d is no launch",
                    Hq, Hc, kv_rep, split_tokens);
  const int wg_heads = kv_rep > 1 ? Hq / kv_rep : Hc;
  const int split = split_tokens ? split_tokens : default_split_tokens(B, wg_heads, max_context, page_size);
  if (!merges_itself(Hq / wg_heads, D)) return 0;
  return merged_pieces(wg_heads, B, n_splits_for(max_context, split), max_context, page_size);
}

extern "C" int64_t fp_paged_decode_workspace_bytes(int32_t B, int32_t Hq, int32_t D, int32_t max_context,
                                                   int32_t split_tokens) {
  if (B < 0 || Hq <= 0 || D <= 0 || max_context < 0 || split_tokens <= 0)
    return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode_workspace_bytes: bad dimension");
  if (split_tokens % 64) return fp::fail(FP_ERR_INVALID_ARGUMENT, "split_tokens must be a multiple of 64");
  const int64_t ns = n_splits_for(max_context, split_tokens);
  if (ns == 1) return 0;
  return static_cast<int64_t>(B) * Hq * ns * (D + 2) * static_cast<int64_t>(sizeof(float));
}

extern "C" int64_t fp_paged_decode_workspace_bytes_up_to(int32_t max_B, int32_t Hq, int32_t Hc, int32_t D,
                                                         int32_t max_context, int32_t page_size) {
  if (max_B < 0 || Hq <= 0 || Hc <= 0 || D <= 0 || max_context < 0 || page_size <= 0)
    return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode_workspace_bytes_up_to: bad dimension");
  int64_t rows = 0;
  for (int B = 1; B <= max_B; ++B) {
    const int ns = n_splits_for(max_context, default_split_tokens(B, Hc, max_context, page_size));
    if (ns > 1 && static_cast<int64_t>(B) * ns > rows) rows = static_cast<int64_t>(B) * ns;
  }
  return rows * Hq * (D + 2) * static_cast<int64_t>(sizeof(float));
}

namespace {

// A plan has a record per chunk of the even cut; a launch has at most two chunks per CU and cache head.
int64_t plan_buffer_bytes() { return 2LL * fp::compute_units() * kPlanInts * static_cast<int64_t>(sizeof(int)); }

struct NewRows {
  const void* k;
  const void* v;
  int64_t k_stride_b, k_stride_h, v_stride_b, v_stride_h;  // elements
};

int decode_entry(int phases, const NewRows* fresh, const void* q, int64_t q_stride_b, int64_t q_stride_h, const void* pool_k,
                 const void* pool_v, const int64_t* page_table, int64_t pt_row_stride,
                 const int64_t* batch_idx, const void* input_pos, int pos_index_type,
                 void* out, int64_t out_stride_b, int64_t out_stride_h, float* lse, const float* sinks,
                 void* workspace, int64_t workspace_bytes, int32_t B, int32_t Hq, int32_t Hc, int32_t kv_rep,
                 int32_t D, int32_t page_size, int32_t n_pages, int32_t max_batch,
                 int64_t n_slots, int32_t max_context, int32_t split_tokens, float scale,
                 int dtype, void* plan, int64_t plan_bytes, void* stream,
                 int32_t* arrivals = nullptr, int32_t* next_arrivals = nullptr, int64_t arrivals_bytes = 0) {
  const bool plan_only = phases == kPhasePlan;  // q, out, lse and the workspace are not touched then
  const int eb = fp::elem_bytes(dtype);
  if (eb == 0) return fp::fail(FP_ERR_UNSUPPORTED, "fp_paged_decode: unknown dtype %d", dtype);
  if (B < 0 || Hq <= 0 || Hc <= 0 || D <= 0 || page_size <= 0 || n_pages <= 0 || max_batch <= 0 ||
      n_slots <= 0 || max_context < 0 || split_tokens < 0)
    return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode: bad dimension");
  if (Hq % Hc) return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode: Hq=%d not a multiple of Hc=%d", Hq, Hc);
  if (kv_rep < 1) return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode: kv_rep must be at least 1");
  if (kv_rep > 1 && (Hc != Hq || Hq % kv_rep))
    return fp::fail(FP_ERR_INVALID_ARGUMENT,
                    "fp_paged_decode: kv_rep = %d needs a cache with one head per query head (Hc = Hq = %d here %d) "
                    "and Hq a multiple of kv_rep", kv_rep, Hq, Hc);
  const int wg_heads = kv_rep > 1 ? Hq / kv_rep : Hc;  // workgroups per sequence and split
  if (n_slots < page_size)
    return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode: n_slots smaller than one page");
  if (max_context > static_cast<int64_t>(n_pages) * page_size)
    return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode: max_context exceeds the page table width");
  if (pos_index_type != FP_INDEX_I32 && pos_index_type != FP_INDEX_I64)
    return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode: bad pos_index_type");
  if (B > 65535 || Hc > 65535 || Hq > 65535)
    return fp::fail(FP_ERR_UNSUPPORTED, "fp_paged_decode: B, Hq or Hc exceeds 65535");
  if (B == 0) return FP_OK;
  if (!page_table || !batch_idx || !input_pos) return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode: null pointer");
  if (plan_only) {
    if (!plan) return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode_plan: null plan");
  } else {
    if (!q || !pool_k || !pool_v || !out || !lse) return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode: null pointer");
    if (!fp::aligned(q, 16) || !fp::aligned(pool_k, 16) || !fp::aligned(pool_v, 16) ||
        (q_stride_b * eb) % 16 || (q_stride_h * eb) % 16)
      return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode: q and pool rows must be 16-byte aligned");
    if (!fp::aligned(out, eb)) return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode: out misaligned");
  }
  if (plan && (!fp::aligned(plan, 4) || plan_bytes < plan_buffer_bytes()))
    return fp::fail(FP_ERR_WORKSPACE, "fp_paged_decode: the plan buffer needs %lld bytes (fp_paged_decode_plan_bytes), %lld given",
                    static_cast<long long>(plan_buffer_bytes()), static_cast<long long>(plan_bytes));

  const int64_t counters = static_cast<int64_t>(B) * wg_heads * 4;
  if (arrivals && (!fp::aligned(arrivals, 4) || arrivals_bytes < counters))
    return fp::fail(FP_ERR_WORKSPACE, "fp_paged_decode_step: %lld bytes of arrival counters needed, %lld given",
                    static_cast<long long>(counters), static_cast<long long>(arrivals_bytes));
  const char *const now = reinterpret_cast<const char*>(arrivals), *const later = reinterpret_cast<const char*>(next_arrivals);
  if (later && (!fp::aligned(later, 4) || (later < now + arrivals_bytes && now < later + arrivals_bytes)))
    return fp::fail(FP_ERR_WORKSPACE, "fp_paged_decode_step: the counters of the next launch overlap those of this one");

  if (split_tokens == 0) split_tokens = default_split_tokens(B, wg_heads, max_context, page_size);
  if (split_tokens % 64) return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode: split_tokens must be a multiple of 64");
  if (split_tokens / page_size + 2 > kMaxSplitPages)
    return fp::fail(FP_ERR_UNSUPPORTED, "fp_paged_decode: split of %d tokens spans more than %d pages", split_tokens,
                    kMaxSplitPages - 2);
  const int ns = n_splits_for(max_context, split_tokens);
  if (ns > 65535) return fp::fail(FP_ERR_UNSUPPORTED, "fp_paged_decode: more than 65535 splits");

  // Counters in lines of 128 bytes of their own where the caller's memory has room: the splits of a short launch arrive together, and adding
  // to words of one line they wait for each other (us a layer with all counters in two lines / apart, 8 heads, limit 8192: 2 sequences of 6157
  // to 7448 tokens, D 64, bf16 12.9 / 10.1, with 2 query heads 14.0 / 11.4, D 128 15.9 / 14.7; one of 7000 9.9 / 8.2; in two passes 10.6, 12.4, 15.0, 9.5).
  const int64_t room = counters > 0 ? arrivals_bytes / counters : 1;
  const int arrivals_step = room >= 32 ? 32 : room >= 1 ? static_cast<int>(room) : 1;
  DecodeArgs a{static_cast<const char*>(q), q_stride_b * eb, q_stride_h * eb,
               static_cast<const char*>(pool_k), static_cast<const char*>(pool_v),
               page_table, pt_row_stride, batch_idx, input_pos, pos_index_type == FP_INDEX_I64,
               static_cast<char*>(out), out_stride_b * eb, out_stride_h * eb, lse, sinks,
               nullptr, nullptr, Hq, wg_heads, fp::PageDiv(page_size), n_pages, max_batch,
               static_cast<int>(n_slots / page_size > INT32_MAX ? INT32_MAX : n_slots / page_size), n_slots,
               max_context, split_tokens, ns, scale * kLog2e,  // scores are kept in log2 units
               nullptr, nullptr, 0, 0, 0, 0, B, 0, static_cast<int*>(plan), arrivals, arrivals_step, next_arrivals};
  if (fresh) {
    if (!fresh->k || !fresh->v) return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode_append: null k_new / v_new");
    if (!fp::aligned(fresh->k, 16) || !fp::aligned(fresh->v, 16) || (fresh->k_stride_b * eb) % 16 ||
        (fresh->k_stride_h * eb) % 16 || (fresh->v_stride_b * eb) % 16 || (fresh->v_stride_h * eb) % 16)
      return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode_append: k_new / v_new rows must be 16-byte aligned");
    a.k_new = static_cast<const char*>(fresh->k);
    a.v_new = static_cast<const char*>(fresh->v);
    a.kn_b = fresh->k_stride_b * eb;
    a.kn_h = fresh->k_stride_h * eb;
    a.vn_b = fresh->v_stride_b * eb;
    a.vn_h = fresh->v_stride_h * eb;
  }
  if (ns > 1 && !plan_only) {
    const int64_t need = static_cast<int64_t>(B) * Hq * ns * (D + 2) * static_cast<int64_t>(sizeof(float));
    if (!workspace || workspace_bytes < need || !fp::aligned(workspace, 16))
      return fp::fail(FP_ERR_WORKSPACE, "fp_paged_decode: workspace of %lld bytes needed, %lld given",
                      static_cast<long long>(need), static_cast<long long>(workspace_bytes));
    a.ws_acc = static_cast<float*>(workspace);
    a.ws_ml = a.ws_acc + static_cast<int64_t>(B) * Hq * ns * D;
  }

  hipStream_t st = static_cast<hipStream_t>(stream);
  int rc;
  switch (dtype) {
    case FP_DTYPE_F32: rc = dispatch_dim<F32>(a, B, D, phases, kv_rep, st); break;
    case FP_DTYPE_BF16: rc = dispatch_dim<BF16>(a, B, D, phases, kv_rep, st); break;
    default: rc = dispatch_dim<F16>(a, B, D, phases, kv_rep, st); break;
  }
  if (rc != FP_OK) return rc;
  return fp::check_launch("fp_paged_decode");
}

}  // namespace

#define FP_DECODE_PARAMS                                                                                   \
  const void *q, int64_t q_stride_b, int64_t q_stride_h, const void *pool_k, const void *pool_v,          \
      const int64_t *page_table, int64_t pt_row_stride, const int64_t *batch_idx, const void *input_pos,  \
      int pos_index_type, void *out, int64_t out_stride_b, int64_t out_stride_h, float *lse,              \
      const float *sinks,                                                                                 \
      void *workspace, int64_t workspace_bytes, int32_t B, int32_t Hq, int32_t Hc, int32_t kv_rep,        \
      int32_t D,                                                                                          \
      int32_t page_size, int32_t n_pages, int32_t max_batch, int64_t n_slots, int32_t max_context,        \
      int32_t split_tokens, float scale, int dtype, void *plan, int64_t plan_bytes, void *stream
#define FP_DECODE_ARGS                                                                                     \
  q, q_stride_b, q_stride_h, pool_k, pool_v, page_table, pt_row_stride, batch_idx, input_pos,             \
      pos_index_type, out, out_stride_b, out_stride_h, lse, sinks, workspace, workspace_bytes, B, Hq, Hc, kv_rep, D, \
      page_size, n_pages, max_batch, n_slots, max_context, split_tokens, scale, dtype, plan, plan_bytes, stream

extern "C" int64_t fp_paged_decode_plan_bytes(void) { return plan_buffer_bytes(); }
extern "C" int fp_paged_decode_plan(FP_DECODE_PARAMS) { return decode_entry(kPhasePlan, nullptr, FP_DECODE_ARGS); }
extern "C" int fp_paged_decode(FP_DECODE_PARAMS) {
  return decode_entry(kPhasePartial | kPhaseMerge, nullptr, FP_DECODE_ARGS);
}
extern "C" int fp_paged_decode_partial(FP_DECODE_PARAMS) { return decode_entry(kPhasePartial, nullptr, FP_DECODE_ARGS); }
extern "C" int fp_paged_decode_merge(FP_DECODE_PARAMS) { return decode_entry(kPhaseMerge, nullptr, FP_DECODE_ARGS); }
extern "C" int fp_paged_decode_append(const void* k_new, const void* v_new, int64_t k_stride_b, int64_t k_stride_h,
                                      int64_t v_stride_b, int64_t v_stride_h, FP_DECODE_PARAMS) {
  const NewRows fresh{k_new, v_new, k_stride_b, k_stride_h, v_stride_b, v_stride_h};
  return decode_entry(kPhasePartial | kPhaseMerge, &fresh, FP_DECODE_ARGS);
}
extern "C" int fp_paged_decode_step(int32_t* arrivals, int32_t* next_arrivals, int64_t arrivals_bytes, const void* k_new, const void* v_new,
                                    int64_t k_stride_b, int64_t k_stride_h, int64_t v_stride_b, int64_t v_stride_h,
                                    FP_DECODE_PARAMS) {
  if (B > 0 && !arrivals) return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode_step: null arrival counters");
  const NewRows fresh{k_new, v_new, k_stride_b, k_stride_h, v_stride_b, v_stride_h};
  return decode_entry(kPhasePartial | kPhaseMerge, k_new || v_new ? &fresh : nullptr, FP_DECODE_ARGS, arrivals, next_arrivals, arrivals_bytes);
}


// ---------------------------------------------------------------------------------------------
// fp_paged_decode for callers that cannot allocate: the split-K partial results go to an array that
// lives in the library's device image instead of a caller-owned workspace.
//
// `scratch` below is, in host code, only a handle of the device symbol: its device address differs
// per GPU and is asked for once per device with hipGetSymbolAddress, on the entry point's first call
// on that device (with that device current).  Only that address is ever handed to a kernel.  Every
// launch on a GPU shares the GPU's one array: calls that overlap on one GPU (two streams, two
// threads) race on it.  The partial pass writes every row the merge pass reads, so the contents left
// by an earlier call never need clearing.
constexpr int64_t kScratchBytes = FP_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch_ptr[kMaxDevices];

// device address of `scratch` on the current device, nullptr + error message on failure
void* scratch_address() {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    fp::fail(FP_ERR_LAUNCH, "fp_paged_decode_noalloc: hipGetDevice: %s (device %d)", hipGetErrorString(e), dev);
    return nullptr;
  }
  void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (p) return p;
  e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !p) {
    (void)hipGetLastError();
    fp::fail(FP_ERR_LAUNCH, "fp_paged_decode_noalloc: hipGetSymbolAddress(scratch) on device %d: %s", dev,
             hipGetErrorString(e));
    return nullptr;
  }
  g_scratch_ptr[dev].store(p, std::memory_order_release);  // two first calls racing store the same address
  return p;
}
}  // namespace

extern "C" int fp_paged_decode_noalloc(const void* q, int64_t q_stride_b, int64_t q_stride_h, const void* pool_k,
                                       const void* pool_v, const int64_t* page_table, int64_t pt_row_stride,
                                       const int64_t* batch_idx, const void* input_pos, int pos_index_type,
                                       void* out, int64_t out_stride_b, int64_t out_stride_h, float* lse,
                                       const float* sinks, int32_t B, int32_t Hq, int32_t Hc, int32_t kv_rep,
                                       int32_t D, int32_t page_size, int32_t n_pages, int32_t max_batch,
                                       int64_t n_slots, int32_t max_context, int32_t split_tokens, float scale,
                                       int dtype, void* stream) {
  // size the partial results exactly as decode_entry will, and refuse what the array cannot hold
  if (B < 0 || Hq <= 0 || Hc <= 0 || D <= 0 || page_size <= 0 || max_context < 0 || split_tokens < 0 || kv_rep < 1)
    return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode_noalloc: bad dimension");
  int st = split_tokens;
  if (st == 0) st = default_split_tokens(B, kv_rep > 1 ? Hq / kv_rep : Hc, max_context, page_size);
  if (st % 64) return fp::fail(FP_ERR_INVALID_ARGUMENT, "fp_paged_decode_noalloc: split_tokens must be a multiple of 64");
  const int64_t ns = n_splits_for(max_context, st);
  const int64_t need = ns > 1 ? static_cast<int64_t>(B) * Hq * ns * (D + 2) * static_cast<int64_t>(sizeof(float)) : 0;
  if (need > kScratchBytes)
    return fp::fail(FP_ERR_WORKSPACE,
                    "fp_paged_decode_noalloc: this launch needs %lld bytes of split-K partial results, the library's "
                    "array holds %lld; use fp_paged_decode with a caller-owned workspace, or a larger split_tokens",
                    static_cast<long long>(need), static_cast<long long>(kScratchBytes));
  void* ws = nullptr;
  if (need) {
    ws = scratch_address();
    if (!ws) return FP_ERR_LAUNCH;
  }
  return decode_entry(kPhasePartial | kPhaseMerge, nullptr, q, q_stride_b, q_stride_h, pool_k, pool_v, page_table,
                      pt_row_stride, batch_idx, input_pos, pos_index_type, out, out_stride_b, out_stride_h, lse, sinks,
                      ws, need ? kScratchBytes : 0, B, Hq, Hc, kv_rep, D, page_size, n_pages, max_batch, n_slots,
                      max_context, st, scale, dtype, nullptr, 0, stream);
}
