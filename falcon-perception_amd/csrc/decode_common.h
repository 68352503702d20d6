// Shared by the decode kernels (paged_decode.hip, paged_decode_mfma.hip): their arguments, the plan of a step, the even
// cut of a launch, the sink gate and lane exchanges.
#pragma once

#include "fp_common.h"
#include "prefill_common.h"

#include <math.h>

namespace fp_decode {

constexpr int kMaxSplitPages = 1024;  // page ids of one split held in LDS
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

struct DecodeArgs {
  const char* q;
  int64_t qs_b, qs_h;  // bytes
  const char* pool_k;
  const char* pool_v;
  const int64_t* page_table;
  int64_t pt_row_stride;
  const int64_t* batch_idx;
  const void* input_pos;
  int pos_i64;
  char* out;
  int64_t os_b, os_h;  // bytes
  float* lse;
  const float* sinks;  // optional [Hq]: out is multiplied by sigmoid(lse - sinks[h])
  float* ws_acc;  // [B, Hq, n_splits, D]
  float* ws_ml;   // [B, Hq, n_splits, 2]
  int Hq, Hc;
  fp::PageDiv pd;
  int n_pages, max_batch, pool_pages;  // pool_pages = n_slots / page_size
  int64_t n_slots;
  int max_context;
  int split_tokens;
  int n_splits;
  float qscale;  // scale * log2(e)
  // fused append (optional): the row of the newest token of every sequence, [B, Hc, 1, D]
  const char* k_new;
  const char* v_new;
  int64_t kn_b, kn_h, vn_b, vn_h;  // bytes
  int B;         // sequences of the launch
  int n_chunks;  // even cut (kFlat): workgroups per cache head; walk_pieces: splits of all sequences together, about
  int* plan;     // optional: the step's plan of the even cut (fp_paged_decode_plan), kPlanInts ints per chunk
  // optional [B, Hc], all 0 between launches: how many splits of a (sequence, workgroup head) have left their
  // partial result.  The workgroup that is the last merges them, and there is no merge pass (last_to_arrive, merge_splits)
  int* arrivals;
  int arrivals_step;  // ints from counter to counter
  int* next_arrivals;  // optional, laid out alike: counters of a launch after this one, which this one sets to 0 (clear_next_counter)
};

// The plan of a decode step: what every workgroup of the even cut needs before it can ask for its first K row,
// computed once per step instead of once per layer and workgroup.  Per chunk (workgroup of a cache head):
//   rec[0]            pieces of the chunk, or -1: no plan for this chunk (more pieces or pages than a record
//                     holds), the workgroup works everything out itself
//   rec[1 .. 3]       B, n_chunks, max_context of the launch the plan was made for: a workgroup that finds other
//                     values ignores the plan
//   rec[4 + 6 k ..]   piece k: sequence, first token, tokens, raw length (position + 1), row of the page table
//                     (-1: not a valid slot), offset of its page ids in the chunk's list
//   pages[..]         page ids of the pieces, piece after piece (unmapped or foreign pages as 0, like the kernel
//                     stages them)
//   chunk 0, rec[126]  a hash of the positions and slots the plan was made from (plan_hash_term)
// The positions, the slots and the page table must not change between the plan and the launches that use it.
// What the launches do if they did: the merge pass recomputes the hash from the step's positions and slots
// (it reads them anyway) and stores NaN in every row of out and lse when it differs, so a stale plan fails
// loudly.  The split-K pass itself does not look (a check of its own position before the fused append's store
// measured 1.2 us per launch): with a stale plan the fresh rows of the sequences that moved land where the plan
// says.
constexpr int kPlanPieces = 20;
constexpr int kPlanHashAt = 126;
constexpr int kPlanRec = 128;            // 4 + 6 * kPlanPieces, rounded up
constexpr int kPlanPages = kMaxSplitPages;
constexpr int kPlanInts = kPlanRec + kPlanPages;
static_assert(4 + 6 * kPlanPieces <= kPlanHashAt && kPlanHashAt < kPlanRec, "a record holds its pieces and the hash");

// Contribution of sequence b to the hash of a step's positions and slots (summed over the sequences, mod 2^32).
__device__ __forceinline__ uint32_t plan_hash_term(int b, int64_t L, int64_t trow) {
  const uint32_t w = 2u * static_cast<uint32_t>(b) + 1u;
  return (static_cast<uint32_t>(L) + static_cast<uint32_t>(trow) * 0x9E3779B1u) * w;
}

// Attention-sink gate of the caller's post-attention step (model.py:122-128), applied where the
// output row and its lse are final: the reference multiplies the attention output, already rounded
// to the model dtype, by sigmoid(lse - sinks[h]) in fp32 and rounds again.
template <typename E>
__device__ __forceinline__ float sink_gate(float o, float lse_nat, const float* sinks, int hq) {
  if (sinks == nullptr) return o;
  const float g = 1.f / (1.f + __expf(sinks[hq] - lse_nat));
  return E::round(o) * g;
}

// ---- cross-lane helpers ---------------------------------------------------
template <int kCtrl>
__device__ __forceinline__ float dpp(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kCtrl, 0xf, 0xf, true));
}

// Sum over the kLanes consecutive lanes that share a row; every lane gets the total.
// All kN values advance one butterfly step at a time, so back-to-back DPP
// instructions are independent of each other.
template <int kLanes, int kN>
__device__ __forceinline__ void row_sum(float (&x)[kN]) {
#pragma unroll
  for (int i = 0; i < kN; ++i) if (kLanes >= 2) x[i] += dpp<0xB1>(x[i]);   // quad_perm [1,0,3,2]
#pragma unroll
  for (int i = 0; i < kN; ++i) if (kLanes >= 4) x[i] += dpp<0x4E>(x[i]);   // quad_perm [2,3,0,1]
#pragma unroll
  for (int i = 0; i < kN; ++i) if (kLanes >= 8) x[i] += dpp<0x141>(x[i]);  // row_half_mirror
#pragma unroll
  for (int i = 0; i < kN; ++i) if (kLanes >= 16) x[i] += dpp<0x140>(x[i]); // row_mirror
#pragma unroll
  for (int i = 0; i < kN; ++i) if (kLanes >= 32) x[i] += __shfl_xor(x[i], 16);
#pragma unroll
  for (int i = 0; i < kN; ++i) if (kLanes >= 64) x[i] += __shfl_xor(x[i], 32);
}

// v_permlane16_swap exchanges the odd rows of 16 lanes of its first operand with the even rows of its second, as
// fp::swap_lane_halves does with the halves of the wavefront (inline assembly for the reason given there).
__device__ __forceinline__ void swap_rows(float& a, float& b) {
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}
__device__ __forceinline__ void swap_halves(float& a, float& b, float& c, float& d) {
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\tv_permlane32_swap_b32 %2, %3\n\ts_nop 1" : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
}
__device__ __forceinline__ void swap_rows(float& a, float& b, float& c, float& d) {
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3\n\ts_nop 1" : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
}
__device__ __forceinline__ float max_across_rows(float x) {
  float y = x;
  swap_rows(x, y);
  return fmaxf(x, y);
}
__device__ __forceinline__ float sum_across_halves(float x) {
  float y = x;
  fp::swap_lane_halves(x, y);
  return x + y;
}
__device__ __forceinline__ float sum_across_rows(float x) {
  float y = x;
  swap_rows(x, y);
  return x + y;
}
// x[0 .. N / 2) of the lower half of the lanes (of the even rows) get the totals of x[0 .. N / 2), of the other those of the rest.
template <int N, int M>
__device__ __forceinline__ void add_across_halves(float (&x)[M]) {
  static_assert(N % 2 == 0, "elements in pairs");
  if constexpr (N % 4 == 0) {
#pragma unroll
    for (int i = 0; i < N / 2; i += 2) swap_halves(x[i], x[i + N / 2], x[i + 1], x[i + 1 + N / 2]);
  } else {
#pragma unroll
    for (int i = 0; i < N / 2; ++i) fp::swap_lane_halves(x[i], x[i + N / 2]);
  }
#pragma unroll
  for (int i = 0; i < N / 2; ++i) x[i] += x[i + N / 2];
}
template <int N, int M>
__device__ __forceinline__ void add_across_rows(float (&x)[M]) {
  static_assert(N % 2 == 0, "elements in pairs");
  if constexpr (N % 4 == 0) {
#pragma unroll
    for (int i = 0; i < N / 2; i += 2) swap_rows(x[i], x[i + N / 2], x[i + 1], x[i + 1 + N / 2]);
  } else {
#pragma unroll
    for (int i = 0; i < N / 2; ++i) swap_rows(x[i], x[i + N / 2]);
  }
#pragma unroll
  for (int i = 0; i < N / 2; ++i) x[i] += x[i + N / 2];
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float safe_max(float m) { return m == -INFINITY ? 0.f : m; }

// ceil(L / part) for L > 0; unsigned, which is two thirds of the instructions of the signed division in front of the first row
__device__ __forceinline__ int pieces_of(int L, int part) {
  return static_cast<int>((static_cast<uint32_t>(L) + part - 1) / static_cast<uint32_t>(part));
}

// tokens per split of a context of L tokens: L is divided evenly over ceil(L / split_tokens)
// splits, rounded up to 64 tokens (so every split starts on a wavefront-iteration boundary)
__device__ __forceinline__ int split_part(int L, int split_tokens) {
  if (L <= 0) return split_tokens;
  const int n = pieces_of(L, split_tokens);
  return (pieces_of(L, n) + 63) & ~63;
}

// Even cut of a launch (kFlat): the contexts of the launch, each rounded up to 64 tokens, are laid end
// to end and cut into n_chunks pieces of equal length.  Sequence b starts at flat_start[b]; chunk c covers
// [c * len, (c + 1) * len); a chunk that spans several sequences works through them one after another.
constexpr int kFlatMaxB = 1024;

// Start of every sequence on the flat axis -> s_start[0 .. B] (s_start[B] = total), by one wavefront.
__device__ __forceinline__ void flat_starts(const DecodeArgs& a, int* s_start) {
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    const int per = (a.B + 63) / 64;  // consecutive sequences per lane
    int sum = 0;
    for (int i = 0; i < per; ++i) {
      const int b = lane * per + i;
      int Lr = 0;
      if (b < a.B) {
        int64_t L = fp::load_index(a.input_pos, b, a.pos_i64) + 1;
        const int64_t trow = a.batch_idx[b];
        if (trow < 0 || trow >= a.max_batch || L < 0) L = 0;
        if (L > a.max_context) L = a.max_context;
        Lr = (static_cast<int>(L) + 63) & ~63;
      }
      sum += Lr;
    }
    int incl = sum;  // inclusive scan over the lanes
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int up = __shfl_up(incl, off);
      if (lane >= off) incl += up;
    }
    int run = incl - sum;
    for (int i = 0; i < per; ++i) {
      const int b = lane * per + i;
      if (b > a.B) break;
      s_start[b] = run;
      if (b < a.B) {
        int64_t L = fp::load_index(a.input_pos, b, a.pos_i64) + 1;
        const int64_t trow = a.batch_idx[b];
        if (trow < 0 || trow >= a.max_batch || L < 0) L = 0;
        if (L > a.max_context) L = a.max_context;
        run += (static_cast<int>(L) + 63) & ~63;
      }
    }
    if (lane == 63 && a.B == 64 * per) s_start[a.B] = incl;
  }
}

// tokens per chunk of the even cut
__device__ __forceinline__ int flat_chunk_len(int total, int n_chunks) {
  const int len = (total + n_chunks - 1) / n_chunks;
  return len < 64 ? 64 : (len + 63) & ~63;
}

// The kernel's arguments (its first parameter) read again where they are used: the merge needs a dozen of them, once, and scalar
// registers that carried them through the loop over the rows would be spilled into vector registers.
__device__ __forceinline__ const DecodeArgs& reread_args() {
  auto p = (const __attribute__((address_space(4))) DecodeArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const DecodeArgs*)p;
}

// ---- splits that meet without a merge pass ----
// A launch with `arrivals` goes split by split and has no merge pass: every workgroup leaves its partial result, counts itself
// in, and the last of a (sequence, workgroup head) merges all of them.  Results are written and read with relaxed device-scope
// atomics, which go past the eight L2s; a workgroup waits until its own have arrived before it counts itself in, so whoever
// counts n - 1 others sees all rows, and no cache is written back or invalidated (a device-scope fence writes back an XCD's L2: +68 us
// at 512 workgroups).  Nobody waits for anybody.  The last one sets its counter back to 0 for the next launch.  The three trips
// (store, count, load) are 0.4 to 0.5 us each; a launch in a replayed graph is 1.7 us before it does anything, and a merge pass
// 2.7 to 3.3.  What a launch of this kind is held to, and its figures: merges_itself.
__device__ __forceinline__ void publish(float* p, float x) {
  __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void publish2(float* p, float x, float y) {
  const uint64_t w = static_cast<uint64_t>(__float_as_uint(y)) << 32 | __float_as_uint(x);
  __hip_atomic_store(reinterpret_cast<uint64_t*>(p), w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float2 take2(const float* p) {
  const uint64_t w = __hip_atomic_load(reinterpret_cast<const uint64_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return float2{__uint_as_float(static_cast<uint32_t>(w)), __uint_as_float(static_cast<uint32_t>(w >> 32))};
}

// x / d for 0 <= x < 2^23, d >= 1 and a quotient below 2^21, in half the instructions of an integer division: it is in front of the
// first row.  The product's error is below x / d * 2^-22 + 1, so a step up or down is all there is to mend.
__device__ __forceinline__ int quotient(int x, int d) {
  const int q = static_cast<int>(static_cast<float>(x) * __builtin_amdgcn_rcpf(static_cast<float>(d)));
  const int rest = x - q * d;
  return q + (rest >= d ? 1 : rest < 0 ? -1 : 0);
}

// Inclusive sum over the lanes up to this one, without a trip through LDS.
__device__ __forceinline__ int scan_lanes(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);  // row_shr:1, 2, 4, 8, then row_bcast:15, 31
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, true);
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, true);
  return x;
}

// Splits of L tokens (> 0) in a launch with arrivals: the launch's length, twice that where there would be more than merge_splits
// takes at once and half as many still give every CU a workgroup (8000 tokens, 16 q / 8 kv heads, D 128: 13.4 us a layer in 64 splits,
// 12.3 in 32; 4 heads of 64 in fp32 9.3 and 9.5).
__device__ __forceinline__ int split_tokens_for(const DecodeArgs& a, int L) {
  const bool twice = a.Hc >= 8 && L > 32 * a.split_tokens && 2 * a.split_tokens < (kMaxSplitPages - 1) * a.pd.page_size;  // pages fit LDS
  return twice ? 2 * a.split_tokens : a.split_tokens;
}

// The workgroup's partial result of sequence b is on its way (publish, by any of its threads): counts it in and says whether it is
// the last of n.  `flag`: one word of LDS.
__device__ __forceinline__ bool last_to_arrive(int b, int n, int* flag) {
  const DecodeArgs& a = reread_args();
  asm volatile("s_waitcnt vmcnt(0)" : : : "memory");  // this wavefront's stores have arrived
  __syncthreads();
  if (threadIdx.x == 0) {
    int* const counter = a.arrivals + (static_cast<int64_t>(b) * a.Hc + blockIdx.x) * a.arrivals_step;
    const bool last = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == n - 1;
    if (last) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *flag = last;
  }
  __syncthreads();
  return __builtin_amdgcn_readfirstlane(*flag) != 0;
}

// Counters are 0 behind a launch because its last workgroups say so; where one was not (launches that overlapped on the same counters, positions
// written while a launch read them), every launch to come would merge too early or never.  A launch that is given the counters of a later one
// sets these to 0, by the workgroup of the first split, so that such a fault does not outlast the next launch.
__device__ __forceinline__ void clear_next_counter(const DecodeArgs& a, int b) {
  if (threadIdx.x != 0 || a.next_arrivals == nullptr) return;
  __hip_atomic_store(a.next_arrivals + (static_cast<int64_t>(b) * a.Hc + blockIdx.x) * a.arrivals_step, 0, __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_AGENT);
}

// Merges the n partial results of sequence b's G heads (rows hq * row_mul + row_add + split of the workspace), normalises, gates and
// stores them.  A wavefront takes 128 elements of the G x D (two per lane); where there are fewer of these than wavefronts, several
// share one and take the splits in batches of kMergeBatch in turn.  Every load of two batches is in flight at once.  `s_part`: 4 * 64 * 4 floats
// of LDS.
constexpr int kMergeBatch = 8;
template <typename E, int D>
__device__ __forceinline__ void merge_splits(int b, int64_t row_mul, int64_t row_add, int n, int G, float* s_part) {
  const DecodeArgs& a = reread_args();
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));  // nothing in here is worked out ahead of the rows and kept in registers through them
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, hc = blockIdx.x;
  const int n_items = (G * D + 127) / 128;        // 1 or 2 (merges_itself)
  const int deep = 4 / n_items, turn = wave / n_items, item = wave & (n_items - 1);
  const int e = item * 128 + lane * 2;
  const bool on = e < G * D;
  const int g = on ? e / D : 0, d = on ? e - g * D : 0, hq = hc * G + g;
  const int64_t row0 = hq * row_mul + row_add;
  const float* const ml_at = a.ws_ml + row0 * 2;
  const float* const acc_at = a.ws_acc + row0 * D + d;
  float m = -INFINITY, den = 0.f, num0 = 0.f, num1 = 0.f;
  float2 ml[2][kMergeBatch], acc[2][kMergeBatch];
  const auto load = [&](int base, float2 (&ml)[kMergeBatch], float2 (&acc)[kMergeBatch]) {
    const float* mp = ml_at + base * 2;
    const float* ap = acc_at + static_cast<int64_t>(base) * D;
#pragma unroll
    for (int s = 0; s < kMergeBatch; ++s) {  // past the last split its row again, dropped below
      ml[s] = take2(mp);
      acc[s] = take2(ap);
      const int next = base + s + 1 < n ? 1 : 0;
      mp += next * 2;
      ap += next * D;
    }
  };
  const auto fold = [&](int base, const float2 (&ml)[kMergeBatch], const float2 (&acc)[kMergeBatch]) {
    float mn = m;
#pragma unroll
    for (int s = 0; s < kMergeBatch; ++s) mn = fmaxf(mn, ml[s].x);
    const float ms = safe_max(mn), keep = fast_exp2(m - ms);
    den *= keep;
    num0 *= keep;
    num1 *= keep;
#pragma unroll
    for (int s = 0; s < kMergeBatch; ++s) {
      if (base + s >= n) break;
      const float w = fast_exp2(ml[s].x - ms);
      den += ml[s].y * w;
      num0 += acc[s].x * w;
      num1 += acc[s].y * w;
    }
    m = mn;
  };
  const int stride = deep * kMergeBatch;
#pragma nounroll
  for (int base = turn * kMergeBatch; base < n; base += 2 * stride) {
    load(base, ml[0], acc[0]);
    if (base + stride < n) load(base + stride, ml[1], acc[1]);
    fold(base, ml[0], acc[0]);
    if (base + stride < n) fold(base + stride, ml[1], acc[1]);
  }
  float4* const slot = reinterpret_cast<float4*>(s_part) + lane;
  slot[wave * 64] = float4{m, den, num0, num1};
  __syncthreads();
  if (turn != 0) return;
#pragma nounroll
  for (int t = 1; t < deep; ++t) {
    const float4 o = slot[(wave + t * n_items) * 64];
    const float mn = fmaxf(m, o.x), ms = safe_max(mn), keep = fast_exp2(m - ms), w = fast_exp2(o.x - ms);  // w: 0 without a split
    den = den * keep + o.y * w;
    num0 = num0 * keep + o.z * w;
    num1 = num1 * keep + o.w * w;
    m = mn;
  }
  if (!on) return;
  const float lse_nat = (m + log2f(den)) * kLn2;
  char* const o = a.out + b * a.os_b + hq * a.os_h + d * sizeof(typename E::type);
  E::store(o, sink_gate<E>(num0 / den, lse_nat, a.sinks, hq));
  E::store(o + sizeof(typename E::type), sink_gate<E>(num1 / den, lse_nat, a.sinks, hq));
  if (d == 0) a.lse[static_cast<int64_t>(b) * a.Hq + hq] = lse_nat;
}

// Which launches merge their splits themselves, where the caller brings the counters: up to 256 elements a merge (query heads x
// head_dim), and not the even cut (merged_pieces: which of these go piece by piece).  A single workgroup takes longer over more than a merge
// pass that has a wavefront per row, and the
// even cut's workgroups end together, so that the three trips come on top of all of them.  us a layer in two passes / one launch, 8 heads: 2 x
// 128 elements, one sequence of 300, 2000 and 8000 tokens 9.1 / 7.7, 9.7 / 8.6 and 12.9 / 12.3, 4 of 100 to 700 13.8 / 11.4; 4 x 64 (matrix cores) 8.6 /
// 7.7, 8.7 / 7.9, 10.4 / 9.9 and 10.0 / 8.9; 4 x 128 9.5 / 8.4, 10.1 / 9.5, but 13.6 / 13.8 at 8000 tokens, and two of 8000 17.8 / 18.6; 8 x 128
// 9.9 / 9.9, 8000 tokens 14.5 / 23.0, 4 of 100 to 700 13.7 / 12.3.  Even cut, 2 x 128: 64 of 1088 to 4096 117.3 / 118.1, 96 of 64 to 400 29.0 / 29.6,
// 16 of 350 to 4620 38.7 / 38.2; 8 x 128: 24 of 512 to 8191 74.5 / 80.1.
constexpr bool merges_itself(int G, int D) { return G * D <= 256; }

// What a workgroup does with its cut: piece(sequence, first token, tokens, which of the sequence's pieces it is (of the even cut only: not the first), and
// where its partial result goes: workspace row head * part_mul + part_add; how many pieces the sequence has in a launch with arrivals; position
// + 1 and page-table row of the sequence; then the page ids of a planned piece).

// tokens a split has at least there, by the bytes of a row: what the wavefronts ask for at once
// (16 sequences of 64 to 500 tokens, head_dim 64, 2 query heads, f16: 10.1 us a layer from 128 on, 9.6 from 256)
constexpr int min_part(int row_bytes) { return row_bytes < 256 ? 256 : 128; }
constexpr int kMostPieces = 16;  // splits a sequence has at most there: what merge_splits asks for at once with two query heads

// One trip to memory for the arguments up to the first row: each is otherwise asked for where it is first used, and a line of 64
// bytes that no load before it touched is a trip of its own.
__device__ __forceinline__ void ask_for_arguments(const DecodeArgs& a) {
  asm volatile("" : : "s"(a.q), "s"(a.batch_idx), "s"(a.input_pos), "s"(a.Hq), "s"(a.Hc), "s"(a.n_slots), "s"(a.n_splits),
               "s"(a.k_new), "s"(a.vn_h), "s"(a.B), "s"(a.arrivals));
}

// Position + 1 of sequence b and its page-table row (-1: not a valid slot), as a piece is given them.
template <bool kUniform>
__device__ __forceinline__ void load_sequence(const DecodeArgs& a, int b, int* raw, int* trow) {
  // one trip to memory: both words of an int64 position or an int32 one twice, so that neither its type nor the slot waits for a load
  const int at = a.pos_i64 ? 2 * b : b;
  const auto pos = (const __attribute__((address_space(4))) int*)a.input_pos;  // no launch writes them: scalar loads
  int lo = pos[at];
  int hi = pos[a.pos_i64 ? at + 1 : at];
  int64_t t = ((const __attribute__((address_space(4))) int64_t*)a.batch_idx)[b];
  if constexpr (kUniform)
    asm volatile("" : "+s"(lo), "+s"(hi), "+s"(t));
  else
    asm volatile("" : "+v"(lo), "+v"(hi), "+v"(t));
  if (a.pos_i64 && hi != lo >> 31) lo = hi < 0 ? INT32_MIN : INT32_MAX;
  *raw = lo == INT32_MAX ? lo : lo + 1;
  *trow = t < 0 || t >= a.max_batch ? -1 : static_cast<int>(t);
}

// Grid (workgroup heads, B, splits).
template <bool kMerges, class Work>
__device__ __forceinline__ void walk_split(const DecodeArgs& a, const Work& piece) {
  // A context of L tokens is cut into ceil(L / split_tokens) parts of equal
  // size (a multiple of 64 tokens), so the workgroups of one sequence carry the same load instead of
  // leaving a short tail split.
  // The workgroup dispatcher deals consecutive workgroups of an XCD to its four shader engines in turn
  // and starts them in order, so with grid y = sequence every split of a sequence would land on the
  // same engine and an engine's load would be the lengths of "its" sequences (12 % apart at 64
  // sequences of 1 k to 4 k tokens).  Rotating the sequences by the split index spreads each sequence
  // over the engines.
  const int split = blockIdx.z;
  ask_for_arguments(a);
  int b = blockIdx.y + blockIdx.z;
  b = static_cast<int>(static_cast<uint32_t>(b) % static_cast<uint32_t>(a.B));
  int raw, trow;
  load_sequence<true>(a, b, &raw, &trow);
  const int L = raw > a.max_context ? a.max_context : raw < 0 ? 0 : raw;
  const int part = split_part(L, kMerges && a.arrivals ? split_tokens_for(a, L) : a.split_tokens);
  piece(b, split * part, part, split, a.n_splits, static_cast<int64_t>(b) * a.Hq * a.n_splits + split, L > 0 ? pieces_of(L, part) : 0,
        raw, trow, nullptr);
}

// Grid (workgroup heads, n_chunks + B) of a launch with arrivals, up to 48 sequences (merged_pieces; a lane of a wavefront each): the splits of all sequences have one length, as long
// as n_chunks of them need to be, and what a workgroup does follows from the lengths of the sequences.  Split by split it follows
// from max_context, and a workgroup that finds nothing to do costs the launch 3 ns: 4 sequences of 300 tokens under a limit of 4096, 1024
// workgroups 10.9 us a layer, 512 9.4, 256 8.1.  Every wavefront works the cut out by itself, a sequence to a lane, without LDS or a barrier; that
// is 0.3 us in front of the first row, which is why launches that gain nothing else go split by split (merged_pieces).
template <int kMinPart, class Work>
__device__ __forceinline__ void walk_pieces(const DecodeArgs& a, const Work& piece) {
  ask_for_arguments(a);
  const int lane = threadIdx.x & 63, c = blockIdx.y, pieces = a.n_chunks;
  int lane_raw, lane_trow;
  load_sequence<false>(a, lane < a.B ? lane : 0, &lane_raw, &lane_trow);
  int L = lane_trow < 0 || lane_raw < 0 || lane >= a.B ? 0 : lane_raw;
  L = L > a.max_context ? a.max_context : L;
  const int total = __builtin_amdgcn_readlane(scan_lanes(L), 63);
  int part = total <= kMinPart * pieces ? kMinPart : (quotient(total, pieces) + 64) & ~63;
  int count, upto;
  for (int tries = 0;; ++tries) {
    count = quotient(L + part - 1, part);
    count = count < 1 ? 1 : count < kMostPieces ? count : kMostPieces;
    upto = scan_lanes(lane < a.B ? count : 0);
    // with the remainders there are up to B more than `pieces`, which would run behind the others: somewhat longer, then
    if (__builtin_amdgcn_readlane(upto, 63) <= pieces || part == kMinPart || tries == 4) break;
    part += 64 + (part >> 4 & ~63);
  }
  // the splits of a sequence are equal, too, and may be fewer for it (every lane its own)
  int own = (quotient(L + count - 1, count) + 63) & ~63;
  own = own < 64 ? 64 : own;
  const int n_own = quotient(L + own - 1, own);
  const unsigned long long behind = __ballot(upto > c);
  if (behind == 0) return;
  const int b = __builtin_ctzll(behind);
  const int raw = __builtin_amdgcn_readlane(lane_raw, b), trow = __builtin_amdgcn_readlane(lane_trow, b);
  const int n = __builtin_amdgcn_readlane(n_own, b);
  part = __builtin_amdgcn_readlane(own, b);
  const int split = c - __builtin_amdgcn_readlane(upto - count, b);
  if (split > 0 && split >= n) return;
  piece(b, split * part, part, split, pieces + a.B, c, n, raw, trow, nullptr);
}

// Grid (workgroup heads, n_chunks): every workgroup streams the same number of rows, whatever the lengths are.  `s_start`
// holds kFlatMaxB + 1 ints, `s_pages` kMaxSplitPages.
template <int kThreads, class Piece>
__device__ __forceinline__ void walk_even_cut(const DecodeArgs& a, int* s_start, int* s_pages, const Piece& piece) {
  const int tid = threadIdx.x;
  if (a.plan) {
    // the chunk's record goes where the sequence starts would go, its page ids where a piece stages its own:
    // one trip to memory instead of positions -> cut -> page table
    const int* src = a.plan + static_cast<int64_t>(blockIdx.y) * kPlanInts;
    if (tid < kPlanRec) s_start[tid] = src[tid];
    s_pages[tid] = src[kPlanRec + tid];  // the first kThreads page ids; more only for very long chunks
    __syncthreads();
    const int n = s_start[0];
    if (n >= 0 && n <= kPlanPieces && s_start[1] == a.B && s_start[2] == a.n_chunks && s_start[3] == a.max_context) {
      int n_pages_used = 0;
      if (n > 0) {
        const int* last = s_start + 4 + 6 * (n - 1);
        n_pages_used = last[5] + last[2] / a.pd.page_size + 2;  // an upper bound of the list's length
      }
      if (n_pages_used > kThreads) {
        for (int i = kThreads + tid; i < n_pages_used && i < kPlanPages; i += kThreads) s_pages[i] = src[kPlanRec + i];
        __syncthreads();
      }
      const int c = blockIdx.y;
      // the records are read from registers of a copy: a piece reuses s_start's LDS for nothing, but keeps s_pages
      for (int k = 0; k < n; ++k) {
        int r[6];
#pragma unroll
        for (int j = 0; j < 6; ++j) r[j] = s_start[4 + 6 * k + j];
        piece(r[0], r[1], r[2], 1, 1, static_cast<int64_t>(c + r[0]) * a.Hq, 0, r[3], r[4], s_pages + r[5]);
        __syncthreads();  // the LDS of the piece is free again
      }
      return;
    }
    __syncthreads();  // no usable plan: s_start and s_pages are written anew below
  }
  flat_starts(a, s_start);
  __syncthreads();
  const int total = s_start[a.B];
  const int len = flat_chunk_len(total, a.n_chunks);
  const int c = blockIdx.y;
  const int64_t lo = static_cast<int64_t>(c) * len;
  const int64_t hi = lo + len < total ? lo + len : total;
  if (lo >= total) return;
  // first sequence that ends after lo
  int b = 0;
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
    if (end == begin) continue;  // a sequence without keys has no piece; the merge pass writes its zeros
    const int t0 = lo > begin ? static_cast<int>(lo - begin) : 0;
    const int t1 = static_cast<int>((hi < end ? hi : end) - begin);
    int raw, trow;
    load_sequence<false>(a, b, &raw, &trow);
    piece(b, t0, t1 - t0, 1, 1, static_cast<int64_t>(c + b) * a.Hq, 0, raw, trow, nullptr);
    __syncthreads();  // the LDS of the piece is free again
  }
}

}  // namespace fp_decode
