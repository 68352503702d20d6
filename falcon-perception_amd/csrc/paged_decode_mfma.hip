// Paged decode attention on the matrix cores: 16-bit caches with four or eight query heads per cache head.
//
// The same work as paged_decode_kernel (paged_decode.hip): a workgroup of 4 wavefronts owns one (cache head, token range)
// of a sequence and reads each K and V row once.  There every row costs G dot products and G multiply-adds per element on
// the vector pipe, which is the limit from four query heads on; here the G heads are columns of a matrix product, whose
// cost does not depend on G.
//   S^T = K Q^T   v_mfma_f32_16x16x32: 16 keys x 16 columns.  Columns 0 .. 7 and 8 .. 15 both hold the heads of the group.
//   O^T += V^T P^T  v_mfma_f32_16x16x16: P^T is in the B operand's layout as the scores leave the first product.  Columns
//         0 .. 7 carry the probabilities rounded to the 16-bit type and columns 8 .. 15 what that rounding left over; the two
//         halves of O^T are added at the end, so P keeps 16 (bf16) or 22 (f16) bits against the 24 of the vector kernel.
//         The result's error against float64 is the rounding of the output either way: 1.648e-3 to 1.664e-3 (bf16) and 2.05e-4 to
//         2.10e-4 (f16) over contexts of 64 to 8191 tokens, 1e-6 of that apart from the vector kernel's.
//   K and V go straight from HBM into LDS (global_load_lds, non-temporal), row-major with the 16-byte chunks permuted
//         against bank conflicts; V^T comes out through ds_read_b64_tr_b16.  Every wavefront has a ring of two stages of
//         4 KB of K and 4 KB of V of its own: no barrier inside a token range, and the next stage is on its way while one
//         is worked on.  Two workgroups to a CU keep 64 to 128 KB in flight per CU.
// HBM-bound.  Per layer-step, merge pass included, against the vector kernel: 24 sequences of 512 to 8191 tokens, 64 q / 8 kv
// heads, bf16 (415 MB) 76.8 us (5.4 TB/s) against 142.7 us; 96 sequences of 4352 to 16384 tokens, 32 q / 8 kv heads (4.0
// GB) 626 us (6.5 TB/s) against 648 us.
#include "decode_common.h"
#include "paged_decode_mfma.h"

#include <type_traits>

namespace {

using namespace fp_decode;

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int kStageBytes = 8192;      // 4 KB of K rows, then 4 KB of V rows
constexpr int kStages = 2;             // per wavefront
constexpr int kMaxGroup = 8;           // query heads per cache head: half of the 16 columns
constexpr float kMaxSlack = 6.f;       // the reference point of the exponentials may lag the maximum by this much (log2)

typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

struct BF16 {
  using type = __bf16;
  typedef __bf16 vec4 __attribute__((ext_vector_type(4)));
  typedef __bf16 vec8 __attribute__((ext_vector_type(8)));
  // Added to the exponents.  Here it keeps the probabilities at 1 and below although the reference point lags the maximum:
  // a product with the largest V of the type stays in fp32.
  static constexpr float kHeadroom = -kMaxSlack;
  static __device__ __forceinline__ f32x4 mfma_k32(const v4u& a, const v4u& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(vec8, a), __builtin_bit_cast(vec8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4 mfma_k16(const s16x4& a, const s16x4& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    typedef __bf16 vec2 __attribute__((ext_vector_type(2)));
    const vec2 v = {static_cast<__bf16>(lo), static_cast<__bf16>(hi)};
    return __builtin_bit_cast(uint32_t, v);
  }
  static __device__ __forceinline__ float above_zero(float p) { return p; }  // fp32's exponents: no p rounds to 0
  static __device__ __forceinline__ float low(uint32_t w) { return __uint_as_float(w << 16); }
  static __device__ __forceinline__ float high(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
  static __device__ __forceinline__ void store(char* p, float v) { *reinterpret_cast<__bf16*>(p) = static_cast<__bf16>(v); }
  static __device__ __forceinline__ float round(float v) { return static_cast<float>(static_cast<__bf16>(v)); }
};
struct F16 {
  using type = _Float16;
  typedef _Float16 vec4 __attribute__((ext_vector_type(4)));
  typedef _Float16 vec8 __attribute__((ext_vector_type(8)));
  // what rounding leaves over of a probability stays a normal number; probabilities up to 2^(8 + kMaxSlack) are below the largest f16
  static constexpr float kHeadroom = 8.f;
  static __device__ __forceinline__ f32x4 mfma_k32(const v4u& a, const v4u& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(vec8, a), __builtin_bit_cast(vec8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4 mfma_k16(const s16x4& a, const s16x4& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(vec4, a), __builtin_bit_cast(vec4, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    typedef _Float16 vec2 __attribute__((ext_vector_type(2)));
    const vec2 v = {static_cast<_Float16>(lo), static_cast<_Float16>(hi)};
    return __builtin_bit_cast(uint32_t, v);
  }
  // a probability that would round to 0 becomes the smallest number of the type, so that an infinite V element still meets
  // something above 0; the other half takes it back (2^-24 - p rounds to 2^-24 again)
  static __device__ __forceinline__ float above_zero(float p) { return fmaxf(p, fminf(p * 0x1p+102f, 0x1p-24f)); }
  static __device__ __forceinline__ float low(uint32_t w) {
    return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(w & 0xffffu)));
  }
  static __device__ __forceinline__ float high(uint32_t w) {
    return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(w >> 16)));
  }
  static __device__ __forceinline__ void store(char* p, float v) { *reinterpret_cast<_Float16*>(p) = static_cast<_Float16>(v); }
  static __device__ __forceinline__ float round(float v) { return static_cast<float>(static_cast<_Float16>(v)); }
};

__device__ __forceinline__ s16x4 lds_read_tr(const char* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p));
}

// this wavefront's staging loads but the `kLater` issued last have landed in LDS
template <int kLater>
__device__ __forceinline__ void wait_staged() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(kLater) : "memory");
}

template <typename E, int D, bool kFlat, bool kPieces = false>
__global__ __launch_bounds__(kThreads, 2) void paged_decode_mfma_kernel(const DecodeArgs a, const Cut cut) {
  constexpr int ROWB = D * 2;             // bytes of a row
  constexpr int CPR = ROWB / 16;          // 16-byte chunks per row
  constexpr int R32 = ROWB / 32;          // 32-byte regions per row
  constexpr int RPI = 64 / CPR;           // rows of one load instruction
  constexpr int TS = 4096 / ROWB;         // tokens per stage
  constexpr int NI = TS / RPI;            // load instructions per stage and tensor
  constexpr int NB = TS / 16;             // 16-key blocks per stage
  constexpr int KK = D / 32;              // k-steps of the score product
  constexpr int DB = D / 16;              // 16-row blocks of O^T
  constexpr bool kMerges = !kFlat && merges_itself(4, D);  // a launch of eight heads comes without arrival counters
  constexpr int NQ = kMaxGroup * ROWB / 1024;  // load instructions of the query rows

  __shared__ __attribute__((aligned(1024))) char s_ring[kWaves * kStages * kStageBytes];
  __shared__ __attribute__((aligned(1024))) char s_q[kMaxGroup * ROWB];
  __shared__ int s_pages[kMaxSplitPages];
  __shared__ float s_ml[kWaves][kMaxGroup][2];

  const int hc = blockIdx.x;
  const int G = a.Hq / a.Hc;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int col = lane & 15;   // column (query head; 8 + head: the same head again) of Q^T, S^T, P^T, O^T
  const int grp = lane >> 4;
  char* const ring = s_ring + wave * (kStages * kStageBytes);

  // staging: instruction i brings rows i * RPI + lane / CPR; this lane fills 16-byte position lane % CPR of its row.
  // The permutations: K chunk c of row r sits at c ^ k_swz(r) (the score product reads one chunk of 16 consecutive rows),
  // V's 32-byte region c of row r at (c + v_rot(r)) % R32 (a transpose read takes one region of 16 consecutive rows).
  const auto k_swz = [](int r) { return CPR == 16 ? r & 15 : (r >> 1) & 7; };
  const auto v_rot = [](int r) { return CPR == 16 ? r & 7 : (r >> 1) & 3; };
  const int lrow = lane / CPR, lpos = lane % CPR;
  uint32_t k_off[NI], v_off[NI];  // byte offset inside the row
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int r = i * RPI + lrow;
    k_off[i] = (lpos ^ k_swz(r)) * 16;
    v_off[i] = (((lpos >> 1) + R32 - v_rot(r)) % R32) * 32 + (lpos & 1) * 16;
  }
  const bool aligned_pages = a.pd.shift >= 0 && a.pd.page_size % TS == 0;  // a full stage lies in one page
  const char* const kplane = a.pool_k + static_cast<int64_t>(hc) * a.n_slots * ROWB;
  const char* const vplane = a.pool_v + static_cast<int64_t>(hc) * a.n_slots * ROWB;

  // Tokens [t0, t0 + part) of sequence b; a partial result goes to row hq * part_mul + part_add of the workspace.
  auto piece = [&](const int b, const int t0, const int part, const int split, const int64_t part_mul,
                   const int64_t part_add, const int n_pieces, const int raw, const int trow, const int* pre_pages) {
    int L = trow < 0 ? 0 : raw;
    const int* pages_lds = pre_pages ? pre_pages : s_pages;
    const bool beyond = L > a.max_context;  // as in paged_decode_kernel: read up to max_context, no fresh row
    if (beyond) L = a.max_context;
    if (t0 >= L) {
      if ((cut.direct || (kMerges && a.arrivals)) && split == 0) {  // no visible key at all: out = 0, lse = -inf
        for (int i = tid; i < G * D; i += kThreads) {
          const int g = i / D, d = i - g * D;
          E::store(a.out + b * a.os_b + (hc * G + g) * a.os_h + d * 2, 0.f);
        }
        if (tid < G) a.lse[static_cast<int64_t>(b) * a.Hq + hc * G + tid] = -INFINITY;
        if (kMerges && a.arrivals) clear_next_counter(a, b);
      }
      return;
    }
    const int t1 = L < t0 + part ? L : t0 + part;
    // fused append: the newest token (position L - 1) is read from k_new / v_new by the workgroup whose range ends with
    // it, and written to its slot
    const bool owns_new = a.k_new != nullptr && !beyond && t1 == L;
    const int t1_pool = owns_new ? t1 - 1 : t1;

    int64_t blk0;
    {
      int off_unused;
      int64_t blk_last;
      a.pd.split(t0, blk0, off_unused);
      a.pd.split(t1 - 1, blk_last, off_unused);
      if (!pre_pages) {
        for (int i = tid; i <= static_cast<int>(blk_last - blk0); i += kThreads) {
          int64_t page = 0;
          if (blk0 + i < a.n_pages) page = a.page_table[static_cast<int64_t>(trow) * a.pt_row_stride + blk0 + i];
          if (page < 0 || page >= a.pool_pages) page = 0;  // not a page of the pool
          s_pages[i] = static_cast<int>(page);
        }
        __syncthreads();
      }
    }
    const char* const k_new = a.k_new + b * a.kn_b + hc * a.kn_h;
    const char* const v_new = a.v_new + b * a.vn_b + hc * a.vn_h;

    // the fresh row travels to its slot through the registers of the last wavefront
    const bool stores_new = owns_new && wave == kWaves - 1 && lane < 2 * CPR;
    v4u fresh = {0, 0, 0, 0};
    if (stores_new) fresh = *reinterpret_cast<const v4u*>((lane < CPR ? k_new : v_new) + lpos * 16);

    // query rows (row of the first head where the group has fewer than 8): every wavefront brings the same bytes
    {
      const char* qrow = a.q + b * a.qs_b + hc * G * a.qs_h;
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        const int r = i * RPI + lrow;
        fp::load_to_lds(qrow + (r < G ? r : 0) * a.qs_h + lpos * 16, s_q + i * 1024);
      }
    }

    auto issue = [&](int c0, char* stage) {
      if (aligned_pages && c0 + TS <= t1_pool) {
        const int page = __builtin_amdgcn_readfirstlane(pages_lds[(c0 >> a.pd.shift) - static_cast<int>(blk0)]);
        const int64_t slot = static_cast<int64_t>(page) * a.pd.page_size + (c0 & (a.pd.page_size - 1));
#pragma unroll
        for (int i = 0; i < NI; ++i)
          fp::load_to_lds_nt(kplane + slot * ROWB, (i * RPI + lrow) * ROWB + k_off[i], stage + i * 1024);
#pragma unroll
        for (int i = 0; i < NI; ++i)
          fp::load_to_lds_nt(vplane + slot * ROWB, (i * RPI + lrow) * ROWB + v_off[i], stage + 4096 + i * 1024);
      } else {
        // the last tokens of the range, the fresh row, pages that do not hold whole stages: row by row.  A row past the
        // range repeats its last one and is masked.
        const char* ksrc[NI];
        const char* vsrc[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          int t = c0 + i * RPI + lrow;
          if (t >= t1) t = t1 - 1;
          if (t >= t1_pool) {
            ksrc[i] = k_new;
            vsrc[i] = v_new;
          } else {
            int64_t blk;
            int off;
            a.pd.split(t, blk, off);
            const int64_t slot = static_cast<int64_t>(pages_lds[blk - blk0]) * a.pd.page_size + off;
            ksrc[i] = kplane + slot * ROWB;
            vsrc[i] = vplane + slot * ROWB;
          }
        }
#pragma unroll
        for (int i = 0; i < NI; ++i) fp::load_to_lds_nt(ksrc[i] + k_off[i], stage + i * 1024);
#pragma unroll
        for (int i = 0; i < NI; ++i) fp::load_to_lds_nt(vsrc[i] + v_off[i], stage + 4096 + i * 1024);
      }
    };

    f32x4 o[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) o[db] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    v4u q[KK];

    // stages wave, wave + 4, ... of the range; the fresh row has its place in the last one
    const int n_stages = (t1 - t0 + TS - 1) / TS;
    if (wave < n_stages) issue(t0 + wave * TS, ring);
    if (wave + kWaves < n_stages) issue(t0 + (wave + kWaves) * TS, ring + kStageBytes);
#pragma nounroll
    for (int s = wave, buf = 0; s < n_stages; s += kWaves, buf ^= 1) {
      const int c0 = t0 + s * TS;
      const char* const k_lds = ring + buf * kStageBytes;
      char* const v_lds = ring + buf * kStageBytes + 4096;
      if (s + kWaves < n_stages) wait_staged<2 * NI>(); else wait_staged<0>();
      if (s == wave) {
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
          q[kk] = *reinterpret_cast<const v4u*>(s_q + (col & 7) * ROWB + (4 * kk + grp) * 16);
          if ((col & 7) >= G) q[kk] = v4u{0, 0, 0, 0};
        }
      }
      // scores of this lane's column: keys 16 * blk + 4 * grp + 0 .. 3
      float sc[NB][4];
#pragma unroll
      for (int blk = 0; blk < NB; ++blk) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        const int r = blk * 16 + col;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
          const v4u ka = *reinterpret_cast<const v4u*>(k_lds + r * ROWB + ((4 * kk + grp) ^ k_swz(r)) * 16);
          acc = E::mfma_k32(ka, q[kk], acc);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) sc[blk][j] = acc[j] * a.qscale;
      }
      if (c0 + TS > t1) {
#pragma unroll
        for (int blk = 0; blk < NB; ++blk)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (c0 + blk * 16 + grp * 4 + j >= t1) sc[blk][j] = -INFINITY;
        // their V rows, copies of the last one, become 0: a probability of 0 against an infinity would be NaN
#pragma unroll
        for (int i = 0; i < NI; ++i)
          if (c0 + i * RPI + lrow >= t1) *reinterpret_cast<v4u*>(v_lds + i * 1024 + lane * 16) = v4u{0, 0, 0, 0};
        asm volatile("" : : : "memory");  // a wavefront's LDS instructions are executed in order
      }
      // Reference point of the exponentials, per column: moves only when the column's maximum has outgrown it by
      // kMaxSlack, so most stages need no exchange between the lanes of a column and no rescale.
      float cand = sc[0][0];
#pragma unroll
      for (int blk = 0; blk < NB; ++blk)
#pragma unroll
        for (int j = 0; j < 4; ++j) cand = fmaxf(cand, sc[blk][j]);
      if (__any(cand > m + (E::kHeadroom + kMaxSlack))) {
        cand = fmaxf(cand, __shfl_xor(cand, 16));
        cand = fmaxf(cand, __shfl_xor(cand, 32));
        if (cand > m + (E::kHeadroom + kMaxSlack)) {
          const float m_new = cand - E::kHeadroom;
          const float alpha = fast_exp2(m - m_new);
          l *= alpha;
#pragma unroll
          for (int db = 0; db < DB; ++db) o[db] *= alpha;
          m = m_new;
        }
      }
      const float ms = safe_max(m);  // no key above -inf so far: its probabilities are 0
#pragma unroll
      for (int blk = 0; blk < NB; ++blk) {
        float p[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          p[j] = fast_exp2(sc[blk][j] - ms);
          l += p[j];
        }
        uint32_t w[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          w[j] = E::pack2(E::above_zero(p[2 * j]), E::above_zero(p[2 * j + 1]));
          const uint32_t rest = E::pack2(p[2 * j] - E::low(w[j]), p[2 * j + 1] - E::high(w[j]));
          if (col >= 8) w[j] = rest;
        }
        const s16x4 pb = __builtin_bit_cast(s16x4, uint2{w[0], w[1]});
        // lanes 4 j + c of a 16-lane block name elements 4 c .. of key 4 * grp + j and receive element `col` of the four keys
        const int r = blk * 16 + grp * 4 + (col >> 2);
        const char* const vrow = v_lds + r * ROWB + (col & 3) * 8;
#pragma unroll
        for (int db = 0; db < DB; ++db) o[db] = E::mfma_k16(lds_read_tr(vrow + ((db + v_rot(r)) % R32) * 32), pb, o[db]);
      }
      if (s + 2 * kWaves < n_stages) {
        asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");  // every operand of this stage has left LDS
        issue(c0 + 2 * kWaves * TS, ring + buf * kStageBytes);
      }
    }

    wait_staged<0>();  // also a wavefront without a stage has its query rows in flight

    // both halves of the columns together, then the wavefront's state to LDS (its ring is free again).  Against an infinite
    // V element what rounding left over of a probability is 0 or negative, and the sum would be NaN: the upper half stands.
    float* const acc_lds = reinterpret_cast<float*>(ring);
#pragma unroll
    for (int db = 0; db < DB; ++db) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float rest = dpp<0x128>(o[db][j]);  // row_ror:8, lane ^ 8
        if ((__float_as_uint(o[db][j]) & 0x7f800000u) != 0x7f800000u) o[db][j] += rest;
      }
      if (col < G) *reinterpret_cast<f32x4*>(acc_lds + col * D + db * 16 + grp * 4) = o[db];
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (lane < G) {
      s_ml[wave][lane][0] = m;
      s_ml[wave][lane][1] = l;
    }
    if (stores_new) {
      int64_t blk;
      int off;
      a.pd.split(t1 - 1, blk, off);
      const int64_t slot = static_cast<int64_t>(pages_lds[blk - blk0]) * a.pd.page_size + off;
      char* dst = const_cast<char*>(lane < CPR ? kplane : vplane) + slot * ROWB + lpos * 16;
      __builtin_nontemporal_store(fresh, reinterpret_cast<v4u*>(dst));
    }
    __syncthreads();

    // combine the wavefronts; one thread per (head of the group, element)
    const DecodeArgs& e = reread_args();
    const bool merges = kMerges && e.arrivals != nullptr;
    const bool direct = cut.direct || (merges && n_pieces == 1);  // the only piece: out and lse, no partial result
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
        num += reinterpret_cast<const float*>(s_ring + w * (kStages * kStageBytes))[i] * wgt;
        den += s_ml[w][g][1] * wgt;
      }
      const int hq = hc * G + g;
      if (direct) {
        const float lse_nat = (mn + log2f(den)) * kLn2;
        E::store(e.out + b * e.os_b + hq * e.os_h + d * 2, sink_gate<E>(num / den, lse_nat, e.sinks, hq));
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
    if constexpr (kMerges) {  // the rings are free behind the barrier inside
      if (merges && split == 0) clear_next_counter(e, b);
      __shared__ int s_last;
      if (merges && !direct && last_to_arrive(b, n_pieces, &s_last)) merge_splits<E, D>(b, part_mul, part_add - split, n_pieces, G, reinterpret_cast<float*>(s_ring));
    }
  };  // piece

  if constexpr (kFlat) {
    __shared__ int s_start[kFlatMaxB + 1];
    walk_even_cut<kThreads>(a, s_start, s_pages, piece);
  } else if constexpr (kPieces) {
    walk_pieces<min_part(ROWB)>(a, piece);
  } else {
    walk_split<kMerges>(a, piece);
  }
}

template <typename E, int D>
void launch(const DecodeArgs& a, const Cut& cut, dim3 grid, hipStream_t st) {
  if (cut.flat)
    hipLaunchKernelGGL((paged_decode_mfma_kernel<E, D, true>), grid, dim3(kThreads), 0, st, a, cut);
  else if (merges_itself(4, D) && cut.pieces)
    hipLaunchKernelGGL((paged_decode_mfma_kernel<E, D, false, merges_itself(4, D)>), grid, dim3(kThreads), 0, st, a, cut);
  else
    hipLaunchKernelGGL((paged_decode_mfma_kernel<E, D, false>), grid, dim3(kThreads), 0, st, a, cut);
}

template <typename E>
int dispatch(const DecodeArgs& a, int D, const Cut& cut, dim3 grid, hipStream_t st) {
  if (D == 64)
    launch<E, 64>(a, cut, grid, st);
  else
    launch<E, 128>(a, cut, grid, st);
  return FP_OK;
}

}  // namespace

int fp_decode::launch_mfma(const DecodeArgs& a, int dtype, int D, const Cut& cut, dim3 grid, hipStream_t st) {
  return dtype == FP_DTYPE_BF16 ? dispatch<BF16>(a, D, cut, grid, st) : dispatch<F16>(a, D, cut, grid, st);
}
