// Chunked-prefill attention over the paged cache under the hybrid mask, fp32 (the reference's
// default dtype, server/config.py:38) on the bf16 matrix instruction: every operand as three bf16 numbers.
//
// Same contract as the bf16 / f16 kernel (paged_prefill.hip; reference attention.py:18 as called
// at model.py:156-162, mask paged_attention.py:343-362): row r of the packed queries sees keys
// 0 .. row_limit[r] - 1 of sequence batch_idx[r], fetched through the page table.
//
// MFMA-bound.  The fp32 matrix instruction does a sixteenth of the bf16 one's work per cycle.  An fp32 number is exactly the sum of three
// bf16 numbers, each the rounding of what the ones before leave (x = x1 + x2 + x3), so a product of two is six bf16 products
// and a rest of 2^-26: k1 q1 + (k1 q2 + k2 q1) + (k1 q3 + k2 q2 + k3 q1), 6 / 16 of the cycles (the method of G. Henry, P. T. P. Tang and
// A. Heinecke, "Leveraging the bfloat16 artificial intelligence datatype for higher-precision computations", 2019).  Sums stay in the instruction's
// fp32 accumulators; in the scores the five small products have accumulators of their own, so that the large one is rounded
// D / 16 times.  K, V and Q are all kept to their 24 bits, and so are probabilities from 2^-100 on; of a smaller one less than 2^-125 is lost.
// us a launch with its merge on the fp32 instruction / so, 16 heads, D 128: whole sequences of 5376 rows 681 / 488, of 17920 2909 /
// 1924 (126 / 190 TFLOP/s: 1.14 PFLOP/s of bf16 products, the rate of a large matrix product here, 1.18 to 1.23), 8 chunks of 512 rows on 8
// cache heads 823 / 570, D 64 390 / 284; relative error against float64 5.7e-7 / 4.6e-7, 8.6e-7 / 6.9e-7, 5.2e-7 / 3.9e-7 and 4.9e-7 / 4.5e-7.
// A workgroup of 8 wavefronts owns one cache head and 256 / G packed query rows of each of its G query heads, a wavefront 32 rows of
// one head.  K/V tiles travel through registers, where they are split (once per workgroup), into three bf16 planes each in LDS,
// double-buffered, one barrier per tile; rows of a plane are laid out and read as in the bf16 kernel.
//   S^T = K Q^T : a lane holds the scores of ONE query (softmax reductions stay in registers plus
//                 one exchange between the lane halves); Q is scaled when it is loaded.
//   O^T = V^T P^T : P^T is the B operand as it leaves the softmax; V^T comes out of LDS through ds_read_b64_tr_b16.
// A run with an infinity, a NaN, or a number too large or too small for the split (from the largest bf16 on, in K and Q from 2^60 on; below
// 2^-100) in a tile or in a row of Q is done again on the fp32 matrix instruction, from the start of the run (a V of 2^-110 in the first / last tile
// of every sequence, all heads: whole sequences of 5376 rows 501 us without, 574 / 588 with it, 8 chunks 536, 577 / 780, D 64 264, 290 / 324).
#include "fp_common.h"
#include "prefill_common.h"

#include <math.h>

namespace {

using fp::load_to_lds;

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * 64;
constexpr int kExactTileN = 32;    // keys per tile of a run on the fp32 matrix instruction
constexpr float kMaxSlack = 6.f;   // the running maximum may lag a row's true maximum by this much (log2)
constexpr int kSlotTable = 4096;   // tiles of a run whose first pool slot is looked up ahead of the tile loop
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) const char* lds_ptr;  // a 32-bit LDS address
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr f32x16 kZero16 = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

template <int N>
struct IntC {
  static constexpr int value = N;
};

struct Args {
  const char* q;
  int64_t qs_row, qs_h;  // bytes
  const char* pool_k;
  const char* pool_v;
  const int64_t* page_table;
  int64_t pt_row_stride;
  const int64_t* batch_idx;
  const int32_t* row_limit;
  char* out;
  int64_t os_row, os_h;  // bytes
  float* lse;            // [Hq, Lq]
  const float* sinks;    // optional [Hq]: out is multiplied by sigmoid(lse - sinks[h])
  int Lq, Hq, Hc;
  fp::PageDiv pd;
  int n_pages, max_batch;
  int64_t n_slots, pool_pages;
  float qscale;  // scale * log2(e)
  int n_tiles;   // query tiles
  // key shares (grid z): unnormalised partial results for the merge pass, as in the bf16 / f16 kernel
  float* ws_acc;  // [shares, Lq, Hq, D]
  float* ws_ml;   // [shares, Lq, Hq, 2]: running maximum (log2 units), denominator
};

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ f32x16 mfma(float a, float b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 mfma(const v4u& a, const v4u& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ s16x4 lds_read_tr(lds_ptr p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p));
}

__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  const bf16x2 v = {static_cast<__bf16>(lo), static_cast<__bf16>(hi)};
  return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ float low(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float high(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// Eight numbers as three bf16 vectors whose sum they are.  What a rounding leaves is x minus one half of a packed pair, a dot product
// with (-1, 0) or (0, -1) added to x: exact, and one instruction instead of two.
struct Split {
  v4u p[3];
};
__device__ __forceinline__ Split split(const float (&x)[8]) {
  // in registers: as a constant in the instruction, (-1, 0) came out as (0, -1)
  uint32_t lo_bits = 0x0000bf80u, hi_bits = 0xbf800000u;
  asm("" : "+s"(lo_bits), "+s"(hi_bits));
  const bf16x2 minus_lo = __builtin_bit_cast(bf16x2, lo_bits), minus_hi = __builtin_bit_cast(bf16x2, hi_bits);
  Split r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float lo = x[2 * i], hi = x[2 * i + 1];
#pragma unroll
    for (int n = 0; n < 3; ++n) {
      const uint32_t w = pack2(lo, hi);
      r.p[n][i] = w;
      lo = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w), minus_lo, lo, false);
      hi = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w), minus_hi, hi, false);
    }
  }
  return r;
}
// Whether one of the numbers is out of the split's range, by its first part: an infinity or a NaN, or below 2^-100 and not 0 (what
// rounds to 0 is below 2^-134).  K and Q also from 2^60 on (kScoreTooLarge): below, no sum of up to 128 products leaves fp32.  Beyond, the
// large and the small products of a score may overflow to opposite infinities, a NaN where plain fp32 has -inf and no weight.
constexpr uint32_t kTooLarge = 0x7f80u, kScoreTooLarge = (127u + 60u) << 7, kTooSmall = 0x0d80u;
__device__ __forceinline__ bool out_of_range(const Split& s, uint32_t too_large) {
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  const u16x2 one = {1, 1};
  u16x2 most = {0, 0}, least = {0xffff, 0xffff};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t w = s.p[0][i] & 0x7fff7fffu;
    const u16x2 b = __builtin_bit_cast(u16x2, w);
    most = __builtin_elementwise_max(most, b);
    least = __builtin_elementwise_min(least, static_cast<u16x2>(b - one));  // 0 comes out above everything
  }
  return max(most.x, most.y) >= too_large || min(least.x, least.y) < kTooSmall - 1u;
}

// LDS layout of a plane of a tile: unpadded rows of D bf16, whose 16-byte chunks are permuted against bank conflicts as in the
// bf16 kernel: K chunk c of row r at position c ^ kswz(r) (the score product reads one chunk of 16 consecutive rows), V's 32-byte
// region c of row r at (c + vrot(r)) % regions (a transpose read takes 4 consecutive rows x 32 bytes per 16-lane block).
template <int D>
struct Swizzle {
  static constexpr int CPR = D * 2 / 16;  // 16-byte chunks per row
  static constexpr int R32 = CPR / 2;     // 32-byte regions per row
  static __device__ __forceinline__ int kswz(int r) { return (r / (16 / CPR)) % CPR; }
  static __device__ __forceinline__ int vrot(int r) { return (2 * ((r / (8 / R32)) & 3)) % R32; }
};

template <int D, int G, bool kPow2>
__global__ __launch_bounds__(kThreads, 2) void paged_prefill_f32_kernel(const Args a) {
  constexpr int RB = kWaves / G;           // 32-row blocks per workgroup
  constexpr int BM = RB * 32;              // query rows per workgroup
  using SW = Swizzle<D>;
  constexpr int ROWB = D * 4;              // bytes of a K/V row in the pool
  constexpr int PROWB = D * 2;             // and of a plane in LDS
  constexpr int LPR = D / 8;               // lanes that bring in a row, 32 bytes each
  constexpr int RPW = 64 / LPR;            // rows a wavefront stages
  constexpr int kTileN = kWaves * RPW;     // keys per tile: 32 at head_dim 128, 64 at head_dim 64
  constexpr int KB = kTileN / 32;          // 32-key blocks of a tile
  constexpr int DS = D / 16;               // MFMA k-steps over head_dim
  constexpr int DB = D / 32;               // 32-wide blocks of head_dim in O^T
  constexpr int R32 = SW::R32;
  constexpr int PLANE = kTileN * PROWB;    // 8 KB
  constexpr int TILE_BYTES = 3 * PLANE;

  __shared__ __attribute__((aligned(1024))) char s_k[2 * TILE_BYTES];
  __shared__ __attribute__((aligned(1024))) char s_v[2 * TILE_BYTES];
  __shared__ int s_bad[2];  // the tile on its way into this buffer (0: or a row of Q) is out of the split's range
  __shared__ int s_bidx[BM];
  __shared__ int s_red[kWaves];
  __shared__ int s_tslot[kSlotTable];

  // linear id = cache head + Hc * tile: all tiles that read one cache head run on the XCD that
  // already holds its K/V in L2
  const int hc = blockIdx.x;
  const int tile = a.n_tiles - 1 - blockIdx.y;  // later rows see more keys: longest first
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hq = hc * G + wave % G;  // query head of this wavefront
  const int rblock = wave / G;       // its block of 32 rows inside the tile
  const int lane = tid & 63;
  const int half = lane >> 5;   // which of the 2 k-values of an MFMA step this lane holds
  const int ln = lane & 31;     // query column (S^T, O^T), key row (K operand) or head_dim row (V operand)
  const int tile0 = tile * BM;

  // Everything the set-up needs from global memory is requested at once: the sequence of each row
  // of the tile, then this wavefront's row limit and Q row.
  const int bi_row = tile0 + tid;
  const int64_t bx_raw = (tid < BM && bi_row < a.Lq) ? a.batch_idx[bi_row] : 0;
  if (tid < BM) {
    int64_t bx = bx_raw;
    if (bx < 0 || bx >= a.max_batch) bx = 0;
    s_bidx[tid] = static_cast<int>(bx);
  }
  __syncthreads();

  const char* kplane = a.pool_k + static_cast<int64_t>(hc) * a.n_slots * ROWB;
  const char* vplane = a.pool_v + static_cast<int64_t>(hc) * a.n_slots * ROWB;

  // ---- what a lane stages and reads ----
  // These numbers follow from the thread's id in a few instructions and are made where they are used: kept, they would not fit beside
  // Q and the accumulators.
  auto thread = [&] {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
  };
  // A lane brings 8 numbers of row `row` of a tile: 16-byte chunk `chunk` of a plane's row.
  struct Place {
    int row, chunk;
  };
  auto staged = [&] {
    const int t = thread();
    return Place{(t >> 6) * RPW + (t & 63) / LPR, (t & 63) % LPR};
  };

  int run0 = 0;
  while (run0 < BM) {
    const int tid = thread(), lane = tid & 63, half = lane >> 5, ln = lane & 31;
    // values every lane agrees on are moved to scalar registers so the control flow that
    // depends on them stays uniform
    const int sq = __builtin_amdgcn_readfirstlane(s_bidx[run0]);
    // end of the run: the first row of another sequence, found 64 rows at a time
    int run1 = BM;
    for (int base = run0; base < BM; base += 64) {
      const int idx = base + lane;
      const unsigned long long other = __ballot(idx < BM && s_bidx[idx] != sq);
      if (other != 0) {
        run1 = base + __builtin_ctzll(other);
        break;
      }
    }
    run1 = __builtin_amdgcn_readfirstlane(run1);

    const int tr = rblock * 32 + ln, row = tile0 + tr;  // this lane's row inside the tile
    const bool active = tr >= run0 && tr < run1 && row < a.Lq;
    int lim = (active && sq != 0) ? a.row_limit[row] : 0;
    if (lim < 0) lim = 0;

    if (sq == 0) {
      const int th = thread(), row = tile0 + rblock * 32 + (th & 31), half = (th >> 5) & 1;
      // padding rows: out = 0, lse = -inf; each lane half clears half of the row
      if (active && gridDim.z > 1) {  // an empty share; the merge pass then writes out = 0, lse = -inf
        const int64_t p = (static_cast<int64_t>(blockIdx.z) * a.Lq + row) * a.Hq + hq;
#pragma unroll
        for (int c = 0; c < D / 8; ++c) *reinterpret_cast<f32x4*>(a.ws_acc + p * D + half * (D / 2) + c * 4) = f32x4{0, 0, 0, 0};
        if (half == 0) *reinterpret_cast<float2*>(a.ws_ml + p * 2) = float2{-INFINITY, 0.f};
      } else if (active) {
        float* o = reinterpret_cast<float*>(a.out + row * a.os_row + hq * a.os_h) + half * (D / 2);
#pragma unroll
        for (int c = 0; c < D / 2; ++c) o[c] = 0.f;
        if (half == 0) a.lse[static_cast<int64_t>(hq) * a.Lq + row] = -INFINITY;
      }
      run0 = run1;
      continue;
    }

    // key range of the run: wavefront maximum, then workgroup maximum
    int wave_max = lim;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) wave_max = max(wave_max, __shfl_xor(wave_max, off));
    wave_max = __builtin_amdgcn_readfirstlane(wave_max);
    int wave_min = active ? lim : 0x7fffffff;  // smallest limit among the active rows (tiles below it need no masking)
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) wave_min = min(wave_min, __shfl_xor(wave_min, off));
    wave_min = __builtin_amdgcn_readfirstlane(wave_min);
    __syncthreads();  // s_red, s_tslot and the LDS tiles of the previous run are free
    if (lane == 0) s_red[wave] = wave_max;
    if (tid < 2) s_bad[tid] = 0;
    __syncthreads();
    int kv_max = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) kv_max = max(kv_max, s_red[w]);
    kv_max = __builtin_amdgcn_readfirstlane(kv_max);
    const int n_run_tiles = (kv_max + kTileN - 1) / kTileN;
    // this workgroup's share of the run's key tiles: [kt_lo, n_kv_tiles)
    uint32_t n_shares = gridDim.z;  // at most 8, and fewer than 2^26 tiles
    asm volatile("" : "+s"(n_shares));  // its reciprocal is not kept in a register through the runs
    const int kt_lo = static_cast<int>(n_run_tiles * blockIdx.z / n_shares);
    const int n_kv_tiles = static_cast<int>(n_run_tiles * (blockIdx.z + 1) / n_shares);

    f32x16 o_acc[DB];
    float m_run, l_run;

    // ---- K/V fetch pipeline ----
    // Every lane brings 32 bytes of a K and of a V row of each tile, requested while the tile before is worked on.  Where a page holds whole
    // tiles (page size a power of two, at least the tile), a tile that lies before the run's last key in a
    // mapped page is contiguous in the pool: its first slot is looked up once per run into s_tslot.  Any other tile (the
    // last one of a run, small or odd page sizes, unmapped pages, runs longer than the table) looks its rows up one by
    // one: a row past the run's last key is 0, and masked; a key below it on a page that is not mapped reads slot 0 of the
    // pool, here and on the fp32 matrix instruction.
    const int64_t* pt_row = a.page_table + static_cast<int64_t>(sq) * a.pt_row_stride;
    const int64_t pool_pages = a.pool_pages;
    // first pool slots of tiles lo .. hi - 1 of n keys each -> s_tslot
    auto look_up_tiles = [&](int lo, int hi, int n) {
      const bool page_holds_tile = kPow2 && a.pd.page_size % n == 0;
      for (int t = lo + tid; t < hi && t - lo < kSlotTable; t += kThreads) {
        int slot = -1;
        if (page_holds_tile && (t + 1) * n <= kv_max) {
          const int key0 = t * n;
          const int blk = key0 >> a.pd.shift;
          if (blk < a.n_pages) {
            const int64_t pg = pt_row[blk];
            if (pg >= 0 && pg < pool_pages) slot = static_cast<int>(pg) * a.pd.page_size + (key0 & (a.pd.page_size - 1));
          }
        }
        s_tslot[t - lo] = slot;
      }
    };
    look_up_tiles(kt_lo, n_kv_tiles, kTileN);
    // first pool slot of tile t of lo .. hi - 1, or -1: wavefront-uniform
    auto tile_slot = [&](int t, int lo, int hi) {
      return __builtin_amdgcn_readfirstlane((t >= lo && t < hi && t - lo < kSlotTable) ? s_tslot[t - lo] : -1);
    };
    auto key_block = [&](int kpos, int& blkid, int& off) {
      if (kPow2) {  // page size is a power of two: shift and mask, no branch on the page size
        blkid = kpos >> a.pd.shift;
        off = kpos & (a.pd.page_size - 1);
      } else {
        int page_size = a.pd.page_size;
        asm volatile("" : "+s"(page_size));  // its reciprocal is not kept in a register
        blkid = kpos / page_size;
        off = kpos - blkid * page_size;
      }
    };
    // Byte offset of this lane's row of tile kt in a plane of the pool, or -1: past the run's last key.
    auto row_offset = [&](int kt) -> int64_t {
      const int ts = tile_slot(kt, kt_lo, n_kv_tiles);
      const Place at = staged();
      if (ts >= 0) return static_cast<int64_t>(ts) * ROWB + (at.row * ROWB + at.chunk * 32);
      asm volatile("");  // rare: keep it out of the way as a branch
      const int kpos = kt * kTileN + at.row;
      int blkid, off;
      key_block(kpos, blkid, off);
      if (kpos >= kv_max) return -1;
      const int64_t pg = blkid < a.n_pages ? pt_row[blkid] : -1;
      const int64_t slot = pg >= 0 && pg < pool_pages ? pg * a.pd.page_size + off : 0;
      return slot * ROWB + at.chunk * 32;
    };
    struct Raw {
      f32x4 lo, hi;
    };
    auto fetch = [&](const char* plane, int64_t off) {
      Raw r{{0, 0, 0, 0}, {0, 0, 0, 0}};
      if (off >= 0) {
        r.lo = *reinterpret_cast<const f32x4*>(plane + off);
        r.hi = *reinterpret_cast<const f32x4*>(plane + off + 16);
      }
      return r;
    };
    // 4 numbers of this lane's query row from head_dim element d on, scaled.  Rows of other sequences count as 0: what they hold neither
    // sends this run through the fp32 instruction nor moves its reference points.
    auto load_q = [&](int d, float* x) {
      f32x4 w = {0, 0, 0, 0};
      const int tr = rblock * 32 + (thread() & 31), r = tile0 + tr;
      if (tr >= run0 && tr < run1 && r < a.Lq) w = *reinterpret_cast<const f32x4*>(a.q + r * a.qs_row + hq * a.qs_h + d * 4);
#pragma unroll
      for (int t = 0; t < 4; ++t) x[t] = w[t] * a.qscale;
    };
    // Online softmax of a tile from key0 on, one query per lane; score x of block kb is key kb * 32 + (x / 4) * 8 + half * 4 + x % 4.
    // Scores become probabilities; returns the factor the accumulators have to take, or -1: none.
    auto softmax = [&](auto& sc, int key0) {
      constexpr int N = sizeof(sc) / sizeof(float);
      if (key0 + N * 2 > wave_min) {
        asm volatile("");  // keeps this a branch: turned into selects it would run on every tile
        const int rel = lim - key0 - half * 4;
#pragma unroll
        for (int x = 0; x < N; ++x) sc[x] = ((x >> 4) * 32 + ((x & 15) >> 2) * 8 + (x & 3)) < rel ? sc[x] : -INFINITY;
      }
      float mx = sc[0];
#pragma unroll
      for (int x = 1; x < N; ++x) mx = fmaxf(mx, sc[x]);
      mx = fp::max_across_lane_halves(mx);
      // Lazy running maximum: the reference point m_run only moves when some row's maximum has grown by
      // more than kMaxSlack (log2 units); until then exp2(s - m_run) may reach 2^kMaxSlack, harmless in
      // fp32, and the accumulators need no rescale.
      const bool moved = __any(mx > m_run + kMaxSlack);
      const float m_new = moved ? fmaxf(m_run, mx) : m_run;
      const float m_safe = m_new == -INFINITY ? 0.f : m_new;
      const float alpha = moved ? fast_exp2(m_run - m_safe) : 1.f;
      m_run = m_new;
      float psum = 0.f;
#pragma unroll
      for (int x = 0; x < N; ++x) {
        sc[x] = fast_exp2(sc[x] - m_safe);
        psum += sc[x];
      }
      l_run = fmaf(l_run, alpha, psum);  // alpha is 1 unless the reference point moved
      return moved ? alpha : -1.f;
    };
    // Splits what fetch brought into the three planes of a tile.
    auto put = [&](const Raw& r, char* tile, bool is_k, int buf, int word) {
      float x[8];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        x[t] = r.lo[t];
        x[4 + t] = r.hi[t];
      }
      const Place at = staged();
      char* const dst = tile + buf * TILE_BYTES + at.row * PROWB +
                        (is_k ? (at.chunk ^ SW::kswz(at.row)) * 16
                              : (((at.chunk >> 1) + SW::vrot(at.row)) % R32) * 32 + (at.chunk & 1) * 16);
      const Split s = split(x);
      if (out_of_range(s, is_k ? kScoreTooLarge : kTooLarge)) s_bad[word] = 1;
#pragma unroll
      for (int n = 0; n < 3; ++n) *reinterpret_cast<v4u*>(dst + n * PLANE) = s.p[n];
    };

    bool bad = false;
    {
      // Q^T operands, scaled: lane (query ln, half) holds d = 16 ds + 8 half .. + 7 of k-step ds
      Split qreg[DS];
#pragma unroll
      for (int ds = 0; ds < DS; ++ds) {
        float x[8];
        load_q(16 * ds + 8 * half, x);
        load_q(16 * ds + 8 * half + 4, x + 4);
        qreg[ds] = split(x);
        if (out_of_range(qreg[ds], kScoreTooLarge)) s_bad[1] = 1;
      }
      __builtin_amdgcn_sched_barrier(0);  // not before: Q as it came and split fills the registers
      m_run = -INFINITY;
      l_run = 0.f;
#pragma unroll
      for (int db = 0; db < DB; ++db) o_acc[db] = kZero16;
      __syncthreads();  // the slot table
      put(fetch(kplane, row_offset(kt_lo)), s_k, true, 0, 1);

      // ---- schedule ----
      // Step i of a wavefront is M(i) = { O^T += V^T P^T of tile i - 1;  S^T = K Q^T of tile i } on the matrix pipe and X(i) = softmax
      // of tile i on the vector pipe.  The two wavefronts that share a SIMD (w and w + 4) run
      // half a step apart: between two barriers the first half does M(i) then X(i), the second half X(i - 1) then M(i) (8 chunks of 512 rows
      // 505 us, 555 us in step; whole sequences 431 and 435).  In step i
      // a wavefront also splits its rows of K of tile i + 1 and of V of tile i into LDS, each requested one product ahead.  K(i)
      // lives in K buffer i % 2, V(i) in V buffer i % 2.
      const int n_my = n_kv_tiles - kt_lo;
      float sc[KB * 16];
      auto works = [&](int i) { return i >= 0 && i < n_my && (kt_lo + i) * kTileN < wave_max; };
      auto fetch_k = [&](int i) { return fetch(kplane, i + 1 < n_my ? row_offset(kt_lo + i + 1) : -1); };
      auto matrix_part = [&](auto parity, int i, const Raw& kr) __attribute__((always_inline)) {
        constexpr int kBuf = decltype(parity)::value;
        if (works(i - 1)) {
          asm volatile("");
          // ---- O^T += V^T P^T: k-step j pairs scores 8 j .. 8 j + 7 of a lane with the same keys of V ----
          // V operand of step (j, db): this lane names 8 bytes of region 2 db + (16-lane block) % 2 of row 16 j + 4 half + lane % 16 / 4 and,
          // for its other four keys, of the row 8 on.  Every plane's operand is asked for again as soon as its last product is on its way.
          const int th = thread();
          const int vrow = ((th >> 5) & 1) * 4 + ((th & 15) >> 2), vsel = ((th >> 4) & 1) + SW::vrot(vrow);
          const lds_ptr vrow_at = (lds_ptr)s_v + vrow * PROWB + (th & 3) * 8;
          auto read_v = [&](int t, int n) {
            const lds_ptr p0 = vrow_at + ((2 * (t % DB) + vsel) % R32) * 32 + (1 - kBuf) * TILE_BYTES + n * PLANE + t / DB * 16 * PROWB;
            const uint2 lo = __builtin_bit_cast(uint2, lds_read_tr(p0)), hi = __builtin_bit_cast(uint2, lds_read_tr(p0 + 8 * PROWB));
            return v4u{lo.x, lo.y, hi.x, hi.y};
          };
          v4u v0 = read_v(0, 0), v1 = read_v(0, 1), v2 = read_v(0, 2);
          Split p;
#pragma unroll
          for (int t = 0; t < 2 * KB * DB; ++t) {
            const int j = t / DB, db = t % DB;
            const bool next = t + 1 < 2 * KB * DB;
            if (db == 0) {
              float x[8];
#pragma unroll
              for (int e = 0; e < 8; ++e) x[e] = sc[8 * j + e];
              p = split(x);
            }
            o_acc[db] = mfma(v2, p.p[0], o_acc[db]);
            if (next) v2 = read_v(t + 1, 2);
            o_acc[db] = mfma(v1, p.p[1], o_acc[db]);
            o_acc[db] = mfma(v1, p.p[0], o_acc[db]);
            if (next) v1 = read_v(t + 1, 1);
            o_acc[db] = mfma(v0, p.p[2], o_acc[db]);
            o_acc[db] = mfma(v0, p.p[1], o_acc[db]);
            o_acc[db] = mfma(v0, p.p[0], o_acc[db]);
            if (next) v0 = read_v(t + 1, 0);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        if (i + 1 < n_my) put(kr, s_k, true, 1 - kBuf, kBuf);
        const Raw vr = fetch(vplane, i < n_my ? row_offset(kt_lo + i) : -1);
        if (works(i)) {
          asm volatile("");
          // ---- S^T = K Q^T ----
          // K operand of k-step ds: row kb * 32 + lane % 32, chunk 2 ds + half at position (2 ds) ^ (half ^ kswz)
          f32x16 s_acc[KB], small[KB];
          const int th = thread();
          const int kofs = (th & 31) * PROWB + (((th >> 5) & 1) ^ SW::kswz(th & 31)) * 16;
          auto read_k = [&](int t, int n) {
            return *reinterpret_cast<__attribute__((address_space(3))) const v4u*>((lds_ptr)s_k + (kofs ^ (32 * (t / KB))) + kBuf * TILE_BYTES + n * PLANE + (t % KB) * 32 * PROWB);
          };
          v4u k0 = read_k(0, 0), k1 = read_k(0, 1), k2 = read_k(0, 2);
#pragma unroll
          for (int t = 0; t < KB * DS; ++t) {
            const int kb = t % KB, ds = t / KB;
            const bool next = t + 1 < KB * DS;
            const Split& q = qreg[ds];
            small[kb] = mfma(k2, q.p[0], ds == 0 ? kZero16 : small[kb]);
            if (next) k2 = read_k(t + 1, 2);
            small[kb] = mfma(k1, q.p[1], small[kb]);
            small[kb] = mfma(k1, q.p[0], small[kb]);
            if (next) k1 = read_k(t + 1, 1);
            small[kb] = mfma(k0, q.p[2], small[kb]);
            small[kb] = mfma(k0, q.p[1], small[kb]);
            s_acc[kb] = mfma(k0, q.p[0], ds == 0 ? kZero16 : s_acc[kb]);
            if (next) k0 = read_k(t + 1, 0);
            __builtin_amdgcn_sched_barrier(0);
          }
#pragma unroll
          for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int x = 0; x < 16; ++x) sc[kb * 16 + x] = s_acc[kb][x] + small[kb][x];
        } else {  // also here a new value: the old ones are not kept through the products above
#pragma unroll
          for (int x = 0; x < KB * 16; ++x) sc[x] = 0.f;
        }
        if (i < n_my) put(vr, s_v, false, kBuf, kBuf);
      };
      auto vector_part = [&](int i) __attribute__((always_inline)) {
        if (!works(i)) return;
        asm volatile("");
        const float alpha = softmax(sc, (kt_lo + i) * kTileN);
        if (alpha >= 0.f) {
          asm volatile("");  // the rescale is rare and must not run unconditionally
#pragma unroll
          for (int db = 0; db < DB; ++db) o_acc[db] *= alpha;
        }
      };
      // Steps 0 .. n_my, the last one without a tile of its own.  A tile out of the split's range ends the loop, and the run is done
      // again below.  All wavefronts leave at the same step: the word of a step is written in it, read in the next and written
      // again in the one after that.
      auto step = [&](auto second, auto parity, int i) __attribute__((always_inline)) {
        __syncthreads();
        bad = __builtin_amdgcn_readfirstlane(s_bad[1 - decltype(parity)::value]) != 0;
        if (bad) return;
        const Raw kr = fetch_k(i);
        if (decltype(second)::value) vector_part(i - 1);
        matrix_part(parity, i, kr);
        if (!decltype(second)::value) vector_part(i);
      };
      if (wave < kWaves / 2) {
        for (int i = 0; i <= n_my && !bad; i += 2) {
          step(IntC<0>{}, IntC<0>{}, i);
          if (!bad && i + 1 <= n_my) step(IntC<0>{}, IntC<1>{}, i + 1);
        }
      } else {
        for (int i = 0; i <= n_my && !bad; i += 2) {
          step(IntC<1>{}, IntC<0>{}, i);
          if (!bad && i + 1 <= n_my) step(IntC<1>{}, IntC<1>{}, i + 1);
        }
      }
    }

    if (bad) {
      asm volatile("");
      // ---- the run on the fp32 matrix instruction: tiles of 32 keys, whole numbers in LDS ----
      m_run = -INFINITY;
      l_run = 0.f;
#pragma unroll
      for (int db = 0; db < DB; ++db) o_acc[db] = kZero16;
      const int xt_lo = kt_lo * (kTileN / kExactTileN);
      const int xt_hi = min(n_kv_tiles * (kTileN / kExactTileN), (kv_max + kExactTileN - 1) / kExactTileN);
      constexpr int XCPR = ROWB / 16;               // 16-byte chunks per row
      constexpr int XRPI = 64 / XCPR;               // rows one wavefront load instruction brings in
      constexpr int NI = kExactTileN / (XRPI * kWaves);
      constexpr int X_BYTES = kExactTileN * ROWB;
      static_assert(NI >= 1 && 2 * X_BYTES <= 2 * TILE_BYTES, "two tiles of whole numbers fit");
      // The 16-byte chunks of a row are permuted on the GLOBAL side of the load so that the operand reads meet no bank conflict: K chunk c
      // of row r at c ^ (r % 16) (S^T takes one chunk of 16 consecutive rows at a time), V's at c ^ 8 when (r / 4) is odd (O^T takes
      // 32 consecutive floats of row k in one lane half and of row k + 4 in the other).
      const int xrow = wave * XRPI + lane / XCPR, xlp = lane % XCPR;
      const uint32_t x_k = xrow * ROWB + (xlp ^ (xrow & 15)) * 16;
      const uint32_t x_v = xrow * ROWB + (xlp ^ (((xrow >> 2) & 1) << 3)) * 16;
      __syncthreads();
      look_up_tiles(xt_lo, xt_hi, kExactTileN);
      __syncthreads();
      f32x4 qx[D / 8];  // lane (query ln, half) holds d = 8 c + 4 half .. + 3 of group c
#pragma unroll
      for (int c = 0; c < D / 8; ++c) {
        float x[4];
        load_q(8 * c + 4 * half, x);
        qx[c] = f32x4{x[0], x[1], x[2], x[3]};
      }
      auto stage = [&](int t, int buf) {
        if (t >= xt_hi) return;
        const int ts = tile_slot(t, xt_lo, xt_hi);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          char* const kdst = s_k + buf * X_BYTES + (i * kWaves + wave) * XRPI * ROWB;  // wavefront-uniform
          char* const vdst = s_v + buf * X_BYTES + (i * kWaves + wave) * XRPI * ROWB;
          if (ts >= 0) {
            const int64_t base = (static_cast<int64_t>(ts) + i * kWaves * XRPI) * ROWB;
            load_to_lds(kplane + base, x_k, kdst);
            load_to_lds(vplane + base, x_v, vdst);
          } else {
            const int kpos = t * kExactTileN + i * kWaves * XRPI + xrow;
            int blkid, off;
            key_block(kpos, blkid, off);
            const bool in_range = kpos < kv_max && blkid < a.n_pages;
            const int64_t pg = pt_row[in_range ? blkid : 0];
            const bool ok = in_range && pg >= 0 && pg < pool_pages;
            const int64_t rowbyte = static_cast<int64_t>(ok ? static_cast<int>(pg) * a.pd.page_size + off : 0) * ROWB;
            load_to_lds(kplane + rowbyte + x_k - xrow * ROWB, kdst);
            load_to_lds(vplane + rowbyte + x_v - xrow * ROWB, vdst);
          }
        }
      };
      stage(xt_lo, 0);
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wavefront's rows have landed in LDS
      __syncthreads();
#pragma nounroll
      for (int t = xt_lo, buf = 0; t < xt_hi; ++t, buf ^= 1) {
        const lds_ptr kcur = (lds_ptr)(s_k + buf * X_BYTES);
        const lds_ptr vcur = (lds_ptr)(s_v + buf * X_BYTES);
        stage(t + 1, buf ^ 1);
        const int key0 = t * kExactTileN;
        if (key0 < wave_max) {
          f32x16 s_acc = kZero16;
          const uint32_t kx = ln * ROWB + (half ^ (ln & 15)) * 16;
#pragma unroll
          for (int c = 0; c < D / 8; ++c) {
            const f32x4 kv = *reinterpret_cast<__attribute__((address_space(3))) const f32x4*>(kcur + (kx ^ (32u * c)));
#pragma unroll
            for (int e = 0; e < 4; ++e) s_acc = mfma(kv[e], qx[c][e], s_acc);
            __builtin_amdgcn_sched_barrier(0);
          }
          float sc[16];
#pragma unroll
          for (int x = 0; x < 16; ++x) sc[x] = s_acc[x];
          const float alpha = softmax(sc, key0);
          if (alpha >= 0.f) {
#pragma unroll
            for (int db = 0; db < DB; ++db) o_acc[db] *= alpha;
          }
          // score x pairs key (x / 4) * 8 + x % 4 (first lane half) with the key 4 rows on
#pragma unroll
          for (int x = 0; x < 16; ++x) {
#pragma unroll
            for (int db = 0; db < DB; ++db) {
              const uint32_t vx = half * 4 * ROWB + (((db * 8 + (ln >> 2)) ^ (half * 8)) * 16) + (ln & 3) * 4;
              const float va = *reinterpret_cast<__attribute__((address_space(3))) const float*>(vcur + vx + ((x >> 2) * 8 + (x & 3)) * ROWB);
              o_acc[db] = mfma(va, sc[x], o_acc[db]);
            }
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);  // this wavefront's share of the next tile has landed
        __syncthreads();
      }
    }

    // ---- finish the run: normalise and store ----
    {
      const int th = thread(), row = tile0 + rblock * 32 + (th & 31), half = (th >> 5) & 1;
      const float l_tot = l_run + __shfl_xor(l_run, 32);
      const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
      if (active && gridDim.z > 1) {
        // one of several key shares: the unnormalised state goes to the merge pass
        const int64_t p = (static_cast<int64_t>(blockIdx.z) * a.Lq + row) * a.Hq + hq;
        float* po = a.ws_acc + p * D;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int i4 = 0; i4 < 4; ++i4)
            *reinterpret_cast<f32x4*>(po + db * 32 + i4 * 8 + half * 4) =
                f32x4{o_acc[db][i4 * 4], o_acc[db][i4 * 4 + 1], o_acc[db][i4 * 4 + 2], o_acc[db][i4 * 4 + 3]};
        if (half == 0) *reinterpret_cast<float2*>(a.ws_ml + p * 2) = float2{m_run, l_tot};
      } else if (active) {
        float* o = reinterpret_cast<float*>(a.out + row * a.os_row + hq * a.os_h);
        const float lse_nat = l_tot > 0.f ? (m_run + log2f(l_tot)) * kLn2 : -INFINITY;
        // attention-sink gate of the caller's post-attention step (model.py:122-128)
        const float gate = a.sinks != nullptr ? 1.f / (1.f + __expf(a.sinks[hq] - lse_nat)) : 1.f;
        const float f = inv * gate;
#pragma unroll
        for (int db = 0; db < DB; ++db) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            // register r holds d = db * 32 + (r / 4) * 8 + half * 4 + r % 4
            o[db * 32 + (r >> 2) * 8 + half * 4 + (r & 3)] = o_acc[db][r] * f;
          }
        }
        if (half == 0) a.lse[static_cast<int64_t>(hq) * a.Lq + row] = lse_nat;
      }
    }
    run0 = run1;
  }
}

// ---- merge of the key shares: one wavefront per (query row, query head) ----
constexpr int kMergeRows = 4;  // (row, head) pairs per workgroup

template <int D>
__global__ __launch_bounds__(kMergeRows * 64) void paged_prefill_f32_merge_kernel(const Args a, int n_shares) {
  constexpr int EPL = D / 64;  // output elements per lane
  const int lane = threadIdx.x & 63;
  const int64_t item = static_cast<int64_t>(blockIdx.x) * kMergeRows + (threadIdx.x >> 6);
  if (item >= static_cast<int64_t>(a.Lq) * a.Hq) return;
  const int row = static_cast<int>(item / a.Hq), hq = static_cast<int>(item % a.Hq);
  const int64_t share_stride = static_cast<int64_t>(a.Lq) * a.Hq;
  constexpr int kBatch = 8;  // the launcher never makes more shares
  float m_s[kBatch], l_s[kBatch], acc_s[kBatch][EPL];
#pragma unroll
  for (int s = 0; s < kBatch; ++s) {
    const bool on = s < n_shares;
    const int64_t p = s * share_stride + item;
    m_s[s] = on ? a.ws_ml[p * 2] : -INFINITY;
    l_s[s] = on ? a.ws_ml[p * 2 + 1] : 0.f;
#pragma unroll
    for (int e = 0; e < EPL; ++e) acc_s[s][e] = on ? a.ws_acc[p * D + lane * EPL + e] : 0.f;
  }
  float mn = -INFINITY;
#pragma unroll
  for (int s = 0; s < kBatch; ++s) mn = fmaxf(mn, m_s[s]);
  const float ms = mn == -INFINITY ? 0.f : mn;
  float den = 0.f, num[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) num[e] = 0.f;
#pragma unroll
  for (int s = 0; s < kBatch; ++s) {
    const float wgt = fast_exp2(m_s[s] - ms);  // 0 for a share that saw no key
    den += l_s[s] * wgt;
#pragma unroll
    for (int e = 0; e < EPL; ++e) num[e] += acc_s[s][e] * wgt;
  }
  const float lse_nat = den > 0.f ? (mn + log2f(den)) * kLn2 : -INFINITY;
  const float gate = a.sinks != nullptr ? 1.f / (1.f + __expf(a.sinks[hq] - lse_nat)) : 1.f;
  const float f = (den > 0.f ? 1.f / den : 0.f) * gate;
  float* o = reinterpret_cast<float*>(a.out + row * a.os_row + hq * a.os_h) + lane * EPL;
#pragma unroll
  for (int e = 0; e < EPL; ++e) o[e] = num[e] * f;
  if (lane == 0) a.lse[static_cast<int64_t>(hq) * a.Lq + row] = lse_nat;
}

template <int D, int G>
void launch_group(const Args& a0, void* workspace, int64_t workspace_bytes, hipStream_t st) {
  Args a = a0;
  constexpr int BM = (kWaves / G) * 32;
  a.n_tiles = (a.Lq + BM - 1) / BM;
  int shares = workspace ? fp::prefill_key_shares(static_cast<int64_t>(a.Hc) * a.n_tiles, FP_DTYPE_F32) : 1;
  while (shares > 1 && fp::prefill_share_bytes(shares, a.Lq, a.Hq, D, 4) > workspace_bytes) --shares;
  if (shares > 1) {
    a.ws_acc = static_cast<float*>(workspace);
    a.ws_ml = a.ws_acc + static_cast<int64_t>(shares) * a.Lq * a.Hq * D;
  }
  dim3 grid(a.Hc, a.n_tiles, shares);
  if (a.pd.shift >= 0)
    hipLaunchKernelGGL((paged_prefill_f32_kernel<D, G, true>), grid, dim3(kThreads), 0, st, a);
  else
    hipLaunchKernelGGL((paged_prefill_f32_kernel<D, G, false>), grid, dim3(kThreads), 0, st, a);
  if (shares > 1) {
    const int64_t items = static_cast<int64_t>(a.Lq) * a.Hq;
    hipLaunchKernelGGL((paged_prefill_f32_merge_kernel<D>), dim3(static_cast<unsigned>((items + kMergeRows - 1) / kMergeRows)),
                       dim3(kMergeRows * 64), 0, st, a, shares);
  }
}

template <int D>
int launch(const Args& a, void* ws, int64_t ws_bytes, hipStream_t st) {
  switch (a.Hq / a.Hc) {
    case 1: launch_group<D, 1>(a, ws, ws_bytes, st); return FP_OK;
    case 2: launch_group<D, 2>(a, ws, ws_bytes, st); return FP_OK;
    case 4: launch_group<D, 4>(a, ws, ws_bytes, st); return FP_OK;
    case 8: launch_group<D, 8>(a, ws, ws_bytes, st); return FP_OK;
    default: return fp::fail(FP_ERR_UNSUPPORTED, "fp_paged_prefill: Hq/Hc = %d (supported: 1, 2, 4, 8)", a.Hq / a.Hc);
  }
}

}  // namespace

namespace fp {

int prefill_mfma_f32(const void* q, int64_t q_stride_row, int64_t q_stride_h, const void* pool_k, const void* pool_v,
                     const int64_t* page_table, int64_t pt_row_stride, const int64_t* batch_idx,
                     const int32_t* row_limit, void* out, int64_t out_stride_row, int64_t out_stride_h, float* lse,
                     const float* sinks, int32_t Lq, int32_t Hq, int32_t Hc, int32_t D, int32_t page_size,
                     int32_t n_pages, int32_t max_batch, int64_t n_slots, float scale, void* workspace,
                     int64_t workspace_bytes, hipStream_t st) {
  if ((static_cast<int64_t>(Lq) + 31) / 32 > 65535) return fail(FP_ERR_UNSUPPORTED, "fp_paged_prefill: too many query rows");
  Args a{static_cast<const char*>(q), q_stride_row * 4, q_stride_h * 4,
         static_cast<const char*>(pool_k), static_cast<const char*>(pool_v),
         page_table, pt_row_stride, batch_idx, row_limit,
         static_cast<char*>(out), out_stride_row * 4, out_stride_h * 4, lse, sinks,
         Lq, Hq, Hc, PageDiv(page_size), n_pages, max_batch, n_slots, n_slots / page_size, scale * kLog2e, 0, nullptr, nullptr};
  return D == 64 ? launch<64>(a, workspace, workspace_bytes, st) : launch<128>(a, workspace, workspace_bytes, st);
}

}  // namespace fp
