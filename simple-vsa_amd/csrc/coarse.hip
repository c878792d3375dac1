// Coarse (pooled-token) attention on gfx950 MFMA, its backward, and the Top-K
// route: the T-dtype softmax attention of common.py:159-166 over the block
// means, the per-row top-k of triton_impl.py:1710, and the autograd of the
// coarse branch.  These replace the one-row-per-workgroup kernels of
// common.hip for bf16 / fp16 with head_dim 64 or 128 (the backward: 256 too, up
// to 768 blocks); other dtypes / widths keep the generic kernels.
//
// Layout of the tiles: a workgroup owns 32 rows (query blocks, or key blocks
// in the column pass) and its 8 waves stride over 32-wide tiles of the other
// side.  Products are taken transposed (S^T = K Q^T, dP^T = V G^T) so that a
// lane owns one row and holds 16 of its columns: row statistics are a lane
// reduction plus one xor-32 exchange.  Results that sum over the strided
// tiles are reduced across the waves in LDS in a fixed order, so every output
// is deterministic.
//
// These passes are a chain of memory and LDS round trips: a few tiles per
// wave, far from any rate limit.  So every load of a tile is issued before the
// first of its values is used, the score / probability tiles of up to 24 key
// tiles (768 blocks) stay in registers between the statistics and their use,
// and the waves' partial sums go to LDS side by side (rows padded by one float)
// and are added by all threads at once.  The version with 4 waves, two passes
// over the keys and one wave after another adding to one unpadded LDS tile (32
// lanes on one bank) took, at 12 heads, head dim 128: forward 14.3 us at 64
// blocks and 38 at 624, rows 12.8 and 34.6, columns 14.6 and 29.3; this one 9.0
// and 25, 7.1 and 19.6, 4.4 and 21.
//
// Rounding points follow the reference in T: scores T(T(q_c k_c) * scale),
// probabilities T(softmax), out_c T(P v_c); backward dP = T(G v_c^T),
// dS = T(T(P (dP - rowsum(P dP))) * scale), d_q_c = T(dS k_c),
// d_k_c = T(dS^T q_c), d_v_c = T(P^T G).
#include "coarse.h"

#include "vsa_device.h"
#include "vsa_launch.h"

namespace vsa {

namespace {

constexpr int kRows = 32;   // rows per workgroup
constexpr int kWaves = 8;
constexpr int kNT = 64 * kWaves;
constexpr int kParts = 4;   // partial sums side by side in LDS

// B-operand fragments of 32 rows of a [rows, D] matrix: lane (r, h) holds
// row base + r (clamped to the last row), dims 16 ks + 8h .. +7.
template <typename T, int D>
__device__ __forceinline__ void load_rows_b(const T* __restrict__ m, int base, int rows,
                                            typename Elem<T>::vec8 (&f)[D / 16]) {
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int row = min(base + r, rows - 1);
  const T* p = m + (int64_t)row * D + 8 * h;
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks)
    f[ks] = as_vec8<T>(*reinterpret_cast<const u32x4*>(p + 16 * ks));
}

// Copy of 32 rows x DH dims of a [rows, D] matrix (rows past the end repeat the
// last row) into this wave's swizzled LDS tile, for transpose reads: load()
// issues the loads, store() writes the tile.
template <typename T, int D, int DH>
struct RowStage {
  static constexpr int CH = 32 * DH / 8;  // 16-byte chunks
  static constexpr int N = CH / 64;       // per lane
  static_assert(CH % 64 == 0, "whole 16-byte chunks per lane");
  u32x4 v[N];
  __device__ __forceinline__ void load(const T* __restrict__ m, int base, int rows) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int c = lane + 64 * i;
      const int src = min(base + c / (DH / 8), rows - 1);
      v[i] = *reinterpret_cast<const u32x4*>(m + (int64_t)src * D + (c % (DH / 8)) * 8);
    }
  }
  __device__ __forceinline__ void store(T* tile) const {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int c = lane + 64 * i;
      *reinterpret_cast<u32x4*>(tile + swz<DH>(c / (DH / 8), c % (DH / 8))) = v[i];
    }
  }
};

// key (or row) index of accumulator element i in a lane with half h
__device__ __forceinline__ int acc_row(int i, int h) { return 8 * (i >> 2) + 4 * h + (i & 3); }

// LDS of a pass: the waves' operand tiles, then (the same memory) the partial
// sums of reduce_rows.
template <typename T, int DH>
union Shared {
  T tile[kWaves][32 * DH];
  float part[kParts][32 * (DH + 1)];
};

// Sum the waves' [32 x DH] transposed accumulators (lane (r, h) holds column r,
// rows mt*32 + acc_row) in a fixed order, round to T and store row `row` at
// dst + row * stride (rows < nrows).  Only waves < ntile hold a sum.  `part` may
// alias the operand tiles.
template <typename T, int DH>
__device__ __forceinline__ void reduce_rows(const f32x16 (&acc)[DH / 32],
                                            float (*part)[32 * (DH + 1)], int ntile,
                                            T* __restrict__ dst, int64_t stride, int nrows) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  static_assert(kWaves == 2 * kParts, "two waves per partial sum");
  float* p = part[wave % kParts] + r * (DH + 1);
  __syncthreads();
  if (ntile > kParts) {
    if (wave >= kParts) {
#pragma unroll
      for (int mt = 0; mt < DH / 32; ++mt)
#pragma unroll
        for (int i = 0; i < 16; ++i) p[mt * 32 + acc_row(i, h)] = acc[mt][i];
    }
    __syncthreads();
    if (wave < kParts) {  // each lane adds to what its own position holds
#pragma unroll
      for (int mt = 0; mt < DH / 32; ++mt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          float* e = p + mt * 32 + acc_row(i, h);
          *e = acc[mt][i] + *e;
        }
    }
  } else if (wave < ntile) {
#pragma unroll
    for (int mt = 0; mt < DH / 32; ++mt)
#pragma unroll
      for (int i = 0; i < 16; ++i) p[mt * 32 + acc_row(i, h)] = acc[mt][i];
  }
  __syncthreads();
  const int np = min(ntile, kParts);
  for (int x = 2 * threadIdx.x; x < 32 * DH; x += 2 * kNT) {
    const int row = x / DH, d = x % DH, at = row * (DH + 1) + d;
    float a = part[0][at], c = part[0][at + 1];
    for (int w = 1; w < np; ++w) {
      a += part[w][at];
      c += part[w][at + 1];
    }
    typedef T pair __attribute__((ext_vector_type(2)));
    if (row < nrows)
      *reinterpret_cast<pair*>(dst + row * stride + d) = pair{Elem<T>::from_f(a), Elem<T>::from_f(c)};
  }
}

// Four consecutive entries key0 .. key0+3 of a [.., kb] fp32 row; entries past
// the row read as zero and are not written.
__device__ __forceinline__ void load4(const float* __restrict__ row, int key0, int kb, bool vec4,
                                      float* v) {
  if (vec4 && key0 + 3 < kb) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(row + key0);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = x[e];
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = key0 + e < kb ? row[key0 + e] : 0.f;
  }
}
__device__ __forceinline__ void store_tile(float* __restrict__ row, int kt, int kb, bool vec4,
                                           int h, const float (&v)[16]) {
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int key0 = kt * 32 + 8 * g + 4 * h;
    if (vec4 && key0 + 3 < kb) {
      *reinterpret_cast<f32x4*>(row + key0) = f32x4{v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]};
    } else {
      for (int e = 0; e < 4; ++e)
        if (key0 + e < kb) row[key0 + e] = v[4 * g + e];
    }
  }
}

// Max / sum of one value per row over the waves (lane (r, h): the wave's value
// of row r, the same in both halves), in wave order.
template <bool MAX>
__device__ __forceinline__ float across_waves(float x, float (*stat)[32]) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 31;
  if (lane < 32) stat[wave][r] = x;
  __syncthreads();
  float y = stat[0][r];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) y = MAX ? fmaxf(y, stat[w][r]) : y + stat[w][r];
  return y;
}

}  // namespace

// ---------------------------------------------------------------------------
// Forward: scores, probabilities, out_c.  grid (ceil(Qb/32), BH).  NCT key
// tiles per wave are kept in registers (8 NCT tiles cover the row); NCT = 0
// recomputes the scores for each use instead.
// ---------------------------------------------------------------------------
template <typename T, int D, int NCT>
__global__ __launch_bounds__(kNT) void coarse_fwd_mfma_kernel(
    const T* __restrict__ qc, const T* __restrict__ kc, const T* __restrict__ vc,
    float* __restrict__ scores, float* __restrict__ probs, T* __restrict__ outc, int qb, int kb,
    float scale) {
  using E = Elem<T>;
  typedef typename E::vec8 V8;
  __shared__ __attribute__((aligned(16))) Shared<T, D> sh;
  __shared__ float smax[kWaves][32], ssum[kWaves][32];
  const int64_t b = blockIdx.y;
  const int q0 = blockIdx.x * kRows;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int myq = q0 + r;
  const bool qvalid = myq < qb;
  const T* kb_ = kc + b * kb * (int64_t)D;
  const T* vb_ = vc + b * kb * (int64_t)D;
  float* srow = scores + (b * qb + myq) * (int64_t)kb;
  float* prow = probs + (b * qb + myq) * (int64_t)kb;
  const int ntile = (kb + 31) / 32;
  const bool vec4 = (kb & 3) == 0;  // rows of the [.., Kb] fp32 buffers are 16-byte aligned

  V8 qf[D / 16];
  load_rows_b<T, D>(qc + b * qb * (int64_t)D, q0, qb, qf);

  // S^T tile (keys x queries) of key tile kt, rounded as the reference does
  auto scores_of = [&](const V8 (&kf)[D / 16], int kt, float (&s)[16]) {
    f32x16 acc = f32x16{};
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) acc = E::mfma32(kf[ks], qf[ks], acc);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int key = kt * 32 + acc_row(i, h);
      s[i] = key < kb ? round_t<T>(round_t<T>(acc[i]) * scale) : -INFINITY;
    }
  };
  f32x16 oacc[D / 32];
#pragma unroll
  for (int mt = 0; mt < D / 32; ++mt) oacc[mt] = f32x16{};
  T* vt = sh.tile[wave];
  auto add_pv = [&](const float (&p)[16]) {  // out_c^T += V^T P^T, V in vt
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const V8 bp = pack8<T>(p + 8 * kk);
#pragma unroll
      for (int mt = 0; mt < D / 32; ++mt)
        oacc[mt] = E::mfma32(tr_a8<T, D>(vt, mt * 32, 16 * kk, 16 * kk + 8), bp, oacc[mt]);
    }
  };
  RowStage<T, D, D> vst;

  if constexpr (NCT > 0) {
    V8 kf[NCT][D / 16];
#pragma unroll
    for (int c = 0; c < NCT; ++c) load_rows_b<T, D>(kb_, (wave + c * kWaves) * 32, kb, kf[c]);
    vst.load(vb_, wave * 32, kb);
    float s[NCT][16];
    float m = -INFINITY;
#pragma unroll
    for (int c = 0; c < NCT; ++c) {
      scores_of(kf[c], wave + c * kWaves, s[c]);  // a tile past the row: all -inf
#pragma unroll
      for (int i = 0; i < 16; ++i) m = fmaxf(m, s[c][i]);
    }
    m = fmaxf(m, __shfl_xor(m, 32, 64));
    const float M = across_waves<true>(m, smax);
    float p[NCT][16];
    float l = 0.f;
#pragma unroll
    for (int c = 0; c < NCT; ++c)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        p[c][i] = expf(s[c][i] - M);
        l += p[c][i];
      }
    l += __shfl_xor(l, 32, 64);
    const float L = across_waves<false>(l, ssum);
#pragma unroll
    for (int c = 0; c < NCT; ++c) {
      const int kt = wave + c * kWaves;
      if (kt >= ntile) break;  // the last tiles of the row: uniform
#pragma unroll
      for (int i = 0; i < 16; ++i) p[c][i] = round_t<T>(p[c][i] / L);  // 0 for padding keys
      vst.store(vt);
      if (c + 1 < NCT) vst.load(vb_, (kt + kWaves) * 32, kb);
      add_pv(p[c]);
      if (qvalid) {
        store_tile(srow, kt, kb, vec4, h, s[c]);
        store_tile(prow, kt, kb, vec4, h, p[c]);
      }
    }
  } else {
    // scores out, running max / sum per query (lane-partial sums)
    V8 kf[D / 16];
    float m = -INFINITY, l = 0.f;
    load_rows_b<T, D>(kb_, wave * 32, kb, kf);
    for (int kt = wave; kt < ntile; kt += kWaves) {
      float s[16];
      scores_of(kf, kt, s);
      load_rows_b<T, D>(kb_, (kt + kWaves) * 32, kb, kf);
      float tmax = -INFINITY;
#pragma unroll
      for (int i = 0; i < 16; ++i) tmax = fmaxf(tmax, s[i]);
      tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
      const float mn = fmaxf(m, tmax);
      float part = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) part += expf(s[i] - mn);
      l = l * expf(m - mn) + part;
      m = mn;
      if (qvalid) store_tile(srow, kt, kb, vec4, h, s);
    }
    load_rows_b<T, D>(kb_, wave * 32, kb, kf);
    vst.load(vb_, wave * 32, kb);
    l += __shfl_xor(l, 32, 64);
    const float M = across_waves<true>(m, smax);
    const float L = across_waves<false>(m == -INFINITY ? 0.f : l * expf(m - M), ssum);
    // probabilities out, out_c^T += V^T P^T
    for (int kt = wave; kt < ntile; kt += kWaves) {
      float p[16];
      scores_of(kf, kt, p);
      load_rows_b<T, D>(kb_, (kt + kWaves) * 32, kb, kf);
#pragma unroll
      for (int i = 0; i < 16; ++i) p[i] = round_t<T>(expf(p[i] - M) / L);
      vst.store(vt);
      vst.load(vb_, (kt + kWaves) * 32, kb);
      add_pv(p);
      if (qvalid) store_tile(prow, kt, kb, vec4, h, p);
    }
  }
  reduce_rows<T, D>(oacc, sh.part, ntile, outc + (b * qb + q0) * (int64_t)D, D, qb - q0);
}

// ---------------------------------------------------------------------------
// Top-K route, a wave per row with the row's keys in registers (R per lane, up
// to 64 R blocks): the k-th largest total-order score key is found bit by bit
// from the top (a ballot per register and bit; the search ends as soon as
// exactly topk keys are above the candidate), then the keys above it and, by
// ascending id, those equal to it are written in id order: the rule "larger
// score, then smaller id" of topk_radix_kernel, which needs a workgroup and
// about eighty barriers per row.  Bound by the ballots' issue.  40 x 160 rows of
// 160 blocks, topk 20: 26.3 -> 6.7 us; 12 x 624 rows of 624, topk 78: 45.6 -> 20.8.
// ---------------------------------------------------------------------------
template <int R>
__global__ __launch_bounds__(256) void topk_wave_kernel(const float* __restrict__ scores,
                                                        int32_t* __restrict__ selected,
                                                        int64_t rows, int kb, int topk) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const float* src = scores + row * kb;
  uint32_t u[R];  // order key as unsigned; 0 past the row (no score has it: -inf is 0x007fffff)
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int j = 64 * i + lane;
    u[i] = j < kb ? (uint32_t)order_key(src[j]) ^ 0x80000000u : 0u;
  }
  uint32_t t = 0;    // largest t found so far with at least topk keys >= t
  int above = kb;    // keys >= t
  auto search = [&](int hi, int lo) {
    for (int bit = hi; bit >= lo && above != topk; --bit) {
      const uint32_t cand = t | (1u << bit);
      int n = 0;
#pragma unroll
      for (int i = 0; i < R; ++i) n += (int)__popcll(__ballot(u[i] >= cand));
      if (n >= topk) {
        t = cand;
        above = n;
      }
    }
  };
  search(31, 16);
  if (above != topk) {
    // several keys share the upper half of the k-th: where they agree in the
    // lower half too (scores rounded to bf16 always do), that half needs no search
    uint32_t low_or = 0, low_and = 0xffffu;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const bool same = (u[i] >> 16) == (t >> 16);
      low_or |= same ? u[i] & 0xffffu : 0u;
      low_and &= same ? u[i] : 0xffffu;
    }
    if (__all(low_or == 0u)) {
    } else if (__all(low_and == 0xffffu)) {
      t |= 0xffffu;
    } else {
      search(15, 0);
    }
  }
  // `drop` of the keys equal to t are not taken: those with the largest ids
  int eq = 0;
  if (above != topk) {
#pragma unroll
    for (int i = 0; i < R; ++i) eq += (int)__popcll(__ballot(u[i] == t));
  }
  int take_eq = eq - (above - topk);  // unused while above == topk
  const uint64_t below = (1ull << lane) - 1ull;
  int32_t* dst = selected + row * topk;
  int at = 0;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    bool sel = u[i] >= t && u[i] != 0u;
    if (above != topk) {
      const uint64_t e = __ballot(u[i] == t);
      if (u[i] == t) sel = (int)__popcll(e & below) < take_eq;
      take_eq -= (int)__popcll(e);
    }
    const uint64_t m = __ballot(sel);
    if (sel) dst[at + __popcll(m & below)] = 64 * i + lane;
    at += __popcll(m);
  }
}

// ---------------------------------------------------------------------------
// Top-K of rows longer than topk_wave_kernel takes, by radix select on the
// total-order score key (one workgroup per row, the keys in LDS):
// the k-th largest key T is found digit by digit (4 x 8 bits); every key above
// T is taken, and keys equal to T are taken by ascending id until topk ids are
// chosen -- the rule "larger score, then smaller id".  Ids are written in
// ascending order.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void topk_radix_kernel(const float* __restrict__ scores,
                                                         int32_t* __restrict__ selected, int kb,
                                                         int topk) {
  extern __shared__ uint32_t keys[];  // kb
  __shared__ int hist[256];
  __shared__ int wsum[4][2];
  __shared__ int digit_sel[2];
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  for (int j = tid; j < kb; j += 256)
    keys[j] = (uint32_t)order_key(scores[row * kb + j]) ^ 0x80000000u;  // unsigned order
  __syncthreads();
  uint32_t prefix = 0, mask = 0;
  int remaining = topk;  // how many of the keys matching `prefix` are still to be taken
  for (int shift = 24; shift >= 0; shift -= 8) {
    hist[tid] = 0;
    __syncthreads();
    for (int j = tid; j < kb; j += 256) {
      const uint32_t u = keys[j];
      if ((u & mask) == prefix) atomicAdd(&hist[(u >> shift) & 255], 1);
    }
    __syncthreads();
    // suffix sums: hist[d] <- number of matching keys with digit >= d
    for (int o = 1; o < 256; o <<= 1) {
      const int add = tid + o < 256 ? hist[tid + o] : 0;
      __syncthreads();
      hist[tid] += add;
      __syncthreads();
    }
    const int above = tid < 255 ? hist[tid + 1] : 0;  // digit > tid
    if (hist[tid] >= remaining && above < remaining) {
      digit_sel[0] = tid;
      digit_sel[1] = above;
    }
    __syncthreads();
    const int d = digit_sel[0];
    remaining -= digit_sel[1];
    prefix |= (uint32_t)d << shift;
    mask |= 255u << shift;
    __syncthreads();
  }
  // prefix = T (k-th largest); `remaining` keys equal to T are taken, by id
  const uint32_t kth = prefix;
  int taken = 0, eq_seen = 0;
  int32_t* dst = selected + row * topk;
  for (int j0 = 0; j0 < kb; j0 += 256) {
    const int j = j0 + tid;
    const uint32_t u = j < kb ? keys[j] : 0u;
    const bool eq = j < kb && u == kth;
    const uint64_t beq = __ballot(eq);
    const int eq_before = __popcll(beq & ((1ull << lane) - 1ull));
    if (lane == 0) wsum[wave][0] = __popcll(beq);
    __syncthreads();
    int eq_off = eq_seen;
    for (int w = 0; w < wave; ++w) eq_off += wsum[w][0];
    const bool sel = j < kb && (u > kth || (eq && eq_off + eq_before < remaining));
    const uint64_t bsel = __ballot(sel);
    const int sel_before = __popcll(bsel & ((1ull << lane) - 1ull));
    if (lane == 0) wsum[wave][1] = __popcll(bsel);
    __syncthreads();
    int sel_off = taken;
    for (int w = 0; w < wave; ++w) sel_off += wsum[w][1];
    if (sel && sel_off + sel_before < topk) dst[sel_off + sel_before] = j;
    for (int w = 0; w < 4; ++w) {
      eq_seen += wsum[w][0];
      taken += wsum[w][1];
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Backward, rows: dP, softmax backward, dS out, d_q_c.  grid (ceil(Qb/32), BH,
// D/DH): a workgroup sums DH dims of d_q_c (dP needs all D; at head dim 256
// both halves form it).  NCT as in the forward.
// ---------------------------------------------------------------------------
template <typename T, int D, int NCT>
__global__ __launch_bounds__(kNT) void coarse_bwd_rows_mfma_kernel(
    const T* __restrict__ kc, const T* __restrict__ vc, const float* __restrict__ probs,
    const T* __restrict__ d_outc, float* __restrict__ ds, T* __restrict__ d_qc, int qb, int kb,
    float scale) {
  using E = Elem<T>;
  typedef typename E::vec8 V8;
  constexpr int DH = D < 128 ? D : 128;
  __shared__ __attribute__((aligned(16))) Shared<T, DH> sh;
  __shared__ float ssum[kWaves][32];
  const int64_t b = blockIdx.y;
  const int q0 = blockIdx.x * kRows, d_off = blockIdx.z * DH;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int myq = q0 + r;
  const int qrow = min(myq, qb - 1);
  const T* kb_ = kc + b * kb * (int64_t)D + d_off;
  const T* vb_ = vc + b * kb * (int64_t)D;
  const float* prow = probs + (b * qb + qrow) * (int64_t)kb;
  float* dsrow = ds + (b * qb + myq) * (int64_t)kb;
  const bool store_ds = myq < qb && blockIdx.z == 0;
  const int ntile = (kb + 31) / 32;
  const bool vec4 = (kb & 3) == 0;  // rows of the [.., Kb] fp32 buffers are 16-byte aligned

  V8 gf[D / 16];
  load_rows_b<T, D>(d_outc + b * qb * (int64_t)D, q0, qb, gf);

  // dP^T tile (keys x queries), rounded to T
  auto dp_of = [&](const V8 (&vf)[D / 16], float (&dp)[16]) {
    f32x16 acc = f32x16{};
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) acc = E::mfma32(vf[ks], gf[ks], acc);
#pragma unroll
    for (int i = 0; i < 16; ++i) dp[i] = round_t<T>(acc[i]);
  };
  auto load_p = [&](int kt, float (&p)[16]) {
#pragma unroll
    for (int g = 0; g < 4; ++g) load4(prow, kt * 32 + 8 * g + 4 * h, kb, vec4, p + 4 * g);
  };
  f32x16 qacc[DH / 32];
#pragma unroll
  for (int mt = 0; mt < DH / 32; ++mt) qacc[mt] = f32x16{};
  T* kt_ = sh.tile[wave];
  RowStage<T, D, DH> kst;
  auto finish_tile = [&](int kt, float (&dp)[16], const float (&p)[16], float rsum, bool more) {
#pragma unroll
    for (int i = 0; i < 16; ++i) dp[i] = round_t<T>(round_t<T>(p[i] * (dp[i] - rsum)) * scale);
    kst.store(kt_);
    if (more) kst.load(kb_, (kt + kWaves) * 32, kb);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const V8 bs = pack8<T>(dp + 8 * kk);
#pragma unroll
      for (int mt = 0; mt < DH / 32; ++mt)
        qacc[mt] = E::mfma32(tr_a8<T, DH>(kt_, mt * 32, 16 * kk, 16 * kk + 8), bs, qacc[mt]);
    }
    if (store_ds) store_tile(dsrow, kt, kb, vec4, h, dp);
  };

  if constexpr (NCT > 0) {
    float dp[NCT][16], p[NCT][16];
    float part = 0.f;
    V8 vf[D / 16];
    load_rows_b<T, D>(vb_, wave * 32, kb, vf);
#pragma unroll
    for (int c = 0; c < NCT; ++c) load_p(wave + c * kWaves, p[c]);  // zero past the row
#pragma unroll
    for (int c = 0; c < NCT; ++c) {
      dp_of(vf, dp[c]);
      if (c + 1 < NCT) load_rows_b<T, D>(vb_, (wave + (c + 1) * kWaves) * 32, kb, vf);
      if (c + 1 == NCT) kst.load(kb_, wave * 32, kb);
#pragma unroll
      for (int i = 0; i < 16; ++i) part = fmaf(p[c][i], dp[c][i], part);
    }
    part += __shfl_xor(part, 32, 64);
    const float rsum = across_waves<false>(part, ssum);
#pragma unroll
    for (int c = 0; c < NCT; ++c) {
      const int kt = wave + c * kWaves;
      if (kt >= ntile) break;
      finish_tile(kt, dp[c], p[c], rsum, c + 1 < NCT);
    }
  } else {
    V8 vf[D / 16];
    float p[16], dp[16];
    float part = 0.f;
    load_rows_b<T, D>(vb_, wave * 32, kb, vf);
    for (int kt = wave; kt < ntile; kt += kWaves) {
      load_p(kt, p);
      dp_of(vf, dp);
      load_rows_b<T, D>(vb_, (kt + kWaves) * 32, kb, vf);
#pragma unroll
      for (int i = 0; i < 16; ++i) part = fmaf(p[i], dp[i], part);
    }
    load_rows_b<T, D>(vb_, wave * 32, kb, vf);
    kst.load(kb_, wave * 32, kb);
    part += __shfl_xor(part, 32, 64);
    const float rsum = across_waves<false>(part, ssum);
    for (int kt = wave; kt < ntile; kt += kWaves) {
      load_p(kt, p);
      dp_of(vf, dp);
      load_rows_b<T, D>(vb_, (kt + kWaves) * 32, kb, vf);
      finish_tile(kt, dp, p, rsum, true);
    }
  }
  reduce_rows<T, DH>(qacc, sh.part, ntile, d_qc + (b * qb + q0) * (int64_t)D + d_off, D, qb - q0);
}

// ---------------------------------------------------------------------------
// Backward, columns: d_k_c = T(dS^T q_c), d_v_c = T(P^T d_out_c).
// grid (ceil(Kb/32), BH, 2 D/DH): a workgroup sums DH dims of one of the two
// (both at once needed more registers than a wave has); waves stride over
// 32-query tiles.
// ---------------------------------------------------------------------------
template <typename T, int D>
__global__ __launch_bounds__(kNT) void coarse_bwd_cols_mfma_kernel(
    const T* __restrict__ qc, const float* __restrict__ probs, const T* __restrict__ d_outc,
    const float* __restrict__ ds, T* __restrict__ d_kc, T* __restrict__ d_vc, int qb, int kb) {
  using E = Elem<T>;
  typedef typename E::vec8 V8;
  constexpr int DH = D < 128 ? D : 128;
  __shared__ __attribute__((aligned(16))) Shared<T, DH> sh;
  const int64_t b = blockIdx.y;
  const bool is_v = blockIdx.z & 1;
  const int k0 = blockIdx.x * kRows, d_off = (blockIdx.z >> 1) * DH;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int mykey = min(k0 + r, kb - 1);
  const T* rows = (is_v ? d_outc : qc) + b * qb * (int64_t)D + d_off;
  const float* weights = (is_v ? probs : ds) + b * qb * (int64_t)kb;
  T* dst = is_v ? d_vc : d_kc;
  const int ntile = (qb + 31) / 32;

  f32x16 acc[DH / 32];
#pragma unroll
  for (int mt = 0; mt < DH / 32; ++mt) acc[mt] = f32x16{};
  T* tile = sh.tile[wave];
  for (int t = wave; t < ntile; t += kWaves) {
    // B operand: the weights [q][key r] of the 16 queries this lane feeds (rows
    // past the end are clamped, loaded and zeroed: a load under the condition
    // would be a branch and a wait per value).  The tile's first row is a 64-bit
    // offset (any number of query blocks is taken), the 32 rows in it 32-bit ones.
    float w[16];
    RowStage<T, D, DH> st;
    const float* wt = weights + (int64_t)t * 32 * kb + mykey;
    const int last = qb - 1 - t * 32;
#pragma unroll
    for (int i = 0; i < 16; ++i) w[i] = wt[min(acc_row(i, h), last) * kb];
    st.load(rows, t * 32, qb);
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (t * 32 + acc_row(i, h) >= qb) w[i] = 0.f;
    st.store(tile);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const V8 bw = pack8<T>(w + 8 * kk);
#pragma unroll
      for (int mt = 0; mt < DH / 32; ++mt)
        acc[mt] = E::mfma32(tr_a8<T, DH>(tile, mt * 32, 16 * kk, 16 * kk + 8), bw, acc[mt]);
    }
  }
  reduce_rows<T, DH>(acc, sh.part, ntile, dst + (b * kb + k0) * (int64_t)D + d_off, D, kb - k0);
}

// ---------------------------------------------------------------------------
// Host launchers (called by the C ABI in common.hip)
// ---------------------------------------------------------------------------
bool coarse_fwd_mfma_supported(int D, int dtype) {
  return (dtype == VSA_BF16 || dtype == VSA_F16) && (D == 64 || D == 128);
}

// key tiles per wave kept in registers, or 0 (recomputed) for longer rows
static int cached_tiles(int kb) {
  const int n = ((kb + 31) / 32 + kWaves - 1) / kWaves;
  return n <= 3 ? n : 0;
}

// The backward also takes head dim 256 up to 768 blocks (the loop for longer
// rows spills there).  Its products only round differently; the forward's
// scores decide the route, whose near-ties the order of a dot product can
// break, so head dim 256 keeps the generic forward's order.
bool coarse_bwd_mfma_supported(int D, int kb, int dtype) {
  return coarse_fwd_mfma_supported(D, dtype) ||
         ((dtype == VSA_BF16 || dtype == VSA_F16) && D == 256 && cached_tiles(kb) > 0);
}

int coarse_fwd_mfma(const void* qc, const void* kc, const void* vc, float* scores, float* probs,
                    void* outc, int64_t bh, int qb, int kb, int D, float scale, int dtype,
                    hipStream_t s) {
  if (bh > 65535) return VSA_ERR_SHAPE;
  const dim3 grid((qb + kRows - 1) / kRows, (unsigned)bh);
  const int nct = cached_tiles(kb);
#define VSA_CF(DD, CC)                                                                         \
  if (D == DD && nct == CC) {                                                                  \
    hipLaunchKernelGGL((coarse_fwd_mfma_kernel<T, DD, CC>), grid, dim3(kNT), 0, s,             \
                       (const T*)qc, (const T*)kc, (const T*)vc, scores, probs, (T*)outc, qb,  \
                       kb, scale);                                                             \
    return vsa_check_launch();                                                                 \
  }
#define VSA_CFD(DD) VSA_CF(DD, 0) VSA_CF(DD, 1) VSA_CF(DD, 2) VSA_CF(DD, 3)
  VSA_DISPATCH_MFMA(dtype, T, { VSA_CFD(64) VSA_CFD(128) });
#undef VSA_CFD
#undef VSA_CF
  return VSA_ERR_UNSUPPORTED;
}

int topk_route(const float* scores, int32_t* selected, int64_t rows, int kb, int topk,
               hipStream_t s) {
  if (rows > 0x7fffffffLL) return VSA_ERR_SHAPE;
  const dim3 grid((unsigned)((rows + 3) / 4));
#define VSA_TK(R)                                                                              \
  if (kb <= 64 * R) {                                                                          \
    hipLaunchKernelGGL((topk_wave_kernel<R>), grid, dim3(256), 0, s, scores, selected, rows,   \
                       kb, topk);                                                              \
    return vsa_check_launch();                                                                 \
  }
  VSA_TK(1) VSA_TK(2) VSA_TK(4) VSA_TK(8) VSA_TK(16) VSA_TK(32)
#undef VSA_TK
  hipLaunchKernelGGL(topk_radix_kernel, dim3((unsigned)rows), dim3(256),
                     (size_t)kb * sizeof(uint32_t), s, scores, selected, kb, topk);
  return vsa_check_launch();
}

int coarse_bwd_mfma(const void* qc, const void* kc, const void* vc, const float* probs,
                    const void* d_outc, float* ds, void* d_qc, void* d_kc, void* d_vc,
                    int64_t bh, int qb, int kb, int D, float scale, int dtype, hipStream_t s) {
  if (bh > 65535) return VSA_ERR_SHAPE;
  const unsigned halves = D > 128 ? D / 128 : 1;
  const dim3 grows((qb + kRows - 1) / kRows, (unsigned)bh, halves);
  const dim3 gcols((kb + kRows - 1) / kRows, (unsigned)bh, 2 * halves);
  const int nct = cached_tiles(kb);
#define VSA_CB(DD, CC)                                                                           \
  if (D == DD && nct == CC) {                                                                    \
    hipLaunchKernelGGL((coarse_bwd_rows_mfma_kernel<T, DD, CC>), grows, dim3(kNT), 0, s,         \
                       (const T*)kc, (const T*)vc, probs, (const T*)d_outc, ds, (T*)d_qc, qb,    \
                       kb, scale);                                                               \
    int rc = vsa_check_launch();                                                                 \
    if (rc) return rc;                                                                           \
    hipLaunchKernelGGL((coarse_bwd_cols_mfma_kernel<T, DD>), gcols, dim3(kNT), 0, s,             \
                       (const T*)qc, probs, (const T*)d_outc, ds, (T*)d_kc, (T*)d_vc, qb, kb);   \
    return vsa_check_launch();                                                                   \
  }
#define VSA_CBD(DD) VSA_CB(DD, 1) VSA_CB(DD, 2) VSA_CB(DD, 3)
  VSA_DISPATCH_MFMA(dtype, T, {
    VSA_CB(64, 0) VSA_CBD(64) VSA_CB(128, 0) VSA_CBD(128) VSA_CBD(256)
  });
#undef VSA_CBD
#undef VSA_CB
  return VSA_ERR_UNSUPPORTED;
}

}  // namespace vsa
