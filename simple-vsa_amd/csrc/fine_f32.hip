// Sparse fine forward, dQ and dK/dV for fp32 inputs (the reference's GPU path
// accepts fp32: triton_impl.py:375-376).  Inputs, sums and results are fp32:
// outputs, LSE (base 2), the fused combine, the pooled-gradient folds and the
// padding masks follow the bf16 / fp16 kernels of fine_fwd.hip and
// fine_bwd.hip with T = fp32.
//
// Head dims 64 / 128 run their products on the bf16 matrix core (the splitting of
// Henry, Tang and Heinecke, 2019, with three parts): every fp32 operand is the
// exact sum of three bf16 values, hi and mid rounded to the nearest, and a product
// is its six largest partial products, accumulated in fp32.  What is left out
// (mid.lo, lo.mid, lo.lo) has either sign and is at most 2^-24 of a product, half
// an fp32 rounding.  With parts that were truncated it had the product's sign and
// reached 2^-21 (dP of near-constant rows off by 4e-7 in common, now 7e-8 rms, 8e-7
// on the fp32 matrix core), for 1 % less time.  A 32x32 tile over 16 dims takes
// 6 x 32 cycles against 8 x 64 on v_mfma_f32_32x32x2_f32, and its sum is rounded 6
// times instead of 16.  At 12 heads, 16 384 tokens, head dim 128, block 256, topk 8
// the forward takes 1.39 ms against 2.89 on the fp32 units, dQ 1.73 against 2.85,
// dK/dV 2.56 against 4.31, and the error against fp64 is 1.0e-6 against 1.1e-6.
// Bound by one wave per SIMD at head dim 128 (registers): the matrix core is busy
// 40 / 48 / 48 % of the time and the vector unit, which splits operands, 36 / 33 /
// 26 %, mostly one after the other.
//
// The parts hold an operand's 24 bits from 2^-110 (7.7e-34) up.  Below, up to
// 2^-133 of each operand is lost (3e-6 rms at 1e-35), bf16's last place; that
// counts for the backward's dS = P (dP - delta) too, so from |dO| of about 1e-32
// down, depending on P.
//
// The forward and dQ at head_dim 256 (split fragments would exceed a wave's
// registers) run on v_mfma_f32_32x32x2_f32 (the fp32 matrix core: 1/16 of the
// bf16 rate, twice the unpacked fp32 VALU rate).  Its operands are one float per lane:
//   A (32 x 2): lane (r, h) = row r, k = h;  B (2 x 32): lane (c, h) = column c, k = h;
//   C (32 x 32): element i of lane (c, h) = row 8(i/4) + 4h + i%4, column c.
// A dot product over D dims is D/2 MFMAs; k-step t pairs dim t (h = 0) with
// dim D/2 + t (h = 1), so each lane reads its row contiguously.  The C tile of
// one product is the B operand of the next with no data movement (element t of
// the accumulator is the k = h value of k-step t, rows 8(t/4) + 4h + t%4), and
// the other operand is read in that row order.  dK/dV at head_dim 256 keeps a
// vector-ALU kernel.
#include "fine_f32.h"
#include "vsa_device.h"
#include "vsa_launch.h"

namespace vsa {

namespace {

constexpr int kRows = 64;   // rows per workgroup
constexpr int kChunk = 32;  // streamed rows per LDS chunk

__device__ __forceinline__ f32x16 mfma_f32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float quad_sum(float x) {
  x += __shfl_xor(x, 1, 64);
  x += __shfl_xor(x, 2, 64);
  return x;
}

// Copy 32 rows of D floats (global row stride D) into LDS with row stride LD;
// rows past `valid` are zero (never used for a valid result, only kept finite).
template <int D, int LD, int NT>
__device__ __forceinline__ void stage32(float* dst, const float* __restrict__ src, int valid) {
  constexpr int V4 = D / 4;  // float4 per row
#pragma unroll 4
  for (int x = threadIdx.x; x < kChunk * V4; x += NT) {
    const int r = x / V4, c = x % V4;
    f32x4 val = {0.f, 0.f, 0.f, 0.f};
    if (r < valid) val = *reinterpret_cast<const f32x4*>(src + (int64_t)r * D + 4 * c);
    *reinterpret_cast<f32x4*>(dst + r * LD + 4 * c) = val;
  }
}

// Copy `rows` rows of D floats (row stride D) into LDS (row stride D) with 256
// threads; rows past `valid` are zero.
template <int D>
__device__ __forceinline__ void stage_rows_f32(float* dst, const float* __restrict__ src,
                                               int rows, int valid) {
  constexpr int V4 = D / 4;  // float4 per row
  for (int x = threadIdx.x; x < rows * V4; x += 256) {
    const int r = x / V4, c = x % V4;
    f32x4 val = {0.f, 0.f, 0.f, 0.f};
    if (r < valid) val = *reinterpret_cast<const f32x4*>(src + (int64_t)r * D + 4 * c);
    *reinterpret_cast<f32x4*>(dst + r * D + 4 * c) = val;
  }
}

// this lane's row fragment: x[row][h * D/2 + t], t < D/2
template <int D>
__device__ __forceinline__ void load_frag(float (&f)[D / 2], const float* __restrict__ row, int h) {
#pragma unroll
  for (int t = 0; t < D / 2; t += 4) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(row + h * (D / 2) + t);
    f[t] = x[0]; f[t + 1] = x[1]; f[t + 2] = x[2]; f[t + 3] = x[3];
  }
}

// acc += rows(lds, 32 x D, stride LD) . frag^T: A = LDS row r (lane r), B = frag
template <int D, int LD>
__device__ __forceinline__ void mma_rows(f32x16& acc, const float* lds, const float (&f)[D / 2],
                                         int r, int h) {
  const float* row = lds + r * LD + h * (D / 2);
#pragma unroll
  for (int t = 0; t < D / 2; t += 4) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(row + t);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = mfma_f32(a[e], f[t + e], acc);
  }
}

// acc[mt] += (LDS rows)^T . B, B = the C tile `bop` (rows 8(t/4) + 4h + t%4 of
// the LDS tile paired with k-step t): A = LDS[row(t, h)][32 mt + r]
template <int D, int LD>
__device__ __forceinline__ void mma_cols(f32x16 (&acc)[D / 32], const float* lds, const f32x16& bop,
                                         int r, int h) {
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    const float* row = lds + (8 * (t >> 2) + 4 * h + (t & 3)) * LD + r;
#pragma unroll
    for (int mt = 0; mt < D / 32; ++mt) acc[mt] = mfma_f32(row[32 * mt], bop[t], acc[mt]);
  }
}

}  // namespace

// ---------------------------------------------------------------------------
// Split-bf16 products
// ---------------------------------------------------------------------------
namespace {

typedef __bf16 bf16_t;

// Eight fp32 values as three bf16 MFMA operands.
struct Split8 {
  bf16x8 hi, mid, lo;
};

// The upper halves of two floats, packed.
__device__ __forceinline__ uint32_t pack_hi16(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
// Two floats rounded to bf16 (v_cvt_pk_bf16_f32), packed, and the packed two as
// floats.
__device__ __forceinline__ uint32_t round_pair(float a, float b) {
  typedef bf16_t pair __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, pair{(bf16_t)a, (bf16_t)b});
}
__device__ __forceinline__ float low_part(uint32_t p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float high_part(uint32_t p) { return __uint_as_float(p & 0xffff0000u); }

// Magnitudes from here on round to a bf16 infinity.
constexpr float kSplitMax = 0x1.ffp127f;

// x = hi + mid + lo of |x| < kSplitMax: hi and mid are rounded to the nearest,
// so that what is left is signed and at most half of the last place (|mid| <=
// 2^-8 |x|, |lo| <= 2^-17 |x|, with x's leading bit); lo has 8 significant bits
// and is exact.
__device__ __forceinline__ Split8 split8(const float (&x)[8]) {
  u32x4 hi, mid, lo;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float a = x[2 * e], b = x[2 * e + 1];
    hi[e] = round_pair(a, b);
    const float a1 = a - low_part(hi[e]), b1 = b - high_part(hi[e]);
    mid[e] = round_pair(a1, b1);
    const float a2 = a1 - low_part(mid[e]), b2 = b1 - high_part(mid[e]);
    lo[e] = pack_hi16(a2, b2);
  }
  return {as_vec8<bf16_t>(hi), as_vec8<bf16_t>(mid), as_vec8<bf16_t>(lo)};
}

// Largest magnitude of the eight (a NaN stays a NaN): split8 needs it below kSplitMax.
__device__ __forceinline__ float absmax8(const float (&x)[8]) {
  float mx = fabsf(x[0]);
#pragma unroll
  for (int e = 1; e < 8; ++e) mx = vmax(mx, fabsf(x[e]));
  return mx;
}

// split8 of any values.  The largest finite ones keep bf16's largest as their hi
// part.  An infinity or NaN goes into the lo part, which only meets the other
// operand's hi part, beside a hi part of +-1: inf * y is then an infinity of the
// right sign (NaN for y = 0), also where y is infinite; an infinite hi part
// would meet the zeros and signs of the other operand's mid and lo parts.
__device__ __forceinline__ Split8 split8_any(const float (&x)[8]) {
  constexpr float kMax = 0x1.fep127f;
  Split8 s;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const bool finite = fabsf(x[e]) < INFINITY;
    const float y = finite ? x[e] : copysignf(1.0f, x[e]);
    s.hi[e] = (bf16_t)__builtin_amdgcn_fmed3f(y, -kMax, kMax);
    const float a1 = y - (float)s.hi[e];
    s.mid[e] = (bf16_t)a1;
    s.lo[e] = (bf16_t)(finite ? a1 - (float)s.mid[e] : x[e]);
  }
  return s;
}

// acc += a . b over 16 dims: the six partial products, the small ones first.
__device__ __forceinline__ f32x16 mma6(const Split8& a, const Split8& b, f32x16 acc) {
  using E = Elem<bf16_t>;
  acc = E::mfma32(a.lo, b.hi, acc);
  acc = E::mfma32(a.hi, b.lo, acc);
  acc = E::mfma32(a.mid, b.mid, acc);
  acc = E::mfma32(a.mid, b.hi, acc);
  acc = E::mfma32(a.hi, b.mid, acc);
  return E::mfma32(a.hi, b.hi, acc);
}

// b . a in the order of mma6(b, a): the same sum bit for bit with the operands'
// places exchanged.
__device__ __forceinline__ f32x16 mma6_as_ba(const Split8& a, const Split8& b, f32x16 acc) {
  using E = Elem<bf16_t>;
  acc = E::mfma32(a.hi, b.lo, acc);
  acc = E::mfma32(a.lo, b.hi, acc);
  acc = E::mfma32(a.mid, b.mid, acc);
  acc = E::mfma32(a.hi, b.mid, acc);
  acc = E::mfma32(a.mid, b.hi, acc);
  return E::mfma32(a.hi, b.hi, acc);
}

// This lane's row of an operand held in registers: dims 16 ks + 8h .. +7.
template <int D>
__device__ __forceinline__ void load_split(Split8 (&f)[D / 16], const float* __restrict__ row,
                                           int h) {
  f32x4 raw[D / 16][2];
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks)
#pragma unroll
    for (int e = 0; e < 2; ++e)
      raw[ks][e] = *reinterpret_cast<const f32x4*>(row + 16 * ks + 8 * h + 4 * e);
#pragma unroll
  for (int ks = 0; ks < D / 16; ++ks) {
    __builtin_amdgcn_sched_barrier(0);  // one piece's temporaries at a time
    const float x[8] = {raw[ks][0][0], raw[ks][0][1], raw[ks][0][2], raw[ks][0][3],
                        raw[ks][1][0], raw[ks][1][1], raw[ks][1][2], raw[ks][1][3]};
    f[ks] = __any(!(absmax8(x) < kSplitMax)) ? split8_any(x) : split8(x);
  }
}

// A streamed tile of 32 rows in LDS: three bf16 planes, each swizzled as the
// bf16 kernels' tiles.
template <int D>
struct SplitTile {
  static constexpr int PLANE = kChunk * D;    // elements
  static constexpr int ELEMS = 3 * PLANE;
};

// The copy of a 32-row tile: load() issues this thread's global loads, put(i)
// splits piece i (8 floats of one row) and writes it to the three planes.  The
// pieces are put between the MFMAs of the product before the tile's own, with
// no branch among them; finish() writes the tile again, value by value, in the
// rare case that it holds an infinity, a NaN or a value that rounds to one.
template <int D, int NT>
struct SplitCopy {
  static constexpr int N = kChunk * D / 8 / NT;
  static_assert(N >= 1 && kChunk * D / 8 % NT == 0, "tile must split evenly over the workgroup");
  f32x4 buf[N][2];
  float mx;  // largest magnitude put so far
  // rows past `valid` are zero (never used for a valid result, only kept finite)
  __device__ __forceinline__ void load(const float* __restrict__ src, int valid) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int x = (int)threadIdx.x + i * NT, r = x / (D / 8), c = x % (D / 8);
      const f32x4* p = reinterpret_cast<const f32x4*>(src + r * D + 8 * c);
      const bool on = r < valid;
      buf[i][0] = on ? p[0] : f32x4{0.f, 0.f, 0.f, 0.f};
      buf[i][1] = on ? p[1] : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    mx = 0.f;
  }
  __device__ __forceinline__ void store(int i, const Split8& s, bf16_t* tile) const {
    const int x = (int)threadIdx.x + i * NT;
    bf16_t* dst = tile + swz<D>(x / (D / 8), x % (D / 8));
    *reinterpret_cast<bf16x8*>(dst) = s.hi;
    *reinterpret_cast<bf16x8*>(dst + SplitTile<D>::PLANE) = s.mid;
    *reinterpret_cast<bf16x8*>(dst + 2 * SplitTile<D>::PLANE) = s.lo;
  }
  __device__ __forceinline__ void put(int i, bf16_t* tile) {
    const float v[8] = {buf[i][0][0], buf[i][0][1], buf[i][0][2], buf[i][0][3],
                        buf[i][1][0], buf[i][1][1], buf[i][1][2], buf[i][1][3]};
    mx = vmax(mx, absmax8(v));
    store(i, split8(v), tile);
  }
  __device__ __forceinline__ void finish(bf16_t* tile) const {
    if (!__any(!(mx < kSplitMax))) return;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const float v[8] = {buf[i][0][0], buf[i][0][1], buf[i][0][2], buf[i][0][3],
                          buf[i][1][0], buf[i][1][1], buf[i][1][2], buf[i][1][3]};
      store(i, split8_any(v), tile);
    }
  }
  __device__ __forceinline__ void put_all(bf16_t* tile) {
#pragma unroll
    for (int i = 0; i < N; ++i) put(i, tile);
    finish(tile);
  }
  // piece to put after step `st` of `of` product steps (spread from step
  // `first` on); -1: none
  static __device__ __forceinline__ constexpr int piece_after(int st, int of, int first) {
    const int per = (of - first) / N;
    return st >= first && (st - first) % per == per - 1 && (st - first) / per < N
               ? (st - first) / per : -1;
  }
};

// Row r of the tile, dims 16 ks + 8h .. +7.
template <int D>
__device__ __forceinline__ Split8 tile_row(const bf16_t* tile, int r, int ks, int h) {
  Split8 s;
  s.hi = row_a8<bf16_t, D>(tile, r, ks, h);
  s.mid = row_a8<bf16_t, D>(tile + SplitTile<D>::PLANE, r, ks, h);
  s.lo = row_a8<bf16_t, D>(tile + 2 * SplitTile<D>::PLANE, r, ks, h);
  return s;
}

// Dims d0 .. d0+31 of the tile's rows 16 kk + (the C tile's row order).
template <int D>
__device__ __forceinline__ Split8 tile_col(const bf16_t* tile, int d0, int kk) {
  Split8 s;
  s.hi = tr_a8<bf16_t, D>(tile, d0, 16 * kk, 16 * kk + 8);
  s.mid = tr_a8<bf16_t, D>(tile + SplitTile<D>::PLANE, d0, 16 * kk, 16 * kk + 8);
  s.lo = tr_a8<bf16_t, D>(tile + 2 * SplitTile<D>::PLANE, d0, 16 * kk, 16 * kk + 8);
  return s;
}

// Half kk of a C tile (16 of its rows) as the other operand of the next product.
__device__ __forceinline__ Split8 split_acc(const f32x16& acc, int kk) {
  float x[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = acc[8 * kk + e];
  return split8(x);
}

// The same of a tile of any values (dS, where an infinite dO or V makes some); the
// look over the tile takes 1 % of dQ and dK / dV.
__device__ __forceinline__ void split_acc_any(const f32x16& acc, Split8 (&s)[2]) {
  float x[2][8];
#pragma unroll
  for (int e = 0; e < 16; ++e) x[e >> 3][e & 7] = acc[e];
  const float mx = vmax(absmax8(x[0]), absmax8(x[1]));
  if (__any(!(mx < kSplitMax))) {
    s[0] = split8_any(x[0]);
    s[1] = split8_any(x[1]);
  } else {
    s[0] = split8(x[0]);
    s[1] = split8(x[1]);
  }
}

// Steps 0 .. N-1 of a product: step st's LDS operand `load(st)` is read one step
// ahead of its use in `mul(st, operand)`.  The scheduler keeps to the steps (it
// would otherwise read many operands ahead and spill).
template <int N, typename L, typename M>
__device__ __forceinline__ void pipelined(L load, M mul) {
  Split8 cur = load(0);
#pragma unroll
  for (int st = 0; st < N; ++st) {
    Split8 next = cur;
    if (st + 1 < N) next = load(st + 1);
    mul(st, cur);
    cur = next;
    __builtin_amdgcn_sched_barrier(0);
  }
}

}  // namespace

// Rows per workgroup: 128 in four waves, or the 64 of a small block in two.
template <int D, int BE>
struct SplitCfg {
  static constexpr int ROWS = BE >= 128 ? 128 : 64;
  static constexpr int NT = 2 * ROWS;
  // backward: the tiles' loads are issued one product ahead of the product they
  // are put under; a two-wave workgroup (twice the registers of loads a thread)
  // issues them as that product starts
  static constexpr bool EARLY = NT == 256;
  static constexpr int FIRST = EARLY ? 0 : D / 32;
  // dK/dV at head_dim 128: the lo parts of the workgroup's V stay in LDS (its
  // fragments and accumulators would take 24 registers too many), and a
  // two-wave workgroup, of which two share a CU, keeps one Q buffer
  static constexpr bool VLO = D == 128;
  static constexpr int QBUF = VLO && NT == 128 ? 1 : 2;
  // waves per SIMD the registers are sized for: the fragments of a row take
  // 3 D/4 registers (one operand in the forward, two backward)
  static constexpr int WPE_FWD = D == 64 ? 2 : 1;
  static constexpr int WPE_DQ = D == 64 && BE >= 128 ? 2 : 1;
};

// Chunk cursor over a query block's route: slot s, key block kv with nvb valid
// keys, first key c0.
template <int BE>
struct RouteCursor {
  const int32_t* sel;
  const int32_t* vbs;
  int topk, kb;
  int s = -1, kv = 0, nvb = 0, c0 = 0;
  __device__ __forceinline__ bool next() {
    c0 += kChunk;
    while (c0 >= nvb) {
      if (++s >= topk) return false;
      kv = sel[s];
      nvb = (kv >= 0 && kv < kb) ? clamp_valid(vbs[kv], BE) : 0;
      c0 = 0;
    }
    return true;
  }
  __device__ __forceinline__ int row() const { return kv * BE + c0; }
  __device__ __forceinline__ int keys() const { return min(kChunk, nvb - c0); }
};

// ---------------------------------------------------------------------------
// Forward: out = softmax(q k^T scale) v over the selected blocks, LSE base 2,
// combine `out_c * gate` in the epilogue.  Per wave (32 queries) and 32-key
// chunk: S^T = K Q^T, online softmax per lane-query (lane halves hold 16 keys
// each, joined by a permlane swap), O^T += V^T P^T.  A row's offset of the
// exponents is a chunk's max and moves only when a later chunk's passes it by
// more than kMaxSlack: O is rescaled on few chunks, and the exponents of the
// largest weights stay near 0, where fp32 resolves them.  The weights are kept
// as 2^-kMaxSlack of their value, at most 1, so that no product passes v's
// largest.  (An offset 8 above the max took 3 % less, 1.355 against 1.397 ms at 12
// heads, 16 384 tokens, head dim 128, and left each weight with a rounding of up to
// 3e-7; a slack of 2 rescales often enough to cost 2 % more, 6 is as fast as 4.)
// The next V tile is split and written under the S products, the next K tile under
// the O products: one buffer each and two barriers a chunk.
// ---------------------------------------------------------------------------
constexpr int kMaxSlack = 4;

// 2^(x - kMaxSlack), with the rounding of exp2f(x).
__device__ __forceinline__ float weight_exp2(float x) {
  const bool tiny = x < -126.0f;  // the instruction's results end at 2^-126
  return __builtin_ldexpf(__builtin_amdgcn_exp2f(tiny ? x + 64.0f : x),
                          tiny ? -64 - kMaxSlack : -kMaxSlack);
}

template <int D, int BE>
__global__ __launch_bounds__((SplitCfg<D, BE>::NT))
    __attribute__((amdgpu_waves_per_eu(SplitCfg<D, BE>::WPE_FWD))) void
    sparse_fwd_f32_kernel(const float* __restrict__ q, const float* __restrict__ k,
                          const float* __restrict__ v, const int32_t* __restrict__ selected,
                          const int32_t* __restrict__ kv_vbs, float* __restrict__ out,
                          float* __restrict__ fine, float* __restrict__ lse,
                          const float* __restrict__ outc, const float* __restrict__ gate,
                          int gate_mode, int gate_heads, int tiles, int tiles_per_head, int sq,
                          int skv, int qb, int kb, int topk, float c2) {
  using C = SplitCfg<D, BE>;
  using Copy = SplitCopy<D, C::NT>;
  __shared__ __attribute__((aligned(16))) bf16_t ks_[SplitTile<D>::ELEMS];
  __shared__ __attribute__((aligned(16))) bf16_t vs_[SplitTile<D>::ELEMS];
  const int tile = xcd_tile(blockIdx.x, tiles);
  if (tile >= tiles) return;
  const int64_t b = tile / tiles_per_head;
  const int q0 = (tile % tiles_per_head) * C::ROWS;
  const int qblk = q0 / BE;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 31, h = lane >> 5;
  const int myq = q0 + wave * 32 + r;
  const int64_t tok = b * sq + myq;
  Split8 qf[D / 16];
  load_split<D>(qf, q + tok * D, h);
  f32x16 o[D / 32];
#pragma unroll
  for (int mt = 0; mt < D / 32; ++mt) o[mt] = f32x16{};
  float m = -INFINITY, l = 0.f;  // offset of the exponents (log2 units), this half's sum of weights
  const float* kbase = k + b * (int64_t)skv * D;
  const float* vbase = v + b * (int64_t)skv * D;
  RouteCursor<BE> cur{selected + (b * qb + qblk) * topk, kv_vbs, topk, kb};
  Copy cp;
  bool have = cur.next();
  if (have) {
    cp.load(kbase + (int64_t)cur.row() * D, cur.keys());
    cp.put_all(ks_);
  }
  while (have) {
    const int nk = cur.keys();
    cp.load(vbase + (int64_t)cur.row() * D, nk);
    __syncthreads();  // K written; every wave is done with V
    f32x16 sacc = f32x16{};
    pipelined<D / 16>([&](int ks) { return tile_row<D>(ks_, r, ks, h); },
                      [&](int ks, const Split8& a) {
                        sacc = mma6(a, qf[ks], sacc);
                        const int i = Copy::piece_after(ks, D / 16, D / 32);
                        if (i >= 0) cp.put(i, vs_);
                      });
    cp.finish(vs_);
    float cmax = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int key = 8 * (i >> 2) + 4 * h + (i & 3);
      sacc[i] = key < nk ? sacc[i] * c2 : -INFINITY;
      cmax = vmax(cmax, sacc[i]);
    }
    cmax = pair_max32(cmax);
    // a row moves its own offset only, so that its values never depend on the
    // other rows of the wave (a NaN moves it too, and stays)
    const bool grow = !(cmax <= m + (float)kMaxSlack);
    if (__any(grow)) {
      const float mnew = grow ? cmax : m;
      const float alpha = exp2f(m - mnew);
      l *= alpha;
#pragma unroll
      for (int mt = 0; mt < D / 32; ++mt) o[mt] *= alpha;
      m = mnew;
    }
    float psum = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      sacc[i] = weight_exp2(sacc[i] - m);
      psum += sacc[i];
    }
    l += psum;
    const Split8 p[2] = {split_acc(sacc, 0), split_acc(sacc, 1)};
    have = cur.next();
    if (have) cp.load(kbase + (int64_t)cur.row() * D, cur.keys());
    __syncthreads();  // V written; every wave is done with K
    // step x: keys 16 (x / (D/32)) .., dims 32 (x % (D/32)) ..
    pipelined<D / 16>(
        [&](int x) { return tile_col<D>(vs_, 32 * (x % (D / 32)), x / (D / 32)); },
        [&](int x, const Split8& a) {
          o[x % (D / 32)] = mma6(a, p[x / (D / 32)], o[x % (D / 32)]);
          const int i = Copy::piece_after(x, D / 16, D / 32);
          if (i >= 0) cp.put(i, ks_);
        });
    cp.finish(ks_);
  }
  // epilogue: normalise, fused combine, LSE
  const float ltot = pair_sum32(l);
  const float inv = 1.0f / ltot;
  if (lse != nullptr && h == 0) lse[tok] = m + log2f(__builtin_ldexpf(ltot, kMaxSlack));
  const float* ocrow = outc ? outc + (b * qb + qblk) * D : nullptr;
  const float* grow = nullptr;
  float gtok = 1.f;
  if (outc && gate_mode == 1) grow = gate + tok * D;
  if (outc && gate_mode == 2) gtok = gate[tok];
  if (outc && gate_mode == 3)
    grow = gate + (((b / gate_heads) * sq + myq) * gate_heads + b % gate_heads) * D;
#pragma unroll
  for (int mt = 0; mt < D / 32; ++mt) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d0 = 32 * mt + 8 * g + 4 * h;
      f32x4 val;
#pragma unroll
      for (int e = 0; e < 4; ++e) val[e] = o[mt][4 * g + e] * inv;
      if (ocrow && fine) *reinterpret_cast<f32x4*>(fine + tok * D + d0) = val;
      if (ocrow) {
        const f32x4 oc = *reinterpret_cast<const f32x4*>(ocrow + d0);
        const f32x4 gv = grow ? *reinterpret_cast<const f32x4*>(grow + d0)
                              : f32x4{gtok, gtok, gtok, gtok};
#pragma unroll
        for (int e = 0; e < 4; ++e) val[e] = fmaf(oc[e], gv[e], val[e]);
      }
      *reinterpret_cast<f32x4*>(out + tok * D + d0) = val;
    }
  }
}

// dQ rows of a wave from its accumulators: scaled, plus the pooled gradient on
// the block's valid rows.
template <int D, int BE>
__device__ __forceinline__ void store_dq(const f32x16 (&acc)[D / 32], float* __restrict__ dq,
                                         const float* __restrict__ dqc,
                                         const int32_t* __restrict__ q_vbs, int64_t b, int64_t tok,
                                         int myq, int qblk, int qb, int h, float scale) {
  float cdiv = 1.f;
  bool cvalid = false;
  if (dqc) {
    const int32_t cnt = q_vbs[qblk];
    cvalid = myq - qblk * BE < clamp_valid(cnt, BE);
    cdiv = (float)(cnt > 1 ? cnt : 1);
  }
#pragma unroll
  for (int mt = 0; mt < D / 32; ++mt) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d0 = 32 * mt + 8 * g + 4 * h;
      f32x4 cv = {0.f, 0.f, 0.f, 0.f};
      if (cvalid) cv = *reinterpret_cast<const f32x4*>(dqc + (b * qb + qblk) * D + d0);
      f32x4 val;
#pragma unroll
      for (int e = 0; e < 4; ++e) val[e] = acc[mt][4 * g + e] * scale + cv[e] / cdiv;
      *reinterpret_cast<f32x4*>(dq + tok * D + d0) = val;
    }
  }
}

// ---------------------------------------------------------------------------
// dQ (query-owned): per wave (32 queries) and 32-key chunk S^T = K Q^T,
// dP^T = V dO^T, P^T = exp2(S^T c2 - lse), dS^T = P^T (dP^T - delta),
// dQ^T += K^T dS^T; dQ = scale dQ plus the pooled gradient d_q_c / count on the
// block's valid rows.  V is split and written under the S products, the next
// K tile (a second buffer) under the dP products.
// ---------------------------------------------------------------------------
template <int D, int BE>
__global__ __launch_bounds__((SplitCfg<D, BE>::NT))
    __attribute__((amdgpu_waves_per_eu(SplitCfg<D, BE>::WPE_DQ))) void
    sparse_dq_f32_kernel(const float* __restrict__ q, const float* __restrict__ k,
                         const float* __restrict__ v, const float* __restrict__ dout,
                         const float* __restrict__ lse, const float* __restrict__ delta,
                         const int32_t* __restrict__ selected, const int32_t* __restrict__ kv_vbs,
                         float* __restrict__ dq, const float* __restrict__ dqc,
                         const int32_t* __restrict__ q_vbs, int tiles, int tiles_per_head, int sq,
                         int skv, int qb, int kb, int topk, float c2, float scale) {
  using C = SplitCfg<D, BE>;
  using Copy = SplitCopy<D, C::NT>;
  __shared__ __attribute__((aligned(16))) bf16_t ks_[2 * SplitTile<D>::ELEMS];
  __shared__ __attribute__((aligned(16))) bf16_t vs_[SplitTile<D>::ELEMS];
  const int tile = xcd_tile(blockIdx.x, tiles);
  if (tile >= tiles) return;
  const int64_t b = tile / tiles_per_head;
  const int q0 = (tile % tiles_per_head) * C::ROWS;
  const int qblk = q0 / BE;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 31, h = lane >> 5;
  const int myq = q0 + wave * 32 + r;
  const int64_t tok = b * sq + myq;
  Split8 qf[D / 16], df[D / 16];
  load_split<D>(qf, q + tok * D, h);
  load_split<D>(df, dout + tok * D, h);
  const float my_lse = lse[tok], my_delta = delta[tok];
  f32x16 acc[D / 32];
#pragma unroll
  for (int mt = 0; mt < D / 32; ++mt) acc[mt] = f32x16{};
  const float* kbase = k + b * (int64_t)skv * D;
  const float* vbase = v + b * (int64_t)skv * D;
  RouteCursor<BE> cur{selected + (b * qb + qblk) * topk, kv_vbs, topk, kb};
  Copy kc, vc;
  int krow = 0;  // first key row of the chunk
  bool have = cur.next();
  if (have) {
    krow = cur.row();
    kc.load(kbase + (int64_t)krow * D, cur.keys());
    if (C::EARLY) vc.load(vbase + (int64_t)krow * D, cur.keys());
    kc.put_all(ks_);
  }
  int buf = 0;
  while (have) {
    const int nk = cur.keys();
    const bool more = cur.next();
    const int row = krow;
    krow = cur.row();
    if (C::EARLY && more) kc.load(kbase + (int64_t)krow * D, cur.keys());
    if (!C::EARLY) vc.load(vbase + (int64_t)row * D, nk);
    const bf16_t* kt = ks_ + buf * SplitTile<D>::ELEMS;
    bf16_t* knext = ks_ + (buf ^ 1) * SplitTile<D>::ELEMS;
    __syncthreads();  // K written; every wave is done with V
    f32x16 sacc = f32x16{}, pacc = f32x16{};
    pipelined<D / 16>([&](int ks) { return tile_row<D>(kt, r, ks, h); },
                      [&](int ks, const Split8& a) {
                        sacc = mma6(a, qf[ks], sacc);
                        const int i = Copy::piece_after(ks, D / 16, C::FIRST);
                        if (i >= 0) vc.put(i, vs_);
                      });
    vc.finish(vs_);
    if (C::EARLY && more) vc.load(vbase + (int64_t)krow * D, cur.keys());
    if (!C::EARLY && more) kc.load(kbase + (int64_t)krow * D, cur.keys());
    __syncthreads();  // V written; every wave is done with the other K buffer
    pipelined<D / 16>([&](int ks) { return tile_row<D>(vs_, r, ks, h); },
                      [&](int ks, const Split8& a) {
                        pacc = mma6(a, df[ks], pacc);
                        const int i = Copy::piece_after(ks, D / 16, C::FIRST);
                        if (i >= 0) kc.put(i, knext);
                      });
    kc.finish(knext);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int key = 8 * (i >> 2) + 4 * h + (i & 3);
      const float p = key < nk ? exp2f(fmaf(sacc[i], c2, -my_lse)) : 0.f;
      sacc[i] = p * (pacc[i] - my_delta);
    }
    Split8 ds[2];
    split_acc_any(sacc, ds);
    pipelined<D / 16>(
        [&](int x) { return tile_col<D>(kt, 32 * (x % (D / 32)), x / (D / 32)); },
        [&](int x, const Split8& a) {
          acc[x % (D / 32)] = mma6(a, ds[x / (D / 32)], acc[x % (D / 32)]);
        });
    have = more;
    buf ^= 1;
  }
  store_dq<D, BE>(acc, dq, dqc, q_vbs, b, tok, myq, qblk, qb, h, scale);
}

// ---------------------------------------------------------------------------
// dK / dV (key-owned over the CSR in-edges of the key block): per wave (32
// keys) and 32-query item S = Q K^T, dP = dO V^T, P = exp2(S c2 - lse),
// dS = P (dP - delta), dV^T += dO^T P, dK^T += Q^T dS; dK *= scale; pooled
// gradients folded on valid keys; padding keys get zero.  dO is split and
// written under the S products, the next item's Q and statistics (a second
// buffer) under the dP products.
// ---------------------------------------------------------------------------
template <int D, int BE>
__global__ __launch_bounds__((SplitCfg<D, BE>::NT))
    __attribute__((amdgpu_waves_per_eu(1))) void
    sparse_dkdv_f32_kernel(const float* __restrict__ q, const float* __restrict__ k,
                           const float* __restrict__ v, const float* __restrict__ dout,
                           const float* __restrict__ lse, const float* __restrict__ delta,
                           const int32_t* __restrict__ counts, const int32_t* __restrict__ offsets,
                           const int32_t* __restrict__ inverse, const int32_t* __restrict__ kv_vbs,
                           float* __restrict__ dk, float* __restrict__ dv,
                           const float* __restrict__ dkc, const float* __restrict__ dvc, int tiles,
                           int tiles_per_head, int sq, int skv, int qb, int kb, int topk, float c2,
                           float scale) {
  using C = SplitCfg<D, BE>;
  using Copy = SplitCopy<D, C::NT>;
  __shared__ __attribute__((aligned(16))) bf16_t qs_[C::QBUF * SplitTile<D>::ELEMS];
  __shared__ __attribute__((aligned(16))) bf16_t vlo_[C::VLO ? C::ROWS * D : 8];
  __shared__ __attribute__((aligned(16))) bf16_t os_[SplitTile<D>::ELEMS];
  __shared__ __attribute__((aligned(16))) float st_[2][2 * kChunk];  // lse, delta of an item
  const int tile = xcd_tile(blockIdx.x, tiles);
  if (tile >= tiles) return;
  const int64_t b = tile / tiles_per_head;
  const int k0 = (tile % tiles_per_head) * C::ROWS;
  const int kvblk = k0 / BE;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 31, h = lane >> 5;
  const int mykey = k0 + wave * 32 + r;
  const int64_t ktok = b * skv + mykey;
  const bool key_valid = mykey - kvblk * BE < clamp_valid(kv_vbs[kvblk], BE);
  Split8 kf[D / 16], vf[D / 16];
  load_split<D>(kf, k + ktok * D, h);
  load_split<D>(vf, v + ktok * D, h);
  if constexpr (C::VLO) {  // each lane reads back what it wrote
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks)
      *reinterpret_cast<bf16x8*>(vlo_ + swz<D>(wave * 32 + r, 2 * ks + h)) = vf[ks].lo;
  }
  f32x16 dka[D / 32], dva[D / 32];
#pragma unroll
  for (int mt = 0; mt < D / 32; ++mt) dka[mt] = dva[mt] = f32x16{};
  const int64_t meta = b * kb + kvblk;
  const int nedge = counts[meta];
  const int32_t* seg = inverse + b * (int64_t)qb * topk + offsets[meta];
  const float* qbase = q + b * (int64_t)sq * D;
  const float* dbase = dout + b * (int64_t)sq * D;
  // item it: 32 queries (rows (it % SUBS) * 32 ..) of in-edge query block it / SUBS
  constexpr int SUBS = BE / kChunk;
  const int items = nedge * SUBS;
  auto row_of = [&](int it) { return seg[it / SUBS] * BE + (it % SUBS) * kChunk; };
  Copy qc, oc;
  float stv = 0.f;  // lse (threads < 32) or delta (32 .. 63) of the item in qc
  auto load_q = [&](int row) {
    qc.load(qbase + (int64_t)row * D, kChunk);
    if (threadIdx.x < 2 * kChunk)
      stv = threadIdx.x < kChunk ? lse[b * sq + row + threadIdx.x]
                                 : delta[b * sq + row + threadIdx.x - kChunk];
  };
  int row = 0;  // first query row of the item
  if (items > 0) {
    row = row_of(0);
    load_q(row);
    if (C::EARLY) oc.load(dbase + (int64_t)row * D, kChunk);
    qc.put_all(qs_);
    if (threadIdx.x < 2 * kChunk) st_[0][threadIdx.x] = stv;
  }
  for (int it = 0; it < items; ++it) {
    const int buf = it & 1;
    const bool more = it + 1 < items;
    const int next = more ? row_of(it + 1) : 0;
    if (C::EARLY && more) load_q(next);
    if (!C::EARLY) oc.load(dbase + (int64_t)row * D, kChunk);
    const bf16_t* qt = qs_ + (C::QBUF == 2 ? buf : 0) * SplitTile<D>::ELEMS;
    bf16_t* qnext = qs_ + (C::QBUF == 2 ? buf ^ 1 : 0) * SplitTile<D>::ELEMS;
    __syncthreads();  // Q and statistics written; every wave is done with dO
    f32x16 sacc = f32x16{}, pacc = f32x16{};
    // S (queries x keys), lane column = key r, as the forward summed it: P is
    // exp2 of its difference to a sum of the forward's S, which shares S's
    // rounding only then
    pipelined<D / 16>([&](int ks) { return tile_row<D>(qt, r, ks, h); },
                      [&](int ks, const Split8& a) {
                        sacc = mma6_as_ba(a, kf[ks], sacc);
                        const int i = Copy::piece_after(ks, D / 16, C::FIRST);
                        if (i >= 0) oc.put(i, os_);
                      });
    oc.finish(os_);
    if (more && C::EARLY) oc.load(dbase + (int64_t)next * D, kChunk);
    if (more && !C::EARLY && C::QBUF == 2) load_q(next);
    row = next;
    __syncthreads();  // dO written; every wave is done with the other Q buffer
    pipelined<D / 16>([&](int ks) { return tile_row<D>(os_, r, ks, h); },
                      [&](int ks, const Split8& a) {
                        Split8 f = vf[ks];
                        if constexpr (C::VLO)
                          f.lo = row_a8<bf16_t, D>(vlo_, wave * 32 + r, ks, h);
                        pacc = mma6(a, f, pacc);
                        const int i = Copy::piece_after(ks, D / 16, C::FIRST);
                        if (C::QBUF == 2 && i >= 0) qc.put(i, qnext);
                      });
    if (C::QBUF == 2) qc.finish(qnext);
    if (C::QBUF == 2 && more && threadIdx.x < 2 * kChunk) st_[buf ^ 1][threadIdx.x] = stv;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 l4 = *reinterpret_cast<const f32x4*>(st_[buf] + 8 * g + 4 * h);
      const f32x4 d4 = *reinterpret_cast<const f32x4*>(st_[buf] + kChunk + 8 * g + 4 * h);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = 4 * g + j;
        sacc[i] = exp2f(fmaf(sacc[i], c2, -l4[j]));
        pacc[i] = sacc[i] * (pacc[i] - d4[j]);
      }
    }
    const Split8 p[2] = {split_acc(sacc, 0), split_acc(sacc, 1)};
    pipelined<D / 16>(  // dV^T += dO^T P
        [&](int x) { return tile_col<D>(os_, 32 * (x % (D / 32)), x / (D / 32)); },
        [&](int x, const Split8& a) {
          dva[x % (D / 32)] = mma6(a, p[x / (D / 32)], dva[x % (D / 32)]);
        });
    Split8 ds[2];
    split_acc_any(pacc, ds);
    pipelined<D / 16>(  // dK^T += Q^T dS
        [&](int x) { return tile_col<D>(qt, 32 * (x % (D / 32)), x / (D / 32)); },
        [&](int x, const Split8& a) {
          dka[x % (D / 32)] = mma6(a, ds[x / (D / 32)], dka[x % (D / 32)]);
        });
    if (C::QBUF == 1 && more) {
      load_q(next);
      __syncthreads();  // every wave is done with Q and the statistics
      qc.put_all(qs_);
      if (threadIdx.x < 2 * kChunk) st_[buf ^ 1][threadIdx.x] = stv;
    }
  }
  const int32_t cnt = kv_vbs[kvblk];
  const float cdiv = (float)(cnt > 1 ? cnt : 1);
  // pooled-gradient rows loaded before the first store (a load issued after a
  // store also waits for that store)
  f32x4 ckr[D / 32][4], cvr[D / 32][4];
#pragma unroll
  for (int mt = 0; mt < D / 32; ++mt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      ckr[mt][g] = f32x4{0.f, 0.f, 0.f, 0.f};
      cvr[mt][g] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (key_valid && dkc) {
        const int d0 = 32 * mt + 8 * g + 4 * h;
        ckr[mt][g] = *reinterpret_cast<const f32x4*>(dkc + meta * D + d0);
        cvr[mt][g] = *reinterpret_cast<const f32x4*>(dvc + meta * D + d0);
      }
    }
#pragma unroll
  for (int mt = 0; mt < D / 32; ++mt) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d0 = 32 * mt + 8 * g + 4 * h;
      const f32x4 ck = ckr[mt][g], cv = cvr[mt][g];
      f32x4 kk, vv;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        kk[e] = (key_valid ? dka[mt][4 * g + e] * scale : 0.f) + ck[e] / cdiv;
        vv[e] = (key_valid ? dva[mt][4 * g + e] : 0.f) + cv[e] / cdiv;
      }
      *reinterpret_cast<f32x4*>(dk + ktok * D + d0) = kk;
      *reinterpret_cast<f32x4*>(dv + ktok * D + d0) = vv;
    }
  }
}

// ---------------------------------------------------------------------------
// Forward at head_dim 256 on the fp32 matrix core: out = softmax(q k^T scale) v
// over the selected blocks, LSE base 2,
// combine `out_c * gate` in the epilogue.  Per wave and 32-key chunk:
//   S^T = K Q^T (D/2 MFMAs), online softmax per lane-query (lane halves hold
//   16 keys each, joined by a permlane swap), O^T += V^T P^T (16 D/32 MFMAs).
// grid: bh * Sq / 64.
// ---------------------------------------------------------------------------
template <int D, int BE>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(1))) void
sparse_fwd_f32m_kernel(const float* __restrict__ q, const float* __restrict__ k,
                       const float* __restrict__ v, const int32_t* __restrict__ selected,
                       const int32_t* __restrict__ kv_vbs, float* __restrict__ out,
                       float* __restrict__ fine, float* __restrict__ lse,
                       const float* __restrict__ outc, const float* __restrict__ gate,
                       int gate_mode, int gate_heads, int tiles_per_head, int sq, int skv, int qb,
                       int kb, int topk, float c2) {
  constexpr int NT = 128, LD = D + 4;  // threads, LDS row stride (floats)
  __shared__ __attribute__((aligned(16))) float ks[kChunk * LD];
  __shared__ __attribute__((aligned(16))) float vs[kChunk * LD];
  const int64_t b = blockIdx.x / tiles_per_head;
  const int q0 = (blockIdx.x % tiles_per_head) * kRows;
  const int qblk = q0 / BE;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 31, h = lane >> 5;
  const int myq = q0 + wave * 32 + r;
  const int64_t tok = b * sq + myq;
  float qf[D / 2];
  load_frag<D>(qf, q + tok * D, h);
  f32x16 o[D / 32];
#pragma unroll
  for (int mt = 0; mt < D / 32; ++mt) o[mt] = f32x16{};
  float m = -INFINITY, l = 0.f;  // running max (log2 units), this half's partial sum
  const int32_t* sel = selected + (b * qb + qblk) * topk;
  const float* kbase = k + b * (int64_t)skv * D;
  const float* vbase = v + b * (int64_t)skv * D;
  for (int s = 0; s < topk; ++s) {
    const int kv = sel[s];
    if (kv < 0 || kv >= kb) continue;
    const int nvb = clamp_valid(kv_vbs[kv], BE);
    for (int c0 = 0; c0 < nvb; c0 += kChunk) {
      const int nk = min(kChunk, nvb - c0);
      __syncthreads();
      stage32<D, LD, NT>(ks, kbase + ((int64_t)kv * BE + c0) * D, nk);
      stage32<D, LD, NT>(vs, vbase + ((int64_t)kv * BE + c0) * D, nk);
      __syncthreads();
      f32x16 sacc = f32x16{};
      mma_rows<D, LD>(sacc, ks, qf, r, h);
      float cmax = -INFINITY;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int key = 8 * (i >> 2) + 4 * h + (i & 3);
        sacc[i] = key < nk ? sacc[i] * c2 : -INFINITY;
        cmax = fmaxf(cmax, sacc[i]);
      }
      const float mnew = fmaxf(m, pair_max32(cmax));
      const float alpha = exp2f(m - mnew);
      m = mnew;
      float psum = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        sacc[i] = exp2f(sacc[i] - m);
        psum += sacc[i];
      }
      l = l * alpha + psum;
#pragma unroll
      for (int mt = 0; mt < D / 32; ++mt) o[mt] *= alpha;
      mma_cols<D, LD>(o, vs, sacc, r, h);
    }
  }
  // epilogue: normalise, fused combine, LSE
  const float ltot = pair_sum32(l);
  const float inv = 1.0f / ltot;
  if (lse != nullptr && h == 0) lse[tok] = m + log2f(ltot);
  const float* ocrow = outc ? outc + (b * qb + qblk) * D : nullptr;
  const float* grow = nullptr;
  float gtok = 1.f;
  if (outc && gate_mode == 1) grow = gate + tok * D;
  if (outc && gate_mode == 2) gtok = gate[tok];
  if (outc && gate_mode == 3)
    grow = gate + (((b / gate_heads) * sq + myq) * gate_heads + b % gate_heads) * D;
#pragma unroll
  for (int mt = 0; mt < D / 32; ++mt) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d0 = 32 * mt + 8 * g + 4 * h;
      f32x4 val;
#pragma unroll
      for (int e = 0; e < 4; ++e) val[e] = o[mt][4 * g + e] * inv;
      if (ocrow && fine) *reinterpret_cast<f32x4*>(fine + tok * D + d0) = val;
      if (ocrow) {
        const f32x4 oc = *reinterpret_cast<const f32x4*>(ocrow + d0);
        const f32x4 gv = grow ? *reinterpret_cast<const f32x4*>(grow + d0)
                              : f32x4{gtok, gtok, gtok, gtok};
#pragma unroll
        for (int e = 0; e < 4; ++e) val[e] = fmaf(oc[e], gv[e], val[e]);
      }
      *reinterpret_cast<f32x4*>(out + tok * D + d0) = val;
    }
  }
}

// ---------------------------------------------------------------------------
// dQ at head_dim 256 (query-owned): per wave and 32-key chunk S^T = K Q^T, dP^T = V dO^T,
// P^T = exp2(S^T c2 - lse), dS^T = P^T (dP^T - delta), dQ^T += K^T dS^T;
// dQ = scale dQ plus the pooled gradient d_q_c / count on the block's valid
// rows.  grid: bh * Sq / 64.
// ---------------------------------------------------------------------------
template <int D, int BE>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(1))) void
sparse_dq_f32m_kernel(const float* __restrict__ q, const float* __restrict__ k,
                      const float* __restrict__ v, const float* __restrict__ dout,
                      const float* __restrict__ lse, const float* __restrict__ delta,
                      const int32_t* __restrict__ selected, const int32_t* __restrict__ kv_vbs,
                      float* __restrict__ dq, const float* __restrict__ dqc,
                      const int32_t* __restrict__ q_vbs, int tiles_per_head, int sq, int skv,
                      int qb, int kb, int topk, float c2, float scale) {
  constexpr int NT = 128, LD = D + 4;  // threads, LDS row stride (floats)
  __shared__ __attribute__((aligned(16))) float ks[kChunk * LD];
  __shared__ __attribute__((aligned(16))) float vs[kChunk * LD];
  const int64_t b = blockIdx.x / tiles_per_head;
  const int q0 = (blockIdx.x % tiles_per_head) * kRows;
  const int qblk = q0 / BE;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 31, h = lane >> 5;
  const int myq = q0 + wave * 32 + r;
  const int64_t tok = b * sq + myq;
  float qf[D / 2], df[D / 2];
  load_frag<D>(qf, q + tok * D, h);
  load_frag<D>(df, dout + tok * D, h);
  const float my_lse = lse[tok], my_delta = delta[tok];
  f32x16 acc[D / 32];
#pragma unroll
  for (int mt = 0; mt < D / 32; ++mt) acc[mt] = f32x16{};
  const int32_t* sel = selected + (b * qb + qblk) * topk;
  const float* kbase = k + b * (int64_t)skv * D;
  const float* vbase = v + b * (int64_t)skv * D;
  // chunk cursor over the route: slot s, key block kv with nvb valid keys, first key c0
  auto advance = [&](int& s, int& kv, int& nvb, int& c0) {
    c0 += kChunk;
    while (c0 >= nvb) {
      if (++s >= topk) return false;
      kv = sel[s];
      nvb = (kv >= 0 && kv < kb) ? clamp_valid(kv_vbs[kv], BE) : 0;
      c0 = 0;
    }
    return true;
  };
  int s = -1, kv = 0, nvb = 0, c0 = 0;
  bool have = advance(s, kv, nvb, c0);
  while (have) {
    const int nk = min(kChunk, nvb - c0);
    __syncthreads();
    stage32<D, LD, NT>(ks, kbase + ((int64_t)kv * BE + c0) * D, nk);
    stage32<D, LD, NT>(vs, vbase + ((int64_t)kv * BE + c0) * D, nk);
    const bool have2 = advance(s, kv, nvb, c0);
    __syncthreads();
    f32x16 sacc = f32x16{}, pacc = f32x16{};
    mma_rows<D, LD>(sacc, ks, qf, r, h);
    mma_rows<D, LD>(pacc, vs, df, r, h);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int key = 8 * (i >> 2) + 4 * h + (i & 3);
      const float p = key < nk ? exp2f(fmaf(sacc[i], c2, -my_lse)) : 0.f;
      sacc[i] = p * (pacc[i] - my_delta);
    }
    mma_cols<D, LD>(acc, ks, sacc, r, h);
    have = have2;
  }
  store_dq<D, BE>(acc, dq, dqc, q_vbs, b, tok, myq, qblk, qb, h, scale);
}

// ---------------------------------------------------------------------------
// dK / dV at head_dim 256 on the vector ALU (key-owned over the CSR in-edges
// of the key block): four lanes per key, each holding 64 dims; for every row of
// every in-edge query block dV += P dO, dK += dS Q; dK *= scale; pooled
// gradients folded on valid keys; padding keys get zero.  grid: bh * Skv / 64.
// ---------------------------------------------------------------------------
template <int D, int BE>
__global__ __launch_bounds__(256) void sparse_dkdv_f32v_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ dout, const float* __restrict__ lse,
    const float* __restrict__ delta, const int32_t* __restrict__ counts,
    const int32_t* __restrict__ offsets, const int32_t* __restrict__ inverse,
    const int32_t* __restrict__ kv_vbs, float* __restrict__ dk, float* __restrict__ dv,
    const float* __restrict__ dkc, const float* __restrict__ dvc, int tiles_per_head, int sq,
    int skv, int qb, int kb, int topk, float c2, float scale) {
  constexpr int DS = D / 4;
  __shared__ __attribute__((aligned(16))) float qs[kChunk * D];
  __shared__ __attribute__((aligned(16))) float ds_[kChunk * D];
  __shared__ float ls[kChunk], es[kChunk];
  const int64_t b = blockIdx.x / tiles_per_head;
  const int k0 = (blockIdx.x % tiles_per_head) * kRows;
  const int kvblk = k0 / BE;
  const int row = threadIdx.x >> 2, sl = threadIdx.x & 3;
  const int mykey = k0 + row;
  const int64_t ktok = b * skv + mykey;
  const bool key_valid = mykey - kvblk * BE < clamp_valid(kv_vbs[kvblk], BE);
  float kvv[DS], vvv[DS], ak[DS], av[DS];
#pragma unroll
  for (int i = 0; i < DS; ++i) {
    kvv[i] = k[ktok * D + sl * DS + i];
    vvv[i] = v[ktok * D + sl * DS + i];
    ak[i] = av[i] = 0.f;
  }
  const int64_t meta = b * kb + kvblk;
  const int nedge = counts[meta];
  const int32_t* seg = inverse + b * (int64_t)qb * topk + offsets[meta];
  const float* qbase = q + b * (int64_t)sq * D;
  const float* dbase = dout + b * (int64_t)sq * D;
  for (int e = 0; e < nedge; ++e) {
    const int qblock = seg[e];
    for (int c0 = 0; c0 < BE; c0 += kChunk) {
      const int qrow0 = qblock * BE + c0;
      __syncthreads();
      stage_rows_f32<D>(qs, qbase + (int64_t)qrow0 * D, kChunk, kChunk);
      stage_rows_f32<D>(ds_, dbase + (int64_t)qrow0 * D, kChunk, kChunk);
      if (threadIdx.x < kChunk) {
        ls[threadIdx.x] = lse[b * sq + qrow0 + threadIdx.x];
        es[threadIdx.x] = delta[b * sq + qrow0 + threadIdx.x];
      }
      __syncthreads();
      for (int qq = 0; qq < kChunk; ++qq) {
        float s = 0.f, dp = 0.f;
#pragma unroll
        for (int i = 0; i < DS; ++i) {
          s = fmaf(qs[qq * D + sl * DS + i], kvv[i], s);
          dp = fmaf(ds_[qq * D + sl * DS + i], vvv[i], dp);
        }
        const float p = exp2f(fmaf(quad_sum(s), c2, -ls[qq]));
        const float dsv = p * (quad_sum(dp) - es[qq]);
#pragma unroll
        for (int i = 0; i < DS; ++i) {
          av[i] = fmaf(p, ds_[qq * D + sl * DS + i], av[i]);
          ak[i] = fmaf(dsv, qs[qq * D + sl * DS + i], ak[i]);
        }
      }
    }
  }
  const int32_t cnt = kv_vbs[kvblk];
  const float cdiv = (float)(cnt > 1 ? cnt : 1);
#pragma unroll
  for (int i = 0; i < DS; ++i) {
    const int d = sl * DS + i;
    const float ck = (key_valid && dkc) ? dkc[meta * D + d] / cdiv : 0.f;
    const float cv = (key_valid && dvc) ? dvc[meta * D + d] / cdiv : 0.f;
    dk[ktok * D + d] = (key_valid ? ak[i] * scale : 0.f) + ck;
    dv[ktok * D + d] = (key_valid ? av[i] : 0.f) + cv;
  }
}

// ---------------------------------------------------------------------------
// Host launchers (the C ABI in fine_fwd.hip / fine_bwd.hip dispatches fp32
// here).  Shapes: head_dim 64 / 128 / 256, block volume 64 / 128 / 256 (the
// Python layer pads other shapes onto these, as for bf16).
// ---------------------------------------------------------------------------
// every kernel shape has 64 | block volume, so a workgroup's 64 rows lie in
// one block and sequence lengths (multiples of the volume) split evenly
static bool f32_shape(int D, int be) {
  return (D == 64 || D == 128 || D == 256) && (be == 64 || be == 128 || be == 256);
}

#define VSA_F32_SHAPES(X) \
  X(64, 64) X(64, 128) X(64, 256) X(128, 64) X(128, 128) X(128, 256) X(256, 64) X(256, 128) X(256, 256)

int sparse_fwd_f32(const void* q, const void* k, const void* v, const int32_t* selected,
                   const int32_t* kv_vbs, void* out, void* fine, float* lse, const void* out_c,
                   const void* gate, int gate_mode, int gate_heads, int64_t bh, int64_t sq,
                   int64_t skv, int D, int be, int topk, float scale, hipStream_t s) {
  if (!f32_shape(D, be)) return VSA_ERR_UNSUPPORTED;
  if (bh * (sq / kRows) > (1LL << 30)) return VSA_ERR_SHAPE;
  const float c2 = scale * kLog2e;
#define VSA_F(DD, BB)                                                                           \
  if (D == DD && be == BB) {                                                                    \
    if constexpr (DD <= 128) {                                                                  \
      using C = SplitCfg<DD, BB>;                                                               \
      const int tph = (int)(sq / C::ROWS), tiles = (int)(bh * tph);                             \
      hipLaunchKernelGGL((sparse_fwd_f32_kernel<DD, BB>), dim3((unsigned)((tiles + 7) / 8 * 8)), \
                         dim3(C::NT), 0, s, (const float*)q, (const float*)k, (const float*)v,  \
                         selected, kv_vbs, (float*)out, (float*)fine, lse, (const float*)out_c, \
                         (const float*)gate, gate_mode, gate_heads, tiles, tph, (int)sq,        \
                         (int)skv, (int)(sq / BB), (int)(skv / BB), topk, c2);                  \
    } else {                                                                                    \
      const int tph = (int)(sq / kRows);                                                        \
      hipLaunchKernelGGL((sparse_fwd_f32m_kernel<DD, BB>), dim3((unsigned)(bh * tph)),          \
                         dim3(128), 0, s, (const float*)q, (const float*)k, (const float*)v,    \
                         selected, kv_vbs, (float*)out, (float*)fine, lse, (const float*)out_c, \
                         (const float*)gate, gate_mode, gate_heads, tph, (int)sq, (int)skv,     \
                         (int)(sq / BB), (int)(skv / BB), topk, c2);                            \
    }                                                                                           \
    return vsa_check_launch();                                                                  \
  }
  VSA_F32_SHAPES(VSA_F)
#undef VSA_F
  return VSA_ERR_UNSUPPORTED;
}

int sparse_dq_f32(const void* q, const void* k, const void* v, const void* dout,
                  const float* lse, const float* delta, const int32_t* selected,
                  const int32_t* kv_vbs, void* dq, const void* dqc, const int32_t* q_vbs,
                  int64_t bh, int64_t sq, int64_t skv, int D, int be, int topk, float scale,
                  hipStream_t s) {
  if (!f32_shape(D, be)) return VSA_ERR_UNSUPPORTED;
  if (bh * (sq / kRows) > (1LL << 30)) return VSA_ERR_SHAPE;
  const float c2 = scale * kLog2e;
#define VSA_F(DD, BB)                                                                           \
  if (D == DD && be == BB) {                                                                    \
    if constexpr (DD <= 128) {                                                                  \
      using C = SplitCfg<DD, BB>;                                                               \
      const int tph = (int)(sq / C::ROWS), tiles = (int)(bh * tph);                             \
      hipLaunchKernelGGL((sparse_dq_f32_kernel<DD, BB>), dim3((unsigned)((tiles + 7) / 8 * 8)), \
                         dim3(C::NT), 0, s, (const float*)q, (const float*)k, (const float*)v,  \
                         (const float*)dout, lse, delta, selected, kv_vbs, (float*)dq,          \
                         (const float*)dqc, q_vbs, tiles, tph, (int)sq, (int)skv,               \
                         (int)(sq / BB), (int)(skv / BB), topk, c2, scale);                     \
    } else {                                                                                    \
      const int tph = (int)(sq / kRows);                                                        \
      hipLaunchKernelGGL((sparse_dq_f32m_kernel<DD, BB>), dim3((unsigned)(bh * tph)),           \
                         dim3(128), 0, s, (const float*)q, (const float*)k, (const float*)v,    \
                         (const float*)dout, lse, delta, selected, kv_vbs, (float*)dq,          \
                         (const float*)dqc, q_vbs, tph, (int)sq, (int)skv, (int)(sq / BB),      \
                         (int)(skv / BB), topk, c2, scale);                                     \
    }                                                                                           \
    return vsa_check_launch();                                                                  \
  }
  VSA_F32_SHAPES(VSA_F)
#undef VSA_F
  return VSA_ERR_UNSUPPORTED;
}

int sparse_dkdv_f32(const void* q, const void* k, const void* v, const void* dout,
                    const float* lse, const float* delta, const int32_t* counts,
                    const int32_t* offsets, const int32_t* inverse, const int32_t* kv_vbs,
                    void* dk, void* dv, const void* dkc, const void* dvc, int64_t bh, int64_t sq,
                    int64_t skv, int D, int be, int topk, float scale, hipStream_t s) {
  if (!f32_shape(D, be)) return VSA_ERR_UNSUPPORTED;
  if (bh * (skv / kRows) > (1LL << 30)) return VSA_ERR_SHAPE;
  const float c2 = scale * kLog2e;
  // head_dim 64 / 128 on the matrix core, 256 on the vector ALU
#define VSA_F(DD, BB)                                                                             \
  if (D == DD && be == BB) {                                                                      \
    if constexpr (DD <= 128) {                                                                    \
      using C = SplitCfg<DD, BB>;                                                                 \
      const int tph = (int)(skv / C::ROWS), tiles = (int)(bh * tph);                              \
      hipLaunchKernelGGL((sparse_dkdv_f32_kernel<DD, BB>), dim3((unsigned)((tiles + 7) / 8 * 8)), \
                         dim3(C::NT), 0, s, (const float*)q, (const float*)k, (const float*)v,    \
                         (const float*)dout, lse, delta, counts, offsets, inverse, kv_vbs,        \
                         (float*)dk, (float*)dv, (const float*)dkc, (const float*)dvc, tiles,     \
                         tph, (int)sq, (int)skv, (int)(sq / BB), (int)(skv / BB), topk, c2,       \
                         scale);                                                                  \
    } else {                                                                                      \
      const int tph = (int)(skv / kRows);                                                         \
      hipLaunchKernelGGL((sparse_dkdv_f32v_kernel<DD, BB>), dim3((unsigned)(bh * tph)),           \
                         dim3(256), 0, s, (const float*)q, (const float*)k, (const float*)v,      \
                         (const float*)dout, lse, delta, counts, offsets, inverse, kv_vbs,        \
                         (float*)dk, (float*)dv, (const float*)dkc, (const float*)dvc, tph,       \
                         (int)sq, (int)skv, (int)(sq / BB), (int)(skv / BB), topk, c2, scale);    \
    }                                                                                             \
    return vsa_check_launch();                                                                    \
  }
  VSA_F32_SHAPES(VSA_F)
#undef VSA_F
  return VSA_ERR_UNSUPPORTED;
}

}  // namespace vsa
