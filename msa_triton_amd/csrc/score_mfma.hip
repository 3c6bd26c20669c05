// Stage 1 on MFMA: block maxima of the indexer logits with a certified exact winner,
// for bf16 and fp16 inputs (score_fwd_mfma_kernel) and fp32 inputs (score_fwd_f32_kernel).
// Measured against the FP64 kernel that fp16 and fp32 used before (score_fwd_exact, one
// wave per row and block): 8192 tokens x 4 groups of 128 dims in fp16 85.8 -> 0.13 ms with
// the top-k, 2048 tokens x 2 groups in fp32 1.05 -> 0.12 ms.
//
// Work unit: a tile of 128 consecutive (t, g) rows of the flattened [T*G] row
// space, 4 waves x 32 rows. A wave keeps its rows' query fragments in
// registers and, for every key block reachable by the tile, evaluates its
// 32 x 128 logits on v_mfma_f32_16x16x32_bf16 (exact bf16 products, fp32
// accumulation) against the block held in LDS. Key blocks are double-buffered:
// the next block is fetched from memory while the current one is used, so one
// barrier per block orders all LDS traffic. With the index dim a multiple of 32
// the blocks go from memory straight to LDS (global_load_lds_dwordx4: 16 bytes
// per lane, no staging registers) into unpadded rows whose 16-byte chunks are
// XOR-swizzled by row, so the fragment reads stay bank-conflict free. Tiles are
// issued heaviest first (the last rows of a sequence see the most blocks), each as one
// or more workgroups (tile_parts). Each key block's largest norm and safety (for the error
// bound below) come from a pre-pass (score_block_norms) instead of being formed per tile.
//
// Exactness (the public score is the reference's FP32 form of the exact winning dot,
// public_score, and the winner set must be the exact one, index_score.py:121-136): with
//   E = (Di_pad + 8) * 2^-22 * ||q|| * max_k ||k||  >=  |s_mfma - s_exact|,
// every key whose approximate directed logit is below (max_approx - 2E) is
// certainly beaten by the approximate winner. The running maximum and runner-up
// are tracked on logits whose 7 low mantissa bits are replaced by the key's
// position (4 kt + i, an inline constant of the and-or; the quarter q4 is
// recovered after the cross-lane merge and the key is 16 kt + 4 q4 + i),
// which moves each by < 2^-16 of its magnitude: the test therefore also allows
// 2^-15 max(|max|, |runner-up|) plus the smallest normal float. If exactly one key
// survives, it is the unique exact winner and only its dot is evaluated in FP64: a lane
// pair owns the row, each lane runs one half of exact_dot's fixed order (two
// sequential chains over the halves of the index dim) from the query half it keeps in
// registers and the key row in LDS, and the halves are added in that order. Each
// bf16 x bf16 product comes from v_dot2_f32_bf16 against a key word with the other
// half masked to zero: exact in fp32 when every nonzero element of the query row and
// the key block lies in [2^-60, 2^55) ("safe": products then are normal fp32 numbers,
// and no MFMA sum can overflow), and adding that exact product in FP64 gives the bits
// of exact_dot's fused multiply-add. (fp16 products are exact in fp32 whatever the finite
// values; v_fma_mix_f32 forms them. fp32 elements are converted and fused in FP64.) Pairs of
// an unsafe row or block go to the resolve kernel below.
// Otherwise the (row, block) pair is marked in a bitmap that a second
// kernel (score_fwd_resolve) settles after the main pass: the keys within the bound of the
// row's maximum are evaluated in FP64 (same order) for the maximum, tie count and first
// winner. Deferring keeps the rare ambiguous rows (a few per
// thousand on random data) from holding the other waves of a workgroup at the
// next block barrier.
// A negative scale flips the query signs once (exact), so every comparison is
// on the directed dot.
#include <algorithm>
#include <type_traits>

#include "mfma_util.hpp"
#include "score_mfma.hpp"

namespace msa {

namespace {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

constexpr int kTileRows = 128;  // 4 waves x 32 rows
constexpr int kShortSeq = 16;   // tokens of the longest sequence that score_fwd_short takes
constexpr int kThreads = 256;

// Workspace: squared key norms (fp32 per key), the key blocks' norms (fp32, at each
// block's first key), then the ambiguous-pair bitmap, block-major: bit
// block * rows_pad + row of 32-bit words, rows_pad = rows rounded up to a whole number
// of resolve chunks.
constexpr int kResolveRows = 4096;  // rows per resolve wave: 64 bits for each of its lanes
int64_t align256(int64_t x) { return (x + 255) & ~int64_t{255}; }
int64_t ws_bnorm_offset(int64_t T) { return align256(4 * (T > 0 ? T : 1)); }
int64_t ws_bitmap_offset(int64_t T) { return 2 * ws_bnorm_offset(T); }
int64_t rows_padded(int64_t rows) { return (rows + kResolveRows - 1) / kResolveRows * kResolveRows; }
int64_t bitmap_words(int64_t rows, int64_t NB) { return rows_padded(rows) / 32 * NB; }

template <int NK>
struct ScoreSmem {
  static constexpr int DP = 32 * NK;
  static constexpr int RS = DP + 8;  // row stride (bf16) of a padded key block (index dim below DP)
  alignas(16) uint16_t k[2][128 * RS];  // full-width blocks use the first 128 * DP entries (swizzled rows)
};

// Offset (bf16 elements) of dims [d, d + 8) of key `row` in a buffered block (d a
// multiple of 8). Full width: rows DP apart, 16-byte chunk c at c ^ swz(row), with
// swz chosen so the 16 rows one fragment read touches land on 16 distinct bank
// groups. Otherwise: rows DP + 8 apart, unswizzled.
template <int NK, bool FULLD>
__device__ __forceinline__ int key_off(int row, int d) {
  constexpr int DP = 32 * NK, CPK = DP / 8;
  if constexpr (FULLD) {
    constexpr int SH = NK == 4 ? 0 : (NK == 2 ? 1 : 2);  // rows sharing a bank base: 16 / CPK apart
    return row * DP + 8 * ((d >> 3) ^ ((row >> SH) & (CPK - 1)));
  } else {
    return row * (DP + 8) + d;
  }
}

// Logit bits with the key position in the 7 low mantissa bits (see the header comment).
__device__ __forceinline__ float pack_key(float v, uint32_t pos) {
  return __uint_as_float((__float_as_uint(v) & 0xffffff80u) | pos);
}
constexpr float kMaskedLogit = -3.0e38f;  // a finite stand-in for masked keys (packing keeps it finite)

// v_max3_f32 on finite values. Written out because the optimiser, given fmaxf, adds a
// canonicalisation of every operand whose bits it cannot trace to an FP operation.
__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

__device__ __forceinline__ float min2(float a, float b) {
  float r;
  asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// The value of this lane and that of lane ^ 32 (or ^ 16), in an order that depends on
// the lane: v_permlane32_swap (v_permlane16_swap) of x with itself. For a symmetric
// combination (max, min, a sum of two) the order does not matter.
struct LanePair {
  uint32_t a, b;
};
__device__ __forceinline__ LanePair pair_xor32(uint32_t x) {
  const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  return LanePair{r[0], r[1]};
}
__device__ __forceinline__ LanePair pair_xor16(uint32_t x) {
  const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  return LanePair{r[0], r[1]};
}

// Both bf16 of a word zero or of magnitude in [2^-60, 2^55) (biased exponent 67 .. 181):
// the product of two such values is zero or a normal fp32 number below 2^110, and a
// sum of up to 128 of them stays below 2^117.
__device__ __forceinline__ bool bf16_safe(uint32_t x16) {
  const uint32_t e = (x16 >> 7) & 0xffu;
  return (x16 & 0x7fffu) == 0u || (e >= 67u && e <= 181u);
}
// fp16: every product of two finite values is exact in fp32 (22 significant bits, from 2^-48
// to 2^32, and sums of 128 stay finite), so only infinities and NaN are unsafe.
template <int DT>
__device__ __forceinline__ bool word_safe(uint32_t w) {
  if constexpr (DT == kF16) return (w & 0x7c00u) != 0x7c00u && (w & 0x7c000000u) != 0x7c000000u;
  else return bf16_safe(w & 0xffffu) && bf16_safe(w >> 16);
}

// fp32: zero or of magnitude in [2^-40, 2^55), so that the products of the bf16 terms (each
// no smaller than 2^-63) are normal and their sums stay finite.
__device__ __forceinline__ bool f32_safe(uint32_t w) {
  const uint32_t e = (w >> 23) & 0xffu;
  return (w & 0x7fffffffu) == 0u || (e >= 87u && e <= 181u);
}

// Eight consecutive elements as loaded.
template <int DT>
struct Words8 {
  static constexpr int N = DT == kF32 ? 8 : 4;
  uint32_t w[N];
};
template <int DT>
__device__ __forceinline__ Words8<DT> load_words(const void* __restrict__ base, int64_t i) {
  Words8<DT> r;
  const uint4* p = reinterpret_cast<const uint4*>(static_cast<const char*>(base) + i * (DT == kF32 ? 4 : 2));
#pragma unroll
  for (int u = 0; u < Words8<DT>::N / 4; ++u) {
    const uint4 x = p[u];
    r.w[4 * u] = x.x, r.w[4 * u + 1] = x.y, r.w[4 * u + 2] = x.z, r.w[4 * u + 3] = x.w;
  }
  return r;
}
// n2 += the square(s) of the word's element(s); safe cleared if one is not safe.
template <int DT>
__device__ __forceinline__ void add_square(uint32_t w, float& n2, bool& safe) {
  if constexpr (DT == kF32) {
    n2 = fmaf(__uint_as_float(w), __uint_as_float(w), n2);
    safe = safe && f32_safe(w);
  } else {
    n2 = fmaf(lo16_f32<DT>(w), lo16_f32<DT>(w), n2);
    n2 = fmaf(hi16_f32<DT>(w), hi16_f32<DT>(w), n2);
    safe = safe && word_safe<DT>(w);
  }
}
// An MFMA operand of eight fp32 elements as two bf16 terms, x ~ hi + mid (to 2^-18 |x|).
struct SplitFrag {
  bf16x8 hi, mid;
};
__device__ __forceinline__ SplitFrag split_frag(const uint32_t (&w)[8]) {
  uint32_t h[4], m[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const float x0 = __uint_as_float(w[2 * u]), x1 = __uint_as_float(w[2 * u + 1]);
    h[u] = cvt_pk_bf16(x0, x1);
    m[u] = cvt_pk_bf16(sub_lo_half(h[u], x0), sub_hi_half(h[u], x1));
  }
  return SplitFrag{__builtin_bit_cast(bf16x8, make_uint4(h[0], h[1], h[2], h[3])),
                   __builtin_bit_cast(bf16x8, make_uint4(m[0], m[1], m[2], m[3]))};
}
// acc += a . b with both operands as two bf16 terms (the smaller products first).
__device__ __forceinline__ f32x4 mfma_split(const SplitFrag& a, const SplitFrag& b, f32x4 acc) {
  acc = mfma(a.mid, b.hi, acc);
  acc = mfma(a.hi, b.mid, acc);
  return mfma(a.hi, b.hi, acc);
}

// fp32 product of the low (lo) or high element of a and of b, exact when both are safe.
template <int DT>
__device__ __forceinline__ float prod_lo(uint32_t a, uint32_t b) {
  if constexpr (DT == kF16)
    return __builtin_fmaf(lo16_f32<DT>(a), lo16_f32<DT>(b), 0.f);  // v_fma_mix_f32
  else
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, a),
                                           __builtin_bit_cast(bf16x2_t, b & 0xffffu), 0.0f, false);
}
template <int DT>
__device__ __forceinline__ float prod_hi(uint32_t a, uint32_t b) {
  if constexpr (DT == kF16)
    return __builtin_fmaf(hi16_f32<DT>(a), hi16_f32<DT>(b), 0.f);
  else
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, a),
                                           __builtin_bit_cast(bf16x2_t, b & 0xffff0000u), 0.0f, false);
}

// Two logits x, y (keys at positions pos, pos + 1) into a running top 2 (m1 the maximum,
// m2 the largest other value, m1 >= m2 throughout): the second largest of {m1, m2, x, y}
// is max(m2, med3(m1, x, y)). med3(a, b, +inf) is max(a, b); unlike fmaxf it needs no
// canonicalised inputs. pinf is +inf in a register the optimiser cannot see through, or it
// would turn the med3 back into a maximum with canonicalisations.
__device__ __forceinline__ void fold_pair(float x, float y, uint32_t pos, float pinf, float& m1, float& m2) {
  x = pack_key(x, pos);
  y = pack_key(y, pos + 1);
  const float t = __builtin_amdgcn_fmed3f(m1, x, y);
  m2 = __builtin_amdgcn_fmed3f(m2, t, pinf);
  m1 = max3(m1, x, y);
}

// A row's top 2 over its four key quarters (lanes c, c + 16, c + 32, c + 48): a1 the
// maximum, a2 the largest other value, and the key index of the maximum (unique whenever
// the row is certified).
struct RowTop {
  float a1, a2;
  int key;
};
__device__ __forceinline__ RowTop merge_quarters(float m1, float m2, int q4) {
  RowTop r{m1, m2, 0};
#pragma unroll
  for (int o = 16; o <= 32; o <<= 1) {  // with the quarter of lane ^ o
    const LanePair p1 = o == 16 ? pair_xor16(__float_as_uint(r.a1)) : pair_xor32(__float_as_uint(r.a1));
    const LanePair p2 = o == 16 ? pair_xor16(__float_as_uint(r.a2)) : pair_xor32(__float_as_uint(r.a2));
    const float u = __uint_as_float(p1.a), v = __uint_as_float(p1.b);
    r.a2 = max3(__uint_as_float(p2.a), __uint_as_float(p2.b), min2(u, v));
    r.a1 = max3(u, v, v);
  }
  int wq = m1 == r.a1 ? q4 : 4;  // the quarter holding the maximum
  const LanePair w16 = pair_xor16(static_cast<uint32_t>(wq));
  wq = min(static_cast<int>(w16.a), static_cast<int>(w16.b));
  const LanePair w32 = pair_xor32(static_cast<uint32_t>(wq));
  wq = min(static_cast<int>(w32.a), static_cast<int>(w32.b));
  const int pos = static_cast<int>(__float_as_uint(r.a1) & 0x7fu);  // 4 kt + i
  r.key = 16 * (pos >> 2) + 4 * wq + (pos & 3);
  return r;
}

// The sum of the two halves of a row's dot, held by lanes l and l ^ 32 (half 0 first; the
// value is that of the lane pair whatever the lane).
__device__ __forceinline__ double add_halves(double half) {
  const uint64_t hbits = static_cast<uint64_t>(__double_as_longlong(half));
  const LanePair hlo = pair_xor32(static_cast<uint32_t>(hbits));
  const LanePair hhi = pair_xor32(static_cast<uint32_t>(hbits >> 32));
  const double h0 = __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hhi.a) << 32) | hlo.a));
  const double h1 = __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hhi.b) << 32) | hlo.b));
  return h0 + h1;
}

// The logits' error bound per ||q|| max ||k||: half the distance below the approximate
// maximum from which a key is certainly beaten. 16-bit inputs: DP exact products summed in
// fp32. fp32 inputs enter as two bf16 terms each (s = qh kh + qh km + qm kh): the terms left
// out are below 3 x 2^-18 |q| |k| in all, and 3 DP products are summed.
template <int DT, int DP>
constexpr float logit_error() {
  return DT == kF32 ? 3.1f * 0x1p-18f + static_cast<float>(3 * DP + 8) * 0x1p-22f
                    : static_cast<float>(DP + 8) * 0x1p-22f;
}

// Iteration space of a tile: (sequence, block) pairs for every sequence overlapping
// the tile rows [r0, r0 + nr), blocks 0 .. the last row's query block.
struct BlockCursor {
  int s;       // sequence
  int b;       // sequence-local block
  int b_last;  // last block of this sequence the tile needs
};

__device__ __forceinline__ int last_block_of(const int32_t* __restrict__ cu, int s, int64_t r0, int nr, int G,
                                             int B) {
  const int64_t start = cu[s], end = cu[s + 1];
  const int64_t t_last = (r0 + nr - 1) / G;
  const int64_t t = t_last < end - 1 ? t_last : end - 1;
  return static_cast<int>((t - start) / B);
}

// Next (s, b) after c; s == nseq when the tile has no more blocks. Sequences of up to `shortest`
// tokens (0: the empty ones) are left out.
__device__ __forceinline__ BlockCursor next_block(const int32_t* __restrict__ cu, int nseq, BlockCursor c,
                                                  int64_t r0, int nr, int G, int B, int shortest) {
  if (c.b < c.b_last) {
    ++c.b;
    return c;
  }
  const int64_t t_last = (r0 + nr - 1) / G;
  for (int s = c.s + 1; s < nseq && cu[s] <= t_last; ++s) {
    if (cu[s + 1] - cu[s] > shortest) return BlockCursor{s, 0, last_block_of(cu, s, r0, nr, G, B)};
  }
  return BlockCursor{nseq, 0, -1};
}

// Part `part` of `parts` equal runs of the tile's (sequence, block) pairs: its first pair and
// their number.
__device__ __forceinline__ BlockCursor tile_share(const int32_t* __restrict__ cu, int nseq, int64_t r0, int nr, int G,
                                                  int B, int shortest, int part, int parts, int& todo) {
  const int64_t t_last = (r0 + nr - 1) / G;
  const int s0 = find_seq(cu, nseq, r0 / G);
  int pairs = 0;
  for (int s = s0; s < nseq && cu[s] <= t_last; ++s)
    if (cu[s + 1] - cu[s] > shortest) pairs += last_block_of(cu, s, r0, nr, G, B) + 1;
  int skip = static_cast<int>(static_cast<int64_t>(pairs) * part / parts);
  todo = static_cast<int>(static_cast<int64_t>(pairs) * (part + 1) / parts) - skip;
  if (todo <= 0) return BlockCursor{nseq, 0, -1};
  for (int s = s0; s < nseq && cu[s] <= t_last; ++s) {
    if (cu[s + 1] - cu[s] <= shortest) continue;
    const int last = last_block_of(cu, s, r0, nr, G, B);
    if (skip <= last) return BlockCursor{s, skip, last};
    skip -= last + 1;
  }
  return BlockCursor{nseq, 0, -1};
}

// Blocks without a causal key: score -inf, tie code 0, for up to 32 rows from `row0` (those
// of one wave); the tile's parts (blockIdx.y) share the rows.
__device__ __forceinline__ void fill_future(const int32_t* __restrict__ cu, int nseq, int64_t row0, int nr, int G,
                                            int NB, int B, float* __restrict__ scores, int32_t* __restrict__ tie) {
  const int lane = threadIdx.x & 63, j0 = lane & 31;
  int own = NB;
  if (j0 < nr) {
    const int64_t t = (row0 + j0) / G;
    own = static_cast<int>((t - cu[find_seq(cu, nseq, t)]) / B);
  }
  for (int j = blockIdx.y; j < 32 && j < nr; j += gridDim.y) {
    const int64_t base = (row0 + j) * NB;
    for (int b = __shfl(own, j, kWave) + 1 + lane; b < NB; b += kWave) {
      scores[base + b] = -__builtin_inff();
      if (tie) tie[base + b] = 0;
    }
  }
}

}  // namespace

// The squared norm of `n` elements from element i, rounded up by 1.0001 (bounds the fp32
// rounding of the sum), with the sign bit set when one of them is not safe.
template <int DT>
__device__ __forceinline__ float signed_norm2(const void* __restrict__ ik, int64_t i, int n) {
  float n2 = 0.f;
  bool safe = true;
#pragma unroll 8  // a row's loads in flight together
  for (int d = 0; d < n; d += 8) {
    const Words8<DT> w = load_words<DT>(ik, i + d);
#pragma unroll
    for (int u = 0; u < Words8<DT>::N; ++u) add_square<DT>(w.w[u], n2, safe);
  }
  return safe ? n2 * 1.0001f : -(fabsf(n2) * 1.0001f) - 1.0f;
}

// The key norms that enter the error bound, and the ambiguous-pair bitmap cleared. Per key
// block, stored at the block's first key: the largest key norm, sqrt(max ||k||^2), negated
// when a key of the block is not safe (or not a number). Safety is read from the sign bit:
// a block whose only unsafe key is NaN (fmaxf skips its NaN entry) and whose other keys are
// zero stores -0. One workgroup per 64 tokens; for each block that starts among them (one or
// two when 64 <= B <= 128, this kernel's range) two threads take each key, half a row each.
// Bound by the latency of its few loads (8.4 us at 2048 keys of 512 bytes; with one lane
// per whole row in one wave per block 14.7 us, with the lanes side by side along a row 39.8 us:
// the shuffles).
template <int DT>
__global__ __launch_bounds__(256) void score_block_norms(const void* __restrict__ ik, const int32_t* __restrict__ cu,
                                                         int nseq, int64_t T, int Di, int B, int shortest,
                                                         float* __restrict__ bnorm, uint32_t* __restrict__ amb,
                                                         int64_t amb_words) {
  __shared__ float part[256];
  __shared__ float wmax[2];
  const int64_t a = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (a < amb_words) amb[a] = 0u;
  const int tid = threadIdx.x, lane = tid & 63, key = tid & 127, hf = tid >> 7;
  const int64_t base = static_cast<int64_t>(blockIdx.x) * 64;
  if (base >= T) return;  // whole workgroup
  int32_t end = 0;
  bool starts = false;
  if (base + lane < T) {  // every wave looks at the same 64 tokens
    const int32_t t = static_cast<int32_t>(base) + lane;
    const int s = find_seq_near(cu, nseq, t);
    end = cu[s + 1];
    starts = end - cu[s] > shortest && (t - cu[s]) % B == 0;
  }
  for (uint64_t m = __ballot(starts); m; m &= m - 1) {
    const int l = __builtin_ctzll(m);
    const int64_t t0 = base + l;
    const int64_t e0 = __shfl(end, l, kWave);
    const int nk = static_cast<int>(t0 + B < e0 ? B : e0 - t0);
    const int n1 = Di / 16 * 8;  // the first half's elements, a multiple of 8
    part[tid] = key < nk ? signed_norm2<DT>(ik, (t0 + key) * Di + (hf ? n1 : 0), hf ? Di - n1 : n1) : 0.f;
    __syncthreads();
    if (tid < 128) {
      const float x = part[tid], y = part[tid + 128];
      const float r = sqrtf(fmaxf(wave_max_f32(fabsf(x) + fabsf(y)), 0.f));  // (maxima skip NaN)
      const bool ok = __ballot(!(x >= 0.f && y >= 0.f)) == 0;
      if (lane == 0) wmax[tid >> 6] = ok ? r : -r;
    }
    __syncthreads();
    if (tid == 0) {
      const float x = wmax[0], y = wmax[1], r = fmaxf(fabsf(x), fabsf(y));
      bnorm[t0] = __builtin_signbit(x) == 0 && __builtin_signbit(y) == 0 ? r : -r;
    }
    __syncthreads();  // part is rewritten for the next block
  }
}

// The same for blocks of fewer than 64 keys, in two passes: the norms of all keys (and the
// bitmap), then one thread per block.
template <int DT>
__global__ __launch_bounds__(256) void score_key_norms(const void* __restrict__ ik, int64_t T, int Di,
                                                       float* __restrict__ knorm2, uint32_t* __restrict__ amb,
                                                       int64_t amb_words) {
  const int64_t j = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (j < amb_words) amb[j] = 0u;
  if (j < T) knorm2[j] = signed_norm2<DT>(ik, j * Di, Di);
}

__global__ __launch_bounds__(256) void score_small_block_norms(const float* __restrict__ knorm2,
                                                               const int32_t* __restrict__ cu, int nseq, int64_t T,
                                                               int B, float* __restrict__ bnorm) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (t >= T) return;
  const int s = find_seq(cu, nseq, t);
  const int64_t start = cu[s], end = cu[s + 1];
  if ((t - start) % B != 0) return;
  const int64_t e = t + B < end ? t + B : end;
  float m = 0.f;
  bool safe = true;
  for (int64_t j = t; j < e; ++j) {
    const float v = knorm2[j];
    m = fmaxf(m, fabsf(v));
    safe = safe && v >= 0.f;
  }
  const float r = sqrtf(m);
  bnorm[t] = safe ? r : -r;
}

// Two workgroups per CU; one for the widest partial-width variant (index dim 72..120),
// whose register staging of the next block does not fit beside two.
template <int DT, int NK, bool FULLD, int SHORTEST>
__global__ __launch_bounds__(kThreads, NK == 4 && !FULLD ? 1 : 2) void score_fwd_mfma_kernel(const uint16_t* __restrict__ iq,
                                                                     const uint16_t* __restrict__ ik,
                                                                     const int32_t* __restrict__ cu, int nseq,
                                                                     int64_t rows, int G, int Di, int NB, int B,
                                                                     double scale, const float* __restrict__ bnorm,
                                                                     uint32_t* __restrict__ amb, int64_t rows_pad,
                                                                     float* __restrict__ scores,
                                                                     int32_t* __restrict__ tie) {
  constexpr int DP = 32 * NK;
  constexpr int CPK = DP / 8;                 // 16-byte chunks per key row
  constexpr int KCH = 128 * CPK / kThreads;   // chunks per thread per key block
  constexpr int HF = DP / 2;                  // max dims of a query half (Di / 2 <= DP / 2)
  __shared__ ScoreSmem<NK> sm;
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, q4 = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform (scalar) index
  const int64_t r0 = static_cast<int64_t>(gridDim.x - 1 - blockIdx.x) * kTileRows;  // heaviest tiles first
  const int nr = static_cast<int>(rows - r0 < kTileRows ? rows - r0 : kTileRows);
  const bool neg = scale < 0.0;
  const float fscale = static_cast<float>(fabs(scale));  // the reference's FP32 |scale|
  const uint32_t flip = neg ? 0x80008000u : 0u;
  constexpr float cerr = logit_error<DT, DP>();
  // exact_dot's split point (Di % 8 == 0, so h % 4 == 0); compile-time for Di == DP
  const int h = FULLD ? DP / 2 : Di / 2;

  // ---- this wave's rows: MFMA B fragments (rows 16 rt + c) ...
  const int wr0 = 32 * wid;  // first tile row of the wave
  bf16x8 qf[2][NK];
  int64_t mtok[2];
  bool min_tile[2];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const int rr = wr0 + 16 * rt + c;
    min_tile[rt] = rr < nr;
    mtok[rt] = min_tile[rt] ? (r0 + rr) / G : -1;
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) {
      const int d0 = 32 * kk + 8 * q4;
      uint4 w = make_uint4(0u, 0u, 0u, 0u);
      if (min_tile[rt] && d0 < Di) w = *reinterpret_cast<const uint4*>(iq + (r0 + rr) * Di + d0);
      w.x ^= flip;
      w.y ^= flip;
      w.z ^= flip;
      w.w ^= flip;
      qf[rt][kk] = __builtin_bit_cast(bf16x8, w);
    }
  }
  // ... and the exact-dot layout: lane (pr = lane & 31, hf = lane >> 5) keeps half hf
  // (dims [hf h, hf h + h)) of row wr0 + pr, sign-flipped, packed two per word.
  const int pr = lane & 31, hf = lane >> 5;
  const int prow = wr0 + pr;
  const bool pin = prow < nr;
  uint32_t qh[HF / 2];
  float pn2 = 0.f;
  bool psafe = true;
#pragma unroll
  for (int w4 = 0; w4 < HF / 4; ++w4) {  // 8-byte loads: 4 dims each
    uint2 x = make_uint2(0u, 0u);
    if (pin && 4 * w4 < h) x = *reinterpret_cast<const uint2*>(iq + (r0 + prow) * Di + hf * h + 4 * w4);
    x.x ^= flip;
    x.y ^= flip;
    qh[2 * w4] = x.x;
    qh[2 * w4 + 1] = x.y;
    pn2 = fmaf(lo16_f32<DT>(x.x), lo16_f32<DT>(x.x), pn2);
    pn2 = fmaf(hi16_f32<DT>(x.x), hi16_f32<DT>(x.x), pn2);
    pn2 = fmaf(lo16_f32<DT>(x.y), lo16_f32<DT>(x.y), pn2);
    pn2 = fmaf(hi16_f32<DT>(x.y), hi16_f32<DT>(x.y), pn2);
    psafe = psafe && word_safe<DT>(x.x) && word_safe<DT>(x.y);
  }
  pn2 += __shfl_xor(pn2, 32, kWave);
  psafe = psafe && __shfl_xor(static_cast<int>(psafe), 32, kWave) != 0;  // both halves of the row
  const float pnorm = sqrtf(pn2) * 1.0001f;  // ||q|| of row prow, rounded up
  float mnorm[2];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) mnorm[rt] = __shfl(pnorm, 16 * rt + c, kWave);
  bool msafe[2];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) msafe[rt] = __shfl(static_cast<int>(psafe), 16 * rt + c, kWave) != 0;
  const int64_t ptok = pin ? (r0 + prow) / G : -1;

  // ---- key block staging
  uint4 kreg[FULLD ? 1 : KCH];  // register staging of partial-width blocks
  // Full width: wave wid's instruction i fills physical chunks p = (wid KCH + i) 64 + lane
  // of the buffer (1 KiB per instruction), holding row p / CPK, logical chunk
  // (p % CPK) ^ swz(row). Rows advance by 16 every KCH / 2 instructions and the swizzle
  // repeats every 16 rows, so the offsets of the first half serve the second.
  constexpr int SH = NK == 4 ? 0 : (NK == 2 ? 1 : 2);
  constexpr int NP = FULLD ? KCH / 2 : 1;
  // element offset of instruction i's chunk within a complete block (block-invariant)
  auto chunk_off = [&](int i) {
    const int p = (wid * KCH + i % NP) * 64 + lane;
    const int row = p / CPK, pc = p % CPK;
    return static_cast<uint32_t>(row * DP + 8 * (pc ^ ((row >> SH) & (CPK - 1))) + (i < NP ? 0 : 16 * DP));
  };
  auto fetch = [&](const BlockCursor& bc, const uint16_t* gsrc, uint16_t* into) {
    if (bc.s >= nseq) return;
    const int64_t kb = cu[bc.s] + static_cast<int64_t>(bc.b) * B;
    const int64_t end = cu[bc.s + 1];
    const int nk = static_cast<int>(end - kb < B ? end - kb : B);
    if constexpr (FULLD) {
      char* dst = reinterpret_cast<char*>(into) + wid * KCH * 1024;
      if (nk == 128) {  // a complete block: scalar base plus the precomputed offsets
        const uint16_t* src = gsrc + kb * DP;
#pragma unroll
        for (int i = 0; i < KCH; ++i)
          __builtin_amdgcn_global_load_lds(src + static_cast<int>(chunk_off(i)),
                                           (__attribute__((address_space(3))) void*)(dst + i * 1024), 16, 0, 0);
      } else {  // rows past the block's end repeat its last key (masked later)
#pragma unroll
        for (int i = 0; i < KCH; ++i) {
          const int p = (wid * KCH + i) * 64 + lane;
          const int row = p / CPK, pc = p % CPK;
          const int lc = pc ^ ((row >> SH) & (CPK - 1));
          const int rowc = row < nk ? row : nk - 1;
          __builtin_amdgcn_global_load_lds(gsrc + (kb + rowc) * Di + 8 * lc,
                                           (__attribute__((address_space(3))) void*)(dst + i * 1024), 16, 0, 0);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < KCH; ++i) {
        const int e = tid + kThreads * i;
        const int kl = e / CPK, d0 = 8 * (e % CPK);
        kreg[i] = (kl < nk && d0 < Di) ? *reinterpret_cast<const uint4*>(gsrc + (kb + kl) * Di + d0)
                                       : make_uint4(0u, 0u, 0u, 0u);
      }
    }
  };
  auto commit = [&](int into) {
    if constexpr (!FULLD) {
#pragma unroll
      for (int i = 0; i < KCH; ++i) {
        const int e = tid + kThreads * i;
        const int kl = e / CPK, d0 = 8 * (e % CPK);
        *reinterpret_cast<uint4*>(sm.k[into] + key_off<NK, FULLD>(kl, d0)) = kreg[i];
      }
    }
  };
  // the block's largest key norm, negated when a key of the block is not safe
  auto block_norm = [&](const BlockCursor& bc) {
    return bc.s < nseq ? bnorm[cu[bc.s] + static_cast<int64_t>(bc.b) * B] : 0.f;
  };

  int todo;
  BlockCursor cur = tile_share(cu, nseq, r0, nr, G, B, SHORTEST, blockIdx.y, gridDim.y, todo);
  const float cn = block_norm(cur);
  fetch(cur, ik, sm.k[0]);
  commit(0);
  __builtin_amdgcn_s_waitcnt(0);  // this thread's direct-to-LDS loads have landed
  __syncthreads();
  float kmax = fabsf(cn);
  bool bsafe = !__builtin_signbit(cn);  // -0 marks an unsafe block too
  int buf = 0;
  while (cur.s < nseq) {
    BlockCursor nxt = next_block(cu, nseq, cur, r0, nr, G, B, SHORTEST);
    if (--todo <= 0) nxt.s = nseq;
    const float nn = block_norm(nxt);
    // The next block's fetch and this block's LDS reads go through the restrict-qualified
    // pointers of one inlined call, so the compiler's wait insertion can tell the fetch's
    // LDS writes (buffer buf ^ 1) from the reads (buffer buf): without that it waits for
    // the whole fetch before the first read, and the fetch would not overlap the block.
    [&](const uint16_t* __restrict__ ksrc, const uint16_t* __restrict__ kt_base, uint16_t* __restrict__ knext) {
    fetch(nxt, ksrc, knext);  // in flight while this block is evaluated (that buffer's readers passed the last barrier)

    const int64_t start = cu[cur.s], end = cu[cur.s + 1];
    const int64_t kb = start + static_cast<int64_t>(cur.b) * B;
    const int nk = static_cast<int>(end - kb < B ? end - kb : B);
    // visible keys of the lane's MFMA rows (0: row not in this sequence or block in its future)
    int lim[2];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      const int64_t t = mtok[rt];
      const int64_t v = (t >= start && t < end) ? t - kb + 1 : 0;
      lim[rt] = v <= 0 ? 0 : (v < nk ? static_cast<int>(v) : nk);
    }
    const bool wave_on = __ballot(lim[0] > 0 || lim[1] > 0) != 0;  // wave-uniform
    // approximate logits, 16 keys at a time, key position packed into their low bits,
    // folded into a per-row running top 2
    float m1[2] = {kMaskedLogit, kMaskedLogit}, m2[2] = {kMaskedLogit, kMaskedLogit};
    float pinf = __builtin_inff();
    asm volatile("" : "+v"(pinf));
    auto scan = [&](auto masked) {
#pragma unroll
      for (int kt = 0; kt < 8; ++kt) {
        bf16x8 kf[NK];
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) kf[kk] = load_frag(kt_base + key_off<NK, FULLD>(16 * kt + c, 32 * kk + 8 * q4));
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
          f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int kk = 0; kk < NK; ++kk) a = mfma_t<DT>(kf[kk], qf[rt][kk], a);
#pragma unroll
          for (int i = 0; i < 4; i += 2) {
            float x = a[i], y = a[i + 1];
            if constexpr (decltype(masked)::value) {
              x = 16 * kt + 4 * q4 + i < lim[rt] ? x : kMaskedLogit;
              y = 16 * kt + 4 * q4 + i + 1 < lim[rt] ? y : kMaskedLogit;
            }
            fold_pair(x, y, 4 * kt + i, pinf, m1[rt], m2[rt]);
          }
        }
      }
    };
    if (wave_on) {
      if (__ballot(lim[0] < 128 || lim[1] < 128) == 0)  // no key masked in the wave
        scan(std::false_type{});
      else
        scan(std::true_type{});
    }
    if (wave_on) {
      // merge the four key quarters of each row; the winner is certified unique iff no
      // other key comes within the bound of the maximum
      int widx[2], wcnt[2];
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        const RowTop top = merge_quarters(m1[rt], m2[rt], q4);
        widx[rt] = top.key;
        const float bound = 2.f * cerr * mnorm[rt] * kmax + 0x1p-15f * fmaxf(fabsf(top.a1), fabsf(top.a2)) + 0x1p-126f;
        // 2: at least two candidates, or products not certainly exact in fp32
        wcnt[rt] = (top.a2 >= top.a1 - bound || !(bsafe && msafe[rt])) ? 2 : 1;
      }
      // lane pair (pr, hf): row wr0 + pr = 16 rt + c with rt = pr >> 4 -- this lane's c matches
      const int prt = pr >> 4;
      const int myidx = prt ? widx[1] : widx[0];
      const int mycnt = prt ? wcnt[1] : wcnt[0];
      const int mylim = prt ? lim[1] : lim[0];
      const bool row_ok = pin && mylim > 0;
      // unique winner: its exact dot, half per lane, in exact_dot's order (exact fp32
      // products of safe bf16 values added in FP64)
      double half = 0.0;
      if (row_ok && mycnt == 1) {
#pragma unroll
        for (int j8 = 0; j8 < HF / 8; ++j8) {  // 8 dims per 16-byte read
          if (FULLD || 8 * j8 < h) {
            const uint16_t* kp = kt_base + key_off<NK, FULLD>(myidx, hf * h + 8 * j8);
            uint32_t kx[4];
            if (FULLD) {
              const uint4 kw = *reinterpret_cast<const uint4*>(kp);
              kx[0] = kw.x, kx[1] = kw.y, kx[2] = kw.z, kx[3] = kw.w;
            } else if (8 * j8 + 8 <= h) {  // the second half may start 8 bytes into a 16-byte unit (h % 8 == 4)
              const uint2 ka = *reinterpret_cast<const uint2*>(kp), kb = *reinterpret_cast<const uint2*>(kp + 4);
              kx[0] = ka.x, kx[1] = ka.y, kx[2] = kb.x, kx[3] = kb.y;
            } else {  // h % 8 == 4: the last four dims of the half
              const uint2 kw = *reinterpret_cast<const uint2*>(kp);
              kx[0] = kw.x, kx[1] = kw.y, kx[2] = kx[3] = 0u;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              if (FULLD || 8 * j8 + 2 * u < h) {
                half += static_cast<double>(prod_lo<DT>(qh[4 * j8 + u], kx[u]));
                half += static_cast<double>(prod_hi<DT>(qh[4 * j8 + u], kx[u]));
              }
            }
          }
        }
      }
      const double dot = add_halves(half);  // lanes pr and pr + 32
      if (row_ok && mycnt == 1 && hf == 0) {
        const int64_t out = (r0 + prow) * NB + cur.b;
        scores[out] = public_score(dot, fscale);
        if (tie) tie[out] = myidx + 1;
      }
      // ambiguous rows: marked for score_fwd_resolve
      if (row_ok && mycnt != 1 && hf == 0) {
        const int64_t bit = static_cast<int64_t>(cur.b) * rows_pad + r0 + prow;
        atomicOr(amb + (bit >> 5), 1u << (bit & 31));
      }
    }
    }(ik, sm.k[buf], sm.k[buf ^ 1]);
    if (nxt.s < nseq) commit(buf ^ 1);  // that buffer's readers finished before the last barrier
    __builtin_amdgcn_s_waitcnt(0);       // the next block's direct-to-LDS loads have landed
    __syncthreads();  // this block's readers are done; the next block is visible
    kmax = fabsf(nn);
    bsafe = !__builtin_signbit(nn);
    buf ^= 1;
    cur = nxt;
  }

  fill_future(cu, nseq, r0 + wr0, nr - wr0, G, NB, B, scores, tie);
}

// The fp32 form: every element enters the MFMA logits as two bf16 terms (three products),
// split from the fp32 key block in LDS as the fragments are read; the certified winner's
// exact dot reads its fp32 row from the same block. One LDS buffer (64 KiB at 128 dims), so
// that two workgroups share a CU and one's fetch runs beside the other's products.
template <int NK>
struct KeyRowsF32 {
  static constexpr int CPK = 8 * NK;  // 16-byte chunks per key row
  // chunk of dims [4p, 4p + 4) of key `row`: swizzled so that the 16 rows of a fragment read
  // (one chunk of each) cover all 64 banks
  static __device__ __forceinline__ int at(int row, int p) {
    return row * CPK + (p ^ (NK == 1 ? (row >> 1) & 7 : row & 15));
  }
};

template <int NK, int SHORTEST>
__global__ __launch_bounds__(kThreads, 2) void score_fwd_f32_kernel(const float* __restrict__ iq,
                                                                    const float* __restrict__ ik,
                                                                    const int32_t* __restrict__ cu, int nseq,
                                                                    int64_t rows, int G, int Di, int NB, int B,
                                                                    double scale, const float* __restrict__ bnorm,
                                                                    uint32_t* __restrict__ amb, int64_t rows_pad,
                                                                    float* __restrict__ scores,
                                                                    int32_t* __restrict__ tie) {
  using Rows = KeyRowsF32<NK>;
  constexpr int DP = 32 * NK, CPK = Rows::CPK, KCH = 128 * CPK / kThreads, HF = DP / 2;
  __shared__ alignas(16) uint4 keys[128 * CPK];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, q4 = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t r0 = static_cast<int64_t>(gridDim.x - 1 - blockIdx.x) * kTileRows;  // heaviest tiles first
  const int nr = static_cast<int>(rows - r0 < kTileRows ? rows - r0 : kTileRows);
  const float fscale = static_cast<float>(fabs(scale));
  const uint32_t flip = scale < 0.0 ? 0x80000000u : 0u;
  constexpr float cerr = logit_error<kF32, DP>();
  const int h = Di / 2;  // exact_dot's split point, a multiple of 4

  // ---- this wave's rows: MFMA operands (rows 16 rt + c), zero past Di
  const int wr0 = 32 * wid;
  SplitFrag qf[2][NK];
  int64_t mtok[2];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    const int rr = wr0 + 16 * rt + c;
    mtok[rt] = rr < nr ? (r0 + rr) / G : -1;
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) {
      const int d0 = 32 * kk + 8 * q4;
      Words8<kF32> w = {};
      if (rr < nr && d0 < Di) w = load_words<kF32>(iq, (r0 + rr) * Di + d0);
#pragma unroll
      for (int u = 0; u < 8; ++u) w.w[u] ^= flip;
      qf[rt][kk] = split_frag(w.w);
    }
  }
  // ... and the exact-dot layout: lane (pr = lane & 31, hf = lane >> 5) keeps half hf of row
  // wr0 + pr
  const int pr = lane & 31, hf = lane >> 5;
  const int prow = wr0 + pr;
  const bool pin = prow < nr;
  float qh[HF];
  float pn2 = 0.f;
  bool psafe = true;
#pragma unroll
  for (int j = 0; j < HF / 4; ++j) {
    uint4 x = make_uint4(0u, 0u, 0u, 0u);
    if (pin && 4 * j < h) x = *reinterpret_cast<const uint4*>(iq + (r0 + prow) * Di + hf * h + 4 * j);
    const uint32_t xs[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      add_square<kF32>(xs[u], pn2, psafe);
      qh[4 * j + u] = __uint_as_float(xs[u] ^ flip);
    }
  }
  pn2 += __shfl_xor(pn2, 32, kWave);
  psafe = psafe && __shfl_xor(static_cast<int>(psafe), 32, kWave) != 0;
  const float pnorm = sqrtf(pn2) * 1.0001f;  // ||q|| of row prow, rounded up
  float mnorm[2];
  bool msafe[2];
#pragma unroll
  for (int rt = 0; rt < 2; ++rt) {
    mnorm[rt] = __shfl(pnorm, 16 * rt + c, kWave);
    msafe[rt] = __shfl(static_cast<int>(psafe), 16 * rt + c, kWave) != 0;
  }

  int todo;
  BlockCursor cur = tile_share(cu, nseq, r0, nr, G, B, SHORTEST, blockIdx.y, gridDim.y, todo);
  float pinf = __builtin_inff();
  asm volatile("" : "+v"(pinf));
  while (cur.s < nseq) {
    const int64_t start = cu[cur.s], end = cu[cur.s + 1];
    const int64_t kb = start + static_cast<int64_t>(cur.b) * B;
    const int nk = static_cast<int>(end - kb < B ? end - kb : B);
    // wave wid's instruction i fills physical chunks (wid KCH + i) 64 + lane; rows past the
    // block's end repeat its last key (masked later), chunks past Di the row's last one (their
    // query operands are zero; a block with a key that is not finite is not certified)
    __syncthreads();  // the previous block's readers are done
#pragma unroll
    for (int i = 0; i < KCH; ++i) {
      const int p = (wid * KCH + i) * 64 + lane;
      const int row = p / CPK, lc = Rows::at(row, p % CPK) - row * CPK;
      const int rowc = row < nk ? row : nk - 1, lcc = 4 * lc < Di ? lc : Di / 4 - 1;
      __builtin_amdgcn_global_load_lds(
          ik + (kb + rowc) * Di + 4 * lcc,
          (__attribute__((address_space(3))) void*)(reinterpret_cast<char*>(keys) + (wid * KCH + i) * 1024), 16, 0, 0);
    }
    const float bn = bnorm[kb];
    const float kmax = fabsf(bn);
    const bool bsafe = !__builtin_signbit(bn);
    int lim[2];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      const int64_t t = mtok[rt];
      const int64_t v = (t >= start && t < end) ? t - kb + 1 : 0;
      lim[rt] = v <= 0 ? 0 : (v < nk ? static_cast<int>(v) : nk);
    }
    const bool wave_on = __ballot(lim[0] > 0 || lim[1] > 0) != 0;  // wave-uniform
    __builtin_amdgcn_s_waitcnt(0);  // this thread's direct-to-LDS loads have landed
    __syncthreads();
    if (wave_on) {
      float m1[2] = {kMaskedLogit, kMaskedLogit}, m2[2] = {kMaskedLogit, kMaskedLogit};
      auto scan = [&](auto masked) {
#pragma unroll
        for (int kt = 0; kt < 8; ++kt) {
          f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
          for (int kk = 0; kk < NK; ++kk) {
            const uint4 a = keys[Rows::at(16 * kt + c, 8 * kk + 2 * q4)];
            const uint4 b = keys[Rows::at(16 * kt + c, 8 * kk + 2 * q4 + 1)];
            const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
            const SplitFrag kf = split_frag(w);
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) acc[rt] = mfma_split(kf, qf[rt][kk], acc[rt]);
          }
#pragma unroll
          for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
              float x = acc[rt][i], y = acc[rt][i + 1];
              if constexpr (decltype(masked)::value) {
                x = 16 * kt + 4 * q4 + i < lim[rt] ? x : kMaskedLogit;
                y = 16 * kt + 4 * q4 + i + 1 < lim[rt] ? y : kMaskedLogit;
              }
              fold_pair(x, y, 4 * kt + i, pinf, m1[rt], m2[rt]);
            }
        }
      };
      if (__ballot(lim[0] < 128 || lim[1] < 128) == 0)  // no key masked in the wave
        scan(std::false_type{});
      else
        scan(std::true_type{});
      int widx[2];
      bool sure[2];  // exactly one candidate
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        const RowTop top = merge_quarters(m1[rt], m2[rt], q4);
        widx[rt] = top.key;
        const float bound =
            2.f * cerr * mnorm[rt] * kmax + 0x1p-15f * fmaxf(fabsf(top.a1), fabsf(top.a2)) + 0x1p-126f;
        sure[rt] = top.a2 < top.a1 - bound && bsafe && msafe[rt];
      }
      // lane pair (pr, hf): row wr0 + pr = 16 rt + c with rt = pr >> 4 -- this lane's c matches
      const int prt = pr >> 4;
      const int myidx = prt ? widx[1] : widx[0];
      const bool row_ok = pin && (prt ? lim[1] : lim[0]) > 0;
      const bool mysure = row_ok && (prt ? sure[1] : sure[0]);
      double half = 0.0;
      if (mysure) {
#pragma unroll
        for (int j = 0; j < HF / 4; ++j) {
          if (4 * j < h) {
            const uint4 kw = keys[Rows::at(myidx, hf * (h / 4) + j)];
            const uint32_t ks[4] = {kw.x, kw.y, kw.z, kw.w};
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              float qv = qh[4 * j + u];
              asm volatile("" : "+v"(qv));  // converted here: hoisted out of the block loop, 64 doubles spill
              half = fma(static_cast<double>(qv), static_cast<double>(__uint_as_float(ks[u])), half);
            }
          }
        }
      }
      const double dot = add_halves(half);
      if (mysure && hf == 0) {
        const int64_t out = (r0 + prow) * NB + cur.b;
        scores[out] = public_score(dot, fscale);
        if (tie) tie[out] = myidx + 1;
      }
      if (row_ok && !mysure && hf == 0) {  // marked for score_fwd_resolve
        const int64_t bit = static_cast<int64_t>(cur.b) * rows_pad + r0 + prow;
        atomicOr(amb + (bit >> 5), 1u << (bit & 31));
      }
    }
    cur = next_block(cu, nseq, cur, r0, nr, G, B, SHORTEST);
    if (--todo <= 0) cur.s = nseq;
  }
  fill_future(cu, nseq, r0 + wr0, nr - wr0, G, NB, B, scores, tie);
}
// exact_dot (two sequential FMA chains over the halves of the index dim) with 4-element loads:
// n % 8 == 0, rows aligned for them.
template <int DT>
__device__ __forceinline__ double exact_dot_wide(const void* __restrict__ a, int64_t ia, const void* __restrict__ b,
                                                 int64_t ib, int n) {
  const int h = n / 2;
  auto load4 = [](const void* base, int64_t i, float (&x)[4]) {
    if constexpr (DT == kF32) {
      const float4 w = *reinterpret_cast<const float4*>(static_cast<const float*>(base) + i);
      x[0] = w.x, x[1] = w.y, x[2] = w.z, x[3] = w.w;
    } else {
      const uint2 w = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(base) + i);
      x[0] = lo16_f32<DT>(w.x), x[1] = hi16_f32<DT>(w.x), x[2] = lo16_f32<DT>(w.y), x[3] = hi16_f32<DT>(w.y);
    }
  };
  double s0 = 0.0, s1 = 0.0;
  for (int d = 0; d < h; d += 4) {
    float a0[4], b0[4], a1[4], b1[4];
    load4(a, ia + d, a0);
    load4(b, ib + d, b0);
    load4(a, ia + h + d, a1);
    load4(b, ib + h + d, b1);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      s0 = fma(static_cast<double>(a0[u]), static_cast<double>(b0[u]), s0);
      s1 = fma(static_cast<double>(a1[u]), static_cast<double>(b1[u]), s1);
    }
  }
  return s0 + s1;
}

// Rows of sequences of up to kShortSeq tokens, 16 lanes each, one key per lane: every visible key's
// exact dot, the maximum, its count and first key (a NaN dot is no candidate). A sequence is one
// step of the MFMA kernels' tiles, of 128 keys and 64 or 128 rows, whatever its length: packs of
// short ones took up to 64 such steps per tile, and the norms of 64 blocks one after the other.
// Bound by the FP64 chains and their conversions (a wave's four rows take as long for one key
// as for 16: 75 to 133 us for 131 072 rows). us, MFMA steps / here, 2 groups of 128 dims: fp16,
// 8192 sequences of one token 356 / 43, 1024 of 8 69 / 31, 512 of 16 47 / 35, 65 536 of one 768 / 139,
// 8192 of 8 154 / 134, 4096 of 16 103 / 175; fp32, 8192 of one 762 / 41, 682 of 12 124 / 32, 4096 of 16 255 /
// 170. (For many fp16 or bf16 sequences of 9 to 16 the steps are the faster: not taken apart.)
template <int DT>
__global__ __launch_bounds__(256) void score_fwd_short(const void* __restrict__ iq, const void* __restrict__ ik,
                                                       const int32_t* __restrict__ cu, int nseq, int64_t rows, int G,
                                                       int Di, int NB, double scale, float* __restrict__ scores,
                                                       int32_t* __restrict__ tie) {
  const int64_t row = static_cast<int64_t>(blockIdx.x) * 16 + (threadIdx.x >> 4);
  if (row >= rows) return;
  const int sub = threadIdx.x & 15;
  const int64_t t = row / G;
  const int s = find_seq(cu, nseq, t);
  const int64_t start = cu[s];
  if (cu[s + 1] - start > kShortSeq) return;  // all 16 lanes
  double best = -__builtin_inf();
  bool seen = start + sub <= t;
  if (seen) {
    const double v = directed(exact_dot_wide<DT>(iq, row * Di, ik, (start + sub) * Di, Di), scale);
    seen = v == v;
    if (seen) best = v;
  }
  const double own = best;
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) best = fmax(best, __shfl_xor(best, o, 16));
  const uint32_t at = static_cast<uint32_t>(__ballot(seen && own == best) >> (threadIdx.x & 48)) & 0xffffu;
  if (sub == 0) {
    const int count = __popc(at);
    scores[row * NB] = public_score(best, static_cast<float>(fabs(scale)));
    if (tie) tie[row * NB] = count == 1 ? __builtin_ctz(at) + 1 : -count;
  }
}

// Monotone map of a double that is not NaN onto uint64 (+0 and -0 collapse; never 0), and back.
__device__ __forceinline__ uint64_t ordered_f64(double x) {
  const uint64_t u = static_cast<uint64_t>(__double_as_longlong(x + 0.0));
  return (u >> 63) ? ~u : (u | (uint64_t(1) << 63));
}
__device__ __forceinline__ double from_ordered_f64(uint64_t k) {
  return __longlong_as_double(static_cast<long long>((k >> 63) ? (k & ~(uint64_t(1) << 63)) : ~k));
}

// The ambiguous (row, block) pairs the main pass marked, settled exactly. For a block and
// kResolveRows rows one wave, or where that gives the chip few (calls of few blocks: short
// sequences) up to kResolveShares, lists the marked rows in order and takes its share of them, up
// to 16 (of one sequence) at a time: about 4 us each, one after the other (341 sequences of 24
// tokens, 2 groups, fp32: 4 waves 165 us, the selection 294, now 91; shared beyond 512 waves the groups
// are smaller and there are more of them: 64 blocks, 8192 tokens, 4 groups, fp16, 2048 waves: 131 for 127). Their MFMA logits against the block are formed again, operands
// straight from memory; the keys within the error bound of a row's maximum (all visible keys
// where the row or the block is not safe) are its candidates, two or three of 128 for most
// rows. The candidates of the 16 rows are spread over the lanes, one exact_dot each; the
// maximum, its count and the first winner come from integer LDS atomics, so the result does
// not depend on their order. (Re-evaluating every key of the block in FP64 took 133 us at
// 32 768 tokens x 4 groups in bf16, this pass 54 us.)
constexpr int kResolveGroup = 16, kResolveShares = 64, kResolveWaves = 512;
template <int DT>
__global__ __launch_bounds__(64) void score_fwd_resolve(const void* __restrict__ iq, const void* __restrict__ ik,
                                                        const int32_t* __restrict__ cu, int nseq, int64_t rows_pad,
                                                        int G, int Di, int NB, int B, double scale,
                                                        const float* __restrict__ bnorm,
                                                        const uint32_t* __restrict__ amb, float* __restrict__ scores,
                                                        int32_t* __restrict__ tie) {
  constexpr int NK = 4;  // Di <= 128
  __shared__ uint16_t list[kResolveRows];
  __shared__ uint16_t cand[kResolveGroup * 128];  // row of the group << 7 | key
  __shared__ uint64_t best[kResolveGroup];
  __shared__ int count[kResolveGroup], first[kResolveGroup];
  const int lane = threadIdx.x, c = lane & 15, q4 = lane >> 4;
  // blockIdx.x: chunk * NB + block; blockIdx.y: share
  const int b = static_cast<int>(blockIdx.x % static_cast<uint32_t>(NB));
  const int64_t c0 = static_cast<int64_t>(blockIdx.x / static_cast<uint32_t>(NB)) * kResolveRows;
  static_assert(kResolveRows == 64 * 64, "one 64-bit bitmap word per lane");
  const uint32_t* words = amb + (static_cast<int64_t>(b) * rows_pad + c0) / 32 + 2 * lane;
  uint64_t mine = (static_cast<uint64_t>(words[1]) << 32) | words[0];
  auto scan = [&](int x) {  // inclusive prefix over the lanes
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(x, o, kWave);
      if (lane >= o) x += y;
    }
    return x;
  };
  {
    const int own = __popcll(mine), incl = scan(own);
    int o = incl - own;
    for (; mine; mine &= mine - 1) list[o++] = static_cast<uint16_t>(64 * lane + __builtin_ctzll(mine));
    count[0] = __shfl(incl, 63, kWave);
  }
  __syncthreads();
  // (the lists are in order, so a share's groups are those of its rows: each row once)
  const int marked = __builtin_amdgcn_readfirstlane(count[0]), shares = gridDim.y;
  const int n = marked * (static_cast<int>(blockIdx.y) + 1) / shares;
  const bool neg = scale < 0.0;
  for (int i = marked * static_cast<int>(blockIdx.y) / shares; i < n;) {
    const int64_t row0 = c0 + __builtin_amdgcn_readfirstlane(list[i]);
    const int s = find_seq(cu, nseq, row0 / G);
    const int64_t start = cu[s], end = cu[s + 1];
    const int64_t end_row = end * G - c0;  // chunk-relative end of the sequence's rows
    const int m = __popcll(__ballot(lane < kResolveGroup && i + lane < n && list[min(i + lane, n - 1)] < end_row));
    const int64_t k0 = start + static_cast<int64_t>(b) * B;
    const int nk = static_cast<int>((k0 + B < end ? k0 + B : end) - k0);  // >= 1: a listed row sees block b
    const int64_t row = c0 + list[c < m ? i + c : i];
    const int64_t vis = row / G + 1 - k0;
    const int lim = c < m ? static_cast<int>(vis < nk ? vis : nk) : 0;
    // ---- approximate logits S[row c][key 16 kt + 4 q4 + i]
    float n2 = 0.f;
    bool safe = true;
    f32x4 acc[8];
#pragma unroll
    for (int kt = 0; kt < 8; ++kt) acc[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < NK; ++kk) {
      if (32 * kk < Di) {
        const int d0 = 32 * kk + 8 * q4;
        const bool in = d0 < Di;
        Words8<DT> qw = load_words<DT>(iq, row * Di + (in ? d0 : 0));
#pragma unroll
        for (int u = 0; u < Words8<DT>::N; ++u) {
          qw.w[u] = in ? qw.w[u] : 0u;
          add_square<DT>(qw.w[u], n2, safe);
          qw.w[u] ^= neg ? (DT == kF32 ? 0x80000000u : 0x80008000u) : 0u;
        }
        Words8<DT> kw[8];
#pragma unroll
        for (int kt = 0; kt < 8; ++kt) {
          const int key = 16 * kt + c < nk ? 16 * kt + c : nk - 1;
          kw[kt] = load_words<DT>(ik, (k0 + key) * Di + (in ? d0 : 0));
        }
        if constexpr (DT == kF32) {
          const SplitFrag qf = split_frag(qw.w);
#pragma unroll
          for (int kt = 0; kt < 8; ++kt) acc[kt] = mfma_split(split_frag(kw[kt].w), qf, acc[kt]);
        } else {
          const bf16x8 qf = __builtin_bit_cast(bf16x8, make_uint4(qw.w[0], qw.w[1], qw.w[2], qw.w[3]));
#pragma unroll
          for (int kt = 0; kt < 8; ++kt)
            acc[kt] = mfma_t<DT>(
                __builtin_bit_cast(bf16x8, make_uint4(kw[kt].w[0], kw[kt].w[1], kw[kt].w[2], kw[kt].w[3])), qf,
                acc[kt]);
        }
      }
    }
    // ---- candidates of each row
    float mx = -__builtin_inff();
#pragma unroll
    for (int kt = 0; kt < 8; ++kt)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (16 * kt + 4 * q4 + j < lim) mx = fmaxf(mx, acc[kt][j]);
#pragma unroll
    for (int o = 16; o <= 32; o <<= 1) {
      mx = fmaxf(mx, __shfl_xor(mx, o, kWave));
      n2 += __shfl_xor(n2, o, kWave);
      safe = __shfl_xor(static_cast<int>(safe), o, kWave) != 0 && safe;
    }
    const float bn = bnorm[k0];
    safe = safe && !__builtin_signbit(bn);
    const float bound = 2.f * logit_error<DT, 32 * NK>() * (sqrtf(n2) * 1.0001f) * fabsf(bn) +
                        0x1p-20f * fabsf(mx) + 0x1p-126f;
    uint32_t cm = 0u;
#pragma unroll
    for (int kt = 0; kt < 8; ++kt)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (16 * kt + 4 * q4 + j < lim && (!safe || !(acc[kt][j] < mx - bound))) cm |= 1u << (4 * kt + j);
    const int own = __popc(cm), incl = scan(own);
    const int total = __shfl(incl, 63, kWave);
    int o = incl - own;
    for (; cm; cm &= cm - 1) {
      const int p = __builtin_ctz(cm);
      cand[o++] = static_cast<uint16_t>(c << 7 | (16 * (p >> 2) + 4 * q4 + (p & 3)));
    }
    if (lane < kResolveGroup) {
      best[lane] = 0u;
      count[lane] = 0;
      first[lane] = 0x7fffffff;
    }
    __syncthreads();
    // ---- their exact dots (NaN dots are skipped; a row without any other visible dot keeps count 0)
    auto value = [&](int e) -> uint64_t {
      const int x = cand[e], key = x & 127;
      double v = exact_dot_wide<DT>(iq, (c0 + list[i + (x >> 7)]) * Di, ik, (k0 + key) * Di, Di);
      v = neg ? -v : v;
      return v == v ? ordered_f64(v) : 0u;
    };
    uint64_t v0 = 0u;
    for (int e = lane; e < total; e += kWave) {
      const uint64_t v = value(e);
      if (e == lane) v0 = v;
      if (v) atomicMax(reinterpret_cast<unsigned long long*>(&best[cand[e] >> 7]), static_cast<unsigned long long>(v));
    }
    __syncthreads();
    for (int e = lane; e < total; e += kWave) {
      const uint64_t v = e == lane ? v0 : value(e);
      const int g = cand[e] >> 7;
      if (v && v == best[g]) {
        atomicAdd(&count[g], 1);
        atomicMin(&first[g], cand[e] & 127);
      }
    }
    __syncthreads();
    if (lane < m) {
      const int k = count[lane];
      const int64_t out = row * NB + b;  // lane < m: row is row `lane` of the group
      scores[out] = public_score(k ? from_ordered_f64(best[lane]) : -__builtin_inf(), static_cast<float>(fabs(scale)));
      if (tie) tie[out] = k == 1 ? first[lane] + 1 : -k;
    }
    __syncthreads();  // the lists are rewritten by the next group
    i += m;
  }
}

bool score_mfma_supported(int Di, int B, double scale) {
  return scale != 0.0 && Di >= 8 && Di <= 128 && Di % 8 == 0 && B >= 1 && B <= 128;
}

int64_t score_fwd_mfma_workspace_bytes(int64_t total_tokens, int64_t rows, int64_t NB) {
  return ws_bitmap_offset(total_tokens) + 4 * bitmap_words(rows, NB);
}

// Workgroups per row tile, each taking an equal run of the tile's key blocks. A tile's work
// grows with its position in the sequence, so with one workgroup per tile the chip waits for
// the heaviest ones unless there are many tiles per CU. A part costs its rows' set-up:
// enough parts for 2048 workgroups while a part keeps about 16 blocks, and for 512 (two per
// CU) while it keeps 2. Measured, us per selection with 1 / 2 / 4 / 8 parts: 256 tiles of up
// to 64 blocks 243 / 179 / 154 / 162; with 1 / 2 / 4 parts: 1024 tiles of up to 256 blocks
// 1275 / 1216 / 1246, 512 tiles of up to 48 blocks (score forward and backward) 472 / 437 / 450.
static unsigned tile_parts(int64_t rows, int64_t NB) {
  const int64_t tiles = (rows + kTileRows - 1) / kTileRows;
  auto parts = [&](int64_t workgroups, int64_t blocks) {
    const int64_t p = (workgroups + tiles - 1) / tiles, most = NB / blocks;
    return p < most ? p : most;
  };
  const int64_t many = parts(2048, 16), fill = parts(512, 2);
  const int64_t p = many > fill ? many : fill;
  return static_cast<unsigned>(p < 1 ? 1 : p);
}

template <int DT>
static int launch(const void* iq, const void* ik, const int32_t* cu, int nseq, int64_t rows, int G, int Di, int NB,
                  int B, double scale, float* scores, int32_t* tie, void* ws, hipStream_t st) {
  const dim3 grid(grid_1d(rows, kTileRows), tile_parts(rows, NB)), block(kThreads);
  const int64_t T = rows / G;
  char* wsb = static_cast<char*>(ws);
  float* knorm2 = reinterpret_cast<float*>(wsb);
  float* bnorm = reinterpret_cast<float*>(wsb + ws_bnorm_offset(T));
  auto* amb = reinterpret_cast<uint32_t*>(wsb + ws_bitmap_offset(T));
  const int64_t words = bitmap_words(rows, NB);
  const int64_t rows_pad = rows_padded(rows);
  // Short sequences apart where they can be a large part of the pack (a mean length below 32; the
  // kernel's pass over all rows takes 4 to 6 us where there are none). They are one block each: B >= 64.
  const bool may_be_short = T < 32 * static_cast<int64_t>(nseq) && (nseq > 1 || T <= kShortSeq);
  const int shortest = B >= 64 && may_be_short && rows < (int64_t{1} << 28) ? kShortSeq : 0;
  if (shortest)
    hipLaunchKernelGGL(score_fwd_short<DT>, dim3(grid_1d(rows, 16)), dim3(256), 0, st, iq, ik, cu, nseq, rows, G, Di, NB,
                       scale, scores, tie);
  if (B >= 64 && T < (int64_t{1} << 30)) {  // (four threads per token: a launch holds fewer than 2^32)
    const unsigned ng = grid_1d(T, 64), wg = grid_1d(words, 256);
    hipLaunchKernelGGL(score_block_norms<DT>, dim3(ng > wg ? ng : wg), dim3(256), 0, st, ik, cu, nseq, T, Di, B, shortest, bnorm, amb, words);
  } else {
    hipLaunchKernelGGL(score_key_norms<DT>, dim3(grid_1d(T > words ? T : words, 256)), dim3(256), 0, st, ik, T, Di, knorm2, amb, words);
    hipLaunchKernelGGL(score_small_block_norms, dim3(grid_1d(T, 256)), dim3(256), 0, st, knorm2, cu, nseq, T, B, bnorm);
  }
  const int nk = Di <= 32 ? 1 : (Di <= 64 ? 2 : 4);
  if constexpr (DT == kF32) {
#define MSA_SCORE_F32(NKV) hipLaunchKernelGGL((shortest ? score_fwd_f32_kernel<NKV, kShortSeq> : score_fwd_f32_kernel<NKV, 0>), grid, block, 0, st, static_cast<const float*>(iq), static_cast<const float*>(ik), cu, nseq, rows, G, Di, NB, B, scale, bnorm, amb, rows_pad, scores, tie)
    if (nk == 1) MSA_SCORE_F32(1); else if (nk == 2) MSA_SCORE_F32(2); else MSA_SCORE_F32(4);
#undef MSA_SCORE_F32
  } else {
#define MSA_SCORE_MFMA(NKV, FD) hipLaunchKernelGGL((shortest ? score_fwd_mfma_kernel<DT, NKV, FD, kShortSeq> : score_fwd_mfma_kernel<DT, NKV, FD, 0>), grid, block, 0, st, static_cast<const uint16_t*>(iq), static_cast<const uint16_t*>(ik), cu, nseq, rows, G, Di, NB, B, scale, bnorm, amb, rows_pad, scores, tie)
    const bool fd = Di == 32 * nk;
    if (nk == 1) { if (fd) MSA_SCORE_MFMA(1, true); else MSA_SCORE_MFMA(1, false); }
    else if (nk == 2) { if (fd) MSA_SCORE_MFMA(2, true); else MSA_SCORE_MFMA(2, false); }
    else { if (fd) MSA_SCORE_MFMA(4, true); else MSA_SCORE_MFMA(4, false); }
#undef MSA_SCORE_MFMA
  }
  const int64_t chunks = rows_pad / kResolveRows;
  const int64_t most = std::min<int64_t>(kResolveShares, std::min<int64_t>(rows, kResolveRows) / 64);  // (of 64 rows)
  const int64_t shares = std::max<int64_t>(1, std::min(most, kResolveWaves / (NB * chunks)));
  hipLaunchKernelGGL(score_fwd_resolve<DT>, dim3(static_cast<unsigned>(NB * chunks), static_cast<unsigned>(shares)), dim3(64), 0,
                     st, iq, ik, cu, nseq, rows_pad, G, Di, NB, B, scale, bnorm, amb, scores, tie);
  return status_from(hipGetLastError());
}

int score_fwd_mfma_launch(int dt, const void* iq, const void* ik, const int32_t* cu, int nseq, int64_t rows, int G,
                          int Di, int NB, int B, double scale, float* scores, int32_t* tie, void* ws, hipStream_t st) {
  if (!ws) return kErrInvalidArgument;
  switch (dt) {
    case kF32: return launch<kF32>(iq, ik, cu, nseq, rows, G, Di, NB, B, scale, scores, tie, ws, st);
    case kF16: return launch<kF16>(iq, ik, cu, nseq, rows, G, Di, NB, B, scale, scores, tie, ws, st);
    default: return launch<kBF16>(iq, ik, cu, nseq, rows, G, Di, NB, B, scale, scores, tie, ws, st);
  }
}

}  // namespace msa
