// Causal top-k selection of one (token, group) row, by sixteen lanes (one DPP row)
// or by a whole wavefront, and the host launch that picks between them.
//
// Semantics follow triton/topk.py:31-46 (eager twin eager/ops.py:94-129): blocks
// b > qb(t) are masked to -inf, blocks in (qb-L, qb] are forced to +inf, the
// min(K, NB) largest are returned in descending order, -inf picks become -1, and
// the row is right-padded with -1 up to K slots. NaN scores rank above +inf (as in
// torch.topk). Ties (equal values, e.g. several +inf local blocks, or NaNs) are
// emitted in ascending block order.
#pragma once
#include "common.hpp"

namespace msa {

// Monotone map of float bits onto uint32 (+0 and -0 collapse to the same key). NaN of
// either sign ranks above +inf, as in torch.topk (the reference's selection,
// triton/topk.py:44-45); 0xfffffffe keeps the 64-bit key of block 0 below the scan's
// initial bound ~0.
__device__ __forceinline__ uint32_t ordered_key(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return 0xfffffffeu;
  if (u == 0x80000000u) u = 0u;
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

constexpr uint32_t kKeyNegInf = 0x007fffffu;  // ordered_key(-inf)
constexpr uint32_t kKeyPosInf = 0xff800000u;  // ordered_key(+inf)

// 64-bit max over the 16 lanes of a DPP row (every lane of the row receives it):
// quad butterflies, then half-row and row mirrors pair disjoint groups.
__device__ __forceinline__ uint64_t row16_max_u64(uint64_t v) {
#define MSA_DPP_MAX(CTRL)                                                                         \
  {                                                                                               \
    const uint32_t lo = static_cast<uint32_t>(v), hi = static_cast<uint32_t>(v >> 32);            \
    const uint32_t olo = __builtin_amdgcn_update_dpp(0u, lo, CTRL, 0xF, 0xF, false);              \
    const uint32_t ohi = __builtin_amdgcn_update_dpp(0u, hi, CTRL, 0xF, 0xF, false);              \
    const uint64_t o = (static_cast<uint64_t>(ohi) << 32) | olo;                                  \
    v = o > v ? o : v;                                                                            \
  }
  MSA_DPP_MAX(0xB1)   // quad_perm [1, 0, 3, 2]
  MSA_DPP_MAX(0x4E)   // quad_perm [2, 3, 0, 1]
  MSA_DPP_MAX(0x141)  // row_half_mirror
  MSA_DPP_MAX(0x140)  // row_mirror
#undef MSA_DPP_MAX
  return v;
}

// A lane's sorted cache of its N largest keys below a bound (0 = empty slot):
// c[0] > c[1] > ... > c[N - 1]. Keys are unique (the block id is in the low word).
template <int N>
struct TopN {
  uint64_t c[N];
  __device__ __forceinline__ void insert(uint64_t x) {
    // x enters at the bottom when it beats the smallest entry, then bubbles up
    if (x > c[N - 1]) c[N - 1] = x;
#pragma unroll
    for (int i = N - 1; i > 0; --i) {
      const uint64_t hi = c[i] > c[i - 1] ? c[i] : c[i - 1];
      const uint64_t lo = c[i] > c[i - 1] ? c[i - 1] : c[i];
      c[i - 1] = hi;
      c[i] = lo;
    }
  }
  template <int VPL>
  __device__ __forceinline__ void fill(const uint64_t (&key)[VPL], uint64_t below) {
#pragma unroll
    for (int i = 0; i < N; ++i) c[i] = 0;
#pragma unroll
    for (int v = 0; v < VPL; ++v)
      if (key[v] < below) insert(key[v]);
  }
  __device__ __forceinline__ void pop() {
#pragma unroll
    for (int i = 0; i + 1 < N; ++i) c[i] = c[i + 1];
    c[N - 1] = 0;
  }
};

// Sixteen lanes (one DPP row) per (token, group) row, four rows per wavefront: lane
// j of a row holds blocks j, j + 16, ... (VPL values). Each pick is a 16-lane DPP
// max of the lanes' best remaining keys. A lane keeps its largest remaining keys
// sorted (TopN: 4 for up to 16 values per lane, 8 above, where a lane more often
// holds several winners); the owner of a pick pops it and refills from its values below the
// popped key only once its cache is empty. The picks are those of a full rescan
// after every pick: the cache always holds the lane's largest keys below its last
// popped one.
// Every lane of the wavefront must call it (row >= rows: no output, but the lanes
// still take part in the DPP and shuffle steps). The selection key is the ordered
// float bits << 32 | ~block, so one 64-bit comparison implements "larger value,
// then smaller block id".
template <int VPL>
__device__ __forceinline__ void topk_row16(const float* __restrict__ scores, const int32_t* __restrict__ cu,
                                           int nseq, int64_t rows, int G, int NB, int B, int K, int L,
                                           int32_t* __restrict__ out, int64_t row, int sub) {
  const bool live = row < rows;
  const int64_t rr = live ? row : rows - 1;
  const int64_t t = rr / G;
  const int s = find_seq(cu, nseq, t);
  const int64_t qb = (t - cu[s]) / B;
  const int n = static_cast<int>(qb + 1 < NB ? qb + 1 : NB);
  const int count = K < NB ? K : NB;
  const int sel = live ? (count < n ? count : n) : 0;
  const float* src = scores + rr * NB;
  int32_t* dst = out + rr * K;

  uint64_t key[VPL];
#pragma unroll
  for (int v = 0; v < VPL; ++v) {
    const int b = v * 16 + sub;
    uint32_t k = 0u;  // below every real key: never selected
    if (b < n) {
      k = (L > 0 && b > qb - L) ? kKeyPosInf : ordered_key(src[b]);
    }
    key[v] = (static_cast<uint64_t>(k) << 32) | static_cast<uint32_t>(~static_cast<uint32_t>(b));
  }
  TopN<(VPL > 16 ? 8 : 4)> top;
  top.fill(key, ~uint64_t(0));

  // every row of the wave runs the same number of picks (the wave maximum)
  int sel_w = sel;
#pragma unroll
  for (int o = 16; o < 64; o <<= 1) sel_w = max(sel_w, __shfl_xor(sel_w, o, kWave));
  for (int it = 0; it < sel_w; ++it) {
    const uint64_t win = row16_max_u64(top.c[0]);
    const int b = static_cast<int>(~static_cast<uint32_t>(win));
    const uint32_t k = static_cast<uint32_t>(win >> 32);
    if (sub == 0 && it < sel) dst[it] = (k == kKeyNegInf) ? -1 : b;
    if ((b & 15) == sub && it < sel) {  // win == top.c[0] of this lane
      top.pop();
      if (top.c[0] == 0) top.fill(key, win);
    }
  }
  if (live)
    for (int it = sel + sub; it < K; it += 16) dst[it] = -1;
}

// The two values of the lanes l and l ^ J, in either order, for J a power of two.
template <int J>
__device__ __forceinline__ void xor_pair(uint32_t v, uint32_t& a, uint32_t& b) {
  a = v;
  if constexpr (J == 1) b = __builtin_amdgcn_update_dpp(0u, v, 0xB1, 0xF, 0xF, false);
  else if constexpr (J == 2) b = __builtin_amdgcn_update_dpp(0u, v, 0x4E, 0xF, 0xF, false);
  else if constexpr (J == 4)  // xor 7 (row_half_mirror), then xor 3 (quad_perm [3, 2, 1, 0])
    b = __builtin_amdgcn_update_dpp(0u, __builtin_amdgcn_update_dpp(0u, v, 0x141, 0xF, 0xF, false), 0x1B, 0xF, 0xF,
                                    false);
  else if constexpr (J == 8) b = __builtin_amdgcn_update_dpp(0u, v, 0x128, 0xF, 0xF, false);  // row_ror:8
  else {
    const auto r = J == 16 ? __builtin_amdgcn_permlane16_swap(v, v, false, false)
                           : __builtin_amdgcn_permlane32_swap(v, v, false, false);
    a = r[0];
    b = r[1];
  }
}

// The lanes that keep the larger value in stage K, step J of a bitonic sort, descending within
// runs of N lanes.
constexpr uint64_t bitonic_mask(int n, int k, int j) {
  uint64_t m = 0;
  for (int l = 0; l < 64; ++l)
    if (((l & j) == 0) == (k == n || (l & k) == 0)) m |= uint64_t(1) << l;
  return m;
}

// One compare-exchange. Keys are doubles: v_max_f64 / v_min_f64 order 52-bit integers in one
// instruction each, written out because the optimiser would canonicalise both operands and
// form the constant lane mask in vector code.
template <int N, int K, int J>
__device__ __forceinline__ double bitonic_step(double x) {
  const uint64_t u = static_cast<uint64_t>(__double_as_longlong(x));
  uint32_t al, bl, ah, bh;
  xor_pair<J>(static_cast<uint32_t>(u), al, bl);
  xor_pair<J>(static_cast<uint32_t>(u >> 32), ah, bh);
  const uint64_t a = (static_cast<uint64_t>(ah) << 32) | al, b = (static_cast<uint64_t>(bh) << 32) | bl;
  uint64_t mx, mn;
  asm("v_max_f64 %0, %1, %2" : "=v"(mx) : "v"(a), "v"(b));
  asm("v_min_f64 %0, %1, %2" : "=v"(mn) : "v"(a), "v"(b));
  uint32_t lo, hi;
  const uint64_t take = bitonic_mask(N, K, J);
  asm("v_cndmask_b32 %0, %1, %2, %3" : "=v"(lo) : "v"(static_cast<uint32_t>(mn)), "v"(static_cast<uint32_t>(mx)), "s"(take));
  asm("v_cndmask_b32 %0, %1, %2, %3"
      : "=v"(hi)
      : "v"(static_cast<uint32_t>(mn >> 32)), "v"(static_cast<uint32_t>(mx >> 32)), "s"(take));
  return __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hi) << 32) | lo));
}
template <int N, int K = 2, int J = 1>
__device__ __forceinline__ double bitonic_sort(double x) {
  x = bitonic_step<N, K, J>(x);
  if constexpr (J > 1) return bitonic_sort<N, K, J / 2>(x);
  else if constexpr (K < N) return bitonic_sort<N, 2 * K, K>(x);
  else return x;
}

// The same for 32-bit keys.
template <int N, int K = 2, int J = 1>
__device__ __forceinline__ uint32_t bitonic_sort_u32(uint32_t x) {
  uint32_t a, b, r;
  xor_pair<J>(x, a, b);
  const uint64_t take = bitonic_mask(N, K, J);
  asm("v_cndmask_b32 %0, %1, %2, %3" : "=v"(r) : "v"(a < b ? a : b), "v"(a < b ? b : a), "s"(take));
  if constexpr (J > 1) return bitonic_sort_u32<N, K, J / 2>(r);
  else if constexpr (K < N) return bitonic_sort_u32<N, 2 * K, K>(r);
  else return r;
}

// The selection of rows of 65 to 1024 blocks with up to 64 slots, by threshold and sort:
// the row's ordered keys sit in the wave's registers (lane j: blocks j, j + 64, ...), the
// sel-th largest of the lane maxima (one bitonic sort over lanes), or a bisection on ballot
// counts from there, gives a key that between `sel` and CAP values reach; those go to LDS and
// a second sort puts them in order. CAP = 32 sorts two rows per wave (up to 24 slots, so that
// most rows need no bisection), CAP = 64 one. Bound by VALU work and, in the bisection, by
// scalar counts (threshold by bisection alone: 410 us where the lane maxima give 325, and 538
// with 32 slots in CAP = 32). Measured against the iterated argmax of topk_row16, a 16-lane
// 64-bit maximum per slot: 65 536 tokens x 8 groups, 512 blocks, 32 slots 757 -> 325 us;
// 32 768 x 4, 256 blocks, 16 slots 71 -> 52 us.
constexpr int kSelectMostSlots = 64, kSelectPairSlots = 24;
// A row's threshold and two sorts cost the same for one slot as for 24, the argmax of topk_row16 by
// the slot: rows of up to 128 (256) blocks take that one up to these many slots. Argmax / sort, us,
// 262 144 rows: 128 blocks with 4 slots 49 / 83, 10 65 / 85, 12 74 / 84, 16 87 / 83; 256 blocks with 4 76 / 97, 8 93 /
// 100, 10 101 / 100; 16 384 rows: 128 blocks with 4 5.4 / 7.4, 10 7.6 / 7.6, 256 with 7 9.3 / 8.6; 257 blocks and
// more: sort (320 blocks, one slot, 262 144 rows: 202 / 107).
constexpr int kArgmaxSlots128 = 11, kArgmaxSlots256 = 7;
template <int VPL, int CAP>
__device__ __forceinline__ void topk_threshold(const float* __restrict__ scores, const int32_t* __restrict__ cu,
                                               int nseq, int64_t rows, int G, int NB, int B, int K, int L,
                                               int32_t* __restrict__ out, int64_t wave, int lane, uint2* cand) {
  constexpr int ROWS = 64 / CAP;
  cand[lane] = make_uint2(0u, 0u);  // below every real key
  int sel_own = 0;
  for (int p = 0; p < ROWS; ++p) {
    const int64_t row = ROWS * wave + p;
    if (row >= rows) break;  // wave-uniform
    const int32_t t = static_cast<int32_t>(rows <= 0x7fffffff ? static_cast<uint32_t>(row) / static_cast<uint32_t>(G)
                                                              : row / G);
    const int32_t qb = (t - cu[find_seq(cu, nseq, t)]) / B;
    const int n = qb + 1 < NB ? qb + 1 : NB;
    const int sel = K < n ? K : n;  // slots to fill
    const int own0 = L > 0 && qb - L + 1 < n ? qb - L + 1 : n;  // the forced local blocks: own0 .. n - 1
    if (ROWS == 1 || (lane >> 5) == p) sel_own = sel;
    const float* src = scores + row * NB;
    uint32_t key[VPL];  // 0 past the causal prefix
#pragma unroll
    for (int v = 0; v < VPL; ++v) {  // raw bits: all loads before the first use
      key[v] = 0u;
      if (64 * v < n) {
        const int b = 64 * v + lane;
        key[v] = __float_as_uint(src[b < n ? b : n - 1]);
      }
    }
    uint32_t top = 0u;  // the lane's largest key
#pragma unroll
    for (int v = 0; v < VPL; ++v) {
      if (64 * v < n) {
        const int b = 64 * v + lane;
        uint32_t k = ordered_key(__uint_as_float(key[v]));
        k = b >= own0 ? kKeyPosInf : k;
        key[v] = k = b < n ? k : 0u;
        top = k > top ? k : top;
      }
    }
    auto reach = [&](uint32_t x) {  // values of key >= x (x > 0)
      int c = 0;
#pragma unroll
      for (int v = 0; v < VPL; ++v) c += __popcll(__ballot(key[v] >= x));
      return c;
    };
    // `at`: the candidates are the keys >= at, and where those are fewer than sel, the
    // first blocks with key at - 1 (more than CAP values share it). The sel-th largest of
    // the 64 lane maxima is reached by sel values at least, and on most rows by not many
    // more (about 42 for sel = 32 of 512 independent values); the bisection is for the rest.
    uint32_t at = 1u;
    if (n > CAP) {
      at = __builtin_amdgcn_readlane(bitonic_sort_u32<64>(top), sel - 1);
      int c = reach(at);
      uint32_t lo = at, hi = 0xffffffffu;  // hi: above every key
      while (c > CAP || c < sel) {
        if (c > CAP) lo = at; else hi = at;
        if (hi - lo <= 1u) {
          at = hi;
          break;
        }
        at = lo + ((hi - lo) >> 1);
        c = reach(at);
      }
    }
    int base = CAP * p;
    const int stop = CAP * (p + 1);
#pragma unroll
    for (int v = 0; v < VPL; ++v) {
      const uint64_t m = __ballot(key[v] >= at);
      if (m) {
        const int pos = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32),
                                                  __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), base));
        if (key[v] >= at) cand[pos] = make_uint2(key[v], 64 * v + lane);
        base += __popcll(m);
      }
    }
    if (base - CAP * p < sel) {  // ties: ascending blocks, as many as there is room for
#pragma unroll
      for (int v = 0; v < VPL; ++v) {
        const uint64_t m = __ballot(key[v] == at - 1u);
        const int pos = base + __popcll(m & ((uint64_t(1) << lane) - 1));
        if (key[v] == at - 1u && pos < stop) cand[pos] = make_uint2(key[v], 64 * v + lane);
        base += __popcll(m);
        if (base > stop) base = stop;
      }
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  // 2^52 + (key << 20 | ~block): larger value first, then the smaller block id
  const uint2 c = cand[lane];
  const uint32_t hw = 0x43300000u | (c.x >> 12), lw = (c.x << 20) | (0xfffffu ^ c.y);
  double x = __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hw) << 32) | lw));
  x = bitonic_sort<CAP>(x);
  const uint64_t u = static_cast<uint64_t>(__double_as_longlong(x));
  const uint32_t k = static_cast<uint32_t>(u >> 20);  // (the exponent bits fall off the top)
  const int b = static_cast<int>((static_cast<uint32_t>(u) & 0xfffffu) ^ 0xfffffu);
  const int slot = lane & (CAP - 1);
  const int64_t row = ROWS * wave + lane / CAP;
  if (row < rows && slot < K) out[row * K + slot] = slot < sel_own && k != kKeyNegInf ? b : -1;
}

// Host launch of the stand-alone selection (topk.hip): 16-lane rows up to 64 blocks,
// threshold and sort up to 1024 (16-lane rows there for more than 64 slots, and up to 256
// blocks for few), one wavefront per row with the row in registers up to 4096, streamed above.
int topk_launch(const float* scores, const int32_t* cu_seqlens, int nseq, int64_t rows, int G, int NB, int B, int K,
                int L, int32_t* indices, hipStream_t st);

// One wavefront per row: lane j holds blocks j, j + 64, ... (VPL values); each pick
// is a 64-lane max. All lanes of the wavefront call it for the same row.
template <int VPL>
__device__ __forceinline__ void topk_row64(const float* __restrict__ scores, const int32_t* __restrict__ cu,
                                           int nseq, int G, int NB, int B, int K, int L,
                                           int32_t* __restrict__ out, int64_t row, int lane) {
  const int64_t t = row / G;
  const int s = find_seq(cu, nseq, t);
  const int64_t qb = (t - cu[s]) / B;
  const int n = static_cast<int>(qb + 1 < NB ? qb + 1 : NB);
  const int count = K < NB ? K : NB;
  const int sel = count < n ? count : n;
  const float* src = scores + row * NB;
  int32_t* dst = out + row * K;
  uint64_t key[VPL];
#pragma unroll
  for (int v = 0; v < VPL; ++v) {
    const int b = v * kWave + lane;
    uint32_t k = 0u;
    if (b < n) k = (L > 0 && b > qb - L) ? kKeyPosInf : ordered_key(src[b]);
    key[v] = (static_cast<uint64_t>(k) << 32) | static_cast<uint32_t>(~static_cast<uint32_t>(b));
  }
  uint64_t best = 0;
#pragma unroll
  for (int v = 0; v < VPL; ++v) best = key[v] > best ? key[v] : best;
  for (int it = 0; it < sel; ++it) {
    const uint64_t win = wave_max_u64(best);
    const int b = static_cast<int>(~static_cast<uint32_t>(win));
    const uint32_t k = static_cast<uint32_t>(win >> 32);
    if (lane == 0) dst[it] = (k == kKeyNegInf) ? -1 : b;
    if ((b & 63) == lane) {
      best = 0;
#pragma unroll
      for (int v = 0; v < VPL; ++v) {
        if (key[v] == win) key[v] = 0;
        best = key[v] > best ? key[v] : best;
      }
    }
  }
  for (int it = sel + lane; it < K; it += kWave) dst[it] = -1;
}

// One wavefront per row with the row left in memory, for any number of blocks (used
// above 4096): lane j scans blocks j, j + 64, ... and keeps its eight largest keys
// below its last pick (TopN<8>); it rescans its blocks only when that cache runs empty,
// so a row is read about once. Picks, order and padding are those of topk_row64.
__device__ __forceinline__ void topk_row_stream(const float* __restrict__ scores, const int32_t* __restrict__ cu,
                                                int nseq, int G, int NB, int B, int K, int L,
                                                int32_t* __restrict__ out, int64_t row, int lane) {
  const int64_t t = row / G;
  const int s = find_seq(cu, nseq, t);
  const int64_t qb = (t - cu[s]) / B;
  const int n = static_cast<int>(qb + 1 < NB ? qb + 1 : NB);
  const int count = K < NB ? K : NB;
  const int sel = count < n ? count : n;
  const float* src = scores + row * NB;
  int32_t* dst = out + row * static_cast<int64_t>(K);
  TopN<8> top;
  auto fill = [&](uint64_t below) {
#pragma unroll
    for (int i = 0; i < 8; ++i) top.c[i] = 0;
    for (int b = lane; b < n; b += kWave) {
      const uint32_t k = (L > 0 && b > qb - L) ? kKeyPosInf : ordered_key(src[b]);
      const uint64_t x = (static_cast<uint64_t>(k) << 32) | static_cast<uint32_t>(~static_cast<uint32_t>(b));
      if (x < below) top.insert(x);
    }
  };
  fill(~uint64_t(0));
  for (int it = 0; it < sel; ++it) {
    const uint64_t win = wave_max_u64(top.c[0]);
    const int b = static_cast<int>(~static_cast<uint32_t>(win));
    const uint32_t k = static_cast<uint32_t>(win >> 32);
    if (lane == 0) dst[it] = (k == kKeyNegInf) ? -1 : b;
    if ((b & 63) == lane) {  // win == top.c[0] of this lane
      top.pop();
      if (top.c[0] == 0) fill(win);
    }
  }
  for (int it = sel + lane; it < K; it += kWave) dst[it] = -1;
}

}  // namespace msa
