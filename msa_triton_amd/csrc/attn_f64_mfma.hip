// Stage 3 for fp32 inputs on v_mfma_f64_16x16x4_f64: the FP64 arithmetic of the VALU kernels
// (attn_scalar.hip: exact products, FP64 logits, softmax and sums), with the products on the
// matrix cores.
//
// Bound by the FP64 matrix rate (69 TFLOP/s measured, the FP64 vector rate): the VALU kernels
// reached 7 % of it, limited by the address unit (a lane per key row). Here a wave reads 16
// rows at a time, 16 bytes per lane, and converts each element once per use (full-rate
// v_cvt_f64_f32 beside 64-cycle MFMAs). Measured at 2048 tokens, 2 groups x 8 heads of 128
// dims, 8 slots: forward 1372 -> 478 us, query pass 2398 -> 661, KV pass 2069 -> 733.
//
// Operand layouts (checked on the device): lane l (c = l % 16, q4 = l / 16) holds A[c][q4] and
// B[q4][c] of a 16x16x4 product, and C[4 i + q4][c] in element i. Two facts follow:
//  * The order of the inner index is free as long as A and B agree. For products over dims the
//    lane reads float4 at dims 16 j + 4 q4; element s belongs to step (j, s).
//  * Element s of a C tile is the A operand of step s of the next product, transposed, with
//    inner index 4 s + q4: P^T feeds P.V, dS^T feeds dS.K and so on, without a shuffle. The B
//    operand then reads row 4 s + q4 with float4 at dims 64 a + 4 c (element b: output tile
//    4 a + b, i.e. column c of that tile is dim 64 a + 4 c + b), and for D % 64 == 32 float2 at
//    the last 32 dims.
//
// Query passes: one workgroup per (token, group), its R heads (3 to 8) the columns of the
// logits (16: the rest is idle; below 3 the VALU kernels waste less; above 8 the dQ pass's two key
// sums no longer fit the 16 rows of one product, nor the waves' sums the 64 KiB of LDS that two
// workgroups per CU leave: 9 to 16 heads stay on the VALU kernels, untried here), its key tiles of 16
// dealt to 4 waves; their sums are added in wave order. The query pass forms its two key sums
// (of u = p (dp - c) and of p) in one product: rows 0-7 of the A operand are u, 8-15 p.
// KV pass: one workgroup per 16 keys and group, the rows (edge, head) of the block's CSR row
// 16 at a time, dealt to 8 waves; the waves' sums are added in wave order. Tiles of few rows and keys
// are the VALU kernel's (kF64FewestPairs).
#include <algorithm>

#include "attn_f64_mfma.hpp"

namespace msa {

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f64x4 mfma64(double a, double b, f64x4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// One row's elements for a product over dims: float4 at dims 16 j + 4 q4.
template <int D>
struct DimFrag {
  float4 x[D / 16];
  __device__ __forceinline__ void load(const float* __restrict__ row, int q4) {
#pragma unroll
    for (int j = 0; j < D / 16; ++j) x[j] = *reinterpret_cast<const float4*>(row + 16 * j + 4 * q4);
  }
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int j = 0; j < D / 16; ++j) x[j] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
};
// x as FP64, converted here: the compiler would keep the 2 D / 4 registers of a fragment that
// stays for a whole loop in FP64 otherwise, and spill.
__device__ __forceinline__ double here_f64(float x) {
  asm volatile("" : "+v"(x));
  return static_cast<double>(x);
}
// sum over dims of a[.][d] b[.][d]: C[row of a][row of b]; b is the fragment that stays
template <int D>
__device__ __forceinline__ f64x4 dot_rows(const DimFrag<D>& a, const DimFrag<D>& b) {
  f64x4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int j = 0; j < D / 16; ++j) {
    acc = mfma64(a.x[j].x, here_f64(b.x[j].x), acc);
    acc = mfma64(a.x[j].y, here_f64(b.x[j].y), acc);
    acc = mfma64(a.x[j].z, here_f64(b.x[j].z), acc);
    acc = mfma64(a.x[j].w, here_f64(b.x[j].w), acc);
  }
  return acc;
}

// One row's elements as the B operand of a product over rows (output dims along the lanes).
template <int D>
struct RowFrag {
  static constexpr int NA = D / 64;
  static constexpr bool TAIL = D % 64 != 0;
  float4 x[NA > 0 ? NA : 1];
  float2 t;
  // (global loads are asked for by name: a row that is chosen from two arrays would be read with
  // flat ones)
  __device__ __forceinline__ void load(const float* __restrict__ row, int c) {
    typedef const __attribute__((address_space(1))) float* Global;
    typedef const __attribute__((address_space(1))) f32x4* Global4;
#pragma unroll
    for (int a = 0; a < NA; ++a) {
      const f32x4 y = *(Global4)(row + 64 * a + 4 * c);
      x[a] = make_float4(y[0], y[1], y[2], y[3]);
    }
    if constexpr (TAIL) {
      const Global y = (Global)(row + 64 * NA + 2 * c);
      t = make_float2(y[0], y[1]);
    }
  }
  // out[tile] += a^T . this row
  __device__ __forceinline__ void accumulate(double a, f64x4 (&out)[D / 16]) const {
#pragma unroll
    for (int n = 0; n < NA; ++n) {
      out[4 * n] = mfma64(a, x[n].x, out[4 * n]);
      out[4 * n + 1] = mfma64(a, x[n].y, out[4 * n + 1]);
      out[4 * n + 2] = mfma64(a, x[n].z, out[4 * n + 2]);
      out[4 * n + 3] = mfma64(a, x[n].w, out[4 * n + 3]);
    }
    if constexpr (TAIL) {
      out[4 * NA] = mfma64(a, t.x, out[4 * NA]);
      out[4 * NA + 1] = mfma64(a, t.y, out[4 * NA + 1]);
    }
  }
};
// dim of column c of output tile n
template <int D>
__device__ __forceinline__ int tile_dim(int n, int c) {
  return n < 4 * (D / 64) ? 64 * (n / 4) + 4 * c + n % 4 : 64 * (D / 64) + 2 * c + (n - 4 * (D / 64));
}

// Stands in for a row that must not enter a product (0 times an infinity or a NaN is NaN).
alignas(16) __device__ const float kZeroRow[128] = {};

// The sum (maximum) over the lanes c, c + 16, c + 32, c + 48.
__device__ __forceinline__ double quarter_sum(double x) {
  x += __shfl_xor(x, 16, kWave);
  return x + __shfl_xor(x, 32, kWave);
}
__device__ __forceinline__ double quarter_max(double x) {
  x = fmax(x, __shfl_xor(x, 16, kWave));
  return fmax(x, __shfl_xor(x, 32, kWave));
}

constexpr int kQueryWaves = 4, kKeyWaves = 8, kMostHeads = 8;

// The (token, group) of a query workgroup and its key tiles: calls fn(first key, keys) for
// every tile of up to 16 visible keys of the selected blocks that falls to wave `wid`.
struct QueryRow {
  int64_t t, start, qb;
  int g;
  const int32_t* sel;
};
__device__ __forceinline__ QueryRow query_row(const int32_t* __restrict__ indices, const int32_t* __restrict__ cu,
                                              int nseq, int G, int K, int B) {
  QueryRow r;
  r.t = blockIdx.x / G;
  r.g = static_cast<int>(blockIdx.x % G);
  r.start = cu[find_seq(cu, nseq, r.t)];
  r.qb = (r.t - r.start) / B;
  r.sel = indices + (r.t * G + r.g) * K;
  return r;
}
template <typename Fn>
__device__ __forceinline__ void for_key_tiles(const QueryRow& r, int K, int B, int wid, Fn fn) {
  int tile = 0;
  for (int slot = 0; slot < K; ++slot) {
    const int blk = r.sel[slot];
    if (blk < 0 || blk > r.qb) continue;
    const int64_t kb0 = r.start + static_cast<int64_t>(blk) * B;
    const int64_t kend = (kb0 + B < r.t + 1) ? kb0 + B : r.t + 1;
    const int n = static_cast<int>(kend - kb0 + 15) / 16;
    for (int i = (wid - tile) & (kQueryWaves - 1); i < n; i += kQueryWaves) {
      const int64_t key = kb0 + 16 * i;
      fn(key, static_cast<int>(kend - key < 16 ? kend - key : 16));
    }
    tile += n;
  }
}

}  // namespace

template <int D>
__global__ __launch_bounds__(64 * kQueryWaves, 2) void attn_f64_fwd(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    const int32_t* __restrict__ indices, const int32_t* __restrict__ cu, int nseq, int Hq, int G, int K, int B,
    double scale, float* __restrict__ out, float* __restrict__ lse, double* __restrict__ row_state,
    float* __restrict__ o32) {
  constexpr int NT = D / 16;
  __shared__ double obuf[kQueryWaves][kMostHeads][D];
  __shared__ double mbuf[kQueryWaves][kMostHeads], lbuf[kQueryWaves][kMostHeads];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, q4 = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const QueryRow r = query_row(indices, cu, nseq, G, K, B);
  const int R = Hq / G;
  const int64_t th0 = r.t * Hq + static_cast<int64_t>(r.g) * R;
  DimFrag<D> qf;  // columns: heads
  if (c < R) qf.load(q + (th0 + c) * D, q4); else qf.zero();
  double m = -__builtin_inf(), l = 0.0;  // head c: running maximum; this lane's keys' sum
  f64x4 o[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) o[n] = f64x4{0.0, 0.0, 0.0, 0.0};
  for_key_tiles(r, K, B, wid, [&](int64_t key, int nk) __attribute__((always_inline)) {
    auto at = [&](int i) { return ((key + (i < nk ? i : nk - 1)) * G + r.g) * D; };
    DimFrag<D> kf;
    kf.load(k + at(c), q4);
    RowFrag<D> vf[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) vf[s].load(4 * s + q4 < nk ? v + at(4 * s + q4) : kZeroRow, c);
    const f64x4 x = dot_rows<D>(kf, qf);  // [key 4 s + q4][head c]
    double p[4], mt = -__builtin_inf();
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      p[s] = 4 * s + q4 < nk ? x[s] * scale : -__builtin_inf();
      mt = fmax(mt, p[s]);
    }
    const double mn = fmax(m, quarter_max(mt));
    if (__ballot(mn != m) != 0) {  // rescale: output rows are heads
      const double alpha = m == -__builtin_inf() ? 0.0 : exp(m - mn);
      l *= alpha;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const double ai = __shfl(alpha, 4 * i + q4, kWave);
#pragma unroll
        for (int n = 0; n < NT; ++n) o[n][i] *= ai;
      }
      m = mn;
    }
    const double base = mn == -__builtin_inf() ? 0.0 : mn;  // (only logits of -inf so far: weights 0, not NaN)
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      p[s] = 4 * s + q4 < nk ? exp(p[s] - base) : 0.0;
      l += p[s];
      vf[s].accumulate(p[s], o);
    }
  });
  l = quarter_sum(l);
  if (q4 == 0 && c < R) {
    mbuf[wid][c] = m;
    lbuf[wid][c] = l;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {  // heads 4 i + q4 < 8
    const int h = 4 * i + q4;
    if (h < R)
#pragma unroll
      for (int n = 0; n < NT; ++n) obuf[wid][h][tile_dim<D>(n, c)] = o[n][i];
  }
  __syncthreads();
  for (int e = tid; e < R * D; e += 64 * kQueryWaves) {
    const int h = e / D, d = e % D;
    double M = -__builtin_inf();
#pragma unroll
    for (int w = 0; w < kQueryWaves; ++w) M = fmax(M, mbuf[w][h]);
    double L = 0.0, x = 0.0;
#pragma unroll
    for (int w = 0; w < kQueryWaves; ++w) {
      const double f = mbuf[w][h] == -__builtin_inf() ? 0.0 : exp(mbuf[w][h] - M);
      L = fma(f, lbuf[w][h], L);
      x = fma(f, obuf[w][h][d], x);
    }
    const float y = static_cast<float>(L > 0.0 ? x / L : 0.0);
    const int64_t th = th0 + h;
    out[th * D + d] = y;
    if (o32) o32[th * D + d] = y;
    if (d == 0) {
      const double full = L > 0.0 ? M + log(L) : -__builtin_inf();
      lse[th] = static_cast<float>(full);
      if (row_state) {
        row_state[th * 4] = full;
        row_state[th * 4 + 1] = 1.0;  // FP64 lse: p = exp(x - lse) needs no mass correction
      }
    }
  }
}

// dQ = scale / mass (sum u k - delta sum p k), u = p (dp - c), and the row statistics for the
// KV pass.
template <int D>
__global__ __launch_bounds__(64 * kQueryWaves, 2) void attn_f64_dq(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ out, const float* __restrict__ dout, double* __restrict__ row_state,
    const int32_t* __restrict__ indices, const int32_t* __restrict__ cu, int nseq, int Hq, int G, int K, int B,
    double scale, float* __restrict__ dq) {
  constexpr int NT = D / 16;
  __shared__ double abuf[kQueryWaves][2 * kMostHeads][D];
  __shared__ double mbuf[kQueryWaves][kMostHeads], dbuf[kQueryWaves][kMostHeads];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, q4 = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const QueryRow r = query_row(indices, cu, nseq, G, K, B);
  const int R = Hq / G;
  const int64_t th0 = r.t * Hq + static_cast<int64_t>(r.g) * R;
  DimFrag<D> qf, gf;  // columns: heads
  double cen = 0.0, row_lse = -__builtin_inf();
  if (c < R) {
    qf.load(q + (th0 + c) * D, q4);
    gf.load(dout + (th0 + c) * D, q4);
    DimFrag<D> of;
    of.load(out + (th0 + c) * D, q4);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      cen = fma(static_cast<double>(of.x[j].x), static_cast<double>(gf.x[j].x), cen);
      cen = fma(static_cast<double>(of.x[j].y), static_cast<double>(gf.x[j].y), cen);
      cen = fma(static_cast<double>(of.x[j].z), static_cast<double>(gf.x[j].z), cen);
      cen = fma(static_cast<double>(of.x[j].w), static_cast<double>(gf.x[j].w), cen);
    }
    row_lse = row_state[(th0 + c) * 4];
  } else {
    qf.zero();
    gf.zero();
  }
  cen = quarter_sum(cen);
  const bool live = row_lse != -__builtin_inf();  // (a row without visible keys has no tiles)
  double mass = 0.0, delta = 0.0;
  f64x4 ab[NT];  // rows 0-7: sum u k of head row; 8-15: sum p k of head row - 8
#pragma unroll
  for (int n = 0; n < NT; ++n) ab[n] = f64x4{0.0, 0.0, 0.0, 0.0};
  for_key_tiles(r, K, B, wid, [&](int64_t key, int nk) __attribute__((always_inline)) {
    auto at = [&](int i) { return ((key + (i < nk ? i : nk - 1)) * G + r.g) * D; };
    DimFrag<D> kf, vf;
    kf.load(k + at(c), q4);
    vf.load(v + at(c), q4);
    const f64x4 x = dot_rows<D>(kf, qf);   // [key 4 s + q4][head c]
    const f64x4 dp = dot_rows<D>(vf, gf);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      RowFrag<D> kr;
      kr.load(k + at(4 * s + q4), c);
      const bool ok = live && 4 * s + q4 < nk;
      const double p = ok ? exp(x[s] * scale - row_lse) : 0.0;
      const double u = ok ? p * (dp[s] - cen) : 0.0;  // (past nk dp repeats the last key's, which may be infinite)
      mass += p;
      delta += u;
      const double p8 = __shfl_xor(p, 8, kWave);  // p of head c - 8
      kr.accumulate(c < 8 ? u : p8, ab);
      if (D == 128) __builtin_amdgcn_sched_barrier(0);  // (one step's rows at a time: registers)
    }
  });
  mass = quarter_sum(mass);
  delta = quarter_sum(delta);
  if (q4 == 0 && c < R) {
    mbuf[wid][c] = mass;
    dbuf[wid][c] = delta;
    if (wid == 0) row_state[(th0 + c) * 4 + 2] = cen;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int n = 0; n < NT; ++n) abuf[wid][4 * i + q4][tile_dim<D>(n, c)] = ab[n][i];
  __syncthreads();
  for (int e = tid; e < R * D; e += 64 * kQueryWaves) {
    const int h = e / D, d = e % D;
    double msum = 0.0, dsum = 0.0, a = 0.0, b = 0.0;
#pragma unroll
    for (int w = 0; w < kQueryWaves; ++w) {
      msum += mbuf[w][h];
      dsum += dbuf[w][h];
      a += abuf[w][h][d];
      b += abuf[w][h + 8][d];
    }
    const bool has = msum > 0.0;
    const double dhat = has ? dsum / msum : 0.0;
    const int64_t th = th0 + h;
    if (dq) dq[th * D + d] = static_cast<float>(has ? scale * (a - dhat * b) / msum : 0.0);
    if (d == 0) {
      row_state[th * 4 + 1] = has ? msum : 1.0;
      row_state[th * 4 + 3] = dhat;
    }
  }
}

// dK, dV of 16 keys of one group: rows (edge, head) of the block's CSR row, 16 per step. With
// `part`, blockIdx.z of gridDim.z workgroups share the rows and leave FP64 sums there
// ([split][dK, dV][key][group][dim], added by attn_f64_dkdv_reduce); without, one workgroup
// has them all and writes dK and dV.
template <int D>
__global__ __launch_bounds__(64 * kKeyWaves, 2) void attn_f64_dkdv(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ dout, const double* __restrict__ row_state, const int32_t* __restrict__ cu,
    const int32_t* __restrict__ cu_blocks, const int32_t* __restrict__ row_ptr, const int32_t* __restrict__ qidx,
    int nseq, int64_t T, int Hq, int G, int B, int64_t compact, int fewest, double scale, float* __restrict__ dk,
    float* __restrict__ dv, double* __restrict__ part) {
  constexpr int NT = D / 16;
  __shared__ double kbuf[16][D], vbuf[16][D];
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, q4 = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  int64_t row, kb, kend;
  const int g = static_cast<int>(blockIdx.x % G);
  const int64_t x = blockIdx.x / G;
  if (compact == 0) {  // x: block * tiles of a whole block + tile
    const int64_t per_block = (static_cast<int64_t>(B) + 15) / 16, gb = x / per_block;
    if (gb >= cu_blocks[nseq]) return;  // whole workgroup
    int s = upper_index(cu_blocks, nseq + 1, gb);
    while (s < nseq && cu_blocks[s + 1] <= gb) ++s;
    const int64_t first = cu[s] + (gb - cu_blocks[s]) * B;
    kb = first + 16 * (x - gb * per_block);
    kend = first + B < cu[s + 1] ? first + B : cu[s + 1];
    row = gb * G + g;
  } else {
    // x: a number of a tile. Tile i of block gb has the number first / 16 + gb + i (first: the
    // block's first token): no two tiles share one, as a block of n keys has at most n / 16 + 1,
    // and all are below T / 16 + blocks. The even numbers go first: with blocks of 16 keys
    // every other number has no tile, and workgroups go to the XCDs round-robin.
    const int64_t w = x < compact ? 2 * x : 2 * (x - compact) + 1;
    int s = 0;  // the last sequence whose first tile is not after w
    for (int hi = nseq; hi - s > 1;) {
      const int mid = (s + hi) >> 1;
      if (cu[mid] / 16 + static_cast<int64_t>(cu_blocks[mid]) <= w) s = mid; else hi = mid;
    }
    const int64_t start = cu[s], gb0 = cu_blocks[s];
    int64_t b = 0;  // its last block whose first tile is not after w
    for (int64_t hi = cu_blocks[s + 1] - gb0; hi - b > 1;) {
      const int64_t mid = (b + hi) >> 1;
      if ((start + mid * B) / 16 + gb0 + mid <= w) b = mid; else hi = mid;
    }
    const int64_t first = start + b * B;
    kb = first + 16 * (w - first / 16 - gb0 - b);
    kend = first + B < cu[s + 1] ? first + B : cu[s + 1];
    row = (gb0 + b) * G + g;
  }
  if (kb >= kend) return;  // whole workgroup: no such tile
  const int nk = static_cast<int>(kend - kb < 16 ? kend - kb : 16);
  const int64_t e0 = row_ptr[row];
  const int R = Hq / G;
  const int64_t nrows = (row_ptr[row + 1] - e0) * R;
  if (nrows * nk < fewest) return;  // whole workgroup: left to the vector kernel
  f64x4 ak[NT], av[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) ak[n] = av[n] = f64x4{0.0, 0.0, 0.0, 0.0};
  const int64_t first = 16 * (wid + kKeyWaves * static_cast<int64_t>(blockIdx.z));
  const int64_t stride = 16 * kKeyWaves * static_cast<int64_t>(gridDim.z);
  uint64_t left_out = 0;
  for (int64_t i0 = first; i0 < nrows; i0 += stride) {
    // this lane's row (c): its token and (token, head); past the end the last row, masked
    const int64_t i = i0 + c < nrows ? i0 + c : nrows - 1;
    const int64_t eo = nrows <= 0x7fffffff ? static_cast<uint32_t>(i) / static_cast<uint32_t>(R) : i / R;
    const int t = qidx[e0 + eo];
    const int64_t th = static_cast<int64_t>(t) * Hq + static_cast<int64_t>(g) * R + (i - eo * R);
    // the key and value rows (columns) are read again each step: 64 registers that the sums need
    int kc = c < nk ? c : nk - 1;
    asm volatile("" : "+v"(kc));
    const int64_t off0 = ((kb + kc) * G + g) * D;
    DimFrag<D> rf, cf;
    rf.load(q + th * D, q4);
    cf.load(k + off0, q4);
    const f64x4 x = dot_rows<D>(rf, cf);  // [row 4 s + q4][key c]
    rf.load(dout + th * D, q4);
    cf.load(v + off0, q4);
    const f64x4 dp = dot_rows<D>(rf, cf);
    double p[4], ds[4];
    int64_t off[4];
    bool zero[4];
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      const int rr = 4 * s4 + q4;
      const int64_t tr = __shfl(t, rr, kWave);
      const int64_t thr = __shfl(th, rr, kWave);
      off[s4] = thr * D;
      const double2 a = reinterpret_cast<const double2*>(row_state)[thr * 2];      // lse, mass
      const double2 b = reinterpret_cast<const double2*>(row_state)[thr * 2 + 1];  // c, delta
      const bool ok = i0 + rr < nrows && c < nk && tr >= kb + c;
      p[s4] = ok ? exp(x[s4] * scale - a.x) / a.y : 0.0;
      ds[s4] = ok ? p[s4] * ((dp[s4] - b.x) - b.y) * scale : 0.0;
      // A masked pair has weight 0, but 0 times a row that holds an infinity or a NaN is NaN
      // (such a row's products with any key are not finite, and sums of finite fp32 products stay
      // far inside the FP64 range): the matrix product takes zeros for this row, and what it gives
      // to the keys that it does attend to is added at the end.
      const uint64_t odd = __ballot(!ok && !(fabs(x[s4]) < __builtin_inf() && fabs(dp[s4]) < __builtin_inf()));
      zero[s4] = (odd >> (16 * q4) & 0xffff) != 0;
      left_out |= odd;
    }
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      RowFrag<D> gr, qr;
      gr.load(zero[s4] ? kZeroRow : dout + off[s4], c);
      qr.load(zero[s4] ? kZeroRow : q + off[s4], c);
      gr.accumulate(p[s4], av);
      qr.accumulate(ds[s4], ak);
      if (D == 128) __builtin_amdgcn_sched_barrier(0);  // (one step's rows at a time: registers)
    }
  }
  // the sums of the waves that had rows, in wave order
  const int64_t steps = (nrows + 15) / 16 - kKeyWaves * static_cast<int64_t>(blockIdx.z);
  const int waves = steps < 1 ? 1 : (steps < kKeyWaves ? static_cast<int>(steps) : kKeyWaves);
  for (int w = 0; w < waves; ++w) {
    if (wid == w) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const int kk = 4 * i + q4, d = tile_dim<D>(n, c);
          kbuf[kk][d] = (w ? kbuf[kk][d] : 0.0) + ak[n][i];
          vbuf[kk][d] = (w ? vbuf[kk][d] : 0.0) + av[n][i];
        }
    }
    __syncthreads();
  }
  // the rows left out: a wave at a time, one row at a time, lane (key c, dims q4, q4 + 4, ...)
  for (int w = 0; __syncthreads_or(left_out != 0) && w < kKeyWaves; ++w) {
    for (int64_t i = first; wid == w && i < nrows; i += (i & 15) == 15 ? stride - 15 : 1) {
      const int64_t t = qidx[e0 + i / R], th = t * Hq + static_cast<int64_t>(g) * R + i % R;
      const int64_t off0 = ((kb + (c < nk ? c : nk - 1)) * G + g) * D;
      double x = 0.0, dp = 0.0;
#pragma unroll 1
      for (int d = q4; d < D; d += 4) {
        x = fma(static_cast<double>(q[th * D + d]), static_cast<double>(k[off0 + d]), x);
        dp = fma(static_cast<double>(dout[th * D + d]), static_cast<double>(v[off0 + d]), dp);
      }
      x = quarter_sum(x);
      dp = quarter_sum(dp);
      const bool ok = c < nk && t >= kb + c;
      if (__ballot(!ok && !(fabs(x) < __builtin_inf() && fabs(dp) < __builtin_inf())) == 0) continue;
      const double* a = row_state + th * 4;  // lse, mass, c, delta
      const double p = exp(x * scale - a[0]) / a[1], ds = p * ((dp - a[2]) - a[3]) * scale;
      if (ok)
#pragma unroll 1
        for (int d = q4; d < D; d += 4) {
          kbuf[c][d] = fma(ds, static_cast<double>(q[th * D + d]), kbuf[c][d]);
          vbuf[c][d] = fma(p, static_cast<double>(dout[th * D + d]), vbuf[c][d]);
        }
    }
  }
  for (int e = tid; e < nk * D; e += 64 * kKeyWaves) {
    const int kk = e / D, d = e % D;
    const int64_t o = ((kb + kk) * G + g) * D + d;
    if (part) {
      double* p = part + 2 * blockIdx.z * T * G * D;
      p[o] = kbuf[kk][d];
      p[T * G * D + o] = vbuf[kk][d];
    } else {
      if (dk) dk[o] = static_cast<float>(kbuf[kk][d]);
      if (dv) dv[o] = static_cast<float>(vbuf[kk][d]);
    }
  }
}

__global__ __launch_bounds__(256) void attn_f64_dkdv_reduce(const double* __restrict__ part, int splits, int64_t n,
                                                            float* __restrict__ dk, float* __restrict__ dv) {
  const int64_t o = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (o >= n) return;
  double a = 0.0, b = 0.0;
  for (int z = 0; z < splits; ++z) {
    a += part[2 * z * n + o];
    b += part[(2 * z + 1) * n + o];
  }
  if (dk) dk[o] = static_cast<float>(a);
  if (dv) dv[o] = static_cast<float>(b);
}

// Workgroups that share one 16-key tile's rows: up to 8, for 2048 in all. A tile's rows grow
// with how often its block is selected, and the earliest blocks of a sequence are visible to
// every query: with one workgroup per tile and about one tile per CU the pass takes as long as
// its longest tile (1262 us at 2048 tokens x 2 groups, split 722 and 11 for the sums).
static int dkdv_splits(int64_t T, int64_t G) {
  const int64_t tiles = (T + 15) / 16 * G, s = (2048 + tiles - 1) / tiles;
  return static_cast<int>(s > 8 ? 8 : s);
}

// Threads of a launch: fewer than 2^32. (The vector kernels have fewer threads per head or key.)
constexpr int64_t kMostThreads = int64_t{1} << 32;

// Head dims of 32, 64, 96 or 128 with rows that start on 16-byte boundaries; the query passes
// also need 3 to 8 heads per group (see above).
bool attn_f64_dims_fit(int D, std::initializer_list<const void*> rows) {
  uintptr_t bits = 0;
  for (const void* p : rows) bits |= reinterpret_cast<uintptr_t>(p);
  return D % 32 == 0 && D <= 128 && (bits & 15) == 0;
}
bool attn_f64_heads_fit(int64_t T, int64_t G, int R) {
  return R >= 3 && R <= kMostHeads && T * G < kMostThreads / (64 * kQueryWaves);
}

#define MSA_F64_DIMS(LAUNCH)  \
  switch (D) {                \
    case 32: LAUNCH(32); break;  \
    case 64: LAUNCH(64); break;  \
    case 96: LAUNCH(96); break;  \
    default: LAUNCH(128); break; \
  }

int attn_f64_fwd_launch(const float* q, const float* k, const float* v, const int32_t* idx, const int32_t* cu, int nseq,
                        int64_t T, int Hq, int G, int D, int K, int B, double scale, float* out, float* lse, double* rs,
                        float* o32, hipStream_t st) {
#define MSA_F64_FWD(DV) hipLaunchKernelGGL(attn_f64_fwd<DV>, dim3(static_cast<unsigned>(T * G)), dim3(64 * kQueryWaves), 0, st, q, k, v, idx, cu, nseq, Hq, G, K, B, scale, out, lse, rs, o32)
  MSA_F64_DIMS(MSA_F64_FWD)
#undef MSA_F64_FWD
  return status_from(hipGetLastError());
}

int attn_f64_dq_launch(const float* q, const float* k, const float* v, const float* out, const float* dout, double* rs,
                       const int32_t* idx, const int32_t* cu, int nseq, int64_t T, int Hq, int G, int D, int K, int B,
                       double scale, float* dq, hipStream_t st) {
#define MSA_F64_DQ(DV) hipLaunchKernelGGL(attn_f64_dq<DV>, dim3(static_cast<unsigned>(T * G)), dim3(64 * kQueryWaves), 0, st, q, k, v, out, dout, rs, idx, cu, nseq, Hq, G, K, B, scale, dq)
  MSA_F64_DIMS(MSA_F64_DQ)
#undef MSA_F64_DQ
  return status_from(hipGetLastError());
}

int64_t attn_f64_dkdv_workspace_bytes(int64_t T, int64_t G, int64_t D) {
  const int n = dkdv_splits(T, G);
  return n > 1 ? int64_t{16} * n * T * G * D : 0;
}

// One workgroup per tile of every block, a block's tiles side by side (they gather the same rows; with
// one block's tiles far apart 4 sequences of 2048 tokens took 8790 us for the backward, so 6257), or,
// where whole blocks would give more than two numbers per tile (short sequences, blocks far longer
// than they), numbered by tile: 8 sequences of 1024 tokens in blocks of 2^19 keys 8815 -> 5538 us.
// blocks: at least as many as there are; numbers without a tile come last, as far as possible
// (spread evenly between the others they leave shader engines idle: 8 x 1024, 8668 us).
struct KeyGrid {
  int64_t compact, numbers;  // numbers per group
};
static KeyGrid key_grid(int64_t T, int64_t nseq, int64_t B) {
  const int64_t blocks = T / B + nseq < T ? T / B + nseq : T, tiles = T / 16 + blocks, per_block = (B + 15) / 16;
  const int64_t compact = per_block * blocks > 2 * tiles ? (tiles + 1) / 2 : 0;
  return KeyGrid{compact, compact ? 2 * compact : blocks * per_block};
}
bool attn_f64_dkdv_fits(int64_t T, int64_t nseq, int64_t G, int64_t B) {
  return key_grid(T, nseq, B).numbers * G < kMostThreads / (64 * kKeyWaves);
}

F64Tile attn_f64_mean_tile(int64_t T, int nseq, int R, int K, int B) {
  const double blocks = static_cast<double>(T / B + nseq < T ? T / B + nseq : T), keys = T / blocks;
  const double slots = std::min<double>(K, (std::max(1.0, blocks / nseq) + 1) / 2);  // that exist
  return F64Tile{R * keys * slots, std::min(16.0, keys)};
}

int attn_f64_dkdv_launch(const float* q, const float* k, const float* v, const float* dout, const double* rs,
                         const int32_t* cu, const int32_t* cu_blocks, const int32_t* row_ptr, const int32_t* qidx,
                         int nseq, int64_t T, int Hq, int G, int D, int K, int B, int fewest, double scale, float* dk,
                         float* dv, void* ws, int64_t ws_bytes, hipStream_t st) {
  // a caller without the workspace gets the unsplit pass
  const int64_t need = attn_f64_dkdv_workspace_bytes(T, G, D);
  const bool split = ws && need > 0 && ws_bytes >= need && (reinterpret_cast<uintptr_t>(ws) & 7) == 0;
  // (a share of at least two steps on average: with fewer its zeros and the sum cost more than they give)
  const double most = attn_f64_mean_tile(T, nseq, Hq / G, K, B).rows / 32;
  const int splits = split ? std::max(1, static_cast<int>(std::min<double>(dkdv_splits(T, G), most))) : 1;
  double* part = splits > 1 ? static_cast<double*>(ws) : nullptr;
  const KeyGrid kg = key_grid(T, nseq, B);
  const dim3 grid(static_cast<unsigned>(kg.numbers * G), 1, splits);
#define MSA_F64_DKDV(DV) hipLaunchKernelGGL(attn_f64_dkdv<DV>, grid, dim3(64 * kKeyWaves), 0, st, q, k, v, dout, rs, cu, cu_blocks, row_ptr, qidx, nseq, T, Hq, G, B, kg.compact, fewest, scale, dk, dv, part)
  MSA_F64_DIMS(MSA_F64_DKDV)
#undef MSA_F64_DKDV
  if (splits > 1)
    hipLaunchKernelGGL(attn_f64_dkdv_reduce, dim3(grid_1d(T * G * D, 256)), dim3(256), 0, st, part, splits, T * G * D, dk,
                       dv);
  return status_from(hipGetLastError());
}

}  // namespace msa
