// fp32 attention on FP64 matrix products (attn_f64_mfma.hip).
#pragma once
#include <initializer_list>

#include "common.hpp"

namespace msa {

// What the kernels take: every pass needs fitting dims and 16-byte aligned rows, the query
// passes (forward, dQ) also fitting heads per group, and each a number of workgroups that one
// launch holds.
bool attn_f64_dims_fit(int D, std::initializer_list<const void*> rows);
bool attn_f64_heads_fit(int64_t T, int64_t G, int R);
bool attn_f64_dkdv_fits(int64_t T, int64_t nseq, int64_t G, int64_t B);

int attn_f64_fwd_launch(const float* q, const float* k, const float* v, const int32_t* idx, const int32_t* cu, int nseq,
                        int64_t T, int Hq, int G, int D, int K, int B, double scale, float* out, float* lse, double* rs,
                        float* o32, hipStream_t st);
int attn_f64_dq_launch(const float* q, const float* k, const float* v, const float* out, const float* dout, double* rs,
                       const int32_t* idx, const int32_t* cu, int nseq, int64_t T, int Hq, int G, int D, int K, int B,
                       double scale, float* dq, hipStream_t st);
int attn_f64_dkdv_launch(const float* q, const float* k, const float* v, const float* dout, const double* rs,
                         const int32_t* cu, const int32_t* cu_blocks, const int32_t* row_ptr, const int32_t* qidx,
                         int nseq, int64_t T, int Hq, int G, int D, int K, int B, int fewest, double scale, float* dk,
                         float* dv, void* ws, int64_t ws_bytes, hipStream_t st);

// The KV pass takes 16 keys of a block at a time against the block's rows (edge, head). A tile
// with fewer than kF64FewestPairs (row, key) pairs goes to the vector kernel, one wave per key:
// the matrix kernel's workgroup, 16 columns and sum cost more than they save. Measured on the
// backward with 2 groups of 128 dims, vector / matrix: 8192 sequences of one token, 8 heads (8 pairs)
// 840 / 1559 us, 4096 x 2 (32) 799 / 996, 2731 x 3 (72) 796 / 856, 2048 x 4 (128) 794 / 721;
// one head, blocks of 4 keys with 4 slots (64) 343 / 514, of 16 with 2 (512) 272 / 266.
constexpr int kF64FewestPairs = 100;
__device__ __forceinline__ bool f64_few_pairs(int64_t rows, int64_t offset, int64_t block_keys) {
  const int64_t left = block_keys - offset / 16 * 16;  // offset: of a key in its block
  return rows * (left < 16 ? left : 16) < kF64FewestPairs;
}
// Mean rows and keys of a call's tiles, as far as the sizes tell (each sequence's slots as if it
// had the mean number of blocks).
struct F64Tile {
  double rows, keys;
};
F64Tile attn_f64_mean_tile(int64_t T, int nseq, int R, int K, int B);

// FP64 partial sums of the KV pass where its rows are shared by several workgroups; 0: none.
int64_t attn_f64_dkdv_workspace_bytes(int64_t T, int64_t G, int64_t D);

}  // namespace msa
