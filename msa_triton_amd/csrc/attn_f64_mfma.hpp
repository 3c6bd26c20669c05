// fp32 attention on FP64 matrix products (attn_f64_mfma.hip).
#pragma once
#include <initializer_list>

#include "common.hpp"

namespace msa {

// What the kernels take: every pass needs fitting dims and 16-byte aligned rows, the query
// passes (forward, dQ) also fitting heads per group.
bool attn_f64_dims_fit(int D, std::initializer_list<const void*> rows);
bool attn_f64_heads_fit(int R);

int attn_f64_fwd_launch(const float* q, const float* k, const float* v, const int32_t* idx, const int32_t* cu, int nseq,
                        int64_t T, int Hq, int G, int D, int K, int B, double scale, float* out, float* lse, double* rs,
                        float* o32, hipStream_t st);
int attn_f64_dq_launch(const float* q, const float* k, const float* v, const float* out, const float* dout, double* rs,
                       const int32_t* idx, const int32_t* cu, int nseq, int64_t T, int Hq, int G, int D, int K, int B,
                       double scale, float* dq, hipStream_t st);
int attn_f64_dkdv_launch(const float* q, const float* k, const float* v, const float* dout, const double* rs,
                         const int32_t* cu, const int32_t* cu_blocks, const int32_t* row_ptr, const int32_t* qidx,
                         int nseq, int64_t T, int Hq, int G, int D, int B, double scale, float* dk, float* dv, void* ws,
                         int64_t ws_bytes, hipStream_t st);

// FP64 partial sums of the KV pass where its rows are shared by several workgroups; 0: none.
int64_t attn_f64_dkdv_workspace_bytes(int64_t T, int64_t G, int64_t D);

}  // namespace msa
