// Host-side helpers shared by the launch code: error recording and kernel entry declarations.
#pragma once
#include <hip/hip_runtime.h>

#include "fa_common.hpp"

namespace fa {

// Records a printf-style message for flexattn_last_error_string() and returns `code`.
int set_error(int code, const char* fmt, ...);

// Returns FLEXATTN_OK, or records hipGetLastError() under `what`.
int check_launch(const char* what);

// bf16, head dim 128 (MFMA kernels)
int fwd_bf16_d128(const FwdArgs& a, hipStream_t stream);
int fwd_bf16_d64(const FwdArgs& a, hipStream_t stream);    // (same tiles as head dim 128; plain scores)
bool fwd_bf16_d64_ok(float sm_scale, int nk);
int fwd_bf16_d256(const FwdArgs& a, hipStream_t stream);   // (same tiles as head dim 128)
void fwd_bf16_d128_tile(int* bq, int* bk);
// the forward with scratch memory for split lists (0 bytes: nothing to split)
int64_t fwd_bf16_work_bytes(const FwdArgs& a, int D);
int fwd_bf16_with_work(const FwdArgs& a, int D, void* work, hipStream_t stream);
// few query rows against long keys, plain scores, no mask (head dim 64 or 128)
bool fwd_decode_ok(int dtype, int B, int Hq, int Hkv, int Sq, int Sk, int D);
int64_t fwd_decode_bytes(int B, int Hq, int Hkv, int Sq, int Sk, int D);
int fwd_decode(const FwdArgs& a, int D, void* work, hipStream_t stream);
int bwd_dq_bf16_d128(const BwdArgs& a, hipStream_t stream);
int bwd_dq_bf16_d64(const BwdArgs& a, hipStream_t stream);
bool bwd_dq_bf16_d64_ok(int nk);
int bwd_dq_bf16_d256(const BwdArgs& a, hipStream_t stream);
void bwd_dq_bf16_d128_tile(int* bq, int* bk);
int bwd_dkv_bf16_d128(const BwdArgs& a, hipStream_t stream);
int bwd_dkv_bf16_d64(const BwdArgs& a, hipStream_t stream);
int bwd_dkv_bf16_d256(const BwdArgs& a, hipStream_t stream);
// (the dk/dv pass of such a request runs the generated stream: its exported dS then lacks sm_scale and the soft-cap's
// factor 4; the kernel with a compiled main loop exports dS complete)
bool bwd_dkv_bf16_d128_on_stream(int kind, int flags, int nq, bool has_ab, int Hq, int Hkv);
void bwd_dkv_bf16_d128_tile(int* bq, int* bk);
// the gradient of a bias that several (batch, head) pairs share, in the bias's own shape; whether it is expected to beat the
// full-size gradient of the dk/dv pass and a sum over it
bool bwd_dab_bf16_pays(const BwdArgs& a);
int bwd_dab_bf16(const BwdArgs& a, hipStream_t stream);
// dq = out_scale dS K from the dS blocks that the dk/dv stream kernels wrote to a.ds (a.map: row lists at the
// dk/dv tiles)
int bwd_dq_from_ds(const BwdArgs& a, int D, float out_scale, hipStream_t stream);

// fp32, head dim 64 or 128 (FMA kernels, exact-arithmetic path)
int fwd_f32(const FwdArgs& a, int D, hipStream_t stream);
int bwd_dq_f32(const BwdArgs& a, int D, hipStream_t stream);
int bwd_dkv_f32(const BwdArgs& a, int D, hipStream_t stream);
void f32_tile(int* bq, int* bk);
// the same on the fp32 matrix cores (the default; FLEXATTN_FLAG_COMPILED_LOOP selects the FMA kernels)
int fwd_f32_mfma(const FwdArgs& a, int D, hipStream_t stream);
int bwd_dq_f32_mfma(const BwdArgs& a, int D, hipStream_t stream);
int bwd_dkv_f32_mfma(const BwdArgs& a, int D, hipStream_t stream);

int bwd_delta(const void* o, const void* dout, float* delta, int64_t rows, int D, int dtype, hipStream_t stream);

// (doc_batches: batch entries the mask's document arrays hold a row for; the map is the union over them)
int build_block_mask(const MaskArgs& mask, int doc_batches, int Sq, int Sk, int block_q, int block_k, uint8_t* state,
                     int* kv_cnt, int* kv_idx, int* q_cnt, int* q_idx, hipStream_t stream);

int build_ds_index(const uint8_t* state, const int* q_cnt, const int* q_idx, int nq, int nk, int* col, int* rank,
                   hipStream_t stream);

}  // namespace fa
