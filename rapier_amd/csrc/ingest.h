// ingest.h - the wide-chunk launches of the engine's prompt ingest: the library's kernels over more columns than one
// entry-point call takes (16), with the bits of the single-column calls.
#pragma once

#include "rmi_common.h"

namespace rmi {

constexpr int kIngestColTile = 128;    // columns are padded to this tile
constexpr int kIngestMaxCols = 4096;

// packed Q6_K GEMM (ingest_gemm.hip): y[col][n_out] = W x_col (+ res, and the 4-row partials of y), bitwise the packed
// GEMV; ws: ingest_operand_bytes(n_in, ncols) bytes of scratch, 16-byte aligned
size_t ingest_operand_bytes(int n_in, int ncols);
int q6k_packed_gemm(const void* w_packed, const void* x_q8_1, float* y, const float* res, float* partials, int n_in,
                    int n_out, int ncols, void* ws, hipStream_t s);

// The column kernels of the entry points of the same names (epilogue.hip, attn.hip), for up to `limit` columns
int embed_cols(int type, const void* emb, const int* tokens, float* x, float* partials, int n_embd, int n_vocab,
               int ncols, int limit, hipStream_t s);
int embed_quant_pair_cols(int type, const void* emb, const int* tokens, const float* w0, const float* x1,
                          const float* w1, const float* partials1, void* y_q8_1, int cols, int n_vocab, float eps,
                          int ncols, int limit, hipStream_t s);
int rms_quant_cols(const float* x, const float* w, const float* partials, void* y_q8_1, int cols, float eps, int ncols,
                   int limit, hipStream_t s);
int rms_quant_self_cols(const float* x, const float* w, void* y_q8_1, int cols, float eps, int ncols, int limit,
                        hipStream_t s);
int rms_norm_out_cols(const float* x, const float* w, const float* partials, float* out, int out_stride,
                      float* out_partials, int cols, float eps, int ncols, int limit, hipStream_t s);
int swiglu_interleaved_cols(const float* up_gate, void* y_q8_1, int n, int ncols, int col_stride, int limit,
                            hipStream_t s);
int swiglu_cols(const float* up, const float* gate, void* y_q8_1, int n, int ncols, int col_stride, int limit,
                hipStream_t s);
int attn_prep_cols(const float* q3, int q3_stride, const float* qn, const float* kn, uint16_t* kcache,
                   uint16_t* vcache, const int* pos, float* qout, int n_head, int n_kv, int head_dim, int n_rot,
                   const rmi_rope_params* rope, float eps, int ntok, int limit, int max_ctx, hipStream_t s);

// split-K attention of ntok tokens at positions pos0 + t (pos: the same on the device, pos[t]), `per` tokens a launch
int flash_wide(const float* q, const uint16_t* kcache, const uint16_t* vcache, const int* pos, int pos0,
               const float* gate_src, int gate_stride, uint8_t* q8, int q8_stride, void* workspace, int per, int n_head,
               int n_kv, int head_dim, int ntok, int max_ctx, int nsub, float scale, hipStream_t s);
size_t flash_wide_bytes(int max_ctx, int n_head, int n_kv, int nsub, int per);

// one Gated-DeltaNet layer over ntok >= 3 tokens (gdn.hip): rmi_gdn_layer_tokens for more than 16 tokens, same bits;
// ws: gdn_wide_bytes
size_t gdn_wide_bytes(int h_k, int h_v, int ntok);
int gdn_wide(float* state_a, float* state_b, float* hist_a, float* hist_b, const int* sel, const float* qkvz,
             int stride, const float* ab, int ab_stride, const float* conv_w, const float* dt, const float* ssm_a,
             const float* gamma, float eps, float* y, uint8_t* q8, int q8_stride, int h_k, int h_v, int ntok, void* ws,
             hipStream_t s);

}  // namespace rmi
