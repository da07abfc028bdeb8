// C-ABI entry points of the delta rule (DeltaNet / GatedDeltaNet), forward and backward.
// Dispatch: the chunked MFMA kernels (delta_rule_chunk.hip) take bf16, per-head beta,
// head_dim 64 .. 128 (a multiple of 8; zero-padded to 128 inside), seq >= 64 (forward and
// backward); every other case takes the row scans (delta_rule_row.hip, delta_rule_row_bwd.hip) or, by
// row_path() below, the exact per-step kernels (delta_rule_seq.hip).
#include "edf_abi.hpp"

#include <algorithm>

namespace edf {
size_t dr_seq_backward_workspace_bytes(int batch, int heads, int seq, int d);
size_t dr_seq_context_bytes(int batch, int heads, int seq, int d);
int dr_seq_run(void* stream, const void* q, const void* k, const void* v, const void* beta, const void* alpha,
               void* out, int batch, int seq, int heads, int d, int dtype, int beta_per_head, int alpha_per_row,
               float* context);
int dr_seq_backward_run(void* stream, const void* q, const void* k, const void* v, const void* beta,
                        const void* alpha, const void* grad_out, void* dq, void* dk, void* dv, void* dbeta,
                        void* dalpha, void* workspace, int batch, int seq, int heads, int d, int dtype,
                        int beta_per_head, int alpha_per_row, const float* context);
bool dr_row_takes(int batch, int heads, int seq, int d);
int dr_row_run(void* stream, const void* q, const void* k, const void* v, const void* beta, const void* alpha,
               void* out, int batch, int seq, int heads, int d, int dtype, int beta_per_head, int alpha_per_row,
               float* ckpt, float* err, int cw);
size_t dr_row_context_bytes(int batch, int heads, int seq, int d, bool decay);
int dr_row_record_run(void* stream, const void* q, const void* k, const void* v, const void* beta, const void* alpha,
                      void* out, int batch, int seq, int heads, int d, int dtype, int beta_per_head,
                      int alpha_per_row, void* context);
size_t dr_row_backward_workspace_bytes(int batch, int heads, int seq, int d, bool decay, bool saved);
int dr_row_backward_run(void* stream, const void* q, const void* k, const void* v, const void* beta,
                        const void* alpha, const void* grad_out, void* dq, void* dk, void* dv, void* dbeta,
                        void* dalpha, void* workspace, int batch, int seq, int heads, int d, int dtype,
                        int beta_per_head, int alpha_per_row, const void* context);
bool dr_chunk_eligible(int seq, int d, int dtype, int beta_per_head);
size_t dr_chunk_workspace_bytes(int batch, int seq, int heads, int d);
int dr_chunk_run(void* stream, const void* q, const void* k, const void* v, const void* beta, const void* alpha,
                 void* out, void* workspace, int batch, int seq, int heads, int d);
size_t dr_chunk_backward_workspace_bytes(int batch, int seq, int heads, int d);
size_t dr_chunk_saved_backward_workspace_bytes(int batch, int seq, int heads, int d);
int dr_chunk_saved_backward_run(void* stream, const void* q, const void* k, const void* v, const void* beta,
                                const void* alpha, const void* grad_out, void* dq, void* dk, void* dv, void* dbeta,
                                void* dalpha, const void* fwd_workspace, void* workspace, int batch, int seq,
                                int heads, int d);
int dr_chunk_backward_run(void* stream, const void* q, const void* k, const void* v, const void* beta,
                          const void* alpha, const void* grad_out, void* dq, void* dk, void* dv, void* dbeta,
                          void* dalpha, void* workspace, int batch, int seq, int heads, int d);

namespace {
int check_dr(int batch, int seq, int heads, int d, int dtype, int beta_mode) {
  EDF_REQUIRE(batch > 0 && seq > 0 && heads > 0 && d > 0, EDF_ERR_INVALID_ARG, "dimensions must be positive");
  EDF_REQUIRE(valid_dtype(dtype), EDF_ERR_INVALID_ARG, "dtype must be 0 (f32) or 1 (bf16)");
  EDF_REQUIRE(d <= 128, EDF_ERR_UNSUPPORTED, "head_dim %d > 128 unsupported", d);
  EDF_REQUIRE(beta_mode == EDF_BETA_PER_ELEMENT || beta_mode == EDF_BETA_PER_HEAD, EDF_ERR_INVALID_ARG,
              "unknown beta mode %d", beta_mode);
  return EDF_OK;
}

// Off the chunked path: the row scans, or the per-step kernels where they are the faster ones with the backward.  The
// row scans cost whole chunks of 16 steps, states at least 32 wide and a workgroup per 16 rows and per 16 (64) steps
// in the gradients; the per-step kernels a chain of steps.  bfloat16, us with gradients, per-step / row scans:
//                                      DeltaNet     GatedDeltaNet
//   one chunk     d 64,  8 heads x 16    17 / 22      18 / 23
//                 d 64,  512 x 16        51 / 44      56 / 39
//                 d 128, 128 x 16        53 / 34      55 / 39
//   narrow        d 16,  8 x 48, 64      22 / 25, 27 / 27    25 / 25, 31 / 27
//                 d 16,  128 x 128       48 / 36      58 / 55
//                 d 16,  512 x 256      109 / 118    125 / 208
//                 d 32,  8 x 32, 48      20 / 23, 27 / 24    22 / 24, 29 / 25
//                 d 32,  512 x 64, 128   60 / 37, 106 / 66   66 / 71, 120 / 119
// float32's row scans take up to a third longer than bfloat16's with a decay (their sums are split), so their lines
// lie further out.  Batch rows of (seq + 96) H d 4 >= 2 GiB, of either type, are past the row scans' byte offsets.
bool row_path(int batch, int heads, int seq, int d, int dtype, bool decay) {
  if (!dr_row_takes(batch, heads, seq, d)) return false;
  const long bh = (long)batch * heads;
  const bool f32 = dtype != EDF_BF16;
  if (d <= 16) return seq >= 64 && bh < (f32 && decay ? 128 : 256);
  if (seq <= 16) return f32 ? d > 64 && bh >= 128 && !decay : (d > 32 && bh >= 512) || (d > 64 && bh >= 128);
  if (d <= 32) return bh < 256 ? seq >= 48 : !decay || (!f32 && seq >= 128);
  return !(f32 && decay && bh < 128 && seq <= 32);
}
// A forward that keeps no record.  On a full grid of short sequences float32 row scans, which hold two or three
// workgroups per CU, are the slower ones although they win with the backward: DeltaNet 512 heads of d 128, 32 steps
// 54 us per-step, 72 row scans; GatedDeltaNet 58 and 88, at 128 steps 232 and 254.
bool row_forward(int batch, int heads, int seq, int d, int dtype, bool decay) {
  if (!row_path(batch, heads, seq, d, dtype, decay)) return false;
  return !(dtype != EDF_BF16 && (long)batch * heads * ((d + 15) / 16) >= 768 && seq < (decay ? 256 : 64));
}

// The record of a forward and the workspace of a backward; saved: with the forward's record at hand.
size_t unchunked_context_bytes(int batch, int heads, int seq, int d, int dtype, bool decay) {
  return row_path(batch, heads, seq, d, dtype, decay) ? dr_row_context_bytes(batch, heads, seq, d, decay)
                                               : dr_seq_context_bytes(batch, heads, seq, d);
}
size_t unchunked_backward_bytes(int batch, int heads, int seq, int d, int dtype, bool decay, bool saved) {
  return row_path(batch, heads, seq, d, dtype, decay) ? dr_row_backward_workspace_bytes(batch, heads, seq, d, decay, saved)
                                               : dr_seq_backward_workspace_bytes(batch, heads, seq, d);
}
// What serves a call with a decay and one without: the queries that do not say which.
size_t any_context_bytes(int batch, int heads, int seq, int d, int dtype) {
  return std::max(unchunked_context_bytes(batch, heads, seq, d, dtype, false),
                  unchunked_context_bytes(batch, heads, seq, d, dtype, true));
}
size_t any_backward_bytes(int batch, int heads, int seq, int d, int dtype) {
  return std::max(unchunked_backward_bytes(batch, heads, seq, d, dtype, false, false),
                  unchunked_backward_bytes(batch, heads, seq, d, dtype, true, false));
}

int unchunked_fwd(void* stream, const void* q, const void* k, const void* v, const void* beta, const void* alpha,
                  void* out, int batch, int seq, int heads, int d, int dtype, int beta_per_head, int alpha_per_row,
                  void* context) {
  const bool decay = alpha != nullptr;
  if (context != nullptr && row_path(batch, heads, seq, d, dtype, decay))
    return dr_row_record_run(stream, q, k, v, beta, alpha, out, batch, seq, heads, d, dtype, beta_per_head,
                             alpha_per_row, context);
  if (context == nullptr && row_forward(batch, heads, seq, d, dtype, decay))
    return dr_row_run(stream, q, k, v, beta, alpha, out, batch, seq, heads, d, dtype, beta_per_head, alpha_per_row,
                      nullptr, nullptr, 0);
  return dr_seq_run(stream, q, k, v, beta, alpha, out, batch, seq, heads, d, dtype, beta_per_head, alpha_per_row,
                    (float*)context);
}

// context null: the record is recomputed
int unchunked_bwd(void* stream, const void* q, const void* k, const void* v, const void* beta, const void* alpha,
                  const void* grad_out, void* dq, void* dk, void* dv, void* dbeta, void* dalpha, void* workspace,
                  int batch, int seq, int heads, int d, int dtype, int beta_per_head, int alpha_per_row,
                  const void* context) {
  if (row_path(batch, heads, seq, d, dtype, alpha != nullptr))
    return dr_row_backward_run(stream, q, k, v, beta, alpha, grad_out, dq, dk, dv, dbeta, dalpha, workspace, batch,
                               seq, heads, d, dtype, beta_per_head, alpha_per_row, context);
  return dr_seq_backward_run(stream, q, k, v, beta, alpha, grad_out, dq, dk, dv, dbeta, dalpha, workspace, batch, seq,
                             heads, d, dtype, beta_per_head, alpha_per_row, (const float*)context);
}

int fwd(void* stream, const void* q, const void* k, const void* v, const void* beta, const void* alpha, void* out,
        void* workspace, size_t ws_bytes, int batch, int seq, int heads, int d, int dtype, int beta_mode) {
  int rc = check_dr(batch, seq, heads, d, dtype, beta_mode);
  if (rc) return rc;
  EDF_REQUIRE(q && k && v && beta && out, EDF_ERR_INVALID_ARG, "null tensor pointer");
  const int per_head = beta_mode == EDF_BETA_PER_HEAD;
  if (dr_chunk_eligible(seq, d, dtype, per_head)) {
    // As the backward: a missing or short workspace is the caller's error, not a reason to
    // run the (exact-state, ~10x slower) per-step kernels with different numerics.
    const size_t need = dr_chunk_workspace_bytes(batch, seq, heads, d);
    EDF_REQUIRE(workspace && ws_bytes >= need, EDF_ERR_WORKSPACE, "workspace too small: need %zu bytes", need);
    return dr_chunk_run(stream, q, k, v, beta, alpha, out, workspace, batch, seq, heads, d);
  }
  // a workspace of edf_delta_rule_forward_context_bytes() (optional) also receives what the saved
  // backward reads
  const bool keep = workspace && ws_bytes >= unchunked_context_bytes(batch, heads, seq, d, dtype, alpha != nullptr);
  return unchunked_fwd(stream, q, k, v, beta, alpha, out, batch, seq, heads, d, dtype, per_head, 0,
                       keep ? workspace : nullptr);
}

int bwd(void* stream, const void* q, const void* k, const void* v, const void* beta, const void* alpha,
        const void* grad_out, void* dq, void* dk, void* dv, void* dbeta, void* dalpha, void* workspace,
        size_t ws_bytes, int batch, int seq, int heads, int d, int dtype, int beta_mode) {
  int rc = check_dr(batch, seq, heads, d, dtype, beta_mode);
  if (rc) return rc;
  EDF_REQUIRE(q && k && v && beta && grad_out && dq && dk && dv && dbeta, EDF_ERR_INVALID_ARG,
              "null tensor pointer");
  const int per_head = beta_mode == EDF_BETA_PER_HEAD;
  if (dr_chunk_eligible(seq, d, dtype, per_head)) {
    const size_t need = dr_chunk_backward_workspace_bytes(batch, seq, heads, d);
    EDF_REQUIRE(workspace && ws_bytes >= need, EDF_ERR_WORKSPACE, "workspace too small: need %zu bytes", need);
    return dr_chunk_backward_run(stream, q, k, v, beta, alpha, grad_out, dq, dk, dv, dbeta, dalpha, workspace, batch,
                                 seq, heads, d);
  }
  const size_t need = unchunked_backward_bytes(batch, heads, seq, d, dtype, alpha != nullptr, false);
  EDF_REQUIRE(workspace && ws_bytes >= need, EDF_ERR_WORKSPACE, "workspace too small: need %zu bytes", need);
  return unchunked_bwd(stream, q, k, v, beta, alpha, grad_out, dq, dk, dv, dbeta, dalpha, workspace, batch, seq, heads,
                       d, dtype, per_head, 0, nullptr);
}
int bwd_saved(void* stream, const void* q, const void* k, const void* v, const void* beta, const void* alpha,
              const void* grad_out, void* dq, void* dk, void* dv, void* dbeta, void* dalpha, const void* fwd_ws,
              size_t fwd_ws_bytes, void* workspace, size_t ws_bytes, int batch, int seq, int heads, int d, int dtype,
              int beta_mode) {
  int rc = check_dr(batch, seq, heads, d, dtype, beta_mode);
  if (rc) return rc;
  EDF_REQUIRE(q && k && v && beta && grad_out && dq && dk && dv && dbeta, EDF_ERR_INVALID_ARG,
              "null tensor pointer");
  EDF_REQUIRE((alpha == nullptr) == (dalpha == nullptr), EDF_ERR_INVALID_ARG,
              "alpha and grad_alpha must both be given (gated) or both be null");
  const int per_head = beta_mode == EDF_BETA_PER_HEAD;
  if (dr_chunk_eligible(seq, d, dtype, per_head)) {
    const size_t need_f = dr_chunk_workspace_bytes(batch, seq, heads, d);
    EDF_REQUIRE(fwd_ws && fwd_ws_bytes >= need_f, EDF_ERR_WORKSPACE,
                "forward workspace too small: need the %zu bytes the forward filled", need_f);
    const size_t need = dr_chunk_saved_backward_workspace_bytes(batch, seq, heads, d);
    EDF_REQUIRE(workspace && ws_bytes >= need, EDF_ERR_WORKSPACE, "workspace too small: need %zu bytes", need);
    return dr_chunk_saved_backward_run(stream, q, k, v, beta, alpha, grad_out, dq, dk, dv, dbeta, dalpha, fwd_ws,
                                       workspace, batch, seq, heads, d);
  }
  // the forward's record when its workspace held one, else the backward recomputes it
  const bool saved = fwd_ws && fwd_ws_bytes >= unchunked_context_bytes(batch, heads, seq, d, dtype, alpha != nullptr);
  const size_t need = unchunked_backward_bytes(batch, heads, seq, d, dtype, alpha != nullptr, saved);
  EDF_REQUIRE(workspace && ws_bytes >= need, EDF_ERR_WORKSPACE, "workspace too small: need %zu bytes", need);
  return unchunked_bwd(stream, q, k, v, beta, alpha, grad_out, dq, dk, dv, dbeta, dalpha, workspace, batch, seq, heads,
                       d, dtype, per_head, 0, saved ? fwd_ws : nullptr);
}
}  // namespace
}  // namespace edf

extern "C" {

size_t edf_delta_rule_saved_backward_workspace_bytes(int batch, int seq_len, int num_heads, int head_dim, int dtype,
                                                     int beta_mode) {
  if (batch <= 0 || seq_len <= 0 || num_heads <= 0 || head_dim <= 0) return 0;
  if (edf::dr_chunk_eligible(seq_len, head_dim, dtype, beta_mode == EDF_BETA_PER_HEAD))
    return edf::dr_chunk_saved_backward_workspace_bytes(batch, seq_len, num_heads, head_dim);
  return edf::any_backward_bytes(batch, num_heads, seq_len, head_dim, dtype);
}

int edf_fused_delta_rule_scan_backward_saved(void* stream, const void* q, const void* k, const void* v,
                                             const void* beta, const void* alpha, const void* grad_out,
                                             void* grad_q, void* grad_k, void* grad_v, void* grad_beta,
                                             void* grad_alpha, const void* forward_workspace,
                                             size_t forward_workspace_bytes, void* workspace, size_t workspace_bytes,
                                             int batch, int seq_len, int num_heads, int head_dim, int dtype,
                                             int beta_mode) {
  return edf::bwd_saved(stream, q, k, v, beta, alpha, grad_out, grad_q, grad_k, grad_v, grad_beta, grad_alpha,
                        forward_workspace, forward_workspace_bytes, workspace, workspace_bytes, batch, seq_len,
                        num_heads, head_dim, dtype, beta_mode);
}

size_t edf_delta_rule_context_bytes(int batch, int seq_len, int num_heads, int head_dim, int dtype, int beta_mode,
                                    int has_alpha) {
  if (batch <= 0 || seq_len <= 0 || num_heads <= 0 || head_dim <= 0 || head_dim > 128) return 0;
  if (edf::dr_chunk_eligible(seq_len, head_dim, dtype, beta_mode == EDF_BETA_PER_HEAD))
    return edf::dr_chunk_workspace_bytes(batch, seq_len, num_heads, head_dim);
  return edf::unchunked_context_bytes(batch, num_heads, seq_len, head_dim, dtype, has_alpha != 0);
}

size_t edf_delta_rule_context_backward_workspace_bytes(int batch, int seq_len, int num_heads, int head_dim, int dtype,
                                                       int beta_mode, int has_alpha) {
  if (batch <= 0 || seq_len <= 0 || num_heads <= 0 || head_dim <= 0) return 0;
  if (edf::dr_chunk_eligible(seq_len, head_dim, dtype, beta_mode == EDF_BETA_PER_HEAD))
    return edf::dr_chunk_saved_backward_workspace_bytes(batch, seq_len, num_heads, head_dim);
  return edf::unchunked_backward_bytes(batch, num_heads, seq_len, head_dim, dtype, has_alpha != 0, true);
}

size_t edf_delta_rule_forward_context_bytes(int batch, int seq_len, int num_heads, int head_dim, int dtype,
                                            int beta_mode) {
  if (batch <= 0 || seq_len <= 0 || num_heads <= 0 || head_dim <= 0 || head_dim > 128) return 0;
  if (edf::dr_chunk_eligible(seq_len, head_dim, dtype, beta_mode == EDF_BETA_PER_HEAD))
    return edf::dr_chunk_workspace_bytes(batch, seq_len, num_heads, head_dim);
  return edf::any_context_bytes(batch, num_heads, seq_len, head_dim, dtype);
}

size_t edf_delta_rule_workspace_bytes(int batch, int seq_len, int num_heads, int head_dim, int dtype,
                                      int beta_mode) {
  if (batch <= 0 || seq_len <= 0 || num_heads <= 0 || head_dim <= 0) return 0;
  if (edf::dr_chunk_eligible(seq_len, head_dim, dtype, beta_mode == EDF_BETA_PER_HEAD))
    return edf::dr_chunk_workspace_bytes(batch, seq_len, num_heads, head_dim);
  return 0;
}

size_t edf_delta_rule_backward_workspace_bytes(int batch, int seq_len, int num_heads, int head_dim, int dtype,
                                               int beta_mode) {
  if (batch <= 0 || seq_len <= 0 || num_heads <= 0 || head_dim <= 0) return 0;
  if (edf::dr_chunk_eligible(seq_len, head_dim, dtype, beta_mode == EDF_BETA_PER_HEAD))
    return edf::dr_chunk_backward_workspace_bytes(batch, seq_len, num_heads, head_dim);
  return edf::any_backward_bytes(batch, num_heads, seq_len, head_dim, dtype);
}

int edf_fused_delta_net_scan(void* stream, const void* q, const void* k, const void* v, const void* beta, void* out,
                             void* workspace, size_t workspace_bytes, int batch, int seq_len, int num_heads,
                             int head_dim, int dtype, int beta_mode) {
  return edf::fwd(stream, q, k, v, beta, nullptr, out, workspace, workspace_bytes, batch, seq_len, num_heads,
                  head_dim, dtype, beta_mode);
}

int edf_fused_gated_delta_net_scan(void* stream, const void* q, const void* k, const void* v, const void* beta,
                                   const void* alpha, void* out, void* workspace, size_t workspace_bytes, int batch,
                                   int seq_len, int num_heads, int head_dim, int dtype, int beta_mode) {
  EDF_REQUIRE(alpha != nullptr, EDF_ERR_INVALID_ARG, "null alpha pointer");
  return edf::fwd(stream, q, k, v, beta, alpha, out, workspace, workspace_bytes, batch, seq_len, num_heads,
                  head_dim, dtype, beta_mode);
}

int edf_fused_delta_rule_scan_backward(void* stream, const void* q, const void* k, const void* v, const void* beta,
                                       const void* forward_out, const void* grad_out, void* grad_q, void* grad_k,
                                       void* grad_v, void* grad_beta, void* workspace, size_t workspace_bytes,
                                       int batch, int seq_len, int num_heads, int head_dim, int dtype,
                                       int beta_mode) {
  (void)forward_out;  // accepted for signature parity; the reference never reads it either
  return edf::bwd(stream, q, k, v, beta, nullptr, grad_out, grad_q, grad_k, grad_v, grad_beta, nullptr, workspace,
                  workspace_bytes, batch, seq_len, num_heads, head_dim, dtype, beta_mode);
}

int edf_fused_gated_delta_net_scan_backward(void* stream, const void* q, const void* k, const void* v,
                                            const void* beta, const void* alpha, const void* forward_out,
                                            const void* grad_out, void* grad_q, void* grad_k, void* grad_v,
                                            void* grad_beta, void* grad_alpha, void* workspace,
                                            size_t workspace_bytes, int batch, int seq_len, int num_heads,
                                            int head_dim, int dtype, int beta_mode) {
  (void)forward_out;
  EDF_REQUIRE(alpha != nullptr && grad_alpha != nullptr, EDF_ERR_INVALID_ARG, "null alpha / grad_alpha pointer");
  return edf::bwd(stream, q, k, v, beta, alpha, grad_out, grad_q, grad_k, grad_v, grad_beta, grad_alpha, workspace,
                  workspace_bytes, batch, seq_len, num_heads, head_dim, dtype, beta_mode);
}

// KDA: per-row log-space decay, per-head beta; never the chunked kernels (which take one decay per head).
size_t edf_kda_scan_backward_workspace_bytes(int batch, int seq_len, int num_heads, int head_dim, int dtype) {
  if (batch <= 0 || seq_len <= 0 || num_heads <= 0 || head_dim <= 0) return 0;
  return edf::unchunked_backward_bytes(batch, num_heads, seq_len, head_dim, dtype, true, false);
}

int edf_fused_kda_scan(void* stream, const void* q, const void* k, const void* v, const void* alpha,
                       const void* beta, void* out, int batch, int seq_len, int num_heads, int head_dim, int dtype) {
  int rc = edf::check_dr(batch, seq_len, num_heads, head_dim, dtype, EDF_BETA_PER_HEAD);
  if (rc) return rc;
  EDF_REQUIRE(q && k && v && alpha && beta && out, EDF_ERR_INVALID_ARG, "null tensor pointer");
  return edf::unchunked_fwd(stream, q, k, v, beta, alpha, out, batch, seq_len, num_heads, head_dim, dtype, 1, 1,
                         nullptr);
}

int edf_fused_kda_scan_backward(void* stream, const void* q, const void* k, const void* v, const void* alpha,
                                const void* beta, const void* forward_out, const void* grad_out, void* grad_q,
                                void* grad_k, void* grad_v, void* grad_alpha, void* grad_beta, void* workspace,
                                size_t workspace_bytes, int batch, int seq_len, int num_heads, int head_dim,
                                int dtype) {
  (void)forward_out;
  int rc = edf::check_dr(batch, seq_len, num_heads, head_dim, dtype, EDF_BETA_PER_HEAD);
  if (rc) return rc;
  EDF_REQUIRE(q && k && v && alpha && beta && grad_out && grad_q && grad_k && grad_v && grad_alpha && grad_beta,
              EDF_ERR_INVALID_ARG, "null tensor pointer");
  const size_t need = edf::unchunked_backward_bytes(batch, num_heads, seq_len, head_dim, dtype, true, false);
  EDF_REQUIRE(workspace && workspace_bytes >= need, EDF_ERR_WORKSPACE, "workspace too small: need %zu bytes", need);
  return edf::unchunked_bwd(stream, q, k, v, beta, alpha, grad_out, grad_q, grad_k, grad_v, grad_beta,
                                  grad_alpha, workspace, batch, seq_len, num_heads, head_dim, dtype, 1, 1, nullptr);
}

size_t edf_kda_scan_context_backward_workspace_bytes(int batch, int seq_len, int num_heads, int head_dim, int dtype) {
  if (batch <= 0 || seq_len <= 0 || num_heads <= 0 || head_dim <= 0) return 0;
  return edf::unchunked_backward_bytes(batch, num_heads, seq_len, head_dim, dtype, true, true);
}

size_t edf_kda_scan_context_bytes(int batch, int seq_len, int num_heads, int head_dim, int dtype) {
  if (batch <= 0 || seq_len <= 0 || num_heads <= 0 || head_dim <= 0 || head_dim > 128) return 0;
  return edf::unchunked_context_bytes(batch, num_heads, seq_len, head_dim, dtype, true);
}

int edf_fused_kda_scan_with_context(void* stream, const void* q, const void* k, const void* v, const void* alpha,
                                    const void* beta, void* out, void* context, size_t context_bytes, int batch,
                                    int seq_len, int num_heads, int head_dim, int dtype) {
  int rc = edf::check_dr(batch, seq_len, num_heads, head_dim, dtype, EDF_BETA_PER_HEAD);
  if (rc) return rc;
  EDF_REQUIRE(q && k && v && alpha && beta && out, EDF_ERR_INVALID_ARG, "null tensor pointer");
  const size_t need = edf::unchunked_context_bytes(batch, num_heads, seq_len, head_dim, dtype, true);
  EDF_REQUIRE(context && context_bytes >= need, EDF_ERR_WORKSPACE, "context too small: need %zu bytes", need);
  return edf::unchunked_fwd(stream, q, k, v, beta, alpha, out, batch, seq_len, num_heads, head_dim, dtype, 1, 1,
                         context);
}

int edf_fused_kda_scan_backward_saved(void* stream, const void* q, const void* k, const void* v, const void* alpha,
                                      const void* beta, const void* grad_out, void* grad_q, void* grad_k,
                                      void* grad_v, void* grad_alpha, void* grad_beta, const void* context,
                                      size_t context_bytes, void* workspace, size_t workspace_bytes, int batch,
                                      int seq_len, int num_heads, int head_dim, int dtype) {
  int rc = edf::check_dr(batch, seq_len, num_heads, head_dim, dtype, EDF_BETA_PER_HEAD);
  if (rc) return rc;
  EDF_REQUIRE(q && k && v && alpha && beta && grad_out && grad_q && grad_k && grad_v && grad_alpha && grad_beta,
              EDF_ERR_INVALID_ARG, "null tensor pointer");
  const size_t needc = edf::unchunked_context_bytes(batch, num_heads, seq_len, head_dim, dtype, true);
  EDF_REQUIRE(context && context_bytes >= needc, EDF_ERR_WORKSPACE,
              "context too small: need the %zu bytes the forward filled", needc);
  const size_t need = edf::unchunked_backward_bytes(batch, num_heads, seq_len, head_dim, dtype, true, true);
  EDF_REQUIRE(workspace && workspace_bytes >= need, EDF_ERR_WORKSPACE, "workspace too small: need %zu bytes", need);
  return edf::unchunked_bwd(stream, q, k, v, beta, alpha, grad_out, grad_q, grad_k, grad_v, grad_beta,
                                  grad_alpha, workspace, batch, seq_len, num_heads, head_dim, dtype, 1, 1,
                                  context);
}

}  // extern "C"
