// Validation and dispatch for the matrix-product entry points.
#include <algorithm>

#include "common.h"

namespace spiral {
int64_t gemv_max_k(int type, bool exact);
int gemv(int type, const void* w, int64_t n_rows, int64_t k, const uint16_t* x, void* y, int y_type, bool exact,
         hipStream_t s);
int64_t gemm_min_workspace_bytes(int64_t m, int64_t k);
int64_t gemm_workspace_bytes(int64_t m, int64_t n_rows, int64_t k);
int64_t gemm_max_k();
int gemm(int type, const void* w, int64_t n_rows, int64_t k, const uint16_t* x, int64_t ldx, int64_t m,
         void* y, int y_type, int64_t ldy, void* workspace, int64_t workspace_bytes, hipStream_t s);
bool dense_fits(int type, int64_t n_rows, int64_t k, int64_t m, int64_t ldx, bool f32);
int64_t dense_workspace_bytes(int64_t n_rows, int64_t k);
int gemm_dense(int type, const void* w, int64_t n_rows, int64_t k, const uint16_t* x, int64_t ldx, int64_t m, void* y,
               int y_type, int64_t ldy, void* workspace, hipStream_t s);
bool skinny_fits(int type, int64_t n_rows, int64_t k, int64_t m);
int skinny(int type, const void* w, int64_t n_rows, int64_t k, const uint16_t* x, int64_t ldx, int64_t m, void* y,
           int y_type, int64_t ldy, hipStream_t s);
int64_t moe_workspace_bytes(int64_t n_expert, int64_t n_pairs);
int moe(int type, const void* w, int64_t expert_stride, int64_t n_expert, int64_t n_rows, int64_t k,
        const uint16_t* x, int64_t x_slots, const int32_t* ids, int64_t n_tokens, int64_t top_k, void* y,
        int y_type, int glu_op, int swapped, void* workspace, hipStream_t s, const void* w_up = nullptr);
int glu(int op, int swapped, const float* x, int64_t ldx, int64_t n, int64_t rows, float* y, int64_t ldy,
        hipStream_t s, float alpha, float limit, uint16_t* copy);
int glu_split(int op, int swapped, const float* xg, int64_t ldg, const float* xu, int64_t ldu, int64_t n,
              int64_t rows, float* y, int64_t ldy, hipStream_t s, float alpha, float limit, uint16_t* copy);
bool moe_glu_fits_k(int64_t k);
void* moe_static_scratch(int& rc);

bool glu_op_ok(int op) {
  return op == SPIRAL_GLU_REGLU || op == SPIRAL_GLU_GEGLU || op == SPIRAL_GLU_SWIGLU ||
         op == SPIRAL_GLU_GEGLU_ERF || op == SPIRAL_GLU_GEGLU_QUICK;
}

// Products that need no workspace: the GEMV and the small-batch form.
bool runs_direct(int type, int64_t n_rows, int64_t k, int64_t m) {
  return (m == 1 && k <= gemv_max_k(type, true)) || skinny_fits(type, n_rows, k, m);
}

// The least workspace a call takes is the fused GEMM's; the forms that want more
// run when the caller's workspace holds it.
int64_t mul_mat_least_workspace(int type, int64_t n_rows, int64_t k, int64_t m) {
  return runs_direct(type, n_rows, k, m) ? 0 : gemm_min_workspace_bytes(m, k);
}

// Checks shared by MUL_MAT_ID and its fused GLU form.
int check_mul_mat_id(int type, const void* w, int64_t expert_stride, int64_t n_expert, int64_t n_rows, int64_t k,
                     const uint16_t* x, int64_t x_slots, const int32_t* ids, int64_t n_tokens, int64_t top_k,
                     void* y, int y_type, void* workspace, int64_t workspace_bytes) {
  if (!is_quant_type(type)) return SPIRAL_ERR_TYPE;
  if (y_type != SPIRAL_TYPE_BF16 && y_type != SPIRAL_TYPE_F32) return SPIRAL_ERR_TYPE;
  if (w == nullptr || x == nullptr || ids == nullptr || y == nullptr || workspace == nullptr)
    return SPIRAL_ERR_NULL;
  if (n_expert <= 0 || n_rows <= 0 || k <= 0 || k % block_elems(type) != 0 || n_tokens < 0 || top_k <= 0)
    return SPIRAL_ERR_SHAPE;
  if (x_slots != 1 && x_slots != top_k) return SPIRAL_ERR_SHAPE;
  const int64_t matrix_bytes = spiral_tensor_bytes(type, n_rows, k);
  if (matrix_bytes == 0 || expert_stride < matrix_bytes || expert_stride % 16 != 0) return SPIRAL_ERR_SHAPE;
  int64_t pairs = 0;
  if (n_expert > INT32_MAX || __builtin_mul_overflow(n_tokens, top_k, &pairs) || pairs > INT32_MAX)
    return SPIRAL_ERR_SHAPE;
  if (workspace_bytes < moe_workspace_bytes(n_expert, pairs)) return SPIRAL_ERR_CAPACITY;
  if (!aligned16(w) || !aligned16(x) || k % 8 != 0) return SPIRAL_ERR_ALIGN;
  if ((reinterpret_cast<uintptr_t>(y) & 3u) != 0 || (reinterpret_cast<uintptr_t>(workspace) & 3u) != 0)
    return SPIRAL_ERR_ALIGN;
  return SPIRAL_OK;
}
}  // namespace spiral

using namespace spiral;

extern "C" {

int64_t spiral_mul_mat_workspace_bytes(int type, int64_t n_rows, int64_t k, int64_t m) {
  if (!is_quant_type(type) || n_rows <= 0 || m <= 0 || k <= 0 || k % block_elems(type) != 0) return 0;
  if (runs_direct(type, n_rows, k, m)) return 0;
  const int64_t need = gemm_workspace_bytes(m, n_rows, k);  // 0 past the GEMM's longest row: spiral_mul_mat refuses that shape
  const bool dense = need > 0 && (dense_fits(type, n_rows, k, m, k, false) || dense_fits(type, n_rows, k, m, k, true));
  return dense ? std::max(need, dense_workspace_bytes(n_rows, k)) : need;
}

int spiral_mul_mat(int type, const void* w, int64_t n_rows, int64_t k, const uint16_t* x, int64_t ldx,
                   int64_t m, void* y, int y_type, int64_t ldy, void* workspace, int64_t workspace_bytes,
                   void* stream) {
  if (!is_quant_type(type)) return SPIRAL_ERR_TYPE;
  if (y_type != SPIRAL_TYPE_BF16 && y_type != SPIRAL_TYPE_F32) return SPIRAL_ERR_TYPE;
  if (w == nullptr || x == nullptr || y == nullptr) return SPIRAL_ERR_NULL;
  if (n_rows <= 0 || m <= 0 || k <= 0 || k % block_elems(type) != 0) return SPIRAL_ERR_SHAPE;
  if (ldx < k || ldy < n_rows || spiral_tensor_bytes(type, n_rows, k) == 0) return SPIRAL_ERR_SHAPE;
  if (!aligned16(w) || !aligned16(x) || ldx % 8 != 0) return SPIRAL_ERR_ALIGN;
  if ((reinterpret_cast<uintptr_t>(y) & 3u) != 0) return SPIRAL_ERR_ALIGN;
  const bool direct = runs_direct(type, n_rows, k, m);
  if (!direct && k > gemm_max_k()) return SPIRAL_ERR_SHAPE;
  const int64_t need = mul_mat_least_workspace(type, n_rows, k, m);
  if (need > 0) {
    if (workspace == nullptr) return SPIRAL_ERR_NULL;
    if (workspace_bytes < need) return SPIRAL_ERR_CAPACITY;
    if (!aligned16(workspace)) return SPIRAL_ERR_ALIGN;
  }
  int rc = require_device();
  if (rc != SPIRAL_OK) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (direct) {
    if (m == 1 && k <= gemv_max_k(type, true)) return gemv(type, w, n_rows, k, x, y, y_type, true, s);
    return skinny(type, w, n_rows, k, x, ldx, m, y, y_type, ldy, s);
  }
  if (dense_fits(type, n_rows, k, m, ldx, y_type == SPIRAL_TYPE_F32) &&
      workspace_bytes >= dense_workspace_bytes(n_rows, k))
    return gemm_dense(type, w, n_rows, k, x, ldx, m, y, y_type, ldy, workspace, s);
  return gemm(type, w, n_rows, k, x, ldx, m, y, y_type, ldy, workspace, workspace_bytes, s);
}

int64_t spiral_gemv_relaxed_max_k(int type) { return is_quant_type(type) ? gemv_max_k(type, false) : 0; }

int spiral_gemv_relaxed(int type, const void* w, int64_t n_rows, int64_t k, const uint16_t* x, void* y, int y_type,
                        void* stream) {
  if (!is_quant_type(type)) return SPIRAL_ERR_TYPE;
  if (y_type != SPIRAL_TYPE_BF16 && y_type != SPIRAL_TYPE_F32) return SPIRAL_ERR_TYPE;
  if (w == nullptr || x == nullptr || y == nullptr) return SPIRAL_ERR_NULL;
  if (n_rows <= 0 || k <= 0 || k % block_elems(type) != 0 || k > gemv_max_k(type, false)) return SPIRAL_ERR_SHAPE;
  if (spiral_tensor_bytes(type, n_rows, k) == 0) return SPIRAL_ERR_SHAPE;
  if (!aligned16(w) || !aligned16(x)) return SPIRAL_ERR_ALIGN;
  if ((reinterpret_cast<uintptr_t>(y) & 3u) != 0) return SPIRAL_ERR_ALIGN;
  const int rc = require_device();
  if (rc != SPIRAL_OK) return rc;
  return gemv(type, w, n_rows, k, x, y, y_type, false, static_cast<hipStream_t>(stream));
}

int64_t spiral_mul_mat_id_workspace_bytes(int64_t n_expert, int64_t n_tokens, int64_t top_k) {
  int64_t pairs = 0;
  if (n_expert <= 0 || n_tokens < 0 || top_k <= 0 || n_expert > INT32_MAX ||
      __builtin_mul_overflow(n_tokens, top_k, &pairs) || pairs > INT32_MAX)
    return 0;  // a shape spiral_mul_mat_id refuses
  return moe_workspace_bytes(n_expert, pairs);
}

int spiral_mul_mat_id(int type, const void* w, int64_t expert_stride, int64_t n_expert, int64_t n_rows,
                      int64_t k, const uint16_t* x, int64_t x_slots, const int32_t* ids, int64_t n_tokens,
                      int64_t top_k, void* y, int y_type, void* workspace, int64_t workspace_bytes,
                      void* stream) {
  if (n_tokens == 0 && is_quant_type(type) && (y_type == SPIRAL_TYPE_BF16 || y_type == SPIRAL_TYPE_F32))
    return SPIRAL_OK;
  int rc = check_mul_mat_id(type, w, expert_stride, n_expert, n_rows, k, x, x_slots, ids, n_tokens, top_k, y, y_type,
                            workspace, workspace_bytes);
  if (rc != SPIRAL_OK) return rc;
  rc = require_device();
  if (rc != SPIRAL_OK) return rc;
  return moe(type, w, expert_stride, n_expert, n_rows, k, x, x_slots, ids, n_tokens, top_k, y, y_type, -1, 0,
             workspace, static_cast<hipStream_t>(stream));
}

int spiral_mul_mat_id_noalloc(int type, const void* w, int64_t expert_stride, int64_t n_expert, int64_t n_rows,
                              int64_t k, const uint16_t* x, int64_t x_slots, const int32_t* ids, int64_t n_tokens,
                              int64_t top_k, void* y, int y_type, void* stream) {
  if (n_tokens == 0 && is_quant_type(type) && (y_type == SPIRAL_TYPE_BF16 || y_type == SPIRAL_TYPE_F32))
    return SPIRAL_OK;
  // Validated as spiral_mul_mat_id with a stand-in workspace of the static
  // array's size (never dereferenced here); the real address comes after.
  static uint32_t probe_ws[4];
  int rc = check_mul_mat_id(type, w, expert_stride, n_expert, n_rows, k, x, x_slots, ids, n_tokens, top_k, y, y_type,
                            probe_ws, SPIRAL_MUL_MAT_ID_STATIC_BYTES);
  if (rc != SPIRAL_OK) return rc;
  rc = require_device();
  if (rc != SPIRAL_OK) return rc;
  void* ws = moe_static_scratch(rc);
  if (rc != SPIRAL_OK) return rc;
  return moe(type, w, expert_stride, n_expert, n_rows, k, x, x_slots, ids, n_tokens, top_k, y, y_type, -1, 0, ws,
             static_cast<hipStream_t>(stream));
}

int spiral_mul_mat_id_glu_fits(int type, int64_t n_rows, int64_t k) {
  if (!is_quant_type(type) || n_rows <= 0 || n_rows % 2 != 0 || k <= 0 || k % block_elems(type) != 0) return 0;
  return moe_glu_fits_k(k) ? 1 : 0;
}

int spiral_mul_mat_id_glu(int type, const void* w, int64_t expert_stride, int64_t n_expert, int64_t n_rows,
                          int64_t k, const uint16_t* x, int64_t x_slots, const int32_t* ids, int64_t n_tokens,
                          int64_t top_k, int glu_op, int swapped, void* y, int y_type, void* workspace,
                          int64_t workspace_bytes, void* stream) {
  if (!glu_op_ok(glu_op) || (swapped != 0 && swapped != 1)) return SPIRAL_ERR_TYPE;
  if (n_tokens == 0 && is_quant_type(type) && (y_type == SPIRAL_TYPE_BF16 || y_type == SPIRAL_TYPE_F32))
    return SPIRAL_OK;
  int rc = check_mul_mat_id(type, w, expert_stride, n_expert, n_rows, k, x, x_slots, ids, n_tokens, top_k, y, y_type,
                            workspace, workspace_bytes);
  if (rc != SPIRAL_OK) return rc;
  if (n_rows % 2 != 0) return SPIRAL_ERR_SHAPE;
  rc = require_device();
  if (rc != SPIRAL_OK) return rc;
  return moe(type, w, expert_stride, n_expert, n_rows, k, x, x_slots, ids, n_tokens, top_k, y, y_type, glu_op,
             swapped, workspace, static_cast<hipStream_t>(stream));
}

int spiral_mul_mat_id_glu_split(int type, const void* w_gate, const void* w_up, int64_t expert_stride,
                                int64_t n_expert, int64_t n_ff, int64_t k, const uint16_t* x, int64_t x_slots,
                                const int32_t* ids, int64_t n_tokens, int64_t top_k, int glu_op, int swapped, void* y,
                                int y_type, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!glu_op_ok(glu_op) || (swapped != 0 && swapped != 1)) return SPIRAL_ERR_TYPE;
  if (n_tokens == 0 && is_quant_type(type) && (y_type == SPIRAL_TYPE_BF16 || y_type == SPIRAL_TYPE_F32))
    return SPIRAL_OK;
  if (w_up == nullptr) return SPIRAL_ERR_NULL;
  int rc = check_mul_mat_id(type, w_gate, expert_stride, n_expert, n_ff, k, x, x_slots, ids, n_tokens, top_k, y,
                            y_type, workspace, workspace_bytes);
  if (rc != SPIRAL_OK) return rc;
  if (!aligned16(w_up)) return SPIRAL_ERR_ALIGN;
  if (n_ff > INT64_MAX / 2 || !spiral_mul_mat_id_glu_fits(type, 2 * n_ff, k)) return SPIRAL_ERR_SHAPE;
  rc = require_device();
  if (rc != SPIRAL_OK) return rc;
  return moe(type, w_gate, expert_stride, n_expert, 2 * n_ff, k, x, x_slots, ids, n_tokens, top_k, y, y_type, glu_op,
             swapped, workspace, static_cast<hipStream_t>(stream), w_up);
}

}  // extern "C"

namespace spiral {

// Argument checks and launch shared by the GLU entry points (alpha and limit
// are read by SWIGLU_OAI only).
int glu_split_entry(int glu_op, int swapped, float alpha, float limit, const float* gate, int64_t ldg,
                    const float* up, int64_t ldu, int64_t F, int64_t rows, float* y, int64_t ldy, uint16_t* copy,
                    void* stream) {
  if (swapped != 0 && swapped != 1) return SPIRAL_ERR_TYPE;
  int64_t span = 0;
  const int64_t ld = std::max(ldg, std::max(ldu, ldy));
  if (F < 0 || rows < 0 || ldg < F || ldu < F || ldy < F || __builtin_mul_overflow(rows, ld, &span))
    return SPIRAL_ERR_SHAPE;
  if (F == 0 || rows == 0) return SPIRAL_OK;
  if (gate == nullptr || up == nullptr || y == nullptr) return SPIRAL_ERR_NULL;
  if ((reinterpret_cast<uintptr_t>(gate) & 3u) != 0 || (reinterpret_cast<uintptr_t>(up) & 3u) != 0 ||
      (reinterpret_cast<uintptr_t>(y) & 3u) != 0)
    return SPIRAL_ERR_ALIGN;
  const int rc = require_device();
  if (rc != SPIRAL_OK) return rc;
  return glu_split(glu_op, swapped, gate, ldg, up, ldu, F, rows, y, ldy, static_cast<hipStream_t>(stream), alpha,
                   limit, copy);
}

int glu_entry(int glu_op, int swapped, float alpha, float limit, const float* x, int64_t ldx, int64_t F, int64_t rows,
              float* y, int64_t ldy, uint16_t* copy, void* stream) {
  if (swapped != 0 && swapped != 1) return SPIRAL_ERR_TYPE;
  int64_t span = 0;
  if (F < 0 || rows < 0 || F > INT64_MAX / 2 || ldx < 2 * F || ldy < F ||
      __builtin_mul_overflow(rows, ldx > ldy ? ldx : ldy, &span))
    return SPIRAL_ERR_SHAPE;
  if (F == 0 || rows == 0) return SPIRAL_OK;
  if (x == nullptr || y == nullptr) return SPIRAL_ERR_NULL;
  if ((reinterpret_cast<uintptr_t>(x) & 3u) != 0 || (reinterpret_cast<uintptr_t>(y) & 3u) != 0)
    return SPIRAL_ERR_ALIGN;
  const int rc = require_device();
  if (rc != SPIRAL_OK) return rc;
  return glu(glu_op, swapped, x, ldx, F, rows, y, ldy, static_cast<hipStream_t>(stream), alpha, limit, copy);
}

}  // namespace spiral

extern "C" {

int spiral_glu_split(int glu_op, int swapped, const float* gate, int64_t ldg, const float* up, int64_t ldu, int64_t F,
                     int64_t rows, float* y, int64_t ldy, void* stream) {
  if (!glu_op_ok(glu_op)) return SPIRAL_ERR_TYPE;
  return glu_split_entry(glu_op, swapped, 0.0f, 0.0f, gate, ldg, up, ldu, F, rows, y, ldy, nullptr, stream);
}

int spiral_glu(int glu_op, int swapped, const float* x, int64_t ldx, int64_t F, int64_t rows, float* y, int64_t ldy,
               void* stream) {
  if (!glu_op_ok(glu_op)) return SPIRAL_ERR_TYPE;
  return glu_entry(glu_op, swapped, 0.0f, 0.0f, x, ldx, F, rows, y, ldy, nullptr, stream);
}

int spiral_glu_swiglu_oai(int swapped, float alpha, float limit, const float* x, int64_t ldx, int64_t F, int64_t rows,
                          float* y, int64_t ldy, void* stream) {
  return glu_entry(SPIRAL_GLU_SWIGLU_OAI, swapped, alpha, limit, x, ldx, F, rows, y, ldy, nullptr, stream);
}

int spiral_glu_split_swiglu_oai(int swapped, float alpha, float limit, const float* gate, int64_t ldg,
                                const float* up, int64_t ldu, int64_t F, int64_t rows, float* y, int64_t ldy,
                                void* stream) {
  return glu_split_entry(SPIRAL_GLU_SWIGLU_OAI, swapped, alpha, limit, gate, ldg, up, ldu, F, rows, y, ldy, nullptr, stream);
}

}  // extern "C"
