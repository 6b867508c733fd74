// Wide dense layer + activation (N > 128): internal interface between the two source files
// behind folx_hip_dense_act_fwdlap.
#pragma once
#include "common.h"

constexpr int FOLX_MAX_PARTS = 8;

// The Jacobian operand as a concatenation along K of up to FOLX_MAX_PARTS arrays (widths multiples
// of 16, so that no chunk of K straddles two).  A broadcast part has one row per `group`
// consecutive positions (a per-walker feature shown to every electron).
struct FolxWideParts {
  const float* jac[FOLX_MAX_PARTS];
  int64_t pstride[FOLX_MAX_PARTS];  // floats between consecutive Jacobian rows of the part
  int32_t width[FOLX_MAX_PARTS];
  int32_t kend[FOLX_MAX_PARTS];     // first k after the part
  int32_t bcast[FOLX_MAX_PARTS];
  int32_t n, group;
};

// Workspace the wide path needs, or a negative error code when the shape is not one it takes.
int64_t folx_dense_act_wide_ws_bytes(int64_t R, int32_t P, int32_t K, int32_t N);

// Jacobian rows of a group in the wide path's tiles (8, 16 or 32), and whether it is expected to be faster than the plain
// product over `plain` features followed by the activation (1 / 0); a negative error code as above.
int folx_dense_act_wide_group(int64_t R, int32_t P, int32_t K, int32_t N);
int folx_dense_act_wide_faster(int64_t R, int32_t P, int32_t K, int32_t N, int32_t plain);

int folx_dense_act_wide(hipStream_t st, int32_t act, float param, const float* x, const float* jac, const float* lap,
                        const float* W, const float* bias, float* y, float* y_jac, float* y_lap, int64_t R,
                        int32_t P, int32_t K, int32_t N, void* workspace, int64_t workspace_bytes);

// The same layers with their products from bf16 pieces (wide_pieces.hip): what they need, whether they are expected to be faster than
// the plain product over `plain` features and the activation after it, and the call (jac, or parts of it).
int64_t folx_wide_pieces_ws_bytes(int64_t R, int32_t P, int32_t K, int32_t N);
int folx_wide_pieces_faster(int64_t R, int32_t P, int32_t K, int32_t N, int32_t plain);
int folx_wide_pieces(hipStream_t st, int32_t act, float param, const float* x, const float* jac, const float* lap,
                     const FolxWideParts* parts, const float* W, const float* bias, const float* res, const float* res_jac,
                     const float* res_lap, const float* pre, const float* pre_jac, const float* pre_lap, int64_t pre_group,
                     float* y, float* y_jac, float* y_lap, int64_t R, int32_t P, int32_t K, int32_t N, void* workspace,
                     int64_t workspace_bytes);
