// What the two forms of a chain of narrow dense + activation layers share.
#pragma once
#include "common.h"

namespace folx_chain {

constexpr int MAXL = FOLX_HIP_CHAIN_MAX_LAYERS;

struct Layer {
  const float *W, *bias;
  int32_t K, N, act;  // act < 0: none (last layer, N = 1)
  float prm;
};

struct Params {
  const float *x, *jac, *lap;
  float *y, *y_jac, *y_lap;
  float *h, *h_jac, *h_lap;  // what goes into a matrix-vector product at the end, where somebody else reads it too
  int64_t R;
  int32_t P, L, ld, vec;
  Layer layer[MAXL];
};

// Over many Jacobian rows (dense_chain_many.hip): whether the chain is for it, and the scratch it takes.
bool many_plan(int L, const int32_t* act, const int32_t* widths, int64_t R, int32_t P, bool& faster, int64_t& ws_bytes);
int many_launch(hipStream_t stream, const Params& prm, const int32_t* act, const int32_t* widths, void* ws);

}  // namespace folx_chain
