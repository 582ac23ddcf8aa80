// Dense (unquantised) products shared by dense.hip, dense_tile.hip and the
// prefill GEMM entry in mm8h.hip.
#pragma once
#include "common.h"

namespace rwkv7mi {

enum { ACT_NONE = 0, ACT_TANH = 1, ACT_SIGMOID = 2, ACT_RELU2 = 3 };

struct DenseProb {
  const void* x;
  const void* W;
  const void* bias;
  const void* residual;  // added after the activation, or null
  void* y;
  int N, K, act, tile0;
};
struct DenseBatch {
  DenseProb p[4];
  int nprob;
};

__device__ __forceinline__ float apply_act(float v, int act) {
  if (act == ACT_TANH) return tanhf(v);
  if (act == ACT_SIGMOID) return 1.0f / (1.0f + expf(-v));
  if (act == ACT_RELU2) {
    v = fmaxf(v, 0.f);
    return v * v;
  }
  return v;
}

// Tile kernel for fp16 / bf16 (dense_tile.hip).  part null: y with the
// epilogue; else S K ranges of fp32 partials [problem][split][row][ldp]
// (problems of one shape).  dense_tile_us: its estimated time for S splits.
bool dense_tile_supported(const DenseBatch& b, int64_t rows, int act_dtype);
double dense_tile_us(const DenseBatch& b, int64_t rows, int S);
int dense_tile_run(const DenseBatch& b, int64_t rows, int act_dtype, int S, float* part, int64_t ldp, void* stream);

}  // namespace rwkv7mi
