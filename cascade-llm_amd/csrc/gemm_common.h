// What the prefill GEMM kernels share: the epilogue kinds, the argument block
// and the launch of the one-pass streaming kernel (gemm_stream.hip).
#pragma once

#include "cascade_device.h"
#include "cascade_internal.h"

namespace cascade {

enum GemmEpilogue : int {
  kGemmStore = 0,
  kGemmResidual = 1,
  kGemmQkvRope = 2,
  kGemmSwiglu = 3,
  kGemmSilu = 4,
  kGemmMul = 5,
  kGemmF32 = 6,
};

constexpr int kXcds = 8;
constexpr int kGemmHead = 128;
constexpr int kGemmHalfHead = 64;

struct GemmArgs {
  const uint16_t *x;  // [m, k]
  const uint16_t *w0;  // store/residual/silu/mul/f32: W; qkv: Wq; swiglu: Wgate
  const uint16_t *w1;  // qkv: Wk; swiglu: Wup
  const uint16_t *w2;  // qkv: Wv
  int64_t n0, n1, n2;  // rows of w0 / w1 / w2 (swiglu: n0 = n_half)
  int64_t m, k;
  uint16_t *y;  // [m, ldy] (qkv: the q rows, ldy = n0)
  int64_t ldy;
  float *yf;    // kGemmF32 output [m, ldy]
  const uint16_t *aux;  // residual (kGemmResidual) or gate (kGemmMul), [m, ldy]
  const uint16_t *rope_cos;  // [positions, 64] bf16
  const uint16_t *rope_sin;
  int64_t pos0;
  uint16_t *k_out;  // position 0 of KV head 0 of this layer's K cache
  uint16_t *v_out;
  int64_t kv_head_stride;
  int64_t slot0;
  // full tiles: a tiles_m x tiles_n grid (tiles of them, per_xcd on each
  // XCD); half-height tiles: an htiles_m x htiles_n grid right of it
  int32_t tiles_m, tiles_n, tiles, per_xcd;
  int32_t htiles_m, htiles_n, htiles, hper_xcd;
  int32_t vec_out;  // row pitches and widths allow 16-byte output accesses
  // split K (fp32 partials, kGemmF32 only): workgroup row blockIdx.y runs
  // slabs [blockIdx.y * split_slabs, + split_slabs) of K and writes its
  // partial at yf + blockIdx.y * split_stride; 0: the whole K
  int32_t split_slabs;
  int64_t split_stride;
  // streaming kernel: start each tile's walk over K at another slab
  int32_t rotate;
};

__device__ __forceinline__ float gemm_silu(float g) {
  return g / (1.0f + expf(-g));
}

// CUs of the device a stream runs on (gemm.hip).
int gemm_device_cus(hipStream_t s);

// The streaming kernel of short prompts (gemm_stream.hip).  A plan names its
// shape: weight rows of a workgroup, 16-token fragments of a workgroup (0: the
// tiles of gemm.hip take the product) and runs of K.
struct StreamPlan {
  int fm, rows, splits;
};
// n: the rows of all weight matrices of the launch (gate and up both count).
StreamPlan stream_plan(int epi, int64_t m, int64_t n, int cus);
// Over split K, fp32 partials (args.split_slabs / split_stride / yf).
StreamPlan stream_split_plan(int64_t m, int64_t n, int64_t k, int cus);
hipError_t launch_stream(int epi, const StreamPlan &p, const GemmArgs &args, hipStream_t s);

}  // namespace cascade
