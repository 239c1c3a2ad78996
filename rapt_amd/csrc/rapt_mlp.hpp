// rapt_mlp.hpp -- what the surrogate's translation units share: the network's
// layout, its activation and the inference kernel's arguments.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rapt {
namespace mlp {

constexpr int H = 256;
constexpr int OFF_W1 = 0;                 // [256][3]
constexpr int OFF_B1 = OFF_W1 + H * 3;    // [256]
constexpr int OFF_W2 = OFF_B1 + H;        // [256][256] (out, in)
constexpr int OFF_B2 = OFF_W2 + H * H;
constexpr int OFF_W3 = OFF_B2 + H;
constexpr int OFF_B3 = OFF_W3 + H * H;
constexpr int OFF_W4 = OFF_B3 + H;        // [3][256]
constexpr int OFF_B4 = OFF_W4 + 3 * H;    // [3]
constexpr int NPARAM = OFF_B4 + 3;        // 133,379
constexpr int NPAD = (NPARAM + 255) / 256 * 256;
constexpr int PACKED = 8 * 16 * 64 * 8;   // bf16 elements of one packed 256x256 layer

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// The network is a SiLU MLP whose parameters are kept in base-2 units.  With
// the plain network's (W1, b1, W2, b2, W3, b3, W4, b4) the stored parameters
// are (log2(e) W1, log2(e) b1, W2, log2(e) b2, W3, log2(e) b3, ln(2) W4, b4):
// every hidden pre-activation is then a = log2(e) z and every hidden output
// g = log2(e) silu(z) = a / (1 + 2^-a), the same function, while the logistic
// factor is rcp(1 + exp2(-a)), one v_exp_f32 and one v_rcp_f32 (about 1 ulp
// each) with no scaling multiply in front.  Training and inference use these
// same definitions, so both round the same hidden values to bf16.
constexpr float LN2 = 0.6931471805599453f;
__device__ __forceinline__ float sig2(float a) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-a));
}
__device__ __forceinline__ float act2(float a) { return a * sig2(a); }
// d act2 / da = s (1 + ln2 a (1 - s)), s = sig2(a)
__device__ __forceinline__ float dact2(float a) {
  const float s = sig2(a);
  return s * (1.0f + LN2 * a * (1.0f - s));
}

constexpr int MAXM = 4;   // largest ensemble

struct InferArgs {
  int64_t n;
  int members;
  const bf16* wb;         // [members][NPAD]
  const bf16* packed;     // [members][2][PACKED]: layers 2 and 3
  const bf16* p1;         // [members][16*64*8]: layer-1 A operands
  const float* norm;      // shift[3], scale[3]
  float thresh;           // relative member deviation that sends a query to the fallback
  const float* prep;      // [n][8] k_prep's features and baselines
  float* out;             // [n][3] physical outputs (T_b, |omega_d|, latitude)
  float* raw;             // optional [members][n][3] normalised outputs
  int32_t* flag;          // [n] in: k_prep's side | near << 1; out: 1 = fallback
};

// a layer's packed K order (k_infer)
__device__ __forceinline__ int pin32(int kb, int h, int j) {
  return 32 * (kb >> 1) + 16 * (kb & 1) + 8 * (j >> 2) + 4 * h + (j & 3);
}
__device__ __forceinline__ int row32(int r, int h) { return 8 * (r >> 2) + 4 * h + (r & 3); }

// Layer-1 operands of one member, bf16 elements
constexpr int P1SIZE = 8 * 64 * 8;
}  // namespace mlp
}  // namespace rapt

// the ensemble inference kernel on n prepared queries (rapt_mlp_infer.hip);
// cus: compute units of the device
void rapt_launch_infer(hipStream_t st, const rapt::mlp::InferArgs& A, int cus);
