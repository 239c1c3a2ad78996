// rapt_mlp_infer.hip -- the surrogate's fused ensemble inference kernel, in a
// translation unit of its own (its scheduling takes minutes to compile).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "rapt_mlp.hpp"

namespace rapt {
namespace mlp {

// ---- fused inference -------------------------------------------------------------------
// One kernel runs the whole ensemble forward pass, the disagreement test and
// the baseline for a batch of queries; activations never leave registers.
//
// v_mfma_f32_32x32x16_bf16, 32 queries per wave: lane l holds query l%32 and
// half h = l/32 of each activation.  A 32x32 output tile t leaves register r
// of lane l holding neuron 32t + row32(r, h), row32(r, h) = 8(r/4) + 4h + r%4
// (the D layout of the instruction: D[8(r/4)+4(l/32)+r%4][l%32]; A operand:
// lane l holds row l%32, K indices 8(l/32)+j; B operand: column l%32, K
// indices 8(l/32)+j).  Registers 8g..8g+7 of tile t form the B operand of
// K-block kb = 2t+g of the next layer, so K index 8h + j of block kb is input
// neuron pin32(kb, h, j) = 32(kb/2) + 16(kb%2) + 8(j/4) + 4h + j%4, and the
// packed weights are P[t][kb][lane][j] = W[32t + lane%32][pin32(kb, lane/32,
// j)].  A block of IW waves stages one member's packed 256x256 layer (128
// KB) in LDS and its waves (IW x 32 queries) read the A fragments from
// there, so L2 supplies each weight once per block instead of once per wave;
// each fragment read from LDS feeds a 32-query MFMA.
// one member's small parameters, staged in LDS: b1, b2, b3, w4 (one float4
// of the three output weights per layer-3 neuron), b4
struct SmallW {
  float b1[H], b2[H], b3[H];
  float4 w4[H];
  float b4[4];
};
typedef float f32x4 __attribute__((ext_vector_type(4)));

// the biases of one 32x32 output tile in a lane's accumulator order: register
// r holds neuron row32(r, h), so b points at the tile's bias + 4h and the 16
// values are four float4 runs at 8-element strides
__device__ __forceinline__ f32x16 bias16(const float* b) {
  f32x16 acc;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float4 v = *(const float4*)(b + 8 * q);
    acc[4 * q] = v.x;
    acc[4 * q + 1] = v.y;
    acc[4 * q + 2] = v.z;
    acc[4 * q + 3] = v.w;
  }
  return acc;
}

// IW = 8 waves per block (two per SIMD), 32 queries per wave.  The biases
// start the accumulators.  Staging is pipelined: each member's two 256x256
// layers pass through LDS as four 64 KB halves (layer 2 tiles 0-3, 4-7, then
// layer 3), alternating between two buffers; while the waves compute with
// one half, the next half (the next member's, or member 0's for the next
// chunk) streams into the other buffer with direct global-to-LDS loads, so
// the loads never wait on a barrier with the matrix cores idle.  A half is
// 64 fragments of 1 KB; wave w loads fragments 8i + w.
constexpr int IW = 8;
constexpr int QW = 32;  // queries per wave
constexpr int HALF = PACKED / 16;  // bf16x8 elements of half a packed layer (64 KB)

// stage s of a member's four: layer 2 + (s >> 1), fragments 64 (s & 1) onward.
// Wave wv loads fragments 8i + wv, starting at i = rot (the block's rotation,
// so that the CUs of an XCD do not all ask the L2 for the same lines at the
// same moment).  The loads go through a buffer resource
// (buffer_load_dwordx4 ... lds), which counts on vmcnt alone: with the FLAT
// form (global_load_lds) in flight the compiler must treat the LDS counter as
// unordered, and every LDS read of the half being computed would then wait
// for all reads issued before it.
__device__ __forceinline__ void stage_load(__amdgpu_buffer_rsrc_t rs, int m, int s, bf16x8* buf,
                                           int wv, int l, int rot) {
  const int base = (m * 2 + (s >> 1)) * PACKED * 2 + (s & 1) * HALF * 16;  // bytes
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int f = 8 * ((i + rot) & 7) + wv;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rs, (__attribute__((address_space(3))) void*)(buf + 64 * f), 16,
        base + (64 * f + l) * 16, 0, 0, 0);
  }
}

__device__ __forceinline__ void wait_loads() { __builtin_amdgcn_s_waitcnt(0); }

// one 32x32 output tile of a hidden layer from the fragments of buf (tile
// t of the half: fragments 16 t .. 16 t + 15).  The A fragments are read
// PF ahead into a ring of registers, so each MFMA's LDS read has PF - 1
// matrix operations of cover (the compiler's own schedule gives one).
constexpr int PF = 4;
__device__ __forceinline__ f32x16 tile32(const bf16x8* buf, int t, const bf16x8* in,
                                         f32x16 acc, int l) {
  const bf16x8* p = buf + 16 * t * 64 + l;
  bf16x8 a[PF];
#pragma unroll
  for (int i = 0; i < PF; ++i) a[i] = p[i * 64];
#pragma unroll
  for (int kb = 0; kb < 16; ++kb) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[kb % PF], in[kb], acc, 0, 0, 0);
    if (kb + PF < 16) a[kb % PF] = p[(kb + PF) * 64];
  }
  // keep that order in the schedule (left alone, the scheduler sinks each
  // read next to its MFMA to save registers): PF LDS reads (mask 0x100),
  // then per step one MFMA (0x008), one LDS read and up to five other
  // vector instructions (0x002)
  __builtin_amdgcn_sched_group_barrier(0x100, PF, 0);
#pragma unroll
  for (int kb = 0; kb < 16; ++kb) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    if (kb + PF < 16) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
  }
  return acc;
}

__global__ __launch_bounds__(IW * 64) void k_infer(InferArgs A) {
  __shared__ bf16x8 buf0[HALF], buf1[HALF];
  __shared__ SmallW sw[MAXM];
  const int l = threadIdx.x & 63, wv = threadIdx.x >> 6, h = l >> 5;
  const int64_t groups = (A.n + QW - 1) / QW;
  const int64_t chunks = (groups + IW - 1) / IW;
  if ((int64_t)blockIdx.x >= chunks) return;  // no work: no barrier is reached
  for (int m = 0; m < A.members; ++m) {
    const bf16* w = A.wb + (int64_t)m * NPAD;
    for (int i = threadIdx.x; i < H; i += IW * 64) {
      sw[m].b1[i] = (float)w[OFF_B1 + i];
      sw[m].b2[i] = (float)w[OFF_B2 + i];
      sw[m].b3[i] = (float)w[OFF_B3 + i];
      sw[m].w4[i] = make_float4((float)w[OFF_W4 + i], (float)w[OFF_W4 + H + i],
                                (float)w[OFF_W4 + 2 * H + i], 0.0f);
    }
    if (threadIdx.x < 3) sw[m].b4[threadIdx.x] = (float)w[OFF_B4 + threadIdx.x];
  }
  // the packed layers 2 and 3 of every member as a raw buffer (stride 0,
  // the gfx9 word-3 format bits); reads past the end return 0
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)A.packed, (short)0, A.members * 2 * PACKED * (int)sizeof(bf16), 0x00020000);
  const int rot = blockIdx.x & 7;
  stage_load(rs, 0, 0, buf0, wv, l, rot);
  for (int64_t ch = blockIdx.x; ch < chunks; ch += gridDim.x) {
    const int64_t g = ch * IW + wv;
    const int64_t qi = g * QW + (l & 31);
    const bool valid = g < groups && qi < A.n;
    const float4* pq = (const float4*)(A.prep + 8 * (valid ? qi : 0));
    const float4 p0 = pq[0];
    const float xin[3] = {p0.x, p0.y, p0.z};
    const int rg = valid ? A.flag[qi] : 0;  // k_prep's side | near << 1
    bf16x8 xb;
#pragma unroll
    for (int j = 0; j < 8; ++j) xb[j] = (bf16)0.0f;
    if (h == 0) {
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const bf16 hv = (bf16)xin[j];
        xb[j] = hv;
        xb[3 + j] = (bf16)(xin[j] - (float)hv);
      }
    }
    float mean[3] = {0.0f, 0.0f, 0.0f}, lo[3], hi[3];
    for (int c = 0; c < 3; ++c) { lo[c] = 3.0e38f; hi[c] = -3.0e38f; }
    for (int m = 0; m < A.members; ++m) {
      const SmallW& W = sw[m];
      const bf16x8* P1 = (const bf16x8*)(A.p1 + (int64_t)m * P1SIZE);
      const int mn = m + 1 < A.members ? m + 1 : 0;  // the member whose layer 2 comes next
      // layer 1 (its operands come from global memory)
      bf16x8 act[16];
      wait_loads();
      __syncthreads();  // first pass: sw written; every pass: this member's half 0 landed
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        f32x16 acc = bias16(&W.b1[32 * t + 4 * h]);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(P1[t * 64 + l], xb, acc, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 16; ++r) act[2 * t + (r >> 3)][r & 7] = (bf16)act2(acc[r]);
      }
      // layer 2, tiles 0-3 from buf0 while tiles 4-7 stream into buf1
      stage_load(rs, m, 1, buf1, wv, l, rot);
      bf16x8 nxt[16];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        f32x16 acc = tile32(buf0, t, act, bias16(&W.b2[32 * t + 4 * h]), l);
#pragma unroll
        for (int r = 0; r < 16; ++r) nxt[2 * t + (r >> 3)][r & 7] = (bf16)act2(acc[r]);
      }
      wait_loads();
      __syncthreads();  // buf1 landed; buf0 free
      stage_load(rs, m, 2, buf0, wv, l, rot);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        f32x16 acc = tile32(buf1, t, act, bias16(&W.b2[32 * (t + 4) + 4 * h]), l);
#pragma unroll
        for (int r = 0; r < 16; ++r) nxt[2 * (t + 4) + (r >> 3)][r & 7] = (bf16)act2(acc[r]);
      }
      wait_loads();
      __syncthreads();  // layer 3 half 0 in buf0; buf1 free
      stage_load(rs, m, 3, buf1, wv, l, rot);
      // layer 3 and the output layer (FP32)
      float o0 = 0.0f, o1 = 0.0f, o2 = 0.0f;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        if (half == 1) {
          wait_loads();
          __syncthreads();  // layer 3 half 1 in buf1; buf0 free
          stage_load(rs, mn, 0, buf0, wv, l, rot);
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int tt = 4 * half + t;
          f32x16 acc = tile32(half ? buf1 : buf0, t, nxt, bias16(&W.b3[32 * tt + 4 * h]), l);
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float4 c = W.w4[32 * tt + row32(r, h)];
            const float v = act2(acc[r]);
            // fused multiply-adds (the library compiles without contraction)
            o0 = __builtin_fmaf(c.x, v, o0);
            o1 = __builtin_fmaf(c.y, v, o1);
            o2 = __builtin_fmaf(c.z, v, o2);
          }
        }
      }
      o0 += __shfl_xor(o0, 32);
      o1 += __shfl_xor(o1, 32);
      o2 += __shfl_xor(o2, 32);
      const float o[3] = {o0 + W.b4[0], o1 + W.b4[1], o2 + W.b4[2]};
      for (int c = 0; c < 3; ++c) {
        mean[c] += o[c];
        lo[c] = fminf(lo[c], o[c]);
        hi[c] = fmaxf(hi[c], o[c]);
      }
      if (A.raw && valid && l < 32)
        for (int c = 0; c < 3; ++c) A.raw[((int64_t)m * A.n + qi) * 3 + c] = o[c];
    }
    if (valid && l < 32) {
      const float4 p1 = pq[1];
      const float bb[3] = {p0.w, p1.x, p1.y};
      int bad = (rg & 2) ? 1 : 0;
      for (int k = 0; k < 3; ++k) {
        const float sc = A.norm[3 + k];
        const float mu = mean[k] / (float)A.members;
        if (expm1f(sc * fmaxf(hi[k] - mu, mu - lo[k])) > A.thresh) bad = 1;
        A.out[qi * 3 + k] = expf(bb[k] + A.norm[k] + sc * mu);
      }
      A.flag[qi] = bad;
    }
  }
  wait_loads();  // the prefetch issued for a chunk this block does not run
}

}  // namespace mlp
}  // namespace rapt

// persistent: one block per CU, each taking chunks of IW x QW queries
void rapt_launch_infer(hipStream_t st, const rapt::mlp::InferArgs& A, int cus) {
  using namespace rapt::mlp;
  const int64_t groups = (A.n + QW - 1) / QW;
  int64_t blocks = (groups + IW - 1) / IW;
  if (blocks > cus) blocks = cus;
  hipLaunchKernelGGL(k_infer, dim3((unsigned)blocks), dim3(IW * 64), 0, st, A);
}
