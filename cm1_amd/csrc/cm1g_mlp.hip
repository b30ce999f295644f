// A small per-cell MLP (8 -> 128 -> 128 -> 128 -> 4, SiLU hidden layers)
// with BF16 operands and FP32 accumulation on the CDNA matrix cores, used as
// a learned surrogate for the local part of Kessler microphysics.  No
// counterpart in the reference.
//
// Operands are rounded from FP32 to BF16 to nearest, ties to even.  Training
// (cm1g_mlp_loss_grad) is three kernels: k_train runs 16-sample groups
// forward and backward in registers and writes the operands of the weight
// gradients, k_wgrad contracts them over the samples, k_grad_final adds the
// partial sums in a fixed order; the loss is the mean squared error of the
// normalised outputs.  Inference runs fused (mlp_tiles in cm1g_mlp.h).
#include "cm1g_mlp.h"

#include <algorithm>
#include <random>

#define ARGCHK(cond, msg)          \
  do {                             \
    if (!(cond)) {                 \
      cm1g_set_error(msg);         \
      return CM1G_E_ARG;           \
    }                              \
  } while (0)

struct cm1g_mlp {
  float *p = nullptr, *g = nullptr, *m1 = nullptr, *m2 = nullptr;  // params, grads, Adam moments
  float *dnorm = nullptr;                                          // normalisation (device)
  int64_t adam_t = 0;
  hipStream_t stream = nullptr;
  MlpPack *pk = nullptr;                                           // BF16 weights in fragment order
  // training workspace for `cap` rows: the weight gradients' operands, and
  // the partial sums of k_train's and k_wgrad's workgroups
  int64_t cap = 0;
  unsigned short *frag = nullptr;
  float *part = nullptr, *wpart = nullptr, *keep = nullptr, *red = nullptr;
};
const MlpPack *mlp_packed(const cm1g_mlp *n) { return n->pk; }

const float *mlp_params(const cm1g_mlp *n) { return n->p; }
const float *mlp_norm(const cm1g_mlp *n) { return n->dnorm; }

// ------------------------------------------------------------ packing
// the fragment positions of parameter i, BF16 (biases stay FP32 in the
// parameters themselves)
__device__ __forceinline__ void mlp_pack_one(MlpPack *pk, int i, float v) {
  const unsigned short b = bf16_rne(v);
  if (i < OB1) {
    const int k = (i - OW1) / MLP_H, n = (i - OW1) % MLP_H;
    ((unsigned short *)pk->f.w1)[mlp_wfrag(k, n, 1)] = b;
  } else if (i >= OW2 && i < OB2) {
    const int k = (i - OW2) / MLP_H, n = (i - OW2) % MLP_H;
    ((unsigned short *)pk->f.w2)[mlp_wfrag32(k, n, 4)] = b;
    ((unsigned short *)pk->b.b2)[mlp_wfrag32(n, k, 4)] = b;
  } else if (i >= OW3 && i < OB3) {
    const int k = (i - OW3) / MLP_H, n = (i - OW3) % MLP_H;
    ((unsigned short *)pk->f.w3)[mlp_wfrag32(k, n, 4)] = b;
    ((unsigned short *)pk->b.b3)[mlp_wfrag32(n, k, 4)] = b;
  } else if (i >= OW4 && i < OB4) {
    const int k = (i - OW4) / MLP_OUT, n = (i - OW4) % MLP_OUT;
    ((unsigned short *)pk->f.w4)[mlp_wfrag32(k, n, 4)] = b;
    ((unsigned short *)pk->b.b4)[mlp_wfrag(n, k, 1)] = b;
  }
}
// (the padding of the first and last layers stays the zero it was allocated
// with)
__global__ void __launch_bounds__(256) k_pack(const float *__restrict__ p, MlpPack *__restrict__ pk) {
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i < MLP_NPARAM) mlp_pack_one(pk, i, p[i]);
}

// ------------------------------------------------------------ training
// The weight gradients' operands of one 16-sample group: tiles of 16
// features x 16 samples in BF16, lane l of a tile holding feature l%16,
// samples 4(l/16)..+3 (what the matrix instructions take with the samples as
// the summed index).
constexpr int T_X = 0, T_H1 = 1, T_H2 = 9, T_H3 = 17, T_D1 = 25, T_D2 = 33, T_D3 = 41, T_DY = 49, T_N = 50;
constexpr int T_ELEM = 256;
constexpr int TP_N = 392;  // one workgroup's partial sums: 3 x 128 + 4 bias gradients, the loss (a double)
constexpr int TP_LOSS = 3 * MLP_H + MLP_OUT;
static_assert(TP_N % 2 == 0 && TP_LOSS % 2 == 0 && TP_LOSS + 2 <= TP_N, "the loss's place");

// (the caller's rows may start on any float)
typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));

struct TrainLds {
  MlpPack w;
  float b[3 * MLP_H + 16];
  unsigned short tr[MLP_WAVES][64][16];  // a wavefront's transposes: 64 features x 16 samples
};
static_assert(sizeof(TrainLds) <= 160 * 1024, "k_train: LDS");

// tiles nt0..nt0+n-1 (n <= 4) of a lane's values, sample l%16 and outputs
// 16nt + 4(l/16) + t, to the layout above
template <int N>
__device__ __forceinline__ void put_tiles(unsigned short (*tr)[16], const bf16x4 *x, unsigned short *dst, int l) {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
  for (int q = 0; q < N; q++)
#pragma unroll
    for (int t = 0; t < 4; t++) tr[16 * q + 4 * (l >> 4) + t][l & 15] = (unsigned short)x[q][t];
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
  for (int q = 0; q < N; q++) {
    const bf16x4 v = *(const bf16x4 *)&tr[16 * q + (l & 15)][4 * (l >> 4)];
    *(bf16x4 *)(dst + q * T_ELEM + 4 * l) = v;
  }
}

template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}
// Sums over the 16 samples (lanes l%16) of a lane's 32 values: each step
// hands half of the values to a partner lane and keeps the other half, so
// lane s ends with values 2s', 2s'+1, s' = s; order fixed.
__device__ __forceinline__ void sum16(const floatx4 (&z)[8], float &r0, float &r1, int l) {
  const bool b3 = l & 8, b2 = l & 4, b1 = l & 2, b0 = l & 1;
  float v[32];
#pragma unroll
  for (int q = 0; q < 32; q++) v[q] = z[q >> 2][q & 3];
#pragma unroll
  for (int q = 0; q < 16; q++) {
    const float keep = b3 ? v[q + 16] : v[q], send = b3 ? v[q] : v[q + 16];
    v[q] = keep + dpp<0x128>(send);  // row_ror:8
  }
#pragma unroll
  for (int q = 0; q < 8; q++) {
    const float keep = b2 ? v[q + 8] : v[q], send = b2 ? v[q] : v[q + 8];
    v[q] = keep + dpp<0x141>(send);  // row_half_mirror
  }
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const float keep = b1 ? v[q + 4] : v[q], send = b1 ? v[q] : v[q + 4];
    v[q] = keep + dpp<0x4E>(send);  // quad_perm [2,3,0,1]
  }
#pragma unroll
  for (int q = 0; q < 2; q++) {
    const float keep = b0 ? v[q + 2] : v[q], send = b0 ? v[q] : v[q + 2];
    v[q] = keep + dpp<0xB1>(send);  // quad_perm [1,0,3,2]
  }
  r0 += v[0];
  r1 += v[1];
  __builtin_amdgcn_sched_barrier(0);
}

// acc (pre-activations) -> x = SiLU in BF16, in inference's form, d = SiLU'.
// The derivative reaches the bias gradients unrounded, so its sigmoid is a
// single-precision one: the hardware forms' error, which BF16 activations do
// not show, grows with |z| (3e-6 of the derivative at z = -80, 5e-7 here; k_train
// 37 us with them, 54 so).
__device__ __forceinline__ void silu_both(const floatx4 (&acc)[1][8], bf16x4 (&x)[1][8], floatx4 (&d)[8]) {
#pragma unroll
  for (int nt = 0; nt < 8; nt++) {
    floatx4 h;
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const float z = acc[0][nt][t];
      h[t] = silu_f(z);
      const float sg = 1.0f / (1.0f + expf(-z));
      d[nt][t] = sg * (1.0f + z * (1.0f - sg));
    }
    x[0][nt] = mlp_pack(h[0], h[1], h[2], h[3]);
    __builtin_amdgcn_sched_barrier(0);
  }
}
// acc += W x, 128 x 128 in four 32-deep steps (one step's weight fragments at
// a time: two would not leave the registers to hold the derivatives)
__device__ __forceinline__ void mlp_prod(floatx4 (&acc)[1][8], const bf16x4 (&x)[1][8], const bf16x8s *wf, int l) {
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int kb = 0; kb < 4; kb++) {
    const bf16x8 xb = mlp_join(x[0][2 * kb], x[0][2 * kb + 1]);
#pragma unroll
    for (int nt = 0; nt < 8; nt++)
      acc[0][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf[(nt * 4 + kb) * 64 + l]), xb,
                                                            acc[0][nt], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Forward and backward of 16-sample groups, one group per wavefront at a
// time, activations, derivatives and gradients in registers throughout: each
// layer is computed transposed (mlp_tiles has the argument), and so is its
// backward product dX^T = W dY^T, whose second operand is again what the lane
// holds.  The operands of the weight gradients (the layers' inputs and
// pre-activation gradients, BF16) leave through a small LDS transpose, 25.6 KB
// a group; bias gradients are summed from the FP32 gradients.  Bound by the
// vector unit (two exponentials, a reciprocal and a division per hidden value)
// and by those stores: 54 us for 65536 rows, k_wgrad 32, k_grad_final 7; the separate
// products and element-wise passes they replace (FP32 activations through
// memory, column sums by one workgroup each) took 1390 us.
__global__ void __launch_bounds__(512) k_train(const MlpPack *__restrict__ pk, const float *__restrict__ prm,
                                               const float *__restrict__ X, const float *__restrict__ T,
                                               int64_t rows, int64_t ngroups, unsigned short *__restrict__ frag,
                                               float *__restrict__ part, float *keep) {
  __shared__ TrainLds S;
  const int tid = (int)threadIdx.x, l0 = tid & 63, w = tid >> 6;
  mlp_stage(&S.w, pk, (int)sizeof(MlpPack), tid);
  mlp_stage_bias(S.b, prm, tid);
  __syncthreads();
  const int64_t count = rows * MLP_OUT;
  double lsum = 0.0;  // (a lane adds 2048 squares at the largest batch)
  float bs[3][2] = {{0.0f, 0.0f}, {0.0f, 0.0f}, {0.0f, 0.0f}};
  floatx4 b4 = {0.0f, 0.0f, 0.0f, 0.0f};
  const floatx4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int64_t g = (int64_t)blockIdx.x * MLP_WAVES + w; g < ngroups; g += (int64_t)gridDim.x * MLP_WAVES) {
    // opaque, so that the biases and weight fragments are read from LDS where
    // they are used and not kept in registers over the loop
    int l = l0;
    asm volatile("" : "+v"(l));
    const int64_t s = 16 * g + (l & 15);
    unsigned short *fg = frag + g * (T_N * T_ELEM);
    unsigned short(*tr)[16] = S.tr[w];
    // the first layer's derivatives wait in memory (L2): three layers' would
    // not fit the registers, and the compiler's own spills wait one by one
    float *dk = keep + ((int64_t)blockIdx.x * MLP_WAVES + w) * (MLP_H * 16);
    bf16x4 x[1][8];
    floatx4 acc[1][8], d1[8], d2[8], d3[8];
    {
      // lanes 0-15 take inputs 0-3, lanes 16-31 inputs 4-7
      floatx4 v = zero;
      if (l < 32 && s < rows) v = *(const floatx4u *)(X + s * MLP_IN + 4 * (l >> 4));
      x[0][0] = mlp_pack(v[0], v[1], v[2], v[3]);
    }
    floatx4 tv = zero;
    if (l < 16 && s < rows) tv = *(const floatx4u *)(T + s * MLP_OUT);
    put_tiles<1>(tr, &x[0][0], fg + T_X * T_ELEM, l);
    mlp_bias_init(acc, S.b, l);
#pragma unroll
    for (int nt = 0; nt < 8; nt++)
      acc[0][nt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(S.w.f.w1[nt * 64 + l], x[0][0], acc[0][nt], 0, 0, 0);
    silu_both(acc, x, d1);
#pragma unroll
    for (int nt = 0; nt < 8; nt++) *(floatx4 *)(dk + nt * 256 + 4 * l) = d1[nt];
    put_tiles<4>(tr, &x[0][0], fg + T_H1 * T_ELEM, l);
    put_tiles<4>(tr, &x[0][4], fg + (T_H1 + 4) * T_ELEM, l);
    mlp_bias_init(acc, S.b + MLP_H, l);
    mlp_prod(acc, x, S.w.f.w2, l);
    silu_both(acc, x, d2);
    put_tiles<4>(tr, &x[0][0], fg + T_H2 * T_ELEM, l);
    put_tiles<4>(tr, &x[0][4], fg + (T_H2 + 4) * T_ELEM, l);
    mlp_bias_init(acc, S.b + 2 * MLP_H, l);
    mlp_prod(acc, x, S.w.f.w3, l);
    silu_both(acc, x, d3);
    put_tiles<4>(tr, &x[0][0], fg + T_H3 * T_ELEM, l);
    put_tiles<4>(tr, &x[0][4], fg + (T_H3 + 4) * T_ELEM, l);
    // outputs (lane l < 16: the 4 of its sample), loss, dY
    floatx4 y = zero;
#pragma unroll
    for (int kb = 0; kb < 4; kb++)
      y = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, S.w.f.w4[kb * 64 + l]),
                                                  mlp_join(x[0][2 * kb], x[0][2 * kb + 1]), y, 0, 0, 0);
    floatx4 dy = zero;
    if (l < 16 && s < rows) {
#pragma unroll
      for (int t = 0; t < 4; t++) {
        const float e = (y[t] + S.b[3 * MLP_H + t]) - tv[t];
        dy[t] = 2.0f * e / (float)count;
        lsum += (double)e * (double)e;
      }
      b4 += dy;
    }
    bf16x4 dyp = mlp_pack(dy[0], dy[1], dy[2], dy[3]);
    put_tiles<1>(tr, &dyp, fg + T_DY * T_ELEM, l);
    // layer 3
#pragma unroll
    for (int nt = 0; nt < 8; nt++) {
      const floatx4 a = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(S.w.b.b4[nt * 64 + l], dyp, zero, 0, 0, 0);
      acc[0][nt] = a * d3[nt];
      x[0][nt] = mlp_pack(acc[0][nt][0], acc[0][nt][1], acc[0][nt][2], acc[0][nt][3]);
    }
    sum16(acc[0], bs[2][0], bs[2][1], l);
    put_tiles<4>(tr, &x[0][0], fg + T_D3 * T_ELEM, l);
    put_tiles<4>(tr, &x[0][4], fg + (T_D3 + 4) * T_ELEM, l);
    // layer 2
#pragma unroll
    for (int nt = 0; nt < 8; nt++) acc[0][nt] = zero;
    mlp_prod(acc, x, S.w.b.b3, l);
#pragma unroll
    for (int nt = 0; nt < 8; nt++) {
      acc[0][nt] = acc[0][nt] * d2[nt];
      x[0][nt] = mlp_pack(acc[0][nt][0], acc[0][nt][1], acc[0][nt][2], acc[0][nt][3]);
    }
    sum16(acc[0], bs[1][0], bs[1][1], l);
    put_tiles<4>(tr, &x[0][0], fg + T_D2 * T_ELEM, l);
    put_tiles<4>(tr, &x[0][4], fg + (T_D2 + 4) * T_ELEM, l);
    // layer 1
#pragma unroll
    for (int nt = 0; nt < 8; nt++) {
      d1[nt] = *(const floatx4 *)(dk + nt * 256 + 4 * l);
      acc[0][nt] = zero;
    }
    mlp_prod(acc, x, S.w.b.b2, l);
#pragma unroll
    for (int nt = 0; nt < 8; nt++) {
      acc[0][nt] = acc[0][nt] * d1[nt];
      x[0][nt] = mlp_pack(acc[0][nt][0], acc[0][nt][1], acc[0][nt][2], acc[0][nt][3]);
    }
    sum16(acc[0], bs[0][0], bs[0][1], l);
    put_tiles<4>(tr, &x[0][0], fg + T_D1 * T_ELEM, l);
    put_tiles<4>(tr, &x[0][4], fg + (T_D1 + 4) * T_ELEM, l);
    if (g == ngroups - 1 && (ngroups & 1))  // k_wgrad takes groups in pairs
      for (int q = 0; q < T_N; q++) *(bf16x4 *)(fg + (T_N + q) * T_ELEM + 4 * l) = bf16x4{0, 0, 0, 0};
  }
  // partial sums: the wavefronts', then the workgroup's
  const int l = l0;
  for (int o = 8; o > 0; o >>= 1) {
    lsum += __shfl_down(lsum, o, 16);
#pragma unroll
    for (int t = 0; t < 4; t++) b4[t] += __shfl_down(b4[t], o, 16);
  }
  __syncthreads();
  float *red = (float *)&S.tr[0][0][0];  // 8 x TP_N floats fit the transposes' space
  static_assert(offsetof(TrainLds, tr) % 8 == 0, "k_train: the loss's place");
  static_assert(MLP_WAVES * TP_N * sizeof(float) <= sizeof(S.tr), "k_train: partial sums");
  const int f = 2 * (l & 15);  // this lane's two values of sum16: 16nt + 4(l/16) + t
#pragma unroll
  for (int q = 0; q < 3; q++)
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const int v = f + e;
      red[w * TP_N + q * MLP_H + 16 * (v >> 2) + 4 * (l >> 4) + (v & 3)] = bs[q][e];
    }
  if (l == 0) {
    for (int t = 0; t < 4; t++) red[w * TP_N + 3 * MLP_H + t] = b4[t];
    *(double *)(red + w * TP_N + TP_LOSS) = lsum;
  }
  __syncthreads();
  if (tid < TP_LOSS) {
    float s = 0.0f;
    for (int q = 0; q < MLP_WAVES; q++) s += red[q * TP_N + tid];
    part[(int64_t)blockIdx.x * TP_N + tid] = s;
  } else if (tid == TP_LOSS) {
    double s = 0.0;
    for (int q = 0; q < MLP_WAVES; q++) s += *(const double *)(red + q * TP_N + tid);
    *(double *)(part + (int64_t)blockIdx.x * TP_N + tid) = s;
  }
}

// One weight gradient over a range of pairs of groups: dW(in, out) = sum over
// samples of a(in) d(out), MA x NB tiles per wavefront, 32 samples a step (the
// lane's four of either group; the same order of samples in both operands).
template <int MA, int NB>
__device__ __forceinline__ void wgrad(const unsigned short *__restrict__ frag, int64_t p0, int64_t p1, int ta, int tb,
                                      float *out, int ld, int min_, int nout, int l) {
  floatx4 acc[MA][NB];
#pragma unroll
  for (int a = 0; a < MA; a++)
#pragma unroll
    for (int b = 0; b < NB; b++) acc[a][b] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  // the workspace holds whole pairs, the group after an odd last one zeroed.
  // The next step's operands load while this one's instructions run.
  bf16x8 av[MA], bv[NB], an[MA], bn[NB];
  auto fetch = [&](int64_t p, bf16x8 (&a_)[MA], bf16x8 (&b_)[NB]) {
    const unsigned short *g0 = frag + 2 * p * (T_N * T_ELEM) + 4 * l, *g1 = g0 + T_N * T_ELEM;
#pragma unroll
    for (int a = 0; a < MA; a++)
      a_[a] = mlp_join(*(const bf16x4 *)(g0 + (ta + a) * T_ELEM), *(const bf16x4 *)(g1 + (ta + a) * T_ELEM));
#pragma unroll
    for (int b = 0; b < NB; b++)
      b_[b] = mlp_join(*(const bf16x4 *)(g0 + (tb + b) * T_ELEM), *(const bf16x4 *)(g1 + (tb + b) * T_ELEM));
  };
  if (p0 < p1) fetch(p0, av, bv);
  for (int64_t p = p0; p < p1; p++) {
    if (p + 1 < p1) fetch(p + 1, an, bn);
#pragma unroll
    for (int a = 0; a < MA; a++)
#pragma unroll
      for (int b = 0; b < NB; b++) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[a], bv[b], acc[a][b], 0, 0, 0);
#pragma unroll
    for (int a = 0; a < MA; a++) av[a] = an[a];
#pragma unroll
    for (int b = 0; b < NB; b++) bv[b] = bn[b];
  }
#pragma unroll
  for (int a = 0; a < MA; a++)
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int t = 0; t < 4; t++) {
        const int in = 16 * a + 4 * (l >> 4) + t, o = 16 * b + (l & 15);
        if (in < min_ && o < nout) out[in * ld + o] = acc[a][b][t];
      }
}

// The four weight gradients (blockIdx.y: W3, W2, W1, W4), each split over
// gridDim.x ranges of samples; bound by reading the 25.6 KB of operands a
// group (W2 and W3: a 64 x 64 quadrant per wavefront).
__global__ void __launch_bounds__(256) k_wgrad(const unsigned short *__restrict__ frag, int64_t ngroups,
                                               float *__restrict__ wpart) {
  const int l = (int)threadIdx.x & 63, w = (int)threadIdx.x >> 6;
  const int64_t np = (ngroups + 1) / 2, per = (np + gridDim.x - 1) / gridDim.x;
  const int64_t p0 = (int64_t)blockIdx.x * per, p1 = p0 + per < np ? p0 + per : np;
  float *out = wpart + (int64_t)blockIdx.x * MLP_NPARAM;
  const int m4 = 4 * (w & 1), n4 = 4 * (w >> 1);
  if (blockIdx.y == 0)
    wgrad<4, 4>(frag, p0, p1, T_H2 + m4, T_D3 + n4, out + OW3 + 16 * (m4 * MLP_H + n4), MLP_H, MLP_H, MLP_H, l);
  else if (blockIdx.y == 1)
    wgrad<4, 4>(frag, p0, p1, T_H1 + m4, T_D2 + n4, out + OW2 + 16 * (m4 * MLP_H + n4), MLP_H, MLP_H, MLP_H, l);
  else if (blockIdx.y == 2)
    wgrad<1, 2>(frag, p0, p1, T_X, T_D1 + 2 * w, out + OW1 + 32 * w, MLP_H, MLP_IN, MLP_H, l);
  else
    wgrad<2, 1>(frag, p0, p1, T_H3 + 2 * w, T_DY, out + OW4 + 32 * w * MLP_OUT, MLP_OUT, MLP_H, MLP_OUT, l);
}

// The gradients and the loss: every parameter's partial sums in order (64
// parameters a workgroup, its four wavefronts a quarter of the partials
// each).  Workgroup 0 also adds the loss, in double.
__global__ void __launch_bounds__(256) k_grad_final(const float *__restrict__ wpart, int splits,
                                                    const float *__restrict__ part, int nwg, int64_t count,
                                                    float *__restrict__ G, float *__restrict__ loss) {
  __shared__ float r[4][64];
  const int l = (int)threadIdx.x & 63, w = (int)threadIdx.x >> 6;
  const int i = (int)blockIdx.x * 64 + l;
  float s = 0.0f;
  if (i < MLP_NPARAM) {
    // a bias's sums come from k_train, a weight's from k_wgrad
    int col = -1;
    if (i >= OB1 && i < OW2) col = i - OB1;
    else if (i >= OB2 && i < OW3) col = MLP_H + i - OB2;
    else if (i >= OB3 && i < OW4) col = 2 * MLP_H + i - OB3;
    else if (i >= OB4) col = 3 * MLP_H + i - OB4;
    const int n = col < 0 ? splits : nwg;
    const float *src = col < 0 ? wpart + i : part + col;
    const int64_t ld = col < 0 ? MLP_NPARAM : TP_N;
    const int per = (n + 3) / 4, q1 = min(n, (w + 1) * per);
#pragma unroll 8
    for (int q = w * per; q < q1; q++) s += src[q * ld];
  }
  r[w][l] = s;
  __syncthreads();
  if (w == 0 && i < MLP_NPARAM) G[i] = ((r[0][l] + r[1][l]) + r[2][l]) + r[3][l];
  if (blockIdx.x == 0) {
    __shared__ double d[256];
    const int q = (int)threadIdx.x;  // nwg <= 256
    const double t = block_reduce256(q < nwg ? *(const double *)(part + (int64_t)q * TP_N + TP_LOSS) : 0.0, d, OpAdd());
    if (q == 0) loss[0] = (float)(t / (double)count);
  }
}

__global__ void __launch_bounds__(256) k_adam(float *__restrict__ p, const float *__restrict__ g,
                                              float *__restrict__ m1, float *__restrict__ m2, int n, float lr,
                                              float bc1, float bc2, MlpPack *__restrict__ pk) {
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i >= n) return;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1.0e-8f;
  const float gi = g[i];
  const float a = b1 * m1[i] + (1.0f - b1) * gi;
  const float b = b2 * m2[i] + (1.0f - b2) * gi * gi;
  m1[i] = a;
  m2[i] = b;
  const float v = p[i] - lr * (a / bc1) / (sqrtf(b / bc2) + eps);
  p[i] = v;
  mlp_pack_one(pk, i, v);
}

// fused inference over a row-major [n x 8] input, [n x 4] output
template <class LOAD, class PREP, class OUT>
__global__ void __launch_bounds__(512) k_mlp(const MlpPack *pk, const float *prm, int64_t n, LOAD load, PREP prep,
                                             OUT out) {
  mlp_tiles(pk, prm, n, nullptr, load, prep, out, (int)blockIdx.x, (int)gridDim.x);
}

// ------------------------------------------------------------ C ABI
static inline unsigned nb256(int64_t n) { return (unsigned)((n + 255) / 256); }

extern "C" int cm1g_mlp_nparams(int64_t *n) {
  ARGCHK(n, "cm1g_mlp_nparams: null argument");
  *n = MLP_NPARAM;
  return 0;
}

extern "C" int cm1g_mlp_destroy(cm1g_mlp *n) {
  if (!n) return 0;
  if (n->stream) hipStreamSynchronize(n->stream);
  void *bufs[] = {n->p, n->g, n->m1, n->m2, n->dnorm, n->pk, n->frag, n->part, n->wpart, n->keep, n->red};
  for (void *b : bufs)
    if (b) hipFree(b);
  if (n->stream) hipStreamDestroy(n->stream);
  delete n;
  return 0;
}

// the packed weights of the parameters as they are on the device
static int pack_params(cm1g_mlp *n) {
  hipLaunchKernelGGL(k_pack, dim3(nb256(MLP_NPARAM)), dim3(256), 0, n->stream, n->p, n->pk);
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(n->stream));
  return 0;
}

extern "C" int cm1g_mlp_create(uint64_t seed, cm1g_mlp **out) {
  ARGCHK(out, "cm1g_mlp_create: null argument");
  cm1g_mlp *n = new cm1g_mlp();
  bool ok = hipStreamCreate(&n->stream) == hipSuccess;
  ok = ok && hipMalloc((void **)&n->p, MLP_NPARAM * sizeof(float)) == hipSuccess;
  ok = ok && hipMalloc((void **)&n->g, MLP_NPARAM * sizeof(float)) == hipSuccess;
  ok = ok && hipMalloc((void **)&n->m1, MLP_NPARAM * sizeof(float)) == hipSuccess;
  ok = ok && hipMalloc((void **)&n->m2, MLP_NPARAM * sizeof(float)) == hipSuccess;
  ok = ok && hipMalloc((void **)&n->dnorm, MLP_NNORM * sizeof(float)) == hipSuccess;
  ok = ok && hipMalloc((void **)&n->pk, sizeof(MlpPack)) == hipSuccess;
  ok = ok && hipMemset(n->pk, 0, sizeof(MlpPack)) == hipSuccess;
  if (!ok) {
    cm1g_mlp_destroy(n);
    cm1g_set_error("cm1g_mlp_create: allocation failed");
    return CM1G_E_HIP;
  }
  // He-uniform weights (fan-in), zero biases; identity normalisation
  std::vector<float> p(MLP_NPARAM, 0.0f);
  std::mt19937_64 rng(seed);
  auto fill = [&](int off, int fin, int fout) {
    const float a = std::sqrt(6.0f / (float)fin);
    std::uniform_real_distribution<float> u(-a, a);
    for (int i = 0; i < fin * fout; i++) p[off + i] = u(rng);
  };
  fill(OW1, MLP_IN, MLP_H);
  fill(OW2, MLP_H, MLP_H);
  fill(OW3, MLP_H, MLP_H);
  fill(OW4, MLP_H, MLP_OUT);
  std::vector<float> nm(MLP_NNORM, 0.0f);
  for (int k = 0; k < MLP_IN; k++) nm[MLP_IN + k] = 1.0f;
  for (int k = 0; k < MLP_OUT; k++) nm[2 * MLP_IN + MLP_OUT + k] = 1.0f;
  for (int k = 0; k < MLP_IN; k++) {
    nm[NM_XLO + k] = -8.0f;
    nm[NM_XHI + k] = 8.0f;
  }
  std::vector<float> z(MLP_NPARAM, 0.0f);
  ok = hipMemcpy(n->p, p.data(), MLP_NPARAM * sizeof(float), hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(n->m1, z.data(), MLP_NPARAM * sizeof(float), hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(n->m2, z.data(), MLP_NPARAM * sizeof(float), hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(n->g, z.data(), MLP_NPARAM * sizeof(float), hipMemcpyHostToDevice) == hipSuccess &&
       hipMemcpy(n->dnorm, nm.data(), MLP_NNORM * sizeof(float), hipMemcpyHostToDevice) == hipSuccess;
  ok = ok && pack_params(n) == 0;
  if (!ok) {
    cm1g_mlp_destroy(n);
    cm1g_set_error("cm1g_mlp_create: upload failed");
    return CM1G_E_HIP;
  }
  *out = n;
  return 0;
}

extern "C" int cm1g_mlp_get_params(cm1g_mlp *n, float *host) {
  ARGCHK(n && host, "cm1g_mlp_get_params: null argument");
  HIPCHK(hipStreamSynchronize(n->stream));
  HIPCHK(hipMemcpy(host, n->p, MLP_NPARAM * sizeof(float), hipMemcpyDeviceToHost));
  return 0;
}

extern "C" int cm1g_mlp_set_params(cm1g_mlp *n, const float *host) {
  ARGCHK(n && host, "cm1g_mlp_set_params: null argument");
  HIPCHK(hipStreamSynchronize(n->stream));
  HIPCHK(hipMemcpy(n->p, host, MLP_NPARAM * sizeof(float), hipMemcpyHostToDevice));
  return pack_params(n);
}

extern "C" int cm1g_mlp_set_norm(cm1g_mlp *n, const float *norm) {
  ARGCHK(n && norm, "cm1g_mlp_set_norm: null argument");
  for (int k = 0; k < MLP_IN; k++) ARGCHK(norm[MLP_IN + k] > 0.0f, "cm1g_mlp_set_norm: xstd must be > 0");
  for (int k = 0; k < MLP_OUT; k++)
    ARGCHK(norm[2 * MLP_IN + MLP_OUT + k] > 0.0f, "cm1g_mlp_set_norm: ystd must be > 0");
  for (int k = 0; k < MLP_IN; k++)
    ARGCHK(norm[NM_XLO + k] < norm[NM_XHI + k], "cm1g_mlp_set_norm: xlo must be < xhi");
  HIPCHK(hipStreamSynchronize(n->stream));
  HIPCHK(hipMemcpy(n->dnorm, norm, MLP_NNORM * sizeof(float), hipMemcpyHostToDevice));
  return 0;
}

extern "C" int cm1g_mlp_forward(cm1g_mlp *n, const float *x, int64_t rows, float *y) {
  ARGCHK(n && x && y && rows >= 0, "cm1g_mlp_forward: bad argument");
  if (rows == 0) return 0;
  auto load = [=] __device__(int64_t s, float *r) {
    for (int k = 0; k < MLP_IN; k++) r[k] = x[s * MLP_IN + k];
  };
  auto prep = [=] __device__(int64_t, const float *r, float *v) {
    for (int k = 0; k < MLP_IN; k++) v[k] = r[k];
  };
  auto out = [=] __device__(int64_t s, const float *v, const float *) {
    for (int k = 0; k < MLP_OUT; k++) y[s * MLP_OUT + k] = v[k];
  };
  const int64_t groups = (rows + 16 * MLP_G * MLP_WAVES - 1) / (16 * MLP_G * MLP_WAVES);
  const int nbx = (int)(groups < 1024 ? groups : 1024);
  hipLaunchKernelGGL((k_mlp<decltype(load), decltype(prep), decltype(out)>), dim3(nbx), dim3(512), 0, n->stream,
                     n->pk, n->p, rows, load, prep, out);
  HIPCHK(hipGetLastError());
  return 0;
}

// k_train's workgroups (one per CU: the weights of both directions fill its
// LDS) and k_wgrad's ranges of samples
constexpr int TRAIN_WGS = 256, WGRAD_SPLITS = 64;

static int ensure_workspace(cm1g_mlp *n, int64_t rows) {
  struct {
    float **p;
    size_t n;
  } fixed[] = {{&n->part, (size_t)TRAIN_WGS * TP_N},
               {&n->wpart, (size_t)WGRAD_SPLITS * MLP_NPARAM},
               {&n->keep, (size_t)TRAIN_WGS * MLP_WAVES * MLP_H * 16},
               {&n->red, 1}};
  for (auto &f : fixed)
    if (!*f.p) HIPCHK(hipMalloc((void **)f.p, f.n * sizeof(float)));
  if (rows <= n->cap) return 0;
  HIPCHK(hipStreamSynchronize(n->stream));
  if (n->frag) hipFree(n->frag);
  n->frag = nullptr;
  n->cap = 0;
  const size_t groups = (size_t)((rows + 31) / 32) * 2;  // whole pairs
  HIPCHK(hipMalloc((void **)&n->frag, groups * T_N * T_ELEM * sizeof(unsigned short)));
  n->cap = rows;
  return 0;
}

// loss and gradients (into n->g) of one batch
extern "C" int cm1g_mlp_loss_grad(cm1g_mlp *n, const float *x, const float *t, int64_t rows, float *loss,
                                  float *grad) {
  ARGCHK(n && x && t && rows >= 1 && rows <= (1 << 24), "cm1g_mlp_loss_grad: bad argument");
  int rc = ensure_workspace(n, rows);
  if (rc) return rc;
  hipStream_t st = n->stream;
  const int64_t groups = (rows + 15) / 16, pairs = (groups + 1) / 2;
  const int nwg = (int)std::min<int64_t>(TRAIN_WGS, (groups + MLP_WAVES - 1) / MLP_WAVES);
  const int splits = (int)std::min<int64_t>(WGRAD_SPLITS, pairs);
  hipLaunchKernelGGL(k_train, dim3(nwg), dim3(512), 0, st, n->pk, n->p, x, t, rows, groups, n->frag, n->part, n->keep);
  hipLaunchKernelGGL(k_wgrad, dim3(splits, 4), dim3(256), 0, st, n->frag, groups, n->wpart);
  hipLaunchKernelGGL(k_grad_final, dim3((MLP_NPARAM + 63) / 64), dim3(256), 0, st, n->wpart, splits, n->part, nwg,
                     rows * MLP_OUT, n->g, n->red);
  HIPCHK(hipGetLastError());
  if (loss) {
    HIPCHK(hipMemcpyAsync(loss, n->red, sizeof(float), hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
  }
  if (grad) {
    HIPCHK(hipStreamSynchronize(st));
    HIPCHK(hipMemcpy(grad, n->g, MLP_NPARAM * sizeof(float), hipMemcpyDeviceToHost));
  }
  return 0;
}

extern "C" int cm1g_mlp_adam(cm1g_mlp *n, float lr) {
  ARGCHK(n && lr > 0.0f, "cm1g_mlp_adam: bad argument");
  n->adam_t++;
  const float bc1 = 1.0f - std::pow(0.9f, (float)n->adam_t), bc2 = 1.0f - std::pow(0.999f, (float)n->adam_t);
  hipLaunchKernelGGL(k_adam, dim3(nb256(MLP_NPARAM)), dim3(256), 0, n->stream, n->p, n->g, n->m1, n->m2,
                     MLP_NPARAM, lr, bc1, bc2, n->pk);
  HIPCHK(hipGetLastError());
  return 0;
}

extern "C" int cm1g_mlp_sync(cm1g_mlp *n) {
  ARGCHK(n, "cm1g_mlp_sync: null argument");
  HIPCHK(hipStreamSynchronize(n->stream));
  return 0;
}
