// libimx learned correction: per-edge MLP 48 -> 128 -> 128 -> 128 -> 2 with
// GELU (tanh form), BF16 weights and activations on MFMA, FP32 accumulation;
// hand-written inference, training (forward + backward), weight-gradient and
// AdamW kernels.
//
// Register-resident layers. v_mfma_f32_16x16x16_bf16 takes, per lane l,
//   A[m = l%16][k = 4(l/16)+i], B[k = 4(l/16)+i][n = l%16], and returns
//   D[m = 4(l/16)+i][n = l%16]                       (i = 0..3).
// Every layer is evaluated transposed, Z^T(features x edges) = W^T A^T, with
// weights as the A operand and the 16 edges of a wave as the columns. The D
// fragment of output-feature tile t is then exactly the B fragment of input
// chunk t of the next layer, so activations never leave registers between
// layers. The backward data pass (dA^T = W dZ^T) has the same shape with a
// second, transposed weight fragment set. Weight gradients
// dW = A^T(features x edges) . dZ(edges x features) contract over edges, in
// the same kernel, from LDS.
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>

#include <cmath>
#include <cstring>
#include <new>
#include <string>
#include <vector>

#include "imx_device.h"

#include "imx_mlp_dev.h"

// load the 3 input fragments of 16 edges (rows of X, 48 bf16 each)
__device__ __forceinline__ void load_x(const short *__restrict__ X, int64_t e0, int64_t n, int lane,
                                       v4s (&x)[3]) {
  const int64_t e = e0 + (lane % 16);
#pragma unroll
  for (int kc = 0; kc < 3; ++kc) {
    if (e < n) x[kc] = *reinterpret_cast<const v4s *>(X + e * MLP_IN + kc * 16 + 4 * (lane / 16));
    else x[kc] = v4s{0, 0, 0, 0};
  }
}

// Training pass: forward, weighted MSE loss
//   L = sum_e w_e sum_o (y_eo - t_eo)^2,
// backward through every layer, and the weight and bias gradients, in one
// kernel. Output o with bit o of gmask set takes T[e][o] as dL/dy_eo itself
// (a loss defined outside the network, e.g. through a divergence) and adds
// nothing to the loss.
//
// A block takes 64 edges at a time. Four of its eight waves, 16 edges each,
// evaluate the layers forward and backward and leave the layer inputs
// A0 = X .. A3 and the pre-activation gradients dZ1 .. dZ4 in LDS,
// feature-major (the transposition the weight gradients need). The other four
// contract them over the 64 edges, one phase behind, with the gradient tiles
// in accumulators over all of the block's edges, and fetch the next layer's
// weight fragments into LDS while one layer runs. The block writes its
// gradient once; the optimiser kernel sums the blocks' partials in order.
//   gradient wave g: output tiles 2g, 2g + 1 of layers 1-3 with all input
//   tiles, input tiles 2g, 2g + 1 of layer 4; biases as products with ones.
// One block per CU (161 KB of LDS), two waves per SIMD: one busy with
// activations, one with MFMAs and LDS.
//
// Against the form that stored A and dZ in memory (1.7 KB per edge, in
// 32-byte pieces) and contracted them in a second and third kernel: 754 us ->
// 90 at glevel 6 (122,886 edges; 320 TFLOP/s). What bounds it now is one
// layer wave's own chain of LDS reads, MFMAs and activations, 29 k cycles a
// batch, of which the matrix cores are busy 6 k. With both roles in four waves the
// accumulators and the layers in flight spilled, and every wait for a spilled
// value or a bias also waited for the weights on their way: 282 us. The
// derivative is formed with the activation and shares its exponential and
// reciprocal.
#define TR_STRIDE 68  // bf16 per LDS row: 64 edges and a pad of 8 bytes
#define TR_A 0        // rows: layer inputs 48 + 3 x 128
#define TR_DA 432     // dZ of layers 3 and 1
#define TR_DB 560     // dZ of layer 2
#define TR_D4 688     // dZ4, 16 rows of which 2 are live
#define TR_ROWS 704
#define TR_BLOCKS 256
#define TR_ILV 4     // MFMA chains a wave runs side by side
#define TR_THREADS (2 * 64 * MLP_WAVES)

// activation (BF16, as the next layer's input) and its derivative
__device__ __forceinline__ v4s gelu_both(const v4f &z, v4f &d) {
  float g[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float x = z[i], s = gelu_s(x);
    g[i] = x * s;
    float t = s + g[i] * (1.0f - s) * GELU_C2 * __builtin_fmaf(3.0f * GELU_A, x * x, 1.0f);
    asm volatile("" : "+v"(t));  // now: left to its use, x and s would be kept instead
    d[i] = t;
  }
  uint32_t p[2] = {f2bf2(g[0], g[1]), f2bf2(g[2], g[3])};
  return __builtin_bit_cast(v4s, p);
}

// rows 16 t + 4 (lane / 16) + i of one edge column
__device__ __forceinline__ void put_rows(short *lds, int row0, int col, int lane, v4s v) {
  short *p = lds + (row0 + 4 * (lane / 16)) * TR_STRIDE + col;
#pragma unroll
  for (int i = 0; i < 4; ++i) p[i * TR_STRIDE] = v[i];
}
// One hidden layer of 16 edges, a tile of 16 features at a time: pre-activations
// from fragments Wf[(n*KT + kc)*64 + lane] and input fragments xin[kc], the
// activation (to the next layer and to rows row0 of LDS) and its derivative.
template <int KT>
__device__ __forceinline__ void layer_act(const v4s *Wf, const float *b, const v4s (&xin)[KT], v4s (&a)[8], v4f (&d)[8],
                                          short *lds, int row0, int col, int lane) {
#pragma unroll
  for (int n = 0; n < 8; n += TR_ILV) {  // independent chains side by side
    v4f z[TR_ILV];
#pragma unroll
    for (int q = 0; q < TR_ILV; ++q) z[q] = *reinterpret_cast<const v4f *>(b + (n + q) * 16 + 4 * (lane / 16));
#pragma unroll
    for (int kc = 0; kc < KT; ++kc)
#pragma unroll
      for (int q = 0; q < TR_ILV; ++q) z[q] = mfma(Wf[((n + q) * KT + kc) * 64 + lane], xin[kc], z[q]);
#pragma unroll
    for (int q = 0; q < TR_ILV; ++q) {
      a[n + q] = gelu_both(z[q], d[n + q]);
      put_rows(lds, row0 + 16 * (n + q), col, lane, a[n + q]);
    }
  }
}
// K32 operand: row lane % 16 of a 16-row tile, 8 edges of chunk c
__device__ __forceinline__ v8s get_rows(const short *lds, int row0, int c, int lane) {
  const v4s *p = reinterpret_cast<const v4s *>(lds + (row0 + lane % 16) * TR_STRIDE + 32 * c + 8 * (lane / 16));
  return __builtin_shufflevector(p[0], p[1], 0, 1, 2, 3, 4, 5, 6, 7);
}

// gradient tiles of one layer: MT input tiles x NB output tiles of this wave
template <int MT, int NB>
__device__ __forceinline__ void grad_tiles(const short *lds, int a_row, int dz_row, int lane, v4f (&acc)[NB][MT],
                                           v4f (&bias)[NB]) {
  const short one = 0x3F80;
  const v8s ones = {one, one, one, one, one, one, one, one};
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    v8s dz[NB];
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      dz[q] = get_rows(lds, dz_row + 16 * q, c, lane);
      bias[q] = mfma32(ones, dz[q], bias[q]);
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const v8s x = get_rows(lds, a_row + 16 * m, c, lane);
#pragma unroll
      for (int q = 0; q < NB; ++q) acc[q][m] = mfma32(x, dz[q], acc[q][m]);
    }
  }
}

// dz (128 features) = (W dZ_next) g'(z): one layer of the backward pass
template <int KT>
__device__ __forceinline__ void back_layer(const v4s *__restrict__ Wb, const v4s (&dzn)[KT], const v4f (&d)[8],
                                           v4s (&dz)[8], int lane) {
#pragma unroll
  for (int m = 0; m < 8; m += TR_ILV) {
    v4f acc[TR_ILV];
#pragma unroll
    for (int q = 0; q < TR_ILV; ++q) acc[q] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kc = 0; kc < KT; ++kc)
#pragma unroll
      for (int q = 0; q < TR_ILV; ++q) acc[q] = mfma(Wb[((m + q) * KT + kc) * 64 + lane], dzn[kc], acc[q]);
#pragma unroll
    for (int q = 0; q < TR_ILV; ++q) {
      const v4f g = acc[q] * d[m + q];
      uint32_t p[2] = {f2bf2(g[0], g[1]), f2bf2(g[2], g[3])};
      dz[m + q] = __builtin_bit_cast(v4s, p);
    }
  }
}

// One layer's weight fragments from memory straight to LDS (16 bytes per lane,
// no registers), a quarter of them by each of four waves; in flight until
// the wave's s_waitcnt.
template <int COUNT>
__device__ __forceinline__ void tr_fetch(const short *__restrict__ src, short *dst, int wave) {
  constexpr int kWave = COUNT / MLP_WAVES;  // bf16 per wave
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < kWave; i += 512)
    __builtin_amdgcn_global_load_lds(
        (const __attribute__((address_space(1))) void *)(src + wave * kWave + i + lane * 8),
        (__attribute__((address_space(3))) void *)(dst + wave * kWave + i), 16, 0, 0);
}
__device__ __forceinline__ void tr_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

__global__ __launch_bounds__(TR_THREADS) void mlp_train(
    int64_t n, int nbatch, const short *__restrict__ X, const float *__restrict__ T,
    const float *__restrict__ w, int gmask, const short *__restrict__ Wf, const short *__restrict__ Wb,
    const float *__restrict__ P, float *__restrict__ part, float *__restrict__ loss_part) {
  __shared__ __align__(16) short lds[TR_ROWS * TR_STRIDE];
  __shared__ __align__(16) short wbuf[2][MLP_H * MLP_H];  // the layer in use and the next
  __shared__ __align__(16) float lb[3 * MLP_H];           // biases of layers 1-3
  __shared__ float lred[MLP_WAVES];
  const int lane = threadIdx.x & 63;
  const int role = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = role & (MLP_WAVES - 1);
  const v4f zero = {0.f, 0.f, 0.f, 0.f};
  for (int i = threadIdx.x; i < 3 * MLP_H; i += TR_THREADS)
    lb[i] = P[(i < MLP_H ? P_B1 : i < 2 * MLP_H ? P_B2 - MLP_H : P_B3 - 2 * MLP_H) + i];
  // Both roles pass the same barriers: one before the loop, five per batch,
  // one after it. wbuf[cur] holds layers 1 and 3 forward and 2 backward.
  int cur = 0;
  if (role < MLP_WAVES) {  // layers
    const int col = 16 * wave + lane % 16;
    const v4s *W4 = reinterpret_cast<const v4s *>(Wf + FF_4), *B4 = reinterpret_cast<const v4s *>(Wb + FB_4);
    v4s w4[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) w4[k] = W4[k * 64 + lane];
    const float y0 = lane < 16 ? P[P_B4] : 0.f, y1 = lane < 16 ? P[P_B4 + 1] : 0.f;
    auto frag = [&](int which) { return reinterpret_cast<const v4s *>(wbuf[which]); };
    __syncthreads();
    for (int b = blockIdx.x; b < nbatch; b += gridDim.x) {
      const int64_t e = (int64_t)b * 64 + col;
      const bool live = lane < 16 && e < n;
      v4s x[3];
      load_x(X, (int64_t)b * 64 + 16 * wave, n, lane, x);
      const float we = live ? w[e] : 0.f, t0 = live ? T[e * 2] : 0.f, t1 = live ? T[e * 2 + 1] : 0.f;
      v4f d1[8], d2[8], d3[8];
      v4s a1[8], a2[8];
      __syncthreads();  // layer 1's weights
      layer_act<3>(frag(cur), lb, x, a1, d1, lds, TR_A + 48, col, lane);
      __syncthreads();  // layer 2's; the previous batch's layer-1 gradient has read X
#pragma unroll
      for (int kc = 0; kc < 3; ++kc) put_rows(lds, TR_A + kc * 16, col, lane, x[kc]);
      layer_act<8>(frag(cur ^ 1), lb + MLP_H, a1, a2, d2, lds, TR_A + 176, col, lane);
      __syncthreads();  // layer 3's
      layer_act<8>(frag(cur), lb + 2 * MLP_H, a2, a1, d3, lds, TR_A + 304, col, lane);
      v4f y = {y0, y1, 0.f, 0.f};
#pragma unroll
      for (int kc = 0; kc < 8; ++kc) y = mfma(w4[kc], a1[kc], y);
      // dL/dy (features 0,1 live in lanes 0..15, elements 0,1)
      v4s dz4[1] = {{0, 0, 0, 0}};
      float lsum = 0.f;
      if (live) {
        const float r0 = y[0] - t0, r1 = y[1] - t1;
        lsum = ((gmask & 1) ? 0.f : we * r0 * r0) + ((gmask & 2) ? 0.f : we * r1 * r1);
        dz4[0][0] = f2bf((gmask & 1) ? t0 : 2.f * we * r0);
        dz4[0][1] = f2bf((gmask & 2) ? t1 : 2.f * we * r1);
      }
      put_rows(lds, TR_D4, col, lane, dz4[0]);
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) lsum += __shfl_xor(lsum, off, 64);
      if (lane == 0) lred[wave] = lsum;
      v4s dz[8], dzn[8];
      back_layer<1>(B4, dz4, d3, dz, lane);
#pragma unroll
      for (int t = 0; t < 8; ++t) put_rows(lds, TR_DA + 16 * t, col, lane, dz[t]);
      __syncthreads();  // layer 3's backward; A, dZ4, dZ3 to the gradients
      if (threadIdx.x == 0) {
        float s = 0.f;
        for (int q = 0; q < MLP_WAVES; ++q) s += lred[q];
        loss_part[b] = s;
      }
      back_layer<8>(frag(cur ^ 1), dz, d2, dzn, lane);
#pragma unroll
      for (int t = 0; t < 8; ++t) put_rows(lds, TR_DB + 16 * t, col, lane, dzn[t]);
      __syncthreads();  // layer 2's backward; dZ2; dZ3 is read: its rows take dZ1
      back_layer<8>(frag(cur), dzn, d1, dz, lane);
#pragma unroll
      for (int t = 0; t < 8; ++t) put_rows(lds, TR_DA + 16 * t, col, lane, dz[t]);
      cur ^= 1;
    }
    __syncthreads();
    return;
  }

  // gradients and weight fetches
  v4f g1[2][3], g2[2][8], g3[2][8], g4[1][2], b1[2], b2[2], b3[2], b4[1];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    b1[q] = b2[q] = b3[q] = g4[0][q] = zero;
#pragma unroll
    for (int m = 0; m < 8; ++m) g2[q][m] = g3[q][m] = zero;
#pragma unroll
    for (int m = 0; m < 3; ++m) g1[q][m] = zero;
  }
  b4[0] = zero;
  tr_fetch<MLP_IN * MLP_H>(Wf + FF_1, wbuf[0], wave);
  __syncthreads();
  for (int b = blockIdx.x; b < nbatch; b += gridDim.x) {
    tr_wait();
    __syncthreads();  // layer 1 runs
    tr_fetch<MLP_H * MLP_H>(Wf + FF_2, wbuf[cur ^ 1], wave);
    if (b != blockIdx.x) grad_tiles<3, 2>(lds, TR_A, TR_DA + 32 * wave, lane, g1, b1);
    tr_wait();
    __syncthreads();  // layer 2
    tr_fetch<MLP_H * MLP_H>(Wf + FF_3, wbuf[cur], wave);
    tr_wait();
    __syncthreads();  // layers 3 and 4, dZ3
    tr_fetch<MLP_H * MLP_H>(Wb + FB_3, wbuf[cur ^ 1], wave);
    tr_wait();
    __syncthreads();  // dZ2
    tr_fetch<MLP_H * MLP_H>(Wb + FB_2, wbuf[cur], wave);
    grad_tiles<2, 1>(lds, TR_A + 304 + 32 * wave, TR_D4, lane, g4, b4);
    grad_tiles<8, 2>(lds, TR_A + 176, TR_DA + 32 * wave, lane, g3, b3);
    tr_wait();
    __syncthreads();  // dZ1
    tr_fetch<MLP_IN * MLP_H>(Wf + FF_1, wbuf[cur ^ 1], wave);  // of the next batch
    grad_tiles<8, 2>(lds, TR_A + 48, TR_DB + 32 * wave, lane, g2, b2);
    cur ^= 1;
  }
  tr_wait();  // the last fetch, which no batch uses
  __syncthreads();
  grad_tiles<3, 2>(lds, TR_A, TR_DA + 32 * wave, lane, g1, b1);
  // the block's partial: D[in = 16 mt + 4 (l/16) + i][out = 16 nt + l % 16]
  float *q = part + (int64_t)blockIdx.x * P_N;
  const int in0 = 4 * (lane / 16), lo = lane % 16;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int out = 32 * wave + 16 * k + lo;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int m = 0; m < 3; ++m) q[P_W1 + (16 * m + in0 + i) * MLP_H + out] = g1[k][m][i];
#pragma unroll
      for (int m = 0; m < 8; ++m) {
        q[P_W2 + (16 * m + in0 + i) * MLP_H + out] = g2[k][m][i];
        q[P_W3 + (16 * m + in0 + i) * MLP_H + out] = g3[k][m][i];
      }
      if (lo < MLP_OUT) q[P_W4 + (32 * wave + 16 * k + in0 + i) * MLP_OUT + lo] = g4[0][k][i];
    }
    if (lane < 16) {
      q[P_B1 + out] = b1[k][0];
      q[P_B2 + out] = b2[k][0];
      q[P_B3 + out] = b3[k][0];
    }
  }
  if (wave == 0 && lane < MLP_OUT) q[P_B4 + lane] = b4[0][0];
}

// The places of weight (row, col) of a layer in the fragment copies (the
// inverse of mlp_pack's maps; layer 0-3, N output features)
__device__ __forceinline__ void put_weight(int layer, int row, int col, short v, short *Ff, short *Fb, short *Ff32,
                                           short *F1g) {
  const int KT = layer == 0 ? 3 : 8;
  const int fbase = layer == 0 ? FF_1 : layer == 1 ? FF_2 : layer == 2 ? FF_3 : FF_4;
  Ff[fbase + (((col / 16) * KT + row / 16) * 64 + (row % 16) / 4 * 16 + col % 16) * 4 + row % 4] = v;
  if (layer > 0) {
    const int bbase = layer == 1 ? FB_2 : layer == 2 ? FB_3 : FB_4, KB = layer == 3 ? 1 : 8;
    Fb[bbase + (((row / 16) * KB + col / 16) * 64 + (col % 16) / 4 * 16 + row % 16) * 4 + col % 4] = v;
  }
  // K32: slot i of lane group g holds row kappa32(g, i) of its chunk
  const int r = row % 32, lane = (r % 16) / 4 * 16 + col % 16, i = r % 4 + (r < 16 ? 0 : 4);
  if (layer == 0) {
    Ff32[(col / 16) * 768 + (row < 32 ? lane * 8 + i : 512 + lane * 4 + row % 4)] = v;
    int g, s;
    mlp_feature_slot(row, &g, &s);
    const int gl = g * 16 + col % 16;
    F1g[(col / 16) * 768 + (s < 8 ? gl * 8 + s : 512 + gl * 4 + s - 8)] = v;
  } else
    Ff32[fbase + (col / 16) * 2048 + (row / 32) * 512 + lane * 8 + i] = v;
}

// AdamW (decoupled weight decay on the matrices, not the biases) on the sum
// of the blocks' partials, and the updated weights' places in the BF16
// fragment copies: 64 parameters per block, eight threads each over an eighth
// of the partials, added in a fixed order.
#define AW_GROUPS 8
__global__ __launch_bounds__(64 * AW_GROUPS) void mlp_adamw(int nsplit, const float *__restrict__ part,
                                                 float *__restrict__ P, float *__restrict__ M,
                                                 float *__restrict__ V, float *__restrict__ G, float lr,
                                                 float b1, float b2, float eps, float wd, float bc1,
                                                 float bc2, int apply, short *__restrict__ Ff,
                                                 short *__restrict__ Fb, short *__restrict__ Ff32,
                                                 short *__restrict__ F1g) {
  const int lane = threadIdx.x & 63, p = blockIdx.x * 64 + lane, grp = threadIdx.x >> 6;
  __shared__ float red[AW_GROUPS][64];
  float g = 0.f;
  if (p < P_N) {
#pragma unroll 8
    for (int s = grp; s < nsplit; s += AW_GROUPS) g += part[(int64_t)s * P_N + p];
  }
  red[grp][lane] = g;
  __syncthreads();
  if (grp || p >= P_N) return;
  g = 0.f;
#pragma unroll
  for (int k = 0; k < AW_GROUPS; ++k) g += red[k][lane];
  G[p] = g;
  if (!apply) return;
  const bool is_bias = (p >= P_B1 && p < P_W2) || (p >= P_B2 && p < P_W3) || (p >= P_B3 && p < P_W4) ||
                       p >= P_B4;
  const float m = b1 * M[p] + (1.f - b1) * g;
  const float v = b2 * V[p] + (1.f - b2) * g * g;
  M[p] = m;
  V[p] = v;
  float x = P[p];
  if (!is_bias) x -= lr * wd * x;
  x -= lr * (m / bc1) / (sqrtf(v / bc2) + eps);
  P[p] = x;
  if (is_bias) return;
  const int layer = p < P_W2 ? 0 : p < P_W3 ? 1 : p < P_W4 ? 2 : 3;
  const int q = p - (layer == 0 ? P_W1 : layer == 1 ? P_W2 : layer == 2 ? P_W3 : P_W4);
  const int N = layer == 3 ? MLP_OUT : MLP_H;
  put_weight(layer, q / N, q % N, f2bf(x), Ff, Fb, Ff32, F1g);
}

// fragment copies from the FP32 master (forward: W^T tiles; backward: W tiles)
// k-permutation of a K32 chunk: operand slot i of lane group g holds
// feature kappa(g, i) of the chunk (the inference kernel's B operand is the
// concatenation of two 16-feature activation tiles)
__device__ __forceinline__ int kappa32(int g, int i) { return i < 4 ? 4 * g + i : 16 + 4 * g + (i - 4); }

__global__ __launch_bounds__(256) void mlp_pack(const float *__restrict__ P, short *__restrict__ Ff,
                                                short *__restrict__ Fb, short *__restrict__ Ff32,
                                                short *__restrict__ F1g) {
  const int q = blockIdx.x * 256 + threadIdx.x;
  if (q < MLP_IN * MLP_H) {  // layer 1 for gathered features
    const int row = q / MLP_H, col = q % MLP_H;
    int g, s;
    mlp_feature_slot(row, &g, &s);
    const int gl = g * 16 + col % 16;
    F1g[(col / 16) * 768 + (s < 8 ? gl * 8 + s : 512 + gl * 4 + s - 8)] = f2bf(P[P_W1 + q]);
  }
  // inference (K32) fragments: index -> (layer, output tile, chunk, lane, i)
  if (q < FF_N) {
    int row, col, N, poff;
    if (q < FF_2) {  // layer 1: per output tile a K32 fragment then a K16 one
      const int nn = q / 768, s = q % 768;
      N = MLP_H;
      poff = P_W1;
      if (s < 512) {
        const int lane = s / 8, i = s % 8;
        row = kappa32(lane / 16, i);
        col = nn * 16 + lane % 16;
      } else {
        const int lane = (s - 512) / 4, i = (s - 512) % 4;
        row = 32 + 4 * (lane / 16) + i;
        col = nn * 16 + lane % 16;
      }
    } else {
      int base;
      if (q < FF_3) { base = FF_2; N = MLP_H; poff = P_W2; }
      else if (q < FF_4) { base = FF_3; N = MLP_H; poff = P_W3; }
      else { base = FF_4; N = MLP_OUT; poff = P_W4; }
      const int r = q - base;
      const int nn = r / 2048, c = (r / 512) % 4, lane = (r / 8) % 64, i = r % 8;
      row = 32 * c + kappa32(lane / 16, i);
      col = nn * 16 + lane % 16;
    }
    Ff32[q] = (col < N) ? f2bf(P[poff + row * N + col]) : (short)0;
  }
  // forward: index -> (layer, n, kc, lane, i)
  if (q < FF_N) {
    int base, K, N, poff, KT;
    int r = q;
    if (r < FF_2) { base = FF_1; K = MLP_IN; N = MLP_H; poff = P_W1; }
    else if (r < FF_3) { base = FF_2; K = MLP_H; N = MLP_H; poff = P_W2; }
    else if (r < FF_4) { base = FF_3; K = MLP_H; N = MLP_H; poff = P_W3; }
    else { base = FF_4; K = MLP_H; N = MLP_OUT; poff = P_W4; }
    r -= base;
    KT = K / 16;
    const int i = r & 3, lane = (r >> 2) & 63, tile = r >> 8;
    const int n = tile / KT, kc = tile % KT;
    const int row = kc * 16 + 4 * (lane / 16) + i;  // k (input feature)
    const int col = n * 16 + lane % 16;             // output feature
    Ff[q] = (col < N) ? f2bf(P[poff + row * N + col]) : (short)0;
  }
  if (q < FB_N) {
    int base, K, N, poff, KT;
    int r = q;
    if (r < FB_3) { base = FB_2; K = MLP_H; N = MLP_H; poff = P_W2; }
    else if (r < FB_4) { base = FB_3; K = MLP_H; N = MLP_H; poff = P_W3; }
    else { base = FB_4; K = MLP_H; N = MLP_OUT; poff = P_W4; }
    r -= base;
    KT = (N == MLP_OUT) ? 1 : N / 16;  // contraction over output features
    const int i = r & 3, lane = (r >> 2) & 63, tile = r >> 8;
    const int m = tile / KT, kc = tile % KT;
    const int row = m * 16 + lane % 16;            // input feature of the layer
    const int col = kc * 16 + 4 * (lane / 16) + i;  // output feature
    (void)K;
    Fb[q] = (col < N) ? f2bf(P[poff + row * N + col]) : (short)0;
  }
}

__global__ void f32_to_bf16(int64_t n, const float *__restrict__ x, short *__restrict__ y) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) y[i] = f2bf(x[i]);
}

// ================================================================= handle ==

namespace imx {

static int mlp_fail(hipError_t e, const char *what) {
  return set_error(IMX_EDEVICE, std::string(what) + ": " + hipGetErrorString(e));
}
#define MTRY(expr, what)                          \
  do {                                            \
    hipError_t _e = (expr);                       \
    if (_e != hipSuccess) return mlp_fail(_e, what); \
  } while (0)

int mlp_reserve(imx_mlp *m, int64_t n) {
  const int64_t npad = ((n + 63) / 64) * 64;
  if (npad <= m->cap) return IMX_OK;
  (void)hipFree(m->X);
  (void)hipFree(m->T);
  (void)hipFree(m->w);
  (void)hipFree(m->Y);
  (void)hipFree(m->Xf);
  (void)hipFree(m->lossp);
  m->X = nullptr;
  m->T = m->w = m->Y = m->Xf = m->lossp = nullptr;
  MTRY(hipMalloc(&m->X, npad * MLP_IN * 2), "mlp scratch");
  MTRY(hipMalloc(&m->T, npad * 2 * 4), "mlp scratch");
  MTRY(hipMalloc(&m->w, npad * 4), "mlp scratch");
  MTRY(hipMalloc(&m->Y, npad * 2 * 4), "mlp scratch");
  MTRY(hipMalloc(&m->Xf, npad * MLP_IN * 4), "mlp scratch");
  MTRY(hipMalloc(&m->lossp, (npad / 64 + 1) * 4), "mlp scratch");
  m->cap = npad;
  return IMX_OK;
}

// He-normal init of the matrices, zero biases (SplitMix64 + Box-Muller)
void mlp_initial_params(uint64_t seed, std::vector<float> &P) {
  P.assign(P_N, 0.f);
  uint64_t s = seed;
  auto next = [&]() {
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
  };
  auto normal = [&]() {
    const double u1 = ((next() >> 11) + 0.5) * (1.0 / 9007199254740992.0);
    const double u2 = ((next() >> 11) + 0.5) * (1.0 / 9007199254740992.0);
    return std::sqrt(-2.0 * std::log(u1)) * std::cos(6.283185307179586 * u2);
  };
  auto init = [&](int off, int fan_in, int count, double gain) {
    for (int i = 0; i < count; ++i) P[off + i] = (float)(normal() * gain * std::sqrt(2.0 / fan_in));
  };
  init(P_W1, MLP_IN, MLP_IN * MLP_H, 1.0);
  init(P_W2, MLP_H, MLP_H * MLP_H, 1.0);
  init(P_W3, MLP_H, MLP_H * MLP_H, 1.0);
  init(P_W4, MLP_H, MLP_H * MLP_OUT, 0.1);  // small output layer: starts near "no correction"
}

int mlp_pack_launch(imx_mlp *m) {
  const int n = FF_N > FB_N ? FF_N : FB_N;
  mlp_pack<<<(n + 255) / 256, 256, 0, m->stream>>>(m->P, m->Ff, m->Fb, m->Ff32, m->F1g);
  MTRY(hipGetLastError(), "mlp_pack");
  return IMX_OK;
}

// Forward on device buffers (X bf16 [n][48]) -> Y fp32 [n][2].
int mlp_forward_dev(imx_mlp *m, int64_t n, const short *X, float *Y, hipStream_t st) {
  if (n <= 0) return IMX_OK;
  MTRY(mlp_fwd_launch(m->Ff32, m->Ff32, m->P, n, RowLoader{X}, Y, st), "mlp_fwd_lds");
  return IMX_OK;
}

// One training pass on the device batch X (m->X when NULL), m->T, m->w (n
// edges), enqueued on m's stream; loss_part [(n + 63) / 64] takes the loss
// partials (m->lossp when NULL).
int mlp_train_dev(imx_mlp *m, int64_t n, const short *X, float lr, float wd, int apply, float *loss_part,
                  int gmask) {
  const int nbatch = (int)((n + 63) / 64), blocks = nbatch < TR_BLOCKS ? nbatch : TR_BLOCKS;
  hipStream_t st = m->stream;
  mlp_train<<<blocks, TR_THREADS, 0, st>>>(n, nbatch, X ? X : m->X, m->T, m->w, gmask, m->Ff, m->Fb, m->P,
                                               m->part, loss_part ? loss_part : m->lossp);
  MTRY(hipGetLastError(), "mlp_train");
  m->t += apply ? 1 : 0;
  const float b1 = 0.9f, b2 = 0.999f;
  const float bc1 = 1.f - powf(b1, (float)(m->t > 0 ? m->t : 1));
  const float bc2 = 1.f - powf(b2, (float)(m->t > 0 ? m->t : 1));
  mlp_adamw<<<(P_N + 63) / 64, 64 * AW_GROUPS, 0, st>>>(blocks, m->part, m->P, m->M, m->V, m->G, lr, b1, b2, 1e-8f,
                                                        wd, bc1, bc2, apply, m->Ff, m->Fb, m->Ff32, m->F1g);
  MTRY(hipGetLastError(), "mlp_adamw");
  return IMX_OK;
}

// Sum of the loss partials of passes over n edges (waits for m's stream).
int mlp_loss(imx_mlp *m, int64_t n, const float *loss_part, int passes, double *loss) {
  const int64_t nb = (n + 63) / 64;
  std::vector<float> lp((size_t)nb * passes);
  MTRY(hipMemcpyAsync(lp.data(), loss_part ? loss_part : m->lossp, lp.size() * 4, hipMemcpyDeviceToHost, m->stream),
       "loss");
  MTRY(hipStreamSynchronize(m->stream), "loss");
  for (int k = 0; k < passes; ++k) {
    double s = 0.0;
    for (int64_t b = 0; b < nb; ++b) s += lp[k * nb + b];
    loss[k] = s;
  }
  return IMX_OK;
}

}  // namespace imx

extern "C" {

int imx_mlp_create(uint64_t seed, imx_mlp **out) {
  if (!out) return imx::set_error(IMX_EINVAL, "imx_mlp_create: NULL out");
  *out = nullptr;
  imx_mlp *m = new (std::nothrow) imx_mlp();
  if (!m) return imx::set_error(IMX_ENOMEM, "imx_mlp_create: out of memory");
  std::vector<float> P;
  imx::mlp_initial_params(seed, P);
  int rc = IMX_OK;
  if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess ||
      hipMalloc(&m->P, P_N * 4) != hipSuccess || hipMalloc(&m->M, P_N * 4) != hipSuccess ||
      hipMalloc(&m->V, P_N * 4) != hipSuccess || hipMalloc(&m->G, P_N * 4) != hipSuccess ||
      hipMalloc(&m->part, (size_t)TR_BLOCKS * P_N * 4) != hipSuccess ||
      hipMalloc(&m->Ff, FF_N * 2) != hipSuccess || hipMalloc(&m->Fb, FB_N * 2) != hipSuccess ||
      hipMalloc(&m->Ff32, FF_N * 2) != hipSuccess || hipMalloc(&m->F1g, FF_2 * 2) != hipSuccess) {
    rc = imx::set_error(IMX_EDEVICE, "imx_mlp_create: device allocation failed");
  } else {
    (void)hipMemcpy(m->P, P.data(), P_N * 4, hipMemcpyHostToDevice);
    // the fills run on the null stream, which m->stream does not wait for
    (void)hipMemsetAsync(m->M, 0, P_N * 4, nullptr);
    (void)hipMemsetAsync(m->V, 0, P_N * 4, nullptr);
    (void)hipMemsetAsync(m->G, 0, P_N * 4, nullptr);
    (void)hipStreamSynchronize(nullptr);
    rc = imx::mlp_pack_launch(m);
    if (!rc && hipStreamSynchronize(m->stream) != hipSuccess)
      rc = imx::set_error(IMX_EDEVICE, "imx_mlp_create: pack failed");
  }
  if (rc) {
    imx_mlp_destroy(m);
    return rc;
  }
  *out = m;
  return IMX_OK;
}

int imx_mlp_nparams(void) { return P_N; }

int imx_mlp_get_params(imx_mlp *m, float *p) {
  if (!m || !p) return imx::set_error(IMX_EINVAL, "imx_mlp_get_params: NULL argument");
  if (hipMemcpy(p, m->P, P_N * 4, hipMemcpyDeviceToHost) != hipSuccess)
    return imx::set_error(IMX_EDEVICE, "imx_mlp_get_params: copy failed");
  return IMX_OK;
}

int imx_mlp_set_params(imx_mlp *m, const float *p) {
  if (!m || !p) return imx::set_error(IMX_EINVAL, "imx_mlp_set_params: NULL argument");
  if (hipMemcpy(m->P, p, P_N * 4, hipMemcpyHostToDevice) != hipSuccess)
    return imx::set_error(IMX_EDEVICE, "imx_mlp_set_params: copy failed");
  int rc = imx::mlp_pack_launch(m);
  if (rc) return rc;
  if (hipStreamSynchronize(m->stream) != hipSuccess) return imx::set_error(IMX_EDEVICE, "imx_mlp_set_params");
  return IMX_OK;
}

int imx_mlp_init(imx_mlp *m, uint64_t seed) {
  if (!m) return imx::set_error(IMX_EINVAL, "imx_mlp_init: NULL handle");
  std::vector<float> P;
  imx::mlp_initial_params(seed, P);
  if (hipStreamSynchronize(m->stream) != hipSuccess ||
      hipMemcpy(m->P, P.data(), P_N * 4, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemsetAsync(m->M, 0, P_N * 4, nullptr) != hipSuccess ||
      hipMemsetAsync(m->V, 0, P_N * 4, nullptr) != hipSuccess ||
      hipMemsetAsync(m->G, 0, P_N * 4, nullptr) != hipSuccess || hipStreamSynchronize(nullptr) != hipSuccess)
    return imx::set_error(IMX_EDEVICE, "imx_mlp_init: device copy failed");
  m->t = 0;
  int rc = imx::mlp_pack_launch(m);
  if (rc) return rc;
  if (hipStreamSynchronize(m->stream) != hipSuccess) return imx::set_error(IMX_EDEVICE, "imx_mlp_init");
  return IMX_OK;
}

// host-array entry points (tests, gradient check, small batches)
int imx_mlp_forward(imx_mlp *m, int64_t n, const float *X, float *Y) {
  if (!m || !X || !Y || n < 0) return imx::set_error(IMX_EINVAL, "imx_mlp_forward: bad argument");
  int rc = imx::mlp_reserve(m, n);
  if (rc) return rc;
  if (hipMemcpyAsync(m->Xf, X, n * MLP_IN * 4, hipMemcpyHostToDevice, m->stream) != hipSuccess)
    return imx::set_error(IMX_EDEVICE, "imx_mlp_forward: upload");
  f32_to_bf16<<<(unsigned)((n * MLP_IN + 255) / 256), 256, 0, m->stream>>>(n * MLP_IN, m->Xf, m->X);
  rc = imx::mlp_forward_dev(m, n, m->X, m->Y, m->stream);
  if (rc) return rc;
  if (hipMemcpyAsync(Y, m->Y, n * 2 * 4, hipMemcpyDeviceToHost, m->stream) != hipSuccess ||
      hipStreamSynchronize(m->stream) != hipSuccess)
    return imx::set_error(IMX_EDEVICE, "imx_mlp_forward: download");
  return IMX_OK;
}

// Gradient of L = sum_e w_e |y_e - t_e|^2 (no update when apply == 0);
// grad receives the P_N parameter gradients (may be NULL).
int imx_mlp_train(imx_mlp *m, int64_t n, const float *X, const float *T, const float *w, float lr,
                  float wd, int32_t apply, double *loss, float *grad, int32_t gmask) {
  if (!m || !X || !T || !w || n <= 0 || gmask < 0 || gmask > 3)
    return imx::set_error(IMX_EINVAL, "imx_mlp_train: bad argument");
  int rc = imx::mlp_reserve(m, n);
  if (rc) return rc;
  hipStream_t st = m->stream;
  if (hipMemcpyAsync(m->Xf, X, n * MLP_IN * 4, hipMemcpyHostToDevice, st) != hipSuccess ||
      hipMemcpyAsync(m->T, T, n * 2 * 4, hipMemcpyHostToDevice, st) != hipSuccess ||
      hipMemcpyAsync(m->w, w, n * 4, hipMemcpyHostToDevice, st) != hipSuccess)
    return imx::set_error(IMX_EDEVICE, "imx_mlp_train: upload");
  f32_to_bf16<<<(unsigned)((n * MLP_IN + 255) / 256), 256, 0, st>>>(n * MLP_IN, m->Xf, m->X);
  rc = imx::mlp_train_dev(m, n, nullptr, lr, wd, apply, nullptr, gmask);
  if (!rc && loss) rc = imx::mlp_loss(m, n, nullptr, 1, loss);
  if (rc) return rc;
  if (grad && (hipMemcpyAsync(grad, m->G, P_N * 4, hipMemcpyDeviceToHost, st) != hipSuccess ||
               hipStreamSynchronize(st) != hipSuccess))
    return imx::set_error(IMX_EDEVICE, "imx_mlp_train: download");
  if (hipStreamSynchronize(st) != hipSuccess) return imx::set_error(IMX_EDEVICE, "imx_mlp_train");
  return IMX_OK;
}

// Inference timing on n synthetic rows already resident (for throughput).
int imx_mlp_forward_timed(imx_mlp *m, int64_t n, int32_t reps, double *ms) {
  if (!m || !ms || n <= 0 || reps < 1) return imx::set_error(IMX_EINVAL, "imx_mlp_forward_timed: bad argument");
  int rc = imx::mlp_reserve(m, n);
  if (rc) return rc;
  hipEvent_t e0, e1;
  (void)hipEventCreate(&e0);
  (void)hipEventCreate(&e1);
  (void)hipMemsetAsync(m->X, 0, n * MLP_IN * 2, m->stream);
  rc = imx::mlp_forward_dev(m, n, m->X, m->Y, m->stream);
  (void)hipEventRecord(e0, m->stream);
  for (int r = 0; r < reps && !rc; ++r) rc = imx::mlp_forward_dev(m, n, m->X, m->Y, m->stream);
  (void)hipEventRecord(e1, m->stream);
  (void)hipEventSynchronize(e1);
  float f = 0.f;
  (void)hipEventElapsedTime(&f, e0, e1);
  *ms = f / reps;
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return rc;
}

void imx_mlp_destroy(imx_mlp *m) {
  if (!m) return;
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  float *fs[] = {m->P, m->M, m->V, m->G, m->part, m->lossp, m->T, m->w, m->Y, m->Xf};
  for (float *p : fs) (void)hipFree(p);
  short *ss[] = {m->Ff, m->Fb, m->Ff32, m->F1g, m->X};
  for (short *p : ss) (void)hipFree(p);
  if (m->stream) (void)hipStreamDestroy(m->stream);
  delete m;
}

}  // extern "C"
