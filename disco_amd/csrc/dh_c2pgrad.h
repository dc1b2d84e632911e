// dh_c2pgrad.h -- the learned guess's loss gradient on the matrix cores: one
// batch of rows as two launches.
//
//   k_mlp_batch   workgroups of 4 wavefronts take tiles of 32 rows: forward
//                 and backward pass in LDS, the 64 x 64 products (hidden
//                 layer, its transpose, the weight gradient H1^T D2) and the
//                 first layer's gradient X^T D1 as 16x16x4 float32 MFMA
//                 products; each workgroup keeps its gradient sums in
//                 registers over its tiles and writes one partial block
//   k_mlp_sum     one thread per parameter adds the partial blocks in order
//                 (and, in training, takes the Adam step); a wavefront adds
//                 the partial losses
//
// What bounds it: a batch of 4096 rows is 0.12 GFLOP and 0.2 MB, both under
// a microsecond at the card's rates, so the time is two launches and the
// chain of layers within one tile.  One thread per row and one per
// parameter, each parameter's sum running over all rows, took 1.49 ms for
// 4096 rows (76 wavefronts with a serial chain of 4096 loads each); the 128
// workgroups here take 22 us, launches included, and a fit of 40,000 rows in
// batches of 2048 goes from 33.3 to 1.8 ms.  32 rows a tile: 64 would halve the
// workgroups (4096 rows then fill a quarter of the CUs), 16 would double the
// partial blocks that k_mlp_sum reads.
//
// The sums are deterministic: the split depends on the row count alone.
// Products and sums are float32 as in the row-by-row form, in another order
// (a tile's 32 rows, then tiles, then workgroups; the row-by-row form adds
// all rows to one sum), the losses double.
#pragma once
#include <hip/hip_runtime.h>

#include "dh_c2ptrain.h"

namespace dh {

typedef float mlp_v4 __attribute__((ext_vector_type(4)));

constexpr int MLP_ROWS = 32;        // rows of a tile
constexpr int MLP_MAX_WG = 128;     // workgroups of a batch (they loop over the tiles)
constexpr int MLP_TPB = 256;
constexpr int MLP_P = C2PNET_H + 1;  // LDS pitch: odd, so that columns too are free of conflicts
constexpr int MLP_XP = 17;           // pitch of the features (8, a constant 1 for the bias, zeros to 16)

// Floats of workspace for a batch: every workgroup's partial gradient and
// (as a double, first) its loss.
constexpr size_t MLP_WS_FLOATS = (size_t)MLP_MAX_WG * (C2PNET_NTRAIN + 2);

inline unsigned mlp_workgroups(long n)
{
   long tiles = (n + MLP_ROWS - 1) / MLP_ROWS;
   return (unsigned)(tiles < MLP_MAX_WG ? tiles : MLP_MAX_WG);
}

__device__ inline mlp_v4 mlp_mfma(float a, float b, mlp_v4 c)
{
   return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Partial gradients part[wg][NTRAIN] and losses lossp[wg] of the batch's
// rows; blockIdx.x takes tiles blockIdx.x, + gridDim.x, ...
// 16x16x4 operands: lane l holds A[l % 16][l / 16], B[l / 16][l % 16] and
// the result's rows 4 (l / 16) + i, column l % 16.
__global__ __launch_bounds__(MLP_TPB) void k_mlp_batch(const float *__restrict__ prm,
                                                       const float *__restrict__ Xg,
                                                       const float *__restrict__ Yg,
                                                       const int *__restrict__ idx, long n,
                                                       double *__restrict__ lossp,
                                                       float *__restrict__ part)
{
   __shared__ float W1[C2PNET_IN * C2PNET_H], W2[C2PNET_H * MLP_P], W3[C2PNET_H * C2PNET_OUT];
   __shared__ float X[MLP_ROWS * MLP_XP], H1[MLP_ROWS * MLP_P], H2[MLP_ROWS * MLP_P];
   __shared__ float D1[MLP_ROWS * MLP_P], D2[MLP_ROWS * MLP_P], D3[MLP_ROWS * C2PNET_OUT];
   __shared__ float ls[MLP_ROWS * C2PNET_OUT];
   const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
   const int col = lane & 15, quad = lane >> 4;
   for (int i = tid; i < C2PNET_IN * C2PNET_H; i += MLP_TPB) W1[i] = prm[C2PNET_W1 + i];
   for (int i = tid; i < C2PNET_H * C2PNET_H; i += MLP_TPB)
      W2[(i / C2PNET_H) * MLP_P + i % C2PNET_H] = prm[C2PNET_W2 + i];
   for (int i = tid; i < C2PNET_H * C2PNET_OUT; i += MLP_TPB) W3[i] = prm[C2PNET_W3 + i];

   mlp_v4 gW2[4], gW1 = {0.f, 0.f, 0.f, 0.f};
   for (int i = 0; i < 4; ++i) gW2[i] = mlp_v4{0.f, 0.f, 0.f, 0.f};
   float gV = 0.f;        // W3 (threads 0..127), b2 (128..191), b3 (192, 193)
   double loss = 0.0;     // thread 0
   const float nout = (float)(C2PNET_OUT * n);

   const long ntiles = (n + MLP_ROWS - 1) / MLP_ROWS;
   for (long t = blockIdx.x; t < ntiles; t += gridDim.x) {
      const long row0 = t * MLP_ROWS;
      const int rows = (int)(n - row0 < MLP_ROWS ? n - row0 : MLP_ROWS);
      __syncthreads();  // the last tile's arrays are read; the weights are in place
      {
         int r = tid >> 3, k = tid & 7;
         float v = 0.f;
         if (r < rows) {
            long i = idx ? idx[row0 + r] : row0 + r;
            v = (Xg[(size_t)i * C2PNET_IN + k] - prm[C2PNET_IN_MU + k]) / prm[C2PNET_IN_SD + k];
         }
         X[r * MLP_XP + k] = v;
         // column 8 turns the bias's gradient into a row of X^T D1
         X[r * MLP_XP + 8 + k] = k == 0 && r < rows ? 1.f : 0.f;
      }
      __syncthreads();
      // layer 1: 8 outputs a thread (output j of 8 rows)
      {
         int j = tid & 63;
         float w[C2PNET_IN], b = prm[C2PNET_B1 + j];
         for (int k = 0; k < C2PNET_IN; ++k) w[k] = W1[k * C2PNET_H + j];
         for (int r = wv; r < MLP_ROWS; r += 4) {
            float s = b;
            for (int k = 0; k < C2PNET_IN; ++k) s += X[r * MLP_XP + k] * w[k];
            H1[r * MLP_P + j] = s > 0.f ? s : 0.f;
         }
      }
      __syncthreads();
      // layer 2: wavefront wv takes columns 16 wv .. + 15 of both row blocks
      {
         float b = prm[C2PNET_B2 + 16 * wv + col];
         mlp_v4 c0 = {b, b, b, b}, c1 = c0;
         for (int ks = 0; ks < C2PNET_H / 4; ++ks) {
            float w = W2[(4 * ks + quad) * MLP_P + 16 * wv + col];
            c0 = mlp_mfma(H1[col * MLP_P + 4 * ks + quad], w, c0);
            c1 = mlp_mfma(H1[(16 + col) * MLP_P + 4 * ks + quad], w, c1);
         }
         for (int i = 0; i < 4; ++i) {
            H2[(4 * quad + i) * MLP_P + 16 * wv + col] = c0[i] > 0.f ? c0[i] : 0.f;
            H2[(16 + 4 * quad + i) * MLP_P + 16 * wv + col] = c1[i] > 0.f ? c1[i] : 0.f;
         }
      }
      __syncthreads();
      // layer 3, the error and its derivative: 4 threads an output
      {
         int r = tid >> 3, o = (tid >> 2) & 1, q = tid & 3;
         float y = 0.f;
         for (int k = q; k < C2PNET_H; k += 4) y += H2[r * MLP_P + k] * W3[k * C2PNET_OUT + o];
         y += __shfl_xor(y, 1, 64);
         y += __shfl_xor(y, 2, 64);
         if (q == 0) {
            float e = 0.f;
            if (r < rows) {
               long i = idx ? idx[row0 + r] : row0 + r;
               float tg = (Yg[(size_t)i * C2PNET_OUT + o] - prm[C2PNET_OUT_MU + o]) /
                          prm[C2PNET_OUT_SD + o];
               e = y + prm[C2PNET_B3 + o] - tg;
            }
            D3[r * C2PNET_OUT + o] = 2.0f * e / nout;
            ls[r * C2PNET_OUT + o] = e * e;
         }
      }
      __syncthreads();
      {
         int j = tid & 63;
         float w0 = W3[j * C2PNET_OUT], w1 = W3[j * C2PNET_OUT + 1];
         for (int r = wv; r < MLP_ROWS; r += 4) {
            float s = D3[r * C2PNET_OUT] * w0 + D3[r * C2PNET_OUT + 1] * w1;
            D2[r * MLP_P + j] = H2[r * MLP_P + j] > 0.f ? s : 0.f;
         }
      }
      __syncthreads();
      // D1 = D2 W2^T where H1 > 0
      {
         mlp_v4 c0 = {0.f, 0.f, 0.f, 0.f}, c1 = c0;
         for (int ks = 0; ks < C2PNET_H / 4; ++ks) {
            float w = W2[(16 * wv + col) * MLP_P + 4 * ks + quad];
            c0 = mlp_mfma(D2[col * MLP_P + 4 * ks + quad], w, c0);
            c1 = mlp_mfma(D2[(16 + col) * MLP_P + 4 * ks + quad], w, c1);
         }
         for (int i = 0; i < 4; ++i) {
            int r0 = (4 * quad + i) * MLP_P + 16 * wv + col, r1 = r0 + 16 * MLP_P;
            D1[r0] = H1[r0] > 0.f ? c0[i] : 0.f;
            D1[r1] = H1[r1] > 0.f ? c1[i] : 0.f;
         }
      }
      __syncthreads();
      // the gradients' sums over the tile's rows
      for (int ks = 0; ks < MLP_ROWS / 4; ++ks) {
         int r = 4 * ks + quad;
         float d2 = D2[r * MLP_P + 16 * wv + col];
         for (int kb = 0; kb < 4; ++kb) gW2[kb] = mlp_mfma(H1[r * MLP_P + 16 * kb + col], d2, gW2[kb]);
         gW1 = mlp_mfma(X[r * MLP_XP + col], D1[r * MLP_P + 16 * wv + col], gW1);
      }
      if (tid < C2PNET_H * C2PNET_OUT) {
         int k = tid / C2PNET_OUT, o = tid % C2PNET_OUT;
         for (int r = 0; r < MLP_ROWS; ++r) gV += H2[r * MLP_P + k] * D3[r * C2PNET_OUT + o];
      } else if (tid < C2PNET_H * C2PNET_OUT + C2PNET_H) {
         int j = tid - C2PNET_H * C2PNET_OUT;
         for (int r = 0; r < MLP_ROWS; ++r) gV += D2[r * MLP_P + j];
      } else if (tid < C2PNET_H * C2PNET_OUT + C2PNET_H + C2PNET_OUT) {
         int o = tid - C2PNET_H * C2PNET_OUT - C2PNET_H;
         for (int r = 0; r < MLP_ROWS; ++r) gV += D3[r * C2PNET_OUT + o];
      }
      if (wv == 3) {  // ls: 64 squared errors, added by halves
         double l = ls[lane];
         for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o, 64);
         loss += l;
      }
   }
   float *out = part + (size_t)blockIdx.x * C2PNET_NTRAIN - C2PNET_TRAIN0;
   for (int kb = 0; kb < 4; ++kb)
      for (int i = 0; i < 4; ++i)
         out[C2PNET_W2 + (16 * kb + 4 * quad + i) * C2PNET_H + 16 * wv + col] = gW2[kb][i];
   for (int i = 0; i < 4; ++i) {
      int k = 4 * quad + i;
      if (k < C2PNET_IN) out[C2PNET_W1 + k * C2PNET_H + 16 * wv + col] = gW1[i];
      else if (k == C2PNET_IN) out[C2PNET_B1 + 16 * wv + col] = gW1[i];
   }
   if (tid < C2PNET_H * C2PNET_OUT) out[C2PNET_W3 + tid] = gV;
   else if (tid < C2PNET_H * C2PNET_OUT + C2PNET_H) out[C2PNET_B2 + tid - C2PNET_H * C2PNET_OUT] = gV;
   else if (tid < C2PNET_H * C2PNET_OUT + C2PNET_H + C2PNET_OUT)
      out[C2PNET_B3 + tid - C2PNET_H * C2PNET_OUT - C2PNET_H] = gV;
   if (tid == 192) lossp[blockIdx.x] = loss;
}

// The Adam state and rates of a training step (KAdam's).
struct MlpAdam {
   float *prm, *m, *v;  // prm null: no step
   float lr, b1, b2, eps, c1, c2;
};

// The batch's gradient from the partial blocks of nwg workgroups: block
// i < MLP_SUM_BLOCKS takes parameters MLP_TPB i .. of the parameter block
// and writes grad[NPARAM] (zero outside the trainable range) where grad is
// given, and takes the Adam step where A.prm is; the last block's first
// wavefront adds the losses: *mean = sum / (2 n) (mean given), *total +=
// sum in float (total given).
constexpr unsigned MLP_SUM_BLOCKS = (C2PNET_NPARAM + MLP_TPB - 1) / MLP_TPB;
__global__ __launch_bounds__(MLP_TPB) void k_mlp_sum(const float *__restrict__ part,
                                                     const double *__restrict__ lossp, int nwg,
                                                     long n, float *grad, MlpAdam A, float *mean,
                                                     float *total)
{
   if (blockIdx.x == MLP_SUM_BLOCKS) {
      if (threadIdx.x >= 64) return;
      double l = 0.0;
      for (int w = threadIdx.x; w < nwg; w += 64) l += lossp[w];
      for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o, 64);
      if (threadIdx.x == 0) {
         if (mean) *mean = (float)(l / (2.0 * n));
         if (total) *total += (float)l;
      }
      return;
   }
   int q = blockIdx.x * MLP_TPB + threadIdx.x;
   if (q >= C2PNET_NPARAM) return;
   int t = q - C2PNET_TRAIN0;
   bool trained = t >= 0 && t < C2PNET_NTRAIN;
   float s = 0.f;
   if (trained) {
      // four sums in flight: the loads of consecutive blocks do not wait for each other
      float s4[4] = {0.f, 0.f, 0.f, 0.f};
      int w = 0;
      for (; w + 4 <= nwg; w += 4)
         for (int i = 0; i < 4; ++i) s4[i] += part[(size_t)(w + i) * C2PNET_NTRAIN + t];
      for (; w < nwg; ++w) s4[0] += part[(size_t)w * C2PNET_NTRAIN + t];
      s = (s4[0] + s4[1]) + (s4[2] + s4[3]);
   }
   if (grad) grad[q] = s;
   if (A.prm && trained) KAdam{A.prm, A.m, A.v, nullptr, A.lr, A.b1, A.b2, A.eps, A.c1, A.c2}.step(t, s);
}

}  // namespace dh
