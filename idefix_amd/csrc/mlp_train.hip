// Training of the learned limiter: hand-written FP32 kernels behind the C ABI of
// include/idefix_amd.h (idfx_mlp_*).  No counterpart in the reference.  A step is two
// kernels: k_train (forward, loss, backward and the weight gradients of a block's rows,
// FP32 matrix cores) and k_reduce (sums the blocks' gradients and applies Adam).
//
// Parameters are packed as in oracle/mlp.py: W1 [48][64], b1 [64], W2 [64][64], b2 [64],
// W3 [64][16], b3 [16] (row-major [in][out]), 8336 floats.  A batch row of X holds
// MLP_ROW = 72 floats: the 48 features, the interface's 16 PPM weights wp and 8 per-variable
// loss weights om; TAU [B][8] holds the normalised targets (t - c) / s.  The network's 16
// outputs z3 shift both PPM states of a variable, wL = wpL + z3[2v], wR = wpR - z3[2v].  Loss = mean over rows of
// sum_v om_v^2 (eL_v^2 + eR_v^2) with eL = x2 + wL (x3 - x2) - tau,
// eR = x3 - wR (x3 - x2) - tau.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "../../include/idefix_amd.h"

namespace {

constexpr int NF = 48, NH = 64, NO = 16;
constexpr int P_W1 = 0, P_B1 = P_W1 + NF * NH, P_W2 = P_B1 + NH, P_B2 = P_W2 + NH * NH,
              P_W3 = P_B2 + NH, P_B3 = P_W3 + NH * NO, P_N = P_B3 + NO;
constexpr float GELU_K = 1.702f;
constexpr int ROW = 72, ROW_WP = 48, ROW_OM = 64;  // batch row: features | wp | om
constexpr int TR = 32;            // rows of a tile: two waves of 16
constexpr int MAX_BLOCKS = 512;   // blocks of k_train: two per CU

__device__ __forceinline__ float sig(float z) { return 1.0f / (1.0f + expf(-z)); }
// derivative of z s with s = sig(GELU_K z)
__device__ __forceinline__ float gelu_d(float z, float s) {
  return s + GELU_K * z * s * (1.0f - s);
}

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));  // batch rows: any float address

// D += A B on 16x16x4 FP32 matrix instructions: lane 16 g + q gives A[q][g] and B[g][q]
// and holds D[4 g + r][q], r = 0 .. 3.
__device__ __forceinline__ f4 mfma(float a, float b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// LDS, in floats.  Weights [in][out], rows padded to strides (68, 20) that keep the reads of
// both passes free of bank conflicts: forward a lane reads one output of four inputs 4 g + r,
// backward four consecutive outputs of one input.  The tile's activations and deltas
// [row][unit] take their place for the weight gradients (strides of 16 mod 32 floats).
constexpr int S_W = 68, S_W3 = 20, L_W1 = 0, L_W2 = L_W1 + NF * S_W, L_W3 = L_W2 + NH * S_W,
              L_B = L_W3 + NH * S_W3, L_WEND = L_B + 2 * NH + NO;
constexpr int S_X = 48, S_H = 80, S_O = 16, L_X = 0, L_H1 = L_X + TR * S_X,
              L_H2 = L_H1 + TR * S_H, L_D1 = L_H2 + TR * S_H, L_D2 = L_D1 + TR * S_H,
              L_D3 = L_D2 + TR * S_H;
constexpr int L_GEND = L_D3 + TR * S_O, L_END = L_GEND > L_WEND ? L_GEND : L_WEND;

// Forward: acc[t] += W^T in over the inputs in[NI] (inputs 16 i + 4 g + r of the lane's row
// in in[i][r]); w points at the lane's input 4 g and output q of tile 0.
template <int NT, int NI>
__device__ __forceinline__ void forward(const float *w, int stride, const f4 *in, f4 *acc) {
#pragma unroll
  for (int i = 0; i < NI; i++)
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int t = 0; t < NT; t++)
        acc[t] = mfma(w[(16 * i + r) * stride + 16 * t], in[i][r], acc[t]);
}
// Backward: acc[t] += W in over the outputs; w points at the lane's input q and output 4 g.
template <int NT, int NI>
__device__ __forceinline__ void backward(const float *w, int stride, const f4 *in, f4 *acc) {
#pragma unroll
  for (int i = 0; i < NI; i++) {
    f4 a[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) a[t] = *reinterpret_cast<const f4 *>(w + 16 * t * stride + 16 * i);
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int t = 0; t < NT; t++) acc[t] = mfma(a[t][r], in[i][r], acc[t]);
  }
}

// Forward pass, loss, backward pass and weight gradients of tiles of 32 rows.  A wave takes
// 16 rows through all layers with the weights as the A operand and the activations as the
// B operand: a layer's accumulator (unit 4 g + r of row q in lane 16 g + q) is the next
// layer's B operand as it stands, so activations stay in registers.  For the gradients
// (sums over rows) the activations and deltas pass through LDS, each wave computing half
// of every layer's output tiles over all 32 rows; they accumulate in registers over the
// block's tiles and go out once per block.  Everything is FP32 (products, accumulators,
// activations).  208 + 128 matrix instructions per 16 rows: 2.2 us of the matrix cores'
// time at 8192 rows; the kernel is bound by its serial chain of layers.  A step of 8192
// rows takes 31 us, 18 of them here (33 with the weights loaded and transposed one float at a
// time); the eleven kernels this replaces (one thread per activation, scalar products) took
// 716, 555 of them in the weight gradients.
__global__ __launch_bounds__(128) void k_train(const float *X, const float *TAU, int B,
                                               const float *P, float *partial,
                                               double *lossp) {
  __shared__ __attribute__((aligned(16))) float lds[L_END];
  __shared__ double lred[2];
  const int tid = threadIdx.x, wave = tid >> 6, q = tid & 15, g = (tid >> 4) & 3;
  f4 g1[3][2], g2[4][2], g3[2];
#pragma unroll
  for (int n = 0; n < 2; n++) {
#pragma unroll
    for (int m = 0; m < 3; m++) g1[m][n] = f4{0, 0, 0, 0};
#pragma unroll
    for (int m = 0; m < 4; m++) g2[m][n] = f4{0, 0, 0, 0};
    g3[n] = f4{0, 0, 0, 0};
  }
  float gb = 0.0f, gb3 = 0.0f;  // bias gradients: unit tid of layers 1 | 2, unit tid of 3
  double loss = 0.0;
  const float inv = 1.0f / (float)B;
  for (int tile = blockIdx.x; tile * TR < B; tile += gridDim.x) {
    __syncthreads();  // the previous tile's gradient buffers have been read
    {
      // 16 consecutive floats of a thread's loads in flight at a time; every block of P
      // starts at a multiple of four floats
      const f4 *p1 = reinterpret_cast<const f4 *>(P + P_W1), *p2 = reinterpret_cast<const f4 *>(P + P_W2);
      const f4 *p3 = reinterpret_cast<const f4 *>(P + P_W3);
      f4 v1[NF * NH / 512], v2[NH * NH / 512], v3[NH * NO / 512];
#pragma unroll
      for (int n = 0; n < NF * NH / 512; n++) v1[n] = p1[tid + 128 * n];
#pragma unroll
      for (int n = 0; n < NH * NH / 512; n++) v2[n] = p2[tid + 128 * n];
#pragma unroll
      for (int n = 0; n < NH * NO / 512; n++) v3[n] = p3[tid + 128 * n];
      const float bias = P[tid < NH ? P_B1 + tid : P_B2 + tid - NH];
      const float bias3 = tid < NO ? P[P_B3 + tid] : 0.0f;
#pragma unroll
      for (int n = 0; n < NF * NH / 512; n++) {
        const int e = tid + 128 * n;  // 16 groups of four per row
        *reinterpret_cast<f4 *>(lds + L_W1 + e / 16 * S_W + e % 16 * 4) = v1[n];
      }
#pragma unroll
      for (int n = 0; n < NH * NH / 512; n++) {
        const int e = tid + 128 * n;
        *reinterpret_cast<f4 *>(lds + L_W2 + e / 16 * S_W + e % 16 * 4) = v2[n];
      }
#pragma unroll
      for (int n = 0; n < NH * NO / 512; n++) {
        const int e = tid + 128 * n;  // four groups per row
        *reinterpret_cast<f4 *>(lds + L_W3 + e / 4 * S_W3 + e % 4 * 4) = v3[n];
      }
      lds[L_B + tid] = bias;
      if (tid < NO) lds[L_B + 2 * NH + tid] = bias3;
    }
    __syncthreads();

    const int row = tile * TR + 16 * wave + q;
    const bool ok = row < B;
    const float *xr = X + (long long)(ok ? row : B - 1) * ROW;
    f4 x[3], z1[4], z2[4], z3;
#pragma unroll
    for (int i = 0; i < 3; i++) x[i] = *reinterpret_cast<const f4u *>(xr + 16 * i + 4 * g);
    // the lane's output variables 2 g and 2 g + 1
    float x2[2], x3[2], d[2], om2[2], tau[2], wpl[2], wpr[2];
#pragma unroll
    for (int n = 0; n < 2; n++) {
      const int v = 2 * g + n;
      x2[n] = xr[6 * v + 2];
      x3[n] = xr[6 * v + 3];
      d[n] = x3[n] - x2[n];
      const float om = xr[ROW_OM + v];
      om2[n] = ok ? om * om : 0.0f;
      wpl[n] = xr[ROW_WP + 2 * v];
      wpr[n] = xr[ROW_WP + 2 * v + 1];
      tau[n] = TAU[(long long)(ok ? row : B - 1) * 8 + v];
    }
    f4 s1[4], s2[4], h[4], h1[4];
#pragma unroll
    for (int t = 0; t < 4; t++) z1[t] = *reinterpret_cast<const f4 *>(lds + L_B + 16 * t + 4 * g);
    forward<4, 3>(lds + L_W1 + 4 * g * S_W + q, S_W, x, z1);
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        s1[t][r] = sig(GELU_K * z1[t][r]);
        h1[t][r] = z1[t][r] * s1[t][r];
      }
#pragma unroll
    for (int t = 0; t < 4; t++) z2[t] = *reinterpret_cast<const f4 *>(lds + L_B + NH + 16 * t + 4 * g);
    forward<4, 4>(lds + L_W2 + 4 * g * S_W + q, S_W, h1, z2);
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        s2[t][r] = sig(GELU_K * z2[t][r]);
        h[t][r] = z2[t][r] * s2[t][r];
      }
    z3 = *reinterpret_cast<const f4 *>(lds + L_B + 2 * NH + 4 * g);
    forward<1, 4>(lds + L_W3 + 4 * g * S_W3 + q, S_W3, h, &z3);
    // loss and dloss/dz3 (1/B included): wL = wpL + z3[2v], wR = wpR - z3[2v]
    f4 d3 = f4{0, 0, 0, 0};
#pragma unroll
    for (int n = 0; n < 2; n++) {
      const float z = z3[2 * n];
      const float el = x2[n] + (wpl[n] + z) * d[n] - tau[n];
      const float er = x3[n] - (wpr[n] - z) * d[n] - tau[n];
      loss += (double)(om2[n] * (el * el + er * er));
      d3[2 * n] = om2[n] * 2.0f * (el + er) * d[n] * inv;
    }
    f4 d2[4], d1[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
      const float *w3 = lds + L_W3 + (16 * t + q) * S_W3 + 4 * g;
      d2[t] = mfma(w3[0], d3[0], f4{0, 0, 0, 0});
      d2[t] = mfma(w3[2], d3[2], d2[t]);
      d1[t] = f4{0, 0, 0, 0};
    }
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) d2[t][r] *= gelu_d(z2[t][r], s2[t][r]);
    backward<4, 4>(lds + L_W2 + q * S_W + 4 * g, S_W, d2, d1);
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) d1[t][r] *= gelu_d(z1[t][r], s1[t][r]);
    __syncthreads();  // both waves are done with the weights
    {
      const int rr = 16 * wave + q;
#pragma unroll
      for (int i = 0; i < 3; i++)
        *reinterpret_cast<f4 *>(lds + L_X + rr * S_X + 16 * i + 4 * g) = x[i];
#pragma unroll
      for (int t = 0; t < 4; t++) {
        const int o = rr * S_H + 16 * t + 4 * g;
        *reinterpret_cast<f4 *>(lds + L_H1 + o) = h1[t];
        *reinterpret_cast<f4 *>(lds + L_H2 + o) = h[t];
        *reinterpret_cast<f4 *>(lds + L_D1 + o) = d1[t];
        *reinterpret_cast<f4 *>(lds + L_D2 + o) = d2[t];
      }
      *reinterpret_cast<f4 *>(lds + L_D3 + rr * S_O + 4 * g) = d3;
    }
    __syncthreads();
    // gradients: this wave's output units are the tiles 2 wave, 2 wave + 1 of layers 1 and
    // 2; of layer 3 its input units are.  Rows past the batch have zero deltas.
#pragma unroll
    for (int k = 0; k < TR; k += 4) {
      const float *b1 = lds + L_D1 + (k + g) * S_H + 32 * wave + q, *b2 = b1 + (L_D2 - L_D1);
      const float *ax = lds + L_X + (k + g) * S_X + q, *ah = lds + L_H1 + (k + g) * S_H + q;
      const float *a2 = lds + L_H2 + (k + g) * S_H + 32 * wave + q;
      const float dz3 = lds[L_D3 + (k + g) * S_O + q];
#pragma unroll
      for (int n = 0; n < 2; n++) {
#pragma unroll
        for (int m = 0; m < 3; m++) g1[m][n] = mfma(ax[16 * m], b1[16 * n], g1[m][n]);
#pragma unroll
        for (int m = 0; m < 4; m++) g2[m][n] = mfma(ah[16 * m], b2[16 * n], g2[m][n]);
        g3[n] = mfma(a2[16 * n], dz3, g3[n]);
      }
    }
#pragma unroll
    for (int r = 0; r < TR; r++) {
      gb += lds[(wave ? L_D2 : L_D1) + r * S_H + (tid & 63)];
      if (tid < NO) gb3 += lds[L_D3 + r * S_O + tid];
    }
  }
  float *out = partial + (long long)blockIdx.x * P_N;
#pragma unroll
  for (int n = 0; n < 2; n++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int col = 32 * wave + 16 * n + q, m0 = 4 * g + r;
#pragma unroll
      for (int m = 0; m < 3; m++) out[P_W1 + (16 * m + m0) * NH + col] = g1[m][n][r];
#pragma unroll
      for (int m = 0; m < 4; m++) out[P_W2 + (16 * m + m0) * NH + col] = g2[m][n][r];
      out[P_W3 + (32 * wave + 16 * n + m0) * NO + q] = g3[n][r];
    }
  out[(wave ? P_B2 : P_B1) + (tid & 63)] = gb;
  if (tid < NO) out[P_B3 + tid] = gb3;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) loss += __shfl_xor(loss, o);
  if ((tid & 63) == 0) lred[wave] = loss;
  __syncthreads();
  if (tid == 0) lossp[blockIdx.x] = lred[0] + lred[1];
}

// G = sum of the blocks' gradients, 32 parameters per block of 256 threads (8 slices of the
// blocks, then the slices, in a fixed order), and with ADAM the step (Kingma & Ba 2015,
// bias correction c1, c2).  Block 0 also sums the loss.  Eight loads in flight per thread: 6
// instead of 11 us for 256 blocks.
struct AdamArgs {
  float lr, b1, b2, eps, c1, c2;
};
template <bool ADAM>
__global__ __launch_bounds__(256) void k_reduce(const float *partial, const double *lossp,
                                                int nblk, int B, float *G, double *loss,
                                                float *P, float *M, float *V, AdamArgs a) {
  __shared__ float red[8][32];
  __shared__ double lred[256];
  const int c = threadIdx.x & 31, sl = threadIdx.x >> 5;
  const int e = blockIdx.x * 32 + c;
  float s = 0.0f;
  if (e < P_N) {
    int b = sl;
    for (; b + 56 < nblk; b += 64) {  // eight loads in flight
      float v[8];
#pragma unroll
      for (int k = 0; k < 8; k++) v[k] = partial[(long long)(b + 8 * k) * P_N + e];
#pragma unroll
      for (int k = 0; k < 8; k++) s += v[k];
    }
    for (; b < nblk; b += 8) s += partial[(long long)b * P_N + e];
  }
  red[sl][c] = s;
  __syncthreads();
  if (sl == 0 && e < P_N) {
    float gr = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; k++) gr += red[k][c];
    G[e] = gr;
    if constexpr (ADAM) {
      const float m = a.b1 * M[e] + (1.0f - a.b1) * gr;
      const float v = a.b2 * V[e] + (1.0f - a.b2) * gr * gr;
      M[e] = m;
      V[e] = v;
      P[e] -= a.lr * (m / a.c1) / (sqrtf(v / a.c2) + a.eps);
    }
  }
  if (blockIdx.x == 0) {
    double l = 0.0;
    for (int b = threadIdx.x; b < nblk; b += 256) l += lossp[b];
    lred[threadIdx.x] = l;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
      if ((int)threadIdx.x < w) lred[threadIdx.x] += lred[threadIdx.x + w];
      __syncthreads();
    }
    if (threadIdx.x == 0) *loss = lred[0] / B;
  }
}

int train_blocks(int B) { return std::min(MAX_BLOCKS, (B + TR - 1) / TR); }

}  // namespace

struct idfx_mlp {
  int cap = 0;
  long step = 0;
  std::vector<void *> allocs;
  float *P = nullptr, *G = nullptr, *M = nullptr, *V = nullptr;
  float *partial = nullptr;                  // gradients per block of k_train
  double *loss = nullptr, *lossp = nullptr;  // mean loss; loss sums per block
};

namespace {

int mlp_alloc(idfx_mlp *h, float **p, long long n) {
  void *q = nullptr;
  if (hipMalloc(&q, sizeof(float) * (size_t)std::max(n, 1LL)) != hipSuccess) return IDFX_E_ALLOC;
  h->allocs.push_back(q);
  if (hipMemset(q, 0, sizeof(float) * (size_t)std::max(n, 1LL)) != hipSuccess) return IDFX_E_ALLOC;
  *p = static_cast<float *>(q);
  return IDFX_OK;
}

// forward + loss + backward + gradient into h->G, with adam its step (asynchronous on s)
int grad_enqueue(idfx_mlp *h, const float *X, const float *TAU, int B, const AdamArgs *adam,
                 hipStream_t s) {
  const int nblk = train_blocks(B);
  const dim3 rgrid((P_N + 31) / 32);
  hipLaunchKernelGGL(k_train, dim3(nblk), dim3(128), 0, s, X, TAU, B, h->P, h->partial, h->lossp);
  if (adam)
    hipLaunchKernelGGL(k_reduce<true>, rgrid, dim3(256), 0, s, h->partial, h->lossp, nblk, B, h->G,
                       h->loss, h->P, h->M, h->V, *adam);
  else
    hipLaunchKernelGGL(k_reduce<false>, rgrid, dim3(256), 0, s, h->partial, h->lossp, nblk, B,
                       h->G, h->loss, h->P, h->M, h->V, AdamArgs{});
  return hipGetLastError() == hipSuccess ? IDFX_OK : IDFX_E_LAUNCH;
}

}  // namespace

extern "C" {

int idfx_mlp_param_count(void) { return P_N; }

int idfx_mlp_create(int max_batch, idfx_mlp **out) {
  if (!out || max_batch < 1) return IDFX_E_ARGS;
  *out = nullptr;
  idfx_mlp *h = new idfx_mlp();
  h->cap = max_batch;
  const int nblk = train_blocks(max_batch);
  int st = IDFX_OK;
  float **bufs[] = {&h->P, &h->G, &h->M, &h->V};
  for (float **b : bufs)
    if (st == IDFX_OK) st = mlp_alloc(h, b, P_N);
  if (st == IDFX_OK) st = mlp_alloc(h, &h->partial, (long long)nblk * P_N);
  if (st == IDFX_OK) {
    float *l = nullptr;
    st = mlp_alloc(h, &l, 2 * (1 + nblk));
    h->loss = reinterpret_cast<double *>(l);
    h->lossp = h->loss ? h->loss + 1 : nullptr;
  }
  if (st != IDFX_OK) {
    idfx_mlp_destroy(h);
    return st;
  }
  *out = h;
  return IDFX_OK;
}

int idfx_mlp_destroy(idfx_mlp *h) {
  if (!h) return IDFX_OK;
  hipDeviceSynchronize();
  for (void *p : h->allocs) hipFree(p);
  delete h;
  return IDFX_OK;
}

int idfx_mlp_set_params(idfx_mlp *h, const float *host) {
  if (!h || !host) return IDFX_E_ARGS;
  if (hipMemcpy(h->P, host, sizeof(float) * P_N, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemset(h->M, 0, sizeof(float) * P_N) != hipSuccess ||
      hipMemset(h->V, 0, sizeof(float) * P_N) != hipSuccess)
    return IDFX_E_LAUNCH;
  h->step = 0;
  return IDFX_OK;
}

int idfx_mlp_get_params(idfx_mlp *h, float *host) {
  if (!h || !host) return IDFX_E_ARGS;
  return hipMemcpy(host, h->P, sizeof(float) * P_N, hipMemcpyDeviceToHost) == hipSuccess
             ? IDFX_OK : IDFX_E_LAUNCH;
}

int idfx_mlp_loss_grad(idfx_mlp *h, const float *X, const float *TAU, int B, double *loss,
                       float *grad, void *stream) {
  if (!h || !X || !TAU || B < 1 || B > h->cap) return IDFX_E_ARGS;
  hipStream_t s = (hipStream_t)stream;
  int st = grad_enqueue(h, X, TAU, B, nullptr, s);
  if (st != IDFX_OK) return st;
  if (hipStreamSynchronize(s) != hipSuccess) return IDFX_E_LAUNCH;
  if (loss && hipMemcpy(loss, h->loss, sizeof(double), hipMemcpyDeviceToHost) != hipSuccess)
    return IDFX_E_LAUNCH;
  if (grad && hipMemcpy(grad, h->G, sizeof(float) * P_N, hipMemcpyDeviceToHost) != hipSuccess)
    return IDFX_E_LAUNCH;
  return IDFX_OK;
}

int idfx_mlp_train_step(idfx_mlp *h, const float *X, const float *TAU, int B, float lr,
                        void *stream) {
  if (!h || !X || !TAU || B < 1 || B > h->cap || !(lr > 0.0f)) return IDFX_E_ARGS;
  hipStream_t s = (hipStream_t)stream;
  const double t = (double)(h->step + 1);
  const AdamArgs adam{lr, 0.9f, 0.999f, 1e-8f, 1.0f - (float)std::pow(0.9, t),
                      1.0f - (float)std::pow(0.999, t)};
  const int st = grad_enqueue(h, X, TAU, B, &adam, s);
  if (st == IDFX_OK) h->step++;
  return st;
}

int idfx_mlp_loss(idfx_mlp *h, double *loss, void *stream) {
  if (!h || !loss) return IDFX_E_ARGS;
  hipStream_t s = (hipStream_t)stream;
  if (hipMemcpyAsync(loss, h->loss, sizeof(double), hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess)
    return IDFX_E_LAUNCH;
  return IDFX_OK;
}

}  // extern "C"
