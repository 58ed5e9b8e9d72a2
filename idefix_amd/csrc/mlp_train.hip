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
constexpr int TR = 32;            // rows of a tile: two groups of 16
constexpr int MAX_BLOCKS = 256;   // blocks of k_train: one per CU

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
// backward four consecutive outputs of one input.  Then the tile's features, activations and
// deltas [row][unit] (strides of 16 mod 32 floats).
constexpr int S_W = 68, S_W3 = 20, L_W1 = 0, L_W2 = L_W1 + NF * S_W, L_W3 = L_W2 + NH * S_W,
              L_B = L_W3 + NH * S_W3, L_WEND = L_B + 2 * NH + NO;
constexpr int S_X = 48, S_H = 80, S_O = 16, L_X = L_WEND, L_H1 = L_X + TR * S_X,
              L_H2 = L_H1 + TR * S_H, L_D1 = L_H2 + TR * S_H, L_D2 = L_D1 + TR * S_H,
              L_D3 = L_D2 + TR * S_H, L_END = L_D3 + TR * S_O;
static_assert(L_X % 4 == 0 && L_B % 4 == 0, "16-byte reads");

// Forward pass, loss, backward pass and weight gradients of tiles of 32 rows.  A group of
// four waves takes 16 rows through the layers, each wave one tile of 16 units of the hidden
// layers (all four compute the 16 outputs), with the weights as the A operand and the
// activations as the B operand: a lane holds units 4 g + r of row q, r = 0 .. 3.  Between
// layers the activations and deltas pass through LDS, where the gradients (sums over rows)
// need them too; each of the block's eight waves computes four of their 32 tiles of 16 x 16
// over all 32 rows.  They accumulate in registers over the block's tiles and go out once per
// block.  Everything is FP32 (products, accumulators, activations).
//
// 208 + 128 matrix instructions per 16 rows: 2.2 us of the matrix cores' time at 8192 rows;
// the kernel is bound by its serial chain of layers, which four waves a row group shorten:
// 14 us at 8192 rows (a step 27), against 18 (31) with one wave per 16 rows and the activations
// in registers; 131,072 rows: a step 109 against 117.
// The eleven kernels this replaces (one thread per activation, scalar products) took 716 us a
// step, 555 of them in the weight gradients.
__global__ __launch_bounds__(512) void k_train(const float *X, const float *TAU, int B,
                                               const float *P, float *partial,
                                               double *lossp) {
  __shared__ __attribute__((aligned(16))) float lds[L_END];
  __shared__ double lred[2];
  const int tid = threadIdx.x, wave = tid >> 6, q = tid & 15, g = (tid >> 4) & 3;
  const int grp = wave >> 2, u = wave & 3;  // row group, tile of 16 hidden units
  {
    // the weights: 16-byte loads, all in flight together; every block of P starts at a
    // multiple of four floats
    const f4 *p1 = reinterpret_cast<const f4 *>(P + P_W1), *p2 = reinterpret_cast<const f4 *>(P + P_W2);
    const f4 *p3 = reinterpret_cast<const f4 *>(P + P_W3);
    constexpr int Q1 = NF * NH / 4, Q2 = NH * NH / 4, Q3 = NH * NO / 4;  // 768, 1024, 256
    const f4 a0 = p1[tid], a1 = p1[min(tid + 512, Q1 - 1)], b0 = p2[tid], b1 = p2[tid + 512];
    const f4 c0 = p3[min(tid, Q3 - 1)];
    const float bias = tid < NH       ? P[P_B1 + tid]
                       : tid < 2 * NH ? P[P_B2 + tid - NH]
                       : tid < 2 * NH + NO ? P[P_B3 + tid - 2 * NH] : 0.0f;
    auto put = [&](int base, int e, f4 v) {  // 16 groups of four per row
      *reinterpret_cast<f4 *>(lds + base + e / 16 * S_W + e % 16 * 4) = v;
    };
    put(L_W1, tid, a0);
    if (tid + 512 < Q1) put(L_W1, tid + 512, a1);
    put(L_W2, tid, b0);
    put(L_W2, tid + 512, b1);
    static_assert(Q2 == 1024, "two 16-byte groups of W2 per thread");
    if (tid < Q3) *reinterpret_cast<f4 *>(lds + L_W3 + tid / 4 * S_W3 + tid % 4 * 4) = c0;
    if (tid < 2 * NH + NO) lds[L_B + tid] = bias;
  }
  // this wave's gradient tiles: waves 0-2 input block `wave` of layer 1, 3-6 input block
  // wave - 3 of layer 2, each with all four output blocks; wave 7 the four input blocks of
  // layer 3
  const int am = wave < 3 ? L_X + 16 * wave : wave < 7 ? L_H1 + 16 * (wave - 3) : L_H2;
  const int as = wave < 3 ? S_X : S_H, an = wave < 7 ? 0 : 16;
  const int bm = wave < 3 ? L_D1 : wave < 7 ? L_D2 : L_D3;
  const int bs = wave < 7 ? S_H : S_O, bnn = wave < 7 ? 16 : 0;
  f4 gr[4];
#pragma unroll
  for (int n = 0; n < 4; n++) gr[n] = f4{0, 0, 0, 0};
  // bias gradients: thread tid sums unit tid of layer 1, tid - 64 of 2, tid - 128 of 3
  const int gcol = tid < NH ? L_D1 + tid : tid < 2 * NH ? L_D2 + tid - NH : L_D3 + tid - 2 * NH;
  const int gstr = tid < 2 * NH ? S_H : S_O;
  float gb = 0.0f;
  double loss = 0.0;
  const float inv = 1.0f / (float)B;
  for (int tile = blockIdx.x; tile * TR < B; tile += gridDim.x) {
    const int lr = 16 * grp + q, row = tile * TR + lr;
    const bool ok = row < B;
    const float *xr = X + (long long)(ok ? row : B - 1) * ROW;
    f4 x[3];
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
    __syncthreads();  // weights stored; the previous tile's gradients have been summed
    if (u < 3) *reinterpret_cast<f4 *>(lds + L_X + lr * S_X + 16 * u + 4 * g) = x[u];
    // hidden layers: this wave's units 16 u + 4 g + r
    const int ho = lr * S_H + 16 * u + 4 * g, hrow = lr * S_H + 4 * g;
    f4 z1 = *reinterpret_cast<const f4 *>(lds + L_B + 16 * u + 4 * g), s1, s2;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        z1 = mfma(lds[L_W1 + (16 * i + 4 * g + r) * S_W + 16 * u + q], x[i][r], z1);
    f4 h;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      s1[r] = sig(GELU_K * z1[r]);
      h[r] = z1[r] * s1[r];
    }
    *reinterpret_cast<f4 *>(lds + L_H1 + ho) = h;
    __syncthreads();
    f4 z2 = *reinterpret_cast<const f4 *>(lds + L_B + NH + 16 * u + 4 * g);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const f4 in = *reinterpret_cast<const f4 *>(lds + L_H1 + hrow + 16 * i);
#pragma unroll
      for (int r = 0; r < 4; r++)
        z2 = mfma(lds[L_W2 + (16 * i + 4 * g + r) * S_W + 16 * u + q], in[r], z2);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
      s2[r] = sig(GELU_K * z2[r]);
      h[r] = z2[r] * s2[r];
    }
    *reinterpret_cast<f4 *>(lds + L_H2 + ho) = h;
    __syncthreads();
    f4 z3 = *reinterpret_cast<const f4 *>(lds + L_B + 2 * NH + 4 * g);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const f4 in = *reinterpret_cast<const f4 *>(lds + L_H2 + hrow + 16 * i);
#pragma unroll
      for (int r = 0; r < 4; r++) z3 = mfma(lds[L_W3 + (16 * i + 4 * g + r) * S_W3 + q], in[r], z3);
    }
    // loss and dloss/dz3 (1/B included): wL = wpL + z3[2v], wR = wpR - z3[2v]
    f4 d3 = f4{0, 0, 0, 0};
#pragma unroll
    for (int n = 0; n < 2; n++) {
      const float z = z3[2 * n];
      const float el = x2[n] + (wpl[n] + z) * d[n] - tau[n];
      const float er = x3[n] - (wpr[n] - z) * d[n] - tau[n];
      if (u == 0) loss += (double)(om2[n] * (el * el + er * er));
      d3[2 * n] = om2[n] * 2.0f * (el + er) * d[n] * inv;
    }
    if (u == 0) *reinterpret_cast<f4 *>(lds + L_D3 + lr * S_O + 4 * g) = d3;
    // deltas; outputs 2 v + 1 have none
    const float *w3 = lds + L_W3 + (16 * u + q) * S_W3 + 4 * g;
    f4 d2 = mfma(w3[0], d3[0], f4{0, 0, 0, 0});
    d2 = mfma(w3[2], d3[2], d2);
#pragma unroll
    for (int r = 0; r < 4; r++) d2[r] *= gelu_d(z2[r], s2[r]);
    *reinterpret_cast<f4 *>(lds + L_D2 + ho) = d2;
    __syncthreads();
    f4 d1 = f4{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const f4 in = *reinterpret_cast<const f4 *>(lds + L_D2 + hrow + 16 * i);
      const f4 w = *reinterpret_cast<const f4 *>(lds + L_W2 + (16 * u + q) * S_W + 16 * i + 4 * g);
#pragma unroll
      for (int r = 0; r < 4; r++) d1 = mfma(w[r], in[r], d1);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) d1[r] *= gelu_d(z1[r], s1[r]);
    *reinterpret_cast<f4 *>(lds + L_D1 + ho) = d1;
    __syncthreads();
    // gradients.  Rows past the batch have zero deltas.
#pragma unroll
    for (int k = 0; k < TR; k += 4) {
      const float *a = lds + am + (k + g) * as + q, *b = lds + bm + (k + g) * bs + q;
#pragma unroll
      for (int n = 0; n < 4; n++) gr[n] = mfma(a[n * an], b[n * bnn], gr[n]);
    }
    if (tid < 2 * NH + NO) {
#pragma unroll
      for (int r = 0; r < TR; r++) gb += lds[gcol + r * gstr];
    }
  }
  float *out = partial + (long long)blockIdx.x * P_N;
  const int om0 = wave < 3 ? P_W1 + 16 * wave * NH : wave < 7 ? P_W2 + 16 * (wave - 3) * NH : P_W3;
#pragma unroll
  for (int n = 0; n < 4; n++)
#pragma unroll
    for (int r = 0; r < 4; r++)
      out[wave < 7 ? om0 + (4 * g + r) * NH + 16 * n + q : om0 + (16 * n + 4 * g + r) * NO + q] = gr[n][r];
  if (tid < 2 * NH + NO) out[tid < NH ? P_B1 + tid : tid < 2 * NH ? P_B2 + tid - NH : P_B3 + tid - 2 * NH] = gb;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) loss += __shfl_xor(loss, o);
  if (u == 0 && (tid & 63) == 0) lred[grp] = loss;
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
  hipLaunchKernelGGL(k_train, dim3(nblk), dim3(512), 0, s, X, TAU, B, h->P, h->partial, h->lossp);
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
  // the clears have ended before the memory is handed out: a non-blocking stream does not wait
  // for them
  if (st == IDFX_OK && hipStreamSynchronize(nullptr) != hipSuccess) st = IDFX_E_ALLOC;
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
  // steps may be under way on a stream that does not wait for the null stream, nor it for them;
  // the moments are clear before the call returns
  if (hipDeviceSynchronize() != hipSuccess ||
      hipMemcpy(h->P, host, sizeof(float) * P_N, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemset(h->M, 0, sizeof(float) * P_N) != hipSuccess ||
      hipMemset(h->V, 0, sizeof(float) * P_N) != hipSuccess || hipStreamSynchronize(nullptr) != hipSuccess)
    return IDFX_E_LAUNCH;
  h->step = 0;
  return IDFX_OK;
}

int idfx_mlp_get_params(idfx_mlp *h, float *host) {
  if (!h || !host) return IDFX_E_ARGS;
  // the steps enqueued so far, on whichever stream
  if (hipDeviceSynchronize() != hipSuccess) return IDFX_E_LAUNCH;
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
