// h-predictor MLP for the h-rho iteration: 6 features -> 32 -> 32 (GELU) -> 1,
// BF16 weights with FP32 accumulation, trained online on the device by the
// kernels below (forward, backward, Adam).  Its output only seeds the
// Newton-Raphson iteration of k_nr_pass, which still converges every particle
// to tolh; the reference's seed is h = h_in + dt dh/dt
// (src/stepND_leapfrog_mhd.f90:153).
//
// Parameter vector (float[NPARAM]): W1[32][6] b1[32] W2[32][32] b2[32] W3[32] b3.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "ndsp_mlp.h"

#define NIN MLP_NIN
#define NH MLP_NH
#define WB 64          // samples per block of the FP32 passes (four waves, eight hidden units each)
#define WU (NH / 4)

__device__ __forceinline__ float bf16_to_f(uint16_t b) { return __uint_as_float(((uint32_t)b) << 16); }

__device__ __forceinline__ uint16_t f_to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  uint32_t r = u + 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even
  return (uint16_t)(r >> 16);
}

__device__ __forceinline__ float gelu(float x) {
  const float c = 0.7978845608028654f;
  return 0.5f * x * (1.0f + tanhf(c * (x + 0.044715f * x * x * x)));
}
__device__ __forceinline__ float dgelu(float x) {
  const float c = 0.7978845608028654f;
  const float u = c * (x + 0.044715f * x * x * x);
  const float t = tanhf(u);
  const float du = c * (1.0f + 3.0f * 0.044715f * x * x);
  return 0.5f * (1.0f + t) + 0.5f * x * (1.0f - t * t) * du;
}

__device__ __forceinline__ void load_weights(const uint16_t* __restrict__ wbf, float* sw) {
  for (int p = threadIdx.x; p < MLP_NPARAM; p += blockDim.x) sw[p] = bf16_to_f(wbf[p]);
  __syncthreads();
}

// The FP32 passes: a block of four waves takes WB samples; lane s of every wave
// works on sample s, wave g on the hidden units WU g .. WU g + WU - 1 (their
// weights are broadcast reads), and the activations pass between the waves
// through LDS.  Each unit's sum runs in the order a single thread would take.
// (One thread a sample left 16384 rows with 256 waves, one per CU: gradient 51 us
// and forward 17; 24 and 9 here.)
struct MlpTile {
  float sw[MLP_NPARAM];
  float a1[WB][NH + 1], a2[WB][NH + 1];
};

// forward of the block's samples: activations in t, the wave's own
// pre-activations in z1, z2, the output of sample threadIdx % 64 returned
__device__ __forceinline__ float mlp_fwd_tile(MlpTile& t, const float (&x)[NIN], float (&z1)[WU], float (&z2)[WU]) {
  const int s = threadIdx.x & 63, g = threadIdx.x >> 6;
  const float* W1 = t.sw;
  const float* b1 = W1 + NH * NIN;
  const float* W2 = b1 + NH;
  const float* b2 = W2 + NH * NH;
  const float* W3 = b2 + NH;
#pragma unroll
  for (int u = 0; u < WU; u++) {
    const int o = WU * g + u;
    float v = b1[o];
#pragma unroll
    for (int i = 0; i < NIN; i++) v += W1[o * NIN + i] * x[i];
    z1[u] = v;
    t.a1[s][o] = gelu(v);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < WU; u++) z2[u] = b2[WU * g + u];
#pragma unroll 8
  for (int i = 0; i < NH; i++) {
    const float a = t.a1[s][i];
#pragma unroll
    for (int u = 0; u < WU; u++) z2[u] += W2[(WU * g + u) * NH + i] * a;
  }
#pragma unroll
  for (int u = 0; u < WU; u++) t.a2[s][WU * g + u] = gelu(z2[u]);
  __syncthreads();
  float y = W3[NH];
#pragma unroll 8
  for (int i = 0; i < NH; i++) y += W3[i] * t.a2[s][i];
  return y;
}

// forward on a feature matrix X[B][ldx] (columns 0..5 are the features)
__global__ __launch_bounds__(256) void k_mlp_forward(const uint16_t* __restrict__ wbf, const float* __restrict__ X,
                                                     int ldx, int B, float* __restrict__ y) {
  __shared__ MlpTile t;
  load_weights(wbf, t.sw);
  const int b = blockIdx.x * WB + (threadIdx.x & 63);
  float x[NIN], z1[WU], z2[WU];
  for (int i = 0; i < NIN; i++) x[i] = b < B ? X[(size_t)b * ldx + i] : 0.0f;
  const float out = mlp_fwd_tile(t, x, z1, z2);
  if (threadIdx.x < 64 && b < B) y[b] = out;
}

// gradient of L = sum (y - t)^2 / B over the samples b < B; sample b is row
// (off + b * stride) mod nrows of X[.][ldx], its target at T[row * ldt]
__global__ __launch_bounds__(256) void k_mlp_grad(const uint16_t* __restrict__ wbf, const float* __restrict__ X, int ldx,
                                                  const float* __restrict__ T, int ldt, int nrows, int B, long long off,
                                                  long long stride, float* __restrict__ grad, float* __restrict__ loss) {
  __shared__ MlpTile t;
  __shared__ float sX[WB][NIN + 1];
  __shared__ float sD1[WB][NH + 1];
  __shared__ float sD2[WB][NH + 1];
  __shared__ float sDy[WB];
  load_weights(wbf, t.sw);
  const int s = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int b = blockIdx.x * WB + s;
  const bool act = b < B;
  const long long row = act ? (off + (long long)b * stride) % nrows : 0;
  float x[NIN], z1[WU], z2[WU];
  for (int i = 0; i < NIN; i++) x[i] = act ? X[row * ldx + i] : 0.0f;
  const float y = mlp_fwd_tile(t, x, z1, z2);
  const float r = act ? y - T[row * ldt] : 0.0f;
  const float dy = act ? 2.0f * r / (float)B : 0.0f;
  const float* W2 = t.sw + NH * NIN + NH;
  const float* W3 = W2 + NH * NH + NH;
#pragma unroll
  for (int u = 0; u < WU; u++) {
    const int o = WU * g + u;
    sD2[s][o] = act ? dy * W3[o] * dgelu(z2[u]) : 0.0f;
  }
  if (g == 0) {
    for (int i = 0; i < NIN; i++) sX[s][i] = x[i];
    sDy[s] = dy;
  }
  __syncthreads();
  float d1[WU];
#pragma unroll
  for (int u = 0; u < WU; u++) d1[u] = 0.0f;
#pragma unroll 8
  for (int o = 0; o < NH; o++) {
    const float d = sD2[s][o];
#pragma unroll
    for (int u = 0; u < WU; u++) d1[u] += W2[o * NH + WU * g + u] * d;
  }
#pragma unroll
  for (int u = 0; u < WU; u++) sD1[s][WU * g + u] = act ? d1[u] * dgelu(z1[u]) : 0.0f;
  __syncthreads();
  // each thread sums whole parameter gradients over the block's samples
  for (int p = threadIdx.x; p < MLP_NPARAM; p += 256) {
    float v = 0.0f;
    int q = p;
    if (q < NH * NIN) {
      const int o = q / NIN, i = q % NIN;
      for (int k = 0; k < WB; k++) v += sD1[k][o] * sX[k][i];
    } else if ((q -= NH * NIN) < NH) {
      for (int k = 0; k < WB; k++) v += sD1[k][q];
    } else if ((q -= NH) < NH * NH) {
      const int o = q / NH, i = q % NH;
      for (int k = 0; k < WB; k++) v += sD2[k][o] * t.a1[k][i];
    } else if ((q -= NH * NH) < NH) {
      for (int k = 0; k < WB; k++) v += sD2[k][q];
    } else if ((q -= NH) < NH) {
      for (int k = 0; k < WB; k++) v += sDy[k] * t.a2[k][q];
    } else {
      for (int k = 0; k < WB; k++) v += sDy[k];
    }
    atomicAdd(&grad[p], v);
  }
  if (g == 0) {
    float l = act ? r * r / (float)B : 0.0f;
    for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o);
    if (s == 0) atomicAdd(loss, l);
  }
}

// Adam update of the FP32 master weights, BF16 copy, gradient and loss reset
__global__ void k_mlp_adam(float* __restrict__ w, uint16_t* __restrict__ wbf, float* __restrict__ m,
                           float* __restrict__ v, float* __restrict__ grad, float* __restrict__ loss, float lr,
                           float bc1, float bc2) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p == 0) *loss = 0.0f;
  if (p >= MLP_NPARAM) return;
  const float g = grad[p];
  const float mm = 0.9f * m[p] + 0.1f * g;
  const float vv = 0.999f * v[p] + 0.001f * g * g;
  m[p] = mm;
  v[p] = vv;
  const float ww = w[p] - lr * (mm / bc1) / (sqrtf(vv / bc2) + 1e-8f);
  w[p] = ww;
  wbf[p] = f_to_bf16(ww);
  grad[p] = 0.0f;
}

__global__ void k_mlp_fill(float* __restrict__ a, int n, float v) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < n) a[p] = v;
}

__global__ void k_mlp_to_bf16(const float* __restrict__ w, uint16_t* __restrict__ wbf) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < MLP_NPARAM) wbf[p] = f_to_bf16(w[p]);
}

// ---------------------------------------------------------------------------
// Inference on the matrix cores (v_mfma_f32_32x32x8bf16_1k): BF16 inputs and
// activations, FP32 accumulation.  A wavefront takes 64 samples as two
// blocks of 32.  Each layer is computed transposed, Z^T = W A^T: the weights
// are the A operand (row = output unit = lane % 32, four inputs 4 (lane / 32)
// + j per lane), the activations the B operand (column = sample = lane % 32,
// four inputs 4 (lane / 32) + j per lane), and the result D holds, in its
// register v, output unit 8 (v / 4) + 4 (lane / 32) + v % 4 of sample
// lane % 32 -- registers 4s..4s+3 are then exactly the B operand of the next
// layer's K-step s, so activations never leave the registers.  Layer 1 pads
// the 6 features to K = 8; layer 2 is four K-steps; layer 3 (32 -> 1) is a
// dot product per lane over its 16 units plus one exchange between the two
// half-waves.
// ---------------------------------------------------------------------------
typedef short mlp_bf16x4 __attribute__((ext_vector_type(4)));
typedef float mlp_f32x16 __attribute__((ext_vector_type(16)));

// tanh-form GELU with the hardware exponential and reciprocal:
// 0.5 x (1 + tanh u) = x / (1 + exp(-2u)); for very negative u the
// exponential overflows to inf and the quotient takes its limit 0
__device__ __forceinline__ float gelu_fast(float x) {
  const float u = 0.7978845608028654f * (x + 0.044715f * x * x * x);
  return x * __builtin_amdgcn_rcpf(1.0f + __expf(-2.0f * u));
}

// per-lane weights of the transposed layers (see above)
struct MlpLaneW {
  mlp_bf16x4 a1, a2[4];
  float b1[16], b2[16], w3[16];
  float b3;
};
__device__ __forceinline__ void mlp_lane_weights(const uint16_t* __restrict__ wbf, MlpLaneW& w) {
  const int lane = threadIdx.x & 63, i = lane & 31, hb = lane >> 5;
  const uint16_t* W1 = wbf;
  const uint16_t* B1 = W1 + NH * NIN;
  const uint16_t* W2 = B1 + NH;
  const uint16_t* B2 = W2 + NH * NH;
  const uint16_t* W3 = B2 + NH;
  for (int j = 0; j < 4; j++) {
    const int kin = 4 * hb + j;
    w.a1[j] = kin < NIN ? (short)W1[i * NIN + kin] : (short)0;
    for (int s = 0; s < 4; s++) w.a2[s][j] = (short)W2[i * NH + 8 * s + 4 * hb + j];
  }
  for (int v = 0; v < 16; v++) {
    const int u = 8 * (v >> 2) + 4 * hb + (v & 3);
    w.b1[v] = bf16_to_f(B1[u]);
    w.b2[v] = bf16_to_f(B2[u]);
    w.w3[v] = bf16_to_f(W3[u]);
  }
  w.b3 = bf16_to_f(W3[NH]);
}

// the network on one block of 32 samples: x0..x3 are the lane's four inputs
// (features 4 (lane / 32) + j of sample lane % 32); returns the output of
// sample lane % 32 in both half-waves
__device__ __forceinline__ float mlp_mfma_block(const MlpLaneW& w, const float (&x)[4]) {
  mlp_bf16x4 b;
  for (int j = 0; j < 4; j++) b[j] = (short)f_to_bf16(x[j]);
  mlp_f32x16 zero;
  for (int v = 0; v < 16; v++) zero[v] = 0.0f;
  const mlp_f32x16 d1 = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(w.a1, b, zero, 0, 0, 0);
  mlp_bf16x4 h[4];
  for (int v = 0; v < 16; v++) h[v >> 2][v & 3] = (short)f_to_bf16(gelu_fast(d1[v] + w.b1[v]));
  mlp_f32x16 d2 = zero;
  for (int s = 0; s < 4; s++) d2 = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(w.a2[s], h[s], d2, 0, 0, 0);
  float part = 0.0f;
  for (int v = 0; v < 16; v++) part += w.w3[v] * gelu_fast(d2[v] + w.b2[v]);
  return part + __shfl_xor(part, 32) + w.b3;
}

// inference on caller rows X[B][ldx] (features in columns 0..5)
__global__ __launch_bounds__(256) void k_mlp_infer(const uint16_t* __restrict__ wbf, const float* __restrict__ X,
                                                   int ldx, int B, float* __restrict__ y) {
  MlpLaneW w;
  mlp_lane_weights(wbf, w);
  const int lane = threadIdx.x & 63, i = lane & 31, hb = lane >> 5;
  // each wave takes 64 samples at a time, strided over the grid (the loop
  // bound is uniform in the wave, so every lane reaches every MFMA)
  const long long step = (long long)gridDim.x * blockDim.x;
  for (long long base = (long long)blockIdx.x * blockDim.x + (threadIdx.x & ~63); base < B; base += step)
    for (int r = 0; r < 2; r++) {
      const long long p = base + 32 * r + i;
      float x[4] = {0.f, 0.f, 0.f, 0.f};
      if (p < B)
        for (int j = 0; j < 4; j++) {
          const int k = 4 * hb + j;
          if (k < NIN) x[j] = X[p * ldx + k];
        }
      const float out = mlp_mfma_block(w, x);
      if (hb == 0 && p < B) y[p] = out;
    }
}

// the seed of the h-rho iteration after the predictor: features formed from
// the particle fields, optionally stored as training rows, and (apply) the
// predictor's h scaled by exp(y / MLP_TSCALE), |y / MLP_TSCALE| <= 0.1;
// fixed boundary particles (itype 1) keep the h the predictor gave them
__global__ __launch_bounds__(256) void k_mlp_seed_mfma(const uint16_t* __restrict__ wbf, MlpSeedFields f) {
  MlpLaneW w;
  mlp_lane_weights(wbf, w);
  const int lane = threadIdx.x & 63, i = lane & 31, hb = lane >> 5;
  const float dtf = (float)f.dt, nexpf = (float)f.nexp, inv_nexp = (float)(1.0 / f.nexp);
  const float dndimf = (float)f.dndim, inv_hfact = (float)(1.0 / f.hfact);
  // 64 particles a wave at a time, strided over the grid, so that the lane
  // weights are loaded once per wave (the loop bound is uniform in the wave)
  const long long step = (long long)gridDim.x * blockDim.x;
  for (long long base = (long long)blockIdx.x * blockDim.x + (threadIdx.x & ~63); base < f.n; base += step)
    for (int r = 0; r < 2; r++) {
      const long long p = base + 32 * r + i;
      const bool ok = p < f.n;
      float x[4] = {0.f, 0.f, 0.f, 0.f};
      double hpred = 0.0;
      // features in FP32 (network inputs; the same arithmetic forms the
      // training rows), the half-wave taking features 0-3 or 4-5
      if (ok) {
        hpred = f.h[p];
        const float hin = (float)f.hin[p], rho = (float)f.rho[p];
        if (hb == 0) {
          x[0] = 100.0f * dtf * (float)f.dhdtin[p] * __builtin_amdgcn_rcpf(hin);
          x[1] = rho > 0.0f ? 100.0f * dtf * (float)f.drhodt[p] * __builtin_amdgcn_rcpf(rho) : 0.0f;
          x[2] = (float)(1000.0 * f.corr[p]);
          x[3] = ((float)f.numneigh[p] - nexpf) * inv_nexp;
        } else {
          x[0] = (float)f.nits[p] - 1.5f;
          x[1] = rho > 0.0f
                     ? 1000.0f * (hin * exp2f(dndimf * __log2f(rho * __builtin_amdgcn_rcpf((float)f.m[p]))) * inv_hfact -
                                  1.0f)
                     : 0.0f;
        }
      }
      const float out = mlp_mfma_block(w, x);
      if (!ok) continue;
      if (f.X) {
        float* row = f.X + p * MLP_LDX;
        if (hb == 0) {
          for (int j = 0; j < 4; j++) row[j] = x[j];
        } else {
          row[4] = x[0];
          row[5] = x[1];
          row[MLP_COL_HPRED] = (float)hpred;
        }
      }
      if (f.apply && hb == 0 && !(f.itype && f.itype[p] == 1)) {
        float yy = out / MLP_TSCALE;
        yy = fminf(fmaxf(yy, -0.1f), 0.1f);
        if (isfinite(yy) && yy != 0.0f && hpred > 0.0) f.h[p] = hpred * (double)__expf(yy);
      }
    }
}

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------

static inline unsigned nb(long long n, int bs) { return (unsigned)((n + bs - 1) / bs); }
// workgroups of the matrix-core inference: four waves each, a few per CU
static constexpr unsigned MLP_MFMA_BLOCKS = 1024;

hipError_t mlp_alloc(MlpState& s, int n) {
  hipError_t e;
  if ((e = hipMalloc(&s.w32, sizeof(float) * MLP_NPARAM))) return e;
  if ((e = hipMalloc(&s.wbf, sizeof(uint16_t) * MLP_NPARAM))) return e;
  if ((e = hipMalloc(&s.m, sizeof(float) * MLP_NPARAM))) return e;
  if ((e = hipMalloc(&s.v, sizeof(float) * MLP_NPARAM))) return e;
  // the loss lies behind the gradient: one copy to the host takes both
  if ((e = hipMalloc(&s.grad, sizeof(float) * (MLP_NPARAM + 1)))) return e;
  s.loss = s.grad + MLP_NPARAM;
  if ((e = hipMalloc(&s.X, sizeof(float) * (size_t)MLP_LDX * n))) return e;
  s.nrows = n;
  hipMemset(s.w32, 0, sizeof(float) * MLP_NPARAM);
  hipMemset(s.wbf, 0, sizeof(uint16_t) * MLP_NPARAM);
  hipMemset(s.m, 0, sizeof(float) * MLP_NPARAM);
  hipMemset(s.v, 0, sizeof(float) * MLP_NPARAM);
  hipMemset(s.grad, 0, sizeof(float) * (MLP_NPARAM + 1));
  hipMemset(s.X, 0, sizeof(float) * (size_t)MLP_LDX * n);
  return hipSuccess;
}

void mlp_free(MlpState& s) {
  void* p[] = {s.w32, s.wbf, s.m, s.v, s.grad, s.X, s.Xext};
  for (void* q : p)
    if (q) (void)hipFree(q);
}

hipError_t mlp_set_params(MlpState& s, const float* host, hipStream_t st) {
  hipError_t e = hipMemcpyAsync(s.w32, host, sizeof(float) * MLP_NPARAM, hipMemcpyHostToDevice, st);
  if (e) return e;
  hipLaunchKernelGGL(k_mlp_to_bf16, dim3(nb(MLP_NPARAM, 256)), dim3(256), 0, st, (const float*)s.w32, s.wbf);
  hipLaunchKernelGGL(k_mlp_fill, dim3(nb(MLP_NPARAM, 256)), dim3(256), 0, st, s.m, MLP_NPARAM, 0.0f);
  hipLaunchKernelGGL(k_mlp_fill, dim3(nb(MLP_NPARAM, 256)), dim3(256), 0, st, s.v, MLP_NPARAM, 0.0f);
  mlp_launch_zero_grad(s, st);
  s.adam_steps = 0;
  s.have_params = 1;
  return hipGetLastError();
}


void mlp_launch_seed_mfma(MlpState& s, const MlpSeedFields& f, hipStream_t st) {
  hipLaunchKernelGGL(k_mlp_seed_mfma, dim3(std::min(nb(f.n, 256), MLP_MFMA_BLOCKS)), dim3(256), 0, st,
                     (const uint16_t*)s.wbf, f);
}

void mlp_launch_infer(MlpState& s, const float* X, int ldx, int B, float* y, hipStream_t st) {
  hipLaunchKernelGGL(k_mlp_infer, dim3(std::min(nb(B, 256), MLP_MFMA_BLOCKS)), dim3(256), 0, st,
                     (const uint16_t*)s.wbf, X, ldx, B, y);
}

void mlp_launch_forward(MlpState& s, const float* X, int ldx, int B, float* y, hipStream_t st) {
  hipLaunchKernelGGL(k_mlp_forward, dim3(nb(B, WB)), dim3(256), 0, st, (const uint16_t*)s.wbf, X, ldx, B, y);
}

void mlp_launch_zero_grad(MlpState& s, hipStream_t st) {
  hipLaunchKernelGGL(k_mlp_fill, dim3(nb(MLP_NPARAM + 1, 256)), dim3(256), 0, st, s.grad, MLP_NPARAM + 1, 0.0f);
  s.grad_zero = true;
}

// (adds to gradient and loss, which a training step or mlp_launch_zero_grad
// leaves zero; a caller that returned early, on an error, left its sums)
void mlp_launch_grad(MlpState& s, const float* X, int ldx, const float* T, int ldt, int nrows, int B, long long off,
                     long long stride, hipStream_t st) {
  if (!s.grad_zero) mlp_launch_zero_grad(s, st);
  s.grad_zero = false;
  hipLaunchKernelGGL(k_mlp_grad, dim3(nb(B, WB)), dim3(256), 0, st, (const uint16_t*)s.wbf, X, ldx, T, ldt, nrows, B, off,
                     stride, s.grad, s.loss);
}

void mlp_launch_adam(MlpState& s, float lr, hipStream_t st) {
  s.adam_steps++;
  const float bc1 = 1.0f - powf(0.9f, (float)s.adam_steps);
  const float bc2 = 1.0f - powf(0.999f, (float)s.adam_steps);
  hipLaunchKernelGGL(k_mlp_adam, dim3(nb(MLP_NPARAM, 256)), dim3(256), 0, st, s.w32, s.wbf, s.m, s.v, s.grad,
                     s.loss, lr, bc1, bc2);
  s.grad_zero = true;
}
