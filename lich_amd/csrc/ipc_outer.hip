// ipc_outer.hip - rank-B outer-product weight update for small batches (gfx950).
//
//   W[m][k] += alpha * sum_{b<B} E[m][b] * f(X[k][b])        (B <= 32)
//
// Replaces SmallBWeightUpdater (src/ipc_tilelang/weight_update_specialization.py:63-128),
// which formed a [B,M,K] temporary with torch.bmm and reduced it; here the
// sum is formed in registers and W is streamed once (read + write), so the
// kernel is bound by HBM traffic on W.  The sign is +alpha as in the GEMM
// weight update and reference.py:57.
//
// A workgroup owns OUTER_TK columns x 4 * RW rows of W, each of its 4 waves RW
// rows, each lane 4 adjacent columns.  What bounds it is W in memory, so a
// thread's loads of W (16 bytes each) are issued before anything else and
// arrive while the rows X[k0 .. k0 + OUTER_TK) are activated, once per element,
// into LDS as [B][OUTER_TK].  MI355X, fp32 2048 x 2048, B = 8: 8.4 us (4.0 TB/s
// of W), against 15.8 with W loaded after the sums, 4 bytes a lane; bf16 8192 x
// 8192, B = 16: 79 us against 246.
#include <type_traits>

#include "ipc_device.h"
#include "ipc_launch.h"

namespace ipc {

constexpr int OUTER_TK = 256;
constexpr int OUTER_LDX = OUTER_TK + 4;

template <typename ST> struct Four { typedef ST T __attribute__((ext_vector_type(4))); };

// VEC: every row of W starts on a multiple of 4 elements (K and the base), so
// that 4 columns are one load and one store.
template <typename ST, int RW, bool VEC>
__global__ void __launch_bounds__(OUTER_TK) outer_kernel(const OuterProblem p) {
  extern __shared__ __align__(16) float xs[];  // [B][OUTER_LDX] f(X), then [B][4 * RW] E
  const int B = p.B, K = p.K, M = p.M;
  const int g = blockIdx.z;
  const int k0 = blockIdx.x * OUTER_TK, m0 = blockIdx.y * (4 * RW);
  const ST* X = reinterpret_cast<const ST*>(p.x) + (long long)g * p.x_gs;
  const ST* E = reinterpret_cast<const ST*>(p.e) + (long long)g * p.e_gs;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int k = k0 + (tid & 63) * 4, mw = m0 + wave * RW;
  ST* W = reinterpret_cast<ST*>(p.w) + (long long)g * p.w_gs + (long long)mw * K + k;
  float* es = xs + B * OUTER_LDX;

  float wv[RW][4];
#pragma unroll
  for (int r = 0; r < RW; ++r) {
#pragma unroll
    for (int j = 0; j < 4; ++j) wv[r][j] = 0.0f;
    if (mw + r >= M) continue;
    if constexpr (VEC) {
      if (k < K) load4(W + (long long)r * K, wv[r]);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (k + j < K) wv[r][j] = to_f32(W[(long long)r * K + j]);
    }
  }

  // f(X): items of up to 8 batch values of a column, in flight together and
  // through one branch on the activation (2, 4, 6 or 8 values, past B the last one
  // again); a thread a column, where the block has at most 64 or 128 columns 4 or
  // 2.  MI355X, us, 8 branches a thread and one thread a column / this: fp32 65 x
  // 65, B = 32, tanh, 6.9 / 4.8; bf16 16 x 64, B = 18, silu, 5.7 / 4.0; fp32 512 x
  // 4096, B = 32, gelu, 10.8 / 9.3.
  const int kn = min(OUTER_TK, K - k0), lg = kn > 128 ? 8 : kn > 64 ? 7 : 6;
  const int col = tid & ((1 << lg) - 1);
  const ST* xrow = X + (long long)(k0 + col) * B;
  const bool xvec = B % 4 == 0 && reinterpret_cast<uintptr_t>(X) % (4 * sizeof(ST)) == 0;
  auto item = [&](auto nv, int b0) {
    constexpr int NV = decltype(nv)::value;
    float v[NV];
    if (xvec && NV % 4 == 0) {
#pragma unroll
      for (int q = 0; q < NV / 4; ++q) {
        float h[4];
        load4(xrow + b0 + q * 4, h);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[q * 4 + j] = h[j];
      }
    } else {
#pragma unroll
      for (int j = 0; j < NV; ++j) v[j] = to_f32(xrow[min(b0 + j, B - 1)]);
    }
    activate<NV>(p.act, v);
#pragma unroll
    for (int j = 0; j < NV; ++j)
      if (b0 + j < B) xs[(b0 + j) * OUTER_LDX + col] = v[j];
  };
  if (col < kn) {
#pragma unroll 1
    for (int b0 = (tid >> lg) * 8; b0 < B; b0 += (OUTER_TK >> lg) * 8) {
      const int left = B - b0;
      if (left > 6) item(std::integral_constant<int, 8>{}, b0);
      else if (left > 4) item(std::integral_constant<int, 6>{}, b0);
      else if (left > 2) item(std::integral_constant<int, 4>{}, b0);
      else item(std::integral_constant<int, 2>{}, b0);
    }
  }
  const int mn = min(4 * RW, M - m0);
  for (int i = tid; i < 4 * RW * B; i += OUTER_TK) {
    const int b = i / (4 * RW), r = i % (4 * RW);
    es[i] = r < mn ? to_f32(E[(long long)(m0 + r) * B + b]) : 0.0f;
  }
  __syncthreads();
  if (k >= K) return;

  float acc[RW][4];
#pragma unroll
  for (int r = 0; r < RW; ++r)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[r][j] = 0.0f;
  for (int b = 0; b < B; ++b) {
    const float4 x = *reinterpret_cast<const float4*>(xs + b * OUTER_LDX + (tid & 63) * 4);
#pragma unroll
    for (int r = 0; r < RW; ++r) {
      const float e = es[b * (4 * RW) + wave * RW + r];
      acc[r][0] += e * x.x;
      acc[r][1] += e * x.y;
      acc[r][2] += e * x.z;
      acc[r][3] += e * x.w;
    }
  }
#pragma unroll
  for (int r = 0; r < RW; ++r) {
    if (mw + r >= M) break;
    ST o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // W + (alpha * acc), each rounded, as the fp32 reference does.
#pragma clang fp contract(off)
      o[j] = cvt<ST>(wv[r][j] + p.alpha * acc[r][j]);
    }
    ST* q = W + (long long)r * K;
    if constexpr (VEC) {
      typename Four<ST>::T v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = o[j];
      *reinterpret_cast<typename Four<ST>::T*>(q) = v;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (k + j < K) q[j] = o[j];
    }
  }
}

// Elementwise activation, used once per batch for the saved input activation
// a[L] = f(x[L]) (trainer.py:510-511).
template <typename ST>
__global__ void __launch_bounds__(256) act_kernel(const ST* src, ST* dst, long long n, int act) {
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256)
    dst[i] = cvt<ST>(act_f(act, to_f32(src[i])));
}

hipError_t launch_act(const void* src, void* dst, long long n, int act, int storage, hipStream_t s) {
  const long long want = (n + 255) / 256;
  const int blocks = (int)(want < 4096 ? (want < 1 ? 1 : want) : 4096);
  if (storage == DT_F32)
    hipLaunchKernelGGL(act_kernel<float>, dim3(blocks), dim3(256), 0, s, (const float*)src, (float*)dst, n, act);
  else if (storage == DT_F16)
    hipLaunchKernelGGL(act_kernel<f16>, dim3(blocks), dim3(256), 0, s, (const f16*)src, (f16*)dst, n, act);
  else
    hipLaunchKernelGGL(act_kernel<bf16>, dim3(blocks), dim3(256), 0, s, (const bf16*)src, (bf16*)dst, n, act);
  return hipGetLastError();
}

template <typename ST, int RW, bool VEC>
static hipError_t run_outer(const OuterProblem& p, hipStream_t s) {
  const dim3 grid((p.K + OUTER_TK - 1) / OUTER_TK, (p.M + 4 * RW - 1) / (4 * RW), p.groups);
  const size_t lds = (size_t)p.B * (OUTER_LDX + 4 * RW) * sizeof(float);  // B <= 32: at most 35,328 bytes
  hipLaunchKernelGGL((outer_kernel<ST, RW, VEC>), grid, dim3(OUTER_TK), lds, s, p);
  return hipGetLastError();
}

template <typename ST>
static hipError_t run_outer_as(const OuterProblem& p, hipStream_t s) {
  const bool vec = p.K % 4 == 0 && reinterpret_cast<uintptr_t>(p.w) % (4 * sizeof(ST)) == 0;
  // 16 rows a workgroup once that gives every CU two of them, else 8 (MI355X,
  // us, 8 / 16 rows and 32, which is not instantiated: fp32 2048 x 2048, B = 8, 8.3 / 7.7 / 7.7 back to back; bf16 8192 x
  // 8192, B = 16, 116 / 79 / 68; fp16, B = 1, 47 / 41 / 44; bf16 1000 x 1531, B =
  // 5, 378 workgroups of 16, 6.3 / 7.3 / 9.8; 8191 x 8191, B = 16, 130 / 104 / 112)
  const long long groups16 = ((p.K + OUTER_TK - 1LL) / OUTER_TK) * ((p.M + 15LL) / 16) * p.groups;
  if (groups16 < 512) return vec ? run_outer<ST, 2, true>(p, s) : run_outer<ST, 2, false>(p, s);
  return vec ? run_outer<ST, 4, true>(p, s) : run_outer<ST, 4, false>(p, s);
}

hipError_t launch_outer(const OuterProblem& p, int storage, hipStream_t s) {
  if (storage == DT_F32) return run_outer_as<float>(p, s);
  if (storage == DT_F16) return run_outer_as<f16>(p, s);
  return run_outer_as<bf16>(p, s);
}

}  // namespace ipc
