// ipc_chunk_kernel.h - the k-chunk GEMM kernel of small and middle-sized problems (gfx950).
//
// The tile kernel of ipc_gemm_kernel.h walks the whole contraction with one
// set of waves, one k-tile's loads in flight at a time: a problem with few
// output tiles then costs (K / 32) memory latencies however little it moves
// (64 x 784 x 128 in fp16: 25 k-tiles of 3 us).  Here the waves of a workgroup
// share one TM x TN output tile and split its contraction instead: wave w
// takes the CHUNK_K columns of chunk w (then w + waves, ...), streams both
// operands from global memory straight into MFMA registers (no LDS staging,
// no barrier; a chunk's loads are issued before the first is used), and the
// chunks' partial products are added through LDS in chunk order.  A problem of
// up to 8 (16 for 16 x 16 tiles) chunks so costs about one memory latency plus
// the reduction.
//
// The sum of an element is ((chunk 0 + chunk 1) + chunk 2) ..., each chunk a
// chain of v_mfma_f32_16x16x32 (16x16x4 for fp32 operands) in k order: the bits
// depend neither on the tile nor on the number of waves, and are those of the
// whole-step kernels' predictions (NARROW_KCHUNK).
//
// Operand lane layout: lane (r = lane % 16, g = lane / 16) of a k-step of KS
// supplies k = k0 + g * KL + q, q < KL, of row / column r.  An operand whose k is contiguous
// is read as KL consecutive values per lane (128 bytes of a row per 4 lanes);
// an operand whose other index is contiguous is read as KL k-rows of NV = tile
// / 16 consecutive values per lane, which makes column tile t the columns
// lr * NV + t (16 lanes read 16 * NV consecutive values).
#pragma once

#include <algorithm>
#include <type_traits>

#include "ipc_device.h"
#include "ipc_gemm_kernel.h"
#include "ipc_launch.h"

namespace ipc {
namespace chunk {

constexpr int CHUNK_K = 128;

template <typename OT> struct Mma;
template <> struct Mma<float> {
  static constexpr int KS = 16, KL = 4;
  typedef f32x4 operand;
  __device__ __forceinline__ static f32x4 run(f32x4 a, f32x4 b, f32x4 c) {
    // instruction s takes k = k0 + 4 g + s from lane group g
#pragma unroll
    for (int s = 0; s < 4; ++s) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], b[s], c, 0, 0, 0);
    return c;
  }
};
template <> struct Mma<f16> {
  static constexpr int KS = 32, KL = 8;
  typedef f16x8 operand;
  __device__ __forceinline__ static f32x4 run(f16x8 a, f16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};
template <> struct Mma<bf16> {
  static constexpr int KS = 32, KL = 8;
  typedef bf16x8 operand;
  __device__ __forceinline__ static f32x4 run(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};

template <typename ST, int N> struct VecOf { typedef ST T __attribute__((ext_vector_type(N))); };

typedef unsigned U2 __attribute__((ext_vector_type(2)));
typedef unsigned U3 __attribute__((ext_vector_type(3)));
typedef unsigned U4 __attribute__((ext_vector_type(4)));
constexpr unsigned OUTSIDE = 0x80000000u;

// An operand matrix of `elements` elements (below 2^31 bytes, which the host
// checks) behind a buffer resource: loads are dword-aligned vectors whatever
// the row length, and a dword past the matrix reads zero.  16-bit matrices
// whose rows or base are not dword-aligned (ODD) load the dwords around the
// values and shift; the resource then ends with the dword that holds the last
// element.
template <typename ST>
struct Mat {
  __amdgpu_buffer_rsrc_t r;
  unsigned mis;  // bytes from the dword-aligned start to element 0
  __device__ __forceinline__ Mat(const ST* base, long long elements) {
    const unsigned long long a = reinterpret_cast<unsigned long long>(base);
    mis = (unsigned)(a & 3);
    r = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(a - mis), (short)0,
                                          (int)((elements * (long long)sizeof(ST) + mis + 3) & ~3LL), 0x00020000);
  }
  __device__ __forceinline__ bool odd(int ld) const { return sizeof(ST) == 2 && ((ld & 1) || mis); }
  // N consecutive elements from element `at` on (`in` false: zeros)
  template <int N, bool ODD>
  __device__ __forceinline__ void ld(unsigned at, bool in, ST* o) const {
    const unsigned off = in ? at * (unsigned)sizeof(ST) + (ODD ? mis : 0u) : OUTSIDE;
    if constexpr (sizeof(ST) == 2 && N == 1) {
      o[0] = __builtin_bit_cast(ST, (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0));
    } else if constexpr (sizeof(ST) == 4) {
      if constexpr (N == 4) put<N>((U4)__builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0), o);
      else if constexpr (N == 2) put<N>((U2)__builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0), o);
      else o[0] = __builtin_bit_cast(ST, (unsigned)__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
    } else if constexpr (!ODD) {
      if constexpr (N == 8) put<N>((U4)__builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0), o);
      else if constexpr (N == 4) put<N>((U2)__builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0), o);
      else put<N>((unsigned)__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0), o);
    } else {
      const unsigned a = off & ~3u, sh = (off & 2u) * 8u;
      unsigned w[N / 2 + 1];
      if constexpr (N == 8) {
        const U4 v = (U4)__builtin_amdgcn_raw_buffer_load_b128(r, a, 0, 0);
        w[0] = v[0]; w[1] = v[1]; w[2] = v[2]; w[3] = v[3];
        w[4] = (unsigned)__builtin_amdgcn_raw_buffer_load_b32(r, a + 16, 0, 0);
      } else if constexpr (N == 4) {
        const U3 v = (U3)__builtin_amdgcn_raw_buffer_load_b96(r, a, 0, 0);
        w[0] = v[0]; w[1] = v[1]; w[2] = v[2];
      } else {
        const U2 v = (U2)__builtin_amdgcn_raw_buffer_load_b64(r, a, 0, 0);
        w[0] = v[0]; w[1] = v[1];
      }
#pragma unroll
      for (int i = 0; i < N / 2; ++i) put<2>(__builtin_amdgcn_alignbit(w[i + 1], w[i], sh), o + 2 * i);
    }
  }
  template <int N, typename U>
  __device__ __forceinline__ static void put(U u, ST* o) {
    const typename VecOf<ST, N>::T v = __builtin_bit_cast(typename VecOf<ST, N>::T, u);
#pragma unroll
    for (int i = 0; i < N; ++i) o[i] = v[i];
  }
};

// One k-step of an operand: T 16-wide tiles of KL values per lane.
template <typename ST, int T, int KL>
struct Raw {
  ST v[T][KL];
};

// k-contiguous operand [rows][ld]: tile t of this lane is row e0 + t*16 + lr,
// KL values from k on.  Values of rows past the matrix may be anything: they
// reach only result rows that are not stored.  `tail` (uniform): the k-step
// reaches past K, where a row's values are the next row's and are zeroed.
template <typename ST, int T, int KL, bool ODD>
__device__ __forceinline__ void load_kmaj(const Mat<ST>& m, int ld, int e0, int k, int K, bool tail, int lr,
                                          Raw<ST, T, KL>& o) {
  constexpr int G = KL * (int)sizeof(ST) > 16 ? 16 / (int)sizeof(ST) : KL;
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const unsigned at = (unsigned)((e0 + t * 16 + lr) * ld + k);
#pragma unroll
    for (int q = 0; q < KL; q += G) m.template ld<G, ODD>(at + q, k + q < K, &o.v[t][q]);
  }
  if (tail) {
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int q = 0; q < KL; ++q) o.v[t][q] = k + q < K ? o.v[t][q] : (ST)0.0f;
  }
}

// [K][ld] operand, the other index contiguous: tile t of this lane is column
// e0 + lr*T + t.  Values of columns past the matrix may be anything (as above).
template <typename ST, int T, int KL, bool ODD>
__device__ __forceinline__ void load_mn(const Mat<ST>& m, int ld, int e0, int k, int K, int lr, Raw<ST, T, KL>& o) {
#pragma unroll
  for (int q = 0; q < KL; ++q) {
    ST x[T];
    m.template ld<T, ODD>((unsigned)((k + q) * ld + e0 + lr * T), k + q < K, x);
#pragma unroll
    for (int t = 0; t < T; ++t) o.v[t][q] = x[t];
  }
}

// The operand registers of a lane's KL values (and their lo terms: v - hi,
// rounded), rounded like cvt: the values are pinned first, so that no product
// behind them is folded into the conversion.
template <typename OT, int KL>
__device__ __forceinline__ typename Mma<OT>::operand round_operand(float (&v)[KL], typename Mma<OT>::operand* lo) {
  typedef typename Mma<OT>::operand V;
  V hi;
  if constexpr (sizeof(OT) == 4) {
#pragma unroll
    for (int q = 0; q < KL; ++q) hi[q] = v[q];
  } else {
    typedef float F8 __attribute__((ext_vector_type(8)));
    F8 f;
#pragma unroll
    for (int q = 0; q < KL; ++q) {
      asm("" : "+v"(v[q]));
      f[q] = v[q];
    }
    hi = __builtin_convertvector(f, V);
    if (lo) {
      F8 d;
#pragma unroll
      for (int q = 0; q < KL; ++q) d[q] = v[q] - to_f32(hi[q]);
      *lo = __builtin_convertvector(d, V);
    }
  }
  return hi;
}

// x_new = x + gamma (-e + f'(x) s) of four elements and, when kept, f(x_new),
// each operation rounded on its own, as in gemm_kernel.
template <typename ST, int ACT>
__device__ __forceinline__ void infer_as(float gamma, bool keep, const float (&x)[4], const float (&e)[4],
                                         const float (&s)[4], ST (&o)[4], ST (&a)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma clang fp contract(off)
    const float xn = x[i] + gamma * (-e[i] + dact_t<ACT>(x[i]) * s[i]);
    o[i] = cvt<ST>(xn);
    if (keep) a[i] = cvt<ST>(act_t<ACT>(xn));
  }
}
template <typename ST>
__device__ __forceinline__ void infer_group(int act, float gamma, bool keep, const float (&x)[4], const float (&e)[4],
                                            const float (&s)[4], ST (&o)[4], ST (&a)[4]) {
  switch (act) {
    case ACT_RELU: return infer_as<ST, ACT_RELU>(gamma, keep, x, e, s, o, a);
    case ACT_TANH: return infer_as<ST, ACT_TANH>(gamma, keep, x, e, s, o, a);
    case ACT_SIGMOID: return infer_as<ST, ACT_SIGMOID>(gamma, keep, x, e, s, o, a);
    case ACT_SILU: return infer_as<ST, ACT_SILU>(gamma, keep, x, e, s, o, a);
    case ACT_GELU: return infer_as<ST, ACT_GELU>(gamma, keep, x, e, s, o, a);
    default: return infer_as<ST, ACT_IDENTITY>(gamma, keep, x, e, s, o, a);
  }
}

// Fewest waves of a launch: enough for one or two epilogue groups per thread,
// also where the contraction has fewer chunks (1792 x 16 x 448 inference, tanh,
// 64 x 64 tiles: 26 us with one wave per tile).
constexpr int min_waves(int TM, int TN, int MAXW) {
  return TM * TN / 256 < MAXW ? TM * TN / 256 : MAXW;
}

// NS: waves that share a chunk, each with TN / NS of the tile's columns, where
// the contraction has fewer chunks than the workgroup waves; OCC: waves per SIMD
// the registers leave room for, that is workgroups a CU holds (run_chunk8).
template <typename ST, typename OT, int LAYOUT, int SPLIT, int TM, int TN, int MAXW, int NS, int OCC>
__global__ void __launch_bounds__(MAXW * 64, OCC) chunk_kernel(const GemmBatch batch) {
  using MM = Mma<OT>;
  typedef typename MM::operand V;
  constexpr int KS = MM::KS, KL = MM::KL, RM = TM / 16, RN = TN / 16 / NS;
  constexpr bool A_KMAJ = LAYOUT != LAYOUT_INF, B_KMAJ = LAYOUT == LAYOUT_WGT;
  constexpr bool SA = SPLIT >= 2, SB = SPLIT >= 3;
  constexpr int LDP = TN + 4;                       // floats per row of a partial tile
  constexpr int STEPS = CHUNK_K / KS;
  extern __shared__ __align__(16) float part[];     // [chunks in flight][TM][LDP]

  const int bid = blockIdx.x;
  int pi = 0;
#pragma unroll 1
  while (pi + 1 < batch.count && bid >= batch.start[pi + 1]) ++pi;
  const GemmProblem& p = batch.p[pi];
  const int M = p.M, N = p.N, K = p.K;
  const int tn = (N + TN - 1) / TN, tm = (M + TM - 1) / TM;
  const int local = bid - batch.start[pi];
  const int g = local / (tn * tm);
  const int rem = local - g * (tn * tm);
  const int m0 = (rem / tn) * TM, n0 = (rem % tn) * TN;
  const int lda = (int)p.lda, ldb = (int)p.ldb;
  const Mat<ST> A(reinterpret_cast<const ST*>(p.a) + (long long)g * p.a_gs, (long long)(A_KMAJ ? M : K) * lda);
  const Mat<ST> B(reinterpret_cast<const ST*>(p.b) + (long long)g * p.b_gs, (long long)(B_KMAJ ? N : K) * ldb);
  ST* out = reinterpret_cast<ST*>(p.out) + (long long)g * p.o_gs;
  const ST* aux = p.aux ? reinterpret_cast<const ST*>(p.aux) + (long long)g * p.x_gs : nullptr;
  ST* out2 = p.out2 ? reinterpret_cast<ST*>(p.out2) + (long long)g * p.o2_gs : nullptr;
  const long long ldo = p.ldo, ldx = p.ldx, ld2 = p.ld2;
  const int act_b = p.act_b, kind = p.kind;

  const int tid = threadIdx.x, nthreads = blockDim.x, lane = tid & 63, lr = tid & 15, lg = lane >> 4;
  // (uniform, so that the chunk's addresses are scalar)
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), slots = (nthreads >> 6) / NS;
  const int slot = wave / NS, nw = wave % NS * (TN / NS);  // this wave's chunk of a round, its first column
  const int chunks = (K + CHUNK_K - 1) / CHUNK_K;

  // The epilogue's 4-column groups: group tid, then every nthreads (at most
  // PRE of them each, min_waves).  Their inputs are fetched before the
  // contraction.
  constexpr int GROUPS = TM * TN / 4, PRE = GROUPS / (64 * min_waves(TM, TN, MAXW));
  const bool need_x = kind != KIND_FWD;
  const ST* xin = kind == KIND_PRED ? aux : out;
  const long long ldin = kind == KIND_PRED ? ldx : ldo;
  auto aligned4 = [](const void* q, long long ld) {
    return ld % 4 == 0 && reinterpret_cast<uintptr_t>(q) % (4 * sizeof(ST)) == 0;
  };
  const bool vx = need_x && aligned4(xin, ldin);
  const bool ve = kind == KIND_INFER && aligned4(aux, ldx);
  const bool vo = aligned4(out, ldo), v2 = out2 && aligned4(out2, ld2);
  auto load_group = [&](const ST* src, long long ld, bool vec, int gi, float (&o)[4]) {
    const int r = gi / (TN / 4), c = (gi % (TN / 4)) * 4;
    const int m = m0 + r, n = n0 + c;
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = 0.0f;
    if (m >= M || n >= N) return;
    const ST* q = src + (long long)m * ld + n;
    if (vec && n + 4 <= N) {
      load4(q, o);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n + i < N) o[i] = to_f32(q[i]);
    }
  };
  float xs[PRE][4], es[PRE][4];
#pragma unroll
  for (int i = 0; i < PRE; ++i) {
    const int gi = tid + i * nthreads;
    if (gi >= GROUPS) continue;
    if (need_x) load_group(xin, ldin, vx, gi, xs[i]);
    if (LAYOUT == LAYOUT_INF) load_group(aux, ldx, ve, gi, es[i]);
  }

  for (int c0 = 0; c0 < chunks; c0 += slots) {
    const int c = c0 + slot;
    if (c < chunks) {
      f32x4 acc[RM][RN];
#pragma unroll
      for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      const int kend = K - c * CHUNK_K < CHUNK_K ? K : (c + 1) * CHUNK_K;
      auto steps = [&](auto ODDV) {
        constexpr bool ODD = decltype(ODDV)::value;
        // k-steps whose loads are issued together: as many as about half of
        // the registers hold
        constexpr int REGS = (RM + RN) * KL * (ODD ? 4 : (int)sizeof(ST)) / 4;
        constexpr int ROOM = MAXW > 8 ? (ODD ? 16 : 48) : OCC >= 4 ? 48 : TM > 32 ? 96 : 128;
        constexpr int AHEAD = REGS * STEPS <= ROOM ? STEPS : REGS * STEPS <= 2 * ROOM ? STEPS / 2
                              : REGS * STEPS <= 4 * ROOM ? STEPS / 4 : 1;
        Raw<ST, RM, KL> ra[AHEAD];
        Raw<ST, RN, KL> rb[AHEAD];
#pragma unroll 1
        for (int k0 = c * CHUNK_K; k0 < kend; k0 += AHEAD * KS) {
          const bool tail = k0 + AHEAD * KS > K;
#pragma unroll
          for (int s = 0; s < AHEAD; ++s) {
            const int k = k0 + s * KS + lg * KL;
            if constexpr (A_KMAJ) load_kmaj<ST, RM, KL, ODD>(A, lda, m0, k, K, tail, lr, ra[s]);
            else load_mn<ST, RM, KL, ODD>(A, lda, m0, k, K, lr, ra[s]);
            if constexpr (B_KMAJ) load_kmaj<ST, RN, KL, ODD>(B, ldb, n0 + nw, k, K, tail, lr, rb[s]);
            else load_mn<ST, RN, KL, ODD>(B, ldb, n0 + nw, k, K, lr, rb[s]);
          }
#pragma unroll
          for (int s = 0; s < AHEAD; ++s) {
            if (k0 + s * KS >= kend) break;
            V ah[RM], al[SA ? RM : 1], bh[RN], bl[SB ? RN : 1];
#pragma unroll
            for (int i = 0; i < RM; ++i) {
              if constexpr (std::is_same<ST, OT>::value) {
#pragma unroll
                for (int q = 0; q < KL; ++q) ah[i][q] = ra[s].v[i][q];
              } else {
                float f[KL];
#pragma unroll
                for (int q = 0; q < KL; ++q) f[q] = to_f32(ra[s].v[i][q]);
                ah[i] = round_operand<OT, KL>(f, SA ? &al[SA ? i : 0] : nullptr);
              }
            }
#pragma unroll
            for (int j = 0; j < RN; ++j) {
              bool raw = false;
              if constexpr (std::is_same<ST, OT>::value) {
                if (LAYOUT == LAYOUT_INF || act_b == ACT_IDENTITY) {
                  raw = true;
#pragma unroll
                  for (int q = 0; q < KL; ++q) bh[j][q] = rb[s].v[j][q];
                }
              }
              if (!raw) {
                float f[KL];
#pragma unroll
                for (int q = 0; q < KL; ++q) f[q] = to_f32(rb[s].v[j][q]);
                if (LAYOUT != LAYOUT_INF) activate<KL>(act_b, f);
                bh[j] = round_operand<OT, KL>(f, SB ? &bl[SB ? j : 0] : nullptr);
              }
            }
#pragma unroll
            for (int i = 0; i < RM; ++i)
#pragma unroll
              for (int j = 0; j < RN; ++j) {
                acc[i][j] = MM::run(ah[i], bh[j], acc[i][j]);
                if (SA) acc[i][j] = MM::run(al[SA ? i : 0], bh[j], acc[i][j]);
                if (SB) acc[i][j] = MM::run(ah[i], bl[SB ? j : 0], acc[i][j]);
              }
          }
        }
      };
      if constexpr (sizeof(ST) == 2) {
        if (A.odd(lda) || B.odd(ldb)) steps(std::integral_constant<bool, true>{});
        else steps(std::integral_constant<bool, false>{});
      } else {
        steps(std::integral_constant<bool, false>{});
      }
      // the partial tile in matrix order: result register q of tile (i, j) is
      // operand row 4 lg + q of row tile i, column lr of column tile j
      float* pw = part + slot * TM * LDP + nw;
#pragma unroll
      for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int r = A_KMAJ ? i * 16 + 4 * lg + q : (4 * lg + q) * RM + i;
          if constexpr (!B_KMAJ && RN == 4) {
            *reinterpret_cast<float4*>(pw + r * LDP + lr * 4) =
                make_float4(acc[i][0][q], acc[i][1][q], acc[i][2][q], acc[i][3][q]);
          } else {
#pragma unroll
            for (int j = 0; j < RN; ++j) pw[r * LDP + (B_KMAJ ? j * 16 + lr : lr * RN + j)] = acc[i][j][q];
          }
        }
    }
    __syncthreads();
    const int have = chunks - c0 < slots ? chunks - c0 : slots;
    const bool last = c0 + slots >= chunks;
#pragma unroll
    for (int u = 0; u < PRE; ++u) {
      const int gi = tid + u * nthreads;
      if (gi >= GROUPS) break;
      const int r = gi / (TN / 4), cc = (gi % (TN / 4)) * 4;
      float* at = part + r * LDP + cc;
      // running sum of the earlier rounds: kept after the chunks' partial tiles
      float* run = part + slots * TM * LDP + r * LDP + cc;
      float4 t = *reinterpret_cast<float4*>(at);
      float s[4] = {t.x, t.y, t.z, t.w};
      if (c0 > 0) {
        const float4 u = *reinterpret_cast<float4*>(run);
        s[0] = u.x + s[0]; s[1] = u.y + s[1]; s[2] = u.z + s[2]; s[3] = u.w + s[3];
      }
      for (int w = 1; w < have; ++w) {
        t = *reinterpret_cast<float4*>(at + w * TM * LDP);
        s[0] = s[0] + t.x; s[1] = s[1] + t.y; s[2] = s[2] + t.z; s[3] = s[3] + t.w;
      }
      if (!last) {
        *reinterpret_cast<float4*>(run) = make_float4(s[0], s[1], s[2], s[3]);
        continue;
      }
      const int m = m0 + r, n = n0 + cc;
      if (m >= M || n >= N) continue;
      const float (&x)[4] = xs[u], (&e)[4] = es[u];
      ST o[4], o2[4];
      if constexpr (LAYOUT == LAYOUT_INF) {
        infer_group<ST>(p.act_epi, p.scal, out2 != nullptr, x, e, s, o, o2);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          // every epilogue operation rounds on its own, as in gemm_kernel
#pragma clang fp contract(off)
          if (LAYOUT == LAYOUT_PF) o[i] = kind == KIND_PRED ? cvt<ST>(x[i] - to_f32(cvt<ST>(s[i]))) : cvt<ST>(s[i]);
          else o[i] = cvt<ST>(x[i] + p.scal * s[i]);
        }
      }
      auto store_group = [&](ST* dst, long long ld, bool vec, const ST (&v)[4]) {
        ST* q = dst + (long long)m * ld + n;
        if (vec && n + 4 <= N) {
          typename VecOf<ST, 4>::T w;
#pragma unroll
          for (int i = 0; i < 4; ++i) w[i] = v[i];
          *reinterpret_cast<typename VecOf<ST, 4>::T*>(q) = w;
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (n + i < N) q[i] = v[i];
        }
      };
      store_group(out, ldo, vo, o);
      if (LAYOUT == LAYOUT_INF && out2) store_group(out2, ld2, v2, o2);
    }
    if (!last) __syncthreads();
  }
}

// Launch of one tile size over a ragged batch.
template <typename ST, typename OT, int LAYOUT, int SPLIT, int TM, int TN, int MAXW, int NS, int OCC>
static hipError_t run_chunk(const GemmProblem* probs, int count, hipStream_t s) {
  const void* fn = reinterpret_cast<const void*>(&chunk_kernel<ST, OT, LAYOUT, SPLIT, TM, TN, MAXW, NS, OCC>);
  constexpr int TILE_BYTES = TM * (TN + 4) * 4;
  constexpr int LDS_MAX = (MAXW / NS + 1) * TILE_BYTES;
  static_assert(LDS_MAX <= 160 * 1024, "partial tiles exceed the LDS");
  if (LDS_MAX > 64 * 1024) {
    static const hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_MAX);
    if (e != hipSuccess) return e;
  }
  for (int base = 0; base < count; base += MAX_BATCH) {
    GemmBatch batch;
    batch.count = count - base < MAX_BATCH ? count - base : MAX_BATCH;
    int total = 0, most = 1;
    for (int i = 0; i < batch.count; ++i) {
      const GemmProblem& q = probs[base + i];
      batch.p[i] = q;
      batch.start[i] = total;
      total += ((q.N + TN - 1) / TN) * ((q.M + TM - 1) / TM) * q.groups;
      most = std::max(most, (q.K + CHUNK_K - 1) / CHUNK_K);
    }
    for (int i = batch.count; i <= MAX_BATCH; ++i) batch.start[i] = total;
    if (total == 0) continue;
    // partial tiles: a round's chunks, and the running sum where there are more
    // rounds; no more than that, so that a CU holds several workgroups of few
    // chunks
    const int slots = std::min(most, MAXW / NS), waves = std::max(min_waves(TM, TN, MAXW), slots * NS);
    const int tiles = most > slots ? slots + 1 : slots;
    void* args[] = {&batch};
    const hipError_t err = hipLaunchKernel(fn, dim3(total), dim3(waves * 64), args, (size_t)tiles * TILE_BYTES, s);
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

// Waves per chunk: where the longest contraction leaves an 8-wave workgroup
// without a chunk for every wave, 2 or 4 waves take columns of one chunk each.
// An operand A is then read by all of them, so the inference update, whose
// narrower transposing reads cost more (1000 x 200 x 1000 10.4 -> 12.9 us), and
// 16-bit storage with two (2000 x 400 x 500 weight update 16.7 -> 24) keep one.
// MI355X, us, one wave a chunk / this rule: weight update 1000 x 1531, B = 300,
// fp32 storage, bf16 operands 29.7 / 20.1, fp32 operands 44.4 / 28.7, bf16
// storage 32.5 / 21.6; 1024 x 1024, B = 128, 13.6 / 9.5, 21.1 / 10.3, 14.6 / 8.9;
// prediction 1000 x 200 x 1000 12.0 / 9.4, 19.0 / 10.8, 12.5 / 9.1.
//
// Workgroups per CU: two of 32 x 32 tiles, each with fewer loads in flight,
// hide one another's latencies and reductions (prediction 1000 x 1531 x 300,
// the three types in the same order, 37.1 -> 27.0 us, 48.8 -> 33.4, 36.1 -> 28.0;
// inference 800 x 800 x 400 17.5 -> 12.3, 26.8 -> 21.0, 14.7 -> 11.4); an inference
// update of at most one tile per CU keeps the loads instead (512 x 4096 x 512,
// fp32, 42.7 us against 54.7).
template <typename ST, typename OT, int LAYOUT, int SPLIT, int TM, int TN>
static hipError_t run_chunk8(const GemmProblem* probs, int count, hipStream_t s) {
  constexpr bool wide = sizeof(ST) == 4;
  int kmax = 0;
  for (int i = 0; i < count; ++i) kmax = std::max(kmax, probs[i].K);
  if constexpr (LAYOUT != LAYOUT_INF && TN == 64)
    if (kmax <= (wide ? 2 : 3) * CHUNK_K) return run_chunk<ST, OT, LAYOUT, SPLIT, TM, TN, 8, 4, 4>(probs, count, s);
  if constexpr (LAYOUT != LAYOUT_INF && (wide || (LAYOUT == LAYOUT_WGT && TN == 32)))
    if (kmax <= 4 * CHUNK_K) return run_chunk<ST, OT, LAYOUT, SPLIT, TM, TN, 8, 2, 4>(probs, count, s);
  if constexpr (TN == 32) {
    long long tiles = 0;
    for (int i = 0; i < count; ++i) tiles += ((probs[i].M + 31LL) / 32) * ((probs[i].N + 31LL) / 32) * probs[i].groups;
    if (LAYOUT != LAYOUT_INF || tiles > 256) return run_chunk<ST, OT, LAYOUT, SPLIT, TM, TN, 8, 1, 4>(probs, count, s);
  }
  return run_chunk<ST, OT, LAYOUT, SPLIT, TM, TN, 8, 1, 2>(probs, count, s);
}

template <typename ST, typename OT, int LAYOUT, int SPLIT>
static hipError_t run_chunks(const GemmProblem* probs, int count, int tile, hipStream_t s) {
  switch (tile) {
    case TILE_CHUNK_16: return run_chunk<ST, OT, LAYOUT, SPLIT, 16, 16, 16, 1, 4>(probs, count, s);
    case TILE_CHUNK_32: return run_chunk8<ST, OT, LAYOUT, SPLIT, 32, 32>(probs, count, s);
    default: return run_chunk8<ST, OT, LAYOUT, SPLIT, 64, 64>(probs, count, s);
  }
}

}  // namespace chunk
}  // namespace ipc
