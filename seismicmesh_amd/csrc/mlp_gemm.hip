// FP32 product on the matrix cores, with the surrogate's elementwise work in
// the epilogue (mlp_gemm.h).
//
// A workgroup of 4 waves computes a 128 x 128 tile (64 x 64 with MT = 1),
// each wave a quarter of it as MT x MT blocks of v_mfma_f32_32x32x2_f32.
// Slices of 16 k go through LDS, double buffered: the next slice's global
// loads are in flight while this one is multiplied, one barrier a slice.  An
// operand contiguous in k is staged as [row][k] (rows of 20 words: the 16-B
// reads of 16 rows fall in 64 different banks) and read four k at a time; one
// contiguous in m or n as [k][column] (rows of 32 mod 64 words, so the two
// k of one instruction use different halves of the banks).  Both halves of a
// wave take their k four apart, in the same order for A and B.
#include "mlp_gemm.h"

#include <algorithm>
#include <type_traits>

namespace smk {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kKT = 16;
constexpr int kRowK = kKT + 4;

// LDS words of one staged operand of T rows or columns
template <int T>
constexpr int stage_words(bool kmajor) {
  return kmajor ? T * kRowK : kKT * (T + 32);
}

// One slice of an operand, T x kKT values by 256 threads: T / 64 float4 each.
// Out of range is zero.
template <int T, bool KM>
struct Stage {
  static constexpr int kV = T / 64;
  float4 v[kV];
  __device__ void load(const float *P, int64_t ld, int64_t t0, int64_t tn, int64_t k0,
                       int64_t kn) {
#pragma unroll
    for (int i = 0; i < kV; ++i) {
      const int e = threadIdx.x + 256 * i;
      v[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (KM) {
        const int64_t r = t0 + e / 4, k = k0 + 4 * (e % 4);
        if (r < tn && k < kn) v[i] = *reinterpret_cast<const float4 *>(P + r * ld + k);
      } else {
        const int64_t k = k0 + e / (T / 4), c = t0 + 4 * (e % (T / 4));
        if (k < kn && c < tn) v[i] = *reinterpret_cast<const float4 *>(P + k * ld + c);
      }
    }
  }
  __device__ void store(float *sh) const {
#pragma unroll
    for (int i = 0; i < kV; ++i) {
      const int e = threadIdx.x + 256 * i;
      float *d = KM ? sh + (e / 4) * kRowK + 4 * (e % 4)
                    : sh + (e / (T / 4)) * (T + 32) + 4 * (e % (T / 4));
      *reinterpret_cast<float4 *>(d) = v[i];
    }
  }
};

template <int T, bool KM>
__device__ inline void fragment(const float *sh, int row, int g, int half, float *f) {
  if (KM) {
    const float4 q = *reinterpret_cast<const float4 *>(sh + row * kRowK + 8 * g + 4 * half);
    f[0] = q.x;
    f[1] = q.y;
    f[2] = q.z;
    f[3] = q.w;
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) f[j] = sh[(8 * g + 4 * half + j) * (T + 32) + row];
  }
}

template <int EPI, bool AK, bool BK, int MT>
__global__ __launch_bounds__(256, EPI == kEpiStore || EPI == kEpiPart ? 3 : 2) void k_gemm32(
    GemmArgs g, int64_t kchunk) {
  constexpr int T = 64 * MT;
  constexpr int kA = stage_words<T>(AK), kB = stage_words<T>(BK);
  __shared__ __align__(16) float As[2][kA];
  __shared__ __align__(16) float Bs[2][kB];
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int r = lane % 32, half = lane / 32;
  const int wm = (wave / 2) * 32 * MT, wn = (wave % 2) * 32 * MT;
  // tiles of one row of tiles are neighbours (they share A's rows); both
  // indices in grid.x, since grid.y ends at 65535
  const unsigned tn = (unsigned)((g.N + T - 1) / T), tm = blockIdx.x / tn;
  const int64_t m0 = (int64_t)tm * T, n0 = (int64_t)(blockIdx.x - tm * tn) * T;
  const int64_t kb = (int64_t)blockIdx.z * kchunk, ke = kb + kchunk < g.K ? kb + kchunk : g.K;
  floatx16 acc[MT][MT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  Stage<T, AK> sa;
  Stage<T, BK> sb;
  sa.load(g.A, g.lda, m0, g.M, kb, ke);
  sb.load(g.B, g.ldb, n0, g.N, kb, ke);
  sa.store(As[0]);
  sb.store(Bs[0]);
  int buf = 0;
  for (int64_t k0 = kb; k0 < ke; k0 += kKT) {
    const bool more = k0 + kKT < ke;
    if (more) {
      sa.load(g.A, g.lda, m0, g.M, k0 + kKT, ke);
      sb.load(g.B, g.ldb, n0, g.N, k0 + kKT, ke);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kKT / 8; ++q) {
      float fa[MT][4], fb[MT][4];
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        fragment<T, AK>(As[buf], wm + 32 * i + r, q, half, fa[i]);
        fragment<T, BK>(Bs[buf], wn + 32 * i + r, q, half, fb[i]);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int a = 0; a < MT; ++a)
#pragma unroll
          for (int b = 0; b < MT; ++b)
            acc[a][b] =
                __builtin_amdgcn_mfma_f32_32x32x2f32(fa[a][j], fb[b][j], acc[a][b], 0, 0, 0);
    }
    if (more) {
      sa.store(As[buf ^ 1]);
      sb.store(Bs[buf ^ 1]);
    }
    buf ^= 1;
  }
  // Element e of a block: row (e % 4) + 8 (e / 4) + 4 half, column r.  A
  // tile inside the matrix takes the epilogue without bounds checks, its
  // loads ahead of the arithmetic.
  float cs[MT];
  const auto epilogue = [&](auto inside) {
    constexpr bool kIn = decltype(inside)::value;
#pragma unroll
    for (int b = 0; b < MT; ++b) {
      const int64_t n = n0 + wn + 32 * b + r;
      cs[b] = 0.0f;
      const float bias = EPI == kEpiSilu && (kIn || n < g.N) ? g.vec[n] : 0.0f;
#pragma unroll
      for (int a = 0; a < MT; ++a) {
        const int64_t m1 = m0 + wm + 32 * a + 4 * half;
        float zv[16];
        if (EPI == kEpiSiluBack)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const int64_t m = m1 + (e % 4) + 8 * (e / 4);
            zv[e] = kIn || (m < g.M && n < g.N) ? g.vec[m * g.ldc + n] : 0.0f;
          }
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int64_t m = m1 + (e % 4) + 8 * (e / 4);
          if (!kIn && (m >= g.M || n >= g.N)) continue;
          const float v = acc[a][b][e];
          if (EPI == kEpiStore) {
            float *c = g.C + m * g.ldc + n;
            *c = g.alpha * v + (g.beta != 0.0f ? g.beta * *c : 0.0f);
          } else if (EPI == kEpiPart) {
            g.C[((int64_t)blockIdx.z * g.M + m) * g.N + n] = v;
          } else if (EPI == kEpiSilu) {
            const float z = v + bias;
            g.C[m * g.ldc + n] = z;
            g.C2[m * g.ldc + n] = train_silu(z);
          } else {
            const float z = zv[e], s = train_sigmoid(z);
            const float d = v * s * (1.0f + z * (1.0f - s));
            g.C[m * g.ldc + n] = d;
            cs[b] += d;
          }
        }
      }
    }
  };
  if (m0 + T <= g.M && n0 + T <= g.N) epilogue(std::true_type{});
  else epilogue(std::false_type{});
  if (EPI == kEpiSiluBack) {
    // column sums of the tile: both halves, then both rows of waves
    __syncthreads();
    float *red = As[0];
#pragma unroll
    for (int b = 0; b < MT; ++b) {
      const float t = cs[b] + __shfl_xor(cs[b], 32);
      if (half == 0) red[(wave / 2) * T + wn + 32 * b + r] = t;
    }
    __syncthreads();
    for (int c = threadIdx.x; c < T; c += 256)
      if (n0 + c < g.N) g.C2[(int64_t)tm * g.N + n0 + c] = red[c] + red[T + c];
  }
}

constexpr int64_t kMaxTiles = (int64_t)1 << 23;

int64_t split_chunk(const GemmArgs &g) {
  const int64_t per = (g.K + g.nsplit - 1) / std::max(g.nsplit, 1);
  return std::max<int64_t>(kKT, (per + kKT - 1) / kKT * kKT);
}

template <int EPI, bool AK, bool BK>
void launch(const GemmArgs &g, bool small, hipStream_t s) {
  const int64_t T = small ? 64 : 128;
  const int64_t chunk = EPI == kEpiPart ? split_chunk(g) : std::max<int64_t>(g.K, 1);
  const dim3 grid((unsigned)(((g.N + T - 1) / T) * ((g.M + T - 1) / T)), 1u,
                  EPI == kEpiPart ? (unsigned)gemm32_splits(g) : 1u);
  if (small)
    hipLaunchKernelGGL((k_gemm32<EPI, AK, BK, 1>), grid, dim3(256), 0, s, g, chunk);
  else
    hipLaunchKernelGGL((k_gemm32<EPI, AK, BK, 2>), grid, dim3(256), 0, s, g, chunk);
}

template <int EPI>
void launch_layout(bool ak, bool bk, const GemmArgs &g, bool small, hipStream_t s) {
  if (ak && bk) launch<EPI, true, true>(g, small, s);
  else if (ak) launch<EPI, true, false>(g, small, s);
  else if (bk) launch<EPI, false, true>(g, small, s);
  else launch<EPI, false, false>(g, small, s);
}

}  // namespace

int gemm32_splits(const GemmArgs &g) {
  const int64_t c = split_chunk(g);
  return (int)std::max<int64_t>(1, (g.K + c - 1) / c);
}

// 16-byte loads: the contiguous index in fours, strides and bases aligned;
// no more tiles than a grid's threads (2^32) have room for
bool gemm32_takes(bool ak, bool bk, const GemmArgs &g) {
  const auto ok = [&](const float *p, int64_t ld, int64_t run) {
    return ((uintptr_t)p & 15) == 0 && ld % 4 == 0 && run % 4 == 0 && ld >= run;
  };
  return g.M > 0 && g.N > 0 && g.K > 0 && ok(g.A, g.lda, ak ? g.K : g.M) &&
         ok(g.B, g.ldb, bk ? g.K : g.N) &&
         (g.M + 63) / 64 <= kMaxTiles / ((g.N + 63) / 64);
}

int gemm32(GemmEpi epi, bool ak, bool bk, const GemmArgs &g, bool small, hipStream_t s) {
  SM_CHECK(gemm32_takes(ak, bk, g), SM_ERR_ARG, "gemm32: shape or alignment not taken");
  switch (epi) {
    case kEpiStore: launch_layout<kEpiStore>(ak, bk, g, small, s); break;
    case kEpiPart: launch_layout<kEpiPart>(ak, bk, g, small, s); break;
    case kEpiSilu: launch<kEpiSilu, true, true>(g, small, s); break;
    case kEpiSiluBack: launch<kEpiSiluBack, true, false>(g, small, s); break;
  }
  SM_LAUNCH_CHECK();
  return SM_OK;
}

}  // namespace smk
