// Pieces shared by the any-shape kernels: a tile of token rows in LDS times a weight matrix read
// from L2, on the matrix cores, for every I/O type.
//
// 16-bit types use v_mfma_f32_32x32x16; fp32 uses v_mfma_f32_32x32x2_f32, four per 16-byte operand,
// so one piece of code serves all three: a lane always holds 16 bytes (VE elements) of a row's k
// range, lane half hl the second half of a k-step of KS = 2 VE elements.
#pragma once

#include "common.hpp"

namespace tops {

template <typename T>
struct TileMma {
  static constexpr int VE = 8, KS = 16;
  using V = vec<T, 8>;
  __device__ static inline f32x16 mma(V a, V b, f32x16 c) { return Mma<T>::m32(a, b, c); }
};
template <>
struct TileMma<float> {
  static constexpr int VE = 4, KS = 8;
  using V = vec<float, 4>;
  __device__ static inline f32x16 mma(V a, V b, f32x16 c) {
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], c, 0, 0, 0);
    return c;
  }
};

// Raw buffer loads: 32-bit byte offsets from one base, reads at or past `bytes` return 0.
using Rsrc = __amdgpu_buffer_rsrc_t;
__device__ inline Rsrc buffer_of(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}
template <typename V>
__device__ inline V buffer_load(Rsrc r, uint32_t off) {
  if constexpr (sizeof(V) == 16)
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
  else if constexpr (sizeof(V) == 4)
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
  else
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0));
}

// Channels of an LDS token row: C rounded up to 32, the tail zero.  Rows are 16 bytes longer than
// that, an odd number of 16-byte slots, so 16 rows read together hit 16 distinct bank groups.
__host__ __device__ inline int tile_kp(int C) { return (C + 31) / 32 * 32; }
template <typename T>
__host__ __device__ inline int tile_row(int C) {
  return tile_kp(C) + TileMma<T>::VE;
}

// Row r of an A operand's 32 rows holds feature (or token) tile_perm(r) of the 32: D slot v of lane
// half hl is then number 16 hl + v, 16 consecutive ones per lane.
__device__ inline int tile_perm(int r) { return 16 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3); }

// Sum over the TPT threads of a token (adjacent lanes).
template <int TPT>
__device__ inline float token_sum(float v) {
  if constexpr (TPT == 32) {
    v = group_sum<16>(v);
    return v + __shfl_xor(v, 16);
  } else {
    return group_sum<TPT>(v);
  }
}

// This thread's 16-byte chunks (part, part + TPT, ...) of one token row into LDS; channels >= C and
// rows that do not exist (ok false) are zero.  VEC: C is a multiple of VE and the rows are 16-byte
// aligned, so chunks are loaded whole (a compile-time choice: a branch at each load would make the
// compiler wait for every load before the next).
template <typename T, int TPT, bool VEC>
__device__ __attribute__((always_inline)) inline void stage_row(T* dst, const T* src, bool ok, int part, int C,
                                                                int KP) {
  using M = TileMma<T>;
  constexpr int U = 4;  // loads in flight per thread
  for (int c0 = part; c0 < KP / M::VE; c0 += U * TPT) {
    typename M::V v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = (c0 + u * TPT) * M::VE;
      if constexpr (VEC) {
        v[u] = ldg<typename M::V>(src + (k < C ? k : 0));
        if (!ok || k >= C) v[u] = typename M::V{};
      } else {
#pragma unroll
        for (int e = 0; e < M::VE; ++e) v[u][e] = ok && k + e < C ? src[k + e] : (T)0.f;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = (c0 + u * TPT) * M::VE;
      if (k < KP) *reinterpret_cast<typename M::V*>(dst + k) = v[u];
    }
  }
}

// Mean and 1 / standard deviation of the C channels of a staged row (fp32, two passes), in every
// thread of the token.  Each thread reads only chunks that it staged itself.
template <typename T, int TPT>
__device__ __attribute__((always_inline)) inline void row_stats(const T* row, int part, int C, float eps, float& mean,
                                                                float& rstd) {
  using M = TileMma<T>;
  float s = 0.f;
  for (int c = part; c * M::VE < C; c += TPT) {
    const typename M::V v = *reinterpret_cast<const typename M::V*>(row + c * M::VE);
#pragma unroll
    for (int e = 0; e < M::VE; ++e) s += (float)v[e];
  }
  mean = token_sum<TPT>(s) / (float)C;
  float q = 0.f;
  for (int c = part; c * M::VE < C; c += TPT) {
    const typename M::V v = *reinterpret_cast<const typename M::V*>(row + c * M::VE);
#pragma unroll
    for (int e = 0; e < M::VE; ++e) {
      const float d = (float)v[e] - mean;
      q = c * M::VE + e < C ? fmaf(d, d, q) : q;
    }
  }
  rstd = rsqrtf(token_sum<TPT>(q) / (float)C + eps);
}

// row = (row - mean) * rstd (* w + b), rounded to T, in place (w, b: per-channel affine or null).
template <typename T, int TPT>
__device__ __attribute__((always_inline)) inline void normalise_row(T* row, int part, int C, float mean, float rstd,
                                                                    const T* __restrict__ w, const T* __restrict__ b) {
  using M = TileMma<T>;
  for (int c = part; c * M::VE < C; c += TPT) {
    typename M::V v = *reinterpret_cast<const typename M::V*>(row + c * M::VE);
#pragma unroll
    for (int e = 0; e < M::VE; ++e) {
      const int k = c * M::VE + e;
      if (k < C) {
        float n = ((float)v[e] - mean) * rstd;
        if (w) n = n * (float)w[k] + (b ? (float)b[k] : 0.f);
        v[e] = (T)n;
      }
    }
    *reinterpret_cast<typename M::V*>(row + c * M::VE) = v;
  }
}

// acc[i][n] += W_i rows x token rows over k < K: the lane's weight row w[i] (row tile_perm(lane % 32) or
// lane % 32 of a 32-feature chunk, already clamped to a row that exists) as one operand, rows
// 32 n + trow of the LDS tile as the other.  A_IS_W puts the weights in the A operand (D rows are
// features, columns tokens); otherwise the tokens.  Weights come straight from L2, PB k-steps ahead in
// two register sets used in turn: each wave of a block needs other rows, so a pass through LDS would
// only add barriers.  (fp32: 2 k-steps of 4 MFMAs each cover the latency; 4 cost registers, 2-6 % slower.)  VEC as
// in stage_row, for the weight rows; a k-step that ends past K and the ones
// left over from the batches are taken one at a time.
template <typename T, int NWT, int NT, bool A_IS_W, bool VEC, int PB>
__device__ __attribute__((always_inline)) inline void tile_gemm_n(f32x16 (&acc)[NWT][NT], const T* tile, int rs,
                                                                  int trow, const T* const (&w)[NWT], int K) {
  using M = TileMma<T>;
  using V = typename M::V;
  const int hk = (threadIdx.x >> 5 & 1) * M::VE, nk = (K + M::KS - 1) / M::KS;
  const int nb = VEC ? K / (M::KS * PB) : 0;
  const T* t0 = tile + trow * rs + hk;
  using Set = V[PB][NWT];
  auto load = [&](Set& r, int b) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < PB; ++j)
#pragma unroll
      for (int i = 0; i < NWT; ++i) r[j][i] = ldg<V>(w[i] + (b * PB + j) * M::KS + hk);
  };
  auto mul = [&](const V(&r)[NWT], int s) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      const V x = *reinterpret_cast<const V*>(t0 + 32 * n * rs + s * M::KS);
#pragma unroll
      for (int i = 0; i < NWT; ++i) acc[i][n] = A_IS_W ? M::mma(r[i], x, acc[i][n]) : M::mma(x, r[i], acc[i][n]);
    }
  };
  auto step = [&](const Set& r, int b) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < PB; ++j) mul(r[j], b * PB + j);
  };
  if (nb > 0) {
    Set wa, wb;
    load(wa, 0);
    int b = 0;
    for (; b + 2 < nb; b += 2) {
      load(wb, b + 1);
      step(wa, b);
      load(wa, b + 2);
      step(wb, b + 1);
    }
    if (b + 1 < nb) {
      load(wb, b + 1);
      step(wa, b);
      step(wb, b + 1);
    } else {
      step(wa, b);
    }
  }
  for (int s = nb * PB; s < nk; ++s) {
    const int k = s * M::KS + hk;
    V r[NWT];
#pragma unroll
    for (int i = 0; i < NWT; ++i) {
      if constexpr (VEC) {
        r[i] = ldg<V>(w[i] + (k < K ? k : 0));
        if (k >= K) r[i] = V{};
      } else {
#pragma unroll
        for (int e = 0; e < M::VE; ++e) r[i][e] = k + e < K ? w[i][k + e] : (T)0.f;
      }
    }
    mul(r, s);
  }
}
template <typename T, int NT, bool A_IS_W, bool VEC, int PB = sizeof(T) == 4 ? 2 : 4>
__device__ __attribute__((always_inline)) inline void tile_gemm(f32x16 (&acc)[1][NT], const T* tile, int rs, int trow,
                                                                const T* w, int K) {
  const T* const ws[1] = {w};
  tile_gemm_n<T, 1, NT, A_IS_W, VEC, PB>(acc, tile, rs, trow, ws, K);
}

// Writes f(v), v = 0..15, to dst[0..15], leaving out elements >= n; VEC: in 16-byte chunks (n a
// multiple of VE, dst 16-byte aligned).
template <typename T, bool VEC, typename F>
__device__ __attribute__((always_inline)) inline void store16(T* dst, int n, F f) {
  using M = TileMma<T>;
#pragma unroll
  for (int c = 0; c < 16; c += M::VE) {
    typename M::V r;
#pragma unroll
    for (int e = 0; e < M::VE; ++e) r[e] = f(c + e);
    if constexpr (VEC) {
      if (c < n) *reinterpret_cast<typename M::V*>(dst + c) = r;
    } else {
#pragma unroll
      for (int e = 0; e < M::VE; ++e)
        if (c + e < n) dst[c + e] = r[e];
    }
  }
}

// The 16 elements f(v) = p[fl + v] of a per-feature vector as floats (0 where p is null or the feature
// does not exist).
template <typename T, bool VEC>
__device__ __attribute__((always_inline)) inline f32x16 load16(const T* p, int n) {
  using M = TileMma<T>;
  f32x16 r = {};
  if (p) {
#pragma unroll
    for (int c = 0; c < 16; c += M::VE) {
      if constexpr (VEC) {
        const typename M::V v = ldg<typename M::V>(p + (c < n ? c : n - M::VE));
#pragma unroll
        for (int e = 0; e < M::VE; ++e) r[c + e] = (float)v[e];
      } else {
#pragma unroll
        for (int e = 0; e < M::VE; ++e) r[c + e] = c + e < n ? (float)p[c + e] : 0.f;
      }
    }
  }
  return r;
}

}  // namespace tops
