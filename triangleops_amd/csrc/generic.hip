// Any-shape kernels: the shapes the tuned kernels do not cover, and fp32 I/O (then every value stays
// fp32).  Products run on the matrix cores, 32x32x16 MFMAs in 16-bit types and 32x32x2 fp32 MFMAs
// in fp32 (tile_mma.hpp); with 16-bit I/O the rounding points follow the tuned path:
//   LN(x) is rounded to the I/O type before the Q / K / V and gate products, Q / K / V and the
//   gated activations are rounded to the I/O type, the pair bias and the attention weights stay fp32.
//
//   tri_generic_prep_kernel   LN(x), Q / K / V of all heads and the row-shared pair bias
//                             bias[h][a][b] = LN(x[a, b]) . Wz[h] + bz[h]
//   tri_generic_attn_kernel   32 queries of one (row i, head h) per wave: online softmax in fp32, scores
//                             q . k * scale + bias, masked keys get the reference's fp32 "+ (-1e9)"
//   gate_generic_kernel       y = (o * sigmoid(g . Wg^T + bg)) -> io, out = y . Wo^T + bo
//                             with g = LN(gin) or gin
//   apb_generic_qkv_kernel, apb_gen_bias_mma_kernel (C_z <= 256), apb_generic_bias_kernel (wider; fp32
//                             FMAs): attention_pair_bias's projections and pair bias
//   tmu_generic_in_kernel     triangle_multiplicative_update input phase at any C / C_out:
//                             ab[f] = (xn . Wp[f] + Bp[f]) * sigmoid(xn . Wg[f] + Bg[f]) * mask,
//                             xn = (x - mean) * rstd (the LN affine is folded into Wp / Wg)
//   tmu_generic_out_kernel    output phase: (yn . Wp + Bp) * sigmoid(xn . Wg + Bg), yn = LN_out(y)
//
// Reference: triangle_attn/module.py:57-125 and benchmarks/references.py:174-205 (the op),
// triangle_attn/kernel.py:230-238 (-1e9 pair mask), :282-290 (D = 16 keeps separate K / V
// weights), tests/test_triangle_attn.py:137-192 (the Apo shape).
#include <initializer_list>
#include <type_traits>

#include "capi.hpp"
#include "common.hpp"
#include "generic.hpp"
#include "tile_mma.hpp"

namespace tops {

constexpr int kGenTok = 16;  // tokens per block; 16 lanes per token for the LayerNorm sums

// Conditions of a kernel's 16-byte accesses (a null pointer is not accessed).
static bool aligned16(std::initializer_list<const void*> ps) {
  for (const void* p : ps)
    if ((uintptr_t)p % 16 != 0) return false;
  return true;
}
static bool multiples_of(int n, std::initializer_list<int64_t> vs) {
  for (int64_t v : vs)
    if (v % n != 0) return false;
  return true;
}

// LayerNorm of kGenTok token rows held in LDS (fp32, row length C, row stride ld): 16
// consecutive lanes per token, two-pass statistics.  Writes normalised rows back in place.
template <typename T>
__device__ void gen_layer_norm(float* rows, int ld, int C, const T* w_ln, const T* b_ln, float eps) {
  const int tid = threadIdx.x, t = tid >> 4, part = tid & 15;
  float* r = rows + t * ld;
  float s = 0.f;
  for (int c = part; c < C; c += 16) s += r[c];
  const float mean = group_sum<16>(s) / (float)C;
  float q = 0.f;
  for (int c = part; c < C; c += 16) q = fmaf(r[c] - mean, r[c] - mean, q);
  const float rstd = rsqrtf(group_sum<16>(q) / (float)C + eps);
  for (int c = part; c < C; c += 16) {
    const float w = w_ln ? (float)w_ln[c] : 1.f, b = b_ln ? (float)b_ln[c] : 0.f;
    r[c] = (r[c] - mean) * rstd * w + b;
  }
}

// Writes 16 consecutive rows f0 .. f0 + 15 (f(v), v < n) of the (H, 3, D) projection of one token to
// its q, k and v rows, in pieces of pw elements.
template <typename T, typename F>
__device__ __attribute__((always_inline)) inline void store_qkv16(T* qo, T* ko, T* vo, int64_t row, int f0, int n,
                                                                  int D, int pw, F f) {
  // the destination is picked by integer selects on address offsets (a pointer choice among the three
  // becomes a table in private memory)
  const uint64_t aq = (uint64_t)qo, dk = (uint64_t)ko - aq, dv = (uint64_t)vo - aq;
  auto dst = [&](int fr) __attribute__((always_inline)) {
    const int h = fr / (3 * D), r = fr - h * 3 * D, which = r / D;
    return reinterpret_cast<T*>(aq + (which == 1 ? dk : 0) + (which == 2 ? dv : 0)) + row + h * D + (r - which * D);
  };
  auto pieces = [&](auto tag) __attribute__((always_inline)) {
    constexpr int W = decltype(tag)::value;
#pragma unroll
    for (int c = 0; c < 16; c += W) {
      if (c >= n) continue;
      vec<T, W> r;
#pragma unroll
      for (int e = 0; e < W; ++e) r[e] = (T)f(c + e);
      *reinterpret_cast<vec<T, W>*>(dst(f0 + c)) = r;
    }
  };
  if (pw == TileMma<T>::VE)
    pieces(std::integral_constant<int, TileMma<T>::VE>{});
  else if (pw == 4)
    pieces(std::integral_constant<int, 4>{});
  else
    pieces(std::integral_constant<int, 1>{});
}

// The widest piece (VE, 4 or 1 elements) that divides D and that the three outputs are aligned to.
template <typename T>
static int qkv_piece(int D, const void* q, const void* k, const void* v) {
  for (int w : {TileMma<T>::VE, 4})
    if (D % w == 0 && ((uintptr_t)q | (uintptr_t)k | (uintptr_t)v) % (w * sizeof(T)) == 0) return w;
  return 1;
}

// ---------------------------------------------------------------------------------------------
// Pre-pass: 32 tokens per block of 4 waves.  LN(x) in LDS (rounded to the I/O type, also written out
// as xln), Q / K / V of all heads on the matrix cores (a wave takes 32-row chunks of the weight in
// turn), the row-shared pair bias from the unrounded LN(x) in fp32 FMAs by the threads that normalise
// the rows (H is small: an MFMA chunk of 32 features would be mostly empty).  Bound by the matrix
// cores and the weight reads; N = 200, C = 128, H = 4, D = 32: fp32 130 -> 57 us, bf16 193 -> 29 us
// against VALU block products; N = 320, C = 256, H = 8 in bf16 3815 -> 210 us.  64 tokens per block
// (each weight row read half as often) measured slower up to C = 128 (68 and 36 us) and 9 % faster
// at C = 256.
// ---------------------------------------------------------------------------------------------
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void tri_generic_prep_kernel(const T* __restrict__ x, int64_t sx0, int64_t sx1,
                                                              const T* __restrict__ w_ln, const T* __restrict__ b_ln,
                                                              int apply_ln, const T* __restrict__ wqkv,
                                                              const T* __restrict__ WZ, const float* __restrict__ BZ,
                                                              T* __restrict__ xln, T* __restrict__ qo,
                                                              T* __restrict__ ko, T* __restrict__ vo,
                                                              float* __restrict__ bias, int64_t N, int C, int H, int D,
                                                              int pw, float eps) {
  using M = TileMma<T>;
  using V = typename M::V;
  constexpr int TT = 32, TPT = 256 / TT;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int rx = tile_row<T>(C);
  T* xs = reinterpret_cast<T*>(smem);  // [TT][rx]  x, then LN(x)
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hl = lane >> 5, col = lane & 31, HD = H * D, F = 3 * HD;
  const int64_t ntok = N * N, tok0 = (int64_t)blockIdx.x * TT;
  {
    const int t = tid / TPT, part = tid % TPT;
    const bool ok = tok0 + t < ntok;
    const int64_t tok = ok ? tok0 + t : ntok - 1, i = tok / N;
    T* row = xs + t * rx;
    stage_row<T, TPT, VEC>(row, x + i * sx0 + (tok - i * N) * sx1, ok, part, C, tile_kp(C));
    float mean = 0.f, rstd = 1.f;
    if (apply_ln) row_stats<T, TPT>(row, part, C, eps, mean, rstd);
    // pair bias, 4 heads at a time
    for (int h0 = 0; h0 < H; h0 += 4) {
      float acc[4] = {};
      for (int k = part * M::VE; k < C; k += TPT * M::VE) {
        const V v = *reinterpret_cast<const V*>(row + k);
        V wz[4], w = {}, b = {};
        if constexpr (VEC) {
#pragma unroll
          for (int j = 0; j < 4; ++j) wz[j] = ldg<V>(WZ + (int64_t)(h0 + j < H ? h0 + j : H - 1) * C + k);
          if (apply_ln) {
            w = ldg<V>(w_ln + k);
            if (b_ln) b = ldg<V>(b_ln + k);
          }
        } else {
#pragma unroll
          for (int e = 0; e < M::VE; ++e) {
            const bool in = k + e < C;
#pragma unroll
            for (int j = 0; j < 4; ++j) wz[j][e] = in ? WZ[(int64_t)(h0 + j < H ? h0 + j : H - 1) * C + k + e] : (T)0.f;
            if (apply_ln) {
              w[e] = in ? w_ln[k + e] : (T)0.f;
              b[e] = in && b_ln ? b_ln[k + e] : (T)0.f;
            }
          }
        }
#pragma unroll
        for (int e = 0; e < M::VE; ++e) {
          float n = (float)v[e];
          if (apply_ln) n = (n - mean) * rstd * (float)w[e] + (float)b[e];
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[j] = fmaf(n, (float)wz[j][e], acc[j]);
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float s = token_sum<TPT>(acc[j]);
        if (part == j && ok && h0 + j < H) bias[(int64_t)(h0 + j) * ntok + tok] = s + (BZ ? BZ[h0 + j] : 0.f);
      }
    }
    if (apply_ln) normalise_row<T, TPT>(row, part, C, mean, rstd, w_ln, b_ln);
    if (ok) {
      T* dst = xln + tok * C;
      for (int k = part * M::VE; k < C; k += TPT * M::VE) {
        const V v = *reinterpret_cast<const V*>(row + k);
        if constexpr (VEC) {
          *reinterpret_cast<V*>(dst + k) = v;
        } else {
#pragma unroll
          for (int e = 0; e < M::VE; ++e)
            if (k + e < C) dst[k + e] = v[e];
        }
      }
    }
  }
  __syncthreads();
  for (int f0 = 32 * wave; f0 < F; f0 += 128) {
    const int row = f0 + tile_perm(col), fl = f0 + 16 * hl;
    f32x16 acc[1][1] = {};
    tile_gemm<T, 1, true, VEC>(acc, xs, rx, col, wqkv + (int64_t)(row < F ? row : F - 1) * C, C);
    if (tok0 + col < ntok)
      store_qkv16<T>(qo, ko, vo, (tok0 + col) * HD, fl, F - fl, D, pw,
                     [&](int v) __attribute__((always_inline)) { return acc[0][0][v]; });
  }
}

// ---------------------------------------------------------------------------------------------
// Attention over R rows of N queries and N keys, any H, D <= DP (16, 32 or 64).  A wave holds 32 queries of one
// (row i, head h) and walks the keys in chunks of 32: S^T = K . Q^T (a lane: one query, the 16 keys
// k0 + 16 hl + v), scores q . k * scale + bias with masked keys (mask[i*sm0 + k*sm1] == 0) getting
// "+ (-1e9)" in fp32 (triangle attention) or -inf (MASK_INF, attention_pair_bias: a row without valid
// keys gives NaN, as torch's softmax does) and keys >= N left out, online softmax in fp32, and
// O^T += V^T . P^T with the score registers as the operand.  fp32 I/O runs the fp32 MFMA throughout;
// with 16-bit I/O each fp32 weight enters as three 16-bit terms that hold all its 24 bits (weight_terms).  Why
// three: two hold 17 bits in bf16 and 22 down to 8 (small weights) in fp16, for 1-6 % and 3-25 % less time (bf16 /
// fp16, N = 500, 2 heads of 64: 239 / 241 against 253 / 275 us; 600 tokens x 16 heads of 24: 11.5 / 12.2 and 11.7 / 12.6);
// V and weights converted to the fp32 MFMA, as in fp32 I/O: 392 / 393 and 13.1 / 13.0.
// K, V and the bias rows come straight from L2 in operand order (K rows as 16-byte chunks, V an element
// per key and lane, which is the transpose): no LDS and no barrier in the loop.  With KSPL = 1 a block is one
// wave and one query tile, and the tiles of a (row, head) share its key reads through their XCD's L2; with
// KSPL = 4 a block's 4 waves take every 4th chunk of one query tile and merge (m, l, o) through LDS.  Bound by
// the fp32 MFMAs in fp32 (N = 200, 4 heads of 32: 246 -> 62 us against a query per lane on the VALU, half of the
// fp32 matrix rate), by the exponentials and the split of the weights in 16 bits (the same in bf16: 248 -> 37).
// ---------------------------------------------------------------------------------------------
// w[0 .. 15] as three terms of the I/O type that add up to all 24 bits: w = t[0] + (t[1] + t[2] / S) / S.  bf16 has
// fp32's range: S = 1 and the terms are the first, second and last 8 bits.  fp16 has not: S = 2^11, a term's
// width, keeps the rests clear of its denormals (with the largest weight at 2^15, the others are whole down to
// 2^-38 of it and off by less than 2^-61 of it below).
template <typename T>
constexpr int kTermScale = std::is_same<T, _Float16>::value ? 1 << 11 : 1;
template <typename T, typename V, int NV>
__device__ __attribute__((always_inline)) inline void weight_terms(const f32x16& w, V (&t)[3][NV]) {
  constexpr int VE = 16 / NV;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    float r = w[v];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      if constexpr (std::is_same<T, __bf16>::value) {
        const uint32_t top = __float_as_uint(r) & 0xffff0000u;
        t[k][v / VE][v % VE] = __builtin_bit_cast(T, (uint16_t)(top >> 16));
        r -= __uint_as_float(top);
      } else {
        t[k][v / VE][v % VE] = (T)r;
        r = (r - (float)t[k][v / VE][v % VE]) * kTermScale<T>;
      }
    }
  }
}

template <typename T, int DP, int KSPL, bool MASK_INF, bool VEC>
__global__ __launch_bounds__(KSPL == 1 ? 64 : 256, DP <= 32 ? 4 : 2) void tri_generic_attn_kernel(
    const T* __restrict__ qi_, const T* __restrict__ ki_, const T* __restrict__ vi_, const float* __restrict__ bias,
    const int8_t* __restrict__ mask, int64_t sm0, int64_t sm1, T* __restrict__ out, int64_t so0, int64_t so1, int N,
    int H, int D, float scale) {
  using M = TileMma<T>;
  using V = typename M::V;
  constexpr int ND = (DP + 31) / 32;               // 32-channel tiles of O
  constexpr int NQ = DP / M::KS, NV = 16 / M::VE;  // k-steps of q . k, 16-byte pieces of 16 keys
  constexpr float kShift = kTermScale<T> == 1 ? 0.f : 15.f;  // weights up to 2^15: fp16's range, used from the top
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hl = lane >> 5, col = lane & 31;
  // consecutive blocks go to the 8 XCDs in turn: XCD x takes the x-th eighth of the work, so the query
  // tiles of one (row, head) read its keys through one L2
  uint32_t w = blockIdx.x;
  if constexpr (KSPL == 1) {
    const uint32_t per = gridDim.x / 8, x = w % 8, rem = gridDim.x % 8;
    w = x * per + (x < rem ? x : rem) + w / 8;
  }
  const uint32_t nqb = (N + 31) / 32, ih = w / nqb, qb = w - ih * nqb;
  const int i = ih / (uint32_t)H, h = ih - i * H;
  const int q0 = qb * 32;
  // all reads go through buffers of the row's keys and of the tile's bias rows: a lane keeps 32-bit byte
  // offsets (64-bit addresses of every element would take the registers of two more waves per SIMD),
  // and keys past N read 0.  kOut is past any buffer's end.
  constexpr uint32_t ES = sizeof(T), kOut = 0x80000000u;
  const uint32_t HDB = H * D * ES;
  const int64_t base = (int64_t)i * N * H * D + h * D;
  const int q = q0 + col < N ? q0 + col : N - 1;
  const uint32_t rbytes = (uint32_t)N * HDB - (uint32_t)h * D * ES;
  const Rsrc qr = buffer_of(qi_ + base, rbytes), kr = buffer_of(ki_ + base, rbytes), vr = buffer_of(vi_ + base, rbytes);
  const int qrows = N - q0 < 32 ? N - q0 : 32;
  const Rsrc br = buffer_of(bias + ((int64_t)h * N + q0) * N, (uint32_t)qrows * N * 4);
  const int8_t* mrow = mask ? mask + i * sm0 : nullptr;
  auto load_row = [&](V(&r)[NQ], Rsrc src, uint32_t row) __attribute__((always_inline)) {  // zero past D
#pragma unroll
    for (int s = 0; s < NQ; ++s) {
      const int d = s * M::KS + hl * M::VE;
      if constexpr (VEC) {
        r[s] = buffer_load<V>(src, row + (d < D ? d * ES : kOut));
      } else {
#pragma unroll
        for (int e = 0; e < M::VE; ++e) r[s][e] = buffer_load<T>(src, row + (d + e < D ? (d + e) * ES : kOut));
      }
    }
  };
  V qf[NQ], kf[NQ];
  load_row(qf, qr, (uint32_t)q * HDB);
  uint32_t vd[ND];  // this lane's V element of a key: channel tile_perm(col) of each 32, so o holds 16 hl + v
#pragma unroll
  for (int n = 0; n < ND; ++n) {
    const int d = 32 * n + tile_perm(col);
    vd[n] = 16 * hl * HDB + (d < D ? d : D - 1) * ES;  // channels past D are computed and not stored
  }
  const uint32_t bd = (uint32_t)(q - q0) * N * 4 + 64 * hl, kd = tile_perm(col) * HDB;
  f32x16 o[ND] = {};
  float m = -INFINITY, l = 0.f;
  const int nch = (N + 31) / 32, c0 = KSPL == 1 ? 0 : wave;
  int c = c0;
  if (c < nch) load_row(kf, kr, kd + 32 * c * HDB);
  for (; c < nch; c += KSPL) {
    const int k0 = 32 * c;
    // this chunk's V, bias and mask, used after the scores
    V vf[ND][NV];
    f32x16 b;
#pragma unroll
    for (int v = 0; v < 16; ++v)
#pragma unroll
      for (int n = 0; n < ND; ++n) vf[n][v / M::VE][v % M::VE] = buffer_load<T>(vr, vd[n] + (k0 + v) * HDB);
    if (k0 + 32 <= N) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 t = buffer_load<f32x4>(br, bd + k0 * 4 + 16 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) b[4 * g + e] = t[e];
      }
    } else {  // (past the end of a row: the next row or 0, replaced by -inf below)
#pragma unroll
      for (int v = 0; v < 16; ++v) b[v] = buffer_load<float>(br, bd + k0 * 4 + 4 * v);
    }
    const bool in = k0 + col < N;
    const bool on = in && (!mrow || mrow[(int64_t)(k0 + col) * sm1] != 0);
    const uint32_t inb = (uint32_t)__builtin_amdgcn_ballot_w64(in), onb = (uint32_t)__builtin_amdgcn_ballot_w64(on);
    f32x16 s = {};
#pragma unroll
    for (int j = 0; j < NQ; ++j) s = M::mma(kf[j], qf[j], s);
    if (c + KSPL < nch) load_row(kf, kr, kd + 32 * (c + KSPL) * HDB);
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] = fmaf(s[v], scale, b[v]);
    if (onb != 0xffffffffu) {  // some key is masked or past the end
      const uint32_t ib = inb >> (16 * hl), ob = onb >> (16 * hl);
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        s[v] = (ob >> v) & 1 ? s[v] : (MASK_INF ? -INFINITY : s[v] - 1e9f);
        s[v] = (ib >> v) & 1 ? s[v] : -INFINITY;
      }
    }
    float cm = s[0];
#pragma unroll
    for (int v = 1; v < 16; ++v) cm = fmaxf(cm, s[v]);
    const float mn = fmaxf(m, halves_max(cm));
    // while every key so far is left out, m = mn = -inf: shift by 0 instead, so those keys get
    // p = 0 and the state stays (m, l, o) = (-inf, 0, 0) instead of NaN
    const float sh = mn == -INFINITY ? 0.f : mn;
    const float corr = fast_exp2((m - sh) * kLog2e);
    m = mn;
    float lc = 0.f;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      s[v] = fast_exp2(fmaf(s[v] - sh, kLog2e, kShift));
      lc += s[v];
    }
    // the chunk's sums start at zero and are added to the running ones: a chain over all keys rounds
    // against the whole sum at every key (fp32, N = 291: 18 % more error than sums over a quarter each)
    l = fmaf(l, corr, lc);
    auto add = [&](int n, const f32x16& t) __attribute__((always_inline)) {
#pragma unroll
      for (int v = 0; v < 16; ++v) o[n][v] = fmaf(o[n][v], corr, t[v]);
    };
    if constexpr (sizeof(T) == 2) {
      V p[3][NV];
      weight_terms<T>(s, p);
#pragma unroll
      for (int n = 0; n < ND; ++n) {
        f32x16 t = {};
#pragma unroll
        for (int k = 2; k >= 0; --k) {  // the smallest terms first
#pragma unroll
          for (int j = 0; j < NV; ++j) t = M::mma(vf[n][j], p[k][j], t);
          if (k > 0 && kTermScale<T> != 1) t *= 1.f / kTermScale<T>;
        }
        add(n, t);
      }
    } else {
#pragma unroll
      for (int n = 0; n < ND; ++n) {
        f32x16 t = {};
#pragma unroll
        for (int v = 0; v < 16; ++v)
          t = __builtin_amdgcn_mfma_f32_32x32x2f32((float)vf[n][v / M::VE][v % M::VE], s[v], t, 0, 0, 0);
        add(n, t);
      }
    }
  }
  if constexpr (sizeof(T) == 2) {
    // an infinity of V times a weight's zero term is NaN where the weight itself gives an infinity: a tile with an
    // element that is not finite takes its products again in fp32, with the weights of the final maximum (some
    // twice the time for such a tile; 16 FMAs per 32 channels for the others)
    float z = 0.f;
#pragma unroll
    for (int n = 0; n < ND; ++n)
#pragma unroll
      for (int v = 0; v < 16; ++v) z = fmaf(o[n][v], 0.f, z);
    if (__builtin_amdgcn_ballot_w64(z != z) != 0) {
      const float sh = m == -INFINITY ? 0.f : m;
#pragma unroll
      for (int n = 0; n < ND; ++n) o[n] = f32x16{};
      for (c = c0; c < nch; c += KSPL) {
        const int k0 = 32 * c;
        load_row(kf, kr, kd + k0 * HDB);
        f32x16 s = {};
#pragma unroll
        for (int j = 0; j < NQ; ++j) s = M::mma(kf[j], qf[j], s);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int key = k0 + 16 * hl + v;
          s[v] = fmaf(s[v], scale, buffer_load<float>(br, bd + k0 * 4 + 4 * v));
          if (mrow && key < N && mrow[(int64_t)key * sm1] == 0) s[v] = MASK_INF ? -INFINITY : s[v] - 1e9f;
          s[v] = key < N ? fast_exp2(fmaf(s[v] - sh, kLog2e, kShift)) : 0.f;
#pragma unroll
          for (int n = 0; n < ND; ++n)
            o[n] = __builtin_amdgcn_mfma_f32_32x32x2f32((float)buffer_load<T>(vr, vd[n] + (k0 + v) * HDB), s[v], o[n],
                                                        0, 0, 0);
        }
      }
    }
  }
  l = halves_sum(l);
  if constexpr (KSPL == 1) {
    const float inv = 1.f / l;
    if (q0 + col >= N) return;
    T* dst = out + i * so0 + (int64_t)q * so1 + h * D;
#pragma unroll
    for (int n = 0; n < ND; ++n) {
      const int d = 32 * n + 16 * hl;
      store16<T, VEC>(dst + d, D - d, [&](int v) __attribute__((always_inline)) { return (T)(o[n][v] * inv); });
    }
  } else {
    // ---- merge the waves' partial states ----
    constexpr int OR = 32 * ND + 4;
    __shared__ __attribute__((aligned(16))) float ob[KSPL][32][OR];
    __shared__ float mls[KSPL][32][2];
#pragma unroll
    for (int n = 0; n < ND; ++n)
#pragma unroll
      for (int v = 0; v < 16; ++v) ob[wave][col][32 * n + 16 * hl + v] = o[n][v];
    mls[wave][col][0] = m;
    mls[wave][col][1] = l;
    __syncthreads();
    const int t = threadIdx.x >> 3, d0 = (threadIdx.x & 7) * 4 * ND;  // 8 threads per query, 4 ND channels each
    float mw[KSPL], mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < KSPL; ++w) {
      mw[w] = mls[w][t][0];
      mx = fmaxf(mx, mw[w]);
    }
    const float sh = mx == -INFINITY ? 0.f : mx;
    float sw[KSPL], lt = 0.f;
#pragma unroll
    for (int w = 0; w < KSPL; ++w) {
      sw[w] = fast_exp2((mw[w] - sh) * kLog2e);
      lt += sw[w] * mls[w][t][1];
    }
    const float inv = 1.f / lt;
    if (q0 + t < N) {
      T* dst = out + i * so0 + (q0 + t) * so1 + h * D;
#pragma unroll
      for (int d = 0; d < 4 * ND; ++d) {
        float acc = 0.f;
#pragma unroll
        for (int w = 0; w < KSPL; ++w) acc += sw[w] * ob[w][t][d0 + d];
        if (d0 + d < D) dst[d0 + d] = (T)(acc * inv);
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// x . W^T for few tokens: 32 tokens x 32 features per block, the k range split over its 4 waves, both
// operands straight from memory in operand order with PB k-steps in flight, partial sums added through
// LDS.  With few tokens a kernel whose blocks read whole weight matrices is bound by what one CU can
// read (600 tokens, C = HD = C_out = 384: gate and output projection in one launch bf16 20 us, fp32 45; as
// two launches of this 9 and 14): here a block reads 32 rows.
// A thread ends up with 4 consecutive features fl .. fl + 3 of token tok: epi(tok, fl, values, count).
// ---------------------------------------------------------------------------------------------
template <typename T, bool VEC, typename Epi>
__device__ __attribute__((always_inline)) inline void few_token_linear(const T* __restrict__ x, int64_t sx,
                                                                       const T* __restrict__ W, int M, int K, int F,
                                                                       Epi epi) {
  using TM = TileMma<T>;
  using V = typename TM::V;
  constexpr int PB = 4;
  __shared__ f32x4 part[4][4][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hl = lane >> 5, col = lane & 31;
  const int tok0 = blockIdx.x * 32, f0 = blockIdx.y * 32;
  const int tok = tok0 + col < M ? tok0 + col : M - 1, row = f0 + tile_perm(col);
  const T* xr = x + tok * sx + hl * TM::VE;
  const T* wr = W + (int64_t)(row < F ? row : F - 1) * K + hl * TM::VE;
  const int nk = (K + TM::KS - 1) / TM::KS, per = (nk + 3) / 4, s1 = per * (wave + 1) < nk ? per * (wave + 1) : nk;
  const int kl = K - hl * TM::VE;  // this lane's k-range
  auto load = [&](V& r, const T* p, int s) __attribute__((always_inline)) {
    const int k = s * TM::KS;
    if constexpr (VEC) {
      r = ldg<V>(p + (k < kl ? k : -hl * TM::VE));
      if (k >= kl) r = V{};
    } else {
#pragma unroll
      for (int e = 0; e < TM::VE; ++e) r[e] = k + e < kl ? p[k + e] : (T)0.f;
    }
  };
  f32x16 acc = {};
  for (int s0 = per * wave; s0 < s1; s0 += PB) {
    V a[PB], b[PB];
#pragma unroll
    for (int j = 0; j < PB; ++j) {  // (past the wave's part: the last k-step again, not used)
      const int s = s0 + j < s1 ? s0 + j : s1 - 1;
      load(a[j], wr, s);
      load(b[j], xr, s);
    }
#pragma unroll
    for (int j = 0; j < PB; ++j)
      if (s0 + j < s1) acc = TM::mma(a[j], b[j], acc);
  }
#pragma unroll
  for (int g = 0; g < 4; ++g) part[wave][g][lane] = f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
  __syncthreads();
  const f32x4 v = (part[0][wave][lane] + part[1][wave][lane]) + (part[2][wave][lane] + part[3][wave][lane]);
  const int fl = f0 + 16 * hl + 4 * wave;
  if (tok0 + col < M && fl < F) epi(tok, fl, v, F - fl < 4 ? F - fl : 4);
}

// Elements p[0 .. 3] as floats (p may be null: zeros; n: those that exist; VEC: n = 4, aligned).
template <typename T, bool VEC>
__device__ inline f32x4 load4(const T* p, int n) {
  f32x4 r = {};
  if (p) {
    if constexpr (VEC) {
      const vec<T, 4> v = ldg<vec<T, 4>>(p);
      r = f32x4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = e < n ? (float)p[e] : 0.f;
    }
  }
  return r;
}
template <typename T, bool VEC>
__device__ inline void store4(T* p, int n, vec<T, 4> v) {
  if constexpr (VEC) {
    *reinterpret_cast<vec<T, 4>*>(p) = v;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (e < n) p[e] = v[e];
  }
}

// y = io(o * sigmoid(gin . Wg^T + bg)), y (M, HD) contiguous.
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void gate_act_few_kernel(const T* __restrict__ o, int64_t so, const T* __restrict__ gin,
                                                          int64_t sg, const T* __restrict__ Wg, const T* __restrict__ bg,
                                                          T* __restrict__ y, int M, int Cin, int HD) {
  few_token_linear<T, VEC>(gin, sg, Wg, M, Cin, HD, [&](int tok, int f, f32x4 v, int n) __attribute__((always_inline)) {
    const f32x4 b = load4<T, VEC>(bg ? bg + f : nullptr, n), ov = load4<T, VEC>(o + tok * so + f, n);
    vec<T, 4> r;
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = (T)(ov[e] * sigmoid(v[e] + b[e]));
    store4<T, VEC>(y + (int64_t)tok * HD + f, n, r);
  });
}

// out = y . Wo^T + bo, with a residual rounded first as a separate add would see it.
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void gate_proj_few_kernel(const T* __restrict__ y, const T* __restrict__ Wo,
                                                           const T* __restrict__ bo, const T* __restrict__ res,
                                                           int64_t sr, T* __restrict__ out, int64_t sd, int M, int HD,
                                                           int Cout) {
  few_token_linear<T, VEC>(y, HD, Wo, M, HD, Cout, [&](int tok, int f, f32x4 v, int n) __attribute__((always_inline)) {
    const f32x4 b = load4<T, VEC>(bo ? bo + f : nullptr, n);
    vec<T, 4> r;
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = (T)(v[e] + b[e]);
    if (res) {
      const f32x4 rv = load4<T, VEC>(res + tok * sr + f, n);
#pragma unroll
      for (int e = 0; e < 4; ++e) r[e] = (T)(rv[e] + (float)r[e]);
    }
    store4<T, VEC>(out + tok * sd + f, n, r);
  });
}

// ---------------------------------------------------------------------------------------------
// Gate + output projection, any (C_in, HD, C_out): 32 tokens per block of NW waves.  Both input
// tiles are staged in LDS; each wave takes 32-feature chunks of the two products in turn (weights
// from L2 as the A operand, tokens as B), so a lane ends up with 16 consecutive features of one
// token: the gated activations overwrite the o tile in place and the output is stored in 16-byte
// pieces.  Few tokens are bound by the latency of the weight reads (600 tokens, C = HD = 384, bf16:
// 373 -> 20 us against a thread per output), many by the matrix cores in fp32 (262144 tokens, C = HD =
// 128: 206 us, 83 TFLOP/s) and by memory otherwise (the same in bf16: 771 -> 79 us).  32 tokens per
// block: 64 were 2 % faster at C = 128 and 15 % slower at C = 64 (fewer blocks per CU).
// ---------------------------------------------------------------------------------------------
template <typename T, int NW, bool VEC>
__global__ __launch_bounds__(64 * NW) void gate_generic_kernel(const T* __restrict__ o, int64_t so0, int64_t so1,
                                                              const T* __restrict__ gin, int64_t sg0, int64_t sg1,
                                                              const T* __restrict__ w_ln, const T* __restrict__ b_ln,
                                                              float eps, int apply_ln, const T* __restrict__ Wg,
                                                              const T* __restrict__ bg, const T* __restrict__ Wo,
                                                              const T* __restrict__ bo, const T* __restrict__ res,
                                                              int64_t sr0, int64_t sr1, T* __restrict__ out,
                                                              int64_t sd0, int64_t sd1, int64_t M1, int64_t M2,
                                                              int Cin, int HD, int Cout) {
  constexpr int TT = 32, TPT = 64 * NW / TT;
  constexpr int PB = sizeof(T) == 4 && NW == 16 ? 2 : 4;  // (fp32, 4 waves: 2 k-steps ahead 7 % slower)
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int rg = tile_row<T>(Cin), ry = tile_row<T>(HD);
  T* gs = reinterpret_cast<T*>(smem);  // [TT][rg] gate input (normalised)
  T* ys = gs + TT * rg;                // [TT][ry] o, then the gated activations
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hl = lane >> 5, col = lane & 31;
  const int64_t M = M1 * M2, tok0 = (int64_t)blockIdx.x * TT;
  {
    const int t = tid / TPT, part = tid % TPT;
    const bool ok = tok0 + t < M;
    const int64_t tok = ok ? tok0 + t : M - 1, m1 = tok / M2, m2 = tok - m1 * M2;
    stage_row<T, TPT, VEC>(gs + t * rg, gin + m1 * sg0 + m2 * sg1, ok, part, Cin, tile_kp(Cin));
    stage_row<T, TPT, VEC>(ys + t * ry, o + m1 * so0 + m2 * so1, ok, part, HD, tile_kp(HD));
    if (apply_ln) {
      float mean, rstd;
      row_stats<T, TPT>(gs + t * rg, part, Cin, eps, mean, rstd);
      normalise_row<T, TPT>(gs + t * rg, part, Cin, mean, rstd, w_ln, b_ln);
    }
  }
  __syncthreads();
  // gate: ys = io(o * sigmoid(g . Wg + bg)), each element rewritten by the lane that reads it
  for (int f0 = 32 * wave; f0 < HD; f0 += 32 * NW) {
    const int row = f0 + tile_perm(col), fl = f0 + 16 * hl;
    f32x16 acc[1][1] = {};
    tile_gemm<T, 1, true, VEC, PB>(acc, gs, rg, col, Wg + (int64_t)(row < HD ? row : HD - 1) * Cin, Cin);
    const f32x16 b = load16<T, VEC>(bg && fl < HD ? bg + fl : nullptr, HD - fl);
    T* y = ys + col * ry + fl;
    store16<T, true>(y, 16, [&](int v) __attribute__((always_inline)) {
      return (T)((float)y[v] * sigmoid(acc[0][0][v] + b[v]));
    });
  }
  __syncthreads();
  // output projection; with a residual, the result is rounded first as a separate add would see it
  const int64_t tok = tok0 + col < M ? tok0 + col : M - 1, m1 = tok / M2, m2 = tok - m1 * M2;
  for (int f0 = 32 * wave; f0 < Cout; f0 += 32 * NW) {
    const int row = f0 + tile_perm(col), fl = f0 + 16 * hl;
    f32x16 acc[1][1] = {};
    tile_gemm<T, 1, true, VEC, PB>(acc, ys, ry, col, Wo + (int64_t)(row < Cout ? row : Cout - 1) * HD, HD);
    if (tok0 + col >= M || fl >= Cout) continue;
    const f32x16 b = load16<T, VEC>(bo ? bo + fl : nullptr, Cout - fl);
    T* dst = out + m1 * sd0 + m2 * sd1 + fl;
    if (res) {
      const f32x16 r = load16<T, VEC>(res + m1 * sr0 + m2 * sr1 + fl, Cout - fl);
      store16<T, VEC>(dst, Cout - fl,
                      [&](int v) __attribute__((always_inline)) { return (T)(r[v] + (float)(T)(acc[0][0][v] + b[v])); });
    } else {
      store16<T, VEC>(dst, Cout - fl, [&](int v) __attribute__((always_inline)) { return (T)(acc[0][0][v] + b[v]); });
    }
  }
}

template <typename T>
static int tri_generic_prep_t(const void* x, int64_t sx0, int64_t sx1, const void* w_ln, const void* b_ln,
                              int apply_ln, const void* wqkv, const void* WZ, const float* BZ, void* xln, void* q,
                              void* k, void* v, float* bias, int64_t N, int C, int H, int D, float eps,
                              hipStream_t st) {
  if (N == 0) return TOPS_OK;
  const bool vec = aligned16({x, w_ln, b_ln, wqkv, WZ, xln}) && multiples_of(TileMma<T>::VE, {sx0, sx1, C});
  const int pw = qkv_piece<T>(D, q, k, v);
  const size_t lds = (size_t)32 * tile_row<T>(C) * sizeof(T);
#define TOPS_GEN_PREP(VEC)                                                                                          \
  do {                                                                                                              \
    (void)hipFuncSetAttribute((const void*)tri_generic_prep_kernel<T, VEC>,                                         \
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);                                \
    hipLaunchKernelGGL((tri_generic_prep_kernel<T, VEC>), dim3((unsigned)((N * N + 31) / 32)), dim3(256), lds, st,   \
                       (const T*)x, sx0, sx1, (const T*)w_ln, (const T*)b_ln, apply_ln, (const T*)wqkv, (const T*)WZ, \
                       BZ, (T*)xln, (T*)q, (T*)k, (T*)v, bias, N, C, H, D, pw, eps);                                 \
  } while (0)
  if (vec)
    TOPS_GEN_PREP(true);
  else
    TOPS_GEN_PREP(false);
#undef TOPS_GEN_PREP
  return launched("tops_tri_generic_prep");
}

// Attention of R rows (q, k, v: (R, N, H, D) contiguous; mask rows sm0 apart, out rows so0 apart).
template <typename T, bool MASK_INF>
static int generic_attention_t(const char* name, const void* q, const void* k, const void* v, const float* bias,
                               const void* mask, int64_t sm0, int64_t sm1, void* out, int64_t so0, int64_t so1,
                               int64_t R, int64_t N, int H, int D, float scale, hipStream_t st) {
  if (R * N == 0) return TOPS_OK;
  const int64_t rh = R * H;
  // Keys split over a block's 4 waves while groups of 4 query tiles are fewer than the CUs: about where the
  // tiles alone would give every SIMD one wave.  us with the split / without, D = 24, at so many tiles: 304 (600
  // tokens x 16 heads) bf16 12 / 20, fp32 19 / 32; 752 (1500 x 16) 41 / 58, 54 / 91; 960 (1900 x 16) 63 / 73, 84 /
  // 115; 576 (N = 96 x 2 heads) 5.4 / 5.6, 7.8 / 7.3.  Past the line: 1152 (N = 96 x 4) 9.4 / 6.9, 14 / 11; 2048
  // (N = 128 x 4) 14 / 10, 23 / 16.  One long row still gains there up to 1264 tiles in bf16 (2500 x 16: 145 /
  // 153; 3000 x 16: 217 / 207) and 1504 in fp32 (237 / 263): the line lies where pair rows need it.
  const bool split = rh * ((N + 127) / 128) < num_cus();
  const int64_t blocks = rh * ((N + 31) / 32);
  TOPS_REQUIRE(blocks < (1LL << 31), "%s: too many query blocks", name);
  const bool vec = aligned16({q, k, v, out}) && multiples_of(TileMma<T>::VE, {D, so0, so1});
#define TOPS_GEN_ATTN(DP, KS, VEC)                                                                                  \
  hipLaunchKernelGGL((tri_generic_attn_kernel<T, DP, KS, MASK_INF, VEC>), dim3((unsigned)blocks),                   \
                     dim3(KS == 1 ? 64 : 256)        , 0, st,                                                       \
                     (const T*)q, (const T*)k, (const T*)v, bias, (const int8_t*)mask, sm0, sm1, (T*)out, so0, so1,  \
                     (int)N, H, D, scale)
#define TOPS_GEN_ATTN_V(DP, KS) \
  do {                          \
    if (vec)                    \
      TOPS_GEN_ATTN(DP, KS, true);  \
    else                        \
      TOPS_GEN_ATTN(DP, KS, false); \
  } while (0)
  if (split && D <= 16)
    TOPS_GEN_ATTN_V(16, 4);
  else if (split && D <= 32)
    TOPS_GEN_ATTN_V(32, 4);
  else if (split)
    TOPS_GEN_ATTN_V(64, 4);
  else if (D <= 16)
    TOPS_GEN_ATTN_V(16, 1);
  else if (D <= 32)
    TOPS_GEN_ATTN_V(32, 1);
  else
    TOPS_GEN_ATTN_V(64, 1);
#undef TOPS_GEN_ATTN_V
#undef TOPS_GEN_ATTN
  return launched(name);
}

template <typename T>
static int gate_generic_t(const void* o, int64_t so0, int64_t so1, const void* gin, int64_t sg0, int64_t sg1,
                          const void* w_ln, const void* b_ln, float eps, int apply_ln, const void* Wg, const void* bg,
                          const void* Wo, const void* bo, const void* res, int64_t sr0, int64_t sr1, void* out,
                          int64_t sd0, int64_t sd1, int64_t M1, int64_t M2, int Cin, int HD, int Cout,
                          hipStream_t st) {
  const int64_t M = M1 * M2;
  if (M == 0) return TOPS_OK;
  using V = TileMma<T>;
  const bool vec = aligned16({gin, o, Wg, bg, Wo, bo, res, out}) &&
                   multiples_of(V::VE, {sg0, sg1, so0, so1, sr0, sr1, sd0, sd1, Cin, HD, Cout});
  const size_t lds = (size_t)32 * (tile_row<T>(Cin) + tile_row<T>(HD)) * sizeof(T);
#define TOPS_GEN_GATE(NW, VEC)                                                                                      \
  do {                                                                                                              \
    const void* fn = (const void*)gate_generic_kernel<T, NW, VEC>;                                                  \
    (void)hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);                            \
    hipLaunchKernelGGL((gate_generic_kernel<T, NW, VEC>), dim3((unsigned)((M + 31) / 32)), dim3(64 * NW), lds, st,  \
                       (const T*)o, so0, so1, (const T*)gin, sg0, sg1, (const T*)w_ln, (const T*)b_ln, eps,         \
                       apply_ln, (const T*)Wg, (const T*)bg, (const T*)Wo, (const T*)bo, (const T*)res, sr0, sr1,    \
                       (T*)out, sd0, sd1, M1, M2, Cin, HD, Cout);                                                   \
  } while (0)
  // 16 waves per block while every block has a CU to itself (bf16 / fp32, 6000 tokens x 384: 21 / 49 us
  // against 23 / 57 with 4; 8000 x 128: equal), 4 beyond (16000 x 128: 10 / 16 against 11 / 19)
  if ((M + 31) / 32 <= num_cus()) {
    if (vec)
      TOPS_GEN_GATE(16, true);
    else
      TOPS_GEN_GATE(16, false);
  } else {
    if (vec)
      TOPS_GEN_GATE(4, true);
    else
      TOPS_GEN_GATE(4, false);
  }
#undef TOPS_GEN_GATE
  return launched(res ? "tops_gate_out_generic_residual" : "tops_gate_out_generic");
}

// True where gate and output projection run as two launches of few_token_linear: tokens in one column, no
// LayerNorm, and weights that one CU would read for longer than a launch takes (bf16 / fp32, 384 / 384 /
// 384, 600 tokens: 20 / 45 us in one launch, 9 / 14 in two; 2048: 20 / 45 and 16 / 24; 6000: 21 / 47 and
// 42 / 62; 128 / 128 / 128, 2000 tokens in bf16: 6.2 and 6.8).
static bool gate_few(int64_t M1, int64_t M2, int64_t Cin, int64_t HD, int64_t Cout, int apply_ln, size_t es) {
  return M2 == 1 && !apply_ln && (M1 + 31) / 32 <= num_cus() / 4 && (int64_t)es * HD * (Cin + Cout) >= 128 * 1024;
}

template <typename T>
static int gate_few_t(const void* o, int64_t so, const void* gin, int64_t sg, const void* Wg, const void* bg,
                      const void* Wo, const void* bo, const void* res, int64_t sr, void* out, int64_t sd, void* y,
                      int M, int Cin, int HD, int Cout, hipStream_t st) {
  constexpr int VE = TileMma<T>::VE;
  const unsigned mt = (unsigned)((M + 31) / 32);
  const dim3 g1(mt, (unsigned)((HD + 31) / 32)), g2(mt, (unsigned)((Cout + 31) / 32));
  if (aligned16({o, gin, Wg, bg, y}) && multiples_of(VE, {so, sg, Cin, HD}))
    hipLaunchKernelGGL((gate_act_few_kernel<T, true>), g1, dim3(256), 0, st, (const T*)o, so, (const T*)gin, sg,
                       (const T*)Wg, (const T*)bg, (T*)y, M, Cin, HD);
  else
    hipLaunchKernelGGL((gate_act_few_kernel<T, false>), g1, dim3(256), 0, st, (const T*)o, so, (const T*)gin, sg,
                       (const T*)Wg, (const T*)bg, (T*)y, M, Cin, HD);
  if (aligned16({y, Wo, bo, res, out}) && multiples_of(VE, {HD, Cout, sr, sd}))
    hipLaunchKernelGGL((gate_proj_few_kernel<T, true>), g2, dim3(256), 0, st, (const T*)y, (const T*)Wo, (const T*)bo,
                       (const T*)res, sr, (T*)out, sd, M, HD, Cout);
  else
    hipLaunchKernelGGL((gate_proj_few_kernel<T, false>), g2, dim3(256), 0, st, (const T*)y, (const T*)Wo, (const T*)bo,
                       (const T*)res, sr, (T*)out, sd, M, HD, Cout);
  return launched("tops_gate_out_generic_work");
}

// ---------------------------------------------------------------------------------------------
// attention_pair_bias, any (C_s, C_z, H, D) (attn_pair_bias/kernel.py:205-257):
//   apb_generic_qkv_kernel   per token m: q / k / v [m][h][d] = X[m] . W (rounded to the I/O type)
//   apb_generic_bias_kernel  per pair (q, k): bias[h][q][k] = zn . Wc[h] + Bc[h], zn = (z - mean) * rstd
//                            of z = Z[q, k, :] (the LN affine is folded into Wc / Bc)
// ---------------------------------------------------------------------------------------------
// 32 tokens and 128 weight rows per block, one 32-row chunk per wave; X rows go through LDS kQkvC
// channels at a time.  Few tokens: bound by latency (600 tokens, C = 384, 16 heads of 24 in bf16: 1031
// -> 8 us against a thread per output).
constexpr int kQkvC = 512;
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void apb_generic_qkv_kernel(const T* __restrict__ X, const T* __restrict__ wqkv,
                                                             T* __restrict__ qo, T* __restrict__ ko,
                                                             T* __restrict__ vo, int64_t M, int C, int H, int D,
                                                             int pw) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  T* xs = reinterpret_cast<T*>(smem);  // [32][tile_row(min(C, kQkvC))]
  const int rx = tile_row<T>(C < kQkvC ? C : kQkvC), HD = H * D, F = 3 * HD;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hl = lane >> 5, col = lane & 31;
  const int64_t tok0 = (int64_t)blockIdx.x * 32;
  const int f0 = 128 * blockIdx.y + 32 * wave, row = f0 + tile_perm(col), fl = f0 + 16 * hl;
  const T* w = wqkv + (int64_t)(row < F ? row : F - 1) * C;
  const int t = tid >> 3, part = tid & 7;
  const bool ok = tok0 + t < M;
  const T* src = X + (ok ? tok0 + t : M - 1) * C;
  f32x16 acc[1][1] = {};
  for (int c0 = 0; c0 < C; c0 += kQkvC) {
    const int kc = C - c0 < kQkvC ? C - c0 : kQkvC;
    if (c0 > 0) __syncthreads();
    stage_row<T, 8, VEC>(xs + t * rx, src + c0, ok, part, kc, tile_kp(kc));
    __syncthreads();
    if (f0 < F) tile_gemm<T, 1, true, VEC, 8>(acc, xs, rx, col, w + c0, kc);
  }
  if (tok0 + col < M && f0 < F)
    store_qkv16<T>(qo, ko, vo, (tok0 + col) * HD, fl, F - fl, D, pw,
                   [&](int v) __attribute__((always_inline)) { return acc[0][0][v]; });
}

// The same for few tokens (pw < 4: element-wise stores).
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void apb_qkv_few_kernel(const T* __restrict__ X, const T* __restrict__ wqkv,
                                                         T* __restrict__ qo, T* __restrict__ ko, T* __restrict__ vo,
                                                         int M, int C, int H, int D, int pw) {
  few_token_linear<T, VEC>(X, C, wqkv, M, C, 3 * H * D, [&](int tok, int f, f32x4 v, int n) __attribute__((always_inline)) {
    const int64_t row = (int64_t)tok * H * D;
    auto dst = [&](int fr) __attribute__((always_inline)) {
      const int h = fr / (3 * D), r = fr - h * 3 * D, which = r / D;
      const uint64_t aq = (uint64_t)qo, dk = (uint64_t)ko - aq, dv = (uint64_t)vo - aq;
      return reinterpret_cast<T*>(aq + (which == 1 ? dk : 0) + (which == 2 ? dv : 0)) + row + h * D + (r - which * D);
    };
    if (pw >= 4) {
      store4<T, true>(dst(f), 4, vec<T, 4>{(T)v[0], (T)v[1], (T)v[2], (T)v[3]});
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (e < n) *dst(f + e) = (T)v[e];
    }
  });
}

template <typename T>
__global__ __launch_bounds__(256) void apb_generic_bias_kernel(const T* __restrict__ Z, int64_t sz0, int64_t sz1,
                                                              const float* __restrict__ Wc,
                                                              const float* __restrict__ Bc, float* __restrict__ bias,
                                                              int64_t M, int Cz, int H, float eps) {
  extern __shared__ float zs[];  // [kGenTok][Cz]
  const int tid = threadIdx.x;
  const int64_t npair = M * M, p0 = (int64_t)blockIdx.x * kGenTok;
  for (int e = tid; e < kGenTok * Cz; e += 256) {
    const int64_t pr = p0 + e / Cz;
    zs[e] = pr < npair ? (float)Z[(pr / M) * sz0 + (pr % M) * sz1 + e % Cz] : 0.f;
  }
  __syncthreads();
  gen_layer_norm<T>(zs, Cz, Cz, nullptr, nullptr, eps);
  __syncthreads();
  for (int e = tid; e < kGenTok * H; e += 256) {
    const int t = e / H, h = e % H;
    const int64_t pr = p0 + t;
    if (pr >= npair) continue;
    const float* z = zs + t * Cz;
    const float* w = Wc + (int64_t)h * Cz;
    float acc = Bc[h];
    for (int c = 0; c < Cz; ++c) acc = fmaf(z[c], w[c], acc);
    bias[(int64_t)h * npair + pr] = acc;
  }
}

// C_z <= 4 VE NKC: 16 pairs and 16 heads (blockIdx.y) per wave and step.  Lane quarter qd holds the
// 16-byte chunks 4 j + qd of pair lane % 16, takes the two-pass LayerNorm in registers and feeds the
// normalised fp32 values to v_mfma_f32_16x16x4_f32 against the fp32 folded weights, which stay in
// registers over all steps.  The next step's loads are issued before this step's arithmetic.  Bound by
// the read of Z and the matrix cores together (600 tokens, 16 heads, C_z = 128, bf16: 148 -> 40 us
// against LDS tiles and FMAs, 3 TB/s).
template <typename T, int NKC, bool VEC>
__global__ __launch_bounds__(256, NKC <= 4 ? 4 : 1) void apb_gen_bias_mma_kernel(const T* __restrict__ Z, int64_t sz0, int64_t sz1,
                                                              const float* __restrict__ Wc,
                                                              const float* __restrict__ Bc, float* __restrict__ bias,
                                                              uint32_t M, int Cz, int H, float eps) {
  using TM = TileMma<T>;
  using V = typename TM::V;
  constexpr int VE = TM::VE;
  const int lane = threadIdx.x & 63, qd = lane >> 4, col = lane & 15;
  const int h0 = 16 * blockIdx.y, hr = h0 + col < H ? h0 + col : H - 1;
  const uint32_t npair = M * M, nstep = (npair + 15) / 16;
  const uint32_t nw = gridDim.x * 4, w0 = blockIdx.x * 4 + (threadIdx.x >> 6);
  float wr[NKC][VE], bc[4];
#pragma unroll
  for (int j = 0; j < NKC; ++j)
#pragma unroll
    for (int e = 0; e < VE; ++e) {
      const int k = (4 * j + qd) * VE + e;
      wr[j][e] = k < Cz ? Wc[(int64_t)hr * Cz + k] : 0.f;
    }
#pragma unroll
  for (int v = 0; v < 4; ++v) bc[v] = h0 + 4 * qd + v < H ? Bc[h0 + 4 * qd + v] : 0.f;
  auto load = [&](V(&z)[NKC], uint32_t step) __attribute__((always_inline)) {
    uint32_t p = step * 16 + col;
    p = p < npair ? p : npair - 1;
    const uint32_t a = p / M, b = p - a * M;
    const T* src = Z + a * sz0 + b * sz1;
#pragma unroll
    for (int j = 0; j < NKC; ++j) {
      const int k = (4 * j + qd) * VE;
      if constexpr (VEC) {
        z[j] = ldg<V>(src + (k < Cz ? k : 0));
        if (k >= Cz) z[j] = V{};
      } else {
#pragma unroll
        for (int e = 0; e < VE; ++e) z[j][e] = k + e < Cz ? src[k + e] : (T)0.f;
      }
    }
  };
  auto quarters = [&](float v) __attribute__((always_inline)) {  // sum over the pair's four lanes
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return halves_sum(__uint_as_float(r[0]) + __uint_as_float(r[1]));
  };
  auto compute = [&](const V(&z)[NKC], uint32_t step) __attribute__((always_inline)) {
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < NKC; ++j)
#pragma unroll
      for (int e = 0; e < VE; ++e) s += (float)z[j][e];
    const float mean = quarters(s) / (float)Cz;
    float q = 0.f, d[NKC][VE];
#pragma unroll
    for (int j = 0; j < NKC; ++j)
#pragma unroll
      for (int e = 0; e < VE; ++e) {
        d[j][e] = (4 * j + qd) * VE + e < Cz ? (float)z[j][e] - mean : 0.f;
        q = fmaf(d[j][e], d[j][e], q);
      }
    const float rstd = rsqrtf(quarters(q) / (float)Cz + eps);
    f32x4 acc = {};
#pragma unroll
    for (int j = 0; j < NKC; ++j)
#pragma unroll
      for (int e = 0; e < VE; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wr[j][e], d[j][e] * rstd, acc, 0, 0, 0);
    const uint32_t p = step * 16 + col;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int h = h0 + 4 * qd + v;
      if (p < npair && h < H) bias[(int64_t)h * npair + p] = acc[v] + bc[v];
    }
  };
  V za[NKC], zb[NKC];
  uint32_t t = w0;
  if (t < nstep) load(za, t);
  for (; t < nstep; t += 2 * nw) {
    if (t + nw < nstep) load(zb, t + nw);
    compute(za, t);
    if (t + nw >= nstep) break;
    if (t + 2 * nw < nstep) load(za, t + 2 * nw);
    compute(zb, t + nw);
  }
}

template <typename T>
static int apb_generic_prep_t(const void* X, const void* wqkv, const void* Z, int64_t sz0, int64_t sz1,
                              const float* Wc, const float* Bc, void* q, void* k, void* v, float* bias, int64_t M,
                              int C, int Cz, int H, int D, float eps, hipStream_t st) {
  if (M == 0) return TOPS_OK;
  const int pw = qkv_piece<T>(D, q, k, v);
  // few tokens: the other kernel's blocks (128 weight rows each) would reach less than half of the CUs (with
  // the bias, 128 tokens, C = 384, 16 heads of 24: bf16 19.3 us, fp32 18.2; 18.8 and 13.1 so; at 600 tokens,
  // 171 blocks, bf16 46.0 and 48.2)
  if ((M + 31) / 32 * ((3 * H * D + 127) / 128) < num_cus() / 2) {
    const dim3 grid((unsigned)((M + 31) / 32), (unsigned)((3 * H * D + 31) / 32));
    if (aligned16({X, wqkv}) && C % TileMma<T>::VE == 0)
      hipLaunchKernelGGL((apb_qkv_few_kernel<T, true>), grid, dim3(256), 0, st, (const T*)X, (const T*)wqkv, (T*)q,
                         (T*)k, (T*)v, (int)M, C, H, D, pw);
    else
      hipLaunchKernelGGL((apb_qkv_few_kernel<T, false>), grid, dim3(256), 0, st, (const T*)X, (const T*)wqkv, (T*)q,
                         (T*)k, (T*)v, (int)M, C, H, D, pw);
  } else {
    const bool vec = aligned16({X, wqkv}) && C % TileMma<T>::VE == 0;
    const size_t lds = (size_t)32 * tile_row<T>(C < kQkvC ? C : kQkvC) * sizeof(T);
    const dim3 grid((unsigned)((M + 31) / 32), (unsigned)((3 * H * D + 127) / 128));
    if (vec) {
      (void)hipFuncSetAttribute((const void*)apb_generic_qkv_kernel<T, true>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      hipLaunchKernelGGL((apb_generic_qkv_kernel<T, true>), grid, dim3(256), lds, st, (const T*)X, (const T*)wqkv,
                         (T*)q, (T*)k, (T*)v, M, C, H, D, pw);
    } else {
      (void)hipFuncSetAttribute((const void*)apb_generic_qkv_kernel<T, false>,
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      hipLaunchKernelGGL((apb_generic_qkv_kernel<T, false>), grid, dim3(256), lds, st, (const T*)X, (const T*)wqkv,
                         (T*)q, (T*)k, (T*)v, M, C, H, D, pw);
    }
  }
  if (Cz <= 256 && M < 65536) {
    const bool vec = aligned16({Z}) && multiples_of(TileMma<T>::VE, {sz0, sz1, Cz});
    const int64_t steps = (M * M + 63) / 64;  // of 4 waves
    // blocks that a CU holds at once: 4 in 128 registers (up to 4 chunks), 2 with more chunks (fp32, 600 tokens x
    // 16 heads, C_z = 128: 50 us, 55 with 4 blocks and 65 with 8, whose waves take uneven step counts)
    constexpr int W = 4 * TileMma<T>::VE;  // channels per chunk of the four lanes
    const int64_t cap = (Cz <= 4 * W ? 4 : 2) * num_cus();
    const dim3 grid((unsigned)(steps < cap ? steps : cap), (unsigned)((H + 15) / 16));
#define TOPS_GEN_BIAS(NKC, VEC)                                                                                     \
  hipLaunchKernelGGL((apb_gen_bias_mma_kernel<T, NKC, VEC>), grid, dim3(256), 0, st, (const T*)Z, sz0, sz1, Wc, Bc, \
                     bias, (uint32_t)M, Cz, H, eps)
#define TOPS_GEN_BIAS_V(NKC)    \
  do {                          \
    if (vec)                    \
      TOPS_GEN_BIAS(NKC, true); \
    else                        \
      TOPS_GEN_BIAS(NKC, false);\
  } while (0)
    if (Cz <= W)
      TOPS_GEN_BIAS_V(1);
    else if (Cz <= 2 * W)
      TOPS_GEN_BIAS_V(2);
    else if (Cz <= 4 * W)
      TOPS_GEN_BIAS_V(4);
    else if (Cz <= 8 * W)
      TOPS_GEN_BIAS_V(8);
    else if constexpr (sizeof(T) == 4)
      TOPS_GEN_BIAS_V(16);
#undef TOPS_GEN_BIAS_V
#undef TOPS_GEN_BIAS
  } else {
    const int64_t b2 = (M * M + kGenTok - 1) / kGenTok;
    hipLaunchKernelGGL((apb_generic_bias_kernel<T>), dim3((unsigned)b2), dim3(256),
                       (size_t)kGenTok * Cz * sizeof(float), st, (const T*)Z, sz0, sz1, Wc, Bc, bias, M, Cz, H, eps);
  }
  return launched("tops_apb_generic_prep");
}

// ---------------------------------------------------------------------------------------------
// triangle_multiplicative_update, any C (triangle_mul/module.py:8-12: x is (B, L, L, D), any D;
// triangle_mul/kernel.py:235-326).  Both phases take 32 NB tokens per block of 4 waves, normalised in LDS
// (rounded to the I/O type as the products' operand); a wave takes units of one 32-feature chunk of
// the weights and 32 NU tokens in turn.
//   input phase:  the tile is part of one row r of the (B, L, ld) store grid (tokens (r, c) or,
//                 transposed, (c, r), c = c0 ..; c >= L stores zeros).  Tokens are the A operand, so a
//                 lane holds 16 consecutive tokens of one feature of P and of G; the gated values go
//                 through a per-wave LDS tile, so each store instruction writes whole 64 NB-byte (fp32:
//                 128 NB) pieces of the features' rows.
//   output phase: tokens (b, i, j0 ..); y, channel-major, is transposed on its way into LDS.  Weights are
//                 the A operand, so a lane holds 16 consecutive features of one token.
// Bound by the fp32 MFMAs in fp32 (L = 256, C = 128: input / output phase 174 / 181 -> 90 / 61 us against
// VALU block products, 95 and 71 TFLOP/s) and by memory and the weight reads in 16-bit types (bf16 L = 512,
// C = 64: 174 / 320 -> 40 / 41 us, 2.5 TB/s).  Three waves per SIMD: left to itself the compiler takes the
// registers of one more (46 / 45 us), four spill (63 / 38).
// ---------------------------------------------------------------------------------------------
template <typename T, int NB, int NU, bool VEC>
__global__ __launch_bounds__(256, 3) void tmu_generic_in_kernel(const T* __restrict__ x, const int8_t* __restrict__ mask,
                                                            const T* __restrict__ Wp, const T* __restrict__ Wg,
                                                            const float* __restrict__ Bp, const float* __restrict__ Bg,
                                                            T* __restrict__ ab, uint32_t L, int C, int Cout, uint32_t ld,
                                                            int64_t fstride, int transpose, float eps) {
  using M = TileMma<T>;
  using V = typename M::V;
  constexpr int TT = 32 * NB, TPT = 256 / TT, UT = 32 * NU, OR = UT + M::VE;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int rx = tile_row<T>(C);
  T* xs = reinterpret_cast<T*>(smem);          // [TT][rx] normalised tokens
  T* ost = xs + TT * rx;                       // [4 waves][32][OR] output features x tokens
  float* msk = reinterpret_cast<float*>(ost + 4 * 32 * OR);  // [TT] 1 for a valid, unmasked token
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hl = lane >> 5, col = lane & 31;
  const uint32_t tpr = ld / TT, rr = blockIdx.x / tpr, c0 = (blockIdx.x - rr * tpr) * TT, bb = rr / L, r = rr - bb * L;
  {
    const int t = tid / TPT, part = tid % TPT;
    const uint32_t c = c0 + t < L ? c0 + t : L - 1;
    const int64_t tok = transpose ? ((int64_t)bb * L + c) * L + r : ((int64_t)bb * L + r) * L + c;
    T* row = xs + t * rx;
    // past L: a row of zeros, normalised by 0 (the values of token L - 1 may not be finite)
    stage_row<T, TPT, VEC>(row, x + tok * C, c0 + t < L, part, C, tile_kp(C));
    float mean, rstd;
    row_stats<T, TPT>(row, part, C, eps, mean, rstd);
    if (c0 + t >= L) rstd = 0.f;
    normalise_row<T, TPT>(row, part, C, mean, rstd, nullptr, nullptr);
    if (part == 0) msk[t] = c0 + t < L && (!mask || mask[tok] != 0) ? 1.f : 0.f;
  }
  __syncthreads();
  T* o = ost + wave * 32 * OR;
  T* abt = ab + ((int64_t)bb * L + r) * ld + c0;
  const int nunits = (Cout + 31) / 32 * (NB / NU);
  for (int u = wave; u < nunits; u += 4) {
    const int f0 = 32 * (u / (NB / NU)), t0 = UT * (u % (NB / NU));
    const int f = f0 + col < Cout ? f0 + col : Cout - 1;
    f32x16 acc[2][NU] = {};
    const T* const w[2] = {Wp + (int64_t)f * C, Wg + (int64_t)f * C};
    tile_gemm_n<T, 2, NU, false, VEC, 2>(acc, xs + t0 * rx, rx, tile_perm(col), w, C);
    const float bp = Bp[f], bg = Bg[f];
#pragma unroll
    for (int n = 0; n < NU; ++n) {
      const float* mk = msk + t0 + 32 * n + 16 * hl;
      store16<T, true>(o + col * OR + 32 * n + 16 * hl, 16, [&](int v) __attribute__((always_inline)) {
        return (T)((acc[0][n][v] + bp) * sigmoid(acc[1][n][v] + bg) * mk[v]);
      });
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    constexpr int LPR = UT / M::VE, FPI = 64 / LPR;  // lanes per feature row, features per instruction
#pragma unroll
    for (int k = 0; k < 32 / FPI; ++k) {
      const int fr = k * FPI + lane / LPR, tc = lane % LPR * M::VE;
      const V v = *reinterpret_cast<const V*>(o + fr * OR + tc);
      if (f0 + fr < Cout) {
        T* dst = abt + (int64_t)(f0 + fr) * fstride + t0 + tc;
        if constexpr (VEC) {
          *reinterpret_cast<V*>(dst) = v;
        } else {
#pragma unroll
          for (int e = 0; e < M::VE; ++e) dst[e] = v[e];
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();  // read before the next unit overwrites it
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

template <typename T, int NB, int NU, bool VEC>
__global__ __launch_bounds__(256, 3) void tmu_generic_out_kernel(const T* __restrict__ y, const T* __restrict__ x,
                                                             const T* __restrict__ Wp, const T* __restrict__ Wg,
                                                             const float* __restrict__ Bp,
                                                             const float* __restrict__ Bg, const T* __restrict__ res,
                                                             T* __restrict__ out, uint32_t L, int C, int Cout,
                                                             uint32_t ldy, int64_t cstride, float eps) {
  using M = TileMma<T>;
  using V = typename M::V;
  constexpr int TT = 32 * NB, TPT = 256 / TT;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int rx = tile_row<T>(C), KP = tile_kp(C);
  T* ys = reinterpret_cast<T*>(smem);  // [TT][rx] LN_out(y)
  T* xs = ys + TT * rx;                // [TT][rx] LN_in(x)
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hl = lane >> 5, col = lane & 31;
  const uint32_t tpr = (L + TT - 1) / TT, bi = blockIdx.x / tpr, j0 = (blockIdx.x - bi * tpr) * TT;  // bi = b * L + i
  const int ntok = (int)(L - j0 < (uint32_t)TT ? L - j0 : TT);
  const int t = tid / TPT, part = tid % TPT;
  stage_row<T, TPT, VEC>(xs + t * rx, x + ((int64_t)bi * L + j0 + (t < ntok ? t : ntok - 1)) * C, true, part, C, KP);
  {
    // y: 16 bytes (VE tokens) of KC channels per thread and step, written as KC-channel pieces of VE token
    // rows (columns up to ldy exist; those past L are dropped at the end)
    constexpr int KC = sizeof(T) == 2 ? 2 : 1, G = TT / M::VE, S = 256 / G * KC, U = 2;
    const T* yr = y + (int64_t)bi * ldy + j0 + tid % G * M::VE;
    for (int k0 = tid / G * KC; k0 < KP; k0 += U * S) {
      V v[U][KC];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int j = 0; j < KC; ++j) {
          const int k = k0 + u * S + j;
          if constexpr (VEC) {
            v[u][j] = ldg<V>(yr + (k < C ? k : 0) * cstride);
            if (k >= C) v[u][j] = V{};
          } else {
#pragma unroll
            for (int e = 0; e < M::VE; ++e) v[u][j][e] = k < C ? yr[k * cstride + e] : (T)0.f;
          }
        }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (k0 + u * S >= KP) continue;
#pragma unroll
        for (int e = 0; e < M::VE; ++e) {
          vec<T, KC> p;
#pragma unroll
          for (int j = 0; j < KC; ++j) p[j] = v[u][j][e];
          *reinterpret_cast<vec<T, KC>*>(ys + (tid % G * M::VE + e) * rx + k0 + u * S) = p;
        }
      }
    }
  }
  __syncthreads();
  {
    float mean, rstd;
    row_stats<T, TPT>(ys + t * rx, part, C, eps, mean, rstd);
    normalise_row<T, TPT>(ys + t * rx, part, C, mean, rstd, nullptr, nullptr);
    row_stats<T, TPT>(xs + t * rx, part, C, eps, mean, rstd);
    normalise_row<T, TPT>(xs + t * rx, part, C, mean, rstd, nullptr, nullptr);
  }
  __syncthreads();
  const int nunits = (Cout + 31) / 32 * (NB / NU);
  for (int u = wave; u < nunits; u += 4) {
    const int f0 = 32 * (u / (NB / NU)), t0 = 32 * NU * (u % (NB / NU));
    const int row = f0 + tile_perm(col), fr = row < Cout ? row : Cout - 1, fl = f0 + 16 * hl;
    f32x16 ap[1][NU] = {}, ag[1][NU] = {};
    tile_gemm<T, NU, true, VEC>(ap, ys + t0 * rx, rx, col, Wp + (int64_t)fr * C, C);
    tile_gemm<T, NU, true, VEC>(ag, xs + t0 * rx, rx, col, Wg + (int64_t)fr * C, C);
    if (fl >= Cout) continue;
    const f32x16 bp = load16<float, false>(Bp + fl, Cout - fl), bg = load16<float, false>(Bg + fl, Cout - fl);
#pragma unroll
    for (int n = 0; n < NU; ++n) {
      const int tk = t0 + 32 * n + col;
      if (tk >= ntok) continue;
      const int64_t off = ((int64_t)bi * L + j0 + tk) * Cout + fl;
      auto val = [&](int v) __attribute__((always_inline)) {
        return (T)((ap[0][n][v] + bp[v]) * sigmoid(ag[0][n][v] + bg[v]));
      };
      if (res) {
        const f32x16 rv = load16<T, VEC>(res + off, Cout - fl);
        store16<T, VEC>(out + off, Cout - fl,
                        [&](int v) __attribute__((always_inline)) { return (T)(rv[v] + (float)val(v)); });
      } else {
        store16<T, VEC>(out + off, Cout - fl, val);
      }
    }
  }
}

// Both phases take 64 tokens per block or 32 (`half`, see the callers), and one 32-token tile per unit
// instead of all where there are fewer chunks of features than waves.
#define TOPS_TMU_SHAPES(CALL, T, half, Cout, vec)  \
  do {                                             \
    if (half) {                                    \
      if (vec)                                     \
        CALL(T, 1, 1, true);                       \
      else                                         \
        CALL(T, 1, 1, false);                      \
    } else if ((Cout) <= 96) {                     \
      if (vec)                                     \
        CALL(T, 2, 1, true);                       \
      else                                         \
        CALL(T, 2, 1, false);                      \
    } else {                                       \
      if (vec)                                     \
        CALL(T, 2, 2, true);                       \
      else                                         \
        CALL(T, 2, 2, false);                      \
    }                                              \
  } while (0)

template <typename T>
static int tmu_generic_in_t(const void* x, const void* mask, const void* Wp, const void* Wg, const float* Bp,
                            const float* Bg, void* ab, int64_t B, int64_t L, int64_t C, int64_t C_out, int64_t ld,
                            int transpose, float eps, hipStream_t st) {
  if (B * L == 0) return TOPS_OK;
  TOPS_REQUIRE(B * L * (ld / 32) < (1LL << 31), "tops_tmu_input_phase: too many tokens");
  const bool vec = aligned16({x, Wp, Wg, ab}) && C % TileMma<T>::VE == 0;
  auto lds = [&](int nb, int nu) {
    return (size_t)(32 * nb * tile_row<T>((int)C) + 4 * 32 * (32 * nu + TileMma<T>::VE)) * sizeof(T) + 32 * nb * 4;
  };
#define TOPS_TMU_IN(T, NB, NU, VEC)                                                                                 \
  do {                                                                                                              \
    (void)hipFuncSetAttribute((const void*)tmu_generic_in_kernel<T, NB, NU, VEC>,                                   \
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds(NB, NU));                        \
    hipLaunchKernelGGL((tmu_generic_in_kernel<T, NB, NU, VEC>), dim3((unsigned)(B * L * (ld / (32 * NB)))), dim3(256), \
                       lds(NB, NU), st, (const T*)x, (const int8_t*)mask, (const T*)Wp, (const T*)Wg, Bp, Bg,       \
                       (T*)ab, (uint32_t)L, (int)C, (int)C_out, (uint32_t)ld, B * L * ld, transpose, eps);           \
  } while (0)
  // 64 tokens (each weight row read half as often) unless they do not fit in LDS or, in fp32, give a CU
  // fewer than 4 blocks: C = 128 fp32 L = 200 (3 per CU) 87 us, 81 with 32; L = 256 91 and 98; bf16 C = 64
  // L = 256 13.5 and 17.6, L = 128 equal
  const bool half = lds(2, 2) > 160 * 1024 || (sizeof(T) == 4 && B * L * (ld / 64) < 4 * num_cus());
  TOPS_TMU_SHAPES(TOPS_TMU_IN, T, half, C_out, vec);
#undef TOPS_TMU_IN
  return launched("tops_tmu_input_phase");
}

template <typename T>
static int tmu_generic_out_t(const void* y, const void* x, const void* Wp, const void* Wg, const float* Bp,
                             const float* Bg, const void* res, void* out, int64_t B, int64_t L, int64_t C,
                             int64_t C_out, int64_t ldy, float eps, hipStream_t st) {
  if (B * L == 0) return TOPS_OK;
  TOPS_REQUIRE(B * L * ((L + 31) / 32) < (1LL << 31), "tops_tmu_output_phase: too many tokens");
  const bool vec = aligned16({y, x, Wp, Wg, res, out}) && multiples_of(TileMma<T>::VE, {C, C_out});
  auto lds = [&](int nb) { return (size_t)2 * 32 * nb * tile_row<T>((int)C) * sizeof(T); };
#define TOPS_TMU_OUT(T, NB, NU, VEC)                                                                                \
  do {                                                                                                              \
    (void)hipFuncSetAttribute((const void*)tmu_generic_out_kernel<T, NB, NU, VEC>,                                  \
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds(NB));                            \
    hipLaunchKernelGGL((tmu_generic_out_kernel<T, NB, NU, VEC>),                                                     \
                       dim3((unsigned)(B * L * ((L + 32 * NB - 1) / (32 * NB)))), dim3(256), lds(NB), st, (const T*)y, \
                       (const T*)x, (const T*)Wp, (const T*)Wg, Bp, Bg, (const T*)res, (T*)out, (uint32_t)L, (int)C, \
                       (int)C_out, (uint32_t)ldy, B * L * ldy, eps);                                                 \
  } while (0)
  // 64 tokens unless they do not fit in LDS or, in fp32, leave a CU room for fewer than 3 blocks: fp32
  // C = 128 L = 200 62 us, 50 with 32, L = 320 104 and 99; C = 64 L = 512 82 and 104; bf16, bound by the weight
  // reads sooner, C = 256 L = 300 95 and 118
  const bool half = lds(2) > 160 * 1024 || (sizeof(T) == 4 && 3 * lds(2) > 160 * 1024);
  TOPS_TMU_SHAPES(TOPS_TMU_OUT, T, half, C_out, vec);
#undef TOPS_TMU_OUT
  return launched("tops_tmu_output_phase");
}

int tmu_generic_input_phase(const void* x, const void* mask, const void* Wp, const void* Wg, const float* Bp,
                            const float* Bg, void* ab, int64_t B, int64_t L, int64_t C, int64_t C_out, int64_t ld,
                            int transpose, float eps, int dtype, hipStream_t st) {
  TOPS_REQUIRE(C >= 1 && C <= 1024 && C_out >= 1 && C_out <= 4096,
               "tops_tmu_input_phase: supports C <= 1024, C_out <= 4096 (got %lld, %lld)", (long long)C,
               (long long)C_out);
  if (dtype == TOPS_DTYPE_BF16)
    return tmu_generic_in_t<__bf16>(x, mask, Wp, Wg, Bp, Bg, ab, B, L, C, C_out, ld, transpose, eps, st);
  if (dtype == TOPS_DTYPE_F16)
    return tmu_generic_in_t<_Float16>(x, mask, Wp, Wg, Bp, Bg, ab, B, L, C, C_out, ld, transpose, eps, st);
  if (dtype == TOPS_DTYPE_F32)
    return tmu_generic_in_t<float>(x, mask, Wp, Wg, Bp, Bg, ab, B, L, C, C_out, ld, transpose, eps, st);
  return fail(TOPS_EUNSUPPORTED, "tops_tmu_input_phase: unsupported dtype code %d", dtype);
}

int tmu_generic_output_phase(const void* y, const void* x, const void* Wp, const void* Wg, const float* Bp,
                             const float* Bg, const void* res, void* out, int64_t B, int64_t L, int64_t C,
                             int64_t C_out, int64_t ldy, float eps, int dtype, hipStream_t st) {
  TOPS_REQUIRE(C >= 1 && C <= 512 && C_out >= 1 && C_out <= 4096,
               "tops_tmu_output_phase: supports C <= 512, C_out <= 4096 (got %lld, %lld)", (long long)C,
               (long long)C_out);
  if (dtype == TOPS_DTYPE_BF16)
    return tmu_generic_out_t<__bf16>(y, x, Wp, Wg, Bp, Bg, res, out, B, L, C, C_out, ldy, eps, st);
  if (dtype == TOPS_DTYPE_F16)
    return tmu_generic_out_t<_Float16>(y, x, Wp, Wg, Bp, Bg, res, out, B, L, C, C_out, ldy, eps, st);
  if (dtype == TOPS_DTYPE_F32)
    return tmu_generic_out_t<float>(y, x, Wp, Wg, Bp, Bg, res, out, B, L, C, C_out, ldy, eps, st);
  return fail(TOPS_EUNSUPPORTED, "tops_tmu_output_phase: unsupported dtype code %d", dtype);
}

}  // namespace tops

using namespace tops;

extern "C" int tops_tri_generic_prep(const void* x, int64_t sx0, int64_t sx1, const void* w_ln, const void* b_ln,
                                     int apply_ln, const void* wqkv, const void* WZ, const float* BZ, void* xln,
                                     void* q, void* k, void* v, float* bias, int64_t N, int64_t C, int64_t H,
                                     int64_t D, float eps, int dtype, void* stream) {
  TOPS_REQUIRE(x && wqkv && WZ && xln && q && k && v && bias, "tops_tri_generic_prep: null pointer argument");
  TOPS_REQUIRE(!apply_ln || w_ln, "tops_tri_generic_prep: w_ln is required when apply_ln != 0");
  TOPS_REQUIRE(N >= 0 && N <= 65536, "tops_tri_generic_prep: bad N %lld", (long long)N);
  TOPS_REQUIRE(C >= 1 && C <= 1024 && H >= 1 && H <= 64 && D >= 1 && D <= 64,
               "tops_tri_generic_prep: supports C <= 1024, H <= 64, D <= 64 (got %lld, %lld, %lld)", (long long)C,
               (long long)H, (long long)D);
  hipStream_t st = (hipStream_t)stream;
  if (dtype == TOPS_DTYPE_BF16)
    return tri_generic_prep_t<__bf16>(x, sx0, sx1, w_ln, b_ln, apply_ln, wqkv, WZ, BZ, xln, q, k, v, bias, N, (int)C,
                                      (int)H, (int)D, eps, st);
  if (dtype == TOPS_DTYPE_F16)
    return tri_generic_prep_t<_Float16>(x, sx0, sx1, w_ln, b_ln, apply_ln, wqkv, WZ, BZ, xln, q, k, v, bias, N,
                                        (int)C, (int)H, (int)D, eps, st);
  if (dtype == TOPS_DTYPE_F32)
    return tri_generic_prep_t<float>(x, sx0, sx1, w_ln, b_ln, apply_ln, wqkv, WZ, BZ, xln, q, k, v, bias, N, (int)C,
                                     (int)H, (int)D, eps, st);
  return fail(TOPS_EUNSUPPORTED, "tops_tri_generic_prep: unsupported dtype code %d", dtype);
}

extern "C" int tops_tri_generic_attention(const void* q, const void* k, const void* v, const float* bias,
                                          const void* mask, int64_t sm0, int64_t sm1, void* out, int64_t so0,
                                          int64_t so1, int64_t N, int64_t H, int64_t D, float scale, int dtype,
                                          void* stream) {
  TOPS_REQUIRE(q && k && v && bias && out, "tops_tri_generic_attention: null pointer argument");
  TOPS_REQUIRE(N >= 0 && N <= 65536 && H >= 1 && H <= 64 && D >= 1 && D <= 64,
               "tops_tri_generic_attention: supports H <= 64, D <= 64 (got N=%lld H=%lld D=%lld)", (long long)N,
               (long long)H, (long long)D);
  hipStream_t st = (hipStream_t)stream;
  if (dtype == TOPS_DTYPE_BF16)
    return generic_attention_t<__bf16, false>("tops_tri_generic_attention", q, k, v, bias, mask, sm0, sm1, out, so0, so1, N, N,
                                      (int)H, (int)D, scale, st);
  if (dtype == TOPS_DTYPE_F16)
    return generic_attention_t<_Float16, false>("tops_tri_generic_attention", q, k, v, bias, mask, sm0, sm1, out, so0, so1, N, N,
                                      (int)H, (int)D, scale, st);
  if (dtype == TOPS_DTYPE_F32)
    return generic_attention_t<float, false>("tops_tri_generic_attention", q, k, v, bias, mask, sm0, sm1, out, so0, so1, N, N,
                                      (int)H, (int)D, scale, st);
  return fail(TOPS_EUNSUPPORTED, "tops_tri_generic_attention: unsupported dtype code %d", dtype);
}

extern "C" int tops_apb_generic_prep(const void* X, const void* wqkv, const void* Z, int64_t sz0, int64_t sz1,
                                     const float* Wc, const float* Bc, void* q, void* k, void* v, float* bias,
                                     int64_t M, int64_t C, int64_t Cz, int64_t H, int64_t D, float eps, int dtype,
                                     void* stream) {
  TOPS_REQUIRE(X && wqkv && Z && Wc && Bc && q && k && v && bias, "tops_apb_generic_prep: null pointer argument");
  TOPS_REQUIRE(M >= 0 && M <= 65536 && C >= 1 && C <= 4096 && Cz >= 1 && Cz <= 1024 && H >= 1 && H <= 64 && D >= 1 &&
                   D <= 64,
               "tops_apb_generic_prep: supports C <= 4096, Cz <= 1024, H <= 64, D <= 64 (got M=%lld C=%lld Cz=%lld "
               "H=%lld D=%lld)",
               (long long)M, (long long)C, (long long)Cz, (long long)H, (long long)D);
  hipStream_t st = (hipStream_t)stream;
  if (dtype == TOPS_DTYPE_BF16)
    return apb_generic_prep_t<__bf16>(X, wqkv, Z, sz0, sz1, Wc, Bc, q, k, v, bias, M, (int)C, (int)Cz, (int)H, (int)D,
                                      eps, st);
  if (dtype == TOPS_DTYPE_F16)
    return apb_generic_prep_t<_Float16>(X, wqkv, Z, sz0, sz1, Wc, Bc, q, k, v, bias, M, (int)C, (int)Cz, (int)H,
                                        (int)D, eps, st);
  if (dtype == TOPS_DTYPE_F32)
    return apb_generic_prep_t<float>(X, wqkv, Z, sz0, sz1, Wc, Bc, q, k, v, bias, M, (int)C, (int)Cz, (int)H, (int)D,
                                     eps, st);
  return fail(TOPS_EUNSUPPORTED, "tops_apb_generic_prep: unsupported dtype code %d", dtype);
}

extern "C" int tops_apb_generic_attention(const void* q, const void* k, const void* v, const float* bias,
                                          const void* mask, void* Og, int64_t M, int64_t H, int64_t D, float scale,
                                          int dtype, void* stream) {
  TOPS_REQUIRE(q && k && v && bias && Og, "tops_apb_generic_attention: null pointer argument");
  TOPS_REQUIRE(M >= 0 && M <= 65536 && H >= 1 && H <= 64 && D >= 1 && D <= 64,
               "tops_apb_generic_attention: supports H <= 64, D <= 64 (got M=%lld H=%lld D=%lld)", (long long)M,
               (long long)H, (long long)D);
  hipStream_t st = (hipStream_t)stream;
  if (dtype == TOPS_DTYPE_BF16)
    return generic_attention_t<__bf16, true>("tops_apb_generic_attention", q, k, v, bias, mask, 0, 1, Og, 0, H * D, 1, M, (int)H,
                                     (int)D, scale, st);
  if (dtype == TOPS_DTYPE_F16)
    return generic_attention_t<_Float16, true>("tops_apb_generic_attention", q, k, v, bias, mask, 0, 1, Og, 0, H * D, 1, M, (int)H,
                                     (int)D, scale, st);
  if (dtype == TOPS_DTYPE_F32)
    return generic_attention_t<float, true>("tops_apb_generic_attention", q, k, v, bias, mask, 0, 1, Og, 0, H * D, 1, M, (int)H,
                                     (int)D, scale, st);
  return fail(TOPS_EUNSUPPORTED, "tops_apb_generic_attention: unsupported dtype code %d", dtype);
}

static int gate_generic_dispatch(const void* o, int64_t so0, int64_t so1, const void* gin, int64_t sg0, int64_t sg1,
                                 const void* w_ln, const void* b_ln, float ln_eps, int apply_ln, const void* Wg,
                                 const void* bg, const void* Wo, const void* bo, const void* res, int64_t sr0,
                                 int64_t sr1, void* out, int64_t sd0, int64_t sd1, int64_t M1, int64_t M2, int64_t Cin,
                                 int64_t HD, int64_t Cout, int dtype, hipStream_t st) {
  if (dtype == TOPS_DTYPE_BF16)
    return gate_generic_t<__bf16>(o, so0, so1, gin, sg0, sg1, w_ln, b_ln, ln_eps, apply_ln, Wg, bg, Wo, bo, res, sr0,
                                  sr1, out, sd0, sd1, M1, M2, (int)Cin, (int)HD, (int)Cout, st);
  if (dtype == TOPS_DTYPE_F16)
    return gate_generic_t<_Float16>(o, so0, so1, gin, sg0, sg1, w_ln, b_ln, ln_eps, apply_ln, Wg, bg, Wo, bo, res,
                                    sr0, sr1, out, sd0, sd1, M1, M2, (int)Cin, (int)HD, (int)Cout, st);
  if (dtype == TOPS_DTYPE_F32)
    return gate_generic_t<float>(o, so0, so1, gin, sg0, sg1, w_ln, b_ln, ln_eps, apply_ln, Wg, bg, Wo, bo, res, sr0,
                                 sr1, out, sd0, sd1, M1, M2, (int)Cin, (int)HD, (int)Cout, st);
  return fail(TOPS_EUNSUPPORTED, "tops_gate_out_generic: unsupported dtype code %d", dtype);
}

extern "C" int tops_gate_out_generic(const void* o, int64_t so0, int64_t so1, const void* gin, int64_t sg0,
                                     int64_t sg1, const void* w_ln, const void* b_ln, float ln_eps, int apply_ln,
                                     const void* Wg, const void* bg, const void* Wo, const void* bo, void* out,
                                     int64_t M1, int64_t M2, int64_t Cin, int64_t HD, int64_t Cout, int dtype,
                                     void* stream) {
  TOPS_REQUIRE(o && gin && Wg && Wo && out, "tops_gate_out_generic: null pointer argument");
  TOPS_REQUIRE(!apply_ln || w_ln, "tops_gate_out_generic: w_ln is required when apply_ln != 0");
  TOPS_REQUIRE(M1 >= 0 && M2 >= 0, "tops_gate_out_generic: bad sizes");
  TOPS_REQUIRE(Cin >= 1 && HD >= 1 && Cout >= 1 && Cin + HD <= 1024 && Cout <= 4096,
               "tops_gate_out_generic: supports C_in + H*D <= 1024, C_out <= 4096 (got %lld, %lld, %lld)",
               (long long)Cin, (long long)HD, (long long)Cout);
  return gate_generic_dispatch(o, so0, so1, gin, sg0, sg1, w_ln, b_ln, ln_eps, apply_ln, Wg, bg, Wo, bo, nullptr, 0, 0,
                               out, M2 * Cout, Cout, M1, M2, Cin, HD, Cout, dtype, (hipStream_t)stream);
}

extern "C" int tops_gate_out_generic_residual(const void* o, int64_t so0, int64_t so1, const void* gin, int64_t sg0,
                                              int64_t sg1, const void* w_ln, const void* b_ln, float ln_eps,
                                              int apply_ln, const void* Wg, const void* bg, const void* Wo,
                                              const void* bo, const void* res, int64_t sr0, int64_t sr1, void* out,
                                              int64_t sd0, int64_t sd1, int64_t M1, int64_t M2, int64_t Cin,
                                              int64_t HD, int64_t Cout, int dtype, void* stream) {
  TOPS_REQUIRE(o && gin && Wg && Wo && res && out, "tops_gate_out_generic_residual: null pointer argument");
  TOPS_REQUIRE(!apply_ln || w_ln, "tops_gate_out_generic_residual: w_ln is required when apply_ln != 0");
  TOPS_REQUIRE(M1 >= 0 && M2 >= 0, "tops_gate_out_generic_residual: bad sizes");
  TOPS_REQUIRE(Cin >= 1 && HD >= 1 && Cout >= 1 && Cin + HD <= 1024 && Cout <= 4096,
               "tops_gate_out_generic_residual: supports C_in + H*D <= 1024, C_out <= 4096 (got %lld, %lld, %lld)",
               (long long)Cin, (long long)HD, (long long)Cout);
  return gate_generic_dispatch(o, so0, so1, gin, sg0, sg1, w_ln, b_ln, ln_eps, apply_ln, Wg, bg, Wo, bo, res, sr0, sr1,
                               out, sd0, sd1, M1, M2, Cin, HD, Cout, dtype, (hipStream_t)stream);
}

static size_t io_size(int dtype) { return dtype == TOPS_DTYPE_F32 ? 4 : 2; }

extern "C" int64_t tops_gate_generic_workspace_bytes(int64_t M1, int64_t M2, int64_t Cin, int64_t HD, int64_t Cout,
                                                     int apply_ln, int dtype) {
  if (M1 <= 0 || M2 <= 0 || !gate_few(M1, M2, Cin, HD, Cout, apply_ln, io_size(dtype))) return 0;
  return M1 * HD * (int64_t)io_size(dtype);
}

extern "C" int tops_gate_out_generic_work(const void* o, int64_t so0, int64_t so1, const void* gin, int64_t sg0,
                                          int64_t sg1, const void* w_ln, const void* b_ln, float ln_eps, int apply_ln,
                                          const void* Wg, const void* bg, const void* Wo, const void* bo,
                                          const void* res, int64_t sr0, int64_t sr1, void* out, int64_t sd0,
                                          int64_t sd1, void* work, int64_t M1, int64_t M2, int64_t Cin, int64_t HD,
                                          int64_t Cout, int dtype, void* stream) {
  TOPS_REQUIRE(o && gin && Wg && Wo && out, "tops_gate_out_generic_work: null pointer argument");
  TOPS_REQUIRE(!apply_ln || w_ln, "tops_gate_out_generic_work: w_ln is required when apply_ln != 0");
  TOPS_REQUIRE(M1 >= 0 && M2 >= 0, "tops_gate_out_generic_work: bad sizes");
  TOPS_REQUIRE(Cin >= 1 && HD >= 1 && Cout >= 1 && Cin + HD <= 1024 && Cout <= 4096,
               "tops_gate_out_generic_work: supports C_in + H*D <= 1024, C_out <= 4096 (got %lld, %lld, %lld)",
               (long long)Cin, (long long)HD, (long long)Cout);
  hipStream_t st = (hipStream_t)stream;
  if (!work || M1 == 0 || !gate_few(M1, M2, Cin, HD, Cout, apply_ln, io_size(dtype)))
    return gate_generic_dispatch(o, so0, so1, gin, sg0, sg1, w_ln, b_ln, ln_eps, apply_ln, Wg, bg, Wo, bo, res, sr0,
                                 sr1, out, sd0, sd1, M1, M2, Cin, HD, Cout, dtype, st);
  if (dtype == TOPS_DTYPE_BF16)
    return gate_few_t<__bf16>(o, so0, gin, sg0, Wg, bg, Wo, bo, res, sr0, out, sd0, work, (int)M1, (int)Cin, (int)HD,
                              (int)Cout, st);
  if (dtype == TOPS_DTYPE_F16)
    return gate_few_t<_Float16>(o, so0, gin, sg0, Wg, bg, Wo, bo, res, sr0, out, sd0, work, (int)M1, (int)Cin, (int)HD,
                                (int)Cout, st);
  if (dtype == TOPS_DTYPE_F32)
    return gate_few_t<float>(o, so0, gin, sg0, Wg, bg, Wo, bo, res, sr0, out, sd0, work, (int)M1, (int)Cin, (int)HD,
                             (int)Cout, st);
  return fail(TOPS_EUNSUPPORTED, "tops_gate_out_generic_work: unsupported dtype code %d", dtype);
}
