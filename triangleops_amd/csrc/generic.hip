// Any-shape kernels for the triangle-attention op and the gate / output projection: the
// shapes the tuned kernels do not cover (C_in != 128, D != 32, H != 4, C_out != 128, e.g. the
// D = 16, C_in = 64 "Apo" configuration).  Plain fp32 VALU arithmetic (no MFMA), written for
// correctness at small and medium sizes, and the path of fp32 I/O (then every value stays fp32);
// with 16-bit I/O the rounding points follow the tuned path:
//   LN(x) is rounded to the I/O type before the Q / K / V and gate products, Q / K / V and the
//   gated activations are rounded to the I/O type, the pair bias stays fp32.
//
//   tri_generic_prep_kernel   per token: LN(x) (fp32, two-pass), Q / K / V of all heads and
//                             the row-shared pair bias bias[h][a][b] = LN(x[a, b]) . Wz[h] + bz[h]
//   tri_generic_attn_kernel   64 queries of one (row i, head h) per block, keys split over 4 waves
//                             in 32-key chunks staged in LDS: online softmax in fp32, scores
//                             q . k * scale + bias, masked keys get the reference's fp32 "+ (-1e9)"
//   gate_generic_kernel       per token: y = (o * sigmoid(g . Wg^T + bg)) -> io, out = y . Wo^T + bo
//                             with g = LN(gin) or gin
//
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
constexpr int kTK = 32;      // k-tile of the weights the tiled kernels stage through LDS

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
// cores and the weight reads; N = 200, C = 128, H = 4, D = 32: fp32 130 -> 60 us, bf16 193 -> 29 us
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
    f32x16 acc[1] = {};
    tile_gemm<T, 1, true, VEC>(acc, xs, rx, col, wqkv + (int64_t)(row < F ? row : F - 1) * C, C);
    if (tok0 + col < ntok)
      store_qkv16<T>(qo, ko, vo, (tok0 + col) * HD, fl, F - fl, D, pw,
                     [&](int v) __attribute__((always_inline)) { return acc[0][v]; });
  }
}

// ---------------------------------------------------------------------------------------------
// Attention over R rows of N queries and N keys, any H, D <= DP (16, 32 or 64).  A wave holds 32 queries of one
// (row i, head h) and walks the keys in chunks of 32: S^T = K . Q^T (a lane: one query, the 16 keys
// k0 + 16 hl + v), scores q . k * scale + bias with masked keys (mask[i*sm0 + k*sm1] == 0) getting
// "+ (-1e9)" in fp32 (triangle attention) or -inf (MASK_INF, attention_pair_bias: a row without valid
// keys gives NaN, as torch's softmax does) and keys >= N left out, online softmax in fp32, and
// O^T += V^T . P^T with the score registers as the operand.  fp32 I/O runs the fp32 MFMA throughout;
// with 16-bit I/O the fp32 weights enter as two 16-bit terms (hi + lo, two MFMAs: 16 bits of each
// weight or more, as fp16 weights are scaled by 2^10 to stay clear of its denormals).
// K, V and the bias rows come straight from L2 in operand order (K rows as 16-byte chunks, V an element
// per key and lane, which is the transpose): no LDS and no barrier in the loop.  With KSPL = 1 a block's
// 4 waves take 4 query tiles and share the key reads through L1; with KSPL = 4 they take every 4th chunk
// of one query tile and merge (m, l, o) through LDS.  Bound by the fp32 MFMAs in fp32 (N = 200, 4 heads
// of 32: 247 -> 75 us against a query per lane on the VALU, half of the fp32 matrix rate), by the
// exponentials and the split of the weights in 16 bits (the same in bf16: 245 -> 44 us).
// ---------------------------------------------------------------------------------------------
template <typename T, int DP, int KSPL, bool MASK_INF, bool VEC>
__global__ __launch_bounds__(256, DP <= 32 ? 4 : 2) void tri_generic_attn_kernel(
    const T* __restrict__ qi_, const T* __restrict__ ki_, const T* __restrict__ vi_, const float* __restrict__ bias,
    const int8_t* __restrict__ mask, int64_t sm0, int64_t sm1, T* __restrict__ out, int64_t so0, int64_t so1, int N,
    int H, int D, float scale) {
  using M = TileMma<T>;
  using V = typename M::V;
  constexpr int ND = (DP + 31) / 32;               // 32-channel tiles of O
  constexpr int NQ = DP / M::KS, NV = 16 / M::VE;  // k-steps of q . k, 16-byte pieces of 16 keys
  constexpr int QB = 128 / KSPL;                          // queries per block
  constexpr float kShift = std::is_same<T, _Float16>::value ? 10.f : 0.f;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hl = lane >> 5, col = lane & 31;
  const uint32_t nqb = (N + QB - 1) / QB, ih = blockIdx.x / nqb, qb = blockIdx.x - ih * nqb;
  const int i = ih / (uint32_t)H, h = ih - i * H;
  const int q0 = qb * QB + (KSPL == 1 ? 32 * wave : 0);
  if (KSPL == 1 && q0 >= N) return;
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
  const int nch = (N + 31) / 32;
  int c = KSPL == 1 ? 0 : wave;
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
    if (__builtin_amdgcn_ballot_w64(mn != m) != 0) {
      const float corr = fast_exp2((m - sh) * kLog2e);
      l *= corr;
#pragma unroll
      for (int n = 0; n < ND; ++n)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[n][v] *= corr;
      m = mn;
    }
    V p[NV], pl[NV];
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const float w = fast_exp2(fmaf(s[v] - sh, kLog2e, kShift));
      l += w;
      const T hi = (T)w;
      p[v / M::VE][v % M::VE] = hi;
      pl[v / M::VE][v % M::VE] = (T)(w - (float)hi);
    }
#pragma unroll
    for (int n = 0; n < ND; ++n)
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        o[n] = M::mma(vf[n][j], p[j], o[n]);
        if constexpr (sizeof(T) == 2) o[n] = M::mma(vf[n][j], pl[j], o[n]);
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
    f32x16 acc[1] = {};
    tile_gemm<T, 1, true, VEC>(acc, gs, rg, col, Wg + (int64_t)(row < HD ? row : HD - 1) * Cin, Cin);
    const f32x16 b = load16<T, VEC>(bg && fl < HD ? bg + fl : nullptr, HD - fl);
    T* y = ys + col * ry + fl;
    store16<T, true>(y, 16, [&](int v) __attribute__((always_inline)) {
      return (T)((float)y[v] * sigmoid(acc[0][v] + b[v]));
    });
  }
  __syncthreads();
  // output projection; with a residual, the result is rounded first as a separate add would see it
  const int64_t tok = tok0 + col < M ? tok0 + col : M - 1, m1 = tok / M2, m2 = tok - m1 * M2;
  for (int f0 = 32 * wave; f0 < Cout; f0 += 32 * NW) {
    const int row = f0 + tile_perm(col), fl = f0 + 16 * hl;
    f32x16 acc[1] = {};
    tile_gemm<T, 1, true, VEC>(acc, ys, ry, col, Wo + (int64_t)(row < Cout ? row : Cout - 1) * HD, HD);
    if (tok0 + col >= M || fl >= Cout) continue;
    const f32x16 b = load16<T, VEC>(bo ? bo + fl : nullptr, Cout - fl);
    T* dst = out + m1 * sd0 + m2 * sd1 + fl;
    if (res) {
      const f32x16 r = load16<T, VEC>(res + m1 * sr0 + m2 * sr1 + fl, Cout - fl);
      store16<T, VEC>(dst, Cout - fl,
                      [&](int v) __attribute__((always_inline)) { return (T)(r[v] + (float)(T)(acc[0][v] + b[v])); });
    } else {
      store16<T, VEC>(dst, Cout - fl, [&](int v) __attribute__((always_inline)) { return (T)(acc[0][v] + b[v]); });
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
  // keys split over the waves while 128-query blocks are fewer than the CUs (80 blocks, 600 tokens x 16
  // heads of 24, bf16: 14 us against 31; 192 blocks, 1500 tokens: 41 against 75; 400 blocks, N = 100 x 4
  // heads: 13 against 10)
  const bool split = rh * ((N + 127) / 128) < num_cus();
  const int64_t blocks = rh * (split ? (N + 31) / 32 : (N + 127) / 128);
  TOPS_REQUIRE(blocks < (1LL << 31), "%s: too many query blocks", name);
  const bool vec = aligned16({q, k, v, out}) && multiples_of(TileMma<T>::VE, {D, so0, so1});
#define TOPS_GEN_ATTN(DP, KS, VEC)                                                                                  \
  hipLaunchKernelGGL((tri_generic_attn_kernel<T, DP, KS, MASK_INF, VEC>), dim3((unsigned)blocks), dim3(256), 0, st, \
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
  f32x16 acc[1] = {};
  for (int c0 = 0; c0 < C; c0 += kQkvC) {
    const int kc = C - c0 < kQkvC ? C - c0 : kQkvC;
    if (c0 > 0) __syncthreads();
    stage_row<T, 8, VEC>(xs + t * rx, src + c0, ok, part, kc, tile_kp(kc));
    __syncthreads();
    if (f0 < F) tile_gemm<T, 1, true, VEC, 8>(acc, xs, rx, col, w + c0, kc);
  }
  if (tok0 + col < M && f0 < F)
    store_qkv16<T>(qo, ko, vo, (tok0 + col) * HD, fl, F - fl, D, pw,
                   [&](int v) __attribute__((always_inline)) { return acc[0][v]; });
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
// the read of Z and the matrix cores together (600 tokens, 16 heads, C_z = 128, bf16: 148 -> 39 us
// against LDS tiles and FMAs, 2.9 TB/s).
template <typename T, int NKC, bool VEC>
__global__ __launch_bounds__(256) void apb_gen_bias_mma_kernel(const T* __restrict__ Z, int64_t sz0, int64_t sz1,
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
  {
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
    // 2 blocks per CU: 600 tokens x 16 heads, C_z = 128 in bf16 39 us against 42 with 4 and 52 with 8 (whose
    // waves take 3 and 1.5 steps each, unevenly), 500 tokens x 2 heads, C_z = 32 equal within 1 us
    const dim3 grid((unsigned)(steps < 2 * num_cus() ? steps : 2 * num_cus()), (unsigned)((H + 15) / 16));
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
    constexpr int W = 4 * TileMma<T>::VE;  // channels per chunk of the four lanes
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
// triangle_mul/kernel.py:235-326).  Tokens t = (b, i, j) in row-major order.
// ---------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void tmu_generic_in_kernel(const T* __restrict__ x, const int8_t* __restrict__ mask,
                                                            const T* __restrict__ Wp, const T* __restrict__ Wg,
                                                            const float* __restrict__ Bp, const float* __restrict__ Bg,
                                                            T* __restrict__ ab, int64_t B, int64_t L, int C, int Cout,
                                                            int64_t ld, int transpose, float eps) {
  extern __shared__ float xs[];  // [kGenTok][C]
  const int tid = threadIdx.x;
  const int64_t ntok = B * L * L, tok0 = (int64_t)blockIdx.x * kGenTok;
  for (int e = tid; e < kGenTok * C; e += 256) {
    const int64_t tok = tok0 + e / C;
    xs[e] = tok < ntok ? (float)x[tok * C + e % C] : 0.f;
  }
  __syncthreads();
  gen_layer_norm<T>(xs, C, C, nullptr, nullptr, eps);
  __syncthreads();
  for (int e = tid; e < kGenTok * C; e += 256) xs[e] = (float)(T)xs[e];  // GEMM operand in the I/O type
  __syncthreads();
  const int64_t fstride = B * L * ld;
  for (int e = tid; e < kGenTok * Cout; e += 256) {
    const int t = e / Cout, f = e % Cout;
    const int64_t tok = tok0 + t;
    if (tok >= ntok) continue;
    const float* r = xs + t * C;
    const T* wp = Wp + (int64_t)f * C;
    const T* wg = Wg + (int64_t)f * C;
    float p = Bp[f], g = Bg[f];
    for (int c = 0; c < C; ++c) {
      p = fmaf(r[c], (float)wp[c], p);
      g = fmaf(r[c], (float)wg[c], g);
    }
    const float m = mask ? (mask[tok] != 0 ? 1.f : 0.f) : 1.f;
    const int64_t b = tok / (L * L), rem = tok % (L * L), i = rem / L, j = rem % L;
    const int64_t row = transpose ? j : i, col = transpose ? i : j;
    T* dst = ab + f * fstride + (b * L + row) * ld;
    dst[col] = (T)(p * sigmoid(g) * m);
    if (col == L - 1)  // zero k-padding of this row for the einsum
      for (int64_t c = L; c < ld; ++c) dst[c] = (T)0.f;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void tmu_generic_out_kernel(const T* __restrict__ y, const T* __restrict__ x,
                                                             const T* __restrict__ Wp, const T* __restrict__ Wg,
                                                             const float* __restrict__ Bp,
                                                             const float* __restrict__ Bg, const T* __restrict__ res,
                                                             T* __restrict__ out, int64_t B, int64_t L, int C,
                                                             int Cout, int64_t ldy, float eps) {
  extern __shared__ float sm[];
  float* ys = sm;                 // [kGenTok][C]  y of the tile's tokens (token-major)
  float* xs = sm + kGenTok * C;   // [kGenTok][C]  x
  const int tid = threadIdx.x;
  const int64_t ntok = B * L * L, tok0 = (int64_t)blockIdx.x * kGenTok, cstride = B * L * ldy;
  for (int e = tid; e < kGenTok * C; e += 256) {
    const int t = e % kGenTok, c = e / kGenTok;  // token fastest: y is channel-major
    const int64_t tok = tok0 + t;
    float v = 0.f;
    if (tok < ntok) {
      const int64_t b = tok / (L * L), rem = tok % (L * L);
      v = (float)y[c * cstride + (b * L + rem / L) * ldy + rem % L];
    }
    ys[t * C + c] = v;
  }
  for (int e = tid; e < kGenTok * C; e += 256) {
    const int64_t tok = tok0 + e / C;
    xs[e] = tok < ntok ? (float)x[tok * C + e % C] : 0.f;
  }
  __syncthreads();
  gen_layer_norm<T>(ys, C, C, nullptr, nullptr, eps);
  gen_layer_norm<T>(xs, C, C, nullptr, nullptr, eps);
  __syncthreads();
  for (int e = tid; e < 2 * kGenTok * C; e += 256) sm[e] = (float)(T)sm[e];
  __syncthreads();
  for (int e = tid; e < kGenTok * Cout; e += 256) {
    const int t = e / Cout, f = e % Cout;
    const int64_t tok = tok0 + t;
    if (tok >= ntok) continue;
    const float* yr = ys + t * C;
    const float* xr = xs + t * C;
    const T* wp = Wp + (int64_t)f * C;
    const T* wg = Wg + (int64_t)f * C;
    float p = Bp[f], g = Bg[f];
    for (int c = 0; c < C; ++c) {
      p = fmaf(yr[c], (float)wp[c], p);
      g = fmaf(xr[c], (float)wg[c], g);
    }
    const T r = (T)(p * sigmoid(g));
    out[tok * Cout + f] = res ? (T)((float)res[tok * Cout + f] + (float)r) : r;
  }
}

// ---------------------------------------------------------------------------------------------
// Tiled forms of the two phases for C <= 256 (the kernels above remain for wider C): a block
// takes a tile of tokens, normalises them into LDS k-major ([channel][token], fp32, rounded to
// the I/O type as the products' operand, exactly as above), stages the weights of a chunk of
// output features k-major through LDS in 32-deep k-tiles, and each thread accumulates 4 tokens
// x 4 features of P and of G in registers (fp32 FMAs), then applies bias, gate and mask.
//   input phase:  64 tokens of one row r of the (B, L, ld) store grid (tokens (r, c) or,
//                 transposed, (c, r), c = c0 .. c0 + 63; c >= L stores zeros), 64-feature chunks,
//                 each thread's 4 tokens stored as one vector per feature (contiguous in ab)
//   output phase: 32 tokens (b, i, j0 .. j0 + 31), y read channel-major 32 tokens per channel,
//                 128-feature chunks, each thread's 4 features stored as one vector per token
// ---------------------------------------------------------------------------------------------
constexpr int kTinTok = 64, kTinRow = kTinTok + 4;    // input phase: tokens per tile, LDS row
constexpr int kToutTok = 32, kToutRow = kToutTok + 4;  // output phase
constexpr int kTF = 128, kTFRow = kTF + 4;              // output phase: features per chunk, LDS row

// LayerNorm of the `ntok` token columns of a k-major LDS tile (4 threads per token, two-pass),
// rounding the normalised values to T; rows k in [C, CK) are set to zero.
template <typename T>
__device__ inline void tiled_layer_norm(float* xs, int row, int ntok, int C, int CK, float eps) {
  const int t = threadIdx.x >> 2, part = threadIdx.x & 3;
  if (t >= ntok) return;  // whole quads drop out together, so the quad sums stay exact
  float s = 0.f;
  for (int k = part; k < C; k += 4) s += xs[k * row + t];
  const float mean = group_sum<4>(s) / (float)C;
  float q = 0.f;
  for (int k = part; k < C; k += 4) {
    const float d = xs[k * row + t] - mean;
    q = fmaf(d, d, q);
  }
  const float rstd = rsqrtf(group_sum<4>(q) / (float)C + eps);
  for (int k = part; k < CK; k += 4) xs[k * row + t] = k < C ? (float)(T)((xs[k * row + t] - mean) * rstd) : 0.f;
}

template <typename T>
__global__ __launch_bounds__(256) void tmu_gen_in_tiled_kernel(const T* __restrict__ x, const int8_t* __restrict__ mask,
                                                              const T* __restrict__ Wp, const T* __restrict__ Wg,
                                                              const float* __restrict__ Bp, const float* __restrict__ Bg,
                                                              T* __restrict__ ab, int64_t L, int C, int Cout, int64_t ld,
                                                              int64_t fstride, int transpose, float eps) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int CK = (C + kTK - 1) / kTK * kTK;
  float* xs = sm;                     // [CK][kTinRow]  normalised tile
  float* wps = xs + CK * kTinRow;     // [kTK][kTinRow] P weights of the chunk, k-major
  float* wgs = wps + kTK * kTinRow;   // [kTK][kTinRow] G weights
  float* msk = wgs + kTK * kTinRow;   // [kTinTok] 1 for a valid, unmasked token
  const int tid = threadIdx.x;
  const int64_t tpr = ld / kTinTok, rr = blockIdx.x / tpr, r = rr % L, b = rr / L;
  const int64_t c0 = (blockIdx.x % tpr) * kTinTok;
  auto token = [&](int t) -> int64_t {  // x / mask index of tile token t (t >= L - c0: position L - 1)
    int64_t c = c0 + t;
    c = c < L ? c : L - 1;
    return transpose ? (b * L + c) * L + r : (b * L + r) * L + c;
  };
  for (int e = tid; e < kTinTok * C; e += 256) {  // row-major reads, k-major LDS
    const int t = e / C, k = e % C;
    xs[k * kTinRow + t] = (float)x[token(t) * C + k];
  }
  if (tid < kTinTok) msk[tid] = c0 + tid < L ? (mask ? (mask[token(tid)] != 0 ? 1.f : 0.f) : 1.f) : 0.f;
  __syncthreads();
  tiled_layer_norm<T>(xs, kTinRow, kTinTok, C, CK, eps);

  const int ty = tid >> 4, tx = tid & 15;  // tokens 4 ty .. + 3, chunk features 4 tx .. + 3
  T* abt = ab + (b * L + r) * ld + c0 + 4 * ty;
  // (64-feature chunk, 32-deep k-tile) steps in one sequence; each step's P and G weights are
  // loaded into registers during the previous step and stored k-major into LDS after a barrier
  const int nk = CK / kTK, nsteps = ((Cout + 63) / 64) * nk;
  float wr[16];  // P (0-7) and G (8-15) weights (f, k) = (e / kTK, e % kTK), e = tid + 256 i
  auto wload = [&](int step) __attribute__((always_inline)) {
    const int f0 = (step / nk) * 64, k0 = (step % nk) * kTK;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int e = tid + 256 * i, ff = f0 + e / kTK, kk = k0 + e % kTK;
      const bool ok = ff < Cout && kk < C;
      wr[i] = ok ? (float)Wp[(int64_t)ff * C + kk] : 0.f;
      wr[8 + i] = ok ? (float)Wg[(int64_t)ff * C + kk] : 0.f;
    }
  };
  wload(0);
  float ap[4][4] = {}, ag[4][4] = {};
  for (int step = 0; step < nsteps; ++step) {
    __syncthreads();  // the previous step's weights are consumed (step 0: the tile is normalised)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int e = tid + 256 * i;
      wps[(e % kTK) * kTinRow + e / kTK] = wr[i];
      wgs[(e % kTK) * kTinRow + e / kTK] = wr[8 + i];
    }
    __syncthreads();
    if (step + 1 < nsteps) wload(step + 1);
    const int k0 = (step % nk) * kTK;
#pragma unroll 8
    for (int k = 0; k < kTK; ++k) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(&xs[(k0 + k) * kTinRow + 4 * ty]);
      const f32x4 wp = *reinterpret_cast<const f32x4*>(&wps[k * kTinRow + 4 * tx]);
      const f32x4 wg = *reinterpret_cast<const f32x4*>(&wgs[k * kTinRow + 4 * tx]);
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          ap[u][v] = fmaf(a[u], wp[v], ap[u][v]);
          ag[u][v] = fmaf(a[u], wg[v], ag[u][v]);
        }
    }
    if (step % nk != nk - 1) continue;
    const int f0 = (step / nk) * 64;  // the chunk's last k-tile: bias, gate, mask, store
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int f = f0 + 4 * tx + v;
      if (f < Cout) {
        const float bp = Bp[f], bg = Bg[f];
        vec<T, 4> o;
#pragma unroll
        for (int u = 0; u < 4; ++u) o[u] = (T)((ap[u][v] + bp) * sigmoid(ag[u][v] + bg) * msk[4 * ty + u]);
        *reinterpret_cast<vec<T, 4>*>(abt + (int64_t)f * fstride) = o;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) ap[u][v] = ag[u][v] = 0.f;
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void tmu_gen_out_tiled_kernel(const T* __restrict__ y, const T* __restrict__ x,
                                                               const T* __restrict__ Wp, const T* __restrict__ Wg,
                                                               const float* __restrict__ Bp,
                                                               const float* __restrict__ Bg, const T* __restrict__ res,
                                                               T* __restrict__ out, int64_t L, int C, int Cout,
                                                               int64_t ldy, int64_t cstride, float eps) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int CK = (C + kTK - 1) / kTK * kTK;
  float* ys = sm;                      // [CK][kToutRow]  LN_out(y), k-major
  float* xs = ys + CK * kToutRow;      // [CK][kToutRow]  LN_in(x)
  float* wps = xs + CK * kToutRow;     // [kTK][kTFRow]
  float* wgs = wps + kTK * kTFRow;     // [kTK][kTFRow]
  const int tid = threadIdx.x;
  const int64_t tpr = (L + kToutTok - 1) / kToutTok, bi = blockIdx.x / tpr;  // bi = b * L + i
  const int64_t j0 = (blockIdx.x % tpr) * kToutTok;
  const int ntok = (int)(L - j0 < kToutTok ? L - j0 : kToutTok);
  for (int e = tid; e < kToutTok * C; e += 256) {  // y channel-major: 32 consecutive tokens per channel
    const int k = e / kToutTok, t = e % kToutTok;
    ys[k * kToutRow + t] = t < ntok ? (float)y[(int64_t)k * cstride + bi * ldy + j0 + t] : 0.f;
  }
  for (int e = tid; e < kToutTok * C; e += 256) {  // x token-major
    const int t = e / C, k = e % C;
    xs[k * kToutRow + t] = t < ntok ? (float)x[(bi * L + j0 + t) * C + k] : 0.f;
  }
  __syncthreads();
  tiled_layer_norm<T>(ys, kToutRow, kToutTok, C, CK, eps);
  tiled_layer_norm<T>(xs, kToutRow, kToutTok, C, CK, eps);

  const int ty = tid >> 5, tx = tid & 31;  // tokens 4 ty .. + 3, chunk features 4 tx .. + 3
  // (128-feature chunk, 32-deep k-tile) steps in one sequence, weights prefetched into registers
  const int nk = CK / kTK, nsteps = ((Cout + kTF - 1) / kTF) * nk;
  float wr[32];  // P (0-15) and G (16-31) weights (f, k) = (e / kTK, e % kTK), e = tid + 256 i
  auto wload = [&](int step) __attribute__((always_inline)) {
    const int f0 = (step / nk) * kTF, k0 = (step % nk) * kTK;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int e = tid + 256 * i, ff = f0 + e / kTK, kk = k0 + e % kTK;
      const bool ok = ff < Cout && kk < C;
      wr[i] = ok ? (float)Wp[(int64_t)ff * C + kk] : 0.f;
      wr[16 + i] = ok ? (float)Wg[(int64_t)ff * C + kk] : 0.f;
    }
  };
  wload(0);
  float ap[4][4] = {}, ag[4][4] = {};
  for (int step = 0; step < nsteps; ++step) {
    __syncthreads();  // the previous step's weights are consumed (step 0: the tiles are normalised)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int e = tid + 256 * i;
      wps[(e % kTK) * kTFRow + e / kTK] = wr[i];
      wgs[(e % kTK) * kTFRow + e / kTK] = wr[16 + i];
    }
    __syncthreads();
    if (step + 1 < nsteps) wload(step + 1);
    const int k0 = (step % nk) * kTK;
#pragma unroll 8
    for (int k = 0; k < kTK; ++k) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(&ys[(k0 + k) * kToutRow + 4 * ty]);
      const f32x4 g = *reinterpret_cast<const f32x4*>(&xs[(k0 + k) * kToutRow + 4 * ty]);
      const f32x4 wp = *reinterpret_cast<const f32x4*>(&wps[k * kTFRow + 4 * tx]);
      const f32x4 wg = *reinterpret_cast<const f32x4*>(&wgs[k * kTFRow + 4 * tx]);
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          ap[u][v] = fmaf(a[u], wp[v], ap[u][v]);
          ag[u][v] = fmaf(g[u], wg[v], ag[u][v]);
        }
    }
    if (step % nk != nk - 1) continue;
    const int f0 = (step / nk) * kTF;  // the chunk's last k-tile: bias, gate, residual, store
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = 4 * ty + u;
      const int64_t o = (bi * L + j0 + t) * Cout;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int f = f0 + 4 * tx + v;
        if (t < ntok && f < Cout) {
          const T rv = (T)((ap[u][v] + Bp[f]) * sigmoid(ag[u][v] + Bg[f]));
          out[o + f] = res ? (T)((float)res[o + f] + (float)rv) : rv;
        }
        ap[u][v] = ag[u][v] = 0.f;
      }
    }
  }
}

int tmu_generic_input_phase(const void* x, const void* mask, const void* Wp, const void* Wg, const float* Bp,
                            const float* Bg, void* ab, int64_t B, int64_t L, int64_t C, int64_t C_out, int64_t ld,
                            int transpose, float eps, int dtype, hipStream_t st) {
  TOPS_REQUIRE(C >= 1 && C <= 1024 && C_out >= 1 && C_out <= 4096,
               "tops_tmu_input_phase: supports C <= 1024, C_out <= 4096 (got %lld, %lld)", (long long)C,
               (long long)C_out);
  if (C <= 256) {  // tiled kernel
    const int64_t tiles = B * L * (ld / kTinTok);
    if (tiles == 0) return TOPS_OK;
    TOPS_REQUIRE(tiles < (1LL << 31), "tops_tmu_input_phase: too many tokens");
    const int CK = (int)((C + kTK - 1) / kTK * kTK);
    const size_t lds = ((size_t)(CK + 2 * kTK) * kTinRow + kTinTok) * sizeof(float);
    const int64_t fstride = B * L * ld;
#define TOPS_GEN_IN_T(TT)                                                                                        \
  do {                                                                                                           \
    hipFuncSetAttribute((const void*)tmu_gen_in_tiled_kernel<TT>, hipFuncAttributeMaxDynamicSharedMemorySize,    \
                        (int)lds);                                                                               \
    hipLaunchKernelGGL((tmu_gen_in_tiled_kernel<TT>), dim3((unsigned)tiles), dim3(256), lds, st, (const TT*)x,     \
                       (const int8_t*)mask, (const TT*)Wp, (const TT*)Wg, Bp, Bg, (TT*)ab, L, (int)C, (int)C_out, ld, \
                       fstride, transpose, eps);                                                                  \
  } while (0)
    if (dtype == TOPS_DTYPE_BF16)
      TOPS_GEN_IN_T(__bf16);
    else if (dtype == TOPS_DTYPE_F16)
      TOPS_GEN_IN_T(_Float16);
    else if (dtype == TOPS_DTYPE_F32)
      TOPS_GEN_IN_T(float);
    else
      return fail(TOPS_EUNSUPPORTED, "tops_tmu_input_phase: unsupported dtype code %d", dtype);
#undef TOPS_GEN_IN_T
    return launched("tops_tmu_input_phase");
  }
  const int64_t blocks = (B * L * L + kGenTok - 1) / kGenTok;
  if (blocks == 0) return TOPS_OK;
  const size_t lds = (size_t)kGenTok * C * sizeof(float);
#define TOPS_GEN_IN(TT)                                                                                            hipLaunchKernelGGL((tmu_generic_in_kernel<TT>), dim3((unsigned)blocks), dim3(256), lds, st, (const TT*)x,                           (const int8_t*)mask, (const TT*)Wp, (const TT*)Wg, Bp, Bg, (TT*)ab, B, L, (int)C, (int)C_out,                      ld, transpose, eps)
  if (dtype == TOPS_DTYPE_BF16)
    TOPS_GEN_IN(__bf16);
  else if (dtype == TOPS_DTYPE_F16)
    TOPS_GEN_IN(_Float16);
  else if (dtype == TOPS_DTYPE_F32)
    TOPS_GEN_IN(float);
  else
    return fail(TOPS_EUNSUPPORTED, "tops_tmu_input_phase: unsupported dtype code %d", dtype);
#undef TOPS_GEN_IN
  return launched("tops_tmu_input_phase");
}

int tmu_generic_output_phase(const void* y, const void* x, const void* Wp, const void* Wg, const float* Bp,
                             const float* Bg, const void* res, void* out, int64_t B, int64_t L, int64_t C,
                             int64_t C_out, int64_t ldy, float eps, int dtype, hipStream_t st) {
  TOPS_REQUIRE(C >= 1 && C <= 512 && C_out >= 1 && C_out <= 4096,
               "tops_tmu_output_phase: supports C <= 512, C_out <= 4096 (got %lld, %lld)", (long long)C,
               (long long)C_out);
  if (C <= 256) {  // tiled kernel
    const int64_t tiles = B * L * ((L + kToutTok - 1) / kToutTok);
    if (tiles == 0) return TOPS_OK;
    TOPS_REQUIRE(tiles < (1LL << 31), "tops_tmu_output_phase: too many tokens");
    const int CK = (int)((C + kTK - 1) / kTK * kTK);
    const size_t lds = ((size_t)2 * CK * kToutRow + (size_t)2 * kTK * kTFRow) * sizeof(float);
    const int64_t cstride = B * L * ldy;
#define TOPS_GEN_OUT_T(TT)                                                                                       \
  do {                                                                                                           \
    hipFuncSetAttribute((const void*)tmu_gen_out_tiled_kernel<TT>, hipFuncAttributeMaxDynamicSharedMemorySize,   \
                        (int)lds);                                                                               \
    hipLaunchKernelGGL((tmu_gen_out_tiled_kernel<TT>), dim3((unsigned)tiles), dim3(256), lds, st, (const TT*)y,    \
                       (const TT*)x, (const TT*)Wp, (const TT*)Wg, Bp, Bg, (const TT*)res, (TT*)out, L, (int)C,    \
                       (int)C_out, ldy, cstride, eps);                                                            \
  } while (0)
    if (dtype == TOPS_DTYPE_BF16)
      TOPS_GEN_OUT_T(__bf16);
    else if (dtype == TOPS_DTYPE_F16)
      TOPS_GEN_OUT_T(_Float16);
    else if (dtype == TOPS_DTYPE_F32)
      TOPS_GEN_OUT_T(float);
    else
      return fail(TOPS_EUNSUPPORTED, "tops_tmu_output_phase: unsupported dtype code %d", dtype);
#undef TOPS_GEN_OUT_T
    return launched("tops_tmu_output_phase");
  }
  const int64_t blocks = (B * L * L + kGenTok - 1) / kGenTok;
  if (blocks == 0) return TOPS_OK;
  const size_t lds = (size_t)2 * kGenTok * C * sizeof(float);
#define TOPS_GEN_OUT(TT)                                                                                        hipLaunchKernelGGL((tmu_generic_out_kernel<TT>), dim3((unsigned)blocks), dim3(256), lds, st, (const TT*)y,                      (const TT*)x, (const TT*)Wp, (const TT*)Wg, Bp, Bg, (const TT*)res, (TT*)out, B, L, (int)C, (int)C_out, ldy, eps)
  if (dtype == TOPS_DTYPE_BF16)
    TOPS_GEN_OUT(__bf16);
  else if (dtype == TOPS_DTYPE_F16)
    TOPS_GEN_OUT(_Float16);
  else if (dtype == TOPS_DTYPE_F32)
    TOPS_GEN_OUT(float);
  else
    return fail(TOPS_EUNSUPPORTED, "tops_tmu_output_phase: unsupported dtype code %d", dtype);
#undef TOPS_GEN_OUT
  return launched("tops_tmu_output_phase");
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
