// gemm_rows.hip — products of at most 64 rows: a linear layer's X W^T (W stored N x K, "NT") or
// X W (W stored K x N, "NN") at a small batch, fp32 and fp16.
//
// Such a product is bound by reading W once. The tiled kernels streamed it from too few
// workgroups, with one K-tile pair in flight each (fp32 16 x 11008 x 4096: 3.0 TB/s), and
// products that neither split K nor fill tiles took a multiple of that (fp32 16 x 3000 x 2000: 0.5
// TB/s). Here a workgroup takes all rows (FM blocks of 16) and 16 FN columns, its KW waves take the K
// steps in turn, and each wave keeps D steps of W and X in registers: it multiplies the oldest
// and reloads its registers D steps ahead, so loads are always in flight. The waves' sums are
// added in LDS in wave order. A CU then reads 30 to 40 KB/us of W in the wide shapes whatever the
// depth (D = 2 to 4, 4 to 16 waves measured within 5%), the chip about 5 TB/s, so what matters is that
// the workgroups cover the CUs evenly: plan_rows picks FN, and S slices of K across workgroups
// (partial products, then the reduce of the split-K path), by that count.
//
// Fragments go from global memory into the MFMA source registers:
//  * NT: lane (i, g) loads 16 bytes of column i's row of W, k = E g .. E g + E - 1 of a KS-element
//    substep (fp32 E = 4, KS = 16; fp16 E = 8, KS = 32), two substeps of a 128-byte line in turn;
//  * NN: lane (i, g) loads FN consecutive columns FN i .. of one k row, so the 16 lanes of a k row read
//    16 FN elements in a run. Register n of those loads is column FN i + n: the MFMA's column i
//    of block n is column FN i + n of the tile, and no data moves between lanes. fp32: the loads of
//    k rows 4 g + s feed step s. fp16: the eight k rows 8 g .. 8 g + 7 are combined two by two with
//    v_perm (one per 4 bytes).
// X's fragments are loaded by every wave (16 bytes per lane; L2): with more columns per wave there are
// fewer of them.
//
// us on MI355X, W from HBM (before -> after): fp32 NT 16 x 11008 x 4096 59 -> 44, 16 x 5000 x 800 21 -> 9,
// 16 x 1024 x 4096 19.6 -> 11, 8 x 3000 x 2000 49 -> 10, 32 x 11008 x 4096 75 -> 53; NN 16 x 11008 x 4096
// 64 -> 41, 1 x 4096 x 4096 30 -> 20; fp16 NT 16 x 4096 x 1024 11.8 -> 5.5, NN 4 x 11008 x 4096 25 -> 20, 1 x
// 2048 x 8192 45 -> 14.
#include <algorithm>

#include "gemm_rows.h"
#include "gemm_tile.h"

namespace gn {
namespace {

template <typename T>
struct RowOps;
template <>
struct RowOps<float> {
  typedef float4_t V;
  static constexpr int E = 4, KS = 16, MPS = 4;
  static __device__ __forceinline__ float4_t mma(const V &a, const V &b, int s, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], b[s], c, 0, 0, 0);
  }
};
template <>
struct RowOps<_Float16> {
  typedef half8_t V;
  static constexpr int E = 8, KS = 32, MPS = 1;
  static __device__ __forceinline__ float4_t mma(const V &a, const V &b, int, float4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

template <typename T, int N>
struct VecOf {
  typedef T type __attribute__((ext_vector_type(N)));
};
template <>
struct VecOf<float, 1> {
  typedef float type;
};

// Steps of H substeps; XV: X's rows allow 16-byte loads. Rows past M and columns past N are
// clamped to the last ones (loaded, multiplied and not stored). NN: N and ldb are multiples of FN.
// NA: sums per element and wave; the substeps in flight take them in turn. An MFMA rounds its sum
// once per product, and where 4 or 8 waves share K one sum each lost up to half the precision the tiled
// kernels have in NN: fp32 4 x 11008 x 4096 5.7e-7 against 2.9e-7 relative to float64, now 2.9e-7 in the
// same time. FLUSH: with 17 to 32 rows there are no registers for that (28 spilled; two sums in AGPRs cost
// 10-20%), and the sum of each round of loads is added to a total instead (with fewer rows, or in the
// 8-wave shapes, that cost up to 20% where K is short). fp32 sums of 4 waves need the two waves per SIMD: the
// compiler then keeps them in VGPRs instead of copying them from AGPRs; fp16 loses 2-4% by it.
template <typename T, bool TB, int FM, int FN, int KW, int D, int H, bool XV>
__global__ void __launch_bounds__(KW * 64) __attribute__((amdgpu_waves_per_eu(KW > 4 ? KW / 4 : sizeof(T) == 4 && FM <= 2 ? 2 : 1)))
gemm_rows_kernel(GemmParams p, int S) {
  typedef RowOps<T> Ops;
  typedef typename Ops::V V;
  constexpr int E = Ops::E, KS = Ops::KS, STEP = KS * H, BN = 16 * FN;
  typedef typename VecOf<T, TB ? E : FN>::type WV;
  constexpr int NW = TB ? FN : E;  // W loads of a substep
  __shared__ float4_t red[KW][FM * FN][64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int li = lane & 15, lg = lane >> 4;
  // Workgroup w runs on XCD w % 8: each XCD takes a contiguous range of (slice, tile) pairs, so that
  // the tiles that share W's lines (NN tiles of 64 bytes) share an L2.
  const int tiles = gridDim.x, total = tiles * gridDim.z;
  int w0 = blockIdx.x + blockIdx.z * tiles;
  w0 = (w0 & 7) * (total >> 3) + min(w0 & 7, total & 7) + (w0 >> 3);
  const int z = w0 / tiles;
  const long n0 = (long)(w0 - z * tiles) * BN;
  const T *X = static_cast<const T *>(p.A), *W = static_cast<const T *>(p.B);
  const T *xp[FM], *wp[TB ? FN : 1];
#pragma unroll
  for (int m = 0; m < FM; ++m) xp[m] = X + min((long)(16 * m + li), p.M - 1) * p.lda + E * lg;
  if (TB) {
#pragma unroll
    for (int n = 0; n < FN; ++n) wp[TB ? n : 0] = W + min(n0 + 16 * n + li, p.N - 1) * p.ldb + E * lg;
  } else {
    wp[0] = W + min(n0 + FN * li, p.N - FN) + (long)(E * lg) * p.ldb;
  }
  V x[D][H][FM];
  WV w[D][H][NW];
  auto load_x = [&](const T *q) -> V {
    if (XV) return *reinterpret_cast<const V *>(q);
    V v;
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = q[e];
    return v;
  };
  auto load = [&](int d, long k) {
#pragma unroll
    for (int h = 0; h < H; ++h) {
#pragma unroll
      for (int j = 0; j < NW; ++j) {
        const T *q = TB ? wp[TB ? j : 0] + k + h * KS : wp[0] + (k + h * KS + j) * p.ldb;
        w[d][h][j] = *reinterpret_cast<const WV *>(q);
      }
#pragma unroll
      for (int m = 0; m < FM; ++m) x[d][h][m] = load_x(xp[m] + k + h * KS);
    }
  };
  constexpr int NA = FM > 1 || KW > 8 || (TB && (KW == 8 || sizeof(T) == 2)) ? 1 : !TB && KW == 4 && sizeof(T) == 4 ? 4 : 2;
  constexpr bool FLUSH = FM == 2 && KW == 4 && sizeof(T) == 4;
  static_assert(D * H % NA == 0, "the sums in turn");
  float4_t acc[NA][FM][FN];
#pragma unroll
  for (int q = 0; q < NA; ++q)
#pragma unroll
    for (int m = 0; m < FM; ++m)
#pragma unroll
      for (int n = 0; n < FN; ++n) acc[q][m][n] = float4_t{0.f, 0.f, 0.f, 0.f};
  float4_t flushed[FLUSH ? FM : 1][FLUSH ? FN : 1];
  if constexpr (FLUSH) {
#pragma unroll
    for (int m = 0; m < FM; ++m)
#pragma unroll
      for (int n = 0; n < FN; ++n) flushed[m][n] = float4_t{0.f, 0.f, 0.f, 0.f};
  }
  // B fragments of a substep: NT as loaded; NN fp32: register n of row j; NN fp16: the 8 rows' column n
  auto mul = [&](const V (&xs)[FM], const WV (&ws)[NW], float4_t (&c)[FM][FN]) {
    V b[FN];
    if constexpr (TB) {
#pragma unroll
      for (int n = 0; n < FN; ++n) b[n] = ws[n];
    } else if constexpr (sizeof(T) == 4) {
#pragma unroll
      for (int n = 0; n < FN; ++n)
#pragma unroll
        for (int e = 0; e < E; ++e) {
          if constexpr (FN == 1) b[n][e] = ws[e];
          else b[n][e] = ws[e][n];
        }
    } else {
      typedef uint32_t WU __attribute__((ext_vector_type(FN / 2 == 1 ? 2 : FN / 2)));
      typedef uint32_t BU __attribute__((ext_vector_type(4)));
      BU bu[FN];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        uint32_t lo[FN / 2], hi[FN / 2];
        if constexpr (FN == 2) {
          lo[0] = __builtin_bit_cast(uint32_t, ws[2 * q]);
          hi[0] = __builtin_bit_cast(uint32_t, ws[2 * q + 1]);
        } else {
          const WU a = __builtin_bit_cast(WU, ws[2 * q]), c = __builtin_bit_cast(WU, ws[2 * q + 1]);
#pragma unroll
          for (int n = 0; n < FN / 2; ++n) lo[n] = a[n], hi[n] = c[n];
        }
#pragma unroll
        for (int n = 0; n < FN / 2; ++n) {
          bu[2 * n][q] = __builtin_amdgcn_perm(hi[n], lo[n], 0x05040100);
          bu[2 * n + 1][q] = __builtin_amdgcn_perm(hi[n], lo[n], 0x07060302);
        }
      }
#pragma unroll
      for (int n = 0; n < FN; ++n) b[n] = __builtin_bit_cast(V, bu[n]);
    }
#pragma unroll
    for (int s = 0; s < Ops::MPS; ++s)
#pragma unroll
      for (int m = 0; m < FM; ++m)
#pragma unroll
        for (int n = 0; n < FN; ++n) c[m][n] = Ops::mma(xs[m], b[n], s, c[m][n]);
  };
  // the slice's whole steps [s0, s1); wave w takes s0 + w, s0 + w + KW, ...
  const long full = p.K / STEP, s0 = full * z / S, s1 = full * (z + 1) / S;
  const long mine = wave < s1 - s0 ? (s1 - s0 - wave + KW - 1) / KW : 0;
  const long k = (s0 + wave) * STEP;
  if (mine >= D) {
#pragma unroll
    for (int d = 0; d < D; ++d) load(d, k + (long)d * KW * STEP);
    long t = D;
    // multiply each buffer and reload it D steps ahead
    for (; t + D <= mine; t += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
#pragma unroll
        for (int h = 0; h < H; ++h) mul(x[d][h], w[d][h], acc[(d * H + h) % NA]);
        load(d, k + (t + d) * KW * STEP);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (FLUSH) {
#pragma unroll
        for (int m = 0; m < FM; ++m)
#pragma unroll
          for (int n = 0; n < FN; ++n) flushed[m][n] = flushed[m][n] + acc[0][m][n], acc[0][m][n] = float4_t{0.f, 0.f, 0.f, 0.f};
      }
    }
#pragma unroll
    for (int d = 0; d < D; ++d) {
#pragma unroll
      for (int h = 0; h < H; ++h) mul(x[d][h], w[d][h], acc[(d * H + h) % NA]);
      if (t + d < mine) load(d, k + (t + d) * KW * STEP);
    }
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (t + d < mine) {
#pragma unroll
        for (int h = 0; h < H; ++h) mul(x[d][h], w[d][h], acc[(d * H + h) % NA]);
      }
  } else {
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (d < mine) load(d, k + (long)d * KW * STEP);
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (d < mine) {
#pragma unroll
        for (int h = 0; h < H; ++h) mul(x[d][h], w[d][h], acc[(d * H + h) % NA]);
      }
  }
  // the last K % STEP: substep by substep, elements at or past K zero in both operands
  if (full * STEP < p.K && z == S - 1 && wave == (s1 - s0) % KW) {
    for (long kb = full * STEP; kb < p.K; kb += KS) {
      V xs[FM];
      WV ws[NW];
      const long kl = kb + E * lg;  // this lane's first k
#pragma unroll
      for (int m = 0; m < FM; ++m)
#pragma unroll
        for (int e = 0; e < E; ++e) xs[m][e] = kl + e < p.K ? xp[m][kb + e] : T(0);
#pragma unroll
      for (int j = 0; j < NW; ++j) {
        if constexpr (TB) {
#pragma unroll
          for (int e = 0; e < E; ++e) ws[j][e] = kl + e < p.K ? wp[j][kb + e] : T(0);
        } else {
          WV z;
          if constexpr (FN == 1 && sizeof(T) == 4) z = 0.0f;
          else {
#pragma unroll
            for (int n = 0; n < FN; ++n) z[n] = T(0);
          }
          ws[j] = z;
          if (kl + j < p.K) ws[j] = *reinterpret_cast<const WV *>(wp[0] + (kb + j) * p.ldb);
        }
      }
      mul(xs, ws, acc[NA - 1]);
    }
  }
#pragma unroll
  for (int m = 0; m < FM; ++m)
#pragma unroll
    for (int n = 0; n < FN; ++n) {
      float4_t v = acc[0][m][n];
#pragma unroll
      for (int q = 1; q < NA; ++q) v = v + acc[q][m][n];
      if constexpr (FLUSH) v = v + flushed[m][n];
      red[wave][m * FN + n][lane] = v;
    }
  __syncthreads();
  for (int f = wave; f < FM * FN; f += KW) {
    float4_t v = red[0][f][lane];
#pragma unroll
    for (int q = 1; q < KW; ++q) v = v + red[q][f][lane];
    const int n = f % FN, m = f / FN;
    const long col = TB ? n0 + 16 * n + li : n0 + FN * li + n, row0 = 16 * m + 4 * lg;
    if (col >= p.N) continue;
    const float bv = p.bias ? p.bias[col] : 0.0f;
    auto finish = [&](auto act_c) {
      constexpr int ACT = decltype(act_c)::value;
      const int act = ACT == kActRuntime ? p.act : ACT;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (row0 + e >= p.M) break;
        float *dst = p.C + z * p.strideC + (row0 + e) * p.ldc + col;
        const float old = p.beta != 0.0f ? *dst : 0.0f;
        *dst = apply_act(act, p.alpha * v[e] + p.beta * old + bv, p.act_alpha);
      }
    };
    switch (p.act) {
      case -1: finish(ActCode<-1>{}); break;
      case 0: finish(ActCode<0>{}); break;
      case 7: finish(ActCode<7>{}); break;
      default: finish(ActCode<kActRuntime>{}); break;
    }
  }
}

// ------------------------------------------------------------------ wide products of few k (GEMV)
// C = act(alpha X W + beta C + bias) for X of R <= 4 rows, W stored K x N: lane l of a workgroup owns
// columns n0 + E l .. + E - 1 (4 bytes of each row of W: 256 contiguous bytes by a wave); the KW waves
// split K into contiguous ranges, summed with fmaf on the VALU, and the partials are added in LDS as a
// tree (in wave order they lost more than the sums did). Bound by reading W, or, where W is short, by launch and the latency of one
// round of loads: nothing else is on the path, where gemm_rows_kernel needs K for its pipeline (it takes
// none below 256) and the tiled kernels 64 rows. us on MI355X, W in the caches (64 x 64 tiles or
// gemm_rows_kernel -> this): fp32 1 x 32768 x 255 17.4 -> 4.9, 4 x 65536 x 128 13.1 -> 7.3, 1 x 16384 x 512
// 5.4 -> 4.6; fp16 2 x 32768 x 128 5.4 -> 2.7, 1 x 65536 x 256 6.0 -> 4.2.
template <typename T, int R, int E, int KW>
__global__ void __launch_bounds__(KW * 64) gemv_nn_kernel(GemmParams p) {
  __shared__ float red[KW][R][64 * E];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const long nb = (long)blockIdx.x * 64 * E, n0 = nb + (long)lane * E;
  const T *__restrict__ W = static_cast<const T *>(p.B);
  const T *__restrict__ X = static_cast<const T *>(p.A);
  const long kb = p.K * wave / KW, ke = p.K * (wave + 1) / KW;
  float acc[R][E];
#pragma unroll
  for (int m = 0; m < R; ++m)
#pragma unroll
    for (int e = 0; e < E; ++e) acc[m][e] = 0.0f;
  if (n0 < p.N) {  // N is a multiple of E: the E columns are all inside or all past N
    typedef typename VecOf<T, E>::type VE;
    auto step = [&](long k) {
      const VE w = *reinterpret_cast<const VE *>(W + k * p.ldb + n0);
#pragma unroll
      for (int m = 0; m < R; ++m) {
        const float x = (float)X[m * p.lda + k];  // the same for the whole wave
        if constexpr (E == 1) {
          acc[m][0] = fmaf(x, (float)w, acc[m][0]);
        } else {
#pragma unroll
          for (int e = 0; e < E; ++e) acc[m][e] = fmaf(x, (float)w[e], acc[m][e]);
        }
      }
    };
    long k = kb;
    for (; k + 8 <= ke; k += 8) {
#pragma unroll
      for (int u = 0; u < 8; ++u) step(k + u);
    }
    for (; k < ke; ++k) step(k);
  }
#pragma unroll
  for (int m = 0; m < R; ++m)
#pragma unroll
    for (int e = 0; e < E; ++e) red[wave][m][lane * E + e] = acc[m][e];
  __syncthreads();
  for (int o = threadIdx.x; o < R * 64 * E; o += KW * 64) {
    const int m = o / (64 * E), c = o % (64 * E);
    const long n = nb + c;
    if (n >= p.N) continue;
    float v[KW];
#pragma unroll
    for (int w = 0; w < KW; ++w) v[w] = red[w][m][c];
#pragma unroll
    for (int h = KW / 2; h > 0; h /= 2)
#pragma unroll
      for (int w = 0; w < h; ++w) v[w] += v[w + h];
    float *dst = p.C + m * p.ldc + n;
    const float old = p.beta != 0.0f ? *dst : 0.0f;
    *dst = apply_act(p.act, p.alpha * v[0] + p.beta * old + (p.bias ? p.bias[n] : 0.0f), p.act_alpha);
  }
}

template <typename T, int R>
hipError_t launch_gemv_r(const GemmParams &p, hipStream_t s) {
  constexpr int E = sizeof(T) == 2 ? 2 : 1;  // 4 bytes per lane and row of W
  const unsigned grid = (unsigned)((p.N + 64 * E - 1) / (64 * E));
  hipLaunchKernelGGL((gemv_nn_kernel<T, R, E, 16>), dim3(grid), dim3(1024), 0, s, p);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_gemv_t(const GemmParams &p, hipStream_t s) {
  switch (p.M) {
    case 1: return launch_gemv_r<T, 1>(p, s);
    case 2: return launch_gemv_r<T, 2>(p, s);
    case 3: return launch_gemv_r<T, 3>(p, s);
    default: return launch_gemv_r<T, 4>(p, s);
  }
}

// ------------------------------------------------------------------ shapes
// Shape fn: NT 16, 32 or 48 columns; NN fp32 16, 32 or 64, fp16 32 or 64 (FN values). Waves and
// depths are the ones that measured best or within 3% of it: 16 waves of two steps for 16 NT columns
// (8 with 33-64 rows, which need the registers; 4 where plan_rows says so), 4 waves for the widest NN
// shapes.
template <typename T, bool TB, int FM, int FN, int KW, int D, bool XV, int H = 2>
hipError_t launch_shape(const GemmParams &p, int S, hipStream_t s) {
  const dim3 grid((unsigned)((p.N + 16 * FN - 1) / (16 * FN)), 1, (unsigned)S);
  hipLaunchKernelGGL((gemm_rows_kernel<T, TB, FM, FN, KW, D, H, XV>), grid, dim3(KW * 64), 0, s, p, S);
  return hipGetLastError();
}

template <typename T, int FM, bool XV>
hipError_t launch_nn(const GemmParams &p, int fn, int S, hipStream_t s) {
  if constexpr (sizeof(T) == 4) {
    if (fn == 1) return launch_shape<T, false, FM, 1, 8, FM <= 2 ? 4 : 2, XV>(p, S, s);
    if (fn == 2) return launch_shape<T, false, FM, 2, 8, 2, XV>(p, S, s);
    return launch_shape<T, false, FM, 4, 4, 2, XV>(p, S, s);
  } else {
    if (fn == 2) return launch_shape<T, false, FM, 2, 8, 2, XV>(p, S, s);
    return launch_shape<T, false, FM, 4, FM == 1 ? 4 : 8, 2, XV, FM <= 3 ? 2 : 1>(p, S, s);
  }
}

template <typename T, int FM>
hipError_t launch_fm(const GemmParams &p, bool tb, bool xv, int fn, bool few, int S, hipStream_t s) {
  if (tb) {
    if constexpr (FM == 1)
      if (few) return launch_shape<T, true, 1, 1, 4, 2, true>(p, S, s);
    if (fn == 1) return launch_shape<T, true, FM, 1, FM <= 2 ? 16 : 8, 2, true>(p, S, s);
    if (fn == 2) return launch_shape<T, true, FM, 2, 8, 2, true>(p, S, s);
    return launch_shape<T, true, FM, 3, 8, 2, true>(p, S, s);
  }
  if (xv) return launch_nn<T, FM, true>(p, fn, S, s);
  if constexpr (FM == 1) return launch_nn<T, FM, false>(p, fn, S, s);
  return hipErrorInvalidValue;  // plan_rows takes unaligned X up to 16 rows
}

template <typename T>
hipError_t launch_rows_t(const GemmParams &p, bool tb, bool xv, int fn, bool few, int S, hipStream_t s) {
  switch ((p.M + 15) / 16) {
    case 1: return launch_fm<T, 1>(p, tb, xv, fn, few, S, s);
    case 2: return launch_fm<T, 2>(p, tb, xv, fn, few, S, s);
    case 3: return launch_fm<T, 3>(p, tb, xv, fn, few, S, s);
    default: return launch_fm<T, 4>(p, tb, xv, fn, few, S, s);
  }
}

bool x_vectors(const GemmDesc &d) {
  const long e = d.dtype == GN_F16 ? 8 : 4;
  return (uintptr_t)d.A % 16 == 0 && d.lda % e == 0;
}

}  // namespace

bool plan_rows(const GemmDesc &d, bool split_ok, RowsPlan *out) {
  const bool f16 = d.dtype == GN_F16, beta = d.beta != 0.0f;
  const long e = f16 ? 8 : 4, esz = f16 ? 2 : 4;
  if (d.batch != 1 || d.ta || d.M > 64 || d.N < 256 || d.K < 256 || d.N > (1L << 30)) return false;
  if ((double)d.N * d.K < (double)(1L << 18)) return false;
  const bool xv = x_vectors(d);
  if (d.tb) {  // 16-byte loads along K for W and X
    if (!xv || (uintptr_t)d.B % 16 || d.ldb % e) return false;
  } else if (!xv && d.M > 16) {
    return false;
  }
  // Prices in us: a fixed part, the larger of the busiest CU's reading (W and X; rounds of 256
  // workgroups) and W at the chip's rate and a quarter of the other, a part of the fp32 MFMAs, and
  // the reduce. They follow the measured times of 220 shapes (1 to 64 rows, W of 256 K to 45 M
  // elements) within 20%; S > 1 has to be 5% ahead.
  const double fm = (double)((d.M + 15) / 16), xrows = std::min(16.0 * fm, (double)d.M) / 16.0;
  const double w_mb = (double)d.N * (double)d.K * esz / 1.0e6;
  out->us = 1e30;
  for (int fn = 1; fn <= 4; ++fn) {
    // KB/us one CU reads W at in this shape, and X's share: rows of X cost about what columns of W
    // do in NT, and a third of the tile's time per 16 rows in NN.
    // hbm (MB/us): NN tiles whose runs are shorter than two 128-byte lines get less of it.
    double rate, x, hbm = 5.2;
    if (d.tb) {
      if (fn > 3) continue;
      rate = f16 ? 31.0 + fn : 27.0 + 5.0 * fn;
      x = 0.95 * xrows;
    } else {
      if (fn == 3 || (f16 && fn == 1)) continue;
      if (d.N % fn || d.ldb % fn || (uintptr_t)d.B % (fn * esz)) continue;
      rate = f16 ? (fn == 2 ? 22.0 : 40.0) : fn == 1 ? 18.0 : fn == 2 ? 36.0 : 58.0;
      x = (f16 ? 0.26 : 0.33) * xrows * fn;
      if (fn < 4) hbm = f16 ? 3.5 : fn == 1 ? 3.7 : 4.4;
    }
    const long tiles = (d.N + 16 * fn - 1) / (16 * fn);
    for (int S = 1; S <= (split_ok ? 8 : 1); ++S) {
      if (S > 1 && d.K / S < 512) break;
      const double rounds = (double)((tiles * S + 255) / 256), ks = (double)d.K / S;
      const double cu = rounds * ks * 16.0 * (double)esz * (fn + x) / (rate * 1e3);
      // fp32 MFMAs: 2 cycles of the four SIMDs per 16 x 16 block and k; a third of them shows
      const double mfma = f16 ? 0.0 : 0.35 * rounds * ks * 2.0 * fm * fn / 2200.0;
      const double red = S > 1 ? 3.0 + (double)(S + 1 + (beta ? 1 : 0)) * (double)(d.M * d.N) * 4.0 / 5.0e6 : 0.0;
      const double w = w_mb / hbm, us = 3.0 + 0.3 * fm * fn + std::max(cu, w) + 0.25 * std::min(cu, w) + mfma + red;
      if (us < (S > 1 ? 0.95 : 1.0) * out->us) out->us = us, out->fn = fn, out->S = S;
    }
  }
  if (out->us >= 1e30) return false;
  // Many NT tiles of 16 columns with little K each: of 16 waves most have no step or one, and two
  // workgroups of them fill a CU, which then waits out one round of loads after another; eight of 4
  // waves do so at a time (16 waves -> 4, warm: fp16 1 x 65536 x 256 22.8 -> 7.2 us, 2 x 32768 x 512 11.3 -> 5.8,
  // 8 x 16384 x 1024 13.6 -> 9.8; fp32 1 x 32768 x 256 14.3 -> 7.2). With more K or rows level or slower
  // (fp16 16 x 16384 x 1024 9.4 -> 11.1).
  out->few = d.tb && d.N >= 4096 &&
             (f16 ? (d.K < 512 && (d.M <= 12 || (d.M <= 16 && (d.N < 16384 || d.N >= 65536)))) || (d.K < 1024 && d.M <= 8) || (d.K <= 1024 && (d.M <= 2 || (d.M <= 8 && d.N >= 8192)))
                  : (d.K < 512 && (d.M <= 4 || (d.M <= 8 && d.N >= 8192))) || (d.M <= 4 && d.N > 8192 && d.K < 1024));
  if (out->few) out->fn = 1, out->S = 1;
  out->part_bytes = out->S > 1 ? (size_t)out->S * splitk_stride(d.M, d.N) * sizeof(float) : 0;
  return true;
}

// Where gemv_nn_kernel beat the other kernels on a grid of 1 to 4 rows, N 256 to 65536 and K 16 to 8192
// (time over the best of theirs): K below 256 from N = 8192, 0.35-0.8 (N = 4096 0.9-1.2); fp32 to K = 1024
// the further N is from M K (1 x 16384 x 1024 0.95, 2 x 11008 x 384 0.91; 2 x 8192 x 512 1.2, 4 rows 0.9-1.1
// whatever the size), fp16 from N = 32768 (0.83-0.98; 16384 x 512 1.05-1.3).
bool takes_gemv(const GemmDesc &d, bool b_ok) {
  if (d.batch != 1 || d.ta || d.tb || d.M > 4 || !b_ok || d.N < 8192 || d.K > 1024 || d.N > (1L << 30)) return false;
  if (d.K < 256) return true;
  if (d.dtype == GN_F32) return d.M <= 3 && d.N >= 13 * d.M * d.K;
  return d.N >= (d.K < 384 ? 5120 * d.M : 32768);
}

hipError_t launch_gemv(const GemmDesc &d, hipStream_t s) {
  GemmParams p{};
  p.A = d.A; p.B = d.B; p.C = d.C;
  p.M = d.M; p.N = d.N; p.K = d.K;
  p.lda = d.lda; p.ldb = d.ldb; p.ldc = d.ldc;
  p.alpha = d.alpha; p.beta = d.beta;
  p.bias = d.bias;
  p.act = d.act; p.act_alpha = d.act_alpha;
  return d.dtype == GN_F16 ? launch_gemv_t<_Float16>(p, s) : launch_gemv_t<float>(p, s);
}

hipError_t launch_rows(const GemmDesc &d, const RowsPlan &plan, float *part, hipStream_t s) {
  GemmParams p{};
  p.A = d.A; p.B = d.B;
  p.M = d.M; p.N = d.N; p.K = d.K;
  p.lda = d.lda; p.ldb = d.ldb;
  if (plan.S == 1) {
    p.C = d.C;
    p.ldc = d.ldc;
    p.alpha = d.alpha; p.beta = d.beta;
    p.bias = d.bias;
    p.act = d.act; p.act_alpha = d.act_alpha;
  } else {
    p.C = part;
    p.ldc = d.N;
    p.strideC = splitk_stride(d.M, d.N);
    p.alpha = 1.0f;
    p.act = -1;
  }
  const bool xv = x_vectors(d);
  return d.dtype == GN_F16 ? launch_rows_t<_Float16>(p, d.tb, xv, plan.fn, plan.few, plan.S, s)
                           : launch_rows_t<float>(p, d.tb, xv, plan.fn, plan.few, plan.S, s);
}

}  // namespace gn
