// gemm_split.hip — large fp32 products on the bf16 matrix cores.
//
// The fp32 matrix cores' 157 TFLOP/s bound a large fp32 product (4096^3: 0.93 ms, the pipe 93%
// busy); the bf16 ones run at 16 times that rate. Every fp32 value v is the exact sum of three
// bf16 values, h = bf16(v), m = bf16(v - h), l = v - h - m (round to nearest: 8 + 8 + 8 bits with
// signs), and of the nine products of parts of a b six are computed in fp32 accumulators: hh, hm,
// mh, mm, hl, lh (Henry, Tang and Heinecke, "Leveraging the bfloat16 artificial intelligence datatype
// for higher-precision computations", ARITH 2019). The others are at most 2^-24 |a b| together (2^-27
// rms, of either sign): a sum of one term is up to 1.67 2^-24 off where the fp32 cores round it to
// 2^-24 (0.435 against 0.425 rms), sums of many come out closer. hh has
// an accumulator of its own: the other five are 2^-8 of it and less, so a sum over K = 4096 rounds
// at full size once per 32 k, where the fp32 cores do so every 4 k. Error against float64, N(0, 1)
// operands, relative Frobenius: 4096^3 4.0e-7 against 1.15e-6 on the fp32 cores, 2048^3 2.7e-7
// against 8.1e-7, 777 x 1234 x 4099 2.2e-7 against 5.1e-7 (with one accumulator 1.0e-6, 7.0e-7,
// 4.0e-7, at the same speed).
//
// Range: the packed parts are of x 2^16, so that the low parts of subnormals are whole bf16
// subnormals, and a product takes this way only when every |x| < 2^36 (for K up to 2^20 no sum of
// x 2^16 y 2^16 overflows). The pack kernel looks, and the product kernel in a B that it splits itself;
// otherwise, infinities and NaN included, the fp32 kernels enqueued behind them compute C (split_gate.h).
//
// Time, 4096^3 NN: 928 -> 605-620 us a call, 56 of them the pack (335 MB, 6 TB/s), about 5 the fp32 kernels
// that return at once; the product's 545-560 are 245-250 TFLOP/s, 1.5 PFLOP/s of bf16 products, which is the
// rate the board's power limit leaves the matrix cores.
#include <algorithm>

#include "gemm_split.h"
#include "gemm_tile.h"

namespace gn {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

// The split layout: for every 16 rows and 32 k the three parts, each 1 KiB in the order of one MFMA
// fragment (lane 16 g + i: row i, k = 8 g .. 8 g + 7). So a copy to LDS moves 1 KiB of consecutive
// bytes, a fragment read takes lane l's 16 bytes at 16 l (no bank conflicts, no swizzle), and the
// product kernel has one form for all layouts, alignments and odd sizes. Rows past the operand
// and k past K are zeros.
//
// One operand's way into it: rows x K values, element (r, k) at r * ld + k
// (kcontig) or k * ld + r.
struct PackSide {
  const float *src;
  char *dst;
  long rows, ld, sstride;  // sstride: elements between the operands of consecutive batches
  long dstride;            // bytes between their packed forms
  int kcontig, vec;
};

// What the product kernel needs beside GemmParams.
struct SplitArgs {
  long sa, sb;   // bytes between the packed operands of consecutive batches
  int nkt, S;    // K-tiles of 32, and the slices they are cut into
  int nra, nrb;  // 16-row blocks of A and of B
};

struct Parts {
  bf16x8_t p[3];
};

// Element e of the three parts of x; bad |= x is none that they hold.
__device__ __forceinline__ void split1(float x, Parts &o, int e, bool &bad) {
  bad |= !(fabsf(x) < kSplitMax);
  const float v = x * kSplitScale;
  const __bf16 h = (__bf16)v;
  const float r1 = v - (float)h;
  const __bf16 m = (__bf16)r1;
  const float r2 = r1 - (float)m;
  o.p[0][e] = h;
  o.p[1][e] = m;
  o.p[2][e] = (__bf16)r2;
}

__device__ __forceinline__ Parts split8(const float (&x)[8], bool &bad) {
  Parts o;
#pragma unroll
  for (int e = 0; e < 8; ++e) split1(x[e], o, e, bad);
  return o;
}

// One K-tile of 64 rows per workgroup: with two or four K-tiles a workgroup the large operands
// took as long, and the small ones longer (1024 x 1024: 13 against 9 us), for want of waves.
__global__ void __launch_bounds__(256) split_pack_kernel(PackSide a, PackSide b, long K, int nkt, int ya,
                                                         SplitGate *gate, unsigned long long seq) {
  const bool is_b = (int)blockIdx.y >= ya;
  const PackSide s = is_b ? b : a;
  const long y = is_b ? blockIdx.y - ya : blockIdx.y;
  const float *src = s.src + (long)blockIdx.z * s.sstride;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  // K-contiguous: wave w packs row block 4 y + w, lane (i, g) row i, k = 8 g .. 8 g + 7 of the
  // K-tile: a row's 128 bytes by four lanes. MN-contiguous: lane = row (64 of them), wave g takes
  // k = 8 g .. 8 g + 7: 256 bytes of a k row by the wave.
  const long r = s.kcontig ? y * 64 + wave * 16 + (lane & 15) : y * 64 + lane;
  const int g = s.kcontig ? lane >> 4 : wave;
  const long k = (long)blockIdx.x * 32 + 8 * g;
  const bool rin = r < s.rows;
  float x[8];
  if (s.kcontig) {
    const float *q = src + r * s.ld + k;
    if (s.vec && rin && k + 8 <= K) {
      const float4_t u = *reinterpret_cast<const float4_t *>(q), v = *reinterpret_cast<const float4_t *>(q + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = u[e], x[4 + e] = v[e];
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = (rin && k + e < K) ? q[e] : 0.0f;
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = (rin && k + e < K) ? src[(k + e) * s.ld + r] : 0.0f;
  }
  const long rb = r >> 4;
  if (rb * 16 >= s.rows) return;  // row blocks past the operand are not stored
  bool bad = false;
  const Parts o = split8(x, bad);
  char *d = s.dst + (long)blockIdx.z * s.dstride + (rb * nkt + blockIdx.x) * kSplitBlock + (g * 16 + (r & 15)) * 16;
#pragma unroll
  for (int q = 0; q < 3; ++q) *reinterpret_cast<bf16x8_t *>(d + q * 1024) = o.p[q];
  if (bad) __hip_atomic_store(&gate->packed, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// 16 bytes per lane from the buffer at voff + soff into LDS at lds + 16 * lane. Every offset is
// inside the packed operand: row blocks past its last are clamped to it, K-tiles past a slice
// are not copied.
__device__ __forceinline__ void dma16s(const BufRsrc &s, unsigned voff, unsigned soff, unsigned lds) {
  int saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %4\n\t"
      "buffer_load_dwordx4 %1, %2, %3 offen lds\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved)
      : "v"(voff), "s"(s.r), "s"(soff), "s"(lds)
      : "memory");
}

// C tile of BM x BN by WM x WN waves over the K-tiles of a slice; BSRC 0: both operands packed, else
// B is split here (see "A raw B"). Per 32-k tile a wave multiplies six
// pairs of part planes (FM x FN MFMAs each); a plane's fragments are read while the two products
// before its first use run, so at most five of the six planes are in registers beside the two
// accumulator sets: 239 of 256 registers with 64 x 64 per wave (all six: 254 and spills). The
// ring holds NS K-tiles; the one barrier per K-tile comes after the third product, when its last
// planes are in registers, and the copies of K-tile t + NS are issued behind it in two parts. Reading
// the next tile's planes together behind the barrier instead ran at 250 TFLOP/s (4096^3) where this
// order reaches 270; at 2048^3 215 against 244.
//  * 256 x 128, 8 waves of 64 x 64: fewest bytes per MFMA (24 LDS reads for 96; 72 KiB of copies per
//    workgroup and K-tile); 144 KiB of LDS;
//  * 128 x 128, 8 waves of 64 x 32: twice the tiles where those leave CUs idle (2048^3: 70 us
//    against 109); three ring slots measured 1-2% slower than two.
template <int BM, int BN, int WM, int WN, int BSRC, int RD>
__global__ void __launch_bounds__(WM * WN * 64) __attribute__((amdgpu_waves_per_eu(2, 2)))
gemm_split_kernel(GemmParams p, SplitArgs q) {
  constexpr int NW = WM * WN, FM = BM / WM / 16, FN = BN / WN / 16, NS = 2;
  constexpr int CA = BM / 16 * 3, CB = BN / 16 * 3;  // 1 KiB chunks of a K-tile of A and of B
  constexpr int IPA = CA / NW, IPB = BSRC ? 0 : CB / NW, LPW = IPA + IPB;
  static_assert(RD == 1 || RD == 2, "raw buffers");
  static_assert(BSRC == 0 || (BN == 128 && NW == 8), "a raw B: one 16-column block, or 64 columns x 8 k, per wave");
  constexpr int SLOT = (CA + CB) * 1024;
  static_assert(CA % NW == 0 && CB % NW == 0, "tile shape");
  static_assert(WM * 16 * (BN + 4) * 4 <= NS * SLOT, "epilogue staging exceeds the ring");
  __shared__ __attribute__((aligned(1024))) char smem[NS * SLOT];
  if (split_product_skipped(*p.gate, p.gate_seq)) return;  // uniform: no workgroup of this launch writes that word
  int tm, tn;
  tile_coords(p, tm, tn);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wm = wave / WN, wn = wave % WN;
  const int z = blockIdx.z, zb = z / q.S, sl = z - zb * q.S;
  const int kt0 = (int)((long)sl * q.nkt / q.S), kt1 = (int)((long)(sl + 1) * q.nkt / q.S);
  const int nt = kt1 - kt0;
  const long m0 = (long)tm * BM, n0 = (long)tn * BN;
  const BufRsrc ra = make_rsrc(static_cast<const char *>(p.A) + zb * q.sa);
  const BufRsrc rb = make_rsrc(static_cast<const char *>(p.B) + zb * q.sb);
  const unsigned sbase = lds_offset(smem);
  const unsigned voff = lane * 16;
  unsigned soa[IPA], sob[IPB ? IPB : 1];
#pragma unroll
  for (int i = 0; i < IPA; ++i) {
    const int c = wave * IPA + i, blk = min((int)(m0 >> 4) + c / 3, q.nra - 1);
    soa[i] = (unsigned)blk * (unsigned)q.nkt * kSplitBlock + (unsigned)kt0 * kSplitBlock + (c % 3) * 1024;
  }
#pragma unroll
  for (int i = 0; i < IPB; ++i) {
    const int c = wave * IPB + i, blk = min((int)(n0 >> 4) + c / 3, q.nrb - 1);
    sob[i] = (unsigned)blk * (unsigned)q.nkt * kSplitBlock + (unsigned)kt0 * kSplitBlock + (c % 3) * 1024;
  }
  // part h of 2 of the wave's copies of K-tile t
  auto issue = [&](int t, int slot, int h) {
    const unsigned st = sbase + slot * SLOT, ko = (unsigned)t * kSplitBlock;
#pragma unroll
    for (int i = 0; i < IPA; ++i)
      if (2 * i / LPW == h)
        dma16s(ra, voff, __builtin_amdgcn_readfirstlane(soa[i] + ko),
               __builtin_amdgcn_readfirstlane(st + (wave * IPA + i) * 1024));
#pragma unroll
    for (int i = 0; i < IPB; ++i)
      if (2 * (IPA + i) / LPW == h)
        dma16s(rb, voff, __builtin_amdgcn_readfirstlane(sob[i] + ko),
               __builtin_amdgcn_readfirstlane(st + (CA + wave * IPB + i) * 1024));
  };
  // A raw B (BSRC 1: K-contiguous, rows of whole 16-byte vectors; 2: N-contiguous): a thread loads
  // eight k of one column of a K-tile into registers, NS + RD K-tiles ahead of their multiplication,
  // and writes their parts into the slot NS K-tiles ahead of it. Every K-tile takes RAW
  // unconditional load instructions, which the waits count on: columns past N are the last
  // one's (multiplied and not stored), k past K is some k before it (A's parts are zero there).
  constexpr int RAW = BSRC == 1 ? 2 : 8;
  constexpr bool MIX = FM * FN <= 8;  // the splits run beside MFMAs where the registers allow it
  const int bg = BSRC == 1 ? lane >> 4 : wave >> 1, bcol = BSRC == 1 ? wave * 16 + (lane & 15) : (wave & 1) * 64 + lane;
  const float *bsrc = static_cast<const float *>(p.B) + zb * p.strideB;
  const long blane = min(n0 + bcol, p.N - 1) * (BSRC == 1 ? p.ldb : 1);
  float raw[RD][8];
  bool bad = false;
  auto load_raw = [&](int r, int t) {
    const long k = (long)(kt0 + t) * 32 + 8 * bg;
    if (BSRC == 1) {
      const float4_t u = *reinterpret_cast<const float4_t *>(bsrc + blane + min(k, p.K - 4));
      const float4_t v = *reinterpret_cast<const float4_t *>(bsrc + blane + min(k + 4, p.K - 4));
#pragma unroll
      for (int e = 0; e < 4; ++e) raw[r][e] = u[e], raw[r][4 + e] = v[e];
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) raw[r][e] = bsrc[min(k + e, p.K - 1) * p.ldb + blane];
    }
  };
  Parts parts;
  auto split_raw = [&](int r, int e0, int e1) {
#pragma unroll
    for (int e = e0; e < e1; ++e) split1(raw[r][e], parts, e, bad);
  };
  auto write_raw = [&](int slot) {
    char *d = smem + slot * SLOT + (CA + (bcol >> 4) * 3) * 1024 + (bg * 16 + (bcol & 15)) * 16;
#pragma unroll
    for (int h = 0; h < 3; ++h) *reinterpret_cast<bf16x8_t *>(d + h * 1024) = parts.p[h];
  };
  bf16x8_t fa[FM][3], fb[FN][3];
  auto read_a = [&](int slot, int h) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
      fa[i][h] = *reinterpret_cast<const bf16x8_t *>(smem + slot * SLOT + ((wm * FM + i) * 3 + h) * 1024 + lane * 16);
  };
  auto read_b = [&](int slot, int h) {
#pragma unroll
    for (int j = 0; j < FN; ++j)
      fb[j][h] = *reinterpret_cast<const bf16x8_t *>(smem + slot * SLOT + (CA + (wn * FN + j) * 3 + h) * 1024 + lane * 16);
  };
  float4_t acc[FM][FN], low[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = low[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
  auto mul = [&](int ha, int hb) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        float4_t &c = ha + hb > 0 ? low[i][j] : acc[i][j];
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i][ha], fb[j][hb], c, 0, 0, 0);
      }
  };
#pragma unroll
  for (int u = 0; u < NS; ++u)
    if (u < nt) {
      issue(u, u, 0);
      issue(u, u, 1);
      if (BSRC) {
        load_raw(0, u);
        split_raw(0, 0, 8);
        write_raw(u);
      }
    }
#pragma unroll
  for (int r = 0; BSRC && r < RD; ++r) load_raw(r, NS + r);
  if (BSRC) __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
  else if (nt >= NS) __builtin_amdgcn_s_waitcnt(vmcnt_imm((NS - 1) * LPW));
  else __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
  __syncthreads();
  read_b(0, 1);
  read_a(0, 1);
  read_b(0, 2);
  int cur = 0;
  auto step = [&](int t, int r) {  // r: the raw buffer of K-tile t + NS
    const int nxt = cur ^ 1;
    const bool more = t + NS < nt;
    __builtin_amdgcn_sched_barrier(0);
    read_a(cur, 0);
    mul(1, 1);
    sched_interleave<FM * FN, FM>();
    __builtin_amdgcn_sched_barrier(0);
    read_b(cur, 0);
    mul(0, 1);
    sched_interleave<FM * FN, FN>();
    __builtin_amdgcn_sched_barrier(0);
    read_a(cur, 2);
    mul(0, 2);
    sched_interleave<FM * FN, FM>();
    __builtin_amdgcn_sched_barrier(0);
    // the copies of K-tile t + 1; a raw B's newest loads, issued behind them, may still be in flight
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(BSRC ? RAW : 0));
    __syncthreads();
    if (BSRC) {
      // raw[r] is waited for here: behind the next copies the compiler's wait would be for those too
#pragma unroll
      for (int e = 0; e < 8; ++e) asm volatile("" : "+v"(raw[r][e]));
    }
    __builtin_amdgcn_sched_barrier(0);
    if (more) issue(t + NS, cur, 0);
    __builtin_amdgcn_sched_barrier(0);
    read_b(nxt, 1);
    if (BSRC && MIX) split_raw(r, 0, 4);
    mul(2, 0);
    if (BSRC && MIX) sched_mix<FM * FN, FN>();
    else sched_interleave<FM * FN, FN>();
    __builtin_amdgcn_sched_barrier(0);
    if (more) issue(t + NS, cur, 1);
    if (BSRC && !MIX) {
      split_raw(r, 0, 8);
      write_raw(cur);
    }
    __builtin_amdgcn_sched_barrier(0);
    read_b(nxt, 2);
    if (BSRC && MIX) {
      split_raw(r, 4, 8);
      write_raw(cur);
    }
    mul(1, 0);
    if (BSRC && MIX) sched_mix<FM * FN, FN>();
    else sched_interleave<FM * FN, FN>();
    __builtin_amdgcn_sched_barrier(0);
    if (BSRC) load_raw(r, t + NS + RD);
    __builtin_amdgcn_sched_barrier(0);
    read_a(nxt, 1);
    mul(0, 0);
    sched_interleave<FM * FN, FM>();
    cur = nxt;
  };
  if constexpr (BSRC && RD == 2) {
    int t = 0;
    for (; t + 1 < nt; t += 2) {
      step(t, 0);
      step(t + 1, 1);
    }
    if (t < nt) step(t, 0);
  } else {
    for (int t = 0; t < nt; ++t) step(t, 0);
  }
  __syncthreads();
  if (BSRC && bad) __hip_atomic_store(&p.gate->multiplied, p.gate_seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = (acc[i][j] + low[i][j]) * (1.0f / (kSplitScale * kSplitScale));
  store_tile_rows<BM, BN, WM, WN>(p, m0, n0, z, reinterpret_cast<float *>(smem), acc);
}

template <int BM, int BN, int WM, int WN, int BSRC = 0, int RD = 1>
hipError_t launch_tile(GemmParams p, const SplitArgs &q, long batch, hipStream_t s) {
  p.tiles_m = (int)((p.M + BM - 1) / BM);
  p.tiles_n = (int)((p.N + BN - 1) / BN);
  const dim3 grid((unsigned)(p.tiles_m * p.tiles_n), 1, (unsigned)(batch * q.S));
  hipLaunchKernelGGL((gemm_split_kernel<BM, BN, WM, WN, BSRC, RD>), grid, dim3(WM * WN * 64), 0, s, p, q);
  return hipGetLastError();
}

hipError_t launch_shape(const SplitPlan &plan, int bsrc, const GemmParams &p, const SplitArgs &q, long batch,
                        hipStream_t s) {
  if (bsrc == 1)
    return plan.tile == 0 ? launch_tile<256, 128, 4, 2, 1, 1>(p, q, batch, s) : launch_tile<128, 128, 2, 4, 1, 2>(p, q, batch, s);
  if (bsrc == 2)
    return plan.tile == 0 ? launch_tile<256, 128, 4, 2, 2, 1>(p, q, batch, s) : launch_tile<128, 128, 2, 4, 2, 2>(p, q, batch, s);
  return plan.tile == 0 ? launch_tile<256, 128, 4, 2>(p, q, batch, s) : launch_tile<128, 128, 2, 4>(p, q, batch, s);
}

long blocks16(long n) { return (n + 15) / 16; }

bool vectors(const void *ptr, long ld, long stride, long batch) {
  return (uintptr_t)ptr % 16 == 0 && ld % 4 == 0 && (batch == 1 || stride % 4 == 0);
}

}  // namespace

bool plan_split(const GemmDesc &d, long nb, long kc, SplitPlan *out) {
  const long M = d.M, N = d.N, K = kc, batch = nb, nkt = (K + 31) / 32;
  const bool beta = d.beta != 0.0f || kc < d.K;
  const long last_k = d.K - (d.K - 1) / kc * kc;  // of the last part
  if (K < 32 || K > kSplitMaxK || batch > 16384 || (M + 63) / 64 + (N + 63) / 64 > 65535) return false;
  const size_t pa = (size_t)blocks16(M) * nkt * kSplitBlock, pb = (size_t)blocks16(N) * nkt * kSplitBlock;
  if (pa >= ring::kNumRecords) return false;  // 32-bit copy offsets
  // Prices in us, fitted to 44 shapes (64 x 8192 x 8192 to 8192 x 8192 x 128, both tiles, S 1-16) and 13
  // with a raw B, within 15%: the packing at 4.6 TB/s, a round of 256 workgroups at a fixed part (launch,
  // first copies, the store of C) plus its K-tiles, which cost more the more CUs share the board's
  // power, and the reduce. Slices keep at least 8 K-tiles. A raw B saves its packing (10 bytes per
  // element) and costs a 256-row tile's K-tile about a tenth, a 128-row tile's half as much again: it
  // pays for up to about 512 rows (512 x 11008 x 4096 NT 323 -> 250 us, 256 rows 217 -> 156; 1024 x 4096 x
  // 1024: level). It reads 16-byte vectors of a K-contiguous B, in every batch and part (kc is a
  // multiple of 32, or K).
  const bool raw_ok = d.tb ? vectors(d.B, d.ldb, d.strideB, d.batch) && d.K % 4 == 0 : true;
  // A K-contiguous operand off 16 bytes is packed element by element: past what the caches hold its packing
  // takes 1.6 times as long (17 x 130 x 2567 x 2071 TT 594 us where 411 were priced and the fp32 cores take 466).
  const bool odd_a = !d.ta && !vectors(d.A, d.lda, d.strideA, d.batch), odd_b = d.tb && !vectors(d.B, d.ldb, d.strideB, d.batch);
  out->us = 1e30;
  for (int form = 0; form < 4; ++form) {
    const int tile = form & 1;
    const bool raw = form >= 2;
    if (raw ? !raw_ok : pb >= ring::kNumRecords) continue;
    const double packed_mb = 6.0e-6 * (double)batch * (double)(M + (raw ? 0 : N)) * (double)K;
    const double a_bytes = odd_a && packed_mb > 100.0 ? 16.0 : 10.0, b_bytes = odd_b && packed_mb > 100.0 ? 16.0 : 10.0;
    const double pack_us = 3.0 + (double)batch * (a_bytes * (double)M + (raw ? 0.0 : b_bytes * (double)N)) * (double)K / 4.6e6;
    const double w_us = raw ? (double)batch * (double)N * (double)K * 4.0 / 4.9e6 : 0.0;
    const long bm = tile == 0 ? 256 : 128;
    const long tiles = ((M + bm - 1) / bm) * ((N + 127) / 128) * batch;
    if (tiles > (1L << 30)) return false;
    for (long S = 1; S <= (batch == 1 ? 32 : 1) && S <= nkt; ++S) {
      if (S > 1 && nkt / S < 8) break;
      // a raw B without slices writes C before its values are known: not where C counts, in any part
      if (raw && beta && std::min(S, (last_k + 31) / 32) == 1) continue;
      const long w = tiles * S, rounds = (w + 255) / 256;
      const double kt = (double)((nkt + S - 1) / S), busy = (double)w / (256.0 * (double)rounds);
      const double wg = raw ? (tile == 0 ? 10.0 + (1.75 + 0.6 * busy) * kt : 8.0 + 1.36 * kt)
                            : tile == 0 ? 9.0 + (1.54 + 0.36 * busy) * kt : 8.0 + (0.66 + 0.26 * busy) * kt;
      const double us = pack_us + std::max((double)rounds * wg, w_us) +
                        (S > 1 ? 2.5 + (double)(S + 1 + (beta ? 1 : 0)) * (double)(M * N) * 4.0 / 5.0e6 : 0.0);
      if (us < out->us) out->us = us, out->tile = tile, out->S = (int)S, out->raw_b = raw;
    }
  }
  if (out->us >= 1e30) return false;
  out->pack_bytes = (size_t)batch * (pa + (out->raw_b ? 0 : pb));
  out->part_bytes = out->S > 1 ? (size_t)out->S * splitk_stride(M, N) * sizeof(float) : 0;
  return true;
}

hipError_t launch_split(const GemmDesc &d, const SplitPlan &plan, char *ws, float *part, SplitGate *gate,
                        unsigned long long seq, hipStream_t s) {
  SplitArgs q{};
  q.nkt = (int)((d.K + 31) / 32);
  q.S = plan.S;
  q.nra = (int)blocks16(d.M);
  q.nrb = (int)blocks16(d.N);
  q.sa = (long)q.nra * q.nkt * kSplitBlock;
  q.sb = (long)q.nrb * q.nkt * kSplitBlock;
  char *pb = ws + d.batch * q.sa;
  const PackSide a{static_cast<const float *>(d.A), ws, d.M, d.lda, d.strideA, q.sa, !d.ta,
                   vectors(d.A, d.lda, d.strideA, d.batch)};
  const PackSide b{static_cast<const float *>(d.B), pb, d.N, d.ldb, d.strideB, q.sb, d.tb,
                   vectors(d.B, d.ldb, d.strideB, d.batch)};
  const int ya = (int)((d.M + 63) / 64), yb = plan.raw_b ? 0 : (int)((d.N + 63) / 64);
  hipLaunchKernelGGL(split_pack_kernel, dim3((unsigned)q.nkt, (unsigned)(ya + yb), (unsigned)d.batch), dim3(256), 0, s,
                     a, b, d.K, q.nkt, ya, gate, seq);
  if (hipError_t e = hipGetLastError()) return e;
  GemmParams p{};
  p.A = ws;
  p.B = plan.raw_b ? d.B : pb;
  p.ldb = d.ldb;
  p.strideB = d.strideB;
  p.M = d.M;
  p.N = d.N;
  p.K = d.K;
  p.gate = gate;
  p.gate_seq = seq;
  if (plan.S == 1) {
    p.C = d.C;
    p.ldc = d.ldc;
    p.strideC = d.strideC;
    p.alpha = d.alpha;
    p.beta = d.beta;
    p.bias = d.bias;
    p.act = d.act;
    p.act_alpha = d.act_alpha;
  } else {
    p.C = part;
    p.ldc = d.N;
    p.strideC = splitk_stride(d.M, d.N);
    p.alpha = 1.0f;
    p.act = -1;
  }
  return launch_shape(plan, plan.raw_b ? (d.tb ? 1 : 2) : 0, p, q, d.batch, s);
}

}  // namespace gn
