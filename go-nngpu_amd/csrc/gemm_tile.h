// gemm_tile.h — what the GEMM kernels share (gemm.hip, gemm_split.hip): the kernel parameters,
// the row-order epilogue, the XCD-aware tile order and the LDS-direct copies.
#pragma once

#include "act.h"
#include "common.h"
#include "ring_plan.h"
#include "split_gate.h"

namespace gn {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef __fp16 trh4_t __attribute__((__vector_size__(4 * sizeof(__fp16))));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));

#define LDS_AS __attribute__((address_space(3)))
#define CONST_AS __attribute__((address_space(4)))

struct GemmParams {
  const void *A;
  const void *B;
  float *C;
  const float *bias;
  long M, N, K;
  long lda, ldb, ldc;
  long strideA, strideB, strideC;
  float alpha, beta, act_alpha;
  int act;
  int tiles_m, tiles_n;
  int group_m;  // tile rows per raster group (tile_coords); 0 selects the default of 4
  // An fp32 product on the bf16 matrix cores (gemm_split.hip) and its fp32 kernels are both
  // enqueued; the gate says whose result counts (split_gate.h). The fp32 kernels (GATED) return at
  // once where the split's does.
  SplitGate *gate;
  unsigned long long gate_seq;
  int slices, nz;  // GATED: slices of K per batch; batch x slices
};

// False in an fp32 kernel that stands behind a split product whose operands allowed it.
__device__ __forceinline__ bool fp32_needed(const GemmParams &p) { return split_fp32_needed(*p.gate, p.gate_seq); }

// p for slice z % slices of K of batch z / slices, cut as the split product's slices are (whole 32-k
// tiles), so that its partial products take the places of the split's.
template <bool TA, bool TB>
__device__ __forceinline__ GemmParams slice_of(GemmParams p, int z) {
  const int S = p.slices, zb = z / S, sl = z - zb * S, nkt = (int)((p.K + 31) / 32);
  const long k0 = (long)sl * nkt / S * 32, k1 = min((long)(sl + 1) * nkt / S * 32, p.K);
  p.A = static_cast<const float *>(p.A) + zb * p.strideA + (TA ? k0 * p.lda : k0);
  p.B = static_cast<const float *>(p.B) + zb * p.strideB + (TB ? k0 : k0 * p.ldb);
  p.strideA = p.strideB = 0;
  p.K = k1 - k0;
  return p;
}

// ------------------------------------------------------------------ epilogue
// Workgroup barrier that orders LDS accesses only (s_waitcnt lgkmcnt(0); s_barrier).
// __syncthreads() also waits for vmcnt(0), i.e. for every global store the wave has
// issued to complete, which between the epilogue's passes serialised each pass behind
// the previous pass's C writes.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int V>
struct ActCode {
  static constexpr int value = V;
};
constexpr int kActRuntime = -1000;  // ActCode value: apply p.act, decided per element

// Writes a workgroup's BM x BN accumulator tile to C in row order. Pass f stages MFMA
// block-row f of every wave (WM x 16 tile rows, all BN columns) in LDS at `stg` (pitch
// BN + 4 floats: the 4 row groups of one ds_write_b32 fall on distinct banks), then the
// workgroup stores those rows as 16-byte vectors with consecutive lanes along a row, so
// each store instruction writes long contiguous row segments (one whole 1 KiB row at
// BN = 256). All CUs write their tiles at about the same time; when each wave stored
// only its own 256-byte row pieces (rows 32 KiB apart), the writes drained so slowly
// that the 8192^3 GEMM took 11% longer (4096^3: 17%). Each thread owns one column quad
// for the whole epilogue, so its bias values are loaded once, before the first pass: a
// load inside the passes would wait for all earlier stores (vmcnt counts stores too).
// The passes are separated by LDS-only barriers, so the stores of one pass drain while
// the next is staged. alpha, beta*C, bias and the activation are applied on the way;
// scalar stores at ragged edges or when ldc / C do not allow aligned 16-byte stores.
// The pass loop is unrolled so every accumulator index is static (a runtime index would
// move the accumulators to scratch memory). stage(f) writes the wave's rows of pass f (wave
// tile rows 16 f .. 16 f + 15) into stg at rows wm * 16 + 0..15, pitch BN + 4, columns
// wn * (BN / WN) + 0..BN / WN - 1.
template <int BM, int BN, int WM, int WN, typename Stage>
__device__ __forceinline__ void store_tile_passes(const GemmParams &p, long m0, long n0, long z, float *stg,
                                                  Stage &&stage) {
  constexpr int WTM = BM / WM, FM = WTM / 16;
  constexpr int LP = BN + 4, CPR = BN / 4, NTH = WM * WN * 64;
  constexpr int ROWS = WM * 16;       // tile rows staged per pass
  constexpr int RPS = NTH / CPR;      // rows one sweep of the workgroup's threads covers
  constexpr int SWEEPS = (ROWS + RPS - 1) / RPS;
  static_assert(BN % 4 == 0 && CPR <= NTH, "row vectors");
  const int c4 = threadIdx.x % CPR, r0 = threadIdx.x / CPR;  // threads with r0 >= RPS only stage
  const long col = n0 + 4 * c4;
  float *C = p.C + z * p.strideC;
  const bool vec = (p.ldc % 4 == 0) && (((uintptr_t)C & 15) == 0) && col + 3 < p.N;
  float bv[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) bv[e] = (p.bias && col + e < p.N) ? p.bias[col + e] : 0.0f;
#pragma unroll
  for (int f = 0; f < FM; ++f) {
    lds_barrier();  // the previous pass (or the main loop) is done with stg
    stage(f);
    lds_barrier();
    // The common activations get their own copy of the row sweep with the code fixed at
    // compile time: the generic one inlines every case of apply_act for every element,
    // and that long branchy code cost 3.5 us per launch at 512 x 11008 x 512 (ReLU).
    auto sweep = [&](auto act_c) {
      constexpr int ACT = decltype(act_c)::value;
      const int act = ACT == kActRuntime ? p.act : ACT;
      // a runtime loop: unrolling it as well made the pass loop too large to unroll
      // fully (the 256 x 256 kernels then kept the accumulators in scratch memory)
#pragma unroll 1
      for (int s = 0; s < SWEEPS; ++s) {
        const int t = r0 + s * RPS;
        if (r0 >= RPS || t >= ROWS) continue;
        const long row = m0 + (t / 16) * WTM + f * 16 + (t % 16);
        if (row >= p.M) continue;
        const float4_t v = *reinterpret_cast<const float4_t *>(stg + t * LP + 4 * c4);
        float *dst = C + row * p.ldc + col;
        if (vec) {
          float4_t o;
          const float4_t old =
              p.beta != 0.0f ? *reinterpret_cast<const float4_t *>(dst) : float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = apply_act(act, p.alpha * v[e] + p.beta * old[e] + bv[e], p.act_alpha);
          __builtin_nontemporal_store(o, reinterpret_cast<float4_t *>(dst));  // C is not re-read: keep L2 for A/B
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (col + e < p.N) {
              float x = p.alpha * v[e];
              if (p.beta != 0.0f) x += p.beta * dst[e];
              dst[e] = apply_act(act, x + bv[e], p.act_alpha);
            }
          }
        }
      }
    };
    switch (p.act) {
      case -1: sweep(ActCode<-1>{}); break;
      case 0: sweep(ActCode<0>{}); break;
      case 7: sweep(ActCode<7>{}); break;
      default: sweep(ActCode<kActRuntime>{}); break;
    }
  }
}

// store_tile_passes for 16 x 16 MFMA accumulators: lane (c, g) of block (f, j) holds rows
// 4 g + 0..3 of column c.
template <int BM, int BN, int WM, int WN>
__device__ __forceinline__ void store_tile_rows(const GemmParams &p, long m0, long n0, long z, float *stg,
                                                const float4_t (&acc)[BM / WM / 16][BN / WN / 16]) {
  constexpr int WTN = BN / WN, FN = WTN / 16, LP = BN + 4;
  const int wave = threadIdx.x >> 6, wm = wave / WN, wn = wave % WN, lane = threadIdx.x & 63;
  const int c = lane & 15, g = lane >> 4;
  store_tile_passes<BM, BN, WM, WN>(p, m0, n0, z, stg, [&](int f) {
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) stg[(wm * 16 + 4 * g + r) * LP + wn * WTN + 16 * j + c] = acc[f][j][r];
  });
}

// Grouped + XCD-aware mapping of the linear workgroup id w to a (tile_m, tile_n) pair.
__device__ __forceinline__ void tile_coords(const GemmParams &p, int w, int &tm, int &tn) {
  // Workgroup w runs on XCD w % 8; give XCD x the contiguous tile range
  // [x*base + min(x, rem), ...) of base (+1 for the first rem XCDs) tiles.
  const int total = p.tiles_m * p.tiles_n;
  {
    const int base = total >> 3, rem = total & 7, x = w & 7;
    w = x * base + min(x, rem) + (w >> 3);
  }
  const int GROUP_M = p.group_m > 0 ? p.group_m : 4;
  const int in_group = GROUP_M * p.tiles_n;
  const int group = w / in_group;
  const int first_m = group * GROUP_M;
  const int gsize = min(p.tiles_m - first_m, GROUP_M);
  const int r = w - group * in_group;
  tm = first_m + r % gsize;
  tn = r / gsize;
}
__device__ __forceinline__ void tile_coords(const GemmParams &p, int &tm, int &tn) { tile_coords(p, blockIdx.x, tm, tn); }

// A GATED kernel's tiles, body(p of the slice, tile, z) for each: its workgroups, at most
// kGatedGrid, take them in turn. An empty workgroup costs about a nanosecond of a product whose
// split counts (512 x 4096 x 11008: 2048 of them 4 us).
constexpr int kGatedGrid = 512;
template <bool TA, bool TB, typename Body>
__device__ __forceinline__ void gated_tiles(const GemmParams &p, Body &&body) {
  if (!fp32_needed(p)) return;
  // The kernel's arguments (p is the only one), read again for every tile: kept beside a tile's own
  // they take more scalar registers than there are.
  auto *args = (const CONST_AS GemmParams *)__builtin_amdgcn_kernarg_segment_ptr();
  for (long u = blockIdx.x;; u += gridDim.x) {
    asm volatile("" : "+s"(args));
    const GemmParams q = *(const GemmParams *)args;
    const int tiles = q.tiles_m * q.tiles_n, z = (int)(u / tiles);
    if (z >= q.nz) return;
    body(slice_of<TA, TB>(q, z), (int)(u - (long)z * tiles), z);
    __syncthreads();  // before the next tile's copies into LDS
  }
}

typedef int i32x4_t __attribute__((ext_vector_type(4)));

struct BufRsrc {
  i32x4_t r;
};

// Raw buffer descriptor: 48-bit base, stride 0, num_records ring::kNumRecords (offsets at
// or beyond it read as zero), gfx9 dword3.
__device__ __forceinline__ BufRsrc make_rsrc(const void *base) {
  const unsigned long long b = (unsigned long long)base;
  BufRsrc s;
  s.r.x = __builtin_amdgcn_readfirstlane((int)(b & 0xffffffffu));
  s.r.y = __builtin_amdgcn_readfirstlane((int)(b >> 32) & 0xffff);
  s.r.z = (int)ring::kNumRecords;
  s.r.w = 0x00020000;
  return s;
}

__device__ __forceinline__ void rsrc_advance(BufRsrc &s, long bytes) {
  unsigned long long b =
      ((unsigned long long)(unsigned)s.r.x) | ((unsigned long long)(unsigned)(s.r.y & 0xffff) << 32);
  b += (unsigned long long)bytes;
  s.r.x = __builtin_amdgcn_readfirstlane((int)(b & 0xffffffffu));
  s.r.y = __builtin_amdgcn_readfirstlane((int)(b >> 32) & 0xffff);
}

// 16 bytes per lane from the buffer at voff into LDS at lds + 16 * lane (lds is
// wave-uniform). M0 is saved and restored around the load.
__device__ __forceinline__ void dma16(const BufRsrc &s, unsigned voff, unsigned lds) {
  int saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %3\n\t"
      "buffer_load_dwordx4 %1, %2, 0 offen lds\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved)
      : "v"(voff), "s"(s.r), "s"(lds)
      : "memory");
}

using ring::hsw;
using ring::kc8_octet;
using ring::kc8_slot;
using ring::kOutOfRange;
using ring::msw32;

// s_waitcnt immediate that waits for vmcnt <= n only (vmcnt[3:0] in bits 3:0 and
// vmcnt[5:4] in bits 15:14; expcnt and lgkmcnt at their maxima).
constexpr int vmcnt_imm(int n) { return (n & 0xF) | ((n >> 4) << 14) | (0x7 << 4) | (0xF << 8); }

__device__ __forceinline__ unsigned lds_offset(const void *p) {
  return (unsigned)(unsigned long)(const LDS_AS void *)p;
}

// A scheduling region of NM MFMAs and NR LDS reads, interleaved 1:1 (then the rest).
template <int NM, int NR>
__device__ __forceinline__ void sched_interleave() {
  constexpr int NP = NR < NM ? NR : NM;
#pragma unroll
  for (int g = 0; g < NP; ++g) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
  }
  if constexpr (NM > NP) __builtin_amdgcn_sched_group_barrier(0x008, NM - NP, 0);
  if constexpr (NR > NP) __builtin_amdgcn_sched_group_barrier(0x100, NR - NP, 0);
}

// The same with up to VPM VALU instructions after every MFMA.
template <int NM, int NR, int VPM = 5>
__device__ __forceinline__ void sched_mix() {
#pragma unroll
  for (int g = 0; g < NM; ++g) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, VPM, 0);
    if (g < NR) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
  }
}

}  // namespace
}  // namespace gn
