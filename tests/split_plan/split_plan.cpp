// split_plan.cpp — CPU check of how fp32 products are cut for the bf16 matrix cores
// (go-nngpu_amd/csrc: cut_split, plan_split), through the built library's own functions; no GPU.
//
// For products of many shapes, layouts, batches, batch strides and alignments it walks the parts
// that run_split launches (nb batches and kc of K at a time) and checks what the kernels assume:
//  * B split by the product kernel and stored K-contiguous (float4 loads): every part's first
//    element and every row is 16-byte aligned and its K a multiple of 4;
//  * B split by the product kernel without slices of K (C is written before the values are known):
//    the part's beta is 0;
//  * no slice is empty, and the workspace holds the part's packed operands and partial products.
// And of the gate (split_gate.h): nothing that workgroups of the product kernel write changes what
// others of the same launch read, and whichever kernel finds a value stops the reduce and calls for the
// fp32 kernels, for this call only.
// Exit 0: no violation; 1: violations. Prints how many cuts of each form it saw. With arguments M N K
// batch layout gap (nn, nt, tn or tt; gap: elements between the batches' B) it prints that product's cut;
// with route f32|f16 layout M N K, the kernel that takes that product (aligned operands).
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "../../go-nngpu_amd/csrc/gemm_rows.h"
#include "../../go-nngpu_amd/csrc/gemm_split.h"

using namespace gn;

namespace {

long g_bad = 0;
void violation(const char *what, const GemmDesc &d, const SplitCut &c, long z, long k) {
  if (++g_bad <= 20)
    std::printf("VIOLATION %s: %ldx%ldx%ld batch %ld %c%c ldb %ld strideB %ld B%%16 %d beta %g: nb %ld kc %ld raw %d S %d, part "
                "z %ld k %ld\n",
                what, d.M, d.N, d.K, d.batch, d.ta ? 't' : 'n', d.tb ? 't' : 'n', d.ldb, d.strideB,
                (int)((uintptr_t)d.B % 16), d.beta, c.nb, c.kc, (int)c.plan.raw_b, c.plan.S, z, k);
}

struct Seen {
  long cuts = 0, raw = 0, raw_in_batch = 0, batch_cut = 0, one_batch = 0, k_cut = 0, raw_k_cut = 0, odd_stride = 0;
} g_seen;

bool cut(const GemmDesc &d, SplitCut *c) {
  const bool a_ok = d.lda % 4 == 0 && (d.batch == 1 || d.strideA % 4 == 0) && (d.ta ? d.M : d.K) % 4 == 0;
  const bool b_ok = (uintptr_t)d.B % 16 == 0 && d.ldb % 4 == 0 && (d.batch == 1 || d.strideB % 4 == 0) &&
                    (d.tb ? d.K : d.N) % 4 == 0;
  return cut_split(d, a_ok, b_ok, c);
}

void check(const GemmDesc &d) {
  SplitCut c;
  if (!cut(d, &c)) return;
  ++g_seen.cuts;
  g_seen.raw += c.plan.raw_b;
  g_seen.raw_in_batch += c.plan.raw_b && d.batch > 1;
  g_seen.batch_cut += c.nb < d.batch;
  g_seen.one_batch += c.nb == 1 && d.batch > 1;
  g_seen.k_cut += c.kc < d.K;
  g_seen.raw_k_cut += c.kc < d.K && c.plan.raw_b;
  g_seen.odd_stride += d.batch > 1 && d.tb && d.strideB % 4 != 0;
  if (c.nb < 1 || c.kc < 1 || (c.kc < d.K && c.kc % 32)) violation("part sizes", d, c, 0, 0);
  for (long z = 0; z < d.batch; z += c.nb)
    for (long k = 0; k < d.K; k += c.kc) {
      const long nb = d.batch - z < c.nb ? d.batch - z : c.nb, kk = d.K - k < c.kc ? d.K - k : c.kc;
      const int S = split_slices(c.plan, kk);
      const float beta = k > 0 ? 1.0f : d.beta;
      const long nkt = (kk + 31) / 32;
      for (int sl = 0; sl < S; ++sl)
        if ((long)(sl + 1) * nkt / S <= (long)sl * nkt / S) violation("empty slice", d, c, z, k);
      if (c.plan.raw_b && S == 1 && beta != 0.0f) violation("raw B writes a C that counts", d, c, z, k);
      if (c.plan.raw_b && d.tb)
        for (long b = z; b < z + nb; ++b) {
          const uintptr_t first = (uintptr_t)d.B + 4 * ((uintptr_t)b * d.strideB + k);
          if (first % 16 || d.ldb % 4 || kk % 4) violation("raw B loads off 16 bytes", d, c, b, k);
        }
      const size_t row = (size_t)nkt * kSplitBlock;
      const size_t pack = (size_t)nb * ((d.M + 15) / 16 + (c.plan.raw_b ? 0 : (d.N + 15) / 16)) * row;
      const size_t part = S > 1 ? ((size_t)S * splitk_stride(d.M, d.N) * 4 + 255) / 256 * 256 : 0;
      if (256 + part + pack > c.ws_bytes) violation("workspace too small", d, c, z, k);
    }
}

GemmDesc product(long M, long N, long K, long batch, bool ta, bool tb, long gap) {
  char *base = reinterpret_cast<char *>(0x700000000000ull);
  GemmDesc d;
  std::memset(&d, 0, sizeof d);
  d.dtype = GN_F32;
  d.ta = ta, d.tb = tb;
  d.M = M, d.N = N, d.K = K, d.batch = batch;
  d.alpha = 1.0f, d.act = -1;
  d.lda = ta ? M : K;
  d.ldb = tb ? K : N;
  d.ldc = N;
  d.strideA = M * K;
  d.strideB = N * K + gap;
  d.strideC = M * N;
  d.A = base;
  d.B = base + (1ull << 44);
  d.C = reinterpret_cast<float *>(base + (2ull << 44));
  return d;
}

}  // namespace

constexpr unsigned long long kSeq = 7, kOld = 6;
// The product kernel's test reads the same before and after workgroups of the same launch wrote.
static_assert(!split_product_skipped({kOld, kOld}, kSeq) && !split_product_skipped({kOld, kSeq}, kSeq), "uniform");
static_assert(split_product_skipped({kSeq, kOld}, kSeq) && split_product_skipped({kSeq, kSeq}, kSeq), "uniform");
static_assert(split_fp32_needed({kSeq, kOld}, kSeq) && split_fp32_needed({kOld, kSeq}, kSeq), "either finder");
static_assert(!split_fp32_needed({kOld, kOld}, kSeq), "an earlier call's values");

int main(int argc, char **argv) {
  if (argc == 7 && std::strcmp(argv[1], "route") == 0) {
    GemmDesc d = product(std::atol(argv[4]), std::atol(argv[5]), std::atol(argv[6]), 1, argv[3][0] == 't', argv[3][1] == 't', 0);
    d.dtype = argv[2][1] == '3' ? GN_F32 : GN_F16;
    const bool small = takes_small(d, true);
    RowsPlan rows;
    if (takes_gemv(d, true)) std::printf("gemv\n");
    else if (plan_rows(d, true, &rows) && takes_rows(d, rows, true, true, small)) std::printf("rows%s\n", rows.few ? "-4" : "");
    else std::printf("%s\n", small ? "small" : "tiles");
    return 0;
  }
  if (argc == 7) {
    const GemmDesc d = product(std::atol(argv[1]), std::atol(argv[2]), std::atol(argv[3]), std::atol(argv[4]),
                               argv[5][0] == 't', argv[5][1] == 't', std::atol(argv[6]));
    SplitCut c;
    if (cut(d, &c))
      std::printf("nb %ld kc %ld raw %d S %d\n", c.nb, c.kc, (int)c.plan.raw_b, c.plan.S);
    else
      std::printf("none\n");
    return 0;
  }
  const long Ms[] = {100, 160, 256, 300, 512, 777, 1024, 1300, 2048, 4096, 6200};
  const long Ns[] = {640, 1500, 4096, 5001, 11008};
  const long Ks[] = {512, 1000, 1533, 2052, 4096, 11008, 33000, 180004, 300033, 1048576};
  for (long M : Ms)
    for (long N : Ns)
      for (long K : Ks)
        for (int lay = 0; lay < 4; ++lay)
          for (long batch : {1L, 2L, 3L, 7L, 64L})
            for (long gap : {0L, 1L, 2L, 4L})
              for (long off : {0L, 4L})
                for (float beta : {0.0f, 0.5f}) {
                  if (gap && batch == 1 && off) continue;
                  GemmDesc d = product(M, N, K, batch, lay & 2, lay & 1, gap);
                  d.beta = beta;
                  if (batch == 1) d.ldb += gap;  // a pitch in place of a gap between batches
                  d.B = static_cast<const char *>(d.B) + off;
                  check(d);
                }
  std::printf("cuts %ld raw %ld raw_in_batch %ld batch_cut %ld one_batch %ld k_cut %ld raw_k_cut %ld odd_stride %ld\n",
              g_seen.cuts, g_seen.raw, g_seen.raw_in_batch, g_seen.batch_cut, g_seen.one_batch, g_seen.k_cut,
              g_seen.raw_k_cut, g_seen.odd_stride);
  std::printf("%ld violations\n", g_bad);
  return g_bad != 0;
}
