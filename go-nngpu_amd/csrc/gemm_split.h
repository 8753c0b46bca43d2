// gemm_split.h — large fp32 products on the bf16 matrix cores (gemm_split.hip), called by the
// GEMM dispatch (gemm.hip).
#pragma once

#include "common.h"
#include "split_gate.h"

namespace gn {

// The values the split layout holds: |x| < kSplitMax; the packed parts are of x * kSplitScale.
constexpr float kSplitScale = 65536.0f;      // 2^16
constexpr float kSplitMax = 68719476736.0f;  // 2^36
constexpr int kSplitBlock = 3072;            // bytes of 16 rows x 32 k in three bf16 parts
constexpr long kSplitMaxK = 1L << 20;        // K up to which no partial sum overflows

// How one launch of a product runs: tile (index into the kernel's shapes), S slices of K, the
// device time it is priced at (us, pack and reduce included), and the bytes of the packed
// operands and the partial products.
struct SplitPlan {
  int tile = 0, S = 1;
  bool raw_b = false;  // B is split by the product kernel instead of packed
  double us = 0;
  size_t pack_bytes = 0, part_bytes = 0;
};
// The plan for the parts of d that a launch takes: nb of its batches and kc of its K (a multiple
// of 32, or all of K; parts of K add to C). It holds for every part: alignments are those of any
// batch's and any part's operands, and the last part may be shorter. false: a shape the split
// kernels do not take.
bool plan_split(const GemmDesc &d, long nb, long kc, SplitPlan *out);
// The slices of a part with K `k` by that plan: none is empty.
inline int split_slices(const SplitPlan &plan, long k) {
  const long nkt = (k + 31) / 32;
  return plan.S < nkt ? plan.S : (int)nkt;
}

// How a product runs through launch_split within the scratch a stream keeps: nb batches and kc
// of K at a time, each by `plan`.
struct SplitCut {
  long nb = 0, kc = 0;
  SplitPlan plan;
  size_t ws_bytes = 0;
};
// true when the product runs on the bf16 matrix cores (gemm.hip). a_ok, b_ok: the operand suits
// the aligned fp32 kernels.
bool cut_split(const GemmDesc &d, bool a_ok, bool b_ok, SplitCut *cut);
// The partials' stride in floats: M x N rounded up to a multiple of 4.
inline long splitk_stride(long M, long N) { return (M * N + 3) / 4 * 4; }

// Packs the operands into ws (plan.pack_bytes) and multiplies them into C (d.C with the
// epilogue when plan.S == 1, else the partial products of the S slices into part). A word
// of *gate becomes seq when an operand holds a value the parts do not. Then d.C still holds what it
// held, except with a raw B and S == 1 (which plan_split gives for beta == 0 only).
hipError_t launch_split(const GemmDesc &d, const SplitPlan &plan, char *ws, float *part, SplitGate *gate,
                        unsigned long long seq, hipStream_t s);

}  // namespace gn
