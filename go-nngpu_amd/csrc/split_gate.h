// split_gate.h — who computes C of an fp32 product that runs on the bf16 matrix cores
// (gemm_split.hip): the split kernels, or the fp32 kernels enqueued behind them because an operand
// holds a value the split does not.
//
// Plain constexpr functions, so that the kernels and the CPU test (tests/split_plan) use the same.
// Each word is written by one launch and tested by later ones only: every workgroup, and every
// wave of it, sees the same value. (A product kernel that tested the word it also writes would
// let some waves of a workgroup leave while the others wait for them at a barrier.)
#pragma once

namespace gn {

// A word holds the number of the last call (seq) that found such a value.
struct SplitGate {
  unsigned long long packed;      // by the pack kernel, in the operands it packs
  unsigned long long multiplied;  // by the product kernel, in a B that it splits itself
};
// The product kernel has nothing to do.
constexpr bool split_product_skipped(const SplitGate &g, unsigned long long seq) { return g.packed == seq; }
// The split's result does not count: the reduce stops, the fp32 kernels run.
constexpr bool split_fp32_needed(const SplitGate &g, unsigned long long seq) {
  return g.packed == seq || g.multiplied == seq;
}

}  // namespace gn
