// gemm_rows.h — products of at most 64 rows (gemm_rows.hip), called by the GEMM dispatch (gemm.hip).
#pragma once

#include "common.h"
#include "gemm_split.h"  // splitk_stride

namespace gn {

// Columns per workgroup (16 fn), slices of K across workgroups, the price in us, and the bytes of
// the slices' partial products.
struct RowsPlan {
  int fn = 0, S = 1;
  bool few = false;  // NT, fn 1: 4 waves per workgroup
  double us = 0;
  size_t part_bytes = 0;
};
// false: a shape, layout or alignment these kernels do not take. split_ok: S > 1 is allowed.
bool plan_rows(const GemmDesc &d, bool split_ok, RowsPlan *out);
// C with the epilogue (plan.S == 1) or the partial products of the slices into part.
hipError_t launch_rows(const GemmDesc &d, const RowsPlan &plan, float *part, hipStream_t s);

// Products of 1 to 4 rows with a wide W stored K x N and little K, W aligned (b_ok): gemv_nn_kernel. One
// launch, no scratch.
bool takes_gemv(const GemmDesc &d, bool b_ok);
hipError_t launch_gemv(const GemmDesc &d, hipStream_t s);
// Whether the small-product kernel takes a product if no other does before it (gemm.hip). vec: the operands suit 16-byte
// vectors.
bool takes_small(const GemmDesc &d, bool vec);
// Whether launch_rows takes a product that plan_rows has planned (gemm.hip). small: takes_small.
bool takes_rows(const GemmDesc &d, const RowsPlan &rows, bool a_ok, bool b_ok, bool small);

}  // namespace gn
