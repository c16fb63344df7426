// The nested-ordered hierarchy of fe_amg_pcg.hip as its other users read it.
#pragma once

#include "fe_hip_internal.h"

struct FeNestedLevel {
  int n, nc;
  int64_t nnz;
  const int2 *sell;             // level 0: (first SELL position, length) per row; columns ja, values valD
  const int *ia, *ja;           // levels >= 1: CSR
  const int *agg, *aggStart;    // not on the coarsest level
  const double *valD;           // level 0
  const float *val32, *l1_32;
};
struct FeNestedView {
  std::vector<FeNestedLevel> lv;
  const int *perm;              // level-0 row -> row of the system
  const double *cinv;           // inverse of the coarsest operator
  const int *flag;              // non-positive coarsest pivot
};
// Pattern (once) and numeric set-up of the current values for FP64 vectors
// with FP32 level values, without the small-level image (feAmgSetup first).
int feAmgNestedPrepare(fe_hip_ctx *ctx, FeNestedView *view);
