// Typed fp32 products of rows sorted by type (typed_rows.hip).
#pragma once

#include "common.h"

namespace ga {

constexpr int kMaxTypedRows = 4;      // weight tensors multiplied with one X

struct TypedRows {
  const int32_t *tp;                  // (n_types + 1) over the rows
  int n_types;
  const float *X;                     // (rows, K)
  int64_t rows;
  int K, M, n_weights;
  const float *W[kMaxTypedRows];      // (n_types, K, M)
  float *Y[kMaxTypedRows];            // (rows, M)
  const float *row_scale;             // Y[r, :] *= row_scale[r]; null: 1
  const float *gate;                  // Y[r, :] *= g(gate[type(r)]); null: 1
  bool gate_sigmoid;                  // g = 1 / (1 + exp(-x)) instead of the identity
};

// GA_OK, GA_EUNSUPPORTED (nothing launched: K not a multiple of 4 or above 128, M not 16, 32 or a
// multiple of 64, rows not 16-byte aligned) or a launch error.
int typed_rows_launch(const TypedRows &p, hipStream_t s);

}  // namespace ga
