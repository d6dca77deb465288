// kore_qmv_rows.h - what libkore_layer.so takes from libkore_qmv.so beside its
// public ABI.
#pragma once

#include "kore_qmv.h"

#include <cstdint>

// kore_qmv_get_row_dev for 1..64 rows in one launch (forward_batch(),
// kore.cpp:1496-1501): rows[z] (a host array, read before the call returns) ->
// out[z][n].
extern "C" KORE_QMV_API int kore_qmv_get_rows_dev(int type, const void *table, const int64_t *rows, int n_rows,
                                                  int64_t n, float *out, void *stream);
