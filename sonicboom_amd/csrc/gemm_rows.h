// Products of up to eight bfloat16 rows whose blocks keep the rows in LDS (gemm_rows.hip), for the entry points that choose among
// the few-row kernels.
#pragma once

#include "common.h"

namespace sb {

// K slices that the raw product of these sizes comes in, 0: not taken.
int rows_slices(int n_rows, int n_out, int n_in);
// The raw product in rows_slices() slices, float [slices][n_rows][n_out].
int rows_partial(float *partial, const void *x, const void *w, int n_rows, int n_out, int n_in, void *stream);

// Whether the whole product of these sizes is taken: gated, or plain with float results and nothing added.
bool rows_whole(int n_rows, int n_out, int n_in, int gated);
// y float [n_rows][n_out] = x w^T.
int rows_plain(float *y, const void *x, const void *w, int n_rows, int n_out, int n_in, void *stream);
// y bfloat16 [n_rows][n_out] = act(f g) * (f u), f a row's factor that follows from ssq [ssq_parts][n_rows] (NULL: 1).
int rows_gated(void *y, const void *x, const double *ssq, int ssq_parts, float eps, const void *w, int n_rows, int n_out, int n_in,
               int gate, void *stream);

// The same from blocks that take a tile of features each and read X's fragments beside W's (gemm_skinny.hip), and where that is ahead.
bool tile_gated_pays(int n_rows, int n_out, int n_in);
int tile_gated(void *y, const void *x, const double *ssq, int ssq_parts, float eps, const void *w, int n_rows, int n_out, int n_in,
               int gate, void *stream);

}  // namespace sb
