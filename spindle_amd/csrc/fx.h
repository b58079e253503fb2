// Launchers of the float-activation products on the bf16 matrix cores (fx.hip): Q8_0 / Q5_0
// weights, 2..128 rows of fp32 activations; a row's bits do not depend on the pass's other rows.
#pragma once
#include "fused.h"

namespace spx {

bool fx_type(int dtype);  // Q8_0 or Q5_0

// The workgroups of launch_fx_mv over all rows of one matrix and m vectors: the grid to give it with
// greedy keys (a task a workgroup; other grids stride).
int fx_mv_wgs(const TensorView &w, int m);
// The segments' rows times m vectors (st null: a.m = m); all segments of one format and width. With greedy
// keys (a.best) the launch has grid_cap = a.nbest workgroups a vector group.
hipError_t launch_fx_mv(const MVArgs &a, int m, const StepRec *st, int grid_cap, hipStream_t s);
// Gate / up + SwiGLU: dense over the step record's m rows (a.jobs null), or over a job list of at
// most 16 users a job (vec = row of x, out = row of h), max_jobs bounding *a.njobs
hipError_t launch_fx_gateup(const GUArgs &a, int m, const StepRec *st, int max_jobs, hipStream_t s);
// Down projection of a job list's users (h rows out[]): y to a.yd [out][dim]
hipError_t launch_fx_down(const DownArgs &a, int max_jobs, hipStream_t s);

}  // namespace spx
