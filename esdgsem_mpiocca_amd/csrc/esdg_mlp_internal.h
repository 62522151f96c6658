// esdg_mlp_internal.h -- the learned indicator's entry points used by the solver (esdg_deviceclass.hip).
#pragma once

#include "esdg_internal.h"
#include "esdg_mlp.h"
#include "esdg_stage.h"

namespace esdg {

// Features + inference over the elements of q; p per element.
int mlp_classify(esdg_ctx* ctx, const esdg_mlp* m, int Nelem, const double* q, const double* B, const double* VdmInv,
                 float* p);
// The network's classes (0 smooth: p <= lo, 1 troubled: p >= hi, 2 unsure) over the elements of the stage
// batch's learned scenarios (tasks: 32-element tiles of N = 7 scenarios, in buffer src of their state), and
// in the same pass the modal sensor with zero viscosity where the class is smooth (from the modal
// coefficients the features already formed).  Each viscous element marks itself and its face neighbours
// for stage `stage` of the step; in stage 0 the viscosities enter each scenario's maximum.  A scenario
// whose time has reached its end is skipped.  counters (IND_SLOTS copies of 5 entries, 8 apart, accumulated):
// [0] element-stages with viscosity, [1] sensor positives declared smooth (audit), [2] sensor positives
// (audit), [3] element-stages not declared smooth, [4] element-stages classified.
int mlp_ensemble_indicator(esdg_ctx* ctx, const esdg_mlp* m, const StageScn* scns, const StageTask* tasks, int ntask,
                           int src, const int* mark, int stage, float lo, float hi, int audit,
                           unsigned long long* counters);


}  // namespace esdg
