// esdg_sequence.h -- the reference's kernel sequence in fewer passes over memory (schedule 0).
#pragma once

#include "esdg_internal.h"

namespace esdg {

// Device pointers of one stage (owned by the deviceclass mirror).  The gradient side traces gtr and the
// viscous volume term Qv are needed with artificial viscosity only.
struct SequenceArgs {
    int Nelem, Nfaces, artificial_viscosity, positivity;
    double *q, *gRK, *Qt;
    const double *Jac, *Yxi, *Yeta, *Xxi, *Xeta, *Bx, *By, *D, *Dhat, *Dstrong, *GLw, *EleSizes;
    const double *nx, *ny, *scal, *bL, *bR, *ViscPara;
    const int *EdgeData, *EdgeReversed, *ElemToEdge, *EMS, *EOR;
    double *qL, *qR, *SurfaceParts, *qGradientX, *qGradientY, *SurfacePartsVisc, *gtr, *Qv;
};

// CollectEdgeData + calcNumFluxes: qL, qR and SurfaceParts of the state.
int sequence_faces(esdg_ctx* ctx, const SequenceArgs& a);
// The stage from there (ViscPara is that of the state): the gradient chain and the viscous fluxes, then volume,
// surface and viscous terms into Qt, gRK = A gRK + Qt, q += cdt gRK and the limiter.
int sequence_update(esdg_ctx* ctx, const SequenceArgs& a, double rkA, double cdt);

}  // namespace esdg
