// esdg_sequence.hip -- the reference's kernel sequence of one RK stage (src/deviceclass.cpp:938-1126) in
// fewer passes over memory:
//   CollectEdgeData + calcNumFluxes                                   -> sequence_faces
//   calcNumFluxesGradient + calcGradient + SurfaceKernelGradient +
//     scaleGradient + the sums of VolumeKernelViscose                 -> sequence_gradient
//   CollectEdgeDataGradient + calcNumFluxesViscose                    -> sequence_viscous_faces
//   VolumeKernel + SurfaceKernel + VolumeKernelViscose +
//     SurfaceKernelVisc + calcRK + UpdateKernel + PosPres             -> sequence_volume (esdg_volume.hip)
// Every value is computed with the expressions and in the order of those kernels, and q, Qt, gRK, qL, qR,
// SurfaceParts and the scaled gradients are stored as they leave them: the same bits.  Kernel by kernel the
// stage reads and writes Qt five times and each gradient four times; at 160 x 160, N = 7, with viscosity
// those 14 launches took 327 us per stage, these and the sensor take 175: sequence_volume 72 (350 MB),
// sequence_gradient 56 (280 MB), sequence_faces 21, the sensor 14, sequence_viscous_faces 10.
#include <type_traits>

#include "esdg_av_device.h"
#include "esdg_device.h"
#include "esdg_sequence.h"

namespace esdg {

int sequence_volume(esdg_ctx* ctx, const SequenceArgs& a, double rkA, double cdt);   // esdg_volume.hip

// One thread per face node, whole faces per block: the right state at the reversed node comes from that
// node's thread.  Bound by the strided reads of the element sides in the xi direction (a 64-byte line per
// value); the fluxes are evaluated while other waves wait for them.  KIND: the numerical flux, a template
// argument so that each instance holds the registers of its own flux only.
template <int KIND>
__global__ void __launch_bounds__(256) k_sequence_faces(int Nfaces, int ngl, FluxConsts c, GatherConsts gc,
                                                        const int* __restrict__ ED, const int* __restrict__ ER,
                                                        const double* __restrict__ q, const double* __restrict__ nxa,
                                                        const double* __restrict__ nya,
                                                        const double* __restrict__ scal,
                                                        const double* __restrict__ BL, const double* __restrict__ BR,
                                                        double* __restrict__ qL, double* __restrict__ qR,
                                                        double* __restrict__ SP) {
    __shared__ double sR[4][256];
    const int fpb = 256 / ngl;
    const int fl = threadIdx.x / ngl, i = threadIdx.x % ngl;
    const int64_t f = (int64_t)blockIdx.x * fpb + fl;
    const bool act = fl < fpb && f < Nfaces;
    const int64_t t = f * ngl + i;
    int cpuR = 0, ir = 0;
    double nx = 0.0, ny = 0.0, sc = 0.0, bl = 0.0;
    FaceState L{0.0, 0.0, 0.0};
    if (act) {
        const int* E = ED + 8 * f;
        const int rv = ER[f];
        ir = (1 - rv) * (ngl - 1 - i) + rv * i;
        cpuR = E[6];
        nx = nxa[t]; ny = nya[t]; sc = scal[t]; bl = BL[t];
        const double br = BR[t];
        FaceState Lq, Rq;
        face_side_traces(q, ngl, E, i, Lq, Rq);
        L = gathered_from(Lq, Rq, E, true, nx, ny, gc, bl, br);
        const FaceState R = gathered_from(Lq, Rq, E, false, nx, ny, gc, bl, br);
        const int64_t eid = f * ngl * ESDG_NEQ + i;
        qL[eid] = L.h; qL[eid + ngl] = L.hu; qL[eid + 2 * ngl] = L.hv;
        qR[eid] = R.h; qR[eid + ngl] = R.hu; qR[eid + 2 * ngl] = R.hv;
        sR[0][threadIdx.x] = R.h;
        sR[1][threadIdx.x] = R.hu;
        sR[2][threadIdx.x] = R.hv;
        sR[3][threadIdx.x] = br;
    }
    __syncthreads();
    if (!act) return;
    const int o = fl * ngl + ir;
    double F0, F1, F2;
    numerical_flux(KIND, c, cpuR, nx, ny, L.h, L.hu, L.hv, sR[0][o], sR[1][o], sR[2][o], bl, sR[3][o], F0, F1, F2);
    const int64_t eid = f * ngl * ESDG_NEQ + i;
    SP[eid] = sc * c.geomFace * F0;
    SP[eid + ngl] = sc * c.geomFace * F1;
    SP[eid + 2 * ngl] = sc * c.geomFace * F2;
}

// Face states from the arrays that sequence_faces stored; the scaled gradients go to gX, gY as well.
struct TraceFromFaces {
    const double *qL, *qR;
    double *gX, *gY;
    __device__ __forceinline__ FaceState operator()(int ngl, int f, const int*, bool left, int k, double, double,
                                                    const GatherConsts&, double, double) const {
        const double* p = (left ? qL : qR) + (int64_t)f * ngl * ESDG_NEQ + k;
        return FaceState{p[0], p[ngl], p[2 * ngl]};
    }
    template <int NN>
    __device__ __forceinline__ void store(int e, int n, double gx0, double gx1, double gy0, double gy1) const {
        const int64_t id = (int64_t)e * NN * 2 + n;
        gX[id] = gx0; gX[id + NN] = gx1;
        gY[id] = gy0; gY[id + NN] = gy1;
    }
};

// The gradient chain, one thread per node, intermediate fields in LDS: reads the state and the metrics
// once, writes the scaled gradients, their side traces and the viscous volume term once.
template <int NGL>
__global__ void __launch_bounds__(256) k_sequence_gradient(int Nelem, AvMesh M, TraceFromFaces src,
                                                           const double* __restrict__ Dh,
                                                           const double* __restrict__ Ds,
                                                           const double* __restrict__ visc) {
    using EB = ElemBlock<NGL>;
    constexpr int NN = NGL * NGL;
    __shared__ double sDh[NN], sDs[NN];
    __shared__ double sA[EB::THREADS], sB[EB::THREADS], sC[EB::THREADS], sE[EB::THREADS], sF[EB::EPB * 16 * NGL];
    __shared__ double sEps[EB::EPB];
    if (threadIdx.x < NN) {
        sDh[threadIdx.x] = Dh[threadIdx.x];
        sDs[threadIdx.x] = Ds[threadIdx.x];
    }
    const int e = blockIdx.x * EB::EPB + threadIdx.x / NN;
    const bool act = e < Nelem;
    av_element_block<NGL>(M, src, act ? e : 0, act, act ? visc[e] : 0.0, sDh, sDs, sA, sB, sC, sE, sF, sEps);
}

// CollectEdgeDataGradient.okl:17-194 + calcNumFluxesViscose.okl:17-107, one thread per face node, from the
// contiguous side traces of the gradients; an absent side's trace is zero and its viscosity the other side's.
__global__ void __launch_bounds__(256) k_sequence_viscous_faces(int Nfaces, int ngl, double geomFace,
                                                                const int* __restrict__ ED,
                                                                const double* __restrict__ gtr,
                                                                const double* __restrict__ visc,
                                                                const double* __restrict__ nxa,
                                                                const double* __restrict__ nya,
                                                                const double* __restrict__ scal,
                                                                double* __restrict__ SPV) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)Nfaces * ngl) return;
    const int f = (int)(t / ngl), i = (int)(t % ngl);
    const int* E = ED + 8 * (int64_t)f;
    const int iel = E[0], ier = E[1], isl = E[2], isr = E[3], rv = E[4], cpuL = E[5], cpuR = E[6];
    const double nx = nxa[t], ny = nya[t], sc = scal[t];
    double N0 = 0.0, N1 = 0.0;
    if (!(cpuL == -1 || cpuR == -1)) {
        const int inc = (rv == 0) ? (ngl - 1) - i : i;
        double XL0 = 0, XL1 = 0, XR0 = 0, XR1 = 0, YL0 = 0, YL1 = 0, YR0 = 0, YR1 = 0;
        double vl = 0.0, vr = 0.0;
        if (cpuL == 0) {
            const double* T = gtr + ((int64_t)iel * 4 + isl) * 4 * ngl + i;
            XL0 = T[0]; XL1 = T[ngl]; YL0 = T[2 * ngl]; YL1 = T[3 * ngl];
            vl = visc[iel];
        }
        if (cpuR == 0) {
            const double* T = gtr + ((int64_t)ier * 4 + isr) * 4 * ngl + inc;
            XR0 = T[0]; XR1 = T[ngl]; YR0 = T[2 * ngl]; YR1 = T[3 * ngl];
            vr = visc[ier];
        }
        const double f2L = nx * XL0 + ny * YL0;
        const double f2R = nx * XR0 + ny * YR0;
        const double f3L = nx * XL1 + ny * YL1;
        const double f3R = nx * XR1 + ny * YR1;
        const double m = fmax(vl, vr);
        N0 = 0.5 * m * (f2L + f2R);
        N1 = 0.5 * m * (f3L + f3R);
    }
    const int64_t eid = (int64_t)f * ngl * 2 + i;
    SPV[eid] = -sc * geomFace * N0;
    SPV[eid + ngl] = -sc * geomFace * N1;
}

template <int NGL>
void launch_sequence_gradient(esdg_ctx* ctx, const SequenceArgs& a) {
    using EB = ElemBlock<NGL>;
    const AvMesh M{a.q, a.Jac, a.Yxi, a.Yeta, a.Xxi, a.Xeta, a.ElemToEdge, a.EMS, a.EOR, a.EdgeData,
                   a.nx, a.ny, a.scal, a.bL, a.bR, GatherConsts{ctx->p.bc_kind, ctx->p.h_zero},
                   ctx->p.geomFace, ctx->p.PosPresTOL, a.gtr, a.Qv};
    k_sequence_gradient<NGL><<<blocks_for(a.Nelem, EB::EPB), EB::THREADS, 0, ctx->stream>>>(
        a.Nelem, M, TraceFromFaces{a.qL, a.qR, a.qGradientX, a.qGradientY}, a.Dhat, a.Dstrong, a.ViscPara);
}

int sequence_faces(esdg_ctx* ctx, const SequenceArgs& a) {
    if (a.Nfaces == 0) return ESDG_OK;
    const int ngl = ctx->p.ngl;
    FluxConsts fc{ctx->p.g, ctx->p.geomFace, ctx->p.PosPresTOL, ctx->p.ES};
    GatherConsts gc{ctx->p.bc_kind, ctx->p.h_zero};
    KernelScope ks(ctx, "sequence_faces");
    auto launch = [&](auto kind_tag) {
        k_sequence_faces<decltype(kind_tag)::value><<<blocks_for(a.Nfaces, 256 / ngl), 256, 0, ctx->stream>>>(
            a.Nfaces, ngl, fc, gc, a.EdgeData, a.EdgeReversed, a.q, a.nx, a.ny, a.scal, a.bL, a.bR, a.qL, a.qR,
            a.SurfaceParts);
    };
    switch (ctx->p.num_flux) {
        case ESDG_FLUX_ES: launch(std::integral_constant<int, ESDG_FLUX_ES>{}); break;
        case ESDG_FLUX_LF: launch(std::integral_constant<int, ESDG_FLUX_LF>{}); break;
        case ESDG_FLUX_ES_ROTATED: launch(std::integral_constant<int, ESDG_FLUX_ES_ROTATED>{}); break;
        case ESDG_FLUX_ROE: launch(std::integral_constant<int, ESDG_FLUX_ROE>{}); break;
        default: launch(std::integral_constant<int, ESDG_FLUX_OCEAN>{}); break;
    }
    return launch_check(ctx, "sequence_faces");
}

int sequence_update(esdg_ctx* ctx, const SequenceArgs& a, double rkA, double cdt) {
    if (a.Nelem == 0) return ESDG_OK;
    const int ngl = ctx->p.ngl;
    if (a.artificial_viscosity) {
        {
            KernelScope ks(ctx, "sequence_gradient");
            ESDG_NGL_DISPATCH(ngl, launch_sequence_gradient, ctx, a);
            const int rc = launch_check(ctx, "sequence_gradient");
            if (rc) return rc;
        }
        KernelScope ks(ctx, "sequence_viscous_faces");
        k_sequence_viscous_faces<<<blocks_for((int64_t)a.Nfaces * ngl, 256), 256, 0, ctx->stream>>>(
            a.Nfaces, ngl, ctx->p.geomFace, a.EdgeData, a.gtr, a.ViscPara, a.nx, a.ny, a.scal, a.SurfacePartsVisc);
        const int rc = launch_check(ctx, "sequence_viscous_faces");
        if (rc) return rc;
    }
    return sequence_volume(ctx, a, rkA, cdt);
}

}  // namespace esdg
