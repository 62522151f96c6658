// esdg_stage.hip -- element-centric single-kernel RK stage over a batch of scenarios (see
// esdg_stage.h).  Per element and stage it performs, in the reference's arithmetic and order:
//   CollectEdgeData + calcNumFluxes for its 4 sides    (SolidWalls/InnerOuter/OceanBoundary.okl,
//                                                       calcESFlux.okl / calcESFluxRotated.okl)
//   VolumeKernel (flux differencing)                   (VolumeKernelFluxDiffV99.okl)
//   SurfaceKernel                                      (SurfaceKernel.okl, DBSurf = 0)
//   calcRK + UpdateKernel                              (rkLS.okl, UpdateKernelLS.okl)
//   [PosPres]                                          (PosPres.okl)
//   [FindLambdaMax of the new state, last stage]      (FindLambdaMax.okl)
//   [ShockCapturing of the new state]                 (ShockCapturing.okl, for the next stage)
//   [ArrivalTimes, MaximumElevation, last stage]      (ArrivalTimes.okl, MaximumElevation.okl)
// and the dt of DGtimeloop (src/deviceclass.cpp:899-930) runs on the device.
#include "esdg_av_device.h"
#include "esdg_device.h"
#include "esdg_mlp_internal.h"
#include "esdg_stage.h"

#include <algorithm>

namespace esdg {

// Per element: the four planes of the volume sweep (VolCfg::ESZ), reused for the face fluxes
// [side][v][k] once the sweeps have read them, and 16 doubles: the side records, and the limiter's and the
// sensor's sums (keeping consecutive elements 8 doubles apart modulo 16, as ESZ does).  At N = 7 a block of 8
// elements then fits 8 blocks per CU.
template <int NGL>
struct StageCfg {
    using V = VolCfg<NGL>;
    static constexpr int EPW = V::EPW;
    static constexpr int FSZ = 12 * NGL;              // face fluxes [side][v][k] of one element
    static_assert(FSZ <= 4 * V::PLANE, "the face fluxes fit in the element's planes");
    static constexpr int ELDS = V::ESZ + 16;          // per element: planes, side records, sums
    static constexpr int LDS = EPW * ELDS;            // doubles of LDS per block
};

constexpr int cmax(int a, int b) { return a > b ? a : b; }
template <int LO, int HI>
struct MaxLds {
    static constexpr int value = cmax(StageCfg<LO>::LDS, MaxLds<LO + 1, HI>::value);
};
template <int HI>
struct MaxLds<HI, HI> {
    static constexpr int value = StageCfg<HI>::LDS;
};

// a double that is the same in all lanes, as a scalar
__device__ __forceinline__ double uniform(double x) {
    const long long b = __double_as_longlong(x);
    const unsigned lo = __builtin_amdgcn_readfirstlane((int)b), hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// LDS accesses of a wave complete in order: the lanes of a block of one wave, or with MW of the wave that the
// caller is, see each other's.
template <bool MW>
__device__ __forceinline__ void wave_sync() {
    if constexpr (MW) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    } else {
        __syncthreads();
    }
}

// Volume term, surface lift, RK update, limiter and wave speed of one block of elements; the
// face fluxes of the elements' sides come from `faces`, into LDS (FS) after the sweeps.  Pointer
// parameters are __restrict__ so that the geometry loads schedule as in a kernel taking them as
// arguments, and global (gptr) so that they compile to global loads and stores.
// AFF: every element's metrics are the same at all of its nodes (a Cartesian mesh), and come from one
// record per element instead of five doubles per node; the bottom slopes too where they are constant.
// MW: the caller is the element wave of a block of five (k_stage_wide), the face fluxes come in mwFS.
// What bounds it: on curved meshes the memory path (512 x 512, N = 7, with viscosity: 618 us per stage for 3.34 GB
// moved, 5.4 TB/s, of which it cannot do without 2.71; an add of three large arrays reaches 5.65 here), on
// Cartesian meshes, whose records leave 11 doubles per node, instruction issue (256 x 256, N = 7: 120 us per
// stage, 157 with metrics per node), and on small ones one wave's chain of dependent steps.
template <int NGL, bool AV, bool AFF, bool MW, class Faces, class Early, class Dt>
__device__ __forceinline__ void stage_core(int e, int r, bool act, double* P, const Faces& faces, const Early& early,
                                           const Dt& step_dt, double g, double tol,
                                           double zero_tol, int positivity, double rkA, double rkC, bool last,
                                           gptr<const double> __restrict__ qi, gptr<double> __restrict__ qo,
                                           gptr<double> __restrict__ gRK, gptr<const double> __restrict__ Yeta,
                                           gptr<const double> __restrict__ Xeta, gptr<const double> __restrict__ Yxi,
                                           gptr<const double> __restrict__ Xxi, gptr<const double> __restrict__ Jac,
                                           gptr<const double> __restrict__ Bx, gptr<const double> __restrict__ By,
                                           gptr<const double> __restrict__ geo,
                                           gptr<const double> __restrict__ EleSizes,
                                           gptr<const double> __restrict__ GLw,
                                           const StageScn* SV, int src, int p,
                                           int mark, int next_mark, double* sD, double* mwFS) {
    using C = VolCfg<NGL>;
    double* FS = MW ? mwFS : P;      // face fluxes, after the sweeps (the planes are free then)
    const int4* rec = reinterpret_cast<const int4*>(P + C::ESZ);   // the element's side records
    double* MS = P + C::ESZ + 8;     // the limiter's and the sensor's sums
    const double* D = sD;
    const int lane = threadIdx.x;
    double h[NGL], hu[NGL], hv[NGL], u[NGL], v[NGL];
    double Y[AFF ? 1 : NGL], X[AFF ? 1 : NGL];
    double a1[NGL], a2[NGL], a3[NGL];
    double G[8];                     // the element's geometry record (AFF)
#pragma unroll
    for (int c = 0; c < NGL; ++c) { a1[c] = 0.0; a2[c] = 0.0; a3[c] = 0.0; }

    double dt = 0.0;
    // whether viscosity is in reach, and the element's own, loaded beside the row data
    bool marked = false;
    double eps0 = 0.0;
    if constexpr (AV) {
        if (act && SV->av) {
            marked = glob(SV->active[src])[e] == mark;
            eps0 = glob((const double*)SV->visc)[e];
        }
    }

    // ---- row phase: eta-row r ---------------------------------------------------------------
    if (act) {
        const int64_t qb = (int64_t)e * C::NN * 3 + r * NGL;
        const int64_t xb = (int64_t)e * C::NN + r * NGL;
        if constexpr (AFF) {
            using d2v = double __attribute__((ext_vector_type(2)));
            const gptr<const d2v> gp = (gptr<const d2v>)(geo + (int64_t)e * 8);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const d2v t = gp[k];
                G[2 * k] = t.x;
                G[2 * k + 1] = t.y;
            }
        }
#pragma unroll
        for (int c = 0; c < NGL; ++c) {
            h[c] = qi[qb + c];
            hu[c] = qi[qb + C::NN + c];
            hv[c] = qi[qb + 2 * C::NN + c];
            if constexpr (!AFF) {
                Y[c] = Yeta[xb + c];
                X[c] = Xeta[xb + c];
            }
        }
        // a step that changes nothing has dt < 0: with -1 the state goes over to the other buffer as it is, with -2
        // both buffers keep theirs.  (dt is loaded beside the rows; a wave that waited for it before loading
        // them cost 3 %.)
        dt = step_dt();
        if (dt < 0.0) {
            if (dt != -2.0) {
#pragma unroll
                for (int c = 0; c < NGL; ++c) {
                    qo[qb + c] = h[c];
                    qo[qb + C::NN + c] = hu[c];
                    qo[qb + 2 * C::NN + c] = hv[c];
                }
            }
        } else {
        early();   // LDS stores of values loaded beside the row data
#pragma unroll
        for (int c = 0; c < NGL; ++c) {
            const double inv = (h[c] > 0) ? 1.0 / h[c] : 0.0;
            u[c] = hu[c] * inv;
            v[c] = hv[c] * inv;
            P[0 * C::PLANE + r * C::RS + c] = h[c];
            P[1 * C::PLANE + r * C::RS + c] = hu[c];
            P[2 * C::PLANE + r * C::RS + c] = hv[c];
            P[3 * C::PLANE + r * C::RS + c] = inv;
        }
        if constexpr (AFF) line_sweep<NGL, false>(D, g, h, hu, hv, u, v, ConstMetrics(G[0], G[1]), a1, a2, a3);
        else line_sweep<NGL, false>(D, g, h, hu, hv, u, v, LineMetrics<NGL>{Y, X}, a1, a2, a3);
        }
    }
    dt = uniform(dt);   // (lane 0 has an element)
    if (dt < 0.0) {
        if constexpr (MW) __syncthreads();   // (every wave of the block meets one barrier)
        return;
    }
    wave_sync<MW>();

    // ---- column phase: xi-column r ----------------------------------------------------------
    const int64_t xb = (int64_t)e * C::NN + r;
    if (act) {
#pragma unroll
        for (int k = 0; k < NGL; ++k) {
            h[k] = P[0 * C::PLANE + k * C::RS + r];
            hu[k] = P[1 * C::PLANE + k * C::RS + r];
            hv[k] = P[2 * C::PLANE + k * C::RS + r];
            const double inv = P[3 * C::PLANE + k * C::RS + r];
            u[k] = hu[k] * inv;
            v[k] = hv[k] * inv;
            if constexpr (!AFF) {
                Y[k] = Yxi[xb + k * NGL];
                X[k] = Xxi[xb + k * NGL];
            }
        }
    }
    wave_sync<MW>();
    if (act) {
#pragma unroll
        for (int c = 0; c < NGL; ++c) {
            P[0 * C::PLANE + r * C::RS + c] = a1[c];
            P[1 * C::PLANE + r * C::RS + c] = a2[c];
            P[2 * C::PLANE + r * C::RS + c] = a3[c];
        }
    }
    wave_sync<MW>();
    double b1[NGL], b2[NGL], b3[NGL], rJ[NGL];
    if (act) {
#pragma unroll
        for (int k = 0; k < NGL; ++k) {
            b1[k] = P[0 * C::PLANE + k * C::RS + r];
            b2[k] = P[1 * C::PLANE + k * C::RS + r];
            b3[k] = P[2 * C::PLANE + k * C::RS + r];
        }
        if constexpr (AFF) line_sweep<NGL, true>(D, g, h, hu, hv, u, v, ConstMetrics(G[2], G[3]), b1, b2, b3);
        else line_sweep<NGL, true>(D, g, h, hu, hv, u, v, LineMetrics<NGL>{Y, X}, b1, b2, b3);
        // the bottom slopes: with AFF from the record where they are the same at every node (a choice of
        // address: a branch here makes the compiler move the whole sweep behind it and spill)
        gptr<const double> bxp = Bx + xb, byp = By + xb;
        int bst = NGL;
        if constexpr (AFF) {
            if (G[7] != 0.0) { bxp = geo + (int64_t)e * 8 + 5; byp = bxp + 1; bst = 0; }
        }
        double bx[NGL], by[NGL];
#pragma unroll
        for (int k = 0; k < NGL; ++k) {
            if constexpr (AFF) rJ[k] = G[4];
            else rJ[k] = Jac[xb + k * NGL];
            bx[k] = bxp[k * bst];
            by[k] = byp[k * bst];
        }
#pragma unroll
        for (int k = 0; k < NGL; ++k) {
            unscale_sums(b1[k], b2[k], b3[k]);
            b1[k] = -rJ[k] * b1[k];
            b2[k] = -rJ[k] * b2[k] - g * h[k] * bx[k];
            b3[k] = -rJ[k] * b3[k] - g * h[k] * by[k];
        }
    }
    // the face fluxes of the element's sides (from the stage-start state) into the planes, which
    // every lane has read by now
    if constexpr (MW) {
        __syncthreads();     // the block's other waves have written them
    } else {
        __syncthreads();
        if (act) faces(FS);
        __syncthreads();
    }
    if (act) {
        // surface lift: bottom/top sides first, then right/left (SurfaceKernel.okl).  FS holds
        // -ms F* (ms = +-1, so the sign is exact and -ms F* rJ equals the okl's -ms rJ F* bitwise).
        {
            const double* F0 = FS;
            const double* F2 = FS + 2 * 3 * NGL;
            b1[0] += F0[r] * rJ[0];
            b2[0] += F0[NGL + r] * rJ[0];
            b3[0] += F0[2 * NGL + r] * rJ[0];
            b1[NGL - 1] += F2[r] * rJ[NGL - 1];
            b2[NGL - 1] += F2[NGL + r] * rJ[NGL - 1];
            b3[NGL - 1] += F2[2 * NGL + r] * rJ[NGL - 1];
        }
        if (r == 0 || r == NGL - 1) {
            const double* F = FS + ((r == 0) ? 3 : 1) * 3 * NGL;
#pragma unroll
            for (int k = 0; k < NGL; ++k) {
                b1[k] += F[k] * rJ[k];
                b2[k] += F[NGL + k] * rJ[k];
                b3[k] += F[2 * NGL + k] * rJ[k];
            }
        }
        if constexpr (AV) {
            // the viscous terms of an element with viscosity in reach, in the reference's order
            // after the surface lift: the viscous volume term (where the element's viscosity is not
            // zero), then the lift of the viscous face fluxes (VolumeKernelViscose.okl,
            // SurfaceKernelVisc.okl), as the fused volume pass adds them
            if (marked) {
                const gptr<const double> SPV = glob((const double*)SV->SPV);
                // every load of the branch is issued before its sums: each side's face, orientation and
                // sign come from its record
                auto side = [&](int s, int& rev, double& nms) {
                    const int4 R4 = rec[s];
                    rev = (int)(((unsigned)R4.w >> 5) & 1u);
                    nms = (((unsigned)R4.w >> 6) & 1u) ? -1.0 : 1.0;    // -EMS
                    return SPV + (int64_t)R4.x * NGL * 2;
                };
                const bool edge = r == 0 || r == NGL - 1;
                int rv0, rv2, rvc;
                double m0, m2, mc;
                const gptr<const double> f0 = side(0, rv0, m0), f2 = side(2, rv2, m2),
                                         fc = side(r == NGL - 1 ? 1 : 3, rvc, mc);
                const int l0 = rv0 ? r : NGL - 1 - r, l2 = rv2 ? r : NGL - 1 - r;
                const double s02 = f0[l0], s03 = f0[l0 + NGL], s22 = f2[l2], s23 = f2[l2 + NGL];
                if (eps0 != 0.0) {
                    const gptr<const double> qv = glob((const double*)SV->Qv) + (int64_t)e * C::NN * 2 + r;
#pragma unroll
                    for (int k = 0; k < NGL; ++k) {
                        b2[k] += qv[k * NGL];
                        b3[k] += qv[C::NN + k * NGL];
                    }
                }
                b2[0] += m0 * rJ[0] * s02;
                b3[0] += m0 * rJ[0] * s03;
                b2[NGL - 1] += m2 * rJ[NGL - 1] * s22;
                b3[NGL - 1] += m2 * rJ[NGL - 1] * s23;
                if (edge) {
#pragma unroll
                    for (int k = 0; k < NGL; ++k) {
                        const int l = rvc ? k : NGL - 1 - k;
                        b2[k] += mc * rJ[k] * fc[l];
                        b3[k] += mc * rJ[k] * fc[l + NGL];
                    }
                }
            }
        }
        // low-storage RK: gRK = A gRK + Qt; q_new = q + (C dt) gRK, q at node (k, r) being this
        // lane's column input (h, hu, hv): the same bits, without a second read of q
        const double cdt = rkC * dt;
        const int64_t ob = (int64_t)e * C::NN * 3 + r;
        // A step's first stage has A = 0: the register starts from Qt and is not read.  What the last
        // stage would leave in it is read by nobody but a checkpoint: it is stored where the caller
        // asks for it.
        if (rkA != 0.0) {
#pragma unroll
            for (int k = 0; k < NGL; ++k) {
                const int64_t id = ob + k * NGL;
                b1[k] = rkA * gRK[id] + b1[k];
                b2[k] = rkA * gRK[id + C::NN] + b2[k];
                b3[k] = rkA * gRK[id + 2 * C::NN] + b3[k];
            }
        }
        if (!last || glob((const double*)SV->clock)[8 * (p ^ 1) + 6] != 0.0) {
#pragma unroll
            for (int k = 0; k < NGL; ++k) {
                const int64_t id = ob + k * NGL;
                gRK[id] = b1[k];
                gRK[id + C::NN] = b2[k];
                gRK[id + 2 * C::NN] = b3[k];
            }
        }
#pragma unroll
        for (int k = 0; k < NGL; ++k) {
            b1[k] = h[k] + cdt * b1[k];
            b2[k] = hu[k] + cdt * b2[k];
            b3[k] = hv[k] + cdt * b3[k];
        }
    }
    if (positivity) {
        // PosPres.okl on the new state: the products h w, hu w, hv w (w = GLw[xi] GLw[eta] / Jinv) to the
        // planes; three lanes of the element add them in the okl's serial order (xi outer, eta inner)
        wave_sync<MW>();
        double hmin = 0.0;
        if (act) {
            const double gx = GLw[r];
#pragma unroll
            for (int k = 0; k < NGL; ++k) {
                const double w = gx * GLw[k] / rJ[k];
                P[0 * C::PLANE + k * C::RS + r] = b1[k] * w;
                P[1 * C::PLANE + k * C::RS + r] = b2[k] * w;
                P[2 * C::PLANE + k * C::RS + r] = b3[k] * w;
                hmin = fmin(hmin, b1[k]);
            }
            P[3 * C::PLANE + r] = hmin;
        }
        wave_sync<MW>();
        if (act && r < 3) {
            const double* F = P + r * C::PLANE;
            double a = 0.0;
            for (int l = 0; l < NGL; ++l)
                for (int k = 0; k < NGL; ++k) a += F[k * C::RS + l];
            MS[r] = a;
        }
        wave_sync<MW>();
        if (act) {
            hmin = 0.0;
#pragma unroll
            for (int k = 0; k < NGL; ++k) hmin = fmin(hmin, P[3 * C::PLANE + k]);
            const double size = EleSizes[e];
            double ha = MS[0] / size;
            if (fabs(ha) < zero_tol) ha = 0.0;
            const double hua = MS[1] / size, hva = MS[2] / size;
            const double th = (ha == hmin) ? 1.0 : fmin(1.0, ha / (ha - hmin));
#pragma unroll
            for (int k = 0; k < NGL; ++k) {
                if (hmin < 0.0) {
                    double hn = 0.0, hun = 0.0, hvn = 0.0;
                    if (ha > 0.0) {
                        hn = fabs(th * (b1[k] - ha) + ha);
                        if (hn > tol) {
                            hun = th * (b2[k] - hua) + hua;
                            hvn = th * (b3[k] - hva) + hva;
                        }
                    }
                    if (ha < 0.0) { hn = -INFINITY; hun = 0.0; hvn = 0.0; }
                    b1[k] = hn; b2[k] = hun; b3[k] = hvn;
                } else if (b1[k] < tol) {
                    b2[k] = 0.0; b3[k] = 0.0;
                }
            }
        }
    }
    // b of row r for the sensor below, loaded before the stores
    // (a step of a failed scenario has marks in its first stage only)
    const bool sensor = AV && SV->av && !SV->learned && (dt != 0.0 || last);
    double w[AV ? NGL : 1];
    if constexpr (AV) {
        if (sensor && act) {
            const gptr<const double> B = glob(SV->B) + (int64_t)e * C::NN + r * NGL;
#pragma unroll
            for (int i = 0; i < NGL; ++i) w[i] = B[i];
        }
    }
    double lam = 0.0;
    if (act) {
        const int64_t ob = (int64_t)e * C::NN * 3 + r;
#pragma unroll
        for (int k = 0; k < NGL; ++k) {
            const int64_t id = ob + k * NGL;
            qo[id] = b1[k];
            qo[id + C::NN] = b2[k];
            qo[id + 2 * C::NN] = b3[k];
        }
        if (last) {
            // FindLambdaMax.okl on the new state (the next step's dt)
#pragma unroll
            for (int k = 0; k < NGL; ++k) {
                const double hh = b1[k];
                const double Qinv = (hh > tol) ? 1.0 / hh : 0.0;
                const double c = sqrt(g * hh);
                lam = fmax(lam, c + fmax(fabs(b2[k] * Qinv), fabs(b3[k] * Qinv)));
            }
        }
    }
    if (last) {
        if (SV->lam) {
            double m = 0.0;
#pragma unroll
            for (int k = 0; k < NGL; ++k) m = fmax(m, __shfl(lam, lane - r + k));
            if (act && r == 0) glob(SV->lam)[e] = m;
        }
        double m = lam;
        for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off));
        if (lane == 0) max_into(SV->lmax + (p ^ 1), m);
        // ArrivalTimes.okl:16-62 and MaximumElevation.okl:16-55 on the state after the step, at its time
        if (act && SV->arrival) {
            const double t = glob(SV->clock)[8 * (p ^ 1) + 1];
            const gptr<double> arr = glob(SV->arrival);
            const gptr<const double> B = glob(SV->B);
#pragma unroll
            for (int k = 0; k < NGL; ++k) {
                const int64_t x = xb + k * NGL;
                if (arr[x] == 1000.0 && fabs((b1[k] + B[x]) - SV->h_zero) > 0.00005) arr[x] = t;
            }
        }
        if (act && SV->maxelev) {
            const gptr<double> mx = glob(SV->maxelev);
            const gptr<const double> B = glob(SV->B);
#pragma unroll
            for (int k = 0; k < NGL; ++k) {
                const int64_t x = xb + k * NGL;
                mx[x] = fmax(mx[x], b1[k] + B[x] - SV->h_zero);
            }
        }
    }
    if constexpr (AV) {
        // ShockCapturing.okl:63-217 on the new state (here 46 us at 512 x 512, N = 7, the stage 573 and without it
        // 527; as a pass of its own 81), with the arithmetic of sensor_rows: lane r forms
        // column r of T = V (h + b) from row r of h + b, then the squares of row r of T V^T; up to four
        // lanes form the energy sums.  An element with viscosity marks what it reaches for the next stage,
        // and after the last stage its viscosity enters the next step's maximum.
        if (sensor) {
            wave_sync<MW>();
            double* Tm = P + 1 * C::PLANE;
            double* V = sD;
            for (int t = lane; t < C::NN; t += 64) V[t] = glob(SV->VdmInv)[t];
            if (act) {
#pragma unroll
                for (int k = 0; k < NGL; ++k) P[k * C::RS + r] = b1[k];
            }
            wave_sync<MW>();
            if (act) {
#pragma unroll
                for (int i = 0; i < NGL; ++i) w[i] = w[i] + P[r * C::RS + i];
#pragma unroll
                for (int a = 0; a < NGL; ++a) {
                    double s = 0.0;
#pragma unroll
                    for (int l = 0; l < NGL; ++l) s += V[a * NGL + l] * w[l];
                    Tm[a * C::RS + r] = s;
                }
            }
            wave_sync<MW>();
            if (act) {
#pragma unroll
                for (int l = 0; l < NGL; ++l) w[l] = Tm[r * C::RS + l];
#pragma unroll
                for (int c = 0; c < NGL; ++c) {
                    double s = 0.0;
#pragma unroll
                    for (int l = 0; l < NGL; ++l) s += w[l] * V[c * NGL + l];
                    Tm[r * C::RS + c] = s * s;
                }
            }
            wave_sync<MW>();
            if (act)
                for (int k = r; k < 4; k += NGL) MS[k] = sensor_sum_lane<NGL, C::RS>(Tm, k);
            wave_sync<MW>();
            double eps = 0.0;
            if (act && r == 0) {
                eps = sensor_ramp(MS[0], MS[1], MS[2], MS[3], SV->sc);
                glob(SV->visc)[e] = eps;
                if (SV->visc_plot) glob(SV->visc_plot)[e] = eps;
            }
            // the marks of an element with viscosity, a side per lane
            if (__shfl(eps, lane - r) != 0.0 && act) {
                for (int s = r; s < 4; s += NGL) mark_side(*SV, e, s, rec[s], next_mark, src ^ 1);
            }
            if (last) {
                // non-negative doubles order as their bit patterns; a NaN stays out, as fmax leaves it
                double m = eps > 0.0 ? eps : 0.0;
                for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_xor(m, off));
                if (lane == 0 && m > 0.0) max_into(SV->emax + (p ^ 1), m);
            }
        }
    }
}


// DGtimeloop's dt (src/deviceclass.cpp:899-930) of the step that starts from the scenario's clock ck: while
// t < T, dt = min(T - t, dti / lambda_max[, dvc / eps_max]) and t += dt; once t >= T the
// steps change nothing: dt = -1 in the first stage, which carries the state over to the other buffer, and -2, with
// which nothing is written, from there on.  From a dt that is not positive and finite on, which is flagged, dt = -2 at
// once: the last good step's state and the one before its last stage stay where they are (see
// StageBatch::repeat_last_stage).  (A batch that does not freeze a failed state goes on with dt = 0 there: what
// is not finite spreads, as in q + 0 gRK.)  Every
// wave of a step's first stage forms it from the maxima that the last step's last stage left, beside its
// row loads; the clock after it is written to `next` by one of them (as a launch of its own before the
// stages it took 4 to 5 us per step).
__device__ __forceinline__ double first_dt(const StageScn& S, gptr<const double> ck, double lm, double em,
                                           gptr<double> next) {
    const double t = ck[1], steps = ck[2], failed = ck[4], until = ck[7];
    double dt = failed != 0.0 || ck[0] < 0.0 ? -2.0 : -1.0, t1 = t, n1 = steps, last = ck[3], err = failed, bad = ck[5], keep = ck[6];
    if (t < S.T && failed == 0.0) {
        const double dt_i = S.dti / lm;
        // with artificial viscosity also the viscous limit dvc / max eps (infinite where no element
        // has viscosity), in the order of src/deviceclass.cpp:920-926
        dt = S.av ? fmin(S.T - t, fmin(dt_i, S.dvc / em)) : fmin(S.T - t, dt_i);
        if (!(dt > 0.0) || isinf(dt)) {
            err = 1.0;
            bad = dt;
            keep = 1.0;
            dt = S.freeze ? -2.0 : 0.0;
        } else {
            t1 = t + dt;
            n1 = steps + 1.0;
            last = dt;
            // the step that ends the run leaves its RK register for a checkpoint
            keep = (n1 == until || t1 >= S.T) ? 1.0 : 0.0;
        }
    } else if (failed != 0.0 && !S.freeze) {
        dt = 0.0;
    }
    if (next) {
        next[0] = dt; next[1] = t1; next[2] = n1; next[3] = last;
        next[4] = err; next[5] = bad; next[6] = keep; next[7] = until;
    }
    return dt;
}

template <int NGL, bool AV, bool AFF, bool MW>
__device__ __forceinline__ void stage_body(const StageScn& S, int e0, double* lds, double* sD, double* mwF, int src, int stage,
                                           double rkA, double rkC, bool last, int mark, int next_mark, int* markp) {
    using C = VolCfg<NGL>;
    using SC = StageCfg<NGL>;
    const int lane = MW ? threadIdx.x & 63 : threadIdx.x;
    const int wave = MW ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
    const int p = src ^ (stage & 1);     // the step's half of the clocks, maxima and marks
    // the marks of the stage's state have been used: the list that the next stage's marks go to is the
    // other one, and this one is empty when its turn comes
    // (the list's first scenario does, a part per lane)
    if (AV && S.av && S.mbase == 0 && e0 == 0 && wave == 0) *mark_count(S.mcount, src, lane) = 0;
    if (stage == 1 && e0 == 0 && lane == 0 && wave == 0) {
        // the first stage has read the step's maxima: they are empty when the next step's last stage adds
        // to them; and the next step's marks
        S.lmax[p] = 0ull;
        if (AV && S.av) S.emax[p] = 0ull;
        if (AV && S.id == 0) markp[p ^ 1] = markp[p] + STAGE_MARKS;
    }
    // D of this degree in LDS (wave-uniform reads, broadcast): keeps it out of the scalar registers
    if (wave == 0)
        for (int t = lane; t < NGL * NGL; t += 64) sD[t] = glob(S.D)[t];
    const int el = lane / NGL, r = lane % NGL;
    const int e = e0 + el;
    const bool act = (el < C::EPW) && (e < S.Nelem);
    double* P = lds + (act ? el : 0) * SC::ELDS;     // planes: h, hu, hv, 1/h (later: the row sums)
    const gptr<const double> qi = glob((const double*)S.q[src]);
    const gptr<double> qo = glob(S.q[src ^ 1]);
    const double g = S.g;

    // The element's four side records (StageScn::srec) are loaded beside the row data and stored
    // to LDS, so the face-flux reads after the sweeps need no dependent round trips through
    // ElemToEdge and EdgeData.
    constexpr int FPL = (4 + NGL - 1) / NGL;   // sides per lane: lane r loads sides r, r + NGL, ...
    int4 rec[FPL];
#pragma unroll
    for (int j = 0; j < FPL; ++j) {
        const int sd = r + j * NGL;
        rec[j] = make_int4(0, 0, 0, 0);
        if (act && sd < 4 && wave == 0) rec[j] = side_record(S, e, sd);
    }
    int4* RS = reinterpret_cast<int4*>(P + C::ESZ);
    auto early = [&]() {
#pragma unroll
        for (int j = 0; j < FPL; ++j)
            if (r + j * NGL < 4) RS[r + j * NGL] = rec[j];
    };

    // ---- fluxes of the element's four sides: lane r takes side node r of every side (called by
    // stage_core once the sweeps are done, with the face-flux area FS) ----------------------------
    auto faces = [&](double* FS) {
        const FluxConsts fc{g, S.geomFace, S.tol, S.ES};
        const GatherConsts gc{S.bc, S.h_zero};
        const gptr<const double> nxp = glob(S.nx), nyp = glob(S.ny), scp = glob(S.scal), bLp = glob(S.bL),
                                 bRp = glob(S.bR);
        // one side's decoded record and loads
        struct Side {
            int E[8];
            int ir, rev;     // the reversed face node (EdgeData[4]) of the lane's node; EOR
            unsigned w;
            FaceState Li, Ri;
            double nx, ny, sc, bl, br;
        };
        auto load = [&](int s, Side& d) {
            const int4 R4 = MW ? side_record(S, e, s) : RS[s];
            const int f = R4.x;
            d.w = (unsigned)R4.w;
            d.rev = (int)((d.w >> 5) & 1u);
            const int i = d.rev * r + (1 - d.rev) * (NGL - 1 - r);      // face node of side node r
            // EdgeData's entries as gathered() reads them
            d.E[0] = R4.y; d.E[1] = R4.z; d.E[2] = (int)(d.w & 3u); d.E[3] = (int)((d.w >> 2) & 3u);
            d.E[4] = (int)((d.w >> 4) & 1u); d.E[5] = (int)((d.w >> 8) & 255u) - 2;
            d.E[6] = (int)((d.w >> 16) & 255u) - 2; d.E[7] = 0;
            const int rv = d.E[4];
            d.ir = (1 - rv) * (NGL - 1 - i) + rv * i;
            const int64_t t = (int64_t)f * NGL + i;
            face_side_traces(qi, NGL, d.E, i, d.Li, d.Ri);
            if constexpr (AFF) {
                // a face whose five values are the same at every node has them in one 64-byte record
                const bool one = (d.w >> 24) & 1u;
                const gptr<const double> fg = glob(S.fgeo) + (int64_t)f * 8;
                d.nx = one ? fg[0] : nxp[t];
                d.ny = one ? fg[1] : nyp[t];
                d.sc = one ? fg[2] : scp[t];
                d.bl = one ? fg[3] : bLp[t];
                d.br = one ? fg[4] : bRp[t];
            } else {
                d.nx = nxp[t]; d.ny = nyp[t]; d.sc = scp[t]; d.bl = bLp[t]; d.br = bRp[t];
            }
        };
        // The element's NGL lanes (one wave) hold the face's NGL nodes: each lane also evaluates
        // the right trace at its own node, and lane r takes node ir's from the lane holding it
        auto flux = [&](int s, const Side& d) {
            const FaceState L = gathered_from(d.Li, d.Ri, d.E, true, d.nx, d.ny, gc, d.bl, d.br);
            const FaceState Ro = gathered_from(d.Li, d.Ri, d.E, false, d.nx, d.ny, gc, d.bl, d.br);
            const int src = lane - r + (d.rev * d.ir + (1 - d.rev) * (NGL - 1 - d.ir));
            const FaceState R{__shfl(Ro.h, src), __shfl(Ro.hu, src), __shfl(Ro.hv, src)};
            const double brr = __shfl(d.br, src);
            double F0, F1, F2;
            numerical_flux(S.num_flux, fc, d.E[6], d.nx, d.ny, L.h, L.hu, L.hv, R.h, R.hu, R.hv, d.bl, brr, F0, F1,
                           F2);
            const double nms = ((d.w >> 6) & 1u) ? -1.0 : 1.0;   // -EMS
            FS[(s * 3 + 0) * NGL + r] = nms * (d.sc * S.geomFace * F0);
            FS[(s * 3 + 1) * NGL + r] = nms * (d.sc * S.geomFace * F1);
            FS[(s * 3 + 2) * NGL + r] = nms * (d.sc * S.geomFace * F2);
        };
        Side a, b;
        if constexpr (MW) {
            load(wave - 1, a);
            flux(wave - 1, a);
            return;
        }
        // two sides at a time, in a loop of one copy of the code: unrolled over the four sides, with each
        // side's loads issued before the fluxes of the one before it, the N = 7 kernels were 87 to 99 KB of
        // code, more than the 64 KB of instruction cache, and slower (us per step with and without the
        // loop: 256 x 256, N = 7, single kernel 596 and 624, 192 x 192 with analysis 352 and 390, 24 mixed
        // scenarios 1073 and 1174, 512 x 512 with viscosity 3155 and 3228)
#pragma unroll 1
        for (int s = 0; s < 4; s += 2) {
            load(s, a);
            load(s + 1, b);
            flux(s, a);
            flux(s + 1, b);
        }
    };

    auto step_dt = [&]() -> double {
        const gptr<double> ck = glob(S.clock);
        if (stage) {
            const double dt = ck[8 * (p ^ 1)];
            return dt < 0.0 ? -2.0 : dt;
        }
        const double lm = __longlong_as_double((long long)glob(S.lmax)[p]);
        const double em = S.av ? __longlong_as_double((long long)glob(S.emax)[p]) : 0.0;
        return first_dt(S, ck + 8 * p, lm, em, e0 == 0 && lane == 0 ? ck + 8 * (p ^ 1) : nullptr);
    };

    double* const FSx = MW ? mwF + (act ? el : 0) * SC::FSZ : nullptr;
    if constexpr (MW) {
        if (wave > 0) {
            if (act) faces(FSx);
            __syncthreads();
            return;
        }
    }
    wave_sync<MW>();   // sD written
    stage_core<NGL, AV, AFF, MW>(e, r, act, P, faces, early, step_dt, g, S.tol, S.zero_tol, S.positivity, rkA, rkC, last, qi, qo, glob(S.gRK), glob(S.Yeta), glob(S.Xeta), glob(S.Yxi),
                             glob(S.Xxi), glob(S.Jac), glob(S.Bx), glob(S.By), glob(S.geo), glob(S.EleSizes), glob(S.GLw),
                             &S, src, p, mark, next_mark, sD, FSx);
}

template <int LO, int HI, bool AV, bool AFF, bool MW = false>
__device__ __forceinline__ void stage_task(const StageScn* __restrict__ scns, const StageTask& tk, double* lds,
                                           double* sD, double* mwF, int src, int stage, double rkA, double rkC, bool last, int mark,
                                           int next_mark, int* markp) {
    const StageScn& S = scns[tk.scn];
    switch (tk.ngl) {
#define ESDG_CASE(n)                                                                \
    case n:                                                                         \
        if constexpr (n >= LO && n <= HI) stage_body<n, AV, AFF, MW>(S, tk.e0, lds, sD, mwF, src, stage, rkA, rkC, last, mark, next_mark, markp); \
        break;
        ESDG_CASE(3) ESDG_CASE(4) ESDG_CASE(5) ESDG_CASE(6) ESDG_CASE(7) ESDG_CASE(8)
#undef ESDG_CASE
        default: break;
    }
}

// One RK stage over tasks[0, n).  Non-persistent: block b takes one task.  Persistent: the tasks
// are cut into chunks of `tile` consecutive tasks and a grid of gridDim.x blocks loops over the
// chunks, one block taking a chunk's tasks one after another (with tile > 1 and a grid of one
// block per chunk this is the element-tile size: a block advances tile element groups).  With
// xcd = 1 the task list is cut into 8 contiguous parts and the blocks that the dispatcher places
// on XCD x (b mod 8 = x) take part x, so tasks that are adjacent in the list (one element tile of
// several scenarios that share geometry) meet in the same L2.  Every block leaves after a bounded
// number of tasks.
template <int LO, int HI, bool PERSIST, bool AV, bool AFF>
__global__ void __launch_bounds__(64, 2) k_stage(const StageScn* __restrict__ scns, const StageTask* __restrict__ tasks,
                                                 int n, int xcd, int tile, int src, double rkA, double rkC,
                                                 int last, int* markp, int stage) {
    __shared__ __attribute__((aligned(16))) double lds[MaxLds<LO, HI>::value];
    __shared__ double sD[HI * HI];
    const int base = AV ? markp[src ^ (stage & 1)] : 0, mark = base + stage, next_mark = last ? base + STAGE_MARKS : mark + 1;
    const int b = blockIdx.x;
    int beg = 0, cnt = n, i0 = b, stride = gridDim.x;
    if (xcd) {
        const int q = n >> 3, rr = n & 7, x = b & 7;
        cnt = q + (x < rr ? 1 : 0);
        beg = x * q + (x < rr ? x : rr);
        i0 = b >> 3;
        stride = gridDim.x >> 3;
    }
    // (the tasks of a single scenario need no list)
    auto task = [&](int i) { return tasks ? tasks[i] : StageTask{0, i * (64 / LO), LO, 0}; };
    if constexpr (!PERSIST) {
        if (i0 < cnt) stage_task<LO, HI, AV, AFF>(scns, task(beg + i0), lds, sD, nullptr, src, stage, rkA, rkC, last != 0, mark, next_mark, markp);
    } else {
        const int nch = (cnt + tile - 1) / tile;
        for (int c = i0; c < nch; c += stride) {
            const int i1 = min(cnt, (c + 1) * tile);
            for (int i = c * tile; i < i1; ++i) {
                if (i != i0 * tile) __syncthreads();   // LDS of the previous task is free
                stage_task<LO, HI, AV, AFF>(scns, task(beg + i), lds, sD, nullptr, src, stage, rkA, rkC, last != 0, mark, next_mark, markp);
            }
        }
    }
}

// The same stage for short lists of tasks of one degree, where a stage takes as long as one wave's chain of
// loads, sweeps and face fluxes: five waves per block, one for the elements and one for each of their
// sides, whose fluxes are ready when the sweeps are.  16 x 16, N = 4: 12.2 us per stage with one wave per block,
// 7.6 with five.
template <int NGL, bool AV, bool AFF>
__global__ void __launch_bounds__(320, 2) k_stage_wide(const StageScn* __restrict__ scns,
                                                       const StageTask* __restrict__ tasks, int n, int xcd, int src,
                                                       double rkA, double rkC, int last, int* markp, int stage) {
    __shared__ __attribute__((aligned(16))) double lds[StageCfg<NGL>::LDS];
    __shared__ double sD[NGL * NGL], mwF[StageCfg<NGL>::EPW * StageCfg<NGL>::FSZ];
    const int base = AV ? markp[src ^ (stage & 1)] : 0, mark = base + stage, next_mark = last ? base + STAGE_MARKS : mark + 1;
    int i = blockIdx.x, beg = 0, cnt = n;
    if (xcd) {
        const int q = n >> 3, rr = n & 7, x = i & 7;
        cnt = q + (x < rr ? 1 : 0);
        beg = x * q + (x < rr ? x : rr);
        i >>= 3;
    }
    if (i >= cnt) return;
    const StageTask tk = tasks ? tasks[beg + i] : StageTask{0, (beg + i) * (64 / NGL), NGL, 0};
    stage_body<NGL, AV, AFF, true>(scns[tk.scn], tk.e0, lds, sD, mwF, src, stage, rkA, rkC, last != 0, mark, next_mark, markp);
}

// lambda_max of the state in buffer src, per scenario (FindLambdaMax.okl + the host max loop).  A block
// takes every gridDim.x-th task and keeps the maximum while the scenario stays the same (one wave per task,
// each with an atomic, took 395 us at 512 x 512, N = 7; this takes 89).
__global__ void __launch_bounds__(256) k_stage_lambda(const StageScn* __restrict__ scns,
                                                      const StageTask* __restrict__ tasks, int n, int src) {
    __shared__ double part[4];
    double lam = 0.0;
    for (int i = blockIdx.x; i < n; i += gridDim.x) {
        const StageTask tk = tasks ? tasks[i] : StageTask{0, i * (64 / scns[0].ngl), scns[0].ngl, 0};
        const StageScn& S = scns[tk.scn];
        const int ngl2 = tk.ngl * tk.ngl;
        const int nodes = min(64 / tk.ngl, S.Nelem - tk.e0) * ngl2;
        const gptr<const double> q = glob((const double*)S.q[src]) + (int64_t)tk.e0 * ngl2 * 3;
        for (int t = threadIdx.x; t < nodes; t += 256) {
            const int id = t / ngl2 * ngl2 * 3 + t % ngl2;
            const double hh = q[id];
            const double Qinv = (hh > S.tol) ? 1.0 / hh : 0.0;
            const double c = sqrt(S.g * hh);
            lam = fmax(lam, c + fmax(fabs(q[id + ngl2] * Qinv), fabs(q[id + 2 * ngl2] * Qinv)));
        }
        const int next = i + (int)gridDim.x;
        if (next < n && (!tasks || tasks[next].scn == tk.scn)) continue;
        for (int off = 32; off > 0; off >>= 1) lam = fmax(lam, __shfl_xor(lam, off));
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = lam;
        __syncthreads();
        if (threadIdx.x == 0) max_into(S.lmax + src, fmax(fmax(part[0], part[1]), fmax(part[2], part[3])));
        __syncthreads();
        lam = 0.0;
    }
}

// ---------------------------------------------------------------------------------------------
// Artificial viscosity of the scenarios with av = 1.  The element viscosity of a stage's state comes from the
// stage that wrote it (ShockCapturing.okl) or from the learned indicator's pass before the stage
// (esdg_mlp.hip), each viscous element marking itself and its face neighbours with the stage's mark.
// Before each stage: the gradient pass
// (calcGradient + SurfaceKernelGradient + scaleGradient + VolumeKernelViscose) over the marked
// elements; the viscous face fluxes (CollectEdgeDataGradient + calcNumFluxesViscose) of the faces
// of marked elements.  The stage kernel then adds the viscous terms of the marked elements.  The
// same work as the fused schedule's AV passes (esdg_fused.hip), element by element, with the face
// traces read from the state instead of a side-trace buffer: the same bits.
// ---------------------------------------------------------------------------------------------

// Before the sensor pass of prime(): fresh marks, empty lists, no viscosity maximum.
__global__ void k_stage_prime(const StageScn* __restrict__ scns, int nscn, int src, int* mark, int* mcount) {
    if (threadIdx.x == 0) mark[src] = max(mark[0], mark[1]) + STAGE_MARKS;
    for (int i = threadIdx.x; i < 2 * MARK_LISTS * MARK_SLOTS; i += blockDim.x) mcount[i * MARK_STRIDE] = 0;
    for (int s = threadIdx.x; s < nscn; s += blockDim.x)
        if (scns[s].av) scns[s].emax[0] = scns[s].emax[1] = 0ull;
}

template <int LO, int HI>
struct MaxRowLds {
    static constexpr int value = cmax(RowBlock<LO>::EPB * RowBlock<LO>::ES, MaxRowLds<LO + 1, HI>::value);
};
template <int HI>
struct MaxRowLds<HI, HI> {
    static constexpr int value = RowBlock<HI>::EPB * RowBlock<HI>::ES;
};

template <int NGL>
__device__ __forceinline__ void ens_sensor_body(const StageScn& S, int e0, int src, int m, double* sV,
                                                double* sT, double (*sSum)[4], unsigned long long* sMax) {
    if (threadIdx.x < NGL * NGL) sV[threadIdx.x] = glob(S.VdmInv)[threadIdx.x];
    const double v = sensor_rows<NGL>(S.Nelem, e0, S.sc, glob((const double*)S.q[src]), glob(S.B), sV, sT, sSum);
    const int el = threadIdx.x / NGL, r = threadIdx.x % NGL;
    const int e = e0 + el;
    if (el < RowBlock<NGL>::EPB && e < S.Nelem && r == 0) {
        glob(S.visc)[e] = v;
        if (S.visc_plot) glob(S.visc_plot)[e] = v;
        if (v != 0.0)
            for (int s = 0; s < 4; ++s) mark_side(S, e, s, side_record(S, e, s), m, src);
        // non-negative doubles order as their bit patterns; a NaN stays out, as fmax leaves it
        if (v > 0.0) atomicMax(sMax, (unsigned long long)__double_as_longlong(v));
    }
}

// ShockCapturing of the state in buffer src over RowBlock tiles (tasks: {scenario, first element, ngl}), for
// the first stage of a run: the stages evaluate it on the states that they write.  A block's largest
// viscosity enters its scenario's eps_max; the marks are those of stage `stage` (even) of the next step.
template <int LO, int HI>
__global__ void __launch_bounds__(256) k_ens_sensor(const StageScn* __restrict__ scns,
                                                    const StageTask* __restrict__ tasks, int src,
                                                    const int* __restrict__ markp, int stage) {
    __shared__ double sV[HI * HI];
    __shared__ double sT[MaxRowLds<LO, HI>::value];
    __shared__ double sSum[RowBlock<LO>::EPB][4];
    __shared__ unsigned long long sMax;
    const StageTask tk = tasks ? tasks[blockIdx.x]
                               : StageTask{0, (int)blockIdx.x * (256 / scns[0].ngl), scns[0].ngl, 0};
    const StageScn& S = scns[tk.scn];
    const int m = markp[src] + stage;
    if (threadIdx.x == 0) sMax = 0ull;   // published by the sensor's first barrier
    switch (tk.ngl) {
#define ESDG_CASE(n)                                                                          \
    case n:                                                                                   \
        if constexpr (n >= LO && n <= HI) ens_sensor_body<n>(S, tk.e0, src, m, sV, sT, sSum, &sMax); \
        break;
        ESDG_CASE(3) ESDG_CASE(4) ESDG_CASE(5) ESDG_CASE(6) ESDG_CASE(7) ESDG_CASE(8)
#undef ESDG_CASE
        default: break;
    }
    __syncthreads();
    if (threadIdx.x == 0 && sMax) max_into(S.emax + src, __longlong_as_double((long long)sMax));
}

// One list's marked elements, ElemBlock<NGL>::EPB at a time, one thread per node; the elements of a
// block may be of different scenarios, so every element brings its own operators and pointers.
template <int NGL, bool ONE>
__device__ __forceinline__ void ens_grad_body(const StageScn* __restrict__ scns, const int2* __restrict__ list, int cnt,
                                              int blk, int nblk, int src, double* sDh, double* sDs, double* sA,
                                              double* sB, double* sC, double* sE, double* sF, double* sEps) {
    using EB = ElemBlock<NGL>;
    constexpr int NN = NGL * NGL;
    const int el = threadIdx.x / NN, n = threadIdx.x % NN;
    for (int g = blk * EB::EPB; g < cnt; g += nblk * EB::EPB) {
        const bool act = el < EB::EPB && g + el < cnt;
        const int2 me = list[act ? g + el : g];
        const StageScn& S = scns[ONE ? 0 : me.x];
        if (el < EB::EPB) {
            sDh[threadIdx.x] = S.Dhat[n];
            sDs[threadIdx.x] = S.Dstrong[n];
        }
        const AvMesh M{S.q[src], S.Jac, S.Yxi, S.Yeta, S.Xxi, S.Xeta, S.E2E, S.EMS, S.EOR, S.EdgeData,
                       S.nx, S.ny, S.scal, S.bL, S.bR, GatherConsts{S.bc, S.h_zero}, S.geomFace, S.tol, S.gtr, S.Qv};
        const int o = (el < EB::EPB ? el : 0) * NN;
        av_element_block<NGL>(M, TraceFromState{S.q[src]}, me.y, act, act ? S.visc[me.y] : 0.0, sDh + o, sDs + o, sA,
                              sB, sC, sE, sF, sEps);
    }
}

// The gradient pass over the lists of marked elements.  A list's blocks stride over it, so a front
// that crosses one part of a mesh spreads over the chip (one block per 256-element tile worked
// through the tile's marked elements in sequence, 248 us for each launch of ten scenarios).  ONE: a batch of one
// scenario, whose pointers are the same in all lanes, and of one degree, whose registers and LDS are all that is
// held: 43 us where every element of 128 x 128, N = 7, has viscosity and 394 at 400 x 400, with the pointers per lane
// and all degrees in one kernel 60 and 675.
template <int LO, int HI, bool ONE>
__global__ void __launch_bounds__(256) k_ens_grad(const StageScn* __restrict__ scns, MarkLists L, int l0, int l1, int src) {
    __shared__ double sDh[256], sDs[256];
    __shared__ double sA[256], sB[256], sC[256], sE[256];
    __shared__ double sF[ElemBlock<LO>::EPB * 16 * LO];   // (the most at the lowest degree)
    __shared__ double sEps[ElemBlock<LO>::EPB];
    int l = l0;
    while (l + 1 < l1 && (int)blockIdx.x >= L.first[l] + L.blocks[l]) ++l;
    const int blk = (int)blockIdx.x - L.first[l], slot = blk % MARK_SLOTS, cnt = *mark_count(L.count[l], src, slot);
    if (blk >= L.blocks[l]) return;
    const int2* list = L.list[l] + slot * L.cap[l];
    switch (L.ngl[l]) {
#define ESDG_CASE(n)                                                                          \
    case n:                                                                                   \
        if constexpr (n >= LO && n <= HI)                                                     \
            ens_grad_body<n, ONE>(scns, list, cnt, blk / MARK_SLOTS, L.blocks[l] / MARK_SLOTS, src, sDh, sDs, sA, sB, sC, sE, \
                             sF, sEps);                                                       \
        break;
        ESDG_CASE(3) ESDG_CASE(4) ESDG_CASE(5) ESDG_CASE(6) ESDG_CASE(7) ESDG_CASE(8)
#undef ESDG_CASE
        default: break;
    }
}

// The viscous face fluxes over the side nodes of the listed elements; each face node once, by the
// face's left element if that is marked, else by its right one (the faces a marked element reads
// are exactly those).
template <bool ONE>
__global__ void __launch_bounds__(256) k_ens_vface(const StageScn* __restrict__ scns, MarkLists L, int l0, int l1, int src,
                                                   const int* __restrict__ markp, int stage) {
    int l = l0;
    while (l + 1 < l1 && (int)blockIdx.x >= L.first[l] + L.blocks[l]) ++l;
    const int blk = (int)blockIdx.x - L.first[l];
    if (blk >= L.blocks[l]) return;
    const int m = markp[src ^ (stage & 1)] + stage, ngl = L.ngl[l];
    const int slot = blk % MARK_SLOTS;
    const int2* list = L.list[l] + slot * L.cap[l];
    const int64_t items = (int64_t)*mark_count(L.count[l], src, slot) * 4 * ngl;
    for (int64_t it = (int64_t)(blk / MARK_SLOTS) * 256 + threadIdx.x; it < items; it += (int64_t)(L.blocks[l] / MARK_SLOTS) * 256) {
        const int li = (int)(it / (4 * ngl)), rem = (int)(it % (4 * ngl));
        const int side = rem / ngl, i = rem % ngl;
        const int2 me = list[li];
        const StageScn& S = scns[ONE ? 0 : me.x];
        const int f = S.E2E[me.y * 4 + side] - 1;
        const int* E = S.EdgeData + 8 * (int64_t)f;
        const int iel = E[0], ier = E[1], isl = E[2], isr = E[3], rv = E[4], cpuL = E[5], cpuR = E[6];
        const int owner = (cpuL == 0 && S.active[src][iel] == m) ? iel : ier;
        if (me.y != owner) continue;
        viscous_face_node(f, i, ngl, S.geomFace, iel, ier, isl, isr, rv, cpuL, cpuR, S.gtr, S.visc, S.nx, S.ny, S.scal,
                          S.SPV);
    }
}

// One record per element (StageScn::geo) of a mesh whose metrics are the same, bit for bit, at all nodes
// of each element: {Yeta, Xeta, Yxi, Xxi, 1/J, Bx, By, 1 if Bx and By are the same at all nodes}.  *bad is
// set where an element's metrics vary: the mesh then has no records.  One wave per element.
__global__ void __launch_bounds__(64) k_geo_records(int Nelem, int nn, const double* __restrict__ Yeta,
                                                    const double* __restrict__ Xeta, const double* __restrict__ Yxi,
                                                    const double* __restrict__ Xxi, const double* __restrict__ Jac,
                                                    const double* __restrict__ Bx, const double* __restrict__ By,
                                                    double* __restrict__ geo, int* __restrict__ bad) {
    const int n = threadIdx.x;      // nn <= 64
    const double* a[7] = {Yeta, Xeta, Yxi, Xxi, Jac, Bx, By};
    for (int e = blockIdx.x; e < Nelem; e += gridDim.x) {
        // (on a curved mesh the first elements settle it)
        if (__hip_atomic_load(bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
        bool metrics = true, slopes = true;
        double first[7];
        for (int k = 0; k < 7; ++k) {
            const double v = a[k][(int64_t)e * nn + (n < nn ? n : 0)];
            first[k] = a[k][(int64_t)e * nn];
            const bool same = __all(__double_as_longlong(v) == __double_as_longlong(first[k]));
            if (k < 5) metrics = metrics && same;
            else slopes = slopes && same;
        }
        if (n == 0) {
            for (int k = 0; k < 7; ++k) geo[8 * (int64_t)e + k] = first[k];
            geo[8 * (int64_t)e + 7] = slopes ? 1.0 : 0.0;
            if (!metrics) *bad = 1;
        }
    }
}

// One record per face of such a mesh: {nx, ny, scal, bL, bR, -, -, 1 if all five are the same at all
// nodes of the face}.
__global__ void __launch_bounds__(256) k_face_records(int Nfaces, int ngl, const double* __restrict__ nx,
                                                      const double* __restrict__ ny, const double* __restrict__ scal,
                                                      const double* __restrict__ bL, const double* __restrict__ bR,
                                                      double* __restrict__ fgeo) {
    const int f = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (f >= Nfaces) return;
    const double* a[5] = {nx, ny, scal, bL, bR};
    bool same = true;
    for (int k = 0; k < 5; ++k) {
        const double* p = a[k] + (int64_t)f * ngl;
        const long long first = __double_as_longlong(p[0]);
        for (int i = 1; i < ngl; ++i) same = same && __double_as_longlong(p[i]) == first;
        fgeo[8 * (int64_t)f + k] = p[0];
    }
    fgeo[8 * (int64_t)f + 7] = same ? 1.0 : 0.0;
}

// One record per element side (StageScn::srec) from the connectivity arrays.
__global__ void __launch_bounds__(256) k_side_records(int Nelem, const int* __restrict__ E2E, const int* __restrict__ EOR,
                                                      const int* __restrict__ EMS, const int* __restrict__ ED,
                                                      const double* __restrict__ fgeo, int4* __restrict__ rec) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)Nelem * 4) return;
    const int f = E2E[t] - 1;
    const int* E = ED + 8 * (int64_t)f;
    // (of another rank only that it is one matters)
    auto rank = [](int c) { return (unsigned)(min(max(c, -2), 253) + 2); };
    const unsigned w = (unsigned)(E[2] & 3) | ((unsigned)(E[3] & 3) << 2) | ((unsigned)(E[4] & 1) << 4) |
                       ((unsigned)(EOR[t] & 1) << 5) | ((EMS[t] > 0 ? 1u : 0u) << 6) |
                       (rank(E[5]) << 8) | (rank(E[6]) << 16) |
                       ((fgeo && fgeo[8 * (int64_t)f + 7] != 0.0 ? 1u : 0u) << 24);
    rec[t] = make_int4(f, E[0], E[1], (int)w);
}

static int face_records(esdg_ctx* ctx, const StageScn& S, double* fgeo, int4* rec) {
    if (fgeo)
        k_face_records<<<blocks_for(S.Nfaces, 256), 256, 0, ctx->stream>>>(S.Nfaces, S.ngl, S.nx, S.ny, S.scal, S.bL, S.bR,
                                                                           fgeo);
    k_side_records<<<blocks_for((int64_t)S.Nelem * 4, 256), 256, 0, ctx->stream>>>(S.Nelem, S.E2E, S.EOR, S.EMS, S.EdgeData,
                                                                                 fgeo, rec);
    return launch_check(ctx, "face and side records");
}

int StageBatch::refresh_faces(esdg_ctx* ctx) {
    const StageScn& S = host[0];
    return S.fgeo ? face_records(ctx, S, const_cast<double*>(S.fgeo), const_cast<int4*>(S.srec)) : ESDG_OK;
}

int StageBatch::init(esdg_ctx* ctx, const std::vector<StageScn>& scns) {
    host = scns;
    if (scns.empty()) return set_error(ctx, ESDG_ERR_ARG, "the single-kernel stage needs at least one scenario");
    for (const StageScn& S : scns) {
        if (S.ngl < 3 || S.ngl > 8) return set_error(ctx, ESDG_ERR_ARG, "the single-kernel stage supports 2 <= N <= 7");
        if (S.Nelem <= 0) return set_error(ctx, ESDG_ERR_ARG, "the single-kernel stage needs at least one element");
    }
    int rc = ESDG_OK;
    // element and face records, once per distinct mesh and bottom (a mesh with varying metrics has
    // none), and side records, once per distinct connectivity and face records
    auto same_mesh = [](const StageScn& A, const StageScn& B) {
        return A.ngl == B.ngl && A.Nelem == B.Nelem && A.Nfaces == B.Nfaces && A.E2E == B.E2E && A.EOR == B.EOR &&
               A.EMS == B.EMS && A.EdgeData == B.EdgeData && A.Yeta == B.Yeta && A.Xeta == B.Xeta && A.Yxi == B.Yxi &&
               A.Xxi == B.Xxi && A.Jac == B.Jac && A.Bx == B.Bx && A.By == B.By && A.nx == B.nx && A.ny == B.ny &&
               A.scal == B.scal && A.bL == B.bL && A.bR == B.bR;
    };
    auto buffer = [&](size_t bytes) {
        void* d = nullptr;
        if (!rc) rc = esdg_malloc(ctx, &d, bytes);
        if (!rc) rec_bufs.push_back(d);
        return d;
    };
    for (size_t a = 0; a < host.size() && !rc; ++a) {
        StageScn& S = host[a];
        size_t b = 0;
        while (b < a && !same_mesh(host[b], S)) ++b;
        if (b < a) {
            S.geo = host[b].geo;
            S.fgeo = host[b].fgeo;
            S.srec = host[b].srec;
            continue;
        }
        S.geo = S.fgeo = nullptr;
        // one buffer (zero-filled): the flag, the element, face and side records.  (Where the mesh turns out to have
        // no element and face records their part, 2 % of the mesh's arrays, stays unused: an
        // allocation and a free of their own took as long as the passes.)
        int bad = 0;
        char* buf = S.rec ? (char*)S.rec : (char*)buffer(record_bytes(S.Nelem, S.Nfaces));
        int* dbad = (int*)buf;
        double* geo = (double*)(buf + 64);
        double* fgeo = geo + (size_t)S.Nelem * 8;
        int4* d = (int4*)(fgeo + (size_t)S.Nfaces * 8);
        if (rc) break;
        k_geo_records<<<(unsigned)std::min(S.Nelem, 16384), 64, 0, ctx->stream>>>(
            S.Nelem, S.ngl * S.ngl, S.Yeta, S.Xeta, S.Yxi, S.Xxi, S.Jac, S.Bx, S.By, geo, dbad);
        rc = launch_check(ctx, "geometry records");
        if (!rc) rc = esdg_memcpy(ctx, &bad, dbad, sizeof bad, ESDG_D2H);
        if (rc) break;
        rc = face_records(ctx, S, bad ? nullptr : fgeo, d);
        if (!bad) {
            S.geo = geo;
            S.fgeo = fgeo;
        }
        S.srec = d;
    }
    if (rc) return rc;
    rc = hip_check(ctx, hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, ctx->device), "CU count");
    if (rc) return rc;
    has_av = false;
    for (const StageScn& S : scns) has_av = has_av || S.av;
    // the scenario table; marks, list lengths, counts, and the lists (zero-filled), which hold every element of their
    // scenarios at most once a stage and whose total size does not depend on which are learned
    size_t all = 0;
    for (const StageScn& S : host)
        if (S.av) all += mark_elements(S.Nelem);
    const size_t table = (host.size() * sizeof(StageScn) + 63) / 64 * 64;
    char* own = host.size() == 1 ? (char*)host[0].rec : nullptr;
    char* buf = own ? own + record_bytes(host[0].Nelem, host[0].Nfaces) : (char*)buffer(table + (has_av ? mark_bytes(all) : 0));
    if (rc) return rc;
    d_scn = (StageScn*)buf;
    rc = esdg_memcpy(ctx, d_scn, host.data(), host.size() * sizeof(StageScn), ESDG_H2D);
    if (!rc && has_av) {
        const size_t counts = 8 * IND_SLOTS * sizeof(unsigned long long);
        const size_t lengths = 2 * MARK_LISTS * MARK_SLOTS * MARK_STRIDE * sizeof(int);
        buf += table;
        d_mark = (int*)buf;
        d_icount = (unsigned long long*)(buf + 128);
        d_mcount = (int*)(buf + 128 + counts);
        d_mlist = (int2*)(buf + 128 + counts + lengths);
        rc = build_av_tasks(ctx);
    }
    if (!rc) rc = set_schedule(ctx, StageSchedule{});
    return rc;
}

// Element tiles of the AV scenarios for the sensor (RowBlock tiles) and the learned indicator
// (32-element tiles), and the layout of the marked-element lists.
int StageBatch::build_av_tasks(esdg_ctx* ctx) {
    std::vector<StageTask> sens, ind;      // (a single scenario's follow from their index)
    int elements[MARK_LISTS] = {0};
    auto list_of = [](const StageScn& S) { return S.learned ? MARK_LISTS - 1 : S.ngl - 3; };
    for (int s = 0; s < (int)host.size(); ++s) {
        StageScn& S = host[s];
        if (!S.av) continue;
        S.mbase = elements[list_of(S)];
        elements[list_of(S)] += mark_elements(S.Nelem);
        const int ngl = S.ngl;
        if (host.size() == 1) {
        } else if (S.learned)
            for (int e0 = 0; e0 < S.Nelem; e0 += 32) ind.push_back(StageTask{s, e0, ngl, 0});
        else
            for (int e0 = 0; e0 < S.Nelem; e0 += 256 / ngl) sens.push_back(StageTask{s, e0, ngl, 0});
    }
    for (int l = 0; l < MARK_LISTS; ++l) {
        mcap[l] = mark_capacity(elements[l]);
        mfirst[l + 1] = mfirst[l] + (int64_t)mcap[l] * MARK_SLOTS;
    }
    for (int s = 0; s < (int)host.size(); ++s) {
        StageScn& S = host[s];
        S.id = s;
        if (!S.av) continue;
        S.mlist = d_mlist + mfirst[list_of(S)];
        S.mcount = d_mcount + 2 * MARK_SLOTS * MARK_STRIDE * list_of(S);
        S.mcap = mcap[list_of(S)];
    }
    int rcs = esdg_memcpy(ctx, d_scn, host.data(), host.size() * sizeof(StageScn), ESDG_H2D);
    if (rcs) return rcs;
    auto put = [&](const std::vector<StageTask>& v, StageTask*& d, int& n) -> int {
        if (d) esdg_free(ctx, d);
        d = nullptr;
        n = (int)v.size();
        if (v.empty()) return ESDG_OK;
        int rc = esdg_malloc(ctx, (void**)&d, v.size() * sizeof(StageTask));
        if (!rc) rc = esdg_memcpy(ctx, d, v.data(), v.size() * sizeof(StageTask), ESDG_H2D);
        return rc;
    };
    int rc = put(sens, d_sens, nsens);
    if (!rc) rc = put(ind, d_ind, nind);
    if (host.size() == 1) {
        const StageScn& S = host[0];
        const int per = S.learned ? 32 : 256 / S.ngl;
        (S.learned ? nind : nsens) = (S.Nelem + per - 1) / per;
    }
    return rc;
}

int StageBatch::take_counts(esdg_ctx* ctx, unsigned long long c[5]) {
    for (int k = 0; k < 5; ++k) c[k] = 0;
    if (!d_icount) return ESDG_OK;
    unsigned long long all[8 * IND_SLOTS];
    int rc = esdg_memcpy(ctx, all, d_icount, sizeof all, ESDG_D2H);
    if (!rc) rc = esdg_fill(ctx, reinterpret_cast<double*>(d_icount), 0.0, 8 * IND_SLOTS);
    if (!rc) rc = esdg_finish(ctx);
    for (int i = 0; i < IND_SLOTS && !rc; ++i)
        for (int k = 0; k < 5; ++k) c[k] += all[8 * i + k];
    return rc;
}

int StageBatch::put_counts(esdg_ctx* ctx, const unsigned long long c[5]) {
    if (!d_icount) return ESDG_OK;
    int rc = esdg_fill(ctx, reinterpret_cast<double*>(d_icount), 0.0, 8 * IND_SLOTS);
    if (!rc) rc = esdg_memcpy(ctx, d_icount, c, 5 * sizeof c[0], ESDG_H2D);
    return rc;
}

int StageBatch::set_indicator(esdg_ctx* ctx, const esdg_mlp* m, float lo, float hi) {
    if (m && !(lo <= hi)) return set_error(ctx, ESDG_ERR_ARG, "set_indicator: lo > hi");
    int learned = 0;
    for (StageScn& S : host) {
        S.learned = (m && S.av && S.ngl == 8) ? 1 : 0;
        learned += S.learned;
    }
    if (m && !learned)
        return set_error(ctx, ESDG_ERR_ARG, "the learned indicator needs a scenario with N = 7 and artificial viscosity");
    primed = false;
    mlp = m;
    ind_lo = lo;
    ind_hi = hi;
    drop_graphs();
    int rc = ESDG_OK;
    if (has_av) rc = build_av_tasks(ctx);
    else rc = esdg_memcpy(ctx, d_scn, host.data(), host.size() * sizeof(StageScn), ESDG_H2D);
    if (!rc) rc = set_schedule(ctx, sched);   // the stage launches split by group (or not)
    return rc;
}

// A fresh start of the marks (the step counter would wrap): every mark array back to 0.
int StageBatch::reset_marks(esdg_ctx* ctx) {
    int rc = esdg_fill(ctx, reinterpret_cast<double*>(d_mark), 0.0, 8);
    for (const StageScn& S : host)
        for (int* a : {S.active[0], S.active[1]})
            if (!rc && S.av) rc = esdg_fill(ctx, reinterpret_cast<double*>(a), 0.0, ((size_t)S.Nelem + 1) / 2);
    marks_used = 0;
    primed = false;
    return rc;
}

int StageBatch::prime(esdg_ctx* ctx, int src, int stage) {
    {
        KernelScope ks(ctx, "stage_mark");
        k_stage_prime<<<1, 256, 0, ctx->stream>>>(d_scn, (int)host.size(), src, d_mark, d_mcount);
        int rc = launch_check(ctx, "stage_prime");
        if (rc) return rc;
    }
    marks_used += 1;
    if (nsens) {
        KernelScope ks(ctx, "ens_sensor");
        k_ens_sensor<3, 8><<<nsens, 256, 0, ctx->stream>>>(d_scn, d_sens, src, d_mark, stage);
        int rc = launch_check(ctx, "ens_sensor");
        if (rc) return rc;
    }
    primed = true;
    return ESDG_OK;
}

int StageBatch::av_terms(esdg_ctx* ctx, int src, int stage, int l0, int l1, hipStream_t st) {
    // blocks per list: enough for a front's elements in one pass (the lists' lengths are known on
    // the device only), never more than the list could use
    auto lay_out = [&](int cap, auto per_block) {
        MarkLists L{};
        int n = 0;
        for (int l = l0; l < l1; ++l) {
            L.ngl[l] = l == MARK_LISTS - 1 ? 8 : l + 3;
            L.list[l] = d_mlist + mfirst[l];
            L.count[l] = d_mcount + 2 * MARK_SLOTS * MARK_STRIDE * l;
            L.cap[l] = mcap[l];
            L.first[l] = n;
            L.blocks[l] = (int)std::min<int64_t>(cap / MARK_SLOTS, per_block(mcap[l], L.ngl[l])) * MARK_SLOTS;
            n += L.blocks[l];
        }
        return std::make_pair(L, n);
    };
    {
        const auto [L, n] = lay_out(1024, [](int64_t e, int ngl) {
            const int epb = std::max(1, 256 / (ngl * ngl));
            return (e + epb - 1) / epb;
        });
        if (n == 0) return ESDG_OK;
        KernelScope ks(ctx, "ens_grad");
        if (host.size() == 1) {
            switch (host[0].ngl) {
#define ESDG_CASE(g) case g: k_ens_grad<g, g, true><<<n, 256, 0, st>>>(d_scn, L, l0, l1, src); break;
                ESDG_CASE(3) ESDG_CASE(4) ESDG_CASE(5) ESDG_CASE(6) ESDG_CASE(7)
                default: k_ens_grad<8, 8, true><<<n, 256, 0, st>>>(d_scn, L, l0, l1, src); break;
#undef ESDG_CASE
            }
        } else {
            k_ens_grad<3, 8, false><<<n, 256, 0, st>>>(d_scn, L, l0, l1, src);
        }
        int rc = launch_check(ctx, "ens_grad");
        if (rc) return rc;
    }
    const auto [L, n] = lay_out(512, [](int64_t e, int ngl) { return (e * 4 * ngl + 255) / 256; });
    KernelScope ks(ctx, "ens_viscous_face");
    if (host.size() == 1) k_ens_vface<true><<<n, 256, 0, st>>>(d_scn, L, l0, l1, src, d_mark, stage);
    else k_ens_vface<false><<<n, 256, 0, st>>>(d_scn, L, l0, l1, src, d_mark, stage);
    return launch_check(ctx, "ens_viscous_face");
}

void StageBatch::drop_graphs() {
    for (auto& x : exec)
        if (x) { (void)hipGraphExecDestroy(x); x = nullptr; }
}

int StageBatch::set_schedule(esdg_ctx* ctx, const StageSchedule& sc) {
    if (sc.order < 0 || sc.order > 2 || sc.blocks_per_cu < 0 || sc.blocks_per_cu > 64 ||
        (sc.tile != 1 && sc.tile != 2 && sc.tile != 4))
        return set_error(ctx, ESDG_ERR_ARG, "stage schedule: order must be 0..2, blocks_per_cu 0..64, tile 1, 2 or 4");
    const int ns = (int)host.size();
    // scenario visiting order
    std::vector<int> scn(ns);
    for (int s = 0; s < ns; ++s) scn[s] = s;
    if (sc.order == 2 || sc.per_degree)
        std::stable_sort(scn.begin(), scn.end(), [&](int a, int b) { return host[a].ngl > host[b].ngl; });
    std::vector<StageTask> tasks;      // (those of a single scenario follow from their index)
    auto tiles = [&](int s) { const int epw = 64 / host[s].ngl; return (host[s].Nelem + epw - 1) / epw; };
    auto task = [&](int s, int t) { return StageTask{s, t * (64 / host[s].ngl), host[s].ngl, 0}; };
    if (ns == 1) {
    } else if (sc.order == 1) {
        // groups of scenarios on the same geometry, in order of first appearance; tile-major inside
        std::vector<int> done(ns, 0);
        for (int a = 0; a < ns; ++a) {
            const int s0 = scn[a];
            if (done[s0]) continue;
            std::vector<int> grp;
            for (int b = a; b < ns; ++b) {
                const int s1 = scn[b];
                if (!done[s1] && host[s1].Jac == host[s0].Jac && host[s1].ngl == host[s0].ngl &&
                    host[s1].Nelem == host[s0].Nelem) {
                    grp.push_back(s1);
                    done[s1] = 1;
                }
            }
            for (int t = 0; t < tiles(s0); ++t)
                for (int s1 : grp) tasks.push_back(task(s1, t));
        }
    } else {
        for (int s : scn)
            for (int t = 0; t < tiles(s); ++t) tasks.push_back(task(s, t));
    }
    // with both modal-sensor and learned scenarios: the other scenarios' tasks first, then the
    // learned ones', each group in the schedule's order and launched on its own stream
    split = has_av && nsens > 0 && nind > 0;
    const int ntasks = ns == 1 ? tiles(0) : (int)tasks.size();
    int nother = ntasks;
    if (split) {
        std::stable_partition(tasks.begin(), tasks.end(), [&](const StageTask& t) { return !host[t.scn].learned; });
        nother = 0;
        while (nother < (int)tasks.size() && !host[tasks[nother].scn].learned) ++nother;
    }
    // launch ranges
    std::vector<Range> rg;
    int cur_learned = 0;
    auto add_range = [&](int beg, int n, int lo, int hi) {
        if (n <= 0) return;
        Range r{beg, n, lo, hi, n, 0, cur_learned, 1};
        for (int i = beg; i < beg + (ns == 1 ? 1 : n); ++i)
            if (!host[ns == 1 ? 0 : tasks[i].scn].geo) { r.affine = 0; break; }
        // chunks of sc.tile tasks; with xcd every XCD's part is chunked on its own
        const int nch = sc.xcd ? 8 * (((n + 7) / 8 + sc.tile - 1) / sc.tile) : (n + sc.tile - 1) / sc.tile;
        const int pgrid = sc.blocks_per_cu * ncu;
        if (sc.blocks_per_cu > 0 && pgrid < nch && (!sc.xcd || pgrid >= 8)) {
            r.grid = sc.xcd ? (pgrid / 8) * 8 : pgrid;
            r.persistent = 1;
        } else if (sc.tile > 1) {
            r.grid = nch;
            r.persistent = 1;
        }
        rg.push_back(r);
    };
    auto add_group = [&](int g0, int g1) {
        if (ns == 1) {
            add_range(g0, g1 - g0, host[0].ngl, host[0].ngl);
        } else if (sc.per_degree) {
            int beg = g0;
            while (beg < g1) {
                int end = beg;
                while (end < g1 && tasks[end].ngl == tasks[beg].ngl) ++end;
                add_range(beg, end - beg, tasks[beg].ngl, tasks[beg].ngl);
                beg = end;
            }
        } else {
            int lo = 99, hi = 0;
            for (int i = g0; i < g1; ++i) { lo = std::min(lo, tasks[i].ngl); hi = std::max(hi, tasks[i].ngl); }
            add_range(g0, g1 - g0, lo, hi);
        }
    };
    add_group(0, nother);
    cur_learned = 1;
    add_group(nother, ntasks);
    if (ns > 1) {
        if (d_task && ntasks != ntask) {
            esdg_free(ctx, d_task);
            d_task = nullptr;
        }
        int rc = ESDG_OK;
        if (!d_task) rc = esdg_malloc(ctx, (void**)&d_task, tasks.size() * sizeof(StageTask));
        if (!rc) rc = esdg_memcpy(ctx, d_task, tasks.data(), tasks.size() * sizeof(StageTask), ESDG_H2D);
        if (rc) return rc;
    }
    ntask = ntasks;
    ranges = rg;
    sched = sc;
    drop_graphs();
    return ESDG_OK;
}

int StageBatch::lambda(esdg_ctx* ctx, int src) {
    KernelScope ks(ctx, "stage_lambda");
    k_stage_lambda<<<std::min(ntask, 4096), 256, 0, ctx->stream>>>(d_scn, d_task, ntask, src);
    return launch_check(ctx, "stage_lambda");
}

// k_stage_wide where its blocks of five waves are all resident at once: one per CU, two at ngl <= 5, whose waves
// need fewer registers.  us per step with it and with k_stage, runs of 40 steps on Cartesian meshes: 16 x 16, N = 4,
// 38 and 61, 48 x 48 43 and 64, 64 x 64 (342 tasks) 67 and 72; 16 x 16, N = 7, 55 and 77, 45 x 45 (254 tasks) 63 and
// 84.  Beyond it k_stage has more waves at work: 56 x 56, N = 7 (392 tasks) 110 and 91, 64 x 64, N = 5 (410 tasks) 82
// and 79, 80 x 80, N = 4 (534 tasks) 89 and 79.
static constexpr int wide_blocks_per_cu(int ngl) { return ngl <= 5 ? 2 : 1; }

template <int LO, int HI, bool AV>
static void launch_stage(hipStream_t st, const StageBatch& b, const StageBatch::Range& r, int src, double rkA,
                         double rkC, int last, int stage) {
    const StageTask* tasks = b.d_task ? b.d_task + r.beg : nullptr;
    if constexpr (LO == HI) {
        if (!r.persistent && r.n <= b.ncu * wide_blocks_per_cu(LO)) {
            if (r.affine)
                k_stage_wide<LO, AV, true><<<r.grid, 320, 0, st>>>(b.d_scn, tasks, r.n, b.sched.xcd, src, rkA, rkC, last,
                                                                   b.d_mark, stage);
            else
                k_stage_wide<LO, AV, false><<<r.grid, 320, 0, st>>>(b.d_scn, tasks, r.n, b.sched.xcd, src, rkA, rkC, last,
                                                                    b.d_mark, stage);
            return;
        }
    }
    if (r.persistent)
        // (the records of a Cartesian mesh serve the launches of one block per task)
        k_stage<LO, HI, true, AV, false><<<r.grid, 64, 0, st>>>(b.d_scn, tasks, r.n, b.sched.xcd, b.sched.tile,
                                                                src, rkA, rkC, last, b.d_mark, stage);
    else if (r.affine)
        k_stage<LO, HI, false, AV, true><<<r.grid, 64, 0, st>>>(b.d_scn, tasks, r.n, b.sched.xcd, 1, src, rkA,
                                                                rkC, last, b.d_mark, stage);
    else
        k_stage<LO, HI, false, AV, false><<<r.grid, 64, 0, st>>>(b.d_scn, tasks, r.n, b.sched.xcd, 1, src, rkA,
                                                                 rkC, last, b.d_mark, stage);
}

template <bool AV>
static void launch_ranges(hipStream_t st, const StageBatch& b, const StageBatch::Range& r, int src, double rkA,
                          double rkC, int last, int stage) {
    if (r.lo != r.hi) launch_stage<3, 8, AV>(st, b, r, src, rkA, rkC, last, stage);
    else switch (r.lo) {
        case 3: launch_stage<3, 3, AV>(st, b, r, src, rkA, rkC, last, stage); break;
        case 4: launch_stage<4, 4, AV>(st, b, r, src, rkA, rkC, last, stage); break;
        case 5: launch_stage<5, 5, AV>(st, b, r, src, rkA, rkC, last, stage); break;
        case 6: launch_stage<6, 6, AV>(st, b, r, src, rkA, rkC, last, stage); break;
        case 7: launch_stage<7, 7, AV>(st, b, r, src, rkA, rkC, last, stage); break;
        default: launch_stage<8, 8, AV>(st, b, r, src, rkA, rkC, last, stage); break;
    }
}

int StageBatch::indicator(esdg_ctx* ctx, int src, int s) {
    if (!nind) return ESDG_OK;
    return mlp_ensemble_indicator(ctx, mlp, d_scn, d_ind, nind, src, d_mark, s, ind_lo, ind_hi, ind_audit, d_icount);
}

int StageBatch::launch_all(esdg_ctx* ctx, int src, double A, double C, int last, int s) {
    for (const Range& r : ranges) {
        KernelScope ks(ctx, "stage");
        if (has_av) launch_ranges<true>(ctx->stream, *this, r, src, A, C, last, s);
        else launch_ranges<false>(ctx->stream, *this, r, src, A, C, last, s);
        const int rc = launch_check(ctx, "stage");
        if (rc) return rc;
    }
    return ESDG_OK;
}

int StageBatch::step(esdg_ctx* ctx, const double* A, const double* C, int stages, int& src) {
    if (nind && !mlp) return set_error(ctx, ESDG_ERR_STATE, "learned scenarios without a network");
    // the learned scenarios' viscosity of the step's state (its maximum enters the dt; the others' is
    // there already)
    int rc = indicator(ctx, src, 0);
    if (rc) return rc;
    for (int s = 0; s < stages; ++s) {
        const int last = (s == stages - 1);
        if (split && ctx->side && !ctx->profile) {
            // the other scenarios on the second stream, the learned ones on the main stream
            (void)hipEventRecord(ctx->fork, ctx->stream);
            (void)hipStreamWaitEvent(ctx->side, ctx->fork, 0);
            rc = av_terms(ctx, src, s, 0, MARK_LISTS - 1, ctx->side);
            for (const Range& r : ranges)
                if (!rc && !r.learned) {
                    launch_ranges<true>(ctx->side, *this, r, src, A[s], C[s], last, s);
                    rc = launch_check(ctx, "stage");
                }
            (void)hipEventRecord(ctx->join, ctx->side);
            if (!rc && s > 0) rc = indicator(ctx, src, s);
            if (!rc) rc = av_terms(ctx, src, s, MARK_LISTS - 1, MARK_LISTS, ctx->stream);
            for (const Range& r : ranges)
                if (!rc && r.learned) {
                    launch_ranges<true>(ctx->stream, *this, r, src, A[s], C[s], last, s);
                    rc = launch_check(ctx, "stage");
                }
            (void)hipStreamWaitEvent(ctx->stream, ctx->join, 0);
            if (rc) return rc;
            src ^= 1;
            continue;
        }
        if (has_av) {
            if (s > 0) rc = indicator(ctx, src, s);
            if (!rc) rc = av_terms(ctx, src, s, 0, MARK_LISTS, ctx->stream);
            if (rc) return rc;
        }
        rc = launch_all(ctx, src, A[s], C[s], last, s);
        if (rc) return rc;
        src ^= 1;
    }
    return ESDG_OK;
}

// Everything of that stage is computed anew from the state before it, the viscosities and marks too, so it writes the
// same bits as it did.  Its clock is in the half that the good step left (ck: the clock after that step).
int StageBatch::repeat_last_stage(esdg_ctx* ctx, const double* A, const double* C, int stages, int dst, const double* ck) {
    const int src = dst ^ 1, s = stages - 1;
    const double clock[8] = {ck[3], ck[1], ck[2], ck[3], 0.0, 0.0, 1.0, ck[7]};
    unsigned long long counts[5];
    int rc = esdg_memcpy(ctx, host[0].clock + 8 * dst, clock, sizeof clock, ESDG_H2D);
    if (!rc) rc = take_counts(ctx, counts);
    if (!rc && has_av) rc = prime(ctx, src, s);
    if (!rc) rc = indicator(ctx, src, s);
    if (!rc && has_av) rc = av_terms(ctx, src, s, 0, MARK_LISTS, ctx->stream);
    if (!rc) rc = launch_all(ctx, src, A[s], C[s], 1, s);
    // the network's viscosities are those of the state that the failed step started from
    if (!rc) rc = indicator(ctx, dst, 0);
    if (!rc) rc = put_counts(ctx, counts);
    primed = false;
    return rc;
}

int StageBatch::capture(esdg_ctx* ctx, const double* A, const double* C, int stages, int start) {
    if (hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal) != hipSuccess) {
        (void)hipGetLastError();
        graph_ok = false;
        return ESDG_OK;
    }
    int rc = ESDG_OK, src = start;
    for (int k = 0; k < 2 && !rc; ++k) rc = step(ctx, A, C, stages, src);
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(ctx->stream, &g);
    if (!rc && (e != hipSuccess || !g || hipGraphInstantiate(&exec[start], g, nullptr, nullptr, 0) != hipSuccess)) {
        (void)hipGetLastError();
        exec[start] = nullptr;
        graph_ok = false;
    }
    if (g) (void)hipGraphDestroy(g);
    return rc;
}

int StageBatch::run(esdg_ctx* ctx, const double* A, const double* C, int stages, int steps, int& src) {
    int n = 0;
    if (has_av) {
        // marks advance by STAGE_MARKS per step: start them afresh long before the int would wrap
        int rc = marks_used + (int64_t)steps + 2 > (int64_t)(1 << 27) ? reset_marks(ctx) : ESDG_OK;
        if (!rc && !primed) rc = prime(ctx, src);
        if (rc) return rc;
        marks_used += steps;
    }
    const int before = issued;
    issued = (int)std::min<int64_t>((int64_t)issued + steps, 1 << 20);
    if (sched.graph && graph_ok && !ctx->profile && steps >= 2 && (exec[src] || std::max(steps, before) >= EAGER_STEPS)) {
        // two steps flip the buffers an even number of times, so the graph that starts from buffer
        // `src` ends there and can be replayed
        if (!exec[src]) {
            const int rc = capture(ctx, A, C, stages, src);
            if (rc) return rc;
        }
        for (; exec[src] && n + 2 <= steps; n += 2) {
            int rc = hip_check(ctx, hipGraphLaunch(exec[src], ctx->stream), "graph launch");
            if (rc) return rc;
        }
    }
    for (; n < steps; ++n) {
        int rc = step(ctx, A, C, stages, src);
        if (rc) return rc;
    }
    return ESDG_OK;
}

void StageBatch::release(esdg_ctx* ctx) {
    drop_graphs();
    for (StageTask** p : {&d_task, &d_sens, &d_ind})
        if (*p) { esdg_free(ctx, *p); *p = nullptr; }
    for (void* p : rec_bufs) esdg_free(ctx, p);
    rec_bufs.clear();
    d_mlist = nullptr;
    d_mcount = nullptr;
    d_scn = nullptr;
    d_mark = nullptr;
    d_icount = nullptr;
}

}  // namespace esdg
