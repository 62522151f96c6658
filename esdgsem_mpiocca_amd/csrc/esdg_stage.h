// esdg_stage.h -- element-centric single-kernel RK stage over a batch of scenarios.
//
// One launch per RK stage covers every element of every scenario in the batch.  A block (one
// wave) owns EPW = 64/ngl elements of one scenario (a task); inside, the degree of that scenario
// selects the instantiation.  Each element computes the entropy-stable fluxes of its own four
// sides from the stage-start state (the neighbour's trace is read from the same buffer, so the two
// elements of a face produce identical bits), then the flux-differencing volume term, the surface
// lift, the low-storage RK step into the other state buffer and, on request, the positivity
// limiter, the shock sensor and the wave speed of the new state (the next stage's viscosity and the next
// step's lambda_max, reduced per scenario with an atomic max).  dt is computed on the device; a whole step needs no host synchronisation,
// so steps are captured in a hipGraph.
#pragma once

#include <vector>

#include "esdg_device.h"
#include "esdg_internal.h"

struct esdg_mlp;

namespace esdg {

struct StageScn {
    int ngl, Nelem, Nfaces, ES, num_flux, positivity, bc;
    double g, geomFace, tol, zero_tol, h_zero;
    double dti;         // (min_ele_size / ngl) * CFL            (dt_i = dti / lambda_max)
    double T;
    const double *Jac, *Yxi, *Yeta, *Xxi, *Xeta, *Bx, *By, *D, *nx, *ny, *scal, *bL, *bR, *EleSizes, *GLw;
    const int *EdgeData, *E2E, *EMS, *EOR;
    double* q[2];       // ping-pong state buffers
    double* gRK;
    // Of the clock, the maxima and the marks there are two, used by steps in turn: a step that starts from the
    // state in buffer p takes half p and leaves the other half for the next (the stages of a step are odd
    // in number, so that one starts from buffer p ^ 1).
    double* clock;      // 2 x 8: [0] dt of the current step (-1 or -2: it changes nothing; 0: a failed scenario), [1] t,
                        // [2] steps taken, [3] dt of the last step taken, [4] 1 if a dt was not positive
                        // and finite ([5] that dt), [6] 1 in the step that brings [2] to [7] or t to T: it stores gRK to the end
    unsigned long long* lmax;   // 2: bit pattern of max lambda (non-negative doubles order as integers)
    // artificial viscosity (av = 1): the modal sensor, or with learned = 1 (N = 7) the learned
    // indicator with the sensor as fallback, evaluated on each stage's state; BR1 gradients and the
    // viscous terms only where viscosity is in reach (active[e] == the stage's mark)
    int av, learned;
    double dvc;         // DFL / ngl^2 * min_ele_size^2            (dt_v = dvc / eps_max)
    SensorConsts sc;
    const double *B, *VdmInv, *Dhat, *Dstrong;
    double* visc;       // element viscosity of the stage's state [Nelem]
    double* gtr;        // side traces of the scaled velocity gradients [Nelem][4][4][ngl]
    double* Qv;         // viscous volume term [Nelem][2][ngl^2] (hu, hv)
    double* SPV;        // viscous face fluxes [Nfaces][2][ngl]
    double* visc_plot;  // its copy (may be null)
    // active[b][e] == the stage's mark: viscosity on the element or a face neighbour in the state of
    // buffer b.  Those elements, each once, with those of every scenario of the same degree and
    // indicator (learned or not), as {scenario, element} in MARK_SLOTS parts of a list: part s is
    // mlist[s mcap .. s mcap + mark_count(mcount, b, s))
    int* active[2];
    int2* mlist;
    int* mcount;
    int mcap, mbase;    // the scenarios of a list number their elements one after another: this one's from mbase on
    int id;             // this scenario's index in the batch
    int freeze;         // after a dt that was not positive and finite: 1 both state buffers stay as they are, 0
                        // the state takes q + 0 gRK
    // a single solver's buffers (each may be null): the element wave speeds of the state after a step,
    // and the analysis buffers, advanced after every step
    double *lam, *arrival, *maxelev;
    unsigned long long* emax;   // 2: bit pattern of the step's max viscosity
    // per element side, what its face flux needs from the connectivity (built by StageBatch::init
    // from E2E, EOR, EMS and EdgeData; one record per side, shared by the scenarios of a mesh):
    // x face, y EdgeData[0] (left element), z EdgeData[1] (right element), w bits: [0,2) left
    // side, [2,4) right side, 4 EdgeData[4] (reversed), 5 EOR, 6 EMS > 0, [8,16) EdgeData[5] + 2,
    // [16,24) EdgeData[6] + 2, 24 the face's geometry is one record of fgeo
    const int4* srec;
    // one record per element and per face of a mesh with element-wise constant metrics (else null)
    const double *geo, *fgeo;
    void* rec;          // batch_bytes of zeroed memory for a batch of this scenario alone, or null: StageBatch::init
                        // allocates it
};

// bytes of a mesh's records
inline size_t record_bytes(int Nelem, int Nfaces) { return 64 + ((size_t)Nelem * 2 + Nfaces) * 64; }

struct StageTask {
    int scn, e0, ngl, pad;
};

// max of a non-negative double into a cell (non-negative doubles order as their bit patterns).  Most blocks
// find a larger value there already and leave the cell alone: atomics of all blocks on one cell queue
// up at about 12 ns each.
__device__ __forceinline__ void max_into(unsigned long long* cell, double m) {
    const unsigned long long bits = (unsigned long long)__double_as_longlong(m);
    if (bits > __hip_atomic_load(cell, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(cell, bits);
}

// The part of its list that an element goes to, and the length of a part.  One length for all was a queue: where every
// element has viscosity the stage took 1057 us at 300 x 300, N = 4, and 223 at 128 x 128, N = 7, and takes 128 and 51 with
// 64 lengths in cache lines of their own.  Four consecutive elements go together (a group of the gradient pass at
// N = 7); any 256 consecutive ones are dealt out evenly, the higher bits keep a front that crosses the rows of a mesh
// from meeting in few parts.  k counts over all scenarios of the list, so that many small meshes fill the parts evenly
// too (numbered mesh by mesh, 512 of 4 x 4 elements met in four parts: 707 us per step instead of 213).
constexpr int MARK_SLOTS = 64, MARK_STRIDE = 16;
__host__ __device__ constexpr int mark_capacity(int elements) { return 4 * ((elements + 255) / 256); }
constexpr int mark_elements(int Nelem) { return (Nelem + 3) / 4 * 4; }     // a scenario's share of the numbers
__host__ __device__ constexpr int mark_slot(int k) { return ((k >> 2) ^ (k >> 8) ^ (k >> 14) ^ (k >> 20)) & (MARK_SLOTS - 1); }
constexpr bool deals_out(int first) {      // 256 elements from `first`: four to each part
    int n[MARK_SLOTS] = {};
    for (int k = 0; k < 256; ++k) n[mark_slot(first + k)] += 1;
    for (int c : n)
        if (c != 4) return false;
    return true;
}
static_assert(deals_out(0) && deals_out(256) && deals_out(77 * 256) && deals_out(0x2a500 * 256), "a part holds mark_capacity elements");
template <class P>
__device__ __forceinline__ P mark_count(P mcount, int b, int slot) { return mcount + (b * MARK_SLOTS + slot) * MARK_STRIDE; }

// An element with viscosity in the state of buffer b marks itself and its face neighbours for the stage that
// starts from it (the elements whose viscous terms can be non-zero), as the fused face pass does for both
// elements of every face with viscosity on either side.  The first to mark an element also lists it.
__device__ __forceinline__ void mark_element(const StageScn& S, int k, int m, int b) {
    if (atomicExch(S.active[b] + k, m) != m) {
        const int s = mark_slot(S.mbase + k);
        S.mlist[s * S.mcap + atomicAdd(mark_count(S.mcount, b, s), 1)] = make_int2(S.id, k);
    }
}
// Side `side` of element e (record R, StageScn::srec): the neighbour there, and with side 0 the element itself.
__device__ __forceinline__ void mark_side(const StageScn& S, int e, int side, const int4& R, int m, int b) {
    const int cpuL = (int)(((unsigned)R.w >> 8) & 255u) - 2, cpuR = (int)(((unsigned)R.w >> 16) & 255u) - 2;
    if (side == 0) mark_element(S, e, m, b);
    if (cpuL == 0 && R.y != e) mark_element(S, R.y, m, b);
    if (cpuR == 0 && R.z != e) mark_element(S, R.z, m, b);
}
__device__ __forceinline__ int4 side_record(const StageScn& S, int e, int side) {
    // one 16-byte load (a vector type: int4's assignment would take a generic reference)
    using i4v = int __attribute__((ext_vector_type(4)));
    const i4v v = ((gptr<const i4v>)glob(S.srec))[(int64_t)e * 4 + side];
    return make_int4(v.x, v.y, v.z, v.w);
}

// The mark of a stage: the step's base (advanced by STAGE_MARKS at each step, on the device, so that
// replays of a captured step take fresh marks) plus the stage.
constexpr int STAGE_MARKS = 8;
constexpr int IND_SLOTS = 64;

// The marked-element lists of a batch: one for the modal-sensor scenarios of each degree (ngl - 3)
// and one for the learned ones (MARK_LISTS - 1).  A pass over them takes, of each list, the blocks
// [first, first + blocks) of its grid, every MARK_SLOTS-th of them for the same part.
constexpr int MARK_LISTS = 7;
struct MarkLists {
    const int2* list[MARK_LISTS];
    const int* count[MARK_LISTS];
    int ngl[MARK_LISTS], first[MARK_LISTS], blocks[MARK_LISTS], cap[MARK_LISTS];
};

// bytes of a batch's marks, counts and marked-element lists, whose scenarios have `elements` numbers in all (each list
// is rounded up to 256)
inline size_t mark_bytes(size_t elements) {
    return 128 + 8 * IND_SLOTS * sizeof(unsigned long long) + 2 * MARK_LISTS * MARK_SLOTS * MARK_STRIDE * sizeof(int) +
           (elements + 256 * MARK_LISTS) * sizeof(int2);
}
// bytes of what a batch of one scenario keeps beside the scenario's arrays (StageScn::rec): its records, its entry of the
// scenario table, its marks
inline size_t batch_bytes(int Nelem, int Nfaces, bool av) {
    return record_bytes(Nelem, Nfaces) + (sizeof(StageScn) + 63) / 64 * 64 +
           (av ? mark_bytes(mark_elements(Nelem)) : 0);
}

// How the tasks of a stage are ordered and launched (the autotuner's search space).
struct StageSchedule {
    int order = 0;          // 0 scenario by scenario; 1 tiles of geometry-sharing scenarios
                            // interleaved (tile-major); 2 degree descending, then scenario by scenario
    int blocks_per_cu = 0;  // 0: one block per task; k > 0: persistent grid of k blocks per CU
    int per_degree = 0;     // 1: one launch per degree group instead of one mixed-degree launch
    int xcd = 0;            // 1: each XCD takes a contiguous range of the task list
    int graph = 1;          // replay pairs of steps from a captured hipGraph
    int tile = 1;           // consecutive tasks (element groups of 64/ngl elements) per block: 1, 2 or 4
};

// Host side: device copies of the scenario table and the task list, plus the per-step sequence.
class StageBatch {
  public:
    int init(esdg_ctx* ctx, const std::vector<StageScn>& scns);
    int set_schedule(esdg_ctx* ctx, const StageSchedule& sc);
    // a batch of one scenario: its face records anew, after something has written the arrays they are made from
    int refresh_faces(esdg_ctx* ctx);
    // initial lambda_max of every scenario from the state in buffer `src`
    int lambda(esdg_ctx* ctx, int src);
    // the sensor, marks and viscosity maximum of the state in buffer src; run() calls it when `primed`
    // is not set, which whoever changes the state, or which scenarios are learned, clears.  stage (even): the
    // stage of the next step that the marks are for
    int prime(esdg_ctx* ctx, int src, int stage = 0);
    bool primed = false;
    // steps that run() has been asked for (as far as it matters).  A captured pair of steps takes about 100 us to
    // capture and instantiate: a batch's first EAGER_STEPS, unless asked for at once, are launched one by one.
    int issued = 0;
    static constexpr int EAGER_STEPS = 8;
    // one time step: the RK stages, the first of which forms dt [each after its viscous terms]; src flips
    // once per stage
    int step(esdg_ctx* ctx, const double* A, const double* C, int stages, int& src);
    // `steps` steps: pairs of steps replayed from a captured graph (schedule.graph), the rest eager
    int run(esdg_ctx* ctx, const double* A, const double* C, int stages, int steps, int& src);
    // A batch of one scenario that freezes a failed state, after a run that failed: the last stage of the last good
    // step again, from buffer dst ^ 1 into buffer dst, for the RK register, which a step stores to the end only
    // where the run is known to end with it.  ck: the clock that the run left.
    int repeat_last_stage(esdg_ctx* ctx, const double* A, const double* C, int stages, int dst, const double* ck);
    void release(esdg_ctx* ctx);

    struct Range {
        int beg, n, lo, hi, grid, persistent;
        int learned;   // 1: the tasks of learned-indicator scenarios (see `split`)
        int affine;    // 1: every scenario of the range has element records (StageScn::geo)
    };
    std::vector<StageScn> host;
    StageSchedule sched;
    std::vector<Range> ranges;
    StageScn* d_scn = nullptr;
    StageTask* d_task = nullptr;
    int ntask = 0;
    int ncu = 0;
    hipGraphExec_t exec[2] = {nullptr, nullptr};   // graph of two steps, one per starting parity
    // artificial viscosity: element tiles of the AV scenarios for the sensor (row tiles) and the
    // learned indicator (32-element tiles of learned scenarios); the gradient and the viscous face
    // pass run over the lists of marked elements; the step's mark counter lives on the device
    // (graph replays advance it)
    bool has_av = false;
    StageTask *d_sens = nullptr, *d_ind = nullptr;
    int nsens = 0, nind = 0;
    int2* d_mlist = nullptr;                       // the marked-element lists, one after another
    int* d_mcount = nullptr;                       // MARK_LISTS x 2 x MARK_SLOTS lengths, MARK_STRIDE apart
    int mcap[MARK_LISTS] = {0};                    // elements that a part of each list has room for
    int64_t mfirst[MARK_LISTS + 1] = {0};          // where each list starts in d_mlist
    // With both modal-sensor and learned scenarios the stage runs as two streams of work: the
    // other scenarios (sensor pass, their AV terms, their stage launches) on the second stream and
    // the learned ones (indicator pass, AV terms, stage launches) on the main stream, so the
    // indicator overlaps the other scenarios' stage.  Their marked elements are in lists of their own.
    bool split = false;
    int* d_mark = nullptr;
    // the learned indicator's 5 counts: IND_SLOTS copies, 8 words apart, to be added
    unsigned long long* d_icount = nullptr;
    int take_counts(esdg_ctx* ctx, unsigned long long c[5]);   // since the last call
    int put_counts(esdg_ctx* ctx, const unsigned long long c[5]);
    const esdg_mlp* mlp = nullptr;
    float ind_lo = 0.5f, ind_hi = 0.5f;
    int ind_audit = 0;
    int64_t marks_used = 0;
    // the learned indicator for the AV scenarios with N = 7 (m = null: the modal sensor everywhere)
    int set_indicator(esdg_ctx* ctx, const esdg_mlp* m, float lo, float hi);

    void drop_graphs();

  private:
    std::vector<void*> rec_bufs;    // allocations: the records of each distinct mesh; table, marks, lists and counts
    bool graph_ok = true;           // no capture has been refused
    // two steps from buffer `start` into exec[start], without running them.  A capture that the runtime refuses is no
    // error: exec[start] stays null and this batch's steps are launched one by one.
    int capture(esdg_ctx* ctx, const double* A, const double* C, int stages, int start);
    int build_av_tasks(esdg_ctx* ctx);
    int reset_marks(esdg_ctx* ctx);
    // the learned scenarios' viscosities and marks of the state in buffer src, for stage s
    int indicator(esdg_ctx* ctx, int src, int s);
    // the stage's launches, one after another on the main stream
    int launch_all(esdg_ctx* ctx, int src, double A, double C, int last, int s);
    // gradients, viscous volume and face terms of the marked elements, of the lists [l0, l1), on
    // stream st
    int av_terms(esdg_ctx* ctx, int src, int stage, int l0, int l1, hipStream_t st);
};

}  // namespace esdg
