// Device-resident AMG hierarchy shared by the single-vector path
// (hier.hip) and the multi-vector path (block.hip).
#pragma once

#include <functional>
#include <vector>

#include "common.hpp"

struct ramd_hier_s;

namespace ramd {

// temp: a product that is only multiplied by other sparse matrices, or read
ramd_csr_s* spgemm(ramd_csr_s* A, ramd_csr_s* B, bool temp = false);
ramd_csr_s* galerkin(ramd_csr_s* A, ramd_csr_s* P);

struct Level {
    ramd_csr_s* A = nullptr;  // diagonal first
    ramd_csr_s* P = nullptr;  // n_l x n_{l+1}
    ramd_csr_s* R = nullptr;  // P^T (owned by P)
    double* diag = nullptr;   // a_ii (0 where absent)
    double *x = nullptr, *b = nullptr, *t = nullptr, *r = nullptr;
    float* diag32 = nullptr;
    float *x32 = nullptr, *b32 = nullptr, *t32 = nullptr, *r32 = nullptr;
    std::vector<int> states;
    int n = 0;
    // multicolour smoothers: rows of colour c are color_rows[color_ptr[c] ..
    // color_ptr[c+1]) (device), ascending
    std::vector<int> color_ptr;
    int* color_rows = nullptr;
};

// Largest coarse system solved by one wavefront (LU staged in LDS).
constexpr int kCoarseWave = 64;

// Lane `lane`'s value of a double held by lane j (j uniform).
__device__ __forceinline__ double lane_value(double v, int j)
{
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(b & 0xffffffffll), j);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(b >> 32), j);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// The substitutions of coarse_solve_wave: lane `lane` of the wavefront
// holds the permuted b_i (i = lane), the LU factors are in ls; returns x_i.
// Every lane of the wavefront calls it.  A chain of n + n dependent steps of
// one wavefront, bound by its instruction issue: b_j goes to all lanes
// through readlane (a scalar register; shuffles through LDS cost about 100
// cycles per step more), the factors' columns are read from LDS four steps
// at a time, ahead of the chain, and there is no branch inside (steps past n
// change nothing).  n = 34: 3000 cycles forward, 7300 back; with the
// division by Markstein's reciprocal form instead of the general one 10100.
__device__ __forceinline__ double coarse_lu_lane(int n, const double* ls, double v, int lane)
{
    constexpr int U = 4;
    const int row = lane < n ? lane : n - 1;
#pragma unroll 1
    for (int j0 = 0; j0 < n; j0 += U) {
        double c[U];
#pragma unroll
        for (int u = 0; u < U; u++) c[u] = ls[row + min(j0 + u, n - 1) * n];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const double bj = lane_value(v, j0 + u);
            const double t = v - bj * c[u];
            v = lane > j0 + u ? t : v;  // lanes past n hold nothing
        }
    }
#pragma unroll 1
    for (int j0 = (n - 1) / U * U; j0 >= 0; j0 -= U) {
        double c[U];
#pragma unroll
        for (int u = 0; u < U; u++) c[u] = ls[row + min(j0 + u, n - 1) * n];
#pragma unroll
        for (int u = U - 1; u >= 0; u--) {
            const int j = j0 + u;
            const double q = v / c[u];  // of use on lane j: row j of column j, the pivot
            v = lane == j ? q : v;
            const double bj = lane_value(v, j);
            const double t = v - bj * c[u];
            v = lane < (j < n ? j : 0) ? t : v;
        }
    }
    return v;
}

// dgetrs_('N') on one right-hand side by one wavefront, n <= kCoarseWave:
// lane i holds b_perm[i] (perm: the row swaps applied in order); the
// unit-lower and the upper substitution run in the reference BLAS column
// order with the same operations per entry as the workgroup kernel
// (b_i -= b_j * l_ij; b_j /= u_jj), so the result is bit-identical.  b and x
// are read and written with element stride `stride`; `ls` is n*n doubles of
// LDS.  All 64 lanes must call it.
template <typename TB, typename TX>
__device__ __forceinline__ void coarse_solve_wave(int n, const double* __restrict__ lu, const int* __restrict__ perm,
                                                  const TB* __restrict__ b, TX* __restrict__ x, size_t stride,
                                                  double* ls)
{
    const int lane = threadIdx.x;
    double v = lane < n ? (double)b[(size_t)perm[lane] * stride] : 0.0;
    // sixteen loads in flight per lane
    constexpr int U = 16;
    for (int t0 = lane; t0 < n * n; t0 += 64 * U) {
        double c[U];
#pragma unroll
        for (int u = 0; u < U; u++) c[u] = lu[min(t0 + 64 * u, n * n - 1)];
#pragma unroll
        for (int u = 0; u < U; u++)
            if (t0 + 64 * u < n * n) ls[t0 + 64 * u] = c[u];
    }
    __syncthreads();
    v = coarse_lu_lane(n, ls, v, lane);
    if (lane < n) x[(size_t)lane * stride] = (TX)v;
}

// Device setup steps (setup_gpu.hip), bit-identical to the host ones.
// (temp: S is only read by the other setup steps)
ramd_csr_s* gpu_classical_strength(ramd_csr_s* A, double theta, bool temp = false);
ramd_csr_s* gpu_symmetric_strength(ramd_csr_s* A, double theta, bool temp = false);
// PMIS on the device; prior_states (host, n; nullptr for plain PMIS) are
// states an earlier pass decided (HMIS), applied before the first round
void gpu_split_pmis(const ramd_csr_s* S, const double* weights, int* states, const int* prior_states = nullptr);
// CLJP on the device (prior_states: Falgout's Ruge-Stuben states, or nullptr)
void gpu_split_cljp(const ramd_csr_s* S, const double* weights, int* states, const int* prior_states = nullptr);
ramd_csr_s* gpu_mod_classical_interpolation(const ramd_csr_s* A, const ramd_csr_s* S, const int* states_d,
                                            const std::vector<int>& states_h);
ramd_csr_s* gpu_direct_interpolation(const ramd_csr_s* A, const ramd_csr_s* S, const int* states_d,
                                     const std::vector<int>& states_h);
ramd_csr_s* gpu_extended_interpolation(const ramd_csr_s* A, const ramd_csr_s* S, const int* states_d,
                                       const std::vector<int>& states_h, double filter);
// Smoothed aggregation's setup steps on the device, with the host
// restatement's results: MIS-2 of S (weights: host, n) into states (device);
// aggregation of A and S (both stored sorted, diagonal first) into agg
// (device; the root row or -1; rand_vals: host, n, or nullptr for zeros),
// returning the number of aggregates; the Jacobi prolongation's scaled
// operator and its subtraction P - Q.
void gpu_mis2(const ramd_csr_s* S, const double* weights, int* states);
int gpu_aggregate(const ramd_csr_s* A, const ramd_csr_s* S, const int* states, int* agg,
                  const double* rand_vals = nullptr);
// fit_candidates with one candidate: T (n x n_aggs) from the aggregates
// (device agg_d and its host copy) and the candidate B_d (device, n); the
// aggregate norms go to R_d (device, n_aggs)
ramd_csr_s* gpu_fit_candidates(ramd_ctx ctx, int n, int n_aggs, const int* agg_d, const std::vector<int>& agg_h,
                               const double* B_d, double* R_d);
ramd_csr_s* gpu_sa_scaled_operator(const ramd_csr_s* A, double omega);
ramd_csr_s* gpu_sa_subtract(const ramd_csr_s* P, const ramd_csr_s* Q);

// One FP64 V-cycle from x = 0 (ParMultilevel::cycle on the fine level).
void vcycle_from_zero(ramd_hier_s* h, double* x, const double* b);

// Coarse tail (tail.hip): one operation of the tail's list.  Offsets are
// into the workgroup's LDS vectors; the matrix's slices of 64 rows start at
// entry slice0 of the slice table (-1: no matrix).
enum TailType { kTailSpmv, kTailSpmvJfz, kTailResidual, kTailJacobi, kTailAdd, kTailFill, kTailCoarse };
struct TailOp {
    int type, n, slice0, x, b, y, y2, d, pad, unused[3];
};
// The tail levels' packed matrices and operation list (per precision where
// two entries: FP64, FP32).  A tail that starts at level l runs operations
// first[l] .. last[l]; the residual and the iterate of the level above go to
// rb_off[l] and cb_off[l], the result comes from rb_off[l].
struct TailPack {
    int l0 = -1;
    int* table = nullptr;  // device: n_ops TailOps, then the slice table
    int n_ops = 0, n_table = 0;
    void* cols[2] = {nullptr, nullptr};
    void* vals[2] = {nullptr, nullptr};
    void* diags[2] = {nullptr, nullptr};
    int diag_off = 0, n_diag = 0;
    size_t lds[2] = {0, 0};
    std::vector<int> first, last, rb_off, cb_off;
};
constexpr int kTailLdsBytes = 160 * 1024;    // LDS of a compute unit
constexpr int64_t kTailMaxPadded = 1 << 18;  // entries of a packed matrix, padding included
void tail_free(TailPack* t);
// Packs levels l0.. for cycles in precision prec (0 FP64, 1 FP32), once.
void tail_pack(ramd_hier_s* h, int l0, int prec);
size_t tail_lds_bytes(const ramd_hier_s* h, int l0, int prec);
bool tail_fits(const ramd_csr_s* M);
// Launches the tail below level lb: restriction of r, the tail levels'
// cycle, out = cur + P_lb x.
template <typename X>
void launch_tail(ramd_hier_s* h, int lb, const X* r, const X* cur, X* out);

struct BlockState;  // multi-vector work space (block.hip)
void block_free(BlockState* b);

// Device-time buckets: pairs of hipEvents recorded on a stream around a
// piece of work, summed per slot when resolved.  Used for the per-level
// solve times (ParMultilevel::track_times) and PCG's precond_t / comm_t.
struct EventSpans {
    struct Span {
        hipEvent_t b, e;
        int slot;
    };
    std::vector<Span> pending;
    std::vector<hipEvent_t> pool;
    // records the start event of a span for `slot`; returns its index
    int open(hipStream_t s, int slot);
    void close(hipStream_t s, int idx);
    // waits for the last recorded event and adds every span's seconds to acc[slot]
    void resolve(std::vector<double>& acc);
    void release();
};

// Stream capture of fn's launches into an instantiated graph (thread-local
// capture mode; no memset node is ever recorded: buffers are cleared by
// kernels).
hipGraphExec_t capture_graph(hipStream_t s, const std::function<void()>& fn);

// Captured flexible-PCG iteration of the single-vector solve: the operator
// step and the preconditioner application (V-cycle and inner products; the
// direction update that writes x runs eagerly), one pair per parity of the
// alternating r.z slots, valid for one (A, hierarchy forms, precision,
// partials).
struct FpcgGraphs {
    hipGraphExec_t gA[2] = {nullptr, nullptr}, gB[2] = {nullptr, nullptr};
    uint64_t a_uid = 0, key = 0;
    int prec = -1;
    const double* part = nullptr;
    uint64_t used = 0;  // last use (least recently used entry is replaced)
};
// captured iterations kept per hierarchy (per outer operator, hierarchy
// forms and precision; no captured kernel touches the solution vector, so
// one capture serves every solution vector)
constexpr int kFpcgGraphSets = 4;
void fpcg_graphs_free(FpcgGraphs* g);

}  // namespace ramd

struct ramd_hier_s {
    ramd_ctx ctx = nullptr;
    ramd_amg_opts opts{};
    std::vector<ramd::Level> levels;
    int coarse_n = 0;
    int coarse_info = 0;   // dgetrf's info for the coarse matrix (> 0: zero pivot)
    double* lu = nullptr;  // column-major LU of the coarse matrix read column-major (A_c^T)
    int* piv = nullptr;
    int* perm = nullptr;   // the pivots' row swaps as one permutation
    ramd::TailPack* tail = nullptr;
    double* cb = nullptr;  // FP64 staging for the FP32 cycle's coarse solve
    double* cx = nullptr;
    double times[5] = {0, 0, 0, 0, 0};
    // host seconds of each level's setup step (the level's extend_hierarchy;
    // the coarsest level gets the dense factorisation), as the reference's
    // setup_times[5 * l] (multilevel/par_multilevel.hpp:171-208)
    std::vector<double> setup_level_s;
    // per-level device seconds of the cycle's work on that level while
    // tracking is on (solve_times[5 * l], multilevel/par_multilevel.hpp:343-456)
    bool track = false;
    std::vector<double> solve_level_s;
    ramd::EventSpans spans;
    bool fp32 = false;
    // coarse tail (the small coarsest levels' cycle as one workgroup
    // kernel; same bits either way): mode -1 off, 0 automatic (timed per
    // precision at the first cycle: tail_pick, -2 not yet), >= 1 forced to
    // start at that level; tail_force overrides both while timing
    int tail_mode = 0;
    int tail_pick[2] = {-2, -2};
    int tail_force = -2;
    // PCG work vectors (fine level)
    double *pr = nullptr, *pz = nullptr, *pp = nullptr, *pAp = nullptr;
    float *pr32 = nullptr, *pz32 = nullptr;
    ramd::BlockState* blk = nullptr;
    // captured FPCG iteration and its own partial-sum buffer (never
    // reallocated while graphs hold it)
    ramd::FpcgGraphs* fg = nullptr;  // kFpcgGraphSets entries (allocated at first use)
    uint64_t fg_tick = 0;
    double* fpart = nullptr;
    size_t fpart_cap = 0;
};

namespace ramd {
// Identity and buffer counts of A and of every level operator, and the
// coarse-tail switch: captured graphs hold raw pointers to all of their
// buffers and the launches these choose, and are keyed on this.
inline uint64_t forms_key(const ramd_hier_s* h, const ramd_csr_s* A)
{
    uint64_t k = A->uid * 1000003ull + A->forms;
    for (int t : {h->tail_mode, h->tail_pick[0], h->tail_pick[1]}) k = k * 131ull + (uint64_t)(t + 3);
    for (const Level& L : h->levels)
        for (const ramd_csr_s* M : {(const ramd_csr_s*)L.A, (const ramd_csr_s*)L.P, (const ramd_csr_s*)L.R})
            if (M) k = k * 1000003ull + M->uid * 31ull + M->forms;
    return k;
}
}  // namespace ramd

namespace ramd {
// Builds the FP32 copies of every level (values, diagonal, level vectors).
void enable_fp32(ramd_hier_s* h);
// Before cycling in precision prec (0 FP64, 1 FP32): the FP32 copies (prec
// 1) and, in the coarse tail's automatic mode, its timed choice.
void cycle_prepare(ramd_hier_s* h, int prec);
inline dim3 grid1(int64_t n, int bs = 256)
{
    int64_t g = (n + bs - 1) / bs;
    return dim3((unsigned)(g > 0 ? g : 1));
}
}  // namespace ramd
