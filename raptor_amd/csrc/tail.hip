// Coarse tail: the restriction into a run of small levels, their whole
// V-cycle (smoothing, residuals, restrictions, the coarse LU solve,
// interpolations) and the interpolation back out, by one workgroup in one
// launch instead of about five launches per level.
//
// Every vector of the tail levels, the residual that enters, the diagonals,
// the coarse LU and the operation list live in LDS; only the iterate the
// result is added to and the matrices come from memory.  The matrices are
// packed once per precision (tail_pack): 64 rows per slice, one lane per row,
// the rows' entries in stored order in groups of four (16-bit columns, then
// values), the slice padded to its longest row.  A wavefront owns every
// kTailWaves-th slice of an operation and adds each row's entries left to
// right on the row's lane, the operations of stream_kernel's phase 2, so
// every value is the one the per-level kernels produce.
//
// What bounds it: an operation is a chain of dependent steps (columns and
// values from memory, x from LDS, the row's additions, a barrier), and the
// kernel's instructions are fetched anew in every cycle, since the other
// levels' kernels run in between.  So the matrices, which do not depend on
// the cycle's vectors, are kept kTailDepth steps ahead in registers, across
// slices and across the operations' barriers (which wait for LDS only, not
// for these loads).  In a long row the loads are unconditional, so that the
// wait before a step covers its own loads and not the younger ones.  Every
// operation runs through one loop of few instructions per entry: the
// residual's subtraction is the addition of the negated product (the same
// value), and padding needs no test: its product is -0.0, and a + (-0.0) is a for every a.  A vector
// that rows gather from starts with an entry for that, one the padding's
// columns point to: +0.0, or -0.0 for the residual, whose values are negated
// (padding's value is -0.0).
#include <algorithm>
#include <cstring>

#include "hier.hpp"

namespace ramd {

constexpr int kTailWaves = 8;
constexpr int kTailThreads = 64 * kTailWaves;
constexpr int kTailUnit = 8;    // entries of a row per step: two groups of four
constexpr int kTailDepth = 4;   // steps in flight per wavefront
// a slice's table entry: 64-group blocks before it << kTailNgBits | its
// groups per row; block 0 of the packed arrays is all padding
constexpr int kTailNgBits = 12;

typedef unsigned short U16x4 __attribute__((ext_vector_type(4)));

// Workgroup barrier that waits for LDS traffic only.
__device__ __forceinline__ void tail_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <typename X>
struct TailUnitRegs {
    U16x4 c[2];  // byte offsets into the gathered vector
    X v[8];
};

// Step u of a slice (first group base, ng groups per row; uniform) into r;
// past the slice's groups: the padding block.
template <typename X>
__device__ __forceinline__ void tail_load(int base, int ng, int u, int lane, const U16x4* __restrict__ cols,
                                          const X* __restrict__ vals, TailUnitRegs<X>& r)
{
    typedef X X4 __attribute__((ext_vector_type(4)));
    const X4* v4 = reinterpret_cast<const X4*>(vals);
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int g = 2 * u + h;
        const int i = g < ng ? base + g * 64 : 0;
        r.c[h] = (cols + i)[lane];
        const X4 v = (v4 + i)[lane];
#pragma unroll
        for (int t = 0; t < 4; t++) r.v[4 * h + t] = v[t];
    }
}

__device__ __forceinline__ double negate_by(double v, unsigned sign)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    return __longlong_as_double((long long)(b ^ ((unsigned long long)sign << 32)));
}
__device__ __forceinline__ float negate_by(float v, unsigned sign)
{
    return __uint_as_float(__float_as_uint(v) ^ sign);
}

// acc + the products of a step's entries, in order, their values negated by
// `sign`; skip: without the first one.
template <typename X>
__device__ __forceinline__ X tail_add(X acc, const TailUnitRegs<X>& r, const X* xv, unsigned sign, bool skip)
{
    X xx[kTailUnit];
#pragma unroll
    for (int t = 0; t < kTailUnit; t++)
        xx[t] = *reinterpret_cast<const X*>(reinterpret_cast<const char*>(xv) + (unsigned)r.c[t >> 2][t & 3]);
#pragma unroll
    for (int t = 0; t < kTailUnit; t++) {
        const X next = acc + negate_by(r.v[t], sign) * xx[t];
        acc = t == 0 && skip ? acc : next;
    }
    return acc;
}

// The operation's record as scalars.
__device__ __forceinline__ TailOp tail_op(const TailOp* ops, int op)
{
    TailOp o = ops[op];
    int* w = reinterpret_cast<int*>(&o);
#pragma unroll
    for (int t = 0; t < (int)(sizeof(TailOp) / sizeof(int)); t++) w[t] = __builtin_amdgcn_readfirstlane(w[t]);
    return o;
}

// The cycle of cycle64 / cycle32 from the restriction into a level to the
// interpolation out of it: operations first .. last of the list.  The
// residual rb and the iterate curb of the level above are copied to LDS
// offsets rb_off and cb_off first, and the result from rb_off to outb at the
// end; all other vectors stay in LDS.
template <typename X>
__global__ __launch_bounds__(kTailThreads) void tail_cycle_kernel(
    const int* __restrict__ table, int n_table, int n_ops, const U16x4* __restrict__ cols,
    const X* __restrict__ vals, const X* __restrict__ diags, const double* __restrict__ lu,
    const int* __restrict__ perm, int first, int last, int nc, int diag_off, int n_diag, int rb_off, int cb_off,
    int n_rb, X omega, const X* __restrict__ rb, const X* __restrict__ curb, X* __restrict__ outb)
{
    extern __shared__ double lds[];
    double* ls = lds;  // nc * nc
    int* tab = reinterpret_cast<int*>(lds + nc * nc);
    const TailOp* ops = reinterpret_cast<const TailOp*>(tab);
    const int* slices = tab + n_ops * (int)(sizeof(TailOp) / sizeof(int));
    X* vec = reinterpret_cast<X*>(lds + nc * nc + (n_table + 1) / 2);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    for (int t = tid; t < n_table; t += kTailThreads) tab[t] = table[t];
    for (int t = tid; t < n_rb; t += kTailThreads) {
        vec[rb_off + 1 + t] = rb[t];
        vec[cb_off + 1 + t] = curb[t];
    }
    for (int t = tid; t < n_diag; t += kTailThreads) vec[diag_off + t] = diags[t];
    for (int t = tid; t < nc * nc; t += kTailThreads) ls[t] = lu[t];
    const int pm = lane < nc ? perm[lane] : 0;
    if (tid == 0) vec[rb_off] = X(0);
    tail_barrier();

    // the wavefront's current slice: operation cop, slice cq, first group cb, groups cn
    TailOp o = tail_op(ops, first);
    int cop = first, cq = wave, cb = 0, cn = 0;
    if (cq * 64 < o.n) {
        const int w = __builtin_amdgcn_readfirstlane(slices[o.slice0 + cq]);
        cb = (w >> kTailNgBits) * 64;
        cn = w & ((1 << kTailNgBits) - 1);
    } else {
        cop = -1;  // none yet
    }
    TailUnitRegs<X> buf[kTailDepth];
#pragma unroll
    for (int d = 0; d < kTailDepth; d++)
        if (2 * d < cn) tail_load(cb, cn, d, lane, cols, vals, buf[d]);

#pragma unroll 1
    for (int op = first; op <= last; op++) {
        // the next operation's record and the wavefront's first slice of it
        TailOp on = o;
        if (op < last) on = tail_op(ops, op + 1);
        const bool have_next = op < last && on.slice0 >= 0 && wave * 64 < on.n;
        const bool idle = cop != op;
        if (idle && have_next) {
            // no slice of this operation: the next one's first steps now
            const int w = __builtin_amdgcn_readfirstlane(slices[on.slice0 + wave]);
            cb = (w >> kTailNgBits) * 64;
            cn = w & ((1 << kTailNgBits) - 1);
#pragma unroll
            for (int d = 0; d < kTailDepth; d++)
                if (2 * d < cn) tail_load(cb, cn, d, lane, cols, vals, buf[d]);
        }
        const int type = o.type;
        const bool jac = type == kTailJacobi;
        if (type == kTailCoarse && wave == 0) {
            // the coarsest level: FP64 LU solve on one wavefront, rounded once
            double v = lane < nc ? (double)vec[o.b + pm] : 0.0;
            v = coarse_lu_lane(nc, ls, v, lane);
            if (lane < nc) vec[o.y + 1 + lane] = (X)v;
        } else if (type == kTailFill) {
            for (int i = tid; i < o.n; i += kTailThreads) vec[o.y + 1 + i] = X(0);
        }
        const unsigned sign = type == kTailResidual ? 0x80000000u : 0u;
        const X* xv = vec + o.x;
        bool mine = !idle;
#pragma unroll 1
        while (mine) {
            // the wavefront's next slice: of this operation, or of the next
            const bool again = (cq + kTailWaves) * 64 < o.n;
            const int nw = again ? slices[o.slice0 + cq + kTailWaves]
                                 : (have_next ? slices[on.slice0 + wave] : 0);
            const int row = cq * 64 + lane;
            const bool valid = row < o.n;
            X acc = X(0), diag = X(0), own = X(0), rhs = X(0);
            if (valid) {
                if (type == kTailResidual || jac) rhs = vec[o.b + row];
                if (type == kTailAdd) rhs = vec[o.b + 1 + row];
                if (jac || type == kTailSpmvJfz) diag = vec[o.d + row];
                if (jac) own = xv[1 + row];
            }
            if (type == kTailResidual) acc = rhs;
            const int nu = (cn + 1) >> 1;
            // all steps but the last kTailDepth, each followed by the load
            // of the step that takes its registers
            int u0 = 0;
            for (; u0 + kTailDepth < nu; u0 += kTailDepth) {
#pragma unroll
                for (int d = 0; d < kTailDepth; d++) {
                    // Jacobi does not add the diagonal, the first entry
                    acc = tail_add(acc, buf[d], xv, sign, d == 0 && jac && u0 == 0);
                    tail_load(cb, cn, u0 + d + kTailDepth, lane, cols, vals, buf[d]);
                }
            }
#pragma unroll
            for (int d = 0; d < kTailDepth; d++)
                if (u0 + d < nu) acc = tail_add(acc, buf[d], xv, sign, d == 0 && jac && u0 == 0);
            // the first steps of the wavefront's next slice
            {
                const int w = __builtin_amdgcn_readfirstlane(nw);
                cb = (w >> kTailNgBits) * 64;
                cn = w & ((1 << kTailNgBits) - 1);
            }
#pragma unroll
            for (int d = 0; d < kTailDepth; d++)
                if (2 * d < cn) tail_load(cb, cn, d, lane, cols, vals, buf[d]);
            if (valid) {
                if (jac) {
                    // a row without a usable diagonal keeps its value
                    acc = (fabs(diag) > X(1e-16)) ? ((X(1.0) - omega) * own) + (omega * ((rhs - acc) / diag)) : own;
                } else if (type == kTailAdd) {
                    acc = rhs + acc;
                } else if (type == kTailSpmvJfz) {
                    vec[o.y2 + 1 + row] = jacobi_zero_row(acc, diag, omega);
                }
                // b is not gathered from and has no padding entry
                vec[o.y + (type == kTailSpmv || type == kTailSpmvJfz ? 0 : 1) + row] = acc;
            }
            cq += kTailWaves;
            mine = again;
        }
        if (tid == 0 && o.pad != 0) vec[(o.pad < 0 ? -o.pad : o.pad) - 1] = o.pad < 0 ? -X(0) : X(0);
        cop = have_next ? op + 1 : -1;
        cq = wave;
        o = on;
        tail_barrier();
    }
    for (int t = tid; t < n_rb; t += kTailThreads) outb[t] = vec[rb_off + 1 + t];
}

// Rows of a matrix into its slices: entry k of row r in group k / 4, as the
// byte offset of its column (the vector's entry 0 is the padding's) and its
// value; padded to the slice's groups (rows past n are all padding).
template <typename X>
__global__ void tail_pack_kernel(int n, int padded, const int* __restrict__ rp, const int* __restrict__ col,
                                 const double* __restrict__ val, const int* __restrict__ slices,
                                 unsigned short* __restrict__ cols, X* __restrict__ vals)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= padded) return;
    const int s = slices[r >> 6];
    const int base = (s >> kTailNgBits) * 64, ng = s & ((1 << kTailNgBits) - 1);
    int b = 0, len = 0;
    if (r < n) {
        b = rp[r];
        len = rp[r + 1] - b;
    }
    for (int k = 0; k < 4 * ng; k++) {
        const size_t i = ((size_t)base + (size_t)(k >> 2) * 64 + (r & 63)) * 4 + (k & 3);
        cols[i] = k < len ? (unsigned short)((col[b + k] + 1) * (int)sizeof(X)) : (unsigned short)0;
        vals[i] = k < len ? (X)val[b + k] : -X(0);
    }
}

// Block 0: padding.
template <typename X>
__global__ void tail_pad_kernel(unsigned short* __restrict__ cols, X* __restrict__ vals)
{
    const int i = threadIdx.x;
    cols[i] = 0;
    vals[i] = -X(0);
}

template <typename X>
__global__ void tail_diag_kernel(int n, const double* __restrict__ d, X* __restrict__ out)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = (X)d[i];
}

void tail_free(TailPack* t)
{
    if (!t) return;
    for (void* p : {(void*)t->table, t->cols[0], t->cols[1], t->vals[0], t->vals[1],
                    t->diags[0], t->diags[1]})
        dfree(p);
    delete t;
}

// Operations of the largest tail (from level l0).
static int tail_ops(const ramd_hier_s* h, int l0)
{
    const int sweeps = std::max(h->opts.num_smooth_sweeps, 0);
    const int above = (int)h->levels.size() - 1 - l0;  // tail levels above the coarsest
    return above * (3 + (sweeps ? 2 * sweeps - 1 : 1)) + 3;
}

static int tail_slices(const ramd_hier_s* h, int l0)
{
    auto q = [&](int l) { return (h->levels[(size_t)l].n + 63) / 64; };
    int s = 0;
    for (int l = l0; l < (int)h->levels.size(); l++) s += q(l) + q(l - 1) + (l + 1 < (int)h->levels.size() ? q(l) : 0);
    return s;
}

size_t tail_lds_bytes(const ramd_hier_s* h, int l0, int prec)
{
    size_t n = 2 * ((size_t)h->levels[(size_t)l0 - 1].n + 1);
    for (size_t l = (size_t)l0; l < h->levels.size(); l++) n += 4 * (size_t)h->levels[l].n + 2;
    const size_t table = (size_t)tail_ops(h, l0) * (sizeof(TailOp) / sizeof(int)) + (size_t)tail_slices(h, l0);
    return sizeof(double) * ((size_t)h->coarse_n * h->coarse_n + (table + 1) / 2) +
           n * (prec ? sizeof(float) : sizeof(double));
}

// 64-lane groups of four entries in the packed form of M.
static int64_t tail_groups(const ramd_csr_s* M)
{
    const int* rp = M->h_rowptr.data();
    int64_t g = 0;
    for (int q = 0; q < M->n_rows; q += 64) {
        int w = 0;
        for (int r = q; r < std::min(M->n_rows, q + 64); r++) w = std::max(w, rp[r + 1] - rp[r]);
        g += (int64_t)64 * ((w + 3) / 4);
    }
    return g;
}

void tail_pack(ramd_hier_s* h, int l0, int prec)
{
    const int nlev = (int)h->levels.size();
    hipStream_t s = h->ctx->stream;
    RAMD_CHECK(l0 >= 1 && l0 < nlev, RAMD_E_STATE, "coarse tail: first level %d of %d", l0, nlev);
    if (h->tail && h->tail->vals[prec]) return;
    // the matrices in the order their slices are laid out: for each tail
    // level the R into it and the P out of it, and A above the coarsest
    struct Mat {
        const ramd_csr_s* M;
        int slice0;
    };
    std::vector<Mat> R((size_t)nlev), P((size_t)nlev), A((size_t)nlev);
    std::vector<int> slices;
    int64_t groups = 64;  // after the padding block
    auto add = [&](const ramd_csr_s* M) {
        Mat m{M, (int)slices.size()};
        const int* rp = M->h_rowptr.data();
        for (int q = 0; q < M->n_rows; q += 64) {
            int w = 0;
            for (int r = q; r < std::min(M->n_rows, q + 64); r++) w = std::max(w, rp[r + 1] - rp[r]);
            slices.push_back((int)(groups / 64) << kTailNgBits | (w + 3) / 4);
            groups += (int64_t)64 * ((w + 3) / 4);
        }
        return m;
    };
    for (int l = l0; l < nlev; l++) {
        R[l] = add(h->levels[l - 1].R);
        P[l] = add(h->levels[l - 1].P);
        if (l + 1 < nlev) A[l] = add(h->levels[l].A);
    }
    if (!h->tail) {
        h->tail = new TailPack();
        h->tail->l0 = l0;
    }
    TailPack& T = *h->tail;
    RAMD_CHECK(T.l0 == l0, RAMD_E_STATE, "coarse tail: packed from level %d, not %d", T.l0, l0);
    if (!T.table) {
        const int sweeps = h->opts.num_smooth_sweeps;
        // LDS offsets (in vector elements): x, t, b per level (x and t after
        // their padding entry), the diagonals, the level above's two vectors
        std::vector<int> xo((size_t)nlev), to((size_t)nlev), bo((size_t)nlev), dof((size_t)nlev);
        int off = 0;
        for (int l = l0; l < nlev; l++) {
            const int n = h->levels[l].n;
            xo[l] = off;
            to[l] = off + n + 1;
            bo[l] = off + 2 * n + 2;
            off += 3 * n + 2;
        }
        T.diag_off = off;
        for (int l = l0; l < nlev; l++) {
            dof[l] = off;
            off += h->levels[l].n;
        }
        T.n_diag = off - T.diag_off;
        T.rb_off.assign((size_t)nlev, off);
        T.cb_off.assign((size_t)nlev, off + h->levels[(size_t)l0 - 1].n + 1);
        std::vector<TailOp> ops;
        std::vector<int> cur((size_t)nlev), oth((size_t)nlev);
        T.first.assign((size_t)nlev, -1);
        T.last.assign((size_t)nlev, -1);
        // pad: the vector whose padding entry the operation sets (its offset
        // + 1; negated: to -0.0, for a residual)
        auto op = [&](int type, int n, int slice0, int x, int b, int y, int y2, int d, int pad) {
            ops.push_back(TailOp{type, n, slice0, x, b, y, y2, d, pad, {0, 0, 0}});
        };
        for (int l = l0; l < nlev; l++) {
            const Level& L = h->levels[l];
            T.first[l] = (int)ops.size();
            // r of the level above sits in that level's spare iterate
            if (l > l0) {
                T.rb_off[l] = oth[l - 1];
                T.cb_off[l] = cur[l - 1];
            }
            const int xin = T.rb_off[l];
            const bool smoothed = l + 1 < nlev && sweeps >= 1;
            if (smoothed)
                op(kTailSpmvJfz, L.n, R[l].slice0, xin, 0, bo[l], xo[l], dof[l],
                   sweeps == 1 ? -(xo[l] + 1) : xo[l] + 1);
            else op(kTailSpmv, L.n, R[l].slice0, xin, 0, bo[l], 0, 0, 0);
            cur[l] = xo[l];
            oth[l] = to[l];
            if (l + 1 == nlev) {
                op(kTailCoarse, L.n, -1, 0, bo[l], xo[l], 0, 0, xo[l] + 1);
                break;
            }
            if (sweeps <= 0) op(kTailFill, L.n, -1, 0, 0, xo[l], 0, 0, -(xo[l] + 1));
            for (int it = 1; it < sweeps; it++) {
                op(kTailJacobi, L.n, A[l].slice0, cur[l], bo[l], oth[l], 0, dof[l],
                   it + 1 == sweeps ? -(oth[l] + 1) : oth[l] + 1);
                std::swap(cur[l], oth[l]);
            }
            op(kTailResidual, L.n, A[l].slice0, cur[l], bo[l], oth[l], 0, 0, oth[l] + 1);
        }
        for (int l = nlev - 1; l >= l0; l--) {
            // out of level l: cur + P x into the spare iterate of the level above
            const Level& B = h->levels[l - 1];
            op(kTailAdd, B.n, P[l].slice0, cur[l], T.cb_off[l], T.rb_off[l], 0, 0, T.rb_off[l] + 1);
            T.last[l] = (int)ops.size() - 1;
            if (l == l0) break;
            std::swap(cur[l - 1], oth[l - 1]);
            for (int it = 0; it < sweeps; it++) {
                op(kTailJacobi, B.n, A[l - 1].slice0, cur[l - 1], bo[l - 1], oth[l - 1], 0, dof[l - 1],
                   oth[l - 1] + 1);
                std::swap(cur[l - 1], oth[l - 1]);
            }
        }
        RAMD_CHECK((int)ops.size() == tail_ops(h, l0) && (int)slices.size() == tail_slices(h, l0), RAMD_E_STATE,
                   "coarse tail: %zu operations, %zu slices", ops.size(), slices.size());
        constexpr int W = (int)(sizeof(TailOp) / sizeof(int));
        std::vector<int> table(ops.size() * W + slices.size());
        std::memcpy(table.data(), ops.data(), ops.size() * sizeof(TailOp));
        std::copy(slices.begin(), slices.end(), table.begin() + (long)ops.size() * W);
        T.n_ops = (int)ops.size();
        T.n_table = (int)table.size();
        T.table = dalloc<int>(table.size());
        RAMD_HIP(hipMemcpyAsync(T.table, table.data(), sizeof(int) * table.size(), hipMemcpyHostToDevice, s));
        RAMD_HIP(hipStreamSynchronize(s));  // the host vector goes out of scope
    }
    const int* d_slices = T.table + (size_t)T.n_ops * (sizeof(TailOp) / sizeof(int));
    const size_t w = prec ? sizeof(float) : sizeof(double);
    void* vals = dmalloc(w * 4 * (size_t)groups);
    unsigned short* cols = nullptr;
    void* diags = nullptr;
    try {
        cols = dalloc<unsigned short>(4 * (size_t)groups);
        if (prec) hipLaunchKernelGGL((tail_pad_kernel<float>), dim3(1), dim3(256), 0, s, cols, (float*)vals);
        else hipLaunchKernelGGL((tail_pad_kernel<double>), dim3(1), dim3(256), 0, s, cols, (double*)vals);
        RAMD_HIP(hipGetLastError());
        diags = dmalloc(w * (size_t)std::max(T.n_diag, 1));
        auto pack = [&](const Mat& m) {
            const int padded = (m.M->n_rows + 63) / 64 * 64;
            if (!padded) return;
            if (prec)
                hipLaunchKernelGGL((tail_pack_kernel<float>), grid1(padded), dim3(256), 0, s, m.M->n_rows, padded,
                                   m.M->rowptr, m.M->col, m.M->val, d_slices + m.slice0, cols, (float*)vals);
            else
                hipLaunchKernelGGL((tail_pack_kernel<double>), grid1(padded), dim3(256), 0, s, m.M->n_rows, padded,
                                   m.M->rowptr, m.M->col, m.M->val, d_slices + m.slice0, cols, (double*)vals);
            RAMD_HIP(hipGetLastError());
        };
        size_t at = 0;
        for (int l = l0; l < nlev; l++) {
            pack(R[l]);
            pack(P[l]);
            if (l + 1 < nlev) pack(A[l]);
            const Level& L = h->levels[l];
            if (prec)
                hipLaunchKernelGGL((tail_diag_kernel<float>), grid1(L.n), dim3(256), 0, s, L.n, L.diag,
                                   (float*)diags + at);
            else
                hipLaunchKernelGGL((tail_diag_kernel<double>), grid1(L.n), dim3(256), 0, s, L.n, L.diag,
                                   (double*)diags + at);
            RAMD_HIP(hipGetLastError());
            at += (size_t)L.n;
        }
        const size_t bytes = tail_lds_bytes(h, l0, prec);
        const void* fn = prec ? (const void*)tail_cycle_kernel<float> : (const void*)tail_cycle_kernel<double>;
        RAMD_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, kTailLdsBytes));
        T.lds[prec] = bytes;
    } catch (...) {
        dfree(vals);
        dfree(cols);
        dfree(diags);
        throw;
    }
    T.vals[prec] = vals;
    T.cols[prec] = cols;
    T.diags[prec] = diags;
}

template <typename X>
void launch_tail(ramd_hier_s* h, int lb, const X* r, const X* cur, X* out)
{
    const int prec = sizeof(X) == 4 ? 1 : 0;
    const TailPack* T = h->tail;
    const int l = lb + 1;
    RAMD_CHECK(T && T->vals[prec] && l >= T->l0 && l < (int)h->levels.size() && T->first[l] >= 0, RAMD_E_STATE,
               "coarse tail: level %d was not packed", l);
    hipLaunchKernelGGL((tail_cycle_kernel<X>), dim3(1), dim3(kTailThreads), T->lds[prec], h->ctx->stream, T->table,
                       T->n_table, T->n_ops, (const U16x4*)T->cols[prec], (const X*)T->vals[prec], (const X*)T->diags[prec], h->lu,
                       h->perm, T->first[l], T->last[l], h->coarse_n, T->diag_off, T->n_diag, T->rb_off[l], T->cb_off[l],
                       h->levels[(size_t)lb].n, (X)h->opts.relax_weight, r, cur, out);
    RAMD_HIP(hipGetLastError());
}
template void launch_tail<double>(ramd_hier_s*, int, const double*, const double*, double*);
template void launch_tail<float>(ramd_hier_s*, int, const float*, const float*, float*);

bool tail_fits(const ramd_csr_s* M)
{
    const int64_t g = tail_groups(M);
    return g * 4 <= kTailMaxPadded && g / 64 < (1 << kTailNgBits);
}

}  // namespace ramd
