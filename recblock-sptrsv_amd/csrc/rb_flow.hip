// Flow schedule: the whole solve in one launch over all compute units, rows
// in level order, every row waiting for its own dependencies.
//
// For factors whose levels are wide and few (power-law rows): rows are put
// in order (level, entries per lane and lanes per row) and cut into steps of
// 64 lanes alike, so a lane's entries (1, 2 or 4) are all read at once and no
// lane idles for a longer neighbour; rows of more than 4 entries take several
// lanes.  A wave takes a step, reads its entries, then x of all of them in
// one go, repeats what still holds the sentinel, and writes x by position for
// other rows and in the caller's order.  b is read and x written in place:
// no pass but the one that puts the sentinel into the x buffer.
//
// Waves take their steps from 16 counters, wave i of a workgroup always from
// counter i, in order and one ahead: any resident workgroup serves every
// counter, so the lowest step not done is always with a wave whose earlier
// steps are done, whatever else runs on the device.  The launch has about 10
// levels' worth of waves, at most 16 per compute unit: fewer leave levels
// waiting for their entries, more only poll (300,001 rows, 90 steps a level:
// 32 / 64 / 128 workgroups 192 / 169 / 198 us; 4M rows, 540 steps a level:
// 128 / 192 / 256 workgroups 625 / 570 / 568 us).  Waiting waves sleep
// between polls, in the end for a 64th of the time waited so far, at most
// about 2 ms: where thousands wait for one line, the polls of it become so
// few that the store they wait for goes through.
//
// Several right-hand sides: a row's x lie together, CP columns per lane on
// CL neighbouring lanes, so that an entry costs one line for all of them
// (300,001 rows backward, 5 columns: 160 us; column by column, an entry at a
// time, 1,210 us).  Groups of columns go side by side in one launch, on as
// many workgroups together as one alone has at most (32 columns of 300,000 rows
// 527 us; with up to twice as many 783, with that many for each 1,567: the
// waves beyond only poll).
//
// x is divided by the diagonal (a product with its reciprocal is no faster
// here, and further off: 1.03e-16 of 4M rows, 5.6e-17 like this).
//
// Bound: the random reads.  4M rows, 16.6M entries outside the caches: 434 us
// with every wait taken out of a copy, 556 with them; 75 us is what its
// bytes would take in order.  On 300,001 rows the chain of levels, 2 us each.
#include <algorithm>
#include <memory>
#include <type_traits>
#include <vector>

#include "rb_internal.h"

namespace rb {

namespace {

constexpr int kT = 256;
constexpr int kEnt = 4;      // entries per lane at a time
constexpr int kWaves = 16;   // waves of a workgroup, each with a ticket counter of its own
constexpr int kPad = 32;     // counters apart (ints)
constexpr int kCtl = (kWaves + 1) * kPad;  // and the count of finished workgroups
constexpr int kCols = 8;     // columns of a row's line of x at most
constexpr int kGroups = 4;   // lines of that many, a launch

inline int nblk(long n, int t = kT) { return (int)((n + t - 1) / t); }

// A step: up to 64 lanes of rows of one level, alike in lanes per row and
// entries per lane.
struct Step {
    int pos;       // position of its first row
    int shape;     // log2 lanes per row | log2 entries per lane << 8 | rows << 16
    unsigned off;  // its entries (64 lanes x entries per lane x chunks), in 64s
    int chunks;    // rounds of kEnt entries per lane (1 but for the longest rows)
};

struct FlowArgs {
    const Step *step;
    const int *col;     // position of an entry, -1: none
    const double *val;  // -a_ij
    const int *row;     // caller's row of a position
    const double *diag; // a_ii by position
    const double *b;
    double *x;
    long ldb, ldx;
    int ncol;           // columns, at most the kernel's times the grid's groups
    int m, nsteps;
    double *xs;         // [groups][m][columns of the kernel] x by position, the
                        // sentinel until solved
    int *ctl;           // [groups][kCtl] tickets; workgroups done
    int *status;
    unsigned spin;
};

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
constexpr int kSC1 = 16;  // cache policy: device-coherent

__device__ inline bool pending(double v) {
    return __double_as_longlong(v) == (long long)kPending;
}

// A lane's CP (1 or 2) neighbouring columns of x
template <int CP>
struct Xv {
    double v[CP];
    __device__ bool wait() const {
        bool w = pending(v[0]);
        if constexpr (CP == 2) w = w || pending(v[1]);
        return w;
    }
};
template <int CP>
__device__ inline Xv<CP> ld_x(__amdgpu_buffer_rsrc_t r, int off) {
    if constexpr (CP == 2)
        return __builtin_bit_cast(Xv<2>, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, kSC1));
    else
        return __builtin_bit_cast(Xv<1>, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, kSC1));
}
template <int CP>
__device__ inline void st_x(Xv<CP> v, __amdgpu_buffer_rsrc_t r, int off) {
    if constexpr (CP == 2)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, off, 0, kSC1);
    else
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, off, 0, kSC1);
}

__global__ void __launch_bounds__(kT) k_flow_reset(double *xs, long n, int *ctl, int nctl) {
    const long i = ((long)blockIdx.x * kT + threadIdx.x) * 2;
    const double s = __longlong_as_double((long long)kPending);
    if (i + 1 < n) *(double2 *)(xs + i) = make_double2(s, s);
    else if (i < n) xs[i] = s;
    if (blockIdx.x == 0)
        for (int k = threadIdx.x; k < nctl; k += kT) ctl[k] = 0;
}

// CP columns per lane, CL lanes beside each other for a row's columns: an
// entry's CP * CL columns of x lie together and are read by CL lanes in one
// access.  A wave takes 64 / CL of a step's 64 lanes at a time.  MULTI:
// blockIdx.y is a group of CP * CL columns, with tickets and x of its own, which
// waits for no other.  (The one group of the others is known to be the first:
// 5 columns of 300,001 rows 194 us, 196 with the multiple form.)
template <int CP, int CL, bool MULTI>
__global__ void __launch_bounds__(kWaves * 64) k_flow(FlowArgs a) {
    constexpr int KC = CP * CL, S = 64 / CL;
    const int grp = MULTI ? blockIdx.y : 0, g0 = grp * KC;
    const int ncol = a.ncol - g0;  // the group's columns
    const double *b = a.b + g0 * a.ldb;
    double *xo = a.x + g0 * a.ldx;
    const int lane = threadIdx.x & 63, c0 = lane % CL * CP;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const __amdgpu_buffer_rsrc_t xs = __builtin_amdgcn_make_buffer_rsrc(
        a.xs + (long)g0 * a.m, (short)0, (int)min((long)a.m * KC * 8, 0x7fffffffL), 0x00020000);
    int *ticket = a.ctl + grp * kCtl + wave * kPad;
    auto take = [&]() {
        int t = 0;
        if (lane == 0)
            t = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return t;  // lane 0
    };
    int nt = take();
    while (true) {
        const int t = __builtin_amdgcn_readfirstlane(nt) * kWaves + wave;
        if (t >= a.nsteps * CL) break;
        nt = take();
        const int s = t / CL, sub = t % CL;
        const Step st = a.step[s];
        const int shape = __builtin_amdgcn_readfirstlane(st.shape), gl = shape & 255,
                  el = (shape >> 8) & 255;
        // a row wider than the wave's slots is taken by the part that it
        // begins in, a lane going on to the slots S further: one sum for
        // each, added up in the order of the shuffles of a single column
        // (same bits)
        const int reps = max(1, (1 << gl) / S);
        if (sub & (reps - 1)) continue;
        const int slot = sub * S + lane / CL;
        const int r = slot >> gl;
        const bool live = r < shape >> 16;
        const int p = st.pos + (live ? r : 0);
        const int row = a.row[p];
        const double dv = a.diag[p];
        double acc[CP], bv[CP];
        bool bad = false;
        auto run = [&](auto ents, int rep) {
            constexpr int E = decltype(ents)::value;
            for (int ch = 0; ch < st.chunks; ch++) {
                const size_t o =
                    ((size_t)st.off + (size_t)ch * E) * 64 + (size_t)(slot + rep * S) * E;
                int cj[E];
                double vj[E];
                Xv<CP> xv[E];
#pragma unroll
                for (int j = 0; j < E; j++) cj[j] = live ? a.col[o + j] : -1;
#pragma unroll
                for (int j = 0; j < E; j++) vj[j] = live ? a.val[o + j] : 0.0;
                // (no entry: out of range, reads zero)
#pragma unroll
                for (int j = 0; j < E; j++) {
                    cj[j] = cj[j] < 0 ? -16 : (cj[j] * KC + c0) * 8;
                    xv[j] = ld_x<CP>(xs, cj[j]);
                }
                unsigned spins = 0;
                while (true) {
                    bool wait = false;
#pragma unroll
                    for (int j = 0; j < E; j++) wait = wait || xv[j].wait();
                    if (!__any(wait)) break;
                    if (spins > a.spin) {
                        bad = true;
                        break;
                    }
                    if (spins < 16) __builtin_amdgcn_s_sleep(6);
                    else if (spins < 64) __builtin_amdgcn_s_sleep(20);
                    else
                        for (unsigned k = 0; k < min(spins / 64, 1024u); k++)
                            __builtin_amdgcn_s_sleep(60);
                    spins += max(1u, min(spins / 64, 1024u));
#pragma unroll
                    for (int j = 0; j < E; j++)
                        if (xv[j].wait()) xv[j] = ld_x<CP>(xs, cj[j]);
                }
#pragma unroll
                for (int j = 0; j < E; j++)
#pragma unroll
                    for (int c = 0; c < CP; c++) acc[c] += vj[j] * xv[j].v[c];
            }
        };
#pragma unroll
        for (int c = 0; c < CP; c++)
            bv[c] = live && c0 + c < ncol ? b[(c0 + c) * a.ldb + row] : 0.0;
        auto tree = [&](int rep, double (&sum)[CP]) {
#pragma unroll
            for (int c = 0; c < CP; c++) acc[c] = 0.0;
            if (el == 0) run(std::integral_constant<int, 1>(), rep);
            else if (el == 1) run(std::integral_constant<int, 2>(), rep);
            else run(std::integral_constant<int, 4>(), rep);
            for (int o = 1; o < min(1 << gl, S); o <<= 1)
#pragma unroll
                for (int c = 0; c < CP; c++) acc[c] += __shfl_xor(acc[c], o * CL, 64);
#pragma unroll
            for (int c = 0; c < CP; c++) sum[c] = rep & 1 ? sum[c] + acc[c] : acc[c];
        };
        double sum[CP], rest[CP];
        for (int rep = 0; rep < min(reps, 2); rep++) tree(rep, sum);
        if (CL > 2 && reps > 2) {
            for (int rep = 2; rep < 4; rep++) tree(rep, rest);
#pragma unroll
            for (int c = 0; c < CP; c++) sum[c] += rest[c];
        }
        if (bad && lane == 0) atomicOr(a.status, 1);
        if (live && (slot & ((1 << gl) - 1)) == 0) {
            Xv<CP> x;
#pragma unroll
            for (int c = 0; c < CP; c++)
                x.v[c] = bad ? __builtin_nan("") : (bv[c] + sum[c]) / dv;
            st_x<CP>(x, xs, (p * KC + c0) * 8);
#pragma unroll
            for (int c = 0; c < CP; c++)
                if (c0 + c < ncol) xo[(c0 + c) * a.ldx + row] = x.v[c];
        }
    }
    // the last workgroup turns every x into a NaN when a wait gave up
    __syncthreads();
    __shared__ int last;
    if (threadIdx.x == 0)
        last = __hip_atomic_fetch_add(a.ctl + kWaves * kPad, 1, __ATOMIC_ACQ_REL,
                                      __HIP_MEMORY_SCOPE_AGENT) ==
                   (int)(gridDim.x * (MULTI ? gridDim.y : 1)) - 1 &&
               (__hip_atomic_load(a.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & 7);
    __syncthreads();
    if (last)
        for (int c = 0; c < a.ncol; c++)
            for (int i = threadIdx.x; i < a.m; i += kWaves * 64)
                a.x[c * a.ldx + i] = __builtin_nan("");
}

// ------------------------------------------------------------- build

struct RowGeom {
    int m, fwd, nlev;
};

// lanes per row and entries per lane of a row length: class (el, gl)
__device__ inline int class_of(int len) {
    if (len <= 1) return 0;
    if (len <= 2) return 1;
    int gl = 0;
    while (gl < 6 && (kEnt << gl) < len) gl++;
    return 2 + gl;
}
__device__ inline int class_el(int c) { return c < 2 ? c : 2; }
__device__ inline int class_gl(int c) { return c < 2 ? 0 : c - 2; }

__global__ void k_fl_key(RowGeom g, const int *__restrict__ rp, const int *__restrict__ lp,
                         int *key, int *val) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= g.m) return;
    const int r = g.fwd ? q : g.m - 1 - q;
    int lo = 0, hi = g.nlev;
    while (hi - lo > 1) {
        const int mid = (lo + hi) / 2;
        if (lp[mid] <= q) lo = mid;
        else hi = mid;
    }
    key[q] = lo * 16 + class_of(rp[r + 1] - rp[r] - 1);
    val[q] = q;
}

__global__ void k_fl_heads(const int *__restrict__ key, int m, int *run) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < m) run[i] = i > 0 && key[i] == key[i - 1] ? 0 : i;
}

// per position: is it the first of a step, and the 64s of entries of that
// step; permuted row -> position
__global__ void k_fl_steps(const int *__restrict__ key, const int *__restrict__ run,
                           const int *__restrict__ order, RowGeom g, int *head, int *rend, int *newpos) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= g.m) return;
    const int c = key[i] & 15, gl = class_gl(c);
    head[i] = ((i - run[i]) & ((64 >> gl) - 1)) == 0;
    if (i + 1 == g.m || key[i + 1] != key[i]) rend[run[i]] = i + 1;
    const int q = order[i];
    newpos[g.fwd ? q : g.m - 1 - q] = i;
}

// the 64s of entries of the step a head starts (a step of the longest rows
// holds one row)
__global__ void k_fl_size(const int *__restrict__ key, const int *__restrict__ order, RowGeom g,
                          const int *__restrict__ rp, const int *__restrict__ head, int *size) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i > g.m) return;
    size[i] = 0;
    if (i == g.m || !head[i]) return;
    const int c = key[i] & 15, r = g.fwd ? order[i] : g.m - 1 - order[i];
    const int len = rp[r + 1] - rp[r] - 1, e = 1 << class_el(c);
    size[i] = class_gl(c) < 6 ? e : e * max(1, (len + 64 * e - 1) / (64 * e));
}

__global__ void k_fl_blank(int *col, double *val, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        col[i] = -1;
        val[i] = 0.0;
    }
}

__global__ void k_fl_fill(const int *__restrict__ key, const int *__restrict__ run,
                          const int *__restrict__ rend, const int *__restrict__ order,
                          const int *__restrict__ head, const int *__restrict__ sidx,
                          const int *__restrict__ off, RowGeom g, const int *__restrict__ rp,
                          const int *__restrict__ cc, const double *__restrict__ cv,
                          const int *__restrict__ newpos, const int *__restrict__ lf, Step *step,
                          int *col, double *val, int *row, double *diag) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < g.m;
    int c = 0, k0 = 0, first = 0, past = 0, o64 = 0;
    if (live) {
        c = key[i] & 15;
        const int gl = class_gl(c), el = class_el(c), e = 1 << el;
        k0 = (i - run[i]) & ((64 >> gl) - 1);
        o64 = off[i - k0];
        const int r = g.fwd ? order[i] : g.m - 1 - order[i];
        // (columns rise along a row: the diagonal is its last entry, in a
        // backward solve its first)
        first = rp[r] + (g.fwd ? 0 : 1);
        past = rp[r + 1] - (g.fwd ? 1 : 0);
        if (head[i]) {
            const int chunks = gl < 6 ? 1 : max(1, (past - first + 64 * e - 1) / (64 * e));
            const int rows = min(64 >> gl, rend[run[i]] - i);
            step[sidx[i]] = Step{i, gl | el << 8 | rows << 16, (unsigned)o64, chunks};
        }
        row[i] = lf[r];
        diag[i] = cv[g.fwd ? past : first - 1];
    }
    each_entry(
        first, past,
        [&](int k, int from, int cl, int at0, int base64) {
            const int gl = class_gl(cl), e = 1 << class_el(cl), n = k - from;
            // entries go round the row's lanes, then round the lane's places
            const int l = (at0 << gl) + (n & ((1 << gl) - 1)), t = n >> gl;
            const size_t at =
                (size_t)(unsigned)base64 * 64 + (size_t)(t / e) * 64 * e + (size_t)l * e + t % e;
            col[at] = newpos[cc[k]];
            val[at] = -cv[k];
        },
        first, c, k0, o64);
}

int bits_for(long n) {
    int b = 1;
    while ((1L << b) < n + 1) b++;
    return b;
}

}  // namespace

struct FlowPlan {
    Arena mem{1 << 20};
    int nsteps = 0;
    Step *d_step = nullptr;
    int *d_col = nullptr, *d_row = nullptr, *d_ctl = nullptr;
    double *d_val = nullptr, *d_diag = nullptr;
    int ncu = 0;
    ~FlowPlan() { mem.release(); }
};

void flow_destroy(rb_plan *p) {
    delete p->flow;
    p->flow = nullptr;
}

size_t flow_bytes(const rb_plan *p) { return p->flow ? p->flow->mem.bytes : 0; }

rb_status build_flow(rb_plan *p, const int *d_rp, const int *d_cc, const double *d_cv,
                     hipStream_t s) {
    const int m = p->m;
    if (m == 0 || p->nparts > 1 || (long)p->nlevel * 16 > 0x7fffffffL ||
        8L * m > 0x7fffffffL)
        return RB_OK;
    Arena tmp(64 * (size_t)m + (1 << 20));
    struct Guard {
        Arena &a;
        ~Guard() { a.release(); }
    } guard{tmp};
    int *k0, *v0, *key, *order, *run, *rend, *newpos, *head, *sidx, *size, *off;
    for (int **q : {&k0, &v0, &key, &order, &run, &rend, &newpos}) RB_TRY(tmp.alloc(q, m));
    for (int **q : {&head, &sidx, &size, &off}) RB_TRY(tmp.alloc(q, (size_t)m + 1));
    const RowGeom g{m, p->subst == 0, p->nlevel};
    RB_HIP(hipMemsetAsync(head + m, 0, sizeof(int), s));
    k_fl_key<<<nblk(m), kT, 0, s>>>(g, d_rp, p->d_levelPtr, k0, v0);
    RB_HIP(hipGetLastError());
    RB_TRY(sort_pairs_i32(k0, key, v0, order, m, bits_for((long)p->nlevel * 16), s, tmp));
    k_fl_heads<<<nblk(m), kT, 0, s>>>(key, m, k0);
    RB_HIP(hipGetLastError());
    RB_TRY(inclusive_max_i32(k0, run, m, s, tmp));
    k_fl_steps<<<nblk(m), kT, 0, s>>>(key, run, order, g, head, rend, newpos);
    k_fl_size<<<nblk((long)m + 1), kT, 0, s>>>(key, order, g, d_rp, head, size);
    RB_HIP(hipGetLastError());
    RB_TRY(exclusive_scan_i32(head, sidx, m + 1, s, tmp));
    RB_TRY(exclusive_scan_i32(size, off, m + 1, s, tmp));
    int nsteps = 0, n64 = 0;
    RB_HIP(hipMemcpyAsync(&nsteps, sidx + m, sizeof(int), hipMemcpyDeviceToHost, s));
    RB_HIP(hipMemcpyAsync(&n64, off + m, sizeof(int), hipMemcpyDeviceToHost, s));
    RB_HIP(hipStreamSynchronize(s));
    std::unique_ptr<FlowPlan> F(new FlowPlan());
    F->nsteps = nsteps;
    Arena &A = F->mem;
    const size_t ne = (size_t)(unsigned)n64 * 64;
    RB_TRY(A.alloc(&F->d_step, nsteps));
    RB_TRY(A.alloc(&F->d_col, ne));
    RB_TRY(A.alloc(&F->d_val, ne));
    RB_TRY(A.alloc(&F->d_row, m));
    RB_TRY(A.alloc(&F->d_diag, m));
    RB_TRY(A.alloc(&F->d_ctl, 2 * kGroups * kCtl));
    k_fl_blank<<<nblk((long)ne), kT, 0, s>>>(F->d_col, F->d_val, (long)ne);
    k_fl_fill<<<nblk(m), kT, 0, s>>>(key, run, rend, order, head, sidx, off, g, d_rp, d_cc, d_cv,
                                     newpos, p->d_levelItem, F->d_step, F->d_col, F->d_val,
                                     F->d_row, F->d_diag);
    RB_HIP(hipGetLastError());
    int dev = 0, ncu = 0;
    RB_HIP(hipGetDevice(&dev));
    RB_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    F->ncu = ncu;
    RB_HIP(hipStreamSynchronize(s));
    p->flow = F.release();
    return RB_OK;
}

template <int CP, int CL>
static rb_status flow_columns(rb_plan *p, const double *b, long ldb, double *x, long ldx,
                              int ncol, double *xs, int *ctl, hipStream_t s) {
    const FlowPlan *F = p->flow;
    const int groups = (ncol + CP * CL - 1) / (CP * CL);
    const long n = (long)p->m * CP * CL * groups;
    k_flow_reset<<<nblk((n + 1) / 2), kT, 0, s>>>(xs, n, ctl, groups * kCtl);
    FlowArgs a{F->d_step, F->d_col, F->d_val, F->d_row, F->d_diag, b, x, ldb, ldx, ncol,
               p->m, F->nsteps, xs, ctl, p->d_status, p->spin_limit};
    const long takes = (long)F->nsteps * CL;
    const int grid = (int)std::max(
        std::min(16L, (takes + kWaves - 1) / kWaves),
        std::min((long)F->ncu / groups, 10 * takes / ((long)kWaves * std::max(1, p->nlevel))));
    mark_start(p, s);
    if (groups > 1)
        k_flow<2, kCols / 2, true><<<dim3(grid, groups), kWaves * 64, 0, s>>>(a);
    else
        k_flow<CP, CL, false><<<grid, kWaves * 64, 0, s>>>(a);
    RB_HIP(hipGetLastError());
    mark_end(p, s);
    return RB_OK;
}

// the x buffer of n columns together: m values each for 1, 2, 4 or 8, or for
// groups of 8
static int flow_width(int n) {
    return n <= 2 ? n : n <= 4 ? 4 : (n + kCols - 1) / kCols * kCols;
}

rb_status solve_flow(rb_plan *p, const double *d_b, int ldb, double *d_x, int ldx, int nrhs,
                     hipStream_t s, double *ws, size_t ws_bytes) {
    const int m = p->m;
    if (m == 0) return RB_OK;
    const size_t col = sizeof(double) * (size_t)m;
    // columns at a time: a power of two up to a group, or whole groups (one
    // after another each pays the chain of levels: 32 columns of 30,000
    // power-law rows 646 us, of 900,000 2,119; together 175 and 1,642; the
    // block walk 416 and 3,274)
    int cap = kCols;
    while (cap > 1 && (long)m * cap * 8 > 0x7fffffffL) cap /= 2;
    if (cap == kCols) cap = std::max(1, std::min(kGroups, walk_cols(p) / kCols)) * kCols;
    // a group's b is copied first where x would overwrite what is still to be
    // read
    const bool copy = part_overlap(d_b, ldb, d_x, ldx, m, nrhs);
    int group = copy ? std::min(nrhs, walk_cols(p)) : nrhs;  // columns copied at a time
    double *xs = ws, *bc = nullptr;
    // (a solve on a caller's workspace may run beside one on the plan's)
    int *ctl = p->flow->d_ctl + (ws ? kGroups * kCtl : 0);
    if (ws) {
        if (copy) group = 1;
        while (cap > kCols && cap * col > ws_bytes) cap -= kCols;
        while (cap > 1 && cap * col > ws_bytes) cap /= 2;
        if ((copy ? 2 : 1) * col > ws_bytes) {
            set_error(RB_ERR_INVALID_ARG, "workspace too small for one column");
            return RB_ERR_INVALID_ARG;
        }
        bc = ws + m;
    } else {
        RB_TRY(scratch_cols(p, copy ? std::max(group, flow_width(std::min(cap, nrhs)))
                                    : flow_width(std::min(cap, nrhs)), s));
        xs = p->d_xperm;
        bc = p->d_bperm;
    }
    ColumnGroups grp;
    RB_TRY(column_groups(d_b, ldb, d_x, ldx, m, nrhs, group, &grp));
    for (int i = 0; i < grp.n; i++) {
        const int g = grp.at(i);
        const int ng = std::min(group, nrhs - g);
        const double *b = d_b + (size_t)g * ldb;
        long lb = ldb;
        if (copy) {
            RB_HIP(hipMemcpy2DAsync(bc, col, b, sizeof(double) * ldb, col, ng,
                                    hipMemcpyDeviceToDevice, s));
            b = bc;
            lb = m;
        }
        for (int k = 0; k < ng; k += cap) {
            const int n = std::min(cap, ng - k);
            const double *bk = b + (size_t)k * lb;
            double *xk = d_x + (size_t)(g + k) * ldx;
            switch (flow_width(n)) {
            case 1: RB_TRY((flow_columns<1, 1>(p, bk, lb, xk, ldx, n, xs, ctl, s))); break;
            case 2: RB_TRY((flow_columns<2, 1>(p, bk, lb, xk, ldx, n, xs, ctl, s))); break;
            case 4: RB_TRY((flow_columns<2, 2>(p, bk, lb, xk, ldx, n, xs, ctl, s))); break;
            default: RB_TRY((flow_columns<2, 4>(p, bk, lb, xk, ldx, n, xs, ctl, s))); break;
            }
        }
    }
    return RB_OK;
}

}  // namespace rb
