// Level schedule: the whole solve in one launch, one workgroup per
// (independent part of the matrix, right-hand side), x in LDS.
//
// For deep factors whose levels are narrow a level costs what it takes one
// row to see another's x.  Through device memory that is 1-3 us; inside one
// workgroup it is an LDS write, a workgroup barrier and an LDS read.  The
// rows are put in order (part, level, lanes per row) and cut into steps of
// 64 lanes; a part's steps go round robin to the workgroup's step waves.  A
// wave reads a step's records into registers as soon as its previous step
// is done -- several levels ahead of the step's turn -- then takes part in
// every level's barrier, and at its own level needs only the LDS: gather
// the entries' x, multiply, add, write x.
//
// The LDS holds a ring of b and x: row u of the part (in the storage order,
// below) has slot u mod ring, which holds b_u until the row is solved
// and x_u afterwards.  The swap waves move blocks of 256 consecutive rows
// through it: once every reader of a block's x is past, x goes out and b of
// the block one ring length ahead comes in, both as contiguous accesses.
// (With b gathered and x scattered by the step waves, 64 addresses per
// access, the address unit of a compute unit was busy 490 cycles per step:
// 64 uneven banded factors of 1e3..2e5 rows, 1002 columns, took 985 us.)
//
// Bound: the serial chain, one level after another.  A level of the banded
// factor takes 0.19 us: about 128 cycles for the gather, 50 for the sums, 70
// for the write, the rest barrier and issue; 2.69 us is what its bytes would
// take.  (A tag and a value polled per entry, one after another: 910 us.)
// A wave sums the entries that read older levels before the last barrier
// (257 -> 243 us) and ends its level before it issues its next loads (22.5
// -> 16.2 us on 3,000 rows).  Batches run at what the address units take.
//
// Storage order: the caller's rows where a ring that fits the LDS exists
// for them (rows that are solved close together lie close together);
// otherwise the rows' solve order, with a pass before and after the launch.
// Parts: the factors of a batch (independent by construction); a single
// factor is one part.
#include <algorithm>
#include <memory>
#include <type_traits>
#include <vector>

#include "rb_internal.h"

namespace rb {

namespace {

constexpr int kT = 256;
constexpr int kEnt = 8;             // entries per lane
constexpr int kMaxLen = 64 * kEnt;  // longest row (off-diagonal entries)
constexpr int kMinRing = 1024, kMaxRing = 16384;  // LDS ring, rows
// Rows a swap moves, and the waves.  Banded factor of 100,000 rows (973
// levels) / the batch of 64 above: 128 rows 200 / 606 us, 256 rows 193 / 606;
// one swap wave (128 rows) 236 / 632, two 200 / 606.  With 8 waves in all
// the records arrive too late (256 us against 242 with 16, before the swaps).
constexpr int kBlock = 256;
constexpr int kWaves = 16, kSwapWaves = 2, kStepWaves = kWaves - kSwapWaves;

inline int nblk(long n, int t = kT) { return (int)((n + t - 1) / t); }

// 16-byte words of a lane's record: the entries' ring slots (16 bits each),
// then their negated values -a_ij
template <class T>
constexpr int words() { return 1 + kEnt * (int)sizeof(T) / 16; }

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// A step: up to 64 lanes of rows of one level, `lanes per row` alike.
struct Step {
    int level;  // within the part
    int shape;  // log2 lanes per row | entries per lane of the previous level << 8 |
                // lanes in use << 16
};

struct Part {
    int step0, step1;  // its steps
    int levels;
    int row0, rows;    // its rows in storage order
    int swap0, swaps;  // its swaps: block k out, block k + ring / kBlock in
};

template <class T>
struct LevelArgs {
    const uint4 *rec;            // [nsteps][words][64] lane records
    const unsigned short *slot;  // [nsteps][64] the row's ring slot; `ring`: none
    const Step *step;            // [nsteps]
    const int *swap;             // level after which a swap may run, ascending per part
    const T *dinv;               // [nsteps][64] 1 / a_ii
    const Part *part;            // [nparts]
    Part only;                   // the part when it is the only one
    int nparts, ring;
    const int *job;  // per workgroup: column << 16 | part, or -1; null: see k_level
    const double *b;             // storage order; or per part where bp is not null
    double *x;
    long ldb, ldx;
    const double *const *bp;
    double *const *xp;
    const int *ldbp, *ldxp;
    const int *cap;          // per part: columns it has (null: all)
    bool add;                // T float: x += the correction, else x = it
    const int *left, *done;  // refinement: nothing to do at 0 / for this column
};

// Buffer resources: a wave-uniform base and a size; an access outside the
// size reads zero or is dropped, so an empty lane needs no branch.  Every
// load of the step loop is one of these: no branch lies between the loads,
// so the waits count them exactly.
__device__ inline __amdgpu_buffer_rsrc_t buf(const void *p, long bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0,
                                             (int)min(bytes, 0x7fffffffL), 0x00020000);
}
// a wave-uniform value in scalar registers
__device__ inline int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
template <class P>
__device__ inline P *uniform(P *p) {
    const unsigned long long v = (unsigned long long)p;
    const unsigned lo = (unsigned)uniform((int)v), hi = (unsigned)uniform((int)(v >> 32));
    return (P *)((unsigned long long)hi << 32 | lo);
}
constexpr int kNone = -8;  // a byte offset outside every buffer

template <class T>
__device__ inline T load_val(__amdgpu_buffer_rsrc_t r, int off, int soff) {
    if constexpr (sizeof(T) == 4)
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, off, soff, 0));
    else
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, off, soff, 0));
}
template <class T>
__device__ inline void store_val(T v, __amdgpu_buffer_rsrc_t r, int off, int soff) {
    if constexpr (sizeof(T) == 4)
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, off, soff, 0);
    else
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, off, soff, 0);
}

// T double: the solve, x = T^-1 b.  T float: the refinement's inner solve,
// x (+)= T^-1 (float) b.
template <class T>
__global__ void __launch_bounds__(kWaves * 64, 8) k_level(LevelArgs<T> a) {
    extern __shared__ double lds_raw[];
    T *ring = (T *)lds_raw;
    constexpr int KW = words<T>();
    constexpr bool f32 = sizeof(T) == 4;
    if (f32 && *a.left == 0) return;
    int part, col;
    if (a.job) {
        const int j = uniform(a.job[blockIdx.x]);
        if (j < 0) return;
        part = j & 0xffff;
        col = j >> 16;
    } else {
        part = blockIdx.x % a.nparts;
        col = blockIdx.x / a.nparts;
    }
    if ((f32 && a.done[col]) || (a.cap && col >= a.cap[part])) return;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    Part pt = a.only;
    if (a.nparts > 1) {
        const Part v = a.part[part];
        pt = Part{uniform(v.step0), uniform(v.step1), uniform(v.levels), uniform(v.row0),
                  uniform(v.rows),  uniform(v.swap0), uniform(v.swaps)};
    }
    const int mask = a.ring - 1;
    const double *pb = a.b + col * a.ldb + pt.row0;
    double *px = a.x + col * a.ldx + pt.row0;
    if (a.bp) {
        pb = uniform(a.bp[part] + col * (long)a.ldbp[part]);
        px = uniform(a.xp[part] + col * (long)a.ldxp[part]);
    }
    const __amdgpu_buffer_rsrc_t bb = buf(pb, 8L * pt.rows), xx = buf(px, 8L * pt.rows);
    const bool add = f32 && a.add;
    int cur = 0;  // levels complete
    auto barrier = [&]() {
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        cur++;
    };
    // the ring's first rows
    for (int u = threadIdx.x; u < min(a.ring, pt.rows); u += kWaves * 64)
        ring[u] = T(pb[u]);
    if (threadIdx.x == 0) ring[a.ring] = T(0);

    if (wave < kStepWaves) {
        const int ns = pt.step1 - pt.step0;
        const size_t l0 = (size_t)pt.step0 * 64;
        const __amdgpu_buffer_rsrc_t rec = buf(a.rec + l0 * KW, (long)ns * KW * 1024),
                                     slots = buf(a.slot + l0, (long)ns * 128),
                                     dinv = buf(a.dinv + l0, (long)ns * 64 * sizeof(T)),
                                     step = buf(a.step + pt.step0, (long)ns * sizeof(Step));
        // A wave's step and its next one: level and shape in scalar
        // registers, those of the one after on their way in `ahead`.
        u32x4 w[KW];
        u32x2 ahead;
        int sl;  // the row's ring slot
        T dv;
        auto load_step = [&](int s) {  // (past the end: zeros, a step without lanes)
            return __builtin_amdgcn_raw_buffer_load_b64(step, min(s, ns) * (int)sizeof(Step), 0, 0);
        };
        auto load = [&](int s, int shape) {
            const int r = lane < shape >> 16 ? lane * 16 : kNone;
            sl = __builtin_amdgcn_raw_buffer_load_b16(slots, lane * 2, s * 128, 0);
            dv = load_val<T>(dinv, lane * (int)sizeof(T), s * (64 * (int)sizeof(T)));
#pragma unroll
            for (int k = 0; k < KW; k++)
                w[k] = __builtin_amdgcn_raw_buffer_load_b128(rec, r, (s * KW + k) * 1024, 0);
        };
        int s = wave;
        u32x2 s1 = load_step(s), s2 = load_step(s + kStepWaves);
        ahead = load_step(s + 2 * kStepWaves);
        asm volatile("" : "+v"(s1), "+v"(s2), "+v"(ahead));
        int lev = uniform((int)s1.x), shape = uniform((int)s1.y);
        int lev1 = uniform((int)s2.x), shape1 = uniform((int)s2.y);
        load(min(s, ns), shape);
        __syncthreads();
        while (s < ns) {
            while (cur < lev - 1) barrier();
            // everything below has been on its way for several levels
#pragma unroll
            for (int k = 0; k < KW; k++) asm volatile("" : "+v"(w[k]));
            asm volatile("" : "+v"(sl), "+v"(dv), "+v"(ahead));
            unsigned at[kEnt];
            const unsigned ow[4] = {w[0].x, w[0].y, w[0].z, w[0].w};
#pragma unroll
            for (int j = 0; j < kEnt; j++) {
                at[j] = (j & 1 ? ow[j / 2] >> 16 : ow[j / 2] & 0xffffu) * (unsigned)sizeof(T);
                asm volatile("" : "+v"(at[j]));
            }
            T c[kEnt];
#pragma unroll
            for (int j = 0; j < kEnt; j++) {
                if constexpr (f32) c[j] = __uint_as_float(w[1 + j / 4][j % 4]);
                else
                    c[j] = __hiloint2double(w[1 + j / 2][j % 2 * 2 + 1], w[1 + j / 2][j % 2 * 2]);
            }
            const int own = sl & 0xffff;
            // (T float: b goes in last, so that the products are rounded at
            // their own size and not at b's)
            const T bv = ring[own];
            T acc0 = f32 ? T(0) : bv, acc1 = 0;
            // entries [late, kEnt) read levels before the previous one and
            // go in before the last barrier
            auto sum = [&](auto from, auto to) {
                T xv[kEnt];
#pragma unroll
                for (int j = from; j < to; j++) xv[j] = *(const T *)((const char *)ring + at[j]);
#pragma unroll
                for (int j = from; j < to; j++) {
                    if (j & 1) acc1 += c[j] * xv[j];
                    else acc0 += c[j] * xv[j];
                }
            };
            auto sums = [&](auto late) {
                sum(late, std::integral_constant<int, kEnt>());
                asm volatile("" : "+v"(acc0), "+v"(acc1) : "v"(bv));
                if (cur < lev) barrier();
                sum(std::integral_constant<int, 0>(), late);
            };
            const int nl = (shape >> 8) & 255, gl = shape & 255;
            if (nl <= 2) sums(std::integral_constant<int, 2>());
            else if (nl <= 4) sums(std::integral_constant<int, 4>());
            else sums(std::integral_constant<int, kEnt>());
            acc0 += acc1;
            for (int o = 1; o < (1 << gl); o <<= 1) acc0 += __shfl_xor(acc0, o, 64);
            if (own < a.ring) ring[own] = (f32 ? acc0 + bv : acc0) * dv;
            // x is in the ring: the level ends before the wave's next loads,
            // whose issue would hold every other wave (unless its next step
            // is of the same level)
            s += kStepWaves;
            if (s >= ns || lev1 != lev) barrier();
            lev = lev1;
            shape = shape1;
            lev1 = uniform((int)ahead.x);
            shape1 = uniform((int)ahead.y);
            ahead = load_step(s + 2 * kStepWaves);
            load(min(s, ns), shape);
        }
    } else {
        // Swap k takes block k's x out and brings block k + ring / kBlock
        // in, kDepth of the wave's swaps on their way.
        constexpr int Q = kBlock / 64, kDepth = 2;
        struct In {
            int level;
            double b[Q], old[Q];  // (old: T float, x so far)
        };
        const __amdgpu_buffer_rsrc_t swap = buf(a.swap + pt.swap0, 4L * pt.swaps);
        auto load = [&](int k, In &in) {  // (past the end: the last one again)
            k = max(0, min(k, pt.swaps - 1));
            const int u = k * kBlock, v = min(u + a.ring, pt.rows);
            in.level = __builtin_amdgcn_raw_buffer_load_b32(swap, 0, k * 4, 0);
#pragma unroll
            for (int q = 0; q < Q; q++) {
                const int l = q * 64 + lane;
                in.b[q] = load_val<double>(bb, l * 8, v * 8);
                if constexpr (f32) in.old[q] = add ? load_val<double>(xx, l * 8, u * 8) : 0.0;
            }
        };
        using Bits = std::conditional_t<f32, unsigned, unsigned long long>;
        auto run = [&](int k, In &in, const In &next) {
            const int lev = uniform(in.level);
            while (cur < lev - 1) barrier();
            T v[Q];
#pragma unroll
            for (int q = 0; q < Q; q++) v[q] = T(in.b[q]);
            if (cur < lev) barrier();
            const bool real = k < pt.swaps;  // (otherwise the spare block)
            T *at = ring + (real ? (k * kBlock) & mask : a.ring + 2) + lane;
#pragma unroll
            for (int q = 0; q < Q; q++)
                v[q] = __builtin_bit_cast(
                    T, __hip_atomic_exchange((Bits *)(at + q * 64), __builtin_bit_cast(Bits, v[q]),
                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
            // the level ends before the stores and loads, whose issue would
            // hold every other wave (unless the next swap is due too)
            if (real && (k + kSwapWaves >= pt.swaps || uniform(next.level) > cur)) barrier();
#pragma unroll
            for (int q = 0; q < Q; q++)
                store_val<double>(f32 ? in.old[q] + (double)v[q] : (double)v[q], xx,
                                  real ? (q * 64 + lane) * 8 : kNone, real ? k * (kBlock * 8) : 0);
            load(k + kDepth * kSwapWaves, in);
        };
        In in[kDepth];
        int k = wave - kStepWaves;
#pragma unroll
        for (int i = 0; i < kDepth; i++) load(k + i * kSwapWaves, in[i]);
        // (all there before the loop: its waits then count the loads of the
        // passes before only)
#pragma unroll
        for (int i = 0; i < kDepth; i++) {
            asm volatile("" : "+v"(in[i].level));
#pragma unroll
            for (int q = 0; q < Q; q++) asm volatile("" : "+v"(in[i].b[q]));
        }
        __syncthreads();
        // whole rounds of kDepth, without a way out in between (which would
        // make the waits at the head count the fewest loads of any way)
        for (; k < pt.swaps; k += kDepth * kSwapWaves)
#pragma unroll
            for (int i = 0; i < kDepth; i++)
                run(k + i * kSwapWaves, in[i], in[(i + 1) % kDepth]);
    }
    while (cur < pt.levels) barrier();
    __syncthreads();
    // the blocks still in the ring
    for (int u = pt.swaps * kBlock + threadIdx.x; u < pt.rows; u += kWaves * 64)
        px[u] = f32 && add ? px[u] + (double)ring[u & mask] : (double)ring[u & mask];
}

constexpr int kPassCols = 8;  // columns per thread of the two passes

// b into storage order (the rows' solve order): sb[u] = b[row[u]].  A
// thread's columns are all read before the first is written, so the loads of
// one are not held up by the others.
__global__ void __launch_bounds__(kT)
    k_level_in(const double *b, long ldb, const int *__restrict__ row, int m, int ncol,
               double *__restrict__ sb, const int *__restrict__ left) {
    if (left && *left == 0) return;
    const int u = blockIdx.x * kT + threadIdx.x, cb = blockIdx.y * kPassCols;
    if (u >= m) return;
    const double *at = b + row[u] + cb * ldb;
    const int n = min(kPassCols, ncol - cb);
    double v[kPassCols];
#pragma unroll
    for (int q = 0; q < kPassCols; q++) v[q] = q < n ? at[q * ldb] : 0.0;
#pragma unroll
    for (int q = 0; q < kPassCols; q++)
        if (q < n) sb[(size_t)(cb + q) * m + u] = v[q];
}

// x out of storage order; ADD: x += (columns not yet converged)
template <bool ADD>
__global__ void __launch_bounds__(kT)
    k_level_out(double *x, long ldx, const int *__restrict__ row, int m, int ncol,
                const double *__restrict__ sx, const int *__restrict__ left,
                const int *__restrict__ done) {
    if (left && *left == 0) return;
    const int u = blockIdx.x * kT + threadIdx.x, cb = blockIdx.y * kPassCols;
    if (u >= m) return;
    double *at = x + row[u] + cb * ldx;
    const int n = min(kPassCols, ncol - cb);
    double v[kPassCols];
#pragma unroll
    for (int q = 0; q < kPassCols; q++) {
        v[q] = q < n ? sx[(size_t)(cb + q) * m + u] : 0.0;
        if (ADD && q < n) v[q] += at[q * ldx];
    }
#pragma unroll
    for (int q = 0; q < kPassCols; q++)
        if (q < n && !(ADD && done[cb + q])) at[q * ldx] = v[q];
}

// ------------------------------------------------------------- build

struct RowGeom {
    int m, fwd, nlev;
};

__device__ inline int glog_of(int len) {
    int g = 0;
    while ((kEnt << g) < len) g++;
    return g;
}

// Levels.  A row may run in any level from its own (the longest path to it)
// to the one before the first row that needs it; it is put kAhead levels
// before that row if it can be: a few rows that are ready early (without
// dependencies, say) would otherwise hold their ring slots for hundreds of
// levels, while rows just before their readers leave those nothing to sum
// ahead of their turn.  A row that no other needs goes where the rest of its
// block of rows begins.
constexpr int kAhead = 8;
__global__ void k_lv_own(RowGeom g, const int *__restrict__ rp, const int *__restrict__ lp,
                         int *level, int *need, int *longest) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    int len = 0;
    if (q < g.m) {
        const int r = g.fwd ? q : g.m - 1 - q;
        len = rp[r + 1] - rp[r] - 1;
        int lo = 0, hi = g.nlev;  // last level that starts at or before q
        while (hi - lo > 1) {
            const int mid = (lo + hi) / 2;
            if (lp[mid] <= q) lo = mid;
            else hi = mid;
        }
        level[r] = lo;
        need[r] = 0x7fffffff;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) len = max(len, __shfl_xor(len, o, 64));
    if ((threadIdx.x & 63) == 0 && len > 0) atomicMax(longest, len);
}

// the first level that needs a row's x
__global__ void k_lv_need(int m, const int *__restrict__ rp, const int *__restrict__ cc,
                          const int *__restrict__ level, int *need) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = r < m;
    each_entry(
        live ? rp[r] : 0, live ? rp[r + 1] : 0,
        [&](int k, int row, int l) {
            int *at = need + cc[k];
            if (cc[k] != row && *(volatile int *)at > l) atomicMin(at, l);
        },
        r, live ? level[r] : 0);
}

// Blocks of kBlock rows, counted part by part (a part's rows lie together; its
// first row and block: off and blk0, null for a single part)
struct RowBlocks {
    const int *part, *off, *blk0;
    __device__ int part_of(int row) const { return part ? part[row] : 0; }
    __device__ int of(int row) const {
        const int p = part_of(row);
        return (off ? blk0[p] : 0) + (row - (off ? off[p] : 0)) / kBlock;
    }
};

__global__ void k_lv_block_start(int m, const int *__restrict__ level,
                                 const int *__restrict__ need, const int *__restrict__ lf,
                                 RowBlocks rb, int *start) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= m || need[r] == 0x7fffffff) return;
    int *at = start + rb.of(lf[r]);
    const int l = max(level[r], need[r] - kAhead);
    if (*(volatile int *)at > l) atomicMin(at, l);
}

// solve-order row q: its sort key (part, level, log2 lanes per row)
__global__ void k_lv_key(RowGeom g, const int *__restrict__ rp, const int *__restrict__ level,
                         const int *__restrict__ need, const int *__restrict__ start,
                         const int *__restrict__ lf, RowBlocks rb, int *key, int *val) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= g.m) return;
    const int r = g.fwd ? q : g.m - 1 - q;
    const int len = rp[r + 1] - rp[r] - 1, p = rb.part_of(lf[r]);
    int l = max(level[r], need[r] - kAhead);
    if (need[r] == 0x7fffffff) {
        const int s = start[rb.of(lf[r])];
        l = s == 0x7fffffff ? level[r] : max(level[r], s);
    }
    key[q] = (p * g.nlev + l) * 8 + glog_of(min(len, kMaxLen));
    val[q] = q;
}

// first positions of every (part, level, lanes) run and (part, level) level
__global__ void k_lv_heads(const int *__restrict__ key, int m, int *run, int *lev) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    run[i] = i > 0 && key[i] == key[i - 1] ? 0 : i;
    lev[i] = i > 0 && (key[i] >> 3) == (key[i - 1] >> 3) ? 0 : i;
}

// per position: first of a step; per run (at its first position): end;
// permuted row -> position
__global__ void k_lv_steps(const int *__restrict__ key, const int *__restrict__ run,
                           const int *__restrict__ lev, const int *__restrict__ order,
                           RowGeom g, int *head, int *rend, int *newpos) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= g.m) return;
    const int gl = key[i] & 7;
    head[i] = ((i - run[i]) & ((64 >> gl) - 1)) == 0;
    const bool last = i + 1 == g.m;
    if (last || key[i + 1] != key[i]) rend[run[i]] = i + 1;
    const int q = order[i];
    newpos[g.fwd ? q : g.m - 1 - q] = i;
}

// What the ring must respect, per block of kBlock rows in the caller's order
// (c) and in solve order (p): the first level with a row of the block and
// the last level that needs one of its x.
__global__ void k_lv_blocks(const int *__restrict__ key, const int *__restrict__ order,
                            RowGeom g, const int *__restrict__ rp, const int *__restrict__ cc,
                            const int *__restrict__ newpos, const int *__restrict__ lf,
                            const int *__restrict__ off, const int *__restrict__ blk0,
                            int *first_c, int *last_c, int *first_p, int *last_p) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = i < g.m;
    const int r = !live ? 0 : g.fwd ? order[i] : g.m - 1 - order[i];
    const int pl = live ? key[i] >> 3 : 0, p = pl / g.nlev;
    // (the plain read first: most atomics would change nothing)
    if (live) {
        const int l = pl - p * g.nlev, o = off ? off[p] : 0;
        int *at = first_c + blk0[p] + (lf[r] - o) / kBlock;
        if (*(volatile int *)at > l) atomicMin(at, l);
        // (levels rise with the position)
        if ((i - o) % kBlock == 0) first_p[blk0[p] + (i - o) / kBlock] = l;
    }
    // (the diagonal: the row itself)
    each_entry(
        live ? rp[r] : 0, live ? rp[r + 1] : 0,
        [&](int k, int q, int l) {
            const int o = off ? off[q] : 0, b0 = blk0[q];
            auto high = [&](int *at) {
                if (*(volatile int *)at < l) atomicMax(at, l);
            };
            high(last_c + b0 + (lf[cc[k]] - o) / kBlock);
            high(last_p + b0 + (newpos[cc[k]] - o) / kBlock);
        },
        p, pl - p * g.nlev);
}

// empty lanes: no row, coefficients 0 on the ring's zero
__global__ void k_lv_blank(uint4 *rec, unsigned short *slot, double *dinv, long nlanes,
                           int ring) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nlanes) return;
    const long s = t / 64;
    const int l = (int)(t & 63);
    const unsigned z = (unsigned)ring << 16 | (unsigned)ring;
    constexpr int KW = words<double>();
    rec[s * KW * 64 + l] = make_uint4(z, z, z, z);
#pragma unroll
    for (int k = 1; k < KW; k++) rec[(s * KW + k) * 64 + l] = make_uint4(0, 0, 0, 0);
    slot[t] = (unsigned short)ring;
    dinv[t] = 0.0;
}

// direct: storage order is the caller's, else the position
__global__ void k_lv_fill(const int *__restrict__ key, const int *__restrict__ run,
                          const int *__restrict__ lev, const int *__restrict__ rend,
                          const int *__restrict__ order, const int *__restrict__ head,
                          const int *__restrict__ sidx, RowGeom g,
                          const int *__restrict__ rp, const int *__restrict__ cc,
                          const double *__restrict__ cv, const double *__restrict__ invd,
                          const int *__restrict__ newpos, const int *__restrict__ lf,
                          const int *__restrict__ off, int ring, bool direct, uint4 *rec,
                          unsigned short *slot, int *row, double *dinv, Step *step,
                          Part *part) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= g.m) return;
    constexpr int KW = words<double>();
    const int gl = key[i] & 7, lv = key[i] >> 3, p = lv / g.nlev;
    const int s = sidx[i] + head[i] - 1;
    const int l0 = ((i - run[i]) & ((64 >> gl) - 1)) << gl;  // the row's first lane
    const int used = min(64, (rend[run[i]] - i) * (1 << gl) + l0);
    const int r = g.fwd ? order[i] : g.m - 1 - order[i];
    const int o = off ? off[p] : 0;
    auto slot_of = [&](int r_, int i_) {
        return (unsigned short)(((direct ? lf[r_] : i_) - o) & (ring - 1));
    };
    if (head[i]) {
        step[s].level = lv - p * g.nlev;
        atomicMax(&part[p].step1, s + 1);
        atomicMax(&part[p].levels, lv - p * g.nlev + 1);
        if (i == 0 || (key[i - 1] >> 3) / g.nlev != p) part[p].step0 = s;
    }
    row[i] = lf[r];
    dinv[(size_t)s * 64 + l0] = invd[r];
    slot[(size_t)s * 64 + l0] = slot_of(r, i);
    // entries go round the row's lanes, those of the previous level first
    uint4 *base = rec + (size_t)s * KW * 64 + l0;
    const int from = lev[i] > 0 ? lev[lev[i] - 1] : 0;
    int n = 0;
    for (int late = 1; late >= 0; late--) {
        for (int k = rp[r]; k < rp[r + 1]; k++) {
            if (cc[k] == r || (newpos[cc[k]] >= from) != late) continue;
            uint4 *b = base + (n & ((1 << gl) - 1));
            const int j = n >> gl;
            ((unsigned short *)b)[j] = slot_of(cc[k], newpos[cc[k]]);
            ((double *)(b + (1 + j / 2) * 64))[j & 1] = -cv[k];
            n++;
        }
        if (late)
            atomicMax(&step[s].shape, gl | ((n + (1 << gl) - 1) >> gl) << 8 | used << 16);
    }
}

__global__ void k_lv_to32(const uint4 *__restrict__ rec, long nlanes, uint4 *rec32) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nlanes) return;
    const long s = t / 64;
    const int l = (int)(t & 63);
    constexpr int K6 = words<double>(), K3 = words<float>();
    rec32[s * K3 * 64 + l] = rec[s * K6 * 64 + l];
#pragma unroll
    for (int k = 0; k < kEnt / 4; k++) {
        const double2 p = ((const double2 *)rec)[(s * K6 + 1 + 2 * k) * 64 + l];
        const double2 q = ((const double2 *)rec)[(s * K6 + 2 + 2 * k) * 64 + l];
        rec32[(s * K3 + 1 + k) * 64 + l] =
            make_uint4(__float_as_uint((float)p.x), __float_as_uint((float)p.y),
                       __float_as_uint((float)q.x), __float_as_uint((float)q.y));
    }
}

__global__ void k_lv_f32(const double *__restrict__ a, long n, float *o) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) o[i] = (float)a[i];
}

__global__ void k_lv_set(int *a, int n, int v) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = v;
}

int bits_for(long n) {
    int b = 1;
    while ((1L << b) < n + 1) b++;
    return b;
}

}  // namespace

struct LevelPlan {
    Arena mem{1 << 20};  // one chunk for a small factor's tables
    int nsteps = 0, nparts = 1, ring = 0;
    bool direct = false;  // storage order is the caller's
    uint4 *d_rec = nullptr, *d_rec32 = nullptr;
    unsigned short *d_slot = nullptr;
    Step *d_step = nullptr;
    int *d_row = nullptr, *d_swap = nullptr;  // caller's row of a position
    double *d_dinv = nullptr;
    float *d_dinv32 = nullptr;
    Part *d_part = nullptr;
    std::vector<Part> parts;  // host copy
    ~LevelPlan() { mem.release(); }
};

// The swaps' levels for a ring, or false when the ring is too short.  Block
// k may leave once every level up to last[k] is complete; block k + ring /
// kBlock comes in then and must be there one level before the first that
// reads its b, which happens a level early.
static bool plan_swaps(const std::vector<Part> &parts, const std::vector<int> &blk0,
                       const int *first, const int *last, int ring,
                       std::vector<int> &swap, std::vector<Part> &out) {
    const int rb = ring / kBlock;
    swap.clear();
    out = parts;
    for (size_t q = 0; q < parts.size(); q++) {
        const int nb = (parts[q].rows + kBlock - 1) / kBlock;
        const int *f = first + blk0[q], *l = last + blk0[q];
        out[q].swap0 = (int)swap.size();
        out[q].swaps = std::max(0, nb - rb);
        int tag = 0;
        for (int k = 0; k + rb < nb; k++) {
            tag = std::max(tag, l[k] + 1);
            if (tag > f[k + rb] - 2) return false;
            swap.push_back(tag);
        }
    }
    return true;
}

void level_destroy(rb_plan *p) {
    delete p->level;
    p->level = nullptr;
}

size_t level_bytes(const rb_plan *p) { return p->level ? p->level->mem.bytes : 0; }

template <class T>
static rb_status allow_lds() {
    RB_HIP(hipFuncSetAttribute((const void *)k_level<T>,
                               hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)(sizeof(double) * (kMaxRing + 2 + kBlock))));
    return RB_OK;
}

// What a single column takes, in us, and what the chain-following schedule
// takes at least where it applies: both from runs on the banded and grid
// factors (973 levels, 1961 steps: 193 us; 549, 1428: 120; 89, 104: 14).
static double level_us(const rb_plan *p, int nsteps) {
    return 0.07 * p->nlevel + 0.06 * nsteps;
}
static double chain_us(const rb_plan *p) { return 20.0 + 0.043 * p->nlevel; }

bool level_beats_chain(const rb_plan *p) {
    return p->level && p->level->nparts == 1 && level_us(p, p->level->nsteps) < chain_us(p);
}

bool level_beats_walk(const rb_plan *p) {
    return p->level && (p->level->nparts > 1 || level_us(p, p->level->nsteps) < 0.45 * p->nlevel);
}

rb_status level_narrow(const rb_plan *p, hipStream_t s, bool *narrow) {
    *narrow = false;
    if (level_us(p, p->nlevel) >= chain_us(p)) return RB_OK;
    std::vector<int> lp(p->nlevel + 1);
    RB_HIP(hipMemcpyAsync(lp.data(), p->d_levelPtr, sizeof(int) * lp.size(),
                          hipMemcpyDeviceToHost, s));
    RB_HIP(hipStreamSynchronize(s));
    int nsteps = 0;
    for (int l = 0; l < p->nlevel; l++) nsteps += (lp[l + 1] - lp[l] + 63) / 64;
    *narrow = level_us(p, nsteps) < chain_us(p);
    return RB_OK;
}

rb_status build_level(rb_plan *p, const int *d_rp, const int *d_cc, const double *d_cv,
                      hipStream_t s) {
    const int m = p->m, np = std::max(1, p->nparts);
    if (m == 0 || np > 0xffff || (long)np * p->nlevel * 8 > 0x7fffffffL) return RB_OK;
    // (levels far too wide for one workgroup are not worth the tables, nor the
    // analysis where their rows alone say so)
    auto too_wide = [&](int nsteps) {
        return p->want_schedule == RB_SCHED_AUTO && np == 1 && level_us(p, nsteps) > 8.0 * chain_us(p);
    };
    if (too_wide(m / 64)) return RB_OK;
    Arena tmp(76 * (size_t)m + (1 << 20));
    struct Guard {
        Arena &a;
        ~Guard() { a.release(); }
    } guard{tmp};
    int *k0, *v0, *key, *order, *run, *lev, *head, *sidx, *rend, *newpos,
        *cnt;
    for (int **q : {&k0, &v0, &key, &order, &run, &lev, &rend, &newpos})
        RB_TRY(tmp.alloc(q, m));
    for (int **q : {&head, &sidx}) RB_TRY(tmp.alloc(q, (size_t)m + 1));
    RB_TRY(tmp.alloc(&cnt, 1));
    const RowGeom g{m, p->subst == 0, p->nlevel};
    RB_HIP(hipMemsetAsync(cnt, 0, sizeof(int), s));
    RB_HIP(hipMemsetAsync(head + m, 0, sizeof(int), s));
    // the parts' rows and blocks
    std::vector<Part> parts(np);
    std::vector<int> blk0(np + 1, 0);
    for (int q = 0; q < np; q++) {
        parts[q] = Part{};
        parts[q].row0 = np > 1 ? p->h_partoff[q] : 0;
        parts[q].rows = (np > 1 && q + 1 < np ? p->h_partoff[q + 1] : m) - parts[q].row0;
        blk0[q + 1] = blk0[q] + (parts[q].rows + kBlock - 1) / kBlock;
    }
    const int nb = blk0[np];
    int *d_blk0, *blk, *start;
    RB_TRY(tmp.alloc(&d_blk0, np));
    RB_TRY(tmp.alloc(&blk, 4 * (size_t)nb));
    RB_TRY(tmp.alloc(&start, nb));
    RB_HIP(hipMemcpyAsync(d_blk0, blk0.data(), sizeof(int) * np, hipMemcpyHostToDevice, s));
    const RowBlocks rb{p->d_part, p->d_partoff, d_blk0};
    // (run, lev and newpos are free until the rows are sorted)
    k_lv_own<<<nblk(m), kT, 0, s>>>(g, d_rp, p->d_levelPtr, lev, newpos, cnt);
    k_lv_need<<<nblk(m), kT, 0, s>>>(m, d_rp, d_cc, lev, newpos);
    k_lv_set<<<nblk(nb), kT, 0, s>>>(start, nb, 0x7fffffff);
    k_lv_block_start<<<nblk(m), kT, 0, s>>>(m, lev, newpos, p->d_levelItem, rb, start);
    k_lv_key<<<nblk(m), kT, 0, s>>>(g, d_rp, lev, newpos, start, p->d_levelItem, rb, k0, v0);
    RB_HIP(hipGetLastError());
    RB_TRY(sort_pairs_i32(k0, key, v0, order, m, bits_for((long)np * p->nlevel * 8), s, tmp));
    k_lv_heads<<<nblk(m), kT, 0, s>>>(key, m, k0, v0);
    RB_HIP(hipGetLastError());
    RB_TRY(inclusive_max_i32(k0, run, m, s, tmp));
    RB_TRY(inclusive_max_i32(v0, lev, m, s, tmp));
    k_lv_steps<<<nblk(m), kT, 0, s>>>(key, run, lev, order, g, head, rend, newpos);
    RB_HIP(hipGetLastError());
    RB_TRY(exclusive_scan_i32(head, sidx, m + 1, s, tmp));
    k_lv_set<<<nblk(2 * nb), kT, 0, s>>>(blk, 2 * nb, 0x7fffffff);
    k_lv_set<<<nblk(2 * nb), kT, 0, s>>>(blk + 2 * nb, 2 * nb, 0);
    k_lv_blocks<<<nblk(m), kT, 0, s>>>(key, order, g, d_rp, d_cc, newpos, p->d_levelItem,
                                       p->d_partoff, d_blk0, blk, blk + 2 * nb, blk + nb,
                                       blk + 3 * nb);
    RB_HIP(hipGetLastError());
    int longest = 0, nsteps = 0;
    std::vector<int> hblk(4 * (size_t)nb);
    RB_HIP(hipMemcpyAsync(&longest, cnt, sizeof(int), hipMemcpyDeviceToHost, s));
    RB_HIP(hipMemcpyAsync(&nsteps, sidx + m, sizeof(int), hipMemcpyDeviceToHost, s));
    RB_HIP(hipMemcpyAsync(hblk.data(), blk, sizeof(int) * hblk.size(), hipMemcpyDeviceToHost,
                          s));
    RB_HIP(hipStreamSynchronize(s));
    if (longest > kMaxLen || 8L * m > 0x7fffffffL) return RB_OK;
    if (too_wide(nsteps)) return RB_OK;
    std::unique_ptr<LevelPlan> L(new LevelPlan());
    std::vector<int> swap;
    for (int c = 1; c >= 0 && L->ring == 0; c--)
        for (int ring = kMinRing; ring <= kMaxRing && L->ring == 0; ring *= 2)
            if (plan_swaps(parts, blk0, hblk.data() + (c ? 0 : nb),
                           hblk.data() + (c ? 2 * nb : 3 * nb), ring, swap, L->parts)) {
                L->ring = ring;
                L->direct = c == 1;
            }
    if (L->ring == 0) return RB_OK;
    L->nsteps = nsteps;
    L->nparts = np;
    Arena &A = L->mem;
    const size_t nl = (size_t)nsteps * 64;
    RB_TRY(A.alloc(&L->d_step, nsteps));
    RB_TRY(A.alloc(&L->d_slot, nl));
    RB_TRY(A.alloc(&L->d_rec, nl * words<double>()));
    RB_TRY(A.alloc(&L->d_row, m));
    RB_TRY(A.alloc(&L->d_dinv, nl));
    RB_TRY(A.alloc(&L->d_part, np));
    RB_TRY(A.alloc(&L->d_swap, swap.size()));
    RB_HIP(hipMemcpyAsync(L->d_part, L->parts.data(), sizeof(Part) * np,
                          hipMemcpyHostToDevice, s));
    if (!swap.empty())
        RB_HIP(hipMemcpyAsync(L->d_swap, swap.data(), sizeof(int) * swap.size(),
                              hipMemcpyHostToDevice, s));
    RB_HIP(hipMemsetAsync(L->d_step, 0, sizeof(Step) * nsteps, s));
    k_lv_blank<<<nblk((long)nl), kT, 0, s>>>(L->d_rec, L->d_slot, L->d_dinv, (long)nl,
                                             L->ring);
    k_lv_fill<<<nblk(m), kT, 0, s>>>(key, run, lev, rend, order, head, sidx, g, d_rp, d_cc,
                                     d_cv, p->d_invd, newpos, p->d_levelItem, p->d_partoff,
                                     L->ring, L->direct, L->d_rec, L->d_slot, L->d_row,
                                     L->d_dinv, L->d_step, L->d_part);
    RB_HIP(hipGetLastError());
    RB_HIP(hipMemcpyAsync(L->parts.data(), L->d_part, sizeof(Part) * np,
                          hipMemcpyDeviceToHost, s));
    RB_HIP(hipStreamSynchronize(s));
    for (const Part &t : L->parts)  // a part's records lie within a buffer's 2 GiB
        if ((long)(t.step1 - t.step0) * words<double>() * 1024 > 0x7fffffffL) return RB_OK;
    if (p->mixed) {
        RB_TRY(A.alloc(&L->d_rec32, nl * words<float>()));
        RB_TRY(A.alloc(&L->d_dinv32, nl));
        k_lv_to32<<<nblk((long)nl), kT, 0, s>>>(L->d_rec, (long)nl, L->d_rec32);
        k_lv_f32<<<nblk((long)nl), kT, 0, s>>>(L->d_dinv, (long)nl, L->d_dinv32);
        RB_HIP(hipGetLastError());
    }
    RB_TRY(allow_lds<double>());
    RB_TRY(allow_lds<float>());
    RB_HIP(hipStreamSynchronize(s));
    p->level = L.release();
    return RB_OK;
}

template <class T>
static LevelArgs<T> level_args(const rb_plan *p) {
    const LevelPlan *L = p->level;
    LevelArgs<T> a{};
    a.slot = L->d_slot;
    a.step = L->d_step;
    a.swap = L->d_swap;
    a.part = L->d_part;
    a.only = L->parts[0];
    if constexpr (sizeof(T) == 4) {
        a.rec = L->d_rec32;
        a.dinv = L->d_dinv32;
    } else {
        a.rec = L->d_rec;
        a.dinv = L->d_dinv;
    }
    a.nparts = L->nparts;
    a.ring = L->ring;
    a.cap = p->d_partcap;
    return a;
}

template <class T>
static rb_status launch_level(rb_plan *p, const LevelArgs<T> &a, int grid, hipStream_t s) {
    const size_t bytes = sizeof(T) * ((size_t)a.ring + 2 + kBlock);
    mark_start(p, s);
    k_level<T><<<grid, kWaves * 64, bytes, s>>>(a);
    RB_HIP(hipGetLastError());
    mark_end(p, s);
    return RB_OK;
}

// nc columns; sb: scratch in storage order (m per column), unless the storage
// order is the caller's and x does not overlap what is still to be read of b
template <class T>
static rb_status level_columns(rb_plan *p, const double *b, long ldb, double *x, long ldx,
                               int nc, double *sb, bool through, const int *left,
                               const int *done, hipStream_t s, bool add = true) {
    const LevelPlan *L = p->level;
    const int m = p->m;
    LevelArgs<T> a = level_args<T>(p);
    a.b = b;
    a.x = x;
    a.ldb = ldb;
    a.ldx = ldx;
    a.add = add;
    a.left = left;
    a.done = done;
    const dim3 pass(nblk(m), (nc + kPassCols - 1) / kPassCols);
    if (L->direct && through) {
        RB_HIP(hipMemcpy2DAsync(sb, sizeof(double) * m, b, sizeof(double) * ldb,
                                sizeof(double) * m, nc, hipMemcpyDeviceToDevice, s));
        a.b = sb;
        a.ldb = m;
    } else if (!L->direct) {
        k_level_in<<<pass, kT, 0, s>>>(b, ldb, L->d_row, m, nc, sb, left);
        RB_HIP(hipGetLastError());
        a.b = a.x = sb;
        a.ldb = a.ldx = m;
        a.add = false;
    }
    RB_TRY(launch_level<T>(p, a, a.nparts * nc, s));
    if (!L->direct) {
        if (sizeof(T) == 4 && add)
            k_level_out<true><<<pass, kT, 0, s>>>(x, ldx, L->d_row, m, nc, sb, left, done);
        else
            k_level_out<false><<<pass, kT, 0, s>>>(x, ldx, L->d_row, m, nc, sb, left, done);
        RB_HIP(hipGetLastError());
    }
    return RB_OK;
}

rb_status solve_level(rb_plan *p, const double *d_b, int ldb, double *d_x, int ldx, int nrhs,
                      hipStream_t s, double *ws, size_t ws_bytes) {
    const int m = p->m;
    if (m == 0) return RB_OK;
    const bool through = part_overlap(d_b, ldb, d_x, ldx, m, nrhs);
    if (p->level->direct && !through)
        return level_columns<double>(p, d_b, ldb, d_x, ldx, nrhs, nullptr, false, nullptr,
                                     nullptr, s);
    int cap = walk_cols(p);
    if (ws) cap = (int)std::min<size_t>(cap, ws_bytes / (sizeof(double) * (size_t)m));
    if (cap < 1) {
        set_error(RB_ERR_INVALID_ARG, "workspace too small for one column");
        return RB_ERR_INVALID_ARG;
    }
    ColumnGroups grp;
    RB_TRY(column_groups(d_b, ldb, d_x, ldx, m, nrhs, cap, &grp));
    if (!ws) RB_TRY(scratch_cols(p, std::min(cap, nrhs), s));
    for (int i = 0; i < grp.n; i++) {
        const int k = grp.at(i);
        RB_TRY(level_columns<double>(p, d_b + (size_t)k * ldb, ldb, d_x + (size_t)k * ldx, ldx,
                                     std::min(cap, nrhs - k), ws ? ws : p->d_bperm, through,
                                     nullptr, nullptr, s));
    }
    return RB_OK;
}

rb_status solve_level32(rb_plan *p, const double *d_r, int ldr, double *d_x, int ldx, int nc,
                        hipStream_t s, const int *left, const int *done, bool first) {
    if (p->m == 0) return RB_OK;
    // (r is the refinement's own: no overlap with x; nc is at most walk_cols)
    if (!p->level->direct) RB_TRY(scratch_cols(p, nc, s));
    return level_columns<float>(p, d_r, ldr, d_x, ldx, nc, p->d_bperm, false, left, done, s,
                                !first);
}

bool level_batches(const rb_plan *p) { return p->use_level && p->level->direct; }

void level_jobs(const rb_plan *p, const int *nrhs, std::vector<int> &out) {
    // Workgroups go round the 8 XCDs: a part's columns, which read the same
    // records, are put on one of them, parts with the most steps first.
    const LevelPlan *L = p->level;
    std::vector<int> order(L->nparts);
    for (int q = 0; q < L->nparts; q++) order[q] = q;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
        return L->parts[a].step1 - L->parts[a].step0 > L->parts[b].step1 - L->parts[b].step0;
    });
    std::vector<int> queue[8];
    long work[8] = {};
    for (int q : order) {
        const long steps = L->parts[q].step1 - L->parts[q].step0;
        if (steps == 0) continue;
        const int k = (int)(std::min_element(work, work + 8) - work);
        work[k] += steps * nrhs[q];
        for (int c = 0; c < nrhs[q]; c++) queue[k].push_back(c << 16 | q);
    }
    size_t len = 0;
    for (auto &k : queue) len = std::max(len, k.size());
    out.assign(8 * len, -1);
    for (int k = 0; k < 8; k++)
        for (size_t i = 0; i < queue[k].size(); i++) out[8 * i + k] = queue[k][i];
}

rb_status solve_level_batch(rb_plan *p, const double *const *d_b, double *const *d_x,
                            const int *d_ldb, const int *d_ldx, const int *d_job, int njobs,
                            hipStream_t s) {
    LevelArgs<double> a = level_args<double>(p);
    a.bp = d_b;
    a.xp = d_x;
    a.ldbp = d_ldb;
    a.ldxp = d_ldx;
    a.job = d_job;
    return launch_level<double>(p, a, njobs, s);
}

}  // namespace rb
