// Level-set analysis on the GPU that reproduces the reference's BFS
// *discovery order* exactly (R/findlevel.h:7-83, R/utils_cuda.h:29-97,
// where it runs on a single GPU thread).
//
// Order rule (the sequential algorithm restated): level 0 holds the rows
// with no off-diagonal entry, ascending.  A row v joins level k+1 when the
// last of its dependencies is visited; in the sequential walk that is its
// dependency u* with the largest level-order position, and v lands at the
// position sorted by (position of u*, offset of v inside column u*).
//
// Parallel form, one level per round inside one cooperative launch:
//   A  every frontier node u (position p) decrements rem[v] and raises
//      par[v] to p for every off-diagonal v in its column (atomics);
//   B  node u counts its children: v with rem[v] == 0 and par[v] == p;
//   S  exclusive scan of the counts in frontier order (grid-wide);
//   C  node u writes its children, in column order, at e + offset.
// A grid barrier separates the phases.
#include <hip/hip_cooperative_groups.h>

#include "rb_internal.h"

namespace cg = cooperative_groups;

namespace rb {

namespace {

// (256 and 1024 threads: 300,001 power-law rows backward 11.1 and 6.6 ms,
// 21,527 forward 1.8 and 1.2, 250,000 rows of a grid 5.6 and 5.5)
constexpr int kBfsThreads = 1024, kBfsWaves = kBfsThreads / 64;
constexpr int kScan = kBfsWaves + 2;  // ints of LDS for a scan

struct BfsCtl {
    int s, e;     // current frontier [s, e) of levelItem
    int nlevel;   // levels emitted so far
    int stalled;  // 1 when a round adds nothing while rows remain
};

// Exclusive scan of one value per thread across the block.  Returns the
// exclusive prefix; *total receives the block sum.  lds may be written again
// after the next barrier.
__device__ inline int block_excl_scan_open(int v, int *lds, int *total) {
    const int lane = threadIdx.x & 63;
    const int wid = threadIdx.x >> 6;
    int x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        int y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) lds[wid] = x;
    __syncthreads();
    // every wave scans the waves' sums for itself
    int w = lane < kBfsWaves ? lds[lane] : 0;
#pragma unroll
    for (int o = 1; o < kBfsWaves; o <<= 1) {
        int y = __shfl_up(w, o, 64);
        if (lane >= o) w += y;
    }
    *total = __shfl(w, kBfsWaves - 1, 64);
    return x - v + (wid > 0 ? __shfl(w, wid - 1, 64) : 0);
}
__device__ inline int block_excl_scan(int v, int *lds, int *total) {
    const int r = block_excl_scan_open(v, lds, total);
    __syncthreads();
    return r;
}

__device__ inline int ld_relaxed(const int *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// workgroup scope: while one workgroup walks narrow levels it is the only
// reader and writer of rem / par / levelItem (every other workgroup waits
// at the grid barrier, whose device-scope release / acquire publishes the
// walk's results and makes earlier writes visible to it)
__device__ inline int ld_wg(const int *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Grid-wide exclusive scan of cnt[0..len) in place (contiguous chunk per
// block).  Returns the grand total to every thread.  Uses two grid syncs.
__device__ int grid_excl_scan(cg::grid_group &g, int *cnt, int len,
                              int *blocksum, int *lds) {
    const int G = gridDim.x;
    const int chunk = (len + G - 1) / G;
    const int b0 = blockIdx.x * chunk;
    const int b1 = min(len, b0 + chunk);
    int local = 0;
    for (int i = b0 + threadIdx.x; i < b1; i += blockDim.x) local += cnt[i];
    int tot;
    (void)block_excl_scan(local, lds, &tot);
    if (threadIdx.x == 0) blocksum[blockIdx.x] = tot;
    g.sync();
    // every block scans the block sums redundantly (G is small)
    int before = 0, grand = 0;
    {
        int run = 0;
        for (int base = 0; base < G; base += blockDim.x) {
            int i = base + threadIdx.x;
            int v = i < G ? ld_relaxed(&blocksum[i]) : 0;
            int t;
            int ex = block_excl_scan(v, lds, &t);
            if (i == blockIdx.x) lds[kBfsWaves] = run + ex;
            run += t;
            __syncthreads();
        }
        before = lds[kBfsWaves];
        grand = run;
        __syncthreads();
    }
    int run = before;
    for (int base = b0; base < b1; base += blockDim.x) {
        int i = base + threadIdx.x;
        int v = i < b1 ? cnt[i] : 0;
        int t;
        int ex = block_excl_scan(v, lds, &t);
        if (i < b1) cnt[i] = run + ex;
        run += t;
    }
    g.sync();
    return grand;
}

constexpr int kNarrow = 4096;  // frontier size handled by one workgroup
constexpr int kIlp = 2;        // frontier nodes per thread, cached levels
constexpr int kE = 4;          // column entries per node kept in registers

// The phases over the entries [a, b) of a node's column (node u at position
// p).  Thread by thread, four entries in flight, or by a whole wave (with
// uniform arguments), 64 entries at a time, for a column of more than
// kLongCol entries: one thread alone needs two trips to memory for every four
// of them, and power-law factors have columns of thousands (300,001 rows
// backward: 47 ms with one thread and one entry at a time, 6.6 like this).
constexpr int kLongCol = 16;
constexpr int kWg = __HIP_MEMORY_SCOPE_WORKGROUP, kDev = __HIP_MEMORY_SCOPE_AGENT;
constexpr auto kCount = [](int, int) {};

template <int SC>
__device__ inline int ld_sc(const int *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, SC);
}

// A: decrement dependants, raise their parent position
template <int SC>
__device__ inline void release(int v, int *rem, int *par, int u, int p) {
    if (v == u) return;
    __hip_atomic_fetch_add(&rem[v], -1, __ATOMIC_RELAXED, SC);
    __hip_atomic_fetch_max(&par[v], p, __ATOMIC_RELAXED, SC);
}

// The children (rem 0, parent p), in column order: B counts them (put does
// nothing), C puts child v at o, o + 1, ...  Returns their number.
template <int SC, class Put>
__device__ inline int children(const int *__restrict__ rowidx, const int *rem, const int *par,
                               int a, int b, int u, int p, int o, Put put) {
    int c = 0;
    for (int q = a; q < b; q += 4) {
        int v[4], r[4], t[4];
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = q + j < b ? rowidx[q + j] : u;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            r[j] = ld_sc<SC>(&rem[v[j]]);
            t[j] = ld_sc<SC>(&par[v[j]]);
        }
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (v[j] != u && r[j] == 0 && t[j] == p) put(o + c++, v[j]);
    }
    return c;
}
template <int SC, class Put>
__device__ inline int wave_children(const int *__restrict__ rowidx, const int *rem,
                                    const int *par, int a, int b, int u, int p, int o, Put put) {
    const int lane = threadIdx.x & 63;
    int n = 0;
    for (int q = a; q < b; q += 64) {
        const int v = q + lane < b ? rowidx[q + lane] : u;
        const int r = ld_sc<SC>(&rem[v]), t = ld_sc<SC>(&par[v]);
        const bool kid = v != u && r == 0 && t == p;
        const unsigned long long kids = __ballot(kid);
        if (kid) put(o + n + __popcll(kids & ((1ull << lane) - 1)), v);
        n += __popcll(kids);
    }
    return n;
}

// The same for every lane's node at once (a == b: none), called by whole
// waves: short columns thread by thread, then the long ones one by one.
template <int SC>
__device__ inline void each_release(const int *__restrict__ rowidx, int *rem, int *par, int a,
                                    int b, int u, int p) {
    const bool wide = b - a > kLongCol;
    if (!wide)
        for (int q = a; q < b; q++) release<SC>(rowidx[q], rem, par, u, p);
    for (unsigned long long todo = __ballot(wide); todo; todo &= todo - 1) {
        const int l = __ffsll(todo) - 1;
        const int la = __shfl(a, l, 64), lb = __shfl(b, l, 64);
        const int lu = __shfl(u, l, 64), lp = __shfl(p, l, 64);
        for (int q = la + (threadIdx.x & 63); q < lb; q += 64)
            release<SC>(rowidx[q], rem, par, lu, lp);
    }
}
template <int SC, class Put>
__device__ inline int each_children(const int *__restrict__ rowidx, const int *rem,
                                    const int *par, int a, int b, int u, int p, int o, Put put) {
    const bool wide = b - a > kLongCol;
    int c = 0;
    if (!wide) c = children<SC>(rowidx, rem, par, a, b, u, p, o, put);
    for (unsigned long long todo = __ballot(wide); todo; todo &= todo - 1) {
        const int l = __ffsll(todo) - 1;
        const int n = wave_children<SC>(rowidx, rem, par, __shfl(a, l, 64), __shfl(b, l, 64),
                                        __shfl(u, l, 64), __shfl(p, l, 64), __shfl(o, l, 64),
                                        put);
        if ((int)(threadIdx.x & 63) == l) c = n;
    }
    return c;
}

// A level's frontier in LDS, left there by a cached level for the next when
// that is cached too: its nodes and their column ranges [a, b).
struct Front {
    int u[kIlp * kBfsThreads];
    int a[kIlp * kBfsThreads];
    int b[kIlp * kBfsThreads];
};
struct Walk {
    Front fr[2];
    int nlong;                        // nodes with long columns ...
    int node[kIlp * kBfsThreads];     // ... which they are
    int kids[kIlp * kBfsThreads];     // ... and their children: how many, then where
    int lds[kScan];
};

// One narrow level [s, e) of at most N * kBfsThreads nodes, N to a thread.
// Each thread keeps its nodes, their entry ranges and the first kE entries of
// their columns in registers from phase A to C, and phase B remembers which
// of those entries are children, so B reads only rem / par and C only writes.
// Entries past the first kE are re-read in each phase, by the thread or, in a
// long column, by the next wave that is free: the nodes with long columns are
// listed in LDS (the first levels of a power-law factor hold most of them).
// N is 1 where the level fits: places without a node still cost the loads of
// phase B (250 nodes a level, 256 threads: 7.3 us with six places, 5.6 with
// one).
template <int N>
__device__ int level_cached_n(const int *__restrict__ colptr, const int *__restrict__ rowidx,
                              int *rem, int *par, int *levelItem, int s, int e, Walk &w,
                              int &held) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, len = e - s;
    const bool in = held >= 0;  // this level's nodes and column ranges are in cur
    const int c0 = in ? held : 0;
    Front &cur = w.fr[c0], &fr = w.fr[c0 ^ 1];
    int u[N], q0[N], q1[N], vc[N][kE], at[N];
    unsigned kid[N];
#pragma unroll
    for (int k = 0; k < N; k++) {
        const int i = tid * N + k;
        u[k] = i >= len ? -1 : in ? cur.u[i] : ld_wg(&levelItem[s + i]);
    }
#pragma unroll
    for (int k = 0; k < N; k++) {
        const int i = tid * N + k;
        q0[k] = u[k] < 0 ? 0 : in ? cur.a[i] : colptr[u[k]];
        q1[k] = u[k] < 0 ? 0 : in ? cur.b[i] : colptr[u[k] + 1];
        if (!in && i < len) {
            cur.u[i] = u[k];
            cur.a[i] = q0[k];
            cur.b[i] = q1[k];
        }
    }
#pragma unroll
    for (int k = 0; k < N; k++)
#pragma unroll
        for (int j = 0; j < kE; j++)
            vc[k][j] = q0[k] + j < q1[k] ? rowidx[q0[k] + j] : -1;
    auto is_long = [&](int k) { return q1[k] - q0[k] > kLongCol; };
    // A: decrement dependants, raise their parent position
#pragma unroll
    for (int k = 0; k < N; k++) {
        const int p = s + tid * N + k;
#pragma unroll
        for (int j = 0; j < kE; j++)
            if (vc[k][j] >= 0) release<kWg>(vc[k][j], rem, par, u[k], p);
        if (is_long(k)) {
            at[k] = __hip_atomic_fetch_add(&w.nlong, 1, __ATOMIC_RELAXED, kWg);
            w.node[at[k]] = tid * N + k;
        } else {
            for (int q = q0[k] + kE; q < q1[k]; q++) release<kWg>(rowidx[q], rem, par, u[k], p);
        }
    }
    auto fence = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __syncthreads();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    };
    fence();
    const int nlong = w.nlong;
    if (nlong > 0) {
        for (int g = wave; g < nlong; g += kBfsWaves) {
            const int i = w.node[g], b = cur.b[i], uu = cur.u[i];
            for (int q = cur.a[i] + kE + lane; q < b; q += 64)
                release<kWg>(rowidx[q], rem, par, uu, s + i);
        }
        fence();
        if (tid == 0) w.nlong = 0;
        for (int g = wave; g < nlong; g += kBfsWaves) {
            const int i = w.node[g];
            const int n = wave_children<kWg>(rowidx, rem, par, cur.a[i] + kE, cur.b[i], cur.u[i],
                                             s + i, 0, kCount);
            if (lane == 0) w.kids[g] = n;
        }
        __syncthreads();
    }
    // B: children (rem 0, parent p) per node.  The cached entries' rem and
    // par are read together (a non-candidate reads row 0, in range, and is
    // ignored), and with them the entries' column ranges, which a child
    // takes into the next level's frontier in LDS.  A narrow level cost
    // about five dependent trips to memory (frontier, column pointers,
    // entries, atomics, rem / par) at ~2 us each on the 1500^2 Laplacian;
    // with the frontier in LDS three are left.  Reading rem / par entry by
    // entry behind branches cost another ~0.5 us.
    int rv[N][kE], pv[N][kE], ca[N][kE], cb[N][kE];
#pragma unroll
    for (int k = 0; k < N; k++)
#pragma unroll
        for (int j = 0; j < kE; j++) {
            const int v = vc[k][j];
            const int va = v >= 0 && v != u[k] ? v : 0;
            rv[k][j] = ld_wg(&rem[va]);
            pv[k][j] = ld_wg(&par[va]);
            ca[k][j] = colptr[va];
            cb[k][j] = colptr[va + 1];
        }
    int cnt[N], own = 0;
#pragma unroll
    for (int k = 0; k < N; k++) {
        const int p = s + tid * N + k;
        int c = 0;
        unsigned bits = 0;
#pragma unroll
        for (int j = 0; j < kE; j++) {
            const int v = vc[k][j];
            const bool cand = v >= 0 && v != u[k];
            if (cand && rv[k][j] == 0 && pv[k][j] == p) {
                c++;
                bits |= 1u << j;
            }
        }
        if (is_long(k)) c += w.kids[at[k]];
        else c += children<kWg>(rowidx, rem, par, q0[k] + kE, q1[k], u[k], p, 0, kCount);
        kid[k] = bits;
        cnt[k] = c;
        own += c;
    }
    int total;
    int o = e + block_excl_scan_open(own, w.lds, &total);
    // C: children in column order at the node's offset; when the next
    // level is cached too, its frontier also goes to the other fr
    const bool out = total <= kIlp * kBfsThreads;
    auto put = [&](int to, int v) {
        if (out) {
            fr.u[to - e] = v;
            fr.a[to - e] = colptr[v];
            fr.b[to - e] = colptr[v + 1];
        }
        __hip_atomic_store(&levelItem[to], v, __ATOMIC_RELAXED, kWg);
    };
#pragma unroll
    for (int k = 0; k < N; k++) {
        const int p = s + tid * N + k;
        int to = o;
#pragma unroll
        for (int j = 0; j < kE; j++)
            if ((kid[k] >> j) & 1u) {
                if (out) {
                    fr.u[to - e] = vc[k][j];
                    fr.a[to - e] = ca[k][j];
                    fr.b[to - e] = cb[k][j];
                }
                __hip_atomic_store(&levelItem[to++], vc[k][j], __ATOMIC_RELAXED, kWg);
            }
        if (is_long(k)) w.kids[at[k]] = to;
        else children<kWg>(rowidx, rem, par, q0[k] + kE, q1[k], u[k], p, to, put);
        o += cnt[k];
    }
    if (nlong > 0) {
        __syncthreads();
        for (int g = wave; g < nlong; g += kBfsWaves) {
            const int i = w.node[g];
            wave_children<kWg>(rowidx, rem, par, cur.a[i] + kE, cur.b[i], cur.u[i], s + i,
                               w.kids[g], put);
        }
    }
    held = out ? c0 ^ 1 : -1;
    return total;
}
__device__ int level_cached(const int *__restrict__ colptr, const int *__restrict__ rowidx,
                            int *rem, int *par, int *levelItem, int s, int e, Walk &w,
                            int &held) {
    static_assert(kIlp == 2);
    if (e - s <= kBfsThreads)
        return level_cached_n<1>(colptr, rowidx, rem, par, levelItem, s, e, w, held);
    return level_cached_n<2>(colptr, rowidx, rem, par, levelItem, s, e, w, held);
}

// One level [s, e) of any width inside one workgroup: the A / B / scan /
// C phases of the narrow levels, with the counts in device memory (cnt,
// indexed by frontier position) and a scan in chunks of the workgroup's
// width.  A thread handles the same positions in B and C, so it reads back
// only its own counts.
__device__ int level_wide(const int *__restrict__ colptr,
                          const int *__restrict__ rowidx, int *rem, int *par,
                          int *levelItem, int s, int e, int *cnt, int *lds) {
    const int tid = threadIdx.x;
    for (int base = s; base < e; base += blockDim.x) {  // uniform trip counts
        const int p = base + tid;
        const int u = p < e ? ld_wg(&levelItem[p]) : -1;
        each_release<kWg>(rowidx, rem, par, u >= 0 ? colptr[u] : 0, u >= 0 ? colptr[u + 1] : 0,
                         u, p);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    int carry = 0;
    for (int base = s; base < e; base += blockDim.x) {
        const int p = base + tid;
        const int u = p < e ? ld_wg(&levelItem[p]) : -1;
        const int c = each_children<kWg>(rowidx, rem, par, u >= 0 ? colptr[u] : 0,
                                    u >= 0 ? colptr[u + 1] : 0, u, p, 0, kCount);
        int tot = 0;
        const int off = block_excl_scan(c, lds, &tot);
        if (p < e) cnt[p] = carry + off;
        carry += tot;
    }
    for (int base = s; base < e; base += blockDim.x) {
        const int p = base + tid;
        const int u = p < e ? ld_wg(&levelItem[p]) : -1;
        each_children<kWg>(rowidx, rem, par, u >= 0 ? colptr[u] : 0, u >= 0 ? colptr[u + 1] : 0, u,
                      p, p < e ? e + cnt[p] : e, [&](int at, int v) {
                          __hip_atomic_store(&levelItem[at], v, __ATOMIC_RELAXED, kWg);
                      });
    }
    return carry;
}

// Consecutive narrow levels inside workgroup 0: the same A / B / scan / C
// phases, separated by workgroup barriers.  rem / par / levelItem are read,
// updated and written at workgroup scope (see ld_wg).
__device__ void bfs_narrow(const int *__restrict__ colptr,
                           const int *__restrict__ rowidx, int m, int *rem,
                           int *par, int *cnt, int *levelItem, int *levelPtr,
                           BfsCtl *ctl) {
    __shared__ Walk w;
    const int tid = threadIdx.x;
    if (tid == 0) w.nlong = 0;
    __syncthreads();
    int s = ld_relaxed(&ctl->s), e = ld_relaxed(&ctl->e);
    int nl = ld_relaxed(&ctl->nlevel);
    int stalled = 0;
    int held = -1;  // which of w.fr holds the level's frontier, -1: neither
    while (e < m && e - s <= kNarrow) {
        int total;
        if (e - s <= kIlp * kBfsThreads) {
            total = level_cached(colptr, rowidx, rem, par, levelItem, s, e, w, held);
        } else {
            total = level_wide(colptr, rowidx, rem, par, levelItem, s, e, cnt, w.lds);
            held = -1;
        }
        if (tid == 0) levelPtr[nl + 1] = e + total;
        nl++;
        s = e;
        e += total;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __syncthreads();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        if (total == 0) {
            stalled = 1;
            break;
        }
    }
    if (tid == 0) {
        ctl->s = s;
        ctl->e = e;
        ctl->nlevel = nl;
        if (stalled) ctl->stalled = 1;
    }
}

__global__ void __launch_bounds__(kBfsThreads)
k_bfs(const int *__restrict__ colptr, const int *__restrict__ rowidx, int m,
      int *rem, int *par, int *cnt, int *levelItem, int *levelPtr,
      int *blocksum, BfsCtl *ctl) {
    cg::grid_group g = cg::this_grid();
    __shared__ int lds[kScan];
    const int gtid = blockIdx.x * blockDim.x + threadIdx.x;
    const int gsz = gridDim.x * blockDim.x;

    // ---- level 0: rows without off-diagonal entries, ascending ----
    {
        const int G = gridDim.x;
        const int chunk = (m + G - 1) / G;
        const int b0 = blockIdx.x * chunk;
        const int b1 = min(m, b0 + chunk);
        for (int i = b0 + threadIdx.x; i < b1; i += blockDim.x)
            cnt[i] = rem[i] == 0 ? 1 : 0;
        g.sync();
        int total = grid_excl_scan(g, cnt, m, blocksum, lds);
        for (int i = b0 + threadIdx.x; i < b1; i += blockDim.x)
            if (rem[i] == 0) levelItem[cnt[i]] = i;
        if (gtid == 0) {
            levelPtr[0] = 0;
            levelPtr[1] = total;
            ctl->s = 0;
            ctl->e = total;
            ctl->nlevel = 1;
            ctl->stalled = (total == 0 && m > 0) ? 1 : 0;
        }
        g.sync();
    }

    while (true) {
        const int s = ld_relaxed(&ctl->s);
        const int e = ld_relaxed(&ctl->e);
        if (e >= m || ld_relaxed(&ctl->stalled)) break;
        const int len = e - s;
        if (len <= kNarrow) {
            // narrow frontier: workgroup 0 walks consecutive narrow levels
            // with workgroup barriers only; the rest wait at the grid sync
            if (blockIdx.x == 0)
                bfs_narrow(colptr, rowidx, m, rem, par, cnt, levelItem, levelPtr, ctl);
            g.sync();
            continue;
        }
        // A: decrement dependants, raise their parent position
        // (uniform trip counts in every phase: whole waves)
        for (int base = s + blockIdx.x * blockDim.x; base < e; base += gsz) {
            const int p = base + threadIdx.x;
            const int u = p < e ? levelItem[p] : -1;
            each_release<kDev>(rowidx, rem, par, u >= 0 ? colptr[u] : 0,
                              u >= 0 ? colptr[u + 1] : 0, u, p);
        }
        g.sync();
        // B: count the children each frontier node discovers
        {
            const int G = gridDim.x;
            const int chunk = (len + G - 1) / G;
            const int b0 = blockIdx.x * chunk;
            const int b1 = min(len, b0 + chunk);
            for (int base = b0; base < b1; base += blockDim.x) {
                const int i = base + threadIdx.x;
                const int u = i < b1 ? levelItem[s + i] : -1;
                const int c = each_children<kDev>(rowidx, rem, par, u >= 0 ? colptr[u] : 0,
                                             u >= 0 ? colptr[u + 1] : 0, u, s + i, 0, kCount);
                if (i < b1) cnt[i] = c;
            }
        }
        g.sync();
        const int total = grid_excl_scan(g, cnt, len, blocksum, lds);
        // C: emit children in column order
        for (int base = blockIdx.x * blockDim.x; base < len; base += gsz) {
            const int i = base + threadIdx.x;
            const int u = i < len ? levelItem[s + i] : -1;
            each_children<kDev>(rowidx, rem, par, u >= 0 ? colptr[u] : 0,
                           u >= 0 ? colptr[u + 1] : 0, u, s + i, i < len ? e + cnt[i] : e,
                           [&](int at, int v) { levelItem[at] = v; });
        }
        if (gtid == 0) {
            const int nl = ctl->nlevel;
            levelPtr[nl + 1] = e + total;
            ctl->nlevel = nl + 1;
            ctl->s = e;
            ctl->e = e + total;
            if (total == 0) ctl->stalled = 1;
        }
        g.sync();
    }
}

// The level analysis of every triangular block at once, one workgroup per
// block (blockIdx.x = t): the same discovery order as the whole-matrix
// walk (R/findlevel.h:7-83), restricted to the block's own entries.  The
// CSC holds the block-diagonal matrix (every row's in-block entries; row
// ids are permuted ids, block t owns [ups[t], ups[t] + bms[t])), so the
// blocks share no row and each workgroup reads and writes only its own
// rows: no grid barrier, only workgroup barriers.  Writes the block's rows
// in discovery order to item[ups[t] ..] (permuted ids), its level starts
// (block-local, level 0 at 0) to lvptr[lvbase[t] ..] and its level count
// to nlv[t]; a block that cannot finish (a row never released) sets
// *stalled.
__global__ void __launch_bounds__(kBfsThreads)
k_bfs_blocks(const int *__restrict__ colptr, const int *__restrict__ rowidx,
             const int *__restrict__ rowcnt, const int *__restrict__ ups,
             const int *__restrict__ bms, const int *__restrict__ lvbase,
             int *item, int *lvptr, int *nlv, int *rem, int *par, int *cnt,
             int *stalled) {
    __shared__ Walk w;
    const int t = blockIdx.x, tid = threadIdx.x;
    const int up = ups[t], bm = bms[t];
    int *lp = lvptr + lvbase[t];
    if (bm == 0) {
        if (tid == 0) {
            lp[0] = 0;
            nlv[t] = 0;
        }
        return;
    }
    int *it = item + up;
    if (tid == 0) w.nlong = 0;
    for (int i = tid; i < bm; i += blockDim.x) {
        rem[up + i] = rowcnt[up + i] - 1;
        par[up + i] = -1;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    // level 0: the rows without an in-block dependency, ascending
    int e = 0;
    for (int base = 0; base < bm; base += blockDim.x) {  // uniform trip count
        const int i = base + tid;
        const int f = i < bm && ld_wg(&rem[up + i]) == 0 ? 1 : 0;
        int tot = 0;
        const int off = block_excl_scan(f, w.lds, &tot);
        if (f)
            __hip_atomic_store(&it[e + off], up + i, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
        e += tot;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    if (tid == 0) {
        lp[0] = 0;
        lp[1] = e;
    }
    int s = 0, nl = 1;
    bool bad = e == 0;
    int held = -1;  // which of w.fr holds the level's frontier, -1: neither
    while (e < bm && !bad) {
        const int len = e - s;
        int total;
        if (len <= kIlp * kBfsThreads) {
            total = level_cached(colptr, rowidx, rem, par, it, s, e, w, held);
        } else {
            total = level_wide(colptr, rowidx, rem, par, it, s, e, cnt + up, w.lds);
            held = -1;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __syncthreads();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        if (total == 0) {
            bad = true;
            break;
        }
        if (tid == 0) lp[nl + 1] = e + total;
        nl++;
        s = e;
        e += total;
    }
    if (tid == 0) {
        nlv[t] = nl;
        if (bad) atomicOr(stalled, 1);
    }
}

__global__ void k_bfs_init(const int *__restrict__ rowcnt, int m, int *rem,
                           int *par) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < m) {
        rem[i] = rowcnt[i] - 1;
        par[i] = -1;
    }
}

}  // namespace

rb_status bfs_blocks(const int *d_colptr, const int *d_rowidx,
                     const int *d_rowcnt, int m, int nblocks, const int *d_ups,
                     const int *d_bms, const int *d_lvbase, int *d_item,
                     int *d_lvptr, int *d_nlv, hipStream_t s) {
    if (m == 0 || nblocks == 0) return RB_OK;
    Arena tmp(12 * (size_t)m + (1 << 20));  // rem, par, cnt and counters
    int *rem, *par, *cnt, *stalled;
    RB_TRY(tmp.alloc(&rem, m));
    RB_TRY(tmp.alloc(&par, m));
    RB_TRY(tmp.alloc(&cnt, m));
    RB_TRY(tmp.alloc(&stalled, 1));
    RB_HIP(hipMemsetAsync(stalled, 0, sizeof(int), s));
    k_bfs_blocks<<<nblocks, kBfsThreads, 0, s>>>(d_colptr, d_rowidx, d_rowcnt,
                                                 d_ups, d_bms, d_lvbase, d_item,
                                                 d_lvptr, d_nlv, rem, par, cnt,
                                                 stalled);
    RB_HIP(hipGetLastError());
    int h = 0;
    hipError_t e = hipMemcpyAsync(&h, stalled, sizeof(int), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    tmp.release();
    if (e != hipSuccess) return status_of_hip(e, "k_bfs_blocks");
    if (h) {
        set_error(RB_ERR_MISSING_DIAG,
                  "block level analysis stalled: a row is never released "
                  "(missing diagonal or cyclic dependency)");
        return RB_ERR_MISSING_DIAG;
    }
    return RB_OK;
}

rb_status bfs_levels(const int *d_colptr, const int *d_rowidx,
                     const int *d_rowcnt, int m, int *d_levelItem,
                     int *d_levelPtr, int *nlevel, hipStream_t s) {
    *nlevel = 0;
    if (m == 0) {
        int z = 0;
        RB_HIP(hipMemcpyAsync(d_levelPtr, &z, sizeof(int),
                              hipMemcpyHostToDevice, s));
        RB_HIP(hipStreamSynchronize(s));
        return RB_OK;
    }
    int dev = 0;
    RB_HIP(hipGetDevice(&dev));
    int ncu = 0;
    RB_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount,
                                 dev));
    int per_cu = 0;
    RB_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_bfs,
                                                        kBfsThreads, 0));
    if (per_cu < 1) per_cu = 1;
    int grid = ncu * (per_cu < 2 ? per_cu : 2);
    int need = (m + kBfsThreads - 1) / kBfsThreads;
    if (grid > need) grid = need;
    if (grid < 1) grid = 1;

    Arena tmp(12 * (size_t)m + (1 << 20));  // rem, par, cnt and counters
    int *rem, *par, *cnt, *blocksum;
    BfsCtl *ctl;
    RB_TRY(tmp.alloc(&rem, m));
    RB_TRY(tmp.alloc(&par, m));
    RB_TRY(tmp.alloc(&cnt, m));
    RB_TRY(tmp.alloc(&blocksum, grid));
    RB_TRY(tmp.alloc(&ctl, 1));
    k_bfs_init<<<(m + 255) / 256, 256, 0, s>>>(d_rowcnt, m, rem, par);
    RB_HIP(hipGetLastError());
    void *args[] = {(void *)&d_colptr, (void *)&d_rowidx, (void *)&m,
                    (void *)&rem,      (void *)&par,      (void *)&cnt,
                    (void *)&d_levelItem, (void *)&d_levelPtr,
                    (void *)&blocksum, (void *)&ctl};
    hipError_t e = hipLaunchCooperativeKernel((const void *)k_bfs, dim3(grid),
                                              dim3(kBfsThreads), args, 0, s);
    if (e != hipSuccess) {
        tmp.release();
        return status_of_hip(e, "hipLaunchCooperativeKernel(k_bfs)");
    }
    BfsCtl h;
    e = hipMemcpyAsync(&h, ctl, sizeof(h), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    tmp.release();
    if (e != hipSuccess) return status_of_hip(e, "k_bfs");
    if (h.stalled) {
        set_error(RB_ERR_MISSING_DIAG,
                  "level analysis stalled: a row is never released "
                  "(missing diagonal or cyclic dependency)");
        return RB_ERR_MISSING_DIAG;
    }
    *nlevel = h.nlevel;
    return RB_OK;
}

}  // namespace rb
