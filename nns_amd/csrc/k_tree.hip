// k_tree.hip -- tree construction, bottom-up summary and the traversal layout.
//
// Cells are prefixes of the 63-bit Morton key.  A cell at level L selects the
// slot of a body by key digit L (bits 62-3L .. 60-3L), so slot order is key
// order and the bodies of any cell are a contiguous range of the sorted keys.
// Single system: the root is node 0 with its slots at child[0..7] (the
// reference's convention, src/Kernels.cu:195,225) and cells take ids n, n+1, ...
// Ensemble: system s has the root cell N + s and cells follow from N + S.
//
// Construction is split along the MI355X memory hierarchy.  Each XCD has its
// own L2, so a fence or atomic at device scope costs a trip past L2; those are
// kept to a handful per subtree:
//   1. top cells -- cells holding more than kSubtreeMax bodies -- are found
//      from the sorted keys by searches (one thread per sample of
//      kSubtreeMax bodies) and wired with their child ranges;
//   2. every child range of a top cell with 2..kSubtreeMax bodies is a subtree
//      built by one workgroup from the shared-digit counts of neighbouring keys:
//      cell ids from a prefix sum, parents from searches over the keys in LDS, the
//      child slots filled in LDS and copied out (subtree_build_kernel).  Every subtree's
//      exact cell count is known first (from the shared-digit counts), and their
//      sums give each its block of cell ids: by a scan of its own, or up to kBuildScan
//      bodies summed by the build's workgroups.
//      The lock-based insertion (compare-and-swap on child slots, -2 = locked,
//      at workgroup scope; subtree_insert_kernel) builds the same cells when
//      nbx_params.build_locked is set;
//   3. the summary runs level by level: subtrees inside their workgroup, then
//      the top cells.  Every cell is summed by one thread over its
//      children in slot order, in FP64: results do not depend on scheduling.
#include "nbx_device.h"

#include <algorithm>

namespace nbx {

// Segments: one system ([0, n), root node 0) or an ensemble (off[], roots n + s).
struct Segs {
    const int32_t *off;       // nullptr: one segment [0, n)
    const int32_t *samp_off;  // nullptr: its samples start at 0
    int nseg, n;
    int batch;                // roots at n + s instead of node 0
};

__device__ inline int seg_lo(const Segs &g, int s) { return g.off ? g.off[s] : 0; }
__device__ inline int seg_hi(const Segs &g, int s) { return g.off ? g.off[s + 1] : g.n; }
__device__ inline int samp_lo(const Segs &g, int s) { return g.samp_off ? g.samp_off[s] : 0; }
__device__ inline int seg_root(const Segs &g, int s) { return g.batch ? g.n + s : 0; }
__device__ inline int seg_of_sample(const Segs &g, int k)
{
    if (!g.samp_off) return 0;
    int lo = 0, hi = g.nseg;  // last s with samp_off[s] <= k
    while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if (g.samp_off[mid] <= k) lo = mid; else hi = mid;
    }
    return lo;
}

__device__ inline uint64_t prefix_of(uint64_t key, int L) { return key >> (63 - 3 * L); }

// The run [a, b) of keys around position q of [lo, hi) that share its first L digits,
// both ends searched at once.
__device__ inline void prefix_run(const uint64_t *k, int lo, int q, int hi, int L, int &a, int &b)
{
    const uint64_t P = prefix_of(k[q], L);
    int la = lo, ha = q, lb = q + 1, hb = hi;
    while (la < ha || lb < hb) {
        const bool ua = la < ha, ub = lb < hb;
        const Quarter x = quarter_probes(la, ua ? ha : la), y = quarter_probes(ub ? lb : q, ub ? hb : q);
        uint64_t kx[3], ky[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            kx[i] = k[x.m[i]];
            ky[i] = k[y.m[i]];
        }
        if (ua) quarter_step(la, ha, x, prefix_of(kx[0], L) < P, prefix_of(kx[1], L) < P, prefix_of(kx[2], L) < P);
        if (ub) quarter_step(lb, hb, y, prefix_of(ky[0], L) <= P, prefix_of(ky[1], L) <= P, prefix_of(ky[2], L) <= P);
    }
    a = la;
    b = lb;
}
// First index in [lo, hi) whose digit L is >= d (all keys share the first L digits).
__device__ inline int lower_digit(const uint64_t *k, int lo, int hi, int d, int L)
{
    while (lo < hi) {
        const Quarter x = quarter_probes(lo, hi);
        const uint64_t k0 = k[x.m[0]], k1 = k[x.m[1]], k2 = k[x.m[2]];
        quarter_step(lo, hi, x, digit_at(k0, L) < d, digit_at(k1, L) < d, digit_at(k2, L) < d);
    }
    return lo;
}

// After the sort, in one launch: the top cells (the first `tb` workgroups), then lcp
// and the key-ordered bodies.
//
// Top cells: one lane per (sample q, level L); q is every kSubtreeMax-th sorted
// position of a segment.  The level-L cell through q is [a, b), found by a search
// over the segment; it is a top cell when it holds more than kSubtreeMax bodies, and
// q owns it when no earlier sample lies in it.  The levels of a sample are searched
// side by side, not one after another.  The table is level-major (entry
// L * nsamples + k), so the scan of its flags numbers the top cells level by level:
// the cells of level L are the ids base0 + [id[L * nsamples], id[(L + 1) * nsamples]).
//
// lcp[k]: the number of leading key digits shared by sorted keys k and k+1 (21 if
// equal).
//
// Bodies in key order as float4 (x, y, z, m) at nodes4[0..n), for the summary: read in
// input order and stored at their sorted positions pos[] (the sort's inverse
// permutation): random 16-byte reads each fetch a whole line, random 16-byte stores
// only dirty their bytes.
__global__ void __launch_bounds__(256) after_sort_kernel(Segs g, int nsamples, int tb,
                                                         const uint64_t *__restrict__ skeys,
                                                         uint32_t *__restrict__ flag, uint32_t *__restrict__ id,
                                                         int32_t *__restrict__ ta, int32_t *__restrict__ tend,
                                                         uint8_t *__restrict__ lcp, const int32_t *__restrict__ pos,
                                                         const float4 *__restrict__ bodies4,
                                                         float4 *__restrict__ nodes4, DeviceState *st)
{
    const int tid = threadIdx.x;
    if (blockIdx.x == 0 && tid == 0) {
        st->nsub = 0;
        st->ntop = 0;
    }
    if (latched(st)) return;
    if ((int)blockIdx.x < tb) {
        const int gt = blockIdx.x * 256 + tid;
        const int k = gt >> 5, L = gt & 31;
        if (k >= nsamples || L >= kLevels) return;
        const int e = L * nsamples + k;
        if (L == 0) {  // the root is wired separately
            flag[e] = id[e] = 0u;
            return;
        }
        const int s = seg_of_sample(g, k);
        const int lo = seg_lo(g, s), hi = seg_hi(g, s);
        const int q = lo + (k - samp_lo(g, s)) * kSubtreeMax;
        int a, b;
        prefix_run(skeys, lo, q, hi, L, a, b);
        const bool top = b - a > kSubtreeMax && (q - kSubtreeMax < a || q == lo);
        flag[e] = id[e] = top ? 1u : 0u;
        if (top) {
            ta[e] = a;
            tend[e] = b;
        }
        return;
    }
    const int stride = (int)(gridDim.x - tb) * 256;
    for (int k = (int)(blockIdx.x - tb) * 256 + tid; k < g.n; k += stride) {
        nodes4[pos[k]] = bodies4[k];
        if (k < g.n - 1) {
            const uint64_t x = (skeys[k] ^ skeys[k + 1]) & ~(1ull << 63);
            lcp[k] = x == 0 ? (uint8_t)kKeyLevels : (uint8_t)((62 - (63 - __clzll((long long)x))) / 3);
        }
    }
}

// Group order of the force walk.  The walk gives each wave 64 consecutive
// bodies of this order.  Key order has jumps (consecutive Morton keys can lie in
// cells far apart), so bodies are ordered by the top kGroupLevels Hilbert digits
// of their key instead, stably over key order (ties keep key order), each system
// by itself.  The order changes which bodies share a wave, never a body's
// interaction list.
//
// A cell's bodies are a range of this order too, and its children's ranges follow
// each other in the order of their Hilbert digits, so the order is read off the
// tree: in state s (a function of the cell's key digits) a child's range starts at its
// cell's plus the counts of the children with smaller digits (its offset), and a
// body's place is the sum of the offsets on its way up.  Below level kGroupLevels the
// digit is the slot (state kPlain).  The build leaves the offsets of the top cells and
// of the subtrees (top_wire_kernel, which has the child ranges in hand); here a
// workgroup takes a subtree: one thread per cell for the offsets of its children, then
// one per body for the sum.  No keys are made and nothing is sorted: the order takes
// 20 us at N = 2,000, 31 at 1M and 98 at 4M, where Hilbert keys and four radix passes (13
// launches) took 51, 138 and 245.  Placing the cells level by level instead took 34,
// 74 and 258 us: few of a level's lanes have a cell.
constexpr int kPlain = 12;

// Digit of each slot and state of each child, a nibble per slot, by state.
struct OrderTables {
    uint32_t dig[kPlain + 1], next[kPlain + 1];
};
__device__ inline void order_tables_fill(OrderTables &o)
{
    const int t = threadIdx.x;
    if (t <= kPlain) {
        uint32_t dig = 0, next = 0;
        for (int s = 0; s < 8; ++s) {
            dig |= (uint32_t)(t < kPlain ? c_hil[t][s] : s) << (4 * s);
            next |= (uint32_t)(t < kPlain ? c_dir[t][s] : kPlain) << (4 * s);
        }
        o.dig[t] = dig;
        o.next[t] = next;
    }
}
// State of the level-`to` cell of `key` from that of its level-`from` cell.
__device__ inline int order_state(const OrderTables &o, uint64_t key, int state, int from, int to)
{
    if (to >= kGroupLevels) return kPlain;
    for (int L = from; L < to; ++L) state = (int)(o.next[state] >> (4 * digit_at(key, L))) & 15;
    return state;
}

// Wires every top cell (and every root): child ranges by digit L; a range of
// one body is a leaf, of more than kSubtreeMax a top cell, otherwise a subtree
// queued for the subtree build.  Eight lanes per entry, lane d for digit d: each
// finds the end of its digit's range by one binary search over the cell's
// range and takes its start from the lane before (the searches run side by
// side, not one after another).  Thread 0 also sets *index past the top cells.
// Every child's place in the group order is left relative to its parent's: {offset,
// the parent's number among the top cells}, or {place, -1} under a root.
//
// SCAN: up to kWireScan entries, which every workgroup numbers for itself (workgroup 0
// also stores the numbers, id[]); otherwise id[] holds the scanned flags.  At 2,000
// and 32,768 bodies this adds 1.0 to 1.5 us and saves a launch of 4; at 150,001 (3,087
// entries) it added 3.6.
constexpr int kWireScan = 2048;
template <bool SCAN>
__global__ void __launch_bounds__(256) top_wire_kernel(
    Segs g, int nsamples, const uint64_t *__restrict__ skeys, const int32_t *__restrict__ perm, int *child,
    int32_t *__restrict__ cell_level, const uint32_t *__restrict__ flag, uint32_t *__restrict__ id,
    const int32_t *__restrict__ ta, const int32_t *__restrict__ tb, int4 *__restrict__ sub, int sub_max,
    int base0, int m, int *index, int *__restrict__ start, int2 *__restrict__ top_place,
    int2 *__restrict__ sub_place, DeviceState *st)
{
    __shared__ OrderTables tab;
    __shared__ uint32_t s_id[SCAN ? kWireScan : 1], s_sum[4];
    __shared__ int s_stop;
    order_tables_fill(tab);
    if (threadIdx.x == 0) s_stop = latched(st);  // one read: this launch raises the latch itself
    __syncthreads();
    if (s_stop) return;
    const int total = nsamples * kLevels;
    if (SCAN) {
        scan_to_lds<kWireScan / 1024>(flag, total, s_id, s_sum);
        if (blockIdx.x == 0)
            for (int k = threadIdx.x; k < total; k += 256) id[k] = s_id[k];
    }
    const auto number = [&](int e) { return (int)(SCAN ? s_id[e] : id[e]); };
    const int gt = blockIdx.x * blockDim.x + threadIdx.x;
    const int t = gt >> 3;  // entry: one (level, sample) of the top table, or one root
    const int d = gt & 7;   // digit, slot
    if (gt == 0) {
        const int ntop = number(total - 1) + (int)flag[total - 1];
        st->ntop = ntop;
        *index = base0 + ntop;
        if ((int64_t)base0 + ntop > m) atomicOr(&st->err, kErrCapacity);
    }
    int c, L, a, b, s;
    if (t < total) {
        if (!flag[t]) return;
        L = t / nsamples;
        const int k = t - L * nsamples;
        c = base0 + number(t);
        a = ta[t];
        b = tb[t];
        s = seg_of_sample(g, k);
        if (c >= m) return;  // capacity error latched by thread 0
        if (d == 0) {
            cell_level[c] = L;
            start[c] = a;
        }
        if (L == kKeyLevels) {  // more than kSubtreeMax bodies on one key
            if (d == 0) atomicOr(&st->err, kErrBucket);
            child[8 * (int64_t)c + d] = -1;
            return;
        }
    } else if (t < total + g.nseg) {
        s = t - total;
        c = seg_root(g, s);
        L = 0;
        a = seg_lo(g, s);
        b = seg_hi(g, s);
        if (g.batch && d == 0) start[c] = a;  // the single system's root is node 0, not a cell
    } else {
        return;
    }
    // the 8 lanes of an entry are consecutive lanes of one wave and all get here
    const int lo = seg_lo(g, s);
    const int db = lower_digit(skeys, a, b, d + 1, L);
    const int up = __shfl_up(db, 1, 8);
    const int da = d == 0 ? a : up;
    const int cnt = db - da;
    const uint32_t dig = tab.dig[order_state(tab, skeys[a], 0, 0, L)];
    int below = 0;
    for (int o = 0; o < 8; ++o) {
        const int w = __shfl(cnt, o, 8);
        below += ((int)(dig >> (4 * o)) & 7) < ((int)(dig >> (4 * d)) & 7) ? w : 0;
    }
    const int2 place = t < total ? make_int2(below, number(t)) : make_int2(a + below, -1);
    const int64_t slot = 8 * (int64_t)c + d;
    if (cnt == 0) {
        child[slot] = -1;
    } else if (cnt == 1) {
        child[slot] = perm[da];
    } else if (cnt > kSubtreeMax) {
        const int kk = samp_lo(g, s) + (da - lo + kSubtreeMax - 1) / kSubtreeMax;
        const int tc = number((L + 1) * nsamples + kk);
        child[slot] = base0 + tc;
        top_place[tc] = place;
    } else {
        child[slot] = -1;  // set by the subtree build
        const int i = atomicAdd(&st->nsub, 1);
        if (i < sub_max) {
            sub[i] = make_int4(da, db, L + 1, (int)slot);
            sub_place[i] = place;
        } else {
            atomicOr(&st->err, kErrCapacity);
        }
    }
}

// Cell ids of the subtrees.  A subtree [a, b) of sorted bodies with its root at
// level L0 has one cell per run of two or more bodies sharing L digits, L0 <= L
// <= 21; body a + i starts the runs of levels P_i < L <= l_i (l_i = lcp[a + i],
// P_i = l_{i-1}, P_0 = L0 - 1; the last body starts none), so the subtree has
//     (lcp[a] - L0 + 1) + sum over a < k < b - 1 of max(0, lcp[k] - lcp[k - 1])
// cells.  subtree_cells_kernel counts them, one wave per subtree (a job the
// builds reject counts 0); subtree_base_kernel turns the counts into the
// exclusive sum cbase[] (cbase[nsub] the total) and sets *index past the last
// subtree cell, so subtree j owns the ids from base0 + ntop + cbase[j] (after
// the top cells).  (Where the build sums the counts itself, cbase[] keeps them and the
// build does the rest.)  Each build workgroup reads or sums its base instead of taking it
// from one shared counter: the device-scope atomics of a shared counter are
// serialised, one per subtree.  A build that counts other than its subtree's number of
// cells latches kErrCapacity and leaves it unbuilt, so no two subtrees can share an id.
__global__ void __launch_bounds__(256) subtree_cells_kernel(const int4 *__restrict__ sub, int sub_max,
                                                            const uint8_t *__restrict__ lcp,
                                                            uint32_t *__restrict__ cbase, const DeviceState *st)
{
    if (latched(st)) return;
    const int nsub = min(__hip_atomic_load(&st->nsub, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), sub_max);
    const int lane = threadIdx.x & 63;
    const int waves = (int)(gridDim.x * blockDim.x) >> 6;
    for (int job = (int)(blockIdx.x * blockDim.x + threadIdx.x) >> 6; job < nsub; job += waves) {
        const int4 jb = sub[job];
        const int a = jb.x, cnt = jb.y - jb.x, L0 = jb.z;
        int c = 0;
        if (cnt >= 2 && cnt <= kSubtreeMax && L0 >= 1 && L0 <= kKeyLevels)
            for (int k = a + lane; k < a + cnt - 1; k += 64)
                c += k == a ? (int)lcp[a] - L0 + 1 : max(0, (int)lcp[k] - (int)lcp[k - 1]);
        for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
        if (lane == 0) cbase[job] = (uint32_t)c;
    }
}

__global__ void __launch_bounds__(1024) subtree_base_kernel(uint32_t *__restrict__ cbase, int sub_max, int base0,
                                                            int m, int *index, DeviceState *st)
{
    __shared__ uint32_t sh[16];
    if (latched(st)) return;
    const int nsub = min(__hip_atomic_load(&st->nsub, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), sub_max);
    const uint32_t carry = scan_in_place(cbase, nsub, sh);
    if (threadIdx.x == 0) {
        cbase[nsub] = carry;  // so that subtree j has cbase[j + 1] - cbase[j] cells for every j
        const int64_t end = (int64_t)base0 + st->ntop + carry;
        if (end > m) atomicOr(&st->err, kErrCapacity);
        else *index = (int)end;
    }
}

__device__ inline int ld_slot_wg(const int *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ inline void st_slot_wg(int *p, int v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ inline int cas_slot_wg(int *p, int expect, int desired)
{
    __hip_atomic_compare_exchange_strong(p, &expect, desired, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_WORKGROUP);
    return expect;
}

__device__ inline int block_max(int v, int *red)
{
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o));
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    int s = red[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) s = max(s, red[w]);
    __syncthreads();
    return s;
}

__device__ inline int block_sum(int v, int *red)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    int s = 0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s += red[w];
    __syncthreads();
    return s;
}

// Subtree build by insertion (nbx_params.build_locked = 1): persistent
// workgroups take subtrees from the queue.  Inside a
// subtree, the bodies are inserted by lock-based descent along their key digits
// (one body per thread per round, bodies strided over the range so that the
// lanes of a wave start in different branches):
//   cell (>= n)  descend;   -1  CAS -1 -> body;   -2  locked, retry next iteration;
//   body         CAS body -> -2 (lock); the winner creates the chain of cells down
//                to the first level where the two keys differ (a level-21 bucket if
//                they are equal), then publishes the first cell with a release store
//                (unlock).
// No lane waits inside an iteration on another lane, so a wave whose lanes
// contend for one slot always makes progress.  All atomics and fences are at
// workgroup scope: only this workgroup touches the subtree.
__global__ void __launch_bounds__(256) subtree_insert_kernel(
    int n, int m, const uint64_t *__restrict__ skeys, const int32_t *__restrict__ perm,
    const uint64_t *__restrict__ keys, const uint8_t *__restrict__ lcp, int *child, int base0,
    const uint32_t *__restrict__ cbase, int32_t *__restrict__ cell_level, int4 *__restrict__ sub, int sub_max,
    int4 *__restrict__ subcells, DeviceState *st)
{
    __shared__ int s_job, s_base, s_next, s_bad;
    __shared__ int red[4];
    const int tid = threadIdx.x;
    const int nsub = min(__hip_atomic_load(&st->nsub, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), sub_max);
    const int top = base0 + __hip_atomic_load(&st->ntop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    int next = blockIdx.x;  // workgroups stride over the jobs, like the summary's
    for (;;) {
        // Thread 0 alone reads the error latch (which other workgroups of this
        // launch may raise at any time) and names the job; every wave reads its
        // decision from LDS after the barrier, so the workgroup continues or
        // leaves as a whole.  A wave that left on its own read would let the
        // others pass the barrier and read an s_job nobody wrote.
        if (tid == 0) s_job = latched(st) ? nsub : next;
        next += gridDim.x;
        __syncthreads();
        const int job = s_job;
        __syncthreads();
        if (job >= nsub) break;
        const int4 jb = sub[job];
        const int a = jb.x, b = jb.y, L0 = jb.z, slot = jb.w;
        // exact cell count of the subtree from the common-prefix lengths
        int contrib = 0, deep = L0;
        for (int k = a + tid; k < b - 1; k += blockDim.x) {
            contrib += (k == a) ? (int)lcp[a] - L0 + 1 : max(0, (int)lcp[k] - (int)lcp[k - 1]);
            deep = max(deep, (int)lcp[k]);
        }
        const int ks = block_sum(contrib, red);
        const int Lmax = block_max(deep, red);
        if (tid == 0) {
            const int base = top + (int)cbase[job];  // ids reserved by subtree_base_kernel
            s_bad = (int64_t)base + ks > (int64_t)m || ks != (int)(cbase[job + 1] - cbase[job]);
            if (s_bad) atomicOr(&st->err, kErrCapacity);
            s_base = base;
            s_next = 1;
            if (!s_bad) {
                for (int d = 0; d < 8; ++d) child[8 * (int64_t)base + d] = -1;
                cell_level[base] = L0;
                child[slot] = base;
                subcells[job] = make_int4(base, ks, L0, Lmax);
            } else {
                subcells[job] = make_int4(0, 0, L0, L0 - 1);
            }
        }
        __syncthreads();
        if (s_bad) continue;
        const int base = s_base, root = base;
        const int count = b - a;
        const int rounds = (count + blockDim.x - 1) / blockDim.x;
        for (int r = 0; r < rounds; ++r) {
            const int off = r + tid * rounds;
            bool done = off >= count;
            const int p = a + off;
            const int body = done ? 0 : perm[p];
            const uint64_t key = done ? 0ull : skeys[p];
            int node = root, L = L0;
            while (__ballot(!done)) {
                if (done) continue;
                if (L == kKeyLevels) {
                    bool placed = false, full = true;
                    for (int s = 0; s < 8 && !placed; ++s) {
                        int ch = ld_slot_wg(&child[8 * (int64_t)node + s]);
                        if (ch == -1) {
                            full = false;
                            if (cas_slot_wg(&child[8 * (int64_t)node + s], -1, body) == -1) placed = true;
                        }
                    }
                    if (placed) {
                        done = true;
                    } else if (full) {
                        atomicOr(&st->err, kErrBucket);
                        done = true;
                    }
                    continue;
                }
                const int64_t addr = 8 * (int64_t)node + digit_at(key, L);
                const int ch = ld_slot_wg(&child[addr]);
                if (ch >= n) {
                    node = ch;
                    ++L;
                } else if (ch == -1) {
                    if (cas_slot_wg(&child[addr], -1, body) == -1) done = true;
                } else if (ch >= 0) {
                    if (cas_slot_wg(&child[addr], ch, -2) == ch) {
                        const uint64_t key2 = keys[ch];
                        int ld = L + 1;
                        while (ld < kKeyLevels && digit_at(key, ld) == digit_at(key2, ld)) ++ld;
                        const int need = ld - L;  // cells at levels L+1 .. ld
                        const int old = atomicAdd(&s_next, need);
                        if (old + need > ks) {
                            atomicOr(&st->err, kErrCapacity);
                            st_slot_wg(&child[addr], ch);
                            done = true;
                            continue;
                        }
                        const int first = base + old;
                        const int4 neg = make_int4(-1, -1, -1, -1);
                        for (int j = 0; j < need; ++j) {
                            const int c = first + j;
                            const int lvl = L + 1 + j;
                            int4 *c4 = reinterpret_cast<int4 *>(child + 8 * (int64_t)c);
                            c4[0] = neg;
                            c4[1] = neg;
                            cell_level[c] = lvl;
                            if (lvl < ld) {
                                child[8 * (int64_t)c + digit_at(key, lvl)] = c + 1;
                            } else if (ld < kKeyLevels) {
                                child[8 * (int64_t)c + digit_at(key2, ld)] = ch;
                                child[8 * (int64_t)c + digit_at(key, ld)] = body;
                            } else {
                                child[8 * (int64_t)c + 0] = ch;  // bucket; index order restored in the summary
                                child[8 * (int64_t)c + 1] = body;
                            }
                        }
                        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
                        st_slot_wg(&child[addr], first);  // publish + unlock
                        done = true;
                    }
                }
            }
        }
        __syncthreads();
    }
}

// Subtree build, without locks or atomics on child slots.  One workgroup builds one
// subtree [a, b) of sorted bodies whose root is at level L0 (a child range of
// a top cell, 2..kSubtreeMax bodies).  With l[i] the number of key digits that
// local bodies i and i+1 share (l[cnt-1] = L0 - 1 at the subtree's edge) and
// P_i = l[i-1] (P_0 = L0 - 1), the cells of the subtree are the runs of two or
// more bodies that share L digits, L = L0..21, and body i starts exactly the
// cells of levels P_i < L <= l[i].  Numbering cells by first body, then level,
//     id(i, L) = base + cs[i] + (L - P_i - 1),   cs = exclusive sum of max(0, l[i] - P_i),
// gives every cell its id from one prefix sum (base from subtree_base_kernel).
// The parent of cell (i, L), L > L0, is (i, L-1) when L-1 > P_i; otherwise the
// level-P_i cell that holds bodies i-1 and i, which starts at the first body s_i
// that shares P_i digits with body i, found by a search over the keys in LDS.  The
// deepest cell of body i is (i, l[i]) when l[i] > P_i, else the same (s_i, P_i).
// A child takes the slot of its key digit at the parent's level; in a level-21
// bucket (equal keys) the bodies take slots 0, 1, ... in sorted order, which is
// ascending index order.  Each slot thus has exactly one writer: every cell and body
// stores itself into its parent's slot in LDS, and the slots go out in one
// contiguous store per cell.  Every id and slot is range-checked before its store.
//
// Latency bounds it: a chain of loads, a scan, a search and stores per subtree.  So
// a thread has at most four bodies (one wave with up to sixteen, a table of
// range minima for s_i and the slots stored to memory twice, empty and filled:
// 2,000 bodies 22 us, now 10; 150,000: 36 and 13.5; 1M:
// 48 and 30; 4M: 104 and 88), and, as in the summary, the subtrees of a launch are those that fit its
// POOL of slots and not one of BELOW bytes; with REST also those that fit none,
// whose slots are stored to memory directly.
constexpr int kBuildSmall = 12672, kBuildSmallT = 128;  // 12 workgroups of 128 threads share a CU
constexpr int kBuildPool = 26752;                       // six of 256; 1,024 bodies with 515 cells
__host__ __device__ constexpr int build_bytes(int ks, int nb) { return 32 * ks + 10 * nb + 32; }
// Workgroups stride over the jobs.  With about one job each at N = 4M (16,400
// subtrees), the dispatcher starts a new workgroup wherever one has finished,
// which balances subtrees of 2 to 1024 bodies better than a few jobs per
// resident workgroup (with one wave each, 0.141 ms with 4096 workgroups, 0.103 ms
// with 16384).
constexpr int kBuildBlocks = 16384;

__device__ inline int shared_digits(uint64_t a, uint64_t b)  // of two keys, 21 if equal
{
    const uint64_t x = (a ^ b) & ~(1ull << 63);
    return x == 0 ? kKeyLevels : (__clzll((long long)x) - 1) / 3;
}

template <int T, int POOL, int BELOW, bool SCAN>
__global__ void __launch_bounds__(T, 6) subtree_build_kernel(
    int m, const uint64_t *__restrict__ skeys, const int32_t *__restrict__ perm, int *__restrict__ child, int base0,
    const uint32_t *__restrict__ cbase, int32_t *__restrict__ cell_level, int *__restrict__ start,
    const int4 *__restrict__ sub, int sub_max, int4 *__restrict__ subcells, int *__restrict__ index, DeviceState *st)
{
    constexpr bool REST = POOL == kBuildPool;
    constexpr int C = 4, W = T / 64;  // bodies per thread at most; waves
    static_assert(!REST || (C * T >= kSubtreeMax && build_bytes(0, kSubtreeMax) <= POOL), "the keys fit without the slots");
    __shared__ int s_stop, s_cnt[C][W], s_deep[W], s_sum[W];
    __shared__ __align__(16) unsigned char s_pool[POOL];
    if (threadIdx.x == 0) s_stop = latched(st);  // one read: this launch raises the latch itself
    __syncthreads();
    if (s_stop) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nsub = min(__hip_atomic_load(&st->nsub, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), sub_max);
    const int top = base0 + __hip_atomic_load(&st->ntop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // SCAN: the cells of the subtrees [from, to), summed by the workgroup from the counts
    const auto cells_of = [&](int from, int to) {
        int c = 0;
        for (int j = from + tid; j < to; j += T) c += (int)cbase[j];
        for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
        if (lane == 0) s_sum[wave] = c;
        __syncthreads();
        c = 0;
        for (int w = 0; w < W; ++w) c += s_sum[w];
        __syncthreads();
        return c;
    };
    if (SCAN && blockIdx.x == 0) {
        const int64_t end = (int64_t)top + cells_of(0, nsub);
        if (tid == 0) {
            if (end > m) atomicOr(&st->err, kErrCapacity);
            else *index = (int)end;
        }
    }
    // SCAN: the cells before a job, kept from job to job, so that a workgroup reads every count once
    uint32_t before = SCAN && (int)blockIdx.x < nsub ? (uint32_t)cells_of(0, blockIdx.x) : 0u;
    const auto next_of = [&](int job) {
        const int next = job + (int)gridDim.x;
        if (SCAN && next < nsub) before += (uint32_t)cells_of(job, next);
        return next;
    };
    for (int job = blockIdx.x; job < nsub; job = next_of(job)) {
        const int4 jb = sub[job];
        const uint32_t cb0 = SCAN ? before : cbase[job], cb1 = SCAN ? cb0 + cbase[job] : cbase[job + 1];
        const int base = top + (int)cb0, ks = (int)(cb1 - cb0);  // the subtree's own ids
        const int a = jb.x, cnt = jb.y - jb.x, L0 = jb.z, slot = jb.w;
        const bool fits = ks >= 0 && ks < 65536 && cnt <= C * T && build_bytes(ks, cnt) <= POOL;
        if (fits ? BELOW > 0 && cnt <= 4 * kBuildSmallT && build_bytes(ks, cnt) <= BELOW : !REST) continue;
        if (cnt < 2 || cnt > kSubtreeMax || L0 < 1 || L0 > kKeyLevels || ks < 1 || ks > 65535 ||
            (int64_t)base + ks > (int64_t)m) {
            if (tid == 0) {
                atomicOr(&st->err, kErrCapacity);
                subcells[job] = make_int4(0, 0, L0, L0 - 1);
            }
            continue;
        }
        uint64_t *key = (uint64_t *)s_pool;
        int *cslots = (int *)(s_pool + ((10 * cnt + 15) & ~15));
        uint16_t *cs = (uint16_t *)(key + cnt);  // cs[i] (ids relative to base)
        int *gslots = child + 8 * (int64_t)base;
        uint64_t kq[C];
        int pq[C];
#pragma unroll
        for (int q = 0; q < C; ++q) {
            const int i = tid + T * q;
            if (i >= cnt) break;
            kq[q] = skeys[a + i];
            pq[q] = perm[a + i];
        }
        const int4 none = make_int4(-1, -1, -1, -1);
        for (int k = tid; k < 2 * ks; k += T) (fits ? (int4 *)cslots : (int4 *)gslots)[k] = none;
#pragma unroll
        for (int q = 0; q < C; ++q)
            if (tid + T * q < cnt) key[tid + T * q] = kq[q];
        if (!fits) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __syncthreads();
        int l[C], P[C], run[C], deep = L0;
#pragma unroll
        for (int q = 0; q < C; ++q) {
            const int i = tid + T * q;
            l[q] = i < cnt - 1 ? shared_digits(kq[q], key[i + 1]) : L0 - 1;
            P[q] = i > 0 && i < cnt ? shared_digits(key[i - 1], kq[q]) : L0 - 1;
            run[q] = i < cnt ? max(0, l[q] - P[q]) : 0;
            deep = max(deep, l[q]);
        }
#pragma unroll
        for (int q = 0; q < C; ++q) {
            const int own = run[q];
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(run[q], o);
                if (lane >= o) run[q] += y;
            }
            if (lane == 63) s_cnt[q][wave] = run[q];
            run[q] -= own;
        }
        for (int o = 32; o > 0; o >>= 1) deep = max(deep, __shfl_xor(deep, o));
        if (lane == 0) s_deep[wave] = deep;
        __syncthreads();
        int total = 0;
#pragma unroll
        for (int q = 0; q < C; ++q)
#pragma unroll
            for (int w = 0; w < W; ++w) {
                if (w == wave) run[q] += total;
                total += s_cnt[q][w];
            }
        for (int w = 0; w < W; ++w) deep = max(deep, s_deep[w]);
#pragma unroll
        for (int q = 0; q < C; ++q)
            if (tid + T * q < cnt) cs[tid + T * q] = (uint16_t)run[q];
        __syncthreads();
        if (total != ks) {  // uniform: the counts of subtree_cells_kernel do not hold
            if (tid == 0) {
                atomicOr(&st->err, kErrCapacity);
                subcells[job] = make_int4(0, 0, L0, L0 - 1);
            }
            __syncthreads();
            continue;
        }
        // every cell (but the root) and every body into its parent's slot
        bool bad = false;
        const auto put = [&](int par, int d, int v) {
            if (par < 0 || par >= ks || d >= 8) bad = true;
            else if (fits) cslots[8 * par + d] = v;
            else gslots[8 * (int64_t)par + d] = v;
        };
#pragma unroll
        for (int q = 0; q < C; ++q) {
            const int i = tid + T * q;
            if (i >= cnt) break;
            const int own = run[q] - P[q] - 1;  // id(i, L) - base = own + L
            int s = 0, up = 0;                  // start of the level-P run through i >= 1, its id - base
            if (i >= 1) {
                const uint64_t want = prefix_of(kq[q], P[q]);
                int hi = i - 1;
                while (s < hi) {
                    const Quarter z = quarter_probes(s, hi);
                    const uint64_t k0 = key[z.m[0]], k1 = key[z.m[1]], k2 = key[z.m[2]];
                    quarter_step(s, hi, z, prefix_of(k0, P[q]) < want, prefix_of(k1, P[q]) < want,
                                 prefix_of(k2, P[q]) < want);
                }
                const int Ps = s == 0 ? L0 - 1 : shared_digits(key[s - 1], key[s]);
                up = (int)cs[s] - Ps - 1 + P[q];
            }
            for (int L = P[q] + 1; L <= l[q]; ++L) {
                const int c = own + L;
                if (c < 0 || c >= ks) { bad = true; break; }
                cell_level[base + c] = L;
                start[base + c] = a + i;
                if (L > L0) put(L - 1 > P[q] ? c - 1 : up, digit_at(kq[q], L - 1), base + c);
            }
            const int D = max(P[q], l[q]);
            put(l[q] > P[q] ? own + l[q] : up, D < kKeyLevels ? digit_at(kq[q], D) : l[q] > P[q] ? 0 : i - s, pq[q]);
        }
        if (bad) atomicOr(&st->err, kErrBucket);
        if (tid == 0) {
            child[slot] = base;
            subcells[job] = make_int4(base, ks, L0, deep);
        }
        __syncthreads();
        if (fits)
            for (int k = tid; k < 2 * ks; k += T) ((int4 *)gslots)[k] = ((const int4 *)cslots)[k];
        __syncthreads();  // the next job overwrites the pool
    }
}

// ------------------------------------------------------------------ summary
struct CellSum {
    double ms, mx, my, mz;
    int cnt, first;
};

// The slots v[] of the level-21 bucket c in ascending index order, the stable key order.
__device__ inline void order_bucket(int *child, int c, int *v)
{
    for (int i = 1; i < 8; ++i) {
        int a = v[i], j = i - 1;
        while (j >= 0 && (v[j] == -1 || (a != -1 && v[j] > a))) { v[j + 1] = v[j]; --j; }
        v[j + 1] = a;
    }
    for (int s = 0; s < 8; ++s) child[8 * (int64_t)c + s] = v[s];
}

// Sums the children of c in slot order; a level-21 bucket first puts its
// bodies (equal keys) in ascending index order, the stable key order.  The
// children of a cell in slot order are consecutive ranges of the sorted
// bodies, so with the cell's first sorted position known (first >= 0) a body
// child is read from the sorted copy at a running cursor; otherwise (first < 0)
// from its own index, with its sorted position from pos[].
// The slots go in batches of B (a divisor of 8): per batch (1) the cell
// children's sums, counts and (without a cursor) first bodies, every load
// issued before the first use (a slot without a cell loads node 0, unused),
// (2) the body children at the cursor (the cell's first body plus the sizes of
// the slots before them), (3) the sums in slot order, in FP64.  B = 2 for the
// subtrees (more would cost occupancy: 4 needs 90 registers against 59), 4 for
// the top cells.  CURSOR: the build has given every cell its first sorted body
// (first >= 0), which the summary then neither reads for the children nor
// stores again.
template <int B, bool CURSOR>
__device__ inline CellSum sum_cell(int c, int first, bool bucket, int n, int *child, const float4 *bodies4,
                                   const float4 *sorted4, const int32_t *pos, const double4 *sum64,
                                   const int *count, const int *start)
{
    int v[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) v[s] = child[8 * (int64_t)c + s];
    if (bucket) order_bucket(child, c, v);
    CellSum r{0.0, 0.0, 0.0, 0.0, 0, 0x7fffffff};
    int cur = first;
#pragma unroll
    for (int s0 = 0; s0 < 8; s0 += B) {
        double cm[B], cx[B], cy[B], cz[B];
        int kc[B], kf[B], bp[B];
        float4 b[B];
#pragma unroll
        for (int t = 0; t < B; ++t) {
            const int64_t q = v[s0 + t] >= n ? v[s0 + t] : 0;
            const double4 cs = sum64[q];  // one 32-byte record: mass and the three moments
            cm[t] = cs.x;
            cx[t] = cs.y;
            cy[t] = cs.z;
            cz[t] = cs.w;
            kc[t] = count[q];
            kf[t] = CURSOR ? 0 : start[q];
        }
#pragma unroll
        for (int t = 0; t < B; ++t) {
            const int ch = v[s0 + t];
            bp[t] = cur;
            if (cur >= 0) cur += ch == -1 ? 0 : (ch < n ? 1 : kc[t]);
        }
#pragma unroll
        for (int t = 0; t < B; ++t) {
            const int ch = v[s0 + t];
            const bool body = ch >= 0 && ch < n;
            const int p = bp[t];
            const float4 *a = body && p >= 0 && p < n ? sorted4 + p : bodies4 + (body ? ch : 0);
            b[t] = *a;
        }
#pragma unroll
        for (int t = 0; t < B; ++t) {
            const int ch = v[s0 + t];
            if (ch == -1) continue;
            if (ch < n) {
                const double mb = (double)b[t].w;
                r.ms = __dadd_rn(r.ms, mb);
                r.mx = __dadd_rn(r.mx, __dmul_rn(mb, (double)b[t].x));
                r.my = __dadd_rn(r.my, __dmul_rn(mb, (double)b[t].y));
                r.mz = __dadd_rn(r.mz, __dmul_rn(mb, (double)b[t].z));
                r.cnt += 1;
                if (!CURSOR) r.first = min(r.first, bp[t] >= 0 ? bp[t] : pos[ch]);
            } else {
                r.ms = __dadd_rn(r.ms, cm[t]);
                r.mx = __dadd_rn(r.mx, cx[t]);
                r.my = __dadd_rn(r.my, cy[t]);
                r.mz = __dadd_rn(r.mz, cz[t]);
                r.cnt += kc[t];
                if (!CURSOR) r.first = min(r.first, kf[t]);
            }
        }
    }
    return r;
}

struct SumOut {
    int n;
    int *child;
    const float4 *bodies4;   // bodies (x, y, z, m) by index
    float *mass;             // cells written (single system)
    float *cx, *cy, *cz;     // cell centre of mass (single system; nullptr for the ensemble)
    int *count, *start;      // start: set by the build for every cell when `cursor`
    const int32_t *pos, *cell_level;
    double4 *sum64;          // FP64 cell sums {mass, moments x, y, z} (written)
    float4 *nodes4;          // bodies in key order at [0, n) (read), cells at [n, m) (written)
    int cursor;              // cell starts known before the summary
};

__device__ inline void store_cell(const SumOut &o, int c, const CellSum &r, DeviceState *st)
{
    if (r.cnt > 0 && !(r.ms > 0.0)) atomicOr(&st->err, kErrNonFinite);
    const float fx = (float)(r.mx / r.ms), fy = (float)(r.my / r.ms), fz = (float)(r.mz / r.ms), fm = (float)r.ms;
    o.sum64[c] = make_double4(r.ms, r.mx, r.my, r.mz);
    if (o.cx) {
        o.cx[c] = fx; o.cy[c] = fy; o.cz[c] = fz; o.mass[c] = fm;
    }
    o.count[c] = r.cnt;
    if (!o.cursor) o.start[c] = r.first;
    o.nodes4[c] = make_float4(fx, fy, fz, fm);
}

// The single system's root, from its mass and moments.
__device__ inline void store_root(double ms, double mx, double my, double mz, int cnt, DeviceState *st)
{
    if (cnt > 0 && !(ms > 0.0)) atomicOr(&st->err, kErrNonFinite);
    const double gx = mx / ms, gy = my / ms, gz = mz / ms;
    st->root64[0] = ms; st->root64[1] = gx; st->root64[2] = gy; st->root64[3] = gz;
    st->root4 = make_float4((float)gx, (float)gy, (float)gz, (float)ms);
}

// lev: the cell's level when the caller has it (else -1).
// B: slots whose loads go together; CURSOR: o.cursor (sum_cell).
template <int B, bool CURSOR>
__device__ inline void summarise(const SumOut &o, int c, DeviceState *st, bool single_root, int root_first = 0,
                                 int lev = -1)
{
    const bool bucket = !single_root && (lev >= 0 ? lev : o.cell_level[c]) == kKeyLevels;
    const int first = !CURSOR ? -1 : single_root ? root_first : o.start[c];
    const CellSum r = sum_cell<B, CURSOR>(c, first, bucket, o.n, o.child, o.bodies4, o.nodes4, o.pos, o.sum64,
                                          o.count, o.start);
    if (!single_root) {
        store_cell(o, c, r, st);
        return;
    }
    store_root(r.ms, r.mx, r.my, r.mz, r.cnt, st);
}

// Subtree summary: workgroup w sums subtrees w, w + gridDim.x, ...: with as many
// workgroups as subtrees, about, the dispatcher hands each free slot of a CU
// the next workgroup, a job queue with no shared counter.  The cells of a
// subtree are the contiguous ids [base, base + ks), its bodies the sorted range
// [a, a + nb), and a cell waits for the level below it: a chain of up to 20 steps
// that sets the time at every size (a subtree has 5 to 15 levels of few cells).  So
// the subtree first comes into LDS, every load issued before the first wait, and its
// cells are listed by level; the levels then run from the deepest up on LDS alone,
// four lanes per cell, one for each of its four sums; and the centres, the divisions
// and every store follow at the end, all cells side by side.  A cell's record holds
// its slots until it is summed, then its sums.  (Sums and bodies read from memory and
// results stored level by level: 2,000 bodies 32 us, now 11; 150,000: 43 and
// 17; 1M: 86 and 43; 4M: 311 and 141.)
//
// What a subtree needs of LDS varies (a mean of 9 KB, at most some 43), and the
// subtrees a CU holds at once are what hides their chains.  A launch takes those that
// fit its POOL and, with BELOW > 0, do not fit a pool of BELOW bytes; with REST, the
// subtrees that fit no pool too, which are summed in memory.
constexpr int kSumSmall = 9920, kSumSmallT = 128;  // 16 workgroups of 128 threads share a CU
constexpr int kSumPool = 40672;                    // four of 256; 1,024 bodies with 620 cells
constexpr int kSumCells = 3;                       // cells a thread stages at most, and four bodies
constexpr int kSubSumBatch = 2;
__device__ inline bool sum_fits(int ks, int nb, int threads, int pool)
{
    return 39 * ks + 16 * nb + 72 <= pool && ks <= kSumCells * threads && nb <= 4 * threads;
}

template <bool CURSOR, int T, int POOL, int BELOW>
__global__ void __launch_bounds__(T, POOL == kSumSmall ? 8 : 4) subtree_summary_kernel(
    SumOut o, const int4 *__restrict__ sub, int sub_max, const int4 *__restrict__ subcells, DeviceState *st)
{
    constexpr bool REST = POOL == kSumPool;
    static_assert(!REST || kSubtreeMax <= 4 * T, "a thread stages four bodies");
    __shared__ int s_stop, s_hist[kLevels], s_from[kLevels + 1];
    __shared__ __align__(32) unsigned char s_pool[POOL];
    const int tid = threadIdx.x;
    const int nsub = min(__hip_atomic_load(&st->nsub, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), sub_max);
    for (int job = blockIdx.x; job < nsub; job += gridDim.x) {
        const int4 sc = subcells[job], jb = sub[job];
        const int base = sc.x, ks = sc.y, L0 = sc.z, a = jb.x, nb = jb.y - jb.x;
        const bool fits = sum_fits(ks, nb, T, POOL);
        if (fits ? BELOW > 0 && sum_fits(ks, nb, kSumSmallT, BELOW) : !REST) continue;
        // One read of the latch per job, by thread 0, published to the workgroup,
        // which continues or leaves as a whole (a zero cell mass raises the latch
        // from inside this launch).
        if (tid == 0) s_stop = latched(st);
        if (tid < kLevels) s_hist[tid] = 0;
        __syncthreads();
        if (s_stop) break;
        if (!fits) {
            for (int L = sc.w; L >= L0; --L) {
                for (int k = tid; k < ks; k += blockDim.x)
                    if (o.cell_level[base + k] == L) summarise<kSubSumBatch, CURSOR>(o, base + k, st, false, 0, L);
                __syncthreads();
            }
            continue;
        }
        // Slots in LDS, 16 bits each, the empty ones left out: a cell's number in the
        // subtree; `none` after the last; and for a body `one`, or with no cursor
        // 0x8000 | its position.  The entries `one` and `none` of cnt[] hold 1 and 0.
        const uint32_t one = ks, none = ks + 1;
        double4 *rec = (double4 *)s_pool;
        float4 *body = (float4 *)(rec + ks + 2);
        uint16_t *cnt = (uint16_t *)(body + nb), *first = cnt + ks + 2, *list = first + ks;
        uint8_t *lev = (uint8_t *)(list + ks);
        float4 bv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (tid + T * u < nb) bv[u] = o.nodes4[a + tid + T * u];
#pragma unroll
        for (int u = 0; u < kSumCells; ++u) {
            const int k = tid + T * u;
            if (k >= ks) break;
            const int4 *c4 = (const int4 *)(o.child + 8 * ((int64_t)base + k));
            const int4 va = c4[0], vb = c4[1];
            const int lv = o.cell_level[base + k], fv = CURSOR ? o.start[base + k] - a : 0;
            int v[8] = {va.x, va.y, va.z, va.w, vb.x, vb.y, vb.z, vb.w};
            if (!CURSOR && lv == kKeyLevels) order_bucket(o.child, base + k, v);
            uint64_t lo = none * 0x0001000100010001ull, hi = lo;
#pragma unroll
            for (int t = 7; t >= 0; --t) {
                const int ch = v[t];
                const bool isb = ch >= 0 && ch < o.n, in = isb || (ch > base && ch - base < ks);
                const uint64_t w = !isb ? (uint32_t)(ch - base)
                                        : CURSOR ? one : 0x8000u | ((uint32_t)(o.pos[ch] - a) & 0x3ffu);
                hi = in ? hi << 16 | lo >> 48 : hi;
                lo = in ? lo << 16 | w : lo;
            }
            *(ulonglong2 *)&rec[k] = make_ulonglong2(lo, hi);
            lev[k] = (uint8_t)lv;
            first[k] = (uint16_t)fv;
            cnt[k] = (uint16_t)atomicAdd(&s_hist[lv], 1);  // for now, its number in its level
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (tid + T * u < nb) body[tid + T * u] = bv[u];
        if (tid < 2) {
            rec[ks + tid] = make_double4(0.0, 0.0, 0.0, 0.0);
            cnt[ks + tid] = tid == 0;
        }
        __syncthreads();
        if (tid < 64) {
            int x = tid < kLevels ? s_hist[tid] : 0;
            for (int d = 1; d < 32; d <<= 1) {
                const int y = __shfl_up(x, d);
                if (tid >= d) x += y;
            }
            if (tid < kLevels) s_from[tid + 1] = x;
            if (tid == 0) s_from[0] = 0;
        }
        __syncthreads();
        for (int k = tid; k < ks; k += T) list[s_from[lev[k]] + cnt[k]] = (uint16_t)k;
        __syncthreads();
        const int q = tid & 3;  // this lane's sum: mass, moments x, y, z
        for (int L = sc.w; L >= L0; --L) {
            const int to = s_from[L + 1];
            for (int i = s_from[L] + (tid >> 2); i < to; i += T / 4) {
                const int k = list[i];
                const ulonglong2 slots = *(const ulonglong2 *)&rec[k];
                int at_first = nb, all = CURSOR ? (int)first[k] : 0;
                const int f0 = all;
                double sum = 0.0;
                for (int half = 0; half < 2; ++half) {
                    const uint64_t wq = half ? slots.y : slots.x;
                    if ((uint32_t)(wq & 0xffffu) == none) break;
                    bool isb[4];
                    int at[4];  // a child's first body
                    double cs[4];
                    float bm[4], br[4];
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const uint32_t w = (uint32_t)(wq >> (16 * t)) & 0xffffu;
                        isb[t] = CURSOR ? w == one : w >= 0x8000u;
                        const uint32_t c = !CURSOR && isb[t] ? one : w;
                        const int kc = cnt[c];
                        cs[t] = ((const double *)rec)[4 * c + q];
                        if (CURSOR) {
                            at[t] = all;
                        } else {
                            at[t] = isb[t] ? (int)(w & 0x3ffu) : c < one ? (int)first[c] : nb;
                            at_first = min(at_first, at[t]);
                        }
                        all += kc;
                    }
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const int e = min(at[t], nb - 1);
                        bm[t] = body[e].w;
                        br[t] = ((const float *)body)[4 * e + ((q + 3) & 3)];  // the mass itself for lane 0
                    }
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const float r = q ? br[t] : 1.0f;
                        const double v = __dmul_rn((double)bm[t], (double)r);
                        sum = __dadd_rn(sum, isb[t] ? v : cs[t]);
                    }
                }
                ((double *)rec)[4 * k + q] = sum;
                if (q == 0) {
                    cnt[k] = (uint16_t)(all - f0);
                    if (!CURSOR) first[k] = (uint16_t)at_first;
                }
            }
            __syncthreads();
        }
        for (int k = tid; k < ks; k += T) {
            const double4 r = rec[k];
            store_cell(o, base + k, CellSum{r.x, r.y, r.z, r.w, (int)cnt[k], a + (int)first[k]}, st);
        }
        __syncthreads();  // the next job overwrites the pool
    }
}

// Top summary: the top cells level by level, deepest first, then the roots.  A
// level's cells read only the levels below.  A cell's sum gathers from up to 8
// children in unrelated cache lines, and one CU's address pipeline takes such
// gathers a few lanes at a time, so while more are left than fit there,
// the levels are spread over kTopBlocks workgroups (a level's cell i to workgroup i mod
// kTopBlocks) that meet at a grid barrier after each (top_levels_kernel); the rest is
// summed by one workgroup alone, in LDS (top_summary_kernel).
// The workgroups of a grid barrier must all be on the device at once.  Those of
// top_levels_kernel hold no LDS to speak of and 256 threads, so 64 fit any partition of an MI355X
// (32 CUs at least) twice over, beside other kernels and launches of their own kind; the
// LDS part, whose workgroup takes a CU for itself, is a launch of its own (a step of 1M
// bodies 2,022 us, with both in one launch 2,014).  The wait is bounded all the same: one that
// runs out latches kErrStall, and every wave still finishes.
constexpr int kTopBlocks = 64, kTopLevelThreads = 256;
// Up to kTopOneGroup bodies there are hardly ever many more top cells than fit, and
// one workgroup sums them all; up to kTopFew bodies in a third of the LDS.  Workgroups that
// need most of a CU's LDS hold up the kernels of other streams: three ensembles of 96
// systems (100,000 bodies) side by side took 1.6 % longer a step with one of 145 KB
// and as long as before with one of 52 KB.
constexpr int kTopOneGroup = 1 << 19;
constexpr int kTopSmall = 160, kTopLarge = 448, kTopFew = 1 << 17;
constexpr int kTopSpin = 1 << 20;  // polls of one barrier wait (about a second)
// Top cells that the LDS part takes with room for `items`; the others leave some to the roots.
constexpr int top_lds_cells(int items) { return items * 7 / 8; }

// Grid barrier number `phase` (1, 2, ...) of the launch.  Every wave waits until its
// stores have reached the XCD's L2; thread 0 then makes them visible device-wide with its
// arrival (one write-back of the L2, not one per wave), waits until every workgroup has
// arrived, and acquires what they wrote for the whole CU.
__device__ inline void top_barrier(DeviceState *st, int phase, bool &stalled)
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        const int target = phase * (int)gridDim.x;
        __hip_atomic_fetch_add(&st->tsync, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        for (int k = 0; !stalled && __hip_atomic_load(&st->tsync, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target;
             ++k) {
            if (k == kTopSpin) {
                atomicOr(&st->err, kErrStall);
                stalled = true;  // no further waits in this workgroup
            }
            __builtin_amdgcn_s_sleep(2);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    __syncthreads();
}

// Few top cells and roots (items): all in the LDS of one workgroup.  The sums of
// every item's children have their places there: those of subtrees and bodies are loaded up
// front, all side by side, and an item that is summed puts its own into its parent's.
// Eight lanes per item, of which four add one component each, in slot order.
// (Level by level in memory, with four times as many write-backs of the L2 at a barrier:
// 150,001 bodies 23 us, now 11; with the levels before it 1M: 49, now 12 + 16; 4M: 48, now
// 23 + 14; 7.5M in 512 systems: 100, now 61 + 20.)
constexpr int kTopThreads = 512;
template <int ITEMS>
struct TopLds {
    double4 slot[8 * ITEMS];  // sums of the children
    double4 rec[ITEMS];       // sums of the items
    int cnt[8 * ITEMS];       // bodies of the children; slot 0 then the item's
    int place[ITEMS];         // an item's place among its parent's children
};
template <bool CURSOR, int ITEMS>
__device__ inline void top_in_lds(TopLds<ITEMS> &t, int *first, const SumOut &o, const Segs &g, int base0, int left,
                                  int roots, const int *first_of_level, int from,
                                  DeviceState *st)
{
    const int tid = threadIdx.x, s = tid & 7, items = left + roots;
    const auto node_of = [&](int j) { return j < left ? base0 + j : seg_root(g, j - left); };
    for (int j = tid; j < left; j += kTopThreads) t.place[j] = -1;  // below a root that is not an item
    __syncthreads();
    for (int k0 = tid; k0 < 8 * items; k0 += 4 * kTopThreads) {
        int q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int k = k0 + u * kTopThreads;
            q[u] = k < 8 * items ? o.child[8 * (int64_t)node_of(k >> 3) + s] : -1;
        }
        double4 v[4];
        int c[4], f[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            v[u] = make_double4(0.0, 0.0, 0.0, 0.0);
            c[u] = 0;
            f[u] = 0x7fffffff;
            if (q[u] >= o.n && (q[u] < base0 || q[u] >= base0 + left)) {
                v[u] = o.sum64[q[u]];
                c[u] = o.count[q[u]];
                if (!CURSOR) f[u] = o.start[q[u]];
            } else if (q[u] >= 0 && q[u] < o.n) {
                const float4 b = o.bodies4[q[u]];
                const double m = (double)b.w;
                v[u] = make_double4(m, __dmul_rn(m, (double)b.x), __dmul_rn(m, (double)b.y), __dmul_rn(m, (double)b.z));
                c[u] = 1;
                if (!CURSOR) f[u] = o.pos[q[u]];
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int k = k0 + u * kTopThreads;
            if (k >= 8 * items) break;
            if (q[u] >= base0 && q[u] < base0 + left) t.place[q[u] - base0] = k;
            t.slot[k] = v[u];
            t.cnt[k] = c[u];
            if (!CURSOR) first[k] = f[u];
        }
    }
    __syncthreads();
    for (int L = from; L >= 0; --L) {
        const int a = L ? first_of_level[L] : left, b = L ? first_of_level[L + 1] : items;
        if (a >= b) continue;
        for (int j = a + (tid >> 3); j < b; j += kTopThreads / 8) {
            int n1 = t.cnt[8 * j + s], lo = CURSOR ? 0 : first[8 * j + s];
            for (int d = 1; d < 8; d <<= 1) {
                n1 += __shfl_xor(n1, d, 8);
                if (!CURSOR) lo = min(lo, __shfl_xor(lo, d, 8));
            }
            double sum = 0.0;
#pragma unroll
            for (int k = 0; k < 8; ++k) sum = __dadd_rn(sum, ((const double *)&t.slot[8 * j + k])[s & 3]);
            const int up = j < left ? t.place[j] : -1;
            if (s < 4) {
                ((double *)&t.rec[j])[s] = sum;
                if (up >= 0) ((double *)&t.slot[up])[s] = sum;
            } else if (s == 4) {
                t.cnt[8 * j] = n1;  // this item's lanes have read it
                if (up >= 0) t.cnt[up] = n1;
                if (!CURSOR) {
                    first[8 * j] = lo;
                    if (up >= 0) first[up] = lo;
                }
            }
        }
        __syncthreads();
    }
    for (int j = tid; j < items; j += kTopThreads) {
        const double4 r = t.rec[j];
        if (j < left || g.batch)
            store_cell(o, node_of(j), CellSum{r.x, r.y, r.z, r.w, t.cnt[8 * j], CURSOR ? 0 : first[8 * j]}, st);
        else
            store_root(r.x, r.y, r.z, r.w, t.cnt[8 * j], st);
    }
}

// The top cells of level L are the ids base0 + [first[L], first[L + 1]) (the scanned,
// level-major top table).  Called by the whole workgroup; ends with a barrier.
__device__ inline void top_levels(int *first, const uint32_t *top_id, int nsamples, const DeviceState *st)
{
    const int tid = threadIdx.x;
    if (tid <= kLevels)
        first[tid] = tid < kLevels ? (int)top_id[tid * nsamples]
                                   : __hip_atomic_load(&st->ntop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
}

// The levels below those that the LDS part takes with room for kTopLarge items.
template <bool CURSOR>
__global__ void __launch_bounds__(kTopLevelThreads) top_levels_kernel(SumOut o, int base0, int nsamples,
                                                                      const uint32_t *__restrict__ top_id,
                                                                      DeviceState *st)
{
    __shared__ int s_first[kLevels + 1];
    __shared__ int s_stop;
    const int tid = threadIdx.x;
    if (tid == 0) s_stop = latched(st);  // one read for the whole workgroup
    top_levels(s_first, top_id, nsamples, st);
    // Latched before this launch: every workgroup reads it so and skips the sums,
    // but still meets every barrier (a latch raised by this launch's own sums may
    // be seen by some workgroups only).
    const bool stop = s_stop != 0;
    bool stalled = false;
    int phase = 0;
    for (int L = kKeyLevels; L >= 1 && s_first[L + 1] > top_lds_cells(kTopLarge); --L) {
        const int cnt = s_first[L + 1] - s_first[L];
        if (cnt <= 0) continue;  // uniform: no barrier for an empty level
        if (!stop)
            for (int i = blockIdx.x + gridDim.x * tid; i < cnt; i += gridDim.x * blockDim.x)
                summarise<4, CURSOR>(o, base0 + s_first[L] + i, st, false, 0, L);
        top_barrier(st, ++phase, stalled);
    }
    if (phase == 0) return;
    if (tid == 0) {  // the last workgroup out (every other one is past its last wait) resets the barrier
        const int out = __hip_atomic_fetch_add(&st->tdone, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        if (out == (int)gridDim.x - 1) {
            __hip_atomic_store(&st->tsync, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(&st->tdone, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// One workgroup.  WIDE: also the levels below those that fit (without a launch of
// top_levels_kernel before).
template <bool CURSOR, int ITEMS, bool WIDE>
__global__ void __launch_bounds__(kTopThreads) top_summary_kernel(SumOut o, Segs g, int base0, int nsamples,
                                                          const uint32_t *__restrict__ top_id, DeviceState *st)
{
    static_assert(WIDE || ITEMS == kTopLarge, "top_levels_kernel leaves off at kTopLarge");
    __shared__ int s_first[kLevels + 1];
    __shared__ int s_stop;
    __shared__ TopLds<ITEMS> s_top;
    __shared__ int s_low[CURSOR ? 1 : 8 * ITEMS];
    const int tid = threadIdx.x;
    if (tid == 0) s_stop = latched(st);  // one read for the whole workgroup
    top_levels(s_first, top_id, nsamples, st);
    if (s_stop) return;
    int L = kKeyLevels;
    for (; L >= 1 && s_first[L + 1] > top_lds_cells(ITEMS); --L) {
        if (!WIDE) continue;
        for (int i = s_first[L] + tid; i < s_first[L + 1]; i += kTopThreads)
            summarise<4, CURSOR>(o, base0 + i, st, false, 0, L);
        __syncthreads();
    }
    const int left = s_first[L + 1];
    const bool roots = left + g.nseg <= ITEMS;
    top_in_lds<CURSOR>(s_top, s_low, o, g, base0, left, roots ? g.nseg : 0, s_first, L, st);
    __syncthreads();
    if (!roots)  // every top cell is summed
        for (int s = tid; s < g.nseg; s += kTopThreads) summarise<4, CURSOR>(o, seg_root(g, s), st, !g.batch);
}

// ------------------------------------------------------------------ layout
// Frame blocks.  Block b lists the non-empty children of one cell, compacted in
// slot order, as the records [off(b), off(b) + k_b) of the packed arrays:
// fnode[off(b) + k] = (x, y, z, m) of the child and fmeta[off(b) + k] its
// descriptor {tag, crit}:
//   body:  tag = sorted position << 4,        crit = -1 (always accepted);
//   cell:  tag = off(block) << 4 | children (1-8), crit = crit_L + eps^2,
// crit_L = (l_L/theta)^2 computed as in the opening test (crit_0 rounded once
// from FP64, scaled by 4^-L exactly) and eps^2 added once in FP32, so the walk
// compares crit < |d|^2 + eps^2 -- the value its interaction needs anyway.
// A cell child is described by the bottom of its chain, the first descendant
// with two or more children: the cells of a one-child chain carry the same mass
// and centre of mass (the FP64 sums of a single child are exact copies), and
// crit_L + eps^2 falls with L, so a body accepts some cell of the chain exactly
// when it accepts the bottom one, and meets the same monopole once either way.  fnode
// keeps the data of the child itself (walk_record).
// Single system: block 0 is the root (slots child[0..7]), block i >= 1 is cell
// n + i - 1.  Ensemble: block i is cell n + i, the roots being blocks 0..S-1.
// froot4 / frootm describe each root as a child of a virtual parent.  The
// parent blocks of every block and of every body (by sorted position) go to
// pblk / bpar for the adjoint's top-down pass.
// Blocks follow in id order with no gaps between them, so off(b) is the number
// of children of the blocks before b: the packed records take 24 bytes per node
// (fnode and fmeta) where blocks of eight slots took 192 bytes per cell, and a
// frame's three block loads come from fewer distinct lines of the L2.
template <bool BATCH>
__device__ inline int block_of(int c, int n)
{
    return BATCH ? c - n : (c == 0 ? 0 : c - n + 1);
}

// Children per block, summed within each run of kOffRun blocks: boff[b] = the
// children of the blocks of b's run before b, bsum[run] = the run's total (the
// runs are then scanned in place).  One workgroup per run.  The slots are read
// as 16-byte halves of the blocks' rows, consecutive threads on consecutive
// halves, and the two halves of a block meet by a lane exchange.
template <bool BATCH>
__global__ void __launch_bounds__(256) frame_count_kernel(int n, const int *__restrict__ index,
                                                          const int *__restrict__ child, uint32_t *__restrict__ boff,
                                                          uint32_t *__restrict__ bsum, const DeviceState *st)
{
    __shared__ uint32_t cnt[kOffRun];
    __shared__ uint32_t sh[4];
    static_assert(kOffRun == 4 * 256, "four blocks per thread");
    if (latched(st)) return;
    const int64_t items = BATCH ? (int64_t)*index - n : (int64_t)*index - n + 1;
    const int64_t r0 = (int64_t)blockIdx.x * kOffRun;
    if (r0 >= items) {  // uniform: a run past the last block
        if (threadIdx.x == 0) bsum[blockIdx.x] = 0u;
        return;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int h = (int)threadIdx.x + 256 * u;  // half h & 1 of the run's block h >> 1
        const int64_t item = r0 + (h >> 1);
        int k = 0;
        if (item < items) {
            const int node = BATCH ? n + (int)item : (item == 0 ? 0 : n + (int)item - 1);
            const int4 q = reinterpret_cast<const int4 *>(child + 8 * (int64_t)node)[h & 1];
            k = (q.x != -1) + (q.y != -1) + (q.z != -1) + (q.w != -1);
        }
        k += __shfl_xor(k, 1);
        if ((h & 1) == 0) cnt[h >> 1] = (uint32_t)k;
    }
    __syncthreads();
    const int j0 = 4 * (int)threadIdx.x;
    uint32_t k[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) k[u] = cnt[j0 + u];
    uint32_t tot;
    uint32_t ex = block_exclusive_scan(k[0] + k[1] + k[2] + k[3], sh, &tot);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        if (r0 + j0 + u < items) boff[r0 + j0 + u] = ex;
        ex += k[u];
    }
    if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

// Opening threshold of a level-L cell as the walk compares it: crit_L + eps^2,
// crit_L = (l_L/theta)^2, l_0 the side of the root cell of the key grid.
__device__ inline float crit_of(double span, float theta, float eps2, int lev)
{
    const double lc0 = ldexp(span / kMaskCoord, kKeyLevels);
    const double r0 = lc0 / (double)theta;
    return ldexpf((float)(r0 * r0), -2 * lev) + eps2;
}

// Descriptor of the bottom of the one-child chain starting at cell c (c = 0 is
// the single-system root).
template <bool BATCH>
__device__ inline int2 chain_bottom(int c, int n, const int *__restrict__ child,
                                    const int32_t *__restrict__ cell_level, bool root, double span, float theta,
                                    float eps2, const uint32_t *__restrict__ boff, const uint32_t *__restrict__ bsum)
{
    for (;;) {
        const int4 *p = reinterpret_cast<const int4 *>(child + 8 * (int64_t)c);
        const int4 a = p[0], b = p[1];
        const int v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        int cnt = 0, last = -1;
        for (int s = 0; s < 8; ++s)
            if (v[s] != -1) { ++cnt; last = v[s]; }
        if (cnt == 1 && last >= n) {
            c = last;
            root = false;
            continue;
        }
        const int lev = root ? 0 : cell_level[c];
        const int off = frame_off(boff, bsum, block_of<BATCH>(c, n));
        return make_int2((off << 4) | cnt, __float_as_int(crit_of(span, theta, eps2, lev)));
    }
}

// chain_bottom of a cell child whose slots (a, b) and level are already loaded:
// the loads of a chain are made only when the child has a single cell child.
template <bool BATCH>
__device__ inline int2 chain_bottom_from(int c, int4 a, int4 b, int lev, int n, const int *__restrict__ child,
                                         const int32_t *__restrict__ cell_level, double span, float theta,
                                         float eps2, const uint32_t *__restrict__ boff,
                                         const uint32_t *__restrict__ bsum)
{
    for (;;) {
        const int v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        int cnt = 0, last = -1;
        for (int s = 0; s < 8; ++s)
            if (v[s] != -1) { ++cnt; last = v[s]; }
        if (cnt == 1 && last >= n) {
            c = last;
            const int4 *p = reinterpret_cast<const int4 *>(child + 8 * (int64_t)c);
            a = p[0];
            b = p[1];
            lev = cell_level[c];
            continue;
        }
        const int off = frame_off(boff, bsum, block_of<BATCH>(c, n));
        return make_int2((off << 4) | cnt, __float_as_int(crit_of(span, theta, eps2, lev)));
    }
}

// A cell's record for the walk, its centre of mass brought into FP32's range (masses that nearly
// cancel can put it past that).  Its monopole is then 0 at every body, d^2 being infinite, and 0
// times the distance stays 0 on all of the wave's lanes, also those that do not meet the cell.
__device__ inline float4 walk_record(const float4 q)
{
    constexpr float M = 3.402823466e38f;
    return make_float4(fminf(fmaxf(q.x, -M), M), fminf(fmaxf(q.y, -M), M), fminf(fmaxf(q.z, -M), M), q.w);
}

// Ensemble: the system of a cell from its first sorted position (sorting leaves every
// system's bodies in the system's own positions, so sys_of holds for both orders).
struct SysInfo {
    const int32_t *sys_of;
    const float *theta;
    const double *ext;
};

// SCAN: up to kLayoutRuns runs, whose totals (brun) every workgroup scans for itself
// (workgroup 0 also stores the sums, bsum[]); otherwise bsum[] holds the scanned totals.
// 0.6 us more at 2,000 and 32,768 bodies for a launch of 3.7; 2.4 more at 150,001.
constexpr int kLayoutRuns = 96;
template <bool BATCH, bool SCAN>
__global__ void __launch_bounds__(256) frame_layout_kernel(
    int n, int nroot, const int *__restrict__ index, const int *__restrict__ child, const int32_t *__restrict__ pos,
    const int32_t *__restrict__ cell_level, const int *__restrict__ count, const int *__restrict__ start,
    const float4 *__restrict__ nodes4, float4 *__restrict__ fnode, int2 *__restrict__ fmeta,
    const uint32_t *__restrict__ boff, const uint32_t *__restrict__ brun, int runs, uint32_t *gsum,
    float4 *__restrict__ froot4, int2 *__restrict__ frootm, int32_t *__restrict__ pblk, int32_t *__restrict__ bpar,
    float theta, float eps2, SysInfo si, const DeviceState *st)
{
    __shared__ uint32_t s_run[SCAN ? kLayoutRuns : 1], s_sum[4];
    if (latched(st)) return;  // one value for the whole launch: nothing in it raises the latch
    if (SCAN) {
        scan_to_lds<1>(brun, runs, s_run, s_sum);
        if (blockIdx.x == 0)
            for (int k = threadIdx.x; k < runs; k += 256) gsum[k] = s_run[k];
    }
    const uint32_t *bsum = SCAN ? s_run : gsum;
    const int ncell = *index - n;
    const int64_t items = BATCH ? ncell : ncell + 1;
    const int64_t total = 8 * items;
    const int64_t bound = (total + 63) & ~(int64_t)63;  // whole waves iterate together (ballot below)
    const int lane = threadIdx.x & 63;
    const int body_crit = __float_as_int(-1.f);
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < bound;
         k += (int64_t)blockDim.x * gridDim.x) {
        const int64_t item = k >> 3;
        const int s = (int)(k & 7);
        const int node = BATCH ? n + (int)item : (item == 0 ? 0 : n + (int)item - 1);
        const int ch = k < total ? child[8 * (int64_t)node + s] : -1;
        // Everything a cell child needs (its slots, level, count and centre) and
        // the node's first sorted body are loaded now, before the scan below: a
        // slot that holds no cell reads node 0, unused.
        const int64_t cq = ch >= n ? ch : 0;
        const int4 *cs4 = reinterpret_cast<const int4 *>(child + 8 * cq);
        const int4 ca = cs4[0], cb = cs4[1];
        const int clev = cell_level[cq];
        const int ccnt = count[cq];
        const float4 cnode = nodes4[cq];
        const int nstart = k >= total || (!BATCH && item == 0) ? 0 : start[node];  // the single root is node 0
        const int boff0 = k < total ? frame_off(boff, bsum, (int)item) : 0;  // the block's first record
        const uint64_t occ = __ballot(ch != -1);
        const unsigned seg = (unsigned)(occ >> (lane & ~7)) & 0xffu;
        const int rank = __popc(seg & ((1u << s) - 1u));
        // Sorted position of a body child: the node's first sorted body plus the
        // bodies of the slots before it (children in slot order are consecutive
        // ranges of the key order).  8-lane exclusive sum of the children's sizes.
        const int w = ch == -1 ? 0 : ch < n ? 1 : ccnt;
        int off = w;
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) {
            const int y = __shfl_up(off, o, 8);
            if (s >= o) off += y;
        }
        off -= w;
        if (ch == -1 && !(k < total && item < nroot && s == 0)) continue;
        double span;
        float th;
        if (BATCH) {
            const int sys = item < nroot ? (int)item : si.sys_of[nstart];
            span = si.ext[4 * sys + 3];
            th = si.theta[sys];
        } else {
            span = st->ext[3];
            th = theta;
        }
        if (k < total && item < nroot && s == 0) {
            froot4[item] = walk_record(BATCH ? nodes4[node] : st->root4);
            frootm[item] = chain_bottom<BATCH>(node, n, child, cell_level, true, span, th, eps2, boff, bsum);
            pblk[item] = -1;
        }
        if (ch == -1) continue;
        const int64_t slot = (int64_t)boff0 + rank;
        if (ch < n) {
            const int q = nstart + off;
            const int ps = q >= 0 && q < n ? q : pos[ch];
            fnode[slot] = nodes4[ps];
            fmeta[slot] = make_int2(ps << 4, body_crit);
            bpar[ps] = (int)item;
        } else {
            fnode[slot] = walk_record(cnode);
            fmeta[slot] = chain_bottom_from<BATCH>(ch, ca, cb, clev, n, child, cell_level, span, th, eps2, boff, bsum);
            pblk[block_of<BATCH>(ch, n)] = (int)item;
        }
    }
}

// Also writes sorted[] (the reference's output of the sort stage).  A subtree of
// more than kOrdCells cells (chains of one-child cells) keeps its cells' offsets in
// `place`, one word per cell.
constexpr int kOrdCells = 1024;
__global__ void __launch_bounds__(256) group_order_kernel(Segs g, int base0, const uint64_t *__restrict__ skeys,
                                                          const int4 *__restrict__ sub,
                                                          const int4 *__restrict__ subcells,
                                                          const int *__restrict__ child, const int *__restrict__ count,
                                                          const int *__restrict__ start,
                                                          const int32_t *__restrict__ cell_level,
                                                          const int2 *__restrict__ top_place,
                                                          const int2 *__restrict__ sub_place, int *place,
                                                          const int32_t *__restrict__ perm, int *__restrict__ sorted,
                                                          int32_t *__restrict__ gorder, const DeviceState *st)
{
    __shared__ uint16_t s_cnt[kOrdCells], s_off[kOrdCells], s_par[kOrdCells];
    __shared__ uint16_t s_boff[kSubtreeMax], s_bpar[kSubtreeMax];  // bodies: offset, cell
    __shared__ OrderTables tab;
    static_assert(kSubtreeMax <= 2048, "offsets of 11 bits");
    if (latched(st)) return;
    const int tid = threadIdx.x, n = g.n;
    const int nsub = __hip_atomic_load(&st->nsub, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int ntop = __hip_atomic_load(&st->ntop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    order_tables_fill(tab);
    __syncthreads();
    // a place under a top cell or root: the offsets from there up
    auto up = [&](int2 e) {
        int p = e.x;
        while (e.y >= 0) {
            e = top_place[e.y];
            p += e.x;
        }
        return p;
    };
    for (int job = blockIdx.x; job < nsub; job += gridDim.x) {
        const int4 sc = subcells[job], jb = sub[job];
        const int base = sc.x, ks = sc.y, L0 = sc.z, a = jb.x, cnt = jb.y - jb.x;
        const bool lds = ks <= kOrdCells;
        const int2 pl = sub_place[job];
        if (lds)
            for (int k = tid; k < ks; k += 256) s_cnt[k] = (uint16_t)count[base + k];
        const int state0 = order_state(tab, skeys[a], 0, 0, L0);
        const int p0 = up(pl);
        __syncthreads();
        for (int k = tid; k < ks; k += 256) {
            const int c = base + k, first = start[c];
            const int4 *row = reinterpret_cast<const int4 *>(child + 8 * (int64_t)c);
            const int4 ra = row[0], rb = row[1];
            const int state = order_state(tab, skeys[first], state0, L0, cell_level[c]);
            const int v[8] = {ra.x, ra.y, ra.z, ra.w, rb.x, rb.y, rb.z, rb.w};
            int w[8], dg[8];
            const uint32_t dig = tab.dig[state];
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                w[s] = v[s] == -1 ? 0 : v[s] < n ? 1 : lds ? (int)s_cnt[v[s] - base] : count[v[s]];
                dg[s] = (int)(dig >> (4 * s)) & 7;
            }
            int cur = first - a;
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                int off = 0;
#pragma unroll
                for (int o = 0; o < 8; ++o) off += dg[o] < dg[s] ? w[o] : 0;
                if (v[s] != -1) {
                    if (v[s] < n) {
                        s_boff[cur] = (uint16_t)off;
                        s_bpar[cur] = (uint16_t)k;
                    } else if (lds) {
                        s_off[v[s] - base] = (uint16_t)off;
                        s_par[v[s] - base] = (uint16_t)k;
                    } else {
                        place[v[s]] = off | k << 11;
                    }
                }
                cur += w[s];
            }
        }
        __syncthreads();
        for (int i = tid; i < cnt; i += 256) {
            int p = p0 + s_boff[i];
            for (int c = s_bpar[i]; c != 0;) {  // the subtree's root is its first cell
                if (lds) {
                    p += s_off[c];
                    c = s_par[c];
                } else {
                    const int e = place[base + c];
                    p += e & 2047;
                    c = e >> 11;
                }
            }
            gorder[p] = a + i;
        }
        __syncthreads();
    }
    // bodies that hang from a top cell or a root themselves: eight lanes per cell
    const int d = tid & 7;
    for (int i = (int)(blockIdx.x * 256 + tid) >> 3; i < ntop + g.nseg; i += (int)(gridDim.x * 256) >> 3) {
        const bool top = i < ntop;
        const int c = top ? base0 + i : seg_root(g, i - ntop);
        const int v = child[8 * (int64_t)c + d];
        if (((__ballot(v >= 0 && v < n) >> (tid & 56)) & 0xff) == 0) continue;  // of the cell's lanes
        const int a = top ? start[c] : seg_lo(g, i - ntop);
        const int w = v == -1 ? 0 : v < n ? 1 : count[v];
        const uint32_t dig = tab.dig[top ? order_state(tab, skeys[a], 0, 0, cell_level[c]) : 0];
        int before = 0, below = 0;
        for (int s = 0; s < 8; ++s) {
            const int ws = __shfl(w, s, 8);
            before += s < d ? ws : 0;
            below += ((int)(dig >> (4 * s)) & 7) < ((int)(dig >> (4 * d)) & 7) ? ws : 0;
        }
        if (v >= 0 && v < n) gorder[up(top ? make_int2(below, i) : make_int2(a + below, -1))] = a + before;
    }
    for (int k = blockIdx.x * 256 + tid; k < n; k += gridDim.x * 256) sorted[k] = perm[k];
}

// ------------------------------------------------------------------ launchers
static inline int capped_grid(int64_t work, int cap = 65536)
{
    int64_t g = (work + 255) / 256;
    if (g < 1) g = 1;
    return (int)(g > cap ? cap : g);
}


// Workgroups of a job loop (subtree build, locked insertion, subtree summary, group
// order): a few per subtree (a subtree averages about 256 bodies) up to kBuildBlocks,
// which leaves about one each at 4M bodies, and about one per subtree above.  With
// many jobs per workgroup the stride balances them worse: at N = 48.8M, 16384 summary
// workgroups took 3.50 ms against 3.30 ms for a shared job counter.  Workgroups that
// find no job still have to be dispatched: at N = 2,000, 16384 of them cost each of these
// kernels several microseconds.
static int job_grid(int nbodies)
{
    return std::min(1 << 20, std::max({256, std::min(kBuildBlocks, nbodies / 64), nbodies / 256}));
}

// From this many bodies on, the subtrees of a launch go to two pools of LDS by size:
// there are then several rounds of workgroups, and the small ones leave room for more at
// once.  Below, nearly all are resident together and a second launch only costs its 4 to
// 5 us.  Summary, one pool and two: 43 and 50 us at 1M, 162 and 141 at 4M, 366 and 286 at
// 7.5M bodies in 512 systems; build: 30 and 37, 89 and 88, 207 and 177.
constexpr int kSumTwoPools = 1 << 21, kBuildTwoPools = 1 << 22;

// Up to this many bodies (some 250 subtrees) and systems (up to eight subtrees each, however
// small) every workgroup of the build adds up the cells of the subtrees before its
// own, instead of a launch that scans the counts: nothing to 0.5 us more at 2,000 and 32,768
// bodies for a launch of 3.9, 3.8 us more at 150,001 and 4.3 for an ensemble of 96 systems
// with 100,000.  Each workgroup reads all counts about once, so without the line of the
// systems 8,192 of 8 bodies would read some 15,000 counts in each of 1,024 workgroups.
constexpr int kBuildScan = 1 << 16, kBuildScanSystems = 192;

static void build_tree(Segs g, int nsamples, int base0, int m, TreeScratch &ts, DeviceState *st, hipStream_t s,
                       int n, const uint64_t *skeys, const int32_t *perm, const uint64_t *keys,
                       const int32_t *pos, const float4 *bodies4, float4 *nodes4, int *child, int *index,
                       int32_t *cell_level, int *start, bool locked)
{
    const int tb = (32 * nsamples + 255) / 256;
    after_sort_kernel<<<tb + capped_grid(n), 256, 0, s>>>(g, nsamples, tb, skeys, ts.top_flag, ts.top_id, ts.top_a,
                                                          ts.top_b, ts.lcp, pos, bodies4, nodes4, st);
    const int wire = nsamples * kLevels + g.nseg;  // entries, 8 lanes each
    const auto wire_with = [&](auto kernel) {
        kernel<<<(8 * wire + 255) / 256, 256, 0, s>>>(g, nsamples, skeys, perm, child, cell_level, ts.top_flag, ts.top_id,
                                                      ts.top_a, ts.top_b, ts.sub, ts.sub_max, base0, m, index, start,
                                                      ts.top_place, ts.sub_place, st);
    };
    if (nsamples * kLevels <= kWireScan) {
        wire_with(top_wire_kernel<true>);
    } else {
        launch_exclusive_scan_u32(ts.top_id, nsamples * kLevels, ts.scan_tmp, s);
        wire_with(top_wire_kernel<false>);
    }
    subtree_cells_kernel<<<capped_grid(64 * (int64_t)ts.sub_max, 4096), 256, 0, s>>>(ts.sub, ts.sub_max, ts.lcp,
                                                                                     ts.cbase, st);
    const bool scan = !locked && g.n <= kBuildScan && g.nseg <= kBuildScanSystems;
    if (!scan) subtree_base_kernel<<<1, 1024, 0, s>>>(ts.cbase, ts.sub_max, base0, m, index, st);
    const int jobs = job_grid(g.n);
    const auto build_with = [&](auto kernel, int threads) {
        kernel<<<jobs, threads, 0, s>>>(m, skeys, perm, child, base0, ts.cbase, cell_level, start, ts.sub, ts.sub_max,
                                        ts.subcells, index, st);
    };
    if (locked) {
        subtree_insert_kernel<<<jobs, 256, 0, s>>>(n, m, skeys, perm, keys, ts.lcp, child, base0, ts.cbase, cell_level,
                                                   ts.sub, ts.sub_max, ts.subcells, st);
    } else if (scan) {
        build_with(subtree_build_kernel<256, kBuildPool, 0, true>, 256);
    } else if (g.n < kBuildTwoPools) {
        build_with(subtree_build_kernel<256, kBuildPool, 0, false>, 256);
    } else {
        build_with(subtree_build_kernel<256, kBuildPool, kBuildSmall, false>, 256);
        build_with(subtree_build_kernel<kBuildSmallT, kBuildSmall, 0, false>, kBuildSmallT);
    }
}

template <bool CURSOR>
static void summarise_tree(Segs g, int base0, int nsamples, TreeScratch &ts, DeviceState *st, hipStream_t s,
                           const SumOut &o)
{
    const int grid = job_grid(g.n);
    if (g.n < kSumTwoPools) {
        subtree_summary_kernel<CURSOR, 256, kSumPool, 0><<<grid, 256, 0, s>>>(o, ts.sub, ts.sub_max, ts.subcells, st);
    } else {
        subtree_summary_kernel<CURSOR, 256, kSumPool, kSumSmall><<<grid, 256, 0, s>>>(o, ts.sub, ts.sub_max, ts.subcells, st);
        subtree_summary_kernel<CURSOR, kSumSmallT, kSumSmall, 0><<<grid, kSumSmallT, 0, s>>>(o, ts.sub, ts.sub_max, ts.subcells, st);
    }
    if (g.n <= kTopFew) {
        top_summary_kernel<CURSOR, kTopSmall, true><<<1, kTopThreads, 0, s>>>(o, g, base0, nsamples, ts.top_id, st);
    } else if (g.n <= kTopOneGroup) {
        top_summary_kernel<CURSOR, kTopLarge, true><<<1, kTopThreads, 0, s>>>(o, g, base0, nsamples, ts.top_id, st);
    } else {
        top_levels_kernel<CURSOR><<<kTopBlocks, kTopLevelThreads, 0, s>>>(o, base0, nsamples, ts.top_id, st);
        top_summary_kernel<CURSOR, kTopLarge, false><<<1, kTopThreads, 0, s>>>(o, g, base0, nsamples, ts.top_id, st);
    }
}
// base0: the first top cell's id; nsamples: the top table's samples.
static void summarise_tree(Segs g, int base0, int nsamples, TreeScratch &ts, DeviceState *st, hipStream_t s,
                           const SumOut &o)
{
    if (o.cursor)
        summarise_tree<true>(g, base0, nsamples, ts, st, s, o);
    else
        summarise_tree<false>(g, base0, nsamples, ts, st, s, o);
}

static inline int samples_of(int n) { return (n + kSubtreeMax - 1) / kSubtreeMax; }

bool alloc_tree_scratch(TreeScratch &ts, int n, int nseg, int samples)
{
    ts.samples_max = samples;
    int64_t sub = 8 * ((int64_t)samples * kKeyLevels + nseg);
    sub = std::min<int64_t>(sub, (int64_t)n / 2 + 8 * (int64_t)nseg + 8);
    ts.sub_max = (int)sub;
    const size_t tt = (size_t)samples * kLevels;
    return hipMalloc((void **)&ts.lcp, (size_t)n + 1) == hipSuccess &&
           hipMalloc((void **)&ts.top_flag, 4 * tt) == hipSuccess &&
           hipMalloc((void **)&ts.top_id, 4 * tt) == hipSuccess &&
           hipMalloc((void **)&ts.top_a, 4 * tt) == hipSuccess &&
           hipMalloc((void **)&ts.top_b, 4 * tt) == hipSuccess &&
           hipMalloc((void **)&ts.top_place, sizeof(int2) * tt) == hipSuccess &&
           hipMalloc((void **)&ts.sub_place, sizeof(int2) * (size_t)ts.sub_max) == hipSuccess &&
           hipMalloc((void **)&ts.sub, sizeof(int4) * (size_t)ts.sub_max) == hipSuccess &&
           hipMalloc((void **)&ts.subcells, sizeof(int4) * (size_t)ts.sub_max) == hipSuccess &&
           hipMalloc((void **)&ts.cbase, sizeof(uint32_t) * ((size_t)ts.sub_max + 1)) == hipSuccess &&
           hipMalloc((void **)&ts.scan_tmp, 4 * 1024) == hipSuccess && (int64_t)samples * kLevels <= (1 << 20);
}

void free_tree_scratch(TreeScratch &ts)
{
    void *p[] = {ts.lcp, ts.top_flag, ts.top_id, ts.top_a, ts.top_b, ts.sub, ts.subcells, ts.scan_tmp,
                 ts.cbase, ts.top_place, ts.sub_place};
    for (void *q : p)
        if (q) hipFree(q);
    ts = TreeScratch{};
}

void launch_build(nbx_context *c, hipStream_t s, int n, int m, int *child, int *index)
{
    if (n <= 0) return;
    Segs g{nullptr, nullptr, 1, n, 0};
    build_tree(g, samples_of(n), n, m, c->ts, c->st, s, n, c->skeys, c->perm, c->keys, c->pos, c->bodies4, c->nodes4,
               child, index, c->cell_level, c->start, c->p.build_locked != 0);
}

void launch_summarize(nbx_context *c, hipStream_t s)
{
    Segs g{nullptr, nullptr, 1, c->n, 0};
    SumOut o{c->n, c->child, c->bodies4, c->mass, c->x, c->y, c->z, c->count, c->start, c->pos,
             c->cell_level, c->sum64, c->nodes4, c->p.build_locked == 0};
    summarise_tree(g, c->n, samples_of(c->n), c->ts, c->st, s, o);
}

// sorted[] and gorder[] (place: scratch of one int per node, free until the frame layout).
static void order_bodies(Segs g, int base0, const TreeScratch &ts, DeviceState *st, hipStream_t s,
                         const uint64_t *skeys, const int *child, const int *count, const int *start,
                         const int32_t *cell_level, int *place, const int32_t *perm, int *sorted, int32_t *gorder)
{
    group_order_kernel<<<job_grid(g.n), 256, 0, s>>>(g, base0, skeys, ts.sub, ts.subcells, child, count, start,
                                                     cell_level, ts.top_place, ts.sub_place, place, perm, sorted, gorder,
                                                     st);
}

void launch_layout(nbx_context *c, hipStream_t s, int *sorted)
{
    Segs g{nullptr, nullptr, 1, c->n, 0};
    order_bodies(g, c->n, c->ts, c->st, s, c->skeys, c->child, c->count, c->start, c->cell_level, c->pblk, c->perm,
                 sorted, c->gorder);
    launch_frame_layout(c, s);
}

// Blocks' children, their runs' totals scanned, then the records.  items: blocks at most.
template <bool BATCH, class... Out>
static void lay_out(hipStream_t s, int64_t items, int n, int nroot, const int *index, const int *child, const int32_t *pos,
                    const int32_t *cell_level, const int *count, const int *start, const float4 *nodes4, float4 *fnode,
                    int2 *fmeta, uint32_t *boff, uint32_t *bsum, uint32_t *brun, DeviceState *st, Out... out)
{
    const int runs = (int)((items + kOffRun - 1) / kOffRun);
    const bool scan = runs <= kLayoutRuns;
    frame_count_kernel<BATCH><<<runs, 256, 0, s>>>(n, index, child, boff, scan ? brun : bsum, st);
    if (!scan) launch_scan_one_block(bsum, runs, s);
    const auto with = [&](auto kernel) {
        kernel<<<capped_grid(8 * items), 256, 0, s>>>(n, nroot, index, child, pos, cell_level, count, start, nodes4, fnode,
                                                      fmeta, boff, brun, runs, bsum, out..., st);
    };
    if (scan) with(frame_layout_kernel<BATCH, true>);
    else with(frame_layout_kernel<BATCH, false>);
}

void launch_frame_layout(nbx_context *c, hipStream_t s)
{
    lay_out<false>(s, (int64_t)c->m - c->n + 1, c->n, 1, c->index, c->child, c->pos, c->cell_level, c->count, c->start,
                   c->nodes4, c->fnode, c->fmeta, c->boff, c->bsum, c->brun, c->st, c->froot4, c->frootm, c->pblk, c->bpar,
                   c->p.theta, layout_eps2(c->p), SysInfo{});
    c->layout_theta = c->p.theta;
    c->layout_eps2 = layout_eps2(c->p);
}

void launch_batch_build(nbx_batch *b, hipStream_t s)
{
    Segs g{b->off, b->samp_off, b->S, b->N, 1};
    build_tree(g, b->ts.samples_max, b->N + b->S, b->m, b->ts, b->st, s, b->N, b->skeys, b->perm, b->keys, b->pos,
               b->bodies4, b->nodes4, b->child, b->index, b->cell_level, b->start, b->p.build_locked != 0);
}

void launch_batch_summarize(nbx_batch *b, hipStream_t s)
{
    Segs g{b->off, b->samp_off, b->S, b->N, 1};
    SumOut o{b->N, b->child, b->bodies4, b->mass, nullptr, nullptr, nullptr, b->count, b->start, b->pos,
             b->cell_level, b->sum64, b->nodes4, b->p.build_locked == 0};
    summarise_tree(g, b->N + b->S, b->ts.samples_max, b->ts, b->st, s, o);
}

void launch_batch_layout(nbx_batch *b, hipStream_t s)
{
    Segs g{b->off, b->samp_off, b->S, b->N, 1};
    order_bodies(g, b->N + b->S, b->ts, b->st, s, b->skeys, b->child, b->count, b->start, b->cell_level, b->pblk,
                 b->perm, b->sorted, b->gorder);
    lay_out<true>(s, (int64_t)b->m - b->N, b->N, b->S, b->index, b->child, b->pos, b->cell_level, b->count, b->start,
                  b->nodes4, b->fnode, b->fmeta, b->boff, b->bsum, b->brun, b->st, b->froot4, b->frootm, b->pblk, b->bpar,
                  0.f, layout_eps2(b->p), SysInfo{b->sys_of, b->theta, b->ext});
}

}  // namespace nbx
