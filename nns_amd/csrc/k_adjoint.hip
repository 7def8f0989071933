// k_adjoint.hip -- vector-Jacobian product of the Barnes-Hut accelerations.
//
// Given u_i = dL/da_i for every body, the walk of the force kernel is repeated
// on the same tree and frame layout (so each body meets exactly the nodes of
// its forward interaction list) and, for every interaction of body i with a
// node n of mass M at X (d = X - x_i, s = (|d|^2 + eps^2)^-3/2),
//     h      = M s (u - 3 (u.d) d / (|d|^2 + eps^2))      = d(u.a_i)/dX
//     dL/dx_i -= h,   dL/dX_n += h,   dL/dM_n += s (u.d).
// The lane's own body contributes nothing (its forward term vanishes
// identically); another body at the same point does when eps > 0 (h = M eps^-3
// u) and is skipped, as in the forward walk, when eps = 0.  The node terms
// of one child step are summed over the lanes that took it by DPP adds and row
// swaps (VjpLog).  Bodies are nodes too.
//
// The per-step sums do not go to the nodes by atomics (one FP64 atomic per
// component and step is a memory-side transaction: at N = 262K they cost more
// than the walk).  They are appended to a log {32-bit node id, float4}: each
// wave takes chunks of records with one atomicAdd and seals the unused tail of a
// chunk with a sentinel node id.  The log is then summed per node in FP64: in
// bins of node ids, tile by tile, through LDS (log_tiles_kernel and after) while
// the ids make at most kLogBins bins (n_max + m_max below 2^22), else by a stable
// radix sort of the ids and a segmented sum (log_reduce_kernel).  The order of a
// node's records is that of the chunk grants, so its FP64 total can differ from run to
// run in its last bits.  A wave that finds the log full adds its remaining sums
// with atomics directly.
//
// A cell's X and M are sums over its bodies, X = sum m_k x_k / M, so the node
// gradients flow down: for every body k
//     dL/dx_k += m_k A,   dL/dm_k += B + A.x_k,
// with A = sum of G_c / M_c and B = sum of (GM_c - G_c.X_c / M_c) over the
// cells c that contain k.  The walk attributes a collapsed one-child chain to
// its bottom cell; the cells of a chain hold the same bodies, mass and centre,
// so the sums over the ancestors are unchanged.
#include "walk_split.h"

namespace nbx {

// Log records taken per atomicAdd: few, so that short walks leave few unused, but
// more where one counter serves all waves (serialised: about 11 ns per grant).
constexpr int kChunkBinned = 128, kChunkSorted = 512;
constexpr int kLogLine = 32;    // ints per counter of the log: a 128-byte line each
constexpr int kLogParts = 64;   // counters, and parts of the log, at most
constexpr int kLogBins = 1024;  // bins of the binned sums at most
// Records of a tile: the larger from kLogTileLine records on, so that a bin's run
// in a tile spans whole lines (N = 262,144: 10 records with the smaller, 40 with the
// larger); shorter logs need the blocks.
constexpr int kLogTile = 8192, kLogTileMax = 32768;
constexpr int64_t kLogTileLine = 8 << 20;
constexpr int kLogShare = 2048, kLogItems = 1024;  // records of a work item at least, items about

// What the walk of one group needs beside the tree's frames.
struct VjpArgs {
    const float4 *nodes4;
    const int32_t *perm, *gorder;
    const float4 *froot4;
    const int2 *frootm;
    const float *ux, *uy, *uz;
    float4 *own;       // [n] the walk's own part of dL/dx by sorted position
    double *tgt;
    uint32_t *log_id;  // [nlogs subcap] the node-term log, nlogs parts
    float4 *log_val;
    int *log_next;     // [kLogLine nlogs] next free record of each part
    int *err;
    int n, nlogs, subcap, chunk;
    uint32_t sentinel;
    float G;
};

// Sums a lane's four values over rows of 16 lanes, down to one register: component
// c = (lane >> 2) & 3, summed over the four quads of the row (lanes of the same
// lane & 3).  Each halving keeps two values apart by the banks a DPP add writes:
// banks 0 and 2 of u become x's sums of two quads, banks 1 and 3 y's.  The waits are
// those of a DPP read after a vector write.
static __device__ __forceinline__ float quad_sums(float x, float y, float z, float w)
{
    float u, v, r;
    asm("s_nop 1\n\t"
        "v_add_f32_dpp %0, %3, %3 row_ror:4 row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %0, %4, %4 row_ror:4 row_mask:0xf bank_mask:0xa\n\t"
        "v_add_f32_dpp %1, %5, %5 row_ror:4 row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %1, %6, %6 row_ror:4 row_mask:0xf bank_mask:0xa\n\t"
        "s_nop 0\n\t"
        "v_add_f32_dpp %2, %0, %0 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %2, %1, %1 row_ror:8 row_mask:0xf bank_mask:0xc"
        : "=&v"(u), "=&v"(v), "=&v"(r)
        : "v"(x), "v"(y), "v"(z), "v"(w));
    return r;
}

// a's sums over lane and lane ^ 32 in lanes 0..31, b's in lanes 32..63.
static __device__ __forceinline__ float halve32(float a, float b)
{
    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}
// The same over lane ^ 16: a's in rows 0 and 2, b's in rows 1 and 3.
static __device__ __forceinline__ float halve16(float a, float b)
{
    const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(p[0]) + __uint_as_float(p[1]);
}
static __device__ __forceinline__ float quad_xor(float v, int ctrl_is_1)
{
    return ctrl_is_1 ? __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, false))   // 1,0,3,2
                     : __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, false));  // 2,3,0,1
}

// The sums of a frame's node terms on their way to the log.  The step of child j
// brings four values per lane and leaves one (quad_sums) in r[j].  After the
// frame the eight registers are halved against each other over lane ^ 32, lane ^ 16
// and lane ^ 2, and summed over lane ^ 1: lane l then holds component (l >> 2) & 3
// of child (l >> 5 & 1) + 2 (l >> 4 & 1) + 4 (l >> 1 & 1).  Six VALU instructions
// per step and 16 per frame, and no LDS.  Through LDS (one float4 per lane written,
// read back transposed) a step took 8 and 2 KB of LDS traffic, and the buffers held
// the kernel to 16 waves per CU.
struct VjpLog {
    float r[8];
    int idv;         // lane j: the node id of child j
    unsigned took;   // children that some lane took
    int cpos, cend;  // the wave's log chunk [cpos, cend), records of the whole log
    int part;        // the part of the log it takes chunks from
    bool full;       // the log is full: add sums with atomics
};

// The arguments that few frames need are read again from the kernel's argument
// block (VjpArgs is the first parameter of the walk kernels), so that they hold no
// scalar registers during the walk.
typedef const __attribute__((address_space(4))) VjpArgs *VjpArgsPtr;
static __device__ __forceinline__ VjpArgsPtr vjp_args()
{
    VjpArgsPtr k = (VjpArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(k));
    return k;
}

static __device__ __forceinline__ void vjp_flush(VjpLog &w, int lane)
{
    const VjpArgsPtr v = vjp_args();
    uint32_t *log_id = v->log_id;
    float *log_val = reinterpret_cast<float *>(v->log_val);
    const float a = halve16(halve32(w.r[0], w.r[1]), halve32(w.r[2], w.r[3]));
    const float b = halve16(halve32(w.r[4], w.r[5]), halve32(w.r[6], w.r[7]));
    int l2 = lane;
    asm volatile("" : "+v"(l2));  // its test is made here, not held in scalar registers
    float t = (l2 & 2 ? b : a) + quad_xor(l2 & 2 ? a : b, 0);
    t += quad_xor(t, 1);
    const int count = __popc(w.took);
    if (!w.full && w.cend - w.cpos < count) {
        if (lane < w.cend - w.cpos) log_id[w.cpos + lane] = v->sentinel;  // seal the old chunk (< 8 records)
        const int part = __builtin_amdgcn_readfirstlane(w.part), subcap = v->subcap, chunk = v->chunk;
        int k = 0;
        if (lane == 0) k = atomicAdd(&v->log_next[part * kLogLine], chunk);
        k = __builtin_amdgcn_readfirstlane(k);
        if (k < 0 || k > subcap - chunk) {
            w.full = true;
            w.cpos = w.cend = 0;
        } else {
            w.cpos = part * subcap + k;  // the whole log holds less than 2^31 records
            w.cend = w.cpos + chunk;
        }
    }
    const int j = (lane >> 5 & 1) | (lane >> 3 & 2) | (lane << 1 & 4), c = lane >> 2 & 3;
    if (!w.full) {
        if (!(lane & 1) && (w.took >> j & 1u))
            log_val[4 * (int64_t)(w.cpos + __popc(w.took & ((1u << j) - 1u))) + c] = t;
        if (lane < 8 && (w.took >> lane & 1u))
            log_id[w.cpos + __popc(w.took & ((1u << lane) - 1u))] = (uint32_t)w.idv;
        w.cpos += count;
    } else {
        const int id = __shfl(w.idv, j);
        if (!(lane & 1) && (w.took >> j & 1u)) unsafeAtomicAdd(v->tgt + 4 * (int64_t)id + c, (double)t);
    }
    w.took = 0u;
}

// The bodies of a group: lane l's body at (x, y, z), u scaled by G.
struct VjpBody {
    float4 me;
    float vx, vy, vz;
    float ox, oy, oz;  // dL/dx of the lane's own body
    int me_tag;        // the descriptor tag of the lane's own body
};

// One child step (child j of a frame, descriptor {tag, crit} as in the force walk);
// returns the lanes that open the child.
template <bool SOFT>
static __device__ __forceinline__ uint64_t vjp_step(VjpBody &o, VjpLog &w, int n, float eps2, const int j,
                                                    const float4 q, const int tag, const float crit,
                                                    const uint64_t mask)
{
    const float dx = q.x - o.me.x;
    const float dy = q.y - o.me.y;
    const float dz = q.z - o.me.z;
    const float d2e = fmaf(dz, dz, fmaf(dy, dy, fmaf(dx, dx, eps2)));  // |d|^2 + eps^2
    const uint64_t ok = __ballot(crit < d2e);  // the force walk's test
    // The lane's own term vanishes identically (a body's tag is its sorted
    // position << 4); another body at the same point keeps its derivative
    // when eps > 0, and is left out, as in the forward walk, when eps = 0.
    const uint64_t keep = SOFT ? ~__ballot(tag == o.me_tag) : __ballot(d2e > 0.f);
    const uint64_t takem = mask & ok & keep;
    if (takem) {
        const bool sel = __builtin_amdgcn_inverse_ballot_w64(takem);
        const float r2 = SOFT ? d2e : (sel ? d2e : 1.f);  // finite on every lane (d2e >= eps^2 > 0 when SOFT)
        const float rs = __builtin_amdgcn_rsqf(r2);
        const float rs2 = rs * rs;
        const float s3 = sel ? rs * rs2 : 0.f;
        const float ud = fmaf(o.vz, dz, fmaf(o.vy, dy, o.vx * dx));
        const float k3 = 3.f * ud * rs2;
        const float ms = q.w * s3;
        const float hx = ms * fmaf(-k3, dx, o.vx);
        const float hy = ms * fmaf(-k3, dy, o.vy);
        const float hz = ms * fmaf(-k3, dz, o.vz);
        const float hw = s3 * ud;
        o.ox -= hx;
        o.oy -= hy;
        o.oz -= hz;
        w.r[j] = quad_sums(hx, hy, hz, hw);
        asm("v_writelane_b32 %0, %1, %2" : "+v"(w.idv) : "s"((tag & 15) == 0 ? tag >> 4 : n + (tag >> 4)), "n"(j));
        w.took |= 1u << j;
    }
    return mask & ~ok;
}

static __device__ __forceinline__ VjpBody vjp_body(const VjpArgs &v, int first, int lane, uint64_t &live, int &p)
{
    const bool valid = lane < min(64, v.n - first);
    VjpBody o;
    p = valid ? v.gorder[first + lane] : 0;  // the lane's body, by sorted position
    o.me = valid ? v.nodes4[p] : make_float4(0.f, 0.f, 0.f, 0.f);
    const int i = valid ? v.perm[p] : 0;
    o.me_tag = valid ? p << 4 : -1;
    o.vx = valid ? v.G * v.ux[i] : 0.f;
    o.vy = valid ? v.G * v.uy[i] : 0.f;
    o.vz = valid ? v.G * v.uz[i] : 0.f;
    o.ox = o.oy = o.oz = 0.f;
    live = __ballot(valid);
    return o;
}

static __device__ __forceinline__ VjpLog vjp_log(int part)
{
    VjpLog w{};
    w.took = 0u;
    w.part = part;
    asm volatile("" : "+v"(w.part));  // rarely used: not in a scalar register
    w.cpos = w.cend = 0;
    w.full = false;
    return w;
}

// Seals the unused rest of the wave's last chunk.
static __device__ __forceinline__ void vjp_seal(VjpLog &w, int lane)
{
    if (!w.full)
        for (int k = w.cpos + lane; k < w.cend; k += 64) vjp_args()->log_id[k] = vjp_args()->sentinel;
}

// One wave per group.
template <int W, bool SOFT>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(8)))
vjp_kernel(VjpArgs v, int ngroups, const float4 *__restrict__ fnode, const int2 *__restrict__ fmeta, float eps2,
           const DeviceState *st)
{
    __shared__ uint4 stk[W][kForceStack];
    if (latched(st)) return;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int g = xcd_swizzle(blockIdx.x, gridDim.x) * W + wave;
    if (g >= ngroups) return;
    const int part = g % v.nlogs;
    uint64_t live;
    int p;
    VjpBody o = vjp_body(v, g * 64, lane, live, p);
    VjpLog w = vjp_log(part);
    uint4 *s = stk[wave];
    int sp = 0;
    {
        const int2 rd = v.frootm[0];
        const int rt = __builtin_amdgcn_readfirstlane(rd.x);
        const float rc = __int_as_float(__builtin_amdgcn_readfirstlane(rd.y));
        const uint64_t om = vjp_step<SOFT>(o, w, v.n, eps2, 0, v.froot4[0], rt, rc, live);
        if (w.took) vjp_flush(w, lane);
        if (om) {
            if (lane == 0) s[0] = make_uint4((unsigned)rt, 0u, (unsigned)om, (unsigned)(om >> 32));
            sp = 1;
        }
    }
    bool overflow = false;
    while (sp > 0) {  // one exit: the accumulators keep their registers between frames
        if (sp > kForceStack - 7) {
            overflow = true;
            sp = 0;
            continue;
        }
        sp = __builtin_amdgcn_readfirstlane(sp - 1);
        uint4 e = s[sp];
        const int tag = __builtin_amdgcn_readfirstlane((int)e.x);
        const int nch = tag & 15, off = tag >> 4;
        float4 q[8];
        int2 d[8];
        load_block(fnode + off, fmeta + off, 0u, q, d);
        asm volatile("" : "+v"(e.z), "+v"(e.w));
        const uint64_t mask = ((uint64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)e.w) << 32) |
                              (uint64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)e.z);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (j >= nch) break;
            const int tj = __builtin_amdgcn_readfirstlane(d[j].x);
            const float cj = __int_as_float(__builtin_amdgcn_readfirstlane(d[j].y));
            const uint64_t om = vjp_step<SOFT>(o, w, v.n, eps2, j, q[j], tj, cj, mask);
            if (om) {
                if (lane == 0) s[sp] = make_uint4((unsigned)tj, 0u, (unsigned)om, (unsigned)(om >> 32));
                sp = __builtin_amdgcn_readfirstlane(sp + 1);
            }
        }
        if (w.took) vjp_flush(w, lane);
    }
    if (overflow && lane == 0) atomicOr(vjp_args()->err, kErrStack);
    vjp_seal(w, lane);
    if (__builtin_amdgcn_inverse_ballot_w64(live)) vjp_args()->own[p] = make_float4(o.ox, o.oy, o.oz, 0.f);
}

// The same walk shared by the S waves of a workgroup (walk_split.h).
template <int S, bool SOFT>
__global__ void __launch_bounds__(64 * S) __attribute__((amdgpu_waves_per_eu(8)))
vjp_split_kernel(VjpArgs v, const float4 *__restrict__ fnode, const int2 *__restrict__ fmeta, float eps2,
                 const DeviceState *st)
{
    __shared__ SplitStack<S> L;
    __shared__ int s_stop;
    static_assert(sizeof(L.stk) >= sizeof(float) * 3 * 64 * S, "the waves' sums meet in the stack's memory");
    if (threadIdx.x == 0) s_stop = latched(st);  // one read: the workgroup stays or leaves as a whole
    __syncthreads();
    if (s_stop) return;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int g = xcd_swizzle(blockIdx.x, gridDim.x);
    const int part = (g * S + wave) % v.nlogs;
    uint64_t live;
    int p;
    VjpBody o = vjp_body(v, g * 64, lane, live, p);
    VjpLog w = vjp_log(part);
    const int2 rd = v.frootm[0];
    const int rt = __builtin_amdgcn_readfirstlane(rd.x);
    const float rc = __int_as_float(__builtin_amdgcn_readfirstlane(rd.y));
    const float4 rq = v.froot4[0];
    uint64_t om;
    if (wave == 0) {  // the root counts once
        om = vjp_step<SOFT>(o, w, v.n, eps2, 0, rq, rt, rc, live);
        if (w.took) vjp_flush(w, lane);
    } else {
        const float dx = rq.x - o.me.x, dy = rq.y - o.me.y, dz = rq.z - o.me.z;
        om = live & ~__ballot(rc < fmaf(dz, dz, fmaf(dy, dy, fmaf(dx, dx, eps2))));
    }
    const bool ok = split_walk<S>(L, wave, lane, make_uint4((unsigned)rt, 0u, (unsigned)om, (unsigned)(om >> 32)),
                                  om != 0, [&](const uint4 *ep, uint4 *out) -> int {
        uint4 e = *ep;
        const int tag = __builtin_amdgcn_readfirstlane((int)e.x);
        const int nch = tag & 15, off = tag >> 4;
        float4 q[8];
        int2 d[8];
        load_block(fnode + off, fmeta + off, 0u, q, d);
        asm volatile("" : "+v"(e.z), "+v"(e.w));
        const uint64_t mask = ((uint64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)e.w) << 32) |
                              (uint64_t)(unsigned)__builtin_amdgcn_readfirstlane((int)e.z);
        int k = 0;
        asm volatile("" : "+s"(k));  // a scalar count
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (j >= nch) break;
            const int tj = __builtin_amdgcn_readfirstlane(d[j].x);
            const float cj = __int_as_float(__builtin_amdgcn_readfirstlane(d[j].y));
            const uint64_t m = vjp_step<SOFT>(o, w, v.n, eps2, j, q[j], tj, cj, mask);
            if (m) {
                if (lane == 0) out[k] = make_uint4((unsigned)tj, 0u, (unsigned)m, (unsigned)(m >> 32));
                k = __builtin_amdgcn_readfirstlane(k + 1);
            }
        }
        if (w.took) vjp_flush(w, lane);
        return k;
    });
    if (!ok && threadIdx.x == 0) atomicOr(vjp_args()->err, kErrStack);
    vjp_seal(w, lane);
    __syncthreads();  // the stack is free
    float *red = reinterpret_cast<float *>(L.stk);
    red[(3 * wave + 0) * 64 + lane] = o.ox;
    red[(3 * wave + 1) * 64 + lane] = o.oy;
    red[(3 * wave + 2) * 64 + lane] = o.oz;
    __syncthreads();
    if (wave == 0 && __builtin_amdgcn_inverse_ballot_w64(live)) {
        float x = 0.f, y = 0.f, z = 0.f;
#pragma unroll
        for (int k = 0; k < S; ++k) {
            x += red[(3 * k + 0) * 64 + lane];
            y += red[(3 * k + 1) * 64 + lane];
            z += red[(3 * k + 2) * 64 + lane];
        }
        vjp_args()->own[p] = make_float4(x, y, z, 0.f);
    }
}

// Clears the gradient sums and the log's counters (of a small system more than its sums).
__global__ void __launch_bounds__(256) vjp_clear_kernel(double *__restrict__ p, int64_t count, int *__restrict__ next,
                                                        int nnext)
{
    const int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x, stride = (int64_t)blockDim.x * gridDim.x;
    for (int64_t k = t; k < count; k += stride) p[k] = 0.0;
    for (int64_t k = t; k < nnext; k += stride) next[k] = 0;
}

// ---- sums of the log, node by node: binned form
// The ids are cut into bins of 2^shift (at most kLogBins).  Each tile of records is
// put in bin order by itself (log_tiles_kernel), so the records of a bin are one
// run per tile, listed in the tile's row of tab; no record moves further than its
// tile, and no count has to be known before.  A workgroup then adds the runs of
// one bin into FP64 sums in LDS (log_bins_kernel) and adds those to the nodes.  A
// bin of many records (the cells near the root, which every group meets) is shared
// by several workgroups (log_plan_kernel), whose sums meet by atomics.  HBM-bound
// passes over 20 bytes per record, the tiles' scattered within 640 KB: at N = 262,144
// (about 14 M records) tiles 0.19, plan 0.013, bins 0.16 ms, where three radix passes
// over (id, index), a gather of the values and a segmented sum took 0.68 ms; at
// N = 20,011 0.041 ms against 0.11.

// Records of part l that were granted (a part's chunks end at subcap).
static __device__ inline int log_part_count(const int *next, int l, int subcap)
{
    return min(next[l * kLogLine], subcap);
}

// Tile v = t nlogs + l is the t-th of part l.  The ids are read twice (counted, then
// placed from running positions) instead of held in registers, so that two
// workgroups fit a CU and one's scan overlaps the other's loads.
__global__ void __launch_bounds__(1024) log_tiles_kernel(const uint32_t *__restrict__ log_id,
                                                         const float4 *__restrict__ log_val,
                                                         const int *__restrict__ next, int nlogs, int subcap, int tile,
                                                         int shift, int nbins, uint32_t sentinel,
                                                         uint32_t *__restrict__ out_id, float4 *__restrict__ out_val,
                                                         uint16_t *__restrict__ tab)
{
    __shared__ uint32_t cnt[kLogBins];
    __shared__ uint32_t sh[16];
    static_assert(kLogBins == 1024 && kLogTileMax < 65536, "one bin per thread, 16-bit places");
    constexpr int U = 4;
    const int tid = threadIdx.x, v = blockIdx.x, l = v % nlogs, t0 = v / nlogs * tile;
    const int n = min(log_part_count(next, l, subcap) - t0, tile);
    if (n <= 0) return;
    const int64_t base = (int64_t)l * subcap + t0;
    const uint32_t *src = log_id + base;
    const float4 *val = log_val + base;
    cnt[tid] = 0u;
    __syncthreads();
    for (int k0 = tid; k0 < n; k0 += 1024 * U) {
        uint32_t id[U];
#pragma unroll
        for (int u = 0; u < U; ++u) id[u] = k0 + 1024 * u < n ? src[k0 + 1024 * u] : sentinel;
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (id[u] != sentinel) atomicAdd(&cnt[id[u] >> shift], 1u);
    }
    __syncthreads();
    uint32_t tot;
    const uint32_t ex = block_exclusive_scan(cnt[tid], sh, &tot);
    cnt[tid] = ex;
    uint16_t *row = tab + (int64_t)v * (nbins + 1);
    if (tid < nbins) row[tid] = (uint16_t)ex;
    if (tid == 0) row[nbins] = (uint16_t)tot;
    __syncthreads();
    for (int k0 = tid; k0 < n; k0 += 1024 * U) {
        uint32_t id[U];
        float4 x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            id[u] = k0 + 1024 * u < n ? src[k0 + 1024 * u] : sentinel;
            x[u] = val[k0 + 1024 * u < n ? k0 + 1024 * u : 0];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (id[u] != sentinel) {
                const int64_t k = base + atomicAdd(&cnt[id[u] >> shift], 1u);
                out_id[k] = id[u];
                out_val[k] = x[u];
            }
    }
}

// One workgroup per bin: its records, then work items {bin, first tile, end,
// shared} of about `share` records each, so that the log makes about kLogItems items
// beside one per bin (fewer records per item leave more sums to meet by atomics).
__global__ void __launch_bounds__(256) log_plan_kernel(const uint16_t *__restrict__ tab, const int *__restrict__ next,
                                                       int nlogs, int subcap, int tile, int nbins, int *__restrict__ nitems,
                                                       int4 *__restrict__ items)
{
    __shared__ int red[4];
    __shared__ int s_first;
    const int tid = threadIdx.x, b = blockIdx.x, lane = tid & 63;
    int most = lane < nlogs ? log_part_count(next, lane, subcap) : 0;  // nlogs <= 64 lanes
    int64_t total = most;
    for (int o = 32; o > 0; o >>= 1) {
        most = max(most, __shfl_xor(most, o));
        total += __shfl_xor(total, o);
    }
    const int tiles = (most + tile - 1) / tile * nlogs;
    const int share = max((int)(total / kLogItems), kLogShare);
    int sum = 0;
    for (int v = tid; v < tiles; v += 256)
        if ((int64_t)(v / nlogs) * tile < log_part_count(next, v % nlogs, subcap)) {
            const uint16_t *row = tab + (int64_t)v * (nbins + 1) + b;
            sum += (int)row[1] - (int)row[0];
        }
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    if (lane == 0) red[tid >> 6] = sum;
    __syncthreads();
    sum = red[0] + red[1] + red[2] + red[3];
    const int parts = min((sum + share - 1) / share, tiles);
    if (parts == 0) return;
    if (tid == 0) s_first = atomicAdd(nitems, parts);
    __syncthreads();
    for (int y = tid; y < parts; y += 256)
        items[s_first + y] = make_int4(b, (int)((int64_t)tiles * y / parts), (int)((int64_t)tiles * (y + 1) / parts),
                                       parts > 1);
}

// Sixteen lanes per run, four workgroups per CU at the smallest bins.
template <int SHIFT>
__global__ void __launch_bounds__(512) log_bins_kernel(const uint32_t *__restrict__ id, const float4 *__restrict__ val,
                                                       const uint16_t *__restrict__ tab, const int *__restrict__ next,
                                                       int nlogs, int subcap, int tile, int nbins,
                                                       const int *__restrict__ nitems, const int4 *__restrict__ items,
                                                       int64_t ntgt, double *__restrict__ tgt)
{
    constexpr int R = 1 << SHIFT;
    __shared__ double acc[4 * R];
    const int tid = threadIdx.x, row = tid >> 4, l16 = tid & 15;
    const int n = *nitems;
    if ((int)blockIdx.x >= n) return;
    for (int k = tid; k < 4 * R; k += 512) acc[k] = 0.0;
    for (int it = blockIdx.x; it < n; it += gridDim.x) {
        const int4 w = items[it];
        __syncthreads();
        auto add = [&](uint32_t i, const float4 x) {
            const int j = (int)(i & (R - 1));  // a plane per component: consecutive nodes in consecutive banks
            unsafeAtomicAdd(&acc[j], (double)x.x);
            unsafeAtomicAdd(&acc[R + j], (double)x.y);
            unsafeAtomicAdd(&acc[2 * R + j], (double)x.z);
            unsafeAtomicAdd(&acc[3 * R + j], (double)x.w);
        };
        // U runs at a time, their bounds and then their first records all in flight
        constexpr int U = 4;
        for (int v0 = w.y + row; v0 < w.z; v0 += 32 * U) {
            int64_t k[U], end[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int v = v0 + 32 * u;
                const int64_t t0 = (int64_t)(v / nlogs) * tile;
                k[u] = end[u] = 0;
                if (v < w.z && t0 < log_part_count(next, v % nlogs, subcap)) {
                    const uint16_t *r = tab + (int64_t)v * (nbins + 1) + w.x;
                    const int64_t base = (int64_t)(v % nlogs) * subcap + t0;
                    k[u] = base + r[0] + l16;
                    end[u] = base + r[1];
                }
            }
            uint32_t i[U];
            float4 x[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t q = k[u] < end[u] ? k[u] : 0;
                i[u] = id[q];
                x[u] = val[q];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (k[u] < end[u]) add(i[u], x[u]);
                for (k[u] += 16; k[u] < end[u]; k[u] += 16) add(id[k[u]], val[k[u]]);
            }
        }
        __syncthreads();
        const int64_t t0 = 4 * ((int64_t)w.x << SHIFT);
        for (int k = tid; k < 4 * R; k += 512) {
            const int j = (k & 3) * R + (k >> 2);
            const double a = acc[j];
            acc[j] = 0.0;
            if (a != 0.0 && t0 + k < ntgt) {
                if (w.w) unsafeAtomicAdd(tgt + t0 + k, a);
                else tgt[t0 + k] += a;
            }
        }
    }
}

// ---- sums of the log, node by node: sorted form (ids past kLogBins bins)
// Sort length: every granted chunk is written in full (records or sentinels).
__global__ void log_count_kernel(DeviceState *st, const int *__restrict__ next, int subcap)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) st->log_count = log_part_count(next, 0, subcap);
}

// Per-node sums of the sorted log in tiles of 64 records (one per lane); a wave
// takes kReduceTiles consecutive tiles and issues all their loads (ids, then the
// values gathered from the log) before the first sum.  Per tile: an inclusive
// scan over the lanes holding the same node (six shuffle steps), then the last
// lane of each run adds it to the node.  A run that continues into the previous
// or the next tile is added with an FP64 atomic; a run inside the tile with a
// plain add (no other tile holds that node).
constexpr int kReduceTiles = 4;

__global__ void __launch_bounds__(256) log_reduce_kernel(const uint32_t *__restrict__ sk,
                                                         const int32_t *__restrict__ sv,
                                                         const float4 *__restrict__ val, const DeviceState *st,
                                                         uint32_t sentinel, double *__restrict__ tgt)
{
    if (latched(st)) return;
    const int64_t count = st->log_count;
    const int lane = threadIdx.x & 63;
    const int64_t ntiles = (count + 63) / 64;
    const int64_t wstride = (int64_t)gridDim.x * (blockDim.x >> 6) * kReduceTiles;
    for (int64_t w0 = ((int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * kReduceTiles; w0 < ntiles;
         w0 += wstride) {
        uint32_t ids[kReduceTiles];
        int32_t src[kReduceTiles];
        float4 vals[kReduceTiles];
#pragma unroll
        for (int t = 0; t < kReduceTiles; ++t) {
            const int64_t k = (w0 + t) * 64 + lane;
            ids[t] = k < count ? sk[k] : sentinel;
            src[t] = k < count ? sv[k] : 0;
        }
#pragma unroll
        for (int t = 0; t < kReduceTiles; ++t)
            vals[t] = ids[t] != sentinel ? val[src[t]] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int t = 0; t < kReduceTiles; ++t) {
            if (w0 + t >= ntiles) break;
            const int64_t k0 = (w0 + t) * 64, k = k0 + lane;
            const uint32_t id = ids[t];
            const bool live = id != sentinel;
            float4 v = vals[t];
            const int id32 = live ? (int)id : -1;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int oid = __shfl_up(id32, o);
                const float tx = __shfl_up(v.x, o), ty = __shfl_up(v.y, o), tz = __shfl_up(v.z, o),
                            tw = __shfl_up(v.w, o);
                if (lane >= o && oid == id32) {
                    v.x += tx; v.y += ty; v.z += tz; v.w += tw;
                }
            }
            const int next = __shfl_down(id32, 1);
            const bool last_of_run = live && (lane == 63 || next != id32);
            const int lane0_id = __shfl(id32, 0);
            const bool from_prev = k0 > 0 && lane0_id == id32 && sk[k0 - 1] == id;
            const bool into_next = lane == 63 && k + 1 < count && sk[k + 1] == id;
            if (last_of_run) {
                double *p = tgt + 4 * (int64_t)id;
                if (from_prev || into_next) {
                    unsafeAtomicAdd(p + 0, (double)v.x); unsafeAtomicAdd(p + 1, (double)v.y);
                    unsafeAtomicAdd(p + 2, (double)v.z); unsafeAtomicAdd(p + 3, (double)v.w);
                } else {
                    p[0] += v.x; p[1] += v.y; p[2] += v.z; p[3] += v.w;
                }
            }
        }
    }
}

// Per block b: A and B summed over b and its ancestors (walk up pblk).
__global__ void __launch_bounds__(256) adj_cells_kernel(int n, const int *__restrict__ index,
                                                        const int32_t *__restrict__ pblk,
                                                        const uint32_t *__restrict__ boff,
                                                        const uint32_t *__restrict__ bsum,
                                                        const double *__restrict__ tgt,
                                                        const double4 *__restrict__ sum64, double *__restrict__ ab,
                                                        const DeviceState *st)
{
    if (latched(st)) return;
    const int nblk = *index - n + 1;
    for (int b = blockIdx.x * blockDim.x + threadIdx.x; b < nblk; b += blockDim.x * gridDim.x) {
        double a0 = 0.0, a1 = 0.0, a2 = 0.0, bb = 0.0;
        for (int c = b; c >= 0; c = pblk[c]) {
            const double *t = tgt + 4 * ((int64_t)n + frame_off(boff, bsum, c));  // the block's node id
            double M, X, Y, Z;
            if (c == 0) {
                M = st->root64[0]; X = st->root64[1]; Y = st->root64[2]; Z = st->root64[3];
            } else {
                const int64_t cell = (int64_t)c + n - 1;
                const double4 cs = sum64[cell];
                M = cs.x;
                X = cs.y / M; Y = cs.z / M; Z = cs.w / M;
            }
            if (M > 0.0) {
                const double g0 = t[0] / M, g1 = t[1] / M, g2 = t[2] / M;
                a0 += g0; a1 += g1; a2 += g2;
                bb += t[3] - (g0 * X + g1 * Y + g2 * Z);
            } else {
                bb += t[3];
            }
        }
        double *o = ab + 4 * (int64_t)b;
        o[0] = a0; o[1] = a1; o[2] = a2; o[3] = bb;
    }
}

// Per body (sorted position p): the node terms of the body itself plus the
// flow-down of the cells above it and the walk's own part.
__global__ void __launch_bounds__(256) adj_bodies_kernel(int n, const int32_t *__restrict__ perm,
                                                         const int32_t *__restrict__ bpar,
                                                         const float4 *__restrict__ nodes4,
                                                         const float4 *__restrict__ own,
                                                         const double *__restrict__ tgt,
                                                         const double *__restrict__ ab, float *__restrict__ gx,
                                                         float *__restrict__ gy, float *__restrict__ gz,
                                                         float *__restrict__ gm, const DeviceState *st)
{
    if (latched(st)) return;
    for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += blockDim.x * gridDim.x) {
        const int i = perm[p];
        const float4 b = nodes4[p];
        const double *t = tgt + 4 * (int64_t)p;
        const double *a = ab + 4 * (int64_t)bpar[p];
        const double m = b.w;
        const float4 w = own[p];
        gx[i] = (float)((double)w.x + t[0] + m * a[0]);
        gy[i] = (float)((double)w.y + t[1] + m * a[1]);
        gz[i] = (float)((double)w.z + t[2] + m * a[2]);
        gm[i] = (float)(t[3] + a[3] + a[0] * (double)b.x + a[1] * (double)b.y + a[2] * (double)b.z);
    }
}

// Radix passes over the node ids: a body's id is its sorted position, a cell's
// n + the first record of its frame block, so ids are below n_max + m_max and
// the sentinel, 2^(kRadixBits passes) - 1, must exceed them.
static int sort_passes(int64_t id_max)
{
    int p = 1;
    while ((int64_t(1) << (kRadixBits * p)) < id_max + 2) ++p;
    return p;
}

// Waves per group of the walk (the force launch's rule, with more work per frame
// and so a later end).  Whole product, us: a sphere and a binary + disk at theta 0.5, with
//   16 and 8 waves:  480 groups 236, 277; 121, 143.   640 groups 321, 341; 155, 165.   1,024
//                    groups 426, 439; 213, 220 (at theta 0.8 the sphere 212, 210)
//   8 and 4 waves:   4,096 groups 1,581, 1,586; 741, 786.   5,120 groups 2,035, 2,008; 984,
//                    1,008.   8,192 groups 3,292, 3,187; 1,556, 1,528
//   4 and 1 wave:    8,192 groups 3,187, 3,310; 1,528, 1,746.   12,288 groups 4,915, 4,963;
//                    2,397, 2,434.   16,384 groups 6,826, 6,680 (sphere)
// Between 640 and 1,024 groups 16 waves and 8 differ by no more than 6 %.
static int vjp_split(int ngroups)
{
    return ngroups <= 640 ? 16 : ngroups <= 5120 ? 8 : ngroups <= 10240 ? 4 : 1;
}

template <class T> static bool dmalloc(T **p, int64_t count)
{
    return hipMalloc(reinterpret_cast<void **>(p), sizeof(T) * (size_t)(count > 0 ? count : 1)) == hipSuccess;
}

bool alloc_vjp_scratch(nbx_context *c)
{
    const int64_t ids = (int64_t)c->n_max + c->m_max + 8;  // node ids: bodies, then n + a record
    const int64_t ngroups = ((int64_t)c->n_max + 63) / 64;
    // bins of the ids: as small as kLogBins of them allow (more workgroups, less LDS each)
    c->adj_shift = 0;
    for (int sh = 10; sh <= 12 && !c->adj_shift; ++sh)
        if (((ids - 1) >> sh) + 1 <= kLogBins) c->adj_shift = sh;
    const bool binned = c->adj_shift != 0;
    c->adj_nbins = binned ? (int)(((ids - 1) >> c->adj_shift) + 1) : 0;
    // one part of the log per counter: chunk grants from a single one are serialised
    c->adj_nlogs = !binned ? 1 : c->n_max >= 65536 ? kLogParts : c->n_max >= 8192 ? 16 : 4;
    // about 60 records per body at theta = 0.5, and a started chunk per wave; a full log falls back to
    // atomics (grants past the end count on: they must not pass 2^31 either)
    const int64_t waves = std::max<int64_t>(ngroups, std::min<int64_t>(16 * ngroups, 65536));
    const int64_t started = (int64_t)(binned ? kChunkBinned : kChunkSorted) * (waves + kLogParts);
    int64_t cap = 64 * (int64_t)c->n_max + started;
    cap = std::min<int64_t>(cap, INT32_MAX - started - (int64_t)kLogTileMax * c->adj_nlogs);
    c->adj_tile = cap >= kLogTileLine ? kLogTileMax : kLogTile;
    const int64_t sub = ((cap + c->adj_nlogs - 1) / c->adj_nlogs + c->adj_tile - 1) / c->adj_tile * c->adj_tile;
    c->adj_subcap = (int)sub;
    cap = sub * c->adj_nlogs;
    bool ok = dmalloc(&c->adj_tgt, 4 * ids) && dmalloc(&c->adj_ab, 4 * ((int64_t)c->m_max + 8)) &&
              dmalloc(&c->adj_own, c->n_max) && dmalloc(&c->adj_next, kLogLine * (kLogParts + 1)) &&
              dmalloc(&c->adj_log_id, cap) && dmalloc(&c->adj_log_val, cap) && dmalloc(&c->adj_sk, cap);
    if (binned) {
        ok = ok && dmalloc(&c->adj_sval, cap) && dmalloc(&c->adj_tab, cap / c->adj_tile * (c->adj_nbins + 1)) &&
             dmalloc(&c->adj_items, c->adj_nbins + kLogItems + 64);
    } else {
        const bool even = sort_passes((int64_t)c->n_max + c->m_max) % 2 == 0;
        const int64_t tiles = (cap + kSortTile - 1) / kSortTile;
        ok = ok && dmalloc(&c->adj_sv, cap) && dmalloc(&c->adj_tv, cap) && (!even || dmalloc(&c->adj_tk, cap)) &&
             dmalloc(&c->adj_hist, tiles * kRadix + kRadix);
    }
    if (!ok) {
        free_vjp_scratch(c);
        return false;
    }
    c->adj_cap = cap;
    return true;
}

void free_vjp_scratch(nbx_context *c)
{
    void *p[] = {c->adj_tgt, c->adj_ab, c->adj_own, c->adj_next, c->adj_log_id, c->adj_log_val, c->adj_sk, c->adj_sv,
                 c->adj_tv, c->adj_tk, c->adj_hist, c->adj_sval, c->adj_tab, c->adj_items};
    for (void *q : p)
        if (q) hipFree(q);
    c->adj_tgt = c->adj_ab = nullptr;
    c->adj_own = c->adj_sval = c->adj_log_val = nullptr;
    c->adj_next = nullptr;
    c->adj_log_id = c->adj_sk = c->adj_tk = nullptr;
    c->adj_sv = c->adj_tv = nullptr;
    c->adj_hist = nullptr;
    c->adj_tab = nullptr;
    c->adj_items = nullptr;
    c->adj_cap = 0;
}

template <bool SOFT>
static void launch_vjp_walk(const VjpArgs &v, const nbx_context *c, int ngroups, float eps2, hipStream_t s)
{
    const int S = vjp_split(ngroups);
    if (S >= 16) vjp_split_kernel<16, SOFT><<<ngroups, 1024, 0, s>>>(v, c->fnode, c->fmeta, eps2, c->st);
    else if (S >= 8) vjp_split_kernel<8, SOFT><<<ngroups, 512, 0, s>>>(v, c->fnode, c->fmeta, eps2, c->st);
    else if (S >= 4) vjp_split_kernel<4, SOFT><<<ngroups, 256, 0, s>>>(v, c->fnode, c->fmeta, eps2, c->st);
    else vjp_kernel<2, SOFT><<<(ngroups + 1) / 2, 128, 0, s>>>(v, ngroups, c->fnode, c->fmeta, eps2, c->st);
}

template <int SHIFT>
static void launch_bins(const nbx_context *c, int64_t ntgt, hipStream_t s)
{
    log_bins_kernel<SHIFT><<<c->adj_nbins + 2 * kLogItems, 512, 0, s>>>(c->adj_sk, c->adj_sval, c->adj_tab, c->adj_next, c->adj_nlogs,
                                                c->adj_subcap, c->adj_tile, c->adj_nbins, c->adj_next + kLogLine * kLogParts, c->adj_items,
                                                ntgt, c->adj_tgt);
}

void launch_vjp(nbx_context *c, hipStream_t s, const float *ux, const float *uy, const float *uz, float *gx,
                float *gy, float *gz, float *gm, float g)
{
    const int n = c->n;
    if (n <= 0) return;
    if (frame_layout_stale(c)) launch_frame_layout(c, s);
    const int64_t ntgt = 4 * ((int64_t)n + c->m + 8);  // bodies, then cells by their block's first record
    vjp_clear_kernel<<<(int)std::min<int64_t>((ntgt + 255) / 256, 65536), 256, 0, s>>>(c->adj_tgt, ntgt, c->adj_next,
                                                                                     kLogLine * (kLogParts + 1));
    const bool binned = c->adj_shift != 0;
    const int passes = sort_passes((int64_t)c->n_max + c->m_max);
    VjpArgs v{};
    v.nodes4 = c->nodes4; v.perm = c->perm; v.gorder = c->gorder; v.froot4 = c->froot4; v.frootm = c->frootm;
    v.ux = ux; v.uy = uy; v.uz = uz;
    v.own = c->adj_own; v.tgt = c->adj_tgt;
    v.log_id = c->adj_log_id; v.log_val = c->adj_log_val; v.log_next = c->adj_next;
    v.err = &c->st->err;
    v.n = n; v.nlogs = c->adj_nlogs; v.subcap = c->adj_subcap;
    v.chunk = binned ? kChunkBinned : kChunkSorted;
    v.sentinel = binned ? 0xffffffffu : (uint32_t)((uint64_t(1) << (kRadixBits * passes)) - 1);
    v.G = g;
    const int ngroups = (n + 63) / 64;
    const float eps2 = layout_eps2(c->p);
    if (eps2 > 0.f) launch_vjp_walk<true>(v, c, ngroups, eps2, s);
    else launch_vjp_walk<false>(v, c, ngroups, eps2, s);
    if (binned) {
        log_tiles_kernel<<<(int)(c->adj_cap / c->adj_tile), 1024, 0, s>>>(
            c->adj_log_id, c->adj_log_val, c->adj_next, c->adj_nlogs, c->adj_subcap, c->adj_tile, c->adj_shift,
            c->adj_nbins, v.sentinel, c->adj_sk, c->adj_sval, c->adj_tab);
        log_plan_kernel<<<c->adj_nbins, 256, 0, s>>>(c->adj_tab, c->adj_next, c->adj_nlogs, c->adj_subcap,
                                                     c->adj_tile, c->adj_nbins, c->adj_next + kLogLine * kLogParts, c->adj_items);
        if (c->adj_shift == 10) launch_bins<10>(c, ntgt, s);
        else if (c->adj_shift == 11) launch_bins<11>(c, ntgt, s);
        else launch_bins<12>(c, ntgt, s);
    } else {
        log_count_kernel<<<1, 1, 0, s>>>(c->st, c->adj_next, c->adj_subcap);
        uint32_t *tk = passes % 2 ? c->adj_log_id : c->adj_tk;  // the input keys are dead after the first pass
        launch_radix_passes(c->adj_hist, s, c->adj_log_id, (int)c->adj_cap, passes, c->adj_sk, c->adj_sv, tk, c->adj_tv,
                            &c->st->log_count);
        const int64_t waves = (c->adj_cap + 64 * kReduceTiles - 1) / (64 * kReduceTiles);
        log_reduce_kernel<<<(int)std::min<int64_t>((waves + 3) / 4, 65536), 256, 0, s>>>(
            c->adj_sk, c->adj_sv, c->adj_log_val, c->st, v.sentinel, c->adj_tgt);
    }
    const int64_t nblk = c->m - n + 1;
    adj_cells_kernel<<<(int)std::min<int64_t>((nblk + 255) / 256, 65536), 256, 0, s>>>(
        n, c->index, c->pblk, c->boff, c->bsum, c->adj_tgt, c->sum64, c->adj_ab, c->st);
    adj_bodies_kernel<<<(int)std::min<int64_t>((n + 255) / 256, 65536), 256, 0, s>>>(
        n, c->perm, c->bpar, c->nodes4, c->adj_own, c->adj_tgt, c->adj_ab, gx, gy, gz, gm, c->st);
}

}  // namespace nbx
