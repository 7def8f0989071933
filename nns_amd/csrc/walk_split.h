// walk_split.h -- one group's tree walk shared by the S waves of a workgroup.
//
// A walk by one wave is a chain of several hundred frames, each a dependent
// trip to the L2, so a launch with few groups waits for its longest chain
// however idle the chip is.  Here the S waves of a workgroup hold the same 64
// bodies (lane l of every wave is body l) and walk the group's frames S at a
// time: in each round wave w takes the w-th frame from the top of a stack in
// LDS, and the frames it opens go to its own staging slots; one barrier ends the
// round.  Which wave walks a frame, and in which order, follows from the tree
// alone, so the sums of every wave, and their total in wave order, are the same
// on every run.
//
// A round starts with the counts of the staged frames: their running sum (DPP,
// S <= 16 lanes of one row) names the frame each wave takes (staged frames in
// wave order first, then the stack) and, when more than S are staged, the stack
// slots of the rest, which their owners copy while the frames' blocks are being
// fetched (the staging slots are double-buffered, so the copies need no barrier
// of their own).
//
// Size of the stack: it stays sorted by depth, deepest on top (wave 0 takes the
// deepest frame, staged frames are taken in wave order, and the rest goes to the
// stack in that order from the top).  Frames of depth l + 1 are pushed only by
// frames of depth l, which are taken only when every deeper frame is taken in
// the same round, so at most 8 S of each depth exist; depths run to kKeyLevels.
// A walk that would pass the bound all the same stops and says so.
#pragma once

#include "nbx_device.h"

namespace nbx {

constexpr int kSplitMax = 16;  // waves of a workgroup at most (one DPP row of counts)

template <int S>
struct SplitStack {
    static constexpr int kCap = 8 * S * kKeyLevels;
    uint4 stk[kCap];
    uint4 stage[2][S][8];
    int cnt[2][S];
};

// Inclusive sum over the first S lanes of a row of 16.
template <int S>
static __device__ inline int row_inclusive_sum(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, true);  // row_shr:1
    if (S > 2) v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, true);  // row_shr:2
    if (S > 4) v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, true);  // row_shr:4
    if (S > 8) v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, true);  // row_shr:8
    return v;
}

// Walks every frame below `root` (walked itself when open; both the same in all
// S waves).  frame(e, out) walks the frame of entry *e = {tag, tag, mask} with the
// calling wave, writes the frames it opens to out[0 .. 8) and returns their
// number.  Returns false (in every wave) if the stack bound was passed.  All
// threads of the workgroup call it.
template <int S, class F>
static __device__ __forceinline__ bool split_walk(SplitStack<S> &L, int wave, int lane, uint4 root, bool open, F frame)
{
    static_assert(S >= 2 && S <= kSplitMax, "waves of a workgroup");
    int sp = 0, P = 0;
    if (threadIdx.x < S) L.cnt[0][threadIdx.x] = threadIdx.x == 0 && open ? 1 : 0;
    if (threadIdx.x == 0) L.stage[0][0][0] = root;
    __syncthreads();
    for (;;) {
        const int c = L.cnt[P][lane & (S - 1)];  // lanes past S repeat the counts
        const int inc = row_inclusive_sum<S>(c);
        const int tot = __builtin_amdgcn_readlane(inc, S - 1);
        const int avail = tot + sp;
        if (avail == 0) return true;
        if (tot > S) {  // the staged frames that no wave takes in this round
            const int mine = __builtin_amdgcn_readlane(c, wave), e = __builtin_amdgcn_readlane(inc, wave) - mine + lane;
            if (lane < mine && e >= S) L.stk[sp + tot - 1 - e] = L.stage[P][wave][lane];
        }
        int pushed = 0;
        if (wave < avail) {
            const uint4 *e;
            if (wave < tot) {
                const int v = __ffsll((unsigned long long)__ballot(inc > wave)) - 1;
                e = &L.stage[P][v][wave - __builtin_amdgcn_readlane(inc, v) + __builtin_amdgcn_readlane(c, v)];
            } else {
                e = &L.stk[sp - 1 - (wave - tot)];
            }
            pushed = frame(e, L.stage[P ^ 1][wave]);
        }
        if (lane == 0) L.cnt[P ^ 1][wave] = pushed;
        sp = tot >= S ? sp + tot - S : max(0, sp + tot - S);
        if (sp + 8 * S > SplitStack<S>::kCap) return false;
        P ^= 1;
        __syncthreads();
    }
}

// A frame's block: eight records from the first (`at`: bytes of the records before it
// in fnode, the tag without its count), every load issued before the first use (three
// scalar loads of 64 bytes, one wait).
static __device__ __forceinline__ void load_block(const float4 *__restrict__ fnode, const int2 *__restrict__ fmeta,
                                                  unsigned at, float4 (&q)[8], int2 (&d)[8])
{
    const float4 *bq = reinterpret_cast<const float4 *>(reinterpret_cast<const char *>(fnode) + at);
    const int2 *bd = reinterpret_cast<const int2 *>(reinterpret_cast<const char *>(fmeta) + (at >> 1));
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        q[j] = bq[j];
        d[j] = bd[j];
    }
    asm volatile("" ::"s"(q[0].x), "s"(q[0].y), "s"(q[0].z), "s"(q[0].w), "s"(q[1].x), "s"(q[1].y), "s"(q[1].z),
                 "s"(q[1].w), "s"(q[2].x), "s"(q[2].y), "s"(q[2].z), "s"(q[2].w), "s"(q[3].x), "s"(q[3].y),
                 "s"(q[3].z), "s"(q[3].w));
    asm volatile("" ::"s"(q[4].x), "s"(q[4].y), "s"(q[4].z), "s"(q[4].w), "s"(q[5].x), "s"(q[5].y), "s"(q[5].z),
                 "s"(q[5].w), "s"(q[6].x), "s"(q[6].y), "s"(q[6].z), "s"(q[6].w), "s"(q[7].x), "s"(q[7].y),
                 "s"(q[7].z), "s"(q[7].w));
    asm volatile("" ::"s"(d[0].x), "s"(d[0].y), "s"(d[1].x), "s"(d[1].y), "s"(d[2].x), "s"(d[2].y), "s"(d[3].x),
                 "s"(d[3].y), "s"(d[4].x), "s"(d[4].y), "s"(d[5].x), "s"(d[5].y), "s"(d[6].x), "s"(d[6].y),
                 "s"(d[7].x), "s"(d[7].y));
}

}  // namespace nbx
