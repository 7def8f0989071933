// k_sort.hip -- stable merge sort of (64-bit key, int32 index) pairs.
//
// Chunks of kSortChunk pairs are sorted by one workgroup each in LDS
// (chunk_sort_kernel), then runs are merged two by two, one launch per doubling
// (merge_pass_kernel), every workgroup producing kMergeTile consecutive outputs.
// Both steps take the left element of equal keys first, so the order is stable.
// A sort of n pairs is 1 + ceil(log2(n / kSortChunk)) launches, where eight radix
// passes of 8 bits were 24; up to 17 chunks are merged in one launch (rank_merge_kernel).
// Keys and permutation on one MI355X, radix -> merge:
// N = 2,000, 95 -> 16 us; 20,011, 127 -> 31; 150,001, 132 -> 71; 1,000,003, 172 -> 127;
// 4,194,304, 388 -> 285 (and its Morton keys are made on the way, 37 us less); 8.4 M by
// radix 737, 8.0 M merged 545.  Chunks of 8,192 pairs take 36 us against 29 at N = 8,192 and 131
// against 127 at 1M (one workgroup per CU instead of three), chunks of 2,048 139.
//
// Segments: the pairs of one system, or of each system of an ensemble, sorted
// by themselves (no system index in the keys): a chunk never straddles two
// segments, and merges pair up the chunks of a segment.
#include "nbx_device.h"

#include <algorithm>

namespace nbx {

constexpr int kSortItems8 = 8;                           // pairs per thread
constexpr int kChunkThreads = kSortChunk / kSortItems8;  // 512
constexpr int kMergeThreads = 256;
constexpr int kMergeTile = kMergeThreads * kSortItems8;  // 2048

// Chunk c: segment [x, y), the chunk's index z within it, system w.
__device__ inline int4 chunk_of(const int4 *__restrict__ chunks, int n, int c)
{
    return chunks ? chunks[c] : make_int4(0, n, c, 0);
}

// Position of pair i in LDS: every eighth place skipped, so that threads that read
// eight consecutive pairs each meet different banks.
__device__ inline int pad8(int i) { return i + (i >> 3); }

// Sorts the eight pairs of a thread by exchanging neighbours that are out of
// order (strictly: stable).
__device__ inline void sort8(uint64_t (&k)[8], uint32_t (&v)[8])
{
#pragma unroll
    for (int r = 0; r < 8; ++r)
#pragma unroll
        for (int i = r & 1; i + 1 < 8; i += 2) {
            const bool swap = k[i + 1] < k[i];
            const uint64_t a = swap ? k[i + 1] : k[i], b = swap ? k[i] : k[i + 1];
            const uint32_t p = swap ? v[i + 1] : v[i], q = swap ? v[i] : v[i + 1];
            k[i] = a; k[i + 1] = b;
            v[i] = p; v[i + 1] = q;
        }
}

// Eight consecutive outputs, from the d-th, of the merge of A = [a, a + na) and
// B = [b, b + nb) in LDS (keys sk, values sv, both at pad8): the split of the
// first d outputs by binary search, then eight steps.
template <class V>
__device__ inline void merge8(const uint64_t *sk, const V *sv, int a, int na, int b, int nb, int d, uint64_t (&k)[8],
                              uint32_t (&v)[8])
{
    int lo = max(0, d - nb), hi = min(d, na);
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (sk[pad8(a + mid)] <= sk[pad8(b + d - 1 - mid)]) lo = mid + 1;
        else hi = mid;
    }
    int i = a + lo, j = b + d - lo;
    const int ea = a + na, eb = b + nb;
    uint64_t ka = sk[pad8(i)], kb = sk[pad8(j)];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const bool left = j >= eb || (i < ea && ka <= kb);
        k[q] = left ? ka : kb;
        v[q] = sv[pad8(left ? i : j)];
        if (left) ++i; else ++j;
        const uint64_t x = sk[pad8(left ? i : j)];
        ka = left ? x : ka;
        kb = left ? kb : x;
    }
}

// Where a chunk's keys come from.
struct SortSource {
    const uint64_t *keys;           // KEYS
    const float *x, *y, *z, *mass;  // BODIES: Morton keys of the bodies in the extent of their system,
    const double *ext;              // also written to keys_out (input order), with (x, y, z, m) to bodies4
    uint64_t *keys_out;
    float4 *bodies4;
};

// One workgroup per chunk.  The pairs are loaded and stored in strides of the
// workgroup (coalesced) and handed to the threads, eight consecutive pairs each, through
// LDS; each thread sorts its eight, then runs of 8, 16, ... are merged in LDS.
// Bound by the LDS round trips of the merges (nine rounds of a split search and
// eight steps each, about 2 us a round, which wait on instruction issue as much as on the
// LDS: a four-way search took 24, the eight steps as a bitonic network in registers
// 28): 20 us for one chunk, 102 us for 4M bodies.
template <bool BODIES>
__global__ void __launch_bounds__(kChunkThreads) chunk_sort_kernel(SortSource src, const int4 *__restrict__ chunks,
                                                                   int n, uint64_t *__restrict__ kout,
                                                                   int32_t *__restrict__ vout,
                                                                   int32_t *__restrict__ inv)
{
    __shared__ uint64_t sk[kSortChunk + kSortChunk / 8 + 2];
    __shared__ uint16_t sv[kSortChunk + kSortChunk / 8 + 2];
    static_assert(kSortChunk <= 65536, "16-bit positions");
    const int t = threadIdx.x;
    const int4 ck = chunk_of(chunks, n, blockIdx.x);
    const int c0 = ck.x + ck.z * kSortChunk, cnt = min(kSortChunk, ck.y - c0);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int q = i * kChunkThreads + t;
        uint64_t key = ~0ull;  // past the chunk's end: last, also among equal keys
        if (q < cnt) {
            const int64_t e = c0 + q;
            if (BODIES) {
                const float x = src.x[e], y = src.y[e], z = src.z[e];
                key = morton_key(x, y, z, src.ext + 4 * ck.w);
                src.keys_out[e] = key;
                src.bodies4[e] = make_float4(x, y, z, src.mass[e]);
            } else {
                key = src.keys[e];
            }
        }
        sk[pad8(q)] = key;
    }
    __syncthreads();
    uint64_t k[8];
    uint32_t v[8];
    const bool live = 8 * t < cnt;
    if (live) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            k[i] = sk[pad8(8 * t + i)];
            v[i] = 8 * t + i;
        }
        sort8(k, v);
    }
    for (int w = 8; w < cnt; w *= 2) {
        // runs of up to 256 pairs are merged by the threads of one wave
        if (2 * w > 512) __syncthreads();
        else __builtin_amdgcn_wave_barrier();
        if (live) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                sk[pad8(8 * t + i)] = k[i];
                sv[pad8(8 * t + i)] = (uint16_t)v[i];
            }
        }
        if (2 * w > 512) __syncthreads();
        else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (live) {
            const int p = (8 * t) & ~(2 * w - 1);
            // threads past the end wrote nothing: their places still hold ~0 keys
            merge8(sk, sv, p, w, p + w, w, 8 * t - p, k, v);
        }
    }
    __syncthreads();
    if (live) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            sk[pad8(8 * t + i)] = k[i];
            sv[pad8(8 * t + i)] = (uint16_t)v[i];
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int q = i * kChunkThreads + t;
        if (q < cnt) {
            const int32_t b = c0 + sv[pad8(q)];
            kout[c0 + q] = sk[pad8(q)];
            vout[c0 + q] = b;
            if (inv) inv[b] = c0 + q;
        }
    }
}

// Steps of a split's rounds in a pass over runs of R, as powers of two of five bits each,
// the first lowest: 64 probes from a multiple of a step reach over the run, or over
// the step before.  From kMergeGrid pairs on, whose passes are bound by what they
// fetch; 0 (probes spread evenly) below: there the lines that all tiles probe at the
// same time, 16 KB apart, cost more than they save.  Sort of 64-bit keys, spread and at
// multiples (tiles in launch order): 1M pairs 126 and 133 us, 1.5M 163 and 156, 2M 182
// and 161, 4,194,304 370 and 308, 8M 728 and 595.
constexpr int kMergeGrid = 5 << 18;
static uint32_t merge_steps(int n, int64_t R)
{
    if (n < kMergeGrid) return 0;
    return R <= 64 << 6 ? 6 : R <= 64 << 11 ? 11 | 6 << 5 : R <= 64 << 17 ? 17 | 11 << 5 | 6 << 10 : 23 | 17 << 5 | 11 << 10 | 6 << 15;
}

// First i in [lo, hi] with i == hi or A[i] > B[d - 1 - i]: how many of the first d
// merged pairs come from A.  One wave, 64 probes per round, a step apart and, with
// steps, at multiples of it: from steps of 2,048 up (d is a multiple of that but
// for the last tile) the tiles of a merge probe the same lines, and the 66 lines of
// the round of 64 are the only ones that a tile fetches for itself.  Spread evenly,
// the probes fetch as much again as the pairs.
__device__ inline int merge_split(const uint64_t *__restrict__ A, const uint64_t *__restrict__ B, int na, int nb, int d,
                                  uint32_t steps, int lane)
{
    const bool grid = steps != 0;
    int lo = max(0, d - nb), hi = min(d, na);
    while (lo < hi) {
        const int step = grid ? 1 << (steps & 31) : (hi - lo + 63) >> 6;
        const int base = grid ? lo & -step : lo;
        steps >>= 5;
        const int i = max(lo, base + lane * step);
        const bool ok = i < hi && A[i] <= B[d - 1 - i];
        const int c = __popcll(__ballot(ok));  // the probes that hold are the first c
        // the answer lies past probe c - 1 and not past probe c
        const int nlo = c ? max(lo, base + (c - 1) * step) + 1 : lo;
        hi = min(hi, max(lo, base + c * step));
        lo = nlo;
    }
    return lo;
}

// Output tile `sub` of a chunk in the pass that merges runs of R into runs of 2 R.
// Bound by its round trips (the split search, the tile's load, the merge in LDS:
// 8 us) while the tiles fit the device at once, then by HBM: 22 us for 4M pairs, 100 MB (the last pass, with inv, 79).
// Large merges (steps) give each XCD consecutive tiles, whose pairs and splits share
// lines of its L2 (block b runs on XCD b mod 8): sort of 1.5M pairs 156 -> 147 us,
// 4,194,304 308 -> 285, 8M 597 -> 545.
__global__ void __launch_bounds__(kMergeThreads) merge_pass_kernel(const uint64_t *__restrict__ kin,
                                                                   const int32_t *__restrict__ vin,
                                                                   const int4 *__restrict__ chunks, int n, int R,
                                                                   uint32_t steps, int ntiles,
                                                                   uint64_t *__restrict__ kout,
                                                                   int32_t *__restrict__ vout,
                                                                   int32_t *__restrict__ inv)
{
    constexpr int kSub = kSortChunk / kMergeTile;
    __shared__ uint64_t sk[kMergeTile + kMergeTile / 8 + 2];
    __shared__ int32_t sv[kMergeTile + kMergeTile / 8 + 2];
    __shared__ int s_split[2];
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int b = blockIdx.x;
    const int tile = steps ? (b & 7) * (int)(gridDim.x >> 3) + (b >> 3) : b;
    if (tile >= ntiles) return;
    const int4 ck = chunk_of(chunks, n, tile / kSub);
    const int o0 = ck.x + ck.z * kSortChunk + tile % kSub * kMergeTile;
    if (o0 >= ck.y) return;
    const int cnt = min(kMergeTile, ck.y - o0);
    const int64_t rel = o0 - ck.x;
    const int p = ck.x + (int)(rel / (2 * (int64_t)R) * (2 * (int64_t)R));
    const int na = min(R, ck.y - p), nb = (int)min((int64_t)R, max((int64_t)0, (int64_t)ck.y - p - R));
    const uint64_t *A = kin + p, *B = kin + p + na;
    if (wave < 2) {
        const int i = merge_split(A, B, na, nb, o0 - p + (wave ? cnt : 0), steps, lane);
        if (lane == 0) s_split[wave] = i;
    }
    __syncthreads();
    const int a0 = s_split[0], ca = s_split[1] - a0, b0 = o0 - p - a0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int q = i * kMergeThreads + t;
        if (q < cnt) {
            const int64_t e = q < ca ? p + a0 + q : p + na + b0 + (q - ca);
            sk[pad8(q)] = kin[e];
            sv[pad8(q)] = vin[e];
        }
    }
    __syncthreads();
    uint64_t k[8];
    uint32_t v[8];
    const bool live = 8 * t < cnt;
    if (live) merge8(sk, sv, 0, ca, ca, cnt - ca, 8 * t, k, v);
    __syncthreads();
    if (live) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            sk[pad8(8 * t + i)] = k[i];
            sv[pad8(8 * t + i)] = (int32_t)v[i];
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int q = i * kMergeThreads + t;
        if (q < cnt) {
            const int32_t b = sv[pad8(q)];
            kout[o0 + q] = sk[pad8(q)];
            vout[o0 + q] = b;
            if (inv) inv[b] = o0 + q;
        }
    }
}

// All merges in one launch, for few pairs in segments of few chunks: a pair's place
// is its position in its own chunk plus, for every other chunk of the segment, the
// number of its keys that come before (in an earlier chunk equal keys too).  Every 64th key
// of every chunk is staged in LDS.  The 64 consecutive pairs of a wave bracket each
// other: the places of the first and the last in a chunk are found by two ballots over
// 64 keys each, and the others search between them, four chunks side by side.  Bound by
// the chain of loads, about 7 us per four chunks, where each doubling of the runs costs a
// launch of 8 us; every wave meets every chunk, so the work grows with the square of the
// chunks, and a last chunk that is not full takes longer (a sixth of it filled, below).  Sort of
// n pairs, merge passes and this, the last chunk full and not: 2 chunks, 29.8 and 29.1 us, 28.6
// and 30.4; 4 chunks, 37.6 and 30.0, 37.4 and 31.2; 12 chunks, 53.5 and 40.3, 53.6 and 46.3;
// 16 chunks, 53.8 and 45.9, 53.8 and 54.2; 17 chunks, 60.9 and 48.7, 60.3 and 56.9; 18 chunks,
// 61.4 and 53.8, 61.7 and 62.4; 22 chunks, 62.0 and 60.3, 61.9 and 71.2; 26 chunks, 62.7 and
// 66.4, 62.1 and 78.2.  The line
// lies below the first count from which on a chunk that is not full only loses.  An ensemble of
// 7.5M pairs in chunks by at most 16, 419 and 673.
constexpr int kRankThreads = 256, kRankWidth = 4;
constexpr int kRankChunks = 17, kRankPairs = 1 << 17;

__device__ inline bool comes_before(uint64_t q, uint64_t k, bool earlier) { return q < k || (earlier && q == k); }
__device__ inline uint64_t lane_key(uint64_t k, int lane)
{
    return (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(k >> 32), lane) << 32 |
           (uint32_t)__builtin_amdgcn_readlane((int)k, lane);
}

__global__ void __launch_bounds__(kRankThreads) rank_merge_kernel(const uint64_t *__restrict__ kin,
                                                                  const int32_t *__restrict__ vin,
                                                                  const int4 *__restrict__ chunks, int n,
                                                                  uint64_t *__restrict__ kout,
                                                                  int32_t *__restrict__ vout,
                                                                  int32_t *__restrict__ inv)
{
    constexpr int kSub = kSortChunk / kRankThreads, kEach = kSortChunk / 64;
    __shared__ uint64_t s_key[kRankChunks * kEach];
    const int4 ck = chunk_of(chunks, n, blockIdx.x / kSub);
    const int lane = threadIdx.x & 63;
    const int own = (int)(blockIdx.x % kSub) * kRankThreads + (int)threadIdx.x;
    const int len = ck.y - ck.x, z = ck.z, e = z * kSortChunk + own;
    if (e - (int)threadIdx.x >= len) return;  // the workgroup as a whole
    const int nc = (len + kSortChunk - 1) / kSortChunk;
    const uint64_t *seg = kin + ck.x;
    const uint64_t k = seg[min(e, len - 1)];
    for (int i = threadIdx.x; i < nc * kEach && i * 64 < len; i += kRankThreads) s_key[i] = seg[64 * i];
    __syncthreads();
    if (e - lane >= len) return;
    const uint64_t kf = lane_key(k, 0), kl = lane_key(k, 63);
    int to = ck.x + own;
    for (int i = 0; i < nc - 1; i += kRankWidth) {
        int from[kRankWidth], lo[kRankWidth], hi[kRankWidth], cf[kRankWidth], cl[kRankWidth], have[kRankWidth];
        bool earlier[kRankWidth];
        uint64_t q[kRankWidth], r[kRankWidth];
#pragma unroll
        for (int u = 0; u < kRankWidth; ++u) {
            const int o = min(i + u, nc - 2), c = o + (o >= z);
            earlier[u] = c < z;
            from[u] = c * kSortChunk;
            have[u] = i + u < nc - 1 ? min(kSortChunk, len - from[u]) : 0;
            q[u] = s_key[c * kEach + lane];
        }
#pragma unroll
        for (int u = 0; u < kRankWidth; ++u) {
            const bool in = lane * 64 < have[u];
            cf[u] = __popcll(__ballot(in && comes_before(q[u], kf, earlier[u])));
            cl[u] = __popcll(__ballot(in && comes_before(q[u], kl, earlier[u])));
            // the place lies past sample c - 1, and not past sample c
            q[u] = seg[from[u] + min(64 * max(cf[u] - 1, 0) + lane, max(have[u] - 1, 0))];
            r[u] = seg[from[u] + min(64 * max(cl[u] - 1, 0) + lane, max(have[u] - 1, 0))];
        }
        int width = 0;
#pragma unroll
        for (int u = 0; u < kRankWidth; ++u) {
            const int bf = 64 * (cf[u] - 1), bl = 64 * (cl[u] - 1);
            const int pf = __popcll(__ballot(bf + lane < have[u] && comes_before(q[u], kf, earlier[u])));
            const int pl = __popcll(__ballot(bl + lane < have[u] && comes_before(r[u], kl, earlier[u])));
            lo[u] = cf[u] ? bf + pf : 0;
            hi[u] = cl[u] ? bl + pl : 0;
            width = max(width, hi[u] - lo[u]);
        }
        for (int w = width; w > 0; w >>= 1) {  // an interval of w halves to w / 2 at most
#pragma unroll
            for (int u = 0; u < kRankWidth; ++u) q[u] = seg[from[u] + min((lo[u] + hi[u]) >> 1, max(have[u] - 1, 0))];
#pragma unroll
            for (int u = 0; u < kRankWidth; ++u) {
                const int mid = (lo[u] + hi[u]) >> 1;
                const bool up = lo[u] < hi[u] && comes_before(q[u], k, earlier[u]);
                hi[u] = up ? hi[u] : mid;
                lo[u] = up ? mid + 1 : lo[u];
            }
        }
#pragma unroll
        for (int u = 0; u < kRankWidth; ++u) to += lo[u];
    }
    if (e < len) {
        const int32_t v = vin[ck.x + e];
        kout[to] = k;
        vout[to] = v;
        if (inv) inv[v] = to;
    }
}

// The chunk sort into whichever buffers make the last pass end in keys_out / perm_out, then the passes.
template <bool BODIES>
static void sort_pairs(const SortSource &src, const SortSegs &g, uint64_t *keys_out, int32_t *perm_out, uint64_t *tmp_k,
                       int32_t *tmp_v, int32_t *inv_out, hipStream_t s)
{
    if (g.n <= 0) return;
    int passes = 0;
    while (((int64_t)kSortChunk << passes) < g.longest) ++passes;
    if (passes > 0 && g.longest <= kRankChunks * kSortChunk && g.n <= kRankPairs) {
        chunk_sort_kernel<BODIES><<<g.nchunks, kChunkThreads, 0, s>>>(src, g.chunks, g.n, tmp_k, tmp_v, nullptr);
        rank_merge_kernel<<<g.nchunks * (kSortChunk / kRankThreads), kRankThreads, 0, s>>>(tmp_k, tmp_v, g.chunks, g.n,
                                                                                        keys_out, perm_out, inv_out);
        return;
    }
    uint64_t *k = passes % 2 ? tmp_k : keys_out, *k2 = passes % 2 ? keys_out : tmp_k;
    int32_t *v = passes % 2 ? tmp_v : perm_out, *v2 = passes % 2 ? perm_out : tmp_v;
    chunk_sort_kernel<BODIES><<<g.nchunks, kChunkThreads, 0, s>>>(src, g.chunks, g.n, k, v, passes ? nullptr : inv_out);
    for (int p = 0; p < passes; ++p) {
        const int ntiles = g.nchunks * (kSortChunk / kMergeTile);
        merge_pass_kernel<<<(ntiles + 7) / 8 * 8, kMergeThreads, 0, s>>>(
            k, v, g.chunks, g.n, kSortChunk << p, merge_steps(g.n, (int64_t)kSortChunk << p), ntiles, k2, v2,
            p == passes - 1 ? inv_out : nullptr);
        std::swap(k, k2);
        std::swap(v, v2);
    }
}

void launch_sort_keys(const SortSegs &g, const uint64_t *keys_in, uint64_t *keys_out, int32_t *perm_out,
                      uint64_t *tmp_k, int32_t *tmp_v, int32_t *inv_out, hipStream_t s)
{
    SortSource src{};
    src.keys = keys_in;
    sort_pairs<false>(src, g, keys_out, perm_out, tmp_k, tmp_v, inv_out, s);
}

void launch_sort_bodies(const SortSegs &g, const float *x, const float *y, const float *z, const float *mass,
                        const double *ext, uint64_t *keys, float4 *bodies4, uint64_t *keys_out, int32_t *perm_out,
                        uint64_t *tmp_k, int32_t *tmp_v, int32_t *inv_out, hipStream_t s)
{
    SortSource src{nullptr, x, y, z, mass, ext, keys, bodies4};
    sort_pairs<true>(src, g, keys_out, perm_out, tmp_k, tmp_v, inv_out, s);
}

void launch_batch_sort(nbx_batch *b, hipStream_t s)
{
    const SortSegs g{b->sort_chunks, b->nsort, b->N, b->longest};
    launch_sort_bodies(g, b->x, b->y, b->z, b->mass, b->ext, b->keys, b->bodies4, b->skeys, b->perm, b->kbuf, b->vbuf,
                       b->pos, s);
}

}  // namespace nbx
