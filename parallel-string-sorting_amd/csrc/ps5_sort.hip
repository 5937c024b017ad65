// ps5_sort.hip -- pS5 string sample sort on MI355X (gfx950): HIP kernels and
// the host orchestration behind the C ABI in include/ps5_mi355x.h.
//
// Reference algorithm (paths relative to the reference checkout):
//   SampleSortStep sample/count/distribute  src/parallel/bingmann-parallel_sample_sort.hpp:1264-1611
//   splitter tree classify                   src/sequential/bingmann-sample_sortBTC.hpp:45-72,297-399
//   bucket recursion rules                   src/parallel/bingmann-parallel_sample_sort.hpp:1492-1584
//   bucket-boundary LCPs                     src/parallel/bingmann-parallel_sample_sort.hpp:311-396
//   LCP insertion sort base case             src/sequential/bingmann-lcp_inssort.hpp:36-187
//   key extraction                           src/tools/stringset.hpp:201-231
// The GPU formulation keeps the reference's outputs but reorganises the work
// breadth-first: every round handles all segments at one 8-byte depth, every
// pass is a kernel over a device-side work list, and buckets small enough for
// LDS are finished by one workgroup without another trip through HBM.
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "ps5_device.hpp"
#include "ps5_internal.hpp"
#include "ps5_kernels.hpp"
#include "../../include/ps5_mi355x.h"

using namespace ps5;

// ===========================================================================
// kernels
// ===========================================================================

// First 8 characters of every string, in input order (the LCP merge's keys).
__global__ __launch_bounds__(kWG) void k_init(Bufs B, key64* key, uint32_t n)
{
    const uint32_t i = blockIdx.x * kWG + tid_x();
    if (i >= n) return;
    key[i] = load_key(B.arena, B.alen, str_off(B, i));
}

// Reset counters and place the root item.
__global__ void k_setup(uint32_t* cnt, Item* list, int c_index, uint32_t n)
{
    if (tid_x() < C_NCNT) cnt[tid_x()] = 0;
    __syncthreads();
    if (tid_x() == 0) {
        list[0] = Item{ 0u, n, 0u, F_IDENT, 0u, 0u };
        cnt[c_index] = 1;
    }
}

// The roots of a batch, staged by kind in mapped host memory: the lists and
// the counters in one launch.
constexpr int kRootKinds = kBlkClasses + 2;      // tiny, blocks by size class, large
struct RootLists {
    const Item* src;                 // all roots, kind by kind
    Item* dst[kRootKinds];
    uint32_t count[kRootKinds];
    int counter[kRootKinds];
};
__global__ __launch_bounds__(kWG) void k_roots(RootLists R, uint32_t* cnt)
{
    if (blockIdx.x == 0) {
        if (tid_x() < C_NCNT) cnt[tid_x()] = 0;
        __syncthreads();
        if (tid_x() == 0) {
#pragma unroll
            for (int k = 0; k < kRootKinds; ++k) cnt[R.counter[k]] = R.count[k];
        }
    }
    uint32_t first = 0;
#pragma unroll
    for (int k = 0; k < kRootKinds; ++k) {
        for (uint32_t i = blockIdx.x * kWG + tid_x(); i < R.count[k]; i += gridDim.x * kWG) R.dst[k][i] = R.src[first + i];
        first += R.count[k];
    }
}

// Counters and the first kPeek items of a work list in one buffer, so that a
// single copy brings both to the host: out[0, C_NCNT) = counters, then
// min(cnt[ci], kPeek) items from byte kStageHead on.
constexpr uint32_t kPeek = 2048;
constexpr uint32_t kStageHead = 128;
constexpr uint32_t kStageSeq = kStageHead - 4;    // the copy's sequence number, written last
static_assert(C_NCNT * 4 <= kStageSeq, "counters must fit the stage head");
// Copy the counters and the head of a list into mapped host memory, then
// publish `seq`: every thread makes its stores visible to the host first, so
// a host that reads seq (acquire) reads the whole copy.  The stream runs
// k_stage after everything enqueued before it, so seq also says that all of
// that work is complete.
__global__ __launch_bounds__(kWG) void k_stage(const uint32_t* cnt, const Item* list, int ci, unsigned char* out,
                                               uint32_t seq)
{
    if (tid_x() < C_NCNT) reinterpret_cast<uint32_t*>(out)[tid_x()] = cnt[tid_x()];
    if (list) {
        const uint32_t nl = min(cnt[ci], kPeek);
        Item* dst = reinterpret_cast<Item*>(out + kStageHead);
        for (uint32_t i = tid_x(); i < nl; i += kWG) dst[i] = list[i];
    }
    __threadfence_system();
    __syncthreads();
    if (tid_x() == 0)
        __hip_atomic_store(reinterpret_cast<uint32_t*>(out + kStageSeq), seq, __ATOMIC_RELEASE,
                           __HIP_MEMORY_SCOPE_SYSTEM);
}

// copy 8-byte words of a level plan from mapped host memory to the device:
// the header with the descriptors, the table of chunks, the table of groups
struct FetchArgs {
    const uint64_t* src[3];
    uint64_t* dst[3];
    uint64_t words[3];
};
__device__ __forceinline__ void fetch_plan(const FetchArgs& F)
{
    const uint64_t stride = (uint64_t)gridDim.x * kWG;
#pragma unroll
    for (int k = 0; k < 3; ++k)
        for (uint64_t i = (uint64_t)blockIdx.x * kWG + tid_x(); i < F.words[k]; i += stride) F.dst[k][i] = F.src[k][i];
}

__global__ __launch_bounds__(kWG) void k_fetch(FetchArgs F)
{
    fetch_plan(F);
}

// The same for the root level of a single root planned on the host, the
// sort's first kernel: its first workgroup also does k_setup's work
// (counters, the root item), one launch fewer before the root level.
__global__ __launch_bounds__(kWG) void k_root_fetch(FetchArgs F, uint32_t* cnt, Item* list, uint32_t n)
{
    if (blockIdx.x == 0) {
        if (tid_x() < C_NCNT) cnt[tid_x()] = 0;
        __syncthreads();
        if (tid_x() == 0) {
            list[0] = Item{ 0u, n, 0u, F_IDENT, 0u, 0u };
            cnt[C_LROUND] = 1;
        }
    }
    fetch_plan(F);
}

// zero the counters whose bit is set in `mask`
__global__ void k_reset(uint32_t* cnt, uint32_t mask)
{
    const int t = tid_x();
    if (t < C_NCNT && ((mask >> t) & 1u)) cnt[t] = 0;
}

// the leaves listed so far are finished (device-driven levels, round parity rp)
__global__ void k_leaves_done(uint32_t* cnt, int rp)
{
    if (tid_x() == 0) {
        cnt[C_TDONE] = cnt[C_TINY + rp];
        cnt[C_RDONE] = cnt[C_RUN + rp];
    }
}

// ---- multi-workgroup sample-sort step (segments > kBlkT) -------------------

// ---- device-planned levels ---------------------------------------------------

// Treebits of a multi-workgroup step on m strings (device copy of the host's
// large_treebits): the fewest levels of at most maxbits that bring buckets
// down to about `target` strings, the fan-out spread evenly over them.
__device__ __forceinline__ uint32_t dev_treebits(uint32_t m, uint32_t target, uint32_t maxbits)
{
    const double need = log2(fmax(2.0, (double)m / target));
    const int levels = max(1, (int)ceil(need / maxbits));
    const int k = (int)ceil(need / levels);
    return (uint32_t)max(1, min((int)maxbits, k));
}

struct PlanArgs {
    const Item* list;        // the level's large segments
    int ci;                  // their counter
    uint32_t cap_large;      // capacity of that list
    unsigned char* plan;     // header, descriptors, tables (at tiles_off and groups_off)
    uint64_t tiles_off, tiles_cap, groups_off, groups_cap, hist_cap, gsum_cap;
    uint32_t leaf_target, max_treebits, max_oversample;
    uint32_t chunk_max, chunk_max_root, min_tiles;    // chunk shapes (ps5_ctx_set_shape)
    uint32_t kmax;           // bound of the level's launches (treebits are clamped to it)
    int done_rp;             // >= 0: mark the blocks of round parity done_rp listed so far as sorted
};

// Plan one level on the device (one workgroup of kBigWG threads): the same
// descriptors, tables and totals that the host's large_step computes
// from a read-back list.  A level that does not fit the buffers is flagged
// (ERR_CAP) and planned empty.
__global__ __launch_bounds__(kBigWG) void k_plan(PlanArgs A, uint32_t* cnt)
{
    __shared__ uint32_t s_tmp[4 * kBigWaves];
    __shared__ uint32_t s_tb[kBigWG], s_gb[kBigWG];   // chunk and group offsets of a block of segments, for the tables
    __shared__ unsigned long long s_tot;
    __shared__ uint32_t s_ident, s_kmax;
    LevelHdr* hdr = reinterpret_cast<LevelHdr*>(A.plan);
    LargeDesc* desc = reinterpret_cast<LargeDesc*>(A.plan + sizeof(LevelHdr));
    TileRef* tiles = reinterpret_cast<TileRef*>(A.plan + A.tiles_off);
    TileRef* groups = reinterpret_cast<TileRef*>(A.plan + A.groups_off);
    const uint32_t tid = tid_x();
    if (A.done_rp >= 0 && tid < kBlkClasses) cnt[C_BDONE + tid] = cnt[C_BLOCK + 2 * tid + A.done_rp];
    uint32_t nl = cnt[A.ci];
    if (nl > A.cap_large) {      // (an overflow of the list has been flagged)
        nl = 0;
        if (tid == 0) flag_error(cnt, ERR_CAP);
    }
    if (tid == 0) {
        s_tot = 0;
        s_ident = 1;
        s_kmax = 1;
    }
    __syncthreads();
    unsigned long long tot = 0;
    bool ident = true;
    for (uint32_t i = tid; i < nl; i += kBigWG) {
        tot += A.list[i].size;
        ident = ident && (A.list[i].flags & F_IDENT);
    }
    atomicAdd(&s_tot, tot);
    if (!ident) atomicAnd(&s_ident, 0u);
    __syncthreads();
    const uint64_t cmax = s_ident ? A.chunk_max_root : A.chunk_max;
    const uint64_t climit = min(cmax, max((uint64_t)kChunkMin, (s_tot + A.min_tiles - 1) / A.min_tiles));
    // descriptors: table, histogram and group bases are exclusive scans over
    // the segments (blocks of kBigWG with carries)
    uint32_t tcarry = 0, gcarry = 0;
    uint64_t hcarry = 0, scarry = 0;
    for (uint32_t b0 = 0; b0 < nl; b0 += kBigWG) {
        const uint32_t i = b0 + tid;
        uint32_t T = 0, G = 0, hc = 0, sc = 0;
        LargeDesc D{};
        if (i < nl) {
            D.seg = A.list[i];
            T = (uint32_t)((D.seg.size + climit - 1) / climit);
            G = hist_groups(T);
            D.nch = T;
            D.chunk = (D.seg.size + T - 1) / T;
            D.k = min(dev_treebits(D.seg.size, A.leaf_target, A.max_treebits), A.kmax);
            const uint32_t nspl = (1u << D.k) - 1;
            D.oversample = max(2u, min(A.max_oversample, (kMaxSamples / nspl) & ~1u));
            hc = (2u << D.k) * T;
            sc = (2u << D.k) * (G + 1);
            atomicMax(&s_kmax, D.k);
        }
        const uint32_t each[4] = { T, G, hc, sc };
        uint32_t ex[4], total[4];
        block_excl_scan_k<kBigWaves, 4>(each, ex, total, s_tmp);
        const uint32_t tex = ex[0], gex = ex[1], hex = ex[2], sex = ex[3];
        const uint32_t ttot = total[0], gtot = total[1], htot = total[2], stot = total[3];
        if (i < nl) {
            D.hist_base = (uint32_t)(hcarry + hex);
            D.gbase = (uint32_t)(scarry + sex);
            desc[i] = D;
        }
        // this block's entries of the two tables, written by the whole
        // workgroup (within their capacity; an overflow is flagged below):
        // entry t of the block belongs to the last segment whose offset is
        // <= t (every segment has at least one chunk and one group)
        s_tb[tid] = tex;
        s_gb[tid] = gex;
        __syncthreads();
        const uint32_t nseg = min(nl - b0, (uint32_t)kBigWG);
        auto fill = [&](TileRef* out, const uint32_t* first, uint32_t total, uint32_t carry, uint64_t cap) {
            for (uint32_t t = tid; t < total && carry + t < cap; t += kBigWG) {
                const uint32_t lo = find_run(first, nseg, t);
                out[carry + t] = TileRef{ b0 + lo, t - first[lo] };
            }
        };
        fill(tiles, s_tb, ttot, tcarry, A.tiles_cap);
        fill(groups, s_gb, gtot, gcarry, A.groups_cap);
        __syncthreads();     // the offsets are written again by the next block
        tcarry += ttot;
        gcarry += gtot;
        hcarry += htot;
        scarry += stot;
    }
    const bool fits = tcarry <= A.tiles_cap && gcarry <= A.groups_cap && hcarry <= A.hist_cap && scarry <= A.gsum_cap &&
                      hcarry <= 0xFFFFFFFFull;
    if (!fits && tid == 0) flag_error(cnt, ERR_CAP);
    if (tid == 0) *hdr = LevelHdr{ fits ? nl : 0u, fits ? tcarry : 0u, fits ? gcarry : 0u, s_kmax, { 0u, 0u, 0u, 0u } };
}

// Splitter trees of the large segments of a level, one workgroup each.
// D.oversample * nspl random keys are sorted (4-key runs per thread by a
// sorting network, then merge-path rounds in LDS); splitter i is sample
// oversample/2 + oversample*i (the reference's choice for oversample factor 2,
// bingmann-sample_sort_tree_builder.hpp:44-58) and the tree is stored in
// level order: trees[gbase + t], t = 1..nspl, followed by the splitters in
// sorted order at trees[gbase + (1 << k) + i], i < nspl.
//
// A root's samples also choose the format of its keys (KeyFmt).  Eight
// characters of a small alphabet leave many strings equal: 20 M windows of
// ACGT text have 65536 different keys, and every equal run then gathers its
// strings again.  When the samples say that a key would be shared by
// kPackRun strings or more beside its own (d equal neighbours among s sorted
// samples of n strings: 2 d n / s^2 strings for each key, one of them the
// string itself, drawn twice) and the sampled strings' first 24 characters
// form an alphabet of at most 31, the root's keys hold 21, 16 or 12 packed
// characters instead.  A character that the samples do not show is found by
// the extraction (ERR_ALPHA), which adds it to the root's alphabet in B.lut;
// no children are listed then, and the sort starts over with the alphabets
// found (B.widen; plain keys where one has more than 31 characters).  20 M
// windows of 100 characters: 1.48 ms, with an N in 10^6 characters 2.00 (4.0 when
// the whole sort started over with plain keys, 2.97 with plain keys alone).

// what the kernels of a level know of its segments' strings: buckets of the
// level before, roots with plain keys, roots that may pack theirs, or
// segments of an earlier round
constexpr int kFromRuns = 0, kRootPlain = 1, kRootPack = 2, kFromPerm = 3;

struct TreeLds {
    key64 samp[kMaxSamples + 1];      // + 1: a merge step reads the slot after the one it takes
    uint32_t alpha[8];                // the alphabet
    uint32_t dups;                    // equal neighbours among the sorted samples
    uint8_t lut[kLutBytes];           // characters seen, then the code table
};
constexpr float kPackRun = 1.0f;
constexpr uint32_t kMaxAlphabet = 31;       // five code bits

template <int SRC>
__device__ __forceinline__ void tree_of_segment(LargeDesc* Dp, uint32_t si, const Bufs& B, uint64_t seed, key64* tree,
                                                TreeLds& S)
{
    const LargeDesc D = *Dp;
    const Item seg = D.seg;
    key64* s_samp = S.samp;
    if (!item_ok(seg, B)) {
        if (tid_x() == 0) flag_error(B.cnt, ERR_BOUNDS);
        return;
    }
    const int k = (int)D.k, nspl = (1 << k) - 1, a = (int)D.oversample;
    const uint32_t ss = (uint32_t)(a * nspl);
    uint32_t P = 64;
    while (P < ss) P <<= 1;
    if (P > (uint32_t)kMaxSamples) {
        if (tid_x() == 0) flag_error(B.cnt, ERR_BOUNDS);
        return;
    }
    // every sample load is issued first (kPer consecutive samples per
    // thread), each thread sorts its kPer keys with a network, then runs are
    // merged pairwise by merge path: a co-rank search places a thread's kPer
    // outputs, then it merges them sequentially (padding ~0 sorts last; equal
    // keys need no tie order, only the splitters are kept)
    constexpr int kPer = kMaxSamples / kBigWG;
    static_assert(kMaxSamples % kBigWG == 0 && kPer == 4, "four samples per thread");
    const uint32_t o = tid_x() * kPer;
    const bool act = o < P;
    constexpr bool may_pack = SRC == kRootPack;
    if (may_pack) {     // (cleared before the merge rounds' barriers)
        if (tid_x() < kLutBytes / 4) reinterpret_cast<uint32_t*>(S.lut)[tid_x()] = 0;
        if (tid_x() == kLutBytes / 4) S.dups = 0;
    }
    auto sample = [&](uint32_t j) {
        const uint64_t h = mix64(seed ^ ((uint64_t)seg.begin << 21) ^ (uint64_t)j);
        return seg.begin + (uint32_t)(((h >> 32) * (uint64_t)seg.size) >> 32);
    };
    key64 v[kPer];
    if (SRC == kFromRuns) {
        // the samples' runs are searched in a copy of the bucket's row of
        // first positions (in LDS, before the samples go there), or of every
        // stride-th entry of it and then in the row itself
        const Runs R = runs_of(B, seg);
        constexpr uint32_t kRowMax = 2 * kMaxSamples;
        uint32_t* s_v = reinterpret_cast<uint32_t*>(s_samp);
        const uint32_t stride = (R.nch + kRowMax - 1) / kRowMax, ns = (R.nch + stride - 1) / stride;
        for (uint32_t c = tid_x(); c < ns; c += kBigWG) s_v[c] = R.V[c * stride];
        __syncthreads();
        uint32_t q[kPer];
#pragma unroll
        for (int e = 0; e < kPer; ++e) {
            const uint32_t pos = sample(min(o + e, ss - 1));
            uint32_t c = find_run(s_v, ns, pos) * stride;
            if (stride > 1) c += find_run(R.V + c, min(stride, R.nch - c), pos);     // (uniform branch)
            q[e] = R.S[c] + (pos - R.V[c]);
        }
#pragma unroll
        for (int e = 0; e < kPer; ++e) {
            const key64 x = rec_key(R.R[checked_place(B, q[e])]);
            v[e] = o + e < ss ? x : ~0ull;
        }
        __syncthreads();     // the row's copy is no longer read
    } else {
        const uint32_t depth = SRC == kFromPerm ? seg_depth(B, seg.rbeg) : 0u;
#pragma unroll
        for (int e = 0; e < kPer; ++e) {
            v[e] = ~0ull;
            if (o + e >= ss) continue;
            const uint32_t pos = sample(o + e);
            v[e] = string_key(B, SRC == kFromPerm ? B.perm[pos] : pos, depth);
        }
    }
    uint32_t fmt = 0;
    for (;;) {
        if (act) {
            constexpr int net[][2] = { { 0, 1 }, { 2, 3 }, { 0, 2 }, { 1, 3 }, { 1, 2 } };
#pragma unroll
            for (int c = 0; c < 5; ++c) {
                const key64 x = v[net[c][0]], y = v[net[c][1]];
                v[net[c][0]] = min(x, y);
                v[net[c][1]] = max(x, y);
            }
#pragma unroll
            for (int e = 0; e < kPer; ++e) s_samp[o + e] = v[e];
        }
        __syncthreads();
        for (uint32_t L = kPer; L < P; L <<= 1) {
            if (act) {
                const uint32_t a0 = (o / (2 * L)) * (2 * L), b0 = a0 + L, diag = o - a0;
                uint32_t lo = diag > L ? diag - L : 0u, hi = min(diag, L);
                while (lo < hi) {
                    const uint32_t mid = (lo + hi) >> 1;
                    if (s_samp[a0 + mid] <= s_samp[b0 + diag - 1 - mid]) lo = mid + 1;
                    else hi = mid;
                }
                // branch-free steps on byte offsets, as in the block sort: one
                // read of the consumed run's next head (unused past the run's
                // end; s_samp has one spare slot)
                const unsigned char* sbase = reinterpret_cast<const unsigned char*>(s_samp);
                uint32_t pa = (a0 + lo) * 8u, pb = (b0 + diag - lo) * 8u;
                const uint32_t ea = (a0 + L) * 8u, eb = (b0 + L) * 8u;
                key64 ka = pa < ea ? *reinterpret_cast<const key64*>(sbase + pa) : 0ull;
                key64 kb = pb < eb ? *reinterpret_cast<const key64*>(sbase + pb) : 0ull;
#pragma unroll
                for (int e = 0; e < kPer; ++e) {
                    const bool take_a = pb >= eb || (pa < ea && ka <= kb);
                    const uint32_t src = take_a ? pa : pb;
                    v[e] = take_a ? ka : kb;
                    const key64 nx = *reinterpret_cast<const key64*>(sbase + src + 8u);
                    pa += take_a ? 8u : 0u;
                    pb += take_a ? 0u : 8u;
                    ka = take_a ? nx : ka;
                    kb = take_a ? kb : nx;
                }
            }
            __syncthreads();
            if (act) {
#pragma unroll
                for (int e = 0; e < kPer; ++e) s_samp[o + e] = v[e];
            }
            __syncthreads();
        }
        if (!may_pack || fmt) break;
        uint32_t d = 0;
#pragma unroll
        for (int e = 0; e < kPer; ++e) {
            const uint32_t j = o + e;
            if (j + 1 < ss) d += s_samp[j] == s_samp[j + 1] && (s_samp[j] & 0xFFull) != 0 ? 1u : 0u;
        }
        if (d) atomicAdd(&S.dups, d);
        __syncthreads();
        const uint32_t dups = S.dups;
        if (dups < 16 || 2.0f * (float)dups * (float)seg.size < (1.0f + kPackRun) * (float)ss * (float)ss) break;     // (uniform)
        uint8_t* code_out = B.lut + (uint64_t)si * kRootCode;
        uint32_t* alpha_out = reinterpret_cast<uint32_t*>(code_out + kLutBytes);
        if (B.widen) {     // (uniform)
            if (tid_x() < kLutBytes) S.lut[tid_x()] = (uint8_t)((alpha_out[tid_x() / 32] >> (tid_x() & 31)) & 1u);
        }
        uint32_t sigma = 0;
        // (a thread's first sample alone shows most alphabets that are too
        // large; all four take 10 us)
#pragma unroll 1
        for (uint32_t part = 0; part < 2; ++part) {
            if (!B.widen && act) {
#pragma unroll 1
                for (uint32_t j = o + part; j < (part ? o + kPer : o + 1) && j < ss; ++j) {
                    const Chars24 c = load_chars24(B.arena, B.alen, str_off(B, sample(j)));
                    const uint32_t len = chars_before_nul(c);
#pragma unroll
                    for (int i = 0; i < 24; ++i)
                        if ((uint32_t)i < len) S.lut[(uint32_t)(c.w[i / 8] >> (8 * (i & 7))) & 0xFFu] = 1;
                }
            }
            __syncthreads();
            if (tid_x() < kLutBytes) {     // (whole waves)
                const uint64_t seen = __ballot(S.lut[tid_x()] != 0);
                if ((tid_x() & 31) == 0) S.alpha[tid_x() / 32] = (uint32_t)(seen >> (tid_x() & 32));
            }
            __syncthreads();
            sigma = 0;
#pragma unroll
            for (int j = 0; j < 8; ++j) sigma += (uint32_t)__popc(S.alpha[j]);
            if (B.widen || sigma > kMaxAlphabet) break;     // (uniform)
        }
        if (tid_x() < 8) alpha_out[tid_x()] = S.alpha[tid_x()];
        fmt = sigma <= 7 ? 1u : sigma <= 15 ? 2u : sigma <= kMaxAlphabet ? 3u : 0u;
        if (fmt == 0) break;     // (uniform)
        if (tid_x() < kLutBytes) {
            const uint32_t c = tid_x();
            uint32_t rank = 1;
            for (uint32_t j = 0; j < c / 32; ++j) rank += (uint32_t)__popc(S.alpha[j]);
            rank += (uint32_t)__popc(S.alpha[c / 32] & ((1u << (c & 31)) - 1));
            const uint32_t code = c == 0 ? 0u : (S.alpha[c / 32] >> (c & 31)) & 1u ? rank : 0x81u;
            S.lut[c] = (uint8_t)code;
            code_out[c] = (uint8_t)code;
        }
        __syncthreads();
        // the same samples with packed keys (a rolled loop: this code runs in
        // few workgroups, where its size would cost more than its latency)
        if (act) {
#pragma unroll 1
            for (uint32_t j = o; j < o + kPer; ++j) {
                bool bad = false;     // (the alphabet holds the samples' characters)
                s_samp[j] = j < ss ? pack_key_fmt(load_chars24(B.arena, B.alen, str_off(B, sample(j))), fmt, S.lut,
                                                  alpha_out, &bad)
                                   : ~0ull;
            }
#pragma unroll
            for (int e = 0; e < kPer; ++e) v[e] = s_samp[o + e];
        }
    }
    if (fmt && tid_x() == 0) Dp->seg.flags = seg.flags | (fmt << kFmtShift);
    const key64* sorted = s_samp;
    for (int t = tid_x() + 1; t <= nspl; t += kBigWG) tree[t] = sorted[a / 2 + a * inorder_of(t, k)];
    for (int i = tid_x(); i < nspl; i += kBigWG) tree[nspl + 1 + i] = sorted[a / 2 + a * i];
}

template <int SRC>
__global__ __launch_bounds__(kBigWG) void k_tree(Plan P, Bufs B, uint64_t seed, key64* trees)
{
    __shared__ TreeLds S;
    const uint32_t nlarge = P.hdr->nlarge;
    for (uint32_t si = blockIdx.x; si < nlarge; si += gridDim.x) {
        __syncthreads();     // the previous segment's samples are consumed
        tree_of_segment<SRC>(P.desc + si, si, B, seed, trees + P.desc[si].gbase, S);
    }
}

// Load a read-only value that every lane of the wave reads at the same
// address, through the constant address space (scalar loads).
template <typename T>
__device__ __forceinline__ T load_uniform(const T* p)
{
    static_assert(sizeof(T) % 4 == 0, "whole dwords");
    using cword = const __attribute__((address_space(4))) uint32_t;
    cword* q = (cword*)(uintptr_t)p;
    uint32_t w[sizeof(T) / 4];
#pragma unroll
    for (uint32_t i = 0; i < sizeof(T) / 4; ++i) w[i] = q[i];
    T v;
    __builtin_memcpy(&v, w, sizeof(T));
    return v;
}

// tid_x() through an opaque move: addresses derived from it are
// recomputed where they are used instead of being hoisted out of loops,
// where they would hold registers
__device__ __forceinline__ uint32_t scat_tid()
{
    uint32_t t;
    asm volatile("v_mov_b32 %0, %1" : "=v"(t) : "v"((uint32_t)threadIdx.x));
    return t;
}

// The places of a bucket's positions [v0, v0 + m) for a workgroup of NW
// waves: position v0 + p lies at p + delta[r] for the run r holding it, and r
// is the number of run starts at or before p in a bitmap, less one.  Runs
// average tens of strings, so a bit per position costs less to build and to
// read than a search per position.
template <int MAXP>
struct RunMap {
    uint32_t delta[MAXP];
    uint32_t bits[MAXP / 32];
    uint32_t pre[MAXP / 32];
    uint32_t tmp[16];
};
template <int NW, int MAXP>
__device__ __forceinline__ void map_runs(const Runs& R, uint32_t vend, uint32_t v0, uint32_t m, RunMap<MAXP>& M)
{
    constexpr uint32_t T = NW * 64;
    constexpr uint32_t W = MAXP / 32;
    static_assert(W <= T, "a thread per bitmap word");
    const uint32_t tid = scat_tid(), w = wave_id(), lane = lane_id();
    if (tid < W) M.bits[tid] = 0;
    // the run holding v0: T samples of the row, then their interval
    const uint32_t step = (R.nch + T - 1) / T;
    const uint32_t si = tid * step;
    const uint32_t le = (uint32_t)__popcll(__ballot(si < R.nch && R.V[si] <= v0));
    if (lane == 0) M.tmp[w] = le;
    __syncthreads();
    uint32_t c0 = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) c0 += M.tmp[i];
    c0 = (c0 ? c0 - 1 : 0u) * step;
    if (step > 1) {     // (uniform) every wave looks at the interval
        if (step <= 64) {
            const uint32_t c = c0 + lane;
            const uint32_t in = (uint32_t)__popcll(__ballot(lane < step && c < R.nch && R.V[c] <= v0));
            c0 += in ? in - 1 : 0u;
        } else {
            c0 += find_run(R.V + c0, min(step, R.nch - c0), v0);
        }
    }
    uint32_t base = 0;       // runs mapped so far
    for (uint32_t cb = c0;; cb += T) {
        __syncthreads();     // tmp is read (first pass: and the bitmap is cleared)
        const uint32_t c = cb + tid;
        uint32_t v = 0, nx = 0, s = 0;
        if (c < R.nch) {
            v = R.V[c];
            nx = c + 1 < R.nch ? R.V[c + 1] : vend;
            s = R.S[c];
        }
        const bool use = nx > v && nx > v0 && v < v0 + m;
        const uint64_t bal = __ballot(use);
        if (lane == 0) M.tmp[w] = (uint32_t)__popcll(bal);
        __syncthreads();
        uint32_t before = 0, all = 0;
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            const uint32_t t = M.tmp[i];
            before += i < (int)w ? t : 0u;
            all += t;
        }
        if (use) {
            const uint32_t r = base + before + (uint32_t)__popcll(bal & lanemask_lt());
            const uint32_t p = v > v0 ? v - v0 : 0u;
            if (r < MAXP) M.delta[r] = s + v0 - v;
            atomicOr(&M.bits[p >> 5], 1u << (p & 31));
        }
        base += all;
        if (cb + T >= R.nch || R.V[cb + T] >= v0 + m) break;     // (uniform)
    }
    __syncthreads();
    // exclusive prefix of the words' bit counts
    const uint32_t pc = tid < W ? (uint32_t)__popc(M.bits[tid]) : 0u;
    uint32_t x = pc;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)x, d, 64);
        if (lane >= (uint32_t)d) x += y;
    }
    if (lane == 63) M.tmp[w] = x;
    __syncthreads();
    uint32_t wp = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) wp += i < (int)w ? M.tmp[i] : 0u;
    if (tid < W) M.pre[tid] = wp + x - pc;
    __syncthreads();
}
template <int MAXP>
__device__ __forceinline__ uint32_t mapped_place(const Bufs& B, const RunMap<MAXP>& M, uint32_t p)
{
    const uint32_t below = M.bits[p >> 5] & (0xFFFFFFFFu >> (31 - (p & 31)));
    const uint32_t r = M.pre[p >> 5] + (uint32_t)__popc(below);
    return checked_place(B, p + M.delta[r ? min(r - 1, (uint32_t)MAXP - 1) : 0u]);
}

// Partition one chunk of a segment (classify, .hpp:1413-1435, and distribute,
// .hpp:1464-1490, in one pass): each wave classifies its part of the chunk
// with the splitter tree in LDS and ranks it stably (ballot matching and
// per-wave bucket counts, ranks follow input order), a scan of the counts
// places every (bucket, wave), and the records are staged in LDS in that
// order and written back in place of the chunk, 16 bytes a lane.  The chunk's
// bucket counts and starts go to its row of hist.
//
// 2 GiB of random strings, root level (reading the arena, 511 splitters):
// 0.66 ms, 4.9 TB/s of the 3.2 GB it reads and writes, against 5.5 of a plain
// copy; counting first and scattering afterwards took 0.71 + 0.50 ms.
//
// LDS: the stage (the lane-mask tables of match_bucket_lds, or the run map of
// a bucket's chunk, before that), the per-wave counts and the tree.
template <int NB>
struct PartLds {
    static constexpr uint32_t kSlots = 1u << NB;             // bucket slots per wave
    static constexpr uint32_t kStageOff = 0;                 // (+ 3 words: the image is aligned like its destination)
    static constexpr uint32_t kCntOff = (kPartStage * kRecWords + 4) * 4;
    static constexpr uint32_t kTreeOff = kCntOff + kPartWaves * kSlots * 2;
    static constexpr uint32_t kTmpOff = kTreeOff + kSlots / 2 * 8;
    static constexpr uint32_t kBytes = kTmpOff + 64;
    static constexpr int kPeerBits = NB < 8 ? NB : 8;
    static_assert(((uint32_t)kPartWaves << kPeerBits << 3) <= kCntOff, "the lane-mask tables fit the stage");
    static_assert(sizeof(RunMap<kPartMax>) <= kTmpOff, "the run map fits the stage and the counts");
    static_assert(kCntOff % 16 == 0 && kPartStage % 4 == 0, "16-byte copies");
};

template <int NB, int SRC>
__device__ __forceinline__ void part_chunk(uint32_t ti, const Plan& P, const Bufs& B, const key64* trees, bool one,
                                           unsigned char* smem)
{
    using L = PartLds<NB>;
    constexpr int kE = kPartGroups;
    constexpr uint32_t T = kPartThreads;
    uint32_t* s_rec = reinterpret_cast<uint32_t*>(smem + L::kStageOff);
    uint64_t* s_peer = reinterpret_cast<uint64_t*>(smem + L::kStageOff);
    uint16_t* s_cnt = reinterpret_cast<uint16_t*>(smem + L::kCntOff);
    key64* s_tree = reinterpret_cast<key64*>(smem + L::kTreeOff);
    uint32_t* s_tmp = reinterpret_cast<uint32_t*>(smem + L::kTmpOff);
    ti = __builtin_amdgcn_readfirstlane(ti);
    // (read-only here, the same for the workgroup)
    const TileRef tr = one ? TileRef{ 0u, ti } : load_uniform(P.tiles + ti);
    const LargeDesc D = load_uniform(P.desc + tr.seg);
    const Item seg = D.seg;
    const int k = (int)D.k;
    const uint32_t cb = tr.t * D.chunk;
    if (!item_ok(seg, B) || k + 1 > NB || tr.t >= D.nch || D.chunk > (uint32_t)kPartMax || cb >= seg.size) {   // (uniform)
        if (tid_x() == 0) flag_error(B.cnt, ERR_BOUNDS);
        return;
    }
    const uint32_t tid = scat_tid(), w = wave_id(), lane = lane_id();
    const uint32_t m = min(seg.size - cb, D.chunk);
    const uint32_t per = ((m + kPartWaves - 1) / kPartWaves + 63) & ~63u;     // positions per wave
    const uint32_t wb = w * per;
    const uint32_t nspl = (1u << k) - 1, nbs = 2u << k;
    const key64* tree = trees + D.gbase;
    const uint32_t fmt = SRC == kRootPack ? (seg.flags & kFmtMask) >> kFmtShift : 0u;
    key64 kv[kE];
    uint32_t iv[kE];        // (indices; a root's are its positions)
    // clamped positions: every load is unconditional, so all of them are in flight together
#define PS5_PART_POS(e) min(wb + (e) * 64 + lane, m - 1)
    if (SRC == kFromRuns) {
        const Runs R = runs_of(B, seg);
        RunMap<kPartMax>& M = *reinterpret_cast<RunMap<kPartMax>*>(smem);
        map_runs<kPartWaves, kPartMax>(R, seg.begin + seg.size, seg.begin + cb, m, M);
#pragma unroll
        for (int e = 0; e < kE; ++e) {
            const Rec r = R.R[mapped_place(B, M, PS5_PART_POS(e))];
            kv[e] = rec_key(r);
            iv[e] = r.id;
        }
        __syncthreads();     // the run map is read
    } else if (SRC == kFromPerm) {
        const uint32_t depth = seg_depth(B, seg.rbeg);
#pragma unroll
        for (int e = 0; e < kE; ++e) iv[e] = B.perm[seg.begin + cb + PS5_PART_POS(e)];
#pragma unroll
        for (int e = 0; e < kE; ++e) kv[e] = string_key(B, iv[e], depth);
    } else if (fmt == 0) {     // (uniform)
        uint64_t off[kE];
        if (B.offs64) {     // (uniform)
#pragma unroll
            for (int e = 0; e < kE; ++e) off[e] = B.offs64[seg.begin + cb + PS5_PART_POS(e)];
        } else {
#pragma unroll
            for (int e = 0; e < kE; ++e) off[e] = B.offs[seg.begin + cb + PS5_PART_POS(e)];
        }
#pragma unroll
        for (int e = 0; e < kE; ++e) kv[e] = load_key(B.arena, B.alen, off[e]);
    }
    for (uint32_t i = tid; i <= nspl; i += T) s_tree[i] = tree[i];
    for (uint32_t i = tid; i < kPartWaves * L::kSlots / 2; i += T) reinterpret_cast<uint32_t*>(s_cnt)[i] = 0;
    if (SRC == kRootPack && fmt) {
        // packed keys are extracted in a rolled loop, four groups at a time
        // through the wave's part of the stage: unrolled with the others they
        // would take twice the registers.  The code table sits where the
        // counts go afterwards
        uint8_t* s_lut = reinterpret_cast<uint8_t*>(s_cnt);
        constexpr int kH = 4;
        static_assert(kPartWaves * kH * 64 * 8 <= L::kCntOff && kE % kH == 0, "the groups' keys fit the stage");
        key64* s_w = reinterpret_cast<key64*>(smem + L::kStageOff) + w * kH * 64;
        __syncthreads();
        uint8_t* code = B.lut + (uint64_t)tr.seg * kRootCode;
        uint32_t* unknown = reinterpret_cast<uint32_t*>(code + kLutBytes);
        if (tid < kLutBytes) s_lut[tid] = code[tid];
        // once a character is missing, the sort starts over: the other chunks
        // only complete the alphabet, or do nothing when it is already too
        // large to pack
        if (tid == 0) {
            uint32_t over = __hip_atomic_load(&B.cnt[C_ERR], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & ERR_ALPHA;
            if (over) {
                uint32_t sigma = 0;
                for (int j = 0; j < 8; ++j)
                    sigma += (uint32_t)__popc(__hip_atomic_load(unknown + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                if (sigma > kMaxAlphabet) over = ~0u;
            }
            s_tmp[15] = over;
        }
        __syncthreads();
        if (s_tmp[15] == ~0u) return;     // (uniform)
        bool bad = false;
#pragma unroll
        for (int e0 = 0; e0 < kE; e0 += kH) {
            if ((uint32_t)e0 * 64 >= per) {     // (uniform)
#pragma unroll
                for (int j = 0; j < kH; ++j) kv[e0 + j] = 0;
                continue;
            }
#pragma unroll 2
            for (int j = 0; j < kH; ++j) {
                const uint32_t q = min(wb + (e0 + j) * 64 + lane, m - 1);
                s_w[j * 64 + lane] = pack_key_fmt(load_chars24(B.arena, B.alen, str_off(B, seg.begin + cb + q)), fmt,
                                                  s_lut, unknown, &bad);
            }
#pragma unroll
            for (int j = 0; j < kH; ++j) kv[e0 + j] = s_w[j * 64 + lane];
        }
        if (bad) flag_error(B.cnt, ERR_ALPHA);
        if (s_tmp[15]) return;     // (uniform)
        __syncthreads();     // the table is read
        if (tid < kLutBytes / 4) reinterpret_cast<uint32_t*>(s_cnt)[tid] = 0;
    }
    for (uint32_t i = tid; i < ((uint32_t)kPartWaves << L::kPeerBits); i += T) s_peer[i] = 0;
    __syncthreads();
    uint16_t* cnt_w = s_cnt + w * L::kSlots;
    uint64_t* peer = s_peer + (w << L::kPeerBits);
    const uint64_t lanebit = 1ull << lane;
    uint32_t br[kE];        // bucket << 16 | rank inside the wave's part, later the staged slot
    constexpr int kG = 4;   // groups whose descents advance together
    static_assert(kE % kG == 0, "whole batches");
#pragma unroll
    for (int e0 = 0; e0 < kE; e0 += kG) {
        if ((uint32_t)e0 * 64 >= per) {     // (uniform) nothing here in a short chunk
#pragma unroll
            for (int j = 0; j < kG; ++j) br[e0 + j] = 0;
            continue;
        }
        key64 kk[kG];
        uint32_t bv[kG];
#pragma unroll
        for (int j = 0; j < kG; ++j) kk[j] = kv[e0 + j];
        classify_keys<kG>(kk, s_tree, k, bv);
#pragma unroll
        for (int j = 0; j < kG; ++j) {
            const uint32_t p = (e0 + j) * 64 + lane;
            const bool act = p < per && wb + p < m;
            if (!act) bv[j] = L::kSlots - 1;     // (above every bucket)
            const uint64_t peers = match_bucket_lds<NB, L::kPeerBits>(bv[j], peer, lanebit);
            const uint32_t r = (uint32_t)__popcll(peers & lanemask_lt());
            const uint32_t old = cnt_w[bv[j]];
            if (act && r == 0) cnt_w[bv[j]] = (uint16_t)(old + (uint32_t)__popcll(peers));
            br[e0 + j] = (bv[j] << 16) | (old + r);
        }
    }
    __syncthreads();
    // places: a thread takes kPB neighbouring buckets, two 16-bit counts to a
    // word; the counts become the wave's first slot per bucket
    constexpr int kPB = (int)L::kSlots / (int)T > 2 ? (int)L::kSlots / (int)T : 2;
    static_assert(kPartMax < 65536, "slots fit 16 bits");
    uint32_t* s_pair = reinterpret_cast<uint32_t*>(s_cnt);
    const uint32_t pair0 = tid * (kPB / 2);
    uint32_t cnt[kPB], sum = 0;
#pragma unroll
    for (int q = 0; q < kPB / 2; ++q) {
        uint32_t run = 0;
        if (pair0 + q < nbs / 2) {
            uint32_t* col = s_pair + pair0 + q;
#pragma unroll
            for (int ww = 0; ww < kPartWaves; ++ww) {
                const uint32_t v = col[ww * (L::kSlots / 2)];
                col[ww * (L::kSlots / 2)] = run;
                run += v;
            }
        }
        cnt[2 * q] = run & 0xFFFFu;
        cnt[2 * q + 1] = run >> 16;
        sum += cnt[2 * q] + cnt[2 * q + 1];
    }
    uint32_t tot;
    uint32_t st = block_excl_scan<kPartWaves>(sum, &tot, s_tmp);
    uint32_t* hrow = B.hist + D.hist_base + (uint64_t)tr.t * nbs;
#pragma unroll
    for (int q = 0; q < kPB / 2; ++q) {
        const uint32_t b0 = st, b1 = st + cnt[2 * q];
        st = b1 + cnt[2 * q + 1];
        if (pair0 + q >= nbs / 2) continue;
        uint32_t* col = s_pair + pair0 + q;
        const uint32_t add = b0 | (b1 << 16);
#pragma unroll
        for (int ww = 0; ww < kPartWaves; ++ww) col[ww * (L::kSlots / 2)] += add;
        *reinterpret_cast<uint2*>(hrow + 2 * (pair0 + q)) =
            make_uint2(cnt[2 * q] | (b0 << 16), cnt[2 * q + 1] | (b1 << 16));
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kE; ++e) {
        const uint32_t p = e * 64 + lane;
        const bool act = p < per && wb + p < m;
        uint32_t slot = act ? cnt_w[br[e] >> 16] + (br[e] & 0xFFFFu) : 0xFFFFFFFFu;
        if (act && slot >= m) { flag_error(B.cnt, ERR_BOUNDS); slot = 0xFFFFFFFFu; }
        br[e] = slot;
    }
    // the records in their new order, kPartStage at a time; the image in LDS
    // is shifted so that it is aligned to 16 bytes where its destination is.
    // The destination is the buffer the segment's strings are not in
    const uint64_t at = (SRC == kFromRuns && !(seg.flags & F_BUFB) ? B.cap : 0ull) + seg.begin + cb;
    uint32_t* out = B.rec + at * kRecWords;
    const uint32_t shift = (uint32_t)((uintptr_t)out >> 2) & 3u;
    for (uint32_t s0 = 0; s0 < m; s0 += kPartStage) {     // (uniform)
        const uint32_t ns = min(m - s0, kPartStage);
        if (s0) __syncthreads();     // the last part is copied (first: the lane-mask tables are read, a barrier ago)
#pragma unroll
        for (int e = 0; e < kE; ++e) {
            const uint32_t r = br[e] - s0;
            if (r < ns) {
                uint32_t* x = s_rec + shift + r * kRecWords;
                x[0] = (uint32_t)kv[e];
                x[1] = (uint32_t)(kv[e] >> 32);
                x[2] = SRC == kRootPlain || SRC == kRootPack ? seg.begin + cb + wb + e * 64 + lane : iv[e];
            }
        }
        __syncthreads();
        const uint32_t words = ns * kRecWords;
        uint32_t* o = out + (uint64_t)s0 * kRecWords - shift;      // (a 16-byte boundary)
        const uint4* img = reinterpret_cast<const uint4*>(s_rec);
        for (uint32_t v = tid; 4 * v < shift + words; v += T) {
            if (4 * v >= shift && 4 * v + 4 <= shift + words) {
                reinterpret_cast<uint4*>(o)[v] = img[v];
            } else {     // the ends
#pragma unroll
                for (uint32_t j = 4 * v; j < 4 * v + 4; ++j)
                    if (j >= shift && j < shift + words) o[j] = s_rec[j];
            }
        }
    }
#undef PS5_PART_POS
}

// XCD-contiguous chunks: workgroup g runs on XCD g % kXcds (the grid is a
// multiple of kXcds), and XCD x takes the chunks [N x / kXcds, N (x+1) /
// kXcds), so neighbouring chunks, whose runs of a bucket share cache lines
// with those of its neighbours, meet in one L2; each workgroup loops over its
// share (one chunk, in a level planned on the host).  ntiles: the level's
// chunks if the host knows them, else 0; one: a level of one segment, whose
// chunks need no table.
template <int NB, int SRC>
__global__ __launch_bounds__(kPartThreads, 4) void k_part(Plan P, Bufs B, const key64* trees, uint32_t ntiles, int one)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const uint32_t N = ntiles ? ntiles : P.hdr->ntiles, per = gridDim.x / kXcds, xcd = blockIdx.x % kXcds;
    const uint32_t thi = (uint32_t)((uint64_t)N * (xcd + 1) / kXcds);
    uint32_t ti = (uint32_t)((uint64_t)N * xcd / kXcds) + blockIdx.x / kXcds;
    for (; ti < thi; ti += per) {
        __syncthreads();     // the previous chunk's stage is written out
        part_chunk<NB, SRC>(ti, P, B, trees, one, smem);
    }
}

// a packed root met a character outside its alphabet: nothing of the level is
// of use, and without children no later one finds any work
__device__ __forceinline__ bool starts_over(const Bufs& B)
{
    return B.lut && (load_uniform(B.cnt + C_ERR) & ERR_ALPHA);
}

// Bucket counts summed over groups of kHistGroup chunks (segments of more
// than one group): row 1 + g of the segment's gsum.
__global__ __launch_bounds__(kWG) void k_hist_sum(Plan P, Bufs B)
{
    if (starts_over(B)) return;
    const uint32_t ng = P.hdr->ngroups;
    for (uint32_t gi = blockIdx.x; gi < ng; gi += gridDim.x) {
        const TileRef gr = load_uniform(P.groups + gi);
        const LargeDesc D = load_uniform(P.desc + gr.seg);
        const uint32_t G = hist_groups(D.nch), nbs = 2u << D.k;
        if (G == 1) continue;     // (k_children sums its rows)
        const uint32_t c0 = gr.t * kHistGroup, c1 = min(D.nch, c0 + kHistGroup);
        const uint32_t* h = B.hist + D.hist_base;
        for (uint32_t b = blockIdx.y * kWG + tid_x(); b < nbs; b += gridDim.y * kWG) {
            uint32_t s = 0;
#pragma unroll 8
            for (uint32_t c = c0; c < c1; ++c) s += h[(uint64_t)c * nbs + b] & 0xFFFFu;
            B.gsum[D.gbase + (1 + gr.t) * nbs + b] = s;
        }
    }
}

// The rows of the run tables: for bucket b and chunk c of a segment,
// vpos = the bucket's first position + its strings in the chunks before c,
// src = the chunk's place + the bucket's start inside it.  A workgroup takes
// 64 chunks x 64 buckets, turned in LDS from chunk-major to bucket-major.
__global__ __launch_bounds__(kWG) void k_hist_runs(Plan P, Bufs B, int buf)
{
    __shared__ uint32_t s_h[64][65];
    static_assert(kHistGroup == 64, "a lane per chunk of a group");
    if (starts_over(B)) return;
    const uint32_t ng = P.hdr->ngroups;
    uint32_t* V = B.vpos + (buf ? B.cap_h : 0ull);
    uint32_t* S = B.src + (buf ? B.cap_h : 0ull);
    const uint32_t w = wave_id(), lane = lane_id();
    for (uint32_t gi = blockIdx.x; gi < ng; gi += gridDim.x) {
        const TileRef gr = load_uniform(P.groups + gi);
        const LargeDesc D = load_uniform(P.desc + gr.seg);
        const uint32_t nbs = 2u << D.k, b0 = blockIdx.y * 64;
        if (b0 >= nbs) continue;     // (uniform)
        const uint32_t c0 = gr.t * kHistGroup, nc = min(D.nch - c0, kHistGroup);
        const uint32_t* h = B.hist + D.hist_base;
        __syncthreads();     // the previous tile is read
#pragma unroll 4
        for (uint32_t r = w; r < 64; r += kWaves)
            s_h[r][lane] = r < nc && b0 + lane < nbs ? h[(uint64_t)(c0 + r) * nbs + b0 + lane] : 0u;
        __syncthreads();
        const uint32_t chunk_at = D.seg.begin + (c0 + lane) * D.chunk;
        // lane: the first position of bucket b0 + lane in this group of chunks
        const uint32_t* g = B.gsum + D.gbase + min(b0 + lane, nbs - 1);
        const uint32_t firsts = g[0] + g[(1 + gr.t) * nbs];
        for (uint32_t r = w; r < 64; r += kWaves) {
            const uint32_t b = b0 + r;
            if (b + 1 >= nbs) break;     // (uniform) the last slot is no bucket
            const uint32_t x = s_h[lane][r], n = x & 0xFFFFu;
            uint32_t inc = n;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const uint32_t y = (uint32_t)__shfl_up((int)inc, d, 64);
                if (lane >= (uint32_t)d) inc += y;
            }
            const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)firsts, (int)r);
            if (lane < nc) {
                const uint32_t at = D.hist_base + b * D.nch + c0 + lane;
                V[at] = first + inc - n;
                S[at] = chunk_at + (x >> 16);
            }
        }
    }
}

// Emit the children buckets of a multi-workgroup step.  Tiny buckets become
// tiny leaves, other equal buckets (odd b) equal-key leaves in chunks, other
// less-than buckets blocks or large segments of the next level
// (distribute_finished, .hpp:1492-1584).  A thread takes the kPer buckets
// from tid * kPer on, of sz[] strings, the first of them starting at
// position start; dst: the buffer they lie in.
//
// spl: the segment's sorted splitters; equal bucket b holds the key spl[b >> 1],
// and one whose key holds no NUL continues into the next round (counted).
constexpr int kChildPer = (kMaxBkt + kBigWG) / kBigWG;     // 2 buckets per thread
constexpr int kChildLists = 3 + kBlkClasses;

__device__ __forceinline__ void emit_children(const LargeDesc& D, uint32_t start, const uint32_t (&sz)[kChildPer], uint32_t dst,
                                              const key64* spl, const Sink& s, uint32_t* sdepth_out, uint32_t* s_tmp)
{
    const Item seg = D.seg;
    const uint32_t base_flags = dst | (seg.flags & kFmtMask);
    const KeyFmt F = key_fmt(seg.flags);
    uint32_t c_t = 0, c_l = 0, c_r = 0, c_b[kBlkClasses] = {}, c_cont = 0;
#pragma unroll
    for (int j = 0; j < kChildPer; ++j) {
        const uint32_t b = tid_x() * kChildPer + j, m = sz[j];
        if (m == 0) continue;
        if (m <= kTinyT) c_t++;
        else if (b & 1) {
            c_r += (m + kRunChunk - 1) / kRunChunk;
            if (!key_ends(spl[b >> 1], F)) c_cont++;
        }
        else if (m <= kBlkT) c_b[block_class(m)]++;
        else c_l++;
    }
    // the list offsets of this thread's children: one scan of all seven
    // counts (tiny, large, equal-key chunks, the block classes), then one
    // atomic per list for the segment's place in it
    uint32_t cv[kChildLists], ov[kChildLists], tv[kChildLists];
    cv[0] = c_t;
    cv[1] = c_l;
    cv[2] = c_r;
#pragma unroll
    for (int c = 0; c < kBlkClasses; ++c) cv[3 + c] = c_b[c];
    block_excl_scan_k<kBigWaves, kChildLists>(cv, ov, tv, s_tmp);
    if (c_cont) atomicAdd(&s.cnt[s.c_runcont], c_cont);
    uint32_t* s_base = s_tmp + kBigWaves * kChildLists;
    if (tid_x() < kChildLists) {     // (a lane per list, so that the atomics are in flight together)
        const uint32_t l = tid_x();
        const int ci = l == 0 ? s.c_tiny : l == 1 ? s.c_large : l == 2 ? s.c_run : s.c_block + 2 * ((int)l - 3);
        uint32_t n = tv[0];
#pragma unroll
        for (int c = 1; c < kChildLists; ++c) n = l == (uint32_t)c ? tv[c] : n;
        s_base[l] = n ? atomicAdd(&s.cnt[ci], n) : 0u;
    }
    __syncthreads();
    uint32_t o_t = ov[0] + s_base[0], o_l = ov[1] + s_base[1], o_r = ov[2] + s_base[2], o_b[kBlkClasses];
#pragma unroll
    for (int c = 0; c < kBlkClasses; ++c) o_b[c] = ov[3 + c] + s_base[3 + c];
#pragma unroll
    for (int j = 0; j < kChildPer; ++j) {
        const uint32_t b = tid_x() * kChildPer + j, m = sz[j];
        if (m == 0) continue;
        const Item it = { start, m, seg.rbeg, base_flags, D.hist_base + b * D.nch, D.nch };
        start += m;
        if (m <= kTinyT) {
            put_item(s.tiny, s.cap_tiny, o_t++, it, s.cnt);
        } else if (b & 1) {
            const uint32_t nch = (m + kRunChunk - 1) / kRunChunk;
            sdepth_out[it.begin >> kDepthShift] = 0xFFFFFFFFu;     // (k_leaf_run's chunks lower it)
            for (uint32_t c = 0; c < nch; ++c) {
                Item r = it;
                r.flags = base_flags | F_SORTED | (c << kFlagShift);
                put_item(s.run, s.cap_run, o_r++, r, s.cnt);
            }
        } else if (m <= kBlkT) {
            const int c = block_class(m);
            put_item(s.block + (uint64_t)c * s.cap_block, s.cap_block, o_b[c]++, it, s.cnt);
        } else {
            put_item(s.large, s.cap_large, o_l++, it, s.cnt);
        }
    }
}

// Bucket sizes of the segments of a level, one workgroup each: their starts
// (gsum), and the children.  A segment of one group of chunks sums its bucket
// counts here, of more it scans the groups' sums, a thread per bucket.  dst:
// the buffer the level wrote.
//
// fused (a level planned on the host whose segments all are of one group and
// few entries, or on the device for one such segment): the segments' run
// tables are written here, after the bucket starts, and k_hist_runs is not
// launched.  It takes 5 to 9 us on its own for so little (40 K strings of ACGT:
// 121 -> 118 us, a burst of 16 served requests 1.45 -> 1.40 ms); a thread
// writes a bucket's row, which for the hundreds of segments of a level planned
// on the device is slower than k_hist_runs's turned tiles (64 M strings: 2.12
// ms fused, 2.09 not).
constexpr uint32_t kFusedRuns = 16384;     // entries of a segment
__global__ __launch_bounds__(kBigWG) void k_children(Plan P, Bufs B, const key64* trees, Sink s, uint32_t dst, int fused)
{
    __shared__ uint32_t s_sz[kMaxBkt + 1];
    __shared__ uint32_t s_tmp[kBigWaves * kChildLists + 8];     // the scans' scratch, then the lists' bases
    if (starts_over(B)) return;
    const uint32_t nlarge = P.hdr->nlarge;
    for (uint32_t si = blockIdx.x; si < nlarge; si += gridDim.x) {
        const LargeDesc D = load_uniform(P.desc + si);
        const uint32_t G = hist_groups(D.nch), nbs = 2u << D.k;
        uint32_t* g = B.gsum + D.gbase;
        uint32_t sz[kChildPer];
        if (G == 1) {     // (uniform)
            const uint32_t* h = B.hist + D.hist_base;
            for (uint32_t b = tid_x(); b < nbs; b += kBigWG) {
                uint32_t n = 0;
#pragma unroll 8
                for (uint32_t c = 0; c < D.nch; ++c) n += h[c * nbs + b] & 0xFFFFu;
                s_sz[b] = n;
            }
        } else {
            for (uint32_t b = tid_x(); b < nbs; b += kBigWG) {
                uint32_t* col = g + nbs + b;
                uint32_t n = 0;
                for (uint32_t i0 = 0; i0 < G; i0 += 8) {     // eight loads in flight
                    uint32_t x[8];
#pragma unroll
                    for (int j = 0; j < 8; ++j) x[j] = i0 + j < G ? col[(i0 + j) * nbs] : 0u;
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        if (i0 + j < G) col[(i0 + j) * nbs] = n;
                        n += x[j];
                    }
                }
                s_sz[b] = n;
            }
        }
        __syncthreads();
        uint32_t sum = 0;
#pragma unroll
        for (int j = 0; j < kChildPer; ++j) {
            const uint32_t b = tid_x() * kChildPer + j;
            sz[j] = b < nbs ? s_sz[b] : 0u;
            sum += sz[j];
        }
        uint32_t tot;
        const uint32_t start = D.seg.begin + block_excl_scan<kBigWaves>(sum, &tot, s_tmp);
        if (tot != D.seg.size) {     // (uniform) the counts must account for every string of the segment
            if (tid_x() == 0) flag_error(B.cnt, ERR_BOUNDS);
        } else {
            uint32_t at = start;
#pragma unroll
            for (int j = 0; j < kChildPer; ++j) {
                const uint32_t b = tid_x() * kChildPer + j;
                if (b < nbs) {
                    if (fused) s_sz[b] = at;
                    else g[b] = at;
                    if (G == 1 && !fused) g[nbs + b] = 0;
                }
                at += sz[j];
            }
            if (fused) {     // (uniform)
                __syncthreads();     // the starts are written
                const uint32_t* h = B.hist + D.hist_base;
                uint32_t* V = B.vpos + (dst ? B.cap_h : 0ull) + D.hist_base;
                uint32_t* S = B.src + (dst ? B.cap_h : 0ull) + D.hist_base;
                for (uint32_t b = tid_x(); b + 1 < nbs; b += kBigWG) {
                    uint32_t first = s_sz[b];
#pragma unroll 8
                    for (uint32_t c = 0; c < D.nch; ++c) {
                        const uint32_t x = h[c * nbs + b];
                        V[b * D.nch + c] = first;
                        S[b * D.nch + c] = D.seg.begin + c * D.chunk + (x >> 16);
                        first += x & 0xFFFFu;
                    }
                }
            }
            emit_children(D, start, sz, dst, trees + D.gbase + (1u << D.k), s, B.sdepth_out, s_tmp);
        }
        __syncthreads();     // the LDS is reused by the next segment
    }
}

// ---- leaves --------------------------------------------------------------------

// Finish one sorted position at depth d: LCP with the predecessor when the
// keys differ; inside a run of equal keys the LCP is known when the key holds
// a NUL (fill_lcp with lcpKeyDepth, .hpp:1546-1547), otherwise the run moves
// on to the next depth, where its keys are read through the permutation.
__device__ __forceinline__ void finish_position(const Bufs& B, uint32_t pos, uint32_t id, key64 k, bool has_prev,
                                                key64 pk, uint32_t depth, KeyFmt F)
{
    B.perm[pos] = id;
    if (!has_prev || !B.lcp) return;
    if (pk != k) B.lcp[pos] = depth + lcp_key(pk, k, F);
    else if (key_ends(k, F)) B.lcp[pos] = depth + key_depth(k, F);
}

// LDS exchange between the lanes of one wave: its LDS operations execute in
// order, so keeping the compiler from reordering them is enough.
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// One wave finishes a leaf of m <= 64 strings at positions [begin, begin+m)
// completely: a rank sort by broadcast compares (the slot each string takes
// in an LCP insertion sort, lcp_inssort.hpp:36-187) at depth `cur` (keys of
// format F), then,
// while runs of equal keys without a NUL remain, their strings fetch their
// next 8 characters and every such run is re-sorted in place.  Runs never
// leave the wave, so deep shared prefixes cost one gather per string per 8
// characters and no work-list traffic (the reference likewise finishes small
// buckets by insertion sort).  k, id: lane's key at `cur` and input index
// (lanes >= m ignored).  s_k, s_i, s_r: this wave's 64-entry LDS arrays.
// write_bkey: record the round-depth keys of the two end positions for the
// leaf-boundary pass.  All 64 lanes must call this.
//
// The wave may also finish several independent runs at once (packed runs of
// a block): slots [run0, run0 + length) of each run are contiguous, `pos` is
// the position this lane's slot stands for (consecutive within a run), and
// every lane of a run passes the run's first slot as run0.  A single leaf is
// run0 = 0, pos = begin + lane.
// NK: keys fetched per string at a time (1..8), or 0 for B.leaf_keys.
template <int NK>
__device__ void wave_finish_leaf(const Bufs& B, uint32_t pos, uint32_t m, key64 k, uint32_t id, uint32_t cur,
                                 KeyFmt F, bool write_bkey, uint32_t run0, key64* s_k, uint32_t* s_i, uint32_t* s_r)
{
    const uint32_t lane = lane_id();
    const bool act = lane < m;
    // every string starts in its run; (key, slot) orders a run stably
    uint32_t run = run0;
    bool live = act;         // position still has an undecided successor relation
    wave_lds_sync();
    if (act) {
        s_k[lane] = k;
        s_r[lane] = run0;
    }
    bool first_pass = write_bkey;
    constexpr int kLeafKeys = 8;
    key64 kbuf[kLeafKeys] = {};     // string bid's next keys (depths cur+8, cur+16, ...)
    // keys fetched per string at a time (the tuned key width of leaf passes)
    const int nk = NK ? NK : (int)min(max(B.leaf_keys, 1u), (uint32_t)kLeafKeys);
    uint32_t bid = 0xFFFFFFFFu;
    int nbuf = 0;
    for (;;) {
        // re-sort every live run by (key, slot); finished positions keep their slot
        wave_lds_sync();
        uint32_t rank = lane;
        if (live) {
            rank = run;
            for (uint32_t j = run; j < m && s_r[j] == run; ++j) {
                const key64 kj = s_k[j];
                rank += (kj < k || (kj == k && j < lane)) ? 1u : 0u;
            }
        }
        wave_lds_sync();
        if (live) {
            s_k[rank] = k;
            s_i[rank] = id;
        } else if (act) {
            s_i[lane] = id;
        }
        wave_lds_sync();
        if (act) {
            k = s_k[lane];
            id = s_i[lane];
        }
        wave_lds_sync();
        // neighbours inside the same run at this depth
        key64 pk = 0;
        bool eqp = false, eqn = false, same_prev = false;
        if (act && live) {
            same_prev = lane > 0 && s_r[lane - 1] == run;
            if (same_prev) pk = s_k[lane - 1];
            eqp = same_prev && pk == k;
            eqn = lane + 1 < m && s_r[lane + 1] == run && s_k[lane + 1] == k;
        }
        const bool term = key_ends(k, F);
        if (act && live) {
            if (first_pass && (lane == 0 || lane == m - 1)) B.bkey[pos] = k;
            if (same_prev && !eqp && B.lcp) B.lcp[pos] = cur + lcp_key(pk, k, F);
            if (eqp && term && B.lcp) B.lcp[pos] = cur + key_depth(k, F);
            if ((!eqp && !eqn) || term) {
                B.perm[pos] = id;     // decided: a single string or identical strings
                live = false;
            }
        }
        // new runs: a live position starts one where it differs from its predecessor
        const uint64_t starts = __ballot(act && live && !eqp);
        const uint64_t alive = __ballot(act && live);
        if (alive == 0) break;
        if (live) {
            const uint64_t below = starts & ((2ull << lane) - 1);   // start bits at or below this lane
            run = 63u - (uint32_t)__clzll((long long)below);
        }
        wave_lds_sync();
        if (act) s_r[lane] = live ? run : 0xFFFFFFFFu;
        // the next 8 characters of every string still in a run: fetched
        // nk keys at a time, so deep shared prefixes cost one memory round
        // trip per 8 * nk characters.  A lane's buffer belongs
        // to the string it was loaded for (bid); when a re-sort moved any
        // string to another lane, the wave loads afresh.
        first_pass = false;
        cur += F.cpk;
        F = key_fmt(0);      // (what is fetched here is plain characters)
        if (nbuf == 0 || __ballot(live && id != bid) != 0) {     // (uniform)
            const bool ok = live && id < B.n;
            if (live && !ok) flag_error(B.cnt, ERR_BOUNDS);
            const uint64_t off = ok ? str_off(B, id) : 0ull;
            bid = id;
            // depths where, in every run, all strings agree with the run's
            // first one and none ends decide nothing: skip them together.
            // While all fetched keys do, the wave fetches on without sorting
            // (the suffixes of a 4.2 MB text with long repeats: 1.24 -> 0.89 ms)
            int skip;
            for (;;) {
                if (live) {
                    if (ok) load_keys<kLeafKeys>(B.arena, B.alen, off + cur, kbuf, nk);
                    else for (int i = 0; i < kLeafKeys; ++i) kbuf[i] = 0;
                }
                skip = nk;
#pragma unroll
                for (int i = 0; i < kLeafKeys; ++i) {
                    if (i >= nk) break;     // (uniform)
                    const uint32_t lo = __shfl((uint32_t)kbuf[i], (int)run, 64);
                    const uint32_t hi = __shfl((uint32_t)(kbuf[i] >> 32), (int)run, 64);
                    const bool same = kbuf[i] == (((uint64_t)hi << 32) | lo) && (kbuf[i] & 0xFFull) != 0;
                    if (skip == nk && __ballot(live && !same) != 0) skip = i;     // (uniform)
                }
                if (skip < nk) break;     // (uniform)
                cur += 8 * (uint32_t)nk;
            }
            nbuf = nk;
            for (int s = 0; s < skip; ++s) {     // (uniform)
#pragma unroll
                for (int i = 0; i + 1 < kLeafKeys; ++i) kbuf[i] = kbuf[i + 1];
            }
            nbuf -= skip;
            cur += 8 * (uint32_t)skip;
        }
        k = kbuf[0];
#pragma unroll
        for (int i = 0; i + 1 < kLeafKeys; ++i) kbuf[i] = kbuf[i + 1];
        --nbuf;
        if (live) s_k[lane] = k;
    }
}

// Key and input index of the string at lane's position L.begin + lane of a
// leaf of at most 64 strings (lane < L.size).  A bucket of at most 64 runs has
// them in the lanes; longer rows are searched.
__device__ __forceinline__ void load_tiny(const Bufs& B, const Item& L, uint32_t depth, key64* k, uint32_t* id)
{
    const uint32_t lane = lane_id(), pos = L.begin + lane;
    const bool act = lane < L.size;
    if (L.flags & (F_IDENT | F_NEXT)) {     // (uniform)
        if (act) {
            *id = (L.flags & F_IDENT) ? pos : B.perm[pos];
            *k = string_key(B, *id, depth);
        }
        return;
    }
    const Runs R = runs_of(B, L);
    uint32_t q = 0;
    if (R.nch <= 64) {     // (uniform)
        uint32_t v = 0, sp = 0;
        if (lane < R.nch) {
            v = R.V[lane];
            sp = R.S[lane];
        }
        // (an empty run starts where the next one does, or at the leaf's end)
        const uint32_t down = (uint32_t)__shfl_down((int)v, 1, 64);     // (by all lanes)
        const uint32_t nx = lane + 1 < R.nch ? down : L.begin + L.size;
        for (uint64_t m = __ballot(lane < R.nch && nx > v); m; m &= m - 1) {     // (uniform)
            const int c = __builtin_ctzll(m);
            const uint32_t rv = (uint32_t)__builtin_amdgcn_readlane((int)v, c);
            const uint32_t rs = (uint32_t)__builtin_amdgcn_readlane((int)sp, c);
            if (pos >= rv) q = rs + (pos - rv);
        }
        if (act) q = checked_place(B, q);
    } else if (act) {
        q = run_place(B, R, pos);
    }
    if (act) {
        const Rec r = R.R[q];
        *k = rec_key(r);
        *id = r.id;
    }
}

// One tiny leaf (at most 64 strings), finished completely by one wave.
// s_k, s_i, s_r: its 64-entry LDS arrays.
template <int NK>
__device__ __forceinline__ void tiny_leaf(const Item& L, const Bufs& B, key64* s_k, uint32_t* s_i, uint32_t* s_r)
{
    const uint32_t lane = lane_id();
    if (!item_ok(L, B) || L.size > kTinyT) {     // (uniform)
        if (lane == 0) flag_error(B.cnt, ERR_BOUNDS);
        return;
    }
    key64 k = ~0ull;
    uint32_t id = 0;
    const uint32_t depth = tiny_depth(B, L);
    load_tiny(B, L, depth, &k, &id);
    wave_finish_leaf<NK>(B, L.begin + lane, L.size, k, id, depth, key_fmt(L.flags), true, 0u, s_k, s_i, s_r);
}

// The tiny leaves from *p_first (first, if null) to entry `end` of a list, a wave each.
template <int NK>
__global__ __launch_bounds__(kWG) void k_leaf_tiny(const Item* items, const uint32_t* p_first, uint32_t first,
                                                   const uint32_t* cnt_items, uint32_t end, Bufs B)
{
    __shared__ key64 s_k[kWaves][64];
    __shared__ uint32_t s_i[kWaves][64];
    __shared__ uint32_t s_r[kWaves][64];     // first sorted position of the run holding a position
    const uint32_t w = wave_id();
    if (B.pending && *B.pending) {      // the round's levels are not finished
        if (B.pending_err && tid_x() == 0) flag_error(B.cnt, ERR_LEVELS);
        return;
    }
    const uint32_t nitems = min(*cnt_items, end);     // (an overflow of the list has been flagged)
    if (p_first) first = *p_first;
    // each wave takes leaves it, it + stride, ... (no workgroup barriers below)
    for (uint32_t it = first + blockIdx.x * kWaves + w; it < nitems; it += gridDim.x * kWaves) {
        const Item L = load_uniform(items + __builtin_amdgcn_readfirstlane((int)it));
        tiny_leaf<NK>(L, B, s_k[w], s_i[w], s_r[w]);
    }
}

// Sorting network over E (key, position) pairs in one thread's registers
// (Batcher's odd-even merge sort: 5 comparators for 4, 19 for 8).  Positions
// are distinct, so the (key, position) order is total and the result stable.
template <int E>
__device__ __forceinline__ void thread_sort(key64 (&k)[E], uint32_t (&p)[E])
{
    static_assert(E == 4 || E == 8, "networks for 4 and 8 elements");
    constexpr int n4[][2] = { { 0, 1 }, { 2, 3 }, { 0, 2 }, { 1, 3 }, { 1, 2 } };
    constexpr int n8[][2] = { { 0, 1 }, { 2, 3 }, { 4, 5 }, { 6, 7 }, { 0, 2 }, { 1, 3 }, { 4, 6 },
                              { 5, 7 }, { 1, 2 }, { 5, 6 }, { 0, 4 }, { 1, 5 }, { 2, 6 }, { 3, 7 },
                              { 2, 4 }, { 3, 5 }, { 1, 2 }, { 3, 4 }, { 5, 6 } };
    constexpr int NC = E == 4 ? 5 : 19;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int a = E == 4 ? n4[c][0] : n8[c][0], b = E == 4 ? n4[c][1] : n8[c][1];
        const bool sw = kp_less(k[b], p[b], k[a], p[a]);
        const key64 ka = k[a], kb = k[b];
        const uint32_t pa = p[a], pb = p[b];
        k[a] = sw ? kb : ka;
        k[b] = sw ? ka : kb;
        p[a] = sw ? pb : pa;
        p[b] = sw ? pa : pb;
    }
}

constexpr uint32_t kBlockRuns = 64;     // short runs a block finishes itself (per batch of runs)

// Long runs (> kTinyT strings) a block in tail mode keeps to sort itself at
// their next depth.  Pending runs are disjoint intervals of the block, so
// at most kBlkT / (kTinyT + 1) = 31 wait at once.
constexpr uint32_t kTailStack = 32;
struct TailStack {
    uint32_t pos[kTailStack], len[kTailStack], depth[kTailStack];
    uint32_t n;
};
// keys per thread of the four block classes (256, 512, 1024, 2048 keys)
constexpr int kBlkE0 = 4, kBlkE1 = 4, kBlkE2 = 4, kBlkE3 = 4;

// Finish a block's short runs of equal keys (each at most 64 strings, at
// sorted positions beg + (s_runs[r] >> 16)) at depth, the block's next one
// (their strings are in perm): the runs are
// packed into batches of at most 64 strings, and a wave finishes all runs of
// a batch in one pass (duplicates come in many short runs).  The batch
// table lives in s_k after the waves' leaf arrays.
template <int NK>
__device__ __forceinline__ void block_finish_runs(const Bufs& B, key64* s_k, const uint32_t* s_runs,
                                                  uint32_t nruns, uint32_t beg, uint32_t depth, uint32_t nwaves)
{
    const uint32_t tid = tid_x(), w = wave_id(), lane = lane_id();
    // the sorted block is no longer needed: each wave's leaf arrays live in
    // s_k, and after them the run batches
    uint32_t* s_rslot = reinterpret_cast<uint32_t*>(s_k + nwaves * 128);      // first slot of a run in its batch
    uint32_t* s_bfirst = s_rslot + kBlockRuns;                                 // first run of each batch
    uint32_t* s_nbatch_p = s_bfirst + kBlockRuns + 1;
    // pack the runs into batches of at most 64 strings: a wave finishes all
    // runs of a batch in one pass (duplicates come in many short runs)
    if (tid == 0) {
        uint32_t nb = 0, fill = 64;
        for (uint32_t r = 0; r < nruns; ++r) {
            const uint32_t len = s_runs[r] & 0xFFFFu;
            if (fill + len > 64) {
                s_bfirst[nb++] = r;
                fill = 0;
            }
            s_rslot[r] = fill;
            fill += len;
        }
        s_bfirst[nb] = nruns;
        *s_nbatch_p = nb;
    }
    __syncthreads();
    key64* wk = s_k + w * 128;
    uint32_t* wi = reinterpret_cast<uint32_t*>(wk + 64);
    uint32_t* wr = wi + 64;
    const uint32_t nbatch = *s_nbatch_p;
    for (uint32_t bt = w; bt < nbatch; bt += nwaves) {
        const uint32_t r0 = s_bfirst[bt], r1 = s_bfirst[bt + 1];
        uint32_t slot0 = 0, total = 0, rs = 0;
        bool mine = false;
        for (uint32_t r = r0; r < r1; ++r) {     // the run whose slots hold this lane
            const uint32_t so = s_rslot[r], len = s_runs[r] & 0xFFFFu;
            if (lane >= so && lane < so + len) {
                mine = true;
                slot0 = so;
                rs = s_runs[r] >> 16;
            }
            total = max(total, so + len);
        }
        key64 kk = 0;
        uint32_t id = 0, pos = 0;
        if (mine) {
            pos = beg + rs + (lane - slot0);
            id = B.perm[pos];
            kk = string_key(B, id, depth);
        }
        wave_finish_leaf<NK>(B, pos, total, kk, id, depth, key_fmt(0), false, slot0, wk, wi, wr);
    }
}

// Merge sort of a block's m keys, in s_k in position order (padding ~0 up
// to the next multiple of E sorts last): each of MAXM / E threads sorts E
// consecutive (key, position) pairs with a sorting network, then runs are
// merged pairwise by merge path: a thread finds where its E outputs start in
// the two runs by binary search (co-rank) and merges them sequentially; on
// equal keys the left run goes first, so the order stays stable.  Leaves the
// sorted keys in s_k and their positions in s_p.
template <uint32_t MAXM, int E>
__device__ __forceinline__ void block_merge_sort(uint32_t m, key64* s_k, uint16_t* s_p)
{
    constexpr uint32_t T = MAXM / E;
    (void)T;
    const uint32_t tid = tid_x();
    const uint32_t Ta = (m + E - 1) / E, Pm = Ta * E;   // threads in use, padded size
    key64 k[E];
    uint32_t p[E];
    const uint32_t o = tid * E;
    if (tid < Ta) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            k[e] = s_k[o + e];
            p[e] = o + e;
        }
        thread_sort<E>(k, p);
    }
    __syncthreads();
    if (tid < Ta) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            s_k[o + e] = k[e];
            s_p[o + e] = (uint16_t)p[e];
        }
    }
    __syncthreads();
    for (uint32_t Lr = E; Lr < Pm; Lr <<= 1) {
        if (tid < Ta) {
            const uint32_t a0 = (o / (2 * Lr)) * (2 * Lr), la = min(Lr, Pm - a0);
            const uint32_t b0 = a0 + Lr, lb = b0 < Pm ? min(Lr, Pm - b0) : 0u;
            const uint32_t diag = o - a0;
            uint32_t lo = diag > lb ? diag - lb : 0u, hi = min(diag, la);
            while (lo < hi) {
                const uint32_t mid = (lo + hi) >> 1;
                if (s_k[a0 + mid] <= s_k[b0 + diag - 1 - mid]) lo = mid + 1;
                else hi = mid;
            }
            // the heads as byte offsets into s_k, and the runs' ends
            uint32_t pa = (a0 + lo) * 8u, pb = (b0 + diag - lo) * 8u;
            const uint32_t ea = (a0 + la) * 8u, eb = (b0 + lb) * 8u;
            const unsigned char* kbase = reinterpret_cast<const unsigned char*>(s_k);
            const unsigned char* pbase = reinterpret_cast<const unsigned char*>(s_p);
            key64 ka = pa < ea ? *reinterpret_cast<const key64*>(kbase + pa) : 0ull;
            key64 kb = pb < eb ? *reinterpret_cast<const key64*>(kbase + pb) : 0ull;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                // branch-free step: the consumed run's next head is the slot
                // after the one taken (past a run's end it is never used:
                // take_a tests pa < ea and pb >= eb; s_k has one spare slot)
                const bool take_a = pb >= eb || (pa < ea && ka <= kb);
                const uint32_t src = take_a ? pa : pb;
                k[e] = take_a ? ka : kb;
                p[e] = *reinterpret_cast<const uint16_t*>(pbase + (src >> 2));
                const key64 nx = *reinterpret_cast<const key64*>(kbase + src + 8u);
                pa += take_a ? 8u : 0u;
                pb += take_a ? 0u : 8u;
                ka = take_a ? nx : ka;
                kb = take_a ? kb : nx;
            }
        }
        __syncthreads();
        if (tid < Ta) {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                s_k[o + e] = k[e];
                s_p[o + e] = (uint16_t)p[e];
            }
        }
        __syncthreads();
    }
}

// Radix partition of a block.  The keys of a block lie between two
// neighbouring splitters, so their offsets from the block's smallest key
// usually fit 48 bits; then v = offset << 16 | position orders the block
// exactly as (key, position) does, in one 64-bit word.  Values are grouped
// by their top log2(MAXM) offset bits and ranked inside their groups.  A
// thread's ranking work grows with the sizes of the groups its slots fall
// in, so a block is merge-sorted instead when its offsets need more than 48
// bits, a group holds more than kRadixMaxGroup keys, or the key-weighted
// mean group size (sum of squared group sizes over the keys) exceeds
// kRadixMeanGroup.
constexpr uint32_t kRadixMaxGroup = 128;
constexpr uint32_t kRadixMeanGroup = 16;

// Exclusive block scan of a, the block totals of a and b and the block
// maximum of b (one uint32 each per thread, NW waves), with one barrier.  The
// caller writes s_tmp again only after another barrier.
template <int NW>
__device__ __forceinline__ uint32_t block_scan_sum_max(uint32_t a, uint32_t b, uint32_t* tot_a, uint32_t* tot_b,
                                                       uint32_t* max_b, uint32_t* s_tmp)
{
    const uint32_t lane = lane_id(), w = wave_id();
    uint32_t x = a, sb = b, mb = b;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)x, d, 64);
        if (lane >= (uint32_t)d) x += y;
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        sb += (uint32_t)__shfl_xor((int)sb, d, 64);
        mb = max(mb, (uint32_t)__shfl_xor((int)mb, d, 64));
    }
    if (lane == 63) {
        s_tmp[w] = x;
        s_tmp[NW + w] = sb;
        s_tmp[2 * NW + w] = mb;
    }
    __syncthreads();
    uint32_t wpre = 0, ta = 0, tb = 0, mx = 0;
#pragma unroll 1
    for (int i = 0; i < NW; ++i) {     // (not unrolled: few registers for the 8-wave class)
        const uint32_t t = s_tmp[i];
        wpre += (i < (int)w) ? t : 0u;
        ta += t;
        tb += s_tmp[NW + i];
        mx = max(mx, s_tmp[2 * NW + i]);
    }
    *tot_a = ta;
    *tot_b = tb;
    *max_b = mx;
    return wpre + x - a;
}

// minimum and maximum over the wave by lane moves inside the vector unit (the
// lanes' values need no trip through the LDS), then over the workgroup (NW
// waves; s_tmp: 2 NW words, written again by the caller only after a barrier)
template <int CTRL, int ROWS>
__device__ __forceinline__ void dpp_min_max(uint32_t& lo, uint32_t& hi)
{
    lo = min(lo, (uint32_t)__builtin_amdgcn_update_dpp((int)0xFFFFFFFFu, (int)lo, CTRL, ROWS, 0xF, false));
    hi = max(hi, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)hi, CTRL, ROWS, 0xF, false));
}
template <int NW>
__device__ __forceinline__ void block_min_max(uint32_t& lo, uint32_t& hi, uint32_t* s_tmp)
{
    dpp_min_max<0x111, 0xF>(lo, hi);     // row_shr:1, 2, 4, 8: lane 15 of a row has the row's
    dpp_min_max<0x112, 0xF>(lo, hi);
    dpp_min_max<0x114, 0xF>(lo, hi);
    dpp_min_max<0x118, 0xF>(lo, hi);
    dpp_min_max<0x142, 0xA>(lo, hi);     // row_bcast:15 into rows 1 and 3
    dpp_min_max<0x143, 0xC>(lo, hi);     // row_bcast:31 into rows 2 and 3: lane 63 has the wave's
    if (NW == 1) {
        lo = (uint32_t)__builtin_amdgcn_readlane((int)lo, 63);
        hi = (uint32_t)__builtin_amdgcn_readlane((int)hi, 63);
        __syncthreads();
        return;
    }
    if (lane_id() == 63) {
        s_tmp[wave_id()] = lo;
        s_tmp[NW + wave_id()] = hi;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NW; ++i) {
        lo = min(lo, s_tmp[i]);
        hi = max(hi, s_tmp[NW + i]);
    }
}

// Radix-partitioned rank sort of a block's m keys (w: thread t's keys of the positions t, t + T, ..):
// values v are grouped in LDS by d = v >> (16 + sh), the top log2(MAXM)
// bits of the offset (slots from LDS atomics, in no particular order), and
// each value's sorted slot is its group's start plus the group members below
// it -- exact, so the result is the stable sort.  Returns false when the
// block is to be merge-sorted; s_k then holds the keys in position order,
// padded with ~0 up to the next multiple of E, for block_merge_sort.  On
// success s_k holds the sorted keys and s_p their positions.  s_cnt: MAXM +
// 2 counters (group counts, the total, a spare for lanes past m).
template <uint32_t MAXM, int E>
__device__ __forceinline__ bool block_radix_sort(key64 (&w)[E], uint32_t m, key64* s_k, uint16_t* s_p,
                                                 uint32_t* s_cnt, uint32_t* s_tmp)
{
    constexpr uint32_t T = MAXM / E;
    constexpr int NW = (int)(T / 64);
    constexpr int D = __builtin_ctz(MAXM);      // digit bits: MAXM groups
    static_assert((MAXM & (MAXM - 1)) == 0 && MAXM / T == (uint32_t)E, "a power-of-two block, E counters per thread");
    // (through an opaque move: indices derived from it are recomputed per
    // block instead of being hoisted out of a tail workgroup's loop)
    const uint32_t tid = scat_tid();
    const uint32_t Pm = (m + E - 1) / E * E;
    // w: this thread's keys (positions e*T + tid, clamped to the block), later
    // their packed values
    for (uint32_t j = tid; j < MAXM + 2; j += T) s_cnt[j] = 0;
    // bounds of the keys from their high words, or from their low words where
    // those agree: any bounds do, and words take a quarter of the instructions
    uint32_t lo32 = ~0u, hi32 = 0u;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        lo32 = min(lo32, (uint32_t)(w[e] >> 32));     // (clamped copies of the last key change neither)
        hi32 = max(hi32, (uint32_t)(w[e] >> 32));
    }
    block_min_max<NW>(lo32, hi32, s_tmp);
    key64 kmin = (key64)lo32 << 32, kmax = ((key64)hi32 << 32) | 0xFFFFFFFFull;
    if (lo32 == hi32) {     // (uniform)
        lo32 = ~0u;
        hi32 = 0u;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            lo32 = min(lo32, (uint32_t)w[e]);
            hi32 = max(hi32, (uint32_t)w[e]);
        }
        block_min_max<NW>(lo32, hi32, s_tmp + 2 * NW);
        kmax = kmin | hi32;
        kmin |= lo32;
    }
    // (s_tmp is written again only after the counting barrier below)
    const key64 range = kmax - kmin;
    if (range == 0) {     // (uniform) all keys equal (a run sorted at its next depth): already in order
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const uint32_t i = (uint32_t)e * T + tid;
            if (i < m) {
                s_k[i] = kmin;
                s_p[i] = (uint16_t)i;
            }
        }
        __syncthreads();
        return true;
    }
    if ((range >> 48) != 0) {     // (uniform) offsets too wide to pack: merge sort
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const uint32_t i = (uint32_t)e * T + tid;
            if (i < Pm) s_k[i] = i < m ? w[e] : ~0ull;
        }
        __syncthreads();
        return false;
    }
    // the packed values, and the shift that leaves a value's group
    const int sh = 16 + max(0, 64 - (int)__clzll((long long)(range | 1)) - D);
    // (positions past m count into the spare counter s_cnt[MAXM + 1])
    uint32_t slot[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const uint32_t i = (uint32_t)e * T + tid;
        w[e] = ((w[e] - kmin) << 16) | i;
        slot[e] = atomicAdd(&s_cnt[i < m ? (uint32_t)(w[e] >> sh) : MAXM + 1], 1u);
    }
    __syncthreads();
    // group starts (exclusive scan in place, E counters per thread); the
    // largest per-thread sum of squared group sizes and their total
    uint32_t sum = 0, sq = 0;
#pragma unroll
    for (int j = 0; j < E; ++j) {
        const uint32_t c = s_cnt[tid * E + j];
        sum += c;
        sq += c * c;
    }
    uint32_t tot, tsq, over;
    // (all counts are read before the scan's barrier: starts may overwrite them)
    uint32_t run = block_scan_sum_max<NW>(sum, sq, &tot, &tsq, &over, s_tmp);
#pragma unroll
    for (int j = 0; j < E; ++j) {
        const uint32_t c = s_cnt[tid * E + j];
        s_cnt[tid * E + j] = run;
        run += c;
    }
    if (tid == 0) s_cnt[MAXM] = tot;
    __syncthreads();
    if (over > kRadixMaxGroup * kRadixMaxGroup || tsq > kRadixMeanGroup * m) {   // (uniform) merge sort instead
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const uint32_t i = (uint32_t)e * T + tid;
            if (i < Pm) s_k[i] = i < m ? (w[e] >> 16) + kmin : ~0ull;
        }
        __syncthreads();
        return false;
    }
    key64* s_v = s_k;     // packed values, grouped
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const uint32_t i = (uint32_t)e * T + tid;
        if (i < m) s_v[s_cnt[(uint32_t)(w[e] >> sh)] + slot[e]] = w[e];
    }
    __syncthreads();
    // sorted places: thread t ranks the slots t + e T (consecutive lanes read
    // consecutive values, free of LDS bank conflicts).  Groups are ordered
    // by their top bits, so a slot's place is its group's start plus the
    // group's values below it; value and place stay in registers until every
    // value has been read.
    uint32_t place[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        if ((uint32_t)e * T >= m) break;     // (uniform) no slot of this pass is in the block
        const uint32_t j = (uint32_t)e * T + tid;
        const uint32_t jc = min(j, m - 1);
        const key64 v = s_v[jc];
        const uint32_t g = (uint32_t)(v >> sh);
        const uint32_t G1 = s_cnt[g + 1];
        uint32_t q = s_cnt[g], r = q;
        for (; q + 1 < G1; q += 2) {     // two values per step: their reads overlap
            const key64 va = s_v[q], vb = s_v[q + 1];
            r += (va < v ? 1u : 0u) + (vb < v ? 1u : 0u);
        }
        if (q < G1) r += s_v[q] < v ? 1u : 0u;
        w[e] = v;
        place[e] = r;
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < E; ++e) {
        if ((uint32_t)e * T >= m) break;     // (uniform)
        if ((uint32_t)e * T + tid < m) {
            s_k[place[e]] = (w[e] >> 16) + kmin;
            s_p[place[e]] = (uint16_t)w[e];
        }
    }
    __syncthreads();
    return true;
}

// The block sort's LDS (one workgroup).
template <uint32_t MAXM, int E, bool TAIL>
struct BlockLds {
    static constexpr uint32_t T = MAXM / E;
    key64 k[MAXM + 1];     // + 1: a merge step reads the slot after the one it takes
    uint16_t p[MAXM];
    uint32_t runs[TAIL ? MAXM / 2 : kBlockRuns];      // (start << 16) | length; in tail mode every short run
    uint32_t nruns;
    uint32_t cnt[MAXM + 2];           // radix partition: group counts, then starts
    alignas(8) uint32_t tmp[4 * (T / 64) + 4];
};

// One workgroup of MAXM / E threads sorts a block of 65..MAXM strings
// completely on chip and finishes every position at this depth (the
// reference's insertion-sort base case, lcp_inssort.hpp:36-187, and the
// equal-bucket rules, .hpp:1531-1557, on sorted keys).  The sort is the
// radix partition with in-group ranks (block_radix_sort) when the block's
// keys spread well over their range, else the merge sort (block_merge_sort);
// both give the stable (key, position) order.  Finishing a sorted position:
// LCP to its neighbour, identical strings done, runs of equal keys without a
// NUL handed to round r+1.
//
// TAIL (a round whose blocks are its last work): a run longer than kTinyT
// is pushed on the workgroup's stack ts at depth + 8 instead of going to the
// next round (k_block sorts it there), and every short run is finished here.
// top: a block of the round's lists (false: a run of one, sorted deeper),
// whose first and last keys at this depth go to bkey for k_leafbound.
template <uint32_t MAXM, int E, int NK, bool TAIL>
__device__ __forceinline__ void block_one(const Item L, const Bufs& B, const Sink& nxt, uint32_t depth,
                                          BlockLds<MAXM, E, TAIL>& S, TailStack* ts, bool top)
{
    constexpr uint32_t T = MAXM / E;
    static_assert(T % 64 == 0 && MAXM <= 65536, "whole waves; positions fit 16 bits");
    // short equal runs finished here (more go to the next round; all of them in tail mode)
    constexpr uint32_t kMaxRuns = TAIL ? MAXM / 2 : kBlockRuns;
    static_assert(MAXM * 8 >= 1024 * (T / 64) + 4 * (2 * kBlockRuns + 2),
                  "the per-wave leaf arrays (1 KB each) and the run batches reuse s_k");
    key64* s_k = S.k;
    uint16_t* s_p = S.p;
    uint32_t* s_runs = S.runs;
    uint32_t& s_nruns = S.nruns;
    uint32_t* s_cnt = S.cnt;
    uint32_t* s_tmp = S.tmp;
    if (!item_ok(L, B) || L.size > MAXM) {
        if (tid_x() == 0) flag_error(B.cnt, ERR_BOUNDS);
        return;
    }
    const uint32_t m = L.size, beg = L.begin;
    uint32_t tid = scat_tid();     // (opaque: see block_radix_sort)
    const KeyFmt F = key_fmt(L.flags);
    if (tid == 0) s_nruns = 0;
    // keys and input indices; every load is unconditional (clamped position),
    // so all of a thread's are in flight at once.  The indices stay in
    // registers through the sort, then are staged in s_cnt (free after either
    // sort), so that sorted positions read them from LDS
    constexpr int kPerThread = MAXM / T;
    key64 w[kPerThread];
    uint32_t idv[kPerThread];
    if (L.flags & (F_IDENT | F_NEXT)) {     // (uniform)
#pragma unroll
        for (int e = 0; e < kPerThread; ++e) {
            const uint32_t pos = beg + min(tid + (uint32_t)e * T, m - 1);
            idv[e] = (L.flags & F_IDENT) ? pos : B.perm[pos];
        }
#pragma unroll
        for (int e = 0; e < kPerThread; ++e) w[e] = string_key(B, idv[e], depth);
    } else {
        // a bucket of at most 64 runs has them in the lanes of every wave, and
        // a wave's 64 consecutive positions walk the few runs they meet (the
        // blocks of 42 M keys are bound by instruction issue: with the bounds
        // below by words, 750 -> 630 us); longer rows are copied to s_k and
        // searched there, or searched where they are
        const Runs R = runs_of(B, L);
        uint32_t* s_v = reinterpret_cast<uint32_t*>(s_k);
        uint32_t q[kPerThread];
        if (R.nch <= 64) {     // (uniform)
            const uint32_t lane = tid & 63u;
            uint32_t v = 0xFFFFFFFFu, sp = 0;
            if (lane < R.nch) {
                v = R.V[lane];
                sp = R.S[lane] - v;     // a string's place less its position
            }
#pragma unroll
            for (int e = 0; e < kPerThread; ++e) {
                const uint32_t pos = beg + min(tid + (uint32_t)e * T, m - 1);
                const uint32_t p0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)pos);
                uint64_t rest = __ballot(v <= p0 + 63u);       // runs starting before the wave's positions end
                uint64_t upto = __ballot(v <= p0);              // the last of them holds its first one
                int c = 63 - (int)__builtin_clzll(upto | 1ull);
                uint32_t d = (uint32_t)__builtin_amdgcn_readlane((int)sp, c);
                for (rest &= ~((2ull << c) - 1ull); rest; rest &= rest - 1) {     // (uniform)
                    c = __builtin_ctzll(rest);
                    const uint32_t rv = (uint32_t)__builtin_amdgcn_readlane((int)v, c);
                    const uint32_t rd = (uint32_t)__builtin_amdgcn_readlane((int)sp, c);
                    if (pos >= rv) d = rd;
                }
                q[e] = checked_place(B, pos + d);
            }
        } else if (R.nch <= MAXM) {     // (uniform)
            for (uint32_t c = tid; c < R.nch; c += T) {
                s_v[c] = R.V[c];
                s_v[R.nch + c] = R.S[c];
            }
            __syncthreads();
#pragma unroll
            for (int e = 0; e < kPerThread; ++e) {
                const uint32_t pos = beg + min(tid + (uint32_t)e * T, m - 1);
                const uint32_t c = find_run(s_v, R.nch, pos);
                q[e] = checked_place(B, s_v[R.nch + c] + (pos - s_v[c]));
            }
        } else {
#pragma unroll
            for (int e = 0; e < kPerThread; ++e) q[e] = run_place(B, R, beg + min(tid + (uint32_t)e * T, m - 1));
        }
#pragma unroll
        for (int e = 0; e < kPerThread; ++e) {
            const Rec r = R.R[q[e]];
            w[e] = rec_key(r);
            idv[e] = r.id;
        }
    }
    // (the sort writes s_k only after a barrier)
    if (!block_radix_sort<MAXM, E>(w, m, s_k, s_p, s_cnt, s_tmp)) block_merge_sort<MAXM, E>(m, s_k, s_p);
    tid = scat_tid();     // (a fresh copy: positions from it are not held through the sort)
#pragma unroll
    for (int e = 0; e < kPerThread; ++e) {
        const uint32_t i = tid + (uint32_t)e * T;
        if (i < m) s_cnt[i] = idv[e];
    }
    __syncthreads();
    // the input index of every sorted position, read before finish_position
    // overwrites its slot in perm (a segment of an earlier round reads it there)
    uint32_t ids[kPerThread];
#pragma unroll
    for (int e = 0; e < kPerThread; ++e) {
        const uint32_t i = tid + (uint32_t)e * T;
        ids[e] = 0;
        if (i < m) ids[e] = s_cnt[s_p[i]];
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kPerThread; ++e) {
        const uint32_t i = tid + (uint32_t)e * T;
        if ((uint32_t)e * T >= m) break;     // (uniform) no position of this pass is in the block
        const bool act = i < m;     // sorted position
        bool eqp = false, eqn = false;
        key64 kk = 0, pk = 0;
        if (act) {
            kk = s_k[i];
            if (i > 0) pk = s_k[i - 1];
            eqp = i > 0 && pk == kk;
            eqn = i + 1 < m && s_k[i + 1] == kk;
            finish_position(B, beg + i, ids[e], kk, i > 0, pk, depth, F);
            if (top && (i == 0 || i == m - 1)) B.bkey[beg + i] = kk;
        }
        // a run of equal keys without a NUL continues at the next depth (its
        // strings are in perm): a run of at most
        // kTinyT strings is finished below by this workgroup, a longer one is
        // a segment of the next round
        const bool nr = act && !eqp && eqn && !key_ends(kk, F);
        if (__ballot(nr) == 0) continue;     // (uniform) nothing to append in this wave
        uint32_t rl = 0;
        if (nr) {     // the run's last position: binary search in the sorted keys
            uint32_t lo = i + 1, hi = m;     // s_k[lo] == kk, s_k[hi] != kk (or hi == m)
            while (hi - lo > 1) {
                const uint32_t mid = (lo + hi) >> 1;
                if (s_k[mid] == kk) lo = mid;
                else hi = mid;
            }
            rl = lo - i + 1;
        }
        const bool small = nr && rl <= kTinyT;
        const uint32_t slot = small ? atomicAdd(&s_nruns, 1u) : kMaxRuns;
        const bool keep = slot < kMaxRuns;
        if (keep) s_runs[slot] = (i << 16) | rl;
        if (TAIL) {
            if (nr && !small) {
                const uint32_t t = atomicAdd(&ts->n, 1u);
                if (t < kTailStack) {
                    ts->pos[t] = beg + i;
                    ts->len[t] = rl;
                    ts->depth[t] = depth + F.cpk;
                } else {
                    flag_error(B.cnt, ERR_BOUNDS);     // (pending runs are disjoint: cannot happen)
                }
            }
        } else {
            Item ni = { beg + i, rl, beg + i, F_NEXT, depth + F.cpk, 0u };
            if (nr && !small) B.sdepth_out[(beg + i) >> kDepthShift] = depth + F.cpk;
            wave_append_segment(nr && !keep, ni, nxt);
        }
    }
    __syncthreads();     // the runs' indices written above are visible to the whole group
    const uint32_t nruns = min(s_nruns, kMaxRuns);
    for (uint32_t r0 = 0; r0 < nruns; r0 += kBlockRuns) {     // (uniform) batches of at most kBlockRuns runs
        block_finish_runs<NK>(B, s_k, s_runs + r0, min(kBlockRuns, nruns - r0), beg, depth + F.cpk, T / 64);
        if (TAIL) __syncthreads();     // the next batch reuses the batch table
    }
}

// A block in tail mode, finished completely by its workgroup.
template <uint32_t MAXM, int E, int NK>
__device__ __forceinline__ void block_tail(Item cur, const Bufs& B, const Sink& nxt, BlockLds<MAXM, E, true>& S, TailStack& ts)
{
    if (tid_x() == 0) ts.n = 0;
    // (every thread reads ts.n after block_one, which returns at once on
    // a malformed item: the count is stored before a barrier each time)
    __syncthreads();
    uint32_t d = seg_depth(B, cur.rbeg);
    for (bool top = true;; top = false) {     // one call site, so that block_one stays inline
        block_one<MAXM, E, NK, true>(cur, B, nxt, d, S, &ts, top);
        // (the pushes precede a barrier in block_one's finish pass)
        const uint32_t n = min(ts.n, kTailStack);
        if (n == 0) break;     // (uniform)
        __syncthreads();     // the last pass's LDS is no longer read, every thread has read ts.n
        cur = Item{ ts.pos[n - 1], ts.len[n - 1], ts.pos[n - 1], F_NEXT, 0u, 0u };
        d = ts.depth[n - 1];
        if (tid_x() == 0) ts.n = n - 1;     // (pushes into the freed entry come after block_one's barriers)
        __syncthreads();     // every thread has read the top entry; the count is stored
    }
}

// Blocks [first, last) of a list (one per workgroup), or with LOOP (levels
// planned on the device) from *p_first to the list's count, each workgroup
// looping over them; a count over the list's capacity has been flagged and
// is clamped.
//
// TAIL (host-planned, the round's last work: no large segments and no
// equal-key chunks are left): the workgroup finishes its block completely,
// sorting each long run again at its next depth until every string is
// decided, so the sort needs no further round.
template <uint32_t MAXM, int E, bool LOOP, int NK, bool TAIL>
__global__ __launch_bounds__(MAXM / E) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_block(const Item* items, uint32_t first, uint32_t last,
                                                     const uint32_t* p_first, const uint32_t* cnt_items, uint32_t cap,
                                                     Bufs B, Sink nxt)
{
    __shared__ BlockLds<MAXM, E, TAIL> S;
    if constexpr (TAIL) {
        static_assert(!LOOP, "tail mode is host-planned");
        __shared__ TailStack ts;
        const uint32_t idx = first + blockIdx.x;
        if (idx >= min(last, cap)) return;
        block_tail<MAXM, E, NK>(items[idx], B, nxt, S, ts);
    } else if constexpr (!LOOP) {
        const uint32_t idx = first + blockIdx.x;
        if (idx >= min(last, cap)) return;
        const Item L = items[idx];
        block_one<MAXM, E, NK, false>(L, B, nxt, seg_depth(B, L.rbeg), S, nullptr, true);
    } else {
        const uint32_t lo = *p_first, hi = min(*cnt_items, cap);
        for (uint32_t idx = lo + blockIdx.x; idx < hi; idx += gridDim.x) {
            __syncthreads();     // the previous block's LDS is no longer read
            const Item L = items[idx];
            block_one<MAXM, E, NK, false>(L, B, nxt, seg_depth(B, L.rbeg), S, nullptr, true);
        }
    }
}

constexpr uint32_t kRunRow = 512;       // runs of a row that k_leaf_run searches

// Characters that string a (from offset off on) shares with the string whose
// next characters are ref[]: at most 64, and none past a NUL of it.
constexpr int kExtKeys = 8;
__device__ __forceinline__ uint32_t common_chars(const Bufs& B, const key64 (&ref)[kExtKeys], uint64_t off)
{
    key64 a[kExtKeys];
    load_keys<kExtKeys>(B.arena, B.alen, off, a);
    uint32_t n = 8 * kExtKeys;
#pragma unroll
    for (int i = kExtKeys - 1; i >= 0; --i) {     // (the first difference or end counts)
        if (a[i] != ref[i]) n = 8 * i + lcp_key(a[i], ref[i]);
        else if ((ref[i] & 0xFFull) == 0) n = 8 * i + key_depth(ref[i]);
    }
    return n;
}

// One chunk of an equal-key leaf (all keys equal), by a workgroup of kWG threads.
//
// A run that continues is a segment of the next round, at the depth its
// strings are known to share.  Strings with a common prefix (URLs of one host)
// share more than one key: without looking ahead, every 8 characters of the
// prefix cost a round of tree, partition and host round trips that split
// nothing.  If 64 strings of the chunk agree in their next character, every
// string of it is compared with the run's first one over 64 characters, and
// the run continues after what they all share.  4.4 M URL-like strings
// (prefixes of 8 to 40 characters, 256 MB): 3.07 -> 1.40 ms, 2 instead of 5
// rounds with large segments.  The sample looks at one key only: most runs of a
// text share nothing more, and over 64 characters it took half as long as the
// rest (20 M windows in plain keys, 65 K runs of 300 strings: 850 -> 549 us).
__device__ __forceinline__ void run_chunk(const Item& L, const Bufs& B, const Sink& nxt, RunMap<kRunChunk>& M)
{
    const uint32_t c = L.flags >> kFlagShift;
    if (!item_ok(L, B) || (uint64_t)c * kRunChunk >= L.size || (L.flags & (F_IDENT | F_NEXT))) {
        if (tid_x() == 0) flag_error(B.cnt, ERR_BOUNDS);
        return;
    }
    const Runs R = runs_of(B, L);
    const uint32_t rend = L.begin + L.size;
    const uint32_t cb = L.begin + c * kRunChunk;
    const uint32_t m = min(rend - cb, kRunChunk);
    // a short row (a bucket of a small segment) is copied and searched, a
    // long one mapped
    uint32_t* s_v = M.delta;
    const bool small = R.nch <= kRunRow;     // (uniform)
    if (small) {
        for (uint32_t i = tid_x(); i < R.nch; i += kWG) {
            s_v[i] = R.V[i];
            s_v[kRunRow + i] = R.S[i];
        }
        __syncthreads();
    } else {
        map_runs<kWaves, (int)kRunChunk>(R, rend, cb, m, M);
    }
    auto place = [&](uint32_t p) {
        if (!small) return mapped_place(B, M, p);
        const uint32_t r = find_run(s_v, R.nch, cb + p);
        return checked_place(B, s_v[kRunRow + r] + (cb + p - s_v[r]));
    };
    const key64 key = rec_key(R.R[place(0u)]);
    const KeyFmt F = key_fmt(L.flags);
    const uint32_t depth = seg_depth(B, L.rbeg);
    // identical strings are done, others continue at the next depth
    const bool term = key_ends(key, F), single = L.size == 1;
    const uint32_t l = depth + key_depth(key, F);
#pragma unroll 4
    for (uint32_t p = tid_x(); p < m; p += kWG) {
        B.perm[cb + p] = R.R[place(p)].id;
        if (term && B.lcp && cb + p > L.begin) B.lcp[cb + p] = l;
    }
    if (!term) {     // (uniform)
        const uint32_t next = depth + F.cpk;
        const uint32_t id0 = R.R[run_place(B, R, L.begin)].id;
        key64 ref[kExtKeys];     // (in vector registers: the scalar ones are short)
        uint32_t zero;
        asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
        load_keys<kExtKeys>(B.arena, B.alen, str_off(B, min(id0, B.n - 1)) + next + zero, ref);
        // all waves take the same sample
        const uint32_t lane = lane_id();
        const uint32_t sp = (uint32_t)(((uint64_t)lane * m) >> 6);
        const key64 ks = string_key(B, R.R[place(sp)].id, next);
        uint32_t ext = 0;
        if (__ballot((ref[0] ^ ks) >> 56 != 0 || (ks >> 56) == 0) == 0) {     // (uniform) a character at least
            ext = 8 * kExtKeys;
#pragma unroll 4     // (1: 549 -> 577 us, the URL-like strings' runs 220 -> 236)
            for (uint32_t p = tid_x(); p < m; p += kWG) {
                const uint32_t id = R.R[place(p)].id;
                ext = min(ext, common_chars(B, ref, str_off(B, min(id, B.n - 1)) + next));
            }
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) ext = min(ext, (uint32_t)__shfl_xor((int)ext, d, 64));     // (this wave's strings)
        }
        if (lane == 0) atomicMin(&B.sdepth_out[L.begin >> kDepthShift], next + ext);
    }
    if (tid_x() < 64) {
        const bool nr = tid_x() == 0 && c == 0 && !term && !single;
        Item ni = { L.begin, L.size, L.begin, F_NEXT, 0u, 0u };
        wave_append_segment(nr, ni, nxt);
        if (tid_x() == 0) {
            if (c == 0) B.bkey[L.begin] = key;
            if (cb + m == rend) B.bkey[rend - 1] = key;
        }
    }
}

// The chunks of equal-key leaves from *p_first (first, if null) to entry `end` of a list.
__global__ __launch_bounds__(kWG) void k_leaf_run(const Item* items, const uint32_t* p_first, uint32_t first,
                                                  const uint32_t* cnt_items, uint32_t end, Bufs B, Sink nxt)
{
    __shared__ RunMap<kRunChunk> M;
    if (B.pending && *B.pending) {      // the round's levels are not finished
        if (B.pending_err && tid_x() == 0) flag_error(B.cnt, ERR_LEVELS);
        return;
    }
    const uint32_t nitems = min(*cnt_items, end);     // (an overflow of the list has been flagged)
    if (p_first) first = *p_first;
    for (uint32_t ii = first + blockIdx.x; ii < nitems; ii += gridDim.x) {
        __syncthreads();     // the previous chunk's map is no longer read
        run_chunk(load_uniform(items + ii), B, nxt, M);
    }
}

// Few leaves of all kinds in one launch (host-planned): workgroups of
// kLeavesWG threads, the largest blocks first; waves that a leaf has no use
// for end at once (a barrier waits for those that are left).  Kernels of one
// kind each run after one another, and with few leaves each lasts as long as
// its slowest workgroup, 20 to 40 us.  40 K strings of ACGT: 147 -> 117 us.
struct LeafRange {
    const Item* list;
    uint32_t first, count;
};
struct LeafSet {          // kinds: tiny, blocks by class, equal-key chunks
    LeafRange r[kBlkClasses + 2];
};
constexpr uint32_t kLeavesWG = kBlkT / kBlkE3;
constexpr uint32_t kLeavesTiny = kLeavesWG / 64;     // tiny leaves of a workgroup

template <uint32_t MAXM, int E, int NK, bool TAIL>
__device__ __forceinline__ void leaves_block(const Item L, const Bufs& B, const Sink& nxt, BlockLds<MAXM, E, TAIL>& S, TailStack& ts)
{
    if constexpr (TAIL) block_tail<MAXM, E, NK>(L, B, nxt, S, ts);
    else block_one<MAXM, E, NK, false>(L, B, nxt, seg_depth(B, L.rbeg), S, nullptr, true);
}
template <int NK, bool TAIL>
__global__ __launch_bounds__(kLeavesWG) __attribute__((amdgpu_waves_per_eu(5))) void k_leaves(LeafSet Q, Bufs B, Sink nxt)
{
    union Lds {
        BlockLds<kBlkT, kBlkE3, TAIL> b3;
        BlockLds<1024, kBlkE2, TAIL> b2;
        RunMap<kRunChunk> m;
        struct { key64 k[kLeavesTiny][64]; uint32_t i[kLeavesTiny][64], r[kLeavesTiny][64]; } t;
    };
    __shared__ Lds S;
    __shared__ TailStack ts;
    uint32_t i = blockIdx.x;
#define PS5_LEAVES_BLOCK(J, M, E, LDS)                                                  \
    if (i < Q.r[J].count) {                                                             \
        if (tid_x() >= (M) / (E)) return;     /* (whole waves) */                       \
        leaves_block<M, E, NK, TAIL>(Q.r[J].list[Q.r[J].first + i], B, nxt, LDS, ts);   \
        return;                                                                         \
    }                                                                                   \
    i -= Q.r[J].count;
    PS5_LEAVES_BLOCK(4, kBlkT, kBlkE3, S.b3)
    PS5_LEAVES_BLOCK(3, 1024, kBlkE2, S.b2)
    // (smaller blocks have as many waves: their LDS is reserved anyway, and a
    // block's runs of equal keys are finished a wave each)
    PS5_LEAVES_BLOCK(2, 1024, kBlkE2, S.b2)
    PS5_LEAVES_BLOCK(1, 1024, kBlkE2, S.b2)
#undef PS5_LEAVES_BLOCK
    if (i < Q.r[5].count) {
        if (tid_x() < kWG) run_chunk(load_uniform(Q.r[5].list + Q.r[5].first + i), B, nxt, S.m);
        return;
    }
    i -= Q.r[5].count;
    const uint32_t w = wave_id(), t = i * kLeavesTiny + w;
    if (t < Q.r[0].count)
        tiny_leaf<NK>(load_uniform(Q.r[0].list + __builtin_amdgcn_readfirstlane((int)(Q.r[0].first + t))), B, S.t.k[w], S.t.i[w], S.t.r[w]);
}

// LCP between neighbouring leaves of one round segment:
// depth + lcp_key(last key of the left leaf, first key of the right leaf)
// (sample_sort_lcp, .hpp:311-396).
struct LeafLists {        // the leaf lists of a round, concatenated in this order
    const Item* list[kBlkClasses + 2];   // tiny, blocks by class, equal-key chunks
    int cnt[kBlkClasses + 2];            // their counters (indices into the counter array)
    uint32_t cap[kBlkClasses + 2];       // their capacities (an overflow has been flagged)
};

__global__ __launch_bounds__(kWG) void k_leafbound(LeafLists LL, Bufs B)
{
    constexpr int NL = kBlkClasses + 2;
    if (B.pending && *B.pending) {      // the round's levels are not finished
        if (B.pending_err && tid_x() == 0) flag_error(B.cnt, ERR_LEVELS);
        return;
    }
    uint32_t end[NL];        // running totals of the list lengths
    uint32_t run = 0;
#pragma unroll
    for (int j = 0; j < NL; ++j) end[j] = run += min(B.cnt[LL.cnt[j]], LL.cap[j]);
    for (uint32_t i = blockIdx.x * kWG + tid_x(); i < end[NL - 1]; i += gridDim.x * kWG) {
        int l = 0;
#pragma unroll
        for (int j = 0; j < NL - 1; ++j) l += i >= end[j] ? 1 : 0;
        const Item L = LL.list[l][i - (l ? end[l - 1] : 0u)];
        if (l == NL - 1 && (L.flags >> kFlagShift) != 0) continue;   // only the first chunk of an equal-key leaf
        if (L.begin <= L.rbeg || !B.lcp) continue;
        if (L.begin >= B.n) { flag_error(B.cnt, ERR_BOUNDS); continue; }
        const key64 a = B.bkey[L.begin - 1], c = B.bkey[L.begin];
        if (a == c) { flag_error(B.cnt, ERR_LCP); continue; }
        B.lcp[L.begin] = seg_depth(B, L.rbeg) + lcp_key(a, c, key_fmt(L.flags));
    }
}

// Batch outputs: input index -> index inside its set (perm[pos] - first of
// the set holding pos; a set occupies the same positions as its inputs).
// A workgroup takes kLocTile positions: two lanes find the sets holding its
// first and last position, and each position searches only between them
// (no search at all in the common case of a tile inside one set).
constexpr uint32_t kLocTile = 16 * kWG;
__global__ __launch_bounds__(kWG) void k_localize(uint32_t* perm, uint32_t n, const uint64_t* set_first,
                                                   uint32_t nsets)
{
    __shared__ uint32_t s_set[2];
    const uint32_t t0 = blockIdx.x * kLocTile;
    if (t0 >= n) return;
    const uint32_t t1 = (uint32_t)min<uint64_t>(n, (uint64_t)t0 + kLocTile);
    if (tid_x() < 2) {
        const uint32_t pos = tid_x() == 0 ? t0 : t1 - 1;
        uint32_t lo = 0, hi = nsets;   // largest s with set_first[s] <= pos
        while (lo + 1 < hi) {
            const uint32_t mid = (lo + hi) / 2;
            if (set_first[mid] <= pos) lo = mid;
            else hi = mid;
        }
        s_set[tid_x()] = lo;
    }
    __syncthreads();
    const uint32_t s0 = s_set[0], s1 = s_set[1];
    if (s0 == s1 && ((uintptr_t)perm & 15) == 0) {     // (uniform) one set: one base, 16-byte accesses
        const uint32_t base = (uint32_t)set_first[s0];
        for (uint32_t q = t0 + 4 * tid_x(); q < t1; q += 4 * kWG) {
            if (q + 4 <= t1) {
                uint4 v = *reinterpret_cast<const uint4*>(perm + q);
                v.x -= base;
                v.y -= base;
                v.z -= base;
                v.w -= base;
                *reinterpret_cast<uint4*>(perm + q) = v;
            } else {
                for (uint32_t pos = q; pos < t1; ++pos) perm[pos] -= base;
            }
        }
        return;
    }
    for (uint32_t pos = t0 + tid_x(); pos < t1; pos += kWG) {
        uint32_t lo = s0, hi = s1 + 1;
        while (lo + 1 < hi) {
            const uint32_t mid = (lo + hi) / 2;
            if (set_first[mid] <= pos) lo = mid;
            else hi = mid;
        }
        perm[pos] -= (uint32_t)set_first[lo];
    }
}

// Distinguishing characters of a sorted order: cache[i] = s_i[lcp[i]] for
// i >= 1, the first character in which the i-th string differs from its
// predecessor, NUL when they are equal (set_cache in sample_sort_lcp,
// bingmann-parallel_sample_sort.hpp:366,385; fill_lcp, stringptr.hpp:950-958;
// checked by verify_lcp_cache, stringptr.hpp:1015-1021).  lcp[i] never
// exceeds the length of s_i, so the byte read is inside the string.
__global__ __launch_bounds__(kWG) void k_dist_chars(const uint8_t* arena, const uint32_t* offs,
                                                    const uint32_t* perm, const uint32_t* lcp, uint32_t n,
                                                    uint8_t* cache, uint32_t* cnt, uint64_t alen)
{
    const uint32_t i = blockIdx.x * kWG + tid_x();
    if (i == 0 || i >= n) return;
    const uint64_t p = (uint64_t)offs[perm[i]] + lcp[i];
    if (p >= alen) { flag_error(cnt, ERR_BOUNDS); return; }
    cache[i] = arena[p];
}

// ptrs[i] = base + offs[perm[i]]: the sorted strings' host pointers
__global__ __launch_bounds__(kWG) void k_gather_ptrs(const uint32_t* perm, const uint32_t* offs, uint64_t base,
                                                     uint64_t n, uint64_t* ptrs)
{
    const uint64_t i = (uint64_t)blockIdx.x * kWG + tid_x();
    if (i < n) ptrs[i] = base + offs[perm[i] < n ? perm[i] : 0u];
}

// wide[i] = lcp[i] as uint64 (entry 0 is copied too; callers skip it)
__global__ __launch_bounds__(kWG) void k_widen_lcp(const uint32_t* lcp, uint64_t n, uint64_t* wide)
{
    const uint64_t i = (uint64_t)blockIdx.x * kWG + tid_x();
    if (i < n) wide[i] = lcp[i];
}

// offs64[i] = base[s] + offs32[i] for the set s holding string i
__global__ __launch_bounds__(kWG) void k_widen(const uint32_t* offs32, const uint64_t* first, const uint64_t* base,
                                               uint32_t nsets, uint64_t n, uint64_t* offs64)
{
    const uint64_t i = (uint64_t)blockIdx.x * kWG + tid_x();
    if (i >= n) return;
    uint32_t lo = 0, hi = nsets;   // largest s with first[s] <= i
    while (lo + 1 < hi) {
        const uint32_t mid = (lo + hi) / 2;
        if (first[mid] <= i) lo = mid;
        else hi = mid;
    }
    offs64[i] = base[lo] + offs32[i];
}

// ---- LCP-aware merge of sorted runs ---------------------------------------

// Compare strings a and b (arena offsets) that share their first h
// characters: returns true if a <= b, and their LCP in *lcp.
__device__ __forceinline__ bool str_leq_from(const uint8_t* arena, uint64_t alen, uint64_t a, uint64_t b,
                                             uint32_t h, uint32_t* lcp)
{
    for (;;) {
        const key64 ka = load_key(arena, alen, a + h), kb = load_key(arena, alen, b + h);
        if (ka != kb) {
            *lcp = h + lcp_key(ka, kb);
            return ka < kb;
        }
        if ((ka & 0xFFull) == 0) {   // both end inside this key: equal strings
            *lcp = h + key_depth(ka);
            return true;
        }
        h += 8;
    }
}

// One round of pairwise merges.  Pair p merges runs A = [first[p], mid[p])
// and B = [mid[p], first[p+1]) of (idx, lcp) into the same positions of the
// output; lcp[q] is the LCP of the strings at q-1 and q within a run (its
// first entry unused).  The output of a pair is cut into tiles of kMergeT
// positions, one workgroup each.  k_merge_part finds, for the first output
// of every tile, how many strings of A precede it (a merge-path co-rank,
// by string comparisons; equal strings take A first, so ties keep run
// order).  k_merge_tile stages the tile's strings of A and B in LDS (index,
// LCP and their first 8 characters), places each thread's kMergeE outputs by
// a co-rank inside the tile, and emits them with the binary LCP merge
// (lcp_merge_binary and lcp_compare, bingmann-lcp_mergesort_binary.hpp),
// which compares characters only where the LCPs to the previous output do
// not decide; the staged characters decide most of those compares without
// touching the arena.  The first round takes the 8 characters from keys
// extracted in input order by one streaming pass (a gather of 8 bytes per
// string instead of an offset and an arena window); every round writes them
// beside its outputs for the next.
// (outputs per thread: a thread's co-rank and LCP chain are serial, and the
// tile's LDS sets how many workgroups hide them.  8 runs of 2 M strings: 977 us
// with 8, 851 with 4, 974 with 2)
constexpr uint32_t kMergeE = 4;
constexpr uint32_t kMergeT = kWG * kMergeE;        // outputs per tile

// a <= b for strings a, b (input indices) whose first 8 characters are ka, kb
__device__ __forceinline__ bool merge_leq(const Bufs& B, uint32_t a, uint32_t b, key64 ka, key64 kb,
                                          uint32_t* lcp)
{
    if (ka != kb) {
        *lcp = lcp_key(ka, kb);
        return ka < kb;
    }
    if ((ka & 0xFFull) == 0) {
        *lcp = key_depth(ka);
        return true;
    }
    return str_leq_from(B.arena, B.alen, str_off(B, a), str_off(B, b), 8, lcp);
}

// first 8 characters of the string at position pos of the source: from the
// previous round's output, else from in_key (indexed by input index)
__device__ __forceinline__ key64 merge_key(const Bufs& B, const uint32_t* src_idx, const key64* src_key,
                                           const key64* in_key, uint64_t pos)
{
    if (src_key) return src_key[pos];
    const uint32_t id = src_idx[pos];
    if (id < B.n) return in_key[id];
    flag_error(B.cnt, ERR_BOUNDS);
    return 0;
}

// the pair holding tile g: the largest p with tstart[p] <= g
__device__ __forceinline__ uint32_t merge_pair(const uint64_t* tstart, uint32_t npairs, uint64_t g)
{
    uint32_t lo = 0, hi = npairs;
    while (lo + 1 < hi) {
        const uint32_t m = (lo + hi) / 2;
        if (tstart[m] <= g) lo = m;
        else hi = m;
    }
    return lo;
}

// co[g] = strings of A (of g's pair) that precede the first output of tile g.
// LANES lanes search together, each testing one of as many positions evenly
// spread over what is left.  A test is a chain of dependent gathers, and
// halving the range takes 21 of them one after another for runs of 2 M strings;
// more lanes take fewer steps and more gathers, which is what counts when the
// tiles are many.  A round of less than kMergeFew tiles takes 8 lanes, of more
// 4, of kMergeMany or more one.  8 runs, us:
//   strings        8 lanes   4      2      1
//   1 M (ASCII)       98    103    116    129
//   4 M              224    231    242    262
//   16 M             835    814    822    852
//   64 M            3340   3233   3178   3136
constexpr uint64_t kMergeFew = 8192, kMergeMany = 32768;
template <uint32_t LANES>
__global__ __launch_bounds__(kWG) void k_merge_part(Bufs B, const uint32_t* src_idx, const key64* src_key,
                                                    const key64* in_key,
                                                    const uint64_t* first, const uint64_t* mid,
                                                    const uint64_t* tstart, uint32_t npairs, uint32_t* co)
{
    const uint64_t g = ((uint64_t)blockIdx.x * kWG + tid_x()) / LANES;
    if (g >= tstart[npairs]) return;
    const uint32_t p = merge_pair(tstart, npairs, g);
    const uint64_t a0 = first[p], b0 = mid[p];
    const uint64_t la = b0 - a0, lb = first[p + 1] - b0;
    const uint64_t diag = (g - tstart[p]) * kMergeT;
    uint64_t i0 = diag > lb ? diag - lb : 0, i1 = min(diag, la);
    const uint32_t lane = lane_id(), l = lane % LANES;
    while (i0 < i1) {     // (the same for the tile's lanes)
        // A[mi] precedes this tile up to some mi in [i0, i1), and none from there on
        const uint64_t step = (i1 - i0 + 1 + LANES) / (LANES + 1);
        const uint64_t mi = i0 + (l + 1) * step - 1;
        bool before = false;
        if (mi < i1) {
            const uint64_t pa = a0 + mi, pb = b0 + diag - 1 - mi;
            const key64 ka = merge_key(B, src_idx, src_key, in_key, pa), kb = merge_key(B, src_idx, src_key, in_key, pb);
            uint32_t lcp;
            // (indices are needed only where the keys do not decide)
            before = ka != kb || (ka & 0xFFull) == 0 ? ka <= kb
                                                     : merge_leq(B, src_idx[pa], src_idx[pb], ka, kb, &lcp);
        }
        const uint64_t ones = (__ballot(before) >> (lane - l)) & ((1ull << LANES) - 1);
        const uint32_t t = (uint32_t)__popcll(ones);
        i0 += t * step;
        i1 = min(i1, i0 + step - 1);     // (lane t's position, if it is in the range, does not precede)
    }
    if (l == 0) co[g] = (uint32_t)i0;
}

// Where keys do not decide, every comparison is a chain of gathers from the
// arena.  A thread finds its first output by ten comparisons, and knows from
// them what its heads share with the output before it, but at the tile's
// ends.  With half, every second thread searches between its neighbours' places
// only: a chain of 12 comparisons, but 6 or 7 for each thread on average.  In a
// round of kMergeHalf tiles or more, which the gathers' traffic bounds, that
// is less (16 M strings of ACGT in 8 runs 5.01 ms, 6.08 without half, 7.56 when
// every thread also compared its heads with the output before it; 16 M of
// ASCII, whose keys decide, 0.81, 0.80 and 0.82); below, the chain counts
// (8 runs of 0.3 M strings: ACGT 171 us with half, 155 without, URL-like ones
// 353 and 308).  The line lies where 8 runs of URL-like strings, whose
// comparisons are the longest, begin to gain (0.5 M 385 and 360 us, 0.7 M 412
// and 524, 1 M 534 and 782); windows gain later (1 M 484 and 431), ASCII, digits
// and ACGT lose 1 to 2% between.
constexpr uint64_t kMergeHalf = 768;
__global__ __launch_bounds__(kWG) void k_merge_tile(Bufs B, const uint32_t* src_idx, const uint32_t* src_lcp,
                                                    const key64* src_key, const key64* in_key,
                                                    uint32_t* dst_idx, uint32_t* dst_lcp,
                                                    key64* dst_key, const uint64_t* first, const uint64_t* mid,
                                                    const uint64_t* tstart, uint32_t npairs, const uint32_t* co,
                                                    bool half)
{
    // slots [0, na+1): A[ia0-1 .. ia1), slots [na+1, na+nb+2): B[jb0-1 .. jb1);
    // slot 0 of a part is unused when the part starts its run
    __shared__ key64 s_key[kMergeT + 2];
    __shared__ uint32_t s_idx[kMergeT + 2];
    __shared__ uint32_t s_lcp[kMergeT + 2];
    __shared__ uint16_t s_oslot[kMergeT];
    __shared__ uint32_t s_olcp[kMergeT];
    const uint64_t g = blockIdx.x;
    const uint32_t p = merge_pair(tstart, npairs, g);
    const uint64_t a0 = first[p], b0 = mid[p];
    const uint64_t la = b0 - a0, lb = first[p + 1] - b0;
    const uint64_t diag0 = (g - tstart[p]) * kMergeT;
    const uint32_t len = (uint32_t)min((uint64_t)kMergeT, la + lb - diag0);
    const uint64_t ia0 = co[g], ia1 = g + 1 < tstart[p + 1] ? co[g + 1] : la;
    const uint64_t jb0 = diag0 - ia0;
    const uint32_t na = (uint32_t)(ia1 - ia0), nb = len - na;
    const uint32_t sb = na + 1;        // first slot of B
    for (uint32_t k = tid_x(); k < len + 2; k += kWG) {
        uint64_t pos;
        bool valid;
        if (k < sb) {
            valid = k > 0 || ia0 > 0;
            pos = a0 + ia0 + k - 1;
        } else {
            valid = k > sb || jb0 > 0;
            pos = b0 + jb0 + (k - sb) - 1;
        }
        if (valid) {
            s_idx[k] = src_idx[pos];
            s_lcp[k] = src_lcp[pos];
            s_key[k] = merge_key(B, src_idx, src_key, in_key, pos);
        }
    }
    __syncthreads();
    auto leq = [&](uint32_t x, uint32_t y, uint32_t* l) {
        return merge_leq(B, s_idx[x], s_idx[y], s_key[x], s_key[y], l);
    };
    // strings of A among the tile's first d outputs, known to be in [i0, i1];
    // l1: the LCP of A[i-1] and B[j], l2: of B[j-1] and A[i], where the search
    // compared them
    constexpr uint32_t kNoLcp = 0xFFFFFFFFu;
    auto corank = [&](uint32_t d, uint32_t i0, uint32_t i1, uint32_t* l1, uint32_t* l2) {
        *l1 = *l2 = kNoLcp;
        while (i0 < i1) {
            const uint32_t mi = (i0 + i1) / 2;
            uint32_t l;
            if (leq(1 + mi, sb + d - mi, &l)) {     // A[mi] <= B[d-1-mi]
                i0 = mi + 1;
                *l1 = l;
            } else {
                i1 = mi;
                *l2 = l;
            }
        }
        return i0;
    };
    const uint32_t d = tid_x() * kMergeE;
    uint32_t i = 0, j = 0, l1 = kNoLcp, l2 = kNoLcp;
    uint32_t lo = d > nb ? d - nb : 0, hi = min(d, na);
    bool found = false;
    if (half) {     // (uniform) every second thread's first output is searched
                    // in the whole tile, by half of the threads; the others'
                    // lie between their neighbours'
        uint32_t* s_co = s_olcp;       // co-rank, l1, l2 of kWG / 2 threads
        static_assert(3 * (kWG / 2) <= kMergeT, "they fit the outputs' memory");
        const uint32_t t = tid_x(), d2 = 2 * d;
        if (t < kWG / 2 && d2 < len) {
            s_co[t] = corank(d2, d2 > nb ? d2 - nb : 0, min(d2, na), &l1, &l2);
            s_co[kWG / 2 + t] = l1;
            s_co[kWG + t] = l2;
        }
        __syncthreads();
        if (d < len) {
            i = s_co[t / 2];
            l1 = s_co[kWG / 2 + t / 2];
            l2 = s_co[kWG + t / 2];
            found = t % 2 == 0;
            lo = max(lo, i);
            hi = min(hi, min(d + kMergeE < len ? s_co[t / 2 + 1] : na, i + kMergeE));
        }
        __syncthreads();     // (their memory takes the outputs)
    }
    uint32_t lcpa = 0, lcpb = 0;       // LCPs of the next A and B string with the previous output
    if (d < len) {
        if (!found) i = corank(d, lo, hi, &l1, &l2);
        j = d - i;
        // the previous output is the larger one of A[i-1] and B[j-1], and of two
        // strings before a third the larger shares at least as much with it
        const bool hasa = ia0 + i > 0, hasb = jb0 + j > 0;
        if (i < na) {
            if (hasa) lcpa = s_lcp[1 + i];
            if (hasb) {
                if (l2 == kNoLcp) leq(sb + j, 1 + i, &l2);
                lcpa = max(lcpa, l2);
            }
        }
        if (j < nb) {
            if (hasb) lcpb = s_lcp[sb + 1 + j];
            if (hasa) {
                if (l1 == kNoLcp) leq(i, sb + 1 + j, &l1);
                lcpb = max(lcpb, l1);
            }
        }
        const uint32_t nout = min(kMergeE, len - d);
        for (uint32_t q = 0; q < nout; ++q) {
            bool take_a;
            uint32_t lab = 0;     // LCP of the two heads
            if (j >= nb) take_a = true;
            else if (i >= na) take_a = false;
            else if (lcpa == lcpb) {
                const uint32_t x = 1 + i, y = sb + 1 + j;
                if (lcpa < 8) take_a = leq(x, y, &lab);
                else take_a = str_leq_from(B.arena, B.alen, str_off(B, s_idx[x]), str_off(B, s_idx[y]), lcpa, &lab);
            }
            else if (lcpa > lcpb) { take_a = true; lab = lcpb; }
            else { take_a = false; lab = lcpa; }
            if (take_a) {
                s_oslot[d + q] = (uint16_t)(1 + i);
                s_olcp[d + q] = lcpa;
                ++i;
                lcpa = i < na ? s_lcp[1 + i] : 0u;
                lcpb = lab;
            } else {
                s_oslot[d + q] = (uint16_t)(sb + 1 + j);
                s_olcp[d + q] = lcpb;
                ++j;
                lcpb = j < nb ? s_lcp[sb + 1 + j] : 0u;
                lcpa = lab;
            }
        }
    }
    __syncthreads();
    const uint64_t o0 = a0 + diag0;
    for (uint32_t k = tid_x(); k < len; k += kWG) {
        const uint32_t s = s_oslot[k];
        dst_idx[o0 + k] = s_idx[s];
        dst_lcp[o0 + k] = s_olcp[k];
        if (dst_key) dst_key[o0 + k] = s_key[s];
    }
}

// plain copy of 16-byte words (calibrates the HBM byte counters)
__global__ __launch_bounds__(kWG) void k_copy16(const uint4* src, uint4* dst, uint64_t n16)
{
    for (uint64_t i = (uint64_t)blockIdx.x * kWG + tid_x(); i < n16; i += (uint64_t)gridDim.x * kWG)
        dst[i] = src[i];
}

// sum of the sizes of a work list range (profiling only)
__global__ __launch_bounds__(kWG) void k_sum_sizes(const Item* items, uint32_t first, const uint32_t* cnt_items,
                                                    unsigned long long* out)
{
    __shared__ uint32_t s_tmp[16];
    const uint32_t n = *cnt_items;
    uint32_t v = 0;
    for (uint32_t i = first + blockIdx.x * kWG + tid_x(); i < n; i += gridDim.x * kWG) {
        const Item it = items[i];
        if (it.flags & F_SORTED) {   // a chunk of an equal-key leaf
            const uint32_t c = it.flags >> kFlagShift, cb = c * kRunChunk;
            v += cb < it.size ? min(kRunChunk, it.size - cb) : 0u;
        } else {
            v += it.size;
        }
    }
    uint32_t tot;
    block_excl_scan<kWaves>(v, &tot, s_tmp);
    if (tid_x() == 0 && tot) atomicAdd(out, (unsigned long long)tot);
}

// ===========================================================================
// host side
// ===========================================================================

namespace {

thread_local std::string g_err;

int set_err(int code, const char* fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_err = buf;
    return code;
}

static_assert(kChunkLimit == kPartMax, "the largest chunk");

#define HIPCHK(x)                                                                  \
    do {                                                                           \
        hipError_t _e = (x);                                                       \
        if (_e != hipSuccess)                                                      \
            return set_err(PS5_ERR_HIP, "%s failed: %s (%s:%d)", #x,               \
                           hipGetErrorString(_e), __FILE__, __LINE__);             \
    } while (0)

enum KernelId {
    K_TREE, K_PART, K_HIST, K_CHILDREN, K_BLOCK,
    K_LEAF_TINY, K_LEAF_RUN, K_LEAFBOUND, K_MISC, K_NUM
};
const char* kKernelNames[K_NUM] = {
    "k_tree", "k_part", "k_hist", "k_children", "k_block",
    "k_leaf_tiny", "k_leaf_run", "k_leafbound", "k_misc"
};

enum { S_BLOCK, S_TINY, S_RUN, S_NUM };

// The work buffers of a sort of up to `cap` strings.  A context owns one set
// (grown with hipMalloc on demand); the allocation-free entry point swaps in
// a set carved from the static device scratch for the duration of a call.
struct WorkBuffers {
    bool fixed = false;              // carved from the static scratch: never grown or freed
    uint64_t cap = 0;
    uint32_t* rec = nullptr;         // two buffers of cap records, one after the other
    key64* bkey = nullptr;
    uint32_t* sdepth[2] = { nullptr, nullptr };
    // large segments: first level of a round [round parity], later levels [level parity]
    Item* l_round[2] = { nullptr, nullptr };
    Item* l_lvl[2] = { nullptr, nullptr };
    // leaves of a round [round parity]
    Item* l_tiny[2] = { nullptr, nullptr };
    Item* l_block[2] = { nullptr, nullptr };
    Item* l_run[2] = { nullptr, nullptr };
    uint32_t cap_large = 0, cap_block = 0, cap_tiny[2] = { 0, 0 }, cap_run = 0;
    Item* h_large = nullptr;         // pinned copy of a large list
    // plan of a level: its nlarge descriptors followed by its tile table, in
    // one buffer so that one copy uploads both
    unsigned char* d_plan = nullptr;
    unsigned char* h_plan = nullptr;     // pinned, mapped: the host's plans are pulled by k_fetch
    unsigned char* h_plan_dev = nullptr; // its device address
    uint64_t tiles_cap = 0, groups_cap = 0;
    uint8_t* lut = nullptr;          // kRootCode bytes per large segment (cap_large of them)
    // bucket counts of a level (hist_cap entries), their group sums and the
    // segments' splitters (gsum_cap entries each), and the run tables
    // (hist_cap entries for each of the two buffers)
    uint32_t* hist = nullptr;
    uint32_t* vpos = nullptr;
    uint32_t* src = nullptr;
    uint64_t hist_cap = 0;
    uint32_t* gsum = nullptr;
    key64* trees = nullptr;
    uint64_t gsum_cap = 0;
};

// List capacities of a sort of up to cap strings (each list bounds what the
// device can append to it; an overflow is flagged, never written).
constexpr uint32_t cap_large_of(uint64_t cap) { return (uint32_t)(cap / kBlkT + 16); }
constexpr uint32_t cap_block_of(uint64_t cap) { return (uint32_t)(cap / kTinyT + 16); }
// Tiny leaves: a batch may consist of as many sets; later rounds' (odd first)
// come from runs of two strings or more, or are buckets of segments with at
// most a sixteenth as many buckets as strings.
constexpr uint32_t cap_tiny_of(uint64_t cap, int rp) { return (uint32_t)(rp ? cap / 4 * 3 + 16 : cap + 16); }
// an equal-key run of m > kTinyT strings yields ceil(m / kRunChunk) <= m / 64 chunks
constexpr uint32_t cap_run_of(uint64_t cap) { return (uint32_t)(cap / 64 + 16); }
// every large segment has at most size / kChunkMin + 1 chunks
constexpr uint64_t tiles_cap_of(uint64_t cap) { return cap / kChunkMin + cap_large_of(cap) + 1; }
constexpr uint64_t groups_cap_of(uint64_t cap) { return tiles_cap_of(cap) / kHistGroup + cap_large_of(cap) + 1; }
// Entries of a level's bucket counts and of its run tables: segments of S
// strings in all, in chunks of `limit` keys, have at most 2048 S / limit +
// S / 16 (2 << treebits is at most 2048 and at most a sixteenth of a segment,
// the leaf target being 64 or more); a level of min_tiles chunks or fewer has
// chunks of kChunkMin or more keys.
constexpr uint64_t hist_cap_of(uint64_t cap, uint64_t chunk_max, uint64_t min_tiles)
{
    const uint64_t limit = chunk_max < (uint64_t)kPartMax ? chunk_max : (uint64_t)kPartMax;
    const uint64_t few = cap < kChunkMin * min_tiles ? cap : kChunkMin * min_tiles, many = cap * 2048 / limit;
    return (few > many ? few : many) + cap / 16 + 4096;
}
constexpr uint64_t sdepth_cap_of(uint64_t cap) { return (cap >> kDepthShift) + 1; }
// per bucket its first position and one sum per group of chunks
constexpr uint64_t gsum_cap_of(uint64_t cap, uint64_t hist_cap) { return hist_cap / kHistGroup + cap / 8 + 8192; }
// a plan: the level header, cap_large descriptors, the tables of chunks and groups
constexpr uint64_t plan_tiles_off(uint64_t cap)
{
    return sizeof(LevelHdr) + (uint64_t)cap_large_of(cap) * sizeof(LargeDesc);
}
constexpr uint64_t plan_groups_off(uint64_t cap) { return plan_tiles_off(cap) + tiles_cap_of(cap) * sizeof(TileRef); }
constexpr uint64_t plan_bytes_of(uint64_t cap) { return plan_groups_off(cap) + groups_cap_of(cap) * sizeof(TileRef); }
static_assert(sizeof(LevelHdr) % 8 == 0 && sizeof(LargeDesc) % 8 == 0 && sizeof(TileRef) % 8 == 0,
              "a plan is copied in 8-byte words");
Plan plan_view(unsigned char* base, uint64_t cap)
{
    Plan P;
    P.hdr = reinterpret_cast<const LevelHdr*>(base);
    P.desc = reinterpret_cast<LargeDesc*>(base + sizeof(LevelHdr));
    P.tiles = reinterpret_cast<const TileRef*>(base + plan_tiles_off(cap));
    P.groups = reinterpret_cast<const TileRef*>(base + plan_groups_off(cap));
    return P;
}

}  // namespace

struct ps5_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    hipStream_t side = nullptr;         // a round's leaves run here beside its last blocks
    hipEvent_t ev_fork = nullptr, ev_join = nullptr;
    WorkBuffers w;                   // the buffers run_sort uses
    // the allocation-free entry point: pinned plan buffers sized for the
    // scratch's largest sort (allocated with the context), and the scratch's
    // device address on this context's device
    Item* na_h_large = nullptr;
    unsigned char* na_h_plan = nullptr;
    unsigned char* na_h_plan_dev = nullptr;
    unsigned char* na_scratch = nullptr;
    uint32_t* d_cnt = nullptr;
    uint32_t* h_cnt = nullptr;       // pinned
    // counters + head of a list, written by k_stage straight into mapped
    // host memory (no copy engine on the readback path)
    unsigned char* h_stage = nullptr;    // pinned, mapped, coherent
    unsigned char* h_stage_dev = nullptr;    // its device address
    uint32_t stage_seq = 0;                  // sequence number of the last staged copy
    uint32_t pending_root = 0;               // strings of a single root whose set-up the next plan fetch does
    Item* h_roots = nullptr;         // pinned, mapped: root items of a batch, kind by kind
    Item* h_roots_dev = nullptr;     // its device address
    uint64_t roots_cap = 0;
    uint64_t* d_merge = nullptr;     // plan of a merge round
    uint64_t merge_cap = 0;
    uint32_t cus = 256;                 // CUs, rounded down to a multiple of kXcds
    uint64_t* d_sets = nullptr;      // set boundaries of a batch
    uint64_t sets_cap = 0;
    unsigned long long* d_sums = nullptr;   // profiling: elements per kernel class
    unsigned long long* h_sums = nullptr;
    // tuning
    uint32_t leaf_target = 768;      // strings per block the multi-workgroup levels aim for
    uint32_t max_treebits = kMaxTreebits;   // splitter-tree depth limit of one level
    uint32_t max_oversample = 32;    // sample keys per splitter (limited by kMaxSamples)
    // tile shapes of the multi-workgroup levels and the leaf passes' key width
    uint32_t chunk_max = kShapeChunkMax;     // keys per chunk, ordinary levels (at most kPartMax take effect)
    uint32_t chunk_max_root = kShapeChunkMaxRoot;    // the same in a level of roots
    uint32_t min_tiles = kMinTiles;          // a small level's chunks shrink to give this many tiles
    uint32_t leaf_keys = 8;                  // keys a leaf pass fetches per string at a time
    uint64_t seed = 0x5EED5EEDull;
    int planning = 0;                // 0: levels planned on the host, 1: on the device (no host synchronisation
                                     // inside a round), 2: on the device for a single sort of fewer than
                                     // kAutoDevMax strings, else on the host
    // a sort's first rounds as one captured HIP graph (0: off), and the
    // instantiated graph of the last sort, replayed while its inputs match
    uint32_t graph_rounds = 0;
    hipGraph_t graph = nullptr;
    hipGraphExec_t graph_exec = nullptr;
    std::vector<uint64_t> graph_key;
    uint64_t w_gen = 0;              // bumped whenever a work buffer is allocated again
    bool tail_blocks = true;         // a round's last blocks finish every string (PS5_TAIL_BLOCKS=0: off)
    bool chain_levels = true;        // a host-planned level's successor is planned on the device, without a
                                     // read-back between them (PS5_CHAIN_LEVELS=0: off)
    uint32_t graph_levels = 0;       // non-zero: fewer levels per captured round (PS5_GRAPH_LEVELS; tests
                                     // use it to reach the host-planned fallback)
    // profiling
    bool profile = false;
    bool trace = false;              // PS5_TRACE set: per-round work to stderr (diagnostics)
    std::vector<hipEvent_t> ev_pool;
    std::vector<std::pair<int, std::pair<hipEvent_t, hipEvent_t>>> ev_used;
    double k_ms[K_NUM] = {};
    uint64_t k_launch[K_NUM] = {};
    uint64_t k_bytes[K_NUM] = {};
    uint64_t st_rounds = 0, st_levels = 0, st_segments = 0, st_leaves = 0, st_syncs = 0;
};

namespace {

void free_tables(ps5_ctx* c)
{
    for (uint32_t** q : { &c->w.hist, &c->w.gsum, &c->w.vpos, &c->w.src }) {
        if (*q) (void)hipFree(*q);
        *q = nullptr;
    }
    if (c->w.trees) (void)hipFree(c->w.trees);
    c->w.trees = nullptr;
    c->w.hist_cap = c->w.gsum_cap = 0;
}

void free_buffers(ps5_ctx* c)
{
    if (c->w.fixed) {     // views into the static scratch: nothing to free
        c->w = WorkBuffers();
        return;
    }
    auto f = [](void* p) { if (p) (void)hipFree(p); };
    for (int i = 0; i < 2; ++i) {
        f(c->w.l_round[i]); f(c->w.l_lvl[i]);
        f(c->w.l_tiny[i]); f(c->w.l_block[i]); f(c->w.l_run[i]); f(c->w.sdepth[i]);
        c->w.l_round[i] = nullptr; c->w.l_lvl[i] = nullptr;
        c->w.l_tiny[i] = nullptr; c->w.l_block[i] = nullptr; c->w.l_run[i] = nullptr;
        c->w.sdepth[i] = nullptr;
    }
    f(c->w.rec); f(c->w.bkey); f(c->w.lut); f(c->w.d_plan);
    c->w.rec = nullptr; c->w.bkey = nullptr; c->w.lut = nullptr; c->w.d_plan = nullptr;
    free_tables(c);
    if (c->w.h_large) (void)hipHostFree(c->w.h_large);
    if (c->w.h_plan) (void)hipHostFree(c->w.h_plan);
    c->w.h_large = nullptr; c->w.h_plan = nullptr; c->w.h_plan_dev = nullptr;
    c->w.cap = 0;
    c->w.tiles_cap = c->w.groups_cap = 0;
}

// The splitter trees, bucket counts and run tables of any level of a sort of
// the context's capacity and shape.  Called before a sort, when its stream is
// idle; they keep their size until the capacity or the shape asks for more
// (a level's tables are still read by the leaves of the one before).
int ensure_tables(ps5_ctx* c)
{
    const uint64_t hist = hist_cap_of(c->w.cap, std::min(c->chunk_max, c->chunk_max_root), c->min_tiles);
    const uint64_t gsum = gsum_cap_of(c->w.cap, hist);
    if (hist <= c->w.hist_cap && gsum <= c->w.gsum_cap) return PS5_OK;
    if (c->w.fixed) return set_err(PS5_ERR_CAPACITY, "the scratch holds no tables of this shape");
    free_tables(c);
    HIPCHK(hipMalloc(&c->w.hist, hist * sizeof(uint32_t)));
    HIPCHK(hipMalloc(&c->w.gsum, gsum * sizeof(uint32_t)));
    HIPCHK(hipMalloc(&c->w.trees, gsum * sizeof(key64)));
    HIPCHK(hipMalloc(&c->w.vpos, 2 * hist * sizeof(uint32_t)));
    HIPCHK(hipMalloc(&c->w.src, 2 * hist * sizeof(uint32_t)));
    c->w.hist_cap = hist;
    c->w.gsum_cap = gsum;
    c->w_gen++;
    return PS5_OK;
}

int ensure_capacity(ps5_ctx* c, uint64_t n)
{
    if (n <= c->w.cap) return PS5_OK;
    if (c->w.fixed)
        return set_err(PS5_ERR_CAPACITY, "%llu strings exceed the scratch's %llu", (unsigned long long)n,
                       (unsigned long long)c->w.cap);
    // a context that has to grow again grows by half at least
    uint64_t cap = std::max<uint64_t>(std::max<uint64_t>(n, 1024), c->w.cap + c->w.cap / 2);
    cap = std::min<uint64_t>(cap, std::max<uint64_t>(n, 0xFFFFFF00ull));
    free_buffers(c);
    HIPCHK(hipMalloc(&c->w.rec, 2 * cap * kRecWords * sizeof(uint32_t)));
    HIPCHK(hipMalloc(&c->w.bkey, cap * sizeof(key64)));
    for (int i = 0; i < 2; ++i) HIPCHK(hipMalloc(&c->w.sdepth[i], sdepth_cap_of(cap) * sizeof(uint32_t)));
    c->w.cap_large = cap_large_of(cap);
    c->w.cap_block = cap_block_of(cap);
    for (int i = 0; i < 2; ++i) c->w.cap_tiny[i] = cap_tiny_of(cap, i);
    c->w.cap_run = cap_run_of(cap);
    for (int i = 0; i < 2; ++i) {
        HIPCHK(hipMalloc(&c->w.l_round[i], (uint64_t)c->w.cap_large * sizeof(Item)));
        HIPCHK(hipMalloc(&c->w.l_lvl[i], (uint64_t)c->w.cap_large * sizeof(Item)));
        HIPCHK(hipMalloc(&c->w.l_tiny[i], (uint64_t)c->w.cap_tiny[i] * sizeof(Item)));
        HIPCHK(hipMalloc(&c->w.l_block[i], (uint64_t)kBlkClasses * c->w.cap_block * sizeof(Item)));
        HIPCHK(hipMalloc(&c->w.l_run[i], (uint64_t)c->w.cap_run * sizeof(Item)));
    }
    HIPCHK(hipMalloc(&c->w.lut, (uint64_t)c->w.cap_large * kRootCode));
    c->w.tiles_cap = tiles_cap_of(cap);
    c->w.groups_cap = groups_cap_of(cap);
    const uint64_t plan_bytes = plan_bytes_of(cap);
    HIPCHK(hipMalloc(&c->w.d_plan, plan_bytes));
    HIPCHK(hipHostMalloc(reinterpret_cast<void**>(&c->w.h_large), (uint64_t)c->w.cap_large * sizeof(Item)));
    HIPCHK(hipHostMalloc(reinterpret_cast<void**>(&c->w.h_plan), plan_bytes, hipHostMallocMapped | hipHostMallocCoherent));
    HIPCHK(hipHostGetDevicePointer(reinterpret_cast<void**>(&c->w.h_plan_dev), c->w.h_plan, 0));
    c->w.cap = cap;
    c->w_gen++;
    return PS5_OK;
}

// ---- the allocation-free entry point's device scratch -----------------------
//
// ps5_sort_device_noalloc takes every work buffer of a sort of up to
// kNoAllocMaxStrings strings from `scratch`, a static device array: each GPU
// the library runs on holds its own copy from the time the code object is
// loaded until the process ends.  Host code never uses the array's name as a
// device address; the address is resolved once per device with
// hipGetSymbolAddress (scratch_address) and kept in the context.
constexpr uint64_t kScratchBytes = 104ull << 20;
constexpr uint64_t kNoAllocMaxStrings = 1ull << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

// Byte offsets of the work buffers of a sort of up to `cap` strings of the
// given shape in one piece of memory, and their sum.
struct WorkLayout {
    uint64_t rec, bkey, sdepth[2], lut, l_round[2], l_lvl[2], l_tiny[2], l_block[2], l_run[2];
    uint64_t desc, trees, hist, gsum, vpos, src, total;
    uint64_t hist_cap, gsum_cap;
};
constexpr uint64_t align256(uint64_t x) { return (x + 255) / 256 * 256; }
constexpr WorkLayout work_layout(uint64_t cap, uint64_t chunk_max, uint64_t min_tiles)
{
    WorkLayout L{};
    uint64_t o = 0;
    auto take = [&o](uint64_t bytes) { const uint64_t at = o; o = align256(o + bytes); return at; };
    const uint64_t cl = cap_large_of(cap), cb = cap_block_of(cap), cr = cap_run_of(cap);
    L.rec = take(2 * cap * kRecWords * sizeof(uint32_t));
    L.bkey = take(cap * sizeof(key64));
    for (int i = 0; i < 2; ++i) L.sdepth[i] = take(sdepth_cap_of(cap) * sizeof(uint32_t));
    for (int i = 0; i < 2; ++i) {
        L.l_round[i] = take(cl * sizeof(Item));
        L.l_lvl[i] = take(cl * sizeof(Item));
        L.l_tiny[i] = take(cap_tiny_of(cap, i) * sizeof(Item));
        L.l_block[i] = take(kBlkClasses * cb * sizeof(Item));
        L.l_run[i] = take(cr * sizeof(Item));
    }
    L.desc = take(plan_bytes_of(cap));
    L.lut = take(cl * kRootCode);
    L.hist_cap = hist_cap_of(cap, chunk_max, min_tiles);
    L.hist = take(L.hist_cap * sizeof(uint32_t));
    L.vpos = take(2 * L.hist_cap * sizeof(uint32_t));
    L.src = take(2 * L.hist_cap * sizeof(uint32_t));
    L.gsum_cap = gsum_cap_of(cap, L.hist_cap);
    L.gsum = take(L.gsum_cap * sizeof(uint32_t));
    L.trees = take(L.gsum_cap * sizeof(key64));
    L.total = o;
    return L;
}
// the scratch's layout: tables for any shape (chunks of kChunkMin keys)
constexpr WorkLayout scratch_layout() { return work_layout(kNoAllocMaxStrings, kChunkMin, kMinTiles); }
static_assert(scratch_layout().total <= kScratchBytes, "the scratch holds the work buffers of its largest sort");

// Device address of `scratch` on `device` (the caller has made it current):
// resolved on the first call per device and remembered.
int scratch_address(int device, unsigned char** out)
{
    static std::mutex mu;
    static std::map<int, unsigned char*> addr;
    std::lock_guard<std::mutex> g(mu);
    auto it = addr.find(device);
    if (it == addr.end()) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return set_err(PS5_ERR_HIP, "hipGetSymbolAddress(scratch) on device %d failed: %s", device,
                           hipGetErrorString(e));
        it = addr.emplace(device, static_cast<unsigned char*>(p)).first;
    }
    *out = it->second;
    return PS5_OK;
}

// Calls of the allocation-free entry point on one device share its scratch:
// they are serialised per device inside this process.
std::mutex& scratch_mutex(int device)
{
    static std::mutex mus[64];
    return mus[(unsigned)device % 64u];
}

// Work buffers of a sort of up to kNoAllocMaxStrings strings carved from the
// scratch at `base` (its device address), with the context's pinned plan
// buffers.  Nothing is allocated.
WorkBuffers scratch_buffers(unsigned char* base, Item* h_large, unsigned char* h_plan, unsigned char* h_plan_dev)
{
    constexpr WorkLayout L = scratch_layout();
    const uint64_t cap = kNoAllocMaxStrings;
    WorkBuffers w;
    w.fixed = true;
    w.cap = cap;
    for (int i = 0; i < 2; ++i) {
        w.l_round[i] = reinterpret_cast<Item*>(base + L.l_round[i]);
        w.l_lvl[i] = reinterpret_cast<Item*>(base + L.l_lvl[i]);
        w.l_tiny[i] = reinterpret_cast<Item*>(base + L.l_tiny[i]);
        w.l_block[i] = reinterpret_cast<Item*>(base + L.l_block[i]);
        w.l_run[i] = reinterpret_cast<Item*>(base + L.l_run[i]);
        w.sdepth[i] = reinterpret_cast<uint32_t*>(base + L.sdepth[i]);
        w.cap_tiny[i] = cap_tiny_of(cap, i);
    }
    w.rec = reinterpret_cast<uint32_t*>(base + L.rec);
    w.vpos = reinterpret_cast<uint32_t*>(base + L.vpos);
    w.src = reinterpret_cast<uint32_t*>(base + L.src);
    w.bkey = reinterpret_cast<key64*>(base + L.bkey);
    w.cap_large = cap_large_of(cap);
    w.cap_block = cap_block_of(cap);
    w.cap_run = cap_run_of(cap);
    w.h_large = h_large;
    w.d_plan = base + L.desc;
    w.h_plan = h_plan;
    w.h_plan_dev = h_plan_dev;
    w.tiles_cap = tiles_cap_of(cap);
    w.groups_cap = groups_cap_of(cap);
    w.trees = reinterpret_cast<key64*>(base + L.trees);
    w.lut = base + L.lut;
    w.hist = reinterpret_cast<uint32_t*>(base + L.hist);
    w.hist_cap = L.hist_cap;
    w.gsum = reinterpret_cast<uint32_t*>(base + L.gsum);
    w.gsum_cap = L.gsum_cap;
    return w;
}

struct Launch {   // counts a launch; brackets it with events when profiling
    ps5_ctx* c;
    int id;
    hipEvent_t a = nullptr, b = nullptr;
    Launch(ps5_ctx* c_, int id_, uint64_t bytes) : c(c_), id(id_)
    {
        c->k_launch[id]++;
        c->k_bytes[id] += bytes;
        if (!c->profile) return;
        a = take();
        b = take();
        (void)hipEventRecord(a, c->stream);
    }
    ~Launch()
    {
        if (!c->profile) return;
        (void)hipEventRecord(b, c->stream);
        c->ev_used.push_back({ id, { a, b } });
    }
    hipEvent_t take()
    {
        if (c->ev_pool.empty()) {
            hipEvent_t e;
            (void)hipEventCreate(&e);
            return e;
        }
        hipEvent_t e = c->ev_pool.back();
        c->ev_pool.pop_back();
        return e;
    }
};

void collect_events(ps5_ctx* c)
{
    for (auto& u : c->ev_used) {
        float ms = 0;
        if (hipEventElapsedTime(&ms, u.second.first, u.second.second) == hipSuccess) c->k_ms[u.first] += ms;
        c->ev_pool.push_back(u.second.first);
        c->ev_pool.push_back(u.second.second);
    }
    c->ev_used.clear();
}

// sink: large -> `large` list, leaves -> lists of round parity `rp`
Sink make_sink(ps5_ctx* c, Item* large, int c_large, int rp)
{
    Sink s;
    s.large = large;
    s.block = c->w.l_block[rp];
    s.tiny = c->w.l_tiny[rp];
    s.run = c->w.l_run[rp];
    s.cnt = c->d_cnt;
    s.c_large = c_large;
    s.c_block = C_BLOCK + rp;
    s.c_tiny = C_TINY + rp;
    s.c_run = C_RUN + rp;
    s.c_runcont = C_RUNCONT + rp;
    s.cap_large = c->w.cap_large;
    s.cap_block = c->w.cap_block;
    s.cap_tiny = c->w.cap_tiny[rp];
    s.cap_run = c->w.cap_run;
    return s;
}

// copy the counters (and the large list `list` with counter `ci`) to the host
// Wait until the staged copy's sequence number reads `seq`, rather than for
// the stream to go idle: the host sees the number as soon as the GPU writes
// it.  The stream is queried every 1024 spins, so that a failed stream ends
// the wait with its error.
constexpr uint32_t kGraphSeqPending = 0xFFFFFFFFu;     // set by the host before a captured graph's replay
int wait_stage(ps5_ctx* c, uint32_t seq)
{
    const uint32_t* f = reinterpret_cast<const uint32_t*>(c->h_stage + kStageSeq);
    for (uint32_t spin = 1;; ++spin) {
        if (__atomic_load_n(f, __ATOMIC_ACQUIRE) == seq) return PS5_OK;
        if ((spin & 1023) == 0) {
            const hipError_t e = hipStreamQuery(c->stream);
            if (e == hipSuccess) {
                if (__atomic_load_n(f, __ATOMIC_ACQUIRE) == seq) return PS5_OK;
                return set_err(PS5_ERR_INTERNAL, "the staged copy's sequence number never arrived");
            }
            if (e != hipErrorNotReady) return set_err(PS5_ERR_HIP, "waiting for a staged copy: %s", hipGetErrorString(e));
        }
        __builtin_ia32_pause();
    }
}

// (not a status of the ABI) the sort's packed keys met a character outside
// their alphabet: run_sort starts over
constexpr int kStartOver = -1;

int readback(ps5_ctx* c, const Item* list, int ci)
{
    // one staged copy holds the counters and the head of the list
    uint32_t seq = ++c->stage_seq;
    if (seq == 0 || seq == kGraphSeqPending) seq = c->stage_seq = 1;     // (values the graph path uses)
    hipLaunchKernelGGL(k_stage, dim3(1), dim3(kWG), 0, c->stream, c->d_cnt, list, ci, c->h_stage_dev, seq);
    HIPCHK(hipGetLastError());
    int rc = wait_stage(c, seq);
    if (rc) return rc;
    c->st_syncs++;
    memcpy(c->h_cnt, c->h_stage, C_NCNT * sizeof(uint32_t));
    if (c->h_cnt[C_ERR] & ERR_ALPHA) return kStartOver;
    if (c->h_cnt[C_ERR] & ERR_CAP) return set_err(PS5_ERR_CAPACITY, "work list capacity exceeded");
    if (c->h_cnt[C_ERR] & ERR_LCP) return set_err(PS5_ERR_INTERNAL, "equal keys across a leaf boundary");
    if (c->h_cnt[C_ERR] & ERR_BOUNDS) return set_err(PS5_ERR_INTERNAL, "device bounds check failed");
    if (c->h_cnt[C_ERR] & ERR_LEVELS) return set_err(PS5_ERR_INTERNAL, "a captured round needed more levels");
    if (list) {
        const uint32_t nl = c->h_cnt[ci];
        if (nl > c->w.cap_large) return set_err(PS5_ERR_CAPACITY, "large list overflow");
        memcpy(c->w.h_large, c->h_stage + kStageHead, std::min(nl, kPeek) * sizeof(Item));
        if (nl > kPeek) {
            HIPCHK(hipMemcpyAsync(c->w.h_large + kPeek, list + kPeek, (nl - kPeek) * sizeof(Item),
                                  hipMemcpyDeviceToHost, c->stream));
            HIPCHK(hipStreamSynchronize(c->stream));
            c->st_syncs++;
        }
    }
    return PS5_OK;
}

uint32_t div_up(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

void sum_sizes(ps5_ctx* c, const Item* list, uint32_t first, const uint32_t* cnt, uint32_t n, int slot)
{
    if (!c->profile || n == 0) return;
    hipLaunchKernelGGL(k_sum_sizes, dim3(std::min<uint32_t>(div_up(n, kWG), 1024)), dim3(kWG), 0, c->stream,
                       list, first, cnt, c->d_sums + slot);
}

// Treebits of a multi-workgroup step on m strings: the fewest levels of at
// most 1023 splitters that bring buckets down to about leaf_target strings,
// with the fan-out spread evenly over those levels.
int large_treebits(uint32_t m, uint32_t target, int maxbits)
{
    const double need = std::log2(std::max(2.0, (double)m / target));
    const int levels = std::max(1, (int)std::ceil(need / maxbits));
    const int k = (int)std::ceil(need / levels);
    return std::max(1, std::min(maxbits, k));
}

void launch_tree(ps5_ctx* c, const Bufs& B, Plan P, uint32_t grid, uint64_t seed, int src)
{
    const auto f = src == kFromRuns ? k_tree<kFromRuns> : src == kRootPlain ? k_tree<kRootPlain>
                 : src == kRootPack ? k_tree<kRootPack> : k_tree<kFromPerm>;
    hipLaunchKernelGGL(f, dim3(grid), dim3(kBigWG), 0, c->stream, P, B, seed, c->w.trees);
}

// the k_part instance for trees of up to kmax treebits, with its LDS
using PartKernel = void (*)(Plan, Bufs, const key64*, uint32_t, int);
template <int NB>
PartKernel part_kernel_nb(int src)
{
    return src == kFromRuns ? k_part<NB, kFromRuns> : src == kRootPlain ? k_part<NB, kRootPlain>
         : src == kRootPack ? k_part<NB, kRootPack> : k_part<NB, kFromPerm>;
}
PartKernel part_kernel(int kmax, int src, uint32_t* lds)
{
    if (kmax <= 7) { *lds = PartLds<8>::kBytes; return part_kernel_nb<8>(src); }
    if (kmax == 8) { *lds = PartLds<9>::kBytes; return part_kernel_nb<9>(src); }
    if (kmax == 9) { *lds = PartLds<10>::kBytes; return part_kernel_nb<10>(src); }
    *lds = PartLds<11>::kBytes;
    return part_kernel_nb<11>(src);
}
void launch_part(ps5_ctx* c, const Bufs& B, Plan P, uint32_t grid, int kmax, int src, uint32_t ntiles, bool one)
{
    uint32_t lds = 0;
    const PartKernel f = part_kernel(kmax, src, &lds);
    hipLaunchKernelGGL(f, dim3(grid), dim3(kPartThreads), lds, c->stream, P, B, c->w.trees, ntiles, (int)one);
}
// bytes per string of a partition: its input, and key 8 + idx 4 written
uint64_t part_bytes(int src)
{
    return src == kFromRuns ? 8 + 4 + 12                 // key, idx
         : src == kFromPerm ? 4 + 4 + 8 + 12             // perm, offset, characters
                            : 4 + 8 + 12;                // offset, characters
}

// What follows a level's partition: bucket sizes, children, run tables.
void launch_hist(ps5_ctx* c, const Bufs& B, Plan P, const Sink& sink, uint32_t dst, int kmax, uint32_t g_sum,
                 uint32_t g_children, uint32_t g_runs, uint64_t hl, bool fused)
{
    const uint32_t nbs = 2u << kmax;
    if (g_sum) {     // (segments of more than one group of chunks)
        Launch L(c, K_HIST, hl * 4);
        hipLaunchKernelGGL(k_hist_sum, dim3(g_sum, div_up(nbs, kWG)), dim3(kWG), 0, c->stream, P, B);
    }
    {
        Launch L(c, K_CHILDREN, g_sum ? hl * 8 / kHistGroup : hl * 4);
        hipLaunchKernelGGL(k_children, dim3(g_children), dim3(kBigWG), 0, c->stream, P, B, c->w.trees, sink, dst, (int)fused);
    }
    if (!fused) {
        Launch L(c, K_HIST, hl * 12);
        hipLaunchKernelGGL(k_hist_runs, dim3(g_runs, div_up(nbs, 64)), dim3(kWG), 0, c->stream, P, B, (int)dst);
    }
}

// One multi-workgroup sample-sort step over all large segments of a level,
// planned on the host from the level's large list (read back into h_large).
// src: where the segments' strings are; dst: the buffer the level writes.
int large_step(ps5_ctx* c, const Bufs& B, uint32_t nlarge, const Sink& sink, uint64_t seed, int src, uint32_t dst)
{
    hipStream_t st = c->stream;
    uint64_t ntiles = 0, ngroups = 0, hl = 0, gs = 0, elems = 0;
    int kmax = 1;
    bool fused = true;
    if (nlarge > c->w.cap_large) return set_err(PS5_ERR_CAPACITY, "large list overflow");
    LevelHdr* h_hdr = reinterpret_cast<LevelHdr*>(c->w.h_plan);
    LargeDesc* h_descs = reinterpret_cast<LargeDesc*>(c->w.h_plan + sizeof(LevelHdr));
    TileRef* h_tiles = reinterpret_cast<TileRef*>(c->w.h_plan + plan_tiles_off(c->w.cap));
    TileRef* h_groups = reinterpret_cast<TileRef*>(c->w.h_plan + plan_groups_off(c->w.cap));
    for (uint32_t i = 0; i < nlarge; ++i) elems += c->w.h_large[i].size;
    const bool roots = src == kRootPlain || src == kRootPack;
    const uint64_t cmax = std::min<uint64_t>(roots ? c->chunk_max_root : c->chunk_max, kPartMax);
    const uint64_t climit = std::min<uint64_t>(cmax, std::max<uint64_t>(kChunkMin, div_up(elems, c->min_tiles)));
    for (uint32_t i = 0; i < nlarge; ++i) {
        const Item seg = c->w.h_large[i];
        const uint32_t T = div_up(seg.size, climit), G = hist_groups(T);
        LargeDesc& D = h_descs[i];
        D.seg = seg;
        D.nch = T;
        D.chunk = div_up(seg.size, T);   // <= climit: equal chunks, the last one short
        D.hist_base = (uint32_t)hl;
        D.gbase = (uint32_t)gs;
        D.k = (uint32_t)large_treebits(seg.size, c->leaf_target, (int)c->max_treebits);
        const uint32_t nspl = (1u << D.k) - 1;
        kmax = std::max(kmax, (int)D.k);
        D.oversample = std::max<uint32_t>(2, std::min<uint32_t>(c->max_oversample, (kMaxSamples / nspl) & ~1u));
        fused = fused && G == 1 && (uint64_t)T * (2u << D.k) <= kFusedRuns;
        if (ntiles + T > c->w.tiles_cap || ngroups + G > c->w.groups_cap)
            return set_err(PS5_ERR_CAPACITY, "chunk table capacity");
        for (uint32_t t = 0; t < T; ++t) h_tiles[ntiles + t] = TileRef{ i, t };
        for (uint32_t g = 0; g < G; ++g) h_groups[ngroups + g] = TileRef{ i, g };
        ntiles += T;
        ngroups += G;
        hl += (uint64_t)(2u << D.k) * T;
        gs += (uint64_t)(2u << D.k) * (G + 1);
        if (hl > c->w.hist_cap || hl > 0xFFFFFFFFull || gs > c->w.gsum_cap)
            return set_err(PS5_ERR_CAPACITY, "histogram capacity");
    }
    *h_hdr = LevelHdr{ nlarge, (uint32_t)ntiles, (uint32_t)ngroups, (uint32_t)kmax, { 0u, 0u, 0u, 0u } };
    {   // the plan: pulled from mapped host memory by a kernel (no copy engine)
        FetchArgs F;
        const uint64_t off[3] = { 0, plan_tiles_off(c->w.cap), plan_groups_off(c->w.cap) };
        F.words[0] = (sizeof(LevelHdr) + nlarge * sizeof(LargeDesc)) / 8;
        F.words[1] = ntiles * sizeof(TileRef) / 8;
        F.words[2] = ngroups * sizeof(TileRef) / 8;
        for (int k = 0; k < 3; ++k) {
            F.src[k] = reinterpret_cast<const uint64_t*>(c->w.h_plan_dev + off[k]);
            F.dst[k] = reinterpret_cast<uint64_t*>(c->w.d_plan + off[k]);
        }
        const dim3 g((uint32_t)std::min<uint64_t>(div_up(std::max(F.words[0], F.words[1]), kWG), 1024));
        if (c->pending_root)
            hipLaunchKernelGGL(k_root_fetch, g, dim3(kWG), 0, st, F, c->d_cnt, c->w.l_round[0], c->pending_root);
        else
            hipLaunchKernelGGL(k_fetch, g, dim3(kWG), 0, st, F);
        c->pending_root = 0;
    }
    const Plan P = plan_view(c->w.d_plan, c->w.cap);
    {
        Launch L(c, K_TREE, (uint64_t)nlarge * kMaxSamples * 8);
        launch_tree(c, B, P, nlarge, seed, src);
    }
    {
        Launch L(c, K_PART, elems * part_bytes(src) + hl * 4);
        launch_part(c, B, P, div_up(ntiles, kXcds) * kXcds, kmax, src, (uint32_t)ntiles, nlarge == 1);
    }
    launch_hist(c, B, P, sink, dst, kmax, ngroups > nlarge ? (uint32_t)ngroups : 0u, nlarge, (uint32_t)ngroups, hl, fused);
    c->st_segments += nlarge;
    return PS5_OK;
}

// Roots of a sort: one segment [0, n), or one per set of a batch (sets never
// mix: every set is its own round segment, so no LCP crosses a set border).
// h_cnt and h_large get what the first round finds in its lists.
int setup_roots(ps5_ctx* c, uint32_t n, const uint64_t* set_first, uint32_t nsets)
{
    hipStream_t st = c->stream;
    for (int i = 0; i < C_NCNT; ++i) c->h_cnt[i] = 0;
    if (!set_first) {
        Item* list; int ci;
        if (n <= kTinyT) { list = c->w.l_tiny[0]; ci = C_TINY; }
        else if (n <= kBlkT) {
            const int cls = block_class(n);
            list = c->w.l_block[0] + (uint64_t)cls * c->w.cap_block;
            ci = C_BLOCK + 2 * cls;
        }
        else { list = c->w.l_round[0]; ci = C_LROUND; }
        c->h_cnt[ci] = 1;
        if (ci == C_LROUND) c->w.h_large[0] = Item{ 0u, n, 0u, F_IDENT, 0u, 0u };
        Launch L(c, K_MISC, 0);
        hipLaunchKernelGGL(k_setup, dim3(1), dim3(64), 0, st, c->d_cnt, list, ci, n);
        HIPCHK(hipGetLastError());
        return PS5_OK;
    }
    // root items staged in mapped host memory and pulled by a kernel (the
    // last sort that read them is complete)
    if ((uint64_t)nsets > c->roots_cap) {
        const uint64_t want = std::max<uint64_t>(nsets, 2 * c->roots_cap);
        if (c->h_roots) (void)hipHostFree(c->h_roots);
        c->h_roots = nullptr;
        c->roots_cap = 0;
        HIPCHK(hipHostMalloc(reinterpret_cast<void**>(&c->h_roots), want * sizeof(Item),
                             hipHostMallocMapped | hipHostMallocCoherent));
        HIPCHK(hipHostGetDevicePointer(reinterpret_cast<void**>(&c->h_roots_dev), c->h_roots, 0));
        c->roots_cap = want;
    }
    // kinds: 0 tiny, 1..kBlkClasses blocks by size class, last large
    auto kind_of = [](uint32_t m) { return m <= kTinyT ? 0 : m <= kBlkT ? 1 + block_class(m) : kRootKinds - 1; };
    RootLists R{};
    for (uint32_t s = 0; s < nsets; ++s) {
        const uint64_t b = set_first[s], e = set_first[s + 1];
        if (e < b || e > n) return set_err(PS5_ERR_ARG, "set boundaries must be non-decreasing and <= n");
        if (e > b) R.count[kind_of((uint32_t)(e - b))]++;
    }
    if (R.count[kRootKinds - 1] > c->w.cap_large || R.count[0] > c->w.cap_tiny[0])
        return set_err(PS5_ERR_CAPACITY, "too many sets");
    uint32_t at[kRootKinds], total = 0;
    for (int k = 0; k < kRootKinds; ++k) {
        at[k] = total;
        total += R.count[k];
        const bool large = k == kRootKinds - 1;
        if (k > 0 && !large && R.count[k] > c->w.cap_block) return set_err(PS5_ERR_CAPACITY, "too many sets");
        R.dst[k] = k == 0 ? c->w.l_tiny[0] : large ? c->w.l_round[0] : c->w.l_block[0] + (uint64_t)(k - 1) * c->w.cap_block;
        R.counter[k] = k == 0 ? C_TINY : large ? C_LROUND : C_BLOCK + 2 * (k - 1);
        c->h_cnt[R.counter[k]] = R.count[k];
    }
    const uint32_t large0 = at[kRootKinds - 1];
    for (uint32_t s = 0; s < nsets; ++s) {
        const uint64_t b = set_first[s], e = set_first[s + 1];
        if (e > b) c->h_roots[at[kind_of((uint32_t)(e - b))]++] =
            Item{ (uint32_t)b, (uint32_t)(e - b), (uint32_t)b, F_IDENT, 0u, 0u };
    }
    memcpy(c->w.h_large, c->h_roots + large0, R.count[kRootKinds - 1] * sizeof(Item));
    R.src = c->h_roots_dev;
    Launch L(c, K_MISC, 0);
    hipLaunchKernelGGL(k_roots, dim3(std::min<uint32_t>(div_up(std::max(total, 1u), kWG), 1024)), dim3(kWG), 0, st, R,
                       c->d_cnt);
    HIPCHK(hipGetLastError());
    return PS5_OK;
}

constexpr uint32_t kMaxGraphRounds = 64;      // rounds one captured graph may hold
constexpr uint32_t kForkLeafGroups = 8192;    // leaf workgroups worth a side stream
// Workgroups per CU of one launch for all kinds of leaves (k_leaves).  Their
// LDS, that of the largest block each, fills a CU with four, so this is twice
// what the chip holds at once.  0.5 M digits (1020 workgroups): 201 us with
// the kinds' own kernels, 159 together; 512 sets, 4.7 K workgroups of two
// block classes and 0.4 K others: 363 us apart, 329 with the others together,
// 316 with those on the side stream, 338 with one of the classes as well.
constexpr uint32_t kFewLeavesPerCu = 8;
// Strings of the largest root from which on roots may pack their keys.
// Packing saves rounds and levels where keys repeat: 4.2 M suffixes of an ACGT
// text take 0.70 ms against 1.07 plain, 20 M windows 1.48 against 3.03.  The
// kernels that can pack cost those that do not a little: 0.5 to 1 M digits or
// ASCII strings 2-3%, URL-like ones 1-2%, less the larger they are (4.2 M: 0-1%).
// From 2^20 on packing gains 13-25% and more where it is of use (1 M suffixes
// 0.63 -> 0.55 ms, 1 M ACGT strings 0.31 -> 0.25); between 2^19 and 2^20 from
// nothing (0.64 and 0.9 M suffixes, 0.64 M ACGT strings) to 29% (0.75 M, where
// plain keys need one more level), below 2^19 from -8% (16 K suffixes) to 14%
// (0.25 M).  The smaller roots of a batch pack with its largest: the line drawn
// for each root took 2.37 ms for 192 sets of 1 K to 2 M strings (a third ACGT)
// instead of 2.21, since the plain ones then keep the batch's rounds going.
constexpr uint64_t kPackMin = 1u << 20;
constexpr uint64_t kChainMin = 1u << 22;       // strings of a level whose successor is chained on the device
// Automatic planning plans a single sort of fewer strings on the device, as
// its callers are told: one synchronisation per round.  The line was drawn
// where the two modes took the same time; the host now sees which leaves are
// few and launches them together, and is ahead at every size (39 K strings of
// ACGT: 115 us, 152 planned on the device; 0.5 M digits: 162 and 214; 4 M
// ASCII strings: 365 and 375).
constexpr uint64_t kAutoDevMax = 1u << 22;

// Largest grids of the device-planned levels: their kernels loop over the
// work the device lists, so these bound the workgroups of a launch.
constexpr uint32_t kDevTreeWgs = 512, kDevHistWgs = 1024, kDevChildWgs = 512,
                   kDevTinyWgs = 8192, kDevRunWgs = 2048, kDevBoundWgs = 1024;
static_assert(kBlkE0 == kBlkE1 && kBlkE1 == kBlkE2 && kBlkE2 == kBlkE3, "one thread count per 256 keys");

// Leaf grids for nt tiny leaves and nr equal-key chunks: the leaf kernels
// loop over their lists, and a bounded grid of them is far faster than a
// workgroup per leaf when leaves number in the millions.
uint32_t leaf_tiny_grid(uint64_t nt) { return (uint32_t)std::min<uint64_t>(kDevTinyWgs, div_up(nt, kWaves)); }
uint32_t leaf_run_grid(uint64_t nr) { return (uint32_t)std::min<uint64_t>(kDevRunWgs, nr); }

// Looping block kernels of size class cls: four workgroups per wave slot
// of the GPU (32 per CU)
uint32_t block_grid_full(const ps5_ctx* c, int cls)
{
    const uint32_t waves = (256u << cls) / (uint32_t)kBlkE0 / 64;
    return (uint32_t)((uint64_t)c->cus * 128 / waves);
}

// Blocks of size class cls and round parity rp: the list entries [first,
// first + count) (or, with dev_first, from the device counter C_BDONE + cls
// to the list's count), `grid` workgroups.
void launch_block_class(ps5_ctx* c, const Bufs& B, int rp, int cls, uint32_t first, uint32_t count, bool dev_first,
                        uint32_t grid, const Sink& nsink, bool tail = false, int flags = 0)
{
    const uint32_t last = first + count;
    hipStream_t st = c->stream;
    const Item* list = c->w.l_block[rp] + (uint64_t)cls * c->w.cap_block;
    const uint32_t* cnt = c->d_cnt + C_BLOCK + 2 * cls + rp;
    const uint32_t* pf = dev_first ? c->d_cnt + C_BDONE + cls : nullptr;
    const uint32_t cap = c->w.cap_block;
    // no more blocks than CUs: small ones are given more waves, which finish
    // more of their runs of equal keys at a time (167 URL-like strings: 40 -> 26 us)
    if (!dev_first && count <= (uint32_t)c->cus) cls = std::max(cls, 2);
    Launch L(c, K_BLOCK, 0);
    // the default key width (8 keys) has its own instances; others share one
#define PS5_BLOCK_LAUNCH(M, E, LOOP, TAIL)                                                                         \
    do {                                                                                                           \
        if (c->leaf_keys == 8)                                                                                     \
            hipExtLaunchKernelGGL((k_block<M, E, LOOP, 8, TAIL>), dim3(grid), dim3(M / E), 0, st, nullptr, nullptr, \
                                  flags, list, first, last, pf, cnt, cap, B, nsink);                                 \
        else                                                                                                       \
            hipExtLaunchKernelGGL((k_block<M, E, LOOP, 0, TAIL>), dim3(grid), dim3(M / E), 0, st, nullptr, nullptr, \
                                  flags, list, first, last, pf, cnt, cap, B, nsink);                                 \
    } while (0)
    if (dev_first) {
        if (cls == 0) PS5_BLOCK_LAUNCH(256, kBlkE0, true, false);
        else if (cls == 1) PS5_BLOCK_LAUNCH(512, kBlkE1, true, false);
        else if (cls == 2) PS5_BLOCK_LAUNCH(1024, kBlkE2, true, false);
        else PS5_BLOCK_LAUNCH(kBlkT, kBlkE3, true, false);
    } else if (tail) {
        if (cls == 0) PS5_BLOCK_LAUNCH(256, kBlkE0, false, true);
        else if (cls == 1) PS5_BLOCK_LAUNCH(512, kBlkE1, false, true);
        else if (cls == 2) PS5_BLOCK_LAUNCH(1024, kBlkE2, false, true);
        else PS5_BLOCK_LAUNCH(kBlkT, kBlkE3, false, true);
    } else {
        if (cls == 0) PS5_BLOCK_LAUNCH(256, kBlkE0, false, false);
        else if (cls == 1) PS5_BLOCK_LAUNCH(512, kBlkE1, false, false);
        else if (cls == 2) PS5_BLOCK_LAUNCH(1024, kBlkE2, false, false);
        else PS5_BLOCK_LAUNCH(kBlkT, kBlkE3, false, false);
    }
#undef PS5_BLOCK_LAUNCH
}

// Tiny leaves and equal-key chunks of round parity rp on stream s: n_tiny and
// n_run of them from the entries done.tiny and done.run on, and no more, since
// what is queued before may have listed leaves that the host does not count
// yet (with dev_first: from the counters C_TDONE and C_RDONE on, all that are
// listed), in grids of g_tiny and g_run workgroups (0 skips a list).
struct LeavesDone { uint32_t tiny = 0, run = 0; };
void launch_leaves(ps5_ctx* c, const Bufs& B, int rp, const Sink& nsink, LeavesDone done, bool dev_first,
                   uint32_t g_tiny, uint32_t g_run, uint64_t n_tiny, uint64_t n_run, hipStream_t s, int flags = 0)
{
    if (g_tiny) {
        const uint32_t* first = dev_first ? c->d_cnt + C_TDONE : nullptr;
        const uint32_t end = dev_first ? c->w.cap_tiny[rp] : (uint32_t)std::min<uint64_t>(c->w.cap_tiny[rp], done.tiny + n_tiny);
        {
            Launch L(c, K_LEAF_TINY, 0);
            const auto f = c->leaf_keys == 8 ? k_leaf_tiny<8> : k_leaf_tiny<0>;
            hipExtLaunchKernelGGL(f, dim3(g_tiny), dim3(kWG), 0, s, nullptr, nullptr, flags, c->w.l_tiny[rp], first,
                                  done.tiny, c->d_cnt + C_TINY + rp, end, B);
        }
        sum_sizes(c, c->w.l_tiny[rp], done.tiny, c->d_cnt + C_TINY + rp, (uint32_t)n_tiny, S_TINY);
    }
    if (g_run) {
        const uint32_t* first = dev_first ? c->d_cnt + C_RDONE : nullptr;
        const uint32_t end = dev_first ? c->w.cap_run : (uint32_t)std::min<uint64_t>(c->w.cap_run, done.run + n_run);
        {
            Launch L(c, K_LEAF_RUN, 0);
            hipExtLaunchKernelGGL(k_leaf_run, dim3(g_run), dim3(kWG), 0, s, nullptr, nullptr, flags, c->w.l_run[rp], first,
                                  done.run, c->d_cnt + C_RUN + rp, end, B, nsink);
        }
        sum_sizes(c, c->w.l_run[rp], done.run, c->d_cnt + C_RUN + rp, (uint32_t)n_run, S_RUN);
    }
}

// The kinds of leaves that go into one launch (k_leaves): of the blocks of
// round parity rp from blk_first on (nblk by class), and the nt tiny leaves
// and nr equal-key chunks from `done` on, the kinds with the fewest
// workgroups, as long as they are few together (kFewLeavesPerCu).  Takes their
// counts; grid 0: none (a single kind is left to its own kernel, and so are
// all when profiling, which asks for each kind's time).
struct FewLeaves {
    LeafSet q;
    uint32_t grid;
};
FewLeaves take_few_leaves(const ps5_ctx* c, int rp, const uint32_t* blk_first, uint32_t* nblk, LeavesDone done, uint32_t* nt,
                          uint32_t* nr)
{
    constexpr int NL = kBlkClasses + 2;
    uint32_t* count[NL];
    FewLeaves F;
    F.grid = 0;
    count[0] = nt;
    F.q.r[0] = LeafRange{ c->w.l_tiny[rp], done.tiny, 0u };
    for (int cls = 0; cls < kBlkClasses; ++cls) {
        count[1 + cls] = nblk + cls;
        F.q.r[1 + cls] = LeafRange{ c->w.l_block[rp] + (uint64_t)cls * c->w.cap_block, blk_first[cls], 0u };
    }
    count[NL - 1] = nr;
    F.q.r[NL - 1] = LeafRange{ c->w.l_run[rp], done.run, 0u };
    uint32_t grid = 0, kinds = 0;
    uint64_t room = c->profile ? 0 : (uint64_t)c->cus * kFewLeavesPerCu;
    for (;;) {
        int best = -1;
        uint64_t bw = 0;
        for (int j = 0; j < NL; ++j) {
            // (a chunk counts twice: its own kernel holds twice as many at once)
            const uint64_t w = j == 0 ? div_up(*nt, kLeavesTiny) : j == NL - 1 ? 2ull * *nr : *count[j];
            if (w == 0 || F.q.r[j].count || (best >= 0 && w >= bw)) continue;
            best = j;
            bw = w;
        }
        if (best < 0 || bw > room) break;
        F.q.r[best].count = *count[best];
        room -= bw;
        grid += best == 0 ? (uint32_t)bw : *count[best];
        ++kinds;
    }
    if (kinds < 2) return F;
    F.grid = grid;
    for (int j = 0; j < NL; ++j)
        if (F.q.r[j].count) *count[j] = 0;
    return F;
}
void launch_few_leaves(ps5_ctx* c, const Bufs& B, const FewLeaves& F, const Sink& nsink, bool tail, hipStream_t s)
{
    if (F.grid == 0) return;
    const auto f = c->leaf_keys == 8 ? (tail ? k_leaves<8, true> : k_leaves<8, false>)
                                     : (tail ? k_leaves<0, true> : k_leaves<0, false>);
    hipLaunchKernelGGL(f, dim3(F.grid), dim3(kLeavesWG), 0, s, F.q, B, nsink);
}

// The leaves known to the host (h_cnt) that are not finished yet, on the
// context's stream: before a level overwrites the buffer and the run tables
// of the level before the last, where some of them lie.
void finish_known_leaves(ps5_ctx* c, const Bufs& B, int rp, const Sink& nsink, LeavesDone* done)
{
    const uint32_t nt = c->h_cnt[C_TINY + rp], nr = c->h_cnt[C_RUN + rp];
    launch_leaves(c, B, rp, nsink, *done, false, leaf_tiny_grid(nt - done->tiny), leaf_run_grid(nr - done->run),
                  nt - done->tiny, nr - done->run, c->stream);
    done->tiny = nt;
    done->run = nr;
}

// LCPs between neighbouring leaves of round parity rp (grid workgroups).
void launch_leafbound(ps5_ctx* c, const Bufs& B, int rp, uint32_t grid, uint64_t nleaves)
{
    Launch L(c, K_LEAFBOUND, nleaves * 36);
    LeafLists LL;
    LL.list[0] = c->w.l_tiny[rp];
    LL.cnt[0] = C_TINY + rp;
    LL.cap[0] = c->w.cap_tiny[rp];
    for (int cls = 0; cls < kBlkClasses; ++cls) {
        LL.list[1 + cls] = c->w.l_block[rp] + (uint64_t)cls * c->w.cap_block;
        LL.cnt[1 + cls] = C_BLOCK + 2 * cls + rp;
        LL.cap[1 + cls] = c->w.cap_block;
    }
    LL.list[kBlkClasses + 1] = c->w.l_run[rp];
    LL.cnt[kBlkClasses + 1] = C_RUN + rp;
    LL.cap[kBlkClasses + 1] = c->w.cap_run;
    hipLaunchKernelGGL(k_leafbound, dim3(grid), dim3(kWG), 0, c->stream, LL, B);
}

// The leaves listed so far, in a round planned on the device (at most n of
// them): before a level from the third on (finish_known_leaves).
void dev_finish_leaves(ps5_ctx* c, const Bufs& B, int rp, const Sink& nsink, uint64_t n)
{
    launch_leaves(c, B, rp, nsink, LeavesDone{}, true, (uint32_t)std::min<uint64_t>(kDevTinyWgs, div_up(n, kWaves)),
                  (uint32_t)std::min<uint64_t>(kDevRunWgs, n / kTinyT + 1), n, n, c->stream);
    hipLaunchKernelGGL(k_leaves_done, dim3(1), dim3(64), 0, c->stream, c->d_cnt, rp);
}

// One level planned on the device: k_plan turns the large list `list`
// (counter ci) into the level's plan, and the step's kernels read their work
// from it, in grids bounded by what the host knows (at most bound_large
// segments holding S strings), so nothing comes back to the host.
void dev_level(ps5_ctx* c, const Bufs& B, const Item* list, int ci, uint32_t bound_large, uint64_t S,
               const Sink& sink, uint64_t seed, int src, uint32_t dst, int kmax, int done_rp)
{
    hipStream_t st = c->stream;
    PlanArgs A;
    A.list = list;
    A.ci = ci;
    A.cap_large = c->w.cap_large;
    A.plan = c->w.d_plan;
    A.tiles_off = plan_tiles_off(c->w.cap);
    A.tiles_cap = c->w.tiles_cap;
    A.groups_off = plan_groups_off(c->w.cap);
    A.groups_cap = c->w.groups_cap;
    A.hist_cap = c->w.hist_cap;
    A.gsum_cap = c->w.gsum_cap;
    A.leaf_target = c->leaf_target;
    A.max_treebits = c->max_treebits;
    A.max_oversample = c->max_oversample;
    A.chunk_max = std::min<uint32_t>(c->chunk_max, kPartMax);
    A.chunk_max_root = std::min<uint32_t>(c->chunk_max_root, kPartMax);
    A.min_tiles = c->min_tiles;
    A.kmax = (uint32_t)kmax;
    A.done_rp = done_rp;
    {
        Launch L(c, K_MISC, 0);
        hipLaunchKernelGGL(k_plan, dim3(1), dim3(kBigWG), 0, st, A, c->d_cnt);
    }
    const Plan P = plan_view(c->w.d_plan, c->w.cap);
    const uint32_t gl = std::max<uint32_t>(1, bound_large);
    {
        Launch L(c, K_TREE, 0);
        launch_tree(c, B, P, std::min(gl, kDevTreeWgs), seed, src);
    }
    const uint64_t tiles_bound = S / kChunkMin + gl;
    {
        // two workgroups per CU are resident
        Launch L(c, K_PART, 0);
        launch_part(c, B, P, (uint32_t)std::min<uint64_t>(2 * c->cus, div_up(tiles_bound, kXcds) * kXcds), kmax, src, 0u,
                    false);
    }
    const uint32_t groups_bound = (uint32_t)std::min<uint64_t>(kDevHistWgs, tiles_bound / kHistGroup + gl);
    // no segment of so few strings has more than one group of chunks, and the
    // tables of a single one are k_children's to write if they are short: two
    // kernels fewer (a sort of 5 K strings 113 -> 105 us, 108 with separate
    // count, scan and scatter passes; 40 K 117 -> 108)
    const bool one_group = S <= (uint64_t)kHistGroup * kChunkMin;
    const bool fused = one_group && gl == 1 && (tiles_bound << (kmax + 1)) <= kFusedRuns;
    launch_hist(c, B, P, sink, dst, kmax, one_group ? 0u : groups_bound, std::min(gl, kDevChildWgs), groups_bound, 0, fused);
}

// Bound on the buckets of a level over segments of at most m strings (its
// treebits in *k): 4x their mean below 16 sample keys per splitter (large
// trees; keys repeated between two splitters can add to the spread of the
// sample spacings, 2.9x has been seen at 8), 1 + 8/sqrt(s) from s = 16 on
// (3x at 16, 2.5x at 32: small trees).  Below 4x, the bound shrinks with
// every level of at least 3 splitters.
uint64_t level_bucket_bound(const ps5_ctx* c, uint64_t m, int* k)
{
    *k = large_treebits((uint32_t)std::min<uint64_t>(m, 0xFFFFFFFFull), c->leaf_target, (int)c->max_treebits);
    const uint32_t nspl = (1u << *k) - 1;
    const uint32_t s = std::max<uint32_t>(2, std::min<uint32_t>(c->max_oversample, (kMaxSamples / nspl) & ~1u));
    const uint64_t quarters = s < 16 ? 16 : 4 + (uint64_t)std::ceil(32.0 / std::sqrt((double)s));   // the factor, in quarters
    return (m * quarters + (4ull << *k) - 1) / (4ull << *k);
}

// Levels a round needs when a segment may hold m strings, each level's
// buckets bounded by level_bucket_bound (blocks are sorted by the level that
// lists them, so no level of blocks alone is needed).  A round whose
// segments outgrow the bound leaves them pending, and the host finishes them.
uint32_t dev_levels_for(const ps5_ctx* c, uint64_t m)
{
    uint32_t L = 0;
    int k;
    while (m > kBlkT && L < 8) {
        m = level_bucket_bound(c, m, &k);
        ++L;
    }
    return std::max<uint32_t>(L, 1);
}

// Largest treebits a device-planned level `level` of a round gives its
// segments, when the round's segments hold at most m strings: the bound of
// dev_levels_for, level by level.  A segment above the bound only gets a
// smaller tree than it would choose, and the next level splits it further.
int dev_level_kmax(const ps5_ctx* c, uint64_t m, uint32_t level)
{
    int k;
    for (uint32_t l = 0; l < level; ++l) m = level_bucket_bound(c, m, &k);
    (void)level_bucket_bound(c, m, &k);
    return k;
}

// The host-planned levels of a round from the large list of counter cur_ci
// (in h_cnt / h_large), the round's level `level` and on: each level's large
// list is read back and planned on the host, and the blocks listed before a
// level are sorted in it (blk_done: blocks already sorted per size class;
// done: leaves already finished).  Level l of a round writes buffer l & 1.
int host_levels(ps5_ctx* c, const Bufs& B, uint32_t round, uint32_t level, int cur_ci, uint32_t* blk_done,
                LeavesDone* done, bool* leaves_forked, uint32_t reset_mask, bool* after_blocks, bool* split)
{
    *after_blocks = false;     // set when the stream's last packets are the last level's block kernels
    *split = false;            // set when a segment of the round is split
    hipStream_t st = c->stream;
    const int rp = round & 1, np = rp ^ 1;
    const Sink nsink = make_sink(c, c->w.l_round[np], C_LROUND + np, np);
    int rc;
    for (;; ++level) {
        if (level > 4096) return set_err(PS5_ERR_INTERNAL, "sample-sort levels do not terminate");
        const uint32_t nlarge = c->h_cnt[cur_ci];
        uint32_t nblk[kBlkClasses], nblk_all = 0;
        for (int cls = 0; cls < kBlkClasses; ++cls) {
            nblk[cls] = c->h_cnt[C_BLOCK + 2 * cls + rp] - blk_done[cls];
            nblk_all += nblk[cls];
        }
        Item* nx_large = c->w.l_lvl[level & 1];
        int nx_ci = C_LLVL + (level & 1);
        if (nx_ci == cur_ci) {      // (a round continued from device levels may start on either list)
            nx_large = c->w.l_lvl[(level & 1) ^ 1];
            nx_ci = C_LLVL + ((level & 1) ^ 1);
        }
        // counters to clear before anything of this level is enqueued (the
        // forked leaves included): the caller's (the next round's lists, at
        // level 0) and, when a large step runs, the next level's list (every
        // counter starts at zero in round 0)
        if (nlarge && (round > 0 || level > 0 || cur_ci != C_LROUND + rp)) reset_mask |= 1u << nx_ci;
        if (reset_mask) {
            Launch L(c, K_MISC, 0);
            hipLaunchKernelGGL(k_reset, dim3(1), dim3(64), 0, st, c->d_cnt, reset_mask);
            reset_mask = 0;
        }
        if (nlarge == 0 && nblk_all == 0) break;
        c->st_levels++;
        const Sink sink = make_sink(c, nx_large, nx_ci, rp);
        const uint64_t seed = c->seed ^ ((uint64_t)round << 40) ^ ((uint64_t)level << 32);
        // a level without large segments, in a round whose equal-key
        // leaves all end here (their keys hold a NUL), holds the round's
        // last work: its blocks finish every string themselves (tail mode)
        // and no further round is needed
        const bool tail = c->tail_blocks && nlarge == 0 && c->h_cnt[C_RUNCONT + rp] == 0;
        auto sort_blocks = [&]() -> int {
            uint32_t blk[kBlkClasses], nt = 0, nr = 0;
            std::copy(nblk, nblk + kBlkClasses, blk);
            if (nlarge == 0) {     // the last level: the round's other leaves are all listed
                nt = c->h_cnt[C_TINY + rp] - done->tiny;
                nr = c->h_cnt[C_RUN + rp] - done->run;
            }
            const uint32_t nt0 = nt, nr0 = nr;
            const FewLeaves few = take_few_leaves(c, rp, blk_done, blk, *done, &nt, &nr);
            // beside many blocks, what is few runs on the side stream, and so
            // do many leaves (not when profiling, whose events time the main
            // stream; with less beside it the fork costs more than it hides)
            uint32_t many = 0;
            for (int cls = 0; cls < kBlkClasses; ++cls) many += blk[cls];
            if (nlarge == 0 && !c->profile && ((few.grid && many >= (uint32_t)c->cus * kFewLeavesPerCu) ||
                                               div_up(nt, kWaves) + nr >= kForkLeafGroups)) {
                HIPCHK(hipEventRecord(c->ev_fork, st));
                HIPCHK(hipStreamWaitEvent(c->side, c->ev_fork, 0));
                launch_few_leaves(c, B, few, nsink, tail, c->side);
                LeavesDone d = *done;
                d.tiny += nt0 - nt;
                d.run += nr0 - nr;
                launch_leaves(c, B, rp, nsink, d, false, leaf_tiny_grid(nt), leaf_run_grid(nr), nt, nr, c->side);
                HIPCHK(hipEventRecord(c->ev_join, c->side));
                *leaves_forked = true;
            } else {
                launch_few_leaves(c, B, few, nsink, tail, st);
            }
            done->tiny += nt0 - nt;
            done->run += nr0 - nr;
            int bflags = 0;     // the first class waits for the level; the others may run beside it
            for (int cls = 0; cls < kBlkClasses; ++cls) {
                if (blk[cls]) {
                    launch_block_class(c, B, rp, cls, blk_done[cls], blk[cls], false, blk[cls], nsink, tail, bflags);
                    if (!c->profile) bflags = hipExtAnyOrderLaunch;
                    *after_blocks = nlarge == 0;
                    sum_sizes(c, c->w.l_block[rp] + (uint64_t)cls * c->w.cap_block, blk_done[cls],
                              c->d_cnt + C_BLOCK + 2 * cls + rp, blk_done[cls] + blk[cls], S_BLOCK);
                }
                blk_done[cls] += nblk[cls];
            }
            return PS5_OK;
        };
        // from level 2 on, the step overwrites the buffer and the run tables
        // of the level before the last: what was listed from them goes first
        if ((level >= 2 || nlarge == 0) && (rc = sort_blocks())) return rc;
        if (nlarge) {
            *split = true;
            if (level >= 2) finish_known_leaves(c, B, rp, nsink, done);
            const int src = level > 0 ? kFromRuns : round > 0 ? kFromPerm : B.lut ? kRootPack : kRootPlain;
            if ((rc = large_step(c, B, nlarge, sink, seed, src, level & 1))) return rc;
            if (level < 2 && (rc = sort_blocks())) return rc;
        }
        HIPCHK(hipGetLastError());
        // blocks only append to the next round's lists: after a level
        // without large segments this round has no more levels
        if (nlarge == 0) break;
        uint64_t S = 0, mmax = 0;     // this level's strings and largest segment
        for (uint32_t i = 0; c->chain_levels && i < nlarge; ++i) {
            S += c->w.h_large[i].size;
            mmax = std::max<uint64_t>(mmax, c->w.h_large[i].size);
        }
        if (c->chain_levels && !c->profile && S >= kChainMin) {
            // the next level planned on the device at once, without reading
            // this level's large list back: its segments hold at most this
            // level's S strings and are no larger than its largest segment
            // (below kChainMin strings the bounded grids of a device level
            // cost more than the read-back they save; a profiled sort plans
            // every level on the host, which knows each launch's bytes)
            const int nn = (nx_ci - C_LLVL) ^ 1;     // the level list the device level fills
            Item* nn_large = c->w.l_lvl[nn];
            const int nn_ci = C_LLVL + nn;
            {
                Launch L(c, K_MISC, 0);
                hipLaunchKernelGGL(k_reset, dim3(1), dim3(64), 0, st, c->d_cnt, 1u << nn_ci);
            }
            ++level;
            c->st_levels++;
            const uint64_t seed2 = c->seed ^ ((uint64_t)round << 40) ^ ((uint64_t)level << 32);
            const int kmax = large_treebits((uint32_t)std::min<uint64_t>(mmax, 0xFFFFFFFFull), c->leaf_target,
                                            (int)c->max_treebits);
            if (level >= 2) finish_known_leaves(c, B, rp, nsink, done);
            dev_level(c, B, nx_large, nx_ci, (uint32_t)std::min<uint64_t>(c->w.cap_large, S / (kBlkT + 1) + 1), S,
                      make_sink(c, nn_large, nn_ci, rp), seed2, kFromRuns, level & 1, kmax, -1);
            HIPCHK(hipGetLastError());
            if ((rc = readback(c, nn_large, nn_ci))) return rc;
            cur_ci = nn_ci;
            continue;
        }
        if ((rc = readback(c, nx_large, nx_ci))) return rc;
        cur_ci = nx_ci;
    }
    return PS5_OK;
}

// Leaves and leaf boundaries of a round planned on the host (h_cnt holds
// the round's final counts), then the read-back of the next round's lists.
int host_round_end(ps5_ctx* c, const Bufs& B, uint32_t round, LeavesDone done, bool leaves_forked, bool after_blocks,
                   bool split)
{
    hipStream_t st = c->stream;
    const int rp = round & 1, np = rp ^ 1;
    const Sink nsink = make_sink(c, c->w.l_round[np], C_LROUND + np, np);
    const uint32_t nt = c->h_cnt[C_TINY + rp], nr = c->h_cnt[C_RUN + rp];
    uint32_t nb = 0;
    for (int cls = 0; cls < kBlkClasses; ++cls) nb += c->h_cnt[C_BLOCK + 2 * cls + rp];
    c->st_leaves += nt + nb + nr;
    if (c->trace) {
        fprintf(stderr, "[ps5] round %u: tiny %u, blocks %u/%u/%u/%u, equal chunks %u, levels %llu\n",
                round, nt, c->h_cnt[C_BLOCK + rp], c->h_cnt[C_BLOCK + 2 + rp], c->h_cnt[C_BLOCK + 4 + rp],
                c->h_cnt[C_BLOCK + 6 + rp], nr, (unsigned long long)c->st_levels);
    }
    if (leaves_forked) HIPCHK(hipStreamWaitEvent(st, c->ev_join, 0));
    // right after the last level's block kernels (the first of which waited
    // for everything before it) the leaves may start beside them; the leaf
    // boundaries below wait for all of them
    else launch_leaves(c, B, rp, nsink, done, false, leaf_tiny_grid(nt - done.tiny), leaf_run_grid(nr - done.run),
                       nt - done.tiny, nr - done.run, st, after_blocks && !c->profile ? hipExtAnyOrderLaunch : 0);
    // (a segment that was not split is one leaf, without a boundary to another:
    // 5 us of a small sort's 55)
    if (split && nt + nb + nr && B.lcp) launch_leafbound(c, B, rp, div_up((uint64_t)nt + nb + nr, kWG), nt + nb + nr);
    HIPCHK(hipGetLastError());
    return readback(c, c->w.l_round[np], C_LROUND + np);
}

// One sort call's state, shared by its rounds.
struct SortRun {
    Bufs B;
    uint32_t n;
    uint64_t alen;
    uint32_t root_kmax;       // largest treebits of a large root
    uint64_t root_max;        // largest root: no segment of any round is larger
    uint64_t root_sum;        // strings in large roots
};

// The depth arrays a round reads (none in round 0: every root starts at
// depth 0) and writes.
void set_depths(ps5_ctx* c, Bufs& B, uint32_t round)
{
    B.sdepth_in = round ? c->w.sdepth[round & 1] : nullptr;
    B.sdepth_out = c->w.sdepth[(round & 1) ^ 1];
}

// Round `round` of a sort, planned on the host or (dev) on the device; sets
// *done when no work is left for another round.
int sort_round(ps5_ctx* c, SortRun& R, uint32_t round, bool dev, bool* done)
{
    int rc;
    hipStream_t st = c->stream;
    Bufs& B = R.B;
    const uint32_t n = R.n;
    const uint64_t alen = R.alen;
    const uint32_t root_kmax = R.root_kmax;
    const uint64_t root_max = R.root_max, root_sum = R.root_sum;
    uint32_t* lcp = B.lcp;
    *done = false;
    const int rp = round & 1, np = rp ^ 1;
    set_depths(c, B, round);
    c->st_rounds++;
    uint32_t round_mask = 0;     // the lists of round r+1 are empty again (consumed in round r-1; set up empty in round 0)
    if (round > 0) {
        round_mask = (1u << (C_LROUND + np)) | (1u << (C_TINY + np)) | (1u << (C_RUN + np));
        for (int cls = 0; cls < kBlkClasses; ++cls)
            round_mask |= (1u << (C_BLOCK + 2 * cls + np)) | (1u << (C_BDONE + cls));
        round_mask |= (1u << (C_RUNCONT + np)) | (1u << C_TDONE) | (1u << C_RDONE);
    }
    if (round_mask && dev) {     // (host-planned levels clear them with their first level's counters)
        Launch L(c, K_MISC, 0);
        hipLaunchKernelGGL(k_reset, dim3(1), dim3(64), 0, st, c->d_cnt, round_mask);
    }
    const Sink nsink = make_sink(c, c->w.l_round[np], C_LROUND + np, np);
    uint32_t blk_done[kBlkClasses] = {};
    LeavesDone done_leaves;
    bool leaves_forked = false, after_blocks = false, split = false;
    if (!dev) {
        if ((rc = host_levels(c, B, round, 0, C_LROUND + rp, blk_done, &done_leaves, &leaves_forked, round_mask,
                              &after_blocks, &split)))
            return rc;
        if ((rc = host_round_end(c, B, round, done_leaves, leaves_forked, after_blocks, split))) return rc;
    } else {
        // every level of the round without a host synchronisation.  The
        // host knows the round's lists (read back with the previous
        // round, or set up): S strings in nl0 large segments bound the
        // grids; a round without large segments is planned on the host
        const uint32_t nl0 = c->h_cnt[C_LROUND + rp];
        uint64_t S = 0, mmax = 0;
        if (round == 0) {
            S = root_sum;
            mmax = root_max;
        } else if (nl0 <= kPeek) {
            for (uint32_t i = 0; i < nl0; ++i) {
                S += c->w.h_large[i].size;
                mmax = std::max<uint64_t>(mmax, c->w.h_large[i].size);
            }
        } else {
            S = n;
            mmax = root_max;
        }
        const uint32_t L = nl0 ? dev_levels_for(c, mmax) : 0;
        if (L == 0) {
            if ((rc = host_levels(c, B, round, 0, C_LROUND + rp, blk_done, &done_leaves, &leaves_forked, 0u,
                                  &after_blocks, &split)))
                return rc;
            if ((rc = host_round_end(c, B, round, done_leaves, leaves_forked, after_blocks, split))) return rc;
        } else {
            int in_ci = C_LROUND + rp;
            const Item* in_list = c->w.l_round[rp];
            const uint32_t deeper_large = (uint32_t)std::min<uint64_t>(c->w.cap_large, S / (kBlkT + 1) + 1);
            for (uint32_t level = 0; level < L; ++level) {
                c->st_levels++;
                const int out_ci = C_LLVL + (level & 1);
                if (!(round == 0 && level == 0)) {
                    Launch Lr(c, K_MISC, 0);
                    hipLaunchKernelGGL(k_reset, dim3(1), dim3(64), 0, st, c->d_cnt, 1u << out_ci);
                }
                const Sink sink = make_sink(c, c->w.l_lvl[level & 1], out_ci, rp);
                const uint64_t seed = c->seed ^ ((uint64_t)round << 40) ^ ((uint64_t)level << 32);
                const bool rootlvl = round == 0 && level == 0;
                const int src = level > 0 ? kFromRuns : round > 0 ? kFromPerm : B.lut ? kRootPack : kRootPlain;
                if (level >= 2) dev_finish_leaves(c, B, rp, nsink, S);
                dev_level(c, B, in_list, in_ci, level == 0 ? nl0 : deeper_large, S, sink, seed, src, level & 1,
                          rootlvl ? (int)root_kmax : dev_level_kmax(c, mmax, level), level > 0 ? rp : -1);
                int bflags = 0;     // the first class waits for the level; the others run beside it
                for (int cls = 0; cls < kBlkClasses; ++cls) {
                    // four workgroups for every wave slot of the GPU (32
                    // per CU): blocks differ in size up to 2x, and the
                    // dispatcher's later workgroups even out the load
                    const uint32_t minm = cls == 0 ? kTinyT + 1 : (128u << cls) + 1;
                    const uint64_t full = block_grid_full(c, cls);
                    const uint64_t known = level == 0 ? c->h_cnt[C_BLOCK + 2 * cls + rp] : 0;
                    const uint32_t g = (uint32_t)std::min<uint64_t>(full, known + S / minm + 1);
                    launch_block_class(c, B, rp, cls, 0, 0, true, g, nsink, false, bflags);
                    if (!c->profile) bflags = hipExtAnyOrderLaunch;
                }
                HIPCHK(hipGetLastError());
                in_ci = out_ci;
                in_list = c->w.l_lvl[level & 1];
            }
            // leaves with persistent grids: they skip their work when
            // large segments remain (counter in_ci), which the host then
            // finishes
            const uint64_t nt0 = c->h_cnt[C_TINY + rp], nr0 = c->h_cnt[C_RUN + rp];
            const uint32_t gt = (uint32_t)std::min<uint64_t>(kDevTinyWgs, div_up(nt0 + S, kWaves));
            const uint32_t gr = (uint32_t)std::min<uint64_t>(kDevRunWgs, nr0 + S / kTinyT + 1);
            B.pending = c->d_cnt + in_ci;
            launch_leaves(c, B, rp, nsink, done_leaves, true, gt, gr, nt0 + S, nr0 + S, st);
            if (lcp) {
                uint64_t known = nt0 + nr0;
                for (int cls = 0; cls < kBlkClasses; ++cls) known += c->h_cnt[C_BLOCK + 2 * cls + rp];
                launch_leafbound(c, B, rp,
                                 (uint32_t)std::min<uint64_t>(kDevBoundWgs, div_up(known + S, kWG)), known + S);
            }
            B.pending = nullptr;
            HIPCHK(hipGetLastError());
            if ((rc = readback(c, c->w.l_round[np], C_LROUND + np))) return rc;
            if (c->h_cnt[in_ci] != 0) {
                // more levels than planned: read the remaining large list
                // back and finish the round on the host
                for (int cls = 0; cls < kBlkClasses; ++cls) blk_done[cls] = c->h_cnt[C_BLOCK + 2 * cls + rp];
                if ((rc = readback(c, in_list, in_ci))) return rc;
                done_leaves = LeavesDone{ c->h_cnt[C_TDONE], c->h_cnt[C_RDONE] };
                if ((rc = host_levels(c, B, round, L, in_ci, blk_done, &done_leaves, &leaves_forked, 0u, &after_blocks, &split)))
                    return rc;
                if ((rc = host_round_end(c, B, round, done_leaves, leaves_forked, after_blocks, split))) return rc;
            } else {
                uint32_t nb = 0;
                for (int cls = 0; cls < kBlkClasses; ++cls) nb += c->h_cnt[C_BLOCK + 2 * cls + rp];
                c->st_leaves += c->h_cnt[C_TINY + rp] + nb + c->h_cnt[C_RUN + rp];
            }
        }
    }
    uint64_t pending = (uint64_t)c->h_cnt[C_LROUND + np] + c->h_cnt[C_TINY + np] + c->h_cnt[C_RUN + np];
    for (int cls = 0; cls < kBlkClasses; ++cls) pending += c->h_cnt[C_BLOCK + 2 * cls + np];
    if (pending == 0) { *done = true; return PS5_OK; }
    if ((uint64_t)round * 8 > alen + 8) return set_err(PS5_ERR_INTERNAL, "depth exceeds the arena: no progress");
    return PS5_OK;
}

// Round `round` for a captured graph: planned on the device with grids
// bounded by what the host knows before the sort (n strings, roots of at
// most root_max), no host synchronisation; L device levels, and a round that
// needs more is flagged (ERR_LEVELS) by its leaf kernels.
void graph_round(ps5_ctx* c, SortRun& R, uint32_t round, uint32_t L, uint32_t nl_root)
{
    hipStream_t st = c->stream;
    Bufs B = R.B;
    const uint64_t n = R.n;
    const int rp = round & 1, np = rp ^ 1;
    set_depths(c, B, round);
    if (round > 0) {
        uint32_t mask = (1u << (C_LROUND + np)) | (1u << (C_TINY + np)) | (1u << (C_RUN + np));
        for (int cls = 0; cls < kBlkClasses; ++cls) mask |= (1u << (C_BLOCK + 2 * cls + np)) | (1u << (C_BDONE + cls));
        mask |= (1u << (C_RUNCONT + np)) | (1u << C_TDONE) | (1u << C_RDONE);
        hipLaunchKernelGGL(k_reset, dim3(1), dim3(64), 0, st, c->d_cnt, mask);
    }
    const Sink nsink = make_sink(c, c->w.l_round[np], C_LROUND + np, np);
    const uint64_t S = round == 0 ? R.root_sum : n;
    const uint32_t any_large = (uint32_t)std::min<uint64_t>(c->w.cap_large, n / (kBlkT + 1) + 1);
    int in_ci = C_LROUND + rp;
    const Item* in_list = c->w.l_round[rp];
    for (uint32_t level = 0; level < L; ++level) {
        const int out_ci = C_LLVL + (level & 1);
        hipLaunchKernelGGL(k_reset, dim3(1), dim3(64), 0, st, c->d_cnt, 1u << out_ci);
        const Sink sink = make_sink(c, c->w.l_lvl[level & 1], out_ci, rp);
        const uint64_t seed = c->seed ^ ((uint64_t)round << 40) ^ ((uint64_t)level << 32);
        const bool rootlvl = round == 0 && level == 0;
        const int src = level > 0 ? kFromRuns : round > 0 ? kFromPerm : kRootPlain;
        if (level >= 2) dev_finish_leaves(c, B, rp, nsink, n);
        dev_level(c, B, in_list, in_ci, rootlvl ? nl_root : any_large, S, sink, seed, src, level & 1,
                  rootlvl ? (int)R.root_kmax : dev_level_kmax(c, R.root_max, level), level > 0 ? rp : -1);
        for (int cls = 0; cls < kBlkClasses; ++cls) {
            launch_block_class(c, B, rp, cls, 0, 0, true, block_grid_full(c, cls), nsink);
        }
        in_ci = out_ci;
        in_list = c->w.l_lvl[level & 1];
    }
    B.pending = c->d_cnt + in_ci;
    B.pending_err = 1;
    launch_leaves(c, B, rp, nsink, LeavesDone{}, true, (uint32_t)std::min<uint64_t>(kDevTinyWgs, div_up(n, kWaves)),
                  (uint32_t)std::min<uint64_t>(kDevRunWgs, c->w.cap_run), n, n, st);
    if (B.lcp) launch_leafbound(c, B, rp, (uint32_t)std::min<uint64_t>(kDevBoundWgs, div_up(n, kWG)), n);
}

// How a sort's roots choose their keys: plain, packed as their samples say, or
// packed with the alphabets that a sort with kPackSampled found.
enum Packing { kPackNone, kPackSampled, kPackWidened };

int run_sort_keys(ps5_ctx* c, const uint8_t* arena, uint64_t alen, const uint32_t* offs, const uint64_t* offs64,
                  uint32_t n, uint32_t* perm, uint32_t* lcp, const uint64_t* set_first, uint32_t nsets, Packing pack)
{
    int rc = ensure_capacity(c, n);
    if (!rc) rc = ensure_tables(c);
    if (rc) return rc;
    for (int i = 0; i < K_NUM; ++i) { c->k_ms[i] = 0; c->k_launch[i] = 0; c->k_bytes[i] = 0; }
    c->st_rounds = c->st_levels = c->st_segments = c->st_leaves = c->st_syncs = 0;
    hipStream_t st = c->stream;
    if (c->profile) HIPCHK(hipMemsetAsync(c->d_sums, 0, S_NUM * sizeof(unsigned long long), st));

    Bufs B;
    B.n = n;
    B.cnt = c->d_cnt;
    B.arena = arena;
    B.alen = alen;
    B.offs = offs;
    B.offs64 = offs64;
    B.rec = c->w.rec;
    B.vpos = c->w.vpos;
    B.src = c->w.src;
    B.cap = c->w.cap;
    B.cap_h = c->w.hist_cap;
    B.perm = perm;
    B.lcp = lcp;
    B.bkey = c->w.bkey;
    B.hist = c->w.hist;
    B.gsum = c->w.gsum;
    B.pending = nullptr;
    B.pending_err = 0;
    B.leaf_keys = c->leaf_keys;
    set_depths(c, B, 0);
    B.lut = nullptr;
    B.widen = pack == kPackWidened;

    // the roots (one, or a batch's sets) and their sizes
    uint32_t root_kmax = 1;                     // largest treebits of a large root
    uint64_t root_max = n;                      // largest root (no segment of any round is larger)
    uint64_t root_sum = n;                      // strings in large roots
    if (!set_first) {
        root_kmax = (uint32_t)large_treebits(n, c->leaf_target, (int)c->max_treebits);
    } else {
        root_max = 0;
        root_sum = 0;
        for (uint32_t s = 0; s < nsets; ++s) {
            const uint64_t m = set_first[s + 1] - set_first[s];
            root_max = std::max(root_max, m);
            if (m <= kBlkT) continue;
            root_sum += m;
            root_kmax = std::max<uint32_t>(root_kmax, (uint32_t)large_treebits((uint32_t)m, c->leaf_target,
                                                                               (int)c->max_treebits));
        }
    }
    const bool single_root = !set_first && n > kBlkT;
    bool dev = c->planning == 1 ||
               (c->planning == 2 && !c->profile && !set_first && n < kAutoDevMax);   // (profiled sorts: host, whose
                                                                                     // launches know their bytes)
    // a single root planned on the host: the root level's plan fetch, the
    // sort's first kernel, also sets the counters and the root item up
    c->pending_root = single_root && !dev && !(c->graph_rounds && !c->profile) ? n : 0u;
    if (c->pending_root) {
        for (int i = 0; i < C_NCNT; ++i) c->h_cnt[i] = 0;
        c->h_cnt[C_LROUND] = 1;
        c->w.h_large[0] = Item{ 0u, n, 0u, F_IDENT, 0u, 0u };
    } else if ((rc = setup_roots(c, n, set_first, nsets))) {
        return rc;
    }
    if (pack != kPackNone && root_max >= kPackMin) B.lut = c->w.lut;     // large roots may pack their keys
    SortRun R{ B, n, alen, root_kmax, root_max, root_sum };
    uint32_t start = 0;
    if (c->graph_rounds && !c->profile) {
        // the first graph_rounds rounds as one captured graph, replayed while
        // the sort's inputs, buffers and shape settings are the same
        uint32_t nl_root = 0;
        for (uint32_t s = 0; set_first && s < nsets; ++s) nl_root += set_first[s + 1] - set_first[s] > kBlkT ? 1 : 0;
        if (!set_first) nl_root = n > kBlkT ? 1 : 0;
        std::vector<uint64_t> key = { (uint64_t)(uintptr_t)arena, alen, (uint64_t)(uintptr_t)offs,
                                      (uint64_t)(uintptr_t)offs64, n, (uint64_t)(uintptr_t)perm,
                                      (uint64_t)(uintptr_t)lcp, nsets, (uint64_t)(uintptr_t)c->w.rec, c->w.cap,
                                      (uint64_t)(uintptr_t)c->w.trees, c->w.gsum_cap, c->leaf_target,
                                      c->max_treebits, c->max_oversample, c->graph_rounds, c->seed,
                                      c->w_gen, c->w.fixed ? 1u : 0u, c->graph_levels, c->chunk_max,
                                      c->chunk_max_root, c->min_tiles, c->leaf_keys };
        for (uint32_t s = 0; set_first && s <= nsets; ++s) key.push_back(set_first[s]);
        if (!c->graph_exec || key != c->graph_key) {
            if (c->graph_exec) (void)hipGraphExecDestroy(c->graph_exec);
            if (c->graph) (void)hipGraphDestroy(c->graph);
            c->graph_exec = nullptr;
            c->graph = nullptr;
            c->graph_key.clear();
            uint32_t L = dev_levels_for(c, root_max);
            if (c->graph_levels) L = std::min(L, c->graph_levels);
            HIPCHK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
            for (uint32_t r = 0; r < c->graph_rounds; ++r) graph_round(c, R, r, L, nl_root);
            hipLaunchKernelGGL(k_stage, dim3(1), dim3(kWG), 0, st, c->d_cnt, c->w.l_round[c->graph_rounds & 1],
                               C_LROUND + (int)(c->graph_rounds & 1), c->h_stage_dev, 0u);
            hipGraph_t g = nullptr;
            const hipError_t ec = hipStreamEndCapture(st, &g);
            if (ec != hipSuccess) return set_err(PS5_ERR_HIP, "graph capture failed: %s", hipGetErrorString(ec));
            c->graph = g;
            HIPCHK(hipGraphInstantiate(&c->graph_exec, c->graph, nullptr, nullptr, 0));
            c->graph_key = key;
        }
        // the graph's k_stage publishes 0 last; the host marks the word first
        __atomic_store_n(reinterpret_cast<uint32_t*>(c->h_stage + kStageSeq), kGraphSeqPending, __ATOMIC_RELEASE);
        HIPCHK(hipGraphLaunch(c->graph_exec, st));
        if ((rc = wait_stage(c, 0u))) return rc;
        c->st_syncs++;
        c->st_rounds += c->graph_rounds;
        memcpy(c->h_cnt, c->h_stage, C_NCNT * sizeof(uint32_t));
        if (c->h_cnt[C_ERR] & ERR_LEVELS) {
            // a round needed more levels than the graph holds: sort again,
            // every level planned on the host
            if ((rc = setup_roots(c, n, set_first, nsets))) return rc;
            dev = false;
        } else {
            if (c->h_cnt[C_ERR] & ERR_CAP) return set_err(PS5_ERR_CAPACITY, "work list capacity exceeded");
            if (c->h_cnt[C_ERR] & ERR_LCP) return set_err(PS5_ERR_INTERNAL, "equal keys across a leaf boundary");
            if (c->h_cnt[C_ERR] & ERR_BOUNDS) return set_err(PS5_ERR_INTERNAL, "device bounds check failed");
            const int rp = c->graph_rounds & 1;
            uint64_t pending = (uint64_t)c->h_cnt[C_LROUND + rp] + c->h_cnt[C_TINY + rp] + c->h_cnt[C_RUN + rp];
            for (int cls = 0; cls < kBlkClasses; ++cls) pending += c->h_cnt[C_BLOCK + 2 * cls + rp];
            if (pending == 0) return PS5_OK;
            // more rounds than captured: continue round by round
            if ((rc = readback(c, c->w.l_round[rp], C_LROUND + rp))) return rc;
            start = c->graph_rounds;
        }
    }
    for (uint32_t round = start;; ++round) {
        bool done = false;
        if ((rc = sort_round(c, R, round, dev, &done))) return rc;
        if (done) break;
    }
    if (c->profile) {
        HIPCHK(hipMemcpyAsync(c->h_sums, c->d_sums, S_NUM * sizeof(unsigned long long), hipMemcpyDeviceToHost, st));
        HIPCHK(hipStreamSynchronize(st));
        // algorithmic bytes per string of the list-driven kernels
        c->k_bytes[K_BLOCK] += c->h_sums[S_BLOCK] * 20;     // key 8 + idx 4 R, perm 4 + lcp 4 W
        c->k_bytes[K_LEAF_TINY] += c->h_sums[S_TINY] * 20;
        c->k_bytes[K_LEAF_RUN] += c->h_sums[S_RUN] * 12;    // idx 4 R, perm 4 + lcp 4 W
        collect_events(c);
    }
    return PS5_OK;
}

// (a captured graph holds plain keys only: its replay cannot start over)
int run_sort(ps5_ctx* c, const uint8_t* arena, uint64_t alen, const uint32_t* offs, const uint64_t* offs64,
             uint32_t n, uint32_t* perm, uint32_t* lcp, const uint64_t* set_first, uint32_t nsets)
{
    const bool graph = c->graph_rounds && !c->profile;
    int rc = run_sort_keys(c, arena, alen, offs, offs64, n, perm, lcp, set_first, nsets, graph ? kPackNone : kPackSampled);
    if (rc != kStartOver) return rc;
    HIPCHK(hipStreamSynchronize(c->side));
    HIPCHK(hipStreamSynchronize(c->stream));
    if (c->profile) collect_events(c);
    // (every root's level saw all of its strings, so this finds no other character)
    if (c->trace) fprintf(stderr, "[ps5] a packed root met a character outside its alphabet: starting over\n");
    rc = run_sort_keys(c, arena, alen, offs, offs64, n, perm, lcp, set_first, nsets, kPackWidened);
    return rc == kStartOver ? set_err(PS5_ERR_INTERNAL, "a packed key outside its whole root's alphabet") : rc;
}

}  // namespace

// ===========================================================================
// C ABI
// ===========================================================================

extern "C" {

const char* ps5_last_error(void) { return g_err.c_str(); }

int ps5_ctx_create(ps5_ctx** out, int device)
{
    if (!out) return set_err(PS5_ERR_ARG, "out is NULL");
    *out = nullptr;
    HIPCHK(hipSetDevice(device));
    for (int kmax = 7; kmax <= kMaxTreebits; ++kmax)
        for (int src : { kFromRuns, kRootPlain, kRootPack, kFromPerm }) {
            uint32_t lds = 0;
            const PartKernel f = part_kernel(kmax, src, &lds);
            HIPCHK(hipFuncSetAttribute((const void*)f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        }
    ps5_ctx* c = new ps5_ctx;
    c->device = device;
    c->trace = getenv("PS5_TRACE") != nullptr;
    if (const char* dl = getenv("PS5_DEV_LEVELS")) c->planning = std::min(std::max(atoi(dl), 0), 2);
    if (const char* gr = getenv("PS5_GRAPH_ROUNDS")) c->graph_rounds = std::min<uint32_t>(atoi(gr), kMaxGraphRounds);
    if (const char* gl = getenv("PS5_GRAPH_LEVELS")) c->graph_levels = (uint32_t)std::max(atoi(gl), 0);
    if (const char* tb = getenv("PS5_TAIL_BLOCKS")) c->tail_blocks = atoi(tb) != 0;
    if (const char* cl = getenv("PS5_CHAIN_LEVELS")) c->chain_levels = atoi(cl) != 0;
    int ncu = 0;
    hipError_t e = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, device);
    c->cus = std::max<uint32_t>(kXcds, (uint32_t)std::max(ncu, 0) / kXcds * kXcds);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipStreamCreateWithFlags(&c->side, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&c->ev_fork, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&c->ev_join, hipEventDisableTiming);
    if (e == hipSuccess) e = hipMalloc(&c->d_cnt, C_NCNT * sizeof(uint32_t));
    if (e == hipSuccess) e = hipHostMalloc(reinterpret_cast<void**>(&c->h_cnt), C_NCNT * sizeof(uint32_t));
    if (e == hipSuccess)
        e = hipHostMalloc(reinterpret_cast<void**>(&c->h_stage), kStageHead + kPeek * sizeof(Item),
                          hipHostMallocMapped | hipHostMallocCoherent);
    // recycled pinned memory may hold an older context's sequence number: the
    // wait for this context's first staged copies must not see it
    if (e == hipSuccess) memset(c->h_stage, 0, kStageHead);
    if (e == hipSuccess) e = hipHostGetDevicePointer(reinterpret_cast<void**>(&c->h_stage_dev), c->h_stage, 0);
    if (e == hipSuccess) e = hipMalloc(&c->d_sums, S_NUM * sizeof(unsigned long long));
    if (e == hipSuccess) e = hipHostMalloc(reinterpret_cast<void**>(&c->h_sums), S_NUM * sizeof(unsigned long long));
    // the allocation-free entry point's pinned plan buffers, sized for the
    // scratch's largest sort
    if (e == hipSuccess)
        e = hipHostMalloc(reinterpret_cast<void**>(&c->na_h_large), cap_large_of(kNoAllocMaxStrings) * sizeof(Item));
    if (e == hipSuccess)
        e = hipHostMalloc(reinterpret_cast<void**>(&c->na_h_plan), plan_bytes_of(kNoAllocMaxStrings),
                          hipHostMallocMapped | hipHostMallocCoherent);
    if (e == hipSuccess) e = hipHostGetDevicePointer(reinterpret_cast<void**>(&c->na_h_plan_dev), c->na_h_plan, 0);
    if (e != hipSuccess) {
        ps5_ctx_destroy(c);
        return set_err(PS5_ERR_HIP, "context setup failed: %s", hipGetErrorString(e));
    }
    if (int rc = scratch_address(device, &c->na_scratch)) {
        ps5_ctx_destroy(c);
        return rc;
    }
    *out = c;
    return PS5_OK;
}

void ps5_ctx_destroy(ps5_ctx* c)
{
    if (!c) return;
    (void)hipSetDevice(c->device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    free_buffers(c);
    if (c->d_cnt) (void)hipFree(c->d_cnt);
    if (c->d_sums) (void)hipFree(c->d_sums);
    if (c->d_sets) (void)hipFree(c->d_sets);
    if (c->d_merge) (void)hipFree(c->d_merge);
    if (c->h_cnt) (void)hipHostFree(c->h_cnt);
    if (c->h_stage) (void)hipHostFree(c->h_stage);
    if (c->h_roots) (void)hipHostFree(c->h_roots);
    if (c->h_sums) (void)hipHostFree(c->h_sums);
    if (c->na_h_large) (void)hipHostFree(c->na_h_large);
    if (c->na_h_plan) (void)hipHostFree(c->na_h_plan);
    for (auto e : c->ev_pool) (void)hipEventDestroy(e);
    for (auto& u : c->ev_used) { (void)hipEventDestroy(u.second.first); (void)hipEventDestroy(u.second.second); }
    if (c->side) (void)hipStreamSynchronize(c->side);
    if (c->graph_exec) (void)hipGraphExecDestroy(c->graph_exec);
    if (c->graph) (void)hipGraphDestroy(c->graph);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    if (c->side) (void)hipStreamDestroy(c->side);
    if (c->ev_fork) (void)hipEventDestroy(c->ev_fork);
    if (c->ev_join) (void)hipEventDestroy(c->ev_join);
    delete c;
}

int ps5_ctx_reserve(ps5_ctx* c, uint64_t n)
{
    if (!c) return set_err(PS5_ERR_ARG, "ctx is NULL");
    if (n >= 0xFFFFFF00ull) return set_err(PS5_ERR_ARG, "n too large (limit 2^32-256 strings)");
    HIPCHK(hipSetDevice(c->device));
    const int rc = ensure_capacity(c, n);
    return rc ? rc : ensure_tables(c);
}

void* ps5_ctx_stream(ps5_ctx* c) { return c ? (void*)c->stream : nullptr; }

int ps5_sort_device(ps5_ctx* c, const uint8_t* d_arena, uint64_t arena_bytes, const uint32_t* d_offs,
                    uint64_t n, uint32_t* d_perm, uint32_t* d_lcp)
{
    if (!c) return set_err(PS5_ERR_ARG, "ctx is NULL");
    if (n == 0) return PS5_OK;
    if (!d_arena || !d_offs || !d_perm) return set_err(PS5_ERR_ARG, "NULL device pointer");
    if (n >= 0xFFFFFF00ull) return set_err(PS5_ERR_ARG, "n too large (limit 2^32-256 strings)");
    if (arena_bytes == 0 || arena_bytes > 0xFFFFFFFFull)
        return set_err(PS5_ERR_ARG, "arena_bytes must be in [1, 2^32)");
    if (((uintptr_t)d_arena & 7u) != 0) return set_err(PS5_ERR_ARG, "arena must be 8-byte aligned");
    HIPCHK(hipSetDevice(c->device));
    int rc = run_sort(c, d_arena, arena_bytes, d_offs, nullptr, (uint32_t)n, d_perm, d_lcp, nullptr, 0);
    if (rc) {
        (void)hipStreamSynchronize(c->stream);
        (void)hipStreamSynchronize(c->side);
        if (c->profile) collect_events(c);
    }
    return rc;
}

int ps5_sort_device_noalloc(ps5_ctx* c, const uint8_t* d_arena, uint64_t arena_bytes, const uint32_t* d_offs,
                            uint64_t n, uint32_t* d_perm, uint32_t* d_lcp)
{
    if (!c) return set_err(PS5_ERR_ARG, "ctx is NULL");
    if (n == 0) return PS5_OK;
    if (!d_arena || !d_offs || !d_perm) return set_err(PS5_ERR_ARG, "NULL device pointer");
    if (n > kNoAllocMaxStrings)
        return set_err(PS5_ERR_ARG, "n = %llu exceeds the allocation-free limit of %llu strings",
                       (unsigned long long)n, (unsigned long long)kNoAllocMaxStrings);
    if (arena_bytes == 0 || arena_bytes > 0xFFFFFFFFull)
        return set_err(PS5_ERR_ARG, "arena_bytes must be in [1, 2^32)");
    if (((uintptr_t)d_arena & 7u) != 0) return set_err(PS5_ERR_ARG, "arena must be 8-byte aligned");
    if (!c->na_scratch) return set_err(PS5_ERR_HIP, "the device scratch of this context is not resolved");
    HIPCHK(hipSetDevice(c->device));
    std::lock_guard<std::mutex> g(scratch_mutex(c->device));
    // the context's own buffers step aside for views into the scratch;
    // profiling (which creates events) and captured graphs (whose
    // instantiation allocates) are off for the call
    WorkBuffers own = scratch_buffers(c->na_scratch, c->na_h_large, c->na_h_plan, c->na_h_plan_dev);
    std::swap(c->w, own);
    const bool prof = c->profile;
    const uint32_t graph_rounds = c->graph_rounds;
    c->profile = false;
    c->graph_rounds = 0;
    int rc = run_sort(c, d_arena, arena_bytes, d_offs, nullptr, (uint32_t)n, d_perm, d_lcp, nullptr, 0);
    if (rc) {
        (void)hipStreamSynchronize(c->stream);
        (void)hipStreamSynchronize(c->side);
    }
    c->profile = prof;
    c->graph_rounds = graph_rounds;
    std::swap(c->w, own);
    return rc;
}

uint64_t ps5_noalloc_max_strings(void) { return kNoAllocMaxStrings; }

int ps5_merge_device(ps5_ctx* c, const uint8_t* d_arena, uint64_t arena_bytes, const uint32_t* d_offs,
                     const uint64_t* run_first, uint32_t nruns, const uint32_t* d_idx, const uint32_t* d_lcp,
                     uint32_t* d_idx_out, uint32_t* d_lcp_out)
{
    if (!c) return set_err(PS5_ERR_ARG, "ctx is NULL");
    if (nruns == 0 || !run_first) return set_err(PS5_ERR_ARG, "no runs");
    const uint64_t n = run_first[nruns];
    if (run_first[0] != 0) return set_err(PS5_ERR_ARG, "run_first[0] must be 0");
    for (uint32_t r = 0; r < nruns; ++r)
        if (run_first[r + 1] < run_first[r]) return set_err(PS5_ERR_ARG, "run boundaries must be non-decreasing");
    if (n == 0) return PS5_OK;
    if (!d_arena || !d_offs || !d_idx || !d_lcp || !d_idx_out || !d_lcp_out)
        return set_err(PS5_ERR_ARG, "NULL device pointer");
    if (n >= 0xFFFFFF00ull) return set_err(PS5_ERR_ARG, "n too large (limit 2^32-256 strings)");
    if (arena_bytes == 0 || arena_bytes > 0xFFFFFFFFull) return set_err(PS5_ERR_ARG, "arena_bytes must be in [1, 2^32)");
    if (((uintptr_t)d_arena & 7u) != 0) return set_err(PS5_ERR_ARG, "arena must be 8-byte aligned");
    HIPCHK(hipSetDevice(c->device));
    hipStream_t st = c->stream;
    if (nruns == 1) {
        HIPCHK(hipMemcpyAsync(d_idx_out, d_idx, n * 4, hipMemcpyDeviceToDevice, st));
        HIPCHK(hipMemcpyAsync(d_lcp_out, d_lcp, n * 4, hipMemcpyDeviceToDevice, st));
        HIPCHK(hipStreamSynchronize(st));
        return PS5_OK;
    }
    int rc = ensure_capacity(c, n);
    if (rc) return rc;
    HIPCHK(hipMemsetAsync(c->d_cnt, 0, C_NCNT * sizeof(uint32_t), st));
    Bufs B{};
    B.n = (uint32_t)n;
    B.cnt = c->d_cnt;
    B.arena = d_arena;
    B.alen = arena_bytes;
    B.offs = d_offs;
    // ping-pong buffers in the records' memory: two of first 8 characters, two
    // of indices; LCPs in the two halves of bkey
    key64* keys = reinterpret_cast<key64*>(c->w.rec);
    uint32_t* idxs = reinterpret_cast<uint32_t*>(keys + 2 * c->w.cap);
    uint32_t* ti[2] = { idxs, idxs + c->w.cap };
    key64* tk[2] = { keys, keys + c->w.cap };
    uint32_t* tl[2] = { reinterpret_cast<uint32_t*>(c->w.bkey), reinterpret_cast<uint32_t*>(c->w.bkey) + c->w.cap };
    std::vector<uint64_t> bounds(run_first, run_first + nruns + 1);
    const uint32_t* si = d_idx;
    const uint32_t* sl = d_lcp;
    // the first round reads every string's first 8 characters from ik, keys
    // extracted in input order by one streaming pass (the previous round's
    // output carries them afterwards); tk[1] is free until the second merge
    // round writes it
    key64* ik = tk[1];
    hipLaunchKernelGGL(k_init, dim3(div_up(n, kWG)), dim3(kWG), 0, st, B, ik, (uint32_t)n);
    HIPCHK(hipGetLastError());
    // every round's plan, uploaded at once: first[np + 1], mid[np], tstart[np + 1]
    struct Round { uint64_t at; uint32_t np; uint64_t tiles; };
    std::vector<Round> rounds;
    std::vector<uint64_t> plan;
    uint64_t most = 0;     // tiles of a round
    while (bounds.size() > 2) {
        const uint32_t nr = (uint32_t)bounds.size() - 1, np = (nr + 1) / 2;
        const uint64_t at = plan.size();
        plan.resize(at + 3 * ((uint64_t)np + 1), 0);
        uint64_t* f = plan.data() + at;
        uint64_t* mdl = f + (np + 1);
        uint64_t* ts = mdl + (np + 1);
        std::vector<uint64_t> nb(np + 1);
        for (uint32_t p = 0; p < np; ++p) {
            f[p] = bounds[2 * p];
            mdl[p] = bounds[2 * p + 1];
            const uint64_t e = 2 * p + 2 <= nr ? bounds[2 * p + 2] : bounds[2 * p + 1];
            ts[p + 1] = ts[p] + (e - f[p] + kMergeT - 1) / kMergeT;
            nb[p] = f[p];
        }
        f[np] = nb[np] = bounds[nr];
        rounds.push_back(Round{ at, np, ts[np] });
        most = std::max(most, ts[np]);
        bounds.swap(nb);
    }
    const uint64_t words = plan.size() + (most + 1) / 2;    // the plans, then co[tiles] as uint32
    if (words > c->merge_cap) {
        if (c->d_merge) (void)hipFree(c->d_merge);
        c->d_merge = nullptr;
        c->merge_cap = 0;
        HIPCHK(hipMalloc(&c->d_merge, words * sizeof(uint64_t)));
        c->merge_cap = words;
    }
    // (the vector outlives the copy: the call ends with a read-back)
    HIPCHK(hipMemcpyAsync(c->d_merge, plan.data(), plan.size() * sizeof(uint64_t), hipMemcpyHostToDevice, st));
    uint32_t* co = reinterpret_cast<uint32_t*>(c->d_merge + plan.size());
    const key64* sk = nullptr;
    int cur = 0;
    for (const Round& R : rounds) {
        const bool last = R.np == 1;
        uint32_t* di = last ? d_idx_out : ti[cur];
        uint32_t* dl = last ? d_lcp_out : tl[cur];
        key64* dk = last ? nullptr : tk[cur];
        const uint64_t* pf = c->d_merge + R.at;
        const uint64_t* pm = pf + (R.np + 1);
        const uint64_t* pt = pm + (R.np + 1);
        if (R.tiles) {
            const uint32_t lanes = R.tiles < kMergeFew ? 8 : R.tiles < kMergeMany ? 4 : 1;
            const auto part = lanes == 8 ? k_merge_part<8> : lanes == 4 ? k_merge_part<4> : k_merge_part<1>;
            hipLaunchKernelGGL(part, dim3(div_up(R.tiles, kWG / lanes)), dim3(kWG), 0, st, B, si, sk, ik, pf, pm, pt, R.np,
                               co);
            HIPCHK(hipGetLastError());
            hipLaunchKernelGGL(k_merge_tile, dim3(R.tiles), dim3(kWG), 0, st, B, si, sl, sk, ik, di, dl, dk, pf, pm, pt,
                               R.np, co, R.tiles >= kMergeHalf);
            HIPCHK(hipGetLastError());
        }
        si = di;
        sl = dl;
        sk = dk;
        cur ^= 1;
    }
    return readback(c, nullptr, 0);
}

int ps5_dist_chars_device(ps5_ctx* c, const uint8_t* d_arena, uint64_t arena_bytes, const uint32_t* d_offs,
                          uint64_t n, const uint32_t* d_perm, const uint32_t* d_lcp, uint8_t* d_cache)
{
    if (!c) return set_err(PS5_ERR_ARG, "ctx is NULL");
    if (n < 2) return PS5_OK;
    if (!d_arena || !d_offs || !d_perm || !d_lcp || !d_cache) return set_err(PS5_ERR_ARG, "NULL device pointer");
    if (n >= 0xFFFFFF00ull) return set_err(PS5_ERR_ARG, "n too large (limit 2^32-256 strings)");
    HIPCHK(hipSetDevice(c->device));
    HIPCHK(hipMemsetAsync(c->d_cnt, 0, C_NCNT * sizeof(uint32_t), c->stream));
    hipLaunchKernelGGL(k_dist_chars, dim3(div_up(n, kWG)), dim3(kWG), 0, c->stream, d_arena, d_offs, d_perm, d_lcp,
                       (uint32_t)n, d_cache, c->d_cnt, arena_bytes);
    HIPCHK(hipGetLastError());
    int rc = readback(c, nullptr, 0);
    return rc;
}

int ps5_sort_batch_device(ps5_ctx* c, const uint8_t* d_arena, uint64_t arena_bytes, const uint64_t* d_offs,
                          const uint64_t* set_first, uint32_t nsets, uint32_t* d_perm, uint32_t* d_lcp)
{
    if (!c) return set_err(PS5_ERR_ARG, "ctx is NULL");
    if (!set_first || nsets == 0) return set_err(PS5_ERR_ARG, "no sets");
    const uint64_t n = set_first[nsets];
    if (n == 0) return PS5_OK;
    if (!d_arena || !d_offs || !d_perm) return set_err(PS5_ERR_ARG, "NULL device pointer");
    if (n >= 0xFFFFFF00ull) return set_err(PS5_ERR_ARG, "n too large (limit 2^32-256 strings)");
    if (set_first[0] != 0) return set_err(PS5_ERR_ARG, "set_first[0] must be 0");
    if (arena_bytes == 0) return set_err(PS5_ERR_ARG, "empty arena");
    if (((uintptr_t)d_arena & 7u) != 0) return set_err(PS5_ERR_ARG, "arena must be 8-byte aligned");
    HIPCHK(hipSetDevice(c->device));
    int rc = run_sort(c, d_arena, arena_bytes, nullptr, d_offs, (uint32_t)n, d_perm, d_lcp, set_first, nsets);
    if (rc == PS5_OK) {
        if (c->sets_cap < (uint64_t)nsets + 1) {
            if (c->d_sets) (void)hipFree(c->d_sets);
            c->d_sets = nullptr;
            c->sets_cap = 0;
            HIPCHK(hipMalloc(&c->d_sets, ((uint64_t)nsets + 1) * sizeof(uint64_t)));
            c->sets_cap = (uint64_t)nsets + 1;
        }
        HIPCHK(hipMemcpyAsync(c->d_sets, set_first, ((uint64_t)nsets + 1) * sizeof(uint64_t), hipMemcpyHostToDevice,
                              c->stream));
        hipLaunchKernelGGL(k_localize, dim3(div_up(n, kLocTile)), dim3(kWG), 0, c->stream, d_perm, (uint32_t)n, c->d_sets,
                           nsets);
        HIPCHK(hipGetLastError());
        HIPCHK(hipStreamSynchronize(c->stream));
    } else {
        (void)hipStreamSynchronize(c->stream);
        (void)hipStreamSynchronize(c->side);
        if (c->profile) collect_events(c);
    }
    return rc;
}

int ps5_sort_device_timed(ps5_ctx* c, const uint8_t* d_arena, uint64_t arena_bytes, const uint32_t* d_offs,
                          uint64_t n, uint32_t* d_perm, uint32_t* d_lcp, double* ms)
{
    if (!c) return set_err(PS5_ERR_ARG, "ctx is NULL");
    hipEvent_t a, b;
    HIPCHK(hipSetDevice(c->device));
    HIPCHK(hipEventCreate(&a));
    HIPCHK(hipEventCreate(&b));
    (void)hipEventRecord(a, c->stream);
    int rc = ps5_sort_device(c, d_arena, arena_bytes, d_offs, n, d_perm, d_lcp);
    (void)hipEventRecord(b, c->stream);
    (void)hipEventSynchronize(b);
    float f = 0;
    (void)hipEventElapsedTime(&f, a, b);
    if (ms) *ms = f;
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    return rc;
}

int ps5_ctx_set_tuning(ps5_ctx* c, uint32_t leaf_target, uint32_t max_treebits, uint32_t max_oversample)
{
    if (!c) return set_err(PS5_ERR_ARG, "ctx is NULL");
    if (leaf_target < kTinyT || leaf_target > kMaxLeafTarget)
        return set_err(PS5_ERR_ARG, "leaf_target must be in [64, 1024]");
    if (max_treebits < 1 || max_treebits > (uint32_t)kMaxTreebits)
        return set_err(PS5_ERR_ARG, "max_treebits must be in [1, 10]");
    if (max_oversample < 2 || max_oversample > 32 || (max_oversample & 1))
        return set_err(PS5_ERR_ARG, "max_oversample must be even and in [2, 32]");
    c->leaf_target = leaf_target;
    c->max_treebits = max_treebits;
    c->max_oversample = max_oversample;
    return PS5_OK;
}

int ps5_ctx_set_shape(ps5_ctx* c, uint32_t chunk_max, uint32_t chunk_max_root, uint32_t min_tiles, uint32_t leaf_keys)
{
    if (!c) return set_err(PS5_ERR_ARG, "ctx is NULL");
    if (chunk_max < (uint32_t)kChunkMin || chunk_max > kShapeChunkMax)
        return set_err(PS5_ERR_ARG, "chunk_max must be in [%d, %u]", kChunkMin, kShapeChunkMax);
    if (chunk_max_root < (uint32_t)kChunkMin || chunk_max_root > kShapeChunkMaxRoot)
        return set_err(PS5_ERR_ARG, "chunk_max_root must be in [%d, %u]", kChunkMin, kShapeChunkMaxRoot);
    if (min_tiles < 1 || min_tiles > 65536) return set_err(PS5_ERR_ARG, "min_tiles must be in [1, 65536]");
    if (leaf_keys < 1 || leaf_keys > 8) return set_err(PS5_ERR_ARG, "leaf_keys must be in [1, 8]");
    c->chunk_max = chunk_max;
    c->chunk_max_root = chunk_max_root;
    c->min_tiles = min_tiles;
    c->leaf_keys = leaf_keys;
    return PS5_OK;
}

int ps5_ctx_get_shape(ps5_ctx* c, uint32_t* chunk_max, uint32_t* chunk_max_root, uint32_t* min_tiles,
                      uint32_t* leaf_keys)
{
    if (!c) return set_err(PS5_ERR_ARG, "ctx is NULL");
    if (chunk_max) *chunk_max = c->chunk_max;
    if (chunk_max_root) *chunk_max_root = c->chunk_max_root;
    if (min_tiles) *min_tiles = c->min_tiles;
    if (leaf_keys) *leaf_keys = c->leaf_keys;
    return PS5_OK;
}

int ps5_ctx_get_tuning(ps5_ctx* c, uint32_t* leaf_target, uint32_t* max_treebits, uint32_t* max_oversample)
{
    if (!c) return set_err(PS5_ERR_ARG, "ctx is NULL");
    if (leaf_target) *leaf_target = c->leaf_target;
    if (max_treebits) *max_treebits = c->max_treebits;
    if (max_oversample) *max_oversample = c->max_oversample;
    return PS5_OK;
}

int ps5_ctx_set_planning(ps5_ctx* c, int mode)
{
    if (!c) return set_err(PS5_ERR_ARG, "ctx is NULL");
    if (mode < 0 || mode > 2) return set_err(PS5_ERR_ARG, "planning mode %d is not 0 (host), 1 (device) or 2 (auto)", mode);
    c->planning = mode;
    return PS5_OK;
}

int ps5_ctx_get_planning(ps5_ctx* c)
{
    return c ? c->planning : -1;
}

int ps5_ctx_set_graph_rounds(ps5_ctx* c, uint32_t rounds)
{
    if (!c) return set_err(PS5_ERR_ARG, "ctx is NULL");
    if (rounds > kMaxGraphRounds) return set_err(PS5_ERR_ARG, "at most %u captured rounds", kMaxGraphRounds);
    if (rounds != c->graph_rounds) {
        HIPCHK(hipSetDevice(c->device));
        HIPCHK(hipStreamSynchronize(c->stream));
        if (c->graph_exec) (void)hipGraphExecDestroy(c->graph_exec);
        if (c->graph) (void)hipGraphDestroy(c->graph);
        c->graph_exec = nullptr;
        c->graph = nullptr;
        c->graph_key.clear();
    }
    c->graph_rounds = rounds;
    return PS5_OK;
}

int ps5_ctx_get_graph_rounds(ps5_ctx* c)
{
    return c ? (int)c->graph_rounds : -1;
}

int ps5_ctx_set_profile(ps5_ctx* c, int on)
{
    if (!c) return set_err(PS5_ERR_ARG, "ctx is NULL");
    c->profile = on != 0;
    return PS5_OK;
}

int ps5_ctx_kernel_count(ps5_ctx*) { return K_NUM; }

int ps5_ctx_kernel_stat(ps5_ctx* c, int i, const char** name, double* ms, uint64_t* launches, uint64_t* bytes)
{
    if (!c || i < 0 || i >= K_NUM) return set_err(PS5_ERR_ARG, "bad kernel index");
    if (name) *name = kKernelNames[i];
    if (ms) *ms = c->k_ms[i];
    if (launches) *launches = c->k_launch[i];
    if (bytes) *bytes = c->k_bytes[i];
    return PS5_OK;
}

int ps5_ctx_work_stats(ps5_ctx* c, uint64_t* rounds, uint64_t* levels, uint64_t* segments, uint64_t* leaves,
                       uint64_t* syncs)
{
    if (!c) return set_err(PS5_ERR_ARG, "ctx is NULL");
    if (rounds) *rounds = c->st_rounds;
    if (levels) *levels = c->st_levels;
    if (segments) *segments = c->st_segments;
    if (leaves) *leaves = c->st_leaves;
    if (syncs) *syncs = c->st_syncs;
    return PS5_OK;
}

int ps5_dev_malloc(void** p, uint64_t bytes)
{
    if (!p) return set_err(PS5_ERR_ARG, "p is NULL");
    hipError_t e = hipMalloc(p, bytes ? bytes : 1);
    if (e != hipSuccess)
        return set_err(PS5_ERR_NOMEM, "hipMalloc(%llu): %s", (unsigned long long)bytes, hipGetErrorString(e));
    return PS5_OK;
}

int ps5_dev_free(void* p)
{
    if (p) HIPCHK(hipFree(p));
    return PS5_OK;
}

int ps5_memcpy_h2d(void* dst, const void* src, uint64_t bytes)
{
    HIPCHK(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
    return PS5_OK;
}

int ps5_memcpy_d2h(void* dst, const void* src, uint64_t bytes)
{
    HIPCHK(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
    return PS5_OK;
}

int ps5_dev_copy(void* dst, const void* src, uint64_t bytes)
{
    if ((bytes & 15) || ((uintptr_t)dst & 15) || ((uintptr_t)src & 15))
        return set_err(PS5_ERR_ARG, "ps5_dev_copy needs 16-byte aligned pointers and size");
    if (bytes == 0) return PS5_OK;
    const uint64_t n16 = bytes / 16;
    const uint32_t grid = (uint32_t)std::min<uint64_t>((n16 + kWG - 1) / kWG, 65536);
    hipLaunchKernelGGL(k_copy16, dim3(grid), dim3(kWG), 0, nullptr, (const uint4*)src, (uint4*)dst, n16);
    HIPCHK(hipGetLastError());
    HIPCHK(hipDeviceSynchronize());
    return PS5_OK;
}

int ps5_device_synchronize(void)
{
    HIPCHK(hipDeviceSynchronize());
    return PS5_OK;
}

}  // extern "C"

namespace ps5 {

int set_error(int code, const char* fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_err = buf;
    return code;
}

uint64_t work_bytes(uint64_t n)
{
    return work_layout(n, std::min(kShapeChunkMax, kShapeChunkMaxRoot), kMinTiles).total;
}

int widen_offsets(ps5_ctx* c, const uint32_t* d_offs32, const uint64_t* d_first, const uint64_t* d_base,
                  uint32_t nsets, uint64_t n, uint64_t* d_offs64)
{
    if (!c || nsets == 0) return set_err(PS5_ERR_ARG, "widen_offsets: no context or no sets");
    if (n == 0) return PS5_OK;
    HIPCHK(hipSetDevice(c->device));
    hipLaunchKernelGGL(k_widen, dim3(div_up(n, kWG)), dim3(kWG), 0, c->stream, d_offs32, d_first, d_base, nsets, n,
                       d_offs64);
    HIPCHK(hipGetLastError());
    return PS5_OK;
}


int gather_pointers(ps5_ctx* c, const uint32_t* d_perm, const uint32_t* d_offs, uint64_t base, uint64_t n,
                    uint64_t* d_ptrs)
{
    if (!c) return set_err(PS5_ERR_ARG, "gather_pointers: no context");
    if (n == 0) return PS5_OK;
    HIPCHK(hipSetDevice(c->device));
    hipLaunchKernelGGL(k_gather_ptrs, dim3(div_up(n, kWG)), dim3(kWG), 0, c->stream, d_perm, d_offs, base, n, d_ptrs);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(c->stream));
    return PS5_OK;
}

int widen_lcps(ps5_ctx* c, const uint32_t* d_lcp, uint64_t n, uint64_t* d_wide)
{
    if (!c) return set_err(PS5_ERR_ARG, "widen_lcps: no context");
    if (n == 0) return PS5_OK;
    HIPCHK(hipSetDevice(c->device));
    hipLaunchKernelGGL(k_widen_lcp, dim3(div_up(n, kWG)), dim3(kWG), 0, c->stream, d_lcp, n, d_wide);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(c->stream));
    return PS5_OK;
}

}  // namespace ps5
