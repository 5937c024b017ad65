// ps5_device.hpp -- device helpers of the gfx950 pS5 kernels (wave64).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "ps5_kernels.hpp"

namespace ps5 {

__device__ __forceinline__ uint64_t mix64(uint64_t z)
{
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// 8 characters of the arena at byte offset `off`, big-endian, zeroed from the
// first NUL on (the reference's get_char_uint64_simple, stringset.hpp:201-231).
// Two aligned 8-byte loads and a funnel shift; near the arena end the bytes
// are fetched one by one so nothing outside arena[0, alen) is read.
// The arena is global memory: loads through address-space-1 pointers are
// global loads, which wait on the vector memory counter alone (a generic
// pointer would compile to flat loads that also wait for LDS operations).
typedef __attribute__((address_space(1))) const uint64_t g_u64;
typedef __attribute__((address_space(1))) const uint8_t g_u8;
__device__ __forceinline__ key64 load_key(const uint8_t* arena, uint64_t alen, uint64_t off)
{
    const uint64_t a8 = off & ~7ull;
    uint64_t lo, hi;
    if (a8 + 16 <= alen) {
        const g_u64* p = (const g_u64*)(arena + a8);
        lo = p[0];
        hi = p[1];
    } else {
        lo = 0;
        hi = 0;
        const g_u8* b = (const g_u8*)arena;
        for (int i = 0; i < 16; ++i) {
            const uint64_t q = a8 + i;
            if (q < alen) {
                const uint64_t c = b[q];
                if (i < 8) lo |= c << (8 * i);
                else hi |= c << (8 * (i - 8));
            }
        }
    }
    const uint32_t sh = (uint32_t)(off & 7) * 8;
    uint64_t v = sh ? ((lo >> sh) | (hi << (64 - sh))) : lo;
    v = __builtin_bswap64(v);
    // high bit of each byte of t is set iff that byte is non-zero (no carries)
    const uint64_t t = ((v & 0x7F7F7F7F7F7F7F7Full) + 0x7F7F7F7F7F7F7F7Full) | v;
    const uint64_t z = ~t & 0x8080808080808080ull;
    if (z) {
        const uint32_t p = (uint32_t)__clzll((long long)z);   // 8 * index of the first NUL
        v = p ? (v & (~0ull << (64 - p))) : 0ull;
    }
    return v;
}

// The keys at depths off, off+8, ..., off+8(KB-1) of one string: KB+1
// aligned 8-byte loads issued together (load_key near the arena end).  Keys
// past the string's NUL hold whatever follows it; callers use a key only
// while every key before it was NUL-free.
template <int KB>
__device__ __forceinline__ void load_keys(const uint8_t* arena, uint64_t alen, uint64_t off, key64 (&k)[KB],
                                          int nk = KB)
{
    const uint64_t a8 = off & ~7ull;
    if (a8 + 8 * (uint64_t)(nk + 1) > alen) {
#pragma unroll
        for (int i = 0; i < KB; ++i) k[i] = i < nk ? load_key(arena, alen, off + 8 * i) : 0ull;
        return;
    }
    const g_u64* p = (const g_u64*)(arena + a8);
    uint64_t w[KB + 1];
#pragma unroll
    for (int i = 0; i <= KB; ++i) w[i] = i <= nk ? p[i] : 0ull;
    const uint32_t sh = (uint32_t)(off & 7) * 8;
#pragma unroll
    for (int i = 0; i < KB; ++i) {
        uint64_t v = sh ? ((w[i] >> sh) | (w[i + 1] << (64 - sh))) : w[i];
        v = __builtin_bswap64(v);
        const uint64_t t = ((v & 0x7F7F7F7F7F7F7F7Full) + 0x7F7F7F7F7F7F7F7Full) | v;
        const uint64_t z = ~t & 0x8080808080808080ull;
        if (z) {
            const uint32_t q = (uint32_t)__clzll((long long)z);
            v = q ? (v & (~0ull << (64 - q))) : 0ull;
        }
        k[i] = v;
    }
}

// characters the two keys share (lcpKeyType, bingmann-parallel_sample_sort.hpp:225-230)
__device__ __forceinline__ uint32_t lcp_key(key64 a, key64 b)
{
    key64 x = a ^ b;
    return x ? ((uint32_t)__clzll((long long)x) >> 3) : 8u;
}
// non-NUL characters of a key (lcpKeyDepth, bingmann-parallel_sample_sort.hpp:232-237)
__device__ __forceinline__ uint32_t key_depth(key64 a)
{
    return a ? 8u - ((uint32_t)__builtin_ctzll(a) >> 3) : 0u;
}

// the same for keys of format F
__device__ __forceinline__ uint32_t lcp_key(key64 a, key64 b, KeyFmt F)
{
    const key64 x = a ^ b;
    return x ? ((uint32_t)__clzll((long long)x) * F.mul) >> 8 : F.cpk;
}
__device__ __forceinline__ uint32_t key_depth(key64 a, KeyFmt F)
{
    return a ? F.cpk - ((((uint32_t)__builtin_ctzll(a) - F.pad) * F.mul) >> 8) : 0u;
}
__device__ __forceinline__ bool key_ends(key64 a, KeyFmt F) { return ((uint32_t)a & F.last) == 0; }

// The 24 characters from byte offset off as three little-endian words
// (zeros past the arena's end).
struct Chars24 { uint64_t w[3]; };
__device__ __forceinline__ Chars24 load_chars24(const uint8_t* arena, uint64_t alen, uint64_t off)
{
    const uint64_t a8 = off & ~7ull;
    uint64_t v[4];
    if (a8 + 32 <= alen) {
        const g_u64* p = (const g_u64*)(arena + a8);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = p[i];
    } else {
        const g_u8* b = (const g_u8*)arena;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = 0;
        for (uint64_t q = a8; q < alen; ++q) {     // (fewer than 32 bytes are left)
            const uint64_t c = (uint64_t)b[q] << (8 * (q & 7));
            const uint32_t j = (uint32_t)(q - a8) >> 3;
            v[0] |= j == 0 ? c : 0ull;
            v[1] |= j == 1 ? c : 0ull;
            v[2] |= j == 2 ? c : 0ull;
            v[3] |= j == 3 ? c : 0ull;
        }
    }
    const uint32_t sh = (uint32_t)(off & 7) * 8;
    Chars24 r;
#pragma unroll
    for (int i = 0; i < 3; ++i) r.w[i] = sh ? ((v[i] >> sh) | (v[i + 1] << (64 - sh))) : v[i];
    return r;
}

// characters of c before its first NUL (24 if there is none)
__device__ __forceinline__ uint32_t chars_before_nul(const Chars24& c)
{
    uint32_t n = 24;
#pragma unroll
    for (int i = 2; i >= 0; --i) {
        const uint64_t t = ((c.w[i] & 0x7F7F7F7F7F7F7F7Full) + 0x7F7F7F7F7F7F7F7Full) | c.w[i];
        const uint64_t z = ~t & 0x8080808080808080ull;
        if (z) n = 8 * i + ((uint32_t)__builtin_ctzll(z) >> 3);
    }
    return n;
}

// The packed key of c under the code table lut (LDS: 0 for the NUL, 1.. for
// the alphabet, 0x81 for anything else).  A character of the key outside the
// alphabet goes into the bitmap *unknown (global memory, shared with other
// workgroups) and sets *bad.  BITS code bits, BITS * 7 or more of them per
// 32-bit word, so that a character costs a byte extract, a table read and a
// shift-or.
template <int BITS>
__device__ __forceinline__ key64 pack_key(const Chars24& c, const uint8_t* lut, uint32_t* unknown, bool* bad)
{
    constexpr int kPerWord = BITS == 3 ? 10 : BITS == 4 ? 8 : 6;
    constexpr int kChars = BITS == 3 ? 21 : BITS == 4 ? 16 : 12;
    constexpr int kPad = 64 - kChars * BITS;
    uint32_t acc[3] = { 0, 0, 0 }, any = 0;
#pragma unroll
    for (int i = 0; i < kChars; ++i) {
        const uint32_t word = (uint32_t)(c.w[i / 8] >> (32 * ((i / 4) & 1)));
        const uint32_t code = lut[(word >> (8 * (i & 3))) & 0xFFu];
        any |= code;
        acc[i / kPerWord] = (acc[i / kPerWord] << BITS) | code;
    }
    key64 k = ((key64)acc[0] << (64 - kPerWord * BITS)) | ((key64)acc[1] << (64 - 2 * kPerWord * BITS));
    if (kChars > 2 * kPerWord) k |= (key64)acc[2] << kPad;
    const uint32_t len = chars_before_nul(c);
    if (any & 0x80u) {     // rare: an unknown character in the key or in what follows the string
        k = 0;
        for (int i = 0; i < kChars && i < (int)len; ++i) {
            const uint64_t w = i < 8 ? c.w[0] : i < 16 ? c.w[1] : c.w[2];
            const uint32_t ch = (uint32_t)(w >> (8 * (i & 7))) & 0xFFu, code = lut[ch];
            if (code & 0x80u) {
                *bad = true;
                uint32_t* word = unknown + (ch >> 5);
                const uint32_t bit = 1u << (ch & 31);
                if (!(__hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & bit)) atomicOr(word, bit);
            }
            k |= (key64)(code & 0x1Fu) << (64 - (i + 1) * BITS);
        }
        return k;
    }
    if (len < (uint32_t)kChars) k = len ? k & (~0ull << (64 - len * BITS)) : 0ull;
    return k;
}
__device__ __forceinline__ key64 pack_key_fmt(const Chars24& c, uint32_t fmt, const uint8_t* lut, uint32_t* unknown, bool* bad)
{
    return fmt == 1 ? pack_key<3>(c, lut, unknown, bad)
         : fmt == 2 ? pack_key<4>(c, lut, unknown, bad) : pack_key<5>(c, lut, unknown, bad);
}

// tid_x() through an opaque move: values derived from it are recomputed
// where they are used, instead of being hoisted out of the persistent loops
// of the kernels and holding registers across every iteration
__device__ __forceinline__ uint32_t tid_x()
{
    uint32_t t;
    asm volatile("v_mov_b32 %0, %1" : "=v"(t) : "v"((uint32_t)threadIdx.x));
    return t;
}
__device__ __forceinline__ uint32_t lane_id() { return tid_x() & 63u; }
__device__ __forceinline__ uint32_t wave_id() { return (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid_x() >> 6)); }
__device__ __forceinline__ uint64_t lanemask_lt() { return (1ull << lane_id()) - 1ull; }

// (key, position) order: positions are distinct, so the order is total and
// equal keys keep their input order (stable).
__device__ __forceinline__ bool kp_less(key64 ka, uint32_t pa, key64 kb, uint32_t pb)
{
    return ka < kb || (ka == kb && pa < pb);
}

// The lanes holding the same NB-bit bucket id, with few vector instructions
// (all 64 lanes must execute this): every lane ORs its bit (lanebit) into this
// wave's table of 64-bit lane masks at the id's low TB bits, reads the entry
// back -- the lanes agreeing on those bits -- and clears it, and ballots on the
// NB - TB high bits keep the lanes agreeing on the whole id.  tab holds 1 << TB
// entries, zero on entry and zero again on return.  The OR of the lanes' bits
// does not depend on the order the LDS applies them in, and a wave's LDS
// operations complete in issue order, so every read sees all of the ORs.
template <int NB, int TB>
__device__ __forceinline__ uint64_t match_bucket_lds(uint32_t b, uint64_t* tab, uint64_t lanebit)
{
    static_assert(TB >= 1 && TB <= NB, "table bits within the id");
    uint64_t* e = tab + (b & ((1u << TB) - 1));
    __hip_atomic_fetch_or(e, lanebit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    const uint64_t got = __hip_atomic_load(e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    __hip_atomic_store(e, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    uint32_t lo = (uint32_t)got, hi = (uint32_t)(got >> 32);
#pragma unroll
    for (int i = TB; i < NB; ++i) {
        const uint32_t m = (uint32_t)((int32_t)(b << (31 - i)) >> 31);
        const uint64_t nbal = ~(uint64_t)__ballot(m != 0u);
        lo &= (uint32_t)nbal ^ m;
        hi &= (uint32_t)(nbal >> 32) ^ m;
    }
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ void flag_error(uint32_t* cnt, uint32_t e) { atomicOr(&cnt[C_ERR], e); }

// characters the strings of the round segment that starts at rbeg share
__device__ __forceinline__ uint32_t seg_depth(const Bufs& B, uint32_t rbeg)
{
    return B.sdepth_in ? B.sdepth_in[rbeg >> kDepthShift] : 0u;
}
// the same of a leaf of at most kTinyT strings
__device__ __forceinline__ uint32_t tiny_depth(const Bufs& B, const Item& it)
{
    return it.flags & F_NEXT ? it.row : seg_depth(B, it.rbeg);
}

// byte offset of input string i in the arena
__device__ __forceinline__ uint64_t str_off(const Bufs& B, uint32_t i)
{
    return B.offs64 ? B.offs64[i] : (uint64_t)B.offs[i];
}

struct Rec { uint32_t lo, hi, id; };
__device__ __forceinline__ key64 rec_key(const Rec& r) { return ((key64)r.hi << 32) | r.lo; }

// Where a bucket's strings lie: run c holds the positions from V[c] on, at
// S[c] and after in R.
struct Runs {
    const Rec* R;
    const uint32_t* V;
    const uint32_t* S;
    uint32_t nch;
};
__device__ __forceinline__ Runs runs_of(const Bufs& B, const Item& it)
{
    const uint64_t b = it.flags & F_BUFB;
    const uint64_t t = it.row + b * B.cap_h;
    return Runs{ reinterpret_cast<const Rec*>(B.rec) + b * B.cap, B.vpos + t, B.src + t, it.nch };
}
// the run holding position pos: the last of n whose first position is not
// above it (an empty run shares its position with the run after it)
__device__ __forceinline__ uint32_t find_run(const uint32_t* V, uint32_t n, uint32_t pos)
{
    uint32_t lo = 0, hi = n;
    while (lo + 1 < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (V[mid] <= pos) lo = mid;
        else hi = mid;
    }
    return lo;
}
// a place computed from run tables, checked against the buffers' size
__device__ __forceinline__ uint32_t checked_place(const Bufs& B, uint32_t q)
{
    if (q >= B.n) { flag_error(B.cnt, ERR_BOUNDS); q = 0; }
    return q;
}
__device__ __forceinline__ uint32_t run_place(const Bufs& B, const Runs& R, uint32_t pos)
{
    const uint32_t c = find_run(R.V, R.nch, pos);
    return checked_place(B, R.S[c] + (pos - R.V[c]));
}
// the key at depth d of input string id
__device__ __forceinline__ key64 string_key(const Bufs& B, uint32_t id, uint32_t d)
{
    if (id >= B.n) { flag_error(B.cnt, ERR_BOUNDS); id = 0; }
    return load_key(B.arena, B.alen, str_off(B, id) + d);
}

// an item must describe a non-empty range inside [0, n)
__device__ __forceinline__ bool item_ok(const Item& it, const Bufs& B)
{
    return it.size != 0 && it.begin < B.n && it.size <= B.n - it.begin &&
           ((it.flags & (F_IDENT | F_NEXT)) || it.nch != 0);
}

__device__ __forceinline__ void put_item(Item* list, uint32_t cap, uint32_t slot, Item it, uint32_t* cnt)
{
    if (slot < cap) list[slot] = it;
    else flag_error(cnt, ERR_CAP);
}

// Append for every lane with pred: returns its slot (wave-aggregated atomic).
__device__ __forceinline__ uint32_t wave_append(bool pred, uint32_t* counter)
{
    const uint64_t m = __ballot(pred);
    if (m == 0) return 0xFFFFFFFFu;
    const uint32_t leader = (uint32_t)__ffsll((long long)m) - 1;
    uint32_t base = 0;
    if (lane_id() == leader) base = atomicAdd(counter, (uint32_t)__popcll(m));
    base = (uint32_t)__shfl((int)base, (int)leader, 64);
    return base + (uint32_t)__popcll(m & lanemask_lt());
}

// Append an unsorted segment (any size) to the list of its size class.
__device__ __forceinline__ void wave_append_segment(bool pred, Item it, const Sink& s)
{
    const uint32_t m = it.size;
    const bool t = pred && m <= kTinyT;
    const bool bl = pred && m > kTinyT && m <= kBlkT;
    const bool lg = pred && m > kBlkT;
    uint32_t slot;
    slot = wave_append(t, &s.cnt[s.c_tiny]);
    if (t) put_item(s.tiny, s.cap_tiny, slot, it, s.cnt);
#pragma unroll
    for (int c = 0; c < kBlkClasses; ++c) {
        const bool bc = bl && block_class(m) == c;
        slot = wave_append(bc, &s.cnt[s.c_block + 2 * c]);
        if (bc) put_item(s.block + (uint64_t)c * s.cap_block, s.cap_block, slot, it, s.cnt);
    }
    slot = wave_append(lg, &s.cnt[s.c_large]);
    if (lg) put_item(s.large, s.cap_large, slot, it, s.cnt);
}

// Exclusive block scan of one uint32 per thread (NW waves); *total = sum.
template <int NW>
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* total, uint32_t* s_tmp)
{
    const uint32_t lane = lane_id(), w = wave_id();
    uint32_t x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        uint32_t y = (uint32_t)__shfl_up((int)x, d, 64);
        if (lane >= (uint32_t)d) x += y;
    }
    if (lane == 63) s_tmp[w] = x;
    __syncthreads();
    uint32_t wpre = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
        uint32_t t = s_tmp[i];
        wpre += (i < (int)w) ? t : 0u;
        tot += t;
    }
    __syncthreads();
    *total = tot;
    return wpre + x - v;
}

// Exclusive block scans of K uint32 per thread at once (NW waves): ex[k] is
// the sum of v[k] over the threads before this one, tot[k] the block total.
// Two barriers for all K (s_tmp: NW * K entries).
template <int NW, int K>
__device__ __forceinline__ void block_excl_scan_k(const uint32_t (&v)[K], uint32_t (&ex)[K], uint32_t (&tot)[K],
                                                  uint32_t* s_tmp)
{
    const uint32_t lane = lane_id(), w = wave_id();
    uint32_t x[K];
#pragma unroll
    for (int k = 0; k < K; ++k) x[k] = v[k];
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const uint32_t y = (uint32_t)__shfl_up((int)x[k], d, 64);
            if (lane >= (uint32_t)d) x[k] += y;
        }
    }
    if (lane == 63) {
#pragma unroll
        for (int k = 0; k < K; ++k) s_tmp[w * K + k] = x[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        uint32_t wpre = 0, t = 0;
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            const uint32_t u = s_tmp[i * K + k];
            wpre += (i < (int)w) ? u : 0u;
            t += u;
        }
        ex[k] = wpre + x[k] - v[k];
        tot[k] = t;
    }
    __syncthreads();
}

// In-order index of level-order node t of a complete tree with k levels.
__device__ __forceinline__ int inorder_of(int t, int k)
{
    const int l = 31 - __clz(t);
    const int j = t - (1 << l);
    return ((2 * j + 1) << (k - l - 1)) - 1;
}

// Buckets of G keys: b = 2 * lower_bound + [splitter == key]
// (ClassifyTreeSimple::find_bkt, bingmann-sample_sortBTC.hpp:45-72).  The
// descent i = 2i + (key > tree[i]) over the level-order tree ends at the
// number x of splitters below the key; the equality test reads splitter x,
// whose node follows from the number of trailing zeros of x + 1 (one load
// instead of tracking a candidate per level, and no second array).
// The G descents advance level by level together, so their LDS reads are in
// flight at the same time.
template <int G>
__device__ __forceinline__ void classify_keys(const key64 (&key)[G], const key64* s_tree, int k, uint32_t (&b)[G])
{
    // the descent tracks byte offsets into s_tree (8 * node): each level is
    // one LDS read, one compare and one shift-add
    uint32_t a[G];
#pragma unroll
    for (int j = 0; j < G; ++j) a[j] = 8;
    const unsigned char* tb = reinterpret_cast<const unsigned char*>(s_tree);
    for (int l = 0; l < k; ++l) {
#pragma unroll
        for (int j = 0; j < G; ++j)
            a[j] = 2 * a[j] + (key[j] > *reinterpret_cast<const key64*>(tb + a[j]) ? 8u : 0u);
    }
    // a / 8 = 2^k + x; splitter x is node (2^k + x + 1) >> (z + 1), z the
    // trailing zeros of x + 1 (node 0 when every splitter is below the key)
#pragma unroll
    for (int j = 0; j < G; ++j) {
        const uint32_t n = (a[j] >> 3) + 1;
        const uint32_t node = n >> (__builtin_ctz(n) + 1);
        const uint32_t x = n - 1 - (1u << k);
        b[j] = 2 * x + ((node != 0 && s_tree[node] == key[j]) ? 1u : 0u);
    }
}

}  // namespace ps5
