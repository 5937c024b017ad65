// ps5_kernels.hpp -- shared definitions of the gfx950 pS5 kernels.
//
// Device data layout (one sort, n strings, positions 0..n-1 of the sorted order):
//   arena      characters as given by the caller (never written)
//   offs[n]    uint32 start offset of input string i
//   rec[2][n]  records of 12 bytes (key and input index) as a level of the
//              sample sort leaves them: every chunk of a segment reordered by
//              bucket, in place of the chunk.  Even levels of a round write
//              buffer 0, odd levels buffer 1.  Key and index lie together
//              because a bucket is gathered in short runs: 8 strings of a
//              511-bucket level's chunk of 4096 touched 340 bytes of cache
//              lines in two arrays
//   vpos[2], src[2]  per buffer: for bucket b and chunk c of a segment, the
//              first sorted position and the place in rec of the bucket's
//              strings in that chunk (its run), bucket-major
//   bkey[n]    uint64 scratch: depth key of the first/last position of a leaf
//   sdepth[2][n / 64] uint32 by round parity: characters the strings of the
//              round segment starting at a position are known to share
//   perm[n], lcp[n]  results (caller memory); between rounds perm holds the
//              input indices of the strings that continue
//
// A sort proceeds in rounds; a round compares one key (8 characters, or up to
// 21 in round 0, see KeyFmt) of every string at the depth of its segment.
// Inside a round, segments (contiguous position ranges whose strings share
// the characters before that depth) are split by multi-workgroup
// splitter-tree steps until every piece is a leaf: a block (at most kBlkT
// strings, sorted completely in LDS by one workgroup), a tiny leaf (at most
// 64 strings, one wave) or an equal-key bucket.  Leaves finish their strings
// at this depth (order, LCPs, permutation) and turn every run of equal keys
// without a NUL into a segment of the next round.
//
// A level moves every string once: its chunks are reordered in LDS and
// written back whole, and whoever reads a bucket gathers its runs, one per
// chunk.  Counting first, so that buckets come out contiguous, would read
// every key once more and write and read its bucket and rank (12 bytes).
#pragma once
#include <cstdint>

namespace ps5 {

typedef uint64_t key64;

constexpr int kWG = 256;                     // threads per workgroup (small kernels)
constexpr int kWaves = kWG / 64;             // wave64
constexpr int kBigWG = 1024;                 // threads of the LDS-heavy kernels
constexpr int kBigWaves = kBigWG / 64;
constexpr uint32_t kXcds = 8;                // MI355X: 8 accelerator complex dies
constexpr int kMaxTreebits = 10;             // reference DefaultTreebits
constexpr int kMaxSpl = (1 << kMaxTreebits) - 1;    // 1023 splitters
constexpr int kMaxBkt = 2 * kMaxSpl + 1;            // 2047 buckets
constexpr int kMaxSamples = 4096;            // sample keys of one splitter tree
// A segment's splitters in `trees`, from its gbase on: the level-order tree in
// [0, 1 << k), the sorted splitters in [1 << k, 2 << k).
// A large segment is cut into the fewest equal chunks of at most a per-level
// limit of keys: kPartMax, unless the level is too small to give min_tiles
// chunks that way; then the limit shrinks (not below kChunkMin) so small
// sorts still spread over the GPU.  A chunk is the unit of k_part: one
// workgroup of kPartWaves waves ranks its keys stably and reorders them.
// Longer chunks make longer runs, which the next reader gathers with fewer
// partial cache lines; the records are staged in parts, so that the LDS of
// two workgroups or more fits a CU and one loads while another ranks.  2 GiB
// of random strings sort in 2.24 ms with chunks of 8192 keys, 2.29 with 6144
// and 2.37 with 4096 (the root level alone is faster with 4096, 0.61 ms
// against 0.66, where three workgroups fit).
constexpr int kPartWaves = 8;
constexpr int kPartThreads = kPartWaves * 64;
constexpr int kPartGroups = 16;              // 64-key groups per wave
constexpr int kPartMax = kPartThreads * kPartGroups;
constexpr uint32_t kPartStage = 2752;        // records staged in LDS at a time (a multiple of 4)
constexpr int kChunkMin = 2048;
constexpr uint32_t kHistGroup = 64;          // chunks whose bucket counts are summed together
// limits and defaults of ps5_ctx_set_shape
constexpr uint32_t kShapeChunkMax = 9216, kShapeChunkMaxRoot = 12032;
constexpr uint32_t kMinTiles = 512;
constexpr uint32_t kTinyT = 64;              // leaves sorted by one wave
constexpr uint32_t kDepthShift = 6;          // a slot of sdepth per kTinyT positions
static_assert(1u << kDepthShift == kTinyT, "segments of more than kTinyT strings start in slots of their own");
constexpr uint32_t kBlkT = 2048;             // leaves sorted on chip by one workgroup
constexpr uint32_t kMaxLeafTarget = 1024;    // largest leaf size the fan-out aims at
constexpr uint32_t kRunChunk = 4096;         // equal-key leaves are processed in chunks
// Blocks are kept in four size classes, each sorted by a kernel whose LDS
// fits its largest block: (64, 256], (256, 512], (512, 1024], (1024, 2048].
constexpr int kBlkClasses = 4;
__host__ __device__ constexpr int block_class(uint32_t m)
{
    return m <= 256 ? 0 : m <= 512 ? 1 : m <= 1024 ? 2 : 3;
}

struct Item {            // a segment or a leaf
    uint32_t begin;      // first position
    uint32_t size;       // number of positions
    uint32_t rbeg;       // first position of the round segment it belongs to
    uint32_t flags;      // F_* | key format << kFmtShift | chunk index << kFlagShift
    uint32_t row, nch;   // a bucket: its first entry in vpos/src and its runs (one per chunk of its segment); row of a
                         // tiny F_NEXT segment: its depth
};
// Where a segment's strings are found: F_IDENT (a root: the string at position
// p is input string p) and F_NEXT (a segment of an earlier round: perm[p]) say
// that its keys are still to be read from the arena; otherwise it is a bucket,
// whose strings lie in the runs of its row in buffer F_BUFB.
constexpr uint32_t F_BUFB = 1u;              // rec[1]/vpos[1]/src[1]
constexpr uint32_t F_SORTED = 2u;            // all keys equal (equal bucket)
constexpr uint32_t F_IDENT = 4u;
constexpr uint32_t F_NEXT = 32u;
constexpr uint32_t kFmtShift = 3;            // (flags >> kFmtShift) & 3: format of the segment's keys (KeyFmt)
constexpr uint32_t kFmtMask = 3u << kFmtShift;
constexpr uint32_t kFlagShift = 8;           // flags >> kFlagShift: chunk index of an equal-key chunk

// device counters
enum : int {
    C_LROUND = 0,  // [2] large segments starting a round (round parity)
    C_LLVL = 2,    // [2] large segments of the next level (level parity)
    C_TINY = 4,    // [2] leaf lists (round parity)
    C_BLOCK = 6,   // [4][2] blocks: C_BLOCK + 2 * size class + round parity
    C_RUN = 14,    // [2]
    C_ERR = 16,    // error flags
    C_BDONE = 17,  // [4] blocks of the current round already sorted, per size class (device-driven levels)
    C_RUNCONT = 21,  // [2] equal-key leaves whose strings continue into the next round (round parity)
    C_TDONE = 23,  // tiny leaves and equal-key chunks of the current round finished before its end (device-driven
    C_RDONE = 24,  // levels)
    C_NCNT = 25
};
constexpr uint32_t ERR_CAP = 1u, ERR_LCP = 2u, ERR_BOUNDS = 4u;
constexpr uint32_t ERR_LEVELS = 8u;          // a captured round had more levels than it was built with
constexpr uint32_t ERR_ALPHA = 16u;          // a packed root holds a character outside the alphabet its samples showed
constexpr uint32_t kLutBytes = 256;          // code table of one packed root
constexpr uint32_t kRootCode = kLutBytes + 32;     // the table, then the alphabet as a bitmap

// Formats of a key.  Format 0: 8 characters of 8 bits.  Formats 1..3: codes
// of 3, 4 or 5 bits, 21, 16 or 12 characters (code 0 is the NUL, the
// characters of the alphabet count up from 1 in byte order), left-aligned
// with `pad` zero bits below.  All formats order like the strings.
struct KeyFmt {
    uint32_t mul;        // (bit index * mul) >> 8 = bit index / code bits, for bit indices below 64
    uint32_t cpk;        // characters per key
    uint32_t pad;        // unused low bits
    uint32_t last;       // mask of the last character's code: zero there = the key holds a NUL
};
__host__ __device__ constexpr KeyFmt key_fmt(uint32_t flags)
{
    const uint32_t f = (flags & kFmtMask) >> kFmtShift;
    return f == 0 ? KeyFmt{ 32, 8, 0, 0xFFu } : f == 1 ? KeyFmt{ 86, 21, 1, 7u << 1 }
         : f == 2 ? KeyFmt{ 64, 16, 0, 15u } : KeyFmt{ 52, 12, 4, 31u << 4 };
}

constexpr uint32_t kRecWords = 3;            // key low, key high, index

struct LargeDesc {       // one segment of the multi-workgroup sample-sort step
    Item seg;
    uint32_t nch;        // chunks
    uint32_t chunk;      // keys per chunk (the last one may be short), <= kPartMax
    uint32_t hist_base;  // first entry of this segment's bucket counts (chunk-major, 2 << k per chunk) and of
                         // its vpos/src rows (bucket-major, nch per bucket)
    uint32_t gbase;      // first entry of its group sums: a row of 2 << k first positions, then a row per group; and
                         // of its splitters
    uint32_t k;          // treebits
    uint32_t oversample; // sample keys per splitter
};
__host__ __device__ constexpr uint32_t hist_groups(uint32_t nch) { return (nch + kHistGroup - 1) / kHistGroup; }

struct TileRef {         // one chunk, or one group of kHistGroup chunks
    uint32_t seg;        // index into the LargeDesc array
    uint32_t t;          // chunk or group inside the segment
};

struct LevelHdr {        // totals of one level's multi-workgroup step
    uint32_t nlarge;     // segments (LargeDesc entries)
    uint32_t ntiles;     // chunks (TileRef entries)
    uint32_t ngroups;    // groups of chunks (TileRef entries of the second table)
    uint32_t kmax;       // largest treebits of the level
    uint32_t pad[4];
};

// A level's plan in device memory: the header, then cap_large descriptors,
// then the tables of chunks and of groups (fixed offsets, so a plan written
// on the device needs no pointer arithmetic on the host).
struct Plan {
    const LevelHdr* hdr;
    LargeDesc* desc;     // (k_tree records a root's key format in it)
    const TileRef* tiles;
    const TileRef* groups;
};

struct Sink {            // where new items are appended
    Item* large; Item* block; Item* tiny; Item* run;
    uint32_t* cnt;       // counter base
    int c_large, c_block, c_tiny, c_run;     // counter indices (c_block: of size class 0)
    int c_runcont;       // counter of equal-key leaves that continue (their key holds no NUL)
    uint32_t cap_large, cap_block, cap_tiny, cap_run;   // cap_block: per size class;
                         // class c lives at block + c * cap_block, counter c_block + 2 * c
};

struct Bufs {
    uint32_t n;          // number of strings (bound of every position and index)
    uint32_t* cnt;       // counters (error flags)
    const uint8_t* arena;
    uint64_t alen;
    const uint32_t* offs;      // string start offsets (uint32), or
    const uint64_t* offs64;    // uint64 offsets when non-null (batches over 4 GiB)
    uint32_t* rec;       // two buffers of cap records (kRecWords words) each, one after the other
    uint32_t* vpos;      // two tables of cap_h entries each
    uint32_t* src;
    uint64_t cap, cap_h;
    uint32_t* perm;
    uint32_t* lcp;       // may be null
    key64* bkey;
    uint32_t* hist;      // bucket counts of the level being split
    uint32_t* gsum;      // their sums over groups of chunks
    const uint32_t* pending;   // non-null and non-zero: large segments remain, the round's leaves wait
    uint32_t pending_err;      // ... and that is an error (ERR_LEVELS: a captured graph cannot continue the round)
    // depths of the segments of more than kTinyT strings that start in each
    // kTinyT positions (at most one does): this round's (null in round 0:
    // depth 0) and the next round's
    const uint32_t* sdepth_in;
    uint32_t* sdepth_out;
    uint8_t* lut;              // code tables and alphabets of packed roots, kRootCode bytes per large segment; null: every
                               // key has format 0
    uint32_t widen;            // non-zero: a root's alphabet is the one in lut, not that of its samples
    uint32_t leaf_keys;        // keys (8 characters each) a leaf pass fetches per string at a time, 1..8
};

}  // namespace ps5
