// Mining a database of small graphs out of LDS.
//
// No embedding leaves its graph, so a database is mined graph by graph: the
// graphs are packed once (pack below) into blocks of a few dozen graphs whose
// vertices, label segments and neighbour lists are 16-bit numbers local to
// the block, and k_resident loads one block at a time into LDS and runs every
// query of the call on it there.  Nothing else is read from HBM, and no table
// of partial embeddings is written to it: a wave expands its rows depth
// first, in levels of at most kRCap rows that live in LDS too.
//
// The queries of a call form a trie of operations over tables (a table = the
// partial embeddings of some first steps): extend (a step that makes a wider
// table), count (the last step) and leaves (trailing leaf groups, counted per
// row).  Queries with the same first steps share the operations that make
// those tables.  Counts and algorithmic bytes are kept per operation and
// added up per query on the host.
//
// What bounds it: a wave's chain of dependent LDS reads and scalar
// instructions for each batch of 64 rows and each 64 of their candidates, so
// the waves a CU holds (its LDS) and how evenly they are kept busy.  Measured
// on MI355X, means of four databases each, before = the table engines (a launch
// or more per step of a query, tables in HBM):
//   10 queries on 1,000 small graphs, one by one      849 ->  375 us
//   24 queries on 20,000 graphs, one by one          4714 -> 1890 us
//   131 queries on 17,321 graphs, one call           3.33 -> 1.65 ms
//   256 queries on 100,000 graphs, one call          18.8 -> 9.79 ms
// The split of the work that gives these (figures below are of earlier states,
// each beside its own reference): workgroups take blocks as they
// become free (with every gridDim-th block 3.05 and 11.1 ms), their waves take
// tasks of a block, and a wave without a task gets half of the next table that
// another one makes: one start vertex can hold most of a block's work (without
// this 3.1 and 10.0 ms; one block of one database kept a single wave at work for
// 3.4 of 4.0 ms).  What a block holds beyond its share goes to the whole chip
// in another launch (kRSpare).
#include "common.h"

#include <memory>

#define GV_CONST __attribute__((address_space(4)))

namespace {

// Rows of a level (of a table held at once).  Tables are cut at the cap after
// each 64 candidates, so 64 rows or 96 leave the lanes of the next step half
// empty (batches of 131 / 256 queries: 96 rows 3.8 / 13.0 ms, 112 3.8 / 12.7,
// 128 3.05 / 11.1); 160 make the waves of a CU fewer (3.07 / 10.2 against
// 3.04 / 10.0).
constexpr uint32_t kRCap = 128;
constexpr uint32_t kRCol = 2 * kRCap;            // bytes of a level's column
constexpr uint32_t kRSlotBytes = 64;
constexpr uint32_t kRMaxOps = 1024;              // operations of a launch (16 B of LDS each)
constexpr uint32_t kRMaxTerms = 256;             // counted operations of a launch
constexpr uint32_t kRSmallBytes = 1024;          // programs of up to this size travel as kernel arguments
constexpr uint32_t kRMaxCombos = 256;            // edge-label partitions x vertex labels
constexpr uint32_t kRGraphSpan = 256;            // graph ids a block may span
constexpr uint32_t kRBlockMax = 64u << 10;       // bytes of a block (one graph at least)
constexpr uint32_t kNone = 0xffffffffu;
constexpr uint32_t kNoCol = 0xffffu;

enum { kOpExtend = 0, kOpCount = 1, kOpLeaves = 2 };

// An operation on a table: one cache line, which a wave reads with one scalar
// load.  Columns are named by where their level keeps them (bytes from the
// wave's levels), operations by their place in the program (bytes).
constexpr uint32_t kInBack = 3, kInColl = 4, kInCopy = 10;   // references held here, the rest in RMore
struct ROp {
    uint32_t head;           // kind | nback << 2 | ncoll << 6 | ncopy << 10 | own number << 16
    uint32_t child;          // extend: first operation on the new table; leaves: the first RLeafStep
    uint32_t next;           // next operation on the same table (kNone: none)
    uint32_t cols;           // restriction column (kNoCol: none) | new vertex's column << 16 (kNoCol: not kept);
                             // leaves: width | leaves << 16
    uint32_t dst;            // extend: the new table's first column; count, leaves: number among the counted
    uint32_t back[kInBack];  // label segment (partition x labels + label) | column << 16
    uint32_t coll[kInColl / 2];   // same-label columns, two a word
    uint32_t copy[kInCopy / 2];   // columns the new table takes over, two a word
    uint32_t more;           // RMore of an operation with more references
};
static_assert(sizeof(ROp) == 64, "one cache line");
struct RMore {
    uint32_t back[GV_MAXK - kInBack], coll[GV_MAXK - kInColl], copy[GV_MAXK - kInCopy];
};
struct RLeafStep {
    uint32_t seg;            // label segment | anchor column << 16
    uint32_t cut;            // restriction column (kNoCol: none) | leaves of its group before it << 16 |
                             // of the group of the leaf before << 31
    uint32_t coll;           // same-label columns: the first two
    uint32_t rest;           // their number | the third << 16, or the first of all of them in the column list
};
constexpr uint32_t kLeafColl = 3;

// A share of a block's work for one wave: an operation on start rows [first,
// first + rows) of its label in the block, and below it the `nchild`
// operations from `child` on.  An operation whose children are spread over
// several tasks is accounted by one of them.
struct RTask {
    uint32_t op, label, first, rows, child, nchild, account, pad;
};

// One block of the packed image: bytes [16 off16, 16 (off16 + n16)).  Its
// sections: masks (mask_words planes of nv words: the label segments each
// vertex has), vertex words (first directory entry | graph << 16, the graph
// counted from graph0 rounded down to 32), then 16-bit arrays: the
// directory (start of each present segment in the neighbours, ndir + 1), the
// neighbours (ne), the vertices by label (nv) and where each label starts in
// them (labels + 1).
struct RBlk {
    uint32_t off16, n16, nv, ndir, ne, v0, graph0, gwords;
};

struct RArgs {
    const RBlk* blk;
    const uint4* img;
    uint32_t mask_words;
    // the program (RProg::image; its list of leaf steps' columns begins at
    // o_col bytes); tasks (kSmall: task t is operation 0 on rows [64 t,
    // 64 (t + 1)) of label0)
    const ROp* ops;
    uint32_t o_col;
    const RTask* tasks;
    uint32_t ntasks, label0;
    uint32_t nops, nterms, lmax, lvl_bytes;   // lmax: widest table; lvl_bytes: a wave's levels
    uint32_t gw;                 // graph words per counted operation in LDS
    uint32_t img_bytes;          // LDS of the largest block
    uint32_t nwords;
    // per operation: list entries (leaves: bytes), survivors (counted:
    // embeddings); kRLines copies of 2 nops words, block b adds to copy b mod
    // kRLines
    unsigned long long* acc;
    uint32_t* next;              // blocks handed out beyond the first of each workgroup
    // tables set aside (kAside...), to read and to write: item_words each
    uint32_t nwork;              // blocks, or with `items` tables to take up
    uint32_t item_words;
    const uint32_t* items;       // set aside by the launch before
    uint32_t* aside;             // for the next launch: `naside` of at most aside_cap
    uint32_t* naside;
    uint32_t aside_cap;
    uint32_t busy;               // set aside with so many workgroups at work, or fewer
    uint32_t* done;              // workgroups that have ended: kRLines counters, kRDoneStep words apart
    uint32_t* bits;              // nterms x nwords (nullable)
    uint32_t prog[kRSmallBytes / 4];   // a small program
};

__host__ __device__ constexpr uint32_t rwave_bytes(uint32_t lvl_bytes, uint32_t lmax) {
    return (lvl_bytes + kRSlotBytes + 16 * lmax + 15) & ~15u;
}
constexpr uint32_t kRLines = 16;                 // copies of the accumulators
constexpr uint32_t kRShares = 32;                // shares of a block's work (make_tasks); 16 or 64: within 3%
constexpr uint32_t kRLeastRows = 16;             // start rows of a share
constexpr uint32_t kRLdsMost = 160u << 10;       // LDS of a CU
constexpr uint32_t kRSmallWaves = 4, kRWaves = 8;   // waves of a workgroup, at most
constexpr uint32_t kRGive = 16;                  // rows of a table worth sharing; 4 or 48: within 2%
// Room for the tables that one launch sets aside: at first (a call on a new
// context pays for the allocation: with 4 MiB 920 us instead of 310), and
// after a call that set aside more (131 queries on 6,000 graphs: with 512 KiB
// 2.95 ms, with 4 MiB 1.55).
constexpr uint64_t kRAsideFirst = 512u << 10, kRAsideMost = 4u << 20;
// A wave sets tables aside once it has worked through kRSpare batches of 64
// rows or 64 candidates in a block (about 80 us alone), while a quarter of the
// workgroups that the chip holds or fewer are at work; it looks again every
// kRAgain.  What is set aside costs another launch and a synchronisation (35
// us) and its block's image again, so it does not pay while the chip is busy
// (9 queries on 5,000 hub graphs, heavy in every block: 2008 us with nothing
// set aside, 2085 without this condition, 1857 with it).  Calls on databases
// with hubs, without and with it, and with the table engines:
//   a star query on 6,000 graphs of 20-400 vertices       1380 ->  341 us  ( 289)
//   131 queries on the same, one call                     3.02 -> 1.56 ms  (2.89)
//   9 queries on 8 graphs of 1,450 vertices, one by one   1684 -> 1038 us  (1448)
//   the same, one call                                     867 ->  329 us  ( 588)
//   9 on 20,000 small and 10 such graphs, one by one      2467 -> 1048 us  (2637)
// 600 queries, one by one, on two databases without such hubs: the sum within
// 1%, on one with them 5% less; batches of 24 to 600 of them between 7% more
// (600 us) and 48% less.  kRSpare 100: the sums 0-1% more, the heaviest 10%
// less; half or an eighth of the workgroups: within 5%.
constexpr uint32_t kRSpare = 160, kRAgain = 64;
constexpr uint32_t kRDoneStep = 16;              // words: a cache line
// a workgroup's control words: tasks taken, next block, waves waiting for a
// share (a bit each), waves at work; then each wave's share: given | first
// operation | rows, width << 16 | operations left on a width-2 table
enum { kCtlTask = 0, kCtlNext = 4, kCtlIdle = 8, kCtlBusy = 12, kCtlShare = 16 };
constexpr uint32_t kRCtlBytes = kCtlShare + 16 * kRWaves;

// A table set aside: a wave that has done much in one block leaves the next
// tables it makes to the whole chip, in another launch (a rare star's centre
// can hold nearly all of a query's work, in one block of a thousand).  Words:
// block, first operation, rows | width << 16, operations left on a width-2
// table, first column (bytes), columns; from kRAside on the columns, kRCap
// 16-bit numbers each.
enum { kAsideBlock = 0, kAsideOp = 1, kAsideRows = 2, kAsideLeft = 3, kAsideCol = 4, kAsideCols = 5, kRAside = 8 };
static_assert(kRCap == 128, "a wave moves a column with one word a lane");

extern __shared__ uint4 rlds[];

__device__ __forceinline__ uint32_t ld8(uint32_t o) { return reinterpret_cast<const uint8_t*>(rlds)[o]; }
__device__ __forceinline__ uint32_t ld16(uint32_t o) { return *reinterpret_cast<const uint16_t*>(reinterpret_cast<const char*>(rlds) + o); }
__device__ __forceinline__ uint32_t ld32(uint32_t o) { return *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(rlds) + o); }
__device__ __forceinline__ void st8(uint32_t o, uint32_t v) { reinterpret_cast<uint8_t*>(rlds)[o] = (uint8_t)v; }
__device__ __forceinline__ void st16(uint32_t o, uint32_t v) { *reinterpret_cast<uint16_t*>(reinterpret_cast<char*>(rlds) + o) = (uint16_t)v; }
__device__ __forceinline__ void st32(uint32_t o, uint32_t v) { *reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(rlds) + o) = v; }
__device__ __forceinline__ void add64(uint32_t o, uint64_t v) {
    atomicAdd(reinterpret_cast<unsigned long long*>(reinterpret_cast<char*>(rlds) + o), (unsigned long long)v);
}

// words that other waves of the workgroup change
__device__ __forceinline__ uint32_t* lds_word(uint32_t o) { return reinterpret_cast<uint32_t*>(rlds) + o / 4; }
__device__ __forceinline__ uint32_t ld32_shared(uint32_t o) {
    return __hip_atomic_load(lds_word(o), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void st32_shared(uint32_t o, uint32_t v) {
    __hip_atomic_store(lds_word(o), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ uint32_t uni(uint32_t x) { return __builtin_amdgcn_readfirstlane(x); }
// x in a vector register: k_resident's scalar registers are all taken, so what
// is seldom read does not live in one (uni gets it back)
__device__ __forceinline__ uint32_t vec(uint32_t x) {
    asm volatile("" : "+v"(x));
    return x;
}
// the kernel's arguments, read where they are used and not before
__device__ __forceinline__ const GV_CONST RArgs& rargs() {
    const GV_CONST char* p = (const GV_CONST char*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const GV_CONST RArgs*)p;
}

// LDS written by other lanes of this wave is visible after it
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// inclusive sums over the wave (all 64 lanes active)
__device__ __forceinline__ uint32_t wave_scan_u32(uint32_t x) {
    x += __builtin_amdgcn_update_dpp(0u, x, 0x111, 0xf, 0xf, false);   // row_shr 1, 2, 4, 8
    x += __builtin_amdgcn_update_dpp(0u, x, 0x112, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0u, x, 0x114, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0u, x, 0x118, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0u, x, 0x142, 0xa, 0xf, false);   // row_bcast 15, 31
    x += __builtin_amdgcn_update_dpp(0u, x, 0x143, 0xc, 0xf, false);
    return x;
}
__device__ __forceinline__ uint32_t wave_total_u32(uint32_t x) {
    return __builtin_amdgcn_readlane(wave_scan_u32(x), 63);
}
// a wave's sum, in 32 bits when no lane's value reaches 2^26
__device__ __forceinline__ uint64_t wave_total_u64(uint64_t x) {
    return __ballot(x >> 26) ? wave_sum_u64(x) : wave_total_u32((uint32_t)x);
}

// The wave's view of its block: LDS offsets of the sections.
struct RView {
    uint32_t nv, vinfo, doff, nbr;
    uint32_t wv;             // the wave's levels
};

// label segment `cl` of vertex v in the neighbours: [b, e).  Without a branch
// on the lane: of an absent segment the directory entries read belong to a
// later one.
__device__ __forceinline__ void rseg(const RView& V, uint32_t cl, uint32_t v, uint32_t& b, uint32_t& e) {
    const uint32_t w = ld32(4 * ((cl >> 5) * V.nv + v)), below = (1u << (cl & 31)) - 1;
    uint32_t d = (ld32(V.vinfo + 4 * v) & 0xffffu) + __popc(w & below);
    if (cl >> 5)
        for (uint32_t m = 0; m < (cl >> 5); ++m) d += __popc(ld32(4 * (m * V.nv + v)));
    b = ld16(V.doff + 2 * d);
    e = ld16(V.doff + 2 * d + 2);
    e = w & (below + 1) ? e : b;
}

// entries of neighbours [b, b + len) below x, for the whole wave (len 0 for a
// lane without a search): steps of halving powers of two, as many for all
// lanes as the longest needs
__device__ __forceinline__ uint32_t rbelow(const RView& V, uint32_t b, uint32_t len, uint32_t x) {
    uint32_t step = 1, p = 0;
    if (__ballot(len > 1)) {
        while (__ballot(len >= 2 * step)) step *= 2;
        for (; step > 1; step >>= 1) {
            const uint32_t q = p + step;
            const uint32_t y = ld16(V.nbr + 2 * (b + (q <= len ? q - 1 : 0)));
            p = q <= len && y < x ? q : p;
        }
    }
    const uint32_t y = ld16(V.nbr + 2 * (b + p));
    return p < len && y < x ? p + 1 : p;
}
// whether x is among the neighbours [b, b + len)
__device__ __forceinline__ bool rcontains(const RView& V, uint32_t b, uint32_t len, uint32_t x) {
    const uint32_t p = rbelow(V, b, len, x);
    return p < len && ld16(V.nbr + 2 * (b + p)) == x;
}

// row idx of a column
__device__ __forceinline__ uint32_t rcol(const RView& V, uint32_t col, uint32_t idx) { return ld16(V.wv + col + 2 * idx); }

// Embeddings of one core row of a leaf-group query and their algorithmic
// bytes: the leaves go in one by one, rows = the rows held after each.  With t
// leaves of a group of s candidates placed the next one turns C(s, t) into
// C(s, t + 1) = C(s, t) (s - t) / (t + 1); the product of a row's groups stays
// below 2^57 (leaves_fit), so the division is exact.  For the whole wave.
__device__ __forceinline__ uint64_t rleaf_count(const RView& V, const GV_CONST RLeafStep* leaf, const GV_CONST uint32_t* cols,
                                                uint32_t L0, uint32_t n, uint32_t idx, uint64_t& bytes) {
    uint64_t rows = 1, by = 0;
    uint32_t s = 0, len = 0;
    for (uint32_t j = 0; j < n; ++j) {
        const uint32_t sg = leaf[j].seg, ct = leaf[j].cut, cl = leaf[j].coll, rest = leaf[j].rest;
        if (!(ct >> 31)) {
            uint32_t b, e, bound = 0xffffffffu;
            rseg(V, sg & 0xffffu, rcol(V, sg >> 16, idx), b, e);
            len = s = e - b;
            if ((ct & 0xffffu) != kNoCol) {
                bound = rcol(V, ct & 0xffffu, idx);
                s = rbelow(V, b, len, bound);
            }
            const uint32_t ncoll = rest & 0xffffu, cut = s;
            for (uint32_t i = 0; i < ncoll; ++i) {
                const uint32_t c = ncoll > kLeafColl ? cols[(rest >> 16) + i] : (i == 0 ? cl & 0xffffu : i == 1 ? cl >> 16 : rest >> 16);
                s -= rcontains(V, b, cut, rcol(V, c, idx));
            }
        }
        if (n == 1) {
            bytes = 4u * L0 + 8u + 4u * len;
            return s;
        }
        const uint32_t t = (ct >> 16) & 0x7fffu;
        by += rows * (4u * (L0 + j) + 8u + 4u * len);
        rows = s > t ? rows * (s - t) : 0ull;
        if (t) rows = div_exact(rows, t + 1);
        if (j + 1 < n) by += 4u * (L0 + j + 1) * rows;
    }
    bytes = by;
    return rows;
}

// One workgroup takes blocks of the database; its waves take the block's
// tasks (a width-1 operation and a range of its start vertices) and run each
// down the trie.
// kAside: what it takes are the tables set aside by the launch before.
template <bool kSmall, bool kAside>
__global__ __launch_bounds__(1024) void k_resident(RArgs a) {
    const GV_CONST char* ops;
    if constexpr (kSmall) ops = (const GV_CONST char*)__builtin_amdgcn_kernarg_segment_ptr() + offsetof(RArgs, prog);
    else ops = (const GV_CONST char*)a.ops;
    const GV_CONST RTask* tasks = (const GV_CONST RTask*)a.tasks;
    const uint32_t lane = __lane_id(), wib = uni(threadIdx.x >> 6);
    const uint32_t o_acc = a.img_bytes, o_bits = o_acc + 16 * a.nops;
    const uint32_t o_ctl = (o_bits + 4 * a.nterms * a.gw + 15) & ~15u;
    RView V;
    V.wv = o_ctl + kRCtlBytes + wib * rwave_bytes(a.lvl_bytes, a.lmax);
    const uint32_t o_slot = V.wv + a.lvl_bytes, o_st = o_slot + kRSlotBytes - 16;
    const uint64_t le = lane == 63 ? ~0ull : (2ull << lane) - 1;   // lanes up to this one
    for (uint32_t i = threadIdx.x; i < 4 * a.nops; i += blockDim.x) st32(o_acc + 4 * i, 0);
    for (uint32_t i = threadIdx.x; i < a.nterms * a.gw; i += blockDim.x) st32(o_bits + 4 * i, 0);
    auto match = [&](uint32_t term, uint32_t v) {   // the graph of vertex v holds an embedding
        const uint32_t g = ld32(V.vinfo + 4 * v) >> 16;
        atomicOr(reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(rlds) + o_bits + 4 * (term * a.gw + (g >> 5))),
                 1u << (g & 31));
    };
    uint32_t loaded = kNone;
    for (uint32_t wi = blockIdx.x; wi < a.nwork;) {
        const uint32_t wv = vec(wi);
        const uint32_t bi = kAside ? uni(a.items[(uint64_t)wi * a.item_words]) : wi;
        const RBlk blk = a.blk[bi];
        // The workgroup's next block: the next free one, or for one small
        // query, whose blocks take a few us each, at a fixed stride (the
        // counter's atomics come back about 100 ns apart, from all XCDs in turn).
        uint32_t then = 0;
        constexpr bool counter = !kSmall || kAside;   // tables set aside differ too much for a stride
        if (counter && threadIdx.x == 0) then = atomicAdd(a.next, 1u);
        if (!kAside || bi != loaded)
            for (uint32_t i = threadIdx.x; i < blk.n16; i += blockDim.x) rlds[i] = a.img[(uint64_t)blk.off16 + i];
        if constexpr (kAside) loaded = bi;
        if (threadIdx.x == 0) {
            st32(o_ctl + kCtlTask, 0);
            st32(o_ctl + kCtlIdle, 0);
            st32(o_ctl + kCtlBusy, blockDim.x >> 6);
        }
        V.nv = blk.nv;
        V.vinfo = 4 * a.mask_words * blk.nv;
        V.doff = V.vinfo + 4 * blk.nv;
        V.nbr = V.doff + 2 * (blk.ndir + 1);
        const uint32_t o_lv = V.nbr + 2 * blk.ne, o_lvo = o_lv + 2 * blk.nv;
        __syncthreads();
        uint32_t spare = vec(kRSpare);    // batches before this wave sets tables aside (as int)
        bool drained = false;   // no task is left: this wave takes shares of the others' work
        for (;;) {
            uint32_t opo, n;              // the operation, and rows of the table it reads
            uint32_t base = 1, left = 0;  // width the work began at; operations left on the width-2 table, the one
                                          // running and those to come
            uint32_t child = kNone, nchild = 0;
            bool account = true;
            if (!drained) {
                uint32_t t = 0;
                if (lane == 0) t = atomicAdd(lds_word(o_ctl + kCtlTask), 1u);
                t = uni(t);
                if (t >= (kAside ? blockDim.x >> 6 : a.ntasks)) {
                    drained = true;
                    continue;
                }
                if constexpr (kAside) {
                    const uint32_t* item = a.items + (uint64_t)uni(wv) * a.item_words;
                    opo = uni(item[kAsideOp]);
                    n = uni(item[kAsideRows]);
                    base = n >> 16;
                    n &= 0xffffu;
                    left = uni(item[kAsideLeft]);
                    // the table's rows in shares for the waves
                    const uint32_t share = max(kRGive, (n + (blockDim.x >> 6) - 1) / (blockDim.x >> 6)), first = t * share;
                    if (first >= n) continue;
                    n = min(share, n - first);
                    const uint32_t at = V.wv + uni(item[kAsideCol]), cols = uni(item[kAsideCols]);
                    const uint16_t* from = reinterpret_cast<const uint16_t*>(item + kRAside) + first;
                    for (uint32_t k = 0; k < cols; ++k)
                        for (uint32_t i = lane; i < n; i += 64) st16(at + k * kRCol + 2 * i, from[kRCap * k + i]);
                } else {
                    RTask task;
                    if constexpr (kSmall) task = RTask{0, a.label0, 64 * t, 64, kNone, 0, 1, 0};
                    else task = {tasks[t].op, tasks[t].label, tasks[t].first, tasks[t].rows, tasks[t].child, tasks[t].nchild, tasks[t].account, 0};
                    opo = task.op;
                    child = vec(task.child);
                    nchild = vec(task.nchild);
                    account = task.account;
                    const uint32_t s0 = uni(ld16(o_lvo + 2 * task.label)) + task.first, s1 = uni(ld16(o_lvo + 2 * task.label + 2));
                    if (s0 >= s1) continue;
                    n = s1 - s0 < task.rows ? s1 - s0 : task.rows;
                    for (uint32_t i = lane; i < n; i += 64) st16(V.wv + 2 * i, ld16(o_lv + 2 * (s0 + i)));
                }
                wave_lds_sync();
            } else {
                // Wait for a share.  A giver counts itself and the taker as at
                // work before it gives, so with none at work nothing can come.
                const uint32_t mine = o_ctl + kCtlShare + 16 * wib;
                if (lane == 0) {
                    st32_shared(mine, 0);
                    __hip_atomic_fetch_or(lds_word(o_ctl + kCtlIdle), 1u << wib, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
                    __hip_atomic_fetch_sub(lds_word(o_ctl + kCtlBusy), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                }
                wave_lds_sync();
                uint32_t given;
                for (;;) {
                    given = uni(ld32_shared(mine));
                    if (given || uni(ld32_shared(o_ctl + kCtlBusy)) == 0) break;
                    __builtin_amdgcn_s_sleep(2);
                }
                if (!given) break;
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
                opo = uni(ld32(mine + 4));
                n = uni(ld32(mine + 8));
                base = n >> 16;
                n &= 0xffffu;
                left = uni(ld32(mine + 12));
            }
            // w: width of the current table; cb: first row of the batch being
            // extended, cc: its next candidate; counted: that batch's lists
            // are in the accumulator already
            uint32_t w = base, cb = 0, cc = 0;
            bool counted = false;
            for (;;) {
                const GV_CONST ROp& op = *(const GV_CONST ROp*)(ops + opo);
                const uint32_t head = op.head, kind = head & 3u;
                uint64_t sum0 = 0, sum1 = 0;   // what the operation adds to its accumulator
                uint32_t nn = 0;
                if (kind == kOpLeaves) {
                    const GV_CONST RLeafStep* lf = (const GV_CONST RLeafStep*)(ops + op.child);
                    const uint32_t L0 = op.cols & 0xffffu, nleaf = op.cols >> 16;
                    for (uint32_t r0 = 0; r0 < n; r0 += 64) {
                        const uint32_t r = r0 + lane < n ? r0 + lane : r0;
                        uint64_t by, c = rleaf_count(V, lf, (const GV_CONST uint32_t*)(ops + rargs().o_col), L0, nleaf, r, by);
                        if (r0 + lane >= n) c = by = 0;
                        sum0 += by;
                        sum1 += c;
                        if (c && a.bits) match(op.dst, rcol(V, lf->seg >> 16, r));
                    }
                    sum0 = wave_total_u64(sum0);
                    sum1 = wave_total_u64(sum1);
                } else {
                    const bool extend = kind == kOpExtend;
                    const uint32_t nback = (head >> 2) & 15u, ncoll = (head >> 6) & 15u, ncopy = (head >> 10) & 15u;
                    const uint32_t cut = op.cols & 0xffffu, back0 = op.back[0];
                    const GV_CONST RMore& more = *(const GV_CONST RMore*)(ops + op.more);
                    auto back = [&](uint32_t i) { return i < kInBack ? op.back[i] : more.back[i - kInBack]; };
                    uint32_t suspended = 0, lists = 0, found = 0;
                    for (; cb < n; cb += 64) {
                        if (extend && nn > kRCap - 64) {
                            suspended = counted ? 2 : 1;
                            break;
                        }
                        // the batch's rows: shortest list, cut at the restriction
                        const uint32_t r = cb + lane < n ? cb + lane : cb;
                        uint32_t beg, end, ai = 0;
                        rseg(V, back0 & 0xffffu, rcol(V, back0 >> 16, r), beg, end);
                        uint32_t len = end - beg, sum = len;
                        for (uint32_t i = 1; i < nback; ++i) {
                            const uint32_t be = back(i);
                            uint32_t b, e;
                            rseg(V, be & 0xffffu, rcol(V, be >> 16, r), b, e);
                            const uint32_t l = e - b;
                            sum += l;
                            ai = l < len ? i : ai;
                            beg = l < len ? b : beg;
                            len = l < len ? l : len;
                        }
                        if (cut != kNoCol) len = rbelow(V, beg, len, rcol(V, cut, r));
                        const bool in = cb + lane < n;
                        len = in ? len : 0;
                        if (!counted) lists += in ? sum : 0;
                        counted = false;
                        uint32_t c0 = cc;
                        cc = 0;
                        if (__ballot(len != 0) == 0) continue;
                        const uint32_t incl = wave_scan_u32(len), excl = incl - len;
                        const uint32_t total = __builtin_amdgcn_readlane(incl, 63);
                        spare = vec(spare - 1 - total / 64);
                        for (; c0 < total; c0 += 64) {
                            if (extend && nn > kRCap - 64) {
                                suspended = 2;
                                cc = c0;
                                break;
                            }
                            // the row of each of the 64 candidates: every row
                            // marks its first candidate of them
                            st8(o_slot + lane, 0);
                            wave_lds_sync();
                            if (len && incl > c0 && excl < c0 + 64) st8(o_slot + (excl > c0 ? excl - c0 : 0), lane + 1);
                            wave_lds_sync();
                            const uint64_t heads = __ballot(ld8(o_slot + lane) != 0);
                            const uint32_t src = ld8(o_slot + (63 - __clzll(heads & le))) - 1;
                            const uint32_t j = c0 + lane;
                            const uint32_t at = __shfl(beg - excl, src, 64) + j;
                            const uint32_t sr = cb + src;
                            bool ok = j < total;
                            const uint32_t v = ld16(V.nbr + 2 * (ok ? at : 0u));
                            if (ncoll) {
                                ok &= rcol(V, op.coll[0] & 0xffffu, sr) != v;
                                if (ncoll > 1) {
                                    ok &= rcol(V, op.coll[0] >> 16, sr) != v;
                                    if (ncoll > 2) ok &= rcol(V, op.coll[1] & 0xffffu, sr) != v;
                                    if (ncoll > 3) ok &= rcol(V, op.coll[1] >> 16, sr) != v;
                                    for (uint32_t k = kInColl; k < ncoll; ++k) ok &= rcol(V, more.coll[k - kInColl], sr) != v;
                                }
                            }
                            if (nback > 1) {
                                const uint32_t skip = __shfl(ai, src, 64);
                                for (uint32_t i = 0; i < nback; ++i) {
                                    const uint32_t be = back(i);
                                    uint32_t b, e;
                                    rseg(V, be & 0xffffu, rcol(V, be >> 16, sr), b, e);
                                    const bool has = rcontains(V, b, ok && i != skip ? e - b : 0u, v);
                                    ok = ok && (i == skip || has);
                                }
                            }
                            const uint64_t m = __ballot(ok);
                            const uint32_t hits = (uint32_t)__popcll(m);
                            if (extend) {
                                // the new rows: the columns still needed, and v
                                if (ok) {
                                    const uint32_t p2 = 2 * (nn + lanes_below(m)), nc = op.cols >> 16;
                                    if (nc != kNoCol) st16(V.wv + nc + p2, v);
                                    uint32_t dst = V.wv + op.dst + p2;
                                    for (uint32_t k = 0; k < ncopy && k < kInCopy; k += 2) {
                                        const uint32_t two = op.copy[k / 2];
                                        const uint32_t x = rcol(V, two & 0xffffu, sr), y = rcol(V, two >> 16, sr);
                                        st16(dst + k * kRCol, x);
                                        if (k + 1 < ncopy) st16(dst + (k + 1) * kRCol, y);
                                    }
                                    for (uint32_t k = kInCopy; k < ncopy; ++k) st16(dst + k * kRCol, rcol(V, more.copy[k - kInCopy], sr));
                                }
                                nn += hits;
                            } else {
                                found += hits;
                                if (ok && a.bits) match(op.dst, v);
                            }
                        }
                        if (suspended) break;
                    }
                    sum0 = wave_total_u32(lists);
                    sum1 = extend ? nn : found;
                    if (nn) {
                        const uint32_t s = o_st + 16 * w;
                        st32(s, opo);
                        st32(s + 4, cb | suspended << 16);
                        st32(s + 8, cc);
                        st32(s + 12, n);
                    }
                }
                if (lane < 2 && (w > 1 || account))
                    add64(o_acc + 16 * (head >> 16) + 8 * lane, lane ? sum1 : sum0);
                cb = cc = 0;
                bool aside = false;
                if (nn) {
                    // down to the operations on the new table
                    wave_lds_sync();
                    opo = op.child;
                    if (!kSmall && w == 1) {
                        opo = uni(child);
                        left = uni(nchild);
                    }
                    n = nn;
                    ++w;
                    if (n >= kRGive) {
                        // (a table whose next operation only counts is soon done)
                        if ((int)uni(spare) < 0 && (((const GV_CONST ROp*)(ops + opo))->head & 3u) == kOpExtend) {
                            const GV_CONST RArgs& b = rargs();
                            uint32_t ended = 0;
                            if (lane < kRLines) ended = __hip_atomic_load(b.done + kRDoneStep * lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            uint32_t at = b.aside_cap;
                            if (gridDim.x - wave_total_u32(ended) <= b.busy && lane == 0) at = atomicAdd(b.naside, 1u);
                            at = uni(at);
                            aside = at < b.aside_cap;
                            spare = vec(aside ? 0xffffffffu : kRAgain);
                            if (aside) {
                                uint32_t* to = b.aside + (uint64_t)at * b.item_words;
                                const uint32_t cols = ((head >> 10) & 15u) + (op.cols >> 16 != kNoCol);
                                if (lane == 0) {
                                    to[kAsideBlock] = kAside ? b.items[(uint64_t)uni(wv) * b.item_words + kAsideBlock] : uni(wv);
                                    to[kAsideOp] = opo;
                                    to[kAsideRows] = n | w << 16;
                                    to[kAsideLeft] = left;
                                    to[kAsideCol] = op.dst;
                                    to[kAsideCols] = cols;
                                }
                                for (uint32_t k = 0; k < cols; ++k)
                                    to[kRAside + 64 * k + lane] = ld32(V.wv + op.dst + k * kRCol + 4 * lane);
                            }
                        }
                    }
                    if (!aside && n >= kRGive) {
                        // half of the rows to a wave that has nothing to do
                        const uint32_t idle = uni(ld32_shared(o_ctl + kCtlIdle));
                        if (idle) {
                            const uint32_t to = __builtin_ctz(idle);
                            uint32_t was = 0;
                            if (lane == 0)
                                was = __hip_atomic_fetch_and(lds_word(o_ctl + kCtlIdle), ~(1u << to), __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP);
                            if (uni(was) >> to & 1u) {
                                const uint32_t keep = n > 64 ? 64 : n / 2, give = n - keep;
                                const uint32_t share = o_ctl + kCtlShare + 16 * to;
                                const uint32_t off = (to - wib) * rwave_bytes(a.lvl_bytes, a.lmax);   // its levels from this wave's
                                const uint32_t nc = op.cols >> 16, ncopy = (head >> 10) & 15u;
                                if (lane == 0) __hip_atomic_fetch_add(lds_word(o_ctl + kCtlBusy), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                                if (lane < give) {
                                    const uint32_t from = V.wv + 2 * (keep + lane), at = V.wv + off + 2 * lane;
                                    for (uint32_t k = 0; k < ncopy; ++k) st16(at + op.dst + k * kRCol, ld16(from + op.dst + k * kRCol));
                                    if (nc != kNoCol) st16(at + nc, ld16(from + nc));
                                }
                                if (lane == 0) {
                                    st32(share + 4, opo);
                                    st32(share + 8, give | w << 16);
                                    st32(share + 12, left);
                                }
                                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
                                if (lane == 0) st32_shared(share, 1);
                                n = keep;
                            }
                        }
                    }
                    if (!aside) continue;
                }
                // the next operation on this table, or back up to the
                // narrowest table that has work left
                uint32_t nx = aside || w == 1 || (!kSmall && w == 2 && --left == 0) ? kNone : op.next;
                while (nx == kNone && w > base) {
                    --w;
                    const uint32_t s = o_st + 16 * w;
                    opo = uni(ld32(s));
                    const uint32_t cs = uni(ld32(s + 4));
                    n = uni(ld32(s + 12));
                    if (cs >> 16) {
                        nx = opo;
                        cb = cs & 0xffffu;
                        cc = uni(ld32(s + 8));
                        counted = (cs >> 16) == 2;
                    } else if (w > 1 && (kSmall || w > 2 || --left != 0)) {
                        nx = ((const GV_CONST ROp*)(ops + opo))->next;
                    }
                }
                if (nx == kNone) break;
                opo = nx;
            }
        }
        if (counter && threadIdx.x == 0) st32(o_ctl + kCtlNext, then);
        __syncthreads();
        const uint32_t wnext = gridDim.x + (counter ? uni(ld32(o_ctl + kCtlNext)) : uni(wv));
        if (a.bits) {
            // (a batch reads them again: they are not worth registers while the
            // block is mined; one small query would wait for them)
            const GV_CONST RArgs& a = rargs();
            uint32_t gwords = blk.gwords, graph0 = blk.graph0;
            if constexpr (!kSmall) {
                const RBlk& again = a.blk[kAside ? a.items[(uint64_t)uni(wv) * a.item_words] : uni(wv)];
                gwords = again.gwords;
                graph0 = again.graph0;
            }
            for (uint32_t i = threadIdx.x; i < a.nterms * gwords; i += blockDim.x) {
                const uint32_t term = i / gwords, x = i - term * gwords;
                const uint32_t o = o_bits + 4 * (term * a.gw + x);
                const uint32_t m = ld32(o);
                if (m) {
                    st32(o, 0);
                    atomicOr(&a.bits[(uint64_t)term * a.nwords + (graph0 >> 5) + x], m);
                }
            }
        }
        wi = wnext;
        __syncthreads();
    }
    if (threadIdx.x == 0) atomicAdd(a.done + kRDoneStep * (blockIdx.x % kRLines), 1u);
    for (uint32_t i = threadIdx.x; i < 2 * a.nops; i += blockDim.x) {
        const uint64_t x = *reinterpret_cast<const uint64_t*>(reinterpret_cast<const char*>(rlds) + o_acc + 8 * i);
        if (x) atomicAdd(&a.acc[(blockIdx.x % kRLines) * 2 * a.nops + i], (unsigned long long)x);
    }
}

// The accumulators (their copies added up) and bitsets into pinned host
// memory, cleared for the next launch; or, when the launch set tables aside,
// only their number (naside[which]).
__global__ __launch_bounds__(256) void k_resident_out(unsigned long long* acc, uint32_t nacc, unsigned long long* hacc,
                                                      uint32_t* next, uint32_t* bits, uint64_t nbits, uint32_t* hbits,
                                                      uint32_t* naside, uint32_t which, uint32_t* haside, uint32_t* done) {
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (uint64_t)gridDim.x * blockDim.x;
    // the first of each thread's words are on their way before `left` is known
    const uint32_t left = naside[which];
    uint64_t x = 0;
    uint32_t m = 0;
    if (t < nacc)
#pragma unroll
        for (uint32_t k = 0; k < kRLines; ++k) x += acc[k * nacc + t];
    if (t < nbits) m = bits[t];
    if (t == 0) {
        *next = 0;
        *haside = left;
        naside[which ^ 1] = 0;   // those have been taken up
    }
    if (t < kRLines) done[kRDoneStep * t] = 0;
    if (left) return;
    for (uint64_t i = t; i < nacc;) {
        hacc[i] = x;
#pragma unroll
        for (uint32_t k = 0; k < kRLines; ++k) acc[k * nacc + i] = 0;
        i += stride;
        x = 0;
        if (i < nacc)
#pragma unroll
            for (uint32_t k = 0; k < kRLines; ++k) x += acc[k * nacc + i];
    }
    for (uint64_t i = t; i < nbits;) {
        hbits[i] = m;
        bits[i] = 0;
        i += stride;
        if (i < nbits) m = bits[i];
    }
}

// ---- packing ---------------------------------------------------------------

// label of each vertex from the start tables
__global__ void k_pack_labels(const uint32_t* lverts, uint64_t n, const uint64_t* lvoff, uint32_t nl, uint32_t* lab) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        uint32_t lo = 0, hi = nl;   // the label l with lvoff[l] <= i < lvoff[l + 1]
        while (hi - lo > 1) {
            const uint32_t m = (lo + hi) >> 1;
            if (lvoff[m] <= i) lo = m;
            else hi = m;
        }
        lab[lverts[i]] = lo;
    }
}

// per vertex: label segments present (capped) and neighbours (capped), and
// whether a neighbour lies in another graph
__global__ void k_pack_count(DevGraph g, uint32_t nparts, uint64_t nv1, uint32_t* nd, uint32_t* ne, uint32_t* cross) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t v = 1 + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < nv1; v += stride) {
        uint32_t d = 0, m = 0;
        for (uint32_t p = 0; p < nparts; ++p) {
            const uint32_t* lo = g.loff + (uint64_t)p * g.part_stride + v * g.nl1;
            for (uint32_t l = 0; l + 1 < g.nl1; ++l) d += lo[l + 1] > lo[l];
            m += lo[g.nl1 - 1] - lo[0];
            for (uint32_t q = lo[0]; q < lo[g.nl1 - 1]; ++q)
                if (g.gof[g.nbr[q]] != g.gof[v]) *cross = 1;
        }
        nd[v] = d;
        ne[v] = m;
    }
}

// one workgroup per block of the image
__global__ __launch_bounds__(256) void k_pack(DevGraph g, uint32_t nparts, uint32_t nl, uint32_t mask_words,
                                              const RBlk* blks, uint32_t nblk, const uint32_t* ord, const uint32_t* pos,
                                              const uint32_t* lab, const uint32_t* nd, const uint32_t* ne, uint4* img) {
    __shared__ uint64_t wsum[kWavesPerBlock];
    __shared__ uint32_t hist[kRMaxCombos + 1];
    for (uint32_t b = blockIdx.x; b < nblk; b += gridDim.x) {
        const RBlk k = blks[b];
        uint32_t* mask = reinterpret_cast<uint32_t*>(img + k.off16);
        uint32_t* vinfo = mask + (uint64_t)mask_words * k.nv;
        uint16_t* doff = reinterpret_cast<uint16_t*>(vinfo + k.nv);
        uint16_t* nbr = doff + k.ndir + 1;
        uint16_t* lv = nbr + k.ne;
        uint16_t* lvo = lv + k.nv;
        for (uint32_t i = threadIdx.x; i <= nl; i += blockDim.x) hist[i] = 0;
        __syncthreads();
        uint64_t carry = 0;   // directory entries << 32 | neighbours before this round
        for (uint32_t v0 = 0; v0 < k.nv; v0 += blockDim.x) {
            const uint32_t i = v0 + threadIdx.x;
            const uint32_t v = i < k.nv ? ord[k.v0 + i] : 0u;
            const uint64_t mine = i < k.nv ? (uint64_t)nd[v] << 32 | ne[v] : 0ull;
            // exclusive prefix over the workgroup
            uint64_t x = mine;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const uint64_t y = __shfl_up(x, o, 64);
                if (__lane_id() >= (unsigned)o) x += y;
            }
            if (__lane_id() == 63) wsum[threadIdx.x >> 6] = x;
            __syncthreads();
            uint64_t before = carry, all = 0;
            for (int q = 0; q < kWavesPerBlock; ++q) {
                if (q < (int)(threadIdx.x >> 6)) before += wsum[q];
                all += wsum[q];
            }
            const uint64_t ex = before + x - mine;
            __syncthreads();
            carry += all;
            if (i >= k.nv) continue;
            uint32_t d = (uint32_t)(ex >> 32), m = (uint32_t)ex;
            vinfo[i] = d | (g.gof[v] - (k.graph0 & ~31u)) << 16;
            for (uint32_t q = 0; q < mask_words; ++q) mask[(uint64_t)q * k.nv + i] = 0;
            for (uint32_t p = 0; p < nparts; ++p) {
                const uint32_t* lo = g.loff + (uint64_t)p * g.part_stride + (uint64_t)v * g.nl1;
                for (uint32_t l = 0; l < nl; ++l) {
                    const uint32_t s = lo[l], e = lo[l + 1];
                    if (s == e) continue;
                    const uint32_t cl = p * nl + l;
                    mask[(uint64_t)(cl >> 5) * k.nv + i] |= 1u << (cl & 31);
                    doff[d++] = (uint16_t)m;
                    for (uint32_t q = s; q < e; ++q) nbr[m++] = (uint16_t)(pos[g.nbr[q]] - k.v0);
                }
            }
            atomicAdd(&hist[lab[v]], 1u);
        }
        if (threadIdx.x == 0) doff[k.ndir] = (uint16_t)k.ne;
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t s = 0;
            for (uint32_t l = 0; l <= nl; ++l) {
                const uint32_t c = l < nl ? hist[l] : 0;
                lvo[l] = (uint16_t)s;
                hist[l] = s;
                s += c;
            }
        }
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < k.nv; i += blockDim.x)
            lv[atomicAdd(&hist[lab[ord[k.v0 + i]]], 1u)] = (uint16_t)i;
        __syncthreads();
    }
}

template <class T>
struct DevBuf {   // device memory freed at the end of its scope
    T* p = nullptr;
    ~DevBuf() {
        if (p) (void)hipFree(p);
    }
    bool make(uint64_t n) { return hipMalloc(&p, std::max<uint64_t>(n, 1) * sizeof(T)) == hipSuccess; }
};

}  // namespace

struct ResImage {
    RBlk* d_blk = nullptr;
    uint4* d_img = nullptr;
    uint32_t nblk = 0, mask_words = 0;
    uint32_t img_bytes = 0;               // largest block
    uint32_t gw = 0;                      // most graph words of a block
    uint64_t bytes = 0;
    std::vector<uint32_t> max_start;      // most vertices of a label in one block
};

void res_image_free(gv_graph* g) {
    ResImage* r = g->res;
    if (!r) return;
    if (r->d_blk) (void)hipFree(r->d_blk);
    if (r->d_img) (void)hipFree(r->d_img);
    g->dev_bytes -= r->bytes;
    delete r;
    g->res = nullptr;
}

// Pack the database (gv_graph_set_owner).  Not every graph can be: with an
// edge between two of its graphs, a graph beyond kRBlockMax bytes, or more
// than kRMaxCombos label segments, g->res stays null and the table engines
// mine it.
int res_image_build(gv_graph* g, const uint32_t* graph_of) {
    res_image_free(g);
    const uint32_t np = g->nparts, nl = g->nlabels;
    const uint64_t nv1 = g->nv1, nlab = g->lvoff.back();
    if (np == 0 || (uint64_t)np * nl > kRMaxCombos || nlab == 0 || g->ngraphs < 2) return GV_OK;
    const uint32_t mw = (np * nl + 31) / 32;
    DevBuf<uint32_t> lab, nd, ne, cross, dord, dpos;
    DevBuf<uint64_t> off;
    if (!lab.make(nv1) || !nd.make(nv1) || !ne.make(nv1) || !cross.make(1) || !off.make(nl + 1) || !dord.make(nlab) ||
        !dpos.make(nv1))
        return GV_ERR_NOMEM;
    const DevGraph dg = dev_view(g);
    HIPCHK(hipMemcpy(off.p, g->lvoff.data(), 8ull * (nl + 1), hipMemcpyHostToDevice));
    HIPCHK(hipMemset(cross.p, 0, 4));
    HIPCHK(hipMemset(lab.p, 0xff, 4 * nv1));
    hipLaunchKernelGGL(k_pack_labels, dim3(grid_for(nlab, 256, 4096)), dim3(256), 0, nullptr, g->d_lverts, nlab, off.p, nl, lab.p);
    hipLaunchKernelGGL(k_pack_count, dim3(grid_for(nv1, 256, 8192)), dim3(256), 0, nullptr, dg, np, nv1, nd.p, ne.p, cross.p);
    HIPCHK(hipGetLastError());
    uint32_t crosses = 0;
    std::vector<uint32_t> hlab(nv1), hnd(nv1), hne(nv1);
    HIPCHK(hipMemcpy(&crosses, cross.p, 4, hipMemcpyDeviceToHost));
    if (crosses) return GV_OK;
    HIPCHK(hipMemcpy(hlab.data(), lab.p, 4 * nv1, hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(hnd.data(), nd.p, 4 * nv1, hipMemcpyDeviceToHost));
    HIPCHK(hipMemcpy(hne.data(), ne.p, 4 * nv1, hipMemcpyDeviceToHost));
    // vertices by graph, ids ascending within one
    std::vector<uint64_t> start(g->ngraphs + 1, 0);
    for (uint64_t v = 1; v < nv1; ++v)
        if (hlab[v] != 0xffffffffu) start[graph_of[v] + 1]++;
    for (uint32_t i = 0; i < g->ngraphs; ++i) start[i + 1] += start[i];
    std::vector<uint32_t> ord(nlab), pos(nv1, 0);
    {
        std::vector<uint64_t> at(start.begin(), start.end() - 1);
        for (uint64_t v = 1; v < nv1; ++v)
            if (hlab[v] != 0xffffffffu) {
                const uint64_t p = at[graph_of[v]]++;
                ord[p] = (uint32_t)v;
                pos[v] = (uint32_t)p;
            }
    }
    auto block_bytes = [&](uint64_t nv, uint64_t d, uint64_t e) {
        return 4 * (mw + 1) * nv + 2 * (d + 1 + e + nv + nl + 1);
    };
    uint64_t td = 0, te = 0;
    for (uint64_t i = 0; i < nlab; ++i) {
        td += hnd[ord[i]];
        te += hne[ord[i]];
    }
    // Bytes a block aims at: enough blocks to give every CU several, but no
    // more than 24 KiB, so that a CU holds several workgroups (a batch of 256
    // queries on 100,000 graphs: 16 KiB 10.6 ms, 24 KiB 10.0, 32 KiB 10.0).
    const uint64_t target = std::min<uint64_t>(24u << 10, std::max<uint64_t>(2048, block_bytes(nlab, td, te) / 1024));
    std::unique_ptr<ResImage> r(new ResImage());
    r->mask_words = mw;
    r->max_start.assign(nl, 0);
    std::vector<RBlk> blks;
    std::vector<uint32_t> hist(nl, 0);
    uint64_t off16 = 0, bv = 0, bd = 0, be = 0;
    uint32_t g0 = 0, glast = 0;           // the open block's first and last graph
    auto close = [&](uint64_t vend) {
        if (bv == 0) return;
        RBlk k;
        const uint64_t by = block_bytes(bv, bd, be);
        k.off16 = (uint32_t)off16;
        k.n16 = (uint32_t)((by + 15) / 16);
        k.nv = (uint32_t)bv;
        k.ndir = (uint32_t)bd;
        k.ne = (uint32_t)be;
        k.v0 = (uint32_t)(vend - bv);
        k.graph0 = g0;
        k.gwords = (glast - (g0 & ~31u)) / 32 + 1;
        off16 += k.n16;
        r->img_bytes = std::max(r->img_bytes, k.n16 * 16);
        r->gw = std::max(r->gw, k.gwords);
        for (uint32_t l = 0; l < nl; ++l) {
            r->max_start[l] = std::max(r->max_start[l], hist[l]);
            hist[l] = 0;
        }
        blks.push_back(k);
    };
    for (uint32_t q = 0; q < g->ngraphs; ++q) {
        const uint64_t n = start[q + 1] - start[q];
        if (n == 0) continue;
        uint64_t d = 0, e = 0;
        for (uint64_t i = start[q]; i < start[q + 1]; ++i) {
            d += hnd[ord[i]];
            e += hne[ord[i]];
        }
        if (n > 0xfff0 || d > 0xfff0 || e > 0xfff0 || block_bytes(n, d, e) > kRBlockMax) return GV_OK;
        if (bv && (block_bytes(bv + n, bd + d, be + e) > target || q - (g0 & ~31u) >= kRGraphSpan)) {
            close(start[q]);
            bv = bd = be = 0;
        }
        if (bv == 0) g0 = q;
        glast = q;
        bv += n;
        bd += d;
        be += e;
        for (uint64_t i = start[q]; i < start[q + 1]; ++i) hist[hlab[ord[i]]]++;
    }
    close(nlab);
    r->nblk = (uint32_t)blks.size();
    r->bytes = 16 * off16;
    if (off16 >= 0xffffffffull) return GV_OK;
    if (hipMalloc(&r->d_blk, sizeof(RBlk) * blks.size()) != hipSuccess) return GV_ERR_NOMEM;
    if (hipMalloc(&r->d_img, 16 * off16) != hipSuccess) {
        (void)hipFree(r->d_blk);
        return GV_ERR_NOMEM;
    }
    g->res = r.release();
    ResImage* R = g->res;
    g->dev_bytes += R->bytes;
    HIPCHK(hipMemcpy(R->d_blk, blks.data(), sizeof(RBlk) * blks.size(), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(dord.p, ord.data(), 4 * nlab, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(dpos.p, pos.data(), 4 * nv1, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_pack, dim3(std::min<uint32_t>(R->nblk, 8192)), dim3(256), 0, nullptr, dg, np, nl, mw, R->d_blk,
                       R->nblk, dord.p, dpos.p, lab.p, nd.p, ne.p, R->d_img);
    HIPCHK(hipGetLastError());
    HIPCHK(hipDeviceSynchronize());
    const int most = kRLdsMost;
    for (const auto kernel : {k_resident<true, false>, k_resident<false, false>, k_resident<true, true>, k_resident<false, true>})
        HIPCHK(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, most));
    return GV_OK;
}

// ---- programs and calls ----------------------------------------------------

constexpr uint64_t kRAccBytes = 16ull * kRMaxOps * kRLines;
// words: blocks handed out, tables set aside (two, in turn), workgroups that ended
enum { kTailNext = 0, kTailAside = 1, kTailDone = kRDoneStep };
constexpr uint64_t kRTailBytes = 4 * kRDoneStep * (1 + kRLines);

// A context's buffers of gv_resident_mine, kept between calls (grow only).
struct ResWork {
    char* d_prog = nullptr;               // the program (RProg::image) and the tasks
    char* h_prog = nullptr;               // pinned
    uint64_t prog_cap = 0;
    // kRLines copies of 2 kRMaxOps words and the counters (kTail...), zero
    // between calls
    unsigned long long* d_acc = nullptr;
    uint32_t* d_aside = nullptr;          // tables set aside: twice aside_bytes
    uint64_t aside_bytes = 0, aside_want = kRAsideFirst;
    unsigned long long* h_acc = nullptr;  // pinned: the number set aside, then 2 kRMaxOps words
    uint32_t* d_bits = nullptr;           // zero between calls
    uint32_t* h_bits = nullptr;           // pinned
    uint64_t bits_cap = 0;
    bool dirty = false;                   // a call failed between launch and fold
};

void res_work_free(gv_ctx* c) {
    ResWork* w = c->resw;
    if (!w) return;
    for (void* p : {(void*)w->d_prog, (void*)w->d_acc, (void*)w->d_aside, (void*)w->d_bits})
        if (p) (void)hipFree(p);
    for (void* p : {(void*)w->h_prog, (void*)w->h_acc, (void*)w->h_bits})
        if (p) (void)hipHostFree(p);
    delete w;
    c->resw = nullptr;
}

namespace {

// The operations of a launch: tables and the steps on them, added query by
// query, then laid out as ROp, RMore and RLeafStep.
struct RProg {
    struct Op {
        uint32_t kind, table, child = kNone, term = kNone;   // child: table
        gv_step_t st{};
        gv_leaves_t lv{};
    };
    struct Table {
        uint32_t width, label0, from;     // from: the operation that makes it (kNone: a start table)
        std::vector<uint32_t> ops;
        uint32_t live = 0;                // columns kept
        uint32_t off = 0;                 // where, in a wave's levels
        double rows = 0;                  // expected in a block
        std::vector<uint32_t> labels;     // of its columns
    };
    const gv_graph* g;
    std::vector<Op> ops;
    std::vector<Table> tables;
    std::map<uint32_t, uint32_t> start;   // label -> its start table
    uint32_t nterms = 0, nleaves = 0, lmax = 1;
    std::vector<ROp> code;
    std::vector<RMore> mores;
    std::vector<RLeafStep> leaves;
    std::vector<uint32_t> cols;           // same-label columns of leaf steps
    std::vector<RTask> tasks;
    uint32_t lvl_bytes = 0, nroots = 0, most_cols = 1;

    explicit RProg(const gv_graph* g_) : g(g_) {}

    static bool same(const gv_step_t& x, const gv_step_t& y) {
        return x.label == y.label && x.nback == y.nback && x.ncoll == y.ncoll && x.restrict_col == y.restrict_col &&
               std::equal(x.back_col, x.back_col + x.nback, y.back_col) &&
               std::equal(x.back_part, x.back_part + x.nback, y.back_part) &&
               std::equal(x.coll_col, x.coll_col + x.ncoll, y.coll_col);
    }
    static bool same(const gv_leaves_t& x, const gv_leaves_t& y) {
        if (x.width != y.width || x.k != y.k || x.ngroups != y.ngroups ||
            !std::equal(x.group_of, x.group_of + (x.k - x.width), y.group_of))
            return false;
        for (uint32_t q = 0; q < x.ngroups; ++q) {
            const gv_leaf_group_t &a = x.group[q], &b = y.group[q];
            if (a.anchor_col != b.anchor_col || a.part != b.part || a.m != b.m || a.restrict_col != b.restrict_col ||
                a.label != b.label || a.ncoll != b.ncoll || !std::equal(a.coll_col, a.coll_col + a.ncoll, b.coll_col))
                return false;
        }
        return true;
    }
    uint32_t table(uint32_t width, uint32_t label0, uint32_t from) {
        Table t;
        t.width = width;
        t.label0 = label0;
        t.from = from;
        tables.push_back(t);
        lmax = std::max(lmax, width);
        return (uint32_t)tables.size() - 1;
    }

    // Adds a query's operations; `path` receives them from the start table
    // down.  Returns whether another query had added the first of them.
    bool add(const gv_query_t& q, const gv_leaves_t* lv, std::vector<uint32_t>& path) {
        bool reused = false;
        auto it = start.find(q.label0);
        if (it == start.end()) it = start.emplace(q.label0, table(1, q.label0, kNone)).first;
        uint32_t t = it->second;
        for (uint32_t w = 1;; ++w) {
            const bool leafy = lv && w == lv->width, end = leafy || w + 1 == q.k;
            const uint32_t kind = leafy ? kOpLeaves : (end ? kOpCount : kOpExtend);
            uint32_t id = kNone;
            for (uint32_t x : tables[t].ops)
                if (ops[x].kind == kind && (leafy ? same(ops[x].lv, *lv) : same(ops[x].st, q.step[w]))) id = x;
            if (id == kNone) {
                id = (uint32_t)ops.size();
                Op o;
                o.kind = kind;
                o.table = t;
                if (leafy) {
                    o.lv = *lv;
                    ++nleaves;
                } else {
                    o.st = q.step[w];
                }
                if (end) o.term = nterms++;
                else o.child = table(w + 1, q.label0, id);
                ops.push_back(o);
                tables[t].ops.push_back(id);
            } else if (w == 1) {
                reused = true;
            }
            path.push_back(id);
            if (end) return reused;
            t = ops[id].child;
        }
    }

    // Columns: every table keeps those that an operation on it, or on a table
    // made from it, reads.  A level (one width) has room for its largest table.
    void finish() {
        for (uint32_t t = (uint32_t)tables.size(); t-- > 0;) {   // a table comes after the one it is made from
            uint32_t& live = tables[t].live;
            for (uint32_t x : tables[t].ops) {
                const Op& o = ops[x];
                if (o.kind == kOpLeaves) {
                    for (uint32_t q = 0; q < o.lv.ngroups; ++q) {
                        const gv_leaf_group_t& gr = o.lv.group[q];
                        live |= 1u << gr.anchor_col;
                        if (gr.restrict_col != GV_NONE) live |= 1u << gr.restrict_col;
                        for (uint32_t j = 0; j < gr.ncoll; ++j) live |= 1u << gr.coll_col[j];
                    }
                    continue;
                }
                for (uint32_t i = 0; i < o.st.nback; ++i) live |= 1u << o.st.back_col[i];
                for (uint32_t j = 0; j < o.st.ncoll; ++j) live |= 1u << o.st.coll_col[j];
                if (o.st.restrict_col != GV_NONE) live |= 1u << o.st.restrict_col;
                if (o.child != kNone) live |= tables[o.child].live & ((1u << tables[t].width) - 1);
            }
        }
        // a table's columns follow those of the table it is made from
        for (Table& t : tables) {
            if (t.from != kNone) {
                const Table& u = tables[ops[t.from].table];
                t.off = u.off + kRCol * (uint32_t)__builtin_popcount(u.live);
            } else {
                t.live = 1;
            }
            lvl_bytes = std::max(lvl_bytes, t.off + kRCol * (uint32_t)__builtin_popcount(t.live));
            most_cols = std::max(most_cols, (uint32_t)__builtin_popcount(t.live));
        }
        auto col = [&](const Table& t, uint32_t c) {
            return t.off + kRCol * (uint32_t)__builtin_popcount(t.live & ((1u << c) - 1));
        };
        auto segment = [&](uint32_t part, uint32_t label) { return part * g->nlabels + label; };
        const uint32_t n = (uint32_t)ops.size();
        code.assign(n, ROp{});
        for (uint32_t x = 0; x < n; ++x) {
            const Op& o = ops[x];
            const Table& t = tables[o.table];
            ROp& c = code[x];
            c.child = c.next = kNone;
            c.cols = kNoCol | kNoCol << 16;
            if (t.width == 1) ++nroots;
            for (size_t i = 0; i + 1 < t.ops.size(); ++i)
                if (t.ops[i] == x) c.next = t.ops[i + 1] * (uint32_t)sizeof(ROp);
            if (o.kind == kOpLeaves) {
                const uint32_t nleaf = o.lv.k - o.lv.width;
                c.head = o.kind | x << 16;
                c.child = (uint32_t)leaves.size();   // placed by image()
                c.cols = o.lv.width | nleaf << 16;
                c.dst = o.term;
                uint32_t placed[GV_MAX_LEAF_GROUPS] = {}, before = kNone;
                for (uint32_t j = 0; j < nleaf; ++j) {
                    const uint32_t q = o.lv.group_of[j];
                    const gv_leaf_group_t& gr = o.lv.group[q];
                    RLeafStep f{};
                    f.seg = segment(gr.part, gr.label) | col(t, gr.anchor_col) << 16;
                    f.cut = (gr.restrict_col == GV_NONE ? kNoCol : col(t, gr.restrict_col)) | placed[q]++ << 16 |
                            (q == before ? 1u << 31 : 0u);
                    auto coll = [&](uint32_t i) { return i < gr.ncoll ? col(t, gr.coll_col[i]) : 0u; };
                    f.coll = coll(0) | coll(1) << 16;
                    f.rest = gr.ncoll | coll(2) << 16;
                    if (gr.ncoll > kLeafColl) {
                        f.rest = gr.ncoll | (uint32_t)cols.size() << 16;
                        for (uint32_t i = 0; i < gr.ncoll; ++i) cols.push_back(coll(i));
                    }
                    leaves.push_back(f);
                    before = q;
                }
                continue;
            }
            std::vector<uint32_t> copy;
            uint32_t fresh = kNoCol;
            if (o.kind == kOpExtend) {
                const Table& u = tables[o.child];
                for (uint32_t k = 0; k < t.width; ++k)
                    if (u.live >> k & 1) copy.push_back(col(t, k));
                if (u.live >> t.width & 1) fresh = col(u, t.width);
                c.child = u.ops[0] * (uint32_t)sizeof(ROp);
                c.dst = u.off;
            } else {
                c.dst = o.term;
            }
            RMore m{};
            for (uint32_t i = 0; i < o.st.nback; ++i)
                (i < kInBack ? c.back[i] : m.back[i - kInBack]) =
                    segment(o.st.back_part[i], o.st.label) | col(t, o.st.back_col[i]) << 16;
            for (uint32_t i = 0; i < o.st.ncoll; ++i) {
                const uint32_t v = col(t, o.st.coll_col[i]);
                if (i < kInColl) c.coll[i / 2] |= v << (16 * (i & 1));
                else m.coll[i - kInColl] = v;
            }
            for (uint32_t i = 0; i < copy.size(); ++i) {
                if (i < kInCopy) c.copy[i / 2] |= copy[i] << (16 * (i & 1));
                else m.copy[i - kInCopy] = copy[i];
            }
            if (o.st.nback > kInBack || o.st.ncoll > kInColl || copy.size() > kInCopy) {
                c.more = (uint32_t)mores.size() + 1;   // placed by image()
                mores.push_back(m);
            }
            c.cols = (o.st.restrict_col == GV_NONE ? kNoCol : col(t, o.st.restrict_col)) | fresh << 16;
            c.head = o.kind | (uint32_t)o.st.nback << 2 | (uint32_t)o.st.ncoll << 6 | (uint32_t)copy.size() << 10 | x << 16;
        }
    }

    // The program as the device reads it, at `to` (bytes() of it).
    uint64_t o_more() const { return sizeof(ROp) * code.size(); }
    uint64_t o_leaf() const { return o_more() + sizeof(RMore) * mores.size(); }
    uint64_t o_col() const { return o_leaf() + sizeof(RLeafStep) * leaves.size(); }
    uint64_t bytes() const { return o_col() + 4 * cols.size(); }
    void image(char* to) const {
        ROp* c = reinterpret_cast<ROp*>(to);
        for (size_t i = 0; i < code.size(); ++i) {
            c[i] = code[i];
            if ((c[i].head & 3u) == kOpLeaves) c[i].child = (uint32_t)(o_leaf() + sizeof(RLeafStep) * code[i].child);
            c[i].more = code[i].more ? (uint32_t)(o_more() + sizeof(RMore) * (code[i].more - 1)) : 0u;
        }
        auto put = [&](uint64_t at, const void* from, uint64_t n) {
            if (n) memcpy(to + at, from, n);
        };
        put(o_more(), mores.data(), sizeof(RMore) * mores.size());
        put(o_leaf(), leaves.data(), sizeof(RLeafStep) * leaves.size());
        put(o_col(), cols.data(), 4 * cols.size());
    }
};

// Shares of a block's work for the waves: an operation on a start table, with
// a run of the operations below it, takes as many start rows as bring it to
// 1 / kRShares of the block's expected work (from the label statistics), and
// at most kRCap.  Heavy shares go first.
void make_tasks(RProg& p, const ResImage* R) {
    const gv_graph* g = p.g;
    const uint32_t nl = g->nlabels, n = (uint32_t)p.ops.size();
    std::vector<double> cost(n, 0);   // batches of an operation and of those below it, in a block
    for (uint32_t t = 0; t < p.tables.size(); ++t) {
        RProg::Table& T = p.tables[t];
        if (T.from == kNone) {
            T.labels.assign(1, T.label0);
            T.rows = (double)(g->lvoff[T.label0 + 1] - g->lvoff[T.label0]) / R->nblk;
        } else {
            const RProg::Op& o = p.ops[T.from];
            const RProg::Table& U = p.tables[o.table];
            double f = 1e300;
            for (uint32_t i = 0; i < o.st.nback; ++i) {
                const uint64_t l = U.labels[o.st.back_col[i]], nv = g->lvoff[l + 1] - g->lvoff[l];
                f = std::min(f, (double)g->pair_edges[(o.st.back_part[i] * (uint64_t)nl + l) * nl + o.st.label] /
                                    std::max<double>(1.0, (double)nv));
            }
            T.labels = U.labels;
            T.labels.push_back(o.st.label);
            T.rows = U.rows * f;
            // the hubs that many rows run through have more neighbours than the mean
            T.rows *= o.st.nback > 1 ? 0.2 : 1.5;
        }
    }
    for (uint32_t x = n; x-- > 0;) {
        const RProg::Op& o = p.ops[x];
        cost[x] += 1.0 + p.tables[o.table].rows / 64 * (o.kind == kOpLeaves ? 1.0 : 2.0);
        const uint32_t up = p.tables[o.table].from;
        if (up != kNone) cost[up] += cost[x];
    }
    double all = 0;
    for (uint32_t x = 0; x < n; ++x)
        if (p.tables[p.ops[x].table].from == kNone) all += cost[x];
    const double share = std::max(all / kRShares, 1.0);
    std::vector<std::pair<double, RTask>> out;
    auto put = [&](uint32_t x, uint32_t child, uint32_t nchild, bool account, double c) {
        const uint32_t l0 = p.tables[p.ops[x].table].label0, most = R->max_start[l0];
        const double parts = std::max(1.0, c / share), rows = p.tables[p.ops[x].table].rows;
        const uint32_t step = std::min<uint32_t>(kRCap, std::max<uint32_t>(kRLeastRows, (uint32_t)(rows / parts) + 1));
        for (uint32_t f = 0; f < most; f += step)
            out.push_back({c * step, RTask{x * (uint32_t)sizeof(ROp), l0, f, step, child, nchild, account ? 1u : 0u, 0}});
    };
    for (uint32_t x = 0; x < n; ++x) {
        const RProg::Op& o = p.ops[x];
        if (p.tables[o.table].from != kNone) continue;
        if (o.kind != kOpExtend) {
            put(x, kNone, 0, true, cost[x]);
            continue;
        }
        const std::vector<uint32_t>& below = p.tables[o.child].ops;
        for (size_t i = 0; i < below.size();) {
            size_t j = i;
            double c = 0;
            do c += cost[below[j++]];
            while (j < below.size() && c + cost[below[j]] <= share);
            put(x, below[i] * (uint32_t)sizeof(ROp), (uint32_t)(j - i), i == 0, c);
            i = j;
        }
    }
    std::stable_sort(out.begin(), out.end(), [](const auto& a, const auto& b) { return a.first > b.first; });
    for (auto& t : out) p.tasks.push_back(t.second);
}

// the products of a row's leaf groups stay below 2^57 (rleaf_count)
bool leaves_fit(const gv_leaves_t& d, const gv_graph* g) {
    return (d.k - d.width) * std::log2((double)g->max_deg + 1.0) < 57.0;
}

bool valid_query(const gv_query_t& q, const gv_graph* g) {
    if (q.k < 2 || q.k > GV_MAXK || q.label0 >= g->nlabels) return false;
    for (uint32_t w = 1; w < q.k; ++w)
        if (!valid_step(&q.step[w], w, g)) return false;
    return true;
}

int res_buffers(gv_ctx* c, uint64_t prog, uint64_t bits) {
    if (!c->resw) c->resw = new ResWork();
    ResWork* w = c->resw;
    // (each of the two on its own: a call that found memory for one of them
    // only leaves that one for the next)
    if (!w->d_acc) {
        if (hipMalloc(&w->d_acc, kRAccBytes + kRTailBytes) != hipSuccess) {
            w->d_acc = nullptr;
            return GV_ERR_NOMEM;
        }
        w->dirty = true;
    }
    if (!w->h_acc) {
        if (hipHostMalloc((void**)&w->h_acc, 16 * kRMaxOps + 16, hipHostMallocCoherent) != hipSuccess) {
            w->h_acc = nullptr;
            return GV_ERR_NOMEM;
        }
        *w->h_acc = 0;
    }
    if (w->aside_want > w->aside_bytes) {
        uint32_t* room = nullptr;
        if (hipMalloc(&room, 2 * w->aside_want) == hipSuccess) {
            HIPCHK(hipStreamSynchronize(c->stream));
            if (w->d_aside) HIPCHK(hipFree(w->d_aside));
            w->d_aside = room;
            w->aside_bytes = w->aside_want;
        } else if (w->d_aside) {
            (void)hipGetLastError();   // what there is does as well
            w->aside_want = w->aside_bytes;
        } else {
            return GV_ERR_NOMEM;
        }
    }
    if (prog > w->prog_cap) {
        HIPCHK(hipStreamSynchronize(c->stream));
        if (w->d_prog) HIPCHK(hipFree(w->d_prog));
        if (w->h_prog) HIPCHK(hipHostFree(w->h_prog));
        w->d_prog = w->h_prog = nullptr;
        w->prog_cap = 0;
        const uint64_t n = std::max<uint64_t>(prog, 64 << 10);
        if (hipMalloc((void**)&w->d_prog, n) != hipSuccess || hipHostMalloc((void**)&w->h_prog, n) != hipSuccess)
            return GV_ERR_NOMEM;
        w->prog_cap = n;
    }
    if (bits > w->bits_cap) {
        HIPCHK(hipStreamSynchronize(c->stream));
        if (w->d_bits) HIPCHK(hipFree(w->d_bits));
        if (w->h_bits) HIPCHK(hipHostFree(w->h_bits));
        w->d_bits = w->h_bits = nullptr;
        w->bits_cap = 0;
        if (hipMalloc(&w->d_bits, 4 * bits) != hipSuccess ||
            hipHostMalloc((void**)&w->h_bits, 4 * bits, hipHostMallocCoherent) != hipSuccess)
            return GV_ERR_NOMEM;
        w->bits_cap = bits;
        w->dirty = true;
    }
    if (w->dirty) {
        HIPCHK(hipMemsetAsync(w->d_acc, 0, kRAccBytes + kRTailBytes, c->stream));
        if (w->d_bits) HIPCHK(hipMemsetAsync(w->d_bits, 0, 4 * w->bits_cap, c->stream));
        w->dirty = false;
    }
    return GV_OK;
}

int resident_mine(gv_ctx_t c, gv_graph_t g, uint32_t n, const gv_query_t* const* qs,
                  const gv_leaves_t* const* leaves, uint64_t* counts, uint64_t* alg_bytes,
                  uint32_t* const* bits, uint32_t nwords, gv_resident_stats_t* stats) {
    if (!c || !g || (n && (!qs || !counts || !alg_bytes))) return GV_ERR_ARG;
    if (bits && nwords != (g->ngraphs + 31) / 32) return GV_ERR_ARG;
    for (uint32_t i = 0; i < n; ++i) {
        if (!qs[i] || !valid_query(*qs[i], g)) return GV_ERR_ARG;
        if (leaves && leaves[i] && (!valid_leaves(leaves[i], g) || leaves[i]->k != qs[i]->k)) return GV_ERR_ARG;
    }
    const ResImage* R = g->res;
    if (!gv_resident_ready(c, g)) return GV_ERR_CAPACITY;
    for (uint32_t i = 0; i < n; ++i)
        if (leaves && leaves[i] && !leaves_fit(*leaves[i], g)) return GV_ERR_CAPACITY;
    HIPCHK(hipSetDevice(c->device));
    gv_resident_stats_t st{};
    std::vector<std::vector<uint32_t>> paths;
    for (uint32_t i0 = 0; i0 < n;) {
        // as many queries as one launch takes
        RProg p(g);
        uint32_t i1 = i0;
        paths.clear();
        while (i1 < n && p.ops.size() + qs[i1]->k <= kRMaxOps && p.nterms < kRMaxTerms) {
            paths.emplace_back();
            if (p.add(*qs[i1], leaves ? leaves[i1] : nullptr, paths.back())) st.shared_queries++;
            ++i1;
        }
        p.finish();
        const uint32_t nops = (uint32_t)p.ops.size();
        const uint64_t pb = (p.bytes() + 15) & ~15ull;
        const bool small = p.bytes() <= kRSmallBytes && p.nroots == 1;
        if (!small) make_tasks(p, R);
        const uint64_t tb = sizeof(RTask) * p.tasks.size();
        const uint64_t nb = bits ? (uint64_t)p.nterms * nwords : 0;
        const int rc = res_buffers(c, small ? 0 : pb + tb, nb);
        if (rc == GV_ERR_NOMEM) {
            // the table engines may have what they need already
            (void)hipGetLastError();
            return GV_ERR_CAPACITY;
        }
        if (rc != GV_OK) return rc;
        ResWork* w = c->resw;
        RArgs a;
        a.blk = R->d_blk;
        a.img = R->d_img;
        a.mask_words = R->mask_words;
        a.ops = nullptr;
        a.tasks = nullptr;
        a.o_col = (uint32_t)p.o_col();
        a.label0 = p.tables[0].label0;
        a.ntasks = small ? (R->max_start[p.tables[0].label0] + 63) / 64 : (uint32_t)p.tasks.size();
        a.nops = nops;
        a.nterms = p.nterms;
        a.lmax = p.lmax;
        a.lvl_bytes = p.lvl_bytes;
        a.gw = R->gw;
        a.img_bytes = R->img_bytes;
        a.nwords = nwords;
        a.acc = w->d_acc;
        uint32_t* const tail = reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(w->d_acc) + kRAccBytes);
        uint32_t* const aside[2] = {w->d_aside, w->d_aside + w->aside_bytes / 4};
        unsigned long long* const sums = w->h_acc + 1;
        uint32_t* const left = reinterpret_cast<uint32_t*>(w->h_acc);
        a.next = tail + kTailNext;
        a.done = tail + kTailDone;
        a.nwork = R->nblk;
        a.item_words = kRAside + 64 * p.most_cols;
        a.aside_cap = (uint32_t)(w->aside_bytes / 4 / a.item_words);
        a.bits = bits ? w->d_bits : nullptr;
        if (small) {
            p.image(reinterpret_cast<char*>(a.prog));
        } else {
            p.image(w->h_prog);
            memcpy(w->h_prog + pb, p.tasks.data(), tb);
            HIPCHK(hipMemcpyAsync(w->d_prog, w->h_prog, pb + tb, hipMemcpyHostToDevice, c->stream));
            a.ops = reinterpret_cast<const ROp*>(w->d_prog);
            a.tasks = reinterpret_cast<const RTask*>(w->d_prog + pb);
        }
        const uint32_t fixed = R->img_bytes + 16 * nops + 4 * p.nterms * R->gw + 16 + kRCtlBytes;
        const uint32_t each = rwave_bytes(p.lvl_bytes, p.lmax);
        uint32_t waves = fixed < kRLdsMost ? std::min(kRSmallWaves, (kRLdsMost - fixed) / each) : 0;
        if (!small) {
            // the split of a CU's LDS that holds the most waves, in two
            // workgroups or more: one alone idles at each change of block
            // (131 queries, one database: two of 4 waves 1.72 ms, one of 8 2.14;
            // 256 queries: two of 8 8.75, two of 4 13.9)
            waves = 0;
            uint32_t most = 0;
            for (uint32_t k = 4; k >= 2; --k) {
                const uint32_t room = kRLdsMost / k;
                const uint32_t f = room > fixed ? std::min(kRWaves, (room - fixed) / each) : 0;
                if (k * f > most) {
                    most = k * f;
                    waves = f;
                }
            }
            if (waves == 0) waves = fixed < kRLdsMost ? std::min(kRWaves, (kRLdsMost - fixed) / each) : 0;
        }
        const uint32_t lds = fixed + waves * each;
        if (waves == 0 || lds > kRLdsMost) return GV_ERR_CAPACITY;
        const uint32_t per_cu = std::max<uint32_t>(1, std::min<uint32_t>(kRLdsMost / lds, 32 / waves));
        a.busy = per_cu * (uint32_t)c->num_cu / 4;
        w->dirty = true;
        for (uint32_t turn = 0;; ++turn) {
            a.aside = aside[turn & 1];
            a.naside = tail + kTailAside + (turn & 1);
            {
                ProfScope ps(c, kKindResident);
                const uint32_t grid = std::min<uint32_t>(a.nwork, per_cu * c->num_cu);
                const auto kernel = turn ? (small ? k_resident<true, true> : k_resident<false, true>)
                                         : (small ? k_resident<true, false> : k_resident<false, false>);
                hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * waves), lds, c->stream, a);
                HIPCHK(hipGetLastError());
            }
            hipLaunchKernelGGL(k_resident_out, dim3(grid_for(std::max<uint64_t>(nb, 2 * nops), 256, 512)), dim3(256), 0,
                               c->stream, w->d_acc, 2 * nops, sums, a.next, w->d_bits, nb, w->h_bits,
                               tail + kTailAside, turn & 1, left, a.done);
            HIPCHK(hipGetLastError());
            HIPCHK(hipStreamSynchronize(c->stream));
            st.launches += 1;
            if (*left == 0) break;
            if (*left > a.aside_cap) w->aside_want = kRAsideMost;
            // the tables that were set aside, over the whole chip
            a.items = a.aside;
            a.nwork = std::min<uint32_t>(*left, a.aside_cap);
        }
        w->dirty = false;
        // bytes of each operation from the rows it read, its lists and what it wrote
        std::vector<uint64_t> by(nops);
        for (uint32_t x = 0; x < nops; ++x) {
            const RProg::Op& o = p.ops[x];
            const RProg::Table& t = p.tables[o.table];
            const uint64_t lists = sums[2 * x], found = sums[2 * x + 1];
            const uint64_t rows = t.from == kNone ? g->lvoff[t.label0 + 1] - g->lvoff[t.label0] : sums[2 * t.from + 1];
            by[x] = o.kind == kOpLeaves ? lists
                                        : rows * (4ull * t.width + 8ull * o.st.nback) + 4 * lists +
                                              (o.kind == kOpExtend ? 4ull * (t.width + 1) * found : 0ull);
            st.bytes += by[x];
            st.rows += rows;
            if (x != t.ops[0]) st.fused_rows += rows;   // read again for another operation
        }
        for (uint32_t i = i0; i < i1; ++i) {
            const std::vector<uint32_t>& path = paths[i - i0];
            uint64_t b = 0;
            for (uint32_t x : path) b += by[x];
            counts[i] = sums[2 * path.back() + 1];
            alg_bytes[i] = b;
            if (bits && bits[i]) memcpy(bits[i], w->h_bits + (uint64_t)p.ops[path.back()].term * nwords, 4ull * nwords);
        }
        i0 = i1;
    }
    if (c->prof) c->res_bytes += st.bytes;
    if (stats) *stats = st;
    return GV_OK;
}

}  // namespace

extern "C" {

int gv_resident_info(gv_graph_t g, uint32_t* blocks, uint64_t* bytes) {
    if (!g) return GV_ERR_ARG;
    if (blocks) *blocks = g->res ? g->res->nblk : 0;
    if (bytes) *bytes = g->res ? g->res->bytes : 0;
    return GV_OK;
}

int gv_resident_ready(gv_ctx_t c, gv_graph_t g) { return c && g && g->res && !c->prof_bytes ? 1 : 0; }

int gv_resident_takes(gv_graph_t g, const gv_query_t* q, const gv_leaves_t* leaves) {
    if (!g || !q || !valid_query(*q, g) || (leaves && (!valid_leaves(leaves, g) || leaves->k != q->k))) return 0;
    return g->res && (!leaves || leaves_fit(*leaves, g)) ? 1 : 0;
}

int gv_resident_mine(gv_ctx_t c, gv_graph_t g, uint32_t n, const gv_query_t* const* qs,
                     const gv_leaves_t* const* leaves, uint64_t* counts, uint64_t* alg_bytes,
                     uint32_t* const* bits, uint32_t nwords, gv_resident_stats_t* stats) {
    try {
        return resident_mine(c, g, n, qs, leaves, counts, alg_bytes, bits, nwords, stats);
    } catch (const std::bad_alloc&) {
        // no host memory, as without device memory: the table engines may do.
        // A launch may still be running with this call's buffers.
        if (hipStreamSynchronize(c->stream) != hipSuccess) return GV_ERR_HIP;
        return GV_ERR_CAPACITY;
    }
}

}  // extern "C"
