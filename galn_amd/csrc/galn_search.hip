// galn_search.hip -- BWA-aln backtracking search on gfx950 (MI355X), and its C ABI.
//
// Two engines. k_heavy searches a read with a wave, many entries of its stack at a
// time (its comment is further down); every form's reads end there. k_search
// searches a read with a lane (thread-per-read): the plain form's first pops, the
// batched form where it is tuned to hand reads over later, penalties that are not
// positive, re-runs. The lane runs the read as a state machine whose every iteration performs exactly one occurrence (LF)
// lookup, whatever the read is doing -- widths (bwt_cal_width), the seed
// widths, expanding a popped stack entry (bwt_2occ4), or an exact-match tail
// (bwt_match_exact_alt) -- so all 64 lanes of a wave issue their random index
// loads together and the memory system sees one independent gather per lane.
//
// Per-lane search state (reference src/bwtgap_hd.h:338-473):
//   * the priority stack: one LIFO per score bucket, built from 16-entry
//     chunks of 16-byte packed entries; the top of each bucket (chunk id,
//     fill) lives in LDS, the non-empty-bucket bitmask in registers, so a pop
//     is one dependent global load and a push is none. Chunks come from a
//     device-wide pool in granules of 64 chunks: a lane takes granules as its
//     stack grows (lock-free tagged free stack, then a bump counter), keeps a
//     few for its next read and hands the rest back, so a read's stack grows to
//     its true peak without re-runs and the pool holds only what is live;
//   * the exact child of an expansion (pushed last, same score, so always the
//     next pop) stays in registers instead of going through the arena;
//   * width[] / seed_width[] as packed u64 (w:48 | bid:16) in the lane's arena.
// Pops, pushes, cut-offs and records follow the reference exactly, so records,
// record order, pop counts and trace hashes are those of the CPU search.
//
// Forms:
//   plain    one launch per 0x40000 reads (one lane per read, input order), then a
//            wave for each read past 32 pops;
//   batched  one persistent launch over the whole read list; waves claim the next
//            read from a device counter as soon as theirs is done;
//   without allocation  the same inside a static device array.
// Reads that outgrow their record slots, or find the pool exhausted, are re-run
// from scratch in a later launch with more room, so results never depend on
// the capacities chosen (the reference's contract, src/bwtgap_hd.h:10-22).

#include <hip/hip_runtime.h>
#include <cstdlib>
#include <cstring>
#include <rocprim/device/device_scan.hpp>
#include <rocprim/iterator/transform_iterator.hpp>

#include <algorithm>
#include <chrono>
#include <atomic>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <numeric>
#include <type_traits>
#include <vector>

#include "galn_hip.h"

__attribute__((visibility("hidden"))) hipError_t galn_hip_dev_malloc(void **p, size_t bytes);  // galn_index.hip

namespace {

constexpr int CH = 16;                       // entries per stack chunk
constexpr int GRAN = 64;                     // chunks per pool granule
constexpr uint32_t MAX_POOL_CHUNKS = 1u << 28;  // 28-bit chunk ids in the bucket tops
constexpr int MAXB = 256;                    // score buckets (bitmask width)
constexpr int MAXLEN = 1023;                 // read length limit (10-bit entry fields)
constexpr int MAXDIFF = 126;                 // 7-bit n_mm / n_gapo fields (n_mm may reach max_diff + 1)
constexpr uint64_t KMASK = (1ull << 38) - 1; // 38-bit k and l
constexpr uint64_t W48 = (1ull << 48) - 1;
constexpr uint32_t NIL = 0xffffffffu;

constexpr int ERR_STACK = -1;   // lane arena full: re-run in a larger tier
constexpr int ERR_ALN = -2;     // record slots full: re-run with more
constexpr int ERR_SCORE = -3;   // final, as the reference
constexpr int ERR_UNSUP = -5;
constexpr int ERR_OUT = -8;     // output arena full: re-run after it grows
constexpr int ERR_INTERNAL = -9; // stack bookkeeping inconsistent (final)
constexpr int ERR_HEAVY = -10;   // pop budget spent: the read moves to the wave-per-read engine
constexpr int NOFIN = 0x7fffffff;  // k_search helpers: the read goes on
constexpr int HITP = 0x7ffffffe;   // k_search pop: the popped entry is a hit
constexpr int STARTS = 0x7ffffffd; // k_search widths: done, the search is set up

constexpr int MODE_GAPE = 0x01, MODE_LOGGAP = 0x04, MODE_NONSTOP = 0x10;
constexpr int ST_M = 0, ST_I = 1, ST_D = 2;

constexpr uint64_t TR_INIT = 1469598103934665603ull;
constexpr uint64_t TR_PRIME = 1099511628211ull;

struct DMeta {
    uint64_t primary;
    uint64_t seq_len;
    const uint64_t *ext;  // counts at the start of each epoch of blocks, or null (one epoch, 32-bit counts)
    uint32_t eshift;      // log2 of an epoch's blocks
};

// packed stack entry (layout below)
struct __align__(16) Ent {
    uint64_t w0, w1;
};

struct KArgs {
    const uint32_t *bwt;
    DMeta meta;
    // reads
    const uint8_t *query;
    const uint64_t *qoff;
    const int32_t *qlen;
    const int32_t *maxdiff;
    const int32_t *batch;
    const galn_search_opt_t *bopts;
    const int32_t *nstacks;
    // work: list positions [0, n_list); read id = list ? list[pos] : list_base + pos
    const int32_t *list;
    int32_t list_base;
    int32_t n_list;
    int32_t *qnext;          // persistent claims
    int32_t n_slots;
    // per-lane region: widths, seed widths, records, owned granules
    uint8_t *scratch;
    uint64_t slot_bytes;
    uint32_t sw_off, rec_off, own_off;
    int32_t own_cap;         // granules a lane may hold (enough for max_entries)
    int32_t keep;            // granules a lane keeps between reads
    int32_t rec_cap;
    // stack pool
    Ent *pool_chk;           // n_gran * GRAN * CH entries
    uint32_t *pool_link;     // per chunk: previous chunk of its bucket, or next free chunk of its lane
    uint32_t *gnext;         // per granule: next granule in the free stack
    unsigned long long *ghead;  // [NSHARD] free stack heads: tag << 32 | granule (0xffffffff = empty)
    uint32_t *gbump;         // granules never handed out start here
    uint32_t n_gran;
    // results (indexed by read id)
    int32_t *out_n;
    uint64_t *out_off;
    uint64_t *out_pops;
    uint64_t *out_trace;
    uint64_t *out_bytes;     // algorithmic index bytes per read
    galn_aln_rec_t *out_rec;
    uint64_t out_cap;
    unsigned long long *out_top;
    int32_t *fail_list;
    int32_t *fail_n;
    int32_t *fail_kind;      // [0] output full, [1] record slots, [2] stack arena
    unsigned long long *algo_bytes;  // this launch's algorithmic index bytes (final results only)
    int32_t fuse;
    uint64_t pop_budget;     // > 0: reads popping more entries go to heavy_list
    int32_t *heavy_list;
    int32_t *heavy_n;
    // hand-off of a heavy read's widths: slot h (its place in heavy_list) holds
    // [bytes | 3 << 62][W[0..len]][SW[0..seed_len]] ... [0], or 0 when the widths were not kept
    uint64_t *hand;
    uint32_t hand_stride;    // u64 words per slot
    int32_t hand_cap;        // slots
};

// The kernel argument segment as k_search reads it, and a load that the compiler must perform
// where it is written (not hoisted out of the loop into registers).
typedef const __attribute__((address_space(4))) KArgs KArgsC;
template <class T>
__device__ __forceinline__ T cold_ld(const __attribute__((address_space(4))) T *p)
{
    return *reinterpret_cast<const volatile __attribute__((address_space(4))) T *>(p);
}
#define CA(f) cold_ld(&A->f)

// ---------------------------------------------------------------------------
// Occurrence counts. Device index layout: blocks of 128 symbols in 64 bytes,
//   4 x u32  C[c]: row of the first suffix that starts with base c, plus the c's before the block
//   4 x {high bits, low bits, prefix}, one per 32 symbols: the symbols' two bit planes (symbol s of the
//            word at bit 31 - s) and, 7 bits each, the set high bits, set low bits and base 3's of the
//            block before this word.
// A count needs C and one 12-byte word, two loads of one 64-byte line and one masked popcount per
// plane; with the counts as u64 and the planes whole (four 16-byte loads, a masked popcount of every
// plane word) it was 55 vector instructions a position against 25, and 16 registers of loaded data
// against 7. An index of 2^32 symbols or more counts C from the start of its epoch (2^24 blocks), and
// `ext` holds the epochs' own counts; 32-bit counts are all a smaller index needs.
//
// Counts are of the first P symbols of the $-less BWT. Row r of the BWT with $ is symbol r - (r > primary)
// (for r != primary), so the symbols at or before row k - 1 are P = k - (k > primary), k = 0 included, and
// those at or before row l are P = l + (l < primary).

// a value the compiler takes as it is
#define OPAQUE(v) asm("" : "+v"(v))

// what a position's count is computed from
struct OccWord {
    uint4 C;
    uint32_t h, l, pre;
};

struct Sub {
    uint32_t h, l, pre;
};

template <class K>
__device__ __forceinline__ void occ_load(const uint32_t *__restrict__ bwt, K P, OccWord &o)
{
    const uint32_t in = 16u + 12u * ((uint32_t)(P >> 5) & 3u);
    const char *const base = reinterpret_cast<const char *>(bwt);
    Sub sub;
    if constexpr (sizeof(K) == 4) {
        const uint32_t off = ((uint32_t)P >> 7) << 6;  // below 2^31
        uint32_t so = off + (in - 16u);
        OPAQUE(so);  // (one 32-bit offset from the scalar base, not a 64-bit address of its own)
        o.C = *reinterpret_cast<const uint4 *>(base + off);
        sub = *reinterpret_cast<const Sub *>(base + 16 + so);
    } else {
        const uint64_t off = ((uint64_t)P >> 7) << 6;
        o.C = *reinterpret_cast<const uint4 *>(base + off);
        sub = *reinterpret_cast<const Sub *>(base + off + in);
    }
    o.h = sub.h;
    o.l = sub.l;
    o.pre = sub.pre;
}

// counts of all four bases among the first P symbols, each plus its base's first row; `wide`: the index
// has epochs (a constant in the wave engine)
template <class K>
__device__ __forceinline__ void occ_count(const DMeta &m, bool wide, const OccWord &o, K P, K (&c)[4])
{
    const uint32_t out = 0xffffffffu >> ((uint32_t)P & 31u);  // the symbols of the word from P on
    const uint32_t h = o.h & ~out, l = o.l & ~out;
    const uint32_t nh = __builtin_popcount(h) + (o.pre & 127u), nl = __builtin_popcount(l) + ((o.pre >> 7) & 127u);
    const uint32_t n3 = __builtin_popcount(h & l) + ((o.pre >> 14) & 127u);
    const uint32_t n0 = ((uint32_t)P & 127u) - nh - nl + n3;
    c[0] = (K)(o.C.x + n0);
    c[1] = (K)(o.C.y + (nl - n3));
    c[2] = (K)(o.C.z + (nh - n3));
    c[3] = (K)(o.C.w + n3);
    if constexpr (sizeof(K) == 8) {
        if (wide) {
            const ulonglong2 *const e = reinterpret_cast<const ulonglong2 *>(m.ext + 4 * ((P >> 7) >> m.eshift));
            const ulonglong2 e01 = e[0], e23 = e[1];
            c[0] += e01.x;
            c[1] += e01.y;
            c[2] += e23.x;
            c[3] += e23.y;
        }
    }
}

template <class K>
__device__ __forceinline__ K pick4(const K (&v)[4], int c)
{
    // (all four are read first: a choice between elements would become an indexed load of the array,
    // which then lives in scratch memory)
    const K v0 = v[0], v1 = v[1], v2 = v[2], v3 = v[3];
    const K a = (c & 1) ? v1 : v0, b = (c & 1) ? v3 : v2;
    return (c & 2) ? b : a;
}

template <class K>
__device__ __forceinline__ K pos_k(const DMeta &m, K k) { return k - (K)(k > (K)m.primary); }
template <class K>
__device__ __forceinline__ K pos_l(const DMeta &m, K l) { return l + (K)(l < (K)m.primary); }

// 64-byte units of an occurrence query at (k - 1, l) as the reference counts them: one block when
// k = 0 or both positions lie in one 128-symbol block of the .bwt, else two (src/bwtgap_hd.h:158-192)
template <class K>
__device__ __forceinline__ uint32_t occ_units(K Pk, K Pl)
{
    return Pk != 0 && (((Pk - 1) ^ (Pl - 1)) >> 7) != 0 ? 2u : 1u;
}

// bwt_2occ4 (src/bwtgap_hd.h:158-192) of the interval [k, l] on an index of any size: ca, cb are the
// counts at rows k - 1 and l, each plus the base's first row, so that a child's interval is
// [ca[c] + 1, cb[c]]. Returns the query's algorithmic bytes.
__device__ __forceinline__ uint32_t lf_pair(const uint32_t *__restrict__ bwt, const DMeta &m, uint64_t k, uint64_t l,
                                            uint64_t (&ca)[4], uint64_t (&cb)[4])
{
    const uint64_t Pk = pos_k<uint64_t>(m, k), Pl = pos_l<uint64_t>(m, l);
    OccWord A, B;
    occ_load<uint64_t>(bwt, Pk, A);
    occ_load<uint64_t>(bwt, Pl, B);
    occ_count<uint64_t>(m, m.ext != nullptr, A, Pk, ca);
    occ_count<uint64_t>(m, m.ext != nullptr, B, Pl, cb);
    return occ_units<uint64_t>(Pk, Pl) << 6;
}

// What the .bwt header says of a body: the bases' first rows (L2[4] = the symbols), and the block that the
// end of the text is counted in where the text fills the block before it (~0 otherwise). A position at the end
// reads that block's counts, which are the totals of the header: of the body's own words only those of
// blocks with symbols are taken, as the .bwt readers of the reference do.
struct Totals {
    uint64_t L2[5], end;
};

// `ext` of an uploaded .bwt body (before k_planes rewrites it): per epoch and base, the base's first row
// plus its count before the epoch's first block
__global__ void k_epochs(const uint32_t *bwt, uint64_t n_blocks, uint32_t eshift, Totals T, uint64_t *ext, uint32_t n)
{
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 4 * n) return;
    const uint64_t blk = (uint64_t)(t >> 2) << eshift;
    const int c = (int)(t & 3);
    const uint64_t before = blk < n_blocks ? reinterpret_cast<const uint64_t *>(bwt + (blk << 4))[c] : 0;
    ext[t] = blk == T.end ? T.L2[c + 1] : T.L2[c] + before;
}

// In-place conversion of the uploaded .bwt body (BWA's blocks: 4 x u64 exclusive counts, 8 words of 16
// two-bit symbols, first symbol in bits 31-30) to the device layout, one block per thread (a last, shorter
// block included: what lies past its symbols is never counted).
__global__ void __launch_bounds__(256)
    k_planes(uint32_t *bwt, uint64_t n_blocks, Totals T, const uint64_t *ext, uint32_t eshift, int wide)
{
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_blocks) return;
    uint4 *const p = reinterpret_cast<uint4 *>(bwt + (i << 4));
    const uint4 c0 = p[0], c1 = p[1], s0 = p[2], s1 = p[3];
    const uint32_t w[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
    uint32_t hp[4] = {0, 0, 0, 0}, lp[4] = {0, 0, 0, 0}, pre[4];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            const int sym = k * 16 + t;  // symbol index in the block
            const uint32_t c = (w[k] >> (30 - 2 * t)) & 3u;
            hp[sym >> 5] |= (c >> 1) << (31 - (sym & 31));
            lp[sym >> 5] |= (c & 1u) << (31 - (sym & 31));
        }
    }
    uint32_t nh = 0, nl = 0, n3 = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        pre[j] = nh | nl << 7 | n3 << 14;
        nh += __builtin_popcount(hp[j]);
        nl += __builtin_popcount(lp[j]);
        n3 += __builtin_popcount(hp[j] & lp[j]);
    }
    // 32 bits: the count from the epoch's start, or (one epoch) the base's first row and the count
    const uint64_t *const e = ext + (wide ? 4 * (i >> eshift) : 0);
    uint64_t C[4] = {(uint64_t)c0.y << 32 | c0.x, (uint64_t)c0.w << 32 | c0.z, (uint64_t)c1.y << 32 | c1.x, (uint64_t)c1.w << 32 | c1.z};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const uint64_t row = i == T.end ? T.L2[c + 1] : C[c] + ext[c];
        C[c] = wide ? row - e[c] : row;
    }
    p[0] = make_uint4((uint32_t)C[0], (uint32_t)C[1], (uint32_t)C[2], (uint32_t)C[3]);
    p[1] = make_uint4(hp[0], lp[0], pre[0], hp[1]);
    p[2] = make_uint4(lp[1], pre[1], hp[2], lp[2]);
    p[3] = make_uint4(pre[2], hp[3], lp[3], pre[3]);
}

// ---------------------------------------------------------------------------
// Packed stack entry (16 bytes); the score is the bucket.
//   w0 = k[0:38) | i[38:48) | n_mm[48:55) | n_gapo[55:62) | state[62:64)
//   w1 = l[0:38) | last_diff_pos[38:48) | n_gape[48:56) | n_ins[56:64)
// n_del = n_gapo + n_gape - n_ins (every gap open or extension adds one
// inserted or one deleted base, src/bwtgap_hd.h:430-454).


__device__ __forceinline__ Ent mk_ent(uint64_t k, uint64_t l, int i, int ldp, int mm, int go, int ge, int ins, int st)
{
    // the fields first, so that children differing only in (k, l) share them
    const uint64_t h0 = ((uint64_t)i << 38) | ((uint64_t)mm << 48) | ((uint64_t)go << 55) | ((uint64_t)st << 62);
    const uint64_t h1 = ((uint64_t)ldp << 38) | ((uint64_t)ge << 48) | ((uint64_t)ins << 56);
    Ent e;
    e.w0 = h0 | (k & KMASK);
    e.w1 = h1 | (l & KMASK);
    return e;
}
__device__ __forceinline__ uint64_t e_k(const Ent &e) { return e.w0 & KMASK; }
__device__ __forceinline__ int e_i(const Ent &e) { return (int)((e.w0 >> 38) & 1023); }
__device__ __forceinline__ int e_mm(const Ent &e) { return (int)((e.w0 >> 48) & 127); }
__device__ __forceinline__ int e_go(const Ent &e) { return (int)((e.w0 >> 55) & 127); }
__device__ __forceinline__ int e_st(const Ent &e) { return (int)(e.w0 >> 62); }
__device__ __forceinline__ uint64_t e_l(const Ent &e) { return e.w1 & KMASK; }
__device__ __forceinline__ int e_ldp(const Ent &e) { return (int)((e.w1 >> 38) & 1023); }
__device__ __forceinline__ int e_ge(const Ent &e) { return (int)((e.w1 >> 48) & 255); }
__device__ __forceinline__ int e_ins(const Ent &e) { return (int)(e.w1 >> 56); }

__device__ __forceinline__ uint64_t tr_mix(uint64_t h, uint64_t v) { return (h ^ v) * TR_PRIME; }

__device__ __forceinline__ int int_log2(uint32_t v) { return v ? 31 - __builtin_clz(v) : 0; }

__device__ __forceinline__ int wbid(uint64_t w) { return (int)(w >> 48); }
__device__ __forceinline__ uint64_t wval(uint64_t w) { return w & W48; }
__device__ __forceinline__ uint64_t wpack(uint64_t w, int bid) { return w | ((uint64_t)bid << 48); }

// what a lane of k_search does with the loads of an iteration: claim a read (no loads), a
// width step, evaluate a popped entry, expand (or prune, or start the exact tail of) an entry,
// one exact-tail step
enum : int { PH_CLAIM = 0, PH_CW = 1, PH_POP = 2, PH_EXP = 3, PH_EXACT = 4 };

// Free granules: NSHARD lock-free stacks, each with a head that carries a tag bumped on every
// change (no ABA), links read and written at device scope; then never-used granules. A
// workgroup uses the shard of its index, so contention on one head stays low.
constexpr int NSHARD = 64;

__device__ __forceinline__ uint32_t shard_pop(unsigned long long *head, uint32_t *gnext)
{
    for (;;) {
        unsigned long long old = __hip_atomic_load(head, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t g = (uint32_t)old;
        if (g == NIL) return NIL;
        const uint32_t nxt = __hip_atomic_load(gnext + g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned long long nw = ((old >> 32) + 1) << 32 | nxt;
        if (__hip_atomic_compare_exchange_strong(head, &old, nw, __ATOMIC_ACQ_REL, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT))
            return g;
    }
}

__device__ __forceinline__ uint32_t gran_pop(unsigned long long *ghead, uint32_t *gnext, uint32_t *gbump, uint32_t n_gran)
{
    const int sh = (int)(blockIdx.x & (NSHARD - 1));
    uint32_t g = shard_pop(ghead + sh, gnext);
    if (g != NIL) return g;
    if (__hip_atomic_load(gbump, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < n_gran) {
        const uint32_t b = atomicAdd(gbump, 1u);
        if (b < n_gran) return b;
    }
    // the never-used granules are gone: look in the other shards
    for (int t = 1; t < NSHARD && g == NIL; ++t) g = shard_pop(ghead + ((sh + t) & (NSHARD - 1)), gnext);
    return g;
}

// push the chain own[from..to) (linked through gnext) onto this workgroup's shard in one exchange
__device__ __forceinline__ void gran_push(unsigned long long *ghead, uint32_t *gnext, const uint32_t *own, int from,
                                          int to)
{
    unsigned long long *const head = ghead + (blockIdx.x & (NSHARD - 1));
    for (int j = from; j + 1 < to; ++j)
        __hip_atomic_store(gnext + own[j], own[j + 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t first = own[from], last = own[to - 1];
    unsigned long long old = __hip_atomic_load(head, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (;;) {
        __hip_atomic_store(gnext + last, (uint32_t)old, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned long long nw = ((old >> 32) + 1) << 32 | first;
        if (__hip_atomic_compare_exchange_strong(head, &old, nw, __ATOMIC_RELEASE, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT))
            return;
    }
}

template <bool TRACE, bool PERSIST>
__global__ void __launch_bounds__(128) k_search(KArgs a)
{
    using TopT = uint32_t;  // chunk id << 4 | fill - 1
    extern __shared__ __align__(16) uint8_t lds_raw[];
    const int slot = blockIdx.x * blockDim.x + threadIdx.x;
    if (slot >= a.n_slots) return;
    // arguments used once per read (claims, results, granules) are read from the kernel
    // argument segment where they are used, so they do not hold scalar registers for the loop
    const KArgsC *const A = (const KArgsC *)__builtin_amdgcn_kernarg_segment_ptr();
    TopT *const tops = reinterpret_cast<TopT *>(lds_raw) + threadIdx.x;
    const int tstride = blockDim.x;

    uint8_t *const base = a.scratch + (uint64_t)slot * a.slot_bytes;
    uint64_t *const W = reinterpret_cast<uint64_t *>(base);
    uint64_t *const SW = reinterpret_cast<uint64_t *>(base + a.sw_off);
    galn_aln_rec_t *const REC = reinterpret_cast<galn_aln_rec_t *>(base + a.rec_off);
    uint32_t *const OWN = reinterpret_cast<uint32_t *>(base + a.own_off);
    uint32_t *const LINK = a.pool_link;
    Ent *const CHK = a.pool_chk;
    const DMeta &M = a.meta;
    const uint64_t seq_len = M.seq_len;

    // ---- lane state ----
    int rid = 0, len = 0;
    const uint8_t *q = nullptr;
    int s_mm = 0, s_gapo = 0, s_gape = 0, mode = 0, ies = 0, mdo = 0, max_entries = 0, max_gapo = 0, max_gape = 0,
        msd = 0, max_top2 = 0, n_stacks = 0, md_read = 0, seed_len = 0;
    bool seeding = false;
    // widths in progress: position cj of `pstr` (the query, or its seed part), interval [ck, cl]
    int cj = 0, plen = 0, cbid = 0, cbase = 0, nN = 0;
    const uint8_t *pstr = nullptr;
    uint64_t *wout = nullptr;
    bool in_seed = false;
    uint64_t ck = 0, cl = 0;
    // search
    int best_score = 0, best_diff = 0, max_diff = 0, best_cnt = 0, n_aln = 0, n_entries = 0;
    uint64_t bm0 = 0, bm1 = 0, bm2 = 0, bm3 = 0;
    Ent cur{0, 0}, e{0, 0}, pf{0, 0};
    bool has_cur = false, pf_valid = false;
    int cur_score = 0, e_score = 0, m = 0, m_seed = 0;
    uint32_t pf_addr = NIL, ld_ntop = NIL;  // prefetched entry; lowest top after a pop being loaded
    uint64_t hk = 0, hl = 0;  // a hit waiting to be applied
    uint32_t spare = NIL, free_head = NIL;
    int n_own = 0, own_next = 0, gleft = 0;  // granules held, next one to use, chunks left in it
    uint32_t gbase = 0;
    uint64_t pops = 0, trace = TR_INIT, obytes = 0, wbytes = 0;  // wbytes: of the widths
    // what the next iteration loads, and what it then does
    int phase = PH_CLAIM;
    bool rq_lf = false, rq_ent = false, rq_pf = false, rq_w = false;
    uint64_t qa = 0, qb = 0;
    uint32_t ent_addr = 0;
    const uint8_t *c1p = nullptr, *c2p = nullptr;  // query bytes to load (null: none)
    bool claimed = false;

    // ---- helpers (all lane-local) ----
    auto bm_test = [&](int s) __attribute__((always_inline)) -> bool {
        const uint64_t w = s < 64 ? bm0 : s < 128 ? bm1 : s < 192 ? bm2 : bm3;
        return (w >> (s & 63)) & 1ull;
    };
    auto bm_set = [&](int s) __attribute__((always_inline)) {
        const uint64_t bit = 1ull << (s & 63);
        const int w = s >> 6;
        bm0 |= w == 0 ? bit : 0ull;
        bm1 |= w == 1 ? bit : 0ull;
        bm2 |= w == 2 ? bit : 0ull;
        bm3 |= w == 3 ? bit : 0ull;
    };
    auto bm_clear = [&](int s) __attribute__((always_inline)) {
        const uint64_t bit = ~(1ull << (s & 63));
        const int w = s >> 6;
        bm0 &= w == 0 ? bit : ~0ull;
        bm1 &= w == 1 ? bit : ~0ull;
        bm2 &= w == 2 ? bit : ~0ull;
        bm3 &= w == 3 ? bit : ~0ull;
    };
    auto bm_any = [&]() __attribute__((always_inline)) -> bool { return (bm0 | bm1 | bm2 | bm3) != 0; };
    auto bm_low = [&]() __attribute__((always_inline)) -> int {
        return bm0 ? __builtin_ctzll(bm0)
                   : bm1 ? 64 + __builtin_ctzll(bm1) : bm2 ? 128 + __builtin_ctzll(bm2) : 192 + __builtin_ctzll(bm3);
    };
    auto chunk_alloc = [&]() __attribute__((always_inline)) -> uint32_t {
        uint32_t c;
        if (spare != NIL) {
            c = spare;
            spare = NIL;
        } else if (free_head != NIL) {
            c = free_head;
            free_head = LINK[c];
        } else if (gleft > 0) {
            c = gbase + (uint32_t)(GRAN - gleft);
            --gleft;
        } else {
            uint32_t g;
            if (own_next < n_own) {
                g = OWN[own_next];
            } else {
                if (n_own >= CA(own_cap)) return NIL;
                g = gran_pop(CA(ghead), CA(gnext), CA(gbump), CA(n_gran));
                if (g == NIL) return NIL;
                OWN[n_own++] = g;
            }
            ++own_next;
            gbase = g * GRAN;
            gleft = GRAN - 1;
            c = gbase;
        }
        return c;
    };
    auto chunk_free = [&](uint32_t c) __attribute__((always_inline)) {
        if (spare == NIL) {
            spare = c;
        } else {
            LINK[c] = free_head;
            free_head = c;
        }
    };
    // gap_push into the arena: src/bwtgap_hd.h:264-286
    auto push_mem = [&](int s, const Ent &en) __attribute__((always_inline)) -> int {
        if (s < 0 || s >= n_stacks) return ERR_SCORE;
        TopT *tp = tops + s * tstride;
        uint32_t chunk, idx;
        if (bm_test(s)) {
            const uint32_t t = *tp;
            chunk = t >> 4;
            idx = (t & 15u) + 1;
            if (idx == CH) {
                const uint32_t nc = chunk_alloc();
                if (nc == NIL) return ERR_STACK;
                LINK[nc] = chunk;
                chunk = nc;
                idx = 0;
            }
        } else {
            const uint32_t nc = chunk_alloc();
            if (nc == NIL) return ERR_STACK;
            LINK[nc] = NIL;
            chunk = nc;
            idx = 0;
            bm_set(s);
        }
        *tp = (TopT)(chunk << 4 | idx);
        CHK[(uint64_t)chunk * CH + idx] = en;
        ++n_entries;
        return 0;
    };
    auto score_of = [&](int mm, int go, int ge) __attribute__((always_inline)) -> int { return mm * s_mm + go * s_gapo + ge * s_gape; };
    // n (<= 16) consecutive pushes into bucket s: the first n1 go to chunk c0 from slot s0,
    // the rest to chunk c1 from slot 0; the bucket's top moves to the last
    auto reserve = [&](int s, int n, uint32_t &c0, uint32_t &s0, uint32_t &n1, uint32_t &c1)
        __attribute__((always_inline)) -> int {
        if (s < 0 || s >= n_stacks) return ERR_SCORE;
        TopT *tp = tops + s * tstride;
        if (bm_test(s)) {
            const uint32_t t = *tp;
            c0 = t >> 4;
            s0 = (t & 15u) + 1;
        } else {
            const uint32_t nc = chunk_alloc();
            if (nc == NIL) return ERR_STACK;
            LINK[nc] = NIL;
            c0 = nc;
            s0 = 0;
            bm_set(s);
        }
        n1 = min((uint32_t)n, (uint32_t)CH - s0);
        if ((uint32_t)n > n1) {
            const uint32_t nc = chunk_alloc();
            if (nc == NIL) return ERR_STACK;
            LINK[nc] = c0;
            c1 = nc;
            *tp = (TopT)(nc << 4 | ((uint32_t)n - n1 - 1));
        } else {
            c1 = NIL;
            *tp = (TopT)(c0 << 4 | (s0 + n1 - 1));
        }
        n_entries += n;
        return 0;
    };

    // result of the current read; the lane then claims the next one
    auto finish = [&](int code) __attribute__((always_inline)) {
        int n = code;
        if (n == ERR_HEAVY) {
            const int h = atomicAdd(CA(heavy_n), 1);
            CA(heavy_list)[h] = rid;
            if (h < CA(hand_cap)) {
                // the widths go along while no hit has changed them (gap_shadow only runs with a
                // new record); the wave engine then skips computing them again
                uint64_t *const dst = CA(hand) + (uint64_t)h * CA(hand_stride);
                if (n_aln == 0) {
                    for (int j = 0; j <= len; ++j) dst[1 + j] = W[j];
                    if (seeding)
                        for (int j = 0; j <= seed_len; ++j) dst[2 + len + j] = SW[j];
                    dst[CA(hand_stride) - 1] = 0;  // (the seed's bytes are among them)
                    dst[0] = wbytes | (3ull << 62);
                } else {
                    dst[0] = 0;
                }
            }
        } else {
            if (n > 0) {
                const unsigned long long b0 = atomicAdd(CA(out_top), (unsigned long long)n);
                if (b0 + (unsigned long long)n > CA(out_cap)) {
                    n = ERR_OUT;
                } else {
                    for (int j = 0; j < n; ++j) CA(out_rec)[b0 + j] = REC[j];
                    CA(out_off)[rid] = b0;
                }
            }
            if (n == ERR_STACK || n == ERR_ALN || n == ERR_OUT) {
                const int f = atomicAdd(CA(fail_n), 1);
                CA(fail_list)[f] = rid;
                atomicOr(CA(fail_kind) + (n == ERR_OUT ? 0 : n == ERR_ALN ? 1 : 2), 1);
            }
            CA(out_n)[rid] = n;
            CA(out_pops)[rid] = pops;
            if (TRACE) CA(out_trace)[rid] = trace;
            if (CA(out_bytes)) CA(out_bytes)[rid] = obytes;
            if (n != ERR_STACK && n != ERR_ALN && n != ERR_OUT) atomicAdd(CA(algo_bytes), (unsigned long long)obytes);
        }
        if (n_own > CA(keep)) {
            gran_push(CA(ghead), CA(gnext), OWN, CA(keep), n_own);
            n_own = CA(keep);
        }
        rq_lf = rq_ent = rq_pf = rq_w = false;
        c1p = c2p = nullptr;
        phase = PH_CLAIM;
    };

    // gap_shadow: src/bwtgap_hd.h:309-320 (widths read eight at a time)
    auto shadow = [&](int x, int ldp) __attribute__((always_inline)) {
        const uint64_t ux = (uint64_t)(int64_t)x;
        int j = 0;
        for (int i0 = 0; i0 < ldp; i0 += 8) {
            uint64_t wv[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) wv[t] = i0 + t < ldp ? W[i0 + t] : 0;
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                if (i0 + t >= ldp) break;
                uint64_t w = wval(wv[t]);
                int bid = wbid(wv[t]);
                if (w > ux) {
                    w -= ux;
                } else if (w == ux) {
                    bid = 1;
                    w = seq_len - (uint64_t)(++j);
                } else {
                    continue;
                }
                W[i0 + t] = wpack(w, bid);
            }
        }
    };

    // a hit (src/bwtgap_hd.h:385-409): NOFIN, or the code the read finishes with
    auto hit = [&](uint64_t k, uint64_t l) __attribute__((always_inline)) -> int {
        const int mm = e_mm(e), go = e_go(e), ge = e_ge(e);
        const int score = e_score;
        bool do_add = true;
        if (n_aln == 0) {
            best_score = score;
            best_diff = mm + go;
            if (mode & MODE_GAPE) best_diff += ge;
            if (!(mode & MODE_NONSTOP)) max_diff = (best_diff + 1 > md_read) ? md_read : best_diff + 1;
        }
        if (score == best_score) {
            best_cnt = (int)(uint32_t)((uint64_t)(int64_t)best_cnt + (l - k + 1));
        } else if (best_cnt > max_top2) {
            return n_aln;
        }
        if (go) {
            for (int j = 0; j < n_aln; ++j)
                if (REC[j].k == k && REC[j].l == l) {
                    do_add = false;
                    break;
                }
        }
        if (do_add) {
            shadow((int)(uint32_t)(l - k + 1), e_ldp(e));
            if (n_aln == CA(rec_cap)) return ERR_ALN;
            const int ins = e_ins(e), del = go + ge - ins;
            galn_aln_rec_t r;
            r.packed = ((uint64_t)(mm & 0xff)) | ((uint64_t)(go & 0xff) << 8) | ((uint64_t)(ge & 0xff) << 16) |
                       ((uint64_t)(score & 0xfffff) << 24) | ((uint64_t)(ins & 0x3ff) << 44) |
                       ((uint64_t)(del & 0x3ff) << 54);
            r.k = k;
            r.l = l;
            REC[n_aln] = r;
            ++n_aln;
        }
        return NOFIN;
    };

    // The top of bwt_match_gap's loop (src/bwtgap_hd.h:357-383): pop entries until one needs
    // an LF lookup (its loads are requested for the next iteration: NOFIN), an entry has to be
    // loaded first (NOFIN), a popped entry is a hit (HITP, at (hk, hl)), or the search ends
    // (the finish code). have_e: `e` was just loaded and not yet evaluated.
    auto pop_loop = [&](bool have_e) __attribute__((always_inline)) -> int {
        uint32_t ntop = NIL;      // the lowest bucket's top after the last pop from memory
        bool popped_mem = have_e;  // ntop is known
        if (have_e) ntop = ld_ntop;
        for (;;) {
            if (!have_e) {
                if (n_entries == 0 || n_entries > max_entries) return n_aln;
                if (has_cur) {
                    e = cur;
                    e_score = cur_score;
                    has_cur = false;
                    popped_mem = false;
                } else {
                    popped_mem = true;
                    if (!bm_any()) return ERR_INTERNAL;  // entries counted but none held: never expected
                    const int s = bm_low();
                    TopT *tp = tops + s * tstride;
                    const uint32_t t = *tp;
                    const uint32_t chunk = t >> 4, idx = t & 15u;
                    // the bucket's new top: the lowest bucket's top unless the bucket empties
                    if (idx > 0) {
                        ntop = t - 1;
                        *tp = (TopT)ntop;
                    } else {
                        const uint32_t p = LINK[chunk];
                        chunk_free(chunk);  // its entries stay readable until a later push
                        if (p != NIL) {
                            ntop = p << 4 | (CH - 1);
                            *tp = (TopT)ntop;
                        } else {
                            bm_clear(s);
                            ntop = bm_any() ? tops[bm_low() * tstride] : NIL;
                        }
                    }
                    e_score = s;
                    if (pf_valid && pf_addr == t) {
                        e = pf;
                        pf_valid = false;
                    } else {
                        ent_addr = t;
                        rq_ent = true;
                        ld_ntop = ntop;
                        phase = PH_POP;
                        // and the entry now on top of the lowest bucket
                        if (ntop != NIL && (!pf_valid || pf_addr != ntop)) {
                            pf_addr = ntop;
                            pf_valid = false;
                            rq_pf = true;
                        }
                        return NOFIN;
                    }
                }
            }
            have_e = false;
            --n_entries;
            ++pops;
            if (a.pop_budget && pops > a.pop_budget) return ERR_HEAVY;
            const int i0 = e_i(e), mm = e_mm(e), go = e_go(e), ge = e_ge(e), st = e_st(e);
            if (TRACE) {
                const int ins = e_ins(e), del = go + ge - ins;
                trace = tr_mix(trace, (uint64_t)((uint32_t)e_score << 21 | (uint32_t)i0));
                trace = tr_mix(trace, e_k(e));
                trace = tr_mix(trace, e_l(e));
                trace = tr_mix(trace, (uint64_t)((uint32_t)mm | (uint32_t)go << 8 | (uint32_t)ge << 16 | (uint32_t)st << 24));
                trace = tr_mix(trace, (uint64_t)ins | (uint64_t)del << 16);
                trace = tr_mix(trace, (uint64_t)(uint32_t)e_ldp(e));
                trace = tr_mix(trace, (uint64_t)(uint32_t)n_entries);
            }
            if (!(mode & MODE_NONSTOP) && (uint32_t)e_score > (uint32_t)(best_score + s_mm)) return n_aln;
            m = max_diff - (mm + go);
            if (mode & MODE_GAPE) m -= ge;
            if (m < 0) continue;
            if (seeding) {
                m_seed = msd - (mm + go);
                if (mode & MODE_GAPE) m_seed -= ge;
            }
            if (i0 == 0) {
                hk = e_k(e);
                hl = e_l(e);
                return HITP;
            }
            // the occurrence query of (k, l), whether the entry expands or starts an exact tail,
            // with the widths and the query bytes it needs
            qa = e_k(e);
            qb = e_l(e);
            rq_lf = true;
            rq_w = true;
            c1p = q + (i0 - 1);
            c2p = i0 >= 2 ? q + (i0 - 2) : nullptr;
            phase = PH_EXP;
            // and the entry on top of the lowest bucket, usually the next pop (after a pop from
            // memory ntop is that entry; after the exact child in registers it is unchanged)
            if (!popped_mem && bm_any()) ntop = tops[bm_low() * tstride];
            if (ntop != NIL && (!pf_valid || pf_addr != ntop)) {
                pf_addr = ntop;
                pf_valid = false;
                rq_pf = true;
            }
            return NOFIN;
        }
    };

    auto start_search = [&]() __attribute__((always_inline)) -> int {
        wbytes = obytes;
        best_score = score_of(md_read + 1, max_gapo + 1, max_gape + 1);
        best_diff = md_read + 1;
        max_diff = md_read;
        best_cnt = 0;
        n_aln = 0;
        pops = 0;
        trace = TR_INIT;
        bm0 = bm1 = bm2 = bm3 = 0;
        n_entries = 0;
        spare = free_head = NIL;
        own_next = 0;
        gleft = 0;
        has_cur = false;
        pf_valid = false;
        if (nN > md_read) return 0;
        if (n_stacks <= 0) return ERR_SCORE;
        // root: (i = len, k = 0, l = seq_len), score 0
        const Ent root = mk_ent(0, seq_len, len, 0, 0, 0, 0, 0, ST_M);
        if (a.fuse) {
            cur = root;
            cur_score = 0;
            has_cur = true;
            ++n_entries;
            return NOFIN;
        }
        const int r = push_mem(0, root);
        return r ? r : NOFIN;
    };

    // widths (bwt_cal_width, src/bwtgap_hd.h:216-242): consume the query byte `c0` of position
    // cj, loaded by the previous iteration; request the next LF lookup or byte (NOFIN), or,
    // when the widths are done, set the search up (STARTS: pop next; or a finish code)
    auto width_char = [&](int c0) __attribute__((always_inline)) -> int {
        for (;;) {
            if (cj == plen) {
                wout[plen] = wpack(0, ++cbid);
                if (!in_seed && seeding) {
                    in_seed = true;
                    pstr = q + (len - seed_len);
                    plen = seed_len;
                    wout = SW;
                    cj = 0;
                    ck = 0;
                    cl = seq_len;
                    cbid = 0;
                    if (plen == 0) continue;
                    c1p = pstr;
                    return NOFIN;
                }
                const int r = start_search();
                return r == NOFIN ? STARTS : r;
            }
            if (!in_seed) nN += c0 > 3;
            if (c0 <= 3) {
                cbase = 3 - c0;
                qa = ck;
                qb = cl;
                rq_lf = true;
                c1p = cj + 1 < plen ? pstr + (cj + 1) : nullptr;
                return NOFIN;
            }
            // N: restart without a lookup
            ck = 0;
            cl = seq_len;
            ++cbid;
            wout[cj] = wpack(seq_len + 1, cbid);
            ++cj;
            if (cj < plen) {
                c1p = pstr + cj;
                return NOFIN;
            }
            c0 = 4;
        }
    };

    auto init_read = [&](int pos) __attribute__((always_inline)) -> int {
        rid = CA(list) ? CA(list)[pos] : CA(list_base) + pos;
        len = CA(qlen)[rid];
        q = CA(query) + CA(qoff)[rid];
        const int b = CA(batch)[rid];
        const galn_search_opt_t o = CA(bopts)[b];
        s_mm = o.s_mm;
        s_gapo = o.s_gapo;
        s_gape = o.s_gape;
        mode = o.mode;
        ies = o.indel_end_skip;
        mdo = o.max_del_occ;
        max_entries = o.max_entries;
        max_gapo = o.max_gapo;
        max_gape = o.max_gape;
        msd = o.max_seed_diff;
        max_top2 = o.max_top2;
        n_stacks = CA(nstacks)[b];
        md_read = CA(maxdiff)[rid];
        seed_len = o.seed_len;
        seeding = seed_len < len;
        pops = 0;
        trace = TR_INIT;
        obytes = 0;
        pf_valid = false;
        if (len < 1 || len > MAXLEN || n_stacks > MAXB || md_read > MAXDIFF || max_gapo > MAXDIFF ||
            max_gapo + max_gape > 255 || max_gape < 0)
            return ERR_UNSUP;
        in_seed = false;
        pstr = q;
        plen = len;
        wout = W;
        cj = 0;
        ck = 0;
        cl = seq_len;
        cbid = 0;
        nN = 0;
        c1p = q;
        phase = PH_CW;
        return NOFIN;
    };

    // ---- main loop: every iteration loads what the lane asked for, then works on it ----
    for (;;) {
        int fin = NOFIN;
        if (phase == PH_CLAIM) {
            int pos;
            if (PERSIST) {
                pos = atomicAdd(CA(qnext), 1);
            } else {
                if (claimed) break;
                pos = slot;
            }
            claimed = true;
            if (pos >= CA(n_list)) break;
            fin = init_read(pos);
        } else {
            // ---- loads, all issued before any is used ----
            uint64_t wA = 0, wB = 0, sA = 0, sB = 0;
            int ch1 = 4, ch2 = 4;
            Ent ld{0, 0};
            uint64_t ca[4] = {0, 0, 0, 0}, cb[4] = {0, 0, 0, 0};
            uint32_t lf_bytes = 0;
            if (rq_w) {
                const int wi = e_i(e);
                wB = W[wi - 1];
                if (wi >= 2) wA = W[wi - 2];
                if (seeding) {
                    const int ii = wi - 1 - (len - seed_len);
                    if (ii > 0) {
                        sA = SW[ii - 1];
                        sB = SW[ii];
                    }
                }
            }
            if (c1p) ch1 = *c1p;
            if (c2p) ch2 = *c2p;
            if (rq_ent) ld = CHK[(uint64_t)(ent_addr >> 4) * CH + (ent_addr & 15u)];
            if (rq_pf) pf = CHK[(uint64_t)(pf_addr >> 4) * CH + (pf_addr & 15u)];
            if (rq_lf) lf_bytes = lf_pair(a.bwt, M, qa, qb, ca, cb);
            if (rq_pf) pf_valid = true;
            const bool had_lf = rq_lf;
            rq_lf = rq_ent = rq_pf = rq_w = false;
            c1p = c2p = nullptr;

            // ---- work: each phase ends in new loads, a hit and/or a pop, or a finish ----
            bool want_pop = false, have_e = false, want_hit = false;
            if (phase == PH_CW) {
                if (had_lf) {
                    obytes += lf_bytes;
                    const int c = cbase;
                    uint64_t k = pick4(ca, c) + 1, l = pick4(cb, c);
                    if (k > l) {
                        k = 0;
                        l = seq_len;
                        ++cbid;
                    }
                    wout[cj] = wpack(l - k + 1, cbid);
                    ck = k;
                    cl = l;
                    ++cj;
                }
                const int r = width_char(ch1);
                if (r == STARTS)
                    want_pop = true;
                else
                    fin = r;
            } else if (phase == PH_POP) {
                e = ld;
                want_pop = have_e = true;
            } else if (phase == PH_EXACT) {
                // one step of an exact tail (bwt_match_exact_alt, src/bwtgap_hd.h:201-208)
                obytes += lf_bytes;
                const int c = cbase;
                const uint64_t k = pick4(ca, c) + 1, l = pick4(cb, c);
                want_pop = true;
                if (k <= l) {
                    if (cj == 0) {
                        want_hit = (int)(uint32_t)(l - k + 1) != 0;
                        hk = k;
                        hl = l;
                    } else if (ch1 <= 3) {
                        --cj;
                        cbase = ch1;
                        qa = k;
                        qb = l;
                        rq_lf = true;
                        c1p = cj >= 1 ? q + (cj - 1) : nullptr;
                        want_pop = false;
                    }
                }
            } else {
                // PH_EXP: the popped entry's lookup, widths and query bytes are here
                const int i0 = e_i(e);
                const int st = e_st(e), ge = e_ge(e);
                const int qbase = ch1;
                want_pop = true;
                if (m < wbid(wB)) {
                    // pruned by the widths
                } else if (m == 0 && (st == ST_M || (mode & MODE_GAPE) || ge == max_gape)) {
                    // exact tail: its first step is this lookup
                    if (qbase <= 3) {
                        obytes += lf_bytes;
                        const uint64_t k = pick4(ca, qbase) + 1, l = pick4(cb, qbase);
                        if (k <= l) {
                            if (i0 < 2) {
                                want_hit = (int)(uint32_t)(l - k + 1) != 0;
                                hk = k;
                                hl = l;
                            } else if (ch2 <= 3) {
                                cj = i0 - 2;
                                cbase = ch2;
                                qa = k;
                                qb = l;
                                rq_lf = true;
                                c1p = cj >= 1 ? q + (cj - 1) : nullptr;
                                phase = PH_EXACT;
                                want_pop = false;
                            }
                        }
                    }
                } else {
                    // expansion: src/bwtgap_hd.h:412-470
                    obytes += lf_bytes;
                    const int i = i0 - 1;
                    const int mm = e_mm(e), go = e_go(e), ins = e_ins(e);
                    const uint64_t k = e_k(e), l = e_l(e), occ = l - k + 1;
                    bool allow_diff = true, allow_M = true;
                    if (i > 0) {
                        if (wbid(wA) > m - 1)
                            allow_diff = false;
                        else if (wbid(wA) == m - 1 && wbid(wB) == m - 1 && wval(wA) == wval(wB))
                            allow_M = false;
                        if (seeding) {
                            const int ii = i - (len - seed_len);
                            if (ii > 0) {
                                if (wbid(sA) > m_seed - 1)
                                    allow_diff = false;
                                else if (wbid(sA) == m_seed - 1 && wbid(sB) == m_seed - 1 && wval(sA) == wval(sB))
                                    allow_M = false;
                            }
                        }
                    }
                    const int tmp = (mode & MODE_LOGGAP) ? int_log2((uint32_t)(ge + go)) / 2 + 1 : go + ge;
                    const bool gap_ok = allow_diff && i >= ies + tmp && len - i >= ies + tmp;
                    // the children, in the order bwt_match_gap pushes them:
                    // bit 0 insertion, bits 1-4 deletions (bases 0..3), bits 5-8 the bases
                    // qbase+1 .. qbase+4 (the last one is the exact child), bit 9 the exact child
                    // alone (when differences are not allowed here)
                    // the children's intervals are [ca + 1, cb] per base
                    uint32_t mask = 0;
                    if (gap_ok) {
                        const bool open = st == ST_M && go < max_gapo;
                        if (open || (st == ST_I && ge < max_gape)) mask |= 1u;
                        if (open || (st == ST_D && ge < max_gape && (ge + go < max_diff || occ < (uint64_t)(int64_t)mdo))) {
    #pragma unroll
                            for (int j = 0; j < 4; ++j)
                                if (ca[j] < cb[j]) mask |= 2u << j;
                        }
                    }
                    if (allow_diff && allow_M) {
    #pragma unroll
                        for (int j = 1; j <= 4; ++j) {
                            const int c = (qbase + j) & 3;
                            if (pick4(ca, c) < pick4(cb, c)) mask |= 16u << j;
                        }
                    } else if (qbase < 4 && pick4(ca, qbase) < pick4(cb, qbase)) {
                        mask |= 512u;
                    }
                    // Pushes, in bwt_match_gap's order: the gap children (bits 0-4) all score sg
                    // and the mismatches sm, so each group takes consecutive slots of one bucket
                    // (two groups with one score share it, gap children first); the exact child
                    // (bit 8 with qbase <= 3, or bit 9) comes last with the parent's score.
                    const uint32_t xbit = (qbase <= 3 ? 256u : 0u) | 512u;
                    const uint32_t mx = mask & xbit;
                    const uint32_t mg = mask & 31u, mmk = mask & 0x1e0u & ~xbit;
                    const int sg = st == ST_M ? score_of(mm, go + 1, ge) : score_of(mm, go, ge + 1);
                    const int sm = score_of(mm + 1, go, ge);
                    const int ng = __builtin_popcount(mg), nm = __builtin_popcount(mmk);
                    const bool merged = ng > 0 && nm > 0 && sg == sm;
                    uint32_t gc0 = 0, gs0 = 0, gn1 = 0, gc1 = 0, mc0 = 0, ms0 = 0, mn1 = 0, mc1 = 0;
                    int err = 0;
                    if (ng + (merged ? nm : 0) > 0) err = reserve(sg, ng + (merged ? nm : 0), gc0, gs0, gn1, gc1);
                    if (!err && nm > 0 && !merged) err = reserve(sm, nm, mc0, ms0, mn1, mc1);
                    if (!err) {
                        uint32_t rest = mg | mmk;
                        int rg = 0, rm = merged ? ng : 0;
                        while (rest) {
                            const int bit = __builtin_ctz(rest);
                            rest &= rest - 1;
                            Ent ch;
                            int r;
                            bool in_g = bit <= 4 || merged;
                            if (bit == 0) {
                                const int go2 = st == ST_M ? go + 1 : go, ge2 = st == ST_M ? ge : ge + 1;
                                ch = mk_ent(k, l, i, i, mm, go2, ge2, ins + 1, ST_I);
                            } else if (bit <= 4) {
                                const int j = bit - 1;
                                const uint64_t kk = pick4(ca, j) + 1, ll = pick4(cb, j);
                                const int go2 = st == ST_M ? go + 1 : go, ge2 = st == ST_M ? ge : ge + 1;
                                ch = mk_ent(kk, ll, i + 1, i + 1, mm, go2, ge2, ins, ST_D);
                            } else {
                                const int c = (qbase + bit - 4) & 3;
                                const uint64_t kk = pick4(ca, c) + 1, ll = pick4(cb, c);
                                ch = mk_ent(kk, ll, i, i, mm + 1, go, ge, ins, ST_M);
                            }
                            if (bit <= 4)
                                r = rg++;
                            else
                                r = rm++;
                            const uint32_t c0 = in_g ? gc0 : mc0, s0 = in_g ? gs0 : ms0, n1 = in_g ? gn1 : mn1,
                                           c1 = in_g ? gc1 : mc1;
                            const uint32_t slot_ = (uint32_t)r < n1 ? c0 * CH + s0 + (uint32_t)r : c1 * CH + ((uint32_t)r - n1);
                            CHK[slot_] = ch;
                        }
                        if (mx) {
                            const uint64_t kk = pick4(ca, qbase) + 1, ll = pick4(cb, qbase);  // (qbase <= 3 here)
                            const Ent ch = mk_ent(kk, ll, i, 0, mm, go, ge, ins, ST_M);
                            if (a.fuse) {
                                // pushed last with the parent's score: the next pop; kept in registers
                                cur = ch;
                                cur_score = e_score;
                                has_cur = true;
                                ++n_entries;
                            } else {
                                uint32_t c0, s0, n1, c1;
                                err = reserve(e_score, 1, c0, s0, n1, c1);
                                if (!err) CHK[n1 ? c0 * CH + s0 : c1 * CH] = ch;
                            }
                        }
                    }
                    if (err) {
                        fin = err;
                        want_pop = false;
                    }
                }
            }
            // ---- hits and pops, until new loads are requested or the read finishes ----
            for (;;) {
                if (want_hit) {
                    want_hit = false;
                    const int h = hit(hk, hl);
                    if (h != NOFIN) {
                        fin = h;
                        break;
                    }
                }
                if (!want_pop) break;
                const int r = pop_loop(have_e);
                have_e = false;
                if (r == HITP) {
                    want_hit = true;
                    continue;
                }
                fin = r;
                break;
            }
        }
        if (fin != NOFIN) finish(fin);
    }
}

// ---------------------------------------------------------------------------
// SA value of BWT rows (bwt_sa with bwt_invPsi, upstream bwt.c:53-59, :88-96): LF steps from each
// row to the nearest row divisible by the sample interval (fewer than intv steps, one 64-byte block
// each), then that row's sample plus the steps. Row 0, the $ row, counts as -1 as bwa sets it (a
// walk that ends there gives steps - 1). samples[j] is the suffix at row (j + 1) * intv; rows are
// at most seq_len (checked by the caller).
__global__ void __launch_bounds__(256) k_sa_walk(const uint32_t *__restrict__ bwt, DMeta m,
                                                  const uint64_t *__restrict__ samples, uint64_t intv,
                                                  const uint64_t *__restrict__ rows, uint64_t n, uint64_t *__restrict__ pos,
                                                  const int32_t *__restrict__ ref_len, int32_t *__restrict__ strand)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        uint64_t k = rows[i], sa = 0;
        while (k & (intv - 1)) {
            ++sa;
            if (k == m.primary) {
                k = 0;
                break;
            }
            // the row's symbol, the one after the first k - (k > primary) symbols, and its rank
            const uint64_t P = pos_k<uint64_t>(m, k);
            OccWord o;
            occ_load<uint64_t>(bwt, P, o);
            uint64_t cnt[4];
            occ_count<uint64_t>(m, m.ext != nullptr, o, P, cnt);
            const uint32_t sh = 31u - ((uint32_t)P & 31u);
            const int c = (int)(((o.h >> sh) & 1u) << 1 | ((o.l >> sh) & 1u));
            k = pick4(cnt, c) + 1;
        }
        uint64_t p = sa + (k == 0 ? ~0ull : samples[k / intv - 1]);
        if (ref_len) {
            // bwa_sa2pos (upstream bwase.c:112-123): a hit across the forward/reverse boundary is -1;
            // on the reverse half, the forward position of the hit's first base, strand 0
            const uint64_t l_pac = m.seq_len >> 1;
            const uint64_t rl = (uint64_t)(int64_t)ref_len[i];
            int st = 0;
            if (p < l_pac && l_pac < p + rl) {
                p = ~0ull;
            } else {
                const bool rev = p >= l_pac;
                if (rev) p = (l_pac << 1) - 1 - p;
                st = rev ? 0 : 1;
                if (rev) p = p + 1 < rl ? 0 : p - rl + 1;
            }
            strand[i] = st;
        }
        pos[i] = p;
    }
}

// ---------------------------------------------------------------------------
// Wave-per-read engine.
//
// Between two hits the search's state (max_diff, widths, best score) is fixed, and with positive
// penalties every non-exact child lands in a higher bucket than its parent. So the entries of the lowest
// bucket b each start an independent "chain" -- the entry, then its exact child, then that child's exact
// child, ... (the sequential search pops exactly this chain next, LIFO) -- whose pushes all go to buckets
// above b. A workgroup of NW waves takes up to CPL chains per thread from the top of bucket b, runs them
// (a thread takes the next chain when its own has ended), then commits them in the sequential order: pops,
// pushes (placed by scans so that every bucket keeps its LIFO order), removal of the heads, and the first
// hit, which changes the state and ends the commit. Chains after that hit are discarded and run again in
// the next round. The result, the pop count and the trace are those of the sequential search.
//
// A bucket is a LIFO list of granules of the stack pool, all full below the top one: entry 0 names the
// granule below, 1023 entries follow. A round's heads come from the top two granules, its pushes fill the
// top one up, and a granule that empties is the next one taken. (Buckets that took a piece of a shared
// granule each round gave a round only the last piece, 91 heads of up to 256 on average, and a read's
// memory grew with its pushes, not with its stack.)
//
// What bounds it: with few reads, the rounds of the longest ones, one after the other; with the chip full, memory
// past L2, 3.2 TB/s of the 4.9 that a copy reaches (10M ancient DNA reads, 1.22 s: 3.9 TB for 1.66 TB of index
// blocks, the vector units 28% busy; the one before, a chain a lane and round, was 70% busy and took 1.26 s). What
// took it from vector issue to there: a wave pays a full iteration while one lane has a lookup left, and the chains of a heavy read are 2.3 steps long on average,
// 5.5 the longest of 64: with one chain per lane and round 37% of the lane slots did work. Taking the next
// chain when one ends, pruning dead heads before the loop, tails as iterations of the same loop (a nested
// one held the wave for the longest tail of every step), 32-bit intervals and packed fields kept in
// registers below 2^32 symbols, and one log per bucket code (a placed push needs no ranks, ballots or score)
// took 2M ancient DNA reads on 100 Mbp from 308 ms of this kernel to 238, and 262,144 from 130 to 80.
//
// The tail: a read's rounds follow each other, and when the last read has been taken the waves that are done
// leave the ones still on a read of a million pops. Those reads are parked and gone on with by workgroups of
// four waves, whose round takes 1024 chains: 4001 reads, the longest of 630k pops, 41 -> 15 ms; 262,144
// reads 80 -> 44 ms.
//
// The log: a thread's own (1 KB a bucket code) touched up to 400 half-filled lines a round, 4.2e9 write
// requests past L2 for 2M reads; one log per wave in the order of the iterations is 16 bytes after 16 bytes
// and stays in L2. Its stores are issued after the next step's lookups, which a pop needs the exact child's
// interval for and nothing else. With choices written as arithmetic instead of branches (186 -> 142 scalar
// instructions an iteration) and the kernel's cold arguments read where they are used (373 -> 87 static
// readlanes of spilled scalars): 2M reads 225 -> 210 ms, 100k of 100 bp 7.75 -> 7.17, the 4001 15 -> 13,
// 100,003 reads of a 700 Mbp repeat-rich genome 142 -> 125.

constexpr int HW = 64;         // lanes of a wave
constexpr int H_STEPS = 60;    // chain steps per round
constexpr int H_STEPS_PLAIN = 32;  // and where lone descents are not walked ahead
constexpr int H_LOG = 8192;    // pushes logged per wave and round
constexpr int H_SPUSH = 9;     // pushes of one step at most
constexpr int H_CPUSH = 127;   // pushes of a chain and round to one bucket at most (7-bit ranks)
constexpr int H_SLOG = 64;    // trace build: steps logged per thread
constexpr int H_KEEP = 64;     // granules a workgroup keeps between reads
constexpr int H_PIECES = 48;   // segment pieces one round may add (three buckets)
constexpr int H_MINCAP = 128;  // the lowest push cap a test may set
constexpr uint32_t GENT = (uint32_t)GRAN * CH;  // entries per granule, its link included
constexpr uint32_t GFULL = GENT - 1;
constexpr int H_LOOK = 16;     // rounds between looks at the queue
constexpr int H_FREE = 32;     // emptied granules kept in LDS
static_assert(H_LOG > 2 * HW * H_SPUSH, "every lane of a wave can log a step's pushes");
static_assert(H_SLOG >= 2 * H_STEPS_PLAIN, "a chain's steps fit the rest of a thread's step log");

enum : int { K_END = 0, K_HIT = 1, K_TRUNC = 2, K_ESCORE = 3, K_TAIL = 4, K_DEAD = 5 };  // (the last two only while walking ahead)
constexpr int H_ALONE = 2;  // iterations with one lane at work after which it walks ahead

struct HArgs {
    const uint32_t *bwt;
    DMeta meta;
    const uint8_t *query;
    const uint64_t *qoff;
    const int32_t *qlen;
    const int32_t *maxdiff;
    const int32_t *batch;
    const galn_search_opt_t *bopts;
    const int32_t *nstacks;
    const int32_t *list;        // read ids by position, or null (the position)
    int32_t n_list;
    const int32_t *n_list_dev;  // when set, the number of reads is read here
    const uint64_t *hand;       // widths by position (k_search or k_widths), or null
    uint32_t hand_stride;
    int32_t hand_cap;
    int32_t *qnext;
    int32_t n_slots;
    uint8_t *scratch;
    uint64_t slot_bytes;
    uint32_t rec_off, own_off, spill_off, plog_off, slog_off;
    int32_t own_cap, rec_cap;
    Ent *pool;
    uint32_t *gnext;
    unsigned long long *ghead;
    uint32_t *gbump;
    uint32_t n_gran;
    int32_t first_gran;         // granules each workgroup holds from the start (gbump begins after them)
    int32_t *out_n;
    uint64_t *out_off, *out_pops, *out_trace, *out_bytes;
    galn_aln_rec_t *out_rec;
    uint64_t out_cap;
    unsigned long long *out_top;
    int32_t *fail_list, *fail_n, *fail_kind;
    unsigned long long *algo_bytes;
    int32_t buckets;  // LDS buckets: the largest n_stacks of the launch
    int32_t wlen;     // LDS widths: longest read + 1
    int32_t swlen;    // LDS seed widths
    int32_t push_cap; // pushes committed per round (more than the logs hold unless a test lowers it)
    // a read that is still running when no other is left to take, after park_pops pops (0: never), is parked:
    // its workgroup writes its state to its scratch, lists itself in park_list and ends; a launch of
    // workgroups of more waves goes on with it
    uint32_t park_pops;
    int32_t *park_list, *park_n;
    uint32_t state_off;
    uint8_t *park_scratch;          // that launch's: the scratch of the launch that parked, its layout
    uint64_t park_slot_bytes;
    uint32_t park_rec_off, park_own_off, park_spill_off, park_state_off;
    unsigned long long *stats;  // [16] engine counters (rounds, chains, steps, cycles)
};

struct HShared {
    int rid, len, n_stacks, md_read, seeding, seed_len;
    int s_mm, s_gapo, s_gape, mode, ies, mdo, max_entries, max_gapo, max_gape, msd, max_top2;
    int best_score, best_diff, max_diff, best_cnt, n_aln, n_entries;
    unsigned long long pops, trace, obytes;
    unsigned long long bm[4];
    int has_pend, claim, status, result, K, b, n_piece, n_own, n_used, n_free, n_spill, nN, bad;
    int root, root_unused;  // steps of the root chain known beyond the root, until the first round's commit
    uint32_t own[H_KEEP], free_g[H_FREE];  // the first granules held; emptied ones (more of them in the spill list)
    int next, stop, lim, l_kind, cut;  // the round's claims, first stopping chain, commit limit
    uint32_t tot01, tot2s, totb;       // committed pushes (16 bits per bucket code), pops, index bytes / 64
    int fp[3];                         // first piece of each bucket code
    uint32_t wsum[3][16];              // per wave: scan totals
    int wlive[16];
    uint64_t hk, hl;                   // the last committed chain's hit, or its pending child
    uint32_t hx, hy;
    struct {                           // per wave, a descent walked ahead: the entry after its steps, their number,
        uint64_t k, l;                 // how it ended, and the chain's pops, index bytes / 64 and pushes before it
        uint32_t n, end, steps, sby, np3, unused;
    } ahead[4];
};
static_assert(sizeof(HShared) % 8 == 0, "the widths follow it in a parked read's state");

// what a read's state is besides HShared: the widths, the buckets
__host__ __device__ constexpr size_t heavy_state_bytes(int buckets, int wlen, int swlen)
{
    return sizeof(HShared) + (size_t)(wlen + swlen + 2) * 8 + (size_t)buckets * 12;
}

__device__ __forceinline__ int hbm_low(const unsigned long long *bm)
{
    return bm[0] ? __builtin_ctzll(bm[0]) : bm[1] ? 64 + __builtin_ctzll(bm[1]) : bm[2] ? 128 + __builtin_ctzll(bm[2])
                 : bm[3] ? 192 + __builtin_ctzll(bm[3]) : -1;
}

// lanes below this one that are set in m
__device__ __forceinline__ int lanes_below(uint64_t m)
{
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// inclusive sum over a wave's lanes in six row moves (no LDS); every lane of the wave must call it
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x)
{
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false);  // row_shr:1
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false);  // row_shr:2
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false);  // row_shr:4
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false);  // row_shr:8
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false);  // row_bcast:15
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return x;
}

template <class K>
__device__ __forceinline__ K lane_value(K v, int lane)
{
    if constexpr (sizeof(K) == 8)
        return (K)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), lane) << 32 | (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, lane);
    else
        return (K)__builtin_amdgcn_readlane((int)v, lane);
}

// A stack entry in registers: the interval, x = i | n_mm << 10 | n_gapo << 17 | state << 24 and
// y = last_diff_pos | n_gape << 10 | n_ins << 18. In memory an index of 2^32 symbols or more packs k and x
// into one 64-bit word, l and y into the other (the layout above); a smaller one stores the four words.
template <bool WIDE>
struct Item {
    using K = typename std::conditional<WIDE, uint64_t, uint32_t>::type;
    K k, l;
    uint32_t x, y;
};
constexpr uint32_t X_I = 1023u, X_MM = 1u << 10, X_GO = 1u << 17, X_ST = 3u << 24, X_INS = 1u << 24, X_DEL = 2u << 24;
constexpr uint32_t Y_LDP = 1023u, Y_GE = 1u << 10, Y_IN = 1u << 18;
__device__ __forceinline__ int x_mm(uint32_t x) { return (int)((x >> 10) & 127u); }
__device__ __forceinline__ int x_go(uint32_t x) { return (int)((x >> 17) & 127u); }
__device__ __forceinline__ int x_st(uint32_t x) { return (int)((x >> 24) & 3u); }
__device__ __forceinline__ int y_ge(uint32_t y) { return (int)((y >> 10) & 255u); }
__device__ __forceinline__ int y_ins(uint32_t y) { return (int)((y >> 18) & 255u); }

template <bool WIDE>
__device__ __forceinline__ void put_item(Ent *p, typename Item<WIDE>::K k, typename Item<WIDE>::K l, uint32_t x, uint32_t y)
{
    if constexpr (WIDE) {
        Ent e;
        e.w0 = (uint64_t)k | (uint64_t)x << 38;
        e.w1 = (uint64_t)l | (uint64_t)y << 38;
        *p = e;
    } else {
        *reinterpret_cast<uint4 *>(p) = make_uint4((uint32_t)k, (uint32_t)l, x, y);
    }
}

template <bool WIDE>
__device__ __forceinline__ Item<WIDE> get_item(const Ent *p)
{
    Item<WIDE> r;
    if constexpr (WIDE) {
        const Ent e = *p;
        r.k = e.w0 & KMASK;
        r.l = e.w1 & KMASK;
        r.x = (uint32_t)(e.w0 >> 38);
        r.y = (uint32_t)(e.w1 >> 38);
    } else {
        const uint4 v = *reinterpret_cast<const uint4 *>(p);
        r.k = v.x;
        r.l = v.y;
        r.x = v.z;
        r.y = v.w;
    }
    return r;
}

// a popped entry's share of the trace hash
__device__ __forceinline__ uint64_t trace_item(uint64_t t, int score, uint64_t k, uint64_t l, uint32_t x, uint32_t y, int n_entries)
{
    const int mm = x_mm(x), go = x_go(x), ge = y_ge(y), st = x_st(x), ins = y_ins(y);
    t = tr_mix(t, (uint64_t)((uint32_t)score << 21 | (x & X_I)));
    t = tr_mix(t, k);
    t = tr_mix(t, l);
    t = tr_mix(t, (uint64_t)((uint32_t)mm | (uint32_t)go << 8 | (uint32_t)ge << 16 | (uint32_t)st << 24));
    t = tr_mix(t, (uint64_t)ins | (uint64_t)(go + ge - ins) << 16);
    t = tr_mix(t, (uint64_t)(y & Y_LDP));
    return tr_mix(t, (uint64_t)(uint32_t)n_entries);
}

// widths in LDS: the value in the low part, the bound above it (32 bits each below 2^32 symbols, so that
// neither needs a shift; the 48 | 16 of the hand-off slots otherwise). A sentinel before position 0 bounds
// nothing, so that the first positions need no case of their own.
constexpr uint32_t NO_BOUND = 0xffffb000u;  // a bound below any number of differences, also as 16 bits
template <bool WIDE>
__device__ __forceinline__ int lw_bid(uint64_t v) { return WIDE ? (int)((int64_t)v >> 48) : (int)(v >> 32); }
template <bool WIDE>
__device__ __forceinline__ uint64_t lw_val(uint64_t v) { return WIDE ? v & W48 : v & 0xffffffffull; }
template <bool WIDE>
__device__ __forceinline__ uint64_t lw_make(uint64_t w, uint32_t bid) { return w | (uint64_t)bid << (WIDE ? 48 : 32); }

// bwt_cal_width by one thread (src/bwtgap_hd.h:216-242); returns the algorithmic bytes. put(i, w, bid)
// stores position i's width.
template <class K, class Put>
__device__ __forceinline__ uint64_t cal_width_one(const uint32_t *bwt, const DMeta &M, int len, const uint8_t *str, Put put)
{
    K k = 0, l = (K)M.seq_len;
    uint32_t units = 0;
    int bid = 0;
    for (int i = 0; i < len; ++i) {
        const int c0 = str[i];
        if (c0 <= 3) {
            const K Pk = pos_k<K>(M, k), Pl = pos_l<K>(M, l);
            OccWord A, B;
            occ_load<K>(bwt, Pk, A);
            occ_load<K>(bwt, Pl, B);
            K ca[4], cb[4];
            occ_count<K>(M, sizeof(K) == 8, A, Pk, ca);
            occ_count<K>(M, sizeof(K) == 8, B, Pl, cb);
            units += occ_units<K>(Pk, Pl);
            k = pick4(ca, 3 - c0) + 1;
            l = pick4(cb, 3 - c0);
        }
        if (k > l || c0 > 3) {
            k = 0;
            l = (K)M.seq_len;
            ++bid;
        }
        put(i, (uint64_t)l - k + 1, bid);
    }
    put(len, 0, ++bid);
    return (uint64_t)units << 6;
}

// Widths and root chains of the reads given to the wave engine, into their hand-off slots (those that k_search
// has filled keep their widths): three threads per read, one for the read's widths, one for its seed's and one
// for the intervals of its exact descent, each a walk of as many dependent lookups as it has positions, all
// reads at once, so that the wave engine does not hold 64 lanes while one of them walks. A slot:
// [bytes | flags][W[0..len]][SW[0..seed_len]] ... [root steps 1 ..][their number][bytes of the seed's].
// The descent from the root is a read's first chain and, for a read of a few hundred pops, four fifths of its
// iterations with one lane at work: with its intervals known, the engine's first round has a lane for each of
// its steps (100k reads of 100 bp 7.2 -> 4.9 ms, this kernel 0.47 -> 0.72).
struct WArgs {
    const uint32_t *bwt;
    DMeta meta;
    const uint8_t *query;
    const uint64_t *qoff;
    const int32_t *qlen;
    const int32_t *batch;
    const galn_search_opt_t *bopts;
    const int32_t *list;
    int32_t n_list;
    const int32_t *n_list_dev;
    uint64_t *hand;
    uint32_t hand_stride;
    int32_t hand_cap;
    int32_t wlen, swlen;
    int32_t root;   // steps of a root chain that a slot has room for (0: none)
    int32_t check;  // slots may hold widths already
};
constexpr int H_ROOT = 127;  // steps of the root chain kept at most (one round's chains with the root itself)
// Only of reads of this length on: a shorter descent saves little, and its pushes come all at once (2M ancient
// DNA reads, median 45, 240 ms with all of them, 228 with those from 90 on, 224 with none).
constexpr int H_ROOT_MIN = 90;
constexpr uint64_t HAND_OK = 1ull << 63, HAND_SEARCH = 1ull << 62;  // a slot's flags: filled; by k_search

template <bool WIDE>
__global__ void __launch_bounds__(256) k_widths(WArgs a)
{
    using K = typename Item<WIDE>::K;
    const int n = min(a.n_list_dev ? *a.n_list_dev : a.n_list, a.hand_cap);
    // a wave's threads do the same work for 64 reads (three walks in one wave follow each other)
    const int64_t span = ((int64_t)n + HW - 1) / HW * HW;
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < (WIDE ? 2 : 3) * span; t += (int64_t)gridDim.x * blockDim.x) {
        const int role = t < span ? 0 : t < 2 * span ? 1 : 2;
        const int pos = (int)(t - role * span);
        if (pos >= n) continue;
        uint64_t *const dst = a.hand + (uint64_t)pos * a.hand_stride;
        if (role < 2 && a.check && (dst[0] & HAND_SEARCH)) continue;
        const int rid = a.list ? a.list[pos] : pos;
        const int len = a.qlen[rid];
        const int sl = a.bopts[a.batch[rid]].seed_len;
        // (a read the wave engine rejects, or a seed it has no room for: no widths)
        const bool none = len < 1 || len + 1 > a.wlen || (sl < len && sl + 1 > a.swlen);
        const uint8_t *const q = a.query + a.qoff[rid];
        if (role == 0) {
            uint64_t *const w = dst + 1;
            dst[0] = none ? 0 : cal_width_one<K>(a.bwt, a.meta, len, q, [w](int i, uint64_t v, int bid) { w[i] = wpack(v, bid); }) | HAND_OK;
        } else if (role == 1) {
            if (none || sl >= len) continue;
            uint64_t *const w = dst + 2 + len;
            dst[a.hand_stride - 1] = cal_width_one<K>(a.bwt, a.meta, sl, q + (len - sl), [w](int i, uint64_t v, int bid) { w[i] = wpack(v, bid); });
        } else if constexpr (!WIDE) {
            uint64_t *const at = dst + 1 + a.wlen + a.swlen;
            const int most = none || len < H_ROOT_MIN ? 0 : min(len, a.root);
            uint32_t k = 0, l = (uint32_t)a.meta.seq_len;
            int s = 0;
            while (s < most) {
                const int c = q[len - 1 - s];
                if (c > 3) break;
                const uint32_t Pk = pos_k<uint32_t>(a.meta, k), Pl = pos_l<uint32_t>(a.meta, l);
                OccWord A, B;
                occ_load<uint32_t>(a.bwt, Pk, A);
                occ_load<uint32_t>(a.bwt, Pl, B);
                uint32_t ca[4], cb[4];
                occ_count<uint32_t>(a.meta, false, A, Pk, ca);
                occ_count<uint32_t>(a.meta, false, B, Pl, cb);
                k = pick4(ca, c) + 1;
                l = pick4(cb, c);
                if (k > l) break;
                at[s] = (uint64_t)l << 32 | k;
                ++s;
            }
            dst[a.hand_stride - 2] = (uint64_t)s;
        }
    }
}

// steps of the root chain that a hand-off slot of reads of up to max_len bases has room for
inline int hand_root(int max_len, bool wide) { return wide || max_len < H_ROOT_MIN ? 0 : std::min(max_len, H_ROOT); }

// words of a hand-off slot
inline uint32_t hand_words(int wlen, int swlen, int root) { return (uint32_t)(1 + wlen + swlen + root + 2); }

// A wave logs a round's pushes in the order it makes them, 16 bytes after 16 bytes. A logged push holds, beside
// the entry, its chain, its rank among the chain's pushes to its bucket and the bucket's code, so that it can
// be placed by itself. A pushed entry's last_diff_pos is its position i (every push is a difference there), so
// its ten bits are free: rank in y[0:7), and below 2^32 symbols code in x[26:28), chain in y[26:32) and
// x[28:32); a larger index keeps code and chain in a word per push after the log.
constexpr int H_CHAIN_BITS = 10;
constexpr size_t heavy_log_bytes(bool wide) { return (size_t)H_LOG * (sizeof(Ent) + (wide ? 4 : 0)); }

// LDS of a workgroup of nw waves, cpl chains per thread (k_heavy carves it up in this order)
constexpr size_t heavy_chain_bytes = 16 + 4 + 4 + 2 + 2;  // head | counts | steps | id | trace place

typedef const __attribute__((address_space(4))) HArgs HArgsC;
#define HA(f) cold_ld(&((HArgsC *)__builtin_amdgcn_kernarg_segment_ptr())->f)

// NW waves per read, at four waves per SIMD (128 VGPRs): a variant of five (96) was 4% faster on light reads, 2%
// slower on heavy ones, before the light reads' descents were taken out of the loop. (The upper bound changes the
// schedule only, not the registers or scratch bytes of any variant; the traced ones and those above 2^32 symbols
// keep the compiler's own, 8, with which their code does not change as the others' bound does.)
template <bool TRACE, bool WIDE, int NW, int CPL>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(4, (TRACE || WIDE) ? 8 : 4))) k_heavy(HArgs a)
{
    using K = typename Item<WIDE>::K;
    constexpr int T = 64 * NW, KMAX = T * CPL;
    static_assert(NW > 1 || H_ROOT < KMAX, "the root's round");
    static_assert(KMAX <= 1 << H_CHAIN_BITS, "a chain's id in its pushes");
    extern __shared__ __align__(16) uint8_t hlds[];
    // the launch of NW > 1 waves goes on with reads that the launch of one wave parked
    constexpr bool RESUME = NW > 1;
    // Steps of exact descents side by side (the root's round, a lone lane's descent): not in the trace build, whose
    // step log has no place for steps that are walked ahead, and not above 2^32 symbols, where hand-off slots have
    // no room for a root chain. Two other builds with this in it were wrong, for a reason that is not known: the
    // traced one above 2^32 symbols read out of range, and one for five waves per SIMD (96 registers) gave records
    // that changed from run to run. What is known: the same source gives the right results lane by lane on the CPU
    // with unwritten memory and registers poisoned and the lanes and waves in any order between two wave operations;
    // and both of those builds keep state of the round in scratch memory, stored from several branches of its loops,
    // while the two kernels that have this code now store to scratch memory in their prologue only, with every
    // lane on (tests/test_device_code.py holds them to that).
    constexpr bool AHEAD = !TRACE && !WIDE;
    static_assert(!AHEAD || (!TRACE && !WIDE), "no step log, no root chain");
    constexpr int STEPS = AHEAD ? H_STEPS : H_STEPS_PLAIN;
    uint4 *const pieces = reinterpret_cast<uint4 *>(hlds);         // {bucket code, rank0, len, base}
    Ent *const hent = reinterpret_cast<Ent *>(pieces + H_PIECES);  // live chains' heads, in order
    uint16_t *const epre = reinterpret_cast<uint16_t *>(hent);     // after them: pushes before each chain, by code
    uint32_t *const cA = reinterpret_cast<uint32_t *>(hent + KMAX);  // pushes by code (8 bits each) | stop kind << 24
    uint32_t *const cC = cA + KMAX;                                  // steps | index bytes / 64 << 6
    uint16_t *const hcid = reinterpret_cast<uint16_t *>(cC + KMAX);  // live chains' ids
    uint16_t *const cS = hcid + KMAX;                                // trace build: place in the step logs
    unsigned long long *const ST = reinterpret_cast<unsigned long long *>(cS + KMAX);  // [16] counters
    HShared &F = *reinterpret_cast<HShared *>(ST + 16);
    uint64_t *const Wp = reinterpret_cast<uint64_t *>(&F + 1);       // Wp[i] = width of position i - 1
    uint64_t *const SW = Wp + HA(wlen) + 1;                          // SW[i] = seed width of position i - 1
    uint32_t *const seg_top = reinterpret_cast<uint32_t *>(SW + HA(swlen) + 1);  // per bucket: its top granule,
    uint32_t *const seg_cnt = seg_top + HA(buckets);                         // that one's entries (0: empty bucket)
    uint32_t *const seg_prev = seg_cnt + HA(buckets);                        // and the granule below, or NIL
    uint16_t *const s0info = reinterpret_cast<uint16_t *>(seg_prev + HA(buckets));  // chain 0's steps: pushes | index bytes / 64 << 4
    uint8_t *const QL = reinterpret_cast<uint8_t *>(s0info + H_STEPS);           // the read's query
    static_assert(MAXLEN * 2 + 2 < 4096, "a step's index bytes fit the step info");

    const int tid = threadIdx.x, lane = tid & (HW - 1), wave = tid >> 6;
    if ((int)blockIdx.x >= HA(n_slots)) return;
    uint8_t *const base = HA(scratch) + (uint64_t)blockIdx.x * HA(slot_bytes);
    galn_aln_rec_t *REC = reinterpret_cast<galn_aln_rec_t *>(base + HA(rec_off));
    uint32_t *OWN = reinterpret_cast<uint32_t *>(base + HA(own_off));
    uint32_t *SPILL = reinterpret_cast<uint32_t *>(base + HA(spill_off));
    // this wave's pushes of the round (all waves' entries, then their words)
    Ent *const LOG = reinterpret_cast<Ent *>(base + HA(plog_off)) + wave * H_LOG;
    uint32_t *const LOGW = reinterpret_cast<uint32_t *>(reinterpret_cast<Ent *>(base + HA(plog_off)) + NW * H_LOG) + wave * H_LOG;
    Ent *const SLOG = reinterpret_cast<Ent *>(base + HA(slog_off));    // trace build: thread t's steps at t * H_SLOG
    uint8_t *const SINFO = reinterpret_cast<uint8_t *>(SLOG + T * H_SLOG);  // and their push counts
    Ent *const POOL = a.pool;
    const DMeta &M = a.meta;
    // (arguments not used in the lookups are read from the kernel argument segment where they are used: held
    // in scalar registers for the whole kernel they spilled, and a fifth of the vector instructions were
    // reads of spilled ones)
    const K seq_len = (K)M.seq_len;

    if (tid == 0) {
        for (int j = 0; j < 16; ++j) ST[j] = 0;
        F.n_own = RESUME ? 0 : HA(first_gran);  // granules this workgroup holds; a read reuses them before taking more
    }
    if (!RESUME && tid < HA(first_gran)) OWN[tid] = F.own[tid] = blockIdx.x * (uint32_t)HA(first_gran) + (uint32_t)tid;
    const int n_list = HA(n_list_dev) ? *HA(n_list_dev) : HA(n_list);
    const bool stats = HA(stats) != nullptr;
    const int state_words = (int)(heavy_state_bytes(HA(buckets), HA(wlen), HA(swlen)) / 4);
    for (;;) {
        const long long t_read = stats ? wall_clock64() : 0;
        if (tid == 0) F.claim = atomicAdd(HA(qnext), 1);
        __syncthreads();
        const int claim = F.claim;
        if (claim >= n_list) break;
        // ---- read set-up ----
        int rid, len;
        if constexpr (RESUME) {
            // a parked read: its state, and its records and granules where its workgroup kept them
            uint8_t *const pb = HA(park_scratch) + (uint64_t)HA(park_list)[claim] * HA(park_slot_bytes);
            const uint32_t *const st = reinterpret_cast<const uint32_t *>(pb + HA(park_state_off));
            __syncthreads();  // (F.claim is part of it)
            for (int j = tid; j < state_words; j += T)
                reinterpret_cast<uint32_t *>(&F)[j] = st[j];
            REC = reinterpret_cast<galn_aln_rec_t *>(pb + HA(park_rec_off));
            OWN = reinterpret_cast<uint32_t *>(pb + HA(park_own_off));
            SPILL = reinterpret_cast<uint32_t *>(pb + HA(park_spill_off));
            __syncthreads();
            rid = F.rid;
            len = F.len;
            const uint8_t *const qg = HA(query) + HA(qoff)[rid];
            for (int j = tid; j < len; j += T) QL[j] = qg[j];
            __syncthreads();
        } else {
            const int pos = claim;
            rid = HA(list) ? HA(list)[pos] : pos;
            len = HA(qlen)[rid];
            const uint8_t *const qg = HA(query) + HA(qoff)[rid];
            const int qn = min(len, HA(wlen));
            for (int j = tid; j < qn; j += T) QL[j] = qg[j];
            if (tid == 0) {
                const int b0 = HA(batch)[rid];
                const galn_search_opt_t o = HA(bopts)[b0];
                F.rid = rid;
                F.len = len;
                F.s_mm = o.s_mm;
                F.s_gapo = o.s_gapo;
                F.s_gape = o.s_gape;
                F.mode = o.mode;
                F.ies = o.indel_end_skip;
                F.mdo = o.max_del_occ;
                F.max_entries = o.max_entries;
                F.max_gapo = o.max_gapo;
                F.max_gape = o.max_gape;
                F.msd = o.max_seed_diff;
                F.max_top2 = o.max_top2;
                F.n_stacks = HA(nstacks)[b0];
                F.md_read = HA(maxdiff)[rid];
                F.seed_len = o.seed_len;
                F.seeding = o.seed_len < len;
                F.nN = 0;
                F.obytes = 0;
                F.n_used = 0;
                F.n_free = 0;
                F.n_spill = 0;
                F.status = 0;
                F.bad = 0;
                F.root = 0;
            }
            __syncthreads();
            const bool unsup = len < 1 || len > MAXLEN || len + 1 > HA(wlen) || F.n_stacks > HA(buckets) || F.md_read > MAXDIFF ||
                               F.max_gapo > MAXDIFF || F.max_gapo + F.max_gape > 255 || F.max_gape < 0;
            const uint64_t h0 = (!unsup && HA(hand) && pos < HA(hand_cap)) ? HA(hand)[(uint64_t)pos * HA(hand_stride)] : 0;
            if (!unsup) {
                if (h0 >> 63) {
                    // the widths computed for this read
                    const uint64_t *src = HA(hand) + (uint64_t)pos * HA(hand_stride);
                    for (int j = tid; j <= len; j += T) Wp[1 + j] = lw_make<WIDE>(wval(src[1 + j]), (uint32_t)wbid(src[1 + j]));
                    if (F.seeding)
                        for (int j = tid; j <= F.seed_len; j += T)
                            SW[1 + j] = lw_make<WIDE>(wval(src[2 + len + j]), (uint32_t)wbid(src[2 + len + j]));
                    if (tid == 0) {
                        F.obytes = (h0 & ~(HAND_OK | HAND_SEARCH)) + (F.seeding ? src[HA(hand_stride) - 1] : 0);
                        if (AHEAD) F.root = (int)src[HA(hand_stride) - 2];
                    }
                } else {
                    uint64_t wb = 0;
                    auto putw = [Wp](int i, uint64_t v, int bid) { Wp[1 + i] = lw_make<WIDE>(v, (uint32_t)bid); };
                    auto puts = [SW](int i, uint64_t v, int bid) { SW[1 + i] = lw_make<WIDE>(v, (uint32_t)bid); };
                    if (tid == 0) wb = cal_width_one<K>(a.bwt, M, len, QL, putw);
                    if (tid == 1 && F.seeding) wb = cal_width_one<K>(a.bwt, M, F.seed_len, QL + (len - F.seed_len), puts);
                    if (wb) atomicAdd(&F.obytes, (unsigned long long)wb);
                }
                int nN = 0;
                for (int j = tid; j < len; j += T) nN += QL[j] > 3;
                if (nN) atomicAdd(&F.nN, nN);
            }
            const int nbk = HA(buckets);
            for (int j = tid; j < nbk; j += T) seg_cnt[j] = 0;
            __syncthreads();
            // ---- search set-up ----
            if (tid == 0) {
                F.best_score = (F.md_read + 1) * F.s_mm + (F.max_gapo + 1) * F.s_gapo + (F.max_gape + 1) * F.s_gape;
                F.best_diff = F.md_read + 1;
                F.max_diff = F.md_read;
                F.best_cnt = 0;
                F.n_aln = 0;
                F.pops = 0;
                F.trace = TR_INIT;
                F.bm[0] = F.bm[1] = F.bm[2] = F.bm[3] = 0;
                F.has_pend = 0;
                F.n_entries = 0;
                Wp[0] = SW[0] = lw_make<WIDE>(0, NO_BOUND);
                if (unsup) {
                    F.status = 1;
                    F.result = ERR_UNSUP;
                } else if (F.nN > F.md_read) {
                    F.status = 1;
                    F.result = 0;
                } else if (F.n_stacks <= 0) {
                    F.status = 1;
                    F.result = ERR_SCORE;
                } else {
                    F.has_pend = 1;
                    F.hk = 0;
                    F.hl = M.seq_len;
                    F.hx = (uint32_t)len;
                    F.hy = 0;
                    F.b = 0;
                    F.n_entries = 1;
                }
                // (the widths' bounds fall towards the read's start: a root that is not dead has no dead step; with
                // no difference allowed the whole descent is one pop)
                if (AHEAD && (F.md_read <= 0 || F.status || F.md_read < lw_bid<WIDE>(Wp[len]))) F.root = 0;
            }
            __syncthreads();
        }
        if (stats && tid == 0) {
            ST[12] += (unsigned long long)(wall_clock64() - t_read);
            if (!RESUME) ST[15] += 1;
        }
        // ---- rounds ----
        int n_round = 0;
        long long t_round_end = 0;  // with stats: end of the last round's commit
        for (;;) {
            const long long t_round = stats ? wall_clock64() : 0;
            if (stats && tid == 0 && t_round_end) ST[14] += (unsigned long long)(t_round - t_round_end);
            int taken_reads = 0;
            if (tid == 0 && F.status == 0) {  // (the others read the status after the barrier)
                // reads taken so far, looked at when this round has been committed. One load in H_LOOK rounds:
                // all workgroups loading this word every round made a round 50% longer. With a workgroup for
                // every read each takes its own, whatever the others do.
                if (!RESUME && HA(park_pops) && F.pops >= HA(park_pops)) {
                    if (n_list <= HA(n_slots))
                        taken_reads = n_list;
                    else if ((++n_round & (H_LOOK - 1)) == 0)
                        taken_reads = __hip_atomic_load(HA(qnext), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                // a pending exact child is the top of the lowest bucket (the bucket it came from)
                const int b = F.has_pend ? F.b : hbm_low(F.bm);
                if (b < 0 || F.n_entries > F.max_entries) {
                    F.status = 1;
                    F.result = F.n_aln;
                } else {
                    F.b = b;
                    const uint32_t cb = seg_cnt[b];
                    const uint32_t avail = (uint32_t)F.has_pend + cb + (cb && seg_prev[b] != NIL ? GFULL : 0u);
                    if (!(F.mode & MODE_NONSTOP) && (uint32_t)b > (uint32_t)(F.best_score + F.s_mm)) {
                        // this pop ends the search (src/bwtgap_hd.h:366)
                        F.pops += 1;
                        F.n_entries -= 1;
                        if (TRACE) {
                            Item<WIDE> e;
                            if (F.has_pend) {
                                e.k = (K)F.hk;
                                e.l = (K)F.hl;
                                e.x = F.hx;
                                e.y = F.hy;
                            } else {
                                e = get_item<WIDE>(POOL + seg_top[b] * GENT + seg_cnt[b]);
                            }
                            F.trace = trace_item(F.trace, b, e.k, e.l, e.x, e.y, F.n_entries);
                        }
                        F.status = 1;
                        F.result = F.n_aln;
                    } else {
                        F.K = AHEAD && !RESUME && F.root ? F.root + 1 : (int)min(avail, (uint32_t)KMAX);
                        F.next = T;
                        F.stop = 0x7fffffff;
                        F.lim = 0x7fffffff;
                        F.l_kind = K_END;
                        F.cut = -1;
                    }
                }
            }
            __syncthreads();
            if (F.status) break;
            const int b = F.b, nK = F.K, hp = F.has_pend;
            // the first round: a chain for every known step of the root chain, of that one pop (the last one goes
            // on as any chain)
            const bool root = AHEAD && !RESUME && F.root != 0;
            const int solo = root ? nK - 1 : 0;
            const long long t_spec = stats ? wall_clock64() : 0;
            if (stats && tid == 0) ST[13] += (unsigned long long)(t_spec - t_round);
            const int s_mm = F.s_mm, s_gapo = F.s_gapo, s_gape = F.s_gape, mode = F.mode, max_diff = F.max_diff;
            const int n_stacks = F.n_stacks, max_gapo = F.max_gapo, max_gape = F.max_gape, ies = F.ies, mdo = F.mdo;
            const int msd = F.msd, sofs = len - F.seed_len;
            const bool seeding = F.seeding != 0;
            // the buckets that pushes go to and their log codes: 0 a mismatch, 1 a gap open, 2 a gap
            // extension, or the lower code of the same bucket (one log, so that its order is kept)
            const int tg0 = b + s_mm, tg1 = b + s_gapo, tg2 = b + s_gape;
            const int sh1 = s_gapo == s_mm ? 0 : 8, sh2 = s_gape == s_mm ? 0 : s_gape == s_gapo ? 8 : 16;
            auto root_step = [&](int c) __attribute__((always_inline)) {
                const uint64_t *const at = HA(hand) + (uint64_t)claim * HA(hand_stride) + 1 + HA(wlen) + HA(swlen) + (c - 1);
                Item<WIDE> e;
                e.k = (K)(uint32_t)at[0];
                e.l = (K)(at[0] >> 32);
                e.x = (uint32_t)(len - c);
                e.y = 0;
                return e;
            };
            // differences still allowed to a chain (constant along it)
            auto left = [&](int lim, uint32_t x, uint32_t y) __attribute__((always_inline)) {
                return lim - x_mm(x) - x_go(x) - ((mode & MODE_GAPE) ? y_ge(y) : 0);
            };
            // ---- chain heads, from the top of bucket b; those that cannot go on end here. Wave w loads
            // heads w * 64 * CPL on; the live ones are listed in order ----
            {
                const uint32_t tc = seg_cnt[b], tb = seg_top[b] * GENT, pb = seg_prev[b] * GENT;
                uint64_t lm[CPL];
                int cnt = 0;
                Item<WIDE> h[CPL];
#pragma unroll
                for (int r = 0; r < CPL; ++r) {
                    const int c = (wave * CPL + r) * HW + lane;
                    if (c < nK) {
                        if (c == 0 && hp) {
                            h[r].k = (K)F.hk;
                            h[r].l = (K)F.hl;
                            h[r].x = F.hx;
                            h[r].y = F.hy;
                        } else if (root) {
                            h[r] = root_step(c);
                        } else {
                            // entry d below the top one: in the top granule, or in the full one below it
                            const uint32_t d = (uint32_t)(c - hp);
                            h[r] = get_item<WIDE>(POOL + (d < tc ? tb + tc - d : pb + GFULL - (d - tc)));
                        }
                    }
                }
#pragma unroll
                for (int r = 0; r < CPL; ++r) {
                    const int c = (wave * CPL + r) * HW + lane;
                    bool live = c < nK;
                    if (!TRACE && live) {
                        const int m = left(max_diff, h[r].x, h[r].y);
                        const uint32_t i0 = h[r].x & X_I;
                        if (m < 0 || (i0 > 0 && m < lw_bid<WIDE>(Wp[i0]))) {
                            live = false;
                            cA[c] = 0;
                            cC[c] = 1;  // one pop, no lookup
                            if (c == 0) s0info[0] = 0;
                        }
                    }
                    lm[r] = __ballot(live);
                    cnt += __builtin_popcountll(lm[r]);
                }
                int at = 0;
                if (NW > 1) {
                    if (lane == 0) F.wlive[wave] = cnt;
                    __syncthreads();
                    for (int w = 0; w < wave; ++w) at += F.wlive[w];
                }
#pragma unroll
                for (int r = 0; r < CPL; ++r) {
                    const int c = (wave * CPL + r) * HW + lane;
                    if ((lm[r] >> lane) & 1ull) {
                        const int p = at + lanes_below(lm[r]);
                        put_item<WIDE>(hent + p, h[r].k, h[r].l, h[r].x, h[r].y);
                        hcid[p] = (uint16_t)c;
                    }
                    at += __builtin_popcountll(lm[r]);
                }
                if (NW == 1 && lane == 0) F.wlive[0] = cnt;
            }
            __syncthreads();
            int nlive = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) nlive += F.wlive[w];
            // ---- speculation: every thread runs chains, one lookup an iteration, and takes the next live
            // one when its own has ended. A step's children are logged while the next step's lookups are on
            // their way ----
            int next = T, stop = 0x7fffffff, its = 0, alone = 0;  // (NW > 1: the claims and the stop are F.next, F.stop)
            uint32_t wl = 0;                           // pushes this wave has logged
            uint64_t stopped = 0;                      // lanes whose chain has stopped
            bool more = true;                          // (uniform) chains are left to take
            // the chain: its pushes by bucket code (8 bits each), pops, index bytes / 64
            uint32_t np3 = 0, sby = 0;
            int cid = -1, kind = K_END, steps = 0, m = 0, m_seed = 0, so = 0, sl = 0;
            bool busy = false, tail = false;
            K k = 0, l = 0;
            uint32_t x = 0, y = 0;
            // children not yet logged: bit 0 an insertion, bits 1-4 deletions by base, bits 5-8 mismatches in
            // their order, bits 9-10 the query's base, bit 11 the gap is opened; their chain, its pushes before
            // them, and what they are made of
            uint32_t ch = 0, p_np3, p_x, p_y;
            int p_cid;
            K pk, pl, ca[4], cb[4];
            constexpr uint32_t ROOM = 0x010101u * (uint32_t)(127 - (H_CPUSH - H_SPUSH));  // sets bit 7 of a full count
            constexpr uint32_t LOG_FULL = H_LOG - 2 * HW * H_SPUSH;
            const bool near = F.n_entries + STEPS * H_SPUSH > F.max_entries;  // chain 0 may cross the limit
            auto finish = [&]() __attribute__((always_inline)) {
                cA[cid] = np3 | (uint32_t)kind << 24;
                cC[cid] = (uint32_t)steps | sby << 6;
                if (TRACE) cS[cid] = (uint16_t)(tid * H_SLOG + so);
                if (NW > 1 && kind != K_END) atomicMin(&F.stop, cid);
                busy = false;
            };
            // pop the entry in k, l, x, y (w: the width of the position before its own): it dies, is a hit, or
            // needs a lookup (src/bwtgap_hd.h:369-396)
            auto pop = [&](uint64_t w) __attribute__((always_inline)) {
                if (TRACE) {
                    put_item<WIDE>(SLOG + tid * H_SLOG + sl, k, l, x, y);
                    SINFO[tid * H_SLOG + sl] = 0;
                    ++sl;
                }
                if (near && cid == 0) s0info[steps] = 0;
                ++steps;
                tail = m == 0 && ((x & X_ST) == 0 || (mode & MODE_GAPE) || y_ge(y) == max_gape);
                const bool dead = m < max(lw_bid<WIDE>(w), 0);
                if (dead || (x & X_I) == 0) {
                    kind = dead ? K_END : K_HIT;
                    finish();
                }
            };
            auto take = [&](int p) __attribute__((always_inline)) {
                const Item<WIDE> e = get_item<WIDE>(hent + p);
                cid = hcid[p];
                k = e.k;
                l = e.l;
                x = e.x;
                y = e.y;
                m = left(max_diff, x, y);
                m_seed = left(msd, x, y);
                steps = 0;
                sby = 0;
                np3 = 0;
                so = sl;
                busy = true;
                pop(Wp[x & X_I]);
            };
            if (tid < nlive) take(tid);
            for (;;) {
                if (more) {
                    const uint64_t wm = __ballot(!busy && kind == K_END && (!TRACE || sl <= H_SLOG - STEPS));
                    if (wm) {
                        int g;
                        if (NW == 1) {
                            g = next;
                            next += __builtin_popcountll(wm);
                            more = next < nlive;
                        } else {
                            g = 0;
                            if (lane == 0) {
                                if (__hip_atomic_load(&F.stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) == 0x7fffffff)
                                    g = atomicAdd(&F.next, __builtin_popcountll(wm));
                                else
                                    g = nlive;
                            }
                            g = __builtin_amdgcn_readlane(g, 0);
                            more = g + __builtin_popcountll(wm) < nlive;
                        }
                        const int p = g + lanes_below(wm);
                        if ((wm >> lane & 1ull) && p < nlive) take(p);
                    }
                }
                uint64_t run_m = __ballot(busy);
                // ---- one lane is left: its exact descent is walked ahead by the wave (a lookup and little more
                // per step), then each of its steps gets a lane of its own in one iteration. With the root's round
                // two thirds of a light read's iterations still had one lane (13 a round of 95 pops; 8
                // now), and a round takes 60 steps of a chain instead of 32: 100k reads of 100 bp 4.9 -> 4.1 ms, 100k pairs of 150 bp
                // 43 -> 34, 100,003 repeat-rich reads 118 -> 105 ----
                bool fan = false;
                if (AHEAD && !more && !near && run_m != 0 && (run_m & (run_m - 1)) == 0 && wl <= LOG_FULL && __ballot(kind != K_END) == 0) {
                    const int L = __builtin_ctzll(run_m);
                    const int wcid = __builtin_amdgcn_readlane(cid, L);
                    if (++alone >= H_ALONE && wcid >= solo) {
                        const bool wtail = (__ballot(tail) >> L & 1ull) != 0;
                        const uint32_t wx = (uint32_t)__builtin_amdgcn_readlane((int)x, L), wy = (uint32_t)__builtin_amdgcn_readlane((int)y, L);
                        const int wm = __builtin_amdgcn_readlane(m, L), ws = __builtin_amdgcn_readlane(steps, L);
                        K wk = lane_value<K>(k, L), wl_ = lane_value<K>(l, L);
                        uint32_t i = wx & X_I, units = 0;
                        int n = 0, end = K_END;
                        for (;;) {
                            if (!wtail && lane == n) {
                                k = wk;
                                l = wl_;
                            }
                            const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)QL[i - 1], 0);
                            ++n;
                            if (c > 3) break;
                            const K Pk = pos_k<K>(M, wk), Pl = pos_l<K>(M, wl_), P = (lane & 1) ? Pl : Pk;
                            OccWord o;
                            occ_load<K>(a.bwt, P, o);
                            K cn[4];
                            occ_count<K>(M, WIDE, o, P, cn);
                            const K v = pick4(cn, (int)c);
                            const K xk = lane_value<K>(v, 0) + 1, xl = lane_value<K>(v, 1);
                            units += occ_units<K>(Pk, Pl);
                            if (xk > xl) break;
                            wk = xk;
                            wl_ = xl;
                            --i;
                            if (wtail) {
                                if (i > 0) continue;
                                if ((uint32_t)(xl - xk + 1) != 0) end = K_HIT;
                                break;
                            }
                            if (ws + n - 1 == STEPS) {
                                end = K_TRUNC;
                                break;
                            }
                            const bool dead = wm < max(__builtin_amdgcn_readlane(lw_bid<WIDE>(Wp[i]), 0), 0);
                            if (dead || i == 0 || wm == 0) {
                                end = dead ? K_DEAD : i == 0 ? K_HIT : K_TAIL;
                                break;
                            }
                        }
                        if (wtail) {
                            if (busy) {
                                sby += units;
                                if (end == K_HIT) {
                                    kind = K_HIT;
                                    k = wk;
                                    l = wl_;
                                }
                                finish();
                            }
                            run_m = 0;
                        } else {
                            if (busy) {
                                F.ahead[wave].k = wk;
                                F.ahead[wave].l = wl_;
                                F.ahead[wave].n = (uint32_t)n;
                                F.ahead[wave].end = (uint32_t)end;
                                F.ahead[wave].steps = (uint32_t)steps;
                                F.ahead[wave].sby = sby;
                                F.ahead[wave].np3 = np3;
                            }
                            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // (all lanes read it below)
                            m_seed = __builtin_amdgcn_readlane(m_seed, L);
                            m = wm;
                            cid = wcid;
                            x = lane ? (wx & ~X_ST) - (uint32_t)lane : wx;
                            y = lane ? wy & ~Y_LDP : wy;
                            np3 = 0;
                            sby = 0;
                            tail = false;
                            busy = lane < n;
                            fan = true;
                        }
                    }
                }
                uint32_t qb = 0, i0 = 0;
                uint64_t wA = 0, wB = 0;
                K Pk = 0, Pl = 0;
                OccWord A, B;
                if (busy) {
                    i0 = x & X_I;
                    Pk = pos_k<K>(M, k);
                    Pl = pos_l<K>(M, l);
                    occ_load<K>(a.bwt, Pk, A);
                    occ_load<K>(a.bwt, Pl, B);
                    qb = QL[i0 - 1];
                    wA = Wp[i0 - 1];
                    wB = Wp[i0];
                }
                // ---- the last step's children to the log, each lane's after those of the lanes before it ----
                if (__ballot((ch & 511u) != 0)) {
                    const uint32_t nch = __builtin_popcount(ch & 511u);
                    const uint32_t incl = wave_incl_scan(nch);
                    if (nch) {
                        uint32_t at = wl + incl - nch;
                        const uint32_t tag_x = (uint32_t)p_cid >> 6 << 28, tag_y = (uint32_t)p_cid << 26;
                        auto put = [&](K ck, K cl, uint32_t cx, uint32_t cy, uint32_t code, uint32_t rank) __attribute__((always_inline)) {
                            if constexpr (WIDE) {
                                put_item<WIDE>(LOG + at, ck, cl, cx, cy | rank);
                                LOGW[at] = (uint32_t)p_cid | code << H_CHAIN_BITS;
                            } else {
                                put_item<WIDE>(LOG + at, ck, cl, cx, cy + rank);
                            }
                            ++at;
                        };
                        if (ch & 31u) {
                            const bool open = (ch >> 11 & 1u) != 0;
                            const uint32_t sh = open ? (uint32_t)sh1 : (uint32_t)sh2, code = sh >> 3;
                            uint32_t xg = p_x + (open ? X_GO : 0u), yg = p_y + (open ? 0u : Y_GE), rank = (p_np3 >> sh) & 127u;
                            if (!WIDE) {
                                xg |= code << 26 | tag_x;
                                yg |= tag_y;
                            }
                            if (ch & 1u) put(pk, pl, (xg - 1) | X_INS, yg + Y_IN, code, rank++);
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                if (ch >> (1 + j) & 1u) put(ca[j] + 1, cb[j], xg | X_DEL, yg, code, rank++);
                            p_np3 += (uint32_t)__builtin_popcount(ch & 31u) << sh;
                        }
                        if (ch >> 5 & 15u) {
                            // slot t of the rotated intervals holds base (query base + t) & 3, the mismatches' order
                            const bool r1 = (ch >> 9 & 1u) != 0, r2 = (ch >> 10 & 1u) != 0;
                            const K k0 = r1 ? ca[1] : ca[0], k1 = r1 ? ca[2] : ca[1], k2 = r1 ? ca[3] : ca[2], k3 = r1 ? ca[0] : ca[3];
                            const K l0 = r1 ? cb[1] : cb[0], l1 = r1 ? cb[2] : cb[1], l2 = r1 ? cb[3] : cb[2], l3 = r1 ? cb[0] : cb[3];
                            uint32_t rank = p_np3 & 127u, xm = p_x - 1 + X_MM, ym = p_y;
                            if (!WIDE) {
                                xm |= tag_x;
                                ym |= tag_y;
                            }
                            if (ch & 32u) put((r2 ? k3 : k1) + 1, r2 ? l3 : l1, xm, ym, 0u, rank++);
                            if (ch & 64u) put((r2 ? k0 : k2) + 1, r2 ? l0 : l2, xm, ym, 0u, rank++);
                            if (ch & 128u) put((r2 ? k1 : k3) + 1, r2 ? l1 : l3, xm, ym, 0u, rank++);
                            if (ch & 256u) put((r2 ? k2 : k0) + 1, r2 ? l2 : l0, xm, ym, 0u, rank++);
                        }
                        ch = 0;
                    }
                    wl += (uint32_t)__builtin_amdgcn_readlane((int)incl, HW - 1);
                    if (wl > LOG_FULL) more = false;
                }
                if (!run_m) break;
                ++its;
                if (busy) {
                    const uint32_t units = occ_units<K>(Pk, Pl);
                    occ_count<K>(M, WIDE, A, Pk, ca);
                    occ_count<K>(M, WIDE, B, Pl, cb);
                    const bool at0 = near && cid == 0;
                    // the exact child's interval
                    const K xk = pick4(ca, (int)qb) + 1, xl = pick4(cb, (int)qb);
                    const bool ex = qb <= 3 && xk <= xl;
                    if (tail) {
                        // exact tail: bwt_match_exact_alt, src/bwtgap_hd.h:195-211
                        if (qb <= 3) {
                            sby += units;
                            if (at0) s0info[steps - 1] += (uint16_t)(units << 4);
                        }
                        if (ex && i0 > 1) {
                            k = xk;
                            l = xl;
                            x -= 1;
                        } else {
                            if (ex && (uint32_t)(xl - xk + 1) != 0) {
                                kind = K_HIT;
                                k = xk;
                                l = xl;
                            }
                            finish();
                        }
                    } else {
                        // expansion: src/bwtgap_hd.h:412-470. The widths before position 0 (and before the seed)
                        // bound nothing.
                        sby += units;
                        const int i = (int)i0 - 1, ge = y_ge(y), go = x_go(x);
                        const int bA = lw_bid<WIDE>(wA);
                        bool allow_diff = bA < m;
                        bool allow_M = !(bA == m - 1 && wA == wB);
                        if (seeding) {
                            const uint64_t *const s = SW + max(i - sofs, 0);
                            const uint64_t sA = s[0], sB = s[1];
                            const int bS = lw_bid<WIDE>(sA);
                            allow_diff = allow_diff && bS < m_seed;
                            allow_M = allow_M && !(bS == m_seed - 1 && sA == sB);
                        }
                        const uint32_t st = x & X_ST;
                        const bool open = st == 0;
                        // bases that occur, and in the mismatches' order: bit t base (qb + t) & 3
                        const uint32_t e4 = (ca[0] < cb[0] ? 1u : 0u) | (ca[1] < cb[1] ? 2u : 0u) | (ca[2] < cb[2] ? 4u : 0u) |
                                            (ca[3] < cb[3] ? 8u : 0u);
                        const uint32_t rot = (e4 * 17u) >> (qb & 3u);
                        // gap children: opened by an entry that ends in a match, or extended
                        const int tmp = (mode & MODE_LOGGAP) ? int_log2((uint32_t)(ge + go)) / 2 + 1 : go + ge;
                        const bool gap = allow_diff && min(i, len - i) >= ies + tmp && (open ? go < max_gapo : ge < max_gape);
                        const bool del = st != X_INS && (open || ge + go < max_diff || (uint64_t)(K)(l - k + 1) < (uint64_t)(int64_t)mdo);
                        ch = gap ? (st != X_DEL ? 1u : 0u) | (del ? e4 << 1 : 0u) : 0u;
                        const int tg = open ? tg1 : tg2;
                        if (ch && (tg < 0 || tg >= n_stacks)) {
                            kind = K_ESCORE;
                            ch = 0;
                        } else if (allow_diff && allow_M) {
                            // mismatches, all four bases at an N
                            const uint32_t mm = (rot >> 1 & 7u) | (qb > 3 ? (rot & 1u) << 3 : 0u);
                            if (mm && (tg0 < 0 || tg0 >= n_stacks))
                                kind = K_ESCORE;
                            else
                                ch |= mm << 5;
                        }
                        p_np3 = np3;
                        p_x = x & ~X_ST;
                        p_y = y & ~Y_LDP;
                        p_cid = cid;
                        pk = k;
                        pl = l;
                        np3 += (uint32_t)__builtin_popcount(ch & 31u) << (open ? sh1 : sh2);
                        np3 += (uint32_t)__builtin_popcount(ch >> 5);
                        if (at0) s0info[steps - 1] = (uint16_t)(__builtin_popcount(ch) | units << 4);
                        if (TRACE) SINFO[tid * H_SLOG + sl - 1] = (uint8_t)__builtin_popcount(ch);
                        ch |= qb << 9 & 0x600u;
                        ch |= open ? 0x800u : 0u;
                        if (fan) {
                        } else if (kind == K_END && ex && cid >= solo) {
                            // the exact child is popped next, or (the round's steps or the log used up) in the
                            // next round
                            k = xk;
                            l = xl;
                            x = p_x - 1;
                            y = p_y;
                            if (steps == STEPS || wl > LOG_FULL || ((np3 + ROOM) & 0x808080u) != 0) {
                                kind = K_TRUNC;
                                finish();
                            } else {
                                pop(wA);
                            }
                        } else {
                            finish();
                        }
                    }
                }
                if (fan) {
                    // the steps' pushes are ranked in their order (10 bits a bucket code); the chain ends at the step
                    // whose pushes fill a code's ranks, or that met a score error; lane 0 goes on with it
                    const auto &W = F.ahead[wave];
                    const uint32_t base = W.np3, own = (np3 & 255u) | (np3 >> 8 & 255u) << 10 | (np3 >> 16 & 255u) << 20;
                    const uint32_t incl = wave_incl_scan(own) + ((base & 255u) | (base >> 8 & 255u) << 10 | (base >> 16 & 255u) << 20);
                    const int n = __builtin_amdgcn_readlane((int)W.n, 0);
                    int end = __builtin_amdgcn_readlane((int)W.end, 0), fin = n - 1;
                    const uint32_t most = max(max(incl & 1023u, incl >> 10 & 1023u), incl >> 20);
                    const uint64_t full = __ballot(busy && most > (uint32_t)(H_CPUSH - H_SPUSH) && lane < n - 1), bad = __ballot(busy && kind == K_ESCORE);
                    if (full) {
                        fin = __builtin_ctzll(full);
                        end = K_TRUNC;
                    }
                    if (bad && __builtin_ctzll(bad) <= fin) {
                        fin = __builtin_ctzll(bad);
                        end = K_ESCORE;
                    }
                    const uint64_t in = ~0ull >> (63 - fin);
                    const uint32_t units = (uint32_t)(__builtin_popcountll(in & __ballot(sby != 0)) + __builtin_popcountll(in & __ballot(sby == 2)));
                    const uint32_t pre = incl - own, tot = (uint32_t)__builtin_amdgcn_readlane((int)incl, fin);
                    p_np3 = (pre & 255u) | (pre >> 10 & 255u) << 8 | (pre >> 20) << 16;
                    const K nk = lane_value<K>(k, (fin + 1) & 63), nl = lane_value<K>(l, (fin + 1) & 63);
                    if (lane > fin) ch = 0;
                    kind = K_END;
                    busy = false;
                    if (lane == 0) {
                        const bool inner = fin < n - 1;
                        k = inner ? nk : (K)W.k;
                        l = inner ? nl : (K)W.l;
                        x = (x & ~X_ST) - (uint32_t)(fin + 1);
                        y &= ~Y_LDP;
                        np3 = (tot & 255u) | (tot >> 10 & 255u) << 8 | (tot >> 20) << 16;
                        sby = W.sby + units;
                        steps = (int)W.steps + fin + (end == K_DEAD || end == K_HIT || end == K_TAIL ? 1 : 0);
                        kind = end == K_DEAD || end == K_TAIL ? K_END : end;
                        if (end == K_TAIL) {
                            busy = true;
                            tail = true;
                        } else {
                            finish();
                        }
                    }
                }
                // the first chain that stops (a hit, a truncation, a score error): those after it run again
                // in the next round
                const uint64_t sm = __ballot(kind != K_END);
                if (sm != stopped) {
                    stopped = sm;
                    more = false;
                    if (NW == 1) {
                        for (uint64_t t = sm; t; t &= t - 1) stop = min(stop, __builtin_amdgcn_readlane(cid, __builtin_ctzll(t)));
                    } else {
                        stop = __hip_atomic_load(&F.stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    }
                    if (cid > stop) busy = false;
                }
            }
            if (NW == 1 && stopped == 0) {  // (a chain that stopped when it was taken last)
                for (uint64_t t = __ballot(kind != K_END); t; t &= t - 1)
                    stop = min(stop, __builtin_amdgcn_readlane(cid, __builtin_ctzll(t)));
            }
            const long long t_commit = stats ? wall_clock64() : 0;
            __syncthreads();
            // ---- commit plan, by scans over the chains (thread t: chains t * CPL on) ----
            if (NW > 1) {
                next = F.next;
                stop = F.stop;
            }
            const int run = next < nlive ? (int)hcid[next] : nK;  // chains before the first one not taken
            const int J = min(stop, run - 1);
            const int push_cap = HA(push_cap);
            uint32_t v01[CPL], v2s[CPL], vb[CPL];
            uint32_t s01 = 0, s2s = 0, sb = 0;
#pragma unroll
            for (int r = 0; r < CPL; ++r) {
                const int c = tid * CPL + r;
                const bool in = c <= J;
                const uint32_t A = in ? cA[c] : 0u, C = in ? cC[c] : 0u;
                v01[r] = (A & 255u) | ((A >> 8) & 255u) << 16;
                v2s[r] = ((A >> 16) & 255u) | (C & 63u) << 16;
                vb[r] = C >> 6;
                s01 += v01[r];
                s2s += v2s[r];
                sb += vb[r];
            }
            uint32_t e01 = wave_incl_scan(s01), e2s = wave_incl_scan(s2s), eb = wave_incl_scan(sb);
            if (NW > 1) {
                if (lane == HW - 1) {
                    F.wsum[0][wave] = e01;
                    F.wsum[1][wave] = e2s;
                    F.wsum[2][wave] = eb;
                }
                __syncthreads();
                for (int w = 0; w < wave; ++w) {
                    e01 += F.wsum[0][w];
                    e2s += F.wsum[1][w];
                    eb += F.wsum[2][w];
                }
            }
            e01 -= s01;
            e2s -= s2s;
            eb -= sb;
            // pushes before each chain by code (over the heads, which are not needed any more), and the first
            // chain that must wait for the next round: the push cap falls in it (chain 0 always fits), or
            // the max_entries check before a pop could (src/bwtgap_hd.h:360); chain 0 is walked step by step
            {
                uint32_t p01 = e01, p2s = e2s;
                int wait = 0x7fffffff;
                bool walk0 = false;
#pragma unroll
                for (int r = 0; r < CPL; ++r) {
                    const int c = tid * CPL + r;
                    if (c <= J) {
                        epre[c] = (uint16_t)p01;
                        epre[KMAX + c] = (uint16_t)(p01 >> 16);
                        epre[2 * KMAX + c] = (uint16_t)p2s;
                        const int pex = (int)((p01 & 0xffffu) + (p01 >> 16) + (p2s & 0xffffu));
                        const int np = (int)((v01[r] & 0xffffu) + (v01[r] >> 16) + (v2s[r] & 0xffffu));
                        // each chain before this one popped its head and left its pushes (in the root's round,
                        // and the next step of the root chain)
                        const bool over = (long)F.n_entries + pex - (root ? 0 : c) + np > (long)F.max_entries;
                        if (c == 0)
                            walk0 = over;
                        else if ((over || pex + np > push_cap) && wait == 0x7fffffff)
                            wait = c;
                        p01 += v01[r];
                        p2s += v2s[r];
                    }
                }
                if (wait != 0x7fffffff) atomicMin(&F.lim, wait);
                if (walk0) {
                    const int s0 = (int)(cC[0] & 63u);
                    long nb = F.n_entries;
                    unsigned long long by = 0;
                    for (int t = 0; t < s0; ++t) {
                        if (nb > F.max_entries) {
                            F.cut = t;
                            break;
                        }
                        nb += s0info[t] & 15;
                        by += s0info[t] >> 4;
                    }
                    if (F.cut >= 0) {
                        // the search stops inside chain 0
                        F.pops += (unsigned long long)F.cut;
                        F.obytes += by << 6;
                        F.status = 1;
                        F.result = F.n_aln;
                    } else {
                        atomicMin(&F.lim, 1);
                    }
                }
            }
            __syncthreads();
            const int last = min(J, F.lim - 1);  // chains 0..last commit
            if (TRACE && tid == 0) {
                // the trace hash runs over the committed pops in order
                uint64_t tr = F.trace;
                int nb = F.n_entries;
                const int cut = F.cut;
                for (int j = 0; j <= (cut >= 0 ? 0 : last); ++j) {
                    const int t0 = (int)cS[j], n = cut >= 0 ? cut : (int)(cC[j] & 63u);
                    for (int t = 0; t < n; ++t) {
                        const Item<WIDE> e = get_item<WIDE>(SLOG + t0 + t);
                        nb -= 1;
                        tr = trace_item(tr, b, e.k, e.l, e.x, e.y, nb);
                        nb += (int)SINFO[t0 + t] + (t + 1 < n || root ? 1 : 0);  // its pushes, and its exact child
                    }
                }
                F.trace = tr;
            }
            if (F.status) break;
            if (last / CPL == tid) {
                uint32_t p01 = e01, p2s = e2s, pb = eb;
#pragma unroll
                for (int r = 0; r < CPL; ++r)
                    if (tid * CPL + r <= last) {
                        p01 += v01[r];
                        p2s += v2s[r];
                        pb += vb[r];
                    }
                F.tot01 = p01;
                F.tot2s = p2s;
                F.totb = pb;
            }
            if (kind != K_END && cid == last) {
                F.l_kind = kind;
                F.hk = k;
                F.hl = l;
                F.hx = x;
                F.hy = y;
            }
            __syncthreads();
            const long long t_c1 = stats ? wall_clock64() : 0;
            const uint32_t tot01 = F.tot01, tot2s = F.tot2s;
            const int T0 = (int)(tot01 & 0xffffu), T1 = (int)(tot01 >> 16), T2 = (int)(tot2s & 0xffffu);
            if (tid == 0) {
                // where each bucket's pushes go: the rest of its top granule, then new ones
                int np_ = 0;
                bool oom = false;
                for (int c = 0; c < 3 && !oom; ++c) {
                    // (selects: arrays indexed by c would live in scratch memory)
                    const int sbk = c == 0 ? tg0 : c == 1 ? tg1 : tg2;
                    uint32_t rem = (uint32_t)(c == 0 ? T0 : c == 1 ? T1 : T2), rk = 0;
                    if (!rem) continue;
                    uint32_t cnt = seg_cnt[sbk], top = cnt ? seg_top[sbk] : NIL;
                    F.fp[c] = np_;
                    if (cnt && cnt < GFULL) {
                        rk = min(rem, GFULL - cnt);
                        pieces[np_++] = make_uint4((uint32_t)c, 0u, rk, top * GENT + 1 + cnt);
                        cnt += rk;
                        rem -= rk;
                    }
                    while (rem > 0) {
                        uint32_t g;
                        if (F.n_free > 0) {
                            g = F.free_g[--F.n_free];
                        } else if (F.n_spill > 0) {
                            g = SPILL[--F.n_spill];
                        } else if (F.n_used < F.n_own) {
                            g = F.n_used < H_KEEP ? F.own[F.n_used] : OWN[F.n_used];
                            ++F.n_used;
                        } else {
                            g = F.n_own < HA(own_cap) ? gran_pop(HA(ghead), HA(gnext), HA(gbump), HA(n_gran)) : NIL;
                            if (g == NIL) {
                                oom = true;
                                break;
                            }
                            if (stats) ST[11] += 1;
                            if (F.n_own < H_KEEP) F.own[F.n_own] = g;
                            OWN[F.n_own++] = g;
                            ++F.n_used;
                        }
                        if (np_ == H_PIECES) {  // (not possible: the push cap spans fewer granules)
                            oom = true;
                            break;
                        }
                        Ent link;
                        link.w0 = top;
                        link.w1 = 0;
                        POOL[g * GENT] = link;
                        seg_prev[sbk] = top;
                        top = g;
                        cnt = min(rem, GFULL);
                        pieces[np_++] = make_uint4((uint32_t)c, rk, cnt, g * GENT + 1);
                        rem -= cnt;
                        rk += cnt;
                    }
                    seg_top[sbk] = top;
                    seg_cnt[sbk] = cnt;
                    F.bm[sbk >> 6] |= 1ull << (sbk & 63);
                }
                F.n_piece = np_;
                if (oom) {
                    F.status = 1;
                    F.result = ERR_STACK;
                }
                F.pops += tot2s >> 16;
                F.obytes += (unsigned long long)F.totb << 6;
            }
            __syncthreads();
            if (F.status) break;
            const long long t_c2 = stats ? wall_clock64() : 0;
            // ---- placement: every logged push of a committed chain to its place among its bucket's pushes of
            // the round ----
            {
                const int npieces = F.n_piece;
                for (uint32_t g = lane; g < wl; g += HW) {
                    Item<WIDE> e = get_item<WIDE>(LOG + g);
                    uint32_t code, chain;
                    if constexpr (WIDE) {
                        const uint32_t w = LOGW[g];
                        chain = w & ((1u << H_CHAIN_BITS) - 1);
                        code = w >> H_CHAIN_BITS;
                    } else {
                        chain = e.x >> 28 << 6 | e.y >> 26;
                        code = (e.x >> 26) & 3u;
                        e.x &= (1u << 26) - 1;
                        e.y &= (1u << 26) - 1;
                    }
                    if ((int)chain > last) continue;
                    const uint32_t R = epre[code * KMAX + chain] + (e.y & 127u);
                    e.y = (e.y & ~Y_LDP) | (e.x & X_I);
                    int p = F.fp[code];
                    uint4 pc = pieces[p];
                    while (R - pc.y >= pc.z && p + 1 < npieces) pc = pieces[++p];
                    if (pc.x == code && R - pc.y < pc.z)
                        put_item<WIDE>(POOL + pc.w + (R - pc.y), e.k, e.l, e.x, e.y);
                    else
                        F.bad = 1;  // a rank outside this round's pieces: not possible
                }
            }
            __syncthreads();
            const long long t_c3 = stats ? wall_clock64() : 0;
            // ---- bucket b: the committed start entries leave its top; the state moves on ----
            const int l_kind = F.l_kind;
            if (tid == 0) {
                const int taken = last + 1;
                const int from_seg = root ? 0 : taken - hp;
                F.has_pend = 0;
                F.root = 0;
                if (from_seg > 0) {
                    uint32_t n = (uint32_t)from_seg, cnt = seg_cnt[b], top = seg_top[b], prev = seg_prev[b];
                    while (n >= cnt) {
                        // the top granule is empty: the next one taken, and the one below is the top
                        n -= cnt;
                        if (F.n_free < H_FREE)
                            F.free_g[F.n_free++] = top;
                        else
                            SPILL[F.n_spill++] = top;
                        if (prev == NIL) {
                            cnt = 0;
                            F.bm[b >> 6] &= ~(1ull << (b & 63));
                            break;
                        }
                        top = prev;
                        cnt = GFULL;
                        prev = (uint32_t)POOL[top * GENT].w0;
                    }
                    seg_cnt[b] = cnt - n;
                    seg_top[b] = top;
                    seg_prev[b] = prev;
                }
                // entries: every chain's head left, its pushes came; a pending child is one more
                int ne = F.n_entries + T0 + T1 + T2 - (root ? 1 : taken);
                if (root && last < solo && l_kind == K_END) {
                    // (cut short: the next step of the root chain waits)
                    const Item<WIDE> e = root_step(last + 1);
                    F.has_pend = 1;
                    F.hk = e.k;
                    F.hl = e.l;
                    F.hx = e.x;
                    F.hy = e.y;
                    ne += 1;
                }
                if (l_kind == K_TRUNC) {
                    F.has_pend = 1;
                    ne += 1;
                }
                F.n_entries = ne;
                if (l_kind == K_ESCORE || F.bad) {
                    F.status = 1;
                    F.result = F.bad ? ERR_INTERNAL : ERR_SCORE;
                }
                if (stats) {
                    ST[0] += 1;
                    ST[1] += (unsigned long long)nK;
                    ST[2] += (unsigned long long)taken;
                    ST[3] += tot2s >> 16;
                    ST[4] += (unsigned long long)its;
                    ST[5] += (unsigned long long)(t_commit - t_spec);
                    const long long t_end = wall_clock64();
                    t_round_end = t_end;
                    ST[6] += (unsigned long long)(t_end - t_commit);
                    ST[7] += (unsigned long long)(t_c1 - t_commit);
                    ST[8] += (unsigned long long)(t_c2 - t_c1);
                    ST[9] += (unsigned long long)(t_c3 - t_c2);
                    ST[10] += (unsigned long long)(t_end - t_c3);
                }
            }
            if (l_kind == K_HIT && wave == 0 && F.status == 0) {
                // a hit ends the last committed chain (src/bwtgap_hd.h:385-409); one wave applies it
                const uint64_t hk = F.hk, hl = F.hl;
                const uint32_t hx = F.hx, hy = F.hy;
                const int n_aln = F.n_aln, mm = x_mm(hx), go = x_go(hx), ge = y_ge(hy);
                const bool same = n_aln == 0 || b == F.best_score;
                const bool stop_hits = !same && F.best_cnt > F.max_top2;
                bool dup = false;
                if (!stop_hits && go) {
                    for (int j0 = 0; j0 < n_aln && !dup; j0 += HW) {
                        const int j = j0 + lane;
                        dup = __ballot(j < n_aln && REC[j].k == hk && REC[j].l == hl) != 0;
                    }
                }
                if (!stop_hits && !dup) {
                    // gap_shadow (src/bwtgap_hd.h:309-320); the widths equal to the hit's are numbered in order
                    const uint64_t ux = (uint64_t)(int64_t)(int)(uint32_t)(hl - hk + 1);
                    const int ldp = (int)(hy & Y_LDP);
                    uint64_t eq = 0;
                    for (int j0 = 0; j0 < ldp; j0 += HW) {
                        const int j = j0 + lane;
                        const uint64_t v = j < ldp ? Wp[1 + j] : 0, w = lw_val<WIDE>(v);
                        const uint64_t em = __ballot(j < ldp && w == ux);
                        if (j < ldp && w > ux) Wp[1 + j] = lw_make<WIDE>(w - ux, (uint32_t)lw_bid<WIDE>(v));
                        if (j < ldp && w == ux) Wp[1 + j] = lw_make<WIDE>(M.seq_len - (eq + (uint64_t)lanes_below(em) + 1), 1);
                        eq += (uint64_t)__builtin_popcountll(em);
                    }
                }
                __builtin_amdgcn_wave_barrier();  // (the wave has read the state that lane 0 changes)
                if (lane == 0) {
                    if (n_aln == 0) {
                        F.best_score = b;
                        F.best_diff = mm + go + ((mode & MODE_GAPE) ? ge : 0);
                        if (!(mode & MODE_NONSTOP)) F.max_diff = (F.best_diff + 1 > F.md_read) ? F.md_read : F.best_diff + 1;
                    }
                    if (same) F.best_cnt = (int)(uint32_t)((uint64_t)(int64_t)F.best_cnt + (hl - hk + 1));
                    if (stop_hits) {
                        F.status = 1;
                        F.result = n_aln;
                    } else if (!dup) {
                        if (n_aln == HA(rec_cap)) {
                            F.status = 1;
                            F.result = ERR_ALN;
                        } else {
                            const int ins = y_ins(hy), del = go + ge - ins;
                            galn_aln_rec_t r;
                            r.packed = ((uint64_t)(mm & 0xff)) | ((uint64_t)(go & 0xff) << 8) | ((uint64_t)(ge & 0xff) << 16) |
                                       ((uint64_t)(b & 0xfffff) << 24) | ((uint64_t)(ins & 0x3ff) << 44) |
                                       ((uint64_t)(del & 0x3ff) << 54);
                            r.k = hk;
                            r.l = hl;
                            REC[n_aln] = r;
                            F.n_aln = n_aln + 1;
                        }
                    }
                }
            }
            if (!RESUME && tid == 0 && F.status == 0 && HA(park_pops) && taken_reads >= n_list) F.status = 2;
            __syncthreads();
        }
        if (!RESUME && F.status == 2) {
            __syncthreads();
            if (tid == 0) F.status = 0;
            __syncthreads();
            uint32_t *const st = reinterpret_cast<uint32_t *>(base + HA(state_off));
            for (int j = tid; j < state_words; j += T)
                st[j] = reinterpret_cast<const uint32_t *>(&F)[j];
            if (tid == 0) {
                HA(park_list)[atomicAdd(HA(park_n), 1)] = (int32_t)blockIdx.x;
                F.n_own = 0;  // its granules stay with it
            }
            break;  // (no read is left to take)
        }
        // ---- the read's result ----
        if (tid == 0) {
            int n = F.result;
            if (n > 0) {
                const unsigned long long b0 = atomicAdd(HA(out_top), (unsigned long long)n);
                if (b0 + (unsigned long long)n > HA(out_cap)) {
                    n = ERR_OUT;
                } else {
                    for (int j = 0; j < n; ++j) HA(out_rec)[b0 + j] = REC[j];
                    HA(out_off)[rid] = b0;
                }
            }
            if (n == ERR_STACK || n == ERR_ALN || n == ERR_OUT) {
                const int f = atomicAdd(HA(fail_n), 1);
                HA(fail_list)[f] = rid;
                atomicOr(HA(fail_kind) + (n == ERR_OUT ? 0 : n == ERR_ALN ? 1 : 2), 1);
            } else {
                atomicAdd(HA(algo_bytes), F.obytes);
            }
            HA(out_n)[rid] = n;
            HA(out_pops)[rid] = F.pops;
            if (TRACE) HA(out_trace)[rid] = F.trace;
            if (HA(out_bytes)) HA(out_bytes)[rid] = F.obytes;
            // keep a few granules for the next read; the rest go back to the pool (a parked read's all)
            const int keep = RESUME ? 0 : H_KEEP;
            if (F.n_own > keep) {
                gran_push(HA(ghead), HA(gnext), OWN, keep, F.n_own);
                F.n_own = keep;
            }
        }
        __syncthreads();
    }
    // the granules this workgroup still holds are for the reads that were parked
    if (tid == 0 && HA(park_pops) && F.n_own > 0) gran_push(HA(ghead), HA(gnext), OWN, 0, F.n_own);
    if (stats && tid < 16) atomicAdd(HA(stats) + tid, ST[tid]);
}

// A read's record count for the output offsets (error codes count none).
struct RecCount {
    __host__ __device__ uint64_t operator()(int32_t v) const { return v > 0 ? (uint64_t)v : 0; }
};

// Records of every read in read order: read i's n_aln[i] records move from the arena (at
// arena_off[i], where the search appended them) to incl[i] - n_aln[i] of the staging array.
__global__ void k_gather_records(const int32_t *n_aln, const uint64_t *arena_off, const uint64_t *incl,
                                 const galn_aln_rec_t *arena, galn_aln_rec_t *stage, uint64_t *rec_off, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int na = n_aln[i] > 0 ? n_aln[i] : 0;
    const uint64_t o = incl[i] - (uint64_t)na;
    rec_off[i] = o;
    for (int j = 0; j < na; ++j) stage[o + j] = arena[arena_off[i] + j];
}

// Fills n words with v: the search's counter and pool-head resets, as kernels so that a
// captured graph holds no memset nodes.
__global__ void k_fill_u32(uint32_t *p, uint32_t v, uint32_t n)
{
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = v;
}

// The resets before a search, and before a launch of the wave engine, in one kernel each.
__global__ void k_reset_search(unsigned long long *algo, int n_algo, unsigned long long *stats, unsigned long long *top, int32_t *ctr)
{
    for (int i = threadIdx.x; i < n_algo; i += blockDim.x) algo[i] = 0;
    if (threadIdx.x < 16) stats[threadIdx.x] = 0;
    if (threadIdx.x < 8) ctr[threadIdx.x] = 0;
    if (threadIdx.x == 0) *top = 0;
}

__global__ void k_reset_heavy(int32_t *qnext, int32_t *park_n, unsigned long long *ghead, uint32_t *gbump, uint32_t first)
{
    for (int i = threadIdx.x; i < NSHARD; i += blockDim.x) ghead[i] = ~0ull;  // an empty free stack
    if (threadIdx.x == 0) {
        *qnext = 0;
        park_n[0] = park_n[1] = 0;
        *gbump = first;  // granules handed out: those the workgroups start with
    }
}

// ---------------------------------------------------------------------------
// host side

thread_local char g_err[512];

int fail(int code, const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

// progress lines on stderr for long calls (GALN_HIP_VERBOSE set and not "0")
bool galn_hip_verbose()
{
    const char *v = getenv("GALN_HIP_VERBOSE");
    return v && *v && strcmp(v, "0") != 0;
}

#define HIP_OK(call)                                                                                   \
    do {                                                                                               \
        hipError_t e_ = (call);                                                                        \
        if (e_ != hipSuccess)                                                                          \
            return fail(e_ == hipErrorOutOfMemory ? GALN_HIP_E_NOMEM : GALN_HIP_E_DEVICE, "%s:%d %s: %s", \
                        __FILE__, __LINE__, #call, hipGetErrorString(e_));                             \
    } while (0)

struct Tier {
    int rec_cap;   // record slots per lane
    int keep;      // granules a lane keeps between reads
};

}  // namespace

// What a search reads back at its end, in pinned memory.
constexpr int galn_max_launch = 256;
struct SearchBack {
    unsigned long long algo[galn_max_launch];
    int32_t failed;
    uint32_t used;
};

// A read set has one of its own; up to eight (2 KB each) wait here for the next read sets of the process, on any
// device, since pinning and unpinning one takes most of what an upload of few reads costs.
struct BackPool {
    std::mutex mu;
    SearchBack *kept[8] = {};
    int n = 0;
    SearchBack *take()
    {
        {
            std::lock_guard<std::mutex> g(mu);
            if (n > 0) return kept[--n];
        }
        SearchBack *b = nullptr;
        return hipHostMalloc((void **)&b, sizeof *b, hipHostMallocPortable) == hipSuccess ? b : nullptr;
    }
    void give(SearchBack *b)
    {
        {
            std::lock_guard<std::mutex> g(mu);
            if (n < 8) {
                kept[n++] = b;
                return;
            }
        }
        (void)hipHostFree(b);
    }
};
static BackPool g_backs;

// Where a search runs: a stream and a stack pool (grown on demand). The read sets of an index
// share its context; a read set of a server slot has one of its own, so that slots' launches run
// at the same time.
struct SearchCtx {
    hipStream_t stream = nullptr;
    Ent *d_pool_chk = nullptr;
    uint32_t *d_pool_link = nullptr, *d_gnext = nullptr, *d_gbump = nullptr;
    unsigned long long *d_ghead = nullptr;
    uint32_t n_gran = 0;
    bool grow = false;  // the last search used every never-used granule: double the pool next time
    // frees the pool (not the stream)
    void free_pool()
    {
        void *p[] = {d_pool_chk, d_pool_link, d_gnext, d_gbump, d_ghead};
        for (void *x : p)
            if (x) (void)hipFree(x);
        d_pool_chk = nullptr, d_pool_link = nullptr, d_gnext = nullptr, d_gbump = nullptr, d_ghead = nullptr;
        n_gran = 0;
    }
};

struct galn_hip_index {
    int device = 0;
    uint32_t *d_bwt = nullptr;
    uint64_t *d_ext = nullptr;  // per epoch: the bases' counts at its start (k_epochs)
    DMeta meta{};
    galn_bwt_meta_t hmeta{};
    int n_cu = 0;
    SearchCtx ctx0;  // the stream and stack pool of the index's own read sets
    // SA samples (galn_hip_index_set_sa): the suffix at rows intv, 2 intv, ...
    uint64_t *d_sa = nullptr;
    uint64_t n_sa = 0;
    uint32_t sa_intv = 0;
    std::atomic<int> n_readsets{0};  // read sets not yet freed (they use the stream and pool)
    std::atomic<int> n_servers{0};   // open servers: the index then belongs to their workers
};

struct GraphKey {
    uint32_t flags;
    int32_t block, slots, hwaves, n;
    uint64_t budget;
    uint32_t rec_cap, keep;
    const int32_t *list;
    const void *ptr[21];
    uint64_t rec_cap_out, n_gran, scratch_bytes, hscratch_bytes;
    int32_t max_len, seed_len, max_stacks, max_entries;
    const void *hand;
    int32_t hand_cap;
    uint32_t hand_stride;
    int32_t push_cap;
    uint32_t park_pops;
};

struct galn_hip_readset {
    galn_hip_index *idx = nullptr;
    SearchCtx *ctx = nullptr;   // &idx->ctx0, or own_ctx
    SearchCtx *own_ctx = nullptr;
    int n = 0;
    int n_batches = 0;
    int seed_len = 0;
    int max_len = 0;
    int max_stacks = 0;
    int max_entries = 0;
    uint64_t qbytes = 0;
    // device inputs
    uint8_t *d_query = nullptr;
    uint64_t *d_qoff = nullptr;
    int32_t *d_qlen = nullptr, *d_maxdiff = nullptr, *d_batch = nullptr, *d_nstacks = nullptr;
    galn_search_opt_t *d_bopts = nullptr;
    int32_t *d_sorted = nullptr;   // read ids, longest first
    // device outputs
    int32_t *d_out_n = nullptr;
    uint64_t *d_out_off = nullptr, *d_pops = nullptr, *d_trace = nullptr, *d_bytes = nullptr;
    galn_aln_rec_t *d_rec = nullptr;
    uint64_t rec_cap = 0;
    unsigned long long *d_top = nullptr;
    int32_t *d_fail[2] = {nullptr, nullptr};
    int32_t *d_ctr = nullptr;      // [0],[1] failure counts, [2] queue head, [3] heavy count, [4..6] failure kinds,
                                   // [8] parked count, [9] parked queue head
    int32_t *d_heavy = nullptr;    // reads handed to the wave-per-read engine
    unsigned long long *d_stats = nullptr;  // wave-per-read engine counters of the last search
    uint8_t *d_hscratch = nullptr; // per-wave regions of the wave-per-read engine
    size_t hscratch_bytes = 0;
    int32_t *d_park = nullptr;     // its workgroups that parked a read
    size_t park_bytes = 0;
    // per-lane regions (grown on demand)
    uint8_t *d_scratch = nullptr;
    size_t scratch_bytes = 0;
    // host copies
    std::vector<galn_search_opt_t> h_bopts;
    // widths handed from k_search to k_heavy, one slot per heavy-list position
    uint64_t *d_hand = nullptr;
    size_t hand_bytes = 0;
    uint32_t hand_stride = 0;
    int32_t hand_root = 0;  // steps of a root chain in each
    int32_t hand_cap = 0;
    // results in read order: inclusive prefix sums of record counts, output offsets, staging
    uint64_t *d_incl = nullptr, *d_roff = nullptr;
    galn_aln_rec_t *d_stage = nullptr;
    size_t stage_bytes = 0;
    void *d_scan_tmp = nullptr;
    size_t scan_tmp_bytes = 0;
    // capacities of the device arrays (reads, query bytes, batches)
    int cap_n = 0, cap_b = 0;
    uint64_t cap_q = 0;
    // last search: one record per kernel launch, timed with events on the search stream
    double first_ms = 0, total_ms = 0;
    // the batched form's tuning chosen by galn_hip_readset_autotune (used when a search passes none)
    bool has_tuned = false;
    galn_hip_tune_t tuned{};
    uint32_t last_flags = 0;
    hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
    struct Launch {
        int tier;
        int slot;
        double ms;
        uint64_t bytes;
    };
    std::vector<Launch> launches;
    // the batched form's captured graph (GALN_HIP_GRAPH), its key and its launch records
    hipGraphExec_t gexec = nullptr, gexec2 = nullptr;  // prologue + first tier; wave engine
    bool capturing = false;  // launches skip their timing events (recorded around the graphs)
    GraphKey gkey{};
    std::vector<Launch> glaunches;
    std::vector<hipEvent_t> lev;           // 2 per launch, reused across searches
    SearchBack *back = nullptr;
    unsigned long long *d_algo = nullptr;  // per-launch algorithmic byte counters
    static constexpr int MAX_LAUNCH = galn_max_launch;
    struct {
        const void *kernel;
        size_t lds;
        int groups;
    } occ[4] = {};                         // workgroups of the wave engine a CU holds, as asked of the runtime
};

namespace {

size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// every device allocation of this file (one that finds no room takes back what earlier builds left)
template <class T>
hipError_t dev_malloc(T **p, size_t bytes)
{
    return galn_hip_dev_malloc(reinterpret_cast<void **>(p), bytes);
}

struct Layout {
    uint64_t slot_bytes;
    uint32_t sw_off, rec_off, own_off;
    int own_cap;
};

Layout make_layout(int max_len, int seed_len, int rec_cap, int own_cap)
{
    Layout L{};
    size_t off = align_up((size_t)(max_len + 1) * 8, 256);
    L.sw_off = (uint32_t)off;
    const int sl = (seed_len > 0 && seed_len < max_len) ? seed_len : 0;
    off += align_up((size_t)(sl + 1) * 8, 256);
    L.rec_off = (uint32_t)off;
    off += align_up((size_t)rec_cap * sizeof(galn_aln_rec_t), 256);
    L.own_off = (uint32_t)off;
    off += align_up((size_t)own_cap * 4, 256);
    // an odd multiple of 256 bytes keeps lanes' regions off the same cache sets
    if ((off / 256) % 2 == 0) off += 256;
    L.slot_bytes = off;
    L.own_cap = own_cap;
    return L;
}

// A device buffer of at least `need` bytes (contents not kept). It grows to twice its size or
// more: hipFree waits for every stream of the device, so a read set whose launches vary in size
// (a server slot) reallocates a few times rather than every launch.
int grow_dev(void **p, size_t &cap, size_t need, hipStream_t s)
{
    if (*p && cap >= need) return 0;
    HIP_OK(hipStreamSynchronize(s));
    if (*p) HIP_OK(hipFree(*p));
    *p = nullptr;
    const size_t c = std::max(need, cap * 2);
    if (dev_malloc(p, c) != hipSuccess) {
        (void)hipGetLastError();
        *p = nullptr;
        cap = 0;
        if (dev_malloc(p, need) != hipSuccess) return fail(GALN_HIP_E_NOMEM, "device allocation of %zu bytes failed", need);
        cap = need;
        return 0;
    }
    cap = c;
    return 0;
}

int ensure_scratch(galn_hip_readset *rs, size_t bytes)
{
    return grow_dev((void **)&rs->d_scratch, rs->scratch_bytes, bytes, rs->ctx->stream);
}

// Granules the stack pool may hold at most: no limit, or the value of GALN_HIP_TEST_POOL_GRANULES,
// which the tests set to exhaust the pool and drive the re-runs with fewer lanes.
uint64_t pool_test_cap()
{
    const char *v = getenv("GALN_HIP_TEST_POOL_GRANULES");
    if (!v || !*v) return ~0ull;
    return (uint64_t)std::max(1L, strtol(v, nullptr, 10));
}

// Granules of a context's first pool: as asked, or the value of GALN_HIP_TEST_POOL_START, which the
// tests set low so that the pool's growth on demand runs.
uint64_t pool_test_start()
{
    const char *v = getenv("GALN_HIP_TEST_POOL_START");
    if (!v || !*v) return ~0ull;
    return (uint64_t)std::max(1024L, strtol(v, nullptr, 10));
}

// The stack pool: `want` granules of 64 chunks (16 KB each), within half the free memory and the
// 28-bit chunk ids of the bucket tops (2^22 granules, 64 GiB).
int ensure_pool(SearchCtx *idx, uint64_t want)
{
    // contexts of one process size their pools one at a time (server slots start together: each
    // would otherwise count the same free memory)
    static std::mutex mu;
    std::lock_guard<std::mutex> lk(mu);
    const uint64_t gbytes = (uint64_t)GRAN * CH * sizeof(Ent);
    const uint64_t have = idx->n_gran;
    if (!idx->grow && have >= std::max<uint64_t>(want, 1024)) return 0;
    size_t freeb = 0, totalb = 0;
    HIP_OK(hipMemGetInfo(&freeb, &totalb));
    uint64_t cap = (uint64_t)((freeb + have * (gbytes + GRAN * 4 + 4)) / 2) / (gbytes + GRAN * 4 + 4);
    cap = std::min<uint64_t>(cap, MAX_POOL_CHUNKS / GRAN);
    cap = std::min<uint64_t>(cap, pool_test_cap());
    // a search that used up the never-used granules made every later allocation search the other
    // shards' free lists (one wave's read can hold millions of entries on a repeat-rich genome: on
    // the 3.1 Gbp human-like workload a 26 GB pool spent 3x the search time allocating)
    if (idx->grow) want = std::max<uint64_t>(want, 2 * have);
    idx->grow = false;
    if (have == 0) want = std::min(want, pool_test_start());
    want = std::min(std::max<uint64_t>(want, 1024), cap);
    if (have >= want) return 0;
    if (!idx->d_ghead) {
        unsigned long long *head = nullptr;
        uint32_t *bump = nullptr;
        HIP_OK(dev_malloc(&head, NSHARD * 8));
        if (dev_malloc(&bump, 4) != hipSuccess) {
            (void)hipFree(head);
            return fail(GALN_HIP_E_NOMEM, "stack pool: allocation of its heads failed");
        }
        idx->d_ghead = head;
        idx->d_gbump = bump;
    }
    // the old pool goes first (it is not copied: no search is running), then all three new
    // arrays are allocated before any of them is installed, so a failure leaves an empty pool
    // (null pointers, no granules) and nothing freed twice
    void *old[] = {idx->d_pool_chk, idx->d_pool_link, idx->d_gnext};
    idx->d_pool_chk = nullptr;
    idx->d_pool_link = nullptr;
    idx->d_gnext = nullptr;
    idx->n_gran = 0;
    for (void *p : old)
        if (p) HIP_OK(hipFree(p));
    Ent *chk = nullptr;
    uint32_t *link = nullptr, *gnext = nullptr;
    // half as many granules while the allocation fails (other allocations of the process, or of
    // other processes, since the free memory was read): a smaller pool only costs re-runs
    for (;;) {
        if (dev_malloc(&chk, want * gbytes) == hipSuccess && dev_malloc(&link, want * GRAN * 4) == hipSuccess &&
            dev_malloc(&gnext, want * 4) == hipSuccess)
            break;
        (void)hipGetLastError();
        for (void *p : {(void *)chk, (void *)link, (void *)gnext})
            if (p) (void)hipFree(p);
        chk = nullptr, link = nullptr, gnext = nullptr;
        if (want <= 1024)
            return fail(GALN_HIP_E_NOMEM, "stack pool of %llu granules does not fit in device memory",
                        (unsigned long long)want);
        want = std::max<uint64_t>(want / 2, 1024);
    }
    idx->d_pool_chk = chk;
    idx->d_pool_link = link;
    idx->d_gnext = gnext;
    idx->n_gran = (uint32_t)want;
    return 0;
}

template <bool TRACE, bool PERSIST>
int launch_one(hipStream_t st, const KArgs &a, int block, int grid, int buckets)
{
    const size_t lds = (size_t)block * buckets * sizeof(uint32_t);
    hipLaunchKernelGGL((k_search<TRACE, PERSIST>), dim3(grid), dim3(block), lds, st, a);
    HIP_OK(hipGetLastError());
    return 0;
}

int launch(hipStream_t st, const KArgs &a, int block, int grid, bool persist, bool trace, int buckets)
{
    if (trace) return persist ? launch_one<true, true>(st, a, block, grid, buckets)
                              : launch_one<true, false>(st, a, block, grid, buckets);
    return persist ? launch_one<false, true>(st, a, block, grid, buckets)
                   : launch_one<false, false>(st, a, block, grid, buckets);
}

int fill_u32(hipStream_t st, void *p, uint32_t v, size_t bytes)
{
    const uint32_t n = (uint32_t)(bytes / 4);
    hipLaunchKernelGGL(k_fill_u32, dim3(std::max(1u, std::min(64u, (n + 255) / 256))), dim3(256), 0, st,
                       reinterpret_cast<uint32_t *>(p), v, n);
    HIP_OK(hipGetLastError());
    return 0;
}
#define FILL(p, v, bytes)                                                                              \
    do {                                                                                               \
        const int fr_ = fill_u32(fst, (p), (v), (bytes));                                              \
        if (fr_) return fr_;                                                                           \
    } while (0)

int buckets_of(const galn_hip_readset *rs) { return std::max(1, std::min(rs->max_stacks, MAXB)); }

// threads per workgroup: the bucket tops of a workgroup must fit 64 KB of LDS
int pick_block(const galn_hip_readset *rs) { return buckets_of(rs) * 128 * 4 <= 65536 ? 128 : 64; }

// persistent grid: the workgroups that are resident at once
int resident_slots(galn_hip_readset *rs, int block, bool trace, int waves_per_cu)
{
    galn_hip_index *idx = rs->idx;
    if (waves_per_cu > 0) return std::max(block, idx->n_cu * waves_per_cu * 64 / block * block);
    int nb = 0;
    const size_t lds = (size_t)block * buckets_of(rs) * 4;
    hipError_t e = trace ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_search<true, true>, block, lds)
                         : hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_search<false, true>, block, lds);
    if (e != hipSuccess || nb < 1) nb = 1;
    return nb * idx->n_cu * block;
}

// Chains per thread and round of the wave engine: 2 (8.5 KB of LDS, 18 waves a CU) against 4 (12.6 KB, 12):
// 2M ancient DNA reads 217 ms against 233, 100k reads of 100 bp 7.5 against 8.9; one wave alone on a read
// runs faster with 4 (262,144 reads 83 ms against 77 without parking), which is what the workgroups that go
// on with parked reads take.
constexpr int HEAVY_CPL = 2;
constexpr int DEEP_NW = 4, DEEP_CPL = 4;
// A read may be parked after this many pops, where it can be expected to pop as many again: 100k pairs of
// 150 bp 39 ms (45 after 8192, 52 after 32768, 42 after 512), 2M ancient DNA reads 222 ms at any of them.
constexpr uint32_t PARK_POPS = 2048;
// With a wave for every read from the start nothing waits for the waves of the parked ones, and going on sooner
// only shortens the tail: 16 reads of 100 bp 0.54 ms after 512 pops, 0.64 after 2048, 0.59 after 256.
constexpr uint32_t PARK_POPS_FEW = 512;
constexpr int FIRST_GRAN = 8;  // granules a workgroup of it starts with
// Granules of the stack pool: POOL_FIRST for each wave's first read and POOL_READ for each read more, up to POOL_MOST
// (34 GB), or POOL_SEEDED where seeds keep the stacks small. It is the longest searches that take them, and more
// reads hold more of those: unseeded ones on a 3.1 Gbp human-like genome use 48k granules (4000 reads), 123k (20,000),
// 340k (60,000), 620k (200,000), 1.15M (2M; 1.84M with 16 waves a CU, where a first search with 1.05M ran dry, each
// granule sought in 64 shards, and took 14.4 s against 3.5); seeded ones 16k (2000) to 247k (1M repeat-rich ones of
// 250 bp). Not POOL_MOST for all: handing out and taking back 17 to 34 GB costs up to 2 s in some phases of the
// driver. 24 times an index opened, one search, closed, 100 bp, default options: of 2000 reads 13.0 s with 512 granules
// a wave and 0.06 so, of 6000 23.1 and 0.16, of 100,000 25.1 and 9.3.
constexpr uint64_t POOL_FIRST = 32, POOL_READ = 4, POOL_SEEDED = 1 << 19, POOL_MOST = 1 << 21;
constexpr int HEAVY_REC = 256;  // record slots of its waves in a search's first launch
constexpr int HEAVY_REC_MAX = 1 << 26;  // and in any (1.6 GB a wave; a slot's offsets are 32-bit)

struct HLayout {
    uint64_t slot_bytes;
    uint32_t rec_off, own_off, spill_off, state_off, plog_off, slog_off;
};

HLayout make_hlayout(int rec_cap, int own_cap, int nw, bool trace, bool wide, size_t state_bytes)
{
    HLayout L{};
    size_t off = 0;
    L.rec_off = 0;
    off += align_up((size_t)rec_cap * sizeof(galn_aln_rec_t), 256);
    L.own_off = (uint32_t)off;
    off += align_up((size_t)own_cap * 4, 256);
    L.spill_off = (uint32_t)off;
    off += align_up((size_t)own_cap * 4, 256);
    L.state_off = (uint32_t)off;
    off += align_up(state_bytes, 256);
    L.plog_off = (uint32_t)off;
    off += nw * heavy_log_bytes(wide);
    off = align_up(off, 16);
    L.slog_off = (uint32_t)off;
    if (trace) off += (size_t)nw * HW * H_SLOG * (sizeof(Ent) + 1);
    off = align_up(off, 256);
    if ((off / 256) % 2 == 0) off += 256;
    L.slot_bytes = off;
    return L;
}

// LDS of a workgroup of the wave engine, in the order k_heavy carves it up
size_t heavy_lds_bytes(int buckets, int wlen, int swlen, int nw, int cpl)
{
    return (size_t)H_PIECES * 16 + (size_t)nw * HW * cpl * heavy_chain_bytes + 16 * 8 + heavy_state_bytes(buckets, wlen, swlen) +
           H_STEPS * 2 + (size_t)wlen;
}

// A wave's scratch has room for the state of any read (5% of a slot): launches of other reads and options
// then fit what the first one allocated (a regrowth of this buffer frees some 2 GB, which waits for every
// stream of the device).
constexpr size_t HEAVY_STATE = heavy_state_bytes(MAXB, MAXLEN + 1, MAXLEN + 1);

size_t heavy_lds_of(const galn_hip_readset *rs, int nw, int cpl)
{
    const int swlen = (rs->seed_len > 0 && rs->seed_len < rs->max_len) ? rs->seed_len + 1 : 1;
    return heavy_lds_bytes(buckets_of(rs), rs->max_len + 1, swlen, nw, cpl);
}

typedef void (*HeavyKernel)(HArgs);

HeavyKernel heavy_kernel(bool wide, bool trace, bool deep)
{
    if (deep)
        return trace ? (wide ? k_heavy<true, true, DEEP_NW, DEEP_CPL> : k_heavy<true, false, DEEP_NW, DEEP_CPL>)
                     : (wide ? k_heavy<false, true, DEEP_NW, DEEP_CPL> : k_heavy<false, false, DEEP_NW, DEEP_CPL>);
    return trace ? (wide ? k_heavy<true, true, 1, HEAVY_CPL> : k_heavy<true, false, 1, HEAVY_CPL>)
                 : (wide ? k_heavy<false, true, 1, HEAVY_CPL> : k_heavy<false, false, 1, HEAVY_CPL>);
}

// Workgroups of the wave engine a CU holds.
int heavy_per_cu(galn_hip_readset *rs, uint32_t flags, bool deep, size_t lds)
{
    const void *const kernel = reinterpret_cast<const void *>(heavy_kernel(rs->idx->meta.ext != nullptr, (flags & GALN_HIP_TRACE) != 0, deep));
    int nb = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, (deep ? DEEP_NW : 1) * HW, lds);
    return e != hipSuccess || nb < 1 ? 1 : nb;
}

// The most workgroups that heavy_grid gives for any reads and options (that of the least LDS).
int heavy_grid_most(galn_hip_readset *rs, uint32_t flags, bool deep)
{
    return heavy_per_cu(rs, flags, deep, heavy_lds_bytes(1, 2, 1, deep ? DEEP_NW : 1, deep ? DEEP_CPL : HEAVY_CPL)) * rs->idx->n_cu;
}

// Workgroups of the wave engine that are resident at once.
int heavy_grid(galn_hip_readset *rs, uint32_t flags, bool deep)
{
    const int nw = deep ? DEEP_NW : 1, cpl = deep ? DEEP_CPL : HEAVY_CPL;
    const bool trace = (flags & GALN_HIP_TRACE) != 0;
    const void *const kernel = reinterpret_cast<const void *>(heavy_kernel(rs->idx->meta.ext != nullptr, trace, deep));
    const size_t lds = heavy_lds_of(rs, nw, cpl);
    auto &o = rs->occ[(trace ? 2 : 0) + (deep ? 1 : 0)];
    if (o.kernel != kernel || o.lds != lds) o = {kernel, lds, heavy_per_cu(rs, flags, deep, lds)};
    // Without seeds a read's stack, log and granules are several times larger, and those of 16 waves a CU go past L2:
    // 12 take 2M ancient DNA reads from 230 to 221 ms, 262,144 from 39.4 to 38.6, 100,003 repeat-rich ones from 105
    // to 101; 100k seeded reads of 100 bp take 4.1 ms with 16, 4.6 with 12, and few reads get a wave each (4001 take
    // 13.1 ms either way). From 2^32 symbols on, where every lookup leaves L2 as well, it depends on the reads: of
    // 30 to 150 bp, 2M on a 3.1 Gbp human-like genome take 3330 to 3480 ms with 16, 2860 to 3000 with 12, 2670 with 8,
    // 2580 with 6, 2690 with 4 (200,000 of them 309 to 330, 290, 283, 278, 295), while 1M of median 45, whose stacks
    // stay small, take 423 with 16, 444 with 12, 524 with 8. The line lies between their means, 90 and 48 bp.
    const bool many = !deep && rs->seed_len == 0 && rs->n >= 16 * o.groups * rs->idx->n_cu;
    const int most = !many ? o.groups : rs->idx->meta.ext == nullptr ? 12 : rs->qbytes >= (uint64_t)rs->n * 64 ? 8 : o.groups;
    return std::min(o.groups, most) * rs->idx->n_cu;
}

// A workgroup's first granules: FIRST_GRAN of them, fewer in a small pool (half of it is left to share).
int first_gran(const SearchCtx *cx, int groups)
{
    return (int)std::min<uint64_t>(FIRST_GRAN, cx->n_gran / 2 / (uint64_t)std::max(groups, 1));
}

// the wave-per-read engine keeps each chain's pops in order only when every child scores above its parent
bool heavy_ok(const galn_hip_readset *rs)
{
    for (const auto &o : rs->h_bopts)
        if (o.s_mm <= 0 || o.s_gapo <= 0 || o.s_gape <= 0) return false;
    return true;
}

KArgs base_args(galn_hip_readset *rs, uint32_t flags)
{
    KArgs a{};
    galn_hip_index *idx = rs->idx;
    a.bwt = idx->d_bwt;
    a.meta = idx->meta;
    a.query = rs->d_query;
    a.qoff = rs->d_qoff;
    a.qlen = rs->d_qlen;
    a.maxdiff = rs->d_maxdiff;
    a.batch = rs->d_batch;
    a.bopts = rs->d_bopts;
    a.nstacks = rs->d_nstacks;
    a.out_n = rs->d_out_n;
    a.out_off = rs->d_out_off;
    a.out_pops = rs->d_pops;
    a.out_trace = rs->d_trace;
    a.out_bytes = rs->d_bytes;
    a.out_rec = rs->d_rec;
    a.out_cap = rs->rec_cap;
    a.out_top = rs->d_top;
    a.pool_chk = rs->ctx->d_pool_chk;
    a.pool_link = rs->ctx->d_pool_link;
    a.gnext = rs->ctx->d_gnext;
    a.ghead = rs->ctx->d_ghead;
    a.gbump = rs->ctx->d_gbump;
    a.n_gran = rs->ctx->n_gran;
    // keeping the exact child in registers relies on children never scoring below their parent
    bool nonneg = true;
    for (const auto &o : rs->h_bopts) nonneg = nonneg && o.s_mm >= 0 && o.s_gapo >= 0 && o.s_gape >= 0;
    a.fuse = ((flags & GALN_HIP_NOFUSE) || !nonneg) ? 0 : 1;
    return a;
}

// One launch over list positions [0, n_list) (read id = list[pos], or list_base + pos);
// failures land in fail buffer `fo`.
// The allocations a first-tier launch over `slots` lanes needs (run before a graph capture).
int prepare_tier(galn_hip_readset *rs, const Tier &t, int slots, int pool_lanes)
{
    const int own_cap = (int)(((int64_t)(rs->max_entries + 16) / CH + MAXB + 2) / GRAN + 2);
    const Layout L = make_layout(rs->max_len, rs->seed_len, t.rec_cap, own_cap);
    int r = ensure_scratch(rs, (size_t)slots * L.slot_bytes);
    if (r) return r;
    // the pool for the lanes that get reads, rounded up to a power of two so that launches of
    // varying size regrow it a few times at most
    uint64_t want = (uint64_t)std::max(pool_lanes, 1) * (uint64_t)(t.keep + 12), p2 = 1024;
    while (p2 < want) p2 <<= 1;
    return ensure_pool(rs->ctx, p2);
}

// Bytes of scratch for the wave engine: `waves` workgroups of one wave, then the workgroups that go on with
// parked reads (which read the former's), `deep` of them at most.
size_t heavy_scratch(galn_hip_readset *rs, int waves, int deep, int rec_cap, uint32_t flags)
{
    const bool trace = (flags & GALN_HIP_TRACE) != 0, wide = rs->idx->meta.ext != nullptr;
    const int own_cap = (int)std::min<uint64_t>(rs->ctx->n_gran, 32768);
    const size_t one = (size_t)waves * make_hlayout(rec_cap, own_cap, 1, trace, wide, HEAVY_STATE).slot_bytes;
    return one + (size_t)std::min(waves, deep) * make_hlayout(0, 0, DEEP_NW, trace, wide, 0).slot_bytes;
}

// Granules of the pool for n reads on `waves` waves, rounded up to a power of two; `most` (one itself) at most.
uint64_t pool_granules(int waves, int n, uint64_t most)
{
    const uint64_t used = std::max(1, std::min(waves, n)), want = used * (POOL_FIRST - POOL_READ) + (uint64_t)std::max(n, 1) * POOL_READ;
    uint64_t p2 = 1024;
    while (p2 < std::min(want, most)) p2 <<= 1;
    return p2;
}

// Seeds that keep every read's stack small: no longer than 32 bases and with 3 differences at most (those measured).
bool pool_seeded(const galn_hip_readset *rs)
{
    for (const auto &o : rs->h_bopts)
        if (o.seed_len > 32 || o.max_seed_diff > 3) return false;
    return true;
}

// The allocations of a wave-engine launch of `waves` waves.
int prepare_heavy(galn_hip_readset *rs, int waves, int rec_cap, uint32_t flags)
{
    SearchCtx *cx = rs->ctx;
    int r = ensure_pool(cx, pool_granules(waves, rs->n, pool_seeded(rs) ? POOL_SEEDED : POOL_MOST));
    if (r) return r;
    if ((r = grow_dev((void **)&rs->d_park, rs->park_bytes, (size_t)waves * 4, cx->stream))) return r;
    return grow_dev((void **)&rs->d_hscratch, rs->hscratch_bytes, heavy_scratch(rs, waves, heavy_grid(rs, flags, true), rec_cap, flags), cx->stream);
}

// Hand-off slots for the widths of reads moving to the wave engine: one per read, up to
// HAND_BYTES or a quarter of the free device memory (reads beyond recompute their widths there,
// one lane walking the read while the wave waits). 10M unseeded reads of up to 150 bp, every read sent
// to the wave engine, need 22.6 GB with their root chains (127 words of a slot's 282) and 12.4 without,
// and where all reads fit only without, the chains are left out: a read then starts with one lane at
// work, but every read has its widths.
constexpr uint64_t HAND_BYTES = 32ull << 30;

// HAND_BYTES, or the value of GALN_HIP_TEST_HAND_BYTES, with which the tests leave slots out.
uint64_t hand_limit(const galn_hip_readset *rs, size_t freeb)
{
    const char *v = getenv("GALN_HIP_TEST_HAND_BYTES");
    const uint64_t most = v && *v ? strtoull(v, nullptr, 10) : HAND_BYTES;
    return std::min<uint64_t>(most, (uint64_t)(freeb + rs->hand_bytes) / 4);
}

int prepare_hand(galn_hip_readset *rs)
{
    const int sl = (rs->seed_len > 0 && rs->seed_len < rs->max_len) ? rs->seed_len : 0;
    int root = hand_root(rs->max_len, rs->idx->meta.ext != nullptr);
    uint32_t stride = hand_words(rs->max_len + 1, sl + 1, root);
    if (!getenv("GALN_HIP_TEST_HAND_BYTES") && rs->d_hand && rs->hand_bytes >= (uint64_t)std::max(rs->n, 1) * stride * 8) {
        rs->hand_stride = stride;
        rs->hand_root = root;
        rs->hand_cap = rs->n;
        return 0;
    }
    size_t freeb = 0, totalb = 0;
    HIP_OK(hipMemGetInfo(&freeb, &totalb));
    const uint64_t limit = hand_limit(rs, freeb);
    if ((uint64_t)rs->n * stride * 8 > limit) {
        root = 0;
        stride = hand_words(rs->max_len + 1, sl + 1, root);
    }
    const int cap = (int)std::min<uint64_t>((uint64_t)rs->n, limit / (stride * 8ull));
    // slots of this stride in the bytes already held (another launch's stride may differ)
    const size_t need = (size_t)std::max(cap, 1) * stride * 8;
    if (!rs->d_hand || rs->hand_bytes < need) {
        if (grow_dev((void **)&rs->d_hand, rs->hand_bytes, need, rs->ctx->stream)) {
            (void)hipGetLastError();
            g_err[0] = 0;
            rs->d_hand = nullptr;  // no hand-off: the wave engine computes the widths itself
            rs->hand_bytes = 0;
            rs->hand_cap = 0;
            return 0;
        }
    }
    rs->hand_stride = stride;
    rs->hand_root = root;
    rs->hand_cap = (int)std::min<uint64_t>((uint64_t)cap, rs->hand_bytes / (stride * 8ull));
    return 0;
}

// The batched form's buffers sized for launches of up to n reads of up to max_len bases: the
// hand-off slots, the stack pool and wave-engine scratch of min(grid, n) waves, the results' scan
// space and two staged records per read. Without it these grow by doubling as launches get larger
// (a server slot's launches vary in size), and each regrowth's hipFree waits for every stream of
// the device: on the 100 Mbp index a slot regrew ~30 times over its first 50 requests, frees of up
// to 190 ms, each holding the slot until the other slots' launches ended. Best effort: what does
// not fit is left to the searches, which allocate what they need.
int reserve_search(galn_hip_readset *rs, int n, int max_len, uint32_t flags)
{
    SearchCtx *cx = rs->ctx;
    hipStream_t s = cx->stream;
    n = std::max(n, 1);
    auto soft = [](int r) {
        if (r) (void)hipGetLastError(), g_err[0] = 0;
        return r;
    };
    // hand-off slots (seed widths of seeds up to 32 bases included), within prepare_hand's limit
    const uint64_t stride = hand_words(max_len + 1, 33, hand_root(max_len, rs->idx->meta.ext != nullptr));
    size_t freeb = 0, totalb = 0;
    HIP_OK(hipMemGetInfo(&freeb, &totalb));
    const uint64_t limit = hand_limit(rs, freeb);
    const uint64_t hand = std::min<uint64_t>((uint64_t)n, limit / (stride * 8)) * stride * 8;
    if (hand > rs->hand_bytes && soft(grow_dev((void **)&rs->d_hand, rs->hand_bytes, hand, s))) {
        rs->d_hand = nullptr;
        rs->hand_bytes = 0;
        rs->hand_cap = 0;
    }
    // the stack pool and the wave engine's per-wave scratch, as prepare_heavy sizes them for the reads and
    // options that get the most waves (this launch's may be fewer)
    const int waves = std::max(1, std::min(heavy_grid_most(rs, flags, false), n));
    if (!soft(ensure_pool(cx, pool_granules(waves, n, POOL_MOST)))) {
        soft(grow_dev((void **)&rs->d_park, rs->park_bytes, (size_t)waves * 4, s));
        soft(grow_dev((void **)&rs->d_hscratch, rs->hscratch_bytes, heavy_scratch(rs, waves, heavy_grid_most(rs, flags, true), HEAVY_REC, flags), s));
    }
    // the results: the record counts' scan over n reads and the staged records
    size_t tmp = 0;
    const rocprim::transform_iterator<const int32_t *, RecCount, uint64_t> cnt(rs->d_out_n, RecCount());
    HIP_OK(rocprim::inclusive_scan(nullptr, tmp, cnt, rs->d_incl, (size_t)n, rocprim::plus<uint64_t>(), s));
    soft(grow_dev(&rs->d_scan_tmp, rs->scan_tmp_bytes, tmp, s));
    soft(grow_dev((void **)&rs->d_stage, rs->stage_bytes, (size_t)2 * n * sizeof(galn_aln_rec_t), s));
    return 0;
}

// What a captured search graph holds: when any of it changes, the graph is captured again.
void fill_key_ptrs(const galn_hip_readset *rs, GraphKey &k)
{
    const void *p[] = {rs->d_query, rs->d_qoff, rs->d_qlen, rs->d_maxdiff, rs->d_batch, rs->d_nstacks, rs->d_bopts,
                       rs->d_sorted, rs->d_out_n, rs->d_out_off, rs->d_pops, rs->d_trace, rs->d_bytes, rs->d_rec,
                       rs->d_fail[0], rs->d_fail[1], rs->d_heavy, rs->d_park, rs->d_scratch, rs->d_hscratch, rs->ctx->d_pool_chk};
    static_assert(sizeof(p) == sizeof(k.ptr), "graph key pointers");
    memcpy(k.ptr, p, sizeof p);
    k.rec_cap_out = rs->rec_cap;
    k.n_gran = rs->ctx->n_gran;
    k.scratch_bytes = rs->scratch_bytes;
    k.hscratch_bytes = rs->hscratch_bytes;
    k.max_len = rs->max_len, k.seed_len = rs->seed_len, k.max_stacks = rs->max_stacks, k.max_entries = rs->max_entries;
    k.hand = rs->d_hand, k.hand_cap = rs->hand_cap, k.hand_stride = rs->hand_stride;
}

// A launch record of this search, its byte counter cleared, its two events ready.
int new_launch(galn_hip_readset *rs, int tier_id, int *li_out)
{
    const int li = (int)rs->launches.size();
    if (li >= galn_hip_readset::MAX_LAUNCH) return fail(GALN_HIP_E_DEVICE, "too many launches in one search");
    while ((int)rs->lev.size() < 2 * (li + 1)) {
        hipEvent_t e;
        HIP_OK(hipEventCreate(&e));
        rs->lev.push_back(e);
    }
    rs->launches.push_back({tier_id, li, 0.0, 0});
    *li_out = li;
    return 0;
}

int run_tier(galn_hip_readset *rs, uint32_t flags, const Tier &t, const int32_t *list, int list_base, int n_list,
             bool persist, int slots, int fo, int block, int tier_id, uint64_t pop_budget = 0)
{
    SearchCtx *cx = rs->ctx;
    hipStream_t fst = cx->stream;
    if (n_list <= 0) return 0;
    if (!persist) slots = n_list;
    // scratch and pool for every lane of a full persistent grid, also when this launch has fewer
    // reads, so that launches of varying size reuse them
    const int alloc_lanes = std::max(1, slots);
    slots = std::max(1, std::min(slots, n_list));
    const int own_cap = (int)(((int64_t)(rs->max_entries + 16) / CH + MAXB + 2) / GRAN + 2);
    Layout L = make_layout(rs->max_len, rs->seed_len, t.rec_cap, own_cap);
    // scratch, and a pool for what the lanes keep plus room for the heavy reads in flight
    int r = prepare_tier(rs, t, alloc_lanes, slots);
    if (r) return r;
    KArgs a = base_args(rs, flags);
    a.list = list;
    a.list_base = list_base;
    a.n_list = n_list;
    a.qnext = rs->d_ctr + 2;
    a.n_slots = slots;
    a.scratch = rs->d_scratch;
    a.slot_bytes = L.slot_bytes;
    a.sw_off = L.sw_off;
    a.rec_off = L.rec_off;
    a.own_off = L.own_off;
    a.own_cap = L.own_cap;
    a.keep = t.keep;
    a.rec_cap = t.rec_cap;
    a.fail_list = rs->d_fail[fo];
    a.fail_n = rs->d_ctr + fo;
    a.fail_kind = rs->d_ctr + 4;
    a.pop_budget = pop_budget;
    a.heavy_list = rs->d_heavy;
    a.heavy_n = rs->d_ctr + 3;
    a.hand = pop_budget ? rs->d_hand : nullptr;
    a.hand_stride = rs->hand_stride;
    a.hand_cap = (pop_budget && rs->d_hand) ? rs->hand_cap : 0;
    if (persist) FILL(rs->d_ctr + 2, 0, sizeof(int32_t));
    // an empty free stack (tag and granule all ones) and no granule handed out yet
    FILL(cx->d_ghead, 0xffffffffu, NSHARD * 8);
    FILL(cx->d_gbump, 0, 4);
    int li = 0;
    if ((r = new_launch(rs, tier_id, &li))) return r;
    a.algo_bytes = rs->d_algo + li;
    const int grid = (slots + block - 1) / block;
    if (!rs->capturing) HIP_OK(hipEventRecord(rs->lev[2 * li], fst));
    r = launch(fst, a, block, grid, persist, (flags & GALN_HIP_TRACE) != 0, buckets_of(rs));
    if (r) return r;
    if (!rs->capturing) HIP_OK(hipEventRecord(rs->lev[2 * li + 1], fst));
    return 0;
}

// Pushes the wave engine commits per round at most: what the logs hold, or a lower value (at least H_MINCAP;
// a round's first chain always fits) from GALN_HIP_TEST_PUSH_CAP, which the tests set to make the cap cut
// rounds short and check that the results do not change.
int heavy_push_cap()
{
    const char *v = getenv("GALN_HIP_TEST_PUSH_CAP");
    if (!v || !*v) return DEEP_NW * H_LOG;
    const long c = strtol(v, nullptr, 10);
    return (int)std::min<long>(DEEP_NW * H_LOG, std::max<long>(H_MINCAP, c));
}

// Pops from which on a read may be parked (0: never); `few`: every read has a wave of its own.
uint32_t heavy_park_pops(bool few)
{
    const char *v = getenv("GALN_HIP_TEST_PARK_POPS");
    return v && *v ? (uint32_t)strtoul(v, nullptr, 10) : few ? PARK_POPS_FEW : PARK_POPS;
}

int launch_widths(galn_hip_index *idx, hipStream_t st, const WArgs &w)
{
    const int64_t threads = 3 * ((int64_t)w.n_list + HW - 1) / HW * HW;
    const int grid = w.n_list_dev ? idx->n_cu * 8 : (int)std::max<int64_t>(1, std::min<int64_t>(idx->n_cu * 8, (threads + 255) / 256));
    if (idx->meta.ext)
        hipLaunchKernelGGL(k_widths<true>, dim3(grid), dim3(256), 0, st, w);
    else
        hipLaunchKernelGGL(k_widths<false>, dim3(grid), dim3(256), 0, st, w);
    HIP_OK(hipGetLastError());
    return 0;
}

// The widths of list[0..n) (n < 0: as many as k_search handed over) into the hand-off slots; `check`:
// those that k_search filled stay.
int launch_widths(galn_hip_readset *rs, const int32_t *list, int n, bool check)
{
    galn_hip_index *idx = rs->idx;
    WArgs w{};
    w.bwt = idx->d_bwt;
    w.meta = idx->meta;
    w.query = rs->d_query;
    w.qoff = rs->d_qoff;
    w.qlen = rs->d_qlen;
    w.batch = rs->d_batch;
    w.bopts = rs->d_bopts;
    w.list = list;
    w.n_list = std::max(n, 0);
    w.n_list_dev = n < 0 ? rs->d_ctr + 3 : nullptr;
    w.hand = rs->d_hand;
    w.hand_stride = rs->hand_stride;
    w.hand_cap = rs->hand_cap;
    w.root = rs->hand_root;
    w.wlen = rs->max_len + 1;
    w.swlen = (rs->seed_len > 0 && rs->seed_len < rs->max_len) ? rs->seed_len + 1 : 1;
    w.check = check ? 1 : 0;
    return launch_widths(idx, rs->ctx->stream, w);
}

// The wave-per-read engine over list[0..n): one wave per read, `waves` resident waves
// claiming reads from a device counter; failures land in fail buffer `fo`.
int run_heavy(galn_hip_readset *rs, uint32_t flags, const int32_t *list, int n, int rec_cap, int fo, int tier_id,
              int waves, bool widths_done = false)
{
    galn_hip_index *idx = rs->idx;
    SearchCtx *cx = rs->ctx;
    hipStream_t fst = cx->stream;
    const bool dev_count = n < 0;  // the count is the heavy-list length k_search leaves on the device
    if (n == 0) return 0;
    waves = std::max(1, dev_count ? waves : std::min(waves, n));
    const bool tr = (flags & GALN_HIP_TRACE) != 0, wide = idx->meta.ext != nullptr;
    int r = prepare_heavy(rs, waves, rec_cap, flags);
    if (r) return r;
    const int own_cap = (int)std::min<uint64_t>(cx->n_gran, 32768);
    const HLayout L = make_hlayout(rec_cap, own_cap, 1, tr, wide, HEAVY_STATE);
    const int wlen = rs->max_len + 1;
    const int swlen = (rs->seed_len > 0 && rs->seed_len < rs->max_len) ? rs->seed_len + 1 : 1;
    const size_t lds = heavy_lds_of(rs, 1, HEAVY_CPL);
    const size_t lds_deep = heavy_lds_of(rs, DEEP_NW, DEEP_CPL);
    if (std::max(lds, lds_deep) > 65536)
        return fail(GALN_HIP_E_UNSUPPORTED, "wave engine: %zu bytes of LDS needed", std::max(lds, lds_deep));
    const uint32_t park_pops = heavy_park_pops(!dev_count && n <= waves);
    HArgs a{};
    a.bwt = idx->d_bwt;
    a.meta = idx->meta;
    a.query = rs->d_query;
    a.qoff = rs->d_qoff;
    a.qlen = rs->d_qlen;
    a.maxdiff = rs->d_maxdiff;
    a.batch = rs->d_batch;
    a.bopts = rs->d_bopts;
    a.nstacks = rs->d_nstacks;
    a.list = list;
    a.n_list = dev_count ? 0 : n;
    a.n_list_dev = dev_count ? rs->d_ctr + 3 : nullptr;
    a.hand = rs->d_hand;  // the list is the heavy list of the k_search launch just before
    a.hand_stride = rs->hand_stride;
    a.hand_cap = rs->d_hand ? rs->hand_cap : 0;
    a.qnext = rs->d_ctr + 2;
    a.n_slots = waves;
    a.scratch = rs->d_hscratch;
    a.slot_bytes = L.slot_bytes;
    a.rec_off = L.rec_off;
    a.own_off = L.own_off;
    a.spill_off = L.spill_off;
    a.plog_off = L.plog_off;
    a.slog_off = L.slog_off;
    a.own_cap = own_cap;
    a.rec_cap = rec_cap;
    a.pool = cx->d_pool_chk;
    a.gnext = cx->d_gnext;
    a.ghead = cx->d_ghead;
    a.gbump = cx->d_gbump;
    a.n_gran = cx->n_gran;
    a.out_n = rs->d_out_n;
    a.out_off = rs->d_out_off;
    a.out_pops = rs->d_pops;
    a.out_trace = rs->d_trace;
    a.out_bytes = rs->d_bytes;
    a.out_rec = rs->d_rec;
    a.out_cap = rs->rec_cap;
    a.out_top = rs->d_top;
    a.fail_list = rs->d_fail[fo];
    a.fail_n = rs->d_ctr + fo;
    a.fail_kind = rs->d_ctr + 4;
    a.buckets = buckets_of(rs);
    a.wlen = wlen;
    a.push_cap = heavy_push_cap();
    a.swlen = swlen;
    a.stats = (flags & GALN_HIP_STATS) ? rs->d_stats : nullptr;
    a.park_pops = park_pops;
    a.park_list = rs->d_park;
    a.park_n = rs->d_ctr + 8;
    a.state_off = L.state_off;
    a.first_gran = first_gran(cx, waves);
    hipLaunchKernelGGL(k_reset_heavy, dim3(1), dim3(256), 0, fst, rs->d_ctr + 2, rs->d_ctr + 8, cx->d_ghead, cx->d_gbump,
                       (uint32_t)(a.first_gran * waves));
    HIP_OK(hipGetLastError());
    int li = 0;
    if ((r = new_launch(rs, tier_id, &li))) return r;
    a.algo_bytes = rs->d_algo + li;
    if (!rs->capturing) HIP_OK(hipEventRecord(rs->lev[2 * li], fst));
    if (a.hand && a.hand_cap > 0 && !widths_done && (r = launch_widths(rs, list, n, true))) return r;
    hipLaunchKernelGGL(heavy_kernel(wide, tr, false), dim3(waves), dim3(HW), lds, fst, a);
    if (park_pops) {
        // the reads still running when the last one was taken, with more waves each (their count is read on
        // the device; the workgroups end at once when there are none)
        HIP_OK(hipGetLastError());
        const int groups = std::min(waves, heavy_grid(rs, flags, true));
        const HLayout D = make_hlayout(0, 0, DEEP_NW, tr, wide, 0);
        HArgs d = a;
        d.n_list_dev = rs->d_ctr + 8;
        d.qnext = rs->d_ctr + 9;
        d.n_slots = groups;
        d.scratch = a.scratch + (size_t)waves * L.slot_bytes;
        d.slot_bytes = D.slot_bytes;
        d.plog_off = D.plog_off;
        d.slog_off = D.slog_off;
        d.park_pops = 0;
        d.park_scratch = a.scratch;
        d.park_slot_bytes = L.slot_bytes;
        d.park_rec_off = L.rec_off;
        d.park_own_off = L.own_off;
        d.park_spill_off = L.spill_off;
        d.park_state_off = L.state_off;
        hipLaunchKernelGGL(heavy_kernel(wide, tr, true), dim3(groups), dim3(DEEP_NW * HW), lds_deep, fst, d);
    }
    HIP_OK(hipGetLastError());
    if (!rs->capturing) HIP_OK(hipEventRecord(rs->lev[2 * li + 1], fst));
    return 0;
}

int read_ctr(galn_hip_readset *rs, int which, int32_t *v)
{
    HIP_OK(hipMemcpyAsync(v, rs->d_ctr + which, sizeof(int32_t), hipMemcpyDeviceToHost, rs->ctx->stream));
    HIP_OK(hipStreamSynchronize(rs->ctx->stream));
    return 0;
}

int grow_records(galn_hip_readset *rs)
{
    hipStream_t st = rs->ctx->stream;
    unsigned long long top = 0;
    HIP_OK(hipMemcpyAsync(&top, rs->d_top, sizeof(top), hipMemcpyDeviceToHost, st));
    HIP_OK(hipStreamSynchronize(st));
    const uint64_t used = std::min<uint64_t>(top, rs->rec_cap);
    const uint64_t ncap = std::max<uint64_t>(rs->rec_cap * 2, top + 4096);
    galn_aln_rec_t *nrec = nullptr;
    HIP_OK(dev_malloc(&nrec, ncap * sizeof(galn_aln_rec_t)));
    if (used) HIP_OK(hipMemcpyAsync(nrec, rs->d_rec, used * sizeof(galn_aln_rec_t), hipMemcpyDeviceToDevice, st));
    HIP_OK(hipStreamSynchronize(st));
    HIP_OK(hipFree(rs->d_rec));
    rs->d_rec = nrec;
    rs->rec_cap = ncap;
    unsigned long long u = used;
    HIP_OK(hipMemcpyAsync(rs->d_top, &u, sizeof(u), hipMemcpyHostToDevice, st));
    HIP_OK(hipStreamSynchronize(st));
    return 0;
}

// Re-run failed reads (fail buffer `fi`, count n) until none is left: a full output arena
// grows, full record slots get 16 times more, an exhausted pool gets fewer lanes sharing it.
// A read past `budget` pops ends in the wave engine, whose record slots grow with each such re-run
// from the 256 of the first launch; where that many for each wave would take more than half of
// the free memory, fewer waves run.
int run_retries(galn_hip_readset *rs, uint32_t flags, int fi, int32_t n, Tier t, int slots, uint64_t budget,
                int hwaves)
{
    hipStream_t fst = rs->ctx->stream;
    const int block = pick_block(rs);
    int heavy_rec = HEAVY_REC;
    for (int round = 0; n > 0; ++round) {
        if (round >= 24) return fail(GALN_HIP_E_NOMEM, "reads still failing after %d re-runs", round);
        int32_t kind[3] = {0, 0, 0};
        HIP_OK(hipMemcpy(kind, rs->d_ctr + 4, sizeof(kind), hipMemcpyDeviceToHost));
        int r;
        if (kind[0] && (r = grow_records(rs))) return r;
        if (kind[1]) {
            // (a lane hands a read on after `budget` pops, each of which gives one record at most)
            if (!budget || (uint64_t)t.rec_cap < budget) t.rec_cap *= 16;
            heavy_rec = std::min(heavy_rec * 16, HEAVY_REC_MAX);
        }
        if (kind[2]) {
            // an exhausted pool: twice the granules when there is room, else fewer lanes sharing it
            const uint32_t before = rs->ctx->n_gran;
            rs->ctx->grow = true;
            if ((r = ensure_pool(rs->ctx, before))) return r;
            if (rs->ctx->n_gran <= before) {
                slots = std::max(block, slots / 4);
                hwaves = std::max(1, hwaves / 4);
            }
        }
        slots = std::min(slots, std::max(block, (int)n));
        const int fo = fi ^ 1;
        FILL(rs->d_ctr + fo, 0, sizeof(int32_t));
        FILL(rs->d_ctr + 3, 0, 4 * sizeof(int32_t));
        if ((r = run_tier(rs, flags, t, rs->d_fail[fi], 0, n, true, slots, fo, block, 1 + round, budget))) return r;
        int32_t nh = 0;
        if ((r = read_ctr(rs, 3, &nh))) return r;
        if (nh > 0) {
            int waves = std::min(hwaves, (int)nh);
            size_t freeb = 0, totalb = 0;
            HIP_OK(hipMemGetInfo(&freeb, &totalb));
            while (waves > 1 && heavy_scratch(rs, waves, heavy_grid(rs, flags, true), heavy_rec, flags) > (freeb + rs->hscratch_bytes) / 2) waves /= 2;
            if ((r = run_heavy(rs, flags, rs->d_heavy, nh, heavy_rec, fo, 11 + round, waves))) return r;
        }
        int32_t nf = 0;
        if ((r = read_ctr(rs, fo, &nf))) return r;
        fi = fo;
        n = nf;
    }
    return 0;
}

// Pops after which the batched form hands a read to the wave-per-read engine when no tuning is given: 1,
// every read from the start, with its widths from k_widths. k_search's lanes take 6 us a pop on a read that is
// searched alone (16 reads of 100 bp: 3.0 ms to 512 pops, 0.5 ms in the wave engine) and its waves
// keep every lane until the last one is done (100k reads of 100 bp: 7.4 ms + 3.1 for the reads past 512
// pops, 7.2 ms in the wave engine; 262,144 ancient DNA reads: 20 ms + 39 against 39).
constexpr int DEFAULT_HEAVY_POPS = 1;

// The plain form's: its lanes wait for the slowest of 64 at 6 us a pop. 100k reads of 100 bp 31 ms without a
// limit, 8.8 after 512 pops, 7.2 after 128, 5.7 after 32, 5.5 after 16; 262,144 ancient DNA reads 67, 56, 51, 53.
constexpr int PLAIN_POPS = 32;

int readset_search(galn_hip_readset *rs, int form, uint32_t flags, const galn_hip_tune_t *tune)
{
    if (!tune && rs->has_tuned) tune = &rs->tuned;
    galn_hip_index *idx = rs->idx;
    HIP_OK(hipSetDevice(idx->device));
    hipStream_t fst = rs->ctx->stream;
    rs->last_flags = flags;
    rs->launches.clear();
    const bool trace = (flags & GALN_HIP_TRACE) != 0;
    const bool graph = form != 0 && (flags & GALN_HIP_GRAPH) != 0;
    auto prologue = [&]() -> int {
        hipLaunchKernelGGL(k_reset_search, dim3(1), dim3(256), 0, fst, rs->d_algo, (int)galn_hip_readset::MAX_LAUNCH, rs->d_stats,
                           rs->d_top, rs->d_ctr);
        HIP_OK(hipGetLastError());
        return 0;
    };
    if (!graph) {
        const int pr = prologue();
        if (pr) return pr;
    }
    int block = pick_block(rs);
    Tier t0{64, 4};
    if (tune && tune->rec_per_lane > 0) t0.rec_cap = tune->rec_per_lane;
    if (tune && tune->chunks_per_lane > 0) t0.keep = std::max(1, tune->chunks_per_lane / GRAN);
    int r = 0, slots = 0, hwaves = 0;
    uint64_t budget = 0;
    if (form == 0) {
        // plain: one launch per 0x40000 reads, one lane per read, input order; the reads past PLAIN_POPS pops then
        // get a wave each
        slots = 0x40000;
        budget = heavy_ok(rs) ? PLAIN_POPS : 0;
        hwaves = heavy_grid(rs, flags, false);
        if (budget && (r = prepare_hand(rs))) return r;
        for (int s = 0; s < rs->n && !r; s += 0x40000)
            r = run_tier(rs, flags, t0, nullptr, s, std::min(0x40000, rs->n - s), false, 0, 0, block, 0, budget);
        int32_t nh = 0;
        if (!r && budget && !(r = read_ctr(rs, 3, &nh)) && nh > 0) r = run_heavy(rs, flags, rs->d_heavy, nh, HEAVY_REC, 0, 10, hwaves);
    } else {
        // batched: one persistent launch over the reads, longest first; with a cutoff above 1 reads that
        // spend their pop budget go from k_search to the wave-per-read engine
        // 64-thread workgroups unless tuned otherwise (the autotuner's choice on every workload
        // measured so far)
        block = 64;
        if (tune && tune->block_threads > 0 && buckets_of(rs) * tune->block_threads * 4 <= 65536)
            block = tune->block_threads;
        const bool sorted = !tune || tune->sort_by_cost != 0;
        const int hp = tune ? tune->heavy_pops : 0;
        budget = (hp < 0 || !heavy_ok(rs)) ? 0 : (uint64_t)(hp > 0 ? hp : DEFAULT_HEAVY_POPS);
        hwaves = heavy_grid(rs, flags, false);
        if (budget && (r = prepare_hand(rs))) return r;
        const int32_t *list = sorted ? rs->d_sorted : nullptr;
        // every read to the wave engine: the widths launch stands in the place of k_search's
        const bool direct = budget == 1;
        slots = direct ? 0 : resident_slots(rs, block, trace, tune ? tune->waves_per_cu : 0);
        auto first_tier = [&]() -> int {
            if (!direct) return run_tier(rs, flags, t0, list, 0, rs->n, true, slots, 0, block, 0, budget);
            int li = 0, rc = new_launch(rs, 0, &li);
            if (rc) return rc;
            if (!rs->capturing) HIP_OK(hipEventRecord(rs->lev[2 * li], fst));
            if (rs->d_hand && rs->hand_cap > 0 && (rc = launch_widths(rs, list, rs->n, false))) return rc;
            if (!rs->capturing) HIP_OK(hipEventRecord(rs->lev[2 * li + 1], fst));
            return 0;
        };
        auto wave_tier = [&](int n) -> int {
            return direct ? run_heavy(rs, flags, list, rs->n, HEAVY_REC, 0, 10, hwaves, true)
                          : run_heavy(rs, flags, rs->d_heavy, n, HEAVY_REC, 0, 10, hwaves);
        };
        if (graph) {
            // the prologue, the persistent launch and the wave-engine launch (its read count read
            // on the device) as one captured graph, replayed while nothing it holds has changed
            GraphKey key;
            memset(&key, 0, sizeof key);  // padding included: keys are compared bytewise
            key.flags = flags, key.block = block, key.slots = slots, key.hwaves = hwaves, key.n = rs->n;
            key.budget = budget, key.rec_cap = (uint32_t)t0.rec_cap, key.keep = (uint32_t)t0.keep, key.list = list;
            key.push_cap = heavy_push_cap();
            key.park_pops = heavy_park_pops(direct && rs->n <= hwaves);
            if ((!direct && (r = prepare_tier(rs, t0, slots, std::min(slots, rs->n)))) ||
                (budget && (r = prepare_heavy(rs, hwaves, HEAVY_REC, flags))))
                return r;
            while (rs->lev.size() < 4) {
                hipEvent_t e;
                HIP_OK(hipEventCreate(&e));
                rs->lev.push_back(e);
            }
            fill_key_ptrs(rs, key);
            if (!rs->gexec || memcmp(&key, &rs->gkey, sizeof key) != 0) {
                for (hipGraphExec_t *ge : {&rs->gexec, &rs->gexec2}) {
                    if (*ge) HIP_OK(hipGraphExecDestroy(*ge));
                    *ge = nullptr;
                }
                // two graphs, so that the timing events sit between them rather than inside
                auto capture = [&](int part, hipGraphExec_t *out) -> int {
                    HIP_OK(hipStreamBeginCapture(fst, hipStreamCaptureModeThreadLocal));
                    rs->capturing = true;
                    int rc = 0;
                    if (part == 0) {
                        rc = prologue();
                        if (!rc) rc = first_tier();
                    } else {
                        rc = wave_tier(-1);
                    }
                    rs->capturing = false;
                    hipGraph_t g = nullptr;
                    const hipError_t ec = hipStreamEndCapture(fst, &g);
                    if (rc) {
                        if (g) (void)hipGraphDestroy(g);
                        return rc;
                    }
                    if (ec != hipSuccess) return fail(GALN_HIP_E_DEVICE, "graph capture: %s", hipGetErrorString(ec));
                    const hipError_t ei = hipGraphInstantiate(out, g, nullptr, nullptr, 0);
                    (void)hipGraphDestroy(g);
                    if (ei != hipSuccess) {
                        *out = nullptr;
                        return fail(GALN_HIP_E_DEVICE, "graph instantiate: %s", hipGetErrorString(ei));
                    }
                    return 0;
                };
                if ((r = capture(0, &rs->gexec))) return r;
                if (budget && (r = capture(1, &rs->gexec2))) return r;
                rs->gkey = key;
                rs->glaunches = rs->launches;
            }
            rs->launches = rs->glaunches;
            HIP_OK(hipEventRecord(rs->lev[0], fst));
            HIP_OK(hipGraphLaunch(rs->gexec, fst));
            HIP_OK(hipEventRecord(rs->lev[1], fst));
            if (rs->gexec2) {
                HIP_OK(hipEventRecord(rs->lev[2], fst));
                HIP_OK(hipGraphLaunch(rs->gexec2, fst));
                HIP_OK(hipEventRecord(rs->lev[3], fst));
            }
        } else {
            r = first_tier();
            int32_t nh = 0;
            if (!r && direct)
                r = wave_tier(rs->n);
            else if (!r && budget && !(r = read_ctr(rs, 3, &nh)) && nh > 0)
                r = wave_tier(nh);
        }
    }
    if (r) return r;
    // what the host needs of the search in one wait: the failures, the granules used, the launches' index bytes
    SearchBack *const back = rs->back;
    auto read_back = [&]() -> int {
        back->used = 0;
        HIP_OK(hipMemcpyAsync(&back->failed, rs->d_ctr, 4, hipMemcpyDeviceToHost, fst));
        if (rs->ctx->d_gbump) HIP_OK(hipMemcpyAsync(&back->used, rs->ctx->d_gbump, 4, hipMemcpyDeviceToHost, fst));
        if (!rs->launches.empty())
            HIP_OK(hipMemcpyAsync(back->algo, rs->d_algo, rs->launches.size() * 8, hipMemcpyDeviceToHost, fst));
        HIP_OK(hipStreamSynchronize(fst));
        return 0;
    };
    if ((r = read_back())) return r;
    if (back->failed > 0) {
        if (!slots) slots = resident_slots(rs, block, trace, tune ? tune->waves_per_cu : 0);
        if ((r = run_retries(rs, flags, 0, back->failed, t0, slots, budget, std::max(1, hwaves)))) return r;
        if ((r = read_back())) return r;
    }
    if (rs->ctx->d_gbump && back->used >= rs->ctx->n_gran) rs->ctx->grow = true;
    rs->first_ms = rs->total_ms = 0;
    for (size_t i = 0; i < rs->launches.size(); ++i) {
        float ms = 0;
        HIP_OK(hipEventElapsedTime(&ms, rs->lev[2 * i], rs->lev[2 * i + 1]));
        rs->launches[i].ms = ms;
        rs->launches[i].bytes = back->algo[i];
        if (rs->launches[i].tier == 0) rs->first_ms += ms;
        rs->total_ms += ms;
    }
    return 0;
}

int check_reads(const galn_hip_reads *r)
{
    if (!r || r->n_reads < 0) return fail(GALN_HIP_E_ARG, "reads: null or negative count");
    if (r->n_reads > 0 && (!r->query || !r->qoff || !r->qlen || !r->max_diff || !r->batch))
        return fail(GALN_HIP_E_ARG, "reads: null array");
    if (r->n_batches < 1 || !r->bopts || !r->n_stacks) return fail(GALN_HIP_E_ARG, "reads: no batch options");
    for (int b = 0; b < r->n_batches; ++b)
        if (r->bopts[b].seed_len < 0) return fail(GALN_HIP_E_UNSUPPORTED, "reads: negative seed length");
    for (int i = 0; i < r->n_reads; ++i)
        if (r->batch[i] < 0 || r->batch[i] >= r->n_batches) return fail(GALN_HIP_E_ARG, "reads: batch index out of range");
    return 0;
}

// Grow the per-read and per-batch device arrays to hold n reads, qbytes query bytes and nb
// batches (contents are not kept).
int readset_reserve(galn_hip_readset *rs, int n, uint64_t qbytes, int nb)
{
    const bool grow_n = n > rs->cap_n, grow_q = qbytes > rs->cap_q, grow_b = nb > rs->cap_b;
    if (!grow_n && !grow_q && !grow_b) return 0;
    HIP_OK(hipStreamSynchronize(rs->ctx->stream));
    auto regrow = [](void **p, size_t bytes) __attribute__((always_inline)) -> bool {
        if (*p) (void)hipFree(*p);
        *p = nullptr;
        return dev_malloc(p, std::max<size_t>(bytes, 16)) == hipSuccess;
    };
    bool ok = true;
    if (grow_q) {
        const uint64_t c = std::max<uint64_t>(qbytes, 2 * rs->cap_q);
        ok = regrow((void **)&rs->d_query, c + 16);
        rs->cap_q = ok ? c : 0;
    }
    if (ok && grow_b) {
        const int c = std::max(nb, 2 * rs->cap_b);
        ok = regrow((void **)&rs->d_nstacks, (size_t)c * 4) && regrow((void **)&rs->d_bopts, (size_t)c * sizeof(galn_search_opt_t));
        rs->cap_b = ok ? c : 0;
    }
    if (ok && grow_n) {
        const size_t c = (size_t)std::min<int64_t>(std::max<int64_t>(n, 2 * (int64_t)rs->cap_n), INT32_MAX);
        ok = regrow((void **)&rs->d_qoff, c * 8) && regrow((void **)&rs->d_qlen, c * 4) &&
             regrow((void **)&rs->d_maxdiff, c * 4) && regrow((void **)&rs->d_batch, c * 4) &&
             regrow((void **)&rs->d_sorted, c * 4) && regrow((void **)&rs->d_out_n, c * 4) &&
             regrow((void **)&rs->d_out_off, c * 8) && regrow((void **)&rs->d_pops, c * 8) &&
             regrow((void **)&rs->d_trace, c * 8) && regrow((void **)&rs->d_bytes, c * 8) &&
             regrow((void **)&rs->d_fail[0], c * 4) && regrow((void **)&rs->d_fail[1], c * 4) &&
             regrow((void **)&rs->d_heavy, c * 4) && regrow((void **)&rs->d_incl, c * 8) &&
             regrow((void **)&rs->d_roff, c * 8);
        rs->cap_n = ok ? (int)c : 0;
        if (ok && rs->rec_cap < 2 * c) {
            rs->rec_cap = std::max<uint64_t>(2 * c, 1 << 16);
            ok = regrow((void **)&rs->d_rec, rs->rec_cap * sizeof(galn_aln_rec_t));
            if (!ok) rs->rec_cap = 0;
        }
    }
    if (!ok) return fail(GALN_HIP_E_NOMEM, "readset: device allocation failed");
    return 0;
}

// Copy a read set (already checked) into rs's device arrays.
int readset_fill(galn_hip_readset *rs, const galn_hip_reads *reads)
{
    const int n = reads->n_reads;
    uint64_t qbytes = 0;
    int max_len = 1;
    for (int i = 0; i < n; ++i) {
        qbytes = std::max<uint64_t>(qbytes, reads->qoff[i] + (uint64_t)std::max(reads->qlen[i], 0));
        max_len = std::max(max_len, reads->qlen[i]);
    }
    int r = readset_reserve(rs, std::max(n, 1), qbytes, reads->n_batches);
    if (r) return r;
    rs->n = n;
    rs->n_batches = reads->n_batches;
    rs->max_len = std::min(max_len, MAXLEN);
    rs->qbytes = qbytes;
    // seed widths are kept for the longest seed that is shorter than some read
    rs->seed_len = 0;
    for (int b = 0; b < reads->n_batches; ++b)
        if (reads->bopts[b].seed_len < rs->max_len) rs->seed_len = std::max(rs->seed_len, reads->bopts[b].seed_len);
    rs->max_stacks = 1;
    for (int b = 0; b < reads->n_batches; ++b) rs->max_stacks = std::max(rs->max_stacks, reads->n_stacks[b]);
    rs->h_bopts.assign(reads->bopts, reads->bopts + reads->n_batches);
    rs->max_entries = 0;
    for (const auto &o : rs->h_bopts) rs->max_entries = std::max(rs->max_entries, std::max(o.max_entries, 0));
    // claim order of the batched form: longest reads first (their searches are the longest); a
    // counting sort by length (stable; lengths above the kernel limit share the top bin)
    std::vector<int32_t> order(n);
    {
        std::vector<int32_t> cnt(MAXLEN + 3, 0);
        auto bin = [&](int i) { return MAXLEN + 1 - std::min(std::max(reads->qlen[i], 0), MAXLEN + 1); };
        for (int i = 0; i < n; ++i) ++cnt[bin(i) + 1];
        for (int b = 1; b <= MAXLEN + 2; ++b) cnt[b] += cnt[b - 1];
        for (int i = 0; i < n; ++i) order[cnt[bin(i)]++] = i;
    }
    hipStream_t s = rs->ctx->stream;
    if (hipMemcpyAsync(rs->d_query, reads->query, qbytes, hipMemcpyHostToDevice, s) != hipSuccess ||
        hipMemcpyAsync(rs->d_qoff, reads->qoff, (size_t)n * 8, hipMemcpyHostToDevice, s) != hipSuccess ||
        hipMemcpyAsync(rs->d_qlen, reads->qlen, (size_t)n * 4, hipMemcpyHostToDevice, s) != hipSuccess ||
        hipMemcpyAsync(rs->d_maxdiff, reads->max_diff, (size_t)n * 4, hipMemcpyHostToDevice, s) != hipSuccess ||
        hipMemcpyAsync(rs->d_batch, reads->batch, (size_t)n * 4, hipMemcpyHostToDevice, s) != hipSuccess ||
        hipMemcpyAsync(rs->d_nstacks, reads->n_stacks, (size_t)reads->n_batches * 4, hipMemcpyHostToDevice, s) != hipSuccess ||
        hipMemcpyAsync(rs->d_bopts, reads->bopts, (size_t)reads->n_batches * sizeof(galn_search_opt_t),
                       hipMemcpyHostToDevice, s) != hipSuccess ||
        hipMemcpyAsync(rs->d_sorted, order.data(), (size_t)n * 4, hipMemcpyHostToDevice, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return fail(GALN_HIP_E_DEVICE, "readset: copy failed");
    return 0;
}

}  // namespace

extern "C" {

int galn_hip_abi_version(void) { return GALN_HIP_ABI_VERSION; }

void galn_hip_get_limits(galn_hip_limits_t *lim)
{
    if (!lim) return;
    lim->max_read_len = MAXLEN;
    lim->max_n_stacks = MAXB;
    lim->max_diff = MAXDIFF;
    lim->max_gapo_plus_gape = 255;
    lim->max_seq_len = KMASK;
}

const char *galn_hip_last_error(void) { return g_err; }

}  // extern "C"

// Used by the serving loop (galn_server.cpp), not exported: this thread's error text, and
// the count of handles that keep an index open.
__attribute__((visibility("hidden"))) void galn_hip_set_error(const char *msg) { snprintf(g_err, sizeof(g_err), "%s", msg); }
__attribute__((visibility("hidden"))) void galn_hip_index_hold(galn_hip_index *idx, int delta) { idx->n_readsets += delta; }
// A server's worker threads mark themselves; while a server is open on an index, only they may
// search it (its stream and stack pool are theirs).
thread_local bool tl_server_worker = false;
__attribute__((visibility("hidden"))) void galn_hip_server_worker_mark() { tl_server_worker = true; }
__attribute__((visibility("hidden"))) void galn_hip_index_serve(galn_hip_index *idx, int delta) { idx->n_servers += delta; }

// A server slot's read set gets a stream and a stack pool of its own, so that the slots' launches
// run at the same time (the read set was made on the index's context).
__attribute__((visibility("hidden"))) int galn_hip_readset_make_private(galn_hip_readset *rs)
{
    if (rs->own_ctx) return 0;
    HIP_OK(hipSetDevice(rs->idx->device));
    HIP_OK(hipStreamSynchronize(rs->ctx->stream));
    SearchCtx *c = new SearchCtx;
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
        delete c;
        return fail(GALN_HIP_E_DEVICE, "readset: stream creation failed");
    }
    // graphs captured on the old stream hold the old pool: captured again on first use
    for (hipGraphExec_t *ge : {&rs->gexec, &rs->gexec2}) {
        if (*ge) (void)hipGraphExecDestroy(*ge);
        *ge = nullptr;
    }
    rs->own_ctx = c;
    rs->ctx = c;
    return 0;
}

// Capacity for launches of up to n reads, qbytes query bytes and nb batches, allocated now (a
// server slot's read set, before its first launch fills it): later launches of up to that size
// then allocate nothing per read. The read set's contents are not kept.
__attribute__((visibility("hidden"))) int galn_hip_readset_reserve(galn_hip_readset *rs, int n, uint64_t qbytes, int nb)
{
    HIP_OK(hipSetDevice(rs->idx->device));
    return readset_reserve(rs, std::max(n, 1), qbytes, std::max(nb, 1));
}

// The search buffers of launches of up to n reads of up to max_len bases (the read set's arrays
// must already hold n reads: galn_hip_readset_reserve).
__attribute__((visibility("hidden"))) int galn_hip_readset_reserve_search(galn_hip_readset *rs, int n, int max_len,
                                                                          uint32_t flags)
{
    HIP_OK(hipSetDevice(rs->idx->device));
    if (n > rs->cap_n) return fail(GALN_HIP_E_ARG, "readset_reserve_search: %d reads, the arrays hold %d", n, rs->cap_n);
    return reserve_search(rs, n, max_len, flags);
}

namespace {
int noalloc_setup(int device);

int busy_check(const galn_hip_index *idx, const char *what)
{
    if (idx && idx->n_servers.load() > 0 && !tl_server_worker)
        return fail(GALN_HIP_E_BUSY, "%s: a server holds this index until galn_hip_server_close", what);
    return 0;
}
}  // namespace

extern "C" {

int galn_hip_index_open(const uint32_t *bwt, const galn_bwt_meta_t *meta, int device, galn_hip_index **out)
{
    if (!bwt || !meta || !out) return fail(GALN_HIP_E_ARG, "index_open: null argument");
    *out = nullptr;
    if (meta->seq_len > KMASK) return fail(GALN_HIP_E_UNSUPPORTED, "index of %llu symbols exceeds 2^38-1",
                                           (unsigned long long)meta->seq_len);
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return fail(GALN_HIP_E_DEVICE, "no HIP device");
    if (device < 0 || device >= ndev) return fail(GALN_HIP_E_DEVICE, "no HIP device %d (%d visible)", device, ndev);
    HIP_OK(hipSetDevice(device));
    galn_hip_index *idx = new galn_hip_index;
    idx->device = device;
    idx->hmeta = *meta;
    idx->meta.primary = meta->primary;
    idx->meta.seq_len = meta->seq_len;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) {
        delete idx;
        return fail(GALN_HIP_E_DEVICE, "hipGetDeviceProperties failed");
    }
    idx->n_cu = prop.multiProcessorCount;
    const size_t bytes = (size_t)meta->bwt_size * 4;
    // whole 64-byte blocks are loaded: pad so the last block's load stays in bounds
    const size_t alloc = align_up(bytes + 256, 256);
    if (dev_malloc(&idx->d_bwt, alloc) != hipSuccess) {
        delete idx;
        return fail(GALN_HIP_E_NOMEM, "index of %zu bytes does not fit in device memory", bytes);
    }
    if (hipStreamCreateWithFlags(&idx->ctx0.stream, hipStreamNonBlocking) != hipSuccess ||
        hipMemsetAsync(idx->d_bwt, 0, alloc, idx->ctx0.stream) != hipSuccess ||
        hipMemcpyAsync(idx->d_bwt, bwt, bytes, hipMemcpyHostToDevice, idx->ctx0.stream) != hipSuccess) {
        if (idx->ctx0.stream) (void)hipStreamDestroy(idx->ctx0.stream);
        (void)hipFree(idx->d_bwt);
        delete idx;
        return fail(GALN_HIP_E_DEVICE, "index upload failed");
    }
    // 32-bit counts reach 2^32 - 1 (row seq_len + 1 included); a larger index counts per epoch of 2^24
    // blocks. GALN_HIP_TEST_EPOCH=n makes the epochs 2^n blocks on an index of any size (tests).
    Totals T;
    for (int c = 0; c < 5; ++c) T.L2[c] = meta->L2[c];
    T.end = meta->seq_len % 128 == 0 ? meta->seq_len / 128 : ~0ull;
    // (the end's block may lie past the body, within the allocation's padding)
    uint64_t n_blocks = ((uint64_t)meta->bwt_size + 15) / 16;
    if (T.end == n_blocks) n_blocks += 1;
    uint32_t eshift = 24;
    bool wide = meta->seq_len >= 0xfffffffeull;
    if (const char *v = getenv("GALN_HIP_TEST_EPOCH"); v && *v) {
        eshift = (uint32_t)std::min(24L, std::max(1L, strtol(v, nullptr, 10)));
        wide = true;
    }
    const uint32_t n_ep = wide ? (uint32_t)((n_blocks >> eshift) + 1) : 1u;
    bool up = dev_malloc(&idx->d_ext, (size_t)n_ep * 32) == hipSuccess;
    if (up && n_blocks > 0) {
        hipLaunchKernelGGL(k_epochs, dim3((4 * n_ep + 255) / 256), dim3(256), 0, idx->ctx0.stream, (const uint32_t *)idx->d_bwt, n_blocks,
                           eshift, T, idx->d_ext, n_ep);
        hipLaunchKernelGGL(k_planes, dim3((unsigned)((n_blocks + 255) / 256)), dim3(256), 0, idx->ctx0.stream, idx->d_bwt,
                           n_blocks, T, (const uint64_t *)idx->d_ext, eshift, wide ? 1 : 0);
    }
    if (!up || hipGetLastError() != hipSuccess || hipStreamSynchronize(idx->ctx0.stream) != hipSuccess) {
        (void)hipStreamDestroy(idx->ctx0.stream);
        (void)hipFree(idx->d_bwt);
        if (idx->d_ext) (void)hipFree(idx->d_ext);
        delete idx;
        return fail(GALN_HIP_E_DEVICE, "index upload failed");
    }
    idx->meta.ext = wide ? idx->d_ext : nullptr;
    idx->meta.eshift = eshift;
    // device address of the no-allocation search's array on this device (once per device); a
    // failure here is reported by that entry point, which looks it up again
    if (noalloc_setup(device) != 0) g_err[0] = 0;
    *out = idx;
    return 0;
}

int galn_hip_index_close(galn_hip_index *idx)
{
    if (!idx) return 0;
    if (idx->n_readsets.load() > 0)
        return fail(GALN_HIP_E_BUSY, "index_close: %d read sets (or servers) of this index are still open",
                    idx->n_readsets.load());
    (void)hipSetDevice(idx->device);
    if (idx->ctx0.stream) (void)hipStreamSynchronize(idx->ctx0.stream);
    (void)hipFree(idx->d_bwt);
    if (idx->d_ext) (void)hipFree(idx->d_ext);
    if (idx->d_sa) (void)hipFree(idx->d_sa);
    idx->ctx0.free_pool();
    if (idx->ctx0.stream) (void)hipStreamDestroy(idx->ctx0.stream);
    delete idx;
    return 0;
}

int galn_hip_index_device(const galn_hip_index *idx) { return idx ? idx->device : -1; }

int galn_hip_readset_free(galn_hip_readset *rs)
{
    if (!rs) return 0;
    (void)hipSetDevice(rs->idx->device);
    (void)hipStreamSynchronize(rs->ctx->stream);
    void *ptrs[] = {rs->d_query, rs->d_qoff, rs->d_qlen, rs->d_maxdiff, rs->d_batch, rs->d_nstacks, rs->d_bopts,
                    rs->d_sorted, rs->d_out_n, rs->d_out_off, rs->d_pops, rs->d_trace, rs->d_bytes, rs->d_rec, rs->d_top,
                    rs->d_fail[0], rs->d_fail[1], rs->d_ctr, rs->d_scratch, rs->d_algo, rs->d_heavy, rs->d_park, rs->d_hscratch,
                    rs->d_stats, rs->d_incl, rs->d_roff, rs->d_stage, rs->d_scan_tmp, rs->d_hand};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    if (rs->back) g_backs.give(rs->back);
    for (auto &e : rs->ev)
        if (e) (void)hipEventDestroy(e);
    for (auto &e : rs->lev) (void)hipEventDestroy(e);
    if (rs->gexec) (void)hipGraphExecDestroy(rs->gexec);
    if (rs->gexec2) (void)hipGraphExecDestroy(rs->gexec2);
    if (rs->own_ctx) {
        rs->own_ctx->free_pool();
        if (rs->own_ctx->stream) (void)hipStreamDestroy(rs->own_ctx->stream);
        delete rs->own_ctx;
    }
    rs->idx->n_readsets.fetch_sub(1);
    delete rs;
    return 0;
}

int galn_hip_readset_upload(galn_hip_index *idx, const galn_hip_reads *reads, galn_hip_readset **out)
{
    if (!idx || !out) return fail(GALN_HIP_E_ARG, "readset_upload: null argument");
    *out = nullptr;
    int r = busy_check(idx, "readset_upload");
    if (r) return r;
    if ((r = check_reads(reads))) return r;
    HIP_OK(hipSetDevice(idx->device));
    galn_hip_readset *rs = new galn_hip_readset;
    rs->idx = idx;
    rs->ctx = &idx->ctx0;
    idx->n_readsets.fetch_add(1);
    auto M = [&](void **p, size_t b) __attribute__((always_inline)) -> bool { return dev_malloc(p, b) == hipSuccess; };
    bool ok = M((void **)&rs->d_top, 8) && M((void **)&rs->d_ctr, 16 * sizeof(int32_t)) && M((void **)&rs->d_stats, 16 * 8) &&
              M((void **)&rs->d_algo, sizeof(unsigned long long) * galn_hip_readset::MAX_LAUNCH) && (rs->back = g_backs.take());
    if (!ok) {
        galn_hip_readset_free(rs);
        return fail(GALN_HIP_E_NOMEM, "readset_upload: device allocation failed");
    }
    for (auto &e : rs->ev)
        if (hipEventCreate(&e) != hipSuccess) {
            galn_hip_readset_free(rs);
            return fail(GALN_HIP_E_DEVICE, "hipEventCreate failed");
        }
    if ((r = readset_fill(rs, reads))) {
        galn_hip_readset_free(rs);
        return r;
    }
    *out = rs;
    return 0;
}

int galn_hip_readset_reload(galn_hip_readset *rs, const galn_hip_reads *reads)
{
    if (!rs) return fail(GALN_HIP_E_ARG, "readset_reload: null handle");
    int r = busy_check(rs->idx, "readset_reload");
    if (r) return r;
    if ((r = check_reads(reads))) return r;
    HIP_OK(hipSetDevice(rs->idx->device));
    return readset_fill(rs, reads);
}

int galn_hip_readset_search(galn_hip_index *idx, galn_hip_readset *rs, int form, uint32_t flags,
                            const galn_hip_tune_t *tune)
{
    if (!idx || !rs || rs->idx != idx) return fail(GALN_HIP_E_ARG, "readset_search: bad handle");
    const int b = busy_check(idx, "readset_search");
    if (b) return b;
    if (rs->n == 0) return 0;
    return readset_search(rs, form, flags, tune);
}

int galn_hip_readset_autotune(galn_hip_index *idx, galn_hip_readset *rs, uint32_t flags, galn_hip_tune_t *out)
{
    if (!idx || !rs || rs->idx != idx) return fail(GALN_HIP_E_ARG, "readset_autotune: bad handle");
    const int b = busy_check(idx, "readset_autotune");
    if (b) return b;
    rs->has_tuned = false;
    galn_hip_tune_t best{};
    best.sort_by_cost = 1;
    const bool verbose = galn_hip_verbose();
    if (rs->n > 0) {
        double best_ms = 0;
        auto trial = [&](const galn_hip_tune_t &t) -> int {
            const auto t0 = std::chrono::steady_clock::now();
            const int r = readset_search(rs, 1, flags, &t);
            if (r) return r;
            const double ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
            if (verbose)
                fprintf(stderr, "[galn_hip] autotune: cutoff %d, %d-thread groups, %d waves/CU, %d record slots, "
                                "%d chunks kept: %.1f ms\n",
                        t.heavy_pops, t.block_threads, t.waves_per_cu, t.rec_per_lane, t.chunks_per_lane, ms);
            if (best_ms == 0 || ms < best_ms) {
                best_ms = ms;
                best = t;
            }
            return 0;
        };
        // the thread-vs-wave cutoff first (when the wave engine may run), then, where k_search runs, the
        // workgroup size, then one change at a time from the best so far: the persistent grid's waves
        // per CU, the record slots per lane, and the stack chunks a lane keeps between reads
        galn_hip_tune_t t{};
        t.sort_by_cost = 1;
        t.block_threads = 128;
        // a search before the trials: the buffers that one allocates are not the first candidate's (on 100k reads of
        // 100 bp the cutoff 1 lost to 16 for them, 4.9 ms a search against 5.9)
        if (const int rw = readset_search(rs, 1, flags, nullptr)) return rw;
        // (1: every read goes to the wave engine, k_search is not launched)
        const int cut[] = {1, 16, 64, 128, 256, 512, 1024, 4096};
        int r;
        if (heavy_ok(rs)) {
            for (int c : cut) {
                t.heavy_pops = c;
                if ((r = trial(t))) return r;
            }
        } else {
            t.heavy_pops = -1;
            if ((r = trial(t))) return r;
        }
        if (best.heavy_pops == 1) {
            best.block_threads = 64;  // (the library's own; this and the remaining settings are k_search's)
        } else {
            t = best;
            t.block_threads = 64;
            if ((r = trial(t))) return r;
            const int waves[] = {4, 6}, recs[] = {16, 256}, keeps[] = {GRAN, 16 * GRAN};
            for (int v : waves) {
                t = best;
                t.waves_per_cu = v;
                if ((r = trial(t))) return r;
            }
            for (int v : recs) {
                t = best;
                t.rec_per_lane = v;
                if ((r = trial(t))) return r;
            }
            for (int v : keeps) {
                t = best;
                t.chunks_per_lane = v;
                if ((r = trial(t))) return r;
            }
        }
    }
    rs->tuned = best;
    rs->has_tuned = true;
    if (out) *out = best;
    return 0;
}

int galn_hip_readset_results(galn_hip_readset *rs, galn_hip_out *out)
{
    if (!rs || !out || (rs->n > 0 && (!out->n_aln || !out->rec_off)))
        return fail(GALN_HIP_E_ARG, "readset_results: null argument");
    galn_hip_index *idx = rs->idx;
    const int b = busy_check(idx, "readset_results");
    if (b) return b;
    HIP_OK(hipSetDevice(idx->device));
    const int n = rs->n;
    if (n == 0) {
        out->n_rec = 0;
        return 0;
    }
    hipStream_t s = rs->ctx->stream;
    // records in read order, arranged on the device: offsets = prefix sums of the record counts
    // (errors count 0), then every read's records gathered from the arena
    size_t tmp_bytes = 0;
    const rocprim::transform_iterator<const int32_t *, RecCount, uint64_t> cnt(rs->d_out_n, RecCount());
    HIP_OK(rocprim::inclusive_scan(nullptr, tmp_bytes, cnt, rs->d_incl, (size_t)n, rocprim::plus<uint64_t>(), s));
    if (int g = grow_dev(&rs->d_scan_tmp, rs->scan_tmp_bytes, tmp_bytes, s)) return g;
    HIP_OK(rocprim::inclusive_scan(rs->d_scan_tmp, tmp_bytes, cnt, rs->d_incl, (size_t)n, rocprim::plus<uint64_t>(), s));
    unsigned long long need = 0;
    HIP_OK(hipMemcpyAsync(&need, rs->d_incl + (n - 1), 8, hipMemcpyDeviceToHost, s));
    HIP_OK(hipMemcpyAsync(out->n_aln, rs->d_out_n, (size_t)n * 4, hipMemcpyDeviceToHost, s));
    if (out->n_pops) HIP_OK(hipMemcpyAsync(out->n_pops, rs->d_pops, (size_t)n * 8, hipMemcpyDeviceToHost, s));
    if (out->trace) HIP_OK(hipMemcpyAsync(out->trace, rs->d_trace, (size_t)n * 8, hipMemcpyDeviceToHost, s));
    if (out->occ_bytes) HIP_OK(hipMemcpyAsync(out->occ_bytes, rs->d_bytes, (size_t)n * 8, hipMemcpyDeviceToHost, s));
    HIP_OK(hipStreamSynchronize(s));
    out->n_rec = need;
    if (need > out->rec_cap || (need > 0 && !out->rec))
        return fail(GALN_HIP_E_RECCAP, "record array holds %llu, %llu needed", (unsigned long long)out->rec_cap,
                    (unsigned long long)need);
    if (int g = grow_dev((void **)&rs->d_stage, rs->stage_bytes, std::max<uint64_t>(need, 1) * sizeof(galn_aln_rec_t), s))
        return g;
    hipLaunchKernelGGL(k_gather_records, dim3((n + 255) / 256), dim3(256), 0, s, rs->d_out_n, rs->d_out_off,
                       (const uint64_t *)rs->d_incl, (const galn_aln_rec_t *)rs->d_rec, rs->d_stage, rs->d_roff, n);
    HIP_OK(hipGetLastError());
    HIP_OK(hipMemcpyAsync(out->rec_off, rs->d_roff, (size_t)n * 8, hipMemcpyDeviceToHost, s));
    if (need) HIP_OK(hipMemcpyAsync(out->rec, rs->d_stage, need * sizeof(galn_aln_rec_t), hipMemcpyDeviceToHost, s));
    HIP_OK(hipStreamSynchronize(s));
    return 0;
}

int galn_hip_readset_kernel_ms(const galn_hip_readset *rs, double *first_tier_ms, double *total_ms)
{
    if (!rs) return fail(GALN_HIP_E_ARG, "readset_kernel_ms: null handle");
    if (first_tier_ms) *first_tier_ms = rs->first_ms;
    if (total_ms) *total_ms = rs->total_ms;
    return 0;
}

int galn_hip_readset_engine_stats(galn_hip_readset *rs, uint64_t out[16])
{
    if (!rs || !out) return fail(GALN_HIP_E_ARG, "readset_engine_stats: null argument");
    HIP_OK(hipMemcpy(out, rs->d_stats, 16 * 8, hipMemcpyDeviceToHost));
    return 0;
}

int galn_hip_readset_launches(const galn_hip_readset *rs, int cap, int32_t *tier, double *ms, uint64_t *algo_bytes)
{
    if (!rs) return fail(GALN_HIP_E_ARG, "readset_launches: null handle");
    const int n = (int)rs->launches.size();
    for (int i = 0; i < n && i < cap; ++i) {
        if (tier) tier[i] = rs->launches[i].tier;
        if (ms) ms[i] = rs->launches[i].ms;
        if (algo_bytes) algo_bytes[i] = rs->launches[i].bytes;
    }
    return n;
}

static int search_once(galn_hip_index *idx, const galn_hip_reads *reads, galn_hip_out *out, int form, uint32_t flags,
                       const galn_hip_tune_t *tune)
{
    galn_hip_readset *rs = nullptr;
    int r = galn_hip_readset_upload(idx, reads, &rs);
    if (r) return r;
    r = galn_hip_readset_search(idx, rs, form, flags, tune);
    if (!r) r = galn_hip_readset_results(rs, out);
    galn_hip_readset_free(rs);
    return r;
}

int galn_hip_search_plain(galn_hip_index *idx, const galn_hip_reads *reads, galn_hip_out *out, uint32_t flags)
{
    return search_once(idx, reads, out, 0, flags, nullptr);
}

int galn_hip_search_batched(galn_hip_index *idx, const galn_hip_reads *reads, galn_hip_out *out, uint32_t flags,
                            const galn_hip_tune_t *tune)
{
    return search_once(idx, reads, out, 1, flags, tune);
}

}  // extern "C"

extern "C" {

int galn_hip_index_set_sa(galn_hip_index *idx, const uint64_t *samples, uint64_t n_samples, uint32_t intv)
{
    if (!idx || (!samples && n_samples)) return fail(GALN_HIP_E_ARG, "index_set_sa: null argument");
    int r = busy_check(idx, "index_set_sa");
    if (r) return r;
    if (intv == 0 || (intv & (intv - 1)) != 0) return fail(GALN_HIP_E_ARG, "index_set_sa: interval %u is not a power of 2", intv);
    const uint64_t want = (idx->hmeta.seq_len + intv) / intv - 1;
    if (n_samples != want)
        return fail(GALN_HIP_E_ARG, "index_set_sa: %llu samples, %llu expected for interval %u",
                    (unsigned long long)n_samples, (unsigned long long)want, intv);
    HIP_OK(hipSetDevice(idx->device));
    if (idx->d_sa) HIP_OK(hipFree(idx->d_sa));
    idx->d_sa = nullptr;
    idx->n_sa = 0;
    HIP_OK(dev_malloc(&idx->d_sa, std::max<uint64_t>(n_samples, 1) * 8));
    if (n_samples) HIP_OK(hipMemcpy(idx->d_sa, samples, n_samples * 8, hipMemcpyHostToDevice));
    idx->n_sa = n_samples;
    idx->sa_intv = intv;
    return 0;
}

int galn_hip_sa_positions(galn_hip_index *idx, const uint64_t *rows, uint64_t n, uint64_t *pos, const int32_t *ref_len,
                          int32_t *strand)
{
    if (!idx || (n && (!rows || !pos)) || (!ref_len != !strand))
        return fail(GALN_HIP_E_ARG, "sa_positions: null argument (ref_len and strand come together)");
    int r = busy_check(idx, "sa_positions");
    if (r) return r;
    if (!idx->sa_intv) return fail(GALN_HIP_E_ARG, "sa_positions: no SA samples (galn_hip_index_set_sa)");
    for (uint64_t i = 0; i < n; ++i)
        if (rows[i] > idx->hmeta.seq_len)
            return fail(GALN_HIP_E_ARG, "sa_positions: row %llu beyond %llu", (unsigned long long)rows[i],
                        (unsigned long long)idx->hmeta.seq_len);
    if (n == 0) return 0;
    HIP_OK(hipSetDevice(idx->device));
    const uint64_t chunk = std::min<uint64_t>(n, 1ull << 24);
    uint64_t *d = nullptr;
    HIP_OK(dev_malloc(&d, chunk * (ref_len ? 24 : 16)));
    int32_t *const d_rl = ref_len ? reinterpret_cast<int32_t *>(d + 2 * chunk) : nullptr;
    int32_t *const d_st = ref_len ? d_rl + chunk : nullptr;
    hipStream_t s = idx->ctx0.stream;
    int rc = 0;
    for (uint64_t a = 0; a < n && !rc; a += chunk) {
        const uint64_t m = std::min(chunk, n - a);
        if (hipMemcpyAsync(d, rows + a, m * 8, hipMemcpyHostToDevice, s) != hipSuccess ||
            (ref_len && hipMemcpyAsync(d_rl, ref_len + a, m * 4, hipMemcpyHostToDevice, s) != hipSuccess)) {
            rc = fail(GALN_HIP_E_DEVICE, "sa_positions: copy failed");
            break;
        }
        hipLaunchKernelGGL(k_sa_walk, dim3((unsigned)std::min<uint64_t>((m + 255) / 256, 65535)), dim3(256), 0, s,
                           (const uint32_t *)idx->d_bwt, idx->meta, (const uint64_t *)idx->d_sa, (uint64_t)idx->sa_intv,
                           (const uint64_t *)d, m, d + chunk, (const int32_t *)d_rl, d_st);
        if (hipGetLastError() != hipSuccess ||
            hipMemcpyAsync(pos + a, d + chunk, m * 8, hipMemcpyDeviceToHost, s) != hipSuccess ||
            (ref_len && hipMemcpyAsync(strand + a, d_st, m * 4, hipMemcpyDeviceToHost, s) != hipSuccess) ||
            hipStreamSynchronize(s) != hipSuccess)
            rc = fail(GALN_HIP_E_DEVICE, "sa_positions: kernel or copy failed");
    }
    (void)hipFree(d);
    return rc;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Search without allocation (galn_hip_search_device_noalloc). Every buffer the search needs
// beyond the caller's inputs and outputs -- counters, failure lists, per-batch options, the
// lanes' regions (widths, record slots, granule lists) and the stack pool -- is carved out of
// one static device array, `scratch`, which each GPU holds from the library's first use on it
// until the process ends. Host code never passes the array's name to a kernel: its device
// address on each GPU comes from hipGetSymbolAddress, taken once per device (with that device
// current) when the first index is opened there.

namespace {
constexpr size_t NA_SCRATCH_BYTES = 256ull << 20;  // the array's size
constexpr int NA_MAX_READS = 1 << 20;              // reads per call
constexpr int NA_MAX_BATCHES = 4096;               // per-batch option sets per call
constexpr int NA_MAX_DEVICES = 64;
constexpr int NA_PARK = 24;  // counters of parked reads, in the i32 at the array's start
}  // namespace

static __device__ __align__(256) uint8_t scratch[NA_SCRATCH_BYTES];

namespace {

uint8_t *g_na_ptr[NA_MAX_DEVICES];  // device address of `scratch` on each device
std::mutex g_na_setup_mu;
std::mutex g_na_mu[NA_MAX_DEVICES];  // calls on one device take turns (they share its array)

// Looks up the device address of `scratch` on `device`, which must be current. Idempotent.
int noalloc_setup(int device)
{
    if (device < 0 || device >= NA_MAX_DEVICES) return fail(GALN_HIP_E_DEVICE, "device %d beyond %d", device, NA_MAX_DEVICES);
    std::lock_guard<std::mutex> lk(g_na_setup_mu);
    if (g_na_ptr[device]) return 0;
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
        (void)hipGetLastError();
        return fail(GALN_HIP_E_DEVICE, "scratch array of device %d: hipGetSymbolAddress: %s", device,
                    hipGetErrorString(e));
    }
    g_na_ptr[device] = static_cast<uint8_t *>(p);
    return 0;
}

// Longest read (capped at MAXLEN + 1) and the number of reads whose batch index is out of range.
__global__ void k_na_scan(const int32_t *qlen, const int32_t *batch, int n, int n_batches, int32_t *res)
{
    int mx = 0, bad = 0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        mx = max(mx, min(qlen[i], MAXLEN + 1));
        bad += (batch[i] < 0 || batch[i] >= n_batches) ? 1 : 0;
    }
    if (mx > 0) atomicMax(res, mx);
    if (bad) atomicAdd(res + 1, bad);
}

// Offsets inside the array.
struct NaLayout {
    size_t ctr, top, algo, scan, ghead, gbump, bopts, nstacks, fail0, fail1, pops, lanes;
};

NaLayout na_layout()
{
    NaLayout L{};
    L.ctr = 0;      // 8 x i32: [0],[1] failure counts, [2] claim counter, [3] unused, [4..6] failure kinds
    L.top = 64;     // u64 records reserved in the caller's array
    L.algo = 72;    // u64 algorithmic index bytes
    L.scan = 80;    // 2 x i32 (k_na_scan); from 96 (NA_PARK) 2 x i32, the parked reads and their claim counter
    L.ghead = 256;  // NSHARD x u64 free-granule stack heads
    L.gbump = L.ghead + NSHARD * 8;
    size_t off = align_up(L.gbump + 4, 256);
    L.bopts = off;
    off = align_up(off + (size_t)NA_MAX_BATCHES * sizeof(galn_search_opt_t), 256);
    L.nstacks = off;
    off = align_up(off + (size_t)NA_MAX_BATCHES * 4, 256);
    L.fail0 = off;
    off += (size_t)NA_MAX_READS * 4;
    L.fail1 = off;
    off += (size_t)NA_MAX_READS * 4;
    L.pops = off;  // pop counts when the caller does not ask for them
    off += (size_t)NA_MAX_READS * 8;
    L.lanes = align_up(off, 256);
    return L;
}

// k_fill's counterpart for the first list of reads: 0, 1, 2, ...
__global__ void k_iota(int32_t *p, int n)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = i;
}

// The array's split for the wave engine. A lane of k_search needs two granules of pool, so 4096 lanes -- 64
// waves on 256 CUs -- filled it, each lane on its read until the last pop; the wave engine's 512 waves each have
// their log (128 KB) and some ten granules, reads take hand-off slots for their widths in turns of what
// NA_HAND_BYTES hold, and NA_DEEP workgroups go on with parked reads: 30k reads of 100 bp 57 -> 7.0 ms.
constexpr int NA_WAVES = 512;
constexpr int NA_DEEP = 32;
constexpr size_t NA_HAND_BYTES = 32ull << 20;

// The array's bytes, or fewer: GALN_HIP_TEST_NA_BYTES, with which the tests reach its limits.
size_t na_bytes()
{
    const char *v = getenv("GALN_HIP_TEST_NA_BYTES");
    return v && *v ? std::min<size_t>(NA_SCRATCH_BYTES, strtoull(v, nullptr, 10)) : NA_SCRATCH_BYTES;
}

// Record slots of a wave at most: three eighths of the array (4,194,304 records), beside which one wave's pool fits.
int na_rec_max() { return (int)(na_bytes() * 3 / 8 / sizeof(galn_aln_rec_t)); }

struct NaWaves {
    int waves = 0, groups = 0, turn = 0, own_cap = 0;  // turn: reads per launch
    uint64_t n_gran = 0;
    HLayout L, D;
    size_t park, hand, slots, deep, pool, gnext;  // offsets
};

// At most `want` waves, halved until each has 12 granules (the last one: whatever is left, at least 32).
// waves = 0: not even one fits.
NaWaves na_waves(int want, int n, uint32_t hand_stride, int rec_cap, bool trace, bool wide, size_t state_bytes)
{
    NaWaves N;
    for (int w = std::max(1, want);; w = w > 1 ? w / 2 : 0) {
        if (w == 0) return N;
        N.own_cap = w > 16 ? 1024 : 16384;
        N.L = make_hlayout(rec_cap, N.own_cap, 1, trace, wide, state_bytes);
        N.D = make_hlayout(0, 0, DEEP_NW, trace, wide, 0);
        N.groups = std::min(w, NA_DEEP);
        N.turn = (int)std::min<uint64_t>((uint64_t)n, std::max<uint64_t>(1, NA_HAND_BYTES / (hand_stride * 8ull)));
        const int turns = (n + N.turn - 1) / N.turn;
        N.turn = (n + turns - 1) / turns;
        N.park = na_layout().lanes;
        N.hand = align_up(N.park + (size_t)w * 4, 256);
        N.slots = align_up(N.hand + (size_t)N.turn * hand_stride * 8, 256);
        N.deep = N.slots + (size_t)w * N.L.slot_bytes;
        N.pool = N.deep + (size_t)N.groups * N.D.slot_bytes;
        if (N.pool + 256 >= na_bytes()) continue;
        N.n_gran = (na_bytes() - N.pool - 256) / (GENT * sizeof(Ent) + 4);
        if (N.n_gran < (w > 1 ? 12ull * (uint64_t)w : 32ull)) continue;
        N.gnext = N.pool + N.n_gran * GENT * sizeof(Ent);
        N.waves = w;
        return N;
    }
}

// Bytes of one pool granule with its chunk links and free-stack link.
constexpr size_t NA_GRAN_BYTES = (size_t)GRAN * CH * sizeof(Ent) + (size_t)GRAN * 4 + 4;

// Lanes that fit the array beside the pool with their region of `slot_bytes`: at most `want`,
// each with at least two granules of pool. Returns 0 if not even one fits.
int na_lanes(size_t slot_bytes, int want, uint64_t *n_gran)
{
    const size_t avail = NA_SCRATCH_BYTES - na_layout().lanes - 3 * 256;
    for (int lanes = std::max(1, want);; lanes = lanes > 1 ? lanes / 2 : 0) {
        if (lanes == 0) return 0;
        const size_t region = align_up((size_t)lanes * slot_bytes, 256);
        if (region >= avail) continue;
        const uint64_t g = std::min<uint64_t>((avail - region) / NA_GRAN_BYTES, MAX_POOL_CHUNKS / GRAN);
        if (g >= 2ull * (uint64_t)lanes) {
            *n_gran = g;
            return lanes;
        }
    }
}

int noalloc_search(galn_hip_index *idx, const galn_hip_reads *reads, galn_hip_out *out, uint32_t flags)
{
    if (!idx || !reads || !out) return fail(GALN_HIP_E_ARG, "search_device_noalloc: null argument");
    const int n = reads->n_reads;
    if (n < 0 || n > NA_MAX_READS)
        return fail(GALN_HIP_E_ARG, "search_device_noalloc: %d reads (at most %d per call)", n, NA_MAX_READS);
    if (reads->n_batches < 1 || reads->n_batches > NA_MAX_BATCHES || !reads->bopts || !reads->n_stacks)
        return fail(GALN_HIP_E_ARG, "search_device_noalloc: %d batches (1 to %d, with host option arrays)",
                    reads->n_batches, NA_MAX_BATCHES);
    for (int b = 0; b < reads->n_batches; ++b)
        if (reads->bopts[b].seed_len < 0) return fail(GALN_HIP_E_UNSUPPORTED, "reads: negative seed length");
    const bool trace = (flags & GALN_HIP_TRACE) != 0;
    if (n > 0 && (!reads->query || !reads->qoff || !reads->qlen || !reads->max_diff || !reads->batch ||
                  !out->n_aln || !out->rec_off || (out->rec_cap > 0 && !out->rec) || (trace && !out->trace)))
        return fail(GALN_HIP_E_ARG, "search_device_noalloc: null array");
    int r = busy_check(idx, "search_device_noalloc");
    if (r) return r;
    HIP_OK(hipSetDevice(idx->device));
    if ((r = noalloc_setup(idx->device))) return r;
    std::lock_guard<std::mutex> lk(g_na_mu[idx->device]);
    out->n_rec = 0;
    if (n == 0) return 0;

    uint8_t *const S = g_na_ptr[idx->device];
    const NaLayout NL = na_layout();
    int32_t *const ctr = reinterpret_cast<int32_t *>(S + NL.ctr);
    unsigned long long *const top = reinterpret_cast<unsigned long long *>(S + NL.top);
    unsigned long long *const algo = reinterpret_cast<unsigned long long *>(S + NL.algo);
    int32_t *const scan = reinterpret_cast<int32_t *>(S + NL.scan);
    unsigned long long *const ghead = reinterpret_cast<unsigned long long *>(S + NL.ghead);
    uint32_t *const gbump = reinterpret_cast<uint32_t *>(S + NL.gbump);
    galn_search_opt_t *const d_bopts = reinterpret_cast<galn_search_opt_t *>(S + NL.bopts);
    int32_t *const d_nstacks = reinterpret_cast<int32_t *>(S + NL.nstacks);
    int32_t *const d_fail[2] = {reinterpret_cast<int32_t *>(S + NL.fail0), reinterpret_cast<int32_t *>(S + NL.fail1)};
    uint64_t *const d_pops = out->n_pops ? out->n_pops : reinterpret_cast<uint64_t *>(S + NL.pops);
    hipStream_t st = idx->ctx0.stream, fst = st;

    // per-batch options in, counters cleared (fill kernels: the array keeps the last call's contents)
    const int nb = reads->n_batches;
    HIP_OK(hipMemcpyAsync(d_bopts, reads->bopts, (size_t)nb * sizeof(galn_search_opt_t), hipMemcpyHostToDevice, st));
    HIP_OK(hipMemcpyAsync(d_nstacks, reads->n_stacks, (size_t)nb * 4, hipMemcpyHostToDevice, st));
    FILL(S, 0, 256);  // counters, record top, byte count, scan results
    FILL(out->rec_off, 0, (size_t)n * 8);
    hipLaunchKernelGGL(k_na_scan, dim3(std::min(1024, (n + 255) / 256)), dim3(256), 0, st, reads->qlen, reads->batch, n,
                       nb, scan);
    HIP_OK(hipGetLastError());
    int32_t hs[2] = {0, 0};
    HIP_OK(hipMemcpyAsync(hs, scan, sizeof hs, hipMemcpyDeviceToHost, st));
    HIP_OK(hipStreamSynchronize(st));
    if (hs[1] > 0) return fail(GALN_HIP_E_ARG, "reads: %d batch indexes out of range", hs[1]);

    // what readset_fill derives from the reads
    const int max_len = std::max(1, std::min(hs[0], MAXLEN));
    int seed_len = 0, max_stacks = 1, max_entries = 0;
    bool nonneg = true, positive = true;
    for (int b = 0; b < nb; ++b) {
        const galn_search_opt_t &o = reads->bopts[b];
        if (o.seed_len < max_len) seed_len = std::max(seed_len, o.seed_len);
        max_stacks = std::max(max_stacks, reads->n_stacks[b]);
        max_entries = std::max(max_entries, std::max(o.max_entries, 0));
        nonneg = nonneg && o.s_mm >= 0 && o.s_gapo >= 0 && o.s_gape >= 0;
        positive = positive && o.s_mm > 0 && o.s_gapo > 0 && o.s_gape > 0;
    }
    const int buckets = std::max(1, std::min(max_stacks, MAXB));
    const bool wide = idx->meta.ext != nullptr;
    const int wlen = max_len + 1, swlen = seed_len > 0 && seed_len < max_len ? seed_len + 1 : 1;
    const size_t lds = heavy_lds_bytes(buckets, wlen, swlen, 1, HEAVY_CPL), lds_deep = heavy_lds_bytes(buckets, wlen, swlen, DEEP_NW, DEEP_CPL);
    const bool engine = positive && std::max(lds, lds_deep) <= 65536;
    const int block = buckets * 128 * 4 <= 65536 ? 128 : 64;
    const int own_full = (int)(((int64_t)(max_entries + 16) / CH + MAXB + 2) / GRAN + 2);

    KArgs a{};
    a.bwt = idx->d_bwt;
    a.meta = idx->meta;
    a.query = reads->query;
    a.qoff = reads->qoff;
    a.qlen = reads->qlen;
    a.maxdiff = reads->max_diff;
    a.batch = reads->batch;
    a.bopts = d_bopts;
    a.nstacks = d_nstacks;
    a.qnext = ctr + 2;
    a.fail_kind = ctr + 4;
    a.algo_bytes = algo;
    a.out_n = out->n_aln;
    a.out_off = out->rec_off;
    a.out_pops = d_pops;
    a.out_trace = out->trace;
    a.out_bytes = out->occ_bytes;
    a.out_rec = out->rec;
    a.out_cap = out->rec_cap;
    a.out_top = top;
    a.ghead = ghead;
    a.gbump = gbump;
    a.fuse = ((flags & GALN_HIP_NOFUSE) || !nonneg) ? 0 : 1;
    a.heavy_n = ctr + 3;  // no pop budget: nothing is handed on

    int rec_cap = engine ? HEAVY_REC : 64, want = std::min(n, engine ? NA_WAVES : 4096), fi = 0;
    int32_t n_todo = n;
    bool out_full = false;
    if (engine) {
        fi = 1;
        hipLaunchKernelGGL(k_iota, dim3(std::min(1024, (n + 255) / 256)), dim3(256), 0, st, d_fail[1], n);
        HIP_OK(hipGetLastError());
    }
    for (int round = 0; n_todo > 0; ++round) {
        if (round >= 24) return fail(GALN_HIP_E_NOMEM, "search_device_noalloc: reads still failing after %d re-runs", round);
        if (engine) {
            // the wave engine over d_fail[fi][0..n_todo), a turn of reads after the other
            const int root = hand_root(max_len, wide);
            const uint32_t stride = hand_words(wlen, swlen, root);
            const NaWaves N = na_waves(std::min(want, (int)n_todo), n_todo, stride, rec_cap, trace, wide, heavy_state_bytes(buckets, wlen, swlen));
            if (N.waves == 0)
                return fail(GALN_HIP_E_UNSUPPORTED, "search_device_noalloc: a wave's regions and its pool do not fit in %zu bytes", na_bytes());
            const int fo = fi ^ 1;
            FILL(ctr + fo, 0, sizeof(int32_t));
            FILL(ctr + 4, 0, 3 * sizeof(int32_t));
            for (int at = 0; at < n_todo; at += N.turn) {
                const int m = std::min(N.turn, (int)n_todo - at);
                WArgs w{};
                w.bwt = idx->d_bwt;
                w.meta = idx->meta;
                w.query = reads->query;
                w.qoff = reads->qoff;
                w.qlen = reads->qlen;
                w.batch = reads->batch;
                w.bopts = d_bopts;
                w.list = d_fail[fi] + at;
                w.n_list = m;
                w.hand = reinterpret_cast<uint64_t *>(S + N.hand);
                w.hand_stride = stride;
                w.hand_cap = m;
                w.root = root;
                w.wlen = wlen;
                w.swlen = swlen;
                if ((r = launch_widths(idx, st, w))) return r;
                HArgs h{};
                h.bwt = w.bwt;
                h.meta = w.meta;
                h.query = w.query;
                h.qoff = w.qoff;
                h.qlen = w.qlen;
                h.maxdiff = reads->max_diff;
                h.batch = w.batch;
                h.bopts = d_bopts;
                h.nstacks = d_nstacks;
                h.list = w.list;
                h.n_list = m;
                h.hand = w.hand;
                h.hand_stride = stride;
                h.hand_cap = m;
                h.qnext = ctr + 2;
                h.n_slots = std::min(N.waves, m);
                h.scratch = S + N.slots;
                h.slot_bytes = N.L.slot_bytes;
                h.rec_off = N.L.rec_off;
                h.own_off = N.L.own_off;
                h.spill_off = N.L.spill_off;
                h.plog_off = N.L.plog_off;
                h.slog_off = N.L.slog_off;
                h.own_cap = N.own_cap;
                h.rec_cap = rec_cap;
                h.pool = reinterpret_cast<Ent *>(S + N.pool);
                h.gnext = reinterpret_cast<uint32_t *>(S + N.gnext);
                h.ghead = ghead;
                h.gbump = gbump;
                h.n_gran = (uint32_t)N.n_gran;
                h.first_gran = (int)std::min<uint64_t>(FIRST_GRAN, N.n_gran / 2 / (uint64_t)N.waves);
                h.out_n = out->n_aln;
                h.out_off = out->rec_off;
                h.out_pops = d_pops;
                h.out_trace = out->trace;
                h.out_bytes = out->occ_bytes;
                h.out_rec = out->rec;
                h.out_cap = out->rec_cap;
                h.out_top = top;
                h.fail_list = d_fail[fo];
                h.fail_n = ctr + fo;
                h.fail_kind = ctr + 4;
                h.algo_bytes = algo;
                h.buckets = buckets;
                h.wlen = wlen;
                h.swlen = swlen;
                h.push_cap = heavy_push_cap();
                h.park_pops = heavy_park_pops(m <= N.waves);
                h.park_list = reinterpret_cast<int32_t *>(S + N.park);
                h.park_n = ctr + NA_PARK;
                h.state_off = N.L.state_off;
                hipLaunchKernelGGL(k_reset_heavy, dim3(1), dim3(256), 0, st, ctr + 2, ctr + NA_PARK, ghead, gbump,
                                   (uint32_t)(h.first_gran * h.n_slots));
                HIP_OK(hipGetLastError());
                hipLaunchKernelGGL(heavy_kernel(wide, trace, false), dim3(h.n_slots), dim3(HW), lds, st, h);
                HIP_OK(hipGetLastError());
                if (h.park_pops) {
                    HArgs d = h;
                    d.n_list_dev = ctr + NA_PARK;
                    d.qnext = ctr + NA_PARK + 1;
                    d.n_slots = std::min(N.groups, h.n_slots);
                    d.scratch = S + N.deep;
                    d.slot_bytes = N.D.slot_bytes;
                    d.plog_off = N.D.plog_off;
                    d.slog_off = N.D.slog_off;
                    d.park_pops = 0;
                    d.park_scratch = h.scratch;
                    d.park_slot_bytes = N.L.slot_bytes;
                    d.park_rec_off = N.L.rec_off;
                    d.park_own_off = N.L.own_off;
                    d.park_spill_off = N.L.spill_off;
                    d.park_state_off = N.L.state_off;
                    hipLaunchKernelGGL(heavy_kernel(wide, trace, true), dim3(d.n_slots), dim3(DEEP_NW * HW), lds_deep, st, d);
                    HIP_OK(hipGetLastError());
                }
            }
            int32_t c[8];
            HIP_OK(hipMemcpyAsync(c, ctr, sizeof c, hipMemcpyDeviceToHost, st));
            HIP_OK(hipStreamSynchronize(st));
            if (c[4]) {  // the caller's record array is full: stop, and report what was reserved
                out_full = true;
                break;
            }
            if (c[5] && rec_cap >= na_rec_max())
                return fail(GALN_HIP_E_UNSUPPORTED, "search_device_noalloc: a read has more than %d records", na_rec_max());
            if (c[5]) rec_cap = std::min(rec_cap * 16, na_rec_max());
            if (c[6]) want = std::max(1, N.waves / 4);
            fi = fo;
            n_todo = c[fo];
            continue;
        }
        const Layout L0 = make_layout(max_len, seed_len, rec_cap, own_full);
        uint64_t n_gran = 0;
        const int lanes = na_lanes(L0.slot_bytes, std::min(want, (int)n_todo), &n_gran);
        if (lanes == 0)
            return fail(GALN_HIP_E_UNSUPPORTED, "search_device_noalloc: a lane's %llu bytes and its pool do not fit in %zu bytes",
                        (unsigned long long)L0.slot_bytes, NA_SCRATCH_BYTES);
        const int own_cap = (int)std::min<uint64_t>((uint64_t)own_full, n_gran);
        const Layout L = make_layout(max_len, seed_len, rec_cap, own_cap);
        uint8_t *const lanes_base = S + NL.lanes;
        uint8_t *const pool = S + align_up(NL.lanes + (size_t)lanes * L.slot_bytes, 256);
        a.scratch = lanes_base;
        a.slot_bytes = L.slot_bytes;
        a.sw_off = L.sw_off;
        a.rec_off = L.rec_off;
        a.own_off = L.own_off;
        a.own_cap = L.own_cap;
        a.keep = 1;
        a.rec_cap = rec_cap;
        a.pool_chk = reinterpret_cast<Ent *>(pool);
        a.pool_link = reinterpret_cast<uint32_t *>(pool + align_up(n_gran * GRAN * CH * sizeof(Ent), 256));
        a.gnext = reinterpret_cast<uint32_t *>(reinterpret_cast<uint8_t *>(a.pool_link) + align_up(n_gran * GRAN * 4, 256));
        a.n_gran = (uint32_t)n_gran;
        a.list = round == 0 ? nullptr : d_fail[fi];
        a.list_base = 0;
        a.n_list = n_todo;
        a.n_slots = lanes;
        const int fo = round == 0 ? 0 : fi ^ 1;
        a.fail_list = d_fail[fo];
        a.fail_n = ctr + fo;
        FILL(ctr + fo, 0, sizeof(int32_t));
        FILL(ctr + 2, 0, 2 * sizeof(int32_t));
        FILL(ctr + 4, 0, 3 * sizeof(int32_t));
        FILL(ghead, 0xffffffffu, NSHARD * 8);
        FILL(gbump, 0, 4);
        r = launch(st, a, block, (lanes + block - 1) / block, true, trace, buckets);
        if (r) return r;
        int32_t c[8];
        HIP_OK(hipMemcpyAsync(c, ctr, sizeof c, hipMemcpyDeviceToHost, st));
        HIP_OK(hipStreamSynchronize(st));
        if (c[4]) {  // the caller's record array is full: stop, and report what was reserved
            out_full = true;
            break;
        }
        if (c[5]) rec_cap *= 16;
        if (c[6]) want = std::max(1, lanes / 4);
        fi = fo;
        n_todo = c[fo];
    }
    unsigned long long t = 0;
    HIP_OK(hipMemcpyAsync(&t, top, sizeof t, hipMemcpyDeviceToHost, st));
    HIP_OK(hipStreamSynchronize(st));
    out->n_rec = t;
    if (out_full)
        return fail(GALN_HIP_E_RECCAP, "search_device_noalloc: record array holds %llu; at least %llu needed",
                    (unsigned long long)out->rec_cap, t);
    return 0;
}

}  // namespace

extern "C" int galn_hip_search_device_noalloc(galn_hip_index *idx, const galn_hip_reads *reads, galn_hip_out *out,
                                              uint32_t flags)
{
    return noalloc_search(idx, reads, out, flags);
}
