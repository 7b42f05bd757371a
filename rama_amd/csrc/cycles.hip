// cycles.hip — conflicted 3-, 4- and 5-cycle search and triangulation
// (src/conflicted_cycles_cuda.cu:13-343, include/rama_utils.h:62-84,296-363).
//
// A conflicted cycle is one repulsive edge (v1, v2) closed by a path of
// attractive edges.  Each stage enumerates "expansions" and intersects two
// sorted attractive neighbour lists per expansion:
//   3-cycles: expansion = rep edge r;                 N(v1) ∩ N(v2)
//   4-cycles: expansion = (r, n1 ∈ N(v1));            N(n1) ∩ N(v2)
//   5-cycles: expansion = (r, n1 ∈ N(v1), n2 ∈ N(v2)); N(n1) ∩ N(n2), n1≠n2
// and writes 1, 2 or 3 triangles per common neighbour `mid`.
//
// Deterministic output order (the reference's atomic slot counter is
// replaced): a count pass stores each expansion's number of mids (uint8,
// saturating) and exact per-tile totals; a scan of the tile totals gives
// every tile its write offset; an emit pass revisits only expansions with
// mids and writes at enumeration position (rep edge, expansion, mid).  The
// triangle budget therefore keeps exactly the first `budget` writes.
#include <cstdlib>
#include <cstring>
#include <optional>

#include "rama_internal.hpp"
#include "tuning.hpp"

namespace rama {

constexpr int kCycTile = kBlock;  // expansions per block

struct CycArgs {
    const int* off;      // attractive CSR offsets (n+1)
    const int* adj;      // attractive CSR neighbours
    const int* rv1;      // repulsive edge rows (v1 < v2)
    const int* rv2;
    const i64* xoff;     // per-rep exclusive expansion offsets (R+1)
    const int* tile_rep; // first rep edge of each tile
    i64 R;
    i64 X;               // number of expansions
    // Several instances packed in one graph (disjoint node ranges): nslot
    // maps a node to its instance; the count kernels add each instance's
    // attempted writes to slot_total, and the emit kernel places instance q's
    // writes at slot_out[q] + slot_base[q] + (global position - slot_first[q]),
    // keeping those below slot_budget[q].  All null for a single instance.
    const int* nslot = nullptr;
    i64* slot_total = nullptr;
    const i64* slot_first = nullptr;
    const i64* slot_base = nullptr;
    const i64* slot_budget = nullptr;
    const i64* slot_out = nullptr;
    // Counting in chunks of blocks (single instance): this launch's first
    // block, and where the blocks add their attempted writes ([0]) and the
    // end of the expansions they covered ([1], a maximum).
    unsigned blk0 = 0;
    i64* counted = nullptr;
    // 4- and 5-cycle counts: 1 if they use their sets (lists and tables), 0 if
    // every entry or expansion goes the general way; the queue of entries to resolve (kQueueParts parts of
    // qcap entries), its counters 128 bytes apart
    int sets = 1;
    int qcap = 0;
    int3* queue = nullptr;
    unsigned* qcount = nullptr;
    int2* wide = nullptr;  // rep edges left to the wide kernel (first, number), count behind qcount's parts;
                           // null: none are, all their entries are resolved
};

// Diagnostic switches (tests force each path on the same inputs; every
// path gives the same counts and triangles):
//   RAMA_COUNT_FORM=sets | lists   the 4- and 5-cycle counts' form, instead of
//                         the choice by what ends the count
//   RAMA_COUNT_QUEUE=none | queue | list   the sets form without queue and list
//                         of hubs, without the list, without the queue, as where
//                         memory is short
//   RAMA_CYCLE_TABLES=0   the same counts without their sets and tables: every
//                         list entry resolved against the lists (sets form),
//                         every expansion counted by its thread (lists form)
//   RAMA_CYCLE_STATS=1    a line per 4- or 5-cycle count
//   RAMA_EMIT_FORM=dense | queue   the emit form, instead of the choice by
//                         the share of expansions with mids
static bool cycle_tables_on() {
    const char* e = std::getenv("RAMA_CYCLE_TABLES");
    return !(e && e[0] == '0' && e[1] == 0);
}
static int count_form_forced() {  // 0: choose, 1: sets, 2: lists
    const char* e = std::getenv("RAMA_COUNT_FORM");
    if (!e) return 0;
    if (std::strcmp(e, "sets") == 0) return 1;
    if (std::strcmp(e, "lists") == 0) return 2;
    return 0;
}
static bool count_queue_part(const char* part) {
    const char* e = std::getenv("RAMA_COUNT_QUEUE");
    return !e || e[0] == 0 || std::strcmp(e, part) == 0;
}
static int emit_form_forced() {  // 0: choose, 1: dense, 2: queue
    const char* e = std::getenv("RAMA_EMIT_FORM");
    if (!e) return 0;
    if (std::strcmp(e, "dense") == 0) return 1;
    if (std::strcmp(e, "queue") == 0) return 2;
    return 0;
}

// Adds the block's attempted writes to its counter line's [0] and raises
// its [1] to the end of its expansions ([2]: entries the sets form resolved).
// The counters are spread over
// kCountedLines lines of 16 i64 (128 bytes): device atomics from every block
// to one address serialise; the host sums the [0]s and takes the largest
// [1].  Block-uniform call.
constexpr int kCountedLines = 16;
__device__ __forceinline__ void block_counted(i64* counted, i64 mine, i64 xend) {
    __shared__ i64 ws[kWaves];
    const i64 s = block_reduce(mine, OpSum(), ws);
    const i64 m = block_reduce(xend, OpMax(), ws);
    if (threadIdx.x == 0) {
        i64* line = counted + (blockIdx.x % kCountedLines) * 16;
        if (s) atomicAdd(reinterpret_cast<unsigned long long*>(line), (unsigned long long)s);
        atomicMax(reinterpret_cast<unsigned long long*>(line + 1), (unsigned long long)m);
    }
}

// Adds v to base[key] for every lane with `on`, one atomic per distinct key
// in the wave (lanes of a wave mostly share their instance).  Wave-uniform
// call.
__device__ __forceinline__ void wave_add_keyed(i64* base, int key, i64 v, bool on) {
    const int lane = lane_id();
    unsigned long long active = __ballot(on && v != 0);
    while (active) {
        const int leader = __builtin_ctzll(active);
        const int kl = __builtin_amdgcn_readlane(key, leader);
        const unsigned long long m = __ballot(key == kl) & active;
        i64 x = ((m >> lane) & 1ull) ? v : 0;
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) x += shfl_down64(x, d);
        if (lane == 0) atomicAdd(reinterpret_cast<unsigned long long*>(base + kl), (unsigned long long)x);
        active &= ~m;
    }
}

// Locate the rep edge owning expansion x: xoff[r] <= x < xoff[r+1], searching
// from the tile's first rep edge.
__device__ __forceinline__ i64 find_rep(const CycArgs& a, i64 x, i64 r0) {
    i64 lo = r0, hi = a.R - 1;
    // galloping upper bound then binary search
    i64 step = 1;
    while (lo + step <= hi && a.xoff[lo + step] <= x) {
        lo += step;
        step <<= 1;
    }
    hi = lo + step < a.R - 1 ? lo + step : a.R - 1;
    while (lo < hi) {
        const i64 mid = (lo + hi + 1) >> 1;
        if (a.xoff[mid] <= x) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// Resolve expansion x to the two vertices whose neighbour lists intersect and
// the triangle writers' (v1, v2, n1, n2).  Returns false if the expansion is
// skipped (5-cycles with n1 == n2).
template <int S>
__device__ __forceinline__ bool resolve(const CycArgs& a, i64 x, i64 r0, int& v1, int& v2, int& n1, int& n2,
                                        int& qa, int& qb) {
    // 3-cycles: expansion x is rep edge x (no offsets, no tile reps)
    const i64 r = S == 3 ? x : find_rep(a, x, r0);
    v1 = a.rv1[r];
    v2 = a.rv2[r];
    const i64 loc = S == 3 ? 0 : x - a.xoff[r];
    if (S == 3) {
        qa = v1;
        qb = v2;
        n1 = n2 = -1;
        return true;
    } else if (S == 4) {
        n1 = a.adj[a.off[v1] + loc];
        n2 = -1;
        qa = n1;
        qb = v2;
        return true;
    } else {
        const int d1 = a.off[v1 + 1] - a.off[v1];
        const int l1 = (int)(loc % d1), l2 = (int)(loc / d1);
        n1 = a.adj[a.off[v1] + l1];
        n2 = a.adj[a.off[v2] + l2];
        qa = n1;
        qb = n2;
        return n1 != n2;
    }
}

// Number of common neighbours of qa and qb (merge walk over sorted lists).
__device__ __forceinline__ int count_common(const int* __restrict__ off, const int* __restrict__ adj, int qa, int qb) {
    int i = off[qa], ie = off[qa + 1], j = off[qb], je = off[qb + 1];
    int c = 0;
    while (i < ie && j < je) {
        const int x = adj[i], y = adj[j];
        c += (x == y);
        i += (x <= y);
        j += (y <= x);
    }
    return c;
}

// Pairs whose two lists hold more than kHeavy entries together are
// intersected by the whole wave instead of by their own lane: after
// contraction a supernode can have thousands of neighbours, and one lane
// walking two such lists would hold up its wave, its block and the launch.
constexpr int kHeavy = 96;

__device__ __forceinline__ int lower_in(const int* __restrict__ adj, int lo, int hi, int x) {
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (adj[mid] < x) lo = mid + 1; else hi = mid;
    }
    return lo;
}

// Whether entry i of the sorted list [sb, se) (value x) has a partner in the
// sorted list [lb, le): its rank among the equal values of its own list is
// below their count in the other, so a value held a and b times matches
// min(a, b) times — the merge walk's rule.
__device__ __forceinline__ bool has_partner(const int* __restrict__ adj, int sb, int i, int x, int lb, int le) {
    const int rank = (i > sb && adj[i - 1] == x) ? i - lower_in(adj, sb, i, x) : 0;
    const int p = lower_in(adj, lb, le, x);
    if (p >= le || adj[p] != x) return false;
    const int cnt = (p + 1 < le && adj[p + 1] == x) ? lower_in(adj, p, le, x + 1) - p : 1;
    return rank < cnt;
}

// The shorter of the lists of qa and qb as [sb, se), the other as [lb, le).
__device__ __forceinline__ void short_long(const int* __restrict__ off, int qa, int qb, int& sb, int& se, int& lb,
                                           int& le) {
    const int ab = off[qa], ae = off[qa + 1], bb = off[qb], be = off[qb + 1];
    if (ae - ab <= be - bb) {
        sb = ab, se = ae, lb = bb, le = be;
    } else {
        sb = bb, se = be, lb = ab, le = ae;
    }
}

// Lane h's 64-bit value, as two 32-bit lane reads (h wave-uniform).
__device__ __forceinline__ i64 readlane64(i64 v, int h) {
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(v & 0xffffffffll), h);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)((unsigned long long)v >> 32), h);
    return (i64)(((unsigned long long)hi << 32) | lo);
}

// Lists at most this long are probed entry by entry into the other list by
// their own lane (binary searches) when the pair is heavy; pairs of two
// longer lists go to the whole wave.
constexpr int kProbe = 16;

// count_common by one lane from the shorter list [sb, se) into [lb, le).
__device__ __forceinline__ int probe_count(const int* __restrict__ adj, int sb, int se, int lb, int le) {
    int c = 0;
    for (int i = sb; i < se; ++i) c += has_partner(adj, sb, i, adj[i], lb, le) ? 1 : 0;
    return c;
}

// count_common of the lists [ia, ie) and [ib, ib + nb) by one lane: from
// the shorter list by binary searches when the pair is heavy and that list
// is short, else the merge walk.
__device__ __forceinline__ int lane_count_common(const int* __restrict__ adj, int ia, int ie, int ib, int nb) {
    const int na = ie - ia;
    if (na + nb > kHeavy && min(na, nb) <= kProbe)
        return na <= nb ? probe_count(adj, ia, ie, ib, ib + nb) : probe_count(adj, ib, ib + nb, ia, ie);
    int i = ia, j = ib, je = ib + nb, c = 0;
    while (i < ie && j < je) {
        const int x = adj[i], y = adj[j];
        c += (x == y);
        i += (x <= y);
        j += (y <= x);
    }
    return c;
}

// count_common by the whole wave (qa, qb wave-uniform): each lane takes
// entries of the shorter list and binary-searches the longer one.
__device__ __forceinline__ int wave_count_common(const int* __restrict__ off, const int* __restrict__ adj, int qa,
                                                 int qb) {
    int sb, se, lb, le;
    short_long(off, qa, qb, sb, se, lb, le);
    int c = 0;
    for (int i = sb + lane_id(); i < se; i += 64) c += has_partner(adj, sb, i, adj[i], lb, le) ? 1 : 0;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) c += __shfl_xor(c, d, 64);
    return c;
}

// Register-list intersection: one sorted list (at most kRegList entries)
// is held in registers, padded with -1, and the other is streamed from
// memory with independent loads.  The k-th copy of a value in the streamed
// list counts when the register list holds more than k copies, so a value
// occurring a and b times counts min(a, b) — the merge walk's rule.
constexpr int kRegList = 16;

__device__ __forceinline__ void load_reg_list(const int* __restrict__ adj, int b, int nb, int (&rb)[kRegList]) {
#pragma unroll
    for (int q = 0; q < kRegList; ++q) rb[q] = q < nb ? adj[b + q] : -1;
}

__device__ __forceinline__ int count_vs_regs(const int* __restrict__ adj, int ia, int ie, const int (&rb)[kRegList]) {
    int c = 0, prev = -1, occ = 0;
    for (int k = ia; k < ie; ++k) {
        const int x = adj[k];
        int m = 0;
#pragma unroll
        for (int q = 0; q < kRegList; ++q) m += (rb[q] == x);
        occ = x == prev ? occ + 1 : 0;
        prev = x;
        c += occ < m;
    }
    return c;
}

// count_vs_regs when the register list has no repeated value (rdup false):
// then a streamed value counts on its first copy only, when some register
// entry equals it.  The comparisons per streamed value become lane masks
// combined on the scalar unit, and the walk stops at the first value above
// the register list's largest entry (rmax; both lists are sorted).  Only
// the first KL register entries are compared (the entries past a list's
// length are -1 and match nothing).
template <int KL>
__device__ __forceinline__ int count_regs_masks(const int* __restrict__ adj, int ia, int ie,
                                                const int (&rb)[kRegList], int rmax) {
    const int lane = lane_id();
    int c = 0, prev = -1;
    // four streamed entries per round of loads (past the end reads as
    // above rmax), walked in order up to the first entry above rmax
    for (int k = ia; k < ie; k += 4) {
        int x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = k + j < ie ? adj[k + j] : 0x7fffffff;
        bool stop = false;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (x[j] > rmax) {
                stop = true;
                break;
            }
            unsigned long long hit = 0;
#pragma unroll
            for (int q = 0; q < KL; ++q) hit |= __ballot(rb[q] == x[j]);
            c += (int)((hit >> lane) & 1ull) & (int)(x[j] != prev);
            prev = x[j];
        }
        if (stop) break;
    }
    return c;
}

// Register entries the lanes about to intersect must compare (the longest
// of their lists: 8, 12 or 16), agreed by the active lanes of the wave.
__device__ __forceinline__ int reg_width(int nb) {
    if (__ballot(nb > 8) == 0ull) return 8;
    if (__ballot(nb > 12) == 0ull) return 12;
    return kRegList;
}

// kw: reg_width of the lanes that call it together.  With repeated
// register entries it falls back to count_vs_regs.
__device__ __forceinline__ int count_vs_regs_fast(const int* __restrict__ adj, int ia, int ie,
                                                  const int (&rb)[kRegList], int rmax, bool rdup, int kw) {
    if (rdup) return count_vs_regs(adj, ia, ie, rb);
    if (kw == 8) return count_regs_masks<8>(adj, ia, ie, rb, rmax);
    if (kw == 12) return count_regs_masks<12>(adj, ia, ie, rb, rmax);
    return count_regs_masks<kRegList>(adj, ia, ie, rb, rmax);
}

// Largest entry and whether a value repeats, for a register list of nb
// sorted entries.
__device__ __forceinline__ void reg_list_props(const int (&rb)[kRegList], int nb, int& rmax, bool& rdup) {
    rmax = -1;
    rdup = false;
#pragma unroll
    for (int q = 0; q < kRegList; ++q) {
        if (q < nb) rmax = rb[q];
        if (q > 0 && q < nb) rdup |= rb[q] == rb[q - 1];
    }
}

// 3-cycles: one thread per repulsive edge r = expansion r; N(v2) in
// registers, N(v1) streamed.  Tile totals by block reduction.
__global__ __launch_bounds__(kBlock) void k_cycle_count3(CycArgs a, unsigned char* __restrict__ cnt8,
                                                         i64* __restrict__ tile_tot) {
    __shared__ i64 ws[kWaves];
    const unsigned blk = xcd_block();
    const i64 r = (i64)blk * kCycTile + threadIdx.x;
    int c = 0;
    int v1 = 0, v2 = 0;
    bool heavy = false;
    if (r < a.R) {
        v1 = a.rv1[r], v2 = a.rv2[r];
        const int b2 = a.off[v2], n2 = a.off[v2 + 1] - b2;
        const int d1 = a.off[v1 + 1] - a.off[v1];
        if (d1 + n2 > kHeavy) {
            if (min(d1, n2) <= kProbe) {
                int sb, se, lb, le;
                short_long(a.off, v1, v2, sb, se, lb, le);
                c = probe_count(a.adj, sb, se, lb, le);
            } else {
                heavy = true;  // counted by the whole wave below
            }
        } else if (n2 <= kRegList) {
            int rb[kRegList];
            load_reg_list(a.adj, b2, n2, rb);
            int rmax;
            bool rdup;
            reg_list_props(rb, n2, rmax, rdup);
            c = count_vs_regs_fast(a.adj, a.off[v1], a.off[v1 + 1], rb, rmax, rdup, reg_width(n2));
        } else {
            c = count_common(a.off, a.adj, v1, v2);
        }
    }
    for (unsigned long long hm = __ballot(heavy); hm; hm &= hm - 1) {
        const int h = __builtin_ctzll(hm);
        const int s = wave_count_common(a.off, a.adj, __builtin_amdgcn_readlane(v1, h),
                                        __builtin_amdgcn_readlane(v2, h));
        if (lane_id() == h) c = s;
    }
    if (r < a.R) cnt8[r] = (unsigned char)(c < 255 ? c : 255);
    if (a.nslot) wave_add_keyed(a.slot_total, r < a.R ? a.nslot[a.rv1[r]] : 0, (i64)c, r < a.R);
    const i64 tot = block_reduce((i64)c, OpSum(), ws);
    if (threadIdx.x == 0) tile_tot[blk] = tot;
}

// The same for up to kFewReps rep edges, which one thread each does not fill
// the chip with: a block of 1024 threads takes a count tile.  Pairs of short
// lists are walked by a thread; the others are listed, and groups of 16 lanes
// take one each and search the shorter list's entries in the longer, a wave
// where both are long.  Contracted random graphs have lists of 20 to 100
// entries, a chain of as many loads for one thread: 62 -> 23 us a launch on
// 50021 nodes (up to 100k rep edges), 71^3 grid 16 -> 13.  Past about 400k rep
// edges threads are enough and walk short lists faster: 1024x2048 grid, 250k
// 44 -> 30 us, 380k 46 -> 42, 610k 47 -> 66; 192^3, 510k 6.6 -> 9.8.
constexpr int kFewReps = 3 << 17;
constexpr int kFewThreads = 1024;
constexpr int kFewGroups = kFewThreads / 16;
constexpr int kFewWalk = 32;    // entries of both lists that a thread walks
constexpr int kFewGroup = 128;  // entries of the shorter list that a group takes

// count_common by a group of 16 lanes, every lane returns it.
__device__ __forceinline__ int group_count_common(const int* __restrict__ adj, int sb, int se, int lb, int le) {
    int c = 0;
    for (int i = sb + (int)(threadIdx.x & 15); i < se; i += 16) c += has_partner(adj, sb, i, adj[i], lb, le) ? 1 : 0;
#pragma unroll
    for (int d = 8; d >= 1; d >>= 1) c += __shfl_xor(c, d, 16);
    return c;
}

__global__ __launch_bounds__(kFewThreads) void k_cycle_count3_few(CycArgs a, unsigned char* __restrict__ cnt8,
                                                                  i64* __restrict__ tile_tot) {
    __shared__ int cnt[kCycTile];
    __shared__ unsigned char list[kCycTile];
    __shared__ int nlist;
    __shared__ i64 ws[kCycTile / 64];
    const int tid = threadIdx.x, w = tid >> 6;
    const i64 r0 = (i64)blockIdx.x * kCycTile, r = r0 + tid;
    const bool on = tid < kCycTile && r < a.R;
    int v1 = 0;
    if (tid == 0) nlist = 0;
    if (tid < kCycTile) cnt[tid] = 0;
    __syncthreads();
    if (on) {
        v1 = a.rv1[r];
        const int v2 = a.rv2[r];
        const int n = a.off[v1 + 1] - a.off[v1] + a.off[v2 + 1] - a.off[v2];
        if (n <= kFewWalk) cnt[tid] = count_common(a.off, a.adj, v1, v2);
        else list[atomicAdd(&nlist, 1)] = (unsigned char)tid;
    }
    __syncthreads();
    const int n = nlist;
    for (int q = tid >> 4; q < n; q += kFewGroups) {
        const int rl = list[q];
        int sb, se, lb, le;
        short_long(a.off, a.rv1[r0 + rl], a.rv2[r0 + rl], sb, se, lb, le);
        if (se - sb > kFewGroup) {
            if ((tid & 15) == 0) cnt[rl] = -1;
            continue;
        }
        const int c = group_count_common(a.adj, sb, se, lb, le);
        if ((tid & 15) == 0) cnt[rl] = c;
    }
    __syncthreads();
    for (int q = w; q < n; q += kFewThreads / 64) {
        const int rl = list[q];
        if (cnt[rl] != -1) continue;  // uniform within the wave
        const int c = wave_count_common(a.off, a.adj, __builtin_amdgcn_readfirstlane(a.rv1[r0 + rl]),
                                        __builtin_amdgcn_readfirstlane(a.rv2[r0 + rl]));
        if (lane_id() == 0) cnt[rl] = c;
    }
    __syncthreads();
    if (w < kCycTile / 64) {
        const int c = cnt[tid];
        if (on) cnt8[r] = (unsigned char)(c < 255 ? c : 255);
        if (a.nslot) wave_add_keyed(a.slot_total, on ? a.nslot[v1] : 0, (i64)c, on);
        i64 t = c;
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) t += shfl_down64(t, d);
        if (lane_id() == 0) ws[w] = t;
    }
    __syncthreads();
    if (tid == 0) {
        i64 t = 0;
#pragma unroll
        for (int q = 0; q < kCycTile / 64; ++q) t += ws[q];
        tile_tot[blockIdx.x] = t;
    }
}

// Adds `v` to the total of the tile holding expansion x, flushing the
// running sum whenever the thread's expansions cross into the next tile.
struct TileAcc {
    i64 tile = -1;
    i64 sum = 0;
    __device__ __forceinline__ void add(i64* tot, i64 x, i64 v) {
        const i64 t = x / kCycTile;
        if (t != tile) {
            flush(tot);
            tile = t;
        }
        sum += v;
    }
    __device__ __forceinline__ void flush(i64* tot) {
        if (tile >= 0 && sum != 0)
            atomicAdd(reinterpret_cast<unsigned long long*>(tot + tile), (unsigned long long)sum);
        sum = 0;
    }
};

// 4- and 5-cycle counts, lists form (the sets form and the choice follow).
//
// 4-cycles: one thread per repulsive edge; its expansions n1 ∈ N(v1) are
// xoff[r] .. xoff[r+1]-1 in order, each intersecting N(n1) with N(v2)
// (held in registers).  tile_tot must be zero on entry.
// Rep edges whose v1 has at least kWideRep neighbours, or whose v2 has more
// than kRegList, are counted by the whole wave, one rep edge at a time: the
// wave puts N(v2) in an LDS hash set (kSetSlots slots, lists of at most
// kSetMax entries) and lane l takes expansions l, l + 64, ..., streaming
// N(n1) and probing each entry.  After contraction supernodes have dozens
// of neighbours: one lane per rep edge would walk long merge walks serially
// while its wave waits.  A repeated value in either list (the min(a, b)
// rule) or a longer N(v2) keeps the merge walk for that expansion.
constexpr int kWideRep = 48;
constexpr int kSetSlots = 256;
constexpr int kSetMax = 128;

__device__ __forceinline__ int set_hash(int m) { return (int)(((unsigned)m * 2654435761u) >> 24); }

__global__ __launch_bounds__(kBlock) void k_cycle_count4(CycArgs a, unsigned char* __restrict__ cnt8,
                                                         i64* __restrict__ tile_tot) {
    __shared__ int wset[kWaves][4 * kSetSlots];
    const int w = threadIdx.x >> 6;
    const i64 r = (i64)(a.blk0 + xcd_block()) * kBlock + threadIdx.x;
    const bool on = r < a.R;
    i64 mine = 0, xend = 0;
    int v1 = 0, v2 = 0, b1 = 0, d1 = 0, b2 = 0, n2 = 0;
    i64 x0 = 0;
    if (on) {
        v1 = a.rv1[r];
        v2 = a.rv2[r];
        b1 = a.off[v1];
        d1 = a.off[v1 + 1] - b1;
        b2 = a.off[v2];
        n2 = a.off[v2 + 1] - b2;
        x0 = a.xoff[r];
        xend = x0 + d1;
    }
    const bool wide = on && a.sets && (d1 >= kWideRep || n2 > kRegList);
    if (on && !wide) {
        int rb[kRegList];
        const bool regs = n2 <= kRegList;
        int rmax = -1, kw = kRegList;
        bool rdup = false;
        if (regs) {
            load_reg_list(a.adj, b2, n2, rb);
            reg_list_props(rb, n2, rmax, rdup);
            kw = reg_width(n2);
        }
        TileAcc acc;
        // the next n1's list bounds are loaded while this one is walked
        int ia = 0, ie = 0;
        if (d1 > 0) {
            const int n1 = a.adj[b1];
            ia = a.off[n1];
            ie = a.off[n1 + 1];
        }
        for (int l = 0; l < d1; ++l) {
            int na = 0, ne = 0;
            if (l + 1 < d1) {
                const int nn = a.adj[b1 + l + 1];
                na = a.off[nn];
                ne = a.off[nn + 1];
            }
            const int c = regs ? count_vs_regs_fast(a.adj, ia, ie, rb, rmax, rdup, kw)
                               : lane_count_common(a.adj, ia, ie, b2, n2);
            cnt8[x0 + l] = (unsigned char)(c < 255 ? c : 255);
            acc.add(tile_tot, x0 + l, 2 * (i64)c);
            mine += 2 * (i64)c;
            ia = na;
            ie = ne;
        }
        acc.flush(tile_tot);
    }
    // wide rep edges: the wave works as four groups of 16 lanes, group g
    // taking the wide rep edges of lanes 16g .. 16g + 15 one after another
    // (four rep edges in flight per wave); the attempted writes are credited
    // to the rep's own lane (its instance, its block total)
    const int lane = lane_id(), g = lane >> 4, gl = lane & 15;
    const unsigned long long wm = __ballot(wide);
    unsigned gm = (unsigned)((wm >> (16 * g)) & 0xffffull);  // this group's wide lanes
    int niter = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) niter = max(niter, __popcll((wm >> (16 * q)) & 0xffffull));
    int* gset = &wset[w][g * kSetSlots];
    const unsigned long long gmask = 0xffffull << (16 * g);
    for (int it = 0; it < niter; ++it) {
        const bool gact = gm != 0u;  // uniform within the group
        const int h = gact ? 16 * g + __builtin_ctz(gm) : lane;
        if (gact) gm &= gm - 1u;
        const int hb1 = __shfl(b1, h, 64), hd1 = gact ? __shfl(d1, h, 64) : 0;
        const int hb2 = __shfl(b2, h, 64), hn2 = gact ? __shfl(n2, h, 64) : 0;
        const i64 hx0 = __shfl(x0, h, 64);
        // N(v2) into the group's set (a repeated value, or too long a list:
        // merge walks instead)
        bool use_set = gact && hn2 <= kSetMax;
        int vmax = -1;
        bool dup = false;
        if (use_set) {
            for (int k = gl; k < kSetSlots; k += 16) gset[k] = -1;
        }
        __builtin_amdgcn_wave_barrier();
        if (use_set) {
            for (int k = gl; k < hn2; k += 16) {
                const int m = a.adj[hb2 + k];
                dup |= k > 0 && a.adj[hb2 + k - 1] == m;
                int hs = set_hash(m);
                while (true) {
                    const int old = atomicCAS(&gset[hs], -1, m);
                    if (old == -1 || old == m) break;
                    hs = (hs + 1) & (kSetSlots - 1);
                }
            }
            vmax = hn2 > 0 ? a.adj[hb2 + hn2 - 1] : -1;
        }
        use_set = use_set && (__ballot(dup) & gmask) == 0ull;
        __builtin_amdgcn_wave_barrier();
        TileAcc acc;
        i64 part = 0;
        for (int l = gl; l < hd1; l += 16) {
            const int n1 = a.adj[hb1 + l];
            const int ia = a.off[n1], ie = a.off[n1 + 1];
            int c = 0;
            bool merge = !use_set;
            if (use_set) {
                // four entries per round of loads (past the end reads as
                // above vmax), walked in order up to the first above vmax
                int prev = -1;
                bool stop = false;
                for (int k = ia; k < ie && !stop; k += 4) {
                    int xs[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) xs[u] = k + u < ie ? a.adj[k + u] : 0x7fffffff;
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const int x = xs[u];
                        if (stop || x > vmax) {
                            stop = true;
                            continue;
                        }
                        if (x == prev) {  // N(n1) repeats a value: the merge walk counts it
                            merge = true;
                            stop = true;
                            continue;
                        }
                        prev = x;
                        int hs = set_hash(x);
                        while (true) {
                            const int key = gset[hs];
                            if (key == x) {
                                ++c;
                                break;
                            }
                            if (key == -1) break;
                            hs = (hs + 1) & (kSetSlots - 1);
                        }
                    }
                }
            }
            if (merge) c = lane_count_common(a.adj, ia, ie, hb2, hn2);
            cnt8[hx0 + l] = (unsigned char)(c < 255 ? c : 255);
            acc.add(tile_tot, hx0 + l, 2 * (i64)c);
            part += 2 * (i64)c;
        }
        acc.flush(tile_tot);
#pragma unroll
        for (int d = 8; d >= 1; d >>= 1) part += __shfl_xor(part, d, 64);  // within the group
        if (gact && lane == h) mine += part;
        __builtin_amdgcn_wave_barrier();
    }
    if (a.nslot) wave_add_keyed(a.slot_total, on ? a.nslot[v1] : 0, mine, on);
    if (a.counted) block_counted(a.counted, mine, xend);
}

// 5-cycles: one thread per (repulsive edge r, n2 = l2-th neighbour of v2);
// its expansions (n1 = l1-th neighbour of v1, n2) are xoff[r] + l2*d1 + l1
// for l1 = 0 .. d1-1, each intersecting N(n1) with N(n2); n1 == n2 is
// skipped.  Threads of rep r are yoff[r] .. yoff[r+1]-1; ytile_rep gives
// each block's first rep.  tile_tot must be zero on entry.
//
// Two ways to count one thread's d1 expansions, with identical counts:
//  * 2-hop table (the common case): the block builds, for each distinct v1
//    among its threads, an LDS hash table of v1's 2-hop neighbourhood,
//    mid -> bitmask of the l1 whose list N(n1) holds mid.  The thread then
//    walks N(n2) once, looks every mid up and adds its mask to bit-sliced
//    per-l1 counters, instead of streaming every N(n1) against N(n2).  Valid
//    when no list involved holds a value twice (then |N(n1) ∩ N(n2)| is the
//    merge walk's min(a, b) count), d1 <= 32 and the 2-hop lists fit.
//  * per expansion (otherwise): N(n2) in registers (or the merge walk /
//    probes for long lists), each N(n1) streamed against it.
constexpr int kT5Tables = 16;      // 2-hop tables (distinct v1 runs) per block
constexpr int kT5SlotBits = 11;
constexpr int kT5Slots = 1 << kT5SlotBits;  // slots of the block's shared hash table
constexpr int kT5MaxFill = 1536;   // entries of all tables together at most this (load <= 3/4)
constexpr int kT5MaxD1 = 32;       // d(v1) at most this (32-bit masks)
constexpr int kT5RepWin = 256;     // rep edges a block locates its threads among in LDS
constexpr int kT5MaxNode = 1 << 27;  // node ids below this: (mid, run) fits one key

// The tables of a block share one open-addressing hash table of keys
// mid * kT5Tables + run.
__device__ __forceinline__ int t5_hash(int key) {
    return (int)(((unsigned)key * 2654435761u) >> (32 - kT5SlotBits));
}

// The per-expansion form for one thread (see above).
__device__ __forceinline__ void count5_direct(const CycArgs& a, int b1, int d1, int n2, int bq, int nq, i64 x0,
                                              unsigned char* __restrict__ cnt8, i64* __restrict__ tile_tot,
                                              i64& mine) {
    int rb[kRegList];
    const bool regs = nq <= kRegList;
    int rmax = -1, kw = kRegList;
    bool rdup = false;
    if (regs) {
        load_reg_list(a.adj, bq, nq, rb);
        reg_list_props(rb, nq, rmax, rdup);
        kw = reg_width(nq);
    }
    TileAcc acc;
    // the next n1 and its list bounds are loaded while this one is walked
    int n1 = d1 > 0 ? a.adj[b1] : 0;
    int ia = d1 > 0 ? a.off[n1] : 0, ie = d1 > 0 ? a.off[n1 + 1] : 0;
    for (int l = 0; l < d1; ++l) {
        const int nn = l + 1 < d1 ? a.adj[b1 + l + 1] : 0;
        const int na = l + 1 < d1 ? a.off[nn] : 0, ne = l + 1 < d1 ? a.off[nn + 1] : 0;
        int c = 0;
        if (n1 != n2)
            c = regs ? count_vs_regs_fast(a.adj, ia, ie, rb, rmax, rdup, kw)
                     : lane_count_common(a.adj, ia, ie, bq, nq);
        cnt8[x0 + l] = (unsigned char)(c < 255 ? c : 255);
        acc.add(tile_tot, x0 + l, 3 * (i64)c);
        mine += 3 * (i64)c;
        n1 = nn;
        ia = na;
        ie = ne;
    }
    acc.flush(tile_tot);
}

__global__ __launch_bounds__(kBlock) void k_cycle_count5(CycArgs a, const i64* __restrict__ yoff,
                                                         const int* __restrict__ ytile_rep, i64 Y, int tables,
                                                         unsigned char* __restrict__ cnt8,
                                                         i64* __restrict__ tile_tot) {
    __shared__ int tkey[kT5Slots];
    __shared__ unsigned tmask[kT5Slots];
    __shared__ int tv1[kT5Tables];
    __shared__ int tok[kT5Tables];
    __shared__ int tfill[kT5Tables];
    __shared__ int sv1[kBlock];
    __shared__ int wruns[kWaves];
    const unsigned blk = a.blk0 + xcd_block();
    const int tid = threadIdx.x, lane = lane_id(), w = tid >> 6;
    const i64 y = (i64)blk * kCycTile + tid;
    const bool on = y < Y;
    i64 mine = 0, xend = 0;
    int slot = 0;
    int v1 = -1, b1 = 0, d1 = 0, n2 = 0, bq = 0, nq = 0;
    i64 x0 = 0;
    // rep owning each thread: the block's threads belong to reps r0, r0 + 1,
    // ...; their thread offsets are loaded once (coalesced) and every thread
    // marks where its rep starts, so a block max-scan (kept as a running max
    // over the marks) hands each thread its rep.  Blocks whose threads span
    // more than kT5RepWin reps fall back to a galloping search.
    const i64 y0 = (i64)blk * kCycTile;
    const i64 r0 = y0 < Y ? (i64)ytile_rep[blk] : 0;
    sv1[tid] = -1;
    __syncthreads();
    bool wide = false;
    for (int k = tid; k < kT5RepWin; k += kBlock) {
        const i64 r = r0 + k;
        if (r < a.R) {
            const i64 ys = yoff[r];
            if (ys >= y0 && ys < y0 + kCycTile && yoff[r + 1] > ys) sv1[ys - y0] = k;
        }
    }
    if (y0 < Y) {
        const i64 rl = r0 + kT5RepWin - 1;
        wide = rl < a.R && yoff[rl + 1] < (y0 + kCycTile < Y ? y0 + kCycTile : Y);
    }
    __syncthreads();
    int mark = sv1[tid];
    // inclusive max-scan of the marks over the block (first thread: its rep
    // r0 starts before the block, mark 0)
    if (tid == 0 && mark < 0) mark = 0;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int t = __shfl_up(mark, d, 64);
        if (lane >= d) mark = max(mark, t);
    }
    __shared__ int wmax[kWaves];
    if (lane == 63) wmax[w] = mark;
    __syncthreads();
    for (int q = 0; q < w; ++q) mark = max(mark, wmax[q]);
    __syncthreads();
    if (on) {
        i64 r = r0 + mark;
        if (wide) {
            // rep owning thread y (galloping from the block's first rep)
            i64 lo = r0, hi = a.R - 1, step = 1;
            while (lo + step <= hi && yoff[lo + step] <= y) {
                lo += step;
                step <<= 1;
            }
            hi = lo + step < a.R - 1 ? lo + step : a.R - 1;
            while (lo < hi) {
                const i64 mid = (lo + hi + 1) >> 1;
                if (yoff[mid] <= y) lo = mid; else hi = mid - 1;
            }
            r = lo;
        }
        v1 = a.rv1[r];
        const int v2 = a.rv2[r];
        const int l2 = (int)(y - yoff[r]);
        b1 = a.off[v1];
        d1 = a.off[v1 + 1] - b1;
        n2 = a.adj[a.off[v2] + l2];
        bq = a.off[n2];
        nq = a.off[n2 + 1] - bq;
        x0 = a.xoff[r] + (i64)l2 * d1;
        if (a.nslot) slot = a.nslot[v1];
    }
    // runs of equal v1 over the block's threads (rep edges are in row order,
    // so a run is usually all threads of one v1); run k < kT5Tables gets
    // table k
    sv1[tid] = v1;
    for (int k = tid; k < kT5Slots; k += kBlock) {
        tkey[k] = -1;
        tmask[k] = 0u;
    }
    __syncthreads();
    const bool start = on && (tid == 0 || sv1[tid - 1] != v1);
    const unsigned long long sm = __ballot(start);
    if (lane == 0) wruns[w] = __popcll(sm);
    __syncthreads();
    int before = 0, runs = 0;
    for (int q = 0; q < kWaves; ++q) {
        before += q < w ? wruns[q] : 0;
        runs += wruns[q];
    }
    // this thread's run index (its run starts at or before it)
    const int run = before + __popcll(sm & ((2ull << lane) - 1ull)) - 1;
    if (start && run < kT5Tables) {
        tv1[run] = v1;
        tok[run] = 1;
    }
    const int ntab = runs < kT5Tables ? runs : kT5Tables;
    __syncthreads();
    // build, in three steps: each wave sizes its tables (w, w + kWaves, ...:
    // lane l holds the bounds of the list of v1's l-th neighbour n1); the
    // tables that fit the shared capacity in run order are kept; each wave
    // inserts its kept tables' (mid, l) pairs, flattened over its 64 lanes
    constexpr int kPerWave = kT5Tables / kWaves;
    int s0[kPerWave], s1[kPerWave];
#pragma unroll
    for (int i = 0; i < kPerWave; ++i) {
        const int k = w + i * kWaves;
        s0[i] = s1[i] = 0;
        if (k >= ntab) continue;
        const int v = tv1[k];
        const int bv = a.off[v], dv = a.off[v + 1] - bv;
        if (dv <= kT5MaxD1 && lane < dv) {
            const int n1 = a.adj[bv + lane];
            s0[i] = a.off[n1];
            s1[i] = a.off[n1 + 1];
        }
        int fill = s1[i] - s0[i];
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) fill += __shfl_xor(fill, d, 64);
        if (lane == 0) tfill[k] = dv <= kT5MaxD1 && tables ? fill : kT5MaxFill + 1;
    }
    __syncthreads();
    if (tid == 0) {
        int used = 0;
        for (int k = 0; k < ntab; ++k) {
            const bool fits = used + tfill[k] <= kT5MaxFill;
            tok[k] = fits ? 1 : 0;
            used += fits ? tfill[k] : 0;
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPerWave; ++i) {
        const int k = w + i * kWaves;
        if (k >= ntab || !tok[k]) continue;  // wave-uniform
        bool dup = false;
        const int fill = tfill[k];
        const int len = s1[i] - s0[i];
        int excl = len;  // where list l starts among the table's pairs
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int t = __shfl_up(excl, d, 64);
            if (lane >= d) excl += t;
        }
        excl -= len;
        const int dv = a.off[tv1[k] + 1] - a.off[tv1[k]];
        for (int f0 = 0; f0 < fill; f0 += 64) {  // wave-uniform: every lane takes part in the shuffles
            const int f = f0 + lane;
            int l = 0;
            for (int j = 1; j < dv; ++j) l = __builtin_amdgcn_readlane(excl, j) <= f ? j : l;
            const int q = __shfl(s0[i], l, 64) + (f - __shfl(excl, l, 64));
            if (f >= fill) continue;
            const int key = a.adj[q] * kT5Tables + k;
            const unsigned bit = 1u << l;
            int h = t5_hash(key);
            while (true) {
                const int old = atomicCAS(&tkey[h], -1, key);
                if (old == -1 || old == key) {
                    dup |= (atomicOr(&tmask[h], bit) & bit) != 0u;
                    break;
                }
                h = (h + 1) & (kT5Slots - 1);
            }
        }
        // a list that repeats a value disables its table
        if (__ballot(dup) != 0ull && lane == 0) tok[k] = 0;
    }
    __syncthreads();
    if (on) {
        const bool table = run < ntab && tok[run] && nq <= 255;
        bool direct = !table;
        if (table) {
            // per-l1 counts of N(n2)'s mids, bit-sliced over 8 planes
            unsigned p[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
            int prev = -1;
            // four entries of N(n2) per round of loads
            for (int q0 = bq; q0 < bq + nq && !direct; q0 += 4) {
                int ms[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) ms[u] = q0 + u < bq + nq ? a.adj[q0 + u] : -1;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if (direct || q0 + u >= bq + nq) continue;
                    const int m = ms[u];
                    if (m == prev) {  // N(n2) repeats a value: the min(a, b) rule needs the direct form
                        direct = true;
                        continue;
                    }
                    prev = m;
                    const int want = m * kT5Tables + run;
                    int h = t5_hash(want);
                    unsigned mk = 0u;
                    while (true) {
                        const int key = tkey[h];
                        if (key == want) {
                            mk = tmask[h];
                            break;
                        }
                        if (key == -1) break;
                        h = (h + 1) & (kT5Slots - 1);
                    }
#pragma unroll
                    for (int b = 0; b < 8; ++b) {
                        const unsigned carry = p[b] & mk;
                        p[b] ^= mk;
                        mk = carry;
                    }
                }
            }
            if (!direct) {
                unsigned nz = 0u;
#pragma unroll
                for (int b = 0; b < 8; ++b) nz |= p[b];
                TileAcc acc;
                for (int l = 0; l < d1; ++l) {
                    int c = 0;
                    if ((nz >> l) & 1u) {
#pragma unroll
                        for (int b = 0; b < 8; ++b) c |= (int)((p[b] >> l) & 1u) << b;
                        if (a.adj[b1 + l] == n2) c = 0;
                    }
                    cnt8[x0 + l] = (unsigned char)(c < 255 ? c : 255);
                    acc.add(tile_tot, x0 + l, 3 * (i64)c);
                    mine += 3 * (i64)c;
                }
                acc.flush(tile_tot);
            }
        }
        if (direct) count5_direct(a, b1, d1, n2, bq, nq, x0, cnt8, tile_tot, mine);
        xend = x0 + d1;
    }
    if (a.nslot) wave_add_keyed(a.slot_total, slot, mine, on);
    if (a.counted) block_counted(a.counted, mine, xend);
}

// 4- and 5-cycle counts, sets form.  Expansions of rep edge r = (v1, v2) are xoff[r] ..
// xoff[r+1]-1: for 4-cycles the neighbours n1 of v1 (l1 = 0 .. d1-1), each
// intersecting N(n1) with N(v2); for 5-cycles the pairs (n1, n2) at
// l2 * d1 + l1, each intersecting N(n1) with N(n2), n1 == n2 left out.
//
// Nearly all of these intersections are empty, so the lists are not walked
// against each other.  Rep edges lie in row order, those of one v1 are a run.
// A group of 16 lanes takes a run, marks the 2-hop neighbourhood of v1 (every
// entry of every N(n1)) in a set of bits in LDS, and looks up, for each rep
// edge of the run, the entries of N(v2) (4-cycles) or of every N(n2)
// (5-cycles): ten entries of one list instead of a hundred of ten lists.
// Entries that pass are queued, first per wave, then in memory, and a second
// launch resolves them against the lists themselves, a lane each: an entry m
// belongs to expansion l1 if n1 is in N(m).  So the counts are exact whatever
// the set lets through, and the few rep edges with most of the cycles (chords
// gather on some vertices) are shared by the whole chip.
//
// A set is words of 32 bits, three bits of one word marked per entry: one LDS
// read per look-up, about one entry in two hundred passes by accident (146
// entries marked on average in the 2D grid).  Runs of hubs (more than
// kSetLists lists or kSetFill entries) and rep edges whose v2 is one are
// listed, and a launch of blocks takes a few of them each with a set of
// kBigWords words.
//
// The lists form takes 9300 vector instructions per wave there and waits on the
// longest of its lanes' lists.  D mode on the 12.47M-edge grid, all 4- and 5-cycle
// counts of a solve: 54.5 + 59.7 ms by lists, 14 + 36 with the sets (a full pass:
// 9.3M rep edges and 100M expansions 5.0 -> 1.4 ms, 1.1G expansions 11 -> 8.2); the
// 192^3 grid's PD+ 14.0 + 8.1 -> 11.0 + 7.7.  5-cycles are bound by the lists' load
// latency (59% of the waves' time, 3.5 to 4 waves per SIMD) and by about 60
// instructions per step of four lists.
constexpr int kSetLanes = 16;                  // lanes per run
constexpr int kSetGroups = kBlock / kSetLanes;
constexpr int kSetWords = 64;                  // words of a group's set
constexpr int kBigWords = 2048;                // words of the block's set
constexpr int kSetLists = 2 * kSetLanes;       // lists of v1 at most
constexpr int kSetFill = 768;                  // entries marked at most
constexpr int kSetQueue = 128;                 // waiting entries per wave
constexpr int kQueueParts = 64;                // of the queue in memory
constexpr int kSetMinReps = 16;                // rep edges per block, at least and at most
constexpr int kSetMaxReps = kBlock;
constexpr int kRunReps = 16;                   // rep edges per run at most: a group takes them in turn
constexpr int kWideReps = 8;                   // rep edges per entry of the list of hubs' runs

// Word and bits of an entry in a set of 2^kLog words.
template <int kLog>
__device__ __forceinline__ unsigned set_bits(int m, unsigned* bits) {
    const unsigned h = (unsigned)m * 2654435761u;
    *bits = (1u << ((h >> (27 - kLog)) & 31)) | (1u << ((h >> (22 - kLog)) & 31)) | (1u << ((h >> (17 - kLog)) & 31));
    return h >> (32 - kLog);
}

// Orders the wave's LDS accesses around it (the lanes of a group share a set).
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// f(x) for the entries x of up to 16 lists, lane i of the group holding the
// bounds [p0, p1) of list i (lists from cnt on are empty); the group's lanes
// share each list, four lists are loaded at a time.
template <class F>
__device__ __forceinline__ void walk_lists(const CycArgs& a, int p0, int p1, int cnt, F f) {
    const int lane = threadIdx.x & (kSetLanes - 1);
    for (int u0 = 0; u0 < cnt; u0 += 4) {  // uniform within the group
        int s[4], e[4], x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            s[u] = __shfl(p0, u0 + u, kSetLanes);
            e[u] = __shfl(p1, u0 + u, kSetLanes);
            x[u] = s[u] + lane < e[u] ? a.adj[s[u] + lane] : -1;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (x[u] >= 0) f(x[u]);
            for (int k = s[u] + kSetLanes + lane; k < e[u]; k += kSetLanes) f(a.adj[k]);
        }
    }
}
// Of the same lists: hit(i, k) for the entries x = adj[k] of list i with
// test(x).
template <class T, class F>
__device__ __forceinline__ void find_in_lists(const CycArgs& a, int p0, int p1, int cnt, T test, F hit) {
    const int lane = threadIdx.x & (kSetLanes - 1);
    for (int u0 = 0; u0 < cnt; u0 += 4) {  // uniform within the group
        int s[4], e[4], x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            s[u] = __shfl(p0, u0 + u, kSetLanes);
            e[u] = __shfl(p1, u0 + u, kSetLanes);
            x[u] = s[u] + lane < e[u] ? a.adj[s[u] + lane] : -1;
        }
        unsigned hits = 0u, more = 0u;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            hits |= x[u] >= 0 && test(x[u]) ? 1u << u : 0u;
            more |= e[u] - s[u] > kSetLanes ? 1u << u : 0u;
        }
        auto pick = [](int v0, int v1, int v2, int v3, int u) {
            const int lo = u & 1 ? v1 : v0, hi = u & 1 ? v3 : v2;
            return u & 2 ? hi : lo;
        };
        for (; hits; hits &= hits - 1u) {
            const int u = __builtin_ctz(hits);
            hit(u0 + u, pick(s[0], s[1], s[2], s[3], u) + lane);
        }
        for (; more; more &= more - 1u) {
            const int u = __builtin_ctz(more);
            const int z = pick(e[0], e[1], e[2], e[3], u);
            for (int k = pick(s[0], s[1], s[2], s[3], u) + kSetLanes + lane; k < z; k += 4 * kSetLanes) {
                int y[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) y[v] = k + v * kSetLanes < z ? a.adj[k + v * kSetLanes] : -1;
                unsigned far = 0u;
#pragma unroll
                for (int v = 0; v < 4; ++v) far |= y[v] >= 0 && test(y[v]) ? 1u << v : 0u;
                for (; far; far &= far - 1u) hit(u0 + u, k + __builtin_ctz(far) * kSetLanes);
            }
        }
    }
}

// Adds c to the (saturating) count byte of expansion x, whose count is at
// most `most`.
__device__ __forceinline__ void bump_count(unsigned char* cnt8, i64 x, int c, int most) {
    unsigned* p = reinterpret_cast<unsigned*>(cnt8 + (x & ~(i64)3));
    const int sh = 8 * (int)(x & 3);
    if (most <= 255) {  // nothing to wait for
        atomicAdd(p, (unsigned)c << sh);
        return;
    }
    unsigned old = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    while (true) {
        const unsigned b = (old >> sh) & 255u, nb = min(255u, b + (unsigned)c);
        if (b == nb) return;
        const unsigned prev = atomicCAS(p, old, (old & ~(255u << sh)) | (nb << sh));
        if (prev == old) return;
        old = prev;
    }
}

// Counts entry k of N(v2) (4-cycles) or of N(n2), n2 the l2-th neighbour of
// v2 (5-cycles), into the expansions of rep edge r; returns the attempted
// writes.  Values repeated in a list count as the merge walk would count
// them, min(a, b) times.
template <int S>
__device__ __forceinline__ i64 resolve_entry(const CycArgs& a, i64 r, int l2, int k, unsigned char* cnt8,
                                             i64* tile_tot) {
    const int v1 = a.rv1[r], v2 = a.rv2[r];
    const int b1 = a.off[v1], e1 = a.off[v1 + 1];
    const int y = S == 4 ? v2 : a.adj[a.off[v2] + l2];
    const int ys = a.off[y], ye = a.off[y + 1];
    const int m = a.adj[k];
    if (k > ys && a.adj[k - 1] == m) return 0;  // counted with the value's first entry
    int mb = 1;
    while (k + mb < ye && a.adj[k + mb] == m) ++mb;
    const int bm = a.off[m], em = a.off[m + 1];
    const i64 x0 = a.xoff[r] + (S == 5 ? (i64)l2 * (e1 - b1) : 0);
    i64 writes = 0;
    auto hit = [&](int l, int c) {
        bump_count(cnt8, x0 + l, c, ye - ys);
        atomicAdd(reinterpret_cast<unsigned long long*>(tile_tot + (x0 + l) / kCycTile),
                  (unsigned long long)(c * (S - 2)));
        writes += c * (S - 2);
    };
    // N(v1) against N(m), which holds n1 as often as N(n1) holds m: a merge
    // walk, or where one list is much longer the other's entries in it
    int i = b1, j = bm;
    const bool far = e1 - b1 > 8 * (em - bm), near = em - bm > 8 * (e1 - b1);
    while (i < e1 && j < em) {
        const int p = a.adj[i], q = a.adj[j];
        if (p != q) {
            if (p < q) i = far ? lower_in(a.adj, i, e1, q) : i + 1;
            else j = near ? lower_in(a.adj, j, em, p) : j + 1;
            continue;
        }
        int ma = 1;
        while (j + ma < em && a.adj[j + ma] == p) ++ma;
        j += ma;
        for (; i < e1 && a.adj[i] == p; ++i)
            if (S == 4 || p != y) hit(i - b1, min(ma, mb));
    }
    return writes;
}

// An entry into part `part` of the queue, in memory (lanes that call it
// together take one place after another), or resolved at once if it is full.
template <int S>
__device__ __forceinline__ i64 queue_entry(const CycArgs& a, int part, i64 r, i64 r0, int l2, int k,
                                           unsigned char* cnt8, i64* tile_tot) {
    const unsigned long long m = __ballot(1);
    const int rank = __popcll(m & ((1ull << lane_id()) - 1ull));
    unsigned at = 0;
    if (rank == 0) at = atomicAdd(a.qcount + part * 32, (unsigned)__popcll(m));
    at = (unsigned)__builtin_amdgcn_readfirstlane((int)at) + (unsigned)rank;
    if (at < (unsigned)a.qcap) {
        a.queue[(i64)part * a.qcap + at] = make_int3((int)(unsigned)(r - r0), l2, k);
        return 0;
    }
    const i64 add = resolve_entry<S>(a, r, l2, k, cnt8, tile_tot);
    if (a.nslot && add)
        atomicAdd(reinterpret_cast<unsigned long long*>(a.slot_total + a.nslot[a.rv1[r]]), (unsigned long long)add);
    return add;
}

// Resolves the queued entries of a count launch, whose first rep edge is r0.
template <int S>
__global__ __launch_bounds__(kBlock) void k_cycle_resolve(CycArgs a, i64 r0, unsigned char* __restrict__ cnt8,
                                                          i64* __restrict__ tile_tot) {
    const int part = blockIdx.x % kQueueParts, step = (int)(gridDim.x / kQueueParts) * kBlock;
    const unsigned passed = a.qcount[part * 32];  // those past the queue's end were resolved at once
    const int n = (int)min(passed, (unsigned)a.qcap);
    if (a.counted && blockIdx.x < kQueueParts && threadIdx.x == 0)
        atomicAdd(reinterpret_cast<unsigned long long*>(a.counted + part % kCountedLines * 16 + 2),
                  (unsigned long long)passed);
    i64 mine = 0;
    for (int q0 = (int)(blockIdx.x / kQueueParts) * kBlock; q0 < n; q0 += step) {  // uniform
        const int q = q0 + (int)threadIdx.x;
        i64 add = 0;
        int slot = 0;
        if (q < n) {
            const int3 e = a.queue[(i64)part * a.qcap + q];
            const i64 r = r0 + (i64)(unsigned)e.x;
            add = resolve_entry<S>(a, r, e.y, e.z, cnt8, tile_tot);
            if (a.nslot) slot = a.nslot[a.rv1[r]];
        }
        if (a.nslot) wave_add_keyed(a.slot_total, slot, add, q < n);
        mine += add;
    }
    if (a.counted) block_counted(a.counted, mine, 0);
}

// A wave's waiting entries, in LDS.
struct WaveQueue {
    int k[kSetQueue], l[kSetQueue];
    unsigned r[kSetQueue];  // from the launch's first rep edge on
    int n;
};
// An entry that passed: into the wave's queue, or past it if it is full.
template <int S>
__device__ __forceinline__ i64 push_entry(const CycArgs& a, WaveQueue& q, i64 r, i64 r0, int l2, int k,
                                          unsigned char* cnt8, i64* tile_tot) {
    const unsigned long long m = __ballot(1);
    const int rank = __popcll(m & ((1ull << lane_id()) - 1ull));
    int at = 0;
    if (rank == 0) at = atomicAdd(&q.n, __popcll(m));
    at = __builtin_amdgcn_readfirstlane(at) + rank;
    if (at >= kSetQueue) return queue_entry<S>(a, blockIdx.x % kQueueParts, r, r0, l2, k, cnt8, tile_tot);
    q.k[at] = k;
    q.l[at] = l2;
    q.r[at] = (unsigned)(r - r0);
    return 0;
}
// Passes the wave's entries on once there are `least` (wave-uniform call).
template <int S>
__device__ __forceinline__ i64 drain_entries(const CycArgs& a, WaveQueue& q, i64 r0, int least, unsigned char* cnt8,
                                             i64* tile_tot) {
    wave_lds_fence();
    const int n = min(q.n, kSetQueue);
    if (n < least) return 0;
    i64 mine = 0;
    for (int i = lane_id(); i < n; i += 64)
        mine += queue_entry<S>(a, blockIdx.x % kQueueParts, r0 + q.r[i], r0, q.l[i], q.k[i], cnt8, tile_tot);
    wave_lds_fence();
    if (lane_id() == 0) q.n = 0;
    wave_lds_fence();
    return mine;
}

// A block takes `reps` rep edges.  tile_tot and cnt8 must be zero on entry;
// cnt8 is accessed in whole words.
template <int S>
__global__ __launch_bounds__(kBlock) void k_cycle_count(CycArgs a, int reps, unsigned char* __restrict__ cnt8,
                                                        i64* __restrict__ tile_tot) {
    __shared__ unsigned sets[kSetGroups * kSetWords];
    __shared__ int sb2[kSetMaxReps], sn2[kSetMaxReps];  // N(v2)
    __shared__ unsigned short runs[kSetMaxReps];        // first rep edge of each run
    __shared__ int rb1[kSetMaxReps], rd1[kSetMaxReps];  // and N(v1)
    __shared__ WaveQueue queue[kWaves];
    __shared__ int wsum[kWaves], next;
    const int tid = threadIdx.x, w = tid >> 6, wl = lane_id(), lane = tid & (kSetLanes - 1);
    const i64 r0 = (i64)(a.blk0 + xcd_block()) * reps, chunk0 = (i64)a.blk0 * reps;
    const int nr = (int)(a.R - r0 < reps ? a.R - r0 : reps);
    WaveQueue& wq = queue[w];
    i64 mine = 0;
    // runs of equal v1, lists of v2
    {
        bool head = false;
        int b1 = 0, e1 = 0;
        if (tid < nr) {
            const i64 r = r0 + tid;
            const int v1 = a.rv1[r], v2 = a.rv2[r];
            head = tid % kRunReps == 0 || a.rv1[r - 1] != v1;
            b1 = a.off[v1];
            e1 = a.off[v1 + 1];
            sb2[tid] = a.off[v2];
            sn2[tid] = a.off[v2 + 1] - sb2[tid];
        }
        const unsigned long long hm = __ballot(head);
        if (wl == 0) {
            wsum[w] = __popcll(hm);
            wq.n = 0;
        }
        if (tid == 0) next = 0;
        __syncthreads();
        int before = 0;
        for (int q = 0; q < w; ++q) before += wsum[q];
        if (head) {
            const int q = before + __popcll(hm & ((1ull << wl) - 1ull));
            runs[q] = (unsigned short)tid;
            rb1[q] = b1;
            rd1[q] = e1 - b1;
        }
    }
    __syncthreads();
    int nruns = 0;
#pragma unroll
    for (int q = 0; q < kWaves; ++q) nruns += wsum[q];
    unsigned* set = sets + tid / kSetLanes * kSetWords;
    constexpr int kMaxN2 = S == 4 ? 16 * kSetLanes : kSetLists;
    while (true) {
        int q = 0;
        if (lane == 0) q = atomicAdd(&next, 1);
        q = __shfl(q, 0, kSetLanes);
        if (!__any(q < nruns)) break;
        if (q < nruns) {
            const int ra = runs[q], rz = q + 1 < nruns ? (int)runs[q + 1] : nr, b1 = rb1[q], d1 = rd1[q];
            // the lists' bounds, two per lane, and their entries together
            int p0[2] = {0, 0}, p1[2] = {0, 0}, fill = 0;
            if (d1 <= kSetLists) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int l = lane + h * kSetLanes;
                    if (l < d1) {
                        const int y = a.adj[b1 + l];
                        p0[h] = a.off[y];
                        p1[h] = a.off[y + 1];
                    }
                    fill += p1[h] - p0[h];
                }
#pragma unroll
                for (int d = kSetLanes / 2; d >= 1; d >>= 1) fill += __shfl_xor(fill, d, kSetLanes);
            }
            const bool hub = d1 > kSetLists || fill > kSetFill;
            if (hub && a.wide) {
                const int n = (rz - ra + kWideReps - 1) / kWideReps;
                unsigned at = 0;
                if (lane == 0) at = atomicAdd(a.qcount + kQueueParts * 32, (unsigned)n);
                at = __shfl(at, 0, kSetLanes);
                for (int i = lane; i < n; i += kSetLanes) {
                    const int rf = ra + i * kWideReps;
                    a.wide[at + i] = make_int2((int)(unsigned)(r0 + rf - chunk0), min(kWideReps, rz - rf));
                }
            } else if (d1 > 0) {
                for (int k = lane; k < kSetWords; k += kSetLanes) set[k] = 0u;
                wave_lds_fence();
                auto mark = [&](int x) {
                    unsigned bits;
                    const unsigned h = set_bits<6>(x, &bits);
                    atomicOr(&set[h], bits);
                };
                // N(v2) of the rep edge, for 5-cycles the bounds of its lists,
                // are loaded while the one before is looked at
                auto ends = [&](int rl) { return rl < rz && lane < sn2[rl] ? a.adj[sb2[rl] + lane] : -1; };
                int y = ends(ra);
                if (!hub) {
                    walk_lists(a, p0[0], p1[0], min(d1, kSetLanes), mark);
                    if (d1 > kSetLanes) walk_lists(a, p0[1], p1[1], d1 - kSetLanes, mark);
                }
                int f0 = 0, f1 = 0;
                if (S == 5) {
                    if (y >= 0) {
                        f0 = a.off[y];
                        f1 = a.off[y + 1];
                    }
                    y = ends(ra + 1);
                }
                wave_lds_fence();
                for (int rl = ra; rl < rz; ++rl) {
                    const int n2 = sn2[rl], x = y, c0 = f0, c1 = f1;
                    if (S == 4) {
                        y = ends(rl + 1);
                    } else {
                        f0 = f1 = 0;
                        if (x >= 0) {
                            f0 = a.off[x];
                            f1 = a.off[x + 1];
                        }
                        y = ends(rl + 2);
                    }
                    if (n2 > kMaxN2 && a.wide) {  // v2 is a hub
                        if (lane == 0)
                            a.wide[atomicAdd(a.qcount + kQueueParts * 32, 1u)] =
                                make_int2((int)(unsigned)(r0 + rl - chunk0), 1);
                        continue;
                    }
                    auto test = [&](int m) {
                        unsigned bits;
                        const unsigned h = set_bits<6>(m, &bits);
                        return hub || !a.sets || (set[h] & bits) == bits;
                    };
                    auto hit = [&](int l2, int k) {
                        mine += push_entry<S>(a, wq, r0 + rl, chunk0, l2, k, cnt8, tile_tot);
                    };
                    const int b2 = sb2[rl];
                    if (S == 4) {
                        if (x >= 0 && test(x)) hit(0, b2 + lane);
                        for (int k = b2 + kSetLanes + lane; k < b2 + n2; k += kSetLanes)
                            if (test(a.adj[k])) hit(0, k);
                    } else {
                        find_in_lists(a, c0, c1, min(n2, kSetLanes), test, hit);
                        for (int l0 = kSetLanes; l0 < n2; l0 += kSetLanes) {
                            int g0 = 0, g1 = 0;
                            if (l0 + lane < n2) {
                                const int z = a.adj[b2 + l0 + lane];
                                g0 = a.off[z];
                                g1 = a.off[z + 1];
                            }
                            find_in_lists(a, g0, g1, min(kSetLanes, n2 - l0), test, [&](int i, int k) { hit(l0 + i, k); });
                        }
                    }
                }
            }
        }
        mine += drain_entries<S>(a, wq, chunk0, 64, cnt8, tile_tot);
    }
    mine += drain_entries<S>(a, wq, chunk0, 1, cnt8, tile_tot);
    if (a.counted) block_counted(a.counted, mine, a.xoff[r0 + nr]);
}

// The listed rep edges of hubs, up to kWideReps of one v1 per block and step.
template <int S>
__global__ __launch_bounds__(kBlock) void k_cycle_count_wide(CycArgs a, i64 chunk0, unsigned char* __restrict__ cnt8,
                                                             i64* __restrict__ tile_tot) {
    __shared__ unsigned set[kBigWords];
    __shared__ WaveQueue queue[kWaves];
    const int tid = threadIdx.x, lane = tid & (kSetLanes - 1), g = tid / kSetLanes;
    const unsigned n = a.qcount[kQueueParts * 32];
    WaveQueue& wq = queue[tid >> 6];
    if (lane_id() == 0) wq.n = 0;
    i64 mine = 0;
    for (unsigned i = blockIdx.x; i < n; i += gridDim.x) {  // uniform
        const int2 e = a.wide[i];
        const i64 ra = chunk0 + (i64)(unsigned)e.x;
        const int v1 = a.rv1[ra], b1 = a.off[v1], d1 = a.off[v1 + 1] - b1;
        __syncthreads();
        for (int k = tid; k < kBigWords; k += kBlock) set[k] = 0u;
        __syncthreads();
        for (int l0 = g; l0 < d1; l0 += kSetGroups * kSetLanes) {
            const int l = l0 + kSetGroups * lane;
            int p0 = 0, p1 = 0;
            if (l < d1) {
                const int y = a.adj[b1 + l];
                p0 = a.off[y];
                p1 = a.off[y + 1];
            }
            walk_lists(a, p0, p1, min(kSetLanes, (d1 - l0 + kSetGroups - 1) / kSetGroups), [&](int x) {
                unsigned bits;
                const unsigned h = set_bits<11>(x, &bits);
                atomicOr(&set[h], bits);
            });
        }
        __syncthreads();
        for (int c = 0; c < e.y; ++c) {
            const i64 r = ra + c;
            auto test = [&](int x) {
                unsigned bits;
                const unsigned h = set_bits<11>(x, &bits);
                return !a.sets || (set[h] & bits) == bits;
            };
            auto hit = [&](int l2, int k) {
                mine += push_entry<S>(a, wq, r, chunk0, l2, k, cnt8, tile_tot);
            };
            const int v2 = a.rv2[r], b2 = a.off[v2], n2 = a.off[v2 + 1] - b2;
            if (S == 4) {
                for (int k = b2 + tid; k < b2 + n2; k += kBlock)
                    if (test(a.adj[k])) hit(0, k);
            } else {
                for (int l0 = g; l0 < n2; l0 += kSetGroups * kSetLanes) {
                    const int l = l0 + kSetGroups * lane;
                    int p0 = 0, p1 = 0;
                    if (l < n2) {
                        const int y = a.adj[b2 + l];
                        p0 = a.off[y];
                        p1 = a.off[y + 1];
                    }
                    find_in_lists(a, p0, p1, min(kSetLanes, (n2 - l0 + kSetGroups - 1) / kSetGroups), test,
                                  [&](int i, int k) { hit(l0 + kSetGroups * i, k); });
                }
            }
            mine += drain_entries<S>(a, wq, chunk0, 64, cnt8, tile_tot);
        }
    }
    mine += drain_entries<S>(a, wq, chunk0, 1, cnt8, tile_tot);
    if (a.counted) block_counted(a.counted, mine, 0);
}

__device__ __forceinline__ void put_tri(int* t1, int* t2, int* t3, i64 g, i64 budget, int a, int b, int c) {
    if (g >= budget) return;
    const int lo = min(a, min(b, c));
    const int hi = max(a, max(b, c));
    const int md = max(min(a, b), min(max(a, b), c));
    t1[g] = lo;
    t2[g] = md;
    t3[g] = hi;
}

// One queued expansion per lane (have: the lane holds one), counted c > 0
// with its first write at `pos` in enumeration order: resolve it, move to the
// instance's triangle region on packed graphs, then write its triangles by
// the merge walk, by probing the short list into the long one, or (two long
// lists) with the whole wave.  Wave-uniform call.
template <int S>
__device__ __forceinline__ void emit_item(const CycArgs& a, bool have, i64 x, i64 pos, i64 budget, int* t1, int* t2,
                                          int* t3) {
    int v1 = 0, v2 = 0, n1 = 0, n2 = 0, qa = 0, qb = 0;
    i64 mypos = pos, tofs = 0;  // tofs: start of the instance's triangle region (packed)
    if (have) {
        resolve<S>(a, x, S == 3 ? 0 : a.tile_rep[x / kCycTile], v1, v2, n1, n2, qa, qb);
        if (a.nslot) {
            // instance q's own position, budget and region
            const int q = a.nslot[v1];
            mypos = a.slot_base[q] + (pos - a.slot_first[q]);
            budget = a.slot_budget[q];
            tofs = a.slot_out[q];
        }
    }
    const bool writes = have && mypos < budget;
    const int i0 = writes ? a.off[qa] : 0, ie = writes ? a.off[qa + 1] : 0;
    const int j0 = writes ? a.off[qb] : 0, je = writes ? a.off[qb + 1] : 0;
    const bool big = writes && (ie - i0) + (je - j0) > kHeavy;
    const bool heavy = big && min(ie - i0, je - j0) > kProbe;
    if (big && !heavy) {
        // one short list: probe its entries into the other, in order
        int sb, se, lb, le;
        short_long(a.off, qa, qb, sb, se, lb, le);
        int* u1 = t1 + tofs;
        int* u2 = t2 + tofs;
        int* u3 = t3 + tofs;
        i64 g = mypos;
        for (int i = sb; i < se && g < budget; ++i) {
            const int mid = a.adj[i];
            if (!has_partner(a.adj, sb, i, mid, lb, le)) continue;
            if (S == 3) {
                put_tri(u1, u2, u3, g++, budget, v1, v2, mid);
            } else if (S == 4) {
                put_tri(u1, u2, u3, g++, budget, v1, v2, n1);
                put_tri(u1, u2, u3, g++, budget, v2, n1, mid);
            } else {
                put_tri(u1, u2, u3, g++, budget, v1, v2, n1);
                put_tri(u1, u2, u3, g++, budget, v2, n1, mid);
                put_tri(u1, u2, u3, g++, budget, v2, mid, n2);
            }
        }
    }
    // heavy items: the whole wave walks the shorter list in order, finds each
    // entry's partner by binary search, and places the k-th common neighbour
    // at mypos + k * (S - 2) as the merge walk would
    for (unsigned long long hm = __ballot(heavy); hm; hm &= hm - 1) {
        const int h = __builtin_ctzll(hm);
        const int hqa = __builtin_amdgcn_readlane(qa, h), hqb = __builtin_amdgcn_readlane(qb, h);
        const int hv1 = __builtin_amdgcn_readlane(v1, h), hv2 = __builtin_amdgcn_readlane(v2, h);
        const int hn1 = __builtin_amdgcn_readlane(n1, h), hn2 = __builtin_amdgcn_readlane(n2, h);
        const i64 hpos = readlane64(mypos, h);
        const i64 hbud = readlane64(budget, h);
        const i64 hofs = readlane64(tofs, h);
        int sb, se, lb, le;
        short_long(a.off, hqa, hqb, sb, se, lb, le);
        const unsigned long long below = (1ull << lane_id()) - 1ull;
        i64 done = 0;
        for (int base = sb; base < se && hpos + done * (S - 2) < hbud; base += 64) {
            const int i = base + lane_id();
            int mid = 0;
            bool m = false;
            if (i < se) {
                mid = a.adj[i];
                m = has_partner(a.adj, sb, i, mid, lb, le);
            }
            const unsigned long long bm = __ballot(m);
            if (m) {
                i64 g = hpos + (done + __popcll(bm & below)) * (S - 2);
                int* u1 = t1 + hofs;
                int* u2 = t2 + hofs;
                int* u3 = t3 + hofs;
                if (S == 3) {
                    put_tri(u1, u2, u3, g, hbud, hv1, hv2, mid);
                } else if (S == 4) {
                    put_tri(u1, u2, u3, g, hbud, hv1, hv2, hn1);
                    put_tri(u1, u2, u3, g + 1, hbud, hv2, hn1, mid);
                } else {
                    put_tri(u1, u2, u3, g, hbud, hv1, hv2, hn1);
                    put_tri(u1, u2, u3, g + 1, hbud, hv2, hn1, mid);
                    put_tri(u1, u2, u3, g + 2, hbud, hv2, mid, hn2);
                }
            }
            done += __popcll(bm);
        }
    }
    if (!writes || big) return;
    t1 += tofs;
    t2 += tofs;
    t3 += tofs;
    int i = i0, j = j0;
    i64 g = mypos;
    while (i < ie && j < je && g < budget) {
        const int p = a.adj[i], q = a.adj[j];
        if (p == q) {
            const int mid = p;
            if (S == 3) {
                put_tri(t1, t2, t3, g++, budget, v1, v2, mid);
            } else if (S == 4) {
                put_tri(t1, t2, t3, g++, budget, v1, v2, n1);
                put_tri(t1, t2, t3, g++, budget, v2, n1, mid);
            } else {
                put_tri(t1, t2, t3, g++, budget, v1, v2, n1);
                put_tri(t1, t2, t3, g++, budget, v2, n1, mid);
                put_tri(t1, t2, t3, g++, budget, v2, mid, n2);
            }
        }
        i += (p <= q);
        j += (q <= p);
    }
}

__device__ __forceinline__ i64 wave_excl_scan64(i64 v, i64* total) {
    i64 x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const i64 t = __shfl_up(x, d, 64);
        if (lane_id() >= d) x += t;
    }
    *total = readlane64(x, 63);
    return x - v;
}

// Dense emit: one thread per expansion (block = one count tile), write
// positions by a block scan of the counts.  Used when a large share of the
// expansions have mids (every lane then has one to write).
template <int S>
__global__ __launch_bounds__(kBlock) void k_cycle_emit_dense(CycArgs a, const unsigned char* __restrict__ cnt8,
                                                             const i64* __restrict__ tile_off, i64 base, i64 budget,
                                                             int* __restrict__ t1, int* __restrict__ t2,
                                                             int* __restrict__ t3) {
    __shared__ i64 ws[kWaves];
    // plain block order: tiles past the budget exit at once, and keeping the
    // working tiles spread over all XCDs balances them
    const unsigned blk = blockIdx.x;
    const bool packed = a.nslot != nullptr;
    if (tile_off[blk + 1] == tile_off[blk]) return;  // uniform: the tile writes nothing
    const i64 tstart = (packed ? 0 : base) + tile_off[blk];
    if (!packed && tstart >= budget) return;  // uniform per block
    const i64 x = (i64)blk * kCycTile + threadIdx.x;
    int c = x < a.X ? (int)cnt8[x] : 0;
    {
        // a saturated count (255): count again (by the wave when both lists
        // are long)
        int v1 = 0, v2 = 0, n1 = 0, n2 = 0, qa = 0, qb = 0;
        bool wave = false;
        if (c == 255) {
            resolve<S>(a, x, S == 3 ? 0 : a.tile_rep[blk], v1, v2, n1, n2, qa, qb);
            int sb, se, lb, le;
            short_long(a.off, qa, qb, sb, se, lb, le);
            if (se - sb <= kProbe) c = probe_count(a.adj, sb, se, lb, le);
            else wave = true;
        }
        for (unsigned long long hm = __ballot(wave); hm; hm &= hm - 1) {
            const int h = __builtin_ctzll(hm);
            const int s = wave_count_common(a.off, a.adj, __builtin_amdgcn_readlane(qa, h),
                                            __builtin_amdgcn_readlane(qb, h));
            if (lane_id() == h) c = s;
        }
    }
    i64 tot;
    const i64 pos = tstart + block_excl_scan((i64)c * (S - 2), ws, &tot);
    emit_item<S>(a, c > 0, x, pos, budget, t1, t2, t3);
}

// Dense emit of 3-cycles for up to kFewReps rep edges: a block of 1024 threads
// per count tile, groups of 16 lanes write one rep edge's triangles each, the
// k-th entry of the shorter list that has a partner at the k-th place, a wave
// where both lists are long.  (k_cycle_emit_dense<3> walks lists of up to 96
// entries by one thread and longer ones one after another in the wave: 127 us a
// launch on 50021 nodes, 43 here.)
__global__ __launch_bounds__(kFewThreads) void k_cycle_emit3_few(CycArgs a, const unsigned char* __restrict__ cnt8,
                                                                 const i64* __restrict__ tile_off, i64 base,
                                                                 i64 budget, int* __restrict__ t1,
                                                                 int* __restrict__ t2, int* __restrict__ t3) {
    __shared__ int cnt[kCycTile];
    __shared__ i64 pos[kCycTile];
    __shared__ i64 wtot[kCycTile / 64];
    const int tid = threadIdx.x, w = tid >> 6, gl = tid & 15;
    const bool packed = a.nslot != nullptr;
    if (tile_off[blockIdx.x + 1] == tile_off[blockIdx.x]) return;  // uniform: the tile writes nothing
    const i64 tstart = (packed ? 0 : base) + tile_off[blockIdx.x];
    if (!packed && tstart >= budget) return;  // uniform
    const i64 r0 = (i64)blockIdx.x * kCycTile;
    if (tid < kCycTile) cnt[tid] = r0 + tid < a.R ? (int)cnt8[r0 + tid] : 0;
    __syncthreads();
    for (int q = w; q < kCycTile; q += kFewThreads / 64) {
        if (cnt[q] != 255) continue;  // uniform within the wave; else saturated: count again
        const int c = wave_count_common(a.off, a.adj, __builtin_amdgcn_readfirstlane(a.rv1[r0 + q]),
                                        __builtin_amdgcn_readfirstlane(a.rv2[r0 + q]));
        if (lane_id() == 0) cnt[q] = c;
    }
    __syncthreads();
    i64 before = 0, tot = 0;
    if (w < kCycTile / 64) {
        before = wave_excl_scan64((i64)cnt[tid], &tot);
        if (lane_id() == 0) wtot[w] = tot;
    }
    __syncthreads();
    if (w < kCycTile / 64) {
        for (int q = 0; q < w; ++q) before += wtot[q];
        pos[tid] = tstart + before;
    }
    __syncthreads();
    // lanes sub, sub + width, ... of `width` share rep edge q
    auto emit = [&](int q, int sub, int width, unsigned long long share) {
        const int v1 = a.rv1[r0 + q], v2 = a.rv2[r0 + q];
        i64 g = pos[q], last = budget;
        int *u1 = t1, *u2 = t2, *u3 = t3;
        if (packed) {
            // the instance's own position, budget and region
            const int z = a.nslot[v1];
            g = a.slot_base[z] + (g - a.slot_first[z]);
            last = a.slot_budget[z];
            u1 += a.slot_out[z];
            u2 += a.slot_out[z];
            u3 += a.slot_out[z];
        }
        int sb, se, lb, le;
        short_long(a.off, v1, v2, sb, se, lb, le);
        const unsigned long long below = share & ((1ull << lane_id()) - 1ull);
        for (int i0 = sb; i0 < se && g < last; i0 += width) {  // uniform among the sharing lanes
            const int i = i0 + sub;
            int mid = 0;
            bool m = false;
            if (i < se) {
                mid = a.adj[i];
                m = has_partner(a.adj, sb, i, mid, lb, le);
            }
            const unsigned long long bm = __ballot(m) & share;
            if (m) put_tri(u1, u2, u3, g + __popcll(bm & below), last, v1, v2, mid);
            g += __popcll(bm);
        }
    };
    auto shorter = [&](int q) {
        const int v1 = a.rv1[r0 + q], v2 = a.rv2[r0 + q];
        return min(a.off[v1 + 1] - a.off[v1], a.off[v2 + 1] - a.off[v2]);
    };
    for (int q = tid >> 4; q < kCycTile; q += kFewGroups)
        if (cnt[q] > 0 && shorter(q) <= kFewGroup) emit(q, gl, 16, 0xffffull << (lane_id() & 48));
    for (int q = w; q < kCycTile; q += kFewThreads / 64)
        if (cnt[q] > 0 && shorter(q) > kFewGroup) emit(q, lane_id(), 64, ~0ull);
}

// Sparse emit: one wave per block walks a contiguous range of count tiles in
// order.  Each tile's 256 counts are read four per lane (expansion order is
// lane-major), a wave scan turns them into write positions (tile start +
// the counts before), and the expansions with mids are queued in LDS; every
// 64 queued expansions are written by the 64 lanes at once (emit_item).
// Most expansions have no mid, so lanes stay busy instead of idling beside
// the few that write.  Saturated counts (255) are counted again first.
constexpr int kEmitQueue = 320;  // at most 63 waiting + 256 from one tile
// Count tiles a queued-emit wave walks, one after another: at most
// kEmitTilesPerWave, and several only once there are more than the waves that
// the chip holds (71^3 grid, eight each -> one: 4-cycles 49 -> 24 us a launch,
// 5-cycles 83 -> 47, 3-cycles 25 -> 10).
constexpr i64 kEmitWaves = 8192;
constexpr i64 kEmitTilesPerWave = 8;

template <int S>
__global__ __launch_bounds__(64) void k_cycle_emit(CycArgs a, const unsigned char* __restrict__ cnt8,
                                                   const i64* __restrict__ tile_off, i64 ntiles, i64 per_block,
                                                   i64 base, i64 budget, int* __restrict__ t1, int* __restrict__ t2,
                                                   int* __restrict__ t3) {
    __shared__ i64 qx[kEmitQueue];
    __shared__ i64 qp[kEmitQueue];
    const int lane = lane_id();
    const bool packed = a.nslot != nullptr;
    const i64 tb = (i64)blockIdx.x * per_block;
    const i64 te = tb + per_block < ntiles ? tb + per_block : ntiles;
    int qn = 0;  // queued expansions (wave-uniform)
    for (i64 t = tb; t < te; ++t) {
        const i64 o0 = tile_off[t], o1 = tile_off[t + 1];
        if (o1 == o0) continue;  // the tile writes nothing (uniform)
        const i64 tstart = (packed ? 0 : base) + o0;
        if (!packed && tstart >= budget) break;  // later tiles start later still
        const i64 x0 = t * kCycTile + 4 * lane;
        int c[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) c[k] = x0 + k < a.X ? (int)cnt8[x0 + k] : 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const bool sat = c[k] == 255;
            if (__ballot(sat) == 0ull) continue;
            // the count saturated its byte: count again (by the wave when
            // both lists are long)
            int v1 = 0, v2 = 0, n1 = 0, n2 = 0, qa = 0, qb = 0;
            bool wave = false;
            if (sat) {
                resolve<S>(a, x0 + k, S == 3 ? 0 : a.tile_rep[t], v1, v2, n1, n2, qa, qb);
                int sb, se, lb, le;
                short_long(a.off, qa, qb, sb, se, lb, le);
                if (se - sb <= kProbe) c[k] = probe_count(a.adj, sb, se, lb, le);
                else wave = true;
            }
            for (unsigned long long hm = __ballot(wave); hm; hm &= hm - 1) {
                const int h = __builtin_ctzll(hm);
                const int s = wave_count_common(a.off, a.adj, __builtin_amdgcn_readlane(qa, h),
                                                __builtin_amdgcn_readlane(qb, h));
                if (lane == h) c[k] = s;
            }
        }
        i64 tot;
        i64 p = tstart + wave_excl_scan64((i64)(c[0] + c[1] + c[2] + c[3]) * (S - 2), &tot);
        const int nz = (c[0] > 0) + (c[1] > 0) + (c[2] > 0) + (c[3] > 0);
        int zx = nz;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int u = __shfl_up(zx, d, 64);
            if (lane >= d) zx += u;
        }
        const int ztot = __builtin_amdgcn_readlane(zx, 63);
        int slot = qn + zx - nz;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (c[k] > 0) {
                qx[slot] = x0 + k;
                qp[slot] = p;
                ++slot;
            }
            p += (i64)c[k] * (S - 2);
        }
        qn += ztot;
        __syncthreads();
        while (qn >= 64) {
            qn -= 64;
            const i64 x = qx[qn + lane], pos = qp[qn + lane];
            __syncthreads();
            emit_item<S>(a, true, x, pos, budget, t1, t2, t3);
        }
    }
    __syncthreads();
    const bool have = lane < qn;
    emit_item<S>(a, have, have ? qx[lane] : 0, have ? qp[lane] : 0, budget, t1, t2, t3);
}

// The emit over `ntiles` count tiles with W attempted writes in all: the
// per-expansion form when at least one expansion in kEmitDenseShare has a
// mid (W counts S - 2 writes per mid), else the queued form.
constexpr i64 kEmitDenseShare = 4;
template <int S>
static void launch_emit(Ctx& ctx, const CycArgs& a, const unsigned char* cnt8, const i64* tile_off, i64 ntiles,
                        i64 W, i64 base, i64 budget, int* t1, int* t2, int* t3) {
    const int forced = emit_form_forced();
    if (forced == 1 || (forced == 0 && W * kEmitDenseShare >= (i64)(S - 2) * a.X)) {
        if (S == 3 && a.R <= kFewReps)
            k_cycle_emit3_few<<<(unsigned)ntiles, kFewThreads, 0, ctx.stream>>>(a, cnt8, tile_off, base, budget, t1, t2,
                                                                               t3);
        else
            k_cycle_emit_dense<S><<<(unsigned)ntiles, kBlock, 0, ctx.stream>>>(a, cnt8, tile_off, base, budget, t1, t2,
                                                                               t3);
    } else {
        const i64 per = std::min<i64>(std::max<i64>(ntiles / kEmitWaves, 1), kEmitTilesPerWave);
        k_cycle_emit<S><<<(unsigned)((ntiles + per - 1) / per), 64, 0, ctx.stream>>>(a, cnt8, tile_off, ntiles, per,
                                                                                     base, budget, t1, t2, t3);
    }
    RAMA_LAUNCHED();
}

static void launch_count3(Ctx& ctx, const CycArgs& a, unsigned ntiles, unsigned char* cnt8, i64* tile) {
    if (a.R <= kFewReps)
        k_cycle_count3_few<<<ntiles, kFewThreads, 0, ctx.stream>>>(a, cnt8, tile);
    else
        k_cycle_count3<<<ntiles, kBlock, 0, ctx.stream>>>(a, cnt8, tile);
    RAMA_LAUNCHED();
}

// Which form counts a single instance's 4- or 5-cycles.  The sets form pays
// about 1.2 ns per entry that passes its filter (true mids, and the filter's own
// errors where 2-hop neighbourhoods are large), the lists form 20 to 50 ps per
// expansion of short lists (5-cycles, through the 2-hop tables) and 300 ps of
// long ones.  So the count starts with the sets and goes over to the lists once
// a chunk has passed on that many entries per expansion: full 5-cycle counts of
// a random graph of degree 20 (5% and more pass) 14.4 ms by sets, 6.2 by lists,
// of a 12-nearest-neighbour graph (two mids per expansion) 2.7 and 0.14, of a
// random graph of degree 8 0.38 and 0.85.  A few thousand rep edges of short
// lists start with the lists (a launch of 378 at a mid per expansion 17 ms by
// sets, whose few groups resolve them in turn, and 0.27).  Where the count may go
// on past kFewWrites writes per rep edge, as verbose ones do, the first chunk is
// smaller, and long lists too are walked from the start.  A pack's counts run to
// the end over all kinds of instances and take the lists (48 mixed instances,
// PD+: 5.3 s by sets, 1.2 by lists).
template <int S>
constexpr i64 kShortLists = S == 4 ? 32 : 1024;  // expansions per rep edge, on average
template <int S>
constexpr double kDenseShare = S == 4 ? 0.25 : 0.03125;
constexpr double kDenseLong = 0.25;
constexpr i64 kFewReps45 = 8192;
constexpr i64 kFewWrites = 4;

// Before a 4- or 5-cycle count, in one launch (a memset each costs the host
// more than this kernel): tile_rep[t] = rep edge containing the first expansion
// of tile t; tile totals, count bytes (whole 16-byte words) and counters
// cleared.
__global__ __launch_bounds__(kBlock) void k_count_begin(const i64* __restrict__ xoff, i64 R, int* __restrict__ tile_rep,
                                                        i64* __restrict__ tile, i64 ntiles, uint4* __restrict__ cnt8,
                                                        i64 words, i64* __restrict__ counted, int ncounted,
                                                        unsigned* __restrict__ qcount, int nqcount) {
    const i64 i0 = (i64)blockIdx.x * kBlock + threadIdx.x, stride = (i64)gridDim.x * kBlock;
    for (i64 r = i0; r < R; r += stride) {
        const i64 b = xoff[r], e = xoff[r + 1];
        for (i64 t = (b + kCycTile - 1) / kCycTile; t * kCycTile < e; ++t) tile_rep[t] = (int)r;
    }
    for (i64 i = i0; i < words; i += stride) cnt8[i] = make_uint4(0u, 0u, 0u, 0u);
    for (i64 i = i0; i < ntiles; i += stride) tile[i] = 0;
    if (i0 < ncounted) counted[i0] = 0;
    for (i64 i = i0; i < nqcount; i += stride) qcount[i] = 0u;
}

// Work of one count launch for the profiler (only while it is on): the
// expansions the launch covers and the neighbour-list entries a merge walk
// of each expansion's two lists reads, deg(a) + deg(b); the launch covers rep
// edges [lo, hi).  nsum[v] = sum of the degrees of v's neighbours.
template <int S>
static void count_work(Ctx& ctx, const Csr& G, const int* rv1, const int* rv2, const i64* nsum, i64 lo, i64 hi,
                       double& x, double& entries) {
    const int* OFF = G.off.get();
    x = entries = 0.0;
    if (hi <= lo) return;
    if (S == 3) {
        x = (double)(hi - lo);
        entries = (double)reduce<i64>(
            ctx,
            [=] __device__(i64 k) {
                const int v = rv1[lo + k], u = rv2[lo + k];
                return (i64)(OFF[v + 1] - OFF[v]) + (i64)(OFF[u + 1] - OFF[u]);
            },
            hi - lo, (i64)0, OpSum());
    } else if (S == 4) {
        x = (double)reduce<i64>(
            ctx, [=] __device__(i64 k) { const int v = rv1[lo + k]; return (i64)(OFF[v + 1] - OFF[v]); }, hi - lo,
            (i64)0, OpSum());
        entries = (double)reduce<i64>(
            ctx,
            [=] __device__(i64 k) {
                const int v = rv1[lo + k], u = rv2[lo + k];
                return nsum[v] + (i64)(OFF[v + 1] - OFF[v]) * (i64)(OFF[u + 1] - OFF[u]);
            },
            hi - lo, (i64)0, OpSum());
    } else {
        x = (double)reduce<i64>(
            ctx,
            [=] __device__(i64 k) {
                const int v = rv1[lo + k], u = rv2[lo + k];
                return (i64)(OFF[v + 1] - OFF[v]) * (i64)(OFF[u + 1] - OFF[u]);
            },
            hi - lo, (i64)0, OpSum());
        entries = (double)reduce<i64>(
            ctx,
            [=] __device__(i64 k) {
                const int v = rv1[lo + k], u = rv2[lo + k];
                return nsum[v] * (i64)(OFF[u + 1] - OFF[u]) + nsum[u] * (i64)(OFF[v + 1] - OFF[v]);
            },
            hi - lo, (i64)0, OpSum());
    }
}

// Rep edges per block of a 4- or 5-cycle count: few where there are few, so
// that every CU has some.
static int count_reps(i64 R) {
    return (int)std::min<i64>(std::max<i64>((R + 2047) / 2048, kSetMinReps), kSetMaxReps);
}

// The queue of a 4- or 5-cycle count over R rep edges with X expansions, and
// the list of hubs' rep edges.  Both are dispensable: without memory for the
// queue entries are resolved as they come, without the list hubs' rep edges
// are treated as the others, unfiltered.
struct CountQueue {
    DBuf<int3> entries;
    DBuf<int2> wide;
    DBuf<unsigned> count;
    template <class T>
    static DBuf<T> try_buf(Ctx& ctx, i64 n) {
        try {
            return ctx.buf<T>(n);
        } catch (const Error& e) {
            if (e.status != RAMA_ERR_OOM) throw;
            return DBuf<T>();
        }
    }
    CountQueue(Ctx& ctx, int S, i64 R, i64 X, CycArgs& a) {
        count = ctx.buf<unsigned>((kQueueParts + 1) * 32);
        a.qcount = count.get();
        if (count_queue_part("list")) wide = try_buf<int2>(ctx, R);
        a.wide = wide.get();
        a.qcap = (int)std::min<i64>(X / (S == 4 ? 16 : 64) / kQueueParts + 1024, (i64)1 << 24);
        if (count_queue_part("queue")) entries = try_buf<int3>(ctx, (i64)kQueueParts * a.qcap);
        a.queue = entries.get();
        if (!a.queue) a.qcap = 0;
    }
};
// k_count_begin for a stage of R rep edges and a.X expansions.
static void count_begin(Ctx& ctx, const CycArgs& a, int* tile_rep, i64* tile, unsigned char* cnt8) {
    const i64 ntiles = (a.X + kCycTile - 1) / kCycTile, words = cnt8 ? (a.X + 15) / 16 : 0;
    const i64 n = std::max<i64>(std::max<i64>(a.R, std::max(words, ntiles)), (kQueueParts + 1) * 32);
    k_count_begin<<<(unsigned)std::min<i64>((n + kBlock - 1) / kBlock, 4096), kBlock, 0, ctx.stream>>>(
        a.xoff, a.R, tile_rep, tile, ntiles, reinterpret_cast<uint4*>(cnt8), words, a.counted,
        a.counted ? kCountedLines * 16 : 0, a.qcount, a.qcount ? (kQueueParts + 1) * 32 : 0);
    RAMA_LAUNCHED();
}
// Counts blocks [a.blk0, a.blk0 + n) of `reps` rep edges.
template <int S>
static void count_blocks(Ctx& ctx, const CycArgs& a, unsigned n, int reps, unsigned char* cnt8, i64* tile) {
    const i64 r0 = (i64)a.blk0 * reps;
    if (a.blk0 > 0) ctx.zero(a.qcount, (kQueueParts + 1) * 32);
    k_cycle_count<S><<<n, kBlock, 0, ctx.stream>>>(a, reps, cnt8, tile);
    RAMA_LAUNCHED();
    if (a.wide) {
        k_cycle_count_wide<S><<<std::min(n, 1024u), kBlock, 0, ctx.stream>>>(a, r0, cnt8, tile);
        RAMA_LAUNCHED();
    }
    const unsigned per_part = std::min<unsigned>(std::max<unsigned>(n * (unsigned)reps / 4096u, 1u), 64u);
    k_cycle_resolve<S><<<kQueueParts * per_part, kBlock, 0, ctx.stream>>>(a, r0, cnt8, tile);
    RAMA_LAUNCHED();
}

// Counts rep edges [r0, a.R) by walking lists, after k_count_begin has cleared
// the count bytes and tile totals, in launches of nblk blocks in all.
template <int S>
struct CountLists {
    CycArgs a;  // of the rep edges from r0 on
    DBuf<i64> yoff;
    DBuf<int> ytile_rep;
    i64 Y = 0;
    unsigned nblk = 0;
    int tables = 0;
    CountLists(Ctx& ctx, const CycArgs& all, i64 r0, int n_nodes) : a(all) {
        a.rv1 += r0;
        a.rv2 += r0;
        a.xoff += r0;
        a.R -= r0;
        if (S == 4) {
            nblk = grid_for(a.R);
            return;
        }
        // thread space: one thread per (rep edge, neighbour of v2)
        tables = a.sets && n_nodes < kT5MaxNode ? 1 : 0;
        yoff = ctx.buf<i64>(a.R + 1);
        const int* OFF = a.off;
        const int* rv2 = a.rv2;
        i64* ym = ctx.mirror<i64>();
        scan_exclusive<i64>(ctx, [=] __device__(i64 r) { const int u = rv2[r]; return (i64)(OFF[u + 1] - OFF[u]); },
                            yoff.get(), a.R, ym);
        ctx.read_mirror(yoff.get() + a.R, ym, &Y);
        const i64 ytiles = (Y + kCycTile - 1) / kCycTile;
        RAMA_REQUIRE(ytiles < ((i64)1 << 31), "too many cycle expansions");
        nblk = (unsigned)ytiles;
        if (Y == 0) return;
        ytile_rep = ctx.buf<int>(ytiles);
        k_count_begin<<<(unsigned)std::min<i64>((a.R + kBlock - 1) / kBlock, 4096), kBlock, 0, ctx.stream>>>(
            yoff.get(), a.R, ytile_rep.get(), nullptr, 0, nullptr, 0, nullptr, 0, nullptr, 0);
        RAMA_LAUNCHED();
    }
    // Blocks [first, first + n).
    void run(Ctx& ctx, unsigned first, unsigned n, unsigned char* cnt8, i64* tile) {
        if (n == 0) return;
        a.blk0 = first;
        if (S == 4)
            k_cycle_count4<<<n, kBlock, 0, ctx.stream>>>(a, cnt8, tile);
        else
            k_cycle_count5<<<n, kBlock, 0, ctx.stream>>>(a, yoff.get(), ytile_rep.get(), Y, tables, cnt8, tile);
        RAMA_LAUNCHED();
    }
};

// Runs one stage over all expansions; returns the number of attempted writes.
template <int S>
static i64 run_stage(Ctx& ctx, const Csr& G, const int* rv1, const int* rv2, i64 R, i64 base, i64 budget,
                     Triangles& T) {
    const int* OFF = G.off.get();
    DBuf<i64> xoff;  // 3-cycles: expansion = rep edge, no offsets
    if (S > 3) xoff = ctx.buf<i64>(R + 1);
    i64* xm = ctx.mirror<i64>();
    if (S == 4) {
        scan_exclusive<i64>(ctx, [=] __device__(i64 r) { const int v = rv1[r]; return (i64)(OFF[v + 1] - OFF[v]); },
                            xoff.get(), R, xm);
    } else if (S == 5) {
        scan_exclusive<i64>(
            ctx,
            [=] __device__(i64 r) {
                const int v = rv1[r], u = rv2[r];
                return (i64)(OFF[v + 1] - OFF[v]) * (i64)(OFF[u + 1] - OFF[u]);
            },
            xoff.get(), R, xm);
    }
    i64 X = R;
    if (S > 3) ctx.read_mirror(xoff.get() + R, xm, &X);
    if (ctx.verbose && S > 3) std::printf("%d-cycles: number of expansions: %lld\n", S, (long long)X);
    if (X == 0) return 0;
    const i64 ntiles = (X + kCycTile - 1) / kCycTile;
    DBuf<int> tile_rep;
    if (S > 3) {
        tile_rep = ctx.buf<int>(ntiles);
    }
    CycArgs a{OFF, G.adj.get(), rv1, rv2, S > 3 ? xoff.get() : nullptr, S > 3 ? tile_rep.get() : nullptr, R, X};
    a.sets = cycle_tables_on() ? 1 : 0;
    DBuf<unsigned char> cnt8 = ctx.buf<unsigned char>((X + 15) / 16 * 16);  // cleared and counted up in whole words
    DBuf<i64> tile = ctx.buf<i64>(ntiles + 1);
    RAMA_REQUIRE(ntiles < ((i64)1 << 31), "too many cycle expansions");
    // profiling only: each count launch's expansions and list entries, and
    // their merge-walk bytes (4 per list entry, 8 of list bounds per expansion)
    const bool work_on = prof::wants(S == 3 ? "cycles3_count" : (S == 4 ? "cycles4_count" : "cycles5_count"));
    DBuf<i64> nsum;
    if (work_on && S > 3) {
        nsum = ctx.buf<i64>(G.n);
        i64* NS = nsum.get();
        const int* ADJ = G.adj.get();
        for_each(ctx, G.n, [=] __device__(i64 v) {
            i64 s = 0;
            for (int k = OFF[v]; k < OFF[v + 1]; ++k) s += OFF[ADJ[k] + 1] - OFF[ADJ[k]];
            NS[v] = s;
        });
    }
    double wx = 0.0, wy = 0.0;
    if (S == 3) {
        if (work_on) count_work<3>(ctx, G, rv1, rv2, nullptr, 0, R, wx, wy);
        prof::Scope ps(ctx, "cycles3_count", 4.0 * wy + 8.0 * wx, wx, wy);
        launch_count3(ctx, a, (unsigned)ntiles, cnt8.get(), tile.get());
    }
    // Stages 4 and 5 count in chunks of blocks, each a prefix of the
    // expansion order, and stop once the attempted writes reach the budget
    // left (budget - base): expansions past that point write nothing, so
    // the triangles, the stage's outcome (total >= budget left) and every
    // later decision are those of a full count.  Only the returned total is
    // then a lower bound of the full one; verbose runs count everything, as
    // they print it.
    //
    // The chunks take the sets form as long as few entries pass, the lists form
    // from there on (kDenseShare).
    i64 tiles_used = ntiles;
    if constexpr (S > 3) {
        DBuf<i64> cnt = ctx.buf<i64>(kCountedLines * 16);
        a.counted = cnt.get();
        const int forced = count_form_forced();
        const bool early = !ctx.verbose && budget > base;
        const i64 need = budget - base;
        const bool few = early && need <= kFewWrites * R, lengthy = X > kShortLists<S> * R;
        const bool sets = forced ? forced == 1 : !(lengthy ? !few : R < kFewReps45);
        std::optional<CountQueue> queue;  // of the sets form
        if (sets) queue.emplace(ctx, S, R, X, a);
        count_begin(ctx, a, tile_rep.get(), tile.get(), cnt8.get());
        i64 hc[3] = {0, 0, 0};  // attempted writes, end of the expansions counted, entries resolved
        auto totals = [&] {
            i64 lines[kCountedLines * 16];
            ctx.read(cnt.get(), lines, kCountedLines * 16);
            hc[0] = hc[1] = hc[2] = 0;
            for (int k = 0; k < kCountedLines; ++k) {
                hc[0] += lines[k * 16];
                hc[1] = std::max(hc[1], lines[k * 16 + 1]);
                hc[2] += lines[k * 16 + 2];
            }
        };
        // the chunk after `done` of n blocks: cycle_chunk_pct percent (default
        // 125) of the blocks that the rate so far says reach the budget (all
        // the rest when it says they will not)
        auto next_chunk = [&](unsigned done, unsigned n, double per_block) {
            const double grow = 0.01 * (double)tune::get(tune::CycleChunkPct, X);
            const double want = early && per_block > 0.0 ? grow * (double)(need - hc[0]) / per_block + 64.0 : 1e30;
            return want >= (double)(n - done) ? n - done : (unsigned)want;
        };
        i64 rdone = 0;
        bool stopped = false;
        if (sets) {
            const int reps = count_reps(R);
            const unsigned nblk = (unsigned)((R + reps - 1) / reps);
            // the first chunk: a sixteenth of the blocks (a count that runs to
            // the end pays this launch's tail once; smaller first chunks cost D
            // mode on the 2D grid 5 ms, larger ones overshoot budgets), less
            // where the count may go on past many mids per rep edge
            unsigned done = 0, chunk = few ? std::max<unsigned>(nblk / 16, 256u) : std::max<unsigned>(nblk / 64, 32u);
            if (forced == 1 && !early) chunk = nblk;
            while (done < nblk) {
                const unsigned n = std::min(chunk, nblk - done);
                a.blk0 = done;
                if (work_on)
                    count_work<S>(ctx, G, rv1, rv2, nsum.get(), rdone, std::min<i64>((i64)(done + n) * reps, R), wx, wy);
                {
                    prof::Scope ps(ctx, S == 4 ? "cycles4_count" : "cycles5_count", 4.0 * wy + 8.0 * wx, wx, wy);
                    count_blocks<S>(ctx, a, n, reps, cnt8.get(), tile.get());
                }
                done += n;
                rdone = std::min<i64>((i64)done * reps, R);
                if (done >= nblk) break;
                totals();
                stopped = early && hc[0] >= need;
                if (stopped) break;
                if (!forced && hc[2] >= (lengthy ? kDenseLong : kDenseShare<S>) * hc[1]) break;
                chunk = next_chunk(done, nblk, (double)hc[0] / (double)done);
            }
        }
        queue.reset();
        const i64 by_sets = rdone;
        if (rdone < R && !stopped) {
            CountLists<S> lists(ctx, a, rdone, G.n);
            const i64 w0 = hc[0];
            unsigned done = 0, chunk = early ? std::max<unsigned>(lists.nblk / 16, 256u) : lists.nblk;
            while (done < lists.nblk) {
                const unsigned n = std::min(chunk, lists.nblk - done);
                if (work_on && done == 0) count_work<S>(ctx, G, rv1, rv2, nsum.get(), rdone, R, wx, wy);
                {
                    // profiling: the first chunk is booked with the work of all
                    prof::Scope ps(ctx, S == 4 ? "cycles4_count" : "cycles5_count", 4.0 * wy + 8.0 * wx, wx, wy);
                    lists.run(ctx, done, n, cnt8.get(), tile.get());
                }
                wx = wy = 0.0;
                done += n;
                if (done >= lists.nblk) break;
                totals();
                stopped = hc[0] >= need;
                if (stopped) break;
                chunk = next_chunk(done, lists.nblk, (double)(hc[0] - w0) / (double)done);
            }
        }
        if (std::getenv("RAMA_CYCLE_STATS")) {
            totals();
            std::fprintf(stderr, "%d-cycle count: %lld rep edges (%lld by sets), %lld expansions, %lld counted, %lld mids, "
                         "%lld entries resolved\n",
                         S, (long long)R, (long long)by_sets, (long long)X, (long long)hc[1],
                         (long long)(hc[0] / (S - 2)), (long long)hc[2]);
        }
        if (stopped) {
            // counted expansions [0, hc[1]): emit the tiles they touch; the
            // rest of the last tile contributes nothing
            tiles_used = (hc[1] + kCycTile - 1) / kCycTile;
        }
    }
    i64* wm = ctx.mirror<i64>();
    scan_exclusive_arr<i64>(ctx, tile.get(), tile.get(), tiles_used, wm);
    i64 W;
    ctx.read_mirror(tile.get() + tiles_used, wm, &W);
    if (W > 0 && base < budget) {
        prof::Scope ps(ctx, S == 3 ? "cycles3_emit" : (S == 4 ? "cycles4_emit" : "cycles5_emit"), 0.0);
        launch_emit<S>(ctx, a, cnt8.get(), tile.get(), tiles_used, W, base, budget, T.t1.get(), T.t2.get(),
                       T.t3.get());
    }
    return W;
}

// One stage over several packed instances.  Instance q's writes go to its
// triangle region (d_out[q] onward) at positions continuing from d_base[q],
// below d_budget[q]; h_total[q] receives its attempted writes (the stage's
// return value in the single-instance form).
template <int S>
void run_stage_packed(Ctx& ctx, const Csr& G, const int* rv1, const int* rv2, i64 R, const int* nslot, int Q,
                      const i64* d_base, const i64* d_budget, const i64* d_out, int* t1, int* t2, int* t3,
                      i64* h_total) {
    for (int q = 0; q < Q; ++q) h_total[q] = 0;
    if (R == 0) return;
    const int* OFF = G.off.get();
    DBuf<i64> xoff;  // 3-cycles: expansion = rep edge, no offsets
    if (S > 3) xoff = ctx.buf<i64>(R + 1);
    i64* xm = ctx.mirror<i64>();
    if (S == 4) {
        scan_exclusive<i64>(ctx, [=] __device__(i64 r) { const int v = rv1[r]; return (i64)(OFF[v + 1] - OFF[v]); },
                            xoff.get(), R, xm);
    } else if (S == 5) {
        scan_exclusive<i64>(
            ctx,
            [=] __device__(i64 r) {
                const int v = rv1[r], u = rv2[r];
                return (i64)(OFF[v + 1] - OFF[v]) * (i64)(OFF[u + 1] - OFF[u]);
            },
            xoff.get(), R, xm);
    }
    i64 X = R;
    if (S > 3) ctx.read_mirror(xoff.get() + R, xm, &X);
    if (X == 0) return;
    const i64 ntiles = (X + kCycTile - 1) / kCycTile;
    RAMA_REQUIRE(ntiles < ((i64)1 << 31), "too many cycle expansions");
    DBuf<int> tile_rep;
    if (S > 3) {
        tile_rep = ctx.buf<int>(ntiles);
    }
    DBuf<i64> slot = ctx.buf<i64>(2 * (i64)Q + 1);  // [0, Q) totals, [Q, 2Q] their exclusive scan
    i64* TOT = slot.get();
    ctx.zero(TOT, Q);
    CycArgs a{OFF, G.adj.get(), rv1, rv2, S > 3 ? xoff.get() : nullptr, S > 3 ? tile_rep.get() : nullptr, R, X};
    a.sets = cycle_tables_on() ? 1 : 0;
    a.nslot = nslot;
    a.slot_total = TOT;
    a.slot_first = TOT + Q;
    a.slot_base = d_base;
    a.slot_budget = d_budget;
    a.slot_out = d_out;
    DBuf<unsigned char> cnt8 = ctx.buf<unsigned char>((X + 15) / 16 * 16);  // cleared and counted up in whole words
    DBuf<i64> tile = ctx.buf<i64>(ntiles + 1);
    if (S > 3 && std::getenv("RAMA_CYCLE_STATS"))
        std::fprintf(stderr, "%d-cycle count of a pack: %lld rep edges (%lld by sets), %lld expansions\n", S, (long long)R,
                     (long long)(count_form_forced() == 1 ? R : 0), (long long)X);
    if constexpr (S == 3) {
        launch_count3(ctx, a, (unsigned)ntiles, cnt8.get(), tile.get());
    } else if (count_form_forced() != 1) {
        // a pack's counts run to the end, past any number of mids
        count_begin(ctx, a, tile_rep.get(), tile.get(), nullptr);
        CountLists<S> lists(ctx, a, 0, G.n);
        lists.run(ctx, 0, lists.nblk, cnt8.get(), tile.get());
    } else {
        const int reps = count_reps(R);
        CountQueue queue(ctx, S, R, X, a);
        count_begin(ctx, a, tile_rep.get(), tile.get(), cnt8.get());
        count_blocks<S>(ctx, a, (unsigned)((R + reps - 1) / reps), reps, cnt8.get(), tile.get());
    }
    scan_exclusive_arr<i64>(ctx, tile.get(), tile.get(), ntiles);
    scan_exclusive_arr<i64>(ctx, TOT, TOT + Q, Q);
    ctx.d2h(h_total, TOT, Q);
    i64 W = 0;
    for (int q = 0; q < Q; ++q) W += h_total[q];
    if (W > 0) {
        launch_emit<S>(ctx, a, cnt8.get(), tile.get(), ntiles, W, 0, 0, t1, t2, t3);
    }
}
template void run_stage_packed<3>(Ctx&, const Csr&, const int*, const int*, i64, const int*, int, const i64*,
                                  const i64*, const i64*, int*, int*, int*, i64*);
template void run_stage_packed<4>(Ctx&, const Csr&, const int*, const int*, i64, const int*, int, const i64*,
                                  const i64*, const i64*, int*, int*, int*, i64*);
template void run_stage_packed<5>(Ctx&, const Csr&, const int*, const int*, i64, const int*, int, const i64*,
                                  const i64*, const i64*, int*, int*, int*, i64*);

// rearrange_triangles / normalize_triangles (include/rama_utils.h:325-363)
// on the first `valid` slots: drop triangles with a repeated vertex, sort
// lexicographically, remove duplicates.  Returns the new count.
i64 rearrange_triangles(Ctx& ctx, Triangles& T, i64 valid, int n_nodes) {
    if (valid <= 0) return 0;
    int* A = T.t1.get();
    int* B = T.t2.get();
    int* C = T.t3.get();
    const int kb = bits_for(n_nodes > 1 ? n_nodes - 1 : 1);
    DBuf<int> cnt = ctx.buf<int>(1);  // unique triangles
    int* CNT = cnt.get();
    DBuf<u64> keys = ctx.buf<u64>(valid);
    DBuf<u32> vals = ctx.buf<u32>(valid);
    u64* K = keys.get();
    u32* V = vals.get();
    if (3 * kb <= 64) {
        // key = the ordered triple (write_triangle already orders it; kept
        // for foreign input); a triangle with a repeated vertex gets the
        // all-ones key of the sort width, which no real triangle has
        // (first < second < third), so it sorts last and is cut below
        const u64 pad = (1ull << (3 * kb)) - 1ull;
        for_each(ctx, valid, [=] __device__(i64 t) {
            const int a = A[t], b = B[t], c = C[t];
            const bool degen = a == b || a == c || b == c;
            const u32 lo = (u32)min(a, min(b, c)), md = (u32)max(min(a, b), min(max(a, b), c)),
                      hi = (u32)max(a, max(b, c));
            K[t] = degen ? pad : ((u64)lo << (2 * kb)) | ((u64)md << kb) | (u64)hi;
            V[t] = (u32)t;
        });
        {
            prof::Site site_("triangles");
            radix_sort_pairs(ctx, keys, vals, valid, 3 * kb);
        }
        K = keys.get();  // an odd pass count hands back the scratch buffers
        const u64 m1 = (1ull << kb) - 1ull;
        // keep the first of each run of equal keys; decode the triple in place
        select_into(
            ctx, valid, [=] __device__(i64 q) { return K[q] != pad && (q == 0 || K[q] != K[q - 1]); },
            [=] __device__(i64 q, int o) {
                const u64 k = K[q];
                A[o] = (int)(k >> (2 * kb));
                B[o] = (int)((k >> kb) & m1);
                C[o] = (int)(k & m1);
            },
            CNT, ctx.mirror<int>());
        int h;
        ctx.read_mirror(CNT, ctx.mirror<int>(), &h);
        return h;
    }
    // ids too wide for one key: two stable passes, by third id and then by
    // (first, second), on the ordered triples kept in S1..S3 (-1: repeated vertex)
    DBuf<int> s1 = ctx.buf<int>(valid), s2 = ctx.buf<int>(valid), s3 = ctx.buf<int>(valid);
    int* S1 = s1.get();
    int* S2 = s2.get();
    int* S3 = s3.get();
    const u64 pad1 = (1ull << kb) - 1ull, pad2 = (1ull << (2 * kb)) - 1ull;
    for_each(ctx, valid, [=] __device__(i64 t) {
        const int a = A[t], b = B[t], c = C[t];
        const bool degen = a == b || a == c || b == c;
        S1[t] = degen ? -1 : min(a, min(b, c));
        S2[t] = degen ? -1 : max(min(a, b), min(max(a, b), c));
        S3[t] = degen ? -1 : max(a, max(b, c));
        K[t] = degen ? pad1 : (u64)(u32)S3[t];
        V[t] = (u32)t;
    });
    prof::Site site_("triangles");
    radix_sort_pairs(ctx, keys, vals, valid, kb);
    K = keys.get();
    V = vals.get();
    for_each(ctx, valid, [=] __device__(i64 q) {
        const u32 o = V[q];
        K[q] = S1[o] < 0 ? pad2 : ((u64)(u32)S1[o] << kb) | (u64)(u32)S2[o];
    });
    radix_sort_pairs(ctx, keys, vals, valid, 2 * kb);
    K = keys.get();
    V = vals.get();
    select_into(
        ctx, valid,
        [=] __device__(i64 q) {
            const u32 a = V[q];
            if (S1[a] < 0) return false;
            if (q == 0) return true;
            const u32 b = V[q - 1];
            return S1[a] != S1[b] || S2[a] != S2[b] || S3[a] != S3[b];
        },
        [=] __device__(i64 q, int o) {
            const u32 a = V[q];
            A[o] = S1[a];
            B[o] = S2[a];
            C[o] = S3[a];
        },
        CNT, ctx.mirror<int>());
    int h;
    ctx.read_mirror(CNT, ctx.mirror<int>(), &h);
    return h;
}

void normalize_triangles(Ctx& ctx, Triangles& T) { T.n = rearrange_triangles(ctx, T, T.n, 1 << 30); }

// The thresholds, the attractive CSR and the repulsive edges of A.
static void cycle_search_inputs(Ctx& ctx, const DCoo& A, float tol, CycleSearch& cs) {
    const float* W = A.val.get();
    const int N = A.max_dim();
    // determine_threshold (:170-174): thr = min(c) * tol; attractive c > -thr
    // (is_positive_edge), repulsive c < thr (is_neg_edge).  The minimum and
    // both class sizes come back in one read.
    struct Sizes {
        float mn;
        float pad;
        u64 counts;  // attractive count << 32 | repulsive count
    };
    DBuf<Sizes> sz = ctx.buf<Sizes>(1);
    Sizes* SZ = sz.get();
    Sizes* SM = ctx.mirror<Sizes>();
    reduce_to<float>(ctx, [=] __device__(i64 e) { return W[e]; }, A.nnz, 3.402823466e38f, OpMin(), &SZ->mn,
                     SM ? &SM->mn : nullptr);
    reduce_to<u64>(
        ctx,
        [=] __device__(i64 e) {
            const float t = SZ->mn * tol;
            return ((u64)(W[e] > -1.0f * t) << 32) | (u64)(W[e] < t);
        },
        A.nnz, (u64)0, OpSum(), &SZ->counts, SM ? &SM->counts : nullptr);
    Sizes h;
    ctx.read_mirror(SZ, SM, &h);
    const float thr = h.mn * tol;
    const i64 npos = (i64)(h.counts >> 32);
    const i64 R = (i64)(h.counts & 0xffffffffull);
    cs.R = R;
    cs.none = npos == 0 || R == 0;
    if (cs.none) return;
    if (A.sym || ctx.last_cycles_empty) {
        // the contraction that made A left its full symmetric CSR, or the
        // last search found nothing, so this dual pass likely leaves A as it
        // is: build that CSR once (the matching reuses it) and take the
        // attractive part out of it
        if (!A.sym) A.sym = std::make_shared<Csr>(symmetric_csr(ctx, A.row.get(), A.col.get(), W, A.nnz, N, false, 0.0f));
        cs.G = csr_filter(ctx, *A.sym, -1.0f * thr, 2 * npos);
    } else {
        cs.G = symmetric_csr(ctx, A.row.get(), A.col.get(), W, A.nnz, N, true, -1.0f * thr, npos);
    }
    cs.rv1 = ctx.buf<int>(R);
    cs.rv2 = ctx.buf<int>(R);
    {
        int* X1 = cs.rv1.get();
        int* X2 = cs.rv2.get();
        const int* AR = A.row.get();
        const int* AC = A.col.get();
        select_into_loaded(
            ctx, A.nnz, [=] __device__(i64 e) { return W[e] < thr; },
            [=] __device__(i64 e) { return make_int2(AR[e], AC[e]); },
            [=] __device__(i64, int q, int2 rc) {
                X1[q] = rc.x;
                X2[q] = rc.y;
            },
            reinterpret_cast<int*>(&SZ->pad));
    }
}

// conflicted_cycles_cuda (src/conflicted_cycles_cuda.cu:222-343), followed by
// the normalisation the message-passing constructor applies.
//
// `known` carries a search that found nothing over to the next one on the same
// graph: the dual pass searches for cycles of up to 3, up to 4, up to 5, and as
// long as nothing is found the graph stays, so each search only has its
// longest cycles left to look at.  A round without cycles of up to five nodes
// then counts three times instead of six and builds its inputs once: 71^3 grid
// PD+ 35.2 -> 31.8 ms, 192^3 116.8 -> 109.8.
Triangles conflicted_cycles(Ctx& ctx, const DCoo& A, int max_len, float factor, float tol, CycleSearch* known) {
    Triangles T;
    if (max_len > 5) throw Error(RAMA_ERR_INVALID, "max_cycle_length should be <= 5. Received: " + std::to_string(max_len));
    if (max_len < 3 || A.nnz == 0) return T;
    CycleSearch own;
    CycleSearch& cs = known ? *known : own;
    if (cs.none) {
        ctx.last_cycles_empty = true;
        return T;
    }
    const int N = A.max_dim();
    if (cs.empty_to == 0) cycle_search_inputs(ctx, A, tol, cs);
    if (cs.none) {
        ctx.last_cycles_empty = true;
        return T;
    }
    const i64 R = cs.R;
    const Csr& G = cs.G;
    const int* rv1 = cs.rv1.get();
    const int* rv2 = cs.rv2.get();
    const i64 budget = (i64)(int)(factor * (float)R);
    T.t1 = ctx.buf<int>(budget > 0 ? budget : 1);
    T.t2 = ctx.buf<int>(budget > 0 ? budget : 1);
    T.t3 = ctx.buf<int>(budget > 0 ? budget : 1);
    const int from = cs.empty_to;  // stages up to this length find nothing
    i64 count = from >= 3 ? 0 : run_stage<3>(ctx, G, rv1, rv2, R, 0, budget, T);
    if (ctx.verbose) std::printf("3-cycles: found # of triangles: %lld, budget: %lld\n", (long long)count, (long long)budget);
    if (max_len >= 4 && count < budget && from < 4) {
        count = rearrange_triangles(ctx, T, count, N);
        count += run_stage<4>(ctx, G, rv1, rv2, R, count, budget, T);
        if (ctx.verbose) std::printf("4-cycles: found # of triangles: %lld, budget: %lld\n", (long long)count, (long long)budget);
    }
    if (max_len >= 5 && count < budget && from < 5) {
        count = rearrange_triangles(ctx, T, count, N);
        count += run_stage<5>(ctx, G, rv1, rv2, R, count, budget, T);
        if (ctx.verbose) std::printf("5-cycles: found # of triangles: %lld, budget: %lld\n", (long long)count, (long long)budget);
    }
    T.raw = count < budget ? count : budget;
    T.n = rearrange_triangles(ctx, T, T.raw, N);
    T.max_id = N - 1;
    ctx.last_cycles_empty = T.raw == 0;
    cs.empty_to = T.raw == 0 && budget > 0 ? max_len : 0;
    return T;
}

}  // namespace rama
