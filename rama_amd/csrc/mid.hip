// mid.hip — matching-contraction rounds queued without reading anything back.
//
// After the first contractions a graph has some ten or hundred thousand
// edges for dozens of rounds.  Stage by stage such a round is 33 launches and
// 4 host waits, about 0.25 ms whatever its size, most of it launch gaps and
// 2 us kernels; with searches for cycles of up to five nodes 48 to 59 launches
// and 18 waits, 0.45 to 0.6 ms.  Here a round is nine to eleven launches (three
// more where matchings are long) whose sizes are read on the device: the host
// queues several rounds over buffers sized by the graph it last saw, then reads one
// small state.  A round that the driver has to handle itself (a conflicted cycle, a
// matching of more than six rounds, a bucket too large for LDS, hubs whose cycle
// test takes too long, the switch to the spanning forest) raises an outcome word of
// the state, and the launches queued behind it leave at once.  So does the first
// matching of more than three rounds: from it on six are queued.
//
//   k_mid_begin    sums of the matching threshold, attractive neighbour lists
//   k_mid_prune    (cycles of 4 and 5) the lists without their leaves
//   k_mid_cycles   (rounds with duals) is there a conflicted cycle
//   k_mid_pick     best neighbours, a launch per matching round (3 or 6)
//   k_mid_resolve  per round's outcome: matched and representative counts
//   k_mid_keys     round that ends the matching, labels, row buckets and each
//                  tile of edges' count per bucket
//   k_mid_scatter  the edges, in both directions, to their row bucket
//   k_mid_bucket   one block per bucket: stable LDS sort, runs of equal keys
//                  summed
//   k_mid_finish   compaction into the contracted graph, its CSR and state
//
// No launch stores an outcome word that it tests itself: its blocks start at
// different times, and the waves of a late one could read the word differently
// and part before a barrier.  `stop` is stored by the finish of the round before
// (all of this round's launches test it), `found` by the cycle test, and by the
// begin where a cost is not a number, `ended` by the keys and `skewed` by the
// scatter (only the launches behind test them); the finish folds them into the next
// state's `stop`.  They are loaded together, not one after another, and a state fills
// a line of its own: every launch begins with them (1024x2048 grid P 15.3 ms otherwise,
// 14.9 so).
//
// The matching needs no matched flags: a vertex v is matched once
// best[best[v]] == v, since matched vertices keep their best.  So a matching
// round is one launch that reads the round before's best array instead of two.
//
// Bound by each launch's chain of dependent loads (0.5 to 1 us each: what the
// launch before wrote comes from memory, not from this XCD's L2), hence the
// merged launches and the loads issued together.  Measured per round of
// 20k to 200k edges: about 60 us on the device (picks 3 x 5.3, bucket 11,
// keys 12, scatter 9, begin 7, finish 6, resolve and prune 4.6 each, cycles 4 to
// 20) against 220 to 320 us stage by stage, 450 to 600 with cycles of up to five
// nodes.  Solves with and without this form (the other forms on): 1024x2048 grid
// with long-range edges P 20.2 -> 15.6 ms, PD 55.2 -> 49.5; 257x509 PD 18.7 -> 15.2;
// 71^3 grid PD+ 31.8 -> 24.3; rounds of 7k to 2k edges of a 187x211 grid PD+ 1.85 ->
// 0.54.  Up to 2^18 edges, the lists whose contraction leaves the symmetric CSR.
//
// Every sum and order is the stage-by-stage path's, so are the results.  (A round
// with a cost that is not a number is the driver's.)
#include "rama_internal.hpp"
#include "tuning.hpp"

namespace rama {

constexpr int kMidGroup = 8;          // lanes per vertex or edge
constexpr int kMidTileEdges = 2048;   // forward edges per scatter tile (each in both directions)
constexpr int kMidThreads = 512;      // keys, scatter and bucket blocks
constexpr int kMidWaves = kMidThreads / 64;
constexpr int kMidEdgeItems = kMidTileEdges / kMidThreads;
constexpr int kMidItems = 16;         // sorted items per thread at most
constexpr int kMidBucketMax = kMidThreads * kMidItems;
constexpr int kMidPicks = 6;          // matching rounds queued per contraction round at most
constexpr int kMidFewPicks = 3;       // and at first
constexpr int kMidVertBlocks = kMidMaxNodes / kBlock;
constexpr int kMidGrid = 1024;        // grid bound of the strided launches
constexpr int kMidFound = 1, kMidTooMuch = 2;  // MidState::found

struct MidGraph {
    int* row;    // forward edges, (row, col) order
    int* col;
    float* val;
    int* off;    // symmetric CSR
    int* adj;
    float* w;
};

struct MidArgs {
    MidGraph g, to;               // this round's graph and the contracted one
    MidState* st;                 // this round's state
    MidState* nx;                 // the next round's
    MidState* mirror;             // host copy, last queued round only
    double* psum;                 // threshold partials
    int* pcnt;
    int* best[kMidPicks];
    u64* rbits[kMidPicks];        // bit v: v keeps its id under round t's outcome
    int* rcnt[kMidPicks];         // per 256 vertices: representatives
    int* mcnt[kMidPicks];         // per 256 vertices: matched
    int* cur;                     // vertex -> its label after the contraction
    u64* ekey;                    // per forward edge: new labels and their row buckets (mid_pack)
    int* rb;                      // 257: first new label of each row bucket
    int* table;                   // per tile: 256 digit counts
    u32* key;                     // scattered items: low key bits and cost
    u32* val;
    int* bstart;                  // 257 bucket starts
    u32* hkey;                    // per bucket, from its start: merged entries
    float* hval;
    int* bstat;                   // 256 x 8: entries, forward entries, largest row, col, kept col, bad, min (bits)
    int* label;
    int* pos;                     // attractive neighbours, from each row's offset on
    int* npos;                    // and how many
    int* npath;                   // and how many of them a path can pass through
    int n0;
    int picks;                    // matching rounds queued
    int len;                      // longest conflicted cycles looked for (0: none)
    int small_words;              // hand over from this many words of bit matrix down
    int small_edges;              // hand over to small_rounds from this many edges down (0: never)
    float mult, ratio, tol;
};

__device__ __forceinline__ int mid_bits(int max_label) {
    int kb = 1;
    while (kb < 31 && (1 << kb) <= max_label) ++kb;
    return kb;
}

// Row buckets hold about equal shares of the entries: a new label's bucket is
// where its representative's row starts in the present CSR, in 256ths of the
// entries (monotone in the label).  Equal ranges of labels instead put up to
// five times the mean into one bucket: supernodes gather.
__device__ __forceinline__ int mid_bucket_of(int off, float scale) { return min(255, (int)((float)off * scale)); }
// Labels below 2^18 and their buckets in one word.
__device__ __forceinline__ u64 mid_pack(u32 lo, u32 hi, u32 blo, u32 bhi) {
    return ((u64)lo << 34) | ((u64)hi << 16) | ((u64)blo << 8) | (u64)bhi;
}
static_assert(kMidMaxNodes <= 1 << 18, "labels in mid_pack");

// Per row v of the present graph: the entries l in [off[v], end(v)) that keep
// accepts, as get(l), in order from the row's offset on in pos, their number in
// count[v].  A group of lanes per row, a wave per long row; get may read pos.
template <class Keep, class Get, class End>
__device__ __forceinline__ void mid_compact(const MidArgs& a, int n, int* count, Keep keep, Get get, End end) {
    constexpr int kLong = 16 * kMidGroup;
    const int lane = lane_id(), sub = lane % kMidGroup, first = lane - sub;
    const unsigned long long lt = (1ull << lane) - 1ull;
    const unsigned long long group = ((1ull << kMidGroup) - 1ull) << first;
    const int stride = (int)gridDim.x * (kBlock / kMidGroup);
    for (int v0 = ((int)xcd_block() * (kBlock / 64) + (threadIdx.x >> 6)) * (64 / kMidGroup); v0 < n; v0 += stride) {
        const int v = v0 + lane / kMidGroup;
        const int b0 = v < n ? a.g.off[v] : 0, e0 = v < n ? end(v) : 0;
        const bool big = e0 - b0 > kLong;
        int k = 0;
        for (int l = b0 + sub; !big && l - sub < e0; l += kMidGroup) {  // uniform per group
            const bool on = l < e0 && keep(l);
            const int x = on ? get(l) : 0;
            const unsigned long long m = __ballot(on) & group;
            if (on) a.pos[b0 + k + __popcll(m & lt)] = x;
            k += __popcll(m);
        }
        if (sub == 0 && v < n && !big) count[v] = k;
        for (unsigned long long rows = __ballot(sub == 0 && big); rows; rows &= rows - 1ull) {
            const int src = __ffsll(rows) - 1;
            const int rb = __shfl(b0, src, 64), re = __shfl(e0, src, 64);
            int q = 0;
            for (int l = rb + lane; l - lane < re; l += 64) {
                const bool on = l < re && keep(l);
                const int x = on ? get(l) : 0;
                const unsigned long long m = __ballot(on);
                if (on) a.pos[rb + q + __popcll(m & lt)] = x;
                q += __popcll(m);
            }
            if (lane == src) count[v] = q;
        }
    }
}

// Threshold partials in reduce_pair_to's blocks and order, and each row's
// attractive neighbours, in order from the row's offset on: a group of lanes
// per row, a wave per long row.
__global__ __launch_bounds__(kBlock) void k_mid_begin(MidArgs a) {
    __shared__ double ws[kWaves];
    __shared__ int wi[kWaves];
    MidState* st = a.st;
    if (st->stop) return;
    const int nnz = 2 * st->nf, n = st->n;
    const int nb = min((nnz + kBlock - 1) / kBlock, (int)kReduceMaxBlocks);
    if ((int)blockIdx.x < nb) {  // uniform per block; the grid covers nb
        double s = 0.0;
        int c = 0;
        bool nan = false;
        for (int i = blockIdx.x * kBlock + threadIdx.x; i < nnz; i += nb * kBlock) {
            const float x = a.g.w[i];
            nan |= x != x;
            s += x >= 0.0f ? (double)x : 0.0;
            c += x >= 0.0f ? 1 : 0;
        }
        // what the launches stage by stage pick from comparisons with a NaN hangs
        // on their shape: the driver's round
        if (nan) __hip_atomic_fetch_or(&st->found, kMidFound, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const double r = block_reduce(s, OpSum(), ws);
        const int rc = block_reduce(c, OpSum(), wi);
        if (threadIdx.x == 0) {
            a.psum[blockIdx.x] = r;
            a.pcnt[blockIdx.x] = rc;
        }
    }
    if (a.len == 0) return;
    const float at = -1.0f * (st->minw * a.tol);
    mid_compact(
        a, n, a.npos, [&](int l) { return a.g.w[l] > at; }, [&](int l) { return a.g.adj[l]; },
        [&](int v) { return a.g.off[v + 1]; });
}

// An attractive path from u to v passes only through vertices with two
// attractive neighbours.  In late rounds most have one: stars remain, of which
// a matching contracts one leaf each.  Without the leaves the lists are one or
// two entries long (k_mid_cycles with them: 123 us a round of the 71^3 grid).
__global__ __launch_bounds__(kBlock) void k_mid_prune(MidArgs a) {
    const MidState* st = a.st;
    if (st->stop) return;
    mid_compact(
        a, st->n, a.npath, [&](int l) { return a.npos[a.pos[l]] > 1; }, [&](int l) { return a.pos[l]; },
        [&](int v) { return a.g.off[v] + a.npos[v]; });
}

// Is x in the ascending list p[0..n)?
__device__ __forceinline__ bool mid_has(const int* __restrict__ p, int n, int x) {
    int lo = 0, hi = n;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (p[mid] < x) lo = mid + 1; else hi = mid;
    }
    return lo < n && p[lo] == x;
}

// Lanes of kLanes that share one of nu x nv pairs: eight where the pairs are
// few, one where they fill the lanes.  Counts past kLanes are all the same here,
// so they are cut before they are multiplied.
constexpr __host__ __device__ int mid_pair_lanes(int nu, int nv, int lanes) {
    const int pairs = (nu < lanes ? nu : lanes) * (nv < lanes ? nv : lanes);
    return pairs * 2 > lanes ? 1 : (pairs * 4 > lanes ? 2 : (pairs * 8 > lanes ? 4 : 8));
}
static_assert(mid_pair_lanes(1, 1, 8) == 8 && mid_pair_lanes(2, 1, 64) == 8 && mid_pair_lanes(3, 3, 64) == 4 &&
              mid_pair_lanes(5, 6, 64) == 2 && mid_pair_lanes(33, 1, 64) == 1, "shares of a pair");
static_assert(mid_pair_lanes(kMidMaxNodes, kMidMaxNodes, 64) == 1, "two hubs (no overflow in a constant)");

// What a lane of the cycle test may load one after another.  In the rounds it is
// made for a lane loads some ten to fifty words; hubs joined by a repulsive edge
// can ask for 10^8 pairs of one wave, and a queued round would take seconds.  A
// lane that runs out hands the round to the driver, whose search spreads such
// edges over the chip.  2048 loads are about 0.8 ms, a searched round's time:
// 257x509 grid with long-range edges, PD+, 45.5 ms, 48 with 8192 loads, 61 without
// a limit; 97x211 22.6, 24.7 and 34.9; grids without long-range edges and random
// graphs the same.
constexpr int kMidWork = 2048;
// Loads of a search in n ascending entries.
__device__ __forceinline__ int mid_search_loads(int n) { return 34 - __clz(n | 1); }

// Is there an attractive path of at most len - 1 edges between u and v, whose
// lists of neighbours to pass through have nu and nv entries?  kLanes lanes
// take the pairs of neighbours (x, y), one each or, of few pairs, a part of
// their lists, and ask for x = y, x next to y, a common neighbour.  left: the
// loads that the lane still has; below zero it gave up.
template <int kLanes>
__device__ __forceinline__ bool mid_joined(const MidArgs& a, const int* num, int u, int v, int nu, int nv, int sub,
                                           int& left) {
    const int* off = a.g.off;
    const int* pu = a.pos + off[u];
    const int* pv = a.pos + off[v];
    const int lanes = mid_pair_lanes(nu, nv, kLanes);
    const int p0 = sub / lanes, step = kLanes / lanes, k0 = sub % lanes;
    int x = p0 / nv, y = p0 % nv;
    const int dx = step / nv, dy = step % nv;
    while (x < nu) {
        const int vx = pu[x], vy = pv[y];
        const int* px = a.pos + off[vx];
        const int* py = a.pos + off[vy];
        int nx = num[vx], ny = num[vy];
        int z = vy;  // looked for in x's list
        if (nx > ny) {
            const int* p = px;
            px = py;
            py = p;
            const int k = nx;
            nx = ny;
            ny = k;
            z = vx;
        }
        const int each = a.len > 4 ? 1 + mid_search_loads(ny) : 1;
        left -= 4;
        bool hit = vx == vy;
        for (int k = k0; k < nx && left >= 0; k += lanes) {
            const int q = px[k];
            hit |= q == z || (a.len > 4 && mid_has(py, ny, q));
            left -= each;
        }
        if (hit) return true;
        if (left < 0) return false;
        x += dx;
        y += dy;
        if (y >= nv) {
            y -= nv;
            ++x;
        }
    }
    return false;
}

// The same for paths of two edges: the shorter list's entries, one per lane, in
// the longer list.
template <int kLanes>
__device__ __forceinline__ bool mid_common(const MidArgs& a, int u, int v, int nu, int nv, int sub, int& left) {
    const int* ps = a.pos + a.g.off[nu < nv ? u : v];
    const int* pl = a.pos + a.g.off[nu < nv ? v : u];
    const int ns = min(nu, nv), nl = max(nu, nv), each = 1 + mid_search_loads(nl);
    for (int k = sub; k < ns && left >= 0; k += kLanes) {
        if (mid_has(pl, nl, ps[k])) return true;
        left -= each;
    }
    return false;
}

// Are a repulsive edge's ends joined by an attractive path of at most len - 1
// edges?  A conflicted cycle exists exactly then: the shortest such path has
// no chord.  A group of lanes per edge, the wave for one with many pairs of
// neighbours.
//
// In the rounds that get here (the search before found nothing) that is one or
// two pairs per edge, of two or three neighbours each: bound by the chain of
// six loads, hence a group for every edge (groups that take eight edges in
// turn: 80 us at 7k edges), and by the few edges between hubs.
__global__ __launch_bounds__(kBlock) void k_mid_cycles(MidArgs a) {
    MidState* st = a.st;
    if (st->stop) return;
    constexpr int kMany = 4 * kMidGroup;  // pairs, or entries of the shorter list
    const int nf = st->nf, lane = lane_id(), sub = lane % kMidGroup;
    const float t = st->minw * a.tol;
    const int* num = a.len > 3 ? a.npath : a.npos;  // of the lists to walk
    const int stride = (int)gridDim.x * (kBlock / kMidGroup);
    bool hit = false;
    int left = kMidWork;
    for (int e0 = ((int)xcd_block() * kWaves + (threadIdx.x >> 6)) * (64 / kMidGroup); e0 < nf; e0 += stride) {
        const int e = e0 + lane / kMidGroup;
        int u = 0, v = 0, nu = 0, nv = 0;
        if (e < nf) {
            const float c = a.g.val[e];
            u = a.g.row[e];
            v = a.g.col[e];
            if (c < t) {
                nu = num[u];
                nv = num[v];
            }
        }
        const bool on = nu > 0 && nv > 0;
        const bool many = on && (a.len == 3 ? min(nu, nv) > kMany : (float)nu * (float)nv > (float)kMany);
        if (on && !many)
            hit = a.len == 3 ? mid_common<kMidGroup>(a, u, v, nu, nv, sub, left)
                             : mid_joined<kMidGroup>(a, num, u, v, nu, nv, sub, left);
        for (unsigned long long rest = __ballot(many && sub == 0); rest && !__any(hit || left < 0); rest &= rest - 1ull) {
            const int src = __ffsll(rest) - 1;
            const int su = __shfl(u, src, 64), sv = __shfl(v, src, 64), mu = __shfl(nu, src, 64), mv = __shfl(nv, src, 64);
            hit = a.len == 3 ? mid_common<64>(a, su, sv, mu, mv, lane, left)
                             : mid_joined<64>(a, num, su, sv, mu, mv, lane, left);
        }
        if (__any(hit || left < 0) || __hip_atomic_load(&st->found, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
    }
    const int found = __any(hit) ? kMidFound : (__any(left < 0) ? kMidTooMuch : 0);
    if (found && lane == 0) __hip_atomic_fetch_or(&st->found, found, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Matching round t's best neighbours (k_pick_best's choice: strongest
// unmatched neighbour above the threshold, first in row order on ties) on
// round t - 1's outcome.  Round 0 combines the threshold first.
template <bool kFirst>
__global__ __launch_bounds__(kBlock) void k_mid_pick(MidArgs a, int t) {
    __shared__ double ws[kWaves];
    __shared__ int wi[kWaves];
    MidState* st = a.st;
    if (st->stop | st->found) return;
    const int n = st->n;
    float thr;
    bool any;
    if (kFirst) {
        const int nnz = 2 * st->nf;
        const int nb = min((nnz + kBlock - 1) / kBlock, (int)kReduceMaxBlocks);
        const double sum = combine_partials(a.psum, (unsigned)nb, 0.0, OpSum(), ws);
        const int cnt = combine_partials(a.pcnt, (unsigned)nb, 0, OpSum(), wi);
        thr = a.mult * (float)sum / (float)cnt;
        any = cnt != 0 && !(thr < 0.0f);
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            st->thr = thr;
            st->any = any ? 1 : 0;
        }
    } else {
        thr = st->thr;
        any = st->any != 0;
    }
    const int* prev = !kFirst ? a.best[t - 1] : nullptr;
    int* best = a.best[t];
    const int sub = threadIdx.x % kMidGroup;
    const int stride = (int)gridDim.x * (kBlock / kMidGroup);
    for (int v = (int)xcd_block() * (kBlock / kMidGroup) + threadIdx.x / kMidGroup; v < n; v += stride) {
        const int b0 = a.g.off[v], e0 = a.g.off[v + 1];
        int pb = -1;
        if (!kFirst) {
            pb = prev[v];
            if (pb >= 0 && prev[pb] != v) pb = -1;  // not matched
        }
        const int e = any && pb < 0 ? e0 : b0;
        float bv = thr;
        int bp = 0x7fffffff, bn = -1;
        for (int l = b0 + sub; l < e; l += kMidGroup) {
            const float c = a.g.w[l];
            const int u = a.g.adj[l];
            if (!(c > bv) || u == v) continue;
            if (!kFirst) {
                const int pu = prev[u];
                if (pu >= 0 && prev[pu] == u) continue;  // matched
            }
            bv = c;
            bp = l;
            bn = u;
        }
#pragma unroll
        for (int d = kMidGroup / 2; d >= 1; d >>= 1) {
            const float ov = __shfl_xor(bv, d, kMidGroup);
            const int op = __shfl_xor(bp, d, kMidGroup);
            const int on = __shfl_xor(bn, d, kMidGroup);
            if (ov > bv || (ov == bv && op < bp)) {
                bv = ov;
                bp = op;
                bn = on;
            }
        }
        if (sub == 0) best[v] = pb >= 0 ? pb : bn;
    }
}

// After each matching round t: which vertices keep their id (all but the
// larger end of a pair), as bits, and counts per 256 vertices.
__global__ __launch_bounds__(kBlock) void k_mid_resolve(MidArgs a) {
    __shared__ int wr[kMidPicks][kWaves], wm[kMidPicks][kWaves];
    const MidState* st = a.st;
    if (st->stop | st->found) return;
    const int n = st->n;
    const int v = blockIdx.x * kBlock + threadIdx.x;
    if ((int)(blockIdx.x * kBlock) >= n) return;  // uniform per block
    const int w = threadIdx.x >> 6;
#pragma unroll
    for (int t = 0; t < kMidPicks; ++t) {
        if (t >= a.picks) break;
        const int b = v < n ? a.best[t][v] : -1;
        const bool m = b >= 0 && a.best[t][b] == v;
        const unsigned long long reps = __ballot(v < n && !(m && b < v));
        const unsigned long long mm = __ballot(m);
        if (lane_id() == 0) {
            a.rbits[t][(blockIdx.x * kBlock >> 6) + w] = reps;
            wr[t][w] = __popcll(reps);
            wm[t][w] = __popcll(mm);
        }
    }
    __syncthreads();
    if ((int)threadIdx.x < a.picks) {
        int r = 0, m = 0;
#pragma unroll
        for (int k = 0; k < kWaves; ++k) {
            r += wr[threadIdx.x][k];
            m += wm[threadIdx.x][k];
        }
        a.rcnt[threadIdx.x][blockIdx.x] = r;
        a.mcnt[threadIdx.x][blockIdx.x] = m;
    }
}

// Exclusive scan over a block of kMidThreads.
__device__ __forceinline__ int mid_block_scan(int x, int* ws, int* total) {
    const int lane = lane_id(), w = threadIdx.x >> 6;
    const int inc = wave_incl_scan(x);
    __syncthreads();
    if (lane == 63) ws[w] = inc;
    __syncthreads();
    int before = 0, tot = 0;
#pragma unroll
    for (int k = 0; k < kMidWaves; ++k) {
        const int t = ws[k];
        before += k < w ? t : 0;
        tot += t;
    }
    *total = tot;
    return before + inc - x;
}

// The matching's end (match_round_active's stop rule on the counts), the
// compressed labels (a vertex's rank among the representatives, from its
// bit's prefix) and each forward edge's new ends; one tile of edges per
// block, with the tile's counts per row bucket in both directions.
__global__ __launch_bounds__(kMidThreads) void k_mid_keys(MidArgs a) {
    __shared__ int pre[kMidVertBlocks];
    __shared__ int ws[kMidWaves];
    __shared__ int cnt[kMidPicks][kMidWaves];
    __shared__ int hist[256];
    MidState* st = a.st;
    const int tid = threadIdx.x, lane = lane_id(), w = tid >> 6;
    const int n = st->n, nf = st->nf, nblk = (n + kBlock - 1) / kBlock, found = st->found;
    if (st->stop) return;
    if (found) {
        if (blockIdx.x == 0 && tid == 0) st->ended = found & kMidFound ? kSmallCycles : kMidSkew;
        return;
    }
    // the edges' ends and what the counts need are loaded together: a chain
    // of dependent loads costs this kernel more than its bytes
    const int e0 = blockIdx.x * kMidTileEdges;
    int er[kMidEdgeItems], ec[kMidEdgeItems];
#pragma unroll
    for (int k = 0; k < kMidEdgeItems; ++k) {
        const int e = e0 + k * kMidThreads + tid;
        er[k] = e < nf ? a.g.row[e] : 0;
        ec[k] = e < nf ? a.g.col[e] : 0;
    }
    constexpr int kPer = kMidVertBlocks / kMidThreads;
    int rc[kMidPicks][kPer], mc[kMidPicks];
#pragma unroll
    for (int t = 0; t < kMidPicks; ++t) {
        mc[t] = 0;
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int b = tid * kPer + k;
            const bool on = t < a.picks && b < nblk;
            rc[t][k] = on ? a.rcnt[t][b] : 0;
            mc[t] += on ? a.mcnt[t][b] : 0;
        }
    }
#pragma unroll
    for (int t = 0; t < kMidPicks; ++t) {
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) mc[t] += __shfl_xor(mc[t], d, 64);
        if (lane == 0) cnt[t][w] = mc[t];
    }
    if (tid < 256) hist[tid] = 0;
    __syncthreads();
    int tr = 0, matched = 0;
    bool ended = false;
#pragma unroll
    for (int t = 0; t < kMidPicks; ++t) {
        if (ended || t >= a.picks) break;  // uniform
        int cur = 0;
#pragma unroll
        for (int k = 0; k < kMidWaves; ++k) cur += cnt[t][k];
        const int nw = cur - matched;
        const float rel = nw / (matched + 1.0f);
        tr = t;
        ended = nw == 0 || rel < 0.1f;
        matched = cur;
    }
    const int outcome = !ended ? kMidMatching : (matched == 0 ? kSmallDone : 0);
    if (outcome) {
        if (blockIdx.x == 0 && tid == 0) st->ended = outcome;
        return;
    }
    // first rank of every 256 vertices
    int reps;
    {
        int x[kPer], s = 0;
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            x[k] = rc[0][k];
#pragma unroll
            for (int t = 1; t < kMidPicks; ++t) x[k] = tr == t ? rc[t][k] : x[k];
            s += x[k];
        }
        int run = mid_block_scan(s, ws, &reps);
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            pre[tid * kPer + k] = run;
            run += x[k];
        }
    }
    __syncthreads();
    const u64* bits = a.rbits[tr];
    const int* best = a.best[tr];
    auto below = [&](int r) {  // representatives below r
        const int q0 = (r >> 8) << 2, q1 = r >> 6;
        int k = pre[r >> 8];
        u64 x[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) x[q] = q0 + q <= q1 ? bits[q0 + q] : 0ull;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            k += __popcll(q0 + q < q1 ? x[q] : (q0 + q == q1 ? x[q] & ((1ull << (r & 63)) - 1ull) : 0ull));
        return k;
    };
    const int* off = a.g.off;
    const float scale = 256.0f / (float)(2 * nf);
    // the tile's edges
    if (e0 < nf) {
        int br[kMidEdgeItems], bc[kMidEdgeItems];
#pragma unroll
        for (int k = 0; k < kMidEdgeItems; ++k) {
            br[k] = best[er[k]];
            bc[k] = best[ec[k]];
        }
        // the representative: the pair's smaller end
#pragma unroll
        for (int k = 0; k < kMidEdgeItems; ++k) {
            const int xr = br[k] >= 0 ? best[br[k]] : -1, xc = bc[k] >= 0 ? best[bc[k]] : -1;
            if (br[k] >= 0 && br[k] < er[k] && xr == er[k]) er[k] = br[k];
            if (bc[k] >= 0 && bc[k] < ec[k] && xc == ec[k]) ec[k] = bc[k];
        }
#pragma unroll
        for (int k = 0; k < kMidEdgeItems; ++k) {
            const int e = e0 + k * kMidThreads + tid;
            const int rl = min(er[k], ec[k]), rh = max(er[k], ec[k]);
            const int bl = mid_bucket_of(off[rl], scale), bh = mid_bucket_of(off[rh], scale);
            const u64 x = mid_pack((u32)below(rl), (u32)below(rh), (u32)bl, (u32)bh);
            if (e < nf) {
                a.ekey[e] = x;
                atomicAdd(&hist[bl], 1);
                if (rl != rh) atomicAdd(&hist[bh], 1);
            }
        }
    }
    // the vertices' labels and each bucket's first label
    for (int v = blockIdx.x * kMidThreads + tid; v < n; v += gridDim.x * kMidThreads) {
        const int b = best[v];
        const int o1 = off[v], o0 = v > 0 ? off[v - 1] : 0;
        const int self = below(v);
        int l = self;
        if (b >= 0 && b < v && best[b] == v) l = below(b);
        a.cur[v] = l;
        const int b1 = mid_bucket_of(o1, scale), b0 = v > 0 ? mid_bucket_of(o0, scale) : -1;
        for (int q = b0 + 1; q <= b1; ++q) a.rb[q] = self;
        if (v == n - 1)
            for (int q = b1 + 1; q <= 256; ++q) a.rb[q] = reps;
    }
    if (blockIdx.x == 0 && tid == 0) {
        st->matched = matched;
        st->kb = mid_bits(n - 1 - matched / 2);
    }
    __syncthreads();
    if (e0 < nf && tid < 256) a.table[blockIdx.x * 256 + tid] = hist[tid];
}

// One tile of edges, each as (lo, hi) and mirrored (a self-loop once), to
// its row bucket, stably: every block adds up the tiles' counts itself.
__global__ __launch_bounds__(kMidThreads) void k_mid_scatter(MidArgs a) {
    __shared__ int wcnt[kMidWaves][256];
    __shared__ int start[256];
    __shared__ int rb[256];
    __shared__ int half[2][256];
    __shared__ int ws[kMidWaves];
    __shared__ int over;
    MidState* st = a.st;
    if (st->stop | st->ended) return;
    const int tid = threadIdx.x, lane = lane_id(), w = tid >> 6;
    const int nf = st->nf, kb = st->kb;
    const int ntiles = (nf + kMidTileEdges - 1) / kMidTileEdges;
    if ((int)blockIdx.x >= ntiles) return;
    if (tid == 0) over = 0;
    for (int k = tid; k < kMidWaves * 256; k += kMidThreads) (&wcnt[0][0])[k] = 0;
    // two threads per digit, each over every other 16 tiles
    int mine = 0, all = 0;
    const int dg = tid & 255;
    for (int t = (tid >> 8) * 16; t < ntiles; t += 32) {
        int x[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) x[u] = t + u < ntiles ? a.table[(t + u) * 256 + dg] : 0;
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            mine += t + u < (int)blockIdx.x ? x[u] : 0;
            all += x[u];
        }
    }
    if (tid >= 256) {
        half[0][dg] = mine;
        half[1][dg] = all;
    }
    __syncthreads();
    if (tid < 256) {
        mine += half[0][dg];
        all += half[1][dg];
    } else {
        mine = all = 0;
    }
    int tot;
    const int beg = mid_block_scan(all, ws, &tot);
    if (tid < 256) {
        start[tid] = beg + mine;
        const int r0 = a.rb[tid], r1 = a.rb[tid + 1];
        rb[tid] = r0;
        if (all > kMidBucketMax || mid_bits(r1 - r0 - 1) + kb > 32) over = 1;
    }
    if (blockIdx.x == 0) {
        if (tid < 256) a.bstart[tid] = beg;
        if (tid == 0) a.bstart[256] = tot;
    }
    __syncthreads();
    if (over) {
        if (blockIdx.x == 0 && tid == 0) st->skewed = kMidSkew;
        return;
    }
    const int e0 = blockIdx.x * kMidTileEdges + w * 64 * kMidEdgeItems;
    const unsigned long long lt = (1ull << lane) - 1ull;
    u32 lo[kMidEdgeItems], hi[kMidEdgeItems];
    u32 dig[kMidEdgeItems];  // buckets of lo (high byte) and hi
    u32 cost[kMidEdgeItems];
    int rnk[2][kMidEdgeItems];
#pragma unroll
    for (int k = 0; k < kMidEdgeItems; ++k) {
        const int e = e0 + k * 64 + lane;
        lo[k] = hi[k] = 0xffffffffu;
        dig[k] = cost[k] = 0u;
        if (e < nf) {
            const u64 x = a.ekey[e];
            lo[k] = (u32)(x >> 34);
            hi[k] = (u32)(x >> 16) & 0x3ffffu;
            dig[k] = (u32)x & 0xffffu;
            cost[k] = __float_as_uint(a.g.val[e]);
        }
    }
    // ranks within the wave, per direction in edge order (the two directions
    // never share a key, a self-loop counts once)
#pragma unroll
    for (int dir = 0; dir < 2; ++dir) {
#pragma unroll
        for (int k = 0; k < kMidEdgeItems; ++k) {
            const bool ok = dir == 0 ? lo[k] != 0xffffffffu : lo[k] != hi[k];
            const u32 d = dir == 0 ? dig[k] >> 8 : dig[k] & 255u;
            unsigned long long peers = __ballot(ok);
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                const unsigned long long m = __ballot((d >> b) & 1u);
                peers &= ((d >> b) & 1u) ? m : ~m;
            }
            const int before = wcnt[w][d];
            __builtin_amdgcn_wave_barrier();
            if (ok && (peers & lt) == 0ull) wcnt[w][d] = before + __popcll(peers);
            __builtin_amdgcn_wave_barrier();
            rnk[dir][k] = before + __popcll(peers & lt);
        }
    }
    __syncthreads();
    if (tid < 256) {
        int run = start[tid];
#pragma unroll
        for (int q = 0; q < kMidWaves; ++q) {
            const int c = wcnt[q][tid];
            wcnt[q][tid] = run;
            run += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kMidEdgeItems; ++k) {
        if (lo[k] == 0xffffffffu) continue;
        const u32 bl = dig[k] >> 8, bh = dig[k] & 255u;
        const int p = wcnt[w][bl] + rnk[0][k];
        a.key[p] = ((lo[k] - rb[bl]) << kb) | hi[k];
        a.val[p] = cost[k];
        if (lo[k] != hi[k]) {
            const int q = wcnt[w][bh] + rnk[1][k];
            a.key[q] = ((hi[k] - rb[bh]) << kb) | lo[k];
            a.val[q] = cost[k];
        }
    }
}

// One row bucket: stable LDS sort by the low key bits, then the head of each
// run of equal keys sums the run in order (double, rounded once) and the
// off-diagonal ones are stored in order from the bucket's start.
__global__ __launch_bounds__(kMidThreads) void k_mid_bucket(MidArgs a) {
    __shared__ u32 sk[kMidBucketMax];
    __shared__ u32 sv[kMidBucketMax];
    __shared__ int wcnt[kMidWaves][256];
    __shared__ int dstart[256];
    __shared__ int ws[kMidWaves];
    __shared__ int agg[8];
    const MidState* st = a.st;
    if (st->stop | st->ended | st->skewed) return;
    const int tid = threadIdx.x, lane = lane_id(), w = tid >> 6, b = blockIdx.x;
    const int n = st->n, kb = st->kb;
    // labels of the nodes at entry, composed with this contraction
    for (int v = b * kMidThreads + tid; v < a.n0; v += gridDim.x * kMidThreads) {
        const int l = a.label[v];
        if (l < n) a.label[v] = a.cur[l];
    }
    const int beg = a.bstart[b], m = a.bstart[b + 1] - beg;
    if (m == 0) {
        if (tid < 8) a.bstat[b * 8 + tid] = tid < 2 ? 0 : (tid < 5 ? -1 : (tid == 5 ? 0 : 0x7f7fffff));
        return;
    }
    const int items = (m + kMidThreads - 1) / kMidThreads;
    const int wbase = w * 64 * items;
    u32 key[kMidItems], val[kMidItems];
#pragma unroll
    for (int k = 0; k < kMidItems; ++k) {
        if (k >= items) break;
        const int i = wbase + k * 64 + lane;
        key[k] = i < m ? a.key[beg + i] : ~0u;
        val[k] = i < m ? a.val[beg + i] : 0u;
    }
    if (tid < 8) agg[tid] = tid >= 2 && tid < 5 ? -1 : (tid == 6 ? 0x7f7fffff : 0);
    const int r0 = a.rb[b];
    const int bits = mid_bits(a.rb[b + 1] - r0 - 1) + kb, passes = (bits + 7) / 8, bw = bits / passes, extra = bits % passes;
    const unsigned long long lt = (1ull << lane) - 1ull;
    int shift = 0;
    for (int p = 0; p < passes; ++p) {
        const int width = bw + (p < extra ? 1 : 0);
        const u32 mask = (1u << width) - 1u;
        for (int k = tid; k < kMidWaves * 256; k += kMidThreads) (&wcnt[0][0])[k] = 0;
        __syncthreads();
        int rnk[kMidItems];
#pragma unroll
        for (int k = 0; k < kMidItems; ++k) {
            if (k >= items) break;
            const u32 d = (key[k] >> shift) & mask;
            unsigned long long peers = ~0ull;
            for (int q = 0; q < width; ++q) {
                const unsigned long long mm = __ballot((d >> q) & 1u);
                peers &= ((d >> q) & 1u) ? mm : ~mm;
            }
            const int r = __popcll(peers & lt);
            const int before = wcnt[w][d];
            __builtin_amdgcn_wave_barrier();
            if (r == 0) wcnt[w][d] = before + __popcll(peers);
            __builtin_amdgcn_wave_barrier();
            rnk[k] = before + r;
        }
        __syncthreads();
        if (tid < 256) {
            int tot = 0;
#pragma unroll
            for (int q = 0; q < kMidWaves; ++q) {
                const int c = wcnt[q][tid];
                wcnt[q][tid] = tot;
                tot += c;
            }
            dstart[tid] = tot;
        }
        __syncthreads();
        if (w == 0) {
            int v[4], s = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                v[q] = dstart[lane * 4 + q];
                s += v[q];
            }
            int run = wave_incl_scan(s) - s;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                dstart[lane * 4 + q] = run;
                run += v[q];
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kMidItems; ++k) {
            if (k >= items) break;
            const u32 d = (key[k] >> shift) & mask;
            const int pos = dstart[d] + wcnt[w][d] + rnk[k];
            sk[pos] = key[k];
            sv[pos] = val[k];
        }
        __syncthreads();
        shift += width;
        if (p + 1 < passes) {
#pragma unroll
            for (int k = 0; k < kMidItems; ++k) {
                if (k >= items) break;
                key[k] = sk[wbase + k * 64 + lane];
                val[k] = sv[wbase + k * 64 + lane];
            }
        }
    }
    const u32 cmask = (1u << kb) - 1u;
    int mrow = -1, mcol = -1, mkept = -1, bad = 0, nfwd = 0, total = 0;
    float mn = 3.402823466e38f;
    for (int k = 0; k < items; ++k) {  // uniform
        const int e = k * kMidThreads + tid;
        bool head = false;
        float f = 0.0f;
        u32 x = 0u;
        if (e < m) {
            x = sk[e];
            head = e == 0 || sk[e - 1] != x;
            if (head) {
                double acc = 0.0;
                for (int y = e; y < m && sk[y] == x; ++y) acc += (double)__uint_as_float(sv[y]);
                f = (float)acc;
                const int r = r0 + (int)(x >> kb), c = (int)(x & cmask);
                if (r <= c) {
                    mrow = r > mrow ? r : mrow;
                    mcol = c > mcol ? c : mcol;
                }
                if (r == c) {
                    bad |= f < 0.0f ? 1 : 0;
                    head = false;
                } else if (r < c) {
                    mkept = c > mkept ? c : mkept;
                    mn = f < mn ? f : mn;
                    ++nfwd;
                }
            }
        }
        int cnt;
        const int pos = mid_block_scan(head ? 1 : 0, ws, &cnt);
        if (head) {
            a.hkey[beg + total + pos] = x;
            a.hval[beg + total + pos] = f;
        }
        total += cnt;
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        mrow = max(mrow, __shfl_xor(mrow, d, 64));
        mcol = max(mcol, __shfl_xor(mcol, d, 64));
        mkept = max(mkept, __shfl_xor(mkept, d, 64));
        bad |= __shfl_xor(bad, d, 64);
        nfwd += __shfl_xor(nfwd, d, 64);
        const float o = __shfl_xor(mn, d, 64);
        mn = o < mn ? o : mn;
    }
    // agg was set before the sort's barriers
    if (lane == 0) {
        atomicAdd(&agg[1], nfwd);
        atomicMax(&agg[2], mrow);
        atomicMax(&agg[3], mcol);
        atomicMax(&agg[4], mkept);
        if (bad) agg[5] = 1;
    }
    __syncthreads();  // ws may still be read by the last scan
    if (lane == 0) ws[w] = __float_as_int(mn);
    __syncthreads();
    if (tid == 0) {
        for (int k = 0; k < kMidWaves; ++k) {
            const float o = __int_as_float(ws[k]);
            mn = o < mn ? o : mn;
        }
        agg[0] = total;
        agg[6] = __float_as_int(mn);
        for (int k = 0; k < 8; ++k) a.bstat[b * 8 + k] = agg[k];
    }
}

// The merged entries into place: CSR, forward edges, row offsets of the
// bucket's rows; block 0 leaves the next round's state.
__global__ __launch_bounds__(kBlock) void k_mid_finish(MidArgs a) {
    __shared__ int ws[kWaves];
    __shared__ int base_s[2];
    __shared__ float wf[kWaves];
    const MidState* st = a.st;
    const int tid = threadIdx.x, b = blockIdx.x;
    if (st->stop | st->ended | st->skewed) {
        if (b == 0 && tid == 0) {
            MidState x = *st;
            x.stop = x.stop ? x.stop : (x.ended ? x.ended : x.skewed);
            *a.nx = x;
            if (a.mirror) *a.mirror = x;
        }
        return;
    }
    const int kb = st->kb;
    const int na = a.bstat[tid * 8], nw = a.bstat[tid * 8 + 1];
    int tot, ftot;
    const int ea = block_excl_scan(na, ws, &tot);
    const int ef = block_excl_scan(nw, ws, &ftot);
    if (tid == b) {
        base_s[0] = ea;
        base_s[1] = ef;
    }
    const int mrow = block_reduce(a.bstat[tid * 8 + 2], OpMax(), ws);
    const int mcol = block_reduce(a.bstat[tid * 8 + 3], OpMax(), ws);
    __syncthreads();
    const int base = base_s[0], fbase = base_s[1];
    const int top = max(mrow, mcol) + 1;  // rows of the CSR
    const int beg = a.bstart[b], m = a.bstat[b * 8];
    const u32 cmask = (1u << kb) - 1u;
    const int r0 = a.rb[b], r1 = a.rb[b + 1];  // the bucket's rows
    int fdone = 0;
    for (int k0 = 0; k0 < m; k0 += kBlock) {  // uniform
        const int k = k0 + tid;
        int r = 0, c = 0, pr = r0 - 1;
        float f = 0.0f;
        if (k < m) {
            const u32 x = a.hkey[beg + k];
            f = a.hval[beg + k];
            r = r0 + (int)(x >> kb);
            c = (int)(x & cmask);
            if (k > 0) pr = r0 + (int)(a.hkey[beg + k - 1] >> kb);
            a.to.adj[base + k] = c;
            a.to.w[base + k] = f;
            for (int q = pr + 1; q <= r; ++q) a.to.off[q] = base + k;
            if (k == m - 1)
                for (int q = r + 1; q < r1 && q <= top; ++q) a.to.off[q] = base + m;
        }
        const int fwd = k < m && r < c ? 1 : 0;
        int cnt;
        const int pos = block_excl_scan(fwd, ws, &cnt);
        if (fwd) {
            const int q = fbase + fdone + pos;
            a.to.row[q] = r;
            a.to.col[q] = c;
            a.to.val[q] = f;
        }
        fdone += cnt;
    }
    if (m == 0)
        for (int q = r0 + tid; q < r1 && q <= top; q += kBlock) a.to.off[q] = base;
    if (b != 0) return;
    // the offset after the last row where the buckets' rows end there
    if (tid == 0 && top >= a.rb[256]) a.to.off[top] = tot;
    const int mkept = block_reduce(a.bstat[tid * 8 + 4], OpMax(), ws);
    const int bad = block_reduce(a.bstat[tid * 8 + 5], OpMax(), ws);
    const float mn = block_reduce(__int_as_float(a.bstat[tid * 8 + 6]), OpMin(), wf);
    if (tid == 0) {
        MidState x{};
        x.iter = st->iter + 1;
        x.nf = ftot;
        x.rows = mrow + 1;
        x.cols = mcol + 1;
        x.max_node = mkept;
        x.n = mkept + 1;
        x.minw = mn;
        x.rounds = st->rounds + 1;
        const bool cross = (float)st->matched < (float)st->rows * a.ratio;
        x.stop = bad ? kSmallBad
                     : (ftot == 0 ? kSmallDone
                                  : (cross ? kSmallForest
                                           : (ftot <= a.small_edges && top <= kSmallMaxNodes && x.n * ((x.n + 31) / 32) <= a.small_words
                                                  ? kMidSmall
                                                  : 0)));
        *a.nx = x;
        if (a.mirror) *a.mirror = x;
    }
}

bool mid_rounds_fit(const DCoo& A, const Options& o) {
    const int n = A.max_node + 1;
    const int len = o.num_dual_itr_primal == 0 ? 0 : o.max_cycle_length_primal;
    return n >= 2 && A.max_dim() <= kMidMaxNodes && A.nnz <= kMidMaxEdges && len <= 5 && A.sym &&
           A.sym->n >= n && tune::get(tune::MidRounds, A.nnz) != 0;
}

MidState mid_rounds(Ctx& ctx, DCoo& A, const Options& o, int iter, int first, int* labels, i64 num_labels) {
    const int n0 = A.max_node + 1, cap_n = A.max_dim();
    const i64 nf0 = A.nnz;
    const int nblk = (n0 + kBlock - 1) / kBlock;
    // the two graphs that rounds alternate between: A's own arrays and these
    DCoo B;
    B.row = ctx.buf<int>(nf0);
    B.col = ctx.buf<int>(nf0);
    B.val = ctx.buf<float>(nf0);
    auto S = std::make_shared<Csr>();
    S->off = ctx.buf<int>((i64)cap_n + 2);
    S->adj = ctx.buf<int>(2 * nf0);
    S->w = ctx.buf<float>(2 * nf0);
    // A's offsets too may receive a round's max_dim() + 1 of them
    auto graph = [](DCoo& G, Csr& C) {
        return MidGraph{G.row.get(), G.col.get(), G.val.get(), C.off.get(), C.adj.get(), C.w.get()};
    };
    const MidGraph gs[2] = {graph(A, *A.sym), graph(B, *S)};
    DBuf<MidState> states = ctx.buf<MidState>(2);
    DBuf<double> psum = ctx.buf<double>(kReduceMaxBlocks);
    DBuf<int> pcnt = ctx.buf<int>(kReduceMaxBlocks);
    DBuf<int> best = ctx.buf<int>((i64)kMidPicks * n0);
    DBuf<u64> rbits = ctx.buf<u64>((i64)kMidPicks * nblk * (kBlock / 64));
    DBuf<int> cnts = ctx.buf<int>((i64)2 * kMidPicks * nblk);
    DBuf<int> cur = ctx.buf<int>(n0), lab = ctx.buf<int>(n0);
    DBuf<u64> ekey = ctx.buf<u64>(nf0);
    const i64 tiles0 = (nf0 + kMidTileEdges - 1) / kMidTileEdges;
    DBuf<int> table = ctx.buf<int>(tiles0 * 256);
    DBuf<u32> key = ctx.buf<u32>(2 * nf0), val = ctx.buf<u32>(2 * nf0);
    DBuf<u32> hkey = ctx.buf<u32>(2 * nf0);
    DBuf<float> hval = ctx.buf<float>(2 * nf0);
    DBuf<int> bstart = ctx.buf<int>(257), rb = ctx.buf<int>(257), bstat = ctx.buf<int>(256 * 8);
    MidArgs a{};
    a.psum = psum.get();
    a.pcnt = pcnt.get();
    for (int t = 0; t < kMidPicks; ++t) {
        a.best[t] = best.get() + (i64)t * n0;
        a.rbits[t] = rbits.get() + (i64)t * nblk * (kBlock / 64);
        a.rcnt[t] = cnts.get() + (i64)t * nblk;
        a.mcnt[t] = cnts.get() + (i64)(kMidPicks + t) * nblk;
    }
    a.cur = cur.get();
    a.ekey = ekey.get();
    a.table = table.get();
    a.key = key.get();
    a.val = val.get();
    a.bstart = bstart.get();
    a.rb = rb.get();
    a.hkey = hkey.get();
    a.hval = hval.get();
    a.bstat = bstat.get();
    a.label = lab.get();
    a.n0 = n0;
    a.picks = kMidFewPicks;
    a.len = o.num_dual_itr_primal != 0 && o.max_cycle_length_primal >= 3 ? o.max_cycle_length_primal : 0;
    DBuf<int> pos, npos;
    if (a.len) {
        pos = ctx.buf<int>(2 * nf0);
        npos = ctx.buf<int>(2 * (i64)n0);
        a.pos = pos.get();
        a.npos = npos.get();
        a.npath = a.npos + n0;
    }
    a.small_words = a.len > 3 ? kSmallBitWords : 0x7fffffff;  // small_rounds_fit's limit
    a.small_edges = tune::get(tune::SmallRounds, kSmallMaxEdges) ? kSmallMaxEdges : 0;
    a.mult = o.mean_multiplier_mm;
    a.ratio = o.matching_thresh_crossover_ratio;
    a.tol = 1e-4f;
    // state at entry; the smallest cost is only needed for the cycle test
    {
        MidState* s0 = states.get();
        const float* W = A.val.get();
        MidState init{};
        init.iter = iter;
        init.nf = (int)nf0;
        init.n = n0;
        init.rows = A.rows;
        init.cols = A.cols;
        init.max_node = A.max_node;
        int* L = lab.get();
        for_each(ctx, n0, [=] __device__(i64 v) {
            L[v] = (int)v;
            if (v == 0) *s0 = init;
        });
        if (a.len)
            reduce_to<float>(ctx, [=] __device__(i64 e) { return W[e]; }, nf0, 3.402823466e38f, OpMin(), &s0->minw);
    }
    MidState h{};
    h.nf = (int)nf0;
    h.n = n0;
    int queued = 0;
    // a few rounds per host wait, more as they keep going
    for (int batch = first;; batch = std::min(2 * batch, 16)) {
        const unsigned ntiles = (unsigned)((h.nf + kMidTileEdges - 1) / kMidTileEdges);
        const unsigned gb = (unsigned)std::min<i64>(
            std::max<i64>((2 * (i64)h.nf + kBlock - 1) / kBlock, ((i64)h.n * kMidGroup + kBlock - 1) / kBlock), kMidGrid);
        const unsigned gc = (unsigned)std::min<i64>(((i64)h.nf * kMidGroup + kBlock - 1) / kBlock, 2 * kMidGrid);
        const unsigned gp = (unsigned)std::min<i64>(((i64)h.n * kMidGroup + kBlock - 1) / kBlock, kMidGrid);
        const unsigned gr = (unsigned)((h.n + kBlock - 1) / kBlock);
        const unsigned gk = std::max(ntiles, 1u);
        for (int r = 0; r < batch; ++r, ++queued) {
            a.g = gs[queued & 1];
            a.to = gs[(queued + 1) & 1];
            a.st = states.get() + (queued & 1);
            a.nx = states.get() + ((queued + 1) & 1);
            a.mirror = r + 1 == batch ? ctx.mirror<MidState>() : nullptr;
            prof::Scope ps(ctx, "mid_round", 0.0);
            k_mid_begin<<<gb, kBlock, 0, ctx.stream>>>(a);
            RAMA_LAUNCHED();
            if (a.len > 3) {
                k_mid_prune<<<gp, kBlock, 0, ctx.stream>>>(a);
                RAMA_LAUNCHED();
            }
            if (a.len) {
                k_mid_cycles<<<gc, kBlock, 0, ctx.stream>>>(a);
                RAMA_LAUNCHED();
            }
            k_mid_pick<true><<<gp, kBlock, 0, ctx.stream>>>(a, 0);
            RAMA_LAUNCHED();
            for (int t = 1; t < a.picks; ++t) {
                k_mid_pick<false><<<gp, kBlock, 0, ctx.stream>>>(a, t);
                RAMA_LAUNCHED();
            }
            k_mid_resolve<<<gr, kBlock, 0, ctx.stream>>>(a);
            RAMA_LAUNCHED();
            k_mid_keys<<<gk, kMidThreads, 0, ctx.stream>>>(a);
            RAMA_LAUNCHED();
            k_mid_scatter<<<gk, kMidThreads, 0, ctx.stream>>>(a);
            RAMA_LAUNCHED();
            k_mid_bucket<<<256, kMidThreads, 0, ctx.stream>>>(a);
            RAMA_LAUNCHED();
            k_mid_finish<<<256, kBlock, 0, ctx.stream>>>(a);
            RAMA_LAUNCHED();
        }
        ctx.read_mirror(states.get() + (queued & 1), ctx.mirror<MidState>(), &h);
        if (h.stop == kMidMatching && a.picks < kMidPicks) {
            // queue this round again with more matching rounds, and the ones after it
            a.picks = kMidPicks;
            const MidState* from = states.get() + (queued & 1);
            queued = h.rounds;  // parity of the set that holds the graph
            MidState* s = states.get() + (queued & 1);
            for_each(ctx, 1, [=] __device__(i64) {
                MidState x = *from;
                x.stop = x.ended = 0;
                *s = x;
            });
            continue;
        }
        if (h.stop) break;
    }
    h.picks = a.picks;
    map_node_labels(ctx, lab.get(), n0, labels, num_labels);
    if (h.rounds & 1) {  // the graph ended up in the second set
        A.row = std::move(B.row);
        A.col = std::move(B.col);
        A.val = std::move(B.val);
        A.sym = S;
    }
    A.nnz = h.nf;
    A.rows = h.rows;
    A.cols = h.cols;
    A.max_node = h.max_node;
    A.sym->n = A.max_dim();
    A.sym->nnz = 2 * A.nnz;
    return h;
}

}  // namespace rama
