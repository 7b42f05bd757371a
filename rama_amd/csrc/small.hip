// small.hip — matching-contraction rounds of a small graph in one launch.
//
// A round of the primal-dual driver (src/rama_cuda.cu:88-158) on a graph of
// a few thousand edges is some 25 to 60 launches of 2 to 20 us each whatever
// the graph's size: a solve spends most of its rounds there, since the last
// 20 to 50 contractions each shrink the graph by a few percent.  Here one
// workgroup holds the whole graph in LDS and runs round after round — the
// conflicted-cycle test, the matching, the label compression, the
// contraction's stable sort and merge — with barriers instead of launches.
// It stops where the driver has something else to do (a conflicted cycle,
// the switch to the spanning forest, nothing left) and hands the graph back.
//
// Bound by LDS latency and barriers: about 60 barriers and 3 or 4 radix
// passes over at most 8192 entries a round.  Measured per round: 16 us
// against 170 stage by stage on 404 edges and fewer, 28 against 160 on 3200
// falling to 400 (primal), 56 against 270 on 4000 (3-cycle test), 50 against
// 500 on 1500 (5-cycle test).  Solves: 64x64 grid PD 8.0 -> 5.2 ms, 187x211
// grid PD+ 26.5 -> 14.3, random graph of 20012 edges P 6.1 -> 3.0, 257x509
// grid with long-range edges PD 22.4 -> 18.7.  The size limit is the LDS: the
// graph takes 72 KB and the sort 81 of the workgroup's 160.
//
// Every decision follows the general path's arithmetic: the same thresholds
// (matching.hip's sums in reduce_pair_to's order), the same stop rule, runs of
// equal keys summed in double in input order.  So the rounds give the same
// labels and costs, bit for bit, as the launches they replace.  A round with a
// cost that is not a number is left to the driver: what its launches pick from
// such comparisons hangs on their shape.
#include "rama_internal.hpp"
#include "tuning.hpp"

namespace rama {

constexpr int kSmThreads = 1024;
constexpr int kSmWaves = kSmThreads / 64;
constexpr int kSmEntries = 2 * kSmallMaxEdges;      // symmetric entries
constexpr int kSmItems = kSmEntries / kSmThreads;   // sorted items per thread at most
constexpr int kSmNodeItems = kSmallMaxNodes / kSmThreads;
constexpr int kSmGroup = 8;                         // lanes per vertex or edge in the list walks
constexpr int kSmRounds = 64;                       // rounds per launch (the host queues another)
constexpr int kSmMatchRounds = 10;

// The graph: symmetric CSR (rows ascending by neighbour) and, per forward
// edge (row < col, in (row, col) order), its row and its place in the CSR.
struct SmGraph {
    float w[kSmEntries];
    unsigned short adj[kSmEntries];
    unsigned short fpos[kSmallMaxEdges];
    unsigned short frow[kSmallMaxEdges];
    unsigned short off[kSmallMaxNodes + 2];
};
struct SmSort {
    u32 key[kSmEntries];
    u32 val[kSmEntries];
    int wcnt[kSmWaves][256];
    int dstart[256];
};
struct SmMatch {
    unsigned short best[kSmallMaxNodes];
    unsigned short map[kSmallMaxNodes];
    unsigned short rank[kSmallMaxNodes];
    unsigned char matched[kSmallMaxNodes];
};
constexpr unsigned short kSmNone = 0xffff;
// One round's scratch: the attractive adjacency as a bit matrix (cycle
// test), then the matching's arrays, then the sort's.
union SmScratch {
    SmSort sort;
    SmMatch match;
    u32 bits[kSmallBitWords];
    double vws[kSmEntries / 64];  // per-wave partial sums of the threshold
};
static_assert(sizeof(SmSort) >= sizeof(u32) * kSmallBitWords, "bit matrix within the sort's scratch");

struct SmShared {
    SmGraph g;
    SmScratch s;
    u32 wsum[kSmWaves];
    float wmin[kSmWaves];
    int newly[kSmMatchRounds];
    int found;     // conflicted cycle
    int st[4];     // contraction: largest row, col, kept col; negative self-loop
    int total;
    int nan;
    int lastrow;
    float pos_sum, pos_cnt;
};
static_assert(sizeof(SmShared) <= 160 * 1024, "LDS of a gfx950 workgroup");

struct SmArgs {
    int* row;     // forward edges in and out
    int* col;
    float* val;
    int* off;     // symmetric CSR in and out
    int* adj;
    float* w;
    int* label;   // out: label of each of the n0 nodes at entry
    int nf, n0, rows, cols;
    int iter;     // round number of the driver
    int max_len;  // primal cycle length (0: no dual pass)
    float mult, ratio, tol;
    SmallState* out;
    SmallState* mirror;
};

// Exclusive scan over the block of one value per thread; *total the sum.
__device__ __forceinline__ u32 sm_scan(u32 x, u32* ws, u32* total) {
    const int lane = lane_id(), w = threadIdx.x >> 6;
    const u32 inc = wave_incl_scan(x);
    __syncthreads();  // ws may still be read by the scan before
    if (lane == 63) ws[w] = inc;
    __syncthreads();
    u32 before = 0, tot = 0;
#pragma unroll
    for (int k = 0; k < kSmWaves; ++k) {
        const u32 t = ws[k];
        before += k < w ? t : 0u;
        tot += t;
    }
    *total = tot;
    return before + inc - x;
}

__device__ __forceinline__ int sm_lower(const unsigned short* a, int lo, int hi, int x) {
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if ((int)a[mid] < x) lo = mid + 1; else hi = mid;
    }
    return lo;
}

// Whether some repulsive edge (cost < t) closes a path of 2 .. max_len - 1
// attractive edges (cost > -t): whether the search of
// conflicted_cycles (src/conflicted_cycles_cuda.cu:222-343) would fill any
// triangle slot.  A 3-cycle is a common neighbour of the two ends, a 4-cycle
// one of N(N(v1)) and N(v2), a 5-cycle one of N(N(v1)) and N(N(v2)); walks
// that step back give such a common element only where a shorter cycle exists.
//
// 3-cycles alone: lanes take the shorter list's entries and search the
// longer one.  Longer ones: rows of the attractive adjacency as bit sets,
// OR-ed over a vertex's neighbours.
__device__ __forceinline__ void sm_find_cycles(SmShared& s, int nf, int n, float t, int max_len) {
    const SmGraph& g = s.g;
    const int sub = threadIdx.x % kSmGroup;
    const float at = -1.0f * t;
    if (max_len == 3) {
        for (int x = threadIdx.x / kSmGroup; x < nf; x += kSmThreads / kSmGroup) {
            const int p = g.fpos[x];
            if (!(g.w[p] < t)) continue;
            int a = g.frow[x], b = g.adj[p];
            if (g.off[a + 1] - g.off[a] > g.off[b + 1] - g.off[b]) {
                const int c = a;
                a = b;
                b = c;
            }
            const int b0 = g.off[b], b1 = g.off[b + 1];
            for (int i = g.off[a] + sub; i < g.off[a + 1]; i += kSmGroup) {
                if (!(g.w[i] > at)) continue;
                const int m = g.adj[i];
                const int q = sm_lower(g.adj, b0, b1, m);
                if (q < b1 && g.adj[q] == m && g.w[q] > at) s.found = 1;
            }
        }
        return;
    }
    const int nw = (n + 31) / 32;
    u32* bits = s.s.bits;
    for (int k = threadIdx.x; k < n * nw; k += kSmThreads) bits[k] = 0u;
    __syncthreads();
    for (int x = threadIdx.x; x < nf; x += kSmThreads) {
        const int p = g.fpos[x], a = g.frow[x], b = g.adj[p];
        if (g.w[p] > at) {
            atomicOr(&bits[a * nw + (b >> 5)], 1u << (b & 31));
            atomicOr(&bits[b * nw + (a >> 5)], 1u << (a & 31));
        }
    }
    __syncthreads();
    for (int x = threadIdx.x / kSmGroup; x < nf; x += kSmThreads / kSmGroup) {
        const int p = g.fpos[x];
        if (!(g.w[p] < t)) continue;
        const int a = g.frow[x], b = g.adj[p];
        const int a0 = g.off[a], a1 = g.off[a + 1], b0 = g.off[b], b1 = g.off[b + 1];
        for (int k = sub; k < nw; k += kSmGroup) {
            const u32 na = bits[a * nw + k], nb = bits[b * nw + k];
            u32 hit = na & nb;
            u32 na2 = 0u, nb2 = 0u;
            for (int i = a0; i < a1; ++i) na2 |= g.w[i] > at ? bits[(int)g.adj[i] * nw + k] : 0u;
            hit |= na2 & nb;
            if (max_len >= 5) {
                for (int i = b0; i < b1; ++i) nb2 |= g.w[i] > at ? bits[(int)g.adj[i] * nw + k] : 0u;
                hit |= na2 & nb2;
            }
            if (hit) s.found = 1;
        }
    }
}

// Sum and count of the non-negative costs of the nnz entries, added as
// reduce_pair_to adds them: blocks of 256 consecutive entries, a wave tree,
// the waves in order, then the blocks' partials by one more tree.  s.nan: some
// cost is not a number.
__device__ __forceinline__ void sm_threshold(SmShared& s, int nnz) {
    const int lane = lane_id(), w = threadIdx.x >> 6;
    int cnt = 0;
    bool nan = false;
    for (int vw = w; vw * 64 < nnz; vw += kSmWaves) {
        const int i = vw * 64 + lane;
        const float x = i < nnz ? s.g.w[i] : -1.0f;
        nan |= x != x;
        double a = x >= 0.0f ? (double)x : 0.0;
        cnt += x >= 0.0f ? 1 : 0;
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) a += shfl_down64(a, d);
        if (lane == 0) s.s.vws[vw] = a;
    }
    if (threadIdx.x == 0) s.total = s.nan = 0;
    __syncthreads();
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) cnt += __shfl_xor(cnt, d, 64);
    if (lane == 0) atomicAdd(&s.total, cnt);
    if (nan) s.nan = 1;
    if (w == 0) {
        const int nvw = (nnz + 63) / 64, nb = (nnz + 255) / 256;
        double a = 0.0;
        if (lane < nb) {
            a = s.s.vws[4 * lane];
#pragma unroll
            for (int k = 1; k < 4; ++k) a += 4 * lane + k < nvw ? s.s.vws[4 * lane + k] : 0.0;
        }
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) a += shfl_down64(a, d);
        if (lane == 0) s.pos_sum = (float)a;
    }
    __syncthreads();
    if (threadIdx.x == 0) s.pos_cnt = (float)s.total;
    __syncthreads();
}
static_assert(kSmEntries / 256 <= 64, "one wave holds the blocks' partials");

// The matching rounds (matching.hip: k_pick_best and k_match with their stop
// rule).  Afterwards s.s.match.map is the mapping; returns the matched vertices.
__device__ __forceinline__ int sm_matching(SmShared& s, int n, float mult) {
    const SmGraph& g = s.g;
    SmMatch& m = s.s.match;
    const int tid = threadIdx.x, sub = tid % kSmGroup;
    const float cnt = s.pos_cnt;
    const float thr = mult * s.pos_sum / cnt;
    for (int v = tid; v < n; v += kSmThreads) {
        m.map[v] = (unsigned short)v;
        m.best[v] = kSmNone;
        m.matched[v] = 0;
    }
    if (tid < kSmMatchRounds) s.newly[tid] = 0;
    __syncthreads();
    if (cnt == 0.0f || thr < 0.0f) return 0;  // uniform
    int prev = 0;
    for (int t = 0; t < kSmMatchRounds; ++t) {
        for (int v = tid / kSmGroup; v < n; v += kSmThreads / kSmGroup) {  // uniform within the group
            if (m.matched[v]) continue;
            const int e = g.off[v + 1];
            float bv = thr;
            int bp = 0x7fffffff, bn = kSmNone;
            for (int l = g.off[v] + sub; l < e; l += kSmGroup) {
                const float c = g.w[l];
                const int u = g.adj[l];
                if (c > bv && !m.matched[u] && u != v) {
                    bv = c;
                    bp = l;
                    bn = u;
                }
            }
#pragma unroll
            for (int d = kSmGroup / 2; d >= 1; d >>= 1) {
                const float ov = __shfl_xor(bv, d, kSmGroup);
                const int op = __shfl_xor(bp, d, kSmGroup);
                const int on = __shfl_xor(bn, d, kSmGroup);
                if (ov > bv || (ov == bv && op < bp)) {
                    bv = ov;
                    bp = op;
                    bn = on;
                }
            }
            if (sub == 0) m.best[v] = (unsigned short)bn;
        }
        __syncthreads();
        int add = 0;
        for (int v = tid; v < n; v += kSmThreads) {
            const int vb = m.best[v];
            // a matched vertex keeps its partner in best[], so best[vb] == v
            // with v unmatched means vb is unmatched too
            if (vb != kSmNone && vb > v && !m.matched[v] && m.best[vb] == v) {
                m.map[vb] = (unsigned short)v;
                m.matched[v] = 1;
                m.matched[vb] = 1;
                add += 2;
            }
        }
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) add += __shfl_xor(add, d, 64);
        if (lane_id() == 0 && add) atomicAdd(&s.newly[t], add);
        __syncthreads();
        const int nw = s.newly[t];
        const int cur = prev + nw;
        const float rel = (cur - prev) / (prev + 1.0f);
        prev = cur;
        if (nw == 0 || rel < 0.1f) break;  // uniform
    }
    return prev;
}

// Lanes of the wave whose digit equals this lane's, among the wave's lanes.
__device__ __forceinline__ unsigned long long sm_peers(u32 d, int bits) {
    unsigned long long peers = ~0ull;
    for (int b = 0; b < bits; ++b) {
        const unsigned long long m = __ballot((d >> b) & 1u);
        peers &= ((d >> b) & 1u) ? m : ~m;
    }
    return peers;
}

// Stable sort of the nk items (key, val per thread in (wave, item, lane)
// order, `items` per thread; items past nk hold ~0) by the low `bits` bits;
// the result is left in s.s.sort.key / val.
__device__ __forceinline__ void sm_sort(SmShared& s, u32 (&key)[kSmItems], u32 (&val)[kSmItems], int items, int bits) {
    SmSort& so = s.s.sort;
    const int tid = threadIdx.x, lane = lane_id(), w = tid >> 6;
    const int wbase = w * 64 * items;
    const unsigned long long lt = (1ull << lane) - 1ull;
    const int passes = (bits + 7) / 8, bw = bits / passes, extra = bits % passes;
    int shift = 0;
    for (int p = 0; p < passes; ++p) {
        const int width = bw + (p < extra ? 1 : 0);
        const u32 mask = (1u << width) - 1u;
        for (int k = tid; k < kSmWaves * 256; k += kSmThreads) (&so.wcnt[0][0])[k] = 0;
        __syncthreads();
        int rnk[kSmItems];
#pragma unroll
        for (int k = 0; k < kSmItems; ++k) {
            if (k >= items) break;
            const u32 d = (key[k] >> shift) & mask;
            const unsigned long long peers = sm_peers(d, width);
            const int r = __popcll(peers & lt);
            const int before = so.wcnt[w][d];
            __builtin_amdgcn_wave_barrier();
            if (r == 0) so.wcnt[w][d] = before + __popcll(peers);
            __builtin_amdgcn_wave_barrier();
            rnk[k] = before + r;
        }
        __syncthreads();
        // wave w's items of digit d start after those of the waves before it
        if (tid < 256) {
            int tot = 0;
#pragma unroll
            for (int q = 0; q < kSmWaves; ++q) {
                const int c = so.wcnt[q][tid];
                so.wcnt[q][tid] = tot;
                tot += c;
            }
            so.dstart[tid] = tot;
        }
        __syncthreads();
        if (w == 0) {  // exclusive scan of the 256 digit totals
            int v[4], sum = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                v[q] = so.dstart[lane * 4 + q];
                sum += v[q];
            }
            int run = wave_incl_scan(sum) - sum;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                so.dstart[lane * 4 + q] = run;
                run += v[q];
            }
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kSmItems; ++k) {
            if (k >= items) break;
            const u32 d = (key[k] >> shift) & mask;
            const int pos = so.dstart[d] + so.wcnt[w][d] + rnk[k];
            so.key[pos] = key[k];
            so.val[pos] = val[k];
        }
        __syncthreads();
        shift += width;
        if (p + 1 < passes) {
#pragma unroll
            for (int k = 0; k < kSmItems; ++k) {
                if (k >= items) break;
                key[k] = so.key[wbase + k * 64 + lane];
                val[k] = so.val[wbase + k * 64 + lane];
            }
            // the next pass writes only after three more barriers
        }
    }
}

__global__ __launch_bounds__(kSmThreads) void k_small_rounds(SmArgs a) {
    __shared__ SmShared s;
    SmGraph& g = s.g;
    const int tid = threadIdx.x, lane = lane_id(), w = tid >> 6;
    int nf = a.nf, n = a.n0, rows = a.rows, cols = a.cols;
    // load: CSR, forward edges and their places (the forward edges of a row
    // are the last entries of its CSR row)
    for (int v = tid; v <= n; v += kSmThreads) g.off[v] = (unsigned short)a.off[v];
    for (int e = tid; e < 2 * nf; e += kSmThreads) {
        g.adj[e] = (unsigned short)a.adj[e];
        g.w[e] = a.w[e];
    }
    for (int e = tid; e < nf; e += kSmThreads) g.frow[e] = (unsigned short)a.row[e];
    __syncthreads();
    for (int e = tid; e < nf; e += kSmThreads) {
        const int r = g.frow[e];
        const int fe = sm_lower(g.frow, e, nf, r + 1);
        g.fpos[e] = (unsigned short)(g.off[r + 1] - (fe - e));
    }
    int lab[kSmNodeItems];
#pragma unroll
    for (int k = 0; k < kSmNodeItems; ++k) lab[k] = tid + k * kSmThreads;
    __syncthreads();

    int iter = a.iter, reason = kSmallMore, done = 0;
    for (int round = 0; round < kSmRounds; ++round) {
        // conflicted cycles: the dual pass is the driver's
        if (a.max_len >= 3 && iter > 0) {
            float mn = 3.402823466e38f;
            for (int x = tid; x < nf; x += kSmThreads) {
                const float c = g.w[g.fpos[x]];
                mn = c < mn ? c : mn;
            }
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) {
                const float o = __shfl_xor(mn, d, 64);
                mn = o < mn ? o : mn;
            }
            if (lane == 0) s.wmin[w] = mn;
            if (tid == 0) s.found = 0;
            __syncthreads();
#pragma unroll
            for (int k = 0; k < kSmWaves; ++k) mn = s.wmin[k] < mn ? s.wmin[k] : mn;
            sm_find_cycles(s, nf, n, mn * a.tol, a.max_len);
            __syncthreads();
            if (s.found) {
                reason = kSmallCycles;
                break;
            }
        }
        sm_threshold(s, 2 * nf);
        if (s.nan) {
            reason = kSmallCycles;
            break;
        }
        const int matched = sm_matching(s, n, a.mult);
        if (matched == 0) {
            reason = kSmallDone;
            break;
        }
        const bool cross = (float)matched < (float)rows * a.ratio;
        // compressed labels: rank of the vertices that keep their id
        SmMatch& m = s.s.match;
        {
            u32 rep[kSmNodeItems], sum = 0;
#pragma unroll
            for (int k = 0; k < kSmNodeItems; ++k) {
                const int v = tid * kSmNodeItems + k;
                rep[k] = v < n && m.map[v] == v ? 1u : 0u;
                sum += rep[k];
            }
            u32 tot;
            u32 run = sm_scan(sum, s.wsum, &tot);
#pragma unroll
            for (int k = 0; k < kSmNodeItems; ++k) {
                const int v = tid * kSmNodeItems + k;
                if (v < n) m.rank[v] = (unsigned short)run;
                run += rep[k];
            }
        }
        if (tid < 4) s.st[tid] = tid < 3 ? -1 : 0;
        if (tid == 4) s.lastrow = -1;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kSmNodeItems; ++k)
            if (lab[k] < n) lab[k] = m.rank[m.map[lab[k]]];
        // contraction keys: every edge as (lo, hi), then every edge mirrored
        const int max_label = n - 1 - matched / 2;
        int kb = 1;
        while ((1 << kb) <= max_label) ++kb;
        const u32 kmask = (1u << kb) - 1u;
        const int nk = 2 * nf;
        const int items = (nk + kSmThreads - 1) / kSmThreads;
        u32 key[kSmItems], val[kSmItems];
#pragma unroll
        for (int k = 0; k < kSmItems; ++k) {
            if (k >= items) break;
            const int i = w * 64 * items + k * 64 + lane;
            key[k] = ~0u;
            val[k] = 0u;
            if (i < nk) {
                const int x = i < nf ? i : i - nf;
                const int p = g.fpos[x];
                const u32 ra = m.rank[m.map[g.frow[x]]], rb = m.rank[m.map[g.adj[p]]];
                const u32 lo = ra < rb ? ra : rb, hi = ra < rb ? rb : ra;
                // a self-loop's mirror sorts after every real key
                key[k] = i < nf ? (lo << kb) | hi : (lo != hi ? (hi << kb) | lo : 1u << (2 * kb));
                val[k] = __float_as_uint(g.w[p]);
            }
        }
        __syncthreads();  // the sort's scratch overlays the matching's arrays
        sm_sort(s, key, val, items, 2 * kb + 1);
        // merge: the head of each run of equal off-diagonal keys sums it in
        // order and becomes an entry of the new CSR; a forward head is a new
        // forward edge too.  Thread t owns positions t * items ..
        const SmSort& so = s.s.sort;
        u32 flag[kSmItems], sum = 0;
#pragma unroll
        for (int k = 0; k < kSmItems; ++k) {
            if (k >= items) break;
            const int e = tid * items + k;
            flag[k] = 0u;
            if (e < nk) {
                const u32 x = so.key[e];
                const u32 r = x >> kb, c = x & kmask;
                const bool head = e == 0 || so.key[e - 1] != x;
                if (head && r <= kmask && r != c) flag[k] = r < c ? 0x10001u : 1u;
            }
            sum += flag[k];
        }
        u32 tot;
        u32 run = sm_scan(sum, s.wsum, &tot);
        int mrow = -1, mcol = -1, mkept = -1, bad = 0, lrow = -1;
#pragma unroll
        for (int k = 0; k < kSmItems; ++k) {
            if (k >= items) break;
            const int e = tid * items + k;
            if (e < nk) {
                const u32 x = so.key[e];
                const int r = (int)(x >> kb), c = (int)(x & kmask);
                const int pr = e > 0 ? (int)(so.key[e - 1] >> kb) : -1;
                const int p = (int)(run & 0xffffu);
                if (r <= (int)kmask) {
                    if (r != pr) {
                        for (int q = pr + 1; q <= r; ++q) g.off[q] = (unsigned short)p;
                        lrow = r;
                    }
                    if (e == 0 || so.key[e - 1] != x) {
                        double acc = 0.0;
                        for (int y = e; y < nk && so.key[y] == x; ++y) acc += (double)__uint_as_float(so.val[y]);
                        const float f = (float)acc;
                        if (r <= c) {
                            mrow = r > mrow ? r : mrow;
                            mcol = c > mcol ? c : mcol;
                            if (r == c) bad |= f < 0.0f ? 1 : 0;
                        }
                        if (r != c) {
                            g.adj[p] = (unsigned short)c;
                            g.w[p] = f;
                            if (r < c) {
                                const int q = (int)(run >> 16);
                                g.fpos[q] = (unsigned short)p;
                                g.frow[q] = (unsigned short)r;
                                mkept = c > mkept ? c : mkept;
                            }
                        }
                    }
                }
            }
            run += flag[k];
        }
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) {
            mrow = max(mrow, __shfl_xor(mrow, d, 64));
            mcol = max(mcol, __shfl_xor(mcol, d, 64));
            mkept = max(mkept, __shfl_xor(mkept, d, 64));
            bad |= __shfl_xor(bad, d, 64);
            lrow = max(lrow, __shfl_xor(lrow, d, 64));
        }
        if (lane == 0) {
            if (mrow >= 0) atomicMax(&s.st[0], mrow);
            if (mcol >= 0) atomicMax(&s.st[1], mcol);
            if (mkept >= 0) atomicMax(&s.st[2], mkept);
            if (bad) s.st[3] = 1;
            if (lrow >= 0) atomicMax(&s.lastrow, lrow);
        }
        __syncthreads();
        rows = s.st[0] + 1;
        cols = s.st[1] + 1;
        const int isbad = s.st[3];
        n = s.st[2] + 1;
        nf = (int)(tot >> 16);
        const int last = s.lastrow, top = max(max(rows, cols), n);
        // rows past the last entry's
        for (int q = last + 1 + tid; q <= top; q += kSmThreads) g.off[q] = (unsigned short)(tot & 0xffffu);
        __syncthreads();
        ++iter;
        ++done;
        if (isbad) {
            reason = kSmallBad;
            break;
        }
        if (nf == 0) {
            reason = kSmallDone;
            break;
        }
        if (cross) {
            reason = kSmallForest;
            break;
        }
    }
    __syncthreads();
    // hand back: graph, CSR (max(rows, cols) rows), labels, state
    if (done) {
        const int top = max(max(rows, cols), n);
        for (int v = tid; v <= top; v += kSmThreads) a.off[v] = g.off[v];
        for (int e = tid; e < 2 * nf; e += kSmThreads) {
            a.adj[e] = g.adj[e];
            a.w[e] = g.w[e];
        }
        for (int e = tid; e < nf; e += kSmThreads) {
            const int p = g.fpos[e];
            a.row[e] = g.frow[e];
            a.col[e] = g.adj[p];
            a.val[e] = g.w[p];
        }
    }
#pragma unroll
    for (int k = 0; k < kSmNodeItems; ++k) {
        const int v = tid + k * kSmThreads;
        if (v < a.n0) a.label[v] = lab[k];
    }
    if (tid == 0) {
        const SmallState st{reason, iter, nf, rows, cols, n - 1};
        *a.out = st;
        if (a.mirror) *a.mirror = st;
    }
}

bool small_rounds_fit(i64 nnz, int max_dim, int max_node, const Options& o) {
    const int n = max_node + 1;
    if (nnz > kSmallMaxEdges || max_dim > kSmallMaxNodes || n < 2) return false;
    if (tune::get(tune::SmallRounds, nnz) == 0) return false;
    const int len = o.num_dual_itr_primal == 0 ? 0 : o.max_cycle_length_primal;
    // cycles of 4 and 5 are looked for in a bit matrix
    if (len > 5 || (len > 3 && n * ((n + 31) / 32) > kSmallBitWords)) return false;
    return true;
}
bool small_rounds_fit(const DCoo& A, const Options& o) { return small_rounds_fit(A.nnz, A.max_dim(), A.max_node, o); }

SmallState small_rounds(Ctx& ctx, DCoo& A, const Options& o, int iter, int* labels, i64 num_labels) {
    const int n0 = A.max_node + 1;
    if (!A.sym)
        A.sym = std::make_shared<Csr>(symmetric_csr(ctx, A.row.get(), A.col.get(), A.val.get(), A.nnz, A.max_dim(),
                                                    false, 0.0f));
    DBuf<int> lab = ctx.buf<int>(n0);
    DBuf<SmallState> out = ctx.buf<SmallState>(1);
    SmArgs a{};
    a.row = A.row.get();
    a.col = A.col.get();
    a.val = A.val.get();
    a.off = A.sym->off.get();
    a.adj = A.sym->adj.get();
    a.w = A.sym->w.get();
    a.label = lab.get();
    a.nf = (int)A.nnz;
    a.n0 = n0;
    a.rows = A.rows;
    a.cols = A.cols;
    a.iter = iter;
    a.max_len = o.num_dual_itr_primal == 0 ? 0 : o.max_cycle_length_primal;
    a.mult = o.mean_multiplier_mm;
    a.ratio = o.matching_thresh_crossover_ratio;
    a.tol = 1e-4f;
    a.out = out.get();
    a.mirror = ctx.mirror<SmallState>();
    {
        prof::Scope ps(ctx, "small_rounds", 0.0);
        k_small_rounds<<<1, kSmThreads, 0, ctx.stream>>>(a);
        RAMA_LAUNCHED();
    }
    map_node_labels(ctx, lab.get(), n0, labels, num_labels);
    SmallState st;
    ctx.read_mirror(out.get(), a.mirror, &st);
    A.nnz = st.nnz;
    A.rows = st.rows;
    A.cols = st.cols;
    A.max_node = st.max_node;
    A.sym->n = A.max_dim();
    A.sym->nnz = 2 * A.nnz;
    return st;
}

}  // namespace rama
