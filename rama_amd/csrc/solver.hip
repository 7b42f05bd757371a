// solver.hip — the primal-dual driver (src/rama_cuda.cu:54-164): initial
// dual pass for the lower bound, then contraction rounds (re-solve a small
// dual, pick contractions by matching or by the conflict-free spanning
// forest, contract, compose labels) until nothing is left to contract.
#include <chrono>
#include <cstdlib>
#include <map>

#include "rama_internal.hpp"

namespace rama {

namespace {
// Wall time per driver stage (stream synchronised at each boundary), printed
// when RAMA_STAGE_TIMES is set.  Diagnostic only.
struct StageTimes {
    bool on = std::getenv("RAMA_STAGE_TIMES") != nullptr;
    std::map<std::string, std::pair<double, int>> acc;
    std::chrono::steady_clock::time_point t0;
    void begin(Ctx& ctx) {
        if (!on) return;
        ctx.sync();
        t0 = std::chrono::steady_clock::now();
    }
    void end(Ctx& ctx, const char* name) {
        if (!on) return;
        ctx.sync();
        auto& a = acc[name];
        a.first += std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
        a.second += 1;
    }
    ~StageTimes() {
        if (!on) return;
        for (auto& kv : acc) std::fprintf(stderr, "stage %-16s %9.3f ms  %d calls\n", kv.first.c_str(), kv.second.first, kv.second.second);
    }
};
}  // namespace

Options to_options(const rama_options_c& c) {
    Options o;
    o.max_cycle_length_lb = c.max_cycle_length_lb;
    o.num_dual_itr_lb = c.num_dual_itr_lb;
    o.max_cycle_length_primal = c.max_cycle_length_primal;
    o.num_dual_itr_primal = c.num_dual_itr_primal;
    o.num_outer_itr_dual = c.num_outer_itr_dual;
    o.mean_multiplier_mm = c.mean_multiplier_mm;
    o.matching_thresh_crossover_ratio = c.matching_thresh_crossover_ratio;
    o.tri_memory_factor = c.tri_memory_factor;
    o.only_compute_lb = c.only_compute_lb != 0;
    o.max_time_sec = c.max_time_sec;
    o.dump_timeline = c.dump_timeline != 0;
    o.verbose = c.verbose != 0;
    o.sanitize_graph = c.sanitize_graph != 0;
    return o;
}

SolveResult solve(Ctx& ctx, DCoo& A, const Options& o) {
    SolveResult out;
    out.t0 = std::chrono::steady_clock::now();
    ctx.last_cycles_empty = false;  // a hint from an earlier solve on this context says nothing here
    scan_reset(ctx);
    StageTimes st;
    st.begin(ctx);
    out.lb = dual_solver(ctx, A, o.max_cycle_length_lb, o.num_dual_itr_lb, o.tri_memory_factor, o.num_outer_itr_dual,
                         1e-4f);
    st.end(ctx, "dual_initial");
    const int N = A.max_dim();
    out.labels = ctx.buf<int>(N);
    iota(ctx, out.labels.get(), N);
    out.num_labels = N;
    if (o.only_compute_lb) {
        out.num_labels = 0;
        scan_check(ctx);
        return out;
    }
    solve_rounds(ctx, A, out, o, 0, !(o.matching_thresh_crossover_ratio > 1.0f));
    return out;
}

// The contraction rounds from round `start_iter` on (src/rama_cuda.cu:88-158):
// out.labels (out.num_labels entries) holds the labels composed so far and
// use_mm whether matching still picks the contractions.
void solve_rounds(Ctx& ctx, DCoo& A, SolveResult& out, const Options& o, int start_iter, bool use_mm, bool quiet) {
    StageTimes st;
    if (start_iter > 0) ctx.last_cycles_empty = quiet;  // resumed on another context
    const auto t0 = out.t0;  // the time budget counts from the start of the solve
    const i64 N = out.num_labels;
    const bool duals = o.max_cycle_length_primal >= 3 && o.num_dual_itr_primal != 0;
    i64 mid_max = kMidMaxEdges;  // largest graph given to mid_rounds
    int mid_first = 2;           // rounds it queues before its first wait
    const bool observed = o.verbose || o.dump_timeline || o.max_time_sec >= 0;
    for (int iter = start_iter; A.nnz > 0; ++iter) {
        const auto r0 = std::chrono::steady_clock::now();
        const int64_t l0 = launch_count(), s0 = ctx.syncs;
        const i64 e0 = A.nnz;
        // A contracted graph of up to a few thousand edges: its rounds run in
        // one launch; of up to 2^18, they are queued without read-backs.
        // Both stop at the next dual pass or the forest.  Not where a round
        // is observed (printing, snapshots, the time budget), nor while the
        // rounds' cycle searches still find something.
        if (use_mm && iter > 0 && (!duals || ctx.last_cycles_empty) && !observed) {
            const bool small = small_rounds_fit(A, o), mid = !small && A.nnz <= mid_max && mid_rounds_fit(A, o);
            int reason = kSmallCycles, next = iter, picks = 0;
            st.begin(ctx);
            if (small) {
                const SmallState ss = small_rounds(ctx, A, o, iter, out.labels.get(), N);
                reason = ss.reason;
                next = ss.iter;
            } else if (mid) {
                const MidState ms = mid_rounds(ctx, A, o, iter, mid_first, out.labels.get(), N);
                reason = ms.stop;
                picks = ms.picks;
                next = ms.iter;
                mid_first = next > iter ? 4 : 1;
                // hubs too large for it: wait until the graph is half as large
                if (reason == kMidSkew) mid_max = ms.nf / 2;
            }
            st.end(ctx, small ? "small_rounds" : "mid_rounds");
            if (st.on && (small || mid))
                std::fprintf(stderr, "rounds %d..%d: %lld edges, %s, reason %d, picks %d, %.3f ms\n", iter, next - 1,
                             (long long)e0, small ? "small" : "mid", reason, picks,
                             std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - r0).count());
            if (reason == kSmallBad) throw Error(RAMA_ERR_BAD_CONTRACTION, "Found bad contractions");
            if (next > iter) out.iterations = next;
            if (reason == kSmallDone) break;
            iter = next;
            if (reason == kSmallForest) use_mm = false;
            if (reason == kSmallMore || reason == kMidSmall) {
                --iter;  // the loop's increment
                continue;
            }
        }
        st.begin(ctx);
        if (iter > 0)
            dual_solver(ctx, A, o.max_cycle_length_primal, o.num_dual_itr_primal, 1.0f, 1, 1e-4f, false);
        st.end(ctx, "dual_primal");
        st.begin(ctx);
        DBuf<int> cur;
        i64 cur_size = 0;
        int n_contract = 0;
        int max_label = 0;
        const bool mm_branch = use_mm;
        if (use_mm) {
            // export_undirected: node count = largest endpoint + 1
            const int Un = A.max_node + 1;
            Csr U;
            if (A.sym && A.sym->n >= Un) {
                // built by this round's cycle search on the same arrays; rows
                // from Un on are empty, so its first Un + 1 offsets are U's
                U = std::move(*A.sym);
                A.sym.reset();
                U.n = Un;
            } else {
                U = symmetric_csr(ctx, A.row.get(), A.col.get(), A.val.get(), A.nnz, Un, false, 0.0f);
            }
            DBuf<int> m;
            n_contract = matching_vertex_based(ctx, U, o.mean_multiplier_mm, m);
            cur = ctx.buf<int>(Un);
            compress_matching(ctx, m.get(), Un, cur.get());
            // largest compressed label (sizes the sort keys): every matched
            // pair shares one label and n_contract counts both its vertices
            max_label = Un - 1 - n_contract / 2;
            cur_size = Un;
            if ((float)n_contract < (float)A.rows * o.matching_thresh_crossover_ratio) {
                if (o.verbose)
                    std::printf("# edges to contract = %d, # vertices = %d\nswitching to MST based contraction edge selection\n",
                                n_contract, A.rows);
                use_mm = false;
            }
        } else {
            n_contract = woc_mapping(ctx, A, cur, cur_size);
            max_label = (int)cur_size - 1;
        }
        st.end(ctx, mm_branch ? "matching" : "mst_mapping");
        st.begin(ctx);
        if (n_contract == 0) {
            if (o.verbose) std::printf("# iterations = %d\n", iter);
            break;
        }
        bool bad = false;
        double diag = 0.0;
        DCoo B = contract(ctx, A, cur.get(), max_label, &bad, o.verbose ? &diag : nullptr);
        if (o.verbose) {
            std::printf("original A size %dx%d\ncontracted A size %dx%d\nenergy reduction %g\n", A.cols, A.rows, B.cols,
                        B.rows, diag);
        }
        if (bad) throw Error(RAMA_ERR_BAD_CONTRACTION, "Found bad contractions");
        A = std::move(B);
        map_node_labels(ctx, cur.get(), cur_size, out.labels.get(), N);
        st.end(ctx, "contract");
        if (st.on)
            std::fprintf(stderr, "round %d: %lld edges, %s, %.3f ms, %lld launches, %lld syncs\n", iter,
                         (long long)e0, mm_branch ? "matching" : "forest",
                         std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - r0).count(),
                         (long long)(launch_count() - l0), (long long)(ctx.syncs - s0));
        out.iterations = iter + 1;
        if (o.dump_timeline) {
            std::vector<int> snap(N);
            ctx.d2h(snap.data(), out.labels.get(), N);
            out.timeline.push_back(std::move(snap));
        }
        if (o.max_time_sec >= 0) {
            // whole elapsed seconds, strictly over the budget (src/rama_cuda.cu:151-157);
            // RAMA_CLOCK_OFFSET_SEC adds whole seconds to the elapsed time, a
            // test hook that makes the rule observable on sub-second solves
            auto t = std::chrono::duration_cast<std::chrono::seconds>(std::chrono::steady_clock::now() - t0).count();
            if (const char* off = std::getenv("RAMA_CLOCK_OFFSET_SEC")) t += std::atol(off);
            if (t > o.max_time_sec) break;
        }
    }
    scan_check(ctx);
    if (st.on) std::fprintf(stderr, "solve: %d rounds, %lld host synchronisations\n", out.iterations, (long long)ctx.syncs);
}

}  // namespace rama
