// Host-side checks of the device form of a grouped GEMM stage -- test code: the operand and output
// addresses of every element of the folded T-GEMMs equal those of the plan's own problems, and the
// work items of a schedule cover every element of C and of its reduction once.
#include <algorithm>
#include <cstdio>
#include <stdexcept>
#include <vector>

#include "descriptors.hpp"
#include "plans.hpp"

using namespace mq;

extern "C" long fold_check(int sym, const mq_mpo_desc* md, const mq_bindex_desc* Ld, const mq_bindex_desc* Rd,
                           const mq_index_desc* li, const mq_index_desc* pi, const mq_index_desc* ri) {
    try {
        MPO mpo(*md);
        BoundaryIndex L = boundary_index_from(*Ld), R = boundary_index_from(*Rd);
        L.layout();
        R.layout();
        HpsiPlanHost P = build_hpsi_plan(Sym(sym), mpo, L, R, Index(*li), Index(*pi), Index(*ri));
        std::vector<GemmDesc> F = fold_batches(P.t_gemms);
        require(F.size() == P.t_gemms.size(), "fold: problems lost");
        long folded = 0;
        for (size_t p = 0; p < F.size(); ++p) {
            GemmDesc const &g = P.t_gemms[p], &f = F[p];
            const bool fold = f.flags & GEMM_NBLOCKS;
            folded += fold;
            require(f.M == g.M && f.K == g.K && f.N * f.batch == g.N * g.batch && f.a == g.a && f.base_a == g.base_a &&
                        f.base_b == g.base_b && f.base_c == g.base_c, "fold: shape");
            require(fold || (f.N == g.N && f.batch == g.batch && f.flags == g.flags), "fold: untouched problem changed");
            for (int32_t b = 0; b < g.batch; ++b)
                for (int32_t n = 0; n < g.N; ++n) {
                    const int32_t nf = fold ? b * g.N + n : n, bf = fold ? 0 : b;
                    for (int32_t k = 0; k < g.K; ++k) {
                        const bool tb = g.flags & GEMM_TRANS_B;
                        const int64_t want = g.b + b * g.sb + (tb ? n + int64_t(k) * g.ldb : k + int64_t(n) * g.ldb);
                        int64_t got = f.b + bf * f.sb;
                        if (fold) got += int64_t(nf / f.nb) * f.sb + nf % f.nb + int64_t(k) * f.ldb;
                        else got += tb ? nf + int64_t(k) * f.ldb : k + int64_t(nf) * f.ldb;
                        require(got == want, "fold: B address");
                    }
                    // column index of C in units of the row's leading dimension
                    require(nf + int64_t(bf) * f.sc == n + int64_t(b) * g.sc, "fold: C column");
                }
        }
        return folded;
    } catch (std::exception const& e) {
        fprintf(stderr, "fold_check: %s\n", e.what());
        return -1;
    }
}

// columns of a stacked transposed problem of `batch` blocks of N once folded, and its column tiles as
// the schedule counts them (32-bit arithmetic)
extern "C" void fold_columns(int N, int batch, long* columns, long* tiles) {
    GemmDesc g{};
    g.M = g.K = 1;
    g.N = N;
    g.batch = batch;
    g.sc = N;
    g.flags = GEMM_ROWMAP | GEMM_TRANS_B;
    const GemmDesc f = fold_batches({g})[0];
    *columns = f.N;
    const int32_t bn = gemm_bn(0);
    *tiles = long(int32_t(uint32_t(f.N) + uint32_t(bn) - 1) / bn);
}

// C problems of the given sizes
static std::vector<GemmDesc> problems(int n, const int* M, const int* N, const int* K, int batch, int flags) {
    std::vector<GemmDesc> G;
    for (int i = 0; i < n; ++i) {
        GemmDesc g{};
        g.M = M[i];
        g.N = N[i];
        g.K = K[i];
        g.batch = batch;
        g.flags = flags;
        G.push_back(g);
    }
    return G;
}

// the policies that the autotuner times for a stage, one bit each
extern "C" long candidate_policies(int n, const int* M, const int* N, const int* K, int batch, int flags) {
    long bits = 0;
    for (GemmCandidate const& c : gemm_candidates(problems(n, M, N, K, batch, flags))) bits |= 1L << c.policy;
    return bits;
}

// the autotuner's key of a stage, and the tiles of its schedule without a split along K
extern "C" uint64_t stage_key(int n, const int* M, const int* N, const int* K, int batch, long* tiles) {
    const std::vector<GemmDesc> G = problems(n, M, N, K, batch, 0);
    *tiles = long(build_gemm_schedule(G, 0, 16).n_tiles());
    return gemm_stage_key(G);
}

// work items of C problems of the given sizes under schedule candidate `policy`; splits or -1
extern "C" long items_check(int n, const int* M, const int* N, const int* K, int batch, int policy) {
    try {
        const std::vector<GemmDesc> G = problems(n, M, N, K, batch, 0);
        const GemmSchedule sch = build_gemm_schedule(G, gemm_policy(policy));
        std::vector<std::vector<int64_t>> done(size_t(n) * batch);
        for (int i = 0; i < n; ++i)
            for (int b = 0; b < batch; ++b) done[size_t(i) * batch + b].assign(size_t(M[i]) * N[i], 0);
        std::vector<char> ws(sch.ws_elems, 0);
        long splits = 0;
        for (GemmItem const& t : gemm_items(G, sch)) {
            GemmDesc const& g = G.at(size_t(t.prob));
            const int nl = std::min(128, g.N - t.n0);
            require(t.ml > 0 && t.ml <= t.bm && t.bm <= 128 && t.m0 + t.ml <= g.M && nl > 0, "items: shape");
            require(t.k0 >= 0 && t.k0 < t.k1 && t.k1 <= g.K && t.k0 % 16 == 0, "items: K range");
            require(t.ws >= 0 || t.k1 - t.k0 == g.K, "items: split without a partial");
            auto& d = done[size_t(t.prob) * batch + t.batch];
            for (int c = 0; c < nl; ++c)
                for (int r = 0; r < t.ml; ++r) {
                    d[size_t(t.m0 + r) + size_t(t.n0 + c) * g.M] += t.k1 - t.k0;
                    if (t.ws >= 0) {
                        char& w = ws.at(size_t(t.ws + r + int64_t(c) * t.bm));
                        require(!w, "items: partials overlap");
                        w = 1;
                    }
                }
            splits += t.ws >= 0;
        }
        for (int i = 0; i < n; ++i)
            for (int b = 0; b < batch; ++b)
                for (int64_t v : done[size_t(i) * batch + b]) require(v == K[i], "items: cover");
        return splits;
    } catch (std::exception const& e) {
        fprintf(stderr, "items_check: %s\n", e.what());
        return -1;
    }
}
