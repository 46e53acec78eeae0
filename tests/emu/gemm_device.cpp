// Host-side check of the device form of a grouped GEMM stage -- test code: the operand and output
// addresses of every element of the folded T-GEMMs equal those of the plan's own problems.
#include <cstdio>
#include <stdexcept>

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
