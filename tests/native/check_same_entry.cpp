// The same-branch entries P(a -> b) that the traceback forms from a block's
// time terms (same_entry), against what the forward of the same block adds to the
// other-branch entry: the products of its coefficient planes.  Internal
// threading prepares both on the host, from ARGs whose removed subtrees have any
// age, with and without a least age of the states.
//
// Tolerance: both are differences of terms no larger than M, rounded a few
// times; exp(x + y) against exp(x) exp(y) differs by half an ulp of x + y, which
// is below 100 here: 64 ulp of M.
#include "fake_hip.h"

#include "engine.h"
#include "instance.h"
#include "internal_prep.h"

using namespace aw;

int main()
{
    long entries = 0, aged = 0;
    for (int k : {4, 9, 25})
        for (double N : {1e4, 5e4})
            for (int minage : {0, 3}) {
                Instance in(k, 1500, N, false);
                ArgTrees &tr = *reinterpret_cast<ArgTrees *>(in.trees);
                Model m;
                model_init(m, in.T, in.times.data(), in.pops.data(), in.rho, in.mu);
                std::vector<int> path(tr.blocks.size());
                srand(k + minage);
                // through an inner node, whose subtree has an age
                arghmm_sample_arg_removal_path(in.trees, k + (int)N % 7 % (k - 2), path.data());
                arghmm_remove_arg_thread_path(in.trees, path.data(), in.T + 1);
                HostPrep hp;
                REQUIRE(prepare_internal(tr, m, in.seqs.data(), minage, hp) == 0);
                const int T1 = in.T - 1, R = hp.R, RW = 64 * R;
                for (size_t b = 0; b < tr.blocks.size(); b++) {
                    const double *pl = &hp.planes[b * NCOEF * RW], *tm = &hp.tm[b * T1 * T1];
                    const double *vec = &hp.tvec[b * time_vecs(T1)];
                    const int S = hp.S[b], *info = &hp.info[b * RW];
                    aged += vec[tv_minage(T1)] > 0;
                    for (int j = 0; j < S; j++)
                        for (int i = 0; i < S; i++) {
                            const int pi = lane_pos(i, R), pj = lane_pos(j, R);
                            if (info_node(info[pi]) != info_node(info[pj])) continue;
                            const int a = info[pi] & INFO_TIME, t = info[pj] & INFO_TIME;
                            const int c = info_age(info[pj]);
                            const double other = tm[a * T1 + t];
                            const double add = a < t   ? pl[CF * RW + pi] * pl[CG * RW + pj]
                                               : a > t ? pl[CD * RW + pi] * pl[CK * RW + pj]
                                                       : pl[CJ * RW + pj];
                            const double DE = vec[TV_D * T1 + a] * vec[TV_E * T1 + t];
                            const auto X = [&](int x) { return x >= 0 && x < t ? vec[tv_x(T1) + x * T1 + t] : 0.0; };
                            const double M = 2 * fabs(other) + DE * (2 * vec[TV_Y * T1 + t] + 2 * X(t - 1) + X(c - 1)) +
                                             (a == t ? vec[TV_NORECOMBS * T1 + a] : 0.0);
                            const double got = same_entry(vec, T1, a, t, c, &tm[a * T1 + t]);
                            REQUIRE(fabs(got - (other + add)) <= 64 * 2.3e-16 * M);
                            entries++;
                        }
                    // no way from or to an age that no thread has
                    for (int a = 0; a < (int)vec[tv_minage(T1)]; a++)
                        for (int t = 0; t < T1; t++)
                            REQUIRE(same_entry(vec, T1, a, t, 0, &tm[a * T1 + t]) == 0.0 &&
                                    same_entry(vec, T1, t, a, 0, &tm[t * T1 + a]) == 0.0);
                }
            }
    printf("%ld entries, %ld blocks of an age above 0\n", entries, aged);
    REQUIRE(entries > 10000 && aged > 20);
    printf("ok\n");
}
