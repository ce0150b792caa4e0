// The server's estimate of a request's device memory against what a batch of it
// allocates, at every count of states per lane.
#include "fake_hip.h"

#include "instance.h"
#include "local_trees.h"
#include "serve.h"

using namespace aw;

int main()
{
    const struct { int k, L; double N; int R; } cases[] = {
        {3, 500, 1e4, 1}, {8, 4000, 1e4, 2}, {20, 3000, 1e4, 4}, {30, 3000, 1e4, 0},
        {100, 2000, 2e4, 0}, {128, 1500, 3e4, 32}};
    for (const auto &c : cases) {
        Instance in(c.k, c.L, c.N);
        HostInstance hi;
        flatten(*reinterpret_cast<ArgTrees *>(in.trees), hi.ft);
        for (char *row : in.seqs) hi.rows.push_back(row);
        model_init(hi.model, in.T, in.times.data(), in.pops.data(), in.rho, in.mu);
        std::vector<int> S;
        instance_states(hi.ft, in.T, &S);
        const int Smax = *std::max_element(S.begin(), S.end());
        if (c.R == 32) REQUIRE(Smax > 1024);
        for (int prec = 0; prec < 2; prec++) {
            const size_t before = fake::device_bytes;
            void *b = awamd_batch_new();
            REQUIRE(in.add(b) == 0 && awamd_batch_upload(b) == 0);
            REQUIRE(awamd_batch_run(b, prec, 2000, 1, nullptr) == 0);
            const size_t used = fake::device_bytes - before;
            const size_t estimate = Server::footprint(hi, prec ? Precision::FP32 : Precision::FP64);
            printf("k %d states %d prec %d: used %zu, estimate %zu\n", c.k, Smax, prec, used, estimate);
            REQUIRE(estimate >= used);
            // no more than the variant rows (this runtime's kernels find none)
            REQUIRE(estimate <= used + 65536 + (size_t)c.L * 64 * 32 * 8);
            awamd_batch_free(b);
        }
    }
    printf("ok\n");
}
