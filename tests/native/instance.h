// A simulated ARG of k haplotypes over L columns, the last removed (a threading
// instance) or not.
#pragma once

#include <cmath>
#include <vector>

#include "../../include/argweaver_amd.h"

struct Instance {
    int k, L, T = 20;
    std::vector<double> times, pops, u;
    std::vector<char> buf;
    std::vector<char *> seqs;
    LocalTrees *trees;
    double rho = 1.6e-7, mu = 1.8e-7;
    Instance(int k, int L, double N = 1e4, bool remove = true) : k(k), L(L), u(L, 0.5), buf((size_t)k * L)
    {
        for (int i = 0; i < T; i++) times.push_back((exp(i / (T - 1.0) * log(1 + .01 * 200e3)) - 1) / .01);
        pops.assign(T, N);
        trees = awamd_simulate(k, L, times.data(), T, pops.data(), rho, mu, 5, buf.data());
        for (int i = 0; i < k; i++) seqs.push_back(&buf[(size_t)i * L]);
        if (remove) awamd_remove_thread(trees, k - 1);
    }
    int add(void *batch)
    {
        return awamd_batch_add(batch, trees, times.data(), T, pops.data(), rho, mu, seqs.data(), k - 1,
                               u.data());
    }
};
