// Device memory kept for the next chain statistic: a batch that finds no memory
// gets it, and a server's budget counts it.
#include "fake_hip.h"

#include "host_stage.h"
#include "instance.h"
#include "local_trees.h"
#include "serve.h"

using namespace aw;

int main()
{
    Instance in(8, 20000);
    // two statistics at once leave two pieces in the pool
    const size_t before = fake::device_bytes, keep = size_t(30) << 20;
    {
        const StageUse a, b;
        REQUIRE(a.s && b.s && a.s->device(keep) && b.s->device(keep));
    }
    REQUIRE(fake::device_bytes == before + 2 * keep);
    // more than is kept of one call goes back with it
    {
        const StageUse a;
        REQUIRE(a.s->device(size_t(65) << 20));
    }
    const size_t kept = fake::device_bytes - before;
    REQUIRE(kept == keep);
    ServeOptions opt;
    opt.drivers = 2;
    REQUIRE(Server::share(opt) == (opt.hbm_budget - kept) / 2);
    opt.hbm_budget = 1000;
    REQUIRE(Server::share(opt) == 0);

    fake::device_limit = fake::device_bytes + (size_t(8) << 20);
    void *b = awamd_batch_new();
    REQUIRE(in.add(b) == 0);
    REQUIRE(awamd_batch_upload(b) == 0);
    REQUIRE(awamd_batch_run(b, 0, 0, 1, nullptr) == 0);
    REQUIRE(hipGetLastError() == hipSuccess);
    REQUIRE(idle_stage_bytes() == 0);
    // memory that is in use stays, and an allocation too large still fails
    const StageUse a;
    REQUIRE(a.s->device(1 << 20) && !free_idle_stage_memory());
    void *p;
    REQUIRE(device_malloc(&p, size_t(1) << 30) != hipSuccess);
    awamd_batch_free(b);
    printf("ok\n");
}
