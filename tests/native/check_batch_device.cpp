// A batch made while one device is current is filled, run and read by a thread
// with another one current.
#include "fake_hip.h"

#include "../../include/argweaver_amd.h"
#include "instance.h"

int main()
{
    Instance in(4, 3000);
    hipSetDevice(1);
    void *b = awamd_batch_new();
    REQUIRE(in.add(b) == 0);
    REQUIRE(awamd_batch_upload(b) == 0);
    hipSetDevice(0);
    for (int prec = 0; prec < 2; prec++) {
        REQUIRE(awamd_batch_run(b, prec, 0, 1, nullptr) == 0);
        std::vector<double> table(awamd_batch_W(b, 0));
        std::vector<int> path(in.L);
        REQUIRE(awamd_batch_alpha(b, 0, table.data()) == 0);
        REQUIRE(awamd_batch_alpha_range(b, 0, 7, 9, table.data()) == 0);
        REQUIRE(awamd_batch_path(b, 0, path.data()) == 0);
    }
    const int tiles[] = {0, 100};
    REQUIRE(awamd_batch_tune(b, 1, tiles, 2, nullptr) >= 0);
    awamd_batch_clear(b);
    REQUIRE(in.add(b) == 0);
    REQUIRE(awamd_batch_upload(b) == 0);
    REQUIRE(fake::device == 0);
    awamd_batch_free(b);
    printf("ok\n");
}
