// A table copy that fails midway returns when nothing writes to its staging memory
// any more, and the next one gets the whole table.
#include "fake_hip.h"

#include "instance.h"

int main()
{
    Instance in(4, 30000);
    void *b = awamd_batch_new();
    REQUIRE(in.add(b) == 0 && awamd_batch_upload(b) == 0 && awamd_batch_run(b, 0, 0, 1, nullptr) == 0);
    std::vector<double> table(awamd_batch_W(b, 0), 1.0);
    fake::kernels = 0;
    REQUIRE(awamd_batch_alpha(b, 0, table.data()) == 0);
    REQUIRE(fake::pending() == 0);
    const int pieces = fake::kernels;
    REQUIRE(pieces > 3);
    for (int good = 0; good < pieces; good++) {
        fake::good_launches = good;
        REQUIRE(awamd_batch_alpha(b, 0, table.data()) != 0);
        REQUIRE(fake::pending() == 0);
    }
    fake::good_launches = -1;
    const std::vector<double> before = table;
    std::fill(table.begin(), table.end(), 1.0);
    REQUIRE(awamd_batch_alpha(b, 0, table.data()) == 0);
    REQUIRE(!memcmp(table.data(), before.data(), table.size() * sizeof(double)));
    awamd_batch_free(b);
    printf("ok\n");
}
