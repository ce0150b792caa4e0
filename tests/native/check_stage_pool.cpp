// Staging memory that cannot be made in full leaves nothing behind.
#include "fake_hip.h"

#include "host_stage.h"

using namespace aw;

int main()
{
    for (int events = 0; events < 2; events++) {
        fake::good_events = events;
        REQUIRE(take_stage() == nullptr);
        REQUIRE(fake::live_events == 0);
    }
    fake::good_events = -1;
    HostStage *s = take_stage();
    REQUIRE(s && fake::live_events == 2);
    give_stage(s);
    REQUIRE(take_stage() == s);
    printf("ok\n");
}
