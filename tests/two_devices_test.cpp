// Contexts on two devices driven from the same and from other threads: every
// buffer of a context lies on the context's device, whichever device is
// current on the thread that calls, small blocks and large ones, new ones and
// those that closed contexts left behind; a call leaves the caller's device
// current.
#include "fake_hip.hpp"
#include "pra.h"

#include <cstdint>
#include <thread>
#include <vector>

#define CHECK(x)                                                     \
    do {                                                             \
        if (!(x)) {                                                  \
            printf("line %d: %s\n", __LINE__, #x);                   \
            std::exit(1);                                            \
        }                                                            \
    } while (0)

static pra_ctx* create(int device)
{
    pra_ctx* c = nullptr;
    CHECK(pra_ctx_create(device, 3, 0, &c) == PRA_OK);
    return c;
}

// loads n equal-width relations of `rows` rows each
static void load(pra_ctx* c, int n, size_t rows)
{
    std::vector<uint64_t> data(rows * 3);
    for (size_t i = 0; i < data.size(); i++) data[i] = i;
    for (int k = 0; k < n; k++) {
        pra_rel* r = nullptr;
        CHECK(pra_rel_create(c, 2, 1, (uint32_t)k, 1, &r) == PRA_OK);
        CHECK(pra_rel_load_rows(r, data.data(), rows, PRA_FULL) == PRA_OK);
    }
}

int main()
{
    const size_t large = 3000000;   // 72 MB
    // a closed context of each device leaves idle blocks behind
    for (int d = 0; d < 2; d++) {
        pra_ctx* c = create(d);
        load(c, 8, 1);
        load(c, 1, large);
        CHECK(pra_ctx_synchronize(c) == PRA_OK);
        CHECK(pra_ctx_destroy(c) == PRA_OK);
    }
    pra_ctx *c0 = create(0), *c1 = create(1);
    for (int current = 0; current < 2; current++)
        for (pra_ctx* c : {c0, c1}) {
            hipSetDevice(current);
            load(c, 2, 1);
            CHECK(fake::current == current);
            load(c, 1, large);
            CHECK(fake::current == current);
        }
    // a new thread's current device is the first
    std::thread t([&] {
        load(c1, 4, 1);
        load(c1, 1, large);
    });
    t.join();
    // beyond what the closed contexts left
    load(c0, 64, 1);
    load(c1, 64, 1);
    hipSetDevice(0);
    CHECK(pra_ctx_destroy(c1) == PRA_OK);
    CHECK(pra_ctx_destroy(c0) == PRA_OK);
    CHECK(fake::foreign == 0);
    printf("ok\n");
    return 0;
}
