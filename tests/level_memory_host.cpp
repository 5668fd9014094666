// level_memory_host.cpp -- levels short of memory, on the host runtime of
// host_runtime.h: memory that only buys speed is given up before a call is
// refused.
#include "host_runtime.h"

#include <cstdio>
#include <vector>

#include "camr_hydro.h"

static int bad = 0;
#define CHECK(c, ...)                                                          \
    do {                                                                       \
        if (!(c)) {                                                            \
            ++bad;                                                             \
            printf("FAILED %s: ", #c);                                         \
            printf(__VA_ARGS__);                                               \
            printf(" (%s)\n", camr_last_error());                              \
        }                                                                      \
    } while (0)

static camr_level_desc desc(int n, const std::vector<int32_t> &boxes) {
    camr_level_desc d;
    camr_default_level_desc(&d);
    for (int x = 0; x < 3; ++x) {
        d.hp.domlo[x] = 0;
        d.hp.domhi[x] = n - 1;
        d.hp.dx[x] = 1.0 / n;
        d.hp.bclo[x] = d.hp.bchi[x] = CAMR_BC_INTERIOR;
        d.is_periodic[x] = 1;
    }
    d.cfl = 0.3;
    d.nbox = (int32_t)boxes.size() / 6;
    d.box_lohi = boxes.data();
    return d;
}

// Method of lines: each allocation of the level-wide source (the last three
// of a creation) may fail; the level is created all the same, steps, and no
// error is left behind for a later launch.
static void mol() {
    const std::vector<int32_t> boxes = {0, 0, 0, 15, 15, 7, 0, 0, 8, 15, 15, 15};
    camr_level_desc d = desc(16, boxes);
    d.hp.do_mol = 1;
    long launches[2] = {0, 0};  // a step's, with and without the level-wide source
    fake::mallocs = 0;
    camr_level *L = nullptr;
    CHECK(camr_level_create(&d, &L) == CAMR_OK, "create");
    const long n = fake::mallocs;
    const size_t all = fake::used;
    auto step = [&](camr_level *l) {
        fake::launches = 0;
        CHECK(camr_level_advance(l, 1e-3) == CAMR_OK, "step");
        return fake::launches;
    };
    launches[0] = step(L);
    camr_level_destroy(L);
    CHECK(fake::used == 0, "%zu bytes left", fake::used);
    for (int k = 0; k < 3; ++k) {
        fake::fail_at = n - k;
        L = nullptr;
        CHECK(camr_level_create(&d, &L) == CAMR_OK, "allocation %ld of %ld refused", n - k, n);
        CHECK(fake::last == hipSuccess, "allocation %ld: error left", n - k);
        if (!L) continue;
        CHECK(fake::used < all, "allocation %ld: %zu bytes of %zu kept", n - k, fake::used, all);
        launches[1] = step(L);
        CHECK(launches[1] > launches[0], "launches %ld, %ld", launches[0], launches[1]);
        camr_level_destroy(L);
        CHECK(fake::used == 0, "%zu bytes left", fake::used);
    }
    fake::fail_at = 0;
    printf("method of lines: %ld launches a step, %ld without the level-wide source\n", launches[0],
           launches[1]);
}

int main() {
    mol();
    printf(bad ? "%d FAILED\n" : "LEVEL MEMORY OK\n", bad);
    return bad != 0;
}
