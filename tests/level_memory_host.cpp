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

// Cut-cell boxes: the buffers per transverse pair (forward and adjoint) are
// given up where the level, its gradient or more checkpoints would not fit
// with them; what pair by pair needs is enough, and less than that is refused.
struct EbRun {
    int made = 0, grad = 0, again = 0;  // return codes of the three
    int back = 0;                       // of a backward pass on what is left
    long launched = 0;                  // by it
    size_t peak = 0;
};
static EbRun eb(int merge, size_t cap, int lose = 0) {
    const int n = 16;
    const std::vector<int32_t> boxes = {0, 0, 0, 15, 15, 7, 0, 0, 8, 15, 15, 15};
    camr_level_desc d = desc(n, boxes);
    d.hp.ppm_type = 0;
    d.engine = 1;
    d.fixed_dt = 1e-3;
    fake::cap = cap;
    fake::peak = 0;
    fake::last = hipSuccess;
    EbRun r;
    camr_level *L = nullptr;
    r.made = camr_level_create(&d, &L);
    const int32_t flo[3] = {-7, -7, -7}, fhi[3] = {n + 6, n + 6, n + 6};
    const int m = n + 14;
    std::vector<int32_t> flags((size_t)m * m * m, (1 << 27) - 1);
    for (int k : {4, 12})  // a cut cell in each box
        flags[(8 + 7) + (8 + 7) * m + (size_t)(k + 7) * m * m] |= 1 << 27;
    if (!r.made) r.made = camr_level_set_eb_merge(L, merge);
    if (!r.made) r.made = camr_level_set_eb(L, flags.data(), flo, fhi);
    std::vector<double> one((size_t)(n + 15) * (n + 15) * 23, 1.0), off(2 * one.size(), 0.0);
    for (int b = 0; b < 2 && !r.made; ++b)
        r.made = camr_level_set_box_eb(L, b, one.data(), one.data(), one.data(), one.data(),
                                       off.data(), off.data(), off.data());
    const std::vector<double> dts(6, 1e-3);
    auto gradient = [&](int steps, int every) {
        int rc = camr_level_adjoint_forward(L, steps, dts.data(), every);
        return rc ? rc : camr_level_adjoint_backward(L);
    };
    if (!r.made && lose) {
        // what a failed gradient gives up is gone (2: after one that fitted): the
        // level neither steps nor goes backward on arrays it no longer has
        if (lose == 2) {
            CHECK(gradient(1, 1) == CAMR_OK, "first gradient");
            fake::cap = fake::used;
        }
        fake::lose_freed = true;
        r.grad = camr_level_adjoint_forward(L, 6, dts.data(), 1);
        fake::lose_freed = false;
        fake::fail_at = 0;
        r.again = camr_level_advance(L, 1e-3);
        fake::launches = 0;
        r.back = camr_level_adjoint_backward(L);
        r.launched = fake::launches;
    } else if (!r.made && !(r.grad = gradient(1, 1))) {
        r.again = gradient(6, 2);
    }
    if (!r.made && !r.grad && !r.again) CHECK(fake::last == hipSuccess, "error left");
    if (L) camr_level_destroy(L);
    CHECK(fake::used == 0, "%zu bytes left", fake::used);
    r.peak = fake::peak;
    fake::cap = size_t(1) << 40;
    return r;
}
static void eb_levels() {
    const EbRun lean = eb(0, fake::cap), full = eb(1, fake::cap);
    CHECK(!lean.made && !lean.grad && !lean.again, "%d %d %d", lean.made, lean.grad, lean.again);
    CHECK(!full.made && !full.grad && !full.again, "%d %d %d", full.made, full.grad, full.again);
    CHECK(full.peak > lean.peak, "%zu, %zu bytes", full.peak, lean.peak);
    for (int s = 0; s <= 40; ++s) {
        const size_t cap = lean.peak + (full.peak - lean.peak) * s / 40;
        const EbRun r = eb(1, cap);
        CHECK(!r.made && !r.grad && !r.again, "%zu of %zu bytes: %d %d %d", cap, full.peak, r.made,
              r.grad, r.again);
    }
    for (int lose : {1, 2}) {
        const EbRun r = eb(1, lose == 1 ? lean.peak + (full.peak - lean.peak) / 4 : fake::cap, lose);
        CHECK(!r.made && r.grad && r.again == CAMR_ERR_ALLOC, "%d: %d %d %d", lose, r.made, r.grad,
              r.again);
        CHECK(r.back && r.launched == 0, "%d: %d after %ld launches", lose, r.back, r.launched);
    }
    for (int merge = 0; merge < 2; ++merge)
        for (int s = 1; s < 40; ++s) {
            const EbRun r = eb(merge, lean.peak * s / 40);
            CHECK(r.made || r.grad || r.again, "%d of 40 accepted", s);
        }
    printf("cut cells: %zu bytes pair by pair, %zu with a buffer per pair\n", lean.peak, full.peak);
}

int main() {
    mol();
    eb_levels();
    printf(bad ? "%d FAILED\n" : "LEVEL MEMORY OK\n", bad);
    return bad != 0;
}
