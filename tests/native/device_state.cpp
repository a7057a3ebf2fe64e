// What the host code keeps on the device between calls, against the runtime of
// fake_hip.cpp: `device_state <scenario>` prints OK, or what went wrong.
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "fake_hip.hpp"
#include "mcdp.h"

namespace {

int failures = 0;
#define CHECK(cond)                                                                                   \
    do {                                                                                              \
        if (!(cond)) {                                                                                \
            std::printf("line %d: %s (%s)\n", __LINE__, #cond, mcdp_last_error());                    \
            ++failures;                                                                               \
        }                                                                                             \
    } while (0)
#define OK(call) CHECK((call) == MCDP_OK)

// `layers` x `width` events, one predecessor each (the same place in the layer
// before), exponential delays.
struct Dag {
    mcdp_propagator *p = nullptr;
    int E, L;
    Dag(int layers, int width) : E(layers * width), L((layers - 1) * width) {
        std::vector<double> earliest(E, 0.0), dur(L, 1.0);
        std::vector<int32_t> idx(L), type(L, 0), target(L), src(L), act(L);
        std::vector<int64_t> off(L + 1);
        for (int l = 0; l < L; ++l) {
            idx[l] = act[l] = src[l] = l;
            target[l] = l + width;
            off[l + 1] = l + 1;
        }
        mcdp_generator *gen = nullptr;
        OK(mcdp_generator_create(&gen));
        OK(mcdp_generator_add_exponential(gen, 0, 2.0, 50.0));
        OK(mcdp_propagator_create(E, earliest.data(), L, idx.data(), dur.data(), type.data(), L, target.data(),
                                  off.data(), src.data(), act.data(), 1800.0, gen, &p));
        mcdp_generator_destroy(gen);
    }
    ~Dag() { mcdp_propagator_destroy(p); }
    Dag(const Dag &) = delete;
};

// A short run whose workspace is beyond what a propagator keeps, again and
// again: a captured graph of it must not outlive the workspace it was captured
// in, which goes back to the pool of the process after each call.
void graph_of_large_workspace() {
    Dag big(40, 90000);  // 4.6 GB for 64 samples
    OK(mcdp_propagator_configure(big.p, 16, 16, 1));
    const std::vector<int32_t> seeds(640, 1);
    for (int i = 0; i < 4; ++i) {
        OK(mcdp_run_many_host(big.p, seeds.data(), 64, nullptr, nullptr, nullptr));
        if (i == 2) {  // no room: the pool's workspaces are freed, and the next call has another one
            void *p = nullptr;
            CHECK(mcdp_malloc(&p, fake::memory) != MCDP_OK);
        }
    }
    CHECK(fake::dead_accesses == 0);
    const int before = fake::graph_launches;
    OK(mcdp_run_many_host(big.p, seeds.data(), 640, nullptr, nullptr, nullptr));
    CHECK(fake::graph_launches > before);  // ten chunks in one workspace still replay a graph
}

}  // namespace

int main(int argc, char **argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "graph_of_large_workspace") {
        graph_of_large_workspace();
    } else {
        std::printf("no such scenario\n");
        return 1;
    }
    CHECK(fake::dead_accesses == 0);
    if (!failures) std::printf("OK\n");
    return failures != 0;
}
