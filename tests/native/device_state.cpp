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

// `layers` x `width` events of `preds` predecessors each (the same place in the
// layer before, and the next ones), exponential delays.
struct Dag {
    mcdp_propagator *p = nullptr;
    int E, L;
    Dag(int layers, int width, int preds = 1) : E(layers * width), L((layers - 1) * width * preds) {
        std::vector<double> earliest(E, 0.0), dur(L, 1.0);
        std::vector<int32_t> idx(L), type(L, 0), target, src(L), act(L);
        std::vector<int64_t> off{0};
        for (int l = 0; l < L; ++l) {
            const int e = width + l / preds, k = l % preds;
            idx[l] = act[l] = l;
            src[l] = (e / width - 1) * width + (e + k) % width;
            if (k == preds - 1) {
                target.push_back(e);
                off.push_back(l + 1);
            }
        }
        mcdp_generator *gen = nullptr;
        OK(mcdp_generator_create(&gen));
        OK(mcdp_generator_add_exponential(gen, 0, 2.0, 50.0));
        OK(mcdp_propagator_create(E, earliest.data(), L, idx.data(), dur.data(), type.data(), (int)target.size(),
                                  target.data(), off.data(), src.data(), act.data(), 1800.0, gen, &p));
        mcdp_generator_destroy(gen);
    }
    // what a run of n samples launches
    int route(int64_t n, bool injected, bool durations, bool two_pass = true) {
        int32_t r = 0;
        void *rows = nullptr;
        OK(mcdp_malloc(&rows, 8));
        auto *x = (double *)rows;
        OK(mcdp_debug_two_pass_mode(p, two_pass ? 0 : 2));
        OK(injected ? mcdp_propagate_device(p, x, n, n, x, (int32_t *)rows, nullptr)
                    : mcdp_run_many_device(p, (int32_t *)rows, n, n, x, durations ? x : nullptr, (int32_t *)rows, nullptr));
        OK(mcdp_debug_last_route(p, &r));
        OK(mcdp_free(rows));
        fake::dead_accesses = 0;  // (the launchers were given no rows)
        return r;
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

// Device arrays of a run of n samples.
struct Rows {
    void *seeds = nullptr, *realized = nullptr, *durations = nullptr, *cause = nullptr;
    int64_t n;
    Rows(const Dag &d, int64_t n_) : n(n_) {
        OK(mcdp_malloc(&seeds, 4 * n));
        OK(mcdp_malloc(&realized, 8 * n * d.E));
        OK(mcdp_malloc(&durations, 8 * n * d.L));
        OK(mcdp_malloc(&cause, 4 * n * d.E));
    }
    int run(const Dag &d, bool with_durations, void *stream) const {
        return mcdp_run_many_device(d.p, (const int32_t *)seeds, n, n, (double *)realized,
                                    with_durations ? (double *)durations : nullptr, (int32_t *)cause, stream);
    }
    ~Rows() {
        for (void *p : {seeds, realized, durations, cause}) OK(mcdp_free(p));
    }
};

// A propagator that has run once, short (two launches) or long (the walk): a
// run of the other kind is captured and replayed, with nothing allocated by
// the replay.
void capture_after_a_run(bool first_short, bool durations, int64_t n) {
    Dag d(20, 30);
    const Rows first(d, first_short ? 10 : 200000), then(d, n);
    void *stream = nullptr, *graph = nullptr;
    OK(mcdp_stream_create(&stream));
    OK(first.run(d, true, nullptr));
    OK(mcdp_graph_capture_begin(stream));
    OK(then.run(d, durations, stream));
    OK(mcdp_graph_capture_end(stream, &graph));
    if (graph) {
        const int allocated = fake::allocations, launched = fake::launches;
        OK(mcdp_graph_launch(graph, stream));
        CHECK(fake::launches > launched && fake::allocations == allocated);
        OK(mcdp_graph_destroy(graph));
    }
    OK(mcdp_stream_destroy(stream));
}

// A propagator that has only walked runs short beside another stream's
// capture, which goes on.
void short_run_beside_a_capture() {
    Dag d(20, 30), other(20, 30);
    const Rows walk(d, 200000), small(d, 10), captured(other, 200000);
    void *stream = nullptr, *beside = nullptr, *graph = nullptr;
    OK(mcdp_stream_create(&stream));
    OK(mcdp_stream_create(&beside));
    OK(walk.run(d, true, nullptr));
    OK(captured.run(other, true, nullptr));
    OK(mcdp_graph_capture_begin(stream));
    OK(captured.run(other, true, stream));
    OK(small.run(d, true, beside));
    OK(mcdp_graph_capture_end(stream, &graph));
    if (graph) OK(mcdp_graph_destroy(graph));
    OK(mcdp_stream_destroy(stream));
    OK(mcdp_stream_destroy(beside));
}

// A propagator that has not run has nothing on the device: a capture of its
// first run fails, and the propagator works afterwards.
void capture_of_a_first_run() {
    Dag d(20, 30);
    const Rows rows(d, 200000);
    void *stream = nullptr, *graph = nullptr;
    OK(mcdp_stream_create(&stream));
    OK(mcdp_graph_capture_begin(stream));
    CHECK(rows.run(d, true, stream) != MCDP_OK);
    CHECK(mcdp_graph_capture_end(stream, &graph) != MCDP_OK);
    OK(rows.run(d, true, stream));
    OK(mcdp_stream_destroy(stream));
}

// Statistics of a short run on a device with room for its rows, but not for
// the durations that the two-pass route would hold beside them.
void statistics_in_little_memory() {
    Dag d(20, 30);
    const int64_t n = 2000, rows = n * d.E * 9;
    const std::vector<int32_t> seeds(n, 1);
    std::vector<double> mean(d.E);
    std::vector<int64_t> counts(d.E + d.L);
    int32_t two_pass = 0;
    OK(mcdp_debug_short_run(d.p, 0, n, &two_pass));
    CHECK(two_pass == 1);
    fake::memory = rows + (4 << 20);
    for (int i = 0; i < 2; ++i)
        OK(mcdp_run_stats_host(d.p, seeds.data(), n, 0, nullptr, mean.data(), nullptr, counts.data()));
    fake::memory = rows / 2;
    CHECK(mcdp_run_stats_host(d.p, std::vector<int32_t>(2 * n, 1).data(), 2 * n, 0, nullptr, mean.data(), nullptr,
                              counts.data()) == MCDP_E_NOMEM);
}

// A short run of a propagator that has walked, on a device with no room left
// for another plan.
void short_run_without_room_for_its_plan() {
    Dag d(20, 30);
    const Rows walk(d, 200000), small(d, 10);
    OK(walk.run(d, true, nullptr));
    fake::memory = fake::used;
    OK(small.run(d, true, nullptr));
    fake::memory += (size_t)1 << 30;
    const int before = fake::allocations;
    OK(small.run(d, true, nullptr));
    CHECK(fake::allocations > before);  // two passes as soon as there is room
}

// Statistics with a workspace of more than a propagator keeps leave it to the
// process, which frees it when asked to; the next call has another one.
void release_of_workspaces() {
    Dag d(20, 500);
    const int64_t n = 60000;  // 5.4 GB of rows
    const std::vector<int32_t> seeds(n, 1);
    std::vector<double> mean(d.E);
    auto stats = [&] {
        OK(mcdp_run_stats_host(d.p, seeds.data(), n, 0, nullptr, mean.data(), nullptr, nullptr));
    };
    stats();
    const size_t held = fake::used;
    CHECK(held > (size_t)5 << 30);
    stats();
    CHECK(fake::used == held);
    OK(mcdp_release_workspaces());
    CHECK(fake::used < (size_t)1 << 30);
    OK(mcdp_release_workspaces());
    stats();
    CHECK(fake::used == held);
}

// Walks of up to 128 groups of 64 samples, where wide steps are the cheaper
// route although one-sample tiles fit the device at once.
void wide_steps_below_a_round() {
    Dag fan(40, 60, 40), net(200, 100, 3), wide(60, 250, 3), light(60, 40, 1);
    CHECK(fan.route(8000, false, false) == MCDP_ROUTE_WIDE_STEPS);
    CHECK(fan.route(8192, true, false, false) == MCDP_ROUTE_WIDE_STEPS);
    CHECK(net.route(6208, true, false, false) == MCDP_ROUTE_WIDE_STEPS);
    CHECK(net.route(8192, true, false, false) == MCDP_ROUTE_WIDE_STEPS);
    CHECK(wide.route(8192, false, true, false) == MCDP_ROUTE_WIDE_STEPS);
    CHECK(light.route(6144, false, false) == MCDP_ROUTE_WIDE_STEPS);
    CHECK(light.route(8192, false, false) == MCDP_ROUTE_ONE_SAMPLE_TILES);
    CHECK(net.route(8193, true, false, false) != MCDP_ROUTE_WIDE_STEPS);
}

// The shape a first walk chooses: two samples per lane wherever a step holds the
// widest level, although one-sample shapes may have more samples resident.
void shapes_of_two_samples_per_lane() {
    for (int width : {10, 30, 40, 60, 66, 80, 96, 100, 128}) {
        Dag d(6, width, 2);
        int64_t info[10] = {};
        (void)d.route(200000, false, true);
        OK(mcdp_propagator_plan_info(d.p, info, 10));
        if (info[9] != 2) std::printf("width %d: waves %d, events per wave %d\n", width, (int)info[1], (int)info[8]);
        CHECK(info[0] == 6 && info[9] == 2);
    }
}

// Short runs take two passes where those were measured to be faster, and walk
// where they were not: with predecessors past an item's inline ones, with
// few samples a workgroup because many values live, with many rounds.
void two_passes_where_they_are_faster() {
    Dag small(20, 10, 2), net(200, 100, 3), wide(60, 250, 3), fan(40, 60, 40), levels2000(6, 2000, 3), seven(9, 59, 7),
        narrow(179, 8, 2), tiny(9, 8, 1);
    CHECK(small.route(1, false, true) == MCDP_ROUTE_TWO_PASS);
    CHECK(net.route(1, false, true) == MCDP_ROUTE_TWO_PASS);
    CHECK(net.route(1000, false, true) == MCDP_ROUTE_TWO_PASS);
    CHECK(net.route(4001, true, false) == MCDP_ROUTE_TWO_PASS);
    CHECK(wide.route(12345, false, true) == MCDP_ROUTE_TWO_PASS);
    CHECK(fan.route(100, false, true) == MCDP_ROUTE_TWO_PASS);
    CHECK(fan.route(6000, false, true) != MCDP_ROUTE_TWO_PASS);
    CHECK(fan.route(6000, true, false) != MCDP_ROUTE_TWO_PASS);
    CHECK(levels2000.route(8000, true, false) != MCDP_ROUTE_TWO_PASS);
    CHECK(levels2000.route(20000, true, false) != MCDP_ROUTE_TWO_PASS);
    CHECK(seven.route(22000, true, false) != MCDP_ROUTE_TWO_PASS);
    CHECK(net.route(20000, false, true) != MCDP_ROUTE_TWO_PASS);
    CHECK(narrow.route(8192, false, true) == MCDP_ROUTE_TWO_PASS);
    (void)tiny.route(200000, false, true);  // a walk: the shape is chosen
    CHECK(tiny.route(1000, false, true) == MCDP_ROUTE_TWO_PASS);
    CHECK(tiny.route(31001, false, true) != MCDP_ROUTE_TWO_PASS);
}

}  // namespace

int main(int argc, char **argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "graph_of_large_workspace") {
        graph_of_large_workspace();
    } else if (what == "capture_of_a_walk_after_a_short_run") {
        capture_after_a_run(true, true, 200000);
    } else if (what == "capture_without_durations_after_a_short_run") {
        capture_after_a_run(true, false, 10);
    } else if (what == "capture_of_a_short_run_after_a_walk") {
        capture_after_a_run(false, true, 10);
    } else if (what == "short_run_beside_a_capture") {
        short_run_beside_a_capture();
    } else if (what == "capture_of_a_first_run") {
        capture_of_a_first_run();
    } else if (what == "statistics_in_little_memory") {
        statistics_in_little_memory();
    } else if (what == "short_run_without_room_for_its_plan") {
        short_run_without_room_for_its_plan();
    } else if (what == "release_of_workspaces") {
        release_of_workspaces();
    } else if (what == "wide_steps_below_a_round") {
        wide_steps_below_a_round();
    } else if (what == "shapes_of_two_samples_per_lane") {
        shapes_of_two_samples_per_lane();
    } else if (what == "two_passes_where_they_are_faster") {
        two_passes_where_they_are_faster();
    } else {
        std::printf("no such scenario\n");
        return 1;
    }
    CHECK(fake::dead_accesses == 0);
    if (!failures) std::printf("OK\n");
    return failures != 0;
}
