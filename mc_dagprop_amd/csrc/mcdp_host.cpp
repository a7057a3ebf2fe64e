// Host side of libmcdp: the delay-generator registry, the context compiler
// that turns a DAG into a levelled, wave-scheduled device plan, and the C ABI
// declared in include/mcdp.h.
//
// Reference semantics followed here (WonJayne/mc_dagprop,
// src/mc_dagprop/monte_carlo/_core.cpp):
//   * validation order and messages: :196-201, :262-264;
//   * link table: link_count = max(idx) + 1, gaps are {0.0, type -1} (:213-229);
//   * the last precedence entry of a target supplies its predecessor list and
//     indegree, every entry adds adjacency, Kahn order with a FIFO (:232-264);
//   * per-event predecessor order is the input order (:266-285);
//   * links without a distribution keep minimal_duration (:303-306).
#include <hip/hip_runtime_api.h>

#include <fcntl.h>
#include <sys/mman.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <cerrno>
#include <cinttypes>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <fstream>
#include <sstream>
#include <limits>
#include <map>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "../../include/mcdp.h"
#include "mcdp_internal.hpp"
#include "mcdp_kernels.hpp"
#include "mcdp_plan.hpp"

using namespace mcdp;

namespace {
thread_local std::string g_last_error;
}  // namespace

namespace mcdp {
int fail(int code, const std::string &msg) {
    g_last_error = msg;
    return code;
}
int hip_fail(hipError_t e, const char *what) {
    return fail(MCDP_E_DEVICE, std::string(what) + ": " + hipGetErrorString(e));
}
}  // namespace mcdp

namespace {

// API-level distribution kinds (the reference's DistVar alternatives, :143).
enum ApiKind { kApiConstant, kApiExponential, kApiGamma, kApiEmpAbs, kApiEmpRel };

struct DistSpec {
    ApiKind kind;
    double a = 0.0, b = 0.0, c = 0.0;
    std::vector<double> values, weights;
};

// ---- regularized lower incomplete gamma P(a, x) ---------------------------
// Series  P = e^{-x} x^a / Gamma(a+1) * sum_n x^n / ((a+1)...(a+n))  for x < a+1,
// continued fraction for Q = 1 - P otherwise (Abramowitz & Stegun 6.5.29,
// 6.5.31; modified Lentz evaluation).  Used only to choose a sampling method.
double reg_lower_gamma(double a, double x) {
    if (!(x > 0.0)) return 0.0;
    if (std::isinf(x)) return 1.0;
    const double lg = std::lgamma(a);
    if (x < a + 1.0) {
        double term = 1.0 / a, sum = term, ap = a;
        for (int n = 0; n < 100000; ++n) {
            ap += 1.0;
            term *= x / ap;
            sum += term;
            if (std::fabs(term) < std::fabs(sum) * 1e-17) break;
        }
        return std::min(1.0, sum * std::exp(-x + a * std::log(x) - lg));
    }
    const double tiny = 1e-300;
    double b = x + 1.0 - a, c = 1.0 / tiny, d = 1.0 / b, h = d;
    for (int i = 1; i < 100000; ++i) {
        const double an = -i * (i - a);
        b += 2.0;
        d = an * d + b;
        if (std::fabs(d) < tiny) d = tiny;
        c = b + an / c;
        if (std::fabs(c) < tiny) c = tiny;
        d = 1.0 / d;
        const double del = d * c;
        h *= del;
        if (std::fabs(del - 1.0) < 1e-16) break;
    }
    const double q = std::exp(-x + a * std::log(x) - lg) * h;
    return std::max(0.0, 1.0 - q);
}

// ---- Vose alias table (M. D. Vose, IEEE TSE 17(9), 1991) -------------------
// P(bin j) = (prob[j] + sum_{i: alias[i] = j} (1 - prob[i])) / n = w_j / sum(w).
// Zero-weight bins get prob 0 and are never an alias target.
void build_alias(const std::vector<double> &w, std::vector<double> &prob, std::vector<int> &alias) {
    const size_t n = w.size();
    long double total = 0.0L;
    for (double x : w) total += x;
    std::vector<long double> p(n);
    std::vector<size_t> small, large;
    size_t heaviest = 0;
    for (size_t i = 0; i < n; ++i) {
        p[i] = (long double)w[i] * (long double)n / total;
        if (w[i] > w[heaviest]) heaviest = i;
    }
    // Zero-weight bins are pushed last so they pair first (stack order).
    for (size_t i = 0; i < n; ++i)
        if (p[i] < 1.0L && w[i] != 0.0) small.push_back(i);
    for (size_t i = 0; i < n; ++i)
        if (w[i] == 0.0) small.push_back(i);
    for (size_t i = 0; i < n; ++i)
        if (p[i] >= 1.0L) large.push_back(i);
    prob.assign(n, 1.0);
    alias.resize(n);
    for (size_t i = 0; i < n; ++i) alias[i] = (int)i;
    while (!small.empty() && !large.empty()) {
        const size_t l = small.back();
        small.pop_back();
        const size_t g = large.back();
        large.pop_back();
        prob[l] = (double)p[l];
        alias[l] = (int)g;
        p[g] = (p[g] + p[l]) - 1.0L;
        if (p[g] < 1.0L)
            small.push_back(g);
        else
            large.push_back(g);
    }
    for (size_t g : large) prob[g] = 1.0;
    for (size_t l : small) {  // rounding leftovers: p[l] is 1 up to rounding
        if (w[l] == 0.0) {
            prob[l] = 0.0;
            alias[l] = (int)heaviest;
        } else {
            prob[l] = 1.0;
        }
    }
}

bool all_finite_nonneg(const std::vector<double> &w, double &sum) {
    sum = 0.0;
    for (double x : w) {
        if (!std::isfinite(x) || x < 0.0) return false;
        sum += x;
    }
    return std::isfinite(sum) && sum > 0.0;
}

int compile_exponential(double lam, double m, DistRec &D) {
    if (std::isnan(lam) || lam < 0.0) return fail(MCDP_E_INVALID, "exponential lambda_ must be non-negative");
    if (std::isnan(m)) m = std::numeric_limits<double>::infinity();  // x > NaN never rejects (:86)
    if (m < 0.0) return fail(MCDP_E_INVALID, "exponential max_scale must be non-negative");
    if (lam == 0.0 || m == 0.0) {  // X == 0 always
        D.kind = kConstant;
        D.p[0] = 0.0;
    } else if (std::isinf(m)) {
        D.kind = kExpInf;
        D.p[0] = lam;
    } else {
        D.kind = kExpTrunc;
        D.p[0] = lam;
        D.p[1] = std::exp(-m / lam);     // q
        D.p[2] = m;
        D.p[3] = -std::expm1(-m / lam);  // 1 - q
    }
    return MCDP_OK;
}

int compile_gamma(double k, double th, double m, DistRec &D) {
    if (std::isnan(k) || !(k > 0.0) || std::isinf(k)) return fail(MCDP_E_INVALID, "gamma shape must be positive and finite");
    if (std::isnan(th) || !(th > 0.0) || std::isinf(th)) return fail(MCDP_E_INVALID, "gamma scale must be positive and finite");
    if (std::isnan(m)) m = std::numeric_limits<double>::infinity();
    if (m < 0.0) return fail(MCDP_E_INVALID, "gamma max_scale must be non-negative");
    if (m == 0.0) {
        D.kind = kConstant;
        D.p[0] = 0.0;
        return MCDP_OK;
    }
    if (k == 1.0) return compile_exponential(th, m, D);  // Gamma(1, th) = Exp(mean th)
    const double mp = m / th;
    const double p_rej = std::isinf(m) ? 1.0 : reg_lower_gamma(k, mp);
    double p_pow = 0.0;
    if (!std::isinf(m)) {
        const double lp = std::lgamma(k + 1.0) + std::log(std::max(p_rej, 1e-300)) - k * std::log(mp);
        p_pow = std::min(1.0, std::exp(lp));
    }
    if (p_rej >= 0.25 || p_rej >= p_pow) {
        if (p_rej < kMinAcceptance) return fail(MCDP_E_INVALID, "gamma max_scale truncation too severe to sample");
        D.p[0] = th;
        D.p[3] = m;
        D.flags = std::isinf(m) ? 0u : kInfoTruncated;
        if (k == 2.0) {
            D.kind = kGammaErlang2;
        } else if (k == 0.5) {
            D.kind = kGammaHalf;
        } else {
            const double kp = k < 1.0 ? k + 1.0 : k;
            D.kind = kGammaMT;
            D.flags |= k < 1.0 ? kInfoBoost : 0u;
            D.p[1] = kp - 1.0 / 3.0;
            D.p[2] = 1.0 / std::sqrt(9.0 * D.p[1]);
            D.p[4] = 1.0 / k;
        }
    } else {
        if (p_pow < kMinAcceptance) return fail(MCDP_E_INVALID, "gamma max_scale truncation too severe to sample");
        D.kind = kGammaPow;
        D.flags = kInfoTruncated;
        D.p[0] = th;
        D.p[1] = mp;
        D.p[2] = 1.0 / k;
        D.p[3] = m;
    }
    return MCDP_OK;
}

int compile_empirical(const DistSpec &s, DistRec &D, std::vector<AliasRec> &table) {
    const size_t n = s.values.size();
    const bool abs = s.kind == kApiEmpAbs;
    if (n == 0) return fail(MCDP_E_INVALID, "empirical distribution needs at least one value");
    if (n == 1) {  // libstdc++ discrete_distribution with < 2 weights always yields 0
        D.kind = abs ? kEmpiricalAbs1 : kEmpiricalRel1;
        D.p[0] = s.values[0];
        return MCDP_OK;
    }
    double sum;
    if (!all_finite_nonneg(s.weights, sum))
        return fail(MCDP_E_INVALID, "empirical weights must be finite, non-negative and not all zero");
    if (n > (size_t)std::numeric_limits<int32_t>::max() / 2) return fail(MCDP_E_INVALID, "empirical table too large");
    std::vector<double> prob;
    std::vector<int> alias;
    build_alias(s.weights, prob, alias);
    if (table.size() + n > (size_t)std::numeric_limits<int32_t>::max()) return fail(MCDP_E_INVALID, "empirical tables too large");
    D.kind = abs ? kEmpiricalAbs : kEmpiricalRel;
    // p0 carries (n, first alias record) as two uint32 (low, high).
    const uint64_t packed = (uint64_t)(uint32_t)n | ((uint64_t)(uint32_t)table.size() << 32);
    std::memcpy(&D.p[0], &packed, sizeof(double));
    for (size_t i = 0; i < n; ++i) table.push_back(AliasRec{prob[i], s.values[i], s.values[(size_t)alias[i]], 0.0});
    return MCDP_OK;
}

int compile_dist(const DistSpec &s, DistRec &D, std::vector<AliasRec> &table) {
    D = DistRec{};
    D.kind = kNone;
    switch (s.kind) {
        case kApiConstant:
            D.kind = kConstant;
            D.p[0] = s.a;
            return MCDP_OK;
        case kApiExponential: return compile_exponential(s.a, s.b, D);
        case kApiGamma: return compile_gamma(s.a, s.b, s.c, D);
        default: return compile_empirical(s, D, table);
    }
}

// Relative cost of one draw (VALU instructions, measured per method), for
// balancing waves within a step.
int draw_cost(const DistRec *D) {
    if (!D) return 2;
    switch (D->kind) {
        case kConstant:
        case kEmpiricalAbs1:
        case kEmpiricalRel1: return 5;
        case kEmpiricalAbs:
        case kEmpiricalRel: return 45;
        case kExpInf: return 75;
        case kExpTrunc: return 80;
        case kGammaErlang2: return (D->flags & kInfoTruncated) ? 160 : 110;
        case kGammaHalf: return (D->flags & kInfoTruncated) ? 180 : 130;
        default: return 250;
    }
}
constexpr int kPredCost = 20;   // propagation work per predecessor record
constexpr int kEventCost = 15;  // per event: header, final cap, stores
// A wide step's launch gap and predecessor loads, in the same units
// (calibrated on the network workload: a 200-step tail run alone costs about
// 12 ns per unit either way).
constexpr int kWideStepCost = 300;
// Wide steps for a partial round of at most this many groups of 64 samples
// (each step launches events x groups single-wave workgroups; up to 128
// groups they were measured to end inside the tiles' time on the network and
// the small workloads).
constexpr int64_t kWideMaxGroups = 128;
// The same where one-sample tiles, whose time does not depend on the number of
// groups, are the better alternative above this many: in sampled runs, unless
// the wide steps cost less than half the tiles or a quarter of the predecessors
// come from global memory in tiles, which makes those dearer.  Measured with
// 8,192 samples, wide steps and one-sample tiles: 200 x 100 events 2.33 and 2.07
// ms (64 groups 1.7); 40 x 60 events of 40 predecessors 1.61 and 2.72; 60 x 250,
// 37% of the predecessors spilled, 2.34 and 2.99; injected durations, whose tiles
// are bound by each event's loads: 200 x 100 1.73 and 2.60, 40 x 60 1.06 and 3.29.
constexpr int64_t kWideMaxGroupsHalved = 96;

size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

}  // namespace

struct mcdp_generator {
    std::map<int32_t, DistSpec> dists;  // last add_* per type wins
};


namespace {

constexpr size_t kLdsBudgetBytes = 64 * 1024;  // LDS per workgroup for predecessor slots (one sample per lane)
// Sample indices and leading dimensions are 32-bit in the kernel; tiles of up
// to 128 samples must not overflow them.
constexpr int64_t kMaxSamplesPerLaunch = ((int64_t)1 << 31) - 256;
// The two-pass route of short runs is considered up to this many samples
// (a round of tiles is 32,768 on 256 CUs).
constexpr int64_t kLevelMaxSamples = (int64_t)1 << 17;

// A predecessor record for edge l: its minimal duration, sampling kind and p0
// inline; the distribution index for the kinds that read more parameters.
Record edge_record(const mcdp_propagator &P, int32_t l) {
    Record r{};
    r.i2 = l;
    if (l >= 0 && l < P.L) {
        r.a = P.dmin[(size_t)l];
        r.info = kInfoEdgeValid;
        const uint32_t di = P.ldist[(size_t)l];
        if (di == kNoDistIndex) {
            r.info |= kNone;
        } else {
            const DistRec &D = P.dist[di];
            r.info |= D.kind | D.flags | (di << kInfoDistShift);
            r.b = D.p[0];
        }
    } else {
        r.info = kNone;  // undefined in the reference: contributes 0.0
    }
    return r;
}

// Relative cost of evaluating event e for one wave.
int event_cost(const mcdp_propagator &P, int32_t e) {
    int c = kEventCost;
    for (int64_t k = P.pred_off[(size_t)e]; k < P.pred_off[(size_t)e + 1]; ++k) {
        const int32_t l = P.preds[(size_t)k].edge;
        const DistRec *D =
            (l >= 0 && l < P.L && P.ldist[(size_t)l] != kNoDistIndex) ? &P.dist[P.ldist[(size_t)l]] : nullptr;
        c += kPredCost + draw_cost(D);
    }
    return c;
}

// Steps, wave assignment, LDS slots and record streams for W waves per
// workgroup and at most K events per wave and step.
int build_schedule(mcdp_propagator &P, int32_t W, int32_t K) {
    const int32_t E = P.E, L = P.L;
    P.waves = W;
    P.k = K;
    P.step_off.assign(1, 0);
    P.ev_off.assign(1, 0);
    P.slot_list.clear();
    P.ev_rec.clear();
    P.recs.clear();
    P.orph.clear();
    P.max_per_wave = 0;
    P.n_global = 0;
    P.tile_cost = 0;
    P.wide_cost = 0;

    // (a) steps: each level in as few steps as W x K events allow, split evenly;
    // within a step, events go to the least-loaded wave (longest first).
    std::vector<int32_t> ev_step((size_t)E, -1);
    std::vector<int32_t> flat_events;  // stream order
    int32_t step = 0;
    for (const auto &lev : P.levels) {
        if (lev.empty()) continue;
        const size_t cap = (size_t)W * (size_t)K;
        const size_t nsteps = (lev.size() + cap - 1) / cap;
        for (size_t c = 0; c < nsteps; ++c) {
            const size_t c0 = lev.size() * c / nsteps, c1 = lev.size() * (c + 1) / nsteps;
            std::vector<std::pair<int, int32_t>> items;
            for (size_t i = c0; i < c1; ++i) items.emplace_back(event_cost(P, lev[i]), lev[i]);
            std::stable_sort(items.begin(), items.end(), [](auto &a, auto &b) { return a.first > b.first; });
            std::vector<std::vector<int32_t>> per((size_t)W);
            std::vector<int64_t> load((size_t)W, 0);
            for (auto &it : items) {
                int best = -1;
                for (int w = 0; w < W; ++w)
                    if ((int)per[(size_t)w].size() < K && (best < 0 || load[(size_t)w] < load[(size_t)best])) best = w;
                per[(size_t)best].push_back(it.second);
                load[(size_t)best] += it.first;
            }
            for (int w = 0; w < W; ++w) {
                for (int32_t e : per[(size_t)w]) {
                    flat_events.push_back(e);
                    ev_step[(size_t)e] = step;
                }
                P.max_per_wave = std::max<int32_t>(P.max_per_wave, (int32_t)per[(size_t)w].size());
                P.ev_off.push_back((int32_t)flat_events.size());
            }
            ++step;
        }
    }
    P.n_steps = step;

    // (b) LDS slots: an event read by a later step occupies a slot from the
    // commit of its step to the end of the last step that reads it.
    std::vector<int32_t> last_use((size_t)E, -1);
    for (int32_t e = 0; e < E; ++e)
        for (int64_t k = P.pred_off[(size_t)e]; k < P.pred_off[(size_t)e + 1]; ++k) {
            const PredEntry &pe = P.preds[(size_t)k];
            if (!pe.stale) last_use[(size_t)pe.src] = std::max(last_use[(size_t)pe.src], ev_step[(size_t)e]);
        }
    const int32_t slot_cap = (int32_t)(kLdsBudgetBytes / (kLanes * sizeof(double)));
    std::vector<int32_t> slot_of((size_t)E, -1);
    {
        std::vector<std::vector<int32_t>> release((size_t)std::max(P.n_steps, 1));
        std::vector<int32_t> free_slots;
        int32_t used = 0;
        for (int32_t t = 0; t < P.n_steps; ++t) {
            for (int32_t e : release[(size_t)t]) free_slots.push_back(slot_of[(size_t)e]);
            const int32_t b = P.ev_off[(size_t)t * W], en = P.ev_off[(size_t)(t + 1) * W];
            for (int32_t i = b; i < en; ++i) {
                const int32_t e = flat_events[(size_t)i];
                if (last_use[(size_t)e] < 0) continue;
                int32_t s = -1;
                if (!free_slots.empty()) {
                    s = free_slots.back();
                    free_slots.pop_back();
                } else if (used < slot_cap) {
                    s = used++;
                }
                slot_of[(size_t)e] = s;
                if (s >= 0) release[(size_t)last_use[(size_t)e]].push_back(e);
            }
        }
        P.slots = used;
    }

    // (c) record streams: for each (step, wave), each event's header then its
    // predecessors in input order.  The first predecessor record of an edge
    // writes its duration row.
    std::vector<uint8_t> referenced((size_t)L, 0);
    P.recs.reserve(flat_events.size() + P.preds.size() + 1);
    P.step_off.assign(1, 0);
    for (size_t g = 0; g + 1 < P.ev_off.size(); ++g) {
        for (int32_t i = P.ev_off[g]; i < P.ev_off[g + 1]; ++i) {
            const int32_t e = flat_events[(size_t)i];
            P.slot_list.push_back(slot_of[(size_t)e]);
            Record h{};
            h.a = P.earliest[(size_t)e];
            h.b = P.earliest[(size_t)e] + P.max_delay;
            h.i0 = e;
            h.i1 = slot_of[(size_t)e];
            h.i2 = (int32_t)(P.pred_off[(size_t)e + 1] - P.pred_off[(size_t)e]);
            h.info = kInfoHeader | (h.i2 == 0 ? kInfoLast : 0u);
            P.ev_rec.push_back((int32_t)P.recs.size());
            P.recs.push_back(h);
            for (int64_t k = P.pred_off[(size_t)e]; k < P.pred_off[(size_t)e + 1]; ++k) {
                const PredEntry &pe = P.preds[(size_t)k];
                Record r = edge_record(P, pe.edge);
                r.i0 = pe.src;
                if (pe.stale) {
                    r.i1 = kSrcStale;
                } else {
                    r.i1 = slot_of[(size_t)pe.src] >= 0 ? slot_of[(size_t)pe.src] : kSrcGlobal;
                    if (r.i1 == kSrcGlobal) ++P.n_global;
                }
                if (pe.edge >= 0 && pe.edge < L && !referenced[(size_t)pe.edge]) {
                    referenced[(size_t)pe.edge] = 1;
                    r.info |= kInfoOwner;
                }
                if (k + 1 == P.pred_off[(size_t)e + 1]) r.info |= kInfoLast;
                P.recs.push_back(r);
            }
        }
        P.step_off.push_back((int32_t)P.recs.size());
    }
    // padding: the walk kernel prefetches one record ahead, a wide step loads
    // kWideBatch predecessor records at a time
    for (int i = 0; i < kWideBatch; ++i) P.recs.push_back(Record{});
    if (P.recs.size() > (size_t)std::numeric_limits<int32_t>::max()) return fail(MCDP_E_INVALID, "plan too large");
    for (int32_t t = 0; t < P.n_steps; ++t) {
        int64_t busiest = 0, costliest = 0;
        for (int32_t w = 0; w < W; ++w) {
            int64_t c = 0;
            for (int32_t i = P.ev_off[(size_t)t * W + w]; i < P.ev_off[(size_t)t * W + w + 1]; ++i) {
                const int64_t ce = event_cost(P, flat_events[(size_t)i]);
                c += ce;
                costliest = std::max(costliest, ce);
            }
            busiest = std::max(busiest, c);
        }
        P.tile_cost += busiest;
        P.wide_cost += kWideStepCost + costliest;
    }
    for (int32_t l = 0; l < L; ++l)
        if (!referenced[(size_t)l]) P.orph.push_back(edge_record(P, l));
    return MCDP_OK;
}

// Threads of a level_kernel workgroup of `group` samples for a widest level of
// `width` events.
int level_threads(int32_t width, int group) {
    const int64_t want = (int64_t)width * group;
    return (int)std::min<int64_t>((want + kLanes - 1) / kLanes * kLanes, kLevelMaxThreads);
}

// Microseconds of a level in level_kernel (see two_pass_us): a pass of the
// workgroup over its items, each of its waves, and in a level with predecessors
// past the items' inline ones these, one after another.
constexpr double kLevelPassUs = 0.40, kLevelWaveUs = 0.045, kLevelExtraUs = 0.5, kLevelExtraEachUs = 0.20;

// LDS slots of the two-pass route: an event that a later level reads has one
// from its own level to the last that reads it.  level_kernel writes a level's
// results while other waves may still read for that level, so a slot is given
// out again from the level after its last read.  Done once, when a run first
// asks for its route.
void build_level_slots(mcdp_propagator &P) {
    if (P.level_ready) return;
    P.level_ready = true;
    const int32_t n_levels = (int32_t)P.levels.size();
    std::vector<int32_t> level((size_t)P.E, 0), last_use((size_t)P.E, -1);
    P.level_width = 0;
    P.walk_cost = P.move_cost = P.level_extra = P.draw_sum = 0;
    std::vector<int64_t> extra((size_t)n_levels, 0);  // the most of an event of the level
    for (int32_t t = 0; t < n_levels; ++t) {
        P.level_width = std::max<int32_t>(P.level_width, (int32_t)P.levels[(size_t)t].size());
        int64_t sum = 0, costliest = 0, moves = 0, most = 0;
        for (int32_t e : P.levels[(size_t)t]) {
            level[(size_t)e] = t;
            const int64_t c = event_cost(P, e);
            sum += c;
            costliest = std::max(costliest, c);
            const int64_t preds = P.pred_off[(size_t)e + 1] - P.pred_off[(size_t)e];
            const int64_t m = kEventCost + kPredCost * preds;
            moves += m;
            most = std::max(most, m);
            extra[(size_t)t] = std::max(extra[(size_t)t], preds - kLevelPreds);
        }
        P.draw_sum += sum - moves;
        P.walk_cost += std::max(costliest, (sum + kMaxWaves - 1) / kMaxWaves);
        P.move_cost += std::max(most, (moves + kMaxWaves - 1) / kMaxWaves);
        P.level_extra += extra[(size_t)t];
    }
    for (int g = 0; g < 7; ++g) {
        const int threads = level_threads(P.level_width, 1 << g);
        const int64_t items = threads >> g;  // of one pass
        P.level_us[g] = 0.0;
        for (int32_t t = 0; t < n_levels; ++t) {
            const int64_t passes = ((int64_t)P.levels[(size_t)t].size() + items - 1) / items, x = extra[(size_t)t];
            P.level_us[g] += (double)passes * (kLevelPassUs + kLevelWaveUs * (threads / kLanes) +
                                               (x > 0 ? kLevelExtraUs + kLevelExtraEachUs * (double)x : 0.0));
        }
    }
    for (int32_t e = 0; e < P.E; ++e)
        for (int64_t k = P.pred_off[(size_t)e]; k < P.pred_off[(size_t)e + 1]; ++k) {
            const PredEntry &pe = P.preds[(size_t)k];
            if (!pe.stale) last_use[(size_t)pe.src] = std::max(last_use[(size_t)pe.src], level[(size_t)e]);
        }
    P.level_slot.assign((size_t)P.E, -1);
    std::vector<std::vector<int32_t>> release((size_t)n_levels + 1);
    std::vector<int32_t> free_slots;
    // slot 0 holds NaN; each event that is read stale has one for its earliest time
    int32_t used = 1;
    P.level_stale.clear();
    P.level_zero_edges = false;
    for (const PredEntry &pe : P.preds) {
        if (pe.stale) P.level_stale.emplace_back(pe.src, 0);
        P.level_zero_edges |= pe.edge < 0 || pe.edge >= P.L;
    }
    std::sort(P.level_stale.begin(), P.level_stale.end());
    P.level_stale.erase(std::unique(P.level_stale.begin(), P.level_stale.end()), P.level_stale.end());
    for (auto &st : P.level_stale) st.second = used++;
    for (int32_t t = 0; t < n_levels; ++t) {
        for (int32_t slot : release[(size_t)t]) free_slots.push_back(slot);
        for (int32_t e : P.levels[(size_t)t]) {
            if (last_use[(size_t)e] < 0) continue;
            int32_t slot;
            if (free_slots.empty()) {
                slot = used++;
            } else {
                slot = free_slots.back();
                free_slots.pop_back();
            }
            P.level_slot[(size_t)e] = slot;
            release[(size_t)last_use[(size_t)e] + 1].push_back(slot);
        }
    }
    P.level_slots = used;
    // the plan packs slots and predecessor counts into 15 and 16 bits
    if (used > 0x7FFF || max_entries(P) > 0xFFFF) P.level_slots = std::numeric_limits<int32_t>::max();
}

// Default (waves, events per wave) for a DAG: enough waves to spread the widest
// level (up to 8), and the smallest compiled bound that holds it in one step.
void default_shape(const mcdp_propagator &P, int32_t &W, int32_t &K) {
    size_t max_width = 0;
    for (const auto &v : P.levels) max_width = std::max(max_width, v.size());
    W = 1;
    while (W < 8 && (size_t)W * 4 < max_width) W *= 2;
    K = kMaxEventsPerWave;
    for (int k : kEventsPerWaveChoices)
        if ((size_t)k * (size_t)W >= max_width) {
            K = k;
            break;
        }
}

int compile_propagator(mcdp_propagator &P, int32_t n_events, const double *earliest, int32_t n_acts,
                       const int32_t *act_idx, const double *act_dur, const int32_t *act_type, int32_t n_entries,
                       const int32_t *entry_target, const int64_t *entry_off, const int32_t *pred_event,
                       const int32_t *pred_act, double max_delay, const mcdp_generator &gen) {
    // (1) validation, in the reference's order.
    if (gen.dists.count(-1)) return fail(MCDP_E_RESERVED_TYPE, "Activity type -1 is reserved for no delay");
    if (max_delay < 0.0) return fail(MCDP_E_MAX_DELAY, "max_delay must be non-negative");
    if (n_events < 0 || n_acts < 0 || n_entries < 0) return fail(MCDP_E_INVALID, "negative count");
    const int32_t E = n_events;
    P.max_delay = max_delay;

    // (2) distributions.
    std::map<int32_t, int32_t> type_to_dist;
    for (const auto &kv : gen.dists) {
        DistRec D;
        int rc = compile_dist(kv.second, D, P.alias);
        if (rc) return fail(rc, g_last_error + " (activity_type " + std::to_string(kv.first) + ")");
        type_to_dist[kv.first] = (int32_t)P.dist.size();
        P.dist.push_back(D);
    }
    if (P.dist.size() > (size_t)kInfoDistMask) return fail(MCDP_E_INVALID, "too many distributions");

    // (3) link table.
    int64_t max_idx = -1;
    for (int32_t i = 0; i < n_acts; ++i) {
        if (act_idx[i] < 0) return fail(MCDP_E_INVALID, "activity index must be non-negative");
        max_idx = std::max<int64_t>(max_idx, act_idx[i]);
    }
    const int32_t L = (int32_t)(max_idx + 1);
    P.dmin.assign((size_t)L, 0.0);
    std::vector<int32_t> ltype((size_t)L, -1);
    std::vector<uint8_t> seen((size_t)L, 0);
    for (int32_t i = 0; i < n_acts; ++i) {
        const int32_t l = act_idx[i];
        if (seen[(size_t)l] &&
            (std::memcmp(&P.dmin[(size_t)l], &act_dur[i], sizeof(double)) != 0 || ltype[(size_t)l] != act_type[i]))
            return fail(MCDP_E_INVALID, "two activities share index " + std::to_string(l) + " with different attributes");
        seen[(size_t)l] = 1;
        P.dmin[(size_t)l] = act_dur[i];
        ltype[(size_t)l] = act_type[i];
    }
    P.ldist.assign((size_t)L, kNoDistIndex);
    for (int32_t l = 0; l < L; ++l) {
        auto it = type_to_dist.find(ltype[(size_t)l]);
        if (it != type_to_dist.end()) P.ldist[(size_t)l] = (uint32_t)it->second;
    }

    // (4) topology.
    if (n_entries > 0 && entry_off[0] != 0) return fail(MCDP_E_INVALID, "entry_offsets[0] must be 0");
    for (int32_t i = 0; i < n_entries; ++i) {
        if (entry_off[i + 1] < entry_off[i]) return fail(MCDP_E_INVALID, "entry_offsets must be non-decreasing");
        if (entry_target[i] < 0 || entry_target[i] >= E) return fail(MCDP_E_INVALID, "precedence target out of range");
        for (int64_t k = entry_off[i]; k < entry_off[i + 1]; ++k)
            if (pred_event[k] < 0 || pred_event[k] >= E) return fail(MCDP_E_INVALID, "predecessor event out of range");
    }
    std::vector<int32_t> win((size_t)E, -1), indeg((size_t)E, 0);
    std::vector<int64_t> adj_off((size_t)E + 1, 0);
    for (int32_t i = 0; i < n_entries; ++i) {
        win[(size_t)entry_target[i]] = i;
        indeg[(size_t)entry_target[i]] = (int32_t)(entry_off[i + 1] - entry_off[i]);
        for (int64_t k = entry_off[i]; k < entry_off[i + 1]; ++k) adj_off[(size_t)pred_event[k] + 1]++;
    }
    for (int32_t i = 0; i < E; ++i) adj_off[(size_t)i + 1] += adj_off[(size_t)i];
    std::vector<int32_t> adj((size_t)adj_off[(size_t)E]);
    {
        std::vector<int64_t> fill(adj_off.begin(), adj_off.end() - 1);
        for (int32_t i = 0; i < n_entries; ++i)
            for (int64_t k = entry_off[i]; k < entry_off[i + 1]; ++k)
                adj[(size_t)fill[(size_t)pred_event[k]]++] = entry_target[i];
    }
    std::vector<int32_t> order;
    order.reserve((size_t)E);
    {
        std::vector<int32_t> q;
        q.reserve((size_t)E);
        for (int32_t i = 0; i < E; ++i)
            if (indeg[(size_t)i] == 0) q.push_back(i);
        size_t head = 0;
        while (head < q.size()) {
            const int32_t n = q[head++];
            order.push_back(n);
            for (int64_t k = adj_off[(size_t)n]; k < adj_off[(size_t)n + 1]; ++k)
                if (--indeg[(size_t)adj[(size_t)k]] == 0) q.push_back(adj[(size_t)k]);
        }
    }
    if ((int32_t)order.size() != E) return fail(MCDP_E_CYCLE, "Invalid DAG: cycle detected in precedence list");

    // (5) predecessor lists and levels.  A predecessor evaluated after its
    // consumer in the reference's order is read before it is written there,
    // i.e. at its earliest time ("stale"); every other predecessor is a true
    // dependency.
    std::vector<int32_t> pos((size_t)E), level((size_t)E, 0);
    for (int32_t i = 0; i < E; ++i) pos[(size_t)order[(size_t)i]] = i;
    P.pred_off.assign((size_t)E + 1, 0);
    for (int32_t e = 0; e < E; ++e) {
        const int32_t w = win[(size_t)e];
        P.pred_off[(size_t)e + 1] = P.pred_off[(size_t)e] + (w >= 0 ? entry_off[w + 1] - entry_off[w] : 0);
    }
    P.preds.resize((size_t)P.pred_off[(size_t)E]);
    for (int32_t e = 0; e < E; ++e) {
        const int32_t w = win[(size_t)e];
        if (w < 0) continue;
        int64_t o = P.pred_off[(size_t)e];
        for (int64_t k = entry_off[w]; k < entry_off[w + 1]; ++k, ++o) {
            const int32_t s = pred_event[k];
            const bool stale = pos[(size_t)s] >= pos[(size_t)e];
            P.preds[(size_t)o] = PredEntry{s, pred_act[k], stale};
            if (stale) ++P.n_stale;
        }
    }
    int32_t n_levels = E > 0 ? 1 : 0;
    for (int32_t e : order) {
        int32_t lv = 0;
        for (int64_t k = P.pred_off[(size_t)e]; k < P.pred_off[(size_t)e + 1]; ++k)
            if (!P.preds[(size_t)k].stale) lv = std::max(lv, level[(size_t)P.preds[(size_t)k].src] + 1);
        level[(size_t)e] = lv;
        n_levels = std::max(n_levels, lv + 1);
    }
    P.levels.assign((size_t)n_levels, {});
    for (int32_t e : order) P.levels[(size_t)level[(size_t)e]].push_back(e);

    P.E = E;
    P.L = L;
    P.earliest.assign(earliest, earliest + E);

    // (6) default schedule.
    int32_t W, K;
    default_shape(P, W, K);
    return build_schedule(P, W, K);
}

// The two-pass route's plan with P's current times: every event in level
// order with its predecessors, and a record per link, costliest laws first
// (waves of draw_kernel take them in turn, so the last ones are short).
struct LevelPlan {
    std::vector<int32_t> off, extra_of;
    std::vector<LevelQuad> quad;
    std::vector<LevelPred> extra;
    std::vector<LevelInit> init;
    std::vector<Record> draws;
};
LevelPlan level_plan(const mcdp_propagator &P) {
    LevelPlan lv;
    const size_t E = (size_t)P.E;
    lv.init.push_back(LevelInit{std::numeric_limits<double>::quiet_NaN(), 0, 0});
    for (const auto &st : P.level_stale) lv.init.push_back(LevelInit{P.earliest[(size_t)st.first], st.second, 0});
    auto entry = [&](const PredEntry &pe) {
        LevelPred pr{0, pe.edge >= 0 && pe.edge < P.L ? pe.edge : -1, pe.src};
        pr.slot = !pe.stale ? P.level_slot[(size_t)pe.src]
                            : std::lower_bound(P.level_stale.begin(), P.level_stale.end(), std::make_pair(pe.src, 0))->second;
        return pr;
    };
    auto pair16 = [](int32_t lo, int32_t hi) { return (int32_t)((uint32_t)(lo & 0xFFFF) | (uint32_t)hi << 16); };
    lv.quad.resize(E * kLevelQuads);
    lv.extra_of.assign(E, 0);
    lv.off.assign(1, 0);
    size_t q = 0;
    for (const auto &level : P.levels) {
        for (int32_t e : level) {
            const int64_t p0 = P.pred_off[(size_t)e], p1 = P.pred_off[(size_t)e + 1];
            const double times[2] = {P.earliest[(size_t)e], P.earliest[(size_t)e] + P.max_delay};
            std::memcpy(&lv.quad[q], times, sizeof(times));
            LevelPred pr[kLevelPreds];
            for (int k = 0; k < kLevelPreds; ++k)
                pr[k] = p0 + k < p1 ? entry(P.preds[(size_t)(p0 + k)]) : LevelPred{0, k ? pr[0].edge : 0, -1};
            lv.extra_of[(size_t)e] = (int32_t)lv.extra.size();
            for (int64_t k = p0 + kLevelPreds; k < p1; ++k) lv.extra.push_back(entry(P.preds[(size_t)k]));
            lv.quad[E + q] = LevelQuad{{e, pair16(P.level_slot[(size_t)e], (int32_t)(p1 - p0)),
                                        pair16(pr[0].slot, pr[1].slot), pair16(pr[2].slot, pr[3].slot)}};
            lv.quad[2 * E + q] = LevelQuad{{pr[0].edge, pr[1].edge, pr[2].edge, pr[3].edge}};
            lv.quad[3 * E + q] = LevelQuad{{pr[0].src, pr[1].src, pr[2].src, pr[3].src}};
            ++q;
        }
        lv.off.push_back((int32_t)q);
    }
    lv.off.push_back((int32_t)q);
    std::vector<std::pair<int, int32_t>> order((size_t)P.L);
    for (int32_t l = 0; l < P.L; ++l) {
        const uint32_t di = P.ldist[(size_t)l];
        // by cost, equal costs by law: a wave's links then mostly share theirs
        const int cost = di == kNoDistIndex ? draw_cost(nullptr) : draw_cost(&P.dist[di]);
        order[(size_t)l] = {-(cost * 64 + (di == kNoDistIndex ? 0 : (int)(P.dist[di].kind & 63))), l};
    }
    std::stable_sort(order.begin(), order.end(), [](auto &a, auto &b) { return a.first < b.first; });
    lv.draws.reserve((size_t)P.L);
    for (auto &o : order) lv.draws.push_back(edge_record(P, o.second));
    return lv;
}

// P's entry for the current device.
int device_entry_impl(mcdp_propagator &P, DeviceCopy *&out) {
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0)
        return fail(MCDP_E_DEVICE, "no HIP device available: the Monte Carlo engine runs on the GPU only");
    int device = 0;
    HIP_TRY(hipGetDevice(&device), "hipGetDevice");
    out = nullptr;
    for (auto &d : P.dev)
        if (d.device == device) out = &d;
    if (!out) {
        P.dev.push_back(DeviceCopy{});
        out = &P.dev.back();
        out->device = device;
    }
    return MCDP_OK;
}

// While one of these lives, its thread may allocate and upload although a
// stream is being captured (the default capture mode forbids that to every
// thread).  A propagator's plans are uploaded when a run first takes a route
// that needs them, so a caller that ran it once, whatever the route, may
// capture any run that follows.
class DuringCapture {
   public:
    explicit DuringCapture(bool allowed)
        : allowed_(allowed && hipThreadExchangeStreamCaptureMode(&mode_) == hipSuccess) {}
    ~DuringCapture() {
        if (allowed_) (void)hipThreadExchangeStreamCaptureMode(&mode_);
    }
    DuringCapture(const DuringCapture &) = delete;
    DuringCapture &operator=(const DuringCapture &) = delete;

   private:
    hipStreamCaptureMode mode_ = hipStreamCaptureModeRelaxed;
    bool allowed_;
};
// Whether a run or a statistics call has used the propagator on d's device.
bool in_use(const DeviceCopy &d) { return d.blob || d.level_blob || d.topo || d.rev; }

// The side stream of d's device and its events (made once).
int ensure_side(DeviceCopy &d) {
    hipError_t e = hipSuccess;
    if (!d.side) e = hipStreamCreateWithFlags(&d.side, hipStreamNonBlocking);
    if (e == hipSuccess && !d.fork) e = hipEventCreateWithFlags(&d.fork, hipEventDisableTiming);
    if (e == hipSuccess && !d.join) e = hipEventCreateWithFlags(&d.join, hipEventDisableTiming);
    return e == hipSuccess ? MCDP_OK : hip_fail(e, "side stream");
}

// A device allocation holding `bytes` of `host`.  For a device in use (see
// DuringCapture) the copy goes through the side stream, which no capture
// waits for.
int upload(DeviceCopy &d, const void *host, size_t bytes, void *&blob) {
    const bool used = in_use(d);
    const DuringCapture allow(used);
    int rc = used ? ensure_side(d) : MCDP_OK;
    if (rc) return rc;
    void *p = nullptr;
    hipError_t e = device_malloc(&p, std::max<size_t>(bytes, 256));
    if (e != hipSuccess) return fail(MCDP_E_NOMEM, std::string("hipMalloc (plan): ") + hipGetErrorString(e));
    if (used) {
        e = hipMemcpyAsync(p, host, bytes, hipMemcpyHostToDevice, d.side);
        if (e == hipSuccess) e = hipStreamSynchronize(d.side);
    } else {
        e = hipMemcpy(p, host, bytes, hipMemcpyHostToDevice);
    }
    if (e != hipSuccess) {
        (void)hipFree(p);
        return hip_fail(e, "hipMemcpy (plan)");
    }
    blob = p;
    return MCDP_OK;
}

// Parts of one device allocation.
class Upload {
   public:
    template <typename T>
    size_t add(const std::vector<T> &v) {
        const size_t o = host_.size();
        host_.resize(o + align_up(std::max<size_t>(v.size() * sizeof(T), 1), 256));
        if (!v.empty()) std::memcpy(host_.data() + o, v.data(), v.size() * sizeof(T));
        return o;
    }
    int send(DeviceCopy &d, void *&blob) { return upload(d, host_.data(), host_.size(), blob); }

   private:
    std::vector<unsigned char> host_;
};
template <typename T>
const T *part(const void *blob, size_t offset) {
    return reinterpret_cast<const T *>(static_cast<const unsigned char *>(blob) + offset);
}

// Uploads the two-pass route's plan to d's device (once).
int ensure_levels(const mcdp_propagator &P, DeviceCopy &d) {
    if (d.level_blob) return MCDP_OK;
    const LevelPlan lv = level_plan(P);
    Upload up;
    const size_t o_off = up.add(lv.off), o_quad = up.add(lv.quad), o_xof = up.add(lv.extra_of), o_init = up.add(lv.init),
                 o_extra = up.add(lv.extra), o_draws = up.add(lv.draws), o_dist = up.add(P.dist),
                 o_alias = up.add(P.alias);
    const int rc = up.send(d, d.level_blob);
    if (rc) return rc;
    const void *b = d.level_blob;
    d.levels.off = part<int32_t>(b, o_off);
    d.levels.quad = part<LevelQuad>(b, o_quad);
    d.levels.extra_of = part<int32_t>(b, o_xof);
    d.levels.init = part<LevelInit>(b, o_init);
    d.levels.n_init = (int32_t)lv.init.size();
    d.levels.extra = part<LevelPred>(b, o_extra);
    d.levels.E = P.E;
    d.levels.n_levels = (int32_t)P.levels.size();
    d.draws.recs = part<Record>(b, o_draws);
    d.draws.dists = part<DistParams>(b, o_dist);
    d.draws.alias = part<AliasRec>(b, o_alias);
    d.draws.n_alias = (int32_t)P.alias.size();
    d.draws.L = P.L;
    return MCDP_OK;
}

// Uploads the walk's plan of `P` to the current device (once per device).
int ensure_device_impl(mcdp_propagator &P, DeviceCopy *&out) {
    const int rc = device_entry_impl(P, out);
    if (rc || out->blob) return rc;
    DeviceCopy &d = *out;
    const size_t a = 256;
    size_t off = 0;
    auto reserve = [&](size_t bytes) {
        const size_t o = off;
        off = align_up(off + bytes, a);
        return o;
    };
    const size_t o_step = reserve(P.step_off.size() * sizeof(int32_t));
    const size_t o_recs = reserve(P.recs.size() * sizeof(Record));
    const size_t o_evoff = reserve(P.ev_off.size() * sizeof(int32_t));
    const size_t o_slots = reserve(P.slot_list.size() * sizeof(int32_t));
    // each (step, wave)'s slots as one row of k, -1 past its events
    std::vector<int32_t> step_slots((size_t)P.n_steps * P.waves * P.k, -1);
    for (size_t g = 0; g + 1 < P.ev_off.size(); ++g)
        for (int32_t i = P.ev_off[g]; i < P.ev_off[g + 1]; ++i)
            step_slots[g * (size_t)P.k + (size_t)(i - P.ev_off[g])] = P.slot_list[(size_t)i];
    const size_t o_sslots = reserve(step_slots.size() * sizeof(int32_t));
    const size_t o_orph = reserve(P.orph.size() * sizeof(Record));
    const size_t o_dist = reserve(P.dist.size() * sizeof(DistParams));
    const size_t o_alias = reserve(P.alias.size() * sizeof(AliasRec));
    const size_t o_earl = reserve(P.earliest.size() * sizeof(double));
    const size_t o_evrec = reserve(P.ev_rec.size() * sizeof(int32_t));
    const size_t total = std::max<size_t>(off, a);
    std::vector<unsigned char> host(total, 0);
    auto put = [&](size_t o, const void *src, size_t bytes) {
        if (bytes) std::memcpy(host.data() + o, src, bytes);
    };
    put(o_step, P.step_off.data(), P.step_off.size() * sizeof(int32_t));
    put(o_recs, P.recs.data(), P.recs.size() * sizeof(Record));
    put(o_evoff, P.ev_off.data(), P.ev_off.size() * sizeof(int32_t));
    put(o_slots, P.slot_list.data(), P.slot_list.size() * sizeof(int32_t));
    put(o_sslots, step_slots.data(), step_slots.size() * sizeof(int32_t));
    put(o_orph, P.orph.data(), P.orph.size() * sizeof(Record));
    put(o_dist, P.dist.data(), P.dist.size() * sizeof(DistParams));
    put(o_alias, P.alias.data(), P.alias.size() * sizeof(AliasRec));
    put(o_earl, P.earliest.data(), P.earliest.size() * sizeof(double));
    put(o_evrec, P.ev_rec.data(), P.ev_rec.size() * sizeof(int32_t));
    void *blob = nullptr;
    const int up = upload(d, host.data(), total, blob);
    if (up) return up;
    // the side stream of wide steps and its fork / join events, made here so
    // that a launch creates nothing (it may be under stream capture)
    const int side = ensure_side(d);
    if (side) {
        (void)hipFree(blob);
        return side;
    }
    d.blob = blob;
    auto *b = static_cast<unsigned char *>(blob);
    d.base.step_off = reinterpret_cast<const int32_t *>(b + o_step);
    d.base.recs = reinterpret_cast<const Record *>(b + o_recs);
    d.base.ev_off = reinterpret_cast<const int32_t *>(b + o_evoff);
    d.base.slot_list = reinterpret_cast<const int32_t *>(b + o_slots);
    d.base.step_slots = reinterpret_cast<const int32_t *>(b + o_sslots);
    d.base.orph = reinterpret_cast<const Record *>(b + o_orph);
    d.base.dists = reinterpret_cast<const DistParams *>(b + o_dist);
    d.base.alias = reinterpret_cast<const AliasRec *>(b + o_alias);
    d.base.earliest = reinterpret_cast<const double *>(b + o_earl);
    d.base.ev_rec = reinterpret_cast<const int32_t *>(b + o_evrec);
    d.base.n_steps = P.n_steps;
    d.base.n_orphans = (int32_t)P.orph.size();
    d.base.waves = P.waves;
    d.base.n_alias = (int32_t)P.alias.size();
    d.base.slots = P.slots;
    return MCDP_OK;
}
// The fast kernel variant needs every read predecessor in LDS (or stale), the
// alias tables small enough to stage in LDS, and no cap of -0 (which only a
// max_delay of -0 gives: its cap is a v_min_f64, where -0 is below +0).
WalkVariant walk_variant(const mcdp_propagator &P, bool injected) {
    const bool alias_fits = P.alias.size() * sizeof(AliasRec) <= kAliasLdsMaxBytes;
    const bool fast = P.n_global == 0 && (injected || alias_fits) && !std::signbit(P.max_delay);
    return WalkVariant{injected, fast ? kPathsFast : kPathsGeneral, P.k, P.spl};
}

size_t walk_lds_bytes(const mcdp_propagator &P, WalkVariant v) {
    size_t bytes = (size_t)P.slots * kLanes * (size_t)v.spl * sizeof(double);
    if (!v.injected && v.paths == kPathsFast) bytes += P.alias.size() * sizeof(AliasRec);
    return bytes;
}

// A schedule shape: waves per workgroup, events per wave and step, samples
// per lane.
struct Shape {
    int32_t waves, k, spl;
};

bool shape_valid(int32_t waves, int32_t k, int32_t spl) {
    if (waves < 1 || waves > kMaxWaves) return false;
    if (spl != 1 && spl != 2) return false;
    bool k_ok = false;
    for (int c : kEventsPerWaveChoices) k_ok |= c == k;
    return k_ok && (spl == 1 || k <= kMaxEventsPerWaveSpl2);
}

// Shapes worth trying: every valid shape whose step holds the widest level
// (or that is the largest shape available).
std::vector<Shape> shape_candidates(const mcdp_propagator &P) {
    size_t max_width = 1;
    for (const auto &v : P.levels) max_width = std::max(max_width, v.size());
    static const int32_t kWaveChoices[] = {1, 2, 4, 6, 8, 10, 12, 14, 16};
    std::vector<Shape> out;
    for (int spl : kSplChoices) {
        const int kmax = spl == 1 ? kMaxEventsPerWave : kMaxEventsPerWaveSpl2;
        const size_t need = std::min<size_t>(max_width, (size_t)kMaxWaves * (size_t)kmax);
        for (int k : kEventsPerWaveChoices)
            for (int32_t w : kWaveChoices)
                if (shape_valid(w, k, spl) && (size_t)w * (size_t)k >= need) out.push_back(Shape{w, k, spl});
    }
    return out;
}

// Picks a shape for the current device without running anything.  Among shapes
// of one number of samples per lane: the most workgroups resident per CU, then
// the least work on the busiest wave of each step (events, summed over steps),
// then more waves.  Of the two winners the one of two samples per lane, unless the
// other has more than one and a half times its work in flight (samples of the
// resident waves that a step gives an event to): a one-sample tile takes 0.72 of
// a two-sample tile's instructions.  Compared by samples resident, three workgroups of 8 waves x 12 events x 1 sample went before one of
// 16 x 8 x 2 for levels of 65 to 96 events: 75 x 80 events, network laws, 65,536
// samples 2.75 ms against 2.26, constants without durations 1.38 against 0.92,
// truncated laws 4.4 against 3.8 (131,072: 7.3 and 7.4); and six of 4 x 12 x 1 before
// two of 8 x 8 x 2 for 33 to 48: 150 x 40 events 2.54 against 2.27, truncated laws
// 4.05 against 3.74.  Candidate schedules are built on the host; P is left with the winner.
int choose_shape(mcdp_propagator &P) {
    struct Best {
        Shape shape{0, 0, 0};
        int bpc = 0;
        int64_t load = 0;
        double flight = 0.0;  // waves with an event, on average over the steps
    } best[2];
    Shape shape{P.waves, P.k, 1};
    for (const Shape &c : shape_candidates(P)) {
        int rc = build_schedule(P, c.waves, c.k);
        if (rc) return rc;
        P.spl = c.spl;
        const WalkVariant v = walk_variant(P, false);
        int bpc = 0;
        if (walk_occupancy(v, P.waves, walk_lds_bytes(P, v), &bpc) != hipSuccess || bpc < 1) continue;
        int64_t load = 0, busy = 0;
        for (int32_t t = 0; t < P.n_steps; ++t) {
            int32_t m = 0;
            for (int32_t w = 0; w < P.waves; ++w) {
                const int32_t events = P.ev_off[(size_t)t * P.waves + w + 1] - P.ev_off[(size_t)t * P.waves + w];
                m = std::max(m, events);
                busy += events > 0 ? 1 : 0;
            }
            load += m;
        }
        Best &b = best[c.spl - 1];
        if (bpc > b.bpc || (bpc == b.bpc && (load < b.load || (load == b.load && c.waves > b.shape.waves))))
            b = Best{c, bpc, load, (double)bpc * (double)busy / std::max(P.n_steps, 1)};
    }
    if (best[0].bpc > 0) shape = best[0].shape;
    if (best[1].bpc > 0 && best[0].flight <= 3.0 * best[1].flight) shape = best[1].shape;
    P.spl = shape.spl;
    return build_schedule(P, shape.waves, shape.k);
}

// Samples per workgroup of level_kernel for a run of n: the fewest that leave
// no more workgroups than CUs (a workgroup costs a level's latency whatever it
// carries, and a second one per CU waits for the first), within what LDS
// holds; 0 if the DAG keeps more realized times live than LDS holds for one
// sample.  Measured on the network DAG, propagation alone: 4,001 samples 0.77 ms
// at 16 a workgroup against 0.86 at 8 and 1.28 at 32; 1,000 samples 0.26 ms at 4
// against 0.38 at 2 and 0.34 at 8.
int level_group(const mcdp_propagator &P, int64_t n, int cus) {
    int group = 1;
    while (group < kLevelMaxGroup && (n + group - 1) / group > cus) group *= 2;
    while (group > 0 && (size_t)P.level_slots * (size_t)group * sizeof(double) > kLevelLdsMaxBytes) group /= 2;
    return group;
}

// Whether a walk of less than a round in one-sample tiles (see launch) takes
// them rather than wide steps above kWideMaxGroupsHalved groups.
bool tiles_early(const mcdp_propagator &P, bool injected) {
    return !injected && 2 * P.wide_cost >= P.tile_cost && 4 * P.n_global <= (int64_t)P.preds.size();
}

// Estimated microseconds of a walk of n samples, at most a round of tiles; one_sample:
// in tiles of one sample per lane (see launch).  Wide steps cost a launch gap
// and their draws or bytes.  A tile's time is its waves' instructions, draws at
// 4.1 ns a cost unit and the rest at 8.9 (three times that where predecessors
// come from global memory); with injected durations, which an event waits for,
// 24 ns a unit of the rest; and some of its bytes.  The plan's costs are those
// of the shape in use, or of 16 waves while no walk has chosen one.
double walk_us(const mcdp_propagator &P, bool injected, int64_t n, bool one_sample) {
    const double bytes = (double)n * (8.0 * (double)P.preds.size() + 12.0 * P.E);
    const int64_t groups = (n + kLanes - 1) / kLanes;
    if (groups <= (one_sample && tiles_early(P, injected) ? kWideMaxGroupsHalved : kWideMaxGroups) &&
        P.wide_cost < P.tile_cost)
        return injected ? 4.1 * P.n_steps + (bytes + (double)n * 8.0 * (double)P.preds.size()) / 10.2e6 + 0.16 * (double)P.level_extra
                        : 11.0 + 4.8 * P.n_steps + (double)n * (double)P.draw_sum * 0.047e-6 + 0.27 * (double)P.level_extra;
    const double shape = P.shape_fixed ? (double)P.tile_cost / (double)std::max<int64_t>(P.walk_cost, 1) : 1.0;
    const double moves = shape * (double)P.move_cost, draws = shape * (double)P.walk_cost - moves;
    const bool spilled = P.n_global > 0;
    const double tile = injected ? 0.0236 * moves * (spilled ? 1.24 : 1.0)
                                 : 0.0041 * draws + 0.0089 * moves * (spilled ? 3.05 : 1.0) + 0.12 * P.n_steps;
    return 11.0 + tile * (one_sample ? 1.0 : injected ? 1.09 : 1.36) + bytes / (injected ? 12.5e6 : 13.9e6);
}

// Estimated microseconds of the two passes.  The draws: their instructions on
// the device's waves or the longest chain of them on one, and the bytes they
// write.  The levels: their latency, for as many rounds of workgroups as there
// are, and the bytes they move, in pieces of a row as long as a workgroup's
// samples.
double two_pass_us(const mcdp_propagator &P, bool injected, int64_t n, int group, int cus) {
    double draws = 0.0;
    if (!injected) {
        // a wave takes 256 samples of a link, or those of a short run for several links
        int64_t samples = (n + 255) / 256 * 256, wave_links = (int64_t)P.L * (samples / 256);
        if (n < kLanes) {
            samples = 1;
            while (samples < n) samples *= 2;
            wave_links = ((int64_t)P.L * samples + kLanes - 1) / kLanes;
        }
        const int64_t waves = (int64_t)cus * 24;
        const double chain = (double)((wave_links + waves - 1) / waves) * (double)P.draw_sum / std::max(P.L, 1) * 0.038;
        const double issue = (double)samples * (double)P.draw_sum * 0.0188e-6;
        draws = 4.0 + std::hypot(std::max(chain, issue), (double)n * 8.0 * P.L / 5.56e6);
    }
    int g = 0;
    while ((1 << g) < group) ++g;
    const int threads = level_threads(P.level_width, group);
    const size_t lds = (size_t)P.level_slots * (size_t)group * sizeof(double);
    const int64_t per_cu = std::max<int64_t>(1, std::min<int64_t>(kLevelMaxThreads / threads, (int64_t)(kLevelLdsMaxBytes / lds)));
    const int64_t groups = (n + group - 1) / group;
    const double rounds = (double)((groups + cus * per_cu - 1) / (cus * per_cu));
    const double beside = std::min((double)per_cu, std::max(1.0, (double)groups / cus)) - 1.0;
    const double us_per_mb = group <= 2 ? 0.54 : group == 4 ? 0.27 : group <= 16 ? 0.16 : 0.128;
    return draws + 3.0 + rounds * P.level_us[g] * (1.0 + 0.3 * beside) +
           (double)n * (8.0 * (double)P.preds.size() + 12.0 * P.E) * 1e-6 * us_per_mb;
}

// Whether a run of n samples takes the two-pass route (draw_kernel, then
// level_kernel) instead of a partial round of the walk (halved: in one-sample
// tiles if it is of at most 64 samples per CU): where its estimate is a
// twentieth below the walk's, a fifth above 64 samples per CU, where the walk's
// estimate is least certain (179 x 8 events, 31,001 samples 0.60 ms against 0.50
// by a twentieth).  Both estimates' constants are fitted to the times
// of both routes on 34 DAGs (layered ones of 1 to 2,000 events a level, up to 40
// predecessors, uneven levels, far predecessors, every kind of law) at up to 11
// sample counts from 100 to 50,000, sampled and injected: 650 pairs, of which
// the rule leaves none more than 5% slower than its other route and 15 walks
// that two passes would have beaten by more.  A rule on bytes and a latency
// per level alone left 54, up to 1.96 times slower: 120 uneven levels of up to 400
// events, far predecessors, 8,000 samples injected 1.34 ms against 0.92; 71 such
// levels, up to 12 predecessors, 6,000 samples 3.7 against 2.2.
constexpr double kTwoPassMargin = 1.05, kTwoPassMarginFull = 1.2;
bool level_route(mcdp_propagator &P, bool injected, int64_t n, int cus, bool halved) {
    if (P.tail_mode != 0 || P.shape_by_caller || P.E == 0 || P.L == 0 || n > kLevelMaxSamples) return false;
    if (P.two_pass_mode == 2) return false;
    build_level_slots(P);
    const int group = level_group(P, n, cus);
    if (group == 0 || P.two_pass_mode == 1) return group != 0;
    const bool full = n > (int64_t)cus * kLanes;
    return (full ? kTwoPassMarginFull : kTwoPassMargin) * two_pass_us(P, injected, n, group, cus) <
           walk_us(P, injected, n, halved && !full);
}

int launch_level_route(const mcdp_propagator &P, const DeviceCopy &d, bool injected, const int32_t *seeds,
                       const double *dur_in, int64_t n, int64_t ld, double *realized, double *durations,
                       int32_t *cause, uint8_t *cause_pos, int cus, hipStream_t stream) {
    if (!injected) {
        DrawParams q = d.draws;
        q.seeds = seeds;
        q.n = (int32_t)n;
        q.ld = (int32_t)ld;
        q.durations = durations;
        HIP_TRY(launch_draws(q, cus, stream), "draw kernel launch");
    }
    LevelParams p = d.levels;
    p.dur = injected ? dur_in : durations;
    p.n = (int32_t)n;
    p.ld = (int32_t)ld;
    p.realized = realized;
    p.cause = cause;
    p.cause_pos = cause_pos;
    const int group = level_group(P, n, cus);
    const int threads = level_threads(P.level_width, group);
    HIP_TRY(launch_levels(p, P.level_zero_edges, group, threads, P.level_slots, stream), "level kernel launch");
    return MCDP_OK;
}

// cause_pos (sampled walks, no cause): the winning entry's position per
// sample instead of the cause event.  scratch: [L][ld] or null, for a sampled
// run without a durations output that may take the two-pass route.  shared:
// other runs use the device beside this one.
int launch(mcdp_propagator &P, bool injected, const int32_t *seeds, const double *dur_in, int64_t n, int64_t ld,
           double *realized, double *durations, int32_t *cause, hipStream_t stream, uint8_t *cause_pos = nullptr,
           double *scratch = nullptr, bool shared = false) {
    if (n < 0) return fail(MCDP_E_INVALID, "n must be non-negative");
    if (cause_pos && (injected || cause)) return fail(MCDP_E_INVALID, "internal error: positions replace sampled causes");
    if (n > 0 && ld < n) return fail(MCDP_E_INVALID, "ld must be >= n");
    if (n > kMaxSamplesPerLaunch || ld > std::numeric_limits<int32_t>::max())
        return fail(MCDP_E_INVALID, "n and ld must be below 2^31 - 256 per call");
    if (injected && !dur_in && P.L > 0 && n > 0) return fail(MCDP_E_INVALID, "durations input is null");
    if (!injected && !seeds && n > 0) return fail(MCDP_E_INVALID, "seeds is null");
    if (!realized && P.E > 0 && n > 0) return fail(MCDP_E_INVALID, "realized must not be null");
    std::lock_guard<std::mutex> lock(P.mu);
    DeviceCopy *d = nullptr;
    int rc = device_entry_impl(P, d);
    if (rc) return rc;
    int cus = 0, bpc = 0;
    HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, d->device), "hipDeviceGetAttribute");
    // A short run takes the two-pass route where there is room for its
    // durations.  Its plan is uploaded by the first such run: one under
    // stream capture, which can upload nothing, walks unless it is there.
    double *const drawn = durations ? durations : scratch;
    // whether rows of doubles that the walk writes, or reads durations from,
    // start on 64-byte sectors
    const auto on_sector = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 63u) == 0; };
    const bool sectors = ld % 8 == 0 && on_sector(realized) && on_sector(durations) && on_sector(dur_in);
    const bool halved_ok = !shared && ((!durations && !injected) || sectors);
    if (n > 0 && (injected || drawn) && level_route(P, injected, n, cus, halved_ok)) {
        hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
        if (!d->level_blob) (void)hipStreamIsCapturing(stream, &capture);
        if (capture == hipStreamCaptureStatusNone) {
            rc = ensure_levels(P, *d);
            P.last_route = MCDP_ROUTE_TWO_PASS;
            if (!rc)
                return launch_level_route(P, *d, injected, seeds, dur_in, n, ld, realized, drawn, cause, cause_pos, cus,
                                          stream);
            if (rc != MCDP_E_NOMEM) return rc;
            (void)hipGetLastError();  // no room for its plan: the walk's may be there
        }
    }
    if (!P.shape_fixed) {  // first walk: fit the schedule to this device
        rc = choose_shape(P);
        if (rc) return rc;
        P.shape_fixed = true;
    }
    rc = ensure_device_impl(P, d);
    if (rc) return rc;
    if (n == 0 || (P.E == 0 && (injected || P.orph.empty()))) return MCDP_OK;
    P.last_route = 0;
    WalkParams p = d->base;
    p.seeds = seeds;
    p.dur_in = dur_in;
    p.ld = (int32_t)ld;
    p.realized = realized;
    p.durations = injected ? nullptr : durations;
    p.cause = cause;
    p.cause_pos = cause_pos;
    WalkVariant v = walk_variant(P, injected);
    v.pos = cause_pos != nullptr;
    const size_t lds = walk_lds_bytes(P, v);
    HIP_TRY(walk_occupancy(v, P.waves, lds, &bpc), "hipOccupancyMaxActiveBlocksPerMultiprocessor");
    if (bpc < 1) return fail(MCDP_E_DEVICE, "walk kernel cannot be resident with " + std::to_string(lds) + " bytes of LDS");
    // Rows that do not start on 64-byte sectors (an odd ld): the pieces that two
    // tiles write of a sector reach memory as two partial writes, and the walk
    // falls to about 2.7-3.8 TB/s where whole sectors reach 5.8.  Overlapping
    // tiles whose stores begin and end on sectors (WalkVariant::shift) compute
    // one sample in sixteen twice instead.  They are taken where the writes are
    // the bound: one workgroup per CU, cheap draws for the bytes (kShiftBytesPerCost
    // of a tile's output per unit of tile_cost; the network and 60 x 100 DAGs with
    // exponential or gamma laws have about 290, with calibrated laws 195, where the
    // overlap costs 3-6%), and three quarters of a round or more.  200 x 100, ld = n,
    // before and after: 17,001 samples 3.7 and 3.2 ms, but 60 x 100 0.95 and 0.98;
    // 30,001 6.8 and 4.0; 32,767 7.2 and 5.7; 65,537 13.8 and 9.0; 98,303 15.7-19.3
    // and 13.2.  Not for injected durations (98,303 samples 13.8 and 14.1 ms), of
    // which most bytes are reads.
    constexpr double kShiftBytesPerCost = 244.0;
    v.shift = !injected && durations && !sectors && v.paths == kPathsFast && v.spl == 2 && !v.pos && P.tail_mode == 0 &&
              bpc == 1 && 4 * n > 3 * (int64_t)cus * kLanes * 2 &&
              (double)(kLanes * 2) * (8.0 * P.L + 12.0 * P.E) > kShiftBytesPerCost * (double)P.tile_cost;
    const int64_t resident = (int64_t)cus * bpc;
    const int64_t tile = v.shift ? kShiftStep : (int64_t)kLanes * v.spl;  // samples a tile adds

    // A tile's run time hardly depends on how many of its lanes are live, so a
    // last round of only a few tiles costs almost a full round.  The samples
    // past the last full round take one of two cheaper routes:
    //   * wide steps: one launch per step, each event of the step a wave of
    //     its own for every group of 64 samples, predecessors read from the
    //     output rows; the tail's latency is then about the steps' launch gaps
    //     plus their costliest events, instead of a whole tile's walk;
    //   * with two samples per lane, the one-sample-per-lane kernel of the
    //     same schedule, whose tiles finish sooner.
    // The wide steps run beside the full rounds' tiles (below), so they cost
    // little as long as they end before the tiles do: they are taken when
    // their estimated latency (from the schedule) is below that of the full
    // rounds.
    // Results do not depend on the split or the route.
    int64_t n_main = n, n_tail = 0;
    bool wide = false;
    WalkVariant v1 = v;
    v1.spl = 1;
    v1.shift = false;
    const size_t lds1 = walk_lds_bytes(P, v1);
    int64_t resident1 = 0;
    // A run of at most one group of 64 samples per CU fits the device in
    // one-sample tiles at once, which take about seven tenths of a two-sample
    // tile's time (200 x 100 events, 16,384 samples: 2.13 against 2.95 ms; a
    // second round of them, from 16,385 samples, 4.2 against 3.6).  They take
    // more of the device in all, which a run beside others pays for (12,000 to
    // 16,384 samples, on two streams at once 1.07-1.28 times the two-sample tiles'
    // time, on four 0.85-0.94, alone 0.63-0.67), and their 512-byte pieces of rows that do not start on cache sectors cost more
    // than they save (16,383 samples: 4.3 against 3.2 ms; without durations no
    // matter).
    const bool halved =
        v.spl == 2 && P.tail_mode == 0 && !P.shape_by_caller && halved_ok && n <= (int64_t)cus * kLanes;
    const int64_t wide_max = halved && tiles_early(P, injected) ? kWideMaxGroupsHalved : kWideMaxGroups;
    {
        const int64_t full_rounds = ((n + tile - 1) / tile) / resident;
        const int64_t rest = n - full_rounds * resident * tile;
        const int64_t groups = (rest + kLanes - 1) / kLanes;
        if (full_rounds == 0 && rest > 0) {
            // less than one round: the wide steps alone against one round of
            // tiles that hardly fills the device
            if (P.tail_mode == 2 || (P.tail_mode == 0 && groups <= wide_max && P.wide_cost < P.tile_cost)) {
                wide = true;
                n_main = 0;
                n_tail = n;
            } else if (halved) {
                int bpc1 = 0;
                HIP_TRY(walk_occupancy(v1, P.waves, lds1, &bpc1), "hipOccupancyMaxActiveBlocksPerMultiprocessor");
                resident1 = (int64_t)cus * bpc1;
                if (groups <= resident1) {
                    n_main = 0;
                    n_tail = n;
                }
            }
        } else if (full_rounds >= 1 && rest > 0) {
            if (P.tail_mode == 2 ||
                (P.tail_mode == 0 && groups <= kWideMaxGroups && P.wide_cost < full_rounds * P.tile_cost)) {
                wide = true;
                n_main = n - rest;
                n_tail = rest;
            } else if (v.spl == 2) {
                int bpc1 = 0;
                HIP_TRY(walk_occupancy(v1, P.waves, lds1, &bpc1), "hipOccupancyMaxActiveBlocksPerMultiprocessor");
                resident1 = (int64_t)cus * bpc1;
                if (bpc1 >= 1 && groups <= resident1) {
                    n_main = n - rest;
                    n_tail = rest;
                }
            }
        }
    }
    p.n = (int32_t)n_main;
    p.n_tiles = (int32_t)(v.shift ? shifted_tiles(n_main) : (n_main + tile - 1) / tile);
    // The wide steps need no LDS and fewer registers than a tile leaves free
    // on a SIMD, so they run on a second stream beside the tiles, forked from
    // the caller's stream before the tiles and joined after.
    hipStream_t tail_stream = stream;
    if (wide && n_main > 0) {
        HIP_TRY(hipEventRecord(d->fork, stream), "hipEventRecord");
        HIP_TRY(hipStreamWaitEvent(d->side, d->fork, 0), "hipStreamWaitEvent");
        tail_stream = d->side;
    }
    if (n_main > 0) {
        P.last_route |= v.shift ? MCDP_ROUTE_OVERLAPPING_TILES : v.spl == 1 ? MCDP_ROUTE_ONE_SAMPLE_TILES : MCDP_ROUTE_TILES;
        HIP_TRY(launch_walk(p, v, (int)std::min<int64_t>(p.n_tiles, resident), lds, stream), "walk kernel launch");
    }
    if (n_tail > 0) {
        WalkParams q = p;
        q.seeds = seeds ? seeds + n_main : nullptr;
        q.dur_in = dur_in ? dur_in + n_main : nullptr;
        q.realized = realized + n_main;
        q.durations = p.durations ? p.durations + n_main : nullptr;
        q.cause = cause ? cause + n_main : nullptr;
        q.cause_pos = cause_pos ? cause_pos + n_main : nullptr;
        q.n = (int32_t)n_tail;
        q.n_tiles = (int32_t)((n_tail + kLanes - 1) / kLanes);
        P.last_route |= wide ? MCDP_ROUTE_WIDE_STEPS : MCDP_ROUTE_ONE_SAMPLE_TILES;
        if (wide) {
            const int32_t groups = q.n_tiles;
            const int32_t W = P.waves;
            for (int32_t t = 0; t < P.n_steps; ++t) {
                const int32_t e0 = P.ev_off[(size_t)t * W], e1 = P.ev_off[(size_t)(t + 1) * W];
                HIP_TRY(launch_walk_wide(q, injected, e0, e1 - e0, groups, tail_stream), "wide step launch");
            }
            if (!injected) HIP_TRY(launch_walk_wide_orphans(q, groups, tail_stream), "wide orphans launch");
            if (tail_stream != stream) {
                HIP_TRY(hipEventRecord(d->join, tail_stream), "hipEventRecord");
                HIP_TRY(hipStreamWaitEvent(stream, d->join, 0), "hipStreamWaitEvent");
            }
        } else {
            HIP_TRY(launch_walk(q, v1, (int)std::min<int64_t>(q.n_tiles, resident1), lds1, stream), "walk kernel launch");
        }
    }
    return MCDP_OK;
}

}  // namespace

namespace {

// Workspaces of more than kHostWorkKeepBytes between calls.  Giving such memory
// back and having it again costs 27 ms per GB (the driver clears it): 171 ms a
// call for the statistics of 32,768 samples of the network DAG, whose kernels
// take 5.  So the process keeps some: per device at most an eighth of its
// memory in all, and only while a quarter of it stays free; the oldest goes
// first.  A propagator's calls and the next propagator's share them (a call
// owns its workspace from taking it to giving it back, its stream idle), they
// are freed with the propagator that used them last, before any allocation of
// this library fails, and when the caller asks for it, whose other allocators
// cannot reach them (mcdp_release_workspaces).
struct LargePool {
    struct Entry {
        int device;
        void *buf;
        size_t bytes;
        const void *owner;
    };
    std::mutex mu;
    std::vector<Entry> kept;  // oldest first

    static void release(const Entry &e) {
        int cur = -1;
        (void)hipGetDevice(&cur);
        (void)hipSetDevice(e.device);
        (void)hipFree(e.buf);
        if (cur >= 0) (void)hipSetDevice(cur);
    }
    // The smallest kept workspace of at least `need` bytes, or null.
    void *take(int device, size_t need, size_t &bytes) {
        std::lock_guard<std::mutex> lock(mu);
        size_t best = kept.size();
        for (size_t i = 0; i < kept.size(); ++i)
            if (kept[i].device == device && kept[i].bytes >= need && (best == kept.size() || kept[i].bytes < kept[best].bytes))
                best = i;
        if (best == kept.size()) return nullptr;
        void *buf = kept[best].buf;
        bytes = kept[best].bytes;
        kept.erase(kept.begin() + (std::ptrdiff_t)best);
        return buf;
    }
    // Keeps or frees an idle workspace of the current device.  (What goes is
    // freed after the lock: hipFree waits for the device.)
    void give(int device, void *buf, size_t bytes, const void *owner) {
        const Entry e{device, buf, bytes, owner};
        std::vector<Entry> gone;
        size_t free_bytes = 0, total = 0;
        if (hipMemGetInfo(&free_bytes, &total) != hipSuccess || bytes > total / 8 || free_bytes < total / 4) {
            gone.push_back(e);
        } else {
            std::lock_guard<std::mutex> lock(mu);
            size_t sum = bytes;
            for (const Entry &k : kept) sum += k.device == device ? k.bytes : 0;
            remove([&](const Entry &k) { return k.device == device && sum > total / 8 && ((sum -= k.bytes), true); }, gone);
            kept.push_back(e);
        }
        for (const Entry &k : gone) release(k);
    }
    // Frees every kept workspace that `which` names; whether there was one.
    template <typename F>
    bool drop(F &&which) {
        std::vector<Entry> gone;
        {
            std::lock_guard<std::mutex> lock(mu);
            remove(which, gone);
        }
        for (const Entry &k : gone) release(k);
        return !gone.empty();
    }

   private:
    // Moves the kept workspaces that `which` names, oldest first, to `gone`.
    template <typename F>
    void remove(F &&which, std::vector<Entry> &gone) {
        std::vector<Entry> left;
        for (const Entry &k : kept) (which(k) ? gone : left).push_back(k);
        kept.swap(left);
    }
};
// (never destroyed: propagators may outlive static objects)
LargePool &large_pool() {
    static LargePool *const pool = new LargePool;
    return *pool;
}

}  // namespace

hipError_t mcdp::device_malloc(void **ptr, size_t bytes) {
    hipError_t e = hipMalloc(ptr, bytes);
    if (e == hipSuccess) return e;
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return e;
    if (!large_pool().drop([&](const LargePool::Entry &k) { return k.device == device; })) return e;
    (void)hipGetLastError();
    return hipMalloc(ptr, bytes);
}

void mcdp::large_pool_drop(const void *owner) {
    (void)large_pool().drop([&](const LargePool::Entry &k) { return k.owner == owner; });
}

int mcdp::host_workspace(mcdp_propagator &P, size_t need, void *&buf, hipStream_t &stream) {
    int device = 0;
    HIP_TRY(hipGetDevice(&device), "hipGetDevice");
    HostWork *hw = nullptr;
    for (auto &h : P.host_work)
        if (h.device == device) hw = &h;
    if (!hw) {
        HostWork h;
        h.device = device;
        HIP_TRY(hipStreamCreateWithFlags(&h.stream, hipStreamNonBlocking), "hipStreamCreate");
        P.host_work.push_back(h);
        hw = &P.host_work.back();
    }
    stream = hw->stream;
    if (need > kHostWorkKeepBytes) {
        hw->large = large_pool().take(device, need, hw->large_bytes);
        if (!hw->large) {
            hipError_t e = device_malloc(&hw->large, need);
            if (e != hipSuccess) {
                hw->large = nullptr;
                return fail(MCDP_E_NOMEM, std::string("hipMalloc (host-call workspace): ") + hipGetErrorString(e));
            }
            hw->large_bytes = need;
        }
        buf = hw->large;
        return MCDP_OK;
    }
    if (hw->bytes < need) {
        if (hw->buf) {
            (void)hipStreamSynchronize(hw->stream);  // idle already: every call ends by waiting on it
            hw->drop_graph();
            (void)hipFree(hw->buf);
            hw->buf = nullptr;
            hw->bytes = 0;
        }
        hipError_t e = device_malloc(&hw->buf, std::max<size_t>(need, 256));
        if (e != hipSuccess) {
            hw->buf = nullptr;
            return fail(MCDP_E_NOMEM, std::string("hipMalloc (host-call workspace): ") + hipGetErrorString(e));
        }
        hw->bytes = std::max<size_t>(need, 256);
    }
    buf = hw->buf;
    return MCDP_OK;
}

void mcdp::host_workspace_trim(mcdp_propagator &P) {
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return;
    for (auto &h : P.host_work)
        if (h.device == device && h.large) {
            (void)hipStreamSynchronize(h.stream);
            h.drop_graph();  // it may have been captured in this workspace
            large_pool().give(device, h.large, h.large_bytes, &P);
            h.large = nullptr;
            h.large_bytes = 0;
        }
}

namespace {

// The caller's output arrays, faulted in by several threads while the device
// works, for calls whose results copy directly (no staging buffers): a page's
// first touch costs a fault, which those copies would otherwise take one page at
// a time on one thread (for the network DAG's 2,048 samples, 1.3 GB: about 50 of
// 130 ms).  The pages get zeros, which the copies then overwrite; regions under
// 64 MB are left alone.
class Prefault {
   public:
    void start(const std::vector<std::pair<char *, size_t>> &regions) {
        size_t total = 0;
        for (const auto &r : regions) total += r.second;
        if (total < ((size_t)64 << 20)) return;
        const unsigned hw = std::max(1u, std::thread::hardware_concurrency());
        const size_t nt = std::min<size_t>(16, hw);
        const size_t share = (total + nt - 1) / nt;
        std::vector<std::pair<char *, size_t>> pieces;  // (start, bytes) of every thread, in order
        size_t taken = 0;
        for (const auto &r : regions)
            for (size_t o = 0; o < r.second;) {
                const size_t room = share - taken % share;
                const size_t len = std::min(room, r.second - o);
                pieces.emplace_back(r.first + o, len);
                o += len;
                taken += len;
            }
        try {
            threads_.reserve(nt);
            for (size_t t = 0; t < nt; ++t) spawn(pieces, t, share);
        } catch (...) {  // no threads to spare: the copies fault the pages in themselves
            join();
        }
    }
    void join() {
        for (auto &t : threads_) t.join();
        threads_.clear();
    }
    ~Prefault() { join(); }

   private:
    void spawn(const std::vector<std::pair<char *, size_t>> &pieces, size_t t, size_t share) {
        threads_.emplace_back([pieces, t, share] {
            size_t at = 0;
            for (const auto &pc : pieces) {  // the pieces whose bytes fall in this thread's share
                const size_t lo = at, hi = at + pc.second;
                at = hi;
                const size_t a = std::max(lo, t * share), b = std::min(hi, (t + 1) * share);
                if (a < b) {
                    char *p = pc.first + (a - lo);
#ifdef MADV_POPULATE_WRITE
                    // whole pages inside the range in one call; the edges by hand
                    const uintptr_t pg = (uintptr_t)sysconf(_SC_PAGESIZE), x = (uintptr_t)p, y = x + (b - a);
                    const uintptr_t x1 = (x + pg - 1) / pg * pg, y1 = y / pg * pg;
                    if (y1 > x1 && madvise((void *)x1, y1 - x1, MADV_POPULATE_WRITE) == 0) {
                        std::memset(p, 0, x1 - x);
                        std::memset((void *)y1, 0, y - y1);
                        continue;
                    }
#endif
                    std::memset(p, 0, b - a);
                }
            }
        });
    }
    std::vector<std::thread> threads_;
};

// Large copies between the device and the caller's (pageable) arrays through
// pinned staging: kStageThreads threads, each with its own stream and pinned
// buffer of kStageBytes, take pieces of the arrays in turn and move each
// through their buffer.  A copy straight to or from pageable memory goes
// through one staging path in the runtime whatever the number of threads
// issuing it; this way several transfers run at once, and the host-side copies
// overlap them.  The buffers and streams exist once per device (64 MB of pinned
// memory, held until the process ends); calls take turns on them.
constexpr int kStageThreads = 8;
constexpr size_t kStageBytes = (size_t)8 << 20;
constexpr size_t kStageMinBytes = (size_t)16 << 20;  // smaller arrays copy directly

struct StageSet {
    int device = -1;
    void *buf[kStageThreads] = {};
    hipStream_t stream[kStageThreads] = {};
};
std::mutex g_stage_mu;
std::vector<StageSet> g_stage;

// One array of a chunk: rows of `width` bytes, `dev_pitch` apart on the device
// and `host_pitch` apart in the caller's array.
struct CopyPlane {
    char *host;
    char *dev;
    size_t rows, width, dev_pitch, host_pitch;
};

// A piece: rows [r0, r0 + k) and bytes [b0, b0 + len) of each of them.  Its
// device bytes are the contiguous span from row r0's byte b0 to row r0+k-1's
// byte b0+len, at most kStageBytes; an upload also writes the span's bytes
// between rows (columns past `width`, which the chunk does not use).
struct CopyPiece {
    const CopyPlane *plane;
    size_t r0, k, b0, len;
};

// The current device's staging set, created on first use; nullptr when its
// buffers cannot be had.  Call with g_stage_mu held.
StageSet *stage_set() {
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return nullptr;
    for (auto &g : g_stage)
        if (g.device == device) return &g;
    StageSet g;
    g.device = device;
    for (int t = 0; t < kStageThreads; ++t) {
        hipError_t e = hipHostMalloc(&g.buf[t], kStageBytes, hipHostMallocDefault);
        if (e == hipSuccess) e = hipStreamCreateWithFlags(&g.stream[t], hipStreamNonBlocking);
        if (e != hipSuccess) {
            for (int u = 0; u <= t; ++u) {
                if (g.buf[u]) (void)hipHostFree(g.buf[u]);
                if (g.stream[u]) (void)hipStreamDestroy(g.stream[u]);
            }
            return nullptr;
        }
    }
    g_stage.push_back(g);
    return &g_stage.back();
}

// True when large arrays of this device can go through the staging buffers.
bool staging_available() {
    std::lock_guard<std::mutex> lock(g_stage_mu);
    return stage_set() != nullptr;
}

// Moves every plane device -> host (to_host) or host -> device, synchronously.
// The device side must be ready (no kernel still writing or reading it).
// Returns an mcdp_status, or -1 when the staging buffers cannot be had (then
// nothing was copied).
int staged_copy(const std::vector<CopyPlane> &planes, bool to_host) {
    std::lock_guard<std::mutex> lock(g_stage_mu);
    StageSet *set = stage_set();
    if (!set) return -1;
    std::vector<CopyPiece> pieces;
    for (const auto &pl : planes) {
        if (pl.rows == 0 || pl.width == 0) continue;
        if (pl.width == pl.dev_pitch && pl.width == pl.host_pitch) {
            // rows back to back on both sides: one long row
            const size_t total = pl.rows * pl.width;
            for (size_t b = 0; b < total; b += kStageBytes)
                pieces.push_back({&pl, 0, 1, b, std::min(kStageBytes, total - b)});
        } else if (pl.dev_pitch <= kStageBytes) {
            const size_t per = kStageBytes / pl.dev_pitch;
            for (size_t r = 0; r < pl.rows; r += per) pieces.push_back({&pl, r, std::min(per, pl.rows - r), 0, pl.width});
        } else {
            for (size_t r = 0; r < pl.rows; ++r)
                for (size_t b = 0; b < pl.width; b += kStageBytes)
                    pieces.push_back({&pl, r, 1, b, std::min(kStageBytes, pl.width - b)});
        }
    }
    std::atomic<size_t> next{0};
    std::atomic<int> failed{0};
    hipError_t first_error = hipSuccess;
    std::mutex err_mu;
    auto work = [&](int t) {
        if (t > 0 && hipSetDevice(set->device) != hipSuccess) return;  // a new thread starts on device 0
        char *stage = static_cast<char *>(set->buf[t]);
        for (size_t i; !failed.load(std::memory_order_relaxed) && (i = next.fetch_add(1)) < pieces.size();) {
            const CopyPiece &pc = pieces[i];
            const CopyPlane &pl = *pc.plane;
            const bool flat = pl.width == pl.dev_pitch && pl.width == pl.host_pitch;
            const size_t pitch = flat ? 0 : pl.dev_pitch;  // of the rows in the staging buffer, as on the device
            const size_t host_pitch = flat ? 0 : pl.host_pitch;
            const size_t span = (pc.k - 1) * pitch + pc.len;
            char *dev = pl.dev + pc.r0 * pitch + pc.b0;
            if (!to_host)
                for (size_t j = 0; j < pc.k; ++j)
                    std::memcpy(stage + j * pitch, pl.host + (pc.r0 + j) * host_pitch + pc.b0, pc.len);
            hipError_t e = to_host ? hipMemcpyAsync(stage, dev, span, hipMemcpyDeviceToHost, set->stream[t])
                                   : hipMemcpyAsync(dev, stage, span, hipMemcpyHostToDevice, set->stream[t]);
            if (e == hipSuccess) e = hipStreamSynchronize(set->stream[t]);
            if (e != hipSuccess) {
                std::lock_guard<std::mutex> g(err_mu);
                if (first_error == hipSuccess) first_error = e;
                failed.store(1);
                return;
            }
            if (to_host)
                for (size_t j = 0; j < pc.k; ++j)
                    std::memcpy(pl.host + (pc.r0 + j) * host_pitch + pc.b0, stage + j * pitch, pc.len);
        }
    };
    std::vector<std::thread> threads;
    try {
        for (int t = 1; t < kStageThreads; ++t) threads.emplace_back(work, t);
    } catch (...) {  // fewer threads: the ones running take every piece
    }
    work(0);
    for (auto &th : threads) th.join();
    if (failed.load()) return hip_fail(first_error, to_host ? "hipMemcpy (outputs)" : "hipMemcpy (inputs)");
    return MCDP_OK;
}

// Short runs through the host path replay a captured graph of their launches
// (HostWork): for up to this many samples, which stay below one round of tiles
// on any device, so the launches are one stream's sequence; and for plans of at
// least kGraphMinSteps steps.  A replay spends about 1.7 us per dependent launch
// against about 3 us for launches one by one, but a graph of a single kernel
// (the tiles' route) is slower to launch than the kernel alone.
constexpr int64_t kGraphMaxSamples = 1024;
constexpr int32_t kGraphMinSteps = 32;

// The chunk's launches (launch()).  A run of one chunk of at most
// kGraphMaxSamples samples whose key (ShortRunKey) matches the previous call's
// is captured into a graph and launched as one; while the key stays, later
// calls replay that graph.  Any other call, or a capture that fails, launches
// directly.  `work` is the workspace that holds the buffers.  The caller holds
// P.host_mu.
int launch_host_chunk(mcdp_propagator &P, HostWork *hw, const void *work, bool injected, const int32_t *d_seeds,
                      double *d_dur, int64_t m, int64_t ld, double *d_real, int32_t *d_cause, hipStream_t st) {
    auto direct = [&] {
        return launch(P, injected, d_seeds, d_dur, m, ld, d_real, injected ? nullptr : d_dur, d_cause, st);
    };
    if (!hw || m != ld || m > kGraphMaxSamples || P.n_steps < kGraphMinSteps) return direct();
    bool two_pass = false;  // two launches: no graph
    const int qc = short_run(P, injected, m, two_pass);
    if (qc) return qc;
    if (two_pass) return direct();
    ShortRunKey key;
    key.buf = work;
    key.n = m;
    key.ld = ld;
    key.injected = injected;
    key.generation = P.generation.load();
    key.tail_mode = P.tail_mode;
    auto replay = [&] {
        {
            std::lock_guard<std::mutex> lock(P.mu);
            P.last_route = MCDP_ROUTE_GRAPH;
        }
        HIP_TRY(hipGraphLaunch(hw->graph, st), "hipGraphLaunch");
        return (int)MCDP_OK;
    };
    if (hw->graph && hw->captured == key) return replay();
    if (!(hw->seen == key)) {  // first sight: the shape and the plan's upload happen here, not in a capture
        hw->seen = key;
        return direct();
    }
    if (hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal) != hipSuccess) {
        (void)hipGetLastError();
        return direct();
    }
    const int rc = direct();
    hipGraph_t g = nullptr;
    const hipError_t ee = hipStreamEndCapture(st, &g);
    hipGraphExec_t exec = nullptr;
    const bool ok = rc == MCDP_OK && ee == hipSuccess && g && hipGraphInstantiate(&exec, g, nullptr, nullptr, 0) == hipSuccess;
    if (g) (void)hipGraphDestroy(g);
    if (!ok) {  // launch directly; this key is not captured again until it is seen twice anew
        (void)hipGetLastError();
        hw->seen = ShortRunKey{};
        return direct();
    }
    if (hw->graph) (void)hipGraphExecDestroy(hw->graph);
    hw->graph = exec;
    hw->captured = key;
    return replay();
}

// The host-path state of the current device (after host_workspace).
HostWork *current_host_work(mcdp_propagator &P) {
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return nullptr;
    for (auto &h : P.host_work)
        if (h.device == device) return &h;
    return nullptr;
}

// Host-buffer convenience: runs in chunks of samples so device memory stays
// bounded, and copies each chunk into the caller's event-major arrays.  The
// device buffers and the stream are the propagator's (HostWork), kept from
// call to call; the call waits on that stream only, so other streams of the
// process (a server's, a caller's own) keep running.
int run_host(mcdp_propagator &P, bool injected, const int32_t *seeds, const double *dur_in, int64_t n,
             double *realized, double *durations, int32_t *cause) {
    if (n < 0) return fail(MCDP_E_INVALID, "n must be non-negative");
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0)
        return fail(MCDP_E_DEVICE, "no HIP device available: the Monte Carlo engine runs on the GPU only");
    if (n == 0) return MCDP_OK;
    const int64_t E = P.E, L = P.L;
    const int64_t per_sample = 12 * E + 8 * L + 8;
    int64_t chunk = std::max<int64_t>(kLanes, ((int64_t)1 << 31) / std::max<int64_t>(per_sample, 1));
    chunk = std::min<int64_t>(n, chunk / kLanes * kLanes);
    const size_t o_cause = align_up(sizeof(double) * E * chunk, 256);
    const size_t o_dur = o_cause + align_up(sizeof(int32_t) * E * chunk, 256);
    const size_t o_seeds = o_dur + align_up(sizeof(double) * L * chunk, 256);
    const size_t need = o_seeds + align_up(sizeof(int32_t) * chunk, 256);

    std::lock_guard<std::mutex> host_lock(P.host_mu);
    void *work = nullptr;
    hipStream_t st = nullptr;
    int rc = host_workspace(P, need, work, st);
    if (rc) return rc;
    HostWork *const hw = current_host_work(P);
    auto *base = static_cast<unsigned char *>(work);
    auto *d_real = reinterpret_cast<double *>(base);
    auto *d_cause = reinterpret_cast<int32_t *>(base + o_cause);
    auto *d_dur = reinterpret_cast<double *>(base + o_dur);
    auto *d_seeds = reinterpret_cast<int32_t *>(base + o_seeds);
    // With staging, the copying threads fault the caller's pages in themselves, in parallel and while
    // other pieces are in flight; without it the copies would take them one at a time.
    const size_t total_out = (size_t)n * ((realized ? 8 * E : 0) + (cause ? 4 * E : 0) +
                                          (durations && !injected ? 8 * L : 0));
    const bool staged = total_out >= kStageMinBytes && staging_available();
    Prefault prefault;
    if (!staged)
        prefault.start({{reinterpret_cast<char *>(realized), realized ? sizeof(double) * (size_t)(E * n) : 0},
                        {reinterpret_cast<char *>(cause), cause ? sizeof(int32_t) * (size_t)(E * n) : 0},
                        {reinterpret_cast<char *>(durations),
                         (durations && !injected) ? sizeof(double) * (size_t)(L * n) : 0}});
    for (int64_t c0 = 0; c0 < n && rc == MCDP_OK; c0 += chunk) {
        const int64_t m = std::min(chunk, n - c0);
        hipError_t e = hipSuccess;
        // one chunk of all samples: host and device rows have the same pitch, so every array moves as
        // one contiguous copy (a 2-D copy of many short rows, e.g. one sample, costs a transfer per row)
        const bool whole = chunk == n;
        if (injected) {
            // the workspace is idle here: every chunk ends by waiting on the stream
            const size_t in_bytes = sizeof(double) * (size_t)L * (size_t)m;
            int sc = -1;
            if (L > 0 && in_bytes >= kStageMinBytes)
                sc = staged_copy({{const_cast<char *>(reinterpret_cast<const char *>(dur_in + c0)),
                                   reinterpret_cast<char *>(d_dur), (size_t)L, sizeof(double) * m,
                                   sizeof(double) * chunk, sizeof(double) * n}},
                                 false);
            if (sc > 0) {
                rc = sc;
                break;
            }
            if (L > 0 && sc < 0)
                e = whole ? hipMemcpyAsync(d_dur, dur_in, sizeof(double) * L * n, hipMemcpyHostToDevice, st)
                          : hipMemcpy2DAsync(d_dur, sizeof(double) * chunk, dur_in + c0, sizeof(double) * n,
                                             sizeof(double) * m, (size_t)L, hipMemcpyHostToDevice, st);
        } else {
            e = hipMemcpyAsync(d_seeds, seeds + c0, sizeof(int32_t) * m, hipMemcpyHostToDevice, st);
        }
        if (e != hipSuccess) {
            rc = hip_fail(e, "hipMemcpy (inputs)");
            break;
        }
        rc = launch_host_chunk(P, hw, work, injected, d_seeds, d_dur, m, chunk, d_real, d_cause, st);
        if (rc) break;
        prefault.join();  // the pages are ready before the first copy writes them
        const size_t out_bytes = (size_t)m * ((realized ? 8 * E : 0) + (cause ? 4 * E : 0) +
                                              (durations && !injected ? 8 * L : 0));
        if (staged && out_bytes >= kStageMinBytes) {
            if ((e = hipStreamSynchronize(st)) != hipSuccess) {
                rc = hip_fail(e, "walk kernel");
                break;
            }
            std::vector<CopyPlane> planes;
            auto plane = [&](void *host, void *dev, size_t elem, int64_t rows) {
                if (host && rows > 0)
                    planes.push_back({static_cast<char *>(host) + elem * c0, static_cast<char *>(dev), (size_t)rows,
                                      elem * m, elem * chunk, elem * n});
            };
            plane(realized, d_real, sizeof(double), E);
            plane(cause, d_cause, sizeof(int32_t), E);
            if (!injected) plane(durations, d_dur, sizeof(double), L);
            const int sc = staged_copy(planes, true);
            if (sc >= 0) {
                rc = sc;
                continue;
            }
        }
        auto copy_out = [&](void *dst, const void *src, size_t elem, int64_t rows) -> hipError_t {
            if (!dst || rows == 0) return hipSuccess;
            if (whole) return hipMemcpyAsync(dst, src, elem * (size_t)n * (size_t)rows, hipMemcpyDeviceToHost, st);
            return hipMemcpy2DAsync(static_cast<char *>(dst) + elem * c0, elem * n, src, elem * chunk, elem * m,
                                    (size_t)rows, hipMemcpyDeviceToHost, st);
        };
        if ((e = copy_out(realized, d_real, sizeof(double), E)) != hipSuccess ||
            (e = copy_out(cause, d_cause, sizeof(int32_t), E)) != hipSuccess ||
            (!injected && (e = copy_out(durations, d_dur, sizeof(double), L)) != hipSuccess)) {
            rc = hip_fail(e, "hipMemcpy (outputs)");
            break;
        }
        if ((e = hipStreamSynchronize(st)) != hipSuccess) rc = hip_fail(e, "walk kernel");
    }
    if (rc) (void)hipStreamSynchronize(st);  // nothing of this call may still use the buffers
    host_workspace_trim(P);
    return rc;
}

}  // namespace

int mcdp::device_entry(mcdp_propagator &P, DeviceCopy *&out) { return device_entry_impl(P, out); }

int mcdp::short_run(mcdp_propagator &P, bool injected, int64_t n, bool &yes) {
    std::lock_guard<std::mutex> lock(P.mu);
    int device = 0, cus = 0;
    HIP_TRY(hipGetDevice(&device), "hipGetDevice");
    HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device), "hipDeviceGetAttribute");
    yes = n > 0 && level_route(P, injected, n, cus, true);
    return MCDP_OK;
}

int mcdp::ensure_device(mcdp_propagator &P, DeviceCopy *&out) {
    // The uploaded plan must be the one the walk kernel will run: fix the
    // schedule shape first, as the first launch would.
    if (!P.shape_fixed) {
        int count = 0;
        if (hipGetDeviceCount(&count) != hipSuccess || count <= 0)
            return fail(MCDP_E_DEVICE, "no HIP device available: the Monte Carlo engine runs on the GPU only");
        int rc = choose_shape(P);
        if (rc) return rc;
        P.shape_fixed = true;
    }
    return ensure_device_impl(P, out);
}
mcdp::WalkVariant mcdp::plan_variant(const mcdp_propagator &P, bool injected) { return walk_variant(P, injected); }
size_t mcdp::plan_lds_bytes(const mcdp_propagator &P, WalkVariant v) { return walk_lds_bytes(P, v); }
mcdp::Record mcdp::link_record(const mcdp_propagator &P, int32_t l) { return edge_record(P, l); }

int32_t mcdp::max_entries(const mcdp_propagator &P) {
    int64_t m = 0;
    for (int32_t e = 0; e < P.E; ++e) m = std::max(m, P.pred_off[(size_t)e + 1] - P.pred_off[(size_t)e]);
    return (int32_t)std::min<int64_t>(m, std::numeric_limits<int32_t>::max());
}

int mcdp::run_many_positions(mcdp_propagator &P, const int32_t *seeds_dev, int64_t n, int64_t ld, double *realized,
                             uint8_t *cause_pos, hipStream_t s, double *scratch, bool shared) {
    if (!cause_pos) return fail(MCDP_E_INVALID, "positions output is null");
    if (max_entries(P) > kMaxPositionEntries)
        return fail(MCDP_E_INVALID, "winner positions need events of at most 254 predecessor entries");
    if (n > 0 && !seeds_dev) return fail(MCDP_E_INVALID, "seeds is null");
    return launch(P, false, seeds_dev, nullptr, n, ld, realized, nullptr, nullptr, s, cause_pos, scratch, shared);
}

int mcdp::run_many_shared(mcdp_propagator &P, const int32_t *seeds_dev, int64_t n, int64_t ld, double *realized,
                          int32_t *cause, hipStream_t s) {
    return launch(P, false, seeds_dev, nullptr, n, ld, realized, nullptr, cause, s, nullptr, nullptr, true);
}

// The range of every duration the sampler can draw for link l, as the device
// rounds it (mcdp_sampler.hpp: base + extra, extra = X * d, one rounding
// each): X in [x0, x1] for the multiplier kinds (exponential and gamma X >= 0,
// at most max_scale), the reachable alias-table values for the empirical
// kinds.  Rounding is monotone, so the two ends bound every draw.  A link
// that can draw NaN gets [-inf, +inf]: a NaN candidate never wins the max, so
// it acts as the smallest candidate.
void mcdp::link_duration_range(const mcdp_propagator &P, int32_t l, double &lo, double &hi) {
    constexpr double inf = std::numeric_limits<double>::infinity();
    const double d = P.dmin[(size_t)l];
    lo = -inf;
    hi = inf;
    if (std::isnan(d)) return;
    const uint32_t di = P.ldist[(size_t)l];
    if (di == kNoDistIndex) {
        lo = hi = d;
        return;
    }
    const DistRec &D = P.dist[di];
    auto rel = [&](double x) {  // d + x d, rounded as the device does
        const double extra = x * d;
        return d + extra;
    };
    auto ends = [&](double a, double b) {
        if (std::isnan(a) || std::isnan(b)) return;
        lo = std::min(a, b);
        hi = std::max(a, b);
    };
    // multiplier X in [x0, x1] (x1 may be +inf while every draw is finite)
    auto mult = [&](double x0, double x1) {
        if (!std::isfinite(d)) return;
        if (d == 0.0) {  // a finite X times a zero is a zero
            lo = hi = rel(0.0);
            return;
        }
        ends(rel(x0), std::isinf(x1) ? (d > 0.0 ? inf : -inf) : rel(x1));
    };
    switch (D.kind) {
        case kNone: lo = hi = d; return;
        case kConstant:
        case kEmpiricalRel1: ends(rel(D.p[0]), rel(D.p[0])); return;
        case kEmpiricalAbs1: ends(d + D.p[0], d + D.p[0]); return;
        case kExpInf: mult(0.0, inf); return;
        case kExpTrunc: mult(0.0, D.p[2]); return;
        case kGammaErlang2:
        case kGammaHalf:
        case kGammaMT:
        case kGammaPow: mult(0.0, D.p[3]); return;
        case kEmpiricalAbs:
        case kEmpiricalRel: {
            uint64_t packed;
            std::memcpy(&packed, &D.p[0], sizeof(double));
            const size_t n = (uint32_t)packed, off = (size_t)(uint32_t)(packed >> 32);
            double vmin = inf, vmax = -inf;
            bool nan = false;
            for (size_t b = 0; b < n; ++b) {  // a bin's own value needs prob > 0; its alias is always reachable
                const AliasRec &a = P.alias[off + b];
                for (int side = 0; side < 2; ++side) {
                    if (side == 0 && !(a.prob > 0.0)) continue;
                    const double v = side == 0 ? a.v_self : a.v_alias;
                    if (std::isnan(v)) nan = true;
                    vmin = std::min(vmin, v);
                    vmax = std::max(vmax, v);
                }
            }
            if (nan) return;
            if (D.kind == kEmpiricalAbs) {
                if (std::isfinite(d)) ends(d + vmin, d + vmax);
            } else if (std::isfinite(d)) {
                if (d == 0.0) {
                    if (std::isfinite(vmin) && std::isfinite(vmax)) lo = hi = rel(0.0);
                } else {
                    ends(rel(vmin), rel(vmax));
                }
            }
            return;
        }
        default: return;
    }
}

// Every event's realized time lies in [ev_lo[e], ev_hi[e]] for every seed:
// the walk's recurrence (upper = earliest + max_delay; per predecessor in
// input order t = min(upper, r_src + duration), best = t when t >= best;
// realized = min(upper, best); a stale predecessor reads its earliest time)
// over the per-link duration ranges, which it preserves because each step is
// monotone.  False when an earliest time or max_delay is not finite.
bool mcdp::event_ranges(const mcdp_propagator &P, std::vector<double> &ev_lo, std::vector<double> &ev_hi) {
    if (!std::isfinite(P.max_delay)) return false;
    for (double e : P.earliest)
        if (!std::isfinite(e)) return false;
    std::vector<double> dlo((size_t)P.L), dhi((size_t)P.L);
    for (int32_t l = 0; l < P.L; ++l) link_duration_range(P, l, dlo[(size_t)l], dhi[(size_t)l]);
    ev_lo.assign((size_t)P.E, 0.0);
    ev_hi.assign((size_t)P.E, 0.0);
    for (const auto &level : P.levels)
        for (int32_t e : level) {
            const double upper = P.earliest[(size_t)e] + P.max_delay;
            double blo = P.earliest[(size_t)e], bhi = blo;
            for (int64_t k = P.pred_off[(size_t)e]; k < P.pred_off[(size_t)e + 1]; ++k) {
                const PredEntry &pe = P.preds[(size_t)k];
                const bool valid = pe.edge >= 0 && pe.edge < P.L;
                const double rlo = pe.stale ? P.earliest[(size_t)pe.src] : ev_lo[(size_t)pe.src];
                const double rhi = pe.stale ? P.earliest[(size_t)pe.src] : ev_hi[(size_t)pe.src];
                double tlo = rlo + (valid ? dlo[(size_t)pe.edge] : 0.0);
                double thi = rhi + (valid ? dhi[(size_t)pe.edge] : 0.0);
                tlo = (upper < tlo) ? upper : tlo;
                thi = (upper < thi) ? upper : thi;
                if (tlo >= blo) blo = tlo;
                if (thi >= bhi) bhi = thi;
            }
            ev_lo[(size_t)e] = (upper < blo) ? upper : blo;
            ev_hi[(size_t)e] = (upper < bhi) ? upper : bhi;
        }
    return true;
}

// ============================================================================
// C ABI
// ============================================================================
extern "C" {

const char *mcdp_last_error(void) { return g_last_error.c_str(); }
int mcdp_abi_version(void) { return MCDP_ABI_VERSION; }

int mcdp_generator_create(mcdp_generator **out) {
    if (!out) return fail(MCDP_E_INVALID, "out is null");
    *out = new (std::nothrow) mcdp_generator();
    return *out ? MCDP_OK : fail(MCDP_E_NOMEM, "out of host memory");
}
void mcdp_generator_destroy(mcdp_generator *gen) { delete gen; }
int mcdp_generator_set_seed(mcdp_generator *gen, int32_t) {
    return gen ? MCDP_OK : fail(MCDP_E_INVALID, "generator is null");
}
int mcdp_generator_add_constant(mcdp_generator *gen, int32_t t, double factor) {
    if (!gen) return fail(MCDP_E_INVALID, "generator is null");
    DistSpec s;
    s.kind = kApiConstant;
    s.a = factor;
    gen->dists[t] = s;
    return MCDP_OK;
}
int mcdp_generator_add_exponential(mcdp_generator *gen, int32_t t, double lambda_, double max_scale) {
    if (!gen) return fail(MCDP_E_INVALID, "generator is null");
    DistSpec s;
    s.kind = kApiExponential;
    s.a = lambda_;
    s.b = max_scale;
    gen->dists[t] = s;
    return MCDP_OK;
}
int mcdp_generator_add_gamma(mcdp_generator *gen, int32_t t, double shape, double scale, double max_scale) {
    if (!gen) return fail(MCDP_E_INVALID, "generator is null");
    DistSpec s;
    s.kind = kApiGamma;
    s.a = shape;
    s.b = scale;
    s.c = max_scale;
    gen->dists[t] = s;
    return MCDP_OK;
}
static int add_empirical(mcdp_generator *gen, int32_t t, const double *v, const double *w, int64_t n, ApiKind k) {
    if (!gen) return fail(MCDP_E_INVALID, "generator is null");
    if (n < 0 || (n > 0 && (!v || !w))) return fail(MCDP_E_INVALID, "invalid empirical table");
    DistSpec s;
    s.kind = k;
    s.values.assign(v, v + n);
    s.weights.assign(w, w + n);
    gen->dists[t] = std::move(s);
    return MCDP_OK;
}
int mcdp_generator_add_empirical_absolute(mcdp_generator *gen, int32_t t, const double *values, const double *weights,
                                          int64_t n) {
    return add_empirical(gen, t, values, weights, n, kApiEmpAbs);
}
int mcdp_generator_add_empirical_relative(mcdp_generator *gen, int32_t t, const double *factors,
                                          const double *weights, int64_t n) {
    return add_empirical(gen, t, factors, weights, n, kApiEmpRel);
}

int mcdp_propagator_create(int32_t n_events, const double *earliest, int32_t n_activities,
                           const int32_t *activity_idx, const double *minimal_duration,
                           const int32_t *activity_type, int32_t n_entries, const int32_t *entry_target,
                           const int64_t *entry_offsets, const int32_t *pred_event, const int32_t *pred_activity,
                           double max_delay, const mcdp_generator *gen, mcdp_propagator **out) {
    if (!out) return fail(MCDP_E_INVALID, "out is null");
    *out = nullptr;
    if (!gen) return fail(MCDP_E_INVALID, "generator is null");
    if ((n_events > 0 && !earliest) || (n_activities > 0 && (!activity_idx || !minimal_duration || !activity_type)) ||
        (n_entries > 0 && (!entry_target || !entry_offsets)) ||
        (n_entries > 0 && entry_offsets[n_entries] > 0 && (!pred_event || !pred_activity)))
        return fail(MCDP_E_INVALID, "null input array");
    try {
        std::unique_ptr<mcdp_propagator> P(new mcdp_propagator());
        int rc = compile_propagator(*P, n_events, earliest, n_activities, activity_idx, minimal_duration,
                                    activity_type, n_entries, entry_target, entry_offsets, pred_event,
                                    pred_activity, max_delay, *gen);
        if (rc) return rc;
        *out = P.release();
        return MCDP_OK;
    } catch (const std::bad_alloc &) {
        return fail(MCDP_E_NOMEM, "out of host memory");
    }
}
void mcdp_propagator_destroy(mcdp_propagator *prop) { delete prop; }
int32_t mcdp_propagator_node_count(const mcdp_propagator *prop) { return prop ? prop->E : -1; }
int32_t mcdp_propagator_activity_count(const mcdp_propagator *prop) { return prop ? prop->L : -1; }

int mcdp_run_many_device(mcdp_propagator *prop, const int32_t *seeds_dev, int64_t n, int64_t ld,
                         double *realized_dev, double *durations_dev, int32_t *cause_dev, void *stream) {
    if (!prop) return fail(MCDP_E_INVALID, "propagator is null");
    return launch(*prop, false, seeds_dev, nullptr, n, ld, realized_dev, durations_dev, cause_dev,
                  static_cast<hipStream_t>(stream));
}
int mcdp_propagate_device(mcdp_propagator *prop, const double *durations_dev, int64_t n, int64_t ld,
                          double *realized_dev, int32_t *cause_dev, void *stream) {
    if (!prop) return fail(MCDP_E_INVALID, "propagator is null");
    return launch(*prop, true, nullptr, durations_dev, n, ld, realized_dev, nullptr, cause_dev,
                  static_cast<hipStream_t>(stream));
}
int mcdp_run_many_host(mcdp_propagator *prop, const int32_t *seeds, int64_t n, double *realized, double *durations,
                       int32_t *cause) {
    if (!prop) return fail(MCDP_E_INVALID, "propagator is null");
    if (n > 0 && !seeds) return fail(MCDP_E_INVALID, "seeds is null");
    return run_host(*prop, false, seeds, nullptr, n, realized, durations, cause);
}
int mcdp_propagate_host(mcdp_propagator *prop, const double *durations, int64_t n, double *realized,
                        int32_t *cause) {
    if (!prop) return fail(MCDP_E_INVALID, "propagator is null");
    if (n > 0 && prop->L > 0 && !durations) return fail(MCDP_E_INVALID, "durations is null");
    return run_host(*prop, true, nullptr, durations, n, realized, nullptr, cause);
}

int mcdp_propagator_plan_info(const mcdp_propagator *prop, int64_t *out, int n_out) {
    if (!prop || !out) return fail(MCDP_E_INVALID, "null argument");
    const int64_t v[12] = {prop->n_steps,
                          prop->waves,
                          prop->slots,
                          (int64_t)prop->slots * kLanes * prop->spl * (int64_t)sizeof(double),
                          prop->n_global,
                          prop->n_stale,
                          (int64_t)prop->orph.size(),
                          prop->max_per_wave,
                          prop->k,
                          prop->spl,
                          prop->tile_cost,
                          prop->wide_cost};
    for (int i = 0; i < n_out && i < 12; ++i) out[i] = v[i];
    return MCDP_OK;
}

int mcdp_propagator_ranges(const mcdp_propagator *prop, double *link_lo, double *link_hi, double *event_lo,
                           double *event_hi) {
    if (!prop) return fail(MCDP_E_INVALID, "propagator is null");
    for (int32_t l = 0; l < prop->L; ++l) {
        double lo, hi;
        link_duration_range(*prop, l, lo, hi);
        if (link_lo) link_lo[l] = lo;
        if (link_hi) link_hi[l] = hi;
    }
    if (!event_lo && !event_hi) return MCDP_OK;
    std::vector<double> elo, ehi;
    if (!event_ranges(*prop, elo, ehi))
        return fail(MCDP_E_INVALID, "event ranges need finite earliest times and a finite max_delay");
    if (event_lo) std::copy(elo.begin(), elo.end(), event_lo);
    if (event_hi) std::copy(ehi.begin(), ehi.end(), event_hi);
    return MCDP_OK;
}

}  // extern "C"

int mcdp::configure_shape(mcdp_propagator *prop, int32_t waves, int32_t events_per_wave, int32_t samples_per_lane,
                          bool by_caller) {
    if (!prop) return fail(MCDP_E_INVALID, "propagator is null");
    if (!shape_valid(waves, events_per_wave, samples_per_lane))
        return fail(MCDP_E_INVALID,
                    "invalid shape: waves in [1, 16], events_per_wave in {4, 8, 12, 16}, samples_per_lane 1 or 2 "
                    "(with events_per_wave <= 8)");
    std::lock_guard<std::mutex> lock(prop->mu);
    int rc = build_schedule(*prop, waves, events_per_wave);
    if (rc) return rc;
    prop->spl = samples_per_lane;
    prop->drop_device_copies();
    prop->shape_fixed = true;
    prop->shape_by_caller = by_caller;
    return MCDP_OK;
}

extern "C" {

int mcdp_propagator_configure(mcdp_propagator *prop, int32_t waves, int32_t events_per_wave,
                              int32_t samples_per_lane) {
    return configure_shape(prop, waves, events_per_wave, samples_per_lane, true);
}

int mcdp_propagator_autotune(mcdp_propagator *prop, int64_t n_samples, int32_t *waves, int32_t *events_per_wave,
                             int32_t *samples_per_lane, float *ms) {
    if (!prop) return fail(MCDP_E_INVALID, "propagator is null");
    if (n_samples < 1) return fail(MCDP_E_INVALID, "n_samples must be positive");
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0) return fail(MCDP_E_DEVICE, "no HIP device available");
    const int64_t n = n_samples, E = prop->E, L = prop->L;
    std::vector<int32_t> hseeds((size_t)n);
    for (int64_t i = 0; i < n; ++i) hseeds[(size_t)i] = (int32_t)i;
    void *buf = nullptr;
    const size_t bytes = align_up((size_t)n * 4, 256) + (size_t)n * (size_t)(12 * E + 8 * L);
    hipError_t e = device_malloc(&buf, bytes);
    if (e != hipSuccess) return fail(MCDP_E_NOMEM, std::string("hipMalloc (autotune): ") + hipGetErrorString(e));
    auto *b = static_cast<unsigned char *>(buf);
    int32_t *d_seeds = reinterpret_cast<int32_t *>(b);
    double *d_real = reinterpret_cast<double *>(b + align_up((size_t)n * 4, 256));
    double *d_dur = d_real + (size_t)(E * n);
    int32_t *d_cause = reinterpret_cast<int32_t *>(d_dur + (size_t)(L * n));
    hipEvent_t t0 = nullptr, t1 = nullptr;
    int rc = MCDP_OK;
    float best_ms = -1.0f;
    Shape best{prop->waves, prop->k, prop->spl};
    std::vector<Shape> cands;
    {
        std::lock_guard<std::mutex> lock(prop->mu);
        cands = shape_candidates(*prop);
    }
    e = hipMemcpy(d_seeds, hseeds.data(), (size_t)n * 4, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipEventCreate(&t0);
    if (e == hipSuccess) e = hipEventCreate(&t1);
    if (e != hipSuccess) rc = hip_fail(e, "autotune setup");
    for (size_t c = 0; rc == MCDP_OK && c < cands.size(); ++c) {
        rc = configure_shape(prop, cands[c].waves, cands[c].k, cands[c].spl, true);  // time the walk, not the two passes
        if (rc) break;
        {  // skip shapes that cannot be resident
            std::lock_guard<std::mutex> lock(prop->mu);
            const WalkVariant v = walk_variant(*prop, false);
            int bpc = 0;
            if (walk_occupancy(v, prop->waves, walk_lds_bytes(*prop, v), &bpc) != hipSuccess || bpc < 1) continue;
        }
        rc = launch(*prop, false, d_seeds, nullptr, n, n, d_real, d_dur, d_cause, nullptr);  // warm-up + upload
        if (rc) break;
        if ((e = hipEventRecord(t0, nullptr)) != hipSuccess) {
            rc = hip_fail(e, "hipEventRecord");
            break;
        }
        rc = launch(*prop, false, d_seeds, nullptr, n, n, d_real, d_dur, d_cause, nullptr);
        if (rc) break;
        float t = 0.0f;
        if ((e = hipEventRecord(t1, nullptr)) != hipSuccess || (e = hipEventSynchronize(t1)) != hipSuccess ||
            (e = hipEventElapsedTime(&t, t0, t1)) != hipSuccess) {
            rc = hip_fail(e, "autotune timing");
            break;
        }
        if (best_ms < 0.0f || t < best_ms) {
            best_ms = t;
            best = cands[c];
        }
    }
    if (t0) (void)hipEventDestroy(t0);
    if (t1) (void)hipEventDestroy(t1);
    (void)hipFree(buf);
    if (rc) {
        std::lock_guard<std::mutex> lock(prop->mu);
        prop->shape_by_caller = false;
        return rc;
    }
    rc = configure_shape(prop, best.waves, best.k, best.spl, false);
    if (rc) return rc;
    if (waves) *waves = best.waves;
    if (events_per_wave) *events_per_wave = best.k;
    if (samples_per_lane) *samples_per_lane = best.spl;
    if (ms) *ms = best_ms;
    return MCDP_OK;
}

// What a schedule shape's speed depends on: the precedence structure (events,
// links, every entry's source, edge and stale flag), which distribution each
// link draws from and each distribution's kind and flags (the code path of a
// draw), and the alias tables' size (LDS).  Times and distribution
// parameters are left out.  FNV-1a, 64 bits, over those values' bytes.
static uint64_t shape_fingerprint(const mcdp_propagator &P) {
    uint64_t h = 0xcbf29ce484222325ull;
    auto mix = [&](const void *data, size_t n) {
        const auto *b = static_cast<const unsigned char *>(data);
        for (size_t i = 0; i < n; ++i) {
            h ^= b[i];
            h *= 0x100000001b3ull;
        }
    };
    auto mix64 = [&](int64_t v) { mix(&v, sizeof v); };
    mix("mcdp-shape-1", 12);
    mix64(P.E);
    mix64(P.L);
    for (int64_t o : P.pred_off) mix64(o);
    for (const PredEntry &pe : P.preds) {
        mix64(pe.src);
        mix64(pe.edge);
        mix64(pe.stale ? 1 : 0);
    }
    for (uint32_t d : P.ldist) mix64(d);
    for (const DistRec &d : P.dist) {
        mix64(d.kind);
        mix64(d.flags);
    }
    mix64((int64_t)P.alias.size());
    return h;
}

int mcdp_propagator_fingerprint(const mcdp_propagator *prop, uint64_t *fingerprint) {
    if (!prop || !fingerprint) return fail(MCDP_E_INVALID, "propagator or fingerprint is null");
    *fingerprint = shape_fingerprint(*prop);
    return MCDP_OK;
}

int mcdp_propagator_autotune_cached(mcdp_propagator *prop, int64_t n_samples, const char *path, int32_t *waves,
                                    int32_t *events_per_wave, int32_t *samples_per_lane, float *ms,
                                    int32_t *from_file) {
    if (!prop) return fail(MCDP_E_INVALID, "propagator is null");
    if (!path || !*path) return fail(MCDP_E_INVALID, "tuning file path is empty");
    if (n_samples < 1) return fail(MCDP_E_INVALID, "n_samples must be positive");
    int dev = 0;
    hipDeviceProp_t props{};
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&props, dev) != hipSuccess)
        return fail(MCDP_E_DEVICE, "no HIP device available");
    // the device kind: architecture name up to its first ':' or space, and compute units
    std::string arch(props.gcnArchName);
    arch = arch.substr(0, arch.find_first_of(": "));
    if (arch.empty()) arch = "unknown";
    int64_t bucket = 1;
    while (bucket < n_samples) bucket *= 2;
    if (arch.size() > 64) arch.resize(64);
    char key[160];
    std::snprintf(key, sizeof key, "mcdp-shape 1 %016" PRIx64 " %s %d %" PRId64, shape_fingerprint(*prop), arch.c_str(),
                  props.multiProcessorCount, bucket);
    const std::string prefix = std::string(key) + " ";

    // the last valid line for this key wins (a later tuning appends a newer choice)
    bool found = false;
    Shape got{0, 0, 0};
    float got_ms = 0.0f;
    {
        std::ifstream in(path);
        std::string line;
        while (in && std::getline(in, line)) {
            if (line.compare(0, prefix.size(), prefix) != 0) continue;
            std::istringstream rest(line.substr(prefix.size()));
            Shape c{0, 0, 0};
            float t = 0.0f;
            if (!(rest >> c.waves >> c.k >> c.spl >> t) || !shape_valid(c.waves, c.k, c.spl)) continue;
            found = true;
            got = c;
            got_ms = t;
        }
    }
    if (found) {
        int rc = configure_shape(prop, got.waves, got.k, got.spl, false);
        if (rc) return rc;
        bool resident = false;
        {
            std::lock_guard<std::mutex> lock(prop->mu);
            const WalkVariant v = walk_variant(*prop, false);
            int bpc = 0;
            resident = walk_occupancy(v, prop->waves, walk_lds_bytes(*prop, v), &bpc) == hipSuccess && bpc >= 1;
        }
        if (resident) {
            if (waves) *waves = got.waves;
            if (events_per_wave) *events_per_wave = got.k;
            if (samples_per_lane) *samples_per_lane = got.spl;
            if (ms) *ms = got_ms;
            if (from_file) *from_file = 1;
            return MCDP_OK;
        }
    }
    int32_t w = 0, k = 0, spl = 0;
    float t = 0.0f;
    int rc = mcdp_propagator_autotune(prop, n_samples, &w, &k, &spl, &t);
    if (rc) return rc;
    if (waves) *waves = w;
    if (events_per_wave) *events_per_wave = k;
    if (samples_per_lane) *samples_per_lane = spl;
    if (ms) *ms = t;
    if (from_file) *from_file = 0;
    // one write of the whole line to a file opened for appending: concurrent
    // tunings add whole lines
    char line[256];
    const int len = std::snprintf(line, sizeof line, "%s%d %d %d %.6f\n", prefix.c_str(), w, k, spl, (double)t);
    if (len <= 0 || (size_t)len >= sizeof line) return fail(MCDP_E_INVALID, "tuning file line too long");
    const int fd = ::open(path, O_WRONLY | O_APPEND | O_CREAT | O_CLOEXEC, 0644);
    if (fd < 0) return fail(MCDP_E_INVALID, std::string("cannot open tuning file ") + path + ": " + std::strerror(errno));
    const ssize_t wr = ::write(fd, line, (size_t)len);
    const int werr = errno;
    ::close(fd);
    if (wr != (ssize_t)len)
        return fail(MCDP_E_INVALID, std::string("cannot write tuning file ") + path + ": " + std::strerror(werr));
    return MCDP_OK;
}

int mcdp_debug_tail_mode(mcdp_propagator *prop, int32_t mode) {
    if (!prop) return fail(MCDP_E_INVALID, "propagator is null");
    if (mode < 0 || mode > 2) return fail(MCDP_E_INVALID, "tail mode must be 0, 1 or 2");
    std::lock_guard<std::mutex> lock(prop->mu);
    prop->tail_mode = mode;
    return MCDP_OK;
}

int mcdp_debug_two_pass_mode(mcdp_propagator *prop, int32_t mode) {
    if (!prop) return fail(MCDP_E_INVALID, "propagator is null");
    if (mode < 0 || mode > 2) return fail(MCDP_E_INVALID, "two-pass mode must be 0, 1 or 2");
    std::lock_guard<std::mutex> lock(prop->mu);
    prop->two_pass_mode = mode;
    return MCDP_OK;
}

int mcdp_debug_last_route(mcdp_propagator *prop, int32_t *route) {
    if (!prop || !route) return fail(MCDP_E_INVALID, "null argument");
    std::lock_guard<std::mutex> lock(prop->mu);
    *route = prop->last_route;
    return MCDP_OK;
}

int mcdp_debug_short_run(mcdp_propagator *prop, int32_t injected, int64_t n, int32_t *two_pass) {
    if (!prop || !two_pass) return fail(MCDP_E_INVALID, "null argument");
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0) return fail(MCDP_E_DEVICE, "no HIP device available");
    bool yes = false;
    const int rc = short_run(*prop, injected != 0, n, yes);
    *two_pass = yes ? 1 : 0;
    return rc;
}

// ---- device plumbing --------------------------------------------------------
int mcdp_device_count(int *count) {
    if (!count) return fail(MCDP_E_INVALID, "count is null");
    *count = 0;
    hipError_t e = hipGetDeviceCount(count);
    if (e != hipSuccess) *count = 0;
    return MCDP_OK;
}
int mcdp_release_workspaces(void) {
    (void)large_pool().drop([](const LargePool::Entry &) { return true; });
    return MCDP_OK;
}
int mcdp_malloc(void **ptr, size_t bytes) {
    if (!ptr) return fail(MCDP_E_INVALID, "ptr is null");
    hipError_t e = device_malloc(ptr, bytes);
    return e == hipSuccess ? MCDP_OK : fail(MCDP_E_NOMEM, std::string("hipMalloc: ") + hipGetErrorString(e));
}
int mcdp_free(void *ptr) {
    HIP_TRY(hipFree(ptr), "hipFree");
    return MCDP_OK;
}
int mcdp_memcpy_htod(void *dst, const void *src, size_t bytes) {
    HIP_TRY(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice), "hipMemcpy HtoD");
    return MCDP_OK;
}
int mcdp_memcpy_dtoh(void *dst, const void *src, size_t bytes) {
    HIP_TRY(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost), "hipMemcpy DtoH");
    return MCDP_OK;
}
int mcdp_memset(void *dst, int value, size_t bytes) {
    HIP_TRY(hipMemset(dst, value, bytes), "hipMemset");
    return MCDP_OK;
}
int mcdp_memcpy2d_dtoh(void *dst, size_t dst_pitch, const void *src, size_t src_pitch, size_t width,
                       size_t height) {
    HIP_TRY(hipMemcpy2D(dst, dst_pitch, src, src_pitch, width, height, hipMemcpyDeviceToHost), "hipMemcpy2D DtoH");
    return MCDP_OK;
}
int mcdp_graph_capture_begin(void *stream) {
    HIP_TRY(hipStreamBeginCapture(static_cast<hipStream_t>(stream), hipStreamCaptureModeGlobal),
            "hipStreamBeginCapture");
    return MCDP_OK;
}
int mcdp_graph_capture_end(void *stream, void **graph_exec) {
    if (!graph_exec) return fail(MCDP_E_INVALID, "graph_exec is null");
    *graph_exec = nullptr;
    hipGraph_t g = nullptr;
    HIP_TRY(hipStreamEndCapture(static_cast<hipStream_t>(stream), &g), "hipStreamEndCapture");
    hipGraphExec_t x = nullptr;
    hipError_t e = hipGraphInstantiate(&x, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e != hipSuccess) return hip_fail(e, "hipGraphInstantiate");
    *graph_exec = x;
    return MCDP_OK;
}
int mcdp_graph_launch(void *graph_exec, void *stream) {
    if (!graph_exec) return fail(MCDP_E_INVALID, "graph_exec is null");
    HIP_TRY(hipGraphLaunch(static_cast<hipGraphExec_t>(graph_exec), static_cast<hipStream_t>(stream)),
            "hipGraphLaunch");
    return MCDP_OK;
}
int mcdp_graph_destroy(void *graph_exec) {
    if (graph_exec) HIP_TRY(hipGraphExecDestroy(static_cast<hipGraphExec_t>(graph_exec)), "hipGraphExecDestroy");
    return MCDP_OK;
}
int mcdp_stream_create(void **stream) {
    if (!stream) return fail(MCDP_E_INVALID, "stream is null");
    hipStream_t s = nullptr;
    HIP_TRY(hipStreamCreate(&s), "hipStreamCreate");
    *stream = s;
    return MCDP_OK;
}
int mcdp_stream_destroy(void *stream) {
    HIP_TRY(hipStreamDestroy(static_cast<hipStream_t>(stream)), "hipStreamDestroy");
    return MCDP_OK;
}
int mcdp_stream_synchronize(void *stream) {
    HIP_TRY(hipStreamSynchronize(static_cast<hipStream_t>(stream)), "hipStreamSynchronize");
    return MCDP_OK;
}
int mcdp_event_create(void **event) {
    if (!event) return fail(MCDP_E_INVALID, "event is null");
    hipEvent_t e = nullptr;
    HIP_TRY(hipEventCreate(&e), "hipEventCreate");
    *event = e;
    return MCDP_OK;
}
int mcdp_event_destroy(void *event) {
    HIP_TRY(hipEventDestroy(static_cast<hipEvent_t>(event)), "hipEventDestroy");
    return MCDP_OK;
}
int mcdp_event_record(void *event, void *stream) {
    HIP_TRY(hipEventRecord(static_cast<hipEvent_t>(event), static_cast<hipStream_t>(stream)), "hipEventRecord");
    return MCDP_OK;
}
int mcdp_event_elapsed_ms(void *start, void *stop, float *ms) {
    if (!ms) return fail(MCDP_E_INVALID, "ms is null");
    HIP_TRY(hipEventElapsedTime(ms, static_cast<hipEvent_t>(start), static_cast<hipEvent_t>(stop)),
            "hipEventElapsedTime");
    return MCDP_OK;
}

int mcdp_debug_copy(double *dst, const double *src, int64_t n, void *stream) {
    if (n < 0 || (n > 0 && (!dst || !src))) return fail(MCDP_E_INVALID, "invalid arguments");
    HIP_TRY(launch_copy(dst, src, n, static_cast<hipStream_t>(stream)), "copy kernel launch");
    return MCDP_OK;
}

int mcdp_debug_philox(int variant, int64_t n, const uint32_t *ctr, const uint32_t *key, uint32_t *out) {
    if (variant != 2 && variant != 4) return fail(MCDP_E_INVALID, "variant must be 2 or 4");
    if (n < 0 || (n > 0 && (!ctr || !key || !out))) return fail(MCDP_E_INVALID, "invalid arguments");
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0) return fail(MCDP_E_DEVICE, "no HIP device available");
    if (n == 0) return MCDP_OK;
    const size_t cw = (size_t)variant, kw = (size_t)(variant / 2);
    uint32_t *d = nullptr;
    const size_t bytes = sizeof(uint32_t) * (size_t)n * (cw + kw + cw);
    HIP_TRY(device_malloc((void **)&d, bytes), "hipMalloc");
    uint32_t *dc = d, *dk = d + (size_t)n * cw, *dout = dk + (size_t)n * kw;
    hipError_t e = hipMemcpy(dc, ctr, sizeof(uint32_t) * n * cw, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dk, key, sizeof(uint32_t) * n * kw, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = launch_philox_debug(variant, n, dc, dk, dout, nullptr);
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e == hipSuccess) e = hipMemcpy(out, dout, sizeof(uint32_t) * n * cw, hipMemcpyDeviceToHost);
    (void)hipFree(d);
    if (e != hipSuccess) return hip_fail(e, "philox debug");
    return MCDP_OK;
}

int mcdp_debug_math(int fn, int64_t n, const double *x, double *out) {
    if (fn < 0 || fn > 2) return fail(MCDP_E_INVALID, "fn must be 0 (log), 1 (cos2pi) or 2 (exp)");
    if (n < 0 || (n > 0 && (!x || !out))) return fail(MCDP_E_INVALID, "invalid arguments");
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0) return fail(MCDP_E_DEVICE, "no HIP device available");
    if (n == 0) return MCDP_OK;
    double *d = nullptr;
    HIP_TRY(device_malloc((void **)&d, sizeof(double) * 2 * (size_t)n), "hipMalloc");
    hipError_t e = hipMemcpy(d, x, sizeof(double) * n, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = launch_math_debug(fn, n, d, d + n, nullptr);
    if (e == hipSuccess) e = hipDeviceSynchronize();
    if (e == hipSuccess) e = hipMemcpy(out, d + n, sizeof(double) * n, hipMemcpyDeviceToHost);
    (void)hipFree(d);
    if (e != hipSuccess) return hip_fail(e, "math debug");
    return MCDP_OK;
}

}  // extern "C"
