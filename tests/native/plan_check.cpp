// Checks of a plan's sizes and of what its searches launch, built with g++
// against the HIP runtime stand-in (hipstub).  One check per run, named by the
// first argument; exit status 0 when it holds.  Test infrastructure only.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "pzl_accel.h"
#include "pzl_geom.h"
#include "pzl_math.h"
#include "pzl_plan.h"

namespace {

int bad = 0;

#define EXPECT(cond, ...)                                     \
    do {                                                      \
        if (!(cond)) {                                        \
            bad++;                                            \
            fprintf(stderr, "line %d: %s: ", __LINE__, #cond); \
            fprintf(stderr, __VA_ARGS__);                     \
            fprintf(stderr, "\n");                            \
        }                                                     \
    } while (0)

PzlConfig config(double N, int zmax, int wmax, int numharm, int batchsize)
{
    PzlConfig c;
    memset(&c, 0, sizeof c);
    c.N = N;
    c.dt = 1e-4;
    c.numbins = (long long)N / 2;
    c.zmax = zmax;
    c.wmax = wmax;
    c.wmaxP = wmax > 0;
    c.numharm = numharm;
    c.sigma = 3.0f;
    c.floP = 1;
    c.flo = 1.0;
    c.fhiP = 1;
    c.fhi = 1e4;
    c.batchsize = batchsize;
    return c;
}

void ok(int rc)
{
    if (rc == 0) return;
    fprintf(stderr, "call failed: %s\n", pzl_last_error());
    exit(2);
}

struct Plan {
    void *h = nullptr;
    PzlConfig c;
    Plan(const PzlConfig &cfg, int launch = 0) : c(cfg)
    {
        ok(pzl_plan_create_launch(&c, 0, launch, &h));
        ok(pzl_set_spectrum_device(h, spectrum().data(), c.numbins));
    }
    ~Plan() { pzl_plan_destroy(h); }
    static std::vector<float> &spectrum()
    {
        static std::vector<float> f(1 << 22, 1.0f);
        return f;
    }
    int launch() const
    {
        int n = 0;
        ok(pzl_plan_launch(h, &n, nullptr));
        return n;
    }
    int asked() const
    {
        int n = 0;
        ok(pzl_plan_launch(h, nullptr, &n));
        return n;
    }
    std::vector<PzlCand> search(PzlStats *st = nullptr)
    {
        long long n = 0;
        ok(pzl_search(h, 0, -1, nullptr, 0, &n, st));
        return cands(n);
    }
    std::vector<PzlCand> cands(long long n)
    {
        std::vector<PzlCand> v((size_t)n);
        ok(pzl_get_cands(h, v.data(), n, &n));
        return v;
    }
};

bool same(const std::vector<PzlCand> &a, const std::vector<PzlCand> &b)
{
    if (a.size() != b.size()) return false;
    for (size_t i = 0; i < a.size(); i++)
        if (a[i].power != b[i].power || a[i].sigma != b[i].sigma || a[i].numharm != b[i].numharm ||
            a[i].r != b[i].r || a[i].z != b[i].z || a[i].w != b[i].w)
            return false;
    return true;
}

// A plan of a given launch size launches by it, holds what the model says, and
// gives the same candidates as any other.
void exact()
{
    const PzlConfig c = config(1 << 18, 8, 0, 2, 8);
    std::vector<PzlCand> ref;
    PzlGeometry g;
    ok(pzl_geometry_from_config(&c, &g));
    for (int b : {1, 3, 8, 20, 1 << 20}) {
        const int want = (int)std::min<long long>(b, g.nrsteps);
        Plan p(c, b);
        EXPECT(p.launch() == want && p.asked() == std::min(want, 8), "%d: %d, %d", b, p.launch(), p.asked());
        PzlStats st;
        const auto v = p.search(&st);
        EXPECT(st.corr_launches == (g.nrsteps + want - 1) / want, "%d: %lld launches", b, st.corr_launches);
        if (ref.empty()) ref = v;
        EXPECT(!v.empty() && same(v, ref), "%d: %zu candidates", b, v.size());
        PzlGeometry gl;
        ok(pzl_geometry_launch(&c, b, &gl));
        long long held = 0;
        ok(pzl_plan_device_bytes(p.h, &held));
        EXPECT(held + (long long)sizeof(float2) * c.numbins == gl.device_bytes, "%d: %lld, model %lld", b, held,
               gl.device_bytes);  // the spectrum is the caller's
    }
    Plan p(c);
    EXPECT(p.launch() > 8 && p.asked() == 8 && same(p.search(), ref), "%d", p.launch());
}

// The rule's launch sizes: within their limits on the bytes of planes, 1 as
// asked, and fewer than the default of 8 raised only while the planes are small.
void rule()
{
    struct Shape {
        double N;
        int zmax, wmax, numharm;
        std::vector<std::pair<int, int>> want;  // asked, launched
    };
    const std::vector<Shape> shapes = {
        {1 << 20, 20, 0, 4, {{8, 512}, {3, 192}, {700, 700}}},       // 0.3 MiB, 540 rsteps
        {1 << 21, 50, 0, 8, {{0, 256}, {8, 256}, {4, 256}}},         // 1.2 MiB
        {1 << 18, 200, 300, 8, {{8, 32}, {4, 4}, {2, 4}, {64, 64}}}, // 88 MiB
        {1 << 22, 200, 300, 16, {{8, 16}, {16, 16}, {7, 7}, {2, 2}}}, // 157 MiB
        {1 << 20, 200, 500, 16, {{8, 8}, {2, 2}}},                   // 612 MiB
    };
    for (const Shape &s : shapes) {
        auto made = [&](int asked, long long *planes, long long *nr) {
            const PzlConfig c = config(s.N, s.zmax, s.wmax, s.numharm, asked);
            Plan p(c);
            PzlGeometry g;
            ok(pzl_plan_geometry(p.h, &g));
            *planes = p.launch() * g.plane_bytes_per_rstep;
            *nr = g.nrsteps;
            return p.launch();
        };
        long long planes, nr;
        for (auto w : s.want) {
            const int n = made(w.first, &planes, &nr);
            EXPECT(n == std::min<long long>(w.second, nr), "(%d, %d, %d) at %d: %d", s.zmax, s.wmax, s.numharm, w.first, n);
        }
        PzlGeometry g;
        const PzlConfig c = config(s.N, s.zmax, s.wmax, s.numharm, 8);
        ok(pzl_geometry_from_config(&c, &g));
        for (int asked : {1, 2, 3, 5, 7, 8, 12, 24, 40, 100}) {
            if (asked * g.plane_bytes_per_rstep > (5LL << 30)) break;  // what this machine's memory takes
            const int n = made(asked, &planes, &nr);
            const bool fits = planes <= (512LL << 20) || (asked >= 8 && planes <= (3LL << 30) && n < 64);
            EXPECT(n == std::min<long long>(asked, nr) || (asked > 1 && n > asked && n <= 512 && fits),
                   "(%d, %d, %d) at %d: %d, %lld bytes", s.zmax, s.wmax, s.numharm, asked, n, planes);
        }
    }
}

// Where the device's memory is short a plan is made at the size asked for, by what
// is reported free or after an allocation that failed.
void memory()
{
    const PzlConfig c = config(1 << 21, 50, 0, 8, 8);
    PzlGeometry full, least;
    ok(pzl_geometry_from_config(&c, &full));
    ok(pzl_geometry_launch(&c, 8, &least));
    EXPECT(full.device_bytes > 3 * least.device_bytes, "%lld, %lld", full.device_bytes, least.device_bytes);
    const long long all = 288LL << 30;
    std::vector<PzlCand> ref;
    const struct {
        long long reported, available;
        bool raised;
    } cases[] = {{all, all, true},
                 {4 * full.device_bytes, all, true},
                 {4 * full.device_bytes - 1, all, false},
                 {all, full.device_bytes / 2, false},
                 {least.device_bytes, least.device_bytes, false}};
    for (auto &k : cases) {
        ok(pzl_bank_cache_clear());
        hipstub_set_memory(k.reported, k.available);
        Plan p(c);
        EXPECT(p.asked() == 8 && (p.launch() > 8) == k.raised, "%lld, %lld: %d", k.reported, k.available, p.launch());
        const auto v = p.search();
        if (ref.empty()) ref = v;
        EXPECT(!v.empty() && same(v, ref), "%zu candidates", v.size());
        EXPECT(pzl_last_error()[0] == 0, "%s", pzl_last_error());
    }
    ok(pzl_bank_cache_clear());
    hipstub_set_memory(all, least.device_bytes / 2);
    void *h = nullptr;
    EXPECT(pzl_plan_create(&c, 0, &h) == PZL_ERR_HIP && !h, "%p", h);
    hipstub_set_memory(all, all);
    EXPECT(hipstub_device_bytes() == 0, "%lld bytes held", hipstub_device_bytes());
}

// A request's footprint: raised where the budget allows, else as asked, and
// refused only where that does not fit.
void server()
{
    const PzlConfig small = config(1 << 21, 50, 0, 8, 8), large = config(1 << 18, 200, 300, 8, 8);
    struct Case {
        const PzlConfig *c;
        int launch, inflight;  // the budget: inflight such footprints
        int want;              // rsteps per launch that the request gets, 0: refused
        long long less;        // ... less this many bytes
    };
    const Case cases[] = {{&small, 0, 1, 256, 0}, {&small, 0, 1, 8, 1}, {&small, 8, 1, 8, 0},   {&small, 8, 1, 0, 1},
                          {&small, 8, 2, 8, 0},   {&large, 0, 2, 32, 0}, {&large, 0, 2, 8, 1},  {&large, 8, 2, 8, 0},
                          {&large, 8, 1, 8, 0},   {&large, 8, 1, 0, 1}};
    for (const Case &k : cases) {
        PzlGeometry g, want;
        ok(pzl_geometry_launch(k.c, k.launch, &g));
        const long long budget = k.inflight * (g.device_bytes + PZL_RUNTIME_BYTES_PER_SEARCH) - k.less;
        void *srv = nullptr;
        ok(pzl_server_create(0, budget, k.inflight, &srv));
        long long id = 0, n = 0;
        const int rc = pzl_server_submit_device(srv, k.c, Plan::spectrum().data(), k.c->numbins, &id);
        EXPECT((rc != 0) == (k.want == 0), "budget %lld: %d", budget, rc);
        if (rc == 0 && k.want) {
            PzlRequestStats st;
            std::vector<PzlCand> v(1 << 16);
            ok(pzl_server_wait(srv, id, v.data(), (long long)v.size(), &n, &st));
            v.resize((size_t)n);
            ok(pzl_geometry_launch(k.c, k.want, &want));
            EXPECT(st.footprint == want.device_bytes + PZL_RUNTIME_BYTES_PER_SEARCH, "budget %lld: %lld, not %lld", budget,
                   st.footprint, want.device_bytes + PZL_RUNTIME_BYTES_PER_SEARCH);
            Plan p(*k.c, 8);
            EXPECT(n > 0 && same(v, p.search()), "%lld candidates", n);
        }
        pzl_server_destroy(srv);
        ok(pzl_bank_cache_clear());
    }
    // memory that others took meanwhile: the plan is made as asked
    PzlGeometry g;
    ok(pzl_geometry_from_config(&small, &g));
    hipstub_set_memory(288LL << 30, g.device_bytes / 2);
    void *srv = nullptr;
    ok(pzl_server_create(0, 8LL << 30, 1, &srv));
    long long id = 0, n = 0;
    ok(pzl_server_submit_device(srv, &small, Plan::spectrum().data(), small.numbins, &id));
    PzlRequestStats st;
    ok(pzl_server_wait(srv, id, nullptr, 0, &n, &st));
    EXPECT(n > 0, "%lld candidates", n);
    pzl_server_destroy(srv);
}

// Batches that overflow their hit slot, anywhere in a search: the same hits and
// candidates as with slots for every cell, and no more than the batches in flight
// launched twice, the search going on at the size asked for.
void overflow()
{
    const PzlConfig c = config(1 << 18, 8, 0, 2, 4);
    PzlGeometry g;
    ok(pzl_geometry_from_config(&c, &g));
    const long long n = g.nrsteps;
    const struct {
        long long lo, hi, every;
    } bursts[] = {{0, n, 8},           // a batch as asked fits, a raised one does not, throughout
                  {0, n, 2},           // nor does one as asked: one rstep at a time
                  {0, 3, 1},           // in the first batch
                  {n - 9, n, 2},       // in the last
                  {n / 2, n / 2 + 12, 3}, {-1, -1, 1}};
    auto hits = [&](Plan &p) {
        long long k = 0;
        ok(pzl_get_hits(p.h, nullptr, nullptr, 0, &k));
        std::vector<long long> keys((size_t)k);
        std::vector<float> pows((size_t)k);
        ok(pzl_get_hits(p.h, keys.data(), pows.data(), k, &k));
        return std::make_pair(keys, pows);
    };
    for (auto &b : bursts) {
        hipstub_set_burst(b.lo, b.hi, b.every);
        Plan all(c, 1);  // a slot for every cell of a batch
        PzlStats st;
        const auto want = all.search();
        const auto want_hits = hits(all);
        PzlConfig cs = c;
        cs.maxhits = 1;  // a slot for one rstep's
        Plan rule(cs), p(cs, 16), asked(cs, 4);
        EXPECT(rule.launch() == 64 && p.asked() == 4 && n > 7 * 16, "%d rsteps per launch of %lld", rule.launch(), n);
        for (Plan *q : {&p, &asked, &rule, &p}) {
            const long long s0 = hipstub_syncs();
            const auto v = q->search(&st);
            const long long syncs = hipstub_syncs() - s0;
            EXPECT(!v.empty() && same(v, want), "burst %lld..%lld: %zu candidates, %zu", b.lo, b.hi, v.size(), want.size());
            EXPECT(hits(*q) == want_hits, "burst %lld..%lld", b.lo, b.hi);
            EXPECT(st.corr_launches <= 4 + (n + 3) / 4, "burst %lld..%lld: %lld launches", b.lo, b.hi, st.corr_launches);
            // once for the batches dropped and once at the end, 5 streams each
            if (b.every == 8) EXPECT(syncs <= 10, "%lld waits", syncs);
        }
    }
    hipstub_set_burst(0, 0, 1);
}

// Near a deadline batches are launched as asked for, and one that has passed stops
// a search before its first batch; a far one and none change nothing.
void deadline()
{
    const PzlConfig c = config(1 << 18, 8, 0, 2, 4);
    Plan p(c);
    PzlGeometry g;
    ok(pzl_plan_geometry(p.h, &g));
    EXPECT(p.launch() >= g.nrsteps, "%d", p.launch());
    PzlStats st;
    const auto want = p.search(&st);
    EXPECT(!want.empty() && st.corr_launches == 1, "%lld launches", st.corr_launches);
    ok(pzl_plan_set_deadline(p.h, 1e7));
    EXPECT(same(p.search(&st), want) && st.corr_launches == 1, "%lld launches", st.corr_launches);
    int in_time = 0;
    for (int k = 0; k < 20; k++) {  // (a busy machine may miss some)
        ok(pzl_plan_set_deadline(p.h, 99.0));
        long long n = 0;
        const int rc = pzl_search(p.h, 0, -1, nullptr, 0, &n, &st);
        EXPECT(rc == 0 || rc == PZL_ERR_TIMEOUT, "%d", rc);
        if (rc) continue;
        in_time++;
        EXPECT(same(p.cands(n), want) && st.corr_launches == (g.nrsteps + 3) / 4, "%lld launches", st.corr_launches);
    }
    EXPECT(in_time > 0, "no search in time");
    ok(pzl_plan_set_deadline(p.h, 1e-6));
    long long n = 0;
    EXPECT(pzl_search(p.h, 0, -1, nullptr, 0, &n, nullptr) == PZL_ERR_TIMEOUT, "%lld candidates", n);
    ok(pzl_plan_set_deadline(p.h, 0));
    EXPECT(same(p.search(&st), want) && st.corr_launches == 1, "%lld launches", st.corr_launches);
}

// The batch-size tuner times each launch size once.
void tuner()
{
    const PzlConfig c = config(1 << 19, 20, 0, 4, 8);
    const int cand[] = {8, 2, 16, 1, 64, 8};
    double ms[6] = {};
    int best = 0;
    ok(pzl_tune_batchsize(&c, 0, Plan::spectrum().data(), c.numbins, cand, 6, 16, &best, ms));
    std::vector<int> launch;
    for (int b : cand) {
        PzlConfig k = c;
        k.batchsize = b;
        launch.push_back(Plan(k).launch());
    }
    EXPECT(launch[0] == launch[2] && launch[0] == launch[4] && launch[1] < launch[0], "%d, %d", launch[0], launch[1]);
    for (int i = 0; i < 6; i++) {
        EXPECT(ms[i] > 0, "%d: %g", cand[i], ms[i]);
        for (int j = 0; j < i; j++)
            EXPECT((ms[i] == ms[j]) == (launch[i] == launch[j]), "%d: %g ms, %d: %g", cand[i], ms[i], cand[j], ms[j]);
    }
    int first = 0;
    for (int i = 1; i < 6; i++)
        if (ms[i] < ms[first]) first = i;
    EXPECT(best == cand[first], "%d, not %d", best, cand[first]);
}

// A server pins nothing before its requests need it.
void pinned()
{
    hipstub_set_pinnable(0);
    void *srv = nullptr;
    EXPECT(pzl_server_create(0, 8LL << 30, 8, &srv) == 0, "%s", pzl_last_error());
    if (!srv) return;
    hipstub_set_pinnable(8 << 20);  // a small buffer and the counts, not a whole chunk of 32 MiB
    const PzlConfig c = config(1 << 18, 8, 0, 2, 4);
    long long id = 0, n = 0;
    PzlRequestStats st;
    ok(pzl_server_submit_device(srv, &c, Plan::spectrum().data(), c.numbins, &id));
    ok(pzl_server_wait(srv, id, nullptr, 0, &n, &st));
    EXPECT(n > 0, "%lld candidates", n);
    pzl_server_destroy(srv);
}

// Rows by width: every row at the shortest length that holds its window and its own
// width, row by row.
void row_sets()
{
    static const int menu[] = {128,  192,  256,  320,  384,  512,  640,  768,  1024,
                               1152, 1280, 1536, 1792, 2048, 2560, 3072, 3584, 4096};
    auto menu_has = [](int n) { return (int)std::binary_search(std::begin(menu), std::end(menu), n); };
    auto even_has = [](int n) { return (int)(n >= 8 && n <= 4096 && n % 2 == 0); };
    auto powers_has = [](int n) { return (int)(n >= 64 && n <= 4096 && (n & (n - 1)) == 0); };
    using Has = int (*)(int);
    const struct {
        int zmax, wmax, numharm;
    } shapes[] = {{0, 0, 1}, {0, 0, 32}, {4, 0, 32}, {2, 20, 4}, {51, 0, 8}, {0, 300, 16}, {20, 500, 8},
                  {200, 300, 16}, {200, 500, 32}, {37, 133, 16}, {600, 0, 4}};
    for (auto &sh : shapes)
        for (Has has : {Has(menu_has), Has(even_has), Has(powers_has)}) {
            const PzlConfig c = config(1 << 17, sh.zmax, sh.wmax, sh.numharm, 8);
            PzlGeometry g;
            std::vector<PzlHarm> harms, sets;
            std::vector<int> rows;
            ok(pzl::compute_geometry(c, g, &harms, nullptr));
            bool held = true;
            for (auto &H : harms) held = held && has(H.fftlen);
            EXPECT(pzl::compute_row_sets(harms, g.corr_uselen, has, &sets, &rows) == held, "(%d, %d)", sh.zmax, sh.wmax);
            if (!held) continue;
            size_t k = 0, at = 0;
            long long bank = 0, seg = 0;
            for (auto &H : harms) {
                std::vector<int> len(H.nrows), khw(H.nrows);
                for (int r = 0; r < H.nrows; r++) {
                    khw[r] = pzl_w_resp_halfwidth(-H.zmax + 2 * (r % H.numz), -H.wmax + 20 * (r / H.numz));
                    const double span = (g.corr_uselen / 2 - 0.5) * H.hf + 0.5;
                    const int window =
                        H.stage == 0 ? g.corr_uselen : std::max(H.max_numrs, 2 * ((int)floor(span + 1.0) + 1));
                    len[r] = window + 4 * khw[r];
                    while (len[r] < H.fftlen && !has(len[r])) len[r]++;
                    if (len[r] > H.fftlen || khw[r] > H.halfwidth) len[r] = H.fftlen;
                }
                for (int n = H.fftlen; n >= 2; n--) {
                    if (std::find(len.begin(), len.end(), n) == len.end()) continue;
                    std::vector<int> want;
                    int widest = 0;
                    for (int r = 0; r < H.nrows; r++)
                        if (len[r] == n) {
                            want.push_back(r);
                            widest = std::max(widest, khw[r]);
                        }
                    EXPECT(k < sets.size(), "(%d, %d)", sh.zmax, sh.wmax);
                    if (k >= sets.size()) return;
                    const PzlHarm &S = sets[k++];
                    EXPECT(S.fftlen == n && S.nrows == (int)want.size() && S.bank_off == bank && S.seg_off == seg &&
                               S.halfwidth == (n == H.fftlen ? H.halfwidth : widest) && S.parent == H.parent &&
                               std::equal(want.begin(), want.end(), rows.begin() + (long)at),
                           "(%d, %d) harmonic %d/%d, %d points", sh.zmax, sh.wmax, H.harmnum, H.numharm, n);
                    at += want.size();
                    bank += (long long)want.size() * n;
                    seg += n / 2;
                }
            }
            EXPECT(k == sets.size() && at == rows.size(), "(%d, %d)", sh.zmax, sh.wmax);
        }
}

}  // namespace

int main(int argc, char **argv)
{
    const std::string name = argc > 1 ? argv[1] : "";
    if (name == "exact") exact();
    else if (name == "rule") rule();
    else if (name == "memory") memory();
    else if (name == "server") server();
    else if (name == "overflow") overflow();
    else if (name == "deadline") deadline();
    else if (name == "tuner") tuner();
    else if (name == "pinned") pinned();
    else if (name == "row_sets") row_sets();
    else {
        fprintf(stderr, "no check '%s'\n", name.c_str());
        return 2;
    }
    printf("%s: %s\n", name.c_str(), bad ? "FAILED" : "OK");
    return bad ? 1 : 0;
}
