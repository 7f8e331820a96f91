// nuc_large_group (lcs_nucleus.hip) on the CPU: its source text, taken from the
// kernel file by the test that builds this program (narrow_group.inc), run by
// 512 threads as coroutines. A wave's lanes go on together between collectives
// and the waves between two barriers run one after the other, in an order that
// the test chooses, so a word that one wave overwrites while another may still
// have to read it gives a wrong result here every time. Each case is compared
// with a sort of the whole group; threads that return different counts, or end
// while others wait at a barrier, fail it.
#include <ucontext.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#define __device__
#define __restrict__

namespace emu {
constexpr int kThreads = 512, kLanes = 64, kWaves = kThreads / kLanes;
constexpr size_t kStack = 64 << 10;
enum Wait { kRun, kWave, kBlock, kDone };
struct Fiber {
    ucontext_t ctx;
    Wait wait;
    uint64_t in[2];
};
Fiber fib[kThreads];
ucontext_t sched;
std::vector<char> stacks((size_t)kThreads * kStack);
int cur;
void (*body)();
bool failed;

void yield(Wait w) {
    fib[cur].wait = w;
    swapcontext(&fib[cur].ctx, &sched);
}
void entry() {
    body();
    fib[cur].wait = kDone;
    swapcontext(&fib[cur].ctx, &sched);
}
// Every lane of the wave has put its word: the lanes' words, by lane.
void collect(uint64_t v, uint64_t (&all)[kLanes]) {
    fib[cur].in[0] = v;
    yield(kWave);
    const int w0 = cur / kLanes * kLanes;
    for (int l = 0; l < kLanes; ++l) all[l] = fib[w0 + l].in[0];
    yield(kWave);   // (every lane has read them)
}
// Runs one wave until its lanes all wait at the barrier or are done.
void run_wave(int w) {
    for (;;) {
        // lanes from the last to the first: a wave's reads precede thread 0's writes
        for (int l = kLanes - 1; l >= 0; --l) {
            cur = w * kLanes + l;
            if (fib[cur].wait == kRun) swapcontext(&sched, &fib[cur].ctx);
        }
        int n[4] = {};
        for (int l = 0; l < kLanes; ++l) ++n[fib[w * kLanes + l].wait];
        if (n[kWave] == kLanes) {
            for (int l = 0; l < kLanes; ++l) fib[w * kLanes + l].wait = kRun;
            continue;
        }
        if (n[kWave] != 0 || (n[kBlock] != 0 && n[kDone] != 0)) failed = true;   // lanes of a wave diverged
        return;
    }
}
// order: the waves' order between barriers. False when the threads diverged.
bool run(void (*fn)(), const int* order) {
    body = fn;
    failed = false;
    for (int t = 0; t < kThreads; ++t) {
        getcontext(&fib[t].ctx);
        fib[t].ctx.uc_stack.ss_sp = stacks.data() + (size_t)t * kStack;
        fib[t].ctx.uc_stack.ss_size = kStack;
        fib[t].ctx.uc_link = &sched;
        makecontext(&fib[t].ctx, entry, 0);
        fib[t].wait = kRun;
    }
    for (int rounds = 0; rounds < 100000; ++rounds) {
        for (int i = 0; i < kWaves; ++i) run_wave(order[i]);
        if (failed) return false;
        int block = 0, done = 0;
        for (int t = 0; t < kThreads; ++t) {
            block += fib[t].wait == kBlock;
            done += fib[t].wait == kDone;
        }
        if (done == kThreads) return true;
        if (block != kThreads) return false;   // some ended while others wait
        for (int t = 0; t < kThreads; ++t) fib[t].wait = kRun;
    }
    return false;
}
}  // namespace emu

// ---- what the kernel text uses ----
constexpr int kWave = 64, kFT = 512, kFW = kFT / kWave;
constexpr uint32_t kNone = 0xffffffffu;
constexpr uint32_t kGroupMax = 4 * kWave;
constexpr uint32_t kNucKeyCache = 2048, kNucList = 32768;
struct Smem {
    struct {
        struct {
            uint64_t lkey[kNucKeyCache], gkey[kGroupMax], gsorted[kGroupMax];
            double gw[kGroupMax];
        } fc;
    } u;
    struct {
        uint32_t lg_n, lg_cb;
        double lg_mb;
        uint32_t nall[kFW], ipen[kFW], imsk[kFW];
        double sraw[kFW];
        uint64_t ck[kFW];
    } l;
};
using NucFinSmem = Smem;
static Smem g_fin;
alignas(16) static uint16_t g_code[kNucList];

static uint32_t tid_x() { return (uint32_t)emu::cur; }
static int lane_id() { return emu::cur % kWave; }
static void __syncthreads() { emu::yield(emu::kBlock); }
template <class T>
static T atomicAdd(T* p, T v) {
    const T o = *p;
    *p = o + v;
    return o;
}
static uint32_t min(uint32_t a, uint32_t b) { return std::min(a, b); }
static uint64_t u64_min(uint64_t a, uint64_t b) { return std::min(a, b); }
static uint64_t ballot(bool p) {
    uint64_t all[kWave], m = 0;
    emu::collect(p, all);
    for (int l = 0; l < kWave; ++l) m |= all[l] << l;
    return m;
}
static uint32_t wave_scan_incl_u(uint32_t v) {
    uint64_t all[kWave];
    emu::collect(v, all);
    uint32_t s = 0;
    for (int l = 0; l <= lane_id(); ++l) s += (uint32_t)all[l];
    return s;
}
static double wave_scan_incl(double v) {
    uint64_t all[kWave], b;
    std::memcpy(&b, &v, 8);
    emu::collect(b, all);
    double s = 0.0;
    for (int l = 0; l <= lane_id(); ++l) {
        double d;
        std::memcpy(&d, &all[l], 8);
        s += d;
    }
    return s;
}
template <int NT>
static uint64_t block_min_u64(uint64_t v, uint64_t* red) {
    uint64_t all[kWave];
    emu::collect(v, all);
    if (lane_id() == 0) red[tid_x() / kWave] = *std::min_element(all, all + kWave);
    __syncthreads();
    const uint64_t r = *std::min_element(red, red + NT / kWave);
    __syncthreads();
    return r;
}
static double exp_f64(double x) { return std::exp(x); }
static float tempered(float p, float maxl, float inv_t) { return (p - maxl) * inv_t; }
static uint64_t rank_key(float v, uint32_t idx) {
    uint32_t u;
    const float z = v == 0.0f ? 0.0f : v;
    std::memcpy(&u, &z, 4);
    u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
    return ((uint64_t)~u << 32) | idx;
}
static float rank_val(uint64_t k) {
    uint32_t u = ~(uint32_t)(k >> 32);
    u = (u & 0x80000000u) ? (u & 0x7fffffffu) : ~u;
    float f;
    std::memcpy(&f, &u, 4);
    return f;
}

#include "narrow_group.inc"

// ---- the cases ----
static std::vector<uint64_t> g_list;
static uint32_t g_ng, g_n, g_ret[emu::kThreads], g_cb[emu::kThreads];
static double g_mb[emu::kThreads];
static float g_max, g_inv_t;
static NucTarget g_tgt;
constexpr uint32_t kC0 = 130, kC1 = 131;

static void thread_body() {
    const uint32_t m = nuc_large_group(kC0, kC1, g_ng, g_n, g_list.data(), g_max, g_inv_t, g_tgt);
    const uint32_t t = tid_x();
    g_ret[t] = m;
    g_cb[t] = g_fin.l.lg_cb;
    g_mb[t] = g_fin.l.lg_mb;
}

static int check(uint32_t n, uint32_t share, float step, int kind, uint32_t seed, const int* order, const char* oname) {
    std::mt19937 rng(seed);
    std::normal_distribution<float> nd;
    g_list.resize(n);
    std::vector<uint64_t> group;
    g_max = 6.0f;
    g_inv_t = 0.75f;
    for (uint32_t i = 0; i < n; ++i) {
        float v = std::min(nd(rng), 5.5f);
        if (step > 0.0f) v = std::round(v / step) * step;
        g_list[i] = rank_key(v, i * 3u + 1u);
        const bool in = rng() % 100 < share;
        g_code[i] = in ? (uint16_t)(kC0 + rng() % 2) : (uint16_t)(rng() % 2 ? 7 : 0xffff);
        if (in) group.push_back(g_list[i]);
        if (i < kNucKeyCache) g_fin.u.fc.lkey[i] = g_list[i];
    }
    g_n = n;
    g_ng = (uint32_t)group.size();
    std::sort(group.begin(), group.end());
    std::vector<double> pre(group.size());
    double s = 0.0;
    for (size_t i = 0; i < group.size(); ++i)
        pre[i] = s += exp_f64((double)tempered(rank_val(group[i]), g_max, g_inv_t));
    // the target: a position, or a share of the weight
    const double at = std::uniform_real_distribution<double>(0.0, 1.0)(rng);
    const uint32_t pos = (uint32_t)(at * (g_ng - 1));
    g_tgt = kind == 0 ? NucTarget{pos, 0.0, 1.0, HUGE_VAL} : NucTarget{kNone, 2.0, s + 4.0, (2.0 + at * s) / (s + 4.0)};
    uint32_t want = pos;
    if (kind != 0)
        for (want = 0; (2.0 + pre[want]) / (s + 4.0) < g_tgt.reach && want + 1 < g_ng;) ++want;
    std::memset(&g_fin.l, 0xff, sizeof g_fin.l);
    int bad = 0;
    auto fail = [&](const char* what) {
        std::printf("FAIL %s: n %u, group %u, step %g, kind %d, seed %u, waves %s\n", what, n, g_ng, step, kind, seed, oname);
        bad = 1;
    };
    if (!emu::run(thread_body, order)) {
        fail("threads diverge at a barrier");
        return 1;
    }
    for (int t = 1; t < emu::kThreads; ++t)
        if (g_ret[t] != g_ret[0] || g_cb[t] != g_cb[0] || g_mb[t] != g_mb[0]) {
            fail("threads disagree");
            return 1;
        }
    const uint32_t m = g_ret[0], cb = g_cb[0];
    if (m == kNone || m > kGroupMax || cb > want || cb + m <= want) {
        fail("the target is not among the candidates left");
        return 1;
    }
    const double before = cb ? pre[cb - 1] : 0.0;
    if (!(std::fabs(g_mb[0] - before) <= 1e-11 * s)) fail("the weight before them");
    for (uint32_t i = 0; i < m; ++i)
        if (g_fin.u.fc.gsorted[i] != group[cb + i] ||
            g_fin.u.fc.gw[i] != exp_f64((double)tempered(rank_val(group[cb + i]), g_max, g_inv_t))) {
            fail("the ranked candidates");
            break;
        }
    return bad;
}

int main() {
    const int up[8] = {0, 1, 2, 3, 4, 5, 6, 7}, down[8] = {7, 6, 5, 4, 3, 2, 1, 0}, mix[8] = {3, 0, 6, 1, 7, 4, 2, 5};
    struct { const int* o; const char* name; } const orders[] = {{up, "ascending"}, {down, "descending"}, {mix, "mixed"}};
    // list length, share of it in the group, spacing of the values
    struct { uint32_t n, share; float step; } const shapes[] = {
        {600, 90, 0.0f}, {600, 100, 100.0f}, {2048, 50, 0.125f}, {5000, 70, 0.0f},
        {16384, 20, 0.0625f}, {16384, 60, 1.0f}, {16385, 10, 0.25f}, {32768, 100, 0.0f}, {32768, 90, 0.5f}};
    int fails = 0, n = 0;
    uint32_t seed = 1;
    for (const auto& s : shapes)
        for (int kind = 0; kind < 2; ++kind)
            for (const auto& o : orders) {
                fails += check(s.n, s.share, s.step, kind, seed++, o.o, o.name);
                ++n;
            }
    std::printf("%d cases, %d failed\n", n, fails);
    return fails != 0;
}
