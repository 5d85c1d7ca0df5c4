// wave_model.cpp — runs the fixed-dt kernels' own source (mc_fixed_dt.h) on the CPU, one fiber a
// lane, with the waves of a workgroup in an order that the test chooses: a wave keeps the
// processor from one wave operation to the next, and the scheduler then picks the wave that
// goes on.  It reports workgroup barriers that meet at different places, waves that wait for one
// that has left, lanes that part within a wave, and stores past the launch's LDS.
// Test infrastructure only (x86-64).
#include "../../mcluminescence_amd/csrc/mc_fixed_dt.h"

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <vector>

namespace mcl {
alignas(64) unsigned char lds_raw[160 * 1024 + 4096];   // the kernels' dynamic LDS
}

namespace wave_model {
namespace {

constexpr int kLanes = 64, kMaxWaves = 8;
constexpr size_t kStack = 128 * 1024;

extern "C" void wave_model_switch(void** save, void* to);
asm(R"(
.text
.globl wave_model_switch
.type wave_model_switch, @function
wave_model_switch:
    pushq %rbp
    pushq %rbx
    pushq %r12
    pushq %r13
    pushq %r14
    pushq %r15
    movq %rsp, (%rdi)
    movq %rsi, %rsp
    popq %r15
    popq %r14
    popq %r13
    popq %r12
    popq %rbx
    popq %rbp
    ret
.size wave_model_switch, .-wave_model_switch
)");

struct Wave {
    void* sp[kLanes];
    uint64_t val[2][kLanes];
    uint32_t op[kLanes];       // where each lane stopped; 0: it has left
    uint32_t phase[kLanes];
    bool waiting;              // at a workgroup barrier
    bool left;
    double prio;
};

Wave g_wave[kMaxWaves];
unsigned char* g_stacks = nullptr;
int g_nw, g_w, g_l;
unsigned g_block;
void* g_main;
void (*g_kernel)(const mcl::LaunchArgs&);
const mcl::LaunchArgs* g_args;
char g_error[256];
// schedule: 0 the waves in turn; 1 + w: wave w only when no other can go on; 100 + w: wave w
// whenever it can; 200: a random order that changes now and then
int g_policy;
uint64_t g_rng;

double random01()
{
    g_rng = g_rng * 6364136223846793005ull + 1442695040888963407ull;
    return (double)(g_rng >> 11) * 0x1p-53;
}

void fail(const char* text, int a, int b)
{
    if (g_error[0] == 0) snprintf(g_error, sizeof g_error, "%s (%d, %d)", text, a, b);
}

void resume(int w, int l, void** save)
{
    g_w = w;
    g_l = l;
    wave_model_switch(save, g_wave[w].sp[l]);
}

// The lane goes to sleep: the wave's next lane runs, or after its last one the scheduler.
void yield()
{
    const int w = g_w, l = g_l;
    void** save = &g_wave[w].sp[l];
    if (l + 1 < kLanes) resume(w, l + 1, save);
    else wave_model_switch(save, g_main);
}

void lane_main()
{
    g_kernel(*g_args);
    g_wave[g_w].op[g_l] = 0;
    for (;;) yield();
}

// Runs wave w from its lanes' present meeting to the next.
void run_wave(int w)
{
    resume(w, 0, &g_main);
    Wave& W = g_wave[w];
    for (int l = 1; l < kLanes; ++l)
        if (W.op[l] != W.op[0]) fail("lanes of a wave are at different operations: lane, wave", l, w);
    W.left = W.op[0] == 0;
    W.waiting = W.op[0] >= kWorkgroupBarrier;
}

int pick()
{
    static int turn = 0;
    if (g_policy >= 200 && random01() < 0.02) g_wave[(int)(random01() * g_nw)].prio = random01();
    int best = -1;
    for (int k = 0; k < g_nw; ++k) {
        const int w = g_policy == 0 ? (turn + 1 + k) % g_nw : k;
        const Wave& W = g_wave[w];
        if (W.left || W.waiting) continue;
        if (best < 0 || (g_policy != 0 && W.prio > g_wave[best].prio)) best = w;
    }
    turn = best;
    return best;
}

void run_block()
{
    for (int w = 0; w < g_nw; ++w) {
        Wave& W = g_wave[w];
        W.waiting = W.left = false;
        W.prio = g_policy >= 200 ? random01() : g_policy == 1 + w ? -1.0 : g_policy == 100 + w ? 1.0 : 0.0;
        for (int l = 0; l < kLanes; ++l) {
            unsigned char* top = g_stacks + (size_t)(w * kLanes + l + 1) * kStack;
            void** s = (void**)top - 2;
            s[0] = (void*)&lane_main;                  // (the stack as a call leaves it)
            s[1] = nullptr;
            W.sp[l] = (void*)(s - 6);
            W.phase[l] = 0;
        }
    }
    while (g_error[0] == 0) {
        const int w = pick();
        if (w >= 0) {
            run_wave(w);
            continue;
        }
        int left = 0;
        for (int k = 0; k < g_nw; ++k) left += g_wave[k].left ? 1 : 0;
        if (left == g_nw) return;
        if (left != 0) return fail("waves wait at a barrier that others will not reach: line, waves gone",
                                   (int)(g_wave[0].left ? 0 : g_wave[0].op[0] & 0xFFFFu), left);
        for (int k = 1; k < g_nw; ++k)
            if (g_wave[k].op[0] != g_wave[0].op[0])
                return fail("workgroup barriers of different places meet: lines",
                            (int)(g_wave[0].op[0] & 0xFFFFu), (int)(g_wave[k].op[0] & 0xFFFFu));
        for (int k = 0; k < g_nw; ++k) g_wave[k].waiting = false;
    }
}

template <int NW, bool GM, bool WIDE>
void kernel(const mcl::LaunchArgs& a)
{
    if constexpr (NW == 1) mcl::fixed_dt_kernel<GM, WIDE>(a);
    else mcl::fixed_dt_mw_kernel<NW, GM, WIDE>(a);
}

template <bool GM, bool WIDE>
void choose(int nw)
{
    g_kernel = nw == 8 ? kernel<8, GM, WIDE> : nw == 4 ? kernel<4, GM, WIDE>
             : nw == 2 ? kernel<2, GM, WIDE> : kernel<1, GM, WIDE>;
}

}  // namespace

Index thread_index() { return {(unsigned)(g_w * kLanes + g_l)}; }
Index block_index() { return {g_block}; }
int lane() { return g_l; }

const uint64_t* meet(uint32_t op, uint64_t v)
{
    Wave& W = g_wave[g_w];
    const int l = g_l;
    const uint32_t ph = W.phase[l]++ & 1u;   // (a lane is at most one meeting ahead of another)
    W.val[ph][l] = v;
    W.op[l] = op;
    yield();
    return W.val[ph];
}

}  // namespace wave_model

// form: 0 everything in LDS, 1 holes in scratch, 2 electrons there too (both take the kernels
// that search wider blocks); wide: those kernels in LDS.  persistent: one workgroup that takes
// every cluster by its ticket (the scratch forms always), else a workgroup a cluster.
extern "C" int wm_run_fixed_dt(const mcl_run_params* runs, int n_runs, uint64_t seed, int n_bins,
                               int row_len, int waves, int form, int wide, int persistent,
                               double holes_per_cell, int policy, uint64_t schedule_seed,
                               uint32_t* counts, uint64_t* live, uint64_t* work, char* error, int error_len)
{
    using namespace wave_model;
    std::vector<mcl::RunDesc> desc;
    std::vector<int32_t> crun, csim;
    int max_h = 0, max_e = 0, cells = 1;
    for (int r = 0; r < n_runs; ++r) {
        const mcl_run_params& p = runs[r];
        mcl::RunDesc d{};
        const double rho = p.rho_prime * (3.0 / (4.0 * 0x1.921fb54442d18p+1) * std::pow(p.alpha, 3.0));
        const double side = std::pow(p.holes / rho, 1.0 / 3.0);
        d.side_nm = side * 1e9;
        d.side_b_nm = (side * p.boundary_factor) * 1e9;
        d.alpha_nm = p.alpha * 1e-9;
        d.s = p.s; d.b = p.b; d.E_cb = p.E_cb; d.E_loc_1 = p.E_loc_1; d.E_loc_2 = p.E_loc_2; d.k_b = p.k_b;
        d.T0_K = p.T_start + 273.15;
        d.T_rate = p.T_rate;
        d.dt = p.dt;
        d.two_channel = p.E_loc_1 != p.E_loc_2 && p.Retrap > 0.0 && p.Retrap < 1.0;
        d.always_chan2 = p.Retrap >= 1.0;
        d.ret_thr = d.two_channel ? (uint64_t)(p.Retrap * 0x1p32) : 0u;
        d.n_e0 = (int32_t)(p.N_e * p.e_ratio_start);
        d.n_h = (int32_t)(p.holes * std::pow(p.boundary_factor, 3.0));
        d.n_steps = p.n_steps;
        d.run_id = r;
        d.grid = mcl::grid_dim(d.n_h, holes_per_cell);
        d.cell_nm = (float)(d.side_b_nm / d.grid);
        d.inv_cell = (float)(d.grid / d.side_b_nm);
        desc.push_back(d);
        for (int s = 0; s < p.sims; ++s) { crun.push_back(r); csim.push_back(s); }
        max_h = max(max_h, d.n_h);
        max_e = max(max_e, d.n_e0);
        cells = max(cells, d.grid * d.grid * d.grid);
    }
    const bool gm = form != 0;
    mcl::LaunchArgs a{};
    a.runs = desc.data();
    a.c_run = crun.data();
    a.c_sim = csim.data();
    a.n_clusters = a.n_order = (int32_t)crun.size();
    a.key0 = (uint32_t)seed;
    a.key1 = (uint32_t)(seed >> 32);
    a.n_bins = n_bins;
    a.row_len = row_len;
    a.counts = counts;
    a.live_steps = live;
    a.work = work;
    a.h_cap = (max_h + 3) / 4 * 4 + 4;
    a.e_cap = max(64, (max_e + 63) / 64 * 64);
    a.g_cap = (cells + 1 + 3) / 4 * 4;
    a.wave_search_max = 32;
    a.wide = wide;
    uint32_t ticket = 0;
    if (persistent || gm) a.queue = &ticket;
    a.e_lds = form == 1;
    const int e_bytes = mcl::fixed_dt_electron_bytes(a.e_cap);
    a.gstride = gm ? mcl::cluster_global_stride(a.h_cap, a.g_cap, e_bytes, a.e_lds != 0) : 0;
    std::vector<unsigned char> scratch((size_t)a.gstride + 256, 0xCD);
    a.gscratch = scratch.data() + (256 - (uintptr_t)scratch.data() % 256) % 256;
    const size_t lds = (size_t)(gm ? mcl::cluster_global_lds(e_bytes, a.e_lds != 0)
                                   : mcl::cluster_lds_bytes(a.h_cap, a.g_cap, e_bytes)) +
                       (size_t)mcl::fixed_dt_waves_lds(waves);
    g_error[0] = 0;
    if (lds > 160 * 1024) snprintf(g_error, sizeof g_error, "the clusters need %zu bytes of LDS", lds);
    if (gm) choose<true, true>(waves);
    else if (wide) choose<false, true>(waves);
    else choose<false, false>(waves);
    g_nw = waves;
    g_args = &a;
    g_policy = policy;
    g_rng = schedule_seed * 2 + 1;
    if (!g_stacks) g_stacks = (unsigned char*)aligned_alloc(4096, (size_t)kMaxWaves * kLanes * kStack);
    const int blocks = a.queue != nullptr ? 1 : a.n_order;
    for (g_block = 0; (int)g_block < blocks && g_error[0] == 0; ++g_block) {
        memset(mcl::lds_raw, 0xCD, sizeof mcl::lds_raw);
        run_block();
        for (size_t i = lds; i < sizeof mcl::lds_raw && g_error[0] == 0; ++i)
            if (mcl::lds_raw[i] != 0xCD) snprintf(g_error, sizeof g_error, "a store past the LDS, at byte %zu of %zu", i, lds);
    }
    snprintf(error, (size_t)error_len, "%s", g_error);
    return g_error[0] == 0 ? 0 : -1;
}
