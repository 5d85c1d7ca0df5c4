// mc_fixed_dt.h — fixed-dt trap/charge-kinetics Monte Carlo, one workgroup per cluster:
// the per-cluster body shared by the LDS kernels (mc_fixed_dt.hip) and the
// global-memory kernels for clusters beyond one workgroup's LDS (mc_fixed_dt_global.hip).
//
// Replaces the run x sim x step loop of simulate.py:36-92 (Box / Physics /
// TLTrapSim: engine.py:44-188, tl_trap_lab.py:24-60).  One workgroup of NW
// wavefronts (1, 2, 4 or 8) owns one cluster; everything it touches lives in LDS:
//
//   hole       [h_cap]   16-byte records {x, y, z, meta}, float32 nm, sorted by
//                        grid cell; meta = (claiming electron << 16) | original
//                        hole index; a removed hole keeps its slot with x = 3e38
//   cstart     [g_cap]   first sorted slot of each cell, cstart[G^3] = n_h
//   est        [e_cap]   live electrons: (nearest hole slot << 16) | electron index
//   ew         [e_cap]   w = exp(-alpha r_nn), float32
//   rowm       [e_cap / 64]  per row of 64 slots: bit j set when an electron of the
//                        row may fire in step j of the window (a superset)
//   nf         [e_cap]   the step of the window in which the electron's draw fires
//                        (kNever: in none)
//   lst        [e_cap + 64]  slots gathered from their rows: each wave's from its own
//                        rows' first entry on, a light step's in the last 64
//   xch        [4 NW + 5] (NW > 1) per-wave values exchanged between the waves, the
//                        persistent launch's ticket, and what wave 0 publishes
//
// A cluster too large for that (GM: the global-memory form) keeps hole and
// cstart in its workgroup's slice of a global scratch buffer (slice blockIdx.x,
// so its launches are persistent: one slice per resident workgroup, reused
// cluster after cluster); xch opens the LDS block, followed by the electron arrays
// when they fit there (e_lds), otherwise those follow cstart in the slice.  The
// code is the same; the workgroup barriers order global memory as they order LDS
// (every wave of a workgroup runs on one CU, behind one L1), and the fences of one
// wave widen to workgroup scope.  Only the slots holes take within a cell can
// differ from the LDS form (global atomics need not serve the lanes of one
// instruction in lane order); no result depends on them: every search keys on
// (distance, original hole index).
//
// First-fire windows.  An electron's draw of step n is the Philox word of counter
// (n >> 2, e, run, sim|FIRE), and its threshold depends on the step and on its w,
// which changes only when the electron is searched again, in a step in which its
// draw fires.  So the step in which it next fires is known in advance: at the start
// of each 64-step window every live electron's first firing step is found (the
// scan), and then only the steps in which some electron fires are simulated, with
// those electrons alone; the others change nothing but the live-step tally.  An
// electron that fires and stays (its new nearest hole is too far for the draw, or
// it lost its hole) is scanned again over the rest of the window with its new w.
// Every draw is tested against exactly the threshold the step-by-step loop would
// use, once.
//   scan      one electron a lane, two Philox blocks (eight steps) an iteration,
//             until every lane of the row has fired.  The draws are compared with
//             one bound per electron and window (the threshold of x with the
//             window's largest band term and largest b dt: the threshold is
//             non-decreasing in x); only a block in which some draw is below its
//             bound takes the exact thresholds of its four steps.  For isothermal
//             one-channel runs the bound is the exact threshold.  Rows with few
//             live electrons take the steps across the lanes instead: 16 lanes
//             cover an electron's whole window.
//   light     a step with at most 64 candidates, wave 0 alone, one candidate a lane,
//             without a workgroup barrier.  (Sharing steps of more than 12 or of more
//             than one among the waves measured slower: 1000 x 1500 decays 2.12 ms at
//             64, 2.28 at 12, 2.65 at 1; 250 x 8000 in scratch memory 14.9, 16.2, 18.2.)
//   together  with several waves, the electrons that fire in the next steps with events and
//             whose hole is gone already are searched by all waves, each its own rows, between
//             two barriers, so that few searches are left to the steps themselves.  Such a
//             search keeps wave 0 waiting about as long as two steps that search for
//             themselves, so it is made every 11 / v steps with candidates, v the stale ones
//             of a step as the steps before and the share of the holes that are gone let
//             expect (11 / sqrt(v) above one, where a step's own search takes several
//             passes; at least every 4).  16 x 500 glow 1.14 ms, 64 x 1000 tunnelling ramps 1.86,
//             500 uneven sets 1.96, 32 x 2000 glow 3.12, 64 isothermal curves 1.94; every 8
//             steps with candidates 1.17, 2.07, 2.03, 3.09 and 1.95; by the other waves beside
//             wave 0's events, none waiting, 1.13, 1.91, 1.81, 2.87 and 2.03, but then the
//             waves' timing decides which searches are made, and with it the number of distances
//             evaluated.  One wave alone leaves every search to its step (the decay measured
//             2 % slower with them).
//   heavy     a step with more candidates: every wave takes the candidates of its
//             own rows, gathered 64 to a chunk, and they meet at barriers (winners,
//             each retry round).
//
// Electron coordinates are not stored: they are a pure function of the
// Philox counter (0, e, run, sim|GEOM_E) and are regenerated (each lane its own
// electron's) when nearest holes have to be searched again.
//
// Nearest holes come from a uniform G^3 cell grid over the hole cube: a search
// scans the 3x3x3 cells around the electron and accepts the minimum of
// (d2 bits, original hole index) only if it is closer than every hole outside
// that block can be (guaranteed face distance, with a margin far above float32
// rounding); otherwise the whole wave scans every hole for that electron.  The
// answer is therefore always the first-index argmin of the full scan
// (engine.py:118-119, 173-175); the grid only removes work.
//
// Per step n (start-of-step temperature T_n = T0 + T_rate n dt, simulate.py:53-54):
//   scalars   A = s e^{-E_cb/kT}, B_i = b e^{-E_loc_i/kT} in float64 (own exp),
//             x_A = A dt, b_i dt in float32; lane j holds those of the window's
//             step j.
//   fire      per live electron: u = Philox(n>>2, e, run, sim|FIRE)[n&3],
//             x = fma(b dt, w, x_A); fire iff u < (uint32)((1 - e^{-x}) 2^32).
//   repair    an electron whose hole was removed keeps its old w until a step in
//             which its draw fires against that old w: only then is it searched
//             again (before its fire test; a conflict loser at once).  Exact: the
//             new nearest hole is no closer, so w and x = k dt can only fall, and
//             the threshold of x is non-decreasing in x (checked for every float x
//             by the oracle), so a draw that fails against the old w fails against
//             the new one.
//   conflict  ds_min_u32 of the electron index into the hole's claim field; the
//             lowest index keeps the hole (src/est_params/functions.py:228-239).
//   remove    winners' slots become dead, their holes get the x sentinel.
//   retry     a conflict loser retries on its new nearest hole within the step,
//             accepted with probability T_new / T_old (one more Philox word), for
//             up to MCL_MAX_ROUNDS rounds; this removes the O(k dt) delay a
//             "loser waits a step" rule would put into the decay curves.
//   compact   between windows, stable, when an eighth of the rows can be dropped.
// Counts go out per bin (bin of step n = n * n_bins / n_steps) into a row that is
// zeroed first, like the reference's padded rows.
#pragma once

#include "mc_common.h"

#include <algorithm>

namespace mcl {

constexpr int kWindow = 64;            // steps of a window (a multiple of 4; rowm's bits)
constexpr uint32_t kNever = 255u;      // nf: no firing step in the window
constexpr uint32_t kSearch = 254u;     // published in place of a heavy step: search all rows
// Steps with candidates between two searches of all rows (see "together" above): at first, at
// least, and the numerator of the rule.
constexpr int kFirstEvents = 8, kMinEvents = 4;
constexpr float kEventsPerStale = 11.0f;
// Rows with at most this many live electrons are scanned four electrons at a time,
// 16 lanes each, instead of one electron a lane.
constexpr int kGroupMax = 16;

// Ordering between one wave's writes and its lanes' reads of them: wavefront scope
// in LDS, whose instructions one wave executes in issue order; workgroup scope
// in the global-memory form, so the wave's global stores come before its loads.
template <bool GM>
__device__ __forceinline__ void wave_sync()
{
    if constexpr (GM) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    } else {
        wave_lds_fence();
    }
}

// Simulate cluster c from its geometry to its last step with NW wavefronts, all
// state in lds_raw (GM: holes and cell starts, and the electron arrays unless
// a.e_lds, in the workgroup's scratch slice).  Every branch that holds a
// workgroup barrier depends only on values all waves share: launch constants, results
// of the exchanges, what wave 0 publishes, and what follows from these alone (the window,
// n_live, n_slots, steps).  rowm is none of them: other waves write it while a wave
// reads it.  WIDE: the build that searches wider blocks before every hole
// (far_search_wave).
template <int NW, bool GM, bool WIDE>
__device__ __forceinline__ void run_cluster(const LaunchArgs& a, const int c,
                                            unsigned char* lds_raw)
{
    const int tid = (int)threadIdx.x;
    const int lane = NW == 1 ? tid : (tid & (kWave - 1));
    const int wv = NW == 1 ? 0 : uniform(tid >> 6);
    const int run = uniform(a.c_run[c]);
    const int sim = uniform(a.c_sim[c]);
    const RunDesc R = a.runs[run];
    const int n_e0 = uniform(R.n_e0);
    const int n_h = uniform(R.n_h);
    const int n_steps = uniform(R.n_steps);
    const int h_cap = a.h_cap, e_cap = a.e_cap, g_cap = a.g_cap;

    unsigned char* hbase;      // hole, cstart
    unsigned char* ebase;      // est, ew, rowm, lst, nf
    uint32_t* xbase;           // xch
    if constexpr (GM) {
        unsigned char* const slice = a.gscratch + (size_t)blockIdx.x * (size_t)a.gstride;
        hbase = slice;
        xbase = (uint32_t*)lds_raw;
        ebase = a.e_lds ? lds_raw + fixed_dt_waves_lds(NW)
                        : slice + 16 * (size_t)h_cap + 4 * (size_t)g_cap;
    } else {
        hbase = lds_raw;
        ebase = lds_raw + 16 * h_cap + 4 * g_cap;
        xbase = (uint32_t*)(ebase + fixed_dt_electron_bytes(e_cap));
    }
    float4* hole = (float4*)hbase;
    float* hole_f = (float*)hbase;                   // word view: x at 4 s, meta at 4 s + 3
    uint32_t* hole_u = (uint32_t*)hbase;
    uint32_t* cstart = (uint32_t*)(hole + h_cap);
    uint32_t* est = (uint32_t*)ebase;
    float* ew = (float*)(est + e_cap);
    unsigned long long* rowm = (unsigned long long*)(ew + e_cap);
    uint16_t* lst = (uint16_t*)(rowm + e_cap / kWave);
    uint8_t* nf = (uint8_t*)(lst + e_cap + kWave);
    uint32_t* const xch = xbase;

    const uint32_t k0 = a.key0, k1 = a.key1;
    const uint32_t prun = (uint32_t)R.run_id;
    const uint32_t psim = (uint32_t)sim << 4;
    const ElectronGen egen{prun, psim | MCL_TAG_GEOM_E, k0, k1, R.side_nm};
    const uint64_t ret_thr = R.ret_thr;
    const uint32_t c3f = psim | MCL_TAG_FIRE, c3c = psim | MCL_TAG_CHAN;
    const int nb = a.n_bins > 0 ? a.n_bins : n_steps;   // n_bins == 0: one bin per step
    uint32_t* cnt = a.counts + (size_t)c * (size_t)a.row_len;

    // The counts row starts as zeros (wave 0, which alone writes it later: one
    // wave's stores to an address keep their order).
    if (wv == 0)
        for (int b = lane; b < a.row_len; b += kWave) cnt[b] = 0u;

    uint64_t dist_evals = 0;
    const Grid grid = setup_cluster_t<NW, WIDE>(R, egen, hole, cstart, est, ew, prun, psim, k0, k1, tid,
                                          dist_evals);
    const float alpha_f = (float)R.alpha_nm;

    const bool two_ch = R.two_channel != 0;
    const bool always2 = R.always_chan2 != 0;
    const bool ramp = R.T_rate != 0.0;
    const bool exact_bound = !ramp && !two_ch;   // the window's bound is every step's threshold
    // single-trap parameter sets share one Boltzmann factor between the channels
    const bool b1_is_a = R.b == R.s && R.E_loc_1 == R.E_cb;
    const bool b2_is_b1 = R.E_loc_2 == R.E_loc_1;
    const int step_limit = a.dump.enabled ? min(a.dump.max_steps, n_steps) : n_steps;

    // The window's steps nb0 .. nb0 + len - 1: lane j holds step nb0 + j's scalars
    // (start-of-step temperature, Boltzmann factors in float64, their float32
    // products with dt), lanes past len those of the last step; x_max and b_max are
    // their largest values (b of the channels a draw can take).
    int nb0 = 0, len = 0;
    float l_xA = 0.0f, l_b1 = 0.0f, l_b2 = 0.0f, x_max = 0.0f, b_max = 0.0f;
    auto window_scalars = [&]() {
        const int m = nb0 + min(lane, len - 1);
        const double t = (double)m * R.dt;
        const double T = R.T0_K + R.T_rate * t;
        const double kT = R.k_b * T;
        const double A = R.s * exp_own(-(R.E_cb / kT));
        const double B1 = b1_is_a ? A : R.b * exp_own(-(R.E_loc_1 / kT));
        const double B2 = b2_is_b1 ? B1 : R.b * exp_own(-(R.E_loc_2 / kT));
        l_xA = (float)(A * R.dt);
        l_b1 = (float)(B1 * R.dt);
        l_b2 = (float)(B2 * R.dt);
        // (non-negative floats order as their bits; a NaN, above every number, makes
        // the bound "always", so the exact thresholds decide)
        const uint32_t xb = __float_as_uint(l_xA);
        const uint32_t b1 = __float_as_uint(l_b1), b2 = __float_as_uint(l_b2);
        x_max = __uint_as_float(wave_max_u32(xb));
        b_max = __uint_as_float(wave_max_u32(two_ch ? max(b1, b2) : always2 ? b2 : b1));
    };
    auto threshold = [&](float w, bool ch2, float xA, float b1, float b2) -> FireThr {
        return fire_threshold(__builtin_fmaf(ch2 ? b2 : b1, w, xA));
    };
    auto fires = [](uint32_t u, const FireThr& t) -> bool { return t.always || u < t.thr; };
    // Does the channel draw of word d pick channel 2?
    auto channel_word = [&](const u32x4& r, int d) -> bool {
        return (uint64_t)pick_word(r, d) < ret_thr;
    };

    // First firing step (window-relative, kNever: none) from step `from` on of the
    // electrons of the lanes in mask (index o, w), four at a time, 16 lanes each:
    // lane q of a row tests block q's four steps.  Writes f in those lanes; returns
    // the mask of the steps found.  (from may differ between the lanes.)
    auto group_scan = [&](uint64_t mask, uint32_t o, float w, int from, uint32_t& f) -> uint64_t {
        uint64_t steps = 0;
        const int g = lane >> 4, q = lane & 15;
        while (mask != 0) {
            int b[4];
            b[0] = __builtin_ctzll(mask);
            mask &= mask - 1;
#pragma unroll
            for (int i = 1; i < 4; ++i) {          // (a missing one repeats the first)
                b[i] = mask != 0 ? (int)__builtin_ctzll(mask) : b[0];
                mask = mask != 0 ? mask & (mask - 1) : 0;
            }
            const uint32_t o0 = lane_value(o, b[0]), o1 = lane_value(o, b[1]),
                           o2 = lane_value(o, b[2]), o3 = lane_value(o, b[3]);
            const float w0 = lane_value(w, b[0]), w1 = lane_value(w, b[1]),
                        w2 = lane_value(w, b[2]), w3 = lane_value(w, b[3]);
            const uint32_t og = g == 0 ? o0 : g == 1 ? o1 : g == 2 ? o2 : o3;
            const float wg = g == 0 ? w0 : g == 1 ? w1 : g == 2 ? w2 : w3;
            const uint32_t f0 = lane_value((uint32_t)from, b[0]), f1 = lane_value((uint32_t)from, b[1]),
                           f2 = lane_value((uint32_t)from, b[2]), f3 = lane_value((uint32_t)from, b[3]);
            const int fg = (int)(g == 0 ? f0 : g == 1 ? f1 : g == 2 ? f2 : f3);
            const uint32_t blk = (uint32_t)(nb0 >> 2) + (uint32_t)q;
            const u32x4 u = philox10(blk, og, prun, c3f, k0, k1);
            uint32_t first = kNever;
            if (exact_bound) {
                const FireThr t = threshold(wg, always2, x_max, b_max, b_max);
#pragma unroll
                for (int d = 3; d >= 0; --d) {
                    const int rel = 4 * q + d;
                    if (rel >= fg && rel < len && fires(pick_word(u, d), t)) first = (uint32_t)rel;
                }
            } else {
                u32x4 cw{0u, 0u, 0u, 0u};
                if (two_ch) cw = philox10(blk, og, prun, c3c, k0, k1);
#pragma unroll
                for (int d = 3; d >= 0; --d) {
                    const int rel = 4 * q + d;
                    const float xA = __shfl(l_xA, rel);
                    const float b1 = __shfl(l_b1, rel), b2 = __shfl(l_b2, rel);
                    const bool ch = two_ch ? channel_word(cw, d) : always2;
                    if (rel >= fg && rel < len && fires(pick_word(u, d), threshold(wg, ch, xA, b1, b2)))
                        first = (uint32_t)rel;
                }
            }
            first = row_min_u32(first);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t fi = lane_value(first, 16 * i);
                if (lane == b[i]) f = fi;
                if (fi != kNever) steps |= 1ull << fi;
            }
        }
        return steps;
    };

    // The same for one electron a lane (live: the lane has one), the blocks of the
    // window in order, until every lane has fired.
    auto lane_scan = [&](bool live, uint32_t o, float w, int from, uint32_t& f) -> uint64_t {
        FireThr tb;
        if (exact_bound) {
            tb = threshold(w, always2, x_max, b_max, b_max);
        } else {
            const float xb = __builtin_fmaf(b_max, w, x_max);
            tb = fire_threshold(xb);
            tb.always = tb.always || !(xb < __builtin_inff());
        }
        bool todo = live && (tb.always || tb.thr != 0u);
        uint32_t first = kNever;
        // the four steps of block q (window-relative) with its draws u
        auto block = [&](int q, const u32x4& u) {
            const uint32_t um = min(min(u.x, u.y), min(u.z, u.w));
            const bool hit = todo && (tb.always || um < tb.thr);
            if (ballot(hit) == 0) return;
            u32x4 cw{0u, 0u, 0u, 0u};
            if (two_ch) cw = philox10((uint32_t)(nb0 >> 2) + (uint32_t)q, o, prun, c3c, k0, k1);
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const int rel = 4 * q + d;
                if (rel < from || rel >= len) continue;
                FireThr t = tb;
                if (!exact_bound) {
                    const bool ch = two_ch ? channel_word(cw, d) : always2;
                    t = threshold(w, ch, lane_value(l_xA, rel), lane_value(l_b1, rel),
                                  lane_value(l_b2, rel));
                }
                if (hit && first == kNever && fires(pick_word(u, d), t)) first = (uint32_t)rel;
            }
            todo = todo && first == kNever;
        };
        const int q_end = (len + 3) >> 2;
        for (int q = from >> 2; q < q_end && ballot(todo) != 0; q += 2) {
            const uint32_t blk = (uint32_t)(nb0 >> 2) + (uint32_t)q;
            const u32x4 ua = philox10(blk, o, prun, c3f, k0, k1);
            const u32x4 ub = philox10(blk + 1u, o, prun, c3f, k0, k1);
            block(q, ua);
            if (q + 1 < q_end) block(q + 1, ub);
        }
        if (live) f = first;
        const uint64_t bit = live && first != kNever ? 1ull << first : 0ull;
        return ((uint64_t)wave_or_u32((uint32_t)(bit >> 32)) << 32) | wave_or_u32((uint32_t)bit);
    };
    auto first_fire = [&](bool live, uint32_t o, float w, int from, uint32_t& f) -> uint64_t {
        const uint64_t m = ballot(live);
        if (__popcll(m) <= kGroupMax) return group_scan(m, o, w, from, f);
        return lane_scan(live, o, w, from, f);
    };
    // The slots of rows [r_lo, r_hi) that fire in the n steps from rel on, to out (at most
    // cap of them); returns how many.  A lane reads eight slots' nf at once, so one trip
    // covers eight rows, and the row masks skip eight rows without one.
    auto gather = [&](int rel, int n, int r_lo, int r_hi, uint16_t* out, int cap) -> int {
        const uint64_t bits = (~0ull >> (kWindow - n)) << rel;
        int k = 0;
        for (int r0 = r_lo; r0 < r_hi; r0 += kWave) {
            const uint64_t rm = r0 + lane < r_hi ? (uint64_t)rowm[r0 + lane] : 0ull;
            const uint64_t ev = ballot((rm & bits) != 0ull);
            for (int r8 = 0; r8 < kWave && (ev >> r8) != 0; r8 += 8) {
                if (((ev >> r8) & 0xFFull) == 0) continue;
                const int p0 = (r0 + r8) * kWave + 8 * lane;
                const uint2 v = p0 < r_hi * kWave ? *(const uint2*)(nf + p0)
                                                  : make_uint2(~0u, ~0u);      // (kNever bytes)
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    const uint32_t f = ((t < 4 ? v.x : v.y) >> (8 * (t & 3))) & 0xFFu;
                    const bool is = f - (uint32_t)rel < (uint32_t)n;
                    const uint64_t m = ballot(is);
                    if (m == 0) continue;
                    const int q = k + lanes_below(m);
                    if (is && q < cap) out[q] = (uint16_t)(p0 + t);
                    k += __popcll(m);
                }
            }
        }
        wave_sync<GM>();
        return k;
    };

    // Claim hole nn for electron o: the claim field keeps the lowest index.
    auto claim = [&](uint32_t nn, uint32_t o) {
        atomicMin(&hole_u[4 * nn + 3], (o << 16) | (hole_u[4 * nn + 3] & 0xFFFFu));
    };
    // Nearest live holes of the lanes in mask (coordinates in the lanes), written to
    // est and ew of their slots p; nn and w follow.
    auto search = [&](uint64_t mask, bool need, float x, float y, float z, uint32_t o, int p,
                      uint32_t& nn, float& w) {
        uint64_t key = ~0ull;
        search_lanes<WIDE>(grid, mask, need, x, y, z, a.wave_search_max, lane, key, dist_evals);
        if (need) {
            nn_from_key(key, alpha_f, nn, w);
            est[p] = (nn << 16) | o;
            ew[p] = w;
        }
    };
    // A conflict loser's retry: accepted with probability T_new / T_old.
    auto accepted = [&](const FireThr& tn, const FireThr& to, uint32_t blk, int word, uint32_t o,
                        uint32_t round) -> bool {
        const uint64_t Tn = tn.always ? 0x100000000ull : (uint64_t)tn.thr;
        const uint64_t To = to.always ? 0x100000000ull : (uint64_t)to.thr;
        if (Tn >= To) return true;
        const u32x4 rr = philox10(blk, o, prun, psim | (MCL_TAG_RETRY0 + round), k0, k1);
        return (uint64_t)pick_word(rr, word) * To < (Tn << 32);
    };
    // Per-wave values between the waves (NW > 1): lane 0 of each wave publishes
    // v (exchange2: and v2, at NW), one workgroup barrier, then every wave reads all NW
    // values.  Consecutive exchanges alternate between two slots of xch and each holds
    // a barrier, so a slot is rewritten only after every wave has read it.
    int xph = 0;
    auto exchange2 = [&](uint32_t v, uint32_t v2) -> const uint32_t* {
        uint32_t* slot = xch + (xph & 1) * (2 * NW);
        if (lane == 0) {
            slot[wv] = v;
            slot[NW + wv] = v2;
        }
        __syncthreads();
        ++xph;
        return slot;
    };
    auto exchange = [&](uint32_t v) -> const uint32_t* {
        uint32_t* slot = xch + (xph & 1) * (2 * NW);
        if (lane == 0) slot[wv] = v;
        __syncthreads();
        ++xph;
        return slot;
    };
    auto any_wave = [&](bool v) -> bool {
        if constexpr (NW == 1) {
            return v;
        } else {
            const uint32_t* x = exchange(v ? 1u : 0u);
            uint32_t r = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) r |= x[w];
            return uniform(r) != 0u;
        }
    };

    int n_live = n_e0, n_slots = n_e0;
    int rows = 0;
    // wave 0's tallies
    uint64_t lsteps = 0;
    int n_acc = 0;               // steps below it are in lsteps
    int bin = 0;
    uint32_t bin_acc = 0;
    const double inv_steps = 1.0 / (double)n_steps;
    // Step n (the next one with candidates) ended with `wins` recombinations.
    auto finish_step = [&](int n, uint32_t wins) {
        lsteps += (uint64_t)n_live * (uint64_t)(n + 1 - n_acc);
        n_acc = n + 1;
        n_live -= (int)wins;
        if (wins == 0u) return;
        int b = n;
        if (nb != n_steps) {
            // floor(n nb / n_steps): the quotient in float64, then one step either way
            const int64_t num = (int64_t)n * (int64_t)nb;
            b = (int)((double)num * inv_steps);
            const int64_t rem = num - (int64_t)b * (int64_t)n_steps;
            b += rem < 0 ? -1 : rem >= (int64_t)n_steps ? 1 : 0;
            b = uniform(b);
        }
        if (b != bin) {
            if (lane == 0 && bin_acc != 0u) cnt[bin] = bin_acc;
            bin = b;
            bin_acc = 0u;
        }
        bin_acc += wins;
    };

    // A step's conflict rounds with at most one candidate a lane (act), one wave:
    // round it = 0 searches the candidates whose hole is gone and tests their draw
    // against the new threshold; later rounds search the losers, which retry.
    auto light_step = [&](int rel, bool act, int p) -> uint64_t {
        const int n = nb0 + rel;
        const uint32_t blk = (uint32_t)n >> 2;
        const int word = n & 3;
        const float xA = lane_value(l_xA, rel), b1 = lane_value(l_b1, rel), b2 = lane_value(l_b2, rel);
        const uint32_t st = act ? est[p] : 0u;
        float w = act ? ew[p] : 0.0f;
        const uint32_t o = st & 0xFFFFu;
        uint32_t nn = st >> 16;
        bool need = act && hole_f[4 * nn] == kDeadHoleX;
        bool cand = act && !need;
        bool ch = always2;
        if (two_ch) ch = channel_word(philox10(blk, o, prun, c3c, k0, k1), word);
        FireThr t{0u, false};
        bool have_t = false, have_xyz = false;
        float x = 0.0f, y = 0.0f, z = 0.0f;
        uint32_t wins = 0;
        bool won = false;
        for (int it = 0;; ++it) {
            const uint64_t nm = ballot(need);
            if (nm != 0) {
                if (!have_xyz) {
                    egen.xyz(o, x, y, z);
                    have_xyz = true;
                }
                if (it > 0 && !have_t) {
                    t = threshold(w, ch, xA, b1, b2);
                    have_t = true;
                }
                uint32_t u = 0u;
                if (it == 0) u = pick_word(philox10(blk, o, prun, c3f, k0, k1), word);
                search(nm, need, x, y, z, o, p, nn, w);
                wave_sync<GM>();
                // (the thresholds of the lanes not searched are unchanged)
                const FireThr tn = threshold(w, ch, xA, b1, b2);
                bool ok = nn != kNoHole;
                if (it == 0) ok = ok && fires(u, tn);
                else ok = ok && accepted(tn, t, blk, word, o, (uint32_t)(it - 1));
                if (need) cand = ok;
                t = tn;
                have_t = true;
            }
            const uint64_t cm = ballot(cand);
            if (cm == 0) break;
            bool win = cand;
            if ((cm & (cm - 1)) != 0) {                  // (a single candidate is not contested)
                if (cand) claim(nn, o);
                wave_sync<GM>();
                // the claim field holds the lowest candidate index for that hole
                uint32_t meta = 0u;
                if (cand) meta = hole_u[4 * nn + 3];
                win = cand && (meta >> 16) == o;
                if (win) hole_u[4 * nn + 3] = 0xFFFF0000u | (meta & 0xFFFFu);
            }
            if (win) {
                hole_f[4 * nn] = kDeadHoleX;
                est[p] = kDeadSlot;
                nf[p] = (uint8_t)kNever;
                won = true;
            }
            wins += (uint32_t)__popcll(ballot(win));
            wave_sync<GM>();
            need = cand && !win;
            cand = false;
            if (it + 1 == MCL_MAX_ROUNDS || ballot(need) == 0) break;
        }
        finish_step(n, wins);
        // the candidates that stay: their next firing step in the window
        const bool stay = act && !won;
        uint64_t more = 0;
        if (ballot(stay) != 0) {
            uint32_t f = kNever;
            if (rel + 1 < len) more = group_scan(ballot(stay && nn != kNoHole), o, w, rel + 1, f);
            if (stay) {
                nf[p] = (uint8_t)f;
                if (f != kNever) atomicOr(&rowm[p >> 6], 1ull << f);
            }
            wave_sync<GM>();
        }
        return more;
    };

    // A step with many candidates, every wave: the candidates of the wave's own rows
    // [r_lo, r_lo + nr), gathered into chunks of 64 (flags per chunk in 64-bit
    // masks).  Returns the cluster's wins.
    auto heavy_step = [&](int rel) -> uint32_t {
        const int n = nb0 + rel;
        const uint32_t blk = (uint32_t)n >> 2;
        const int word = n & 3;
        const float xA = lane_value(l_xA, rel), b1 = lane_value(l_b1, rel), b2 = lane_value(l_b2, rel);
        int r_lo = 0, nr = rows;
        if constexpr (NW > 1) {
            const int per = (rows + NW - 1) / NW;
            r_lo = min(rows, wv * per);
            nr = min(rows, r_lo + per) - r_lo;
        }
        uint16_t* const my = lst + r_lo * kWave;
        const int k = gather(rel, 1, r_lo, r_lo + nr, my, nr * kWave);
        nr = (k + kWave - 1) / kWave;    // chunks from here on
        uint64_t cand = 0;               // per chunk: this lane's candidate claims a hole
        uint32_t wins = 0, step_wins = 0;
        uint64_t todo = nr >= 64 ? ~0ull : (1ull << nr) - 1ull;   // chunks with a search or test
        uint64_t lose = 0;
        for (int round = 0;; ++round) {
            // round 0: the candidates whose hole is gone; later: the losers, retried
            cand = 0;
            uint64_t m = todo;
            while (m != 0) {
                const int r = __builtin_ctzll(m);
                m &= m - 1;
                const int q = r * kWave + lane;
                const bool is = round == 0 ? q < k : ((lose >> r) & 1ull) != 0;
                const int p = is ? (int)my[q] : 0;
                const uint32_t st = is ? est[p] : 0u;
                float w = is ? ew[p] : 0.0f;
                const uint32_t o = st & 0xFFFFu;
                uint32_t nn = st >> 16;
                bool ch = always2;
                if (two_ch) ch = channel_word(philox10(blk, o, prun, c3c, k0, k1), word);
                const bool need = round == 0 ? is && hole_f[4 * nn] == kDeadHoleX : is;
                bool ok = is;
                const uint64_t nm = ballot(need);
                if (nm != 0) {
                    float x, y, z;
                    egen.xyz(o, x, y, z);
                    const FireThr to = threshold(w, ch, xA, b1, b2);
                    search(nm, need, x, y, z, o, p, nn, w);
                    const FireThr tn = threshold(w, ch, xA, b1, b2);
                    bool good;
                    if (round == 0)
                        good = fires(pick_word(philox10(blk, o, prun, c3f, k0, k1), word), tn);
                    else
                        good = accepted(tn, to, blk, word, o, (uint32_t)(round - 1));
                    if (need) ok = nn != kNoHole && good;
                }
                if (ok) {
                    claim(nn, o);
                    cand |= 1ull << r;
                }
            }
            const uint64_t crows = rows_any(cand, nr);
            if constexpr (NW == 1) {
                if (crows == 0) break;
                wave_sync<GM>();
            } else {
                if (!any_wave(crows != 0)) break;        // also the claims' barrier
            }
            // winners: the claim field holds the lowest candidate index for that hole
            lose = 0;
            m = crows;
            while (m != 0) {
                const int r = __builtin_ctzll(m);
                m &= m - 1;
                bool win = false;
                if ((cand >> r) & 1ull) {
                    const int p = (int)my[r * kWave + lane];
                    const uint32_t st = est[p];
                    const uint32_t nn = st >> 16;
                    const uint32_t meta = hole_u[4 * nn + 3];
                    win = (meta >> 16) == (st & 0xFFFFu);
                    if (win) {
                        hole_u[4 * nn + 3] = 0xFFFF0000u | (meta & 0xFFFFu);
                        hole_f[4 * nn] = kDeadHoleX;
                        est[p] = kDeadSlot;
                    } else {
                        lose |= 1ull << r;
                    }
                }
                wins += (uint32_t)__popcll(ballot(win));
            }
            todo = rows_any(lose, nr);
            bool any_lose;
            if constexpr (NW == 1) {
                wave_sync<GM>();
                step_wins = wins;
                any_lose = todo != 0;
            } else {
                // the removed holes are visible to every wave after this barrier
                const uint32_t* x = exchange(wins | (todo != 0 ? 0x80000000u : 0u));
                uint32_t t = 0, l = 0;
#pragma unroll
                for (int w = 0; w < NW; ++w) {
                    t += x[w] & 0x7FFFFFFFu;
                    l |= x[w] >> 31;
                }
                step_wins = uniform(t);
                any_lose = uniform(l) != 0u;
            }
            if (round + 1 == MCL_MAX_ROUNDS || !any_lose) break;
        }
        // the candidates that stay: their next firing step in the window
        for (int r = 0; r < nr; ++r) {
            const int q = r * kWave + lane;
            const bool is = q < k;
            const int p = is ? (int)my[q] : 0;
            const uint32_t st = is ? est[p] : kDeadSlot;
            const float w = is ? ew[p] : 0.0f;
            uint32_t f = kNever;
            if (rel + 1 < len)
                (void)first_fire(st != kDeadSlot && (st >> 16) != kNoHole, st & 0xFFFFu, w, rel + 1, f);
            if (is) {
                nf[p] = (uint8_t)f;
                if (f != kNever) atomicOr(&rowm[p >> 6], 1ull << f);
            }
        }
        if constexpr (NW == 1) wave_sync<GM>();
        else __syncthreads();
        return step_wins;
    };

    // The electrons of rows [r_lo, r_hi) that fire in the n steps from rel0 on and whose
    // nearest hole is gone already: searched now, together, instead of one step after the
    // other.  Exact: the hole found is no farther than the one a search in the firing step
    // would find, and is that one if it still lives then (else it is searched again
    // there); an electron whose draw fails against the new threshold is scanned again.
    auto pre_search = [&](int rel0, int n_rel, int r_lo, int r_hi) {
        uint16_t* const my = lst + r_lo * kWave;
        const int k = gather(rel0, n_rel, r_lo, r_hi, my, (r_hi - r_lo) * kWave);
        for (int c0 = 0; c0 < k; c0 += kWave) {
            const bool is = c0 + lane < k;
            const int p = is ? (int)my[c0 + lane] : 0;
            const uint32_t st = is ? est[p] : 0u;
            const uint32_t o = st & 0xFFFFu;
            uint32_t nn = st >> 16;
            const bool need = is && hole_f[4 * nn] == kDeadHoleX;
            const uint64_t nm = ballot(need);
            if (nm == 0) continue;
            float x, y, z, w = 0.0f;
            egen.xyz(o, x, y, z);
            search(nm, need, x, y, z, o, p, nn, w);
            const int rel = need ? (int)nf[p] : 0;
            const int n = nb0 + rel;
            const uint32_t u = pick_word(philox10((uint32_t)n >> 2, o, prun, c3f, k0, k1), n & 3);
            bool ch = always2;
            if (two_ch) ch = channel_word(philox10((uint32_t)n >> 2, o, prun, c3c, k0, k1), n & 3);
            const FireThr t = threshold(w, ch, __shfl(l_xA, rel), __shfl(l_b1, rel), __shfl(l_b2, rel));
            const bool again = need && !(nn != kNoHole && fires(u, t));
            if (ballot(again) != 0) {
                uint32_t f = kNever;
                (void)group_scan(ballot(again && nn != kNoHole), o, w, rel + 1, f);
                if (again) {
                    nf[p] = (uint8_t)f;
                    if (f != kNever) atomicOr(&rowm[p >> 6], 1ull << f);
                }
            }
        }
        wave_sync<GM>();
    };

    // ---- windows (the step loop, simulate.py:51-92) ------------------------------
    // (NW > 1) what wave 0 publishes: {heavy step, kSearch or kNever (the window is done),
    // n_live, and the first step and end of the search; at a window's end `events`}
    uint32_t* const pub = xch + 4 * NW + 1;
    int events = kFirstEvents;           // steps with candidates between searches of all rows
    while (nb0 < step_limit && n_live > 0) {
        const int w_len = min(kWindow, step_limit - nb0);
        if (nb0 == 0 || ramp || w_len != len) {
            len = w_len;
            window_scalars();
        }
        rows = (n_slots + kWave - 1) / kWave;
        // stable compaction in place, wave 0 (an electron waiting for a new search moves
        // with its stale nearest hole)
        if ((n_live + kWave - 1) / kWave <= rows - max(1, rows >> 3)) {
            if (wv == 0) {
                int base = 0;
                for (int r = 0; r < rows; ++r) {
                    const int p = r * kWave + lane;
                    const uint32_t st = p < n_slots ? est[p] : kDeadSlot;
                    const float w = p < n_slots ? ew[p] : 0.0f;
                    const bool keep = st != kDeadSlot;
                    const uint64_t km = ballot(keep);
                    if (keep) {
                        const int q = base + lanes_below(km);
                        est[q] = st;
                        ew[q] = w;
                    }
                    base += __popcll(km);
                    wave_sync<GM>();
                }
            }
            n_slots = n_live;
            rows = (n_slots + kWave - 1) / kWave;
            __syncthreads();
        }
        // scan: the wave's own rows
        const int per = (rows + NW - 1) / NW, my_lo = min(rows, wv * per), my_hi = min(rows, my_lo + per);
        uint64_t steps = 0;              // steps of the window that may have candidates
        for (int r = my_lo; r < my_hi; ++r) {
            const int p = r * kWave + lane;
            const uint32_t st = p < n_slots ? est[p] : kDeadSlot;
            const float w = p < n_slots ? ew[p] : 0.0f;
            uint32_t f = kNever;
            const uint64_t m =
                first_fire(st != kDeadSlot && (st >> 16) != kNoHole, st & 0xFFFFu, w, 0, f);
            nf[p] = (uint8_t)f;
            if (lane == 0) rowm[r] = m;
            steps |= m;
        }
        if constexpr (NW == 1) {
            wave_sync<GM>();
        } else {
            // (each wave's from its own rows: a read of the others' rowm here would race with
            // the next window's scan when this one has no events)
            const uint32_t* x = exchange2((uint32_t)steps, (uint32_t)(steps >> 32));
            uint32_t lo = 0, hi = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                lo |= x[w];
                hi |= x[NW + w];
            }
            steps = ((uint64_t)uniform(hi) << 32) | uniform(lo);
        }

        // The events: wave 0 takes the steps one after another; the other waves wait until it
        // publishes a heavy step or a search of all rows, and take part in it.  (steps is
        // wave 0's alone from here on.)
        auto all_rows = [&](int above) {
            uint64_t s = 0;
            for (int r = lane; r < rows; r += kWave) s |= (uint64_t)rowm[r];
            steps = ((uint64_t)wave_or_u32((uint32_t)(s >> 32)) << 32) | wave_or_u32((uint32_t)s);
            steps &= above >= kWindow ? 0ull : ~0ull << above;
        };
        // the step after the next `events` of the mask
        auto events_end = [&](uint64_t m) -> int {
            for (int i = 0; i < events && m != 0; ++i) m &= m - 1;
            return m != 0 ? (int)__builtin_ctzll(m) : kWindow;
        };
        int n_ev = 0, n_cand = 0;        // light steps and candidates since the last search
        auto next_events = [&]() {
            if (n_ev == 0) return;
            const float v = (float)n_cand * (float)(n_e0 - n_live) / ((float)n_ev * (float)n_h);
            events = (int)fminf(fmaxf(kEventsPerStale / (v < 1.0f ? v : __builtin_sqrtf(v)),
                                      (float)kMinEvents), (float)kWindow);
            n_ev = 0;
            n_cand = 0;
        };
        uint32_t todo = steps != 0 ? kSearch : kNever;
        int from = steps != 0 ? (int)__builtin_ctzll(steps) : 0, to = events_end(steps);
        while (todo != kNever) {
            if (todo != kSearch) {
                const uint32_t w = heavy_step((int)todo);
                if (wv == 0) {
                    finish_step(nb0 + (int)todo, w);
                    all_rows((int)todo + 1);
                    if (n_live == 0) steps = 0;
                }
            } else if constexpr (NW > 1) {
                pre_search(from, to - from, my_lo, my_hi);
                __syncthreads();
                if (wv == 0) all_rows(from);
            }
            todo = kNever;
            if (wv == 0) {
                while (steps != 0) {
                    const int rel = __builtin_ctzll(steps);
                    if (NW > 1 && rel >= to) {
                        next_events();
                        todo = kSearch;
                        from = rel;
                        to = events_end(steps);
                        break;
                    }
                    const int k = gather(rel, 1, 0, rows, lst + e_cap, kWave);
                    if (k > kWave) {
                        todo = (uint32_t)rel;
                        break;
                    }
                    steps &= steps - 1;
                    n_ev += 1;
                    n_cand += k;
                    if (k == 0) continue;
                    steps |= light_step(rel, lane < k, lane < k ? (int)lst[e_cap + lane] : 0);
                    if (n_live == 0) {
                        steps = 0;
                        break;
                    }
                }
            }
            if constexpr (NW > 1) {
                if (todo == kNever) {    // the window is done: `events` for the next one
                    next_events();
                    to = events;
                }
                if (tid == 0) {
                    pub[0] = todo;
                    pub[1] = (uint32_t)n_live;
                    pub[2] = (uint32_t)from;
                    pub[3] = (uint32_t)to;
                }
                __syncthreads();
                todo = uniform(pub[0]);
                n_live = (int)uniform(pub[1]);
                from = (int)uniform(pub[2]);
                to = (int)uniform(pub[3]);
                if (todo == kNever) events = to;
            }
        }
        nb0 += len;
    }
    int steps_run = n_acc;               // up to the step that emptied the cluster
    if (n_live > 0) {
        lsteps += (uint64_t)n_live * (uint64_t)(step_limit - n_acc);
        steps_run = step_limit;
    }
    if (tid == 0 && bin_acc != 0u) cnt[bin] = bin_acc;
    if (a.live_steps != nullptr && tid == 0) a.live_steps[c] = lsteps;

    // (state dumps are one-wave launches only)
    if (NW == 1 && a.dump.enabled) {
        // searches deferred to a later step happen now, so the dump shows every
        // survivor's current nearest hole
        __syncthreads();
        for (int r = 0; r * kWave < n_slots; ++r) {
            const int p = r * kWave + lane;
            const uint32_t st = p < n_slots ? est[p] : kDeadSlot;
            const uint32_t nn = st >> 16;
            const bool s = nn != kNoHole && hole_f[4 * (nn != kNoHole ? nn : 0u)] == kDeadHoleX;
            float x = 0.0f, y = 0.0f, z = 0.0f;
            if (s) egen.xyz(st & 0xFFFFu, x, y, z);
            const uint64_t key = nn_resolve<WIDE>(grid, s, x, y, z, lane, dist_evals);
            if (s) {
                uint32_t slot;
                float w;
                nn_from_key(key, alpha_f, slot, w);
                est[p] = (slot << 16) | (st & 0xFFFFu);
                ew[p] = w;
            }
        }
        __syncthreads();
    }

    // lanes counted their own evaluations in the lane-private searches
    uint64_t evals_total = dist_evals;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)evals_total, off);
        const uint32_t hi = (uint32_t)__shfl_xor((int)(uint32_t)(evals_total >> 32), off);
        evals_total += ((uint64_t)hi << 32) | lo;
    }
    if constexpr (NW > 1) {
        const uint32_t* xl = exchange((uint32_t)evals_total);
        uint64_t lo_sum = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) lo_sum += xl[w];
        const uint32_t* xh = exchange((uint32_t)(evals_total >> 32));
        uint64_t hi_sum = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) hi_sum += xh[w];
        evals_total = lo_sum + (hi_sum << 32);
    }
    if (a.work != nullptr && tid == 0) {
        a.work[4 * (size_t)c] = lsteps;
        a.work[4 * (size_t)c + 1] = evals_total;
        a.work[4 * (size_t)c + 2] = (uint64_t)(n_e0 - n_live);
        a.work[4 * (size_t)c + 3] = (uint64_t)steps_run;
    }

    if (NW == 1 && a.dump.enabled) {
        const StateDump& d = a.dump;
        for (int e = lane; e < n_e0; e += kWave) {
            float x, y, z;
            egen.xyz((uint32_t)e, x, y, z);
            d.e_live[e] = 0;
            d.nn[e] = kNoHole;
            d.w[e] = 0.0f;
            d.e_xyz[3 * e] = x;
            d.e_xyz[3 * e + 1] = y;
            d.e_xyz[3 * e + 2] = z;
        }
        __syncthreads();
        for (int p = lane; p < n_slots; p += kWave) {
            const uint32_t st = est[p];
            const uint32_t o = st & 0xFFFFu, slot = st >> 16;
            if (st != kDeadSlot && o < (uint32_t)n_e0) {
                d.e_live[o] = 1;
                d.nn[o] = slot == kNoHole ? kNoHole : (hole_u[4 * slot + 3] & 0xFFFFu);
                d.w[o] = ew[p];
            }
        }
        for (int s = lane; s < n_h; s += kWave) {
            const float4 hv = hole[s];
            const uint32_t h = __float_as_uint(hv.w) & 0xFFFFu;
            if (h >= (uint32_t)n_h) continue;
            d.h_alive[h] = hv.x != kDeadHoleX;
            d.h_xyz[3 * h] = hv.x;
            d.h_xyz[3 * h + 1] = hv.y;
            d.h_xyz[3 * h + 2] = hv.z;
        }
    }
}

// One workgroup per cluster (queue == null: cluster order[blockIdx.x], or
// blockIdx.x when order is null), or persistent workgroups that take clusters
// from order[] (null: 0 .. n_order-1) through a global atomic ticket until the
// list is exhausted.  Every workgroup leaves the loop when the ticket passes
// n_order.  The global-memory form always runs persistent.
template <bool GM, bool WIDE>
__global__ __launch_bounds__(64, GM ? 2 : 1) void fixed_dt_kernel(LaunchArgs a)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    if (a.queue == nullptr) {
        const int i = blockIdx.x;
        if (i < a.n_order) run_cluster<1, GM, WIDE>(a, a.order != nullptr ? a.order[i] : i, lds_raw);
        return;
    }
    for (;;) {
        int i = 0;
        if (threadIdx.x == 0) i = (int)atomicAdd(a.queue, 1u);
        i = __shfl(i, 0);
        if (i >= a.n_order) break;
        run_cluster<1, GM, WIDE>(a, a.order != nullptr ? a.order[i] : i, lds_raw);
        __syncthreads();
    }
}

// The same with NW wavefronts per cluster (at least two waves per SIMD, so at
// most 256 VGPRs a wave, as the one-wave kernel).  The persistent ticket goes
// through LDS (the word after the exchange slots), read by every wave between
// two barriers, so all waves take the same cluster and leave the loop together.
template <int NW, bool GM, bool WIDE>
__global__ __launch_bounds__(NW * 64, 2) void fixed_dt_mw_kernel(LaunchArgs a)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    if (a.queue == nullptr) {
        const int i = blockIdx.x;
        if (i < a.n_order) run_cluster<NW, GM, WIDE>(a, a.order != nullptr ? a.order[i] : i, lds_raw);
        return;
    }
    uint32_t* const ticket =
        (GM ? (uint32_t*)lds_raw
            : (uint32_t*)(lds_raw + 16 * a.h_cap + 4 * a.g_cap +
                          fixed_dt_electron_bytes(a.e_cap))) + 4 * NW;
    for (;;) {
        if (threadIdx.x == 0) *ticket = atomicAdd(a.queue, 1u);
        __syncthreads();
        const int i = (int)uniform(*ticket);
        __syncthreads();
        if (i >= a.n_order) break;
        run_cluster<NW, GM, WIDE>(a, a.order != nullptr ? a.order[i] : i, lds_raw);
        __syncthreads();
    }
}

template <bool GM, bool WIDE>
const void* fixed_dt_fn(int waves)
{
    return waves == 8 ? (const void*)fixed_dt_mw_kernel<8, GM, WIDE>
         : waves == 4 ? (const void*)fixed_dt_mw_kernel<4, GM, WIDE>
         : waves == 2 ? (const void*)fixed_dt_mw_kernel<2, GM, WIDE>
                      : (const void*)fixed_dt_kernel<GM, WIDE>;
}

template <bool GM, bool WIDE>
hipError_t launch_fixed_dt_t(const LaunchArgs& a, int grid, unsigned lds, int waves,
                             hipStream_t stream)
{
    const dim3 g((unsigned)grid);
    if (waves == 8)
        hipLaunchKernelGGL((fixed_dt_mw_kernel<8, GM, WIDE>), g, dim3(8 * kWave), lds, stream, a);
    else if (waves == 4)
        hipLaunchKernelGGL((fixed_dt_mw_kernel<4, GM, WIDE>), g, dim3(4 * kWave), lds, stream, a);
    else if (waves == 2)
        hipLaunchKernelGGL((fixed_dt_mw_kernel<2, GM, WIDE>), g, dim3(2 * kWave), lds, stream, a);
    else
        hipLaunchKernelGGL((fixed_dt_kernel<GM, WIDE>), g, dim3(kWave), lds, stream, a);
    return hipGetLastError();
}

// Resident workgroups per CU of the NW-wave kernel with this much dynamic LDS.
template <bool GM, bool WIDE>
hipError_t fixed_dt_occupancy_t(size_t lds, int waves, int* blocks_per_cu)
{
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, fixed_dt_fn<GM, WIDE>(waves),
                                                        waves * kWave, lds);
}

// Dynamic-LDS limits of the kernels of one form.
template <bool GM, bool WIDE>
hipError_t prepare_fixed_dt_t(int bytes_one_wave, int max_lds)
{
    hipError_t e = hipSuccess;
    for (int w : {1, 2, 4, 8}) {
        int b = bytes_one_wave + fixed_dt_waves_lds(w);
        b = b < max_lds ? b : max_lds;
        if (e == hipSuccess)
            e = hipFuncSetAttribute(fixed_dt_fn<GM, WIDE>(w), hipFuncAttributeMaxDynamicSharedMemorySize, b);
    }
    return e;
}

}  // namespace mcl
