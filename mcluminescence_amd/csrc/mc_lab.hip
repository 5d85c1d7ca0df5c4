// mc_lab.hip — the lab experiments of TLTrapSim.TL_lab / ISO_lab
// (tl_trap_lab.py:65-179): an event-mode Monte Carlo with dose filling
// (_filling_time, tl_trap_lab.py:53-60; Box.add_electron, engine.py:133-152) that
// records the trapped fraction n_e / N_e at observation times.  One wave64 per
// (experiment, sim).  Lab clusters are small (N_e ~ 100), so electrons and holes
// keep explicit float32 coordinates in LDS in creation order — the order of the
// reference's arrays, where add_electron appends and remove_pair deletes — and a
// nearest-hole search is a full wave scan (first index on ties).
//
// Step (t = time so far, float64):
//   T = (T_start + 273.15) + T_rate t; A = s e^{-E_cb/kT}, B_c = b e^{-E_loc_c/kT};
//   k_e = fma(B_ch, w_e, A) per live electron (channel as in the other kernels);
//   K summed by 64-electron row scans added in order (as the event kernel).
//   One Philox block (i, 0xFFFFFFFF, run, sim|FIRE): E_t, U_w, E_f as in the event
//   kernel.  lambda = 1e-20 if D = 0 or n_e = int(N_e), else (D/D0)(int(N_e) - n_e);
//   dt_fill = (1 / lambda) E_f; dt_rec = E_t / K (dt_fill without electrons, +inf
//   when K = 0); dt = min(dt_rec, dt_fill), no cap (tl_trap_lab.py:86-89,142-144).
//   t += dt.  dt == dt_fill: a fill — electron f of the run at Philox
//   (f, 0xFFFFFFFE, run, sim|GEOM_E) in the core cube and a hole at
//   (f, 0xFFFFFFFE, run, sim|GEOM_H) in the boundary cube.  The new electron's
//   nearest hole is searched among the holes before the new one and the other
//   electrons keep theirs (engine.py:141-152, the reference's stale update), or,
//   with exact_fill, among all holes with every electron compared against the new
//   hole.  Otherwise a recombination: the electron whose running sum first
//   exceeds U_w K goes with its nearest hole; electrons that had that hole search
//   again (engine.py:154-175).
//   After the step every observation time <= t not yet passed records n_e / N_e
//   (tl_trap_lab.py:163-172); the run ends when all are recorded.
//
// Options of the legacy lab loops (src/est_params/functions.py:270-434):
//   MCL_LAB_SHARED_CHANNEL  one channel draw per step for every electron
//                           (lifetime_fading, functions.py:115-135), word i & 3 of
//                           Philox (i >> 2, 0xFFFFFFFD, run, sim|CHAN);
//   MCL_LAB_FIRST_ELECTRON  the recombining electron is the first one in creation
//                           order that has a hole (recomber as the lab loops call it,
//                           functions.py:241-261: its np.where over a (1, n_e) mask
//                           returns row indices, all 0);
//   MCL_LAB_RETRAP          after a recombination, with probability Retrap (word w
//                           of the step block), one more pair with exact nearest
//                           holes (functions.py:328-331).
//
// The chain of steps bounds this kernel: one cluster issues some 300 vector instructions a
// step, and it takes several waves on a SIMD to keep it busy.  So whatever depends on an index
// only is evaluated for many steps or pairs at once, a lane each: the step draws 64 at a time, the
// channel draws once per Philox block and not for each of its four steps, a step's independent
// exponentials and quotients in one evaluation.  Pairs are prepared 32 at a time, two lanes each:
// coordinates and the electron's nearest hole, which then follows the holes (a new one is
// compared with all pairs to come at once, a removed one searched for again) instead of one wave
// scan and one w per pair.  Holes and electrons are arrays of coordinates, 12 bytes a hole slot
// and 18 an electron, without a table for packing the slots again: 18 clusters a CU instead of
// 12 at 100 electrons (16 by registers).  45,056 clusters of 100 electrons (88 steps each), whole
// call: 4.37 ms with a Philox block per electron and step and two per pair; 3.11 with the draws
// batched; 2.73 with the smaller layout; 2.50 with the pairs' searches batched (the vector units
// then issue 92 % of the time).  Held to 96 registers for a fifth wave a SIMD it spilled and
// measured the same.
#include "mc_common.h"

namespace mcl {

namespace {

constexpr uint32_t kFillCtr = 0xFFFFFFFEu;
constexpr uint32_t kSharedChanCtr = 0xFFFFFFFDu;

// Pairs whose electrons' nearest holes are searched at once, two lanes each (of 77 pairs a
// cluster 16 lanes of the last batch stay unused on average; with 64, a lane each, 32).
constexpr int kFillBatch = 32;


__device__ __forceinline__ double lab_exp1(uint32_t u)
{
    return -log_own(((double)u + 0.5) * 0x1p-32);
}

struct LabHoles {
    const float *x, *y, *z;
};

// First-index nearest live hole among slots [0, n) for the point (x, y, z):
// returns (d2 bits << 32 | slot), d2 = +inf (no live hole) as 0x7f800000.
__device__ __forceinline__ uint64_t lab_nearest(const LabHoles& hole, int n, float x, float y,
                                                float z, int lane)
{
    // a lane's slots ascend, so a strictly smaller distance is the smaller key
    float best = __builtin_inff();
    uint32_t at = 0xFFFFFFFFu;
    auto take = [&](int s, float hx, float hy, float hz) {
        const float dx = hx - x, dy = hy - y, dz = hz - z;
        const float d2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
        const bool closer = hx != kDeadHoleX && d2 < best;
        best = closer ? d2 : best;
        at = closer ? (uint32_t)s : at;
    };
    int s = lane;
    for (; s + kWave < n; s += 2 * kWave) {
        const float xa = hole.x[s], ya = hole.y[s], za = hole.z[s];
        const float xb = hole.x[s + kWave], yb = hole.y[s + kWave], zb = hole.z[s + kWave];
        take(s, xa, ya, za);
        take(s + kWave, xb, yb, zb);
    }
    if (s < n) take(s, hole.x[s], hole.y[s], hole.z[s]);
    return wave_min_u64(((uint64_t)__float_as_uint(best) << 32) | at);
}

// The same for every lane's own point at once: each lane scans all n slots (the
// lanes read the same slot together, one LDS broadcast), the same key per
// (point, slot) as lab_nearest, so the same minimum.
__device__ __forceinline__ uint64_t lab_nearest_own(const LabHoles& hole, int n, float x, float y,
                                                    float z)
{
    uint64_t key = ~0ull;
    for (int s = 0; s < n; ++s) {
        const float hx = hole.x[s];
        const float dx = hx - x, dy = hole.y[s] - y, dz = hole.z[s] - z;
        const float d2 = hx == kDeadHoleX ? __builtin_inff()
                                          : __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
        const uint64_t k = ((uint64_t)__float_as_uint(d2) << 32) | (uint32_t)s;
        key = k < key ? k : key;
    }
    return key;
}

}  // namespace

__device__ __forceinline__ void run_cluster_lab(const LabArgs& a, const int c,
                                                unsigned char* lds_raw)
{
    const int lane = (int)threadIdx.x;
    const int run = uniform(a.c_run[c]);
    const int sim = uniform(a.c_sim[c]);
    const RunDesc& R = a.runs[run];
    const int h_cap = a.h_cap, e_cap = a.e_cap;
    double* rtot = (double*)lds_raw;                  // [e_cap / 64] row sums
    float* hx = (float*)(rtot + e_cap / kWave);       // [h_cap] hole coordinates, creation order
    float* hy = hx + h_cap;
    float* hz = hy + h_cap;
    float* ex = hz + h_cap;                           // [e_cap] electrons, creation order
    float* ey = ex + e_cap;
    float* ez = ey + e_cap;
    float* ew = ez + e_cap;
    uint16_t* enn = (uint16_t*)(ew + e_cap);          // [e_cap] nearest hole slot
    const LabHoles hole{hx, hy, hz};

    const uint32_t k0 = a.key0, k1 = a.key1;
    const uint32_t prun = (uint32_t)R.run_id;
    const uint32_t psim = (uint32_t)sim << 4;
    const float alpha_f = (float)R.alpha_nm;
    const int N_int = (int)R.N_e;

    // ---- seed (Box.seed, engine.py:124-129) --------------------------------------
    int n_e = uniform(R.n_e0);
    int n_hs = uniform(R.n_h);                        // hole slots in use (live or dead)
    for (int h = lane; h < n_hs; h += kWave) {
        const u32x4 o = philox10(0u, (uint32_t)h, prun, psim | MCL_TAG_GEOM_H, k0, k1);
        hx[h] = unit_coord(o.x, R.side_b_nm);
        hy[h] = unit_coord(o.y, R.side_b_nm);
        hz[h] = unit_coord(o.z, R.side_b_nm);
    }
    for (int e = lane; e < n_e; e += kWave) {
        const u32x4 o = philox10(0u, (uint32_t)e, prun, psim | MCL_TAG_GEOM_E, k0, k1);
        ex[e] = unit_coord(o.x, R.side_nm);
        ey[e] = unit_coord(o.y, R.side_nm);
        ez[e] = unit_coord(o.z, R.side_nm);
    }
    __syncthreads();
    // initial nearest holes (Box._rebuild, engine.py:113-119), one electron a lane
    for (int e = lane; e < n_e; e += kWave) {
        const uint64_t key = lab_nearest_own(hole, n_hs, ex[e], ey[e], ez[e]);
        uint32_t slot;
        float w;
        nn_from_key(key, alpha_f, slot, w);
        enn[e] = (uint16_t)slot;
        ew[e] = w;
    }
    __syncthreads();

    const bool two_ch = R.two_channel != 0;
    const bool always2 = R.always_chan2 != 0;
    const bool exact_fill = (a.options & MCL_LAB_EXACT_FILL) != 0;
    const bool shared_ch = two_ch && (a.options & MCL_LAB_SHARED_CHANNEL) != 0;
    const bool own_ch = two_ch && !shared_ch;
    const bool first_e = (a.options & MCL_LAB_FIRST_ELECTRON) != 0;
    const bool retrap = (a.options & MCL_LAB_RETRAP) != 0;
    const uint64_t ret_thr = R.ret_thr;
    const uint32_t c3f = psim | MCL_TAG_FIRE, c3c = psim | MCL_TAG_CHAN;
    const double* obs = a.obs + a.obs_offset[run];
    const int n_obs = a.obs_count[run];
    double* out = a.ratio + (size_t)c * (size_t)a.max_obs;

    double t = 0.0;
    int i = 0, k_obs = 0, fills = 0;
    int32_t status = 0;
    uint64_t lsteps = 0, recomb = 0;
    // The step draws depend on the step index only: lane j holds those of step
    // sb_base + j (E_t, U_w, E_f and the retrap word, each computed as the step
    // would), 64 steps in one parallel evaluation; a step reads its own with
    // scalar reads.
    int sb_base = -kWave;
    uint32_t l_uw = 0u, l_rw = 0u, l_ch = 0u;
    double l_et = 0.0, l_ef = 0.0;
    // The channel draws of a row's slots serve the four steps of a Philox block: a nibble of a
    // lane's word for each of up to 8 rows, those from row ch_row0 on, ch_rows of them, in
    // block ch_blk.
    constexpr int kChanRows = 8;
    uint32_t l_chan = 0u, ch_blk = 0xFFFFFFFFu;
    int ch_row0 = 0, ch_rows = 0;
    // Lanes j and j + 32 hold the pair of fill fb_base + j: its coordinates, and for its electron
    // the nearest of the holes there are now (squared distance, slot, w), which follow the holes
    // until the pair is used.
    int fb_base = -kFillBatch;
    float f_ex = 0.f, f_ey = 0.f, f_ez = 0.f, f_hx = 0.f, f_hy = 0.f, f_hz = 0.f;
    float f_d2 = __builtin_inff(), f_w = 0.f;
    uint32_t f_at = kNoHole;
    const double dose = R.D / R.D0;
    const double T0 = R.T0_K, T_rate = R.T_rate, k_b = R.k_b;
    const bool no_dose = R.D == 0.0;
    double next_obs = obs[0];
    // E of the factor that lane 0 (A), 1 (B1) or 2 (B2) evaluates, and what precedes it
    const double l_E = lane == 0 ? R.E_cb : lane == 1 ? R.E_loc_1 : R.E_loc_2;
    const double l_pre = lane == 0 ? R.s : R.b;
    while (k_obs < n_obs) {
        if ((int64_t)i >= a.max_steps) {
            status = -1;
            break;
        }
        lsteps += (uint64_t)n_e;
        const double T = T0 + T_rate * t;
        const double kT = k_b * T;
        // the three factors at once, a lane each
        const double l_fac = l_pre * exp_own(-(l_E / kT));
        const double A = lane_value_d(l_fac, 0), B1 = lane_value_d(l_fac, 1),
                     B2 = lane_value_d(l_fac, 2);
        const uint32_t blk = (uint32_t)i >> 2;
        const int word = i & 3;
        const int rows = (n_e + kWave - 1) / kWave;
        if (i - sb_base >= kWave) {
            const u32x4 o = philox10((uint32_t)(i + lane), 0xFFFFFFFFu, prun, c3f, k0, k1);
            l_et = lab_exp1(o.x);
            l_uw = o.y;
            l_ef = lab_exp1(o.z);
            l_rw = o.w;
            if (shared_ch)
                l_ch = pick_word(philox10((uint32_t)(i + lane) >> 2, kSharedChanCtr, prun, c3c, k0, k1),
                                 (i + lane) & 3);
            sb_base = i;
        }
        const int js = i - sb_base;
        const bool ch_step = shared_ch ? (uint64_t)lane_value(l_ch, js) < ret_thr : always2;
        // the channel draws of row r (and of the rows of its group) are in l_chan
        auto channels = [&](int r) {
            if (!own_ch) return;
            const int r0 = r & ~(kChanRows - 1);
            const int n = rows - r0 < kChanRows ? rows - r0 : kChanRows;
            if (blk == ch_blk && r0 == ch_row0 && n <= ch_rows) return;
            l_chan = 0u;
            for (int q = 0; q < n; ++q) {
                const u32x4 o = philox10(blk, (uint32_t)((r0 + q) * kWave + lane), prun, c3c, k0, k1);
                const uint32_t m = ((uint64_t)o.x < ret_thr ? 1u : 0u) | ((uint64_t)o.y < ret_thr ? 2u : 0u) |
                                   ((uint64_t)o.z < ret_thr ? 4u : 0u) | ((uint64_t)o.w < ret_thr ? 8u : 0u);
                l_chan |= m << (4 * q);
            }
            ch_blk = blk;
            ch_row0 = r0;
            ch_rows = n;
        };
        // k_e of a lane's slot of row r, 0 past the live ones and for electrons with no hole;
        // branch-free: every slot of a row lies within e_cap, so the reads are in
        // bounds, and the selects drop what the slots past n_e hold
        auto rate_of = [&](int r) -> double {
            const int p = r * kWave + lane;
            const uint32_t nn = enn[p];
            const float w = ew[p];
            const bool ch = own_ch ? ((l_chan >> (4 * (r & (kChanRows - 1)) + word)) & 1u) != 0u : ch_step;
            const double k = __builtin_fma(ch ? B2 : B1, (double)w, A);
            return p < n_e && nn != kNoHole ? k : 0.0;
        };
        // one electron-hole pair (Box.add_electron); false when the cluster is full
        auto add_pair = [&](bool exact) -> bool {
            if (n_e >= e_cap) return false;
            if (n_hs >= h_cap) {
                // stable compaction of the hole slots (creation order kept), 64 at a time; the
                // electrons of those holes (live ones: an electron whose hole goes is searched
                // again) take the new slots, which the later slots' test does not see again
                int base = 0;
                for (int s0 = 0; s0 < n_hs; s0 += kWave) {
                    const int s = s0 + lane;
                    const int sr = s < n_hs ? s : 0;
                    const float vx = hx[sr], vy = hy[sr], vz = hz[sr];
                    const bool live = s < n_hs && vx != kDeadHoleX;
                    const uint64_t m = ballot(live);
                    const int q = base + lanes_below(m);
                    wave_lds_fence();
                    if (live) {
                        hx[q] = vx;
                        hy[q] = vy;
                        hz[q] = vz;
                    }
                    const int fn = (int)f_at - s0;
                    if (fn >= 0 && fn < kWave && f_at != kNoHole)
                        f_at = (uint32_t)(base + __popcll(m & ((1ull << fn) - 1)));
                    for (int e = lane; e < n_e; e += kWave) {
                        const int nn = (int)enn[e] - s0;
                        if (nn >= 0 && nn < kWave && enn[e] != kNoHole)
                            enn[e] = (uint16_t)(base + __popcll(m & ((1ull << nn) - 1)));
                    }
                    wave_lds_fence();
                    base += __popcll(m);
                }
                n_hs = base;
                if (n_hs >= h_cap) return false;
            }
            if (fills - fb_base >= kFillBatch) {
                const uint32_t f = (uint32_t)(fills + (lane & (kFillBatch - 1)));
                const u32x4 oe = philox10(f, kFillCtr, prun, psim | MCL_TAG_GEOM_E, k0, k1);
                const u32x4 oh = philox10(f, kFillCtr, prun, psim | MCL_TAG_GEOM_H, k0, k1);
                f_ex = unit_coord(oe.x, R.side_nm);
                f_ey = unit_coord(oe.y, R.side_nm);
                f_ez = unit_coord(oe.z, R.side_nm);
                f_hx = unit_coord(oh.x, R.side_b_nm);
                f_hy = unit_coord(oh.y, R.side_b_nm);
                f_hz = unit_coord(oh.z, R.side_b_nm);
                fb_base = fills;
                // each of a pair's two lanes takes every other hole (its slots ascend, so a strictly
                // smaller distance is the smaller key)
                f_d2 = __builtin_inff();
                f_at = kNoHole;
#pragma unroll 4        // (four trips' reads in flight)
                for (int s = lane / kFillBatch; s < n_hs; s += 2) {
                    const float dx = hx[s] - f_ex, dy = hy[s] - f_ey, dz = hz[s] - f_ez;
                    const float d2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
                    const bool closer = d2 < f_d2;         // (a removed hole's is infinite)
                    f_d2 = closer ? d2 : f_d2;
                    f_at = closer ? (uint32_t)s : f_at;
                }
                const float od2 = __shfl_xor(f_d2, kFillBatch, kWave);
                const uint32_t oat = (uint32_t)__shfl_xor((int)f_at, kFillBatch, kWave);
                const bool other = od2 < f_d2 || (od2 == f_d2 && oat < f_at);
                f_d2 = other ? od2 : f_d2;
                f_at = other ? oat : f_at;
                f_w = f_at == kNoHole ? 0.0f : w_of(__float_as_uint(f_d2), alpha_f);
            }
            const int jf = fills - fb_base;
            const float px = lane_value(f_ex, jf), py = lane_value(f_ey, jf),
                        pz = lane_value(f_ez, jf);
            const float nx = lane_value(f_hx, jf), ny = lane_value(f_hy, jf),
                        nz = lane_value(f_hz, jf);
            const int hs = n_hs;
            // the new electron's nearest hole: before the new hole (reference) or all
            uint32_t slot = lane_value(f_at, jf);
            float w = lane_value(f_w, jf);
            // the new hole (the last slot: it wins only when strictly closer)
            if (lane == jf) {
                hx[hs] = f_hx;
                hy[hs] = f_hy;
                hz[hs] = f_hz;
            }
            wave_lds_fence();
            {
                const float dx = nx - f_ex, dy = ny - f_ey, dz = nz - f_ez;
                const float d2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
                const bool closer = d2 < f_d2;
                if (ballot(closer) != 0) {
                    f_d2 = closer ? d2 : f_d2;
                    f_at = closer ? (uint32_t)hs : f_at;
                    f_w = closer ? w_of(__float_as_uint(d2), alpha_f) : f_w;
                }
            }
            if (exact) {
                slot = lane_value(f_at, jf);
                w = lane_value(f_w, jf);
            }
            if (exact) {
                // existing electrons: the new hole wins only when strictly closer
                for (int e = lane; e < n_e; e += kWave) {
                    const float x = ex[e], y = ey[e], z = ez[e];
                    const uint32_t s0 = enn[e];
                    const float dx = nx - x, dy = ny - y, dz = nz - z;
                    const float d2n = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
                    float d2o = __builtin_inff();
                    if (s0 != kNoHole) {
                        const float ox = hx[s0] - x, oy = hy[s0] - y, oz = hz[s0] - z;
                        d2o = __builtin_fmaf(oz, oz, __builtin_fmaf(oy, oy, ox * ox));
                    }
                    if (d2n < d2o) {
                        enn[e] = (uint16_t)hs;
                        ew[e] = w_of(__float_as_uint(d2n), alpha_f);
                    }
                }
            }
            wave_lds_fence();
            if (lane == 0) {
                ex[n_e] = px;
                ey[n_e] = py;
                ez[n_e] = pz;
                ew[n_e] = w;
                enn[n_e] = (uint16_t)slot;
            }
            wave_lds_fence();
            n_e += 1;
            n_hs += 1;
            fills += 1;
            return true;
        };
        double K = 0.0;
        // row totals (the scan's lane-63 values), two rows at a time (independent
        // chains), added in order
        int r = 0;
        for (; r + 1 < rows; r += 2) {
            channels(r);
            const double ra = row_total_d(rate_of(r));
            const double rb = row_total_d(rate_of(r + 1));
            if (lane == 0) {
                rtot[r] = ra;
                rtot[r + 1] = rb;
            }
            K = K + ra;
            K = K + rb;
        }
        if (r < rows) {
            channels(r);
            const double rt = row_total_d(rate_of(r));
            if (lane == 0) rtot[r] = rt;
            K = K + rt;
        }
        wave_lds_fence();
        const double lam = (no_dose || n_e == N_int) ? 1e-20
                                                         : dose * (double)(N_int - n_e);
        // the step's two quotients at once: 1 / lam in lane 0, E_t / K in lane 1
        const double e_t = lane_value_d(l_et, js);
        const double quo = (lane == 0 ? 1.0 : e_t) / (lane == 0 ? lam : K);
        const double dt_fill = lane_value_d(quo, 0) * lane_value_d(l_ef, js);
        double dt_rec = dt_fill;
        if (n_e > 0) dt_rec = K > 0.0 ? lane_value_d(quo, 1) : __builtin_inf();
        const double dt = fmin(dt_rec, dt_fill);
        t += dt;
        if (dt == dt_fill) {
            // ---- filling: one electron-hole pair (Box.add_electron) ------------
            if (!add_pair(exact_fill)) {
                status = -2;
                break;
            }
        } else if (dt == dt_rec) {
            // ---- recombination (Box.remove_pair) --------------------------------
            int pw = -1;
            if (first_e) {
                for (int r = 0; r < rows && pw < 0; ++r) {
                    const int p = r * kWave + lane;
                    const uint64_t m = ballot(p < n_e && enn[p] != kNoHole);
                    if (m != 0) pw = r * kWave + (int)__builtin_ctzll(m);
                }
            } else {
                const double target = (double)lane_value(l_uw, js) * 0x1p-32 * K;
                double carry = 0.0;
                for (int r = 0; r < rows; ++r) {
                    const double c2 = carry + rtot[r];
                    if (c2 > target) {
                        channels(r);
                        const double v = row_scan_d(rate_of(r), lane);
                        const uint64_t m = ballot(carry + v > target);
                        pw = r * kWave + (int)__builtin_ctzll(m);
                        break;
                    }
                    carry = c2;
                }
            }
            if (pw < 0) {
                for (int r = rows - 1; r >= 0 && pw < 0; --r) {
                    channels(r);
                    const uint64_t m = ballot(rate_of(r) > 0.0);
                    if (m != 0) pw = r * kWave + 63 - (int)__builtin_clzll(m);
                }
            }
            pw = uniform(pw);
            const uint32_t hw = enn[pw];
            if (lane == 0) hx[hw] = kDeadHoleX;
            // electrons after pw move down one slot (np.delete keeps the order)
            for (int r0 = 0; r0 < n_e; r0 += kWave) {
                const int p = r0 + lane;
                const bool mv = p > pw && p < n_e;
                const int pr = mv ? p : 0;
                const float vx = ex[pr], vy = ey[pr], vz = ez[pr], vw = ew[pr];
                const uint16_t nv = enn[pr];
                wave_lds_fence();
                if (mv) {
                    ex[p - 1] = vx;
                    ey[p - 1] = vy;
                    ez[p - 1] = vz;
                    ew[p - 1] = vw;
                    enn[p - 1] = nv;
                }
                wave_lds_fence();
            }
            n_e -= 1;
            recomb += 1;
            // the electrons whose nearest hole was hw, found row by row by a ballot, each
            // searched by the whole wave (the holes do not change meanwhile, so the
            // order of the searches does not matter)
            for (int r0 = 0; r0 < n_e; r0 += kWave) {
                uint64_t m = ballot(r0 + lane < n_e && enn[r0 + lane] == hw);
                while (m != 0) {
                    const int e = r0 + (int)__builtin_ctzll(m);
                    m &= m - 1;
                    const uint64_t key = lab_nearest(hole, n_hs, ex[e], ey[e], ez[e], lane);
                    if (lane == 0) {
                        uint32_t slot;
                        float w;
                        nn_from_key(key, alpha_f, slot, w);
                        enn[e] = (uint16_t)slot;
                        ew[e] = w;
                    }
                }
            }
            // and so are the pairs to come
            uint64_t mf = ballot(f_at == hw && (lane & (kFillBatch - 1)) >= fills - fb_base) &
                          ((1ull << kFillBatch) - 1);
            while (mf != 0) {
                const int j = (int)__builtin_ctzll(mf);
                mf &= mf - 1;
                const uint64_t key = lab_nearest(hole, n_hs, lane_value(f_ex, j), lane_value(f_ey, j),
                                                 lane_value(f_ez, j), lane);
                if ((lane & (kFillBatch - 1)) == j) {
                    f_d2 = __uint_as_float((uint32_t)(key >> 32));
                    nn_from_key(key, alpha_f, f_at, f_w);
                }
            }
            wave_lds_fence();
            // legacy retrapping: a new pair after the recombination
            if (retrap && (uint64_t)lane_value(l_rw, js) < R.retrap_thr && !add_pair(true)) {
                status = -2;
                break;
            }
        }
        ++i;
        while (k_obs < n_obs && t >= next_obs) {
            if (lane == 0) out[k_obs] = (double)n_e / R.N_e;
            ++k_obs;
            if (k_obs < n_obs) next_obs = obs[k_obs];
        }
    }
    for (int k = k_obs + lane; k < a.max_obs; k += kWave) out[k] = 0.0;
    if (lane == 0) {
        a.status[c] = status;
        if (a.work != nullptr) {
            a.work[4 * (size_t)c] = lsteps;
            a.work[4 * (size_t)c + 1] = (uint64_t)fills;
            a.work[4 * (size_t)c + 2] = recomb;
            a.work[4 * (size_t)c + 3] = (uint64_t)i;
        }
    }
}

__global__ __launch_bounds__(64, 4) void lab_kernel(LabArgs a)
{
    extern __shared__ __align__(16) unsigned char lds_raw[];
    if ((int)blockIdx.x < a.n_clusters) run_cluster_lab(a, (int)blockIdx.x, lds_raw);
}

int lab_lds_bytes(int h_cap, int e_cap)
{
    return 8 * (e_cap / kWaveHost) + 12 * h_cap + 18 * e_cap;
}

int lab_capacity_bytes(int h_cap, int e_cap)
{
    return 20 * h_cap + 20 * e_cap + 8 * (e_cap / kWaveHost);
}

hipError_t prepare_lab(int lds_bytes)
{
    return hipFuncSetAttribute((const void*)lab_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                               lds_bytes);
}

hipError_t launch_lab(const LabArgs& a, int lds_bytes, hipStream_t stream)
{
    hipLaunchKernelGGL(lab_kernel, dim3((unsigned)a.n_clusters), dim3(kWave), (unsigned)lds_bytes,
                       stream, a);
    return hipGetLastError();
}

}  // namespace mcl
