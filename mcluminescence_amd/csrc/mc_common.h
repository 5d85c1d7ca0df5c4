// mc_common.h — device pieces shared by the fixed-dt and event-mode kernels:
// coordinates from Philox words, the hole cell grid, nearest-hole searches (lane
// private, wave cooperative, full scan; every one returns the first-index argmin
// of the float32 squared distance over live holes, engine.py:113-119,168-175)
// and the per-cluster setup (Box.seed / Box._rebuild, engine.py:113-129).
#pragma once

#include "mcl_device.h"
#include "mcl_internal.h"
#include "../../include/mcl.h"

namespace mcl {

__device__ __forceinline__ float unit_coord(uint32_t word, double side)
{
    return (float)(((double)word * 0x1p-32) * side);
}

__device__ __forceinline__ int cell_of(float v, float inv_cell, int G)
{
    const int c = (int)(v * inv_cell);   // v >= 0
    return c < G ? c : G - 1;
}

__device__ __forceinline__ uint64_t hole_key(float d2, uint32_t meta, uint32_t slot)
{
    // (d2 bits, original index, slot): the min is the first-index argmin of d2
    return ((uint64_t)__float_as_uint(d2) << 32) | ((meta & 0xFFFFu) << 16) | slot;
}

__device__ __forceinline__ float sq_dist(const float4& h, float x, float y, float z)
{
    const float dx = h.x - x, dy = h.y - y, dz = h.z - z;
    return __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
}

__device__ __forceinline__ uint64_t key_of(const float4& h, float x, float y, float z, int slot)
{
    return hole_key(sq_dist(h, x, y, z), __float_as_uint(h.w), (uint32_t)slot);
}

// Distance from v to the nearest face of cells [lo, hi] that has cells beyond it.
__device__ __forceinline__ float face_gap(float v, int lo, int hi, int G, float cell)
{
    float g = __builtin_inff();
    if (lo > 0) g = v - (float)lo * cell;
    if (hi < G - 1) g = fminf(g, (float)(hi + 1) * cell - v);
    return g;
}

// Is the block minimum d2 provably below every hole outside the block?
__device__ __forceinline__ bool block_conclusive(float best_d2, float gap, float cell)
{
    const float m = gap - 1e-4f * cell;
    return m > 0.0f && best_d2 < m * m * (1.0f - 1e-5f);
}

struct Grid {
    const float4* hole;
    const uint32_t* cstart;
    int G;
    float cell, inv_cell;
    int n_h;
};

struct ElectronGen {
    uint32_t run, sim_tag, k0, k1;
    double side_nm;
    __device__ __forceinline__ void xyz(uint32_t e, float& x, float& y, float& z) const
    {
        const u32x4 o = philox10(0u, e, run, sim_tag, k0, k1);
        x = unit_coord(o.x, side_nm);
        y = unit_coord(o.y, side_nm);
        z = unit_coord(o.z, side_nm);
    }
};

constexpr int kChunk = 8;   // hole records fetched per LDS round trip in a search

// Lane-private search of the (2 RAD + 1)^3 cell block around (x, y, z).
template <int RAD>
__device__ __forceinline__ uint64_t block_search_lane(const Grid& g, float x, float y, float z,
                                                      bool& conclusive, uint64_t& evals)
{
    constexpr int W = 2 * RAD + 1;
    const int G = g.G;
    const int cx = cell_of(x, g.inv_cell, G), cy = cell_of(y, g.inv_cell, G),
              cz = cell_of(z, g.inv_cell, G);
    const int x0 = max(cx - RAD, 0), x1 = min(cx + RAD, G - 1);
    uint64_t key = ~0ull;
    // (a loop: unrolled, its nine copies at every call are most of a kernel's code)
#pragma unroll 1
    for (int k = 0; k < W * W; ++k) {
        const int zz = cz + k / W - RAD, yy = cy + k % W - RAD;
        // rows outside the grid are empty: the reads go to the nearest row inside
        const bool in = (unsigned)zz < (unsigned)G && (unsigned)yy < (unsigned)G;
        const int base = (min(max(zz, 0), G - 1) * G + min(max(yy, 0), G - 1)) * G;
        const int s = (int)g.cstart[base + x0], s1 = (int)g.cstart[base + x1 + 1];
        const int e = in ? s1 : s;
        evals += (uint64_t)(e - s);
        for (int i0 = s; i0 < e; i0 += kChunk) {
            float4 hv[kChunk];
#pragma unroll
            for (int t = 0; t < kChunk; ++t) hv[t] = g.hole[min(i0 + t, e - 1)];
#pragma unroll
            for (int t = 0; t < kChunk; ++t) {
                const uint64_t kk = key_of(hv[t], x, y, z, min(i0 + t, e - 1));
                key = kk < key ? kk : key;
            }
        }
    }
    const int y0 = max(cy - RAD, 0), y1 = min(cy + RAD, G - 1);
    const int z0 = max(cz - RAD, 0), z1 = min(cz + RAD, G - 1);
    const bool whole = x0 == 0 && y0 == 0 && z0 == 0 && x1 == G - 1 && y1 == G - 1 && z1 == G - 1;
    const float gap = fminf(face_gap(x, x0, x1, G, g.cell),
                            fminf(face_gap(y, y0, y1, G, g.cell), face_gap(z, z0, z1, G, g.cell)));
    conclusive = whole || block_conclusive(__uint_as_float((uint32_t)(key >> 32)), gap, g.cell);
    return key;
}

constexpr int kSearchBatch = 4;   // electrons searched at once by the whole wave

// The whole wave scans every hole for one electron (x, y, z wave-uniform).
__device__ __forceinline__ uint64_t full_scan_wave(const Grid& g, float x, float y, float z,
                                                   int lane, uint64_t& evals)
{
    if (lane == 0) evals += (uint64_t)g.n_h;   // evaluations are summed over lanes
    uint64_t key = ~0ull;
    for (int i = lane; i < g.n_h; i += kWave) {
        const uint64_t k = key_of(g.hole[i], x, y, z, i);
        key = k < key ? k : key;
    }
    return wave_min_u64(key);
}

// Nearest live hole of one electron (x, y, z wave-uniform) whose 3x3x3 block was
// inconclusive, by the whole wave.  WIDE: blocks of 5 and 9 cells an axis while they
// leave out most of the grid, each accepted by the same test as the 3x3x3 block,
// then every hole.  A block's (z, y) rows of cells are contiguous slot ranges; a row is
// split over two lanes (5 cells) or three (9 cells), each fetching four holes a trip.
// Not WIDE: every hole at once (kernels for small grids, without the blocks' code).
template <bool WIDE>
__device__ __forceinline__ uint64_t far_search_wave(const Grid& g, float x, float y, float z, int lane,
                                                    uint64_t& evals)
{
    const int G = g.G;
    for (int R = 2; WIDE && R <= 4 && 4 * R + 1 <= G; R += 2) {
        const int cx = cell_of(x, g.inv_cell, G), cy = cell_of(y, g.inv_cell, G),
                  cz = cell_of(z, g.inv_cell, G);
        const int x0 = max(cx - R, 0), x1 = min(cx + R, G - 1);
        const int y0 = max(cy - R, 0), y1 = min(cy + R, G - 1);
        const int z0 = max(cz - R, 0), z1 = min(cz + R, G - 1);
        const int ny = y1 - y0 + 1, parts = R == 2 ? 2 : 3;
        const int items = (z1 - z0 + 1) * ny * parts;
        uint64_t key = ~0ull;
        for (int i = lane; i < items; i += kWave) {
            const int row = i / parts, part = i - row * parts;
            const int zz = z0 + row / ny, yy = y0 + row % ny;
            const int base = (zz * G + yy) * G;
            const int s = (int)g.cstart[base + x0], e = (int)g.cstart[base + x1 + 1];
            if (part == 0) evals += (uint64_t)(e - s);
            for (int i0 = s + part; i0 < e; i0 += 4 * parts) {
                float4 hv[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) hv[t] = g.hole[min(i0 + t * parts, e - 1)];
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const uint64_t k = key_of(hv[t], x, y, z, min(i0 + t * parts, e - 1));
                    key = k < key ? k : key;
                }
            }
        }
        key = wave_min_u64(key);
        const float gap = fminf(face_gap(x, x0, x1, G, g.cell),
                                fminf(face_gap(y, y0, y1, G, g.cell), face_gap(z, z0, z1, G, g.cell)));
        if (block_conclusive(__uint_as_float((uint32_t)(key >> 32)), gap, g.cell)) return key;
    }
    return full_scan_wave(g, x, y, z, lane, evals);
}

// Nearest live hole for every active lane's electron: 3x3x3 block search per
// lane, then one wave-wide search per lane whose block was inconclusive.  (A
// lane-private 5x5x5 level in between measured slower: it is divergent, so one
// open lane makes the wave pay 25 serialized LDS round trips.)
template <bool WIDE>
__device__ __forceinline__ uint64_t nn_resolve(const Grid& g, bool act, float x, float y, float z,
                                               int lane, uint64_t& evals)
{
    bool ok = true;
    uint64_t key = ~0ull;
    if (act) key = block_search_lane<1>(g, x, y, z, ok, evals);
    uint64_t fb = ballot(act && !ok);
    while (fb != 0) {
        const int l = __builtin_ctzll(fb);
        fb &= fb - 1;
        const float fx = lane_value(x, l), fy = lane_value(y, l), fz = lane_value(z, l);
        const uint64_t k = far_search_wave<WIDE>(g, fx, fy, fz, lane, evals);
        if (lane == l) key = k;
    }
    return key;
}

// Nearest live holes for the electrons of the lanes in mask (act: the lane is one of
// them; x, y, z its electron's coordinates), each lane's key in key.  Up to
// wave_search_max electrons are searched by the whole wave, up to four at a time;
// beyond, lane-parallel.  A batch of one, two or four gives each electron 64, 32 or
// 16 lanes; its 3x3x3 block is at most 9 contiguous slot ranges (one per (z, y) row of
// cells), each shared by 7, 3 or 1 of those lanes, which fetch four holes a trip.
// (Every lane taking a slot of every range instead, nine range bounds and nine
// holes a lane, was 550 instructions a batch against 320: the bounds of one range
// cost as much as three holes.)
template <bool WIDE>
__device__ __forceinline__ void search_lanes(const Grid& g, uint64_t mask, bool act, float x, float y,
                                             float z, int wave_search_max, int lane, uint64_t& key,
                                             uint64_t& evals)
{
    if (__popcll(mask) > wave_search_max) {
        const uint64_t k = nn_resolve<WIDE>(g, act, x, y, z, lane, evals);
        if (act) key = k;
        return;
    }
    const int G = g.G;
    while (mask != 0) {
        int b[kSearchBatch];
        int nb = 0;
#pragma unroll
        for (int i = 0; i < kSearchBatch; ++i) {       // (a missing one repeats the first)
            b[i] = mask != 0 ? (int)__builtin_ctzll(mask) : b[0];
            nb += mask != 0 ? 1 : 0;
            mask = mask != 0 ? mask & (mask - 1) : 0;
        }
        const int log_l = nb == 1 ? 6 : nb == 2 ? 5 : 4;          // log2 lanes of an electron
        const int parts = nb == 1 ? 7 : nb == 2 ? 3 : 1;          // lanes of a range
        const int e = lane >> log_l, l = lane & ((1 << log_l) - 1);
        const int j = nb == 1 ? (l * 37) >> 8 : nb == 2 ? (l * 11) >> 5 : l;   // l / parts
        const float qx = e == 0 ? lane_value(x, b[0]) : e == 1 ? lane_value(x, b[1])
                       : e == 2 ? lane_value(x, b[2]) : lane_value(x, b[3]);
        const float qy = e == 0 ? lane_value(y, b[0]) : e == 1 ? lane_value(y, b[1])
                       : e == 2 ? lane_value(y, b[2]) : lane_value(y, b[3]);
        const float qz = e == 0 ? lane_value(z, b[0]) : e == 1 ? lane_value(z, b[1])
                       : e == 2 ? lane_value(z, b[2]) : lane_value(z, b[3]);
        const int cx = cell_of(qx, g.inv_cell, G), cy = cell_of(qy, g.inv_cell, G),
                  cz = cell_of(qz, g.inv_cell, G);
        const int x0 = max(cx - 1, 0), x1 = min(cx + 1, G - 1);
        const int jz = (j * 11) >> 5, zz = cz - 1 + jz, yy = cy - 1 + (j - 3 * jz);
        // range j of the unclamped block; ranges outside the grid are empty
        uint64_t k = ~0ull;
        if (j < 9 && (unsigned)zz < (unsigned)G && (unsigned)yy < (unsigned)G) {
            const int base = (zz * G + yy) * G;
            const int s0 = (int)g.cstart[base + x0], end = (int)g.cstart[base + x1 + 1];
            const int part = l - j * parts;
            if (part == 0 && e < nb) evals += (uint64_t)(end - s0);   // summed over lanes at the end
            for (int i0 = s0 + part; i0 < end; i0 += 4 * parts) {
                float4 hv[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) hv[t] = g.hole[min(i0 + t * parts, end - 1)];
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const uint64_t kt = key_of(hv[t], qx, qy, qz, min(i0 + t * parts, end - 1));
                    k = kt < k ? kt : k;
                }
            }
        }
        k = row_min_u64(k);
        const int y0 = max(cy - 1, 0), y1 = min(cy + 1, G - 1);
        const int z0 = max(cz - 1, 0), z1 = min(cz + 1, G - 1);
        const bool whole = x0 == 0 && y0 == 0 && z0 == 0 && x1 == G - 1 && y1 == G - 1 && z1 == G - 1;
        const float gap = fminf(face_gap(qx, x0, x1, G, g.cell),
                                fminf(face_gap(qy, y0, y1, G, g.cell), face_gap(qz, z0, z1, G, g.cell)));
        // the rows of 16 lanes of each electron combined
        uint64_t kr[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            kr[i] = ((uint64_t)lane_value((uint32_t)(k >> 32), 16 * i) << 32) |
                    lane_value((uint32_t)k, 16 * i);
        if (nb <= 2) {
            kr[0] = kr[1] < kr[0] ? kr[1] : kr[0];
            kr[1] = kr[3] < kr[2] ? kr[3] : kr[2];
            if (nb == 1) kr[0] = kr[1] < kr[0] ? kr[1] : kr[0];
        }
        const uint64_t own = e == 0 ? kr[0] : e == 1 ? kr[1] : e == 2 ? kr[2] : kr[3];
        const bool ok = e >= nb || whole ||
                        block_conclusive(__uint_as_float((uint32_t)(own >> 32)), gap, g.cell);
        uint64_t open = ballot(l == 0 && !ok);
#pragma unroll
        for (int i = kSearchBatch - 1; i >= 0; --i)     // (the first last: it repeats)
            if (lane == b[i]) key = i < nb ? kr[i] : kr[0];
        // electrons whose block was inconclusive
        while (open != 0) {
            const int lo = (int)__builtin_ctzll(open);
            open &= open - 1;
            const uint64_t kf = far_search_wave<WIDE>(g, lane_value(qx, lo), lane_value(qy, lo),
                                                      lane_value(qz, lo), lane, evals);
            const int i = lo >> log_l;
            if (lane == (i == 0 ? b[0] : i == 1 ? b[1] : i == 2 ? b[2] : b[3])) key = kf;
        }
    }
}

// Inclusive prefix sum of a float64 value over the 64 lanes (all active), in a
// fixed order the CPU replay repeats: within each 16-lane row, steps of 1, 2, 4
// and 8 lanes (v[l] += v[l - o] for l % 16 >= o, by DPP row shifts); then rows
// 1, 2, 3 add t0, t0 + t1 and (t0 + t1) + t2, the totals t_r of the rows before.
template <int kCtrl>
__device__ __forceinline__ double dpp_row_shift_d(double v)
{
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, kCtrl, 0xF, 0xF, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), kCtrl, 0xF,
                                                              0xF, true);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

__device__ __forceinline__ double lane_value_d(double v, int l)
{
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint64_t r = ((uint64_t)lane_value((uint32_t)(b >> 32), l) << 32) |
                       lane_value((uint32_t)b, l);
    return __longlong_as_double((long long)r);
}

__device__ __forceinline__ double row_scan_d(double v, int lane)
{
    v = v + dpp_row_shift_d<0x111>(v);    // row_shr:1 (0 shifted in)
    v = v + dpp_row_shift_d<0x112>(v);    // row_shr:2
    v = v + dpp_row_shift_d<0x114>(v);    // row_shr:4
    v = v + dpp_row_shift_d<0x118>(v);    // row_shr:8
    const double t0 = lane_value_d(v, 15), t1 = lane_value_d(v, 31), t2 = lane_value_d(v, 47);
    const double o2 = t0 + t1, o3 = o2 + t2;
    const int row = lane >> 4;
    if (row > 0) v = v + (row == 1 ? t0 : row == 2 ? o2 : o3);
    return v;
}

// The value row_scan_d leaves in lane 63 (the total of the 64 lanes), in every
// lane, without the scan's cross-row pass: the same four in-row steps, then
// ((t0 + t1) + t2) + t3 from the row totals (lane 63 holds t3 + ((t0 + t1) + t2),
// the same sum), read to scalar registers, so no LDS permute returns it.
__device__ __forceinline__ double row_total_d(double v)
{
    v = v + dpp_row_shift_d<0x111>(v);
    v = v + dpp_row_shift_d<0x112>(v);
    v = v + dpp_row_shift_d<0x114>(v);
    v = v + dpp_row_shift_d<0x118>(v);
    const double t0 = lane_value_d(v, 15), t1 = lane_value_d(v, 31), t2 = lane_value_d(v, 47),
                 t3 = lane_value_d(v, 63);
    return ((t0 + t1) + t2) + t3;
}

// w = exp(-alpha r) of a squared distance (every path computes it this one way).
__device__ __forceinline__ float w_of(uint32_t d2bits, float alpha_f)
{
    return exp_own(-(alpha_f * __builtin_sqrtf(__uint_as_float(d2bits))));
}

__device__ __forceinline__ void nn_from_key(uint64_t key, float alpha_f, uint32_t& slot, float& w)
{
    const uint32_t d2bits = (uint32_t)(key >> 32);
    const bool none = d2bits >= 0x7f800000u;        // no live hole left
    slot = none ? kNoHole : (uint32_t)(key & 0xFFFFu);
    w = none ? 0.0f : w_of(d2bits, alpha_f);
}

// Orders the LDS accesses of one wave around it, for a workgroup of one wave: a
// wavefront-scope fence for the compiler; the wave's LDS instructions execute in
// issue order.
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Bit r set iff any lane has bit r of its row mask set (rows <= 64), by ballots.
__device__ __forceinline__ uint64_t rows_any(uint64_t bits, int rows)
{
    uint64_t m = 0;
    for (int r = 0; r < rows; ++r)
        if (ballot((bits >> r) & 1ull) != 0) m |= 1ull << r;
    return m;
}

// Holes of one cluster counting-sorted by grid cell (Box.seed, engine.py:124-129)
// and every electron's initial nearest hole (Box._rebuild, engine.py:113-119):
// fills hole, cstart, est and ew.  NW wavefronts per workgroup (tid = thread
// index): the hole counts and the electrons' searches are split over the waves;
// the cell prefix, the scatter (slots within a cell in hole-index order) and the
// shift are wave 0's, between the workgroup's barriers.  Shared by the fixed-dt
// and event kernels.
template <int NW, bool WIDE>
__device__ __forceinline__ Grid setup_cluster_t(const RunDesc& R, const ElectronGen& egen,
                                                float4* hole, uint32_t* cstart, uint32_t* est,
                                                float* ew, uint32_t prun, uint32_t psim,
                                                uint32_t k0, uint32_t k1, int tid,
                                                uint64_t& dist_evals)
{
    constexpr int NT = NW * kWave;
    const int lane = NW == 1 ? tid : (tid & (kWave - 1));
    const bool w0 = NW == 1 || tid < kWave;
    const int wv = NW == 1 ? 0 : uniform(tid >> 6);
    const int n_e0 = uniform(R.n_e0);
    const int n_h = uniform(R.n_h);
    const int G = uniform(R.grid);
    const int n_cells = G * G * G;
    const float cell = R.cell_nm, inv_cell = R.inv_cell;
    // ---- holes (Box.seed, engine.py:124-129), counting-sorted by grid cell ------
    for (int i = tid; i <= n_cells; i += NT) cstart[i] = 0u;
    __syncthreads();
    for (int h = tid; h < n_h; h += NT) {
        const u32x4 o = philox10(0u, (uint32_t)h, prun, psim | MCL_TAG_GEOM_H, k0, k1);
        const float x = unit_coord(o.x, R.side_b_nm), y = unit_coord(o.y, R.side_b_nm),
                    z = unit_coord(o.z, R.side_b_nm);
        const int cc = (cell_of(z, inv_cell, G) * G + cell_of(y, inv_cell, G)) * G +
                       cell_of(x, inv_cell, G);
        atomicAdd(&cstart[cc + 1], 1u);
    }
    __syncthreads();
    if (w0) {
        uint32_t carry = 0;
        for (int base = 0; base <= n_cells; base += kWave) {
            const int i = base + lane;
            uint32_t v = i <= n_cells ? cstart[i] : 0u;
#pragma unroll
            for (int off = 1; off < kWave; off <<= 1) {
                const uint32_t u = (uint32_t)__shfl_up((int)v, off);
                if (lane >= off) v += u;
            }
            v += carry;
            if (i <= n_cells) cstart[i] = v;
            carry = (uint32_t)__shfl((int)v, kWave - 1);
        }
    }
    __syncthreads();
    if (w0) {
        for (int h = lane; h < n_h; h += kWave) {
            const u32x4 o = philox10(0u, (uint32_t)h, prun, psim | MCL_TAG_GEOM_H, k0, k1);
            const float x = unit_coord(o.x, R.side_b_nm), y = unit_coord(o.y, R.side_b_nm),
                        z = unit_coord(o.z, R.side_b_nm);
            const int cc = (cell_of(z, inv_cell, G) * G + cell_of(y, inv_cell, G)) * G +
                           cell_of(x, inv_cell, G);
            const uint32_t slot = atomicAdd(&cstart[cc], 1u);
            hole[slot] = make_float4(x, y, z, __uint_as_float(0xFFFF0000u | (uint32_t)h));
        }
    }
    __syncthreads();
    // cstart[c] now holds the end of cell c: shift right by one (top chunk first)
    for (int base = (n_cells / kWave) * kWave; base >= 0; base -= kWave) {
        const int i = base + lane;
        const uint32_t v = (w0 && i >= 1 && i <= n_cells) ? cstart[i - 1] : 0u;
        __syncthreads();
        if (w0 && i <= n_cells) cstart[i] = v;
        __syncthreads();
    }

    const Grid grid{hole, cstart, G, cell, inv_cell, n_h};
    const float alpha_f = (float)R.alpha_nm;

    // ---- electrons and their initial nearest hole (Box._rebuild, engine.py:113-119)
    const int rows0 = (n_e0 + kWave - 1) / kWave;
    for (int r = wv; r < rows0; r += NW) {
        const int e = r * kWave + lane;
        const bool act = e < n_e0;
        float x = 0.0f, y = 0.0f, z = 0.0f;
        if (act) egen.xyz((uint32_t)e, x, y, z);
        const uint64_t key = nn_resolve<WIDE>(grid, act, x, y, z, lane, dist_evals);
        if (act) {
            uint32_t slot;
            float w;
            nn_from_key(key, alpha_f, slot, w);
            est[e] = (slot << 16) | (uint32_t)e;
            ew[e] = w;
        }
    }
    __syncthreads();

    return grid;
}

template <bool WIDE>
__device__ __forceinline__ Grid setup_cluster(const RunDesc& R, const ElectronGen& egen,
                                              float4* hole, uint32_t* cstart, uint32_t* est,
                                              float* ew, uint32_t prun, uint32_t psim,
                                              uint32_t k0, uint32_t k1, int lane,
                                              uint64_t& dist_evals)
{
    return setup_cluster_t<1, WIDE>(R, egen, hole, cstart, est, ew, prun, psim, k0, k1, lane, dist_evals);
}

}  // namespace mcl
