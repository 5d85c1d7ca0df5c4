// de.hip — kernels of the network-scored differential evolution: the population
// of the surrogate-assisted fit lives in device memory, and a generation runs
// with no host round trip.
//
// Two forms of a generation, with identical results:
//   - fused (de_generation_kernel): one kernel.  A workgroup takes 4, 8 or 16
//     members: their trials, the whole network forward with the activations in LDS
//     and the weights read from L2 straight into matrix-core registers, the
//     objectives and the selection; 16 waves, one 32-wide output tile each, so
//     for networks whose layers are at most 512 wide.  The matrix-core tiles are
//     32 rows: the members' and zero rows, whose outputs no epilogue computes.
//     What bounds it: every CU streams the whole weight set (1.9 MB at 64 B a cycle,
//     29.8 k cycles of the kernel's 39 k with 8 members: the hidden layers run at
//     that rate), so the members are spread over more CUs until those contend for
//     the L2s; the rest is the start (arguments, keys and partner rows, the best
//     member's row: three trips to memory one after another, 6 k cycles) and the
//     objectives (2 k).  The weights are read from a copy in fragment order
//     (de_pack_kernel, made when the search is created), so that one load
//     instruction of a wave reads 1 KB of contiguous memory instead of 32 bytes of
//     32 rows.
//   - layered: a propose kernel that writes the trials into the network's packed
//     BF16 input rows, the network's own GEMM kernels (mlp.hip), and a
//     score-and-accept kernel.
// Both run the same matrix-core products in the same K order with the same
// roundings (BF16 activations, the same SiLU), and the same objective sum.
//
// The population is double-buffered: a generation reads members and argmin keys
// from (x, keys) and writes the selected members and their keys to (x_next,
// keys_next), so a trial never reads a partner that another workgroup of the same
// generation has already replaced.
//
// DE/rand-to-best/1/bin, the step of scipy's differential_evolution that the
// reference's fit calls (src/class/optimizer.py:98-111):
//   mutant  = x_a + F (x_best - x_a) + F (x_b - x_c), a, b, c distinct and != i
//   trial_j = mutant_j if U_j < CR or j == j_rand, else x_ij
//   a coordinate outside [-1, 1] is redrawn uniformly
//   the trial replaces x_i when its objective is not worse.
// Draws: Philox4x32-10 with key = seed, counter = (generation, member, block, 0).
#include "mcl_device.h"
#include "mlp_internal.h"

namespace mcl {
namespace mlp {
namespace {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr uint32_t kInitGen = 0xFFFFFFFFu;   // counter word 0 of the initial population
constexpr int kRows = 32;                    // rows of the fused kernel's matrix-core tiles
constexpr int kMembers = 16;                 // members of a workgroup at other shapes
constexpr int kFusedThreads = 1024;          // its 16 waves: one 32-wide output tile each

__device__ __forceinline__ float unit_f(uint32_t w) { return ((float)(w >> 8) + 0.5f) * 0x1p-24f; }

// uniform integer in [0, n) from one 32-bit word (n < 2^31)
__device__ __forceinline__ uint32_t below(uint32_t w, uint32_t n)
{
    return (uint32_t)(((uint64_t)w * n) >> 32);
}

__global__ __launch_bounds__(256) void de_init_kernel(DeArgs a)
{
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= a.pop_pad) return;
    float* X = a.X + (int64_t)i * a.n_in;
    if (i >= a.pop) {
        for (int j = 0; j < a.n_in; ++j) X[j] = 0.0f;   // padding rows of the forward batch
        return;
    }
    const u32x4 w0 = philox10(kInitGen, (uint32_t)i, 0u, 0u, a.key0, a.key1);
    const u32x4 w1 = philox10(kInitGen, (uint32_t)i, 1u, 0u, a.key0, a.key1);
    for (int j = 0; j < a.dim; ++j) {
        const uint32_t w = j < 4 ? pick_word(w0, j) : pick_word(w1, j - 4);
        const float v = 2.0f * unit_f(w) - 1.0f;
        X[j] = v;
        a.x[(int64_t)i * a.dim + j] = v;
    }
    for (int k = 0; a.dim + k < a.n_in; ++k) X[a.dim + k] = a.fixed[k];
    a.f[i] = __builtin_inff();
}

// Population argmin from the members' keys (objective bits << 32 | member; the
// objectives are >= 0, so their float bits order as the values, and ties go to
// the lowest member), reduced by each workgroup of NT threads: a strided minimum
// per thread (k: its first key, first_key), then across the wave and, through LDS,
// across the waves.
__device__ __forceinline__ uint64_t first_key(const DeArgs& a)
{
    // (threads past the population repeat its last key)
    return a.keys[(int)threadIdx.x < a.pop ? (int)threadIdx.x : a.pop - 1];
}

template <int NT>
__device__ __forceinline__ int population_argmin(const DeArgs& a, uint64_t k)
{
    __shared__ uint64_t wmin[NT / 64];
    for (int j = (int)threadIdx.x + NT; j < a.pop; j += NT) k = a.keys[j] < k ? a.keys[j] : k;
    k = wave_min_u64(k);
    if ((threadIdx.x & 63u) == 0u) wmin[threadIdx.x >> 6] = k;
    lds_barrier();
    const int lane = (int)(threadIdx.x & 63u);
    return (int)(uint32_t)wave_min_u64(lane < NT / 64 ? wmin[lane] : ~0ull);
}

// The members that member i (< pop) is crossed with, three distinct offsets in [1, P) from
// one Philox block's words: they differ from i and from one another.
struct Partners {
    uint32_t a, b, c;
};

__device__ __forceinline__ Partners partners(uint32_t rx, uint32_t ry, uint32_t rz, uint32_t P)
{
    const uint32_t oa = 1u + below(rx, P - 1u);
    uint32_t ob = 1u + below(ry, P - 2u);
    ob += ob >= oa ? 1u : 0u;
    uint32_t oc = 1u + below(rz, P - 3u);
    const uint32_t lo = oa < ob ? oa : ob, hi = oa < ob ? ob : oa;
    oc += oc >= lo ? 1u : 0u;
    oc += oc >= hi ? 1u : 0u;
    return {oa, ob, oc};
}

// A coordinate of the trial: mutant, crossover, and the redraw of one outside [-1, 1].
__device__ __forceinline__ float trial_coord(const DeArgs& a, float xi, float x0, float x1, float x2,
                                             float xb, bool always, uint32_t uc, uint32_t ud)
{
    const float m = x0 + a.F * (xb - x0) + a.F * (x1 - x2);
    const float v = unit_f(uc) < a.CR || always ? m : xi;
    return v < -1.0f || v > 1.0f ? 2.0f * unit_f(ud) - 1.0f : v;
}

// The trial of member i by one lane, for the layered form: its searched coordinates into
// t[0 .. dim) and the network's input row into in[16] (trials, fixed inputs, zeros).
__device__ __forceinline__ void propose_member(const DeArgs& a, int i, int best, uint32_t gen,
                                               float* t, float (&in)[16])
{
    const uint32_t P = (uint32_t)a.pop;
    const u32x4 r = philox10(gen, (uint32_t)i, 0u, 0u, a.key0, a.key1);
    const Partners o = partners(r.x, r.y, r.z, P);
    const int jr = (int)below(r.w, (uint32_t)a.dim);     // it always crosses over
    const float* xi = a.x + (int64_t)i * a.dim;
    const float* x0 = a.x + (int64_t)((i + o.a) % P) * a.dim;
    const float* x1 = a.x + (int64_t)((i + o.b) % P) * a.dim;
    const float* x2 = a.x + (int64_t)((i + o.c) % P) * a.dim;
    const float* xb = a.x + (int64_t)best * a.dim;
    const u32x4 c0 = philox10(gen, (uint32_t)i, 1u, 0u, a.key0, a.key1);   // crossover
    const u32x4 c1 = philox10(gen, (uint32_t)i, 2u, 0u, a.key0, a.key1);
    const u32x4 d0 = philox10(gen, (uint32_t)i, 3u, 0u, a.key0, a.key1);   // redraws
    const u32x4 d1 = philox10(gen, (uint32_t)i, 4u, 0u, a.key0, a.key1);
    float tv[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        tv[j] = 0.0f;
        if (j >= a.dim) continue;
        tv[j] = trial_coord(a, xi[j], x0[j], x1[j], x2[j], xb[j], j == jr,
                            j < 4 ? pick_word(c0, j) : pick_word(c1, j - 4),
                            j < 4 ? pick_word(d0, j) : pick_word(d1, j - 4));
        t[j] = tv[j];
    }
#pragma unroll
    for (int k = 0; k < 16; ++k)
        in[k] = k < a.dim ? tv[k & 7] : (k < a.n_in ? a.fixed[k - a.dim] : 0.0f);
}

// The same trial with a lane a coordinate, eight lanes a member, for the fused kernel: each
// lane draws one Philox block, and the words it needs come from its member's lanes.
struct CoordTrial {
    uint32_t uc, ud;            // crossover and redraw words of the coordinate
    int jr;                     // the coordinate that always crosses over
    float xi, x0, x1, x2;
};

// threads that form trials: whole waves, so that every lane of a shuffle is there
template <int M>
constexpr int kTrialThreads = 8 * M < 64 ? 64 : 8 * M;

__device__ __forceinline__ uint32_t word_of(const u32x4& o, int src, int word)
{
    const u32x4 v{(uint32_t)__shfl((int)o.x, src, 64), (uint32_t)__shfl((int)o.y, src, 64),
                  (uint32_t)__shfl((int)o.z, src, 64), (uint32_t)__shfl((int)o.w, src, 64)};
    return pick_word(v, word);
}

// (i < pop; lanes with j past the last coordinate repeat it)
__device__ __forceinline__ void coord_fetch(const DeArgs& a, int i, int j, uint32_t gen, CoordTrial& T)
{
    const int jc = j < a.dim ? j : a.dim - 1;
    const uint32_t P = (uint32_t)a.pop;
    const int g = (int)(threadIdx.x & 56u);          // the member's first lane of the wave
    // blocks: 0 the partners and the crossing coordinate, 1 and 2 crossover, 3 and 4 redraws
    const u32x4 o = philox10(gen, (uint32_t)i, (uint32_t)(j < 4 ? j : 4), 0u, a.key0, a.key1);
    const uint32_t rx = (uint32_t)__shfl((int)o.x, g, 64), ry = (uint32_t)__shfl((int)o.y, g, 64);
    const uint32_t rz = (uint32_t)__shfl((int)o.z, g, 64), rw = (uint32_t)__shfl((int)o.w, g, 64);
    T.uc = word_of(o, g + 1 + (j >> 2), j & 3);
    T.ud = word_of(o, g + 3 + (j >> 2), j & 3);
    const Partners p = partners(rx, ry, rz, P);
    T.jr = (int)below(rw, (uint32_t)a.dim);
    auto row = [&](uint32_t off) {                   // coordinate j of member (i + off) mod P
        const uint32_t m = (uint32_t)i + off;
        return a.x[(int64_t)(m >= P ? m - P : m) * a.dim + jc];
    };
    T.xi = row(0u);
    T.x0 = row(p.a);
    T.x1 = row(p.b);
    T.x2 = row(p.c);
}

// Objective of one network output row y [n_out], reduced over the wave (every
// lane returns it): the mean squared difference of the de-normalised curve and
// the target (tgt: a.target or a copy of it), over the target's squared peak.
__device__ __forceinline__ float member_objective(const DeArgs& a, const float* y, const float* tgt,
                                                  int lane)
{
    float s = 0.0f;
    for (int b = lane; b < a.n_out; b += 64) {
        const float d = expm1_own(y[b] * a.log_span) * a.out_scale - tgt[b];
        s = __builtin_fmaf(d, d, s);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    return s / (float)a.n_out * a.inv_peak2;
}

// Greedy selection of member i by one wave: the trial t replaces the member's
// row xi when its objective ft is not worse than fo (its current one, a.f[i]);
// writes the member's next row and argmin key.
__device__ __forceinline__ void select_member(const DeArgs& a, int i, float ft, float fo,
                                              const float* t, const float* xi, int lane)
{
    const bool take = ft <= fo;
    if (lane < a.dim) a.x_next[(int64_t)i * a.dim + lane] = take ? t[lane] : xi[lane];
    if (lane == 0) {
        const float fn = take ? ft : fo;
        if (take) a.f[i] = ft;
        a.keys_next[i] = ((unsigned long long)__float_as_uint(fn) << 32) | (unsigned long long)i;
    }
}

__global__ __launch_bounds__(256) void de_propose_kernel(DeArgs a, uint32_t gen)
{
    const int best = population_argmin<256>(a, first_key(a));     // of the previous generation
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= a.pop) return;
    float in[16];
    propose_member(a, i, best, gen, a.X + (int64_t)i * a.n_in, in);
    // the whole packed row, as pack_input writes it (trials, fixed inputs, zeros),
    // eight BF16 values per 16-byte store
    uint4* X0 = reinterpret_cast<uint4*>(a.X0 + (int64_t)i * a.kp0);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        uint32_t w[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const bf16 lo = (bf16)in[8 * c + 2 * t], hi = (bf16)in[8 * c + 2 * t + 1];
            w[t] = (uint32_t)__builtin_bit_cast(unsigned short, lo) |
                   ((uint32_t)__builtin_bit_cast(unsigned short, hi) << 16);
        }
        X0[c] = make_uint4(w[0], w[1], w[2], w[3]);
    }
    for (int c = 2; c < a.kp0 / 8; ++c) X0[c] = make_uint4(0u, 0u, 0u, 0u);
}

// One wave per member: objective of its trial (the network output row), greedy
// selection, and the member's argmin key.
__global__ __launch_bounds__(256) void de_score_kernel(DeArgs a)
{
    const int lane = (int)(threadIdx.x & 63u);
    const int i = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    if (i >= a.pop) return;
    const float ft = member_objective(a, a.Y + (int64_t)i * a.n_out, a.target, lane);
    select_member(a, i, ft, a.f[i], a.X + (int64_t)i * a.n_in, a.x + (int64_t)i * a.dim, lane);
}

// Weights in fragment order: for output tile t (32 rows), K step s (16 columns)
// and lane l, the 8 BF16 values W[32 t + l % 32][16 s + 8 (l / 32) .. +7] that lane
// l supplies to the 32x32x16 product, at ((t KS + s) 64 + l) 8, KS = kp / 16.
__global__ __launch_bounds__(256) void de_pack_kernel(const bf16* W, int out, int kp, bf16* Wf)
{
    const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;   // (t, s, l)
    const int KS = kp / 16;
    if (g >= (int64_t)(out / 32) * KS * 64) return;
    const int l = (int)(g % 64), s = (int)((g / 64) % KS), t = (int)(g / (64 * KS));
    *reinterpret_cast<uint4*>(Wf + g * 8) = *reinterpret_cast<const uint4*>(
        W + (int64_t)(32 * t + (l & 31)) * kp + 16 * s + 8 * (l >> 5));
}

// Matrix-core products of one layer for the wave's NT output tiles (w[j] points
// at the lane's fragment of K step 0 of tile j, in fragment order) over the 32
// rows in LDS (act, row stride lda): acc[j][r] = sum_k act[m][k] W[n][k], with m
// and n where the 32x32x16 layout puts them (lane l supplies A[l % 32][8 (l / 32)
// .. +7] and B^T[l % 32][8 (l / 32) .. +7]).  K in steps of 16 in order, CH steps
// per chunk (kp a multiple of 16 CH); the next chunk's weights are fetched while
// the current one is multiplied, alternating between p and q.  p holds the
// layer's first chunk on entry (fetched before the layer's input was ready).  The
// fetch past the last chunk is the next layer's first chunk (wn, when next; else
// the last chunk again), left in flight over the epilogue and the barrier: in p
// after an even number of chunks, in q after an odd one (returned).  The loads
// are unconditional (a uniform choice of address), so the wait before each
// chunk's products counts exactly the loads issued after it.
template <int CH, int NT>
__device__ __forceinline__ bool layer_products(const bf16* act, int lda, const bf16* const (&w)[NT],
                                               int kp, f32x16 (&acc)[NT], bf16x8 (&p)[NT][CH],
                                               bf16x8 (&q)[NT][CH], const bf16* const (&wn)[NT],
                                               bool next)
{
    const int lane = (int)(threadIdx.x & 63u);
    const bf16* ar = act + (lane & 31) * lda + 8 * (lane >> 5);
    constexpr int KC = 16 * CH;
    static_assert(NT >= 1, "at least one tile");
    auto fetch = [&](bf16x8 (&d)[NT][CH], int k0) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const bf16* src = k0 < kp ? w[t] + (int64_t)(k0 / 16) * 512
                                      : (next ? wn[t] : w[t] + (int64_t)((kp - KC) / 16) * 512);
#pragma unroll
            for (int j = 0; j < CH; ++j) d[t][j] = *reinterpret_cast<const bf16x8*>(src + j * 512);
        }
    };
    auto multiply = [&](const bf16x8 (&d)[NT][CH], int k0) {
#pragma unroll
        for (int j = 0; j < CH; ++j) {
            const bf16x8 av = *reinterpret_cast<const bf16x8*>(ar + k0 + 16 * j);
#pragma unroll
            for (int t = 0; t < NT; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, d[t][j], acc[t], 0, 0, 0);
        }
    };
    // the scheduling barriers keep each chunk's loads ahead of the previous chunk's
    // products (the scheduler would otherwise sink them next to their own uses)
    for (int k0 = 0; k0 < kp; k0 += 2 * KC) {
        fetch(q, k0 + KC);
        __builtin_amdgcn_sched_barrier(0);
        multiply(p, k0);
        if (k0 + KC >= kp) return true;
        fetch(p, k0 + 2 * KC);
        __builtin_amdgcn_sched_barrier(0);
        multiply(q, k0 + KC);
    }
    return false;
}

// The lane's fragment of K step 0 of output tile t of layer L, in fragment order.
__device__ __forceinline__ const bf16* tile_fragments(const DeLayer& L, int t, int lane)
{
    return L.w + ((int64_t)t * (L.kp / 16) * 64 + lane) * 8;
}

// One whole generation for M members per workgroup (see the file comment).
// Dynamic LDS: two activation buffers [32][lda] BF16, the output rows
// [32][n_out + 4] FP32, the trials [32][8] FP32, the target [n_out], the
// members' current objectives [32] and rows [32][8] FP32.
// The fixed network shapes of the unrolled form (the surrogate networks): five
// layers, 64 padded inputs, hidden layers 512 wide, 256 outputs.
constexpr int kFixedLayers = 5, kLdaFixed = 512 + 8, kYsFixed = 256 + 4;
constexpr int kAheadDe = 2;     // chunks in flight ahead of the products (4 KB a wave each; 150
                                // generations of 64 members 3.87 ms with 1, 3.79 with 2, and
                                // 4.08 with 3, at 126 registers)

// The fixed shapes as one stream of weight chunks (four K steps, 4 KB per wave):
// chunk 0 is layer 0's only chunk (K = 64), chunks 1 + 8 (l - 1) .. + 7 are layer
// l's (K = 512).  wl[l] is the wave's tile of layer l in fragment order.
constexpr int kFixedChunks = 8, kFixedStream = 1 + kFixedChunks * (kFixedLayers - 1);

__device__ __forceinline__ const bf16* stream_chunk(const bf16* const (&wl)[kFixedLayers], int g)
{
    return g == 0 ? wl[0] : wl[1 + (g - 1) / kFixedChunks] + ((g - 1) % kFixedChunks) * 2048;
}

// The tile row of member u of a workgroup's M.  Accumulator r of a lane holds row 8 (r / 4) +
// 4 (lane / 32) + r % 4, and the members' rows are those of r < M / 2: 0-15, 0-7, or 0, 1, 4
// and 5, so that both halves of the wave share an epilogue evenly.
template <int M>
__device__ __forceinline__ int member_row(int u)
{
    static_assert(M == 16 || M == 8 || M == 4, "rows of M members");
    return M == 4 ? (u & 1) + 4 * (u >> 1) : u;
}

// Layer L of the fixed shapes (bn: the bias of the lane's output column, loaded at
// the kernel's start), its products unrolled over the chunk stream: chunk
// g sits in buf[g % D] and is fetched D - 1 chunks ahead of its products, across
// the layer boundaries too (the next layer's first chunks are in flight over the
// epilogue and the barrier).  Every buffer index is known at compile time, so
// the ring needs no register copies; within a layer the loads are unconditional,
// so the wait before each chunk's products counts exactly the loads issued after
// it (the output layer's eight idle waves skip it whole).  The same products in
// the same K order as layer_products.
template <int L, int M, int D, int LDA, int YS>
__device__ __forceinline__ void fixed_layer(const bf16* const (&wl)[kFixedLayers], float bn,
                                            bf16x8 (&buf)[D][4], bf16*& cur, bf16*& nxt,
                                            float* yrow, int t, int lane)
{
    constexpr bool kLastL = L == kFixedLayers - 1;
    constexpr int G0 = L == 0 ? 0 : 1 + kFixedChunks * (L - 1), NC = L == 0 ? 1 : kFixedChunks;
    const bool has = !kLastL || t < 8;                // the output layer has 8 tiles
    const int n = 32 * (kLastL ? (t & 7) : t) + (lane & 31);
    const bf16* ar = cur + (lane & 31) * LDA + 8 * (lane >> 5);
    auto fetch = [&](int gf) {
        const bf16* src = stream_chunk(wl, gf);
#pragma unroll
        for (int j = 0; j < 4; ++j) buf[gf % D][j] = *reinterpret_cast<const bf16x8*>(src + j * 512);
    };
    if (has) {
        f32x16 acc = f32x16{};
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int g = G0 + c, gf = g + D - 1;
            // a chunk of this layer goes out before the products of chunk g; one of
            // the next layer after them (its products wait for the barrier anyway),
            // and only by the waves that have a tile there
            const bool cross = gf >= G0 + NC;
            if (!cross && gf < kFixedStream) fetch(gf);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bf16x8 av = *reinterpret_cast<const bf16x8*>(ar + 64 * c + 16 * j);
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, buf[g % D][j], acc, 0, 0, 0);
            }
            if (cross && gf < kFixedStream) {
                const bool next_last = gf >= 1 + kFixedChunks * (kFixedLayers - 2);
                if (!next_last || t < 8) fetch(gf);
            }
        }
#pragma unroll
        for (int r = 0; r < M / 2; ++r) {          // the members' rows
            const int m = 8 * (r / 4) + 4 * (lane >> 5) + (r % 4);
            if constexpr (kLastL) {
                yrow[m * YS + n] = acc[r] + bn;
            } else {
                const float z = acc[r] + bn;
                nxt[m * LDA + n] = (bf16)(z * sigmoid(z));
            }
        }
    }
    lds_barrier();
    bf16* done = cur;
    cur = nxt;
    nxt = done;
}

// LDA, YS: the activation and output row strides when fixed at compile time (the
// fixed shapes, laid out by a fully unrolled forward), so that the epilogue's LDS
// addresses are one base and immediate offsets; 0: any shape the fused kernel
// takes, net.lda and n_out + 4 at run time.
template <int M, int LDA, int YS>
__global__ __launch_bounds__(kFusedThreads) void de_generation_kernel(DeArgs a, DeNet net,
                                                                      uint32_t gen)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int lda = LDA > 0 ? LDA : net.lda, ys = YS > 0 ? YS : a.n_out + 4;
    bf16* act0 = reinterpret_cast<bf16*>(smem);
    bf16* act1 = act0 + kRows * lda;
    float* yrow = reinterpret_cast<float*>(act1 + kRows * lda);
    float* trial = yrow + kRows * ys;
    float* tgt = trial + kRows * 8;           // [n_out] the target curve
    float* fcur = tgt + a.n_out;              // [kRows] the members' current objectives
    float* xown = fcur + kRows;               // [kRows][8] the members' current rows
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row0 = (int)blockIdx.x * M;
    constexpr int kChunk = 4;                // K steps per weight chunk
    const int t = wave;                      // the wave's output tile in every layer
    __builtin_assume(t < kFusedThreads / 64);   // every wave has a tile of a hidden layer

    // every argument is asked for at once: one trip to memory, not one at each first use
    asm volatile("" ::"s"(a.keys), "s"(a.target), "s"(a.f), "s"(a.x), "s"(a.x_next),
                 "s"(a.keys_next), "s"(a.pop), "s"(a.n_out), "s"(a.dim), "s"(a.key0), "s"(a.key1), "s"(gen));
    if constexpr (LDA > 0) {
#pragma unroll
        for (int l = 0; l < kFixedLayers; ++l) asm volatile("" ::"s"(net.L[l].w), "s"(net.L[l].b));
    }
    // the keys, the target, the members' current objectives and the trials' draws and
    // partner rows go out first of all, so that their latencies overlap; a lane takes
    // coordinate j of member u
    const uint64_t key = first_key(a);
    // (unconditional loads, clamped: a load under a branch is waited for at its end)
    const float tg = a.target[tid < a.n_out ? tid : 0];
    const float fc = a.f[tid < M && row0 + tid < a.pop ? row0 + tid : row0];
    const int u = tid >> 3, j = tid & 7;
    const bool own = u < M && row0 + u < a.pop;
    const bool coord = own && j < a.dim;
    CoordTrial T;
    if (tid < kTrialThreads<M>) coord_fetch(a, own ? row0 + u : row0, j, gen, T);
    __builtin_amdgcn_sched_barrier(0);
    // the fixed shapes: the wave's tiles of every layer, and a ring of kAheadDe + 1
    // chunk buffers over the stream, whose first chunks go out behind the loads above (loads return in
    // order, so the trials do not wait for weights)
    constexpr int D = kAheadDe + 1;
    const bf16* wl[kFixedLayers];
    float bl[kFixedLayers];                  // the lane's output-column bias of every layer
    bf16x8 buf[D][4];
    if constexpr (LDA > 0) {
#pragma unroll
        for (int l = 0; l < kFixedLayers; ++l) {
            const int tl = l + 1 == kFixedLayers ? (t & 7) : t;
            wl[l] = net.L[l].w + ((int64_t)tl * (l == 0 ? 4 : 32) * 64 + lane) * 8;
            bl[l] = net.L[l].b[32 * tl + (lane & 31)];
        }
#pragma unroll
        for (int g = 0; g < D - 1; ++g) {
            const bf16* src = stream_chunk(wl, g);
#pragma unroll
            for (int j = 0; j < 4; ++j) buf[g][j] = *reinterpret_cast<const bf16x8*>(src + j * 512);
        }
    }

    __builtin_amdgcn_sched_barrier(0);
    // the other rows of both activation buffers hold zeros (16-byte stores; the
    // row stride lda is a multiple of 8)
    constexpr int kFirstZero = M == 4 ? 2 : M;
    for (int e = tid; e < (kRows - kFirstZero) * lda / 8; e += kFusedThreads) {
        reinterpret_cast<uint4*>(act0 + kFirstZero * lda)[e] = make_uint4(0u, 0u, 0u, 0u);
        reinterpret_cast<uint4*>(act1 + kFirstZero * lda)[e] = make_uint4(0u, 0u, 0u, 0u);
    }
    if (tid < a.n_out) tgt[tid] = tg;                 // n_out <= 512
    if (tid < M) fcur[tid] = fc;
    const int best = population_argmin<kFusedThreads>(a, key);   // of the previous generation
    if (u < M) {
        float t_j = 0.0f;
        if (coord)
            t_j = trial_coord(a, T.xi, T.x0, T.x1, T.x2, a.x[(int64_t)best * a.dim + j], j == T.jr,
                              T.uc, T.ud);
        if (coord) {
            trial[8 * u + j] = t_j;
            xown[8 * u + j] = T.xi;
        }
        // the network's input row: trial, fixed inputs, zeros
        bf16* r = act0 + member_row<M>(u) * lda;
        r[j] = (bf16)(coord ? t_j : (own && j < a.n_in ? a.fixed[j - a.dim] : 0.0f));
        for (int k = 8 + j; k < (LDA > 0 ? 64 : net.L[0].kp); k += 8)
            r[k] = (bf16)(own && k < a.n_in ? a.fixed[k - a.dim] : 0.0f);
    }
    // wave w computes output tile w of every layer that is that wide.  The layer
    // loop is unrolled (layer l's descriptor at a fixed kernel-argument offset:
    // scalar loads, which leave the weight prefetch in flight), and each layer's
    // bias is fetched before its products, so waiting for it does not wait for the
    // next layer's first chunk.
    bf16* cur = act0;
    bf16* nxt = act1;
    if constexpr (LDA > 0) {
        lds_barrier();
        static_assert(kFixedLayers == 5, "the unrolled form is written for five layers");
        fixed_layer<0, M, D, LDA, YS>(wl, bl[0], buf, cur, nxt, yrow, t, lane);
        fixed_layer<1, M, D, LDA, YS>(wl, bl[1], buf, cur, nxt, yrow, t, lane);
        fixed_layer<2, M, D, LDA, YS>(wl, bl[2], buf, cur, nxt, yrow, t, lane);
        fixed_layer<3, M, D, LDA, YS>(wl, bl[3], buf, cur, nxt, yrow, t, lane);
        fixed_layer<4, M, D, LDA, YS>(wl, bl[4], buf, cur, nxt, yrow, t, lane);
    } else {
        bf16x8 pre[1][kChunk], alt[1][kChunk];
        if (t < net.L[0].out / 32) {
            const bf16* w0 = tile_fragments(net.L[0], t, lane);
#pragma unroll
            for (int j = 0; j < kChunk; ++j)
                pre[0][j] = *reinterpret_cast<const bf16x8*>(w0 + j * 512);
        }
        lds_barrier();
        bool in_alt = false;          // the layer's first chunk is in alt, not pre
#pragma unroll
        for (int l = 0; l < kMaxLayers; ++l) {
            if (l >= net.n_layers) break;
            const DeLayer L = net.L[l];
            if (t < L.out / 32) {
                if (in_alt) {
#pragma unroll
                    for (int j = 0; j < kChunk; ++j) pre[0][j] = alt[0][j];
                }
                const int n = 32 * t + (lane & 31);
                const float bn = L.b[n];
                const bf16* const w[1] = {tile_fragments(L, t, lane)};
                const int ln = l + 1 < kMaxLayers ? l + 1 : l;
                const bool next = l + 1 < net.n_layers && t < net.L[ln].out / 32;
                const bf16* const wn[1] = {next ? tile_fragments(net.L[ln], t, lane) : w[0]};
                f32x16 acc[1] = {f32x16{}};
                in_alt = layer_products<kChunk, 1>(cur, lda, w, L.kp, acc, pre, alt, wn, next);
                const bool last = l + 1 == net.n_layers;
#pragma unroll
                for (int r = 0; r < M / 2; ++r) {      // the members' rows
                    const int m = 8 * (r / 4) + 4 * (lane >> 5) + (r % 4);
                    if (last) {
                        yrow[m * ys + n] = acc[0][r] + bn;
                    } else {
                        const float z = acc[0][r] + bn;
                        nxt[m * lda + n] = (bf16)(z * sigmoid(z));
                    }
                }
            }
            lds_barrier();
            bf16* done = cur;
            cur = nxt;
            nxt = done;
        }
    }

    // objectives and selection: wave w takes member w of the workgroup
    static_assert(M <= kFusedThreads / 64, "a wave a member");
    if (wave < M && row0 + wave < a.pop) {
        const float ft = member_objective(a, yrow + member_row<M>(wave) * ys, tgt, lane);
        select_member(a, row0 + wave, ft, fcur[wave], trial + wave * 8, xown + wave * 8, lane);
    }
}

// Members of a workgroup for a population: as few as keep to 128 workgroups, half the CUs.
// Every CU streams the whole weight set either way, and the epilogues are the members' share
// of it; with all 256 CUs streaming the L2s are the limit.  150 generations: 1,024 members 3.96
// ms at 8 a workgroup, 4.46 at 4 (256 workgroups), 4.38 at 16; 64 members 3.87 at 4, 4.26 at
// 16; 2,048 members 4.44 at 16, 4.79 at 8.
constexpr int kGroups = 128;
int members_per_group(int pop) { return pop <= 4 * kGroups ? 4 : pop <= 8 * kGroups ? 8 : 16; }

template <int M>
hipError_t launch_fixed(const DeArgs& a, const DeNet& net, uint32_t gen, int lds_bytes,
                        hipStream_t stream)
{
    hipLaunchKernelGGL((de_generation_kernel<M, kLdaFixed, kYsFixed>), dim3((unsigned)((a.pop + M - 1) / M)),
                       dim3(kFusedThreads), (unsigned)lds_bytes, stream, a, net, gen);
    return hipGetLastError();
}

}  // namespace

hipError_t de_init(const DeArgs& a, hipStream_t stream)
{
    hipLaunchKernelGGL(de_init_kernel, dim3((unsigned)((a.pop_pad + 255) / 256)), dim3(256), 0,
                       stream, a);
    return hipGetLastError();
}

hipError_t de_propose(const DeArgs& a, uint32_t gen, hipStream_t stream)
{
    hipLaunchKernelGGL(de_propose_kernel, dim3((unsigned)((a.pop + 255) / 256)), dim3(256), 0,
                       stream, a, gen);
    return hipGetLastError();
}

hipError_t de_score(const DeArgs& a, hipStream_t stream)
{
    hipLaunchKernelGGL(de_score_kernel, dim3((unsigned)((a.pop + 3) / 4)), dim3(256), 0, stream,
                       a);
    return hipGetLastError();
}

hipError_t de_pack(const __bf16* W, int out, int kp, __bf16* Wf, hipStream_t stream)
{
    const int64_t n = (int64_t)(out / 32) * (kp / 16) * 64;
    hipLaunchKernelGGL(de_pack_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, W,
                       out, kp, Wf);
    return hipGetLastError();
}

int de_fused_lds(const DeNet& net, int n_out)
{
    return (int)(2 * kRows * net.lda * sizeof(bf16) + kRows * (n_out + 4) * sizeof(float) +
                 kRows * 8 * sizeof(float) + n_out * sizeof(float) + kRows * sizeof(float) +
                 kRows * 8 * sizeof(float));
}


hipError_t de_fused_prepare(int lds_bytes)
{
    hipError_t e = hipSuccess;
    for (const void* f : {reinterpret_cast<const void*>(de_generation_kernel<4, kLdaFixed, kYsFixed>),
                          reinterpret_cast<const void*>(de_generation_kernel<8, kLdaFixed, kYsFixed>),
                          reinterpret_cast<const void*>(de_generation_kernel<16, kLdaFixed, kYsFixed>),
                          reinterpret_cast<const void*>(de_generation_kernel<kMembers, 0, 0>)})
        if (e == hipSuccess)
            e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    return e;
}

// Whether a network has the fixed shapes of the unrolled form.
bool de_fixed_shapes(const DeNet& net, int n_out)
{
    if (net.n_layers != kFixedLayers || net.lda != kLdaFixed || n_out + 4 != kYsFixed) return false;
    for (int l = 0; l < net.n_layers; ++l) {
        const bool last = l + 1 == net.n_layers;
        if (net.L[l].kp != (l == 0 ? 64 : 512) || net.L[l].out != (last ? 256 : 512)) return false;
    }
    return true;
}

hipError_t de_generation_fused(const DeArgs& a, const DeNet& net, uint32_t gen, int lds_bytes,
                               hipStream_t stream)
{
    if (de_fixed_shapes(net, a.n_out)) {
        switch (members_per_group(a.pop)) {
        case 4: return launch_fixed<4>(a, net, gen, lds_bytes, stream);
        case 8: return launch_fixed<8>(a, net, gen, lds_bytes, stream);
        default: return launch_fixed<16>(a, net, gen, lds_bytes, stream);
        }
    }
    hipLaunchKernelGGL((de_generation_kernel<kMembers, 0, 0>), 
                       dim3((unsigned)((a.pop + kMembers - 1) / kMembers)),
                       dim3(kFusedThreads), (unsigned)lds_bytes, stream, a, net, gen);
    return hipGetLastError();
}

}  // namespace mlp
}  // namespace mcl
