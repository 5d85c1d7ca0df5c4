// mlp_train.hip — a training step of the surrogate network in two kernels: the
// forward and backward chain of the batch, and the weight gradients with the
// AdamW update.
//
// The layered form (mlp.hip) is some 17 launches of products of a few GFLOP each at
// batch 4096 (190 us of kernels, 250 us with the gaps between them), with every
// activation, pre-activation and error written and read in two orders.
//
//   chain   a workgroup takes 32 rows of the batch through every layer forward, the
//           loss, and every layer backward.  Activations and errors pass from layer to
//           layer in LDS; the pre-activations the backward needs stay in registers:
//           a wave computes the same output tiles (wave, wave + 8) of a layer forward
//           and backward, so each lane meets its own z again, rounded to BF16 as it
//           was when it went through memory.  Weights come from L2 in fragment order,
//           as in the inference kernel; the backward reads W^T in that order.  Bound by
//           the stream of weights into each CU: 3.7 MB forward and backward at up to 146
//           GB/s per CU, 25 us whatever the batch up to 32 rows a CU.
//   update  a workgroup takes a 64 x 64 tile of one layer's weights: dW = dZ^T A over the
//           whole batch, the contraction split over its eight waves and summed in order
//           through LDS, then AdamW on the tile and its BF16 copies (row-major and
//           the two fragment orders), so no partial sums go through memory.  Further
//           workgroups take 32 biases each (row sums of dZ), one the loss.
//
// Operands of dW are features x batch, contracted over the batch.  The chain writes them
// (the packed input, every activation, every error) as fragments of the update's
// products: for each 32 features and 16 batch rows, 64 lanes of 8 rows.  A lane of the
// chain holds one feature and four consecutive rows, half of such a fragment, so its
// store is 8 bytes and a wave's 512 contiguous ones.
//
// Products, their K order, the parts the batch is summed in, the bias sums' order and all
// roundings are those of the layered kernels, so the weights after a step are bit for bit
// theirs (only the reported loss adds its squares in another order).
#include "mlp_internal.h"

namespace mcl {
namespace mlp {
namespace {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kWaves = 8, kThreadsT = 64 * kWaves;
constexpr int kR = kTrainRows;          // batch rows of a chain workgroup
constexpr int kLda = 512 + 8;           // LDS row stride of its activations
constexpr int kAhead = 4;               // K steps fetched ahead of their products

struct Ring {                           // weight fragments in flight
    bf16x8 f[kAhead + 1][2];
};

template <int FN>
__device__ __forceinline__ void fetch_first(const bf16* w0, const bf16* w1, Ring& r)
{
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
        r.f[s][0] = *reinterpret_cast<const bf16x8*>(w0 + s * 512);
        if (FN > 1) r.f[s][1] = *reinterpret_cast<const bf16x8*>(w1 + s * 512);
    }
}

// acc[j] += the 32 rows of act times the wave's tile j over KS K steps; the first
// kAhead steps' fragments are in the ring.  The scheduling barriers keep each load
// kAhead steps ahead of its product.
template <int FN, int KS>
__device__ __forceinline__ void products(const bf16* act, const bf16* w0, const bf16* w1, Ring& ring,
                                         f32x16 (&acc)[2], int lane)
{
    static_assert(KS >= kAhead, "the ring is filled before the first product");
    const bf16* ar = act + (lane & 31) * kLda + 8 * (lane >> 5);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        if (s + kAhead < KS) {
            ring.f[(s + kAhead) % (kAhead + 1)][0] =
                *reinterpret_cast<const bf16x8*>(w0 + (s + kAhead) * 512);
            if (FN > 1)
                ring.f[(s + kAhead) % (kAhead + 1)][1] =
                    *reinterpret_cast<const bf16x8*>(w1 + (s + kAhead) * 512);
        }
        __builtin_amdgcn_sched_barrier(0);
        const bf16x8 av = *reinterpret_cast<const bf16x8*>(ar + 16 * s);
#pragma unroll
        for (int j = 0; j < FN; ++j)
            acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, ring.f[s % (kAhead + 1)][j], acc[j], 0, 0, 0);
    }
}

// Four consecutive batch rows (8 q + 4 h ..) of feature tile T, as half of the
// update's fragment (q = 2 (step of 16 rows) + half of 8 rows).
__device__ __forceinline__ void store_quad(bf16* frag, int T, int64_t S, int64_t s0, int q, int lane,
                                           bf16x4 v)
{
    const int64_t o = (((int64_t)T * S + s0 + (q >> 1)) * 64 + (lane & 31) + 32 * (q & 1)) * 8 +
                      4 * (lane >> 5);
    *reinterpret_cast<bf16x4*>(frag + o) = v;
}

// NH hidden layers of 512, NO output tiles of 32 a wave (n_out = 256 NO).
template <int NH, int NO>
__global__ __launch_bounds__(kThreadsT, 2) void train_chain_kernel(TrainArgs a)
{
    extern __shared__ __align__(16) unsigned char smem_t[];
    bf16* cur = reinterpret_cast<bf16*>(smem_t);            // the layer's input
    bf16* nxt = cur + kR * kLda;                            // its output
    int* rows = reinterpret_cast<int*>(nxt + kR * kLda);    // [kR] batch rows in x and t
    float* red = reinterpret_cast<float*>(rows + kR);       // [kWaves]
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t row0 = (int64_t)blockIdx.x * kR;
    const int64_t S = a.B / 16, s0 = row0 / 16;
    constexpr int n_out = 256 * NO;

    auto frag_ptr = [&](const bf16* w, int j, int ks) {
        return w + ((int64_t)(wave + kWaves * j) * ks * 64 + lane) * 8;
    };
    Ring ring;
    const bf16* w0 = frag_ptr(a.net.L[0].w, 0, 4);
    const bf16* w1 = frag_ptr(a.net.L[0].w, 1, 4);
    fetch_first<2>(w0, w1, ring);

    if (tid < kR) rows[tid] = a.idx ? a.idx[row0 + tid] : (int)(row0 + tid);
    __syncthreads();
    for (int e = tid; e < kR * 64; e += kThreadsT) {
        const int r = e >> 6, k = e & 63;
        cur[r * kLda + k] = (bf16)(k < a.n_in ? a.x[(int64_t)rows[r] * a.n_in + k] : 0.0f);
    }
    __syncthreads();
    if (tid < 256) {       // the packed input's fragments: two feature tiles, two steps
        const int l = tid & 63, st = (tid >> 6) & 1, T = tid >> 7;
        bf16x8 v;
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = cur[(16 * st + 8 * (l >> 5) + i) * kLda + 32 * T + (l & 31)];
        *reinterpret_cast<bf16x8*>(a.xf + (((int64_t)T * S + s0 + st) * 64 + l) * 8) = v;
    }

    uint32_t zr[NH][2][8];                // z of the lane's outputs, two BF16 a word
    // ---- forward ------------------------------------------------------------------
#pragma unroll
    for (int l = 0; l < NH; ++l) {
        f32x16 acc[2] = {f32x16{}, f32x16{}};
        float bn[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) bn[j] = a.net.L[l].b[32 * (wave + kWaves * j) + (lane & 31)];
        if (l == 0) products<2, 4>(cur, w0, w1, ring, acc, lane);
        else products<2, 32>(cur, w0, w1, ring, acc, lane);
        w0 = frag_ptr(a.net.L[l + 1].w, 0, 32);
        w1 = frag_ptr(a.net.L[l + 1].w, 1, 32);
        if (l + 1 < NH || NO > 1) fetch_first<2>(w0, w1, ring);
        else fetch_first<1>(w0, w0, ring);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int T = wave + kWaves * j, n = 32 * T + (lane & 31);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                bf16x4 av, zv;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float z = acc[j][4 * q + r] + bn[j];
                    zv[r] = (bf16)z;
                    av[r] = (bf16)(z * sigmoid(z));
                    nxt[(8 * q + 4 * (lane >> 5) + r) * kLda + n] = av[r];
                }
                const uint2 zw = __builtin_bit_cast(uint2, zv);
                zr[l][j][2 * q] = zw.x;
                zr[l][j][2 * q + 1] = zw.y;
                store_quad(a.af[l], T, S, s0, q, lane, av);
            }
        }
        lds_barrier();
        bf16* t = cur;
        cur = nxt;
        nxt = t;
    }
    // ---- output layer, loss -------------------------------------------------------
    {
        f32x16 acc[2] = {f32x16{}, f32x16{}};
        float tg[NO][16], bn[NO];
#pragma unroll
        for (int j = 0; j < NO; ++j) {
            const int n = 32 * (wave + kWaves * j) + (lane & 31);
            bn[j] = a.net.L[NH].b[n];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int m = 8 * (i / 4) + 4 * (lane >> 5) + i % 4;
                tg[j][i] = a.t[(int64_t)rows[m] * n_out + n];
            }
        }
        products<NO, 32>(cur, w0, w1, ring, acc, lane);
        w0 = frag_ptr(a.wtf[NH], 0, n_out / 16);
        w1 = frag_ptr(a.wtf[NH], 1, n_out / 16);
        fetch_first<2>(w0, w1, ring);
        float se = 0.0f;
#pragma unroll
        for (int j = 0; j < NO; ++j) {
            const int T = wave + kWaves * j, n = 32 * T + (lane & 31);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                bf16x4 gv;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float y = acc[j][4 * q + r] + bn[j];
                    const float d = y - tg[j][4 * q + r];
                    se += d * d;
                    gv[r] = (bf16)(d * a.grad_scale);
                    nxt[(8 * q + 4 * (lane >> 5) + r) * kLda + n] = gv[r];
                }
                store_quad(a.dzf[NH], T, S, s0, q, lane, gv);
            }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) se += __shfl_xor(se, o, 64);
        if (lane == 0) red[wave] = se;
        lds_barrier();
        if (tid == 0) {
            float s = 0.0f;
            for (int w = 0; w < kWaves; ++w) s += red[w];
            a.loss_part[blockIdx.x] = s;
        }
        bf16* t = cur;
        cur = nxt;
        nxt = t;
    }
    // ---- backward: dZ_{l-1} = (dZ_l W_l) * silu'(Z_{l-1}) --------------------------
#pragma unroll
    for (int l = NH; l >= 1; --l) {
        f32x16 acc[2] = {f32x16{}, f32x16{}};
        if (l == NH) products<2, n_out / 16>(cur, w0, w1, ring, acc, lane);
        else products<2, 32>(cur, w0, w1, ring, acc, lane);
        if (l > 1) {
            w0 = frag_ptr(a.wtf[l - 1], 0, 32);
            w1 = frag_ptr(a.wtf[l - 1], 1, 32);
            fetch_first<2>(w0, w1, ring);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int T = wave + kWaves * j, n = 32 * T + (lane & 31);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const bf16x4 zv =
                    __builtin_bit_cast(bf16x4, make_uint2(zr[l - 1][j][2 * q], zr[l - 1][j][2 * q + 1]));
                bf16x4 dv;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float z = (float)zv[r];
                    const float s = sigmoid(z);
                    dv[r] = (bf16)(acc[j][4 * q + r] * (s * (1.0f + z * (1.0f - s))));
                    if (l > 1) nxt[(8 * q + 4 * (lane >> 5) + r) * kLda + n] = dv[r];
                }
                store_quad(a.dzf[l - 1], T, S, s0, q, lane, dv);
            }
        }
        if (l > 1) lds_barrier();
        bf16* t = cur;
        cur = nxt;
        nxt = t;
    }
}

constexpr int kTile = 64;                       // weight tile of an update workgroup
constexpr int kChunk = 4;                       // batch steps fetched together
constexpr int kTileLd = kTile + 2;              // row stride of the BF16 transpose
constexpr int kBiasRows = 32;                   // biases of a bias workgroup

// P x Q products of 32 x 32 over the batch steps [sb, se) (rows of fragments at pa, columns
// at pb, S steps each), into the tile's partial sums at part.
template <int P, int Q>
__device__ __forceinline__ void dw_products(const bf16* pa, const bf16* pb, int64_t S, int64_t sb,
                                            int64_t se, float* part, int lane)
{
    f32x16 acc[P][Q];
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
        for (int q = 0; q < Q; ++q) acc[p][q] = f32x16{};
    struct Chunk {
        bf16x8 a[kChunk][P], b[kChunk][Q];
    };
    // steps past the last one repeat it (in bounds) and are not multiplied
    auto fetch = [&](Chunk& c, int64_t s) {
#pragma unroll
        for (int i = 0; i < kChunk; ++i) {
            const int64_t o = (s + i < se ? s + i : se - 1) * 512;
#pragma unroll
            for (int p = 0; p < P; ++p) c.a[i][p] = *reinterpret_cast<const bf16x8*>(pa + p * S * 512 + o);
#pragma unroll
            for (int q = 0; q < Q; ++q) c.b[i][q] = *reinterpret_cast<const bf16x8*>(pb + q * S * 512 + o);
        }
    };
    auto multiply = [&](const Chunk& c, int64_t s) {
#pragma unroll
        for (int i = 0; i < kChunk; ++i) {
            if (s + i < se) {
#pragma unroll
                for (int p = 0; p < P; ++p)
#pragma unroll
                    for (int q = 0; q < Q; ++q)
                        acc[p][q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c.a[i][p], c.b[i][q],
                                                                            acc[p][q], 0, 0, 0);
            }
        }
    };
    Chunk c0, c1;
    fetch(c0, sb);
    for (int64_t s = sb; s < se; s += 2 * kChunk) {
        fetch(c1, s + kChunk);
        __builtin_amdgcn_sched_barrier(0);
        multiply(c0, s);
        fetch(c0, s + 2 * kChunk);
        __builtin_amdgcn_sched_barrier(0);
        multiply(c1, s + kChunk);
    }
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
        for (int q = 0; q < Q; ++q)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                part[(32 * p + 8 * (r / 4) + 4 * (lane >> 5) + r % 4) * kTile + 32 * q + (lane & 31)] =
                    acc[p][q][r];
}

// 32 biases of a layer: the gradient is the row sum of dZ, in the order of a wave whose
// lane c adds groups c, c + 64, .. of eight batch rows and then halves of lanes.
__device__ __forceinline__ void update_biases(const UpdateArgs& a, const UpdateLayer& L, int T,
                                              float* sums, int tid)
{
    constexpr int kLd = kBiasRows + 1;
    const int n = tid & 31;
    const int64_t groups = 2 * a.S;
    // a thread takes four of a row's 64 lanes, 16 fragments in flight: one at a time, its 32
    // dependent trips at batch 4096 were longer than the tiles' products
    constexpr int kC = 64 / (kThreadsT / 32), kU = 4;
    const int c0 = tid >> 5;
    float acc[kC];
#pragma unroll
    for (int j = 0; j < kC; ++j) acc[j] = 0.0f;
    for (int64_t g0 = 0; g0 < groups; g0 += 64 * kU) {
        bf16x8 v[kU][kC];
#pragma unroll
        for (int u = 0; u < kU; ++u)
#pragma unroll
            for (int j = 0; j < kC; ++j) {
                const int64_t gr = g0 + 64 * u + c0 + (kThreadsT / 32) * j;
                const int64_t gl = gr < groups ? gr : 0;
                v[u][j] = *reinterpret_cast<const bf16x8*>(
                    L.dzf + (((int64_t)T * a.S + (gl >> 1)) * 64 + n + 32 * (gl & 1)) * 8);
            }
#pragma unroll
        for (int u = 0; u < kU; ++u)
#pragma unroll
            for (int j = 0; j < kC; ++j)
                if (g0 + 64 * u + c0 + (kThreadsT / 32) * j < groups) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) acc[j] += (float)v[u][j][i];
                }
    }
#pragma unroll
    for (int j = 0; j < kC; ++j) sums[(c0 + (kThreadsT / 32) * j) * kLd + n] = acc[j];
    __syncthreads();
    for (int o = 32; o > 0; o >>= 1) {
        for (int c = tid >> 5; c < o; c += kThreadsT / 32) sums[c * kLd + n] += sums[(c + o) * kLd + n];
        __syncthreads();
    }
    if (tid >= kBiasRows) return;
    const int nb = T * kBiasRows + n;
    if (a.mode == kOptExportGrad) a.flat[L.flat_b + nb] = sums[n];
    else adamw(L.bw[nb], L.bm[nb], L.bv[nb], sums[n], a.hp);
}

__global__ __launch_bounds__(kThreadsT, 2) void train_update_kernel(UpdateArgs a)
{
    extern __shared__ __align__(16) unsigned char smem_u[];
    float* part = reinterpret_cast<float*>(smem_u);                    // [kWaves][kTile][kTile]
    bf16* tr = reinterpret_cast<bf16*>(part + kWaves * kTile * kTile); // [kTile][kTileLd]
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // Biases and the loss first: they are short, and the tiles left when every CU is
    // taken start in their place.  Tiles then go to the XCDs (workgroups are dealt
    // round-robin over them) in contiguous runs of a layer's row-major tiles, about four rows
    // of dZ fragments and all columns of A: 5.8 MB through each L2 instead of the 16 that
    // a column of every layer per XCD reads.
    int blk = (int)blockIdx.x;
    if (blk < a.n_bias) {
        int li = 0;
        while (li + 1 < a.n_layers && blk >= a.L[li + 1].bias0) ++li;
        update_biases(a, a.L[li], blk - a.L[li].bias0, part, tid);
        return;
    }
    blk -= a.n_bias;
    if (blk == 0) {                             // the loss: chain partials in a fixed order
        if (a.loss == nullptr) return;
        float s = 0.0f;
        for (int i = tid; i < a.n_part; i += kThreadsT) s += a.loss_part[i];
        part[tid] = s;
        __syncthreads();
        for (int w = kThreadsT / 2; w > 0; w >>= 1) {
            if (tid < w) part[tid] += part[tid + w];
            __syncthreads();
        }
        if (tid == 0) *a.loss = part[0] * a.loss_scale;
        return;
    }
    {
        const int i = blk - 1, whole = a.n_tiles / 8 * 8;
        const int x = ((int)blockIdx.x) % 8, first = (a.n_bias + 1) % 8;   // XCD; of tile 0
        blk = i < whole ? ((x - first + 8) % 8) * (a.n_tiles / 8) + i / 8 : i;
    }
    int li = 0;
    while (li + 1 < a.n_layers && blk >= a.L[li + 1].tile0) ++li;
    const UpdateLayer& L = a.L[li];
    const int t = blk - L.tile0, tk_n = L.kp / kTile;
    const int tn = t / tk_n, tk = t % tk_n;
    // the batch in `parts` contiguous ranges of steps; eight waves over the parts, and with
    // fewer than eight over the tile's 32 x 32 quarters too
    const int64_t S = a.S, per = S / a.parts;
    const bf16* pa = L.dzf + ((int64_t)(2 * tn) * S * 64 + lane) * 8;
    const bf16* pb = L.xf + ((int64_t)(2 * tk) * S * 64 + lane) * 8;
    if (a.parts == 8) {
        dw_products<2, 2>(pa, pb, S, wave * per, (wave + 1) * per, part + wave * kTile * kTile, lane);
    } else if (a.parts == 4) {
        const int z = wave >> 1, p = wave & 1;
        dw_products<1, 2>(pa + p * S * 512, pb, S, z * per, (z + 1) * per,
                          part + (z * kTile + 32 * p) * kTile, lane);
    } else if (wave < 4 * a.parts) {
        const int z = wave >> 2, p = (wave >> 1) & 1, q = wave & 1;
        dw_products<1, 1>(pa + p * S * 512, pb + q * S * 512, S, z * per, (z + 1) * per,
                          part + (z * kTile + 32 * p) * kTile + 32 * q, lane);
    }
    // the weights this thread updates: row n, eight columns from k on
    const int nl = tid >> 3, kl = (tid & 7) * 8;
    const int n = tn * kTile + nl, k = tk * kTile + kl;
    const int64_t o = (int64_t)n * L.kp + k;
    float w[8], m[8], v[8];
    if (a.mode == kOptAdamW) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            *reinterpret_cast<float4*>(w + 4 * h) = *reinterpret_cast<const float4*>(L.w + o + 4 * h);
            *reinterpret_cast<float4*>(m + 4 * h) = *reinterpret_cast<const float4*>(L.m + o + 4 * h);
            *reinterpret_cast<float4*>(v + 4 * h) = *reinterpret_cast<const float4*>(L.v + o + 4 * h);
        }
    }
    __syncthreads();
    float g[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) g[i] = 0.0f;
    for (int z = 0; z < a.parts; ++z) {
        const float* pz = part + (z * kTile + nl) * kTile + kl;
#pragma unroll
        for (int i = 0; i < 8; ++i) g[i] += pz[i];
    }
    if (a.mode == kOptExportGrad) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (k + i < L.k_in) a.flat[L.flat_w + (int64_t)n * L.k_in + k + i] = g[i];
        return;
    }
    bf16x8 wb;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        if (k + i < L.k_in) adamw(w[i], m[i], v[i], g[i], a.hp);
        wb[i] = (bf16)w[i];
        tr[nl * kTileLd + kl + i] = wb[i];
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        *reinterpret_cast<float4*>(L.w + o + 4 * h) = *reinterpret_cast<const float4*>(w + 4 * h);
        *reinterpret_cast<float4*>(L.m + o + 4 * h) = *reinterpret_cast<const float4*>(m + 4 * h);
        *reinterpret_cast<float4*>(L.v + o + 4 * h) = *reinterpret_cast<const float4*>(v + 4 * h);
    }
    *reinterpret_cast<bf16x8*>(L.wb + o) = wb;
    *reinterpret_cast<bf16x8*>(L.wf + fragment_offset(n, k, L.kp)) = wb;
    if (L.wtf != nullptr) {
        __syncthreads();
        const int kk = tk * kTile + nl, nn = tn * kTile + kl;     // row of W^T, eight columns
        bf16x8 wv;
#pragma unroll
        for (int i = 0; i < 8; ++i) wv[i] = tr[(kl + i) * kTileLd + nl];
        *reinterpret_cast<bf16x8*>(L.wtf + fragment_offset(kk, nn, L.out)) = wv;
    }
}

constexpr int kChainLds = 2 * kR * kLda * (int)sizeof(bf16) + kR * (int)sizeof(int) +
                          kWaves * (int)sizeof(float);
constexpr int kUpdateLds = kWaves * kTile * kTile * (int)sizeof(float) +
                           kTile * kTileLd * (int)sizeof(bf16);

}  // namespace

bool train_fused_ok(const DeNet& net, int max_lds)
{
    if (net.n_layers != kTrainHidden + 1 || kUpdateLds > max_lds || kChainLds > max_lds) return false;
    for (int l = 0; l + 1 < net.n_layers; ++l)
        if (net.L[l].out != 512 || net.L[l].kp != (l == 0 ? 64 : 512)) return false;
    const DeLayer& o = net.L[net.n_layers - 1];
    return (o.out == 256 || o.out == 512) && o.kp == 512;
}

hipError_t train_fused_prepare()
{
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(train_chain_kernel<kTrainHidden, 1>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, kChainLds);
    if (e == hipSuccess)
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(train_chain_kernel<kTrainHidden, 2>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, kChainLds);
    if (e == hipSuccess)
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(train_update_kernel),
                                hipFuncAttributeMaxDynamicSharedMemorySize, kUpdateLds);
    return e;
}

hipError_t train_chain(const TrainArgs& a, int n_out, hipStream_t stream)
{
    const dim3 grid((unsigned)(a.B / kR));
    if (n_out == 256)
        hipLaunchKernelGGL((train_chain_kernel<kTrainHidden, 1>), grid, dim3(kThreadsT), kChainLds, stream, a);
    else
        hipLaunchKernelGGL((train_chain_kernel<kTrainHidden, 2>), grid, dim3(kThreadsT), kChainLds, stream, a);
    return hipGetLastError();
}

hipError_t train_update(const UpdateArgs& a, hipStream_t stream)
{
    hipLaunchKernelGGL(train_update_kernel, dim3((unsigned)(a.n_bias + 1 + a.n_tiles)), dim3(kThreadsT), kUpdateLds,
                       stream, a);
    return hipGetLastError();
}

}  // namespace mlp
}  // namespace mcl
