// mlp_fused.hip — the surrogate network's whole inference forward in one kernel.
//
// A workgroup takes 32 MT rows of the batch through every layer: the rows'
// activations stay in LDS (one BF16 buffer, rewritten in place by each hidden layer
// between two barriers), the weights come from L2 in fragment order (one 1 KB load
// per wave per 32-wide output tile and 16-wide K step), and only the input rows (FP32)
// and the output rows (FP32) touch HBM.  The layered form writes and re-reads every
// hidden activation (64 MiB each way per hidden layer at batch 65,536).
//
// Eight waves; in a layer of N outputs wave w takes the 32-wide output tiles w, w + 8
// (N = 512: two; N = 256: one) for all MT 32-row M tiles.  A hidden layer computes the
// transposed product (weights as the first operand), so a lane holds four consecutive
// features of one row and writes its BF16 activations eight bytes at a time, a quarter
// of the LDS writes and addresses of one value each.  K runs in 16-wide steps in order
// with v_mfma_f32_32x32x16_bf16, the same products in the same order and the same
// epilogue roundings (bias, SiLU, BF16) as the layered GEMM kernels, so the outputs are
// bit-identical to theirs.
//
// What bounds it: up to 8,192 rows a workgroup takes 32 rows, so that the batch spreads over
// the CUs, and the time is one CU's stream of the weights (1.85 MB at 64 B a cycle, 13 us)
// and the layers' latencies: 24 us up to 2,048 rows, 31 at 8,192 (57 and 63 us with 128
// rows a workgroup).  Beyond, 64 rows, two workgroups on a CU at 122 registers: matrix
// cores (49 us at batch 65,536), SiLU epilogues (an exp2 and a reciprocal at a quarter rate
// each, 42 us) and the weight stream (50 us) follow one another, 0.141-0.144 ms in all, as
// with one workgroup of 128 rows.
#include "mcl_device.h"
#include "mlp_internal.h"

namespace mcl {
namespace mlp {
namespace {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

constexpr int kWavesF = 8;

// Weight fragments in flight: kAhead K steps of the wave's two tiles.
template <int PD>
struct Ring {
    bf16x8 f[PD + 1][2];
};

template <int PD, int FN>
__device__ __forceinline__ void fetch_first(const bf16* const (&w)[2], Ring<PD>& r)
{
#pragma unroll
    for (int s = 0; s < PD; ++s)
#pragma unroll
        for (int j = 0; j < FN; ++j) r.f[s][j] = *reinterpret_cast<const bf16x8*>(w[j] + s * 512);
}

// acc[i][j] += rows 32 i .. of act (LDS, stride lda) and the wave's output tile j over
// KS K steps; SWAP: transposed (lane: a row, registers: features).  Straight-line
// code, each step's weight fragments fetched PD steps ahead of its products (the
// first PD by fetch_first, during the layer before); the scheduling barriers keep
// that order.
template <int MT, int FN, int KS, int PD, bool SWAP>
__device__ __forceinline__ void fused_products(const bf16* act, int lda, const bf16* const (&w)[2],
                                               Ring<PD>& ring, f32x16 (&acc)[MT][2])
{
    static_assert(KS >= PD, "the ring is filled before the first product");
    const int lane = (int)(threadIdx.x & 63u);
    const bf16* ar = act + (lane & 31) * lda + 8 * (lane >> 5);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        if (s + PD < KS) {
#pragma unroll
            for (int j = 0; j < FN; ++j)
                ring.f[(s + PD) % (PD + 1)][j] = *reinterpret_cast<const bf16x8*>(w[j] + (s + PD) * 512);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const bf16x8 av = *reinterpret_cast<const bf16x8*>(ar + i * 32 * lda + 16 * s);
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const bf16x8 wv = ring.f[s % (PD + 1)][j];
                acc[i][j] = SWAP ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv, av, acc[i][j], 0, 0, 0)
                                 : __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, wv, acc[i][j], 0, 0, 0);
            }
        }
    }
}

// The wave's tiles of layer L; a 256-wide layer has one a wave, and the second pointer
// repeats it (it is fetched ahead like the first, so it stays inside the weights).
__device__ __forceinline__ void tile_ptrs(const DeLayer& L, const bf16* (&w)[2])
{
    const int lane = (int)(threadIdx.x & 63u), wave = (int)(threadIdx.x >> 6);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int t = wave + kWavesF * j;
        w[j] = L.w + ((int64_t)(32 * t < L.out ? t : wave) * (L.kp / 16) * 64 + lane) * 8;
    }
}

// A hidden layer: products, then (after every wave has read the layer's input) bias, SiLU
// and the BF16 activations in place; the next layer's first fragments (FNX tiles) are
// fetched before the epilogue.
template <int MT, int KS, int PD, int FNX>
__device__ __forceinline__ void hidden_layer(bf16* act, int lda, const DeLayer& L, const DeLayer& next,
                                             const bf16* (&w)[2], Ring<PD>& ring)
{
    const int lane = (int)(threadIdx.x & 63u), wave = (int)(threadIdx.x >> 6);
    f32x16 acc[MT][2];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x16{};
    fused_products<MT, 2, KS, PD, true>(act, lda, w, ring, acc);
    tile_ptrs(next, w);
    fetch_first<PD, FNX>(w, ring);
    lds_barrier();                                 // the layer's input is read
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int n = 32 * (wave + kWavesF * j) + 8 * q + 4 * (lane >> 5);
            const float4 b = *reinterpret_cast<const float4*>(L.b + n);
            const float bn[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                bf16x4 v;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float z = acc[i][j][4 * q + r] + bn[r];
                    v[r] = (bf16)(z * sigmoid(z));
                }
                *reinterpret_cast<bf16x4*>(act + (32 * i + (lane & 31)) * lda + n) = v;
            }
        }
    }
    lds_barrier();                                 // the layer's output is written
}

// MT: 32-row M tiles of a workgroup; NO: output tiles of a wave (n_out = 256 NO); PD: K
// steps fetched ahead.
template <int MT, int NO, int PD>
__global__ __launch_bounds__(64 * kWavesF) __attribute__((amdgpu_waves_per_eu(4, 4)))
void infer_fused_kernel(const float* x, int B, int n_in, DeNet net, float* y)
{
    extern __shared__ __align__(16) unsigned char smem_f[];
    bf16* act = reinterpret_cast<bf16*>(smem_f);
    constexpr int kRows = 32 * MT, n_out = 256 * NO;
    const int lda = net.lda;
    const int lane = (int)(threadIdx.x & 63u), wave = (int)(threadIdx.x >> 6);
    const int64_t row0 = (int64_t)blockIdx.x * kRows;
    const int valid = (int)(B - row0 < kRows ? B - row0 : kRows);    // a multiple of 32
    const bf16* w[2];
    Ring<PD> ring;
    tile_ptrs(net.L[0], w);
    fetch_first<PD, 2>(w, ring);
    // input rows: FP32 -> BF16, zero-padded to the first layer's K (and beyond B)
    for (int e = (int)threadIdx.x; e < kRows * 64; e += 64 * kWavesF) {
        const int r = e >> 6, k = e & 63;
        act[r * lda + k] = (bf16)(k < n_in && r < valid ? x[(row0 + r) * n_in + k] : 0.0f);
    }
    lds_barrier();
    // the shapes the host admits: hidden layers 512 wide (the first with 64 padded
    // inputs), the output layer 256 or 512 wide
    const int last = net.n_layers - 1;
    hidden_layer<MT, 4, PD, 2>(act, lda, net.L[0], net.L[1], w, ring);
    for (int l = 1; l < last; ++l) hidden_layer<MT, 32, PD, 2>(act, lda, net.L[l], net.L[l + 1], w, ring);
    f32x16 acc[MT][2];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x16{};
    fused_products<MT, NO, 32, PD, false>(act, lda, w, ring, acc);
#pragma unroll
    for (int j = 0; j < NO; ++j) {
        const int n = 32 * (wave + kWavesF * j) + (lane & 31);
        const float bn = net.L[last].b[n];
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            if (32 * i >= valid) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = 32 * i + 8 * (r / 4) + 4 * (lane >> 5) + (r % 4);
                y[(row0 + m) * n_out + n] = acc[i][j][r] + bn;
            }
        }
    }
}

template <int MT, int PD>
const void* fused_fn(int n_out)
{
    return n_out == 256 ? reinterpret_cast<const void*>(infer_fused_kernel<MT, 1, PD>)
                        : reinterpret_cast<const void*>(infer_fused_kernel<MT, 2, PD>);
}

template <int MT, int PD>
hipError_t launch_fused(const float* x, int B, int n_in, const DeNet& net, float* y, int n_out,
                        hipStream_t stream)
{
    const dim3 grid((unsigned)((B + 32 * MT - 1) / (32 * MT))), block(64 * kWavesF);
    const unsigned lds = (unsigned)(32 * MT * net.lda * sizeof(bf16));
    if (n_out == 256)
        hipLaunchKernelGGL((infer_fused_kernel<MT, 1, PD>), grid, block, lds, stream, x, B, n_in, net, y);
    else
        hipLaunchKernelGGL((infer_fused_kernel<MT, 2, PD>), grid, block, lds, stream, x, B, n_in, net, y);
    return hipGetLastError();
}

// Largest batch at which a workgroup takes 32 rows: as many workgroups as CUs (8,192 rows: 31
// us, 63 with 128 a workgroup; just past it 64 rows take 40 us).
constexpr int kSmallBatch = 32 * 256;
constexpr int kAheadSmall = 4, kAheadLarge = 2;

}  // namespace

int infer_fused_lds(const DeNet& net) { return (int)(64 * net.lda * sizeof(bf16)); }

bool infer_fused_ok(const DeNet& net)
{
    if (net.n_layers < 2) return false;
    for (int l = 0; l + 1 < net.n_layers; ++l)
        if (net.L[l].out != 512 || net.L[l].kp != (l == 0 ? 64 : 512)) return false;
    const DeLayer& o = net.L[net.n_layers - 1];
    return (o.out == 256 || o.out == 512) && o.kp == 512;
}

hipError_t infer_fused_prepare(int lds_bytes)
{
    hipError_t e = hipSuccess;
    for (int n_out : {256, 512}) {
        for (const void* f : {fused_fn<1, kAheadSmall>(n_out), fused_fn<2, kAheadLarge>(n_out)})
            if (e == hipSuccess)
                e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    }
    return e;
}

hipError_t infer_fused(const float* x, int B, int n_in, const DeNet& net, float* y, int n_out,
                       hipStream_t stream)
{
    return B <= kSmallBatch ? launch_fused<1, kAheadSmall>(x, B, n_in, net, y, n_out, stream)
                            : launch_fused<2, kAheadLarge>(x, B, n_in, net, y, n_out, stream);
}

}  // namespace mlp
}  // namespace mcl
