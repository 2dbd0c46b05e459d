// hd_mlp.hip -- learned Lanczos start vector: an amplitude MLP evaluated and
// trained with BF16 MFMA kernels (FP32 accumulation, FP32 master weights).
//
// No reference counterpart: the reference's only warm-start hook is the ARPACK
// initial-vector file (src/utilities/wrappers/arpack_wrapper.hpp:753-774,
// --use-initial).  The network maps an occupation bitstring plus Hamiltonian
// parameters to (log|psi_s|, sign logit_s) for S amplitudes (the S lowest
// eigenvectors it was trained on; S = 1: the ground state):
//     features (n_bits occupations, n_params parameters, zero padded to 64)
//     -> 256 -> 256 -> 256 (SiLU) -> 2 S
//
// Training runs its layers through one GEMM kernel, C[M x N] = A[M x K] . B[N x K]^T with
// both operands K-contiguous in BF16, FP32 accumulation in
// v_mfma_f32_32x32x16_bf16 (a 64-lane wavefront owns a 32x32 output tile; four
// waves make a 64x64 block tile).  Epilogues fuse bias + SiLU (forward) and the
// SiLU derivative (backward) and write BF16 activations in row-major and, for
// training, transposed layout so that every backward GEMM again sees
// K-contiguous operands.  MFMA operand layout (lane l, 0..63):
//     A: row l%32, k = 8*(l/32) .. +7      B: column l%32, k = 8*(l/32) .. +7
//     D: column l%32, register i -> row (i/4)*8 + (l/32)*4 + i%4
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>

#include "hd_internal.hpp"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

namespace hd {

constexpr int kIn = 64;      // padded input width
constexpr int kW = 256;      // hidden width
constexpr int kOutPad = 64;  // padded output width (2 used)

enum { EPI_STORE = 0, EPI_BIAS_SILU = 1, EPI_DSILU = 2, EPI_BIAS = 3 };

HD_DEV float silu(float z) { return z / (1.f + __expf(-z)); }
HD_DEV float dsilu(float z)
{
    const float s = 1.f / (1.f + __expf(-z));
    return s * (1.f + z * (1.f - s));
}

struct GemmArgs {
    int M, N, K;
    const __bf16* A; int lda;
    const __bf16* B; int ldb;
    float* C; int ldc;          // FP32 output (pre-activation z, or raw result)
    const float* bias;          // EPI_BIAS_SILU / EPI_BIAS
    const float* zin; int ldz;  // EPI_DSILU: pre-activation of the layer below
    __bf16* H; int ldh;         // BF16 output, row-major (nullable)
    __bf16* HT; int ldht;       // BF16 output, transposed (nullable)
};

// acc += A . B^T over K columns (a multiple of 16) from a lane's operand addresses.
// Eight steps' loads are issued together: the grids leave few waves per CU, so
// a step that waited for its own loads cost a memory latency.
HD_DEV f32x16 mfma_strip(const __bf16* pa, const __bf16* pb, int K, f32x16 acc)
{
    constexpr int U = 8;
    int k = 0;
    for (; k + 16 * U <= K; k += 16 * U) {
        bf16x8 a[U], b[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            a[u] = *reinterpret_cast<const bf16x8*>(pa + k + 16 * u);
            b[u] = *reinterpret_cast<const bf16x8*>(pb + k + 16 * u);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[u], b[u], acc, 0, 0, 0);
    }
    for (; k < K; k += 16) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(pa + k);
        const bf16x8 b = *reinterpret_cast<const bf16x8*>(pb + k);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
    }
    return acc;
}

// M, N multiples of 64, K a multiple of 16 (buffers are padded by the callers).
template <int EPI>
__global__ void __launch_bounds__(256) k_gemm(GemmArgs g)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m0 = blockIdx.y * 64 + (wave >> 1) * 32;
    const int n0 = blockIdx.x * 64 + (wave & 1) * 32;
    const int r = lane & 31, kh = (lane >> 5) * 8;
    const __bf16* pa = g.A + (size_t)(m0 + r) * g.lda + kh;
    const __bf16* pb = g.B + (size_t)(n0 + r) * g.ldb + kh;
    f32x16 acc = {};
    acc = mfma_strip(pa, pb, g.K, acc);
    const int col = n0 + r;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int row = m0 + (i >> 2) * 8 + (lane >> 5) * 4 + (i & 3);
        float v = acc[i];
        if (EPI == EPI_BIAS_SILU || EPI == EPI_BIAS) v += g.bias[col];
        if (g.C) g.C[(size_t)row * g.ldc + col] = v;
        float h = v;
        if (EPI == EPI_BIAS_SILU) h = silu(v);
        if (EPI == EPI_DSILU) h = v * dsilu(g.zin[(size_t)row * g.ldz + col]);
        if (g.H) g.H[(size_t)row * g.ldh + col] = (__bf16)h;
        if (g.HT) g.HT[(size_t)col * g.ldht + row] = (__bf16)h;
    }
}

// Input features: occupations of n_bits orbitals, then n_params parameters.  A
// thread makes eight columns of one state: 16 bytes of the row-major copy, and
// two bytes in each of eight rows of the transposed one, neighbouring states
// side by side (32 states x 8 column groups per block).
__global__ void __launch_bounds__(256) k_featurize(int64_t n, int64_t npad, const uint64_t* __restrict__ states,
                            const float* __restrict__ params, int per_sample, int n_bits, int n_params,
                            __bf16* __restrict__ H0, __bf16* __restrict__ H0T)
{
    const int64_t b = (int64_t)blockIdx.x * 32 + (threadIdx.x & 31);
    const int k0 = (threadIdx.x >> 5) * 8;
    if (b >= npad) return;
    const bool live = b < n;
    const uint64_t s = live ? states[b] : 0ull;
    const float* p = params + (per_sample ? b * n_params : 0);
    bf16x8 v;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int k = k0 + j;
        float f = 0.f;
        if (live) {
            if (k < n_bits) f = (float)((s >> k) & 1ull);
            else if (k < n_bits + n_params) f = p[k - n_bits];
        }
        v[j] = (__bf16)f;
        H0T[(size_t)k * npad + b] = v[j];
    }
    *reinterpret_cast<bf16x8*>(H0 + b * kIn + k0) = v;
}

// loss and dL/dout for out = (log|psi_s|, sign logit_s), s < S, against
// targets (log|psi_s|, sign_s, weight_s) per state (3 S floats per sample);
// lambda weights the sign term.  A thread takes four amplitudes (eight columns)
// of one state, as k_featurize.
__global__ void __launch_bounds__(256) k_loss(int64_t n, int64_t npad, int S, const float* __restrict__ out, const float* __restrict__ tgt,
                       float lambda, float inv_n, __bf16* __restrict__ d4, __bf16* __restrict__ d4T,
                       float* __restrict__ partial)
{
    __shared__ float red[256];
    const int64_t b = (int64_t)blockIdx.x * 32 + (threadIdx.x & 31);
    const int c0 = (threadIdx.x >> 5) * 8;
    float l = 0.f;
    if (b < npad) {
        bf16x8 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int st = (c0 >> 1) + j;
            float g0 = 0.f, g1 = 0.f;
            if (b < n && st < S) {
                const float o0 = out[b * kOutPad + 2 * st], o1 = out[b * kOutPad + 2 * st + 1];
                const float* t = tgt + (b * S + st) * 3;
                const float a = t[0], sg = t[1], w = t[2];
                const float e = o0 - a;
                const float m = -sg * o1;  // softplus(m) = log(1 + exp(-s o1))
                const float sp = m > 20.f ? m : log1pf(__expf(m));
                l += w * (e * e + lambda * sp) * inv_n;
                g0 = 2.f * w * e * inv_n;
                g1 = -lambda * w * sg * (1.f / (1.f + __expf(-m))) * inv_n;
            }
            v[2 * j] = (__bf16)g0;
            v[2 * j + 1] = (__bf16)g1;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) d4T[(size_t)(c0 + j) * npad + b] = v[j];
        *reinterpret_cast<bf16x8*>(d4 + b * kOutPad + c0) = v;
    }
    red[threadIdx.x] = l;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// The parameters, their moments and gradients are flat arrays in the order of
// hd_mlp_get_weights: per layer W (rows x cols, padded shape), then b.
constexpr int kRows[4] = {kW, kW, kW, kOutPad};
constexpr int kCols[4] = {kIn, kW, kW, kW};
HD_DEV constexpr int rows_of(int l) { return l == 3 ? kOutPad : kW; }
HD_DEV constexpr int cols_of(int l) { return l == 0 ? kIn : kW; }
constexpr int kOff[5] = {0, kW * kIn + kW, kW * kIn + kW + kW * kW + kW, kW * kIn + kW + 2 * (kW * kW + kW),
                         kW * kIn + kW + 2 * (kW * kW + kW) + kOutPad * kW + kOutPad};
constexpr int kParams = kOff[4];
HD_DEV constexpr int off_of(int l)
{
    return l == 0 ? 0 : l == 1 ? kW * kIn + kW : l == 2 ? kW * kIn + kW + kW * kW + kW : kW * kIn + kW + 2 * (kW * kW + kW);
}

// Weight and bias gradients of all layers, dW_l = d_{l+1}^T h_l and db_l = sum d_{l+1},
// split over the batch: block (t, z) adds the samples [z kc, (z+1) kc) of one 64 x 64
// tile into part[z].  A batch of 4,096 gives 40 tiles, 16 for the largest layer alone:
// unsplit, 16 blocks walked 256 K-steps each (66 us per layer); split 16 ways the four
// layers take 18 us together.
struct WgradArgs {
    const __bf16* dT[4];  // [rows][M]
    const __bf16* hT[4];  // [cols][M]
    int64_t M;
    int kc;
    float* part;
};
constexpr int kWgradTiles = 4 + 16 + 16 + 4;
constexpr int kMaxSplits = 16;

__global__ void __launch_bounds__(256) k_wgrad(WgradArgs g)
{
    int t = blockIdx.x, l = 0;
    if (t >= 36) { l = 3; t -= 36; }
    else if (t >= 20) { l = 2; t -= 20; }
    else if (t >= 4) { l = 1; t -= 4; }
    const int cols = cols_of(l), nt = cols / 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m0 = (t / nt) * 64 + (wave >> 1) * 32, n0 = (t % nt) * 64 + (wave & 1) * 32;
    const int r = lane & 31, kh = (lane >> 5) * 8;
    const int64_t k0 = (int64_t)blockIdx.y * g.kc, k1 = min(k0 + g.kc, g.M);
    const __bf16* pa = g.dT[l] + (size_t)(m0 + r) * g.M + kh;
    const __bf16* pb = g.hT[l] + (size_t)(n0 + r) * g.M + kh;
    const bool bias = n0 == 0;
    f32x16 acc = {};
    float bs = 0.f;
    const int K = (int)(k1 - k0);
    acc = mfma_strip(pa + k0, pb + k0, K, acc);
    if (bias)
        for (int k = 0; k < K; k += 16) {
            const bf16x8 a = *reinterpret_cast<const bf16x8*>(pa + k0 + k);
            bs += (((float)a[0] + (float)a[1]) + ((float)a[2] + (float)a[3])) +
                  (((float)a[4] + (float)a[5]) + ((float)a[6] + (float)a[7]));
        }
    float* w = g.part + (size_t)blockIdx.y * kParams + off_of(l);
#pragma unroll
    for (int i = 0; i < 16; ++i) w[(m0 + (i >> 2) * 8 + (lane >> 5) * 4 + (i & 3)) * cols + n0 + r] = acc[i];
    if (bias) {
        bs += __shfl_xor(bs, 32, 64);
        if (lane < 32) w[rows_of(l) * cols + m0 + r] = bs;
    }
}

// One pass over all parameters.  GRAD: the splits' partial gradients summed in
// order.  STEP: Adam (Kingma and Ba, ICLR 2015) on the FP32 master copy.  COPY: the
// BF16 copies W, W^T and, for inference, the fragment order.  One launch instead
// of four bias sums, eight Adam launches, four conversions and a packing.
struct ParamArgs {
    const float* part;
    int splits;
    float *w, *g, *m, *v;
    float lr, b1, b2, c1, c2, eps;
    __bf16* wb[4];
    __bf16* wbT[4];
    __bf16* wf;
};

template <bool GRAD, bool STEP, bool COPY>
__global__ void __launch_bounds__(256) k_params(ParamArgs a)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= kParams) return;
    float gr = 0.f;
    if (GRAD) {
        for (int z = 0; z < a.splits; ++z) gr += a.part[(size_t)z * kParams + i];
        a.g[i] = gr;
    }
    float w = a.w[i];
    if (STEP) {
        const float mi = a.b1 * a.m[i] + (1.f - a.b1) * gr;
        const float vi = a.b2 * a.v[i] + (1.f - a.b2) * gr * gr;
        a.m[i] = mi;
        a.v[i] = vi;
        w -= a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
        a.w[i] = w;
    }
    if (COPY) {
        const int l = i >= off_of(3) ? 3 : i >= off_of(2) ? 2 : i >= off_of(1) ? 1 : 0;
        const int q = i - off_of(l), cols = cols_of(l), rows = rows_of(l);
        if (q >= rows * cols) return;  // a bias
        const int r = q / cols, k = q % cols;
        const __bf16 v = (__bf16)w;
        a.wb[l][q] = v;
        a.wbT[l][(size_t)k * rows + r] = v;
        // fragment f = tile * (K/16) + k/16 of each layer in turn, lane's eight
        // values W[32 tile + lane%32][16 (k/16) + 8 (lane/32) ..+7]; of the last layer
        // the first 32 rows
        const int base = l == 0 ? 0 : l == 1 ? 32 : l == 2 ? 160 : 288;
        if (r < (l == 3 ? 32 : kW))
            a.wf[(size_t)(base + (r >> 5) * (cols >> 4) + (k >> 4)) * 512 + ((r & 31) + ((k >> 3) & 1) * 32) * 8 + (k & 7)] = v;
    }
}

// ---------------------------------------------------------------- inference
//
// The whole network for NW * 32 states per group in one launch, a wavefront per
// 32 states.  The products run transposed, D = W . H^T: the weights are the A
// operand, the activations the B operand, so a lane's 16 outputs all belong to
// its own state (column l%32) and go through bias and SiLU into the next
// layer's B operand without leaving the registers: only the rows 4-7 / 8-11 of
// every 16 change lane halves (v_permlane32_swap).  Every output is the MFMA
// sequence of k_gemm (32x32x16 tiles, K ascending in steps of 16).
//
// The weights are read in the order of the A fragments (k_params: 1 KiB per
// 32 x 16 fragment, lane l's 16 bytes at 16 l), ten chunks of 32 fragments
// (layer 1 in one, layers 2 and 3 in four each, the output layer in the last),
// double-buffered in LDS: the next chunk's loads are in flight into registers
// while the waves multiply the current one.  Blocks are persistent (one per CU)
// and walk the state groups, so the pipeline also runs across groups.
//
// Bound: the vector instructions (67% of the cycles; the SiLU is 768 of 44 cycles
// per state) beside the MFMAs (31%) and the fragment reads from LDS.  Over the
// N=12, 2S=33 sector (7.76M states, S = 5) 3.55 ms, 0.68 PFLOP/s on the padded
// work, against 11.6 ms for a kernel that kept the activations in LDS (512-byte
// rows, every access a bank conflict, two barriers per 32 columns of weights).
// Two sets of 32 states per wave, which halve the fragment reads, need the AGPRs
// for the activations and were slower (4.1 ms), as was a SiLU pass after each
// tile pair's products instead of between them (3.9 ms).
constexpr int kFrag = 512;          // BF16 elements of one 32 x 16 weight fragment
constexpr int kChunk = 32 * kFrag;  // elements of one staged chunk (32 KiB)
constexpr int kChunks = 10;
constexpr int kOutT = 32;           // outputs of the last layer's tile (n_out <= 32)

struct InferArgs {
    int64_t n;
    const uint64_t* states;
    const float* params;  // n_params values, per state when per_sample
    int per_sample, n_bits, n_params;
    const __bf16* wf;     // packed weights, kChunks * kChunk elements
    const float* b[4];
    int n_out;            // live outputs per state: 2 per amplitude (log|psi|, sign logit)
    float* out;           // n x n_out
    float* partial_max;   // per workgroup and amplitude s: largest output 2s over its states
};

// z / (1 + exp(-z)) with the quotient from v_rcp_f32 and one correction step (the
// remainder z - q d, exact in the fma), instead of the IEEE division sequence.
// v_div_fixup_f32 gives the special cases (+inf for z = +inf, -0 where the exponential
// overflows, NaN for -inf and NaN).  Of all 2^32 floats the bits differ from the
// division's in -88.72 < z < -87.33 alone, where 1 / d is subnormal and v_rcp_f32 gives
// 0: -0 instead of -9e-37 to -3e-37.
HD_DEV float silu_fast(float z)
{
    const float d = 1.f + __builtin_amdgcn_exp2f(z * -1.44269504088896341f);
    const float r = __builtin_amdgcn_rcpf(d);
    const float q = z * r;
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-q, d, z), r, q), d, z);
}

HD_DEV uint32_t pack_bf16(float a, float b)
{
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    bf16x2 v;
    v[0] = (__bf16)a;
    v[1] = (__bf16)b;
    return __builtin_bit_cast(uint32_t, v);
}

// Eight consecutive outputs (bias and SiLU applied) of the lane's state for one
// 16-row block: lo holds rows 4h .. 4h+3 and hi rows 8+4h .. 8+4h+3 of lane half h;
// the swap leaves half h with rows 8h .. 8h+7, the B operand's order.
HD_DEV bf16x8 to_operand(const float (&lo)[4], const float (&hi)[4])
{
    uint32_t v[4];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const auto r = __builtin_amdgcn_permlane32_swap(pack_bf16(lo[2 * q], lo[2 * q + 1]),
                                                        pack_bf16(hi[2 * q], hi[2 * q + 1]), false, false);
        v[q] = r[0];
        v[2 + q] = r[1];
    }
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 p = {v[0], v[1], v[2], v[3]};
    return __builtin_bit_cast(bf16x8, p);
}

// One output tile (32 rows): acc = the tile's weights times `in`, KS steps of one
// fragment each.  Between the MFMAs the previous tile's 16 outputs `prev` go
// through bias (pb, in LDS) and SiLU into out[0] and out[1]: a step's vector
// instructions issue while its MFMA runs in the matrix core.  All of `prev` is
// done two steps before the end, so a tile that opens the next layer may have the
// previous layer's last tile as its last two inputs.
template <int KS, bool PREV>
HD_DEV f32x16 infer_tile(const __bf16* wt, const bf16x8* in, const f32x16& prev, const float* pb, bf16x8* out, int lane)
{
    const bf16x8* w = reinterpret_cast<const bf16x8*>(wt) + lane;
    const float* pl = pb + (lane >> 5) * 4;
    constexpr int kAhead = 2;  // fragments read ahead
    bf16x8 a[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) a[i] = w[i * (kFrag / 8)];
    f32x16 acc = {};
    float v[16];
    float4 b4 = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[ks % kAhead], in[ks], acc, 0, 0, 0);
        if (ks + kAhead < KS) a[ks % kAhead] = w[(ks + kAhead) * (kFrag / 8)];
        if constexpr (PREV) {
            // steps 0 and 1 take two elements, steps 2 to 13 one (KS = 16); four each (KS = 4)
            const int e0 = KS == 4 ? 4 * ks : ks < 2 ? 2 * ks : ks + 2;
            const int e1 = KS == 4 ? 4 * ks + 4 : ks < 2 ? 2 * ks + 2 : ks < 14 ? ks + 3 : ks + 2;
#pragma unroll
            for (int e = e0; e < e1; ++e) {
                if ((e & 3) == 0) b4 = *reinterpret_cast<const float4*>(pl + (e >> 2) * 8);
                const float be = (e & 3) == 0 ? b4.x : (e & 3) == 1 ? b4.y : (e & 3) == 2 ? b4.z : b4.w;
                v[e] = silu_fast(prev[e] + be);
                if ((e & 7) == 7) {
                    const float lo[4] = {v[e - 7], v[e - 6], v[e - 5], v[e - 4]};
                    const float hi[4] = {v[e - 3], v[e - 2], v[e - 1], v[e]};
                    out[e >> 3] = to_operand(lo, hi);
                }
            }
        }
        // keeps pairs of steps apart: hoisting more fragments and SiLUs spills
        if (ks % 2 == 1) __builtin_amdgcn_sched_barrier(0);
    }
    return acc;
}

template <int NW>
__global__ void __launch_bounds__(NW * 64, NW / 4) k_mlp_infer(InferArgs g)
{
    constexpr int T = NW * 64, NS = NW * 32, NP = kChunk / (T * 8);
    __shared__ __align__(16) __bf16 wbuf[2][kChunk];
    __shared__ __align__(16) float sb[3 * kW + kOutT];
    __shared__ float stage[NS * kOutT];  // one group's outputs, n_out per state
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 31, half = lane >> 5;
    for (int i = tid; i < 3 * kW + kOutT; i += T) sb[i] = g.b[i / kW][i % kW];
    // chunk c into buffer `buf`, straight from global memory to LDS (each wave
    // instruction moves 64 x 16 bytes to consecutive LDS addresses); settle() waits
    // for the loads and for every wave
    auto fetch = [&](int c, int buf) {
#pragma unroll
        for (int i = 0; i < NP; ++i)
            __builtin_amdgcn_global_load_lds(
                (const __attribute__((address_space(1))) void*)(g.wf + (size_t)c * kChunk + (i * T + tid) * 8),
                (__attribute__((address_space(3))) void*)&wbuf[buf][(i * T + wave * 64) * 8], 16, 0, 0);
    };
    auto settle = [&]() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    };
    fetch(0, 0);
    settle();
    float mx[16 / NW];  // running maxima of amplitudes wave + NW q (16 at most)
#pragma unroll
    for (float& m : mx) m = -3.0e38f;
    const int64_t groups = (g.n + NS - 1) / NS;
    for (int64_t grp = blockIdx.x; grp < groups; grp += gridDim.x) {
        const int64_t s0 = grp * NS + wave * 32;
        bf16x8 x[kIn / 16], h1[kW / 16], h2[kW / 16];
        {   // features of state s0 + r, columns 16 ks + 8 half ..+7
            const int64_t b = s0 + r;
            const bool live = b < g.n;
            uint64_t st = live ? g.states[b] : 0ull;
            if (g.n_bits < 64) st &= (1ull << g.n_bits) - 1;
            const float* p = g.params + (g.per_sample && live ? b * g.n_params : 0);
            uint32_t xd[kIn / 16][4];  // two features per word, 0 or 1.0 (0x3F80) each
#pragma unroll
            for (int ks = 0; ks < kIn / 16; ++ks)
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    const uint32_t t = (uint32_t)(st >> (ks * 16 + half * 8 + 2 * d));
                    xd[ks][d] = ((t & 1u) | ((t & 2u) << 15)) * 0x3F80u;
                }
            for (int i = 0; i < g.n_params; ++i) {
                const int k = g.n_bits + i;
                const uint32_t v = pack_bf16(live ? p[i] : 0.f, 0.f) << ((k & 1) * 16);
                const bool mine = half == ((k >> 3) & 1);
#pragma unroll
                for (int w = 0; w < kIn / 4; ++w)  // word w: columns 16 (w/4) + 8 half + 2 (w%4)
                    if (w == (k >> 4) * 4 + ((k & 7) >> 1) && mine) xd[w >> 2][w & 3] |= v;
            }
#pragma unroll
            for (int ks = 0; ks < kIn / 16; ++ks) x[ks] = __builtin_bit_cast(bf16x8, xd[ks]);
        }
        // chunk c is in wbuf[c & 1]; ten chunks per group keep the parity
        fetch(1, 1);
        f32x16 acc = infer_tile<kIn / 16, false>(wbuf[0], x, f32x16{}, sb, h1, lane);
#pragma unroll
        for (int t = 1; t < 8; ++t)
            acc = infer_tile<kIn / 16, true>(wbuf[0] + t * (kIn / 16) * kFrag, x, acc, sb + (t - 1) * 32, h1 + 2 * t - 2, lane);
        settle();
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            fetch(2 + c, c & 1);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int t = 2 * c + u;  // tile t of layer 2; tile t - 1 (or layer 1's last) is finished
                acc = infer_tile<kW / 16, true>(wbuf[(1 + c) & 1] + u * (kW / 16) * kFrag, h1, acc,
                                                sb + (t ? kW + (t - 1) * 32 : 7 * 32), t ? h2 + 2 * t - 2 : h1 + 14, lane);
            }
            settle();
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            fetch(6 + c, c & 1);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int t = 2 * c + u;
                acc = infer_tile<kW / 16, true>(wbuf[(5 + c) & 1] + u * (kW / 16) * kFrag, h2, acc,
                                                sb + kW + (t ? kW + (t - 1) * 32 : 7 * 32), t ? h1 + 2 * t - 2 : h2 + 14, lane);
            }
            settle();
        }
        fetch(0, 0);
        acc = infer_tile<kW / 16, true>(wbuf[1], h1, acc, sb + 2 * kW + 7 * 32, h1 + 14, lane);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int row = (i >> 2) * 8 + half * 4 + (i & 3);
            if (row < g.n_out) stage[(wave * 32 + r) * g.n_out + row] = acc[i] + sb[3 * kW + row];
        }
        settle();
        // the group's outputs are contiguous in g.out
        const int64_t left = g.n - grp * NS;
        const int live_states = left < NS ? (int)left : NS;
        const int live = live_states * g.n_out;
        float* o = g.out + grp * NS * g.n_out;
        for (int i = tid; i < live; i += T) o[i] = stage[i];
#pragma unroll
        for (int q = 0; q < 16 / NW; ++q) {
            const int s = wave + NW * q;
            if (2 * s < g.n_out)
                for (int i = lane; i < live_states; i += 64) mx[q] = fmaxf(mx[q], stage[i * g.n_out + 2 * s]);
        }
        // the next write to `stage` comes after the next group's barriers
    }
#pragma unroll
    for (int q = 0; q < 16 / NW; ++q) {
        const int s = wave + NW * q;
        float m = mx[q];
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
        if (lane == 0 && 2 * s < g.n_out) g.partial_max[(int64_t)blockIdx.x * (g.n_out / 2) + s] = m;
    }
}

// Launch shape: one persistent block per CU.  Eight waves (two per SIMD, so one's
// SiLU overlaps the other's MFMAs) once every CU has a group of 256 states; below
// that four waves and 128 states, which spreads a small sector over twice the CUs.
struct InferGrid {
    int nw;
    unsigned blocks;
};
static InferGrid infer_grid(int64_t n, int n_cu)
{
    InferGrid q;
    q.nw = n >= (int64_t)n_cu * 256 ? 8 : 4;
    q.blocks = (unsigned)std::min<int64_t>(n_cu, (n + q.nw * 32 - 1) / (q.nw * 32));
    return q;
}

static void infer_launch(const InferArgs& a, const InferGrid& q, hipStream_t st)
{
    if (q.nw == 8) hipLaunchKernelGGL(k_mlp_infer<8>, dim3(q.blocks), dim3(512), 0, st, a);
    else hipLaunchKernelGGL(k_mlp_infer<4>, dim3(q.blocks), dim3(256), 0, st, a);
}

// shift[s] = max over workgroups of partial[w * S + s] (one block per amplitude, fixed order)
__global__ void __launch_bounds__(256) k_max_states(int64_t nblk, int S, const float* __restrict__ partial,
                                                    float* __restrict__ shift)
{
    __shared__ float red[256];
    const int s = blockIdx.x;
    float m = -3.0e38f;
    for (int64_t i = threadIdx.x; i < nblk; i += 256) m = fmaxf(m, partial[i * S + s]);
    red[threadIdx.x] = m;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + o]);
        __syncthreads();
    }
    if (threadIdx.x == 0) shift[s] = red[0];
}

// part[blk * S + s] = sum over this block's states of exp(2 (o_2s - shift_s)); all
// amplitudes in one pass over the outputs (S <= MS), each state's outputs read by
// one thread.
template <int MS>
__global__ void __launch_bounds__(256) k_norm2_states(int64_t n, int S, const float* __restrict__ out,
                                                      const float* __restrict__ shift, double* __restrict__ part)
{
    __shared__ double red[4][MS];
    double acc[MS];
    float sh[MS];
#pragma unroll
    for (int s = 0; s < MS; ++s) {
        acc[s] = 0.0;
        sh[s] = s < S ? shift[s] : 0.f;
    }
    for (int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x; b < n; b += (int64_t)gridDim.x * 256) {
#pragma unroll
        for (int s = 0; s < MS; ++s)
            if (s < S) acc[s] += exp(2.0 * (double)(out[b * 2 * S + 2 * s] - sh[s]));
    }
#pragma unroll
    for (int s = 0; s < MS; ++s) {
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) acc[s] += __shfl_xor(acc[s], d, 64);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][s] = acc[s];
    }
    __syncthreads();
    if ((int)threadIdx.x < S) {
        const int s = threadIdx.x;
        part[(int64_t)blockIdx.x * S + s] = (red[0][s] + red[1][s]) + (red[2][s] + red[3][s]);
    }
}

// inv[s] = 1 / sqrt(sum over blocks of part[blk * S + s]) (one block per amplitude,
// fixed order)
__global__ void __launch_bounds__(256) k_inv_norm_states(int nb, int S, const double* __restrict__ part,
                                                         double* __restrict__ inv)
{
    __shared__ double red[256];
    const int s = blockIdx.x;
    double t = 0.0;
    for (int b = threadIdx.x; b < nb; b += 256) t += part[(int64_t)b * S + s];
    red[threadIdx.x] = t;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) inv[s] = red[0] > 0.0 ? 1.0 / sqrt(red[0]) : 0.0;
}

// psi_b = sum_s exp(o_2s - shift_s) sign(o_2s+1) * scale_s; with one amplitude
// the scale is 1 (psi = exp(o0 - max o0) sign(o1)), with several each
// amplitude is normalised to unit length before the sum
__global__ void k_amplitude(int64_t n, int S, const float* __restrict__ out, const float* __restrict__ shift,
                            const double* __restrict__ inv, double* __restrict__ psi)
{
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= n) return;
    double v = 0.0;
    for (int s = 0; s < S; ++s) {
        const float o0 = out[b * 2 * S + 2 * s], o1 = out[b * 2 * S + 2 * s + 1];
        const double a = exp((double)(o0 - shift[s])) * (S > 1 ? inv[s] : 1.0);
        v += o1 >= 0.f ? a : -a;
    }
    psi[b] = v;
}

}  // namespace hd

using namespace hd;

// ------------------------------------------------------------------ handle

struct hd_mlp {
    int n_bits = 0, n_params = 0;
    int n_states = 1;  // amplitudes the network predicts (2 outputs each)
    hipStream_t stream = nullptr;
    int live_rows[4] = {kW, kW, kW, 2};
    // flat arrays of kParams: FP32 master (padding kept at zero), gradients, Adam moments
    float *params = nullptr, *grads = nullptr, *mom1 = nullptr, *mom2 = nullptr;
    __bf16* wb[4] = {};   // BF16 copy
    __bf16* wbT[4] = {};  // BF16 transposed copy
    __bf16* wf = nullptr; // BF16 copy in the inference kernel's fragment order
    int64_t step = 0;
    // work buffers for a batch of `cap` rows
    int64_t cap = 0;
    __bf16 *h[4] = {}, *hT[4] = {};  // h[0] = features; h[l] = layer-l output (l=1..3)
    float* z[4] = {};                // pre-activations of layers 1..3 (z[1..3]); z[0] unused
    float* out = nullptr;            // npad x 64
    __bf16 *d[5] = {}, *dT[5] = {};  // deltas: d[4] output layer, d[3..1] hidden
    float* partial = nullptr;
    float* wpart = nullptr;          // kMaxSplits x kParams partial gradients
    uint64_t* st_buf = nullptr;      // staging for host-provided batches
    float* pr_buf = nullptr;
    float* tg_buf = nullptr;
    int64_t st_cap = 0;
};

namespace {

void mlp_free_work(hd_mlp* m)
{
    for (int l = 0; l < 4; ++l) {
        dfree(m->h[l]); dfree(m->hT[l]); dfree(m->z[l]);
        m->h[l] = m->hT[l] = nullptr;
        m->z[l] = nullptr;
    }
    for (int l = 0; l < 5; ++l) {
        dfree(m->d[l]); dfree(m->dT[l]);
        m->d[l] = m->dT[l] = nullptr;
    }
    dfree(m->out); dfree(m->partial); dfree(m->wpart);
    m->out = nullptr;
    m->partial = nullptr;
    m->wpart = nullptr;
    m->cap = 0;
}

int mlp_work(hd_mlp* m, int64_t npad)
{
    if (m->cap >= npad) return HD_OK;
    mlp_free_work(m);
    const int64_t c = std::max<int64_t>(npad, 64);
    HD_CHECK(dalloc_t(&m->h[0], (size_t)c * kIn, "MLP features"));
    for (int l = 1; l < 4; ++l) {
        HD_CHECK(dalloc_t(&m->h[l], (size_t)c * kW, "MLP activations"));
        HD_CHECK(dalloc_t(&m->z[l], (size_t)c * kW, "MLP pre-activations"));
    }
    HD_CHECK(dalloc_t(&m->out, (size_t)c * kOutPad, "MLP output"));
    HD_CHECK(dalloc_t(&m->partial, (size_t)(c / 32 + 1024), "MLP partials"));
    HD_CHECK(dalloc_t(&m->wpart, (size_t)kMaxSplits * kParams, "MLP partial gradients"));
    HD_CHECK(dalloc_t(&m->hT[0], (size_t)c * kIn, "MLP features^T"));
    for (int l = 1; l < 4; ++l) HD_CHECK(dalloc_t(&m->hT[l], (size_t)c * kW, "MLP activations^T"));
    HD_CHECK(dalloc_t(&m->d[4], (size_t)c * kOutPad, "MLP output delta"));
    HD_CHECK(dalloc_t(&m->dT[4], (size_t)c * kOutPad, "MLP output delta^T"));
    for (int l = 1; l < 4; ++l) {
        HD_CHECK(dalloc_t(&m->d[l], (size_t)c * kW, "MLP deltas"));
        HD_CHECK(dalloc_t(&m->dT[l], (size_t)c * kW, "MLP deltas^T"));
    }
    m->cap = c;
    return HD_OK;
}

ParamArgs param_args(const hd_mlp* m, int splits)
{
    ParamArgs a{};
    a.part = m->wpart;
    a.splits = splits;
    a.w = m->params;
    a.g = m->grads;
    a.m = m->mom1;
    a.v = m->mom2;
    for (int l = 0; l < 4; ++l) {
        a.wb[l] = m->wb[l];
        a.wbT[l] = m->wbT[l];
    }
    a.wf = m->wf;
    return a;
}
const dim3 kParamGrid((kParams + 255) / 256);

int mlp_refresh_bf16(hd_mlp* m)
{
    hipLaunchKernelGGL((k_params<false, false, true>), kParamGrid, dim3(256), 0, m->stream, param_args(m, 0));
    HD_HIP(hipGetLastError());
    return HD_OK;
}

void gemm(hipStream_t st, int epi, const GemmArgs& g)
{
    const dim3 grid(g.N / 64, g.M / 64);
    switch (epi) {
    case EPI_STORE: hipLaunchKernelGGL(k_gemm<EPI_STORE>, grid, dim3(256), 0, st, g); break;
    case EPI_BIAS_SILU: hipLaunchKernelGGL(k_gemm<EPI_BIAS_SILU>, grid, dim3(256), 0, st, g); break;
    case EPI_DSILU: hipLaunchKernelGGL(k_gemm<EPI_DSILU>, grid, dim3(256), 0, st, g); break;
    default: hipLaunchKernelGGL(k_gemm<EPI_BIAS>, grid, dim3(256), 0, st, g); break;
    }
}

GemmArgs ga(int M, int N, int K, const __bf16* A, int lda, const __bf16* B, int ldb)
{
    GemmArgs g{};
    g.M = M; g.N = N; g.K = K;
    g.A = A; g.lda = lda; g.B = B; g.ldb = ldb;
    return g;
}

InferArgs infer_args(const hd_mlp* m, int64_t n, const uint64_t* states, const float* params, int per_sample,
                     float* out, float* partial_max)
{
    InferArgs a{};
    a.n = n;
    a.states = states;
    a.params = params;
    a.per_sample = per_sample;
    a.n_bits = m->n_bits;
    a.n_params = m->n_params;
    a.wf = m->wf;
    for (int l = 0; l < 4; ++l) a.b[l] = m->params + kOff[l] + kRows[l] * kCols[l];
    a.n_out = m->live_rows[3];
    a.out = out;
    a.partial_max = partial_max;
    return a;
}

// training's forward pass over npad rows already featurized in h[0] and hT[0]
void mlp_forward_core(hd_mlp* m, int64_t npad)
{
    const int M = (int)npad;
    for (int l = 0; l < 3; ++l) {
        const int K = l == 0 ? kIn : kW;
        GemmArgs g = ga(M, kW, K, m->h[l], K, m->wb[l], kCols[l]);
        g.C = m->z[l + 1]; g.ldc = kW;
        g.bias = m->params + kOff[l] + kRows[l] * kCols[l];
        g.H = m->h[l + 1]; g.ldh = kW;
        g.HT = m->hT[l + 1]; g.ldht = M;
        gemm(m->stream, EPI_BIAS_SILU, g);
    }
    GemmArgs g = ga(M, kOutPad, kW, m->h[3], kW, m->wb[3], kW);
    g.C = m->out; g.ldc = kOutPad;
    g.bias = m->params + kOff[3] + kRows[3] * kCols[3];
    gemm(m->stream, EPI_BIAS, g);
}

// partial gradients of the loss into wpart (*splits of them); the per-block losses
// into `partial`
int mlp_backward(hd_mlp* m, int64_t n, int64_t npad, const float* d_tgt, float lambda, int* splits)
{
    const hipStream_t st = m->stream;
    const int M = (int)npad;
    hipLaunchKernelGGL(k_loss, dim3((unsigned)((npad + 31) / 32)), dim3(256), 0, st, n, npad, m->n_states, m->out, d_tgt,
                       lambda, 1.f / (float)n, m->d[4], m->dT[4], m->partial);
    // hidden layers l = 3, 2, 1: d_l = (d_{l+1} W_{l+1}) * silu'(z_l)
    for (int l = 3; l >= 1; --l) {
        const int Kd = l == 3 ? kOutPad : kW;  // width of d_{l+1}
        GemmArgs g = ga(M, kW, Kd, m->d[l + 1], Kd, m->wbT[l], kRows[l]);
        g.zin = m->z[l]; g.ldz = kW;
        g.H = m->d[l]; g.ldh = kW;
        g.HT = m->dT[l]; g.ldht = M;
        gemm(st, EPI_DSILU, g);
    }
    WgradArgs w{};
    for (int l = 0; l < 4; ++l) {
        w.dT[l] = m->dT[l + 1];
        w.hT[l] = m->hT[l];
    }
    w.M = npad;
    // at least 64 samples per block, a multiple of 16
    w.kc = (int)std::max<int64_t>(64, ((npad + kMaxSplits - 1) / kMaxSplits + 15) / 16 * 16);
    w.part = m->wpart;
    *splits = (int)((npad + w.kc - 1) / w.kc);
    hipLaunchKernelGGL(k_wgrad, dim3(kWgradTiles, *splits), dim3(256), 0, st, w);
    HD_HIP(hipGetLastError());
    return HD_OK;
}

// The loss of the batch, after everything enqueued.
int mlp_loss(hd_mlp* m, int64_t npad, float* loss)
{
    std::vector<float> part((size_t)((npad + 31) / 32));
    HD_HIP(hipMemcpyAsync(part.data(), m->partial, sizeof(float) * part.size(), hipMemcpyDeviceToHost, m->stream));
    HD_HIP(hipStreamSynchronize(m->stream));
    double s = 0.0;
    for (float p : part) s += p;
    if (loss) *loss = (float)s;
    return HD_OK;
}

int stage_batch(hd_mlp* m, const uint64_t* states, const float* params, const float* tgt, int64_t n, bool host,
                const uint64_t** ds, const float** dp, const float** dt, int per_sample)
{
    if (!host) {
        *ds = states;
        *dp = params;
        *dt = tgt;
        return HD_OK;
    }
    if (m->st_cap < n) {
        dfree(m->st_buf); dfree(m->pr_buf); dfree(m->tg_buf);
        m->st_buf = nullptr; m->pr_buf = nullptr; m->tg_buf = nullptr;
        HD_CHECK(dalloc_t(&m->st_buf, (size_t)n, "MLP staged states"));
        HD_CHECK(dalloc_t(&m->pr_buf, (size_t)n * std::max(m->n_params, 1), "MLP staged params"));
        HD_CHECK(dalloc_t(&m->tg_buf, (size_t)n * 3 * m->n_states, "MLP staged targets"));
        m->st_cap = n;
    }
    HD_HIP(hipMemcpyAsync(m->st_buf, states, sizeof(uint64_t) * n, hipMemcpyHostToDevice, m->stream));
    HD_HIP(hipMemcpyAsync(m->pr_buf, params, sizeof(float) * (per_sample ? n : 1) * m->n_params,
                          hipMemcpyHostToDevice, m->stream));
    if (tgt)
        HD_HIP(hipMemcpyAsync(m->tg_buf, tgt, sizeof(float) * n * 3 * m->n_states, hipMemcpyHostToDevice, m->stream));
    *ds = m->st_buf;
    *dp = m->pr_buf;
    *dt = m->tg_buf;
    return HD_OK;
}

int64_t pad64(int64_t n) { return (n + 63) / 64 * 64; }

// forward and backward passes of a batch, up to the partial gradients
int batch_pass(hd_mlp* m, const uint64_t* states, const float* params, const float* tgt, int64_t n, float lambda,
               int host, int* splits)
{
    if (n <= 0) return fail(HD_ERR_ARG, "empty batch");
    const int64_t npad = pad64(n);
    HD_CHECK(mlp_work(m, npad));
    const uint64_t* ds;
    const float *dp, *dt;
    HD_CHECK(stage_batch(m, states, params, tgt, n, host != 0, &ds, &dp, &dt, 1));
    hipLaunchKernelGGL(k_featurize, dim3((unsigned)(npad / 32)), dim3(256), 0, m->stream, n, npad, ds, dp, 1, m->n_bits,
                       m->n_params, m->h[0], m->hT[0]);
    mlp_forward_core(m, npad);
    return mlp_backward(m, n, npad, dt, lambda, splits);
}

}  // namespace

extern "C" {

int hd_mlp_create(int32_t n_bits, int32_t n_params, uint64_t seed, hd_mlp** out)
{
    return hd_mlp_create_states(n_bits, n_params, 1, seed, out);
}

int hd_mlp_create_states(int32_t n_bits, int32_t n_params, int32_t n_states, uint64_t seed, hd_mlp** out)
{
    if (!out || n_bits <= 0 || n_params < 0 || n_bits + n_params > kIn)
        return fail(HD_ERR_ARG, "hd_mlp_create: need 0 < n_bits and n_bits + n_params <= 64");
    if (n_states < 1 || n_states > 16) return fail(HD_ERR_ARG, "hd_mlp_create_states: 1 to 16 amplitudes");
    *out = nullptr;
    hd_mlp* m = new hd_mlp();
    m->n_bits = n_bits;
    m->n_params = n_params;
    m->n_states = n_states;
    m->live_rows[3] = 2 * n_states;
    if (stream_get(&m->stream) != hipSuccess) {
        delete m;
        return fail(HD_ERR_HIP, "stream creation failed");
    }
    std::mt19937_64 rng(seed);
    int st = HD_OK;
    HipErrors q;
    for (float** p : {&m->params, &m->grads, &m->mom1, &m->mom2})
        if (st == HD_OK) st = dalloc_t(p, (size_t)kParams, "MLP parameters");
    std::vector<float> flat(kParams, 0.f);
    for (int l = 0; l < 4 && st == HD_OK; ++l) {
        const int R = kRows[l], C = kCols[l];
        float* w = flat.data() + kOff[l];
        // He-normal over the live fan-in (n_bits + n_params for the first layer)
        const int fan_in = l == 0 ? n_bits + n_params : kW;
        std::normal_distribution<float> nd(0.f, std::sqrt(2.f / (float)fan_in) * (l == 3 ? 0.1f : 1.f));
        for (int r = 0; r < m->live_rows[l]; ++r)
            for (int c = 0; c < (l == 0 ? fan_in : C); ++c) w[(size_t)r * C + c] = nd(rng);
        if ((st = dalloc_t(&m->wb[l], (size_t)R * C, "MLP bf16 weights")) != HD_OK) break;
        if ((st = dalloc_t(&m->wbT[l], (size_t)R * C, "MLP bf16 weights^T")) != HD_OK) break;
    }
    if (st == HD_OK) {
        HD_ENQ(q, hipMemcpy(m->params, flat.data(), sizeof(float) * kParams, hipMemcpyHostToDevice));
        HD_ENQ(q, hipMemsetAsync(m->mom1, 0, sizeof(float) * kParams, m->stream));
        HD_ENQ(q, hipMemsetAsync(m->mom2, 0, sizeof(float) * kParams, m->stream));
    }
    if (st == HD_OK) st = q.status();
    if (st == HD_OK) st = dalloc_t(&m->wf, (size_t)kChunks * kChunk, "MLP packed weights");
    if (st == HD_OK && hipMemsetAsync(m->wf, 0, sizeof(__bf16) * kChunks * kChunk, m->stream) != hipSuccess)
        st = fail(HD_ERR_HIP, "MLP init failed");  // its last half chunk is padding
    if (st == HD_OK) st = mlp_refresh_bf16(m);
    if (st == HD_OK && hipStreamSynchronize(m->stream) != hipSuccess) st = fail(HD_ERR_HIP, "MLP init failed");
    if (st != HD_OK) {
        const std::string msg = hd_last_error();
        hd_mlp_destroy(m);
        set_error(msg);
        return st;
    }
    *out = m;
    return HD_OK;
}

int hd_mlp_destroy(hd_mlp* m)
{
    if (!m) return HD_OK;
    mlp_free_work(m);
    for (int l = 0; l < 4; ++l) {
        dfree(m->wb[l]);
        dfree(m->wbT[l]);
    }
    for (float* p : {m->params, m->grads, m->mom1, m->mom2}) dfree(p);
    dfree(m->st_buf); dfree(m->pr_buf); dfree(m->tg_buf); dfree(m->wf);
    if (m->stream) stream_put(m->stream);
    delete m;
    return HD_OK;
}

int hd_mlp_num_weights(const hd_mlp* m, int64_t* count)
{
    if (!m || !count) return fail(HD_ERR_ARG, "null argument");
    *count = kParams;
    return HD_OK;
}

// Flat FP32 layout: for each layer, W (rows x cols, padded shape) then b.
static int copy_to_host(hd_mlp* m, float* h, const float* d)
{
    HD_HIP(hipMemcpyAsync(h, d, sizeof(float) * kParams, hipMemcpyDeviceToHost, m->stream));
    HD_HIP(hipStreamSynchronize(m->stream));
    return HD_OK;
}

int hd_mlp_get_weights(hd_mlp* m, float* h_out)
{
    if (!m || !h_out) return fail(HD_ERR_ARG, "null argument");
    return copy_to_host(m, h_out, m->params);
}

int hd_mlp_set_weights(hd_mlp* m, const float* h_in)
{
    if (!m || !h_in) return fail(HD_ERR_ARG, "null argument");
    HD_HIP(hipMemcpyAsync(m->params, h_in, sizeof(float) * kParams, hipMemcpyHostToDevice, m->stream));
    HD_CHECK(mlp_refresh_bf16(m));
    HD_HIP(hipStreamSynchronize(m->stream));
    return HD_OK;
}

int hd_mlp_forward(hd_mlp* m, const uint64_t* h_states, const float* h_params, int64_t n, float* h_out)
{
    if (!m || !h_states || !h_params || !h_out || n <= 0) return fail(HD_ERR_ARG, "hd_mlp_forward: bad argument");
    const uint64_t* ds;
    const float *dp, *dt;
    HD_CHECK(stage_batch(m, h_states, h_params, nullptr, n, true, &ds, &dp, &dt, 1));
    int n_cu = 256;
    HD_CHECK(device_props(&n_cu, nullptr));
    const InferGrid grid = infer_grid(n, n_cu);
    const int64_t nblk = grid.blocks;
    float *dout = nullptr, *dmax = nullptr;
    const int S = m->n_states;
    HD_CHECK(dalloc_t(&dout, (size_t)n * 2 * S, "MLP outputs"));
    int st = dalloc_t(&dmax, (size_t)nblk * S, "MLP output maxima");
    if (st == HD_OK) {
        InferArgs a = infer_args(m, n, ds, dp, 1, dout, dmax);
        infer_launch(a, grid, m->stream);
        HipErrors q;
        HD_ENQ(q, hipGetLastError());
        HD_ENQ(q, hipMemcpyAsync(h_out, dout, sizeof(float) * 2 * S * n, hipMemcpyDeviceToHost, m->stream));
        HD_ENQ(q, hipStreamSynchronize(m->stream));
        st = q.status();
    }
    dfree(dout);
    dfree(dmax);
    return st;
}

int hd_mlp_gradients(hd_mlp* m, const uint64_t* h_states, const float* h_params, const float* h_targets, int64_t n,
                     float lambda, float* loss, float* h_grads)
{
    if (!m || !h_states || !h_params || !h_targets || n <= 0) return fail(HD_ERR_ARG, "hd_mlp_gradients: bad argument");
    int splits = 0;
    HD_CHECK(batch_pass(m, h_states, h_params, h_targets, n, lambda, 1, &splits));
    hipLaunchKernelGGL((k_params<true, false, false>), kParamGrid, dim3(256), 0, m->stream, param_args(m, splits));
    HD_HIP(hipGetLastError());
    HD_CHECK(mlp_loss(m, pad64(n), loss));
    if (h_grads) HD_CHECK(copy_to_host(m, h_grads, m->grads));
    return HD_OK;
}

int hd_mlp_train_step(hd_mlp* m, const uint64_t* d_states, const float* d_params, const float* d_targets, int64_t n,
                      float lambda, float lr, float* loss)
{
    if (!m || !d_states || !d_params || !d_targets || n <= 0) return fail(HD_ERR_ARG, "hd_mlp_train_step: bad argument");
    int splits = 0;
    HD_CHECK(batch_pass(m, d_states, d_params, d_targets, n, lambda, 0, &splits));
    m->step += 1;
    ParamArgs a = param_args(m, splits);
    a.lr = lr;
    a.b1 = 0.9f;
    a.b2 = 0.999f;
    a.c1 = 1.f - std::pow(a.b1, (float)m->step);
    a.c2 = 1.f - std::pow(a.b2, (float)m->step);
    a.eps = 1e-8f;
    hipLaunchKernelGGL((k_params<true, true, true>), kParamGrid, dim3(256), 0, m->stream, a);
    HD_HIP(hipGetLastError());
    return mlp_loss(m, pad64(n), loss);
}

int hd_mlp_start_vector(hd_mlp* m, const hd_basis* basis, const float* h_params, double* d_vec)
{
    if (!m || !basis || !h_params || !d_vec) return fail(HD_ERR_ARG, "hd_mlp_start_vector: bad argument");
    if (basis->Norb != m->n_bits) return fail(HD_ERR_ARG, "network input width differs from the orbital count");
    const int64_t n = basis->dim;
    if (n == 0) return HD_OK;
    const int S = m->n_states;
    int n_cu = 256;
    HD_CHECK(device_props(&n_cu, nullptr));
    const InferGrid grid = infer_grid(n, n_cu);
    const int64_t nblk = grid.blocks;
    const int nred = (int)std::min<int64_t>((n + 255) / 256, 1024);
    float *dpar = nullptr, *dout = nullptr, *dmax = nullptr;
    double* dnorm = nullptr;
    const int np = std::max(m->n_params, 1);
    int st = dalloc_t(&dpar, (size_t)np + S, "MLP parameters and shifts");
    if (st == HD_OK) st = dalloc_t(&dout, (size_t)n * 2 * S, "start vector outputs");
    if (st == HD_OK) st = dalloc_t(&dmax, (size_t)nblk * S, "start vector output maxima");
    if (st == HD_OK) st = dalloc_t(&dnorm, (size_t)(nred + 1) * S, "start vector norms");
    if (st == HD_OK) {
        // one pass of the fused network over the sector, then per amplitude the
        // largest log-amplitude (and, with several, the norm), then the sum
        HipErrors q;
        HD_ENQ(q, hipMemcpyAsync(dpar, h_params, sizeof(float) * m->n_params, hipMemcpyHostToDevice, m->stream));
        InferArgs a = infer_args(m, n, basis->d_states, dpar, 0, dout, dmax);
        infer_launch(a, grid, m->stream);
        HD_ENQ(q, hipGetLastError());
        float* shift = dpar + np;
        hipLaunchKernelGGL(k_max_states, dim3(S), dim3(256), 0, m->stream, nblk, S, dmax, shift);
        HD_ENQ(q, hipGetLastError());
        double* inv = dnorm + (size_t)nred * S;
        if (S > 1) {
            if (S <= 8)
                hipLaunchKernelGGL(k_norm2_states<8>, dim3(nred), dim3(256), 0, m->stream, n, S, dout, shift, dnorm);
            else
                hipLaunchKernelGGL(k_norm2_states<16>, dim3(nred), dim3(256), 0, m->stream, n, S, dout, shift, dnorm);
            hipLaunchKernelGGL(k_inv_norm_states, dim3(S), dim3(256), 0, m->stream, nred, S, dnorm, inv);
            HD_ENQ(q, hipGetLastError());
        }
        hipLaunchKernelGGL(k_amplitude, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, m->stream, n, S, dout, shift,
                           inv, d_vec);
        HD_ENQ(q, hipGetLastError());
        HD_ENQ(q, hipStreamSynchronize(m->stream));
        st = q.status();
    }
    dfree(dpar);
    dfree(dout);
    dfree(dmax);
    dfree(dnorm);
    return st;
}

int hd_mlp_num_states(const hd_mlp* m, int32_t* n_states)
{
    if (!m || !n_states) return fail(HD_ERR_ARG, "hd_mlp_num_states: null argument");
    *n_states = m->n_states;
    return HD_OK;
}

// Raw GEMM check: C (M x N, FP32) = A (M x K, BF16 bits) . B (N x K, BF16 bits)^T
// through the MFMA kernel; M, N multiples of 64, K of 16 (host buffers).
int hd_mlp_gemm_check(int32_t M, int32_t N, int32_t K, const uint16_t* h_a, const uint16_t* h_b, float* h_c)
{
    if (M <= 0 || N <= 0 || K <= 0 || M % 64 || N % 64 || K % 16 || !h_a || !h_b || !h_c)
        return fail(HD_ERR_ARG, "hd_mlp_gemm_check: M, N multiples of 64 and K of 16");
    __bf16 *a = nullptr, *b = nullptr;
    float* c = nullptr;
    HD_CHECK(dalloc_t(&a, (size_t)M * K, "gemm A"));
    int st = dalloc_t(&b, (size_t)N * K, "gemm B");
    if (st == HD_OK) st = dalloc_t(&c, (size_t)M * N, "gemm C");
    if (st == HD_OK) {
        HipErrors q;
        HD_ENQ(q, hipMemcpy(a, h_a, (size_t)M * K * 2, hipMemcpyHostToDevice));
        HD_ENQ(q, hipMemcpy(b, h_b, (size_t)N * K * 2, hipMemcpyHostToDevice));
        st = q.status();
    }
    if (st == HD_OK) {
        GemmArgs g = ga(M, N, K, a, K, b, K);
        g.C = c; g.ldc = N;
        gemm(0, EPI_STORE, g);
        if (hipGetLastError() != hipSuccess || hipMemcpy(h_c, c, (size_t)M * N * 4, hipMemcpyDeviceToHost) != hipSuccess)
            st = fail(HD_ERR_HIP, "gemm check failed");
    }
    dfree(a); dfree(b); dfree(c);
    return st;
}

}  // extern "C"
