// qs_learned.hip -- learned heavy-hitter routing in front of the MSWS sketch.
//
// No counterpart in the reference (it has no learned component).  The network
// is a 64 -> 64 -> 64 -> 1 MLP with ReLU on the 64 bits of a key, BF16 weights
// and activations, FP32 accumulation:
//   h1 = bf16(relu(W1 x + b1)),  h2 = bf16(relu(W2 h1 + b2)),  y = w3 . h2 + b3
// Training kernels (VALU, one unit per lane):
//   k_mlp_grad  forward + backward of a minibatch, each block's gradients in a row
//               of its own
//   k_grad_sum  sums the blocks' partial gradients; Adam on the FP32 master weights
//               and their BF16 copies
// Serving kernels:
//   k_mlp_mfma  the same forward on the matrix cores: a wavefront scores 32
//               keys with v_mfma_f32_32x32x8_bf16, computing H^T = W X^T so that
//               the accumulator layout of one layer is the B-operand layout of
//               the next (no transpose between layers)
//   k_route     k_mlp_mfma + routing: keys with score >= threshold and the others
//               are packed apart, chunk by chunk
//   k_heavy_*   the heavy keys counted in LDS tables, whose entries are added to
//               the exact GPU table; long calls group them by bin first
//   k_light_move  the light keys put together, in stream order: the sketch's input
//   k_reflag    after a routing pass the table could not hold: heavy keys
//               without a slot go to the sketch instead
//   k_table_query / k_learned_query  the query: the table count of a key
//               held in the table, else the sketch estimate (the second
//               kernel scores keys first and probes only heavy-scored ones)
#include "qs_internal.h"

#include "../../include/qsketch_learned.h"

#include <cmath>
#include <cstring>
#include <vector>

#define CK(x)                                                                                    \
    do {                                                                                         \
        hipError_t e__ = (x);                                                                    \
        if (e__ != hipSuccess)                                                                   \
            return QS_ERR_HIP;                                                                   \
    } while (0)

#define OFF_W1 0
#define OFF_B1 4096
#define OFF_W2 4160
#define OFF_B2 8256
#define OFF_W3 8320
#define OFF_B3 8384
#define NPAR QS_MLP_PARAMS

#define T_EMPTY 0xffffffffffffffffull
#define T_NONE 0xffffffffu
#define T_PROBES 4096u
// error bits of one insert call
#define LE_FULL 1u // the table turned a key away
#define LE_SORT 2u // the grouping computed a position outside the call

#define ROUTE_THREADS 1024
#define ROUTE_CHUNK 1024u // keys per chunk, a wavefront's unit of routing
#define HBINS 256u        // bins of heavy keys
#define LT_BUCKETS 1024u  // per-block LDS table of heavy keys: buckets of 4 slots (48 KB)
// Calls of at least this many keys group their heavy keys by bin before they
// are counted: one launch more, but fewer updates of the exact table (whole
// windows of 2^20 keys 302 us straight, 356 grouped; of 2^25 keys 1.9 and 1.46 ms;
// the lines meet near 2^21, where both take about 370 us).
#define HEAVY_PART_MIN (1u << 21)

struct qs_learned {
    qs_sketch *sk;
    uint32_t key_bytes;
    float *d_p;        // FP32 master parameters
    uint16_t *d_pb;    // BF16 copies
    float *d_m, *d_v;  // Adam moments
    float *d_part;     // partial gradients, a row per block of k_mlp_grad
    float *d_g;        // gradient of the last batch (the row after d_part's)
    float *d_loss;     // its loss (the element after the gradient)
    uint64_t step;
    float thr;
    uint32_t tlog2;
    uint64_t tcap;
    uint64_t *d_tkeys;
    uint32_t *d_tcnt;
    uint32_t *d_bins;  // heavy keys per bin and the bins' write cursors (both of one call)
    uint32_t *d_err;   // (after them) [0] error bits of one call (LE_*), [1] slots in use
    uint64_t inserted; // keys inserted since create / clear
    uint32_t full;     // the table has turned a key away since create / clear
    uint32_t used;     // table slots in use after the last insert
    // routing scratch
    uint64_t rcap;     // keys
    uint8_t *d_flag;   // 1 = goes to the sketch
    uint32_t *d_count; // light keys per chunk, scanned in place (+ total)
    uint32_t *d_bsum;  // block sums of that scan (+ total)
    void *d_stage;     // per chunk: its light keys, packed at the front
    void *d_light;     // the light keys of the call, in stream order
    uint32_t cus;      // routing blocks at most
    uint32_t *h_pin;   // pinned: light total, error flag, slots in use
};

// ---------------------------------------------------------------------------
// BF16 (round to nearest even) and key bits
// ---------------------------------------------------------------------------
__device__ static inline uint16_t f2bf(float f)
{
    // v_cvt_pk_bf16_f32: round to nearest even, as f2bf_host's bit arithmetic
    // for every finite value
    return __builtin_bit_cast(uint16_t, (__bf16)f);
}
__device__ static inline float bf2f(uint16_t h)
{
    return __uint_as_float((uint32_t)h << 16);
}
static inline uint16_t f2bf_host(float f)
{
    uint32_t u;
    memcpy(&u, &f, 4);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

// the key at i, or at n - 1 past the end (n > 0): loads that prefetch the next
// tile's keys stay unconditional, so the wait for this tile's keys does not also
// wait for them
template <int KB> __device__ static inline uint64_t key64(const KeyT<KB> *keys, uint64_t i);
template <int KB>
__device__ static inline uint64_t key_at(const KeyT<KB> *keys, uint64_t i, uint64_t n)
{
    return key64<KB>(keys, i < n ? i : n - 1u);
}

template <int KB>
__device__ static inline uint64_t key64(const KeyT<KB> *keys, uint64_t i)
{
    return (uint64_t)keys[i];
}

// ---------------------------------------------------------------------------
// training: forward + backward
//
// A block takes groups of GK keys in turn.  In the forward and the deltas a
// wavefront works on GK / 4 keys with one unit per lane (each unit's sum still
// runs over its inputs in order, so activations and deltas equal the per-key
// forward's bit for bit); the weights lie in LDS so that the lanes read
// neighbouring words, and a read serves the wavefront's keys.  The
// weight gradients are 64 x 64 outer-product sums over the group, GR elements of
// each per thread, kept in registers over all of the block's groups and
// written as the block's row of partial gradients (k_grad_sum adds the rows).  Bound by LDS reads (about five per 16
// FMAs); the first form had one key per lane, 64 keys per block and one
// wavefront per CU on a quarter of the chip: 356 us for 4096 keys, now 15.
// ---------------------------------------------------------------------------
#define GK 16u        // keys per group
#define GT 512u       // threads
#define GNW (GT / 64u) // wavefronts
#define GW (GK / GNW)  // keys per wavefront
#define GR (64u / GNW) // rows of a weight gradient per wavefront
static_assert(GR % 4u == 0 && GW * GNW == GK && 192u * GNW <= GK * 64u * 2u, "work per wavefront");
#define GRAD_BLOCKS 256u // one per CU: rows of partial gradients at most
#define PART_STRIDE 8448u // floats per row (parameters and loss, in whole 64s)
static_assert(PART_STRIDE > NPAR && PART_STRIDE % 64u == 0, "a row holds the gradients and the loss");
#define WT 66u        // row stride of a transposed weight matrix in LDS

// orders a wavefront's LDS writes before its later reads (the hardware keeps
// one wavefront's LDS accesses in order; this holds the compiler to it)
__device__ static inline void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ static inline float wave_sum(float v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        v += __shfl_xor(v, o, 64);
    return v;
}

template <int KB>
__global__ __launch_bounds__(GT) void k_mlp_grad(const KeyT<KB> *__restrict__ keys, const float *__restrict__ tgt,
                                                 uint32_t n, const uint16_t *__restrict__ pb,
                                                 const float *__restrict__ p, float inv_n,
                                                 float *__restrict__ part)
{
    __shared__ uint16_t sW1t[64 * WT], sW2t[64 * WT]; // [input][unit]
    __shared__ uint16_t sW2[64 * 64];                 // [unit][input]
    __shared__ float4 srows[3][GK][16]; // per key: h1, and the deltas of layers 2 and 1
    float4(*const sh1)[16] = srows[0], (*const sd2)[16] = srows[1], (*const sd1)[16] = srows[2];
    __shared__ unsigned long long sx[GK];
    const uint32_t t = threadIdx.x, lane = t & 63u, wv = t >> 6;
    for (uint32_t e = t; e < 2048u; e += GT) { // two weights of row j at a time
        const uint32_t j = e >> 5, k = 2u * (e & 31u);
        const uint32_t a = reinterpret_cast<const uint32_t *>(pb + OFF_W1)[e];
        const uint32_t b = reinterpret_cast<const uint32_t *>(pb + OFF_W2)[e];
        sW1t[k * WT + j] = (uint16_t)a;
        sW1t[(k + 1u) * WT + j] = (uint16_t)(a >> 16);
        sW2t[k * WT + j] = (uint16_t)b;
        sW2t[(k + 1u) * WT + j] = (uint16_t)(b >> 16);
        reinterpret_cast<uint32_t *>(sW2)[e] = b;
    }
    const float b1 = p[OFF_B1 + lane], b2 = p[OFF_B2 + lane], w3 = bf2f(pb[OFF_W3 + lane]), b3 = p[OFF_B3];
    // gradient sums of this thread: W2 and W1 elements (row GR wv + i, column
    // lane), and this wavefront's part of unit lane's b1, b2, w3
    float a2[GR], a1[GR], gb1 = 0.f, gb2 = 0.f, gw3 = 0.f, gb3 = 0.f, l = 0.f;
#pragma unroll
    for (uint32_t i = 0; i < GR; ++i)
        a2[i] = a1[i] = 0.f;
    __syncthreads();
    for (uint64_t g0 = (uint64_t)blockIdx.x * GK; g0 < n; g0 += (uint64_t)gridDim.x * GK) {
        uint64_t x[GW];
        float z[GW], h1[GW];
        bool m1[GW];
#pragma unroll
        for (uint32_t q = 0; q < GW; ++q) {
            const uint64_t i = g0 + wv * GW + q;
            const uint64_t xv = i < n ? key64<KB>(keys, i) : 0ull; // one address per wavefront:
            x[q] = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)xv) | // in scalar registers
                   (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(xv >> 32)) << 32;
            if (lane == 0)
                sx[wv * GW + q] = x[q];
            z[q] = b1;
        }
#pragma unroll 8
        for (uint32_t k = 0; k < 64u; ++k) {
            const float w = bf2f(sW1t[k * WT + lane]);
#pragma unroll
            for (uint32_t q = 0; q < GW; ++q)
                z[q] += ((x[q] >> k) & 1ull) ? w : 0.f;
        }
#pragma unroll
        for (uint32_t q = 0; q < GW; ++q) {
            m1[q] = z[q] > 0.f;
            h1[q] = bf2f(f2bf(fmaxf(z[q], 0.f)));
            reinterpret_cast<float *>(sh1[wv * GW + q])[lane] = h1[q];
            z[q] = b2;
        }
        wave_lds_fence(); // a wavefront reads back its own rows only
#pragma unroll 4
        for (uint32_t k4 = 0; k4 < 16u; ++k4) {
            float4 h[GW];
#pragma unroll
            for (uint32_t q = 0; q < GW; ++q)
                h[q] = sh1[wv * GW + q][k4];
#pragma unroll
            for (uint32_t e = 0; e < 4u; ++e) {
                const float w = bf2f(sW2t[(4u * k4 + e) * WT + lane]);
#pragma unroll
                for (uint32_t q = 0; q < GW; ++q)
                    z[q] = fmaf(w, e == 0 ? h[q].x : e == 1 ? h[q].y : e == 2 ? h[q].z : h[q].w, z[q]);
            }
        }
        float d1[GW];
#pragma unroll
        for (uint32_t q = 0; q < GW; ++q) {
            const uint64_t i = g0 + wv * GW + q;
            const float h2 = bf2f(f2bf(fmaxf(z[q], 0.f)));
            const float y = wave_sum(w3 * h2) + b3;
            const float diff = i < n ? y - tgt[i] : 0.f;
            const float dy = diff * inv_n;
            const float d2 = z[q] > 0.f ? dy * w3 : 0.f;
            l += 0.5f * diff * diff * inv_n;
            gw3 = fmaf(dy, h2, gw3);
            gb3 += dy;
            gb2 += d2;
            reinterpret_cast<float *>(sd2[wv * GW + q])[lane] = d2;
            d1[q] = 0.f;
        }
        wave_lds_fence();
#pragma unroll 4
        for (uint32_t j4 = 0; j4 < 16u; ++j4) {
            float4 d[GW];
#pragma unroll
            for (uint32_t q = 0; q < GW; ++q)
                d[q] = sd2[wv * GW + q][j4];
#pragma unroll
            for (uint32_t e = 0; e < 4u; ++e) {
                const float w = bf2f(sW2[(4u * j4 + e) * 64u + lane]);
#pragma unroll
                for (uint32_t q = 0; q < GW; ++q)
                    d1[q] = fmaf(w, e == 0 ? d[q].x : e == 1 ? d[q].y : e == 2 ? d[q].z : d[q].w, d1[q]);
            }
        }
#pragma unroll
        for (uint32_t q = 0; q < GW; ++q) {
            const float d = m1[q] ? d1[q] : 0.f;
            gb1 += d;
            reinterpret_cast<float *>(sd1[wv * GW + q])[lane] = d;
        }
        __syncthreads(); // every wavefront's keys
        for (uint32_t s = 0; s < GK; ++s) {
            const float h = reinterpret_cast<const float *>(sh1[s])[lane];
            const bool on = (sx[s] >> lane) & 1ull;
#pragma unroll
            for (uint32_t c = 0; c < GR / 4u; ++c) {
                const float4 u = sd2[s][GR / 4u * wv + c], v = sd1[s][GR / 4u * wv + c];
                a2[4 * c + 0] = fmaf(u.x, h, a2[4 * c + 0]);
                a2[4 * c + 1] = fmaf(u.y, h, a2[4 * c + 1]);
                a2[4 * c + 2] = fmaf(u.z, h, a2[4 * c + 2]);
                a2[4 * c + 3] = fmaf(u.w, h, a2[4 * c + 3]);
                a1[4 * c + 0] += on ? v.x : 0.f;
                a1[4 * c + 1] += on ? v.y : 0.f;
                a1[4 * c + 2] += on ? v.z : 0.f;
                a1[4 * c + 3] += on ? v.w : 0.f;
            }
        }
        __syncthreads(); // the next group rewrites the rows
    }
    // this block's row of partial gradients, with its loss in the element after
    // them; the wavefronts' unit sums meet in LDS (the rows are free now)
    float *const red = reinterpret_cast<float *>(srows), *const row = part + (size_t)blockIdx.x * PART_STRIDE;
    red[wv * 192u + lane] = gb1;
    red[wv * 192u + 64u + lane] = gb2;
    red[wv * 192u + 128u + lane] = gw3;
    float *const red2 = reinterpret_cast<float *>(sd1);
    if (lane == 0) {
        red2[2u * wv] = gb3;
        red2[2u * wv + 1u] = l;
    }
#pragma unroll
    for (uint32_t i = 0; i < GR; ++i) {
        row[OFF_W2 + (GR * wv + i) * 64u + lane] = a2[i];
        row[OFF_W1 + (GR * wv + i) * 64u + lane] = a1[i];
    }
    __syncthreads();
    if (t < 194u) {
        float v = 0.f;
#pragma unroll
        for (uint32_t w = 0; w < GNW; ++w)
            v += t < 192u ? red[w * 192u + t] : red2[2u * w + (t - 192u)];
        row[t < 64u ? OFF_B1 + t : t < 128u ? OFF_B2 + t - 64u : t < 192u ? OFF_W3 + t - 128u : t == 192u ? OFF_B3 : NPAR] = v;
    }
}

// The blocks' partial gradients summed (64 elements per block, 16 wavefronts a
// share of the rows each), left in g with the loss after them; with `update`,
// Adam on the master weights and their BF16 copies follows.  (Adding the
// partials with atomics to one gradient took 40 of a step's 49 us.)
#define SUM_WAVES 16u
__global__ __launch_bounds__(64 * SUM_WAVES) void k_grad_sum(const float *__restrict__ part, uint32_t nrows,
                                                             float *__restrict__ g, bool update,
                                                             float *__restrict__ p, uint16_t *__restrict__ pb,
                                                             float *__restrict__ m, float *__restrict__ v, float lr,
                                                             float b1, float b2, float eps, float c1, float c2)
{
    __shared__ float s[SUM_WAVES][64];
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    const uint32_t e = blockIdx.x * 64u + lane; // < PART_STRIDE
    float x = 0.f;
#pragma unroll 8
    for (uint32_t r = wv; r < nrows; r += SUM_WAVES)
        x += part[(size_t)r * PART_STRIDE + e];
    s[wv][lane] = x;
    __syncthreads();
    if (wv != 0 || e > NPAR)
        return;
    float gr = 0.f;
#pragma unroll
    for (uint32_t w = 0; w < SUM_WAVES; ++w)
        gr += s[w][lane];
    g[e] = gr;
    if (!update || e == NPAR)
        return;
    const float mm = b1 * m[e] + (1.f - b1) * gr;
    const float vv = b2 * v[e] + (1.f - b2) * gr * gr;
    m[e] = mm;
    v[e] = vv;
    const float pp = p[e] - lr * (mm / c1) / (sqrtf(vv / c2) + eps);
    p[e] = pp;
    pb[e] = f2bf(pp);
}

// new parameters: their BF16 copies, and moments that start over
__global__ void k_set_params(const float *__restrict__ p, uint16_t *__restrict__ pb, float *__restrict__ m,
                             float *__restrict__ v)
{
    for (uint32_t e = blockIdx.x * blockDim.x + threadIdx.x; e < NPAR; e += gridDim.x * blockDim.x) {
        m[e] = v[e] = 0.f;
        pb[e] = f2bf(p[e]);
    }
}

// per-key VALU forward (the training forward)
template <int KB>
__global__ __launch_bounds__(256) void k_mlp_fwd(const KeyT<KB> *__restrict__ keys, uint64_t n,
                                                 const uint16_t *__restrict__ pb, const float *__restrict__ p,
                                                 float *__restrict__ out)
{
    __shared__ uint16_t sW1[64 * 64], sW2[64 * 64];
    __shared__ float sb1[64], sb2[64], sw3[64];
    for (uint32_t e = threadIdx.x; e < 4096u; e += 256u) {
        sW1[e] = pb[OFF_W1 + e];
        sW2[e] = pb[OFF_W2 + e];
    }
    if (threadIdx.x < 64) {
        sb1[threadIdx.x] = p[OFF_B1 + threadIdx.x];
        sb2[threadIdx.x] = p[OFF_B2 + threadIdx.x];
        sw3[threadIdx.x] = bf2f(pb[OFF_W3 + threadIdx.x]);
    }
    __syncthreads();
    const float b3 = p[OFF_B3];
    for (uint64_t i = (uint64_t)blockIdx.x * 256u + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256u) {
        const uint64_t x = key64<KB>(keys, i);
        float h1[64];
#pragma unroll
        for (int j = 0; j < 64; ++j) {
            float acc = sb1[j];
            for (int k = 0; k < 64; ++k)
                acc += ((x >> k) & 1ull) ? bf2f(sW1[j * 64 + k]) : 0.f;
            h1[j] = bf2f(f2bf(fmaxf(acc, 0.f)));
        }
        float y = b3;
        for (int j = 0; j < 64; ++j) {
            float acc = sb2[j];
#pragma unroll
            for (int k = 0; k < 64; ++k)
                acc = fmaf(bf2f(sW2[j * 64 + k]), h1[k], acc);
            y = fmaf(sw3[j], bf2f(f2bf(fmaxf(acc, 0.f))), y);
        }
        out[i] = y;
    }
}

// ---------------------------------------------------------------------------
// matrix-core forward.  v_mfma_f32_32x32x16_bf16 (8 BF16 per lane, gfx950):
//   A (32 x 16):  lane l holds A[l % 32][8 (l / 32) + i],   i = 0..7
//   B (16 x 32):  lane l holds B[8 (l / 32) + i][l % 32]
//   D (32 x 32):  lane l, register r holds D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32]
// Layer 1 computes H1^T (64 units x 32 keys) = W1 X^T as 2 row tiles x 4 K
// steps; lane l's key is key l % 32, and K step s, half h = l / 32 is key byte
// 2 s + h.  Layer 2 sums over the units in the order the accumulators hold
// them: K step s takes registers 8 (s % 2) .. 8 (s % 2) + 7 of row tile s / 2,
// so slot i of half h is unit 32 (s / 2) + 8 (2 (s % 2) + i / 4) + 4 h + i % 4
// (every unit once), and W2's columns are laid out in that order.  The output
// layer is one more row tile in the same K order: W3 is its row 0 (the other
// rows are zero), so the score of key l is register 0 of lane l < 32.
// ---------------------------------------------------------------------------
typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef short bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16v8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// The whole network lives in LDS: the weight operands in MFMA A-operand order
// (layer, row tile, K step, lane -> 8 BF16), so each MFMA reads its operand
// with one 16-byte LDS load, plus the biases and output weights.  Registers
// then hold only accumulators and activations, for several waves per SIMD.
struct mlp_lds {
    bf16x8 a[2][2][4][64];
    bf16x8 a3[4][64]; // output layer: W3 in row 0 of the A operand, other rows 0
    bf16x4 nib[16];   // layer-1 B operand of a key nibble: bit i -> 1.0 or 0.0 in BF16
    float b1[64], b2[64], b3;
};

// BF16(max(lo, 0)), BF16(max(hi, 0)) packed: one conversion of the pair, then
// max(., 0) on the two 16-bit halves (rounding keeps the sign, and negative
// BF16 values and -0 are negative 16-bit integers: the same bits as rounding
// max(x, 0))
typedef short s16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2v __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
__device__ static inline uint32_t relu_bf16x2(float lo, float hi)
{
    const bf16x2v b = __builtin_convertvector((f32x2v){lo, hi}, bf16x2v); // v_cvt_pk_bf16_f32
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(s16x2, b), (s16x2)0));
}

// a layer's activations as the next layer's B operands: K step s takes
// registers 8 (s % 2) .. 8 (s % 2) + 7 of row tile s / 2
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
__device__ static inline void acts_to_b(const float *acc0, const float *acc1, bf16x8 hb[4])
{
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const float *a = s < 2 ? acc0 : acc1;
        u32x4v w;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int r = 8 * (s % 2) + 2 * p;
            w[p] = relu_bf16x2(a[r], a[r + 1]);
        }
        hb[s] = __builtin_bit_cast(bf16x8, w);
    }
}

// input column of K slot i, half h, K step s of layer 0 / 1
__device__ static inline uint32_t kcol(uint32_t layer, uint32_t s, uint32_t h, uint32_t i)
{
    return layer == 0 ? 16u * s + 8u * h + i : 32u * (s / 2u) + 8u * (2u * (s % 2u) + i / 4u) + 4u * h + i % 4u;
}

__device__ static inline void load_mlp(mlp_lds &S, const uint16_t *__restrict__ pb, const float *__restrict__ p)
{
    for (uint32_t e = threadIdx.x; e < 2u * 2u * 4u * 64u; e += blockDim.x) {
        const uint32_t l = e & 63u, s = (e >> 6) & 3u, t = (e >> 8) & 1u, layer = e >> 9;
        const uint32_t h = l >> 5, c = l & 31u;
        const uint16_t *w = pb + (layer ? OFF_W2 : OFF_W1) + (32u * t + c) * 64u;
        bf16x8 v;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            v[i] = (short)w[kcol(layer, s, h, (uint32_t)i)];
        S.a[layer][t][s][l] = v;
    }
    for (uint32_t e = threadIdx.x; e < 4u * 64u; e += blockDim.x) {
        const uint32_t l = e & 63u, s = e >> 6, h = l >> 5, c = l & 31u;
        bf16x8 v;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            v[i] = c == 0 ? (short)pb[OFF_W3 + kcol(1, s, h, (uint32_t)i)] : (short)0;
        S.a3[s][l] = v;
    }
    for (uint32_t e = threadIdx.x; e < 16u; e += blockDim.x) {
        bf16x4 v;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            v[i] = ((e >> i) & 1u) ? (short)0x3f80 : (short)0;
        S.nib[e] = v;
    }
    for (uint32_t e = threadIdx.x; e < 64u; e += blockDim.x) {
        S.b1[e] = p[OFF_B1 + e];
        S.b2[e] = p[OFF_B2 + e];
    }
    if (threadIdx.x == 0)
        S.b3 = p[OFF_B3];
    __syncthreads();
}

// D row held by register r of row tile t in this lane
__device__ static inline uint32_t drow(int t, int r, uint32_t h)
{
    return 32u * t + 8u * (r / 4) + 4u * h + (r % 4);
}

__device__ static inline f32x16 mfma16(const bf16x8 &a, const bf16x8 &b, const f32x16 &c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16v8, a), __builtin_bit_cast(bf16v8, b), c,
                                                   0, 0, 0);
}

// score of key x: lane l < 32 returns the score of its key (lanes 32..63
// return another value of the output tile)
__device__ static inline float mlp_mfma(const mlp_lds &S, uint64_t x)
{
    const uint32_t lane = threadIdx.x & 63u, h = lane >> 5;
    // reload the network from LDS for every key tile instead of letting the
    // compiler hoist it into (occupancy-limiting) registers
    asm volatile("" ::: "memory");
    f32x16 acc0, acc1;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        acc0[r] = S.b1[drow(0, r, h)];
        acc1[r] = S.b1[drow(1, r, h)];
    }
    const uint64_t xs = x >> (8u * h); // this half-wave's bytes: byte 2 s + h at bits 16 s
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const uint32_t byte = (uint32_t)(xs >> (16 * s)) & 0xffu;
        const bf16x4 lo = S.nib[byte & 0xfu], hi = S.nib[byte >> 4];
        const bf16x8 b = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        acc0 = mfma16(S.a[0][0][s][lane], b, acc0);
        acc1 = mfma16(S.a[0][1][s][lane], b, acc1);
    }
    bf16x8 hb[4];
    {
        float a0[16], a1[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            a0[r] = acc0[r];
            a1[r] = acc1[r];
        }
        acts_to_b(a0, a1, hb);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        acc0[r] = S.b2[drow(0, r, h)];
        acc1[r] = S.b2[drow(1, r, h)];
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        acc0 = mfma16(S.a[1][0][s][lane], hb[s], acc0);
        acc1 = mfma16(S.a[1][1][s][lane], hb[s], acc1);
    }
    {
        float a0[16], a1[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            a0[r] = acc0[r];
            a1[r] = acc1[r];
        }
        acts_to_b(a0, a1, hb);
    }
    f32x16 acc3 = {};
#pragma unroll
    for (int s = 0; s < 4; ++s)
        acc3 = mfma16(S.a3[s][lane], hb[s], acc3);
    return acc3[0] + S.b3;
}

// the key that lane src of the wavefront holds
__device__ static inline uint64_t lane_key(uint64_t x, uint32_t src)
{
    return (uint64_t)(uint32_t)__shfl((int)(uint32_t)x, (int)src, 64) |
           (uint64_t)(uint32_t)__shfl((int)(uint32_t)(x >> 32), (int)src, 64) << 32;
}

template <int KB>
__global__ __launch_bounds__(256) void k_mlp_mfma(const KeyT<KB> *__restrict__ keys, uint64_t n,
                                                  const uint16_t *__restrict__ pb, const float *__restrict__ p,
                                                  float *__restrict__ out)
{
    __shared__ mlp_lds S;
    load_mlp(S, pb, p);
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t gw = ((uint64_t)blockIdx.x * 256u + threadIdx.x) >> 6;
    const uint64_t nw = ((uint64_t)gridDim.x * 256u) >> 6;
    if (n == 0)
        return;
    uint64_t i = gw * 32u + (lane & 31u);
    uint64_t x = key_at<KB>(keys, i, n);
    for (uint64_t base = gw * 32u; base < n; base += nw * 32u) {
        // the next key is loaded while this one is scored
        const uint64_t i2 = i + nw * 32u;
        const uint64_t x2 = key_at<KB>(keys, i2, n);
        const float y = mlp_mfma(S, x);
        if (i < n && lane < 32u)
            out[i] = y;
        i = i2;
        x = x2;
    }
}

// ---------------------------------------------------------------------------
// exact table: open addressing with linear probing, u64 keys (all-ones =
// empty; that key value is never routed to the table), u32 counts
// ---------------------------------------------------------------------------
__device__ static inline uint32_t t_home(uint64_t key, uint32_t tlog2)
{
    return (uint32_t)((key * 0x9E3779B97F4A7C15ull) >> (64u - tlog2));
}

// slot of key, claiming a free one if it is absent (claims counts them)
__device__ static inline uint32_t t_insert(uint64_t *tkeys, uint32_t tlog2, uint64_t key, uint32_t &claims)
{
    const uint32_t mask = (1u << tlog2) - 1u;
    uint32_t s = t_home(key, tlog2);
    for (uint32_t pr = 0; pr < T_PROBES; ++pr, s = (s + 1u) & mask) {
        uint64_t cur = __hip_atomic_load(tkeys + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (cur == key)
            return s;
        if (cur == T_EMPTY) {
            unsigned long long prev =
                atomicCAS((unsigned long long *)(tkeys + s), (unsigned long long)T_EMPTY, (unsigned long long)key);
            claims += prev == T_EMPTY ? 1u : 0u;
            if (prev == T_EMPTY || prev == key)
                return s;
        }
    }
    return T_NONE;
}

__device__ static inline uint32_t t_find(const uint64_t *tkeys, uint32_t tlog2, uint64_t key)
{
    const uint32_t mask = (1u << tlog2) - 1u;
    uint32_t s = t_home(key, tlog2);
    for (uint32_t pr = 0; pr < T_PROBES; ++pr, s = (s + 1u) & mask) {
        const uint64_t cur = tkeys[s];
        if (cur == key)
            return s;
        if (cur == T_EMPTY)
            return T_NONE;
    }
    return T_NONE;
}

// err[0] gets LE_FULL when the table has no slot for key
__device__ static inline void t_add(uint64_t *tkeys, uint32_t *tcnt, uint32_t tlog2, uint64_t key, uint32_t c,
                                    uint32_t *err, uint32_t &claims)
{
    const uint32_t s = t_insert(tkeys, tlog2, key, claims);
    if (s == T_NONE)
        atomicOr(err, LE_FULL);
    else
        atomicAdd(tcnt + s, c);
}

// the bin of a heavy key
__device__ static inline uint32_t heavy_bin(uint64_t x)
{
    return (uint32_t)((x * 0x9E3779B97F4A7C15ull) >> 56);
}

// Routing.  A wavefront owns chunks of ROUTE_CHUNK consecutive keys and takes 64
// at a time: two matrix-core tiles score them, then every lane places one key:
// light keys, in stream order, at the front of the chunk's own slots of
// `stage`, heavy ones at the back (from the end), the light ones' number in
// `ccount` and the heavy ones' per bin in `bins`.  The heavy keys are counted by
// the kernels below; k_light_move puts the light ones together after a scan.
// The chunks of a short call go to different CUs.  Counting in this kernel held
// every wavefront to its slowest lane's probes between two scorings: 1.24 ms for
// 2^25 keys, now 0.60 and 0.23 for the counting; the forward alone takes 0.55.
template <int KB>
__global__ __launch_bounds__(ROUTE_THREADS) void k_route(const KeyT<KB> *__restrict__ keys, uint64_t n,
                                                         uint32_t nchunks, const uint16_t *__restrict__ pb,
                                                         const float *__restrict__ p, float thr,
                                                         uint8_t *__restrict__ flag, KeyT<KB> *__restrict__ stage,
                                                         uint32_t *__restrict__ ccount, uint32_t *__restrict__ bins)
{
    __shared__ mlp_lds S;
    __shared__ uint32_t s_bin[HBINS]; // heavy keys per bin
    for (uint32_t e = threadIdx.x; e < HBINS; e += ROUTE_THREADS)
        s_bin[e] = 0;
    load_mlp(S, pb, p); // ends with a barrier
    const uint32_t lane = threadIdx.x & 63u, l32 = lane & 31u;
    const uint64_t below = (1ull << lane) - 1ull;
    const uint32_t nw = gridDim.x * (ROUTE_THREADS / 64u);
    uint32_t c = (threadIdx.x >> 6) * gridDim.x + blockIdx.x;
    uint64_t xn = key_at<KB>(keys, (uint64_t)c * ROUTE_CHUNK + lane, n);
    for (; c < nchunks; c += nw) {
        const uint64_t base = (uint64_t)c * ROUTE_CHUNK;
        uint32_t light = 0;
        for (uint32_t st = 0; st < ROUTE_CHUNK / 64u; ++st) {
            const uint64_t i = base + st * 64u + lane;
            if (base + st * 64u >= n) // uniform
                break;
            const bool valid = i < n;
            const uint64_t x = xn;
            // the next keys are loaded while these are scored
            xn = key_at<KB>(keys, st + 1u < ROUTE_CHUNK / 64u ? i + 64u : base + (uint64_t)nw * ROUTE_CHUNK + lane, n);
            const float ya = mlp_mfma(S, lane_key(x, l32));
            const float yb = mlp_mfma(S, lane_key(x, 32u + l32));
            const float y2 = __shfl(yb, (int)l32, 64);
            const float y = lane < 32u ? ya : y2;
            const bool heavy = y >= thr && x != T_EMPTY;
            const uint64_t m = __ballot(valid && !heavy); // the whole wavefront, outside any branch
            const uint32_t before = light + (uint32_t)__popcll(m & below); // light keys before this one
            if (valid) {
                flag[i] = heavy ? 0 : 1;
                stage[base + (heavy ? ROUTE_CHUNK - 1u - (st * 64u + lane - before) : before)] = (KeyT<KB>)x;
                if (heavy)
                    atomicAdd(&s_bin[heavy_bin(x)], 1u);
            }
            light += (uint32_t)__popcll(m);
        }
        if (lane == 0)
            ccount[c] = light;
    }
    __syncthreads();
    for (uint32_t e = threadIdx.x; e < HBINS; e += ROUTE_THREADS)
        if (s_bin[e])
            atomicAdd(bins + e, s_bin[e]);
}

// The block's LDS table of heavy keys: LT_BUCKETS buckets of 4 slots, a key in
// the one bucket its hash names (two 16-byte reads and no loop but for a lost
// race); a key whose bucket is full goes to the exact table directly.
struct heavy_lds {
    ulonglong2 key2[LT_BUCKETS * 2u];
    uint32_t cnt[LT_BUCKETS * 4u];
};

__device__ static inline void heavy_clear(heavy_lds &T)
{
    unsigned long long *key = reinterpret_cast<unsigned long long *>(T.key2);
    for (uint32_t e = threadIdx.x; e < LT_BUCKETS * 4u; e += blockDim.x) {
        key[e] = T_EMPTY;
        T.cnt[e] = 0;
    }
    __syncthreads();
}

// one insert of x by every lane with `act` (the whole wavefront calls it)
__device__ static inline void heavy_add(heavy_lds &T, bool act, unsigned long long x, uint64_t *tkeys, uint32_t *tcnt,
                                        uint32_t tlog2, uint32_t *err, uint32_t &claims)
{
    // The lanes that hold the same key as the first lane, and then as the first
    // of the others, are counted by one of them: a hot key would serialise
    // its lanes on one LDS counter.
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t w = act ? 1u : 0u;
    uint64_t left = __ballot(act);
#pragma unroll
    for (int peel = 0; peel < 2; ++peel) {
        if (left == 0)
            break;
        const uint32_t first = (uint32_t)__builtin_ctzll(left);
        const uint64_t same = __ballot(w == 1u && x == lane_key(x, first)) & left;
        left &= ~same;
        if ((same >> lane) & 1ull)
            w = lane == first ? (uint32_t)__popcll(same) : 0u;
    }
    if (w == 0)
        return;
    const uint32_t b = (uint32_t)((x * 0x9E3779B97F4A7C15ull) >> 32) & (LT_BUCKETS - 1u); // (not the bin's bits)
    unsigned long long *key = reinterpret_cast<unsigned long long *>(T.key2) + 4u * b;
    int sl = -1;
    for (int tries = 0; tries < 4; ++tries) { // again only when another lane took the free slot
        const ulonglong2 p = T.key2[2u * b], q = T.key2[2u * b + 1u];
        const unsigned long long v[4] = {p.x, p.y, q.x, q.y};
        int fr = -1;
#pragma unroll
        for (int e = 3; e >= 0; --e) {
            sl = v[e] == x ? e : sl;
            fr = v[e] == T_EMPTY ? e : fr;
        }
        if (sl >= 0 || fr < 0)
            break;
        const unsigned long long old = atomicCAS(key + fr, (unsigned long long)T_EMPTY, x);
        if (old == T_EMPTY || old == x) {
            sl = fr;
            break;
        }
    }
    if (sl >= 0)
        atomicAdd(&T.cnt[4u * b + sl], w);
    else
        t_add(tkeys, tcnt, tlog2, x, w, err, claims);
}

// The table's entries to the exact table; the slots the block claimed there
// (also while counting) are added to err[1] at once (an atomic per claim on
// that one word serialised: 0.24 ms for 1.1e5 keys).
__device__ static inline void heavy_flush(heavy_lds &T, uint64_t *tkeys, uint32_t *tcnt, uint32_t tlog2, uint32_t *err,
                                          uint32_t claims)
{
    __syncthreads();
    const unsigned long long *key = reinterpret_cast<const unsigned long long *>(T.key2);
    for (uint32_t e = threadIdx.x; e < LT_BUCKETS * 4u; e += blockDim.x)
        if (T.cnt[e])
            t_add(tkeys, tcnt, tlog2, key[e], T.cnt[e], err, claims);
    __syncthreads();
    uint32_t *total = T.cnt; // free now
    if (threadIdx.x == 0)
        *total = 0;
    __syncthreads();
    if (claims)
        atomicAdd(total, claims);
    __syncthreads();
    if (threadIdx.x == 0 && *total)
        atomicAdd(err + 1, *total);
}

// the heavy keys of chunk c, rows of 64 (0 past their number, returned)
template <int KB>
__device__ static inline uint32_t load_heavy(const KeyT<KB> *__restrict__ stage, uint64_t n, uint32_t c,
                                             uint32_t nchunks, const uint32_t *__restrict__ ccount,
                                             KeyT<KB> k[ROUTE_CHUNK / 64u])
{
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t heavy = 0;
    const uint64_t base = (uint64_t)c * ROUTE_CHUNK;
    if (c < nchunks)
        heavy = (n - base < ROUTE_CHUNK ? (uint32_t)(n - base) : ROUTE_CHUNK) - ccount[c];
    const KeyT<KB> *src = stage + base + ROUTE_CHUNK - heavy;
#pragma unroll
    for (uint32_t r = 0; r < ROUTE_CHUNK / 64u; ++r)
        k[r] = r * 64u + lane < heavy ? __builtin_nontemporal_load(src + r * 64u + lane) : (KeyT<KB>)0;
    return heavy;
}

// Heavy keys counted straight from the chunks (short calls): every block meets
// every key, so each key costs an update of the exact table per block.
template <int KB>
__global__ __launch_bounds__(256) void k_heavy_count(const KeyT<KB> *__restrict__ stage, uint64_t n, uint32_t nchunks,
                                                     const uint32_t *__restrict__ ccount,
                                                     uint64_t *__restrict__ tkeys, uint32_t *__restrict__ tcnt,
                                                     uint32_t tlog2, uint32_t *__restrict__ err)
{
    __shared__ heavy_lds T;
    heavy_clear(T);
    uint32_t claims = 0;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t nw = gridDim.x * 4u;
    for (uint32_t c = blockIdx.x * 4u + (threadIdx.x >> 6); c < nchunks; c += nw) {
        KeyT<KB> k[ROUTE_CHUNK / 64u];
        const uint32_t heavy = load_heavy<KB>(stage, n, c, nchunks, ccount, k);
#pragma unroll
        for (uint32_t r = 0; r < ROUTE_CHUNK / 64u; ++r)
            if (r * 64u < heavy) // uniform
                heavy_add(T, r * 64u + lane < heavy, (unsigned long long)k[r], tkeys, tcnt, tlog2, err,
                          claims);
    }
    heavy_flush(T, tkeys, tcnt, tlog2, err, claims);
}

// Long calls group the heavy keys by bin first (any order within a bin), so
// that a key's inserts meet in the LDS tables of few blocks: updates of the exact
// table (about 5 M of them, 0.89 ms at 2^25 keys, when every block counted
// whatever came) then number little more than its keys.
// A block takes 8 chunks, one per wavefront, ranks their heavy keys per bin in
// LDS, reserves each bin's run with one atomic, and writes the runs in order.
#define HP_WAVES 8u
template <int KB>
__global__ __launch_bounds__(64 * HP_WAVES) void k_heavy_part(const KeyT<KB> *__restrict__ stage, uint64_t n,
                                                              uint32_t nchunks, const uint32_t *__restrict__ ccount,
                                                              const uint32_t *__restrict__ bins,
                                                              uint32_t *__restrict__ cursor,
                                                              KeyT<KB> *__restrict__ out, uint32_t *__restrict__ err)
{
    __shared__ KeyT<KB> s_key[HP_WAVES * ROUTE_CHUNK];
    __shared__ uint32_t s_cnt[HBINS], s_start[HBINS], s_goff[HBINS], s_red[2][4];
    const uint32_t t = threadIdx.x, lane = t & 63u, wv = t >> 6;
    if (t < HBINS)
        s_cnt[t] = 0;
    __syncthreads();
    KeyT<KB> k[ROUTE_CHUNK / 64u];
    uint32_t rank[ROUTE_CHUNK / 64u];
    const uint32_t heavy = load_heavy<KB>(stage, n, blockIdx.x * HP_WAVES + wv, nchunks, ccount, k);
#pragma unroll
    for (uint32_t r = 0; r < ROUTE_CHUNK / 64u; ++r)
        rank[r] = r * 64u + lane < heavy ? atomicAdd(&s_cnt[heavy_bin((uint64_t)k[r])], 1u) : 0u;
    __syncthreads();
    // exclusive scans over the bins: of the block's counts and of the totals
    uint32_t x = 0, y = 0, cx = 0, cy = 0;
    if (t < HBINS) {
        x = cx = s_cnt[t];
        y = cy = bins[t];
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t u = (uint32_t)__shfl_up((int)x, o, 64), v = (uint32_t)__shfl_up((int)y, o, 64);
            x += lane >= (uint32_t)o ? u : 0u;
            y += lane >= (uint32_t)o ? v : 0u;
        }
        if (lane == 63u) {
            s_red[0][wv] = x;
            s_red[1][wv] = y;
        }
    }
    __syncthreads();
    if (t < HBINS) {
        for (uint32_t w = 0; w < wv; ++w) {
            x += s_red[0][w];
            y += s_red[1][w];
        }
        const uint32_t at = cx ? atomicAdd(cursor + t, cx) : 0u;
        s_start[t] = x - cx;
        s_goff[t] = y - cy + at - (x - cx);
    }
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < ROUTE_CHUNK / 64u; ++r)
        if (r * 64u + lane < heavy)
            s_key[s_start[heavy_bin((uint64_t)k[r])] + rank[r]] = k[r];
    __syncthreads();
    const uint32_t total = s_start[HBINS - 1u] + s_cnt[HBINS - 1u];
    for (uint32_t q = t; q < total; q += 64u * HP_WAVES) {
        const KeyT<KB> v = s_key[q];
        const uint32_t dst = s_goff[heavy_bin((uint64_t)v)] + q;
        if (dst < n) // the counts and the ranks agree; checked, never trusted
            out[dst] = v;
        else
            atomicOr(err, LE_SORT);
    }
}

// counts windows of HS_WINDOW grouped heavy keys (few bins each) per block
#define HS_THREADS 512u
#define HS_WINDOW (HS_THREADS * 64u)
template <int KB>
__global__ __launch_bounds__(HS_THREADS) void k_heavy_sum(const KeyT<KB> *__restrict__ keys,
                                                          const uint32_t *__restrict__ bins,
                                                          uint64_t *__restrict__ tkeys, uint32_t *__restrict__ tcnt,
                                                          uint32_t tlog2, uint32_t *__restrict__ err)
{
    __shared__ heavy_lds T;
    __shared__ uint32_t s_n;
    if (threadIdx.x == 0)
        s_n = 0;
    __syncthreads();
    if (threadIdx.x < HBINS)
        atomicAdd(&s_n, bins[threadIdx.x]);
    __syncthreads();
    const uint32_t n = s_n; // heavy keys
    const uint64_t w0 = (uint64_t)blockIdx.x * HS_WINDOW;
    if (w0 >= n)
        return;
    heavy_clear(T);
    uint32_t claims = 0;
    for (uint32_t g = 0; g < HS_WINDOW; g += HS_THREADS * 8u) {
        KeyT<KB> k[8];
#pragma unroll
        for (uint32_t r = 0; r < 8u; ++r) { // every load first, from clamped positions
            const uint64_t i = w0 + g + r * HS_THREADS + threadIdx.x;
            k[r] = __builtin_nontemporal_load(keys + (i < n ? i : n - 1u));
        }
#pragma unroll
        for (uint32_t r = 0; r < 8u; ++r)
            heavy_add(T, w0 + g + r * HS_THREADS + threadIdx.x < n, (unsigned long long)k[r], tkeys, tcnt, tlog2, err,
                          claims);
    }
    heavy_flush(T, tkeys, tcnt, tlog2, err, claims);
}

// every chunk moves its staged light keys to its scanned offset
template <int KB>
__global__ __launch_bounds__(256) void k_light_move(const KeyT<KB> *__restrict__ stage, uint32_t nchunks,
                                                    const uint32_t *__restrict__ coff, KeyT<KB> *__restrict__ out)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t nw = gridDim.x * 4u;
    for (uint32_t c = blockIdx.x * 4u + (threadIdx.x >> 6); c < nchunks; c += nw) {
        const uint32_t off = coff[c], cnt = coff[c + 1] - off; // cnt <= ROUTE_CHUNK
        const KeyT<KB> *src = stage + (size_t)c * ROUTE_CHUNK;
        KeyT<KB> v[ROUTE_CHUNK / 64u];
#pragma unroll
        for (uint32_t r = 0; r < ROUTE_CHUNK / 64u; ++r)
            v[r] = r * 64u + lane < cnt ? __builtin_nontemporal_load(src + r * 64u + lane) : (KeyT<KB>)0;
#pragma unroll
        for (uint32_t r = 0; r < ROUTE_CHUNK / 64u; ++r)
            if (r * 64u + lane < cnt)
                out[(size_t)off + r * 64u + lane] = v[r];
    }
}

// After a routing pass in which the table turned keys away (*err set): every
// key flagged heavy that is not in the table goes to the sketch instead, and
// the chunks are staged again.  A key is either in the table for all of
// its occurrences or for none: slots only fill, so a key's probe window that
// had no room for it never gains room, and once the key holds a slot every
// later probe finds it.  Blocks exit at once when *err is clear.
template <int KB>
__global__ __launch_bounds__(256) void k_reflag(const KeyT<KB> *__restrict__ keys, uint64_t n, uint32_t nchunks,
                                                const uint64_t *__restrict__ tkeys, uint32_t tlog2,
                                                const uint8_t *__restrict__ flag, KeyT<KB> *__restrict__ stage,
                                                uint32_t *__restrict__ ccount, const uint32_t *__restrict__ err)
{
    if (*err == 0)
        return;
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t below = (1ull << lane) - 1ull;
    const uint32_t nw = gridDim.x * 4u;
    for (uint32_t c = blockIdx.x * 4u + (threadIdx.x >> 6); c < nchunks; c += nw) {
        const uint64_t base = (uint64_t)c * ROUTE_CHUNK;
        uint32_t light = 0;
        for (uint32_t st = 0; st < ROUTE_CHUNK / 64u; ++st) {
            const uint64_t i = base + st * 64u + lane;
            bool f = false;
            KeyT<KB> x = 0;
            if (i < n) {
                x = keys[i];
                f = flag[i] || t_find(tkeys, tlog2, (uint64_t)x) == T_NONE;
            }
            const uint64_t m = __ballot(f);
            if (f)
                stage[base + light + (uint32_t)__popcll(m & below)] = x;
            light += (uint32_t)__popcll(m);
        }
        if (lane == 0)
            ccount[c] = light;
    }
}

// Queries of the learned form.  A key is counted entirely in one part: only
// keys the network scores heavy ever enter the table, and a heavy key either
// holds a slot for all its occurrences or for none (k_reflag).  So a key found
// in the table is answered with its table count, and every other key with
// the sketch estimate.  Two kernels give that same answer:
//   k_table_query    looks every key up in the table first (no network); the
//                    probe ends at the first empty slot, so it is used while
//                    the table is at most half full and has never filled
//   k_learned_query  scores 32 keys per wavefront on the matrix cores and
//                    probes the table only for heavy-scored keys
// Both read a key's sketch bucket only when the table does not answer it.
typedef unsigned int lq_u32x4 __attribute__((ext_vector_type(4)));

__device__ static inline uint32_t lq_sel4(const uint4 &v, uint32_t k)
{
    const uint32_t lo = (k & 1u) ? v.y : v.x;
    const uint32_t hi = (k & 1u) ? v.w : v.z;
    return (k & 2u) ? hi : lo;
}

// Sketch estimate of key x by a pair of lanes PAIR apart, one 16-byte half of
// the bucket each (as k_query); need is the same on both lanes of a pair,
// and the exchanges stay outside the branches.
template <int KB, int PAIR>
__device__ static inline uint32_t lq_sketch(bool need, uint64_t x, uint32_t half, const qs_sdesc &d0,
                                            const uint32_t *s_masks, const uint32_t *__restrict__ low,
                                            const uint32_t *__restrict__ high)
{
    uint4 v = make_uint4(0u, 0u, 0u, 0u);
    uint32_t Mh = 0;
    if (need) {
        const KeyT<KB> key = (KeyT<KB>)x;
        const uint32_t M = s_masks[qs_maskidx_d(key, d0)];
        const uint32_t b = qs_bucket_d(key, d0);
        const lq_u32x4 vv = __builtin_nontemporal_load(reinterpret_cast<const lq_u32x4 *>(low + (size_t)b * 8u) + half);
        v = make_uint4(vv[0], vv[1], vv[2], vv[3]);
        Mh = half ? (M >> 16) : (M & 0xffffu);
    }
    uint32_t lo = 0xffffffffu;
    for (uint32_t m = Mh; m; m &= m - 1u) {
        const uint32_t jj = (uint32_t)__builtin_ctz(m);
        lo = min(lo, (lq_sel4(v, jj >> 2) >> ((jj & 3u) * 8u)) & 0xffu);
    }
    lo = min(lo, (uint32_t)__shfl_xor((int)lo, PAIR, 64));
    const uint32_t wo = (uint32_t)__shfl_xor((int)v.w, PAIR, 64);
    const uint32_t w = half ? v.w : wo;
    uint32_t hi = 0xffffffffu;
    if (need && w > QS_LINK_START) {
        const uint32_t *g = high + (size_t)(w - QS_LINK_START) * 32u + 16u * half;
        for (uint32_t m = Mh; m; m &= m - 1u)
            hi = min(hi, g[__builtin_ctz(m)]);
    }
    hi = min(hi, (uint32_t)__shfl_xor((int)hi, PAIR, 64));
    return lo + (w > QS_LINK_START ? hi : 0u);
}

template <int KB>
__global__ __launch_bounds__(256) void k_table_query(const KeyT<KB> *__restrict__ keys, uint64_t n,
                                                     const uint64_t *__restrict__ tkeys,
                                                     const uint32_t *__restrict__ tcnt, uint32_t tlog2, qs_sdesc d0,
                                                     const uint32_t *__restrict__ low,
                                                     const uint32_t *__restrict__ high,
                                                     const uint32_t *__restrict__ masks, uint32_t *__restrict__ out)
{
    __shared__ uint32_t s_masks[QS_MAX_MASKS];
    for (uint32_t e = threadIdx.x; e < d0.n_masks; e += blockDim.x)
        s_masks[e] = masks[e];
    __syncthreads();
    const uint32_t half = threadIdx.x & 1u;
    const uint64_t stride = (uint64_t)gridDim.x * 128u;
    for (uint64_t i = (uint64_t)blockIdx.x * 128u + (threadIdx.x >> 1); i < n; i += stride) {
        const uint64_t x = key64<KB>(keys, i);
        // the all-ones key is the empty-slot marker and is never in the table
        const uint32_t s = x != T_EMPTY ? t_find(tkeys, tlog2, x) : T_NONE;
        const bool need = s == T_NONE;
        const uint32_t est = lq_sketch<KB, 1>(need, x, half, d0, s_masks, low, high);
        if (!half)
            out[i] = need ? est : tcnt[s];
    }
}

template <int KB>
__global__ __launch_bounds__(256) void k_learned_query(const KeyT<KB> *__restrict__ keys, uint64_t n,
                                                       const uint16_t *__restrict__ pb, const float *__restrict__ p,
                                                       float thr, const uint64_t *__restrict__ tkeys,
                                                       const uint32_t *__restrict__ tcnt, uint32_t tlog2,
                                                       qs_sdesc d0, const uint32_t *__restrict__ low,
                                                       const uint32_t *__restrict__ high,
                                                       const uint32_t *__restrict__ masks,
                                                       uint32_t *__restrict__ out)
{
    __shared__ mlp_lds S;
    __shared__ uint32_t s_masks[QS_MAX_MASKS];
    for (uint32_t e = threadIdx.x; e < d0.n_masks; e += blockDim.x)
        s_masks[e] = masks[e];
    load_mlp(S, pb, p); // ends with a barrier
    const uint32_t lane = threadIdx.x & 63u, l32 = lane & 31u, half = lane >> 5;
    const uint64_t gw = ((uint64_t)blockIdx.x * 256u + threadIdx.x) >> 6;
    const uint64_t nw = ((uint64_t)gridDim.x * 256u) >> 6;
    if (n == 0)
        return;
    uint64_t xn = key_at<KB>(keys, gw * 32u + l32, n);
    for (uint64_t base = gw * 32u; base < n; base += nw * 32u) {
        const uint64_t i = base + l32;
        const bool valid = i < n;
        const uint64_t x = xn;
        xn = key_at<KB>(keys, i + nw * 32u, n); // the next tile's key, loaded while this one is scored
        const float y = mlp_mfma(S, x);         // lanes 0..31: the scores of keys 0..31
        uint32_t s = T_NONE;
        if (lane < 32u && valid && y >= thr && x != T_EMPTY)
            s = t_find(tkeys, tlog2, x);
        s = (uint32_t)__shfl((int)s, (int)l32, 64); // lane l + 32 takes key l's answer
        const bool need = valid && s == T_NONE;
        const uint32_t est = lq_sketch<KB, 32>(need, x, half, d0, s_masks, low, high);
        if (lane < 32u && valid)
            out[i] = need ? est : tcnt[s];
    }
}

__global__ void k_table_clear(uint64_t *__restrict__ tkeys, uint32_t *__restrict__ tcnt, uint64_t cap)
{
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < cap; e += (uint64_t)gridDim.x * blockDim.x) {
        tkeys[e] = T_EMPTY;
        tcnt[e] = 0;
    }
}

// ===========================================================================
// host
// ===========================================================================
static uint32_t lgrid(uint64_t want, uint32_t cap)
{
    return (uint32_t)(want < 1 ? 1 : (want > cap ? cap : want));
}

extern "C" void qs_learned_destroy(qs_learned *L)
{
    if (!L)
        return;
    hipDeviceSynchronize();
    qs_destroy(L->sk);
    hipFree(L->d_p);
    hipFree(L->d_pb);
    hipFree(L->d_m);
    hipFree(L->d_v);
    hipFree(L->d_part); // and d_g and d_loss, its tail
    hipFree(L->d_tkeys);
    hipFree(L->d_tcnt);
    hipFree(L->d_bins); // and d_err, its tail
    hipFree(L->d_flag);
    hipFree(L->d_count);
    hipFree(L->d_bsum);
    hipFree(L->d_stage);
    hipFree(L->d_light);
    if (L->h_pin)
        hipHostFree(L->h_pin);
    free(L);
}

extern "C" qs_sketch *qs_learned_sketch(qs_learned *L)
{
    return L ? L->sk : nullptr;
}

extern "C" int qs_learned_create(const qs_params *p, uint32_t table_log2, uint64_t init_seed, qs_learned **out)
{
    if (!out || !p || table_log2 < 10 || table_log2 > 28)
        return QS_ERR_PARAM;
    *out = nullptr;
    qs_learned *L = (qs_learned *)calloc(1, sizeof(qs_learned));
    if (!L)
        return QS_ERR_NOMEM;
    int rc = qs_create(p, &L->sk);
    if (rc) {
        free(L);
        return rc;
    }
    L->key_bytes = p->key_bytes;
    L->tlog2 = table_log2;
    L->tcap = 1ull << table_log2;
    L->thr = INFINITY;
    bool ok = hipMalloc(&L->d_p, NPAR * 4) == hipSuccess && hipMalloc(&L->d_pb, NPAR * 2) == hipSuccess &&
              hipMalloc(&L->d_m, NPAR * 4) == hipSuccess && hipMalloc(&L->d_v, NPAR * 4) == hipSuccess &&
              hipMalloc(&L->d_part, 4ull * PART_STRIDE * (GRAD_BLOCKS + 1u)) == hipSuccess &&
              hipMalloc(&L->d_tkeys, L->tcap * 8) == hipSuccess && hipMalloc(&L->d_tcnt, L->tcap * 4) == hipSuccess &&
              hipMalloc(&L->d_bins, 4ull * (2u * HBINS + 2u)) == hipSuccess &&
              hipHostMalloc(&L->h_pin, 16, hipHostMallocDefault) == hipSuccess;
    if (!ok) {
        qs_learned_destroy(L);
        return qs_alloc_failed();
    }
    L->d_err = L->d_bins + 2u * HBINS;
    L->d_g = L->d_part + (size_t)PART_STRIDE * GRAD_BLOCKS;
    L->d_loss = L->d_g + NPAR;
    // initial weights: uniform in +-1/sqrt(64) from a SplitMix64 stream, biases 0
    std::vector<float> h(NPAR, 0.f);
    uint64_t st = init_seed;
    auto next = [&]() {
        uint64_t z = (st += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
    };
    auto uni = [&]() { return (float)((double)(next() >> 11) * (1.0 / 9007199254740992.0) * 2.0 - 1.0) * 0.125f; };
    for (int e = 0; e < 4096; ++e)
        h[OFF_W1 + e] = uni();
    for (int e = 0; e < 4096; ++e)
        h[OFF_W2 + e] = uni();
    for (int e = 0; e < 64; ++e)
        h[OFF_W3 + e] = uni();
    rc = qs_mlp_set_params(L, h.data());
    if (rc == QS_OK)
        rc = qs_learned_clear(L);
    if (rc) {
        qs_learned_destroy(L);
        return rc;
    }
    *out = L;
    return QS_OK;
}

extern "C" int qs_mlp_get_params(qs_learned *L, float *hp)
{
    if (!L || !hp)
        return QS_ERR_PARAM;
    CK(hipDeviceSynchronize());
    CK(hipMemcpy(hp, L->d_p, NPAR * 4, hipMemcpyDeviceToHost));
    return QS_OK;
}

extern "C" int qs_mlp_set_params(qs_learned *L, const float *hp)
{
    if (!L || !hp)
        return QS_ERR_PARAM;
    if (L->inserted)
        return QS_ERR_STATE; // the routing of the keys already in would change
    CK(hipDeviceSynchronize());
    CK(hipMemcpy(L->d_p, hp, NPAR * 4, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_set_params, dim3(33), dim3(256), 0, 0, L->d_p, L->d_pb, L->d_m, L->d_v);
    CK(hipGetLastError());
    CK(hipDeviceSynchronize());
    L->step = 0;
    return QS_OK;
}

// the gradient of a batch and its loss, to d_g and d_loss; with `update`, one
// Adam step on them
static int grad_launch(qs_learned *L, const void *d_keys, const float *d_t, uint32_t n, bool update, float lr,
                       float beta1, float beta2, float eps, float c1, float c2)
{
    const uint32_t groups = n / GK + (n % GK != 0);
    const uint32_t rows = groups < GRAD_BLOCKS ? groups : GRAD_BLOCKS;
    const dim3 grid(rows), block(GT);
    const float inv = 1.0f / (float)n;
    if (L->key_bytes == 4)
        hipLaunchKernelGGL(k_mlp_grad<4>, grid, block, 0, 0, (const uint32_t *)d_keys, d_t, n, L->d_pb, L->d_p, inv,
                           L->d_part);
    else
        hipLaunchKernelGGL(k_mlp_grad<8>, grid, block, 0, 0, (const uint64_t *)d_keys, d_t, n, L->d_pb, L->d_p, inv,
                           L->d_part);
    hipLaunchKernelGGL(k_grad_sum, dim3(PART_STRIDE / 64u), dim3(64 * SUM_WAVES), 0, 0, L->d_part, rows, L->d_g, update,
                       L->d_p, L->d_pb, L->d_m, L->d_v, lr, beta1, beta2, eps, c1, c2);
    CK(hipGetLastError());
    return QS_OK;
}

extern "C" int qs_mlp_grad(qs_learned *L, const void *d_keys, const float *d_t, uint32_t n, float *loss,
                           float *h_grad)
{
    if (!L || !d_keys || !d_t || n == 0)
        return QS_ERR_PARAM;
    int rc = grad_launch(L, d_keys, d_t, n, false, 0.f, 0.f, 0.f, 0.f, 1.f, 1.f);
    if (rc)
        return rc;
    CK(hipDeviceSynchronize());
    if (loss)
        CK(hipMemcpy(loss, L->d_loss, 4, hipMemcpyDeviceToHost));
    if (h_grad)
        CK(hipMemcpy(h_grad, L->d_g, NPAR * 4, hipMemcpyDeviceToHost));
    return QS_OK;
}

extern "C" int qs_mlp_step(qs_learned *L, const void *d_keys, const float *d_t, uint32_t n, float lr, float beta1,
                           float beta2, float eps, float *loss, float *h_grad)
{
    if (!L || !d_keys || !d_t || n == 0)
        return QS_ERR_PARAM;
    if (L->inserted)
        return QS_ERR_STATE; // the routing of the keys already in would change
    const float step = (float)(L->step + 1);
    int rc = grad_launch(L, d_keys, d_t, n, true, lr, beta1, beta2, eps, 1.f - powf(beta1, step), 1.f - powf(beta2, step));
    if (rc)
        return rc;
    L->step++;
    if (loss || h_grad)
        CK(hipDeviceSynchronize());
    if (h_grad)
        CK(hipMemcpy(h_grad, L->d_g, NPAR * 4, hipMemcpyDeviceToHost));
    if (loss)
        CK(hipMemcpy(loss, L->d_loss, 4, hipMemcpyDeviceToHost));
    return QS_OK;
}

extern "C" int qs_mlp_score(qs_learned *L, const void *d_keys, uint64_t n, float *d_scores, int mfma)
{
    if (!L || (!d_keys && n) || (!d_scores && n))
        return QS_ERR_PARAM;
    if (n == 0)
        return QS_OK;
    if (mfma) {
        const dim3 grid(lgrid((n + 127) / 128, 4096)), block(256);
        if (L->key_bytes == 4)
            hipLaunchKernelGGL(k_mlp_mfma<4>, grid, block, 0, 0, (const uint32_t *)d_keys, n, L->d_pb, L->d_p,
                               d_scores);
        else
            hipLaunchKernelGGL(k_mlp_mfma<8>, grid, block, 0, 0, (const uint64_t *)d_keys, n, L->d_pb, L->d_p,
                               d_scores);
    } else {
        const dim3 grid(lgrid((n + 255) / 256, 4096)), block(256);
        if (L->key_bytes == 4)
            hipLaunchKernelGGL(k_mlp_fwd<4>, grid, block, 0, 0, (const uint32_t *)d_keys, n, L->d_pb, L->d_p,
                               d_scores);
        else
            hipLaunchKernelGGL(k_mlp_fwd<8>, grid, block, 0, 0, (const uint64_t *)d_keys, n, L->d_pb, L->d_p,
                               d_scores);
    }
    CK(hipGetLastError());
    CK(hipDeviceSynchronize());
    return QS_OK;
}

extern "C" int qs_learned_set_threshold(qs_learned *L, float thr)
{
    if (!L || std::isnan(thr))
        return QS_ERR_PARAM;
    if (L->inserted && thr != L->thr)
        return QS_ERR_STATE; // the routing of the keys already in would change
    L->thr = thr;
    return QS_OK;
}

extern "C" float qs_learned_threshold(const qs_learned *L)
{
    return L ? L->thr : NAN;
}

extern "C" int qs_learned_clear(qs_learned *L)
{
    if (!L)
        return QS_ERR_PARAM;
    int rc = qs_clear(L->sk);
    if (rc)
        return rc;
    hipLaunchKernelGGL(k_table_clear, dim3(lgrid((L->tcap + 255) / 256, 2048)), dim3(256), 0, 0, L->d_tkeys,
                       L->d_tcnt, L->tcap);
    CK(hipGetLastError());
    CK(hipMemset(L->d_err, 0, 8));
    CK(hipDeviceSynchronize());
    L->inserted = 0;
    L->full = 0;
    L->used = 0;
    return QS_OK;
}

// the routing buffers freed; the light keys of the call may be kept
static void free_route(qs_learned *L, bool keep_light)
{
    hipFree(L->d_flag);
    hipFree(L->d_count);
    hipFree(L->d_bsum);
    hipFree(L->d_stage);
    L->d_flag = nullptr;
    L->d_count = nullptr;
    L->d_bsum = nullptr;
    L->d_stage = nullptr;
    L->rcap = 0;
    if (keep_light)
        return;
    hipFree(L->d_light);
    L->d_light = nullptr;
}

static int ensure_route(qs_learned *L, uint64_t n)
{
    if (!L->cus) {
        int cu = 0;
        if (hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, L->sk->device) != hipSuccess || cu <= 0)
            cu = 256;
        L->cus = (uint32_t)cu;
    }
    if (L->rcap >= n)
        return QS_OK;
    free_route(L, false);
    const uint64_t chunks = (n + ROUTE_CHUNK - 1) / ROUTE_CHUNK;
    if (hipMalloc(&L->d_flag, n) != hipSuccess || hipMalloc(&L->d_count, (chunks + 1) * 4) != hipSuccess ||
        hipMalloc(&L->d_bsum, 4ull * qs_scan_sums(chunks)) != hipSuccess ||
        hipMalloc(&L->d_stage, chunks * ROUTE_CHUNK * L->key_bytes) != hipSuccess ||
        hipMalloc(&L->d_light, n * L->key_bytes) != hipSuccess) {
        free_route(L, false);
        return qs_alloc_failed();
    }
    L->rcap = n;
    return QS_OK;
}

// one piece of a call; *n_heavy grows by its heavy keys
template <int KB>
static int learned_piece(qs_learned *L, const KeyT<KB> *keys, uint64_t n, uint64_t *n_heavy)
{
    if (L->sk->sticky_err == QS_ERR_INTERNAL)
        return QS_ERR_INTERNAL;
    int rc = ensure_route(L, n);
    if (rc)
        return rc;
    const uint32_t chunks = (uint32_t)((n + ROUTE_CHUNK - 1) / ROUTE_CHUNK); // n < 2^32
    KeyT<KB> *stage = (KeyT<KB> *)L->d_stage;
    CK(hipMemsetAsync(L->d_bins, 0, 4u * (2u * HBINS + 1u), 0)); // bins, cursors and this call's flag
    hipLaunchKernelGGL(k_route<KB>, dim3(chunks < L->cus ? chunks : L->cus), dim3(ROUTE_THREADS), 0, 0, keys, n, chunks,
                       L->d_pb, L->d_p, L->thr, L->d_flag, stage, L->d_count, L->d_bins);
    if (n < HEAVY_PART_MIN) {
        hipLaunchKernelGGL(k_heavy_count<KB>, dim3(lgrid((chunks + 3u) / 4u, 2u * L->cus)), dim3(256), 0, 0, stage, n,
                           chunks, L->d_count, L->d_tkeys, L->d_tcnt, L->tlog2, L->d_err);
    } else {
        // (grouped in the buffer that takes the light keys afterwards)
        KeyT<KB> *grouped = (KeyT<KB> *)L->d_light;
        hipLaunchKernelGGL(k_heavy_part<KB>, dim3((chunks + HP_WAVES - 1u) / HP_WAVES), dim3(64 * HP_WAVES), 0, 0,
                           stage, n, chunks, L->d_count, L->d_bins, L->d_bins + HBINS, grouped, L->d_err);
        hipLaunchKernelGGL(k_heavy_sum<KB>, dim3((uint32_t)((n + HS_WINDOW - 1) / HS_WINDOW)), dim3(HS_THREADS), 0, 0,
                           grouped, L->d_bins, L->d_tkeys, L->d_tcnt, L->tlog2, L->d_err);
    }
    const dim3 wgrid(lgrid((chunks + 3u) / 4u, 8u * L->cus)); // a wavefront per chunk
    // keys the table turned away go to the sketch (no work unless it did)
    hipLaunchKernelGGL(k_reflag<KB>, wgrid, dim3(256), 0, 0, keys, n, chunks, L->d_tkeys, L->tlog2, L->d_flag, stage,
                       L->d_count, L->d_err);
    if (chunks <= 16384u) // one launch while one block is quick enough
        qs_scan_digits(L->d_count, chunks, 1, L->d_count + chunks, 0);
    else
        qs_scan_u32(L->d_count, chunks, L->d_bsum, 0);
    hipLaunchKernelGGL(k_light_move<KB>, wgrid, dim3(256), 0, 0, stage, chunks, L->d_count, (KeyT<KB> *)L->d_light);
    CK(hipGetLastError());
    CK(hipMemcpy(L->h_pin, L->d_count + chunks, 4, hipMemcpyDeviceToHost));
    CK(hipMemcpy(L->h_pin + 1, L->d_err, 8, hipMemcpyDeviceToHost));
    const uint64_t n_light = L->h_pin[0];
    if (L->h_pin[1] & LE_FULL)
        L->full = 1;
    if (L->h_pin[1] & LE_SORT) {
        L->sk->sticky_err = QS_ERR_INTERNAL; // keys are missing from the table: invalid until the clear
        return QS_ERR_INTERNAL;
    }
    L->used = L->h_pin[2];
    L->inserted += n;
    *n_heavy += n - n_light;
    if (n_light == 0)
        return QS_OK;
    rc = qs_insert(L->sk, L->d_light, n_light);
    if (rc == QS_ERR_NOMEM) { // nothing was inserted: again without the buffers that the routing is done with
        free_route(L, true);
        rc = qs_insert(L->sk, L->d_light, n_light);
    }
    return rc;
}

// A call is one piece when the routing buffers for it fit the device, else as many as
// it takes: the pieces one after the other are the same insert.  (The buffers hold a
// flag and two copies of a key; a form that placed the light keys at once held one, so
// calls that fitted then must not be refused for the second.)
#define ROUTE_PIECE_MIN (1ull << 20)
template <int KB>
static int learned_insert(qs_learned *L, const KeyT<KB> *keys, uint64_t n, uint64_t *n_heavy)
{
    uint64_t piece = n, heavy = 0;
    int rc = ensure_route(L, piece);
    while (rc == QS_ERR_NOMEM && piece > ROUTE_PIECE_MIN) {
        piece = (piece + 1) / 2;
        rc = ensure_route(L, piece);
    }
    for (uint64_t off = 0; rc == QS_OK && off < n; off += piece)
        rc = learned_piece<KB>(L, keys + off, n - off < piece ? n - off : piece, &heavy);
    if (n_heavy)
        *n_heavy = heavy;
    return rc;
}

extern "C" int qs_learned_insert(qs_learned *L, const void *d_keys, uint64_t n, uint64_t *n_heavy)
{
    if (!L || (!d_keys && n))
        return QS_ERR_PARAM;
    if (n == 0) {
        if (n_heavy)
            *n_heavy = 0;
        return QS_OK;
    }
    if (n > 0xffffffffull)
        return QS_ERR_PARAM; // tile offsets are 32-bit
    return L->key_bytes == 4 ? learned_insert<4>(L, (const uint32_t *)d_keys, n, n_heavy)
                             : learned_insert<8>(L, (const uint64_t *)d_keys, n, n_heavy);
}

extern "C" int qs_learned_query(qs_learned *L, const void *d_keys, uint64_t n, uint32_t *d_counts)
{
    if (!L || ((!d_keys || !d_counts) && n))
        return QS_ERR_PARAM;
    if (n == 0)
        return QS_OK;
    if (n > 0xffffffffull)
        return QS_ERR_PARAM; // the sketch's query bound
    const qs_sketch *s = L->sk;
    const dim3 block(256);
    if (!L->full && 2ull * L->used <= L->tcap) {
        // probes of absent keys stay short: look the table up first
        const dim3 grid(lgrid((2 * n + 255) / 256, 2048));
        if (L->key_bytes == 4)
            hipLaunchKernelGGL(k_table_query<4>, grid, block, 0, 0, (const uint32_t *)d_keys, n, L->d_tkeys,
                               L->d_tcnt, L->tlog2, s->h_desc[0], s->d_low, s->d_high, s->d_masks, d_counts);
        else
            hipLaunchKernelGGL(k_table_query<8>, grid, block, 0, 0, (const uint64_t *)d_keys, n, L->d_tkeys,
                               L->d_tcnt, L->tlog2, s->h_desc[0], s->d_low, s->d_high, s->d_masks, d_counts);
    } else {
        const dim3 grid(lgrid((n + 127) / 128, 8192));
        if (L->key_bytes == 4)
            hipLaunchKernelGGL(k_learned_query<4>, grid, block, 0, 0, (const uint32_t *)d_keys, n, L->d_pb, L->d_p,
                               L->thr, L->d_tkeys, L->d_tcnt, L->tlog2, s->h_desc[0], s->d_low, s->d_high,
                               s->d_masks, d_counts);
        else
            hipLaunchKernelGGL(k_learned_query<8>, grid, block, 0, 0, (const uint64_t *)d_keys, n, L->d_pb, L->d_p,
                               L->thr, L->d_tkeys, L->d_tcnt, L->tlog2, s->h_desc[0], s->d_low, s->d_high,
                               s->d_masks, d_counts);
    }
    CK(hipGetLastError());
    CK(hipDeviceSynchronize());
    return QS_OK;
}

extern "C" int qs_learned_table(qs_learned *L, uint64_t *h_keys, uint32_t *h_counts, uint64_t cap,
                                uint64_t *n_used)
{
    if (!L || !n_used)
        return QS_ERR_PARAM;
    std::vector<uint64_t> k(L->tcap);
    std::vector<uint32_t> c(L->tcap);
    CK(hipDeviceSynchronize());
    CK(hipMemcpy(k.data(), L->d_tkeys, L->tcap * 8, hipMemcpyDeviceToHost));
    CK(hipMemcpy(c.data(), L->d_tcnt, L->tcap * 4, hipMemcpyDeviceToHost));
    uint64_t u = 0;
    for (uint64_t e = 0; e < L->tcap; ++e) {
        if (k[e] == T_EMPTY)
            continue;
        if (u < cap && h_keys && h_counts) {
            h_keys[u] = k[e];
            h_counts[u] = c[e];
        }
        ++u;
    }
    *n_used = u;
    return QS_OK;
}

extern "C" int qs_learned_table_full(const qs_learned *L)
{
    return L ? (int)L->full : QS_ERR_PARAM;
}

extern "C" int qs_learned_memory(const qs_learned *L, uint64_t *table_bytes, uint64_t *mlp_bytes,
                                 uint64_t *sketch_bytes)
{
    if (!L)
        return QS_ERR_PARAM;
    if (table_bytes)
        *table_bytes = L->tcap * 12u;
    if (mlp_bytes)
        *mlp_bytes = (4096u * 2 + 64u) * 2u + (64u * 2 + 1u) * 4u; // BF16 weights + FP32 biases
    if (sketch_bytes)
        *sketch_bytes = L->sk->low_words * 4u + L->sk->high_words * 4u;
    return QS_OK;
}
