// Matrix-core projections of up to 32 tokens (a short message): one or two
// 16-token MFMA tiles, every workgroup the whole K of its rows, so that no partial sums
// leave it and the consumers' work is its epilogue (mfma.hip describes the
// activation planes and the general kernels).
//
// Bound: HBM, one pass over the weights. 256 workgroups of eight waves, one per
// CU, own 1/256 of the rows each: 24 of q|k|v (12 RoPE pairs), 12 of o and
// down, 72 of gate|up (36 gate rows and the matching up rows); rows are padded
// to 16-row operand tiles in registers only (the spare lanes repeat the last
// row). Wave s takes the s-th eighth of the columns and keeps DEPTH 64-column
// stages of weights and activations in flight, straight to registers: no other
// wave needs them. The eight sums meet in LDS. (Plain weight loads: a stage is
// half of its rows' 128-byte lines, and non-temporal ones fetched those twice,
// gate|up 18 against 13 us.)
// Measured at 7 tokens, with the 64-token tiles of mfma.hip before (128 to 288
// workgroups with one stage in flight each, and partials to sum afterwards):
// q|k|v 8.6 us (15.1 + 3.8 epilogue), o 6.6 (11.8), gate|up 13.6 (22.4 + 4.8),
// down 11.8 (14.5 + 3.8); the layer after 1203 positions 102 -> 68 us. At 32
// tokens the activations, read by every workgroup, weigh as much as the
// weights: the layer after 1200 positions 100 -> 86 us; at 33 the 64-token
// tiles take over.
#include "lh_device.h"
#include "lh_internal.h"
#include "lh_mfma.h"

#include <type_traits>

namespace lh {

enum { EPI_RESIDUAL, EPI_QKV, EPI_GATEUP };

constexpr uint32_t SMALL_GROUPS = 256;

struct SmallArgs {
    const uint8_t* W;          // weight rows (q|k|v, o, gate, down)
    const uint8_t* W1;         // up rows (EPI_GATEUP)
    float s0, s1, s2;          // tensor scales
    const uint16_t* xs;        // activation planes (xs_at)
    uint32_t stride;           // tokens per plane
    uint32_t count;
    const float* row_scale;    // EPI_GATEUP: 2^-e per token
    const float* wave_scale;   // o: 2^-e per (token, K eighth), NULL otherwise
    float* x;                  // EPI_RESIDUAL: rows of 3072, updated in place
    const lh_step_params* params;
    float* q;
    float* kcache;
    float* vcache;
    uint32_t capacity;
    uint16_t* planes;          // EPI_GATEUP: three BF16 planes of 9216 columns
};

// K columns, P activation planes, MT token tiles, NR rows per workgroup in RT
// operand tiles, DEPTH stages in flight. grid 256, block 512.
template <int K, int P, int MT, int NR, int DEPTH, int EPI>
__device__ __forceinline__ void small_body(const SmallArgs& a)
{
    constexpr int RT = (NR + 15) / 16, STAGES = K / 64 / 8, D = DEPTH < STAGES ? DEPTH : STAGES;
    constexpr uint32_t RS = 16 * RT + 4;   // reduction row stride
    using V = typename std::conditional<P == PLANES_BF16, bf16x8, f16x8>::type;
    __shared__ __attribute__((aligned(16))) float red[8 * 16 * MT * RS];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wg = blockIdx.x;
    const uint32_t s = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t col = lane & 15, g = lane >> 4;
    // Where a tile has at most eight tokens, its spare lanes read them again
    // (half the lines).
    const size_t plane = (size_t)a.stride * K;
    const uint16_t* xsrc[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) {
        const uint32_t tl = a.count <= 16u * m + 8 ? col & 7 : col;
        xsrc[m] = a.xs + ((size_t)m * (K / 64) + s * STAGES) * 1024 + (g * 16 + tl) * 8;
    }
    const uint8_t* wsrc[RT];
#pragma unroll
    for (int r = 0; r < RT; r++) {
        const uint32_t n = 16 * r + col < NR ? 16 * r + col : NR - 1;
        const uint8_t* W = a.W;
        uint32_t row;
        if constexpr (EPI == EPI_QKV) {
            const uint32_t pair = wg * (NR / 2) + n % (NR / 2);
            row = (pair >> 6) * 128 + (pair & 63) + (n >= NR / 2 ? 64 : 0);
        } else if constexpr (EPI == EPI_GATEUP) {
            row = wg * (NR / 2) + n % (NR / 2);
            W = n >= NR / 2 ? a.W1 : a.W;
        } else {
            row = wg * NR + n;
        }
        wsrc[r] = W + (size_t)row * K + s * STAGES * 64 + 16 * g;
    }
    u32x4 w[D][RT], x[D][MT][P][2];
    auto issue = [&](int st, int slot) {
#pragma unroll
        for (int r = 0; r < RT; r++) {
            w[slot][r] = *reinterpret_cast<const u32x4*>(wsrc[r] + st * 64);
        }
#pragma unroll
        for (int m = 0; m < MT; m++) {
#pragma unroll
            for (int p = 0; p < P; p++) {
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    x[slot][m][p][h] = *reinterpret_cast<const u32x4*>(
                        xsrc[m] + p * plane + st * 1024 + h * 512);
                }
            }
        }
    };
#pragma unroll
    for (int st = 0; st < D; st++) {
        issue(st, st);
    }
    floatx4 acc[MT][RT];
#pragma unroll
    for (int m = 0; m < MT; m++) {
#pragma unroll
        for (int r = 0; r < RT; r++) {
            acc[m][r] = floatx4{};
        }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int st = 0; st < STAGES; st++) {
        const int slot = st % D;
#pragma unroll
        for (int r = 0; r < RT; r++) {
            V b[2];
            if constexpr (P == PLANES_BF16) {
                fp8x16_to_bf16x8x2(w[slot][r], b[0], b[1]);
            } else {
                fp8x16_to_f16x8x2(w[slot][r], b[0], b[1]);
            }
#pragma unroll
            for (int p = P - 1; p >= 0; p--) {   // from the smallest plane up
#pragma unroll
                for (int h = 0; h < 2; h++) {
#pragma unroll
                    for (int m = 0; m < MT; m++) {
                        const V v = __builtin_bit_cast(V, x[slot][m][p][h]);
                        if constexpr (P == PLANES_BF16) {
                            acc[m][r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, b[h],
                                acc[m][r], 0, 0, 0);
                        } else {
                            acc[m][r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v, b[h],
                                acc[m][r], 0, 0, 0);
                        }
                    }
                }
            }
        }
        if (st + D < STAGES) {
            issue(st + D, slot);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    // Lane: tokens 16m + 4g + k, row col of each tile.
#pragma unroll
    for (int m = 0; m < MT; m++) {
        float f[4] = {1.0f, 1.0f, 1.0f, 1.0f};
        if (a.wave_scale) {
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint32_t t = 16 * m + 4 * g + k;
                f[k] = a.wave_scale[(t < a.count ? t : 0) * 8 + s];
            }
        }
#pragma unroll
        for (int r = 0; r < RT; r++) {
#pragma unroll
            for (int k = 0; k < 4; k++) {
                red[(s * 16 * MT + 16 * m + 4 * g + k) * RS + 16 * r + col] = acc[m][r][k] * f[k];
            }
        }
    }
    __syncthreads();
    // Four rows n .. n + 3 of token t, the waves' sums in K order.
    auto total4 = [&](uint32_t t, uint32_t n) {
        const floatx4* p = reinterpret_cast<const floatx4*>(red + t * RS + n);
        floatx4 v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            v[i] = p[i * 16 * MT * RS / 4];
        }
#pragma unroll
        for (int i = 1; i < 8; i++) {
            v[0] = v[0] + v[i];
        }
        return v[0];
    };
    if constexpr (EPI == EPI_RESIDUAL) {
        const uint32_t t = tid / (NR / 4), n = tid % (NR / 4) * 4;
        if (t < a.count) {
            floatx4* px = reinterpret_cast<floatx4*>(a.x + (size_t)t * LH_HIDDEN + wg * NR + n);
            const floatx4 old = *px, v = total4(t, n);
            *px = old + v * a.s0;
        }
    } else if constexpr (EPI == EPI_QKV) {
        constexpr uint32_t NP = NR / 2;
        const uint32_t t = tid / (NP / 4), n = tid % (NP / 4) * 4;
        if (t < a.count) {
            // Four consecutive pairs lie in one head (12 and 64 are multiples of 4).
            const uint32_t pair = wg * NP + n, head = pair >> 6, i = pair & 63;
            const float scale = head < 32 ? a.s0 : (head < 40 ? a.s1 : a.s2);
            const floatx4 lo = total4(t, n) * scale, hi = total4(t, n + NP) * scale;
            const lh_token_params* tp = &a.params->tokens[t];
            const uint32_t position = a.params->length + t;
            if (head >= 40) {
                floatx4* vr = reinterpret_cast<floatx4*>(a.vcache +
                    lh_kv_index(a.capacity, 0, head - 40, position) + i);
                vr[0] = lo;
                vr[16] = hi;
                return;
            }
            // column i < 64 rotates with -x[i+64]; column i+64 with x[i].
            const floatx4 cl = *reinterpret_cast<const floatx4*>(tp->cosine + i);
            const floatx4 sl = *reinterpret_cast<const floatx4*>(tp->sine + i);
            const floatx4 ch = *reinterpret_cast<const floatx4*>(tp->cosine + i + 64);
            const floatx4 sh = *reinterpret_cast<const floatx4*>(tp->sine + i + 64);
            const floatx4 out_lo = lo * cl + (-hi) * sl, out_hi = hi * ch + lo * sh;
            if (head < 32) {
                floatx4* qh = reinterpret_cast<floatx4*>(a.q + (size_t)t * LH_QUERY + head * 128 +
                    i);
                qh[0] = out_lo * tp->qfactor;
                qh[16] = out_hi * tp->qfactor;
            } else {
                *reinterpret_cast<floatx4*>(a.kcache +
                    lh_k_index(a.capacity, 0, head - 32, position, i)) = out_lo;
                *reinterpret_cast<floatx4*>(a.kcache +
                    lh_k_index(a.capacity, 0, head - 32, position, i + 64)) = out_hi;
            }
        }
    } else {
        constexpr uint32_t NP = NR / 2;
        const uint32_t t = tid % (16 * MT), n = tid / (16 * MT) * 4;
        if (n < NP && t < a.count) {
            const float f = a.row_scale[t];
            const floatx4 gate = total4(t, n) * f, up = total4(t, n + NP) * f;
            float4 y;
            y.x = silu(gate[0] * a.s0) * (up[0] * a.s1);
            y.y = silu(gate[1] * a.s0) * (up[1] * a.s1);
            y.z = silu(gate[2] * a.s0) * (up[2] * a.s1);
            y.w = silu(gate[3] * a.s0) * (up[3] * a.s1);
            store_split4(a.planes, (size_t)a.stride * LH_INNER, xs_at(t, wg * NP + n, LH_INNER), y);
        }
    }
}

// (Device code only: the host pass has no matrix instructions.)
template <int K, int P, int MT, int NR, int DEPTH, int EPI>
__global__ void __launch_bounds__(512, 2)
k_small(SmallArgs a)
{
#ifdef __HIP_DEVICE_COMPILE__
    small_body<K, P, MT, NR, DEPTH, EPI>(a);
#endif
}

}  // namespace lh

using namespace lh;

// DEPTH1, DEPTH2: stages in flight with one and two token tiles (what 256
// registers hold).
template <int K, int P, int NR, int DEPTH1, int DEPTH2, int EPI>
static int launch_small(const SmallArgs& a, hipStream_t s)
{
    if (!a.count || a.count > 32 || a.stride < (a.count + 15) / 16 * 16) {
        return -1;
    }
    if (a.count <= 16) {
        hipLaunchKernelGGL((k_small<K, P, 1, NR, DEPTH1, EPI>), dim3(SMALL_GROUPS), dim3(512), 0,
            s, a);
    } else {
        hipLaunchKernelGGL((k_small<K, P, 2, NR, DEPTH2, EPI>), dim3(SMALL_GROUPS), dim3(512), 0,
            s, a);
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

extern "C" int lh_launch_small_qkv(const uint8_t* W, float sq, float sk, float sv,
    const uint16_t* xs, uint32_t stride, const lh_step_params* params, uint32_t count, float* q,
    float* kcache_layer, float* vcache_layer, uint32_t capacity, hipStream_t s)
{
    SmallArgs a = {};
    a.W = W, a.s0 = sq, a.s1 = sk, a.s2 = sv;
    a.xs = xs, a.stride = stride, a.count = count, a.params = params;
    a.q = q, a.kcache = kcache_layer, a.vcache = vcache_layer, a.capacity = capacity;
    return launch_small<LH_HIDDEN, PLANES_BF16, LH_QKV_ROWS / SMALL_GROUPS, 6, 3, EPI_QKV>(a, s);
}

extern "C" int lh_launch_small_o(const uint8_t* W, float scale, const uint16_t* xs,
    uint32_t stride, const float* head_scale, uint32_t count, float* x, hipStream_t s)
{
    SmallArgs a = {};
    a.W = W, a.s0 = scale, a.xs = xs, a.stride = stride, a.count = count;
    a.wave_scale = head_scale, a.x = x;
    static_assert(LH_KV_HEADS == 8, "one kv head's columns per wave");
    return launch_small<LH_QUERY, PLANES_F16, LH_HIDDEN / SMALL_GROUPS, 8, 4, EPI_RESIDUAL>(a, s);
}

extern "C" int lh_launch_small_gateup(const uint8_t* Wgate, const uint8_t* Wup, float sg, float su,
    const uint16_t* xs, uint32_t stride, const float* row_scale, uint32_t count, uint16_t* planes,
    hipStream_t s)
{
    SmallArgs a = {};
    a.W = Wgate, a.W1 = Wup, a.s0 = sg, a.s1 = su, a.xs = xs, a.stride = stride, a.count = count;
    a.row_scale = row_scale, a.planes = planes;
    return launch_small<LH_HIDDEN, PLANES_F16, 2 * LH_INNER / SMALL_GROUPS, 5, 3, EPI_GATEUP>(a, s);
}

extern "C" int lh_launch_small_down(const uint8_t* W, float scale, const uint16_t* xs,
    uint32_t stride, uint32_t count, float* x, hipStream_t s)
{
    SmallArgs a = {};
    a.W = W, a.s0 = scale, a.xs = xs, a.stride = stride, a.count = count, a.x = x;
    return launch_small<LH_INNER, PLANES_BF16, LH_HIDDEN / SMALL_GROUPS, 6, 3, EPI_RESIDUAL>(a, s);
}
