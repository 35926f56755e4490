// Projections of the precise multi-token path (prefill mode CUSTOM and every
// multi-token call of the resident strategy) on the FP32 matrix
// instructions, bit for bit the canonical row dots of the decode kernels
// (lh_schedule.h).
//
// v_mfma_f32_16x16x1_4b_f32 is four independent 16 x 16 outer products whose
// every element is one correctly rounded fused multiply-add (subnormals kept),
// so a run of them is exactly the canonical chain acc = fma(w, x, acc): block
// b of an instruction holds one lane-chain of the schedule for 16 tokens x 16
// weight rows. The 64 chains of a dot are split over the workgroup's eight
// waves by chain number mod 8: wave s owns chains 8m + s, m = 4g + b, as two
// accumulators g of four blocks b each, so the first three levels of the
// halving tree (distances 32, 16, 8) add inside the wave's registers and the
// last three (4, 2, 1) join the eight waves through LDS.
//
// Activations arrive in the tile order of lh_xt_word (written by the producing
// kernel): a wave's operand for one (chunk, g) is four contiguous 1 KiB loads
// straight to registers, since no other wave of the workgroup reads it. Weight
// rows stay as stored; one stage (16 RT rows x 512 columns, every wave's
// chains of one g) goes to LDS by direct loads of whole row segments, its
// 16-byte words XOR-permuted by row so that the operand reads (16 rows, one
// column word each) are free of bank conflicts. FP8 codes decode in registers
// (v_cvt_pk_f32_fp8, exact). The next stages' loads are in flight while this
// one's 16 RT MFMAs per wave run.
//
// Bound: the FP32 matrix rate (32 products per SIMD and cycle; 59.6 GFLOP of a
// layer's projections at 256 tokens take 0.45 ms at the 2.0 GHz the chip
// holds under this load). Measured there 0.61 ms (65 to 75% of that rate),
// where the row dots it replaces, one token per workgroup, took 3.7 ms (each
// token read and decoded every weight again: 16 TFLOP/s).
#include "lh_attention_blocks.h"
#include "lh_device.h"
#include "lh_internal.h"

namespace lh {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

enum { K_FP8 = 0, K_F32 = 2 };
enum { EPI_RESIDUAL, EPI_QKV, EPI_GATEUP };

struct TileArgs {
    const char* W;         // weight rows (q|k|v, o, gate, down)
    const char* W1;        // up rows (EPI_GATEUP)
    float s0, s1, s2;      // tensor scales (q, k, v; gate, up; or the one scale)
    const f32x4* xt;       // activations, lh_xt_word order
    uint32_t count;        // tokens
    uint32_t tiles;        // row tiles * token tiles
    uint32_t token_tiles;  // ceil(count / 16)
    float* x;              // EPI_RESIDUAL: rows of 3072, updated in place
    const lh_step_params* params;  // EPI_QKV
    float* q;
    float* kcache;
    float* vcache;
    uint32_t capacity;
    f32x4* gated;          // EPI_GATEUP: lh_xt_word order, 9216 columns
};

// The weight rows of a workgroup's 16 RT tile rows n. EPI_RESIDUAL: consecutive
// rows. EPI_QKV: the lower halves of 8 RT consecutive RoPE pairs of one head,
// then their upper halves. EPI_GATEUP: 8 RT gate rows, then the matching up
// rows (of W1). tile_base: the first row; tile_row: row n relative to it, the
// same for every tile.
template <int RT, int EPI>
__device__ __forceinline__ uint32_t tile_base(uint32_t rt)
{
    constexpr uint32_t NP = 8 * RT;
    return EPI == EPI_RESIDUAL ? rt * 16 * RT
        : EPI == EPI_QKV ? (rt * NP >> 6) * 128 + (rt * NP & 63) : rt * NP;
}

template <int RT, int EPI>
__device__ __forceinline__ uint32_t tile_row(uint32_t n)
{
    constexpr uint32_t NP = 8 * RT;
    return EPI == EPI_RESIDUAL || n < NP ? n : n - NP + (EPI == EPI_QKV ? 64 : 0);
}

// Tiles of 16 TT tokens x 16 RT weight rows of a K = 1024 NCH projection.
// Workgroup id (512 threads) takes tiles id, id + gridDim.x, ...; gridDim.x and the
// row tiles are multiples of 8. Tile j's token tiles follow each other on XCD
// j % 8, so a row tile's weights come from HBM once. A tile's first stage is
// requested during the last stages of the tile before it and lands under that
// tile's reduction and epilogue.
template <int KIND, int NCH, int TT, int RT, int EPI>
__device__ __forceinline__ void tile_body(const TileArgs& a)
{
    constexpr uint32_t K = NCH * LH_CHUNK, ES = KIND == K_FP8 ? 1 : 4;
    constexpr uint32_t ROW_WORDS = 512 * ES / 16;       // LDS words of a row's stage
    constexpr uint32_t STAGE_WORDS = 16 * RT * ROW_WORDS;
    constexpr int LOADS = STAGE_WORDS / 512;            // direct loads per wave and stage
    constexpr int WQ = ES;                              // LDS words per lane and (row, chain)
    constexpr uint32_t NP = 8 * RT;
    constexpr uint32_t RS = 16 * RT + 4;                // reduction row stride: no bank conflicts
    // The 2 NCH stages of a tile take NB buffers in turn, a whole number of
    // turns per tile, NB - 1 stages of weights ahead. Three turns do not divide
    // the 8-stage projection. FP32 rows keep to two: with one token tile two
    // workgroups then fit a CU's LDS (74 KB each, 106 KB with three buffers);
    // with more tiles one workgroup runs per CU either way, and a third buffer
    // has not been measured there.
    constexpr int STAGES = 2 * NCH, NB = STAGES % 3 || KIND == K_F32 ? 2 : 3;
    constexpr int UNROLL = 2 * (NB == 3 ? 3 : 1), AHEAD = NB - 1;
    __shared__ u32x4 w0[STAGE_WORDS];
    __shared__ u32x4 w1[STAGE_WORDS];
    __shared__ u32x4 w2[NB == 3 ? STAGE_WORDS : 1];
    __shared__ __attribute__((aligned(16))) float red[8 * 16 * TT * RS];
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t s = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint32_t tile = blockIdx.x, tt, rt;
    // Scalar offsets of the stage loads (the tensors are below 4 GiB).
    const char* const W = EPI == EPI_GATEUP && s >= 4 ? a.W1 : a.W;
    uint32_t src, xsrc[TT];
    // Direct loads: load i of wave s fills LDS words (s * LOADS + i) * 64 + lane,
    // row n = word / ROW_WORDS; LDS word w of row n holds the row's word w ^ (n & 15).
    // Waves 0..3 load the lower half of the rows.
    uint32_t off[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; i++) {
        const uint32_t word = (s * LOADS + i) * 64 + lane;
        const uint32_t n = word / ROW_WORDS, w = word % ROW_WORDS;
        off[i] = tile_row<RT, EPI>(n) * K * ES + 16 * (w ^ (n & 15));
    }
    auto locate = [&](uint32_t j) {
        const uint32_t rest = j >> 3, groups = (a.token_tiles + TT - 1) / TT;
        tt = rest % groups * TT;
        rt = (rest / groups) * 8 + (j & 7);
    };
    auto weights = [&]() { src = tile_base<RT, EPI>(rt) * K * ES; };
    // (A group's token tiles past the last repeat it; their rows lie past count.)
    auto activations = [&]() {
#pragma unroll
        for (int m = 0; m < TT; m++) {
            const uint32_t tile = tt + m < a.token_tiles ? tt + m : a.token_tiles - 1;
            xsrc[m] = (tile * (K >> 9) * 2048 + s * 256) * 16;
        }
    };
    auto load_w = [&](uint32_t stage, u32x4* buf) {
        const char* p = W + __builtin_amdgcn_readfirstlane(src + stage * 512 * ES);
#pragma unroll
        for (int i = 0; i < LOADS; i++) {
            __builtin_amdgcn_global_load_lds(p + off[i], buf + (s * LOADS + i) * 64, 16, 0, 0);
        }
    };
    f32x4 xn[TT][4], xc[TT][4];
    auto load_x = [&](uint32_t stage) {
#pragma unroll
        for (int m = 0; m < TT; m++) {
            const f32x4* p = reinterpret_cast<const f32x4*>(reinterpret_cast<const char*>(a.xt) +
                __builtin_amdgcn_readfirstlane(xsrc[m] + stage * 2048 * 16));
#pragma unroll
            for (int i = 0; i < 4; i++) {
                xn[m][i] = p[i * 64 + lane];
            }
        }
    };
    // Operand words of row tile r: row n = 16 r + lane % 16, chain 8 (lane / 16) + s.
    const uint32_t n16 = lane & 15, wbase = ((lane >> 4) * 8 + s) * WQ;
    f32x16 acc[TT][RT][2];
    auto compute = [&](const u32x4* buf, int g) {
        u32x4 raw[RT][KIND == K_FP8 ? 1 : 4];
#pragma unroll
        for (int r = 0; r < RT; r++) {
#pragma unroll
            for (int i = 0; i < WQ; i++) {
                raw[r][i] = buf[(16 * r + n16) * ROW_WORDS + ((wbase + i) ^ n16)];
            }
        }
        // Columns 4i .. 4i + 3 of the chains, decoded while the four columns
        // before them multiply. The scheduling barriers let only vector and
        // scalar arithmetic cross, so consecutive MFMAs belong to different
        // row tiles and the stage's loads stay where they are issued.
        float w[2][RT][4];
        auto decode = [&](int i) {
#pragma unroll
            for (int r = 0; r < RT; r++) {
                if constexpr (KIND == K_FP8) {
                    fp8x4_to_f32(raw[r][0][i], w[i & 1][r]);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        w[i & 1][r][e] = __uint_as_float(raw[r][i][e]);
                    }
                }
            }
        };
        decode(0);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (i < 3) {
                decode(i + 1);
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
#pragma unroll
                for (int m = 0; m < TT; m++) {
#pragma unroll
                    for (int r = 0; r < RT; r++) {
                        acc[m][r][g] = __builtin_amdgcn_mfma_f32_16x16x1f32(xc[m][i][e],
                            w[i & 1][r][e], acc[m][r][g], 0, 0, 0);
                    }
                }
                __builtin_amdgcn_sched_barrier(0x6);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // Four rows n .. n + 3 of token t of the tile: levels 4, 2 and 1 over the waves.
    auto total4 = [&](uint32_t t, uint32_t n) {
        const f32x4* p = reinterpret_cast<const f32x4*>(red + t * RS + n);
        f32x4 v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            v[i] = p[i * 16 * TT * RS / 4];
        }
        return ((v[0] + v[4]) + (v[2] + v[6])) + ((v[1] + v[5]) + (v[3] + v[7]));
    };
    if (tile >= a.tiles) {
        return;
    }
    locate(tile);
    weights();
    activations();
    load_w(0, w0);
    load_x(0);
    if (AHEAD == 2) {
        load_w(1, w1);
    }
    u32x4* const bufs[3] = {w0, w1, w2};
    while (true) {
#pragma unroll
        for (int m = 0; m < TT; m++) {
#pragma unroll
            for (int r = 0; r < RT; r++) {
                acc[m][r][0] = acc[m][r][1] = f32x16{};
            }
        }
        const uint32_t t0 = tt * 16, n0 = rt;
        const bool more = tile + gridDim.x < a.tiles;
        for (int st = 0; st < STAGES; st += UNROLL) {
#pragma unroll
            for (int u = 0; u < UNROLL; u++) {
                const int k = st + u;
                // Stage k has landed in every wave's part (two ahead, stage
                // k + 1's weight loads, issued last, may be in flight), and
                // every wave has read the buffer of stage k - 1.
                __builtin_amdgcn_s_waitcnt(0x0f70 | (AHEAD == 2 ? LOADS : 0));
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int m = 0; m < TT; m++) {
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        xc[m][i] = xn[m][i];
                    }
                }
                // Stage k + 1's activations, then stage k + AHEAD's weights;
                // past this tile's last stage, the next tile's (the last
                // tile requests its own first stages again, unused).
                if (k + AHEAD == STAGES) {
                    tile = more ? tile + gridDim.x : tile;
                    locate(tile);
                    weights();
                }
                if (k + 1 == STAGES) {
                    activations();
                }
                load_x(k + 1 < STAGES ? k + 1 : 0);
                load_w(k + AHEAD < STAGES ? k + AHEAD : k + AHEAD - STAGES,
                    bufs[(u + AHEAD) % NB]);
                __builtin_amdgcn_sched_barrier(0);
                compute(bufs[u % NB], u & 1);
            }
        }
        // Tree levels 32 (the two accumulators), 16 and 8 (their blocks): lane
        // holds tokens 4 (lane / 16) + k, row lane % 16 of each row tile.
#pragma unroll
        for (int m = 0; m < TT; m++) {
#pragma unroll
            for (int r = 0; r < RT; r++) {
                const f32x16 v = acc[m][r][0] + acc[m][r][1];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    red[((s * TT + m) * 16 + 4 * (lane >> 4) + k) * RS + 16 * r + n16] =
                        (v[k] + v[8 + k]) + (v[4 + k] + v[12 + k]);
                }
            }
        }
        // LDS only: the next tile's first stage stays in flight.
        __builtin_amdgcn_s_waitcnt(0xc07f);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if constexpr (EPI == EPI_RESIDUAL) {
            const uint32_t tl = tid / (4 * RT), n = tid % (4 * RT) * 4, t = t0 + tl;
            if (tid < 64 * RT * TT && t < a.count) {
                f32x4* px = reinterpret_cast<f32x4*>(a.x + (size_t)t * LH_HIDDEN +
                    n0 * 16 * RT + n);
                const f32x4 old = *px, v = total4(tl, n);
                *px = old + v * a.s0;
            }
        } else if constexpr (EPI == EPI_QKV) {
            const uint32_t tl = tid / (2 * RT), n = tid % (2 * RT) * 4, t = t0 + tl;
            if (tid < 32 * RT * TT && t < a.count) {
                const uint32_t pair = n0 * NP + n, head = pair >> 6, i = pair & 63;
                const float scale = head < 32 ? a.s0 : (head < 40 ? a.s1 : a.s2);
                const f32x4 lo = total4(tl, n) * scale, hi = total4(tl, n + NP) * scale;
                const lh_token_params* tp = &a.params->tokens[t];
                const uint32_t position = a.params->length + t;
                if (head < 40) {
                    // column i < 64 rotates with -x[i+64]; column i+64 with x[i].
                    const f32x4 cl = *reinterpret_cast<const f32x4*>(tp->cosine + i);
                    const f32x4 sl = *reinterpret_cast<const f32x4*>(tp->sine + i);
                    const f32x4 ch = *reinterpret_cast<const f32x4*>(tp->cosine + i + 64);
                    const f32x4 sh = *reinterpret_cast<const f32x4*>(tp->sine + i + 64);
                    f32x4 out_lo = lo * cl + (-hi) * sl;
                    f32x4 out_hi = hi * ch + lo * sh;
                    if (head < 32) {
                        f32x4* qh = reinterpret_cast<f32x4*>(a.q + (size_t)t * LH_QUERY +
                            head * 128 + i);
                        qh[0] = out_lo * tp->qfactor;
                        qh[16] = out_hi * tp->qfactor;
                    } else {
                        *reinterpret_cast<f32x4*>(a.kcache +
                            lh_k_index(a.capacity, 0, head - 32, position, i)) = out_lo;
                        *reinterpret_cast<f32x4*>(a.kcache +
                            lh_k_index(a.capacity, 0, head - 32, position, i + 64)) = out_hi;
                    }
                } else {
                    f32x4* vr = reinterpret_cast<f32x4*>(a.vcache +
                        lh_kv_index(a.capacity, 0, head - 40, position) + i);
                    vr[0] = lo;
                    vr[16] = hi;
                }
            }
        } else {
            // One word of the next projection's tile order per thread. Rows
            // past count are written too (their products are never stored).
            const uint32_t tl = tid % (16 * TT), n = tid / (16 * TT) * 4;
            if (tid < 32 * RT * TT && t0 + tl < a.token_tiles * 16) {
                const f32x4 g = total4(tl, n) * a.s0, u = total4(tl, n + NP) * a.s1;
                f32x4 y;
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    y[k] = silu(g[k]) * u[k];
                }
                a.gated[lh_xt_word(t0 + tl, n0 * NP + n, LH_INNER)] = y;
            }
        }
        if (!more) {
            // The unused direct loads land before the LDS is given back.
            __builtin_amdgcn_s_waitcnt(0);
            return;
        }
    }
}

// (The body is device code only: the host pass has no matrix instructions.)
template <int KIND, int NCH, int TT, int RT, int EPI>
__global__ void __launch_bounds__(512, TT == 1 ? 4 : 2)
k_tile(TileArgs a)
{
#ifdef __HIP_DEVICE_COMPILE__
    tile_body<KIND, NCH, TT, RT, EPI>(a);
#endif
}

// Canonical RMSNorm of a 3072-wide row per workgroup, written in the tile
// order of the next projection. grid (count), block 768: thread i owns columns
// 4i .. 4i+3.
__global__ void __launch_bounds__(768)
k_norm_tile(const float* __restrict__ x, const float* __restrict__ gamma, f32x4* __restrict__ xt)
{
    // Lane l's 16 values of chunk c (columns c*1024 + 16l .. +15) are words
    // (4c + q)*64 + l.
    __shared__ f32x4 row_l[LH_HIDDEN / 4];
    __shared__ float r_s;
    const uint32_t t = blockIdx.x, tid = threadIdx.x;
    const f32x4 g = reinterpret_cast<const f32x4*>(gamma)[tid];
    const f32x4 v = reinterpret_cast<const f32x4*>(x + (size_t)t * LH_HIDDEN)[tid];
    const uint32_t c = tid >> 8, w = tid & 255;
    row_l[(4 * c + (w & 3)) * 64 + (w >> 2)] = v;
    __syncthreads();
    if (tid < 64) {
        float acc = 0.0f;
#pragma unroll
        for (int k = 0; k < LH_HIDDEN / 256; k++) {
            const f32x4 u = row_l[k * 64 + tid];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                acc = __builtin_fmaf(u[e], u[e], acc);
            }
        }
        const float ss = wave_tree64(acc);
        if (tid == 0) {
            r_s = 1.0f / __builtin_sqrtf(ss / (float)LH_HIDDEN + 1e-5f);
        }
    }
    __syncthreads();
    const float r = r_s;
    f32x4 y;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        y[e] = g[e] * (v[e] * r);
    }
    xt[lh_xt_word(t, 4 * tid, LH_HIDDEN)] = y;
}

// The attention block partials of several tokens at once, bit for bit those of
// attn_block (lh_attention_blocks.h). The 4 query heads of a kv head times 4
// tokens are the 16 columns (query rows) of the products, one tile per wave.
//   Scores, transposed: v_mfma_f32_16x16x1_4b with A = K (16 positions) and
// B = Q; block c of the instruction is the chain c_c over dims 32c .. 32c + 31.
// Lane l then holds, for query row l % 16, positions 16 pt + 4 (l / 16) + r.
//   The maximum and the 64-position tree run over the lane's registers and
// the four lane groups; a 4 x 4 transpose of registers and lane groups
// (v_permlane32_swap, v_permlane16_swap) puts positions 4 st .. 4 st + 3 into
// the lane groups of register st, in position order.
//   P.V, transposed: v_mfma_f32_16x16x4_f32, whose four products add one after
// the other, each rounded (k ascending), with A = V columns, B = P: the
// canonical chain over the positions.
// K and V come by direct loads to LDS, shared by the workgroup's four waves; the
// next block's K is requested after the scores, its V after the chains.
// Masked positions (past a token's own) carry e = 0: their products add +-0,
// which can only turn a -0 sum into +0, and the combine's chain from +0 gives
// the same bits for both. A nonfinite V among them would not be neutral: such
// a block redoes its chains without them.
// Bound: FP32 matrix instructions, 8192 cycles per wave and block: 256 tokens
// after 4096 positions are 17.6 GFLOP, 0.13 ms at 2 GHz, and write 285 MB of
// partials. Measured there 0.24 ms (0.76 ms with one token per workgroup,
// k_attn_blocks) plus 0.04 ms for the combine, which reads the partials back;
// 37 tokens after 777: 19 us plus 5 (30 and 5).
//
// grid 8 * query groups * ranges, block 256: id = (range * groups + group) * 8 +
// kv head; a group is 16 tokens, a range `per` consecutive blocks.
__global__ void __launch_bounds__(256, 2)
k_attn_tiles(const float* __restrict__ q, const float* __restrict__ kcache,
    const float* __restrict__ vcache, uint32_t length, uint32_t count, uint32_t capacity,
    uint32_t groups, uint32_t per, float* __restrict__ PM, float* __restrict__ PT,
    float* __restrict__ PA)
{
#ifdef __HIP_DEVICE_COMPILE__
    constexpr uint32_t WORDS = LH_ATTN_BLOCK * LH_HEAD_DIM / 4;
    __shared__ f32x4 ks[WORDS];
    __shared__ f32x4 vs[WORDS];
    const uint32_t kvh = blockIdx.x & 7, rest = blockIdx.x >> 3;
    const uint32_t group = rest % groups, range = rest / groups;
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t col = lane & 15, lg = lane >> 4;
    // Blocks of this workgroup: up to its last token's position.
    const uint32_t last = group * 16 + 15 < count ? group * 16 + 15 : count - 1;
    const uint32_t need = (length + last) / LH_ATTN_BLOCK + 1;
    const uint32_t b0 = range * per, b1 = b0 + per < need ? b0 + per : need;
    if (b0 >= b1) {
        return;
    }
    // Query row col: token t, head kvh * 4 + col % 4; rows past count repeat
    // the last token, whose bits they store once more. A row also stores the
    // partials of its group's blocks past its own last position, which no
    // combine reads: every store is issued by every wave, so the waits below
    // can count them.
    const uint32_t tr = group * 16 + wave * 4 + (col >> 2), t = tr < count ? tr : count - 1;
    const uint32_t n = length + t + 1;   // positions the row attends
    const uint32_t nbc = capacity / LH_ATTN_BLOCK;
    const size_t th = (size_t)t * LH_HEADS + kvh * 4 + (col & 3);
    const float* const kh = kcache + lh_kv_index(capacity, 0, kvh, 0);
    const float* const vh = vcache + lh_kv_index(capacity, 0, kvh, 0);
    // K: LDS word (8 pt + i) * 64 + l holds dims 32 (l / 16) + 4i .. + 3 of position
    // 16 pt + l % 16 (the tile's words in lane order). V: rows as they are.
    auto load_k = [&](uint32_t b) {
        const f32x4* p = reinterpret_cast<const f32x4*>(kh + (size_t)b * 64 * LH_HEAD_DIM) +
            wave * 512 + col * 4 + lg;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            __builtin_amdgcn_global_load_lds(p + i * 64, ks + (wave * 8 + i) * 64, 16, 0, 0);
        }
    };
    auto load_v = [&](uint32_t b) {
        const f32x4* p = reinterpret_cast<const f32x4*>(vh + (size_t)b * 64 * LH_HEAD_DIM) +
            wave * 512 + lane;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            __builtin_amdgcn_global_load_lds(p + i * 64, vs + (wave * 8 + i) * 64, 16, 0, 0);
        }
    };
    f32x4 qr[8];
    const f32x4* qp = reinterpret_cast<const f32x4*>(q + th * LH_HEAD_DIM) + lg * 8;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        qr[i] = qp[i];
    }
    load_k(b0);
    load_v(b0);
    __builtin_amdgcn_s_waitcnt(0);
    // Barrier after this wave's LDS reads; direct loads stay in flight.
    auto sync = [&]() {
        __builtin_amdgcn_s_waitcnt(0xc07f);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    auto swap32 = [](float& a, float& b) {   // a's lanes 32..63 <-> b's lanes 0..31
        const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b),
            false, false);
        a = __uint_as_float(s[0]);
        b = __uint_as_float(s[1]);
    };
    auto swap16 = [](float& a, float& b) {   // a's odd rows <-> b's even rows
        const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b),
            false, false);
        a = __uint_as_float(s[0]);
        b = __uint_as_float(s[1]);
    };
    for (uint32_t b = b0; b < b1; b++) {
        const uint32_t first = b * LH_ATTN_BLOCK;
        const bool whole = first + LH_ATTN_BLOCK <= length + 1;   // for every token
        const uint32_t valid = n > first ? (n - first < 64 ? n - first : 64) : 0;
        // K has landed; V's eight loads and the ten stores of the block
        // before, issued after it, may be in flight.
        __builtin_amdgcn_s_waitcnt(0x4f72);
        sync();
        float e[4][4];
#pragma unroll
        for (int pt = 0; pt < 4; pt += 2) {
            f32x16 c0 = {}, c1 = {};
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const f32x4 k0 = ks[(pt * 8 + i) * 64 + lane];
                const f32x4 k1 = ks[(pt * 8 + 8 + i) * 64 + lane];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    c0 = __builtin_amdgcn_mfma_f32_16x16x1f32(k0[j], qr[i][j], c0, 0, 0, 0);
                    c1 = __builtin_amdgcn_mfma_f32_16x16x1f32(k1[j], qr[i][j], c1, 0, 0, 0);
                }
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                e[pt][r] = ((c0[r] + c0[4 + r]) + (c0[8 + r] + c0[12 + r])) * LH_SCORE_SCALE;
                e[pt + 1][r] = ((c1[r] + c1[4 + r]) + (c1[8 + r] + c1[12 + r])) * LH_SCORE_SCALE;
            }
        }
        sync();   // every wave has read K
        // (The last block requests itself again, unused.)
        const uint32_t next = b + 1 < b1 ? b + 1 : b;
        load_k(next);
        __builtin_amdgcn_sched_barrier(0);
        if (!whole) {
#pragma unroll
            for (int pt = 0; pt < 4; pt++) {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    if (16 * pt + 4 * lg + r >= valid) {
                        e[pt][r] = -__builtin_inff();
                    }
                }
            }
        }
        float m = e[0][0];
#pragma unroll
        for (int i = 1; i < 16; i++) {
            m = fmaxf(m, e[i >> 2][i & 3]);
        }
        float x = m, y = m;
        swap32(x, y);
        m = fmaxf(x, y);
        x = m, y = m;
        swap16(x, y);
        m = fmaxf(x, y);
#pragma unroll
        for (int pt = 0; pt < 4; pt++) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float v = expf_flat(e[pt][r] - m);
                e[pt][r] = whole || 16 * pt + 4 * lg + r < valid ? v : 0.0f;
            }
        }
        // T_b: the halving tree over positions (32, 16 by pt; 8, 4 by lane
        // group; 2, 1 by register).
        float u[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            u[r] = (e[0][r] + e[2][r]) + (e[1][r] + e[3][r]);
            x = u[r], y = u[r];
            swap32(x, y);
            u[r] = x + y;
            x = u[r], y = u[r];
            swap16(x, y);
            u[r] = x + y;
        }
        const float total = (u[0] + u[2]) + (u[1] + u[3]);
        // Register e[pt][a] of lane group k: position 16 pt + 4a + k.
#pragma unroll
        for (int pt = 0; pt < 4; pt++) {
            swap32(e[pt][0], e[pt][2]);
            swap32(e[pt][1], e[pt][3]);
            swap16(e[pt][0], e[pt][1]);
            swap16(e[pt][2], e[pt][3]);
        }
        // V has landed; the ten stores and the next K may be in flight.
        __builtin_amdgcn_s_waitcnt(0x4f72);
        sync();
        // A operand row i of tile (h, j): dim 64h + 4 ((i % 4) * 4 + i / 4) + j, so
        // that a lane's results for fixed (h, r) are words 4r + lg: contiguous
        // over the lane groups.
        const uint32_t vw = (col & 3) * 4 + (col >> 2);
        f32x4 o[2][4];
#pragma unroll
        for (int h = 0; h < 2; h++) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                o[h][j] = f32x4{};
            }
        }
        bool redo = false;
        if (whole) {
#pragma unroll
            for (int st = 0; st < 16; st++) {
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const f32x4 v = vs[(4 * st + lg) * 32 + 16 * h + vw];
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        o[h][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[j], e[st >> 2][st & 3],
                            o[h][j], 0, 0, 0);
                    }
                }
            }
        } else {
            // Rows past the call's last token are stale: they enter as 0.
            const uint32_t live = length + count - first;
#pragma unroll
            for (int st = 0; st < 16; st++) {
                const uint32_t p = 4 * st + lg;
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const f32x4 v = vs[p * 32 + 16 * h + vw];
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const float vj = p < live ? v[j] : 0.0f;
                        redo = redo || (__float_as_uint(vj) & 0x7f800000u) == 0x7f800000u;
                        o[h][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(vj, e[st >> 2][st & 3],
                            o[h][j], 0, 0, 0);
                    }
                }
            }
            if (__builtin_amdgcn_ballot_w64(redo)) {
                // The chains over the row's own positions only.
#pragma unroll
                for (int h = 0; h < 2; h++) {
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        o[h][j] = f32x4{};
                    }
                }
#pragma unroll
                for (int st = 0; st < 16; st++) {
#pragma unroll 1
                    for (uint32_t k = 0; k < 4; k++) {
                        const uint32_t p = 4 * st + k;
                        const float ep = __int_as_float(__builtin_amdgcn_ds_bpermute(
                            4 * (16 * k + col), __float_as_int(e[st >> 2][st & 3])));
#pragma unroll
                        for (int h = 0; h < 2; h++) {
#pragma unroll
                            for (int r = 0; r < 4; r++) {
                                const f32x4 v = vs[p * 32 + 16 * h + 4 * r + lg];
#pragma unroll
                                for (int j = 0; j < 4; j++) {
                                    o[h][j][r] = p < valid
                                        ? __builtin_fmaf(ep, v[j], o[h][j][r]) : o[h][j][r];
                                }
                            }
                        }
                    }
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        sync();   // every wave has read V
        load_v(next);
        __builtin_amdgcn_sched_barrier(0);
        float* const pa = PA + (th * nbc + b) * LH_HEAD_DIM;
#pragma unroll
        for (int h = 0; h < 2; h++) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                reinterpret_cast<f32x4*>(pa)[16 * h + 4 * r + lg] =
                    f32x4{o[h][0][r], o[h][1][r], o[h][2][r], o[h][3][r]};
            }
        }
        PM[th * nbc + b] = m;
        PT[th * nbc + b] = total;
    }
    // The unused direct loads land before the LDS is given back.
    __builtin_amdgcn_s_waitcnt(0);
#endif
}

// The combine of the block partials above, operation for operation that of
// attn_combine, into the o projection's tile order. The length comes with the
// launch, so only the valid blocks are read, and a workgroup takes a whole
// head: thread (c = tid % 32, s = tid / 32) owns dims 4c .. 4c + 3 of group s of
// each 64-block round. grid (32 heads, count), block 256. Bound: latency, and
// from about 100 MB of partials HBM. Four workgroups per head (attn_combine's
// dimension quarters) took 10.3 us for 48 tokens after 517 positions and 58 us for
// 256 after 4096, this 5.6 and 43 us (6.6 TB/s).
__global__ void __launch_bounds__(256)
k_combine_tiles(const float* __restrict__ PM, const float* __restrict__ PT,
    const float* __restrict__ PA, uint32_t length, uint32_t capacity, f32x4* __restrict__ xt)
{
    constexpr uint32_t GROUPS = 8, STEP = GROUPS * GROUP;   // blocks per round
    __shared__ float wmax[4], fs[STEP], ts[STEP], ug[GROUPS];
    __shared__ f32x4 sg[GROUPS][32];
    const uint32_t h = blockIdx.x, t = blockIdx.y, tid = threadIdx.x, c = tid & 31, s = tid >> 5;
    const uint32_t nb = (length + t) / LH_ATTN_BLOCK + 1, nbc = capacity / LH_ATTN_BLOCK;
    const size_t th = (size_t)t * LH_HEADS + h;
    const float* pm = PM + th * nbc;
    const float* pt = PT + th * nbc;
    const f32x4* pa = reinterpret_cast<const f32x4*>(PA + th * nbc * LH_HEAD_DIM) + c;
    f32x4 a[GROUP];
    float tb = 0.0f;
    // Rows past the valid blocks repeat the last one and enter no arithmetic.
    auto load_round = [&](uint32_t r0) {
#pragma unroll
        for (uint32_t k = 0; k < GROUP; k++) {
            const uint32_t b = r0 + s * GROUP + k;
            a[k] = pa[(size_t)(b < nb ? b : nb - 1) * (LH_HEAD_DIM / 4)];
        }
        if (tid < STEP) {
            tb = pt[r0 + tid < nb ? r0 + tid : nb - 1];
        }
    };
    load_round(0);
    float M = -__builtin_inff();
    for (uint32_t b = tid; b < nb; b += 256) {
        M = fmaxf(M, pm[b]);
    }
    M = wave_max64(M);
    if ((tid & 63) == 0) {
        wmax[tid >> 6] = M;
    }
    __syncthreads();
    M = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
    f32x4 A = {};
    float T = 0.0f;
    for (uint32_t r0 = 0; r0 < nb; r0 += STEP) {
        if (r0) {
            load_round(r0);
        }
        if (tid < STEP) {
            const uint32_t b = r0 + tid;
            fs[tid] = b < nb ? expf_cw(pm[b] - M) : 0.0f;
            ts[tid] = b < nb ? tb : 0.0f;
        }
        __syncthreads();
        f32x4 S = {};
        float U = 0.0f;
#pragma unroll
        for (uint32_t k = 0; k < GROUP; k++) {
            if (r0 + s * GROUP + k < nb) {
                const float f = fs[s * GROUP + k];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    S[e] = __builtin_fmaf(f, a[k][e], S[e]);
                }
                U = __builtin_fmaf(f, ts[s * GROUP + k], U);
            }
        }
        sg[s][c] = S;
        if (c == 0) {
            ug[s] = U;
        }
        __syncthreads();
        if (tid < 32) {
            for (uint32_t g = 0; g < GROUPS && r0 + g * GROUP < nb; g++) {
                A = r0 + g ? A + sg[g][c] : sg[g][c];
                T = r0 + g ? T + ug[g] : ug[g];
            }
        }
        __syncthreads();
    }
    if (tid < 32) {
        xt[lh_xt_word(t, h * LH_HEAD_DIM + 4 * c, LH_QUERY)] = f32x4{A[0] / T, A[1] / T, A[2] / T,
            A[3] / T};
    }
}

}  // namespace lh

using namespace lh;

static int launched()
{
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// One token tile per workgroup: two workgroups fit a CU (128 registers, at most
// 76 KB of LDS); more: one.
template <int KIND, int NCH, int TT, int RT, int EPI>
static void launch_tile(uint32_t rows, TileArgs a, hipStream_t s)
{
    a.tiles = rows / (16 * RT) * ((a.token_tiles + TT - 1) / TT);
    const uint32_t resident = TT == 1 ? 512 : 256;
    hipLaunchKernelGGL((k_tile<KIND, NCH, TT, RT, EPI>),
        dim3(a.tiles < resident ? a.tiles : resident), dim3(512), 0, s, a);
}

// FP8 projections take two row tiles per workgroup where that leaves no CU
// with more of them than single ones would (the CU with the most work holds
// ceil(workgroups / 256) workgroups): at 256 tokens 0.61 ms a layer against
// 0.66 ms with one, at 16 tokens 77 against 62 us. Four per workgroup (one
// resident per CU) measured the same as two at 256 tokens and worse below; two
// or three token tiles instead were slower (37 tokens: 183 against 172 us).
// FP32 rows, four times as large, take one row tile and up to three token
// tiles, which then share one read of the rows (layers after 517 positions of 24,
// 48, 64 and 90 tokens: 198, 254, 308, 408 us with one token tile, 186, 228, 290,
// 368 us so).
template <int KIND, int NCH, int EPI>
static int run_tile(uint32_t rows, const TileArgs& a, hipStream_t s)
{
    if constexpr (KIND == K_FP8) {
        const uint32_t single = rows / 16 * a.token_tiles;
        if ((single / 2 + 255) / 256 * 2 <= (single + 255) / 256) {
            launch_tile<KIND, NCH, 1, 2, EPI>(rows, a, s);
        } else {
            launch_tile<KIND, NCH, 1, 1, EPI>(rows, a, s);
        }
    } else if (a.token_tiles == 1) {
        launch_tile<KIND, NCH, 1, 1, EPI>(rows, a, s);
    } else if (a.token_tiles % 3) {
        launch_tile<KIND, NCH, 2, 1, EPI>(rows, a, s);
    } else {
        launch_tile<KIND, NCH, 3, 1, EPI>(rows, a, s);
    }
    return launched();
}

extern "C" int lh_launch_norm_tile(const float* x, const float* gamma, float* xt, uint32_t count,
    hipStream_t s)
{
    hipLaunchKernelGGL(k_norm_tile, dim3(count), dim3(768), 0, s, x, gamma,
        reinterpret_cast<f32x4*>(xt));
    return launched();
}

// Ranges: the query groups of the 8 kv heads times the ranges fill the 512
// workgroups that two per CU (64 KB of LDS each) hold at once.
extern "C" int lh_launch_attention_tiles(const float* q, const float* kcache_layer,
    const float* vcache_layer, uint32_t length, uint32_t count, uint32_t capacity, float* PM,
    float* PT, float* PA, float* xt, hipStream_t s)
{
    if (!count || capacity % LH_ATTN_BLOCK || length + count > capacity) {
        return -1;
    }
    const uint32_t groups = (count + 15) / 16, nblk = lh_attention_blocks(length, count);
    const uint32_t ranges = groups < 64 ? 64 / groups : 1, per = (nblk + ranges - 1) / ranges;
    hipLaunchKernelGGL(k_attn_tiles, dim3(8 * groups * ((nblk + per - 1) / per)), dim3(256), 0, s,
        q, kcache_layer, vcache_layer, length, count, capacity, groups, per, PM, PT, PA);
    if (launched()) {
        return -1;
    }
    hipLaunchKernelGGL(k_combine_tiles, dim3(LH_HEADS, count), dim3(256), 0, s, PM, PT, PA, length,
        capacity, reinterpret_cast<f32x4*>(xt));
    return launched();
}

extern "C" int lh_launch_qkv_tile(int resident, const void* Wqkv, float sq, float sk, float sv,
    const float* xt, const lh_step_params* params, uint32_t count, float* q, float* kcache_layer,
    float* vcache_layer, uint32_t capacity, hipStream_t s)
{
    TileArgs a = {};
    a.W = static_cast<const char*>(Wqkv);
    a.s0 = sq, a.s1 = sk, a.s2 = sv;
    a.xt = reinterpret_cast<const f32x4*>(xt);
    a.count = count, a.token_tiles = (count + 15) / 16;
    a.params = params, a.q = q, a.kcache = kcache_layer, a.vcache = vcache_layer;
    a.capacity = capacity;
    return resident ? run_tile<K_F32, 3, EPI_QKV>(LH_QKV_ROWS, a, s)
                    : run_tile<K_FP8, 3, EPI_QKV>(LH_QKV_ROWS, a, s);
}

extern "C" int lh_launch_gateup_tile(int resident, const void* Wgate, const void* Wup, float sg,
    float su, const float* xt, uint32_t count, float* gated_xt, hipStream_t s)
{
    TileArgs a = {};
    a.W = static_cast<const char*>(Wgate), a.W1 = static_cast<const char*>(Wup);
    a.s0 = sg, a.s1 = su;
    a.xt = reinterpret_cast<const f32x4*>(xt);
    a.count = count, a.token_tiles = (count + 15) / 16;
    a.gated = reinterpret_cast<f32x4*>(gated_xt);
    return resident ? run_tile<K_F32, 3, EPI_GATEUP>(2 * LH_INNER, a, s)
                    : run_tile<K_FP8, 3, EPI_GATEUP>(2 * LH_INNER, a, s);
}

extern "C" int lh_launch_residual_tile(int resident, const void* W, float scale, uint32_t cols,
    const float* xt, uint32_t count, float* x, hipStream_t s)
{
    TileArgs a = {};
    a.W = static_cast<const char*>(W);
    a.s0 = scale;
    a.xt = reinterpret_cast<const f32x4*>(xt);
    a.count = count, a.token_tiles = (count + 15) / 16;
    a.x = x;
    if (cols == LH_QUERY) {
        return resident ? run_tile<K_F32, 4, EPI_RESIDUAL>(LH_HIDDEN, a, s)
                        : run_tile<K_FP8, 4, EPI_RESIDUAL>(LH_HIDDEN, a, s);
    }
    if (cols == LH_INNER) {
        return resident ? run_tile<K_F32, 9, EPI_RESIDUAL>(LH_HIDDEN, a, s)
                        : run_tile<K_FP8, 9, EPI_RESIDUAL>(LH_HIDDEN, a, s);
    }
    return -1;
}
