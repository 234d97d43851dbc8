// Dense layer for some tens to some hundreds of tokens:  C[token, feature] = act(X[token, :] . W[:, feature] + bias).
// X is [tokens, K] row-major; W is [features, K] for 2-byte weights and [K, features] for 4-byte weights (the layouts
// the models keep, contiguous 128-byte pieces either way).
//
// What bounds it: a launch of this size moves a few MB and multiplies for 1-5 us, so its time is the chain dispatch ->
// first operands from the Infinity Cache (about 2 us) -> the rest of a compute unit's operands -> hand-over, and what
// shortens it is operands requested early, in whole cache lines, by every compute unit.  Hence:
//   - a workgroup of four wavefronts owns a tile of TM tokens x TN features; the wavefronts share the K axis, not the
//     tile: each walks every fourth 128-byte step of K through LDS of its own, so nothing in the main loop waits for
//     another wavefront, and the four partial tiles meet in LDS once at the end (in wavefront order);
//   - operands go from memory straight to LDS (16 bytes per lane, eight lanes per 128-byte row piece, DEPTH steps
//     requested ahead), laid out so that the matrix-core operand reads hit all banks: the 16-byte unit u of row r
//     sits at u ^ (r / 2 % 8) (two rows span the 64 banks), which the loads get by asking for permuted units;
//   - K can also be cut into slices over workgroups when the consumer adds them (LayerNorm over slices);
//   - fp32 layers of more than 64 tokens come as rows of pairs of fp16 numbers (split.hip): as many bytes, and three products of 32
//     cycles for 16 values of K where fp32 operands take eight of 64, which is most of an fp32 launch (768 -> 3072 with GELU, 120
//     tokens 12.2 -> 8.0 us, 300 18.7 -> 10.8; 3072 -> 768 with its LayerNorm, 300 30 -> 15.1), in shorter sums (error against
//     float64 2.5e-7 -> 1.3e-7 of the 2-norm at 768 inputs, in slices 1.8e-7 -> 1.1e-7).
#include <type_traits>

#include "activations.h"
#include "cubert_kernels.h"
#include "device_common.h"

namespace cubert {
namespace {

typedef float v16f32 __attribute__((ext_vector_type(16)));
typedef float v4f32 __attribute__((ext_vector_type(4)));
typedef _Float16 v8f16 __attribute__((ext_vector_type(8)));

constexpr int kMidWaves = 4;
constexpr int kMidThreads = kMidWaves * kWave;
constexpr int kStepBytes = 128;  // of a row of X that a wavefront consumes per step

// What a kernel reads and what it stores: T and T, or, for fp32 layers on the fp16 matrix cores, rows of pairs (split.hip: for every
// 32 values of K their 32 high and their 32 low terms, a step) on both sides and floats.
struct Pairs {};
template <typename T>
struct MidTypes { typedef T Operand, Value; };
template <>
struct MidTypes<Pairs> { typedef half_t Operand; typedef float Value; };
template <typename T>
constexpr bool is_pairs() { return std::is_same<T, Pairs>::value; }
// K values per step: 128 bytes of a row of X
template <typename T>
constexpr int mid_step() { return kStepBytes / (is_pairs<T>() ? 4 : (int) sizeof(typename MidTypes<T>::Operand)); }

template <int TM, int TN, int DEPTH>
struct MidShape {
    static constexpr int kXBytes = TM * kStepBytes;                // of one step in LDS
    static constexpr int kWBytes = TN * kStepBytes;                // the same size in either weight layout
    static constexpr int kStageBytes = kXBytes + kWBytes;
    static constexpr int kLoads = kStageBytes / 1024;              // requests per lane and step
    static constexpr int kRedPitch = TN + 4;                       // floats between token rows of a partial tile
    static constexpr int kWaveBytes = DEPTH * kStageBytes > TM * kRedPitch * 4 ? DEPTH * kStageBytes : TM * kRedPitch * 4;
    static constexpr int kLdsBytes = kMidWaves * kWaveBytes;
};

enum MidOutput { kMidStore = 0, kMidGelu = 1, kMidSlices = 2 };

// CHAINS (a power of two; pairs: 2 or 3, see there) accumulators per block take turns over a wavefront's K values and are added at the end: a
// single fp32 chain over 192 of 768 K values has 2.5e-7 relative error against float64 (the library's GEMM 2.5e-7 to
// 5.0e-7), eight 1.1e-7 (with K slices 0.9e-7; the few-token kernel, which adds runs of 16 values, 1.1e-7), for 0.2 to
// 0.5 us a launch.
template <typename T, int TM, int TN, int DEPTH, int OUT, int CHAINS>
__global__ __launch_bounds__(kMidThreads) void dense_mid_kernel(
        const typename MidTypes<T>::Operand *__restrict__ W, int ldw, const typename MidTypes<T>::Operand *__restrict__ X, int ldx,
        const typename MidTypes<T>::Value *__restrict__ bias, typename MidTypes<T>::Value *__restrict__ C, int ldc, int tokens,
        int features, int steps_total, int steps_per_slice, int token_tiles, int feature_tiles, float *__restrict__ partials,
        int pitch, long long slice_stride, float alpha, float scale, int *__restrict__ overflow) {
    static_assert(DEPTH == 1 || DEPTH == 2, "steps requested ahead");
    typedef MidShape<TM, TN, DEPTH> S;
    typedef typename MidTypes<T>::Operand Operand;
    typedef typename MidTypes<T>::Value Value;
    constexpr int FB = TN / 32, TB = TM / 32;  // 32 x 32 blocks of the tile
    constexpr int U = 16 / sizeof(Operand);    // elements of a 16-byte unit
    constexpr int kRowStep = kStepBytes / sizeof(Operand);  // elements of a row per step
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & (kWave - 1), wave = wave_in_block();
    const int r = lane & 31, hh = lane >> 5;

    // Workgroups are handed to the eight dies in turn.  Each die gets a contiguous run of the (slice, feature tile, token
    // tile) triples, token tiles innermost: the token tiles of a feature tile mostly share a die, so its weights come to
    // that die's L2 once, and no die gets more than one workgroup more than another.  (Feature tiles dealt out to the dies
    // one by one: 12 of them over 8 dies, 7 slices, put 42 workgroups on the 32 compute units of four dies.)
    const int die = blockIdx.x & 7, die_share = gridDim.x >> 3, extra = gridDim.x & 7;
    const int index = die * die_share + (die < extra ? die : extra) + (int) (blockIdx.x >> 3);
    const int pair = index / token_tiles, tt = index - pair * token_tiles;
    const int slice = pair / feature_tiles, ft = pair - slice * feature_tiles;
    const int m0 = tt * TM, n0 = ft * TN;
    const int s_begin = slice * steps_per_slice;
    const int s_end = s_begin + steps_per_slice < steps_total ? s_begin + steps_per_slice : steps_total;
    const int steps = s_end - s_begin > wave ? (s_end - s_begin - wave + kMidWaves - 1) / kMidWaves : 0;

    unsigned char *mine = smem + wave * S::kWaveBytes;

    // lane l of request i brings the 16-byte unit l % 8 of the LDS row 8 i + l / 8; rows past the end are read from the last
    const int lrow = lane >> 3;
    auto unit_of = [&](int i) { return ((lane & 7) ^ (((i * 8 + lrow) >> 1) & 7)) * U; };
    const Operand *xsrc[TM / 8], *wsrc[TN / 8];
    const int k_first = (s_begin + wave) * kRowStep;
#pragma unroll
    for (int i = 0; i < TM / 8; ++i) {
        const int row = m0 + i * 8 + lrow;
        xsrc[i] = X + (size_t) (row < tokens ? row : tokens - 1) * ldx + k_first + unit_of(i);
    }
    size_t w_advance;
    if constexpr (sizeof(Operand) == 2) {
        w_advance = kMidWaves * kRowStep;
#pragma unroll
        for (int i = 0; i < TN / 8; ++i) {
            const int row = n0 + i * 8 + lrow;
            wsrc[i] = W + (size_t) (row < features ? row : features - 1) * ldw + k_first + unit_of(i);
        }
    } else {
        // [K, features]: the 32 K values of a step are LDS rows of TN features; lane l brings 4 features
        constexpr int kLanes = TN / 4, kRows = kWave / kLanes;
        w_advance = (size_t) kMidWaves * kRowStep * ldw;
        const int f = n0 + (lane % kLanes) * 4;
#pragma unroll
        for (int i = 0; i < TN / 8; ++i) {
            wsrc[i] = W + (size_t) (k_first + i * kRows + lane / kLanes) * ldw + (f < features ? f : features - 4);
        }
    }

    auto request = [&](int slot) {
        unsigned char *stage = mine + slot * S::kStageBytes;
#pragma unroll
        for (int i = 0; i < TN / 8; ++i) {
            load_to_lds(wsrc[i], stage + S::kXBytes + i * 1024);
            wsrc[i] += w_advance;
        }
#pragma unroll
        for (int i = 0; i < TM / 8; ++i) {
            load_to_lds(xsrc[i], stage + i * 1024);
            xsrc[i] += kMidWaves * kRowStep;
        }
    };

    // the bias of the four features this thread stores, on its way together with the first operands
    Vec<Value, 4> b = {};
    const bool has_bias = OUT != kMidSlices && bias != nullptr;
    if (has_bias) {
        const int f = n0 + (int) (threadIdx.x % (TN / 4)) * 4;
        b = load_vec<Value, 4>(bias + (f < features ? f : 0));
    }

    v16f32 chains[CHAINS][TB][FB];
#pragma unroll
    for (int c = 0; c < CHAINS; ++c)
#pragma unroll
        for (int t = 0; t < TB; ++t)
#pragma unroll
            for (int f = 0; f < FB; ++f) chains[c][t][f] = v16f32{};
    v16f32 (&acc)[TB][FB] = chains[0];

#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
        if (d < steps) request(d);
    }
    int slot = 0;
    for (int s = 0; s < steps; ++s) {
        if (DEPTH == 2 && s + 1 < steps) {  // the step after this one has been requested too
            wait_loads<S::kLoads>();
        } else {
            wait_loads<0>();
        }
        __builtin_amdgcn_sched_barrier(0);
        const unsigned char *stage = mine + slot * S::kStageBytes;
        auto refill = [&] {
            __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this step has been read, its LDS may be written again
            __builtin_amdgcn_sched_barrier(0);
            if (s + DEPTH < steps) request(slot);
            __builtin_amdgcn_sched_barrier(0);
        };
        if constexpr (is_pairs<T>()) {
            // The small products, low x high and high x low, have accumulators of their own: a chain of additions that rounds at
            // the size of the sum is a sixteenth of K / 4 long.
            v8f16 x[2][2][TB], w[2][2][FB];  // [16 K values][high, low]
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int term = 1; term >= 0; --term) {
                    const int unit = ((term * 4 + q * 2 + hh) ^ ((r >> 1) & 7)) * 16;
#pragma unroll
                    for (int f = 0; f < FB; ++f)
                        w[q][term][f] = *reinterpret_cast<const v8f16 *>(stage + S::kXBytes + (f * 32 + r) * kStepBytes + unit);
#pragma unroll
                    for (int t = 0; t < TB; ++t)
                        x[q][term][t] = *reinterpret_cast<const v8f16 *>(stage + (t * 32 + r) * kStepBytes + unit);
                }
            refill();
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int kind = 0; kind < 3; ++kind)  // high x high, low x high, high x low
#pragma unroll
                    for (int t = 0; t < TB; ++t)
#pragma unroll
                        for (int f = 0; f < FB; ++f) {
                            v16f32 &sum = chains[kind < CHAINS ? kind : CHAINS - 1][t][f];
                            sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[q][kind == 1][f], x[q][kind == 2][t], sum, 0, 0, 0);
                        }
        } else if constexpr (sizeof(T) == 2) {
            // every operand of the step is read before the first product, and the slot is asked for again right then
            v8f16 x[4][TB], w[4][FB];  // 16 K values per q: 8 per lane half
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int unit = ((q * 2 + hh) ^ ((r >> 1) & 7)) * 16;
#pragma unroll
                for (int f = 0; f < FB; ++f)
                    w[q][f] = *reinterpret_cast<const v8f16 *>(stage + S::kXBytes + (f * 32 + r) * kStepBytes + unit);
#pragma unroll
                for (int t = 0; t < TB; ++t)
                    x[q][t] = *reinterpret_cast<const v8f16 *>(stage + (t * 32 + r) * kStepBytes + unit);
            }
            refill();
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int t = 0; t < TB; ++t)
#pragma unroll
                    for (int f = 0; f < FB; ++f)
                        acc[t][f] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[q][f], x[q][t], acc[t][f], 0, 0, 0);
        } else {
            // The fp32 products take sixteen times as long: they start with the first operands and the rest is read
            // between them (all reads first: 1056 workgroups of 32 x 32 x 768 27.1 instead of 23.1 us).
#pragma unroll
            for (int q = 0; q < 4; ++q) {  // 8 K values: 4 per lane half
                v4f32 x[TB];
                float w[FB][4];
                const int unit = ((q * 2 + hh) ^ ((r >> 1) & 7)) * 16;
#pragma unroll
                for (int f = 0; f < FB; ++f)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        w[f][e] = *reinterpret_cast<const float *>(stage + S::kXBytes +
                                                                   ((q * 8 + hh * 4 + e) * TN + f * 32 + r) * 4);
#pragma unroll
                for (int t = 0; t < TB; ++t)
                    x[t] = *reinterpret_cast<const v4f32 *>(stage + (t * 32 + r) * kStepBytes + unit);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int t = 0; t < TB; ++t)
#pragma unroll
                        for (int f = 0; f < FB; ++f) {
                            v16f32 &chain = chains[(q * 4 + e) * CHAINS / 16][t][f];
                            chain = __builtin_amdgcn_mfma_f32_32x32x2f32(w[f][e], x[t][e], chain, 0, 0, 0);
                        }
            }
            refill();
        }
        slot = slot + 1 < DEPTH ? slot + 1 : 0;
    }

    if constexpr (is_pairs<T>()) {
#pragma unroll
        for (int t = 0; t < TB; ++t)
#pragma unroll
            for (int f = 0; f < FB; ++f) chains[0][t][f] += CHAINS == 3 ? chains[1][t][f] + chains[2][t][f] : chains[1][t][f];
    }
#pragma unroll
    for (int half = is_pairs<T>() ? 0 : CHAINS / 2; half >= 1; half /= 2)
#pragma unroll
        for (int c = 0; c < half; ++c)
#pragma unroll
            for (int t = 0; t < TB; ++t)
#pragma unroll
                for (int f = 0; f < FB; ++f) chains[c][t][f] += chains[c + half][t][f];

    // partial tiles to LDS (each wavefront over its own operands, which it has read): a lane owns one token and, per
    // four accumulator registers, four consecutive features
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_sched_barrier(0);
    float *red = reinterpret_cast<float *>(mine);
#pragma unroll
    for (int t = 0; t < TB; ++t)
#pragma unroll
        for (int f = 0; f < FB; ++f)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                v4f32 v = {acc[t][f][g * 4], acc[t][f][g * 4 + 1], acc[t][f][g * 4 + 2], acc[t][f][g * 4 + 3]};
                *reinterpret_cast<v4f32 *>(red + (t * 32 + r) * S::kRedPitch + f * 32 + g * 8 + hh * 4) = v;
            }
    __syncthreads();
    constexpr int kQuads = TN / 4;
#pragma unroll
    for (int it = 0; it < TM * kQuads / kMidThreads; ++it) {
        const int item = it * kMidThreads + threadIdx.x;
        const int token = item / kQuads, q = item % kQuads;
        v4f32 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < kMidWaves; ++w) {
            sum += *reinterpret_cast<const v4f32 *>(smem + w * S::kWaveBytes + (token * S::kRedPitch + q * 4) * 4);
        }
        const int row = m0 + token, col = n0 + q * 4;
        if (row >= tokens || col >= features) continue;
        if constexpr (OUT == kMidSlices) {
            if (is_pairs<T>()) sum *= alpha;
            *reinterpret_cast<v4f32 *>(partials + slice * slice_stride + (size_t) row * pitch + col) = sum;
        } else if constexpr (is_pairs<T>() && OUT == kMidGelu) {
            Vec<half_t, 4> hi, lo;
            bool over = false;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float v = GeluOp<float>()(fmaf(sum[e], alpha, b.v[e])) * scale;
                split_two_terms(v, hi.v[e], lo.v[e]);
                over = over || two_term_overflow(v);
            }
            half_t *at = reinterpret_cast<half_t *>(C + (size_t) row * ldc) + pair_at(col);
            store_vec<half_t, 4>(at, hi);
            store_vec<half_t, 4>(at + kPairBlock, lo);
            if (over && overflow != nullptr) *overflow = 1;
        } else {
            Vec<Value, 4> out;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v = is_pairs<T>() ? fmaf(sum[e], alpha, to_f32(b.v[e])) : sum[e] + to_f32(b.v[e]);
                if (OUT == kMidGelu) v = GeluOp<Value>()(v);
                out.v[e] = from_f32<Value>(v);
            }
            store_vec<Value, 4>(C + (size_t) row * ldc + col, out);
        }
    }
}

struct MidPlan {
    int tile = 0;  // 0: 32 x 32, 1: 64 x 32, 2: 64 x 64
    int depth = 2, slices = 1, steps_per_slice = 0;
    int chains = 1;
};

constexpr int kShortSumTokens = 64, kShortSumChains = 8, kShortSumSteps = 32;

// The tile and the number of K slices, by a model of the launch time (in microseconds): 2.3 for dispatch, the first
// operands and the drain, then as many rounds as the fullest of the 256 compute units has workgroups.  A workgroup takes its
// operands at 80 KB per microsecond in half precision and in pairs (768 x 768 in 32 x 32 tiles: 98 KB, 1.4 us with its epilogue); in fp32 a
// tile of 32 x 32 takes 4.1 us per 768 K values, 64 x 32 8.0, 64 x 64 14.5.  Workgroups that share a compute unit gain
// nothing over taking turns.  Slices cost their way through memory, and at most eight are worth it: the LayerNorm has eight
// of a row on their way together (32 tokens, 3072 -> 768, fp32, with the LayerNorm: 8 slices 8.6 us, 10 9.6, 16 10.6).
// Measured with the LayerNorm or GELU over every tile, depth and 1 to 16 slices at the four Dense shapes of BERT-base and
// BERT-large, 8 to 320 fp32 and 8 to 1280 half-precision tokens as far as models take this kernel: the choice is within
// 9 % of the best one at 151 of 152, within 17 % at the other.  Pairs, 32 to 1280 tokens as far as
// models take this kernel: within 4 % of the best at 27 of 28, within 13 % at the other.
// Depth: two steps ahead where one workgroup per compute unit is all there is (96 workgroups of 32 x 32 x 768, fp16: one
// step ahead 4.2, two 3.8 us), one where more workgroups fit the LDS that way (672: 6.1 against 6.9 us); in fp32 two pay
// off for every tile (1056: 24.8 against 22.6 us).
// fp32 up to 64 tokens, where a caller would otherwise have the few-token kernel's short sums: eight chains of at most 32
// values each where K is cut (longer slices have 1.7e-7 instead of 1.3e-7, the few-token kernel 1.3e-7 to 1.5e-7), which
// the registers hold for a tile of 32 x 32.
template <typename T>
MidPlan plan_mid(int tokens, int features, int steps, bool sliced, size_t partial_floats) {
    static const int kTile[3][2] = {{32, 32}, {64, 32}, {64, 64}};
    static const float kEpilogue[3] = {0.15f, 0.5f, 1.3f};             // us, half precision
    static const float kF32Step[3] = {4.1f / 24, 8.0f / 24, 14.5f / 24};  // us per step of a workgroup
    constexpr bool kHalfOperands = sizeof(typename MidTypes<T>::Operand) == 2;
    const bool short_sums = !kHalfOperands && tokens <= kShortSumTokens;
    const int most_slices = !sliced ? 1 : short_sums && steps >= 8 * kShortSumSteps ? 16 : 8;
    MidPlan best;
    float best_us = 0.f;
    for (int t = 0; t < (short_sums ? 1 : 3); ++t) {
        const long long tiles = (long long) ((tokens + kTile[t][0] - 1) / kTile[t][0]) *
                                ((features + kTile[t][1] - 1) / kTile[t][1]);
        for (int want = 1; want <= most_slices; ++want) {
            const int per = (steps + want - 1) / want, slices = (steps + per - 1) / per;
            if (slices != want) continue;
            if (slices > 1 && (per < kMidWaves || (size_t) slices * tokens * features > partial_floats)) break;
            const float rounds = (float) ((tiles * slices + 255) / 256);
            const float each = kHalfOperands
                                   ? per * (kTile[t][0] + kTile[t][1]) * (kStepBytes / 80e3f) + kEpilogue[t]
                                   : per * kF32Step[t];
            float us = 2.3f + rounds * each;
            if (slices > 1) us += slices * (0.1f + (float) tokens * features * (8.f / 5e6f));
            if (short_sums && per > kShortSumSteps) us += 1e6f;  // taken only if no finer cut fits
            if (best_us == 0.f || us < best_us) {
                best_us = us;
                best.tile = t, best.slices = slices, best.steps_per_slice = per;
                best.depth = !kHalfOperands || tiles * slices <= 256 ? 2 : 1;
            }
        }
    }
    best.chains = short_sums ? kShortSumChains : 1;
    return best;
}

// the arguments of a launch
template <typename T>
struct MidCall {
    typedef typename MidTypes<T>::Operand Operand;
    typedef typename MidTypes<T>::Value Value;
    const Operand *W;
    int ldw;
    const Operand *X;
    int ldx;
    const Value *bias;
    Value *C;
    int ldc, tokens, features, steps;
    float *partials;
    hipStream_t stream;
    float alpha = 1.f, scale = 1.f;
    int *overflow = nullptr;
};

template <typename T, int TM, int TN, int DEPTH, int OUT, int CHAINS>
int launch_mid(const MidPlan &plan, const MidCall<T> &c) {
    typedef MidShape<TM, TN, DEPTH> S;
    static_assert(S::kLdsBytes <= 160 * 1024, "LDS of a compute unit");
    static std::atomic<unsigned long long> raised{0};  // per kernel
    if (!allow_large_lds(dense_mid_kernel<T, TM, TN, DEPTH, OUT, CHAINS>, raised)) return CUBERT_UNSUPPORTED;
    const int token_tiles = (c.tokens + TM - 1) / TM, feature_tiles = (c.features + TN - 1) / TN;
    const dim3 grid((unsigned) (feature_tiles * token_tiles * plan.slices)), block(kMidThreads);
    return launch_lds(dense_mid_kernel<T, TM, TN, DEPTH, OUT, CHAINS>, grid, block, (unsigned) S::kLdsBytes, c.stream, c.W, c.ldw,
                      c.X, c.ldx, c.bias, c.C, c.ldc, c.tokens, c.features, c.steps, plan.steps_per_slice, token_tiles,
                      feature_tiles, c.partials, c.features, (long long) c.tokens * c.features, c.alpha, c.scale, c.overflow);
}

template <typename T, int OUT>
int launch_mid_tile(const MidPlan &plan, const MidCall<T> &c) {
    // accumulators per block: of a pair's three products each its own where a wavefront has one block, else one for the small two
    constexpr int kOne = is_pairs<T>() ? 3 : 1, kMany = is_pairs<T>() ? 2 : 1;
    if constexpr (sizeof(typename MidTypes<T>::Operand) == 2) {
        if (plan.depth == 1) {
            switch (plan.tile) {
                case 0: return launch_mid<T, 32, 32, 1, OUT, kOne>(plan, c);
                case 1: return launch_mid<T, 64, 32, 1, OUT, kMany>(plan, c);
                default: return launch_mid<T, 64, 64, 1, OUT, kMany>(plan, c);
            }
        }
    }
    if constexpr (std::is_same<T, float>::value) {
        if (plan.chains != 1) return launch_mid<T, 32, 32, 2, OUT, kShortSumChains>(plan, c);
    }
    switch (plan.tile) {
        case 0: return launch_mid<T, 32, 32, 2, OUT, kOne>(plan, c);
        case 1: return launch_mid<T, 64, 32, 2, OUT, kMany>(plan, c);
        default: return launch_mid<T, 64, 64, 2, OUT, kMany>(plan, c);
    }
}

// What the kernel assumes of its operands: whole steps of K, 16-byte pieces of X and W, four features per store.
template <typename T>
int check_mid(int tokens, int features, int in, const T *X, int ldx, const T *W, int ldw) {
    if (!X || !W || tokens < 0 || features < 0 || in < 0) return CUBERT_BAD_ARGUMENT;
    if (ldx < in || ldw < (sizeof(T) == 2 ? in : features)) return CUBERT_BAD_ARGUMENT;
    constexpr int U = 16 / sizeof(T);
    if (in == 0 || in % (int) (kStepBytes / sizeof(T)) != 0 || features % 4 != 0 || tokens > 65535 || features > (1 << 20) ||
        !is_aligned(X, 16) || !is_aligned(W, 16) || ldx % U != 0 || ldw % U != 0) {
        return CUBERT_UNSUPPORTED;
    }
    return 0;
}

}  // namespace

// C[token, feature] = act(X W + bias) in one launch; CUBERT_UNSUPPORTED (and nothing launched) where it does not fit.
template <typename T>
int dense_mid(int tokens, int features, int in, const T *X, int ldx, const T *W, int ldw, const T *bias, int activation,
              T *C, int ldc, hipStream_t stream) {
    if (!C || ldc < features || (activation != 0 && activation != 1)) return CUBERT_BAD_ARGUMENT;
    const int rc = check_mid(tokens, features, in, X, ldx, W, ldw);
    if (rc) return rc;
    if (ldc % 4 != 0 || !is_aligned(C, 4 * sizeof(T)) || !is_aligned(bias, 4 * sizeof(T))) return CUBERT_UNSUPPORTED;
    if (tokens == 0 || features == 0) return 0;
    const int steps = in / (int) (kStepBytes / sizeof(T));
    const MidPlan plan = plan_mid<T>(tokens, features, steps, false, 0);
    const MidCall<T> c = {W, ldw, X, ldx, bias, C, ldc, tokens, features, steps, nullptr, stream};
    return activation == 1 ? launch_mid_tile<T, kMidGelu>(plan, c) : launch_mid_tile<T, kMidStore>(plan, c);
}

// The product left as *slices slices partials[slice][token][feature] for a consumer that adds them; where one slice is
// the best cut this declines (dense_mid stores the finished product).
template <typename T>
int dense_mid_slices(int tokens, int features, int in, const T *X, int ldx, const T *W, int ldw, float *partials,
                     size_t partial_floats, int *slices, hipStream_t stream) {
    if (!partials || !slices) return CUBERT_BAD_ARGUMENT;
    const int rc = check_mid(tokens, features, in, X, ldx, W, ldw);
    if (rc) return rc;
    if (!is_aligned(partials, 16) || tokens == 0 || features == 0) return CUBERT_UNSUPPORTED;
    const int steps = in / (int) (kStepBytes / sizeof(T));
    const MidPlan plan = plan_mid<T>(tokens, features, steps, true, partial_floats);
    if (plan.slices < 2) return CUBERT_UNSUPPORTED;
    *slices = plan.slices;
    return launch_mid_tile<T, kMidSlices>(plan, {W, ldw, X, ldx, nullptr, nullptr, features, tokens, features, steps, partials, stream});
}

// The same over rows of pairs, [tokens, 2 * in] and [features, 2 * in] halves: C = alpha * sum + bias as floats, or GELU of that, times
// scale, as such rows again (overflow: see split.hip), or alpha * sum in slices.
int check_mid_pairs(int tokens, int features, int in, const half_t *X, const half_t *W) {
    if (in < 0 || in > (1 << 20)) return in < 0 ? CUBERT_BAD_ARGUMENT : CUBERT_UNSUPPORTED;
    return check_mid<half_t>(tokens, features, 2 * in, X, 2 * in, W, 2 * in);
}

int dense_mid_pairs(int tokens, int features, int in, const half_t *X, const half_t *W, const float *bias, int activation,
                    float alpha, float scale, float *C, int ldc, int *overflow, hipStream_t stream) {
    if (!C || ldc < features || (activation != 0 && activation != 1)) return CUBERT_BAD_ARGUMENT;
    const int rc = check_mid_pairs(tokens, features, in, X, W);
    if (rc) return rc;
    if (ldc % 4 != 0 || !is_aligned(C, 16) || !is_aligned(bias, 16) ||
        (activation == 1 && (features % kPairBlock != 0 || ldc != features))) {
        return CUBERT_UNSUPPORTED;
    }
    if (tokens == 0 || features == 0) return 0;
    const int steps = in / mid_step<Pairs>();
    const MidPlan plan = plan_mid<Pairs>(tokens, features, steps, false, 0);
    const MidCall<Pairs> c = {W, 2 * in, X, 2 * in, bias, C, ldc, tokens, features, steps, nullptr, stream, alpha, scale, overflow};
    return activation == 1 ? launch_mid_tile<Pairs, kMidGelu>(plan, c) : launch_mid_tile<Pairs, kMidStore>(plan, c);
}

int dense_mid_pairs_slices(int tokens, int features, int in, const half_t *X, const half_t *W, float alpha, float *partials,
                           size_t partial_floats, int *slices, hipStream_t stream) {
    if (!partials || !slices) return CUBERT_BAD_ARGUMENT;
    const int rc = check_mid_pairs(tokens, features, in, X, W);
    if (rc) return rc;
    if (!is_aligned(partials, 16) || tokens == 0 || features == 0) return CUBERT_UNSUPPORTED;
    const int steps = in / mid_step<Pairs>();
    const MidPlan plan = plan_mid<Pairs>(tokens, features, steps, true, partial_floats);
    if (plan.slices < 2) return CUBERT_UNSUPPORTED;
    *slices = plan.slices;
    return launch_mid_tile<Pairs, kMidSlices>(
            plan, {W, 2 * in, X, 2 * in, nullptr, nullptr, features, tokens, features, steps, partials, stream, alpha});
}

// What dense_mid (as_slices = 0) or dense_mid_slices would launch.
template <typename T>
int dense_mid_plan(int tokens, int features, int in, bool as_slices, size_t partial_floats, int *tile, int *depth, int *slices) {
    if (tokens <= 0 || features <= 0 || in <= 0 || !tile || !depth || !slices) return CUBERT_BAD_ARGUMENT;
    if (in % (int) (kStepBytes / sizeof(T)) != 0) return CUBERT_UNSUPPORTED;
    const MidPlan plan = plan_mid<T>(tokens, features, in / (int) (kStepBytes / sizeof(T)), as_slices, partial_floats);
    if (as_slices && plan.slices < 2) return CUBERT_UNSUPPORTED;
    *tile = plan.tile, *depth = plan.depth, *slices = plan.slices;
    return 0;
}

template int dense_mid_plan<float>(int, int, int, bool, size_t, int *, int *, int *);
template int dense_mid_plan<half_t>(int, int, int, bool, size_t, int *, int *, int *);
template int dense_mid<float>(int, int, int, const float *, int, const float *, int, const float *, int, float *, int,
                              hipStream_t);
template int dense_mid<half_t>(int, int, int, const half_t *, int, const half_t *, int, const half_t *, int, half_t *, int,
                               hipStream_t);
template int dense_mid_slices<float>(int, int, int, const float *, int, const float *, int, float *, size_t, int *,
                                     hipStream_t);
template int dense_mid_slices<half_t>(int, int, int, const half_t *, int, const half_t *, int, float *, size_t, int *,
                                      hipStream_t);

}  // namespace cubert
