// Dense layers of hundreds to thousands of tokens on the fp16 matrix cores, C[token, feature] = sum_k x[token, k] w[feature, k],
// in two forms:
//   - halves: fp16 rows of X and W, C = fp16(sum + bias) or fp16(GELU(sum + bias)); a step takes 64 values of K;
//   - pairs: fp32 operands as pairs of fp16 numbers, x = xh + xl, w = wh + wl (see split.hip).  A row of X or W holds, for every
//     32 values of K, their 32 high terms and then their 32 low terms, a step.  The library's form of the same sum is one fp16
//     GEMM over [hi | hi | lo] rows, which reads the high terms twice and multiplies each operand it reads once; here an operand
//     that has come to LDS takes part in three products of one step, high x low, low x high and high x high.
// Either way a step takes 128 bytes of a row, a whole line: a compute unit gets 40 bytes per cycle from its L2 in such pieces and
// 23 in pieces of 64 (measured without any products).
//
// What bounds it: the matrix cores, which throttle the clock to 1.7 to 2.1 GHz while they are busy, and which both forms keep
// busy for some 60 (halves) to 80 % (pairs) of a step.  What it took to get there, each measured at 4096 tokens, 768 -> 2304:
//   - two rings in LDS, X two steps deep and W three: the next step's X is asked for when its slot has been read, W earlier;
//   - requests go out between the products of a phase: asked for in one go after the barrier, a wavefront stands at its
//     requests while its matrix core idles (halves 28.1 -> 25.3 us at 256 x 256);
//   - LDS reads of the next phase also go out between the products, one by one (in one go in front of them: pairs 54.5 us, 47.5);
//   - one barrier per step, in front of its last phase, whose operands are in registers by then.
// 32 x 32 blocks of C per wavefront; a finished part of C passes through LDS of its wavefront and leaves in whole row segments.
#include "activations.h"
#include "cubert_kernels.h"
#include "device_common.h"

namespace cubert {
namespace {

typedef float v16f32 __attribute__((ext_vector_type(16)));
typedef _Float16 v8f16 __attribute__((ext_vector_type(8)));

constexpr int kRowBytes = 128;             // of a row of X or W that a step takes
constexpr int kHalfStep = kRowBytes / 2;   // values of K in them
constexpr int kPairStep = kRowBytes / 4;

// the LDS accesses of this wavefront in front of it are done before those behind it start
__device__ __forceinline__ void order_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// What the kernel reads and what leaves it.  Pairs: alpha * sum + bias as fp32, or GELU of that, times scale, as operand rows of
// the next layer.
enum DenseForm { kHalves = 0, kHalvesGelu = 1, kPairsFloat = 2, kPairsGelu = 3 };
constexpr bool has_pairs(int form) { return form >= kPairsFloat; }
template <int FORM>
struct FormTypes { typedef float Value; };  // of bias and C
template <>
struct FormTypes<kHalves> { typedef half_t Value; };
template <>
struct FormTypes<kHalvesGelu> { typedef half_t Value; };

// TM tokens x TN features by WM x WN wavefronts, or twice as many that take a half of each step (KW = 2); rings of XS steps of X
// and WS steps of W
template <int FORM, int TM, int TN, int WM, int WN, int KW, int XS, int WS>
struct TileShape {
    static constexpr int kTileWaves = WM * WN, kWaves = kTileWaves * KW, kThreads = kWaves * kWave;
    static constexpr int kTB = TM / WM / 32, kFB = TN / WN / 32;  // 32 x 32 blocks of a wavefront
    static constexpr int kXBytes = TM * kRowBytes, kWBytes = TN * kRowBytes;
    // requests of a wavefront per step, eight rows each; some wavefronts may have one of W less
    static constexpr int kXLoads = TM / 8 / kWaves, kWLoads = (TN / 8 + kWaves - 1) / kWaves, kWLoadsAtLeast = TN / 8 / kWaves;
    static constexpr int kOutRow = kFB * 32 * (has_pairs(FORM) ? 4 : 2);  // bytes of a token in a wavefront's part of C
    static constexpr int kOutPitch = kOutRow + 16, kOutBytes = 32 * kOutPitch;
    // of a wavefront at the end: its rows on their way out, and before them what the second half of the wavefronts hands over
    static constexpr int kHalfBytes = KW == 2 ? kTB * kFB * 16 * kWave * 4 : 0;
    static constexpr int kPart = kOutBytes > kHalfBytes ? kOutBytes : kHalfBytes;
    static constexpr int kRings = XS * kXBytes + WS * kWBytes, kOut = kTileWaves * kPart + TN * 4;
    static constexpr int kLdsBytes = kRings > kOut ? kRings : kOut;
    static_assert(kXLoads * kWaves * 8 == TM && TN % 32 == 0 && kWLoadsAtLeast > 0, "whole requests");
    static_assert(XS >= 2 && WS >= XS, "weights are further ahead, or as far");
    static_assert(TN <= kThreads && kLdsBytes <= 160 * 1024, "a thread per bias, LDS of a compute unit");
};

template <int FORM, int TM, int TN, int WM, int WN, int KW, int XS, int WS>
__global__ __launch_bounds__(WM * WN * KW * kWave) void dense_large_kernel(
        const half_t *__restrict__ W, const half_t *__restrict__ X, const typename FormTypes<FORM>::Value *__restrict__ bias,
        typename FormTypes<FORM>::Value *__restrict__ C, int ldc, int tokens, int features, int steps_total, int token_tiles,
        int feature_tiles, float alpha, float scale, int *__restrict__ overflow, int steps_per_slice) {
    typedef TileShape<FORM, TM, TN, WM, WN, KW, XS, WS> S;
    constexpr int TB = S::kTB, FB = S::kFB;
    constexpr bool kPairs = has_pairs(FORM);
    constexpr int kTerms = kPairs ? 2 : 1, kPhases = kPairs ? 2 : 4;  // high and low; phases of a step, 16 values of K each
    typedef typename FormTypes<FORM>::Value Value;
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & (kWave - 1), wave = wave_in_block();
    const int r = lane & 31, hh = lane >> 5;
    const int tile_wave = wave % S::kTileWaves, half = wave / S::kTileWaves;
    const int wm = tile_wave / WN, wn = tile_wave % WN;

    // Workgroups are handed to the eight dies in turn; each die gets a contiguous run of tiles, which go down groups of eight
    // token tiles and then across features: the 32 tiles that a die works on at a time are about 8 x 4 of them.
    const int die = blockIdx.x & 7, die_share = gridDim.x >> 3, extra = gridDim.x & 7;
    const int index = die * die_share + (die < extra ? die : extra) + (int) (blockIdx.x >> 3);
    // (K slices, where a LayerNorm adds them: the first slice's tiles first)
    const int slice = FORM == kPairsFloat ? index / (token_tiles * feature_tiles) : 0;
    const int steps = FORM != kPairsFloat                                          ? steps_total
                      : steps_total - slice * steps_per_slice < steps_per_slice ? steps_total - slice * steps_per_slice
                                                                                : steps_per_slice;
    const int tile = index - slice * (token_tiles * feature_tiles);
    const int per_group = 8 * feature_tiles;
    const int first = tile / per_group * 8, in_group = tile % per_group;
    const int height = token_tiles - first < 8 ? token_tiles - first : 8;
    const int ft = in_group / height, tt = first + in_group - ft * height;
    const int m0 = tt * TM, n0 = ft * TN;

    // The bias of a feature per thread, on its way before the first operands and looked at behind the products.  (Read without a
    // branch, from any valid address where there is none: a branch would end with the wait for it.)
    const int my_feature = n0 + (int) threadIdx.x;
    const bool has_bias = bias != nullptr && threadIdx.x < TN && my_feature < features;
    const Value b = *(has_bias ? bias + my_feature : reinterpret_cast<const Value *>(W));

    // lane l of a request brings the 16-byte unit l % 8 of row l / 8 of eight rows to unit (l % 8) ^ (row / 2 % 8), which
    // spreads the operand reads over all banks; rows past the end are read from the last one
    const unsigned row_bytes = (unsigned) steps_total * kRowBytes, slice_at = (unsigned) (slice * steps_per_slice) * kRowBytes;
    const char *xbase = reinterpret_cast<const char *>(X) + (size_t) m0 * row_bytes + slice_at;
    const char *wbase = reinterpret_cast<const char *>(W) + (size_t) n0 * row_bytes + slice_at;
    if (FORM == kPairsFloat) C += (size_t) slice * tokens * ldc;
    unsigned xo[S::kXLoads], wo[S::kWLoads];
    auto offset_of = [&](int i, int rows_left) {
        const int row = (wave + i * S::kWaves) * 8 + (lane >> 3);
        return (unsigned) (row < rows_left ? row : rows_left - 1) * row_bytes + ((lane & 7) ^ ((row >> 1) & 7)) * 16;
    };
#pragma unroll
    for (int i = 0; i < S::kXLoads; ++i) xo[i] = offset_of(i, tokens - m0);
#pragma unroll
    for (int i = 0; i < S::kWLoads; ++i) wo[i] = offset_of(i, features - n0);

    // request number i of a step's: X of a step, then W of one
    constexpr int kRequests = S::kXLoads + S::kWLoads;
    auto request = [&](int i, int xslot, bool with_x, int wslot, bool with_w) {
        if (i < S::kXLoads) {
            if (with_x) load_to_lds(xbase + xo[i], smem + xslot * S::kXBytes + (wave + i * S::kWaves) * 1024);
            if (with_x && i == S::kXLoads - 1) xbase += kRowBytes;
        } else {
            const int j = i - S::kXLoads;
            if (with_w && (j < S::kWLoadsAtLeast || wave + j * S::kWaves < TN / 8)) {
                load_to_lds(wbase + wo[j], smem + XS * S::kXBytes + wslot * S::kWBytes + (wave + j * S::kWaves) * 1024);
            }
            if (with_w && i == kRequests - 1) wbase += kRowBytes;
        }
    };

    v16f32 acc[TB][FB];
#pragma unroll
    for (int t = 0; t < TB; ++t)
#pragma unroll
        for (int f = 0; f < FB; ++f) acc[t][f] = v16f32{};

    // operand number j of a phase: the blocks of W, then those of X, low terms first
    constexpr int kReads = kTerms * (TB + FB);
    const int xoff = (wm * TB * 32 + r) * kRowBytes, woff = XS * S::kXBytes + (wn * FB * 32 + r) * kRowBytes;
    v8f16 x[2][kTerms][TB], w[2][kTerms][FB];
    auto read = [&](int j, int xslot, int wslot, int phase, int buffer) {
        const int term = kTerms - 1 - j / (TB + FB), k = j % (TB + FB);
        const int unit = ((term * 4 + phase * 2 + hh) ^ ((r >> 1) & 7)) * 16;
        const unsigned char *at = k < FB ? smem + wslot * S::kWBytes + woff + k * 32 * kRowBytes
                                         : smem + xslot * S::kXBytes + xoff + (k - FB) * 32 * kRowBytes;
        (k < FB ? w[buffer][term][k < FB ? k : 0] : x[buffer][term][k < FB ? 0 : k - FB]) =
                *reinterpret_cast<const v8f16 *>(at + unit);
    };

    int xslot = 0, wslot = 0, xfree = 0, wfree = 0;  // slots of the next operands, and those that were read last
    bool more_x = false, more_w = false;
    // The products of a phase; in between go the reads of the wavefront's next phase, in the first three quarters, and this
    // phase's share of the requests into the free slots, which starts with the last phase of a step.
    constexpr int kMyPhases = kPhases / KW;
    const int my_first = half * kMyPhases;
    auto multiply = [&](int phase, int buffer) {
        constexpr int kProducts = (kPairs ? 3 : 1) * TB * FB;
        const int next = (phase + 1) % kMyPhases;
        const int from = next * kRequests / kMyPhases, until = (next + 1) * kRequests / kMyPhases;
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int m = 0; m < kProducts; ++m) {
            const int kind = m / (TB * FB), t = m / FB % TB, f = m % FB;  // low x high, high x low, high x high
            acc[t][f] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[buffer][kPairs && kind == 0 ? 1 : 0][f],
                                                               x[buffer][kPairs && kind == 1 ? 1 : 0][t], acc[t][f], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < kReads; ++j) {
                if (j * kProducts * 3 / (4 * kReads) == m) read(j, xslot, wslot, my_first + next, buffer ^ 1);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < kRequests; ++i) {
                if (i >= from && i < until && (i - from) * kProducts / (until - from) == m) {
                    request(i, xfree, more_x, wfree, more_w);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
    };

#pragma unroll
    for (int d = 0; d < WS; ++d)
#pragma unroll
        for (int i = 0; i < kRequests; ++i) request(i, d, d < XS && d < steps, d, d < steps);
    if (steps >= WS) {
        wait_loads<(WS - 1) * S::kWLoadsAtLeast + (XS - 1) * S::kXLoads>();
    } else {
        wait_loads<0>();
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < kReads; ++j) read(j, 0, 0, my_first, 0);
    auto step = [&](int s, int buffer) {
#pragma unroll
        for (int q = 0; q + 1 < kMyPhases; ++q) multiply(q, (buffer + q) & 1);
        xfree = xslot, wfree = wslot;
        xslot = xslot + 1 < XS ? xslot + 1 : 0, wslot = wslot + 1 < WS ? wslot + 1 : 0;
        more_x = s + XS < steps, more_w = s + WS < steps;
        if (s + 1 < steps) {
            // The next step has landed.  Younger than it: X of XS - 2 steps, and W of as many, or of one more where the ring
            // of W is the deeper one (W of step j + WS follows X of step j + XS).  In the last steps nothing is.
            constexpr int kYounger = (XS - 2) * S::kXLoads + (XS == WS ? XS - 2 : XS - 1) * S::kWLoadsAtLeast;
            if (s + WS <= steps) {
                wait_loads<kYounger>();
            } else {
                wait_loads<0>();
            }
            __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wavefront has read this step
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
        }
        // (behind the last step this reads a slot that holds nothing of use, for a phase that does not follow)
        multiply(kMyPhases - 1, (buffer + kMyPhases - 1) & 1);
    };
    constexpr int kUnroll = kMyPhases % 2 == 0 ? 1 : 2;  // the operand registers alternate
    for (int s = 0; s < steps; s += kUnroll) {
        step(s, 0);
        if (kUnroll == 2 && s + 1 < steps) step(s + 1, 1);
    }

    __syncthreads();
    float *bias_lds = reinterpret_cast<float *>(smem + S::kTileWaves * S::kPart);
    if (threadIdx.x < TN) bias_lds[threadIdx.x] = to_f32(keep_or_zero(b, has_bias));
    if constexpr (KW == 2) {
        float *other = reinterpret_cast<float *>(smem + tile_wave * S::kPart) + lane * 4;
        if (half == 1) {
#pragma unroll
            for (int t = 0; t < TB; ++t)
#pragma unroll
                for (int f = 0; f < FB; ++f)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const Vec<float, 4> v = {acc[t][f][g * 4], acc[t][f][g * 4 + 1], acc[t][f][g * 4 + 2], acc[t][f][g * 4 + 3]};
                        store_vec<float, 4>(other + ((t * FB + f) * 4 + g) * (4 * kWave), v);
                    }
        }
        __syncthreads();
        if (half == 1) return;
#pragma unroll
        for (int t = 0; t < TB; ++t)
#pragma unroll
            for (int f = 0; f < FB; ++f)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const Vec<float, 4> v = load_vec<float, 4>(other + ((t * FB + f) * 4 + g) * (4 * kWave));
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[t][f][g * 4 + e] += v.v[e];
                }
        order_lds();
    } else {
        __syncthreads();
    }
    // 32 tokens at a time: a lane owns a token and, per four accumulator registers, four consecutive features
    unsigned char *out = smem + tile_wave * S::kPart;
    const int col0 = n0 + wn * FB * 32;
    bool over = false;
#pragma unroll
    for (int t = 0; t < TB; ++t) {
        unsigned char *at = out + r * S::kOutPitch;
#pragma unroll
        for (int f = 0; f < FB; ++f) {
            bool fits = true;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int col = g * 8 + hh * 4;
                const Vec<float, 4> bv = load_vec<float, 4>(bias_lds + (wn * FB + f) * 32 + col);
                Vec<float, 4> y;
#pragma unroll
                for (int e = 0; e < 4; ++e) y.v[e] = kPairs ? fmaf(acc[t][f][g * 4 + e], alpha, bv.v[e]) : acc[t][f][g * 4 + e] + bv.v[e];
                if constexpr (FORM == kPairsGelu) {
                    Vec<half_t, 4> hi, lo;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        // (as split_two_terms; GELU is never below -0.2, and a low term that does not fit is one of a value
                        // that raises the flag)
                        const float v = GeluOp<float>()(y.v[e]) * scale;
                        hi.v[e] = (half_t) fminf(v, 65504.f);
                        lo.v[e] = (half_t) fmaf(-1.f, (float) hi.v[e], v);
                        fits = fits && fabsf(v) <= 65504.f;
                    }
                    store_vec<half_t, 4>(reinterpret_cast<half_t *>(at) + f * 64 + col, hi);
                    store_vec<half_t, 4>(reinterpret_cast<half_t *>(at) + f * 64 + 32 + col, lo);
                } else if constexpr (FORM == kPairsFloat) {
                    store_vec<float, 4>(reinterpret_cast<float *>(at) + f * 32 + col, y);
                } else {
                    Vec<half_t, 4> v;
#pragma unroll
                    for (int e = 0; e < 4; ++e) v.v[e] = from_f32<half_t>(FORM == kHalvesGelu ? GeluOp<half_t>()(y.v[e]) : y.v[e]);
                    store_vec<half_t, 4>(reinterpret_cast<half_t *>(at) + f * 32 + col, v);
                }
            }
            over = over || (!fits && m0 + (wm * TB + t) * 32 + r < tokens && col0 + f * 32 < features);
        }
        order_lds();
        constexpr int kPieces = S::kOutRow / 16, kPiece = 16 / sizeof(Value);
        const int token0 = m0 + (wm * TB + t) * 32;
        Value *rows = C + (size_t) token0 * ldc + col0;
#pragma unroll
        for (int i = 0; i < 32 * kPieces / kWave; ++i) {
            const int item = i * kWave + lane, row = item / kPieces, piece = item - row * kPieces;
            const auto v = load_vec<Value, kPiece>(reinterpret_cast<const Value *>(out + row * S::kOutPitch + piece * 16));
            if (token0 + row < tokens && col0 + piece * kPiece < features) {
                store_vec<Value, kPiece>(rows + (size_t) row * ldc + piece * kPiece, v);
            }
        }
        order_lds();
    }
    if (FORM == kPairsGelu && over && overflow != nullptr) *overflow = 1;
}

// the arguments of a launch
template <typename Value>
struct DenseCall {
    const half_t *W, *X;
    const Value *bias;
    Value *C;
    int ldc, tokens, features, steps;
    float alpha, scale;
    int *overflow;
    hipStream_t stream;
    int slices = 1, steps_per_slice = 0;
};

template <int FORM, int TM, int TN, int WM, int WN, int KW, int XS, int WS>
int launch_large(const DenseCall<typename FormTypes<FORM>::Value> &c) {
    typedef TileShape<FORM, TM, TN, WM, WN, KW, XS, WS> S;
    static std::atomic<unsigned long long> raised{0};  // per kernel
    auto kernel = dense_large_kernel<FORM, TM, TN, WM, WN, KW, XS, WS>;
    if (!allow_large_lds(kernel, raised)) return CUBERT_UNSUPPORTED;
    const int token_tiles = (c.tokens + TM - 1) / TM, feature_tiles = (c.features + TN - 1) / TN;
    return launch_lds(kernel, dim3((unsigned) (token_tiles * feature_tiles * c.slices)), dim3(S::kThreads), (unsigned) S::kLdsBytes,
                      c.stream, c.W, c.X, c.bias, c.C, c.ldc, c.tokens, c.features, c.steps, token_tiles, feature_tiles, c.alpha,
                      c.scale, c.overflow, c.slices > 1 ? c.steps_per_slice : c.steps);
}

// The tile, by a model of the launch time in microseconds, fitted to 768 and 3072 inputs, 384 to 16384 tokens and 768 to 3072
// features.  With u tiles per compute unit a launch takes what a tile takes by itself, slowed down by the others', or what the
// tiles of a compute unit take one after the other; where one or two tiles fill a compute unit, rounds are whole.
struct TileModel {
    int tm, tn;
    float alone, alone_step, crowd, each, each_step, start;
    int round;  // tiles per compute unit that run as one round (0: no rounds)
};

constexpr int kTiles = 5;

// Pairs.  Two halves of the wavefronts take a half of each step where a tile would otherwise have one wavefront per matrix core
// or little to do.  Measured at 768 -> 2304 / 768 -> 768 / 768 -> 3072 with GELU / 3072 -> 768, in halves marked *:
//   tokens   256 x 192            128 x 128            128 x 96           *128 x 96            *64 x 64
//      384   35 / 34 / 43 / 117   17 / 15 / 20 / 56    16 / 15 / 19 / 60    15 / 15 / 19 / 44   10 / 8.9 / 14 / 26
//     1280   36 / 34 / 45 / 116   19 / 16 / 24 / 57    20 / 16 / 29 / 59    18 / 16 / 35 / 45   21 / 10 / 27 / 28
//     2080   38 / 35 / 46 / 116   30 / 17 / 36 / 56    27 / 18 / 48 / 59    31 / 16 / 52 / 45   31 / 13 / 46 / 40
//     3072   38 / 35 / 52 / 116   34 / 18 / 55 / 59    43 / 19 / 50 / 61    45 / 16 / 57 / 49   42 / 20 / 59 / 65
//     4096   44 / 35 / 59 / 121   48 / 19 / 60 / 64    44 / 19 / 61 / 67    48 / 18 / 76 / 58   55 / 20 / 86 / 71
//     8192   87 / 41 / 116 / 131  83 / 32 / 114 / 115  83 / 30 / 122 / 105  94 / 34 / 155 / 113  108 / 37 / 164 / 135
constexpr TileModel kPairTiles[kTiles] = {
        {256, 192, 7.5f, 1.14f, 0.55f, 11.2f, 1.71f, 0.f, 1},
        {128, 128, 2.3f, 0.556f, 0.25f, 0.8f, 0.72f, 7.f, 0},
        {128, 96, 1.6f, 0.57f, 0.12f, 0.6f, 0.55f, 5.f, 2},
        {128, 96, 5.4f, 0.407f, 0.22f, 4.f, 0.54f, 0.f, 1},
        {64, 64, 3.2f, 0.237f, 0.12f, 0.33f, 0.236f, 4.f, 0},
};

// Halves, measured in the same way at 768 -> 2304 / 768 -> 768 / 768 -> 3072 with GELU, in halves of a step marked *:
//   tokens   256 x 256          256 x 192          128 x 128          128 x 96           *128 x 64
//      512   19 / 18 / 24       16 / 15 / 20       8.7 / 8.1 / 10     8.7 / 8.2 / 10     7.5 / 6.9 / 8.8
//     1280   20 / 19 / 26       16 / 16 / 22       10 / 8.9 / 12      10 / 8.4 / 15      11 / 7.2 / 13
//     2080   20 / 19 / 26       18 / 16 / 22       17 / 8.9 / 19      13 / 8.8 / 24      16 / 7.5 / 22
//     3072   22 / 19 / 28       19 / 16 / 24       17 / 9.2 / 27      22 / 9.8 / 26      21 / 10 / 29
//     4096   24 / 20 / 30       21 / 16 / 27       24 / 9.6 / 29      23 / 9.5 / 31      26 / 11 / 34
//     4992   25 / 20 / 32       22 / 17 / 44       25 / 11 / 36       26 / 12 / 39       30 / 11 / 43
//     8192   45 / 22 / 59       38 / 18 / 53       39 / 16 / 53       38 / 15 / 59       45 / 17 / 66
//    16384   71 / 25 / 95       65 / 23 / 100      75 / 26 / 102      73 / 27 / 113      92 / 32 / 132
constexpr TileModel kHalfTiles[kTiles] = {
        {256, 256, 6.3f, 1.015f, 0.55f, 8.5f, 1.4f, 0.f, 1},
        {256, 192, 4.8f, 0.858f, 0.55f, 6.7f, 1.24f, 0.f, 1},
        {128, 128, 1.3f, 0.567f, 0.25f, 2.4f, 0.434f, 5.f, 0},
        {128, 96, 0.8f, 0.61f, 0.15f, 1.0f, 0.408f, 4.f, 2},
        {128, 64, 3.0f, 0.322f, 0.18f, 1.3f, 0.306f, 4.f, 0},
};

int plan_large(int form, int tokens, int features, int steps) {
    int best = 0;
    float best_us = 0.f;
    for (int i = 0; i < kTiles; ++i) {
        const TileModel &t = has_pairs(form) ? kPairTiles[i] : kHalfTiles[i];
        const long long tiles = (long long) ((tokens + t.tm - 1) / t.tm) * ((features + t.tn - 1) / t.tn);
        const float u = (float) tiles / 256.f;
        const float alone = t.alone + t.alone_step * steps, each = t.each + t.each_step * steps;
        float us = 0.f, left = u;
        if (t.round > 0) {
            const float rounds = (float) (tiles / (256 * t.round));
            left = u - rounds * t.round;
            us = rounds * t.round * each + (rounds > 0.f ? t.start : 0.f);
        }
        if (left > 0.f) {
            const float crowded = alone * (1.f + t.crowd * (t.round == 1 ? left * left : left));
            const float in_turn = t.start + each * left;
            us += left > 1.f && in_turn > crowded ? in_turn : crowded;
        }
        if (form == kPairsGelu) us += 2.f + u * (t.tm * t.tn) * 0.12e-3f;
        if (form == kHalvesGelu) us += 0.6f + u * (t.tm * t.tn) * 0.08e-3f;
        if (i == 0 || us < best_us) best = i, best_us = us;
    }
    return best;
}

template <int FORM>
int launch_tile(const DenseCall<typename FormTypes<FORM>::Value> &c, int tile) {
    if constexpr (has_pairs(FORM)) {
        switch (tile) {
            case 0: return launch_large<FORM, 256, 192, 4, 2, 1, 2, 3>(c);
            case 1: return launch_large<FORM, 128, 128, 4, 2, 1, 2, 3>(c);
            case 2: return launch_large<FORM, 128, 96, 4, 1, 1, 2, 3>(c);
            case 3: return launch_large<FORM, 128, 96, 4, 1, 2, 3, 3>(c);
            default: return launch_large<FORM, 64, 64, 2, 2, 2, 4, 4>(c);
        }
    } else {
        switch (tile) {
            case 0: return launch_large<FORM, 256, 256, 2, 4, 1, 2, 3>(c);
            case 1: return launch_large<FORM, 256, 192, 4, 2, 1, 2, 3>(c);
            case 2: return launch_large<FORM, 128, 128, 4, 2, 1, 2, 3>(c);
            case 3: return launch_large<FORM, 128, 96, 4, 1, 1, 2, 3>(c);
            default: return launch_large<FORM, 128, 64, 4, 1, 2, 3, 3>(c);
        }
    }
}

// (an offset inside a tile's rows has 32 bits, a grid 31)
bool fits_large(int tokens, int features, int in, int step) {
    return in > 0 && in % step == 0 && in <= (1 << 20) && ((long long) tokens / 64 + 1) * (features / 64 + 1) <= 0x7fffffffLL;
}

}  // namespace

// C = fp16(X W^T + bias), or GELU of it; CUBERT_UNSUPPORTED (and nothing launched) where it does not fit.
int dense_large(int tokens, int features, int in, const half_t *x, const half_t *w, const half_t *bias, int activation,
                half_t *out, int ldo, hipStream_t stream) {
    if (!x || !w || !out || tokens < 0 || features < 0 || in < 0 || ldo < features || (activation != 0 && activation != 1)) {
        return CUBERT_BAD_ARGUMENT;
    }
    if (!fits_large(tokens, features, in, kHalfStep) || features % 8 != 0 || ldo % 8 != 0 || !is_aligned(x, 16) ||
        !is_aligned(w, 16) || !is_aligned(out, 16)) {
        return CUBERT_UNSUPPORTED;
    }
    if (tokens == 0 || features == 0) return 0;
    const DenseCall<half_t> c = {w, x, bias, out, ldo, tokens, features, in / kHalfStep, 1.f, 1.f, nullptr, stream};
    const int form = activation == 1 ? kHalvesGelu : kHalves, tile = plan_large(form, tokens, features, c.steps);
    return activation == 1 ? launch_tile<kHalvesGelu>(c, tile) : launch_tile<kHalves>(c, tile);
}

int dense_pairs(int tokens, int features, int in, const half_t *x, const half_t *w, const float *bias, int activation,
                float alpha, float scale, float *out, int ldo, int *overflow, hipStream_t stream) {
    if (!x || !w || !out || tokens < 0 || features < 0 || in < 0 || ldo < features || (activation != 0 && activation != 1)) {
        return CUBERT_BAD_ARGUMENT;
    }
    if (!fits_large(tokens, features, in, kPairStep) || features % (activation == 1 ? kPairBlock : 4) != 0 || ldo % 4 != 0 ||
        (activation == 1 && ldo != features) || !is_aligned(x, 16) || !is_aligned(w, 16) || !is_aligned(out, 16)) {
        return CUBERT_UNSUPPORTED;
    }
    if (tokens == 0 || features == 0) return 0;
    const DenseCall<float> c = {w, x, bias, out, ldo, tokens, features, in / kPairStep, alpha, scale, overflow, stream};
    const int form = activation == 1 ? kPairsGelu : kPairsFloat, tile = plan_large(form, tokens, features, c.steps);
    return activation == 1 ? launch_tile<kPairsGelu>(c, tile) : launch_tile<kPairsFloat>(c, tile);
}

// alpha * x w^T of a narrowing layer as K slices for the LayerNorm behind it, tiles of 128 x 128: a reduction of 3072 in one piece is
// a long time for few tiles.  As many slices as leave a tile to a compute unit, four at most (the LayerNorm reads them all).  With the
// LayerNorm, 3072 -> 768, the best tile in one piece / so, us: 800 tokens 32.7 / 24.0, 1024 34.4 / 25.2, 1280 36.3 / 29.3, 1600 45.1 / 33.8,
// 2000 47.7 / 39.5, 2304 50.6 / 42.7, 2600 53.7 / 46.1, and with two tiles to a unit 3072 60.2 / 63.9; 4096 -> 1024: 640 41.6 / 28.3, 1280 58.8 /
// 41.8, 2000 70.9 / 57.7, 2304 76.7 / 82.1; five slices 3072 -> 768 at 900 tokens 24.9, four 24.5.  768 -> 768 gains nothing (1600 19.3 / 22.7).
// Up to 128 tiles of 64 x 64 the kernel for small requests cuts K (dense_mid.hip): 640 tokens, 3072 -> 768 19.9 us against 23.1 here.
int pairs_slices(int tokens, int features, int in, size_t partial_floats) {
    if (in <= features || in < 64 * kPairStep) return 1;
    if ((long long) ((tokens + 63) / 64) * ((features + 63) / 64) <= 128) return 1;
    const long long tiles = (long long) ((tokens + 127) / 128) * ((features + 127) / 128);
    const long long room = (long long) (partial_floats / ((size_t) tokens * features));
    long long slices = 256 / tiles < 4 ? 256 / tiles : 4;
    slices = slices < room ? slices : room;
    return slices < 1 ? 1 : (int) slices;
}

int dense_pairs_slices(int tokens, int features, int in, const half_t *x, const half_t *w, float alpha, float *partials,
                       size_t partial_floats, int *slices, hipStream_t stream) {
    if (!x || !w || !partials || !slices || tokens < 0 || features < 0 || in < 0) return CUBERT_BAD_ARGUMENT;
    if (tokens == 0 || features == 0 || !fits_large(tokens, features, in, kPairStep) || features % 4 != 0 || !is_aligned(x, 16) ||
        !is_aligned(w, 16) || !is_aligned(partials, 16)) {
        return CUBERT_UNSUPPORTED;
    }
    const int steps = in / kPairStep, want = pairs_slices(tokens, features, in, partial_floats);
    if (want < 2) return CUBERT_UNSUPPORTED;
    const int per = (steps + want - 1) / want;
    *slices = (steps + per - 1) / per;
    const DenseCall<float> c = {w, x, nullptr, partials, features, tokens, features, steps, alpha, 1.f, nullptr, stream, *slices, per};
    return launch_tile<kPairsFloat>(c, 1);
}

// the tile's number, 0 to 4, and its size
int dense_large_plan(int pairs, int tokens, int features, int in, int activation, int *tile, int *tile_tokens,
                     int *tile_features) {
    if (tokens <= 0 || features <= 0 || in <= 0 || !tile || !tile_tokens || !tile_features) return CUBERT_BAD_ARGUMENT;
    const int step = pairs ? kPairStep : kHalfStep;
    if (in % step != 0) return CUBERT_UNSUPPORTED;
    *tile = plan_large((pairs ? kPairsFloat : kHalves) + (activation == 1), tokens, features, in / step);
    const TileModel &t = pairs ? kPairTiles[*tile] : kHalfTiles[*tile];
    *tile_tokens = t.tm, *tile_features = t.tn;
    return 0;
}

}  // namespace cubert
