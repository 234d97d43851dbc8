#include "Transformer.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <string>
#include <stdexcept>

namespace cuBERT {

namespace {
template <typename T>
void upload(T *dst, const T *src, size_t count) {
    if (dst != nullptr) cuBERT::memcpy(dst, src, count * sizeof(T), 1);
}

// device memory for the duration of a scope (a missing weight name throws out of the constructor)
struct ScopedDeviceBuffer {
    void *ptr = nullptr;
    explicit ScopedDeviceBuffer(size_t bytes) : ptr(bytes ? cuBERT::malloc(bytes) : nullptr) {}
    ScopedDeviceBuffer(const ScopedDeviceBuffer &) = delete;
    ScopedDeviceBuffer &operator=(const ScopedDeviceBuffer &) = delete;
    ~ScopedDeviceBuffer() {
        if (ptr != nullptr) cubert_free(ptr);
    }
};
}  // namespace

template <typename T>
Transformer<T>::Transformer(void *cublas, const std::string &var_prefix,
                            const std::unordered_map<std::string, T *> &var, size_t max_batch_size,
                            size_t seq_length, size_t hidden_size, size_t num_hidden_layers,
                            size_t num_attention_heads, size_t intermediate_size)
        : cublas(cublas), max_batch_size(max_batch_size), seq_length(seq_length), hidden_size(hidden_size),
          num_hidden_layers(num_hidden_layers), num_attention_heads(num_attention_heads),
          intermediate_size(intermediate_size), layers(num_hidden_layers) {
    if (num_attention_heads == 0 || hidden_size % num_attention_heads != 0) {
        throw std::invalid_argument("hidden_size must be a multiple of num_attention_heads");
    }
    const size_t H = hidden_size, I = intermediate_size;
    // The re-ordered copies pay off for 2-byte weights (the plain layout makes the few-token kernel read 64-byte
    // pieces): measured 2 us per GEMM at hidden 768; for 4-byte weights the gain is within 5 %, not worth the memory.
    // (Only where the layer sizes are not whole steps of the library's own Dense kernel, which reads them as they are.)
    own_dense = H % (128 / sizeof(T)) == 0 && I % (128 / sizeof(T)) == 0;
    keep_packed = !own_dense && sizeof(T) == 2 && seq_length <= 64 && H % 16 == 0 && I % 16 == 0;
    // The library's fp16 GEMMs are 10-19 % faster with both operands contiguous along the reduction (measured at
    // 32768 tokens on every Dense shape of BERT-base and BERT-large, same bits out); its fp32 GEMMs do not care.
    // Half-precision models therefore keep their Dense kernels [out, in], transposed once here.
    transposed_kernels = sizeof(T) == 2;
    if constexpr (sizeof(T) == 4) {
        const char *setting = std::getenv("CUBERT_FP32_DENSE");
        const std::string dense_mode = setting != nullptr ? setting : "";
        if (dense_mode != "f16x3" && dense_mode != "f32" && dense_mode != "") {
            fprintf(stderr, "cuBERT: CUBERT_FP32_DENSE=%s is not understood (f32 or f16x3); using f32\n", setting);
        }
        // (where the library's own kernel is switched off by CUBERT_GEMM the rows are the ones of the library GEMM)
        int tile = 0, tile_tokens = 0, tile_features = 0;
        pair_dense = H % 32 == 0 && I % 32 == 0 &&
                     cubert_dense_large_plan(1, 1, (int) H, (int) H, 0, &tile, &tile_tokens, &tile_features) == 0;
        split_asked = dense_mode == "f16x3";
        split_dense = two_terms_pay(max_batch_size * seq_length) && (split_asked || (dense_mode == "" && pair_dense));
        if (split_dense) {
            const TwoTermProof proof = two_term_scales(var_prefix, var);
            split_dense = proof.finite && (proof.held || split_asked);
        }
        pair_dense = pair_dense && split_dense;
    }

    if (split_dense) {
        split_overflow = static_cast<int *>(cubert_malloc_host(64));
        if (split_overflow == nullptr) throw std::runtime_error("no page-locked host memory for the two-term overflow flag");
        *split_overflow = 0;
    }

    // Weight names as the reference resolves them (Transformer.cpp:54-101, AttentionSelf.cpp:27-44);
    // a missing name throws std::out_of_range from unordered_map::at, as it does there.
    layout_weights();
    weights.allocate();
    layout_weights();

    void *stream = cuBERT::blas_get_stream(cublas);
    const size_t largest = H * (3 * H > I ? 3 * H : I);
    ScopedDeviceBuffer staging_memory(transposed_kernels || split_dense ? largest * sizeof(T) : 0);
    T *staging = static_cast<T *>(staging_memory.ptr);
    // one Dense kernel, [in, out] on the host, into its place on the device (and its few-token copy)
    auto load_kernel = [&](T *dst, T *few_token_copy, SplitKernel &split, const T *host, size_t in, size_t out, size_t parts = 1) {
        T *plain = transposed_kernels ? staging : dst;
        upload(plain, host, in * out);
        if (keep_packed) cuBERT::pack_few_token_weights(cublas, plain, (int) out, (int) out, (int) in, few_token_copy);
        if (transposed_kernels) {
            cuBERT::transpose(plain, (int) in, (int) out, dst, stream);
            cuBERT::cuda_stream_synchronize(stream);  // the staging buffer is written again by the next upload
        }
        if constexpr (sizeof(T) == 4) {
            if (split_dense) {
                cuBERT::transpose(dst, (int) in, (int) out, staging, stream);
                // (weights are finite and scaled to at most 1024: no overflow flag needed on this side)
                const size_t features = out / parts, terms = pair_dense ? 2 : 3;
                for (size_t part = 0; part < parts; ++part) {
                    const T *rows = staging + part * features * in;
                    half *to = split.weights + part * features * in * terms;
                    const float scale = std::ldexp(1.f, split.exponent[part]);
                    if (pair_dense) {
                        cuBERT::split_pairs(rows, (int) features, (int) in, scale, to, nullptr, stream);
                    } else {
                        cuBERT::split3(rows, (int) features, (int) in, scale, true, to, nullptr, stream);
                    }
                }
                cuBERT::cuda_stream_synchronize(stream);
            }
        }
    };

    std::vector<T> packed(H * 3 * H), packed_bias(3 * H);
    for (size_t l = 0; l < num_hidden_layers; ++l) {
        const std::string p = var_prefix + "/layer_" + std::to_string(l);
        const T *q = var.at(p + "/attention/self/query/kernel"), *qb = var.at(p + "/attention/self/query/bias");
        const T *k = var.at(p + "/attention/self/key/kernel"), *kb = var.at(p + "/attention/self/key/bias");
        const T *v = var.at(p + "/attention/self/value/kernel"), *vb = var.at(p + "/attention/self/value/bias");
        // [in, out] row-major kernels side by side: row i = [Wq[i,:] | Wk[i,:] | Wv[i,:]]
        for (size_t i = 0; i < H; ++i) {
            std::memcpy(&packed[i * 3 * H], q + i * H, H * sizeof(T));
            std::memcpy(&packed[i * 3 * H + H], k + i * H, H * sizeof(T));
            std::memcpy(&packed[i * 3 * H + 2 * H], v + i * H, H * sizeof(T));
        }
        std::memcpy(&packed_bias[0], qb, H * sizeof(T));
        std::memcpy(&packed_bias[H], kb, H * sizeof(T));
        std::memcpy(&packed_bias[2 * H], vb, H * sizeof(T));
        Layer &w = layers[l];
        load_kernel(w.qkv_kernel, w.qkv_packed, w.qkv_split, packed.data(), H, 3 * H, 3);
        upload(w.qkv_bias, packed_bias.data(), 3 * H);
        if constexpr (sizeof(T) == 4) {
            if (split_dense) {
                for (size_t i = 0; i < 3 * H; ++i) packed_bias[i] = std::ldexp(packed_bias[i], w.qkv_split.shift(i / H));
                upload(w.qkv_split_bias, packed_bias.data(), 3 * H);
            }
        }
        load_kernel(w.attention_output_kernel, w.attention_output_packed, w.attention_output_split,
                    var.at(p + "/attention/output/dense/kernel"), H, H);
        upload(w.attention_output_bias, var.at(p + "/attention/output/dense/bias"), H);
        upload(w.attention_norm_beta, var.at(p + "/attention/output/LayerNorm/beta"), H);
        upload(w.attention_norm_gamma, var.at(p + "/attention/output/LayerNorm/gamma"), H);
        load_kernel(w.intermediate_kernel, w.intermediate_packed, w.intermediate_split,
                    var.at(p + "/intermediate/dense/kernel"), H, I);
        upload(w.intermediate_bias, var.at(p + "/intermediate/dense/bias"), I);
        load_kernel(w.output_kernel, w.output_packed, w.output_split, var.at(p + "/output/dense/kernel"), I, H);
        upload(w.output_bias, var.at(p + "/output/dense/bias"), H);
        upload(w.output_norm_beta, var.at(p + "/output/LayerNorm/beta"), H);
        upload(w.output_norm_gamma, var.at(p + "/output/LayerNorm/gamma"), H);
    }
    cuBERT::cuda_stream_synchronize(stream);  // nothing reads the staging buffer after this

    layout_buffers();
    buffers.allocate();
    layout_buffers();
}

template <typename T>
Transformer<T>::~Transformer() {
    cubert_free_host(split_overflow);  // null is accepted
}

template <typename T>
bool Transformer<T>::two_term_overflowed() {
    if (split_overflow == nullptr || *static_cast<volatile int *>(split_overflow) == 0) return false;
    *split_overflow = 0;
    return true;
}

// The scales of every layer's operands, each the largest power of two that keeps within fp16 what the operand cannot exceed, || || the
// 2-norm:
//   - a LayerNorm's result: norm_result;
//   - the context, an average of rows of V: ||row|| times the norm of the value kernel's largest column, + its largest |bias|;
//   - GELU's result: the same with the intermediate kernel;
// and those of the kernels.  finite: whether all weights are numbers (two terms, which are clamped to fp16's range, would make finite
// results of the others); held: whether every bound allows the smallest scale and two terms at these scales hold every layer (layer
// 0's attention: set_input).  (The bounds allow 1 % for rounding.  A variance that cancellation makes too small can still leave them:
// the overflow flag stays.)
template <typename T>
typename Transformer<T>::TwoTermProof Transformer<T>::two_term_scales(const std::string &var_prefix,
                                                                      const std::unordered_map<std::string, T *> &var) {
    TwoTermProof proof;
    if constexpr (sizeof(T) == 4) {
        const size_t H = hidden_size, I = intermediate_size;
        DenseInput input;
        for (size_t l = 0; l < num_hidden_layers; ++l) {
            const std::string p = var_prefix + "/layer_" + std::to_string(l);
            Layer &w = layers[l];
            if (l > 0) {
                proof.add(attention_scales(p, var, input, w));
            } else {
                auto largest = [&](const char *name) { return largest_size(var.at(p + name + "/kernel"), H * H); };
                proof.finite = set_attention_exponents(w, largest("/attention/self/query"), largest("/attention/self/key"),
                                                       largest("/attention/self/value"), largest("/attention/output/dense"));
            }
            const DenseInput norm = norm_result(var.at(p + "/attention/output/LayerNorm/gamma"),
                                                var.at(p + "/attention/output/LayerNorm/beta"), H);
            const DenseProducts inner = dense_products(var.at(p + "/intermediate/dense/kernel"), H, I, norm);
            const T *bias = var.at(p + "/intermediate/dense/bias");
            DenseInput gelu;
            gelu.element = norm.row * inner.column + largest_or_nan(bias, I);
            gelu.squares.resize(I);
            for (size_t j = 0; j < I; ++j) gelu.squares[j] = (float) gelu_mean_square(inner.squares[j], bias[j]);
            const DenseProducts output = dense_products(var.at(p + "/output/dense/kernel"), I, H, gelu);
            w.intermediate_split.set_exponent(inner.largest_weight);
            w.output_split.set_exponent(output.largest_weight);
            const bool norm_fits = set_scale(w.norm_scale, norm.element), inner_fits = set_scale(w.inner_scale, gelu.element);
            proof.add({std::isfinite(inner.largest_weight) && std::isfinite(output.largest_weight),
                       norm_fits && inner_fits && two_terms_hold(inner, w.norm_scale, w.intermediate_split.exponent[0]) &&
                           two_terms_hold(output, w.inner_scale, w.output_split.exponent[0])});
            input = norm_result(var.at(p + "/output/LayerNorm/gamma"), var.at(p + "/output/LayerNorm/beta"), H);
        }
    }
    return proof;
}

template <typename T>
void Transformer<T>::layout_weights() {
    const size_t H = hidden_size, I = intermediate_size;
    for (Layer &w : layers) {
        w.qkv_kernel = weights.take<T>(H * 3 * H);
        w.qkv_bias = weights.take<T>(3 * H);
        w.attention_output_kernel = weights.take<T>(H * H);
        w.attention_output_bias = weights.take<T>(H);
        w.attention_norm_beta = weights.take<T>(H);
        w.attention_norm_gamma = weights.take<T>(H);
        w.intermediate_kernel = weights.take<T>(H * I);
        w.intermediate_bias = weights.take<T>(I);
        w.output_kernel = weights.take<T>(I * H);
        w.output_bias = weights.take<T>(H);
        w.output_norm_beta = weights.take<T>(H);
        w.output_norm_gamma = weights.take<T>(H);
        if (keep_packed) {
            w.qkv_packed = weights.take<T>(cubert_gemm_skinny_packed_elements(3 * (int) H, (int) H));
            w.attention_output_packed = weights.take<T>(cubert_gemm_skinny_packed_elements((int) H, (int) H));
            w.intermediate_packed = weights.take<T>(cubert_gemm_skinny_packed_elements((int) I, (int) H));
            w.output_packed = weights.take<T>(cubert_gemm_skinny_packed_elements((int) H, (int) I));
        }
        if (split_dense) {
            const size_t terms = pair_dense ? 2 : 3;
            w.qkv_split.weights = weights.take<half>(terms * H * 3 * H);
            w.attention_output_split.weights = weights.take<half>(terms * H * H);
            w.intermediate_split.weights = weights.take<half>(terms * H * I);
            w.output_split.weights = weights.take<half>(terms * I * H);
            w.qkv_split_bias = weights.take<T>(3 * H);
        }
    }
}

template <typename T>
void Transformer<T>::layout_buffers() {
    const size_t M = max_batch_size * seq_length, H = hidden_size;
    // 64 elements between one token's Q | K | V row and the next: the attention kernels read 128-byte pieces of these
    // rows at the row pitch, and a pitch of 3 * hidden elements (6 KB for BERT-large in fp16) spreads those pieces
    // badly over the memory channels.  Measured at 256 sequences x 16 heads x 128 keys, fp16, with and without the
    // padding in alternation on one box: attention kernel 57.4 -> 51.3 us, forward pass 20.34 -> 20.24 ms; BERT-base
    // shapes (pitch 4.5 KB fp16, 9 KB fp32) move by less than the run-to-run noise.
    qkv_ld = 3 * H + 64;
    qkv_out = buffers.take<T>(M * qkv_ld);
    context_out = buffers.take<T>(M * H);
    attention_order = buffers.take<int>(8 * max_batch_size);  // indices, then a record of live tiles per position
    attention_output = buffers.take<T>(M * H);
    intermediate_output = buffers.take<T>(M * intermediate_size);
    layer_output[0] = buffers.take<T>(M * H);
    layer_output[1] = buffers.take<T>(M * H);
    if (split_dense && pair_dense) {
        split_operand = buffers.take<half>(M * 2 * H);
        split_intermediate = buffers.take<half>(M * 2 * intermediate_size);
    } else if (split_dense) {
        split_operand = buffers.take<half>(M * 3 * (H > intermediate_size ? H : intermediate_size));
    }
    if (seq_length <= 64 || own_dense) few_token_partials = buffers.take<float>(kFewTokenPartialFloats);
}

template <typename T>
T *Transformer<T>::scores() {
    if (attention_scores == nullptr) {
        const size_t count = max_batch_size * num_attention_heads * seq_length * seq_length;
        score_memory.take<T>(count);
        score_memory.allocate();
        attention_scores = score_memory.take<T>(count);
    }
    return attention_scores;
}

template <typename T>
T *Transformer<T>::compute(size_t batch_size, T *input_gpu, int8_t *attention_mask) {
    _pre_compute(batch_size);
    return _in_compute(batch_size, input_gpu, attention_mask);
}

template <typename T>
void Transformer<T>::_pre_compute(size_t) {}

// scores[b, a, q, k] = (1/sqrt d) * sum_j Q[b, q, a, j] K[b, k, a, j];  softmax with mask;
// ctx[b, q, a, :] = sum_k p[b, a, q, k] V[b, k, a, :].   Q, K, V are column blocks of qkv[M, 3H].
// The contractions run as one matrix-core launch each where the shape allows.  Otherwise: the (b, a)
// problems have two strides (b: seq*3H, a: d), a strided-batched GEMM has one, so the shorter of the two
// axes is looped on the host and the longer one is the GEMM batch.
template <typename T>
bool Transformer<T>::attention(size_t batch_size, const T *qkv, const int8_t *mask, half *split_context, float scale,
                               float score_unscale) {
    void *stream = cuBERT::blas_get_stream(cublas);
    const int S = (int) seq_length, A = (int) num_attention_heads, H = (int) hidden_size, d = H / A;
    const int B = (int) batch_size, ld = (int) qkv_ld;
    const float alpha = (float) (1.0 / std::sqrt((double) d)) * score_unscale;
    const T *Q = qkv, *K = qkv + H, *V = qkv + 2 * H;
    const long long seq_stride = (long long) S * ld, head_stride = d;
    const long long score_b = (long long) A * S * S, score_a = (long long) S * S;

    // One launch with the score tensor held in registers where the shape allows (seq_length <= 512, K and V
    // of a head within LDS).  CUBERT_ATTENTION=split in the
    // environment keeps the three-operator path below (scores, mask + softmax, context) for every shape.
    static const bool split_only = [] {
        const char *e = std::getenv("CUBERT_ATTENTION");
        return e != nullptr && std::string(e) == "split";
    }();
    if (!split_only && fused_attention_fits) {
        Timed t(profiler, Profiler::kAttentionFused, stream);
        if constexpr (sizeof(T) == 4) {
            if (split_context != nullptr &&
                (pair_dense ? cuBERT::attention_fused_split_pairs(Q, K, V, ld, mask, scale, split_context, alpha, B, A, S, d,
                                                                  split_overflow, stream)
                            : cuBERT::attention_fused_split3(Q, K, V, ld, mask, scale, split_context, alpha, B, A, S, d,
                                                             split_overflow, stream))) {
                return true;
            }
        }
        if (cuBERT::attention_fused(Q, K, V, ld, mask, context_out, H, alpha, B, A, S, d, stream,
                                    order_ready ? attention_order : nullptr)) {
            return false;
        }
        fused_attention_fits = false;  // seq_length and head size are fixed per model: do not ask again
        t.cancel();
    }

    T *score_tensor = scores();
    const bool loop_heads = A <= B;
    const int outer = loop_heads ? A : B, inner = loop_heads ? B : A;
    const long long in_outer = loop_heads ? head_stride : seq_stride, in_inner = loop_heads ? seq_stride : head_stride;
    const long long sc_outer = loop_heads ? score_a : score_b, sc_inner = loop_heads ? score_b : score_a;
    const long long ctx_outer = loop_heads ? (long long) d : (long long) S * H;
    const long long ctx_inner = loop_heads ? (long long) S * H : (long long) d;

    {
        Timed t(profiler, Profiler::kAttentionGemm, stream);
        if (!cuBERT::attention_scores(Q, K, ld, score_tensor, alpha, B, A, S, d, stream)) {
            for (int o = 0; o < outer; ++o) {
                // column-major: scores_ba (S_k x S_q, ld S) = K_ba^T (d x S_k, ld 3H)^T * Q_ba (d x S_q, ld 3H)
                cuBERT::blas_gemm_strided_batch(cublas, true, false, S, S, d, alpha, K + o * in_outer, ld, in_inner,
                                                Q + o * in_outer, ld, in_inner, 0.f, score_tensor + o * sc_outer,
                                                S, sc_inner, inner);
            }
        }
    }
    {
        Timed t(profiler, Profiler::kMaskScaleSoftmax, stream);
        cuBERT::mask_scale_softmax_(score_tensor, mask, 1.0f, B, A, S, stream);
    }
    Timed t(profiler, Profiler::kAttentionGemm, stream);
    if (!cuBERT::attention_context(score_tensor, V, ld, context_out, H, B, A, S, d, stream)) {
        for (int o = 0; o < outer; ++o) {
            // column-major: ctx_ba (d x S_q, ld H) = V_ba (d x S_k, ld 3H) * p_ba (S_k x S_q, ld S)
            cuBERT::blas_gemm_strided_batch(cublas, false, false, d, S, S, 1.f, V + o * in_outer, ld, in_inner,
                                            score_tensor + o * sc_outer, S, sc_inner, 0.f,
                                            context_out + o * ctx_outer, H, ctx_inner, inner);
        }
    }
    return false;
}

// Whether a Dense layer of this size runs on the library's own kernel (kernels/dense_mid.hip) instead of a library
// GEMM or the few-token kernel: up to where they cross, which depends on what follows.  A library GEMM adds the bias of
// Q|K|V by itself, pays a launch for GELU, and leaves K uncut in front of a LayerNorm.  A layer with its GELU or
// LayerNorm, weights from a model's worth of them, library against own, us:
//   half Q|K|V      512 in: 1280 tokens 8.7 / 7.3; 640: 1024 8.2 / 8.4, 1152 9.0 / 11.0; 768: 384 7.6 / 6.1, 896
//                   9.0 / 9.1, 1024 11.1 / 12.0, 1280 10.6 / 13.0; 1024: 512 10.2 / 9.6, 640 10.2 / 10.7, 896
//                   11.8 / 13.7; 1536: 256 15.5 / 14.0, 320 12.4 / 13.9
//   attention out   1024: 1280 13.2 / 12.8; 1536: 640 12.8 / 11.6, 768 15.4 / 16.9; 2048: 640 17.3 / 20.7
//   intermediate    768 in: 1280 19.1 / 16.6; 1024 in: 896 20.7 / 19.5; 2048 in: 320 23.7 / 23.5
//   output          3072 in: 1280 19.0 / 18.2; 4096 in: 896 20.8 / 18.5
//   attention out   fp32, 768: 320 10.5 / 9.9; 1024: 256 12.1 / 11.5, 320 14.5 / 15.3
//   intermediate    768 in: 320 20.0 / 18.2; 1024 in: 160 20.8 / 19.2, 224 23.7 / 23.1, 320 29.0 / 29.7
//   output          3072 in: 256 21.6 / 19.5, 320 22.0 / 22.9; 4096 in: 160 26.0 / 20.4
// fp32 Q|K|V by whole requests, whose weights come from memory rather than from a cache, library against own: BERT-base 120
// tokens 652 / 644, 160 640 / 634, 264 955 / 935, 300 945 / 950, 320 888 / 901; BERT-large 96 1441 / 1449, 128 1447 / 1459.
// fp32, more than 1024 inputs: only as K slices for the LayerNorm.  Otherwise a few workgroups walk all of K (32 tokens,
// 6144 -> 1536 with its LayerNorm: 41.6 us, few-token kernel 23.5) in sums longer than the few-token kernel's (2.6e-7
// against 1.4e-7 of float64; 1536 -> 4608: 1.43e-7 against 1.33e-7).
// fp32, at most 32 tokens, 640 inputs or more and no more inputs than outputs: the few-token kernel, which cuts K for
// these, is the faster one where no GELU follows (Q|K|V of 768 6.7 against 7.2 us, of 1024 8.6 / 8.8, of 512 6.1 / 5.7;
// attention output with its LayerNorm 768 6.2 / 6.4, 1024 7.2 / 7.5, 512 5.3 / 5.2; the intermediate layer of 768 9.0 / 7.4,
// of 1024 8.7 / 9.0; output 768 9.9 / 9.5, 1024 10.3 / 9.8).
bool own_dense_is_best(bool half_precision, int tokens, int out_features, int in_features, DenseUse use, bool as_slices) {
    const double products = (double) tokens * out_features * in_features;
    const bool narrowing = in_features > out_features;
    if (half_precision) {
        if (tokens > 1280) return false;
        if (use == DenseUse::kPlain) return products <= (tokens <= 1024 ? 1.65e9 : 1.3e9);
        return products <= (use == DenseUse::kGelu || narrowing ? 3.05e9 : 1.7e9);
    }
    if (in_features > 1024 && !(use == DenseUse::kNorm && as_slices)) return false;
    if (tokens <= 32 && in_features >= 640 && !narrowing && use != DenseUse::kGelu) return false;
    if (tokens > 320) return false;
    return products <= (use == DenseUse::kPlain ? 4.7e8 : use == DenseUse::kGelu ? 7.6e8 : 7.0e8);
}

// Whether a half Dense layer runs on the library's own kernel for large requests (kernels/dense_large.hip), which applies bias
// and GELU, instead of the one for small requests or a library GEMM (with its GELU pass).  What that saves, us a layer (negative:
// what it costs), by whole requests of 12 layers (1024 inputs: 24) with the one layer on the one kernel or the other in
// alternation.  Against the small kernel one figure; against the library's GEMM two, hipBLASLt 1.2 of ROCm 7.2 / the copy that a
// PyTorch for ROCm 7.0 brings and that a process uses that has loaded PyTorch first: their choices differ by more than the lines.
//   Q|K|V           512 in: 1024 tokens -0.9, 1280 -0.3, 1408 2.3 / 4.8, 4096 0.9 / 3.8, 5120 -0.4 / 2.2; 576: 1024 1.3, 1152 -0.7,
//                   1280 1.7; 640: 640 1.5, 3072 0.0 / 1.4, 3584 -0.8 / 0.4; 768: 512 1.5, 640 1.1, 1280 1.0, 1312 3.5 / 1.9, 2048
//                   1.9 / 5.0, 2560 0.2 / 2.4, 2816 -0.3 / -1.2, 4096 0.4 / 0.6, 8192 -4.9 / -2.8; 1024: 512 0.8, 1152 -1.4 / 0.1,
//                   1408 0.6 / 1.2, 2048 -1.9 / -1.2; 1536: 512 -4.6 / -1.2; 256: 16384 2.6 / 9.2; 128: 65536 13 / 5.9
//   intermediate    512 in: 1024 -1.5, 1152 1.0, 1536 5.0 / 7.2, 3072 0.4 / 2.1, 32768 20 / 11; 640: 640 0.8; 768: 512 0.3, 768 1.0,
//                   1280 4.2 / 3.4, 1312 6.2 / 7.3, 4096 6.8 / 8.5, 16384 16 / 11, 24576 15 / 21, 32768 14 / 12; 1024: 512 1.0, 1024
//                   4.6 / 6.4, 2048 0.2 / 2.0, 8192 5.7 / 2.9, 14336 -1.0 / 1.4, 16384 -1.1 / 4.7, 32768 0.4 / 5.7; 1536: 512 -0.2 /
//                   2.2, 6144 8.0 / 9.1; 2048: 512 5.9 / 4.7, 1024 -0.1 / 2.9, 2048 1.8 / 2.3, 2304 -0.9 / -2.1, 2560 -14 / -4.9, 3072
//                   -10 / -6.2, 4096 1.1 / 5.4; 256: 8192 3.8 / 5.4; 128: 32768 14 / 9.6
//   attention out   512 in: 1280 -2.3, 1408 0.8 / 2.3, 3072 -0.5 / 0.9, 4096 -0.5 / 1.9, 8192 0.4 / 2.4, 16384 -4.1 / -0.8; 640: 3072
//                   0.8 / 1.8, 3584 -0.8 / 0.3, 8192 -0.1 / 1.7; 768: 1280 -0.6, 1312 1.7 / 0.5, 2048 1.2 / 1.8, 2688 1.0 / 1.5, 3072
//                   -1.1 / 0.8, 4096 -0.5 / 1.5, 4992 -0.1 / 1.6, 6144 -0.7 / 1.6, 12288 -2.9 / 8.0, 20480 -3.4 / -4.4; 896: 1408
//                   -0.5 / 1.5, 2048 0.6 / 2.6; 1024: 1312 0.2 / 3.4, 1536 -1.0 / 2.5, 2048 0.2 / 2.8, 4096 -0.8 / 2.4, 6144 -1.7 /
//                   -0.5; 256: 8192 1.5 / 3.9; 128: 8192 2.4 / 1.2
//   output          3072 in: 1536 -1.8 / -1.4, 2048 -1.3 / -0.5, 2560 -0.2 / 0.5, 4096 -2.7 / -3.0, 8192 -7.2 / -6.7: left to the library
// The lines are where the sum of the two changes sign.
static bool large_dense_is_best(int tokens, int out_features, int in_features, DenseUse use) {
    const double products = (double) tokens * out_features * in_features;
    if (tokens < 512) return false;
    switch (use) {
        // (narrow layers: the small kernel is ahead for all of its 1280 tokens)
        case DenseUse::kPlain: return products > 7.5e8 && products <= 4.6e9 && in_features <= 1024 && (in_features > 512 || tokens > 1280);
        case DenseUse::kGelu: return products > 1.2e9 && products <= (in_features <= 1536 ? 7e10 : 3.5e10);
        default: return in_features <= out_features && products <= 4.4e9 && tokens <= 8192;
    }
}

DenseRoute dense_route(bool half_precision, int tokens, int out_features, int in_features, DenseUse use, bool as_slices) {
    const bool small = own_dense_is_best(half_precision, tokens, out_features, in_features, use, as_slices);
    const bool large = half_precision && !(small && use == DenseUse::kNorm) &&
                       large_dense_is_best(tokens, out_features, in_features, use);
    return large ? DenseRoute::kLarge : small ? DenseRoute::kSmall : DenseRoute::kOther;
}

// CUBERT_FEW_TOKEN_SLICES=0 in the environment keeps the Dense kernels of small requests adding their own K slices.
static bool few_token_slices_enabled() {
    static const bool on = [] {
        const char *e = std::getenv("CUBERT_FEW_TOKEN_SLICES");
        return e == nullptr || std::string(e) != "0";
    }();
    return on;
}

static DenseUse use_of(Profiler::Kind kind) {
    return kind == Profiler::kDenseQkv            ? DenseUse::kPlain
           : kind == Profiler::kDenseIntermediate ? DenseUse::kGelu
                                                  : DenseUse::kNorm;
}

template <typename T>
DenseRoute Transformer<T>::route_of(int tokens, int out_features, int in_features, Profiler::Kind kind) const {
    if (!own_dense) return DenseRoute::kOther;
    return dense_route(sizeof(T) == 2, tokens, out_features, in_features, use_of(kind),
                       own_slices_to_norm && few_token_slices_enabled());
}

// One Dense layer.  The bias goes into the GEMM only where the caller asks for it (bias_in_gemm: the Q/K/V
// projection, whose consumer has no fused bias) or where the few-token kernel applies it together with the GELU;
// otherwise it is left to the fused kernel that follows (which then reads the GEMM output once anyway).
template <typename T>
bool Transformer<T>::dense(int out_features, int tokens, int in_features, const T *kernel, const T *packed, const T *in,
                           T *out, const T *bias, bool bias_in_gemm, bool gelu, Profiler::Kind kind, int ld_out) {
    void *stream = cuBERT::blas_get_stream(cublas);
    Timed t(profiler, profiler != nullptr ? profiler->dense_kind(kind) : Profiler::kDenseGemm, stream);
    if (ld_out == 0) ld_out = out_features;
    const DenseRoute route = route_of(tokens, out_features, in_features, kind);
    if constexpr (sizeof(T) == 2) {
        const bool with_bias = bias_in_gemm || gelu;
        if (route == DenseRoute::kLarge && cuBERT::dense_large(tokens, out_features, in_features, in, kernel,
                                                               with_bias ? bias : nullptr, gelu, out, ld_out, stream)) {
            return with_bias;
        }
    }
    if (route == DenseRoute::kSmall) {
        const bool with_bias = bias_in_gemm || gelu;
        if (cuBERT::dense_mid(tokens, out_features, in_features, in, in_features, kernel,
                              transposed_kernels ? in_features : out_features, with_bias ? bias : nullptr, gelu, out, ld_out,
                              stream)) {
            return with_bias;
        }
    }
    // (the few-token kernel reads [in, out] kernels or its own copy of them, not transposed ones)
    if (tokens <= few_token_limit(kind) && (packed != nullptr || (!transposed_kernels && (gelu || tokens > 32) && dense_gelu_fits))) {
        const bool with_bias = bias_in_gemm || gelu;
        if (cuBERT::dense_few_tokens(cublas, out_features, tokens, in_features, kernel, out_features, packed, in,
                                     in_features, out, ld_out, with_bias ? bias : nullptr, gelu)) {
            return with_bias;
        }
        if (gelu) dense_gelu_fits = false;  // the layer sizes are fixed per model: do not ask again
    }
    cuBERT::blas_gemm(cublas, transposed_kernels, false, out_features, tokens, in_features, 1.f, kernel,
                      transposed_kernels ? in_features : out_features, in, in_features, 0.f, out, ld_out,
                      bias_in_gemm ? bias : nullptr);
    return bias_in_gemm;
}

// Whether a Dense layer over rows of pairs runs on the kernel for small requests (kernels/dense_mid.hip) instead of the one for
// large ones: as long as no compute unit has two of its 64 x 64 tiles.  A layer, with its GELU or LayerNorm, small / large, us:
//   Q|K|V           768 in: 120 tokens 7.4 / 10.3, 300 9.7 / 10.3, 384 9.8 / 10.4, 512 14.9 / 12.5; 1024: 300 11.7 / 12.8, 384 18.6 / 16.0
//   attention out   768: 120 7.5 / 12.0, 640 10.0 / 12.9, 1280 14.3 / 15.0; 1024: 800 14.6 / 16.2, 1024 18.4 / 17.8, 1280 23.8 / 22.1
//   intermediate    768 in: 120 8.0 / 11.1, 300 10.8 / 11.1, 384 15.9 / 13.7; 1024: 200 12.5 / 13.2, 300 19.7 / 18.6
//   output          3072 in: 120 10.7 / 32, 640 19.9 / 33.5, 1280 30.9 / 34.6; 4096: 300 19.0 / 40.0, 1024 37.4 / 44.1, 1280 59.7 / 64.3;
//                   in K slices for the LayerNorm up to 128 of these tiles (pairs_slices in kernels/dense_large.hip)
static bool small_pairs_are_best(int tokens, int out_features) {
    return (long long) ((tokens + 63) / 64) * ((out_features + 63) / 64) <= 256;
}

// Up to 64 tokens the fp32 kernels stay: theirs are the shorter sums (tokens of BERT-base against float64, 1e-7 of their 2-norm,
// pairs / fp32: 32 tokens 3.4 / 3.2, 64 3.4 / 3.2; 96 3.5 / 5.1, 120 3.4 / 4.8, 256 3.5 / 5.0, 300 3.5 / 11, 640 4.2 / 12.7, 1600 6.7 /
// 12.7), and no slower (us a request: 32 476 / 454, 64 485 / 487).  Above, BERT-base: 96 506 / 546, 100 633 / 734, 160 633 / 684, 256 720 /
// 852, 300 798 / 1024, 321 760 / 1128, 352 (11 x 32) 732 / 1165, 383 875 / 1285, 384 745 / 1205.  Narrow layers, whose launches are all there is to them, four layers, us, pairs / fp32: hidden
// 256 192 tokens 157 / 147, 320 155 / 151, 640 190 / 245; 512 96 159 / 161, 192 186 / 210; and, where the LayerNorm kernel writes no rows
// of pairs (no multiple of 256) and a pass of its own does, 128 320 174 / 141, 4096 263 / 298; 384 192 189 / 177, 512 232 / 281; 640 96 182 / 174, 192 217 / 230.
template <typename T>
bool Transformer<T>::two_terms_pay(size_t tokens) const {
    if (split_asked && tokens >= kTwoTermMinTokens) return true;
    return pair_dense && tokens > 64 && (double) tokens * hidden_size * hidden_size >= (hidden_size % 256 == 0 ? 3.8e7 : 6.7e7);
}

template <typename T>
void Transformer<T>::make_operand(const T *in, int tokens, int width, float scale) {
    if constexpr (sizeof(T) == 4) {
        void *stream = cuBERT::blas_get_stream(cublas);
        Timed t(profiler, Profiler::kDenseSplit, stream);
        if (pair_dense) {
            cuBERT::split_pairs(in, tokens, width, scale, split_operand, split_overflow, stream);
        } else {
            cuBERT::split3(in, tokens, width, scale, false, split_operand, split_overflow, stream);
        }
    }
}

template <typename T>
void Transformer<T>::dense_split(int out_features, int tokens, int in_features, const SplitKernel &kernel, float scale,
                                 const T *in, T *out, const T *bias, Profiler::Kind kind, int ld_out, float inner_scale) {
    if (ld_out == 0) ld_out = out_features;
    if constexpr (sizeof(T) == 4) {
        void *stream = cuBERT::blas_get_stream(cublas);
        if (in != nullptr) make_operand(in, tokens, in_features, scale);
        Timed t(profiler, profiler != nullptr ? profiler->dense_kind(kind) : Profiler::kDenseGemm, stream);
        if (pair_dense) {
            const bool gelu = kind == Profiler::kDenseIntermediate;
            if (small_pairs_are_best(tokens, out_features) &&
                cuBERT::dense_pairs_small(tokens, out_features, in_features,
                                          kind == Profiler::kDenseOutput ? split_intermediate : split_operand, kernel.weights, bias,
                                          gelu, kernel.unscale() / scale, inner_scale,
                                          gelu ? reinterpret_cast<float *>(split_intermediate) : out, ld_out, split_overflow,
                                          stream)) {
                return;
            }
            cuBERT::dense_pairs(tokens, out_features, in_features, kind == Profiler::kDenseOutput ? split_intermediate : split_operand,
                                kernel.weights, bias, gelu, kernel.unscale() / scale, inner_scale,
                                gelu ? reinterpret_cast<float *>(split_intermediate) : out, ld_out, split_overflow, stream);
            return;
        }
        cuBERT::blas_gemm_f16_f32(cublas, true, false, out_features, tokens, 3 * in_features,
                                  kernel.unscale() / scale, kernel.weights, 3 * in_features, split_operand, 3 * in_features, 0.f, out,
                                  ld_out, bias);
    } else {
        throw std::logic_error("the two-term fp16 Dense form is for fp32 models");
    }
}

template <typename T>
bool Transformer<T>::norm_split(const T *residual, T *inout, int tokens, const T *bias, const T *beta, const T *gamma,
                               float scale) {
    if constexpr (sizeof(T) == 4) {
        void *stream = cuBERT::blas_get_stream(cublas);
        const int H = (int) hidden_size;
        return pair_dense ? cuBERT::layer_norm_split_pairs(residual, inout, tokens, H, bias, beta, gamma, scale, split_operand,
                                                           split_overflow, stream)
                          : cuBERT::layer_norm_split3(residual, inout, tokens, H, bias, beta, gamma, scale, split_operand,
                                                      split_overflow, stream);
    } else {
        throw std::logic_error("the two-term fp16 Dense form is for fp32 models");
    }
}

template <typename T>
bool Transformer<T>::norm_to_operand(const T *residual, T *inout, int tokens, const T *bias, const T *beta, const T *gamma,
                                     float scale) {
    Timed t(profiler, Profiler::kBiasResLayerNorm, cuBERT::blas_get_stream(cublas));
    if (scale > 0.f && norm_writes_operand) {
        if (norm_split(residual, inout, tokens, bias, beta, gamma, scale)) return true;
        norm_writes_operand = false;  // the hidden size is fixed per model: do not ask again
    }
    cuBERT::layer_norm_(residual, inout, tokens, (int) hidden_size, bias, beta, gamma, cuBERT::blas_get_stream(cublas));
    return false;
}

template <typename T>
bool Transformer<T>::dense_split_norm(int tokens, int in_features, const SplitKernel &kernel, float scale, const T *bias,
                                      const T *residual, const T *beta, const T *gamma, T *out, Profiler::Kind kind,
                                      float next_scale) {
    if constexpr (sizeof(T) == 4) {
        void *stream = cuBERT::blas_get_stream(cublas);
        const int H = (int) hidden_size;
        if (pair_dense && own_slices_to_norm && few_token_slices_enabled()) {
            int slices = 0;
            bool done = false;
            // (the two-term form has GELU's result as rows of pairs, elsewhere: room that grows with the model; one opened for few tokens
            // has more in the buffer for small requests, 128 tokens, 768 hidden and 768 intermediate 432 -> 415 us a request)
            float *partials = intermediate_output;
            size_t room = max_batch_size * seq_length * intermediate_size;
            if (few_token_partials != nullptr && room < kFewTokenPartialFloats) partials = few_token_partials, room = kFewTokenPartialFloats;
            {
                Timed t(profiler, profiler != nullptr ? profiler->dense_kind(kind) : Profiler::kDenseGemm, stream);
                done = cuBERT::dense_pairs_slices(tokens, H, in_features,
                                                  kind == Profiler::kDenseOutput ? split_intermediate : split_operand,
                                                  kernel.weights, kernel.unscale() / scale, partials,
                                                  room, &slices, stream);
                if (!done) t.cancel();
            }
            if (done) {
                Timed t(profiler, Profiler::kBiasResLayerNorm, stream);
                if (next_scale > 0.f && norm_writes_operand &&
                    cuBERT::layer_norm_slices_pairs(out, partials, slices, residual, bias, beta, gamma, tokens, H, next_scale,
                                                    split_operand, split_overflow, stream)) {
                    return true;
                }
                if (cuBERT::layer_norm_slices(out, partials, slices, residual, bias, beta, gamma, tokens, H, stream)) {
                    return false;
                }
                t.cancel();
                own_slices_to_norm = false;  // the hidden size is fixed per model: do not ask again
            }
        }
        dense_split(H, tokens, in_features, kernel, scale, nullptr, out, nullptr, kind);
        return norm_to_operand(residual, out, tokens, bias, beta, gamma, next_scale);
    } else {
        throw std::logic_error("the two-term fp16 Dense form is for fp32 models");
    }
}

// Up to how many tokens a Dense layer that the own Dense kernel does not take runs on the few-token kernel.  32 for all of
// them; 64 where the kernel with two
// blocks of 32 tokens per wavefront is ahead of the library.  Measured at BERT-base, batch 2 x seq 32, a launch
// event-timed inside the forward pass, library against kernel -- fp32: attention output 9.1 / 7.6 us, output
// 20.4 / 15.1 us, but Q|K|V 11.7 / 12.5 and intermediate + GELU 16.4 / 18.7 (the fp32 MFMAs of a second token block
// cost what the library's tiles do not); fp16: attention output 8.6 / 6.5, intermediate + GELU 14.6 / 10.7, output
// 10.4 / 7.7, Q|K|V 8.5 / 10.1.  Forward pass 0.665 -> 0.61 ms (fp32), 0.541 -> 0.423 ms (fp16).
template <typename T>
int Transformer<T>::few_token_limit(Profiler::Kind kind) const {
    switch (kind) {
        case Profiler::kDenseAttentionOutput:
        case Profiler::kDenseOutput: return 64;
        case Profiler::kDenseIntermediate: return sizeof(T) == 2 ? 64 : 32;
        default: return 32;
    }
}

template <typename T>
void Transformer<T>::dense_norm(int tokens, int in_features, const T *kernel, const T *packed, const T *in, const T *bias,
                                const T *residual, const T *beta, const T *gamma, T *out, Profiler::Kind kind) {
    void *stream = cuBERT::blas_get_stream(cublas);
    const int H = (int) hidden_size;
    if (route_of(tokens, H, in_features, kind) == DenseRoute::kSmall && own_slices_to_norm && few_token_slices_enabled()) {
        int slices = 0;
        bool done = false;
        {
            Timed t(profiler, profiler != nullptr ? profiler->dense_kind(kind) : Profiler::kDenseGemm, stream);
            done = cuBERT::dense_mid_slices(tokens, H, in_features, in, in_features, kernel,
                                            transposed_kernels ? in_features : H, few_token_partials,
                                            kFewTokenPartialFloats, &slices, stream);
            if (!done) t.cancel();
        }
        if (done) {
            Timed t(profiler, Profiler::kBiasResLayerNorm, stream);
            if (cuBERT::layer_norm_slices(out, few_token_partials, slices, residual, bias, beta, gamma, tokens, H, stream)) {
                return;
            }
            t.cancel();
            own_slices_to_norm = false;  // the hidden size is fixed per model: do not ask again
        }
    }
    // (also for an fp32 layer too short to be cut by the own kernel: 128 -> 128 at 32 tokens 4.4 against 5.0 us)
    if (tokens <= few_token_limit(kind) && slices_to_norm && few_token_partials != nullptr && few_token_slices_enabled() &&
        (packed != nullptr || !transposed_kernels)) {
        int slices = 0, pitch = 0;
        bool done = false;
        {
            Timed t(profiler, profiler != nullptr ? profiler->dense_kind(kind) : Profiler::kDenseGemm, stream);
            done = cuBERT::dense_few_tokens_partials(cublas, H, tokens, in_features, kernel, H, packed, in, in_features,
                                                     few_token_partials, kFewTokenPartialFloats, &slices, &pitch);
            if (!done) t.cancel();
        }
        if (done) {
            Timed t(profiler, Profiler::kBiasResLayerNorm, stream);
            if (cuBERT::layer_norm_partials(out, few_token_partials, slices, pitch, residual, bias, beta, gamma, tokens, H,
                                            stream)) {
                return;
            }
            t.cancel();
        }
        slices_to_norm = false;  // the layer sizes are fixed per model: do not ask again
    }
    const bool bias_done = dense(H, tokens, in_features, kernel, packed, in, out, bias, false, false, kind);
    Timed t(profiler, Profiler::kBiasResLayerNorm, stream);
    cuBERT::layer_norm_(residual, out, tokens, H, bias_done ? nullptr : bias, beta, gamma, stream);
}

template <typename T>
T *Transformer<T>::_in_compute(size_t batch_size, T *input_gpu, int8_t *attention_mask) {
    if (batch_size > max_batch_size) throw std::invalid_argument("batch_size > max_batch_size");
    void *stream = cuBERT::blas_get_stream(cublas);
    const int M = (int) (batch_size * seq_length), H = (int) hidden_size, I = (int) intermediate_size;

    const bool split = split_dense && two_terms_pay((size_t) M) && !fp32_dense_once;
    fp32_dense_once = false;
    bool operand_ready = false;

    // long half-precision sequences: the attention kernels take the sequences longest first (the mask is the same for every layer)
    order_ready = attention_mask != nullptr && fused_attention_fits &&
                  cubert_attention_wants_order(sizeof(T) == 2, (int) batch_size, (int) num_attention_heads, (int) seq_length,
                                               (int) (hidden_size / num_attention_heads)) &&
                  cuBERT::attention_order(attention_mask, (int) batch_size, (int) seq_length, attention_order, stream);

    T *prev_output = input_gpu;
    for (size_t l = 0; l < num_hidden_layers; ++l) {
        const Layer &w = layers[l];
        T *layer_input = prev_output;
        T *out = layer_output[l & 1];

        if (split) {
            if constexpr (sizeof(T) == 4) {
                // split_operand holds the two-term rows of the next Dense input whenever the kernel before it could
                // write them itself (LayerNorm, GELU); otherwise dense_split makes them from the fp32 rows
                // (making them is a pass of 4.2 us, which the first Q|K|V of a small request does not gain: BERT-base, us a request, fp32 /
                // pass and pairs: 100 tokens 531 / 529, 160 552 / 552, 256 658 / 658, 288 670 / 658, 300 792 / 783, 320 681 / 672, 352
                // 748 / 732, 383 894 / 875)
                const bool held = l > 0 || input_held || split_asked;
                const bool fp32_projection = l == 0 && (!held || M <= 256);
                if (fp32_projection) {
                    dense(3 * H, M, H, w.qkv_kernel, w.qkv_packed, layer_input, qkv_out, w.qkv_bias, true, false,
                          Profiler::kDenseQkv, (int) qkv_ld);
                } else {
                    dense_split(3 * H, M, H, w.qkv_split, w.input_scale, operand_ready ? nullptr : layer_input, qkv_out,
                                w.qkv_split_bias, Profiler::kDenseQkv, (int) qkv_ld);
                }
                // (powers of two that the two-term projection leaves in Q, K and V)
                const int query_key = fp32_projection ? 0 : w.qkv_split.shift(0) + w.qkv_split.shift(1);
                const float context_scale = std::ldexp(w.context_scale, fp32_projection ? 0 : -w.qkv_split.shift(2));
                if (!held) {
                    attention(batch_size, qkv_out, attention_mask);
                    dense(H, M, H, w.attention_output_kernel, w.attention_output_packed, context_out, attention_output,
                          w.attention_output_bias, false, false, Profiler::kDenseAttentionOutput);
                    operand_ready = norm_to_operand(layer_input, attention_output, M, w.attention_output_bias,
                                                    w.attention_norm_beta, w.attention_norm_gamma, w.norm_scale);
                } else {
                    const bool context_ready = attention(batch_size, qkv_out, attention_mask, split_operand, context_scale,
                                                         std::ldexp(1.f, -query_key));
                    if (!context_ready) make_operand(context_out, M, H, context_scale);
                    operand_ready = dense_split_norm(M, H, w.attention_output_split, w.context_scale, w.attention_output_bias,
                                                     layer_input, w.attention_norm_beta, w.attention_norm_gamma, attention_output,
                                                     Profiler::kDenseAttentionOutput, w.norm_scale);
                }
                dense_split(I, M, H, w.intermediate_split, w.norm_scale, operand_ready ? nullptr : attention_output,
                            intermediate_output, pair_dense ? w.intermediate_bias : nullptr, Profiler::kDenseIntermediate, 0,
                            w.inner_scale);
                if (!pair_dense) {
                    // bias + GELU straight into the two-term rows the output Dense reads
                    Timed t(profiler, Profiler::kBiasGelu, stream);
                    cuBERT::bias_gelu_split3(intermediate_output, w.intermediate_bias, M, I, w.inner_scale, split_operand,
                                             split_overflow, stream);
                }
                // (nobody reads the last layer's result as an operand)
                const bool last = l + 1 == num_hidden_layers;
                operand_ready = dense_split_norm(M, I, w.output_split, w.inner_scale, w.output_bias, attention_output,
                                                 w.output_norm_beta, w.output_norm_gamma, out, Profiler::kDenseOutput,
                                                 last ? 0.f : layers[l + 1].input_scale);
            }
            prev_output = out;
            continue;
        }

        // attention/self: row-major Y[M, N] = X[M, K] W[K, N] is the column-major gemm(N, M, K) on (W, X)
        dense(3 * H, M, H, w.qkv_kernel, w.qkv_packed, layer_input, qkv_out, w.qkv_bias, true, false, Profiler::kDenseQkv,
              (int) qkv_ld);
        attention(batch_size, qkv_out, attention_mask);

        // attention/output: dense, then bias + residual(layer input) + LayerNorm
        dense_norm(M, H, w.attention_output_kernel, w.attention_output_packed, context_out, w.attention_output_bias,
                   layer_input, w.attention_norm_beta, w.attention_norm_gamma, attention_output,
                   Profiler::kDenseAttentionOutput);

        // intermediate: dense, then bias + GELU (one launch for all three in a small request)
        if (!dense(I, M, H, w.intermediate_kernel, w.intermediate_packed, attention_output, intermediate_output,
                   w.intermediate_bias, false, true, Profiler::kDenseIntermediate)) {
            Timed t(profiler, Profiler::kBiasGelu, stream);
            cuBERT::gelu(intermediate_output, w.intermediate_bias, M, I, stream);
        }

        // output: dense, then bias + residual(attention output) + LayerNorm
        dense_norm(M, I, w.output_kernel, w.output_packed, intermediate_output, w.output_bias, attention_output,
                   w.output_norm_beta, w.output_norm_gamma, out, Profiler::kDenseOutput);

        prev_output = out;
    }
    return prev_output;
}

template class Transformer<float>;
template class Transformer<half>;

}  // namespace cuBERT
