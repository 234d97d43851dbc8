// The encoder stack on one device.  Public surface of the reference's
// Transformer<T> (src/cuBERT/op_att/Transformer.h:17-39): construct from the
// named-weight map under a variable prefix, then compute(batch, input, mask)
// with device pointers, returning a device pointer to [batch, seq, hidden].
//
// Inside, a layer is 8 launches (7 for small requests, whose intermediate Dense applies its GELU and whose two Dense
// layers in front of a LayerNorm may leave their K slices to it, and for large half ones, whose intermediate Dense applies its
// GELU too; which of the own Dense kernels, the few-token kernel and the library's GEMM a layer runs on: dense_route,
// few_token_limit):
//   qkv   = x * [Wq|Wk|Wv] + [bq|bk|bv]          one GEMM, bias in its epilogue
//   ctx   = softmax((1/sqrt d) Q K^T + mask) V    one attention kernel (scores stay in registers); where its
//                                                 shape limits do not hold: scores kernel or batched GEMM into
//                                                 scores[B, A, S, S], mask_scale_softmax_, context kernel or GEMM
//   a     = LN(ctx * Wo + bo + x)                 GEMM, then layer_norm_   (fused kernel)
//   i     = GELU(a * Wi + bi)                     GEMM, then gelu          (fused kernel; one launch for both on
//                                                 the own Dense kernels)
//   out   = LN(i * Wout + bout + a)               GEMM, then layer_norm_   (fused kernel)
// Activation buffers are shared by all layers (the reference keeps four private
// buffers per layer); weights live in one device allocation.  A half-precision model of seq_length
// <= 64 whose layer sizes are not whole steps of the own Dense kernel also keeps its four Dense kernels in the few-token
// GEMM kernel's own order.
//
// The Dense layers of an fp32 model run on the fp16 matrix cores for requests of more than 64 tokens (where they pay:
// two_terms_pay): every fp32 operand is written as the sum of two fp16 numbers and the product as hi*hi + hi*lo + lo*hi with fp32
// accumulation (one pass of the own kernels, kernels/dense_mid.hip and dense_large.hip, which also apply GELU).  Everything
// between them stays fp32.  The error is smaller than that of the fp32 GEMM (BERT-base against float64, relative 2-norm of the
// tokens, two-term / fp32: 5 x 24 3.4e-7 / 4.8e-7, 3 x 100 3.5 / 11, 20 x 100 6.7 / 12.7, 128 x 32 6.8 / 13.0, 16 x 128 6.7 / 12.7) as long as
// fp16's range holds both terms, which the weights decide when the model is opened: two_term_scales(), TwoTerm.h.
// CUBERT_FP32_DENSE in the environment at that time: f32 keeps the fp32 GEMM, f16x3 takes the two-term form of finite weights also
// where they prove nothing (a request that leaves the range is recomputed in fp32) and, for layer sizes that are no multiple of 32, as one
// library GEMM over three times the reduction length.
#ifndef CUBERT_HOST_TRANSFORMER_H
#define CUBERT_HOST_TRANSFORMER_H

#include <cmath>
#include <cstddef>
#include <cstdint>
#include <string>
#include <unordered_map>
#include <vector>

#include "Arena.h"
#include "common.h"
#include "Profiler.h"
#include "TwoTerm.h"

namespace cuBERT {

// What follows a Dense layer: nothing (its bias is added in the GEMM), bias + GELU, or bias + residual + LayerNorm.
enum class DenseUse { kPlain, kGelu, kNorm };

// What a Dense layer of this size runs on where its sizes are whole steps of the own Dense kernels: the one for small requests
// (kernels/dense_mid.hip), the one for large requests (dense_large.hip), or the few-token kernel or a library GEMM; as_slices: the
// LayerNorm that follows can add K slices.
enum class DenseRoute { kOther, kSmall, kLarge };
DenseRoute dense_route(bool half_precision, int tokens, int out_features, int in_features, DenseUse use, bool as_slices);
// ... and whether the one for small requests is better than the few-token kernel and the library's GEMM
bool own_dense_is_best(bool half_precision, int tokens, int out_features, int in_features, DenseUse use, bool as_slices);

template <typename T>
class Transformer {
public:
    explicit Transformer(void *cublas, const std::string &var_prefix, const std::unordered_map<std::string, T *> &var,
                         size_t max_batch_size, size_t seq_length, size_t hidden_size, size_t num_hidden_layers,
                         size_t num_attention_heads, size_t intermediate_size);

    virtual ~Transformer();

    Transformer(const Transformer &) = delete;
    Transformer &operator=(const Transformer &) = delete;

    T *compute(size_t batch_size, T *input_gpu, int8_t *attention_mask);

    // Kept for source compatibility with callers of the reference: there the
    // Dense outputs had to be pre-filled with their biases before a request;
    // here biases are applied inside the GEMM epilogue or the fused kernels.
    void _pre_compute(size_t batch_size);

    T *_in_compute(size_t batch_size, T *input_gpu, int8_t *attention_mask);

    // Optional per-kernel timing (owned by the caller; null = off).
    void set_profiler(Profiler *p) { profiler = p; }

    // Two-term fp16 Dense form only.  An activation beyond the fp16 range (times its scale) cannot be written as two fp16 terms; the kernels that write two-term rows then raise a flag instead of
    // handing a clamped operand to the GEMM in silence.  Once the stream has drained, two_term_overflowed() says
    // whether any request since the last call raised it (and clears it); the caller then runs the request again
    // after use_fp32_dense_once(), which makes the next _in_compute take the fp32 GEMMs whatever its size.
    bool two_term_overflowed();
    void use_fp32_dense_once() { fp32_dense_once = true; }

    // What _in_compute is given (two-term form; where this is not known, or two terms do not hold it, layer 0 of a model that was not
    // asked for the form by name has its attention in fp32).
    void set_input(const std::string &var_prefix, const std::unordered_map<std::string, T *> &var, const DenseInput &input) {
        if (split_dense && !layers.empty()) input_held = attention_scales(var_prefix + "/layer_0", var, input, layers[0]).held;
    }

private:
    // A Dense kernel for the two-term fp16 form: rows of pairs of 2^exponent * W^T, [out, 2 * in], or, for the library's GEMM, rows
    // [hi | lo | hi], [out, 3 * in]; the GEMM multiplies by unscale = 2^-common.  Q, K and V have an exponent each, and leave the GEMM
    // 2^shift too large.
    static constexpr size_t kTwoTermMinTokens = 384;  // asked for by name, on the library's GEMM too
    struct SplitKernel {
        half *weights = nullptr;
        int exponent[3] = {}, common = 0;
        int shift(size_t part) const { return exponent[part] - common; }
        float unscale() const { return std::ldexp(1.f, -common); }
        void set_exponent(float largest_weight) { exponent[0] = common = two_term_exponent(largest_weight); }
    };

    struct Layer {
        // Dense kernels are [in, out] as in the model file, or [out, in] when transposed_kernels is set
        T *qkv_kernel, *qkv_bias;            // [hidden, 3*hidden] (query | key | value side by side), [3*hidden]
        T *attention_output_kernel, *attention_output_bias;
        T *attention_norm_beta, *attention_norm_gamma;
        T *intermediate_kernel, *intermediate_bias;
        T *output_kernel, *output_bias;
        T *output_norm_beta, *output_norm_gamma;
        // the Dense kernels again, in the few-token GEMM kernel's order (null when not kept)
        T *qkv_packed = nullptr, *attention_output_packed = nullptr, *intermediate_packed = nullptr,
          *output_packed = nullptr;
        SplitKernel qkv_split, attention_output_split, intermediate_split, output_split;  // (null when not kept)
        T *qkv_split_bias = nullptr;  // qkv_bias with the powers of two that the two-term form leaves in Q, K and V
        // of the four operands: what the layer is given, context, attention output behind its LayerNorm, GELU's result
        float input_scale = kTwoTermActivationScale, context_scale = kTwoTermActivationScale,
              norm_scale = kTwoTermActivationScale, inner_scale = kTwoTermActivationScale;
    };

    struct TwoTermProof {
        bool finite = true, held = true;
        void add(const TwoTermProof &other) { finite = finite && other.finite, held = held && other.held; }
    };
    TwoTermProof two_term_scales(const std::string &var_prefix, const std::unordered_map<std::string, T *> &var);
    // the same for one layer's attention, given x
    TwoTermProof attention_scales(const std::string &layer, const std::unordered_map<std::string, T *> &var, const DenseInput &x, Layer &w) {
        TwoTermProof proof;
        if constexpr (sizeof(T) == 4) {
            const size_t H = hidden_size;
            auto products = [&](const char *name, const DenseInput &of) { return dense_products(var.at(layer + name + "/kernel"), H, H, of); };
            const DenseProducts query = products("/attention/self/query", x), key = products("/attention/self/key", x),
                                value = products("/attention/self/value", x);
            const T *bias = var.at(layer + "/attention/self/value/bias");
            DenseInput context;
            context.element = x.row * value.column + largest_or_nan(bias, H);
            // (at worst the mean of all rows of V)
            context.squares.resize(H);
            for (size_t j = 0; j < H; ++j) {
                context.squares[j] = (float) ((double) value.squares[j] / seq_length + (double) bias[j] * bias[j]);
            }
            const DenseProducts output = products("/attention/output/dense", context);
            proof.finite = set_attention_exponents(w, query.largest_weight, key.largest_weight, value.largest_weight, output.largest_weight);
            const bool x_fits = set_scale(w.input_scale, x.element), context_fits = set_scale(w.context_scale, context.element);
            proof.held = x_fits && context_fits && two_terms_hold(query, w.input_scale, w.qkv_split.exponent[0]) &&
                         two_terms_hold(key, w.input_scale, w.qkv_split.exponent[1]) &&
                         two_terms_hold(value, w.input_scale, w.qkv_split.exponent[2]) &&
                         two_terms_hold(output, w.context_scale, w.attention_output_split.exponent[0]);
        }
        return proof;
    }
    // Q, K and V have an exponent each, at most 40 apart; false: a weight is not finite
    static bool set_attention_exponents(Layer &w, float query, float key, float value, float output) {
        int *e = w.qkv_split.exponent;
        e[0] = two_term_exponent(query), e[1] = two_term_exponent(key), e[2] = two_term_exponent(value);
        w.qkv_split.common = e[0] < e[1] ? e[0] : e[1];
        w.qkv_split.common = e[2] < w.qkv_split.common ? e[2] : w.qkv_split.common;
        for (int part = 0; part < 3; ++part) e[part] = e[part] < w.qkv_split.common + 40 ? e[part] : w.qkv_split.common + 40;
        w.attention_output_split.set_exponent(output);
        return std::isfinite(query) && std::isfinite(key) && std::isfinite(value) && std::isfinite(output);
    }
    // the scale for an operand that does not exceed bound; false: there is none, and it is the smallest
    static bool set_scale(float &scale, double bound) {
        const float s = two_term_scale(bound);
        scale = s >= kTwoTermActivationScale ? s : kTwoTermActivationScale;
        return s >= kTwoTermActivationScale;
    }

    void layout_weights();
    void layout_buffers();
    // The [max_batch, heads, seq, seq] score tensor.  Only the three-kernel attention path touches it, and the
    // one-launch kernel takes every BERT shape up to seq_length 512, so it is not part of `buffers` (it would be the
    // largest of them: 403 MB at batch 64 x 12 heads x seq 512 in fp16) but allocated on first use.
    T *scores();
    // context_out = attention(qkv); with `split_context` (fp32 models in the two-term Dense form) the one-launch
    // kernel writes the context, times scale, there as two-term rows instead and true is returned; Q K^T is multiplied by score_unscale
    bool attention(size_t batch_size, const T *qkv, const int8_t *mask, half *split_context = nullptr, float scale = 1.f,
                   float score_unscale = 1.f);
    // out[tokens, out_features] = in[tokens, in_features] * kernel (+ bias) (, GELU); returns whether bias and
    // activation were applied (false: the caller's fused kernel still has to).
    bool dense(int out_features, int tokens, int in_features, const T *kernel, const T *packed, const T *in, T *out,
               const T *bias, bool bias_in_gemm, bool gelu, Profiler::Kind kind, int ld_out = 0);
    // The same on the fp16 matrix cores from two-term operands (fp32 models only): `in` is split into
    // split_operand first, or, when null, split_operand already holds its two-term rows.  `bias` may be null.  With pair_dense
    // the intermediate layer applies GELU and leaves two-term rows in split_intermediate, where the output layer finds them.
    // scale: of the operand; inner_scale: of the intermediate layer's result
    void make_operand(const T *in, int tokens, int width, float scale);
    void dense_split(int out_features, int tokens, int in_features, const SplitKernel &kernel, float scale, const T *in, T *out,
                     const T *bias, Profiler::Kind kind, int ld_out = 0, float inner_scale = 1.f);
    // out = LayerNorm(dense_split of split_operand + bias + residual), and with a next_scale its two-term rows in split_operand; whether they were written
    bool dense_split_norm(int tokens, int in_features, const SplitKernel &kernel, float scale, const T *bias,
                          const T *residual, const T *beta, const T *gamma, T *out, Profiler::Kind kind, float next_scale);
    // whether a request of this many tokens is faster in the two-term form
    bool two_terms_pay(size_t tokens) const;
    // inout = LayerNorm(inout + bias + residual), and its two-term rows in split_operand; false: the hidden size is declined
    bool norm_split(const T *residual, T *inout, int tokens, const T *bias, const T *beta, const T *gamma, float scale);
    // the same, or without the rows where they are declined or nobody asks for them (scale 0); whether they were written
    bool norm_to_operand(const T *residual, T *inout, int tokens, const T *bias, const T *beta, const T *gamma, float scale);
    // out = LayerNorm(in * kernel + bias + residual): dense(), then layer_norm_; for a small request the Dense kernel
    // leaves its K slices in few_token_partials and the LayerNorm kernel adds them while it loads (no hand-over between
    // the GEMM's workgroups).
    void dense_norm(int tokens, int in_features, const T *kernel, const T *packed, const T *in, const T *bias,
                    const T *residual, const T *beta, const T *gamma, T *out, Profiler::Kind kind);

    // dense_route for a layer of this model
    DenseRoute route_of(int tokens, int out_features, int in_features, Profiler::Kind kind) const;

    // up to how many tokens the Dense layer of this kind runs on the few-token kernel (32 or 64)
    int few_token_limit(Profiler::Kind kind) const;

    void *cublas;
    Profiler *profiler = nullptr;
    bool slices_to_norm = true;        // few-token Dense layers hand their K slices to the LayerNorm (cleared when declined)
    bool dense_gelu_fits = true;       // cleared when the few-token Dense + GELU kernel declines this model's shape
    bool own_dense = false;            // layer sizes are whole steps of the library's own Dense kernel (any few tokens)
    bool own_slices_to_norm = true;    // cleared when the LayerNorm over its slices declines the hidden size
    bool keep_packed = false;          // Dense kernels are also kept in the few-token kernel's order
    bool transposed_kernels = false;   // Dense kernels are stored [out, in] instead of [in, out] (half precision)
    bool split_dense = false;          // fp32 model with Dense layers in the two-term fp16 form
    bool split_asked = false;          // ... because it was asked for by name (CUBERT_FP32_DENSE=f16x3)
    bool input_held = false;           // set_input gave layer 0 its scales
    bool pair_dense = false;           // ... on the library's own kernel, whose operand rows hold every term once
    bool fp32_dense_once = false;      // the next request takes the fp32 GEMMs (set after a two-term overflow)
    int *split_overflow = nullptr;     // page-locked host word the two-term kernels set to 1 on overflow (split_dense)
    bool norm_writes_operand = true;   // cleared when the LayerNorm that also writes two-term rows declines the hidden size
    bool fused_attention_fits = true;  // cleared when the one-launch attention kernel declines this model's shape
    size_t max_batch_size, seq_length, hidden_size, num_hidden_layers, num_attention_heads, intermediate_size;

    Arena weights;
    Arena buffers;
    Arena score_memory;  // the score tensor of the three-kernel attention path: claimed when a request first takes it
    std::vector<Layer> layers;

    size_t qkv_ld = 0;       // elements from one token's Q | K | V row to the next (>= 3*hidden)
    T *qkv_out;              // [M, qkv_ld]
    T *attention_scores = nullptr;  // [B, heads, seq, seq], in score_memory (null until scores() is first called)
    T *context_out;          // [M, hidden]
    int *attention_order = nullptr;  // [8 * max_batch]: sequence indices, most live key tiles first, and their tile lists (seq_length > 128)
    bool order_ready = false;        // attention_order holds the current request's order
    T *attention_output;     // [M, hidden]
    T *intermediate_output;  // [M, intermediate]
    T *layer_output[2];      // [M, hidden], alternating between layers
    half *split_operand = nullptr;  // [M, 3 * max(hidden, intermediate)] two-term rows of the current Dense input; with pair_dense
    half *split_intermediate = nullptr;  // [M, 2 * hidden], and those of the output layer's input, [M, 2 * intermediate], here
    static constexpr size_t kFewTokenPartialFloats = (size_t) 1 << 21;
    float *few_token_partials = nullptr;  // K slices of the current Dense layer of a small request
};

}  // namespace cuBERT

#endif  // CUBERT_HOST_TRANSFORMER_H
