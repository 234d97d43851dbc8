// What a model's weights say of its Dense layers in the two-term fp16 form (kernels/split.hip): the scales of their operands, and
// whether two terms keep what fp32 operands do.
//
// A tensor has one power of two for a scale.  fp16's range bounds it from above.  From below, the spacing of fp16's subnormals rounds
// values that are small next to the tensor's largest, by up to 2^-25 over the scale, which fp32 operands do not know.  The form is
// therefore taken only where this does not show: in every output feature of every Dense layer, the 2-norm of what is lost that way is to be
// below 2^-23 of the 2-norm of the feature's products (an fp32 GEMM of 768 inputs is 2.5e-7, 2^-22, from float64).  BERT-base with
// weights of one size is 2^8 (context) to 2^9 above the line; a model whose channels differ by more than that keeps the fp32 GEMM (channels
// of the value kernel over 2^-R, undone by the rows of the attention output kernel, error of the tokens with and without this: R = 8
// 1.5e-7 and 1.5e-7, 16 3.3e-7 and 3.5e-7, 24 3.3e-7 and 7e-5, 32 3.3e-7 and 1.4e-2; the fp32 GEMM's own is 3.3e-7).
#ifndef CUBERT_HOST_TWOTERM_H
#define CUBERT_HOST_TWOTERM_H

#include <cmath>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <limits>
#include <vector>

namespace cuBERT {

// Activations are multiplied by a power of two before they are taken apart (undone by the GEMM's alpha).  At this one, the
// smallest that is used, entries of 2^-7 to 2^12 keep full accuracy (fp16 subnormals below, clamping above).
constexpr float kTwoTermActivationScale = 16.f;

// the largest power of two that leaves `bound` inside the range of fp16 (0: there is none)
inline float two_term_scale(double bound) {
    if (!(bound >= 0) || !std::isfinite(bound)) return 0.f;
    int exponent = 0;
    (void) std::frexp(65504.0 / (1.01 * bound + 1e-6), &exponent);  // f * 2^exponent, f in [0.5, 1)
    return (float) std::ldexp(1.0, exponent - 1 < 20 ? exponent - 1 : 20);
}

// the power of two that brings the largest weight to [512, 1024): far from fp16's subnormals and its limit
inline int two_term_exponent(float largest_weight) {
    if (!(largest_weight > 0.f)) return 0;
    int exponent = 0;
    (void) std::frexp(largest_weight, &exponent);  // largest = f * 2^exponent, f in [0.5, 1)
    return 10 - exponent < 100 ? 10 - exponent : 100;
}

// the largest |x|, or something that is not finite where one is not (non-negative numbers are in the order of their bits, which is
// a loop over whole vectors)
inline float largest_size(const float *x, size_t count) {
    uint32_t largest = 0;
    for (size_t i = 0; i < count; ++i) {
        uint32_t bits;
        std::memcpy(&bits, x + i, 4);
        bits &= 0x7fffffffu;
        largest = bits > largest ? bits : largest;
    }
    float size;
    std::memcpy(&size, &largest, 4);
    return size;
}

// the larger one, or whichever is not a number
inline double larger_or_nan(double a, double b) { return a >= b || a != a ? a : b; }
inline double largest_or_nan(const float *x, size_t count) {
    double largest = 0;
    for (size_t i = 0; i < count; ++i) largest = larger_or_nan(largest, std::fabs((double) x[i]));
    return largest;
}

// What a Dense layer is given: no value exceeds `element` and no row `row` in 2-norm (not a number where a weight behind them is
// not); squares: the mean square of each channel.
struct DenseInput {
    double element = 0, row = 0;
    std::vector<float> squares;
};

// A LayerNorm's result: no value is further than sqrt(H - 1) standard deviations from the mean, so an element is at most
// |gamma_j| sqrt(H) + |beta_j| and a row max |gamma| sqrt(H) + ||beta||.  (The mean square takes every channel to vary as the row does.
// One that does not, because what comes in is small in it, shows in the column of the Dense layer before; in the embeddings the mean that
// is taken off leaves none of them small.)
inline DenseInput norm_result(const float *gamma, const float *beta, size_t hidden_size) {
    const double root = std::sqrt((double) hidden_size);
    DenseInput x;
    x.squares.resize(hidden_size);
    double largest_gamma = 0, beta_squares = 0;
    for (size_t j = 0; j < hidden_size; ++j) {
        const double g = std::fabs((double) gamma[j]), b = std::fabs((double) beta[j]);
        x.element = larger_or_nan(x.element, g * root + b);
        largest_gamma = larger_or_nan(largest_gamma, g);
        beta_squares += b * b;
        x.squares[j] = (float) (g * g + b * b);
    }
    x.row = largest_gamma * root + std::sqrt(beta_squares);
    return x;
}

// Of a Dense kernel, by columns: the largest weight, the sum of the weights' squares, and the mean square of its product with x.
struct DenseProducts {
    std::vector<float> largest, weights, squares;
    double input = 0;             // mean square of a row of x
    float largest_weight = 0.f;   // (not finite where one is not)
    double column = 0;            // 2-norm of the largest column
};

inline DenseProducts dense_products(const float *kernel, size_t in, size_t out, const DenseInput &x) {
    DenseProducts y;
    y.largest.assign(out, 0.f), y.weights.assign(out, 0.f), y.squares.assign(out, 0.f);
    float *__restrict most = y.largest.data(), *__restrict weights = y.weights.data(), *__restrict squares = y.squares.data();
    for (size_t i = 0; i < in; ++i) {
        const float *__restrict row = kernel + i * out;
        const float square = x.squares[i];
        y.input += square;
        for (size_t j = 0; j < out; ++j) {
            const float w = std::fabs(row[j]), ww = w * w;
            most[j] = w > most[j] ? w : most[j];
            weights[j] += ww;
            squares[j] += ww * square;
        }
    }
    double column = 0;
    for (size_t j = 0; j < out; ++j) {
        column = larger_or_nan(column, weights[j]);
        y.largest_weight = most[j] > y.largest_weight ? most[j] : y.largest_weight;
    }
    y.column = std::sqrt(column);
    if (!(column >= 0)) y.largest_weight = std::numeric_limits<float>::quiet_NaN();  // (no comparison finds one)
    return y;
}

// Whether two terms of x times input_scale and of the kernel times 2^exponent lose nothing that shows (at the top).  A column of
// zeros loses nothing.  (Squares that leave fp32's range make it no.)
inline bool two_terms_hold(const DenseProducts &y, float input_scale, int exponent) {
    const double of_input = std::ldexp(1.0, -25) / input_scale, of_weights = std::ldexp(1.0, -25 - exponent), shows = std::ldexp(1.0, -23);
    for (size_t j = 0; j < y.weights.size(); ++j) {
        const double lost = of_input * of_input * y.weights[j] + of_weights * of_weights * y.input;
        if (y.largest[j] != 0.f && !(lost <= shows * shows * y.squares[j] && std::isfinite(lost))) return false;
    }
    return true;
}

// the mean square of GELU(x) of a normal x, by five points of Gauss-Hermite quadrature
inline double gelu_mean_square(double variance, double mean) {
    static const double kAt[3] = {0, 1.3556261799742659, 2.8569700138728056}, kShare[3] = {8.0 / 15, 0.22207592200561266, 0.011257411327720691};
    double sum = 0;
    for (int i = -2; i <= 2; ++i) {
        const int n = i < 0 ? -i : i;
        const double x = mean + std::sqrt(variance) * (i < 0 ? -kAt[n] : kAt[n]), y = x * 0.5 * (1 + std::erf(x * 0.70710678118654752));
        sum += kShare[n] * y * y;
    }
    return sum;
}

}  // namespace cuBERT

#endif  // CUBERT_HOST_TWOTERM_H
