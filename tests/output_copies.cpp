// Test driver, not part of the library: csrc/host/Bert.cpp over a pretended device in host memory, with an encoder that does
// nothing, under AddressSanitizer and UndefinedBehaviorSanitizer (tests/test_output_copies.py builds and runs it).  It
// looks at how outputs reach the caller's arrays.  Copies are carried out either as soon as they are asked for or
// only when somebody waits for them: a host that reads a slot too early, or has it filled again too early, gets
// wrong values in one of the two.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <memory>
#include <string>
#include <unordered_map>
#include <vector>

#include "Bert.h"

#define EXPECT(condition)                                                            \
    do {                                                                             \
        if (!(condition)) {                                                          \
            fprintf(stderr, "output_copies: line %d: %s\n", __LINE__, #condition); \
            exit(1);                                                                 \
        }                                                                            \
    } while (0)

// ---- allocations that fail on demand ------------------------------------------------------------------------
static bool g_count_allocations = false;
static long g_allocations_left = 0;

void *operator new(size_t n) {
    if (g_count_allocations && g_allocations_left-- <= 0) throw std::bad_alloc();
    if (void *p = std::malloc(n == 0 ? 1 : n)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

// ---- the pretended device ----------------------------------------------------------------------------------
struct Copy {
    void *dst;
    const void *src;
    size_t bytes;
};
static bool g_late = false;
static std::vector<Copy> *g_copies = nullptr;  // asked for, in order
static size_t g_copied = 0;                    // of them carried out
static const void *g_known = nullptr;          // an array that is not ordinary host memory
static size_t g_locked_bytes = 0, g_locked_limit = (size_t) 1 << 40;  // page-locked memory: asked for so far, to be had
static size_t g_records = 0;                   // of events
static size_t g_events[64];                    // copies in front of each event

static void carry_out(size_t until) {
    for (; g_copied < until; ++g_copied) std::memcpy((*g_copies)[g_copied].dst, (*g_copies)[g_copied].src, (*g_copies)[g_copied].bytes);
}

extern "C" {
void *cubert_stream_create(void) { return std::malloc(1); }
int cubert_stream_destroy(void *s) { return std::free(s), 0; }
int cubert_stream_synchronize(void *) { return carry_out(g_copies->size()), 0; }
void *cubert_blas_create(void) { return std::malloc(1); }
int cubert_blas_destroy(void *h) { return std::free(h), 0; }
int cubert_blas_set_stream(void *, void *) { return 0; }
void *cubert_malloc(size_t n) { return std::malloc(n); }
int cubert_free(void *p) { return std::free(p), 0; }
void *cubert_malloc_host(size_t n) {
    if (g_locked_bytes + n > g_locked_limit) return nullptr;
    g_locked_bytes += n;
    return std::malloc(n);
}
int cubert_free_host(void *p) { return std::free(p), 0; }
int cubert_memcpy(void *dst, const void *src, size_t n, int) { return std::memcpy(dst, src, n), 0; }
int cubert_memcpy_async(void *dst, const void *src, size_t n, int kind, void *) {
    const bool counted = g_count_allocations;
    g_count_allocations = false;
    g_copies->push_back(Copy{dst, src, n});
    g_count_allocations = counted;
    if (!g_late || kind != 2) carry_out(g_copies->size());
    return 0;
}
int cubert_is_pageable(const void *p) { return p != nullptr && p != g_known; }
void *cubert_event_create(void) {
    static size_t next = 0;
    return &g_events[next++ % 64];
}
void *cubert_copy_event_create(void) { return cubert_event_create(); }
int cubert_event_destroy(void *) { return 0; }
int cubert_event_record(void *e, void *) { return ++g_records, *static_cast<size_t *>(e) = g_copies->size(), 0; }
int cubert_event_synchronize(void *e) { return carry_out(*static_cast<size_t *>(e)), 0; }
int cubert_event_elapsed_ms(void *, void *, float *) { return 0; }
int cubert_time_next_launch(void *, void *) { return 0; }

// the forward pass: values that belong to a request
static int g_request = 0;
static float value(int output, size_t i) { return (float) (output * 1000003 + g_request * 7 + (int) (i % 99991)); }
int cubert_embed_ln_f32(const int *, const int8_t *, const float *, const float *, const float *, const float *,
                        const float *, float *out, int batch, int seq, int hidden, void *) {
    for (size_t i = 0; i < (size_t) batch * seq * hidden; ++i) out[i] = value(1, i);
    return 0;
}
int cubert_mean_pool_f32(const float *, float *out, int batch, int, int hidden, void *) {
    for (size_t i = 0; i < (size_t) batch * hidden; ++i) out[i] = value(2, i);
    return 0;
}
// what the models here do not reach
#define NOT_REACHED(name, ...) \
    int name(__VA_ARGS__) { abort(); }
NOT_REACHED(cubert_embed_ln_f16, const int *, const int8_t *, const cubert_half *, const cubert_half *, const cubert_half *,
            const cubert_half *, const cubert_half *, cubert_half *, int, int, int, void *)
NOT_REACHED(cubert_mean_pool_f16, const cubert_half *, cubert_half *, int, int, int, void *)
NOT_REACHED(cubert_bias_tanh_f32, float *, const float *, int, int, void *)
NOT_REACHED(cubert_bias_tanh_f16, cubert_half *, const cubert_half *, int, int, void *)
NOT_REACHED(cubert_row_softmax_f32, const float *, float *, int, int, void *)
NOT_REACHED(cubert_row_softmax_f16, const cubert_half *, cubert_half *, int, int, void *)
NOT_REACHED(cubert_gemm_f32, void *, int, int, int, int, int, float, const float *, int, const float *, int, float, float *, int,
            const float *)
NOT_REACHED(cubert_gemm_f16, void *, int, int, int, int, int, float, const cubert_half *, int, const cubert_half *, int, float,
            cubert_half *, int, const cubert_half *)
NOT_REACHED(cubert_classifier_head_f32, float *, const float *, const float *, const float *, float *, float *, int, int, int,
            void *)
NOT_REACHED(cubert_classifier_head_f16, cubert_half *, const cubert_half *, const cubert_half *, const cubert_half *,
            cubert_half *, cubert_half *, int, int, int, void *)
}

// ---- an encoder that does nothing -------------------------------------------------------------------------
namespace cuBERT {
template <typename T>
Transformer<T>::Transformer(void *, const std::string &, const std::unordered_map<std::string, T *> &, size_t max_batch_size,
                            size_t seq_length, size_t hidden_size, size_t, size_t, size_t)
        : cublas(nullptr), max_batch_size(max_batch_size), seq_length(seq_length), hidden_size(hidden_size), num_hidden_layers(0),
          num_attention_heads(1), intermediate_size(0) {
    buffers.take<T>(max_batch_size * seq_length * hidden_size);
    buffers.allocate();
    layer_output[0] = buffers.take<T>(max_batch_size * seq_length * hidden_size);
}
template <typename T>
Transformer<T>::~Transformer() {}
template <typename T>
T *Transformer<T>::_in_compute(size_t batch_size, T *, int8_t *) {
    for (size_t i = 0; i < batch_size * seq_length * hidden_size; ++i) layer_output[0][i] = (T) value(3, i);
    return layer_output[0];
}
template <typename T>
bool Transformer<T>::two_term_overflowed() { return false; }
template class Transformer<float>;
template class Transformer<half>;
}  // namespace cuBERT

struct Model {
    static constexpr size_t kHidden = 128, kSeq = 64, kVocab = 5;
    std::vector<float> weights = std::vector<float>(kSeq * kHidden);
    std::vector<int> ids;
    std::vector<int8_t> zeros;
    std::unique_ptr<cuBERT::Bert<float>> bert;
    size_t batch;

    explicit Model(size_t batch) : ids(batch * kSeq), zeros(batch * kSeq), batch(batch) {
        std::unordered_map<std::string, float *> var;
        for (const char *name : {"word_embeddings", "token_type_embeddings", "position_embeddings", "LayerNorm/beta", "LayerNorm/gamma"})
            var["bert/embeddings/" + std::string(name)] = weights.data();
        bert.reset(new cuBERT::Bert<float>(var, batch, kSeq, kVocab, 2, kHidden, 0, 1, 0, 1));
    }
    void request() {
        ++g_request;
        bert->compute(batch, ids.data(), zeros.data(), zeros.data());
    }
};

struct Arrays {
    std::vector<float> sequence, embedding, pooled;
    explicit Arrays(size_t batch)
            : sequence(batch * Model::kSeq * Model::kHidden, -1.f), embedding(sequence), pooled(batch * Model::kHidden, -1.f) {}
    cuBERT_Output output() {
        cuBERT_Output o = {};
        o.sequence_output = sequence.data(), o.embedding_output = embedding.data(), o.pooled_output = pooled.data();
        return o;
    }
    void expect_request() const {
        for (size_t i = 0; i < sequence.size(); ++i) EXPECT(sequence[i] == value(3, i) && embedding[i] == value(1, i));
        for (size_t i = 0; i < pooled.size(); ++i) EXPECT(pooled[i] == value(2, i));
    }
};

// from less than a piece to several pieces and a remainder, two requests each; what fits one slot waits for no event
static void arrive() {
    for (size_t batch : {1, 2, 3, 40, 64, 65, 127, 128, 129, 300, 384, 385}) {
        Model m(batch);
        for (int repeat = 0; repeat < 2; ++repeat) {
            Arrays a(batch);
            cuBERT_Output o = a.output();
            m.request();
            g_records = 0;
            m.bert->output(batch, &o);
            a.expect_request();
            EXPECT((g_records == 0) == (2 * a.sequence.size() * sizeof(float) <= (4 << 20)));
        }
    }
}

// an array that only the runtime can write to: one copy, to its address
static void leave_to_the_runtime() {
    for (size_t batch : {2, 200}) {
        Model m(batch);
        Arrays a(batch);
        cuBERT_Output o = a.output();
        g_known = a.sequence.data();
        m.request();
        const size_t before = g_copies->size();
        m.bert->output(batch, &o);
        size_t direct = 0;
        for (size_t i = before; i < g_copies->size(); ++i) {
            if ((*g_copies)[i].dst == g_known) direct += (*g_copies)[i].bytes == a.sequence.size() * sizeof(float);
        }
        EXPECT(direct == 1);
        a.expect_request();
    }
}

// page-locked memory for large outputs: only where one is asked for, and the runtime's copy where there is none
static void lock_on_demand() {
    const size_t batch = 200;
    g_locked_bytes = 0;
    Model m(batch);
    Arrays a(batch);
    cuBERT_Output o = a.output();
    m.request();
    m.bert->pooled_output(1, a.pooled.data());
    EXPECT(g_locked_bytes < (1 << 20));
    const size_t limit = g_locked_limit;
    g_locked_limit = g_locked_bytes;
    m.bert->output(batch, &o);
    a.expect_request();
    g_locked_limit = limit;
    for (int repeat = 0; repeat < 2; ++repeat) {
        m.request();
        m.bert->output(batch, &o);
        a.expect_request();
        EXPECT(g_locked_bytes > (8 << 20) && g_locked_bytes < (9 << 20));
    }
}

// an output call that throws half-way, with arrays that are gone before the next one
static void throw_half_way() {
    for (size_t batch : {1, 3, 200}) {
        bool done = false;
        for (long allocations = 0; !done; ++allocations) {
            Model m(batch);
            m.request();
            {
                std::unique_ptr<Arrays> gone(new Arrays(batch));
                cuBERT_Output o = gone->output();
                g_count_allocations = true, g_allocations_left = allocations;
                try {
                    m.bert->output(batch, &o);
                    done = true;
                } catch (const std::bad_alloc &) {
                }
                g_count_allocations = false;
                if (done) EXPECT(allocations > 0);
            }
            Arrays a(batch);
            m.request();
            m.bert->pooled_output(batch, a.pooled.data());
            cuBERT_Output o = a.output();
            m.bert->output(batch, &o);
            a.expect_request();
        }
    }
}

int main(int argc, char **argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    std::vector<Copy> copies;
    g_copies = &copies;
    for (bool late : {false, true}) {
        g_late = late;
        if (what == "arrive") arrive();
        else if (what == "throw") throw_half_way();
        else if (what == "known") leave_to_the_runtime();
        else if (what == "lock") lock_on_demand();
        else return 2;
    }
    printf("output_copies ok\n");
    return 0;
}
