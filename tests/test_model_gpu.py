"""End-to-end parity of the host classes (Transformer, Bert, BertM behind cuBERT_open) with the
CPU oracle, through the C ABI: the reference's encoder known-answer vectors, seeded random models
at small and full BERT-base / BERT-large shapes, every output type, the GraphDef file path and the
error behaviour of the public API.

Tolerances: fp32 within 1e-5 relative (norm-wise) of the oracle; fp16 storage within 1e-2 relative
on pooled / logit outputs of the fp32 oracle run on the same weights rounded to fp16 (the
reference's own fp16-vs-fp32 bound, BertTest.cpp:109-110)."""
import os

import numpy as np
import pytest

import oracle
from test_oracle_golden import transformer_weights
from util import FP16_TOL, FP32_TOL, assert_close, rel_err

pytestmark = pytest.mark.gpu

T = "test/cuBERT/"


@pytest.fixture(scope="module")
def cb():
    import torch
    if not torch.cuda.is_available():
        pytest.fail("no GPU visible: the -m gpu tests must run on the MI355X box")
    import cubert_amd
    return cubert_amd


# ------------------------------------------------------------------ reference encoder vectors

@pytest.mark.parametrize("name,layers", [("transformer", 1), ("transformer_complex", 2)])
def test_transformer_reference_vectors(cb, case, name, layers):
    c = case(T + "op_att/TransformerTest.cpp", name)
    mask = np.ones((2, 4), np.int8)
    mask[0, 0] = 0
    out = cb.transformer_run(transformer_weights(c, layers), "encoder",
                             np.array(c.arrays["tensor"], np.float32).reshape(2, 4, 6), mask, layers, 2, 5)
    assert c.check(out) == 12  # the reference's own tolerances: 1e-6 (1 layer), 1e-5 (2 layers)


def test_transformer_reference_vectors_half(cb, case):
    c = case(T + "op_att/TransformerTest.cpp", "transformer_complex_half")
    mask = np.ones((2, 4), np.int8)
    mask[0, 0] = 0
    out = cb.transformer_run(transformer_weights(c, 2), "encoder",
                             np.array(c.arrays["tensor"], np.float32).reshape(2, 4, 6), mask, 2, 2, 5,
                             compute_type=cb.ComputeType.HALF)
    assert c.check(out.astype(np.float32)) == 12  # 1e-3 .. 1e-2 absolute, as the reference asserts for half


def test_missing_weight_raises_like_unordered_map_at(cb, case):
    c = case(T + "op_att/TransformerTest.cpp", "transformer")
    w = transformer_weights(c, 1)
    del w["encoder/layer_0/output/dense/bias"]
    with pytest.raises(IndexError):
        cb.transformer_run(w, "encoder", np.zeros((2, 4, 6), np.float32), np.ones((2, 4), np.int8), 1, 2, 5)


# ------------------------------------------------------------------ seeded models vs the oracle

SMALL = dict(vocab=211, hidden=128, layers=3, heads=4, intermediate=512, max_position=64, type_vocab=2)
# an intermediate size that is no whole number of steps of the own Dense kernel: few-token kernel and library
ODD = dict(SMALL, intermediate=528)


def run_both(cb, weights, ids, mask, seg, layers, heads, max_batch, compute_type=0, oracle_rows=None):
    from cubert_amd.testing import random_bert_weights  # noqa: F401  (kept importable for -k runs)
    S = ids.shape[1]
    bert = cb.Bert(weights, max_batch, S, layers, heads, compute_type)
    got = bert.forward(ids, mask, seg)
    bert.close()
    if compute_type == 1:
        weights = {k: oracle.round_to_half(v) for k, v in weights.items()}
    n = ids.shape[0] if oracle_rows is None else oracle_rows
    want = oracle.bert_forward(weights, ids[:n], mask[:n], seg[:n], layers, heads)
    return got, want, n


@pytest.mark.parametrize("pooler,bias,scattered", [(True, True, False), (False, False, True), (True, False, True)])
def test_small_model_all_outputs_fp32(cb, pooler, bias, scattered):
    from cubert_amd.testing import random_bert_weights, random_inputs
    w = random_bert_weights(seed=3, labels=3, pooler=pooler, classifier=True, classifier_bias=bias, ln_random=True,
                            **SMALL)
    ids, mask, seg = random_inputs(seed=4, batch=7, seq_length=32, vocab=SMALL["vocab"], min_valid=2,
                                   segment_split="random", scattered_mask=scattered)
    got, want, _ = run_both(cb, w, ids, mask, seg, 3, 4, max_batch=9)
    for k in ("embedding_output", "sequence_output", "pooled_output", "logits", "probs"):
        assert_close(got[k], want[k], FP32_TOL, k)


@pytest.mark.parametrize("compute_type", [0, 1])
@pytest.mark.parametrize("pooler", [True, False])
def test_many_labels_take_the_three_kernel_classifier(cb, compute_type, pooler):
    """More than 64 labels: the one-launch classifier head declines and the model runs bias + tanh, the classifier
    GEMM and the row softmax separately; with or without a pooler dense layer (MeanPooler)."""
    from cubert_amd.testing import random_bert_weights, random_inputs
    w = random_bert_weights(seed=11, labels=70, pooler=pooler, classifier=True, ln_random=True, **SMALL)
    ids, mask, seg = random_inputs(seed=12, batch=5, seq_length=32, vocab=SMALL["vocab"], min_valid=4, segment_split=11)
    got, want, _ = run_both(cb, w, ids, mask, seg, 3, 4, max_batch=6, compute_type=compute_type)
    for k in ("pooled_output", "logits", "probs"):
        assert_close(got[k], want[k], FP16_TOL if compute_type else FP32_TOL, k)
    assert got["probs"].shape == (5, 70)


def test_small_model_fp16(cb):
    from cubert_amd.testing import random_bert_weights, random_inputs
    w = random_bert_weights(seed=5, labels=2, pooler=True, classifier=True, ln_random=True, **SMALL)
    ids, mask, seg = random_inputs(seed=6, batch=8, seq_length=64, vocab=SMALL["vocab"], min_valid=5, segment_split=20)
    got, want, _ = run_both(cb, w, ids, mask, seg, 3, 4, max_batch=8, compute_type=1)
    for k in ("pooled_output", "logits", "probs", "sequence_output", "embedding_output"):
        assert_close(got[k], want[k], FP16_TOL, k)


@pytest.mark.parametrize("model", [SMALL, ODD], ids=["own_dense", "odd_intermediate"])
@pytest.mark.parametrize("compute_type", [0, 1])
@pytest.mark.parametrize("seq_length", [32, 16])
def test_requests_of_at_most_32_tokens(cb, compute_type, seq_length, model):
    """Batch 1 (and batch 2 at seq 16) of a model whose layer sizes are whole steps of the own Dense kernel run on that one;
    with an odd intermediate size the Dense layers run on the few-token kernel, the intermediate layer with its GELU in the
    same launch, and a half-precision model on its re-ordered weight copies.  A larger batch of the same model (1312 tokens,
    of the odd one 192) takes the library GEMM.  Both must match the oracle, and the single request must match itself as a
    row of the larger batch."""
    from cubert_amd.testing import random_bert_weights, random_inputs
    w = random_bert_weights(seed=11, labels=2, pooler=True, classifier=True, ln_random=True, **model)
    total = (1312 if model is SMALL else 192) // seq_length
    ids, mask, seg = random_inputs(seed=12, batch=total, seq_length=seq_length, vocab=SMALL["vocab"], min_valid=3,
                                   segment_split=7)
    tol = FP16_TOL if compute_type else FP32_TOL
    wo = {k: oracle.round_to_half(v) for k, v in w.items()} if compute_type else w
    want = oracle.bert_forward(wo, ids, mask, seg, 3, 4)
    bert = cb.Bert(w, total, seq_length, 3, 4, compute_type)
    bert.profile(["bias_gelu"])
    full = bert.forward(ids, mask, seg)
    assert bert.profile_read()["bias_gelu"][1] == 3  # a GELU launch of its own per layer: the library's GEMM
    for n in (1, 2):
        if n * seq_length > 32:
            continue
        few = bert.forward(ids[:n], mask[:n], seg[:n])
        assert "bias_gelu" not in bert.profile_read()
        for k in ("sequence_output", "pooled_output", "logits", "probs"):
            assert_close(few[k], want[k][:n], tol, "%s, %d request(s)" % (k, n))
            assert_close(few[k], full[k][:n], tol, "%s vs the same rows of a batch of %d" % (k, total))
    bert.close()
    for k in ("sequence_output", "pooled_output", "logits"):
        assert_close(full[k], want[k], tol, k)


@pytest.mark.parametrize("model", [SMALL, ODD], ids=["own_dense", "odd_intermediate"])
@pytest.mark.parametrize("compute_type", [0, 1])
@pytest.mark.parametrize("seq_length,batches", [(32, (2,)), (64, (1,)), (16, (3, 4)), (8, (5, 8))])
def test_requests_of_33_to_64_tokens(cb, compute_type, seq_length, batches, model):
    """From 33 to 64 tokens: the own Dense kernel, or with an odd intermediate size the few-token kernel with two blocks of
    32 tokens per wavefront for the layers in front of a LayerNorm (and, in half precision, the intermediate layer with its
    GELU) and the library for the others.  The request must match the oracle and itself as rows of a larger batch, which
    runs on the library's GEMMs."""
    from cubert_amd.testing import random_bert_weights, random_inputs
    w = random_bert_weights(seed=21, labels=2, pooler=True, classifier=True, ln_random=True, **model)
    total = (1312 if model is SMALL else 192) // seq_length
    ids, mask, seg = random_inputs(seed=22, batch=total, seq_length=seq_length, vocab=SMALL["vocab"], min_valid=3,
                                   segment_split=5)
    tol = FP16_TOL if compute_type else FP32_TOL
    wo = {k: oracle.round_to_half(v) for k, v in w.items()} if compute_type else w
    want = oracle.bert_forward(wo, ids, mask, seg, 3, 4)
    bert = cb.Bert(w, total, seq_length, 3, 4, compute_type)
    full = bert.forward(ids, mask, seg)
    for n in batches:
        assert 32 < n * seq_length <= 64
        few = bert.forward(ids[:n], mask[:n], seg[:n])
        for k in ("sequence_output", "pooled_output", "logits", "probs"):
            assert_close(few[k], want[k][:n], tol, "%s, %d request(s) of %d tokens" % (k, n, seq_length))
            assert_close(few[k], full[k][:n], tol, "%s vs the same rows of a batch of %d" % (k, total))
    bert.close()


@pytest.mark.parametrize("compute_type,batches", [(0, ((8, True), (10, True), (11, False))),
                                                  (1, ((17, True), (28, True), (37, True), (40, True), (41, True)))])
def test_requests_around_the_switch_to_the_library(cb, monkeypatch, compute_type, batches):
    """Two layers of BERT-base's width, 32 tokens a sequence, on either side of the token counts where a Dense layer (of an fp32 model
    with CUBERT_FP32_DENSE=f32) goes over to the library's GEMM (whose GELU is a launch of its own), or in half precision to the own kernel for large
    requests (whose epilogue applies it); between them some layers run on one and some on the
    other.  Against the oracle, the first and the last sequences of each batch."""
    from cubert_amd.testing import random_bert_weights, random_inputs
    monkeypatch.setenv("CUBERT_FP32_DENSE", "f32")
    m = dict(vocab=97, hidden=768, layers=2, heads=12, intermediate=3072, max_position=64, type_vocab=2)
    w = random_bert_weights(seed=41, labels=2, pooler=True, classifier=True, ln_random=True, **m)
    largest = batches[-1][0]
    ids, mask, seg = random_inputs(seed=42, batch=largest, seq_length=32, vocab=97, min_valid=3, segment_split=9)
    wo = {k: oracle.round_to_half(v) for k, v in w.items()} if compute_type else w
    want = oracle.bert_forward(wo, ids, mask, seg, 2, 12)
    bert = cb.Bert(w, largest, 32, 2, 12, compute_type)
    bert.profile(["bias_gelu"])
    for n, own in batches:
        got = bert.forward(ids[:n], mask[:n], seg[:n])
        assert ("bias_gelu" not in bert.profile_read()) == own, n
        for k in ("sequence_output", "pooled_output", "logits", "probs"):
            assert_close(got[k], want[k][:n], FP16_TOL if compute_type else FP32_TOL, "%s, %d sequences" % (k, n))
    bert.close()


@pytest.mark.parametrize("seq_length,heads,hidden,three_steps,one_launch", [
    (333, 2, 128, (1, 24), (25,)), (320, 3, 192, (16,), (17,)), (511, 2, 128, (2,), (25,)), (288, 2, 128, (), (1, 2)),
    (333, 2, 64, (1, 8), (9,)), (352, 2, 64, (), (1,)), (512, 2, 128, (), (1,)), (333, 1, 128, (1, 25), ()), (289, 6, 192, (1, 8), (9,)),
    (511, 12, 768, (4,), ())])
def test_long_fp32_sequences_by_number_of_problems(cb, seq_length, heads, hidden, three_steps, one_launch):
    """fp32 sequences of more than 288 keys, few (sequence, head) problems and more of them than kernels of a workgroup per problem were
    better with: one launch, which is ahead of scores, softmax and context in three steps at every one of these; a head size of 128, which
    it declines, takes the three steps.  Either way the outputs are the oracle's."""
    from cubert_amd.testing import random_bert_weights, random_inputs
    m = dict(vocab=97, hidden=hidden, layers=1, heads=heads, intermediate=4 * hidden, max_position=512, type_vocab=2)
    w = random_bert_weights(seed=31, labels=2, pooler=True, classifier=True, ln_random=True, **m)
    largest = max(three_steps + one_launch)
    ids, mask, seg = random_inputs(seed=32, batch=largest, seq_length=seq_length, vocab=97, min_valid=3, segment_split=9)
    rows = 2  # rows of a batch are independent
    want = oracle.bert_forward(w, ids[:rows], mask[:rows], seg[:rows], 1, heads)
    bert = cb.Bert(w, largest, seq_length, 1, heads, 0)
    bert.profile(["attention_fused", "attention_gemm", "mask_scale_softmax"])
    for n in three_steps + one_launch:
        got = bert.forward(ids[:n], mask[:n], seg[:n])
        kinds = set(bert.profile_read())
        assert kinds == ({"attention_gemm", "mask_scale_softmax"} if hidden // heads == 128 else {"attention_fused"}), (n, kinds)
        for k in ("sequence_output", "pooled_output", "logits", "probs"):
            assert_close(got[k][:rows], want[k][:n], FP32_TOL, "%s, %d sequences" % (k, n))
    bert.close()


def test_score_tensor_of_few_long_sequences_is_small(cb):
    """A model for 256 sequences of 511 tokens that is asked for one: no score tensor of its largest batch (535 MB), and, in one launch,
    none at all."""
    import ctypes
    from cubert_amd._lib import lib
    from cubert_amd.testing import random_bert_weights, random_inputs
    m = dict(vocab=97, hidden=128, layers=1, heads=2, intermediate=512, max_position=512, type_vocab=2)
    w = random_bert_weights(seed=31, labels=2, pooler=True, classifier=True, ln_random=True, **m)
    ids, mask, seg = random_inputs(seed=32, batch=1, seq_length=511, vocab=97, min_valid=3, segment_split=9)
    bert = cb.Bert(w, 256, 511, 1, 2, 0)
    free = [ctypes.c_size_t(), ctypes.c_size_t()]
    assert lib().cubert_mem_info(ctypes.byref(free[0]), None) == 0
    bert.profile(["attention_fused", "mask_scale_softmax"])
    bert.forward(ids, mask, seg)
    assert set(bert.profile_read()) == {"attention_fused"}
    assert lib().cubert_mem_info(ctypes.byref(free[1]), None) == 0
    bert.close()
    assert free[0].value - free[1].value < 50e6


def test_repeated_calls_and_smaller_batches_reuse_buffers(cb):
    """The reference's BertMTest calls one model four times; results must not depend on what ran before."""
    from cubert_amd.testing import random_bert_weights, random_inputs
    w = random_bert_weights(seed=7, labels=2, **SMALL)
    ids, mask, seg = random_inputs(seed=8, batch=6, seq_length=32, vocab=SMALL["vocab"], min_valid=4)
    bert = cb.Bert(w, 6, 32, 3, 4)
    first = bert.forward(ids, mask, seg)
    small = bert.forward(ids[:2], mask[:2], seg[:2])
    again = bert.forward(ids, mask, seg)
    bert.close()
    for k in first:
        assert np.array_equal(first[k], again[k]), k
        # rows of a batch are independent of the batch they are computed in (different GEMM shapes: not bit-equal)
        assert_close(small[k], first[k][:2], FP32_TOL, k)


CONFIG_CASES = [
    # name, oracle rows (None = all; rows of a batch are independent, so a prefix is enough at big shapes)
    ("C0", None),
    ("C1", None),
    ("C2", 8),
    ("C3", 2),
    ("C4", 4),
]


@pytest.mark.parametrize("two_term", [False, True])
@pytest.mark.parametrize("seed", [11, 12, 13])
def test_randomly_drawn_model_configurations(cb, seed, two_term, monkeypatch):
    """(two_term: the same draws with CUBERT_FP32_DENSE=f16x3 in the environment, fp32 cases only -- requests of at
    least 384 tokens then run their Dense layers on the fp16 matrix cores from two-term operands, same bound.)
    Fifteen models per seed with every size drawn at random -- heads, head size (also ones no matrix-core kernel
    takes), seq_length (1 ... 512, not only multiples of 32), intermediate size, layers, labels (few and many), with and
    without pooler / classifier / classifier bias, both compute types, prefix and scattered masks, a batch below the
    maximum -- against the oracle, every output; two calls in a row must agree bit for bit.  The fp32 bound here is
    5e-5, not 1e-5: weights are drawn with a standard deviation of 0.05 instead of 0.02, and on such a model the
    oracle itself is up to 1e-5 away from a float64 evaluation (summation order over 1536 ... 3080 terms), so two fp32
    evaluations are up to 3e-5 apart (measured over 480 drawn models: 2.8e-5; fp16: 1.3e-2)."""
    from cubert_amd.testing import random_bert_weights, random_inputs
    if two_term:
        monkeypatch.setenv("CUBERT_FP32_DENSE", "f16x3")
    rng = np.random.default_rng(seed)
    for case in range(15):
        heads = int(rng.choice([1, 2, 3, 4, 8, 12]))
        d = int(rng.choice([32, 64, 64, 64, 128, 16, 24]))
        hidden = heads * d
        seq = int(rng.choice([1, 4, 7, 32, 32, 64, 96, 128, 160, 256, 512, 33]))
        if seq * hidden > 512 * 512:
            seq = 32
        max_batch = int(rng.integers(1, 9))
        batch = int(rng.integers(1, max_batch + 1))
        layers = int(rng.integers(1, 4))
        inter = int(rng.choice([hidden * 4, hidden * 2 + 8, 100, 3 * hidden]))
        labels = int(rng.choice([1, 2, 3, 7, 70]))
        pooler, classifier, cbias = bool(rng.integers(0, 2)), bool(rng.integers(0, 4) > 0), bool(rng.integers(0, 2))
        compute_type = int(rng.integers(0, 2))
        vocab = int(rng.integers(5, 400))
        scattered = bool(rng.integers(0, 2))
        what = "seed %d case %d: B=%d/%d S=%d H=%d A=%d I=%d L=%d labels=%d pooler=%s classifier=%s bias=%s %s %s" % (
            seed, case, batch, max_batch, seq, hidden, heads, inter, layers, labels, pooler, classifier, cbias,
            "f16" if compute_type else "f32", "scattered" if scattered else "prefix")
        if two_term and compute_type == 1:
            continue
        print(what, flush=True)
        w = random_bert_weights(seed=seed * 100 + case, vocab=vocab, hidden=hidden, layers=layers, heads=heads,
                                intermediate=inter, max_position=max(seq, 8), type_vocab=2, labels=labels, pooler=pooler,
                                classifier=classifier, classifier_bias=cbias, ln_random=True, stddev=0.05)
        ids, mask, seg = random_inputs(seed=seed * 100 + case, batch=batch, seq_length=seq, vocab=vocab,
                                       min_valid=None if scattered else 1, max_valid=None if scattered else seq,
                                       segment_split="random" if seq > 1 else None, scattered_mask=scattered)
        bert = cb.Bert(w, max_batch, seq, layers, heads, compute_type=compute_type)
        got, again = bert.forward(ids, mask, seg), bert.forward(ids, mask, seg)
        bert.close()
        seen = {k: (oracle.round_to_half(v) if compute_type else v) for k, v in w.items()}
        want = oracle.bert_forward(seen, ids, mask, seg, layers, heads)
        for k, ref in want.items():
            assert np.array_equal(got[k], again[k]), what + ": " + k + " differs between two calls"
            assert_close(got[k], ref, 5e-5 if compute_type == 0 else 2 * FP16_TOL, what + ": " + k)


@pytest.mark.parametrize("name,rows", CONFIG_CASES)
def test_benchmark_configurations(cb, name, rows):
    """The five workloads at their real shapes (BERT-base / BERT-large, random-init N(0, 0.02))."""
    from cubert_amd.testing import CONFIGS, config_inputs, config_weights
    cfg = CONFIGS[name]
    m = cfg["model"]
    w = config_weights(name, seed=0)
    ids, mask, seg = config_inputs(name, seed=0)
    half = cfg["dtype"] == "f16"
    got, want, n = run_both(cb, w, ids, mask, seg, m["layers"], m["heads"], cfg["batch"], int(half), oracle_rows=rows)
    tol = FP16_TOL if half else FP32_TOL
    report = {}
    for k in ("pooled_output", "logits", "probs") + (() if half else ("sequence_output", "embedding_output")):
        report[k] = assert_close(got[k][:n], want[k], tol, "%s %s" % (name, k))
    if half:
        # Token-level outputs of the fp16 path, element by element, with the reference's own absolute tolerances for
        # outputs of order 1: 3e-4 on the embedding output (BertTest.cpp:96-101; its 2e-3 is for one larger element)
        # and 1e-2 on the encoder output (TransformerTest.cpp:330-341).  LayerNorm outputs of 768 ... 1024 channels
        # reach 5 ... 9, where one fp16 rounding alone is up to 2^-11 |x| (2e-3 at 4, 3.9e-3 at 8), so the embedding
        # bound carries that term and the encoder bound scales with elements above 1.
        d = {k: np.abs(got[k][:n].astype(np.float64) - want[k]) for k in ("embedding_output", "sequence_output")}
        size = {k: np.abs(want[k]) for k in d}
        assert (d["embedding_output"] <= 3e-4 + size["embedding_output"] * 2.0 ** -11).all(), \
            (name, float((d["embedding_output"] - size["embedding_output"] * 2.0 ** -11).max()))
        assert (d["sequence_output"] <= 1e-2 * np.maximum(1.0, size["sequence_output"])).all(), \
            (name, float((d["sequence_output"] / np.maximum(1.0, size["sequence_output"])).max()))
        for k in d:
            report[k] = rel_err(got[k][:n], want[k])
            report[k + " (abs)"] = float(d[k].max())
            report[k + " (rms)"] = float(np.sqrt((d[k] ** 2).mean()))
            report[k + " (largest)"] = float(size[k].max())
    print("\n%s relative errors vs oracle: %s" % (name, {k: "%.2e" % v for k, v in report.items()}))
    # size-independent properties at the full batch
    np.testing.assert_allclose(got["probs"].sum(-1), 1.0, atol=2e-3 if half else 1e-5)
    assert np.isfinite(got["sequence_output"]).all()
    if cfg["pooler"]:
        assert np.abs(got["pooled_output"]).max() <= 1.0
    else:
        np.testing.assert_allclose(got["pooled_output"], got["sequence_output"].mean(1), atol=2e-3)
    # LayerNorm with gamma = 1, beta = 0: every output row has mean 0 and variance 1
    seq = got["sequence_output"].astype(np.float64)
    np.testing.assert_allclose(seq.mean(-1), 0.0, atol=2e-3 if half else 1e-5)
    np.testing.assert_allclose(seq.var(-1), 1.0, atol=1e-2 if half else 1e-4)


def test_two_term_fp16_dense_of_an_fp32_model(cb, monkeypatch):
    """CUBERT_FP32_DENSE=f16x3 (read when a model is opened): the Dense layers of an fp32 model on the fp16 matrix
    cores from two-term operands.  Same bound as the default path, 1e-5 of the oracle, at the full C1 shape and on a
    small model with a scattered mask and random LayerNorm weights at 416 tokens; a request of 32 tokens keeps the
    fp32 kernels."""
    from cubert_amd.testing import CONFIGS, config_inputs, config_weights, random_bert_weights, random_inputs
    monkeypatch.setenv("CUBERT_FP32_DENSE", "f16x3")
    cfg = CONFIGS["C1"]
    m = cfg["model"]
    w = config_weights("C1", seed=0)
    ids, mask, seg = config_inputs("C1", seed=0)
    bert = cb.Bert(w, cfg["batch"], cfg["seq_length"], m["layers"], m["heads"], 0)
    bert.profile(["dense_split", "dense_gemm"])
    got = bert.forward(ids, mask, seg)
    counts = bert.profile_read()
    # the form was in use: one split pass, for the first layer's input (the other Dense inputs are written in two-term
    # form by the attention, LayerNorm and GELU kernels themselves)
    assert counts["dense_split"][1] == 1 and counts["dense_gemm"][1] >= 4 * m["layers"], counts
    one = bert.forward(ids[:1], mask[:1], seg[:1])               # 32 tokens: fp32 few-token kernels
    assert "dense_split" not in bert.profile_read()
    few = bert.forward(ids[:11], mask[:11], seg[:11])            # 352 tokens: the form on the kernels for small requests
    assert bert.profile_read()["dense_split"][1] == 1
    bert.close()
    want = oracle.bert_forward(w, ids, mask, seg, m["layers"], m["heads"])
    report = {}
    for k in ("pooled_output", "logits", "probs", "sequence_output", "embedding_output"):
        report[k] = assert_close(got[k], want[k], FP32_TOL, "C1 two-term " + k)
        assert_close(one[k], want[k][:1], FP32_TOL, "C1 single request " + k)
        assert_close(few[k], want[k][:11], FP32_TOL, "C1 eleven requests " + k)
    print("\nC1 two-term Dense, relative errors vs oracle: %s" % {k: "%.2e" % v for k, v in report.items()})

    w = random_bert_weights(seed=3, labels=3, pooler=True, classifier=True, classifier_bias=True, ln_random=True,
                            **SMALL)
    ids, mask, seg = random_inputs(seed=4, batch=13, seq_length=32, vocab=SMALL["vocab"], min_valid=2,
                                   segment_split="random", scattered_mask=True)
    got, want, _ = run_both(cb, w, ids, mask, seg, 3, 4, max_batch=14)
    for k in ("embedding_output", "sequence_output", "pooled_output", "logits", "probs"):
        assert_close(got[k], want[k], FP32_TOL, "small two-term " + k)


def test_sequences_of_a_batch_are_independent_at_full_size(cb):
    """A size-independent property at a benchmark shape (C2: fp16, batch 32 x seq 128, heavy padding): permuting the
    sequences of a batch permutes the outputs, and a sequence computed alone gives what it gives inside the batch."""
    from cubert_amd.testing import CONFIGS, config_inputs, config_weights
    cfg = CONFIGS["C2"]
    m = cfg["model"]
    w = config_weights("C2", seed=0)
    ids, mask, seg = config_inputs("C2", seed=0)
    perm = np.random.default_rng(5).permutation(cfg["batch"])
    bert = cb.Bert(w, cfg["batch"], cfg["seq_length"], m["layers"], m["heads"], 1)
    first = bert.forward(ids, mask, seg)
    moved = bert.forward(ids[perm], mask[perm], seg[perm])
    alone = bert.forward(ids[3:4], mask[3:4], seg[3:4])
    bert.close()
    for k in ("pooled_output", "sequence_output"):
        assert_close(moved[k], first[k][perm], 2e-3, "permuted batch, " + k)
        assert_close(alone[k], first[k][3:4], 2e-3, "single sequence, " + k)


@pytest.mark.parametrize("name", ["C1", "C3"])
def test_masked_positions_reach_no_kept_position_at_full_size(cb, name):
    """A size-independent property of the mask at benchmark shapes (C1: fp32, 128 x 32, prefix masks; C3: fp16, 64 x 512,
    heavy padding, where the attention kernel leaves out key tiles without a kept key): a masked key sits 10000 below
    every kept one, its exponential is exactly 0 in fp32, so what the tokens at masked positions are -- ids and segment
    ids -- cannot change a single bit at any kept position, nor in the BertPooler's output, the logits or the
    probabilities (all from position 0, which is kept).  The outputs at the masked positions themselves do change."""
    from cubert_amd.testing import CONFIGS, config_inputs, config_weights
    cfg = CONFIGS[name]
    m = cfg["model"]
    batch = min(cfg["batch"], 32)
    w = config_weights(name, seed=0)
    ids, mask, seg = config_inputs(name, seed=0, batch=batch)
    assert mask[:, 0].all() and not mask.all()
    rng = np.random.default_rng(17)
    other_ids = np.where(mask != 0, ids, rng.integers(0, m["vocab"], ids.shape, dtype=np.int32)).astype(np.int32)
    other_seg = np.where(mask != 0, seg, 1 - seg).astype(np.int8)
    bert = cb.Bert(w, batch, cfg["seq_length"], m["layers"], m["heads"], 0 if cfg["dtype"] == "f32" else 1)
    first = bert.forward(ids, mask, seg, to_float=False)
    second = bert.forward(other_ids, mask, other_seg, to_float=False)
    bert.close()
    kept = mask != 0
    for k in ("logits", "probs"):
        assert np.array_equal(first[k], second[k]), k
    if cfg["pooler"]:
        assert np.array_equal(first["pooled_output"], second["pooled_output"])
    for k in ("sequence_output", "embedding_output"):
        assert np.array_equal(first[k][kept], second[k][kept]), k + " at kept positions"
    assert not np.array_equal(first["embedding_output"][~kept], second["embedding_output"][~kept])


# ------------------------------------------------------------------ the public C API on a GraphDef file

@pytest.fixture(scope="module")
def small_pb(tmp_path_factory):
    from cubert_amd.graphdef import write_graphdef
    from cubert_amd.testing import random_bert_weights
    w = random_bert_weights(seed=9, labels=2, **SMALL)
    path = str(tmp_path_factory.mktemp("pb") / "bert_small.pb")
    write_graphdef(path, w)
    return path, w


def test_open_compute_every_output_type(cb, small_pb):
    from cubert_amd.testing import random_inputs
    path, w = small_pb
    ids, mask, seg = random_inputs(seed=10, batch=5, seq_length=32, vocab=SMALL["vocab"], min_valid=3, segment_split=9)
    want = oracle.bert_forward(w, ids, mask, seg, 3, 4)
    model = cb.Model(path, 8, 32, 3, 4)
    assert (model.hidden_size, model.num_labels, model.seq_length) == (128, 2, 32)
    shapes = {cb.OutputType.LOGITS: ("logits", (5, 2)), cb.OutputType.PROBS: ("probs", (5, 2)),
              cb.OutputType.POOLED_OUTPUT: ("pooled_output", (5, 128)),
              cb.OutputType.SEQUENCE_OUTPUT: ("sequence_output", (5, 32, 128)),
              cb.OutputType.EMBEDDING_OUTPUT: ("embedding_output", (5, 32, 128))}
    for ot, (key, shape) in shapes.items():
        out = np.zeros(shape, np.float32)
        model.compute(ids, mask, seg, out, ot)
        assert_close(out, want[key], FP32_TOL, key)
    # several outputs in one call
    o = cb.Output()
    o.logits = np.zeros((5, 2), np.float32)
    o.sequence_output = np.zeros((5, 32, 128), np.float32)
    model.compute_m(ids, mask, seg, o)
    assert_close(o.logits, want["logits"], FP32_TOL)
    assert_close(o.sequence_output, want["sequence_output"], FP32_TOL)
    model.close()


@pytest.mark.parametrize("compute_type", ["float", "half"])
def test_open_a_graphdef_written_the_way_tensorflow_writes_one(cb, compute_type):
    """cuBERT_open on the protobuf-library-written fixture (scalar Consts in float_val / half_val, non-Const nodes,
    a function library, a DT_HALF weight among DT_FLOAT ones): all five outputs against the oracle on the tensors
    the fixture's generator recorded."""
    from cubert_amd.testing import random_bert_weights, random_inputs
    from util import tf_style_fixture
    path, w, _ = tf_style_fixture()
    model_names = set(random_bert_weights(seed=0, labels=3, vocab=37, hidden=16, layers=2, heads=2, intermediate=32,
                                          max_position=12, type_vocab=2))
    w = {k: v for k, v in w.items() if k in model_names}   # the fixture keeps each tensor's shape
    assert len(w) == len(model_names)
    half = compute_type == "half"
    if half:
        w = {k: oracle.round_to_half(v) for k, v in w.items()}
    ids, mask, seg = random_inputs(seed=31, batch=3, seq_length=8, vocab=37, min_valid=2, segment_split=5)
    want = oracle.bert_forward(w, ids, mask, seg, 2, 2)
    ct = cb.ComputeType.HALF if half else cb.ComputeType.FLOAT
    model = cb.Model(path, 4, 8, 2, 2, ct)
    assert (model.hidden_size, model.num_labels, model.seq_length) == (16, 3, 8)
    o = cb.Output()
    dt = np.float16 if half else np.float32
    o.logits, o.probs = np.zeros((3, 3), dt), np.zeros((3, 3), dt)
    o.pooled_output = np.zeros((3, 16), dt)
    o.sequence_output, o.embedding_output = np.zeros((3, 8, 16), dt), np.zeros((3, 8, 16), dt)
    model.compute_m(ids, mask, seg, o)
    model.close()
    for k in ("logits", "probs", "pooled_output", "sequence_output", "embedding_output"):
        assert_close(getattr(o, k).astype(np.float32), want[k], FP16_TOL if half else FP32_TOL, k)


def test_open_half_and_output_to_float(cb, small_pb):
    from cubert_amd.testing import random_inputs
    path, w = small_pb
    ids, mask, seg = random_inputs(seed=11, batch=4, seq_length=32, vocab=SMALL["vocab"], min_valid=3)
    want = oracle.bert_forward({k: oracle.round_to_half(v) for k, v in w.items()}, ids, mask, seg, 3, 4)
    model = cb.Model(path, 4, 32, 3, 4, cb.ComputeType.HALF)  # float file converted to half at load
    out16 = np.zeros((4, 2), np.float16)
    model.compute(ids, mask, seg, out16, cb.OutputType.LOGITS)
    o = cb.Output()
    o.logits = np.zeros((4, 2), np.float32)
    o.pooled_output = np.zeros((4, 128), np.float32)
    model.compute_m(ids, mask, seg, o, output_to_float=True)
    model.close()
    assert_close(out16.astype(np.float32), want["logits"], FP16_TOL)
    assert np.array_equal(out16.astype(np.float32), o.logits)
    assert_close(o.pooled_output, want["pooled_output"], FP16_TOL)


def test_tokenize_compute(cb, small_pb, tmp_path):
    """cuBERT_tokenize_compute(_m) (reference: src/cuBERT.cpp:216-280, test/cuBERT_test.cpp:58-107): texts in,
    outputs equal to cuBERT_compute on the ids the oracle's convert_single_example gives, and to the oracle's
    forward pass on them.  The vocabulary is made of characters and word pieces with ids inside the small
    model's 211-row embedding table."""
    from oracle import tokenizer as otok
    path, w = small_pb
    lines = ["[PAD]", "[UNK]", "[CLS]", "[SEP]"] + list("abcdefghijklmnopqrstuvwxyz0123456789,.!?") + \
            ["##" + c for c in "abcdefghijklmnopqrstuvwxyz"] + ["the", "##ing", "run", "知", "乎", "在", "家", "刷"]
    assert len(lines) < SMALL["vocab"]
    vocab_path = tmp_path / "vocab.txt"
    vocab_path.write_text("\n".join(lines) + "\n", encoding="utf8")
    vocab = otok.load_vocab(lines)
    text_a = ["知乎", "The running DOG, again!", "x", "Ünïcödé and more and more and more words than fit in here ok"]
    text_b = ["在家刷知乎", "what?", "", "second part that is also rather long, to force truncation of both"]
    model = cb.Model(path, 8, 32, 3, 4, vocab_file=str(vocab_path))
    for b in (text_b, None):
        feats = [otok.convert_single_example(vocab, 32, a, None if b is None else b[i]) for i, a in enumerate(text_a)]
        ids = np.array([f[0] for f in feats], np.int32)
        mask = np.array([f[1] for f in feats], np.int8)
        seg = np.array([f[2] for f in feats], np.int8)
        want = oracle.bert_forward(w, ids, mask, seg, 3, 4)
        direct = np.zeros((4, 2), np.float32)
        model.compute(ids, mask, seg, direct, cb.OutputType.LOGITS)
        out = np.zeros((4, 2), np.float32)
        model.tokenize_compute(text_a, b, out, cb.OutputType.LOGITS)
        assert np.array_equal(out, direct)
        assert_close(out, want["logits"], FP32_TOL, "tokenize_compute logits")
        o = cb.Output()
        o.probs = np.zeros((4, 2), np.float32)
        o.pooled_output = np.zeros((4, 128), np.float32)
        model.tokenize_compute_m(text_a, b, o)
        assert_close(o.probs, want["probs"], FP32_TOL, "tokenize_compute_m probs")
        assert_close(o.pooled_output, want["pooled_output"], FP32_TOL, "tokenize_compute_m pooled")
    with pytest.raises(ValueError):
        model.tokenize_compute(text_a, text_b[:2], np.zeros((4, 2), np.float32))
    model.close()
    plain = cb.Model(path, 8, 32, 3, 4)
    with pytest.raises(ValueError, match="vocab_file"):
        plain.tokenize_compute(text_a, None, np.zeros((4, 2), np.float32))
    plain.close()


def test_models_per_gpu_must_be_a_sane_count(cb, small_pb, monkeypatch):
    path, _ = small_pb
    for bad in ("0", "-2", "1000", "x"):
        monkeypatch.setenv("CUBERT_MODELS_PER_GPU", bad)
        with pytest.raises(ValueError):
            cb.Model(path, 4, 32, 3, 4)


def test_two_term_dense_falls_back_to_fp32_when_an_activation_does_not_fit(cb, monkeypatch):
    """CUBERT_FP32_DENSE=f16x3 with a model whose LayerNorm scales push activations beyond what two fp16 terms can
    hold (|16 x| > 65504): the request is recomputed on the fp32 GEMMs and its outputs are, bit for bit, those of the
    same model opened without the variable; a request that fits still runs (and stays within 1e-5 of the oracle) in the
    two-term form afterwards."""
    from cubert_amd.testing import random_bert_weights, random_inputs
    w = random_bert_weights(seed=23, labels=3, pooler=True, classifier=True, classifier_bias=True, ln_random=True,
                            **SMALL)
    big = dict(w)
    name = "bert/encoder/layer_1/attention/output/LayerNorm/gamma"
    big[name] = (w[name] * 9000.0).astype(np.float32)            # that layer's LayerNorm outputs reach ~ 3e4
    ids, mask, seg = random_inputs(seed=24, batch=13, seq_length=32, vocab=SMALL["vocab"], min_valid=2,
                                   segment_split="random", scattered_mask=True)
    plain = cb.Bert(big, 14, 32, 3, 4)
    want_big = plain.forward(ids, mask, seg)
    plain.close()
    monkeypatch.setenv("CUBERT_FP32_DENSE", "f16x3")
    for weights, expect_fallback in ((big, True), (w, False)):
        bert = cb.Bert(weights, 14, 32, 3, 4)
        bert.profile(["dense_split", "dense_gemm"])
        got = bert.forward(ids, mask, seg)                       # 416 tokens: the two-term form applies
        counts = bert.profile_read()
        assert counts["dense_split"][1] >= 1                     # ... and was tried
        if expect_fallback:
            # tried (4 GEMMs per layer + pooler and classifier), then all of it again in fp32
            assert counts["dense_gemm"][1] >= 2 * 4 * 3, counts
            for k in ("embedding_output", "sequence_output", "pooled_output", "logits", "probs"):
                assert np.array_equal(got[k].view(np.uint32), want_big[k].view(np.uint32)), k
            # single outputs through the other output methods take the same route
            again = bert.forward(ids, mask, seg)
            assert np.array_equal(again["logits"].view(np.uint32), want_big["logits"].view(np.uint32))
        else:
            assert counts["dense_gemm"][1] < 2 * 4 * 3, counts
            want = oracle.bert_forward(weights, ids, mask, seg, 3, 4)
            for k in ("embedding_output", "sequence_output", "pooled_output", "logits", "probs"):
                assert_close(got[k], want[k], FP32_TOL, "two-term " + k)
        bert.close()


def scaled_layers(w, factors):
    """The model with the named tensors of every layer multiplied by their factors."""
    out = dict(w)
    for name in w:
        for part, factor in factors.items():
            if name.endswith(part) and "/layer_" in name:
                out[name] = (w[name] * np.float32(factor)).astype(np.float32)
    return out


@pytest.mark.parametrize("factors", [
    {},
    {"value/kernel": 2.0 ** -12, "value/bias": 2.0 ** -12, "attention/output/dense/kernel": 2.0 ** 12},  # the same function
    {"LayerNorm/gamma": 2.0 ** -9, "LayerNorm/beta": 2.0 ** -9},
    {"LayerNorm/gamma": 2.0 ** 4, "LayerNorm/beta": 2.0 ** 4, "intermediate/dense/kernel": 2.0 ** -4}], ids=str)
def test_two_term_scales_follow_the_weights(cb, monkeypatch, factors):
    """An fp32 model opened without CUBERT_FP32_DENSE runs requests of enough tokens in the two-term form, with operand scales
    that its weights prove to be safe: however sizes are shared out between neighbouring tensors, the result is no further
    from float64 than the fp32 GEMM's."""
    from cubert_amd.testing import random_bert_weights, random_inputs
    m = dict(vocab=97, hidden=512, layers=2, heads=8, intermediate=2048, max_position=64, type_vocab=2)
    w = scaled_layers(random_bert_weights(seed=61, labels=2, pooler=True, classifier=True, ln_random=True, **m), factors)
    ids, mask, seg = random_inputs(seed=62, batch=20, seq_length=32, vocab=97, min_valid=3, segment_split=9)
    want = float64_tokens(w, ids, mask, seg, 2, 8)
    error = {}
    for mode in ("f32", ""):
        monkeypatch.setenv("CUBERT_FP32_DENSE", mode)
        bert = cb.Bert(w, 20, 32, 2, 8, 0)
        bert.profile(["dense_split", "bias_gelu"])
        got = bert.forward(ids, mask, seg)["sequence_output"]
        assert ("dense_split" in bert.profile_read()) == (mode == "")
        bert.close()
        error[mode] = np.linalg.norm(got - want) / np.linalg.norm(want)
    print("\nrelative error against float64: fp32 GEMM %.2e, two-term %.2e" % (error["f32"], error[""]))
    assert error[""] <= error["f32"]


def uneven_channels(w, what, most, rng):
    """The model with the channels of one operand over a range of 2^-most to 1, and what reads them scaled the other way."""
    out = dict(w)

    def scale(name, axis, factors):
        shape = [1] * out[name].ndim
        shape[axis] = -1
        out[name] = (out[name] * factors.reshape(shape).astype(np.float32)).astype(np.float32)

    for layer in range(2):
        p = "bert/encoder/layer_%d" % layer
        inner = w[p + "/intermediate/dense/kernel"].shape[1]
        s = 2.0 ** -rng.uniform(0, most, inner if what == "inner" else 512)
        if what in ("value", "query"):  # the same function
            scale(p + "/attention/self/%s/kernel" % what, 1, s)
            scale(p + "/attention/self/%s/bias" % what, 0, s)
            scale(p + ("/attention/output/dense/kernel" if what == "value" else "/attention/self/key/kernel"), 0 if what == "value" else 1, 1 / s)
            if what == "query":
                scale(p + "/attention/self/key/bias", 0, 1 / s)
        elif what == "value part":  # the same function
            for name, factor in (("/attention/self/value/kernel", 2.0 ** -most), ("/attention/self/value/bias", 2.0 ** -most),
                                 ("/attention/output/dense/kernel", 2.0 ** most)):
                scale(p + name, 0, np.full(1, factor))
        elif what == "inner":
            scale(p + "/intermediate/dense/kernel", 1, s)
            scale(p + "/intermediate/dense/bias", 0, s)
            scale(p + "/output/dense/kernel", 0, 1 / s)
        elif what == "norm":
            for name in ("/gamma", "/beta"):
                scale(p + "/attention/output/LayerNorm" + name, 0, s)
            scale(p + "/intermediate/dense/kernel", 0, 1 / s)
        elif what == "column":  # the same function
            factors = np.ones(512)
            factors[7] = 2.0 ** most
            scale(p + "/attention/self/value/kernel", 1, factors)
            scale(p + "/attention/self/value/bias", 0, factors)
            scale(p + "/attention/output/dense/kernel", 0, 1 / factors)
    return out


@pytest.mark.parametrize("what,most", [(what, most) for what in ("value", "inner", "norm", "query", "column")
                                       for most in (8, 10, 12, 14, 16, 24, 32)] + [("value part", 12), ("value part", 16), ("value part", 20)])
def test_two_term_form_of_uneven_channels(cb, monkeypatch, what, most):
    """Channels of very different sizes, which fp32 operands do not mind: the model as it is opened is no further from float64
    than with the fp32 GEMM, which it keeps where two terms of one scale a tensor do not hold them."""
    from cubert_amd.testing import random_bert_weights, random_inputs
    m = dict(vocab=97, hidden=512, layers=2, heads=8, intermediate=2048, max_position=64, type_vocab=2)
    w = uneven_channels(random_bert_weights(seed=67, labels=2, pooler=True, classifier=True, ln_random=True, **m), what, most,
                        np.random.default_rng(68))
    ids, mask, seg = random_inputs(seed=69, batch=20, seq_length=32, vocab=97, min_valid=3, segment_split=9)
    want = float64_tokens(w, ids, mask, seg, 2, 8)
    error = {}
    for mode in ("f32", ""):
        monkeypatch.setenv("CUBERT_FP32_DENSE", mode)
        bert = cb.Bert(w, 20, 32, 2, 8, 0)
        bert.profile(["dense_split"])
        got = bert.forward(ids, mask, seg)["sequence_output"]
        two_term = "dense_split" in bert.profile_read()
        bert.close()
        error[mode] = np.linalg.norm(got - want) / np.linalg.norm(want)
    print("\nrelative error against float64: fp32 GEMM %.2e, as opened %.2e" % (error["f32"], error[""]))
    assert error[""] <= error["f32"]
    if most <= 8 or (what == "value part" and most <= 16):
        assert two_term
    if most >= 16 and what != "value part":
        assert not two_term


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("name", ["attention/self/query", "attention/self/key", "attention/self/value", "attention/output/dense",
                                  "intermediate/dense", "output/dense"])
def test_weights_that_are_not_finite_keep_the_fp32_gemm(cb, monkeypatch, name, value):
    """Two fp16 terms cannot hold them: whether the form is asked for by name or not, the outputs are the fp32 GEMM's."""
    from cubert_amd.testing import random_bert_weights, random_inputs
    m = dict(vocab=97, hidden=256, layers=2, heads=4, intermediate=1024, max_position=64, type_vocab=2)
    w = random_bert_weights(seed=63, labels=2, pooler=True, classifier=True, ln_random=True, **m)
    ids, mask, seg = random_inputs(seed=65, batch=20, seq_length=32, vocab=97, min_valid=3, segment_split=9)
    for layer in (0, 1):
        bad = dict(w)
        kernel = "bert/encoder/layer_%d/%s/kernel" % (layer, name)
        bad[kernel] = w[kernel].copy()
        bad[kernel][3, 5] = value
        got = {}
        for mode in ("f32", "", "f16x3"):
            monkeypatch.setenv("CUBERT_FP32_DENSE", mode)
            bert = cb.Bert(bad, 20, 32, 2, 4, 0)
            got[mode] = bert.forward(ids, mask, seg)["sequence_output"]
            bert.close()
        assert np.isnan(got["f32"]).any()
        assert np.array_equal(got[""], got["f32"], equal_nan=True) and np.array_equal(got["f16x3"], got["f32"], equal_nan=True)


@pytest.mark.parametrize("batch,seq", [(1, 64), (1, 65), (3, 37), (2, 128), (1, 257), (3, 107), (11, 32), (4, 96), (2, 300), (20, 64)])
@pytest.mark.parametrize("hidden", [768, 640])
def test_two_term_form_of_small_requests(cb, monkeypatch, batch, seq, hidden):
    """From 65 tokens on the Dense layers run in the two-term form on the kernels for small requests (K slices into the LayerNorm,
    which writes rows of pairs where hidden is a multiple of 256): no further from float64 than the fp32 kernels; below, their bits."""
    from cubert_amd.testing import random_bert_weights, random_inputs
    m = dict(vocab=97, hidden=hidden, layers=2, heads=hidden // 64, intermediate=4 * hidden, max_position=300, type_vocab=2)
    w = random_bert_weights(seed=71, labels=2, pooler=True, classifier=True, ln_random=True, **m)
    ids, mask, seg = random_inputs(seed=72, batch=batch, seq_length=seq, vocab=97, min_valid=seq // 4, segment_split=9)
    want = float64_tokens(w, ids, mask, seg, 2, m["heads"])
    got = {}
    for mode in ("f32", ""):
        monkeypatch.setenv("CUBERT_FP32_DENSE", mode)
        bert = cb.Bert(w, batch, seq, 2, m["heads"], 0)
        got[mode] = bert.forward(ids, mask, seg)["sequence_output"]
        again = bert.forward(ids, mask, seg)["sequence_output"]
        assert np.array_equal(again, got[mode])
        bert.close()
    error = {k: np.linalg.norm(v - want) / np.linalg.norm(want) for k, v in got.items()}
    print("\nrelative error against float64: fp32 %.2e, as opened %.2e" % (error["f32"], error[""]))
    pays = batch * seq > 64 and batch * seq * hidden ** 2 >= (3.8e7 if hidden % 256 == 0 else 6.7e7)
    assert np.array_equal(got[""], got["f32"]) == (not pays)
    assert error[""] <= error["f32"]


@pytest.mark.parametrize("intermediate", [768, 3072])
def test_slices_have_room_whatever_the_model_was_opened_for(cb, intermediate):
    """A layer in front of a LayerNorm is cut into as many K slices in a model opened for the request alone, whose own buffers have room for
    intermediate / hidden of them, as in one opened for ten times as much: the same bits."""
    from cubert_amd.testing import random_bert_weights, random_inputs
    m = dict(vocab=97, hidden=768, layers=2, heads=12, intermediate=intermediate, max_position=64, type_vocab=2)
    w = random_bert_weights(seed=73, labels=2, pooler=True, classifier=True, ln_random=True, **m)
    ids, mask, seg = random_inputs(seed=74, batch=4, seq_length=32, vocab=97, min_valid=3, segment_split=9)
    got = []
    for most in (4, 40):
        bert = cb.Bert(w, most, 32, 2, 12, 0)
        got.append(bert.forward(ids, mask, seg)["sequence_output"])
        bert.close()
    assert np.array_equal(got[0], got[1])


def float64_tokens(w, ids, mask, seg, layers, heads):
    """The encoder's output in float64."""
    from scipy.special import erf
    w = {k: v.astype(np.float64) for k, v in w.items()}

    def norm(x, p):
        return (x - x.mean(-1, keepdims=True)) / np.sqrt(x.var(-1, keepdims=True) + 1e-12) * w[p + "/gamma"] + w[p + "/beta"]
    e = "bert/embeddings/"
    x = w[e + "word_embeddings"][ids] + w[e + "position_embeddings"][:ids.shape[1]] + w[e + "token_type_embeddings"][seg]
    x = norm(x, e + "LayerNorm")
    B, S, H = x.shape
    for layer in range(layers):
        p = "bert/encoder/layer_%d" % layer

        def dense(y, name):
            return y @ w[p + name + "/kernel"] + w[p + name + "/bias"]
        q, k, v = (dense(x, "/attention/self/" + n).reshape(B, S, heads, H // heads).transpose(0, 2, 1, 3)
                   for n in ("query", "key", "value"))
        s = q @ k.transpose(0, 1, 3, 2) / np.sqrt(H // heads) - 10000.0 * (1 - mask[:, None, None, :].astype(np.float64))
        s = np.exp(s - s.max(-1, keepdims=True))
        c = (s / s.sum(-1, keepdims=True) @ v).transpose(0, 2, 1, 3).reshape(B, S, H)
        a = norm(dense(c, "/attention/output/dense") + x, p + "/attention/output/LayerNorm")
        h = dense(a, "/intermediate/dense")
        x = norm(dense(0.5 * h * (1 + erf(h / np.sqrt(2))), "/output/dense") + a, p + "/output/LayerNorm")
    return x


def test_two_term_form_is_left_alone_where_nothing_bounds_the_input(cb, monkeypatch):
    """The encoder by itself, on inputs of any size: layer 0's attention, whose operands no weight bounds, is computed in fp32;
    tiny and huge rows come out as from the fp32 GEMM.  A model with a weight that is not a number keeps the fp32 GEMM."""
    from cubert_amd.testing import random_bert_weights, random_inputs
    m = dict(vocab=97, hidden=512, layers=2, heads=8, intermediate=2048, max_position=64, type_vocab=2)
    w = random_bert_weights(seed=63, labels=2, pooler=True, classifier=True, ln_random=True, **m)
    rng = np.random.default_rng(64)
    mask = np.ones((13, 32), np.int8)
    for size in (1e-6, 1e6):
        x = (rng.standard_normal((13, 32, 512)) * size).astype(np.float32)
        got = cb.transformer_run(w, "bert/encoder", x, mask, 2, 8, 2048, 0)
        monkeypatch.setenv("CUBERT_FP32_DENSE", "f32")
        plain = cb.transformer_run(w, "bert/encoder", x, mask, 2, 8, 2048, 0)
        monkeypatch.delenv("CUBERT_FP32_DENSE")
        assert np.isfinite(got).all() and not np.array_equal(got, plain)
        assert np.abs(got - plain).max() <= FP32_TOL * np.abs(plain).max()
    ids, mask, seg = random_inputs(seed=65, batch=13, seq_length=32, vocab=97, min_valid=3, segment_split=9)
    bad = dict(w)
    name = "bert/encoder/layer_1/attention/output/LayerNorm/beta"
    bad[name] = w[name].copy()
    bad[name][0] = np.nan
    bert = cb.Bert(bad, 13, 32, 2, 8, 0)
    bert.profile(["dense_split"])
    bert.forward(ids, mask, seg)
    assert "dense_split" not in bert.profile_read()
    bert.close()


def test_first_request_does_not_pay_for_gemm_planning(cb):
    """The constructor runs one forward pass at max_batch_size (Bert<T>::_pre_compute), so the GEMM shapes of that
    batch size are planned and timed before the first request: BERT-base width, 2 layers, batch 128 x seq 32 (Dense
    GEMMs of 4.8 ... 19 GFLOP, the size whose algorithms are chosen by timing 32 candidates)."""
    import time
    from cubert_amd.testing import BERT_BASE, random_bert_weights, random_inputs
    shape = dict(BERT_BASE, layers=2, vocab=1000, max_position=32)
    w = random_bert_weights(seed=5, labels=2, **shape)
    ids, mask, seg = random_inputs(seed=6, batch=128, seq_length=32, vocab=1000, min_valid=8)
    bert = cb.Bert(w, 128, 32, 2, 12)
    out = cb.Output(np.empty((128, 768), np.float32), cb.OutputType.POOLED_OUTPUT)
    times = []
    for _ in range(6):
        t = time.perf_counter()
        bert.compute(ids, mask, seg)
        bert.output(128, out)
        times.append((time.perf_counter() - t) * 1e3)
    bert.close()
    later = float(np.median(times[1:]))
    print("\nfirst request %.2f ms, later requests %.2f ms (median of 5)" % (times[0], later))
    assert times[0] <= 3 * later + 2.0, times
    want = oracle.bert_forward(w, ids[:4], mask[:4], seg[:4], 2, 12)["pooled_output"]
    assert_close(out.pooled_output[:4], want, FP32_TOL, "pooled output after the timed requests")


def test_listed_batch_sizes_are_prepared_at_open(cb, monkeypatch):
    """CUBERT_OPEN_WARMUP=48,max: the model prepares batch 48 as well as its maximum when it is opened, so the first
    request of 48 sequences (1536 tokens: library GEMMs of 1.8 ... 7 GFLOP, chosen by timing) costs what later ones
    cost; results are those of the oracle."""
    import time
    from cubert_amd.testing import BERT_BASE, random_bert_weights, random_inputs
    shape = dict(BERT_BASE, layers=2, vocab=1000, max_position=32)
    w = random_bert_weights(seed=15, labels=2, **shape)
    ids, mask, seg = random_inputs(seed=16, batch=48, seq_length=32, vocab=1000, min_valid=8)
    monkeypatch.setenv("CUBERT_OPEN_WARMUP", "48,max")
    bert = cb.Bert(w, 96, 32, 2, 12)
    out = cb.Output(np.empty((48, 768), np.float32), cb.OutputType.POOLED_OUTPUT)
    times = []
    for _ in range(6):
        t = time.perf_counter()
        bert.compute(ids, mask, seg)
        bert.output(48, out)
        times.append((time.perf_counter() - t) * 1e3)
    bert.close()
    later = float(np.median(times[1:]))
    print("\nfirst request of a listed size %.2f ms, later requests %.2f ms (median of 5)" % (times[0], later))
    assert times[0] <= 3 * later + 2.0, times
    want = oracle.bert_forward(w, ids[:4], mask[:4], seg[:4], 2, 12)["pooled_output"]
    assert_close(out.pooled_output[:4], want, FP32_TOL, "pooled output after the timed requests")


def test_api_error_behaviour(cb, small_pb):
    path, _ = small_pb
    with pytest.raises(ValueError, match="model file not found"):
        cb.Model("/nonexistent/model.pb", 4, 32, 3, 4)
    empty = os.path.join(os.path.dirname(path), "empty.pb")
    open(empty, "wb").close()
    with pytest.raises(ValueError, match="model file invalid"):
        cb.Model(empty, 4, 32, 3, 4)
    model = cb.Model(path, 2, 32, 3, 4)
    ids = np.zeros((3, 32), np.int32)
    m8 = np.ones((3, 32), np.int8)
    out = np.full((3, 2), 7.0, np.float32)
    with pytest.raises(ValueError, match="batch_size > max_batch_size"):
        model.compute(ids, m8, m8, out)
    with pytest.raises(ValueError, match="invalid output type"):
        model.compute(ids[:1], m8[:1], m8[:1], out, 17)
    # batch_size == 0 is a silent no-op
    model.compute(ids[:0], m8[:0], m8[:0], out)
    assert (out == 7.0).all()
    # ids outside the embedding tables are refused on the host, before anything is enqueued (the reference reads
    # out of bounds, op/Embedding.cpp:16-19); the model keeps working afterwards
    bad = ids[:2].copy()
    bad[1, 5] = SMALL["vocab"]
    with pytest.raises(ValueError, match=r"input id out of range: input_ids\[37\] = %d" % SMALL["vocab"]):
        model.compute(bad, m8[:2], m8[:2], out[:2])
    bad[1, 5] = -1
    with pytest.raises(ValueError, match="input id out of range"):
        model.compute(bad, m8[:2], m8[:2], out[:2])
    seg = m8[:2].copy()
    seg[0, 31] = 2
    with pytest.raises(ValueError, match=r"segment id out of range: segment_ids\[31\] = 2, type_vocab_size = 2"):
        model.compute(ids[:2], m8[:2], seg, out[:2])
    assert (out == 7.0).all()
    model.compute(ids[:2], m8[:2], m8[:2], out[:2])
    assert np.isfinite(out[:2]).all() and not (out[:2] == 7.0).any()
    model.close()


@pytest.mark.parametrize("models_per_gpu", [None, "3"])
def test_concurrent_callers_share_one_model(cb, small_pb, monkeypatch, models_per_gpu):
    """cuBERT_compute is thread-safe per handle (one mutex per replica held for compute + copy-out), with one
    replica per device and with CUBERT_MODELS_PER_GPU replicas (requests then overlap on the device)."""
    import threading
    from cubert_amd.testing import random_inputs
    path, w = small_pb
    if models_per_gpu is not None:
        monkeypatch.setenv("CUBERT_MODELS_PER_GPU", models_per_gpu)
    model = cb.Model(path, 4, 32, 3, 4)
    cases = [random_inputs(seed=20 + i, batch=1 + i % 4, seq_length=32, vocab=SMALL["vocab"], min_valid=2)
             for i in range(8)]
    wants = [oracle.bert_forward(w, *c, 3, 4)["logits"] for c in cases]
    errors = []

    def worker(i):
        try:
            for _ in range(5):
                out = np.zeros(wants[i].shape, np.float32)
                model.compute(*cases[i], out)
                assert_close(out, wants[i], FP32_TOL, "thread %d" % i)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=worker, args=(i,)) for i in range(8)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    model.close()
    assert not errors, errors


@pytest.mark.parametrize("batch,seq", [(1, 33), (3, 85), (32, 128), (33, 128), (64, 128), (130, 126), (200, 128)])
def test_large_outputs_reach_pageable_and_page_locked_arrays(cb, batch, seq):
    """Outputs beyond the small staging block: together less than a slot of 4 MB, more than one (pieces through two slots), a
    whole piece each, a remainder, and more pieces than slots; into ordinary and into page-locked arrays, together with small ones,
    twice in a row.  hidden 128 fp32: 512 bytes a token."""
    cfg = dict(vocab=211, hidden=128, layers=1, heads=4, intermediate=256, max_position=128, type_vocab=2)
    from cubert_amd.testing import random_bert_weights, random_inputs
    torch = pytest.importorskip("torch")
    w = random_bert_weights(seed=3, labels=2, ln_random=True, **cfg)
    bert = cb.Bert(w, batch, seq, cfg["layers"], cfg["heads"])
    for seed in (1, 2):
        ids, mask, seg = random_inputs(seed=seed, batch=batch, seq_length=seq, vocab=cfg["vocab"], min_valid=1)
        want = oracle.bert_forward(w, ids, mask, seg, cfg["layers"], cfg["heads"])
        for locked in (False, True):
            o = cb.Output()
            keep = {}
            for k, shape in (("sequence_output", (batch, seq, 128)), ("embedding_output", (batch, seq, 128)),
                             ("pooled_output", (batch, 128))):
                keep[k] = torch.full(shape, float("nan"), pin_memory=locked).numpy()
                setattr(o, k, keep[k])
            bert.compute(ids, mask, seg)
            bert.output(batch, o)
            for k, got in keep.items():
                assert_close(got, want[k], FP32_TOL, "%s %s" % (k, locked))
    bert.close()


def test_large_output_into_device_memory(cb):
    """An output that is no host array is the runtime's to write, whatever its size; NULL is no ordinary memory either."""
    from cubert_amd._lib import lib
    from cubert_amd.testing import random_bert_weights, random_inputs
    torch = pytest.importorskip("torch")
    cfg = dict(vocab=211, hidden=128, layers=1, heads=4, intermediate=256, max_position=128, type_vocab=2)
    w = random_bert_weights(seed=3, labels=2, ln_random=True, **cfg)
    bert = cb.Bert(w, 200, 128, cfg["layers"], cfg["heads"])
    ids, mask, seg = random_inputs(seed=1, batch=200, seq_length=128, vocab=cfg["vocab"], min_valid=1)
    want = bert.forward(ids, mask, seg)["sequence_output"]
    device = torch.full((200, 128, 128), float("nan"), device="cuda")
    locked, plain = torch.empty(16, pin_memory=True), np.empty(16, np.float32)
    assert [lib().cubert_is_pageable(p) for p in (None, device.data_ptr(), locked.data_ptr(), plain.ctypes.data)] == [0, 0, 0, 1]
    torch.cuda.synchronize()
    o = cb.Output()
    o._c.sequence_output = device.data_ptr()
    bert.output(200, o)
    assert np.array_equal(device.cpu().numpy(), want)
    bert.close()
