"""The requests whose speed counts: what a program that serves BERT with this library has it do.

A case is one request through the public Python interface: host arrays (or texts) in, host arrays out, on a model that
was opened before and is kept.  Sizes are those of the benchmark definition (`cubert_amd.testing.CONFIGS`: BERT-base and
BERT-large, the five workloads), of the tests (sequence lengths that are not a multiple of 32, batches of any size) and
generic ones between them.

    model       "base" or "large"
    dtype       "f32", "f16", or "two_term": an fp32 model whose Dense layers run on the fp16 matrix cores
                (CUBERT_FP32_DENSE=f16x3 when it is opened)
    batch, seq  sequences of a request; seq_length of the model
    pad         how much of a sequence is real: "none"; "some" = uniform from a quarter of it to all of it; "most" =
                16 + an exponential length of mean 96, cut at the sequence length (the benchmark's long documents)
    pooler      True: first-token dense + tanh, False: mean over the sequence
    output      "logits" (logits and probabilities), "pooled", "sequence", "embedding" or "all"
    text        True: the request is a batch of text pairs that the library tokenizes itself
"""
import functools
import math
import os
import random
import tempfile
import weakref

import numpy as np

import cubert_amd
from cubert_amd import graphdef
from cubert_amd.testing import BERT_BASE, BERT_LARGE, random_inputs

MODELS = {"base": BERT_BASE, "large": BERT_LARGE}
LABELS = 3


def _case(name, model, dtype, batch, seq, pad="some", pooler=True, output="logits", text=False):
    return {"name": name, "model": model, "dtype": dtype, "batch": batch, "seq": seq, "pad": pad, "pooler": pooler,
            "output": output, "text": text}


def listed():
    return [
        # one short query, answered while the user waits: the latency half of the headline benchmark
        _case("query f32", "base", "f32", 1, 32, pad="none"),
        # one question with its passage in half precision
        _case("query f16", "base", "f16", 1, 128, pooler=False, output="pooled"),
        # a handful of queries that arrived together, at a sequence length somebody chose for their data
        _case("few f32", "base", "f32", 5, 24),
        _case("few f16", "base", "f16", 7, 50, output="all"),
        # the headline throughput benchmark: 128 short sequences, fp32, pooled output
        _case("batch f32", "base", "f32", 128, 32, output="pooled"),
        # the same with the Dense layers in their two-term fp16 form
        _case("batch two-term", "base", "two_term", 128, 32, output="pooled"),
        # fp32 passages, a length that is no multiple of 32
        _case("passages f32", "base", "f32", 20, 100),
        # fp16 throughput at moderate length, mean-pooled embeddings
        _case("batch f16", "base", "f16", 32, 128, pooler=False, output="pooled"),
        # tagging and question answering: every token's vector goes back to the host
        _case("tagging f16", "base", "f16", 13, 384, output="sequence"),
        # long documents, mostly padding
        _case("documents f16", "base", "f16", 64, 512, pad="most"),
        # the largest job: BERT-large over a full batch
        _case("large f16", "large", "f16", 256, 128, pad="none"),
        # pairs of texts, tokenized by the library
        _case("texts f32", "base", "f32", 48, 48, text=True),
    ]


# operations of one request of the two largest listed cases per operand type: a drawn case costs no more
MAX_FLOPS = {"f32": 1.2e12, "two_term": 1.2e12, "f16": 1.5e13}


def draw(rng):
    def spread(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    while True:
        dtype = rng.choice(["f32", "f32", "f16", "f16", "f16", "two_term"])
        model = "large" if dtype == "f16" and rng.random() < 0.3 else "base"
        text = dtype != "two_term" and model == "base" and rng.random() < 0.1
        seq = spread(8, 512)
        if rng.random() < 0.4:  # many choose a power of two or a multiple of 32
            seq = rng.choice([32, 64, 96, 128, 256, 384, 512])
        case = _case("", model, dtype, spread(1, 256), seq, pad=rng.choice(["none", "some", "some", "most"]),
                     pooler=rng.random() < 0.7, output=rng.choice(["logits", "logits", "pooled", "sequence", "embedding"]),
                     text=text)
        del case["name"]
        if text and seq > 128:
            continue
        # an answer of a vector per token is asked for in batches that a host can take
        if case["output"] in ("sequence", "embedding") and case["batch"] * seq > 8192:
            case["output"] = "pooled"
        if _flops(case) <= MAX_FLOPS[dtype]:
            return case


# ---- models: opened once and kept for as long as a state uses them, as a server keeps them ---------------

class _Handle(object):
    def __init__(self, model, tokenizer_words=None):
        self.model, self.words = model, tokenizer_words


_OPEN = weakref.WeakValueDictionary()


@functools.lru_cache(maxsize=None)
def _pool(f16):
    rng = np.random.Generator(np.random.PCG64(20191))
    pool = rng.standard_normal(1 << 25, dtype=np.float32) * np.float32(0.02)
    return pool.astype(np.float16) if f16 else pool


def _weights(m, pooler, f16):
    """Normal weights (stddev 0.02, LayerNorm scales around 1), each tensor a window of one pool of random numbers."""
    pool, dt = _pool(f16), np.float16 if f16 else np.float32
    rng = np.random.Generator(np.random.PCG64(7))
    w = {}

    def normal(name, *shape):
        n = int(np.prod(shape))
        at = int(rng.integers(0, pool.size - n)) & ~7
        w[name] = pool[at:at + n].reshape(shape)

    def norm(prefix):
        w[prefix + "/gamma"] = (1 + 0.1 * rng.standard_normal(H)).astype(dt)
        w[prefix + "/beta"] = (0.1 * rng.standard_normal(H)).astype(dt)

    H, I = m["hidden"], m["intermediate"]
    normal("bert/embeddings/word_embeddings", m["vocab"], H)
    normal("bert/embeddings/token_type_embeddings", m["type_vocab"], H)
    normal("bert/embeddings/position_embeddings", m["max_position"], H)
    norm("bert/embeddings/LayerNorm")
    for layer in range(m["layers"]):
        p = "bert/encoder/layer_%d" % layer
        for n, rows, cols in (("/attention/self/query", H, H), ("/attention/self/key", H, H),
                              ("/attention/self/value", H, H), ("/attention/output/dense", H, H),
                              ("/intermediate/dense", H, I), ("/output/dense", I, H)):
            normal(p + n + "/kernel", rows, cols)
            normal(p + n + "/bias", cols)
        norm(p + "/attention/output/LayerNorm")
        norm(p + "/output/LayerNorm")
    if pooler:
        normal("bert/pooler/dense/kernel", H, H)
        normal("bert/pooler/dense/bias", H)
    normal("output_weights", LABELS, H)
    normal("output_bias", LABELS)
    return w


def _vocabulary(size):
    """[PAD], the special tokens, Chinese characters, Latin words and word endings, `size` entries in all."""
    rng = random.Random(3)
    words = ["[PAD]", "[UNK]", "[CLS]", "[SEP]", "[MASK]"] + list("abcdefghijklmnopqrstuvwxyz0123456789.,!?-")
    words += [chr(0x4E00 + i) for i in range(7000)]
    syllables = ["an", "ber", "con", "de", "er", "fi", "gra", "hi", "in", "ka", "lo", "mi", "no", "ous", "pre", "qui",
                 "ra", "ser", "tion", "un", "ver", "wo", "ly", "ing"]
    have = set(words)
    while len(words) < size:
        word = "".join(rng.choice(syllables) for _ in range(rng.randint(1, 4)))
        word = word if rng.random() < 0.7 else "##" + word
        if word not in have:
            have.add(word)
            words.append(word)
    return words[:size]


def _open(case):
    key = tuple(case[k] for k in ("model", "dtype", "batch", "seq", "pooler", "text"))
    handle = _OPEN.get(key)
    if handle is not None:
        return handle
    m, f16 = MODELS[case["model"]], case["dtype"] == "f16"
    weights = _weights(m, case["pooler"], f16)
    compute_type = cubert_amd.ComputeType.HALF if f16 else cubert_amd.ComputeType.FLOAT
    kept = os.environ.get("CUBERT_FP32_DENSE")
    if case["dtype"] == "two_term":
        os.environ["CUBERT_FP32_DENSE"] = "f16x3"
    try:
        if case["text"]:
            words = _vocabulary(m["vocab"])
            with tempfile.TemporaryDirectory() as folder:
                model_file, vocab_file = os.path.join(folder, "model.pb"), os.path.join(folder, "vocab.txt")
                graphdef.write_graphdef(model_file, weights)
                with open(vocab_file, "w", encoding="utf8") as f:
                    f.write("\n".join(words) + "\n")
                handle = _Handle(cubert_amd.Model(model_file, case["batch"], case["seq"], m["layers"], m["heads"],
                                                  compute_type, vocab_file=vocab_file), words)
        else:
            handle = _Handle(cubert_amd.Bert(weights, case["batch"], case["seq"], m["layers"], m["heads"], compute_type))
    finally:
        if kept is None:
            os.environ.pop("CUBERT_FP32_DENSE", None)
        else:
            os.environ["CUBERT_FP32_DENSE"] = kept
    _OPEN[key] = handle
    return handle


def _texts(rng, words, count, longest):
    """Titles and questions: Chinese with Latin words in between, up to about `longest` tokens."""
    latin = [w for w in words[5000:] if w.isascii() and not w.startswith("##")]
    texts = []
    for _ in range(count):
        parts = []
        for _ in range(rng.randint(4, max(5, longest))):
            r = rng.random()
            if r < 0.75:
                parts.append(chr(0x4E00 + rng.randrange(7200)))
            elif r < 0.9:
                word = rng.choice(latin)
                parts.append(" " + (word.capitalize() if rng.random() < 0.3 else word) + rng.choice(["", "ing", "s"]) + " ")
            else:
                parts.append(rng.choice("。，！？、.,?!0123456789"))
        texts.append("".join(parts))
    return texts


class _State(object):
    pass


def prepare(case, seed):
    m = MODELS[case["model"]]
    B, S, H = case["batch"], case["seq"], m["hidden"]
    s = _State()
    s.handle, s.batch = _open(case), B
    if case["text"]:
        rng = random.Random(seed)
        s.text_a = _texts(rng, s.handle.words, B, S // 2)
        s.text_b = _texts(rng, s.handle.words, B, S // 2)
    else:
        lengths = None
        rng = np.random.Generator(np.random.PCG64([seed, 1]))
        if case["pad"] == "some":
            lengths = rng.integers(max(1, S // 4), S + 1, B)
        elif case["pad"] == "most":
            lengths = np.minimum(S, 16 + np.floor(rng.exponential(96.0, B))).astype(np.int64)
        s.inputs = random_inputs(seed, B, S, m["vocab"], valid_lengths=lengths, segment_split="random" if S > 1 else None)
    f32 = case["dtype"] != "f16"
    dt = np.float32 if f32 else np.float16
    s.output = cubert_amd.Output()
    s.arrays = {}
    for field, shape, kinds in (("logits", (B, LABELS), ("logits", "all")), ("probs", (B, LABELS), ("logits", "all")),
                                ("pooled_output", (B, H), ("pooled", "all")),
                                ("sequence_output", (B, S, H), ("sequence", "all")),
                                ("embedding_output", (B, S, H), ("embedding", "all"))):
        if case["output"] in kinds:
            s.arrays[field] = np.zeros(shape, dt)
            setattr(s.output, field, s.arrays[field])
    return s


def run(state):
    model = state.handle.model
    if state.handle.words is not None:
        model.tokenize_compute_m(state.text_a, state.text_b, state.output)
    else:
        model.compute(*state.inputs)
        model.output(state.batch, state.output)
    return state.arrays


def _live_share(case):
    """The mean share of a sequence that is not padding: no other key takes part in attention."""
    S = case["seq"]
    if case["text"] or case["pad"] == "none":
        return 1.0
    if case["pad"] == "some":
        return (max(1, S // 4) + S) / (2.0 * S)
    return min(1.0, (16 + 96 * (1 - math.exp(-max(0, S - 16) / 96.0))) / S)


def _flops(case):
    m = MODELS[case["model"]]
    B, S, H, I = case["batch"], case["seq"], m["hidden"], m["intermediate"]
    tokens = B * S
    layer = 2 * tokens * (4 * H * H + 2 * H * I) + 4 * tokens * S * _live_share(case) * H
    return m["layers"] * layer + 2 * B * H * ((H if case["pooler"] else S) + LABELS)


def work(case):
    m = MODELS[case["model"]]
    B, S, H, I, e = case["batch"], case["seq"], m["hidden"], m["intermediate"], 2 if case["dtype"] == "f16" else 4
    tokens = B * S
    weights = m["layers"] * (4 * H * H + 2 * H * I + 9 * H + I) + (min(m["vocab"], tokens) + S + 2 + 2) * H
    weights += (H * H + H if case["pooler"] else 0) + LABELS * (H + 1)
    outputs = {"logits": 2 * B * LABELS, "pooled": B * H, "sequence": tokens * H, "embedding": tokens * H,
               "all": 2 * B * LABELS + B * H + 2 * tokens * H}[case["output"]]
    return {"bytes": float(e * (weights + outputs) + 6 * tokens), "flops": float(_flops(case))}


def tolerance(case):
    # About four times what the same requests differ by when every GEMM runs on the plain kernel and attention in three
    # steps (CUBERT_GEMM=naive, CUBERT_ATTENTION=split: other summation orders, scores rounded in between).  Largest seen
    # over the listed cases and ten drawn ones, relative 2-norm and largest element: f32 1.6e-6 and 6.8e-6, two_term 3.0e-6
    # and 1.4e-5, f16 1.6e-3 and 9.2e-3.
    return {"f32": {"rel": 7e-6, "max": 4e-5}, "two_term": {"rel": 1.2e-5, "max": 8e-5},
            "f16": {"rel": 6.5e-3, "max": 4e-2}}[case["dtype"]]
