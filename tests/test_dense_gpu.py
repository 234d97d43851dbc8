"""The library's own Dense kernels against float64 on the same (storage-rounded) operands."""
import numpy as np
import pytest
from scipy.special import erf

from util import DENSE_SIZES, DENSE_SLICE_SIZES

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def K():
    if not torch.cuda.is_available():
        pytest.fail("no GPU visible: the -m gpu tests must run on the MI355X box")
    from cubert_amd import kernels
    return kernels


def operands(name, tokens, features, width, pad):
    """x [tokens, width] in rows of width + pad, w as the models keep it, bias: device tensors and their float64 values."""
    rng = np.random.default_rng(tokens + 3 * features + 7 * width)
    dtype = torch.float32 if name == "f32" else torch.float16
    x = torch.from_numpy(rng.normal(0, 1, (tokens, width + pad)).astype(np.float32)).to(dtype)
    w = torch.from_numpy(rng.normal(0, 0.3, (width, features) if name == "f32" else (features, width)).astype(np.float32)).to(dtype)
    bias = torch.from_numpy(rng.normal(0, 1, features).astype(np.float32)).to(dtype)
    x64 = x[:, :width].double().numpy()
    w64 = w.double().numpy() if name == "f32" else w.double().numpy().T
    return x.cuda()[:, :width], w.cuda(), bias.cuda(), x64, w64, bias.double().numpy()


def product_bound(x64, w64):
    # fp32 additions: the longest chain holds a quarter of the products (four wavefronts share the reduction)
    return (x64.shape[1] / 4 + 16) * 2.0 ** -24 * (np.abs(x64) @ np.abs(w64))


def result_bound(name, want, product):
    # the product's error (GELU's slope is below 1.13), its approximation (1e-6 |x|), and the rounding to the storage type
    return 1.13 * product + 2e-6 * (1 + np.abs(want)) + (2.0 ** -24 if name == "f32" else 2.0 ** -11) * np.abs(want) + 6e-8


@pytest.mark.parametrize("name", ["f32", "f16"])
@pytest.mark.parametrize("tokens,features,width", DENSE_SIZES)
def test_dense_against_float64(K, name, tokens, features, width):
    x, w, bias, x64, w64, bias64 = operands(name, tokens, features, width, 16)
    bound = product_bound(x64, w64)
    for use_bias, gelu in ((True, False), (False, False), (True, True)):
        out = torch.full((tokens + 1, features + 8), 7.0, dtype=x.dtype, device="cuda")
        assert K.dense(x, w, bias if use_bias else None, gelu, out[:tokens, :features]) is not None
        got = out.double().cpu().numpy()
        want = x64 @ w64 + (bias64 if use_bias else 0.0)
        if gelu:
            want = 0.5 * want * (1 + erf(want / np.sqrt(2.0)))
        assert (np.abs(got[:tokens, :features] - want) <= result_bound(name, want, bound)).all(), (use_bias, gelu)
        assert (got[tokens:] == 7).all() and (got[:, features:] == 7).all()  # nothing beyond the result


@pytest.mark.parametrize("name", ["f32", "f16"])
@pytest.mark.parametrize("tokens,H,width", DENSE_SLICE_SIZES)
def test_dense_slices_add_up_and_reach_the_layer_norm(K, name, tokens, H, width):
    x, w, bias, x64, w64, _ = operands(name, tokens, H, width, 0)
    slices = K.dense_slices(x, w)
    assert slices is not None and slices.shape[0] >= 2
    assert (np.abs(slices.double().sum(0).cpu().numpy() - x64 @ w64) <= product_bound(x64, w64)).all()
    rng = np.random.default_rng(tokens)
    residual, beta, gamma = (torch.from_numpy(rng.normal(0, 1, s).astype(np.float32)).to(x.dtype).cuda()
                             for s in ((tokens, H), H, H))
    got = K.bias_res_ln_slices(slices, residual, bias, beta, gamma)
    if name == "f32" and H > 1024:
        assert got is None  # no fp32 row of this width in registers
        return
    added = torch.zeros_like(slices[0])
    for s in slices:  # in slice order from 0.f, then rounded: what a finished product would be
        added += s
    plain = K.bias_res_ln_(added.to(x.dtype), residual, bias, beta, gamma)
    if name == "f32":
        assert torch.equal(got, plain)
    else:
        # separately compiled kernels, at 768 halves one that adds a row in another order: the last bit of a few elements
        diff = (got.float() - plain.float()).abs()
        assert (diff <= plain.float().abs() * 2.0 ** -9 + 1e-6).all()
        assert (diff > 0).float().mean().item() < 0.01


@pytest.mark.parametrize("tokens", [1, 32, 33, 64])
@pytest.mark.parametrize("features,width", [(3072, 768), (768, 768), (768, 3072), (1024, 1024), (1024, 4096), (256, 8192),
                                            (9216, 512)])
def test_fp32_sums_of_few_tokens_are_as_short_as_the_few_token_kernels(K, tokens, features, width):
    """fp32 up to 64 tokens: the error against float64 is no larger than the few-token kernel's (K slices where the layer
    stands in front of a LayerNorm).  The two have at least 768 errors each of the same size, so their root mean squares are
    known to 1 / sqrt(2 * 768) = 2.6 % each; a single chain over a wavefront's K is 1.3 to 3.5 times as far off."""
    x, w, _, x64, w64, _ = operands("f32", tokens, features, width, 0)
    want = x64 @ w64

    def error(y):
        return np.sqrt(((y.double().cpu().numpy() - want) ** 2).mean())
    blas = K.Blas()
    few, _, _ = blas.gemm_skinny_partials(features, tokens, width, w, features, x, width)
    slices = K.dense_slices(x, w) if width >= features else None
    own = slices.sum(0) if slices is not None else K.dense(x, w)
    few = few[:, :tokens, :features].sum(0)
    blas.close()
    assert error(own) <= (1 + 2 * 0.026) * error(few), (error(own), error(few))


@pytest.mark.parametrize("name", ["f32", "f16"])
def test_dense_declines_what_it_cannot_do(K, name):
    dtype = torch.float32 if name == "f32" else torch.float16
    x = torch.zeros(64 * 1024, dtype=dtype, device="cuda")

    def operands_of(width, features, shift=0, pad=0):
        rows = x[shift:shift + 8 * (width + pad)].view(8, width + pad)[:, :width]
        return rows, x[:width * features].view((width, features) if name == "f32" else (features, width))
    assert K.dense(*operands_of(128, 64)) is not None
    assert K.dense(*operands_of(48, 64)) is None            # not whole steps of the reduction
    assert K.dense(*operands_of(128, 62)) is None           # features not a multiple of four
    assert K.dense(*operands_of(128, 64, shift=1)) is None  # misaligned rows
    assert K.dense(*operands_of(128, 64, pad=1)) is None    # rows of unaligned pitch
    assert K.dense_slices(*operands_of(128, 64)) is None    # too short to cut
    assert K.dense_slices(*operands_of(1024, 64), partial_floats=8 * 64) is None  # no room for two slices


# ---- large requests (kernels/dense_large.hip): fp32 operands as pairs of fp16 numbers --------------------------

def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _pairs(x, scale):
    """The operand rows by numpy: for every 32 values their high terms and then their low terms."""
    y = x.astype(np.float32) * np.float32(scale)
    hi = np.clip(y, -65504, 65504).astype(np.float16)
    lo = np.clip(y - hi.astype(np.float32), -65504, 65504).astype(np.float16)
    rows, width = x.shape
    return np.stack([hi.reshape(rows, -1, 32), lo.reshape(rows, -1, 32)], axis=2).reshape(rows, 2 * width)


@pytest.mark.parametrize("rows,width", [(5, 768), (3, 32), (2, 96)])
def test_rows_of_pairs_bit_exact(K, rows, width):
    rng = np.random.default_rng(rows + width)
    x = rng.normal(0, 1, (rows, width)).astype(np.float32)
    x.flat[::5] *= 1e-4
    x.flat[0] = 70000.0
    got = K.split_pairs(dev(x), 4.0).cpu().numpy()
    assert np.array_equal(got.view(np.uint16), _pairs(x, 4.0).view(np.uint16))
    # element path: an input that is not 16-byte aligned
    base = torch.zeros(rows * width + 1, device="cuda")
    base[1:] = dev(x).flatten()
    assert np.array_equal(K.split_pairs(base[1:].view(rows, width), 4.0).cpu().numpy().view(np.uint16), got.view(np.uint16))
    if width % 256 == 0:
        res = dev(rng.normal(0, 1, (rows, width)).astype(np.float32))
        beta, gamma = dev(np.zeros(width, np.float32)), dev(np.ones(width, np.float32))
        plain = K.bias_res_ln_(dev(x), res, None, beta, gamma)
        inout = dev(x)
        terms = K.bias_res_ln_split_pairs_(inout, res, None, beta, gamma, scale=16.0)
        assert torch.equal(inout, plain) and torch.equal(terms, K.split_pairs(plain, 16.0))


@pytest.mark.parametrize("batch,heads,seq,d", [(1, 12, 32, 64), (24, 12, 32, 64), (3, 4, 100, 64), (2, 3, 200, 32), (1, 2, 512, 64)])
def test_attention_rows_of_pairs(K, batch, heads, seq, d):
    rng = np.random.default_rng(batch + seq)
    qkv = dev(rng.normal(0, 1, (batch * seq, 3 * heads * d)).astype(np.float32))
    mask = (rng.random((batch, seq)) < 0.7).astype(np.int8)
    mask[:, 0] = 1
    plain = K.attention_fused(qkv, dev(mask), batch, heads, seq, d, d ** -0.5)
    got = K.attention_fused_split_pairs(qkv, dev(mask), batch, heads, seq, d, d ** -0.5, scale=16.0)
    assert torch.equal(got, K.split_pairs(plain, 16.0))


# every tile, one and fewer steps than the rings hold, tokens and features that end inside a tile
PAIR_SHAPES = [(1, 4, 32), (65, 68, 64), (129, 36, 160), (400, 768, 96), (1283, 2308, 768), (1281, 3072, 768), (2080, 2304, 768),
               (3071, 772, 3072), (4090, 2308, 768)]


@pytest.mark.parametrize("tokens,features,width", PAIR_SHAPES)
@pytest.mark.parametrize("gelu", [False, True])
def test_dense_pairs(K, tokens, features, width, gelu):
    features = (features + 31) // 32 * 32 if gelu else features
    rng = np.random.default_rng(tokens + width)
    x = dev(rng.normal(0, 1, (tokens, width)).astype(np.float32))
    w = dev(rng.normal(0, 0.05, (features, width)).astype(np.float32))
    bias = dev(rng.normal(0, 0.5, features).astype(np.float32)) if width != 160 else None
    ldo = features if gelu else features + 8
    got = K.dense_pairs(K.split_pairs(x, 16.0), K.split_pairs(w, 8192.0), bias, gelu, 1 / (16.0 * 8192.0), 16.0, ldo)
    assert got is not None
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    if bias is not None:
        want, size = want + bias.double(), size + bias.double().abs()
    # 3 width / 16 additions of 16 products each, every one rounded once relative to what has been added so far, and the dropped
    # low x low terms and representation errors (2^-22 of a product together); GELU has a slope of at most 1.13
    bound = size * ((3 * width / 16 + 16) * 2.0 ** -23 + 2.0 ** -22)
    if gelu:
        want = 0.5 * want * (1 + torch.erf(want / 2 ** 0.5))
        terms = got.double().view(tokens, -1, 2, 32)
        got = (terms[:, :, 0] + terms[:, :, 1]).reshape(tokens, features) / 16
        bound = 1.13 * bound + 5e-7 * (1 + want.abs())  # (the approximation of erf, and the two terms)
    assert bool(torch.isfinite(got).all()) and bool(((got.double() - want).abs() <= bound).all())


# the kernel for small requests: one token, tiles of 32 and 64 and what ends inside them, a step for one wavefront only, K in slices
@pytest.mark.parametrize("tokens,features,width", [(1, 4, 32), (33, 36, 96), (65, 768, 768), (120, 772, 160), (129, 3072, 768),
                                                   (300, 768, 3072), (383, 2304, 768), (1279, 768, 768)])
@pytest.mark.parametrize("gelu", [False, True])
def test_dense_pairs_small(K, tokens, features, width, gelu):
    features = (features + 31) // 32 * 32 if gelu else features
    rng = np.random.default_rng(tokens + width)
    x = dev(rng.normal(0, 1, (tokens, width)).astype(np.float32))
    w = dev(rng.normal(0, 0.05, (features, width)).astype(np.float32))
    bias = dev(rng.normal(0, 0.5, features).astype(np.float32)) if width != 160 else None
    ldo = features if gelu else features + 8
    xs, ws, alpha = K.split_pairs(x, 16.0), K.split_pairs(w, 8192.0), 1 / (16.0 * 8192.0)
    flag = torch.zeros(1, dtype=torch.int32, device="cuda")
    out = K.dense_pairs(xs, ws, bias, gelu, alpha, 16.0, ldo, overflow=flag, small=True)
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    # as in test_dense_pairs, a quarter of K to a wavefront
    bound = size * ((3 * width / 64 + 24) * 2.0 ** -23 + 2.0 ** -22)
    slices = K.dense_pairs_slices(xs, ws, alpha) if not gelu else None
    if slices is not None:
        assert slices.shape[0] >= 2
        assert bool(((slices.double().sum(0) - want).abs() <= bound).all())
        if features % 256 == 0:
            res = dev(rng.normal(0, 1, (tokens, features)).astype(np.float32))
            beta, gamma = dev(rng.normal(0, 1, features).astype(np.float32)), dev(rng.normal(1, 0.1, features).astype(np.float32))
            plain = K.bias_res_ln_slices(slices, res, bias, beta, gamma)
            norm, terms = K.bias_res_ln_slices_split_pairs(slices, res, bias, beta, gamma, scale=16.0, overflow=flag)
            assert torch.equal(norm, plain) and torch.equal(terms, K.split_pairs(plain, 16.0))
    if bias is not None:
        want, bound = want + bias.double(), bound + bias.double().abs() * 2.0 ** -22
    got = out
    if gelu:
        want = 0.5 * want * (1 + torch.erf(want / 2 ** 0.5))
        terms = out.double().view(tokens, -1, 2, 32)
        got = (terms[:, :, 0] + terms[:, :, 1]).reshape(tokens, features) / 16
        bound = 1.13 * bound + 5e-7 * (1 + want.abs())
    assert bool(torch.isfinite(got).all()) and bool(((got.double() - want).abs() <= bound).all())
    assert int(flag) == 0
    if gelu:  # values of 70000 and more in the result: the flag, and nothing that is not finite
        big = K.dense_pairs(xs, ws, bias, True, alpha, 2.0 ** 20, overflow=flag, small=True)
        assert int(flag) == (1 if float(want.abs().max()) * 2.0 ** 20 > 65536 else 0) and bool(torch.isfinite(big).all())


# tiles of 128 x 128 in two to four K slices, the last of them shorter, and what ends inside a tile; or none
@pytest.mark.parametrize("tokens,features,width,slices", [(800, 768, 3072, 4), (1537, 772, 2560, 2), (1700, 640, 2080, 3), (2700, 772, 2048, None),
                                                          (700, 768, 3072, 4)])
def test_dense_pairs_slices_of_large_requests(K, tokens, features, width, slices):
    rng = np.random.default_rng(tokens)
    x = dev(rng.normal(0, 1, (tokens, width)).astype(np.float32))
    w = dev(rng.normal(0, 0.05, (features, width)).astype(np.float32))
    xs, ws, alpha = K.split_pairs(x, 16.0), K.split_pairs(w, 8192.0), 1 / (16.0 * 8192.0)
    got = K.dense_pairs_slices(xs, ws, alpha, partial_floats=1 << 23)
    assert (got if slices is None else got.shape[0]) == slices
    if slices is not None:
        want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
        bound = size * ((3 * width / 32 + 16) * 2.0 ** -23 + 2.0 ** -22)  # as in test_dense_pairs, half of K at most to a slice
        assert bool(((got.double().sum(0) - want).abs() <= bound).all())
        # room for fewer slices than are best
        fewer = K.dense_pairs_slices(xs, ws, alpha, partial_floats=2 * tokens * features)
        assert fewer.shape[0] == 2 and bool(((fewer.double().sum(0) - want).abs() <= bound).all())


def test_dense_pairs_small_refusals(K):
    x, w = torch.zeros(40, 2 * 64, dtype=torch.float16, device="cuda"), torch.zeros(96, 2 * 64, dtype=torch.float16, device="cuda")
    assert K.dense_pairs(x, w[:94].contiguous(), None, True, small=True) is None   # rows of pairs need whole blocks of 32
    assert K.dense_pairs(x, w[:94].contiguous(), None, small=True) is None         # four features per store
    assert K.dense_pairs(x, w, None, ldo=98, small=True) is None
    assert K.dense_pairs_slices(x, w, partial_floats=40 * 96) is None              # no room for two slices
    part = torch.zeros(2, 40, 320, device="cuda")
    row = torch.zeros(40, 320, device="cuda")
    assert K.bias_res_ln_slices_split_pairs(part, row, None, row[0], row[1]) is None  # hidden = 256 k


def test_dense_pairs_takes_every_tile(K):
    tiles = {K.dense_large_plan(True, t, f, w, g) for t, f, w in PAIR_SHAPES for g in (False, True)}
    assert tiles == {(0, 256, 192), (1, 128, 128), (2, 128, 96), (3, 128, 96), (4, 64, 64)}


def test_dense_pairs_overflow_and_refusals(K):
    flag = torch.zeros(1, dtype=torch.int32, device="cuda")
    x, w = torch.zeros(70, 64, device="cuda"), torch.zeros(96, 64, device="cuda")
    xs, ws = K.split_pairs(x, 16.0), K.split_pairs(w, 16.0)
    bias = torch.full((96,), 4000.0, device="cuda")
    assert K.dense_pairs(xs, ws, bias, True, 1 / 256, 16.0, overflow=flag) is not None
    torch.cuda.synchronize()
    assert int(flag.item()) == 0       # 16 * 4000 fits
    bias[95] = 4100.0
    assert K.dense_pairs(xs, ws, bias, True, 1 / 256, 16.0, overflow=flag) is not None
    torch.cuda.synchronize()
    assert int(flag.item()) == 1
    assert K.dense_pairs(xs, ws[:94].contiguous(), None, True) is None      # rows of pairs need whole blocks of 32
    assert K.dense_pairs(xs, ws[:94].contiguous(), None) is None            # four features per store
    assert K.dense_pairs(xs, ws, None, ldo=98) is None


@pytest.mark.parametrize("tokens,features,width,tile", [(4000, 2976, 128, 0), (900, 3104, 64, 1), (70, 32, 64, 2), (900, 3008, 768, 3),
                                                        (70, 32, 256, 4)])
def test_dense_pairs_overflow_past_the_last_feature(K, tokens, features, width, tile):
    """Past the last feature a tile multiplies that feature's weights again, without its bias: a sum that only the bias brings
    into range does not raise the flag there, whatever the tile."""
    number, _, tile_features = K.dense_large_plan(True, tokens, features, width, True)
    assert number == tile and features % tile_features != 0
    flag = torch.zeros(1, dtype=torch.int32, device="cuda")
    x, w, bias = torch.ones(tokens, width, device="cuda"), torch.zeros(features, width, device="cuda"), torch.zeros(features, device="cuda")
    w[-1] = 8192.0 / width  # 16 * 8192 is out of range
    xs, ws = K.split_pairs(x, 16.0), K.split_pairs(w, 16.0)
    for last, raised in ((-6144.0, 0), (0.0, 1)):
        bias[-1] = last
        out = K.dense_pairs(xs, ws, bias, True, 1 / 256, 16.0, overflow=flag)
        torch.cuda.synchronize()
        assert int(flag.item()) == raised
        if not raised:
            assert bool((out[:, 2 * features - 33] == 16 * 2048.0).all())  # the last feature's high terms


# ---- large requests: half operands ----------------------------------------------------------------------------

LARGE_SHAPES = [(1, 8, 64), (129, 72, 128), (130, 64, 192), (700, 768, 256), (1537, 2304, 768), (2083, 3080, 768), (4090, 2312, 768),
                (4990, 3072, 768), (3001, 776, 3072), (2080, 2304, 768)]


@pytest.mark.parametrize("tokens,features,width", LARGE_SHAPES)
@pytest.mark.parametrize("gelu", [False, True])
def test_dense_large(K, tokens, features, width, gelu):
    rng = np.random.default_rng(tokens + width)
    x = dev(rng.normal(0, 1, (tokens, width)).astype(np.float16))
    w = dev(rng.normal(0, 0.05, (features, width)).astype(np.float16))
    bias = dev(rng.normal(0, 0.5, features).astype(np.float16)) if width != 192 else None
    got = K.dense_large(x, w, bias, gelu, features + 8)
    assert got is not None
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    if bias is not None:
        want, size = want + bias.double(), size + bias.double().abs()
    bound = size * (width / 16 + 16) * 2.0 ** -23  # additions of 16 products each, rounded relative to what has been added
    if gelu:
        want = 0.5 * want * (1 + torch.erf(want / 2 ** 0.5))
        bound = 1.13 * bound + 7.2e-7 * (1 + want.abs())  # (the approximation of erf)
    bound = bound + want.abs() * 2.0 ** -11 + 2.0 ** -25  # the store
    assert bool(torch.isfinite(got).all()) and bool(((got.double() - want).abs() <= bound).all())


def test_dense_large_tiles_and_refusals(K):
    tiles = {K.dense_large_plan(False, t, f, w, g) for t, f, w in LARGE_SHAPES for g in (False, True)}
    assert tiles == {(0, 256, 256), (1, 256, 192), (2, 128, 128), (3, 128, 96), (4, 128, 64)}
    x, w = torch.zeros(64, 128, dtype=torch.float16, device="cuda"), torch.zeros(64, 128, dtype=torch.float16, device="cuda")
    assert K.dense_large(x[:, :96].contiguous(), w[:, :96].contiguous()) is None  # whole lines of K
    assert K.dense_large(x, w[:60].contiguous()) is None                          # eight features per store
    assert K.dense_large(x, w, ldo=68) is None
    base = torch.zeros(64 * 128 + 1, dtype=torch.float16, device="cuda")
    assert K.dense_large(base[1:].view(64, 128), w) is None                       # 16-byte requests


def _beyond(out, tokens, features):
    """What a launch has left in the rows behind the last token and in the columns between `features` and the row pitch."""
    return torch.cat([out[tokens:].flatten(), out[:tokens, features:].flatten()])


# (256 rows more than there are tokens: what any tile could write to)
@pytest.mark.parametrize("gelu", [False, True])
@pytest.mark.parametrize("tokens,features,width", PAIR_SHAPES)
def test_dense_pairs_writes_nothing_else(K, tokens, features, width, gelu):
    from cubert_amd._lib import lib
    features = (features + 31) // 32 * 32 if gelu else features
    ldo = features if gelu else features + 200
    out = torch.full((tokens + 256, ldo), 7.0, device="cuda")
    x = K.split_pairs(torch.ones(tokens, width, device="cuda"), 16.0)
    w = K.split_pairs(torch.full((features, width), 3.0, device="cuda"), 16.0)
    assert lib().cubert_dense_pairs_f32(torch.cuda.current_stream().cuda_stream, tokens, features, width, x.data_ptr(), w.data_ptr(), None,
                                        int(gelu), 1 / 256, 16.0, out.data_ptr(), ldo, None) == 0
    assert bool((_beyond(out, tokens, features) == 7).all()) and not bool((out[:tokens, :features] == 7).any())


@pytest.mark.parametrize("gelu", [False, True])
@pytest.mark.parametrize("tokens,features,width", LARGE_SHAPES)
def test_dense_large_writes_nothing_else(K, tokens, features, width, gelu):
    from cubert_amd._lib import lib
    ldo = features + 264
    out = torch.full((tokens + 256, ldo), 7.0, dtype=torch.float16, device="cuda")
    x = torch.ones(tokens, width, dtype=torch.float16, device="cuda")
    w = torch.full((features, width), 3.0, dtype=torch.float16, device="cuda")
    assert lib().cubert_dense_large_f16(torch.cuda.current_stream().cuda_stream, tokens, features, width, x.data_ptr(), w.data_ptr(), None,
                                        int(gelu), out.data_ptr(), ldo) == 0
    assert bool((_beyond(out, tokens, features) == 7).all()) and bool((out[:tokens, :features] == 3 * width).all())
