import os

import numpy as np

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def rel_err(got, want):
    """Norm-wise relative error of a tensor: max|got - want| / max|want|."""
    got = np.asarray(got, dtype=np.float64)
    want = np.asarray(want, dtype=np.float64)
    scale = np.abs(want).max()
    return np.abs(got - want).max() / (scale if scale > 0 else 1.0)


def assert_close(got, want, tol, what=""):
    assert got.shape == want.shape, "%s: shape %s != %s" % (what, got.shape, want.shape)
    assert np.isfinite(np.asarray(got, dtype=np.float64)).all(), "%s: non-finite values" % what
    e = rel_err(got, want)
    assert e <= tol, "%s: relative error %.3g > %.3g" % (what, e, tol)
    return e


FP32_TOL = 1e-5        # north star: fp32 within 1e-5 relative of the reference path
FP16_TOL = 1e-2        # fp16 storage: 1e-2 relative on pooled / logit outputs (the reference's own fp16-vs-fp32 bound)


# (tokens, features, width) of the own Dense kernel's tests: one step, fewer steps than wavefronts, remainders of token and
# feature tiles; with DENSE_SLICE_SIZES every tile, depth and output that a model's Dense layers run with (checked in
# test_host_cpu.py, where the plan is asked)
DENSE_SIZES = [(1, 4, 64), (33, 100, 128), (31, 36, 320), (32, 2304, 768), (64, 3072, 768), (65, 768, 3072),
               (120, 3072, 768), (200, 2304, 768), (350, 2304, 768), (350, 3072, 768), (777, 1028, 192), (450, 3072, 768),
               (600, 3072, 768), (1279, 3072, 768), (130, 2304, 768)]
DENSE_SLICE_SIZES = [(1, 768, 768), (32, 768, 3072), (65, 768, 3072), (120, 768, 768), (200, 768, 3072), (350, 768, 3072),
                     (250, 768, 3072), (97, 768, 3072), (322, 1536, 6144)]


def tf_style_fixture():
    """The GraphDef written by google.protobuf from the reference's .proto field numbers
    (tests/golden/make_tf_graphdef_fixture.py): path, {name: tensor a loader must find}, [names it must not]."""
    z = np.load(os.path.join(GOLDEN, "tf_style_graphdef_expected.npz"))
    names = [str(n) for n in z["names"]]
    return (os.path.join(GOLDEN, "tf_style_graphdef.pb"), {n: z["w%03d" % i] for i, n in enumerate(names)},
            [str(n) for n in z["absent"]])
