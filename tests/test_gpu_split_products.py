"""fp32 products on the bf16 matrix cores (csrc/split_mfma.h): sizes at the edges of the tiles, the order of accuracy
of fp32 products, and operands that have no finite three-part sum."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

# Of nine partial products three are left out, together below 2^-22 of a product; the six kept are summed in fp32
# like the fp32 path's, whose own bound over n terms is n * 2^-24 of the sum of the magnitudes.
EPS_PRODUCT, EPS_SUM = 2.0 ** -22, 2.0 ** -24


@pytest.fixture(scope="module")
def lib():
    import fastconv_amd as F
    L = F.load(0, 2 << 30)
    yield L
    L.close()


def cshape(s):
    import fastconv_amd as F
    return F.ConvShape(*[getattr(s, n) for n, _ in F.ConvShape._fields_])


def bound(s, x, w):
    terms = s.C * s.kh * s.kw
    return (EPS_PRODUCT + (terms + 40) * EPS_SUM) * O.naive_conv_f64(s, np.abs(x), np.abs(w)) + 1e-30


@pytest.mark.parametrize("shp", [
    (1, 16, 8, 8, 64, 1, 1, 1, 1, 0),        # one stage, one tile, pointwise
    (2, 48, 9, 7, 65, 1, 1, 1, 1, 0),        # a pixel count no tile divides, one channel past a tile
    (1, 32, 11, 13, 127, 3, 3, 1, 1, 1),     # tap-major with border taps
    (3, 16, 10, 10, 130, 3, 3, 2, 2, 1),     # strided
    (2, 7, 12, 9, 70, 3, 3, 1, 1, 1),        # reduction with no whole channels per tap, 63 rows of 64
    (1, 3, 20, 20, 64, 7, 7, 2, 2, 3),       # 49 taps
    (1, 64, 16, 16, 256, 5, 5, 1, 1, 0),     # window inside the image
])
def test_implicit_gemm_split_products(lib, shp):
    s = O.shape(*shp)
    x, w = O.make_inputs(s, seed=sum(shp))
    # magnitudes over 2^40, as a product's rounding must not depend on the scale of its row
    x = (x * np.exp2(np.arange(s.N * s.C) % 41 - 20).reshape(s.N, s.C, 1, 1)).astype(np.float32)
    truth, tol = O.naive_conv_f64(s, x, w), bound(s, x, w)
    for cfg in lib.igemm_configs():
        if cfg.waves_k > 1 or cfg.bm % 64:
            continue
        print("split products", shp, cfg.bm, cfg.bn, flush=True)
        assert (np.abs(lib.implicit_gemm_conv(cshape(s), x, w, config=cfg.id) - truth) <= tol).all(), cfg.id


@pytest.mark.parametrize("C,K,T", [(16, 513, 9), (129, 64, 65), (100, 130, 129), (256, 33, 200)])
def test_winograd_gemm_split_products(lib, C, K, T):
    """C*K above 8192: M = U * V per frequency against fp64, every tile shape; T tiles in one row of an image."""
    s = cshape(O.shape(1, C, 6, 6 * T, K)) if T <= 170 else cshape(O.shape(T // 100, C, 60, 60, K))
    for cfg in lib.wino_configs():
        plan = lib.wino_plan(s, cfg.id)
        mark = lib.mark()
        U = O.rng_uniform(C, (64, plan.C_pad, plan.K_pad))
        V = O.rng_uniform(K, (64, plan.C_pad, plan.T_pad))
        M = lib.alloc(plan.M_bytes)
        print("split products", (C, K, T), cfg.bm, cfg.bn, cfg.bk, flush=True)
        lib.wino_gemm(plan, lib.upload(U), lib.upload(V), M)
        got = lib.download(M, (64, plan.K_pad, plan.T_pad))
        lib.release(mark)
        for f in (0, 9, 63):
            a, b = U[f].T.astype(np.float64), V[f].astype(np.float64)
            tol = (EPS_PRODUCT + (plan.C_pad + 40) * EPS_SUM) * (np.abs(a) @ np.abs(b))
            assert (np.abs(got[f] - a @ b) <= tol).all(), (cfg.id, f)


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, np.finfo(np.float32).max])
def test_values_without_a_finite_split(lib, value):
    """An infinity meets weights of both signs and nothing else: infinities of the right sign, and no NaN next to
    them; the largest float passes through a weight of 1 unchanged."""
    s = O.shape(1, 64, 14, 14, 160, 1, 1, 1, 1, 0)
    x, w = O.make_inputs(s, seed=5)
    w[0] = 0.0
    w[0, 3] = 1.0
    x[0, :, 5, 6] = 0.0
    x[0, 3, 5, 6] = value
    w[np.abs(w) < 1e-6] = 1e-6
    w[0] = 1e-6
    w[0, 3] = 1.0
    expect = (w[:, 3, 0, 0] * np.float32(value)).astype(np.float32)
    truth = O.naive_conv_f64(s, x, w)
    for cfg in lib.igemm_configs():
        print("value", value, cfg.id, flush=True)
        y = lib.implicit_gemm_conv(cshape(s), x, w, config=cfg.id)
        got = y[0, :, 5, 6]
        if np.isfinite(value):
            assert np.allclose(got, expect, rtol=2.0 ** -21, atol=0)
        else:
            assert np.array_equal(got, expect, equal_nan=True), cfg.id
        rest = np.ones((14, 14), bool)
        rest[5, 6] = False
        assert np.abs(y[0][:, rest] - truth[0][:, rest]).max() <= 1e-4
