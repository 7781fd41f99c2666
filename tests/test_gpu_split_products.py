"""fp32 products on the bf16 matrix cores (csrc/split_mfma.h): sizes at the edges of the tiles, the order of accuracy
of fp32 products, and operands that have no finite three-part sum."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

# Of nine partial products three are left out, together below 2^-24 of a product; the six kept are summed in fp32
# like the fp32 path's, whose own bound over n terms is n * 2^-24 of the sum of the magnitudes.
EPS_PRODUCT, EPS_SUM = 2.0 ** -24, 2.0 ** -24
# A sum of one term: what is left out, a last place of the last addition, which the matrix core does not round to nearest
# (2^-23), and five additions of parts of 2^-8 and less.
EPS_SINGLE = 3.1 * 2.0 ** -24


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


def tiles_in_a_row(C, K, T):
    return cshape(O.shape(1, C, 6, 6 * T, K)) if T <= 170 else cshape(O.shape(T // 100, C, 60, 60, K))


def winograd_gemm(lib, plan, U, V):
    mark = lib.mark()
    M = lib.alloc(plan.M_bytes)
    lib.wino_gemm(plan, lib.upload(U), lib.upload(V), M)
    got = lib.download(M, (64, plan.K_pad, plan.T_pad))
    lib.release(mark)
    return got


@pytest.mark.parametrize("C,K,T", [(64, 129, 9), (129, 64, 65), (100, 130, 129), (256, 33, 200), (160, 64, 65)])
def test_winograd_gemm_split_products(lib, C, K, T):
    """More than 48 channels and C*K above 8192: M = U * V per frequency against fp64, every tile shape; T tiles in one
    row of an image."""
    s = tiles_in_a_row(C, K, T)
    for cfg in lib.wino_configs():
        plan = lib.wino_plan(s, cfg.id)
        U = O.rng_uniform(C, (64, plan.C_pad, plan.K_pad))
        V = O.rng_uniform(K, (64, plan.C_pad, plan.T_pad))
        print("split products", (C, K, T), cfg.bm, cfg.bn, cfg.bk, flush=True)
        got = winograd_gemm(lib, plan, U, V)
        for f in (0, 9, 63):
            a, b = U[f].T.astype(np.float64), V[f].astype(np.float64)
            tol = (EPS_PRODUCT + (plan.C_pad + 40) * EPS_SUM) * (np.abs(a) @ np.abs(b))
            assert (np.abs(got[f] - a @ b) <= tol).all(), (cfg.id, f)


@pytest.mark.parametrize("C,K,N", [
    (48, 200, 1), (49, 200, 1),              # channels from which products are split, here with 128x128 tiles
    (64, 130, 38), (64, 130, 39),            # V and M on either side of 320 MB with these
    (64, 130, 1), (65, 130, 1),              # channels from which the smaller tiles follow
    (80, 130, 36), (80, 130, 37),            # V and M on either side of 256 MB with 64x64 tiles
    (144, 130, 30), (145, 130, 30),          # channels from which they follow at any size
    (176, 130, 1), (177, 130, 1),            # and the 256-wide tiles
])
def test_fused_and_staged_pipeline_agree_at_the_lines_of_the_split(lib, C, K, N):
    s = O.shape(N, C, 60, 60, K)
    x, w = O.make_inputs(s, seed=C)
    for cfg in (0, 1, 3, 7):
        print("line", (C, K, N), cfg, flush=True)
        assert np.array_equal(lib.winograd_conv_fused(cshape(s), x, w, config=cfg), lib.winograd_conv(cshape(s), x, w, config=cfg)), cfg


def test_sums_of_one_term_keep_fp32_accuracy(lib):
    """One channel of the filter is not zero: a partial product left out, or a first part that is cut off and not
    rounded, shows in every result (test_split_products.py)."""
    C, K, T = 160, 130, 129
    s = tiles_in_a_row(C, K, T)
    for cfg in lib.wino_configs():
        plan = lib.wino_plan(s, cfg.id)
        U = np.zeros((64, plan.C_pad, plan.K_pad), np.float32)
        k = np.arange(plan.K_pad)
        U[:, k % C, k] = O.rng_uniform(1, (64, plan.K_pad))
        V = O.rng_uniform(2, (64, plan.C_pad, plan.T_pad))
        print("one term", cfg.bm, cfg.bn, cfg.bk, flush=True)
        got = winograd_gemm(lib, plan, U, V)
        exact = U[:, k % C, k].astype(np.float64)[:, :, None] * V[:, k % C]
        assert (np.abs(got - exact) <= EPS_SINGLE * np.abs(exact)).all(), cfg.id
    s = O.shape(2, 64, 13, 11, 130, 1, 1, 1, 1, 0)
    x, w = O.make_inputs(s, seed=7)
    k = np.arange(s.K)
    keep = w[k, k % s.C, 0, 0]
    w[:] = 0.0
    w[k, k % s.C, 0, 0] = keep
    exact = keep.astype(np.float64)[None, :, None, None] * x[:, k % s.C]
    for cfg in lib.igemm_configs():
        print("one term, implicit gemm", cfg.bm, cfg.bn, cfg.waves_k, flush=True)
        assert (np.abs(lib.implicit_gemm_conv(cshape(s), x, w, config=cfg.id) - exact) <= EPS_SINGLE * np.abs(exact)).all(), cfg.id


def test_sums_with_few_terms_are_no_less_exact_than_with_fp32_products(lib):
    """n of 256 channels of the filter are not zero: the 2-norm error of every tile shape against 64 bits is no larger
    than that of the shapes that run on fp32 instructions (a tenth for the single term, whose parts are not rounded alike)."""
    C, K, T = 256, 130, 129
    s = tiles_in_a_row(C, K, T)
    for n in (1, 4, 16, 64, 256):
        err = {}
        for cfg in lib.wino_configs():
            plan = lib.wino_plan(s, cfg.id)
            rng = np.random.default_rng(n)
            U = rng.standard_normal((64, plan.C_pad, plan.K_pad), np.float32)
            U *= np.argsort(rng.random((C, plan.K_pad)), axis=0) < n
            V = rng.standard_normal((64, plan.C_pad, plan.T_pad), np.float32)
            print("terms", n, cfg.bm, cfg.bn, cfg.bk, flush=True)
            got = winograd_gemm(lib, plan, U, V)
            exact = U[::9].transpose(0, 2, 1).astype(np.float64) @ V[::9].astype(np.float64)
            err[cfg.bm % 64 == 0 and cfg.bn % 64 == 0 and cfg.bk == 16, cfg.id] = np.linalg.norm(got[::9] - exact) / np.linalg.norm(exact)
        fp32 = min(e for (split, _), e in err.items() if not split)
        assert all(e <= (1.1 if n == 1 else 1.0) * fp32 for (split, _), e in err.items() if split), (n, err)


def test_small_operands_keep_their_last_places(lib):
    """Filter values down to the smallest subnormal float (one channel an output) meet large inputs, and the other way
    round: the product is an ordinary number and as exact as any other."""
    C, K, T = 160, 130, 129
    s = tiles_in_a_row(C, K, T)
    for cfg in lib.wino_configs():
        plan = lib.wino_plan(s, cfg.id)
        k, t = np.arange(plan.K_pad), np.arange(plan.T_pad)
        for small_filter in (True, False):
            small = np.exp2(-149.0 + np.arange(C) % 50)[None, :, None]      # 2^-149 .. 2^-100, by channel
            large = np.exp2(90.0)
            U = np.zeros((64, plan.C_pad, plan.K_pad), np.float32)
            V = np.zeros((64, plan.C_pad, plan.T_pad), np.float32)
            U[:, k % C, k] = O.rng_uniform(1, (64, plan.K_pad), 1.0, 2.0)
            V[:, :C] = O.rng_uniform(2, (64, C, plan.T_pad), 1.0, 2.0)
            if small_filter:
                U[:, :C] *= small
                V *= np.float32(large)
            else:
                U *= np.float32(large)
                V[:, :C] *= small
            print("small operands", cfg.bm, cfg.bn, cfg.bk, small_filter, flush=True)
            got = winograd_gemm(lib, plan, U, V)
            exact = U[:, k % C, k].astype(np.float64)[:, :, None] * V[:, k % C]
            assert (np.abs(got - exact) <= EPS_SINGLE * np.abs(exact)).all(), (cfg.id, small_filter)
    s = O.shape(1, 64, 13, 11, 130, 1, 1, 1, 1, 0)
    x = O.rng_uniform(3, (s.N, s.C, s.H, s.W), 1.0, 2.0) * np.float32(2.0 ** 90)
    w = np.zeros((s.K, s.C, 1, 1), np.float32)
    k = np.arange(s.K)
    w[k, k % s.C, 0, 0] = O.rng_uniform(4, (s.K,), 1.0, 2.0) * np.exp2(-149.0 + k % 50)
    exact = w[k, k % s.C, 0, 0].astype(np.float64)[None, :, None, None] * x[:, k % s.C]
    for cfg in lib.igemm_configs():
        print("small operands, implicit gemm", cfg.bm, cfg.bn, cfg.waves_k, flush=True)
        assert (np.abs(lib.implicit_gemm_conv(cshape(s), x, w, config=cfg.id) - exact) <= EPS_SINGLE * np.abs(exact)).all(), cfg.id


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


POISON = [np.inf, -np.inf, np.nan, 3e38, 1e30]      # the last two are finite, but their scaled parts or sums are not


@pytest.mark.parametrize("value", POISON)
def test_winograd_gemm_forms_only_values_that_are_not_finite_again(lib, value):
    """One value in V and one in U, in different quarters of the larger tiles: their column and row as fp64 has them,
    everything else with the bits of a run without them."""
    C, K, T = 160, 200, 200
    s = tiles_in_a_row(C, K, T)
    for cfg in lib.wino_configs():
        plan = lib.wino_plan(s, cfg.id)
        U = O.rng_uniform(C, (64, plan.C_pad, plan.K_pad))
        V = O.rng_uniform(K, (64, plan.C_pad, plan.T_pad))
        print("poison", value, cfg.bm, cfg.bn, cfg.bk, flush=True)
        clean = winograd_gemm(lib, plan, U, V)
        V[9, 100, 150] = value
        U[9, 3, 70] = value
        U[9, 100, 70] = V[9, 3, 150] = 0.5      # the two meet numbers
        got = winograd_gemm(lib, plan, U, V)
        rest = np.ones(got.shape, bool)
        rest[9, 70, :] = rest[9, :, 150] = False
        assert np.array_equal(got[rest], clean[rest]), cfg.id
        with np.errstate(invalid="ignore"):
            a, b = U[9].T.astype(np.float64), V[9].astype(np.float64)
            exact, size = a @ b, np.abs(a) @ np.abs(b)
        for line, e, z in ((got[9, 70], exact[70], size[70]), (got[9, :, 150], exact[:, 150], size[:, 150])):
            fin = np.isfinite(e)
            assert np.array_equal(line[~fin], e[~fin].astype(np.float32), equal_nan=True), cfg.id
            assert (np.abs(line[fin] - e[fin]) <= (plan.C_pad + 40) * EPS_SUM * z[fin]).all(), cfg.id


@pytest.mark.parametrize("value", POISON)
def test_winograd_layer_with_values_that_are_not_finite(lib, value):
    """One pixel of one image: the other images keep their bits, staged and fused pipeline give the same."""
    s = O.shape(3, 160, 13, 12, 72)
    x, w = O.make_inputs(s, seed=9)
    bias = O.rng_uniform(5, (s.K,))
    for cfg in lib.wino_configs():
        print("poison", value, cfg.bm, cfg.bn, cfg.bk, flush=True)
        clean = lib.winograd_conv(cshape(s), x, w, bias, True, config=cfg.id)
        bad = x.copy()
        bad[1, 100, 6, 5] = value
        staged = lib.winograd_conv(cshape(s), bad, w, bias, True, config=cfg.id)
        assert np.array_equal(staged[[0, 2]], clean[[0, 2]]), cfg.id
        assert np.array_equal(lib.winograd_conv_fused(cshape(s), bad, w, bias, True, config=cfg.id), staged, equal_nan=True), cfg.id
        hit = staged[1, :, 5:8, 4:7]      # the 3x3 windows that hold the pixel
        assert np.isnan(hit).all() if np.isnan(value) else not np.array_equal(hit, clean[1, :, 5:8, 4:7])


@pytest.mark.parametrize("value", POISON)
@pytest.mark.parametrize("shp", [
    (2, 64, 9, 10, 130, 3, 3, 1, 1, 1),      # split reduction, border taps, channels past a tile
    (2, 64, 12, 12, 256, 1, 1, 1, 1, 0),     # whole tiles, no split reduction
    (2, 7, 11, 12, 128, 3, 3, 1, 1, 1),      # table gather
])
def test_implicit_gemm_forms_only_values_that_are_not_finite_again(lib, shp, value):
    s = O.shape(*shp)
    x, w = O.make_inputs(s, seed=11)
    bias = O.rng_uniform(6, (s.K,))
    bad = x.copy()
    bad[1, 3, 4, 5] = value
    truth = np.maximum(O.naive_conv_f64(s, bad, w, bias), 0.0)
    size = O.naive_conv_f64(s, np.abs(bad), np.abs(w)) + 1.0
    r = s.kh // 2
    hit = np.zeros(truth.shape, bool)
    hit[1, :, 4 - r:5 + r, 5 - r:6 + r] = True
    for cfg in lib.igemm_configs():
        print("poison", value, shp, cfg.bm, cfg.bn, cfg.waves_k, flush=True)
        clean = lib.implicit_gemm_conv(cshape(s), x, w, bias, True, config=cfg.id)
        got = lib.implicit_gemm_conv(cshape(s), bad, w, bias, True, config=cfg.id)
        assert np.array_equal(got[~hit], clean[~hit]), cfg.id
        fin = hit & np.isfinite(truth) & np.isfinite(size)
        assert (np.abs(got[fin] - truth[fin]) <= (s.C * s.kh * s.kw + 40) * EPS_SUM * size[fin]).all(), cfg.id
        odd = hit & ~(np.isfinite(truth) & np.isfinite(size))
        assert np.array_equal(got[odd], truth[odd].astype(np.float32), equal_nan=True), cfg.id
