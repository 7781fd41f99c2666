"""Implicit GEMM of short reductions (csrc/implicit_gemm_short.h): wavefronts that walk over blocks of 32 pixels with the whole
filter in LDS, at the edges of blocks of pixels and channels, of stages, and of the image; and pointwise layers of few output
channels whose filter is split on its way to LDS."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -24      # of a product and of an addition, as for the other kernels of split products


@pytest.fixture(scope="module")
def lib():
    import fastconv_amd as F
    L = F.load(0, 1 << 30)
    yield L
    L.close()


def cshape(s):
    import fastconv_amd as F
    return F.ConvShape(*[getattr(s, n) for n, _ in F.ConvShape._fields_])


SHAPES = [
    (1, 1, 140, 143, 321, 3, 3, 1, 1, 1),    # one channel, a part of a block of channels and of pixels
    (9, 3, 150, 151, 33, 3, 3, 1, 1, 1),     # runs of four, windows before x, more blocks than wavefronts: every one walks
    (4, 4, 89, 88, 1030, 3, 3, 2, 2, 1),     # many groups of channels
    (6, 5, 101, 103, 100, 3, 3, 1, 1, 0),    # four stages in runs of four, as many rows as are padded
    (3, 1, 223, 222, 200, 7, 7, 2, 2, 3),    # runs of eight
    (8, 1, 99, 98, 97, 5, 5, 1, 1, 2),       # runs of eight in three stages, the last one half filled
    (1, 18, 231, 297, 85, 1, 1, 1, 1, 0),    # four pixels a lane, odd image
    (3, 40, 160, 166, 70, 1, 1, 1, 1, 0),    # three stages, channels past the last
    (3, 48, 131, 133, 129, 1, 1, 1, 1, 0),   # images that are no whole groups of four pixels
    (2, 16, 101, 101, 330, 1, 1, 1, 1, 0),   # one stage, many channels
    (2, 32, 130, 130, 500, 1, 1, 1, 1, 0),   # 64 MB of y
]
FEW = [      # of 33 to 64 output channels
    (5, 64, 140, 141, 64, 1, 1, 1, 1, 0),    # split in the kernel from the fp32 filter
    (2, 112, 223, 224, 40, 1, 1, 1, 1, 0),   # the same with 32 of its rows unused in part
    (1, 64, 332, 331, 33, 1, 1, 1, 1, 0),    # and all but one of them
]
PACKED = [   # the same, of which the filter is packed in parts
    (2, 100, 223, 224, 40, 1, 1, 1, 1, 0),   # channels past the last
    (1, 52, 333, 331, 33, 1, 1, 1, 1, 0),    # images that are no whole groups of four pixels
]


def kernel_of(lib, s):
    plan = lib.igemm_plan(cshape(s), lib.igemm_default_config(cshape(s)))
    return lib.igemm_kernel_name(plan), lib.igemm_splits_products(plan)


@pytest.mark.parametrize("shp", SHAPES + FEW + PACKED)
def test_short_reductions_against_fp64(lib, shp):
    s = O.shape(*shp)
    if shp in SHAPES:
        assert kernel_of(lib, s)[0] == "igemm_short_kernel"
    else:
        assert kernel_of(lib, s) == ("igemm_split_kernel", shp in PACKED)
    x, w = O.make_inputs(s, seed=sum(shp))
    bias = O.rng_uniform(3, (s.K,))
    # magnitudes over 2^40, as a product's rounding must not depend on the scale of its row
    x = (x * np.exp2(np.arange(s.N * s.C) % 41 - 20).reshape(s.N, s.C, 1, 1)).astype(np.float32)
    size = O.naive_conv_f64(s, np.abs(x), np.abs(w)) + np.abs(bias)[:, None, None]
    tol = (s.C * s.kh * s.kw + 41) * EPS * size + 1e-30
    truth = O.naive_conv_f64(s, x, w) + bias[:, None, None]
    for cfg in sorted({lib.igemm_default_config(cshape(s)), 1, 3, 4}):
        print("short", shp, cfg, flush=True)
        assert (np.abs(lib.implicit_gemm_conv(cshape(s), x, w, bias, False, config=cfg) - truth) <= tol).all(), cfg
        assert (np.abs(lib.implicit_gemm_conv(cshape(s), x, w, bias, True, config=cfg) - np.maximum(truth, 0.0)) <= tol).all(), cfg


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3e38, 1e30])
@pytest.mark.parametrize("shp", [SHAPES[1], SHAPES[3], SHAPES[4], SHAPES[7], SHAPES[8], FEW[1], PACKED[0]])
def test_only_values_that_are_not_finite_are_formed_again(lib, shp, value):
    s = O.shape(*shp)
    x, w = O.make_inputs(s, seed=11)
    bad = x.copy()
    bad[-1, s.C - 1, 4, 5] = value
    truth, size = O.naive_conv_f64(s, bad, w), O.naive_conv_f64(s, np.abs(bad), np.abs(w))
    hit = O.naive_conv_f64(s, (bad != x).astype(np.float32) if not np.isnan(value) else np.isnan(bad).astype(np.float32), np.ones_like(w)) > 0
    print("poison", shp, value, flush=True)
    clean, got = (lib.implicit_gemm_conv(cshape(s), v, w) for v in (x, bad))
    assert np.array_equal(got[~hit], clean[~hit])
    fin = hit & np.isfinite(truth) & np.isfinite(size)
    assert (np.abs(got[fin] - truth[fin]) <= (s.C * s.kh * s.kw + 40) * EPS * size[fin]).all()
    odd = hit & ~fin
    assert np.array_equal(got[odd], truth[odd].astype(np.float32), equal_nan=True)


@pytest.mark.parametrize("shp", PACKED + [(48, 72, 56, 56, 56, 1, 1, 1, 1, 0), (9, 68, 106, 104, 64, 1, 1, 1, 1, 0)])
def test_a_filter_packed_in_parts_is_not_split_again_in_the_kernel(lib, shp):
    """Few output channels, but channels that are no whole blocks or an odd image, so that the packed filter is split: the tile reads its
    parts (and the fp32 filter before them only for values that are not finite)."""
    s = O.shape(*shp)
    x, w = O.make_inputs(s, seed=5)
    plan = lib.igemm_plan(cshape(s), lib.igemm_default_config(cshape(s)))
    assert lib.igemm_splits_products(plan) and plan.split_k == 1 and lib.igemm_kernel_name(plan) == "igemm_split_kernel"
    mark = lib.mark()
    try:
        dx, dw, Wp, tab = lib.upload(x), lib.upload(w), lib.alloc(plan.Wp_bytes), lib.alloc(plan.table_bytes)
        y, got = lib.alloc(4 * s.K * plan.Npix), []
        lib.igemm_pack_filter(plan, dw, Wp, tab)
        for fp32 in (True, False):
            if not fp32:
                lib.fill_zero(Wp, 4 * plan.Kred_pad * plan.K_pad)
            lib.conv_implicit_gemm(plan, dx, Wp, tab, y)
            got.append(lib.download(y, (s.N, s.K, plan.OH, plan.OW)))
    finally:
        lib.release(mark)
    assert np.abs(got[0]).max() > 0 and np.array_equal(got[0], got[1])


@pytest.mark.parametrize("shp", [(8, 1, 112, 112, 100, 1, 1, 1, 1, 0), (9, 1, 140, 141, 40, 1, 1, 1, 1, 0), (16, 1, 223, 224, 70, 1, 1, 2, 2, 0)])
def test_a_single_product_is_rounded_once(lib, shp):
    s = O.shape(*shp)
    x, w = O.make_inputs(s, seed=3)
    want = x[:, :, ::s.sh, ::s.sw] * w.reshape(1, s.K, 1, 1)
    print("single product", shp, flush=True)
    assert np.array_equal(lib.implicit_gemm_conv(cshape(s), x, w), want)
