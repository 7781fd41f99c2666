"""Implicit GEMM on split products: columns read by wider loads (window rows of three taps, four pixels of a pointwise layer), at the
edges of the image, of the tensor, of the channels and of the parts of a split reduction; parts chosen by time and their sums."""
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


WINDOWS = [      # tiles of 128 rows, strided, three columns
    (3, 15, 11, 13, 130, 3, 3, 2, 2, 1),     # a channel missing, windows before x and past its end
    (2, 47, 9, 30, 128, 3, 3, 2, 2, 0),      # no padding
    (2, 32, 12, 11, 200, 3, 3, 3, 3, 1),     # stride 3: a column no window reads
    (2, 16, 9, 8, 130, 5, 3, 1, 2, 1),       # five window rows
    (4, 64, 15, 15, 256, 3, 3, 2, 2, 1),     # parts of the reduction that begin and end within a window row
    (3, 208, 9, 9, 129, 3, 3, 2, 2, 1),
    (1, 16, 3, 3, 129, 3, 3, 2, 2, 1),       # one image no larger than the window
]
POINTWISE = [      # tiles of 64 rows
    (1, 64, 9, 7, 130, 1, 1, 1, 1, 0),       # one odd image: the last group reads past the last pixel, and past x
    (3, 70, 6, 6, 96, 1, 1, 1, 1, 0),        # channels missing
    (2, 100, 14, 14, 65, 1, 1, 1, 1, 0),     # four of the last eight channels missing
    (5, 64, 2, 2, 72, 1, 1, 1, 1, 0),        # images of one group of pixels
    (1, 49, 1, 3, 70, 1, 1, 1, 1, 0),        # fewer pixels than a group
    (2, 720, 4, 4, 66, 1, 1, 1, 1, 0),       # 45 stages in parts of five
    (2, 720, 92, 92, 66, 1, 1, 1, 1, 0),     # 45 stages of few wavefronts: 64x64 tiles read a pixel a lane
]
LEVELS = [       # tiles of 128 rows cut by time: sums in two levels, the second begun within a part
    (32, 64, 28, 28, 128, 3, 3, 2, 2, 1),
    (6, 144, 92, 91, 272, 3, 3, 2, 2, 0),    # no padding, rows past the last channel
]


def test_the_long_reduction_of_few_wavefronts_is_one(lib):
    s = O.shape(*POINTWISE[-1])
    plan = lib.igemm_plan(cshape(s), 3)
    assert -(-(plan.Kred_pad // 16) // plan.split_k) > 40 and (plan.K_pad // 64) * -(-plan.Npix // 64) * plan.split_k < 1024


@pytest.mark.parametrize("shp,configs", [(s, (0, 2)) for s in WINDOWS + LEVELS] + [(s, (1, 3)) for s in POINTWISE])
def test_columns_against_fp64(lib, shp, configs):
    s = O.shape(*shp)
    x, w = O.make_inputs(s, seed=sum(shp))
    bias = O.rng_uniform(3, (s.K,))
    # magnitudes over 2^40, as a product's rounding must not depend on the scale of its row
    x = (x * np.exp2(np.arange(s.N * s.C) % 41 - 20).reshape(s.N, s.C, 1, 1)).astype(np.float32)
    # products and the sums of them, of the parts of a split reduction (at most 32) and of the bias
    tol = (s.C * s.kh * s.kw + 73) * EPS * (O.naive_conv_f64(s, np.abs(x), np.abs(w)) + np.abs(bias)[:, None, None]) + 1e-30
    truth = O.naive_conv_f64(s, x, w) + bias[:, None, None]
    for cfg in configs:
        print("columns", shp, cfg, flush=True)
        assert (np.abs(lib.implicit_gemm_conv(cshape(s), x, w, bias, False, config=cfg) - truth) <= tol).all(), cfg
        assert (np.abs(lib.implicit_gemm_conv(cshape(s), x, w, bias, True, config=cfg) - np.maximum(truth, 0.0)) <= tol).all(), cfg


@pytest.mark.parametrize("shp", WINDOWS)
def test_window_rows_give_the_bits_of_single_taps(lib, shp):
    """Tiles of 64 rows read a tap at a time and add up the same products in the same order, in as many parts."""
    s = O.shape(*shp)
    x, w = O.make_inputs(s, seed=sum(shp))
    parts = [lib.igemm_plan(cshape(s), cfg).split_k for cfg in range(4)]
    assert len(set(parts)) == 1
    print("window rows", shp, parts, flush=True)
    a, b, c, d = (lib.implicit_gemm_conv(cshape(s), x, w, config=cfg) for cfg in range(4))
    assert np.abs(a).max() > 0 and np.array_equal(a, b) and np.array_equal(c, d) and np.array_equal(a, c)


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3e38])
@pytest.mark.parametrize("shp,cfg", [(WINDOWS[0], 0), (WINDOWS[4], 2), (WINDOWS[5], 2), (LEVELS[0], 2), (LEVELS[1], 0), (POINTWISE[1], 1), (POINTWISE[2], 3)])
def test_only_values_that_are_not_finite_are_formed_again(lib, shp, cfg, value):
    s = O.shape(*shp)
    x, w = O.make_inputs(s, seed=11)
    bad = x.copy()
    bad[-1, s.C - 1, 4, 5] = value
    truth, size = O.naive_conv_f64(s, bad, w), O.naive_conv_f64(s, np.abs(bad), np.abs(w))
    hit = O.naive_conv_f64(s, (bad != x).astype(np.float32), np.ones_like(w)) > 0
    print("poison", shp, cfg, value, flush=True)
    clean, got = (lib.implicit_gemm_conv(cshape(s), v, w, config=cfg) for v in (x, bad))
    assert hit.any() and np.array_equal(got[~hit], clean[~hit])
    fin = hit & np.isfinite(truth) & np.isfinite(size)
    # products and the sums of them and of at most 32 parts
    assert (np.abs(got[fin] - truth[fin]) <= (s.C * s.kh * s.kw + 72) * EPS * size[fin]).all()
    odd = hit & ~fin
    assert np.array_equal(got[odd], truth[odd].astype(np.float32), equal_nan=True)


@pytest.mark.parametrize("shp", [(4, 64, 15, 15, 256, 3, 3, 2, 2, 1), (2, 208, 9, 9, 129, 3, 3, 2, 2, 1)])
def test_plans_in_other_parts_of_the_reduction_run_and_inconsistent_ones_do_not(lib, shp):
    """A plan kept by a program, of a library that chose another number of parts; the packed filter does not depend on it."""
    import fastconv_amd as F
    s = O.shape(*shp)
    x, w = O.make_inputs(s, seed=sum(shp))
    tol = (s.C * s.kh * s.kw + 73) * EPS * O.naive_conv_f64(s, np.abs(x), np.abs(w)) + 1e-30
    truth = O.naive_conv_f64(s, x, w)
    mark = lib.mark()
    try:
        for cfg in (0, 2, 3):
            plan = lib.igemm_plan(cshape(s), cfg)
            dx, dw, Wp, tab = lib.upload(x), lib.upload(w), lib.alloc(plan.Wp_bytes), lib.alloc(plan.table_bytes)
            y, one = lib.alloc(4 * s.N * s.K * plan.OH * plan.OW), 4 * s.K * plan.Npix
            ws = lib.alloc(32 * one)
            lib.igemm_pack_filter(plan, dw, Wp, tab)
            stages = plan.Kred_pad // 16
            for parts in range(1, 34):
                print("parts", shp, cfg, parts, flush=True)
                plan.split_k, plan.ws_bytes = parts, parts * one if parts > 1 else 0
                if parts <= stages // 4 and -(-stages // -(-stages // parts)) == parts:
                    lib.conv_implicit_gemm(plan, dx, Wp, tab, y, None, False, ws)
                    assert (np.abs(lib.download(y, (s.N, s.K, plan.OH, plan.OW)) - truth) <= tol).all(), (cfg, parts)
                else:
                    with pytest.raises(F.FastConvError):
                        lib.conv_implicit_gemm(plan, dx, Wp, tab, y, None, False, ws)
            for parts, nbytes in ((2, one), (2, 0), (1, one), (0, 0), (-1, 0)):
                plan.split_k, plan.ws_bytes = parts, nbytes
                with pytest.raises(F.FastConvError):
                    lib.conv_implicit_gemm(plan, dx, Wp, tab, y, None, False, ws)
    finally:
        lib.release(mark)


@pytest.mark.parametrize("shp,cfg,images", [
    ((32, 256, 28, 28, 256, 3, 3, 2, 2, 1), 2, 3), ((32, 128, 56, 56, 128, 3, 3, 2, 2, 1), 0, 2), ((3, 144, 92, 92, 528, 3, 3, 2, 2, 0), 0, 1),
    ((21, 256, 38, 38, 128, 5, 5, 2, 2, 2), 2, 4), ((12, 800, 10, 52, 128, 3, 3, 1, 1, 1), 0, 2), ((6, 144, 30, 30, 160, 3, 3, 2, 2, 1), 0, 4),
])
def test_a_reduction_in_fewer_parts_is_as_exact(lib, shp, cfg, images):
    """Parts chosen by time against those that fill the chip, whose sums are shorter: root mean square of the differences from 64 bits, over
    the first images."""
    from test_dispatch import parts_that_fill
    s = O.shape(*shp)
    x, w = O.make_inputs(s, seed=sum(shp))
    truth = O.naive_conv_f64(O.shape(images, *shp[1:]), x[:images], w)
    plan = lib.igemm_plan(cshape(s), cfg)
    fill = parts_that_fill(plan, ((128, 128), None, (128, 64))[cfg])
    assert plan.split_k < fill
    mark = lib.mark()
    try:
        dx, dw, Wp, tab = lib.upload(x), lib.upload(w), lib.alloc(plan.Wp_bytes), lib.alloc(plan.table_bytes)
        y, one, errors = lib.alloc(4 * s.K * plan.Npix), 4 * s.K * plan.Npix, []
        ws = lib.alloc(fill * one)
        lib.igemm_pack_filter(plan, dw, Wp, tab)
        for parts in (plan.split_k, fill):
            print("parts by time", shp, cfg, parts, flush=True)
            plan.split_k, plan.ws_bytes = parts, parts * one if parts > 1 else 0
            lib.conv_implicit_gemm(plan, dx, Wp, tab, y, None, False, ws)
            errors.append(np.sqrt(np.mean((lib.download(y, (s.N,) + truth.shape[1:])[:images] - truth) ** 2)))
    finally:
        lib.release(mark)
    # 100 000 values and more: each root mean square is known to about 1 / sqrt(2 * 100000), 0.3 %, of itself
    print("rms", errors, flush=True)
    assert truth.size >= 100000 and errors[0] <= 1.01 * errors[1], errors
