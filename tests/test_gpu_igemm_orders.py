"""Implicit GEMM on the bf16 matrix cores: every order of the reduction (blocks of channels whole, padded and inside the
image, window rows in runs of 8 and of 4), part-filled tiles, windows that start before the input, split reductions."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_split_products import bound, cshape, lib  # noqa: F401

pytestmark = pytest.mark.gpu

SHAPES = [
    O.shape(3, 16, 7, 9, 32, 3, 3, 1, 1, 1),            # one block of channels, 32 rows of a 64-row tile
    O.shape(1, 48, 12, 13, 97, 3, 3, 2, 2, 1),          # strided, half of the last rows
    O.shape(1, 16, 9, 9, 64, 9, 9, 1, 1, 0),            # 81 taps inside the image, one pixel
    O.shape(1, 64, 15, 15, 65, 1, 1, 2, 2, 0),          # 1x1, stride 2
    O.shape(2, 65, 6, 6, 64, 1, 1, 1, 1, 0),            # one channel past a block
    O.shape(2, 29, 10, 11, 96, 3, 3, 1, 1, 1),          # padded channels with taps outside the image
    O.shape(1, 300, 6, 6, 70, 3, 3, 1, 1, 1),           # split reduction, padded channels
    O.shape(1, 17, 9, 8, 64, 3, 3, 1, 1, 1),            # runs of 4
    O.shape(2, 7, 12, 9, 160, 3, 3, 2, 2, 1),           # runs of 4, strided
    O.shape(1, 90, 7, 7, 64, 3, 2, 1, 1, 1),            # runs of 4 half filled
    O.shape(1, 5, 13, 12, 33, 5, 5, 2, 2, 2),           # runs of 8
    O.shape(2, 3, 17, 16, 20, 7, 7, 2, 2, 3),           # runs of 8, 32 rows of a tile, windows before the input
    O.shape(1, 1, 40, 31, 64, 7, 7, 1, 1, 3),           # one channel: every stage has such windows
    O.shape(1, 6, 9, 41, 64, 3, 11, 1, 1, 1),           # two runs a window row
    O.shape(2, 3, 19, 70, 64, 2, 31, 1, 1, 0),          # four runs, the widest window
    O.Shape(2, 20, 9, 9, 64, 3, 3, 1, 1, 0, 2, 2, 0),   # padding on two sides only
    # images smaller than the left padding: windows start before the input in more channels than the first
    O.Shape(2, 5, 1, 4, 64, 1, 15, 1, 1, 0, 0, 7, 7),   # two channels, two runs a window row
    O.shape(2, 3, 1, 2, 64, 7, 7, 1, 1, 3),
    O.shape(3, 3, 1, 1, 64, 5, 5, 1, 1, 2),
    O.shape(2, 8, 1, 3, 64, 5, 5, 1, 1, 4),
    O.shape(1, 20, 1, 1, 64, 5, 5, 1, 1, 4),            # four of twenty channels, split reduction
    O.shape(2, 2, 1, 1, 33, 7, 7, 1, 1, 6),             # all channels
    O.Shape(2, 70, 1, 2, 64, 2, 4, 1, 1, 1, 1, 3, 3),   # runs of 4
    # tiles of which some wavefronts hold such windows and others none
    O.shape(1, 3, 9, 100, 64, 5, 5, 1, 1, 2),
    O.shape(3, 3, 5, 70, 128, 7, 7, 1, 1, 3),
    O.shape(1, 40, 1, 140, 64, 1, 7, 1, 1, 0, pl=150, pr=3),      # more than one image row before x, split reduction
]


@pytest.mark.parametrize("s", SHAPES, ids=lambda s: "-".join(str(getattr(s, n)) for n, _ in type(s)._fields_))
def test_orders_of_the_reduction(lib, s):  # noqa: F811
    x, w = O.make_inputs(s, seed=s.C + s.K)
    bias = O.rng_uniform(3, (s.K,))
    truth, tol = O.naive_conv_f64(s, x, w), bound(s, x, w)
    with_bias = np.maximum(truth + bias[None, :, None, None], 0.0)
    seen = 0
    for cfg in lib.igemm_configs():
        if cfg.waves_k > 1 or not lib.igemm_splits_products(lib.igemm_plan(cshape(s), cfg.id)):
            continue
        print("order", [getattr(s, n) for n, _ in type(s)._fields_], cfg.bm, cfg.bn, flush=True)
        assert (np.abs(lib.implicit_gemm_conv(cshape(s), x, w, config=cfg.id) - truth) <= tol).all(), cfg.id
        got = lib.implicit_gemm_conv(cshape(s), x, w, bias, True, config=cfg.id)
        assert (np.abs(got - with_bias) <= tol + 2.0 ** -23 * (np.abs(truth) + 1)).all(), cfg.id
        seen += 1
    assert seen


@pytest.mark.parametrize("c", [29120, 29125])
def test_longest_reductions(lib, c):  # noqa: F811
    """262125 rows of the filter, 262224 of the packed one; 29120 channels need no padding."""
    s = O.shape(1, c, 3, 3, 33, 3, 3, 1, 1, 0)
    x, w = O.make_inputs(s, seed=c)
    truth, tol = O.naive_conv_f64(s, x, w), bound(s, x, w)
    for cfg in (3, 4):
        print("longest", c, cfg, flush=True)
        assert (np.abs(lib.implicit_gemm_conv(cshape(s), x, w, config=cfg) - truth) <= tol).all()
