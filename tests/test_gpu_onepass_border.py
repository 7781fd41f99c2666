"""Patch rows of the single-kernel Winograd path beside the image border: they are read past the image row and masked, or,
at the ends of the tensor, clamped to the row and shifted.  And rows of y, stored six floats at a time wherever they start."""
import numpy as np
import pytest

import fastconv_amd as F
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL_WINO = 1e-3      # of every Winograd path against 64 bits, as elsewhere in these tests

SHAPES = [
    ((1, 5, 20, 20, 7), {}),                          # both ends of the tensor in one image
    ((2, 16, 14, 26, 70), {}),                        # last column of tiles 2 wide
    ((3, 17, 13, 31, 20), {}),                        # a channel alone in the last chunk
    ((1, 6, 9, 8, 3), {"pl": 2, "pr": 2}),            # the smallest width
    ((2, 5, 8, 9, 4), {"pt": 2, "pb": 2, "pl": 2, "pr": 0}),
    ((2, 7, 12, 12, 5), {"pt": 9, "pb": 9, "pl": 9, "pr": 9}),      # whole tiles in the padding
    ((2, 6, 13, 13, 65), {}), ((1, 8, 12, 15, 33), {}), ((1, 5, 9, 11, 3), {"pr": 2}),      # rows of 13, 15 and 12 floats
    ((1, 16, 12, 18, 64), {"pt": 0, "pb": 0, "pl": 0, "pr": 0}),    # no border inside a patch but in the ragged tiles
]


@pytest.fixture(scope="module")
def lib():
    L = F.load(0, 1 << 30)
    yield L
    L.close()


def cshape(s):
    return F.ConvShape(*[getattr(s, n) for n, _ in F.ConvShape._fields_])


@pytest.mark.parametrize("shp,pads", SHAPES)
def test_border_rows_against_oracle(lib, shp, pads):
    s = O.shape(*shp, **pads)
    x, w = O.make_inputs(s, seed=shp[1])
    print("border rows", shp, pads, flush=True)
    assert O.max_rel_err(lib.winograd_conv_onepass(cshape(s), x, w), O.naive_conv_f64(s, x, w)) <= TOL_WINO


@pytest.mark.parametrize("shp,pads", SHAPES)
def test_what_lies_beyond_the_border_is_dropped(lib, shp, pads):
    """Infinities in the first and last column: tiles whose patch does not hold one keep their bits, though the rows of
    their patches are read across the border into the row that does."""
    s = O.shape(*shp, **pads)
    x, w = O.make_inputs(s, seed=shp[1])
    clean = lib.winograd_conv_onepass(cshape(s), x, w)
    for row, col in ((s.H // 2, 0), (s.H // 2, s.W - 1), (s.H - 1, s.W - 1), (0, 0)):
        bad = x.copy()
        bad[:, 1, row, col] = np.inf
        print("beyond the border", shp, pads, row, col, flush=True)
        y = lib.winograd_conv_onepass(cshape(s), bad, w)
        keep = np.ones(y.shape, bool)
        for th in range((y.shape[2] + 5) // 6):
            for tw in range((y.shape[3] + 5) // 6):
                if 0 <= row + s.pt - 6 * th < 8 and 0 <= col + s.pl - 6 * tw < 8:
                    keep[:, :, 6 * th:6 * th + 6, 6 * tw:6 * tw + 6] = False
        assert keep.any() or y.shape[3] <= 12
        assert np.array_equal(y[keep], clean[keep])


@pytest.mark.parametrize("shp,pads", SHAPES)
def test_rows_of_the_fused_kernel_are_those_of_the_staged_pipeline(lib, shp, pads):
    s = O.shape(*shp, **pads)
    x, w = O.make_inputs(s, seed=shp[1])
    print("fused rows", shp, pads, flush=True)
    assert np.array_equal(lib.winograd_conv_fused(cshape(s), x, w), lib.winograd_conv(cshape(s), x, w))


@pytest.mark.parametrize("shp", [(1, 3, 13, 13, 65), (2, 1, 12, 15, 16), (1, 4, 9, 11, 17), (3, 2, 14, 9, 5), (1, 2, 8, 67, 33)])
def test_odd_rows_of_the_small_channel_kernel(lib, shp):
    """Whole tiles six floats a row, ragged ones a float at a time."""
    s = O.shape(*shp)
    x, w = O.make_inputs(s, seed=shp[1])
    bias = O.rng_uniform(3, (s.K,))
    print("odd rows", shp, flush=True)
    y = lib.winograd_conv_onepass(cshape(s), x, w, bias=bias, relu=True)
    assert O.max_rel_err(y, np.maximum(O.naive_conv_f64(s, x, w, bias), 0.0)) <= TOL_WINO
