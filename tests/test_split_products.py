"""The arithmetic of csrc/split_mfma.h on the CPU: three bf16 parts add up to a float, six of their nine products give a
single term to fp32 accuracy, and the bound that the GPU test holds the kernels to is broken by any other choice."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_split_products import EPS_SINGLE

HI, MID, LO = 0, 1, 2
PRODUCTS = ((LO, HI), (MID, MID), (HI, LO), (MID, HI), (HI, MID), (HI, HI))      # smallest first, as the kernels add them


def bf16(x, cut=False):
    """float32 rounded to nearest bf16, or cut off."""
    u = x.view(np.uint32)
    return ((u if cut else u + 0x7fff + ((u >> 16) & 1)) & np.uint32(0xffff0000)).view(np.float32)


def parts(x, cut=False):
    hi = bf16(x, cut)
    mid = bf16(x - hi)
    return hi, mid, bf16(x - hi - mid)


def single_term_error(products, cut=False):
    """Largest relative error of a * b over many operands, each product added in fp32."""
    a, b = O.rng_uniform(1, (200000,)), O.rng_uniform(2, (200000,))
    pa, pb = parts(a, cut), parts(b, cut)
    total = np.zeros_like(a)
    for i, j in products:
        total = (total.astype(np.float64) + pa[i].astype(np.float64) * pb[j]).astype(np.float32)
    exact = a.astype(np.float64) * b
    ok = exact != 0
    return (np.abs(total - exact)[ok] / np.abs(exact)[ok]).max()


def test_three_parts_are_the_float():
    x = O.rng_uniform(3, (100000,)) * np.exp2(np.arange(100000) % 180 - 80).astype(np.float32)
    hi, mid, lo = parts(x)
    assert np.array_equal(hi.astype(np.float64) + mid + lo, x)


def test_six_products_keep_the_bound():
    assert single_term_error(PRODUCTS) <= EPS_SINGLE


@pytest.mark.parametrize("left_out", PRODUCTS)
def test_five_products_break_it(left_out):
    assert single_term_error([p for p in PRODUCTS if p != left_out]) > EPS_SINGLE


def test_a_first_part_that_is_cut_off_breaks_it():
    assert single_term_error(PRODUCTS, cut=True) > EPS_SINGLE
