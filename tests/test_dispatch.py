"""Which Winograd pipeline the library advises (host code only): where the single-kernel path hands a layer to the
pipelines with V and M in memory, they accept it."""
import ctypes as C
import os
import subprocess
import sys

import pytest

from fastconv_amd import capi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib():
    return capi.load_cdll()


def shape(n, c, k, h, w=None):
    return capi.ConvShape(n, c, h, h if w is None else w, k, 3, 3, 1, 1, 1, 1, 1, 1)


@pytest.mark.parametrize("layer,onepass,fused", [
    ((32, 64, 64, 224), 1, 0), ((32, 64, 128, 112), 1, 0), ((32, 64, 256, 112), 1, 0),   # V and M far beyond the last-level cache
    ((32, 64, 64, 56), 0, 0), ((50, 64, 64, 63), 0, 0), ((20, 64, 64, 119), 1, 0),        # the line for fp32 instructions
    ((32, 64, 256, 56), 0, 0), ((6, 64, 1024, 110), 0, 0), ((14, 32, 512, 69), 0, 0), ((2, 24, 512, 202), 1, 0),
    ((23, 32, 256, 62), 0, 1), ((32, 16, 512, 112), 0, 1), ((32, 32, 128, 112), 1, 1),    # few channels in, many out
    ((1, 64, 64, 56), 0, 0), ((4, 24, 64, 112, 1200), 1, 1),                              # too few blocks; too wide for a plan
])
def test_single_kernel_line(lib, layer, onepass, fused):
    s = shape(*layer)
    assert lib.fc_wino_prefer_onepass(C.byref(s)) == onepass
    if not onepass:
        assert lib.fc_wino_prefer_fused(C.byref(s)) == fused


def test_layers_that_leave_the_single_kernel_path_have_a_plan(lib):
    plan, seen = capi.WinoPlan(), 0
    for c in (16, 17, 33, 48, 64):
        for k in (1, 64, 65, 200, 512, 1031):
            for n, h, w in ((1, 8, 1020), (1, 400, 1021), (3, 200, 5000), (64, 30, 31), (200, 223, 223), (4000, 7, 8)):
                s = shape(n, c, k, h, w)
                if not lib.fc_wino_prefer_onepass(C.byref(s)):
                    rc = lib.fc_wino_make_plan(C.byref(s), lib.fc_wino_gemm_default_config(C.byref(s)), C.byref(plan))
                    blocks = (n * ((h + 5) // 6) * ((w + 5) // 6) + 15) // 16 * ((k + 63) // 64)
                    assert rc == 0 or blocks < 512, (c, k, n, h, w)
                    seen += 1
    assert seen > 30


@pytest.mark.parametrize("k,onepass", [(65535, 0), (65536, 1), (70000, 1)])
def test_more_output_channels_than_the_staged_pipeline_takes_stay_on_the_single_kernel(lib, k, onepass):
    """The output transform of the staged pipeline refuses more than 65535 output channels; with as many the layer is
    otherwise one for the staged pipeline."""
    s = shape(1, 16, k, 12)
    assert lib.fc_prefer_winograd(C.byref(s)) == 1
    assert lib.fc_wino_prefer_onepass(C.byref(s)) == onepass
    assert onepass or not lib.fc_wino_prefer_fused(C.byref(s))


@pytest.mark.parametrize("layer,onepass", [
    ((17, 48, 32, 87), 1), ((9, 40, 24, 112), 1), ((10, 32, 32, 120), 1), ((32, 64, 64, 56), 1),      # staged is faster still
    ((32, 64, 256, 56), 0), ((6, 64, 1024, 110), 0), ((10, 48, 96, 100), 0), ((23, 32, 256, 62), 0),
    ((32, 64, 64, 224), 1), ((32, 64, 128, 112), 1), ((32, 3, 64, 224), 1), ((1, 64, 64, 56), 0),
])
def test_single_kernel_against_the_fused_pipeline_alone(lib, layer, onepass):
    """What the blocked layer class asks, which has no staged pipeline."""
    s = shape(*layer)
    assert lib.fc_wino_prefer_onepass_to_fused(C.byref(s)) == onepass
    assert onepass or not lib.fc_wino_prefer_onepass(C.byref(s))


@pytest.mark.parametrize("geo,bm", [
    ((32, 256, 56, 56, 256, 1, 1, 1, 0), 128), ((12, 85, 150, 150, 128, 3, 3, 1, 1), 128),
    ((39, 256, 230, 230, 256, 1, 1, 1, 0), 128), ((40, 256, 230, 230, 256, 1, 1, 1, 0), 64),      # 2 GiB of input between them
    ((64, 64, 400, 400, 256, 3, 3, 2, 1), 64),
])
def test_large_implicit_gemm_tiles_only_where_they_run_on_the_bf16_matrix_cores(lib, geo, bm):
    """128x128 tiles are ahead of 64x64 ones there, and behind on fp32 instructions, which inputs of 2 GiB run on."""
    n, c, h, w, k, kh, kw, st, p = geo
    s, g = capi.ConvShape(n, c, h, w, k, kh, kw, st, st, p, p, p, p), capi.GemmConfig()
    assert lib.fc_igemm_get_config(lib.fc_igemm_default_config(C.byref(s)), C.byref(g)) == 0
    assert (g.bm, g.bn, g.waves_k) == (bm, bm, 1)


@pytest.mark.parametrize("n,c,k,h,tile,split", [
    (1, 48, 200, 60, (128, 128), 0), (1, 49, 200, 60, (128, 128), 1), (1, 64, 128, 60, (128, 128), 0), (1, 64, 129, 60, (128, 128), 1),
    (38, 64, 130, 60, (128, 128), 1), (39, 64, 130, 60, (128, 128), 0), (40, 96, 130, 60, (128, 128), 1),      # V and M of 320 MB
    (1, 64, 130, 60, (64, 64), 0), (1, 65, 130, 60, (64, 64), 1), (36, 80, 130, 60, (64, 64), 1), (37, 80, 130, 60, (64, 64), 0),      # 256 MB
    (30, 144, 130, 60, (64, 64), 0), (30, 145, 130, 60, (64, 64), 1), (1, 176, 200, 60, (256, 128), 0), (1, 177, 200, 60, (256, 128), 1),
    (8, 512, 512, 28, (64, 32), 0),
])
def test_which_winograd_products_are_split(lib, n, c, k, h, tile, split):
    s, g, plan = shape(n, c, k, h), capi.GemmConfig(), capi.WinoPlan()
    for i in range(lib.fc_wino_gemm_num_configs()):
        assert lib.fc_wino_gemm_get_config(i, C.byref(g)) == 0
        if (g.bm, g.bn) != tile:
            continue
        assert lib.fc_wino_make_plan(C.byref(s), i, C.byref(plan)) == 0
        assert lib.fc_wino_gemm_splits_products(C.byref(plan)) == (split if g.bk == 16 else 0)
    assert lib.fc_wino_make_onepass_plan(C.byref(s), C.byref(plan)) == 0
    assert lib.fc_wino_gemm_splits_products(C.byref(plan)) == 0 and lib.fc_wino_gemm_splits_products(None) == 0


@pytest.mark.parametrize("geo,split", [
    ((32, 256, 56, 56, 256, 1, 1, 0), 1), ((32, 256, 56, 56, 64, 1, 1, 0), 0), ((32, 256, 56, 56, 64, 1, 2, 0), 1),
    ((1, 3, 32, 32, 64, 3, 1, 1), 0), ((1, 3, 32, 32, 64, 5, 1, 2), 1), ((1, 3, 32, 32, 64, 9, 1, 4), 0), ((1, 16, 32, 32, 64, 9, 1, 0), 1),
    ((40, 256, 230, 230, 256, 1, 1, 0), 0),
])
def test_which_implicit_gemm_products_are_split(lib, geo, split):
    n, c, h, w, k, ks, st, p = geo
    s, g, plan = capi.ConvShape(n, c, h, w, k, ks, ks, st, st, p, p, p, p), capi.GemmConfig(), capi.IgemmPlan()
    for i in range(lib.fc_igemm_num_configs()):
        assert lib.fc_igemm_get_config(i, C.byref(g)) == 0
        if lib.fc_igemm_make_plan(C.byref(s), i, C.byref(plan)) == 0:
            assert lib.fc_igemm_splits_products(C.byref(plan)) == (split if g.waves_k == 1 and g.bm % 64 == 0 else 0), i


@pytest.mark.parametrize("geo", [(1, 256, 56, 56, 256, 3, 1, 1), (32, 256, 28, 28, 256, 3, 2, 1), (4, 512, 28, 28, 100, 1, 1, 0), (8, 3, 61, 61, 700, 7, 2, 3)])
def test_plans_are_made_for_the_tile_that_runs(lib, geo):
    """256x128, 128x256 and 64x256 run as 128x128, 128x128 and 64x128 where products are split."""
    n, c, h, w, k, ks, st, p = geo
    s, a, b = capi.ConvShape(n, c, h, w, k, ks, ks, st, st, p, p, p, p), capi.IgemmPlan(), capi.IgemmPlan()
    for big, runs in ((5, 0), (6, 0), (7, 1)):
        assert lib.fc_igemm_make_plan(C.byref(s), big, C.byref(a)) == 0 and lib.fc_igemm_make_plan(C.byref(s), runs, C.byref(b)) == 0
        assert lib.fc_igemm_splits_products(C.byref(a)) == 1 and a.config == big
        assert (a.K_pad, a.Kred_pad, a.split_k, a.ws_bytes, a.Wp_bytes) == (b.K_pad, b.Kred_pad, b.split_k, b.ws_bytes, b.Wp_bytes), big
    whole = capi.ConvShape(n, 4, h, w, k, 3, 3, st, st, 1, 1, 1, 1)      # 36 rows: not split
    assert lib.fc_igemm_make_plan(C.byref(whole), 5, C.byref(a)) == 0 and a.K_pad % 256 == 0
    assert lib.fc_igemm_splits_products(C.byref(a)) == 0


@pytest.mark.parametrize("k", [65535, 65536, 70000, 100000])
def test_untuned_plans_of_very_many_channels_can_run(lib, k):
    """The sum over the parts of a split reduction takes 65535 output channels."""
    s, plan = capi.ConvShape(1, 4096, 4, 4, k, 1, 1, 1, 1, 0, 0, 0, 0), capi.IgemmPlan()
    assert lib.fc_igemm_make_plan(C.byref(s), lib.fc_igemm_default_config(C.byref(s)), C.byref(plan)) == 0
    assert plan.split_k == 1 or k <= 65535


@pytest.mark.parametrize("geo,parts,untuned", [
    ((32, 256, 28, 28, 256, 3, 2, 1), 4, (2, 5)), ((32, 128, 56, 56, 128, 3, 2, 1), 2, (0, 2)), ((32, 512, 14, 14, 512, 3, 2, 1), 9, (0, 9)),
])
def test_parts_of_a_reduction_put_the_large_tiles_on_the_chip_at_once(lib, geo, parts, untuned):
    """128x128 tiles, two a compute unit: at most 512 workgroups as launched, in whole eights of tiles, and more than half of that.  Left to
    the library the first layer runs in tiles of 128x64, four a compute unit, all on the chip at once too."""
    n, c, h, w, k, ks, st, p = geo
    s, plan = capi.ConvShape(n, c, h, w, k, ks, ks, st, st, p, p, p, p), capi.IgemmPlan()
    assert lib.fc_igemm_make_plan(C.byref(s), 0, C.byref(plan)) == 0
    tiles = (plan.K_pad // 128) * -(-plan.Npix // 128)
    assert plan.split_k == parts and 256 < -(-tiles // 8) * 8 * plan.split_k <= 512
    stages = plan.Kred_pad // 16
    assert -(-stages // -(-stages // parts)) == parts and plan.ws_bytes == 4 * parts * k * plan.Npix      # no part is empty
    assert lib.fc_igemm_make_plan(C.byref(s), lib.fc_igemm_default_config(C.byref(s)), C.byref(plan)) == 0
    assert (plan.config, plan.split_k) == untuned
    if untuned[0] == 2:
        tiles = (plan.K_pad // 128) * -(-plan.Npix // 64)
        assert 512 < -(-tiles // 8) * 8 * plan.split_k <= 1024


@pytest.mark.parametrize("geo", [
    (1, 16, 32, 32, 64, 32, 32, 1, 0), (1, 4, 8, 64, 64, 1, 33, 1, 0), (8, 16, 64, 64, 64, 33, 1, 2, 0), (1, 16, 64, 64, 64, 32, 1, 1, 16),      # windows of more than 31
    (1, 65536, 8, 8, 64, 64, 64, 1, 32),      # and a reduction past the longest
])
def test_untuned_choice_answers_for_layers_that_have_no_plan(geo):
    """fc_igemm_default_config is asked before a plan is made: the refusal is fc_igemm_make_plan's."""
    code = ("import ctypes as C; from fastconv_amd import capi; lib = capi.load_cdll(); n, c, h, w, k, kh, kw, st, p = %r; "
            "s = capi.ConvShape(n, c, h, w, k, kh, kw, st, st, p, p, p, p); d = lib.fc_igemm_default_config(C.byref(s)); "
            "assert 0 <= d < lib.fc_igemm_num_configs(); assert lib.fc_igemm_make_plan(C.byref(s), d, C.byref(capi.IgemmPlan())) == -6") % (geo,)
    assert subprocess.run([sys.executable, "-c", code], cwd=ROOT).returncode == 0


def parts_that_fill(plan, tile):
    """About three workgroups a compute unit, six where the reduction is long, of at least four stages; no empty part."""
    stages, blocks = plan.Kred_pad // 16, (plan.K_pad // tile[0]) * -(-plan.Npix // tile[1])
    below, target = (1024, 1536) if stages >= 64 else (512, 768)
    parts = max(1, min(-(-target // blocks), stages // 4, 32)) if blocks < below else 1
    return -(-stages // -(-stages // parts))


@pytest.mark.parametrize("geo", [
    (5, 176, 136, 136, 336, 5, 2, 2), (6, 240, 154, 154, 64, 5, 1, 2), (8, 64, 16, 35, 736, 7, 1, 3), (32, 864, 44, 44, 752, 7, 2, 3),
    (7, 432, 207, 207, 48, 3, 2, 1), (8, 464, 153, 153, 16, 5, 1, 2), (32, 256, 28, 28, 256, 3, 2, 1), (6, 389, 143, 109, 114, 7, 2, 3),
    (8, 512, 28, 28, 512, 3, 1, 1), (32, 128, 28, 28, 512, 1, 1, 0), (43, 768, 18, 18, 112, 5, 2, 2), (3, 144, 92, 92, 528, 3, 2, 1),
])
def test_no_reduction_is_cut_into_more_parts_than_fill_the_chip(lib, geo):
    """A caller with room for the partial sums of the parts that fill the chip has it for the plan; the static workspace takes the same plans."""
    n, c, h, w, k, ks, st, p = geo
    s, plan = capi.ConvShape(n, c, h, w, k, ks, ks, st, st, p, p, p, p), capi.IgemmPlan()
    for i, tile in enumerate([(128, 128), (64, 128), (128, 64), (64, 64), None, (128, 128), (128, 128), (64, 128)]):
        if tile and lib.fc_igemm_make_plan(C.byref(s), i, C.byref(plan)) == 0:
            fill = parts_that_fill(plan, tile)
            assert 1 <= plan.split_k <= fill and plan.ws_bytes == (4 * plan.split_k * k * plan.Npix if plan.split_k > 1 else 0), i


@pytest.mark.parametrize("geo,ws_mb,static", [
    # partial sums of the untuned plan in MiB at most; tiles whose plans fit the static workspace of 32 MiB or are the untuned ones
    ((6, 240, 154, 154, 64, 5, 1, 2), 0, (0, 1, 2, 3, 5, 6, 7)), ((5, 176, 136, 136, 336, 5, 2, 2), 89, (1, 2, 3, 7)),
    ((32, 864, 44, 44, 752, 7, 2, 3), 134, (1, 2, 3, 7)), ((7, 432, 207, 207, 48, 3, 2, 1), 42, (2, 3)), ((8, 64, 16, 35, 736, 7, 1, 3), 51, (2,)),
    ((6, 389, 143, 109, 114, 7, 2, 3), 93, (0,)),
])
def test_plans_that_the_static_workspace_takes(lib, geo, ws_mb, static):
    n, c, h, w, k, ks, st, p = geo
    s, plan = capi.ConvShape(n, c, h, w, k, ks, ks, st, st, p, p, p, p), capi.IgemmPlan()
    untuned = lib.fc_igemm_default_config(C.byref(s))
    for i in (untuned,) + static:
        assert lib.fc_igemm_make_plan(C.byref(s), i, C.byref(plan)) == 0
        assert plan.ws_bytes <= capi.IGEMM_STATIC_WS_BYTES or i == untuned, i
        assert i != untuned or plan.ws_bytes <= ws_mb << 20


@pytest.mark.parametrize("geo,kernel,bf16,split", [      # untuned plans
    ((32, 3, 224, 224, 64, 3, 1, 1), "igemm_short_kernel", 1, 0), ((16, 18, 99, 99, 100, 1, 1, 0), "igemm_short_kernel", 1, 0),
    ((3, 1, 223, 222, 200, 7, 2, 3), "igemm_short_kernel", 1, 1), ((32, 256, 56, 56, 64, 1, 1, 0), "igemm_split_kernel", 1, 0),
    ((32, 256, 56, 56, 256, 1, 1, 0), "igemm_split_kernel", 1, 1), ((32, 256, 28, 28, 256, 3, 2, 1), "igemm_split_kernel", 1, 1),
    ((16, 256, 56, 56, 64, 1, 1, 0), "igemm_conv_kernel", 0, 0), ((1, 256, 56, 56, 256, 3, 2, 1), "igemm_wavesplit_kernel", 0, 0),
])
def test_the_library_says_which_kernel_runs_a_plan_and_on_which_matrix_cores(lib, geo, kernel, bf16, split):
    """What a rate is a fraction of: layers whose filter is split in the kernel run on the bf16 matrix cores too."""
    n, c, h, w, k, ks, st, p = geo
    s, plan = capi.ConvShape(n, c, h, w, k, ks, ks, st, st, p, p, p, p), capi.IgemmPlan()
    assert lib.fc_igemm_make_plan(C.byref(s), lib.fc_igemm_default_config(C.byref(s)), C.byref(plan)) == 0
    assert lib.fc_igemm_kernel_name(C.byref(plan)).decode() == kernel
    assert (lib.fc_igemm_on_bf16(C.byref(plan)), lib.fc_igemm_splits_products(C.byref(plan))) == (bf16, split)
    assert lib.fc_igemm_on_bf16(None) == 0 and lib.fc_igemm_kernel_name(None) == b""
    plan.config = lib.fc_igemm_num_configs()
    assert lib.fc_igemm_on_bf16(C.byref(plan)) == 0 and lib.fc_igemm_kernel_name(C.byref(plan)) == b""


@pytest.mark.parametrize("geo", [(32, 3, 224, 224, 64, 3, 1, 1), (16, 18, 99, 99, 100, 1, 1, 0), (3, 1, 223, 222, 200, 7, 2, 3), (32, 256, 56, 56, 64, 1, 1, 0),
                                 (6, 512, 128, 128, 64, 1, 1, 0)])
def test_a_configuration_that_is_not_the_untuned_one_runs_its_own_tile(lib, geo):
    """Tuning compares tiles: only the untuned plan of such layers goes to the kernels of short reductions and few output channels."""
    n, c, h, w, k, ks, st, p = geo
    s, plan = capi.ConvShape(n, c, h, w, k, ks, ks, st, st, p, p, p, p), capi.IgemmPlan()
    untuned = lib.fc_igemm_default_config(C.byref(s))
    for i in range(8):
        assert lib.fc_igemm_make_plan(C.byref(s), i, C.byref(plan)) == 0
        name, split = lib.fc_igemm_kernel_name(C.byref(plan)).decode(), lib.fc_igemm_splits_products(C.byref(plan))
        if i == untuned:
            assert name == "igemm_short_kernel" or (name == "igemm_split_kernel" and not split)
        else:
            assert name == ("igemm_split_kernel" if split else "igemm_conv_kernel"), i


def test_no_kernel_is_compiled_that_nothing_launches():
    """Tile and mode of igemm_split_kernel, stages and mode of igemm_short_kernel, as their names are mangled (modes: 2
    channels missing, 4 runs of four columns, 5 16-byte pointwise columns, 7 12-byte window rows)."""
    built = open(capi.LIB_PATH, "rb").read()
    for rows, cols, waves in ((64, 64, 2), (64, 128, 4), (128, 64, 2), (128, 128, 4)):
        tile = b"IgSplitILi%dELi%dELi%dEEELi" % (rows, cols, waves)
        assert tile + b"2E" in built
        assert (tile + b"5E" in built) == (rows == 64) and (tile + b"7E" in built) == (rows == 128)
    assert b"igemm_short_kernelILi4ELi4E" in built and b"igemm_short_kernelILi3ELi5E" in built
    assert b"igemm_short_kernelILi4ELi5E" not in built and b"igemm_short_kernelILi4ELi2E" not in built
