"""Which products and convolution passes the host gives to the ring kernels, and on which of their tiles (CPU only): the
layers and products that the GPU tests run reach every tile, on a chip of 256 CUs."""
import ctypes as ct
import os
import subprocess

import pytest

import test_gpu_conv as conv
import test_gpu_deferred as deferred
import test_gpu_dot as dot
from oracle import conv_oracle as co

HERE = os.path.dirname(os.path.abspath(__file__))
CUS = 256
UP, DOWN, OUTP = 0, 1, 2
TILES = [(64, 64), (64, 32), (32, 64), (32, 32), (32, 16), (16, 32)]


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("plans") / "ring_plans.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", os.path.join(HERE, "ring_plans.cpp"), "-o", lib],
                   check=True)
    return ct.CDLL(lib)


def gemm_tile(plans, m, n, k, vec=False):
    """Tile of a product; None: another kernel.  vec: of operands that the other kernels read in 16-byte groups."""
    t = plans.gemm_tile(m, n, k, CUS, vec)
    return TILES[t] if t >= 0 else None


def conv_tile(plans, mode, N, C, H, F, k, s, p, G=1, local=False, partial_sum=0):
    """(tile, whether it lies in one module or pixel, splits, LDS bytes, us) of a pass; None: another kernel."""
    out = (ct.c_double * 5)()
    plans.conv_tile(mode, N, C, H, F, k, co.n_modules(H, k, s, p), s, -p, G, int(local), 1 if local and mode == OUTP else partial_sum, CUS, out)
    return (TILES[int(out[0])], bool(out[1]), out[2], out[3], out[4]) if out[0] >= 0 else None


def test_the_products_of_the_gpu_tests_reach_every_tile(plans):
    got = [gemm_tile(plans, *shape) for shape in dot.RING_SHAPES]
    assert None not in got
    for tile in TILES:
        edges = [(m % tile[0] != 0) + (n % tile[1] != 0) for (m, n, k), t in zip(dot.RING_SHAPES, got) if t == tile]
        assert edges and max(edges) == 2, tile           # one of them hangs over both edges


def test_the_products_of_the_other_kernels_are_not_on_ring_tiles(plans):
    assert [shape for shape in dot.OTHER_SHAPES if gemm_tile(plans, *shape)] == []
    assert [shape for shape in dot.VEC_SHAPES if gemm_tile(plans, *shape, vec=True) or not gemm_tile(plans, *shape)] == []
    assert [shape for shape in dot.RING_SHAPES if gemm_tile(plans, *shape, vec=True) != gemm_tile(plans, *shape)] == []
    slabs = {64: dot.SLAB64_SHAPES, 128: dot.SLAB128_SHAPES}
    assert {side: {plans.gemm_slab(*shape, CUS, vec) for shape in shapes for vec in (0, 1)} for side, shapes in slabs.items()} == {64: {64}, 128: {128}}
    assert [shape for shape in dot.OTHER_SHAPES + dot.VEC_SHAPES + dot.RING_SHAPES for vec in (0, 1) if plans.gemm_split(*shape, CUS, vec)] == []


def test_the_split_products_of_the_gpu_tests_are_k_gemm_split_s(plans):
    assert [shape for shape in dot.SPLIT_SHAPES + [(1409, 1537, 705)] for vec in (0, 1) if not plans.gemm_split(*shape, CUS, vec)] == []
    assert [s for s in deferred.SHAPES if plans.gemm_split(s[0], s[2], s[1], CUS, 0)] == deferred.SHAPES[-1:]
    # tiles have to lie inside the product, and offsets in 31 bits
    assert [shape for shape in ((127, 30000, 4000), (30000, 127, 4000), (65536, 256, 8192), (256, 65536, 8192), (4096, 4096, 199))
            if plans.gemm_split(*shape, CUS, 0)] == []


@pytest.mark.parametrize("cus", [16, 32, 64, 128, 256, 304])
def test_products_that_may_draw_a_sample_do_not_change_their_kernel_for_it(plans, cus):
    """k_gemm_split draws no samples: it takes no product that is small enough for one, however few CUs there are."""
    limit = 16 * 96 * 128
    sides = [(128, n) for n in (128, 700, 1536)] + [(m, limit // m) for m in (129, 200, 298, 384, 435, 443)]
    shapes = [s + (k,) for m, n in sides for s in ((m, n), (n, m)) for k in (200, 640, 2008, 5000)]
    assert [s for s in shapes for vec in (0, 1) if plans.gemm_split(*s, cus, vec)] == []
    assert cus > 32 or plans.gemm_split(444, 444, 2008, cus, 0)                  # 197136 outputs


def test_the_layers_of_the_gpu_tests_reach_every_tile(plans):
    reached = set()
    for mode in (UP, DOWN, OUTP):
        for layer in conv.CASES + conv.RING_LAYERS:
            t = conv_tile(plans, mode, *layer)
            if t:
                reached.add((mode, t[1], t[0]))
    want = {(mode, single, tile) for mode in (UP, DOWN, OUTP) for single in (False, True) for tile in TILES if not (mode == OUTP and single)}
    assert reached == want, sorted(want - reached)


def test_the_layers_of_the_gpu_tests_reach_every_tile_of_the_bf16_matrix_cores(plans):
    def tile(mode, N, C, H, F, k, s, p, G=1, local=False):
        out = (ct.c_double * 5)()
        partial = 1 if local and mode == OUTP else 0
        plans.conv_tile(4 + mode, N, C, H, F, k, co.n_modules(H, k, s, p), s, -p, G, int(local), partial, CUS, out)
        assert out[0] < 6 or out[3] <= 160 << 10                     # (tile and table are a workgroup's LDS)
        return (mode, bool(out[1]), int(out[0])) if out[0] >= 6 else None

    modes = (UP, DOWN, OUTP)
    reached = {tile(mode, *layer) for mode in modes for layer in conv.SPLIT_LAYERS} - {None}
    want = {(mode, single, t) for mode in (UP, DOWN) for single in (False, True) for t in range(6, 11)} - {(UP, False, 10), (UP, True, 10)}
    assert reached == want | {(OUTP, False, t) for t in range(6, 9)}, sorted(want - reached)
    local = [{tile(mode, *layer, local=True) for mode in modes} - {None} for layer in conv.SPLIT_LOCAL]
    assert all(local) and (OUTP, False, 9) in set.union(*local)
    number = dict(up=UP, down=DOWN, outp=OUTP)
    odd = {tile(number[mode], *layer) for mode, layer in conv.NOT_FINITE} | {tile(number[mode], *layer, local=True) for mode, layer in conv.NOT_FINITE_LOCAL}
    assert odd == reached | {(OUTP, False, 9)}
    assert [layer for mode, layer in conv.FEW_SMALL_TILES if tile(number[mode], *layer)] == []
    assert [tile(number[mode], *layer, local=True) for mode, layer in conv.FEW_SMALL_TILES_LOCAL] == [None, None, (OUTP, False, 8)]
    moved = [layer for layer, passes in conv.OTHER_LAYERS.items() if any(tile(number[n], *layer) for n in passes.split())]
    assert moved == [(128, 16, 48, 208, 4, 4, 0, 1)]


def test_a_workgroup_that_is_alone_on_its_cu_costs_more(plans):
    """convUp on 32 x 16 tiles: with 24 stages of table two workgroups fit the 160 KB of a CU, with 25 one."""
    two, one = (conv_tile(plans, UP, 100, colors, 24, 16, 5, 1, 0) for colors in (122, 126))
    assert two[0] == one[0] == (32, 16) and two[3] <= 80 << 10 < one[3]
    assert one[4] > 1.15 * two[4]


def test_layers_are_planned_as_their_comments_say(plans):
    t = conv_tile(plans, OUTP, 128, 40, 13, 188, 7, 2, 0)
    assert t[2] == 1
    t = conv_tile(plans, OUTP, 100, 1, 34, 32, 7, 2, 0)
    assert t[2] > 40
    for layer in conv.RING_LOCAL:
        assert any(conv_tile(plans, mode, *layer, local=True) for mode in (UP, DOWN, OUTP))


@pytest.mark.parametrize("m,n,k", [(5899, 21, 312), (23, 4407, 250), (4585, 22, 381), (28, 4655, 180), (6641, 17, 198), (31, 8192, 139)])
def test_strips_that_a_16_wide_tile_halves_stay_on_32_wide_blocks(plans, m, n, k):
    assert gemm_tile(plans, m, n, k) is None
    assert gemm_tile(plans, m + 16 if m < 32 else m, n + 16 if n < 32 else n, k) is not None
    assert gemm_tile(plans, m, n, 4 * k + 400) is not None


@pytest.mark.parametrize("mode,layer", [(OUTP, (160, 1, 97, 48, 7, 2, 0)), (OUTP, (128, 1, 38, 48, 7, 1, 0)), (DOWN, (100, 16, 30, 208, 7, 1, 0)),
                                        (DOWN, (80, 16, 19, 172, 5, 1, 0)), (UP, (100, 3, 64, 48, 7, 1, 0)),
                                        (UP, (100, 3, 161, 48, 7, 2, 0)), (UP, (128, 4, 38, 48, 3, 1, 0, 2)), (UP, (100, 1, 90, 32, 7, 1, 3)), (UP, (234, 1, 79, 40, 7, 1, 3))])
def test_layers_of_few_colours_that_other_kernels_are_faster_on(plans, mode, layer):
    assert conv_tile(plans, mode, *layer) is None


@pytest.mark.parametrize("layer", [(160, 78, 24, 32, 3, 1, 1), (256, 200, 25, 32, 3, 1, 1, 2), (128, 90, 30, 32, 3, 1, 1),
                                   (256, 156, 15, 32, 3, 1, 0, 2), (128, 96, 32, 48, 3, 1, 1), (32, 96, 62, 64, 3, 1, 1)])
def test_gradients_of_many_colours_from_few_filters_that_slab_tiles_are_faster_on(plans, layer):
    assert conv_tile(plans, DOWN, *layer) is None
    assert conv_tile(plans, DOWN, 48 if layer[0] > 48 else 8, *layer[1:]) is not None          # fewer images: fewer tiles than two per CU


@pytest.mark.parametrize("mode,layer", [(DOWN, (100, 16, 28, 208, 7, 1, 3)), (DOWN, (117, 16, 25, 64, 7, 1, 3)), (DOWN, (202, 16, 8, 224, 5, 1, 0)),
                                        (UP, (100, 3, 74, 64, 5, 1, 0)), (UP, (100, 1, 54, 32, 7, 2, 0))])
def test_layers_of_few_colours_that_ring_tiles_are_faster_on(plans, mode, layer):
    assert conv_tile(plans, mode, *layer) is not None


def test_the_layers_of_the_other_kernels_are_not_on_ring_tiles(plans):
    """Most layers of the tests are small, and small layers go to ring tiles: these are there for the other kernels."""
    for layers, local in ((conv.OTHER_LAYERS, False), (conv.OTHER_LOCAL, True)):
        for layer, passes in layers.items():
            for name in passes.split():
                assert conv_tile(plans, dict(up=UP, down=DOWN, outp=OUTP)[name], *layer, local=local) is None, (layer, name)


def test_aligned_operands_take_the_ring_for_long_reductions_only(plans):
    for m, n, k in ((16384, 147, 160), (128, 18880, 240), (10368, 196, 400), (18432, 49, 208), (1648, 96, 224)):
        assert gemm_tile(plans, m, n, k, vec=True) is None
    for m, n, k in ((16384, 147, 416), (8192, 256, 400), (18432, 49, 272), (7000, 49, 208), (1648, 96, 160), (1648, 96, 272)):
        assert gemm_tile(plans, m, n, k, vec=True) is not None


def test_strips_of_one_or_two_tiles_per_cu(plans):
    for m, n, k in ((12800, 18, 288), (24200, 25, 144), (27, 15300, 160), (23636, 81, 243), (80, 17144, 135)):
        assert gemm_tile(plans, m, n, k) is None
    for m, n, k in ((20000, 25, 256), (27, 15300, 416), (23636, 81, 272), (23636, 92, 243)):
        assert gemm_tile(plans, m, n, k) is not None


def test_long_strips_of_33_to_63_are_not_on_ring_tiles(plans):
    for m, n, k in ((57, 25160, 149), (44, 38103, 167), (26761, 44, 168)):
        assert gemm_tile(plans, m, n, k) is None
    for m, n, k in ((19399, 49, 252), (57, 17393, 163), (26761, 64, 168), (32, 26761, 168)):
        assert gemm_tile(plans, m, n, k) is not None


def pixels_tile(plans, N, C, H, F, k, s, p, G=1):
    out = (ct.c_double * 4)()
    plans.conv_pixels_tile(N, C, H, F, k, co.n_modules(H, k, s, p), s, -p, G, CUS, out)
    return tuple(int(v) for v in out) if out[0] >= 0 else None


def test_gradients_of_the_gpu_tests_reach_every_kind_of_pixel_tile(plans):
    got = [pixels_tile(plans, *layer) for layer in conv.PIXEL_LAYERS]
    assert None not in got and {t[1] for t in got} == {-1, 0, 1, 2, 4}
    assert {t[0] >= 6 for t in got if t[1] == -1} == {t[0] >= 6 for t in got if t[1] > 0} == {False, True}
    odd = {t[0] for layer, t in zip(conv.PIXEL_LAYERS, got) if t[1] == -1 and layer[3] // layer[7] % 4}
    assert {0, 1, 3, 4, 7, 10} <= odd                    # (an instance of its own)
    for tile, blocks, stages, lds in got:
        assert lds <= 160 << 10 and stages >= 1
    assert [layer for layer in conv.PIXEL_LAYERS if conv_tile(plans, DOWN, *layer)] == []
    for layer in conv.SIXTEEN:
        assert pixels_tile(plans, *layer) is None and conv_tile(plans, DOWN, *layer) is None


def test_tables_of_pixel_tiles_fit(plans):
    import random
    rng, taken = random.Random(5), 0
    for _ in range(3000):
        k = rng.randint(1, 16)
        H, s, p = rng.randint(k, 60), rng.randint(1, min(k, 5)), rng.choice([0, k // 2])
        t = pixels_tile(plans, rng.randint(1, 260), rng.randint(1, 130), H, rng.randint(1, 260), k, s, p)
        taken += t is not None
        assert t is None or (t[3] <= 160 << 10 and k <= 15)
    assert taken > 800


def test_the_loose_layers_of_the_gpu_tests_are_loose(plans):
    for layer, passes in conv.LOOSE_LAYERS.items():
        N, C, H, F, k, s, p, G = layer
        got = [n for n, mode in (('up', UP), ('outp', OUTP)) if plans.conv_tile_is_loose(mode, N, C, H, F, k, co.n_modules(H, k, s, p), s, -p, G, CUS)]
        assert got == passes.split(), layer


def test_the_busiest_xcd_counts_for_every_tile_of_few_colours(plans):
    """convDown of at most 16 colours on tiles of one pixel is expected to be faster than the patch form on the busiest XCD too, also where
    the tile is larger than the layer; among random layers are some that only that refuses."""
    import random
    rng, taken, refused, out = random.Random(6), 0, 0, (ct.c_double * 6)()
    for _ in range(4000):
        N, C, k, F = rng.randint(16, 260), rng.randint(4, 16), rng.randint(1, 11), 4 * rng.randint(2, 64)
        H, p = rng.randint(k, 40), rng.choice([0, k // 2])
        plans.conv_route(DOWN, N, C, H, F, k, co.n_modules(H, k, 1, p), 1, -p, 1, CUS, out)
        tile, single, pixels, us, other, crowd = out
        if tile >= 0 and single and not pixels:
            assert us * crowd <= other + 6 * (crowd - 1)
            taken += 1
        refused += tile < 0 and crowd > 1.2
    assert taken > 200 and refused > 50


# convDown, us: on the other kernels / on the tiles that coarser estimates took it to (of one pixel, of blocks of pixels)
SLOWER_ON_TILES = [
    (173, 13, 15, 244, 7, 1, 0, 1), (205, 8, 12, 236, 5, 1, 0, 1), (146, 13, 20, 220, 6, 1, 0, 1),       # 86 / 142, 46 / 70, 132 / 172
    (256, 82, 22, 256, 7, 4, 3, 2), (128, 43, 45, 128, 6, 4, 0, 1), (256, 88, 32, 64, 6, 2, 3, 2),       # 104 / 137, 86 / 108, 154 / 189
    (128, 74, 28, 96, 7, 2, 3, 2), (128, 70, 23, 192, 5, 2, 2, 2), (112, 46, 15, 48, 3, 3, 0, 1)]        # 120 / 145, 91 / 109, 8.2 / 10.3


def test_layers_that_tiles_made_slower_are_on_the_other_kernels(plans):
    out = (ct.c_double * 6)()
    for N, C, H, F, k, s, p, G in SLOWER_ON_TILES:
        plans.conv_route(DOWN, N, C, H, F, k, co.n_modules(H, k, s, p), s, -p, G, CUS, out)
        assert out[0] < 0, (N, C, H, F, k, s, p, G)


def test_the_choice_of_a_layer_is_kept_by_all_that_it_depends_on(plans):
    layer = [DOWN, 128, 24, 14, 96, 5, 10, 1, 0, 2, 0, 100, 1, 1, 1, CUS]

    def key(values):
        out = (ct.c_int * 32)()
        return list(out[:plans.conv_key_of((ct.c_int * 16)(*values), out)])
    for i, other in enumerate([UP, 100, 48, 16, 64, 3, 12, 2, -2, 1, 1, 50, 2, 0, 0, 304]):
        assert other != layer[i] and key(layer) != key(layer[:i] + [other] + layer[i + 1:]), i
    assert key(layer) == key(list(layer))
