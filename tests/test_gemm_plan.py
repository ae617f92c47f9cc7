"""How products are cut into tiles (cacti_hip_gemm_plan; no GPU: the device is taken to have 256 CUs then)."""
import ctypes as C
import random

import pytest

from cacti_amd import ffi


def plan(M, N, K, nz):
    out = (C.c_int64 * 6)()
    assert ffi.lib().cacti_hip_gemm_plan(M, N, K, nz, out) == 0
    return list(out)


@pytest.mark.parametrize("nz", [1, 2, 3, 4, 8])
def test_small_outputs_take_64_by_64_tiles_while_those_fit_the_device(nz):
    assert plan(512, 512, 1024, nz)[:2] == [64, 64]
    assert plan(1024, 256, 128, nz)[:2] == [64, 64]
    assert plan(128, 256, 688, nz)[:2] == [64, 64]


@pytest.mark.parametrize("M,N,K,nz", [(512, 512, 1024, 16), (512, 512, 1024, 32), (512, 512, 192, 64), (256, 1024, 4096, 32)])
def test_many_small_outputs_are_cut_by_cost(M, N, K, nz):
    """More 64 x 64 tiles than the device runs at once: tiles of twice the side need fewer rounds per k tile."""
    p = plan(M, N, K, nz)
    assert p[0] * p[1] > 64 * 64 and p[5] == 1


def test_a_group_is_cut_by_the_same_rule_as_its_products():
    """Small or not is decided for one product where up to four share a launch, so that a group has the bits of its
    products' own launches."""
    for M, N in ((128, 688), (688, 256), (1024, 256), (5, 20000), (512, 512)):
        assert all(plan(M, N, 256, nz)[:2] == [64, 64] for nz in (1, 2, 3, 4))


@pytest.mark.parametrize("M,N,K,how", [(300, 8640, 256, "128, 128, 2, false"), (300, 8640, 1024, "128, 128, 1, false"),
                                       (64, 5504, 256, "64, 64, 2, false"), (64, 256, 256, "64, 64, 2, true")])
def test_kernel_names_tell_the_kernels_of_one_tile_shape_apart(M, N, K, how):
    """128 x 128 exists with one and with two workgroups to a CU, 64 x 64 with either instruction."""
    import bench
    assert bench.kernel_symbol("matmul[NT,1x%dx%dx%d]" % (M, N, K)) == "gemm_direct_kernel<false, true, %s, false>" % how


@pytest.mark.parametrize("label,kernel", [("matmul[NN,1x2048x3200x8640]x2", "gemm_chain_kernel<160, 192, 1, false>"),
                                          ("matmul[NN,1x128x256x256]x3", "gemm_chain_kernel<64, 64, 2, true>"),
                                          ("matmul[TN,1x3200x3200x2048]x3", "gemm_direct_kernel<true, false, 256, 256, 1, false, false>"),
                                          ("matmul[TN,1x8640x3200x2048]x2", None),
                                          ("matmul[NN,1x2048x3200x32000,parts2]", None), ("matmul[NN,1x2048x3200x8640]", "gemm_direct_kernel<false, false, 160, 192, 1, false, false>"),
                                          ("matmul[NN,1x2048x3200x8640,acc]x2", None), ("matmul[NN,1x600x1000x1004]x2", None),
                                          ("matmul_grads[611x1024x1024]x3", None), ("block_matmul[NT,32x2048x2048x100]", None)])
def test_the_kernel_of_a_group_or_a_chain(label, kernel):
    """None: several launches, or products of two layouts in one."""
    import bench
    assert bench.kernel_symbol(label) == kernel


@pytest.mark.parametrize("n,S,N,K,one", [(1, 611, 1024, 1024, 1), (3, 611, 1024, 1024, 1), (2, 611, 2816, 1024, 1), (1, 2048, 2048, 2048, 1),
                                         (2, 603, 9280, 3200, 0), (1, 1267, 17088, 1600, 0), (2, 777, 8640, 3200, 0), (1, 1351, 24104, 2048, 0),
                                         (1, 1854, 2984, 3200, 0), (3, 2048, 3200, 3200, 0)])
def test_all_gradients_in_one_launch_where_that_is_quicker(n, S, N, K, one):
    """Not where the launches apart are as quick: those of 200 us and more, and one of 73, measured 4 to 15 % slower as one."""
    assert ffi.lib().cacti_hip_gemm_f16_grads_one_launch(n, S, N, K) == one


def test_a_kernel_name_needs_its_room():
    name = C.create_string_buffer(128)
    assert ffi.lib().cacti_hip_gemm_kernel_name(1, 0, 2048, 8640, 3200, 1, name, 20) == -1
    assert ffi.lib().cacti_hip_gemm_kernel_name(1, 0, 2048, 8640, 3200, 1, name, 128) == 0
    assert name.value == b"gemm_direct_kernel<true, false, 256, 256, 1, false, false>"
    n = C.c_int(7)
    assert ffi.lib().cacti_hip_gemm_chain_kernel_name(2, 2048, 3200, 8640, name, 20, C.byref(n)) == -1
    assert ffi.lib().cacti_hip_gemm_chain_kernel_name(2, 2048, 3200, 8640, name, 128, C.byref(n)) == 0 and n.value == 1


def parts_plan(M, N, K, parts=0, lent=2 ** 64 - 1):
    """((parts of K, rows and columns of the tile), expected us); parts 0: as a product with a workspace of `lent` bytes is cut, 1: whole."""
    out, us = (C.c_int64 * 3)(), C.c_double()
    assert ffi.lib().cacti_hip_gemm_plan_ws(M, N, K, lent, parts, out, C.byref(us)) == 0
    return tuple(out), us.value


@pytest.mark.parametrize("lent", [2 ** 64 - 1, 64 << 20, 1 << 20])
def test_parts_of_k_are_the_cheapest_that_gain(lent):
    """Of those that fit in what is lent, whatever the order in which tiles and numbers of parts are looked at: none of those that gain the 4 % asked of large tiles on the
    whole product is expected to take less than the cut that is taken."""
    r = random.Random(5)
    drawn = [(round(33 * (2048 / 33) ** r.random()), 8 * round(32 * (400 / 32) ** r.random()), 8 * round(125 * 32 ** r.random())) for _ in range(1500)]
    split = 0
    for M, N, K in drawn + [(1378, 768, 19288), (1325, 3200, 24392), (2048, 3200, 32000), (2048, 2048, 32000), (2056, 2048, 32000)]:
        (parts, _, _), us = parts_plan(M, N, K, lent=lent)
        room = lambda s: s * M * ((N + 3) // 4 * 4) * 4 <= lent
        assert parts == 1 or room(parts), (M, N, K, parts)
        _, whole = parts_plan(M, N, K, 1)
        assert us <= whole, (M, N, K)
        split += parts > 1
        for s in range(2, 9):
            (n, bm, bn), cost = parts_plan(M, N, K, s)
            assert n in (0, s)
            if n and room(n) and cost * 1.04 < whole:
                assert us <= cost, (M, N, K, parts, us, s, bm, bn, cost)
    assert split > (300 if lent > 1 << 20 else 50)


@pytest.mark.parametrize("size,cut", [((3320, 136, 10176), (8, 160, 64)), ((2953, 136, 12288), (8, 160, 64)), ((319, 1248, 19240), (5, 64, 128)),
                                      ((109, 2264, 14936), (7, 64, 128))])
def test_parts_on_long_narrow_tiles(size, cut):
    """Few columns or few rows over a long K: 28 and 25 us, 34 and 27 on the tiles that are next by the costs."""
    assert parts_plan(*size)[0] == cut


def test_a_product_that_is_lent_too_little_for_its_best_parts_is_cut_into_fewer():
    for M, N, K, most in ((2056, 2048, 32000, 270), (1325, 3200, 24392, 220)):
        (parts, _, _), us = parts_plan(M, N, K, lent=64 << 20)
        assert parts > 1 and us < most, (parts, us)


def test_the_products_of_the_traffic_table_are_cut_as_their_labels_say():
    """In a training cycle, which lends 64 MiB to what has no grouped form and is no weight gradient."""
    import bench
    from cacti_amd.gemm_traffic import STEP_PRODUCTS
    for label in STEP_PRODUCTS:
        ta, tb, _, M, N, K = bench.gemm_dims(label)
        lent = 0 if ta or bench.gemm_group(label) > 1 else 64 << 20
        assert parts_plan(M, N, K, lent=lent)[0][0] == bench.gemm_parts(label), label
        assert bench.gemm_launches(label)[1] in (1, 2) and bench.gemm_flops(label) == 2.0 * M * N * K * bench.gemm_group(label)
