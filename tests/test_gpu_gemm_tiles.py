"""Every tile shape of the direct products at the edges of its tiles and of K, each layout, against float64."""
import ctypes as C

import pytest
import torch

from cacti_amd import ffi, ops

TILES = [(64, 64), (96, 64), (160, 64), (64, 128), (96, 128), (128, 128), (160, 128), (128, 192), (160, 192), (192, 192),
         (160, 256), (192, 256), (256, 256)]
# one k tile and a tail of 8; as many k tiles as there are buffers; a tail behind them; enough to go round the buffers
DEPTHS = [72, 128, 200, 328, 520]


def plan(M, N, K):
    out = (C.c_int64 * 6)()
    ffi.call("cacti_hip_gemm_plan", M, N, K, 1, out)
    return tuple(out)


def size_for(tile, K, launches=1):
    """A ragged M x N that is cut into this tile (8 columns of its last one in use), or None."""
    bm, bn = tile
    for tm in list(range(1, 14)) + [17, 27, 34]:
        for tn in list(range(1, 24)) + [33, 40, 60, 101, 126]:
            M, N = tm * bm - bm // 2 - 3, (tn - 1) * bn + 8
            if M * N > 1 << 18 and M * N < 40_000_000:
                p = plan(M, N, K)
                if p[:2] == tile and p[5] == launches:
                    return M, N
    return None


def check(A, B, ta, tb, got, old=None, alpha=1.0):
    """|error| <= half an ulp of the f16 result, and fp32 sums of K products in any order: K 2^-24 sum |a b|."""
    a, b = (A.T if ta else A).double(), (B.T if tb else B).double()
    want, K = alpha * (a @ b), a.shape[1]
    room = abs(alpha) * (a.abs() @ b.abs()) * ((K + 2) * 2.0 ** -24)
    if old is not None:
        want, room = want + old.double(), room + old.double().abs() * 2.0 ** -23
    err = (got.double() - want).abs() - want.abs() * 2.0 ** -11 - room - 2.0 ** -25
    assert err.max().item() <= 0, "worst excess %.3e" % err.max().item()


def operands(M, N, K, ta, tb):
    g = torch.Generator(device="cuda")
    g.manual_seed(M * 7 + N * 3 + K)
    r = lambda *s: torch.randn(s, generator=g, device="cuda", dtype=torch.float16)
    A, B = r(M, K), r(N, K) * 0.1
    return A, B, A.T.contiguous() if ta else A, B if tb else B.T.contiguous()


@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES, ids=lambda t: "%dx%d" % t)
def test_direct_tiles_at_their_edges(tile):
    seen = 0
    for K in DEPTHS:
        size = size_for(tile, K)
        if size is None:
            continue
        seen += 1
        M, N = size
        A, B, _, Bt = operands(M, N, K, False, False)
        base = ops.gemm(A, Bt)
        check(A, B, False, True, base)
        old = torch.randn(M, N, device="cuda", dtype=torch.float16)
        acc = ops.gemm(A, Bt, beta=1.0, out=old.clone())
        check(A, B, False, True, acc, old)
        # the sums are formed in one order whatever the layout: the same bits (a transposed A has rows of 8 elements and more)
        M8 = M // 8 * 8
        for ta, tb in ((False, True), (True, False), (True, True)):
            a, b = (A[:M8].T.contiguous() if ta else A), (B if tb else Bt)
            m = M8 if ta else M
            if plan(m, N, K) == plan(M, N, K):
                assert torch.equal(ops.gemm(a, b, ta=ta, tb=tb), base[:m]), (ta, tb)
                assert torch.equal(ops.gemm(a, b, ta=ta, tb=tb, beta=1.0, out=old[:m].clone()), acc[:m]), (ta, tb)
    assert seen, "no size is cut into %dx%d" % tile


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(2048, 8640, 264), (1531, 11008, 136), (777, 23000, 200)])
def test_columns_beyond_the_full_sets_in_a_second_launch(M, N, K):
    A, B, _, _ = operands(M, N, K, False, True)
    check(A, B, False, True, ops.gemm(A, B, tb=True))
    old = torch.randn(M, N, device="cuda", dtype=torch.float16)
    check(A, B, False, True, ops.gemm(A, B, tb=True, alpha=0.7, beta=1.0, out=old.clone()), old, alpha=0.7)


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K", [(8, 8, 8), (64, 64, 64), (65, 72, 56), (7, 264, 136), (200, 1304, 1000), (512, 512, 328)])
def test_small_outputs(M, N, K, ta, tb):
    """64 x 64 tiles: fewer rows, columns and k than a tile, and a tail of K that comes last."""
    if ta:
        M = (M + 7) // 8 * 8
    A, B, a, b = operands(M, N, K, ta, tb)
    old = torch.randn(M, N, device="cuda", dtype=torch.float16)
    check(A, B, False, True, ops.gemm(a, b, ta=ta, tb=tb))
    check(A, B, False, True, ops.gemm(a, b, ta=ta, tb=tb, beta=1.0, out=old.clone()), old)


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K", [(9, 11, 65), (509, 1003, 770), (130, 4099, 131), (1999, 3001, 203), (1535, 2047, 75), (1537, 2047, 75)])
def test_products_of_any_alignment(M, N, K, ta, tb):
    A, B, a, b = operands(M, N, K, ta, tb)
    old = torch.randn(M, N, device="cuda", dtype=torch.float16)
    check(A, B, False, True, ops.gemm(a, b, ta=ta, tb=tb))
    check(A, B, False, True, ops.gemm(a, b, ta=ta, tb=tb, beta=1.0, out=old.clone()), old)


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K", [(8, 8, 65), (9, 15, 127), (63, 65, 128), (71, 130, 129), (64, 9, 193), (200, 77, 257), (66, 74, 1999),
                                   (5, 3, 200), (7, 300, 77), (9, 11, 8), (33, 70, 13), (130, 9, 63)])
def test_operands_that_start_at_any_half(M, N, K, ta, tb):
    """Edges of tiles and of K with operands between 16-byte boundaries, up to the last half of their memory; strided ones of
    fewer than 8 columns too."""
    A, B, a, b = operands(M, N, K, ta, tb)
    for shift in (1, 3):
        place = lambda t: torch.cat([t.new_full((shift,), float("nan")), t.reshape(-1)])[shift:].view(t.shape)
        got = ops.gemm(place(a), place(b), ta=ta, tb=tb)
        check(A, B, False, True, got)
        old = torch.randn(M, N, device="cuda", dtype=torch.float16)
        check(A, B, False, True, ops.gemm(place(a), place(b), ta=ta, tb=tb, beta=1.0, out=place(old)), old)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(37, 3200, 8640), (5, 2048, 5504), (100, 1000, 9001), (33, 4104, 6000)])
def test_parts_of_k(M, N, K):
    A, B, _, _ = operands(M, N, K, False, True)
    check(A, B, False, True, ops.gemm(A, B, tb=True))


# a product for each tile that parts are formed on but 64 x 64 (above), with rows, columns and a K that no tile divides
PARTS = [((1001, 520, 8200), (96, 64)), ((3321, 136, 10184), (160, 64)), ((109, 2264, 14936), (64, 128)), ((400, 808, 20000), (96, 128)),
         ((227, 1656, 12664), (128, 128)), ((600, 1000, 16008), (160, 128)), ((520, 2008, 20000), (160, 128)), ((1184, 1352, 7048), (160, 192)),
         ((1500, 1000, 12008), (192, 256)), ((1505, 3208, 20000), (256, 256))]


def test_every_tile_of_parts_is_some_product_s():
    """(No GPU: the device is taken to have 256 CUs then.)"""
    out, us = (C.c_int64 * 3)(), C.c_double()
    for size, tile in PARTS:
        ffi.call("cacti_hip_gemm_plan_ws", *size, 2 ** 64 - 1, 0, out, C.byref(us))
        assert out[0] > 1 and tuple(out[1:]) == tile, (size, list(out))


@pytest.mark.gpu
@pytest.mark.parametrize("ta,tb", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("M,N,K", [size for size, _ in PARTS])
def test_parts_of_k_on_large_tiles(M, N, K, ta, tb):
    if ta:
        M = (M + 7) // 8 * 8
    A, B, a, b = operands(M, N, K, ta, tb)
    check(A, B, False, True, ops.gemm(a, b, ta=ta, tb=tb))
    old = torch.randn(M, N, device="cuda", dtype=torch.float16)
    check(A, B, False, True, ops.gemm(a, b, ta=ta, tb=tb, beta=1.0, out=old.clone()), old)


def test_every_tile_is_some_products():
    """(No GPU.)  The sizes above are looked for; at the largest depth each tile has to be found."""
    assert all(size_for(t, DEPTHS[-1]) for t in TILES)
