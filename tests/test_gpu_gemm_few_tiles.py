"""The GEMM forms for launches of few tiles (64-wide tiles with the reduction split over a workgroup's wavefronts;
128-wide tiles on a four-slot ring) at the sizes where they can go wrong: fewer k slabs than wavefronts or ring
slots, slab counts that are no multiple of either, one tile, tile counts on both sides of each rule.  References
are float64 products of the same bf16 inputs; the bound on the mean error is that of one bf16 rounding of the result
(2^-9 of its magnitude at most) plus fp32 accumulation."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _lib():
    from dion_amd import _lib as L

    return L.load(), L.check, torch.cuda.current_stream().cuda_stream


def _close(res, ref):
    """Every element within one bf16 rounding of the float64 value, with the fp32 sums (K terms, relative 2^-24
    each, of the magnitude of the row's products) on top."""
    err = (res.double() - ref).abs()
    bound = ref.abs() * 2.0 ** -8 + ref.abs().mean() * 1e-4
    assert bool((err <= bound).all()), float((err - bound).max())


# (batch, m, n, tile edge of the symmetric products, of B X)
CASES = [
    (1, 128, 128, 64, 64), (1, 128, 384, 64, 64), (3, 256, 640, 64, 64), (1, 896, 128, 64, 64),
    (2, 384, 1664, 64, 128), (4, 512, 2048, 64, 128), (14, 512, 128, 64, 64), (15, 512, 128, 128, 64),
    (1, 1408, 1408, 64, 128), (1, 2048, 2048, 128, 128), (1, 1920, 2176, 64, 128), (7, 1024, 1152, 128, 128),
]


@pytest.mark.parametrize("batch,m,n,sym_edge,full_edge", CASES)
def test_products_of_few_tiles(batch, m, n, sym_edge, full_edge):
    lib, check, st = _lib()
    assert lib.dion_gemm_tile_edge(batch, m, m, 1) == sym_edge
    assert lib.dion_gemm_tile_edge(batch, m, n, 0) == full_edge
    g = torch.Generator(device=DEV).manual_seed(m + n)
    X = torch.randn(batch, m, n, device=DEV, generator=g).to(torch.bfloat16)
    A = torch.full((batch, m, m), float("nan"), device=DEV, dtype=torch.bfloat16)
    B = torch.full_like(A, float("nan"))
    Y = torch.full_like(X, float("nan"))
    check(lib.dion_ns_line_1(X.data_ptr(), A.data_ptr(), batch, m, n, st), "line_1")
    ref = X.double() @ X.double().mT.contiguous()
    _close(A, ref)
    assert torch.equal(A, A.mT)
    S = (A.float() / n).to(torch.bfloat16)
    check(lib.dion_ns_line_2(S.data_ptr(), B.data_ptr(), batch, m, ctypes.c_float(0.5), ctypes.c_float(2.0), st), "line_2")
    Sd = S.double()
    _close(B, 0.5 * (Sd @ Sd) + 2.0 * Sd)
    assert torch.equal(B, B.mT)
    check(lib.dion_ns_line_3(B.data_ptr(), X.data_ptr(), Y.data_ptr(), batch, m, n, ctypes.c_float(0.0), st), "line_3")
    _close(Y, B.double() @ X.double())
    A2 = torch.empty_like(A)
    check(lib.dion_ns_line_1(X.data_ptr(), A2.data_ptr(), batch, m, n, st), "line_1")
    assert torch.equal(A, A2)


@pytest.mark.parametrize("shape,cautious", [((1, 256, 512), False), ((1, 512, 256), True), ((1, 2048, 2048), False),
                                            ((2, 384, 384), True)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_fused_update_of_few_tiles(shape, cautious, dtype):
    """The update applied by these kernels equals the update pass on their stored result, bit for bit."""
    from dion_amd import ops
    from dion_amd.newton_schulz import NS5_COEFFS

    torch.manual_seed(5)
    batch = shape[0]
    G = (torch.randn(*shape, device=DEV) * 0.02).to(torch.bfloat16)
    X = [(torch.randn(*shape[1:], device=DEV) * 0.02).to(dtype) for _ in range(batch)]
    X2 = [x.clone() for x in X]
    lr = torch.tensor(0.02, device=DEV)
    ops.ns_orthogonalize_update(G, X, NS5_COEFFS, 1.0, 1e-7, lr, 0.7, 0.01, cautious)
    ops.muon_post(X2, ops.ns_orthogonalize(G, NS5_COEFFS, 1.0, 1e-7).view(batch, -1), lr, 0.7, 0.01, cautious)
    assert all(torch.equal(a, b) for a, b in zip(X, X2))


@pytest.mark.parametrize("batch,m,n,sym_edge,full_edge", [(86, 128, 128, 128, 128), (128, 128, 256, 128, 128), (100, 128, 1024, 128, 128),
                                                          (26, 256, 256, 128, 128), (26, 256, 512, 128, 128), (13, 384, 384, 64, 128),
                                                          (14, 512, 256, 64, 128)])
def test_products_at_the_line_of_short_reductions(batch, m, n, sym_edge, full_edge):
    test_products_of_few_tiles(batch, m, n, sym_edge, full_edge)


# Slab counts (64 columns of the reduction each) from fewer than a ring has slots, remainders of its length among them.
# 504 tiles of 64 from n = 384 on and 140 of 128 on the four-slot ring below; 160 on the four-slot ring; 300 on the two-slot one
@pytest.mark.parametrize("batch", [14, 16, 30])
@pytest.mark.parametrize("n", [128, 256, 384, 512, 640, 768, 896, 1152])
def test_reduction_lengths_of_symmetric_products(batch, n):
    lib, check, st = _lib()
    assert lib.dion_ns_line_kernel(1, batch, 512, n, 0) == (128 if batch == 30 else 129 if batch == 16 or n < 384 else 64)
    g = torch.Generator(device=DEV).manual_seed(n)
    X = torch.randn(batch, 512, n, device=DEV, generator=g).to(torch.bfloat16)
    A = torch.full((batch, 512, 512), float("nan"), device=DEV, dtype=torch.bfloat16)
    check(lib.dion_ns_line_1(X.data_ptr(), A.data_ptr(), batch, 512, n, st), "line_1")
    _close(A, X.double() @ X.double().mT.contiguous())
    assert torch.equal(A, A.mT)


@pytest.mark.parametrize("m", [128, 256, 384, 512, 640, 1152])
def test_reduction_lengths_of_products_with_a_k_major_operand(m):
    lib, check, st = _lib()
    batch, n = -(-12800 // m), 384  # 300 tiles and a few more, of a width that has no 256-wide ones
    assert lib.dion_gemm_tile_edge(batch, m, n, 0) == 128
    g = torch.Generator(device=DEV).manual_seed(m)
    B = torch.randn(batch, m, m, device=DEV, generator=g)
    B = (B + B.mT).to(torch.bfloat16)
    X = torch.randn(batch, m, n, device=DEV, generator=g).to(torch.bfloat16)
    Y = torch.full_like(X, float("nan"))
    check(lib.dion_ns_line_3(B.data_ptr(), X.data_ptr(), Y.data_ptr(), batch, m, n, ctypes.c_float(0.0), st), "line_3")
    _close(Y, B.double() @ X.double())


# The addend travels through the ring behind the last slab: slab counts (m / 64) from two, remainders of the ring's length,
# more than eight tile rows; four-slot and two-slot rings of 128-wide tiles, and 256-wide tiles.
@pytest.mark.parametrize("m,batch,sym_edge", [(128, 300, 128), (256, 70, 128), (256, 200, 256), (384, 42, 128), (384, 60, 128), (512, 20, 128),
                                              (512, 60, 256), (640, 16, 128), (768, 30, 256), (1152, 3, 128), (1152, 8, 128), (2304, 4, 256)])
def test_addend_at_every_slab_count(m, batch, sym_edge):
    lib, check, st = _lib()
    assert lib.dion_gemm_tile_edge(batch, m, m, 1) == sym_edge
    g = torch.Generator(device=DEV).manual_seed(m + batch)
    S = torch.randn(batch, m, m, device=DEV, generator=g)
    S = ((S + S.mT) * (0.5 / m ** 0.5)).to(torch.bfloat16)
    X = torch.randn(batch, m, m, device=DEV, generator=g).to(torch.bfloat16)
    B, Y = (torch.full_like(S, float("nan")) for _ in range(2))
    Sd = S.double()
    check(lib.dion_ns_line_2(S.data_ptr(), B.data_ptr(), batch, m, ctypes.c_float(0.5), ctypes.c_float(2.0), st), "line_2")
    _close(B, 0.5 * (Sd @ Sd) + 2.0 * Sd)
    assert torch.equal(B, B.mT)
    check(lib.dion_ns_line_3(S.data_ptr(), X.data_ptr(), Y.data_ptr(), batch, m, m, ctypes.c_float(0.75), st), "line_3")
    _close(Y, Sd @ X.double() + 0.75 * X.double())


# K-major operand and addend on the four-slot ring: slab counts (m / 64) that leave the addend in either of its slots.
@pytest.mark.parametrize("m", [1152, 1280, 1408, 1536])
def test_k_major_products_on_the_four_slot_ring(m):
    lib, check, st = _lib()
    assert lib.dion_ns_line_kernel(3, 1, m, m, 0) == 129 and lib.dion_ns_line_kernel(3, 1, m, m, 1) == 129
    g = torch.Generator(device=DEV).manual_seed(m)
    B = (torch.randn(1, m, m, device=DEV, generator=g) / m ** 0.5).to(torch.bfloat16)
    X = torch.randn(1, m, m, device=DEV, generator=g).to(torch.bfloat16)
    for a in (0.0, 0.75):
        Y = torch.full_like(X, float("nan"))
        check(lib.dion_ns_line_3(B.data_ptr(), X.data_ptr(), Y.data_ptr(), 1, m, m, ctypes.c_float(a), st), "line_3")
        _close(Y, B.double() @ X.double() + a * X.double())


# Full products on both sides of the lines between 128- and 256-wide tiles: one round of the CUs, and most of two.
@pytest.mark.parametrize("batch,m,n,edge", [(32, 512, 512, 128), (43, 256, 768, 256), (32, 512, 1024, 256), (17, 1024, 1024, 128),
                                            (42, 512, 1024, 256), (7, 1536, 1536, 256), (10, 1536, 1536, 128), (9, 1024, 1152, 128)])
def test_full_products_at_the_lines_of_256_wide_tiles(batch, m, n, edge):
    lib, check, st = _lib()
    assert lib.dion_gemm_tile_edge(batch, m, n, 0) == edge
    g = torch.Generator(device=DEV).manual_seed(batch)
    B = torch.randn(batch, m, m, device=DEV, generator=g)
    B = ((B + B.mT) * (0.5 / m ** 0.5)).to(torch.bfloat16)
    X = torch.randn(batch, m, n, device=DEV, generator=g).to(torch.bfloat16)
    Y = torch.full_like(X, float("nan"))
    check(lib.dion_ns_line_3(B.data_ptr(), X.data_ptr(), Y.data_ptr(), batch, m, n, ctypes.c_float(0.0), st), "line_3")
    _close(Y, B.double() @ X.double())


# Symmetric products on both sides of the lines between 64-, 128- (129: on the four-slot ring) and 256-wide tiles.
@pytest.mark.parametrize("batch,m,n,kernel", [(6, 768, 768, 64), (6, 768, 1024, 64), (7, 768, 1024, 129), (1, 1920, 1920, 64),
                                              (1, 1920, 2048, 64), (1, 2048, 2048, 129), (21, 512, 1024, 129), (51, 512, 512, 128),
                                              (52, 512, 512, 256), (85, 512, 640, 256), (86, 512, 640, 128), (36, 1024, 1024, 128),
                                              (32, 1024, 2176, 128), (33, 1024, 2176, 256), (20, 1536, 1536, 256)])
def test_symmetric_products_at_the_lines(batch, m, n, kernel):
    lib, check, st = _lib()
    assert lib.dion_ns_line_kernel(1, batch, m, n, 0) == kernel
    g = torch.Generator(device=DEV).manual_seed(batch + n)
    X = torch.randn(batch, m, n, device=DEV, generator=g).to(torch.bfloat16)
    A = torch.full((batch, m, m), float("nan"), device=DEV, dtype=torch.bfloat16)
    check(lib.dion_ns_line_1(X.data_ptr(), A.data_ptr(), batch, m, n, st), "line_1")
    _close(A, X.double() @ X.double().mT.contiguous())
    assert torch.equal(A, A.mT)


# 257-512 tiles of 64: the reduction is added up in four partial sums, slab (64 columns) by slab in turn, whether it is
# longer than the matrix is wide or not.  Slabs 0 and 4 bring 2^26 and -2^26 to one partial sum, slab 1 a 1 to another: exact
# there, lost in one chain, where 2^26 + 1 rounds to 2^26.
@pytest.mark.parametrize("batch,m,n", [(86, 128, 1024), (113, 128, 2048), (26, 256, 512), (13, 512, 2048), (6, 768, 3072), (2, 1024, 4096),
                                       (1, 1920, 2176), (14, 512, 512), (2, 1024, 1024)])
def test_partial_sums_of_symmetric_products(batch, m, n):
    lib, check, st = _lib()
    X = torch.zeros(batch, m, n, device=DEV, dtype=torch.bfloat16)
    X[:, :, 0] = 2.0 ** 13
    X[:, :, 64] = 1.0
    X[:, 0::2, 256] = 2.0 ** 13
    X[:, 1::2, 256] = -(2.0 ** 13)
    A = torch.full((batch, m, m), float("nan"), device=DEV, dtype=torch.bfloat16)
    check(lib.dion_ns_line_1(X.data_ptr(), A.data_ptr(), batch, m, n, st), "line_1")
    assert bool((A[:, 0::2, 1::2] == 1).all())
    assert torch.equal(A, A.mT)


def test_addend_with_rows_too_long_for_32_bit_offsets():
    lib, check, st = _lib()
    m, n = 128, 1 << 26
    if torch.cuda.mem_get_info()[0] < 64 << 30:
        pytest.skip("needs 35 GB")
    assert lib.dion_ns_line_kernel(3, 1, m, n, 1) == 64
    g = torch.Generator(device=DEV).manual_seed(1)
    B = torch.randn(1, m, m, device=DEV, generator=g).to(torch.bfloat16)
    X = torch.zeros(1, m, n, device=DEV, dtype=torch.bfloat16)
    Y = torch.empty_like(X)
    parts = [slice(c, c + 4096) for c in (0, n // 2 - 2048, n - 4096)]
    for p in parts:
        X[:, :, p] = torch.randn(1, m, 4096, device=DEV, generator=g).to(torch.bfloat16)
    check(lib.dion_ns_line_3(B.data_ptr(), X.data_ptr(), Y.data_ptr(), 1, m, n, ctypes.c_float(0.75), st), "line_3")
    for p in parts:
        Xd = X[:, :, p].double()
        _close(Y[:, :, p], B.double() @ Xd + 0.75 * Xd)
    assert not bool(Y[:, :, 4096:n // 2 - 2048].any()) and not bool(Y[:, :, n // 2 + 2048:n - 4096].any())
