"""Matrices that do not fill whole GEMM tiles: the padded copy (with or without the momentum update in it), the last
product stored without its padding, and the Muon update of parameters without padding, at the edges of the tiles and of
the vector widths, on every GEMM form.

Bounds: the copy and the momentum update are exact; an operator's result is compared with float64 by the error the same
matrices show embedded in zeros up to whole tiles (same polynomial, same rounding points, the zeros change no sum), with
a factor 1.5 for sums taken in another order."""
import pytest
import torch

from dion_amd import newton_schulz as ns
from dion_amd import ops
from oracle import dion_oracle as oracle

pytestmark = pytest.mark.gpu
DEV = "cuda"

# (batch, rows, cols): GEMM form of the last product
SHAPES = [
    (1, 65, 65), (2, 127, 129), (2, 129, 127), (1, 66, 1026), (3, 130, 200), (3, 200, 130),   # 64-wide tiles
    (40, 130, 201), (40, 201, 130), (30, 190, 254), (30, 254, 190),                             # 128-wide, two slots
    (3, 1100, 1151), (3, 1151, 1100), (2, 1090, 1150),                                          # 128-wide, four slots
    (264, 130, 300), (264, 301, 130), (264, 255, 257),                                          # 256-wide
]


def _rand(shape, seed, dtype=torch.bfloat16):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(shape, device=DEV, generator=g) * 0.02).to(dtype)


def _pad_up(G, extents):
    """The matrices in zeros, to whole tiles, in their own orientation."""
    m, n = extents
    r, c = (m, n) if G.shape[-2] <= G.shape[-1] else (n, m)
    out = torch.zeros(G.shape[0], r, c, device=DEV, dtype=G.dtype)
    out[:, :G.shape[-2], :G.shape[-1]] = G
    return out


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", SHAPES)
def test_operator(shape, dtype):
    b, r, c = shape
    G = _rand(shape, b + r + c, dtype)
    extents = ops.ns_padded_extents(b, r, c, 5)
    assert extents is not None
    O = ns.zeropower_via_newtonschulz5(G)
    assert torch.equal(O, ns.zeropower_via_newtonschulz5(G))
    assert torch.equal(ns.zeropower_via_newtonschulz5(G.mT.contiguous()), O.mT) or r == c
    pick = [0, b - 1]
    exact = torch.stack([torch.from_numpy(oracle.ns_fp64(G[i].bfloat16().double().cpu().numpy(), oracle.NS5_COEFFS))
                         for i in pick]).to(DEV)
    whole = ns.zeropower_via_newtonschulz5(_pad_up(G, extents))[:, :r, :c]
    assert _rel(O[pick], exact) <= 1.5 * _rel(whole[pick], exact) + 1e-4


@pytest.mark.parametrize("shape", [(2, 127, 129), (40, 201, 130), (264, 130, 300), (3, 1151, 1100), (2, 130, 500)])
def test_nothing_is_written_beside_the_result(shape):
    import ctypes

    from dion_amd import _lib
    b, r, c = shape
    lib = _lib.load()
    G = _rand(shape, 7)
    want = ns.polar_express(G)
    n = b * r * c
    buf = torch.full((n + 256,), 3.0, device=DEV, dtype=torch.bfloat16)
    ws = torch.full((lib.dion_ns_workspace_bytes(b, r, c, 0),), 0xff, device=DEV, dtype=torch.uint8)
    flat = [x for co in ns.POLAR_EXPRESS_COEFFS for x in co]
    _lib.check(lib.dion_ns_orthogonalize(G.data_ptr(), 0, buf[128:].data_ptr(), b, r, c, (ctypes.c_float * 15)(*flat), 5,
                                         ns.POLAR_EXPRESS_SAFETY, 1e-6, 0, 0, ws.data_ptr(), ws.numel(),
                                         torch.cuda.current_stream().cuda_stream), "ns")
    assert torch.equal(buf[128:128 + n].view(shape), want)
    assert bool((buf[:128] == 3).all()) and bool((buf[128 + n:] == 3).all())


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("g_dtype,m_dtype", [(torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16),
                                             (torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16)])
@pytest.mark.parametrize("mats,rows,cols", [(1, 66, 72), (1, 129, 130), (2, 67, 131), (1, 131, 67), (2, 136, 72), (1, 200, 127)])
def test_momentum_and_padded_copy(mats, rows, cols, g_dtype, m_dtype, offset):
    n = 3

    def tensors(seed, dtype):
        return [_rand((mats * rows * cols + offset,), seed + i, dtype)[offset:].view(mats, rows, cols) for i in range(n)]

    G, M = tensors(1, g_dtype), tensors(11, m_dtype)
    M2 = [m.clone() for m in M]
    extents = ops.ns_padded_extents(n * mats, rows, cols, 5)
    for nesterov in (True, False):
        U = ops.muon_pre([g.clone() for g in G], M2, 0.95, nesterov).view(n * mats, rows, cols)
        X, sumsq = ops.muon_pre_padded(G, M, 0.95, nesterov, mats, rows, cols, extents)
        assert all(torch.equal(a, b) for a, b in zip(M, M2))
        U = U if rows <= cols else U.mT
        assert torch.equal(X[:, :U.shape[1], :U.shape[2]], U)
        assert int((X != 0).sum()) == int((U != 0).sum())
        # fp32 sums of 4096 squares per tile: at most 4096 * 2^-24 relative
        exact = U.double().square().sum((1, 2))
        assert bool(((sumsq.double().sum(1) - exact).abs() <= 2.5e-4 * exact).all())


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("x_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("cautious", [False, True])
@pytest.mark.parametrize("n,mats,rows,cols", [(2, 1, 127, 130), (2, 1, 130, 127), (3, 2, 202, 130), (20, 2, 130, 201),
                                              (20, 2, 202, 130), (3, 1, 1100, 1151), (3, 1, 1152, 1100), (66, 4, 130, 300),
                                              (66, 4, 302, 130), (66, 4, 301, 255)])
def test_update_without_padding(n, mats, rows, cols, cautious, x_dtype, offset):
    """The update in the last product against the operator followed by the update pass: the same bits, and nothing
    outside the parameters (between which a few elements lie)."""
    numel = mats * rows * cols
    pitch = numel + 64 + offset - numel % 8

    def params():
        buf = _rand((n * pitch + 64,), 5, x_dtype)
        return buf, [buf[i * pitch + offset:i * pitch + offset + numel].view(mats, rows, cols) for i in range(n)]

    b1, X1 = params()
    b2, X2 = params()
    lr = torch.tensor(0.02, device=DEV)
    G = _rand((n * mats, rows, cols), 3)
    ns.orthogonalize_update(ns.polar_express, G, 1e-6, X1, lr, 0.7, 0.1, cautious)
    O = ns.polar_express(G, 1e-6)
    ops.muon_post(X2, O.view(n, -1), lr, 0.7, 0.1, cautious)
    assert torch.equal(b1, b2)


@pytest.mark.parametrize("cls", ["Muon", "NorMuon"])
@pytest.mark.parametrize("shape", [(130, 201), (201, 130), (2, 100, 70)])
def test_step_with_and_without_the_padded_hand_over(shape, cls):
    """One step through the padded form against the step whose orthogonalization makes the padded copy itself."""
    import dion

    def build(handed_over):
        ps = []
        for i in range(3):
            p = torch.nn.Parameter(_rand(shape, i, torch.float32))
            p.grad = _rand(shape, 20 + i, torch.float32)
            ps.append(p)
        opt = getattr(dion, cls)(ps, lr=0.02, weight_decay=0.1, cautious_wd=True)
        opt.prepared_input = handed_over
        for _ in range(2):
            opt.step()
        return [p.data for p in ps] + [opt.state[p]["momentum"] for p in ps]

    assert all(torch.equal(a, b) for a, b in zip(build(True), build(False)))


def _both_forms(G, func, eps):
    """The operator on G, and on its padded form from the momentum pass (M = 0, no momentum: U = G)."""
    b, r, c = G.shape
    yield func(G, eps)
    extents = ns.padded_extents(func, b, r, c)
    U, sumsq = ops.muon_pre_padded([G], [torch.zeros_like(G)], 0.0, False, b, r, c, extents)
    yield ns.orthogonalize_prepared(func, U, sumsq, r, c, eps, padded=True)


@pytest.mark.parametrize("shape", [(2, 130, 200), (2, 200, 130), (3, 1100, 1151), (40, 130, 201)])
@pytest.mark.parametrize("exponent", [-58, -46, -34, 34, 46, 54])
def test_inputs_of_any_magnitude(shape, exponent):
    """The scale of the input cancels, also where squares of the values as they came leave the range of fp32: powers of two
    on both sides of where the copy is scaled (squared norms of 2^-80 and 2^80).  The bound is the error without the power
    of two; one more rounding of the scaled matrix is within the factor."""
    G = _rand(shape, 5)
    exact = torch.stack([torch.from_numpy(oracle.ns_fp64(g.double().cpu().numpy(), oracle.NS5_COEFFS, 1.0, 0.0)) for g in G[:2]]).to(DEV)
    bound = 1.5 * _rel(ns.zeropower_via_newtonschulz5(G, 0.0)[:2], exact) + 1e-4
    scaled = torch.ldexp(G.float(), torch.tensor(exponent, device=DEV)).bfloat16()
    for O in _both_forms(scaled, ns.zeropower_via_newtonschulz5, 0.0):
        assert _rel(O[:2], exact) <= bound


@pytest.mark.parametrize("shape", [(3, 130, 200), (3, 200, 130)])
def test_norms_past_fp32_and_values_that_are_not_finite(shape):
    """X / inf is 0 where X is finite; a value that is not makes its own matrix NaN and no other."""
    G = _rand(shape, 6)
    G[0] = 2.0 ** 64
    G[1, 5, 7] = float("inf")
    want = ns.polar_express(_rand(shape, 6))[2]
    for O in _both_forms(G, ns.polar_express, 1e-6):
        assert not bool(O[0].any())
        assert bool(O[1].isnan().all())
        assert torch.equal(O[2], want)
