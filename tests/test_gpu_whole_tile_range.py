"""Magnitudes of inputs that fill 128-wide tiles and not 256-wide ones, in batches for which 256-wide tiles would pad them: the norm
is taken out of a copy (or of the prepared input), as where they are padded, so that a norm out of the range of fp32's squares
comes out as it does there."""
import pytest
import torch

from dion_amd import newton_schulz as ns
from dion_amd import ops
from oracle import dion_oracle as oracle

DEV = "cuda"
SHAPES = [(90, 384, 640), (90, 640, 384), (90, 384, 1280)]  # the last one long enough for the Gram form


def test_these_are_whole_tiles():
    for b, r, c in SHAPES:
        assert ops.ns_padded_extents(b, r, c, 5) is None and ops.ns_accepts_prepared(b, r, c, 5)


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


def _rand(shape, seed, dtype=torch.bfloat16):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(shape, device=DEV, generator=g) * 0.02).to(dtype)


def _forms(G, func, eps):
    """The operator on G as it is and in float32, and on the prepared form from the momentum pass (M = 0, no momentum: U = G)."""
    b, r, c = G.shape
    yield func(G, eps)
    yield func(G.float(), eps)
    U, sumsq = ops.muon_pre_prepared([G], [torch.zeros_like(G)], 0.0, False, b, r, c)
    yield ns.orthogonalize_prepared(func, U, sumsq, r, c, eps)


@pytest.mark.gpu
@pytest.mark.parametrize("func,shape", [(ns.zeropower_via_newtonschulz5, s) for s in SHAPES] + [(ns.gram_newton_schulz, SHAPES[2])])
@pytest.mark.parametrize("exponent", [-58, -46, -34, 34, 46, 54])
def test_inputs_of_any_magnitude(func, shape, exponent):
    """Powers of two on both sides of squared norms of 2^-80 and 2^80; bound: the error without the power of two, with a factor
    for one more rounding of the scaled matrix."""
    coeffs, scale = (oracle.NS5_COEFFS, 1.0) if func is ns.zeropower_via_newtonschulz5 else (ns.POLAR_EXPRESS_COEFFS, 1.02)
    G = _rand(shape, 5)
    pick = [0, shape[0] - 1]
    exact = torch.stack([torch.from_numpy(oracle.ns_fp64(G[i].double().cpu().numpy(), coeffs, scale, 0.0)) for i in pick]).to(DEV)
    bound = 1.5 * _rel(func(G, 0.0)[pick], exact) + 1e-4
    for O in _forms(torch.ldexp(G.float(), torch.tensor(exponent, device=DEV)).bfloat16(), func, 0.0):
        assert _rel(O[pick], exact) <= bound


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES[:2])
def test_norms_past_fp32_and_values_that_are_not_finite(shape):
    """X / inf is 0 where X is finite; a value that is not makes its own matrix NaN and no other."""
    plain, G = _rand(shape, 6), _rand(shape, 6)
    G[0] = 2.0 ** 64
    G[1, 5, 7] = float("inf")
    for want, O in zip(_forms(plain, ns.polar_express, 1e-6), _forms(G, ns.polar_express, 1e-6)):
        assert not bool(O[0].any())
        assert bool(O[1].isnan().all())
        assert torch.equal(O[2:], want[2:])
    assert float(G[0, 0, 0]) == 2.0 ** 64  # a plain call leaves its input alone


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("gram", [False, True])
def test_launches_stay_in_their_buffers(shape, gram):
    """Every launch of plain, updating, in-place and prepared calls inside the call's buffers; in a short workspace, not."""
    from dion_amd import _lib

    lib, (b, r, c), flags = _lib.load(), shape, _lib.DION_NS_GRAM if gram else 0
    for in_dtype in (_lib.DION_BF16, _lib.DION_F32):
        for update in (0, 1):
            assert lib.dion_ns_plan_audit(b, r, c, in_dtype, 5, flags, 2, update, _lib.DION_F32, 3, 0) > 0
    assert lib.dion_ns_plan_audit_prepared(b, r, c, 5, flags, 2, 1, _lib.DION_F32, 3, 0) > 0
    assert lib.dion_ns_plan_audit_overlap(b, r, c, _lib.DION_BF16, 5, flags, 2, 0) > 0
    assert lib.dion_ns_plan_audit(b, r, c, _lib.DION_BF16, 5, flags, 2, 0, _lib.DION_F32, 1, 1 << 20) < 0


@pytest.mark.gpu
@pytest.mark.parametrize("x_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", SHAPES[:2])
def test_update_on_the_last_product(shape, x_dtype):
    """One call against orthogonalization and update, bit for bit."""
    b, r, c = shape
    G, lr = _rand(shape, 3), torch.tensor(0.02, device=DEV)
    X1 = [_rand((3, r, c), 10 + i, x_dtype) for i in range(b // 3)]
    X2 = [x.clone() for x in X1]
    ns.orthogonalize_update(ns.polar_express, G, 1e-6, X1, lr, 0.7, 0.1, True)
    ops.muon_post(X2, ns.polar_express(G, 1e-6).view(b // 3, -1), lr, 0.7, 0.1, True)
    assert all(torch.equal(x, y) for x, y in zip(X1, X2))
