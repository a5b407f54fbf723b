"""What the long side of matrices that are padded to 128 is padded to: 256 where that gives the full products more than 384
256-wide tiles.  Bound of the operator test: the error the same matrices show embedded in zeros up to those whole tiles (same
polynomial, same rounding points), with a factor 1.5 for a norm summed in another order."""
import pytest
import torch

from dion_amd import newton_schulz as ns
from dion_amd import ops
from oracle import dion_oracle as oracle

DEV = "cuda"
# (batch, rows, cols) -> padded extents (short, long)
PADDED = {
    (24, 512, 2168): (512, 2304), (24, 2168, 512): (512, 2304), (24, 500, 2176): (512, 2304), (49, 511, 1025): (512, 1280),
    (12, 512, 4216): (512, 4352), (11, 512, 4216): (512, 4224),  # 408 tiles, 374
    (24, 500, 1920): (512, 1920), (48, 500, 1000): (512, 1024),  # 384; an even multiple
    (60, 256, 2168): (256, 2176), (24, 640, 2168): (640, 2176),  # one row of tiles; a short side of 128
}


def test_extents():
    for (b, r, c), want in PADDED.items():
        assert ops.ns_padded_extents(b, r, c, 5) == want, (b, r, c)
    # whole tiles stay as they are
    assert ops.ns_padded_extents(24, 512, 2176, 5) is None and ops.ns_accepts_prepared(24, 512, 2176, 5)
    assert ops.ns_padded_extents(24, 512, 2168, 5, True) == (512, 2304)  # the Gram form too


@pytest.mark.gpu
@pytest.mark.parametrize("func", [ns.zeropower_via_newtonschulz5, ns.polar_express])
@pytest.mark.parametrize("shape", [(24, 512, 2168), (24, 2168, 512), (24, 500, 2176), (49, 511, 1025)])
def test_operator(shape, func):
    b, r, c = shape
    coeffs, scale = (oracle.NS5_COEFFS, 1.0) if func is ns.zeropower_via_newtonschulz5 else (ns.POLAR_EXPRESS_COEFFS, 1.02)
    g = torch.Generator(device=DEV).manual_seed(b + r + c)
    G = (torch.randn(shape, device=DEV, generator=g) * 0.02).bfloat16()
    m, n = PADDED[shape]
    whole = torch.zeros(b, *((m, n) if r <= c else (n, m)), device=DEV, dtype=G.dtype)
    whole[:, :r, :c] = G
    O, W = func(G), func(whole)[:, :r, :c]
    exact = []
    for i in (0, b - 1):
        X = G[i].double()
        X = X / (X.norm() * scale)
        if r > c:
            X = X.T
        for a2, b2, c2 in coeffs:
            A = X @ X.T
            X = a2 * X + (b2 * A + c2 * A @ A) @ X
        exact.append(X.T if r > c else X)
    exact = torch.stack(exact)
    rel = lambda t: float((t[[0, b - 1]].double() - exact).norm() / exact.norm())
    print(shape, rel(O), rel(W))
    assert rel(O) <= 1.5 * rel(W) + 1e-4
    assert torch.equal(func(G.mT.contiguous()), O.mT)
