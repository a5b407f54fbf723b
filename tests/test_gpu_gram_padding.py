"""The Gram form on both sides of the lines of the padding (128 or 256, and 256 for the long side alone): its iteration weighs the
products otherwise than the one the lines were measured on, and a restart reads the padded matrix once more.

Bound: the error the same matrices show embedded in zeros up to whole tiles that take the Gram form too, three times as long as
wide at least (same polynomial, same rounding points), with a factor 1.5 for a norm summed in another order."""
import pytest
import torch

from dion_amd import newton_schulz as ns
from dion_amd import ops

DEV = "cuda"
# (batch, rows, cols) -> padded extents (short, long)
PADDED = {
    (264, 130, 500): (256, 512), (90, 300, 1000): (384, 1024), (90, 1000, 300): (384, 1024), (46, 600, 2000): (640, 2048),
    (26, 300, 1000): (384, 1024), (12, 900, 2800): (1024, 2816),  # less than a round of 256-wide tiles
    (24, 512, 2168): (512, 2304), (24, 2168, 512): (512, 2304), (24, 500, 1900): (512, 1920),
}


def test_extents():
    for (b, r, c), want in PADDED.items():
        assert ops.ns_padded_extents(b, r, c, 5, True) == ops.ns_padded_extents(b, r, c, 5) == want, (b, r, c)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", list(PADDED))
def test_operator(shape):
    b, r, c = shape
    g = torch.Generator(device=DEV).manual_seed(b + r + c)
    G = (torch.randn(shape, device=DEV, generator=g) * 0.02).bfloat16()
    m, n = PADDED[shape]
    n = max(n, 3 * m)
    whole = torch.zeros(b, *((m, n) if r <= c else (n, m)), device=DEV, dtype=G.dtype)
    whole[:, :r, :c] = G
    O, W = ns.gram_newton_schulz(G), ns.gram_newton_schulz(whole)[:, :r, :c]
    exact = []
    for i in (0, b - 1):
        X = G[i].double() if r <= c else G[i].double().T
        X = X / (X.norm() * ns.POLAR_EXPRESS_SAFETY)
        for a2, b2, c2 in ns.POLAR_EXPRESS_COEFFS:
            A = X @ X.T
            X = a2 * X + (b2 * A + c2 * A @ A) @ X
        exact.append(X if r <= c else X.T)
    exact = torch.stack(exact)
    rel = lambda t: float((t[[0, b - 1]].double() - exact).norm() / exact.norm())  # noqa: E731
    assert rel(O) <= 1.5 * rel(W) + 1e-4
    assert torch.equal(ns.gram_newton_schulz(G.mT.contiguous()), O.mT)
