"""What matrices are padded to where the symmetric products offer 256-wide tiles a full round of the CUs: 128 when that
leaves 18 % or more of the operations out, else 256.  One shape on either side of that line, wide and tall; those that keep
256-wide tiles are also the bounded last product on them.

Bound: the error the same matrices show embedded in zeros up to whole tiles (same polynomial, same rounding points), with a
factor 1.5 for sums taken in another order."""
import pytest
import torch

from dion_amd import newton_schulz as ns
from dion_amd import ops
from oracle import dion_oracle as oracle

DEV = "cuda"
# (batch, rows, cols) -> padded extents (short, long)
PADDED = {
    (264, 130, 500): (256, 512), (264, 501, 130): (256, 512), (264, 255, 511): (256, 512),  # nothing to gain
    (264, 130, 300): (256, 384), (264, 300, 130): (256, 384), (90, 300, 301): (384, 384), (90, 320, 640): (384, 640),
    (46, 600, 1000): (640, 1024),
    (26, 900, 1024): (1024, 1024), (8, 1900, 1910): (2048, 2048),
}


def test_extents():
    for (b, r, c), want in PADDED.items():
        assert ops.ns_padded_extents(b, r, c, 5) == want, (b, r, c)
    # multiples of 128 that were padded to 256 are whole tiles now, and taken in the prepared form
    assert ops.ns_padded_extents(90, 384, 640, 5) is None and ops.ns_accepts_prepared(90, 384, 640, 5)
    # below one round of 256-wide tiles: 128 whatever it leaves out
    assert ops.ns_padded_extents(3, 300, 301, 5) == (384, 384)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [s for s in PADDED if s[0] != 8])
def test_operator(shape):
    b, r, c = shape
    g = torch.Generator(device=DEV).manual_seed(b + r + c)
    G = (torch.randn(shape, device=DEV, generator=g) * 0.02).bfloat16()
    m, n = PADDED[shape]
    whole = torch.zeros(b, *((m, n) if r <= c else (n, m)), device=DEV, dtype=G.dtype)
    whole[:, :r, :c] = G
    O, W = ns.zeropower_via_newtonschulz5(G), ns.zeropower_via_newtonschulz5(whole)[:, :r, :c]
    pick = [0, b // 2, b - 1]
    exact = torch.stack([torch.from_numpy(oracle.ns_fp64(G[i].double().cpu().numpy(), oracle.NS5_COEFFS)) for i in pick])
    rel = lambda t: float((t[pick].cpu().double() - exact).norm() / exact.norm())
    assert rel(O) <= 1.5 * rel(W) + 1e-4
    assert torch.equal(ns.zeropower_via_newtonschulz5(G.mT.contiguous()), O.mT)
