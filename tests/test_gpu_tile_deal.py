"""Order in which tiles are dealt to the XCDs: every tile of a launch is computed once, for launches in interleaved chunks
with and without a last part of fewer than 256 tiles.  Operands of -1, 0 and 1: every sum is a whole number that float32 holds, so
the product is known to the last bit."""
import pytest
import torch

from dion_amd import ops

pytestmark = pytest.mark.gpu


def _signs(shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(-1, 2, shape, device="cuda", generator=g).to(torch.bfloat16)


# tiles of the symmetric product / of the full one (256-wide unless it says otherwise)
@pytest.mark.parametrize("batch,m,n", [
    (1, 4096, 4096),    # 136 / 256: less than a chunk; one whole chunk
    (2, 4096, 4352),    # 272 / 544: a chunk and a part
    (5, 3072, 3584),    # 390 / 840
    (1, 4608, 3584),    # 171 / 252, not a multiple of 8 workgroups
    (12, 1536, 6144),   # 252 / 1728
    (6, 1024, 8192),    # 216 of 128, contiguous / 768
    (8, 1024, 8192),    # 288 of 128
])
def test_every_tile_once(batch, m, n):
    X, S = _signs((batch, m, n), 1), _signs((batch, m, m), 2)
    S = torch.triu(S) + torch.triu(S, 1).mT
    got1, got2, got3 = ops.ns_line_1(X), ops.ns_line_2(S, 1.0, 1.0), ops.ns_line_3(S, X, 0.0)
    for b in range(batch):
        Xf, Sf = X[b].float(), S[b].float()
        assert torch.equal(got1[b], (Xf @ Xf.T).to(torch.bfloat16))
        assert torch.equal(got2[b], (Sf @ Sf + Sf).to(torch.bfloat16))
        assert torch.equal(got3[b], (Sf @ Xf).to(torch.bfloat16))
