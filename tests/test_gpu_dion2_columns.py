"""Selected columns of tall matrices with M += G in the gathering pass: the same norms, selection, update of M and selected
block, bit for bit, as accumulating first and gathering after (the form that takes any shape)."""
import pytest
import torch

from dion_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(autouse=True, params=[True, False], ids=["late", "by the rule"])
def late(request, monkeypatch):
    """Both forms at every size: the rule leaves small launches and bf16 momenta to the other one."""
    if request.param:
        monkeypatch.setattr(ops, "_late_add_pays", lambda *a: True)


@pytest.mark.parametrize("sdt,gdt", [(torch.float32, torch.bfloat16), (torch.bfloat16, torch.bfloat16),
                                     (torch.float32, torch.float32), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("where", ["anywhere", "first", "last", "ends", "every fourth"])
@pytest.mark.parametrize("n,mats,rows,cols,k", [(2, 1, 128, 64, 64), (2, 2, 128, 68, 64), (1, 1, 192, 260, 128),
                                                (3, 1, 320, 1028, 192), (1, 3, 576, 300, 64), (2, 1, 1088, 1024, 256)])
def test_same_as_accumulate_then_gather(n, mats, rows, cols, k, where, sdt, gdt):
    gen = torch.Generator(device=DEV).manual_seed(rows + cols)
    mk = lambda dt: [(torch.randn(mats, rows, cols, device=DEV, generator=gen) * 0.1).to(dt) for _ in range(n)]  # noqa: E731
    G, M = mk(gdt), mk(sdt)
    big = {"first": range(k), "last": range(cols - k, cols), "every fourth": range(0, cols, 4),
           "ends": [*range(k // 2), *range(cols - k // 2, cols)]}.get(where, [])
    for m in M:
        if len(big):
            m[..., list(big)] += 3.0
    M2 = [m.clone() for m in M]
    U, idx, imap, sumsq = ops.dion2_select(G, M, k, -1, 0.5, prepared=True)
    U2, idx2, imap2 = ops.dion2_select(G, M2, k, -1, 0.5)
    assert torch.equal(idx, idx2) and torch.equal(imap, imap2)
    assert all(torch.equal(a, b) for a, b in zip(M, M2))
    assert torch.equal(U, U2.view(n * mats, rows, k).mT)
    # fp32 sums of 4096 squares a tile
    exact = U.double().square().sum((1, 2))
    assert bool(((sumsq.double().sum(1) - exact).abs() <= 2.5e-4 * exact).all())


def test_past_the_caches():
    gen = torch.Generator(device=DEV).manual_seed(1)
    n, rows, cols, k = 9, 4160, 2048, 512
    G = [(torch.randn(rows, cols, device=DEV, generator=gen)).bfloat16() for _ in range(n)]
    M = [torch.randn(rows, cols, device=DEV, generator=gen) for _ in range(n)]
    M2 = [m.clone() for m in M]
    U, idx, imap, _ = ops.dion2_select(G, M, k, -1, 0.95, prepared=True)
    U2, idx2, _ = ops.dion2_select(G, M2, k, -1, 0.95)
    assert torch.equal(idx, idx2) and all(torch.equal(a, b) for a, b in zip(M, M2))
    assert torch.equal(U, U2.view(n, rows, k).mT)
