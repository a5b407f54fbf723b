"""``split_sizes`` with neighbours of one height: the blocks behind one address, in several runs, off the 16-byte grid, more than a
pointer table holds, and stacked past what one call takes.  Updated where they lie, they get bit for bit what separate parameters
of the blocks' shapes get."""
import pytest
import torch

from dion import Muon, NorMuon
from dion_amd import optimizers

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _two_steps(cls, split, cols, dtype, **kw):
    g = torch.Generator(device=DEV).manual_seed(sum(split) + cols)
    rand = lambda *s: torch.randn(*s, device=DEV, generator=g) * 0.02  # noqa: E731
    fused = [torch.nn.Parameter(rand(sum(split), cols).to(dtype)) for _ in range(3)]
    parts = [[torch.nn.Parameter(b.clone()) for b in w.detach().split(list(split))] for w in fused]
    kw = dict(lr=0.02, weight_decay=0.01, adjust_lr=None, **kw)
    a, b = cls([{"params": fused, "split_sizes": split}], **kw), cls([p for blocks in zip(*parts) for p in blocks], **kw)
    for _ in range(2):
        for w, blocks in zip(fused, parts):
            w.grad = rand(*w.shape).to(dtype)
            for p, gb in zip(blocks, w.grad.split(list(split))):
                p.grad = gb.clone()
        a.step()
        b.step()
    out = []
    for w, blocks in zip(fused, parts):
        out.append((w.detach(), torch.cat([p.detach() for p in blocks])))
        out += [(t, torch.cat([b.state[p][k] for p in blocks])) for k, t in a.state[w].items()]
    return out


@pytest.mark.parametrize("cls", [Muon, NorMuon])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("split,cols", [((64,) * 12, 96), ((128, 128, 64, 128, 128, 64), 256), ((128, 128, 64, 128), 129),
                                        ((65, 64) * 25, 67), ((256, 256, 384), 512), ((3, 3, 3, 300), 257)])
def test_blocks_are_updated_like_parameters(cls, dtype, split, cols):
    assert all(torch.equal(x, y) for x, y in _two_steps(cls, split, cols, dtype))


@pytest.mark.parametrize("cls", [Muon, NorMuon])
@pytest.mark.parametrize("split,cols", [((64,) * 12, 96), ((128, 128, 64, 128), 129)])
def test_stacked_blocks(cls, split, cols, monkeypatch):
    """Without lr adjustment the blocks are not rescaled, and the stacked form takes the same steps: the momentum to the bit, the
    update within the rounding of another order of sums in the norm (a bf16 rounding of each element, 2^-8, at most)."""
    monkeypatch.setattr(optimizers, "_MOST_ROW_BLOCKS", 1)
    for (x, y) in _two_steps(cls, split, cols, torch.float32, mu=0.9):
        assert float((x - y).norm()) <= 2.0 ** -8 * float(y.norm())
