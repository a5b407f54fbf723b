"""``split_sizes``: the row blocks of a fused weight are updated where they lie, as shape groups of their own.  Bit for bit
what separate parameters of the blocks' shapes get: sizes that fill tiles, padded ones, blocks that start off the 16-byte
grid, blocks for the kernel of one workgroup a matrix, equal and unequal heights, with and without lr adjustment."""
import pytest
import torch

from dion import Muon, NorMuon

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("cls", [Muon, NorMuon])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("split,cols", [((256, 128, 128), 256), ((200, 50, 50), 200), ((130, 67, 130), 133), ((64, 32, 64), 96),
                                        ((7, 300), 129), ((512, 512, 512), 384), ((1, 1), 5)])
def test_blocks_are_updated_like_parameters(cls, dtype, split, cols):
    g = torch.Generator(device=DEV).manual_seed(sum(split) + cols)
    rand = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    for adjust in ("spectral_norm", "rms_norm", None):
        fused = [torch.nn.Parameter((rand(sum(split), cols) * 0.02).to(dtype)) for _ in range(3)]
        parts = [[torch.nn.Parameter(b.clone()) for b in w.detach().split(list(split))] for w in fused]
        kw = dict(lr=0.02, weight_decay=0.01, nesterov=True, cautious_wd=adjust is None, adjust_lr=adjust)
        # (the blocks of one height in the order of the fused step: the first block of every weight, then the second)
        a = cls([{"params": fused, "split_sizes": split}], **kw)
        b = cls([p for blocks in zip(*parts) for p in blocks], **kw)
        for _ in range(2):
            for w, blocks in zip(fused, parts):
                w.grad = rand(*w.shape).to(dtype) * 0.02
                for p, gb in zip(blocks, w.grad.split(list(split))):
                    p.grad = gb.clone()
            a.step()
            b.step()
        for w, blocks in zip(fused, parts):
            assert torch.equal(w.detach(), torch.cat([p.detach() for p in blocks])), adjust
            assert torch.equal(a.state[w]["momentum"], torch.cat([b.state[p]["momentum"] for p in blocks])), adjust
            if cls is NorMuon:
                assert torch.equal(a.state[w]["variance_neuron"], torch.cat([b.state[p]["variance_neuron"] for p in blocks]))
