"""``split_sizes``: the row blocks of a fused weight are updated where they lie.  Bit for bit what separate parameters of the
blocks' shapes get: sizes that fill tiles, padded ones, blocks that start off the 16-byte grid, blocks for the kernel of one
workgroup a matrix, equal and unequal heights, with and without lr adjustment.

With lr adjustment, NorMuon's second moments of a block are those of the block rescaled by the ratio of its lr to the whole
weight's: its square times the separate parameter's, apart from roundings.  In float32 five in each of two steps, under 2^-19;
into a bf16 state one a step, of 2^-8 at most, on each side: 4 x 2^-8.  Half their relative error is in the update."""
import pytest
import torch

from dion import Muon, NorMuon
from dion_amd.optim_base import adjust_lr_ratio, split_lr_scales

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
            assert torch.equal(a.state[w]["momentum"], torch.cat([b.state[p]["momentum"] for p in blocks])), adjust
            whole = torch.cat([p.detach() for p in blocks])
            if cls is Muon or adjust is None:
                assert torch.equal(w.detach(), whole), adjust
            if cls is NorMuon:
                scales = split_lr_scales(split, w.shape, adjust) or (1.0,) * len(split)
                V = torch.cat([b.state[p]["variance_neuron"].float() * f ** 2 for p, f in zip(blocks, scales)])
                off = float((a.state[w]["variance_neuron"].float() - V).abs().div(V).max())
                tol = 2.0 ** -19 if dtype == torch.float32 else 2.0 ** -6
                assert off == 0 if adjust is None else off <= tol, (adjust, off)
                # the weight itself: a rounding to its type a step on each side, and lr * ratio * (an update of norm sqrt(rows)
                # at most, twice)
                step = 4 * float(whole.float().norm()) * (2.0 ** -24 if dtype == torch.float32 else 2.0 ** -8)
                lr = 0.02 * max(adjust_lr_ratio((rows, cols), adjust, False) for rows in split)
                assert float((w.detach() - whole).float().norm()) <= step + 2 * lr * max(split) ** 0.5 * tol * len(split), adjust
