"""How row blocks of ``split_sizes`` become matrices and addresses: neighbours of one height lie behind one address, as heads do,
so that a weight cut into many equal blocks costs the host no more than its heads."""
import random

import pytest
import torch

import dion
from dion_amd import ops, optimizers


def test_every_block_once():
    rng = random.Random(0)
    cases = [(64,) * 36, (1000, 250, 250), (5, 7), (1, 1), (4, 4, 2, 4, 4), (4, 4, 2, 4), (3, 3, 3, 1, 3, 3, 3, 3, 3, 3)]
    cases += [tuple(rng.choice((1, 2, 2, 5)) for _ in range(rng.randint(2, 30))) for _ in range(50)]
    for split in cases:
        want = [(sum(split[:i]), rows) for i, rows in enumerate(split)]
        got = [(at + i * rows, rows) for rows, mats, first in optimizers._equal_blocks(split) for at in first
               for i in range(mats)]
        assert sorted(got) == want, split
    assert optimizers._equal_blocks((64,) * 36) == [(64, 36, [0])]
    assert optimizers._equal_blocks((1000, 250, 250)) == [(1000, 1, [0]), (250, 2, [1000])]
    assert optimizers._equal_blocks((4, 4, 2, 4, 4)) == [(4, 2, [0, 10]), (2, 1, [8])]


def test_addresses():
    w = [torch.arange(24.0).view(8, 3) + 100 * i for i in range(2)]
    blocks = ops.RowBlocks(w, 2, [4, 0])
    assert len(blocks) == 4 and [b.tolist() for b in blocks] == [t[at:at + 2].tolist() for at in (4, 0) for t in w]
    assert [b.data_ptr() for b in blocks] == [t.data_ptr() + at for at in blocks.offsets() for t in w]
    assert not ops.aligned16(ops.RowBlocks([torch.zeros(8, 3)], 1, [0, 1])) and ops.aligned16(ops.RowBlocks([torch.zeros(8, 4)], 1, [0, 1]))


@pytest.mark.parametrize("cls", [dion.Muon, dion.NorMuon])
@pytest.mark.parametrize("split,calls", [
    ((64,) * 36, [(2, 36, 64)]), ((100, 25, 25), [(2, 1, 100), (2, 2, 25)]), ((8, 4) * 10, [(20, 1, 8), (20, 1, 4)]),
    ((8, 4) * 2049, [(2, 1, 8 * 2049 + 4 * 2049)]), ((1,) * 16385, [(2, 1, 16385)]),  # past one call: stacked
])
def test_addresses_a_step_hands_over(cls, split, calls, monkeypatch):
    params = [torch.nn.Parameter(torch.zeros(sum(split), 4)) for _ in range(2)]
    for p in params:
        p.grad = torch.zeros_like(p)
    opt = cls([{"params": params, "split_sizes": split}])
    seen = []

    def phases(group, X, G, M, V, shape, mats, rows, cols, ratio_shape, split_sizes, block_scale=1.0):
        seen.append((len(X), mats, rows))
        assert len(G) == len(M) == len(X) and (V is None or len(V) == len(X)) and cols == 4
        assert (split_sizes is not None) == (len(split) > 4096) and tuple(ratio_shape) == (rows, cols)
        return iter(())

    monkeypatch.setattr(opt, "_matrix_phases", phases)
    opt.step()
    assert seen == calls
