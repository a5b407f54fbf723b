"""dion2_select into the padded form: same selection and momentum as the plain call bit for bit, the same block with zeros around
it, partial sums per 64 x 64 tile; and a Dion2 / NorDion2 step that takes it, against the step that pads in a pass of its own."""
import pytest
import torch

import dion
from dion_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rand(shape, seed, dtype=torch.float32):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(shape, device=DEV, generator=g) * 0.02).to(dtype)


@pytest.mark.parametrize("mdtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,cols,k,offset", [
    (256, 328, 200, 0),    # eight elements a lane
    (300, 330, 75, 0),     # two
    (131, 257, 33, 0),     # one
    (256, 328, 200, 1),    # unaligned momentum
    (600, 200, 300, 0),    # a tall block: transposed
    (601, 203, 300, 3),
    (192, 192, 192, 0),    # everything
    (129, 129, 1, 0),      # one row
])
def test_select_into_the_padded_form(rows, cols, k, offset, mdtype):
    n, mats, select_dim = 2, 2, -2

    def tensors(seed, dtype):
        out = []
        for i in range(n):
            flat = torch.zeros(mats * rows * cols + 8, device=DEV, dtype=dtype)
            t = flat[offset:offset + mats * rows * cols].view(mats, rows, cols)
            out.append(t.copy_(_rand((mats, rows, cols), seed + i)))
        return out

    G, Ma, Mb = tensors(1, torch.bfloat16), tensors(11, mdtype), tensors(11, mdtype)
    sr, sc = k, cols
    lo, hi = min(sr, sc), max(sr, sc)
    extents = (-(-lo // 128) * 128, -(-hi // 128) * 128)
    want, idx_a, map_a = ops.dion2_select(G, Ma, k, select_dim, 0.9)
    U, idx_b, map_b, sumsq = ops.dion2_select(G, Mb, k, select_dim, 0.9, extents=extents)
    assert torch.equal(idx_a, idx_b) and torch.equal(map_a, map_b)
    assert all(torch.equal(a, b) for a, b in zip(Ma, Mb))
    want = want.reshape(n * mats, sr, sc)
    full = torch.zeros(n * mats, *extents, device=DEV, dtype=torch.bfloat16)
    full[:, :lo, :hi] = want.mT if sr > sc else want
    assert torch.equal(U, full)
    tiles = full.double().view(n * mats, extents[0] // 64, 64, extents[1] // 64, 64).pow(2).sum(dim=(2, 4)).flatten(1)
    # float32 sums of 4096 squares in chains of at most 16 and a tree: under 32 roundings of 2^-24 each
    assert sumsq.shape == tiles.shape and bool(((sumsq.double() - tiles).abs() <= 32 * 2.0 ** -24 * tiles).all())


# (Dion2 selects rows of matrices that are no taller than wide, NorDion2 always; the last block is a tall one, 600 x 300)
@pytest.mark.parametrize("cls,shape", [
    (dion.Dion2, (600, 900)), (dion.Dion2, (768, 1000)), (dion.Dion2, (1100, 1100)),
    (dion.NorDion2, (600, 900)), (dion.NorDion2, (900, 600)), (dion.NorDion2, (2304, 768)), (dion.NorDion2, (768, 1000)),
    (dion.NorDion2, (1100, 1100)), (dion.NorDion2, (2400, 300)),
])
def test_step_is_the_unprepared_one(cls, shape, monkeypatch):
    select, forms = ops.dion2_select, []

    def seen(*args, **kw):
        forms.append(kw.get("extents"))
        return select(*args, **kw)

    monkeypatch.setattr(ops, "dion2_select", seen)
    got = []
    for handed_over in (True, False):
        params = [torch.nn.Parameter(_rand(shape, i)) for i in range(3)]
        opt = cls(params, lr=0.02, weight_decay=0.01)
        opt.prepared_input = handed_over
        for step in range(2):
            for i, p in enumerate(params):
                p.grad = _rand(shape, 50 + 10 * step + i)
            opt.step()
        got.append([p.data for p in params] + [opt.state[p]["momentum"] for p in params])
    assert all(forms[:2]) and forms[2:] == [None, None]  # the padded gather in both steps of the first run, in none of the second
    assert all(torch.equal(a, b) for a, b in zip(*got))
