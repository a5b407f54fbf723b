"""NorMuon's second moments under ``split_sizes`` are those of the block as it is rescaled by the ratio of its lr to the whole
weight's, whichever way the step goes: row blocks updated where they lie, or stacked for a caller's orthogonalization.  State is
interchangeable between the two, and with checkpoints of either."""
import pytest
import torch

from dion import NorMuon
from dion_amd import newton_schulz as ns
from dion_amd import ops
from dion_amd.optim_base import split_lr_scales

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _weights(split, cols, dtype, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    rand = lambda *s: torch.randn(*s, device=DEV, generator=g)  # noqa: E731
    w, d = [(rand(sum(split), cols) * 0.02).to(dtype) for _ in range(2)], [(rand(sum(split), cols) * 0.02).to(dtype) for _ in range(2)]
    return w, d, [(0.5 + rand(sum(split), 1).abs()).to(dtype) / cols for _ in range(2)]


@pytest.mark.parametrize("adjust", ["spectral_norm", "rms_norm", None])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("split,cols", [((1000, 250, 250), 1000), ((100, 25, 25), 96), ((256, 128, 128), 256), ((64,) * 6, 128)])
def test_state_of_a_run_continues_either_way(split, cols, dtype, adjust):
    """Bounds.  Stacked, the rescaled block is rounded to bf16 once more (2^-8 of an element at most, either way, so less of a mean
    of squares) and the norm is summed in another order (a few more elements rounded the other way); a bf16 state is rounded on
    each side, 2 x 2^-8.  Half the relative error of a second moment enters the update, beside the rounding of its elements."""
    start, grads, var = _weights(split, cols, dtype, sum(split) + cols)
    got = []
    for func in (None, lambda G, epsilon: ns.polar_express(G, epsilon=epsilon)):
        params = [torch.nn.Parameter(w.clone()) for w in start]
        opt = NorMuon([{"params": params, "split_sizes": split}], lr=0.5, weight_decay=0.0, adjust_lr=adjust,
                      newton_schulz_func=func)
        for p, d, v in zip(params, grads, var):
            opt.state[p]["variance_neuron"].copy_(v)
            p.grad = d
        opt.step()
        got.append([(p.data.float() - w.float(), opt.state[p]["variance_neuron"].float()) for p, w in zip(params, start)])
    own = 0.0 if dtype == torch.float32 else 2.0 ** -7
    for (da, va), (db, vb) in zip(*got):
        assert bool(((va - vb).abs() <= (2.0 ** -7 + own) * vb).all())
        # (the weight is rounded to its type on each side)
        steps = 0.0 if dtype == torch.float32 else 2.0 ** -7 * float(torch.stack(start).float().norm())
        assert float((da - db).norm()) <= 2.0 ** -6 * float(db.norm()) + steps


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,cols", [(1, 5), (250, 1000), (67, 129)])
def test_scaled_statistics(rows, cols, dtype):
    """What the statistics of the multiplied block are in float64: sums of at most 1000 squares and 20 roundings after them."""
    g = torch.Generator(device=DEV).manual_seed(rows * cols)
    U = (torch.randn(3, 2, rows, cols, device=DEV, generator=g) * 0.05).bfloat16()
    V = [(torch.rand(2, rows, 1, device=DEV, generator=g) * 0.01).to(dtype) for _ in range(3)]
    for scale in split_lr_scales((1, 3), (4, 7), "spectral_norm"):
        got, new = [v.clone() for v in V], []
        row_scale = ops.normuon_stats(U, got, 0.9, scale).view(3, 2, rows, 1)
        for u, v, have, rs in zip(U.double() * scale, V, got, row_scale.double()):
            want = torch.lerp(v.double(), u.pow(2).mean(-1, keepdim=True), 1 - 0.9)
            tol = 2.0 ** -18 + (0.0 if dtype == torch.float32 else 2.0 ** -8)
            assert bool(((have.double() - want).abs() <= tol * want).all())
            d = have.double().sqrt() + 1e-8
            rs_want = 1 / d * (u.pow(2).sum((-1, -2), keepdim=True) / (u / d).pow(2).sum((-1, -2), keepdim=True)).sqrt()
            assert bool(((rs - rs_want).abs() <= 2.0 ** -18 * rs_want).all())
            new.append(have)
