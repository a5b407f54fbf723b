"""``split_sizes``: all row blocks of a weight are in one shape group, which runs on one stream.  State that is missing (cleared,
or not in the loaded checkpoint) is made by the group that first needs it, so a second group of the same weight on another
stream could read it before it is cleared, or have it cleared after its update."""
import pytest
import torch

import dion


@pytest.mark.parametrize("lost", ["nothing", "all of it", "second moments"])
@pytest.mark.parametrize("cls", [dion.Muon, dion.NorMuon])
def test_a_weight_is_in_one_shape_group(cls, lost):
    fused, plain = [torch.nn.Parameter(torch.randn(150, 100)) for _ in range(2)], torch.nn.Parameter(torch.randn(100, 100))
    groups = lambda: [{"params": fused, "split_sizes": (100, 25, 25)}, {"params": [plain]}]  # noqa: E731
    opt = cls(groups())
    if lost == "all of it":
        opt.state.clear()
    elif lost == "second moments":
        saved = opt.state_dict()
        opt.load_state_dict({**saved, "state": {i: {"momentum": s["momentum"]} for i, s in saved["state"].items()}})
    for p in (*fused, plain):
        p.grad = torch.ones_like(p)
    seen = []
    opt._run_shape_groups = lambda work: seen.extend(id(p) for entry in work for p in entry[1])
    opt.step()
    assert sorted(seen) == sorted(id(p) for p in (*fused, plain))


@pytest.mark.gpu
@pytest.mark.parametrize("cls", [dion.Muon, dion.NorMuon])
@pytest.mark.parametrize("split", [(1000, 250, 250), (100, 25, 25), (512, 128, 128)])
def test_missing_state_is_fresh_state(cls, split):
    g = torch.Generator(device="cuda").manual_seed(sum(split))
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g) * 0.02  # noqa: E731
    start, grads = [rand(sum(split), 200) for _ in range(2)], [rand(sum(split), 200) for _ in range(2)]
    got = []
    for lose in (lambda o: None, lambda o: o.state.clear(), lambda o: o.load_state_dict({**o.state_dict(), "state": {}})):
        params = [torch.nn.Parameter(w.clone()) for w in start]
        opt = cls([{"params": params, "split_sizes": split}], lr=0.02)
        lose(opt)
        for p, d in zip(params, grads):
            p.grad = d.mT.contiguous().mT  # a gradient that is not contiguous is copied
        opt.step()
        got.append([p.data for p in params] + [t for p in params for t in opt.state[p].values()])
    for other in got[1:]:
        assert len(other) == len(got[0]) and all(torch.equal(a, b) for a, b in zip(got[0], other))
