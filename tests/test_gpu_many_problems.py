"""Several orthogonalizations in one call whose products share launches (``ops.ns_orthogonalize_many``): every problem has
the bits of its own call, on every kernel that takes several products -- the comments name what the joined launches run on --
with problems of different reduction lengths, pitches and numbers of tiles side by side, in every form."""
import pytest
import torch

from dion_amd import newton_schulz as ns
from dion_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"

BUNDLES = [
    [(1, 128, 128), (1, 128, 384)],                                            # 64-wide tiles throughout
    [(2, 192, 768), (3, 256, 1024), (1, 768, 768)],                            # 64-wide, B X on 128-wide ones
    [(12, 250, 1000), (6, 1000, 1000)],                                        # 64- and 128-wide, padded
    [(4, 640, 640), (3, 768, 2304)],                                           # 128-wide, four slots
    [(12, 640, 640), (12, 768, 768), (2, 1024, 256), (5, 384, 512)],           # two slots
    [(12, 768, 768), (12, 768, 2304), (12, 3072, 768), (12, 768, 3072)],       # two slots, B X walking 256-wide tiles
    [(20, 512, 512), (40, 512, 1024), (3, 1024, 1024), (1, 256, 4096)],        # walking: one tile to a member's last walker
    [(40, 1024, 1024), (24, 512, 1024)],                                       # symmetric products on 256-wide tiles
    [(3, 2304, 2304), (3, 2560, 2560)],                                        # B X on 256-wide tiles, one workgroup each
    [(2, 300, 300), (9, 128, 640), (2, 65, 1030), (1, 700, 130), (4, 256, 300), (1, 130, 140), (2, 1000, 999), (3, 512, 512)],
]


def _rand(shape, seed, dtype=torch.bfloat16):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(shape, device=DEV, generator=g) * 0.02).to(dtype)


def _own(G, func):
    return func(G)


@pytest.mark.parametrize("func", [ns.zeropower_via_newtonschulz5, ns.gram_newton_schulz])
@pytest.mark.parametrize("bundle", range(len(BUNDLES)))
def test_plain_problems(bundle, func):
    Gs = [_rand(s, 100 * bundle + i, torch.float32 if i == 1 else torch.bfloat16) for i, s in enumerate(BUNDLES[bundle])]
    want = [func(G) for G in Gs]
    got = ns.run_many([ns.Problem(func, G, None, G.shape[1], G.shape[2], 1e-7) for G in Gs])
    for s, a, b in zip(BUNDLES[bundle], got, want):
        assert torch.equal(a, b), s


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("bundle", [2, 3, 5, 9])
def test_updates_of_prepared_and_padded_problems(bundle, dtype):
    func, lr = ns.polar_express, torch.tensor(0.02, device=DEV)
    made, want = [], []
    for i, (b, r, c) in enumerate(BUNDLES[bundle]):
        G, M = [_rand((r, c), 7 * i + k) for k in range(b)], [torch.zeros(r, c, device=DEV, dtype=dtype) for _ in range(b)]
        X = [_rand((r, c), 70 * i + k, dtype) for k in range(b)]
        extents = ns.padded_extents(func, b, r, c)
        if extents is None and not ns.accepts_prepared(func, b, r, c):
            continue  # the kernel of one workgroup a matrix
        args = (G, M, 0.9, False, 1, r, c)
        U, sq = ops.muon_pre_prepared(*args) if extents is None else ops.muon_pre_padded(*args, extents)
        update = (lr, 0.7, 0.01, i % 2 == 1)
        Y = [x.clone() for x in X]
        ns.orthogonalize_update_prepared(func, U.clone(), sq, r, c, 1e-7, Y, *update, padded=extents is not None)
        want.append(Y)
        made.append((ns.Problem(func, U, sq, r, c, 1e-7, extents is not None, (X, *update)), X))
    assert len(made) >= 2
    assert ns.run_many([p for p, _x in made]) == [None] * len(made)
    for (_p, X), Y in zip(made, want):
        assert all(torch.equal(x, y) for x, y in zip(X, Y))
