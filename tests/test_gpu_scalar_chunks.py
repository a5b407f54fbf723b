"""AdamW / Lion over tensors around the run a workgroup owns (8192 elements), past it by a few elements, empty and
unaligned ones in between, and with enough bytes for the non-temporal form: the result of one call over the whole list
equals, bit for bit, the same elements updated as many short tensors (the element-wise path)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _update(kind, X, G, M, V, steps, lr):
    from dion_amd import ops

    if kind == "adamw":
        ops.adamw_step(X, G, M, V, steps, lr, 0.9, 0.95, 0.01, 1e-8, True)
    else:
        ops.lion_step(X, G, M, lr, 0.9, 0.95, 0.01, True)


@pytest.mark.parametrize("kind", ["adamw", "lion"])
@pytest.mark.parametrize("sdt,gdt", [(torch.float32, torch.bfloat16), (torch.bfloat16, torch.bfloat16),
                                     (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("sizes", [[1, 8191, 0, 8192, 8193, 4096, 3 * 8192 + 5], [8192 * 12, 0, 2], [40_000_003]])
def test_runs_and_rests(kind, sdt, gdt, sizes):
    g = torch.Generator(device=DEV).manual_seed(3)
    lr = torch.tensor(1e-2, device=DEV)
    mk = lambda n, dt, s=1.0: (torch.randn(n, device=DEV, generator=g) * s).to(dt)  # noqa: E731
    X, G, M = ([mk(n, dt) for n in sizes] for dt in (sdt, gdt, sdt))
    V = [mk(n, sdt).abs() for n in sizes]
    st = [torch.full((), 3.0, device=DEV) for _ in sizes]
    # a copy cut into pieces of 1023 elements where that is feasible, else into unaligned halves
    Xc, Mc, Vc = ([t.clone() for t in ts] for ts in (X, M, V))
    cut = lambda t: list(t.split(1023 if t.numel() < 200_000 else t.numel() // 2 + 1)) if t.numel() else []  # noqa: E731
    _update(kind, X, G, M, V, st, lr)
    assert all(float(s) == (4.0 if kind == "adamw" else 3.0) for s in st)
    for x, gr, m, v in zip(Xc, G, Mc, Vc):
        parts = [cut(t) for t in (x, gr, m, v)]
        for lo in range(0, len(parts[0]), 48):
            _update(kind, *(p[lo:lo + 48] for p in parts),
                    [torch.full((), 3.0, device=DEV) for _ in parts[0][lo:lo + 48]], lr)
    for a, b in zip(X + M + (V if kind == "adamw" else []), Xc + Mc + (Vc if kind == "adamw" else [])):
        assert torch.equal(a, b)


@pytest.mark.parametrize("kind", ["adamw", "lion"])
@pytest.mark.parametrize("sdt,gdt", [(torch.float32, torch.bfloat16), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("sizes", [[1, 1023, 0, 1024, 1025, 3 * 1024 + 5], [(1 << 20) - 1], [(1 << 20) - 4095, 2047, 2048, 2049, 0, 7],
                                   [(5 << 20) - 8192, 8191], [(5 << 20) - 8192, 8192, 8193, 3]])
def test_short_runs_and_rests(kind, sdt, gdt, sizes):
    """The same at the edges of the short runs (1024, 2048 elements) and of the launch sizes that take them."""
    test_runs_and_rests(kind, sdt, gdt, sizes)
