"""Dion2's streaming kernels around the batches a thread loads at once, and the selection of the k largest around the
counts of keys a thread holds: exact against the definition, element by element."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dim", [1, 63, 64, 1023, 1024, 1025, 2048, 2049, 4097, 8192, 8193, 20000])
@pytest.mark.parametrize("values", ["close", "ties", "specials"])
def test_k_largest(dim, values):
    """The k first entries of a stable descending sort (ties to the lower index, NaN as +inf), ascending."""
    from dion_amd import _lib

    lib = _lib.load()
    g = torch.Generator().manual_seed(dim)
    n = 3
    v = 10.0 + 0.1 * torch.randn(n, dim, generator=g)
    if values == "ties":
        v = torch.randint(0, 3, (n, dim), generator=g).float()
    elif values == "specials":
        pick = torch.randint(0, 12, (n, dim), generator=g)
        for code, x in enumerate((float("nan"), float("inf"), 0.0, -0.0, 1e-42, 3e38)):
            v[pick == code] = x
    order = torch.nan_to_num(v, nan=float("inf"), posinf=float("inf")).sort(dim=-1, descending=True, stable=True).indices
    vd = v.to(DEV)
    for k in sorted({0, 1, dim // 4, dim // 2 + 1, dim - 1, dim}):
        idx = torch.full((n, k + 1), -7, dtype=torch.int32, device=DEV)  # the last column stays untouched
        imap = torch.full((n, dim), -7, dtype=torch.int32, device=DEV)
        flat = idx.flatten()[: n * k + 1]
        _lib.check(lib.dion_dion2_topk(vd.data_ptr(), n, dim, k, flat.data_ptr(), imap.data_ptr(),
                                       torch.cuda.current_stream().cuda_stream), "topk")
        ref = order[:, :k].sort(-1).values.to(torch.int32)
        inv = torch.full((n, dim), -1, dtype=torch.int32)
        inv.scatter_(1, ref.long(), torch.arange(k, dtype=torch.int32).expand(n, k).contiguous())
        assert torch.equal(flat[: n * k].view(n, k).cpu(), ref) and int(flat[n * k]) == -7
        assert torch.equal(imap.cpu(), inv)


@pytest.mark.parametrize("sdt,gdt", [(torch.float32, torch.bfloat16), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("n,rows,cols,sd", [
    (2, 5, 64 * 16 + 64 * 4 + 9, -2), (2, 9, 1023, -2), (1, 3, 1, -2), (2, 33, 64, -2),
    (2, 131, 36, -1), (1, 517, 260, -1), (2, 7, 8, -1), (3, 66, 5, -1),
    (1, 9, 4 * 2052, -1), (1, 5, 4 * 8196, -1), (1, 3, 4 * 16388, -1),  # fewer and fewer rows per workgroup
    (9, 2048, 4096, -2), (9, 4100, 2048, -1)])  # the last two: past the caches at either dtype
def test_accumulate_select_and_update(n, rows, cols, sd, sdt, gdt):
    """M + G, its slice norms, the selection and the update, against the same arithmetic in torch.  Norms: fp32 sums of
    L non-negative terms are within L * 2^-24 of the exact sum (relative)."""
    from dion_amd import ops

    gen = torch.Generator(device=DEV).manual_seed(rows)
    mk = lambda *s, dt: (torch.randn(*s, device=DEV, generator=gen) * 0.1).to(dt)  # noqa: E731
    G, M, X = ([mk(1, rows, cols, dt=dt) for _ in range(n)] for dt in (gdt, sdt, sdt))
    dim, length = (rows, cols) if sd == -2 else (cols, rows)
    k = max(1, dim // 4)
    ref_m = [(m.float() + g.float()).to(sdt) for m, g in zip(M, G)]
    U, idx, imap = ops.dion2_select(G, M, k, sd, 0.5)
    lr, wd, ratio = torch.tensor(0.25, device=DEV), 0.5, 1.5
    O = mk(*U.shape, dt=torch.bfloat16)
    Xr = [x.clone() for x in X]
    ops.dion2_post(X, O, imap, lr, ratio, wd, sd)
    a, b = torch.tensor(0.875, device=DEV, dtype=torch.float64), torch.tensor(0.375, device=DEV)
    for i in range(n):
        sel = idx[i].long()
        norms = ref_m[i][0].double().abs().sum(-1 if sd == -2 else -2)
        chosen = torch.zeros(dim, dtype=torch.bool, device=DEV)
        chosen[sel] = True
        if k < dim:
            assert float(norms[~chosen].max()) <= float(norms[chosen].min()) * (1 + 2 * length * 2.0 ** -24)
        assert torch.equal(imap[i][sel], torch.arange(k, dtype=torch.int32, device=DEV))
        picked = ref_m[i][0].index_select(0 if sd == -2 else 1, sel)
        assert torch.equal(U[i, 0], picked.to(torch.bfloat16))
        decayed = ref_m[i][0].clone()
        decayed.index_copy_(0 if sd == -2 else 1, sel, (picked.float() * 0.5).to(sdt))
        assert torch.equal(M[i][0], decayed)
        full = torch.zeros(rows, cols, device=DEV)
        full.index_copy_(0 if sd == -2 else 1, sel, b * O[i, 0].float())
        exact = a * Xr[i][0].double() - full.double()  # exact in float64 but for its last bits: one rounding to fp32
        assert torch.equal(X[i][0], exact.float().to(sdt))
