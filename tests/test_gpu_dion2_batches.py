"""The selection of the k largest around the counts of keys a thread holds: exact against the definition."""
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
