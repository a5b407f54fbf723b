"""The one-workgroup-per-matrix kernel (X in registers) at the edges of its row tiles, column groups and wavefront counts,
tall and wide, at every alignment.  The reference is float64; the bound is the error of the same iteration carried out
with torch in float32 with A, B and X rounded to bf16 where the kernel rounds them (factor 1.5: the sums run in another
order; the scaled X too, which the forms beyond 64 x 1024 leave unrounded: test_the_norm_is_no_rounding_of_its_own)."""
import pytest
import torch

from dion_amd import newton_schulz as ns
from dion_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
CO = ns.POLAR_EXPRESS_COEFFS


def _iterate(G, coeffs, round_):
    X = G.mT.contiguous() if G.shape[-2] > G.shape[-1] else G
    X = round_(X / (X.flatten(1).norm(dim=1)[:, None, None] * 1.02 + 1e-6))
    for a, b, c in coeffs:
        A = round_(X @ X.mT.contiguous())
        B = round_(b * A + c * (A @ A) + a * torch.eye(A.shape[-1], device=DEV, dtype=A.dtype))
        X = round_(B @ X)
    return X.mT if G.shape[-2] > G.shape[-1] else X


def _check(G, n_iters):
    O = ops.ns_orthogonalize(G, CO[:n_iters], 1.02, 1e-6)
    assert torch.equal(O, ops.ns_orthogonalize(G, CO[:n_iters], 1.02, 1e-6))
    exact = _iterate(G.bfloat16().double(), CO[:n_iters], lambda t: t)
    same = _iterate(G.bfloat16().float(), CO[:n_iters], lambda t: t.bfloat16().float())
    err = lambda t: float((t.double() - exact).norm() / exact.norm())
    assert err(O) <= 1.5 * err(same) + 1e-4, (err(O), err(same))


# short sides: edges of 32-row pairs of tiles; long sides: edges of 32-column groups, of 4 and 8 wavefronts' shares and of
# every compiled group count
SHAPES = [(1, 1, 1), (2, 1, 33), (3, 16, 16), (2, 17, 100), (2, 31, 257), (1, 32, 1024), (3, 33, 40), (2, 48, 255),
          (2, 63, 512), (2, 64, 513), (1, 64, 769), (2, 64, 1023),                          # any batch
          (260, 32, 129), (257, 20, 640), (300, 30, 1000), (260, 64, 64), (257, 64, 257), (260, 50, 768), (270, 64, 776),
          (16, 32, 1025), (17, 5, 4096), (16, 64, 1025), (16, 60, 1536), (16, 64, 1544), (17, 64, 2048),
          (16, 65, 256), (20, 72, 513), (16, 96, 768), (16, 90, 1024), (17, 96, 1280),
          (16, 97, 256), (18, 128, 512), (16, 120, 520), (16, 128, 769), (17, 128, 1024)]


@pytest.mark.parametrize("tall", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
def test_against_float64(shape, tall):
    b, m, n = shape
    g = torch.Generator(device=DEV).manual_seed(m * 5000 + n)
    G = torch.randn((b, n, m) if tall else (b, m, n), device=DEV, generator=g).mul_(0.02).bfloat16()
    _check(G, 5)


@pytest.mark.parametrize("n_iters", [0, 1, 3])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(3, 64, 768), (3, 768, 64), (300, 48, 200), (16, 128, 264), (16, 300, 100)])
@pytest.mark.parametrize("offset", [0, 1])
def test_iterations_dtypes_and_alignment(shape, dtype, n_iters, offset):
    numel = shape[0] * shape[1] * shape[2]
    g = torch.Generator(device=DEV).manual_seed(numel)
    flat = torch.randn(numel + offset, device=DEV, generator=g).mul_(0.02).to(dtype)
    _check(flat[offset:].view(shape), n_iters)


@pytest.mark.parametrize("shape", [(3, 63, 100), (3, 100, 63), (16, 72, 264), (2, 64, 256)])
def test_nothing_is_written_beside_the_result(shape):
    import ctypes

    from dion_amd import _lib
    b, r, c = shape
    lib = _lib.load()
    g = torch.Generator(device=DEV).manual_seed(1)
    G = torch.randn(shape, device=DEV, generator=g).bfloat16()
    want = ns.polar_express(G)
    for offset in (128, 129):
        n = b * r * c
        buf = torch.full((n + 256,), 3.0, device=DEV, dtype=torch.bfloat16)
        flat = [x for co in CO for x in co]
        _lib.check(lib.dion_ns_orthogonalize(G.data_ptr(), 0, buf[offset:].data_ptr(), b, r, c,
                                             (ctypes.c_float * 15)(*flat), 5, ns.POLAR_EXPRESS_SAFETY, 1e-6, 0, 0, None, 0,
                                             torch.cuda.current_stream().cuda_stream), "ns")
        assert torch.equal(buf[offset:offset + n].view(shape), want)
        assert bool((buf[:offset] == 3).all()) and bool((buf[offset + n:] == 3).all())


def _decaying(b, m, n, tall, seed):
    """Matrices whose singular values fall over 2.5 decades, as a gradient's do."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    Q = torch.linalg.qr(torch.randn(m, m, device=DEV, generator=g))[0] * torch.logspace(0, -2.5, m, device=DEV)
    G = Q @ torch.randn(b, m, n, device=DEV, generator=g).mul_(0.02)
    return (G.mT if tall else G).contiguous().bfloat16()


@pytest.mark.parametrize("tall", [False, True])
@pytest.mark.parametrize("shape", [(16, 128, 256), (24, 128, 1024), (17, 96, 1280), (260, 96, 512), (24, 64, 1536), (17, 64, 2048), (24, 32, 2048), (16, 32, 4096)])
def test_the_norm_is_no_rounding_of_its_own(shape, tall):
    """Shapes that single matrices run on the GEMMs: the distance to float64 is that of the iteration whose first products take
    the values as they came (rounded to bf16 once), A, B and X rounded once per iteration.  Sums in another order move single roundings, and with them a
    distance over this many elements by a few per cent; X rounded once more after the scaling is 1.3 to 1.4 times as far."""
    b, m, n = shape
    G = _decaying(b, m, n, tall, m + n)
    exact = _iterate(G.bfloat16().double(), CO, lambda t: t)
    to_bf16 = lambda t: t.bfloat16().float()
    first = []  # the first value _iterate rounds is the scaled X
    round_ = lambda t: to_bf16(t) if first else (first.append(1), t)[1]
    err = lambda t: float((t.double() - exact).norm() / exact.norm())
    as_it_came, rounded = err(_iterate(G.float(), CO, round_)), err(_iterate(G.float(), CO, to_bf16))
    got = err(ops.ns_orthogonalize(G, CO, 1.02, 1e-6))
    print(f"{shape} {tall}: {got:.3e}, emulated {as_it_came:.3e}, with X rounded again {rounded:.3e}")
    assert got <= 1.1 * as_it_came


@pytest.mark.parametrize("tall", [False, True])
@pytest.mark.parametrize("exponent", [-58, -46, -34, -20, 20, 34, 46, 54])
def test_inputs_of_any_magnitude(exponent, tall):
    """The scale of the input cancels: powers of two on both sides of where the factor moves from the sums into X (squared
    norms of 2^-80 and 2^80), with the bound of the iteration that rounds the scaled X."""
    g = torch.Generator(device=DEV).manual_seed(7)
    G = torch.randn((24, 256, 128) if tall else (24, 128, 256), device=DEV, generator=g).bfloat16()
    O = ops.ns_orthogonalize(torch.ldexp(G.float(), torch.tensor(exponent, device=DEV)).bfloat16(), CO, 1.02, 0.0)
    exact = _iterate(G.double(), CO, lambda t: t)
    same = _iterate(G.float(), CO, lambda t: t.bfloat16().float())
    err = lambda t: float((t.double() - exact).norm() / exact.norm())
    assert err(O) <= 1.5 * err(same) + 1e-4, (err(O), err(same))


def test_a_norm_past_the_range_of_fp32_gives_zeros():
    """X / (inf * s + eps)."""
    G = torch.full((24, 128, 256), 2.0 ** 64, device=DEV).bfloat16()
    assert not bool(ops.ns_orthogonalize(G, CO, 1.02, 1e-6).any())


@pytest.mark.parametrize("shape", [(100, 64, 768), (100, 128, 1024)])
def test_no_workspace_is_allocated(shape):
    ops.release_workspaces()
    G = torch.randn(shape, device=DEV).bfloat16()
    ns.polar_express(G)
    assert not ops._workspaces
    X = [torch.zeros(shape[1:], device=DEV) for _ in range(shape[0])]
    ops.ns_orthogonalize_update(G, X, CO, 1.02, 1e-6, torch.tensor(0.1, device=DEV), 1.0, 0.0)
    assert [w.numel() for w in ops._workspaces.values()] == [G.numel() * 2]
    assert torch.equal(torch.stack(X), -0.1 * ns.polar_express(G).float())
