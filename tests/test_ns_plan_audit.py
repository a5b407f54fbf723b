"""Host-only walk over the launch lists of the orthogonalization driver (no GPU, no device work).

dion_ns_orthogonalize plans a call first -- workspace layout and every kernel launch with its operands
-- and checks the list against the buffers the call owns before the first launch.  This test runs
that planner and checker through dion_ns_plan_audit for every shape of the benchmark configurations
(wide, tall, padded, per-head, Dion2 sub-matrices), every schedule length, Gram on and off and the
fused-update form: each launch must read inside {input, workspace} and write inside {workspace,
output, parameter}, with tile shapes that divide the padded extents.  It also shows the check has
teeth: the same plans audited against a workspace that is too short must be refused, naming the
launch and the operand."""
import os

import pytest

from dion_amd import _lib

pytestmark = pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH), reason="libdion_hip.so not built in this checkout")

BF16, F32, GRAM = _lib.DION_BF16, _lib.DION_F32, _lib.DION_NS_GRAM

# (batch, rows, cols) of every shape group of the benchmark configurations, plus ragged ones
CONFIG_SHAPES = [
    (1, 768, 3072),                                                            # one matrix
    (12, 2304, 768), (12, 768, 768), (12, 3072, 768), (12, 768, 3072),         # GPT-small
    (432, 64, 768),                                                            # per-head (LDS-resident kernel)
    (24, 6144, 2048), (24, 2048, 2048), (24, 8192, 2048), (24, 2048, 8192),    # GPT-1.3B
    (24, 6144, 512), (24, 512, 2048), (24, 8192, 512), (24, 512, 8192),        # Dion2 sub-matrices, fraction 0.25
    (64, 4096, 4096), (64, 1024, 4096), (64, 14336, 4096), (32, 4096, 14336),  # Llama-3-8B
    (8, 4096, 4096), (8, 1024, 4096), (8, 14336, 4096), (4, 4096, 14336),      # one GPU's share of eight
]
RAGGED_SHAPES = [(3, 256, 512), (3, 512, 256), (3, 128, 128), (3, 100, 36), (1, 17, 33), (2, 48, 1000), (2, 1000, 130),
                 (5, 768, 64), (2, 100, 200), (3, 100, 300), (1, 200, 136), (7, 65, 65), (2, 129, 257), (1, 1, 1),
                 (300, 72, 80)]


def _audit(lib, shape, n_iters=5, flags=0, in_dtype=BF16, with_update=0, x_dtype=F32, mats_per_ptr=1, ws=0, reset=2):
    b, r, c = shape
    return lib.dion_ns_plan_audit(b, r, c, in_dtype, n_iters, flags, reset, with_update, x_dtype, mats_per_ptr, ws)


@pytest.mark.parametrize("shape", CONFIG_SHAPES + RAGGED_SHAPES)
def test_every_launch_stays_inside_the_calls_buffers(shape):
    lib = _lib.load()
    b, r, c = shape
    small = min(r, c) <= 64
    for flags in (0, GRAM):
        for n_iters in (0, 1, 5):
            for in_dtype in (BF16, F32):
                n = _audit(lib, shape, n_iters, flags, in_dtype)
                assert n > 0, (shape, flags, n_iters, lib.dion_last_error().decode())
                if small:
                    assert n == 1  # one LDS-resident launch
                elif not flags or max(r, c) < 3 * min(r, c):
                    # norm + prepare + three GEMMs per iteration (+ unpad when padding is in the way); a wide
                    # bf16 input that fills whole tiles is read where it lies: no prepare pass
                    in_place = (in_dtype == BF16 and r <= c and n_iters > 0
                                and bool(lib.dion_ns_accepts_prepared(b, r, c, flags, n_iters)))
                    want = (1 + 3 * n_iters,) if in_place else (2 + 3 * n_iters, 3 + 3 * n_iters)
                    assert n in want, (shape, n_iters, in_dtype, n)
                else:
                    assert n >= 2 + n_iters


@pytest.mark.parametrize("shape", [s for s in CONFIG_SHAPES if min(s[1:]) > 64 and s[1] % 128 == 0 and s[2] % 128 == 0])
def test_fused_update_launches_stay_inside_the_parameters(shape):
    lib = _lib.load()
    b = shape[0]
    for x_dtype in (F32, BF16):
        for flags in (0, GRAM):
            for mpp in sorted({1, 2 if b % 2 == 0 else 1, b}):
                n = _audit(lib, shape, 5, flags, BF16, with_update=1, x_dtype=x_dtype, mats_per_ptr=mpp)
                assert n > 0, (shape, flags, mpp, lib.dion_last_error().decode())
    # more than 64 parameters: the last GEMM is split into launches of 64 pointers each
    n1 = _audit(lib, (shape[0], shape[1], shape[2]), 5, 0, BF16, with_update=1)
    in_place = shape[1] <= shape[2] and bool(lib.dion_ns_accepts_prepared(b, shape[1], shape[2], 0, 5))
    assert n1 == (1 if in_place else 2) + 3 * 4 + 2 + (b + 63) // 64  # norm (+ prepare), 4 iterations, A, B, last X' 


def test_padded_shapes_do_not_take_the_fused_update():
    lib = _lib.load()
    for shape in [(3, 100, 300), (5, 768, 64), (432, 64, 768)]:
        assert _audit(lib, shape, 5, 0, BF16, with_update=1) == -1
        assert "does not take the fused update" in lib.dion_last_error().decode()


@pytest.mark.parametrize("shape", [(1, 768, 3072), (12, 2304, 768), (3, 512, 256), (3, 100, 300), (2, 1000, 130),
                                   (32, 4096, 14336)])
def test_a_short_workspace_is_caught_launch_by_launch(shape):
    lib = _lib.load()
    for flags in (0, GRAM):
        total = lib.dion_ns_workspace_bytes(*shape, flags)
        assert _audit(lib, shape, 5, flags, ws=total) > 0
        # short by the last buffer of the layout (the reciprocal norms, one 256-byte slot)
        assert _audit(lib, shape, 5, flags, ws=total - 256) == -1
        msg = lib.dion_last_error().decode()
        # (the norm is launch 0, or launch 1 behind the transposing copy of a tall input)
        assert "(frobenius norm)" in msg and "reciprocal norms" in msg, msg
        # cut in the middle of the layout: whatever launch first touches a buffer past the cut is named
        x_bytes = 2 * shape[0] * max(shape[1], shape[2]) * min(shape[1], shape[2])
        assert _audit(lib, shape, 5, flags, ws=x_bytes // 2) == -1
        msg = lib.dion_last_error().decode()
        assert "outside the call's buffers" in msg, msg


def test_static_scratch_limit_is_checked_before_any_device_work():
    import ctypes

    lib = _lib.load()
    c = (ctypes.c_float * 15)(*[1.0] * 15)
    rc = lib.dion_ns_orthogonalize_static(0x1000, BF16, 0x2000, 8, 2048, 4096, c, 5, ctypes.c_float(1.0),
                                          ctypes.c_float(0.0), 0, 0, None)
    assert rc == -2
    msg = lib.dion_last_error().decode()
    assert str(_lib.DION_NS_STATIC_SCRATCH_BYTES) in msg and "caller workspace" in msg


def _audit_prepared(lib, shape, n_iters=5, flags=0, with_update=0, x_dtype=F32, mats_per_ptr=1, ws=0, reset=2):
    b, r, c = shape
    return lib.dion_ns_plan_audit_prepared(b, r, c, n_iters, flags, reset, with_update, x_dtype, mats_per_ptr, ws)


@pytest.mark.parametrize("shape", CONFIG_SHAPES + RAGGED_SHAPES)
def test_prepared_input_plans(shape):
    """The prepared form (input in the iteration's layout, norm partials from the caller): taken exactly by
    the shapes that fill whole tiles; no norm pass over the input (one small launch turns the partial sums
    into the per-matrix factor) and no transposing copy of a tall one, every launch
    inside the call's buffers, the fused update included."""
    lib = _lib.load()
    b, r, c = shape
    for flags in (0, GRAM):
        takes = bool(lib.dion_ns_accepts_prepared(b, r, c, flags, 5))
        whole = min(r, c) > 64 and r % 128 == 0 and c % 128 == 0
        if takes:
            assert whole, shape
        if not whole:
            assert not takes, shape
        n = _audit_prepared(lib, shape, 5, flags)
        if not takes:
            assert n == -1 and "does not take a prepared input" in lib.dion_last_error().decode(), shape
            continue
        # the plain form of the same call: a norm launch where this one finalizes the caller's partial sums,
        # plus the transposing copy of a tall input (a wide one is read where it lies in both forms)
        plain = _audit(lib, shape, 5, flags)
        assert n == plain - (1 if r > c else 0), (shape, flags, n, plain)
        assert _audit_prepared(lib, shape, 0, flags) == -1  # no iteration to carry the normalisation
        for x_dtype in (F32, BF16):
            assert _audit_prepared(lib, shape, 5, flags, with_update=1, x_dtype=x_dtype) > 0, \
                (shape, lib.dion_last_error().decode())
        # a workspace cut short is caught for this form too
        assert _audit_prepared(lib, shape, 5, flags, ws=4096) == -1


@pytest.mark.parametrize("shape", [(16, 128, 256), (24, 128, 1024), (20, 768, 128)])
def test_prepared_input_of_matrices_the_small_kernel_takes(shape):
    """Where plain calls of a batch run the small-matrix kernel, a prepared input is not advised but still taken: the GEMMs
    of a batch too small for that kernel, within the workspace the library reports."""
    lib = _lib.load()
    b, r, c = shape
    assert not lib.dion_ns_accepts_prepared(b, r, c, 0, 5) and lib.dion_ns_accepts_prepared(15, r, c, 0, 5)
    assert _audit(lib, shape, 5, 0) == 1
    for with_update in (0, 1):
        n = _audit_prepared(lib, shape, 5, 0, with_update=with_update)
        assert n == _audit_prepared(lib, (15, r, c), 5, 0, with_update=with_update) > 1
    assert lib.dion_ns_update_workspace_bytes(b, r, c, 0, 5) >= lib.dion_ns_workspace_bytes(b, r, c, 0)


@pytest.mark.parametrize("shape", [s for s in RAGGED_SHAPES if min(s[1:]) > 64 and (s[1] % 128 or s[2] % 128)])
def test_padded_plans_with_the_update(shape):
    """Matrices with padding: one copy in, the update in the last product, stored extents without the padding."""
    lib = _lib.load()
    b = shape[0]
    for flags in (0, GRAM):
        for x_dtype in (F32, BF16):
            for in_dtype in (F32, BF16):
                n = _audit(lib, shape, 5, flags, in_dtype, with_update=2, x_dtype=x_dtype)
                assert n > 0, lib.dion_last_error().decode()
                if not flags or max(shape[1:]) < 3 * min(shape[1:]):
                    assert n == 2 + 3 * 4 + 2 + (b + 63) // 64


@pytest.mark.parametrize("shape", [(16, 128, 256), (400, 128, 1024), (24, 1024, 128), (17, 64, 2048), (40, 100, 500)])
def test_an_output_over_another_matrix_keeps_a_batch_off_the_small_kernel(shape):
    """One workgroup per matrix stores its result while others have not read their input: a batch of that kernel whose
    output overlaps the input runs the GEMMs, which copy the input first.  In place in bf16 every workgroup holds its own
    matrix before it stores."""
    lib = _lib.load()
    b, r, c = shape
    mat = 2 * r * c
    for in_dtype in (BF16, F32):
        size = b * mat * (1 if in_dtype == BF16 else 2)
        audit = lambda offset, n=5: lib.dion_ns_plan_audit_overlap(b, r, c, in_dtype, n, 0, 0, offset)
        assert audit(size) == 1 and audit(-b * mat) == 1  # side by side
        assert audit(0) == 1 if in_dtype == BF16 else audit(0) > 1
        for offset in (mat, -mat, 2, size - 2, 2 - b * mat):
            if offset % 16 == 0:
                assert audit(offset) > 1 and audit(offset, 0) > 1, offset
            else:  # what the GEMM path refuses anyway
                assert audit(offset) == -1 and "16-byte" in lib.dion_last_error().decode()
    # the GEMMs need the workspace that is reported for the shape: refused on the host without it
    import ctypes
    co = (ctypes.c_float * 15)(*[1.0] * 15)
    base = 0x100000000000
    assert lib.dion_ns_orthogonalize(base, BF16, base + mat, b, r, c, co, 5, 1.0, 0.0, 0, 0, None, 0, None) == -2
    if lib.dion_ns_workspace_bytes(b, r, c, 0) > _lib.DION_NS_STATIC_SCRATCH_BYTES:
        assert lib.dion_ns_orthogonalize_static(base, BF16, base + mat, b, r, c, co, 5, 1.0, 0.0, 0, 0, None) == -2


def test_overlap_of_matrices_that_only_the_small_kernel_takes():
    lib = _lib.load()
    for offset in (0, 64 * 768 * 2, -64 * 768 * 2):
        assert lib.dion_ns_plan_audit_overlap(432, 64, 768, BF16, 5, 0, 0, offset) == 1


@pytest.mark.parametrize("batch", [1, 15, 32768, 32769, 32773, 65537, 98305, 200001])
def test_a_batch_of_several_calls_runs_one_kernel(batch):
    """The calls that ops.ns_orthogonalize cuts a batch into cover it once and plan the same launches: a matrix's result does
    not depend on which of them it falls into."""
    from dion_amd import ops
    lib = _lib.load()
    calls = ops._calls(batch)
    assert [b0 for b0, _n in calls] == [sum(n for _b, n in calls[:i]) for i in range(len(calls))]
    assert sum(n for _b, n in calls) == batch and all(0 < n <= 32768 for _b, n in calls)
    sizes = sorted({n for _b, n in calls})
    assert sizes[-1] - sizes[0] <= 1
    for shape in [(128, 256), (64, 2048), (100, 500), (128, 128), (256, 256), (300, 40)]:
        for flags in (0, GRAM):
            plans = {(_audit(lib, (n, *shape), 5, flags), lib.dion_gemm_tile_edge(n, 256, 256, 1)) for n in sizes}
            assert len(plans) == 1 and min(plans)[0] > 0, (shape, plans)


@pytest.mark.parametrize("shape", CONFIG_SHAPES + RAGGED_SHAPES + [(1000, 128, 1024), (1024, 32, 4096), (24, 1024, 128)])
def test_the_workspace_of_a_plain_call(shape):
    """What a call uses: nothing where one workgroup takes a whole matrix (432 x (64 x 768) would report 0.6 GB of GEMM
    buffers), the orthogonalized matrices alone where the update follows."""
    lib = _lib.load()
    b, r, c = shape
    for flags in (0, GRAM):
        for n_iters in (0, 5, 9):
            full = lib.dion_ns_workspace_bytes(b, r, c, flags)
            plain = lib.dion_ns_call_workspace_bytes(b, r, c, flags, n_iters, 0)
            update = lib.dion_ns_call_workspace_bytes(b, r, c, flags, n_iters, 1)
            tail = -(-b * r * c * 2 // 256) * 256
            small = _audit(lib, shape, n_iters, flags) == 1
            assert plain == (0 if small else full)
            fuses = not small and n_iters > 0
            assert update == (tail if small else full + (0 if fuses else tail))
            # an upper bound for prepared inputs too, as before
            assert lib.dion_ns_update_workspace_bytes(b, r, c, flags, n_iters) >= update


@pytest.mark.parametrize("batch,m,edge", [(85, 128, 64), (86, 128, 128), (128, 128, 128), (25, 256, 64), (26, 256, 128), (51, 256, 128),
                                          (13, 384, 64), (24, 384, 64), (25, 384, 128), (14, 512, 64), (15, 512, 128)])
def test_tiles_of_symmetric_products_with_short_reductions(batch, m, edge):
    """64-wide tiles split a reduction over four wavefronts; past one such tile per CU a short one is left with less than it
    costs to add the parts (128 x (128 x 128): 6.8 us against 5.1)."""
    assert _lib.load().dion_gemm_tile_edge(batch, m, m, 1) == edge


@pytest.mark.parametrize("line,m,n,addend,edge", [
    (1, 2048, 1 << 24, 0, 64), (1, 2048, (1 << 24) - 128, 0, 129), (1, 2048, 16911104, 0, 64),  # 128 rows past 2^31 elements
    (1, 4096, 1 << 25, 0, 64), (1, 4096, 1 << 24, 0, 256),
    (3, 128, 1 << 26, 1, 64), (3, 128, (1 << 26) - 128, 1, 128), (3, 128, 1 << 26, 0, 128), (3, 128, 1 << 27, 0, 64)])
def test_rows_too_long_for_32_bit_offsets(line, m, n, addend, edge):
    """128- and 256-wide tiles address a tile's rows with 32-bit offsets, which the rows of X X^T from 2^24 columns on (2^25 with
    256-wide tiles), of the addend from 2^26, of the K-major operand from 2^27 do not fit: 64-wide tiles take those."""
    assert _lib.load().dion_ns_line_kernel(line, 1, m, n, addend) == edge


@pytest.mark.parametrize("line,batch,m,n,edge", [
    (1, 64, 768, 1536, 256), (1, 36, 1024, 2048, 256), (1, 32, 1024, 1280, 128), (1, 33, 1024, 1280, 256),  # 1152 | 1188 128-wide tiles
    (1, 110, 512, 2048, 256), (1, 110, 512, 1920, 128), (1, 102, 512, 2048, 128), (1, 54, 768, 3072, 256), (1, 342, 256, 1024, 128),
    (1, 10, 1792, 7168, 128), (1, 42, 1024, 1024, 128), (1, 43, 1024, 1024, 256), (2, 42, 1024, 1024, 128), (2, 43, 1024, 1024, 256),
    (1, 13, 1024, 3072, 128), (1, 16, 1024, 3072, 256), (1, 26, 1024, 3072, 128)])
def test_tiles_of_symmetric_products_by_rounds(line, batch, m, n, edge):
    """128-wide tiles of a symmetric product in their third round of two per CU: no more than soon after its begin where the
    reduction is longer than the matrix is wide (a call on 42 x (1024 x 2048) took 1846 us so, 1781 with 256-wide ones)."""
    assert _lib.load().dion_ns_line_kernel(line, batch, m, n, 0) == edge


@pytest.mark.parametrize("batch,m,n,edges", [  # per form: stored, with an addend, update, transposed update, both of padded parameters
    (42, 512, 1024, (256, 128, 128, 128, 128, 128)), (41, 512, 1024, (128,) * 6), (48, 512, 1024, (256,) * 6),
    (11, 1024, 2048, (256, 128, 128, 128, 128, 128)), (10, 1536, 1536, (128,) * 6),
    (27, 512, 1024, (256, 256, 256, 256, 256, 128)), (43, 256, 768, (256, 256, 256, 256, 256, 128)), (15, 768, 768, (256,) * 6),
    (1, 4096, 4096, (256,) * 6), (8, 1024, 1024, (128,) * 6)])
def test_tiles_of_full_products_by_form(batch, m, n, edges):
    """The lines between 128- and 256-wide tiles of B X lie elsewhere where the epilogue reads memory (336 tiles of
    42 x (512 x 1024): stored 33.9 us against 31.2, with an addend 34.6 / 36.5, updating padded transposed parameters 70.7 / 84.3)."""
    assert tuple(_lib.load().dion_ns_line_kernel(3, batch, m, n, form) for form in range(6)) == edges
