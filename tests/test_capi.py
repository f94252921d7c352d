"""C-ABI library: loads, exports every declared entry point, validates
arguments on the host.  CPU only: nothing here launches a kernel (every call
below fails argument validation before any HIP call)."""

import ctypes

import pytest

from torch_spyre import _capi

from oracle import layout as L

from helpers import gemm_plan


def test_library_exports_every_declared_function():
    lib = _capi.lib()
    declared = _capi.header_functions()
    assert len(declared) >= 20
    missing = [name for name in declared if not hasattr(lib, name)]
    assert not missing, f"declared in include/spyre_hip.h but not exported: {missing}"
    # every declared function has a ctypes signature in the binding
    assert set(declared) <= set(_capi._SIGS), set(declared) - set(_capi._SIGS)


def test_abi_version():
    assert _capi.lib().sph_abi_version() == 1


@pytest.mark.parametrize("shape,order,eb", [([128], [0], 2), ([512, 256], [0, 1], 2),
                                            ([512, 256], [1, 0], 2), ([3, 5, 100], [2, 0, 1], 4),
                                            ([7], [0], 1)])
def test_stick_nbytes_matches_oracle(shape, order, eb):
    got = _capi.lib().sph_stick_nbytes(len(shape), _capi.i64_array(shape),
                                       _capi.i32_array(order), eb)
    assert got == L.stick_nbytes(shape, eb, order)


def test_host_side_argument_errors():
    lib = _capi.lib()
    rc = lib.sph_gemm(_capi.F16, 0, 0, -1, 4, 4, 1.0, None, 4, None, 4, 0.0, None, 0, 0,
                      None, 4, 0, None)
    assert rc == 1001
    assert b"negative" in lib.sph_last_error()
    rc = lib.sph_gemm(_capi.F32, 0, 0, 4, 4, 4, 1.0, None, 4, None, 4, 0.0, None, 0, 0,
                      None, 4, 0, None)
    assert rc == 1002
    rc = lib.sph_softmax_rows(_capi.F16, _capi.F16, None, 2, None, 2, 4, 8, 1.0, 0, 0, 0, None)
    assert rc == 1001  # ld < cols
    with pytest.raises(_capi.SpyreKernelError, match="dim_order"):
        _capi.call("sph_stick_pack", None, None, 2, _capi.i64_array([2, 2]),
                   _capi.i64_array([2, 1]), _capi.i32_array([0, 0]), 2, None)
    rc = lib.sph_pointwise(999, 1, None, 1, None, 0.0, 0.0, None)
    assert rc == 1001
    # zero-size work is a no-op that succeeds without touching the device
    assert lib.sph_gemm_f16(0, 4, 4, None, None, None, None) == 0
    assert lib.sph_softmax_rows_f16(None, None, 0, 8, None) == 0
    assert ctypes.c_int(lib.sph_tri(0, 0, 2, None, None, 0, 4, 4, None)).value == 0


@pytest.mark.parametrize("batch,m,n,k,split", [
    (1, 4096, 4096, 4096, False),    # 256 tiles: one whole round
    (1, 2048, 4096, 4096, True),     # c4 O: a 2-way split beats 128-wide tiles on cold weights
    (1, 2048, 4096, 2048, False),    # K = 2048: a round of 128-wide tiles beats the split
    (1, 2048, 4096, 12800, True),    # c4 down: the split tail beats 128-wide tiles
    (1, 2048, 25600, 4096, True),    # c4 gate/up: 800 tiles, a 32-tile tail in 8 slices
    (1, 256, 256, 2048, True),       # one tile in 8 slices
    (2, 2048, 4096, 12800, False),   # batched: never split
    (1, 2048, 4096, 1024, False)])   # K < 2048: slices too short
def test_gemm_workspace_bytes(batch, m, n, k, split):
    # host-side sizing of the split-K workspace (no device call): nonzero
    # exactly where the GEMM would split its last round along K
    got = _capi.lib().sph_gemm_workspace_bytes(batch, m, n, k)
    assert (got > 0) == split, got
    if split:
        assert got % (256 * 256 * 4) == 0 and got <= 256 * 256 * 256 * 4


def test_gemm_workspace_bytes_covers_each_layout():
    # the size without a layout covers the calls of either, leading dimensions of
    # whole 16-byte chunks need no copies, a transposed A takes neither copies
    # nor slices, and the size is what the plan of the call uses: the padded
    # copies and at most eight slices of partial sums (or one 256 x 256 tile per
    # CU of a split tail)
    lib = _capi.lib()
    for batch in (1, 3):
        for m in (1, 8, 9, 33, 255, 300, 2100):
            for n in (64, 65, 504, 4097):
                for k in (8, 63, 520, 1029, 4096):
                    both = lib.sph_gemm_workspace_bytes(batch, m, n, k)
                    for tb in (0, 1):
                        ldb = k if tb else n
                        one = lib.sph_gemm_workspace_bytes_ex(0, tb, batch, m, n, k, k, ldb)
                        _, tile, slices, packed, _ = gemm_plan(batch, m, n, k, tb)
                        assert 0 <= one <= both
                        assert (one > 0) == (slices > 1 or packed != "")
                        pads = 2 * (k + 64) * ((m if "A" in packed else 0) + (n + 8 if "B" in packed else 0))
                        # (few padded rows: sized for slices, run on a small-row kernel)
                        parts = (max(8 * m * (n + 3) * 4, 256 ** 3 * 4) if slices > 1 else
                                 8 * m * (n + 3) * 4 if m <= 16 else 0)
                        assert one <= batch * pads + 512 + parts
                        # less than that: the call runs without slices or copies
                        if one > 0:
                            _, _, fewer, unpacked, _ = gemm_plan(batch, m, n, k, tb, workspace=0)
                            assert fewer == 1 and unpacked == ""
                    assert lib.sph_gemm_workspace_bytes_ex(1, 0, batch, m, n, k, m, n) == 0
                    if batch > 1 and n % 8 == 0 and k % 8 == 0:
                        assert both == 0


@pytest.mark.parametrize("batch,m,n,k,tb,want", [
    # short K on the register-staged kernel where the ring kernel's epilogue or
    # its 192 x 128 tiles cost more than its loads save
    (10, 250, 1024, 32, 1, "staged"), (24, 552, 512, 128, 1, "staged"),
    (4, 1608, 608, 224, 1, "staged"), (1, 2184, 5424, 32, 1, "staged"),
    (16, 110, 744, 64, 1, "staged"), (10, 1571, 328, 128, 0, "staged"),
    (16, 1152, 528, 64, 0, "staged"),
    # the ring kernel elsewhere: one round of tiles, longer K, a transposing B
    (4, 256, 2115, 384, 1, "ring"), (8, 1280, 146, 640, 1, "ring"),
    (24, 128, 5671, 448, 1, "ring"), (64, 128, 4864, 96, 1, "ring"),
    (8, 401, 463, 320, 0, "ring"), (1, 333, 6144, 4096, 1, "ring"), (10, 1571, 328, 2048, 0, "ring"),
    # whole 256-row tiles of such a product stay on the direct-load kernel
    (8, 512, 1280, 64, 0, "direct")])
def test_gemm_plan_short_k(batch, m, n, k, tb, want):
    assert gemm_plan(batch, m, n, k, tb)[0] == want


@pytest.mark.parametrize("batch,m,n,k,ws,want", [
    # 9 to 16 rows, few columns, long K: the small-row kernel where the ring
    # kernel has no K slices
    (8, 15, 128, 4096, None, "skinny"), (2, 9, 256, 1024, None, "skinny"),
    (16, 16, 128, 8192, None, "skinny"), (1, 12, 1024, 2048, 0, "skinny"),
    (1, 12, 1024, 2048, None, "ring"), (16, 16, 128, 1024, None, "ring"),
    (8, 17, 128, 4096, None, "ring"), (2, 16, 512, 512, None, "ring"),
    (32, 12, 128, 4096, None, "ring"), (32, 12, 128, 8192, None, "skinny")])
def test_gemm_plan_16_rows(batch, m, n, k, ws, want):
    assert gemm_plan(batch, m, n, k, 1, workspace=ws)[0] == want


@pytest.mark.parametrize("batch,max_len,rc", [
    (512, (1 << 30) - 1, 1003),   # 2^24 chunks of 64 positions x 4096 units: past the grid
    (512, 64 * 4096, 1003),       # exactly 2^24 workgroups
    (512, 64 * 4096 - 64, 1001)])  # the largest grid: refused for its workspace only
def test_decode_step_grid_limit(batch, max_len, rc):
    # refused before any launch (the pointers below are never read)
    a = 4096
    got = _capi.lib().sph_decode_attention_step(
        _capi.F16, batch, 8, 8, 128, a, 24 * 128, a, a, 128, a, None, a, 8 * max_len * 128,
        max_len * 128, 128, a, 8 * max_len * 128, max_len * 128, 128, 1, max_len,
        ctypes.c_float(0.1), a, 8 * 128, a, 1 << 62 if rc != 1001 else 16, None)
    assert got == rc
