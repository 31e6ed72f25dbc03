"""cmk_iq2_matmul_kernel (host only): the kernel behind a call, and for the register-
dequantising matmul its passes, tiles and split."""

import pytest


def test_kernels(cabi):
    k = lambda *a, **kw: cabi.matmul_kernel(*a, **kw)["kernel"]  # noqa: E731
    F32, F16, BF16, W8A8 = cabi.CMK_F32, cabi.CMK_F16, cabi.CMK_BF16, cabi.CMK_ACT_QUANT_W8A8
    # IQ2_XXS: decode shapes, batches, short prompts, prompts
    assert k(F32, 1, 4096, 4096) == k(F32, 16, 14336, 4096) == k(F16, 4, 14336, 4096) == "decode"
    assert k(F16, 8, 14336, 4096) == k(BF16, 16, 14336, 4096) == "register_matmul"
    assert k(F32, 16, 14336, 4096, mode=W8A8) == k(F32, 32, 14336, 4096, mode=W8A8) == "register_matmul"
    assert k(F16, 128, 14336, 4096) == k(F32, 128, 1024, 8192) == "register_matmul"
    assert k(F16, 512, 14336, 4096) == k(F32, 128, 8192, 8192) == "gemm"
    # the other formats
    for v in (1, 2, 3):
        assert k(F32, 1, 4096, 4096, variant=v) == "decode"
        assert k(F16, 16, 4096, 4096, variant=v) == k(F32, 2048, 4096, 4096, variant=v) \
            == "register_matmul"
    # the exact-weight paths by weights, not by kernel
    assert cabi.matmul_path(F16, 8, 14336, 4096) == "gemv"
    assert cabi.matmul_path(F16, 128, 14336, 4096) == "gemm"


def test_register_matmul_passes_and_tiles(cabi):
    d = cabi.matmul_kernel(cabi.CMK_F16, 600, 4096, 4096, variant=1)
    assert d == {"kernel": "register_matmul", "rows_per_pass": 600, "row_tile": 64, "splits": 1}
    d = cabi.matmul_kernel(cabi.CMK_F32, 600, 4096, 4096, variant=1)
    assert d == {"kernel": "register_matmul", "rows_per_pass": 600, "row_tile": 128, "splits": 1}
    # without room to stage one tile of rows: the decode launches
    assert cabi.matmul_kernel(cabi.CMK_F32, 600, 4096, 4096, variant=1,
                              workspace_bytes=0)["kernel"] == "decode"
    # room for 130 staged rows: a pass of 128
    room = 130 * 4096 * 4 + 2048
    assert cabi.matmul_kernel(cabi.CMK_F32, 600, 4096, 4096, variant=1,
                              workspace_bytes=room)["rows_per_pass"] == 128
    assert cabi.matmul_kernel(cabi.CMK_F32, 65536, 28672, 28672, variant=1)["rows_per_pass"] == 2304


def test_refused_arguments(cabi):
    with pytest.raises(cabi.CmkError, match="expects non-zero dimensions"):
        cabi.matmul_kernel(cabi.CMK_F32, 1, 0, 256)
    with pytest.raises(cabi.CmkError, match="workspace too small"):
        cabi.matmul_kernel(cabi.CMK_F32, 512, 14336, 4096, workspace_bytes=0)
