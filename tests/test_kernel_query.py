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


@pytest.mark.parametrize("x,m,n,k,v,w8a8,kernel", [
    # staged rows: decode launches are the faster ones at short K
    ("bf16", 5, 2048, 2048, 1, False, "decode"), ("f32", 8, 4096, 1024, 2, False, "decode"),
    ("f32", 8, 28672, 1024, 1, False, "decode"), ("bf16", 5, 4096, 4096, 1, False, "register_matmul"),
    ("bf16", 8, 4096, 1024, 1, True, "register_matmul"), ("bf16", 8, 28672, 1024, 1, True, "decode"),
    ("bf16", 5, 12288, 2048, 1, False, "register_matmul"), ("bf16", 5, 12288, 1024, 1, False, "decode"),
    ("f32", 8, 12288, 1024, 2, False, "register_matmul"), ("f32", 5, 20480, 2048, 2, False, "decode"),
    ("f16", 2, 4099, 1027, 1, False, "decode"), ("f32", 5, 4099, 1027, 1, False, "register_matmul"),
    ("bf16", 5, 5000, 900, 1, False, "decode"),
    ("f32", 16, 4096, 512, 1, False, "decode"), ("f32", 16, 4096, 512, 2, False, "register_matmul"),
    ("f32", 17, 4096, 512, 1, False, "register_matmul"),
    # two rows of long ones
    ("f32", 2, 1536, 28672, 3, False, "decode"), ("f32", 2, 2048, 16384, 3, False, "register_matmul"),
    ("f32", 3, 1536, 28672, 1, False, "register_matmul"),
    # few f16 rows of many columns
    ("f16", 2, 28672, 2048, 1, False, "decode"), ("f16", 5, 28672, 2048, 1, False, "register_matmul"),
    ("f16", 2, 28672, 4096, 1, False, "register_matmul")])
def test_lines_between_kernels(cabi, x, m, n, k, v, w8a8, kernel):
    code = {"f32": cabi.CMK_F32, "f16": cabi.CMK_F16, "bf16": cabi.CMK_BF16}[x]
    mode = cabi.CMK_ACT_QUANT_W8A8 if w8a8 else cabi.CMK_ACT_QUANT_OFF
    assert cabi.matmul_kernel(code, m, n, k, variant=v, mode=mode)["kernel"] == kernel
