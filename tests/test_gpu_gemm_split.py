"""The MFMA GEMM itself (asked of cmk_iq2_matmul_kernel) on shapes beyond the register-
dequantising matmul's: its k split in a caller's workspace of garbage, every staging of x, NaN and
infinities, and the no-alloc entry point.  Bars of test_gpu_parity.py: against the product
with the weights rounded to f16, cond <= 1e-5 and rel <= 1e-3 (W8A8, whose q / inv the
reference rounds: 1e-4 and 1e-2)."""

import numpy as np
import pytest
import torch

from test_gpu_mm import _DT, _run
from test_gpu_parity import dev, errors, to_dev, x_as_f32, x_tensor  # noqa: F401

pytestmark = pytest.mark.gpu

SHAPES = [(600, 1000, 1792, "f16", False), (600, 1024, 8192, "f16", True), (128, 8192, 8192, "f32", False),
          (300, 1000, 2824, "f32", False), (600, 1000, 1800, "bf16", False),
          (600, 520, 2048, "bf16", True), (600, 520, 2048, "f32", True)]


@pytest.mark.parametrize("m,n,k,dtype,w8a8", SHAPES)
def test_split_in_garbage(pkg, cabi, oracle, inputs, dev, m, n, k, dtype, w8a8):  # noqa: F811
    code = {"f32": cabi.CMK_F32, "f16": cabi.CMK_F16, "bf16": cabi.CMK_BF16}[dtype]
    mode = cabi.CMK_ACT_QUANT_W8A8 if w8a8 else cabi.CMK_ACT_QUANT_OFF
    assert cabi.matmul_kernel(code, m, n, k, mode=mode)["kernel"] == "gemm"
    need = cabi.workspace_size(code, m, n, k, mode=mode)
    assert need >= 2 * m * n * 4  # partial sums of a split
    wb, ws = inputs.synthetic_weights(n, k, seed=m)
    wbt, wst = to_dev(wb, dev), to_dev(ws, dev)
    x = x_tensor(inputs.synthetic_x(m, k, seed=n), _DT[dtype], dev)
    ref = _run(pkg, 0, x, n, k, wbt, wst, w8a8)
    work = torch.full((need + 256,), 0xFF, dtype=torch.uint8, device=dev)
    args = (x.data_ptr(), code, x.numel(), m, wbt.data_ptr(), wbt.numel(), wst.data_ptr(),
            wst.numel(), n, k)
    for _ in range(2):
        out = torch.full((m, n), float("nan"), device=dev)
        cabi.matmul_raw(*args, out.data_ptr(), mode=mode, workspace_ptr=work.data_ptr(),
                        workspace_bytes=need)
        assert torch.equal(out, ref)
    assert bool((work[need:] == 0xFF).all())
    if need <= cabi.NOALLOC_SCRATCH_BYTES:
        out = torch.full((m, n), float("nan"), device=dev)
        cabi.matmul_noalloc_raw(*args, out.data_ptr(), mode=mode)
        assert torch.equal(out, ref)
    w = pkg.iq2_dequantize_to_f16(wbt, wst, n, k, pkg.Iq2MatmulVariant(0),
                                  out_dtype=torch.float16).double()
    x64 = x.double()
    if w8a8:
        x64 = to_dev(oracle.rowwise_qdq_w8a8(np.ascontiguousarray(x_as_f32(x)), m, k)
                     .astype(np.float64), dev)
    cond, rel = errors(ref.cpu().numpy(), (x64 @ w.T).cpu().numpy(),
                       (x64.abs() @ w.abs().T).cpu().numpy())
    assert cond <= (1e-4 if w8a8 else 1e-5) and rel <= (1e-2 if w8a8 else 1e-3), (cond, rel)


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_non_finite_row_stays_alone(pkg, cabi, inputs, dev, dtype, bad):  # noqa: F811
    m, n, k = 600, 520, 2048
    code = {"f32": cabi.CMK_F32, "f16": cabi.CMK_F16, "bf16": cabi.CMK_BF16}[dtype]
    assert cabi.matmul_kernel(code, m, n, k)["kernel"] == "gemm"
    wb, ws = inputs.synthetic_weights(n, k, seed=1)
    x = inputs.synthetic_x(m, k, seed=2)
    x[5, 300] = bad
    y = _run(pkg, 0, x_tensor(x, _DT[dtype], dev), n, k, to_dev(wb, dev), to_dev(ws, dev), False)
    assert not bool(torch.isfinite(y[5]).any())
    y[5] = 0.0
    assert bool(torch.isfinite(y).all())
