"""The register-dequantising matmul in tiles of 64 and 128 rows, several super-blocks deep, with
ragged last row and column tiles, parts of K that run out unevenly, and a split of K; each
case asks cmk_iq2_matmul_kernel for its tile, so that it cannot miss it.

Bars of test_gpu_mm.py (cond <= 1e-5, rel <= 1e-3) against the 64-bit product with the
dequantised weights: exact, or rounded to f16 where IQ2_XXS has them so (cmk_iq2_matmul_path);
W8A8 with its bars in test_gpu_parity.py for rounded weights."""

import numpy as np
import pytest
import torch

from test_gpu_mm import _DT, _run
from test_gpu_parity import x_as_f32, x_tensor
from test_gpu_variants import dev, errors, random_weights, to_dev  # noqa: F401

pytestmark = pytest.mark.gpu

ALL, OTHERS = (0, 1, 2, 3), (1, 2, 3)
# formats, m, n, k, x, W8A8, tile rows, split or not
SHAPES = [
    (ALL, 129, 4100, 776, "f16", False, 64, False), (OTHERS, 300, 8000, 520, "f16", False, 64, False),
    (OTHERS, 300, 2000, 8200, "f16", False, 64, True), (ALL, 130, 4100, 777, "bf16", False, 64, False),
    (ALL, 500, 8010, 1288, "bf16", False, 64, False), (ALL, 90, 9000, 1288, "f32", False, 64, False),
    (ALL, 260, 8010, 1288, "bf16", True, 64, False), ((0,), 300, 8000, 520, "f16", False, 128, False),
    (ALL, 150, 8010, 520, "f32", False, 128, False), (OTHERS, 600, 4100, 1288, "f32", False, 128, False),
    (OTHERS, 300, 2000, 8200, "f32", False, 128, True), ((0,), 128, 2000, 8200, "f32", False, 128, True),
    (ALL, 300, 8000, 520, "f16", True, 128, False), (OTHERS, 1000, 8010, 1288, "bf16", True, 128, False),
    (OTHERS, 600, 1030, 9000, "bf16", True, 128, True)]
CASES = [(v,) + s[1:] for s in SHAPES for v in s[0]]


@pytest.mark.parametrize("v,m,n,k,dtype,w8a8,tile,split", CASES)
def test_tiles(pkg, cabi, oracle, inputs, dev, v, m, n, k, dtype, w8a8, tile, split):  # noqa: F811
    code = {"f32": cabi.CMK_F32, "f16": cabi.CMK_F16, "bf16": cabi.CMK_BF16}[dtype]
    mode = cabi.CMK_ACT_QUANT_W8A8 if w8a8 else cabi.CMK_ACT_QUANT_OFF
    plan = cabi.matmul_kernel(code, m, n, k, variant=v, mode=mode)
    assert (plan["kernel"], plan["row_tile"], plan["splits"] > 1) == ("register_matmul", tile, split)
    wb, ws = (to_dev(t, dev) for t in random_weights(oracle, v, n, k, seed=m + n + k))
    x = x_tensor(inputs.synthetic_x(m, k, seed=m + k), _DT[dtype], dev)
    y = _run(pkg, v, x, n, k, wb, ws, w8a8)
    assert torch.equal(y, _run(pkg, v, x, n, k, wb, ws, w8a8))
    rounded = v == 0 and cabi.matmul_path(code, m, n, k, mode) == "gemm"
    w = pkg.iq2_dequantize_to_f16(wb, ws, n, k, pkg.Iq2MatmulVariant(v),
                                  out_dtype=torch.float16 if rounded else torch.float32).double()
    x64 = x.double()
    if w8a8:
        x64 = to_dev(oracle.rowwise_qdq_w8a8(np.ascontiguousarray(x_as_f32(x)), m, k)
                     .astype(np.float64), dev)
    cond, rel = errors(y.cpu().numpy(), (x64 @ w.T).cpu().numpy(),
                       (x64.abs() @ w.abs().T).cpu().numpy())
    loose = w8a8 and rounded
    assert cond <= (1e-4 if loose else 1e-5) and rel <= (1e-2 if loose else 1e-3), (cond, rel)
