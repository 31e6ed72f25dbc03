"""Rows of very wide range on the register-dequantising matmul: super-blocks of x far below the
row's largest, met by weight rows whose block of large x is empty (d = 0), so that only the small
ones count; and f16 rows of subnormals.  The decode launches scale x by 32 columns.  Bar of the
decode kernels: cond <= 1e-5 and rel <= 1e-3 against the fp64 oracle."""

import numpy as np
import pytest
import torch

from test_gpu_mm import _DT, _expected, _run
from test_gpu_parity import x_tensor
from test_gpu_variants import dev, errors, random_weights, to_dev  # noqa: F401

pytestmark = pytest.mark.gpu


def _weights(oracle, v, n, k, seed):
    """d = 0 in block 0 of every second weight row, in blocks 0 and 1 of every fourth."""
    wb, ws = random_weights(oracle, v, n, k, seed)
    spb, bpr = oracle.scales_per_block(v), -(-k // 256)
    d = ws.reshape(n, bpr, spb)
    d[1::2, 0, :2] = 0
    d[3::4, 1, :2] = 0
    return wb, ws


# 16 rows: tiles of 32; 300: of 64 (bf16) and 128 rows (f32); a long K is split.  (IQ2_XXS:
# f32 rows on the decode kernel, many rows on weights rounded to f16.)
@pytest.mark.parametrize("v,dtype,m,n,k", [
    (v, d, m, n, k) for v in (0, 1, 2, 3) for d in ("f32", "bf16")
    for m, n, k in ((16, 1100, 4096), (300, 8000, 520), (16, 300, 17000))
    if v > 0 or (d == "bf16" and m == 16)])
def test_blocks_far_below_the_row(pkg, cabi, oracle, inputs, dev, v, dtype, m, n, k):  # noqa: F811
    code = {"f32": cabi.CMK_F32, "bf16": cabi.CMK_BF16}[dtype]
    assert cabi.matmul_kernel(code, m, n, k, variant=v)["kernel"] == "register_matmul"
    x = inputs.synthetic_x(m, k, seed=m + k)
    x[::3, :256] *= 1e20  # every third row: 1e20, then 1, then 1e-12
    x[::3, 512:] *= 1e-12
    x[1::3, :256] *= 1e6
    wb, ws = _weights(oracle, v, n, k, seed=v + n)
    xt = x_tensor(x, _DT[dtype], dev)
    y = _run(pkg, v, xt, n, k, to_dev(wb, dev), to_dev(ws, dev), False).cpu().numpy()
    y64, sc = _expected(oracle, v, xt, n, k, wb, ws, False)
    # (by row and group of weight rows: outputs of one scale)
    for r in (0, 1, 2, m - 1):
        for c in (slice(0, None, 2), slice(1, None, 4), slice(3, None, 4)):
            cond, rel = errors(y[r:r + 1, c], y64[r:r + 1, c], sc[r:r + 1, c])
            assert cond <= 1e-5 and rel <= 1e-3, (r, c, cond, rel)


@pytest.mark.parametrize("m,n,k", [(12, 1100, 4096), (300, 2000, 520)])
@pytest.mark.parametrize("v", [1, 2, 3])
def test_subnormal_f16_rows(pkg, cabi, oracle, inputs, dev, v, m, n, k):  # noqa: F811
    assert cabi.matmul_kernel(cabi.CMK_F16, m, n, k, variant=v)["kernel"] == "register_matmul"
    x = inputs.synthetic_x(m, k, seed=5).astype(np.float16)
    x[0] = (x[0].astype(np.float32) * 2.0 ** -20).astype(np.float16)
    x[m // 2] = (x[m // 2].astype(np.float32) * 2.0 ** -22).astype(np.float16)
    assert (np.abs(x[m // 2].astype(np.float32)) < 2.0 ** -14).all()
    wb, ws = random_weights(oracle, v, n, k, seed=v)
    xt = to_dev(x, dev)
    y = _run(pkg, v, xt, n, k, to_dev(wb, dev), to_dev(ws, dev), False).cpu().numpy()
    y64, sc = _expected(oracle, v, xt, n, k, wb, ws, False)
    for r in (slice(0, 1), slice(m // 2, m // 2 + 1), slice(1, 2)):
        cond, rel = errors(y[r], y64[r], sc[r])
        assert cond <= 1e-5 and rel <= 1e-3, (r, cond, rel)


@pytest.mark.parametrize("v", [1, 2, 3])
@pytest.mark.parametrize("m,n,k,dtype", [(12, 1100, 4096, "f16"), (130, 1500, 2048, "f16"),
                                         (130, 1500, 2048, "bf16"), (300, 8000, 520, "f32")])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_non_finite_x(pkg, cabi, oracle, inputs, dev, v, m, n, k, dtype, bad):  # noqa: F811
    """A NaN or an infinity reaches its row as in the reference (NaN where it meets a weight of
    0) and no other row."""
    code = {"f32": cabi.CMK_F32, "f16": cabi.CMK_F16, "bf16": cabi.CMK_BF16}[dtype]
    assert cabi.matmul_kernel(code, m, n, k, variant=v)["kernel"] == "register_matmul"
    wb, ws = _weights(oracle, v, n, k, seed=m)
    x = inputs.synthetic_x(m, k, seed=k)
    x[m // 2, 100] = bad
    xt = x_tensor(x, _DT[dtype], dev)
    y = _run(pkg, v, xt, n, k, to_dev(wb, dev), to_dev(ws, dev), False).cpu().numpy()
    row = np.ascontiguousarray(xt[m // 2:m // 2 + 1].float().cpu().numpy())
    ref = oracle.variant_matmul_reference(v, row, 1, n, k, wb, ws).reshape(n)
    got = y[m // 2]
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(np.isposinf(got), np.isposinf(ref))
    assert np.array_equal(np.isneginf(got), np.isneginf(ref))
    assert np.isfinite(np.delete(y, m // 2, axis=0)).all()
