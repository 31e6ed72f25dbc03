"""The register-dequantising MFMA matmul at the edges of its 32-row tiles (test_gpu_mm_tiles.py
has the wider ones): one and several super-blocks (the parts of K that waves share run out
unevenly), partial and odd K, staged rows of every type, W8A8, and less scratch than it would
like.  The smallest shapes stay on the decode launches, in IQ2_XXS more of them.

Bar: exact weights and fp32 sums, so the bars of the decode kernels hold: cond <= 1e-5 and
rel <= 1e-3 against the fp64 oracle (test_gpu_parity.py).  IQ2_XXS above 16 rows (W8A8 32)
of K a multiple of 8 has weights rounded once to f16, as the GEMM has: there the same bar
holds against the product with those weights.
"""

import numpy as np
import pytest
import torch

from test_gpu_parity import x_as_f32, x_tensor
from test_gpu_variants import dev, errors, random_weights, to_dev  # noqa: F401

pytestmark = pytest.mark.gpu

_DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
FORMATS = [0, 1, 2, 3]


def _expected(oracle, v, x, n, k, wb, ws, w8a8, exact=False):
    m = x.shape[0]
    xf = np.ascontiguousarray(x_as_f32(x), np.float32)
    if w8a8:
        xf = np.ascontiguousarray(oracle.rowwise_qdq_w8a8(xf, xf.shape[0], k), np.float32)
    if v == 0 and not exact and k % 8 == 0 and m > (32 if w8a8 else 16):
        w = oracle.dequantize_f16_bits(wb, ws, n, k).view(np.float16).reshape(n, k)
        w = w.astype(np.float64)
        return xf @ w.T, np.abs(xf) @ np.abs(w).T
    if v == 0:
        return oracle.matmul_f64(xf, xf.shape[0], n, k, wb, ws)
    return oracle.variant_matmul_f64(v, xf, xf.shape[0], n, k, wb, ws)


def _run(pkg, v, x, n, k, wb, ws, w8a8):
    ve = pkg.Iq2MatmulVariant(v)
    if w8a8:
        cfg = pkg.ActivationQuantConfig(pkg.ActivationQuantMode.W8A8, False)
        return pkg.iq2_matmul_with_activation_quant(x, wb, ws, n, k, ve, cfg)
    return pkg.iq2_matmul(x, wb, ws, n, k, ve)


@pytest.mark.parametrize("v", FORMATS)
@pytest.mark.parametrize("m,n,k,dtype,w8a8", [
    (9, 1, 8, "f16", False), (17, 31, 256, "f16", False), (32, 64, 1024, "f16", False),
    (33, 65, 1288, "f16", False), (64, 129, 2048, "f16", False), (65, 257, 520, "f16", False),
    (128, 256, 768, "f16", False), (129, 100, 4104, "f16", False), (300, 70, 512, "f16", False),
    (20, 96, 2051, "f16", False), (40, 333, 777, "bf16", False), (16, 64, 4096, "bf16", False),
    (65, 130, 1000, "f32", False), (12, 33, 2872, "f32", False), (17, 40, 515, "f32", False),
    (20, 600, 2051, "f16", False), (16, 300, 4096, "bf16", False), (12, 400, 2872, "f32", False),
    (17, 2050, 515, "f32", False),
    (33, 96, 1024, "f16", True), (70, 65, 1291, "bf16", True), (130, 64, 2304, "f32", True)])
def test_tile_edges(pkg, oracle, inputs, dev, v, m, n, k, dtype, w8a8):  # noqa: F811
    wb, ws = random_weights(oracle, v, n, k, seed=m + 3 * n + k)
    x = x_tensor(inputs.synthetic_x(m, k, seed=m + k), _DT[dtype], dev)
    wbt, wst = to_dev(wb, dev), to_dev(ws, dev)
    y = _run(pkg, v, x, n, k, wbt, wst, w8a8)
    again = _run(pkg, v, x, n, k, wbt, wst, w8a8)
    assert torch.equal(y, again)
    cond, rel = errors(y.cpu().numpy(), *_expected(oracle, v, x, n, k, wb, ws, w8a8))
    assert cond <= 1e-5 and rel <= 1e-3, (cond, rel)


@pytest.mark.parametrize("v,share", [(v, s) for v in (1, 2, 3) for s in (0.0, 0.4, 0.7, 1.0)])
def test_scratch_limits(pkg, cabi, oracle, inputs, dev, v, share):  # noqa: F811
    """Any workspace serves: all rows at once, passes of whole tiles, or the decode
    launches; nothing past the workspace's end is touched."""
    m, n, k = 290, 96, 520
    wb, ws = random_weights(oracle, v, n, k, seed=v)
    x = x_tensor(inputs.synthetic_x(m, k, seed=9), torch.float32, dev)
    wbt, wst = to_dev(wb, dev), to_dev(ws, dev)
    need = cabi.workspace_size(cabi.CMK_F32, m, n, k, v)
    assert need > 0
    have = int(need * share) // 16 * 16
    work = torch.full((have + 256,), 0x5A, dtype=torch.uint8, device=dev)
    out = torch.full((m + 1, n), -7.0, device=dev)
    cabi.matmul_raw(x.data_ptr(), cabi.CMK_F32, x.numel(), m, wbt.data_ptr(), wbt.numel(),
                    wst.data_ptr(), wst.numel(), n, k, out.data_ptr(), v, cabi.CMK_ACT_QUANT_OFF,
                    False, work.data_ptr() if have else None, have, None)
    y = out.cpu().numpy()
    assert (y[m] == -7.0).all()
    assert (work[have:].cpu().numpy() == 0x5A).all()
    cond, rel = errors(y[:m], *_expected(oracle, v, x, n, k, wb, ws, False))
    assert cond <= 1e-5 and rel <= 1e-3, (cond, rel)


@pytest.mark.parametrize("v", FORMATS)
def test_unaligned_rows(pkg, cabi, oracle, inputs, dev, v):  # noqa: F811
    """f16 rows that start 2 bytes off: copied to aligned rows in the workspace (IQ2_XXS with
    exact weights, as the decode kernel serves such rows without one)."""
    m, n, k = 40, 70, 520
    wb, ws = random_weights(oracle, v, n, k, seed=v + 50)
    x = x_tensor(inputs.synthetic_x(m, k, seed=3), torch.float16, dev)
    big = torch.zeros(m * k + 1, dtype=torch.float16, device=dev)
    big[1:] = x.reshape(-1)
    y = _run(pkg, v, big[1:].view(m, k), n, k, to_dev(wb, dev), to_dev(ws, dev), False)
    cond, rel = errors(y.cpu().numpy(), *_expected(oracle, v, x, n, k, wb, ws, False, exact=True))
    assert cond <= 1e-5 and rel <= 1e-3, (cond, rel)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_more_rows_than_one_launch_holds(pkg, oracle, dev, dtype):  # noqa: F811
    """Rows past what grid y counts in 32-row tiles, and past 2^32 threads of one staging
    workgroup a row: every row is one of 8, so every output row is known."""
    m, n, k, v = (1 << 24) + 40, 2, 8, 1
    wb, ws = random_weights(oracle, v, n, k, seed=11)
    kinds = torch.randn(8, k, generator=torch.Generator().manual_seed(5)).to(_DT[dtype])
    x = kinds.to(dev).repeat(m // 8, 1)
    y = _run(pkg, v, x, n, k, to_dev(wb, dev), to_dev(ws, dev), False).view(m // 8, 8, n)
    assert bool((y == y[0]).all())
    cond, rel = errors(y[0].cpu().numpy(), *_expected(oracle, v, kinds, n, k, wb, ws, False))
    assert cond <= 1e-5 and rel <= 1e-3, (cond, rel)
