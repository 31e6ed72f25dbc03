"""The register-dequantising matmul in several passes of staged rows: more rows than one pass
takes (256 MB of them), the last pass a short one."""

import pytest
import torch

from test_gpu_mm import _expected, _run
from test_gpu_parity import x_tensor
from test_gpu_variants import dev, errors, random_weights, to_dev  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("v", [0, 3])
def test_last_pass_short(pkg, oracle, inputs, dev, v):  # noqa: F811
    m, n, k = 2304 + 70, 40 if v == 0 else 2, 28670  # (IQ2_XXS from 2^20 weights of odd K)
    wb, ws = random_weights(oracle, v, n, k, seed=v)
    few = inputs.synthetic_x(8, k, seed=3)  # every row is one of 8
    x = x_tensor(few, torch.float32, dev).repeat(m // 8 + 1, 1)[:m].contiguous()
    y = _run(pkg, v, x, n, k, to_dev(wb, dev), to_dev(ws, dev), False)
    for r0, r1 in ((0, 8), (2304, 2312)):
        cond, rel = errors(y[r0:r1].cpu().numpy(),
                           *_expected(oracle, v, x[:8], n, k, wb, ws, False, exact=True))
        assert cond <= 1e-5 and rel <= 1e-3, (cond, rel)
    whole = m // 8 * 8
    tiles = y[:whole].view(-1, 8, n)
    first = 2304 // 8
    assert bool((tiles[:first] == tiles[0]).all()) and bool((tiles[first:] == tiles[first]).all())
