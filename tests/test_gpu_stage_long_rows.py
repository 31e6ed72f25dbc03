"""Staging of more than 512 rows past 16384 columns, which workgroups of 1024 hold, and of rows
past 32768, which are read twice: against the fp64 oracle, bars of test_gpu_parity.py."""

import pytest
import torch

from test_gpu_mm import _DT, _expected, _run
from test_gpu_parity import x_tensor
from test_gpu_variants import dev, errors, random_weights, to_dev  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k", [(513, 16384), (513, 16392), (530, 32768), (513, 32776)])
@pytest.mark.parametrize("dtype,w8a8", [("f32", False), ("bf16", False), ("f16", True)])
def test_long_rows(pkg, oracle, inputs, dev, m, k, dtype, w8a8):  # noqa: F811
    n, v = 2, 1
    wb, ws = random_weights(oracle, v, n, k, seed=k)
    x = x_tensor(inputs.synthetic_x(m, k, seed=m), _DT[dtype], dev)
    y = _run(pkg, v, x, n, k, to_dev(wb, dev), to_dev(ws, dev), w8a8).cpu().numpy()
    cond, rel = errors(y, *_expected(oracle, v, x, n, k, wb, ws, w8a8))
    assert cond <= 1e-5 and rel <= 1e-3, (cond, rel)
