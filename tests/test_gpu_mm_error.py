"""Rounding of the register-dequantising matmul against the decode launches it replaces: the
2-norm error against the 64-bit product is no larger, in tiles of 32 rows (16 rows), of 64
(600 rows), and with a long K (28672) and its split.

The decode launches serve the same call when x starts two bytes off its alignment and there
is no workspace (such rows would have to be staged).  Bar: 1.03 times their error; a 2-norm
over at least 16 x 1000 results varies by 1 / sqrt(2 x 16000) < 0.6 % from inputs to inputs.
"""

import pytest
import torch

from test_gpu_variants import dev, random_weights, to_dev  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("v,m,n,k,dtype", [
    (0, 16, 1536, 4096, "f16"), (0, 16, 1000, 28672, "bf16"), (1, 600, 4096, 4096, "f16"),
    (1, 600, 4096, 4096, "bf16"), (2, 16, 1000, 28672, "bf16"), (2, 600, 4096, 4096, "f16"),
    (3, 32, 1000, 28672, "bf16"), (3, 600, 4096, 4096, "f16"), (3, 600, 4096, 4096, "bf16")])
def test_error_no_larger_than_decode_launches(pkg, cabi, oracle, dev, v, m, n, k, dtype):  # noqa: F811
    wb, ws = (to_dev(t, dev) for t in random_weights(oracle, v, n, k, seed=m + v))
    g = torch.Generator(device=dev)
    g.manual_seed(k + v)
    x = torch.randn(m, k, generator=g, device=dev)
    x[:, ::512] *= 12.0  # strong channels
    dt, code = {"f16": (torch.float16, cabi.CMK_F16), "bf16": (torch.bfloat16, cabi.CMK_BF16)}[dtype]
    x = x.to(dt)
    ve = pkg.Iq2MatmulVariant(v)
    w = pkg.iq2_dequantize_to_f16(wb, ws, n, k, ve, out_dtype=torch.float32).double()
    exact = x.double() @ w.T

    def error(y):
        return ((y.double() - exact).norm() / exact.norm()).item()

    shifted = torch.zeros(m * k + 1, dtype=dt, device=dev)
    shifted[1:] = x.reshape(-1)
    decode = torch.empty(m, n, device=dev)
    cabi.matmul_raw(shifted[1:].data_ptr(), code, m * k, m, wb.data_ptr(), wb.numel(),
                    ws.data_ptr(), ws.numel(), n, k, decode.data_ptr(), v)
    here = pkg.iq2_matmul(x, wb, ws, n, k, ve)
    assert not torch.equal(here, decode)  # two kernels
    assert error(here) <= 1.03 * error(decode), (error(here), error(decode))
