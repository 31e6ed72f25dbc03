"""cmk_iq2_matmul_noalloc where the register-dequantising matmul runs: other formats, decode-sized
batches, W8A8; bit for bit cmk_iq2_matmul with a workspace, and where the array is smaller than
what the query reports, cmk_iq2_matmul with a workspace of the array's size."""

import numpy as np
import pytest
import torch

from test_gpu_mm import _DT, _expected
from test_gpu_parity import x_tensor
from test_gpu_variants import dev, errors, random_weights, to_dev  # noqa: F401

pytestmark = pytest.mark.gpu


def _case(cabi, oracle, inputs, dev, v, m, n, k, dtype, w8a8=False):  # noqa: F811
    code = {"f32": cabi.CMK_F32, "f16": cabi.CMK_F16, "bf16": cabi.CMK_BF16}[dtype]
    mode = cabi.CMK_ACT_QUANT_W8A8 if w8a8 else cabi.CMK_ACT_QUANT_OFF
    assert cabi.matmul_kernel(code, m, n, k, variant=v, mode=mode)["kernel"] == "register_matmul"
    host = random_weights(oracle, v, n, k, seed=m + k)
    wb, ws = (to_dev(t, dev) for t in host)
    x = x_tensor(inputs.synthetic_x(m, k, seed=n), _DT[dtype], dev)
    args = (x.data_ptr(), code, x.numel(), m, wb.data_ptr(), wb.numel(), ws.data_ptr(),
            ws.numel(), n, k)
    return (x, wb, ws, host), args, dict(variant=v, mode=mode)


def _with_workspace(cabi, args, kw, size, dev):  # noqa: F811
    work = torch.empty(max(size, 16), dtype=torch.uint8, device=dev)
    out = torch.full((args[3], args[8]), float("nan"), device=dev)
    cabi.matmul_raw(*args, out.data_ptr(), workspace_ptr=work.data_ptr(), workspace_bytes=size, **kw)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("v,m,n,k,dtype,w8a8", [
    (0, 8, 2048, 4096, "f16", False), (0, 12, 2048, 4096, "bf16", False), (0, 24, 700, 1024, "f16", True),
    (1, 16, 1024, 8192, "bf16", False), (2, 6, 1100, 4096, "f16", False), (3, 77, 1001, 2872, "f32", False),
    (1, 24, 1000, 2048, "bf16", True), (3, 300, 2000, 2048, "f16", False)])
def test_equals_workspace_entry_point(pkg, cabi, oracle, inputs, dev, v, m, n, k, dtype, w8a8):  # noqa: F811
    keep, args, kw = _case(cabi, oracle, inputs, dev, v, m, n, k, dtype, w8a8)
    need = cabi.workspace_size(args[1], m, n, k, **kw)
    assert need <= cabi.NOALLOC_SCRATCH_BYTES
    out = torch.full((m, n), float("nan"), device=dev)
    cabi.matmul_noalloc_raw(*args, out.data_ptr(), **kw)
    assert torch.equal(out, _with_workspace(cabi, args, kw, need, dev))


def test_more_than_the_array_runs_in_passes(pkg, cabi, oracle, inputs, dev):  # noqa: F811
    v, m, n, k = 1, 1300, 130, 8192  # 43 MB of staged row pairs
    keep, args, kw = _case(cabi, oracle, inputs, dev, v, m, n, k, "f32")
    assert cabi.workspace_size(args[1], m, n, k, **kw) > cabi.NOALLOC_SCRATCH_BYTES
    passes = cabi.matmul_kernel(args[1], m, n, k, workspace_bytes=cabi.NOALLOC_SCRATCH_BYTES, **kw)
    assert passes["kernel"] == "register_matmul" and passes["rows_per_pass"] < m
    out = torch.full((m, n), float("nan"), device=dev)
    cabi.matmul_noalloc_raw(*args, out.data_ptr(), **kw)
    assert torch.equal(out, _with_workspace(cabi, args, kw, cabi.NOALLOC_SCRATCH_BYTES, dev))
    rows = np.r_[0:20, m - 20:m]
    x, _, _, (wb, ws) = keep
    cond, rel = errors(out.cpu().numpy()[rows], *_expected(oracle, v, x[torch.from_numpy(rows).to(dev)],
                                                         n, k, wb, ws, False))
    assert cond <= 1e-5 and rel <= 1e-3, (cond, rel)


def test_graph_replays(pkg, cabi, oracle, inputs, dev):  # noqa: F811
    """Captured (staging, split of K and its sum); replays between eager calls that write the
    same array."""
    keep, args, kw = _case(cabi, oracle, inputs, dev, 1, 16, 1024, 8192, "bf16")
    assert cabi.matmul_kernel(args[1], 16, 1024, 8192, **kw)["splits"] > 1
    keep2, args2, kw2 = _case(cabi, oracle, inputs, dev, 3, 77, 1001, 2872, "f32")
    ref = _with_workspace(cabi, args, kw, cabi.workspace_size(args[1], 16, 1024, 8192, **kw), dev)
    out = torch.full((16, 1024), float("nan"), device=dev)
    other = torch.empty((77, 1001), device=dev)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        cabi.matmul_noalloc_raw(*args, out.data_ptr(), stream=s.cuda_stream, **kw)  # warm-up
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        cabi.matmul_noalloc_raw(*args, out.data_ptr(), stream=s.cuda_stream, **kw)
    for _ in range(4):
        out.fill_(float("nan"))
        cabi.matmul_noalloc_raw(*args2, other.data_ptr(), **kw2)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)
