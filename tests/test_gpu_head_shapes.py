"""The head's forward and backward against the float64 oracle where its forms
change: lanes per row (4 to 64), float4 and scalar columns, more than 256
columns, one and several row ranges; and the loss around the size one block
reduces."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rel(a, b):
    a = np.asarray(a, dtype=np.float64)
    b = np.asarray(b, dtype=np.float64)
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-30))


@pytest.mark.parametrize("rows,hidden", [(1, 1), (5, 16), (4097, 15), (1030, 20), (300, 33), (77, 64), (65, 129),
                                         (9000, 128), (257, 256), (64, 260), (130, 768), (33, 767)])
@pytest.mark.parametrize("offset", [0, 1])  # floats past a 16-byte boundary
def test_head_forms_match_oracle(gpu, oracle, hip_lib, rows, hidden, offset):
    from rnn_kernel_amd import _lib

    print(f"head rows={rows} hidden={hidden} offset={offset}", flush=True)
    g = torch.Generator().manual_seed(rows + hidden)
    out = torch.randn(rows, hidden, generator=g)
    w = torch.randn(1, hidden, generator=g) / hidden ** 0.5
    b = torch.randn(1, generator=g)
    dpred = torch.randn(rows, generator=g)
    buf = torch.empty(rows * hidden + 1, device=gpu)[offset:offset + rows * hidden].copy_(out.flatten())
    dout = torch.full((rows * hidden + 1,), float("nan"), device=gpu)[offset:offset + rows * hidden]
    wd, bd, dp = w.to(gpu), b.to(gpu), dpred.to(gpu)
    pred, dw, db = torch.empty(rows, device=gpu), torch.empty(hidden, device=gpu), torch.empty(1, device=gpu)
    nbytes = hip_lib.rka_head_backward_workspace_bytes(rows, hidden)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=gpu)
    stream = torch.cuda.current_stream().cuda_stream
    _lib.check(hip_lib.rka_head_forward(buf.data_ptr(), wd.data_ptr(), bd.data_ptr(), pred.data_ptr(), rows, hidden,
                                        stream), "rka_head_forward")
    _lib.check(hip_lib.rka_head_backward(buf.data_ptr(), wd.data_ptr(), dp.data_ptr(), dout.data_ptr(), dw.data_ptr(),
                                         db.data_ptr(), ws.data_ptr(), nbytes, rows, hidden, stream),
               "rka_head_backward")
    torch.cuda.synchronize()
    ref = oracle.head_forward(out.numpy(), w.numpy(), b.numpy())
    rdout, rdw, rdb = oracle.head_backward(out.numpy(), w.numpy(), dpred.numpy())
    assert _rel(pred.cpu(), ref) <= 1e-5
    assert _rel(dout.cpu().view(rows, hidden), rdout) <= 1e-6
    assert _rel(dw.cpu(), rdw) <= 1e-5
    # a float32 sum of `rows` values is within rows * 2^-24 of their absolute sum
    assert abs(db.item() - rdb) <= rows * 2.0 ** -24 * float(dpred.double().abs().sum()) + 1e-7


@pytest.mark.parametrize("n", [3, 4096, 16383, 16384, 16385])
def test_mse_around_one_block(gpu, oracle, n):
    from rnn_kernel_amd import mse_loss

    g = torch.Generator().manual_seed(n)
    pred, target = torch.randn(n, generator=g), torch.randn(n, generator=g)
    loss = mse_loss(pred.to(gpu), target.to(gpu))
    ref = oracle.mse_forward(pred.numpy(), target.numpy())
    assert abs(loss.item() - ref) <= 1e-5 * max(ref, 1e-3)
