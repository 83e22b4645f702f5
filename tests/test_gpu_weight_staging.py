"""The forward recurrences' two ways of reading W_hh (whole rows through LDS,
or each lane its own entries) give the same bits: aligned weights take the
first at short sequences, weights one float past a 16-byte boundary always the
second."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# one to four slices, whole and partial, at one, two and four rows per
# workgroup; three slices on both sides of the sequence length where aligned
# weights change over
@pytest.mark.parametrize("B,T,H", [(3, 4, 64), (2, 3, 40), (5, 4, 128), (4, 3, 100), (3, 5, 192), (2, 3, 132),
                                   (2, 600, 192), (2, 601, 192), (3, 4, 256), (2, 3, 196), (70, 3, 256), (120, 3, 132),
                                   (300, 3, 128), (200, 3, 244)])
def test_weight_reads_agree_bitwise(gpu, hip_lib, B, T, H):
    from rnn_kernel_amd import _lib

    print(f"weights B={B} T={T} H={H} {_lib.describe_recurrence(0, B, H)}", flush=True)
    g = torch.Generator().manual_seed(B + T + H)
    gx, h0, bhh = (torch.randn(*s, generator=g).to(gpu) for s in ((B, T, 3 * H), (B, H), (3 * H,)))
    w = (torch.rand(3 * H, H, generator=g) * 2 - 1) / H ** 0.5
    nb = hip_lib.rka_gru_recurrence_workspace_bytes(B, H)
    ws = torch.empty(nb, dtype=torch.uint8, device=gpu)
    out = []
    for off in (0, 1):
        wd = torch.empty(3 * H * H + 4, device=gpu)[off:off + 3 * H * H].copy_(w.flatten())
        y, hn, res = (torch.empty(*s, device=gpu) for s in ((B, T, H), (B, H), (B, T, 4 * H)))
        _lib.check(hip_lib.rka_gru_recurrence_forward(gx.data_ptr(), h0.data_ptr(), wd.data_ptr(), bhh.data_ptr(),
                                                      y.data_ptr(), hn.data_ptr(), res.data_ptr(), ws.data_ptr(), nb,
                                                      B, T, H, torch.cuda.current_stream().cuda_stream), "forward")
        torch.cuda.synchronize()
        out.append((y, hn, res))
    for a, b in zip(*out):
        assert not torch.isnan(a).any()
        assert torch.equal(a, b)
