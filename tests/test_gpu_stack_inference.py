"""Inference through a stack in one library call equals the layers called one
by one, bit for bit, and raises what they raise."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,B,T,I,H", [(1, 1, 1, 3, 5), (2, 3, 7, 16, 33), (3, 5, 1, 9, 256), (4, 2, 9, 20, 130),
                                       (5, 4, 3, 8, 300)])
@pytest.mark.parametrize("strided", [False, True])
def test_stack_equals_layer_by_layer(gpu, L, B, T, I, H, strided):
    from rnn_kernel_amd import GRU, gru_forward_inference

    torch.manual_seed(L * 100 + H)
    model = GRU(I, H, num_layers=L).to(gpu)
    x = torch.randn(B, T, I, device=gpu)
    hx = torch.randn(L, B, H, device=gpu)
    if strided:
        x = torch.randn(T, B, 2 * I, device=gpu)[:, :, ::2].transpose(0, 1)
        hx = torch.randn(B, L, H, device=gpu).transpose(0, 1)
    with torch.no_grad():
        out, hn = model(x, hx)
    seq, states = x, []
    for k in range(L):
        seq, h = gru_forward_inference(seq, hx[k], *model._layer_parameters(k))
        states.append(h)
    assert torch.equal(out, seq) and torch.equal(hn, torch.cat(states, dim=0))
    out2, hn2 = model.forward_inference(x.clone().requires_grad_(True), hx)
    assert not out2.requires_grad and torch.equal(out2, out) and torch.equal(hn2, hn)


def test_stack_rejects_what_the_layers_reject(gpu):
    from rnn_kernel_amd import GRU

    model = GRU(4, 8, num_layers=2).to(gpu)
    x = torch.randn(2, 3, 4, device=gpu)
    with torch.no_grad():
        with pytest.raises(RuntimeError, match="GPU"):
            model(x.cpu())
        with pytest.raises(RuntimeError, match="fp32"):
            model(x.double())
        with pytest.raises(ValueError, match="weight_ih"):
            model(torch.randn(2, 3, 5, device=gpu))
        with pytest.raises(ValueError, match="same CUDA device"):
            model(x, torch.zeros(2, 2, 8))
        with pytest.raises(ValueError, match=">= 1"):
            model(x[:, :0])
        model.weight_hh_l1.data = model.weight_hh_l1.data.double()
        with pytest.raises(RuntimeError, match="fp32"):
            model(x)
