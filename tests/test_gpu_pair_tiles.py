"""The weight-gradient products where their form or number of slices changes,
against float64 sums of the gate gradients that the library itself returns:
one slice (the results written by the products' own launch), few, and a
multiple of 8; sequences shorter than a 16-deep stage and of one step (the
[h0 ; y[:, :-1]] rows); a last slice shorter than the others; aligned and
unaligned rows; 64x64, 128x64 and split tiles, and under RKA_GEMM_TILES_128 the
ring with its narrow last columns."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1, 1), (2, 3, 5, 7), (127, 1, 16, 20), (128, 1, 12, 64), (9, 14, 33, 65), (5, 100, 100, 100),
          (40, 25, 64, 128), (7, 300, 129, 129), (16, 520, 128, 256), (33, 331, 16, 64), (16, 2001, 256, 256), (61, 500, 132, 260),
          (64, 512, 129, 129), (61, 500, 131, 255), (16, 2001, 257, 513)]


@pytest.mark.parametrize("B,T,I,H", SHAPES)
@pytest.mark.parametrize("need_dx", [True, False])
def test_weight_gradients_match_float64(gpu, hip_lib, B, T, I, H, need_dx):
    _check_pair(gpu, hip_lib, B, T, I, H, need_dx)


# tile mode, form, whether one launch writes the results, B, T, I, H.  The ring: one
# tile, several, 5, 7 and 8 last columns summed apart (in 32 slices and in one), the
# remainder just too wide for that
FORMS = [(0, "64x64", True, 3, 5, 4, 4), (0, "64x64", False, 21, 25, 36, 68), (0, "64x64", False, 23, 47, 35, 67),
         (0, "128x64", False, 99, 376, 2, 66), (0, "split", False, 16, 129, 204, 584),
         (0, "split", False, 15, 52, 595, 342), (0, "split", False, 121, 149, 5, 65),
         (1, "ring", False, 3, 5, 4, 4), (1, "ring", False, 9, 14, 33, 65), (1, "ring", False, 40, 25, 64, 128),
         (1, "ring", False, 8, 512, 135, 133), (1, "ring", False, 2, 70, 136, 136), (1, "ring", False, 3, 50, 137, 140),
         (1, "ring", False, 7, 300, 129, 129)]


@pytest.mark.parametrize("mode,form,direct,B,T,I,H", FORMS)
@pytest.mark.parametrize("need_dx", [True, False])
def test_weight_gradient_forms_match_float64(gpu, hip_lib, mode, form, direct, B, T, I, H, need_dx):
    from rnn_kernel_amd import _lib

    try:
        _lib.set_gemm_tiles(mode)
        d = _lib.describe_weight_gradients(B, T, I, H)
        assert (d["form"], d["direct"]) == (form, direct)
        _check_pair(gpu, hip_lib, B, T, I, H, need_dx)
    finally:
        _lib.set_gemm_tiles(0)


def _check_pair(gpu, hip_lib, B, T, I, H, need_dx):
    from rnn_kernel_amd import _lib

    print(f"pair B={B} T={T} I={I} H={H} dx={need_dx}", flush=True)
    gen = torch.Generator(device=gpu).manual_seed(B + T + I + H)

    def randn(*shape):
        return torch.randn(*shape, generator=gen, device=gpu)

    x, h0, y, dy, dhn = randn(B, T, I), randn(B, H), torch.tanh(randn(B, T, H)), randn(B, T, H), randn(B, H)
    w_ih, w_hh = 0.1 * randn(3 * H, I), 0.1 / H ** 0.5 * randn(3 * H, H)
    res = torch.sigmoid(randn(B, T, H, 4))
    stream = torch.cuda.current_stream().cuda_stream
    g, dh0 = torch.empty(B, T, 4, H, device=gpu), torch.empty(B, H, device=gpu)
    nb = hip_lib.rka_gru_recurrence_workspace_bytes(B, H)
    ws = torch.empty(nb, dtype=torch.uint8, device=gpu)
    _lib.check(hip_lib.rka_gru_recurrence_backward(dy.data_ptr(), dhn.data_ptr(), res.data_ptr(), h0.data_ptr(),
                                                   y.data_ptr(), w_hh.data_ptr(), g.data_ptr(), dh0.data_ptr(),
                                                   ws.data_ptr(), nb, B, T, H, stream), "recurrence_backward")
    nan = float("nan")
    dx = torch.full((B, T, I), nan, device=gpu)
    dw_ih, dw_hh = torch.full((3 * H, I), nan, device=gpu), torch.full((3 * H, H), nan, device=gpu)
    db_ih, db_hh = torch.full((3 * H,), nan, device=gpu), torch.full((3 * H,), nan, device=gpu)
    nb = hip_lib.rka_gru_backward_workspace_bytes(B, T, I, H)
    ws = torch.empty(nb, dtype=torch.uint8, device=gpu)
    _lib.check(hip_lib.rka_gru_backward(x.data_ptr(), h0.data_ptr(), w_ih.data_ptr(), w_hh.data_ptr(), y.data_ptr(),
                                        res.data_ptr(), dy.data_ptr(), dhn.data_ptr(), dx.data_ptr() if need_dx else None,
                                        dh0.data_ptr(), dw_ih.data_ptr(), dw_hh.data_ptr(), db_ih.data_ptr(),
                                        db_hh.data_ptr(), ws.data_ptr(), nb, B, T, I, H, stream), "backward")
    # G = (da_n, dr^, dz^, dn^) per step
    G = g.double().view(B * T, 4 * H)
    g_ih = G[:, H:]
    g_hh = torch.cat([G[:, H:3 * H], G[:, :H]], dim=1)
    hprev = torch.cat([h0[:, None], y[:, :-1]], dim=1).double().reshape(B * T, H)
    # a float32 sum of n products, in chains of at most 4096 (to n = 2^20) and their
    # sum, is within (4096 + 256) 2^-24 of the sum of the products' magnitudes
    n = min(B * T, 4352)
    for name, out, a, b in (("dw_ih", dw_ih, g_ih, x.double().reshape(B * T, I)), ("dw_hh", dw_hh, g_hh, hprev),
                            ("db_ih", db_ih, g_ih, None), ("db_hh", db_hh, g_hh, None)):
        if b is None:
            ref, mag = a.sum(0), a.abs().sum(0)
        else:
            ref, mag = a.t().contiguous() @ b, a.abs().t().contiguous() @ b.abs()
        assert bool(((out.double() - ref).abs() <= n * 2.0 ** -24 * mag + 1e-30).all()), name
    if need_dx:
        ref = (g_ih @ w_ih.double()).view(B, T, I)
        mag = (g_ih.abs() @ w_ih.double().abs()).view(B, T, I)
        assert bool(((dx.double() - ref).abs() <= 3 * H * 2.0 ** -24 * mag + 1e-30).all())


# sizes whose few long slices had chains of up to 4096 additions; B, T, I, H
@pytest.mark.parametrize("B,T,I,H", [(16, 256, 256, 256), (236, 19, 12, 412), (6, 549, 2, 389), (115, 155, 1, 242),
                                     (164, 51, 51, 130), (75, 258, 3, 308), (6, 1622, 12, 653)])
def test_weight_gradients_are_no_further_off_than_the_ring(gpu, hip_lib, B, T, I, H):
    """Error against float64 (2-norm) of the chosen form at most that of the
    128x128 ring's short slices (one fifth more: two samples of rounding)."""
    from rnn_kernel_amd import _lib

    print(f"pair B={B} T={T} I={I} H={H}", flush=True)
    gen = torch.Generator(device=gpu).manual_seed(B + T + I + H)

    def randn(*shape):
        return torch.randn(*shape, generator=gen, device=gpu)

    x, h0, y, dy = randn(B, T, I), randn(B, H), torch.tanh(randn(B, T, H)), randn(B, T, H)
    w_ih, w_hh, res = 0.1 * randn(3 * H, I), 0.1 / H ** 0.5 * randn(3 * H, H), torch.sigmoid(randn(B, T, H, 4))
    stream = torch.cuda.current_stream().cuda_stream
    g, dh0 = torch.empty(B, T, 4, H, device=gpu), torch.empty(B, H, device=gpu)
    nb = hip_lib.rka_gru_recurrence_workspace_bytes(B, H)
    ws = torch.empty(nb, dtype=torch.uint8, device=gpu)
    _lib.check(hip_lib.rka_gru_recurrence_backward(dy.data_ptr(), None, res.data_ptr(), h0.data_ptr(), y.data_ptr(),
                                                   w_hh.data_ptr(), g.data_ptr(), dh0.data_ptr(), ws.data_ptr(), nb, B,
                                                   T, H, stream), "recurrence_backward")
    G = g.double().view(B * T, 4 * H)
    g_ih, g_hh = G[:, H:], torch.cat([G[:, H:3 * H], G[:, :H]], dim=1)
    hprev = torch.cat([h0[:, None], y[:, :-1]], dim=1).double().reshape(B * T, H)
    refs = (g_ih.t().contiguous() @ x.double().reshape(B * T, I), g_hh.t().contiguous() @ hprev)
    nb = hip_lib.rka_gru_backward_workspace_bytes(B, T, I, H)
    ws = torch.empty(nb, dtype=torch.uint8, device=gpu)

    def errors(mode):
        # (a pair that the split form takes runs in it in either mode: then
        # unaligned sizes of the same slices are compared with themselves)
        _lib.set_gemm_tiles(mode)
        out = [torch.empty(*s, device=gpu) for s in ((3 * H, I), (3 * H, H), (3 * H,), (3 * H,))]
        _lib.check(hip_lib.rka_gru_backward(x.data_ptr(), h0.data_ptr(), w_ih.data_ptr(), w_hh.data_ptr(), y.data_ptr(),
                                            res.data_ptr(), dy.data_ptr(), None, None, dh0.data_ptr(),
                                            *[o.data_ptr() for o in out], ws.data_ptr(), nb, B, T, I, H, stream),
                   "backward")
        return [((o.double() - r).norm() / r.norm()).item() for o, r in zip(out, refs)]

    try:
        ring, own = errors(1), errors(0)
    finally:
        _lib.set_gemm_tiles(0)
    assert all(e <= 1.2 * r for e, r in zip(own, ring)), (own, ring)


def test_tile_mode_changed_by_another_thread(gpu, hip_lib):
    """A call takes its plan once: with another thread switching the tile mode
    all along, a pass with one slice per product (whose launch writes the
    results itself, or leaves partial sums to a reduction) gives one mode's
    weight gradients or the other's, never unwritten ones."""
    from rnn_kernel_amd import _lib

    B, T, I, H = 2, 8, 16, 16
    gen = torch.Generator(device=gpu).manual_seed(4)

    def randn(*shape):
        return torch.randn(*shape, generator=gen, device=gpu)

    x, h0, y, dy = randn(B, T, I), randn(B, H), torch.tanh(randn(B, T, H)), randn(B, T, H)
    w_ih, w_hh, res = 0.1 * randn(3 * H, I), 0.1 * randn(3 * H, H), torch.sigmoid(randn(B, T, H, 4))
    nb = hip_lib.rka_gru_backward_workspace_bytes(B, T, I, H)
    dx, dh0, nan = torch.empty(B, T, I, device=gpu), torch.empty(B, H, device=gpu), float("nan")

    def run():
        ws = torch.full((nb,), 255, dtype=torch.uint8, device=gpu)  # (NaN where read as float)
        out = [torch.full(s, nan, device=gpu) for s in ((3 * H, I), (3 * H, H), (3 * H,), (3 * H,))]
        _lib.check(hip_lib.rka_gru_backward(x.data_ptr(), h0.data_ptr(), w_ih.data_ptr(), w_hh.data_ptr(), y.data_ptr(),
                                            res.data_ptr(), dy.data_ptr(), None, dx.data_ptr(), dh0.data_ptr(),
                                            *[o.data_ptr() for o in out], ws.data_ptr(), nb, B, T, I, H,
                                            torch.cuda.current_stream().cuda_stream), "backward")
        return torch.cat([o.flatten() for o in out])

    stop = threading.Event()

    def switch():
        mode = 0
        while not stop.is_set():
            mode ^= 1
            hip_lib.rka_set_gemm_tiles(mode)

    thread = threading.Thread(target=switch)
    try:
        want = []
        for mode in (0, 1):
            _lib.set_gemm_tiles(mode)
            want.append(run())
        assert torch.isfinite(want[0]).all() and torch.allclose(want[0], want[1], rtol=1e-5, atol=1e-6)
        thread.start()
        got = [run() for _ in range(600)]
    finally:
        stop.set()
        if thread.is_alive():
            thread.join()
        _lib.set_gemm_tiles(0)
    assert all(any(torch.equal(g, w) for w in want) for g in got)
