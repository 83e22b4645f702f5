"""The direct products' tile forms (128x128 ring, 128x64, 64x64 and 32x32
register-staged tiles) against float64 at the edges of each, and the rule
between them on aligned and unaligned storage."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# m, n, k: 32x32 tiles with one row, partial tiles, k below, at and past one
# and two 64-deep stages; 64x64 and 128x64 tiles (more than one tile per CU, the
# last ones partial; k of one, two, three and a partial 16-deep stage)
SHAPES = [(1, 768, 256), (1, 1, 3), (33, 31, 64), (31, 65, 65), (200, 96, 128), (64, 100, 130), (50, 40, 4),
          (8192, 130, 16), (8200, 192, 32), (8192, 188, 52), (16500, 129, 17), (33000, 65, 33)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("b_kmajor", [0, 1])
@pytest.mark.parametrize("pad", [0, 1])  # floats between rows and before the first: not 16-byte aligned
def test_direct_product_tiles_match_float64(gpu, hip_lib, m, n, k, b_kmajor, pad):
    from rnn_kernel_amd import _lib

    print(f"direct m={m} n={n} k={k} b_kmajor={b_kmajor} pad={pad}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(m + n + k)

    def stored(rows, cols):
        # NaN around the matrix: nothing past an operand may reach the result
        buf = torch.full((rows * (cols + pad) + 2 * pad,), float("nan"), device=gpu)
        view = buf[pad:pad + rows * (cols + pad)].view(rows, cols + pad)[:, :cols]
        view.copy_(torch.randn(rows, cols, generator=g, device=gpu))
        return buf, view

    a_buf, a = stored(m, k)
    b_buf, b = stored(k, n) if b_kmajor else stored(n, k)
    bias = torch.randn(n, generator=g, device=gpu)
    c = torch.full((m + 1, n), float("nan"), device=gpu)
    rc = hip_lib.rka_gemm_f32(m, n, k, a.data_ptr(), k + pad, 0, b.data_ptr(), (n if b_kmajor else k) + pad, b_kmajor,
                              bias.data_ptr(), c.data_ptr(), n, torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "rka_gemm_f32")
    ref = a.double() @ (b.double() if b_kmajor else b.double().t().contiguous()) + bias.double()
    assert (c[:m].double() - ref).abs().max().item() <= 1e-6 * k + 1e-5
    assert torch.isnan(c[m]).all()  # nothing stored past the last row


@pytest.mark.parametrize("k", [1028, 1029])  # float4 and single loads of the row-major operand
def test_direct_product_of_a_wide_k_major_operand(gpu, hip_lib, k):
    """k rows of 2^20 floats are more than 2^32 bytes: offsets within a stage
    must not be limited by the whole extent taken in 32 bits."""
    from rnn_kernel_amd import _lib

    m, n, ld = 64, 64, 1 << 20
    g = torch.Generator(device=gpu).manual_seed(k)
    a = torch.randn(m, k, generator=g, device=gpu)
    b = torch.zeros(k, ld, device=gpu)
    b[:, :n] = torch.randn(k, n, generator=g, device=gpu)
    c = torch.empty(m, n, device=gpu)
    rc = hip_lib.rka_gemm_f32(m, n, k, a.data_ptr(), k, 0, b.data_ptr(), ld, 1, None, c.data_ptr(), n,
                              torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "rka_gemm_f32")
    ref = a.double() @ b[:, :n].double().contiguous()
    assert (c.double() - ref).abs().max().item() <= 1e-6 * k + 1e-5


@pytest.mark.parametrize("m,n", [((1 << 29) - 1, 3), ((1 << 30) + 33, 1)])
def test_direct_product_of_very_many_rows(gpu, hip_lib, m, n):
    """So many rows that 32x32 tiles (the second: 64x64 ones too) would be a
    launch of 2^32 threads: a form of larger tiles takes the product."""
    from rnn_kernel_amd import _lib

    print(f"direct m={m} n={n}", flush=True)
    a = torch.arange(m, device=gpu, dtype=torch.float32).remainder_(1021.0)
    b = torch.arange(1, n + 1, device=gpu, dtype=torch.float32)
    c = torch.empty(m, n, device=gpu)
    rc = hip_lib.rka_gemm_f32(m, n, 1, a.data_ptr(), 1, 0, b.data_ptr(), 1, 0, None, c.data_ptr(), n,
                              torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "rka_gemm_f32")
    for r in range(0, m, 1 << 27):
        assert torch.equal(c[r:r + (1 << 27)], a[r:r + (1 << 27), None] * b)
