"""The direct products' fp32 tile forms (128x128 ring, 128x64, 64x64 and 32x32
register-staged tiles) against float64 at the edges of each, on aligned and
unaligned storage.  The ring takes row-major products under
RKA_GEMM_TILES_128 only."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# m, n, k: 32x32 tiles (one row, partial tiles, k below, at and past one and two
# 64-deep stages, several tiles per CU) and, at (8200, 192, 32), 128x64 ones
SHAPES = [(1, 768, 256), (1, 1, 3), (33, 31, 64), (31, 65, 65), (200, 96, 128), (64, 100, 130), (50, 40, 4),
          (8192, 130, 16), (8200, 192, 32), (8192, 188, 52), (16500, 129, 17), (33000, 65, 33)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("b_kmajor", [0, 1])
@pytest.mark.parametrize("pad", [0, 1])  # floats between rows and before the first: not 16-byte aligned
def test_direct_product_tiles_match_float64(gpu, hip_lib, m, n, k, b_kmajor, pad):
    _check_direct(gpu, hip_lib, m, n, k, b_kmajor, pad)


# tile mode, form, floats between rows and before the first, m, n, k: the last
# tiles partial along m and n; k of less than one 16-deep stage, of one, two, a part
# more and of many
FORMS = [(0, "64x64", 0, 12600, 36, 4), (0, "64x64", 0, 16400, 252, 36), (0, "64x64", 0, 8300, 512, 256),
         (0, "64x64", 1, 13657, 33, 1), (0, "64x64", 1, 16385, 255, 34), (0, "64x64", 1, 8200, 513, 387),
         (0, "128x64", 0, 24612, 36, 4), (0, "128x64", 0, 8200, 192, 32), (0, "128x64", 0, 8196, 188, 260),
         (0, "128x64", 1, 26747, 35, 1), (0, "128x64", 1, 24613, 37, 33),
         (1, "ring", 0, 1, 4, 4), (1, "ring", 0, 300, 200, 52), (1, "ring", 0, 1028, 388, 16),
         (1, "ring", 1, 31, 65, 65), (1, "ring", 1, 1000, 390, 70), (1, "ring", 1, 129, 1, 3)]


@pytest.mark.parametrize("mode,form,pad,m,n,k", FORMS)
@pytest.mark.parametrize("b_kmajor", [0, 1])
def test_direct_product_forms_match_float64(gpu, hip_lib, mode, form, pad, m, n, k, b_kmajor):
    from rnn_kernel_amd import _lib

    try:
        _lib.set_gemm_tiles(mode)
        assert _lib.describe_gemm(m, n, k, aligned=pad == 0) == form
        _check_direct(gpu, hip_lib, m, n, k, b_kmajor, pad)
    finally:
        _lib.set_gemm_tiles(0)


def _check_direct(gpu, hip_lib, m, n, k, b_kmajor, pad):
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
