"""The large fp32 products on the bf16 matrix cores (three bf16 pieces per
value): error against float64 at the edges of their tiles and over magnitudes,
and infinities, NaN and overflow as a float32 product has them."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# m, n, k: partial tiles along m and n, k of a part of a stage, one, two and many;
# then the same without aligned float4 rows, where loads that would cross an
# operand's end start earlier.  (16400, 252, 36), (8300, 512, 256), (16385, 255, 34),
# (8300, 510, 129) and (8200, 513, 387) take fp32 64x64 tiles; SPLIT_SHAPES below are
# all of this form
SHAPES = [(32700, 124, 4), (32768, 128, 16), (32641, 132, 20), (16400, 252, 36), (8300, 512, 256), (16384, 256, 772),
          (32701, 125, 5), (32641, 127, 17), (16385, 255, 34), (8300, 510, 129), (8200, 513, 387), (8257, 643, 63)]


def _product(gpu, hip_lib, a, b, b_kmajor, bias=None):
    from rnn_kernel_amd import _lib

    m, k = a.shape
    n = b.shape[1] if b_kmajor else b.shape[0]
    c = torch.full((m + 1, n), float("nan"), device=gpu)
    rc = hip_lib.rka_gemm_f32(m, n, k, a.data_ptr(), k, 0, b.data_ptr(), b.shape[1], b_kmajor,
                              None if bias is None else bias.data_ptr(), c.data_ptr(), n,
                              torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "rka_gemm_f32")
    torch.cuda.synchronize()
    assert torch.isnan(c[m]).all()  # nothing stored past the last row
    return c[:m]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("b_kmajor", [0, 1])
@pytest.mark.parametrize("scale", [1.0, 1e-30, 1e15])
def test_split_product_error(gpu, hip_lib, m, n, k, b_kmajor, scale):
    _check_error(gpu, hip_lib, m, n, k, b_kmajor, scale)


# aligned: two columns of tiles, the last of 4 to 132 columns; unaligned: a last
# tile of one, two, three and more columns (and rows), k of many stages that end with
# one, two, three and more values
SPLIT_SHAPES = [(32641, 132, 772), (16384, 388, 260), (32765, 128, 1028),
                (32641, 129, 257), (32642, 130, 242), (32643, 131, 243), (32767, 257, 401), (32765, 387, 513)]


@pytest.mark.parametrize("m,n,k", SPLIT_SHAPES)
@pytest.mark.parametrize("b_kmajor", [0, 1])
def test_split_product_edges(gpu, hip_lib, m, n, k, b_kmajor):
    from rnn_kernel_amd import _lib

    assert _lib.describe_gemm(m, n, k, aligned=n % 4 == 0 and k % 4 == 0) == "split"
    _check_error(gpu, hip_lib, m, n, k, b_kmajor, 1.0)


def _check_error(gpu, hip_lib, m, n, k, b_kmajor, scale):
    print(f"split m={m} n={n} k={k} b_kmajor={b_kmajor} scale={scale}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(m + n + k)
    a = scale * torch.randn(m, k, generator=g, device=gpu)
    b = torch.randn((k, n) if b_kmajor else (n, k), generator=g, device=gpu)
    b *= torch.exp(6 * torch.randn(b.shape, generator=g, device=gpu))  # 10 decades within a sum
    bias = scale * torch.randn(n, generator=g, device=gpu)
    c = _product(gpu, hip_lib, a, b, b_kmajor, bias)
    bd = b.double() if b_kmajor else b.double().t().contiguous()
    ref = a.double() @ bd + bias.double()
    mag = a.double().abs() @ bd.abs() + bias.double().abs()
    # six float32 roundings per 16-deep stage and the left-out products of pieces
    # (2^-24); the least normal value for each product and operand besides (looser
    # than need be, see test_split_product_of_small_magnitudes)
    stages = (k + 15) // 16
    tiny = 2.0 ** -126 * (6 * k + a.double().abs().sum(1, keepdim=True) + bd.abs().sum(0))
    assert bool(((c.double() - ref).abs() <= (6 * stages + 4) * 2.0 ** -24 * mag + tiny).all())


@pytest.mark.parametrize("m,n,k", [(32768, 128, 16), (32641, 132, 20), (32701, 125, 5), (32768, 129, 387)])
@pytest.mark.parametrize("b_kmajor", [0, 1])
@pytest.mark.parametrize("sa,sb", [(1e-36, 1.0), (1.0, 1e-38), (1e-41, 1.0), (1.0, 1e-41), (1e-19, 1e-19), (1e-41, 1e36)])
def test_split_product_of_small_magnitudes(gpu, hip_lib, m, n, k, b_kmajor, sa, sb):
    """Operands and products down to the smallest float32 keep the bits that a
    float32 product keeps."""
    print(f"split m={m} n={n} k={k} b_kmajor={b_kmajor} sa={sa} sb={sb}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(m + n + k)
    a = sa * torch.randn(m, k, generator=g, device=gpu)
    b = sb * torch.randn((k, n) if b_kmajor else (n, k), generator=g, device=gpu)
    c = _product(gpu, hip_lib, a, b, b_kmajor)
    bd = b.double() if b_kmajor else b.double().t().contiguous()
    ref = a.double() @ bd
    mag = a.double().abs() @ bd.abs()
    # as in test_split_product_error, and one rounding of a result below the
    # normal range (half of 2^-149)
    stages = (k + 15) // 16
    assert bool(((c.double() - ref).abs() <= (6 * stages + 4) * 2.0 ** -24 * mag + 2.0 ** -150).all())


@pytest.mark.parametrize("m,n,k", [(32768, 128, 256), (32768, 129, 387), (32768, 128, 2304)])
@pytest.mark.parametrize("b_kmajor", [0, 1])
def test_split_product_error_has_no_mean(gpu, hip_lib, m, n, k, b_kmajor):
    """The errors cancel in a sum over the rows (a bias gradient of the layer
    below sums thousands of them), as roundings to nearest do."""
    print(f"split m={m} n={n} k={k} b_kmajor={b_kmajor}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(m + n + k)
    a = torch.randn(m, k, generator=g, device=gpu)
    b = torch.randn((k, n) if b_kmajor else (n, k), generator=g, device=gpu)
    ref = a.double() @ (b.double() if b_kmajor else b.double().t().contiguous())
    mean = (_product(gpu, hip_lib, a, b, b_kmajor).double() - ref).mean() / ref.abs().mean()
    # six roundings per 16-deep stage, each at most 2^-24 of an output's size and
    # of either sign alike: six standard deviations of the mean of m n outputs
    # (measured: below one)
    stages = (k + 15) // 16
    assert abs(mean.item()) <= 6 * 2.0 ** -24 * (6 * stages / (m * n)) ** 0.5


@pytest.mark.parametrize("m,n,k", [(32768, 128, 16), (32768, 128, 256), (32641, 129, 387)])
@pytest.mark.parametrize("b_kmajor", [0, 1])
def test_split_product_rows_do_not_depend_on_their_place(gpu, hip_lib, m, n, k, b_kmajor):
    """Equal sequences of a batch give equal results: a row's result is the same
    bit for bit wherever the row stands."""
    print(f"split m={m} n={n} k={k} b_kmajor={b_kmajor}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(m + n + k)
    a = torch.randn(m, k, generator=g, device=gpu)
    b = torch.randn((k, n) if b_kmajor else (n, k), generator=g, device=gpu)
    c = _product(gpu, hip_lib, a, b, b_kmajor)
    for shift in (1, 37):
        assert torch.equal(_product(gpu, hip_lib, a.roll(shift, 0).contiguous(), b, b_kmajor), c.roll(shift, 0))


@pytest.mark.parametrize("b_kmajor", [0, 1])
def test_split_product_non_finite(gpu, hip_lib, b_kmajor):
    """Rows with an infinity, a NaN, values that round past the largest bf16 and
    a sum that overflows equal the float32 results; all other rows equal the
    same product without them, bit for bit."""
    m, n, k = 32768, 128, 64
    g = torch.Generator(device=gpu).manual_seed(3)
    a = torch.randn(m, k, generator=g, device=gpu)
    b = torch.randn((k, n) if b_kmajor else (n, k), generator=g, device=gpu)
    plain = _product(gpu, hip_lib, a, b, b_kmajor)
    bn = b.t() if b_kmajor else b  # [n, k]
    inf = float("inf")
    a2 = a.clone()
    a2[5, 7] = inf
    a2[130, 0] = -inf
    a2[131, 3], a2[131, 9] = inf, -inf
    a2[200, 63] = float("nan")
    a2[300] = 0.0
    a2[300, 2] = 3.4e38  # finite, but its first bf16 piece is not
    a2[400] = 3e38
    c = _product(gpu, hip_lib, a2, b, b_kmajor)
    touched = torch.zeros(m, dtype=torch.bool, device=gpu)
    touched[[5, 130, 131, 200, 300, 400]] = True
    assert torch.equal(c[~touched], plain[~touched])
    assert torch.equal(c[5], inf * bn[:, 7].sign()) and torch.equal(c[130], -inf * bn[:, 0].sign())
    want = torch.where(bn[:, 3].sign() == bn[:, 9].sign(), torch.full((n,), float("nan"), device=gpu), inf * bn[:, 3].sign())
    assert torch.equal(torch.isnan(c[131]), torch.isnan(want)) and torch.equal(c[131][~torch.isnan(want)], want[~torch.isnan(want)])
    assert torch.isnan(c[200]).all()
    ref = a2[300, 2].double() * bn[:, 2].double()
    fits = ref.abs() < 3.4e38
    assert torch.allclose(c[300][fits].double(), ref[fits], rtol=1e-6) and torch.isinf(c[300][ref.abs() > 3.5e38]).all()
    ref = (a2[400].double() @ bn.double().t().contiguous())
    big = ref.abs() > 1e39
    assert bool((~torch.isfinite(c[400][big])).all())


# aligned and unaligned rows, the last tile partial along m and n, one to three
# 64x64 tiles of it without outputs
@pytest.mark.parametrize("m,n,k", [(32768, 128, 64), (32641, 132, 20), (32701, 125, 37), (32641, 129, 5)])
@pytest.mark.parametrize("b_kmajor", [0, 1])
def test_split_product_all_non_finite(gpu, hip_lib, m, n, k, b_kmajor):
    """Every output infinite or NaN, the bias added: the signs of a float32
    product, nothing stored elsewhere, and the time of two products rather than
    of a hundred."""
    print(f"split m={m} n={n} k={k} b_kmajor={b_kmajor}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(m + n + k)
    a = torch.randn(m, k, generator=g, device=gpu)
    b = torch.randn((k, n) if b_kmajor else (n, k), generator=g, device=gpu)
    bias = torch.randn(n, generator=g, device=gpu)

    def timed():
        best = 1e30
        for _ in range(5):
            start, stop = torch.cuda.Event(True), torch.cuda.Event(True)
            start.record()
            c = _product(gpu, hip_lib, a, b, b_kmajor, bias)
            stop.record()
            stop.synchronize()
            best = min(best, start.elapsed_time(stop))
        return c, best

    _, plain = timed()
    inf, col = float("inf"), (b if b_kmajor else b.t())[3]
    a[:, 3] = inf
    a[::7, 3] = -inf
    a[5::11, 1] = float("nan")
    c, odd = timed()
    want = a[:, 3:4].sign() * col.sign() * inf
    nan = torch.zeros(m, dtype=torch.bool, device=gpu)
    nan[5::11] = True
    assert torch.isnan(c[nan]).all() and torch.equal(c[~nan], want[~nan])
    # (a second product in fp32, 1.5 to 2 times the first; one after the other
    # in each lane it was 40 to 130 times)
    assert odd <= 8 * plain


def test_split_weight_gradients_non_finite(gpu):
    """An infinite upstream gradient in one unit reaches that unit's weight
    gradient rows only."""
    from rnn_kernel_amd import GRUFunction

    B, T, H = 64, 512, 256
    g = torch.Generator(device=gpu).manual_seed(9)
    w = [((torch.rand(*s, generator=g, device=gpu) * 2 - 1) / 16).requires_grad_(True)
         for s in ((3 * H, H), (3 * H, H), (3 * H,), (3 * H,))]
    x = torch.randn(B, T, H, generator=g, device=gpu)
    dy = torch.randn(B, T, H, generator=g, device=gpu)
    y, _ = GRUFunction.apply(x, torch.zeros(B, H, device=gpu), *w)
    dy[3, 0, 17] = float("inf")  # the first step: its gradient goes no further back
    y.backward(dy)
    bad = torch.zeros(3 * H, dtype=torch.bool, device=gpu)
    bad[[17, H + 17, 2 * H + 17]] = True
    for p in w:
        rows = torch.isfinite(p.grad.reshape(3 * H, -1)).all(dim=1)
        assert bool(rows[~bad].all())
        assert not bool(rows[bad].any())


@pytest.mark.parametrize("H", [256, 129])  # aligned and unaligned rows
def test_split_backward_non_finite_leaves_the_rest(gpu, H):
    """The same with dx (in the launch that also reduces the partial sums): what
    the infinity does not reach equals the pass without it, bit for bit."""
    from rnn_kernel_amd import GRUFunction, _lib

    B, T = 64, 512
    assert _lib.describe_weight_gradients(B, T, H, H)["form"] == "split"
    assert _lib.describe_gemm(B * T, H, 3 * H, aligned=H % 4 == 0) == "split"
    g = torch.Generator(device=gpu).manual_seed(H)
    w = [((torch.rand(*s, generator=g, device=gpu) * 2 - 1) / 16).requires_grad_(True)
         for s in ((3 * H, H), (3 * H, H), (3 * H,), (3 * H,))]
    x = torch.randn(B, T, H, generator=g, device=gpu).requires_grad_(True)
    dy = torch.randn(B, T, H, generator=g, device=gpu)
    grads = []
    for value in (dy[3, 0, 17].item(), float("inf")):
        dy[3, 0, 17] = value
        y, _ = GRUFunction.apply(x, torch.zeros(B, H, device=gpu), *w)
        grads.append(torch.autograd.grad(y, [x] + w, dy))
    bad = torch.zeros(3 * H, dtype=torch.bool, device=gpu)
    bad[[17, H + 17, 2 * H + 17]] = True
    hit = torch.zeros(B, T, dtype=torch.bool, device=gpu)
    hit[3, 0] = True
    for k, (plain, odd) in enumerate(zip(*grads)):
        mask = hit if k == 0 else bad
        assert torch.equal(plain[~mask], odd[~mask])
        assert not torch.isfinite(odd[mask].reshape(int(mask.sum()), -1)).all(dim=1).any()
