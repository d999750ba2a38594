"""Products whose operands are requested straight into LDS (K a multiple of 64) against the product in fp64.

bf16 inputs, fp32 sums: a sum of K products is off by at most a few 2^-24 of sum |x w| and is rounded once to bf16 (2^-9 of the
value), hence |d| <= 2^-8 |value| + 2^-18 sqrt(K) for inputs of size one."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# K from one step to more than two turns of the buffers, M and N around the tile's edge and at one row past it
@pytest.mark.parametrize("km,kn", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(40, 8, 64), (64, 64, 128), (72, 72, 192), (256, 200, 256), (136, 64, 320), (64, 1032, 576), (520, 136, 2048), (136, 6144, 320),
                                   (264, 8200, 192), (2200, 2048, 192)])
def test_product(M, N, K, km, kn):
    from jaxrwkv_amd import blocks7
    g = torch.Generator("cuda").manual_seed(M + N + K)
    x = torch.randn((K, M) if km else (M, K), device="cuda", generator=g).bfloat16()
    w = torch.randn((K, N) if kn else (N, K), device="cuda", generator=g).bfloat16()
    guard = torch.full((M + 2, N), 7.0, device="cuda", dtype=torch.bfloat16)
    blocks7._gemm([(guard[1:-1], x, w, km, kn, 0, None)])
    want = (x.double().T if km else x.double()) @ (w.double() if kn else w.double().T)
    d = (guard[1:-1].double() - want).abs()
    assert (d <= want.abs() * 2.0 ** -8 + 2.0 ** -18 * K ** 0.5).all()
    assert (guard[0] == 7).all() and (guard[-1] == 7).all()


def test_several_products_in_one_launch():
    from jaxrwkv_amd import blocks7
    g = torch.Generator("cuda").manual_seed(5)
    x = torch.randn((300, 256), device="cuda", generator=g).bfloat16()
    ws = [torch.randn((n, 256), device="cuda", generator=g).bfloat16() for n in (8, 256, 96)]
    outs = [torch.empty((300, w.shape[0]), device="cuda", dtype=torch.bfloat16) for w in ws]
    blocks7._gemm([(o, x, w, 0, 0, 0, None) for o, w in zip(outs, ws)])
    for o, w in zip(outs, ws):
        want = x.double() @ w.double().T
        assert ((o.double() - want).abs() <= want.abs() * 2.0 ** -8 + 2.0 ** -14).all()


def test_long_and_short_products_in_one_launch():
    """Beside a long product the short ones go straight to LDS as well, whatever their K."""
    from jaxrwkv_amd import blocks7
    g = torch.Generator("cuda").manual_seed(6)
    jobs, want = [], []
    for M, N, K, km, kn in ((200, 32, 1030, 1, 1), (136, 264, 8, 0, 0), (72, 128, 40, 0, 1), (72, 72, 72, 1, 0), (64, 64, 5, 1, 1)):
        x = torch.randn((K, M) if km else (M, K), device="cuda", generator=g).bfloat16()
        w = torch.randn((K, N) if kn else (N, K), device="cuda", generator=g).bfloat16()
        jobs.append((torch.empty((M, N), device="cuda", dtype=torch.bfloat16), x, w, km, kn, 0, None))
        want.append((x.double().T if km else x.double()) @ (w.double() if kn else w.double().T))
    blocks7._gemm(jobs)
    for j, v in zip(jobs, want):
        assert ((j[0].double() - v).abs() <= v.abs() * 2.0 ** -8 + 2.0 ** -18 * 1030 ** 0.5).all()


@pytest.mark.parametrize("M,K", [(8, 64), (40, 64), (40, 72)])
def test_tanh_of_small_values(M, K):
    """The first low-rank factor of the decay starts at zero, so its hidden values start small: tanh keeps their relative precision.
    x is one times a power of two in one place, so the sum is exact in bf16, and the result is tanh rounded once: 2^-8 of it.
    The three shapes are the three kernels."""
    from jaxrwkv_amd import blocks7
    N = 64
    g = torch.Generator("cuda").manual_seed(K)
    x = torch.zeros((M, K), device="cuda")
    x[:, 3] = 2.0 ** -torch.arange(M, device="cuda").float()
    w = torch.zeros((K, N), device="cuda")
    w[3] = torch.rand(N, device="cuda", generator=g) + 0.5
    x, w = x.bfloat16(), w.bfloat16()
    out = torch.empty((M, N), device="cuda", dtype=torch.bfloat16)
    blocks7._gemm([(out, x, w, 0, 1, 1, None)])
    want = torch.tanh((x.double() @ w.double()).bfloat16().double())
    assert ((out.double() - want).abs() <= 2.0 ** -8 * want.abs()).all()


# a last step that is not full, in each tile: 64 x 64, 128 x 64, 128 x 128 with three buffers and with two
@pytest.mark.parametrize("km,kn", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N", [(72, 136), (264, 2056), (2048, 776), (2056, 2312)])
@pytest.mark.parametrize("K", [256, 264, 376, 520])
def test_product_of_any_k(M, N, K, km, kn):
    from jaxrwkv_amd import blocks7
    K += 1 if km and kn and K > 256 else 0                # without rows of k, K may be odd
    g = torch.Generator("cuda").manual_seed(M + N + K)

    def operand(rows, k_major):                           # what lies behind the last k of an operand must not be seen
        shape, used = ((K + 64, rows), slice(0, K)) if k_major else ((rows + 1, K), slice(0, rows))
        full = torch.randn(shape, device="cuda", generator=g).bfloat16()
        full[used.stop:] = float("nan")
        return full[used]
    x, w = operand(M, km), operand(N, kn)
    guard = torch.full((M + 2, N), 7.0, device="cuda", dtype=torch.bfloat16)
    blocks7._gemm([(guard[1:-1], x, w, km, kn, 0, None)])
    want = (x.double().T if km else x.double()) @ (w.double() if kn else w.double().T)
    d = (guard[1:-1].double() - want).abs()
    assert (d <= want.abs() * 2.0 ** -8 + 2.0 ** -18 * K ** 0.5).all()
    assert (guard[0] == 7).all() and (guard[-1] == 7).all()


# few rows: a wave's steps of K from none to one more than a round of requests, one and two tiles of rows, either layout of the weights
@pytest.mark.parametrize("kn", [0, 1])
@pytest.mark.parametrize("M", [1, 16, 17, 32])
@pytest.mark.parametrize("K", [32, 256, 544, 768, 1280, 1792, 2048, 2336])
def test_product_of_few_rows(M, K, kn):
    test_product(M, 48, K, 0, kn)


def test_products_of_few_rows_in_one_launch():
    from jaxrwkv_amd import blocks7
    g = torch.Generator("cuda").manual_seed(7)
    jobs, want = [], []
    for N, K, kn in ((64, 768, 0), (32, 768, 1), (16, 96, 1), (80, 32, 0)):
        x = torch.randn((5, K), device="cuda", generator=g).bfloat16()
        w = torch.randn((K, N) if kn else (N, K), device="cuda", generator=g).bfloat16()
        jobs.append((torch.empty((5, N), device="cuda", dtype=torch.bfloat16), x, w, 0, kn, 0, None))
        want.append(x.double() @ (w.double() if kn else w.double().T))
    blocks7._gemm(jobs)
    for j, v in zip(jobs, want):
        assert ((j[0].double() - v).abs() <= v.abs() * 2.0 ** -8 + 2.0 ** -18 * 768 ** 0.5).all()


# 256 x 128 tiles: the edge of a tile each way, one turn of the buffers and more, a last step that is not full
@pytest.mark.parametrize("M,N", [(2056, 3080), (2040, 3072)])
@pytest.mark.parametrize("K", [256, 264, 320, 520])
def test_product_in_the_largest_tiles(M, N, K):
    test_product_of_any_k(M, N, K, 0, 0)


def test_products_of_several_k_in_large_tiles():
    """A product of few steps and one of many, 128 x 128 tiles, transposed operands."""
    from jaxrwkv_amd import blocks7
    g = torch.Generator("cuda").manual_seed(8)
    jobs, want = [], []
    for M, N, K, km, kn in ((2056, 3080, 264, 0, 1), (776, 3080, 2056, 1, 1)):
        x = torch.randn((K, M) if km else (M, K), device="cuda", generator=g).bfloat16()
        w = torch.randn((K, N) if kn else (N, K), device="cuda", generator=g).bfloat16()
        jobs.append((torch.empty((M, N), device="cuda", dtype=torch.bfloat16), x, w, km, kn, 0, None))
        want.append((x.double().T if km else x.double()) @ (w.double() if kn else w.double().T))
    blocks7._gemm(jobs)
    for j, v in zip(jobs, want):
        assert ((j[0].double() - v).abs() <= v.abs() * 2.0 ** -8 + 2.0 ** -18 * 2056 ** 0.5).all()
