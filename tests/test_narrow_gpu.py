"""Gated MLPs and grouped products around the sizes where their tiles change: narrow ones with two groups of waves and one, 128-row
and tall ones."""
import pytest
import torch

from gpu_util import ALL, DT, NAMES, dev_dequantize, dev_quantize, ggml, stream, weights

pytestmark = pytest.mark.gpu
TILED = ggml.LAYOUT_TILED


def products(x, blob, qtype, n, k):
    """x w^T in fp64 with the weights that the GEMM forms make, rounded once to x's type, and the bound of its error: fp32 sums of k
    terms; asym_int4 (q * d + m) rounds a second time in dev_dequantize"""
    w = dev_dequantize(blob, qtype, n, k, TILED, torch.float32).to(x.dtype).double()
    size = x.double().abs() @ w.abs().t()
    return x.double() @ w.t(), size * (k * 2.0 ** -24 + (torch.finfo(x.dtype).eps if qtype == 3 else 0.0))


def mlp_close(y, x, blobs, qtype, n, k, act):
    """act(x Wg^T) * (x Wu^T), rounded once; exp2 and rcp of an ulp each; the activation's slope is at most 1.13"""
    (g, dg), (u, du) = (products(x, b, qtype, n, k) for b in blobs)
    a = torch.nn.functional.silu(g) if act == 0 else torch.nn.functional.gelu(g, approximate="tanh")
    eps = torch.finfo(x.dtype).eps
    # (tanh as 1 - 2 / (1 + e^2u) cancels: an absolute 2^-23 of g)
    bound = (a * u).abs() * (eps / 2 + 2.0 ** -20) + 1.13 * dg * u.abs() + a.abs() * du + dg * du + (g * u).abs() * 2.0 ** -21 + \
        torch.finfo(x.dtype).smallest_normal
    return ((y.double() - a * u).abs() <= bound).all()


# 64 rows and two groups of waves per tile: 1, 2, 3 and 4 row blocks, an odd number of K steps, a last tile of 16 columns; one
# group: fewer than eight steps, more than one tile per CU, tall tiles little more than one per CU; tall tiles beyond
@pytest.mark.parametrize("m,n,k", [(65, 144, 1152), (100, 2064, 1024), (130, 1040, 1408), (256, 4096, 1024), (200, 272, 640), (300, 6400, 256),
                                   (260, 16400, 256), (513, 11008, 128), (384, 24576, 256)])
@pytest.mark.parametrize("qtype", ALL, ids=NAMES.values())
def test_gated_mlp_tiles(qtype, m, n, k):
    dtype, act = (torch.bfloat16, 1) if k % 512 == 128 else (torch.float16, 0)
    blobs = [dev_quantize(weights(60 + i, (n, k)), qtype, TILED) for i in range(2)]
    x = torch.randn((m, k), generator=torch.Generator().manual_seed(m)).to(dtype).cuda()
    y = torch.full((m + 1, n), float("nan"), dtype=dtype, device="cuda")
    ggml.lowbit_mlp_forward(x.data_ptr(), blobs[0].data_ptr(), blobs[1].data_ptr(), y.data_ptr(), qtype, DT[dtype], m, n, k, act, stream())
    assert torch.isnan(y[m]).all() and mlp_close(y[:m], x, blobs, qtype, n, k, act)


@pytest.mark.parametrize("m,n,k", [(90, 5008, 1152), (176, 8208, 256), (192, 11008, 1024), (270, 4112, 1152), (288, 11024, 256)])
@pytest.mark.parametrize("qtype", ALL, ids=NAMES.values())
def test_gated_mlp_in_row_tiles_of_three_blocks(qtype, m, n, k):
    test_gated_mlp_tiles(qtype, m, n, k)


@pytest.mark.parametrize("m,n,k", [(400, 16400, 256), (600, 11008, 128), (576, 11008, 256), (577, 11008, 256)])
@pytest.mark.parametrize("qtype", ALL, ids=NAMES.values())
def test_gated_mlp_tiles_around_a_second_round(qtype, m, n, k):
    """Tall tiles little more than one per CU: narrow ones in their place, but not with a last row tile of 64 rows at most."""
    test_gated_mlp_tiles(qtype, m, n, k)


@pytest.mark.parametrize("rows,n,k", [((3, 0, 40, 129, 1), 144, 1152), ((130, 257, 64), 2064, 1024), ((5, 31, 33), 272, 640), ((200, 9), 16400, 256),
                                      ((300, 100, 20), 40960, 128)])
@pytest.mark.parametrize("qtype", ALL, ids=NAMES.values())
def test_grouped_tiles(qtype, rows, n, k):
    """Groups of no, few and more than 128 rows in narrow tiles with two groups of waves and one, and in the forms beyond; the plain
    product and the fused gate/up."""
    dtype = torch.float16 if n % 32 else torch.bfloat16
    offsets = torch.tensor([0, *rows]).cumsum(0).int().cuda()
    total = sum(rows)
    blobs = [[dev_quantize(weights(10 * e + i, (n, k)), qtype, TILED) for e in range(len(rows))] for i in range(2)]
    tables = [torch.tensor([b.data_ptr() for b in bs], device="cuda") for bs in blobs]
    x = torch.randn((total, k), generator=torch.Generator().manual_seed(1)).to(dtype).cuda()
    y = torch.full((total + 1, n), float("nan"), dtype=dtype, device="cuda")
    h = torch.full_like(y, float("nan"))
    ggml.lowbit_grouped_forward(x.data_ptr(), tables[0].data_ptr(), y.data_ptr(), offsets.data_ptr(), len(rows), total, qtype, DT[dtype], n, k,
                                stream())
    ggml.lowbit_grouped_mlp_forward(x.data_ptr(), tables[0].data_ptr(), tables[1].data_ptr(), h.data_ptr(), offsets.data_ptr(), len(rows),
                                    total, qtype, DT[dtype], n, k, 0, stream())
    assert torch.isnan(y[total]).all() and torch.isnan(h[total]).all()
    for e, (a, b) in enumerate(zip(offsets.tolist(), offsets.tolist()[1:])):
        if a == b:
            continue
        want, bound = products(x[a:b], blobs[0][e], qtype, n, k)
        assert ((y[a:b].double() - want).abs() <= want.abs() * torch.finfo(dtype).eps / 2 + bound + torch.finfo(dtype).smallest_normal).all()
        assert mlp_close(h[a:b], x[a:b], (blobs[0][e], blobs[1][e]), qtype, n, k, 0)


def random_blob(qtype, n, k, seed):
    w = torch.randn((n, k), generator=torch.Generator("cuda").manual_seed(seed), device="cuda") * 0.02
    blob = torch.empty(ggml.lowbit_blob_bytes(qtype, n * k), dtype=torch.uint8, device="cuda")
    ggml.lowbit_quantize(w.data_ptr(), blob.data_ptr(), qtype, n, k, TILED, stream())
    return blob


# 1 .. 8 row blocks of 32 per tall tile, eight waves (up to 192 rows per group) and four
@pytest.mark.parametrize("rows", [(5, 33, 70, 100, 130, 170, 200, 256), (300, 700, 250, 513)], ids=["eight waves", "four waves"])
@pytest.mark.parametrize("k", [384, 512, 640, 768, 896])
@pytest.mark.parametrize("qtype", ALL, ids=NAMES.values())
def test_tall_tiles_over_several_steps(qtype, k, rows):
    """The tall forms, fused and plain, where narrow tiles would be more than two per CU: three to seven K steps, so that the
    pipeline of two steps ahead runs its loop of three and ends with one, two and three steps after it."""
    dtype = torch.bfloat16 if k % 256 else torch.float16
    offsets = torch.tensor([0, *rows]).cumsum(0).int().cuda()
    total, groups = sum(rows), len(rows)
    x = torch.randn((total, k), generator=torch.Generator().manual_seed(k)).to(dtype).cuda()
    for fused, n in ((True, 5136), (False, 10256)):
        blobs = [random_blob(qtype, n, k, 7 * k + i) for i in range(3)]
        of = lambda e, up: blobs[(e + up) % 3]
        tables = [torch.tensor([of(e, up).data_ptr() for e in range(groups)], device="cuda") for up in range(2)]
        # more narrow tiles than two per CU of 256, were every group's rows to fill theirs; the plain product says what it takes
        assert sum((r + 127) // 128 for r in rows) * ((n + 63) // 64 if fused else (n + 127) // 128) > 512
        y = torch.full((total + 1, n), float("nan"), dtype=dtype, device="cuda")
        if fused:
            ggml.lowbit_grouped_mlp_forward(x.data_ptr(), tables[0].data_ptr(), tables[1].data_ptr(), y.data_ptr(), offsets.data_ptr(), groups,
                                            total, qtype, DT[dtype], n, k, 0, stream())
        else:
            tall, splits = ggml.lowbit_grouped_forward_plan(groups, total, n, k, False)[:2]
            assert (tall, splits) == (1, 1)
            ggml.lowbit_grouped_forward(x.data_ptr(), tables[0].data_ptr(), y.data_ptr(), offsets.data_ptr(), groups, total, qtype, DT[dtype],
                                        n, k, stream())
        assert torch.isnan(y[total]).all()
        for e, (a, b) in enumerate(zip(offsets.tolist(), offsets.tolist()[1:])):
            if fused:
                assert mlp_close(y[a:b], x[a:b], (of(e, 0), of(e, 1)), qtype, n, k, 0)
            else:
                want, bound = products(x[a:b], of(e, 0), qtype, n, k)
                assert ((y[a:b].double() - want).abs() <= want.abs() * torch.finfo(dtype).eps / 2 + bound + torch.finfo(dtype).smallest_normal).all()
