"""lowbit_linear: row-major weights of any shape, float32 activations and the bias, against the oracle."""
import numpy as np
import pytest
import torch

import ipex_llm.ggml.model.llama.llama_cpp as ggml
import lowbit_oracle as orc
from gpu_util import ALL, DT, FP8, NF4, acts, dev_dequantize, dev_quantize, stream, weights
from ipex_llm.transformers.low_bit_linear import FP4Params, LowBitLinear

pytestmark = pytest.mark.gpu
GGML, TILED = ggml.LAYOUT_GGML, ggml.LAYOUT_TILED
TOL = {torch.float16: 2e-3, torch.bfloat16: 8e-3, torch.float32: 3e-5}


def _check(qtype, dtype, layout, m, n, k, biased, seed):
    w, x = weights(seed, (n, k)), acts(seed + 1, m, k, dtype)
    bias = torch.from_numpy(np.random.default_rng(seed + 2).standard_normal(n).astype(np.float32)).to(dtype) if biased else None
    blob, xd = dev_quantize(w, qtype, layout), x.cuda()
    bd = bias.cuda() if biased else None
    need = ggml.lowbit_linear_workspace_bytes(qtype, layout, DT[dtype], m, n, k, 64 << 20)
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    # guard rows on both sides: the kernel writes the m x n results and nothing else
    y = torch.full((m + 2, n), float("nan"), dtype=dtype, device="cuda")
    if (n * y.element_size()) % 16:
        y = torch.full(((m + 2) * n + 16,), float("nan"), dtype=dtype, device="cuda")[n % 8:][:(m + 2) * n].view(m + 2, n)
    ggml.lowbit_linear(xd.data_ptr(), blob.data_ptr(), bd.data_ptr() if biased else None, y[1].data_ptr(), qtype, layout, DT[dtype],
                       m, n, k, ws.data_ptr() if need else None, need, stream())
    torch.cuda.synchronize()
    assert torch.isnan(y[0]).all() and torch.isnan(y[m + 1]).all()
    want = orc.mul_mat_exact(orc.quantize(w, qtype), x.float().numpy(), (n, k), qtype)
    if biased:
        want = want + bias.float().numpy()
    got = y[1:m + 1].float().cpu().numpy()
    assert np.abs(got - want).max() <= TOL[dtype] * np.abs(want).max()


# rows of x around the kernel's passes and tiles, weight rows around 16, columns around 128 (whole blocks)
@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,n,k", [(1, 1, 128), (2, 17, 64), (3, 37, 192), (5, 48, 4160), (8, 8203, 320), (9, 15, 1088),
                                   (16, 16401, 128), (13, 8203, 8256), (17, 33, 576), (33, 3200, 1344), (70, 250, 2240),
                                   (130, 129, 448), (257, 515, 704)])
def test_row_major_weights_of_any_shape(qtype, dtype, m, n, k):
    if qtype == FP8:
        k = (k + 127) // 128 * 128
    _check(qtype, dtype, GGML, m, n, k, m % 2 == 1, 100 * m + n)


@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("m,n,k", [(1, 64, 256), (4, 8192, 384), (7, 8192, 128), (8, 48, 4096), (12, 4096, 1408), (16, 272, 128), (35, 64, 512)])
def test_float32_activations_in_one_pass(qtype, m, n, k):
    _check(qtype, torch.float32, TILED, m, n, k, m % 2 == 0, 300 * m + n)


# one shape for every kernel of the choice: streaming, ring (cut and whole tiles), GEMM, its K split, narrow and tall tiles
@pytest.mark.parametrize("qtype,dtype", [(2, torch.float16), (3, torch.bfloat16), (8, torch.float16), (10, torch.bfloat16), (15, torch.bfloat16)])
@pytest.mark.parametrize("m,n,k", [(3, 512, 256), (40, 4096, 1024), (50, 2048, 6400), (300, 272, 2048), (512, 16384, 128), (1030, 2048, 256), (200, 1040, 128)])
def test_bias_of_every_kernel(qtype, dtype, m, n, k):
    _check(qtype, dtype, TILED, m, n, k, True, 500 * m + n)


# Every form of the row-major kernels: 1 .. 4, 5 .. 8, up to 16 rows, the one-pass kernel, the GEMM with and without K splits
ROW_MAJOR = [(1, 2000, 4160), (7, 1000, 4160), (12, 1000, 4160), (16, 16399, 1088), (30, 1000, 4160), (70, 1000, 4160), (333, 1000, 4160)]


@pytest.mark.parametrize("qtype,dtype", [(2, torch.float16), (3, torch.bfloat16), (8, torch.float16), (10, torch.bfloat16), (15, torch.bfloat16)])
@pytest.mark.parametrize("m", [65, 96, 97, 129, 161, 192, 193, 257, 288, 289])
@pytest.mark.parametrize("n,k", [(1040, 4096), (2064, 1152), (16400, 256)], ids=["splits", "narrow", "wide"])
def test_row_tiles_of_three_blocks(qtype, dtype, m, n, k):
    """Three 32-row blocks in a tile, as a last one and as the height of all (129 .. 192 and 257 .. 288 rows), and the counts beside
    them; with K splits, in narrow tiles and in 128 x 256 tiles."""
    _check(qtype, dtype, ggml.LAYOUT_TILED, m, n, k, m % 2 == 1, m + n)


@pytest.mark.parametrize("qtype,dtype", [(2, torch.float16), (3, torch.float16), (8, torch.bfloat16), (10, torch.float16), (15, torch.float16)])
@pytest.mark.parametrize("m", [224, 225, 352, 480])
@pytest.mark.parametrize("n,k", [(1040, 4096), (2064, 1152), (16400, 256)], ids=["splits", "narrow", "wide"])
def test_last_row_tile_of_three_blocks_behind_whole_ones(qtype, dtype, m, n, k):
    _check(qtype, dtype, ggml.LAYOUT_TILED, m, n, k, m % 2 == 1, m + n)


@pytest.mark.parametrize("m,n,k,dtype", [(385, 17136, 256, torch.float16), (700, 11520, 384, torch.bfloat16)])
@pytest.mark.parametrize("qtype", ALL)
def test_rounds_of_tall_tiles_that_are_partly_filled(qtype, m, n, k, dtype):
    """Tiles of 256 rows over half a round of the GPU and more, which lowbit_linear takes ahead of the estimates."""
    _check(qtype, dtype, ggml.LAYOUT_TILED, m, n, k, True, m + n)


def _plain(qtype, m, n, k, dtype):
    if qtype == FP8 and k % 128:
        n, k = n + 1, (k + 127) // 128 * 128
    w, x = weights(m, (n, k), outliers=False), acts(m + 1, m, k, dtype)
    layer = LowBitLinear(k, n, qtype, bias=False, conver_to_half=False).eval()
    layer.weight = FP4Params(torch.from_numpy(w), qtype=qtype).to("cuda")
    with torch.no_grad():
        y = layer(x.cuda()).cpu()
    return y, x, torch.from_numpy(orc.dequantize(orc.quantize(w, qtype), qtype, (n, k)).astype(np.float64))


@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("m,n,k", ROW_MAJOR)
def test_row_major_weights_are_as_exact_as_in_fp32(qtype, m, n, k):
    """What is left beside the results' own rounding is that of fp32 sums: 2^-24 per step, in at most K / 32 = 136 random
    steps of at most the result's size, is 7e-7 of the norm."""
    y, x, w = _plain(qtype, m, n, k, torch.float32)
    hi = x.bfloat16().double()
    want = (hi + (x.double() - hi).bfloat16().double()) @ w.t()                   # float32 activations go in as two bf16 planes
    assert (y.double() - want).norm() <= 7e-7 * want.norm()
    y, x, w = _plain(qtype, m, n, k, torch.bfloat16)
    want = x.double() @ w.t()
    # an error of 7e-7 moves a result over a rounding border of bf16 (2^-9 to 2^-8 apart) in 2 * 7e-7 / 2^-9 of the cases
    assert (y != want.bfloat16()).float().mean() <= 7e-4


# streaming up to 8 rows in its shapes, the one-pass kernel beyond
@pytest.mark.parametrize("qtype", [t for t in ALL if t != NF4])                   # (nf4: the code book in two bf16 parts)
@pytest.mark.parametrize("m,n,k", [(1, 4096, 4096), (3, 1024, 4096), (8, 1024, 4096), (7, 8192, 1024), (12, 4096, 4096), (16, 8192, 1024),
                                   (24, 1024, 4096), (70, 4112, 2048)])
def test_tiled_weights_with_float32_activations_are_as_exact_as_fp32_sums(qtype, m, n, k):
    y, x, w = _plain(qtype, m, n, k, torch.float32)
    hi = x.bfloat16().double()
    want = (hi + (x.double() - hi).bfloat16().double()) @ w.t()
    assert (y.double() - want).norm() <= 7e-7 * want.norm()                       # (K / 32 = 128 steps at most, as above)


def classes(t):
    """0 finite, 1 nan, 2 +inf, 3 -inf"""
    return np.isnan(t) * 1 + np.isposinf(t) * 2 + np.isneginf(t) * 3


# row-major weights in every form, and tiled ones in the one-pass kernel (1 .. 4 tile rows, 16 .. 64 rows)
@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,n,k", [(1, 37, 640), (4, 8203, 192), (8, 37, 640), (8, 8203, 192), (12, 37, 192), (12, 16399, 64), (24, 37, 192), (70, 37, 192),
                                   (333, 300, 2112), (9, 48, 256), (24, 4112, 256), (40, 8208, 128), (31, 12304, 128), (64, 48, 256)])
def test_infinities_meet_the_weights_and_not_their_codes(qtype, dtype, m, n, k):
    if qtype == FP8:
        k = (k + 127) // 128 * 128
    w, x = weights(m, (n, k)), acts(m + 1, m, k, dtype)
    x[0, 5], x[m // 2, k - 3] = float("inf"), -float("inf")
    if m > 2:
        x[m - 1, 7] = float("nan")
    if dtype != torch.float16 and m > 3:
        x[1, 3] = 1e38                                                            # finite: its codes' sums need not be
    layer = LowBitLinear(k, n, qtype, bias=True, conver_to_half=False).eval()
    layer.weight = FP4Params(torch.from_numpy(w), qtype=qtype).to("cuda")
    layer.bias = torch.nn.Parameter(torch.randn(n).to(dtype).cuda(), requires_grad=False)
    with torch.no_grad(), np.errstate(invalid="ignore"):
        y = layer(x.cuda()).float().cpu().numpy()
        want = x.double().numpy() @ orc.dequantize(orc.quantize(w, qtype), qtype, (n, k)).astype(np.float64).T
    assert (classes(y) == classes(want)).all()
    if m > 1:
        assert (classes(want) != 0).any() and (classes(want) == 0).any()


# tiles times splits that eighths of either do not divide: 1 tile in 16 splits, 9 in 5 to 7, 50 in 5, more than 256 workgroups
@pytest.mark.parametrize("qtype,dtype", [(2, torch.float16), (3, torch.bfloat16), (8, torch.float16), (10, torch.bfloat16), (15, torch.bfloat16)])
@pytest.mark.parametrize("m,n,k", [(70, 256, 8192), (300, 784, 4096), (178, 6288, 1920), (100, 2320, 2176)])
@pytest.mark.parametrize("splits", [2, 5, 7, 16])
def test_k_splits_over_the_xcds(qtype, dtype, m, n, k, splits):
    blob, x = dev_quantize(weights(m, (n, k)), qtype, TILED), acts(m, m, k, dtype).cuda()
    if k // 128 < 2 * splits:
        splits = k // 256
    tiles = (m + 127) // 128 * ((n + 255) // 256)
    ws = torch.full((tiles * splits * 128 * 256 * 4 + 64,), 255, dtype=torch.uint8, device="cuda")
    y = torch.full((m + 1, n), float("nan"), dtype=dtype, device="cuda")
    ggml.lowbit_gemm_ws(x.data_ptr(), blob.data_ptr(), y.data_ptr(), qtype, TILED, DT[dtype], m, n, k, ws.data_ptr(), ws.numel() - 64, splits, stream())
    want = x.double() @ dev_dequantize(blob, qtype, n, k, TILED, torch.float32).double().t()
    assert torch.isnan(y[m]).all() and (ws[-64:] == 255).all()
    assert ((y[:m].double() - want).abs().max() <= TOL[dtype] * want.abs().max())


# parts that are summed in one round of loads (up to 9), in one and a rest, and in two: a part left out or added twice is a tenth of y
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("splits", [3, 4, 6, 8, 9, 10, 14, 16])
def test_sums_of_splits(dtype, splits):
    m, n, k, qtype = 137, 272, 256 * splits, 8
    blob, x = dev_quantize(weights(splits, (n, k)), qtype, TILED), acts(splits, m, k, dtype).cuda()
    ws = torch.empty(2 * 2 * 128 * 256 * 4 * splits, dtype=torch.uint8, device="cuda")
    y = torch.empty(m, n, dtype=dtype, device="cuda")
    ggml.lowbit_gemm_ws(x.data_ptr(), blob.data_ptr(), y.data_ptr(), qtype, TILED, DT[dtype], m, n, k, ws.data_ptr(), ws.numel(), splits, stream())
    want = x.double() @ dev_dequantize(blob, qtype, n, k, TILED, torch.float32).double().t()
    assert ((y.double() - want).abs().max() <= TOL[dtype] * want.abs().max())


# sizes that the one-pass kernel leaves to the kernels that deal tiles or K, with the kernel asserted; row counts around three 32-row blocks
SPLIT, RING, NARROW, GEMM = ggml.PLAN_GEMM_SPLIT, ggml.PLAN_RING, ggml.PLAN_GEMM_NARROW, ggml.PLAN_GEMM
THREE_BLOCKS = [65, 96, 97, 129, 161, 192, 193, 224, 225, 257, 288, 289, 352, 480]
KERNELS = ([(SPLIT, q, m, 1040, 16512) for q in ALL if q != NF4 for m in THREE_BLOCKS] + [(SPLIT, NF4, 129, 4112, 8192), (SPLIT, NF4, 161, 4112, 8192)]
           + [(SPLIT, NF4, m, 2064, 16512) for m in (129, 257, 288, 289, 480)] + [(RING, NF4, m, 1040, 16512) for m in THREE_BLOCKS]
           + [(RING, q, m, 272, 16512) for q in ALL for m in (96, 97, 192, 193, 224, 225)] + [(RING, q, 40, 1040, 16512) for q in ALL]
           + [(RING, q, 128, 528, 20480) for q in ALL] + [(NARROW, q, m, 6160, 1152) for q in ALL for m in THREE_BLOCKS if m < 300]
           + [(NARROW, q, m, 8208, 384) for q in ALL for m in THREE_BLOCKS] + [(GEMM, q, 480, 8208, 2048) for q in ALL if q != NF4])


@pytest.mark.parametrize("plan,qtype,m,n,k", KERNELS)
def test_bias_of_every_kernel_that_deals_tiles(plan, qtype, m, n, k):
    dtype = torch.bfloat16 if (m + n + qtype) % 2 else torch.float16
    need = ggml.lowbit_linear_scratch_bytes(qtype, TILED, DT[dtype], m, n, k, 64 << 20)
    assert ggml.lowbit_linear_plan(qtype, TILED, DT[dtype], m, n, k, need)[0] == plan
    blob = dev_quantize((np.random.default_rng(m + n).standard_normal((n, k), dtype=np.float32) * 0.02), qtype, TILED)
    x, bias = acts(m, m, k, dtype).cuda(), torch.randn(n, generator=torch.Generator().manual_seed(m)).to(dtype).cuda()
    ws = torch.full((need + 64,), 255, dtype=torch.uint8, device="cuda")
    y = torch.full((m + 2, n), float("nan"), dtype=dtype, device="cuda")
    ggml.lowbit_linear(x.data_ptr(), blob.data_ptr(), bias.data_ptr(), y[1].data_ptr(), qtype, TILED, DT[dtype], m, n, k,
                       ws.data_ptr() if need else None, need, stream())
    want = x.double() @ dev_dequantize(blob, qtype, n, k, TILED, torch.float32).double().t() + bias.double()
    assert torch.isnan(y[0]).all() and torch.isnan(y[m + 1]).all() and (ws[need:] == 255).all()
    assert (y[1:m + 1].double() - want).abs().max() <= TOL[dtype] * want.abs().max()
