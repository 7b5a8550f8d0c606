"""The batch kernel for row-major weights: rows of x around its 32-row blocks and its tiles of 32, 64 and 128, weight rows around a
wave's 32 and a workgroup's 128, last steps of one to four blocks, one step, odd and even numbers of them, K splits."""
import numpy as np
import pytest
import torch

import lowbit_oracle as orc
from gpu_util import ALL, DT, FP8, acts, dev_dequantize, dev_quantize, ggml, stream, weights
from test_linear_gpu import GGML, _check, classes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(65, 31, 64), (66, 33, 192), (97, 127, 320), (128, 129, 448), (129, 257, 576), (20, 40, 12864), (40, 70, 8704),
                                   (250, 8203, 192), (300, 145, 4288)])
def test_edges(qtype, dtype, m, n, k):
    if qtype not in (FP8, 10) and m % 2:
        k -= 32                                             # an odd number of blocks
    if qtype == FP8:
        k = (k + 127) // 128 * 128
    _check(qtype, dtype, GGML, m, n, k, m % 2 == 0, 1100 * m + n)


@pytest.mark.parametrize("qtype", ALL)
def test_infinities_at_the_columns_read_past_the_end(qtype):
    """Columns past K are read as the first ones of their group, times a scale of zero."""
    m, n, k = 70, 37, 448 if qtype != FP8 else 512
    w, x = weights(m, (n, k)), acts(m, m, k, torch.float16)
    x[3, 384], x[5, 391], x[40, 388] = float("inf"), -float("inf"), float("nan")
    blob, xd, y = dev_quantize(w, qtype, GGML), x.cuda(), torch.empty((m, n), dtype=torch.float16, device="cuda")
    ggml.lowbit_linear(xd.data_ptr(), blob.data_ptr(), None, y.data_ptr(), qtype, GGML, DT[torch.float16], m, n, k, None, 0, stream())
    with np.errstate(invalid="ignore"):
        want = x.double().numpy() @ orc.dequantize(orc.quantize(w, qtype), qtype, (n, k)).astype(np.float64).T
    assert (classes(y.float().cpu().numpy()) == classes(want)).all()
    assert (classes(want) > 0).any() and (classes(want) == 0).any()


# Tiles of 128 rows, which take more than 256 tiles times splits: K splits where the steps are four times as many or more
@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k,splits", [(333, 3201, 2240, 4), (229, 16523, 192, 1), (97, 16771, 1088, 2), (128, 33003, 96, 1)])
def test_tiles_of_128_rows(qtype, dtype, m, n, k, splits):
    """With a workspace and without; last steps of one to three blocks; infinities and a nan among the activations, also at columns
    that are read past the end."""
    if qtype in (FP8, 10):
        k = (k + 127) // 128 * 128 if qtype == FP8 else (k + 63) // 64 * 64
    tiles = (m + 127) // 128 * ((n + 127) // 128)
    need = ggml.lowbit_linear_workspace_bytes(qtype, GGML, DT[dtype], m, n, k, 256 << 20)
    assert need == (splits * tiles * 128 * 128 * 4 if splits > 1 else 0) and tiles * max((k + 127) // 128 // 4, 1) > 256
    blob, x = dev_quantize(weights(m, (n, k)), qtype, GGML), acts(m, m, k, dtype).cuda()
    w = dev_dequantize(blob, qtype, n, k, GGML, torch.float32).double()
    ws, bias = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda"), torch.randn(n, device="cuda").to(dtype)
    for odd in (False, True):
        if odd:
            x[3, k - k % 128 - 128 if k % 128 == 0 else k - k % 128], x[m // 2, k - 3], x[m - 1, 5] = float("inf"), -float("inf"), float("nan")
        want = x.double() @ w.t()
        # fp32 sums of at most k / 32 scaled partial sums, themselves fp32; the sum with the bias; one rounding
        size = x.double().nan_to_num(posinf=0.0, neginf=0.0).abs() @ w.t().abs()
        bound = size * (k // 32 + 8) * 2.0 ** -24 + (want + bias).abs() * torch.finfo(dtype).eps / 2 * (1 + 2.0 ** -10) + torch.finfo(dtype).smallest_normal
        for workspace in (ws.data_ptr() if need else None, None):
            y = torch.full((m + 2, n), float("nan"), dtype=dtype, device="cuda")
            ggml.lowbit_linear(x.data_ptr(), blob.data_ptr(), bias.data_ptr(), y[1].data_ptr(), qtype, GGML, DT[dtype], m, n, k, workspace,
                               need if workspace else 0, stream())
            assert torch.isnan(y[0]).all() and torch.isnan(y[m + 1]).all()
            got, finite = y[1:m + 1].double(), want.isfinite()
            assert ((got - want - bias).abs() <= bound)[finite].all()
            assert (got.isnan() == want.isnan()).all() and (got == want)[want.isinf()].all()
            assert finite.all() != odd


@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(65, 9001, 2112), (96, 33001, 576), (180, 12001, 704), (129, 9001, 4160), (159, 9011, 4288)])
def test_tiles_of_96_and_160_rows(qtype, dtype, m, n, k):
    """Tiles of three and five 32-row blocks, with and without K splits; infinities in the last block's rows."""
    if qtype in (FP8, 10):
        k = (k + 127) // 128 * 128 if qtype == FP8 else (k + 63) // 64 * 64
    _check(qtype, dtype, GGML, m, n, k, m % 2 == 0, 1300 * m + n)
    blob, x = dev_quantize(weights(m, (37, k)), qtype, GGML), acts(m, m, k, dtype).cuda()
    x[m - 1, k - 1], x[m - 2, 3] = float("inf"), -float("inf")
    y = torch.empty((m, 37), dtype=dtype, device="cuda")
    ggml.lowbit_linear(x.data_ptr(), blob.data_ptr(), None, y.data_ptr(), qtype, GGML, DT[dtype], m, 37, k, None, 0, stream())
    want = x.double() @ dev_dequantize(blob, qtype, 37, k, GGML, torch.float32).double().t()
    assert (classes(y.float().cpu().numpy()) == classes(want.cpu().numpy())).all()


@pytest.mark.parametrize("qtype,dtype", [(2, torch.float16), (3, torch.bfloat16), (8, torch.float16), (10, torch.bfloat16), (15, torch.float16)])
@pytest.mark.parametrize("m,n,k,splits", [(56, 8670, 2176, 4), (52, 17372, 1408, 2), (60, 16383, 1664, 3), (60, 16500, 1664, 3)])
def test_short_last_splits(qtype, dtype, m, n, k, splits):
    """Last splits that are shorter than the others, of workgroups that are a few more than the CUs (they go out last), as many more as
    there are tiles, and more than that."""
    tiles, steps = -(-n // 128), -(-(k // 128) // splits)
    assert ggml.lowbit_linear_workspace_bytes(qtype, GGML, DT[dtype], m, n, k, 256 << 20) == splits * tiles * 64 * 128 * 4
    assert splits * steps > k // 128
    _check(qtype, dtype, GGML, m, n, k, False, m + n)


# sizes that the one-pass kernel leaves to this one: more than 1024 rows, more than 16384 columns; short K at the edges of 32 and 128 weight rows
@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(1025, 31, 64), (1057, 33, 192), (1089, 127, 320), (1120, 128, 128), (1151, 129, 448), (1153, 257, 576),
                                   (20, 40, 16448), (40, 70, 16704), (66, 9001, 320)])
def test_edges_beyond_the_one_pass_kernel(qtype, dtype, m, n, k):
    if qtype not in (FP8, 10) and m % 2:
        k -= 32                                             # an odd number of blocks
    if qtype == FP8:
        k = (k + 127) // 128 * 128
    need = ggml.lowbit_linear_scratch_bytes(qtype, GGML, DT[dtype], m, n, k, 64 << 20)
    assert ggml.lowbit_linear_plan(qtype, GGML, DT[dtype], m, n, k, need)[0] == ggml.PLAN_ROWS
    _check(qtype, dtype, GGML, m, n, k, m % 2 == 0, 1500 * m + n)


# lowbit_forward keeps this kernel above 64 rows, whatever the weight: last blocks of 1 to 32 rows of every height of a tile
@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(65, 31, 64), (66, 33, 192), (70, 37, 448), (96, 37, 576), (97, 127, 320), (128, 129, 448), (129, 257, 576),
                                   (129, 37, 4160), (159, 37, 4288), (180, 37, 704), (300, 145, 4288)])
def test_small_weights_through_lowbit_forward(qtype, dtype, m, n, k):
    """Sums, and infinities and a nan in the first and the last block of rows, at the last column and at ones that are read past the end."""
    if qtype in (FP8, 10):
        k = (k + 127) // 128 * 128 if qtype == FP8 else (k + 63) // 64 * 64
    blob, x = dev_quantize(weights(m, (n, k)), qtype, GGML), acts(m, m, k, dtype).cuda()
    w = dev_dequantize(blob, qtype, n, k, GGML, torch.float32).double()
    for odd in (False, True):
        if odd:
            x[3, k - k % 128 if k % 128 else k - 128], x[5, k - 1], x[m - 1, 5], x[m - 2, 3] = float("inf"), -float("inf"), float("nan"), -float("inf")
        want = x.double() @ w.t()
        size = x.double().nan_to_num(posinf=0.0, neginf=0.0).abs() @ w.t().abs()
        # fp32 sums of at most k / 32 scaled partial sums, themselves fp32; one rounding
        bound = size * (k // 32 + 8) * 2.0 ** -24 + want.abs() * torch.finfo(dtype).eps / 2 * (1 + 2.0 ** -10) + torch.finfo(dtype).smallest_normal
        y = torch.full((m + 2, n), float("nan"), dtype=dtype, device="cuda")
        ggml.lowbit_forward(x.data_ptr(), blob.data_ptr(), y[1].data_ptr(), qtype, GGML, DT[dtype], m, n, k, stream())
        assert torch.isnan(y[0]).all() and torch.isnan(y[m + 1]).all()
        got, finite = y[1:m + 1].double(), want.isfinite()
        assert ((got - want).abs() <= bound)[finite].all()
        assert (got.isnan() == want.isnan()).all() and (got == want)[want.isinf()].all()
        assert finite.all() != odd
