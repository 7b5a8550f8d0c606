"""The one-pass kernel for up to 64 rows: rows around its 16-row blocks, tile rows around the 1 .. 4 a workgroup owns, fewer
and more column groups than waves; both layouts, float32 activations, and the fused gate/up form."""
import numpy as np
import pytest
import torch

import lowbit_oracle as orc
import ipex_llm.ggml.model.llama.llama_cpp as ggml
from gpu_util import ALL, DT, FP8, NF4, acts, dev_dequantize, dev_quantize, stream, weights
from ipex_llm.transformers.low_bit_linear import mlp_forward_xpu
from ipex_llm.transformers.models.utils import SILU
from test_linear_gpu import GGML, TILED, _check, classes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(9, 16, 128), (16, 48, 3200), (16, 4112, 256), (17, 1040, 1408), (32, 8208, 128), (33, 4144, 256),
                                   (48, 12304, 128), (49, 272, 1152), (64, 8224, 256), (64, 16, 6144), (18, 16416, 256), (31, 12304, 640)])
def test_tiled_weights(qtype, dtype, m, n, k):
    _check(qtype, dtype, TILED, m, n, k, m % 2 == 0, 700 * m + n)


@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(5, 4099, 192), (8, 17, 1600), (16, 8201, 128), (17, 4101, 320), (48, 8199, 64), (64, 1023, 1216), (32, 16387, 192)])
def test_row_major_weights(qtype, dtype, m, n, k):
    if qtype == FP8:
        k = (k + 127) // 128 * 128
    _check(qtype, dtype, GGML, m, n, k, m % 2 == 0, 800 * m + n)


@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("layout,m,n,k", [(TILED, 9, 48, 1408), (TILED, 16, 4112, 128), (TILED, 17, 4112, 384), (TILED, 32, 16, 128),
                                          (TILED, 75, 64, 512), (GGML, 10, 4099, 192), (GGML, 31, 33, 1088)])
def test_float32_activations(qtype, layout, m, n, k):
    if qtype == FP8:
        k = (k + 127) // 128 * 128
    _check(qtype, torch.float32, layout, m, n, k, m % 2 == 0, 900 * m + n)


# rows dealt to several workgroups: rests of 1 to 4 blocks of rows, tile rows that 1 to 4 a workgroup do not divide, one workgroup and 256
@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("layout,m,n,k", [(TILED, 17, 1024, 2176), (TILED, 33, 528, 1152), (TILED, 64, 2064, 384), (TILED, 65, 1040, 1152),
                                          (TILED, 97, 48, 3200), (TILED, 130, 2064, 640), (TILED, 217, 1024, 1408), (TILED, 128, 4096, 2048),
                                          (TILED, 500, 512, 384), (TILED, 1024, 272, 256), (TILED, 1024, 16, 128), (GGML, 40, 1003, 704),
                                          (GGML, 66, 1001, 1088), (GGML, 200, 2003, 320), (GGML, 513, 300, 192), (GGML, 1024, 7, 64)])
def test_rows_dealt_to_several_workgroups(qtype, dtype, layout, m, n, k):
    if qtype == FP8:
        k = (k + 127) // 128 * 128
    assert ggml.lowbit_linear_scratch_bytes(qtype, layout, DT[dtype], m, n, k, 64 << 20) == 0
    _check(qtype, dtype, layout, m, n, k, m % 2 == 0, 720 * m + n)


def dealt_sizes(qtype, layout, dtype):
    """(tile rows, blocks of rows) per workgroup -> a size of it, of 17 to 1024 rows on up to 4 million weights."""
    rng, sizes = np.random.default_rng(11), {}
    for lm, ln, lk in rng.random((6000, 3)):
        m, n, k = int(17 * 60.3 ** lm), int(20 * 300 ** ln), int(64 * 40 ** lk) // 32 * 32
        n = (n + 15) // 16 * 16 if layout == TILED else n
        k = (k + 127) // 128 * 128 if layout == TILED or qtype == FP8 else (k + 63) // 64 * 64 if qtype == NF4 else k
        plan, shape = ggml.lowbit_linear_plan(qtype, layout, dtype, m, n, k, 64 << 20)
        if plan == ggml.PLAN_ONE_PASS and n * k <= 4e6 and m * n <= 2e6 and m > 16 * shape[2]:
            sizes.setdefault((shape[0], shape[2]), (m, n, k))
    return sizes


@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("layout", [TILED, GGML])
def test_every_shape_of_rows_dealt_to_several_workgroups(qtype, dtype, layout):
    sizes = dealt_sizes(qtype, layout, DT[dtype])
    assert len(sizes) >= 8
    for m, n, k in sizes.values():
        blob, x = dev_quantize(weights(n, (n, k)), qtype, layout), acts(m, m, k, dtype).cuda()
        dense = dev_dequantize(blob, qtype, n, k, layout, torch.float32).double()
        y = torch.full((m + 1, n), float("nan"), dtype=dtype, device="cuda")
        ggml.lowbit_linear(x.data_ptr(), blob.data_ptr(), None, y.data_ptr(), qtype, layout, DT[dtype], m, n, k, None, 0, stream())
        want, eps = x.double() @ dense.t(), torch.finfo(dtype).eps
        # as in test_few_rows_of_many_tile_rows
        err = 2.0 ** -24 * 2 * 17 * (k / 32 + 33) + (eps / 2 if qtype == NF4 else 0.0)
        bound = want.abs() * eps / 2 + x.double().abs().sum(1, keepdim=True) * dense.abs().amax(1) * err + torch.finfo(dtype).smallest_normal
        assert ((y[:m].double() - want).abs() <= bound).all() and torch.isnan(y[m]).all(), (m, n, k)


@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("layout,m,n,k", [(TILED, 17, 1024, 1408), (TILED, 32, 6160, 256), (TILED, 33, 5440, 256), (TILED, 48, 1040, 1152),
                                          (TILED, 64, 48, 128), (GGML, 20, 3001, 320), (GGML, 40, 1001, 1088), (GGML, 63, 2003, 192)])
def test_float32_rows_dealt_to_several_workgroups(qtype, layout, m, n, k):
    if qtype == FP8:
        k = (k + 127) // 128 * 128
    _check(qtype, torch.float32, layout, m, n, k, m % 2 == 0, 730 * m + n)


@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("layout,m,n,k", [(TILED, 100, 1040, 256), (GGML, 70, 301, 320)])
def test_infinities_in_rows_dealt_to_several_workgroups(qtype, dtype, layout, m, n, k):
    if qtype == FP8:
        k = (k + 127) // 128 * 128
    w, x = weights(m, (n, k)), acts(m + 1, m, k, dtype)
    x[0, 5], x[m // 2, k - 3], x[m - 1, 7] = float("inf"), -float("inf"), float("nan")
    blob, xd = dev_quantize(w, qtype, layout), x.cuda()
    y = torch.empty((m, n), dtype=dtype, device="cuda")
    ggml.lowbit_linear(xd.data_ptr(), blob.data_ptr(), None, y.data_ptr(), qtype, layout, DT[dtype], m, n, k, None, 0, stream())
    with np.errstate(all="ignore"):
        want = x.double().numpy() @ orc.dequantize(orc.quantize(w, qtype), qtype, (n, k)).astype(np.float64).T
    assert (classes(y.float().cpu().numpy()) == classes(want)).all()


# where 5 to 16 rows go to this kernel: around 512, 768, 1024, 1536 and 2048 tile rows, 24 and 64 groups
@pytest.mark.parametrize("qtype,dtype", [(2, torch.float16), (3, torch.bfloat16), (8, torch.float16), (10, torch.bfloat16), (15, torch.bfloat16)])
@pytest.mark.parametrize("layout,m,n,k", [(TILED, 5, 8208, 3072), (TILED, 8, 12288, 3072), (TILED, 7, 4112, 8192), (TILED, 8, 8192, 8192),
                                          (TILED, 6, 19456, 3072), (TILED, 8, 24592, 3072), (TILED, 9, 16400, 256), (TILED, 16, 24576, 128),
                                          (TILED, 12, 24592, 3072), (TILED, 9, 32784, 128), (GGML, 9, 16401, 3072), (GGML, 16, 24577, 3072),
                                          (GGML, 13, 32769, 3072)])
def test_few_rows_of_many_tile_rows(qtype, dtype, layout, m, n, k):
    w = np.random.default_rng(m + n).standard_normal((n, k), dtype=np.float32) * 0.02
    blob, x = dev_quantize(w, qtype, layout), acts(m, m, k, dtype).cuda()
    y = torch.full((m + 1, n), float("nan"), dtype=dtype, device="cuda")
    x_inf = x.clone()
    x_inf[0, 5], x_inf[m - 1, k - 3] = float("inf"), -float("inf")
    dense = dev_dequantize(blob, qtype, n, k, layout, torch.float32).double()
    ggml.lowbit_linear(x.data_ptr(), blob.data_ptr(), None, y.data_ptr(), qtype, layout, DT[dtype], m, n, k, None, 0, stream())
    want, eps = x.double() @ dense.t(), torch.finfo(dtype).eps
    # one rounding, those of fp32 sums over k / 32 blocks of 32 products each, of codes that carry 17 times their value at most, and of
    # nf4's levels to x's type
    err = 2.0 ** -24 * 2 * 17 * (k / 32 + 33) + (eps / 2 if qtype == NF4 else 0.0)
    bound = want.abs() * eps / 2 + x.double().abs().sum(1, keepdim=True) * dense.abs().amax(1) * err + torch.finfo(dtype).smallest_normal
    assert ((y[:m].double() - want).abs() <= bound).all() and torch.isnan(y[m]).all()
    if m > 8 or layout == GGML:                            # (fewer rows may go to the streaming kernel, which gives NaN for some of these)
        ggml.lowbit_linear(x_inf.data_ptr(), blob.data_ptr(), None, y.data_ptr(), qtype, layout, DT[dtype], m, n, k, None, 0, stream())
        want = torch.where(dense[:, 5] == 0, torch.nan, torch.copysign(torch.full_like(dense[:, 5], torch.inf), dense[:, 5]))
        assert torch.equal(torch.nan_to_num(y[0].float(), nan=7.0, posinf=1.0, neginf=-1.0),
                           torch.nan_to_num(want.float(), nan=7.0, posinf=1.0, neginf=-1.0))


# the sizes of 5 to 16 rows that only lowbit_linear gives to this kernel
@pytest.mark.parametrize("qtype,dtype", [(2, torch.float16), (3, torch.bfloat16), (8, torch.float16), (10, torch.bfloat16), (15, torch.bfloat16)])
@pytest.mark.parametrize("layout,m,n,k", [(TILED, 5, 8208, 3072), (TILED, 8, 12288, 3072), (TILED, 7, 4880, 8192), (TILED, 8, 8192, 8192),
                                          (TILED, 6, 24592, 3072), (TILED, 9, 16400, 256), (TILED, 12, 24592, 3072), (GGML, 9, 16401, 3072),
                                          (GGML, 13, 32769, 3072)])
def test_forward_keeps_the_streaming_kernel(qtype, dtype, layout, m, n, k):
    """lowbit_forward and lowbit_forward_ws give the streaming kernel's bits, with whatever alignment of y."""
    blob = dev_quantize(np.random.default_rng(m + n).standard_normal((n, k), dtype=np.float32) * 0.02, qtype, layout)
    x = acts(m, m, k, dtype).cuda()
    y = torch.full((4, (m * n + 23) // 8 * 8), float("nan"), dtype=dtype, device="cuda")
    args = (qtype, layout, DT[dtype], m, n, k)
    ggml.lowbit_gemv(x.data_ptr(), blob.data_ptr(), y[0].data_ptr(), *args, 0, stream())
    ggml.lowbit_forward(x.data_ptr(), blob.data_ptr(), y[1].data_ptr(), *args, stream())
    ggml.lowbit_forward_ws(x.data_ptr(), blob.data_ptr(), y[2].data_ptr(), *args, None, 0, stream())
    ggml.lowbit_forward(x.data_ptr(), blob.data_ptr(), y[3][1:].data_ptr(), *args, stream())
    want = y[0, :m * n]
    assert want.isfinite().all() and torch.equal(y[1, :m * n], want) and torch.equal(y[2, :m * n], want) and torch.equal(y[3, 1:m * n + 1], want)


# tile rows that three and four do not divide, 12 waves with fewer and more groups, several workgroups of four waves per CU
@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("layout,m,n,k", [(TILED, 12, 48, 1664), (TILED, 9, 8224, 256), (TILED, 32, 8240, 1152), (TILED, 16, 12336, 1152),
                                          (TILED, 17, 12336, 640), (TILED, 10, 16400, 640), (TILED, 24, 16416, 128), (GGML, 12, 33, 1728),
                                          (GGML, 9, 8215, 1088), (GGML, 31, 8231, 192), (GGML, 16, 12299, 320), (GGML, 18, 16401, 320)])
def test_float32_activations_shared_by_tile_rows(qtype, layout, m, n, k):
    if qtype == FP8:
        k = (k + 127) // 128 * 128
    _check(qtype, torch.float32, layout, m, n, k, m % 2 == 0, 950 * m + n)


# 12 waves and 8 beside them: fewer groups than waves, one more, a whole second round, and long walks
@pytest.mark.parametrize("qtype,layout,m,n,k,waves", [(q, TILED, m, 48, k, 12) for q in (2, 3, NF4) for m, k in ((9, 1152), (13, 1536), (10, 1664), (13, 3968))]
                         + [(q, GGML, m, 33, k, 12) for q in (2, 3) for m, k in ((9, 1600), (13, 3904))] + [(NF4, TILED, 16, 48, k, 12) for k in (1664, 3968)]
                         + [(q, TILED, 16, 48, k, 8) for q in (2, 3) for k in (1536, 1664, 3968)]
                         + [(q, TILED, 9, 48, 1664, 8) for q in (8, FP8)] + [(q, GGML, 9, 33, 1664, 8) for q in (8, NF4, FP8)])
def test_float32_activations_in_8_and_12_waves(qtype, layout, m, n, k, waves):
    assert ggml.lowbit_linear_plan(qtype, layout, ggml.DT_F32, m, n, k) == (ggml.PLAN_ONE_PASS, (1, waves, 1))
    _check(qtype, torch.float32, layout, m, n, k, m % 2 == 0, 960 * m + n)


@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("layout,m,n,k", [(TILED, 9, 48, 256), (TILED, 20, 8224, 128), (TILED, 16, 12336, 128), (GGML, 17, 8215, 128)])
def test_float32_activations_beyond_bfloat16(qtype, layout, m, n, k):
    """Infinities, a NaN, and a finite value that rounds to an infinity in bfloat16: what its second plane would be is not used."""
    w, x = weights(m + n, (n, k)), acts(m, m, k, torch.float32)
    x[0, 5], x[m // 2, k - 3], x[1, 7], x[2, 9] = float("inf"), -float("inf"), float("nan"), 3.4e38
    blob, y = dev_quantize(w, qtype, layout), torch.empty((m, n), dtype=torch.float32, device="cuda")
    xd = x.cuda()
    ggml.lowbit_linear(xd.data_ptr(), blob.data_ptr(), None, y.data_ptr(), qtype, layout, ggml.DT_F32, m, n, k, None, 0, stream())
    got = y.cpu().numpy()
    dense = orc.dequantize(orc.quantize(w, qtype), qtype, (n, k)).astype(np.float64)
    with np.errstate(all="ignore"):
        want = (x.double().numpy() @ dense.T).astype(np.float32)
    assert (classes(got) == classes(want)).all()
    assert np.isfinite(want[2]).all() and (classes(want[0]) > 1).any()
    # float32 sums of products in float32
    assert np.abs(got[2] - want[2]).max() <= k * 2.0 ** -23 * 3.4e38 * np.abs(dense[:, 9]).max()


@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("m,n,k", [(7, 8208, 128), (9, 16, 128), (16, 4144, 1152), (17, 4112, 128), (33, 8208, 128), (48, 4112, 384),
                                   (49, 4112, 256), (64, 272, 1408), (32, 16400, 128)])
def test_fused_gate_up(qtype, m, n, k):
    dtype = torch.float16 if m % 2 else torch.bfloat16
    wg, wu, x = weights(m + n, (n, k)), weights(m + n + 1, (n, k)), acts(m, m, k, dtype)
    y = mlp_forward_xpu(x.cuda(), dev_quantize(wg, qtype, TILED), dev_quantize(wu, qtype, TILED), m, k, n, SILU, qtype).float().cpu().numpy()
    g, u = (orc.mul_mat_exact(orc.quantize(w, qtype), x.float().numpy(), (n, k), qtype) for w in (wg, wu))
    want = g / (1.0 + np.exp(-g)) * u
    assert np.abs(y - want).max() <= (2e-3 if dtype == torch.float16 else 8e-3) * np.abs(want).max()


def gated_mlp(x, wg, wu, m, k, n, act, qtype):
    y = torch.full((m + 1, n), float("nan"), dtype=x.dtype, device="cuda")
    ggml.lowbit_gated_mlp(x.data_ptr(), wg.data_ptr(), wu.data_ptr(), y.data_ptr(), qtype, DT[x.dtype], m, n, k, 0, stream())
    assert torch.isnan(y[m]).all()
    return y[:m]


# 17 rows and more, dealt to several workgroups
@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(17, 1040, 1152), (33, 272, 640), (64, 2064, 384), (65, 1040, 1408), (130, 1024, 2048), (200, 528, 3200),
                                   (600, 256, 2176), (1024, 48, 1280)])
def test_fused_gate_up_rows_dealt(qtype, dtype, m, n, k):
    test_fused_gate_up_of_many_workgroups(qtype, dtype, m, n, k, gated_mlp)


@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(12, 16400, 640), (20, 8336, 512), (40, 8336, 640), (48, 12304, 1152)])
def test_fused_gate_up_of_many_workgroups(qtype, dtype, m, n, k, run=mlp_forward_xpu):
    """More workgroups of four waves than the GPU holds at once in the form of more registers; K of as many groups as waves, and more."""
    blobs = [dev_quantize(weights(m + i, (n, k)), qtype, TILED) for i in range(2)]
    x = acts(m, m, k, dtype).cuda()
    y = run(x, *blobs, m, k, n, SILU, qtype).double()
    eps = torch.finfo(dtype).eps
    # fp32 sums of exact products; the levels of nf4 are rounded to x's type
    err = k * 2.0 ** -24 + (eps / 2 if qtype == NF4 else 0.0)
    (g, dg), (u, du) = ((x.double() @ w.t(), x.double().abs() @ w.abs().t() * err)
                        for w in (dev_dequantize(b, qtype, n, k, TILED, torch.float32).double() for b in blobs))
    a = g * torch.sigmoid(g)
    # one rounding; exp2 and rcp of an ulp each; silu's slope is at most 1.13
    bound = (a * u).abs() * (eps / 2 + 2.0 ** -20) + 1.13 * dg * u.abs() + a.abs() * du + dg * du + torch.finfo(dtype).smallest_normal
    assert ((y - a * u).abs() <= bound).all()


@pytest.mark.parametrize("qtype", ALL)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(9, 48, 256), (24, 4112, 128), (64, 48, 256)])
def test_fused_gate_up_with_infinities(qtype, dtype, m, n, k):
    wg, wu, x = weights(m, (n, k)), weights(m + 1, (n, k)), acts(m, m, k, dtype)
    x[0, 5], x[m // 2, k - 3] = float("inf"), -float("inf")
    y = mlp_forward_xpu(x.cuda(), dev_quantize(wg, qtype, TILED), dev_quantize(wu, qtype, TILED), m, k, n, SILU, qtype).float().cpu().numpy()
    with np.errstate(all="ignore"):
        g, u = (x.double().numpy() @ orc.dequantize(orc.quantize(w, qtype), qtype, (n, k)).astype(np.float64).T for w in (wg, wu))
        want = g / (1.0 + np.exp(-g)) * u
    assert (classes(y) == classes(want)).all()
    assert (classes(want) > 1).any() and (classes(want) == 0).any()
