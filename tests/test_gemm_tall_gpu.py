"""The 256-row tile of the GEMM where M is no multiple of its rows: last row tiles of 129 to 255 rows (rows of x past M),
one, two and three 128-column steps, a last column tile that is not full, columns left to the 128-row form."""
import pytest
import torch

from gpu_util import ALL, DT, NAMES, dev_dequantize, dev_quantize, ggml, stream, weights

pytestmark = pytest.mark.gpu
TILED = ggml.LAYOUT_TILED


def check(qtype, m, n, k, dtype, gemm, shift=0):
    blob = dev_quantize(weights(77, (n, k)), qtype, TILED)
    gen = torch.Generator().manual_seed(m)
    x = torch.randn((m, k), generator=gen).to(dtype).cuda()
    y = torch.full(((m + 1) * n + shift,), float("nan"), dtype=dtype, device="cuda")[shift:].view(m + 1, n)
    gemm(x.data_ptr(), blob.data_ptr(), y.data_ptr(), qtype, TILED, DT[dtype], m, n, k, stream())
    w = dev_dequantize(blob, qtype, n, k, TILED, torch.float32).to(dtype).float()
    want, size = x.double() @ w.double().t(), x.abs().float() @ w.abs().t()
    assert torch.isnan(y[m]).all()
    # one rounding of the result; fp32 sums over k terms; 16-bit weights rounded once from the same fp32 value, which
    # asym_int4 (q * d + m) rounds a second time here
    eps = torch.finfo(dtype).eps
    bound = want.abs() * eps / 2 + size * (k * 2.0 ** -24 + (eps if qtype == 3 else 0.0)) + torch.finfo(dtype).smallest_normal
    assert ((y[:m].double() - want).abs() <= bound).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("m,n,k", [(897, 16384, 256), (1023, 16368, 384), (1000, 28672, 128), (767, 38160, 256)])
@pytest.mark.parametrize("qtype", ALL, ids=NAMES.values())
def test_last_row_tile(qtype, m, n, k, dtype):
    check(qtype, m, n, k, dtype, ggml.lowbit_gemm)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("m,n,k", [(385, 17136, 256), (700, 11520, 384), (512, 32752, 128), (897, 24832, 1024), (1000, 20496, 2048)])
@pytest.mark.parametrize("qtype", ALL, ids=NAMES.values())
def test_rounds_that_are_partly_filled(qtype, m, n, k, dtype):
    """All columns in tall tiles: half a round and more of them, a last round that is half full; and whole rounds with a rest."""
    check(qtype, m, n, k, dtype, ggml.lowbit_gemm)


@pytest.mark.parametrize("qtype", ALL, ids=NAMES.values())
def test_rest_of_the_columns_ends_on_three_blocks(qtype):
    """2016 rows: a last tall tile of 224 rows, and what is left of the columns in tiles of 128 rows, the last of 96."""
    check(qtype, 2016, 11008, 512, torch.bfloat16, ggml.lowbit_gemm)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("m,n,k", [(1, 16, 128), (32, 144, 256), (33, 128, 384), (64, 272, 640), (65, 1040, 512), (200, 4096, 1152)])
def test_narrow_nf4(m, n, k, dtype):
    """Row blocks 1, 2 and 4 of the narrow tile, whose nf4 lookups are in registers."""
    check(10, m, n, k, dtype, ggml.lowbit_gemm_narrow)


@pytest.mark.parametrize("m,n,k,shift", [(1, 16, 1024, 0), (33, 144, 1152, 4), (64, 272, 1024, 0), (65, 1040, 1152, 0), (129, 144, 1408, 4),
                                         (250, 2048, 1152, 0), (2048, 2048, 1024, 0), (2040, 2064, 1024, 0), (100, 512, 896, 0)])
@pytest.mark.parametrize("qtype", ALL, ids=NAMES.values())
def test_narrow_two_groups(qtype, m, n, k, shift):
    """Two groups of waves on one tile: 1, 2 and 4 row blocks, half tiles, an odd number of K steps, a last column tile that
    is not full, a y off the 16-byte boundaries; 256 workgroups and 272, eight K steps and seven, where the form ends."""
    check(qtype, m, n, k, torch.bfloat16 if n % 32 else torch.float16, ggml.lowbit_gemm_narrow, shift)


def test_row_major_weights_of_very_long_rows():
    """Rows of x beyond 2^24 bytes: past the 32-bit offsets of the batch kernel for row-major weights."""
    m, n, k = 17, 3, (1 << 23) + 32
    gen = torch.Generator(device="cuda").manual_seed(5)
    w = torch.randn((n, k), generator=gen, device="cuda") * 0.02
    x = torch.randn((m, k), generator=gen, device="cuda").half()
    blob = torch.empty(ggml.lowbit_blob_bytes(2, n * k), dtype=torch.uint8, device="cuda")
    ggml.lowbit_quantize(w.data_ptr(), blob.data_ptr(), 2, n, k, ggml.LAYOUT_GGML, stream())
    y = torch.empty((m, n), dtype=torch.float16, device="cuda")
    ggml.lowbit_forward(x.data_ptr(), blob.data_ptr(), y.data_ptr(), 2, ggml.LAYOUT_GGML, DT[torch.float16], m, n, k, stream())
    w = dev_dequantize(blob, 2, n, k, ggml.LAYOUT_GGML, torch.float32).double()
    want = torch.stack([(x.double() * w[i]).sum(1) for i in range(n)], 1)
    # one rounding to 16 bits (sums of about 60); fp32 sums of 2^23 terms, whose rounding errors add up like a random walk
    assert (y.double() - want).abs().max() <= 2.0 ** -11 * want.abs().max() + 0.05
