"""The batch kernel for row-major weights: rows of x around its 32-row blocks and its tiles of 32, 64 and 128, weight rows around a
wave's 32 and a workgroup's 128, last steps of one to four blocks, one step, odd and even numbers of them, K splits."""
import numpy as np
import pytest
import torch

import lowbit_oracle as orc
from gpu_util import ALL, DT, FP8, acts, dev_quantize, ggml, stream, weights
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
