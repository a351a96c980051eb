"""Decode attention where one wave's keys weigh next to nothing beside another's: the weights of the merge keep what
32 bits hold of them."""
import math

import pytest
import torch

from llm_inference_lab_amd.cache import layout as cache_layout
from test_kernels_gpu import DEV, ops      # noqa: F401 (fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d", [16, 64, 128, 256])
@pytest.mark.parametrize("splits", [1, 2])
def test_weights_below_the_smallest_normal_number(ops, dtype, d, splits):      # noqa: F811
    """The first 32 keys score 0 with values of zero, one of the last 32 scores -90 with values of 1e38, all others -200:
    the last wave's weight is e^-90, 2^-129.8, and its sum 1e38."""
    page, keys = 64, 256 * splits
    far = [keys - 27]
    kc, vc = torch.zeros(keys // page, 1, page, d), torch.zeros(keys // page, 1, d, page)
    for k in range(32, keys):
        kc[k // page, 0, k % page, 0] = -90.0 if k in far else -200.0
    for k in far:
        vc[k // page, 0, :, k % page] = 1e38
    kc, vc = cache_layout.keys_to_cache_order(kc.to(dtype)), cache_layout.values_to_cache_order(vc.to(dtype))
    q = torch.zeros(1, 3 * d, dtype=dtype)
    q[0, 0] = 1.0
    out = torch.zeros(1, d, dtype=dtype, device=DEV)
    ints = [torch.tensor(v, dtype=torch.int32, device=DEV) for v in ([list(range(keys // page))], [0, 1], [keys - 1])]
    with ops.debug.force(attention_splits=(d, splits)):
        ops.paged_attention(q.to(DEV), 1, 1, d, kc.to(DEV), vc.to(DEV), ints[0], page, ints[1], ints[2], 1, 1, keys, None,
                            1.0, out)
    want = len(far) * math.exp(-90.0) * float(torch.tensor(1e38).to(dtype)) / 32
    # (a weight below 2^-126 has 19 of its 24 bits; bfloat16: the result's one rounding)
    assert bool(((out.double().cpu() - want).abs() <= want * (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -15)).all())
