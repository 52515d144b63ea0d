"""The weight gradient whose tile stores overlap the next tile's loads (bf16 dW,
few tokens per expert) against the fp32 weight gradient.

Both accumulate the same products in the same order, so dW must be the fp32
result rounded to bf16, bit for bit."""
import numpy as np
import pytest
import torch

from mxfp8gg import ops

pytestmark = pytest.mark.gpu

# tokens of the experts: none, one stage (128), the last of one and first of
# two, two, three and more stages, and many empty experts between full ones
GROUPS = [[1], [128], [129], [256], [257], [385], [0, 0, 300, 0], [640, 0, 31, 128, 0, 256, 7, 500],
          [0] * 5, [33] * 16,
          # an average on either side of the 768 tokens the dispatch changes at
          [640], [740, 736], [770], [900, 1100]]
# tiles of 256, halves of 128 and remainders on both sides
WIDTHS = [(256, 256), (512, 768), (384, 128), (40, 264), (1, 8), (520, 1056), (2048, 1024)]


@pytest.mark.parametrize("sizes", GROUPS)
@pytest.mark.parametrize("n,k", WIDTHS)
def test_equals_rounded_fp32(gpu, sizes, n, k):
    g = torch.Generator(device=gpu).manual_seed(n + k)
    rows = max(sum(sizes), 1)
    ends = torch.tensor(np.cumsum(sizes), dtype=torch.int32, device=gpu)
    dy = torch.randn((rows, (n + 7) // 8 * 8), generator=g, device=gpu).to(torch.bfloat16)
    x = torch.randn((rows, k), generator=g, device=gpu).to(torch.bfloat16)
    go, gos, pad = ops.to_mxfp8_dim1(dy, ends)
    ia, ias, _ = ops.to_mxfp8_dim1(x, ends)
    go, gos = go[:n], gos[:n]
    want = ops.grouped_wgrad(go, ia, pad, gos, ias, out_dtype=torch.float32, split_tokens=0)
    out = torch.full((len(sizes), n, k), 7.0, dtype=torch.bfloat16, device=gpu)
    for _ in range(3):
        ops.grouped_wgrad(go, ia, pad, gos, ias, out=out, out_dtype=torch.bfloat16, split_tokens=0)
        assert torch.equal(out, want.to(torch.bfloat16))


def test_boundary_inside_a_block_is_nan(gpu):
    x = torch.ones((256, 256), dtype=torch.bfloat16, device=gpu)
    q, s, _ = ops.to_mxfp8_dim1(x)
    ends = torch.tensor([40, 128, 256], dtype=torch.int32, device=gpu)
    dw = ops.grouped_wgrad(q, q, ends, s, s, out_dtype=torch.bfloat16, split_tokens=0)
    assert dw[:2].isnan().all() and (dw[2] == 128.0).all()
