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


# ---------------------------------------------------------------------------
# Several rounds of the grid: the stores of a tile stay in flight behind the
# next tile's loads from a workgroup's second tile on.
# ---------------------------------------------------------------------------
def _operands(gpu, sizes, n, k):
    g = torch.Generator(device=gpu).manual_seed(n + k + len(sizes))
    rows = sum(sizes)
    ends = torch.tensor(np.cumsum(sizes), dtype=torch.int32, device=gpu)
    dy = torch.randn((rows, (n + 31) // 32 * 32), generator=g, device=gpu).to(torch.bfloat16)
    x = torch.randn((rows, (k + 31) // 32 * 32), generator=g, device=gpu).to(torch.bfloat16)
    go, gos, pad = ops.to_mxfp8_dim1(dy, ends)
    ia, ias, _ = ops.to_mxfp8_dim1(x, ends)
    return go[:n], gos[:n], ia[:k], ias[:k], pad


@pytest.mark.parametrize("n,k", [(2048, 1024),     # every wave inside dW
                                 (2000, 1032)])    # guarded waves beside interior ones
@pytest.mark.parametrize("sizes", [
    [64] * 32, [128] * 32,            # one stage
    [200] * 32, [256] * 32,           # two, or three where the start is off the 128-token grid
    [385] * 32, [640] * 32,           # three to six
    [200, 256, 385, 640, 33, 128, 100, 500] * 4,
    [640, 0, 31, 128, 0, 256, 7, 500] * 4,          # empty experts last, without loads
    [700] + [0] * 15 + [90] * 16,
])
def test_several_rounds_equal_rounded_fp32(gpu, sizes, n, k):
    tiles = len(sizes) * ((n + 255) // 256) * ((k + 255) // 256)
    assert tiles >= 3 * torch.cuda.get_device_properties(gpu).multi_processor_count
    go, gos, ia, ias, pad = _operands(gpu, sizes, n, k)
    want = ops.grouped_wgrad(go, ia, pad, gos, ias, out_dtype=torch.float32, split_tokens=0)
    out = torch.full((len(sizes), n, k), 7.0, dtype=torch.bfloat16, device=gpu)
    for _ in range(3):
        ops.grouped_wgrad(go, ia, pad, gos, ias, out=out, out_dtype=torch.bfloat16, split_tokens=0)
        assert torch.equal(out.view(torch.int16), want.to(torch.bfloat16).view(torch.int16))


@pytest.mark.parametrize("at", [0, 7, 30])
def test_nan_experts_between_full_ones(gpu, at):
    """A boundary inside a 32-token block: both experts at it are NaN, without
    loads, among experts of several stages in the same workgroups."""
    n, k, sizes = 2048, 1024, [300, 160, 512, 96] * 8
    go, gos, ia, ias, pad = _operands(gpu, sizes, n, k)
    ends = pad.as_subclass(torch.Tensor).clone()
    ends[at] += 8
    want = ops.grouped_wgrad(go, ia, ends, gos, ias, out_dtype=torch.float32, split_tokens=0)
    out = torch.full((len(sizes), n, k), 7.0, dtype=torch.bfloat16, device=gpu)
    for _ in range(3):
        ops.grouped_wgrad(go, ia, ends, gos, ias, out=out, out_dtype=torch.bfloat16,
                          split_tokens=0)
        nan = out.isnan().flatten(1)
        assert nan[at:at + 2].all() and not nan[:at].any() and not nan[at + 2:].any()
        keep = [e for e in range(len(sizes)) if e not in (at, at + 1)]
        assert torch.equal(out[keep], want[keep].to(torch.bfloat16))
