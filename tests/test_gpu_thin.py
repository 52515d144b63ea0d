"""The grouped forward's thin tiles (experts of at most 64 rows).

The launch takes the thin-capable kernel where the average expert has at most
128 rows; the same groups inside a taller operand (rows past the last group
end) take the 256-row kernel.  Every output element is the same chain of MFMAs
in both, so the rows inside the groups must be equal bit for bit, and both are
held against the float64 oracle.  N off the 128-column grid leaves a partial
tile and an empty second half.  The small launches give every workgroup at most
one work item (their load stream crosses from a tile's first 128 columns to its
second, with K below, at and past the six ring stages); the launches of several
rounds cross from tile to tile and from expert to expert.
"""
import numpy as np
import pytest
import torch

import mxfp8gg
from mxfp8gg import ops
from oracle import oracle as O
from tests._helpers import assert_close_to_oracle, u8
from tests.test_gpu_split import _rand_q

pytestmark = pytest.mark.gpu

SIZES = {
    "thin": [64, 0, 1, 60, 3, 61, 2, 64],          # starts on and off the 4-row grid
    "mixed": [5, 65, 64, 0, 128, 1, 300, 17],      # both kinds in one launch
    "one": [33],
}


def _case(gpu, sizes, N, K, scaled, seed):
    M, E = sum(sizes), len(sizes)
    a, a_s = _rand_q((M, K), gpu, seed)
    w, w_s = _rand_q((E, N, K), gpu, seed + 1)
    ends = torch.tensor(np.cumsum(sizes), dtype=torch.int32, device=gpu)
    return a, (a_s if scaled else None), w, (w_s if scaled else None), ends


def _taller(a, a_s, E):
    """The same rows in an operand of more than 128 rows per expert."""
    rows = 128 * E + 1 + a.shape[0]
    big = torch.zeros((rows, a.shape[1]), dtype=torch.uint8, device=a.device)
    big[:a.shape[0]] = a.view(torch.uint8)
    s = None
    if a_s is not None:
        s = torch.full((rows, a_s.shape[1]), 127, dtype=torch.uint8, device=a.device)
        s[:a.shape[0]] = a_s
    return big.view(a.dtype), s


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("scaled", [True, False])
@pytest.mark.parametrize("sizes,N,K", [
    ("thin", 128, 32), ("thin", 260, 640), ("thin", 136, 2080), ("mixed", 384, 768),
    ("mixed", 100, 1056), ("one", 512, 896),
])
def test_thin_tiles_equal_wide_tiles(gpu, sizes, N, K, scaled, out_dtype):
    sizes = SIZES[sizes]
    a, a_s, w, w_s, ends = _case(gpu, sizes, N, K, scaled, 11)
    y = ops.grouped_mm(a, w, ends, a_s, w_s, out_dtype=out_dtype, split_tail=False)
    big, big_s = _taller(a, a_s, len(sizes))
    wide = ops.grouped_mm(big, w, ends, big_s, w_s, out_dtype=out_dtype, split_tail=False)
    bits = torch.int16 if out_dtype == torch.bfloat16 else torch.int32
    assert torch.equal(y.view(bits), wide[:a.shape[0]].view(bits))
    ref = O.grouped_fwd(u8(a), u8(a_s) if scaled else None, u8(w), u8(w_s) if scaled else None,
                        np.cumsum(sizes))
    assert_close_to_oracle(y, ref)


@pytest.mark.parametrize("mode", ["rceil", "floor"])
@pytest.mark.parametrize("sizes,F,K", [("thin", 128, 96), ("mixed", 256, 1024), ("one", 128, 800)])
def test_thin_swiglu_equals_wide(gpu, sizes, F, K, mode):
    sizes = SIZES[sizes]
    g = torch.Generator(device=gpu).manual_seed(5)
    M, E = sum(sizes), len(sizes)
    x = torch.randn((M, K), generator=g, device=gpu).to(torch.bfloat16)
    w = (torch.randn((E, 2 * F, K), generator=g, device=gpu) * 0.05).to(torch.bfloat16)
    ends = torch.tensor(np.cumsum(sizes), dtype=torch.int32, device=gpu)
    a, a_s = mxfp8gg.to_mxfp8_dim0(x, mode)
    wq, ws = mxfp8gg.to_mxfp8_dim0(w, mode)
    q, s, h = ops.grouped_mm_swiglu_quant(a, wq, ends, a_s, ws, mode, return_h=True)
    q1, s1 = ops.grouped_mm_swiglu_quant(a, wq, ends, a_s, ws, mode)
    big, big_s = _taller(a, a_s.contiguous(), E)
    qw, sw, hw = ops.grouped_mm_swiglu_quant(big, wq, ends, big_s, ws, mode, return_h=True)
    assert torch.equal(h.view(torch.int16), hw[:M].view(torch.int16))
    for got in ((q, s), (q1, s1)):
        assert torch.equal(got[0].view(torch.uint8), qw[:M].view(torch.uint8))
        assert torch.equal(got[1], sw[:M])
    aq, as_ = ops.swiglu_quant(h, mode)
    assert torch.equal(q.view(torch.uint8), aq.view(torch.uint8)) and torch.equal(s, as_)


# ---------------------------------------------------------------------------
# Several rounds of the grid: a workgroup's second and later tiles, the load
# stream crossing from one expert's tile to another's, and the ring passing
# between thin and 256-row tiles.
# ---------------------------------------------------------------------------
def _tiles(sizes, n):
    """(256-row or thin) x 256-column tiles of a launch."""
    beg = np.cumsum(sizes) - sizes
    rows = np.where(np.asarray(sizes) > 0, np.asarray(sizes) + beg % 4, 0)
    return int(((rows + 255) // 256).sum()) * ((n + 255) // 256)


def _cus(gpu):
    return torch.cuda.get_device_properties(gpu).multi_processor_count


THIN_64 = [(37 * i) % 61 for i in range(64)]             # 0 .. 60 rows, all thin
MIXED_48 = [5, 65, 64, 0, 128, 1, 300, 17] * 6
WIDE_48 = [65 + 4 * (i % 16) for i in range(48)]         # no thin tile


def _equals_wide(gpu, sizes, N, K, scaled, out_dtype, split):
    a, a_s, w, w_s, ends = _case(gpu, sizes, N, K, scaled, 3)
    big, big_s = _taller(a, a_s, len(sizes))
    wide = ops.grouped_mm(big, w, ends, big_s, w_s, out_dtype=out_dtype, split_tail=split)
    bits = torch.int16 if out_dtype == torch.bfloat16 else torch.int32
    for _ in range(3):
        y = ops.grouped_mm(a, w, ends, a_s, w_s, out_dtype=out_dtype, split_tail=split)
        assert torch.equal(y.view(bits), wide[:a.shape[0]].view(bits))


@pytest.mark.parametrize("out_dtype,scaled", [(torch.bfloat16, True), (torch.float32, True),
                                              (torch.bfloat16, False)])
@pytest.mark.parametrize("sizes,K", [
    (THIN_64, 32),       # one stage a tile: six tiles of up to six experts in flight
    (THIN_64, 640), (THIN_64, 2080),
    (MIXED_48, 32), (MIXED_48, 640), (MIXED_48, 2080),
    (WIDE_48, 640),
])
def test_several_rounds_equal_wide_tiles(gpu, sizes, K, out_dtype, scaled):
    N = 4096
    assert _tiles(sizes, N) >= 2.5 * _cus(gpu)
    _equals_wide(gpu, sizes, N, K, scaled, out_dtype, False)


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("sizes,N,K", [
    # both kinds where a nearly full last round leaves the thin tiles out: whole
    # rounds of a long contraction, and the only round
    ([5, 65] * 16, 4096, 5280), ([5, 65, 20, 64, 1, 70, 33, 66], 7168, 2080),
    # every group index: 1024 groups, empty, thin and larger ones in any order
    ([(7 * i) % 5 + (70 if i % 97 == 3 else 0) for i in range(1024)], 128, 96),
    ([0] * 1000 + [66, 3, 0, 300] * 6, 300, 160),
])
def test_mixed_orders_equal_wide_tiles(gpu, sizes, N, K, out_dtype):
    _equals_wide(gpu, sizes, N, K, True, out_dtype, False)


def test_split_last_round_of_both_kinds(gpu):
    """The split cuts other tiles than in the 256-row kernel (groups of 256-row
    tiles come first), so sums differ by their order: fp32 sums of K products in
    two orders differ by at most 2 K 2^-24 times the sum of their magnitudes."""
    sizes, N, K = [30, 66, 0, 64, 5, 80, 1, 300, 17, 2, 40] * 3, 4096, 2080
    rem = _tiles(sizes, N) % _cus(gpu)
    assert _tiles(sizes, N) > _cus(gpu) and 0 < rem <= _cus(gpu) // 2
    a, a_s, w, w_s, ends = _case(gpu, sizes, N, K, True, 3)
    y = ops.grouped_mm(a, w, ends, a_s, w_s, out_dtype=torch.float32, split_tail=True)
    whole = ops.grouped_mm(a, w, ends, a_s, w_s, out_dtype=torch.float32, split_tail=False)
    size = ops.grouped_mm((a.view(torch.uint8) & 0x7F).view(a.dtype),
                          (w.view(torch.uint8) & 0x7F).view(w.dtype), ends, a_s, w_s,
                          out_dtype=torch.float32, split_tail=False)
    assert ((y.double() - whole.double()).abs() <= 2 * K * 2.0 ** -24 * size.double()).all()
    for _ in range(3):   # the same bits on every call
        again = ops.grouped_mm(a, w, ends, a_s, w_s, out_dtype=torch.float32, split_tail=True)
        assert torch.equal(again, y)


def test_split_last_round_of_thin_tiles(gpu):
    """33 thin experts over 16 column tiles: two whole rounds, then 16 tiles cut
    along K, each of two thin pieces; the same tiles and ranges as in the
    256-row kernel, so the same bits."""
    sizes, N, K = [1 + (7 * i) % 60 for i in range(33)], 4096, 2080
    rem = _tiles(sizes, N) % _cus(gpu)
    assert _tiles(sizes, N) > _cus(gpu) and 0 < rem <= _cus(gpu) // 2
    for dtype in (torch.bfloat16, torch.float32):
        _equals_wide(gpu, sizes, N, K, True, dtype, True)


@pytest.mark.parametrize("keep", [False, True])
@pytest.mark.parametrize("sizes,K", [(THIN_64 * 2, 32), (THIN_64 * 2, 800), (MIXED_48 * 2, 96),
                                     (MIXED_48 * 2, 800), (WIDE_48 * 2, 800)])
def test_swiglu_several_rounds_equal_wide(gpu, sizes, K, keep):
    F, E, M = 1024, len(sizes), sum(sizes)
    assert _tiles(sizes, 2 * F) >= 2.5 * _cus(gpu)
    a, a_s, w, w_s, ends = _case(gpu, sizes, 2 * F, K, True, 9)
    big, big_s = _taller(a, a_s, E)
    want = ops.grouped_mm_swiglu_quant(big, w, ends, big_s, w_s, return_h=keep)
    for _ in range(3):
        got = ops.grouped_mm_swiglu_quant(a, w, ends, a_s, w_s, return_h=keep)
        for x, y in zip(got, want):
            assert torch.equal(x.contiguous().view(torch.uint8),
                               y[:M].contiguous().view(torch.uint8))
