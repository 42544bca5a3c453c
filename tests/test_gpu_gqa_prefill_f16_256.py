"""Chunks over f16 rows of head_dim 256, the walks of 576 keys and more in two halves (gqa_prefill_f16_256.hpp): pages they address by scalars and
others, ranges that end in either half's tile and inside a run of sixteen rows, windows, given and empty ranges, groups, KV splits, row
tiles on both sides of the line in one call, against 64-bit attention."""
import numpy as np
import pytest
import torch

from tests.test_gpu_gqa_prefill_f16 import reference
from zllm_amd import capi, ops

pytestmark = pytest.mark.gpu

D = 256


def run(rows, position, heads, kv_heads, page=16, window=0, softcap=0.0, given=None, workspace=True, q_dtype=torch.bfloat16, spread=1.0, gain=1.0):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rows + 7 * position + heads)
    n = position + rows
    pages = (n + page - 1) // page
    planes = [torch.full((pages * page, kv_heads * D), float("nan"), dtype=torch.float16, device="cuda") for _ in range(2)]  # behind the rows: garbage
    order = torch.randperm(pages, generator=gen, device="cuda").to(torch.int32)
    at = (order.long()[:, None] * page + torch.arange(page, device="cuda")).view(-1)[:n]
    data = [torch.randn(n, kv_heads * D, generator=gen, device="cuda") for _ in range(2)]
    data[0] *= torch.linspace(1.0, gain, n, device="cuda")[:, None]  # rising keys move the softmax reference all the way
    data = [data[0].to(torch.float16), data[1].to(torch.float16)]
    for plane, x in zip(planes, data):
        plane[at] = x
    q = (torch.randn(rows, heads * D, generator=gen, device="cuda") * spread).to(q_dtype)
    r = torch.arange(rows, device="cuda")
    hi = position + r + 1
    lo, kw = torch.clamp(hi - window, min=0) if window else torch.zeros_like(r), {}
    if given == "ends":  # rows read to the end of their block of 50
        hi = torch.minimum((r // 50 + 1) * 50, torch.tensor(rows, device="cuda")) + position
        kw = dict(visible_ends=hi.to(torch.int32))
    elif given == "segments":  # the rows of the third see nothing
        cuts = torch.tensor([0, 3, 64, 131] if rows < 300 else [0, 300, 360, 610, 1250, 1256], device="cuda")
        which = torch.searchsorted(cuts, r, right=True) - 1
        lo, hi = cuts[which], torch.cat([cuts[1:], torch.tensor([rows], device="cuda")])[which]
        hi = torch.where(which == 2, lo, hi)
        kw = dict(visible_starts=lo.to(torch.int32), visible_ends=hi.to(torch.int32))
    out = ops.gqa_prefill_chunk(q, planes[0], None, planes[1], None, order, position, heads, kv_heads, D, page, D**-0.5, window=window, softcap=softcap,
                                kv_format=capi.KV_F16, workspace=workspace, **kw).view(rows, heads, D)
    for head in sorted({0, heads // 2, heads - 1}):
        k, v = (x.view(n, kv_heads, D)[:, head // (heads // kv_heads)] for x in data)
        want = reference(q.view(rows, heads, D)[:, head], k, v, lo, hi, D**-0.5, softcap)
        # probabilities carried as f16 are off by at most 2^-12 of themselves and sum to one: 2^-12 of the largest value, all errors
        # of one sign; f32 scores (|s| < 64 in base 2, the sum of 256 products) move a probability by less than 2^-14
        bound = (2.0**-12 + 2.0**-14) * v.abs().max().item()
        err = (out[:, head].double() - want).abs().max().item()
        assert np.isfinite(err) and err <= bound, f"head {head}: {err:.3e} > {bound:.3e}"


@pytest.mark.parametrize("page", [16, 64, 256, 8, 24])  # the last two keep the tile kernel
def test_pages(page):
    run(150, 300, 16, 8, page)
    run(150, 700, 16, 8, page, workspace=False)


# ranges that end at every edge: a run of sixteen rows, a tile of 32, a pass of two tiles; walks of 576 keys are the shortest in halves
@pytest.mark.parametrize("rows,position", [(64, 511), (64, 512), (64, 513), (65, 527), (65, 528), (79, 529), (64, 544), (97, 543), (575, 0), (576, 0), (700, 3)])
def test_edges_of_halves(rows, position):
    run(rows, position, 4, 2, workspace=False)


@pytest.mark.parametrize("rows,position", [(64, 192), (64, 193), (65, 207), (65, 208), (79, 209), (64, 224), (97, 223), (255, 0), (256, 0), (257, 0), (289, 2),
                                           (63, 300), (64, 191)])
def test_edges(rows, position):
    run(rows, position, 4, 2)


@pytest.mark.parametrize("heads,kv_heads,rows", [(3, 3, 140), (12, 4, 90), (16, 1, 40), (128, 1, 60), (100, 1, 60)])
def test_groups(heads, kv_heads, rows):
    run(rows, 200, heads, kv_heads)
    run(rows, 600, heads, kv_heads, workspace=False)


@pytest.mark.parametrize("window", [200, 256, 300, 511, 512, 1024])  # a row tile of 64 and a window of 512: 575 keys from a tile's first on, in halves
def test_windows(window):
    run(170, 900, 4, 2, window=window)
    run(300, 0, 4, 2, window=window)


@pytest.mark.parametrize("given,position", [("ends", 0), ("ends", 77), ("segments", 0)])
def test_given_ranges(given, position):
    run(260, position, 8, 2, given=given)


# walks on both sides of the line in one launch: segments of 300, 60, none, 640, 6 and 150 rows, their row tiles across them, and ends inside a prefix
@pytest.mark.parametrize("heads,kv_heads", [(8, 2), (16, 16), (6, 3)])
@pytest.mark.parametrize("given,position,workspace", [("segments", 0, True), ("segments", 0, False), ("segments", 37, True), ("segments", 1100, False), ("ends", 0, False), ("ends", 530, False), ("ends", 530, True)])
def test_given_ranges_of_both_lengths(heads, kv_heads, given, position, workspace):
    run(1406, position, heads, kv_heads, given=given, workspace=workspace)


@pytest.mark.parametrize("workspace", [True, False])
def test_splits(workspace):  # parts of a length that is no multiple of a pass
    run(70, 5003, 4, 1, workspace=workspace)


@pytest.mark.parametrize("softcap,spread,gain,q_dtype", [(50.0, 1.0, 1.0, torch.float16), (5.0, 4.0, 1.0, torch.bfloat16), (300.0, 1.0, 1.0, torch.bfloat16),
                                                         (0.0, 4.0, 8.0, torch.float16), (0.0, 0.05, 1.0, torch.bfloat16)])
def test_scores(softcap, spread, gain, q_dtype):
    run(200, 400, 8, 4, softcap=softcap, spread=spread, gain=gain, q_dtype=q_dtype, workspace=False)
    run(200, 1500, 8, 4, softcap=softcap, spread=spread, gain=gain, q_dtype=q_dtype)
