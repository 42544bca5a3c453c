"""The chunk kernel over f16 rows of head_dim 128 that takes launches of more than 512 tiles of 128 (row, head) pairs
(gqa_prefill_f16.hip): pages it addresses by scalars and others, groups that do and do not divide a tile, ranges that end inside
a load's four rows, empty ranges, KV splits, output gate and types, against 64-bit attention on a few heads."""
import numpy as np
import pytest
import torch

from zllm_amd import capi, ops

pytestmark = pytest.mark.gpu

D = 128


def reference(q, k, v, lo, hi, scale, softcap):
    """One head in 64 bits: q [rows, D], k / v [tokens, D], visible tokens [lo, hi) of each row."""
    s = (q.double() @ k.double().T.contiguous()) * scale
    if softcap:
        s = torch.tanh(s / softcap) * softcap
    t = torch.arange(k.shape[0], device=q.device)[None]
    s = s.masked_fill(~((t >= lo[:, None]) & (t < hi[:, None])), float("-inf"))
    top = s.amax(dim=1, keepdim=True)
    p = torch.exp(s - torch.where(top == float("-inf"), torch.zeros_like(top), top))
    total = p.sum(dim=1, keepdim=True)
    return torch.where(total > 0, (p @ v.double()) / total, torch.zeros_like(q, dtype=torch.float64))


def run(rows, position, heads, kv_heads, page, mode="causal", softcap=0.0, table=True, out_dtype=torch.float32, gate=False, workspace=True,
        q_dtype=torch.bfloat16, spread=1.0):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rows + 7 * position + heads)
    n = position + rows
    pages = (n + page - 1) // page
    cols = kv_heads * D
    planes = [torch.full((pages * page, cols), float("nan"), dtype=torch.float16, device="cuda") for _ in range(2)]  # behind the rows: garbage
    order = torch.randperm(pages, generator=gen, device="cuda").to(torch.int32) if table else torch.arange(pages, dtype=torch.int32, device="cuda")
    at = (order.long()[:, None] * page + torch.arange(page, device="cuda")).view(-1)[:n]
    data = [torch.randn(n, cols, generator=gen, device="cuda").to(torch.float16) * f for f in (spread, 1.0)]
    for plane, x in zip(planes, data):
        plane[at] = x
    q = torch.randn(rows, heads * D, generator=gen, device="cuda").to(q_dtype)
    r = torch.arange(rows, device="cuda")
    lo, hi, given = torch.zeros_like(r), position + r + 1, {}
    if mode == "ends":  # rows read to the end of their block of 50
        hi = torch.minimum((r // 50 + 1) * 50, torch.tensor(rows, device="cuda")) + position
        given = dict(visible_ends=hi.to(torch.int32))
    elif mode == "segments":  # unequal ones, the rows of every fifth see nothing
        cuts = torch.tensor([0, 3, 130, 131, 400, 401, 700, 995], device="cuda")
        which = torch.searchsorted(cuts, r, right=True) - 1
        ends = torch.cat([cuts[1:], torch.tensor([rows], device="cuda")])
        lo, hi = cuts[which], ends[which]
        hi = torch.where(which % 5 == 4, lo, hi)
        given = dict(visible_starts=lo.to(torch.int32), visible_ends=hi.to(torch.int32))
    g = torch.randn(rows, heads * D, generator=gen, device="cuda") if gate else None
    scale = D**-0.5
    out = ops.gqa_prefill_chunk(q, planes[0], None, planes[1], None, order if table else None, position, heads, kv_heads, D, page, scale, softcap=softcap,
                                kv_format=capi.KV_F16, out_dtype=out_dtype, gate=g, workspace=workspace, **given)
    out = out.view(rows, heads, D)
    for head in (0, heads // 2, heads - 1):
        kvh = head // (heads // kv_heads)
        k, v = (x.view(n, kv_heads, D)[:, kvh] for x in data)
        want = reference(q.view(rows, heads, D)[:, head], k, v, lo, hi, scale, softcap)
        if gate:
            want = want * torch.sigmoid(g.view(rows, heads, D)[:, head].double())
        # probabilities carried as f16 are off by at most 2^-12 of themselves and sum to one: 2^-12 of the largest value, all errors
        # of one sign; f32 scores (|s| < 64 in base 2, the sum of 128 products) move a probability by less than 2^-14
        bound = (2.0**-12 + 2.0**-14) * v.abs().max().item()
        if out_dtype != torch.float32:
            bound += want.abs().max().item() * (2.0**-8 if out_dtype == torch.bfloat16 else 2.0**-11)
        err = (out[:, head].double() - want).abs().max().item()
        assert np.isfinite(err) and err <= bound, f"head {head}: {err:.3e} > {bound:.3e}"


# 64 KV heads: nine tiles of 128 rows each, 576 in all.  Pages of 8 and more are addressed by scalars
@pytest.mark.parametrize("page", [8, 16, 64, 1024, 4, 1, 24])
def test_pages(page):
    run(1030, 0, 64, 64, page)


@pytest.mark.parametrize("rows", [1025, 1027, 1055, 1056, 1057])  # the last tile of keys ends inside a load's four rows
def test_row_remainders(rows):
    run(rows, 0, 64, 64, 16)


@pytest.mark.parametrize("heads,kv_heads,rows", [(24, 8, 2800), (72, 72, 900), (63, 9, 1100), (600, 600, 40)])
def test_groups(heads, kv_heads, rows):
    run(rows, 0, heads, kv_heads, 16)


@pytest.mark.parametrize("mode", ["ends", "segments"])
@pytest.mark.parametrize("page,table", [(16, True), (24, True), (16, False)])
def test_given_ranges(mode, page, table):
    run(1030, 0, 64, 64, page, mode=mode, table=table)


@pytest.mark.parametrize("workspace", [True, False])
@pytest.mark.parametrize("position", [37, 300, 2051])
def test_behind_a_prefix(position, workspace):
    run(1030, position, 64, 64, 16, workspace=workspace)


@pytest.mark.parametrize("softcap", [5.0, 50.0, 300.0])
def test_soft_caps(softcap):
    run(1030, 0, 64, 64, 16, softcap=softcap)


@pytest.mark.parametrize("out_dtype,gate,q_dtype,spread", [(torch.bfloat16, True, torch.float16, 1.0), (torch.float16, False, torch.bfloat16, 1.0),
                                                           (torch.float32, True, torch.bfloat16, 4.0)])
def test_outputs_and_queries(out_dtype, gate, q_dtype, spread):
    run(1030, 0, 64, 64, 16, out_dtype=out_dtype, gate=gate, q_dtype=q_dtype, spread=spread)


@pytest.mark.parametrize("spread", [0.02, 0.2, 1.0])
def test_short_ranges_carry_both_terms(spread):
    """Segments of up to 400 keys, scores from near-even to ordinary: every step weighs more than a sixteenth of its row, so all
    probabilities have 22 bits."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(7)
    rows, heads = 3000, 32
    lens = torch.tensor([400, 390, 310, 400, 200, 400, 100, 400, 400], device="cuda")
    ends = torch.cumsum(lens, 0)
    start, end = torch.repeat_interleave(ends - lens, lens), torch.repeat_interleave(ends, lens)
    q = (torch.randn(rows, heads * D, generator=gen, device="cuda") * spread).to(torch.bfloat16)
    k, v = (torch.randn((rows + 63) // 64 * 64, heads * D, generator=gen, device="cuda").to(torch.float16) for _ in range(2))
    table = torch.arange(len(k) // 64, dtype=torch.int32, device="cuda")
    out = ops.gqa_prefill_chunk(q, k, None, v, None, table, 0, heads, heads, D, 64, D**-0.5, kv_format=capi.KV_F16, visible_starts=start.to(torch.int32),
                                visible_ends=end.to(torch.int32)).view(rows, heads, D)
    for head in (0, heads - 1):
        want = reference(q.view(rows, heads, D)[:, head], k.view(-1, heads, D)[:rows, head], v.view(-1, heads, D)[:rows, head], start, end, D**-0.5, 0.0)
        # f32 sums of 400 products in numerator and denominator, 2^-24 sqrt(400) each, and scores of 128 products, 2^-24 sqrt(128) of |s| < 8
        err = ((out[:, head].double() - want).norm() / want.norm()).item()
        assert err <= 5e-6, f"head {head}: {err:.2e}"


def workspace_bytes(rows, position, heads, kv_heads, page=16, **given):
    q = torch.empty(rows, heads * D, dtype=torch.bfloat16, device="cuda")
    table = torch.zeros((position + rows + page - 1) // page, dtype=torch.int32, device="cuda")
    args, _, _ = ops.gqa_prefill_chunk_args(q, None, None, None, None, table, position, heads, kv_heads, D, page, 0.1, kv_format=capi.KV_F16, workspace=False,
                                            **given)
    return capi.load().zllm_attn_gqa_prefill_workspace_bytes(args)


@pytest.mark.parametrize("gate", [None, "rows", "columns"])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_outputs_and_gates_of_the_kernel_itself(out_dtype, gate):
    """Packed segments run unsplit: the kernel's own epilogue gates and converts, where split calls leave both to the merge."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(11)
    rows, heads = 1100, 64
    r = torch.arange(rows, device="cuda")
    start, end = r // 220 * 220, r // 220 * 220 + 220
    given = dict(visible_starts=start.to(torch.int32), visible_ends=end.to(torch.int32))
    assert workspace_bytes(rows, 0, heads, heads, **given) == 0
    q = torch.randn(rows, heads * D, generator=gen, device="cuda").to(torch.bfloat16)
    k, v = (torch.randn((rows + 15) // 16 * 16, heads * D, generator=gen, device="cuda").to(torch.float16) for _ in range(2))
    table = torch.arange(len(k) // 16, dtype=torch.int32, device="cuda")
    g = None if gate is None else torch.randn(rows, 1 if gate == "rows" else heads * D, generator=gen, device="cuda").to(torch.bfloat16)
    out = ops.gqa_prefill_chunk(q, k, None, v, None, table, 0, heads, heads, D, 16, D**-0.5, kv_format=capi.KV_F16, out_dtype=out_dtype, gate=g,
                                **given).view(rows, heads, D)
    for head in (0, 31, heads - 1):
        want = reference(q.view(rows, heads, D)[:, head], k.view(-1, heads, D)[:rows, head], v.view(-1, heads, D)[:rows, head], start, end, D**-0.5, 0.0)
        if gate == "rows":
            want = want * torch.sigmoid(g.double())
        elif gate == "columns":
            want = want * torch.sigmoid(g.view(rows, heads, D)[:, head].double())
        # all probabilities carry two terms (220 keys): f32 sums of 220 products and f32 scores, then one rounding of the output type
        bound = 1e-5 * v.abs().max().item() + want.abs() * {torch.float32: 0.0, torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}[out_dtype]
        if out_dtype == torch.float16:
            bound = bound + 2.0**-25  # subnormal halves
        assert ((out[:, head].double() - want).abs() <= bound).all(), f"head {head}"


@pytest.mark.parametrize("position", [1, 200, 2051])
def test_given_ranges_behind_a_prefix(position):
    """Rows that see the prefix and their own segment, others only part of either, in no order."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(position)
    rows, heads = 1030, 64
    n = position + rows
    r = torch.arange(rows, device="cuda")
    lo = torch.where(r % 3 == 0, 0, torch.where(r % 3 == 1, position // 2, position + r // 2))
    hi = torch.where(r % 5 == 0, position + rows, torch.minimum(position + (r // 100 + 1) * 100, torch.tensor(n, device="cuda")))
    hi = torch.where(r % 97 == 5, lo, torch.maximum(lo, hi))  # some see nothing
    pages = (n + 15) // 16
    table = torch.randperm(pages, generator=gen, device="cuda").to(torch.int32)
    at = (table.long()[:, None] * 16 + torch.arange(16, device="cuda")).view(-1)[:n]
    planes = [torch.full((pages * 16, heads * D), float("nan"), dtype=torch.float16, device="cuda") for _ in range(2)]
    data = [torch.randn(n, heads * D, generator=gen, device="cuda").to(torch.float16) for _ in range(2)]
    for plane, x in zip(planes, data):
        plane[at] = x
    q = torch.randn(rows, heads * D, generator=gen, device="cuda").to(torch.bfloat16)
    for workspace in (True, False):
        out = ops.gqa_prefill_chunk(q, planes[0], None, planes[1], None, table, position, heads, heads, D, 16, D**-0.5, kv_format=capi.KV_F16,
                                    visible_starts=lo.to(torch.int32), visible_ends=hi.to(torch.int32), workspace=workspace).view(rows, heads, D)
        for head in (0, 40, heads - 1):
            k, v = (x.view(n, heads, D)[:, head] for x in data)
            want = reference(q.view(rows, heads, D)[:, head], k, v, lo, hi, D**-0.5, 0.0)
            err = (out[:, head].double() - want).abs().max().item()
            bound = (2.0**-12 + 2.0**-14) * v.abs().max().item()  # as in run()
            assert np.isfinite(err) and err <= bound, f"head {head}: {err:.3e} > {bound:.3e}"


# (rows, position) on both sides of each line of the dispatch, 64 heads: full-size tiles hold 256 rows, the smaller ones 128
@pytest.mark.parametrize("rows,position,given", [
    (1024, 0, False), (1025, 0, False),        # 512 and 576 tiles of 128
    (4096, 0, True), (4097, 0, True),          # four whole rounds of full-size tiles, and a row
    (1400, 300, False), (1800, 300, False),    # 384 and 512 full-size tiles behind fewer keys than rows
    (1536, 1537, False), (1537, 1538, False),  # the last of two rounds half full, and a row
    (1100, 16384, False), (1100, 16385, False),
    (2048, 512, True), (2048, 513, True),      # given ranges behind a quarter of the rows
])
def test_both_sides_of_the_dispatch_lines(rows, position, given):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rows)
    heads, n = 64, position + rows
    pages = (n + 63) // 64
    table = torch.randperm(pages, generator=gen, device="cuda").to(torch.int32)
    at = (table.long()[:, None] * 64 + torch.arange(64, device="cuda")).view(-1)[:n]
    planes = [torch.randn(pages * 64, heads * D, generator=gen, device="cuda").to(torch.float16) for _ in range(2)]
    q = torch.randn(rows, heads * D, generator=gen, device="cuda").to(torch.bfloat16)
    r = torch.arange(rows, device="cuda")
    lo, hi, ranges = torch.zeros_like(r), position + r + 1, {}
    if given:
        lo, hi = torch.where(r < rows // 3, 0, position + rows // 3), torch.where(r < rows // 3, position + rows // 3, n)
        ranges = dict(visible_starts=lo.to(torch.int32), visible_ends=hi.to(torch.int32))
    out = ops.gqa_prefill_chunk(q, planes[0], None, planes[1], None, table, position, heads, heads, D, 64, D**-0.5, kv_format=capi.KV_F16, **ranges)
    few = torch.cat([r[:40], r[rows // 3 - 20:rows // 3 + 20], r[-40:]])  # the edges of the rows
    for head in (0, 33, heads - 1):
        k, v = (plane[at, head * D:(head + 1) * D] for plane in planes)
        want = reference(q.view(rows, heads, D)[few, head], k, v, lo[few], hi[few], D**-0.5, 0.0)
        err = (out.view(rows, heads, D)[few, head].double() - want).abs().max().item()
        bound = (2.0**-12 + 2.0**-14) * v.abs().max().item()  # as in run()
        assert np.isfinite(err) and err <= bound, f"head {head}: {err:.3e} > {bound:.3e}"
