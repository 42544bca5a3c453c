"""Chunks over Q8g64 rows that are converted once a call (gqa_prefill_staged.hip), taken with the workspace that
zllm_attn_gqa_prefill_preferred_bytes names: against the CPU oracle, and against the same call without a workspace."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from tests.test_gpu_gqa_prefill import run_case

torch = pytest.importorskip("torch")


def staged_bytes(rows, position, heads, kv_heads, **fields):
    """What the call asks for beyond the workspace it needs (256 compute units where no device says otherwise)."""
    from zllm_amd import capi

    lib = capi.load()
    pre = capi.GqaPrefillArgs(rows=rows, position=position, num_heads=heads, num_kv_heads=kv_heads, head_dim=128, block_tokens=16, score_scale=0.1,
                              kv_format=capi.KV_Q8G64, scale_dtype=capi.SCALE_F16, q_dtype=capi.DTYPE_BF16, out_dtype=capi.DTYPE_F32)
    for name, value in fields.items():
        setattr(pre, name, value)
    return lib.zllm_attn_gqa_prefill_preferred_bytes(C.byref(pre)) - lib.zllm_attn_gqa_prefill_workspace_bytes(C.byref(pre))


def test_which_calls_ask_for_staged_rows():
    from zllm_amd import capi

    tile = 2 * 32 * 128 * 2 + 512  # f16 rows of a tile, and its scales
    assert 0 < staged_bytes(2048, 50000, 32, 8) - 8 * 1627 * tile < 8 * 1627 * 256 + 9 * tile
    assert staged_bytes(192, 5000, 32, 8) == 0 < staged_bytes(193, 5000, 32, 8)            # three and four row tiles a KV head
    assert staged_bytes(65, 959, 32, 8) > 0 and staged_bytes(65, 960, 32, 8) == 0          # few tiles: up to 1,024 keys
    assert 0 < staged_bytes(400, 50000, 32, 8, window=600) < 8 * 33 * (tile + 256) + 9 * tile  # only what a window leaves
    assert staged_bytes(512, 240000, 32, 8) > 0 and staged_bytes(512, 260000, 32, 8) == 0  # at most 1 GiB
    for scales in (capi.SCALE_F32, capi.SCALE_F16):  # few tiles: half of one has to be filled, whatever the scales
        assert staged_bytes(31, 100, 32, 8, scale_dtype=scales) == 0 == staged_bytes(127, 500, 16, 16, scale_dtype=scales)
        assert staged_bytes(33, 100, 32, 8, scale_dtype=scales) > 0 == staged_bytes(24, 8, 64, 8, scale_dtype=scales)
    for other in (dict(q_dtype=capi.DTYPE_F32), dict(kv_format=capi.KV_F16), dict(head_dim=64), dict(head_dim=256)):
        assert staged_bytes(2048, 50000, 32, 8, **other) == 0
    ends = (C.c_uint32 * 1)()
    assert staged_bytes(2048, 50000, 32, 8, visible_ends=C.addressof(ends)) == 0
    # a first chunk: half-size row tiles, more than one a compute unit
    assert staged_bytes(1024, 0, 32, 8) == 0 < staged_bytes(1025, 0, 32, 8)
    assert staged_bytes(16, 500, 32, 8) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("prefix,chunk,hq,hkv,kw", [
    (300, 257, 4, 1, {}),                                            # five row tiles, a last tile of 13 tokens, an odd number of them
    (1500, 97, 8, 1, dict(block_tokens=24)),                         # four row tiles, one row in the last; pages of no power of two
    (31, 33, 64, 1, dict(block_tokens=1)),                           # two tiles of 32 tokens, both at an edge of every row
    (950, 65, 6, 2, dict(gate_cols=6 * 128)),                        # groups of three heads leave a column of the tile free
    (700, 130, 16, 2, dict(window=200, gate_cols=1)),                # the first staged tile is not the first of the sequence
    (900, 300, 8, 2, dict(window=5)),                                # ranges of one and two tiles
    (1200, 260, 8, 2, dict(softcap=30.0, rule=O.RULE_ROCM_MLA)),
    (800, 140, 8, 2, dict(softcap=400.0, rule=O.RULE_CUDA_GQA)),     # the precise form of the soft cap; f32 scales
    (2500, 200, 8, 2, dict(rule=O.RULE_ROCM_MLA, block_tokens=64, v_gain=2.0 ** np.repeat(np.arange(-10, 10), 135))),  # the V window moves on
    (2500, 200, 8, 2, dict(rule=O.RULE_ROCM_MLA, block_tokens=64, v_gain=2.0 ** np.repeat(np.arange(20, 0, -1), 135))),  # and scales that fall behind it
    (400, 40, 130, 1, {}),                                           # one row a tile
    # half-size tiles, the keys in two halves: first chunks
    (0, 1031, 32, 8, dict(block_tokens=24)),                         # 33 tiles of keys: the odd half ends a pass earlier; a last tile of seven rows
    (0, 1000, 33, 11, {}),                                           # the fewest keys; row tiles that see one tile, or the even half's only
    (7, 1100, 56, 8, dict(softcap=30.0, rule=O.RULE_ROCM_MLA, gate_cols=1)),
    (0, 1200, 32, 8, dict(rule=O.RULE_ROCM_MLA, block_tokens=64, v_gain=2.0 ** np.repeat(np.arange(-10, 10), 60)))])  # the halves' windows differ
def test_staged_rows_against_the_oracle(prefix, chunk, hq, hkv, kw):
    named = {"rule": "scale_dtype", "block_tokens": "block_tokens", "window": "window"}
    fields = {named[n]: v for n, v in kw.items() if n in named}
    if "scale_dtype" in fields:
        from zllm_amd import capi

        fields["scale_dtype"] = {O.RULE_ROCM_MLA: capi.SCALE_BF16, O.RULE_CUDA_GQA: capi.SCALE_F32}[fields["scale_dtype"]]
    assert staged_bytes(chunk, prefix, hq, hkv, **fields) > 0, "this shape is meant to be staged"
    outs = []
    for workspace in (True, False):
        out, want = run_case(200 + chunk, prefix, chunk, hq, hkv, workspace=workspace, outliers="v_gain" not in kw, **kw)
        got = out.float().cpu().numpy()
        assert np.abs(got - want).max() <= 2e-3 * max(1.0, float(np.abs(want).max())), (workspace, np.abs(got - want).max())
        outs.append(got)
    # the two kernels round the same products to f16 (2^-12 a term below a sixteenth of the row, both terms above)
    assert np.linalg.norm(outs[0] - outs[1]) <= 2.0 ** -11 * np.linalg.norm(outs[1])


@pytest.mark.gpu
@pytest.mark.parametrize("rows,prefix,tile_rows", [(290, 300, 64), (1100, 7, 32)])  # a row tile of 256 pairs; of 128, the keys in two halves
@pytest.mark.parametrize("k_bits,v_bits", [(0x7E00, 0x7C00), (0x0001, 0x7BFF)])  # a NaN and an infinity; the smallest and the largest scale
def test_row_tiles_are_independent_of_later_tokens(rows, prefix, tile_rows, k_bits, v_bits):
    """A token in the 32-token tile in which a row tile ends, but behind its rows: they come out bit for bit as with an ordinary one there."""
    from zllm_amd import capi, ops

    gen = torch.Generator(device="cuda")
    gen.manual_seed(9)
    total, page = prefix + rows, 16
    table = torch.randperm((total + page - 1) // page, generator=gen, device="cuda").to(torch.int32)
    planes = [torch.zeros(table.numel() * page, n, dtype=t, device="cuda") for n, t in ((1024, torch.int8), (16, torch.int16)) * 2]
    for n in (0, 2):
        ops.q8g64_append(torch.randn(total, 1024, generator=gen, device="cuda", dtype=torch.bfloat16), planes[n], planes[n + 1], table, 0, page,
                         capi.QUANT_METAL_GQA)
    q = torch.randn(rows, 32 * 128, generator=gen, device="cuda", dtype=torch.bfloat16)
    assert staged_bytes(rows, prefix, 32, 8) > 0

    def call():
        return ops.gqa_prefill_chunk(q, *planes, table, prefix, 32, 8, 128, page, 128 ** -0.5)

    clean = call()
    seen = 3 * tile_rows  # rows of the first three tiles
    token = (prefix + seen) | 31  # the last of the 32 tokens in which they end
    assert (prefix + seen) % 32 and token < total
    at = int(table[token // page]) * page + token % page
    planes[1][at], planes[3][at] = k_bits, v_bits
    got = call()
    assert torch.equal(got[:seen], clean[:seen])
    assert not torch.equal(got[seen:], clean[seen:])


@pytest.mark.gpu
def test_staged_rows_in_a_graph():
    """Staging and attention recorded together, replayed over caches that change in between."""
    from zllm_amd import capi, ops

    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    rows, prefix, page = 160, 700, 16
    total = prefix + rows
    table = torch.randperm((total + page - 1) // page + 3, generator=gen, device="cuda")[: (total + page - 1) // page].to(torch.int32)
    pool = ((total + page - 1) // page + 3) * page
    planes = [torch.zeros(pool, n, dtype=t, device="cuda") for n, t in ((256, torch.int8), (4, torch.int16)) * 2]
    q = torch.randn(rows, 16 * 128, generator=gen, device="cuda", dtype=torch.bfloat16)
    args, out, scratch = ops.gqa_prefill_chunk_args(q, *planes, table, prefix, 16, 2, 128, page, 128 ** -0.5)
    lib = capi.load()

    def fill():
        for n in (0, 2):
            x = torch.randn(total, 256, generator=gen, device="cuda", dtype=torch.bfloat16)
            ops.q8g64_append(x, planes[n], planes[n + 1], table, 0, page, capi.QUANT_METAL_GQA)

    def call():
        capi.check(lib.zllm_attn_gqa_prefill_chunk(C.byref(args), ops._stream()))

    fill()
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for _ in range(3):
        fill()
        call()
        eager = out.clone()
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager) and float(out.abs().max()) > 0
