"""Chunked MLA prefill over latents that are converted once a call (mla_staged.hip), taken with the workspace that
zllm_attn_mla_decode_preferred_bytes names: against the CPU oracle, and against the same call with no room for it."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from tests.cases import assert_attention_close, to_torch_bf16, upload
from tests.test_gpu_mla_decode import make_mla_chunk_case, oracle_mla_chunk, weight_args

torch = pytest.importorskip("torch")


def chunk_args(heads, rows, longest, batch=1, **fields):
    from zllm_amd import capi

    args = capi.MlaDecodeArgs(batch=batch, heads=heads, q_head_dim=192, kv_head_dim=256, latent_dim=512, rope_dim=64, block_tokens=64,
                              max_ctx_len=longest, table_stride=0, q_dtype=capi.DTYPE_BF16, out_dtype=capi.DTYPE_F32, query_rows=rows)
    for name, value in fields.items():
        setattr(args, name, value)
    return args


def staged_bytes(*a, **kw):
    """What the call asks for beyond the workspace it needs (256 compute units where no device says otherwise)."""
    from zllm_amd import capi

    args = chunk_args(*a, **kw)
    return capi.load().zllm_attn_mla_decode_preferred_bytes(C.byref(args)) - capi.load().zllm_attn_mla_decode_workspace_bytes(C.byref(args))


def test_which_calls_ask_for_staged_latents():
    from zllm_amd import capi

    tile = 39 * 1024 + 128
    assert staged_bytes(128, 512, 16896) >= (16896 // 32) * tile
    assert staged_bytes(128, 512, 16896, stage_mask=15) > 0
    assert staged_bytes(128, 20, 10020) == 0 == staged_bytes(64, 16, 30016) == staged_bytes(16, 32, 8032) == staged_bytes(128, 1, 60000)
    for stages in (1, 2, 14, capi.MLA_WIDE_TILES):
        assert staged_bytes(128, 512, 16896, stage_mask=stages) == 0  # records for the caller, or another kernel asked for
    ids = (C.c_uint32 * 1)()
    assert staged_bytes(128, 512, 16896, selection=C.addressof(ids), top_k=2048) == 0
    assert staged_bytes(16, 1000, 850000) > 0 and staged_bytes(16, 1000, 870000) == 0  # at most 1 GiB


def test_the_preferred_workspace_is_at_most_a_gigabyte_more():
    """Tiles and records together, over shapes drawn up to where the bound bites; the four are some that went beyond it."""
    rng = np.random.default_rng(7)
    shapes = [(8, 208, 213548, 4), (4, 2093, 844747, 1), (128, 23, 835389, 1), (16, 1000, 850000, 1)]
    for _ in range(4000):
        batch = int(np.exp(rng.uniform(0, np.log(32))))
        rows = min(int(np.exp(rng.uniform(np.log(2), np.log(8000)))), 65535 // batch)
        shapes.append((int(rng.choice([1, 4, 8, 16, 32, 64, 128, 200])), rows, int(np.exp(rng.uniform(np.log(500), np.log(1e6)))), batch))
    more = np.array([staged_bytes(*shape) for shape in shapes])
    assert more.max() <= 1 << 30 and np.count_nonzero(more > 900 << 20) > 10


def test_few_rows_over_many_tokens_are_not_staged():
    """Converting a token costs about as much as attending to it with four rows of 16 heads: speculated tokens and short chunks stay out, alone
    and in batches, and so do ragged batches whose records follow the tokens there are."""
    assert staged_bytes(16, 4, 64000, 8) == staged_bytes(16, 3, 48000, 16) == staged_bytes(16, 4, 300000) == staged_bytes(32, 8, 64000, 8) == 0
    assert staged_bytes(16, 16, 64000, 8) > 0 < staged_bytes(16, 16, 300000)
    ragged = dict(total_ctx_tokens=101500)
    assert staged_bytes(16, 8, 100000, 4, **ragged) == staged_bytes(64, 4, 100000, 4, **ragged) == 0 < staged_bytes(16, 32, 100000, 4, **ragged)


@pytest.mark.parametrize("heads,rows,length", [(128, 300, 1400), (128, 850, 1150), (32, 700, 1500)])
def test_splits_have_to_save_more_than_their_records_cost(heads, rows, length):
    """Some more than one round of workgroups with two splits' worth of keys: unsplit."""
    args = chunk_args(heads, rows, length)
    assert staged_bytes(heads, rows, length) > 0
    from zllm_amd import capi

    args.workspace_bytes = capi.load().zllm_attn_mla_decode_preferred_bytes(C.byref(args))
    layout = capi.SplitRecordLayout()
    capi.check(capi.load().zllm_attn_mla_decode_record_layout(C.byref(args), C.byref(layout)))
    assert layout.max_chunks == 1 and layout.record_rows == rows


def record_layout(args):
    from zllm_amd import capi

    layout = capi.SplitRecordLayout()
    capi.check(capi.load().zllm_attn_mla_decode_record_layout(C.byref(args), C.byref(layout)))
    return [getattr(layout, name) for name, _ in layout._fields_]


def test_the_workspace_size_names_the_plan_of_every_stage():
    """Records lie under one plan for all stage masks and for the layout; only the preferred size itself asks for that of the converted latents."""
    from zllm_amd import capi

    args = chunk_args(16, 1000, 3000)
    lib = capi.load()
    least, preferred = lib.zllm_attn_mla_decode_workspace_bytes(C.byref(args)), lib.zllm_attn_mla_decode_preferred_bytes(C.byref(args))
    plain = record_layout(args)
    args.workspace_bytes = preferred
    staged = record_layout(args)
    assert staged != plain
    for stages in (0, 1, 2, 3, 8, 12, 15, 2 | capi.MLA_WIDE_TILES):
        args.stage_mask = stages
        for size, want in ((preferred, staged), (0, plain), (least, plain), (preferred - 1, plain), (preferred + 1, plain), (1 << 40, plain)):
            args.workspace_bytes = size
            assert record_layout(args) == want, (stages, size)


def run_chunk(case, room, out_dtype=None, hint=False):
    """The call with the preferred workspace, or with the least; max_ctx_len is the longest context, `hint` states the tokens there are."""
    from zllm_amd import capi, ops

    weights, form = weight_args(case)
    rows, heads, batch = case["rows"], case["heads"], len(case["lens"])
    args = chunk_args(heads, rows, int(case["lens"].max()), batch, block_tokens=case["block_tokens"],
                      total_ctx_tokens=int(case["lens"].sum()) if hint else 0)
    lib = capi.load()
    need = (lib.zllm_attn_mla_decode_preferred_bytes if room else lib.zllm_attn_mla_decode_workspace_bytes)(C.byref(args))
    assert not room or need > lib.zllm_attn_mla_decode_workspace_bytes(C.byref(args)), "this shape is meant to be staged"
    workspace = torch.full((need + 4096,), 0x7F, dtype=torch.uint8, device="cuda")
    out = ops.mla_decode(to_torch_bf16(case["q_bits"], "cuda"), weights, upload(case["codes"]), upload(case["scales"]), upload(case["rope"]),
                         upload(case["tables"]), upload(case["lens"]), heads, 192, 256, 512, 64, case["block_tokens"], int(case["lens"].max()),
                         out_dtype=out_dtype or torch.float32, query_rows=rows, workspace=workspace[:need], total_ctx_tokens=args.total_ctx_tokens, **form)
    torch.cuda.synchronize()
    assert int(workspace[need:].min()) == int(workspace[need:].max()) == 0x7F, "written past the workspace"
    return out.float().cpu().numpy()


@pytest.mark.gpu
@pytest.mark.parametrize("heads,lens,rows,kw", [
    (1, [1500], 1000, {}),                                             # 128 rows a tile, a last tile of 104
    (4, [3001], 101, dict(block_tokens=24)),                           # four row tiles, the last with five rows; pages of no power of two
    (5, [1031, 700], 257, dict(block_tokens=1)),                       # two sequences; 25 rows a tile leave three pairs free
    (16, [1400], 300, dict(w_std=0.2)),                                # a last tile of four rows; scores of a large spread
    (8, [900], 900, {}),                                               # a first chunk: the first row sees one token
    (40, [2200], 180, dict(poison=True)),                              # three rows a tile, the last wave part empty; rows past the end hold NaN
    (250, [1999], 102, {}),                                            # one row a tile, two blocks of heads, the second three short
    (8, [1800], 200, dict(latent_gain=2.0 ** np.repeat(np.arange(-9, 9), 100)))])  # the value window moves on, references too
def test_staged_latents_against_the_oracle(heads, lens, rows, kw):
    case = make_mla_chunk_case(heads + rows, lens, rows, heads, **kw)
    want, _ = oracle_mla_chunk(case)
    outs = [run_chunk(case, room) for room in (True, False)]
    for got in outs:
        scale = max(1.0, float(np.abs(want).max()))
        assert_attention_close(got / scale, want / scale, f"heads={heads} lens={lens} rows={rows}")
    # the two kernels round the same probabilities and products to f16 (2^-12 a term, independent over the tokens)
    assert np.linalg.norm(outs[0] - outs[1]) <= 2.0 ** -11 * np.linalg.norm(outs[1])


def rope_score_chunk(heads, rows, length, first_gain, spread):
    """A chunk whose scores come from the rope columns alone, its first 64 latents `first_gain` above the others and seen with a weight of some
    e^-40; and its attention in 64 bits, before the projection by the value rows, which pick columns 4 v of the latents.  The case's context is `length`."""
    case = make_mla_chunk_case(11, [length], rows, heads, block_tokens=64, latent_gain=np.where(np.arange(length) < 64, first_gain, 1.0))
    rng = np.random.default_rng(5)
    direction = rng.standard_normal(64)
    q = rng.standard_normal((rows, heads, 192)) * 0.5
    q[..., 128:] = (q[..., 128:] + direction) * spread * np.sqrt(192.0) / np.sqrt(64 * 1.25)  # scores of deviation `spread`
    kv_b = np.zeros((heads, 256, 512), dtype=np.float32)
    kv_b[:, 128 + np.arange(128), 4 * np.arange(128)] = 1.0
    k_rope = rng.standard_normal((length, 64)) - np.where(np.arange(length) < 64, 6.0 / spread, 0.0)[:, None] * direction
    case["q_bits"], case["kv_b_bits"] = O.f32_to_bf16(q.reshape(rows, -1).astype(np.float32)), O.f32_to_bf16(kv_b.reshape(-1, 512))
    pages = case["tables"][0].astype(np.int64)
    at = (pages[:, None] * 64 + np.arange(64)).reshape(-1)[:length]
    case["rope"][at] = O.f32_to_bf16(k_rope.astype(np.float32))
    latents = case["codes"][at].astype(np.float64) * np.repeat(O.bf16_to_f32(case["scales"][at]).astype(np.float64), 64, axis=1)
    q64 = O.bf16_to_f32(case["q_bits"]).astype(np.float64).reshape(rows, heads, 192)[..., 128:]
    scores = q64 @ O.bf16_to_f32(case["rope"][at]).astype(np.float64).T / np.sqrt(192.0)
    scores = np.where(np.arange(length) < length - rows + 1 + np.arange(rows)[:, None, None], scores, -np.inf)
    p = np.exp(scores - scores.max(axis=2, keepdims=True))
    return case, (p / p.sum(axis=2, keepdims=True)) @ latents[:, ::4]


@pytest.mark.gpu
@pytest.mark.parametrize("lens", [[2600, 901, 700], [1400, 300, 301]])
def test_ragged_batches_with_the_token_count(lens):
    """Sequences of unequal lengths whose sum is stated, one of them no longer than its chunk: each split of each sequence where the merges
    look for it, and the workgroups behind a short one's end write that they have seen nothing."""
    case = make_mla_chunk_case(21, lens, 300, 16, block_tokens=64)
    want, _ = oracle_mla_chunk(case)
    scale = max(1.0, float(np.abs(want).max()))
    for hint in (True, False):
        assert_attention_close(run_chunk(case, True, hint=hint) / scale, want / scale, f"lens={lens} hint={hint}")


@pytest.mark.gpu
@pytest.mark.parametrize("spread", [0.5, 2.0])
@pytest.mark.parametrize("gain", [8, 14, 17, 20, 24])
def test_scales_that_fall_keep_their_bits(gain, spread):
    """Latents 2^gain below those before them, which hold the exponent window of the values: the staged call is as far from 64 bits as the
    call that converts them for every row (f16 weights and products whose factors are rounded alike, in another order)."""
    case, want = rope_score_chunk(8, 300, 2000, 2.0 ** gain, spread)
    staged, plain = (run_chunk(case, room).reshape(want.shape) for room in (True, False))
    err = [float(np.linalg.norm(got - want) / np.linalg.norm(want)) for got in (staged, plain)]
    print("mla falling scales", gain, spread, err)
    assert err[0] <= 1.05 * err[1]


@pytest.mark.gpu
@pytest.mark.parametrize("heads,rows,length", [(16, 300, 2403), (128, 110, 4005), (40, 185, 2231), (1, 1001, 1500)])  # 8, 1, 3 and 128 rows a workgroup
def test_rows_are_independent_of_later_tokens(heads, rows, length):
    """The last five tokens hold infinite scales, NaN and NaN rope columns: rows that do not see them come out as with ordinary ones there."""
    case = make_mla_chunk_case(heads + 1, [length], rows, heads, block_tokens=64)
    clean = run_chunk(case, True)[:rows - 5]
    assert (length - 5) % 64 <= 59
    at = int(case["tables"][0][(length - 5) // 64]) * 64 + (length - 5) % 64  # five tokens of one page
    case["scales"][at:at + 2], case["scales"][at + 2:at + 4], case["rope"][at + 4] = 0x7F80, 0x7FC0, 0x7FC0
    for room in (True, False):
        got = run_chunk(case, room)[:rows - 5]
        assert np.linalg.norm(got - clean) <= 2.0 ** -11 * np.linalg.norm(clean)


@pytest.mark.gpu
def test_a_row_keeps_its_bits_before_a_far_larger_token():
    """One row a workgroup: a last token 2^24 above the others is no part of the rows before it, though it lies in their last tile."""
    case, want = rope_score_chunk(128, 110, 4007, 1.0, 2.0)
    at = int(case["tables"][0][4006 // 64]) * 64 + 4006 % 64
    case["scales"][at] = O.f32_to_bf16(O.bf16_to_f32(case["scales"][at]) * np.float32(2.0 ** 24))
    err = [float(np.linalg.norm((run_chunk(case, room).reshape(want.shape) - want)[:109]) / np.linalg.norm(want[:109])) for room in (True, False)]
    print("mla row before a large token", err)
    assert err[0] <= 1.05 * err[1]


@pytest.mark.gpu
def test_later_stages_take_up_the_records_of_a_whole_call():
    """With the preferred workspace, more, and the least: merge and projection again over the records that a whole call has left, and the
    call stage by stage, give the bits of the whole call; the layout's statistics are those of every live split."""
    from zllm_amd import capi, ops

    heads, rows, lens = 16, 300, [2400, 1700]
    case = make_mla_chunk_case(3, lens, rows, heads, block_tokens=64)
    keep = [upload(case[n]) for n in ("codes", "scales", "rope", "tables", "lens")]  # the argument block holds addresses only
    q, (weights, form) = to_torch_bf16(case["q_bits"], "cuda"), weight_args(case)
    args, out, workspace = ops.mla_decode_args(q, weights, *keep, heads, 192, 256, 512, 64, 64, max(lens),
                                               query_rows=rows, **form)
    lib = capi.load()
    preferred, least = args.workspace_bytes, lib.zllm_attn_mla_decode_workspace_bytes(C.byref(args))
    assert preferred > least, "this shape is meant to be staged"
    workspace = torch.empty(preferred + 4096, dtype=torch.uint8, device="cuda")
    args.workspace = workspace.data_ptr()
    for size in (preferred, preferred + 4096, least):
        args.workspace_bytes = size
        workspace.fill_(0xFF)
        outs = []
        for masks in ((0,), (12,), (3, 12), (1, 2, 4, 8), (1, 2 | capi.MLA_WIDE_TILES, 12)):
            out.zero_()
            for mask in masks:
                args.stage_mask = mask
                capi.check(lib.zllm_attn_mla_decode(C.byref(args), ops._stream()))
            outs.append(out.clone())
            layout = capi.SplitRecordLayout()
            capi.check(lib.zllm_attn_mla_decode_record_layout(C.byref(args), C.byref(layout)))
            stats = workspace[layout.stats_offset:layout.stats_offset + layout.record_rows * heads * 8].view(torch.float32).view(-1, heads, 2)
            for row in (0, rows - 1, rows, 2 * rows - 1):
                length = lens[row // rows] - (rows - 1 - row % rows)
                live = stats[row * layout.max_chunks:row * layout.max_chunks + -(-length // layout.chunk_tokens)]
                assert bool(torch.isfinite(live).all()) and float(live[..., 1].min()) > 0
        assert float(outs[0].abs().max()) > 0
        # merge and projection are one kernel in a whole call and two stage by stage: f32 sums in another order
        assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
        assert float((outs[3] - outs[0]).norm() / outs[0].norm()) <= 1e-5
        # the other partial kernels write the same places: an f16 weight is within 2^-11 of its value in
        # each of the two kernels, so a term of one is within 2^-10 of the other's
        assert float((outs[4] - outs[0]).norm() / outs[0].norm()) <= 2.0 ** -10


@pytest.mark.gpu
def test_staged_latents_in_a_graph():
    """Staging and attention recorded together, replayed over caches that change in between."""
    from zllm_amd import capi, ops

    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    heads, rows, total, page = 8, 240, 2000, 64
    table = torch.randperm(40, generator=gen, device="cuda")[:32].to(torch.int32)[None].contiguous()
    codes, scales, rope = (torch.zeros(40 * page, n, dtype=t, device="cuda") for n, t in ((512, torch.int8), (8, torch.int16), (64, torch.int16)))
    lens = torch.tensor([total], dtype=torch.int32, device="cuda")
    q = torch.randn(rows, heads * 192, generator=gen, device="cuda", dtype=torch.bfloat16)
    weights = (torch.randn(heads * 256, 512, generator=gen, device="cuda") / 512 ** 0.5).to(torch.bfloat16)
    args, out, workspace = ops.mla_decode_args(q, weights, codes, scales, rope, table, lens, heads, 192, 256, 512, 64, page, total, query_rows=rows)
    lib = capi.load()
    assert workspace.numel() > lib.zllm_attn_mla_decode_workspace_bytes(C.byref(args)), "this shape is meant to be staged"

    def fill():
        ops.mla_append(torch.randn(total, 512, generator=gen, device="cuda"), torch.randn(total, 64, generator=gen, device="cuda"), codes, scales, rope,
                       table[0], 0, page)

    def call():
        capi.check(lib.zllm_attn_mla_decode(C.byref(args), ops._stream()))

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
