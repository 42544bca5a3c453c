"""The online softmax of the chunk kernels where its reference point moves, behind a prefix of 2,000 keys of two kinds, so that
the scores of a row are two exact levels.  Against 64-bit attention on three heads."""
import numpy as np
import pytest
import torch

from zllm_amd import capi, ops

pytestmark = pytest.mark.gpu

POSITION = 2000
PAGE = 16
# every chunk kernel and tile size: rows, query heads, KV heads, head_dim, cache, scales, query
KERNELS = {
    "q8 tiles of 64": (16, 16, 4, 128, "q8", "f16", torch.bfloat16),
    "q8 tiles of 128": (32, 16, 4, 128, "q8", "f16", torch.bfloat16),
    "q8 tiles of 128, f32 query": (100, 16, 4, 128, "q8", "f16", torch.float32),
    "q8 tiles of 256": (100, 16, 4, 128, "q8", "f16", torch.bfloat16),
    "q8 tiles of 256, f32 scales": (100, 16, 4, 128, "q8", "f32", torch.bfloat16),
    "q8 64 wide": (100, 16, 4, 64, "q8", "f16", torch.bfloat16),
    "q8 256 wide": (100, 8, 4, 256, "q8", "f16", torch.bfloat16),
    "f16 tiles of 128": (32, 16, 4, 128, "f16", None, torch.bfloat16),
    "f16 tiles of 256": (100, 16, 4, 128, "f16", None, torch.bfloat16),
    "f16 256 wide": (100, 8, 4, 256, "f16", None, torch.bfloat16),
    "f16 waves of 32 pairs": (1030, 64, 64, 128, "f16", None, torch.bfloat16),
}


def attend(kernel, q, low, high, rise, k_scale, score_scale):
    """Distance (2-norm) from 64 bits of a chunk behind POSITION keys.  K of a key is `low` [KV heads, head_dim], from key `rise` on
    `high`, times k_scale; V is random."""
    rows, heads, kv_heads, dim, cache, scales, q_dtype = KERNELS[kernel]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rows + dim)
    n = POSITION + rows
    pages = (n + PAGE - 1) // PAGE
    order = torch.randperm(pages, generator=gen, device="cuda").to(torch.int32)
    at = (order.long()[:, None] * PAGE + torch.arange(PAGE, device="cuda")).view(-1)[:n]
    groups = kv_heads * dim // 64
    k_codes = torch.where(torch.arange(n, device="cuda")[:, None] < rise, low.reshape(1, -1), high.reshape(1, -1))
    v_codes = torch.randint(-100, 101, (n, kv_heads * dim), generator=gen, device="cuda")
    planes = []
    for codes, scale in ((k_codes, k_scale), (v_codes, 2.0**-6)):
        value = codes.double() * scale
        if cache == "f16":
            plane, scale_plane = torch.zeros(pages * PAGE, kv_heads * dim, dtype=torch.float16, device="cuda"), None
            plane[at] = value.to(torch.float16)
            assert torch.equal(plane[at].double(), value)
        else:
            plane = torch.zeros(pages * PAGE, kv_heads * dim, dtype=torch.int8, device="cuda")
            scale_plane = torch.full((pages * PAGE, groups), scale, dtype=torch.float16 if scales == "f16" else torch.float32, device="cuda")
            plane[at] = codes.to(torch.int8)
        planes.append((plane, scale_plane, value.view(n, kv_heads, dim)))
    (k_plane, k_scales, k), (v_plane, v_scales, v) = planes
    q = q.to(q_dtype).view(rows, heads * dim).contiguous()
    out = ops.gqa_prefill_chunk(q, k_plane, k_scales, v_plane, v_scales, order, POSITION, heads, kv_heads, dim, PAGE, score_scale, workspace=False,
                                kv_format=capi.KV_F16 if cache == "f16" else capi.KV_Q8G64,
                                scale_dtype=capi.SCALE_F32 if scales == "f32" else capi.SCALE_F16).view(rows, heads, dim)
    off = []
    hidden = torch.arange(n, device="cuda")[None] > POSITION + torch.arange(rows, device="cuda")[:, None]
    for head in (0, heads // 2, heads - 1):
        kvh = head // (heads // kv_heads)
        s = (q.view(rows, heads, dim)[:, head].double() @ k[:, kvh].T.contiguous()) * score_scale
        want = torch.softmax(s.masked_fill(hidden, float("-inf")), dim=-1) @ v[:, kvh]
        off.append(((out[:, head].double() - want).norm() / want.norm()).item())
    assert np.isfinite(off).all(), off
    return max(off)


@pytest.mark.parametrize("kernel", KERNELS)
def test_scores_too_large_to_add_a_few_units_to(kernel):
    """Scores around 2^25 (base 2), where f32 has multiples of four: a rise by eight units is a rise, not a probability of 2^8, which
    the f16 of the second product has no room for.  Products and sums are exact: 2^13 times 2^12, and 2^-3 times 0 or 2^6."""
    rows, heads, kv_heads, dim, _, _, _ = KERNELS[kernel]
    log2e = np.float32(1.4426950408889634)
    near = np.float32(np.log(2.0)) + np.arange(-4, 5, dtype=np.float32) * np.float32(2.0**-24)
    score_scale = next(s for s in near if s * log2e == 1)
    low, high = torch.zeros(kv_heads, dim, device="cuda"), torch.zeros(kv_heads, dim, device="cuda")
    low[:, 0] = high[:, 0] = 64.0
    high[:, -1] = 1.0
    q = torch.zeros(rows, heads, dim, device="cuda")
    q[:, :, 0], q[:, :, -1] = 2.0**13, 2.0**-3
    # numerator and denominator are f32 sums of 2,000 products: 2^-24 sqrt(2000) = 3e-6 each
    assert attend(kernel, q, low, high, 40, 2.0**6, float(score_scale)) < 1e-5


@pytest.mark.parametrize("kernel", KERNELS)
def test_tied_scores_behind_a_rise_lose_no_bits(kernel):
    """A score that rises by 0.8 to 5.6 units (base 2) after two steps and stays: the probabilities of the 2,000 keys that share the
    maximum are ones, exact in the f16 of a step that carries no low-order term.  Against a reference left at the first level
    they are rounded, all by the same 2^-12."""
    rows, heads, kv_heads, dim, _, _, _ = KERNELS[kernel]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(dim)
    low = torch.randint(10, 51, (kv_heads, dim), generator=gen, device="cuda") * (torch.randint(0, 2, (kv_heads, dim), generator=gen, device="cuda") * 2 - 1)
    # scores of the two levels: beta dim^0.5 x (mean magnitude 30) / 64, times one and two
    beta = torch.linspace(0.55, 3.7, rows * heads, device="cuda")[torch.randperm(rows * heads, generator=gen, device="cuda")].view(rows, heads, 1)
    q = low.sign().float().repeat_interleave(heads // kv_heads, dim=0)[None] * (beta * dim**-0.5 * 64 / 30)
    # numerator and denominator are f32 sums of 2,000 products: 2^-24 sqrt(2000) = 3e-6 each
    assert attend(kernel, q, low, 2 * low, 40, 2.0**-6, dim**-0.5) < 1e-5


@pytest.mark.parametrize("kernel", KERNELS)
def test_a_reference_that_lags_as_far_as_it_may(kernel):
    """Twelve steps of 32 keys whose scores rise by 5.9 units (base 2) each, under V scales that fill their power of two or pass into
    the next with every other step, and then the maximum for the rest: the largest values the second product's f16 may meet."""
    rows, heads, kv_heads, dim, cache, scales, q_dtype = KERNELS[kernel]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rows + dim)
    n = POSITION + rows
    pages = (n + PAGE - 1) // PAGE
    order = torch.randperm(pages, generator=gen, device="cuda").to(torch.int32)
    at = (order.long()[:, None] * PAGE + torch.arange(PAGE, device="cuda")).view(-1)[:n]
    level = torch.clamp(torch.arange(n, device="cuda") // 32, max=12)
    k_codes = torch.zeros(n, kv_heads, dim, device="cuda")
    k_codes[:, :, 0] = level[:, None]  # one product a score: exact
    v_codes = torch.randint(-100, 101, (n, kv_heads * dim), generator=gen, device="cuda")
    v_scale = 2.0**-6 * 1.9990234375 * 2.0 ** torch.clamp(level // 2, max=4)  # exact in f16
    planes = []
    for codes, scale in ((k_codes.view(n, -1), torch.ones(n, device="cuda")), (v_codes, v_scale)):
        value = codes.double() * scale[:, None].double()
        if cache == "f16":
            plane, scale_plane = torch.zeros(pages * PAGE, kv_heads * dim, dtype=torch.float16, device="cuda"), None
            plane[at] = value.to(torch.float16)
            value = plane[at].double()
        else:
            plane = torch.zeros(pages * PAGE, kv_heads * dim, dtype=torch.int8, device="cuda")
            scale_plane = torch.zeros((pages * PAGE, kv_heads * dim // 64), dtype=torch.float16 if scales == "f16" else torch.float32, device="cuda")
            plane[at] = codes.to(torch.int8)
            scale_plane[at] = scale[:, None].expand(n, kv_heads * dim // 64).to(scale_plane.dtype)
        planes.append((plane, scale_plane, value.view(n, kv_heads, dim)))
    (k_plane, k_scales, k), (v_plane, v_scales, v) = planes
    q = torch.zeros(rows, heads, dim, device="cuda")
    q[:, :, 0] = 1.0
    score_scale = 5.9 * float(np.log(2.0))
    out = ops.gqa_prefill_chunk(q.to(q_dtype).view(rows, heads * dim), k_plane, k_scales, v_plane, v_scales, order, POSITION, heads, kv_heads, dim, PAGE,
                                score_scale, workspace=False, kv_format=capi.KV_F16 if cache == "f16" else capi.KV_Q8G64,
                                scale_dtype=capi.SCALE_F32 if scales == "f32" else capi.SCALE_F16).view(rows, heads, dim)
    hidden = torch.arange(n, device="cuda")[None] > POSITION + torch.arange(rows, device="cuda")[:, None]
    for head in (0, heads // 2, heads - 1):
        kvh = head // (heads // kv_heads)
        s = (q[:, head].double() @ k[:, kvh].T.contiguous()) * score_scale
        want = torch.softmax(s.masked_fill(hidden, float("-inf")), dim=-1) @ v[:, kvh]
        # sums of 1,600 tied keys, numerator and denominator, 2^-24 sqrt(1600) = 2.4e-6 each; against a reference left 5.9 units below
        # the maximum, without the low-order term, the keys would be rounded alike by up to 2^-12
        off = ((out[:, head].double() - want).norm() / want.norm()).item()
        assert off < 1e-5, off


@pytest.mark.parametrize("cache,rows,heads,kv_heads,q_dtype", [("q8", 1000, 32, 8, torch.bfloat16), ("q8", 500, 32, 8, torch.float32), ("f16", 500, 64, 8, torch.bfloat16)])
@pytest.mark.parametrize("spread", [0.05, 0.3])
def test_the_first_512_keys_of_a_walk_carry_both_terms(cache, rows, heads, kv_heads, q_dtype, spread):
    """Near-even rows of first chunks in the kernels whose reference lags: a wave walks 512 keys at most (in tiles of 64 pairs each half of
    the waves takes every other 32 of 1,000), and eight of them weigh more than a sixteenth of their lane's sum."""
    dim = 128
    gen = torch.Generator(device="cuda")
    gen.manual_seed(rows + heads)
    pages = (rows + PAGE - 1) // PAGE
    table = torch.arange(pages, dtype=torch.int32, device="cuda")
    planes = []
    for _ in range(2):
        if cache == "f16":
            plane = torch.randn(pages * PAGE, kv_heads * dim, generator=gen, device="cuda").to(torch.float16)
            planes.append((plane, None, plane.double().view(-1, kv_heads, dim)))
        else:
            plane = torch.clamp(torch.randn(pages * PAGE, kv_heads * dim, generator=gen, device="cuda") * 40, -127, 127).to(torch.int8)
            scales = (0.02 + 0.01 * torch.rand(pages * PAGE, kv_heads * 2, generator=gen, device="cuda")).to(torch.float16)
            planes.append((plane, scales, (plane.view(-1, kv_heads * 2, 64).double() * scales.double()[:, :, None]).view(-1, kv_heads, dim)))
    (k_plane, k_scales, k), (v_plane, v_scales, v) = planes
    q = (torch.randn(rows, heads * dim, generator=gen, device="cuda") * spread).to(q_dtype)
    out = ops.gqa_prefill_chunk(q, k_plane, k_scales, v_plane, v_scales, table, 0, heads, kv_heads, dim, PAGE, dim**-0.5, workspace=False,
                                kv_format=capi.KV_F16 if cache == "f16" else capi.KV_Q8G64).view(rows, heads, dim)
    hidden = torch.ones(rows, rows, dtype=torch.bool, device="cuda").triu(1)
    for head in (0, heads - 1):
        kvh = head // (heads // kv_heads)
        s = (q.view(rows, heads, dim)[:, head].double() @ k[:rows, kvh].T.contiguous()) * dim**-0.5
        want = torch.softmax(s.masked_fill(hidden, float("-inf")), dim=-1) @ v[:rows, kvh]
        # f32 sums of 1,000 products in numerator and denominator, 2^-24 sqrt(1000) each, and of 128 products a score, 2^-24 sqrt(128)
        off = ((out[:, head].double() - want).norm() / want.norm()).item()
        assert off < 5e-6, off
