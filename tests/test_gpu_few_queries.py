"""Rows of few queries on MFMA items (csrc/few_query.hip): drafted tokens, and decode rows of wide or odd GQA groups.

The cases sit on the edges of the item: (position, head) query rows per kv head that fill one 16-row block, spill into
the next, and reach 64; pages of one tile, of several and of none (48); rows of one query beside rows of several; rows
split over items and merged, on one kv head per item or a pair. Against the fp32 oracle, at the tolerances of the other
attention tests."""

import math

import pytest
import torch

from helpers import context_for, dense_expected, guarded_workspace, paged_step, plan_counts
from lvattn import Context, MI355XAttention, _capi

pytestmark = pytest.mark.gpu

TOL = {torch.float16: dict(atol=6e-3, rtol=6e-3), torch.bfloat16: dict(atol=2e-2, rtol=1e-2)}

# id: (query heads, kv heads), queries of each row, keys before them, page size, kv heads per item
STEPS = {
    "group5-decode": ((10, 2), [1] * 4, [0, 15, 300, 900], 16, 1),
    "group3-pairs-decode": ((6, 2), [1] * 8, [11_000] * 8, 16, 2),
    "group40-decode": ((40, 1), [1] * 3, [7, 64, 700], 64, 1),
    "16-rows": ((8, 2), [4, 4, 1], [500, 0, 33], 16, 1),
    "17-rows-odd-page": ((17, 1), [1, 1], [600, 47], 48, 1),
    "20-of-32-rows": ((8, 2), [5, 2, 3], [31, 2000, 64], 32, 1),
    "33-rows": ((6, 2), [11, 1, 11], [300, 1000, 5], 16, 1),
    "64-rows": ((8, 2), [16, 16], [0, 700], 64, 1),
    "one-head-drafts": ((3, 3), [4, 4, 4], [1500, 20, 3], 16, 1),
    "long-row-drafts": ((8, 2), [4, 4], [9000, 100], 256, 1),
}


def _run(cuda, heads, dim, dtype, new, cached, bs, layout="NHD", max_q=None):
    hq, hkv = heads
    need = [-(-(c + n) // bs) for c, n in zip(cached, new)]
    width, at, tables = max(need) + 1, 1, []
    for k in need:
        tables.append(list(range(at, at + k)) + [-1] * (width - k))
        at += k
    b = MI355XAttention(hq, dim, 1 / math.sqrt(dim), hkv)
    # Page 0 and the unused slots of every last page hold NaN: no item may let one through.
    qs, kf, vf, kn, vn, kc, vc, slots = paged_step(cached, new, tables, at, heads=hq, kv_heads=hkv, dim=dim, bs=bs,
                                                   device=cuda, dtype=dtype, seed=4, layout=layout, fill=float("nan"))
    b.store_kvcache(kn, vn, kc, vc, slots)
    ctx = context_for(cached, new, tables, cuda, is_prefill=max(new) > 1)
    if max_q is not None:
        ctx.max_seqlen_q = max_q
    b.launch_trace = []
    out = b.forward(torch.cat(qs), kn, vn, kc, vc, ctx)
    torch.cuda.synchronize()
    torch.testing.assert_close(out.float().cpu(), dense_expected(qs, kf, vf, 1 / math.sqrt(dim)), **TOL[dtype])
    return b.launch_trace[-1]


@pytest.mark.parametrize("step", list(STEPS))
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_few_query_items_match_the_oracle(cuda, dtype, dim, step):
    heads, new, cached, bs, hp = STEPS[step]
    info = _run(cuda, heads, dim, dtype, new, cached, bs)
    assert info["decode_kernel"] == "decode_list" and info["prompt_kernel"] == "none", info
    assert info["kv_heads_per_item"] == hp, info


# id: (query heads, kv heads), head dim, queries of each row, keys before them, max_seqlen_q if not theirs, and the number of
# splits of the longest row, within a split's rounding
UNEQUAL = {
    # Half the even share (of 512 workgroups 64 per kv head, less the rows' remainders), 15 and 14 for the average row.
    "8-queries-beside-decodes": ((32, 8), 128, [8] + [1] * 15, [64_000] + [300] * 15, None, (28, 32)),
    "two-of-many-queries": ((32, 8), 128, [9, 1, 16, 2], [5000, 3, 60_000, 900], None, (25, 30)),
    # As many as the merge pays for, lk / sqrt(0.3 lk lq G); 26 for the average row.
    "merge-bound-d64": ((8, 2), 64, [16] + [1] * 7, [64_000] + [10] * 7, None, (53, 58)),
    "merge-bound-d128": ((8, 2), 128, [1] * 7 + [16], [10] * 7 + [64_000], None, (53, 58)),
    "merge-bound-wide-group": ((40, 1), 64, [1], [64_000], None, (70, 74)),
    # A row of 7 queries in a step said to have one a row: its items attend all seven, and 79 splits of them (the
    # bound of one) have no room.
    "queries-of-a-one-query-step": ((6, 2), 64, [7] + [1] * 6, [20_000] + [5] * 6, 1, (51, 55)),
    # Slots for 4 queries a row at most: grown twice.
    "more-queries-than-the-step-says": ((8, 2), 64, [1] * 9 + [16] + [1] * 6, [10] * 9 + [64_000] + [20] * 6, 4, (32, 34)),
}


@pytest.mark.parametrize("case", list(UNEQUAL))
def test_a_long_row_of_more_queries_than_the_others_is_spread(cuda, monkeypatch, case):
    """Partials have room for the splits of a long row that has more queries than the step's average, and a row has no more
    splits than its merge is worth. Nothing is written past the workspace that the step asked for."""
    (hq, hkv), dim, new, cached, max_q, (least, most) = UNEQUAL[case]
    ws = guarded_workspace(monkeypatch, cuda)
    info = _run(cuda, (hq, hkv), dim, torch.bfloat16, new, cached, 16, max_q=max_q)
    assert info["decode_kernel"] == "decode_list" and info["prompt_kernel"] == "none", info
    lens = [c + n for c, n in zip(cached, new)]
    need = _capi.query("lv_paged_attention_workspace_bytes", len(new), sum(new), hq, hkv, dim, 16 * (-(-max(lens) // 16) + 1),
                       int(max_q == 1 or max(new) == 1))
    assert (ws[need:] == 0x5A).all()
    items, split = plan_counts(ws, info["decode_workgroups"] * info["kv_heads_per_item"] // hkv)
    assert items == sum(-(-n // split) for n in lens)
    assert least <= -(-max(lens) // split) <= most


@pytest.mark.parametrize("layout", ["NHD", "HND"])
def test_many_rows_of_drafts_take_kv_head_pairs(cuda, layout):
    """260 rows over 4 kv heads: two rounds of workgroups without splits, so each item takes a pair of kv heads; one row
    is long enough to be split all the same."""
    new = [3, 2, 1, 4] * 65
    cached = [(37 * i) % 150 for i in range(259)] + [6000]
    info = _run(cuda, (16, 4), 64, torch.bfloat16, new, cached, 16, layout)
    assert info["kv_heads_per_item"] == 2 and info["prompt_kernel"] == "none" and info["splitk_merge"], info


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_pairs_of_two_row_blocks(cuda, dtype, dim):
    """Items of a pair of kv heads whose query rows fill a 16-row block and spill into the next: 5 heads, up to 4 queries."""
    new = [3, 2, 1, 4] * 65
    cached = [(37 * i) % 90 for i in range(259)] + [6000]
    info = _run(cuda, (20, 4), dim, dtype, new, cached, 16)
    assert info["kv_heads_per_item"] == 2 and info["prompt_kernel"] == "none" and info["splitk_merge"], info


def test_a_row_of_more_queries_than_the_step_says(cuda):
    """max_seqlen_q sizes the item; a row of more query rows than it holds takes several passes over its keys."""
    info = _run(cuda, (8, 2), 64, torch.bfloat16, [7, 1, 1, 1], [900, 3, 4, 5], 16, max_q=3)
    assert info["decode_kernel"] == "decode_list" and info["prompt_kernel"] == "none", info


def test_drafts_share_one_plan_over_layers_and_graph_replays(cuda):
    """Two layers on one Context (the second reuses the plan), captured and replayed with new queries."""
    heads, dim, bs = (8, 2), 128, 16
    cached, new = [3000, 40], [4, 4]
    tables = [list(range(190)), list(range(190, 193)) + [-1] * 187]
    qs, kf, vf, kn, vn, kc, vc, slots = paged_step(cached, new, tables, 193, heads=8, kv_heads=2, dim=dim, bs=bs,
                                                   device=cuda, dtype=torch.bfloat16, seed=5)
    b = MI355XAttention(8, dim, 1 / math.sqrt(dim), 2)
    b.store_kvcache(kn, vn, kc, vc, slots)
    q = torch.cat(qs)
    template = context_for(cached, new, tables, cuda)

    def context():
        return Context(**{k: getattr(template, k) for k in Context.__slots__ if k not in ("attn_metadata",
                                                                                          "decode_splits")})

    def layers(outs):
        ctx = context()
        for out in outs:
            b.forward(q, None, None, kc, vc, ctx, out=out)

    outs = [torch.empty_like(q) for _ in range(2)]
    layers(outs)  # warm: allocates the workspace outside capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        layers(outs)
    gen = torch.Generator().manual_seed(6)
    for _ in range(3):
        q.copy_(torch.randn(q.shape, generator=gen).to(q.dtype))
        graph.replay()
        torch.cuda.synchronize()
        eager = b.forward(q, None, None, kc, vc, context())
        torch.cuda.synchronize()
        for out in outs:
            assert torch.equal(out, eager)


@pytest.mark.parametrize("new, cached, bs", [([40], [3000], 16), ([33, 20], [2100, 2], 64), ([70], [2500], 256),
                                              ([17, 1], [4000, 900], 32)])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_few_prompt_items_are_split_over_their_keys(cuda, dtype, dim, new, cached, bs):
    """Chunks of too few query tiles to fill the GPU, on cached prefixes: each tile's keys are cut into pieces (of a short
    row's tile some are empty) and merged. One query past a tile, one row beside another, and a decode row."""
    order = sorted(range(len(new)), key=lambda i: new[i] > 1)
    new, cached = [new[i] for i in order], [cached[i] for i in order]
    hq, hkv = (8, 2)
    info = _run(cuda, (hq, hkv), dim, dtype, new, cached, bs)
    items = -(-sum(new) // (128 // (hq // hkv))) + len(new)
    if info["prompt_kernel"] == "prompt_list":
        assert info["prompt_workgroups"] > items * hkv, info
    else:  # beside a decode row the schedule may overlap
        assert min(new) == 1, info


@pytest.mark.parametrize("rows", [1, 1024, 1025, 1300])
def test_a_step_of_prompts_lists_every_tile_once(cuda, monkeypatch, rows):
    """Rows of more queries than few-query items take, on both sides of the plan's rows per thread: the prompt tiles that the
    plan left in the workspace, last tile of a row first, no decode item, and the step's outputs against the oracle."""
    hq, hkv, dim, bs = 8, 1, 64, 16
    new = [17 + (7 * r) % 20 for r in range(rows)]
    ws = guarded_workspace(monkeypatch, cuda)
    info = _run(cuda, (hq, hkv), dim, torch.bfloat16, new, [0] * rows, bs)
    assert info["prompt_kernel"] == "prompt_list" and info["decode_kernel"] == "none", info
    qp = 128 // hq
    listed = -(-sum(new) // qp) + rows
    tiles = [(r, -1 - t) for r, n in enumerate(new) for t in reversed(range(-(-n // qp)))]
    assert ws[:8 * len(tiles)].view(torch.int32).view(-1, 2).tolist() == [list(t) for t in tiles]
    # The decode items' room behind the prompt items': one unsplit item a row.
    items, _ = plan_counts(ws, listed + rows)
    assert items == 0
