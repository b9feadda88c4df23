"""Queries and keys that are not finite, on every path that merges partial outputs, against the fp32 oracle.

A query of NaN, or one with an infinite element, makes its own output NaN and leaves every other row and head as it was:
an engine that watches outputs for NaN has to see it. A merge that drops NaN from its maximum, or takes a sum that is
not positive for "no key seen", turns such a row into zeros. Tolerances as test_gpu_attention.py's."""

import math

import pytest
import torch

from helpers import context_for, dense_expected, paged_step, slots_for
from lvattn import Context, MI355XAttention
from oracle import attention as A

pytestmark = pytest.mark.gpu

TOL = dict(atol=2e-2, rtol=1e-2, equal_nan=True)
LATENT, VDIM, SCALE = 576, 512, 0.137

# id: (query heads, kv heads), queries of each row, keys before them, page size
PAGED = {
    "decode": ((8, 2), [1, 1], [40, 900], 16),
    "decode-split": ((8, 2), [1, 1, 1], [9000, 40, 12_000], 16),
    "decode-pairs": ((8, 2), [1] * 520, [30] * 519 + [9000], 16),
    "few": ((8, 2), [4, 2], [300, 20], 16),
    "few-split": ((8, 2), [4, 4], [9000, 500], 16),
    "few-two-sets": ((8, 2), [12, 12], [5000, 30], 64),
    "few-wide-group": ((12, 1), [1, 1], [6000, 3], 16),
    "prompt": ((8, 2), [200, 40], [100, 0], 16),
    "prompt-split": ((8, 2), [70], [4000], 256),
    "prompt-split-rows": ((8, 2), [33, 40], [3000, 2], 64),
}


def _spoil(q, kind, key):
    """q: one query head row; key: a key that it sees, whose score an infinite element raises to +inf."""
    if kind == "nan":
        q.fill_(float("nan"))
    else:
        q[0] = math.copysign(math.inf, float(key[0]))


@pytest.mark.parametrize("kind", ["nan", "inf"])
@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("step", list(PAGED))
def test_a_query_that_is_not_finite_gives_nan(cuda, step, dim, kind):
    (hq, hkv), new, cached, bs = PAGED[step]
    need = [-(-(c + n) // bs) for c, n in zip(cached, new)]
    width, at, tables = max(need), 0, []
    for k in need:
        tables.append(list(range(at, at + k)) + [-1] * (width - k))
        at += k
    b = MI355XAttention(hq, dim, 1 / math.sqrt(dim), hkv)
    qs, kf, vf, kn, vn, kc, vc, slots = paged_step(cached, new, tables, at, heads=hq, kv_heads=hkv, dim=dim, bs=bs,
                                                   device=cuda, dtype=torch.bfloat16, seed=3)
    for q, k in zip(qs, kf):
        _spoil(q[0, 1], kind, k[0, 1 // (hq // hkv)])
        _spoil(q[-1, hq - 1], kind, k[0, hkv - 1])
    b.store_kvcache(kn, vn, kc, vc, slots)
    out = b.forward(torch.cat(qs), kn, vn, kc, vc, context_for(cached, new, tables, cuda, is_prefill=max(new) > 1))
    torch.cuda.synchronize()
    want = dense_expected(qs, kf, vf, 1 / math.sqrt(dim))
    assert want.isnan().any()
    torch.testing.assert_close(out.float().cpu(), want, **TOL)


def _mla(cuda, bs, lens, queries, heads, spoil_queries=False, spoil_latents=None):
    """Random rows of `lens` latents; spoil_latents(row's latents) plants values. The step's output
    and the oracle's."""
    gen = torch.Generator().manual_seed(5)
    need = [-(-n // bs) for n in lens]
    width, at, tables = max(need), 0, []
    for k in need:
        tables.append(list(range(at, at + k)) + [-1] * (width - k))
        at += k
    latents = [torch.randn(n, LATENT, generator=gen).to(torch.bfloat16) for n in lens]
    q = torch.randn(len(lens) * queries, heads, LATENT, generator=gen).to(torch.bfloat16)
    if spoil_queries:
        for i in range(len(lens)):
            _spoil(q[i * queries, 1], "nan", None)
            _spoil(q[(i + 1) * queries - 1, heads - 1], "inf", latents[i][0])
    cache = torch.zeros(at, bs, LATENT, dtype=torch.bfloat16)
    for lat, table in zip(latents, tables):
        if spoil_latents is not None:
            spoil_latents(lat)
        cache.view(-1, LATENT)[torch.tensor(slots_for(table, bs, 0, lat.size(0)))] = lat
    ctx = Context(context_lens=torch.tensor(lens, dtype=torch.int32, device=cuda),
                  block_tables=torch.tensor(tables, dtype=torch.int32, device=cuda))
    out = MI355XAttention(heads, LATENT, SCALE, heads).mla_decode(q.to(cuda), cache.to(cuda), VDIM, ctx)
    torch.cuda.synchronize()
    want = []
    for i, lat in enumerate(latents):
        for j in range(queries):  # each query over the latents it sees: masked ones must not reach it
            seen = lat[:lat.size(0) - queries + j + 1]
            s = A.dense_scores(q[i * queries + j:i * queries + j + 1], seen.unsqueeze(1), SCALE)
            want.append((s.softmax(-1) @ seen[:, :VDIM].float()).transpose(0, 1))
    return out.float().cpu(), torch.cat(want)


# Pages of 40 latents run on the split schedule.
@pytest.mark.parametrize("bs", [64, 40])
@pytest.mark.parametrize("heads, queries", [(16, 1), (16, 2), (32, 1)])
def test_a_latent_query_that_is_not_finite_gives_nan(cuda, heads, queries, bs):
    """Rows finished in one run, and rows cut over several."""
    out, want = _mla(cuda, bs, [40, 9000, 700], queries, heads, spoil_queries=True)
    assert want.isnan().any()
    torch.testing.assert_close(out, want, **TOL)


@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("bs", [64, 40])
@pytest.mark.parametrize("heads, queries", [(16, 2), (16, 4), (11, 3), (4, 5), (1, 16)])
def test_a_drafts_latent_reaches_no_earlier_query(cuda, heads, queries, bs, value):
    """The row's last latents, one per draft, are seen by the queries from their own on; the others' outputs do not
    change. Row lengths put the drafts at a stage's end, across its border and at a row's start, in one run and in several."""
    def spoil(lat):
        lat[-1, :VDIM:7] = value  # the last query's alone
        lat[-queries // 2, 3] = value
    lens = [queries, 31, 32, 33, 34, 64 + queries // 2, 5000, 9000]
    out, want = _mla(cuda, bs, lens, queries, heads, spoil_latents=spoil)
    assert not want.isfinite().all() and want.isfinite().any()
    torch.testing.assert_close(out, want, **TOL)
