"""The packed tables of an eager step against tables formed token by token, and how their slots are looked up."""
import random

import numpy as np
import pytest
import torch

from tffinfer_amd.cache import CacheManager
from tffinfer_amd.engine.batch import StepEntry, build_step_batch
from tffinfer_amd.parts.base import KVCacheSpec

FULL = KVCacheSpec(2, 16, 0)
WIN = KVCacheSpec(2, 16, 24)


def a_step(rng, decoding, portions, ps=8):
    """A cache of two groups with ``decoding`` requests that bring a token and further ones that bring ``portions`` more."""
    held = [rng.randrange(1, 90) for _ in range(decoding)] + [rng.choice((0, 0, 3, 29, 64)) for _ in portions]
    news = [1] * decoding + list(portions)
    pages = sum((h + n) // ps + 1 for h, n in zip(held, news)) + 4
    cache = CacheManager([(0, True, FULL, None), (1, True, WIN, None)], ps, pages, len(held))
    entries = []
    for r in rng.sample(range(len(held)), len(held)):
        cache.add_request(r)
        for _ in range(held[r] // 3):               # (portion by portion, so that the window's group gives pages back)
            cache.reserve(r, 3)
            cache.commit(r, 3)
        cache.reserve(r, news[r])
        entries.append(StepEntry(r, [rng.randrange(1000) for _ in range(news[r])], sorted(rng.sample(range(news[r]), rng.randrange(min(3, news[r]) + 1)))))
    return cache, entries


def one_by_one(cache, entries):
    """What the step's tables have to say: (token ids, positions, request of each token, cu, start, context, state slots, logit
    rows), and per group (block tables, slots)."""
    ps = cache.page_size
    tok, pos, treq, cu, start, ctx, state, rows = [], [], [], [0], [], [], [], []
    for r, e in enumerate(entries):
        P = cache.num_tokens(e.req)
        rows += [len(tok) + w for w in e.want]
        for i, t in enumerate(e.tokens):
            tok.append(t)
            pos.append(P + i)
            treq.append(r)
        cu.append(len(tok))
        start.append(P)
        ctx.append(P + len(e.tokens))
        state.append(cache.slot(e.req))
    groups = []
    for g in range(len(cache.groups)):
        tables = [cache.block_table(g, e.req) for e in entries]
        width = max(1, max(map(len, tables)))
        slots = [tables[r][p // ps] * ps + p % ps for p, r in zip(pos, treq)]
        groups.append(([[max(p, 0) for p in t] + [0] * (width - len(t)) for t in tables], slots))
    return (tok, pos, treq, cu, start, ctx, state, rows), groups


STEPS = [(1, ()), (5, ()), (0, (1,)), (0, (20,)), (3, (60,)), (60, (60,)), (7, (127, 128, 129)), (0, (255,)),
         (0, (256,)), (2, (255, 5)), (20, (300, 1, 40, 700)), (0, (40, 40, 40, 40))]


@pytest.mark.parametrize("decoding,portions", STEPS)
def test_tables_are_those_of_the_tokens_one_by_one(decoding, portions):
    for seed in range(6):
        cache, entries = a_step(random.Random(seed), decoding, portions)
        b = build_step_batch(entries, cache, "cpu")
        flat, groups = one_by_one(cache, entries)
        for got, want in zip((b.token_ids, b.positions, b.token_req, b.cu_tokens, b.start_pos, b.context_lens, b.state_slots, b.logit_rows), flat):
            assert got.dtype == torch.int32 and got.tolist() == want
        for g, (tables, slots) in zip(b.groups, groups):
            assert g.block_tables.tolist() == tables and g.slot_mapping.tolist() == slots
            assert g.no_slot_mapping.tolist() == [-1] * len(slots)
        assert b.max_new_tokens == max(len(e.tokens) for e in entries) and b.max_context == max(flat[5])
        assert b.host_cu_tokens == flat[3] and b.host_start_pos == flat[4] and b.host_state_slots == flat[6]


@pytest.mark.parametrize("decoding,portions", STEPS)
def test_only_long_portions_look_their_slots_up_as_arrays(monkeypatch, decoding, portions):
    """A look-up by arrays costs six microseconds whatever it finds: sixty requests of one token each may not pay for it."""
    cache, entries = a_step(random.Random(3), decoding, portions)
    asked = []
    inner = CacheManager.slot_array
    monkeypatch.setattr(CacheManager, "slot_array", lambda self, g, req, start, n: asked.append(n) or inner(self, g, req, start, n))
    build_step_batch(entries, cache, "cpu")
    assert all(n >= 48 for n in asked), asked
    assert len(asked) <= 2 * len(portions)


def test_slots_of_spans_as_of_their_tokens():
    rng = random.Random(5)
    ps = 8
    cache = CacheManager([(0, True, FULL, None), (1, True, WIN, None)], ps, 400, 3)
    for r in ("a", "b", "c"):
        cache.add_request(r)
    for _ in range(60):                              # (the requests' pages lie between each other)
        for r in ("a", "b", "c"):
            cache.reserve(r, 7)
            cache.commit(r, 7)
    for _ in range(200):
        spans = []
        for r in rng.sample(("a", "b", "c"), rng.randrange(1, 4)):
            start = rng.randrange(420)
            spans.append((r, start, rng.choice((0, 1, 2, 9, 100, 127, 128, 250)) if start < 170 else 1))
        want = [cache.block_table(0, r)[j // ps] * ps + j % ps for r, s, n in spans for j in range(s, s + n)]
        got = cache.slots_of(0, spans)
        assert list(got) == want and (isinstance(got, list) or got.dtype == np.int32)
        for r, s, n in spans:
            one = [cache.block_table(0, r)[j // ps] * ps + j % ps for j in range(s, s + n)]
            assert cache.slot_array(0, r, s, n).tolist() == one == cache.slot_mapping(0, r, s, n)
    # behind the pages there are, and in a page that the window has left (at either length)
    for n in (1, 200):
        with pytest.raises(IndexError):
            cache.slots_of(0, [("a", 425, n)])
        with pytest.raises(RuntimeError, match="'a': token 5 lies in a page already given back"):
            cache.slots_of(1, [("b", 419, 1), ("a", 5, n)])
    live = (420 - 24 + 1) // ps * ps                 # the first token whose page the window still holds
    assert len(cache.slots_of(1, [("a", live, 420 - live)])) == 420 - live
    with pytest.raises(RuntimeError, match=f"token {live - 1} lies in a page already given back"):
        cache.slot_array(1, "a", live - 1, 3)


@pytest.mark.parametrize("n", [1, 16, 17, 40])
def test_the_check_of_a_portions_tokens(n):
    """Plain whole numbers pass at once where there are more than sixteen; what is outside the vocabulary, or no whole number, is named
    wherever it stands, and a truth value counts as the number it is, as in short portions."""
    from types import SimpleNamespace
    from tffinfer_amd.engine.runner import ModelRunner, StepError
    cache = CacheManager([(0, True, FULL, None)], 8, 16, 1)
    cache.add_request("r")
    runner = SimpleNamespace(cache=cache, vocab_size=100, max_model_len=64)
    good = [(7 * i) % 100 for i in range(n)]
    check = lambda toks: ModelRunner._validate(runner, [StepEntry("r", toks, [len(toks) - 1])])      # noqa: E731
    check(good)
    check(tuple(good))
    for at in {0, n // 2, n - 1}:
        for fine in (0, 99, True, False):
            check(good[:at] + [fine] + good[at + 1:])
        for bad in (-1, 100, 1 << 40, -(1 << 40), 3.0, "3", None, np.int64(3), np.int32(200), float("nan")):
            with pytest.raises(StepError, match="outside the vocabulary"):
                check(good[:at] + [bad] + good[at + 1:])
