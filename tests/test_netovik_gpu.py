"""The Netovik design in the engine against the plain implementation: each mechanism alone at
the level of its op, then whole models through the step function (whole prompts, decoding
token by token, portions down to two tokens, mixed batches on a pool whose pages and slots are
used again), and greedy generation through the engine's own entry point and scheduler."""
import math
import types

import pytest
import torch

import plain_netovik as plain
import replay_lib as rl
from helpers import note_error, oracle_logits, random_tokens, read_config, rel_err, tol
from netovik_models import CLOSE_CALL, NETOVIK_LENGTHS, NETOVIK_PAGE, comparable_tokens

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16}
NAMES = ["nvA", "nvB", "nvC", "nvD"]


def _ops():
    from tffinfer_amd.kernels import ops
    return ops


def _err(got, ref):
    got, ref = got.double().cpu(), ref.double().cpu()
    return float((got - ref).abs().max() / ref.abs().max().clamp_min(1e-30))


def _i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


def _batch(lengths, starts, slots=None):
    """The device tables of a step in which request r brings lengths[r] tokens after starts[r]."""
    cu, pos, req = [0], [], []
    for r, (n, s) in enumerate(zip(lengths, starts)):
        cu.append(cu[-1] + n)
        pos += list(range(s, s + n))
        req += [r] * n
    return types.SimpleNamespace(token_req=_i32(req), positions=_i32(pos), cu_tokens=_i32(cu), num_reqs=len(lengths),
                                 max_new_tokens=max(lengths), host_cu_tokens=cu,
                                 state_slots=_i32(slots if slots is not None else list(range(len(lengths)))))


# ---------------------------------------------------------------- mechanisms, one by one ---

@pytest.mark.parametrize("H,groups", [(60, 1), (60, 3), (256, 2), (1000, 5), (4096, 2), (5000, 1)])
@pytest.mark.parametrize("planes", [1, 3])
def test_norm_on_a_sublayers_output(H, groups, planes):
    ops = _ops()
    g = torch.Generator().manual_seed(H + planes)
    n, eps = 5, 1e-3
    x = torch.randn(n, H, generator=g) * 2
    w = 1 + 0.2 * torch.randn(H, generator=g)
    delta = torch.randn(planes, n, H, generator=g) * 3
    normed = plain.group_norm(delta.double().sum(0), w.double(), groups, eps)
    resid = x.clone().to(DEV)
    d = (delta[0] if planes == 1 else delta).contiguous().to(DEV)
    out = ops.group_rmsnorm_add(resid, d, w.to(DEV), groups, eps, torch.bfloat16)
    assert _err(resid, x.double() + normed) < 2e-6
    assert torch.equal(out.cpu(), resid.cpu().to(torch.bfloat16))      # the copy is the stream, rounded once
    resid = x.clone().to(DEV)
    assert ops.group_rmsnorm_add(resid, d, w.to(DEV), groups, eps, None) is None
    assert _err(resid, x.double() + normed) < 2e-6
    if planes == 1:     # the norm of chosen rows of the stream itself (the model's last norm)
        rows = _i32([4, 0, 2])
        y = ops.group_rmsnorm_add(None, d, w.to(DEV), groups, eps, torch.float32, rows=rows)
        assert _err(y, normed[[4, 0, 2]]) < 2e-6


@pytest.mark.parametrize("T,W", [(1, 48), (7, 321), (33, 1024)])
def test_sum_over_depth(T, W):
    ops = _ops()
    g = torch.Generator().manual_seed(T)
    depths = 5
    hist = torch.zeros(depths, T, W, device=DEV)
    ref_hist = []
    x = torch.randn(T, W, generator=g)
    for n in range(1, depths + 1):
        coef = torch.randn(n, generator=g)
        ref_hist.append(x.double())
        want = sum(coef[j].double() * ref_hist[j] for j in range(n))
        xd = x.to(DEV)
        out = ops.depth_average(hist, n, coef.to(DEV), xd, torch.bfloat16)
        assert _err(xd, want) < 2e-6 and torch.equal(out.cpu(), xd.cpu().to(torch.bfloat16))
        assert torch.equal(hist[n - 1].cpu(), x)
        x = xd.cpu() + torch.randn(T, W, generator=g)      # what a next layer would make of it


def test_mixes_with_the_token_before():
    """Three requests in one step: one at its start (zeros before it), one whose portion goes on from the
    state, one of a single token; the row before a portion's first token comes from the request's slot."""
    ops = _ops()
    g = torch.Generator().manual_seed(3)
    W, lengths, starts, slots = 40, [5, 1, 3], [0, 7, 2], [2, 0, 3]
    x = torch.randn(sum(lengths), W, generator=g)
    mu = torch.rand(5, W, generator=g)
    state = torch.randn(5, 16 + W, generator=g)
    state[2, 16:] = 0
    out = ops.token_shift_mix(x.to(DEV), state.to(DEV), 16, mu.to(DEV), _batch(lengths, starts, slots), torch.float32).cpu()
    at = 0
    for n, s, slot in zip(lengths, starts, slots):
        rows = x[at:at + n].double()
        before = plain.shifted(rows, state[slot, 16:].double())
        for m in range(5):
            assert _err(out[m, at:at + n], rows + (before - rows) * mu[m].double()) < 1e-6
        at += n


@pytest.mark.parametrize("H,D", [(3, 8), (2, 16), (2, 24), (1, 40), (2, 48), (2, 64), (1, 100), (2, 128)])
def test_recurrence_whole_and_in_portions(H, D):
    """The recurrence over 70 tokens at once, and the same tokens in portions of 1 to 30 beside another
    request, with the state carried in a slot: the same numbers, bit for bit; decays from almost 0 to almost 1."""
    ops = _ops()
    g = torch.Generator().manual_seed(D)
    T, W = 70, 16
    r, k, v = (torch.randn(T, H * D, generator=g) for _ in range(3))
    z = 3 * torch.randn(T, H * D, generator=g)
    w0 = torch.rand(H * D, generator=g) * 3.5 - 3
    u = torch.randn(H * D, generator=g)
    x = torch.randn(T, W, generator=g)
    w = torch.exp(-torch.exp(z.double() + w0.double()))
    ref, S_ref = plain.wkv_recurrence(r.double().view(T, H, D), k.double().view(T, H, D), v.double().view(T, H, D),
                                      w.view(T, H, D), u.double().view(H, D))
    row = H * D * D + W
    state = torch.zeros(4, row, device=DEV)
    dev = [t.to(DEV) for t in (r, k, v, z)]
    whole = ops.wkv_recurrence(*dev, w0.to(DEV), u.to(DEV), state, _batch([T], [0], [1]), H, D, x=x.to(DEV), prev_off=H * D * D)
    assert _err(whole, ref.reshape(T, H * D)) < 2e-5
    assert _err(state[1, :H * D * D].view(H, D, D), S_ref) < 2e-5
    assert torch.equal(state[1, H * D * D:].cpu(), x[-1])
    assert float(state[0].abs().max()) == 0 and float(state[2].abs().max()) == 0
    # in portions, in slot 3, beside a second request in slot 0 whose tokens are the same ones shifted
    state.zero_()
    got, at = [], 0
    for n in (1, 2, 30, 1, 7, 29):
        other = min(at + 1, T - n)
        idx = list(range(at, at + n)) + [other]
        step = [t[idx].contiguous() for t in dev]
        o = ops.wkv_recurrence(*step, w0.to(DEV), u.to(DEV), state, _batch([n, 1], [at, 0], [3, 0]), H, D,
                               x=x[idx].to(DEV), prev_off=H * D * D)
        got.append(o[:n])
        at += n
    # (heads of 64 and 128 run long portions in a form of their own, whose sums go in another order)
    if D in (64, 128):
        assert _err(torch.cat(got, 0), whole) < 2e-6
    else:
        assert torch.equal(torch.cat(got, 0), whole)


@pytest.mark.parametrize("group", [1, 255, 257, 512, 513, 1025, 2048, 2049, 2600])
def test_output_norm_and_depth_at_the_edges_of_a_block(group):
    """Groups around the sizes at which a thread has one element more, as a sum of planes; the sum over the depth of rows that
    are whole float4 and of rows that are not.  A float32 sum of n terms in chains of n / 256 and a tree is within 2^-24 (n / 256 + 10)
    of its size, the planes' and the levels' sums within 2^-24 of each addition: 32 times 2^-24 covers both."""
    ops = _ops()
    g = torch.Generator().manual_seed(group)
    n, groups, planes, levels = 3, 2, 5, 11
    H = groups * group
    d, x = torch.randn(planes, n, H, generator=g), torch.randn(n, H, generator=g)
    w, hist, coef = torch.randn(H, generator=g), torch.randn(levels, n, H, generator=g), torch.rand(levels, generator=g)
    resid = x.to(DEV)
    ops.group_rmsnorm_add(resid, d.to(DEV), w.to(DEV), groups, 1e-6, None)
    y = d.double().sum(0).view(n, groups, group)
    y = (y / torch.sqrt((y * y).mean(-1, keepdim=True) + 1e-6)).view(n, H) * w.double() + x.double()
    assert _err(resid, y) < 32 * 2 ** -24
    at, deep = x.to(DEV), hist.to(DEV)
    ops.depth_average(deep, levels, coef.to(DEV), at, torch.bfloat16)
    want = (coef[:-1, None, None].double() * hist[:-1].double()).sum(0) + coef[-1].double() * x.double()
    assert _err(at, want) < 32 * 2 ** -24
    assert torch.equal(deep[-1].cpu(), x) and torch.equal(deep[:-1].cpu(), hist[:-1])


@pytest.mark.parametrize("group,planes", [(1025, 3), (1025, 5), (2048, 5), (2049, 1), (2600, 3)])
def test_output_norm_of_many_rows_is_that_of_few(group, planes):
    """More blocks than are there at once take another form of the kernel: the same sums, the same bits."""
    ops = _ops()
    g = torch.Generator().manual_seed(group)
    n, groups = 520, 2
    H = groups * group
    d, x, w = torch.randn(planes, n, H, generator=g), torch.randn(n, H, generator=g), torch.randn(H, generator=g).to(DEV)
    many, few = x.to(DEV), x[:7].to(DEV)
    o_many = ops.group_rmsnorm_add(many, d.to(DEV), w, groups, 1e-6, torch.float32)
    o_few = ops.group_rmsnorm_add(few, d[:, :7].contiguous().to(DEV), w, groups, 1e-6, torch.float32)
    assert torch.equal(many[:7], few) and torch.equal(o_many[:7], o_few)


@pytest.mark.parametrize("H,D", [(4, 64), (2, 128)])
def test_recurrence_in_chunks_is_no_less_exact(H, D):
    """400 tokens in chunks against the same tokens in the two forms for shorter portions, all against 64 bits, in the 2-norm: no further
    off than those (products and sums within a chunk are formed in 64 bits), and under 1.5 units of 2^-23.  Roundings of 0.29 units each
    add up at random: those of a sum of D terms in chains of eight and of the sixteen or so chunks that a state remembers are some
    sqrt(16) x 0.29 = 1.2 units; measured 0.62 in chunks, 0.77 to 1.06 token by token."""
    ops = _ops()
    g = torch.Generator().manual_seed(D)
    T = 400
    r, k, v, z = (torch.randn(T, H * D, generator=g) for _ in range(4))
    w0, u = torch.rand(H * D, generator=g) * 3.5 - 3, torch.randn(H * D, generator=g)
    w = torch.exp(-torch.exp(z.double() + w0.double()))
    ref, _ = plain.wkv_recurrence(*(t.double().view(T, H, D) for t in (r, k, v, w)), u.double().view(H, D))
    ref, errors = ref.reshape(T, H * D), []
    for most in (T, 100, 10):
        state, out = torch.zeros(1, H * D * D, device=DEV), []
        for at in range(0, T, most):
            part = [t[at:at + most].contiguous().to(DEV) for t in (r, k, v, z)]
            out.append(ops.wkv_recurrence(*part, w0.to(DEV), u.to(DEV), state, _batch([part[0].shape[0]], [at], [0]), H, D))
        errors.append(float((torch.cat(out).double().cpu() - ref).norm() / ref.norm()))
    assert errors[0] < min(errors[1:]) and max(errors) < 1.5 * 2 ** -23, errors


@pytest.mark.parametrize("H,D", [(2, 64), (2, 128)])
@pytest.mark.parametrize("what", ["v", "k", "r", "z", "last v", "state"])
def test_recurrence_what_is_not_finite_reaches_later_tokens_only(H, D, what):
    """An infinity or NaN in a token's row of a portion in chunks, in its last token's, or in the state: what is not finite is so
    token by token as well, every other value is what it was within the bound of that form, the other head keeps its bits."""
    ops = _ops()
    g = torch.Generator().manual_seed(D)
    T = 170
    rows = {n: torch.randn(T, H * D, generator=g).to(DEV) for n in "rkvz"}
    w0, u = torch.randn(H * D, generator=g).to(DEV), torch.randn(H * D, generator=g).to(DEV)
    begin = torch.randn(1, H * D * D, generator=g).to(DEV)

    def outputs(rows, first, pieces):
        out, state = [], first.clone()
        for at in range(0, T, pieces):
            part = [rows[n][at:at + pieces].contiguous() for n in "rkvz"]
            out.append(ops.wkv_recurrence(*part, w0, u, state, _batch([part[0].shape[0]], [at], [0]), H, D))
        return torch.cat(out, 0).view(T, H, D), state.view(H, D, D)
    clean, clean_state = outputs(rows, begin, T)
    t = {"last v": T - 1, "state": 0}.get(what, 105)
    for x in (float("nan"),) if what in ("k", "r", "z") else (float("inf"), float("nan")):
        bad, first = {n: y.clone() for n, y in rows.items()}, begin.clone()
        if what == "state":
            first[0, 7] = x
        else:
            bad[what[-1]][t, 5] = x
        (got, state), (few, few_state) = outputs(bad, first, T), outputs(bad, first, 50)
        assert torch.equal(got[:, 1:], clean[:, 1:]) and torch.equal(state[1:], clean_state[1:])
        assert torch.equal(torch.isfinite(got), torch.isfinite(few)) and not bool(torch.isfinite(got).all())
        assert torch.equal(torch.isfinite(state), torch.isfinite(few_state))
        if t:
            assert _err(got[:t].flatten(1), clean[:t].flatten(1)) < 2e-5


@pytest.mark.parametrize("H,D", [(2, 64), (1, 128), (2, 48)])
@pytest.mark.parametrize("portions", [(1, 200, 2), (15, 16, 0, 127, 128, 1), (17, 3), (140, 300), (150, 20)])
def test_recurrence_of_a_portion_is_its_own_in_any_step(H, D, portions):
    """Portions on both sides of every limit between the forms, one of no tokens among them: outputs, states and kept rows
    of every request are the bits that it gives alone."""
    ops = _ops()
    g = torch.Generator().manual_seed(D + len(portions))
    T, R, W = sum(portions), len(portions), 8
    r, k, v, z = (torch.randn(T, H * D, generator=g).to(DEV) for _ in range(4))
    w0, u, x = (torch.randn(*s, generator=g).to(DEV) for s in ((H * D,), (H * D,), (T, W)))
    row = H * D * D + W
    many = torch.randn(R, row, generator=g).to(DEV)
    alone = many.clone()
    o = ops.wkv_recurrence(r, k, v, z, w0, u, many, _batch(list(portions), [0] * R, list(range(R))), H, D, x=x, prev_off=H * D * D)
    for i, n in enumerate(portions):
        at = sum(portions[:i])
        if n:
            part = [t[at:at + n].contiguous() for t in (r, k, v, z)]
            one = ops.wkv_recurrence(*part, w0, u, alone, _batch([n], [0], [i]), H, D, x=x[at:at + n].contiguous(), prev_off=H * D * D)
            assert torch.equal(one, o[at:at + n]), (i, n)
        assert torch.equal(alone[i], many[i]), (i, n)


@pytest.mark.parametrize("H,D,portions", [(2, 64, (128,)), (3, 64, (129, 3, 250)), (1, 128, (145, 128)), (2, 128, (16, 15, 200))])
def test_recurrence_in_chunks_of_sixteen(H, D, portions):
    """Portions beside one another, the longest of 128 tokens and more, from states that are not zero, with rows
    wider than the heads: against 64 bits, outputs, state and kept row; no other slot is touched.  A sum of some
    D terms and a product of up to 16 decays, each kept to half a unit of 2^-23, stay under 16 such units."""
    ops = _ops()
    g = torch.Generator().manual_seed(D + len(portions))
    T, W, R = sum(portions), 8, len(portions)
    wide = torch.randn(T, 4 * H * D, generator=g)
    wide[:, 3 * H * D:] *= 3
    w0 = torch.rand(H * D, generator=g) * 3.5 - 3
    u = torch.randn(H * D, generator=g)
    x = torch.randn(T, W, generator=g)
    row = H * D * D + W
    state = torch.randn(R + 2, row, generator=g)
    start = state.clone().double()
    dev, slots = wide.to(DEV), list(range(R, 0, -1))
    state = state.to(DEV)
    r, k, v, z = (dev[:, i * H * D:(i + 1) * H * D] for i in range(4))
    o = ops.wkv_recurrence(r, k, v, z, w0.to(DEV), u.to(DEV), state, _batch(list(portions), [0] * R, slots), H, D, x=x.to(DEV),
                           prev_off=H * D * D)
    R64, K64, V64, Z64 = (t.double().view(T, H, D) for t in wide.split(H * D, 1))
    w = torch.exp(-torch.exp(Z64 + w0.double().view(H, D)))
    at = 0
    for n, slot in zip(portions, slots):
        S, out = start[slot, :H * D * D].view(H, D, D).clone(), []
        for t in range(at, at + n):
            kv = K64[t][:, :, None] * V64[t][:, None]
            out.append((R64[t][:, :, None] * (S + u.double().view(H, D)[:, :, None] * kv)).sum(1))
            S = w[t][:, :, None] * S + kv
        assert _err(o[at:at + n], torch.stack(out).view(n, H * D)) < 16 * 2 ** -23
        assert _err(state[slot, :H * D * D].view(H, D, D), S) < 16 * 2 ** -23
        assert torch.equal(state[slot, H * D * D:].cpu(), x[at + n - 1])
        at += n
    for slot in (0, R + 1):
        assert torch.equal(state[slot].cpu().double(), start[slot])


def test_mixes_of_many_tokens_in_pieces():
    """Four tokens a block (1,030 rows of 4,096): requests that begin inside a block, one of a single token, a last block that is not full.
    The same bits as row by row (a request alone, one token a block)."""
    ops = _ops()
    g = torch.Generator().manual_seed(4)
    W, lengths, starts, slots = 4096, [501, 1, 526, 2], [0, 7, 2, 9], [2, 0, 3, 1]
    x, mu, state = (torch.randn(*s, generator=g).to(DEV) for s in ((sum(lengths), W), (5, W), (5, 16 + W)))
    for dtype in (torch.bfloat16, torch.float32):
        out, at = ops.token_shift_mix(x, state, 16, mu, _batch(lengths, starts, slots), dtype), 0
        for n, s, slot in zip(lengths, starts, slots):
            rows = x[at:at + n]
            one = ops.token_shift_mix(rows.contiguous(), state, 16, mu, _batch([n], [s], [slot]), dtype)
            assert torch.equal(out[:, at:at + n], one)
            before = torch.cat((state[slot, 16:][None], rows[:-1])).double()
            ref = rows.double() + (before - rows.double()) * mu[:, None].double()
            assert _err(one.float(), ref) < (1e-6 if dtype == torch.float32 else 2.0 ** -8)
            at += n


@pytest.mark.parametrize("T", [1, 37])
@pytest.mark.parametrize("H,D", [(3, 16), (5, 32), (3, 64), (7, 128), (2, 256)])
def test_norm_over_each_head_in_pieces(H, D, T):
    """Heads of a power of two on aligned rows, several a wave, a last wave that is not full; the shared weight and scale of the
    delta rule's form too.  bfloat16: one rounding, 2^-8 of the largest value."""
    ops = _ops()
    g = torch.Generator().manual_seed(H + D)
    o, gz = 5 * torch.randn(T, H * D, generator=g), 2 * torch.randn(T, H * D + 4, generator=g)
    w = 1 + 0.3 * torch.randn(H * D, generator=g)
    unit = plain.unit_rms(o.double().view(T, H, D), 1e-4).reshape(T, H * D) * plain.silu(gz[:, 4:].double())
    for dtype, tol in ((torch.float32, 2e-6), (torch.bfloat16, 2.0 ** -8)):
        got = ops.head_norm_gate(o.to(DEV), gz.to(DEV)[:, 4:], w.to(DEV), 1e-4, H, D, dtype)
        assert _err(got.float(), unit * w.double()) < tol
        wide = torch.zeros(T, H * D + 8, device=DEV, dtype=dtype)
        ops.head_norm_silu_gate(o.to(DEV), gz.to(DEV)[:, 4:], w[:D].to(DEV), 1e-4, H, D, wide[:, 8:], 0.7)
        assert _err(wide[:, 8:].float(), 0.7 * unit * w[:D].double().repeat(H)) < tol and float(wide[:, :8].abs().max()) == 0


@pytest.mark.parametrize("H,D", [(3, 8), (2, 40), (1, 128)])
def test_norm_over_each_head_and_gate(H, D):
    ops = _ops()
    g = torch.Generator().manual_seed(H)
    T, eps = 9, 1e-4
    o, gz = 5 * torch.randn(T, H * D, generator=g), 2 * torch.randn(T, H * D, generator=g)
    w = 1 + 0.3 * torch.randn(H * D, generator=g)
    ref = plain.unit_rms(o.double().view(T, H, D), eps).reshape(T, H * D) * w.double() * plain.silu(gz.double())
    assert _err(ops.head_norm_gate(o.to(DEV), gz.to(DEV), w.to(DEV), eps, H, D, torch.float32), ref) < 2e-6


def test_distance_buckets_of_the_package():
    from tffinfer_amd.parts.mixed_attention import distance_buckets
    for B, Dmax in ((32, 120), (6, 25), (16, 64), (8, 33), (12, 40)):
        got = distance_buckets(B, Dmax).tolist()
        assert got == [plain.distance_bucket(n, B, Dmax) for n in range(Dmax + 1)]
        assert got[-1] == B - 1 and plain.distance_bucket(10 * Dmax, B, Dmax) == B - 1


class _Cache:
    """Keys and values of one request (or several) in pages that lie in a shuffled order."""

    def __init__(self, G, D, page, lengths, dtype, seed=0):
        self.page = page
        blocks = [-(-n // page) for n in lengths]
        total = sum(blocks) + 3
        perm = torch.randperm(total, generator=torch.Generator().manual_seed(seed)).tolist()
        self.tables, at = [], 0
        for b in blocks:
            self.tables.append(perm[at:at + b])
            at += b
        self.k = torch.zeros(total, G, page, D, dtype=dtype, device=DEV)
        self.v = torch.zeros(total, G, D, page, dtype=dtype, device=DEV)
        width = max(blocks)
        self.bt = _i32([t + [0] * (width - len(t)) for t in self.tables])

    def view(self, reqs, starts, lengths):
        slots = []
        for r, s, n in zip(reqs, starts, lengths):
            slots += [self.tables[r][j // self.page] * self.page + j % self.page for j in range(s, s + n)]
        bt = self.bt[torch.tensor(reqs, device=DEV)].contiguous()
        return types.SimpleNamespace(k_cache=self.k, v_cache=self.v, block_tables=bt, slot_mapping=_i32(slots),
                                     page_size=self.page)


def _attention_case(H, G, D, T, seed, loud=None):
    """Random unit queries and keys; ``loud`` = (query, key, head): that pair's score stands out."""
    g = torch.Generator().manual_seed(seed)
    qk = torch.randn(T, (H + G) * D, generator=g)
    qb, kb = 0.3 * torch.randn(H * D, generator=g), 0.3 * torch.randn(G * D, generator=g)
    if loud is not None:
        i, j, h = loud
        kv = h // (H // G)
        direction = torch.randn(D, generator=g)
        qk[i, h * D:(h + 1) * D] = 6 * direction - qb[h * D:(h + 1) * D]
        qk[j, (H + kv) * D:(H + kv + 1) * D] = 6 * direction - kb[kv * D:(kv + 1) * D]
    return qk, qb, kb


def _plain_attention(qk, qb, kb, H, G, D, eps, **kw):
    T = qk.shape[0]
    q = (qk[:, :H * D].double() + qb.double()).view(T, H, D)
    k = (qk[:, H * D:].double() + kb.double()).view(T, G, D)
    kw = {n: (v.double() if isinstance(v, torch.Tensor) else v) for n, v in kw.items()}
    return plain.attend(plain.unit_rms(q, eps), plain.unit_rms(k, eps), k, **kw).reshape(T, H * D)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,G,D,page", [(4, 2, 16, 16), (3, 3, 8, 8), (12, 4, 8, 32), (1, 1, 40, 8), (6, 1, 64, 16), (5, 5, 12, 16),
                                        (5, 5, 32, 16), (32, 8, 128, 32), (9, 3, 64, 8), (16, 16, 32, 16), (12, 4, 64, 16), (20, 2, 32, 32)])
def test_attention_with_every_term(H, G, D, page, dtype):
    """Bias, cap, exchange between heads, window with kept first tokens and the 1 in the denominator, on a
    prompt in one step and on the same tokens as a prompt's portion followed by single tokens; then each
    term left out in turn.  (In bfloat16, heads of 32, 64 and 128 run portions of 64 tokens and more on the
    matrix cores, sixteen queries a block.)"""
    ops = _ops()
    g = torch.Generator().manual_seed(H * D)
    T, eps, window, keep, B, Dmax = 150, 1e-5, 37, 5, 10, 50
    qk, qb, kb = _attention_case(H, G, D, T, H + D)
    rel = torch.randn(B, H, generator=g)
    talk = torch.eye(H) + 0.5 * torch.randn(H, H, generator=g)
    from tffinfer_amd.parts.mixed_attention import distance_buckets
    table = rel[distance_buckets(B, Dmax)].contiguous().to(DEV)
    limit = 2e-5 if dtype == torch.float32 else 3e-2
    scale = min(0.7, 6.0 / D)       # (unit queries and keys: their products reach D)
    variants = [dict(cap=4.0, rel=rel, talk=talk, window=window, keep=keep, sink=True),
                dict(cap=0.0, rel=None, talk=None, window=None, keep=0, sink=False),
                dict(cap=4.0, rel=rel, talk=None, window=window, keep=0, sink=True),
                dict(cap=0.0, rel=None, talk=talk, window=window, keep=keep, sink=False)]
    for kw in variants:
        ref = _plain_attention(qk, qb, kb, H, G, D, eps, scale=scale, bias_max=Dmax, **kw)
        args = dict(scale=scale, softcap=kw["cap"], bias=table if kw["rel"] is not None else None,
                    mix=kw["talk"].to(DEV) if kw["talk"] is not None else None, window=kw["window"] or 0,
                    keep_first=kw["keep"], sink=kw["sink"])
        for cuts in ([T], [100] + [1] * 50, [3, 2, 61, 64, 20]):
            cache = _Cache(G, D, page, [T], dtype, seed=len(cuts))
            outs, at = [], 0
            for n in cuts:
                kv = cache.view([0], [at], [n])
                q = ops.qk_bias_norm_store(qk[at:at + n].contiguous().to(DEV), qb.to(DEV), kb.to(DEV), eps, H, G, D, kv)
                outs.append(ops.mixed_attention(q, H, G, D, kv, _batch([n], [at]), **args))
                at += n
            err = _err(torch.cat(outs, 0), ref)
            assert err < limit, f"{[k for k, v in kw.items() if v is not None and v is not False and v != 0]} cut {cuts[:3]}: {err:.3e}"


@pytest.mark.parametrize("H,G,D,page", [(32, 8, 128, 16), (32, 32, 64, 16), (20, 5, 64, 48), (9, 3, 32, 16), (24, 24, 32, 64), (16, 1, 128, 32)])
def test_attention_on_the_matrix_cores_at_the_tiles_edges(H, G, D, page):
    """Portions of 64 tokens and more in bfloat16 (tiles of 64 keys, blocks of 16 queries) and single tokens (tiles of 32) whose
    contexts, windows and kept tokens end just before, at and just behind a tile's border; slots that no token has written
    hold NaN, which reaches nothing."""
    ops = _ops()
    from tffinfer_amd.parts.mixed_attention import distance_buckets
    g = torch.Generator().manual_seed(H + G)
    eps, B, Dmax = 1e-5, 10, 50
    talk = torch.eye(H) + 0.3 * torch.randn(H, H, generator=g)
    rel = torch.randn(B, H, generator=g)
    table = rel[distance_buckets(B, Dmax)].contiguous().to(DEV)
    for T, first, window, keep in ((65, 64, 0, 0), (193, 127, 64, 1), (258, 192, 65, 64), (320, 255, 128, 33), (129, 113, 31, 32)):
        qk, qb, kb = _attention_case(H, G, D, T, T + H)
        ref = _plain_attention(qk, qb, kb, H, G, D, eps, scale=min(0.7, 6.0 / D), cap=4.0, rel=rel, bias_max=Dmax, talk=talk,
                               window=window or None, keep=keep, sink=True)
        for cuts in ([first] + [1] * (T - first), [T - 64, 64], [first // 16 * 16, T - first // 16 * 16]):
            cache = _Cache(G, D, page, [T], torch.bfloat16, seed=T)
            cache.k.fill_(float("nan"))
            cache.v.fill_(float("nan"))
            outs, at = [], 0
            for n in cuts:
                if n:
                    kv = cache.view([0], [at], [n])
                    q = ops.qk_bias_norm_store(qk[at:at + n].contiguous().to(DEV), qb.to(DEV), kb.to(DEV), eps, H, G, D, kv)
                    outs.append(ops.mixed_attention(q, H, G, D, kv, _batch([n], [at]), scale=min(0.7, 6.0 / D), softcap=4.0, bias=table,
                                                    mix=talk.to(DEV), window=window, keep_first=keep, sink=True))
                at += n
            err = _err(torch.cat(outs, 0), ref)
            assert err < 3e-2, (T, window, keep, cuts[:2], err)      # (bfloat16 queries, keys, weights and results, as above)


@pytest.mark.parametrize("H,G,D,page", [(32, 8, 128, 16), (20, 5, 64, 16), (32, 32, 64, 16), (16, 1, 32, 32)])
@pytest.mark.parametrize("lengths", [[64], [111], [20, 37, 1, 28], [20, 37, 1, 50]])
def test_short_prompts_a_block_a_token(H, G, D, page, lengths):
    """Steps of 64 tokens and more whose requests hold little: a block a token, several of a request among them.  (Bound as above.)"""
    ops = _ops()
    from tffinfer_amd.parts.mixed_attention import distance_buckets
    g = torch.Generator().manual_seed(H + len(lengths))
    eps, B, Dmax, T = 1e-5, 10, 50, sum(lengths)
    talk, rel = torch.eye(H) + 0.3 * torch.randn(H, H, generator=g), torch.randn(B, H, generator=g)
    table = rel[distance_buckets(B, Dmax)].contiguous().to(DEV)
    qk, qb, kb = _attention_case(H, G, D, T, T + H)
    cache = _Cache(G, D, page, lengths, torch.bfloat16, seed=T)
    cache.k.fill_(float("nan"))
    cache.v.fill_(float("nan"))
    kv = cache.view(list(range(len(lengths))), [0] * len(lengths), lengths)
    q = ops.qk_bias_norm_store(qk.to(DEV), qb.to(DEV), kb.to(DEV), eps, H, G, D, kv)
    batch = _batch(lengths, [0] * len(lengths))
    batch.max_context = max(lengths)
    args = dict(scale=min(0.7, 6.0 / D), softcap=4.0, bias=table, mix=talk.to(DEV), window=33, keep_first=5, sink=True)
    out = ops.mixed_attention(q, H, G, D, kv, batch, **args)
    at = 0
    for n in lengths:
        ref = _plain_attention(qk[at:at + n], qb, kb, H, G, D, eps, scale=min(0.7, 6.0 / D), cap=4.0, rel=rel, bias_max=Dmax, talk=talk, window=33, keep=5, sink=True)
        assert _err(out[at:at + n], ref) < 3e-2
        at += n


def _queries_keys_values(H, G, D, T, seed):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(T, n, D, generator=g).to(torch.bfloat16) for n in (H, G, G)]


def _filled_cache(k, v, page, seed=0):
    """A cache of one request that holds keys and values [T, G, D]."""
    T, G, D = k.shape
    cache = _Cache(G, D, page, [T], k.dtype, seed=seed)
    at = torch.tensor([cache.tables[0][j // page] for j in range(T)]), torch.arange(T) % page
    cache.k[at[0].to(DEV), :, at[1].to(DEV)] = k.to(DEV)
    cache.v[at[0].to(DEV), :, :, at[1].to(DEV)] = v.to(DEV)
    return cache


def _softmax_of_values(scores, v, rep, sink):
    """scores [H, T] of one query in 64 bits, v [T, G, D]: the weighted values, without the keys of weight zero."""
    m = torch.clamp(scores.max(1, keepdim=True).values, min=0.0 if sink else -math.inf)
    p = torch.exp(scores - torch.where(m > -math.inf, m, 0.0))
    total = p.sum(1, keepdim=True) + (torch.exp(-m) if sink else 0.0)
    p = torch.where(total > 0, p / total, 0.0)
    out = torch.zeros(scores.shape[0], v.shape[2], dtype=torch.float64)
    for h in range(scores.shape[0]):
        keep = p[h] > 0
        out[h] = (p[h, keep, None] * v[keep, h // rep].double()).sum(0)
    return out


@pytest.mark.parametrize("splits", [1, 3, None])
@pytest.mark.parametrize("H,G,D,page", [(8, 4, 32, 16), (32, 8, 128, 16), (12, 12, 64, 8), (16, 16, 128, 16), (32, 32, 64, 16)])
def test_infinite_values_of_single_tokens(H, G, D, page, splits):
    """A key whose values are infinite in some elements gives these elements their infinity and leaves the others alone, also where its
    weight is one exactly; a NaN stays a NaN; keys that the token does not see reach nothing."""
    ops = _ops()
    rep, inf = H // G, math.inf
    for T, at in ((1, 0), (20, 7), (100, 99), (161, 31)):
        q, k, v = _queries_keys_values(H, G, D, T + 1, T + H)
        v[at, :, 3], v[at, :, 10], v[at, 0, 17], v[T, :, 20] = inf, -inf, math.nan, inf
        if at > 5:
            v[at - 3, :, 5], v[at - 3, :, 10] = -inf, -inf
        cache = _filled_cache(k, v, page)
        kv = cache.view([0], [T - 1], [1])
        out = ops.mixed_attention(q[T - 1:T].reshape(1, H * D).to(DEV), H, G, D, kv, _batch([1], [T - 1]), scale=0.5 / D ** 0.5, splits=splits)
        scores = torch.einsum("hd,thd->ht", q[T - 1].double(), k[:T].double().repeat_interleave(rep, 1)) * (0.5 / D ** 0.5)
        ref = _softmax_of_values(scores, v[:T], rep, False)
        got = out.double().cpu().view(H, D)
        for what in (torch.isnan, torch.isposinf, torch.isneginf):
            assert torch.equal(what(got), what(ref)), (T, what.__name__)
        fine = torch.isfinite(ref)
        assert fine.sum() > 0.8 * H * D
        assert float((got - ref)[fine].abs().max()) < 3e-2 * float(ref[fine].abs().max())


def test_capped_scores_of_single_tokens_are_as_exact_as_the_library_s():
    """Two keys whose scores differ by some sixteen units in the last place of the cap, values of 1 and -1: the result is half the scores'
    difference, so it shows the cap's rounding a thousand times enlarged.  Scores are sums of few products and exact in float32; their
    difference (2^-14 before the cap) and a weight near one lose 2^-9 of it at most, like the result's bfloat16.  Over 8,192 pairs a root mean
    square within 5 % (three deviations of such an estimate) of what float32 division and tanh of the library leave."""
    ops, g = _ops(), torch.Generator().manual_seed(3)
    H, G, D, R, cap, step = 32, 8, 32, 256, 30.0, 2.0 ** -14
    a = torch.randint(160, 240, (R, H), generator=g).float() / 64                   # (2.5 .. 3.75 in steps of 2^-6, eight bits)
    b = torch.randint(240, 256, (R, G), generator=g).float() / 32                   # (7.5 .. 8 in steps of 2^-5)
    cache = _Cache(G, D, 16, [2] * R, torch.bfloat16)
    q = torch.zeros(R, H, D)
    q[:, :, 0], q[:, :, 1] = a, 1
    for r in range(R):
        p = cache.tables[r][0]
        cache.k[p, :, :2, 0] = b[r, :, None].to(DEV)
        cache.k[p, :, 1, 1] = step
        cache.v[p, :, :, 0], cache.v[p, :, :, 1] = -1, 1
    out = ops.mixed_attention(q.bfloat16().to(DEV).view(R, H * D), H, G, D, cache.view(list(range(R)), [1] * R, [1] * R), _batch([1] * R, [1] * R),
                              scale=1.0, softcap=cap)
    s = (a * b.repeat_interleave(H // G, 1)).to(DEV)
    two = torch.stack([s, s + step])
    assert torch.equal(two.double()[1] - s.double(), torch.full_like(s, step).double()) and 18 < float(s.min()) and float(s.max()) <= 30

    def half_difference(capped):
        return torch.tanh((capped[1].double() - capped[0].double()) / 2)
    ref = half_difference(cap * torch.tanh(two.double() / cap))

    def rms(x):
        return float(((x.double() - ref) / ref).square().mean().sqrt())
    library, ours = rms(half_difference(cap * torch.tanh(two / cap))), rms(out.view(R, H, D)[:, :, 5])
    assert 1e-3 < library < 0.2 and ours < 1.05 * library, (ours, library)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("low", [-math.inf, torch.finfo(torch.float32).min])
def test_biases_that_shut_keys_out_of_single_tokens(low, dtype):
    """A bias of minus infinity, or of the lowest number there is, for distances from 40 on: whole tiles of visible keys without a weight
    of their own, before keys that have one, in one block and in splits of their own; or no weight at all."""
    ops = _ops()
    H, G, D, page = 8, 4, 32, 16
    bias = torch.zeros(60, H)
    bias[40:] = low
    bias[:, 5] = low                             # (head 5: for all distances)
    for T in (30, 100, 300):
        q, k, v = (t.to(dtype) for t in _queries_keys_values(H, G, D, T, T))
        cache = _filled_cache(k, v, page)
        kv = cache.view([0], [T - 1], [1])
        scores = torch.einsum("hd,thd->ht", q[T - 1].float(), k.float().repeat_interleave(H // G, 1)) * 0.1
        scores = (scores + bias[(T - 1 - torch.arange(T)).clamp(max=59)].T).double()      # (sums as float32 has them)
        for sink in (False, True):
            ref = _softmax_of_values(scores, v, H // G, sink)
            for splits in (1, 3, None):
                out = ops.mixed_attention(q[T - 1:T].reshape(1, H * D).to(DEV), H, G, D, kv, _batch([1], [T - 1]), scale=0.1, bias=bias.to(DEV),
                                          sink=sink, splits=splits).double().cpu().view(H, D)
                assert float((out - ref).abs().max()) < (3e-2 if dtype == torch.bfloat16 else 2e-5) * float(ref.abs().max()), (T, sink, splits)


@pytest.mark.parametrize("low", [-math.inf, torch.finfo(torch.float32).min, -1e37])
def test_biases_that_shut_keys_out_of_prompts(low):
    """The same for prompts of 64 tokens and more: tiles in which all that a query sees has the lowest score there is, before the tiles
    that count; head 5 sees nothing else, and the keys count alike (minus infinity: nothing)."""
    ops = _ops()
    H, G, D, page, T = 8, 4, 32, 16, 300
    bias = torch.zeros(60, H)
    bias[40:] = low
    bias[:, 5] = low
    q, k, v = _queries_keys_values(H, G, D, T, T)
    cache = _filled_cache(k, v, page)
    kv = cache.view([0], [0], [T])
    raw = torch.einsum("ihd,thd->iht", q.float(), k.float().repeat_interleave(H // G, 1)) * 0.1
    for sink in (False, True):
        out = ops.mixed_attention(q.reshape(T, H * D).to(DEV), H, G, D, kv, _batch([T], [0]), scale=0.1, bias=bias.to(DEV), sink=sink)
        got = out.double().cpu().view(T, H, D)
        for i in (0, 15, 16, 39, 40, 63, 64, 103, 104, 128, 200, 299):
            scores = (raw[i, :, :i + 1] + bias[(i - torch.arange(i + 1)).clamp(max=59)].T).double()
            ref = _softmax_of_values(scores, v[:i + 1], H // G, sink)
            assert float((got[i] - ref).abs().max()) < 3e-2 * float(ref.abs().max()), (i, sink)


@pytest.mark.parametrize("loudest", [0.0, 30.7, 100.3, 255.1, 700.1])
def test_a_prompt_whose_maximum_stays_gives_all_keys_alike(loudest):
    """Keys that all score the same, over 128 tiles without a window: a weight of one each, so the sums are whole numbers and exact,
    and values of +1 in the first half and of -1 in the second leave (first - second) / keys.  A factor that is not quite one where the
    maximum stays would take from the first tiles at every later one."""
    ops = _ops()
    H, G, D, page, T = 8, 8, 32, 16, 8192
    q, k = torch.zeros(T, H, D, dtype=torch.bfloat16), torch.ones(T, G, D, dtype=torch.bfloat16)
    v = torch.ones(T, G, D, dtype=torch.bfloat16)
    v[T // 2:] = -1
    cache = _filled_cache(k, v, page)
    kv = cache.view([0], [0], [T])
    bias = torch.full((1, H), loudest, device=DEV)
    out = ops.mixed_attention(q.reshape(T, H * D).to(DEV), H, G, D, kv, _batch([T], [0]), scale=1.0, bias=bias).float().cpu().view(T, H * D)
    sums = v[:, 0, 0].double().cumsum(0) / torch.arange(1, T + 1)
    # (the quotient's rounding and that to bfloat16; where the sum is zero nothing at all)
    assert bool(((out.double() - sums[:, None]).abs() <= sums.abs()[:, None] * 2 ** -8).all())


@pytest.mark.parametrize("decode", [False, True])
@pytest.mark.parametrize("edge", ["inside", "outside", "kept", "not_kept"])
def test_a_loud_key_at_the_windows_and_the_kept_tokens_edges(edge, decode):
    """One key whose score with the last query stands far out: just inside the window the output is that
    key's value, just outside it is not; the last of the kept first tokens is seen from anywhere, the one
    after it is not.  Among 300 keys, across page borders, in a prompt and in decoding."""
    ops = _ops()
    H, G, D, T, page, eps, window, keep = 2, 1, 16, 300, 16, 1e-6, 130, 6
    j = {"inside": T - window, "outside": T - window - 1, "kept": keep - 1, "not_kept": keep}[edge]
    qk, qb, kb = _attention_case(H, G, D, T, 5, loud=(T - 1, j, 1))
    cache = _Cache(G, D, page, [T], torch.float32)
    outs, at = [], 0
    for n in ([T - 1, 1] if decode else [T]):
        kv = cache.view([0], [at], [n])
        q = ops.qk_bias_norm_store(qk[at:at + n].contiguous().to(DEV), qb.to(DEV), kb.to(DEV), eps, H, G, D, kv)
        outs.append(ops.mixed_attention(q, H, G, D, kv, _batch([n], [at]), scale=3.0, window=window, keep_first=keep,
                                        sink=True))
        at += n
    out = torch.cat(outs, 0)[-1].view(H, D)[1].cpu()
    value = (qk[j, H * D:] + kb).float()
    near = torch.allclose(out, value, atol=2e-2)
    assert near == (edge in ("inside", "kept")), edge
    ref = _plain_attention(qk, qb, kb, H, G, D, eps, scale=3.0, cap=0.0, rel=None, bias_max=0, talk=None, window=window, keep=keep)
    assert _err(torch.cat(outs, 0), ref) < 2e-5


def test_the_sink_takes_weight():
    """Keys that all score far below zero: the 1 in the denominator takes nearly all the weight and the
    output nearly vanishes; without it the output is an average of values."""
    ops = _ops()
    H, G, D, T, eps = 2, 2, 8, 20, 1e-6
    qk, qb, kb = _attention_case(H, G, D, T, 9)
    cache = _Cache(G, D, 8, [T], torch.float32)
    kv = cache.view([0], [0], [T])
    q = ops.qk_bias_norm_store(qk.to(DEV), qb.to(DEV), kb.to(DEV), eps, H, G, D, kv)
    low = torch.full((4, H), -12.0, device=DEV)
    with_sink = ops.mixed_attention(q, H, G, D, kv, _batch([T], [0]), scale=0.1, bias=low, sink=True)
    without = ops.mixed_attention(q, H, G, D, kv, _batch([T], [0]), scale=0.1, bias=low, sink=False)
    assert float(with_sink.abs().max()) < 1e-3 < float(without.abs().max())


def test_batches_of_unequal_requests_share_the_attention():
    """Three requests in one step (a prompt's portion, a single token, a whole short prompt) give what each
    gives alone, bit for bit."""
    ops = _ops()
    H, G, D, page, eps = 4, 2, 16, 16, 1e-6
    lengths = [90, 41, 7]
    cases = [_attention_case(H, G, D, n, 20 + n) for n in lengths]
    qb, kb = cases[0][1], cases[0][2]
    args = dict(scale=0.5, softcap=6.0, window=33, keep_first=2, sink=True, splits=1)
    alone, cache = [], _Cache(G, D, page, lengths, torch.float32, seed=4)
    for r, (n, c) in enumerate(zip(lengths, cases)):
        kv = cache.view([r], [0], [n])
        q = ops.qk_bias_norm_store(c[0].to(DEV), qb.to(DEV), kb.to(DEV), eps, H, G, D, kv)
        alone.append(ops.mixed_attention(q, H, G, D, kv, _batch([n], [0]), **args))
    cache2 = _Cache(G, D, page, lengths, torch.float32, seed=5)
    firsts = [60, 40, 0]
    for r in (0, 1):        # what came before this step
        kv = cache2.view([r], [0], [firsts[r]])
        ops.qk_bias_norm_store(cases[r][0][:firsts[r]].contiguous().to(DEV), qb.to(DEV), kb.to(DEV), eps, H, G, D, kv)
    news = [n - f for n, f in zip(lengths, firsts)]
    kv = cache2.view([0, 1, 2], firsts, news)
    rows = torch.cat([c[0][f:] for c, f in zip(cases, firsts)], 0).contiguous().to(DEV)
    q = ops.qk_bias_norm_store(rows, qb.to(DEV), kb.to(DEV), eps, H, G, D, kv)
    got = ops.mixed_attention(q, H, G, D, kv, _batch(news, firsts), **args)
    want = torch.cat([a[f:] for a, f in zip(alone, firsts)], 0)
    assert torch.equal(got, want)
    # the keys of each token dealt to several blocks and merged: the same to rounding
    for splits in (None, 2, 5):
        assert _err(ops.mixed_attention(q, H, G, D, kv, _batch(news, firsts), **dict(args, splits=splits)), want) < 2e-6


@pytest.mark.parametrize("n,H,groups,planes,levels", [(1, 256, 1, 1, 2), (3, 1000, 2, 2, 5), (1, 4096, 2, 1, 8), (700, 2048, 2, 4, 3), (600, 4096, 2, 6, 4),
                                                      (2, 6000, 1, 1, 1), (5, 2049, 1, 2, 9), (1, 4096, 2, 1, 10), (1, 4096, 2, 1, 11), (64, 1024, 2, 1, 20),
                                                      (128, 2048, 2, 2, 20), (128, 2048, 2, 2, 21), (256, 2048, 2, 1, 33)])
def test_output_norm_with_the_sum_over_depth(n, H, groups, planes, levels):
    """Every form of the kernel, and what is better left to two launches (groups longer than it holds, many levels of few rows): the same bits
    as the two launches."""
    ops = _ops()
    g = torch.Generator().manual_seed(n + H)
    r = lambda *s: torch.randn(*s, generator=g).to(DEV)       # noqa: E731
    x, d, w, hist, coef = r(n, H), r(planes, n, H), r(H), r(levels + 1, n, H), r(levels)
    d = d if planes > 1 else d[0]
    for out_dtype in (torch.bfloat16, None):
        x1, x2, h1, h2 = x.clone(), x.clone(), hist.clone(), hist.clone()
        ops.group_rmsnorm_add(x1, d, w, groups, 1e-5)
        o1 = ops.depth_average(h1, levels, coef, x1, out_dtype)
        o2 = ops.group_rmsnorm_add(x2, d, w, groups, 1e-5, out_dtype, depth=(h2, levels, coef))
        assert torch.equal(x1, x2) and torch.equal(h1, h2) and ((o1 is None and o2 is None) or torch.equal(o1, o2))


@pytest.mark.parametrize("E,top", [(8, 3), (2, 2), (5, 1), (70, 4)])
def test_softmax_router_and_plain_gated_experts(E, top):
    ops = _ops()
    g = torch.Generator().manual_seed(E)
    T, W, ff = 40, 48, 24
    x = torch.randn(T, W, generator=g)
    P = {"router": torch.randn(E, W, generator=g).double()}
    for e in range(E):
        P[f"e{e}.gate"], P[f"e{e}.up"] = (0.3 * torch.randn(ff, W, generator=g).double() for _ in range(2))
        P[f"e{e}.down"] = 0.3 * torch.randn(W, ff, generator=g).double()
    ref = plain.moe_ff({"router": {"top": top}}, P, x.double())
    s = plain.router_scores(P, x.double())
    logits = (x.double() @ P["router"].T).float().to(DEV)
    idx, wts = ops.route_topk(None, None, None, top, logits=logits, softmax=True)
    want_idx = torch.argsort(s, dim=-1, descending=True, stable=True)[:, :top]
    assert torch.equal(idx.cpu().long(), want_idx)
    assert _err(wts, torch.gather(s, 1, want_idx)) < 1e-5
    stack = lambda n: torch.stack([P[f"e{e}.{n}"] for e in range(E)], 0).float().to(DEV)     # noqa: E731
    out = ops.routed_experts(x.to(DEV), stack("gate"), stack("up"), stack("down"), idx, wts, float("inf"), 1.0, up_offset=0.0)
    assert _err(ops.as_tensor(out), ref) < 2e-5
    b16 = lambda t: t.to(torch.bfloat16)        # noqa: E731
    for by_tiles in (False, True):
        out = ops.routed_experts(b16(x).to(DEV), b16(stack("gate")), b16(stack("up")), b16(stack("down")), idx, wts,
                                 float("inf"), 1.0, by_tiles=by_tiles, up_offset=0.0)
        assert _err(ops.as_tensor(out), ref) < 3e-2


# ---------------------------------------------------------------------- whole models ---

def requests_for(name, model_dir):
    V = read_config(model_dir)["vocab"]
    return {f"{name}{i}": random_tokens(n, V, 2000 + 11 * i + n) for i, n in enumerate(NETOVIK_LENGTHS[name])}


def check(model_dir, reqs, steps, results, dtype, name):
    """A request's rows before its first close call: in bfloat16 among the experts' scores, in both types a first
    token whose recurrence output all but cancels."""
    before = {rid: comparable_tokens(model_dir, tuple(toks), dtype) for rid, toks in reqs.items()}
    total = sum(len(t) for t in reqs.values())
    assert sum(before.values()) >= total // (5 if dtype == "bfloat16" else 2), "too little of these requests can be compared"
    return rl.check_against_oracle(model_dir, reqs, steps, results, tol(dtype, name), dtype, compare_before=before)


def make_runner(model_dir, dtype, page_size, num_pages, max_seqs=4, use_graphs=False):
    from tffinfer_amd.engine.runner import ModelRunner
    from tffinfer_amd.models import load_model
    model = load_model(model_dir, DTYPES[dtype], DEV)
    return ModelRunner(model, page_size=page_size, num_pages=num_pages, max_seqs=max_seqs, max_model_len=512,
                       use_graphs=use_graphs)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", NAMES)
def test_residual_stream_after_every_layer(netovik_dirs, name, dtype):
    """Layer by layer, so that a fault names its layer."""
    from tffinfer_amd.engine.batch import StepEntry, build_step_batch
    from tffinfer_amd.engine.runner import StepContext
    d = netovik_dirs[name]
    V = read_config(d)["vocab"]
    # (the first of a few sequences of which bfloat16 can be compared for twenty tokens and more)
    toks = next(t for t in (random_tokens(45, V, 77 + s) for s in range(40)) if comparable_tokens(d, tuple(t)) >= 20)
    want = []
    plain.forward(*plain.load(d), toks, want)
    upto = len(toks) if dtype == "float32" else comparable_tokens(d, tuple(toks))
    runner = make_runner(d, dtype, NETOVIK_PAGE[name], 16)
    model = runner.model
    runner.add_request("a")
    e = [StepEntry("a", toks, [])]
    runner.reserve(e)
    batch = build_step_batch(e, runner.cache, runner.device, runner._pinned)
    ctx = StepContext(runner.ops, runner.act_dtype, batch, runner.max_model_len, runner._calls, runner.cache)
    resid, pending = model.embedding.forward(ctx, batch.token_ids), None
    assert len(model.schedule) == len(want)
    for it, call in enumerate(model.schedule):
        pending = model.blocks[call.layer].forward(ctx.for_call(it), resid, pending)
        assert pending is None
        err = _err(resid[:upto], want[it][:upto])
        assert err < (4e-5 if dtype == "float32" else 4e-2), f"layer call {it} (layer {call.layer}): {err:.3e}"


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", NAMES)
@pytest.mark.parametrize("mode", ["whole", "tail", "chunks", "mixed"])
def test_replay_modes(netovik_dirs, name, dtype, mode):
    model_dir = netovik_dirs[name]
    reqs = requests_for(name, model_dir)
    steps = {"whole": rl.trace_whole, "tail": rl.trace_tail, "chunks": rl.trace_chunks,
             "mixed": rl.trace_mixed}[mode](reqs)
    ps = NETOVIK_PAGE[name]
    # the pool holds what is live at the worst moment and no more, so pages and slots are used again
    num_pages = rl.max_live_tokens(steps, unit=ps) // ps
    runner = make_runner(model_dir, dtype, ps, num_pages)
    results = rl.run_steps_in_process(runner, steps)
    worst = check(model_dir, reqs, steps, results, dtype, name)
    print(f"{name} {dtype} {mode}: worst rel. error {worst:.3e} over {len(steps)} steps, {num_pages} pages")
    assert all(g.pool.num_used == 0 for g in runner.cache.groups)


def test_a_windows_pages_go_back_but_the_kept_tokens_stay(netovik_dirs):
    """While a request grows far past its windows, every group with a window holds the pages of the window
    and of its kept first tokens and no more."""
    from tffinfer_amd.engine.batch import StepEntry
    d = netovik_dirs["nvB"]
    ps = NETOVIK_PAGE["nvB"]
    toks = random_tokens(130, read_config(d)["vocab"], 2130)
    runner = make_runner(d, "float32", ps, 20)
    runner.add_request("a")
    ref = oracle_logits(d, toks)
    at = 0
    for n in [50] + [1] * 80:
        lg = runner.step([StepEntry("a", toks[at:at + n], [n - 1])])
        at += n
        assert rel_err(lg[0], ref[at - 1]) <= tol("float32", "nvB")
    for g in runner.cache.groups:
        if g.spec.window:
            held = [b for b, p in enumerate(g.tables["a"]) if p >= 0]
            kept = -(-g.spec.keep_first // ps)
            assert held[:kept] == list(range(kept)) and len(held) <= kept + -(-(g.spec.window - 1) // ps) + 1
            assert held[kept] > kept        # (pages in between went back)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", ["nvB", "nvC"])
def test_long_decoding_through_captured_graphs(netovik_dirs, name, dtype):
    """Three requests decode some 150 tokens each, far past every window, as replays of captured
    HIP graphs beside eager prompt steps; state slots and pages of windows are used again."""
    model_dir = netovik_dirs[name]
    V = read_config(model_dir)["vocab"]
    reqs = {f"g{i}": random_tokens(n, V, 300 + n) for i, n in enumerate((160, 171, 190))}
    steps = rl.trace_mixed(reqs, max_live=3, prompt_frac=0.1, want_all=True)
    ps = NETOVIK_PAGE[name]
    runner = make_runner(model_dir, dtype, ps, rl.max_live_tokens(steps, unit=ps) // ps, use_graphs=True)
    results = rl.run_steps_in_process(runner, steps)
    check(model_dir, reqs, steps, results, dtype, name)
    assert runner._graphs, "no decode step ran as a graph"


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_trace_run_program(netovik_dirs, tmp_path, dtype):
    """The program itself, as a user calls it, on a model of this architecture, with its four state slots."""
    model_dir = netovik_dirs["nvA"]
    reqs = requests_for("nvA", model_dir)
    steps = rl.trace_mixed(reqs, want_all=False)
    out = rl.run_steps_subprocess(model_dir, dtype, steps, str(tmp_path / "out"), rl.max_live_tokens(steps, 64))
    check(model_dir, reqs, steps, out, dtype, "nvA")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", ["nvA", "nvB"])
def test_greedy_generation_through_the_engine(netovik_dirs, name, dtype):
    """The engine's own entry point: scheduler, portions beside decoding requests, graphs, sampler.
    Every kept row of logits matches the plain logits of the engine's own sequence, and every
    token is the first maximum of its row."""
    from tffinfer_amd import EngineOptions, LLMEngine
    d = netovik_dirs[name]
    V = read_config(d)["vocab"]
    prompts = [random_tokens(n, V, 80 + n) for n in (1, 9, 40, 70)]
    eng = LLMEngine.from_model_dir(d, EngineOptions(dtype=dtype, page_size=16, kv_tokens=512, max_num_seqs=3,
                                                    max_num_batched_tokens=48, prefill_chunk=24, max_model_len=256))
    eng.keep_logits = True
    res = eng.generate(prompts, max_new_tokens=40, ignore_eos=True)
    for r in res:
        assert len(r.output) == 40 and r.finish_reason == "length"
        ref = oracle_logits(d, r.prompt + r.output)
        margins = []
        plain.forward(*plain.load(d), r.prompt + r.output, margins=margins)
        close = torch.stack(margins).min(0).values < CLOSE_CALL if margins else torch.zeros(len(ref), dtype=torch.bool)
        for i, (row, tok) in enumerate(zip(r.logits, r.output)):
            assert tok == int(torch.argmax(row))
            if dtype == "bfloat16" and bool(close[:len(r.prompt) + i].any()):
                break       # (the sequence the engine chose made a close call: what follows may differ by more than rounding)
            err = rel_err(row, ref[len(r.prompt) + i - 1])
            note_error(dtype, d, err)
            assert err <= tol(dtype, d), f"output {i}: {err:.3e}"
    if dtype == "float32":
        cfg, W = plain.load(d)
        assert res[1].output[:8] == plain.greedy(cfg, W, prompts[1], 8)


def test_a_preempted_request_starts_its_state_again(netovik_dirs):
    """A pool so small that requests are preempted and computed again gives the tokens of a large pool:
    the state of a request that comes back starts at zero."""
    from tffinfer_amd import EngineOptions, LLMEngine
    d = netovik_dirs["nvC"]        # (its second layer keeps every key, so a small pool runs out)
    V = read_config(d)["vocab"]
    prompts = [random_tokens(n, V, 400 + n) for n in (30, 33, 28)]
    outs, preempted = [], []
    for pages in (64, 9):
        eng = LLMEngine.from_model_dir(d, EngineOptions(dtype="float32", page_size=16, num_pages=pages, max_num_seqs=3,
                                                        max_model_len=128))
        res = eng.generate(prompts, max_new_tokens=30, ignore_eos=True)
        outs.append([r.output for r in res])
        preempted.append(sum(r.num_preemptions for r in res))
    assert outs[0] == outs[1]
    assert preempted[0] == 0 and preempted[1] > 0


def test_the_command_line_with_a_configuration_file_of_this_architecture(tmp_path):
    """--config FILE --random-weights through bin/tffinfer: the weights are those of the folder that
    --save-model writes, the dumped rows are the logits that chose each token; a pool so small that
    requests are preempted and computed again gives the same tokens."""
    import json
    import os
    import subprocess
    import sys
    import numpy as np
    from netovik_models import NV_C
    prog = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bin", "tffinfer")
    cfg = tmp_path / "config.json"
    cfg.write_text(json.dumps(NV_C))
    folder, dump = str(tmp_path / "nvC"), str(tmp_path / "logits.f32")
    common = [sys.executable, prog, "--config", str(cfg), "--random-weights", "--seed", "5", "--fp32", "--n-ctx", "256",
              "--n-predict", "12", "--ignore-eos", "--json", "--random-prompts", "3:30", "--page-size", "8",
              "--max-batches", "3"]
    p = subprocess.run(common + ["--save-model", folder, "--dump-logits", dump, "--kv-tokens", "512"],
                       capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stderr[-3000:]
    recs = [json.loads(ln) for ln in p.stdout.strip().splitlines()]
    meta = json.load(open(dump + ".json"))
    V = NV_C["vocab"]
    rows = np.fromfile(dump, dtype="<f4").reshape(meta["shape"])
    assert meta["shape"] == [36, V]
    for i, r in enumerate(recs):
        ref = oracle_logits(folder, r["prompt"] + r["output"])
        first = meta["requests"][i]["first_row"]
        for j, tok in enumerate(r["output"]):
            row = torch.from_numpy(rows[first + j].copy())
            assert rel_err(row, ref[len(r["prompt"]) - 1 + j]) <= tol("float32", "nvC")
            assert tok == int(torch.argmax(row))
    tight = subprocess.run(common + ["--num-pages", "11"], capture_output=True, text=True, timeout=300)
    assert tight.returncode == 0, tight.stderr[-3000:]
    assert "preemption" in tight.stderr
    assert [json.loads(ln)["output"] for ln in tight.stdout.strip().splitlines()] == [r["output"] for r in recs]


@pytest.mark.parametrize("mode", ["chunks", "mixed"])
def test_prompt_attention_on_the_matrix_cores_beside_single_tokens(netovik_dirs, mode, monkeypatch):
    """Steps in which a prompt's portion of 16 tokens and more stands beside other requests' single tokens and
    short portions, all run by the kernel for prompts (its threshold on a step's tokens lowered for the test)."""
    ops = _ops()
    monkeypatch.setattr(ops, "MIXED_ATTENTION_Q16_TOKENS", 16)
    model_dir = netovik_dirs["nvC"]
    reqs = requests_for("nvC", model_dir)
    steps = {"chunks": rl.trace_chunks, "mixed": rl.trace_mixed}[mode](reqs)
    assert any(max(len(e["tokens"]) for e in s["entries"]) >= 16 and len(s["entries"]) > (1 if mode == "mixed" else 0) for s in steps)
    ps = NETOVIK_PAGE["nvC"]
    runner = make_runner(model_dir, "bfloat16", ps, rl.max_live_tokens(steps, unit=ps) // ps)
    results = rl.run_steps_in_process(runner, steps)
    check(model_dir, reqs, steps, results, "bfloat16", "nvC")
