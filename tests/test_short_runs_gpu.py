"""Decode attention of short rows: a run a row, its keys among a block's eight waves."""
import math

import numpy as np
import pytest
import torch

from test_kernels_gpu import ATTN_TOL, DEV, _attn_ref, _close, _fake_step, _ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nq,nkv,d,ps,window", [(16, 8, 128, 16, 0), (32, 8, 128, 8, 0), (8, 2, 32, 8, 300), (16, 4, 64, 128, 0), (14, 7, 112, 32, 100)])
def test_short_rows_on_a_block_of_waves(nq, nkv, d, ps, window):
    """One step and as many as the waves, one more and less, up to the most a short row has and beyond it (the run is the row whatever its
    length); tables narrower and wider than the 64 pages asked for early; runs that are not in use behind the rows'."""
    ops = _ops()
    from tffinfer_amd.kernels.key_runs import max_key_runs
    lengths = [0, 1, 30, 31, 32, 63, 64, 100, 223, 224, 255, 256, 257, 447, 480, 500, 511, 512, 640, 703, 767, 768, 1100]
    entries = [(P, 1) for P in lengths]
    batch, kv, ks, vs, positions, _ = _fake_step(entries, ps, nkv, d, torch.bfloat16, seed=d + ps)
    R = len(entries)
    g = torch.Generator().manual_seed(11)
    qkv = torch.randn(R, (nq + 2 * nkv) * d, generator=g).to(torch.bfloat16)
    q = qkv[:, :nq * d].reshape(R, nq, d)
    k_new = qkv[:, nq * d:(nq + nkv) * d].reshape(R, nkv, d)
    v_new = qkv[:, (nq + nkv) * d:].reshape(R, nkv, d)
    bt = kv.block_tables.cpu()
    slots = torch.tensor([int(bt[r, P // ps]) * ps + P % ps for r, P in enumerate(lengths)], dtype=torch.int32, device=DEV)
    slots[4] = -1           # a row that writes no key reads what its page holds
    scale = 1 / math.sqrt(d)
    ref = torch.stack([_attn_ref(q[r:r + 1], torch.cat([ks[r][:P], k_new[r:r + 1]]), torch.cat([vs[r][:P], v_new[r:r + 1]]), positions[r:r + 1],
                                 window, scale)[0] for r, P in enumerate(lengths)])
    cap = max_key_runs(R, nkv)
    runs = np.full((cap, 4), -1, dtype=np.int32)
    for r, P in enumerate(lengths):
        runs[r] = (r, max(0, P - window + 1) // 32 * 32 if window else 0, P + 1, P)
    out = ops.attention_decode_fused(qkv.to(DEV), nq, nkv, d, None, None, 1e-6, None, 0, kv, batch, window, scale, slot_mapping=slots,
                                     key_runs=torch.from_numpy(runs).to(DEV), run_start=torch.arange(R + 1, dtype=torch.int32, device=DEV),
                                     runs_for_blocks=False, runs_merge=False)
    live = [r for r in range(R) if r != 4]
    _close(out.reshape(R, nq, d)[live], ref[live], ATTN_TOL, "short rows")
    for r, P in enumerate(lengths):
        if r != 4:
            page, at = int(bt[r, P // ps]), P % ps
            assert torch.equal(kv.k_cache[page, :, at].cpu(), k_new[r]) and torch.equal(kv.v_cache[page, :, :, at].cpu(), v_new[r]), r
    same = ops.attention_decode_fused(qkv.to(DEV), nq, nkv, d, None, None, 1e-6, None, 0, kv, batch, window, scale)
    _close(out.reshape(R, nq, d)[live], same.reshape(R, nq, d).double().cpu()[live], ATTN_TOL, "against keys split alike")


@pytest.mark.parametrize("nq,nkv,d,R", [(16, 8, 128, 13), (8, 2, 32, 24), (6, 3, 256, 9), (32, 32, 64, 11)])
def test_rows_of_one_run_each_in_any_order(nq, nkv, d, R):
    """A run's own number says whose it is: runs in another order than the rows', with runs that are not in use in front, between and behind,
    give the bits of runs in order.  Blocks of eight waves and (more pairs than CUs, heads of 256) single waves."""
    ops = _ops()
    ps = 16
    lengths = [(97 * r + 5) % 700 for r in range(R)]
    batch, kv, _, _, _, _ = _fake_step([(P, 1) for P in lengths], ps, nkv, d, torch.bfloat16, seed=R)
    qkv = torch.randn(R, (nq + 2 * nkv) * d, generator=torch.Generator().manual_seed(R)).to(torch.bfloat16).to(DEV)
    bt = kv.block_tables.cpu()
    slots = torch.tensor([int(bt[r, P // ps]) * ps + P % ps for r, P in enumerate(lengths)], dtype=torch.int32, device=DEV)
    start = torch.arange(R + 1, dtype=torch.int32, device=DEV)
    order = np.random.default_rng(R).permutation(R)

    def run(rows_at):
        runs = np.full((64, 4), -1, dtype=np.int32)
        for at, r in rows_at:
            runs[at] = (r, 0, lengths[r] + 1, lengths[r])
        return ops.attention_decode_fused(qkv, nq, nkv, d, None, None, 1e-6, None, 0, kv, batch, 0, 1 / math.sqrt(d), slot_mapping=slots,
                                          key_runs=torch.from_numpy(runs).to(DEV), run_start=start, runs_for_blocks=False, runs_merge=False)

    want = run([(r, r) for r in range(R)])
    assert torch.equal(run([(i, int(r)) for i, r in enumerate(order)]), want)
    assert torch.equal(run([(2 * i + 1 + (i > 4) * 9, int(r)) for i, r in enumerate(order)]), want)
