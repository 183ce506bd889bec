"""The pinned buffers that a step's tables leave through, with the device several steps behind the host."""
import random

import pytest
import torch

pytestmark = pytest.mark.gpu


def keep_busy():
    """Some tens of milliseconds of work on the current stream."""
    a = torch.ones(8192, 8192, dtype=torch.bfloat16, device="cuda")
    for _ in range(24):
        torch.mm(a, a)


def test_buffers_go_round_behind_a_busy_device():
    """Eleven copies of patterns of their own, more than there are buffers, queued behind work that takes longer than the host
    needs for them; one is too long for the buffers and makes them grow in between."""
    from tffinfer_amd.engine.batch import PinnedTables
    p = PinnedTables(64)
    sizes = [50, 64, 1, 64, 33, 64, 5000, 9, 6000, 64, 10001]
    dev = [torch.zeros(n, dtype=torch.int32, device="cuda") for n in sizes]
    torch.cuda.synchronize()
    keep_busy()
    for k, (n, d) in enumerate(zip(sizes, dev)):
        host = p.take(n)
        assert host.numel() == n and host.is_pinned()
        host.copy_(torch.arange(n, dtype=torch.int32) * 16 + k)
        d.copy_(host, non_blocking=True)
        p.copied()
    torch.cuda.synchronize()
    for k, (n, d) in enumerate(zip(sizes, dev)):
        assert torch.equal(d.cpu(), torch.arange(n, dtype=torch.int32) * 16 + k), k


def test_decode_graphs_ahead_of_the_device(model_dirs):
    """Decode steps through a graph whose requests come, go and come back under the same id: launched behind a busy device and one at
    a time, the same bits.  A step's tables are written where they leave from: nothing of their size is copied on the host."""
    from tffinfer_amd import EngineOptions, LLMEngine
    from tffinfer_amd.engine.batch import StepEntry

    def run(wait):
        eng = LLMEngine.from_model_dir(model_dirs["A"], EngineOptions(dtype="bfloat16", page_size=8, num_pages=64, max_num_seqs=4,
                                                                      max_num_batched_tokens=64))
        rn, rng, out = eng.runner, random.Random(3), []
        assert rn._graph_buckets
        live, steps = [], 0

        def step(entries):
            out.append(rn.step(entries).clone())
            if wait:
                torch.cuda.synchronize()

        def come(r):
            rn.add_request(r)
            step([StepEntry(r, [rng.randrange(1, 100) for _ in range(rng.randrange(2, 30))], [0])])
            live.append(r)
        for r in range(4):
            come(r)
        if not wait:
            keep_busy()
        while steps < 40:
            step([StepEntry(r, [rng.randrange(1, 100)], [0]) for r in live])
            steps += 1
            if steps % 5 == 0:                       # (one leaves; the next time it comes back as another's pages have moved)
                gone = live.pop(rng.randrange(len(live)))
                rn.free_request(gone)
                if steps % 10 == 0:
                    come(gone)
            if len(live) < 3:
                come(next(r for r in range(4) if r not in live))
        torch.cuda.synchronize()
        for g in rn._graphs.values():
            assert torch.from_numpy(g.tables.hv).is_pinned()
        return out

    one, many = run(True), run(False)
    assert len(one) == len(many)
    for a, b in zip(one, many):
        assert torch.equal(a, b)
