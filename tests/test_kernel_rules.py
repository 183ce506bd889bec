"""The host's rules between kernels: which steps the recurrences take in chunks on the matrix cores (the dispatch asks the kernels' own
rule, and what the rule refuses stays with the forms that have no such limit), when the draw forms the maxima of runs, and what the
sources' inline assembly keeps to."""
import glob
import os
import re
import types

import pytest
import torch

from tffinfer_amd.kernels import build


def _lib():
    from tffinfer_amd.kernels import lib
    return lib.load()


def test_wkv_chunks_up_to_what_a_launch_holds():
    L = _lib()
    for tokens, heads, fits in ((128, 64, 1), (16 * 65535 + 1, 64, 1), (1 << 30, 31, 1), (1 << 30, 32, 0), (1 << 30, 64, 0)):
        assert L.tff_wkv_chunks_supported(tokens, 3, heads, 64, 4096) == fits, tokens
    assert L.tff_wkv_chunks_supported(128, 65535, 1, 128, 4096) == 1 and L.tff_wkv_chunks_supported(128, 65536, 1, 128, 4096) == 0
    assert [L.tff_wkv_chunks_supported(128, 1, 1, D, 4096) for D in (48, 64, 96, 128, 256)] == [0, 1, 0, 1, 0]
    assert [L.tff_wkv_chunks_supported(128, 1, 1, 64, row) for row in (4098, (1 << 25) - 4, 1 << 25)] == [0, 1, 0]


def test_every_chunk_of_a_step_has_a_place_of_its_own():
    """The numbering that the chunks' kernels and their workspaces share: place t / 16 + r, T / 16 + R places, and the way back
    from a place to its request (the last one whose first place is not behind it)."""
    import random
    rng = random.Random(1)
    for _ in range(300):
        ns = [rng.choice((0, 1, 2, 15, 16, 17, 31, 32, 33, 96, rng.randrange(300))) for _ in range(rng.randrange(1, 150))]
        cu = [sum(ns[:i]) for i in range(len(ns) + 1)]
        seen = {}
        for r, n in enumerate(ns):
            for i in range(-(-n // 16)):
                place = (cu[r] + 16 * i) // 16 + r
                assert place == cu[r] // 16 + r + i and place not in seen and place < cu[-1] // 16 + len(ns)
                seen[place] = r
        for place, r in seen.items():
            assert sum(cu[q] // 16 + q <= place for q in range(len(ns))) - 1 == r


def test_gated_delta_chunks_up_to_32_bit_offsets():
    """Seventeen rows of channels in bytes stay under 2^32; the token-by-token form takes rows up to twice as long."""
    L = _lib()
    H, G, D = 2, 1, 64

    def bytes_of(E):
        return (2 * G * D + H * E + 2 * H) * 17 * 4
    for E in (64, 1 << 20, 31_580_000, 31_581_000, 40_000_000):
        assert L.tff_gdelta_chunks_supported(1, H, G, D, E, 4096) == (bytes_of(E) < 1 << 32 and E <= 16 * 65535), E
    H = 65534
    for E in (480, 960, 964, 1928):
        assert L.tff_gdelta_chunks_supported(1, H, G, D, E, 4096) == (bytes_of(E) < 1 << 32), E
    assert L.tff_gdelta_chunks_supported(65536, 2, 1, 64, 64, 4096) == 0 and L.tff_gdelta_chunks_supported(65535, 2, 1, 64, 64, 4096) == 1
    assert L.tff_gdelta_chunks_supported(1, 3, 1, 64, 64, 4096) == 0 and L.tff_gdelta_chunks_supported(1, 4, 2, 64, 64, 4098) == 0


@pytest.mark.parametrize("longest,chunks", [(127, False), (128, True), (16 * 65535, True), (16 * 65535 + 1, True), ((1 << 20) - 1, True)])
def test_wkv_dispatch_keeps_to_the_rule(monkeypatch, longest, chunks):
    """The op calls the entry for chunks exactly where the rule takes the step (the entries themselves are not run)."""
    from tffinfer_amd.kernels import ops
    real, called = _lib(), []

    class Library:
        def __getattr__(self, name):
            if name in ("tff_wkv_recurrence", "tff_wkv_recurrence_chunks"):
                return lambda *a: called.append(name) or 0
            return getattr(real, name)

    class OnGpu(torch.Tensor):
        is_cuda = True
    monkeypatch.setattr(ops._lib, "load", lambda: Library())
    monkeypatch.setattr(ops, "_req", lambda t, *a, **k: t)
    monkeypatch.setattr(ops, "_state_rows", lambda t, *a: t.shape[1])
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    H, D, T = 1, 64, 4
    r, k, v, z = (torch.zeros(T, H * D).as_subclass(OnGpu) for _ in range(4))
    i32 = torch.zeros(2, dtype=torch.int32)
    batch = types.SimpleNamespace(num_reqs=1, max_new_tokens=longest, host_cu_tokens=[0, longest], cu_tokens=i32, state_slots=i32)
    ops.wkv_recurrence(r, k, v, z, torch.zeros(H * D), torch.zeros(H * D), torch.zeros(1, H * D * D), batch, H, D)
    assert called == ["tff_wkv_recurrence_chunks" if chunks else "tff_wkv_recurrence"]


@pytest.mark.parametrize("lengths,starts,window,sixteen", [
    ([64], [0], 0, False), ([88], [0], 0, False), ([89], [0], 0, False), ([100], [0], 0, False), ([111], [0], 0, False), ([112], [0], 0, True), ([300], [0], 0, True), ([112], [0], 37, False),
    ([113], [0], 37, True), ([64], [1000], 0, True), ([64], [1000], 100, False), ([20] * 5, [0] * 5, 0, False), ([60] + [1] * 10, [0] + [900] * 10, 0, True),
    ([63], [5000], 0, False), ([15] * 40, [5000] * 40, 0, False)])
def test_short_prompts_of_mixed_heads_take_a_block_a_token(monkeypatch, lengths, starts, window, sixteen):
    """Sixteen queries a block from 64 tokens on, with an entry of 16 and more, where the tokens see enough keys; a batch that does not
    hold its contexts is taken to see all that a window lets it."""
    from tffinfer_amd.kernels import ops
    real, called = _lib(), []

    class Library:
        def __getattr__(self, name):
            if name in ("tff_mixed_attention", "tff_mixed_attention_q16"):
                return lambda *a: called.append(name) or 0
            return getattr(real, name)
    monkeypatch.setattr(ops._lib, "load", lambda: Library())
    monkeypatch.setattr(ops, "_req", lambda t, *a, **k: t)
    monkeypatch.setattr(ops, "_check_cache", lambda *a: None)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    H, G, D, page, T = 20, 5, 64, 16, sum(lengths)
    contexts = [s + n for s, n in zip(starts, lengths)]
    i32 = torch.zeros(max(T, len(lengths)), dtype=torch.int32)
    kv = types.SimpleNamespace(k_cache=torch.zeros(1, dtype=torch.bfloat16), v_cache=torch.zeros(1, dtype=torch.bfloat16), page_size=page,
                               block_tables=torch.zeros(len(lengths), -(-max(contexts) // page), dtype=torch.int32))
    batch = types.SimpleNamespace(token_req=i32, positions=i32, max_new_tokens=max(lengths), host_cu_tokens=[sum(lengths[:i]) for i in range(len(lengths) + 1)])
    q = torch.zeros(T, H * D, dtype=torch.bfloat16)
    ops.mixed_attention(q, H, G, D, kv, types.SimpleNamespace(max_context=max(contexts), **vars(batch)), 1.0, window=window)
    ops.mixed_attention(q, H, G, D, kv, batch, 1.0, window=window)
    blind = T >= 64 and max(lengths) >= 16 and (window == 0 or T > 112)
    assert called == ["tff_mixed_attention_q16" if x else "tff_mixed_attention" for x in (sixteen, blind)]
    if T in (88, 89) and max(contexts) < 100:                 # (more than one kv head a wave: up to 88 tokens)
        del called[:]
        ops.mixed_attention(q[:, :20 * 32].contiguous(), 20, 20, 32, kv, types.SimpleNamespace(max_context=T, **vars(batch)), 1.0)
        assert called == ["tff_mixed_attention_q16" if T == 89 else "tff_mixed_attention"]


@pytest.mark.parametrize("n,H,groups,levels,one", [
    (1, 4096, 2, 10, 1), (1, 4096, 2, 11, 0), (1, 4096, 1, 2, 0), (1, 2049, 1, 1, 0), (1, 2048, 1, 1, 1), (31, 4096, 2, 12, 0), (32, 4096, 2, 12, 1), (32, 4096, 2, 13, 0),
    (127, 4096, 2, 20, 0), (128, 4096, 2, 20, 1), (128, 4096, 2, 21, 0), (256, 4096, 2, 40, 1), (4000, 8192, 2, 2, 0), (4000, 8192, 4, 40, 1)])
def test_the_sum_over_depth_goes_with_a_norm_that_it_does_not_hold_up(n, H, groups, levels, one):
    """Not behind groups that a block reads more than once, nor over many levels of few rows."""
    assert _lib().tff_group_depth_in_norm(n, H, groups, levels) == one


@pytest.mark.parametrize("fits", [True, False])
def test_a_wkv_layer_asks_the_kernels_rule_for_its_four_products(monkeypatch, fits):
    """One packed weight where the rule takes it, else four: whatever the rule comes to be."""
    from tffinfer_amd.kernels import ops
    from tffinfer_amd.parts import wkv
    assert [ops.planes_supported(N, K) for N, K in ((128, 64), (4096, 4096), (64, 64), (192, 64), (128, 32), (128, 96))] == [True, True] + [False] * 4
    asked = []
    monkeypatch.setattr(ops, "planes_supported", lambda N, K: asked.append((N, K)) or fits)
    monkeypatch.setattr(wkv, "to_device", lambda t, dtype, device: t)
    monkeypatch.setattr(torch.Tensor, "to", lambda t, *a, **k: t)              # (nothing goes to a device here)
    mixer = wkv.WKVMixer(64, 2, 32, decay_rank=4)
    shapes = {name: spec.shape for name, spec in mixer.weight_specs().items()}
    mixer.load_weights({name: torch.zeros(shape) for name, shape in shapes.items()}, torch.bfloat16, "cuda:0")
    assert asked == [(64, 64)] and (mixer.w_four is not None) == fits and (mixer.w_each is None) == fits
    assert not fits or tuple(mixer.w_four.shape) == (256, 64)


@pytest.mark.parametrize("lengths,heads,dim,groups", [
    ([901], 32, 128, 1), ([901] + [1] * 63, 32, 128, 1), ([1] * 30 + [95, 500], 32, 128, 1), ([901, 400, 400], 32, 128, 1), ([2000] + [200] * 5, 32, 128, 1),
    ([901, 848, 677, 664], 32, 128, 2), ([500] * 6, 32, 128, 2), ([901, 848, 677, 664], 16, 128, 1), ([200] * 16, 16, 128, 2), ([200] * 16, 8, 128, 2),
    ([901, 848, 677, 664], 32, 64, 1), ([500] * 6, 32, 64, 2), ([901] * 8, 64, 128, 2), ([901], 200, 128, 2), ([901] * 6, 32, 256, 1)])
def test_the_delta_rules_scan_takes_two_groups_where_portions_would_wait(lengths, heads, dim, groups):
    """Not by the number of requests: those that decode, and portions that are through before a longer one, keep no block waiting."""
    from tffinfer_amd.kernels import ops
    cu = [sum(lengths[:i]) for i in range(len(lengths) + 1)]
    batch = types.SimpleNamespace(num_reqs=len(lengths), host_cu_tokens=cu)
    assert ops.gdelta_scan_groups(batch, heads, dim, dim, 512) == groups
    assert ops.gdelta_scan_groups(batch, heads, dim, 16, 512) == 1


def test_portions_start_in_turn_where_blocks_run():
    from tffinfer_amd.kernels.ops import _through
    assert _through([], 8, 16) == 0 and _through([5], 8, 16) == 5 and _through([5, 9], 8, 16) == 9
    assert _through([5, 9, 3], 8, 16) == 9 and _through([5, 9, 7], 8, 16) == 12 and _through([4, 4], 32, 16) == 16


def test_the_draw_forms_maxima_only_where_they_bound_something(monkeypatch):
    """A top_k over half the number of a row's runs (or 256) does not ask for them, nor does a small vocabulary; one row that
    profits is enough."""
    from tffinfer_amd.kernels import ops
    from tffinfer_amd.sampling.params import SamplingConfig
    from tffinfer_amd.sampling.sampler import Sampler
    assert [ops.sample_few_limit(V) for V in (1, 16383, 16384, 16385, 32768, 65536, 151936, 1 << 20)] == [0, 0, 64, 64, 128, 256, 256, 256]
    sampler = Sampler(torch.device("cpu"), types.SimpleNamespace(sample=lambda *a, few=False: few))
    monkeypatch.setattr(sampler, "_send", lambda columns: [torch.from_numpy(c) for c in columns])

    def asks(V, *ks):
        return sampler.sample_on_device(torch.zeros(len(ks), V), [SamplingConfig("random", temperature=1.0, top_k=k) for k in ks], [0] * len(ks))
    assert asks(16384, 64) and not asks(16384, 65) and not asks(16384, 0) and not asks(16000, 20)
    assert asks(32768, 128) and not asks(32768, 200, 256) and asks(32768, 200, 20)
    assert asks(151936, 256) and not asks(151936, 257)


@pytest.mark.parametrize("tiles,col_blocks", [(1, 1), (3, 2), (5, 3), (63, 3), (126, 6), (220, 4), (7, 8), (40, 11), (9, 16)])
def test_the_experts_blocks_cover_every_tile_and_load_the_xcds_alike(tiles, col_blocks):
    """Every (column block, tile) pair has one block of a launch for up to as many tiles and more; blocks go to the eight XCDs in turn:
    none has more than its eighth, and each walks neighbouring pairs."""
    L = _lib()
    for most in (tiles, tiles + 5):
        ids = [L.tff_experts_block(b, tiles, col_blocks) for b in range(-(-most * col_blocks // 8) * 8)]
        assert sorted(i for i in ids if i >= 0) == list(range(tiles * col_blocks))
        for x in range(8):
            own = [i for i in ids[x::8] if i >= 0]
            assert len(own) <= -(-tiles * col_blocks // 8) and own == list(range(own[0], own[0] + len(own)) if own else [])


@pytest.mark.parametrize("col_blocks", [1, 3, 16])
@pytest.mark.parametrize("counts", [[1], [3, 1, 8], [9, 16, 25], [2, 0, 17, 1]])
def test_an_experts_pairs_lie_together_and_cover_its_tiles(counts, col_blocks):
    """Pairs in order: an expert after the other, groups of up to eight of its tiles, all column blocks of a group, tiles fastest; the
    entry of tile id / col_blocks, which the kernels look up, is one of the same expert."""
    L = _lib()
    first = 0
    for n in counts:
        seen = [divmod(L.tff_experts_place(i, col_blocks, first, n), col_blocks) for i in range(first * col_blocks, (first + n) * col_blocks)]
        want = [(first + t, c) for g in range(0, n, 8) for c in range(col_blocks) for t in range(g, min(n, g + 8))]
        assert seen == want
        assert all(first <= i // col_blocks < first + n for i in range(first * col_blocks, (first + n) * col_blocks))
        first += n


def test_loads_into_lds_leave_a_wait_state_behind_m0():
    """A load into LDS takes its LDS address from M0 and may follow the scalar instruction that writes it one wait state later at the earliest.
    The compiler does not look into inline assembly, so every piece of it that writes M0 has an instruction between the two."""
    pieces = 0
    for path in sorted(glob.glob(os.path.join(build.CSRC_DIR, "*.h")) + glob.glob(os.path.join(build.CSRC_DIR, "*.hip"))):
        with open(path) as f:
            for text in re.findall(r'asm volatile\(((?:\s*"[^"]*")+)', f.read()):
                lines = "".join(re.findall(r'"([^"]*)"', text)).replace("\\t", "").split("\\n")
                for first, second in zip(lines, lines[1:]):
                    if re.match(r"s_\w+ m0,", first):
                        pieces += 1
                        assert "_lds_" not in second, (os.path.basename(path), lines)
                assert "_lds_" not in lines[0], (os.path.basename(path), lines)      # (M0 is written beside its load)
    assert pieces >= 7, pieces


def test_products_whose_weights_stream_wants_more_blocks_split_k():
    """Some hundred rows of a weight that comes from memory: fewer columns of tiles than keep it coming split K.  Kept sums, up to 64
    rows, long products and K in no units of 64 have plans of their own."""
    import ctypes
    L = _lib()

    def plan(M, N, K, glu=0, keep=0):
        r, c, s = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
        assert L.tff_gemm_plan(M, N, K, glu, keep, ctypes.byref(r), ctypes.byref(c), ctypes.byref(s)) == 0
        return r.value, c.value, s.value

    assert plan(110, 6144, 2560) == (128, 128, 4) and plan(78, 6144, 2560, glu=1) == (64, 128, 2)
    assert plan(202, 6144, 4096) == plan(330, 4096, 4096) == (128, 128, 2)
    assert plan(110, 6144, 2560, keep=1)[2] > 1 and plan(60, 6144, 2560) == (64, 128, 4)
    assert plan(16384, 24576, 4096, glu=1) == (256, 256, 1) and plan(2048, 6144, 4096) == (256, 192, 1)


def test_an_activation_counts_the_kernel_that_adds_up_the_parts():
    """With an activation behind it a product in one part has the kernel that adds up the parts as well, so that two parts may be the
    sooner; the room that is asked for is that plan's."""
    L = _lib()
    for M, N, K, parts in ((200, 18432, 4096, 2), (128, 12288, 4096, 2), (90, 9216, 2048, 2), (1055, 4096, 4096, 2), (333, 512, 192, 1), (16, 18432, 4096, 0), (2048, 18432, 4096, 0)):
        assert L.tff_gemm_unary_workspace_bytes(M, N, K) == parts * M * N * 4, (M, N, K)
        assert L.tff_gemm_takes_unary(M, N, K) == (parts > 0 or M <= 16)


def _plan(M, N, K, glu=0, keep=0):
    import ctypes
    r, c, s = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    assert _lib().tff_gemm_plan(M, N, K, glu, keep, ctypes.byref(r), ctypes.byref(c), ctypes.byref(s)) == 0
    return r.value, c.value, s.value


def test_few_gated_rows_go_on_tiles_by_how_these_fill_the_cus():
    """Not by the number of the weight's elements alone: nine rows and more on tiles that fill three quarters of one round, else the stream."""
    for N, K in ((28672, 8192), (27648, 5120), (24576, 2048), (24576, 4096), (51200, 5120)):
        assert _plan(9, N, K, 1)[0] == _plan(16, N, K, 1)[0] == 32, (N, K)
        assert _plan(8, N, K, 1)[0] == (32 if N * K >= 2.4e8 else 0), (N, K)
    # half a round of tiles and less, a second round, K in no units of 64
    for N, K in ((8192, 12288), (22016, 8192), (34816, 5120), (16384, 8192), (73728, 4096), (28672, 8200)):
        assert _plan(9, N, K, 1) == _plan(16, N, K, 1) == (0, 0, 1), (N, K)


def test_parts_of_k_pay_for_the_kernel_that_adds_them_up():
    """Products of some hundred rows and a short K stay whole; sums kept for a norm are cut as finely as the norm's reads of the parts allow, and few columns
    of many rows too."""
    assert _plan(68, 4096, 1024) == _plan(90, 4096, 1024) == (64, 128, 1)
    assert _plan(107, 512, 768)[2] == _plan(78, 640, 832)[2] == 1
    assert _plan(116, 2048, 2048, keep=1) == (64, 128, 4)
    assert _plan(2219, 128, 15424, keep=1)[2] == 8 and _plan(2210, 4096, 18432, keep=1)[2] <= 2


def test_parts_of_k_in_threes_fit_the_cus_of_every_xcd():
    """An XCD takes an eighth of the tiles in all their parts: blocks that are no more than the CUs may still be more than one XCD's CUs, a second round."""
    for M, N, K in ((160, 8064, 14144), (303, 3584, 15232), (411, 10496, 13120), (382, 896, 6144)):
        assert _plan(M, N, K, keep=1)[2] % 3 != 0, (M, N, K)
    seen = 0
    for M in range(130, 1025, 37):
        for N in range(512, 8193, 384):
            for K in (N, 9728, 14144):
                rows, cols, parts = _plan(M, N, K, keep=1)
                tiles = -(-M // rows) * -(-N // cols)
                if parts % 3 == 0 and rows > 64 and tiles * parts <= 256:
                    seen += 1
                    assert -(-tiles // 8) * parts <= 32, (M, N, K, rows, cols, parts)
    assert seen > 50


def test_gated_products_of_some_hundred_rows_are_bound_by_their_weights_stream():
    """A gated weight of 200 MB is bound by its stream: two parts of K do not make it faster, and cost their sums."""
    for M in (65, 70, 139, 145, 160, 200):
        assert _plan(M, 24576, 4096, 1)[2] == 1, M


def test_an_activation_keeps_the_float32_sums_that_it_had():
    """Products in more parts of K before an activation, which would be in one by the constants of products without: plans of their own."""
    L = _lib()
    for M, N, K in ((666, 9216, 5120), (1507, 3072, 2048), (523, 9920, 3840), (8651, 6080, 14912), (8941, 512, 2048)):
        assert L.tff_gemm_takes_unary(M, N, K) == 1, (M, N, K)
