"""The streaming bfloat16 product of up to 16 rows: what a load packs, units of 128 k dealt to the waves, ends of K."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
ROWS = (1, 3, 4, 5, 8, 9, 16)


def _ops():
    from tffinfer_amd.kernels import ops
    return ops


def _close(got, ref, K, scale, what):
    """Float32 sums of K products in runs on the matrix cores: within (K / 8 + 8) roundings of the terms' root mean square, sqrt(K) terms' worth."""
    bound = 2.0 ** -24 * (K / 8 + 8) * K ** 0.5 * scale * 4
    err = float((got.double() - ref).abs().max())
    assert err <= bound, f"{what}: {err:.3e} > {bound:.3e}"


# up to 256 groups of 16 columns: eight waves, two units of K each in flight; more: four waves, one group a block or two; K of less than a step, no whole
# unit, as many units as waves and one more or less, several rounds with every remainder
@pytest.mark.parametrize("N,K", [(40, 8), (16, 40), (304, 128), (4096, 1016), (4090, 1032), (1000, 2048), (520, 3080), (2050, 4104), (4104, 136), (4112, 640),
                                 (5000, 1160), (7168, 2056), (8200, 520), (24592, 2568)])
def test_rows_of_every_number(N, K):
    """Against 64 bits, the rows strided and one of them not finite; a row's bits do not depend on how many there are."""
    ops = _ops()
    g = torch.Generator(device=DEV).manual_seed(N + K)
    x = torch.randn(16, K + 24, generator=g, device=DEV).bfloat16()[:, :K]
    w = torch.randn(N, K, generator=g, device=DEV).bfloat16()
    pw = ops.pack_weight(w)
    ref = x.double() @ w.double().T
    whole = ops.linear(x, pw, out_dtype=torch.float32)
    _close(whole, ref, K, 1.0, "sixteen rows")
    for once in (0, 1):
        pw.once = once
        for m in ROWS:
            assert torch.equal(ops.linear(x[:m], pw, out_dtype=torch.float32), whole[:m]), m
    y = x.clone()
    y[2, K // 2] = float("nan")
    got = ops.linear(y[:5], pw, out_dtype=torch.float32)
    assert got[2].isnan().all() and torch.equal(got[[0, 1, 3, 4]], whole[[0, 1, 3, 4]])


@pytest.mark.parametrize("I,K", [(100, 192), (4096, 1032), (4100, 520), (6000, 1920), (4200, 2568), (9000, 2184)])
def test_gated_rows_of_every_number(I, K):
    """A pair of groups a CU or less, short and long K of wider weights.  A row's bits do not depend on how many there are but where the waves that share
    K change: from nine rows on, with more than four groups a CU and K of 2,048 and more."""
    ops = _ops()
    g = torch.Generator(device=DEV).manual_seed(I + K)
    x = torch.randn(16, K, generator=g, device=DEV).bfloat16()
    gate, up = (torch.randn(I, K, generator=g, device=DEV).mul_(K ** -0.5).bfloat16() for _ in range(2))
    a, b = x.double() @ gate.double().T, x.double() @ up.double().T
    silu = a * torch.sigmoid(a)
    # Sums of about 1 whose (K / 8 + 8) roundings of at most 2^-24 are independent: four times their root.  silu's derivative is at most 1.1; the exponential
    # and the quotient are within 2^-20 of the result.
    bound = 2.0 ** -24 * 4 * (K / 8 + 8) ** 0.5 * (1.1 * b.abs() + silu.abs() + 1) + 2.0 ** -20 * (silu * b).abs()
    pw = ops.pack_gate_up(gate, up)
    outs = {m: ops.linear(x[:m], pw, out_dtype=torch.float32) for m in ROWS}
    for m, out in outs.items():
        over = (out.double() - silu[:m] * b[:m]).abs() / bound[:m]
        assert float(over.max()) <= 1, f"{m} rows: {float(over.max()):.2f} times the bound"
        same = 16 if I <= 8192 or K < 2048 or m > 8 else 8
        assert torch.equal(out, outs[same][:m]), m


# one and two waves a block: K of less than a unit, ragged units, every number of them up to the last that few waves share, and one more; columns that
# end within a group
@pytest.mark.parametrize("N,K", [(16404, 40), (16400, 128), (18000, 520), (16600, 896), (16600, 904), (8200, 72), (8210, 1016), (12000, 1024), (16000, 1032), (4100, 1000),
                                 (4090, 136), (4000, 256), (700, 264)])
def test_short_inner_sizes_on_few_waves(N, K):
    ops = _ops()
    g = torch.Generator(device=DEV).manual_seed(N + K)
    x = torch.randn(16, K + 8, generator=g, device=DEV).bfloat16()[:, :K]
    w = torch.randn(N, K, generator=g, device=DEV).bfloat16()
    bias = torch.randn(-(-N // 16) * 16, generator=g, device=DEV)
    pw = ops.pack_weight(w)
    ref = x.double() @ w.double().T
    whole = ops.linear(x, pw, out_dtype=torch.float32)
    _close(whole, ref, K, 1.0, "sixteen rows")
    for once in (0, 1):
        pw.once = once
        for m in ROWS:
            assert torch.equal(ops.linear(x[:m], pw, out_dtype=torch.float32), whole[:m]), m
        _close(ops.linear(x, pw, out_dtype=torch.float32, bias=bias), ref + bias[:N].double(), K, 2.0, "with a bias")


@pytest.mark.parametrize("I,K", [(40, 72), (4096, 512), (4100, 264), (8192, 136), (8200, 1064), (12864, 2112), (12864, 2056)])
@pytest.mark.parametrize("scaled", [False, True])
def test_gated_widths_on_few_waves(I, K, scaled):
    """Gated products on two waves a block, eight and four, on either side of the lines, with and without the rows' factors."""
    ops = _ops()
    g = torch.Generator(device=DEV).manual_seed(I + K)
    gate, up = (torch.randn(I, K, generator=g, device=DEV).mul_(K ** -0.5).bfloat16() for _ in range(2))
    pw = ops.pack_gate_up(gate, up)
    rows = torch.randn(16, K, generator=g, device=DEV).bfloat16()
    for m in (3, 8, 9, 16):
        x, factor = rows[:m], torch.ones(m, 1, dtype=torch.float64, device=DEV)
        if scaled:
            w1 = torch.randn(K, 64, generator=g, device=DEV).mul_(0.125).bfloat16()
            stream = torch.randn(m, K, generator=g, device=DEV)
            p = ops.linear(torch.randn(m, 64, generator=g, device=DEV).bfloat16(), ops.pack_weight(w1), out_dtype=torch.float32, partials=True)
            x = ops.add_rmsnorm(stream, p, torch.ones(K, device=DEV), 1e-6, torch.bfloat16, for_linear=True)
            assert isinstance(x, ops.ScaledRows)
            factor = 1 / torch.sqrt((stream.double() ** 2).mean(-1, keepdim=True) + 1e-6)
        v = (x.x if scaled else x).double()
        a, b = factor * (v @ gate.double().T), factor * (v @ up.double().T)
        silu = a * torch.sigmoid(a)
        # (as above; the factor's own sum and square root are within 2^-21 of it)
        bound = 2.0 ** -24 * (4 * (K / 8 + 8) ** 0.5 + 8) * (1.1 * b.abs() + silu.abs() + 1) * 2 + 2.0 ** -19 * (silu * b).abs()
        over = (ops.linear(x, pw, out_dtype=torch.float32).double() - silu * b).abs() / bound
        assert float(over.max()) <= 1, f"{m} rows: {float(over.max()):.2f} times the bound"


def _us(fn):
    """The best of some runs of twenty calls in a graph."""
    fn(0)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for i in range(20):
            fn(i)
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    best = 1e9
    for _ in range(8):
        ev[0].record()
        graph.replay()
        ev[1].record()
        ev[1].synchronize()
        best = min(best, ev[0].elapsed_time(ev[1]) * 50)
    return best


def test_rows_beyond_eight_do_not_halve_the_rate():
    """Sixteen rows' registers leave a SIMD fewer waves: with a short K and many columns, and with a gated product that takes no factors, 9 to 16 rows took
    half as long again as eight (9.9 and 6.6 us, 29.6 and 20.1; 4.8 and 4.0, 24.1 and 20.1)."""
    ops = _ops()
    pw = ops.pack_weight(torch.randn(59520, 64, device=DEV).bfloat16())
    x = torch.randn(16, 64, device=DEV).bfloat16()
    eight, twelve = (_us(lambda i, m=m: ops.linear(x[:m], pw)) for m in (8, 12))
    assert twelve <= 1.35 * eight, (eight, twelve)
    I, K = 12864, 2056
    weights = [ops.pack_gate_up(*(torch.randn(I, K, device=DEV).mul_(K ** -0.5).bfloat16() for _ in range(2))) for _ in range(8)]
    for w in weights:
        w.once = 1
    x = torch.randn(16, K, device=DEV).bfloat16()
    eight, sixteen = (_us(lambda i, m=m: ops.linear(x[:m], weights[i % 8])) for m in (8, 16))
    assert sixteen <= 1.35 * eight, (eight, sixteen)


@pytest.mark.parametrize("M", [1, 4, 5, 9, 16])
@pytest.mark.parametrize("H,K,N", [(1032, 264, 4096), (5128, 520, 4400), (5136, 1160, 520)])
def test_factors_of_rows_whose_norm_is_split(M, H, K, N):
    """The sums of squares of a row's groups: less than a wave's load of them, more, and no multiple of four."""
    ops = _ops()
    g = torch.Generator(device=DEV).manual_seed(M + H)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    w1 = torch.randn(H, K, generator=g, device=DEV).mul_(K ** -0.5).bfloat16()
    w2 = torch.randn(N, H, generator=g, device=DEV).bfloat16()
    resid = torch.randn(M, H, generator=g, device=DEV)
    nw = 1 + 0.1 * torch.randn(H, generator=g, device=DEV)
    p = ops.linear(x, ops.pack_weight(w1), out_dtype=torch.float32, partials=True)
    stream = resid.clone()
    rows = ops.add_rmsnorm(stream, p, nw, 1e-6, torch.bfloat16, for_linear=True)
    assert isinstance(rows, ops.ScaledRows)
    s = resid.double() + x.double() @ w1.double().T
    _close(stream, s, K, K ** -0.5 + 8.0 * K ** -0.5, "the stream")
    ref = rows.x.double() @ w2.double().T / torch.sqrt((s * s).mean(-1, keepdim=True) + 1e-6)
    _close(ops.linear(rows, ops.pack_weight(w2), out_dtype=torch.float32), ref, H, 2.0, "the product after the norm")
