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
    """A pair of groups a CU or less, short and long K of wider weights."""
    ops = _ops()
    g = torch.Generator(device=DEV).manual_seed(I + K)
    x = torch.randn(16, K, generator=g, device=DEV).bfloat16()
    gate, up = (torch.randn(I, K, generator=g, device=DEV).mul_(K ** -0.5).bfloat16() for _ in range(2))
    a, b = x.double() @ gate.double().T, x.double() @ up.double().T
    ref = a * torch.sigmoid(a) * b
    pw = ops.pack_gate_up(gate, up)
    for m in ROWS:
        # (scores around 1: silu's derivative is at most 1.1, |up| and |gate| stay below 6, and the exponential is within 2^-21 of its argument's size)
        _close(ops.linear(x[:m], pw, out_dtype=torch.float32), ref[:m], K, K ** -0.5 * 14 + 2.0, f"{m} rows")


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
