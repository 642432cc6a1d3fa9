"""Each HIP kernel alone against its plain reference, at sizes other than the engine's."""
import ctypes
import math

import pytest
import torch

from tests import plain

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
DTYPES = [torch.float32, torch.bfloat16]


def K():
    from tensorline_amd.ops import kernels
    return kernels


def tol(dtype, f32=1e-5, bf16=2e-2):
    return dict(atol=f32, rtol=f32) if dtype == torch.float32 else dict(atol=bf16, rtol=bf16)


@pytest.mark.parametrize("dtype", DTYPES)
def test_embed(dtype):
    torch.manual_seed(0)
    table = torch.randn(1000, 192, device=DEV).to(dtype)
    ids = torch.tensor([0, 999, 5, 5, 17], dtype=torch.int32, device=DEV)
    x = K().embed(ids, table)
    assert x.dtype == torch.float32
    torch.testing.assert_close(x, table[ids.long()].float(), atol=0, rtol=0)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("T", [1, 5, 64])
def test_add_rmsnorm_reference_vector(dtype, T):
    # sizes of the reference's own test: H=896, eps=1e-6, w ~ U(0.5, 1.5) (tests/test_quant.py:100-113)
    torch.manual_seed(0)
    H, eps = 896, 1e-6
    w = torch.empty(H, device=DEV).uniform_(0.5, 1.5)
    x = torch.randn(T, H, device=DEV)
    r = torch.randn(T, H, device=DEV).to(dtype)
    want_x = x + r.float()
    want = plain.rmsnorm(want_x.double(), w.double(), eps)
    got = K().add_rmsnorm(x, r, w, eps, dtype)
    torch.testing.assert_close(x, want_x, atol=0, rtol=0)          # updated in place, exactly
    torch.testing.assert_close(got.double(), want, **tol(dtype, 2e-6, 2e-2))
    # no residual, odd width, rows picked
    H2 = 193
    x2 = torch.randn(7, H2, device=DEV)
    w2 = torch.randn(H2, device=DEV)
    keep = x2.clone()
    got2 = K().add_rmsnorm(x2, None, w2, 1e-5, dtype)
    torch.testing.assert_close(x2, keep, atol=0, rtol=0)
    torch.testing.assert_close(got2.double(), plain.rmsnorm(keep.double(), w2.double(), 1e-5), **tol(dtype, 2e-6, 2e-2))
    rows = torch.tensor([6, 0, 3], dtype=torch.int32, device=DEV)
    r2 = torch.randn(7, H2, device=DEV).to(dtype)
    got3 = K().add_rmsnorm(x2, r2, w2, 1e-5, dtype, rows=rows)
    torch.testing.assert_close(x2, keep, atol=0, rtol=0)            # with rows, x is left alone
    want3 = plain.rmsnorm((keep + r2.float())[rows.long()].double(), w2.double(), 1e-5)
    torch.testing.assert_close(got3.double(), want3, **tol(dtype, 2e-6, 2e-2))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M", [1, 3, 16, 17, 64, 130])
@pytest.mark.parametrize("N,Kd", [(176, 64), (1000, 192), (64, 100), (3, 7)])
def test_linear(dtype, M, N, Kd):
    torch.manual_seed(M * 1000 + N)
    a = torch.randn(M, Kd, device=DEV).to(dtype)
    w = (torch.randn(N, Kd, device=DEV) / math.sqrt(Kd)).to(dtype)
    b = torch.randn(N, device=DEV)
    want = a.double() @ w.double().T + b.double()
    got = K().linear(a, w, b)
    assert got.dtype == dtype
    torch.testing.assert_close(got.double(), want, **tol(dtype, 1e-5, 3e-2))
    got32 = K().linear(a, w, None, out_dtype=torch.float32)
    torch.testing.assert_close(got32.double(), a.double() @ w.double().T, **tol(dtype, 1e-5, 1e-5))


@pytest.mark.parametrize("H", [896, 193, 3584])
def test_add_rmsnorm_takes_a_product_in_its_shares(H):
    """A residual given as the K shares of a product: the shares are added in order, then to x; the
    result has the bits of adding them first."""
    torch.manual_seed(H)
    T, eps = 37, 1e-6
    w = torch.empty(H, device=DEV).uniform_(0.5, 1.5)
    for P in (2, 3):
        x = torch.randn(T, H, device=DEV)
        x2 = x.clone()
        parts = torch.randn(P, T, H, device=DEV)
        got = K().add_rmsnorm(x, K().ShareSum(parts), w, eps, torch.bfloat16)
        want = K().add_rmsnorm(x2, parts.sum(0), w, eps, torch.bfloat16)
        torch.testing.assert_close(x, x2, atol=0, rtol=0)
        torch.testing.assert_close(got, want, atol=0, rtol=0)
        rows = torch.tensor([5, 0, 36], dtype=torch.int32, device=DEV)
        got_r = K().add_rmsnorm(x, K().ShareSum(parts), w, eps, torch.float32, rows=rows)
        want_r = K().add_rmsnorm(x2, parts.sum(0), w, eps, torch.float32, rows=rows)
        torch.testing.assert_close(got_r, want_r, atol=0, rtol=0)


def test_linear_many_rows_keeps_its_shares_on_request():
    """A many-row product with a long K and few output tiles runs as shares of K: on request they
    come back unsummed, and their sum is the product."""
    torch.manual_seed(3)
    M, N, Kd = 256, 512, 9216
    a = torch.randn(M, Kd, device=DEV).to(torch.bfloat16)
    w = (torch.randn(N, Kd, device=DEV) / math.sqrt(Kd)).to(torch.bfloat16)
    want = a.double() @ w.double().T
    whole = K().linear(a, w, None, out_dtype=torch.float32)
    kept = K().linear(a, w, None, out_dtype=torch.float32, keep_shares=True)
    assert isinstance(kept, K().ShareSum) and kept.parts.shape[1:] == (M, N) and kept.parts.shape[0] > 1
    torch.testing.assert_close(kept.sum(), whole, atol=0, rtol=0)
    torch.testing.assert_close(whole.double(), want, atol=2e-3, rtol=2e-3)
    # a product that is not cut into shares comes back as a tensor either way
    small = K().linear(a[:, :1024].contiguous(), w[:, :1024].contiguous(), None, out_dtype=torch.float32, keep_shares=True)
    assert isinstance(small, torch.Tensor)


@pytest.mark.parametrize("tile", range(7))
@pytest.mark.parametrize("M,N,Kd,shares", [(65, 36, 64, 1), (257, 272, 128, 2), (129, 516, 320, 1), (200, 96, 832, 3), (1, 4, 192, 1), (193, 260, 1024, 4)])
def test_many_row_product_in_every_tile(tile, M, N, Kd, shares):
    """Every tile of the many-row product at the edges of tiles, with one step of K and fewer steps than stages, in shares,
    rows with a stride, columns that are no whole block; bias and activation behind the sum.  The products of bfloat16 numbers are
    exact in float, so a sum of K of them is off by at most K 2^-24 of the sum of their sizes."""
    torch.manual_seed(tile)
    a = torch.randn(M, Kd + 24, device=DEV).to(torch.bfloat16)[:, :Kd]
    w = (torch.randn(N, Kd, device=DEV) / math.sqrt(Kd)).to(torch.bfloat16)
    bias = torch.randn(N, device=DEV)
    sh = K().shuffle_weight(w)
    want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    run = lambda b, dt, **kw: K()._tiles(a, sh, b, dt, M, N, Kd, a.stride(0), shares * 256 + tile, **kw)
    err = (Kd + shares) * 2.0 ** -24 * size
    assert bool(((run(None, torch.float32).double() - want).abs() <= err).all())
    with_bias = want + bias.double()
    assert bool(((run(bias, torch.float32).double() - with_bias).abs() <= err + 2.0 ** -24 * with_bias.abs()).all())
    got, relu2 = run(bias, torch.bfloat16, act=1).double(), with_bias.clamp_min(0) ** 2      # (the square doubles what its argument is off by)
    assert bool(((got - relu2).abs() <= 2.0 ** -8 * relu2 + 2.1 * with_bias.abs() * err + 1e-6).all())
    kept = run(None, torch.float32, keep_shares=True)
    if shares > 1:
        assert isinstance(kept, K().ShareSum) and kept.parts.shape == (shares, M, N)
        torch.testing.assert_close(kept.sum(), run(None, torch.float32), atol=0, rtol=0)
    if tile == 1 or shares > 1:                                       # (a wave of that tile has three blocks of columns: no pairs)
        return
    for I in (16, 80):
        w = (torch.randn(2 * I, Kd, device=DEV) / math.sqrt(Kd)).to(torch.bfloat16)
        both = a.double() @ w.double().T
        for act, fn in ((0, torch.nn.functional.silu), (2, lambda z: torch.nn.functional.gelu(z, approximate="tanh"))):
            got = K()._tiles(a, K().shuffle_weight(w), None, torch.bfloat16, M, 2 * I, Kd, a.stride(0), 256 + tile, gated=True, act=act)
            want_g = fn(both[:, :I]) * both[:, I:]
            torch.testing.assert_close(got.double(), want_g, rtol=2.0 ** -8, atol=1e-4)


TILE_SIZES = [(256, 256), (256, 192), (128, 256), (128, 128), (64, 128), (64, 64), (192, 256)]      # rows and columns, as gemm_tiles.hip numbers them


def _gate_error(gate, up, err_gate, err_up, act):
    """What errors of a float gate and up leave of ``act(gate) * up`` in bfloat16: neither activation is steeper than 1.13."""
    return 1.13 * err_gate * (up.abs() + err_up) + act(gate).abs() * err_up + (2.0 ** -8 * (act(gate) * up).abs()) + 1e-6


@pytest.mark.parametrize("tile", range(7))
@pytest.mark.parametrize("Kd", [128, 384, 448, 832])
def test_many_row_product_beyond_one_panel(tile, Kd):
    """More rows than a panel (2,048) and three tiles of columns, the last one partial, over 2, 6, 7 and 13 steps (fewer than the
    stages, and several rounds of them); gated: three tiles of pairs, the last one partial.  Bounds as in the test above."""
    bm, bn = TILE_SIZES[tile]
    torch.manual_seed(tile)
    M, N = 2048 + bm + 9, 2 * bn + 20
    a = torch.randn(M, Kd, device=DEV).to(torch.bfloat16)
    w = (torch.randn(N, Kd, device=DEV) / math.sqrt(Kd)).to(torch.bfloat16)
    want, err = a.double() @ w.double().T, Kd * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)
    got = K()._tiles(a, K().shuffle_weight(w), None, torch.float32, M, N, Kd, Kd, 256 + tile)
    assert bool(((got.double() - want).abs() <= err).all())
    if tile == 1:
        return
    M, I = 2048 + bm + 9 if Kd == 448 else bm + 9, bn + 48
    a, w = a[:M], (torch.randn(2 * I, Kd, device=DEV) / math.sqrt(Kd)).to(torch.bfloat16)
    both, err = a.double() @ w.double().T, Kd * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)
    for act, fn in ((0, torch.nn.functional.silu), (2, lambda z: torch.nn.functional.gelu(z, approximate="tanh"))):
        got = K()._tiles(a, K().shuffle_weight(w), None, torch.bfloat16, M, 2 * I, Kd, Kd, 256 + tile, gated=True, act=act)
        gate, up = both[:, :I], both[:, I:]
        assert bool(((got.double() - fn(gate) * up).abs() <= _gate_error(gate, up, err[:, :I], err[:, I:], fn)).all())


@pytest.mark.parametrize("tile,M,Kd,shares", [(3, 1, 64, 1), (3, 129, 192, 1), (3, 300, 256, 1), (3, 257, 320, 1), (3, 129, 832, 2), (3, 2048, 576, 1),
                                              (4, 65, 1216, 1), (4, 65, 1280, 1), (4, 130, 1344, 1), (4, 63, 2624, 2), (4, 512, 1600, 1)])
def test_tiles_with_a_cu_of_their_own(tile, M, Kd, shares):
    """A grid of at most one work-group to a CU (tile 4: of 20 steps or more) has more stages, from fewer steps than stages on: bit for bit
    the rows of a call of more tiles than CUs, which has the other form (every sum is of the same order)."""
    bm, N = TILE_SIZES[tile][0], 2048
    many = 2048 // shares // 2 if tile == 4 else 2048 // shares       # rows that fill the CUs
    assert M <= many
    torch.manual_seed(Kd)
    a = torch.randn(many + bm, Kd, device=DEV).to(torch.bfloat16)
    w = (torch.randn(N, Kd, device=DEV) / math.sqrt(Kd)).to(torch.bfloat16)
    sh = K().shuffle_weight(w)
    run = lambda rows, dt, **kw: K()._tiles(a[:rows], sh, None, dt, rows, N, Kd, Kd, shares * 256 + tile, **kw)
    for dt in (torch.float32, torch.bfloat16):
        torch.testing.assert_close(run(M, dt), run(many + bm, dt)[:M], atol=0, rtol=0)
    if shares == 1:
        torch.testing.assert_close(run(M, torch.bfloat16, gated=True), run(many + bm, torch.bfloat16, gated=True)[:M], atol=0, rtol=0)


@pytest.mark.parametrize("M,I,Kd", [(1, 16, 64), (65, 144, 128), (127, 128, 192), (128, 272, 256), (129, 112, 320), (257, 400, 832), (2200, 48, 448)])
def test_gated_product_with_the_matrix_in_registers(M, I, Kd):
    """Tiles whose matrix goes straight into registers, from one step of K to fewer and more than are under way, at the edges of rows
    and of columns, rows with a stride: bit for bit what tiles of the same rows with the matrix in LDS give (every sum is
    of the same order)."""
    torch.manual_seed(Kd)
    a = torch.randn(M, Kd + 8, device=DEV).to(torch.bfloat16)[:, :Kd]
    sh = K().shuffle_weight((torch.randn(2 * I, Kd, device=DEV) / math.sqrt(Kd)).to(torch.bfloat16))
    for act in (0, 2):
        got, want = (K()._tiles(a, sh, None, torch.bfloat16, M, 2 * I, Kd, a.stride(0), 256 + tile, gated=True, act=act) for tile in (7, 2))
        assert bool(torch.isfinite(got).all()) and torch.equal(got, want)


@pytest.mark.parametrize("tile", [0, 3, 5, 6, 7])
def test_gate_of_every_size(tile):
    """SiLU behind the product for every finite bfloat16 number as the gate: sorted, so that waves have middling numbers only, and in
    disorder, so that they have some beyond.  The same bits both ways (a number's steps do not depend on its wave's others), and within
    the rounding of the float steps (2^-21) and of the result; where e^-v passes the largest float, 2^128, the result is 0 for at
    most 89 / 2^128 < 2^-121."""
    v = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    v = v[torch.isfinite(v)].to(DEV)
    v = v[v.float().abs().sort().indices]
    M, I, Kd = v.numel(), 16, 64
    w = torch.zeros(2 * I, Kd, device=DEV, dtype=torch.bfloat16)
    w[:I, 0], w[I:, 1] = 1, 0.75
    sh = K().shuffle_weight(w)

    def run(values):
        a = torch.zeros(M, Kd, device=DEV, dtype=torch.bfloat16)
        a[:, 0], a[:, 1] = values, 1
        return K()._tiles(a, sh, None, torch.bfloat16, M, 2 * I, Kd, Kd, 256 + tile, gated=True)[:, 3]
    got, mixed = run(v), torch.randperm(M, device=DEV)
    assert torch.equal(run(v[mixed]).view(torch.int16), got[mixed].view(torch.int16))
    want = v.double() / (1 + (-v.double()).exp()) * 0.75
    assert bool(((got.double() - want).abs() <= (2.0 ** -8 + 2.0 ** -21) * want.abs() + 2.0 ** -121).all())


@pytest.mark.parametrize("M,N,Kd,gated,tile,shares", [(2049, 17920, 1536, True, 7, 1), (801, 17920, 1536, True, 7, 1), (513, 17920, 1536, True, 6, 1),
                                                      (1521, 9728, 896, True, 0, 1), (300, 17920, 1536, True, 2, 1), (700, 9728, 896, True, 3, 1), (65, 9728, 896, True, 4, 1), (1300, 1536, 8960, False, 1, 5),
                                                      (801, 1536, 8960, False, 2, 6), (1025, 1536, 8960, False, 6, 7), (2049, 6144, 1024, False, 0, 1),
                                                      (801, 2048, 1536, False, 4, 1), (2049, 2048, 1536, False, 3, 1), (65, 2048, 1536, False, 5, 4)])
def test_many_row_calls_in_the_tiles_of_real_steps(M, N, Kd, gated, tile, shares):
    """linear and swiglu_gate_up at sizes that the rule gives each of the tiles, with bias, activation and in every result type."""
    torch.manual_seed(M)
    a = torch.randn(M, Kd, device=DEV).to(torch.bfloat16)
    w = (torch.randn(N, Kd, device=DEV) / math.sqrt(Kd)).to(torch.bfloat16)
    bias, sh = torch.randn(N, device=DEV), K().shuffle_weight(w)
    assert K()._tiles_plan(a, sh, M, N, Kd, Kd, gated=gated) == 256 * shares + tile
    want, err = a.double() @ w.double().T, (Kd + shares) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T)
    if gated:
        gate, up, eg, eu = want[:, :N // 2], want[:, N // 2:], err[:, :N // 2], err[:, N // 2:]
        for activation, fn in (("silu", torch.nn.functional.silu), ("gelu_tanh", lambda z: torch.nn.functional.gelu(z, approximate="tanh"))):
            got = K().swiglu_gate_up(a, w, shuffled=sh, activation=activation)
            assert got.dtype == torch.bfloat16 and bool(((got.double() - fn(gate) * up).abs() <= _gate_error(gate, up, eg, eu, fn)).all())
        return
    want = want + bias.double()
    err = err + 2.0 ** -24 * want.abs()
    got = K().linear(a, w, bias, out_dtype=torch.float32, shuffled=sh)
    assert bool(((got.double() - want).abs() <= err).all())
    got = K().linear(a, w, bias, shuffled=sh)
    assert got.dtype == torch.bfloat16 and bool(((got.double() - want).abs() <= err + 2.0 ** -8 * want.abs()).all())
    relu2 = want.clamp_min(0) ** 2                                    # (the square doubles what its argument is off by)
    for dt, rel in ((torch.float32, 2.0 ** -23), (torch.bfloat16, 2.0 ** -8)):
        got = K().linear(a, w, bias, out_dtype=dt, shuffled=sh, act="relu2")
        assert got.dtype == dt and bool(((got.double() - relu2).abs() <= rel * relu2 + 2 * want.abs() * err + err ** 2 + 1e-6).all())
    if shares > 1:
        kept = K().linear(a, w, None, out_dtype=torch.float32, shuffled=sh, keep_shares=True)
        assert isinstance(kept, K().ShareSum) and bool(((kept.sum().double() + bias.double() - want).abs() <= err + 2.0 ** -24 * want.abs()).all())


def test_many_row_product_by_its_rule():
    """linear and swiglu_gate_up take the tiles the rule picks, for the library's own results: a product with its K in shares, one
    without, and a K the tiles do not take."""
    torch.manual_seed(5)
    for M, N, Kd in ((2100, 256, 512), (70, 512, 9216), (130, 320, 96)):
        a = torch.randn(M, Kd, device=DEV).to(torch.bfloat16)
        w = (torch.randn(N, Kd, device=DEV) / math.sqrt(Kd)).to(torch.bfloat16)
        sh = K().shuffle_weight(w)
        assert bool(K()._tiles_plan(a, sh, M, N, Kd, Kd)) == (Kd % 64 == 0)
        want = a.double() @ w.double().T
        torch.testing.assert_close(K().linear(a, w, None, out_dtype=torch.float32, shuffled=sh).double(), want, atol=1e-4, rtol=1e-4)
        torch.testing.assert_close(K().linear(a, w, None, shuffled=sh).double(), want, atol=1e-4, rtol=2.0 ** -8)
        silu = torch.nn.functional.silu(want[:, :N // 2]) * want[:, N // 2:]
        torch.testing.assert_close(K().swiglu_gate_up(a, w, shuffled=sh).double(), silu, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("M", [1, 7, 16])
@pytest.mark.parametrize("N,Kd", [(1000, 1184), (3584, 18944), (50, 1030), (70, 513), (130, 7), (16, 512), (37, 40000)])
def test_linear_few_rows_float32(M, N, Kd):
    """The float product for at most 16 rows: K in segments of 512 shared by a work-group's waves (one
    segment, a partial last one, more segments than waves, a K that is no multiple of 4 and one too
    long for the segments' sums in LDS, which the many-row kernel takes), N no multiple of 16.  A
    row's result has the same bits whatever other rows come along."""
    torch.manual_seed(M + N)
    a = torch.randn(M, Kd, device=DEV)
    w = torch.randn(N, Kd, device=DEV) / math.sqrt(Kd)
    b = torch.randn(N, device=DEV)
    want = a.double() @ w.double().T + b.double()
    got = K().linear(a, w, b)
    assert got.dtype == torch.float32
    torch.testing.assert_close(got.double(), want, atol=1e-5, rtol=1e-5)
    alone = K().linear(a[M - 1:].contiguous(), w, b)
    torch.testing.assert_close(alone[0], got[M - 1], atol=0, rtol=0)
    # from the matrix-core ordered copy of the weight (what the engine's decode steps stream): the same bits
    ws = K().shuffle_weight_float(w)
    assert ws.shape == (-(-N // 16), -(-Kd // 16), 4, 16, 4)
    torch.testing.assert_close(K().linear(a, w, b, shuffled=ws), got, atol=0, rtol=0)
    strided = torch.randn(M, Kd + 5, device=DEV)[:, 1:Kd + 1]          # rows neither aligned nor contiguous
    torch.testing.assert_close(K().linear(strided, w, b, shuffled=ws), K().linear(strided, w, b), atol=0, rtol=0)


@pytest.mark.parametrize("M", [17, 32, 33, 70, 129, 300])
@pytest.mark.parametrize("N,Kd", [(1, 1), (31, 15), (33, 16), (130, 17), (257, 2047), (96, 2048), (132, 2049), (40, 4100), (1152, 896)])
def test_linear_float_by_three_bfloat16(M, N, Kd):
    """The float product of more than 16 rows (every float as the sum of three bfloat16): tiles' and segments' edges,
    rows neither aligned nor contiguous, columns that the segments' adding kernel takes four at a time or one.  The bound is
    that of K float multiply-adds in any order.  A row has the same bits whatever rows come along."""
    torch.manual_seed(M + N)
    w = torch.randn(N, Kd, device=DEV)
    b = torch.randn(N, device=DEV)
    ws = K().shuffle_weight_float(w)
    for a in (torch.randn(M, Kd, device=DEV), torch.randn(M, Kd + 5, device=DEV)[:, 1:Kd + 1]):
        want = a.double() @ w.double().T + b.double()
        size = a.double().abs() @ w.double().abs().T + b.double().abs()
        got = K().linear(a, w, b, shuffled=ws)
        assert bool(((got.double() - want).abs() <= (Kd + 8) * 2.0 ** -24 * size).all())
        few = K().linear(a[M - 17:], w, b, shuffled=ws)
        assert torch.equal(few, got[M - 17:])
        wide = torch.full((M, N + 3), 7.0, device=DEV)
        K().linear(a, w, b, out=wide[:, 1:N + 1], shuffled=ws)
        assert torch.equal(wide[:, 1:N + 1], got) and bool((wide[:, [0, N + 1, N + 2]] == 7.0).all())


def test_linear_float_by_three_bfloat16_not_finite():
    """Infinities, NaN and values that round to infinity as bfloat16, on either side and across segments: what plain float
    arithmetic gives."""
    torch.manual_seed(3)
    a, w = torch.randn(40, 2100, device=DEV), torch.randn(70, 2100, device=DEV)
    a[3, 5], a[7, 2070], a[9, 1], w[5, 2], w[6, 2090] = float("inf"), float("nan"), 3.4e38, float("-inf"), 3.4e38
    w[:, 1] *= 1e-3
    got = K().linear(a, w, shuffled=K().shuffle_weight_float(w)).cpu()
    want = (a.cpu().double() @ w.cpu().double().T).float()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[want.isinf()], want[want.isinf()])
    fine = want.isfinite()
    torch.testing.assert_close(got[fine], want[fine], atol=1e-3, rtol=1e-5)


@pytest.mark.parametrize("Kd", [1, 2, 3, 7, 15, 16, 33, 64, 128, 896, 3584])
@pytest.mark.parametrize("values", ["normal", "positive", "one column large"])
def test_linear_float_is_no_further_from_64_bits_than_the_float_instruction(Kd, values):
    """More than 16 float rows, at every K: not further from the exact product, in the 2-norm, than the product on the float
    matrix instruction (the call without the ordered copy), and a K of one is rounded once."""
    torch.manual_seed(Kd)
    M, N = 200, 512
    a = torch.rand(M, Kd, device=DEV) if values == "positive" else torch.randn(M, Kd, device=DEV)
    w = torch.rand(N, Kd, device=DEV) if values == "positive" else torch.randn(N, Kd, device=DEV)
    if values == "one column large":
        a[:, Kd // 3] *= 3000.0
    want = a.double() @ w.double().T
    got, other = K().linear(a, w, shuffled=K().shuffle_weight_float(w)), K().linear(a, w)
    assert (got.double() - want).norm() <= (other.double() - want).norm()
    if Kd == 1:
        assert bool(((got.double() - want).abs() <= 2.0 ** -24 * want.abs()).all())


@pytest.mark.parametrize("N,Kd", [(33, 64), (70, 68), (130, 76), (1000, 100), (257, 128), (40, 252), (1152, 256),
                                  (129, 384), (70, 388), (40, 772), (33, 1000), (300, 2044), (128, 2048), (32769, 64), (33000, 156)])
@pytest.mark.parametrize("M", [17, 30, 32])
def test_linear_float_of_at_most_32_rows_splits_them_where_they_are_used(M, N, Kd):
    """One launch for 17 to 32 aligned rows: the bits that the same rows get from parts made beforehand (rows that are not
    aligned, or among more rows), the last step's missing units of k and rows' ends untouched by what lies behind them."""
    torch.manual_seed(M + Kd)
    behind = torch.full((40, Kd + 8), float("nan"), device=DEV)
    behind[:, :Kd] = torch.randn(40, Kd, device=DEV)
    a, odd = behind[:M, :Kd], torch.full((M, Kd + 5), float("nan"), device=DEV)
    odd[:, 1:Kd + 1] = a
    w, b = torch.randn(N, Kd, device=DEV), torch.randn(N, device=DEV)
    ws = K().shuffle_weight_float(w)
    got = K().linear(a, w, b, shuffled=ws)
    want, size = a.double() @ w.double().T + b.double(), a.double().abs() @ w.double().abs().T + b.double().abs()
    assert bool(((got.double() - want).abs() <= (Kd + 8) * 2.0 ** -24 * size).all())
    assert torch.equal(K().linear(odd[:, 1:Kd + 1], w, b, shuffled=ws), got)
    assert torch.equal(K().linear(behind[:, :Kd], w, b, shuffled=ws)[:M], got)
    # infinities, NaN and values past the split's range, in the rows and in the matrix
    behind[3, Kd - 1], behind[16, 5], behind[9, Kd // 2], w[7, 2], w[N - 1, Kd - 2] = float("inf"), float("nan"), 2.0 ** 110, 2.0 ** 120, float("-inf")
    odd[:, 1:Kd + 1] = a
    ws = K().shuffle_weight_float(w)
    torch.testing.assert_close(K().linear(a, w, b, shuffled=ws), K().linear(odd[:, 1:Kd + 1], w, b, shuffled=ws), rtol=0, atol=0, equal_nan=True)


@pytest.mark.parametrize("M,N,Kd", [(40003, 40, 8200), (9000, 5000, 8200)])
def test_linear_float_of_very_many_rows_has_a_bounded_workspace(M, N, Kd):
    """At most 512 MB for the rows' parts (here in several launches) and 512 MB for the segments' sums; rows on either side of
    a launch's edge have the bits that they have alone."""
    torch.manual_seed(M)
    a, w = torch.randn(M, Kd, device=DEV), torch.randn(N, Kd, device=DEV)
    ws, out = K().shuffle_weight_float(w), torch.empty(M, N, device=DEV)
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    K().linear(a, w, out=out, shuffled=ws)
    assert torch.cuda.max_memory_allocated() - before <= 1 << 30
    edge = K().FLOAT_SPLIT_BYTES // (-(-Kd // 16) * 96) // 128 * 128
    for r in (0, min(edge - 10, M - 20), M - 20):
        assert torch.equal(K().linear(a[r:r + 20], w, shuffled=ws), out[r:r + 20])


# (tile, K dealt out by segments, M, N, K): every tile of the float product of more than 16 rows, with the whole of K (two
# segments) and in segments, none of them filled by its rows, its columns or its last step
FLOAT_TILES = [(0, False, 701, 66003, 2100), (0, True, 2049, 2051, 4101), (1, False, 1501, 4101, 2100), (1, True, 97, 16401, 4100),
               (2, False, 301, 16399, 2101), (2, True, 97, 8201, 4100), (3, False, 201, 8201, 2100), (3, True, 97, 2051, 2101)]


def _float_tile(tile, parts, M, N, Kd):
    assert K().library().tl_gemm_float_split_tile(M, N, Kd) == tile + (4 if parts else 0)


@pytest.mark.parametrize("tile,parts,M,N,Kd", FLOAT_TILES)
def test_linear_float_in_every_tile(tile, parts, M, N, Kd):
    """The bound of K float multiply-adds, ends of rows, columns and k, and a row's bits whatever rows come along: 17 rows (the
    smallest tile) and 70 (the next) against the tile that M rows take; columns either side of the result untouched."""
    _float_tile(tile, parts, M, N, Kd)
    torch.manual_seed(tile + 20)
    a, w, b = torch.randn(M, Kd, device=DEV), torch.randn(N, Kd, device=DEV), torch.randn(N, device=DEV)
    ws = K().shuffle_weight_float(w)
    wide = torch.full((M, N + 3), 7.0, device=DEV)
    got = K().linear(a, w, b, out=wide[:, 1:N + 1], shuffled=ws)
    assert bool((wide[:, [0, N + 1, N + 2]] == 7.0).all())
    want, size = a.double() @ w.double().T + b.double(), a.double().abs() @ w.double().abs().T + b.double().abs()
    assert bool(((got.double() - want).abs() <= (Kd + 8) * 2.0 ** -24 * size).all())
    for n in (17, 70):
        assert torch.equal(K().linear(a[M - n:], w, b, shuffled=ws), got[M - n:])
        assert torch.equal(K().linear(a[:n].contiguous(), w, b, shuffled=ws), got[:n])
    assert K().library().tl_gemm_float_split_tile(17, N, Kd) & 3 == 3 and (tile == 3 or K().library().tl_gemm_float_split_tile(70, N, Kd) & 3 != tile)


@pytest.mark.parametrize("tile,parts,M,N,Kd", FLOAT_TILES)
def test_linear_float_not_finite_in_every_tile(tile, parts, M, N, Kd):
    """Infinities, NaN, values that round to infinity as bfloat16 and a product just below the largest float whose rounded
    parts' product is above it, in either segment: what plain float arithmetic gives; every other element as without them."""
    _float_tile(tile, parts, M, N, Kd)
    torch.manual_seed(tile)
    a, w, bias = torch.randn(M, Kd, device=DEV), torch.randn(N, Kd, device=DEV), torch.randn(N, device=DEV)
    w[:, 2] *= 1e-3                                          # 3.4e38 times that stays a float
    a[:, 2080] *= 1e-3
    plain_rows = K().linear(a, w, bias, shuffled=K().shuffle_weight_float(w))
    a[3, 5], a[40, 2070], a[M - 1, 2] = float("inf"), float("nan"), 3.4e38
    w[6, 2080], w[N - 1, 7] = 3.4e38, float("-inf")
    big = 2.0 ** 64 - 2.0 ** 40                              # big^2 rounds to 2^128 (1 - 2^-23), finite; big rounds to 2^64 as bfloat16
    bias[9] = 0.0
    for row, at in ((11, 8), (M - 2, 2090)):                 # that product alone in row 9 of the matrix, in the first and the second segment
        a[row, at], w[9, at] = big if row == 11 else -big, big
    w[9, :8] = w[9, 9:2090] = w[9, 2091:] = 0.0
    a[11, 2090] = a[M - 2, 8] = 0.0
    got = K().linear(a, w, bias, shuffled=K().shuffle_weight_float(w))
    rows, cols = [3, 11, 40, M - 2, M - 1], [6, 9, N - 1]
    top = (2.0 ** 128 * (1.0 - 2.0 ** -23))
    assert got[11, 9].item() == top and got[M - 2, 9].item() == -top
    want = (a.double() @ w.double().T + bias.double()).float()
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[want.isinf()], want[want.isinf()])
    fine = want.isfinite()
    size = (a.double().abs() @ w.double().abs().T + bias.double().abs())[fine]
    assert bool(((got[fine].double() - want[fine].double()).abs() <= (Kd + 8) * 2.0 ** -24 * size).all())
    other_rows = torch.ones(M, dtype=torch.bool, device=DEV)
    other_cols = torch.ones(N, dtype=torch.bool, device=DEV)
    other_rows[rows], other_cols[cols] = False, False
    assert torch.equal(got[other_rows][:, other_cols], plain_rows[other_rows][:, other_cols])


@pytest.mark.parametrize("tile,parts,M,N,Kd", FLOAT_TILES)
def test_linear_float_of_small_and_large_values_in_every_tile(tile, parts, M, N, Kd):
    """Rows and matrix rows of every magnitude a float has, 2^-140 (subnormal, rounded by that) to 2^120, whose products come out
    around one: the bound of K float multiply-adds, the same for all of them."""
    _float_tile(tile, parts, M, N, Kd)
    torch.manual_seed(tile + 10)
    a, w = torch.randn(M, Kd, device=DEV), torch.randn(N, Kd, device=DEV)
    up = torch.tensor([0, -100, -112, -120, -126, -140, 60, 100, 120], device=DEV)
    at, wt = up[torch.arange(M, device=DEV) % 9], up[torch.arange(N, device=DEV) % 9]
    a, w = torch.ldexp(a, at[:, None].float()), torch.ldexp(w, wt[:, None].float())
    got = K().linear(a, w, shuffled=K().shuffle_weight_float(w))
    want, size = a.double() @ w.double().T, a.double().abs() @ w.double().abs().T
    fits = (at[:, None] + wt[None, :] >= -90) & (at[:, None] + wt[None, :] <= 100)      # products and sums that are normal floats
    ok = (got.double() - want).abs() <= (Kd + 8) * 2.0 ** -24 * size
    assert bool(ok[fits].all())


@pytest.mark.parametrize("M", [1, 2, 8, 16, 17, 33, 48, 64])
@pytest.mark.parametrize("N,Kd", [(1000, 1184), (4608, 3584), (136, 8), (50, 264), (3584, 18944), (5120, 1184), (2090, 72),
                                  (5120, 9728)])
def test_linear_few_rows_bfloat16(M, N, Kd):
    """The streaming MFMA kernels (up to 16 rows, and 17 to 64): N no multiple of 16 or 128, K with a
    partial chunk, K cut into shares; numbers of tiles that fill the CUs unevenly (224, 288, 320, 131),
    the last with a K so long that few rows too go to the kernel that cuts K into shares."""
    assert K()._few_rows_go_to_rows64(N, Kd) == ((N, Kd) == (5120, 9728))
    torch.manual_seed(M + N)
    a = torch.randn(M, Kd, device=DEV).to(torch.bfloat16)
    w = (torch.randn(N, Kd, device=DEV) / math.sqrt(Kd)).to(torch.bfloat16)
    b = torch.randn(N, device=DEV)
    want = a.double() @ w.double().T + b.double()
    ws = K().shuffle_weight(w)
    got = K().linear(a, w, b, out_dtype=torch.float32, shuffled=ws)
    torch.testing.assert_close(got.double(), want, atol=2e-4 * math.sqrt(Kd / 1000 + 1), rtol=2e-4)
    got16 = K().linear(a, w, b, shuffled=ws)
    torch.testing.assert_close(got16.double(), want, atol=3e-2, rtol=3e-2)
    # the value of a row does not depend on the rows beside it
    alone = K().linear(a[M - 1:M].contiguous(), w, b, out_dtype=torch.float32, shuffled=ws)
    same_class = M <= 16          # up to 16 rows run the same code with the same split of K: same bits
    t = 0 if same_class else 2e-4 * math.sqrt(Kd / 1000 + 1)
    torch.testing.assert_close(alone[0], got[M - 1], atol=t, rtol=t)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("M", [1, 8, 40, 64, 200])
@pytest.mark.parametrize("I,Kd", [(176, 64), (1184, 3584), (100, 48), (48, 136)])
def test_swiglu_gate_up(dtype, M, I, Kd):
    torch.manual_seed(M + I)
    h = torch.randn(M, Kd, device=DEV).to(dtype)
    w = (torch.randn(2 * I, Kd, device=DEV) / math.sqrt(Kd) * 2).to(dtype)
    got = K().swiglu_gate_up(h, w, K().shuffle_weight(w))
    gu = h.double() @ w.double().T
    want = torch.nn.functional.silu(gu[:, :I]) * gu[:, I:]
    assert got.dtype == dtype and tuple(got.shape) == (M, I)
    # float32 accumulation over K terms: the error grows with sqrt(K)
    torch.testing.assert_close(got.double(), want, **tol(dtype, 2e-6 * math.sqrt(Kd) + 1e-5, 4e-2))


@pytest.mark.parametrize("dtype", DTYPES)
def test_linear_strided_rows(dtype):
    torch.manual_seed(1)
    big = torch.randn(9, 300, device=DEV).to(dtype)
    a = big[:, 20:120]
    w = torch.randn(33, 100, device=DEV).to(dtype)
    got = K().linear(a, w, None, out_dtype=torch.float32)
    torch.testing.assert_close(got.double(), a.double() @ w.double().T, **tol(dtype, 2e-5, 2e-5))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,d,rot", [(14, 2, 64, 64), (5, 1, 48, 48), (4, 4, 16, 8), (28, 4, 128, 128)])
def test_rope_store(dtype, nq, nkv, d, rot):
    torch.manual_seed(0)
    T, bs, pages, theta = 37, 8, 12, 50000.0
    qkv = torch.randn(T, (nq + 2 * nkv) * d, device=DEV).to(dtype)
    pos = torch.randint(0, 3000, (T,), dtype=torch.int32, device=DEV)
    slots = torch.randperm(pages * bs, device=DEV)[:T].to(torch.int32)
    slots[5] = -1
    kc = torch.full((pages, bs, nkv, d), 7.0, device=DEV).to(dtype)
    vc = torch.full((pages, nkv, d, bs), 7.0, device=DEV).to(dtype)       # values: transposed within the page
    i = torch.arange(0, rot, 2, dtype=torch.float64)
    inv_freq = (theta ** (-i / rot)).float().to(DEV)
    heads = qkv.float().cpu().view(T, nq + 2 * nkv, d)
    want_q = plain.rope(heads[:, :nq], pos.cpu(), theta, rot)
    want_k = plain.rope(heads[:, nq:nq + nkv], pos.cpu(), theta, rot)
    want_v = heads[:, nq + nkv:]
    K().rope_store(qkv, pos, inv_freq, nq, nkv, d, kc, vc, slots)
    got = qkv.float().cpu().view(T, nq + 2 * nkv, d)
    t = tol(dtype, 2e-5, 2e-2)
    torch.testing.assert_close(got[:, :nq], want_q, **t)
    kf, vf = kc.float().cpu().view(-1, nkv, d), vc.float().cpu().permute(0, 3, 1, 2).reshape(-1, nkv, d)
    ok = slots.cpu() >= 0
    torch.testing.assert_close(kf[slots.cpu()[ok].long()], want_k[ok], **t)
    torch.testing.assert_close(vf[slots.cpu()[ok].long()], want_v[ok], atol=0, rtol=0)
    untouched = torch.ones(pages * bs, dtype=torch.bool)
    untouched[slots.cpu()[ok].long()] = False
    assert torch.all(kf[untouched] == 7.0) and torch.all(vf[untouched] == 7.0)
    # position 0 is the identity
    qkv0 = torch.randn(3, (nq + 2 * nkv) * d, device=DEV).to(dtype)
    keep = qkv0.clone()
    K().rope_store(qkv0, torch.zeros(3, dtype=torch.int32, device=DEV), inv_freq, nq, nkv, d, None, None, None)
    torch.testing.assert_close(qkv0, keep, atol=0, rtol=0)
    # an owed bias: the same as adding it beforehand (in float32: to the bit)
    bias = torch.randn((nq + 2 * nkv) * d, device=DEV)
    outs = []
    for owed in (True, False):
        x = qkv.clone() if owed else (qkv.float() + bias).to(dtype)      # qkv holds rotated queries by now: any input will do
        kc2, vc2 = torch.zeros_like(kc), torch.zeros_like(vc)
        K().rope_store(x, pos, inv_freq, nq, nkv, d, kc2, vc2, slots, bias if owed else None)
        outs.append((x[:, :nq * d], kc2, vc2))
    for a, b in zip(*outs):
        if dtype == torch.float32:
            torch.testing.assert_close(a, b, atol=0, rtol=0)
        else:
            torch.testing.assert_close(a.float(), b.float(), atol=3e-2, rtol=3e-2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nq,nkv,d,rot,shift", [
    (7, 1, 16, 16, 0), (3, 1, 8, 8, 0), (30, 2, 128, 128, 0),      # one pair group a head; as many as 256 threads and their half
    (31, 2, 128, 128, 1), (60, 8, 120, 120, 0),                    # one head more, a bias at 4 bytes; groups that no power of two counts
    (33, 2, 512, 512, 0), (3, 1, 512, 512, 3),                     # more groups than a work-group has threads; every wave has an angle
    (5, 2, 40, 12, 0), (9, 3, 37, 2, 1),                           # single pairs with dims that pass through
])
def test_rope_store_in_groups_of_pairs(dtype, nq, nkv, d, rot, shift):
    """Pairs by the 16 bytes and one by one, at the numbers of threads a token gets: against the rotation in float64."""
    torch.manual_seed(d)
    T, bs, width = 5, 8, (nq + 2 * nkv) * d
    qkv, bias = torch.randn(T, width, device=DEV).to(dtype), torch.randn(width + shift, device=DEV)[shift:]
    pos, slots = torch.tensor([0, 1, 77, 900, 1500], dtype=torch.int32, device=DEV), torch.tensor([3, 15, -1, 0, 9], dtype=torch.int32, device=DEV)
    inv = (10000.0 ** (-torch.arange(0, rot, 2, dtype=torch.float64) / rot)).float().to(DEV)
    x = (qkv.double() + bias.double()).view(T, nq + 2 * nkv, d)
    theta = (pos.float()[:, None] * inv).double()[:, None]         # (the angle is a float32 product)
    a, b, heads = x[:, :nq + nkv, :rot // 2], x[:, :nq + nkv, rot // 2:rot], x.clone()
    heads[:, :nq + nkv, :rot // 2], heads[:, :nq + nkv, rot // 2:rot] = a * theta.cos() - b * theta.sin(), b * theta.cos() + a * theta.sin()
    kc, vc = torch.full((2, bs, nkv, d), 7.0, device=DEV).to(dtype), torch.full((2, nkv, d, bs), 7.0, device=DEV).to(dtype)
    K().rope_store(qkv, pos, inv, nq, nkv, d, kc, vc, slots, bias)
    keys, values = kc.double().view(-1, nkv, d), vc.double().permute(0, 3, 1, 2).reshape(-1, nkv, d)
    # of values up to 12: a sum with the bias, two products, their sum and a sine rounded in float32, and one rounding of the result
    t = dict(atol=12 * 8 * 2.0 ** -24, rtol=2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -22)
    torch.testing.assert_close(qkv.double().view(T, -1, d)[:, :nq], heads[:, :nq], **t)
    for t_, s in enumerate(slots.tolist()):
        if s >= 0:
            torch.testing.assert_close(keys[s], heads[t_, nq:nq + nkv], **t)
            torch.testing.assert_close(values[s], heads[t_, nq + nkv:], **t)
    left = [s for s in range(2 * bs) if s not in slots.tolist()]
    assert bool((keys[left] == 7).all()) and bool((values[left] == 7).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,nq,nkv,d,rot", [(2051, 20, 2, 128, 128), (4100, 20, 2, 128, 32), (3000, 3, 3, 192, 0), (513, 4, 4, 24, 24), (2049, 33, 1, 128, 128),
                                             (2048, 28, 2, 128, 128)])
def test_rope_store_of_many_tokens(dtype, T, nq, nkv, d, rot):
    """Steps of many tokens, whose work-groups are smaller and whose values come last, leave what the same tokens in small steps do."""
    torch.manual_seed(T)
    pages, bs, width = T // 16 + 2, 16, (nq + 2 * nkv) * d
    rows, bias = torch.randn(T, width, device=DEV).to(dtype), torch.randn(width, device=DEV)
    pos, slots = torch.randint(0, 5000, (T,), dtype=torch.int32, device=DEV), torch.randperm(pages * bs, device=DEV)[:T].int()
    slots[::7] = -1
    inv = (10000.0 ** (-torch.arange(0, rot, 2, dtype=torch.float64) / rot)).float().to(DEV) if rot else None
    left = []
    for step in (T, 100):
        x, kc, vc = rows.clone(), torch.full((pages, bs, nkv, d), 7.0, device=DEV).to(dtype), torch.full((pages, nkv, d, bs), 7.0, device=DEV).to(dtype)
        for t in range(0, T, step):
            K().rope_store(x[t:t + step], pos[t:t + step], inv, nq, nkv, d, kc, vc, slots[t:t + step], bias)
        left.append((x, kc, vc))
    assert all(torch.equal(a, b) for a, b in zip(*left)) and not torch.equal(left[0][0], rows)


@pytest.mark.parametrize("M", [1, 5, 16, 17, 40, 64])
@pytest.mark.parametrize("nq,nkv,d,Kd", [(6, 2, 32, 192), (28, 4, 128, 3584), (4, 4, 64, 264), (5, 1, 96, 120)])
def test_fused_projection_rotation_and_cache_write(M, nq, nkv, d, Kd):
    """One kernel for q/k/v projection + bias + RoPE + cache write against the three separate kernels."""
    torch.manual_seed(M + nq)
    bs, pages, theta = 8, 12, 1e6
    pages = max(pages, M // bs + 4)
    N = (nq + 2 * nkv) * d
    h = torch.randn(M, Kd, device=DEV).to(torch.bfloat16)
    w = (torch.randn(N, Kd, device=DEV) / math.sqrt(Kd)).to(torch.bfloat16)
    b = torch.randn(N, device=DEV)
    pos = torch.randint(0, 4000, (M,), dtype=torch.int32, device=DEV)
    slots = torch.randperm(pages * bs, device=DEV)[:M].to(torch.int32)
    if M > 2:
        slots[2] = -1
    inv_freq = (theta ** (-torch.arange(0, d, 2, dtype=torch.float64) / d)).float().to(DEV)
    mk = lambda: (torch.full((pages, bs, nkv, d), 7.0, device=DEV).to(torch.bfloat16),
                  torch.full((pages, nkv, d, bs), 7.0, device=DEV).to(torch.bfloat16))
    kc, vc = mk()
    q = K().qkv_rope_store(h, K().shuffle_weight(w), b, pos, inv_freq, nq, nkv, d, kc, vc, slots)
    if M > 16 and K().library().tl_gemm_rows64_shares(M, N, Kd) == 1:
        assert q is None                                      # K too short to be cut: the separate kernels serve
        return
    assert q is not None and tuple(q.shape) == (M, nq * d)
    # the same from the plain formulas in float64
    qkv = (h.double() @ w.double().T + b.double()).cpu().view(M, nq + 2 * nkv, d)
    want_q = plain.rope(qkv[:, :nq], pos.cpu(), theta)
    want_k = plain.rope(qkv[:, nq:nq + nkv], pos.cpu(), theta)
    torch.testing.assert_close(q.double().cpu().view(M, nq, d), want_q, atol=3e-2, rtol=3e-2)
    ok = slots.cpu() >= 0
    sl = slots.cpu()[ok].long()
    kf = kc.double().cpu().view(-1, nkv, d)
    vf = vc.double().cpu().permute(0, 3, 1, 2).reshape(-1, nkv, d)
    torch.testing.assert_close(kf[sl], want_k[ok], atol=3e-2, rtol=3e-2)
    torch.testing.assert_close(vf[sl], qkv[:, nq + nkv:][ok], atol=3e-2, rtol=3e-2)
    untouched = torch.ones(pages * bs, dtype=torch.bool)
    untouched[sl] = False
    assert torch.all(kf[untouched] == 7.0) and torch.all(vf[untouched] == 7.0)
    # cases it declines: float32, too many rows, partial rotation
    assert K().qkv_rope_store(h.float(), None, b, pos, inv_freq, nq, nkv, d, kc, vc, slots) is None
    assert K().qkv_rope_store(h, K().shuffle_weight(w), b, pos, inv_freq[: d // 4].contiguous(), nq, nkv, d, kc, vc, slots) is None


def _normed_rows(h, gamma, eps, parts):
    """NormedRows of float rows ``h`` as a product's residual sink would leave them, with the sum of
    squares cut into ``parts`` uneven partials."""
    M, H = h.shape
    cuts = sorted(set([0, H] + torch.randint(1, H, (parts - 1,)).tolist()))
    ss = torch.stack([(h[:, a:b].double() ** 2).sum(1) for a, b in zip(cuts[:-1], cuts[1:])], 0).float()
    return K().NormedRows((h * gamma).to(torch.bfloat16), ss.contiguous(), H, eps)


@pytest.mark.parametrize("M", [1, 7, 16, 17, 40, 64])
@pytest.mark.parametrize("N,Kd,parts", [(176, 64, 4), (1000, 1184, 74), (3584, 3584, 224), (50, 264, 1), (37888, 3584, 14),
                                        (5120, 9728, 38)])
def test_products_apply_an_owed_norm(M, N, Kd, parts):
    """A product of rows h * g with the division by rms(h) owed equals the product of RMSNorm(h) * g:
    plain, gate/up with SiLU, and q/k/v with rotation and cache write."""
    torch.manual_seed(M * 1000 + N)
    eps = 1e-5
    h = torch.randn(M, Kd, device=DEV) * torch.logspace(-1, 2, M, device=DEV)[:, None]   # rows of very different size
    if N > 30000 and M not in (16, 64):
        pytest.skip("the wide case is for the fullest row counts")
    gamma = 1 + 0.1 * torch.randn(Kd, device=DEV)
    owed = _normed_rows(h, gamma, eps, parts)
    rstd = 1 / torch.sqrt((h.double() ** 2).mean(1, keepdim=True) + eps)
    x = owed.rows.double() * rstd                        # what the product must multiply, given the rounded rows
    w = (torch.randn(N, Kd, device=DEV) / math.sqrt(Kd)).to(torch.bfloat16)
    b = torch.randn(N, device=DEV)
    sh = K().shuffle_weight(w)
    got = K().linear(owed, w, b, out_dtype=torch.float32, shuffled=sh)
    torch.testing.assert_close(got.double(), x @ w.double().T + b.double(), atol=2e-3, rtol=2e-3)
    if N % 32 == 0:
        act = K().swiglu_gate_up(owed, w, sh)
        y = x @ w.double().T
        want = torch.nn.functional.silu(y[:, :N // 2]) * y[:, N // 2:]
        torch.testing.assert_close(act.double(), want, atol=2e-2, rtol=2e-2)
    with pytest.raises(K().KernelError, match="streaming"):
        K().linear(owed, w, b, out_dtype=torch.float32, shuffled=None)


@pytest.mark.parametrize("M,Kd", [(5, 192), (40, 1184)])
def test_fused_projection_applies_an_owed_norm(M, Kd):
    torch.manual_seed(3)
    nq, nkv, d, bs, pages, eps = 6, 2, 32, 8, 12, 1e-6
    N = (nq + 2 * nkv) * d
    h = torch.randn(M, Kd, device=DEV) * 30
    gamma = 1 + 0.1 * torch.randn(Kd, device=DEV)
    owed = _normed_rows(h, gamma, eps, 12)
    x = (owed.rows.double() / torch.sqrt((h.double() ** 2).mean(1, keepdim=True) + eps)).to(torch.bfloat16)
    w = (torch.randn(N, Kd, device=DEV) / math.sqrt(Kd)).to(torch.bfloat16)
    b = torch.randn(N, device=DEV)
    pos = torch.randint(0, 4000, (M,), dtype=torch.int32, device=DEV)
    slots = torch.randperm(pages * bs, device=DEV)[:M].to(torch.int32)
    inv_freq = (1e6 ** (-torch.arange(0, d, 2, dtype=torch.float64) / d)).float().to(DEV)
    out = []
    for inp in (owed, x):
        kc = torch.zeros(pages, bs, nkv, d, device=DEV, dtype=torch.bfloat16)
        vc = torch.zeros(pages, nkv, d, bs, device=DEV, dtype=torch.bfloat16)
        q = K().qkv_rope_store(inp, K().shuffle_weight(w), b, pos, inv_freq, nq, nkv, d, kc, vc, slots)
        assert q is not None
        out.append((q, kc, vc))
    for a, c in zip(out[0], out[1]):                     # against the same kernel on rows normalised beforehand
        torch.testing.assert_close(a.float(), c.float(), atol=3e-2, rtol=3e-2)


@pytest.mark.parametrize("M", [1, 6, 16, 17, 33, 64])
@pytest.mark.parametrize("N,Kd", [(176, 64), (1000, 1184), (3584, 18944), (40, 264), (5000, 256), (5120, 520), (5120, 9728)])
def test_product_adds_into_the_residual_and_prepares_the_next_norm(M, N, Kd):
    torch.manual_seed(M + N)
    eps = 1e-6
    a = torch.randn(M, Kd, device=DEV).to(torch.bfloat16)
    w = (torch.randn(N, Kd, device=DEV) / math.sqrt(Kd)).to(torch.bfloat16)
    b = torch.randn(N, device=DEV)
    gamma = 1 + 0.1 * torch.randn(N, device=DEV)
    resid0 = torch.randn(M, N, device=DEV) * 5
    resid = resid0.clone()
    nxt = K().linear(a, w, b, out_dtype=torch.float32, shuffled=K().shuffle_weight(w), sink=K().NormSink(resid, gamma, eps))
    want = resid0.double() + a.double() @ w.double().T + b.double()
    torch.testing.assert_close(resid.double(), want, atol=1e-3, rtol=1e-4)
    assert isinstance(nxt, K().NormedRows) and nxt.dim == N and nxt.eps == eps
    torch.testing.assert_close(nxt.rows.float(), (resid * gamma).to(torch.bfloat16).float(), atol=0, rtol=2 ** -7)
    assert nxt.sumsq.shape[1] == M and nxt.sumsq.shape[0] in (-(-N // 16), -(-N // 256))
    torch.testing.assert_close(nxt.sumsq.double().sum(0), (resid.double() ** 2).sum(1), atol=0, rtol=1e-5)
    # handed on: the next product's result equals that of the norm kernel followed by the product
    w2 = (torch.randn(48, N, device=DEV) / math.sqrt(N)).to(torch.bfloat16)
    got = K().linear(nxt, w2, None, out_dtype=torch.float32, shuffled=K().shuffle_weight(w2))
    x = K().add_rmsnorm(resid.clone(), None, gamma, eps, torch.bfloat16)
    want2 = K().linear(x, w2, None, out_dtype=torch.float32, shuffled=K().shuffle_weight(w2))
    torch.testing.assert_close(got, want2, atol=2e-2, rtol=2e-2)


def _attention_case(dtype, nq, nkv, d, bs, lens, q_lens=None, window=0, seed=0, spike=False, path=None, split_keys=None,
                    route_singles=None, pool_pages=None, spike_at=None, sink=False, spike_gain=4.0, score_shift=0.0,
                    keep_first=0, chunk=0, softcap=0.0, bias=None, pads=0):
    """Sequences of context ``lens``; the last ``q_lens[i]`` positions of each are queries.
    pool_pages: the sequences' pages are the last ones of a pool of that many.  ``spike``: the key
    at position 1 (or at ``spike_at(position of the query)``, if that is a key at all) is made to
    match its query, so that it dominates the sum if it is seen.  ``score_shift``: the first dimension of
    every key and query is set so that it takes that much off every score.  ``sink``: True for a logit of 0 in every head, or
    the heads' logits; ``softcap``: scores bent by that cap; ``bias`` [nq, reach + 1]: added by distance.  ``pads``: so many padding
    sequences of one token behind the others, which the step's facts do not list."""
    torch.manual_seed(seed)
    real = len(lens)
    q_lens = (q_lens or [1] * real) + [1] * pads
    lens = lens + [1] * pads
    S = len(lens)
    nb = max(-(-n // bs) for n in lens)
    num_blocks = S * nb + 8
    kc = torch.randn(num_blocks, bs, nkv, d, device=DEV).to(dtype)
    vc = torch.randn(num_blocks, nkv, d, bs, device=DEV).to(dtype)
    tables = torch.randperm(num_blocks, device=DEV)[:S * nb].view(S, nb).to(torch.int32)   # scattered pages
    if pool_pages:
        first = pool_pages - num_blocks
        big_k = torch.zeros(pool_pages, bs, nkv, d, dtype=dtype, device=DEV)
        big_v = torch.zeros(pool_pages, nkv, d, bs, dtype=dtype, device=DEV)
        big_k[first:], big_v[first:] = kc, vc
        kc, vc, tables = big_k, big_v, tables + first
    seq_of, pos = [], []
    for s, (n, ql) in enumerate(zip(lens, q_lens)):
        for p in range(n - ql, n):
            seq_of.append(s)
            pos.append(p)
    T = len(pos)
    q = torch.randn(T, nq * d, device=DEV).to(dtype)
    if score_shift:
        c = (score_shift * d ** 0.5) ** 0.5
        kc[..., 0] = c
        q.view(T, nq, d)[..., 0] = -c
    if spike:
        # one far key among hundreds must dominate: scale a query and a matching early key
        kflat = kc.view(-1, nkv, d)
        for t in range(T):
            s = seq_of[t]
            far = 1 if lens[s] > 2 else 0
            if spike_at is not None:
                far = spike_at(pos[t])
                if not 0 <= far < lens[s]:
                    continue
            row = int(tables[s, far // bs]) * bs + far % bs
            kflat[row] = (q[t].view(nq, d)[:nkv].float() * spike_gain).to(dtype)
    from tensorline_amd.engine.batch import StepFacts
    qs = [0]
    for ql in q_lens:
        qs.append(qs[-1] + ql)
    plan = StepFacts(max_context=max(lens), max_query_len=max(q_lens), decode_only=max(q_lens) == 1,
                     num_seqs=S, q_lens=list(q_lens[:real]), starts=[n - ql for n, ql in zip(lens, q_lens)][:real])
    single_seqs = None
    logits = None if sink is False else torch.zeros(nq) if sink is True else torch.as_tensor(sink, dtype=torch.float32)
    if K().one_token_sequences(plan):
        single_seqs = torch.tensor(K().one_token_sequences(plan), dtype=torch.int32, device=DEV)
    out = K().paged_attention(q, kc, vc, tables, torch.tensor(seq_of, dtype=torch.int32, device=DEV),
                              torch.tensor(pos, dtype=torch.int32, device=DEV), nq, nkv, d, d ** -0.5, window=window,
                              q_start=torch.tensor(qs, dtype=torch.int32, device=DEV),
                              ctx_start=torch.tensor(plan.starts + [0] * pads, dtype=torch.int32, device=DEV), plan=plan,
                              path=path, split_keys=split_keys, single_seqs=single_seqs, route_singles=route_singles,
                              sink=None if logits is None else logits.to(DEV), keep_first=keep_first, chunk=chunk, softcap=softcap,
                              bias=None if bias is None else bias.to(DEV))
    if pool_pages:
        kc, vc, tables = kc[first:], vc[first:], tables - first
    kf, vf = kc.double().cpu().view(-1, nkv, d), vc.double().cpu().permute(0, 3, 1, 2).reshape(-1, nkv, d)
    want = torch.empty(T, nq, d, dtype=torch.float64)
    tcpu = tables.cpu().long()
    t0 = 0
    for s, (n, ql) in enumerate(zip(lens, q_lens)):
        keys = torch.arange(n)
        rows = tcpu[s][keys // bs] * bs + keys % bs
        qs = q[t0:t0 + ql].double().cpu().view(ql, nq, d)
        if keep_first or chunk or softcap or bias is not None or (logits is not None and bool(logits.any())):
            want[t0:t0 + ql] = _masked_attention(qs, kf[rows], vf[rows], d ** -0.5, n - ql, window, keep_first, chunk, softcap, logits, bias)
        else:
            want[t0:t0 + ql] = plain.causal_attention(qs, kf[rows], vf[rows], d ** -0.5, window=window, q_offset=n - ql, sink=sink)
        t0 += ql
    return out.double().cpu().view(T, nq, d), want


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads", [(14, 2), (12, 2), (16, 2), (4, 4)])
@pytest.mark.parametrize("lens", [[1], [15, 16, 17], [63, 64, 65, 300], [1400] * 3 + [2, 129]])
def test_attention_decode_reference_cases(dtype, heads, lens):
    # the cases of the reference's kernel test (tests/test_paged_attn.py:22-38): D=64, page 16
    got, want = _attention_case(dtype, heads[0], heads[1], 64, 16, lens)
    torch.testing.assert_close(got, want, **tol(dtype, 2e-5, 1e-2))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("nq,nkv,d,bs", [(5, 1, 48, 16), (4, 2, 16, 8), (28, 4, 128, 16), (6, 2, 32, 8), (3, 3, 80, 4)])
def test_attention_portions_and_spike(dtype, nq, nkv, d, bs):
    lens, q_lens = [70, 9, 300, 2], [33, 9, 2, 1]
    got, want = _attention_case(dtype, nq, nkv, d, bs, lens, q_lens, spike=True, seed=3)
    torch.testing.assert_close(got, want, **tol(dtype, 3e-5, 2e-2))


def _pages_beyond_32_bits(bs, nkv, d):
    """Pages of a pool whose planes hold more than 2^31 elements (2^32 bytes and more)."""
    return (1 << 31) // (bs * nkv * d) + 4096


@pytest.mark.parametrize("dtype,path", [(torch.bfloat16, "mfma"), (torch.bfloat16, "generic"), (torch.float32, "generic")])
def test_attention_reads_pages_at_offsets_beyond_32_bits(dtype, path):
    """The sequences' pages are the last ones of a pool of several GB per plane: a page's offset in
    elements is above 2^31 and must be computed in 64 bits, in one-token steps and in portions."""
    nq, nkv, d, bs = 4, 2, 128, 16
    pool = _pages_beyond_32_bits(bs, nkv, d)
    try:
        for lens, q_lens in (([700, 33], None), ([300, 40, 65], [33, 40, 1])):
            got, want = _attention_case(dtype, nq, nkv, d, bs, lens, q_lens, spike=True, seed=11, path=path, pool_pages=pool)
            torch.testing.assert_close(got, want, **tol(dtype, 3e-5, 2e-2))
    finally:
        torch.cuda.empty_cache()


@pytest.mark.parametrize("dtype", DTYPES)
def test_cache_writes_at_offsets_beyond_32_bits(dtype):
    """The kernels that write the cache (rotation and store; the fused projections for few rows and
    for 17 to 64 rows) with slots on the last pages of a pool of several GB per plane leave there
    what they leave in a small pool, and nothing anywhere else."""
    nq, nkv, d, bs, Kd, small = 4, 2, 128, 16, 3584, 12
    pool = _pages_beyond_32_bits(bs, nkv, d)
    first = pool - small
    torch.manual_seed(4)
    inv_freq = (1e6 ** (-torch.arange(0, d, 2, dtype=torch.float64) / d)).float().to(DEV)
    N = (nq + 2 * nkv) * d
    try:
        big_k = torch.zeros(pool, bs, nkv, d, dtype=dtype, device=DEV)
        big_v = torch.zeros(pool, nkv, d, bs, dtype=dtype, device=DEV)
        for M in (5, 40):
            pos = torch.randint(0, 4000, (M,), dtype=torch.int32, device=DEV)
            slots = torch.randperm(small * bs, device=DEV)[:M].to(torch.int32)
            writers = [lambda kc, vc, sl: K().rope_store(qkv.clone(), pos, inv_freq, nq, nkv, d, kc, vc, sl)]
            qkv = torch.randn(M, N, device=DEV).to(dtype)
            if dtype == torch.bfloat16:
                h = torch.randn(M, Kd, device=DEV).to(dtype)
                ws = K().shuffle_weight((torch.randn(N, Kd, device=DEV) / math.sqrt(Kd)).to(dtype))
                b = torch.randn(N, device=DEV)
                fused = lambda kc, vc, sl: K().qkv_rope_store(h, ws, b, pos, inv_freq, nq, nkv, d, kc, vc, sl)
                assert fused(torch.zeros(small, bs, nkv, d, dtype=dtype, device=DEV),
                             torch.zeros(small, nkv, d, bs, dtype=dtype, device=DEV), slots) is not None
                writers.append(fused)
            for write in writers:
                kc = torch.zeros(small, bs, nkv, d, dtype=dtype, device=DEV)
                vc = torch.zeros(small, nkv, d, bs, dtype=dtype, device=DEV)
                write(kc, vc, slots)
                assert kc.abs().sum() > 0 and vc.abs().sum() > 0
                big_k[first:].zero_()
                big_v[first:].zero_()
                write(big_k, big_v, slots + first * bs)
                assert torch.equal(big_k[first:], kc) and torch.equal(big_v[first:], vc)
        # nothing was written below the last pages (a 32-bit offset would land there)
        assert not big_k[:first].any() and not big_v[:first].any()
    finally:
        del big_k, big_v
        torch.cuda.empty_cache()


@pytest.mark.parametrize("lens,split", [([33000], None), ([70001, 9], None), ([70001], 32)])
def test_attention_decode_long_contexts(lens, split):
    """Decoded tokens over tens of thousands of keys: hundreds of key splits, and beyond the most
    splits the merge takes the splits grow; a far key dominates."""
    got, want = _attention_case(torch.bfloat16, 28, 4, 128, 16, lens, None, spike=True, seed=5, path="mfma", split_keys=split)
    torch.testing.assert_close(got, want, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("lens,split,d,bs", [([33000], None, 128, 16), ([5000, 9, 257], None, 48, 8), ([5000, 256], 512, 64, 24),
                                              ([1300, 70], 0, 128, 16), ([700, 9, 257], None, 256, 16), ([1025], None, 144, 24)])
def test_attention_any_shape_kernel_splits_keys_in_one_token_steps(dtype, lens, split, d, bs):
    """The any-shape kernel (the float32 path's attention) in steps of one token per sequence: keys in
    runs of 256 (or as asked) at absolute positions, a work-group per run, merged by a second kernel;
    a far key dominates, contexts of a few keys beside thousands, a context that ends exactly at a
    run's edge, pages of no power of two, head sizes above 128 (tiles of 32 keys: two of the four
    waves have a key block).  0: no split, the same kernel walking all keys."""
    got, want = _attention_case(dtype, 6, 2, d, bs, lens, None, spike=True, seed=11, path="generic", split_keys=split)
    torch.testing.assert_close(got, want, **tol(dtype, 3e-5, 2e-2))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("window", [1, 100, 101, 300])
@pytest.mark.parametrize("split", [None, 64])
def test_attention_any_shape_kernel_window_with_split_keys(dtype, window, split):
    """A window in steps of one token per sequence on the any-shape kernel, where the keys are split
    into runs: the window's first key inside a run (700 keys, window 100: key 600 of the run from
    512), exactly on a run's edge (357 keys, window 101: key 256), whole leading runs empty, a
    window longer than the context.  The key just outside the window matches its query: seen, it
    would carry the sum."""
    lens = [700, 257, 256, 9, 357]
    got, want = _attention_case(dtype, 6, 2, 32, 8, lens, None, window=window, seed=21, spike=True, path="generic",
                                split_keys=split, spike_at=lambda p: p - window)
    torch.testing.assert_close(got, want, **tol(dtype, 3e-5, 2e-2))
    inside, _ = _attention_case(dtype, 6, 2, 32, 8, lens, None, window=window, seed=21, spike=True, path="generic",
                                split_keys=split, spike_at=lambda p: p - window + 1)
    if window > 1:
        assert not torch.allclose(inside, got, atol=1e-3)      # the same key one place further in is seen, and shows


@pytest.mark.parametrize("d,bs", [(128, 8), (128, 16), (128, 32), (128, 64), (128, 128), (128, 24), (64, 8), (64, 16),
                                  (64, 32), (64, 64), (32, 16), (32, 32), (32, 64), (32, 256)])
def test_attention_prompt_tiles_page_sizes_and_long_tables(d, bs):
    """Prompt portions on the kernel that stages 64-key tiles in LDS: pages smaller than, equal to
    and larger than a tile, a page table of more than 512 entries (8 and 16-token pages), a far key
    that dominates, a portion that starts and ends inside a tile, a short sequence beside it.  Pages
    of 24 tokens (no power of two) take the independent-wave kernel instead.  Where the 64 units of
    each of a wave's loads lie in one page (head size x page size >= 2048) the loader works with one
    page id per load, and the values' tile in LDS is cut by pages; elsewhere with one per lane."""
    lens, q_lens = [9000, 131, 70], [300, 131, 3]
    # 16 columns per wave, one chain of tiles per work-group and two; 32 (head sizes 64 and 128, else as before)
    for path in ("mfma-tile16", "mfma-tile16x2", "mfma-tile32"):
        got, want = _attention_case(torch.bfloat16, 28, 4, d, bs, lens, q_lens, spike=True, seed=bs, path=path)
        torch.testing.assert_close(got, want, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("path", ["generic", "mfma", "mfma-direct", "mfma-tile16x2", "mfma-tile32"])
@pytest.mark.parametrize("heads", [(14, 2), (12, 2), (16, 2), (4, 4), (28, 4)])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_attention_matrix_core_kernel(path, heads, d):
    """The matrix-core kernel against the plain attention: decode rows and prompt portions in one
    batch, scattered pages, a key that dominates, contexts around block and page edges, and the
    key range split 1, 3 and many ways."""
    dtype = torch.bfloat16
    lens = [1, 31, 32, 33, 65, 300, 1400, 2, 129]
    q_lens = [1, 1, 32, 5, 64, 1, 9, 2, 100]
    for split_keys in (0, 32, 96, None):
        got, want = _attention_case(dtype, heads[0], heads[1], d, 16, lens, q_lens, seed=7, spike=True, path=path,
                                    split_keys=split_keys)
        torch.testing.assert_close(got, want, atol=2e-2, rtol=2e-2)
    lens = [63, 64, 65, 300, 1400, 1400, 17]                  # decode only, page of 8
    for split_keys in (0, 64, 256, None):
        got, want = _attention_case(dtype, heads[0], heads[1], d, 8, lens, seed=8, path=path, split_keys=split_keys)
        torch.testing.assert_close(got, want, atol=1e-2, rtol=1e-2)
    for window in (1, 7, 32, 100):
        for split_keys in (0, 64):
            got, want = _attention_case(dtype, heads[0], heads[1], d, 16, [50, 7, 130, 700], [20, 7, 1, 33],
                                        window=window, seed=9, path=path, split_keys=split_keys)
            torch.testing.assert_close(got, want, atol=1e-2, rtol=1e-2)


@pytest.mark.parametrize("heads", [(14, 2), (4, 4), (28, 4), (40, 2)])
@pytest.mark.parametrize("d,bs", [(32, 16), (64, 24), (128, 16), (128, 8)])
def test_attention_one_token_sequences_beside_prompt_portions(heads, d, bs):
    """In a step with prompt portions the one-token sequences may be computed by a launch of their
    own with split keys (they are, by default, when their contexts are long beside the portions): first,
    last and between portions, contexts of one key and of thousands, a dominating far key, a
    window, pages of no power of two (where the portions run on independent waves)."""
    dtype = torch.bfloat16
    lens = [5000, 40, 1, 1400, 700, 31, 2, 1025]
    q_lens = [1, 40, 1, 1, 300, 1, 2, 1]
    for window in (0, 100):
        outs = []
        for route in (True, False, None):
            got, want = _attention_case(dtype, heads[0], heads[1], d, bs, lens, q_lens, window=window, seed=11,
                                        spike=window == 0, route_singles=route)
            torch.testing.assert_close(got, want, atol=2e-2, rtol=2e-2)
            outs.append(got)
        # the same with the portions on the kernel of 32 columns per wave
        got, want = _attention_case(dtype, heads[0], heads[1], d, bs, lens, q_lens, window=window, seed=11,
                                    spike=window == 0, route_singles=True, path="mfma-tile32")
        torch.testing.assert_close(got, want, atol=2e-2, rtol=2e-2)
        if window == 0:
            assert torch.equal(outs[0], outs[2])              # 5,000 keys: routed when left to choose
        portion_rows = [r for r in range(sum(q_lens)) if r not in (0, 41, 42, 343, sum(q_lens) - 1)]
        assert torch.equal(outs[0][portion_rows], outs[1][portion_rows])
    short = _attention_case(dtype, heads[0], heads[1], d, bs, [500, 40, 9], [1, 40, 1], seed=12, route_singles=None)
    unrouted = _attention_case(dtype, heads[0], heads[1], d, bs, [500, 40, 9], [1, 40, 1], seed=12, route_singles=False)
    assert torch.equal(short[0], unrouted[0])                 # short contexts stay with the portions


def _masked_attention(q, k, v, scale, q_offset, window, keep_first, chunk, softcap=0.0, logits=None, bias=None):
    """q [n, nq, d] at positions q_offset.., k and v [keys, nkv, d]: the query at position i sees key j <= i if it
    lies in the window (i - j < window) or among the first ``keep_first`` keys, and (with ``chunk``) in i's chunk.
    ``softcap`` bends the scores, ``bias`` [nq, reach + 1] is then added by distance (the last column for all farther keys),
    ``logits`` [nq] are one more entry of each head's softmax, without a value."""
    n, nq, d = q.shape
    nkv = k.shape[1]
    i = (q_offset + torch.arange(n)).view(n, 1)
    j = torch.arange(k.shape[0]).view(1, -1)
    seen = j <= i
    if window:
        seen &= (i - j < window) | (j < keep_first)
    if chunk:
        seen &= (j // chunk) == (i // chunk)
    out = torch.zeros(n, nq, d, dtype=torch.float64)
    for h in range(nq):
        g = h // (nq // nkv)
        s = (q[:, h] @ k[:, g].T) * scale
        if softcap:
            s = softcap * torch.tanh(s / softcap)
        if bias is not None:
            s = s + bias[h].double()[(i - j).clamp(0, bias.shape[1] - 1)]
        s = s.masked_fill(~seen, float("-inf"))
        if logits is not None:
            s = torch.cat((s, torch.full((n, 1), float(logits[h]), dtype=torch.float64)), dim=1)
        out[:, h] = torch.softmax(s, dim=1)[:, :k.shape[0]] @ v[:, g]
    return out


MASK_PATHS = [("generic", torch.float32), ("generic", torch.bfloat16), ("mfma-direct", torch.bfloat16),
              ("mfma-tile16", torch.bfloat16), ("mfma-tile16x2", torch.bfloat16), ("mfma-tile32", torch.bfloat16), (None, torch.bfloat16)]


@pytest.mark.parametrize("path,dtype", MASK_PATHS)
@pytest.mark.parametrize("window,keep_first,chunk", [(44, 5, 0), (100, 70, 0), (33, 1, 0), (64, 64, 0), (0, 0, 48), (0, 0, 64), (0, 0, 7)])
def test_attention_masks_in_prompt_portions(path, dtype, window, keep_first, chunk):
    """A window beside which the first keys stay in sight, and chunks of positions, in every kernel that takes
    prompt portions: portions that start at 0, behind cached tokens and in the middle of a window or chunk, beside
    one-token sequences."""
    lens, q_lens = [150, 9, 301, 77, 130], [150, 9, 40, 1, 1]
    got, want = _attention_case(dtype, 4, 2, 64, 16, lens, q_lens, window=window, seed=31, path=path, keep_first=keep_first,
                                chunk=chunk)
    torch.testing.assert_close(got, want, **tol(dtype, 3e-5, 2e-2))


@pytest.mark.parametrize("path,dtype", [("generic", torch.float32), ("generic", torch.bfloat16), ("mfma-direct", torch.bfloat16),
                                        (None, torch.bfloat16)])
@pytest.mark.parametrize("split", [None, 64])
@pytest.mark.parametrize("window,keep_first,chunk", [(44, 5, 0), (100, 70, 0), (200, 130, 0), (0, 0, 48), (0, 0, 128)])
def test_attention_masks_in_one_token_steps(path, dtype, split, window, keep_first, chunk):
    """The same masks where every sequence brings one token and the keys are split into runs: the kept first keys
    in a run of their own, in the run the window starts in, and over several runs."""
    lens = [700, 257, 256, 9, 357, 41, 130]
    got, want = _attention_case(dtype, 6, 2, 32, 8, lens, None, window=window, seed=33, path=path, split_keys=split,
                                keep_first=keep_first, chunk=chunk)
    torch.testing.assert_close(got, want, **tol(dtype, 3e-5, 2e-2))


@pytest.mark.parametrize("path,dtype", MASK_PATHS)
@pytest.mark.parametrize("where", ["first_in", "first_out", "window_in", "window_out", "chunk_in", "chunk_out"])
def test_attention_masks_show_a_loud_key_on_the_right_side_of_every_edge(path, dtype, where):
    """One key is made to match its query: the last kept first key and the one after it, the window's first key and
    the one before it, a chunk's first key and the one before it.  Seen, it carries the sum, so an edge that is
    off by one shows; prompt portions and one-token sequences."""
    window, keep_first, chunk = (0, 0, 50) if where.startswith("chunk") else (37, 5, 0)
    at = {"first_in": lambda p: keep_first - 1, "first_out": lambda p: keep_first, "window_in": lambda p: p - window + 1,
          "window_out": lambda p: p - window, "chunk_in": lambda p: (p // chunk) * chunk,
          "chunk_out": lambda p: (p // chunk) * chunk - 1}[where]
    for lens, q_lens in (([160, 99, 300], [60, 1, 1]), ([120, 333, 64], None)):
        if q_lens is None and path in ("mfma-tile16", "mfma-tile16x2", "mfma-tile32"):
            continue
        got, want = _attention_case(dtype, 4, 2, 64, 16, lens, q_lens, window=window, seed=35, spike=True, path=path,
                                    spike_at=at, keep_first=keep_first, chunk=chunk, spike_gain=6.0)
        torch.testing.assert_close(got, want, **tol(dtype, 3e-5, 2e-2))


@pytest.mark.parametrize("path", ["mfma-tile32", "mfma-tile16", "mfma-tile16x2", "mfma-direct", "generic"])
@pytest.mark.parametrize("window,keep_first,chunk", [(700, 100, 0), (300, 3, 0), (0, 0, 4096), (0, 0, 1000)])
def test_attention_masks_in_a_long_portion_behind_thousands_of_keys(path, window, keep_first, chunk):
    """1,200 tokens behind 7,800 cached ones: the kept first keys lie thousands of keys before the window, in tiles
    of their own at the head of every work-group's walk; a chunk's edge falls inside the portion."""
    got, want = _attention_case(torch.bfloat16, 8, 2, 64, 32, [9000], [1200], window=window, seed=5, path=path,
                                keep_first=keep_first, chunk=chunk)
    torch.testing.assert_close(got, want, **tol(torch.bfloat16, 3e-5, 2e-2))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("window", [1, 7, 16, 100])
def test_attention_window(dtype, window):
    got, want = _attention_case(dtype, 6, 2, 32, 8, [50, 7, 130], [20, 7, 1], window=window, seed=5)
    torch.testing.assert_close(got, want, **tol(dtype, 2e-5, 1e-2))


def test_attention_special_cases():
    # one key: o = v;  q = 0: o = mean of the visible values
    dtype, nq, nkv, d, bs = torch.float32, 4, 2, 16, 8
    kc = torch.randn(4, bs, nkv, d, device=DEV)
    vc = torch.randn(4, nkv, d, bs, device=DEV)
    tables = torch.tensor([[2, 0]], dtype=torch.int32, device=DEV)
    z = torch.zeros(1, dtype=torch.int32, device=DEV)
    q = torch.randn(1, nq * d, device=DEV)
    o = K().paged_attention(q, kc, vc, tables, z, z, nq, nkv, d, 0.25).view(nq, d)
    torch.testing.assert_close(o, vc[2, :, :, 0].repeat_interleave(2, 0), atol=1e-6, rtol=1e-6)
    p = torch.tensor([10], dtype=torch.int32, device=DEV)
    o = K().paged_attention(torch.zeros_like(q), kc, vc, tables, z, p, nq, nkv, d, 0.25).view(nq, d)
    vis = torch.cat([vc[2].permute(2, 0, 1), vc[0].permute(2, 0, 1)[:3]]).mean(0)
    torch.testing.assert_close(o, vis.repeat_interleave(2, 0), atol=1e-6, rtol=1e-6)


@pytest.mark.parametrize("dtype", DTYPES)
def test_silu_mul(dtype):
    torch.manual_seed(0)
    gu = (torch.randn(9, 2 * 176, device=DEV) * 3).to(dtype)
    got = K().silu_mul(gu)
    g, u = gu[:, :176].double(), gu[:, 176:].double()
    torch.testing.assert_close(got.double(), torch.nn.functional.silu(g) * u, **tol(dtype, 1e-5, 2e-2))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("I", [8, 1032, 2044, 2047])
def test_silu_mul_of_gates_beyond_middling_ones(dtype, I):
    """By 16 bytes, with a last thread of the row alone, and one by one; rows of middling gates beside rows with zeros, gates past where
    the exponent leaves the range, and infinities: what a row alone gives, and the float64 gate."""
    torch.manual_seed(I)
    gu = (torch.randn(5, 2 * I, device=DEV) * torch.tensor([3.0, 30.0, 90.0, 1e-20, 1.0], device=DEV)[:, None]).to(dtype)
    gu[4, :I:3], gu[4, 1:I:3], gu[4, 2] = 0.0, float("-inf"), float("inf")
    got, g, u = K().silu_mul(gu), gu[:, :I].double(), gu[:, I:].double()
    bits = torch.int16 if dtype == torch.bfloat16 else torch.int32
    assert all(torch.equal(got[t:t + 1].view(bits), K().silu_mul(gu[t:t + 1]).view(bits)) for t in range(5))
    beside = gu.clone()
    beside[:, 3:I:7] = 100.0                                          # a column's bits do not depend on the columns beside it
    kept = torch.arange(I, device=DEV) % 7 != 3
    assert torch.equal(K().silu_mul(beside)[:, kept].view(bits), got[:, kept].view(bits))
    want = g / (1 + (-g).exp()) * u
    assert torch.equal(got.isnan(), want.isnan())
    # e^-v has no float beyond 2^128: there the result is 0, for 89 / 2^128 < 2^-121 times |u| at most (|u| is up to some hundreds here)
    t = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -21
    ok = ~want.isnan() & ~want.isinf()
    assert bool(((got.double() - want).abs() <= t * want.abs() + 2.0 ** -121 * u.abs() + 2.0 ** -126)[ok].all()) and bool((got.double() == want)[want.isinf()].all())


def test_gates_of_middling_numbers_have_the_bits_of_the_general_form():
    """All 2^32 floats: of those that a wave may take the short steps for, |v| <= 40 and for SiLU 2^-60 and more, none comes out with other bits
    than by expf and the division."""
    import ctypes
    counts = torch.zeros(4, dtype=torch.int32, device=DEV)
    K()._call("tl_gate_forms_differ", ctypes.c_uint32(0), ctypes.c_longlong(1 << 32), ctypes.c_void_p(counts.data_ptr()), K()._stream())
    bits = lambda x: int(torch.tensor(x).view(torch.int32))
    silu, sigmoid, mid_silu, mid_sigmoid = (c & 0xffffffff for c in counts.tolist())
    assert (silu, sigmoid) == (0, 0)
    assert mid_silu == 2 * (bits(40.0) - bits(2.0 ** -60) + 1) and mid_sigmoid == 2 * (bits(40.0) + 1)


def test_argmax_and_ties():
    torch.manual_seed(0)
    lg = torch.randn(6, 1000, device=DEV)
    lg[2, 17] = lg[2, 900] = 50.0        # tie: the lower index wins
    got = K().argmax(lg)
    want = lg.argmax(-1)
    want[2] = 17
    assert got.tolist() == want.tolist()
    big = torch.randn(3, 152064, device=DEV)
    assert K().argmax(big).tolist() == big.argmax(-1).tolist()


def test_sample_keep_rule_and_draws():
    # hand vector of the keep rule: p = [.5, .3, .2]; top_p .5 keeps one token, .51 keeps two
    lg = torch.log(torch.tensor([[0.5, 0.3, 0.2]], device=DEV))
    one = torch.ones(1, device=DEV)
    for tp, u, want in [(0.5, 0.99, 0), (0.51, 0.99, 1), (0.51, 0.1, 0), (0.81, 0.99, 2), (1.0, 0.99, 2), (1.0, 0.6, 1)]:
        got = K().sample(lg, one, one * tp, one * u)
        assert got.tolist() == [want], (tp, u, got.tolist())
    # greedy rows inside a sampling batch, and agreement with the plain rule on random rows
    torch.manual_seed(1)
    R, V = 64, 1000
    lg = torch.randn(R, V, device=DEV) * 3
    temp = torch.rand(R, device=DEV) + 0.3
    temp[::7] = 0.0
    tp = torch.rand(R, device=DEV) * 0.9 + 0.1
    tp[::5] = 1.0
    u = torch.rand(R, device=DEV)
    got = K().sample(lg, temp, tp, u).tolist()
    miss = 0
    for r in range(R):
        want = plain.sample_with_uniform(lg[r].cpu(), float(temp[r]), float(tp[r]), float(u[r]))
        if temp[r] <= 0:
            assert got[r] == want
        elif got[r] != want:
            # a float32 running sum may land on the other side of a boundary next to the target
            probs = torch.softmax(lg[r].double().cpu() / float(temp[r]), -1)
            if tp[r] < 1:
                assert plain.top_p_keep(probs, float(tp[r]))[got[r]], "drew a token outside the kept set"
            miss += 1
    assert miss <= 2
    # same inputs, same tokens, whatever else is in the batch
    again = K().sample(lg[10:20].contiguous(), temp[10:20].contiguous(), tp[10:20].contiguous(), u[10:20].contiguous())
    assert again.tolist() == got[10:20]


def test_sample_wide_rows_ties_and_masked_logits():
    """Rows of several chunks: agreement with the plain rule, a row of equal logits (the kept set is
    a number of ties, lowest indices first), a row with all but two logits at -inf, a dominant token."""
    torch.manual_seed(4)
    V = 10007
    R = 12
    lg = torch.randn(R, V, device=DEV) * 4
    temp = torch.rand(R, device=DEV) * 1.2 + 0.2
    tp = torch.rand(R, device=DEV) * 0.95 + 0.04
    tp[::4] = 1.0
    u = torch.rand(R, device=DEV)
    got = K().sample(lg, temp, tp, u).tolist()
    miss = 0
    for r in range(R):
        want = plain.sample_with_uniform(lg[r].cpu(), float(temp[r]), float(tp[r]), float(u[r]))
        if got[r] != want:
            probs = torch.softmax(lg[r].double().cpu() / float(temp[r]), -1)
            if tp[r] < 1:
                assert plain.top_p_keep(probs, float(tp[r]))[got[r]], "drew a token outside the kept set"
            miss += 1
    assert miss <= 1
    # equal logits: top_p 0.3 keeps tokens while k / V < 0.3, that is the first 3003; u picks evenly among them
    us = torch.tensor([0.0, 0.25, 0.5, 0.999999], device=DEV)
    n = us.numel()
    flat = torch.zeros(n, V, device=DEV)
    got = K().sample(flat, torch.ones(n, device=DEV), torch.full((n,), 0.3, device=DEV), us).tolist()
    assert got == [int(float(x) * 3003) for x in us.tolist()]
    got = K().sample(flat, torch.ones(n, device=DEV), torch.ones(n, device=DEV), us).tolist()
    assert got == [int(float(x) * V) for x in us.tolist()]
    # two live tokens far apart, the rest -inf: p = (0.25, 0.75)
    two = torch.full((3, V), float("-inf"), device=DEV)
    two[:, 5000] = math.log(0.25)
    two[:, 9999] = math.log(0.75)
    one = torch.ones(3, device=DEV)
    assert K().sample(two, one, one, torch.tensor([0.1, 0.3, 0.9], device=DEV)).tolist() == [5000, 9999, 9999]
    assert K().sample(two, one, one * 0.7, torch.tensor([0.1, 0.3, 0.9], device=DEV)).tolist() == [9999] * 3
    # the vocabulary of the 7B shape: a dominant token wins whatever u is
    big = torch.randn(2, 152064, device=DEV)
    big[0, 151000] = 60.0
    big[1, 3] = 60.0
    assert K().sample(big, torch.ones(2, device=DEV), torch.tensor([0.9, 1.0], device=DEV),
                      torch.tensor([0.9999, 0.5], device=DEV)).tolist() == [151000, 3]


def test_sample_frequencies():
    torch.manual_seed(2)
    V, R = 50, 20000
    row = torch.randn(V, device=DEV) * 2
    lg = row.repeat(R, 1)
    u = torch.rand(R, device=DEV)
    t = torch.full((R,), 0.8, device=DEV)
    got = K().sample(lg, t, torch.ones(R, device=DEV), u)
    freq = torch.bincount(got.long(), minlength=V).double().cpu() / R
    probs = torch.softmax(row.double().cpu() / 0.8, -1)
    assert (freq - probs).abs().max() < 0.015
    # temperature -> 0+ is arg-max
    cold = K().sample(lg[:4], torch.full((4,), 1e-4, device=DEV), torch.ones(4, device=DEV), u[:4])
    assert cold.tolist() == [int(row.argmax())] * 4


def test_bad_arguments_are_refused():
    from tensorline_amd.ops.kernels import KernelError
    with pytest.raises(KernelError):
        K().linear(torch.randn(2, 8, device=DEV), torch.randn(4, 9, device=DEV))
    with pytest.raises(KernelError):
        K().embed(torch.zeros(2, dtype=torch.int64, device=DEV), torch.randn(4, 8, device=DEV))
    with pytest.raises(KernelError):
        K().add_rmsnorm(torch.randn(2, 8), None, torch.ones(8), 1e-6, torch.float32)
    with pytest.raises(KernelError):
        kc = torch.randn(2, 4, 1, 512, device=DEV)
        K().paged_attention(torch.randn(1, 512, device=DEV), kc, kc.permute(0, 2, 3, 1).contiguous(), torch.zeros(1, 1, dtype=torch.int32, device=DEV),
                            torch.zeros(1, dtype=torch.int32, device=DEV), torch.zeros(1, dtype=torch.int32, device=DEV),
                            1, 1, 512, 1.0)


def test_attention_long_portions_take_the_kernel_of_32_columns_per_wave(monkeypatch):
    """Left to choose, a long prompt portion behind thousands of keys runs on the kernel with 32
    columns per wave and work-groups of 256 columns, a short one on that with 16 and 128; both give
    the plain attention, a dominating far key included, and a prompt with a window too."""
    called = []
    call = K()._call
    monkeypatch.setattr(K(), "_call", lambda name, *a: (called.append(name), call(name, *a))[1])
    got, want = _attention_case(torch.bfloat16, 28, 4, 128, 16, [10000, 40], [1300, 40], spike=True, seed=4)
    torch.testing.assert_close(got, want, atol=2e-2, rtol=2e-2)
    assert called == ["tl_attention_tile32"]
    called.clear()
    got, want = _attention_case(torch.bfloat16, 28, 4, 128, 16, [3000, 40], [1300, 40], spike=True, seed=4)
    torch.testing.assert_close(got, want, atol=2e-2, rtol=2e-2)
    assert called == ["tl_attention_mfma"]
    got, want = _attention_case(torch.bfloat16, 8, 2, 64, 32, [9000], [1200], window=700, seed=5, path="mfma-tile32")
    torch.testing.assert_close(got, want, atol=2e-2, rtol=2e-2)


def test_attention_short_portions_behind_long_contexts_walk_their_keys_as_two_chains(monkeypatch):
    """Left to choose, a step with at most one work-group of 128 columns per CU and a walk of 16 tiles
    or more asks the prompt kernel for two chains of tiles per work-group, a step with more
    work-groups or only short walks for one; all give the plain attention where one far key
    dominates, with an odd number of tiles (the second chain has one fewer), a window, and a
    one-token sequence beside the portion."""
    asked = []
    call = K()._call
    monkeypatch.setattr(K(), "_call", lambda name, *a: (asked.append((name, a[25] if len(a) > 25 else None)), call(name, *a))[1])
    for lens, q_lens, window in (([4200, 40], [300, 40], 0), ([2900, 1], [64, 1], 0), ([1100], [33], 0), ([5000], [500], 700)):
        asked.clear()
        got, want = _attention_case(torch.bfloat16, 28, 4, 128, 16, lens, q_lens, window=window, spike=True, seed=6)
        torch.testing.assert_close(got, want, atol=2e-2, rtol=2e-2)
        assert asked == [("tl_attention_mfma", 2)], asked
    for lens, q_lens in (([3000, 40], [1300, 40]), ([60], [33]), ([1000, 9], [700, 9])):
        asked.clear()
        got, want = _attention_case(torch.bfloat16, 28, 4, 128, 16, lens, q_lens, spike=True, seed=4)
        torch.testing.assert_close(got, want, atol=2e-2, rtol=2e-2)
        assert asked == [("tl_attention_mfma", 1)], asked


# ---- the softmax sink: one added to the denominator, in every attention kernel ---------------------------------
SINK_CASES = [
    # (dtype, nq, nkv, d, page, lens, q_lens, window, path, split_keys)
    (torch.float32, 6, 2, 48, 8, [50, 7, 130, 700], [20, 7, 1, 33], 0, "generic", None),        # any-shape kernel, portions
    (torch.float32, 6, 2, 32, 16, [900, 3, 257], None, 0, "generic", 256),                      # its key splits and merge
    (torch.float32, 4, 4, 16, 16, [5, 1], None, 0, "generic", None),                            # its waves sharing a tile's keys
    (torch.bfloat16, 12, 2, 80, 16, [300, 9], [40, 9], 0, None, None),                            # a head size the matrix-core kernels do not take
    (torch.bfloat16, 28, 4, 128, 16, [1400, 1400, 2, 129], None, 0, "mfma", 64),                  # independent waves, splits, merge
    (torch.bfloat16, 8, 2, 64, 16, [63, 64, 65, 300], None, 0, "mfma-direct", None),              # independent waves, one run
    (torch.bfloat16, 8, 2, 64, 16, [700, 40, 9], [300, 40, 1], 0, "mfma-tile16", None),           # tiles shared through LDS
    (torch.bfloat16, 28, 4, 128, 16, [4200, 40], [300, 40], 0, "mfma-tile16x2", None),            # two chains of tiles
    (torch.bfloat16, 8, 2, 64, 32, [9000], [1200], 700, "mfma-tile32", None),                     # 32 columns per wave, a window
    (torch.bfloat16, 28, 4, 128, 16, [5000, 1, 600], [64, 1, 1], 0, None, None),                  # one-token sequences beside a portion
    (torch.bfloat16, 4, 2, 256, 16, [900, 70, 3], [200, 1, 3], 0, None, None),                    # a head size of 256: one column tile per wave
    (torch.bfloat16, 4, 1, 256, 16, [2500, 300], None, 0, "mfma", 128),                           # the same, decoded, with splits
    (torch.bfloat16, 6, 3, 192, 16, [700, 20], [100, 1], 0, None, None),                          # 192: the any-shape kernel
]


@pytest.mark.parametrize("case", range(len(SINK_CASES)))
@pytest.mark.parametrize("gain", [0.0, 4.0])
def test_attention_with_a_sink_in_every_kernel(case, gain):
    """``p_j = exp(s_j) / (1 + sum exp(s))``.  Every score has 8 taken off (a common dimension of keys and
    queries), so that the sink holds a visible share of a row's weight also among thousands of keys; with
    one key made to match its query the row's maximum is large and the sink's share nearly vanishes: both
    ends of the added term's range, in every kernel and through every merge."""
    dtype, nq, nkv, d, bs, lens, q_lens, window, path, split = SINK_CASES[case]
    kw = dict(window=window, seed=case, spike=gain > 0, path=path, split_keys=split, spike_gain=gain or 4.0, score_shift=8.0)
    got, want = _attention_case(dtype, nq, nkv, d, bs, lens, q_lens, sink=True, **kw)
    without, _ = _attention_case(dtype, nq, nkv, d, bs, lens, q_lens, sink=False, **kw)
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    torch.testing.assert_close(got, want, atol=tol, rtol=tol)
    if gain == 0:
        assert (got - without).norm() > 0.1 * without.norm(), "the sink changed nothing where it must"


@pytest.mark.parametrize("case", range(len(SINK_CASES)))
@pytest.mark.parametrize("gain", [0.0, 4.0])
def test_capped_scores_and_a_sink_per_head_in_every_kernel(case, gain):
    """``s -> cap tanh(s / cap)``, then ``p_j = exp(s_j) / (exp(sink_h) + sum exp(s))`` with a logit of each head's own, from
    one that vanishes to one that outweighs every key: in every kernel and through every merge.  With one key made to
    match its query the uncapped score would be tens; capped it is not, so a cap that is left out shows."""
    dtype, nq, nkv, d, bs, lens, q_lens, window, path, split = SINK_CASES[case]
    logits = torch.linspace(-6.0, 9.0, nq) if nq > 1 else torch.tensor([2.0])
    kw = dict(window=window, seed=case + 50, spike=gain > 0, path=path, split_keys=split, spike_gain=gain or 4.0, sink=logits)
    got, want = _attention_case(dtype, nq, nkv, d, bs, lens, q_lens, softcap=2.5, **kw)
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    torch.testing.assert_close(got, want, atol=tol, rtol=tol)
    uncapped, want = _attention_case(dtype, nq, nkv, d, bs, lens, q_lens, softcap=0.0, **kw)
    torch.testing.assert_close(uncapped, want, atol=tol, rtol=tol)
    if gain:
        assert (got - uncapped).norm() > 0.1 * uncapped.norm(), "the cap changed nothing where it must"


@pytest.mark.parametrize("path,dtype", MASK_PATHS)
def test_capped_scores_with_chunks_in_portions_and_one_token_steps(path, dtype):
    logits = torch.tensor([-1.0, 3.0, 0.5, 6.0])
    for lens, q_lens in (([160, 99, 300, 9], [60, 1, 200, 9]), ([120, 333, 64], None)):
        if q_lens is None and path in ("mfma-tile16", "mfma-tile16x2", "mfma-tile32"):
            continue
        for chunk in (50, 64, 7):
            got, want = _attention_case(dtype, 4, 2, 64, 16, lens, q_lens, seed=chunk, spike=True, path=path, chunk=chunk, spike_gain=6.0,
                                        spike_at=lambda p: (p // chunk) * chunk, softcap=9.0, sink=logits)
            torch.testing.assert_close(got, want, **tol(dtype, 3e-5, 2e-2))


@pytest.mark.parametrize("case", range(len(SINK_CASES)))
@pytest.mark.parametrize("reach", [0, 1, 40, 700])
def test_attention_with_a_bias_by_distance_in_every_kernel(case, reach):
    """A number per head and distance, the last one for all farther keys, of the scores' size and larger: in every kernel and
    through every merge, with and without cap and sink; tables that fit LDS beside the tiles and ones that do not."""
    dtype, nq, nkv, d, bs, lens, q_lens, window, path, split = SINK_CASES[case]
    torch.manual_seed(case + reach)
    bias = torch.randn(nq, reach + 1) * 3.0
    kw = dict(window=window, seed=case + 70, path=path, split_keys=split)
    tol = 2e-5 if dtype == torch.float32 else 2e-2
    got, want = _attention_case(dtype, nq, nkv, d, bs, lens, q_lens, softcap=4.0, sink=torch.linspace(-2.0, 3.0, nq) if nq > 1 else torch.tensor([1.0]),
                                bias=bias, **kw)
    torch.testing.assert_close(got, want, atol=tol, rtol=tol)
    got, want = _attention_case(dtype, nq, nkv, d, bs, lens, q_lens, bias=bias, **kw)
    torch.testing.assert_close(got, want, atol=tol, rtol=tol)
    plain_scores, _ = _attention_case(dtype, nq, nkv, d, bs, lens, q_lens, **kw)
    if reach >= 40:
        assert (got - plain_scores).norm() > 0.1 * plain_scores.norm(), "the bias changed nothing where it must"


@pytest.mark.parametrize("path,dtype", MASK_PATHS)
@pytest.mark.parametrize("window,keep_first", [(44, 5), (100, 70), (0, 0)])
def test_bias_at_every_distance_with_windows_and_kept_keys(path, dtype, window, keep_first):
    """One distance at a time stands out by so much that the key there carries the sum: the key itself, its neighbour, tiles'
    and blocks' borders, the distance before the reach, the reach and beyond it; kept first keys count their true distance."""
    reach = 90
    for at in (0, 1, 15, 16, 31, 32, 43, 63, 64, 65, 89, 90):
        if at and window and at >= window and at < reach:
            continue
        bias = torch.randn(4, reach + 1, generator=torch.Generator().manual_seed(at)) * 0.5
        bias[:, at] += 12.0
        for lens, q_lens in (([300, 99, 160, 9], [130, 1, 60, 9]), ([120, 333, 64], None)):
            if q_lens is None and path in ("mfma-tile16", "mfma-tile16x2", "mfma-tile32"):
                continue
            got, want = _attention_case(dtype, 4, 2, 64, 16, lens, q_lens, seed=at, path=path, window=window, keep_first=keep_first,
                                        softcap=9.0, sink=True, bias=bias)
            torch.testing.assert_close(got, want, **tol(dtype, 3e-5, 2e-2))


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("Kd,F,N", [(64, 64, 64), (320, 192, 320), (1024, 448, 1024)])
def test_experts_in_wide_tiles(gated, Kd, F, N, monkeypatch):
    """The grouped product's tiles of up to 256 rows: experts of no pair, one, a tile's edges and several tiles, matrices of
    fewer rows than a tile, input rows wider than K: against the sums in float64, and bit for bit what tiles of 64 rows give."""
    torch.manual_seed(F)
    loads = [0, 1, 63, 64, 65, 130, 193, 255, 256, 257, 300, 513]
    E, top = len(loads), 1
    ids = torch.tensor([e for e, n in enumerate(loads) for _ in range(n)], dtype=torch.int32)
    ids = ids[torch.randperm(len(ids))].to(DEV)[:, None].contiguous()
    T = ids.shape[0]
    h = torch.randn(T, Kd + 8, device=DEV).to(torch.bfloat16)[:, :Kd]
    up = (torch.randn(E, (2 if gated else 1) * F, Kd, device=DEV) / math.sqrt(Kd)).to(torch.bfloat16)
    down = (torch.randn(E, N, F, device=DEV) / math.sqrt(F)).to(torch.bfloat16)
    weights = torch.rand(T, top, device=DEV)
    got = {}
    for wide in (True, False):
        monkeypatch.setattr(K(), "_moe_takes_wide_tiles", lambda *a: wide)
        got[wide] = K().moe_experts(h, up, down, ids, weights, 7.0 if gated else float("inf"), 1.702 if gated else 1.0, gated=gated)
    assert torch.equal(got[True], got[False])
    want = torch.zeros(T, N, dtype=torch.float64, device=DEV)
    for e in range(E):
        rows = (ids[:, 0] == e).nonzero()[:, 0]
        z = h[rows].double() @ up[e].double().T
        if gated:
            g = z[:, :F].clamp(max=7.0)
            act = g * torch.sigmoid(1.702 * g) * (z[:, F:].clamp(-7.0, 7.0) + 1.0)
        else:
            act = z.clamp(min=0) ** 2
        # the activations are kept as bfloat16 (2^-9 of each at most): what that can move in a sum of F products
        want[rows] = weights[rows].double() * (act @ down[e].double().T)
        slack = weights[rows].double() * ((act.abs() * 2.0 ** -8 + 1e-4) @ down[e].double().abs().T) + 1e-4
        assert bool(((got[True][rows].double() - want[rows]).abs() <= slack).all()), e


@pytest.mark.parametrize("limit,alpha,shift", [(float("inf"), 1.0, 0.0), (float("inf"), 1.702, 0.0), (7.0, 1.702, 1.0)])
def test_experts_gates_of_every_size(limit, alpha, shift, monkeypatch):
    """The experts' gate for every finite bfloat16 number: sorted, so that waves of wide tiles have middling numbers only, and in disorder, so that they
    have some beyond; and in tiles of 64 rows, which know one form.  The same bits each way, and within the rounding of the result (2^-9) and
    of the float steps (of the exponent's argument, 89 at most: 2^-17; the others 2^-21); where e^-x passes the largest float the
    result is 0 for at most 89 / 2^128 < 2^-121."""
    v = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    v = v[torch.isfinite(v)].to(DEV)
    v = v[v.float().abs().sort().indices]
    T, E, Kd, F = v.numel(), 3, 64, 64
    up, down = torch.zeros(E, 2 * F, Kd, device=DEV, dtype=torch.bfloat16), torch.eye(F, device=DEV, dtype=torch.bfloat16).repeat(E, 1, 1)
    up[:, :F, 0], up[:, F:, 1] = 1, 0.75
    ids, one = (torch.arange(T, dtype=torch.int32, device=DEV) * E // T)[:, None].contiguous(), torch.ones(T, 1, device=DEV)

    def run(values, wide):
        monkeypatch.setattr(K(), "_moe_takes_wide_tiles", lambda *a: wide)
        h = torch.zeros(T, Kd, device=DEV, dtype=torch.bfloat16)
        h[:, 0], h[:, 1] = values, 1
        out = K().moe_experts(h, up, down, ids, one, limit, alpha, shift=shift)
        assert torch.equal(out[:, :1].expand_as(out), out)
        return out[:, 0].contiguous()
    got, mixed = run(v, True), torch.randperm(T, device=DEV)
    assert torch.equal(run(v[mixed], True).view(torch.int32), got[mixed].view(torch.int32))
    assert torch.equal(run(v, False).view(torch.int32), got.view(torch.int32))
    g = v.double().clamp(max=limit)
    want = g / (1 + (-alpha * g).exp()) * (0.75 + shift)
    assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -121).all())


@pytest.mark.parametrize("E,top,F,N", [(7, 1, 64, 260), (9, 3, 320, 768), (13, 2, 640, 516), (37, 33, 192, 1280), (9, 2, 2176, 4352), (15, 3, 2112, 4100)])
def test_wide_tiles_that_are_no_multiple_of_the_xcds(E, top, F, N, monkeypatch):
    """Row tiles of which fewer than eight are left over, alone or behind whole eights, whole (one to five column tiles) or dealt out over the XCDs
    (seventeen), and choices of one to many: every tile once, bit for bit what tiles of 64 rows give."""
    torch.manual_seed(E)
    T, Kd = 190, 128
    ids = torch.rand(T, E, device=DEV).topk(top, 1).indices.int().contiguous()
    h, weights = torch.randn(T, Kd, device=DEV).to(torch.bfloat16), torch.rand(T, top, device=DEV)
    up = (torch.randn(E, 2 * F, Kd, device=DEV) / 11).to(torch.bfloat16)
    down = (torch.randn(E, N, F, device=DEV) / 16).to(torch.bfloat16)
    got = {}
    for wide in (True, False):
        monkeypatch.setattr(K(), "_moe_takes_wide_tiles", lambda *a: wide)
        got[wide] = K().moe_experts(h, up, down, ids, weights, 7.0, 1.0)
    assert torch.equal(got[True], got[False])


def test_a_large_stack_of_few_experts_takes_wide_tiles(monkeypatch):
    """Four experts of 4,096 x 1,024 have 32 wide tiles for 256 CUs and take them for their size: bit for bit what small tiles give."""
    torch.manual_seed(4)
    T, E, Kd, F, top = 70, 4, 4096, 1024, 2
    ids = torch.rand(T, E, device=DEV).topk(top, 1).indices.int().contiguous()
    h, weights = torch.randn(T, Kd, device=DEV).to(torch.bfloat16), torch.rand(T, top, device=DEV)
    up = (torch.randn(E, 2 * F, Kd, device=DEV) / 64).to(torch.bfloat16)
    down = (torch.randn(E, Kd, F, device=DEV) / 32).to(torch.bfloat16)
    assert K()._moe_takes_wide_tiles(T * top, E, F, Kd)
    wide = K().moe_experts(h, up, down, ids, weights, 7.0, 1.0)
    monkeypatch.setattr(K(), "_moe_takes_wide_tiles", lambda *a: False)
    assert torch.equal(wide, K().moe_experts(h, up, down, ids, weights, 7.0, 1.0))


@pytest.mark.parametrize("N", [66, 68, 3])
def test_a_large_stack_of_experts_with_few_columns_of_result(N):
    """Stacks that take wide tiles by their size, with a result of so many columns, whole quads (which wide tiles store) or not:
    against the sums in float64."""
    torch.manual_seed(N)
    T, E, Kd, F, top = 600, 16, 1024, 1024, 2
    ids = torch.rand(T, E, device=DEV).topk(top, 1).indices.int().contiguous()
    h, weights = torch.randn(T, Kd, device=DEV).to(torch.bfloat16), torch.rand(T, top, device=DEV)
    up = (torch.randn(E, 2 * F, Kd, device=DEV) / 32).to(torch.bfloat16)
    down = (torch.randn(E, N, F, device=DEV) / 32).to(torch.bfloat16)
    got = K().moe_experts(h, up, down, ids, weights, 7.0, 1.0)
    want, slack = torch.zeros(T, N, dtype=torch.float64, device=DEV), torch.full((T, N), 1e-4, dtype=torch.float64, device=DEV)
    for e in range(E):
        rows, place = (ids == e).nonzero(as_tuple=True)
        z = h[rows].double() @ up[e].double().T
        g = z[:, :F].clamp(max=7.0)
        act, w = g * torch.sigmoid(g) * (z[:, F:].clamp(-7.0, 7.0) + 1.0), weights[rows, place].double()[:, None]
        want[rows] += w * (act @ down[e].double().T)
        # the activations are kept as bfloat16 (2^-9 of each at most): what that can move in a sum of F products
        slack[rows] += w * ((act.abs() * 2.0 ** -8 + 1e-4) @ down[e].double().abs().T)
    assert bool(((got.double() - want).abs() <= slack).all())


@pytest.mark.parametrize("keep_rows", [False, True])
def test_experts_in_passes_over_the_tokens(keep_rows, monkeypatch):
    """Where the wide tiles' offsets do not reach all rows, passes over the tokens: bit for bit what one pass gives, with input
    rows wider than K, a shared expert and its gate."""
    torch.manual_seed(8)
    T, E, Kd, F, top = 700, 16, 1024, 1024, 2
    ids = torch.rand(T, E, device=DEV).topk(top, 1).indices.int().contiguous()
    h, weights = torch.randn(T, Kd + 8, device=DEV).to(torch.bfloat16)[:, :Kd], torch.rand(T, top, device=DEV)
    up = (torch.randn(E, 2 * F, Kd, device=DEV) / 32).to(torch.bfloat16)
    down = (torch.randn(E, Kd, F, device=DEV) / 32).to(torch.bfloat16)
    extra = dict(keep_rows=True) if keep_rows else dict(shared=torch.randn(T, Kd, device=DEV), shared_gate=torch.randn(T, 3, device=DEV)[:, 1:2])
    passes = []
    run_pass = K()._experts_pass
    monkeypatch.setattr(K(), "_experts_pass", lambda *a: passes.append(a[0].shape[0]) or run_pass(*a))
    once = K().moe_experts(h, up, down, ids, weights, 7.0, 1.0, **extra)
    monkeypatch.setattr(K(), "MOE_WIDE_REACH", (256 * (E + 2) + 2 * 300) * (Kd + 8))
    parts = K().moe_experts(h, up, down, ids, weights, 7.0, 1.0, **extra)
    assert passes == [700, 300, 300, 100]
    assert torch.equal(once.rows, parts.rows) and torch.equal(parts.weights, weights) if keep_rows else torch.equal(once, parts)


@pytest.mark.parametrize("P,E,BM", [(1, 1, 16), (7, 3, 256), (1000, 70, 16), (5000, 64, 256), (12288, 64, 64), (9000, 200, 256), (3000, 1024, 16)])
def test_pairs_in_tiles_by_expert(P, E, BM):
    """The order of the pairs and the tiles made of it: every pair once, in a tile of its expert, tiles within BM rows."""
    torch.manual_seed(P)
    ids = (torch.rand(P, device=DEV) ** 2 * E).to(torch.int32).clamp(max=E - 1)
    order, tiles = torch.full((P,), -1, dtype=torch.int32, device=DEV), torch.zeros(1 + 3 * (P // BM + E), dtype=torch.int32, device=DEV)
    K()._call("tl_moe_sort", K()._ptr(ids), K()._ptr(order), K()._ptr(tiles), P, E, BM, K()._stream())
    order, tiles, ids = order.tolist(), tiles.tolist(), ids.tolist()
    assert sorted(order) == list(range(P)) and 0 < tiles[0] <= P // BM + E
    at = 0
    for t in range(tiles[0]):
        e, first, rows = tiles[1 + 3 * t:4 + 3 * t]
        assert first == at and 0 < rows <= BM and all(ids[order[p]] == e for p in range(first, first + rows))
        at += rows
    assert at == P


@pytest.mark.parametrize("nq,nkv,bs,lens,q_lens,kw", [
    (4, 1, 16, [300, 65, 64, 2], [300, 64, 17, 2], {}),                              # tiles' edges; fewer columns than a wave, a work-group
    (32, 1, 8, [700, 130], [41, 130], {}),                                           # a portion behind cached tokens, pages of 8
    (16, 2, 64, [257, 900], [257, 3], dict(window=100)),                             # two key/value heads, a window
    (8, 1, 16, [900, 64], [500, 64], dict(window=70, keep_first=5)),
    (8, 1, 16, [900, 200], [300, 200], dict(chunk=96, softcap=20.0)),
    (8, 1, 32, [400, 1, 300], [200, 1, 1], dict(sink=True)),                         # one-token requests beside a portion
    (8, 1, 24, [300], [100], {}),                                                    # pages that are no power of two: independent waves
])
def test_attention_tiles_at_head_size_256(nq, nkv, bs, lens, q_lens, kw):
    """Prompt portions at a head size of 256 on the kernel that shares key tiles through LDS (probabilities are rounded to
    bfloat16 ahead of their product with the values: 2^-9 of each, as at the other head sizes)."""
    got, want = _attention_case(torch.bfloat16, nq, nkv, 256, bs, lens, q_lens, seed=9, **kw)
    torch.testing.assert_close(got, want, **tol(torch.bfloat16, 3e-5, 2e-2))


@pytest.mark.parametrize("nq,lens,q_lens", [(16, [600], [600]), (32, [300, 803], [300, 803]), (16, [2000], [300])])
def test_attention_tiles_at_head_size_256_are_as_close_to_64_bits_as_independent_waves(nq, lens, q_lens):
    """Both round a weight to bfloat16 once; the 2-norm of the error may differ by what the order of float sums and the keys
    that set a maximum do (measured 0.5%; a running maximum that lags behind costs 3%)."""
    error = {}
    for path in ("mfma-tile16", "mfma-direct"):
        got, want = _attention_case(torch.bfloat16, nq, 1, 256, 16, lens, q_lens, seed=1, path=path)
        error[path] = (got.double() - want.double()).norm()
    assert error["mfma-tile16"] <= 1.015 * error["mfma-direct"]


@pytest.mark.parametrize("T", [1, 17, 32, 33, 130])
@pytest.mark.parametrize("B,N,Kd", [(3, 1, 8), (2, 63, 24), (3, 64, 40), (2, 65, 192), (2, 192, 128), (1, 70, 1024), (2, 40, 1032)])
def test_batched_linear_bfloat16(T, B, N, Kd):
    """The product per head: remainders of rows, columns and k, operands that are column blocks of wider rows, a K too long
    for the kernel without LDS, and rows that are not aligned (the any-shape kernel)."""
    torch.manual_seed(T + N)
    w = torch.randn(B, N, Kd, device=DEV).to(torch.bfloat16)
    for off in (0, 8, 1):
        a = torch.randn(T, B, Kd + 16, device=DEV).to(torch.bfloat16)[:, :, off:off + Kd]
        wide = torch.full((T, B, N + 3), 7.0, dtype=torch.bfloat16, device=DEV)
        got = K().batched_linear(a, w, wide[:, :, 2:N + 2])
        want = torch.stack([a[:, b].double() @ w[b].double().T for b in range(B)], 1)
        size = torch.stack([a[:, b].double().abs() @ w[b].double().abs().T for b in range(B)], 1)
        # a float sum of Kd products in any order, then one rounding to bfloat16
        assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + (Kd + 8) * 2.0 ** -24 * size).all())
        assert bool((wide[:, :, [0, 1, N + 2]] == 7.0).all())


@pytest.mark.parametrize("N,Kd", [(1, 8), (16, 32), (17, 40), (33, 520), (48, 512), (100, 1032), (40, 4104), (16 * 65535 + 5, 8)])
@pytest.mark.parametrize("dtype,step", [("bfloat16", 32), ("float32", 16)])
def test_ordered_copy_of_a_matrix(N, Kd, dtype, step):
    """The matrix-core ordered copy, made on the GPU or (rows that are not contiguous) by torch: the definition, zeros where it pads."""
    w = torch.randn(N, Kd, device=DEV).to(getattr(torch, dtype))
    make = K().shuffle_weight if dtype == "bfloat16" else K().shuffle_weight_float
    padded = torch.zeros(-(-N // 16) * 16, -(-Kd // step) * step, dtype=w.dtype, device=DEV)
    padded[:N, :Kd] = w
    want = padded.view(-1, 16, padded.shape[1] // step, 4, step // 4).permute(0, 2, 3, 1, 4)
    assert torch.equal(make(w), want)
    assert torch.equal(make(torch.cat([w, w], 1)[:, :Kd]), want)


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_ordered_copy_of_a_matrix_on_another_gpu(dtype, monkeypatch):
    """Where the matrix is not on the current GPU, whose stream a kernel of ours would run on, the copy is torch's, the same."""
    w = torch.randn(33, 72, device=DEV).to(getattr(torch, dtype))
    make = K().shuffle_weight if dtype == "bfloat16" else K().shuffle_weight_float
    want, calls = make(w), []
    monkeypatch.setattr(K(), "_call", lambda name, *a: calls.append(name))
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 1)
    assert torch.equal(make(w), want) and not calls


@pytest.mark.parametrize("T,B,N,Kd", [(1, 2, 16, 8), (31, 3, 48, 40), (33, 2, 192, 128), (130, 1, 112, 96), (2049, 32, 128, 192), (257, 32, 272, 192),
                                      (1300, 43, 128, 128)])
def test_batched_linear_by_whole_rows_and_not(T, B, N, Kd):
    """Results that are whole aligned sixteens of columns are stored by 16 bytes, from 64 rows a wave where there are many: the same
    bits as through a result that is not aligned, and within a float sum of the product in 64 bits; nothing beside them is written."""
    torch.manual_seed(T + N)
    w, a = torch.randn(B, N, Kd, device=DEV).to(torch.bfloat16), torch.randn(T, B, Kd, device=DEV).to(torch.bfloat16)
    wide = [torch.full((T, B, N + pad), 7.0, dtype=torch.bfloat16, device=DEV) for pad in (16, 3)]
    got, other = K().batched_linear(a, w, wide[0][:, :, 8:N + 8]), K().batched_linear(a, w, wide[1][:, :, 2:N + 2])
    assert torch.equal(got, other)
    for b in {0, B - 1}:
        want, size = a[:, b].double() @ w[b].double().T, a[:, b].double().abs() @ w[b].double().abs().T
        assert bool(((got[:, b].double() - want).abs() <= 2.0 ** -8 * want.abs() + (Kd + 8) * 2.0 ** -24 * size).all())
    assert bool((wide[0][:, :, :8] == 7.0).all()) and bool((wide[0][:, :, N + 8:] == 7.0).all()) and bool((wide[1][:, :, [0, 1, N + 2]] == 7.0).all())


@pytest.mark.parametrize("W,skew", [(4, 0), (1020, 0), (1024, 1), (1028, 0), (2050, 0), (2048, 0)])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_token_shift_by_quads_and_not(W, skew, dtype):
    """Rows of whole aligned quads and others: the formula in float, a sequence's first row against what its slot keeps, which its last row
    becomes."""
    import types
    torch.manual_seed(W)
    dt, lens = getattr(torch, dtype), [3, 1, 7]
    T, starts = sum(lens), [0, 3, 4, 11]
    h = torch.randn(T * W + skew, device=DEV).to(dt)[skew:].view(T, W)
    mu = torch.randn(5, W, device=DEV)
    slots = [2, 0, 1]
    dev = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    ctx = types.SimpleNamespace(num_tokens=T, num_seqs=3, seq_of_token=dev([0] * 3 + [1] + [2] * 7), q_start=dev(starts), state_slots=dev(slots))
    state = torch.randn(4, W + 9, device=DEV)
    before = torch.empty(T, W, device=DEV)
    before[1:] = h[:-1].float()
    for s in range(3):
        before[starts[s]] = state[slots[s], 5:5 + W]
    want = torch.stack([(h.float() + (before - h.float()) * mu[m]).to(dt) for m in range(5)])
    want_state = state.clone()
    for s in range(3):
        want_state[slots[s], 5:5 + W] = h[starts[s + 1] - 1].float()
    got = K().token_shift(h, mu, ctx, state, 5)
    assert torch.equal(got, want) and torch.equal(state, want_state)


@pytest.mark.parametrize("nq,nkv,d,bs,lens,q_lens,kw", [
    (12, 2, 128, 16, [3200, 40, 1, 300, 129], [70, 40, 1, 1, 129], {}),                 # behind a long context, beside one-token requests
    (12, 2, 128, 16, [3200, 40], [70, 40], dict(pads=3)),                               # beside padding sequences
    (14, 2, 64, 16, [4097, 300], [65, 1], dict(spike=True)),                            # one far key dominates
    (4, 1, 32, 8, [2048, 2047], [3, 130], {}),                                          # runs' edges
    (8, 1, 256, 16, [3000, 64], [40, 64], dict(sink=True)),
    (8, 2, 128, 16, [4000, 900], [100, 1], dict(window=1500, keep_first=70)),           # leading runs empty, first keys in a run of their own
    (8, 2, 64, 16, [4000, 2100], [100, 30], dict(chunk=1600, softcap=20.0)),
    (4, 4, 32, 64, [2500, 2000], [60, 5], dict(bias=True)),
    (6, 1, 128, 24, [3000], [40], {}),                                                  # pages of no power of two: independent waves in runs
    (4, 1, 128, 16, [3000, 1500], [4, 2], {}),                                          # one column tile of 16: independent waves in runs
])
def test_attention_portions_in_runs_of_keys(nq, nkv, d, bs, lens, q_lens, kw, monkeypatch):
    """Prompt portions of few columns behind long contexts, their walks cut into runs that a second kernel puts together; the
    one-token sequences beside them stay in the step."""
    if kw.get("bias"):
        kw = dict(kw, bias=torch.randn(nq, 41))
    chosen, choose = [], K()._attention_launch
    monkeypatch.setattr(K(), "_attention_launch", lambda *a: chosen.append(choose(*a)) or chosen[-1])
    got, want = _attention_case(torch.bfloat16, nq, nkv, d, bs, lens, q_lens, seed=21, **kw)
    launch, = chosen
    assert launch.nsplit > 1 and launch.chains > 0 and launch.own_split is None
    assert launch.nt == (1 if d == 256 or max(q_lens) * nq // nkv <= 16 else 2)
    torch.testing.assert_close(got, want, **tol(torch.bfloat16, 3e-5, 2e-2))


@pytest.mark.parametrize("runs,bs,first", [(True, 16, 3), (True, 128, 66), (False, 32, 63), (False, 128, 0)])
def test_attention_of_portions_among_many_sequences(runs, bs, first, monkeypatch):
    """Steps of more sequences than a wave has lanes, portions ahead of, between and behind one-token requests, in runs of keys
    (where the portions' work-groups come first) and in whole walks; pages smaller and larger than a tile of keys."""
    lens, q_lens = [5 + 3 * i for i in range(70)], [1] * 70
    for at, n, ql in ((first, 2100 if runs else 150, 43), (first + 1, 200, 130), (len(lens), 77, 70)):
        lens.insert(at, n), q_lens.insert(at, ql)
    chosen, choose = [], K()._attention_launch
    monkeypatch.setattr(K(), "_attention_launch", lambda *a: chosen.append(choose(*a)) or chosen[-1])
    got, want = _attention_case(torch.bfloat16, 6, 1, 128, bs, lens, q_lens, seed=bs, route_singles=None if runs else False)
    assert (chosen[0].nsplit > 1) == runs and chosen[0].chains > 0 and chosen[0].own_split is None
    torch.testing.assert_close(got, want, **tol(torch.bfloat16, 3e-5, 2e-2))


@pytest.mark.parametrize("M", [1, 5, 16])
@pytest.mark.parametrize("N,Kd", [(784, 2048), (1000, 2056), (2048, 4864), (1030, 520), (896, 2336), (1030, 776), (1030, 904)])
def test_few_rows_in_half_tiles(M, N, Kd):
    """Few-row products whose work-groups own eight columns: an N that ends in either half of a tile, a last step with one
    chunk, a part of one, or only the first of a load's two; a residual sink and the product that reads its partial
    sums.  A row has the same bits whatever rows come along."""
    torch.manual_seed(N + M)
    a = torch.randn(M, Kd, device=DEV).to(torch.bfloat16)
    w = (torch.randn(N, Kd, device=DEV) / math.sqrt(Kd)).to(torch.bfloat16)
    b = torch.randn(N, device=DEV)
    ws = K().shuffle_weight(w)
    want = a.double() @ w.double().T + b.double()
    size = a.double().abs() @ w.double().abs().T + b.double().abs()
    got = K().linear(a, w, b, out_dtype=torch.float32, shuffled=ws)
    assert bool(((got.double() - want).abs() <= (Kd + 8) * 2.0 ** -24 * size).all())     # Kd float sums in any order
    assert torch.equal(K().linear(a[M - 1:], w, b, out_dtype=torch.float32, shuffled=ws)[0], got[M - 1])
    if N % 8:
        return                                                   # (the rows a sink leaves are another product's input)
    resid, gamma = torch.randn(M, N, device=DEV), 1 + 0.1 * torch.randn(N, device=DEV)
    x = resid.clone()
    nxt = K().linear(a, w, b, shuffled=ws, sink=K().NormSink(x, gamma, 1e-6))
    torch.testing.assert_close(x.double(), resid.double() + want, atol=1e-5, rtol=1e-5)
    assert nxt.sumsq.shape[0] == -(-N // (8 if Kd >= 2048 else 16))      # 1,000: the last tile's second half has no row
    torch.testing.assert_close(nxt.sumsq.sum(0).double(), x.double().pow(2).sum(1), atol=0, rtol=1e-5)
    w2 = (torch.randn(512, N, device=DEV) / math.sqrt(N)).to(torch.bfloat16)
    got2 = K().linear(nxt, w2, None, out_dtype=torch.float32, shuffled=K().shuffle_weight(w2))
    h = (x * gamma).to(torch.bfloat16).double() / torch.sqrt(x.double().pow(2).mean(1, keepdim=True) + 1e-6)
    torch.testing.assert_close(got2.double(), h @ w2.double().T, atol=2e-4, rtol=2e-4)


@pytest.mark.parametrize("nq,nkv,d,bs", [(3, 3, 128, 4), (6, 2, 64, 16), (28, 4, 128, 16), (18, 2, 64, 8), (17, 1, 128, 512), (18, 2, 128, 8), (16, 1, 128, 512), (16, 2, 64, 8)])
@pytest.mark.parametrize("split", [None, 0, 64])
@pytest.mark.parametrize("kw", [{}, dict(sink=True), dict(window=70), dict(window=44, keep_first=5), dict(chunk=96)])
def test_float_attention_of_one_token_steps(nq, nkv, d, bs, split, kw):
    """The float kernel of steps of one token per sequence: one, four and eight heads to a work-group and a second group of one,
    contexts that end inside four keys, inside a wave's 32, at the end of a work-group's 128 and of a run, each mask,
    with runs and without.  Against 64 bits: 4,096 float roundings would be 2.4e-4; sums of random sign stay under 2e-5."""
    lens = [1, 2, 5, 31, 32, 33, 65, 127, 128, 129, 256, 257, 1030]
    got, want = _attention_case(torch.float32, nq, nkv, d, bs, lens, None, seed=nq + d, path="generic", split_keys=split, **kw)
    torch.testing.assert_close(got, want, **tol(torch.float32, 2e-5))


def test_draws_queued_one_behind_the_other_keep_their_own_numbers():
    """Draws whose numbers come from pinned memory, none awaited before the next is issued: what the kernels give for the same
    numbers in tensors of their own."""
    from tensorline_amd.sampling.sampler import Sampler, uniform_for
    torch.manual_seed(5)
    sampler, R, V = Sampler(DEV), 6, 9000
    logits = torch.randn(R, V, device=DEV) * 3
    busy = torch.randn(2048, 2048, device=DEV)
    cases = [([0.3 + 0.05 * ((i + r) % 30) if (i + r) % 5 else 0.0 for r in range(R)], [1.0 - 0.1 * ((i * r) % 7) for r in range(R)],
              [i * 100 + r for r in range(R)], [i] * R) for i in range(200)]
    got = []
    for case in cases:
        busy = torch.mm(busy, busy) * 1e-3                   # the GPU stays behind the host
        got.append(sampler.sample_device(logits, *case))
    for (temps, tops, seeds, at), tokens in zip(cases, got):
        u = [uniform_for(s, i) for s, i in zip(seeds, at)]
        t, p, x = (torch.tensor(v, dtype=torch.float32).to(DEV) for v in (temps, tops, u))
        assert torch.equal(K().sample(logits, t, p, x, any_top_p=True, any_greedy=True), tokens)


@pytest.mark.parametrize("V", [4096, 4097, 262144, 262145, 270001])
def test_sample_ties_over_one_to_more_than_64_chunks(V):
    """Equal logits: the kept set is the first tokens whose count stays under 0.3 V, across one chunk, at the edges of a
    chunk and of the 64 chunks a wave adds up at a time, and beyond; u picks evenly among them.  Whole numbers, exact."""
    us = torch.tensor([0.0, 0.25, 0.5, 0.75, 0.999999], device=DEV)
    n, kept = us.numel(), int(0.3 * V) + 1
    flat, one = torch.zeros(n, V, device=DEV), torch.ones(n, device=DEV)
    assert K().sample(flat, one, one * 0.3, us).tolist() == [int(float(x) * kept) for x in us.tolist()]
    assert K().sample(flat, one, one, us).tolist() == [int(float(x) * V) for x in us.tolist()]


def _off_by_one_float(t):
    """The same values at an address that is a multiple of 4 bytes and not of 16."""
    return torch.cat([t.new_zeros(1), t])[1:]


@pytest.mark.parametrize("M", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("N,Kd", [(160, 512), (896, 896), (1024, 2304), (512, 2688), (512, 3456), (800, 4864), (8192, 1024)])
def test_few_rows_asked_for_whole(M, N, Kd):
    """Few-row products whose waves ask for their whole share of K at once: one to four steps a wave, last waves with fewer or
    none, whole and half tiles, an owed norm with as many partial sums as there are columns / 16.  Operands at an address that the
    kernel does not take send the product to the general one, which adds in the same order: the same bits."""
    torch.manual_seed(N + M)
    a = torch.randn(M, Kd, device=DEV).to(torch.bfloat16)
    w = (torch.randn(N, Kd, device=DEV) / math.sqrt(Kd)).to(torch.bfloat16)
    b, ws = torch.randn(N, device=DEV), K().shuffle_weight(w)
    owed = K().NormedRows(a, torch.rand(Kd // 16, M, device=DEV) + 0.5, Kd, 1e-6)
    for rows in (a, owed):
        for kw in (dict(out_dtype=torch.float32), dict(out_dtype=torch.bfloat16)):
            got, general = (K().linear(rows, w, bias, shuffled=ws, **kw) for bias in (b, _off_by_one_float(b)))
            assert torch.equal(got, general)
    want, size = a.double() @ w.double().T + b.double(), a.double().abs() @ w.double().abs().T + b.double().abs()
    got = K().linear(a, w, b, out_dtype=torch.float32, shuffled=ws)
    assert bool(((got.double() - want).abs() <= (Kd + 8) * 2.0 ** -24 * size).all())     # Kd float sums in any order
    resid, gamma = torch.randn(M, N, device=DEV), 1 + 0.1 * torch.randn(N, device=DEV)
    left = []
    for g in (gamma, _off_by_one_float(gamma)):
        x = resid.clone()
        nxt = K().linear(a, w, b, shuffled=ws, sink=K().NormSink(x, g, 1e-6))
        left.append((x, nxt.rows, nxt.sumsq))
    assert all(torch.equal(x, y) for x, y in zip(*left))


@pytest.mark.parametrize("M", [1, 4, 5, 9, 16])
@pytest.mark.parametrize("I,Kd", [(2048, 1024), (3072, 1024), (4864, 896), (6144, 2048), (688, 1408)])
def test_few_rows_gated_asked_for_whole(M, I, Kd):
    """The gated form of the above in pairs of tiles and of half tiles, behind an owed norm and without, against 64 bits: gate and up are float sums of
    Kd products; then one rounding to bfloat16."""
    torch.manual_seed(I + M)
    a = torch.randn(M, Kd, device=DEV).to(torch.bfloat16)
    w = (torch.randn(2 * I, Kd, device=DEV) / math.sqrt(Kd)).to(torch.bfloat16)
    ss = torch.rand(Kd // 16, M, device=DEV) + 0.5
    for rows, factor in ((a, torch.ones(M, 1, device=DEV).double()), (K().NormedRows(a, ss, Kd, 1e-6), 1 / (ss.double().sum(0)[:, None] / Kd + 1e-6).sqrt())):
        got = K().swiglu_gate_up(rows, w, K().shuffle_weight(w))
        gate, up = ((a.double() @ w.double().T) * factor).chunk(2, 1)
        torch.testing.assert_close(got.double(), torch.nn.functional.silu(gate) * up, atol=1e-4, rtol=2.0 ** -8 + 1e-4)


@pytest.mark.parametrize("M", [1, 4, 8, 13])
@pytest.mark.parametrize("nq,nkv,d,Kd", [(14, 2, 64, 896), (3, 1, 96, 512), (12, 4, 128, 2688), (28, 4, 128, 1024), (40, 8, 128, 1024)])
def test_few_rows_qkv_asked_for_whole(M, nq, nkv, d, Kd):
    """The fused q/k/v projection of the above: whole pairs (more than 128) and halves, a head of three pairs, a row without a slot: the
    general kernel's bits, queries and both caches."""
    torch.manual_seed(d + M)
    h = torch.randn(M, Kd, device=DEV).to(torch.bfloat16)
    N = (nq + 2 * nkv) * d
    ws = K().shuffle_weight((torch.randn(N, Kd, device=DEV) / math.sqrt(Kd)).to(torch.bfloat16))
    b, pos = torch.randn(N, device=DEV), torch.randint(0, 5000, (M,), dtype=torch.int32, device=DEV)
    freq = (10000.0 ** (-torch.arange(d // 2, device=DEV).float() * 2 / d)).contiguous()
    slots = (torch.randperm(64, device=DEV)[:M]).to(torch.int32)
    slots[M // 2] = -1 if M > 1 else slots[0]
    owed = K().NormedRows(h, torch.rand(Kd // 16, M, device=DEV) + 0.5, Kd, 1e-6)
    for rows in (h, owed):
        left = []
        for bias in (b, _off_by_one_float(b)):
            kc, vc = torch.zeros(4, 16, nkv, d, dtype=torch.bfloat16, device=DEV), torch.zeros(4, nkv, d, 16, dtype=torch.bfloat16, device=DEV)
            left.append((K().qkv_rope_store(rows, ws, bias, pos, freq, nq, nkv, d, kc, vc, slots), kc, vc))
        assert all(torch.equal(x, y) for x, y in zip(*left))
        assert bool(left[0][1].any()) and bool(left[0][2].any())


@pytest.mark.parametrize("nq,nkv,d,bs", [(14, 2, 64, 16), (12, 2, 128, 16), (16, 1, 128, 64), (6, 2, 32, 32), (4, 1, 128, 8), (16, 1, 256, 16)])
@pytest.mark.parametrize("split", [32, 64, 160, 512])
@pytest.mark.parametrize("kw", [{}, dict(window=70, keep_first=5), dict(chunk=96, softcap=20.0, sink=True)])
def test_decode_attention_in_splits_of_one_wave(nq, nkv, d, bs, split, kw):
    """One-token sequences in splits of one to sixteen blocks of 32 keys (the ring of two, its remainder of none to three), contexts at the edges of a
    block, a page and a split, first keys in splits of their own, more than 64 splits (32) and few, pages of one, two and four to a block."""
    lens = [1, 2, 16, 31, 32, 33, 63, 65, 160, 161, 511, 512, 513, 700, 2049]
    got, want = _attention_case(torch.bfloat16, nq, nkv, d, bs, lens, None, seed=nq + split, split_keys=split, path="mfma", **kw)
    torch.testing.assert_close(got, want, **tol(torch.bfloat16, 3e-5, 2e-2))


@pytest.mark.parametrize("bs,blocks", [(128, 255), (256, 510), (256, 511), (128, 254), (128, 256), (64, 127)])
def test_decode_attention_in_splits_of_some_64_pages(bs, blocks):
    """Splits that begin inside a page and touch 64 pages or 65: more than a wave has lanes for their ids.  The spiked key is in the last page
    that the second split touches; chunks keep the sums to its keys."""
    split = 32 * blocks
    page = (2 * split - 1) // bs * bs
    for kw in (dict(spike=True, spike_at=lambda p: p - 3), dict(chunk=page)):
        got, want = _attention_case(torch.bfloat16, 4, 2, 64, bs, [page + 40, 2 * split, 77], None, seed=blocks, split_keys=split, path="mfma", **kw)
        torch.testing.assert_close(got, want, **tol(torch.bfloat16, 3e-5, 2e-2))


@pytest.mark.parametrize("split", [64, 512])
def test_few_tokens_in_splits_of_one_wave(split):
    """Several tokens of a sequence whose columns fit one tile of 16."""
    got, want = _attention_case(torch.bfloat16, 8, 2, 64, 16, [700, 3, 40, 1030], [4, 3, 1, 2], seed=5, split_keys=split, path="mfma")
    torch.testing.assert_close(got, want, **tol(torch.bfloat16, 3e-5, 2e-2))


@pytest.mark.parametrize("n", [64, 256, 1000, 4096])
def test_block_sums_take_every_lane_once(n):
    """The norm of rows with one entry each, at every place: an entry that a sum left out or took twice would not come out as sqrt(n)."""
    x = torch.diag(torch.linspace(1.0, 2.0, n, device=DEV))
    got = K().norm_rows(x, torch.ones(n, device=DEV), 0.0, torch.float32)
    torch.testing.assert_close(got, math.sqrt(n) * torch.eye(n, device=DEV), atol=0, rtol=5e-7)


@pytest.mark.parametrize("M", [17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("N,Kd", [(896, 896), (1026, 1032), (2048, 2048), (896, 4864), (8192, 512)])
def test_17_to_64_rows_in_tiles_of_what_is_there(M, N, Kd):
    """Two, three and four tiles of rows, with K whole and in shares, rows that end a tile and begin one, an N of no whole quads: plain, with a residual
    sink, and gate/up pairs, against 64 bits."""
    torch.manual_seed(N + M)
    a = torch.randn(M, Kd, device=DEV).to(torch.bfloat16)
    w = (torch.randn(N, Kd, device=DEV) / math.sqrt(Kd)).to(torch.bfloat16)
    b, ws = torch.randn(N, device=DEV), K().shuffle_weight(w)
    want, size = a.double() @ w.double().T + b.double(), a.double().abs() @ w.double().abs().T + b.double().abs()
    got = K().linear(a, w, b, out_dtype=torch.float32, shuffled=ws)
    assert bool(((got.double() - want).abs() <= (Kd + 8) * 2.0 ** -24 * size).all())     # Kd float sums in any order
    resid, gamma = torch.randn(M, N, device=DEV), 1 + 0.1 * torch.randn(N, device=DEV)
    x = resid.clone()
    nxt = K().linear(a, w, b, shuffled=ws, sink=K().NormSink(x, gamma, 1e-6))
    torch.testing.assert_close(x.double(), resid.double() + want, atol=1e-5, rtol=1e-5)
    assert torch.equal(nxt.rows, (x * gamma).to(torch.bfloat16))
    torch.testing.assert_close(nxt.sumsq.sum(0).double(), x.double().pow(2).sum(1), atol=0, rtol=1e-5)
    if N % 32 == 0:
        got = K().swiglu_gate_up(K().NormedRows(a, nxt.sumsq, N, 1e-6), w, ws)
        gate, up = (a.double() @ w.double().T / (x.double().pow(2).mean(1, keepdim=True) + 1e-6).sqrt()).chunk(2, 1)
        torch.testing.assert_close(got.double(), torch.nn.functional.silu(gate) * up, atol=1e-4, rtol=2.0 ** -8 + 1e-4)


@pytest.mark.parametrize("M,N,Kd", [(17, 130, 64), (32, 300, 2048), (33, 129, 2064), (97, 2051, 4112), (300, 1000, 896), (700, 5000, 2050)])
def test_linear_float_where_large_values_meet_zeros(M, N, Kd):
    """Rows whose large values meet zeros in the matrix, and the other way round, so that a result is made of values 2^-30 of their
    row's largest: the bound of K float multiply-adds all the same.  A value that is picked out of a row comes out as it is, rows and
    columns of zeros give zeros, and a row has the same bits whatever rows come along."""
    torch.manual_seed(M + Kd)
    a, w, b = torch.randn(M, Kd, device=DEV), torch.randn(N, Kd, device=DEV), torch.randn(N, device=DEV)
    a[1, ::2] *= 2.0 ** 30                                   # meets columns that are zero there
    w[3, ::2] = 0.0
    w[5, 1::2] *= 2.0 ** 40                                  # meets a row that is zero there
    a[2, 1::2] = 0.0
    a[4], w[7] = 0.0, 0.0
    w[8] = 0.0
    w[8, Kd - 1] = 1.0                                       # picks one value out of every row, the smallest too
    a[6, Kd - 1], a[9, Kd - 1] = 2.0 ** -30, 2.0 ** -100
    ws = K().shuffle_weight_float(w)
    got = K().linear(a, w, b, shuffled=ws)
    want, size = a.double() @ w.double().T + b.double(), a.double().abs() @ w.double().abs().T + b.double().abs()
    assert bool(((got.double() - want).abs() <= (Kd + 8) * 2.0 ** -24 * size).all())
    plain_sums = K().linear(a, w, shuffled=ws)
    assert bool((plain_sums[4] == 0).all()) and bool((plain_sums[:, 7] == 0).all())
    assert torch.equal(plain_sums[:, 8], a[:, Kd - 1])
    assert torch.equal(K().linear(a[:17], w, b, shuffled=ws), got[:17])


@pytest.mark.parametrize("M", [17, 32, 40, 200])
@pytest.mark.parametrize("Kd", [64, 80, 896, 2048])
def test_linear_float_keeps_all_bits_of_small_values(M, Kd):
    """Values 2^-17 to 2^-25 of their row's largest, which meets a zero, all of one sign and with the same last bits, so that what is lost of
    each would add up: the sum is off by what its own roundings make of it, six a step of 16 k, each at most 2^-24 of it and of either
    sign (four times the root of their number), and 2^-22 for the partial products that are left out.  The roles of both operands."""
    torch.manual_seed(Kd + M)
    limit = 2.0 ** -22 + 4.0 * math.sqrt(6 * Kd / 16) * 2.0 ** -24
    small = torch.empty(M, Kd, dtype=torch.float64)
    for r in range(M):                                       # multiples of 2^-38, all 2^-40 off one
        c = 2.0 ** -(17 + r % 9) * (1.0 + 0.9 * torch.rand((), dtype=torch.float64))
        small[r] = (c * 2.0 ** 38).floor() * 2.0 ** -38 + torch.randint(0, 4, (Kd,)) * 2.0 ** -38 + 2.0 ** -40
    small[:, 0] = 1.0
    small = small.float().to(DEV)
    ones = torch.ones(48, Kd, device=DEV)
    ones[:, 0] = 0.0
    want = small.double()[:, 1:].sum(1, keepdim=True)
    for a, w in ((small, ones), (ones, small)):
        got = K().linear(a, w, shuffled=K().shuffle_weight_float(w))
        off = (got if a is small else got.T).double() / want - 1.0
        assert off.shape == (M, 48) and off.abs().max().item() <= limit


def test_linear_float_of_more_rows_than_fit_a_grid_by_eights():
    """524,300 rows of a short K, one launch: every row the bits of the same row in a call of a few hundred."""
    M, N, Kd = 65535 * 8 + 20, 16, 64
    torch.manual_seed(5)
    a, w = torch.randn(M, Kd, device=DEV), torch.randn(N, Kd, device=DEV)
    ws = K().shuffle_weight_float(w)
    got = K().linear(a, w, shuffled=ws)
    for r in (0, M // 2, M - 300):
        assert torch.equal(got[r:r + 300], K().linear(a[r:r + 300].contiguous(), w, shuffled=ws))


@pytest.mark.parametrize("nq,nkv,d,bs", [(4, 4, 64, 4), (14, 2, 64, 16), (28, 4, 128, 16), (3, 1, 128, 8), (40, 2, 64, 128), (130, 1, 128, 16)])
@pytest.mark.parametrize("kw", [{}, dict(sink=True), dict(window=70), dict(window=44, keep_first=5), dict(window=9, keep_first=40), dict(chunk=96)])
def test_float_attention_of_prompt_portions(nq, nkv, d, bs, kw):
    """The float kernel of portions: columns that end within a wave's 32 and a work-group's 128, one token beside portions, keys that end
    within a page, four keys and a tile of 32, every mask.  Against 64 bits, as the one-token steps."""
    lens, q_lens = [33, 1, 32, 300, 257, 129, 70], [33, 1, 31, 65, 1, 128, 17]
    got, want = _attention_case(torch.float32, nq, nkv, d, bs, lens, q_lens, seed=nq + d, **kw)
    torch.testing.assert_close(got, want, **tol(torch.float32, 2e-5))


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("what", ["cut", "strided", "not finite", "tiny", "huge"])
def test_float_attention_of_prompt_portions_at_their_limits(d, what):
    """A position's bits do not depend on how its sequence is cut (of finite numbers that are neither all tiny nor huge), nor on rows' strides.  Infinities and NaN in a key, a value or a query give
    what plain float arithmetic gives, in the tiles and columns that see them, and every other column stays as it is; values of
    2^-70 and 2^70 are as close to 64 bits as others."""
    torch.manual_seed(d)
    nq, nkv, bs, n = 6, 2, 16, 200
    kc, vc = torch.randn(16, bs, nkv, d, device=DEV), torch.randn(16, nkv, d, bs, device=DEV)
    table = torch.randperm(16, device=DEV)[:13].to(torch.int32)[None].contiguous()
    q = torch.randn(n, nq * d, device=DEV)
    if what in ("tiny", "huge"):
        by = 2.0 ** -70 if what == "tiny" else 2.0 ** 70
        kc, q, vc = kc * by, q / by, vc * by

    def run(lo, hi, rows=None):
        from tensorline_amd.engine.batch import StepFacts
        facts = StepFacts(max_context=hi, max_query_len=hi - lo, decode_only=False, num_seqs=1, q_lens=[hi - lo], starts=[lo])
        i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device=DEV)
        return K().paged_attention(q[lo:hi] if rows is None else rows, kc, vc, table, i32(*[0] * (hi - lo)), i32(*range(lo, hi)), nq, nkv, d, d ** -0.5,
                                   q_start=i32(0, hi - lo), ctx_start=i32(lo), plan=facts)
    rows = table[0].long()
    def want():
        kf = kc[rows].view(-1, nkv, d)[:n].double().cpu()
        vf = vc[rows].permute(0, 3, 1, 2).reshape(-1, nkv, d)[:n].double().cpu()
        return plain.causal_attention(q.double().cpu().view(n, nq, d), kf, vf, d ** -0.5).reshape(n, nq * d).to(DEV)
    got = run(0, n)
    scale = vc.abs().max().item()
    torch.testing.assert_close(got.double() / scale, want() / scale, atol=2e-5, rtol=2e-5)
    if what == "cut":
        for cut in (10, 33, 100, 160):
            assert torch.equal(torch.cat((run(0, cut), run(cut, n))), got)
    if what == "strided":
        wide = torch.full((n, nq * d + 3), float("nan"), device=DEV)
        wide[:, 1:nq * d + 1] = q
        assert torch.equal(run(0, n, wide[:, 1:nq * d + 1]), got)
    if what == "not finite":
        key = 70                                             # of key/value head 1: heads 3 to 5
        page, at = int(table[0, key // bs]), key % bs
        vc[page, 1, 5, at] = float("inf")
        after = run(0, n).view(n, nq, d)
        assert bool((after[key:, 3:, 5] == float("inf")).all())
        near = key // 32 * 32                                # (what a masked weight of zero makes of an infinity in its tile is left open)
        same = torch.ones(n, nq, d, dtype=torch.bool, device=DEV)
        same[near:, 3:, 5] = False
        assert torch.equal(after[same].isfinite(), torch.ones_like(after[same], dtype=torch.bool))
        torch.testing.assert_close(after[same], got.view(n, nq, d)[same], atol=1e-5, rtol=1e-5)
        vc[page, 1, 5, at] = 1.0
        kc[page, at, 1, 7] = float("-inf")                   # a score of -inf hides the key, +inf makes the row NaN
        after, sign = run(0, n).view(n, nq, d), q.view(n, nq, d)[key:, 3:, 7] > 0
        assert bool(after[key:, 3:][sign].isfinite().all()) and bool(after[key:, 3:][~sign].isnan().all())
        assert torch.equal(after[:near], got.view(n, nq, d)[:near]) and torch.equal(after[:, :3], got.view(n, nq, d)[:, :3])
        kc[page, at, 1, 7] = 0.5
        q[40, 2 * d + 3] = float("nan")
        after, before = run(0, n).view(n, nq, d), None
        assert bool(after[40, 2].isnan().all()) and int(after.isnan().sum()) == d


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("odd", [float("nan"), float("inf"), 2.0 ** 70, 2.0 ** -60])
def test_float_attention_beside_queries_of_another_size(d, odd):
    """A query with NaN, an infinity or a number past 2^60, or a tiny one as a whole, leaves the bits of its neighbours among a wave's columns as they
    are, however the sequence is cut; itself as close to 64 bits as others where its scores are numbers."""
    from tensorline_amd.engine.batch import StepFacts
    torch.manual_seed(d)
    nq, nkv, bs, n = 6, 2, 16, 120
    kc, vc = torch.randn(8, bs, nkv, d, device=DEV), torch.randn(8, nkv, d, bs, device=DEV)
    table = torch.randperm(8, device=DEV).to(torch.int32)[None].contiguous()
    q = torch.randn(n, nq, d, device=DEV)
    def run(q, lo, hi):
        i32 = lambda *v: torch.tensor(v, dtype=torch.int32, device=DEV)
        facts = StepFacts(max_context=hi, max_query_len=hi - lo, decode_only=False, num_seqs=1, q_lens=[hi - lo], starts=[lo])
        return K().paged_attention(q[lo:hi].reshape(hi - lo, nq * d), kc, vc, table, i32(*[0] * (hi - lo)), i32(*range(lo, hi)), nq, nkv, d, d ** -0.5,
                                   q_start=i32(0, hi - lo), ctx_start=i32(lo), plan=facts).view(hi - lo, nq, d)
    before, other = run(q, 0, n), q.clone()
    at = ((3, 0), (40, 2), (41, 3), (90, 5))
    for t, h in at:
        if odd < 1.0:
            other[t, h] *= odd
        else:
            other[t, h, 7] = odd
    after, mine = run(other, 0, n), torch.zeros(n, nq, dtype=torch.bool, device=DEV)
    for t, h in at:
        mine[t, h] = True
    assert torch.equal(after[~mine], before[~mine])
    for cut in (20, 50, 100):
        cuts = torch.cat((run(other, 0, cut), run(other, cut, n)))
        assert torch.equal(cuts[~mine], before[~mine]) and torch.equal(cuts[mine].isnan(), after[mine].isnan())
        assert odd != odd or torch.equal(cuts[mine].nan_to_num(), after[mine].nan_to_num())
    if odd < 1.0:
        rows = table[0].long()
        kf, vf = kc[rows].view(-1, nkv, d)[:n].double().cpu(), vc[rows].permute(0, 3, 1, 2).reshape(-1, nkv, d)[:n].double().cpu()
        want = plain.causal_attention(other.double().cpu(), kf, vf, d ** -0.5).to(DEV)
        torch.testing.assert_close(after.double(), want, atol=2e-5, rtol=2e-5)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("size", [-20, -76, -109, -112, -118, -126])
@pytest.mark.parametrize("dims", ["one", "all"])
def test_float_attention_of_values_of_every_size(d, size, dims):
    """A head dimension whose values are all some power of two, down to the smallest normal float, beside others or alone: as close to 64 bits as any,
    where what is left of 24 bits is a normal float (a result below 2^-126 is off by up to 2^-149)."""
    torch.manual_seed(d)
    nq, bs, n = 2, 16, 96
    kc, vc = torch.randn(6, bs, nq, d, device=DEV), torch.rand(6, nq, d, bs, device=DEV) + 1.0
    at = slice(None) if dims == "all" else 5
    vc[:, :, at] *= 2.0 ** size
    table, q = torch.randperm(6, device=DEV).to(torch.int32)[None].contiguous(), torch.randn(n, nq, d, device=DEV)
    from tensorline_amd.engine.batch import StepFacts
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    facts = StepFacts(max_context=n, max_query_len=n, decode_only=False, num_seqs=1, q_lens=[n], starts=[0])
    got = K().paged_attention(q.view(n, nq * d), kc, vc, table, i32([0] * n), i32(list(range(n))), nq, nq, d, d ** -0.5,
                              q_start=i32([0, n]), ctx_start=i32([0]), plan=facts).view(n, nq, d)
    rows = table[0].long()
    want = plain.causal_attention(q.double().cpu(), kc[rows].view(-1, nq, d).double().cpu(), vc[rows].permute(0, 3, 1, 2).reshape(-1, nq, d).double().cpu(), d ** -0.5).to(DEV)
    torch.testing.assert_close(got.double()[:, :, at] * 2.0 ** -size, want[:, :, at] * 2.0 ** -size, atol=2.0 ** (-149 - size), rtol=2e-6)


@pytest.mark.parametrize("form", ["decay", "channels", "steps"])
@pytest.mark.parametrize("dk,dv", [(16, 16), (24, 40), (64, 64), (128, 17)])
def test_recurrences_of_portions_with_helping_waves(form, dk, dv):
    """Sequences that end at a chunk of 16 tokens, one behind it and far behind it, zeros and numbers past 40 among the inputs: the waves
    that bring the chunks and write the outputs change no bit of them nor of the states (a caller that does not say how many
    tokens come gets none), whatever the cutting."""
    from types import SimpleNamespace
    torch.manual_seed(dk + dv)
    heads, lens = 3, [1, 16, 17, 32, 33, 100]
    T, S = sum(lens), len(lens)
    q, k, v = torch.randn(T, heads * dk, device=DEV), 0.1 * torch.randn(T, heads * dk, device=DEV), torch.randn(T, heads * dv, device=DEV)
    q[5], k[7, ::2], v[20, 0], q[30, 1], q[31, 2] = 0.0, -0.0, 70.0, -70.0, 1e-30
    kw = {"decay": dict(decay=torch.rand(heads, device=DEV), silu_inputs=True),
          "channels": dict(wlog=torch.randn(T, heads * dk, device=DEV), bonus=torch.randn(heads, dk, device=DEV)),
          "steps": dict(steps=torch.randn(T, heads, device=DEV), rate_log=torch.randn(heads, device=DEV), step_bias=torch.randn(heads, device=DEV),
                        skip=torch.randn(heads, device=DEV))}[form]
    starts = [0]
    for n in lens:
        starts.append(starts[-1] + n)
    def run(longest):
        state = torch.linspace(-1, 1, S * heads * dk * dv, device=DEV).view(S, -1).contiguous()
        facts = None if longest is None else SimpleNamespace(max_query_len=longest, decode_only=True)     # (decode_only: no chunked form of steps)
        ctx = SimpleNamespace(num_seqs=S, state_slots=torch.arange(S, dtype=torch.int32, device=DEV), facts=facts,
                              q_start=torch.tensor(starts, dtype=torch.int32, device=DEV))
        return K().linear_recurrence(q, k, v, ctx, state, heads, dk, dv, **kw), state
    (out, state), (want, want_state) = run(max(lens)), run(None)
    assert torch.equal(out.view(torch.int32), want.view(torch.int32)) and torch.equal(state.view(torch.int32), want_state.view(torch.int32))


@pytest.mark.parametrize("what", ["dyt", "cast", "clamp", "gate", "latent"])
@pytest.mark.parametrize("rows,width", [(1, 4), (3, 1020), (5, 2052)])
def test_four_values_at_a_time_and_one(what, rows, width):
    """Rows of aligned quads, and the same numbers where an access of four would be misaligned: the same bits, and within a rounding to
    bfloat16 (2^-8 of the value) of the expression in 64 bits."""
    k, bf = K(), torch.bfloat16
    torch.manual_seed(rows)
    def placed(t, off):                                      # contiguous, `off` numbers behind an aligned address
        room = torch.empty(t.numel() + off, dtype=t.dtype, device=DEV)
        room[off:] = t.flatten()
        return room[off:].view(t.shape)
    x, y, w, b = torch.randn(rows, width, device=DEV), torch.randn(rows, width, device=DEV), torch.randn(width, device=DEV), torch.randn(width, device=DEV)
    gu = 4.0 * torch.randn(rows, 2 * width, device=DEV)
    gu[0, 0], gu[0, 1], gu[0, 2], gu[0, 3] = float("inf"), -300.0, 0.0, float("nan")
    gate = torch.randn(rows, 4, device=DEV)
    proj, alpha = torch.randn(rows, 2 * 48 + 24 + 16, device=DEV), torch.tensor([0.6], device=DEV)
    def run(off):
        if what == "dyt":
            a = placed(x, off)
            return k.add_dyt(a, placed(y, off), w, b, alpha, bf), a
        if what == "cast":
            a = placed(x, off)
            return k.add_cast(a, placed(y, off), bf), a
        if what == "clamp":
            return k.clamp_glu(placed(gu, off), 7.0, 1.702, bf), placed(gu.to(bf), off)
        if what == "gate":
            return k.head_gate(placed(x.to(bf), off), gate, 4), gate
        kc, vc = torch.zeros(1, 16, 1, 48, dtype=bf, device=DEV), torch.zeros(1, 1, 48, 16, dtype=bf, device=DEV)
        n = torch.arange(rows, dtype=torch.int32, device=DEV)
        plain, lat = k.latent_prepare(placed(proj, off), 7 * n, torch.linspace(0.01, 1, 8, device=DEV), 1.25, w[:1].expand(24).contiguous(), 1e-5, n, kc, vc, 2, 32, 16, 24)
        return plain, torch.cat([lat.view(rows, -1, 48)[:, :, 24:].flatten(), kc.flatten()])
    got, one = run(0), run(1)
    assert all(torch.equal(g.view(torch.int16) if g.dtype == bf else g.view(torch.int32), o.view(torch.int16) if o.dtype == bf else o.view(torch.int32))
               for g, o in zip(got, one))
    s = (x + y).double()
    if what == "dyt":
        want = torch.tanh(0.6 * s) * w.double() + b.double()
    elif what == "cast":
        want = s
    elif what == "clamp":
        g, u = gu[:, :width].double(), gu[:, width:].double()
        g = torch.where(g.isnan(), 7.0, g.clamp(max=7.0))    # (the smaller of NaN and the limit is the limit)
        want = g * torch.sigmoid(1.702 * g) * (u.clamp(-7.0, 7.0) + 1.0)
    elif what == "gate":
        want = (x.to(bf).double().view(rows, 4, -1) * torch.sigmoid(gate.double()).unsqueeze(2)).view(rows, width)
    else:
        want = proj[:, :96].reshape(rows, 2, 48)[:, :, :32].reshape(rows, 64).double()
    torch.testing.assert_close(got[0].double(), want, rtol=2 ** -8, atol=2e-6)


@pytest.mark.parametrize("rows,width", [(1, 4), (255, 4), (257, 4), (65, 16), (33, 64), (17, 68), (3, 512), (5, 516), (2, 1024), (3, 1028)])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_narrow_rows_share_a_work_group(rows, width, dtype):
    """The clamped gate and the gate of heads over rows from one quad to more than a work-group's 256: the bits of one number at a time, and
    nothing beside the rows is written."""
    k, dt = K(), getattr(torch, dtype)
    torch.manual_seed(rows + width)
    gu, heads = 4.0 * torch.randn(rows, 2 * width, device=DEV), 1 if width % 16 else width // 16
    room = torch.empty(gu.numel() + 1, dtype=dt, device=DEV)
    room[1:] = gu.to(dt).flatten()
    assert torch.equal(k.clamp_glu(gu.to(dt), 7.0, 1.702), k.clamp_glu(room[1:].view(rows, 2 * width), 7.0, 1.702))
    gate, x = torch.randn(rows, heads, device=DEV), torch.randn(rows, width, device=DEV).to(dt)
    both = torch.full((2, rows * width + 8), 3.0, dtype=dt, device=DEV)
    outs = []
    for room, off in zip(both, (4, 5)):                      # (a row of `both` starts at a whole quad)
        o = room[off:off + rows * width].view(rows, width)
        o.copy_(x)
        outs.append(k.head_gate(o, gate, heads))
        assert bool((room[:off] == 3.0).all()) and bool((room[off + rows * width:] == 3.0).all())
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("halves", [False, True])
@pytest.mark.parametrize("d,dv,D,turned", [(128, 128, 128, 64), (50, 40, 64, 20), (63, 63, 63, 30), (200, 256, 256, 200)])
def test_heads_of_small_and_large_steps_alike(d, dv, D, turned, halves):
    """A head of up to 128 dimensions has 64 lanes in a small step and 16 in a large one, accesses of two numbers where sizes and addresses are
    even: the same bits of queries, keys and values."""
    H, G, T, page, few = 5, 2, 672, 16, 300
    assert [K().library().tl_head_lanes(t, H + G, D) for t in (few, T)] == ([64, 16] if D <= 128 else [64, 64])
    torch.manual_seed(d)
    cols = (H + G) * d + G * dv
    proj, wide = torch.randn(T, cols + cols % 2, device=DEV), torch.empty(T, cols + 3 - cols % 2, device=DEV)
    wide[:, 1:cols + 1] = proj[:, :cols]
    n = torch.arange(T, dtype=torch.int32, device=DEV)
    slots, freq = n.flip(0).contiguous(), torch.linspace(0.01, 1.0, turned // 2, device=DEV)
    slots[3] = -1
    w = torch.randn(2, d, device=DEV)
    def run(x):
        t = x.shape[0]
        kc, vc = torch.zeros(T // page, page, G, D, dtype=torch.bfloat16, device=DEV), torch.zeros(T // page, G, D, page, dtype=torch.bfloat16, device=DEV)
        q = K().head_norm_rotate_store(x, n[:t], w[0].contiguous(), w[1].contiguous(), 1e-5, freq, 1.1, kc, vc, slots[:t], H, G, d, dv, False, torch.bfloat16, halves=halves)
        return q, kc.view(-1, G, D), vc.permute(0, 3, 1, 2).reshape(-1, G, D)
    (q, kc, vc), (q1, kc1, vc1), (q2, kc2, vc2) = run(proj), run(wide[:, 1:cols + 1]), run(proj[:few])
    assert torch.equal(q, q1) and torch.equal(kc, kc1) and torch.equal(vc, vc1)
    assert torch.equal(q[:few], q2) and torch.equal(kc[T - few:], kc2[T - few:]) and torch.equal(vc[T - few:], vc2[T - few:])   # (token i's slot: T - 1 - i)
    x = proj[:, :H * d].double().view(T, H, d)
    x = x / torch.sqrt(x.square().mean(2, keepdim=True) + 1e-5) * w[0].double()
    angle = (n.unsqueeze(1).float() * freq).double()
    cs, sn = 1.1 * angle.cos().unsqueeze(1), 1.1 * angle.sin().unsqueeze(1)
    a, b = (x[:, :, :turned // 2], x[:, :, turned // 2:turned]) if halves else (x[:, :, :turned:2], x[:, :, 1:turned:2])
    ra, rb = a * cs - b * sn, b * cs + a * sn
    rot = torch.cat([ra, rb], 2) if halves else torch.stack([ra, rb], 3).flatten(2)
    want = torch.nn.functional.pad(torch.cat([rot, x[:, :, turned:]], 2), (0, D - d))
    torch.testing.assert_close(q.view(T, H, D).double(), want, rtol=2 ** -8, atol=2e-5)


@pytest.mark.parametrize("pairs,experts,tile", [(1, 1, 16), (257, 8, 16), (1023, 64, 64), (1024, 3, 64), (4095, 64, 64), (4096, 64, 256), (16385, 256, 256), (40000, 64, 256)])
def test_pairs_sorted_by_expert(pairs, experts, tile):
    """Numbers of pairs on both sides of what the sort's threads keep: every pair once, among its expert's, the tiles cover them in order;
    experts out of range are left out."""
    k = K()
    ids = torch.randint(0, experts, (pairs,), generator=torch.Generator().manual_seed(pairs)).to(torch.int32)
    if pairs > 300:
        ids[::97], ids[5] = -1, experts
    order, tiles = torch.full((pairs,), -1, dtype=torch.int32, device=DEV), torch.zeros(1 + 3 * (pairs // tile + experts), dtype=torch.int32, device=DEV)
    dev = ids.to(DEV)
    k._call("tl_moe_sort", k._ptr(dev), k._ptr(order), k._ptr(tiles), pairs, experts, tile, k._stream())
    order, tiles = order.cpu().long(), tiles.cpu()
    at = covered = 0
    for e in range(experts):
        mine = (ids == e).nonzero().flatten()
        assert torch.equal(order[at:at + mine.numel()].sort().values, mine)
        rows = [r for r in tiles[1:1 + 3 * int(tiles[0])].view(-1, 3).tolist() if r[0] == e]
        assert sum(r[2] for r in rows) == mine.numel() and all(0 < r[2] <= tile for r in rows)
        for _, first, n in rows:
            assert first == at
            at += n
        covered += len(rows)
    assert covered == int(tiles[0]) and bool((order[at:] == -1).all())


@pytest.mark.parametrize("glu", [0, 1, 2])
def test_wide_expert_tiles_of_every_height(glu):
    """Experts whose rows end at each height a wide tile is multiplied in and one beyond it: the bits of the tiles of 64 rows, which take the
    same sums in the same order."""
    k, (N, W) = K(), (260, 192)
    rows = [1, 64, 65, 96, 97, 128, 129, 160, 161, 192, 193, 224, 225, 256, 257]
    E, P = len(rows), sum(rows)
    torch.manual_seed(glu)
    ids = torch.repeat_interleave(torch.arange(E), torch.tensor(rows)).to(torch.int32).to(DEV)
    a = torch.randn(P, W, device=DEV).to(torch.bfloat16)
    w = (0.1 * torch.randn(E, (2 if glu == 1 else 1) * N, W, device=DEV)).to(torch.bfloat16)
    f = ctypes.c_float
    def run(tile):
        most = P // tile + E
        order, tiles = torch.empty(P, dtype=torch.int32, device=DEV), torch.empty(1 + 3 * most, dtype=torch.int32, device=DEV)
        k._call("tl_moe_sort", k._ptr(ids), k._ptr(order), k._ptr(tiles), P, E, tile, k._stream())
        order.copy_(torch.arange(P))                         # (the sort leaves open where in its expert's places a pair goes)
        out = torch.zeros(P, N, dtype=torch.bfloat16 if glu else torch.float32, device=DEV)
        k._call("tl_moe_gemm", k._ptr(a), k.BF16, W, k._ptr(w), k.BF16, k._ptr(out), k.BF16 if glu else k.F32, N, k._ptr(order), k._ptr(tiles),
                most, E, tile, 1, N, W, glu, f(7.0), f(1.702), f(1.0), k._stream())
        return out
    got, want = run(256), run(64)
    assert torch.equal(got.float(), want.float()) and bool(got.isfinite().all()) and bool((got != 0).any(1).all())
