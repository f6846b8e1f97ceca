"""The decode kernel's tiles (csrc/decode.hip): its 16- and 32-column blocks,
plane words through LDS by 16-byte and 4-byte loads and straight into
registers, the waves' shares of a tile at every bit width, ranges of one to
many tiles, scale groups past the ones kept in flight and waits that expire,
against the float64 oracle at the tolerance of the other products."""
import numpy as np
import pytest
import torch

from tests._helpers import assert_output_close, own_product, rand_weight, to_dtype_np, TORCH_DTYPES

pytestmark = pytest.mark.gpu


def _check(M, K, N, b, gs, dtype, mode, shift=0):
    from grinqh.kernel import run_product
    from grinqh.utils import prepare_weight
    rng = np.random.default_rng(M * 7 + K + N + b)
    W = rand_weight(rng, K, N, b)
    s = to_dtype_np(np.abs(rng.standard_normal((-(-K // gs), N))) * 0.02 + 1e-3, dtype)
    x = to_dtype_np(rng.standard_normal((M, K)), dtype)
    t = [0.0, 1.2, 1.9, 2.4]
    P = prepare_weight(torch.from_numpy(W).cuda(), b)
    if shift:  # planes that are not 16-byte aligned take the 4-byte loads
        buf = torch.empty(P.numel() + shift, dtype=torch.int32, device="cuda")
        buf[shift:] = P.view(torch.int32).reshape(-1)
        P = buf[shift:].view(P.shape)
    dt = TORCH_DTYPES[dtype]
    xt, st = torch.from_numpy(x).to(dt).cuda(), torch.from_numpy(s).to(dt).cuda()
    y = run_product(xt, P, st, None, b, gs, N // 4, t, mode)
    again = run_product(xt, P, st, None, b, gs, N // 4, t, mode)
    torch.cuda.synchronize()
    assert torch.equal(y, again), "not repeatable"
    pre = own_product(x, W, s, t, b, gs, dtype, mode == "union")
    assert_output_close(y, pre, to_dtype_np(pre, dtype), dtype, what=f"{M}x{K}x{N} b={b} {mode}")


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("mode", ["union", "dense"])
@pytest.mark.parametrize("b", [2, 4, 6, 8])
@pytest.mark.parametrize("M", [5, 16, 17, 32, 33, 64])
def test_shares_of_a_tile(M, b, mode, dtype):
    """Every bit width (2 to 32 KiB of plane words per tile set) at the edges
    of the row ranges; 5 tiles of K leave some sub-ranges one tile, some two."""
    _check(M, 160, 1024, b, 32, dtype, mode)


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("M,K,N", [(16, 32, 64), (32, 64, 16), (7, 2080, 6160), (20, 1056, 4112), (64, 1056, 400)])
def test_ragged(M, K, N, dtype):
    """One tile in all, row widths that are not whole 16-byte pieces, and a
    last column block of a few word columns."""
    _check(M, K, N, 8, 128, dtype, "union")


@pytest.mark.parametrize("M", [9, 30, 64])
def test_unaligned_planes(M):
    _check(M, 512, 1024, 8, 64, "float16", "union", shift=1)


@pytest.mark.parametrize("mode", ["union", "dense"])
@pytest.mark.parametrize("M,gs", [(16, 32), (16, 128), (30, 32), (30, 128)])
def test_wide_column_blocks(M, gs, mode):
    """Weights large enough for 32-column blocks in the dense dispatch, with a
    partial last one (N / 16 = 1804 word columns)."""
    _check(M, 2048, 28864, 8, gs, "float16", mode)


# ---- large weights: every block runs many tiles, the oracle a part of the columns

_LARGE = {}


def _large(K, N, b):
    """A weight shared by the cases of one shape and width: codes of the
    checked columns (the first, some in the middle and the last word columns of
    all 16 column tiles), and the planes of all."""
    from grinqh.utils import prepare_weight
    key = (K, N, b)
    if key not in _LARGE:
        _LARGE.clear()
        g = torch.Generator(device="cuda").manual_seed(K + N + b)
        W = torch.randint(-(1 << (b - 1)), 1 << (b - 1), (K, N), generator=g, device="cuda", dtype=torch.int8)
        NW = N // 16
        words = np.r_[0:20, NW // 2:NW // 2 + 20, NW - 20:NW]
        cols = (np.arange(16)[:, None] * NW + words[None, :]).reshape(-1)
        ct = torch.from_numpy(cols).cuda()
        _LARGE[key] = (prepare_weight(W, b), W[:, ct].cpu().numpy(), ct)
    return _LARGE[key]


def _check_large(M, K, N, b, gs, dtype, mode):
    from grinqh.kernel import run_product
    P, W, ct = _large(K, N, b)
    rng = np.random.default_rng(M + b)
    s = to_dtype_np(np.abs(rng.standard_normal((-(-K // gs), N))) * 0.02 + 1e-3, dtype)
    x = to_dtype_np(rng.standard_normal((M, K)), dtype)
    t = [0.0] + np.quantile(np.abs(x).max(0), [0.5, 0.8, 0.95]).tolist()
    dt = TORCH_DTYPES[dtype]
    xt, st = torch.from_numpy(x).to(dt).cuda(), torch.from_numpy(s).to(dt).cuda()
    y = run_product(xt, P, st, None, b, gs, N // 4, t, mode)
    again = run_product(xt, P, st, None, b, gs, N // 4, t, mode)
    torch.cuda.synchronize()
    assert torch.equal(y, again), "not repeatable"
    cols = ct.cpu().numpy()
    pre = own_product(x, W, s[:, cols], t, b, gs, dtype, mode == "union")
    assert_output_close(y[:, ct], pre, to_dtype_np(pre, dtype), dtype, what=f"{M}x{K}x{N} b={b} {mode} {dtype}")


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("mode", ["union", "dense"])
@pytest.mark.parametrize("M", [16, 32, 64])
@pytest.mark.parametrize("N", [28864, 28848])
@pytest.mark.parametrize("b", [2, 4, 6, 8])
def test_slots_are_reused(b, N, M, mode, dtype):
    """1000 and more rows of K per block, 8 to 16 tiles and more per sub-range:
    every LDS slot and tile buffer is filled and read several times, at every
    bit width (uneven shares among four waves at 6 bits in bf16), with 16-byte
    plane loads (28864 columns; dense 4-8 bits at 16 rows and 6-8 bits at 32:
    blocks of 32 word columns) and 4-byte or direct ones (28848)."""
    _check_large(M, 4096, N, b, 128, dtype, mode)


@pytest.mark.parametrize("mode", ["union", "dense"])
@pytest.mark.parametrize("M", [16, 30, 64])
def test_scale_groups_past_the_ones_in_flight(M, mode):
    """Groups of 32 rows: 64 per block (graded, and 33-64 rows) where a thread
    keeps 32 in flight, 32 per block of 32 word columns where it keeps 24."""
    _check_large(M, 4096, 28864, 8, 32, "float16", mode)


@pytest.mark.parametrize("M", [20, 64])
def test_overflow_guard_sees_late_scale_groups(M):
    """The one scale past the fp16 weight range lies in group 40 of its block,
    stored ahead of the first barrier with the groups that are not kept in
    flight."""
    from grinqh.kernel import grinqh_gemv_batch_union
    from oracle import grinqh_oracle as O
    K, N, b, gs = 4096, 28864, 8, 32
    P, W, ct = _large(K, N, b)
    cols = ct.cpu().numpy()
    rng = np.random.default_rng(M)
    s = np.full((K // gs, N), 0.25)
    s[40, cols[::3]] = 1500.0
    x = to_dtype_np(rng.standard_normal((M, K)) * 1e-3, "float16")
    t = [0.0] + np.quantile(np.abs(x).max(0), [0.5, 0.8, 0.95]).tolist()
    y = grinqh_gemv_batch_union(torch.from_numpy(x).half().cuda(), P, torch.from_numpy(s).half().cuda(), None, b, gs,
                                N // 4, t)
    weff = O.effective_weight(W, O.grade(O.union_sigma(x), t, b), b).astype(np.float64)
    m, e = np.frexp(weff * np.repeat(s[:, cols], gs, axis=0))  # 11 significant bits, no exponent limit
    pre = x @ np.ldexp(np.round(m * 2.0 ** 11) / 2.0 ** 11, e)
    assert np.abs(pre).max() < 65504
    assert_output_close(y[:, ct], pre, to_dtype_np(pre, "float16"), "float16", what=f"late scale group M={M}")


@pytest.mark.parametrize("dtype", ["float16", "bfloat16"])
@pytest.mark.parametrize("M,K,N,mode", [
    (5, 32, 64, "dense"), (16, 1024, 1024, "dense"), (9, 2048, 28864, "union"), (32, 2048, 28864, "dense"),
    (32, 2048, 28864, "union"), (33, 160, 400, "dense"), (33, 160, 400, "union"), (64, 2048, 1024, "union")])
def test_expired_wait_gives_nan(M, K, N, mode, dtype):
    """(Forms that share tiles.)  A wait for another wave's share of a tile that
    expires (here: is taken to) turns its block's outputs into NaN, and the next
    call is whole again."""
    from grinqh import _lib
    from grinqh.kernel import run_product
    from grinqh.utils import prepare_weight
    lib = _lib.load_library()
    rng = np.random.default_rng(M + K + N)
    P = prepare_weight(torch.from_numpy(rand_weight(rng, K, N, 8)).cuda(), 8)
    dt = TORCH_DTYPES[dtype]
    s = torch.full((-(-K // 32), N), 0.01, dtype=dt, device="cuda")
    x = torch.from_numpy(rng.standard_normal((M, K))).to(dt).cuda()
    call = lambda: run_product(x, P, s, None, 8, 32, N // 4, [0.0, 1.2, 1.9, 2.4], mode)
    want = call()
    assert lib.grinqh_expire_tile_waits(1) == 0
    try:
        got = call()
    finally:
        assert lib.grinqh_expire_tile_waits(0) == 1
    after = call()
    torch.cuda.synchronize()
    assert bool(want.isfinite().all())
    assert bool(got.isnan().all())
    assert torch.equal(after, want)
