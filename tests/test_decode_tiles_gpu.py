"""The decode kernel's tiles in LDS (csrc/decode.hip): its 16- and 32-column
blocks, 16-byte and 4-byte plane loads, the waves' shares of a tile at every
bit width, ranges of one to a few tiles, and scale groups past the ones kept in
flight, against the float64 oracle at the tolerance of the other products."""
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
    partial last one (N / 16 = 1804 word columns), and more scale groups than a
    thread keeps in flight."""
    _check(M, 2048, 28864, 8, gs, "float16", mode)


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
