"""bf16 results are rounded to nearest even by the conversion instruction: every
bf16 scale (subnormals, infinities and NaN among them) times integer weights
against the same products rounded on the CPU."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path", ["dequantize", "one_row"])
def test_every_bf16_scale(path):
    from grinqh.kernel import run_product
    from grinqh.utils import dequantize, prepare_weight
    K, N = 32, 65536
    w = torch.tensor([-128, -127, -77, -64, -3, -2, -1, 0, 1, 2, 3, 5, 63, 64, 77, 127] * 2, dtype=torch.int8)
    W = w.unsqueeze(1).expand(K, N).contiguous()
    s = torch.arange(N, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).unsqueeze(0).contiguous()
    P = prepare_weight(W.cuda(), 8)
    if path == "dequantize":
        got = dequantize(P, s.cuda(), 8, 32, N // 4).cpu()
        ref = (W.float() * s.float()).to(torch.bfloat16)
    else:  # the products' output rounding: one exact term per output (the others 0 * w * s), all zones active
        x = torch.zeros((1, K), dtype=torch.bfloat16)
        x[0, 14] = 1.0  # w = 77
        got = run_product(x.cuda(), P, s.cuda(), None, 8, 32, N // 4, [-1.0] * 4, "union").cpu()
        ref = (torch.tensor(77.0) * s.float()).to(torch.bfloat16)
        inside = s.float().abs() < 2.0 ** 120  # no 0 * inf from the other rows' terms
        got, ref = got[inside], ref[inside]
    assert torch.equal(got.isnan(), ref.isnan())
    ok = ~ref.isnan()
    assert torch.equal(got[ok], ref[ok])  # by value: a sum of signed zeros is +0
