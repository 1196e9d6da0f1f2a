"""bf16 / fp32 activation rows as scaled fp16 (kq_prepare.hip), at the edges of
its two forms: one wave a row up to 2048 values, a workgroup a row beyond, with
values past a lane's registers read twice past 16384.  The scaling is by a
power of two, so a call on prepared rows equals, bit for bit, the fp16 call on
rows scaled by hand, scaled back."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype_name", ["bfloat16", "float32"])
@pytest.mark.parametrize("M,K", [(1, 256), (9, 2048), (7, 2304), (3, 16384), (2, 16640)])
def test_prepared_rows_equal_rows_scaled_by_hand(M, K, dtype_name):
    import torch
    from gmlx_amd import ops
    gen = torch.Generator().manual_seed(M * K)
    x = torch.randn(M, K, generator=gen) * torch.exp2(torch.arange(M)[:, None].float() * 9 - 30)
    x[:, K - 1] = 3 * x.abs().amax(1)  # the largest in the last chunk
    if M > 2:
        x[2] = 0
    x = x.to(getattr(torch, dtype_name))
    big = x.double().abs().amax(1).numpy()
    e = torch.from_numpy(np.where(big > 0, np.frexp(big)[1] - 15, 0)).double()[:, None]
    by_hand = (x.double() * torch.exp2(-e)).to(torch.float16)
    w, _ = ops.quantize(torch.randn(48, K, generator=gen).cuda() * 0.02, "q4_k")
    got = ops.quantized_matmul(x.cuda(), w, None, "q4_k", out_dtype=torch.float32)
    want = ops.quantized_matmul(by_hand.cuda(), w, None, "q4_k", out_dtype=torch.float32)
    assert torch.equal(got.cpu().double(), want.cpu().double() * torch.exp2(e))
