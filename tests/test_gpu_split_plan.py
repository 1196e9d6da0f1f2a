"""The attention split plan at the lines between its lengths (64, 256, 512 and
1024 tokens) and at a caller's workspace too small for the short splits, against
fp64 attention."""
import numpy as np
import pytest

from helpers import BF16_TOL, TOL, attention_ref, q8_affine
from oracle import kquant as okq

pytestmark = pytest.mark.gpu


def _rows(rng, torch, B, Hq, Hkv, L, D, dt):
    mk = lambda *s: torch.from_numpy(rng.normal(0, 1, size=s).astype(np.float32)).to(dt)  # noqa: E731
    return mk(B, Hq, 1, D), mk(B, Hkv, L, D), mk(B, Hkv, L, D)


# head-tokens B * Hkv * L on both sides of seven 64-token waves a CU (114688 on
# 256 CUs), of 2048 waves of 1024 tokens, a wide group whose 64-token partials
# would pass 16 MB, and rows of a few tokens
@pytest.mark.parametrize("B,Hq,Hkv,L,D,dtype_name", [
    (1, 16, 8, 14336, 64, "float16"), (1, 16, 8, 14337, 64, "float16"), (2, 16, 1, 9001, 512, "float16"),
    (32, 8, 8, 7200, 64, "bfloat16"), (3, 8, 2, 65, 128, "bfloat16"), (2, 4, 4, 3, 128, "float16")])
def test_lengths_on_both_sides_of_the_lines(B, Hq, Hkv, L, D, dtype_name):
    import torch
    from gmlx_amd import ops
    rng = np.random.default_rng(B + L + D)
    q, k, v = _rows(rng, torch, B, Hq, Hkv, L, D, getattr(torch, dtype_name))
    starts = [int(s) for s in rng.integers(0, L, size=B)]
    starts[0] = 0
    out = ops.sdpa_decode_gqa(q.cuda(), k.cuda(), v.cuda(), D ** -0.5, starts=starts).float().cpu().numpy()[:, :, 0]
    for b in range(0, B, 7):
        ref = attention_ref(q[b, :, 0].double().numpy(), k[b, :, starts[b]:].double().numpy(),
                            v[b, :, starts[b]:].double().numpy(), D ** -0.5)
        assert okq.max_rel(out[b], ref) <= (TOL if dtype_name == "float16" else BF16_TOL), b


@pytest.mark.parametrize("dtype_name", ["float16", "bfloat16"])
@pytest.mark.parametrize("B,Hkv,L", [(2, 8, 700), (4, 8, 5000), (17, 8, 4100)])
def test_8bit_lengths(B, Hkv, L, dtype_name):
    import torch
    from gmlx_amd import ops
    rng = np.random.default_rng(L)
    D, Hq = 64, 2 * Hkv
    q, k, v = _rows(rng, torch, B, Hq, Hkv, L, D, getattr(torch, dtype_name))
    kw, ks, kb, kd = q8_affine(k.float().numpy(), dtype_name)
    vw, vs, vb, vd = q8_affine(v.float().numpy(), dtype_name)
    starts = [int(s) for s in rng.integers(0, L, size=B)]
    out = ops.sdpa_decode_gqa(q.cuda(), kw.cuda(), vw.cuda(), D ** -0.5, starts=starts, k_scales=ks.cuda(),
                              k_biases=kb.cuda(), v_scales=vs.cuda(), v_biases=vb.cuda()).float().cpu().numpy()
    for b in range(0, B, 5):
        ref = attention_ref(q[b, :, 0].double().numpy(), kd[b, :, starts[b]:], vd[b, :, starts[b]:], D ** -0.5)
        assert okq.max_rel(out[b, :, 0], ref) <= (TOL if dtype_name == "float16" else BF16_TOL), b


def test_a_workspace_of_the_long_splits_is_enough():
    """A caller's buffer that holds only 512-token splits' partials is served
    with those; one below that is refused."""
    import torch
    from gmlx_amd import _lib
    B, Hq, Hkv, L, D = 3, 8, 2, 3000, 128
    rng = np.random.default_rng(7)
    q, k, v = (t.cuda() for t in _rows(rng, torch, B, Hq, Hkv, L, D, torch.float16))
    lib = _lib.lib()
    long_need = B * Hq * 6 * (D + 2) * 4
    assert long_need < lib.kq_sdpa_workspace_bytes(B, Hq, Hkv, D, L)

    def call(nbytes):
        out = torch.full_like(q, float("nan"))
        ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
        rc = lib.kq_sdpa_decode_gqa(q.data_ptr(), k.data_ptr(), v.data_ptr(), k.stride(0), k.stride(1), L, None, B,
                                    Hq, Hkv, D, D ** -0.5, _lib.DTYPE_F16, out.data_ptr(), ws.data_ptr(), nbytes,
                                    torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        return rc, out.float().cpu().numpy()[:, :, 0]

    rc, out = call(long_need)
    assert rc == _lib.KQ_OK
    for b in range(B):
        ref = attention_ref(*(t[b].double().cpu().numpy() for t in (q[:, :, 0], k, v)), D ** -0.5)
        assert okq.max_rel(out[b], ref) <= TOL
    assert call(long_need - 4)[0] == _lib.KQ_ERR_WORKSPACE_TOO_SMALL
