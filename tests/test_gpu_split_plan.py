"""The attention split plan at the lines between its lengths (one split, 64,
128, 256, 512 and 1024 tokens), for a row alone and in a batch, and at a
caller's workspace too small for the short splits, against fp64 attention."""
import numpy as np
import pytest

from helpers import BF16_TOL, TOL, attention_ref, q8_affine
from oracle import kquant as okq

pytestmark = pytest.mark.gpu


def _rows(rng, torch, B, Hq, Hkv, L, D, dt):
    mk = lambda *s: torch.from_numpy(rng.normal(0, 1, size=s).astype(np.float32)).to(dt)  # noqa: E731
    return mk(B, Hq, 1, D), mk(B, Hkv, L, D), mk(B, Hkv, L, D)


# rows of L and L - 1 keys on both sides of each line: 256 (512 past eight query heads
# a kv head), 512, 4096 (1024 past four) and 8192 up to head dim 128; 128, 1024, 8192 and 32768
# past it; and 2048 waves of 1024 tokens
@pytest.mark.parametrize("B,Hq,Hkv,L,D,dtype_name", [
    (3, 8, 2, 257, 64, "float16"), (3, 8, 2, 513, 128, "float16"), (3, 8, 2, 4097, 128, "bfloat16"),
    (2, 16, 2, 1025, 128, "float16"), (2, 16, 1, 513, 64, "bfloat16"), (2, 16, 1, 1025, 128, "float16"),
    (3, 4, 1, 8193, 96, "float16"), (3, 4, 2, 129, 256, "bfloat16"), (2, 2, 2, 1025, 256, "float16"),
    (2, 16, 1, 8193, 512, "float16"), (2, 2, 1, 32769, 256, "float16"), (32, 8, 8, 7200, 64, "bfloat16"),
    (3, 8, 2, 65, 128, "bfloat16"), (2, 4, 4, 3, 128, "float16")])
def test_lengths_on_both_sides_of_the_lines(B, Hq, Hkv, L, D, dtype_name):
    import torch
    from gmlx_amd import ops
    rng = np.random.default_rng(B + L + D)
    q, k, v = _rows(rng, torch, B, Hq, Hkv, L, D, getattr(torch, dtype_name))
    starts = [int(s) for s in rng.integers(0, L, size=B)]
    starts[:2] = [0, 1]
    out = ops.sdpa_decode_gqa(q.cuda(), k.cuda(), v.cuda(), D ** -0.5, starts=starts).float().cpu().numpy()[:, :, 0]
    for b in sorted({0, 1, B - 1}):
        ref = attention_ref(q[b, :, 0].double().numpy(), k[b, :, starts[b]:].double().numpy(),
                            v[b, :, starts[b]:].double().numpy(), D ** -0.5)
        assert okq.max_rel(out[b], ref) <= (TOL if dtype_name == "float16" else BF16_TOL), b


@pytest.mark.parametrize("dtype_name", ["float16", "bfloat16"])
@pytest.mark.parametrize("B,Hkv,L", [(2, 8, 700), (4, 8, 5000), (17, 8, 4100), (2, 2, 65), (2, 1, 257), (2, 2, 1025), (2, 2, 2049),
                                     (2, 1, 32769)])
def test_8bit_lengths(B, Hkv, L, dtype_name):
    import torch
    from gmlx_amd import ops
    rng = np.random.default_rng(L)
    D, Hq = 64, (16 if L == 257 else 2) * Hkv  # (one split up to 256 past eight query heads a kv head)
    q, k, v = _rows(rng, torch, B, Hq, Hkv, L, D, getattr(torch, dtype_name))
    kw, ks, kb, kd = q8_affine(k.float().numpy(), dtype_name)
    vw, vs, vb, vd = q8_affine(v.float().numpy(), dtype_name)
    starts = [int(s) for s in rng.integers(0, L, size=B)]
    starts[:2] = [0, 1]
    out = ops.sdpa_decode_gqa(q.cuda(), kw.cuda(), vw.cuda(), D ** -0.5, starts=starts, k_scales=ks.cuda(),
                              k_biases=kb.cuda(), v_scales=vs.cuda(), v_biases=vb.cuda()).float().cpu().numpy()
    for b in sorted({0, 1, B - 1}):
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


@pytest.mark.parametrize("Hq,Hkv,D,dtype_name,q8", [
    (32, 8, 128, "float16", False), (32, 8, 128, "bfloat16", True), (16, 2, 64, "bfloat16", False),
    (16, 8, 256, "float16", False), (16, 8, 256, "float16", True)])
def test_a_row_keeps_its_bits_in_any_batch(Hq, Hkv, D, dtype_name, q8):
    """Rows of very different lengths in one padded batch, each bitwise the call
    on the row alone, in the batch's cache and in one of its own length; the
    16-bit rows as slabs too.  A sequence's bits do not change as others join."""
    import torch
    from gmlx_amd import ops
    rng = np.random.default_rng(D + Hq)
    dt = getattr(torch, dtype_name)
    lens = [8000, 200, 900, 3000, 1]
    B, L = len(lens), max(lens)
    q, k, v = _rows(rng, torch, B, Hq, Hkv, L, D, dt)
    starts = [L - n for n in lens]
    if q8:
        (kw, ks, kb, kd), (vw, vs, vb, vd) = (q8_affine(t.float().numpy(), dtype_name) for t in (k, v))
        cache = [t.cuda() for t in (kw, vw, ks, kb, vs, vb)]
    else:
        kd, vd = k.double().numpy(), v.double().numpy()
        cache = [k.cuda(), v.cuda()]
    qd = q.cuda()

    def call(sl, cache, starts):
        kw = dict(zip(("k_scales", "k_biases", "v_scales", "v_biases"), cache[2:]))
        return ops.sdpa_decode_gqa(qd[sl], cache[0], cache[1], D ** -0.5, starts=starts, **kw)

    full = call(slice(None), cache, starts)
    for b, n in enumerate(lens):
        sl = slice(b, b + 1)
        assert torch.equal(call(sl, [t[sl] for t in cache], starts[sl])[0], full[b]), n
        own = [t[sl, :, L - n:].contiguous() for t in cache]
        assert torch.equal(call(sl, own, [0])[0], full[b]), n
        ref = attention_ref(q[b, :, 0].double().numpy(), kd[b, :, L - n:], vd[b, :, L - n:], D ** -0.5)
        assert okq.max_rel(full[b, :, 0].float().cpu().numpy(), ref) <= (TOL if dtype_name == "float16" else BF16_TOL)
    if not q8:
        kf, vf = (torch.cat([t[b, :, L - n:].reshape(-1) for b, n in enumerate(lens)]) for t in cache)
        offs = [0]
        for n in lens[:-1]:
            offs.append(offs[-1] + Hkv * n * D)
        assert torch.equal(ops.sdpa_decode_slabs(qd[:, :, 0].contiguous(), kf, vf, offs, lens, Hkv, D ** -0.5),
                           full[:, :, 0])


def test_noalloc_serves_what_the_long_splits_need():
    """A call whose short splits' partials pass the library's own scratch, and
    whose long ones' do not, is served as the workspace entry serves it with
    that many bytes."""
    import torch
    from gmlx_amd import _lib
    B, Hq, Hkv, L, D = 16, 128, 8, 8192, 128
    limit, lib = _lib.SDPA_NOALLOC_SCRATCH_BYTES, _lib.lib()
    assert lib.kq_sdpa_workspace_bytes(B, Hq, Hkv, D, L) > limit >= B * Hq * (L // 512) * (D + 2) * 4
    gen = torch.Generator(device="cuda").manual_seed(5)
    q, k, v = (torch.randn(B, h, n, D, device="cuda", generator=gen).half() for h, n in ((Hq, 1), (Hkv, L), (Hkv, L)))
    ws = torch.empty(limit, dtype=torch.uint8, device="cuda")
    outs = [torch.empty_like(q) for _ in range(2)]
    args = (k.stride(0), k.stride(1), L, None, B, Hq, Hkv, D, D ** -0.5, _lib.DTYPE_F16)
    ptrs = (q.data_ptr(), k.data_ptr(), v.data_ptr())
    s = torch.cuda.current_stream().cuda_stream
    assert lib.kq_sdpa_decode_gqa_noalloc(*ptrs, *args, outs[0].data_ptr(), s) == _lib.KQ_OK
    assert lib.kq_sdpa_decode_gqa(*ptrs, *args, outs[1].data_ptr(), ws.data_ptr(), limit, s) == _lib.KQ_OK
    assert torch.equal(outs[0], outs[1])
    ref = attention_ref(*(t[3].double().cpu().numpy() for t in (q[:, :, 0], k, v)), D ** -0.5)
    assert okq.max_rel(outs[0][3, :, 0].float().cpu().numpy(), ref) <= TOL
