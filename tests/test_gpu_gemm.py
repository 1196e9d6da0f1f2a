"""The matrix-core tiles (kq_gemm.hip): dense groups and the dense GLU past 64
rows, in every tile height and in K slices, and the MoE gathers of long
segments, against fp64 over the same wire bytes (max |err| / max |ref| within
the suite's tolerances; fp32 outputs to 1e-5 for Q4_K and IQ2_XXS, whose
integer codes fp16 holds exactly: what is left is fp32 accumulation over K)."""
import numpy as np
import pytest

from helpers import BF16_TOL, TOL, fp16_rows, quantized_weights
from oracle import kquant as okq

pytestmark = pytest.mark.gpu

CODECS = ("q4_k", "q6_k", "iq2_xxs")


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _wire(rng, codec, n, k):
    if codec == "iq2_xxs":
        return okq.random_valid_blocks(rng, codec, n * k // 256).reshape(n, -1)
    return quantized_weights(rng, codec, n, k)


def _tol(codec):
    return TOL if codec == "q6_k" else 1e-5


@pytest.fixture(autouse=True)
def _plain(monkeypatch):
    for k in ("GMLX_KQ_GEMM", "GMLX_KQ_GEMM_MT", "GMLX_KQ_GEMM_S"):
        monkeypatch.delenv(k, raising=False)


# rows and columns on both sides of every tile edge, one super-block up to an
# odd count; each tile height
@pytest.mark.parametrize("mt", ["1", "2", "4"])
@pytest.mark.parametrize("codec", CODECS)
@pytest.mark.parametrize("M,N,K", [(65, 1, 256), (128, 128, 512), (129, 257, 768), (200, 515, 2816)])
def test_tiles_match_fp64(codec, M, N, K, mt, monkeypatch):
    import torch
    from gmlx_amd import ops
    monkeypatch.setenv("GMLX_KQ_GEMM_MT", mt)
    rng = np.random.default_rng(M + N + K)
    wire, x = _wire(rng, codec, N, K), fp16_rows(rng, M, K)
    got = ops.quantized_matmul(_dev(x), _dev(wire), None, codec, out_dtype=torch.float32).cpu().numpy()
    ref = okq.qmm_ref(x, wire, codec)
    assert okq.max_rel(got, ref) <= _tol(codec), okq.max_rel(got, ref)


@pytest.mark.parametrize("dtype_name", ["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("mt,s", [("2", "3"), ("1", "2"), ("4", "5")])
def test_k_slices(mt, s, dtype_name, monkeypatch):
    """A group of two codecs and widths in uneven K slices: fp64, repeats
    bitwise, counters left zero; rows strided and one-signed."""
    import torch
    from gmlx_amd import _lib, ops
    monkeypatch.setenv("GMLX_KQ_GEMM_MT", mt)
    monkeypatch.setenv("GMLX_KQ_GEMM_S", s)
    rng = np.random.default_rng(int(s))
    M, K = 97, 256 * 23
    x = (fp16_rows(rng, M, K) + np.float16(2.0)).astype(np.float16)
    xd = torch.zeros(M, K + 8).to(getattr(torch, dtype_name)).cuda()
    xd[:, :K] = _dev(x).to(xd.dtype)
    xd = xd[:, :K]
    mats = [(_wire(rng, c, n, K), c) for c, n in (("q4_k", 300), ("q6_k", 33))]
    items = [(xd, _dev(w), c) for w, c in mats]
    outs = [ops.quantized_matmul_grouped(items, out_dtype=torch.float32) for _ in range(3)]
    torch.cuda.synchronize()
    for (w, c), y in zip(mats, outs[0]):
        ref = okq.qmm_ref(xd.float().cpu().numpy(), w, c)
        assert okq.max_rel(y.cpu().numpy(), ref) <= TOL, c
    for o in outs[1:]:
        assert all(torch.equal(a, b) for a, b in zip(o, outs[0]))
    ws = ops._WS._ws[("matmul", xd.device.index, ops._stream(xd).value)]
    assert not ws[:_lib.MATMUL_COUNTER_BYTES].any()


def test_slices_replay_in_a_graph():
    """The plan's own K slices (a down projection of a ragged prompt) captured
    and replayed between eager calls of another shape, each replay bitwise the
    eager result."""
    import torch
    from gmlx_amd import _lib, ops
    rng = np.random.default_rng(3)
    M, N, K = 100, 1024, 12288
    w, x = _dev(_wire(rng, "q6_k", N, K)), _dev(fp16_rows(rng, M, K))
    P = _lib.MatmulProblem
    arr = (P * 1)(P(w.data_ptr(), w.stride(0), x.data_ptr(), K, 1 << 22, N, M, N, K, _lib.CODEC_ID["q6_k"]))
    assert _lib.lib().kq_matmul_workspace_bytes(arr, 1, _lib.DTYPE_F16) > 0  # slices
    want = ops.quantized_matmul(x, w, None, "q6_k")
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        ops.quantized_matmul(x, w, None, "q6_k")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        y = ops.quantized_matmul(x, w, None, "q6_k")
    for m in (70, 300, 65):
        y.zero_()
        g.replay()
        other = ops.quantized_matmul(x[:m].contiguous() if m <= M else x.repeat(3, 1), w, None, "q6_k")
        torch.cuda.synchronize()
        assert torch.equal(y, want)
        assert okq.max_rel(other[:65].float().cpu().numpy(), want[:65].float().cpu().numpy()) <= TOL


@pytest.mark.parametrize("dtype_name", ["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("M,I,codec,act,mt", [(65, 128, "q4_k", "silu", "1"), (130, 200, "q6_k", "gelu", "2"),
                                              (300, 517, "iq2_xxs", "silu", "4")])
def test_dense_glu(M, I, codec, act, mt, dtype_name, monkeypatch):
    import torch
    from gmlx_amd import ops
    monkeypatch.setenv("GMLX_KQ_GEMM_MT", mt)
    rng = np.random.default_rng(M)
    K = 1024
    gw, uw = _wire(rng, codec, I, K), _wire(rng, codec, I, K)
    x = _dev(fp16_rows(rng, M, K)).to(getattr(torch, dtype_name))
    h = ops._glu_matmul(x, _dev(gw), _dev(uw), codec, act, ops._stream(x))
    xf = x.float().cpu().numpy()
    g, u = okq.qmm_ref(xf, gw, codec), okq.qmm_ref(xf, uw, codec)
    a = 0.5 * g * (1 + np.tanh(0.5 * g)) if act == "silu" else \
        0.5 * g * (1 + np.tanh(0.7978845608028654 * (g + 0.044715 * g ** 3)))
    assert h.dtype == x.dtype
    assert okq.max_rel(h.float().cpu().numpy(), a * u) <= (BF16_TOL if dtype_name == "bfloat16" else TOL)
    assert ops._glu_matmul(x[:64], _dev(gw), _dev(uw), codec, act, ops._stream(x)) is None


@pytest.mark.parametrize("dtype_name", ["float16", "bfloat16", "float32"])
@pytest.mark.parametrize("mt", ["1", "2"])
@pytest.mark.parametrize("codec", CODECS)
def test_long_segments(codec, mt, dtype_name, monkeypatch):
    """Gathers whose segments are longer than a tile, one row, empty and out of
    range: plain with a bias, clamped GLU with biases, the shared-expert
    layout's spare rows and the down gather over them, against the small-batch
    gathers (GMLX_KQ_GEMM=0) and fp64.  bf16 and fp32 rows are 2^-20 to 2^20 in
    size, and every pair row is held to its own largest value."""
    import torch
    from gmlx_amd import ops
    rng = np.random.default_rng(11)
    E, T, k, D, I = 5, 150, 2, 768, 200
    idx = np.full((T, k), 1)
    idx[:, 1] = rng.integers(2, 4, T)
    idx[7] = [0, 5]      # one row for expert 0, an id out of range; expert 4 empty
    idx[149, 1] = -1
    w = np.stack([_wire(rng, codec, I, D) for _ in range(E)])
    wu = np.stack([_wire(rng, codec, I, D) for _ in range(E)])
    wd = np.stack([_wire(rng, codec, 130, 256) for _ in range(E)])
    x, hid = fp16_rows(rng, T, D).astype(np.float32), fp16_rows(rng, T * (k + 1), 256).astype(np.float32)
    xc = x
    if dtype_name != "float16":
        size = np.exp2(rng.integers(-20, 21, (T, 1))).astype(np.float32)
        # (the clamps bound h: against large gates its fp32 error has no bound relative to the row)
        x, xc = x * size, x * np.minimum(size, 1)
        hid *= np.exp2(rng.integers(-20, 21, (T * (k + 1), 1))).astype(np.float32)
    dt = getattr(torch, dtype_name)
    b0, b1 = (rng.normal(0, 1, (E, I)).astype(np.float32) for _ in range(2))
    idxd, wgd, wud, wdd, b0d, b1d = (_dev(a) for a in (idx.astype(np.int32), w, wu, wd, b0, b1))
    xd, xcd, hd = _dev(x).to(dt), _dev(xc).to(dt), _dev(hid).to(dt).reshape(T, k + 1, 256)
    sg, su, sd = wgd[0].contiguous(), wud[0].contiguous(), wdd[0].contiguous()
    ones = torch.zeros(T, k + 1, device="cuda")

    def run(mode):
        monkeypatch.setenv("GMLX_KQ_GEMM", mode)
        monkeypatch.setenv("GMLX_KQ_GEMM_MT", mt)
        y = ops.gather_qmm(xd, wgd, None, codec, indices=idxd, out_dtype=torch.float32, bias=b0d).reshape(T, k, I)
        h = ops.moe_glu_gather_kq(xcd, wgd, wud, codec, idxd, act="swiglu_clamp", gate_bias=b0d, up_bias=b1d)
        hs = ops.moe_glu_gather_shexp_kq(xd, wgd, wud, sg, su, codec, idxd)
        dn = []
        for s in range(k + 1):  # the mix with one weight of 1: slot s alone
            one = ones.clone()
            one[:, s] = 1
            dn.append(ops.gather_qmv_mix_kq(hd, wdd, sd, codec, idxd, one))
        return [t.cpu().numpy() for t in (y, h, hs, torch.stack(dn, 1))]

    def rows_rel(a, b):
        a, b = (t.reshape(-1, t.shape[-1]).astype(np.float64) for t in (a, b))
        big = np.abs(b).max(1)
        assert not a[big == 0].any()
        return (np.abs(a - b).max(1)[big > 0] / big[big > 0]).max()

    old, new = run("0"), run("2")
    for a, b in zip(new, old):
        assert rows_rel(a, b) <= 2e-6 * 16  # fp32 sums in another order
    xf, hf = xd.double().cpu().numpy(), hd.double().cpu().numpy()
    W, Wd = (okq.dequantize(t, codec).astype(np.float64) for t in (w, wd))
    ref, refd = np.zeros((T, k, I)), np.zeros((T, k + 1, 130))
    for t in range(T):
        for s in range(k):
            e = idx[t, s]
            if 0 <= e < E:
                ref[t, s] = W[e] @ xf[t] + b0[e]
                refd[t, s] = Wd[e] @ hf[t, s]
        refd[t, k] = Wd[0] @ hf[t, k]
    # (fp32 rows enter rounded to 11 bits)
    tol = TOL if dtype_name == "float32" else _tol(codec)
    assert rows_rel(new[0], ref) <= tol
    assert rows_rel(new[3], refd) <= tol


@pytest.mark.parametrize("codec", CODECS)
def test_more_segments_than_a_wave(codec, monkeypatch):
    """130 experts, a third of them empty, segments of one row to four tiles: the
    chunk table runs over three rounds of 64 segments.  Plain, GLU and per-pair
    gathers of bf16 rows against fp64."""
    import torch
    from gmlx_amd import ops
    monkeypatch.setenv("GMLX_KQ_GEMM", "2")
    monkeypatch.setenv("GMLX_KQ_GEMM_MT", "1")
    rng = np.random.default_rng(130)
    E, N, K = 130, 72, 256
    counts = rng.integers(1, 6, E)
    counts[rng.random(E) < 1 / 3] = 0
    counts[[3, 63, 64, 65, 128, 129]] = [100, 33, 0, 32, 70, 1]
    ids = rng.permutation(np.repeat(np.arange(E), counts))
    k = 2
    idx = ids[:len(ids) // k * k].reshape(-1, k)
    T = len(idx)
    w, wu = (np.stack([_wire(rng, codec, N, K) for _ in range(E)]) for _ in range(2))
    W, U = (okq.dequantize(t, codec).astype(np.float64) for t in (w, wu))
    xd = _dev(fp16_rows(rng, T, K)).bfloat16()
    hd = _dev(fp16_rows(rng, T * k, K)).bfloat16().reshape(T, k, K)
    idxd, wd, wud = _dev(idx.astype(np.int32)), _dev(w), _dev(wu)
    y = ops.gather_qmm(xd, wd, None, codec, indices=idxd, out_dtype=torch.float32).reshape(T, k, N).cpu().numpy()
    h = ops.moe_glu_gather_kq(xd, wd, wud, codec, idxd).cpu().numpy()
    p = ops.gather_qmv_kq(hd, wd, codec, idxd).cpu().numpy()
    xf, hf = xd.double().cpu().numpy(), hd.double().cpu().numpy()
    g, u = (np.einsum("tknj,tj->tkn", M[idx], xf) for M in (W, U))
    assert okq.max_rel(y, g) <= _tol(codec)
    assert okq.max_rel(h, 0.5 * g * (1 + np.tanh(0.5 * g)) * u) <= TOL
    assert okq.max_rel(p, np.einsum("tknj,tkj->tkn", W[idx], hf)) <= _tol(codec)


@pytest.mark.parametrize("codec", CODECS)
def test_dense_kernel_past_64_rows(codec, monkeypatch):
    """The dense kernel over more than one chunk of 64 rows (GMLX_KQ_GEMM=0), and
    where a group of a longer and a shorter problem takes it by itself."""
    import torch
    from gmlx_amd import ops
    rng = np.random.default_rng(64)
    K = 1024
    x, (w, v) = fp16_rows(rng, 150, K), (_wire(rng, codec, n, K) for n in (40, 77))
    xd = _dev(x)
    a, b = ops.quantized_matmul_grouped([(xd, _dev(w), codec), (xd[:20], _dev(v), codec)], out_dtype=torch.float32)
    monkeypatch.setenv("GMLX_KQ_GEMM", "0")
    c = ops.quantized_matmul(xd, _dev(w), None, codec, out_dtype=torch.float32)
    assert torch.equal(a, c)
    assert okq.max_rel(c.cpu().numpy(), okq.qmm_ref(x, w, codec)) <= TOL
    assert okq.max_rel(b.cpu().numpy(), okq.qmm_ref(x[:20], v, codec)) <= TOL


@pytest.mark.parametrize("T,tiles", [(9, False), (33, False), (512, True)])
def test_one_expert_takes_the_tiles_only_when_they_fill_the_gpu(T, tiles, monkeypatch):
    """A shared expert's GLU and down gathers (one expert of 768 x 2048: 12 to
    96 tiles on 256 CUs): the default call's bits are those of the small-batch
    gathers at 9 and 33 tokens, of the tiles at 512, where they are faster."""
    import torch
    from gmlx_amd import ops
    rng = np.random.default_rng(T)
    D, I = 2048, 768
    gw, uw, dw = (_dev(okq.random_valid_blocks(rng, "q4_k", n * k // 256).reshape(1, n, -1))
                  for n, k in ((I, D), (I, D), (D, I)))
    x = _dev(fp16_rows(rng, T, D))
    h = _dev(fp16_rows(rng, T, I)).reshape(T, 1, I)
    idx = torch.zeros(T, 1, dtype=torch.int32, device="cuda")

    def run():
        return (ops.moe_glu_gather_kq(x, gw, uw, "q4_k", idx), ops.gather_qmv_kq(h, dw, "q4_k", idx))

    got = run()
    outs = {}
    for mode in ("0", "2"):
        monkeypatch.setenv("GMLX_KQ_GEMM", mode)
        outs[mode] = run()
    for a, old, new in zip(got, outs["0"], outs["2"]):
        assert not torch.equal(old, new)
        assert torch.equal(a, new if tiles else old)


@pytest.mark.parametrize("M,mats,tiles", [
    (100, [("q6_k", 1000)], False), (65, [("q4_k", 2048), ("q4_k", 1024), ("q6_k", 1024)], False),
    (100, [("iq2_xxs", 300)], False), (300, [("q6_k", 3072)], True), (100, [("q4_k", 1000)], True)])
def test_short_rows_take_the_tiles_only_past_one_round(M, mats, tiles, monkeypatch):
    """Groups of rows shorter than 8 super-blocks with Q6_K or IQ2_XXS among
    them: the default call's bits are the dense kernel's while its workgroups
    fit one a CU, else the tiles'."""
    import torch
    from gmlx_amd import ops
    rng = np.random.default_rng(M)
    K = 1536 if mats[0][0] == "iq2_xxs" else 1024
    x = _dev(fp16_rows(rng, M, K))
    items = [(x, _dev(okq.random_valid_blocks(rng, c, n * K // 256).reshape(n, -1)), c) for c, n in mats]
    got = ops.quantized_matmul_grouped(items, out_dtype=torch.float32)
    outs = {}
    for mode in ("0", "2"):
        monkeypatch.setenv("GMLX_KQ_GEMM", mode)
        outs[mode] = ops.quantized_matmul_grouped(items, out_dtype=torch.float32)
    for a, dense, tile in zip(got, outs["0"], outs["2"]):
        assert not torch.equal(dense, tile)
        assert torch.equal(a, tile if tiles else dense)
