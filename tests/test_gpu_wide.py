"""The wide-batch GEMM (zt_gemm_wide_f32 and the engine's batches past 16
tokens) against the oracle's dequantizers and a float64 product.

Bar per output: |y - ref| <= (K / 32 + 24) 2^-24 sum |w x| + 2^-38 max|x| sum|w|.
The sums are K / 32 block sums added in fp32, each an fp32 sum inside the
MFMAs (16 roundings), and the operand splits add up to 2^-22 sum |w x| (fp16
hi + lo of the activations and of IQ4_NL's codebook) and the split's absolute
floor of 2^-39 of the token's largest value.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from ztensor_amd import _lib, storage as st, synth  # noqa: E402
from ztensor_amd.engine import ROCmEngine  # noqa: E402

pytestmark = pytest.mark.gpu

G = st.GGMLType
FORMATS = ["gptq", "awq", "q4_0", "q8_0", "q5_0", "q4_k", "q5_k", "q6_k", "iq4_nl", "iq4_nl_f16",
           "mmap_q4_0", "mmap_q8_0", "mmap_q5_0", "mmap_q4_k", "mmap_q5_k", "mmap_q6_k"]


@pytest.fixture(scope="module")
def eng():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return ROCmEngine()


def weights(fmt, rows, K, seed, orc, group=128):
    """(storage, the oracle's dequantized matrix in float64)"""
    n = rows * K
    if fmt in ("gptq", "awq"):
        w = synth.w4a16(rows, K, seed, group)
        z = np.random.default_rng(seed).integers(3, 13, w.zeros.shape).astype(np.float16).view(np.uint16)
        if fmt == "gptq":
            s = st.GPTQStorage.from_raw(w.packed, w.scales, z, n, group, 4)
        else:
            s = st.AWQStorage(np.ascontiguousarray(w.packed).reshape(-1).view("<u4"), w.scales, z, n, group)
        d = orc.gptq_dequant(np.ascontiguousarray(w.packed).reshape(-1), w.scales, z, n, group)
    elif fmt in ("q4_0", "mmap_q4_0"):
        raw = synth.q4_0(rows, K, seed).raw
        s, d = st.Q4Storage.from_raw(raw, n), orc.q4_dequant(raw, n)
        s = s if fmt == "q4_0" else st.MmapStorage(raw, n, G.Q4_0)
    elif fmt == "q8_0":
        raw = synth.q8_0(rows, K, seed).raw
        s, d = st.Q8Storage(raw, n), orc.q8_dequant(raw, n)
    elif fmt == "mmap_q8_0":
        raw = synth.gguf_q8_0(rows, K, seed)
        s, d = st.MmapStorage(raw, n, G.Q8_0), orc.gguf_q8_0_dequant(raw, n)
    elif fmt.startswith("iq4"):
        raw = synth.iq4nl(rows, K, seed).raw
        s, d = st.IQ4NLStorage.from_raw(raw, n), orc.iq4nl_dequant(raw, n)
    else:
        name = fmt.replace("mmap_", "")
        raw = synth.kquant(name, rows, K, seed).raw
        d = orc.q5_0_dequant(raw, n) if name == "q5_0" else orc.kq_dequant(name, raw, n)
        kind = {"q5_0": st.Q5_0Storage, "q4_k": st.Q4KStorage, "q5_k": st.Q5KStorage, "q6_k": st.Q6KStorage}[name]
        g = {"q5_0": G.Q5_0, "q4_k": G.Q4_K, "q5_k": G.Q5_K, "q6_k": G.Q6_K}[name]
        s = st.MmapStorage(raw, n, g) if fmt.startswith("mmap") else kind.from_raw(raw, n)
    return s, np.asarray(d, np.float64).reshape(rows, K)


def half(fmt):
    return fmt in ("gptq", "awq", "iq4_nl_f16")


def activations(fmt, T, K, seed):
    x = np.random.default_rng(seed).standard_normal((T, K)).astype(np.float32)
    return x.astype(np.float16) if half(fmt) else x


def check(y, x, w):
    """y [T, rows] against x [T, K] w [rows, K]^T, by the module's bound."""
    y, x = np.asarray(y, np.float64), np.asarray(x, np.float64)
    K = x.shape[1]
    bound = ((K / 32 + 24) * 2.0**-24 * (np.abs(x) @ np.abs(w).T) +
             2.0**-38 * np.abs(x).max(axis=1, keepdims=True) * np.abs(w).sum(axis=1))
    bad = np.abs(y - x @ w.T) > bound
    assert not bad.any(), (int(bad.sum()), float((np.abs(y - x @ w.T) / np.maximum(bound, 1e-300)).max()))


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("rows,K,T", [(1, 256, 17), (37, 768, 33), (200, 1280, 100), (129, 3328, 65)])
def test_wide_matmul_both_sides(eng, orc, fmt, rows, K, T):
    """Tile edges and ragged rows, tokens and K units, in every format and on both operand sides."""
    s, w = weights(fmt, rows, K, rows + T, orc)
    x = activations(fmt, T, K, T)
    xd = torch.from_numpy(x).cuda()
    y = eng.matmul(xd, st.Tensor((K, rows), s))
    assert y.shape == (T, rows) and y.is_contiguous()
    check(y.cpu().numpy(), x, w)
    z = eng.matmul(st.Tensor((rows, K), s), xd.t().contiguous())
    assert z.shape == (rows, T)
    if T > 32:  # on this side the wide path starts past two 16-column chunks
        assert torch.equal(z.t(), y)
    else:
        check(z.t().cpu().numpy(), x, w)
    # a transposed activation, three dimensions and an unaligned base give the same bits
    assert torch.equal(eng.matmul(xd.t().contiguous().t(), st.Tensor((K, rows), s)), y)
    assert torch.equal(eng.matmul(xd.reshape(1, T, K), st.Tensor((K, rows), s)), y.reshape(1, T, rows))
    off = torch.empty(T * K + 1, dtype=xd.dtype, device="cuda")[1:].view(T, K).copy_(xd)
    assert torch.equal(eng.matmul(off, st.Tensor((K, rows), s)), y)


@pytest.mark.parametrize("fmt", FORMATS)
def test_one_token_of_any_strides(eng, orc, fmt):
    """One token whose elements are not neighbours in memory gives the bits of its copy."""
    rows, K = 40, 512
    s, w = weights(fmt, rows, K, 17, orc)
    x = torch.from_numpy(activations(fmt, 8, 2 * K, 18)).cuda()
    t = st.Tensor((K, rows), s)
    cols = x[:, :K].t().contiguous()  # channel-major
    for v in (cols.t()[3:4], cols[:, 3], x[2:3, ::2], x[2, 1::2], x[2, :1].expand(K), x[2, :1].expand(1, K)):
        y = eng.matmul(v, t)
        assert y.shape == (*v.shape[:-1], rows)
        assert torch.equal(y, eng.matmul(v.contiguous(), t))
        check(y.reshape(1, rows).cpu().numpy(), v.reshape(1, K).cpu().numpy(), w)


@pytest.mark.parametrize("fmt", ["gptq", "q4_0", "q4_k", "q6_k"])
@pytest.mark.parametrize("rows,T", [(2304, 17), (4100, 20), (4100, 40), (4100, 100), (4100, 200), (4100, 300),
                                    (4100, 520), (9000, 500), (9000, 1030), (20000, 900)])
def test_wide_every_tile(eng, orc, fmt, rows, T):
    """Every tile of the dispatch, by rows and tokens; a few tokens are checked."""
    K = 512
    s, w = weights(fmt, rows, K, 7, orc)
    x = activations(fmt, T, K, 8)
    y = eng.matmul(torch.from_numpy(x).cuda(), st.Tensor((K, rows), s)).cpu().numpy()
    pick = np.unique(np.r_[0, 15, 16, T // 2, T - 17, T - 2, T - 1])
    check(y[pick], x[pick], w)


@pytest.mark.parametrize("fmt", ["gptq", "iq4_nl_f16", "q4_0", "q5_k", "q6_k"])
@pytest.mark.parametrize("rows,K,T", [(1, 256, 2), (33, 768, 5), (100, 1280, 16), (4096, 512, 3), (4100, 2304, 16),
                                      (8200, 1024, 13), (24600, 512, 7), (50, 8448, 8)])
def test_few_tokens(eng, orc, fmt, rows, K, T):
    """2 to 16 tokens: one to all of a tile's tokens, K of whole and partial 512-value quads, every workgroup shape."""
    s, w = weights(fmt, rows, K, rows + T, orc)
    x = activations(fmt, T, K, T)
    y = eng.matmul(torch.from_numpy(x).cuda(), st.Tensor((K, rows), s))
    check(y.cpu().numpy(), x, w)
    assert torch.equal(eng.matmul(torch.from_numpy(x).cuda(), st.Tensor((K, rows), s)), y)


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("rows,K", [(1, 256), (37, 768), (130, 1280), (2060, 3328), (16400, 5120)])
def test_tiled_tokens_are_the_columns(eng, orc, monkeypatch, fmt, rows, K):
    """The token-major calls on the tiled copies give the column-major calls' bits: every token count, one and
    several K ranges and chunks, ragged rows, an unaligned and a transposed X."""
    if rows > 3000 and fmt not in ("gptq", "q4_0", "q6_k", "iq4_nl_f16"):
        pytest.skip("one format of each kernel on the large matrix")
    import ztensor_amd.engine as E

    # the columns on the tiled copy too
    monkeypatch.setattr(E, "_block_rowblock", lambda *a: False)
    monkeypatch.setattr(E, "_w4a16_rowblock", lambda *a: False)
    if fmt in ("iq4_nl", "iq4_nl_f16"):
        fmt, K = "iq4_nl_f16", K + 8192  # past 8192 they always are
    s, _ = weights(fmt, rows, K, rows + K, orc)
    for T in range(2, 17) if rows < 3000 else (3, 8, 11, 16):
        x = torch.from_numpy(activations(fmt, T, K, T)).cuda()
        y = eng._tiled_tokens(s, rows, K, x)
        n = -(-T // 4) * 4
        xp = torch.zeros((K, n), dtype=x.dtype, device="cuda")
        xp[:, :T] = x.t()
        assert torch.equal(y, eng._weight_times(s, rows, K, xp)[:, :T].t()), T
        off = torch.empty(T * K + 1, dtype=x.dtype, device="cuda")[1:].view(T, K).copy_(x)
        assert torch.equal(eng._tiled_tokens(s, rows, K, off), y)
        assert torch.equal(eng._tiled_tokens(s, rows, K, x.t().contiguous().t()), y)


@pytest.mark.parametrize("fmt", ["q4_0", "q8_0", "q5_0", "q4_k", "q5_k", "q6_k", "mmap_q8_0", "mmap_q4_k"])
@pytest.mark.parametrize("rows,K", [(1, 256), (37, 768), (130, 1280), (2060, 3328)])
def test_tiled_tokens_to_32(eng, orc, fmt, rows, K):
    """Two column tiles: partial and whole second tiles, one and several K ranges, ragged rows."""
    s, w = weights(fmt, rows, K, rows + K, orc)
    for T in (17, 18, 31, 32):
        x = activations(fmt, T, K, T)
        x[T - 1] *= 30.0
        y = eng._tiled_tokens(s, rows, K, torch.from_numpy(x).cuda()).cpu().numpy()
        assert y.shape == (T, rows)
        check(y, x, w)
        check(eng._wide_times(s, rows, K, torch.from_numpy(x).cuda()).cpu().numpy(), x, w)  # the other way


@pytest.mark.parametrize("fmt", ["q4_0", "q8_0", "q5_0", "q4_k", "q5_k", "q6_k", "mmap_q8_0", "mmap_q4_k"])
@pytest.mark.parametrize("T", [3, 4, 8, 12, 16, 20, 32])
@pytest.mark.parametrize("columns", [False, True])
def test_tiled_tokens_keep_to_themselves(eng, orc, monkeypatch, fmt, T, columns):
    """Tokens 40 decades apart are each as exact as alone, and infinities and NaN stay in theirs, on the tiled copies:
    token-major, and as columns.  One and several K ranges, and a last one that is shorter."""
    import ztensor_amd.engine as E

    if columns and (T > 16 or T % 4):
        pytest.skip("columns come in 4, 8, 12 or 16")
    monkeypatch.setattr(E, "_block_rowblock", lambda *a: False)
    for rows, K in ((40, 256), (70, 1280)):
        s, w = weights(fmt, rows, K, rows + T, orc)
        x = activations(fmt, T, K, T)
        x *= (10.0 ** np.linspace(-20, 20, T)).astype(np.float32)[:, None]
        x[1, 5], x[T - 2, K - 3] = np.inf, np.nan
        xd = torch.from_numpy(x).cuda()
        y = eng._weight_times(s, rows, K, xd.t().contiguous()).t() if columns else eng._tiled_tokens(s, rows, K, xd)
        y = y.cpu().numpy()
        fine = [t for t in range(T) if t not in (1, T - 2)]
        check(y[fine], x[fine], w)
        # (T = 3: one token holds both)
        assert not np.isfinite(y[1]).any() and np.isnan(y[T - 2]).all()


def relative_error(eng, s, w, x):
    """2-norm of matmul's error against 64 bits, relative."""
    rows, K = w.shape
    xd = torch.from_numpy(x).cuda()
    ref = xd.double() @ torch.from_numpy(w).cuda().t()
    return float((eng.matmul(xd, st.Tensor((K, rows), s)).double() - ref).norm() / ref.norm())


# root mean square of a rounding to fp32, relative: 2^-23 / sqrt(12) over the mean mantissa
_ROUND = 2.4e-8


@pytest.mark.parametrize("fmt", ["q4_0", "q8_0", "q5_0", "q4_k", "q5_k", "q6_k"])
@pytest.mark.parametrize("T", [3, 8, 16, 20, 32])
def test_error_of_tiled_tokens(eng, orc, fmt, T):
    """A sum of n terms of one size met in n fp32 additions is off by sqrt(n / 2) roundings.  Products are exact, so
    what is left is one such sum over the K / 32 blocks (in K ranges, which only shortens it) and, inside a block and
    in the activations' hi + lo, less than 6e-8."""
    rows, K = 1024, 4096
    s, w = weights(fmt, rows, K, 51, orc)
    x = activations(fmt, T, K, 52)
    assert relative_error(eng, s, w, x) <= np.sqrt(K / 32 / 2) * _ROUND + 6e-8


@pytest.mark.parametrize("fmt", ["gptq", "awq"])
@pytest.mark.parametrize("T", [3, 8, 16, 20, 32])
def test_error_of_tiled_fp16_tokens(eng, orc, fmt, T):
    """As above with two terms a unit of 128, its weights about the middle zero and the rest of its zero."""
    rows, K = 1024, 4096
    s, w = weights(fmt, rows, K, 61, orc)
    x = torch.from_numpy(activations(fmt, T, K, 62)).cuda()
    ref = x.double() @ torch.from_numpy(w).cuda().t()
    err = float((eng._tiled_tokens(s, rows, K, x).double() - ref).norm() / ref.norm())
    assert err <= np.sqrt(K / 64 / 2) * _ROUND + 6e-8


@pytest.mark.parametrize("fmt", ["q4_k", "q5_k"])
def test_error_of_wide_kquants(eng, orc, fmt):
    """One sum over the units of 128; inside one, eight MFMAs one after another, the activations' hi + lo and the minima:
    less than 1e-7."""
    rows, K, T = 2304, 4096, 2048  # all of K in one wave
    s, w = weights(fmt, rows, K, 71, orc)
    assert relative_error(eng, s, w, activations(fmt, T, K, 72)) <= np.sqrt(K / 128 / 2) * _ROUND + 1e-7


@pytest.mark.parametrize("fmt,terms,inside", [("q4_0", 160, 6e-8), ("q8_0", 160, 6e-8), ("mmap_q8_0", 160, 6e-8), ("q5_0", 50, 6e-8),
                                              ("iq4_nl_f16", 50, 6e-8), ("q4_k", 22, 1e-7), ("q5_k", 22, 1e-7)])
def test_error_of_long_rows(eng, orc, fmt, terms, inside):
    """Long rows: no chain of sums past 160 blocks, or two of about the root of their number."""
    rows, K, T = 1100, 14336, 2048
    s, w = weights(fmt, rows, K, 81, orc)
    assert relative_error(eng, s, w, activations(fmt, T, K, 82)) <= np.sqrt(terms / 2) * _ROUND + inside


@pytest.mark.parametrize("K,T", [(4096, 3), (4096, 37), (14336, 9), (14336, 317)])
def test_error_of_fp32_tokens_on_iq4nl(eng, orc, K, T):
    """As the column kernel, in fp32 throughout: the codebook's 24 bits, two chains of at most 8 terms a wave, and the
    activations' hi + lo."""
    rows = 512
    s, w = weights("iq4_nl", rows, K, 91, orc)
    assert relative_error(eng, s, w, activations("iq4_nl", T, K, 92)) <= np.sqrt(16 / 2) * _ROUND + 6e-8


@pytest.mark.parametrize("fmt,rows,K,T", [("gptq", 100, 8192, 5), ("q4_0", 100, 512, 4), ("q8_0", 300, 1024, 3),
                                          ("mmap_q4_0", 64, 512, 8), ("mmap_q5_k", 64, 512, 6), ("q4_k", 64, 512, 20),
                                          ("iq4_nl_f16", 64, 5120, 8)])
def test_tiled_tokens_build_a_copy_only_at_no_risk(eng, orc, fmt, rows, K, T):
    """Where the columns need no tiled copy the tokens make one, but neither in a capture nor at the memory limit, nor
    where the engine was told not to; both ways give the result."""
    s, w = weights(fmt, rows, K, rows + T, orc)
    x = activations(fmt, T, K, T)
    xd = torch.from_numpy(x).cuda()
    careful = ROCmEngine(split_reserve_bytes=1 << 60)
    for e in (careful, ROCmEngine(token_copies=False)):
        check(e.matmul(xd, st.Tensor((K, rows), s)).cpu().numpy(), x, w)
        assert getattr(s, "_gpu_tiled", None) is None
    side = torch.cuda.Stream()
    cap = ROCmEngine(stream=side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side), torch.cuda.graph(g, stream=side):
        y = cap.matmul(xd, st.Tensor((K, rows), s))
    assert getattr(s, "_gpu_tiled", None) is None
    for _ in range(3):
        with torch.cuda.stream(side):
            g.replay()
        torch.cuda.synchronize()
        check(y.cpu().numpy(), x, w)
    z = eng.matmul(xd, st.Tensor((K, rows), s))
    assert s._gpu_tiled is not None
    check(z.cpu().numpy(), x, w)
    assert torch.equal(careful.matmul(xd, st.Tensor((K, rows), s)), z)  # the copy is there


@pytest.mark.parametrize("fmt,rows,K,T", [
    ("q6_k", 64, 512, 1), ("q6_k", 64, 512, 20), ("q6_k", 64, 512, 40), ("mmap_q6_k", 64, 512, 1),
    ("mmap_q6_k", 64, 512, 20), ("mmap_q6_k", 64, 512, 40), ("q6_k", 64, 512, 8), ("q4_k", 64, 512, 7),
    ("q5_k", 64, 512, 16), ("q5_0", 64, 512, 5), ("q4_0", 64, 512, 12), ("q8_0", 64, 512, 16),
    ("mmap_q8_0", 64, 512, 12), ("gptq", 4100, 512, 12), ("iq4_nl_f16", 64, 8448, 8)])
def test_a_copy_made_in_a_capture_is_the_graphs_own(eng, orc, fmt, rows, K, T):
    """A weight's first call in a capture: nothing is kept whose kernels have only been recorded, so eager calls
    before the first replay are right, and so is every replay after them."""
    s, w = weights(fmt, rows, K, rows + T, orc)
    x = activations(fmt, T, K, T)
    xd = torch.from_numpy(x).cuda()
    side = torch.cuda.Stream()
    cap = ROCmEngine(stream=side)
    cap.upload_weights([s])
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side), torch.cuda.graph(g, stream=side):
        y = cap.matmul(xd, st.Tensor((K, rows), s))
        # (columns of a mapped file end in a library's GEMM, whose first call is not one to capture)
        a = cap.matmul(st.Tensor((rows, K), s), xd.t()) if not fmt.startswith("mmap") else y.t()
    assert getattr(s, "_gpu_split", None) is None and getattr(s, "_gpu_tiled", None) is None
    with torch.cuda.stream(side):
        check(cap.matmul(xd, st.Tensor((K, rows), s)).cpu().numpy(), x, w)
    check(eng.matmul(xd, st.Tensor((K, rows), s)).cpu().numpy(), x, w)
    for _ in range(3):
        with torch.cuda.stream(side):
            g.replay()
        torch.cuda.synchronize()
        check(y.cpu().numpy(), x, w)
        check(a.t().cpu().numpy(), x, w)
        junk = torch.full((1 << 22,), 255, dtype=torch.uint8, device="cuda")
        del junk


@pytest.mark.parametrize("fmt,T", [("q4_0", 4), ("gptq", 4), ("q8_0", 20), ("mmap_q5_k", 6), ("mmap_q6_k", 40)])
def test_engines_on_two_streams_share_a_storage(orc, fmt, T):
    """A second engine finds the copy the first has just made behind other work on its stream."""
    rows, K = 640, 8192 if fmt == "gptq" else 1024
    s, w = weights(fmt, rows, K, rows + T, orc)
    x = activations(fmt, T, K, T)
    xd = torch.from_numpy(x).cuda()
    first, second = (ROCmEngine(stream=torch.cuda.Stream()) for _ in range(2))
    first.upload_weights([s])
    torch.cuda.synchronize()
    with torch.cuda.stream(first.stream):
        torch.cuda._sleep(20_000_000)
    y = first.matmul(xd, st.Tensor((K, rows), s))
    z = second.matmul(xd, st.Tensor((K, rows), s))
    torch.cuda.synchronize()
    assert getattr(s, "_gpu_tiled", None) is not None or getattr(s, "_gpu_split", None) is not None
    check(y.cpu().numpy(), x, w)
    assert torch.equal(y, z)


@pytest.mark.parametrize("fmt", ["gptq", "iq4_nl_f16"])
@pytest.mark.parametrize("rows,K", [(1, 256), (130, 1280), (2060, 3328), (16400, 5120)])
def test_tiled_fp16_tokens_to_32(eng, orc, fmt, rows, K):
    """Two column tiles of fp16 tokens give the bits of the calls on each 16 (padded), one and several K ranges and
    chunks."""
    s, _ = weights(fmt, rows, K, rows + K, orc)
    for T in (17, 30, 32):
        x = torch.from_numpy(activations(fmt, T, K, T)).cuda()
        y = eng._tiled_tokens(s, rows, K, x)
        assert y.shape == (T, rows)
        pad = torch.zeros((16, K), dtype=x.dtype, device="cuda")
        pad[: T - 16] = x[16:]
        assert torch.equal(y[:16], eng._tiled_tokens(s, rows, K, x[:16].contiguous()))
        assert torch.equal(y[16:], eng._tiled_tokens(s, rows, K, pad)[: T - 16])


def test_graph_keeps_its_workspace(orc):
    """A graph captured before the engine's workspace grew replays on the one it was captured with."""
    small, w = weights("q4_0", 512, 4096, 1, orc)
    large, _ = weights("q4_0", 4096, 4096, 2, orc)
    side = torch.cuda.Stream()
    e = ROCmEngine(stream=side)
    x = activations("q4_0", 8, 4096, 3)
    xd, xl = torch.from_numpy(x).cuda(), torch.randn(32, 4096, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        e.matmul(xd, st.Tensor((4096, 512), small))  # builds the tiled copy
        held = e._wsbuf.data_ptr()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=side):
            y = e.matmul(xd, st.Tensor((4096, 512), small))
        e.matmul(xl, st.Tensor((4096, 4096), large))
        assert e._wsbuf.data_ptr() != held and any(b.data_ptr() == held for b in e._wskept)
        junk = [torch.full((1 << 20,), 7, dtype=torch.uint8, device="cuda") for _ in range(8)]
        for _ in range(3):
            g.replay()
            torch.cuda.synchronize()
            check(y.cpu().numpy(), x, w)
            assert all(bool((j == 7).all()) for j in junk)


def test_tiled_tokens_entry_point_errors(eng):
    lib, p = eng.lib, 1 << 20
    for t in (0, 33):
        assert lib.zt_gemm_blkt_tokens_f32(1, p, p, 0, p, p, 16, 128, t, 0, 0, 0) == 1
        assert lib.zt_gemm_blkt_tokens_workspace_bytes(1, 16, 128, t) == -1
        assert lib.zt_gemm_w4a16t_tokens_f32(p, p, p, p, 16, 128, t, 128, 0, 0, 0) == 1
        assert lib.zt_gemm_iq4nlt_tokens_f16(p, p, p, p, 16, 128, t, 0, 0, 0) == 1
    assert lib.zt_gemm_blkt_tokens_f32(0, p, p, 0, p, p, 16, 128, 4, 0, 0, 0) == 1  # W4A16 and IQ4_NL have their own
    assert lib.zt_gemm_blkt_tokens_f32(4, p, p, 0, p, p, 16, 128, 4, 0, 0, 0) == 1  # no fifth bits
    assert lib.zt_gemm_blkt_tokens_f32(1, p, p, 0, p + 4, p, 16, 128, 4, 0, 0, 0) == 1  # X alignment
    assert lib.zt_gemm_blkt_tokens_f32(1, p, p, 0, p, p, 16, 1 << 24, 4, 0, 0, 0) == 1
    # 32 tokens: two column tiles of partials
    one, two = lib.zt_gemm_q8t_workspace_bytes(4096, 4096, 16), lib.zt_gemm_blkt_tokens_workspace_bytes(2, 4096, 4096, 17)
    assert two == 2 * one > 0 and lib.zt_gemm_blkt_tokens_workspace_bytes(2, 4096, 4096, 16) == one
    assert lib.zt_gemm_blkt_tokens_f32(2, p, p, 0, p, p, 4096, 4096, 17, p, two - 1, 0) == 1
    assert lib.zt_gemm_w4a16t_tokens_f32(p, p, p, p, 16, 1 << 25, 4, 128, 0, 0, 0) == 1


def test_few_tokens_special_values(eng, orc):
    """Infinities and NaN stay in their tokens."""
    s, w = weights("gptq", 40, 640, 3, orc)
    x = activations("gptq", 6, 640, 4)
    x[1, 7], x[3, 600] = np.inf, np.nan
    y = eng.matmul(torch.from_numpy(x).cuda(), st.Tensor((640, 40), s)).cpu().numpy()
    check(y[[0, 2, 4, 5]], x[[0, 2, 4, 5]], w)
    assert np.all(np.isnan(y[3])) and not np.any(np.isfinite(y[1]))


def test_wide_long_k(eng, orc):
    """The longest rows the packing holds, and a K past them (the other paths)."""
    for K in (16512, 32768, 33024):
        s, w = weights("q4_0", 24, K, 3, orc)
        x = activations("q4_0", 18, K, 4)
        y = eng.matmul(torch.from_numpy(x).cuda(), st.Tensor((K, 24), s)).cpu().numpy()
        if K <= 32768:
            check(y, x, w)
        else:
            assert np.max(np.abs(y - x.astype(np.float64) @ w.T)) <= 1e-5 * np.max(np.abs(x.astype(np.float64) @ w.T))


@pytest.mark.parametrize("K,group", [(768, 256), (640, 64)])
@pytest.mark.parametrize("T", [6, 35])
def test_wide_w4a16_groups(eng, orc, K, group, T):
    """A group of several 128-K units; a group the wide path does not take."""
    s, w = weights("gptq", 40, K, 5, orc, group)
    x = activations("gptq", T, K, 6)
    y = eng.matmul(torch.from_numpy(x).cuda(), st.Tensor((K, 40), s)).cpu().numpy()
    assert np.max(np.abs(y - x.astype(np.float64) @ w.T)) <= 1e-5 * np.max(np.abs(x.astype(np.float64) @ w.T))


@pytest.mark.parametrize("T", [11, 50])
def test_wide_w4a16_zeros_of_any_value(eng, orc, T):
    """Zeros that are no whole numbers, and large ones, in some groups."""
    rows, K = 70, 1024
    w = synth.w4a16(rows, K, 11)
    z = np.full(w.zeros.shape, 8.0, np.float16)
    z.reshape(-1)[::5] = 7.3
    z.reshape(-1)[3::11] = -0.125
    z.reshape(-1)[6::31] = 3000.5
    zb = z.view(np.uint16)
    s = st.GPTQStorage.from_raw(w.packed, w.scales, zb, rows * K, 128, 4)
    d = np.asarray(orc.gptq_dequant(np.ascontiguousarray(w.packed).reshape(-1), w.scales, zb, rows * K, 128), np.float64)
    x = activations("gptq", T, K, 12)
    y = eng.matmul(torch.from_numpy(x).cuda(), st.Tensor((K, rows), s)).cpu().numpy().astype(np.float64)
    x, d = x.astype(np.float64), d.reshape(rows, K)
    # the whole part and the rest of a zero are summed apart: (|q| + |zero|) |s x| instead of |w x|
    sc = w.scales.view(np.float16).astype(np.float64).repeat(128).reshape(rows, K)
    mag = np.abs(x) @ (np.abs(d) + 15 * sc + np.abs(z.astype(np.float64)).repeat(128).reshape(rows, K) * sc).T
    assert np.all(np.abs(y - x @ d.T) <= (K / 32 + 24) * 2.0**-24 * mag)


def test_wide_token_scales_and_special_values(eng, orc):
    """Tokens far apart in scale, all-zero tokens, and infinities and NaN, which stay in their tokens."""
    rows, K, T = 48, 512, 40
    s, w = weights("q8_0", rows, K, 21, orc)
    x = activations("q8_0", T, K, 22)
    x *= (10.0 ** np.linspace(-30, 30, T)).astype(np.float32)[:, None]
    x[7] = 0.0
    x[9, 5] = np.inf
    x[11, 3] = np.nan
    x[13] = np.float32(1e-42)  # subnormal
    y = eng.matmul(torch.from_numpy(x).cuda(), st.Tensor((K, rows), s)).cpu().numpy()
    fine = [t for t in range(T) if t not in (9, 11, 13)]
    check(y[fine], x[fine], w)
    assert np.all(y[7] == 0.0) and np.all(np.isnan(y[11]))
    with np.errstate(invalid="ignore"):
        ref = x[9].astype(np.float64) @ w.T
    assert np.array_equal(np.isnan(y[9]), np.isnan(ref)) and np.array_equal(y[9][np.isinf(ref)], ref[np.isinf(ref)])
    assert np.allclose(y[13], x[13].astype(np.float64) @ w.T, rtol=1e-5, atol=3e-45)


def test_wide_in_a_captured_graph(eng, orc):
    """A captured call replays as the eager one, also after wider eager calls of the same engine."""
    stream = torch.cuda.Stream()
    eng = ROCmEngine(stream=stream)
    s, _ = weights("q4_k", 300, 1024, 31, orc)
    big, _ = weights("q8_0", 500, 2048, 32, orc)
    t = st.Tensor((1024, 300), s)
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):  # all work in the engine's stream order
        x = torch.from_numpy(activations("q4_k", 24, 1024, 33)).cuda()
        eng.matmul(x, t)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=stream):
            y = eng.matmul(x, t)
        for i in range(3):
            x.copy_(torch.from_numpy(activations("q4_k", 24, 1024, 40 + i)))
            want = eng.matmul(x, t).clone()
            eng.matmul(torch.randn(700, 2048, device="cuda"), st.Tensor((2048, 500), big))
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, want)


def test_wide_arguments(eng):
    lib, need = eng.lib, eng.lib.zt_gemm_wide_workspace_bytes
    assert need(1, 0, 64, 256, 20) > 0
    for bad in [(-1, 0, 64, 256, 20), (9, 0, 64, 256, 20), (1, 1, 64, 256, 20), (0, 0, 64, 256, 20), (1, 0, 64, 160, 20),
                (5, 0, 64, 384, 20), (1, 0, 64, 32896, 20), (2, 0, 1 << 16, 32768, 20), (1, 0, 0, 256, 20)]:
        assert need(*bad) == -1, bad
    b = torch.zeros(1 << 20, dtype=torch.uint8, device="cuda")
    p, s = b.data_ptr(), torch.cuda.current_stream().cuda_stream
    ws = need(1, 0, 64, 256, 20)

    def call(w=p, o1=1024, x=p, c=p + (1 << 19), k=256, t=20, wsp=p + (1 << 18), wsb=ws, rows=64):
        return lib.zt_gemm_wide_f32(1, w, o1, 0, 0, 0, x, 0, c, rows, k, t, wsp, wsb, s)

    assert call() == 0 and call(rows=0) == 0 and call(t=0) == 0
    for bad in (dict(w=0), dict(x=0), dict(c=0), dict(wsp=0), dict(wsb=ws - 1), dict(w=p + 8), dict(x=p + 4),
                dict(o1=1032), dict(o1=-16), dict(c=p + 2), dict(wsp=p + 8), dict(k=-128), dict(t=-1), dict(k=96)):
        assert call(**bad) == _lib.HIP_ERROR_INVALID_VALUE, bad
    torch.cuda.synchronize()
