"""What ROCmEngine.matmul hands to its kernels, without a GPU: the engine's
methods run on CPU tensors, with stand-ins for the calls that launch."""
import pytest

torch = pytest.importorskip("torch")

from ztensor_amd import storage as st  # noqa: E402
from ztensor_amd.engine import ROCmEngine  # noqa: E402

ROWS, K = 6, 256


def _engine():
    """An engine whose _weight_times reads its activations as a kernel does: K
    elements (times the columns) in a row from the tensor's address."""
    w = torch.randn(ROWS, K, generator=torch.Generator().manual_seed(1))
    eng = object.__new__(ROCmEngine)

    def weight_times(s, rows, k, x):
        n = x.numel() // k
        assert x.is_contiguous(), (tuple(x.shape), x.stride())
        return w @ torch.as_strided(x, (k, n), (n, 1))

    eng._weight_times = weight_times
    return eng, w


def _vectors():
    x = torch.arange(8.0 * K).reshape(8, K) % 17 - 8
    wide = torch.arange(2.0 * K).reshape(1, 2 * K) % 13 - 6
    return {
        "row": x[3:4], "vector": x[3], "three dimensions": x[3].reshape(1, 1, K),
        "row of channel-major tokens": x.t().contiguous().t()[3:4],
        "column": x.t().contiguous()[:, 3],
        "every other element": wide[:, ::2], "second of each pair": wide.reshape(K, 2)[:, 1],
        "one value for all": torch.tensor([1.5]).expand(K), "one value, a row": torch.tensor([[1.5]]).expand(1, K),
    }


@pytest.mark.parametrize("name", list(_vectors()))
def test_one_token_of_any_strides(name):
    x = _vectors()[name]
    eng, w = _engine()
    y = ROCmEngine.matmul.__wrapped__(eng, x, st.Tensor((K, ROWS), object()))
    assert y.shape == (*x.shape[:-1], ROWS)
    assert torch.allclose(y.reshape(-1), w @ x.reshape(-1), rtol=1e-5, atol=1e-3)


@pytest.mark.parametrize("name", ["vector", "column", "second of each pair", "one value for all"])
def test_grouped_vector_of_any_strides(name):
    x = _vectors()[name]
    eng, w = _engine()
    eng.device = x.device
    for y in ROCmEngine.gemv_group.__wrapped__(eng, [st.Tensor((ROWS, K), object())] * 2, x):
        assert torch.allclose(y, w @ x, rtol=1e-5, atol=1e-3)


class _Lib:
    """Entry points that only note their calls."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        if name.endswith("_bytes"):
            return lambda *a: 64
        raise AttributeError(name)

    def call(self, name, *args):
        self.calls.append(name)


@pytest.mark.parametrize("capturing", [False, True])
def test_copies_made_in_a_capture_are_not_kept(monkeypatch, capturing):
    """A captured copy has only been recorded: no later call may find it on the storage."""
    from types import SimpleNamespace

    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda d=None: (1 << 40, 1 << 40))
    eng = object.__new__(ROCmEngine)
    eng.lib, eng.device = _Lib(), torch.device("cpu")
    eng.stream = SimpleNamespace(cuda_stream=0, synchronize=lambda: eng.lib.calls.append("synchronize"))
    eng.q6k_split, eng.split_reserve_bytes = True, 0
    buf = SimpleNamespace(tensor=torch.zeros(64, dtype=torch.uint8), data_offset=0)

    def storage():
        return SimpleNamespace(gpu_ptr=lambda: buf, group_size=128, _gpu_scales=buf.tensor, _gpu_zeros=None)

    builders = [lambda s: eng._w4a16_tiled(s, 16, 256), lambda s: eng._iq4nl_tiled(s, buf, 16, 256),
                lambda s: eng._block_tiled(s, buf, 16, 256, "q4"), lambda s: eng._kq_tiled(s, buf, 16, 256, "q5k"),
                lambda s: eng._q5_0_tiled(s, buf, 16, 256, 0, 0)]
    for build in builders:
        s = storage()
        assert build(s) is not None
        assert (getattr(s, "_gpu_tiled", None) is None) == capturing
        # a kept copy is complete: an engine on another stream may find it next
        assert (eng.lib.calls[-1] == "synchronize") != capturing
    s = storage()
    assert (eng._q6k_split_copy(s, 0, 16, 256) is None) == capturing  # (the GEMV then reads the super-blocks)
    assert (getattr(s, "_gpu_split", None) is None) == capturing
    assert eng._q6k_split_copy(storage(), 0, 16, 256, for_one_call=True) is not None


@pytest.mark.parametrize("rows,k,wide", [(1024, 1024, True), (20480, 1024, True), (6144, 1536, True), (8448, 1536, False),
                                         (4096, 2048, True), (10240, 2048, False), (16384, 2048, True), (20480, 2048, False),
                                         (4096, 3072, False), (8448, 4096, False), (14336, 4096, False)])
def test_w4a16_tokens_on_the_faster_gemm(rows, k, wide):
    """17 to 32 tokens: the side that measured faster, at both ends of the rule's rows and K."""
    from ztensor_amd.engine import _few_tokens

    s = object.__new__(st.GPTQStorage)
    for t in (17, 32):
        assert _few_tokens(s, rows, k, torch.empty(t, k, dtype=torch.float16)) == wide
        assert not _few_tokens(s, rows, k, torch.empty(t, k))
