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
