"""Tensors in host memory never reach a kernel: what has no path for them refuses them before anything is launched."""
import pytest
import torch

from copilot_for_consensus_amd.ops import kernels as K


class _Launched(Exception):
    pass


@pytest.fixture
def no_launch(monkeypatch):
    """Any call of the native library is one too many."""
    class Lib:
        def __getattr__(self, name):
            def call(*a):
                raise _Launched(name)
            return call
    monkeypatch.setattr(K, "kernels", Lib)
    # what a process with a GPU gives for a device of -1: the current device's stream
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda device: 0)


def test_the_stream_of_a_host_tensor(no_launch):
    with pytest.raises(ValueError, match="cpu"):
        K._stream(torch.empty(1))


def _quantized():
    return K.QWeight(8, 4, 32, torch.zeros(64, dtype=torch.uint8), (0,))


@pytest.mark.parametrize("call", [
    lambda: K.qgemv(torch.zeros(1, 32, dtype=torch.bfloat16), _quantized()),
    lambda: K.knn_queries(torch.zeros(2, 64), True),
    lambda: K.ivf_topk(torch.zeros(8, 64, dtype=torch.bfloat16), torch.zeros(1, 64, dtype=torch.bfloat16), torch.zeros(1, 1, dtype=torch.int32),
                       torch.tensor([0, 8]), 1, 4),
], ids=["qgemv", "knn_queries", "ivf_topk"])
def test_what_has_no_host_path(no_launch, call):
    with pytest.raises(ValueError, match="cpu"):
        call()


class _Rows(torch.Tensor):
    """Rows of an index that say to be on a GPU."""
    @property
    def device(self):
        return torch.device("cuda", 0)

    def get_device(self):
        return 0


def test_queries_of_a_search_lie_beside_the_index(no_launch, monkeypatch):
    monkeypatch.setattr(K, "_topk_parts", lambda n: 1)
    X = torch.zeros(8, 64, dtype=torch.bfloat16).as_subclass(_Rows)
    for q in (torch.zeros(1, 64), torch.zeros(1, 64, device="meta")):
        with pytest.raises(ValueError, match="queries on"):
            K.knn_search(X, q, 4, True)
    with pytest.raises(_Launched):                   # what lies there goes on to the kernels
        K.knn_search(X, torch.zeros(1, 64).as_subclass(_Rows), 4, True)


def test_rows_of_a_norm_lie_beside_what_they_are_of(no_launch):
    class OnGpu(_Rows):
        is_cuda = True
    x = torch.zeros(4, 8, dtype=torch.bfloat16).as_subclass(OnGpu)
    with pytest.raises(ValueError, match="rows"):
        K.rmsnorm_rows(x, x, torch.zeros(1, dtype=torch.int32), x[0], 1e-5)


@pytest.mark.gpu
def test_queries_of_a_search_on_the_gpu():
    X, q = torch.zeros(8, 128, dtype=torch.bfloat16, device="cuda"), torch.zeros(130, device="cuda")
    with pytest.raises(ValueError, match="queries on"):
        K.knn_search(X, q[:128].view(1, 128).cpu(), 4, True)
    with pytest.raises(ValueError, match="16 bytes"):
        K.knn_search(X, q[1:129].view(1, 128), 4, True)
    assert K.knn_search(X, q[:128].view(1, 128), 4, True)[1].tolist() == [[0, 1, 2, 3]]
