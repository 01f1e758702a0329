"""Host side of the FP8 linears without a GPU: the library and the stream lookup are replaced by stubs, so nothing is
launched."""
import pytest
import torch

from lingbot_world_v2_realtime_amd import kernels

F8 = torch.float8_e4m3fn


class StubLib:
    """Stands for the loaded library: every entry point notes its call and reports success."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        return lambda *args: self.calls.append((name, args)) or 0


@pytest.fixture
def stub(monkeypatch):
    lib = StubLib()
    monkeypatch.setattr(kernels._lib, "load", lambda *a: lib)
    monkeypatch.setattr(kernels, "_raw_stream", lambda idx: 0)
    return lib


def test_gemm_refuses_host_tensors(stub):
    """A host pointer must not reach a kernel: all operands on the host, and the stream of a host tensor."""
    m, n, k = 32, 16, 128
    x8, w8 = torch.zeros(m, k).to(F8), torch.zeros(n, k).to(F8)
    with pytest.raises(ValueError, match="device tensor"):
        kernels.gemm_fp8_rows(x8, torch.ones(m, 1), w8, torch.ones(1, n))
    with pytest.raises(ValueError, match="device tensor"):
        kernels.gemm_fp8_mx(x8, torch.zeros(k // 128, m, 4, dtype=torch.uint8), w8,
                            torch.zeros(k // 128, n, 4, dtype=torch.uint8))
    with pytest.raises(ValueError, match="device tensor"):
        kernels._stream(x8)
    assert stub.calls == []
