"""Plan.execute and Istft.execute through the extension module (py_exec.cpp) against the ctypes way,
which tensor subclasses take: same bits, same stream, same errors."""
import pytest

pytestmark = pytest.mark.gpu


def make(kind, dims, batch):
    import torch

    import sip_amd
    p = sip_amd.Plan(kind, dims, batch, inverse=(kind == "c2r"))
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(p.in_shape(), generator=g, device="cuda",
                    dtype=torch.float32 if kind == "r2c" else torch.complex64)
    return p, x


@pytest.mark.parametrize("kind,dims,batch", [("c2c", (64,), 3), ("c2c", (65536,), 2), ("c2c", (32, 48), 2),
                                             ("r2c", (100,), 1), ("r2c", (131072,), 1), ("c2r", (4, 6, 20), 2)])
@pytest.mark.parametrize("side", [False, True])
def test_same_as_ctypes(kind, dims, batch, side):
    import torch

    class Other(torch.Tensor):
        pass

    p, x = make(kind, dims, batch)
    try:
        torch.cuda.synchronize()
        with torch.cuda.stream(torch.cuda.Stream() if side else torch.cuda.default_stream()):
            got = p.execute(x)
            ref = p.execute(x.as_subclass(Other), out=torch.empty_like(got))
            again = p.execute(x, out=torch.empty_like(got))
        torch.cuda.synchronize()
        for y in (ref, again):
            assert torch.equal(torch.view_as_real(got) if got.is_complex() else got,
                               torch.view_as_real(y) if y.is_complex() else y)
    finally:
        p.close()


def test_istft_same_as_ctypes():
    import torch

    import sip_amd

    class Other(torch.Tensor):
        pass

    p = sip_amd.Istft(2, 60, 7, 15)
    try:
        x = torch.randn(2, 60, 7, device="cuda", dtype=torch.complex64)
        w = torch.hann_window(60, device="cuda")
        got = p.execute(x, w)
        ref = p.execute(x.as_subclass(Other), w)
        torch.cuda.synchronize()
        assert torch.equal(torch.view_as_real(got), torch.view_as_real(ref))
        with pytest.raises(sip_amd.fft.N.FftError):
            p.execute(x, w[:-1])
    finally:
        p.close()


def test_errors_and_capture():
    import torch

    from sip_amd._native import FftError
    p, x = make("c2c", (256,), 4)
    want = p.execute(x)
    with pytest.raises(FftError, match="asdFftExecC2C returned 100000"):
        p.execute(x[:3])
    with pytest.raises(FftError, match="asdFftExecC2C returned 100000"):
        p.execute(x.real.contiguous())
    out = torch.empty_like(x)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        p.execute(x, out=out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(torch.view_as_real(out), torch.view_as_real(want))
    p.close()
    with pytest.raises(FftError):
        p.execute(x)
