"""The extension module behind Plan.execute and Istft.execute runs the calls itself (it does not fall through
to ctypes), and on torch's current stream: a call queued behind a producer that is still running on a side
stream sees its output."""
import pytest

pytestmark = pytest.mark.gpu


def test_calls_are_native():
    import torch

    import sip_amd
    native = sip_amd.fft.N.py_exec()

    class Other(torch.Tensor):
        pass

    p = sip_amd.Plan("c2c", (64,), 3)
    s = sip_amd.Istft(2, 60, 7, 15)
    try:
        x = torch.randn(3, 64, device="cuda", dtype=torch.complex64)
        out = torch.empty_like(x)
        assert native.execute(p.handle.value, p._code, None, x, out) is None
        torch.cuda.synchronize()
        assert torch.equal(torch.view_as_real(out), torch.view_as_real(p.execute(x)))
        assert native.execute(p.handle.value, p._code, None, x.as_subclass(Other), out) is NotImplemented
        assert native.execute(p.handle.value, p._code, None, x.cpu(), out) is NotImplemented
        spec = torch.randn(2, 60, 7, device="cuda", dtype=torch.complex64)
        w = torch.hann_window(60, device="cuda")
        y = torch.empty(2, s.out_len, device="cuda", dtype=torch.complex64)
        ws = s.workspace_on(spec.device)
        assert native.execute_istft(s.handle.value, ws, spec, w, y) is None
        assert native.execute_istft(s.handle.value, ws, spec.as_subclass(Other), w, y) is NotImplemented
        torch.cuda.synchronize()
    finally:
        p.close()
        s.close()


def test_current_stream():
    import torch

    import sip_amd
    n, batch = 1024, 64
    p = sip_amd.Plan("c2c", (n,), batch)
    try:
        late = torch.randn(batch, n, device="cuda", dtype=torch.complex64)
        want = p.execute(late)
        x, out = torch.zeros_like(late), torch.empty_like(late)
        a = torch.randn(4096, 4096, device="cuda")
        torch.mm(a, a)
        torch.cuda.synchronize()
        side = torch.cuda.Stream()
        with torch.cuda.stream(side):
            for _ in range(20):  # some ms in front of the copy
                a = torch.mm(a, a).mul_(1e-2)
            x.copy_(late)
            p.execute(x, out=out)
        side.synchronize()
        assert torch.equal(torch.view_as_real(out), torch.view_as_real(want))
    finally:
        torch.cuda.synchronize()
        p.close()
