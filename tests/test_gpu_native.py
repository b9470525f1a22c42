"""The native per-call path (flicker_amd/_native) against the Python path it stands in for: the
same bits for the calls it takes, and every other call left to the Python path's handling."""

import pytest
import torch

from flicker_amd import _lib, kernels, modules, w8a8

pytestmark = pytest.mark.gpu
D = 128


class Declines:
    """A native path that takes no call."""

    def __getattr__(self, name):
        return lambda *_: None


def python_path(monkeypatch, f):
    with monkeypatch.context() as m:
        for mod in (kernels, modules, w8a8):
            m.setattr(mod, "_native", Declines())
        return f()


def same(got, want):
    got, want = (x if isinstance(x, tuple) else (x,) for x in (got, want))
    torch.cuda.synchronize()
    for a, b in zip(got, want, strict=True):
        assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride() and a.device == b.device
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))


def stream(device, batch, length, heads, scale_dtype, seed):
    g = torch.Generator().manual_seed(seed)
    qkv = torch.randn(batch, length, 3 * heads * D + 16, generator=g).to(torch.bfloat16).to(device)
    scales = tuple((1 + 0.1 * torch.randn(D, generator=g)).to(scale_dtype).to(device) for _ in range(2))
    return qkv[..., :3 * heads * D], scales


def tables(device, length, width=D, gain=0.3):
    t = torch.randn(2, length, width, generator=torch.Generator().manual_seed(length)).to(device)[..., :D]
    return kernels.Freqs(t[0], t[1], gain)


@pytest.mark.parametrize("batch,length,heads,scale_dtype", [(1, 512, 24, torch.bfloat16), (2, 64, 3, torch.float32)])
@pytest.mark.parametrize("width", [D, D + 4])   # a wider table row stride is the Python path's
def test_qk_prep(device, monkeypatch, batch, length, heads, scale_dtype, width):
    qkv, scales = stream(device, batch, length, heads, scale_dtype, 1)
    freqs = tables(device, length, width)
    taken = kernels._native.qk_prep(qkv, *scales, freqs.cos, freqs.sin, freqs.q_gain, heads)
    assert (taken is not None) == (width == D)
    f = lambda: kernels.qk_prep(qkv, *scales, freqs, heads)   # noqa: E731
    same(f(), python_path(monkeypatch, f))


@pytest.mark.parametrize("heads,lengths", [(24, (512, 256)), (2, (64, 128)), (24, (512, 1024)), (3, (512, 4096))])
def test_double_attention(device, monkeypatch, heads, lengths):
    """The last shape's attention takes the key split, whose workspace is the Python path's."""
    (txt, ts), (img, im) = (stream(device, 1, n, heads, torch.bfloat16, n) for n in lengths)
    freqs = tables(device, sum(lengths), gain=D ** -0.5)
    taken = kernels._native.double_attention(txt, *ts, img, *im, freqs.cos, freqs.sin, freqs.q_gain, heads)
    assert (taken is None) == (lengths == (512, 4096))
    f = lambda: modules.double_attention(txt, img, ts, im, freqs, heads)   # noqa: E731
    same(f(), python_path(monkeypatch, f))


@pytest.mark.parametrize("shape", [(1, 24, 640, D), (2, 24, 1536, D), (1, 3, 4608, D)])
def test_attend_merged(device, monkeypatch, shape):
    g = torch.Generator().manual_seed(shape[2])
    q, k, v = (0.2 * torch.randn(3, *shape, generator=g)).to(torch.bfloat16).to(device)
    taken = kernels._native.attend_merged(q, k, v)
    assert (taken is None) == (shape == (1, 3, 4608, D))   # the key split, whose workspace is the Python path's
    f = lambda: kernels.attend_merged(q, k, v)   # noqa: E731
    same(f(), python_path(monkeypatch, f))
    t = v.transpose(1, 2).contiguous().transpose(1, 2)   # not dense
    assert kernels._native.attend_merged(q, k, t) is None
    same(kernels.attend_merged(q, k, t), f())


@pytest.mark.parametrize("lead", [(17,), (2, 33), ()])
def test_linear(device, monkeypatch, lead):
    g = torch.Generator().manual_seed(4)
    x = torch.randn(*lead, 256, generator=g).to(torch.bfloat16).to(device)
    qw = w8a8.quantize_linear((0.02 * torch.randn(256, 136, generator=g)).to(torch.bfloat16).to(device),
                              x.reshape(-1, 256).abs().amax(0).float())
    assert kernels._native.linear(x, qw.wq_t, qw.w_scale, qw.inv_smooth) is not None
    f = lambda: w8a8.linear(x, qw)   # noqa: E731
    same(f(), python_path(monkeypatch, f))


def test_other_operands_are_left_alone(device):
    """Anything but plain dense operands of the current device gets None, before any launch."""
    n = kernels._native
    qkv, (qs, ks) = stream(device, 1, 64, 2, torch.bfloat16, 9)
    f = tables(device, 64)
    ok = (qkv, qs, ks, f.cos, f.sin, 0.5, 2)
    assert n.qk_prep(*ok) is not None
    for i, bad in ((0, qkv.cpu()), (0, qkv.float()), (0, qkv[0]), (0, None), (1, qs.cpu()), (1, qs.float()),
                   (2, ks[:64]), (3, f.cos[:32]), (3, f.cos.double()), (4, f.sin.t()), (5, 1), (6, 3), (6, 0),
                   (6, "2")):
        args = list(ok)
        args[i] = bad
        assert n.qk_prep(*args) is None, (i, bad)
    assert n.qk_prep() is None and n.attend_merged(1, 2, 3) is None and n.linear(qkv, None, None, None) is None
    with pytest.raises((RuntimeError, ValueError)):
        torch.vmap(lambda t: kernels.qk_prep(t, qs, ks, f, 2)[0])(qkv[None])


@pytest.mark.parametrize("call", ["qk_prep", "attend_merged", "double_attention", "linear"])
def test_runtime_errors_are_raised(device, monkeypatch, call):
    """An error that the HIP runtime holds when a call launches (here one of a refused host call) is
    that call's HipKernelError, as on the Python path, and not hidden by a second attempt."""
    qkv, scales = stream(device, 1, 64, 2, torch.bfloat16, 3)
    q = torch.ones(3, 1, 2, 64, D, dtype=torch.bfloat16, device=device)
    x = torch.ones(4, 128, dtype=torch.bfloat16, device=device)
    qw = w8a8.quantize_linear(torch.ones(128, 8, dtype=torch.bfloat16, device=device), torch.ones(128, device=device))
    f, joint = tables(device, 64), tables(device, 128)
    run = {"qk_prep": lambda: kernels.qk_prep(qkv, *scales, f, 2),
           "attend_merged": lambda: kernels.attend_merged(*q),
           "double_attention": lambda: modules.double_attention(qkv, qkv, scales, scales, joint, 2),
           "linear": lambda: w8a8.linear(x, qw)}[call]

    def pending():
        run()
        torch.cuda.synchronize()
        assert _lib.lib().hipSetDevice(99) != 0
        try:
            with pytest.raises(_lib.HipKernelError) as error:
                run()
        finally:
            _lib.lib().hipGetLastError()
        run()   # the error is reported once
        return str(error.value).split("failed")[1]

    assert pending() == python_path(monkeypatch, pending)
