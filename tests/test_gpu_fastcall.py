"""The native calls (h3mi._fast) give the bytes of the Python path, leave every
other form of a call to it, and raise what it raises."""
import pytest
import torch

from util import gemm_inputs, norm_inputs

pytestmark = pytest.mark.gpu


class _Never:
    """_fast with every call declined."""

    def __getattr__(self, name):
        return lambda *a: None


def _both(monkeypatch, f):
    """f() through the native calls and through Python alone: their results, or the exceptions' types."""
    import h3mi
    from h3mi import fused, gemm, linear, quant, rope

    def outcome():
        try:
            return f(h3mi)
        except Exception as e:  # noqa: BLE001
            return type(e)

    fast = outcome()
    with monkeypatch.context() as m:
        for mod in (fused, gemm, linear, quant, rope):
            m.setattr(mod, "_fast", _Never())
        return fast, outcome()


def _same(a, b):
    if isinstance(a, type) or isinstance(b, type):
        return a is b
    a, b = (a,) if torch.is_tensor(a) else a, (b,) if torch.is_tensor(b) else b
    return len(a) == len(b) and all(x.shape == y.shape and x.dtype == y.dtype and x.stride() == y.stride()
                                    and torch.equal(x.contiguous().view(torch.uint8), y.contiguous().view(torch.uint8))
                                    for x, y in zip(a, b))


def test_linear_and_quantizers(monkeypatch):
    x, w, ws, bias = (t.cuda() for t in gemm_inputs(37, 100, 512, seed=3))
    wide = torch.cat([x, x], 1)
    from torch.nn import Parameter
    forms = [
        lambda h: h.w8a8_linear(x, w, ws, bias=bias), lambda h: h.w8a8_linear(x, w, ws),
        lambda h: h.w8a8_linear(wide[:, 512:], w, ws),                       # a strided view
        lambda h: h.w8a8_linear(x[None], w, ws, bias=bias),                  # 3-D
        lambda h: h.w8a8_linear(x, Parameter(w, requires_grad=False), ws),
        lambda h: h.w8a8_linear(x, w, ws[:1]), lambda h: h.w8a8_linear(x, w, ws.double()),
        lambda h: h.w8a8_linear(x[:0], w, ws), lambda h: h.w8a8_linear(x.float(), w, ws),
        lambda h: h.w8a8_linear(x[:, :500], w, ws), lambda h: h.w8a8_linear(x, w.cpu(), ws),
        lambda h: h.w8a8_linear(x[:, :200].contiguous(), w[:, :200].contiguous(), ws),   # K % 128
        lambda h: h.w8a8_linear(x, w, ws, bias=bias.float()), lambda h: h.w8a8_linear(x.t(), w, ws),
        lambda h: h.quantize_rowwise(x), lambda h: h.quantize_rowwise(wide[:, 8:520]), lambda h: h.quantize_rowwise(x.cpu()),
        lambda h: h.quantize_rowwise_convrot(x), lambda h: h.quantize_rowwise_convrot(wide, "swiglu"),
        lambda h: h.quantize_rowwise_convrot(x, group_size=128), lambda h: h.quantize_rowwise_convrot(x[:, :257], "swiglu"),
        lambda h: h.quantize_rowwise_convrot(x, "gelu"),
        lambda h: h.int8_mm_scaled(*(q := h.quantize_rowwise(x))[:1], w, q[1], ws, bias=bias),
        lambda h: h.int8_mm_scaled(h.quantize_rowwise(x)[0], w, ws, ws),     # xs of the wrong size
    ]
    for i, f in enumerate(forms):
        a, b = _both(monkeypatch, f)
        assert _same(a, b), (i, a, b)
    import h3mi
    h3mi.w8a8_linear(x, w, ws)
    from h3mi.gemm import _int8_mm_scaled_kernel
    assert _int8_mm_scaled_kernel.best_config == h3mi.config_for(37, 100, 512)


def test_norms_and_rope(monkeypatch):
    x, w, s1, sh, g, o, ridx = (t.cuda() for t in norm_inputs(33, 1032, 3, seed=5, stress=False))
    e = 1e-6
    q, k = (torch.randn(1, 9, 2, 128, device="cuda").bfloat16() for _ in range(2))
    tab = torch.randn(1, 9, 64, 2, 2, device="cuda").bfloat16()
    qw = torch.randn(128, device="cuda").bfloat16()
    c = lambda t: t.clone()
    forms = [
        lambda h: h.norm_mod(x, w, e, ridx, s1, sh), lambda h: h.norm_mod(x, w, torch.tensor(e), ridx, s1, sh),
        lambda h: h.norm_mod(x, w, e, ridx.long(), s1, sh), lambda h: h.norm_mod(x, w, e, ridx, s1[:2], sh),
        lambda h: h.norm_mod(x.t(), w, e, ridx, s1, sh), lambda h: h.norm_mod(x, w, "x", ridx, s1, sh),
        lambda h: h.norm_mod(x, w.cpu(), e, ridx, s1, sh), lambda h: h.norm_mod(x[:, :1030].contiguous(), w, e, ridx, s1, sh),
        lambda h: [y := c(x), h.gate_norm_mod_(y, o, g, w, e, ridx, s1, sh)],
        lambda h: h.gate_norm_mod_(c(x), o[:1], g, w, e, ridx, s1, sh), lambda h: h.gate_norm_mod_(x, x, g, w, e, ridx, s1, sh),
        lambda h: [h.gate_(c(x), o, g, ridx)], lambda h: h.gate_(x, o, g, ridx[:3]), lambda h: h.gate_(x, x, g, ridx),
        lambda h: h.norm_mod_q(x, w, e, ridx, s1, sh), lambda h: h.norm_mod_q(x, w, e, ridx, s1, sh, want_h=True),
        lambda h: [y := c(x), *h.gate_norm_mod_q_(y, o, g, w, e, ridx, s1, sh)],
        lambda h: h.rms_rope_split_half_(c(q), c(k), tab, qw, qw, epsilon=e),
        lambda h: h.rms_rope_split_half_(c(q)[0], c(k)[0], tab[0], qw, qw, epsilon=e, rot_dim=128),
        lambda h: h.rms_rope_split_half_(c(q), c(k), tab, qw, qw, rot_dim=64),
        lambda h: h.rms_rope_split_half_(c(q), c(k), tab[:, :8], qw, qw), lambda h: h.rms_rope_split_half_(c(q), c(k), None, qw, qw),
        lambda h: h.rms_rope_split_half_(c(q), c(k)[:, :, :1], tab, qw, qw), lambda h: h.rms_rope_split_half_(q, q, tab, qw, qw),
    ]
    for i, f in enumerate(forms):
        a, b = _both(monkeypatch, f)
        assert _same(a, b), (i, a, b)


def test_autograd_and_modes(monkeypatch):
    """A call inside vmap, under a dispatch mode, on another stream.  (Autograd: the next test.)"""
    import h3mi
    from torch.utils._python_dispatch import TorchDispatchMode
    x, w, ws, _ = (t.cuda() for t in gemm_inputs(16, 64, 256, seed=1))
    ref = h3mi.w8a8_linear(x, w, ws)

    class Count(TorchDispatchMode):
        n = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            Count.n += 1
            return func(*args, **(kwargs or {}))

    with Count():
        assert torch.equal(h3mi.w8a8_linear(x, w, ws), ref)
    assert Count.n > 0
    a, b = _both(monkeypatch, lambda h: torch.vmap(lambda t: h.w8a8_linear(t, w, ws))(x[None]))
    assert a is b or _same(a, b), (a, b)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        y = h3mi.w8a8_linear(x, w, ws)
    s.synchronize()
    assert torch.equal(y, ref)


def test_requires_grad_and_function_modes(monkeypatch):
    """Arguments that require grad give the same bytes, without a graph, on both
    paths; under a torch-function mode the call is Python's, and the mode sees it."""
    import h3mi
    from torch.overrides import TorchFunctionMode
    x, w, ws, bias = (t.cuda() for t in gemm_inputs(16, 64, 256, seed=2))
    ref = h3mi.w8a8_linear(x, w, ws, bias)
    xg, wsg = x.clone().requires_grad_(), ws.clone().requires_grad_()
    a, b = _both(monkeypatch, lambda h: h.w8a8_linear(xg, w, wsg, bias))
    assert _same(a, b) and torch.equal(a, ref) and not a.requires_grad
    n = norm_inputs(9, 264, 2, seed=4, stress=False)
    nx, nw, s1, sh, g, o, ridx = (t.cuda() for t in n)
    a, b = _both(monkeypatch, lambda h: h.norm_mod(nx.clone().requires_grad_(), nw, 1e-6, ridx, s1, sh))
    assert _same(a, b) and not a.requires_grad
    with torch.no_grad():
        a, b = _both(monkeypatch, lambda h: [h.gate_(nx.clone().requires_grad_(), o, g, ridx)])
    assert _same(a, b)

    class Seen(TorchFunctionMode):
        n = 0

        def __torch_function__(self, func, types, args=(), kwargs=None):
            Seen.n += 1
            return func(*args, **(kwargs or {}))

    with Seen():
        assert torch.equal(h3mi.w8a8_linear(x, w, ws, bias), ref)
        before = Seen.n
        h3mi.norm_mod(nx, nw, 1e-6, ridx, s1, sh)
    assert before > 0 and Seen.n > before
