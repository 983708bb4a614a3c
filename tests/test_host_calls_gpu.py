"""The module's calls in native code (csrc/host/calls.cc) against the Python functions they shorten: same bits in the
ordinary case, and everything that is not ordinary left to Python -- errors, subclasses, captures, missing workspaces."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


class _Leaves:
    """stands in for the native module: leaves every call to Python"""

    @staticmethod
    def fc_Q4A(*a):
        return NotImplemented

    attention_rope2 = fc_Q4A


@pytest.fixture()
def ops():
    import llmops
    from llmops import _lib
    _lib.host()
    yield llmops
    _lib._host = None


def _python_only(fn):
    from llmops import _lib
    _lib._host = _Leaves
    try:
        return fn()
    finally:
        _lib._host = None


def _normal(seed, *shape):
    return torch.randn(*shape, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda")


@pytest.mark.parametrize("G", [32, 128])
@pytest.mark.parametrize("B,M", [(1, 1), (2, 3), (1, 40)])
def test_fc_native_call_gives_the_same_bits(ops, G, B, M):
    w = ops.offline_FC_quant_Q4A(_normal(1, 200, 1024) * 0.02, G)
    x = _normal(2, B, M, 1024)
    want = _python_only(lambda: ops.fc_Q4A(x, w, 200))
    native = ops._lib.host().fc_Q4A(ops._workspaces, x, w, 200)
    assert native is not NotImplemented and native.shape == (B, M, 200) and not native.requires_grad
    assert torch.equal(native, want) and torch.equal(ops.fc_Q4A(x, w, 200), want)
    other = torch.cuda.Stream()  # no workspace of its own yet: Python makes it, then the native call finds it
    with torch.cuda.stream(other):
        assert ops._lib.host().fc_Q4A(ops._workspaces, x, w, 200) is NotImplemented
        first = ops.fc_Q4A(x, w, 200)
        assert torch.equal(ops._lib.host().fc_Q4A(ops._workspaces, x, w, 200), first)
    other.synchronize()
    assert torch.equal(first, want)


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("tokens", [1, 5, 40])
def test_attention_native_call_gives_the_same_bits(ops, tokens, half):
    H, S, past = 4, 128, 70
    inv = 1.0 / (10000.0 ** (torch.arange(0, S, 2, device="cuda").float() / S))
    slots = torch.arange(past, past + tokens, dtype=torch.int32, device="cuda")
    q, k, v = _normal(1, 1, tokens, H * S), _normal(2, 1, tokens, H * S), _normal(3, 1, tokens, H * S)
    cache = _normal(4, 2, 1, H, 128, S).to(torch.float16 if half else torch.float32)

    def run():
        a = [t.clone() for t in (q, k, cache)]
        assert ops.attention_rope2(a[0], a[1], v, inv, a[2], slots, past, 0) is None
        return a

    want = _python_only(run)
    native = [t.clone() for t in (q, k, cache)]
    assert ops._lib.host().attention_rope2(ops._workspaces, native[0], native[1], v, inv, native[2], slots, past, 0) is None
    for a, b, c in zip(run(), native, want):
        assert torch.equal(a, c) and torch.equal(b, c)


def test_native_calls_leave_the_rest_to_python(ops):
    w = ops.offline_FC_quant_Q4A(_normal(1, 64, 256) * 0.02, 128)
    x = _normal(2, 1, 2, 256)
    ops.fc_Q4A(x, w, 64)
    call = ops._lib.host().fc_Q4A

    class Sub(torch.Tensor):
        pass

    left = [(x.as_subclass(Sub), w, 64), (x[:, :, ::2], w, 64), (x.double(), w, 64), (x.cpu(), w, 64), (x[0], w, 64), (x, w.float(), 64),
            (x, w[:, :, :100].contiguous(), 64), (x, w, 64.0), (x, w, True), (x, w, -1), (x, w, 1 << 70), (None, w, 64),
            (torch._neg_view(x), w, 64)]
    for a in left:
        assert call(ops._workspaces, *a) is NotImplemented
    for a in left[1:7]:  # ... where the errors are raised
        with pytest.raises(RuntimeError):
            ops.fc_Q4A(*a)
    with pytest.raises(RuntimeError, match="K"):  # what only the library can refuse, with its own words
        ops.fc_Q4A(x[:, :, :100].contiguous(), w, 64)
    g, s = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.stream(s):
        ops.fc_Q4A(x, w, 64)
    s.synchronize()
    with torch.cuda.graph(g, stream=s):  # a capture has to be noted in the module's bookkeeping
        assert call(ops._workspaces, x, w, 64) is NotImplemented
        y = ops.fc_Q4A(x, w, 64)
    want = ops.fc_Q4A(x, w, 64)
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
