"""The native front (hexmi/_front.so) against the route through ops.py, and the calls it leaves to that route."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def _calls(hexmi, g, dtype=torch.float16):
    """(name, call without out, the same call through ops.py: an out buffer keeps it from the front)"""
    def r(*shape, dt=dtype):
        return torch.randn(*shape, generator=g).to(dt).cuda()
    x, w, b = r(33, 768), r(768), r(768)
    a, m, n = r(70, 264), r(264, 96), r(96, 264)
    bias, res = r(96), r(70, 96)
    q, k, v = r(2, 3, 130, 64), r(2, 3, 130, 64), r(2, 3, 130, 64)
    qs, ks, vs = (t.view(2, 130, 3, 64).transpose(1, 2) for t in r(2, 130, 3 * 3 * 64).split(192, dim=-1))
    aq, ak, av, mask = r(4, 9, 64), r(4, 1000, 64), r(4, 1000, 64), r(4, 9, 1000)
    long = r(3, 40000)
    out = [("softmax", lambda o: hexmi.softmax(x, out=o)), ("softmax split", lambda o: hexmi.softmax(long, out=o)),
           ("rms", lambda o: hexmi.rms_norm(x, w, 1e-5, out=o)), ("rms bare", lambda o: hexmi.rms_norm(x, out=o)),
           ("layer", lambda o: hexmi.layer_norm(x, w, b, 1e-5, out=o)), ("layer split", lambda o: hexmi.layer_norm(long, out=o)),
           ("matmul", lambda o: hexmi.matmul(a, m, out=o)), ("matmul nt", lambda o: hexmi.matmul(a, n, trans_b=True, out=o)),
           ("linear", lambda o: hexmi.matmul(a, m, bias=bias, residual=res, out=o)),
           ("flash", lambda o: hexmi.flash_attention(q, k, v, 0.2, True, out=o)), ("flash plain", lambda o: hexmi.flash_attention(q, k, v, out=o)),
           ("flash slices", lambda o: hexmi.flash_attention(qs, ks, vs, 0.2, True, out=o)),
           ("attention", lambda o: hexmi.attention(aq, ak, av, out=o)), ("attention mask", lambda o: hexmi.attention(aq, ak, av, mask, 0.1, out=o)),
           ("gelu", lambda o: hexmi.gelu(x, out=o)), ("silu", lambda o: hexmi.silu(x, out=o)),
           ("add", lambda o: hexmi.binary("add", x, x, out=o)), ("div", lambda o: hexmi.binary("div", x, w.expand(33, 768).contiguous(), out=o))]
    if dtype == torch.float16:
        wi, s, z = torch.randint(-127, 128, (96, 264), generator=g, dtype=torch.int8).cuda(), r(96), torch.randint(-9, 9, (96,), generator=g, dtype=torch.int8).cuda()
        out += [("w8", lambda o: hexmi.w8a16_matmul(a, wi, s, out=o)), ("w8 zero", lambda o: hexmi.w8a16_matmul(a, wi, s, zero_points=z, out=o))]
    return out


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_front_gives_what_ops_gives(hexmi, dtype):
    for name, call in _calls(hexmi, torch.Generator().manual_seed(1), dtype):
        got = call(None)
        want = call(torch.empty_like(got))
        assert got.dtype == want.dtype and got.is_contiguous() and torch.equal(got, want), name


def test_front_on_streams_threads_and_under_capture(hexmi):
    calls = _calls(hexmi, torch.Generator().manual_seed(2))
    want = [c(None) for _, c in calls]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for (name, c), w in list(zip(calls, want))[i:] + list(zip(calls, want))[:i]:
                if not torch.equal(c(None), w):
                    bad.append(name)
        s.synchronize()
    threads = [threading.Thread(target=work, args=(3 * i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            got = [c(None) for _, c in calls]
    for _ in range(3):
        for t in got:
            t.fill_(7)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for (name, _), a, b in zip(calls, got, want):
            assert torch.equal(a, b), name


def test_front_only_reads_its_operands(hexmi):
    # A copy-on-write operand stays shared: reading it neither copies it nor needs the memory of a copy (whose allocation may fail).
    f = hexmi.ops._front
    hexmi.lib()
    g = torch.Generator().manual_seed(3)

    def lazy(*shape, dtype=torch.float16):
        base = torch.randn(*shape, generator=g).to(dtype).cuda()
        t = torch._lazy_clone(base)
        assert torch._C._is_cow_tensor(t)
        return base, t
    x, w, b, m, q, kv, ks = (lazy(*s) for s in ((5, 768), (768,), (768,), (768, 64), (2, 3, 130, 64), (4, 1000, 64), (1, 200, 2, 64)))
    wi, s = torch.ones(64, 768, dtype=torch.int8, device="cuda"), torch.ones(64, device="cuda").half()
    for call, operands in ((lambda x, w: f.rms_norm(x, w, 1e-5), (x, w)), (lambda x, w, b: f.layer_norm(x, w, b, 1e-5), (x, w, b)),
                           (f.softmax, (x,)), (lambda x, m: f.matmul(x, m, False, None, None), (x, m)),
                           (lambda x: f.w8a16_matmul(x, wi, s, None), (x,)), (lambda q: f.flash_attention(q, q, q, None, True), (q,)),
                           (lambda k: f.flash_attention(k.transpose(1, 2), k.transpose(1, 2), k.transpose(1, 2), None, True), (ks,)),
                           (lambda k: f.attention(k, k, k, None, None), (kv,)), (lambda x: f.unary(0, x), (x,)),
                           (lambda x: f.binary(0, x, x), (x,))):
        want, got = call(*(t[0] for t in operands)), call(*(t[1] for t in operands))
        assert want is not None and torch.equal(got, want) and all(torch._C._is_cow_tensor(t[1]) for t in operands)


class _Sub(torch.Tensor):
    pass


def test_front_leaves_other_calls_alone(hexmi):
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    hexmi.lib()
    f = hexmi.ops._front
    x = torch.randn(8, 64, device="cuda")
    assert f.softmax(x) is not None and f.softmax(torch.nn.Parameter(x)) is not None
    for other in (x.cpu(), x.t(), x[:, :63], x.double(), x[:0], x.as_subclass(_Sub), 3, None):
        assert f.softmax(other) is None
        assert f.layer_norm(other, None, None, 1e-5) is None and f.unary(0, other) is None and f.binary(0, x, other) is None
    w = torch.ones(64, device="cuda")
    for bad in (w[:63], w.half(), w.cpu(), w[None], "w"):
        assert f.rms_norm(x, bad, 1e-5) is None and f.layer_norm(x, w, bad, 1e-5) is None
    assert f.rms_norm(x, w, "1e-5") is None and f.rms_norm(x, w, 10 ** 400) is None
    h = x.half()
    assert f.matmul(h, h, False, None, None) is None and f.matmul(h, x, True, None, None) is None
    assert f.matmul(h, h, 1, None, None) is None and f.matmul(h, h, True, w, None) is None and f.matmul(h, h, True, None, h) is None
    wi, s = torch.ones(32, 64, device="cuda", dtype=torch.int8), torch.ones(32, device="cuda", dtype=torch.float16)
    assert f.w8a16_matmul(h, wi, s, None) is not None and f.w8a16_matmul(x, wi, s, None) is None
    assert f.w8a16_matmul(h, wi, s[:1], None) is None and f.w8a16_matmul(h, wi, None, None) is None
    q = torch.randn(1, 2, 16, 64, device="cuda").half()
    assert f.flash_attention(q, q, q[:, :, :8], None, False) is None and f.flash_attention(q, q, q, None, 0) is None
    assert f.attention(q[0], q[0], q[0], q[0], None) is None

    class F(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class D(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))
    for mode in (F, D):
        with mode():
            assert f.softmax(x) is None
            assert torch.equal(hexmi.softmax(x), f_want(hexmi, x))
    seen = []
    torch.vmap(lambda t: (seen.append(f.softmax(t)), t)[1])(x)
    assert seen == [None]


def f_want(hexmi, x):
    return hexmi.softmax(x, out=torch.empty_like(x))


def test_front_errors_are_those_of_ops(hexmi):
    q = torch.zeros(1, 4, 300, device="cuda", dtype=torch.float16)          # no kernel for heads of 300
    with pytest.raises(hexmi.HexmiError) as a:
        hexmi.attention(q, q, q)
    with pytest.raises(hexmi.HexmiError) as b:
        hexmi.attention(q, q, q, out=torch.empty_like(q))
    assert str(a.value) == str(b.value) and a.value.status == b.value.status
    with pytest.raises(ValueError):
        hexmi.matmul(q[0], q[0])
    with pytest.raises(TypeError):
        hexmi.softmax(q.double())


def test_dynamo_breaks_its_graph_at_the_front_without_a_warning(hexmi):
    import warnings
    x, w = torch.randn(8, 64, device="cuda"), torch.ones(64, device="cuda")
    for f in (lambda t: hexmi.softmax(t * 2) + 1, lambda t: hexmi.layer_norm(t, w, w, 1e-5) * 2, lambda t: hexmi.gelu(t + 1),
              lambda t: hexmi.binary("add", t, t) * 2, lambda t: hexmi.matmul(t + 1, t, trans_b=True)):
        want = f(x)
        torch._dynamo.reset()
        with warnings.catch_warnings(record=True) as seen:
            warnings.simplefilter("always")
            assert torch.equal(torch.compile(f, backend="eager")(x), want)
        assert not [s for s in seen if "_front" in str(s.message) or "C/C++" in str(s.message)]
