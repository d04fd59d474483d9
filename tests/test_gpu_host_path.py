"""The native host path (`_host`) against the general way through the same entry
points: the same bits on the forms it takes, and the forms it leaves to the general
way (views, subclasses, hooks, refused arguments) behave as they do there."""
import contextlib

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture
def general(pkg):
    """A context in which every native call answers None: the general way runs."""
    from importlib import import_module
    lib = import_module("fni8serve_amd._lib")

    class Nothing:
        def __getattr__(self, name):
            return lambda *a: None

    @contextlib.contextmanager
    def ctx():
        kept, lib._host = lib.host(), Nothing()
        try:
            yield
        finally:
            lib._host = kept
    return ctx


@pytest.fixture
def taken(pkg):
    """taken(f): the native calls that f() makes, as (name, whether it took the call)."""
    from importlib import import_module
    lib = import_module("fni8serve_amd._lib")
    native = lib.host()

    class Recorder:
        def __init__(self):
            self.calls = []

        def __getattr__(self, name):
            def call(*a):
                out = getattr(native, name)(*a)
                self.calls.append((name, out is not None))
                return out
            return call

    def run(f):
        lib._host = Recorder()
        try:
            f()
            return lib._host.calls
        finally:
            lib._host = native
    return run


def _same(a, b):
    a, b = (t if isinstance(t, (tuple, list)) else (t,) for t in (a, b))
    assert len(a) == len(b)
    for p, q in zip(a, b):
        assert p.dtype == q.dtype and p.shape == q.shape and p.device == q.device
        assert p.is_contiguous() == q.is_contiguous()
        assert torch.equal(p, q)


def _weight(pkg, N, K, G, seed):
    g = torch.Generator().manual_seed(seed)
    if G:
        return pkg.QTensor(torch.randint(0, 256, (N, K // 2), generator=g, dtype=torch.uint8).cuda(),
                           (torch.rand(N, K // G, generator=g) * 0.01).cuda(),
                           scheme="per_group_i4", group_size=G, codebook="int4")
    return pkg.QTensor(torch.randint(-127, 128, (N, K), generator=g, dtype=torch.int8).cuda(),
                       (torch.rand(N, generator=g) * 1e-3).cuda(), scheme="per_row_i8")


def _inputs(K):
    g = torch.Generator().manual_seed(K)
    x = torch.randn(70, 2, K, generator=g).half().cuda()
    yield from (x[:m, 0].contiguous() for m in (1, 4, 5, 16, 64, 65))
    yield x                      # 3-D
    yield x[3, 1]                # 1-D
    yield x[:, 1]                # rows with a stride
    yield x[:1, 1]               # one such row
    yield x[:, :, ::2].repeat(1, 1, 2)
    yield x.transpose(0, 1)      # not viewable as rows: copied by the general way
    yield x[:, :1].expand(70, 2, K)
    yield torch.as_strided(x, (3, K), (8, 1))  # overlapping rows
    yield x[:0, 0]               # no rows


# whether the native path takes each of _inputs
_TAKEN = [True] * 11 + [False] * 4


@pytest.mark.parametrize("G", [0, 64])
def test_forms_taken(pkg, cuda, taken, G):
    """The forms that the native path is there for go through it, and the others do not:
    without this, tests that compare it with the general way would pass if it declined
    everything."""
    K = 512
    qt, w = _weight(pkg, 64, K, G, 1), torch.randn(K).half().cuda()
    bias = torch.randn(64).half().cuda()
    m = pkg.GatedMLP(_weight(pkg, 2 * 256, K, G, 3), _weight(pkg, K, 256, G, 4))
    xs = list(_inputs(K))
    assert len(xs) == len(_TAKEN)
    for x, take in zip(xs, _TAKEN):
        assert taken(lambda: pkg.linear(x, qt)) == [("linear", take)]
        assert taken(lambda: pkg.linear(x, qt, bias)) == [("linear", take)]
        assert taken(lambda: pkg.rmsnorm(x, w)) == [("rmsnorm", take)]
        assert taken(lambda: pkg.rmsnorm_quant(x, w)) == [("rmsnorm", take)]
        assert taken(lambda: m(x))[:1] == [("mlp", take)]
        res = x.contiguous()
        assert taken(lambda: pkg.rmsnorm(x, w, residual=res)) == [("rmsnorm", take)]
        xq, s = pkg.quantize_rowwise(x)
        assert taken(lambda: pkg.gemm_quantized(xq, s, qt)) == [("gemm", x.numel() > 0)]
    x = xs[2]
    assert taken(lambda: pkg.linear(x, qt, torch.stack([bias, bias], 1)[:, 0])) == [("linear", False)]
    assert taken(lambda: pkg.rmsnorm(x, w, residual=xs[8][:x.shape[0]])) == [("rmsnorm", False)]
    graph = torch.cuda.CUDAGraph()
    m(x)

    def capture():
        with torch.cuda.graph(graph):
            m(x)
    assert taken(capture) == [("mlp", True)]


@pytest.mark.parametrize("G", [0, 64])
def test_moe_taken(pkg, cuda, taken, G):
    H, I, E = 512, 256, 16
    experts = [(_weight(pkg, 2 * I, H, G, 10 + e), _weight(pkg, H, I, G, 50 + e)) for e in range(E)]
    for scoring, kw in (("softmax", {}), ("sigmoid", {"num_expert_groups": 4, "topk_group": 2})):
        moe = pkg.SparseMoE(gate=(torch.randn(E, H) / 16).half().cuda(), experts=experts, top_k=3,
                            scoring_func=scoring, **kw)
        for T in (1, 9, 300):
            x = torch.randn(1, T, H).half().cuda()
            assert taken(lambda: moe(x)) == [("moe", True)]
            assert taken(lambda: moe(torch.cat([x, x], 2)[..., :H])) == [("moe", T == 1)]


@pytest.mark.parametrize("G", [0, 32, 128])
def test_linear_forms(pkg, cuda, general, G):
    K = 512
    qt = _weight(pkg, 136, K, G, 1)
    bias = torch.randn(136).half().cuda()
    for x in _inputs(K):
        for b in (None, bias, bias.reshape(1, -1), torch.stack([bias, bias], 1)[:, 0]):
            with general():
                want = pkg.linear(x, qt, b)
            _same(pkg.linear(x, qt, b), want)


@pytest.mark.parametrize("G", [0, 64])
def test_gemm_and_norm_forms(pkg, cuda, general, G):
    K = 512
    qt = _weight(pkg, 72, K, G, 2)
    w = torch.randn(K).half().cuda()
    for x in _inputs(K):
        for res in (None, x, x * 0.5):
            for unit in (False, True):
                with general():
                    want = pkg.rmsnorm(x, w, 1e-5, residual=res, unit_offset=unit)
                    wq = pkg.rmsnorm_quant(x, w, 1e-5, residual=res, unit_offset=unit)
                _same(pkg.rmsnorm(x, w, 1e-5, residual=res, unit_offset=unit), want)
                _same(pkg.rmsnorm_quant(x, w, 1e-5, residual=res, unit_offset=unit), wq)
        xq, xs = wq[:2]
        for a in (xq, torch.cat([xq, xq], 1)[:, :K]):
            with general():
                want = pkg.gemm_quantized(a, xs, qt)
            _same(pkg.gemm_quantized(a, xs, qt), want)


@pytest.mark.parametrize("G1,G2", [(0, 0), (64, 128), (0, 32)])
@pytest.mark.parametrize("act", ["silu", "gelu_pytorch_tanh", "gelu"])
def test_mlp_forms(pkg, cuda, general, G1, G2, act):
    H, I = 256, 512
    m = pkg.GatedMLP(_weight(pkg, 2 * I, H, G1, 3), _weight(pkg, H, I, G2, 4), act=act,
                     bias_down=torch.randn(H).half().cuda())
    for x in _inputs(H):
        with general():
            want = m(x)
        _same(m(x), want)


def test_mlp_module_surgery(pkg, cuda):
    """A hook on a part, a part of another class and a part with its own forward all
    still run: the one-call chain is for untouched modules."""
    H, I = 256, 128
    m = pkg.GatedMLP(_weight(pkg, 2 * I, H, 0, 5), _weight(pkg, H, I, 0, 6))
    x = torch.randn(2, H).half().cuda()
    plain, seen = m(x), []
    for part in (m.gate_up_proj, m.down_proj, m.act_fn):
        h = part.register_forward_hook(lambda mod, a, out: seen.append(type(mod).__name__))
        _same(m(x), plain)
        h.remove()
    assert seen == ["LinearW8A8", "LinearW8A8", "SiluAndMul"]
    m.gate_up_proj.forward = lambda v: pkg.linear(v, m.gate_up_proj.weight) * 0
    assert not torch.equal(m(x), plain)


@pytest.mark.parametrize("M", [2, 9])
def test_mlp_replaced_steps_run(pkg, cuda, general, monkeypatch, M):
    """A compiled part, a rule of its own and a forward put on the class run in the MLP as
    they do the general way."""
    H, I = 256, 128
    x = torch.randn(M, H).half().cuda()
    linear = pkg.LinearW8A8

    def changed(surgery):
        with monkeypatch.context() as mp:
            m = pkg.GatedMLP(_weight(pkg, 2 * I, H, 0, 5), _weight(pkg, H, I, 0, 6))
            before = m(x)
            surgery(m, mp)
            with general():
                want = m(x)
            _same(m(x), want)
            return not torch.equal(want, before)

    assert changed(lambda m, mp: mp.setattr(
        m.gate_up_proj, "_compiled_call_impl", lambda v: 2 * linear.forward(m.gate_up_proj, v)))
    assert changed(lambda m, mp: mp.setattr(
        linear, "forward", lambda self, v: 2 * pkg.linear(v, self.weight)))
    changed(lambda m, mp: mp.setattr(m.gate_up_proj, "_int8_ok", lambda v: False, raising=False))
    changed(lambda m, mp: mp.setattr(type(m.act_fn), "forward", lambda self, v: v[..., :I] * 0))


@pytest.mark.parametrize("G", [0, 64])
@pytest.mark.parametrize("T", [1, 9, 300])
@pytest.mark.parametrize("scoring,groups", [("softmax", None), ("sigmoid", 4)])
def test_moe_forms(pkg, cuda, general, G, T, scoring, groups):
    H, I, E = 512, 256, 16
    experts = [(_weight(pkg, 2 * I, H, G, 10 + e), _weight(pkg, H, I, G, 50 + e)) for e in range(E)]
    moe = pkg.SparseMoE(gate=(torch.randn(E, H) / 16).half().cuda(), experts=experts, top_k=3,
                        scoring_func=scoring, num_expert_groups=groups,
                        topk_group=2 if groups else None, routed_scaling_factor=1.5,
                        e_score_correction_bias=torch.randn(E).cuda() if groups else None)
    x = torch.randn(1, T, H).half().cuda()
    for v in (x, x.transpose(0, 1), torch.cat([x, x], 2)[..., :H]):
        with general():
            want = moe(v)
        _same(moe(v), want)
    moe.route = lambda xf: type(moe).route(moe, xf * 0)   # an instance's own step is used
    with general():
        want = moe(x)
    _same(moe(x), want)


@pytest.mark.parametrize("G", [0, 64])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_moe_under_autocast_is_refused(pkg, cuda, G, dtype):
    """Autocast makes the router's product a 16-bit tensor, half the bytes that the
    routing kernel would read: the native call declines and `moe_route` refuses.  A
    region with autocast off inside it routes as outside."""
    H, I, E = 512, 256, 16
    experts = [(_weight(pkg, 2 * I, H, G, 10 + e), _weight(pkg, H, I, G, 50 + e)) for e in range(E)]
    moe = pkg.SparseMoE(gate=(torch.randn(E, H) / 16).half().cuda(), experts=experts, top_k=3)
    x = torch.randn(1, 9, H).half().cuda()
    want = moe(x)
    with torch.autocast("cuda", dtype):
        with pytest.raises(ValueError, match="fp32 logits"):
            moe(x)
        with torch.autocast("cuda", enabled=False):
            _same(moe(x), want)


def test_refusals_are_the_general_ways(pkg, cuda):
    qt = _weight(pkg, 64, 128, 0, 7)
    x = torch.randn(2, 128).half().cuda()
    for bad in (x.float(), x[:, :64].contiguous(), x.cpu()):
        with pytest.raises(ValueError):
            pkg.linear(bad, qt)
    with pytest.raises(ValueError):
        pkg.linear(x, qt, torch.zeros(63, dtype=torch.float16, device="cuda"))
    with pytest.raises(ValueError):
        pkg.linear(x, qt, torch.zeros(64, device="cuda"))
    with pytest.raises(ValueError):
        pkg.linear(x, pkg.QTensor(qt.data.cpu(), qt.scale, scheme="per_row_i8"))
    with pytest.raises(ValueError):
        pkg.rmsnorm(x, torch.ones(64, dtype=torch.float16, device="cuda"))

    class Sub(torch.Tensor):
        pass
    _same(pkg.linear(x.as_subclass(Sub), qt), pkg.linear(x, qt))


def test_streams_and_graphs(pkg, cuda):
    """The chain runs on the current stream and can be captured."""
    m = pkg.GatedMLP(_weight(pkg, 1024, 256, 0, 8), _weight(pkg, 256, 512, 0, 9))
    x = torch.randn(8, 256).half().cuda()
    want = m(x)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        y = m(x)
    torch.cuda.current_stream().wait_stream(s)
    _same(y, want)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = m(x)
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        _same(out, want)
