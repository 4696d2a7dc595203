"""The native host side against the Python binding it stands in for: the same bits on every form of call that either takes, the same
errors on calls that both refuse."""
import math

import pytest
import torch

from oracle import rope_attn_oracle as O

pytestmark = pytest.mark.gpu


class _Refuses:
    """A native host side to which no call is a plain one."""
    def __getattr__(self, name):
        return lambda *args: None


@pytest.fixture
def both_ways(pkg, monkeypatch):
    """run(f) -> [f() through the native host side, f() through the Python binding]; an exception counts as its type and text.  run.seen: (name, whether
    it took the call) for the calls that the native side was asked for."""
    lib = pkg._lib.load()
    native, seen = lib.host, []

    class _Counts:
        def __getattr__(self, name):
            def call(*args):
                out = getattr(native[0], name)(*args)
                seen.append((name, out is not None))
                return out
            return call

    def attempt(f):
        try:
            return f()
        except Exception as e:
            return type(e), str(e)

    def run(f):
        results = []
        for host in (_Counts(), _Refuses()):
            monkeypatch.setattr(lib, "host", (host, native[1]))
            results.append(attempt(f))
            torch.cuda.synchronize()
        monkeypatch.setattr(lib, "host", native)
        return results

    run.seen = seen
    return run


def _views(layout, B, H, Hkv, N, D, dtype, gen):
    def one(h, kind):
        if kind == "bnhd":
            return torch.randn(B, N, h, D, device="cuda", generator=gen).to(dtype).transpose(1, 2)
        if kind == "narrow":         # rows of another tensor: row stride a multiple of 8, batch stride larger than the rows
            return torch.randn(B, h, N + 3, D + 8, device="cuda", generator=gen).to(dtype)[:, :, 2:N + 2, :D]
        if kind == "odd_rows":       # row stride no multiple of 8: read by neither, copied
            return torch.randn(B, h, N, D + 3, device="cuda", generator=gen).to(dtype)[..., :D]
        if kind == "misaligned":     # contiguous, two bytes past a 16-byte boundary
            return torch.randn(B * h * N * D + 1, device="cuda", generator=gen).to(dtype)[1:].view(B, h, N, D)
        if kind == "transposed":     # columns apart
            return torch.randn(B, h, D, N, device="cuda", generator=gen).to(dtype).transpose(2, 3)
        return torch.randn(B, h, N, D, device="cuda", generator=gen).to(dtype)
    if layout == "qkv":
        f = torch.randn(B, N, 3, H, D, device="cuda", generator=gen).to(dtype)
        return [f[:, :, i].transpose(1, 2) for i in range(3)]
    return [one(h, layout) for h in (H, Hkv, Hkv)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,H,Hkv,N,D", [(1, 2, 2, 1, 64), (2, 4, 2, 70, 128), (1, 3, 3, 130, 256), (2, 2, 2, 520, 64)])
@pytest.mark.parametrize("layout", ["bhnd", "bnhd", "qkv", "narrow", "odd_rows", "misaligned", "transposed"])
def test_rope_same_bits_both_ways(pkg, both_ways, layout, B, H, Hkv, N, D, dtype):
    if layout == "qkv":
        Hkv = H
    gen = torch.Generator(device="cuda").manual_seed(7)
    q, k, v = _views(layout, B, H, Hkv, N, D, dtype, gen)
    g = _views(layout if layout != "qkv" else "bnhd", B, H, H, N, D, dtype, gen)[0]
    c, s = (t.cuda() for t in O.precompute_freqs_cis(D, N))
    scale = 1 / math.sqrt(D)

    def forward():
        return [pkg.attention(q.detach(), k.detach(), v.detach(), True, scale, c, s)]

    def train():
        x = [t.detach().requires_grad_(True) for t in (q, k, v)]
        out = pkg.attention(*x, False, scale, c, s)
        return [out.detach(), *torch.autograd.grad(out, x, g)]

    plain = layout in ("bhnd", "bnhd", "qkv", "narrow") or (layout == "transposed" and N == 1)
    for f in (forward, train):
        both_ways.seen.clear()
        a, b = both_ways(f)
        # (what a forward keeps is plain in any case, and a gradient of another layout is copied)
        assert both_ways.seen == [("rope_forward", plain)] + [("rope_backward", True)] * (f is train and layout != "misaligned")
        if layout == "misaligned":
            assert a[0] is ValueError and a == b
        else:
            assert all(torch.equal(x, y) and x.is_contiguous() and y.is_contiguous() for x, y in zip(a, b)), f.__name__


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("layout", ["bhnd", "bnhd", "misaligned"])
def test_corope_same_bits_both_ways(pkg, both_ways, layout, dtype):
    gen = torch.Generator(device="cuda").manual_seed(8)
    q, k, v = _views(layout, 2, 4, 2, 90, 64, dtype, gen)
    g = _views(layout, 2, 4, 4, 90, 64, dtype, gen)[0]

    def train():
        x = [t.detach().requires_grad_(True) for t in (q, k, v)]
        out = pkg.corope_attention(*x, True, 0.125, 10000.0)
        return [out.detach(), *torch.autograd.grad(out, x, g)]

    a, b = both_ways(train)
    if layout == "misaligned":
        assert a[0] is ValueError and a == b and both_ways.seen == [("gqa_forward", False)]
    else:
        assert both_ways.seen == [("gqa_forward", True), ("gqa_backward", True)]
        assert len(a) == len(b) == 4 and all(torch.equal(x, y) for x, y in zip(a, b))


def test_tables_of_other_forms_both_ways(pkg, both_ways):
    B, H, N, D = 1, 2, 70, 64
    gen = torch.Generator(device="cuda").manual_seed(9)
    q, k, v = (torch.randn(B, H, N, D, device="cuda", generator=gen).bfloat16() for _ in range(3))
    c, s = (t.cuda() for t in O.precompute_freqs_cis(D, N + 5))
    forms = [(c, s), (c.double(), s.double()), (c[:, :D // 2], s[:, :D // 2]), (c[:, :D // 2].contiguous(), s), (c[1:], s[1:]), (c.t().contiguous().t(), s),
             (c.clone().requires_grad_(True), s), (c[:N - 1], s), (c.cpu(), s), (c[:, :D // 2 - 2], s), (c[None], s[None])]
    for fc, fs in forms:
        a, b = both_ways(lambda: [pkg.attention(q, k, v, True, 0.125, fc, fs).detach()])
        assert a == b if isinstance(a, tuple) else torch.equal(a[0], b[0]), (fc.shape, fc.stride(), fc.dtype, a, b)


def test_refused_calls_both_ways(pkg, both_ways):
    t = lambda *s, d=torch.bfloat16, dev="cuda": torch.zeros(*s, device=dev, dtype=d)
    c, s = (x.cuda() for x in O.precompute_freqs_cis(64, 40))
    good = t(1, 2, 40, 64)
    calls = [(good, t(1, 2, 41, 64), good), (good, t(1, 3, 40, 64), t(1, 3, 40, 64)), (good, good, t(1, 1, 40, 64)), (t(1, 2, 40, 48),) * 3, (t(2, 40, 64),) * 3,
             (good, good, t(1, 2, 40, 64, d=torch.float16)), (t(1, 2, 40, 64, d=torch.float32),) * 3, (good, good, t(1, 2, 40, 64, dev="cpu")),
             (t(1, 2, 40, 64, dev="cpu"),) * 3, (t(0, 2, 40, 64),) * 3, (t(2, 2, 40, 64), good, good)]
    for x in calls:
        for args in ((True, 0.125, c, s), (True, -1.0, c, s)):
            a, b = both_ways(lambda: pkg.attention(*x, *args))
            assert isinstance(a, tuple) and a == b, (x[0].shape, x[1].shape, a, b)
        a, b = both_ways(lambda: pkg.corope_attention(*x, True, 0.125, 10000.0))
        assert isinstance(a, tuple) and a == b, (x[0].shape, x[1].shape, a, b)
    for args in ((True, 0.0, c, s), (True, float("inf"), c, s)):
        a, b = both_ways(lambda: pkg.attention(good, good, good, *args))
        assert a[0] is ValueError and a[0] == b[0]


def test_transforms_and_hooks_meet_the_operator_as_before(pkg, both_ways):
    B, H, N, D = 1, 2, 70, 64
    gen = torch.Generator(device="cuda").manual_seed(10)
    q, k, v = (torch.randn(B, H, N, D, device="cuda", generator=gen).bfloat16() for _ in range(3))
    c, s = (t.cuda() for t in O.precompute_freqs_cis(D, N))
    f = lambda q, k, v: pkg.attention(q, k, v, True, 0.125, c, s)
    batch = [t[None].expand(2, *t.shape).contiguous() for t in (q, k, v)]
    for call in (lambda: torch.func.vmap(f)(*batch), lambda: torch.func.grad(lambda x: f(x, k, v).float().sum())(q),
                 lambda: torch.func.jvp(lambda x: f(x, k, v), (q,), (q,))):
        a, b = both_ways(call)
        assert isinstance(a, tuple) and isinstance(a[0], type) and a == b
    packed = []

    def train():
        x = [t.clone().requires_grad_(True) for t in (q, k, v)]
        with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.shape), t.cpu())[1], lambda t: t.cuda()):
            out = f(*x)
        return [out.detach(), *torch.autograd.grad(out, x, out.detach())]

    a, b = both_ways(train)
    assert all(torch.equal(x, y) for x, y in zip(a, b)) and len(packed) == 14
