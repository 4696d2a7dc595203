"""GPU parity of the Co-RoPE GQA backward against autograd through the dense CPU oracle (through the C ABI).

The oracle's gradients come from torch.autograd over its dense fp64 forward, which is how the reference checks its
own manual backward (corope-exp/corope_attn_gqa_pytorch.py:326-355).  Bar: max-abs <= 2e-2 for the bf16 gradients,
scaled by sqrt(G) for dK and dV, which sum G heads' contributions before the one rounding."""
import math

import pytest
import torch

from conftest import bf16_round, seeded
from oracle import corope_gqa_oracle as C

pytestmark = pytest.mark.gpu
TOL = 2e-2


def _inputs(B, Hq, Hkv, N, D, seed=42):
    return (bf16_round(seeded((B, Hq, N, D), seed)), bf16_round(seeded((B, Hkv, N, D), seed + 1)),
            bf16_round(seeded((B, Hkv, N, D), seed + 2)), bf16_round(seeded((B, Hq, N, D), seed + 3)))


def _oracle_grads(q, k, v, d_o, scale, theta):
    cd = torch.float64 if q.shape[2] <= 160 else torch.float32   # the dense form holds (B, Hq, N, N, D/2) temporaries
    q, k, v = (t.to(cd).clone().requires_grad_(True) for t in (q, k, v))   # (.to is a no-op for fp32 inputs: never mark the caller's tensor)
    o = C.corope_gqa_forward(q, k, v, True, scale, theta, cd)
    return [g.float() for g in torch.autograd.grad(o, (q, k, v), d_o.to(cd))]


def _gpu_grads(pkg, q, k, v, d_o, scale, theta):
    dev = torch.device("cuda:0")
    qg, kg, vg = (t.to(dev, torch.bfloat16).requires_grad_(True) for t in (q, k, v))
    o = pkg.corope_attention(qg, kg, vg, True, scale, theta)
    o.backward(d_o.to(dev, torch.bfloat16))
    torch.cuda.synchronize()
    return [t.grad.float().cpu() for t in (qg, kg, vg)]


def _compare(got, ref, G):
    for name, a, b, bar in zip(("dQ", "dK", "dV"), got, ref, (TOL, TOL * math.sqrt(G), TOL * math.sqrt(G))):
        err = (a - b).abs()
        print(f"  {name} max-abs {err.max():.3e} mean-abs {err.mean():.3e} (max |ref| {b.abs().max():.3f})", flush=True)
        assert torch.isfinite(a).all()
        assert err.max() <= bar, name


# (B, Hq, Hkv, N, D): every group size, ragged lengths around the 16/32/64 tile edges, both head dims
CASES = [(1, 4, 2, 32, 64), (2, 4, 2, 64, 64), (1, 2, 2, 96, 64), (1, 6, 2, 100, 64), (1, 8, 2, 130, 128),
         (1, 8, 1, 150, 64), (2, 5, 1, 77, 128), (1, 3, 1, 64, 128), (1, 7, 1, 65, 64), (1, 4, 1, 1, 64),
         (1, 1, 1, 33, 128), (1, 4, 2, 384, 64), (1, 4, 1, 449, 128), (1, 8, 1, 100, 128), (1, 7, 1, 70, 128),
         # head dims below the kernels' own run padded to 64 (32 is the shape of the reference's self-check,
         # corope_attn_gqa_pytorch.py:309-321)
         (2, 4, 2, 64, 32), (1, 6, 3, 130, 32), (1, 4, 1, 77, 16)]


@pytest.mark.parametrize("B,Hq,Hkv,N,D", CASES)
def test_corope_backward_parity(pkg, B, Hq, Hkv, N, D):
    print(f"case B={B} Hq={Hq} Hkv={Hkv} N={N} D={D}", flush=True)
    q, k, v, d_o = _inputs(B, Hq, Hkv, N, D)
    scale = 1 / math.sqrt(D)
    _compare(_gpu_grads(pkg, q, k, v, d_o, scale, 10000.0), _oracle_grads(q, k, v, d_o, scale, 10000.0), Hq // Hkv)


def test_corope_backward_unit_scale_small_theta(pkg):
    """sm_scale = 1 and a small base: fast rotations make the path through the gates a large part of dQ and dK.
    dO is halved so that the gradients stay below 4, where half a bf16 step of the result alone is under 8e-3."""
    q, k, v, d_o = _inputs(1, 4, 2, 48, 64, seed=7)
    q, k, d_o = bf16_round(q * 0.3), bf16_round(k * 0.3), d_o * 0.5
    _compare(_gpu_grads(pkg, q, k, v, d_o, 1.0, 100.0), _oracle_grads(q, k, v, d_o, 1.0, 100.0), 2)


def test_corope_backward_hot_softmax(pkg):
    """sm_scale = 1 on unit-variance inputs (the reference's comparison script, compare_corope.py:23): scores of +-20, rows
    dominated by one or two keys.  dO is scaled down so that the gradients stay of order one; the bar is the usual one."""
    q, k, v, d_o = _inputs(1, 4, 2, 64, 64, seed=21)
    d_o = bf16_round(d_o * 0.125)
    _compare(_gpu_grads(pkg, q, k, v, d_o, 1.0, 10000.0), _oracle_grads(q, k, v, d_o, 1.0, 10000.0), 2)


@pytest.mark.parametrize("trend", ["growing", "shrinking"])
def test_corope_score_trend_along_the_sweep(pkg, trend):
    """The kernels sweep a row's keys from the diagonal towards key 0 and move the reference value of their exponentials
    only when a score rises well above it.  Key norms that grow (resp. shrink) towards key 0 make the scores rise chunk
    after chunk (the reference moves again and again) or fall away (it stays at the first chunk's maximum while the
    weights become tiny): forward and all gradients against the oracle in both regimes."""
    B, Hq, Hkv, N, D = 1, 4, 2, 320, 64
    q, k, v, d_o = _inputs(B, Hq, Hkv, N, D, seed=33)
    ramp = torch.linspace(3.0, 0.5, N) if trend == "growing" else torch.linspace(0.3, 2.0, N)
    k = bf16_round(k * ramp[None, None, :, None])
    d_o = bf16_round(d_o * 0.25)
    scale = 1 / math.sqrt(D)
    print(f"case trend={trend}", flush=True)
    dev = torch.device("cuda:0")
    o = pkg.corope_attention(*(t.to(dev, torch.bfloat16) for t in (q, k, v)), True, scale, 10000.0).float().cpu()
    ro = C.corope_gqa_forward(q.double(), k.double(), v.double(), True, scale, 10000.0, torch.float64).float()
    print(f"  O max-abs {(o - ro).abs().max():.3e}", flush=True)
    assert torch.isfinite(o).all() and (o - ro).abs().max() <= TOL
    _compare(_gpu_grads(pkg, q, k, v, d_o, scale, 10000.0), _oracle_grads(q, k, v, d_o, scale, 10000.0), Hq // Hkv)


def test_corope_backward_gate_path_is_material_and_right(pkg):
    """On this input the gradient through the leader's gates is a large part of dQ and dK (the oracle with the
    position offsets cut out of the graph differs by far more than the bar), so parity here pins that path; a
    central finite difference through the dense forward pins the oracle's own gradient for one leader coordinate."""
    q, k, v, d_o = _inputs(1, 4, 2, 48, 64, seed=7)
    q, k, d_o = bf16_round(q * 0.3), bf16_round(k * 0.3), d_o * 0.5
    full = _oracle_grads(q, k, v, d_o, 1.0, 100.0)
    qd, kd, vd = (t.double().requires_grad_(True) for t in (q, k, v))
    o = C.corope_gqa_forward(qd, kd, vd, True, 1.0, 100.0, torch.float64, detach_gates=True)
    cut = [g.float() for g in torch.autograd.grad(o, (qd, kd, vd), d_o.double())]
    assert (full[0] - cut[0]).abs().max() > 10 * TOL and (full[1] - cut[1]).abs().max() > 10 * TOL
    assert torch.equal(full[0][:, 1::2], cut[0][:, 1::2])   # only the leaders' queries feed the gates
    got = _gpu_grads(pkg, q, k, v, d_o, 1.0, 100.0)
    _compare(got, full, 2)
    eps, idx = 1e-4, (0, 0, 40, 5)
    qp, qm = q.double(), q.double()
    qp[idx] += eps
    qm[idx] -= eps

    def loss(qq):
        return (C.corope_gqa_forward(qq, k.double(), v.double(), True, 1.0, 100.0, torch.float64) * d_o.double()).sum()

    fd = float((loss(qp) - loss(qm)) / (2 * eps))
    print(f"  finite difference {fd:.5f}, autograd {float(full[0][idx]):.5f}, gpu {float(got[0][idx]):.5f}")
    assert abs(fd - float(full[0][idx])) <= 1e-5 * max(1.0, abs(fd))
    assert abs(fd - float(got[0][idx])) <= TOL


def test_corope_backward_caller_workspace_and_reuse(pkg):
    """A caller-owned workspace filled with garbage gives the same gradients, whether it holds every group's matrices
    (one pass), some of them (the groups are walked in passes of as many as fit) or a single group's; one that cannot
    hold a single group's is refused."""
    mod = pkg.corope_gqa
    dev = torch.device("cuda:0")
    B, Hq, Hkv, N, D = 2, 6, 3, 70, 64
    q, k, v, d_o = (t.to(dev, torch.bfloat16) for t in _inputs(B, Hq, Hkv, N, D, seed=3))
    need = mod.backward_workspace_bytes(B, Hq, Hkv, N, D)
    packed = sum(64 * (i // 64 + 1) for i in range(N))          # rows hold the keys j <= i, padded to 64-key chunks
    assert need == 4 * (packed * (2 * B * Hkv + 3 * B * Hq) + B * Hkv * N * D)   # + the leader's fp32 dq rows
    a = mod.corope_gqa_backward(q, k, v, d_o, 0.125, 1e4)
    ws = torch.full((need // 4 + 64,), float("nan"), device=dev)
    b = mod.corope_gqa_backward(q, k, v, d_o, 0.125, 1e4, workspace=ws)
    torch.cuda.synchronize()
    for x, y in zip(a, b):
        assert torch.equal(x, y)
    one = mod.backward_min_workspace_bytes(B, Hq, Hkv, N, D)
    assert one * B * Hkv == need
    for groups in (1, 2, 4):              # 6 groups in passes of 1, of 2, and of 4 + 2
        ws.fill_(float("nan"))
        c = mod.corope_gqa_backward(q, k, v, d_o, 0.125, 1e4, workspace=ws[: groups * one // 4 + 3])
        torch.cuda.synchronize()
        for x, y in zip(a, c):
            assert torch.equal(x, y), groups
    with pytest.raises(ValueError):
        mod.corope_gqa_backward(q, k, v, d_o, 0.125, 1e4, workspace=ws[: one // 4 - 1])


def test_corope_backward_keeps_its_own_workspace_between_calls(pkg, monkeypatch):
    """Without a caller's workspace the operator uses one buffer per device and stream, sized by the shape and a cap alone: the second
    call allocates nothing new, a smaller cap walks the groups in passes with the same gradients, release frees it."""
    mod = pkg.corope_gqa
    dev = torch.device("cuda:0")
    B, Hq, Hkv, N, D = 2, 6, 3, 70, 64
    q, k, v, d_o = (t.to(dev, torch.bfloat16) for t in _inputs(B, Hq, Hkv, N, D, seed=5))
    mod.release_backward_workspace()
    key = (dev.index, torch.cuda.current_stream(dev).cuda_stream)
    a = mod.corope_gqa_backward(q, k, v, d_o, 0.125, 1e4)
    ws = mod._workspaces[key]
    assert ws.numel() == mod.backward_workspace_bytes(B, Hq, Hkv, N, D)
    b = mod.corope_gqa_backward(q, k, v, d_o, 0.125, 1e4)
    assert mod._workspaces[key].data_ptr() == ws.data_ptr() and len(mod._workspaces) == 1
    one = mod.backward_min_workspace_bytes(B, Hq, Hkv, N, D)
    mod.release_backward_workspace(dev)
    assert not mod._workspaces
    monkeypatch.setattr(mod, "BACKWARD_WORKSPACE_CAP_BYTES", 2 * one + 5)
    c = mod.corope_gqa_backward(q, k, v, d_o, 0.125, 1e4)
    assert mod._workspaces[key].numel() == 2 * one
    torch.cuda.synchronize()
    for x, y, z in zip(a, b, c):
        assert torch.equal(x, y) and torch.equal(x, z)
    mod.release_backward_workspace()


def test_corope_random_shapes_forward_and_backward(pkg):
    """A seeded sweep over batch, group size, head dim, ragged lengths, temperature and rotation base: forward and
    backward in one go, each tensor against the dense oracle with the bar of conftest.within_bar (2e-2, or one bf16 step
    of the value where it exceeds 2.56; dK and dV scaled by sqrt(G) as above)."""
    import random
    from conftest import within_bar
    rnd = random.Random(5)
    dev = torch.device("cuda:0")
    for case in range(16):
        B, Hkv, G, D = rnd.choice([1, 2]), rnd.choice([1, 2, 3]), rnd.randint(1, 8), rnd.choice([64, 128])
        N = rnd.choice([1, 2, 31, 63, 64, 65, 100, 127, 128, 129, 190])
        scale, theta = rnd.choice([1 / math.sqrt(D), 0.25, 0.05]), rnd.choice([100.0, 10000.0, 500000.0])
        Hq = Hkv * G
        print(f"case {case}: B={B} Hq={Hq} Hkv={Hkv} N={N} D={D} scale={scale:.3f} theta={theta}", flush=True)
        q, k, v, d_o = _inputs(B, Hq, Hkv, N, D, seed=1000 + 4 * case)
        d_o = bf16_round(d_o * 0.5)
        cd = torch.float64 if N <= 130 else torch.float32
        qr, kr, vr = (t.to(cd).clone().requires_grad_(True) for t in (q, k, v))
        o_ref = C.corope_gqa_forward(qr, kr, vr, True, scale, theta, cd)
        g_ref = torch.autograd.grad(o_ref, (qr, kr, vr), d_o.to(cd))
        qg, kg, vg = (t.to(dev, torch.bfloat16).requires_grad_(True) for t in (q, k, v))
        o = pkg.corope_attention(qg, kg, vg, True, scale, theta)
        o.backward(d_o.to(dev, torch.bfloat16))
        torch.cuda.synchronize()
        checks = [("O", o.detach(), o_ref.detach(), TOL)]
        checks += [(n, t.grad, r, TOL * (1.0 if n == "dQ" else math.sqrt(G))) for n, t, r in zip(("dQ", "dK", "dV"), (qg, kg, vg), g_ref)]
        for name, got, ref, tol in checks:
            ok, err = within_bar(got.float().cpu(), ref.float(), tol)
            assert torch.isfinite(got).all() and ok, (case, name, err)


@pytest.mark.parametrize("with_o", [True, False])
@pytest.mark.parametrize("B,Hq,Hkv,N,D", [(1, 4, 2, 130, 64), (1, 8, 2, 100, 128)])
def test_corope_backward_does_not_depend_on_the_scale_of_dO(pkg, B, Hq, Hkv, N, D, with_o):
    """Upstream gradients of a mean-reduced loss (1e-6 and below) and unnormalised ones (1e3): the backward is linear in
    dO, and a power-of-two factor commutes with every rounding in it (the fp16 weights of the dQ sums are normalised per
    row by a power of two of |dO_i|), so grad(2^k dO) == 2^k grad(dO) bit for bit -- and both match the oracle."""
    mod = pkg.corope_gqa
    dev = torch.device("cuda:0")
    q, k, v, d_o = _inputs(B, Hq, Hkv, N, D, seed=11)
    scale = 1 / math.sqrt(D)
    qd, kd, vd, gd = (t.to(dev, torch.bfloat16) for t in (q, k, v, d_o))
    out = pkg.corope_attention(qd, kd, vd, True, scale, 10000.0) if with_o else None
    base = [t.float().cpu() for t in mod.corope_gqa_backward(qd, kd, vd, gd, scale, 10000.0, out=out)]
    _compare(base, _oracle_grads(q, k, v, d_o, scale, 10000.0), Hq // Hkv)
    for kexp in (-24, -20, 10, 14):      # 6e-8, 1e-6, 1e3, 1.6e4
        f = 2.0 ** kexp
        got = [t.float().cpu() for t in mod.corope_gqa_backward(qd, kd, vd, (gd.float() * f).to(torch.bfloat16), scale, 10000.0,
                                                                  out=out)]
        torch.cuda.synchronize()
        for name, a, b in zip(("dQ", "dK", "dV"), got, base):
            assert torch.isfinite(a).all(), (name, kexp)
            assert torch.equal(a, b * f), f"{name} at dO x 2^{kexp}: max rel diff {((a - b * f).abs() / (b.abs() * f + 1e-30)).max():.3e}"


def _f16_round(x):
    return x.to(torch.float16).float()


@pytest.mark.parametrize("B,Hq,Hkv,N,D", [(1, 4, 2, 32, 64), (1, 6, 2, 100, 64), (1, 8, 2, 130, 128), (2, 5, 1, 77, 128),
                                           (1, 4, 1, 449, 128), (2, 4, 2, 64, 32)])
def test_corope_backward_parity_fp16(pkg, B, Hq, Hkv, N, D):
    """fp16 tensors, the dtype of the reference's callers (corope-exp/compare_corope.py:18), forward and backward: the same
    kernels built for fp16 elements, against the oracle on the fp16-rounded inputs, at the bf16 bar (fp16 carries three
    mantissa bits more)."""
    print(f"case fp16 B={B} Hq={Hq} Hkv={Hkv} N={N} D={D}", flush=True)
    q, k, v, d_o = (_f16_round(t) for t in _inputs(B, Hq, Hkv, N, D, seed=11))
    scale = 1 / math.sqrt(D)
    dev = torch.device("cuda:0")
    qg, kg, vg = (t.to(dev, torch.float16).requires_grad_(True) for t in (q, k, v))
    o = pkg.corope_attention(qg, kg, vg, True, scale, 10000.0)
    o.backward(d_o.to(dev, torch.float16))
    torch.cuda.synchronize()
    assert all(t.grad.dtype == torch.float16 for t in (qg, kg, vg))
    ro = C.corope_gqa_forward(q.double(), k.double(), v.double(), True, scale, 10000.0, torch.float64).float()
    print(f"  O max-abs {(o.float().cpu() - ro).abs().max():.3e}", flush=True)
    assert (o.float().cpu() - ro).abs().max() <= TOL
    _compare([t.grad.float().cpu() for t in (qg, kg, vg)], _oracle_grads(q, k, v, d_o, scale, 10000.0), Hq // Hkv)


@pytest.mark.parametrize("kexp", [-8, 5])
def test_corope_backward_fp16_scaled_upstream_gradient(pkg, kexp):
    """fp16 tensors with an upstream gradient of 2^-8 and 2^5 times unit size (fp16's own range leaves room for little
    more): the gradients stay finite and match the oracle at the bar scaled by the same factor."""
    B, Hq, Hkv, N, D = 1, 4, 2, 130, 64
    f = 2.0 ** kexp
    q, k, v, d_o = (_f16_round(t) for t in _inputs(B, Hq, Hkv, N, D, seed=11))
    d_o = _f16_round(d_o * f)
    scale = 1 / math.sqrt(D)
    dev = torch.device("cuda:0")
    qg, kg, vg = (t.to(dev, torch.float16).requires_grad_(True) for t in (q, k, v))
    pkg.corope_attention(qg, kg, vg, True, scale, 10000.0).backward(d_o.to(dev, torch.float16))
    torch.cuda.synchronize()
    ref = _oracle_grads(q, k, v, d_o, scale, 10000.0)
    G = Hq // Hkv
    for name, t, b, bar in zip(("dQ", "dK", "dV"), (qg, kg, vg), ref, (TOL, TOL * math.sqrt(G), TOL * math.sqrt(G))):
        a = t.grad.float().cpu()
        err = (a - b).abs().max()
        print(f"  {name} at dO x 2^{kexp}: max-abs {err:.3e} (bar {bar * f:.3e}, max |ref| {b.abs().max():.3e})", flush=True)
        assert torch.isfinite(a).all() and err <= bar * f, name


@pytest.mark.parametrize("B,Hq", [(8200, 8), (65600, 1)])
def test_corope_more_heads_than_a_grid_axis(pkg, B, Hq):
    """Hkv1 N16 D64 with 65600 query heads, more than the 65535 a grid axis holds; as many groups, the second time, are walked in two
    passes by the backward.  The first, a middle and the last group against the same groups run on their own."""
    mod = pkg.corope_gqa
    dev = torch.device("cuda:0")
    Hkv, N, D = 1, 16, 64
    g = torch.Generator(device=dev).manual_seed(3)
    q, d_o = (torch.randn((B, Hq, N, D), device=dev, dtype=torch.bfloat16, generator=g) for _ in range(2))
    k, v = (torch.randn((B, Hkv, N, D), device=dev, dtype=torch.bfloat16, generator=g) for _ in range(2))
    o = pkg.corope_attention(q, k, v, True, 0.125, 1e4)
    grads = mod.corope_gqa_backward(q, k, v, d_o, 0.125, 1e4)
    torch.cuda.synchronize()
    for b in (0, B // 2, B - 1):
        sl = slice(b, b + 1)
        o1 = pkg.corope_attention(q[sl], k[sl], v[sl], True, 0.125, 1e4)
        g1 = mod.corope_gqa_backward(q[sl], k[sl], v[sl], d_o[sl], 0.125, 1e4)
        torch.cuda.synchronize()
        assert torch.equal(o[sl], o1), b
        for a, r in zip(grads, g1):
            assert torch.equal(a[sl], r), b
    mod.release_backward_workspace()


# One key block cut among many workgroups, a cut inside and across blocks, a ragged last block, more groups than one round of
# workgroups, and lengths whose scratch leaves room for few or no partial sums.
@pytest.mark.parametrize("B,Hq,Hkv,N,D", [(1, 4, 1, 128, 64), (1, 2, 1, 129, 128), (1, 2, 2, 257, 64), (1, 1, 1, 256, 128), (1, 2, 1, 655, 64)])
def test_corope_backward_cut_key_blocks(pkg, B, Hq, Hkv, N, D):
    q, k, v, d_o = _inputs(B, Hq, Hkv, N, D, seed=11)
    scale = 1 / math.sqrt(D)
    _compare(_gpu_grads(pkg, q, k, v, d_o, scale, 1e4), _oracle_grads(q, k, v, d_o, scale, 1e4), Hq // Hkv)


# Many short groups: every number of query rows a wave of the scores kernel takes (by group size and by how many rows there are), with
# lengths that end inside a wave's rows, a block of 16 keys and a chunk.  Three of the groups against the oracle.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("groups,G,N,D", [(240, 1, 70, 64), (240, 2, 69, 128), (240, 3, 73, 128), (240, 4, 70, 64), (120, 4, 75, 128),
                                          (120, 5, 71, 64), (120, 8, 70, 128), (120, 7, 97, 64), (120, 2, 81, 64)])
def test_corope_backward_many_groups(pkg, groups, G, N, D, dtype):
    dev = torch.device("cuda:0")
    q, k, v, d_o = _inputs(groups, G, 1, N, D, seed=23)
    scale = 1 / math.sqrt(D)
    qd, kd, vd = (t.to(dev, dtype).requires_grad_(True) for t in (q, k, v))
    pkg.corope_attention(qd, kd, vd, True, scale, 10000.0).backward(d_o.to(dev, dtype))
    torch.cuda.synchronize()
    for g in (0, groups // 2, groups - 1):
        sl = slice(g, g + 1)
        _compare([t.grad[sl].float().cpu() for t in (qd, kd, vd)], _oracle_grads(q[sl], k[sl], v[sl], d_o[sl], scale, 10000.0), G)


# The phase delta w_d is reduced only where it can leave the sine unit's domain: N w_d / 2 pi <= 255 keeps it inside, so with w_0 = 1
# the kernels change form between N = 1602 and 1603; theta = 1 makes every pair that fast.  dO is zero but for the rows that the oracle
# follows, the last ones -- the largest phases -- among them, so their gradients are all there is.
@pytest.mark.parametrize("theta", [10000.0, 1.0])
@pytest.mark.parametrize("Hq,Hkv,N,D", [(2, 1, 1602, 64), (2, 1, 1603, 64), (4, 1, 1602, 128), (4, 1, 1603, 128), (1, 1, 2100, 128)])
def test_corope_phase_beyond_the_sine_units_domain(pkg, Hq, Hkv, N, D, theta):
    dev = torch.device("cuda:0")
    rows = list(range(0, 6)) + [N // 2] + list(range(N - 6, N))
    q, k, v, d_o = _inputs(1, Hq, Hkv, N, D, seed=29)
    keep = torch.zeros(N, 1)
    keep[rows] = 1.0
    d_o, scale = d_o * keep, 1 / math.sqrt(D)
    qg, kg, vg = (t.to(dev, torch.bfloat16).requires_grad_(True) for t in (q, k, v))
    o = pkg.corope_attention(qg, kg, vg, True, scale, theta)
    got = (o[:, :, rows],) + torch.autograd.grad(o, (qg, kg, vg), d_o.to(dev, torch.bfloat16))
    qr, kr, vr = (t.double().requires_grad_(True) for t in (q, k, v))
    ref = C.corope_gqa_forward_rows(qr, kr, vr, True, scale, theta, torch.tensor(rows), torch.float64)
    ref = (ref,) + torch.autograd.grad(ref, (qr, kr, vr), d_o[:, :, rows].double())
    for name, a, b in zip(("O", "dQ", "dK", "dV"), got, ref):
        # bf16 operands of the products and bf16 results: 1.7e-3 to 2.4e-3 where nothing cancels, and the bar at about four times that
        err = ((a.double().cpu() - b).norm() / b.norm()).item()
        print(f"  {name} rel {err:.3e}", flush=True)
        assert err <= 8e-3, name


# A zero and a negative temperature: O, the reference value of the row sums, and through it every gradient.
@pytest.mark.parametrize("scale", [0.0, -0.125])
@pytest.mark.parametrize("B,Hq,Hkv,N,D", [(1, 4, 2, 100, 64), (1, 8, 1, 77, 128), (1, 1, 1, 130, 128)])
def test_corope_backward_scale_zero_or_negative(pkg, B, Hq, Hkv, N, D, scale):
    q, k, v, d_o = _inputs(B, Hq, Hkv, N, D, seed=51)
    _compare(_gpu_grads(pkg, q, k, v, d_o, scale, 10000.0), _oracle_grads(q, k, v, d_o, scale, 10000.0), Hq // Hkv)


def _bad_row_grads(pkg, groups, G, N, D, row, head, what, dtype):
    """Gradients of many short groups, and the same with one query row of group 3 spoilt; everything the spoilt row cannot reach (other
    groups are compared bit for bit) has to stay as it was."""
    dev = torch.device("cuda:0")
    q, k, v, d_o = (t.to(dev, dtype) for t in _inputs(groups, G, 1, N, D, seed=61))
    bad = q.clone()
    bad[3, head, row, 1] = what
    out = []
    for x in (q, bad):
        x, kd, vd = (t.clone().requires_grad_(True) for t in (x, k, v))
        out.append(torch.autograd.grad(pkg.corope_attention(x, kd, vd, True, 1 / math.sqrt(D), 10000.0), (x, kd, vd), d_o))
    torch.cuda.synchronize()
    for clean, spoilt in zip(*out):
        assert torch.equal(clean[:3], spoilt[:3]) and torch.equal(clean[4:], spoilt[4:])
    return [[t[3].float().cpu() for t in side] for side in out]


BAD_ROWS = [(240, 4, 70, 64, 37), (240, 2, 70, 128, 50), (240, 4, 70, 128, 0), (60, 8, 139, 64, 66), (4, 4, 200, 128, 101), (240, 1, 70, 64, 69)]


# A row whose leader's or own query is not finite has NaN statistics.  Keys behind it do not see it.  (Where a rescaling falls moves by
# what the spoilt row does, so its neighbours agree to the suite's bar, not bit for bit.)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("what", [float("nan"), float("inf")])
@pytest.mark.parametrize("groups,G,N,D,row", BAD_ROWS)
def test_corope_dv_of_keys_behind_a_row_that_is_not_finite(pkg, groups, G, N, D, row, what, dtype):
    for head in {0, G - 1}:
        clean, spoilt = _bad_row_grads(pkg, groups, G, N, D, row, head, what, dtype)
        assert torch.isfinite(spoilt[2][:, row + 1:]).all()
        if row + 1 < N:
            assert (clean[2][:, row + 1:] - spoilt[2][:, row + 1:]).abs().max() <= TOL
        assert not torch.isfinite(spoilt[2][:, :row + 1]).any()


# Rows of one wave share matrix products: a row whose rotated keys are not finite must not reach the dq of the rows beside it.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("what", [float("nan"), float("inf")])
@pytest.mark.parametrize("groups,G,N,D,row", BAD_ROWS)
def test_corope_dq_beside_a_row_that_is_not_finite(pkg, groups, G, N, D, row, what, dtype):
    clean, spoilt = _bad_row_grads(pkg, groups, G, N, D, row, 0, what, dtype)
    others = [i for i in range(N) if i != row]
    assert torch.isfinite(spoilt[0][:, others]).all()
    assert (clean[0][:, others] - spoilt[0][:, others]).abs().max() <= TOL
    assert not torch.isfinite(spoilt[0][0, row]).any()


# A key that is NaN spoils the rows that see it and no row before its block of 32 (the leader's gate path multiplies 32 rows at once).  One that leaves fp16's range only where its rotation
# takes it there (here |cos| + |sin| > 65504 / 49920 of the first pair, about half of the rows) spoils none of the others.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("groups,G,N,D,key", [(240, 4, 70, 64, 33), (240, 2, 70, 128, 20), (240, 3, 73, 128, 34)])
def test_corope_dq_of_rows_beside_those_a_key_spoils(pkg, groups, G, N, D, key, dtype):
    dev = torch.device("cuda:0")
    q, k, v, d_o = _inputs(groups, G, 1, N, D, seed=71)
    for what in (float("nan"), 49920.0):
        bad = k.clone()
        bad[3, 0, key, ::D // 2] = what
        x, kd, vd = (t.to(dev, dtype).requires_grad_(True) for t in (q, bad, v))
        dq = torch.autograd.grad(pkg.corope_attention(x, kd, vd, True, 1 / math.sqrt(D), 10000.0), x, d_o.to(dev, dtype))[0][3].float().cpu()
        assert torch.isfinite(dq[:, :key // 32 * 32]).all()
        if what != what:
            assert not torch.isfinite(dq[:, key:]).any()
            continue
        sl = slice(3, 4)
        aux = C.corope_gqa_forward(q[sl].double(), bad[sl].double(), v[sl].double(), True, 1 / math.sqrt(D), 10000.0, torch.float64, return_aux=True)[1]
        phi = aux["delta"][0, 0, :, key]   # the first pair turns by delta itself
        kept = (phi.cos().abs() + phi.sin().abs()) * what < 65000
        kept[:key] = False
        assert 5 < kept.sum() < N - key - 5
        assert torch.isfinite(dq[:, kept]).all()


# The slow pairs' products of the dk kernel (D = 128): every group size they are built for and one beyond, key blocks of 128 cut short, one row past a
# tile; theta = 3000 turns too fast for them.  "open": leaders that see every gate open, so that delta moves by 128 over a block and the
# polynomials are used out to their ends; "shut": by next to nothing.
@pytest.mark.parametrize("gates", ["random", "open", "shut"])
@pytest.mark.parametrize("Hq,Hkv,N,theta,dtype", [(1, 1, 257, 1e4, torch.float16), (4, 2, 129, 1e4, torch.bfloat16), (3, 1, 300, 5e5, torch.float16),
                                                  (8, 2, 265, 1e4, torch.float16), (5, 1, 200, 1e4, torch.bfloat16), (5, 1, 136, 1e4, torch.float16),
                                                  (6, 1, 150, 1e4, torch.float16), (4, 1, 140, 3000.0, torch.float16)])
def test_corope_backward_slow_pairs(pkg, Hq, Hkv, N, theta, dtype, gates):
    """Relative 2-norm of the gradients' error: rounding the result alone costs up to 2^-12 (fp16) or 2^-9 (bf16), the scores' fp16 rounded keys about as
    much as the former; the bar is twice their sum.  A leader's score of +-12 nats moves by 12 times that rounding, and its weights with it."""
    print(f"case Hq={Hq} Hkv={Hkv} N={N} theta={theta} {dtype} {gates}", flush=True)
    G, D = Hq // Hkv, 128
    scale = 1 / math.sqrt(D)
    q, k, v, d_o = (torch.randn(1, h, N, D, generator=torch.Generator().manual_seed(19 + i)).to(dtype) for i, h in enumerate((Hq, Hkv, Hkv, Hq)))
    if gates != "random":   # logits of +-12 from the slowest pair: sigmoid within 1e-4 of 1 or 0
        k[..., D // 2 - 1] = 4.0
        q[:, ::G, :, D // 2 - 1] = (1 if gates == "open" else -1) * 3.0 * math.sqrt(D)
    dev = torch.device("cuda:0")
    qg, kg, vg = (t.to(dev).requires_grad_(True) for t in (q, k, v))
    o = pkg.corope_attention(qg, kg, vg, True, scale, theta)
    got = torch.autograd.grad(o, (qg, kg, vg), d_o.to(dev), retain_graph=True)
    bad = d_o.clone()
    bad[0, 0, N - 60] = float("nan")
    dk_bad = torch.autograd.grad(o, kg, bad.to(dev))[0]
    torch.cuda.synchronize()
    qd, kd, vd = (t.double().requires_grad_(True) for t in (q, k, v))
    ref = torch.autograd.grad(C.corope_gqa_forward(qd, kd, vd, True, scale, theta, torch.float64), (qd, kd, vd), d_o.double())
    bar = 2 * (2.0 ** -12 + (2.0 ** -12 if dtype == torch.float16 else 2.0 ** -9)) + (0 if gates == "random" else 12 * 2.0 ** -12)
    for name, a, b in zip(("dQ", "dK", "dV"), got, ref):
        err = ((a.double().cpu() - b).norm() / b.norm()).item()
        print(f"  {name} relative error {err:.3e}")
        assert err <= bar, name
    assert torch.isnan(dk_bad[0, 0, : N - 59]).any() and torch.equal(dk_bad[0, 0, N - 59:], got[1][0, 0, N - 59:])


@pytest.mark.parametrize("N", [15, 16, 17, 31, 32, 33, 63, 64, 65, 112, 113, 129, 177])
@pytest.mark.parametrize("D", [64, 128])
def test_corope_backward_leader_lengths(pkg, N, D):
    """The leader's dq, whose gate path four waves sum in turn, 16 keys a step: lengths at which some of them have no step, or one fewer.  One head a
    group, so that all of dQ is the leader's; small dO and sm_scale = 1 as where the gate path is material, with that test's bar."""
    print(f"case N={N} D={D}", flush=True)
    q, k, v, d_o = _inputs(1, 2, 2, N, D, seed=7)
    q, k, d_o = bf16_round(q * 0.3), bf16_round(k * 0.3), d_o * 0.5
    _compare(_gpu_grads(pkg, q, k, v, d_o, 1.0, 100.0), _oracle_grads(q, k, v, d_o, 1.0, 100.0), 1)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Hq,Hkv,N,D", [(8, 2, 513, 128), (5, 1, 449, 128), (6, 1, 449, 128)])
def test_corope_dk_of_slow_pairs_keeps_its_bits(pkg, Hq, Hkv, N, D, dtype):
    """dk's slow pairs as sums of products carry their operands to as many bits as rotated ones (six heads a group: rotated), so that no more
    values are rounded the other way.  Every gate is open (delta moves by 128 over a block of keys), the leaders' slow columns are zero and the
    other heads' scores next to nothing: what is left are the errors of delta, of dS in two parts and of fp32 sums, with which 3.2 % of the values
    (fp16: up to 16.2 %) are not the correctly rounded ones.  An operand in one bf16 part at the power that is 0.23 of the whole adds 2.4e-4, a
    sixteenth of bf16's step, and half as many values again; three such parts less, 2e-5, are a tenth of that."""
    print(f"case Hq={Hq} Hkv={Hkv} N={N} D={D} {dtype}", flush=True)
    G, h = Hq // Hkv, D // 2
    q, k, v, g = (seeded((1, n, N, D), 70 + i) for i, n in enumerate((Hq, Hkv, Hkv, Hq)))
    k, v, g = k * 2.0 ** -8, v * 0.5, g * 4.0
    q[:, ::G], q[..., 0], k[..., 0] = 0.0, 0.0, 4.0
    q[:, ::G, :, 0] = 4.0 * math.sqrt(D)
    dev = torch.device("cuda:0")
    q, k, v, g = (t.to(dev, dtype) for t in (q, k, v, g))
    qg, kg, vg = (t.clone().requires_grad_(True) for t in (q, k, v))
    dk = torch.autograd.grad(pkg.corope_attention(qg, kg, vg, True, 1 / math.sqrt(D), 10000.0), kg, g)[0]
    fast = torch.cat([torch.arange(p, p + 3) for p in (h // 2, 3 * h // 4, h + h // 2, h + 3 * h // 4)])   # of each class
    moved = total = 0
    for kv in range(Hkv):
        hs = slice(kv * G, (kv + 1) * G)
        q64, k64, v64 = (t.double().requires_grad_(True) for t in (q[:, hs], k[:, kv:kv + 1], v[:, kv:kv + 1]))
        ref = torch.autograd.grad(C.corope_gqa_forward(q64, k64, v64, True, 1 / math.sqrt(D), 10000.0, torch.float64), k64, g[:, hs].double())[0]
        moved += (dk[:, kv:kv + 1] != ref.to(dtype))[..., fast].sum().item()
        total += ref[..., fast].numel()
    print(f"  {100 * moved / total:.2f} % of {total} values are not the rounded ones")
    assert moved <= (0.045 if dtype == torch.bfloat16 else 0.165) * total
