"""GPU parity of the Co-RoPE GQA forward against the CPU oracle (through the C ABI).

Bar: max-abs <= 2e-2 for the bf16 output against the oracle evaluated in fp64/fp32 on the same bf16-rounded
inputs.  Small shapes use the dense oracle; long sequences use its row-sampled form."""
import math

import pytest
import torch

from conftest import bf16_round, seeded
from oracle import corope_gqa_oracle as C

pytestmark = pytest.mark.gpu
TOL = 2e-2


def _inputs(B, Hq, Hkv, N, D, seed=42):
    return (bf16_round(seeded((B, Hq, N, D), seed)), bf16_round(seeded((B, Hkv, N, D), seed + 1)),
            bf16_round(seeded((B, Hkv, N, D), seed + 2)))


def _run(pkg, q, k, v, scale, theta):
    dev = torch.device("cuda:0")
    o = pkg.corope_attention(q.to(dev, torch.bfloat16), k.to(dev, torch.bfloat16), v.to(dev, torch.bfloat16), True,
                             scale, theta)
    torch.cuda.synchronize()
    return o.float().cpu()


# (B, Hq, Hkv, N, D): the reference's compare_corope.py shape first, then every group size and ragged lengths
CASES = [(1, 4, 2, 32, 64), (2, 4, 2, 64, 64), (1, 2, 2, 96, 64), (1, 6, 2, 100, 64), (1, 8, 2, 130, 128),
         (1, 8, 1, 257, 64), (2, 5, 1, 77, 128), (1, 6, 1, 64, 128), (1, 7, 1, 65, 64), (1, 4, 1, 1, 64),
         (2, 8, 2, 512, 128)]


@pytest.mark.parametrize("B,Hq,Hkv,N,D", CASES)
def test_corope_forward_parity(pkg, B, Hq, Hkv, N, D):
    print(f"case B={B} Hq={Hq} Hkv={Hkv} N={N} D={D}", flush=True)
    q, k, v = _inputs(B, Hq, Hkv, N, D)
    scale = 1 / math.sqrt(D)
    o = _run(pkg, q, k, v, scale, 10000.0)
    if N <= 130:
        ref = C.corope_gqa_forward(q, k, v, True, scale, 10000.0, torch.float64).float()
    else:
        ref = C.corope_gqa_forward_rows(q, k, v, True, scale, 10000.0, torch.arange(N), torch.float32)
    err = (o - ref).abs()
    print(f"  O max-abs {err.max():.3e} mean-abs {err.mean():.3e}")
    assert torch.isfinite(o).all()
    assert err.max() <= TOL


def test_corope_unit_scale_small_theta(pkg):
    """sm_scale = 1 and a small base (fast rotations), as in the reference's comparison script (sm_scale=1.0)."""
    q, k, v = _inputs(1, 4, 2, 32, 64, seed=7)
    q, k = bf16_round(q * 0.3), bf16_round(k * 0.3)
    o = _run(pkg, q, k, v, 1.0, 100.0)
    ref = C.corope_gqa_forward(q, k, v, True, 1.0, 100.0, torch.float64).float()
    assert (o - ref).abs().max() <= TOL


def test_corope_zero_leader_matches_rope_kernel(pkg):
    """With a zero leader every gate is 1/2, so the follower heads equal RoPE attention at positions m/2:
    the Co-RoPE kernel and the RoPE-attention kernel must then agree with each other."""
    B, Hq, Hkv, N, D = 1, 4, 2, 256, 64
    G = Hq // Hkv
    q, k, v = _inputs(B, Hq, Hkv, N, D, seed=11)
    q[:, ::G] = 0
    scale = 1 / math.sqrt(D)
    o = _run(pkg, q, k, v, scale, 10000.0)
    w = C.corope_inv_freq(D, 10000.0)
    ang = (torch.arange(N, dtype=torch.float32) / 2).unsqueeze(1) * w.unsqueeze(0)
    cos, sin = torch.cat([ang.cos()] * 2, -1), torch.cat([ang.sin()] * 2, -1)
    dev = torch.device("cuda:0")
    kx, vx = k.repeat_interleave(G, 1), v.repeat_interleave(G, 1)
    o_rope, _ = pkg.rope_attn_forward_with_lse(q.to(dev, torch.bfloat16), kx.to(dev, torch.bfloat16),
                                                vx.to(dev, torch.bfloat16), True, scale, cos.to(dev), sin.to(dev))
    followers = [h for h in range(Hq) if h % G]
    assert (o[:, followers] - o_rope.float().cpu()[:, followers]).abs().max() <= TOL


def test_corope_validation_errors(pkg):
    dev = torch.device("cuda:0")
    q = torch.zeros(1, 4, 64, 64, device=dev, dtype=torch.bfloat16)
    k = torch.zeros(1, 2, 64, 64, device=dev, dtype=torch.bfloat16)
    with pytest.raises(ValueError):
        pkg.corope_attention(q, k, k, False, 1.0, 1e4)
    with pytest.raises(ValueError):
        pkg.corope_attention(q, k[:, :, :32], k[:, :, :32], True, 1.0, 1e4)
    with pytest.raises(ValueError):
        pkg.corope_attention(torch.zeros(1, 18, 64, 64, device=dev, dtype=torch.bfloat16), k, k, True, 1.0, 1e4)
    with pytest.raises(ValueError):
        pkg.corope_attention(q.float(), k.float(), k.float(), True, 1.0, 1e4)


@pytest.mark.parametrize("scale", [None, 1.0])
@pytest.mark.parametrize("B,Hq,Hkv,N,D", [(1, 4, 2, 32, 64), (1, 6, 2, 100, 64), (1, 8, 2, 130, 128), (2, 8, 2, 512, 128)])
def test_corope_forward_fp16(pkg, B, Hq, Hkv, N, D, scale):
    """fp16 tensors, the dtype of the reference's kernel and comparison script (compare_corope.py:18, whose shape comes
    first and which runs at sm_scale = 1): the same kernel built for fp16 elements, against the oracle on the same
    fp16-rounded inputs.  Bar: max-abs <= 2e-2 at 1/sqrt(D); at sm_scale = 1 (logits with a standard deviation of 8 to 11)
    max <= 0.15 and mean <= 5e-3 as for the other hot cases.  (The fp16 backward: test_gpu_corope_bwd.py.)"""
    print(f"case fp16 B={B} Hq={Hq} Hkv={Hkv} N={N} D={D} scale={scale}", flush=True)
    q, k, v = (t.to(torch.float16).float() for t in (seeded((B, Hq, N, D), 5), seeded((B, Hkv, N, D), 6), seeded((B, Hkv, N, D), 7)))
    sc = 1 / math.sqrt(D) if scale is None else scale
    dev = torch.device("cuda:0")
    qd = q.to(dev, torch.float16).requires_grad_(True)
    o = pkg.corope_attention(qd, k.to(dev, torch.float16), v.to(dev, torch.float16), True, sc, 10000.0)
    torch.cuda.synchronize()
    assert o.dtype == torch.float16
    if N <= 130:
        ref = C.corope_gqa_forward(q, k, v, True, sc, 10000.0, torch.float64).float()
    else:
        ref = C.corope_gqa_forward_rows(q, k, v, True, sc, 10000.0, torch.arange(N), torch.float32)
    err = (o.float().cpu() - ref).abs()
    print(f"  O max-abs {err.max():.3e} mean-abs {err.mean():.3e}")
    assert torch.isfinite(o).all()
    if scale is None:
        assert err.max() <= TOL
    else:
        assert err.max() <= 0.15 and err.mean() <= 5e-3


# Many short groups: every number of query rows a wave takes (by group size and by how many rows there are), with lengths that end
# inside a wave's rows, a workgroup's rows and a chunk.  Three of the groups against the oracle.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("groups,G,N,D", [(470, 1, 70, 64), (480, 2, 69, 128), (240, 3, 73, 128), (240, 4, 70, 64), (120, 4, 75, 128),
                                          (120, 5, 71, 64), (120, 8, 70, 128), (60, 1, 139, 128)])
def test_forward_many_groups(pkg, groups, G, N, D, dtype):
    dev = torch.device("cuda:0")
    q, k, v = (bf16_round(seeded((groups, h, N, D), 20 + i)) for i, h in enumerate((G, 1, 1)))
    scale = 1 / math.sqrt(D)
    o = pkg.corope_attention(*(t.to(dev, dtype) for t in (q, k, v)), True, scale, 10000.0)
    torch.cuda.synchronize()
    for g in (0, groups // 2, groups - 1):
        ref = C.corope_gqa_forward(q[g:g + 1].double(), k[g:g + 1].double(), v[g:g + 1].double(), True, scale, 10000.0, torch.float64)
        err = (o[g:g + 1].double().cpu() - ref).abs().max().item()
        assert err <= 2e-2, (g, err)


# A zero temperature (every weight the same) and a negative one: what lies beyond the diagonal has to vanish whatever the scale does to
# it.  One, two and four query rows per wave, lengths that end inside a chunk.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("scale", [0.0, -0.0, -0.125])
@pytest.mark.parametrize("groups,G,N,D", [(1, 2, 100, 64), (2, 8, 77, 128), (130, 4, 70, 64), (240, 4, 70, 64), (240, 3, 73, 128)])
def test_forward_scale_zero_or_negative(pkg, groups, G, N, D, scale, dtype):
    dev = torch.device("cuda:0")
    q, k, v = (bf16_round(seeded((groups, h, N, D), 50 + i)) for i, h in enumerate((G, 1, 1)))
    o = pkg.corope_attention(*(t.to(dev, dtype) for t in (q, k, v)), True, scale, 10000.0)
    torch.cuda.synchronize()
    for g in {0, groups // 2, groups - 1}:
        ref = C.corope_gqa_forward(q[g:g + 1].double(), k[g:g + 1].double(), v[g:g + 1].double(), True, scale, 10000.0, torch.float64)
        assert (o[g:g + 1].double().cpu() - ref).abs().max() <= TOL, g


# Sizes at which the forward takes the slow pairs through the polynomial: two, four and eight rows per wave (the group sizes' most), both
# head dims, ragged lengths, fewer columns than 16.  "open": leaders that see every gate open, so that delta moves by 64 over a chunk of 64 keys
# and the polynomials are used out to their ends; "shut": by next to nothing.
LOW_CASES = [(1, 64, 16, 257, 64, 1e4), (1, 64, 8, 385, 128, 1e4), (1, 64, 8, 449, 128, 1e4), (1, 64, 16, 449, 128, 1e4), (2, 48, 16, 259, 64, 1e4), (2, 64, 32, 129, 128, 1e4),
             (4, 32, 32, 130, 64, 1e4), (4, 64, 32, 131, 128, 1e4), (1, 256, 32, 130, 64, 9300.0), (1, 64, 16, 449, 128, 5e5), (1, 64, 16, 449, 128, 3000.0)]


@pytest.mark.parametrize("gates", ["random", "open", "shut"])
@pytest.mark.parametrize("B,Hq,Hkv,N,D,theta", LOW_CASES)
def test_corope_forward_slow_pairs(pkg, B, Hq, Hkv, N, D, theta, gates):
    """fp16, because its rounding hides the least: |O - O64| <= 4e-3 follows from P's rounding (2^-11 of sum P |v|, |v| < 4.7) and the
    output's own (2^-12 of |O|), a fourth of which is left for the scores; where theta is too small for the polynomial a rotated key
    is rounded, 12 nats of a leader's score by 2^-12, and |O| moves by up to 2e-2.  A leader row that is not finite stays its own."""
    print(f"case B={B} Hq={Hq} Hkv={Hkv} N={N} D={D} theta={theta} {gates}", flush=True)
    G, scale = Hq // Hkv, 1 / math.sqrt(D)
    q, k, v = (torch.randn(B, h, N, D, generator=torch.Generator().manual_seed(9 + i)).half() for i, h in enumerate((Hq, Hkv, Hkv)))
    if gates != "random":   # logits of +-12 from the slowest pair (no rounded rotation in them): sigmoid within 1e-4 of 1 or 0
        k[..., D // 2 - 1] = 4.0
        q[:, ::G, :, D // 2 - 1] = (1 if gates == "open" else -1) * 3.0 * math.sqrt(D)
    dev = torch.device("cuda:0")
    o = pkg.corope_attention(q.to(dev), k.to(dev), v.to(dev), True, scale, theta)
    q_bad = q.clone()
    q_bad[0, 0, N - 3] = float("nan")
    o_bad = pkg.corope_attention(q_bad.to(dev), k.to(dev), v.to(dev), True, scale, theta)
    torch.cuda.synchronize()
    rows = torch.ones(N, dtype=torch.bool)
    rows[N - 3] = False
    assert torch.isfinite(o).all() and torch.isnan(o_bad[0, 0, N - 3]).all()
    assert torch.equal(o_bad[0, :, rows], o[0, :, rows]) and torch.equal(o_bad[1:], o[1:])
    for b, kv in ((0, 0), (B - 1, Hkv - 1)):
        hs, sl = (slice(b, b + 1), slice(kv * G, (kv + 1) * G)), (slice(b, b + 1), slice(kv, kv + 1))
        ref = C.corope_gqa_forward_rows(q[hs].double(), k[sl].double(), v[sl].double(), True, scale, theta, torch.arange(N), torch.float64)
        err = (o[hs].double().cpu() - ref).abs()
        print(f"  O max-abs {err.max():.3e} mean-abs {err.mean():.3e}")
        assert err.max() <= (4e-3 if theta > 8860 else TOL)


@pytest.mark.parametrize("size", [1e-6, 3e-5, 1.1e4])
@pytest.mark.parametrize("B,Hq,Hkv,N,D", [(1, 32, 8, 449, 128), (1, 64, 16, 449, 128), (1, 32, 32, 260, 128), (2, 64, 16, 257, 64)])
def test_corope_forward_fp16_query_sizes(pkg, B, Hq, Hkv, N, D, size):
    """fp16 queries near either end of the type's range, with an sm_scale that makes the logits those of ordinary ones: the rotation must
    keep fp16's bits whatever the queries' size.  Same bar as with ordinary queries (test_corope_forward_slow_pairs, |O - O64| <= 4e-3), on
    the queries as fp16 holds them (1e-6: to five bits)."""
    print(f"case B={B} Hq={Hq} Hkv={Hkv} N={N} D={D} size={size}", flush=True)
    G, scale = Hq // Hkv, 1 / math.sqrt(D) / size
    q, k, v = (torch.randn(B, h, N, D, generator=torch.Generator().manual_seed(60 + i)) for i, h in enumerate((Hq, Hkv, Hkv)))
    q, k, v = (q * size).half(), k.half(), v.half()
    assert torch.isfinite(q).all()
    dev = torch.device("cuda:0")
    o = pkg.corope_attention(q.to(dev), k.to(dev), v.to(dev), True, scale, 10000.0)
    torch.cuda.synchronize()
    for b, kv in ((0, 0), (B - 1, Hkv - 1)):
        hs, sl = (slice(b, b + 1), slice(kv * G, (kv + 1) * G)), (slice(b, b + 1), slice(kv, kv + 1))
        ref = C.corope_gqa_forward_rows(q[hs].double(), k[sl].double(), v[sl].double(), True, scale, 10000.0, torch.arange(N), torch.float64)
        err = (o[hs].double().cpu() - ref).abs()
        print(f"  O max-abs {err.max():.3e} mean-abs {err.mean():.3e}")
        assert err.max() <= 4e-3
