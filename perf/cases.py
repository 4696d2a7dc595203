"""The calls a user of the two attention operators makes, from the smallest to the largest.

Every case names an operator ("rope": fused RoPE attention, "corope": Co-RoPE grouped-query attention), a mode ("forward": a
prefill that keeps nothing, "train": forward and backward through autograd), the tensor type, the sizes, whether the mask is
causal, and how q, k, v lie in memory:

  bhnd  contiguous (batch, heads, positions, head dim), as the reference's own scripts hold them
  bnhd  (batch, positions, heads, head dim) seen as (batch, heads, positions, head dim), which is what a model gets from its
        projections; the gradient of the output arrives in that layout too
  qkv   three views of one fused (batch, positions, 3, heads, head dim) projection
"""
import math

import torch

import corope_amd

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
_THETA = 10000.0


def _case(op, mode, dtype, B, H, Hkv, N, D, causal=True, layout="bhnd", name=None):
    c = {"op": op, "mode": mode, "dtype": dtype, "B": B, "H": H, "Hkv": Hkv, "N": N, "D": D, "causal": causal, "layout": layout}
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # one short prompt, 32 heads: a call that is all latency
        _case("rope", "forward", "bf16", 1, 32, 32, 96, 128, name="rope_prompt_96"),
        # the smallest shape of the 19-shape sweep, one training step: launches and host work
        _case("rope", "train", "bf16", 4, 8, 8, 512, 64, name="rope_train_512_d64"),
        # an encoder's step: every position sees every other, a ragged length, head dim 64
        _case("rope", "train", "bf16", 4, 16, 16, 1000, 64, causal=False, name="rope_train_1000_d64_full"),
        # prefill of a batch of prompts out of a fused projection
        _case("rope", "forward", "bf16", 4, 32, 32, 1024, 128, layout="qkv", name="rope_prefill_1k_qkv"),
        # training in the reference's own type
        _case("rope", "train", "fp16", 2, 32, 32, 2048, 128, name="rope_train_2k_fp16"),
        # grouped-query training inside a model: projections as they come, a length that is no multiple of any tile
        _case("rope", "train", "bf16", 1, 32, 8, 3001, 128, layout="bnhd", name="rope_train_gqa_3001"),
        # the headline shape of the benchmark
        _case("rope", "train", "bf16", 2, 32, 32, 4096, 128, name="rope_train_4k"),
        # the largest head dim
        _case("rope", "train", "bf16", 2, 16, 16, 2048, 256, name="rope_train_2k_d256"),
        # prefill of one very long sequence
        _case("rope", "forward", "bf16", 1, 8, 8, 65536, 128, name="rope_prefill_64k"),
        # Co-RoPE: a small training step
        _case("corope", "train", "bf16", 2, 8, 2, 512, 64, name="corope_train_512_d64"),
        # Co-RoPE prefill, fp16, a ragged length
        _case("corope", "forward", "fp16", 1, 32, 8, 1111, 128, name="corope_prefill_1111_fp16"),
        # Co-RoPE training at the benchmark's shape
        _case("corope", "train", "bf16", 2, 32, 8, 4096, 128, name="corope_train_4k"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = "corope" if rng.random() < 0.3 else "rope"
    mode = rng.choice(["forward", "train"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    D = rng.choice([64, 128] if op == "corope" else [64, 64, 128, 128, 128, 256])
    causal = op == "corope" or rng.random() < 0.75
    layout = rng.choice(["bhnd", "bnhd"] + (["qkv"] if mode == "forward" and op == "rope" else []))
    while True:
        B = _log_int(rng, 1, 8)
        Hkv = _log_int(rng, 1, 32)
        group = 1 if layout == "qkv" else rng.choice([1, 2, 4, 8] if op == "corope" else [1, 1, 2, 4, 8])
        # lengths over the whole range, odd ones as often as multiples of 64
        N = _log_int(rng, 64, 4096 if op == "corope" else 65536)
        if rng.random() < 0.5:
            N = max(64, N // 64 * 64)
        c = _case(op, mode, dtype, B, Hkv * group, Hkv, N, D, causal, layout)
        # no larger than the largest listed case of the operator, and not so small that nothing is left to time
        cap = 0.6 * work(listed()[8 if op == "rope" else 11])["flops"]
        if B * Hkv * group <= 256 and 2.0e7 <= work(c)["flops"] <= cap and B * Hkv * group * N * D <= 1 << 27:
            return c


def _laid_out(gen, c, heads, dtype):
    B, N, D = c["B"], c["N"], c["D"]
    if c["layout"] == "bhnd":
        return torch.randn(B, heads, N, D, device="cuda", generator=gen).to(dtype)
    return torch.randn(B, N, heads, D, device="cuda", generator=gen).to(dtype).transpose(1, 2)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]
    if case["layout"] == "qkv":
        fused = torch.randn(case["B"], case["N"], 3, case["H"], case["D"], device="cuda", generator=gen).to(dtype)
        q, k, v = (fused[:, :, i].transpose(1, 2) for i in range(3))
    else:
        q, k, v = (_laid_out(gen, case, h, dtype) for h in (case["H"], case["Hkv"], case["Hkv"]))
    state = {"case": case, "q": q, "k": k, "v": v, "sm_scale": case["D"] ** -0.5}
    if case["op"] == "rope":
        state["cos"], state["sin"] = corope_amd.precompute_freqs_cis(case["D"], case["N"], _THETA, device="cuda")
    if case["mode"] == "train":
        state["grad_out"] = _laid_out(gen, case, case["H"], dtype)
        for name in ("q", "k", "v"):
            state[name].requires_grad_(True)
    return state


def run(state):
    case, q, k, v = state["case"], state["q"], state["k"], state["v"]
    if case["op"] == "rope":
        out = corope_amd.attention(q, k, v, case["causal"], state["sm_scale"], state["cos"], state["sin"])
    else:
        out = corope_amd.corope_attention(q, k, v, case["causal"], state["sm_scale"], _THETA)
    if case["mode"] == "forward":
        return out
    dq, dk, dv = torch.autograd.grad(out, (q, k, v), state["grad_out"])
    return {"out": out.detach(), "dq": dq, "dk": dk, "dv": dv}


def work(case):
    B, H, Hkv, N, D = (case[n] for n in ("B", "H", "Hkv", "N", "D"))
    train = case["mode"] == "train"
    q_like, kv_like = 2 * B * H * N * D, 2 * B * Hkv * N * D
    # q, k, v in and the output out; in training also its gradient in and dq, dk, dv out
    nbytes = 2 * q_like + 2 * kv_like
    if train:
        nbytes += 2 * q_like + 2 * kv_like
    pairs = B * N * (N + 1) // 2 if case["causal"] else B * N * N
    if case["op"] == "rope":
        nbytes += 2 * 4 * N * (D // 2)
        # scores and P V; backward: scores again, dP, dV, dK, dQ
        flops = pairs * H * 2 * D * (7 if train else 2)
    else:
        # per group: the leader's logits and one rotation of the key (a sine, a cosine and 7 operations per pair of columns);
        # backward: the logits and the rotation again, one rotation of the summed queries, and the gate's two products
        flops = pairs * (H * 2 * D * (8 if train else 2) + Hkv * (2 * D * (4 if train else 1) + 9 * (D // 2) * (3 if train else 1)))
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # Measured against the same path in 64 bits (per output, 2-norm), and stated at three to four times that: bf16 2.6e-3 to
    # 3.9e-3 (RoPE) and 1.7e-3 to 2.4e-3 (Co-RoPE); fp16 3.1e-4 to 4.8e-4, except the fp16 RoPE forward that keeps nothing for a
    # backward, whose probabilities are bf16 (2.2e-3).
    if case["dtype"] == "bf16":
        return {"rel": 1.2e-2 if case["op"] == "rope" else 8e-3}
    return {"rel": 8e-3 if case["op"] == "rope" and case["mode"] == "forward" else 1.8e-3}
