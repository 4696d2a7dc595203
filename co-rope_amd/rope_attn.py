"""Fused RoPE flash-attention behind the reference's call surface.

``attention(q, k, v, causal, sm_scale, freqs_cos, freqs_sin[, warp_specialize])`` is positional-only, exactly
like the reference's ``attention = _attention.apply`` (fused-rope/fused_rope_attn.py:652-780); the last argument is
accepted and ignored (it selects a Triton code path there).  ``fused_rope_attn`` is a keyword-friendly wrapper.

Forward and backward run hand-written gfx950 kernels through the C ABI in ``include/corope_amd.h``; there is no
other implementation behind this module.  Tensors are bfloat16 or float16 (the reference's dtype, fused_rope_attn.py:236;
the same kernel sources built for fp16 elements)."""
from __future__ import annotations

import ctypes
import functools

import torch

from . import _lib

# 256 (the largest head dim of the reference, fused_rope_attn.py:661) runs one wave per SIMD, on rotated copies a pipelined forward (bf16; fp16
# takes the single-launch kernel there) and, like the others, dQ and fused dK+dV.
_SUPPORTED_D = (64, 128, 256)
_ROTATED_PATH_MAX_D = 256
# Head dims of the reference (fused_rope_attn.py:661) below the kernels' own: run at D = 64 with each half of a row padded
# with zeros (the rotation pairs column j with column j + D/2, so the halves must stay the starts of the new halves).
_PADDED_D = (16, 32)


def spread_halves(x, d_to):
    """(..., D) -> (..., d_to): [x[:D/2], 0, x[D/2:], 0]; zero columns add nothing to any dot product."""
    d = x.shape[-1]
    h, z = d // 2, x.new_zeros(x.shape[:-1] + ((d_to - d) // 2,))
    return torch.cat([x[..., :h], z, x[..., h:], z], dim=-1)


def gather_halves(y, d):
    """Inverse of spread_halves on the columns that carry data."""
    h, hp = d // 2, y.shape[-1] // 2
    return torch.cat([y[..., :h], y[..., hp:hp + h]], dim=-1)


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _stream_ptr(t):
    """The current HIP stream of t's device as an integer handle (the short way when this torch has it: at the small
    shapes the operator is bound by the host, and torch.cuda.current_stream() builds a Python object per call)."""
    if _raw_stream is not None:
        return _raw_stream(t.device.index)
    return torch.cuda.current_stream(t.device).cuda_stream


class _NoGuard:
    def __enter__(self):
        return None

    def __exit__(self, *exc):
        return False


_NO_GUARD = _NoGuard()


def _on_device(t):
    """Context in which t's device is the current one; nothing to enter when it already is."""
    return _NO_GUARD if torch.cuda.current_device() == t.device.index else torch.cuda.device(t.device)


def _check_inputs(q, k, v, freqs_cos, freqs_sin):
    # shape constraints of the reference (fused_rope_attn.py:657-661)
    assert q.dim() == 4 and k.dim() == 4 and v.dim() == 4, "q, k, v must be (B, H, N, D)"
    d = q.shape[-1]
    assert d == k.shape[-1] and d == v.shape[-1], "q, k, v must share the head dim"
    # grouped-query attention (an extension: the reference requires one shape): k, v may have fewer heads
    assert k.shape == v.shape, "k and v must share one shape"
    assert q.shape[0] == k.shape[0] and q.shape[2:] == k.shape[2:], "q and k must agree in batch, sequence and head dim"
    assert q.shape[1] % k.shape[1] == 0, "the number of query heads must be a multiple of the number of key/value heads"
    if d not in _SUPPORTED_D:
        raise ValueError(f"head dim {d} not built for gfx950 (kernels: {_SUPPORTED_D}; padded to 64: {_PADDED_D})")
    if not (q.is_cuda and k.is_cuda and v.is_cuda and freqs_cos.is_cuda and freqs_sin.is_cuda):
        raise ValueError("fused RoPE attention runs on the GPU only: all tensors must be on a HIP device")
    if not (q.dtype == k.dtype == v.dtype and q.dtype in (torch.bfloat16, torch.float16)):
        raise ValueError(f"q, k, v must all be bfloat16 or all float16 (got {q.dtype}, {k.dtype}, {v.dtype})")
    n = q.shape[2]
    for name, f in (("freqs_cos", freqs_cos), ("freqs_sin", freqs_sin)):
        if f.dim() != 2 or f.shape[0] < n or f.shape[1] < d // 2:
            raise ValueError(f"{name} must be (N, D) or (N, D/2) with N >= {n}, got {tuple(f.shape)}")


def _freq_table(f):
    """fp32 table with unit column stride and a row stride the kernels accept."""
    if f.dtype != torch.float32:
        f = f.float()
    if f.stride(1) != 1 or f.stride(0) % 4 != 0 or f.data_ptr() % 16 != 0:
        f = f.contiguous()
        if f.stride(0) % 4 != 0:
            f = torch.nn.functional.pad(f, (0, 4 - f.shape[1] % 4)).contiguous()
    return f


# Shapes from which the operator rotates its operands ahead of the attention kernels: K once into a scratch buffer for
# the forward (every K tile is otherwise rotated again by each query block of its head), and, when a gradient will be asked
# for, q and k once for the backward (fused dK+dV, no tables in its loops, blocks cut into equal pieces where they are few).
# Measured on MI355X, in us, unrotated -> rotated.  Forward and backward: always, B4 H8 N512 D64 52.1 -> 45.9, B1 H32 N96 D128
# 64.3 -> 39.2, B3 Hq64 Hkv32 N64 D64 30.9 -> 26.7, B2 Hq32 Hkv4 N700 D64 299 -> 71, B2 Hq16 Hkv4 N400 D128 243 -> 77, B2 H8 N200
# D256 133 -> 84, B128 H32 N64 D64 265 -> 249, B512 H32 N16 D64 920 -> 869, B128 H32 N16 D256 1013 -> 571 (from N * D = 65536 on it was before).
# The forward alone pays the rotation pass's launch (3 to 4 us) and its way through memory (_forward_pays_rotation).
# What it costs: the rotated q and k beside the caller's own between forward and backward (537 MB at B256 H32 N256 D64, where the step on unrotated
# operands kept references), and a short forward with gradients whose backward never runs (B4 H8 N300 D64 fp16 9.8 -> 11.6).
TWO_LAUNCH_MIN_N = 1024
TRAIN_ROTATED_MIN_ND = 0
_FWD_ROTATED_MIN_ND = 65536


def _forward_pays_rotation(N, D, slabs, kv_slabs, causal, cus):
    """Whether a forward alone that is shorter than 1024 rows and 65536 elements a head takes rotated keys.  Both sides measured on MI355X, in us,
    unrotated -> rotated, B1, 256 compute units:

    D = 64, causal: the unrotated kernel rotates its tiles beside the products of other waves.  H16 N832 19.0 -> 17.4, H32 N832 19.2 -> 18.5, grouped Hq192
    Hkv24 N1000 56.6 -> 54.2; beyond, H48 N896 20.5 -> 21.6, H80 N768 19.3 -> 23.3, H192 N768 40.3 -> 45.9, H224 N960 65.4 -> 71.7.
    D = 64, not causal: H112 N832 46.5 -> 44.3, H256 N896 101.9 -> 91.4; not where the 256-row items are just one round or a little less
    (H64 N832 25.2 -> 27.3, H80 N768 24.8 -> 27.5).
    D = 128, fewer 256-row items than compute units (from there on the unrotated kernel's 256-row form holds out: H128 N300 25.2 -> 26.6): H8 N129
    15.4 -> 14.4, H96 N257 27.4 -> 26.1, H255 N129 not causal 33.0 -> 31.4; causal, up to three blocks of 128 rows, only while those are about one
    round: H128 N160 18.1 -> 18.2; beyond, H160 N160 23.0 -> 26.6, H192 N256 28.4 -> 31.2, H112 N320 28.4 -> 29.9.
    D = 256: H32 N128 26.1 -> 26.7, N160 35.5 -> 27.1, H255 N129 75.9 -> 48.9.
    fp16 (D = 64 and 128; the pipelined kernel with P and V in fp16) goes the same way: D = 64 H32 N1000 22.1 -> 21.2, H192 N800 not causal 74.8 -> 67.5; D = 128
    H32 N160 16.2 -> 14.7, N300 22.5 -> 17.6, and beyond H192 N160 23.4 -> 29.2."""
    items = (N + 255) // 256 * slabs
    if D == 256:
        return N > 128
    if D == 128:
        return N > 128 and items < cus and not (causal and N <= 384 and (N + 127) // 128 * slabs * 8 > cus * 9)
    if D == 64 and causal:
        return N >= 768 and kv_slabs * 8 <= cus
    return D == 64 and N > 768 and not cus * 3 < items * 4 <= cus * 4


@functools.lru_cache(maxsize=None)
def _compute_units(device_index):
    """As the library asks for its own rules: a partition of the card has fewer than its 256."""
    return torch.cuda.get_device_properties(device_index).multi_processor_count


# fp16 tensors, forward of a call that will be differentiated: "exact" keeps P and V in fp16 (O within 1.2e-2 of the fp32 oracle at the
# reference's verification temperature sm_scale = 0.5, gradients within its 0.15 / 5e-3 thresholds): the pipelined forward that looks at
# each half tile's probabilities before it uses them, at D = 256 the single-launch kernel on a key copy rotated beforehand;
# "fast" = the pipelined forward (bf16 probabilities against a V converted to bf16 on its way into LDS: as fast as with
# bf16 tensors, O within one bf16 ulp), whose O carries bf16's rounding of V into delta = rowsum(O * dO) and through it
# into dQ and dK: up to 0.24 there instead of 0.05.  A forward that will not be differentiated always takes the fast form.
FP16_TRAINING_FORWARD = "exact"


def use_rotated_path(N, D, training, slabs=None, kv_slabs=None, causal=True, cus=256):
    """Whether the operator rotates the operands ahead of the attention kernels at this shape.  slabs, kv_slabs: batch times query and key/value heads;
    None leaves out the lengths that depend on them (an fp16 forward at D = 256 has only the single-launch kernel there).  cus: compute units."""
    if N * D < TRAIN_ROTATED_MIN_ND or D > _ROTATED_PATH_MAX_D:
        return N >= TWO_LAUNCH_MIN_N and D <= _ROTATED_PATH_MAX_D
    if training or N >= TWO_LAUNCH_MIN_N or N * D >= _FWD_ROTATED_MIN_ND:
        return True
    return slabs is not None and _forward_pays_rotation(N, D, slabs, slabs if kv_slabs is None else kv_slabs, causal, cus)


def _view_strides(t):
    """(batch, head, row) strides in elements if the kernels can read t where it lies -- last dimension contiguous, rows
    16-byte aligned and at least D apart, as the reference's forward reads q and k through their strides
    (fused_rope_attn.py:709-710) -- else None."""
    sb, sh, sn, sd = t.stride()
    d = t.shape[-1]
    if sd != 1 or sn < d or min(sb, sh) < 0 or sb % 8 or sh % 8 or sn % 8 or t.data_ptr() % 16 or t.shape[2] * sn * 2 >= 1 << 32:
        return None
    return (ctypes.c_int64 * 3)(sb, sh, sn)


def _readable(t):
    """t, or a copy where the kernels cannot read it where it lies, with its (batch, head, row) strides."""
    strides = None if t.is_contiguous() else _view_strides(t)
    if strides is not None:
        return t, strides
    _, h, n, d = t.shape
    return t.contiguous(), (ctypes.c_int64 * 3)(h * n * d, n * d, d)   # (an axis of length 1 may say otherwise)


def _route(q, k, causal, keep_rotated, two_launch=None):
    """(rotate K ahead?, keep P and V in fp16 there?) for a forward."""
    B, H, N, D = q.shape
    asked, fp16 = two_launch is not None, q.dtype == torch.float16
    if not asked:
        two_launch = use_rotated_path(N, D, True) if keep_rotated else use_rotated_path(
            N, D, False, None if fp16 and D > 128 else B * H, B * k.shape[1], causal, _compute_units(q.device.index))
    # fp16 with gradients, or so short that the fast form's kernel never served it: P and V stay fp16 (no key-norm maxima)
    return two_launch, (fp16 and two_launch and
                        (FP16_TRAINING_FORWARD != "fast" if keep_rotated else not asked and not use_rotated_path(N, D, False)))


def _scratch(nbytes, device):
    """Scratch in which launches leave the partial sums of blocks that they cut among workgroups (0 bytes: none are cut), or None.  Only
    speed needs it."""
    try:
        return torch.empty(nbytes, device=device, dtype=torch.uint8) if nbytes > 0 else None
    except torch.cuda.OutOfMemoryError:
        return None


def _fwd_parts(lib, q, causal):
    B, H, N, D = q.shape
    nbytes = lib.corope_rope_attn_fwd_parts_bytes(B, H, N, D, int(bool(causal))) if D <= 128 else 0
    return _scratch(nbytes, q.device), nbytes


def _native_forward(lib, q, k, v, causal, sm_scale, fc, fs, keep):
    """What _forward returns, and the v to keep, by the native host side; None where this is not a plain call (then _check_inputs and
    _forward do it)."""
    if q.dim() != 4 or k.dim() != 4 or not q.is_cuda or q.shape[3] not in _SUPPORTED_D or torch.cuda.current_device() != q.device.index:
        return None
    rotated, exact = _route(q, k, causal, keep)
    host, table = lib.host
    out = host.rope_forward(table, q, k, v, fc, fs, causal, float(sm_scale), rotated, exact, keep, q.device.index, _stream_ptr(q),
                            _fwd_parts(lib, q, causal)[0] if rotated else None)
    if type(out) is int:
        _lib.check(out, "corope_rope_attn_fwd_keep")
    return out and (out[0], out[1], fc, fs, out[2:4] if out[2] is not None else None, out[4])


def _forward(q, k, v, causal, sm_scale, freqs_cos, freqs_sin, two_launch=None, keep_rotated=False):
    """Runs the forward kernels; returns (o, M, fc, fs, rotated) with the tables in the form the kernels were given.
    ``rotated`` is (q_rot, k_rot) when ``keep_rotated`` was asked for and the two-launch path ran, else None.
    q, k, v may be strided views (a (B, N, H, D) tensor seen as (B, H, N, D), a slice of a fused projection): they are read
    where they lie when their layout allows it, else copied."""
    lib = _lib.load()
    fc, fs = _freq_table(freqs_cos), _freq_table(freqs_sin)
    if fc.stride(0) != fs.stride(0):
        fc, fs = fc.contiguous(), fs.contiguous()
    B, H, N, D = q.shape
    Hkv = k.shape[1]
    (q, q_st), (k, k_st), (v, v_st) = (_readable(t) for t in (q, k, v))
    two_launch, exact = _route(q, k, causal, keep_rotated, two_launch)
    empty = lambda shape, dtype=torch.float32: torch.empty(shape, device=q.device, dtype=dtype)
    ptr = lambda t: None if t is None else t.data_ptr()
    with _on_device(q):
        parts, nbytes = _fwd_parts(lib, q, causal) if two_launch else (None, 0)
        o, M = empty(q.shape, q.dtype), empty((B, H, N))
        q_rot = empty(q.shape, q.dtype) if two_launch and keep_rotated else None
        k_rot = empty(k.shape, q.dtype) if two_launch else None
        # with key-norm maxima: the pipelined kernel, for fp16 with bf16 probabilities against a V converted to bf16 on its way into LDS; without:
        # P and V in fp16, pipelined as well up to D = 128, in the single-launch kernel on the rotated copy at 256
        kmax = empty((B, Hkv, (N + 63) // 64)) if two_launch and not exact else None
        rc = lib.corope_rope_attn_fwd_keep(q.data_ptr(), q_st, k.data_ptr(), k_st, v.data_ptr(), v_st, fc.data_ptr(), fs.data_ptr(), fc.stride(0),
                                           o.data_ptr(), M.data_ptr(), ptr(q_rot), ptr(k_rot), ptr(kmax), B, H, Hkv, N, D, float(sm_scale),
                                           int(bool(causal)), int(q.dtype == torch.float16), ptr(parts), nbytes, None, _stream_ptr(q))
    _lib.check(rc, "corope_rope_attn_fwd_keep")
    return o, M, fc, fs, (None if q_rot is None else (q_rot, k_rot))


def _backward_rotated(lib, q_rot, k_rot, v, o, do, M, fc, fs, sm_scale, causal):
    """(dq, dk, dv, ...) of the operator from the rotated q and k its forward kept."""
    B, H, N, D = q_rot.shape
    Hkv = k_rot.shape[1]
    # (how many pieces there are depends on the device: at most 128 MiB with 256 compute units)
    with _on_device(q_rot):
        nbytes = lib.corope_rope_attn_bwd_rotated_parts_bytes(B, H, Hkv, N, D, int(causal))
        parts = _scratch(nbytes, q_rot.device)
        host, table = lib.host
        out = host.rope_backward(table, q_rot, k_rot, v, o, do, M, fc, fs, causal, sm_scale, q_rot.device.index, _stream_ptr(q_rot), parts)
        if type(out) is int:
            _lib.check(out, "corope_rope_attn_bwd_rotated")
        if out is not None:
            return *out, None, None, None, None, None
        do_st = None
        if not do.is_contiguous():
            do_st = _view_strides(do) if D <= 128 else None
            do = do if do_st is not None else do.contiguous()
        dq, dk, dv = torch.empty_like(q_rot), torch.empty_like(k_rot), torch.empty_like(k_rot)
        delta = torch.empty_like(M)
        rc = lib.corope_rope_attn_bwd_rotated(q_rot.data_ptr(), k_rot.data_ptr(), v.data_ptr(), None, o.data_ptr(), do.data_ptr(), do_st,
                                              M.data_ptr(), delta.data_ptr(), fc.data_ptr(), fs.data_ptr(), fc.stride(0), dq.data_ptr(),
                                              dk.data_ptr(), dv.data_ptr(), B, H, Hkv, N, D, sm_scale, int(causal),
                                              int(q_rot.dtype == torch.float16), parts.data_ptr() if parts is not None else None, nbytes,
                                              _stream_ptr(q_rot))
    _lib.check(rc, "corope_rope_attn_bwd_rotated")
    return dq, dk, dv, None, None, None, None, None


class _FusedRopeAttn(torch.autograd.Function):

    @staticmethod
    def forward(ctx, q, k, v, causal, sm_scale, freqs_cos, freqs_sin, warp_specialize=True):
        needs = ctx.needs_input_grad
        training = needs[0] or needs[1] or needs[2]
        # v is kept for the backward, and a view kept as it is would hold the fused projection it is cut from, and would be lost
        # if the caller overwrites that before the backward: a view is copied (by the launch that rotates K), q and k are kept
        # rotated, in tensors of their own
        # when a gradient will be asked for, the forward keeps its rotated q and k for the backward and the originals
        # are not saved (the reference saves q and k, fused_rope_attn.py:718, and re-rotates them in its backward)
        out = _native_forward(_lib.load(), q, k, v, causal, sm_scale, freqs_cos, freqs_sin, training)
        if out is None:
            _check_inputs(q, k, v, freqs_cos, freqs_sin)
            if training:
                v = v.contiguous()
            out = *_forward(q, k, v, causal, sm_scale, freqs_cos, freqs_sin, keep_rotated=training), v
        o, M, fc, fs, rotated, v = out
        # nothing to differentiate, nothing kept: saving q and k would copy strided views of a fused projection.  (Tables that
        # ask for a gradient get None, but the backward that says so runs and wants its tensors.)
        if not any(needs):
            return o
        ctx.rotated = rotated is not None
        if ctx.rotated:
            ctx.save_for_backward(rotated[0], rotated[1], v, o, M, fc, fs)
        else:
            ctx.save_for_backward(q.contiguous(), k.contiguous(), v.contiguous(), o, M, fc, fs)
        ctx.sm_scale = float(sm_scale)
        ctx.HEAD_DIM = q.shape[-1]
        ctx.causal = bool(causal)
        return o

    @staticmethod
    def backward(ctx, do):
        q, k, v, o, M, fc, fs = ctx.saved_tensors
        lib = _lib.load()
        if do.dtype != q.dtype:
            do = do.to(q.dtype)
        B, H, N, D = q.shape
        if ctx.rotated:   # q, k are the rotated copies the forward kept; dO is read where it lies if its layout allows it
            return _backward_rotated(lib, q, k, v, o, do, M, fc, fs, ctx.sm_scale, ctx.causal)
        # A forward of which only the tables ask for a gradient kept nothing rotated: the copies are made here.  (Without them, the kernels on unrotated
        # operands, whose entry points callers of the C ABI have: here only where TRAIN_ROTATED_MIN_ND and TWO_LAUNCH_MIN_N are raised.)
        do = do.contiguous()
        dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
        delta = torch.empty_like(M)
        with _on_device(q):
            if q.dtype == torch.float16:
                ws, nbytes = None, 0
                if use_rotated_path(N, D, training=True):   # rotate q and k once, then the kernels on the copies
                    nbytes = lib.corope_rope_attn_bwd_workspace_bytes(B, H, N, D)
                    ws = torch.empty(nbytes, device=q.device, dtype=torch.uint8)
                rc = lib.corope_rope_attn_bwd_f16(q.data_ptr(), k.data_ptr(), 0, v.data_ptr(), o.data_ptr(), do.data_ptr(),
                                                  M.data_ptr(), delta.data_ptr(), fc.data_ptr(), fs.data_ptr(), fc.stride(0),
                                                  dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), B, H, k.shape[1], N, D,
                                                  ctx.sm_scale, int(ctx.causal), ws.data_ptr() if ws is not None else None,
                                                  nbytes, _stream_ptr(q))
            elif k.shape[1] != H:         # grouped-query attention
                rc = lib.corope_rope_attn_bwd_gqa(q.data_ptr(), k.data_ptr(), 0, v.data_ptr(), o.data_ptr(),
                                                  do.data_ptr(), M.data_ptr(), delta.data_ptr(), fc.data_ptr(), fs.data_ptr(),
                                                  fc.stride(0), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), B, H,
                                                  k.shape[1], N, D, ctx.sm_scale, int(ctx.causal), _stream_ptr(q))
            elif use_rotated_path(N, D, training=True):   # rotate q and k once, then run the kernels on the rotated copies
                nbytes = lib.corope_rope_attn_bwd_workspace_bytes(B, H, N, D)
                ws = torch.empty(nbytes, device=q.device, dtype=torch.uint8)
                rc = lib.corope_rope_attn_bwd_ws(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), do.data_ptr(),
                                                 M.data_ptr(), delta.data_ptr(), fc.data_ptr(), fs.data_ptr(),
                                                 fc.stride(0), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), B, H, N, D,
                                                 ctx.sm_scale, int(ctx.causal), ws.data_ptr(), nbytes, _stream_ptr(q))
            else:
                rc = lib.corope_rope_attn_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), do.data_ptr(),
                                              M.data_ptr(), delta.data_ptr(), fc.data_ptr(), fs.data_ptr(), fc.stride(0),
                                              dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), B, H, N, D, ctx.sm_scale,
                                              int(ctx.causal), _stream_ptr(q))
        _lib.check(rc, "corope_rope_attn_bwd")
        return dq, dk, dv, None, None, None, None, None


def attention(q, k, v, causal, sm_scale, freqs_cos, freqs_sin, warp_specialize=True):
    """The reference's ``attention = _attention.apply`` (fused-rope/fused_rope_attn.py:780): positional arguments in its
    order.  Head dims 64 and 128 go to the kernels as they are; 16 and 32 are padded to 64 around the same kernels (zero
    columns, tables padded with the identity rotation), which changes no value of the result."""
    d = q.shape[-1]
    if d in _PADDED_D and q.dim() == 4 and k.shape[-1] == d and v.shape[-1] == d:
        h, pad = d // 2, (64 - d) // 2
        fc = torch.cat([freqs_cos[:, :h].float(), freqs_cos.new_ones((freqs_cos.shape[0], pad), dtype=torch.float32)], dim=1)
        fs = torch.cat([freqs_sin[:, :h].float(), freqs_sin.new_zeros((freqs_sin.shape[0], pad), dtype=torch.float32)], dim=1)
        o = _FusedRopeAttn.apply(spread_halves(q, 64), spread_halves(k, 64), spread_halves(v, 64), causal, sm_scale, fc, fs,
                                 warp_specialize)
        return gather_halves(o, d)
    return _FusedRopeAttn.apply(q, k, v, causal, sm_scale, freqs_cos, freqs_sin, warp_specialize)


def fused_rope_attn(q, k, v, freqs_cos, freqs_sin, causal=True, sm_scale=None):
    """Keyword-friendly form: ``sm_scale`` defaults to 1/sqrt(D)."""
    if sm_scale is None:
        sm_scale = q.shape[-1] ** -0.5
    return attention(q, k, v, causal, sm_scale, freqs_cos, freqs_sin)


def rope_attn_forward_with_lse(q, k, v, causal, sm_scale, freqs_cos, freqs_sin, two_launch=None):
    """Forward only, returning (O, M) where M is the saved base-2 log-sum-exp statistic (B, H, N) fp32.
    ``two_launch`` forces (True / False) or leaves to the length rule (None) the choice of forward path."""
    _check_inputs(q, k, v, freqs_cos, freqs_sin)
    o, M, _, _, _ = _forward(q, k, v, causal, sm_scale, freqs_cos, freqs_sin, two_launch)
    return o, M


def rope_rotate(x, freqs_cos, freqs_sin, with_tile_max=False, scale=1.0):
    """``scale`` times the half-layout rotation of x (B, H, N, D) bf16 on the device (fp32 arithmetic, one rounding to
    bf16).  Returns y, or (y, tile_max) with the largest row norm of y in every 64-row tile, (B, H, ceil(N/64)) fp32.
    The pre-rotated operands of the backward kernels are ``rope_rotate(k, ...)`` and
    ``rope_rotate(q, ..., scale=sm_scale * log2(e))``."""
    _check_inputs(x, x, x, freqs_cos, freqs_sin)
    if x.dtype != torch.bfloat16:
        raise ValueError("the rotation pass is built for bfloat16 only")
    lib = _lib.load()
    x = x.contiguous()
    fc, fs = _freq_table(freqs_cos), _freq_table(freqs_sin)
    if fc.stride(0) != fs.stride(0):
        fc, fs = fc.contiguous(), fs.contiguous()
    B, H, N, D = x.shape
    y = torch.empty_like(x)
    tm = torch.empty((B, H, (N + 63) // 64), device=x.device, dtype=torch.float32) if with_tile_max else None
    with _on_device(x):
        rc = lib.corope_rope_rotate(x.data_ptr(), fc.data_ptr(), fs.data_ptr(), fc.stride(0), y.data_ptr(),
                                    tm.data_ptr() if with_tile_max else None, B, H, N, D, float(scale), _stream_ptr(x))
    _lib.check(rc, "corope_rope_rotate")
    return (y, tm) if with_tile_max else y
