"""The reference's four operators (module `KVmix`, quant_cuda/csrc/pybind.cpp:6-15) on top of
the gfx950 C ABI.  Names, positional argument order, return types and error texts follow the
reference; the tensors are torch ROCm tensors, everything else is the HIP library.

    quantize_pack_last_dim_cuda(input, group_length, quant_bits) -> (code, scale, min)
    quantized_gemm(group_size, fA, qB, scales, zeros, bits) -> out
    process_key_quantization_cuda(input, prev_code, prev_scale, prev_min, group_length, quant_bits)
    process_value_quantization_cuda(input, prev_code, prev_scale, prev_min, group_length, quant_bits)

All four launch on torch's current stream of the input's device and do not synchronise.
"""
from __future__ import annotations

from typing import Tuple

import functools

import torch

from . import _lib

_DT = {torch.float16: _lib.F16, torch.float32: _lib.F32}


_native = None


def _host():
    """The native host side of the operators (csrc/host.cpp)."""
    global _native
    if _native is None:
        _native = _lib.load_host()
    return _native


def _need_gpu(*tensors: torch.Tensor) -> None:
    for t in tensors:
        if not t.is_cuda:
            raise RuntimeError("KVmix operators run on the GPU only: got a tensor on " + str(t.device))


def _stream(t: torch.Tensor) -> int:
    return torch.cuda.current_stream(t.device).cuda_stream


def _values_per_word(bits: int) -> int:
    return 11 if bits == 3 else 32 // bits


def _check_bits(bits: int) -> None:
    if bits not in (1, 2, 3, 4):
        raise RuntimeError("Supported quantization bits: 1, 2, 3, 4")


def _rows3(t: torch.Tensor) -> Tuple[torch.Tensor, int, int]:
    """View a 4-D tensor [B, H, R, S] as [B*H, R, S] without copying when its strides allow it;
    returns (tensor, outer_stride, inner_stride) in elements."""
    B, H, R, S = t.shape
    ok = (S <= 1 or t.stride(3) == 1) and (B <= 1 or t.stride(0) == H * t.stride(1))
    if ok and R > 1 and t.stride(2) < S:
        ok = False
    if ok and H > 1 and t.stride(1) < t.stride(2):
        ok = False
    if not ok:
        t = t.contiguous()
    return t, (t.stride(1) if B * H > 1 else max(R * t.stride(2), 1)), (t.stride(2) if R > 1 else max(S, 1))


def _quantize_into(x: torch.Tensor, group: int, bits: int, fmt: int, scale_mode: int,
                   code: torch.Tensor, scale: torch.Tensor, mn: torch.Tensor) -> None:
    """x [B,H,R,S]; code/scale/mn 4-D views (possibly slices of larger buffers) to fill."""
    L = _lib.load()
    B, H, R, S = x.shape
    x, xo, xi = _rows3(x)
    with torch.cuda.device(x.device):
        _lib.check(L.kvmix_quant_pack_last_dim(
            x.data_ptr(), _DT[x.dtype], B * H, R, S, xo, xi, group, bits, fmt, scale_mode,
            code.data_ptr(), code.stride(1), code.stride(2),
            scale.data_ptr(), mn.data_ptr(), scale.stride(1), scale.stride(2), _stream(x)))


def quantize_pack_last_dim_cuda(input: torch.Tensor, group_length: int, quant_bits: int):
    """Group-quantize the last dimension of a 4-D fp16/fp32 tensor and bit-pack the codes.

    Reference: quantize_pack_last_dim_cuda, quant_cuda/csrc/quantization_cuda.cu:631-721.
    Returns (code int32 [B,H,R,S/vpw], scale [B,H,R,S/g], min [B,H,R,S/g]); scale and min have the
    input's dtype.  3-bit uses the reference's 11-codes-per-word layout and needs group_length 11."""
    return _host().quantize_pack_last_dim(input, group_length, quant_bits)


def quantize_pack_dense3(input: torch.Tensor, group_length: int = 32):
    """Extension (no reference counterpart): 3-bit codes with qmax 7 for every value, stored as a
    little-endian bit stream (32 codes in three uint32), group a multiple of 32.  Same min / max /
    scale / rounding arithmetic as quantize_pack_last_dim_cuda.  Pair with
    quantized_gemm(..., bits=3, fmt=FMT_DENSE3).
    Returns (code int32 [B,H,R,3S/32], scale [B,H,R,S/g], min [B,H,R,S/g])."""
    return _host().quantize_pack_dense3(input, group_length)


FMT_REF = _lib.FMT_REF
FMT_DENSE3 = _lib.FMT_DENSE3


def quantize_kv_flush(k_chunk: torch.Tensor, k_group: int, k_bits: int, v_chunk: torch.Tensor, v_group: int,
                      v_bits: int, k_fmt: int = _lib.FMT_REF, v_fmt: int = _lib.FMT_REF):
    """Extension (no reference counterpart): both flushes of a decode step in ONE launch.

    k_chunk [B,H,n,D] fp16 are the oldest n tokens of the key tail, token-major as the tail is
    stored; the result is what quantize_pack_last_dim_cuda(k_chunk.transpose(2, 3).contiguous(),
    k_group, k_bits) returns (models/modeling_llama_KVmix.py:131-133), without the transpose copy.
    v_chunk [B,H,nv,D] fp16 is quantized along D as quantize_pack_last_dim_cuda(v_chunk, v_group,
    v_bits) does (:157-159).  Bit-identical to the two separate operators.
    Returns (k_code [B,H,D,n/vpw], k_scale, k_min [B,H,D,n/g], v_code [B,H,nv,D/vpw], v_scale, v_min)."""
    for t in (k_chunk, v_chunk):
        if t.dim() != 4:
            raise RuntimeError("input_tensor must be a 4D tensor")
        if t.dtype != torch.float16:
            raise RuntimeError(f"expected scalar type Half but found {t.dtype}")
    _check_bits(k_bits)
    _check_bits(v_bits)
    _need_gpu(k_chunk, v_chunk)
    L = _lib.load()
    B, H, n, D = k_chunk.shape
    Bv, Hv, nv, Dv = v_chunk.shape
    dev = k_chunk.device

    def words(steps, bits, fmt):
        return steps * 3 // 32 if (bits == 3 and fmt == _lib.FMT_DENSE3) else steps // _values_per_word(bits)

    kc = torch.empty((B, H, D, words(n, k_bits, k_fmt)), dtype=torch.int32, device=dev)
    ks = torch.empty((B, H, D, n // k_group if k_group > 0 else 0), dtype=torch.float16, device=dev)
    km = torch.empty_like(ks)
    vc = torch.empty((Bv, Hv, nv, words(Dv, v_bits, v_fmt)), dtype=torch.int32, device=dev)
    vs = torch.empty((Bv, Hv, nv, Dv // v_group if v_group > 0 else 0), dtype=torch.float16, device=dev)
    vm = torch.empty_like(vs)
    quantize_kv_flush_into(k_chunk, k_group, k_bits, (kc, ks, km), v_chunk, v_group, v_bits, (vc, vs, vm), k_fmt, v_fmt)
    return kc, ks, km, vc, vs, vm


def _flush_descriptors(k_chunk, k_group: int, k_bits: int, k_out, v_chunk, v_group: int, v_bits: int, v_out,
                       k_fmt: int = _lib.FMT_REF, v_fmt: int = _lib.FMT_REF):
    """The (KeyFlush, ValueFlush, tensors to keep alive) of one flush, or None when there is nothing to do.  Keys in
    groups the token-major key kernel does not take (other than 32, or 11 for the reference's 3 bits) are quantized
    here and now through the one-shot quantizer; the key descriptor then stays empty."""
    kf, vf = _lib.KeyFlush(), _lib.ValueFlush()
    kf.group, kf.bits, kf.fmt, kf.scale_mode = max(k_group, 1), k_bits, k_fmt, _lib.SCALE_RECIPROCAL
    vf.group, vf.bits, vf.fmt, vf.scale_mode = max(v_group, 1), v_bits, v_fmt, _lib.SCALE_RECIPROCAL
    ref = k_chunk if k_chunk is not None else v_chunk
    if ref is None:
        return None
    _need_gpu(ref)
    keep = [ref]

    def out_strides(code, scale, mn, B, H):
        for t in (code, scale, mn):
            if t.dim() != 4 or (t.shape[3] > 1 and t.stride(3) != 1) or (B > 1 and t.stride(0) != H * t.stride(1)):
                raise RuntimeError("output views must be 4-D, unit-stride along the last dimension, (B, H) collapsible")
        if (scale.stride(1), scale.stride(2)) != (mn.stride(1), mn.stride(2)):
            raise RuntimeError("scale and min outputs must share their strides")

    if k_chunk is not None and k_chunk.shape[2] > 0:
        B, H, n, D = k_chunk.shape
        ref3 = k_bits == 3 and k_fmt == _lib.FMT_REF
        if not ref3 and k_group != 32:
            # the token-major key kernel is built for group 32 (and the reference's 3-bit group 11)
            _quantize_into(k_chunk.transpose(2, 3).contiguous(), k_group, k_bits, k_fmt, _lib.SCALE_RECIPROCAL, *k_out)
        else:
            if k_chunk.stride(3) != 1 or (B > 1 and k_chunk.stride(0) != H * k_chunk.stride(1)):
                k_chunk = k_chunk.contiguous()
            kc, ks, km = k_out
            out_strides(kc, ks, km, B, H)
            kf.k, kf.outer, kf.n, kf.D = k_chunk.data_ptr(), B * H, n, D
            kf.k_outer_stride, kf.k_token_stride = k_chunk.stride(1), k_chunk.stride(2)
            kf.code, kf.code_outer_stride, kf.code_inner_stride = kc.data_ptr(), kc.stride(1), kc.stride(2)
            kf.scale, kf.zero = ks.data_ptr(), km.data_ptr()
            kf.sz_outer_stride, kf.sz_inner_stride = ks.stride(1), ks.stride(2)
            keep += [k_chunk, kc, ks, km]
    if v_chunk is not None and v_chunk.shape[2] > 0:
        Bv, Hv, nv, Dv = v_chunk.shape
        v_chunk, vo, vi = _rows3(v_chunk)
        vc, vs, vm = v_out
        out_strides(vc, vs, vm, Bv, Hv)
        vf.x, vf.outer, vf.inner, vf.steps = v_chunk.data_ptr(), Bv * Hv, nv, Dv
        vf.x_outer_stride, vf.x_inner_stride = vo, vi
        vf.code, vf.code_outer_stride, vf.code_inner_stride = vc.data_ptr(), vc.stride(1), vc.stride(2)
        vf.scale, vf.zero = vs.data_ptr(), vm.data_ptr()
        vf.sz_outer_stride, vf.sz_inner_stride = vs.stride(1), vs.stride(2)
        keep += [v_chunk, vc, vs, vm]
    return kf, vf, keep


def quantize_kv_flush_into(k_chunk, k_group: int, k_bits: int, k_out, v_chunk, v_group: int, v_bits: int, v_out,
                           k_fmt: int = _lib.FMT_REF, v_fmt: int = _lib.FMT_REF) -> None:
    """quantize_kv_flush writing into tensors the caller owns: k_out = (code [B,H,D,n/vpw],
    scale, min [B,H,D,n/g]) and v_out = (code [B,H,nv,D/vpw], scale, min [B,H,nv,D/g]) may be
    slices of larger pre-allocated cache buffers (unit stride along the last dimension, (B, H)
    collapsible).  Either half may be None (k_chunk and k_out, or v_chunk and v_out)."""
    import ctypes

    d = _flush_descriptors(k_chunk, k_group, k_bits, k_out, v_chunk, v_group, v_bits, v_out, k_fmt, v_fmt)
    if d is None:
        return
    kf, vf, keep = d
    with torch.cuda.device(keep[0].device):
        _lib.check(_lib.load().kvmix_quant_pack_kv_flush(ctypes.byref(kf), ctypes.byref(vf), _stream(keep[0])))


def quantize_kv_flush_batch(flushes) -> None:
    """The flushes of several caches at once (kvmix_quant_pack_kv_flush_batch: eight to a launch): `flushes` is a
    sequence of argument tuples of quantize_kv_flush_into, all on one device; the results are those of calling it
    on each tuple, bit for bit.  What a decode step flushes are the oldest tokens of the fp16 tails
    (models/modeling_llama_KVmix.py:122-127,152-156), so a caller can issue the flushes of all layers of a step
    together before its first layer runs."""
    ds = [d for d in (_flush_descriptors(*f) for f in flushes) if d is not None]
    if not ds:
        return
    dev = ds[0][2][0].device
    if any(d[2][0].device != dev for d in ds):
        raise RuntimeError("the flushes of one batch must be on one device")
    with torch.cuda.device(dev):
        _lib.check(_lib.flush_batch([d[0] for d in ds], [d[1] for d in ds], _stream(ds[0][2][0])))


def quantized_gemm(group_size: int, fA: torch.Tensor, qB: torch.Tensor, scales: torch.Tensor,
                   zeros: torch.Tensor, bits: int, fmt: int = _lib.FMT_REF) -> torch.Tensor:
    """out[b,h,m,:] = fA[b,h,m,:] @ dequant(qB[b,h',:,:]) with h' = h // (nh // nh_kv).

    Reference: quantized_gemm, quant_cuda/csrc/dequantization_gemv_cuda.cu:127-248.
    fA [B,nh,M,K] f16; qB [B,nh_kv,K,N/vpw] i32; scales, zeros [B,nh_kv,K,N/g] f16 -> [B,nh,M,N] f16.
    The packed operands are read in place (views of a larger cache buffer are fine); GQA inputs
    may be passed un-repeated.  `fmt` is an extension (dense 3-bit); the default is the reference's."""
    return _host().quantized_gemm(group_size, fA, qB, scales, zeros, bits, fmt)


def prefer_single_pass(batch: int, heads: int, kv_heads: int, head_dim: int, width: int, k_bits: int, k_fmt: int,
                       k_group: int, v_bits: int, v_fmt: int, v_group: int, k_tokens: int = None,
                       v_tokens: int = None, weights: bool = False) -> bool:
    """Policy for callers that do not need the probabilities (weights: that do): whether the single-pass step is both
    available for this layout and the faster of the two at this size.  The library holds the measured rule
    (kvmix_decode_attention_fused_plan: `recommended`); k_tokens / v_tokens are the quantized lengths, where the
    caller knows them (they decide whether a large step can use the matrix cores; without them a step is
    taken to have nothing quantized on both sides)."""
    if kv_heads <= 0 or heads % kv_heads != 0:
        return False
    if not single_pass_supported(head_dim, heads // kv_heads, k_bits, k_fmt, k_group, v_bits, v_fmt, v_group):
        return False
    if k_tokens is None or v_tokens is None or width < max(k_tokens, v_tokens):
        k_tokens = v_tokens = 0
    return _host().prefer_single_pass(batch, heads, kv_heads, head_dim, width, k_bits, k_fmt, k_group, v_bits, v_fmt, v_group,
                                      k_tokens, v_tokens, weights)


def _set_tail(st, prefix: str, tail: torch.Tensor, slot) -> None:
    """The fields of a tail window and the slot the new token goes to (an int, or a device int64 read by the kernel)."""
    setattr(st, prefix + "_tail", tail.data_ptr())
    setattr(st, prefix + "_tail_batch_stride", tail.stride(0))
    setattr(st, prefix + "_tail_head_stride", tail.stride(1))
    setattr(st, prefix + "_tail_token_stride", tail.stride(2))
    setattr(st, prefix + "_tail_slots", tail.shape[2])
    if torch.is_tensor(slot):
        if slot.dtype != torch.int64 or slot.numel() != 1 or not slot.is_cuda:
            raise RuntimeError("a device-side slot must be one int64 element on the GPU")
        setattr(st, prefix + "_slot_dev", slot.data_ptr())
    else:
        setattr(st, prefix + "_slot", int(slot))


def rope_append(qkv: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, heads: int, kv_heads: int,
                k_tail: torch.Tensor, v_tail: torch.Tensor, k_slot, v_slot) -> torch.Tensor:
    """Rotary embedding of the new token's query and key heads and the append of its key and value
    heads to the cache tails, in one launch (models/modeling_llama_KVmix.py:102-112 for one token).

    qkv [B, 1, (heads + 2 kv_heads) * D] or [B, heads + 2 kv_heads, D] fp16: query, key, value heads
    of the new token; cos, sin: D fp16 values for its position (any shape with D elements);
    k_tail, v_tail [B, kv_heads, slots, D] fp16 windows, written in place at slot k_slot / v_slot
    (ints, or one-element int64 device tensors read when the kernel runs).
    Returns the rotated queries [B, heads, 1, D].  Bit-identical to x * cos + rotate_half(x) * sin
    in fp16 tensor arithmetic."""
    import ctypes

    for t in (qkv, cos, sin, k_tail, v_tail):
        if t.dtype != torch.float16:
            raise RuntimeError(f"expected scalar type Half but found {t.dtype}")
    _need_gpu(qkv, cos, sin, k_tail, v_tail)
    B, D = qkv.shape[0], k_tail.shape[-1]
    total = heads + 2 * kv_heads
    if qkv.numel() != B * total * D or cos.numel() != D or sin.numel() != D:
        raise RuntimeError("rope_append: qkv must hold heads + 2 * kv_heads rows of D values per batch element, cos and sin D values")
    if k_tail.dim() != 4 or v_tail.dim() != 4 or k_tail.shape[:2] != (B, kv_heads) or v_tail.shape[:2] != (B, kv_heads) \
            or v_tail.shape[-1] != D or k_tail.stride(3) != 1 or v_tail.stride(3) != 1:
        raise RuntimeError("rope_append: tails must be [B, kv_heads, slots, D] with unit stride along D")
    qkv = qkv.reshape(B, total * D)
    if qkv.stride(1) != 1:
        qkv = qkv.contiguous()
    cos, sin = cos.reshape(D).contiguous(), sin.reshape(D).contiguous()
    q_out = torch.empty((B, heads, 1, D), dtype=torch.float16, device=qkv.device)
    st = _lib.RopeAppend()
    st.qkv, st.qkv_batch_stride, st.cos, st.sin = qkv.data_ptr(), qkv.stride(0) if B > 1 else total * D, cos.data_ptr(), sin.data_ptr()
    st.q_out, st.q_batch_stride = q_out.data_ptr(), heads * D
    for prefix, tail, slot in (("k", k_tail, k_slot), ("v", v_tail, v_slot)):
        _set_tail(st, prefix, tail, slot)
    st.batch, st.heads, st.kv_heads, st.D = B, heads, kv_heads, D
    with torch.cuda.device(qkv.device):
        _lib.check(_lib.load().kvmix_rope_append(ctypes.byref(st), _stream(qkv)))
    return q_out


@functools.lru_cache(maxsize=None)
def linear_rows_supported(m: int, k: int, rows: int, epilogue: int = _lib.LINEAR_PLAIN, norm: bool = False,
                          head_dim: int = 0, kv_rows: int = 0) -> bool:
    """Whether kvmix_linear_rows takes a projection of these sizes (dense fp16 rows; asks the library)."""
    import ctypes

    st = _lib.LinearRows()
    st.m, st.k, st.x_stride, st.w_stride, st.epilogue = m, k, k, k, epilogue
    st.rows[0], st.out_stride, st.residual_stride = rows, rows, rows
    st.norm_weight = 16 if norm else None
    if epilogue == _lib.LINEAR_SWIGLU:
        st.rows[1] = rows
    if epilogue == _lib.LINEAR_ROPE_APPEND:
        st.rows[1] = st.rows[2] = kv_rows
        st.head_dim = st.k_tail_token_stride = st.v_tail_token_stride = head_dim
        st.k_tail_slots = st.v_tail_slots = 1
    return bool(_lib.load().kvmix_linear_rows_supported(ctypes.byref(st)))


def linear_rows(x: torch.Tensor, w: torch.Tensor, norm_weight: torch.Tensor = None, eps: float = 0.0,
                residual: torch.Tensor = None, fp32: bool = False) -> torch.Tensor:
    """x @ w.T for a few rows of x (kvmix_linear_rows): x [..., k], w [n, k] fp16 -> [..., n].  norm_weight: x is
    RMS-normalised first; residual [..., n]: added to the fp16 product (without a norm); fp32: the fp16
    product as fp32 (without a residual)."""
    return _host().linear_rows(x, w, norm_weight, eps, residual, fp32)


def swiglu_rows(x: torch.Tensor, w, norm_weight: torch.Tensor = None, eps: float = 0.0) -> torch.Tensor:
    """silu(x @ gate.T) * (x @ up.T) for a few rows of x, fp16, in one launch (kvmix_linear_rows); w = the stacked
    [2 n, k] weight, gate over up, or the pair."""
    return _host().swiglu_rows(x, w if isinstance(w, (tuple, list)) else (w,), norm_weight, eps)


def qkv_rope_append(x: torch.Tensor, w, heads: int, kv_heads: int, cos: torch.Tensor, sin: torch.Tensor,
                    k_tail: torch.Tensor, v_tail: torch.Tensor, k_slot, v_slot, norm_weight: torch.Tensor = None,
                    eps: float = 0.0) -> torch.Tensor:
    """The query, key and value projections of one new token per sequence, the rotary embedding of queries and keys and
    the append to the tail windows, in one launch: rope_append(linear(x)) with the same roundings.

    x [B, (1,) k]; w = the stacked [(heads + 2 kv_heads) D, k] weight or the (query, key, value) weights; cos, sin: D
    values shared by the sequences, or [B, (1,) D]; tails and slots as in rope_append.
    Returns the rotated queries [B, heads, 1, D]."""
    slots = []
    for slot in (k_slot, v_slot):
        slots += (0, slot) if torch.is_tensor(slot) else (int(slot), None)
    return _host().qkv_rope_append(x, w if isinstance(w, (tuple, list)) else (w,), heads, kv_heads, cos, sin, k_tail, v_tail,
                                   *slots, norm_weight, eps)


def plain_call(*tensors) -> bool:
    """Whether a call on these tensors is an ordinary one, which a kernel without an autograd formula may serve: no
    gradient (backward or forward mode) is being recorded, nothing is traced, compiled, transformed, cast (autocast) or
    dispatched to a tensor subclass or mode."""
    if torch.is_grad_enabled() and any(t.requires_grad for t in tensors):
        return False
    if any(type(t) is not torch.Tensor and type(t) is not torch.nn.Parameter for t in tensors):
        return False
    return not (torch.jit.is_tracing() or torch.compiler.is_compiling() or torch._C._len_torch_dispatch_stack()
                or torch._C._len_torch_function_stack() or torch._C._functorch.peek_interpreter_stack() is not None
                or torch.autograd.forward_ad._current_level >= 0 or torch.is_autocast_enabled("cuda"))


def _aligned_heads(t: torch.Tensor) -> torch.Tensor:
    """[B, H, T, D] fp16 as 16-byte pieces can be read from it: unit stride along D, the others multiples of 8."""
    if t.stride(3) == 1 and t.data_ptr() % 16 == 0 and not any(t.stride(i) % 8 for i in range(3) if t.shape[i] > 1):
        return t
    return t.clone(memory_format=torch.contiguous_format)


def prefill_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, attention_mask: torch.Tensor = None):
    """softmax(q k^T / sqrt(D) + mask) v of a prompt (kvmix_prefill_attention): q [B, nh, Q, D], k, v [B, nkv, T, D] fp16,
    D 64 or 128, any strides; attention_mask None or [1|B, 1|nh, Q, T] fp32 or fp16, clamped at the lowest half, rows
    masked everywhere weighing all positions alike.  Returns [B, nh, Q, D] fp16 (stored token by token), or None
    where the kernel does not take the call."""
    import ctypes

    if any(t.dim() != 4 or t.dtype != torch.float16 or not t.is_cuda or t.device != q.device for t in (q, k, v)):
        return None
    B, nh, Q, D = q.shape
    nkv, T = k.shape[1], k.shape[2]
    if v.shape != k.shape or k.shape[0] != B or k.shape[3] != D or nkv == 0 or nh % nkv or min(B, nh, Q, T) == 0:
        return None
    st = _lib.PrefillAttn()
    if attention_mask is not None:
        m = attention_mask
        if m.dim() != 4 or m.dtype not in _DT or m.device != q.device or m.shape[0] not in (1, B) or m.shape[1] not in (1, nh) \
                or m.shape[2:] != (Q, T):
            return None
        if T > 1 and m.stride(3) != 1:
            m = m.contiguous()
        st.mask, st.mask_dtype, st.mask_batch, st.mask_heads = m.data_ptr(), _DT[m.dtype], m.shape[0], m.shape[1]
        st.mask_batch_stride, st.mask_head_stride, st.mask_row_stride = m.stride(0), m.stride(1), m.stride(2)
    q, k, v = _aligned_heads(q), _aligned_heads(k), _aligned_heads(v)
    out = torch.empty((B, Q, nh, D), dtype=torch.float16, device=q.device).transpose(1, 2)
    for name, t in (("q", q), ("k", k), ("v", v), ("out", out)):
        setattr(st, name, t.data_ptr())
        setattr(st, name + "_batch_stride", t.stride(0) if t.shape[0] > 1 else 0)
        setattr(st, name + "_head_stride", t.stride(1) if t.shape[1] > 1 else 0)
        setattr(st, name + "_token_stride", t.stride(2) if t.shape[2] > 1 else 0)
    st.batch, st.heads, st.kv_heads, st.q_len, st.kv_len, st.head_dim = B, nh, nkv, Q, T, D
    st.scale = D ** -0.5
    L = _lib.load()
    if not L.kvmix_prefill_attention_supported(ctypes.byref(st)):
        return None
    ws_bytes = L.kvmix_prefill_attention_workspace_bytes(ctypes.byref(st))
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=q.device) if ws_bytes else None
    with torch.cuda.device(q.device):
        _lib.check(L.kvmix_prefill_attention(ctypes.byref(st), ws.data_ptr() if ws is not None else None, ws_bytes, _stream(q)))
    return out


@functools.lru_cache(maxsize=None)
def single_pass_supported(head_dim: int, heads_per_kv: int, k_bits: int, k_fmt: int, k_group: int, v_bits: int,
                          v_fmt: int, v_group: int) -> bool:
    """Whether decode_attention(single_pass=True) takes a cache of this layout (asks the library)."""
    import ctypes

    st = _lib.DecodeAttn()
    st.D, st.heads_per_kv, st.heads, st.samples = head_dim, heads_per_kv, heads_per_kv, heads_per_kv
    st.k_bits, st.k_fmt, st.k_group, st.k_tokens = k_bits, k_fmt, k_group, (11 if k_group == 11 else 32) * 32
    st.v_bits, st.v_fmt, st.v_group, st.v_tokens = v_bits, v_fmt, v_group, 32
    return bool(_lib.load().kvmix_decode_attention_fused_supported(ctypes.byref(st)))


def decode_attention(q: torch.Tensor, k_packed, v_packed, k_tail: torch.Tensor, v_tail: torch.Tensor,
                     k_group: int, k_bits: int, v_group: int, v_bits: int, k_fmt: int = _lib.FMT_REF,
                     v_fmt: int = _lib.FMT_REF, attention_mask=None, k_tail_len=None, v_tail_len=None,
                     single_pass: bool = False, weights: bool = False):
    """One decode step of attention over the packed cache plus its fp16 tails, in four or five
    launches (no reference operator: it is what models/modeling_llama_KVmix.py:180-211 composes
    from quantized_gemm, matmul, cat and softmax).

    single_pass=True runs the step as one pass over the positions instead (two launches, logits and
    probabilities stay on chip); no probabilities are returned (probs is None; weights=True: they are, at
    the price of writing the logits) and the roundings after the softmax are not the reference's (see the header).  Layouts the single-pass kernels do
    not take raise RuntimeError; `single_pass_supported` tells beforehand.

    q [B,nh,1,D] fp16; k_packed = (code [B,Hkv,D,Tk/vpw], scale, min) or None; v_packed =
    (code [B,Hkv,Tv,D/vpw], scale, min) or None; k_tail, v_tail [B,Hkv,slots,D] fp16.
    *_tail_len: None (every slot holds a token), an int, or a device int64 tensor of one element
    read when the kernels run (for steps replayed from a captured graph).
    attention_mask: None or fp32 [B,1,1,width].
    Returns (out [B,nh,1,D] fp16, probs [B,nh,1,width] fp16), width = max(Tk + key slots, Tv + value slots)."""
    lengths = []
    for n in (k_tail_len, v_tail_len):
        lengths += (None, n) if torch.is_tensor(n) else (None if n is None else int(n), None)
    return _host().decode_attention(q, k_packed, v_packed, k_tail, v_tail, k_group, k_bits, v_group, v_bits, k_fmt, v_fmt,
                                    attention_mask, *lengths, single_pass, weights)


def copy_rows(pairs) -> None:
    """dst.copy_(src) for a sequence of (dst, src) pairs of equal 4-D shape and type on one device, which do not overlap,
    in one launch per sixteen (kvmix_copy_rows)."""
    _host().copy_rows(list(pairs))


def grow_tuple(past, key_states, value_states, nk: int, nv: int, k_bits: int, k_group: int, v_bits: int):
    """The first eight entries of the reference's cache tuple after one call's tokens (models/modeling_llama_KVmix.py:
    117-167), in new tensors: the tails grown by them, the oldest nk key and nv value tokens of the OLD tails quantized to
    behind the packed part, in one launch (kvmix_grow; more for the values of a long prompt).  Keys in
    groups of 32 (3 bits: 11), values in groups of 32.  None where that does not take the call."""
    kc, k_tail, ks, km, vc, v_tail, vs, vm, _ = past
    return _host().grow_tuple(kc, k_tail, ks, km, vc, v_tail, vs, vm, key_states, value_states, nk, nv, k_bits, k_group, v_bits)


def process_key_quantization_cuda(input: torch.Tensor, previous_code: torch.Tensor,
                                  previous_scale: torch.Tensor, previous_min: torch.Tensor,
                                  group_length: int, quant_bits: int):
    """Append form for keys: input [B,H,D,n] (groups along n) is quantized and returned
    concatenated after previous_* along the last dimension.

    Reference: process_key_quantization_cuda, quant_cuda/csrc/quantization_cuda.cu:298-411.
    The returned scale is (max-min)/qmax rounded to the input dtype (the reference's append
    kernels divide in-kernel, :49-51,:149-151)."""
    return _host().append_keys(input, previous_code, previous_scale, previous_min, group_length, quant_bits)


def process_value_quantization_cuda(input: torch.Tensor, previous_code: torch.Tensor,
                                    previous_scale: torch.Tensor, previous_min: torch.Tensor,
                                    group_length: int, quant_bits: int):
    """Append form for values: input [B,H,n,D] (groups along D) is quantized and returned
    concatenated after previous_* along the token dimension.

    Reference: process_value_quantization_cuda, quant_cuda/csrc/quantization_cuda.cu:413-537.
    3-bit follows the reference's placeholder branch literally (plain 3*j shifts, so the
    eleventh code of a word keeps only its low two bits)."""
    return _host().append_values(input, previous_code, previous_scale, previous_min, group_length, quant_bits)
