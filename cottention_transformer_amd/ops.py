"""Host-side operators over torch tensors: thin wrappers that validate, allocate outputs and
workspace with torch, and enqueue the HIP kernels on torch's current stream through the C ABI.

Tensor contract is the reference's: (B, H, N, D) for q/k/v/o (Cuda_Kernel/combined_kernel_general.cu
:360-369), state (B, H, Dk, Dv) for decode.  Nothing here computes on the CPU.
"""
import ctypes

import torch

from . import _loader

_DTYPES = {torch.float32: _loader.F32, torch.float64: _loader.F64, torch.float16: _loader.F16,
           torch.bfloat16: _loader.BF16}


def _check(rc, what):
    if rc == _loader.OK:
        return
    msg = _loader.last_error() or f"{what} failed with status {rc}"
    raise RuntimeError(msg)


def _dtype_code(t):
    try:
        return _DTYPES[t.dtype]
    except KeyError:
        raise ValueError("Only float32, float64, float16, and bfloat16 are supported") from None


def _require_gpu(**tensors):
    dev = None
    for name, t in tensors.items():
        if not t.is_cuda:
            raise RuntimeError(f"{name} must be a CUDA tensor")  # wording of combined_kernel_general.cu:355-357
        if dev is None:
            dev = t.device
        elif t.device != dev:
            devs = sorted({str(x.device) for x in tensors.values()})
            raise RuntimeError(f"all tensors must be on the same device, got {devs}")


def _shapes(q, k, v):
    if q.dim() != 4 or k.dim() != 4 or v.dim() != 4:
        raise RuntimeError("Q, K and V must have shape (N, H, S, D)")
    if q.size(3) != k.size(3):
        raise RuntimeError("Q and K must have the same dimension")  # combined_kernel_general.cu:365
    if q.shape[:3] != k.shape[:3] or q.shape[:3] != v.shape[:3]:
        raise RuntimeError(f"Q, K and V must agree in (N, H, S): {tuple(q.shape)} {tuple(k.shape)} {tuple(v.shape)}")
    b, h, n, dk = q.shape
    return b, h, n, dk, v.size(3)


def _workspace(nbytes, device):
    if nbytes == 0:
        return None, 0
    ws = torch.empty(nbytes, dtype=torch.uint8, device=device)
    return ws, ws.data_ptr()


# The host side of a call costs about as much as the kernels of a small problem run, so the fixed parts are kept
# short: workspace sizes are remembered per shape, the device is only switched when it is not the current one, and
# the stream handle comes from torch's raw accessor.
_CACHE_LIMIT = 4096  # shapes remembered per cache; a caller that sweeps sequence lengths starts over, it does not grow


def _remember(cache, key, value):
    if len(cache) >= _CACHE_LIMIT:
        cache.clear()
    cache[key] = value
    return value


_ws_bytes_cache = {}


def _ws_bytes(query, *key):
    k = (query, key)
    n = _ws_bytes_cache.get(k)
    if n is None:
        n = _remember(_ws_bytes_cache, k, getattr(_loader.lib(), query)(*key))
    return n


class _NoSwitch:
    def __enter__(self):
        return None

    def __exit__(self, *exc):
        return False


_NO_SWITCH = _NoSwitch()


def _on(device):
    """Context that makes `device` current for the launch (a no-op when it already is)."""
    return _NO_SWITCH if torch.cuda.current_device() == device.index else torch.cuda.device(device)


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _stream(device=None):
    if _raw_stream is not None and device is not None:
        return _raw_stream(device.index)
    return torch.cuda.current_stream(device).cuda_stream


def _overlaps(a, b):
    """Whether the storage ranges spanned by two tensors intersect."""
    if a.numel() == 0 or b.numel() == 0 or a.untyped_storage().data_ptr() != b.untyped_storage().data_ptr():
        return False
    span = lambda t: (t.data_ptr(), t.data_ptr() + (sum((s - 1) * st for s, st in zip(t.shape, t.stride())) + 1) * t.element_size())
    (a0, a1), (b0, b1) = span(a), span(b)
    return a0 < b1 and b0 < a1


def merged_heads_supported(dtype, n, h, dk, dv):
    """Whether the causal ops can write o / read grad_out as (B,N,H,Dv) (see causal_dot_product)."""
    ok = lambda d: 32 <= d <= 128 and d % 16 == 0
    return dtype in (torch.bfloat16, torch.float16) and ok(dk) and ok(dv) and n * h * max(dk, dv) <= 1 << 30


def causal_dot_product(q, k, v, reversed=False, merged_heads=False, into_v=False):
    """o[s,j] = sum_i q[s,i] sum_{s'<=s (>=s if reversed)} k[s',i] v[s',j]; all of one dtype.

    merged_heads: return o as (B,N,H,Dv), the rows of the (B,N,H*Dv) tensor an output projection reads, instead
    of (B,H,N,Dv): the head merge of GPT_Trainer/GPTCosAttention.py:500 without its copy (bf16 / fp16 only, see
    merged_heads_supported).
    into_v: the result overwrites v and v is returned (inplace=True of Cuda_Kernel/combined_kernel_general.cu
    :403-404).  Where the library allows it (cott_causal_fwd_may_alias_v: the MFMA kernels) the kernels write
    straight into v's memory; otherwise the result is computed beside it and copied.  v must be contiguous."""
    if not merged_heads and not into_v:
        o = _loader.native().causal(q, k, v, reversed)
        if o is not None:
            return o
    _require_gpu(Q=q, K=k, V=v)
    b, h, n, dk, dv = _shapes(q, k, v)
    if not (q.dtype == k.dtype == v.dtype):
        raise RuntimeError("Q, K and V must have the same dtype")
    code = _dtype_code(q)
    if into_v:
        if merged_heads or not v.is_contiguous():
            raise RuntimeError("into_v needs a contiguous (B,H,N,Dv) v")
        if _overlaps(q, v) or _overlaps(k, v):
            raise RuntimeError("into_v: Q and K must not share memory with V")
    q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
    L = _loader.lib()
    if into_v and not L.cott_causal_fwd_may_alias_v(b, h, n, dk, dv, code):
        v.copy_(causal_dot_product(q, k, v, reversed))
        return v
    if merged_heads:
        if reversed:
            raise RuntimeError("merged_heads is only available for the forward direction")
        o = torch.empty((b, n, h, dv), dtype=q.dtype, device=q.device)
        with _on(q.device):
            ws, ws_ptr = _workspace(_ws_bytes("cott_causal_workspace_bytes", b, h, n, dk, dv, code), q.device)
            rc = L.cott_causal_fwd_bnhd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), b, h, n, dk, dv, code,
                                        ws_ptr, ws.numel() if ws is not None else 0, _stream(q.device))
        _check(rc, "cott_causal_fwd_bnhd")
        return o
    o = v if into_v else torch.empty((b, h, n, dv), dtype=q.dtype, device=q.device)
    with _on(q.device):
        ws, ws_ptr = _workspace(_ws_bytes("cott_causal_workspace_bytes", b, h, n, dk, dv, code), q.device)
        rc = L.cott_causal_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), b, h, n, dk, dv, code,
                               int(bool(reversed)), ws_ptr, ws.numel() if ws is not None else 0, _stream(q.device))
    _check(rc, "cott_causal_fwd")
    return o


_f32in_cache = {}


def causal_dot_product_as(q, k, v, dtype):
    """causal_dot_product(q.to(dtype), k.to(dtype), v.to(dtype)): the rule of an autocast forward pass
    (Cuda_Kernel/combined_kernel_general.cu:377-389).  fp32 tensors computed in bf16 are rounded inside the kernel where that
    is built (cott_causal_fwd_f32in_supported), bit for bit as the conversions round them."""
    if dtype is torch.bfloat16 and q.dtype == k.dtype == v.dtype == torch.float32 and q.is_cuda:
        o = _loader.native().causal_f32in(q, k, v)
        if o is not None:
            return o
        _require_gpu(Q=q, K=k, V=v)
        b, h, n, dk, dv = shape = _shapes(q, k, v)
        ok = _f32in_cache.get(shape)
        if ok is None:
            ok = _remember(_f32in_cache, shape, bool(_loader.lib().cott_causal_fwd_f32in_supported(*shape)))
        if ok:
            q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
            if not (q.data_ptr() | k.data_ptr() | v.data_ptr()) & 15:
                o = torch.empty((b, h, n, dv), dtype=dtype, device=q.device)
                with _on(q.device):
                    rc = _loader.lib().cott_causal_fwd_f32in(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), b, h, n,
                                                             dk, dv, _stream(q.device))
                _check(rc, "cott_causal_fwd_f32in")
                return o
    return causal_dot_product(q.to(dtype), k.to(dtype), v.to(dtype))


_saved_plan_cache = {}


def saved_states_plan(dtype, b, h, n, dk, dv):
    """(chunks_per_cut, ncuts, floats per slot, backward workspace bytes) of the states the forward pass can leave for the backward
    pass of this shape, or None when that backward pass takes none (it only does on sequences long enough, for the
    number of heads, to be cut into groups; bf16 / fp16).  cott_causal_saved_plan, remembered per shape."""
    if dtype not in (torch.bfloat16, torch.float16):
        return None
    key = (dtype, b, h, n, dk, dv)
    plan = _saved_plan_cache.get(key, False)
    if plan is False:
        cpc, cuts, slot, ws = ctypes.c_int(0), ctypes.c_int(0), ctypes.c_int(0), ctypes.c_size_t(0)
        rc = _loader.lib().cott_causal_saved_plan(b, h, n, dk, dv, _DTYPES[dtype], ctypes.byref(cpc),
                                                  ctypes.byref(cuts), ctypes.byref(slot), ctypes.byref(ws))
        _check(rc, "cott_causal_saved_plan")
        plan = _remember(_saved_plan_cache, key, (cpc.value, cuts.value, slot.value, ws.value) if cuts.value > 0 else None)
    return plan


def causal_dot_product_saving(q, k, v, merged_heads=False):
    """(o, saved): causal_dot_product(q, k, v) that also leaves, where saved_states_plan() has cuts for the shape,
    the (B,H,ncuts,slot) fp32 states (in the kernels' tile layout, see include/cottention.h) that causal_backward(..., saved=saved) starts dQ from instead of passing over
    k and v once more (what CustomAttention.forward keeps for backward, Cuda_Kernel/Custom_Kernel.py:16, plus this
    one small tensor).  saved is None where the plan has no cuts.  merged_heads: o as (B,N,H,Dv), see causal_dot_product."""
    if not merged_heads:
        pair = _loader.native().causal_saving(q, k, v)
        if pair is not None:
            return pair
    _require_gpu(Q=q, K=k, V=v)
    b, h, n, dk, dv = _shapes(q, k, v)
    if not (q.dtype == k.dtype == v.dtype):
        raise RuntimeError("Q, K and V must have the same dtype")
    plan = saved_states_plan(q.dtype, b, h, n, dk, dv)
    if plan is None:
        return causal_dot_product(q, k, v, merged_heads=merged_heads), None
    cpc, cuts, slot, _ = plan
    code = _dtype_code(q)
    q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
    o = torch.empty((b, n, h, dv) if merged_heads else (b, h, n, dv), dtype=q.dtype, device=q.device)
    saved = torch.empty((b, h, cuts, slot), dtype=torch.float32, device=q.device)
    L = _loader.lib()
    fn = L.cott_causal_fwd_save_bnhd if merged_heads else L.cott_causal_fwd_save
    with _on(q.device):
        ws, ws_ptr = _workspace(_ws_bytes("cott_causal_workspace_bytes", b, h, n, dk, dv, code), q.device)
        rc = fn(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), saved.data_ptr(), cpc, cuts,
                b, h, n, dk, dv, code, ws_ptr, ws.numel() if ws is not None else 0, _stream(q.device))
    _check(rc, "cott_causal_fwd_save")
    return o, saved


_prep_supported_cache = {}


def fused_preparation_supported(dtype, b, h, n, dk, dv, rotary_dim=0):
    """Whether causal_dot_product_prepared has a kernel for the shape: bf16 / fp16, head dims 32..128 in steps of 16
    (128-wide q / k rows with value tiles of at least 64 columns), a rotary width that is a multiple of 8
    (cott_causal_fwd_prep_supported)."""
    if dtype not in (torch.bfloat16, torch.float16):
        return False
    key = (dtype, b, h, n, dk, dv, rotary_dim)
    ok = _prep_supported_cache.get(key)
    if ok is None:
        ok = _remember(_prep_supported_cache, key, bool(
            _loader.lib().cott_causal_fwd_prep_supported(b, h, n, dk, dv, _DTYPES[dtype], rotary_dim)))
    return ok


def fused_preparation_preferred(dtype, b, h, n, dk, dv, rotary_dim=0):
    """Whether the one launch of causal_dot_product_prepared is also the better form for the shape (all but those planned
    as column halves in sequence groups, and few heads past a short length: cott_causal_fwd_prep_preferred); the modules
    take prepare_inputs + causal_dot_product elsewhere."""
    if dtype not in (torch.bfloat16, torch.float16):
        return False
    key = ("preferred", dtype, b, h, n, dk, dv, rotary_dim)
    ok = _prep_supported_cache.get(key)
    if ok is None:
        ok = _remember(_prep_supported_cache, key, bool(
            _loader.lib().cott_causal_fwd_prep_preferred(b, h, n, dk, dv, _DTYPES[dtype], rotary_dim)))
    return ok


def causal_dot_product_prepared(q, k, v, keep=None, cnt=None, sig=None, rotary=None, bnhd=False, merged_heads=False,
                                want_prepared=True, save_states=False):
    """Causal forward on the RAW projections q, k, v: rotation, normalisation, value scaling and masking
    (prepare_inputs) happen inside the attention kernel (GPT_Trainer/GPTCosAttention.py:229-248, 462-476 in front
    of :282 as one launch).  rotary = (table (P,R) fp32, positions): positions is either an int, the table row of
    position s then being that int + s, or the (B,N) integer position_ids tensor of the block (:458), any values
    (rows outside the table are clamped to it on the device; nothing is read back).  bnhd: q, k, v are (B,N,H,D);
    merged_heads: o is returned as (B,N,H,Dv).
    Returns (o, (q_hat, k_hat, v_hat)) with the prepared tensors (B,H,N,D) that the backward pass needs, or
    (o, None) when want_prepared is false.  Raises where fused_preparation_supported() is false.
    save_states: returns (o, prepared, saved) with the states causal_backward(q_hat, k_hat, v_hat, ..., saved=saved)
    takes (None where saved_states_plan() has none for the shape)."""
    _require_gpu(Q=q, K=k, V=v)
    b, h, n, dk, dv = _prep_shapes(q, k, v, bnhd)
    if not (q.dtype == k.dtype == v.dtype):
        raise RuntimeError("Q, K and V must have the same dtype")
    code = _dtype_code(q)
    keep, cnt, sig = _prep_side_inputs(b, h, n, keep, cnt, sig, q.device)
    table, pos0, rdim, rows, pos_ids = None, 0, 0, 0, None
    if rotary is not None:
        table, pos0 = rotary
        if table.dim() != 2 or table.size(1) % 8 != 0 or table.size(1) > dk:
            raise RuntimeError("rotary table must be (positions, rotary_dim), rotary_dim a multiple of 8 and <= Dk")
        table = table.to(device=q.device, dtype=torch.float32).contiguous()
        rows, rdim = table.shape
        if torch.is_tensor(pos0):
            if pos0.dim() == 1:
                pos0 = pos0[None, :]
            if pos0.shape[-1] != n or pos0.shape[0] not in (1, b) or pos0.dim() != 2:
                raise RuntimeError(f"position ids must be (B,N) = {(b, n)}, got {tuple(pos0.shape)}")
            pos_ids = pos0.to(device=q.device, dtype=torch.int64).expand(b, n).contiguous()
            pos0 = 0
    q, k, v, layout = _input_layout(q, k, v, bnhd, b, h, n, dk, dv)
    o = torch.empty((b, n, h, dv) if merged_heads else (b, h, n, dv), dtype=q.dtype, device=q.device)
    prepared = None
    if want_prepared:
        prepared = (torch.empty((b, h, n, dk), dtype=q.dtype, device=q.device),
                    torch.empty((b, h, n, dk), dtype=q.dtype, device=q.device),
                    torch.empty((b, h, n, dv), dtype=q.dtype, device=q.device))
    L = _loader.lib()
    plan = saved_states_plan(q.dtype, b, h, n, dk, dv) if save_states else None
    saved = None
    with _on(q.device):
        head = (q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
                *((t.data_ptr() for t in prepared) if prepared else (None, None, None)),
                _ptr(keep), _ptr(cnt), _ptr(sig), _ptr(table), _ptr(pos_ids), int(pos0), rdim, rows, layout,
                int(bool(merged_heads)))
        ws, ws_ptr = _workspace(_ws_bytes("cott_causal_workspace_bytes", b, h, n, dk, dv, code), q.device)
        tail = (b, h, n, dk, dv, code, ws_ptr, ws.numel() if ws is not None else 0, _stream(q.device))
        if plan is not None:
            cpc, cuts, slot, _ = plan
            saved = torch.empty((b, h, cuts, slot), dtype=torch.float32, device=q.device)
        if layout > 1:
            rc = L.cott_causal_fwd_prep_strided(*head, _ptr(saved), *(plan[:2] if plan is not None else (0, 0)), *tail)
        elif plan is not None:
            rc = L.cott_causal_fwd_prep_save(*head, saved.data_ptr(), cpc, cuts, *tail)
        else:
            rc = L.cott_causal_fwd_prep(*head, *tail)
    _check(rc, "cott_causal_fwd_prep")
    return (o, prepared, saved) if save_states else (o, prepared)


def noncausal_fused_preparation_supported(dtype, b, h, n, dk, dv):
    """Whether noncausal_dot_product_prepared has a kernel for the shape: bf16 / fp16, head dims 32..128 in steps of
    16, enough heads, or positions few enough, that a head is handled by one workgroup
    (cott_noncausal_fwd_prep_supported)."""
    if dtype not in (torch.bfloat16, torch.float16):
        return False
    key = ("nc", dtype, b, h, n, dk, dv)
    ok = _prep_supported_cache.get(key)
    if ok is None:
        ok = _remember(_prep_supported_cache, key, bool(
            _loader.lib().cott_noncausal_fwd_prep_supported(b, h, n, dk, dv, _DTYPES[dtype])))
    return ok


def noncausal_fused_preparation_preferred(dtype, b, h, n, dk, dv):
    """Whether noncausal_dot_product_prepared is also the better form for the shape (cott_noncausal_fwd_prep_preferred); the
    modules take prepare_inputs + noncausal_dot_product elsewhere."""
    if dtype not in (torch.bfloat16, torch.float16):
        return False
    key = ("nc preferred", dtype, b, h, n, dk, dv)
    ok = _prep_supported_cache.get(key)
    if ok is None:
        ok = _remember(_prep_supported_cache, key, bool(
            _loader.lib().cott_noncausal_fwd_prep_preferred(b, h, n, dk, dv, _DTYPES[dtype])))
    return ok


def noncausal_dot_product_prepared(q, k, v, keep=None, cnt=None, sig=None, bnhd=False, merged_heads=False):
    """Non-causal Q (K^T V) on the RAW projections: normalisation, value scaling and masking (prepare_inputs without a
    rotation) happen inside the attention kernel (BERT_Trainer/BertCosAttention.py:162-178 in front of :249 as one
    launch).  bnhd: q, k, v are (B,N,H,D); merged_heads: o is returned as (B,N,H,Dv).  Returns
    (o, (q_hat, k_hat, v_hat)) with the prepared tensors (B,H,N,D) that the backward pass needs.  Raises where
    noncausal_fused_preparation_supported() is false."""
    _require_gpu(Q=q, K=k, V=v)
    b, h, n, dk, dv = _prep_shapes(q, k, v, bnhd)
    if not (q.dtype == k.dtype == v.dtype):
        raise RuntimeError("Q, K and V must have the same dtype")
    code = _dtype_code(q)
    keep, cnt, sig = _prep_side_inputs(b, h, n, keep, cnt, sig, q.device)
    q, k, v, layout = _input_layout(q, k, v, bnhd, b, h, n, dk, dv)
    o = torch.empty((b, n, h, dv) if merged_heads else (b, h, n, dv), dtype=q.dtype, device=q.device)
    prepared = (torch.empty((b, h, n, dk), dtype=q.dtype, device=q.device),
                torch.empty((b, h, n, dk), dtype=q.dtype, device=q.device),
                torch.empty((b, h, n, dv), dtype=q.dtype, device=q.device))
    with _on(q.device):
        L = _loader.lib()
        rc = (L.cott_noncausal_fwd_prep_strided if layout > 1 else L.cott_noncausal_fwd_prep)(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), *(t.data_ptr() for t in prepared), _ptr(keep), _ptr(cnt), _ptr(sig),
            layout, int(bool(merged_heads)), b, h, n, dk, dv, code, _stream(q.device))
    _check(rc, "cott_noncausal_fwd_prep")
    return o, prepared


def causal_prefill(q, k, v, state=None, return_state=True):
    """Causal forward over a whole prompt (or one piece of a sequence) with the recurrence state handed over:
    returns (o, state_out) with o[s] = q[s] (state + sum_{s'<=s} k[s'] v[s']^T) and
    state_out = state + sum_{s'} k[s'] v[s']^T, the tensor `decode_step` continues from.  Replaces the
    per-token loop over the prompt of GPT_Trainer/GPTCosAttention.py:253-272.
    state: None (zero) or (B,H,Dk,Dv) fp32 (fp64 for fp64 inputs); it is not modified."""
    _require_gpu(Q=q, K=k, V=v)
    b, h, n, dk, dv = _shapes(q, k, v)
    if not (q.dtype == k.dtype == v.dtype):
        raise RuntimeError("Q, K and V must have the same dtype")
    code = _dtype_code(q)
    sdt = torch.float64 if q.dtype == torch.float64 else torch.float32
    if state is not None:
        _require_gpu(state=state)
        if state.shape != (b, h, dk, dv) or state.dtype != sdt or not state.is_contiguous():
            raise RuntimeError(f"causal_prefill: state must be a contiguous {sdt} tensor of shape {(b, h, dk, dv)}")
    q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
    o = torch.empty((b, h, n, dv), dtype=q.dtype, device=q.device)
    s_out = torch.empty((b, h, dk, dv), dtype=sdt, device=q.device) if return_state else None
    L = _loader.lib()
    with _on(q.device):
        ws, ws_ptr = _workspace(_ws_bytes("cott_causal_workspace_bytes", b, h, n, dk, dv, code), q.device)
        rc = L.cott_causal_fwd_state(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(),
                                     state.data_ptr() if state is not None else None,
                                     s_out.data_ptr() if s_out is not None else None, b, h, n, dk, dv, code, ws_ptr,
                                     ws.numel() if ws is not None else 0, _stream(q.device))
    _check(rc, "cott_causal_fwd_state")
    return o, s_out


def causal_backward(q, k, v, grad_out, merged_heads=False, saved=None):
    """(dQ, dK, dV) of causal_dot_product(q, k, v) for upstream gradient grad_out ((B,N,H,Dv) with merged_heads).
    saved: the states causal_dot_product_saving() (or causal_dot_product_prepared(save_states=True)) returned for
    the same q, k, v."""
    if not merged_heads and grad_out.dtype == q.dtype:
        grads = _loader.native().causal_backward(q, k, v, grad_out, saved)
        if grads is not None:
            return grads
    _require_gpu(Q=q, K=k, V=v, prev_grad=grad_out)
    b, h, n, dk, dv = _shapes(q, k, v)
    want = (b, n, h, dv) if merged_heads else tuple(v.shape)
    if tuple(grad_out.shape) != want:
        raise RuntimeError(f"prev_grad must have shape {want}, got {tuple(grad_out.shape)}")
    if not (q.dtype == k.dtype == v.dtype == grad_out.dtype):
        raise RuntimeError("Q, K, V and prev_grad must have the same dtype")
    code = _dtype_code(q)
    q, k, v, g = q.contiguous(), k.contiguous(), v.contiguous(), grad_out.contiguous()
    dq, dk_, dv_ = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    L = _loader.lib()
    if saved is not None:
        plan = saved_states_plan(q.dtype, b, h, n, dk, dv)
        if plan is None:
            raise RuntimeError("causal_backward: this call takes no saved states")
        cpc, cuts, slot, ws_bytes = plan
        _require_gpu(saved=saved)
        if tuple(saved.shape) != (b, h, cuts, slot) or saved.dtype != torch.float32 or not saved.is_contiguous():
            raise RuntimeError(f"causal_backward: saved must be a contiguous fp32 tensor of shape {(b, h, cuts, slot)}")
        with _on(q.device):
            ws, ws_ptr = _workspace(ws_bytes, q.device)
            fn = L.cott_causal_bwd_saved_bnhd if merged_heads else L.cott_causal_bwd_saved
            rc = fn(q.data_ptr(), k.data_ptr(), v.data_ptr(), g.data_ptr(), dq.data_ptr(),
                    dk_.data_ptr(), dv_.data_ptr(), saved.data_ptr(), cpc, cuts, b, h, n, dk, dv, code,
                    ws_ptr, ws.numel() if ws is not None else 0, _stream(q.device))
        _check(rc, "cott_causal_bwd_saved")
        return dq, dk_, dv_
    with _on(q.device):
        ws, ws_ptr = _workspace(_ws_bytes("cott_causal_bwd_workspace_bytes", b, h, n, dk, dv, code), q.device)
        fn = L.cott_causal_bwd_bnhd if merged_heads else L.cott_causal_bwd
        rc = fn(q.data_ptr(), k.data_ptr(), v.data_ptr(), g.data_ptr(), dq.data_ptr(), dk_.data_ptr(), dv_.data_ptr(), b, h,
                n, dk, dv, code, ws_ptr, ws.numel() if ws is not None else 0, _stream(q.device))
    _check(rc, "cott_causal_bwd_bnhd" if merged_heads else "cott_causal_bwd")
    return dq, dk_, dv_


_g16_cache = {}


def causal_backward_from(q, k, v, grad_out):
    """causal_backward(q, k, v, grad_out.to(q.dtype)): the backward of an autocast step saves fp32 tensors and is handed the
    gradient of a bf16 output (Cuda_Kernel/Custom_Kernel.py:38).  Where that is built (cott_causal_bwd_g16_supported) the
    kernels read the bf16 gradient as it is, with the results of the converted one."""
    if (grad_out.dtype is torch.bfloat16 and q.dtype == k.dtype == v.dtype == torch.float32 and grad_out.is_cuda
            and tuple(grad_out.shape) == tuple(v.shape)):
        grads = _loader.native().causal_backward(q, k, v, grad_out, None)
        if grads is not None:
            return grads
        _require_gpu(Q=q, K=k, V=v, prev_grad=grad_out)
        b, h, n, dk, dv = shape = _shapes(q, k, v)
        ok = _g16_cache.get(shape)
        if ok is None:
            ok = _remember(_g16_cache, shape, bool(_loader.lib().cott_causal_bwd_g16_supported(*shape)))
        q, k, v, g = q.contiguous(), k.contiguous(), v.contiguous(), grad_out.contiguous()
        grad_out = g
        if ok and not (q.data_ptr() | k.data_ptr() | v.data_ptr() | g.data_ptr()) & 15:
            dq, dk_, dv_ = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
            with _on(q.device):
                ws, ws_ptr = _workspace(_ws_bytes("cott_causal_bwd_workspace_bytes", *shape, _loader.F32), q.device)
                rc = _loader.lib().cott_causal_bwd_g16(q.data_ptr(), k.data_ptr(), v.data_ptr(), g.data_ptr(), dq.data_ptr(),
                                                       dk_.data_ptr(), dv_.data_ptr(), *shape, ws_ptr,
                                                       ws.numel() if ws is not None else 0, _stream(q.device))
            _check(rc, "cott_causal_bwd_g16")
            return dq, dk_, dv_
    return causal_backward(q, k, v, grad_out.contiguous().to(q.dtype))


def noncausal_dot_product(q, k, v, merged_heads=False):
    """o = q (k^T v) per (batch, head): BERT_Trainer/BertCosAttention.py:249.  merged_heads: o as (B,N,H,Dv)
    (the context-layer permute of :317 without its copy; see merged_heads_supported)."""
    if not merged_heads:
        o = _loader.native().noncausal(q, k, v)
        if o is not None:
            return o
    _require_gpu(Q=q, K=k, V=v)
    b, h, n, dk, dv = _shapes(q, k, v)
    if not (q.dtype == k.dtype == v.dtype):
        raise RuntimeError("Q, K and V must have the same dtype")
    code = _dtype_code(q)
    q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
    o = torch.empty((b, n, h, dv) if merged_heads else (b, h, n, dv), dtype=q.dtype, device=q.device)
    L = _loader.lib()
    with _on(q.device):
        ws, ws_ptr = _workspace(_ws_bytes("cott_noncausal_workspace_bytes", b, h, n, dk, dv, code), q.device)
        fn = L.cott_noncausal_fwd_bnhd if merged_heads else L.cott_noncausal_fwd
        rc = fn(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), b, h, n, dk, dv, code, ws_ptr,
                ws.numel() if ws is not None else 0, _stream(q.device))
    _check(rc, "cott_noncausal_fwd_bnhd" if merged_heads else "cott_noncausal_fwd")
    return o


def noncausal_backward(q, k, v, grad_out, merged_heads=False):
    """(dQ, dK, dV) of noncausal_dot_product (grad_out (B,N,H,Dv) with merged_heads)."""
    if not merged_heads:
        grads = _loader.native().noncausal_backward(q, k, v, grad_out)
        if grads is not None:
            return grads
    _require_gpu(Q=q, K=k, V=v, prev_grad=grad_out)
    b, h, n, dk, dv = _shapes(q, k, v)
    want = (b, n, h, dv) if merged_heads else tuple(v.shape)
    if tuple(grad_out.shape) != want:
        raise RuntimeError(f"prev_grad must have shape {want}, got {tuple(grad_out.shape)}")
    if not (q.dtype == k.dtype == v.dtype == grad_out.dtype):
        raise RuntimeError("Q, K, V and prev_grad must have the same dtype")
    code = _dtype_code(q)
    q, k, v, g = q.contiguous(), k.contiguous(), v.contiguous(), grad_out.contiguous()
    dq, dk_, dv_ = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    L = _loader.lib()
    with _on(q.device):
        ws, ws_ptr = _workspace(_ws_bytes("cott_noncausal_workspace_bytes", b, h, n, dk, dv, code), q.device)
        fn = L.cott_noncausal_bwd_bnhd if merged_heads else L.cott_noncausal_bwd
        rc = fn(q.data_ptr(), k.data_ptr(), v.data_ptr(), g.data_ptr(), dq.data_ptr(), dk_.data_ptr(), dv_.data_ptr(), b, h,
                n, dk, dv, code, ws_ptr, ws.numel() if ws is not None else 0, _stream(q.device))
    _check(rc, "cott_noncausal_bwd_bnhd" if merged_heads else "cott_noncausal_bwd")
    return dq, dk_, dv_


def _decode_out(out, *inputs):
    """Where a decode step may write its output: `out` itself, also when it IS one of q, k, v, but not when it shares memory
    with one of them in another way (heads run in any order, each reads its own rows before it writes them)."""
    for t in inputs:
        if _overlaps(out, t) and (out.data_ptr() != t.data_ptr() or out.shape != t.shape):
            return torch.empty_like(out)
    return out


def decode_step(state, q, k, v, out=None):
    """One recurrent step, in place on `state` (B,H,Dk,Dv; fp32, or fp64 for fp64 inputs):
    state += k v^T ; returns o = q state  (GPT_Trainer/GPTCosAttention.py:264,267).
    q,k: (B,H,Dk); v: (B,H,Dv); out: may share memory with q, k or v.  The reference's `past_KV` is
    `state.transpose(-1,-2)`."""
    _require_gpu(state=state, q=q, k=k, v=v)
    if state.dim() != 4 or q.dim() != 3 or k.dim() != 3 or v.dim() != 3:
        raise RuntimeError("decode_step: state (B,H,Dk,Dv), q/k (B,H,Dk), v (B,H,Dv)")
    b, h, dk, dv = state.shape
    if q.shape != (b, h, dk) or k.shape != (b, h, dk) or v.shape != (b, h, dv):
        raise RuntimeError("decode_step: q/k/v do not match the state shape")
    if not (q.dtype == k.dtype == v.dtype):
        raise RuntimeError("q, k and v must have the same dtype")
    code = _dtype_code(q)
    want = torch.float64 if q.dtype == torch.float64 else torch.float32
    if state.dtype != want or not state.is_contiguous():
        raise RuntimeError(f"decode_step: state must be a contiguous {want} tensor (it is updated in place)")
    q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
    if out is None:
        o = out = torch.empty((b, h, dv), dtype=q.dtype, device=q.device)
    elif out.shape != (b, h, dv) or out.dtype != q.dtype or not out.is_contiguous() or out.device != q.device:
        raise RuntimeError("decode_step: bad `out` tensor")
    else:
        o = _decode_out(out, q, k, v)
    L = _loader.lib()
    with _on(q.device):
        rc = L.cott_decode_step(state.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), b, h, dk,
                                dv, code, _stream(q.device))
    _check(rc, "cott_decode_step")
    return out if o is out else out.copy_(o)


def _check_norm_const(norm_const, sig, h, device):
    if (sig is not None or norm_const.numel() != h or norm_const.dtype not in _DTYPES or norm_const.device != device
            or not norm_const.is_contiguous()):
        raise RuntimeError(f"norm_const must be a contiguous floating tensor of {h} elements on the inputs' device, in place of sig")


def decode_step_prepared(state, q, k, v, sig=None, cnt=0.0, rotary=None, out=None, norm_const=None):
    """decode_step on the RAW projections of the new token: rotation (rotary = (table (P,R) fp32, position int)),
    L2 normalisation of q and k and v / max(cnt^sig[h], 1) run inside the kernel (one launch instead of
    prepare_inputs + decode_step).  q, k: (B,H,Dk) or the (B,1,H,Dk) projection output; v likewise; sig: (H) or
    None; cnt: number of tokens so far including this one.  norm_const, in place of sig: the H elements of the
    parameter, whose sigmoid the kernel forms."""
    if q.dim() == 4 and q.shape[1] == 1:
        q, k, v = q[:, 0], k[:, 0], v[:, 0]
    _require_gpu(state=state, q=q, k=k, v=v)
    if state.dim() != 4 or q.dim() != 3 or k.dim() != 3 or v.dim() != 3:
        raise RuntimeError("decode_step_prepared: state (B,H,Dk,Dv), q/k (B,H,Dk), v (B,H,Dv)")
    b, h, dk, dv = state.shape
    if q.shape != (b, h, dk) or k.shape != (b, h, dk) or v.shape != (b, h, dv):
        raise RuntimeError("decode_step_prepared: q/k/v do not match the state shape")
    if not (q.dtype == k.dtype == v.dtype):
        raise RuntimeError("q, k and v must have the same dtype")
    code = _dtype_code(q)
    want = torch.float64 if q.dtype == torch.float64 else torch.float32
    if state.dtype != want or not state.is_contiguous():
        raise RuntimeError(f"decode_step_prepared: state must be a contiguous {want} tensor")
    q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
    if out is None:
        o = out = torch.empty((b, h, dv), dtype=q.dtype, device=q.device)
    elif out.shape != (b, h, dv) or out.dtype != q.dtype or not out.is_contiguous() or out.device != q.device:
        raise RuntimeError("decode_step_prepared: bad `out` tensor")
    else:
        o = _decode_out(out, q, k, v)
    if sig is not None:
        if sig.shape != (h,):
            raise RuntimeError(f"sig must have shape {(h,)}")
        sig = sig.detach().to(device=q.device, dtype=torch.float32).contiguous()
    if norm_const is not None:
        _check_norm_const(norm_const, sig, h, q.device)
    table, pos, rdim, rows = None, 0, 0, 0
    if rotary is not None:
        table, pos = rotary
        if table.dim() != 2 or table.dtype != torch.float32 or table.device != q.device or not table.is_contiguous():
            raise RuntimeError("rotary table must be a contiguous float32 (positions, rotary_dim) tensor on the inputs' device")
        rows, rdim = table.shape
        pos = int(pos)
    L = _loader.lib()
    with _on(q.device):
        fn, scaling = L.cott_decode_step_prep, (_ptr(sig),)
        if norm_const is not None:
            fn, scaling = L.cott_decode_step_norm, (norm_const.data_ptr(), _DTYPES[norm_const.dtype])
        rc = fn(state.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), *scaling, float(cnt), _ptr(table), pos,
                rdim, rows, b, h, dk, dv, code, _stream(q.device))
    _check(rc, "cott_decode_step_prep")
    return out if o is out else out.copy_(o)


DECODE_BLOCK_ROWS = 16  # sequences up to which decode_block is built (kTokenRows, csrc/cott_launch.h)


def decode_block(x, wq, wk, wv, wo, state, sig=None, cnt=0.0, rotary=None, norm_const=None):
    """One new token of up to DECODE_BLOCK_ROWS sequences through a whole attention block without biases, three launches:
    q, k, v = x wq^T, x wk^T, x wv^T, then decode_step_prepared on them (state (B,H,D,D) fp32, updated in place), then
    the returned y = o wo^T.  x: (B,E) bf16 / fp16; weights (E,E), contiguous and 16-byte aligned, in x's type;
    sig, cnt, rotary, norm_const as in decode_step_prepared."""
    if sig is None and norm_const is not None and rotary is not None:
        y = _loader.native().decode_block(x, wq, wk, wv, wo, state, norm_const, float(cnt), rotary[0], int(rotary[1]))
        if y is not None:
            return y
    _require_gpu(x=x, wq=wq, wk=wk, wv=wv, wo=wo, state=state)
    dt = x.dtype
    code = _dtype_code(x)
    if x.dim() != 2 or state.dim() != 4:
        raise RuntimeError("decode_block: x (B,E), state (B,H,D,D)")
    b, e = x.shape
    sb, h, d, d2 = state.shape
    if sb != b or d2 != d or h * d != e or state.dtype != torch.float32 or not state.is_contiguous():
        raise RuntimeError(f"decode_block: state must be a contiguous float32 (B,H,D,D) tensor with H * D = {e}")
    for w in (wq, wk, wv, wo):
        if w.shape != (e, e) or w.dtype != dt or not w.is_contiguous():
            raise RuntimeError(f"decode_block: weights must be contiguous {(e, e)} tensors of type {dt}")
    if sig is not None and (sig.shape != (h,) or sig.dtype != torch.float32 or sig.device != x.device or not sig.is_contiguous()):
        raise RuntimeError(f"decode_block: sig must be a contiguous float32 tensor of shape {(h,)} on x's device")
    if norm_const is not None:
        _check_norm_const(norm_const, sig, h, x.device)
    table, pos, rdim, rows = None, 0, 0, 0
    if rotary is not None:
        table, pos = rotary
        if table.dim() != 2 or table.dtype != torch.float32 or table.device != x.device or not table.is_contiguous():
            raise RuntimeError("rotary table must be a contiguous float32 (positions, rotary_dim) tensor on the inputs' device")
        rows, rdim = table.shape
    x = x.contiguous()
    scratch = torch.empty((4, b, e), dtype=x.dtype, device=x.device)
    y = torch.empty((b, e), dtype=x.dtype, device=x.device)
    with _on(x.device):
        fn, scaling = _loader.lib().cott_decode_block, (_ptr(sig),)
        if norm_const is not None:
            fn, scaling = _loader.lib().cott_decode_block_norm, (norm_const.data_ptr(), _DTYPES[norm_const.dtype])
        rc = fn(x.data_ptr(), wq.data_ptr(), wk.data_ptr(), wv.data_ptr(), wo.data_ptr(), state.data_ptr(), y.data_ptr(),
                *scaling, float(cnt), _ptr(table), int(pos), rdim, rows, b, h, d, code, scratch.data_ptr(),
                scratch.numel() * 2, _stream(x.device))
    _check(rc, "cott_decode_block")
    return y


def _prep_side_inputs(b, h, n, keep, cnt, sig, device):
    if keep is not None:
        if keep.shape != (b, n):
            raise RuntimeError(f"keep must have shape {(b, n)}, got {tuple(keep.shape)}")
        if keep.dtype == torch.bool and keep.device == device and keep.is_contiguous():
            keep = keep.view(torch.uint8)  # a bool tensor already holds one 0 / 1 byte per element: no copy
        else:
            keep = keep.to(device=device, dtype=torch.uint8).contiguous()
    if (cnt is None) != (sig is None):
        raise RuntimeError("cnt and sig are given together (or neither)")
    if cnt is not None:
        if cnt.shape != (b, n) or sig.shape != (h,):
            raise RuntimeError(f"cnt must have shape {(b, n)} and sig {(h,)}")
        cnt = cnt.to(device=device, dtype=torch.float32).contiguous()
        sig = sig.detach().to(device=device, dtype=torch.float32).contiguous()
    return keep, cnt, sig


def _ptr(t):
    return t.data_ptr() if t is not None else None


def _prep_shapes(q, k, v, bnhd):
    """(b, h, n, dk, dv) of q, k, v given as (B,H,N,D), or as (B,N,H,D) when `bnhd`."""
    if bnhd:
        if q.dim() != 4 or k.dim() != 4 or v.dim() != 4 or q.shape != k.shape or q.shape[:3] != v.shape[:3]:
            raise RuntimeError("Q, K and V must have shape (N, S, H, D) and agree in (N, S, H)")
        b, n, h, dk = q.shape
        return b, h, n, dk, v.size(3)
    return _shapes(q, k, v)


_CONVERT_MAX = 8  # COTT_CONVERT_MAX
_PLAIN = (torch.Tensor, torch.nn.Parameter)


def plain(*tensors):
    """Whether all are ordinary tensors, whose numbers lie at their data pointer (a subclass may keep them elsewhere)."""
    return all(type(t) in _PLAIN for t in tensors)


def convert_into(pairs, dtype):
    """dst.copy_(src) for every (src, dst) of `pairs`, dst contiguous of dtype `dtype`: fp32 sources become bf16 / fp16 in one
    launch."""
    pairs = [(src, dst) for src, dst in pairs if src.numel()]
    if not pairs:
        return
    device = pairs[0][0].device
    if (dtype not in (torch.bfloat16, torch.float16) or len(pairs) > _CONVERT_MAX
            or any(src.dtype != torch.float32 or src.device != device or not src.is_cuda or not plain(src, dst)
                   or src.shape != dst.shape or not src.is_contiguous() or (src.data_ptr() | dst.data_ptr()) & 15
                   or src.numel() > 1 << 30 for src, dst in pairs)):
        for src, dst in pairs:
            dst.copy_(src)
        return
    n = len(pairs)
    pointers = ctypes.c_void_p * n
    with _on(device):
        rc = _loader.lib().cott_convert(pointers(*(src.data_ptr() for src, _ in pairs)), pointers(*(dst.data_ptr() for _, dst in pairs)),
                                        (ctypes.c_long * n)(*(src.numel() for src, _ in pairs)), n, _DTYPES[dtype], _stream(device))
    _check(rc, "cott_convert")


def keep_and_counts(mask, b, n, running):
    """(keep, cnt) of the surrounding model's additive mask with b * n entries, 0 at real tokens: keep (b,n) bool = (mask == 0)
    and cnt (b,n) fp32, the kept positions up to each one (running) or in its sequence, as one launch; None where the mask is
    of another kind (its type, strided, on the CPU)."""
    code = _DTYPES.get(mask.dtype)
    if (not mask.is_cuda or not plain(mask) or code is None or code == _loader.F64 or mask.numel() != b * n or not mask.is_contiguous()
            or n > 1 << 24):
        return None
    keep = torch.empty((b, n), dtype=torch.bool, device=mask.device)
    cnt = torch.empty((b, n), dtype=torch.float32, device=mask.device)
    with _on(mask.device):
        rc = _loader.lib().cott_keep_counts(mask.data_ptr(), code, keep.data_ptr(), cnt.data_ptr(), b, n, int(running),
                                            _stream(mask.device))
    _check(rc, "cott_keep_counts")
    return keep, cnt


def keep_and_counts_preferred(b, n, running):
    """Whether keep_and_counts, one workgroup per sequence, is the better form against `mask == 0` and torch's reductions: not for
    long sequences that are too few to fill the chip.  us, this kernel / torch: running, 1 sequence N 16384 18 / 21, 20000 21 / 21,
    32768 33 / 21; 2 sequences N 16384 18 / 44, 131072 129 / 298; totals, 1 sequence N 32768 21 / 28, 49152 30 / 27, 64 sequences N
    65536 43 / 47."""
    few, longest = (b < 2, 1 << 14) if running else (b < 64, 1 << 15)
    return not few or n <= longest


def head_sums(rows):
    """Sums of rows (B,H,N) fp32, contiguous, over B and N.  One workgroup per head adds up to 32768 rows; more are added by one
    workgroup per head and sequence, or piece of a sequence, first (us, 16 heads, in one step / in two, of which 13 host / torch: 8 x
    2048 5 / - / 8, 32 x 2048 15 / 13 / 17, 64 x 2048 27 / 13 / 13, 64 x 8192 103 / 14 / 18, 256 x 4096 215 / 24 / 28)."""
    b, h, n = rows.shape
    if b * n > 1 << 15:
        pieces = 1
        while n % (2 * pieces) == 0 and n // (2 * pieces) >= 4096:
            pieces *= 2
        if not 512 <= n // pieces <= 1 << 15 or b * h * pieces > 1 << 22:  # too little or too much for one workgroup
            return rows.sum(dim=(0, 2))
        return head_sums(_head_sums(rows, 1, b * h * pieces, n // pieces).view(b, h, pieces))
    return _head_sums(rows, b, h, n)


def _head_sums(rows, b, h, n):
    out = torch.empty(h, dtype=torch.float32, device=rows.device)
    with _on(rows.device):
        _check(_loader.lib().cott_head_sums(rows.data_ptr(), out.data_ptr(), b, h, n, _stream(rows.device)), "cott_head_sums")
    return out


def column_sums(x, sizes=None):
    """Sums over the rows of x (rows, cols), in fp32 at least; with `sizes` a list of tensors of their own with that many of them."""
    rows, cols = x.shape
    if (not x.is_cuda or not plain(x) or x.dtype not in (torch.bfloat16, torch.float16) or rows < 2 or cols == 0 or cols % 8 or x.stride(1) != 1
            or x.stride(0) < cols or x.stride(0) % 8 or x.data_ptr() % 16
            or sizes is not None and (len(sizes) > _CONVERT_MAX or any(n % 8 for n in sizes))):
        total = x.sum(0, dtype=torch.promote_types(x.dtype, torch.float32))
        return total if sizes is None else [block.clone() for block in total.split(sizes)]
    outs, count, where, lengths = _blocks([cols] if sizes is None else sizes, 1, x.device)
    with _on(x.device):
        ws, ws_ptr = _workspace(_ws_bytes("cott_column_sums_workspace_bytes", rows, cols), x.device)
        rc = _loader.lib().cott_column_sums_blocks(x.data_ptr(), where, lengths, count, rows, x.stride(0), _DTYPES[x.dtype], ws_ptr,
                                                   ws.numel() if ws is not None else 0, _stream(x.device))
    _check(rc, "cott_column_sums")
    return outs[0].view(cols) if sizes is None else [out.view(-1) for out in outs]


def _blocks(sizes, width, device):
    """(tensors (size, width) fp32, their number, and the arrays of their addresses and lengths) for the library."""
    outs = [torch.empty((n, width), dtype=torch.float32, device=device) for n in sizes]
    n = len(outs)
    return outs, n, (ctypes.c_void_p * n)(*[out.data_ptr() for out in outs]), (ctypes.c_long * n)(*[width * rows for rows in sizes])


def add_pieces(parts, sizes):
    """Sums over the first dimension of parts (pieces, rows, width) fp32, as tensors of their own with `sizes` rows each."""
    if (not parts.is_cuda or not plain(parts) or parts.dtype != torch.float32 or not parts.is_contiguous() or parts.shape[2] % 4 or parts.data_ptr() % 16
            or len(sizes) > _CONVERT_MAX or parts.numel() == 0):
        return [block.sum(0) for block in parts.split(sizes, dim=1)]
    outs, count, where, lengths = _blocks(sizes, parts.shape[2], parts.device)
    with _on(parts.device):
        rc = _loader.lib().cott_add_pieces(parts.data_ptr(), where, lengths, count, parts.shape[0], _stream(parts.device))
    _check(rc, "cott_add_pieces")
    return outs


def _token_stride(q, k, v, b, h, n, dk, dv):
    """Elements from one position to the next when q, k, v are neighbouring column slices, in that order, of one (B,N,H*(2 Dk +
    Dv)) tensor, as `autograd.InputProjections` hands them out; else 0.  The kernels read that layout as it is."""
    row = h * (2 * dk + dv)
    if row % 8 or n * row > 1 << 30 or q.numel() == 0:
        return 0
    for t, d in ((q, dk), (k, dk), (v, dv)):
        for size, have, want in zip((b, n, h, d), t.stride(), (n * row, row, d, 1)):
            if size != 1 and have != want:
                return 0
    size = q.element_size()
    at = q.data_ptr()
    if (at % 16 or h * dk * size % 16 or k.data_ptr() != at + h * dk * size or v.data_ptr() != at + 2 * h * dk * size
            or not q.untyped_storage().data_ptr() == k.untyped_storage().data_ptr() == v.untyped_storage().data_ptr()):
        return 0
    return row


def preparation_rows(q, k, v, bnhd):
    """q, k, v as the preparation takes them without a copy of its own: column slices of one tensor as they are (bnhd), anything
    else contiguous."""
    if bnhd and q.is_cuda and k.is_cuda and v.is_cuda and q.dtype == k.dtype == v.dtype and not q.is_contiguous():
        if _token_stride(q, k, v, *_prep_shapes(q, k, v, bnhd)):
            return q, k, v
    return q.contiguous(), k.contiguous(), v.contiguous()


def _input_layout(q, k, v, bnhd, b, h, n, dk, dv):
    """(q, k, v, layout): 0 and 1 are the library's in_bnhd, larger ones the token_stride of its strided forms."""
    stride = _token_stride(q, k, v, b, h, n, dk, dv) if bnhd and not q.is_contiguous() else 0
    if stride:
        return q, k, v, stride
    return q.contiguous(), k.contiguous(), v.contiguous(), int(bool(bnhd))


def _rotary_args(rotary, b, n, dk, device, check=True):
    if rotary is None:
        return None, None, 0, 0
    table, pos = rotary
    if table.dim() != 2 or table.size(1) % 4 != 0 or table.size(1) > dk:
        raise RuntimeError("rotary table must be (positions, rotary_dim), rotary_dim a multiple of 4 and <= Dk")
    if pos.dim() == 2 and pos.shape == (1, n):  # one row for the whole batch, as GPT-J's model makes them
        pos = pos.expand(b, n)
    if pos.shape != (b, n):
        raise RuntimeError(f"position ids must have shape {(b, n)}")
    # (this check reads the positions back and so waits for the device; callers in a hot loop pass check=False,
    # the kernel then clamps stray positions to the table)
    if check and pos.numel() and (int(pos.max()) >= table.size(0) or int(pos.min()) < 0):
        raise RuntimeError("position id outside the rotary table")
    table = table.to(device=device, dtype=torch.float32).contiguous()
    pos = pos.to(device=device, dtype=torch.int64).contiguous()
    return table, pos, table.size(1), table.size(0)


def prepare_inputs(q, k, v, keep=None, cnt=None, sig=None, out_dtype=None, rotary=None, bnhd=False,
                   check_positions=True):
    """Fused input preparation of the cosine-attention module, one pass per tensor:
        q_out = keep * q / max(|q|, 1e-12),  k_out likewise,  v_out = keep * v / max(cnt ** sig[h], 1)
    converted to `out_dtype` (default: the input dtype) and returned as (B,H,N,D).  Replaces
    GPT_Trainer/GPTCosAttention.py:229-248 and BERT_Trainer/BertCosAttention.py:162-178.
    keep: (B,N) bool/0-1, True = real token; cnt: (B,N) number of kept keys each position attends to;
    sig: (H,) = sigmoid(norm_const).
    rotary=(table, position_ids): also applies the GPT-J rotary embedding to the first table.size(1) columns of
    q and k (GPTCosAttention.py:462-476); bnhd=True: q, k, v are given as (B,N,H,D), the layout the projections
    produce, and the head permute of :478-479 happens in the same pass."""
    _require_gpu(Q=q, K=k, V=v)
    b, h, n, dk, dv = _prep_shapes(q, k, v, bnhd)
    if not (q.dtype == k.dtype == v.dtype):
        raise RuntimeError("Q, K and V must have the same dtype")
    code = _dtype_code(q)
    out_dtype = out_dtype or q.dtype
    if out_dtype not in _DTYPES:
        raise ValueError("Only float32, float64, float16, and bfloat16 are supported")
    keep, cnt, sig = _prep_side_inputs(b, h, n, keep, cnt, sig, q.device)
    table, pos, rdim, rows = _rotary_args(rotary, b, n, dk, q.device, check_positions)
    q, k, v, layout = _input_layout(q, k, v, bnhd, b, h, n, dk, dv)
    qo, ko = (torch.empty((b, h, n, dk), dtype=out_dtype, device=q.device) for _ in range(2))
    vo = torch.empty((b, h, n, dv), dtype=out_dtype, device=q.device)
    L = _loader.lib()
    with _on(q.device):
        rc = (L.cott_prep_strided_fwd if layout > 1 else L.cott_prep_ex_fwd)(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), qo.data_ptr(), ko.data_ptr(), vo.data_ptr(), _ptr(keep), _ptr(cnt), _ptr(sig),
            _ptr(table), _ptr(pos), rdim, rows, layout, b, h, n, dk, dv, code, _DTYPES[out_dtype], _stream(q.device))
    _check(rc, "cott_prep_ex_fwd")
    return qo, ko, vo


def prepare_inputs_backward(q, k, v, gq, gk, gv, keep=None, cnt=None, sig=None, want_dsig=False, rotary=None,
                            bnhd=False, check_positions=True):
    """Gradients of `prepare_inputs` with respect to q, k, v (their dtype and layout, slices of one tensor where q, k, v are) and, if asked, to sig (H,).
    gq, gk, gv: gradients with respect to the outputs, (B,H,N,D)."""
    _require_gpu(Q=q, K=k, V=v, gq=gq, gk=gk, gv=gv)
    b, h, n, dk, dv = _prep_shapes(q, k, v, bnhd)
    if gq.shape != (b, h, n, dk) or gk.shape != (b, h, n, dk) or gv.shape != (b, h, n, dv):
        raise RuntimeError("gradient shapes must be (B,H,N,D)")
    if not (q.dtype == k.dtype == v.dtype) or not (gq.dtype == gk.dtype == gv.dtype):
        raise RuntimeError("q, k, v share one dtype and their gradients share one dtype")
    code, gcode = _dtype_code(q), _dtype_code(gq)
    keep, cnt, sig = _prep_side_inputs(b, h, n, keep, cnt, sig, q.device)
    table, pos, rdim, rows = _rotary_args(rotary, b, n, dk, q.device, check_positions)
    q, k, v, layout = _input_layout(q, k, v, bnhd, b, h, n, dk, dv)
    gq, gk, gv = gq.contiguous(), gk.contiguous(), gv.contiguous()
    if layout > 1:  # the gradients as column slices of one tensor, too
        dq, dk_, dv_ = (t.view(b, n, h, d) for t, d in zip(torch.empty((b, n, layout), dtype=q.dtype, device=q.device).split(
            (h * dk, h * dk, h * dv), dim=-1), (dk, dk, dv)))
    else:
        dq, dk_, dv_ = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    drows = torch.empty((b, h, n), dtype=torch.float32, device=q.device) if (want_dsig and sig is not None) else None
    L = _loader.lib()
    with _on(q.device):
        rc = (L.cott_prep_strided_bwd if layout > 1 else L.cott_prep_ex_bwd)(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), gq.data_ptr(), gk.data_ptr(), gv.data_ptr(), dq.data_ptr(), dk_.data_ptr(),
            dv_.data_ptr(), _ptr(drows), _ptr(keep), _ptr(cnt), _ptr(sig), _ptr(table), _ptr(pos), rdim, rows, layout, b, h, n, dk, dv, code,
            gcode, _stream(q.device))
    _check(rc, "cott_prep_ex_bwd")
    dsig = head_sums(drows) if drows is not None else None
    return dq, dk_, dv_, dsig
