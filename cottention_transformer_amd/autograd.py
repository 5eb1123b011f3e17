"""torch.autograd boundary: `CustomAttention` with the reference's signature, plus the
non-causal counterpart.  Reference: Cuda_Kernel/Custom_Kernel.py:7-141."""
import torch
import torch.nn.utils.parametrize

from . import ops

_SUPPORTED = (torch.float32, torch.float64, torch.float16, torch.bfloat16)


def _autocast_target(q, half_entry=False):
    """Forward-time dtype rule of forward_<T>, Cuda_Kernel/combined_kernel_general.cu:377-389:
    under autocast an fp32 Q is computed in the autocast type (fp16 only for the `float16` entry),
    otherwise in Q's own type; K and V are converted to match."""
    try:
        enabled = torch.is_autocast_enabled("cuda")
    except TypeError:  # older signature
        enabled = torch.is_autocast_enabled()
    if enabled and q.dtype == torch.float32:
        return torch.float16 if half_entry else torch.bfloat16
    return q.dtype


class CustomAttention(torch.autograd.Function):
    """O = causal cosine-attention core of (Q, K, V), tensors (N, H, S, D); apply(Q, K, V) -> O.

    backward_in_forward_dtype (class attribute, default False = the reference's behaviour): under autocast the
    reference computes the forward in bf16 but saves the fp32 tensors (Custom_Kernel.py:16) and runs the backward on
    them in fp32 (:38, :106-108).  Set to True, the tensors are saved as the forward pass rounded them and the
    backward runs in that 16-bit type too (gradients returned in the inputs' types): the gradients of the function
    that was actually evaluated, from the 16-bit kernels (several times faster than the fp32 ones) and from half
    the saved bytes."""

    backward_in_forward_dtype = False

    @staticmethod
    def forward(ctx, Q, K, V):
        if Q.dtype not in _SUPPORTED:
            raise ValueError("Only float32, float64, float16, and bfloat16 are supported")
        Q, K, V = Q.contiguous(), K.contiguous(), V.contiguous()
        dt = _autocast_target(Q, half_entry=(Q.dtype == torch.float16))
        ctx.grad_dtypes = None
        if dt in (torch.float16, torch.bfloat16) and CustomAttention.backward_in_forward_dtype:
            ctx.grad_dtypes = (Q.dtype, K.dtype, V.dtype)
            Q, K, V = Q.to(dt), K.to(dt), V.to(dt)
        if dt == Q.dtype == K.dtype == V.dtype and dt in (torch.float16, torch.bfloat16):
            # 16-bit tensors, forward and backward in the same type: on sequences long enough to be cut into groups
            # the forward pass also leaves the states the backward pass starts dQ from (None otherwise)
            out, states = ops.causal_dot_product_saving(Q, K, V)
            ctx.save_for_backward(Q, K, V, *(() if states is None else (states,)))
            return out
        ctx.save_for_backward(Q, K, V)  # saved before any autocast conversion (Custom_Kernel.py:16)
        return ops.causal_dot_product_as(Q, K, V, dt)

    @staticmethod
    def backward(ctx, grad_output):
        Q, K, V, *states = ctx.saved_tensors
        if Q.dtype not in _SUPPORTED:
            raise ValueError("Only float32, float64, float16, and bfloat16 are supported")
        # One fused call in the saved tensors' dtype replaces the three launches of
        # Custom_Kernel.py:106-108 (same operand permutations inside the library).
        if states:
            grads = ops.causal_backward(Q, K, V, grad_output.contiguous().to(Q.dtype), saved=states[0])
        else:
            grads = ops.causal_backward_from(Q, K.to(Q.dtype), V.to(Q.dtype), grad_output)
        if ctx.grad_dtypes is not None:
            grads = tuple(x.to(t) for x, t in zip(grads, ctx.grad_dtypes))
        return grads


class CustomAttentionMergedHeads(torch.autograd.Function):
    """CustomAttention with the head merge folded in: apply(Q, K, V) -> O of shape (N, S, H, Dv), i.e. the rows
    of the (N, S, H*Dv) input of the output projection (GPT_Trainer/GPTCosAttention.py:106-113, called at :500), and a backward
    that reads the gradient in that layout.  Only where ops.merged_heads_supported() holds for the dtype the
    forward computes in; callers fall back to CustomAttention + permute otherwise."""

    @staticmethod
    def forward(ctx, Q, K, V):
        if Q.dtype not in _SUPPORTED:
            raise ValueError("Only float32, float64, float16, and bfloat16 are supported")
        dt = _autocast_target(Q, half_entry=(Q.dtype == torch.float16))
        Q, K, V = Q.contiguous().to(dt), K.contiguous().to(dt), V.contiguous().to(dt)
        # in the computed (16-bit) type: the backward reads the merged layout too; with the states for its dQ
        out, states = ops.causal_dot_product_saving(Q, K, V, merged_heads=True)
        ctx.save_for_backward(Q, K, V, *(() if states is None else (states,)))
        return out

    @staticmethod
    def backward(ctx, grad_output):
        Q, K, V, *states = ctx.saved_tensors
        return ops.causal_backward(Q, K, V, grad_output.contiguous().to(Q.dtype), merged_heads=True,
                                   saved=states[0] if states else None)


class NonCausalAttention(torch.autograd.Function):
    """O = Q (K^T V): the BERT form (BERT_Trainer/BertCosAttention.py:249) as one fused operator."""

    @staticmethod
    def forward(ctx, Q, K, V):
        if Q.dtype not in _SUPPORTED:
            raise ValueError("Only float32, float64, float16, and bfloat16 are supported")
        Q, K, V = Q.contiguous(), K.contiguous(), V.contiguous()
        ctx.save_for_backward(Q, K, V)
        dt = _autocast_target(Q)
        return ops.noncausal_dot_product(Q.to(dt), K.to(dt), V.to(dt))

    @staticmethod
    def backward(ctx, grad_output):
        Q, K, V = ctx.saved_tensors
        g = grad_output.contiguous().to(Q.dtype)
        return ops.noncausal_backward(Q, K.to(Q.dtype), V.to(Q.dtype), g)


class NonCausalAttentionMergedHeads(torch.autograd.Function):
    """NonCausalAttention returning O as (N, S, H, Dv) and reading its gradient in that layout
    (BERT_Trainer/BertCosAttention.py:317); same conditions as CustomAttentionMergedHeads."""

    @staticmethod
    def forward(ctx, Q, K, V):
        if Q.dtype not in _SUPPORTED:
            raise ValueError("Only float32, float64, float16, and bfloat16 are supported")
        dt = _autocast_target(Q)
        Q, K, V = Q.contiguous().to(dt), K.contiguous().to(dt), V.contiguous().to(dt)
        ctx.save_for_backward(Q, K, V)
        return ops.noncausal_dot_product(Q, K, V, merged_heads=True)

    @staticmethod
    def backward(ctx, grad_output):
        Q, K, V = ctx.saved_tensors
        return ops.noncausal_backward(Q, K, V, grad_output.contiguous().to(Q.dtype), merged_heads=True)


class PrepareInputs(torch.autograd.Function):
    """(q, k, v, keep, cnt, sig, out_dtype[, rot_table, position_ids, bnhd]) -> (q_hat, k_hat, v_scaled), (B,H,N,D):
    the normalise / value-scale / mask steps in front of the attention op (GPT_Trainer/GPTCosAttention.py:229-248),
    optionally with the rotary embedding and the head permute before them (:462-476), as one fused operator with a
    fused backward.  `sig` = sigmoid(norm_const) per head, differentiable; the other side inputs are constants."""

    @staticmethod
    def forward(ctx, q, k, v, keep, cnt, sig, out_dtype, rot_table=None, position_ids=None, bnhd=False):
        q, k, v = ops.preparation_rows(q, k, v, bnhd)
        ctx.save_for_backward(q, k, v, keep, cnt, sig, rot_table, position_ids)
        ctx.bnhd = bool(bnhd)
        rotary = (rot_table, position_ids) if rot_table is not None else None
        # positions are not read back here (that would stall the launch queue): the kernel clamps them to the table
        return ops.prepare_inputs(q, k, v, keep, cnt, sig, out_dtype, rotary=rotary, bnhd=bnhd, check_positions=False)

    @staticmethod
    def backward(ctx, gq, gk, gv):
        q, k, v, keep, cnt, sig, rot_table, position_ids = ctx.saved_tensors
        want = sig is not None and ctx.needs_input_grad[5]
        rotary = (rot_table, position_ids) if rot_table is not None else None
        dq, dk, dv, dsig = ops.prepare_inputs_backward(q, k, v, gq.contiguous(), gk.contiguous(), gv.contiguous(), keep,
                                                       cnt, sig, want_dsig=want, rotary=rotary, bnhd=ctx.bnhd,
                                                       check_positions=False)
        if dsig is not None:
            dsig = dsig.to(sig.dtype)
        return dq, dk, dv, None, None, dsig, None, None, None, None


class PreparedCausalAttention(torch.autograd.Function):
    """(q, k, v, keep, cnt, sig, rot_table, first_position, bnhd, merged_heads) -> O: the preparation steps of
    PrepareInputs and the causal attention op as ONE forward launch on the raw projections
    (ops.causal_dot_product_prepared).  The kernel also leaves the prepared q, k, v for the backward pass, which is
    the attention gradient on them followed by the fused backward of the preparation.  first_position: an int (the
    table row of position s is first_position + s) or the block's (B,N) position_ids tensor, any values, which is never
    read back to the host.  Only where ops.fused_preparation_supported() holds."""

    @staticmethod
    def forward(ctx, q, k, v, keep, cnt, sig, rot_table=None, first_position=0, bnhd=False, merged_heads=False):
        q, k, v = ops.preparation_rows(q, k, v, bnhd)
        ids = first_position if torch.is_tensor(first_position) else None
        if ids is not None and bnhd and ids.dim() == 2 and ids.shape == (1, q.shape[1]):
            ids = ids.expand(q.shape[0], -1).contiguous()  # once, not again in the backward
        rotary = (rot_table, ids if ids is not None else int(first_position)) if rot_table is not None else None
        out, prepared, states = ops.causal_dot_product_prepared(q, k, v, keep, cnt, sig, rotary=rotary, bnhd=bnhd,
                                                                merged_heads=merged_heads, want_prepared=True,
                                                                save_states=True)
        ctx.save_for_backward(q, k, v, keep, cnt, sig, rot_table, ids, *prepared, *(() if states is None else (states,)))
        ctx.first_position = 0 if ids is not None else int(first_position)
        ctx.bnhd, ctx.merged = bool(bnhd), bool(merged_heads)
        return out

    @staticmethod
    def backward(ctx, grad_output):
        q, k, v, keep, cnt, sig, rot_table, ids, qh, kh, vh, *states = ctx.saved_tensors
        gq, gk, gv = ops.causal_backward(qh, kh, vh, grad_output.contiguous().to(qh.dtype), merged_heads=ctx.merged,
                                         saved=states[0] if states else None)
        rotary = None
        if rot_table is not None:
            b, n = (q.shape[0], q.shape[1]) if ctx.bnhd else (q.shape[0], q.shape[2])
            if ids is not None:
                pos = (ids if ids.dim() == 2 else ids[None, :]).expand(b, n)
            else:
                pos = torch.arange(ctx.first_position, ctx.first_position + n, device=q.device).expand(b, n)
            rotary = (rot_table, pos)
        want = sig is not None and ctx.needs_input_grad[5]
        dq, dk, dv, dsig = ops.prepare_inputs_backward(q, k, v, gq, gk, gv, keep, cnt, sig, want_dsig=want, rotary=rotary,
                                                       bnhd=ctx.bnhd, check_positions=False)
        if dsig is not None:
            dsig = dsig.to(sig.dtype)
        return dq, dk, dv, None, None, dsig, None, None, None, None


class PreparedNonCausalAttention(torch.autograd.Function):
    """(q, k, v, keep, cnt, sig, bnhd, merged_heads) -> O: the preparation steps of PrepareInputs (no rotation) and
    the non-causal op Q (K^T V) as ONE forward launch on the raw projections (ops.noncausal_dot_product_prepared;
    BERT_Trainer/BertCosAttention.py:162-178 in front of :249).  The kernel leaves the prepared q, k, v for the
    backward pass: the attention gradients on them, then the fused backward of the preparation.  Only where
    ops.noncausal_fused_preparation_supported() holds."""

    @staticmethod
    def forward(ctx, q, k, v, keep, cnt, sig, bnhd=False, merged_heads=False):
        q, k, v = ops.preparation_rows(q, k, v, bnhd)
        out, prepared = ops.noncausal_dot_product_prepared(q, k, v, keep, cnt, sig, bnhd=bnhd, merged_heads=merged_heads)
        ctx.save_for_backward(q, k, v, keep, cnt, sig, *prepared)
        ctx.bnhd, ctx.merged = bool(bnhd), bool(merged_heads)
        return out

    @staticmethod
    def backward(ctx, grad_output):
        q, k, v, keep, cnt, sig, qh, kh, vh = ctx.saved_tensors
        gq, gk, gv = ops.noncausal_backward(qh, kh, vh, grad_output.contiguous().to(qh.dtype), merged_heads=ctx.merged)
        want = sig is not None and ctx.needs_input_grad[5]
        dq, dk, dv, dsig = ops.prepare_inputs_backward(q, k, v, gq, gk, gv, keep, cnt, sig, want_dsig=want, bnhd=ctx.bnhd,
                                                       check_positions=False)
        if dsig is not None:
            dsig = dsig.to(sig.dtype)
        return dq, dk, dv, None, None, dsig, None, None


def _row_pieces(rows, out, inner):
    """Pieces that the rows of a weight gradient (out, inner) are cut into: until the pieces' 256 x 128 tiles fill the chip (no
    limit up to 1 M elements), as long as a piece keeps 2048 rows and more than out * inner / 2048, below which forming
    and adding an fp32 piece costs what the fuller chip gives.  bf16, us in 1 / 2 / 4 / 8 pieces with their sum: 16384 rows x 1024 x
    1024 104 / 69 / 50 / 46, 2304 x 768 128 / 85 / 90 / 78, 1536 x 1536 152 / 119 / 90 / 106, 3072 x 1024 156 / 121 / 106 / 121, 2048 x
    2048 160 / 138 / 135 / 159; 8192 rows: 2304 x 768 71 / 49 / 56 / 52, 3072 x 1024 86 / 69 / 66, 2048 x 2048 86 / 80 / 84, 4608 x
    1536 126 / 129; 4096 rows: 3072 x 1024 50 / 43, 2048 x 2048 50 / 51, 4608 x 1536 72 / 79."""
    tiles = 0 if out * inner <= 1 << 20 else -(-out // 256) * -(-inner // 128)
    pieces = 1
    while (pieces < 16 and tiles * pieces < 256 and rows % (2 * pieces) == 0 and rows // (2 * pieces) >= 2048
           and rows // (2 * pieces) * 2048 > out * inner):
        pieces *= 2
    return pieces


def _weight_gradient(gy, x, sizes=None):
    """gy^T x for gy (R, out), x (R, in), or with `sizes` a list of its blocks of that many rows.  With many rows and a small
    weight the library's single GEMM fills the chip with too few tiles over a long reduction; the rows are cut into pieces
    (`_row_pieces`) multiplied as one batched GEMM instead.  The pieces leave it in fp32 and are added in fp32, each block into
    a tensor of its own, so the result has the sums of the single GEMM."""
    r = x.shape[0]
    pieces = 1
    # (with a second derivative to record, the single product: the batched one has none with fp32 results, and its own
    # backward would multiply by transposed views, which has faulted in 16 bits; contiguous() for the same reason)
    recording = torch.is_grad_enabled() and (gy.requires_grad or x.requires_grad)
    if x.is_cuda and x.dtype in (torch.float16, torch.bfloat16) and not recording:
        pieces = _row_pieces(r, gy.shape[1], x.shape[1])
    if pieces == 1:
        product = gy.t() @ x
        return product if sizes is None else product.split(sizes)
    a, b = gy.view(pieces, r // pieces, -1).transpose(1, 2), x.contiguous().view(pieces, r // pieces, -1)
    blocks = ops.add_pieces(torch.bmm(a, b, out_dtype=torch.float32), [gy.shape[1]] if sizes is None else sizes)
    return blocks[0] if sizes is None else blocks


def own(t, dtype=None):
    """t as `dtype`, in memory that holds nothing else: for what is kept, saved or dropped by itself."""
    out = t if dtype is None else t.to(dtype)
    return out.clone() if out.untyped_storage().nbytes() != out.numel() * out.element_size() else out


def _joined(parts, sizes):
    """(R, n_0), (R, n_1), ... side by side as one (R, sum n) matrix: without a copy when they are neighbouring column slices of
    one and nothing is recorded for a second derivative (which would see a view of the first slice alone)."""
    if torch.is_grad_enabled():
        return torch.cat(parts, dim=1)
    first, total, size = parts[0], sum(sizes), parts[0].element_size()
    at, rows = first.data_ptr(), first.shape[0]
    for t, n in zip(parts, sizes):
        if (t.data_ptr() != at or t.dtype != first.dtype or n != 1 and t.stride(1) != 1 or rows != 1 and t.stride(0) != total
                or t.untyped_storage().data_ptr() != first.untyped_storage().data_ptr()):
            return torch.cat(parts, dim=1)
        at += n * size
    return first.as_strided((rows, total), (total, 1))


def _of_column_blocks(f, g, sizes, wanted):
    """What f(g, sizes) makes of each column block of g: of the whole at once where all are wanted, else of each wanted one by
    itself (16384 x 3072 x 1024: the weight gradients of all three 106 us, of one 46)."""
    if all(wanted):
        return f(g, sizes)
    return [f(part, [part.shape[1]])[0] if want else None for part, want in zip(g.split(sizes, dim=1), wanted)]


def _joint_form(x, weights, biases, cd):
    """Whether the weights, and the biases if there are any, can be converted to `cd` into one matrix and one vector: all of them have
    to be converted, are ordinary tensors on x's device, fit x, and a bias has an entry for every output (nn.functional.linear would
    also spread one of another shape)."""
    if len(weights) < 2 or not ops.plain(x, *weights):
        return False
    if any(w.dtype == cd or w.device != x.device or w.dim() != 2 or w.shape[1] != x.shape[-1] for w in weights):
        return False
    if all(b is None for b in biases):
        return True
    return all(b is not None and ops.plain(b) and b.device == x.device and b.shape == w.shape[:1] for w, b in zip(weights, biases))


class InputProjections(torch.autograd.Function):
    """(x, w_0, b_0, w_1, b_1, ...) -> (x w_0^T + b_0, x w_1^T + b_1, ...): the q / k / v projections of an attention
    block (GPT_Trainer/GPTCosAttention.py:443-445, BERT_Trainer/BertCosAttention.py:121,143-144 with biases) as one
    operator.  Under autocast x is converted once for all of them, the gradient of x is accumulated by the GEMMs
    themselves and converted back once, and the weight gradients take `_weight_gradient`.  b_i may be None.

    Several weights that have to be converted anyway (fp32 parameters under autocast) are converted into one matrix, and all
    the products are one GEMM each: the outputs are then column slices of one tensor, which the input preparation
    reads, and whose gradients it writes, as such; dx leaves the GEMM in fp32.  Forward / dx / dW of three projections, us, one
    by one and together: 16384 x 1024 98 / 124 / 157 and 94 / 91 / 106, 16384 x 768 75 / 86 / 133 and 65 / 55 / 78,
    2048 x 512 60 / 54 / 59 and 19 / 19 / 20."""

    @staticmethod
    def forward(ctx, x, *wb):
        # the type nn.Linear would compute in: the autocast type for 16- and 32-bit inputs on the GPU, else x's own
        cd = x.dtype
        if x.is_cuda and x.dtype != torch.float64 and torch.is_autocast_enabled("cuda"):
            cd = torch.get_autocast_dtype("cuda")
        weights, biases = wb[0::2], wb[1::2]
        ctx.x_meta = (x.shape, x.dtype)
        ctx.wb_dtypes = [None if t is None else t.dtype for t in wb]
        ctx.sizes = [w.shape[0] for w in weights]
        ctx.joint = x.is_cuda and _joint_form(x, weights, biases, cd)
        if ctx.joint:
            x2 = x.reshape(-1, x.shape[-1])
            w = torch.empty((sum(ctx.sizes), x2.shape[1]), dtype=cd, device=x.device)
            convert = list(zip(weights, w.split(ctx.sizes)))
            bias = None
            if biases[0] is not None:
                bias = torch.empty(sum(ctx.sizes), dtype=cd, device=x.device)
                convert += zip(biases, bias.split(ctx.sizes))
            if x2.dtype != cd:
                convert.append((x2, torch.empty(x2.shape, dtype=cd, device=x.device)))
                x2 = convert[-1][1]
            ops.convert_into(convert, cd)
            ctx.save_for_backward(x2, w)
            y = torch.nn.functional.linear(x2, w, bias)
            return tuple(part.view(x.shape[:-1] + (n,)) for part, n in zip(y.split(ctx.sizes, dim=1), ctx.sizes))
        x2 = x.reshape(-1, x.shape[-1]).to(cd)
        ws = [w.to(cd) for w in weights]
        ctx.save_for_backward(x2, *ws)
        outs = []
        for w, b in zip(ws, biases):
            y = torch.nn.functional.linear(x2, w, None if b is None else b.to(cd))
            outs.append(y.view(x.shape[:-1] + (w.shape[0],)))
        return tuple(outs)

    @staticmethod
    def backward(ctx, *gys):
        x2, *ws = ctx.saved_tensors
        shape, xdt = ctx.x_meta
        gys = [g.reshape(-1, g.shape[-1]).to(x2.dtype) for g in gys]
        if ctx.joint:
            gys = [_joined(gys, ctx.sizes)]
        gx = None
        if ctx.needs_input_grad[0]:
            # (with a second derivative to record, products that have one)
            if (ctx.joint and xdt == torch.float32 and x2.dtype in (torch.float16, torch.bfloat16)
                    and not torch.is_grad_enabled()):
                gx = torch.mm(gys[0], ws[0], out_dtype=torch.float32)
            else:
                gx = gys[0] @ ws[0]
                for g, w in zip(gys[1:], ws[1:]):
                    gx.addmm_(g, w)
            gx = gx.view(shape).to(xdt)
        column_sums = ops.column_sums
        if torch.is_grad_enabled():  # (likewise)
            def column_sums(g, sizes=None):
                total = g.sum(0, dtype=torch.promote_types(g.dtype, torch.float32))
                return total if sizes is None else total.split(sizes)
        want_w = [ctx.needs_input_grad[1 + 2 * i] for i in range(len(ctx.sizes))]
        want_b = [t is not None and ctx.needs_input_grad[2 + 2 * i] for i, t in enumerate(ctx.wb_dtypes[1::2])]
        if ctx.joint:
            gws = _of_column_blocks(lambda g, sizes: _weight_gradient(g, x2, sizes), gys[0], ctx.sizes, want_w)
            gbs = _of_column_blocks(column_sums, gys[0], ctx.sizes, want_b)
        else:
            gws = [_weight_gradient(g, x2) if want else None for g, want in zip(gys, want_w)]
            gbs = [column_sums(g) if want else None for g, want in zip(gys, want_b)]
        # (in memory of their own, each a gradient that is kept, saved or dropped by itself: blocks of a joint 16-bit product are
        # by their conversion, sums as they come but for recorded ones)
        convert = own if torch.is_grad_enabled() else torch.Tensor.to
        grads = [gx]
        for i in range(len(ctx.sizes)):
            grads.append(convert(gws[i], ctx.wb_dtypes[2 * i]) if want_w[i] else None)
            grads.append(convert(gbs[i], ctx.wb_dtypes[2 * i + 1]) if want_b[i] else None)
        return tuple(grads)


def linear_hooks_installed():
    """Whether hooks are registered for every module of the process."""
    m = torch.nn.modules.module
    return bool(getattr(m, "_global_forward_hooks", None) or getattr(m, "_global_forward_pre_hooks", None))


def _is_plain_linear(lin):
    """Whether calling the layer is nothing but x w^T + b with the parameters it holds: exactly torch.nn.Linear, no
    forward (pre-)hooks, no `forward` of its own on the instance (as offloading and casting wrappers put there) and no
    parametrization.  Adapters, quantised linears and hooked layers must be CALLED."""
    if type(lin) is not torch.nn.Linear or "forward" in lin.__dict__:
        return False
    if lin._forward_hooks or lin._forward_pre_hooks or getattr(lin, "_forward_hooks_with_kwargs", None):
        return False
    if linear_hooks_installed():
        return False
    return not torch.nn.utils.parametrize.is_parametrized(lin)


def project(x, *linears):
    """The outputs of the given nn.Linear layers on x: through `InputProjections` when every layer is a plain
    nn.Linear, else by calling the layers as the reference does (GPT_Trainer/GPTCosAttention.py:443-445), so that hooks,
    parametrizations and subclasses (LoRA adapters, quantised linears) keep their effect."""
    if not all(_is_plain_linear(lin) for lin in linears):
        return tuple(lin(x) for lin in linears)
    args = []
    for lin in linears:
        args += [lin.weight, lin.bias]
    return InputProjections.apply(x, *args)
