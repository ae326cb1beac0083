"""AutoFocusFormer classifier assembled around the CLUSTEN operators.

This is the build's own counterpart of models/aff_transformer.py, kept to what drives the three operators and
what an end-to-end images/s figure needs.  Parameter names and shapes equal the reference's, so a reference
`state_dict` loads unchanged.  What each class must reproduce:

  ClusterAttention  (aff_transformer.py:87-160)  q scaled by head_dim^-0.5 before QK; q/key/v handed to the
                    operators as permuted views of the Linear outputs; position bias, padding mask (-100),
                    blank token and softmax between QK and AV; dense branch when a stage attends globally.
  ClusterMerging    (aff_transformer.py:276-365) merge centres = top scores of grid prior + alpha * learned
                    score, reserve tokens on the coarse grid; weights (b, n', m, 4) = weight_net(table)[pe_idx] *
                    learned score * mask; WF output (b, n', 4, c) flattened so that channel = ic * c + c'.
  BasicLayer        (aff_transformer.py:441-507) balanced clusters, the nnc nearest clusters of every token, the
                    neighbourhood list = members of those clusters, nearest cluster first.

Differences from the reference, none of which change results: the relative-position table is a module buffer
instead of a module-level global; the neighbourhoods of the first stage, whose tokens sit on the image grid,
are computed once and reused (the reference caches the clustering but repeats the neighbour search); nearest
neighbours use a sort of exact distances instead of an external library; the operators are reached through
`self.ops`, so a test can run the very same modules on another implementation of the three functions.
"""
import functools
import math
import operator
import threading
from types import SimpleNamespace

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.nn.modules import module as _module

from .points import knn, space_filling_cluster


def default_ops():
    """The three operators as the HIP library provides them."""
    from clusten import CLUSTENAVFunction, CLUSTENQKFunction, CLUSTENWFFunction, _native
    return SimpleNamespace(qk=CLUSTENQKFunction.apply, av=CLUSTENAVFunction.apply, wf=CLUSTENWFFunction.apply,
                           attn_softmax=_native.attn_softmax, attn_softmax_supported=_native.attn_softmax_supported,
                           qk_clusters=_native.qk_forward_clusters, av_clusters=_native.av_forward_clusters,
                           clusters_supported=_native.clusters_supported,
                           cluster_attention=_native.cluster_attention,
                           cluster_attention_plan=_native.cluster_attention_plan,
                           cluster_attention_supported=_native.cluster_attention_supported,
                           cluster_attention_backward=_native.cluster_attention_backward,
                           cluster_attention_backward_supported=_native.cluster_attention_backward_supported,
                           cluster_pairs=_native.cluster_pairs, scatter_rows=_native.scatter_rows,
                           dense_attention_train=_native.dense_attention_train,
                           dense_attention=_native.dense_attention,
                           dense_attention_supported=_native.dense_attention_supported,
                           layer_norm_train=_native.layer_norm_train, layer_norm_backward=_native.layer_norm_backward,
                           layer_norm=_native.layer_norm, layer_norm_supported=_native.layer_norm_supported,
                           linear=_native.linear, linear_supported=_native.linear_supported,
                           add_layer_norm=_native.add_layer_norm, add_layer_norm_supported=_native.add_layer_norm_supported,
                           merge_weights=_native.merge_weights, merge_weights_supported=_native.merge_weights_supported,
                           merge_table=_native.merge_table, merge_table_backward=_native.merge_table_backward,
                           merge_table_supported=_native.merge_table_supported,
                           merge_weights_backward=_native.merge_weights_backward,
                           row_score=_native.row_score, row_score_backward=_native.row_score_backward,
                           row_score_supported=_native.row_score_supported,
                           channel_affine_gelu=_native.channel_affine_gelu,
                           channel_affine_gelu_supported=_native.channel_affine_gelu_supported,
                           add_row_score=_native.add_row_score, add_row_score_supported=_native.add_row_score_supported,
                           bias_table_grad=_native.bias_table_grad,
                           attn_softmax_backward=_native.attn_softmax_backward,
                           neighbour_lists=_native.neighbour_lists,
                           neighbour_lists_supported=_native.neighbour_lists_supported,
                           gather_rows=_native.gather_rows, gather_rows_supported=_native.gather_rows_supported,
                           merge_centres=_native.merge_centres, merge_centres_supported=_native.merge_centres_supported,
                           merge_rows=_native.merge_rows, merge_rows_supported=_native.merge_rows_supported,
                           block_pack=_native.block_pack, block_layout=_native.BlockLayout, block_supported=_native.block_supported,
                           norm_linear=_native.norm_linear, block_tail=_native.block_tail,
                           block_stands_for=(("linear", _native.linear), ("layer_norm", _native.layer_norm),
                                             ("add_layer_norm", _native.add_layer_norm)),
                           weight_grad=_native.weight_grad, weight_grad_supported=_native.weight_grad_supported,
                           block_tail_backward=_native.block_tail_backward, norm_linear_backward=_native.norm_linear_backward,
                           cluster_pairs_from_numbers=_native.cluster_pairs_from_numbers,
                           cluster_pairs_from_numbers_stands_for=(("cluster_pairs", _native.cluster_pairs),),
                           block_train_forward=_native.block_train_forward, block_train_backward=_native.block_train_backward,
                           block_train_supported=_native.block_train_supported,
                           block_train_stands_for=(("norm_linear", _native.norm_linear), ("block_tail", _native.block_tail),
                                                   ("cluster_attention", _native.cluster_attention),
                                                   ("cluster_attention_backward", _native.cluster_attention_backward),
                                                   ("norm_linear_backward", _native.norm_linear_backward),
                                                   ("block_tail_backward", _native.block_tail_backward),
                                                   ("scatter_rows", _native.scatter_rows), ("weight_grad", _native.weight_grad),
                                                   ("block_pack", _native.block_pack), ("bias_table_grad", _native.bias_table_grad)),
                           blocks_forward=_native.blocks_forward, block_params=_native.BlockParams,
                           blocks_stand_for=(("cluster_attention", _native.cluster_attention),
                                             ("dense_attention", _native.dense_attention),
                                             ("dense_attention_train", _native.dense_attention_train),
                                             ("norm_linear", _native.norm_linear), ("block_tail", _native.block_tail)))


def _types_of_forward(backward):
    """A `backward` that works in the types its forward kept, also when it is called under autocast (of another type, or after a
    forward without it): its products would come back in another type than the kernels behind them are given."""
    @functools.wraps(backward)
    def outside(ctx, *grads):
        if not torch.is_autocast_enabled("cuda"):
            return backward(ctx, *grads)
        with torch.autocast("cuda", enabled=False):
            return backward(ctx, *grads)
    return outside


def _by_kernels(*grads):
    """True when a backward pass may hand its incoming gradients to kernels: it is not itself recorded, and they are no batch of
    gradients (`is_grads_batched`), which has no memory to point at."""
    if torch.is_grad_enabled():
        return False
    try:
        for g in grads:
            g.data_ptr()
    except RuntimeError:
        return False
    return True


def _dense(t):
    """`t` as rows the kernels read in place: contiguous and from a 16-byte boundary on, as a gradient that is part of a larger
    buffer need not be."""
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


class _Linear(torch.autograd.Function):
    """`F.linear(x, weight, bias)` in x's dtype for parameters of any, with the parameters' gradients from the library's kernel:
    both in one pass over the rows, in fp32 (not rounded to 16 bits on the way to fp32 parameters)."""

    @staticmethod
    def forward(ctx, x, weight, bias, grad_kernel, supported):
        ctx.save_for_backward(x, weight)
        ctx.meta = (None if bias is None else bias.dtype, grad_kernel, supported)
        return F.linear(x, weight.to(x.dtype), None if bias is None else bias.to(x.dtype))

    @staticmethod
    def backward(ctx, d_y):
        x, weight = ctx.saved_tensors
        bias_dtype, grad_kernel, supported = ctx.meta
        need_x, need_w, need_b = ctx.needs_input_grad[:3]
        d_x = d_y @ weight.to(x.dtype) if need_x else None
        rows, x_rows = d_y.reshape(-1, d_y.shape[-1]), x.reshape(-1, x.shape[-1])
        if need_w and _by_kernels(d_y):
            if not supported(rows, x_rows):
                rows = rows.contiguous()                 # e.g. the gradient of a column range
            if supported(rows, x_rows):
                (d_w, d_b), = grad_kernel([(rows, x_rows, need_b)])
                return d_x, d_w.to(weight.dtype), None if d_b is None else d_b.to(bias_dtype), None, None
        return (d_x, (rows.t() @ x_rows).to(weight.dtype) if need_w else None, rows.sum(0).to(bias_dtype) if need_b else None,
                None, None)


def _hooked(mod):
    """True when calling `mod` runs more than its class' `forward`, or another one that was set on the module itself."""
    return bool("forward" in mod.__dict__ or mod._forward_hooks or mod._forward_pre_hooks or mod._backward_hooks or mod._backward_pre_hooks
                or _module._global_forward_hooks or _module._global_forward_pre_hooks or _module._global_backward_hooks
                or _module._global_backward_pre_hooks)


def _train_linear(lin, x, ops):
    """`lin(x)` of a training step: through `_Linear` for plain layers of a shape and type that the library's parameter
    gradients take."""
    w = lin.weight
    if (getattr(ops, "weight_grad", None) is None or not x.is_cuda or type(lin) is not nn.Linear or _hooked(lin) or _transformed()
            or not w.requires_grad or w.shape[0] % 8 or w.shape[1] % 8 or w.shape[0] * w.shape[1] >= 1 << 26 or x.numel() == 0):
        return lin(x)
    floats = (torch.float32, torch.float16, torch.bfloat16)
    dt = torch.get_autocast_dtype("cuda") if torch.is_autocast_enabled("cuda") else w.dtype
    if dt not in floats or x.dtype not in floats or w.dtype not in floats or (not torch.is_autocast_enabled("cuda") and x.dtype != dt):
        return lin(x)
    return _Linear.apply(x.to(dt), w, lin.bias, ops.weight_grad, ops.weight_grad_supported)


# .reads: what the `CapturedForward` being made by this thread has read so far; .parts: what was kept for the value being made
_thread = threading.local()


class _Kept:
    """What a module keeps between forwards under a key of addresses and versions.  `held` are the tensors behind these
    addresses: as long as they are held no other tensor can come to lie there.  Copies and pickles of the module start
    without it, as `value` may hold device addresses.

    A value is computed by the stream that was current then, and its memory belongs to that stream.  Another stream that
    takes it up waits for it first, and is noted in its memory's list of users, so that the memory is not handed out
    again before that stream is done."""

    __slots__ = ("key", "value", "held", "made", "stream", "ready", "streams")

    def __init__(self, key, value, held, made=None):
        self.key, self.value, self.held = key, value, held
        self.made = _tensors(value if made is None else made)
        self.stream = torch.cuda.current_stream(self.made[0].device) if self.made and self.made[0].is_cuda else None
        self.ready = None               # an event behind the computation; until there is one, the end of the stream
        self.streams = () if self.stream is None else (self.stream.cuda_stream,)

    def join(self):
        """Makes the value usable on the current stream."""
        if self.stream is None or torch._C._cuda_getCurrentRawStream(self.stream.device_index) in self.streams:
            return
        stream = torch.cuda.current_stream(self.stream.device)
        stream.wait_event(self.ready or self.stream.record_event())
        for t in self.made:
            t.record_stream(stream)
        self.streams += (stream.cuda_stream,)

    def __reduce__(self):
        return type(None), ()


def _tensors(value):
    """The tensors of a value: one, or a sequence that may hold other things as well."""
    return [t for t in (value if isinstance(value, (tuple, list)) else (value,)) if isinstance(t, torch.Tensor)]


def _kept(table, slot, key, make, lasting=False):
    """The `_Kept` in `table[slot]`, made by `make()` - (value, tensors to hold[, tensors computed for it, if they are not the
    value]) - when there is none under `key`.

    A recorded graph reads the addresses it was recorded with for as long as it is replayed, which a kept value does not
    outlive its key for.  `CapturedForward` holds what its recording reads; any other recording computes it again as a part of
    itself, but for what is `lasting` (never replaced while its owner lives).  What is made during a recording has no
    contents until the first replay, so it is not kept."""
    kept = table.get(slot)
    hit = type(kept) is _Kept and kept.key == key
    if torch.cuda.is_initialized() and torch.cuda.is_current_stream_capturing():
        reads = getattr(_thread, "reads", None)
        if not hit or not (lasting or reads is not None):
            return _Kept(key, *make())
        if reads is not None:
            reads.append(kept)
    elif hit:
        kept.join()
    else:
        outer, _thread.parts = getattr(_thread, "parts", None), []
        try:
            kept = _Kept(key, *make())
            parts = _thread.parts + [kept]
        finally:
            _thread.parts = outer
        if outer is not None:
            outer += parts                           # the event behind the whole will do for them: 10 us each
        elif kept.stream is not None:
            ready = kept.stream.record_event()
            for part in parts:
                part.ready = ready
        table[slot] = kept                           # in a module's __dict__: no parameter, no buffer, not in the state_dict
    return kept


_modules_of = operator.attrgetter("_modules")


class _Module(nn.Module):
    """A module that drops what it and the modules in it keep, and with it the old parameters it holds, when it is moved or converted."""

    def _apply(self, fn, recurse=True):
        for mod in self.modules():
            for slot in [name for name, value in mod.__dict__.items() if type(value) is _Kept]:
                del mod.__dict__[slot]
        return super()._apply(fn, recurse)


def _cast_params(lin, dt):
    """(weight, bias) of an nn.Linear in dtype `dt` as a `_Kept` value, remade when the parameters change."""
    weight, bias = lin.weight, lin.bias
    key = (dt, weight._version, weight.data_ptr(), None if bias is None else (bias._version, bias.data_ptr()))

    def make():
        held = [t.detach() for t in (weight, bias) if t is not None]
        return (held[0].to(dt), None if bias is None else held[1].to(dt)), held

    return _kept(lin.__dict__, "_cast_cache", key, make)


def _linear(lin, x, ops=None, gelu=False):
    """`lin(x)` for an nn.Linear, followed by the exact GELU when `gelu`.  In inference under mixed precision the
    16-bit copies of weight and bias are kept between calls (autocast makes them anew in every forward; they are
    remade when the parameters change), and the small layers on many rows go through the library's kernel when
    `ops` has it."""
    if torch.is_grad_enabled() or not x.is_cuda or not torch.is_autocast_enabled("cuda"):
        y = _train_linear(lin, x, ops) if torch.is_grad_enabled() else lin(x)
        return F.gelu(y) if gelu else y
    dt = torch.get_autocast_dtype("cuda")
    weight, bias = _cast_params(lin, dt).value
    x = x if x.dtype == dt else x.to(dt)
    fn = getattr(ops, "linear", None)
    if fn is not None and ops.linear_supported(x, weight, gelu):
        return fn(x, weight, bias, gelu)
    y = F.linear(x, weight, bias)
    return F.gelu(y) if gelu else y


def _linear_pair(first, second, x, ops=None):
    """`(first(x), second(x))` for two nn.Linear layers that read the same input (the query and the key / value
    projections of an attention layer, aff_transformer.py:103-106).  In inference under mixed precision they run as
    one matrix product over the stacked 16-bit weights, kept between calls like the single copies; the results are
    the two column ranges of its output (views).  Layers that the library's small-layer kernel takes stay apart."""
    if (torch.is_grad_enabled() or not x.is_cuda or not torch.is_autocast_enabled("cuda")
            or first.bias is None or second.bias is None):
        return _linear(first, x, ops), _linear(second, x, ops)
    dt = torch.get_autocast_dtype("cuda")
    kept = _cast_params(first, dt), _cast_params(second, dt)
    a, b = (k.value for k in kept)
    x = x if x.dtype == dt else x.to(dt)
    fn = getattr(ops, "linear", None)
    if fn is not None and ops.linear_supported(x, a[0], False) and ops.linear_supported(x, b[0], False):
        return fn(x, *a, False), fn(x, *b, False)
    weight, bias = _kept(first.__dict__, "_pair_cache", tuple(k.key for k in kept),
                         lambda: ((torch.cat([a[0], b[0]], 0), torch.cat([a[1], b[1]], 0)), kept)).value
    y = F.linear(x, weight, bias)
    n_first = a[0].shape[0]
    return y[..., :n_first], y[..., n_first:]


class _LayerNormRows(torch.autograd.Function):
    """`F.layer_norm(x.float(), ...)` returned as `out_dtype`, one pass over the rows a direction."""

    @staticmethod
    def forward(ctx, x, weight, bias, eps, out_dtype, ops):
        out, stats = ops.layer_norm_train(x, weight, bias, eps, out_dtype)
        ctx.save_for_backward(x, weight, bias, stats)
        ctx.meta = (eps, out_dtype, ops)
        return out

    @staticmethod
    @_types_of_forward
    def backward(ctx, d_y):
        x, weight, bias, stats = ctx.saved_tensors
        eps, out_dtype, ops = ctx.meta
        if not _by_kernels(d_y):
            return (*_recorded_backward(lambda x, w, b: F.layer_norm(x.float(), (x.shape[-1],), w, b, eps).to(out_dtype), ctx, (x, weight, bias),
                                        (d_y,)), None, None, None)
        grads = ops.layer_norm_backward(_dense(d_y), x, stats, weight)
        return (*(g if need else None for g, need in zip(grads, ctx.needs_input_grad)), None, None, None)


def _train_layer_norm(norm, x, ops, linear):
    """`norm(x)` of a training step by the library's kernels, or None where they do not stand for it."""
    w, b = norm.weight, norm.bias
    amp = torch.is_autocast_enabled("cuda")
    if (getattr(ops, "layer_norm_backward", None) is None or not x.is_cuda or type(norm) is not nn.LayerNorm or _hooked(norm) or _transformed()
            or not ops.layer_norm_supported(x) or not (x.dtype == torch.float32 or amp) or not 0 < x.numel() // x.shape[-1] < 1 << 31
            or tuple(norm.normalized_shape) != x.shape[-1:] or not (_kernel_parameter(w, x) and _kernel_parameter(b, x))):
        return None
    narrow = amp and type(linear) is nn.Linear and not _hooked(linear)
    out_dtype = torch.get_autocast_dtype("cuda") if narrow else torch.float32
    x = x.contiguous()
    if out_dtype not in (torch.float32, torch.float16, torch.bfloat16) or x.data_ptr() % 16 or (
            narrow and x.dtype not in (torch.float32, out_dtype)):
        return None
    return _LayerNormRows.apply(x, w, b, norm.eps, out_dtype, ops)


def _layer_norm(norm, x, ops, feeds_linear=False, linear=None):
    """`norm(x)` for an nn.LayerNorm; on the GPU through the library's one-pass kernels when `ops` has them.

    `feeds_linear`: the result is only read by Linear layers, so under mixed precision it is produced in the
    autocast dtype directly (the rounding those layers would apply to their input, done once); in training only for the one layer
    `linear` that reads it."""
    fn = getattr(ops, "layer_norm", None)
    if torch.is_grad_enabled():
        out = _train_layer_norm(norm, x, ops, linear)
        return norm(x) if out is None else out
    if fn is None or torch.is_grad_enabled() or not ops.layer_norm_supported(x):
        return norm(x)
    out_dtype = torch.get_autocast_dtype("cuda") if (feeds_linear and torch.is_autocast_enabled("cuda")) else None
    return fn(x, norm.weight, norm.bias, norm.eps, out_dtype)


def _one_pass_norm_available(ops, x):
    return (getattr(ops, "layer_norm", None) is not None and not torch.is_grad_enabled() and ops.layer_norm_supported(x))


def _add_layer_norm(norm, x, branch, ops):
    """(x + branch, norm(x + branch)) — just (x, norm(x)) when `branch` is None — with the norm's output feeding
    Linear layers only.  In inference under mixed precision addition and norm are one pass of the library's kernel
    when `ops` has it."""
    if branch is None:
        return x, _layer_norm(norm, x, ops, True)
    fn = getattr(ops, "add_layer_norm", None)
    if (fn is not None and not torch.is_grad_enabled() and torch.is_autocast_enabled("cuda")
            and branch.dtype == torch.get_autocast_dtype("cuda") and ops.add_layer_norm_supported(x, branch)):
        return fn(x, branch, norm.weight, norm.bias, norm.eps)
    x = x + branch
    return x, _layer_norm(norm, x, ops, True)


def _table_rows(table, idx):
    """table[idx] for a (rows, k) table and an index tensor of any shape, written as the reference writes it
    (aff_transformer.py:131: a `gather` along dim 0): the values are those of `table[idx]`, but the backward is a
    scatter-add, where the framework's backward of advanced indexing sorts the indices (19 ms per attention layer at
    batch 64 on this device: nine tenths of a training step)."""
    k = table.shape[1]
    return table.gather(0, idx.reshape(-1, 1).expand(-1, k)).reshape(*idx.shape, k)


class _PositionBias(torch.autograd.Function):
    """bias[pe_idx] laid out as (b, h, n, m), with the table's gradient from the library's kernel (sums per workgroup
    in LDS) instead of the framework's scatter-add of b*h*n*m values into a table of 12 000 rows."""

    @staticmethod
    def forward(ctx, bias, pe_idx, grad_kernel):
        ctx.save_for_backward(pe_idx)
        ctx.rows, ctx.dtype, ctx.grad_kernel = bias.shape[0], bias.dtype, grad_kernel
        return _table_rows(bias, pe_idx).permute(0, 3, 1, 2)

    @staticmethod
    def backward(ctx, grad):
        (pe_idx,) = ctx.saved_tensors
        if not _by_kernels(grad):
            rows = grad.permute(0, 2, 3, 1).reshape(-1, grad.shape[1])
            table = torch.zeros(ctx.rows, grad.shape[1], dtype=torch.float32, device=grad.device)
            return table.scatter_add(0, pe_idx.reshape(-1, 1).expand(-1, grad.shape[1]), rows.float()).to(ctx.dtype), None, None
        return ctx.grad_kernel(grad, pe_idx, ctx.rows).to(ctx.dtype), None, None


class _AttnSoftmax(torch.autograd.Function):
    """Position bias, padding mask, blank token and softmax between QK and AV as one kernel forward and one backward
    (aff_transformer.py:125-147), with the bias table's gradient from `bias_table_grad`: the training counterpart of
    the inference path's `attn_softmax`."""

    @staticmethod
    def forward(ctx, attn, bias, pe_idx, mask, blank_logit, ops):
        probs, blank_prob = ops.attn_softmax(attn, bias, pe_idx, mask, blank_logit=blank_logit)
        ctx.save_for_backward(probs, blank_prob, pe_idx)
        ctx.meta = (attn.dtype, bias.shape[0], bias.dtype, blank_logit.dtype, ops)
        return probs, blank_prob

    @staticmethod
    def backward(ctx, d_probs, d_blank_prob):
        probs, blank_prob, pe_idx = ctx.saved_tensors
        attn_dtype, rows, bias_dtype, blank_dtype, ops = ctx.meta
        d_logit, d_blank = ops.attn_softmax_backward(probs, blank_prob, d_probs, d_blank_prob, attn_dtype)
        d_bias = ops.bias_table_grad(d_logit, pe_idx, rows).to(bias_dtype)
        return d_logit, d_bias, None, None, d_blank.to(blank_dtype), None


def _recorded_backward(fn, ctx, tensors, grads, needs=None):
    """The gradients of `fn(*tensors)` by recorded operations, for a backward pass that is itself differentiated or batched.  `needs`: of
    `tensors`, when they are not the first inputs."""
    needs = ctx.needs_input_grad[:len(tensors)] if needs is None else needs
    with torch.enable_grad(), torch.autocast("cuda", enabled=False):
        out = fn(*tensors)
        out, grads = zip(*((o, g) for o, g in zip(out if isinstance(out, tuple) else (out,), grads) if o.requires_grad))
        wanted = torch.autograd.grad(out, [t for t, need in zip(tensors, needs) if need], grads, create_graph=True, allow_unused=True)
    wanted = iter(wanted)
    return [next(wanted) if need else None for need in needs]


def _local_attention(q, key, v, bias, blank_k, blank_v, mask, pe_idx, member_idx, scale):
    """The local attention of a block in recorded operations, fp32 inside: what the kernel computes (aff_transformer.py:120-155)."""
    b, h, n, ch = q.shape
    m = member_idx.shape[-1]
    rows = member_idx.reshape(b, 1, n * m, 1).expand(-1, h, -1, ch)
    dtype = q.dtype
    q, key, v, bias, blank_k, blank_v = (t.float() for t in (q, key, v, bias, blank_k.reshape(1, h, 1, ch), blank_v.reshape(1, h, 1, ch)))
    logits = (q.unsqueeze(3) * key.gather(2, rows).view(b, h, n, m, ch)).sum(-1) * scale + _table_rows(bias, pe_idx).permute(0, 3, 1, 2)
    if mask is not None:
        logits = logits + (1 - mask.reshape(b, 1, n, m)) * (-100)
    probs = torch.softmax(torch.cat([logits, (q * blank_k).sum(-1, keepdim=True) * scale], dim=-1), dim=-1)
    out = (probs[..., :-1, None] * v.gather(2, rows).view(b, h, n, m, ch)).sum(3) + probs[..., -1:] * blank_v
    return out.permute(0, 2, 1, 3).reshape(b, n, h * ch).to(dtype)


class _ClusterAttention(torch.autograd.Function):
    """The local attention of a block between its projections (aff_transformer.py:120-155) as one kernel forward and,
    backward, one kernel for the query side - the probabilities are recomputed from the softmax denominators the
    forward saved - followed by the sums that complete it: the scatters over the stage's sorted pair lists (d_key,
    d_value), the bias table's gradient, the blank token's.  No (b,h,n,m) tensor is kept between the two passes.
    The scatters go through the operators' own scatter, which reads the flag of the pair lists on the device: lists
    that turn out not to be made of whole clusters (never the model's own) take its atomic kernels, so d_key and d_value
    are complete sums whatever `member_idx` holds."""

    @staticmethod
    def forward(ctx, q, key, v, bias, blank_k, blank_v, plan, pairs, pe_idx, member_idx, mask, scale, ops):
        out, lse = ops.cluster_attention(q, key, v, None, bias, None, None, blank_k, blank_v, scale=scale, plan=plan,
                                         return_lse=True)
        ctx.save_for_backward(q, key, v, out, lse, bias, blank_k, blank_v, plan, pairs, pe_idx, member_idx, mask)
        ctx.meta = (scale, ops)
        return out

    @staticmethod
    @_types_of_forward
    def backward(ctx, d_out):
        q, key, v, out, lse, bias, blank_k, blank_v, plan, pairs, pe_idx, member_idx, mask = ctx.saved_tensors
        scale, ops = ctx.meta
        if not _by_kernels(d_out):
            return (*_recorded_backward(lambda *t: _local_attention(*t, mask, pe_idx, member_idx, scale), ctx,
                                        (q, key, v, bias, blank_k, blank_v), (d_out,)), *(None,) * 7)
        b, h, n, ch = q.shape
        d_q, probs, d_logit, blank_prob, d_blank = ops.cluster_attention_backward(
            q, key, v, d_out, out, lse, plan, bias, blank_k, blank_v, scale=scale)
        g = d_out.to(q.dtype).reshape(b, n, h, ch).permute(0, 2, 1, 3)
        d_v = ops.scatter_rows(probs, g, member_idx, pairs)
        d_k = ops.scatter_rows(d_logit, q, member_idx, pairs) * scale
        d_bias = ops.bias_table_grad(d_logit, pe_idx, bias.shape[0]).to(bias.dtype)
        d_bk = torch.einsum("bhn,bhnc->hc", d_blank, q.float()) * scale
        d_bv = torch.einsum("bhn,bhnc->hc", blank_prob, g.float())
        return (d_q, d_k.to(key.dtype), d_v.to(v.dtype), d_bias, d_bk.reshape(blank_k.shape).to(blank_k.dtype),
                d_bv.reshape(blank_v.shape).to(blank_v.dtype), *(None,) * 7)


class _NormLinearRows(torch.autograd.Function):
    """`norm1` and the q / kv projections of a block as the inference kernel computes them, keeping the norm's result and
    statistics.  Also hands x through: its other use is the residual addition, whose gradient then meets the norm's inside
    the norm's backward kernel."""

    @staticmethod
    def forward(ctx, x, norm_w, norm_b, w_q, b_q, w_kv, b_kv, eps, dt, ops):
        c = x.shape[-1]
        # packed in every forward, not kept: the weights of a training step are new ones
        packed, at = ops.block_pack(c, dt, [(w_q, False), (w_kv, False), (w_q, True), (w_kv, True)])
        qkv, normed, stats = ops.norm_linear(x, norm_w, norm_b, eps, packed, at[0], b_q, b_kv, 3 * c, keep=True)
        ctx.save_for_backward(x, norm_w, norm_b, w_q, b_q, w_kv, b_kv, normed, stats, packed)
        ctx.meta = (eps, dt, ops, at[2:])
        return qkv, x

    @staticmethod
    @_types_of_forward
    def backward(ctx, d_qkv, d_res):
        x, norm_w, norm_b, w_q, b_q, w_kv, b_kv, normed, stats, packed = ctx.saved_tensors
        eps, dt, ops, at = ctx.meta
        c = x.shape[-1]
        if not _by_kernels(d_qkv, d_res):
            def layers(x, norm_w, norm_b, w_q, b_q, w_kv, b_kv):
                y = F.layer_norm(x.float(), (c,), norm_w, norm_b, eps).to(dt)
                return F.linear(y, torch.cat([w_q, w_kv]).to(dt), torch.cat([b_q, b_kv]).to(dt)), x
            return (*_recorded_backward(layers, ctx, (x, norm_w, norm_b, w_q, b_q, w_kv, b_kv), (d_qkv, d_res)), None, None, None)
        need = ctx.needs_input_grad
        rows = _dense(d_qkv).view(-1, 3 * c)
        flat = normed.view(-1, c)
        grads = [None] * 7
        if need[0] or need[1] or need[2]:
            grads[0], grads[1], grads[2] = ops.norm_linear_backward(rows, x, stats, norm_w, packed, at, _dense(d_res))
        wanted = [(i, rows[:, cols], need[i + 1]) for i, cols in ((3, slice(0, c)), (5, slice(c, 3 * c))) if need[i] or need[i + 1]]
        if wanted:
            for (i, _, _), (grads[i], grads[i + 1]) in zip(wanted, ops.weight_grad([(d, flat, bias) for _, d, bias in wanted])):
                pass
        return (*(g if n else None for g, n in zip(grads, need)), None, None, None)


class _BlockTail(torch.autograd.Function):
    """A block behind its attention as the inference kernel computes it, keeping the rows between its two branches, their
    norm and the hidden layer.  `scale`: (2, b) factors of stochastic depth, or None."""

    @staticmethod
    def forward(ctx, attn, x, w_p, b_p, norm_w, norm_b, w_1, b_1, w_2, b_2, scale, eps, dt, ops):
        weights = (w_p, w_1, w_2)
        packed, at = ops.block_pack(x.shape[-1], dt, [(w, False) for w in weights] + [(w, True) for w in weights])
        out, x1, normed, hidden, stats = ops.block_tail(attn, x, packed, at, b_p, norm_w, norm_b, eps, b_1, b_2, scale, keep=True)
        ctx.save_for_backward(attn, x, w_p, b_p, norm_w, norm_b, w_1, b_1, w_2, b_2, scale, x1, normed, hidden, stats, packed)
        ctx.meta = (eps, dt, ops, at[3:])
        return out

    @staticmethod
    @_types_of_forward
    def backward(ctx, d_out):
        attn, x, w_p, b_p, norm_w, norm_b, w_1, b_1, w_2, b_2, scale, x1, normed, hidden, stats, packed = ctx.saved_tensors
        eps, dt, ops, at = ctx.meta
        b, c, h = x.shape[0], x.shape[-1], hidden.shape[-1]
        if not _by_kernels(d_out):
            def layers(attn, x, w_p, b_p, norm_w, norm_b, w_1, b_1, w_2, b_2):
                s = (1.0, 1.0) if scale is None else scale.to(dt).view(2, b, *(1,) * (x.dim() - 1))
                x1 = x + (F.linear(attn, w_p.to(dt), b_p.to(dt)) * s[0]).to(x.dtype)
                y = F.layer_norm(x1.float(), (c,), norm_w, norm_b, eps).to(dt)
                y = F.gelu(F.linear(y, w_1.to(dt), b_1.to(dt)))
                return x1 + (F.linear(y, w_2.to(dt), b_2.to(dt)) * s[1]).to(x.dtype)
            return (*_recorded_backward(layers, ctx, (attn, x, w_p, b_p, norm_w, norm_b, w_1, b_1, w_2, b_2), (d_out,)),
                    None, None, None, None)
        need = ctx.needs_input_grad
        grads = [None] * 10
        grads[1], branch, d_f, g, d_h, grads[0], grads[4], grads[5] = ops.block_tail_backward(_dense(d_out), x1, stats, norm_w, hidden,
                                                                                              packed, at, scale)
        branch, d_f, g, d_h = branch.view(-1, c), d_f.view(-1, c), g.view(-1, h), d_h.view(-1, h)
        wanted = [(i, d, y, need[i + 1]) for i, d, y in ((2, branch, attn.view(-1, c)), (6, d_h, normed.view(-1, c)), (8, d_f, g))
                  if need[i] or need[i + 1]]
        if wanted:
            for (i, *_), (grads[i], grads[i + 1]) in zip(wanted, ops.weight_grad([item[1:] for item in wanted])):
                pass
        return (*(t if n else None for t, n in zip(grads, need)), None, None, None, None)


class _BlockRows(torch.autograd.Function):
    """A whole block in training by one native call a direction: norm and projections, attention with the position bias' layer inside, and
    everything behind it, as the inference kernels compute them; what the backward reads is one block of memory.  `params`: as
    `ClusterTransformerBlock.tensors` gives them.  `plan` and `pairs` of a local attention, else None; `member_idx` and `mask` are read only
    by a backward that is itself recorded."""

    @staticmethod
    def forward(ctx, x, table, pe_idx, plan, pairs, factors, member_idx, mask, dt, heads, hidden, eps, scale, ops, *params):
        out, kept = ops.block_train_forward(x, params, table, pe_idx, plan, pairs, factors, dt, heads, hidden, eps, scale)
        ctx.save_for_backward(x, table, pe_idx, plan, pairs, factors, member_idx, mask, kept, *params)
        ctx.meta = (dt, heads, hidden, eps, scale, ops)
        return out

    @staticmethod
    @_types_of_forward
    def backward(ctx, d_out):
        x, table, pe_idx, plan, pairs, factors, member_idx, mask, kept, *params = ctx.saved_tensors
        dt, heads, hidden, eps, scale, ops = ctx.meta
        need = ctx.needs_input_grad
        if not _by_kernels(d_out):
            b, n, c = x.shape
            everyone = torch.arange(n, device=x.device).expand(b, n, n) if plan is None else member_idx
            t = table.to(dt)

            def layers(x, n1_w, n1_b, n2_w, n2_b, b_q, b_kv, b_p, b_1, b_2, blank_k, blank_v, w_q, w_kv, w_p, w_1, w_2, pe_w, pe_b):
                s = (1.0, 1.0) if factors is None else factors.to(dt).view(2, b, 1, 1)
                y = F.layer_norm(x.float(), (c,), n1_w, n1_b, eps[0]).to(dt)
                qkv = F.linear(y, torch.cat([w_q, w_kv]).to(dt), torch.cat([b_q, b_kv]).to(dt))
                a = _local_attention(*_columns(qkv, heads), F.linear(t, pe_w.to(dt), pe_b.to(dt)), blank_k, blank_v,
                                     None if plan is None else mask, pe_idx, everyone, scale)
                x1 = x + (F.linear(a, w_p.to(dt), b_p.to(dt)) * s[0]).to(x.dtype)
                y = F.gelu(F.linear(F.layer_norm(x1.float(), (c,), n2_w, n2_b, eps[1]).to(dt), w_1.to(dt), b_1.to(dt)))
                return x1 + (F.linear(y, w_2.to(dt), b_2.to(dt)) * s[1]).to(x.dtype)

            d_x, *grads = _recorded_backward(layers, ctx, (x, *params), (d_out,), need[:1] + need[14:])
        else:
            d_x, grads = ops.block_train_backward(_dense(d_out), kept, need[14:], x, params, table, pe_idx, plan, pairs, factors, dt, heads, hidden,
                                                  eps, scale)
        return (d_x if need[0] else None, *(None,) * 13, *(g if n else None for g, n in zip(grads, need[14:])))


class _ClusterAttentionRows(_BlockRows):
    """A block whose tokens attend to the members of their nearest clusters."""


class _DenseAttentionRows(_BlockRows):
    """A block whose tokens attend to all."""


class _MergeTable(torch.autograd.Function):
    """A merge's weight of every relative position - Linear, norm and GELU over the table - by one kernel a direction."""

    @staticmethod
    def forward(ctx, table, weight, bias, norm_w, norm_b, eps, dt, ops):
        ctx.save_for_backward(table, weight, bias, norm_w, norm_b)
        ctx.meta = (eps, dt, ops)
        return ops.merge_table(table, weight, bias, norm_w, norm_b, eps, dt)

    @staticmethod
    @_types_of_forward
    def backward(ctx, d_out):
        table, *params = ctx.saved_tensors
        eps, dt, ops = ctx.meta
        if not _by_kernels(d_out):
            def layers(w, b, norm_w, norm_b):
                return F.gelu(F.layer_norm(F.linear(table.to(dt), w.to(dt), b.to(dt)).float(), (4,), norm_w, norm_b, eps))
            return (None, *_recorded_backward(layers, ctx, params, (d_out,), ctx.needs_input_grad[1:5]), None, None, None)
        grads = ops.merge_table_backward(_dense(d_out), table, *params, eps, dt)
        return (None, *(g if need else None for g, need in zip(grads, ctx.needs_input_grad[1:5])), None, None, None)


def _weight_table(net, table, ops):
    """`net(table)` for a merge's weight net."""
    if (torch.is_grad_enabled() and getattr(ops, "merge_table_backward", None) is not None and table.is_cuda and not table.requires_grad
            and type(net) is nn.Sequential and tuple(map(type, net)) == (nn.Linear, nn.LayerNorm, nn.GELU) and net[2].approximate == "none"
            and not any(map(_hooked, (net, *net))) and not _transformed()):
        params = (net[0].weight, net[0].bias, net[1].weight, net[1].bias)
        dt = torch.get_autocast_dtype("cuda") if torch.is_autocast_enabled("cuda") else torch.float32
        if all(p is not None for p in params) and tuple(net[1].normalized_shape) == (4,) and ops.merge_table_supported(table, *params, dt):
            return _MergeTable.apply(table, *params, net[1].eps, dt, ops)
    return net(table)


class _MergeWeights(torch.autograd.Function):
    """The weights a merge's WF operator takes - table rows by position, times importance, times mask - with both gradients from
    the library's kernels; fp32."""

    @staticmethod
    def forward(ctx, table_w, prob, pe_idx, member_idx, mask, ops):
        ctx.save_for_backward(table_w, prob, pe_idx, member_idx, mask)
        ctx.ops = ops
        return ops.merge_weights(table_w, pe_idx, member_idx, prob, mask)

    @staticmethod
    @_types_of_forward
    def backward(ctx, d_w):
        table_w, prob, pe_idx, member_idx, mask = ctx.saved_tensors
        if not _by_kernels(d_w):
            b, n_out, m = pe_idx.shape

            def layers(table_w, prob):
                weights = _table_rows(table_w, pe_idx) * prob.gather(1, member_idx.reshape(b, -1)).reshape(b, n_out, m, 1)
                return weights if mask is None else weights * mask.unsqueeze(3)
            return (*_recorded_backward(layers, ctx, (table_w, prob), (d_w,)), None, None, None, None)
        d_table, d_prob = ctx.ops.merge_weights_backward(d_w, table_w, pe_idx, member_idx, prob, mask)
        return d_table, d_prob, None, None, None, None


class _RowScore(torch.autograd.Function):
    """`sigmoid(linear(x))` of a layer of one output, one pass over the rows a direction."""

    @staticmethod
    def forward(ctx, x, weight, bias, dt, ops):
        score = ops.row_score(x, weight, bias, dt)
        ctx.save_for_backward(x, weight, bias, score)
        ctx.meta = (dt, ops)
        return score

    @staticmethod
    @_types_of_forward
    def backward(ctx, d_score):
        x, weight, bias, score = ctx.saved_tensors
        dt, ops = ctx.meta
        if not _by_kernels(d_score):
            return (*_recorded_backward(lambda x, w, b: F.linear(x.to(dt), w.to(dt), b.to(dt)).sigmoid(), ctx, (x, weight, bias), (d_score,)),
                    None, None)
        d_x, d_w, d_b = ops.row_score_backward(x, weight, score, d_score.contiguous())
        return (*(g if need else None for g, need in zip((d_x, d_w.view(weight.shape), d_b.view(bias.shape)), ctx.needs_input_grad)), None, None)


def _score(lin, x, ops):
    """`lin(x).sigmoid()` for a layer of one output."""
    if torch.is_grad_enabled() and getattr(ops, "row_score_backward", None) is not None and x.is_cuda:
        w, b = lin.weight, lin.bias
        dt = torch.get_autocast_dtype("cuda") if torch.is_autocast_enabled("cuda") else torch.float32
        if (type(lin) is nn.Linear and w is not None and w.shape[0] == 1 and b is not None and b.dtype == torch.float32 and not _hooked(lin)
                and not _transformed() and b.device == x.device and ops.row_score_supported(x, w, dt)):
            return _RowScore.apply(x, w, b, dt, ops)
    return _linear(lin, x).sigmoid()


def _columns(qkv, heads):
    """(q, key, v), each (b,h,n,ch), of (b,n,3c) rows of stacked projections (views)."""
    b, n, c3 = qkv.shape
    c = c3 // 3
    q = qkv[..., :c].view(b, n, heads, c // heads).permute(0, 2, 1, 3)
    kv = qkv[..., c:].view(b, n, heads, 2, c // heads)
    return q, kv[:, :, :, 0].permute(0, 2, 1, 3), kv[:, :, :, 1].permute(0, 2, 1, 3)


def _transformed():
    """True under forward-mode differentiation or a function transform (vmap, jvp, ...), which a custom Function without
    rules for them does not take."""
    return torch.autograd.forward_ad._current_level >= 0 or torch._C._functorch.peek_interpreter_stack() is not None


def _position_bias(bias, pe_idx, ops):
    """(b, h, n, m) position bias of an attention layer: row pe_idx[b,i,j] of the (rows, h) table for every pair."""
    kernel = getattr(ops, "bias_table_grad", None)
    if (kernel is not None and torch.is_grad_enabled() and bias.requires_grad and bias.is_cuda
            and bias.dtype in (torch.float32, torch.float16, torch.bfloat16)):
        return _PositionBias.apply(bias, pe_idx, kernel)
    return _table_rows(bias, pe_idx).permute(0, 3, 1, 2)


def _autocast_key():
    return torch.get_autocast_dtype("cuda") if torch.is_autocast_enabled("cuda") else None


def _table_function(owner, slot, module, table, compute):
    """`compute()`, a function of `module`'s parameters and of the relative-position table only, kept between
    inference forwards: the position-bias table of an attention layer and the weight table of a merge are the same
    for every batch.  Recomputed when a parameter or the table changes (in place or by replacement) or the autocast
    state does; never kept while gradients are enabled."""
    if torch.is_grad_enabled() or not table.is_cuda:
        return compute()
    key = (tuple((q.data_ptr(), q._version) for q in module.parameters()), table.data_ptr(), table._version, table.dtype,
           _autocast_key())
    return _kept(owner.__dict__, slot, key, lambda: (compute(), [table] + [q.detach() for q in module.parameters()])).value


def relative_position_table(img_size):
    """(table_width^2, 5) rows (dx, dy, distance, sin, cos) for every offset between two stride-4 tokens.

    aff_transformer.py:14-33: offsets range over [-R, R] with R = img_size // 4 - 1; the row of offset (dx, dy)
    is (dy + R) * (2R + 1) + (dx + R); the undefined angle at the origin is 0.
    """
    r = img_size // 4 - 1
    axis = torch.arange(2 * r + 1).float() - r
    dy, dx = torch.meshgrid(axis, axis, indexing="ij")
    dist = (dx ** 2 + dy ** 2) ** 0.5
    table = torch.stack([dx, dy, dist, dy / dist, dx / dist], dim=2)
    table[~torch.isfinite(table)] = 0
    return table.reshape(-1, 5), r


class DropPath(nn.Module):
    """Stochastic depth: drops the whole residual branch of a sample with probability p while training."""

    def __init__(self, p):
        super().__init__()
        self.p = float(p)

    def forward(self, x):
        if not self.training or self.p == 0.0:
            return x
        return x * self.factors(x.shape[0], x.dtype, x.device).view((-1,) + (1,) * (x.dim() - 1))

    def factors(self, samples, dtype, device):
        """The factor of every sample: 0 with probability p, else 1 / (1 - p)."""
        keep = 1.0 - self.p
        return torch.empty(samples, dtype=dtype, device=device).bernoulli_(keep).div_(keep)


def _drops(mod):
    """True for a Dropout or DropPath that drops: by its own mode, which need not be that of the layer it is in."""
    return mod.training and type(mod) is not nn.Identity and mod.p > 0


class Mlp(_Module):
    def __init__(self, dim, hidden, drop=0.0, ops=None):
        super().__init__()
        self.fc1 = nn.Linear(dim, hidden)
        self.act = nn.GELU()
        self.fc2 = nn.Linear(hidden, dim)
        self.drop = nn.Dropout(drop)
        self.ops = ops

    def forward(self, x):
        hidden = _linear(self.fc1, x, self.ops, gelu=True)        # self.act is the exact GELU
        return self.drop(_linear(self.fc2, self.drop(hidden), self.ops))


class ClusterAttention(_Module):
    """Attention of every token over the members of its nearest clusters, plus one learned blank token."""

    def __init__(self, dim, num_heads, attn_drop=0.0, proj_drop=0.0, ops=None):
        super().__init__()
        self.dim, self.num_heads = dim, num_heads
        self.scale = (dim // num_heads) ** -0.5
        self.q = nn.Linear(dim, dim)
        self.kv = nn.Linear(dim, 2 * dim)
        self.blank_k = nn.Parameter(torch.randn(dim))
        self.blank_v = nn.Parameter(torch.randn(dim))
        self.pos_embed = nn.Linear(5, num_heads)
        self.attn_drop = nn.Dropout(attn_drop)
        self.proj = nn.Linear(dim, dim)
        self.proj_drop = nn.Dropout(proj_drop)
        self.ops = ops
        self.cluster_size = 8     # tokens per cluster of the lists this layer is given (its stage sets it)

    def bias_table(self, table):
        """(rows, heads) position bias for every row of the relative-position table (aff_transformer.py:125-129)."""
        return _table_function(self, "_bias_table_cache", self.pos_embed, table, lambda: _linear(self.pos_embed, table))

    def forward(self, feat, member_idx, cluster_mask, pe_idx, global_attn, table, cluster_idx=None, grid_lists=None):
        """`grid_lists`: (cluster_idx, pe_idx, cluster_mask) with a leading 1 instead of the batch size, when the
        lists are the same for every image (tokens of a regular grid); the one-kernel path reads those."""
        q, kv = _linear_pair(self.q, self.kv, feat, self.ops)
        out = self.attend(q, kv, member_idx, cluster_mask, pe_idx, global_attn, table, cluster_idx, grid_lists)
        return self.proj_drop(_linear(self.proj, out, self.ops))

    def _trains_in_one_kernel(self, q, global_attn, cluster_idx, grid_lists):
        """True when the layer's training pass is the one-kernel attention; q: (b,n,c) rows of the queries."""
        b, n, c = q.shape
        h = self.num_heads
        return (getattr(self.ops, "cluster_attention_backward", None) is not None and torch.is_grad_enabled()
                and cluster_idx is not None and not global_attn and self.cluster_size == 8 and grid_lists is not None
                and len(grid_lists) > 4 and not _drops(self.attn_drop)
                and self.ops.cluster_attention_backward_supported(q.view(b, n, h, c // h).permute(0, 2, 1, 3), cluster_idx.shape[2]))

    def _attend_to_all(self, q, kv, pe_idx, table):
        """`attend` of an fp32 inference pass over all tokens by one kernel, or None where it is not built for the call."""
        rows_op = getattr(self.ops, "dense_attention_train", None)
        b, n, c = q.shape
        if (rows_op is None or _drops(self.attn_drop) or _transformed() or c != 32 * self.num_heads or not 0 < n <= 64 or b == 0
                or kv.dtype != q.dtype or pe_idx.shape != (b, n, n) or pe_idx.dtype != torch.int64
                or not all(_kernel_parameter(t, q) and t.numel() == c for t in (self.blank_k, self.blank_v))):
            return None
        bias = self.bias_table(table)
        if bias.dtype != torch.float32:
            return None
        one = q.stride() == kv.stride() == (n * 3 * c, 3 * c, 1) and kv.data_ptr() == q.data_ptr() + 4 * c and q.data_ptr() % 16 == 0
        qkv = q.as_strided((b, n, 3 * c), (n * 3 * c, 3 * c, 1)) if one else torch.cat([q, kv], dim=2)
        return rows_op(qkv.detach(), bias.detach().t().contiguous(), pe_idx.contiguous(), self.blank_k.detach(), self.blank_v.detach(),
                       self.num_heads, self.scale)

    def attend(self, q, kv, member_idx, cluster_mask, pe_idx, global_attn, table, cluster_idx=None, grid_lists=None):
        """The attention between its projections: q (b,n,c) and kv (b,n,2c) in, what the output projection reads (b,n,c)
        out.  The query is not scaled yet; q and kv may be column ranges of one matrix."""
        b, n, c = q.shape
        h = self.num_heads
        ch = c // h
        # inference: the neighbourhoods as (b,n,nnc) cluster numbers instead of the expanded (b,n,m*nnc) row lists
        numbered = cluster_idx is not None and not global_attn and not torch.is_grad_enabled()
        compact = numbered and getattr(self.ops, "qk_clusters", None) is not None
        sized = {} if self.cluster_size == 8 else {"cluster_size": self.cluster_size}
        key, v = kv.view(b, n, h, 2, ch).permute(3, 0, 2, 1, 4).unbind(0)                                   # (b,h,n,ch) views
        one_kernel = getattr(self.ops, "cluster_attention", None)
        if (numbered and one_kernel is not None and not _drops(self.attn_drop)
                and self.ops.cluster_attention_supported(q.view(b, n, h, ch).permute(0, 2, 1, 3), cluster_idx.shape[2],
                                                         self.cluster_size)):
            # inference on 16-bit or fp32 data: scores, position bias, mask, blank token, softmax and the weighted sum
            # of the values in one kernel; the query scale is applied to the scores inside it
            lists = grid_lists if grid_lists is not None else (cluster_idx, pe_idx, cluster_mask)
            plan = lists[3] if len(lists) > 3 else None     # what the kernel makes of the lists, once per stage
            out = one_kernel(q.view(b, n, h, ch).permute(0, 2, 1, 3), key, v, lists[0], self.bias_table(table),
                             lists[1], lists[2], self.blank_k, self.blank_v, scale=self.scale,
                             **({"plan": plan} if plan is not None else {}))
            return out
        if self._trains_in_one_kernel(q, global_attn, cluster_idx, grid_lists):
            # training: the same kernel forward, one kernel and four sums backward
            bias = self.bias_table(table)
            out = _ClusterAttention.apply(q.view(b, n, h, ch).permute(0, 2, 1, 3), key, v, bias, self.blank_k,
                                          self.blank_v, grid_lists[3], grid_lists[4], pe_idx, member_idx,
                                          cluster_mask, self.scale, self.ops)
            return out
        dense = getattr(self.ops, "dense_attention", None)
        if (global_attn and dense is not None and not torch.is_grad_enabled()
                and not _drops(self.attn_drop)
                and self.ops.dense_attention_supported(q.view(b, n, h, ch).permute(0, 2, 1, 3))):
            # inference on 16-bit data, every token attending to every token: one kernel as well
            out = dense(q.view(b, n, h, ch).permute(0, 2, 1, 3), key, v, self.bias_table(table), pe_idx,
                        self.blank_k, self.blank_v, scale=self.scale)
            return out
        if global_attn and q.dtype == torch.float32 and not torch.is_grad_enabled() and q.is_cuda:
            out = self._attend_to_all(q, kv, pe_idx, table)
            if out is not None:
                return out
        q = (q * self.scale).reshape(b, n, h, ch).permute(0, 2, 1, 3)                    # (b,h,n,ch) view
        if global_attn:
            attn = q @ key.transpose(-1, -2)                                             # (b,h,n,n)
        elif compact and self.ops.clusters_supported(q, cluster_idx.shape[2], **sized):
            attn = self.ops.qk_clusters(q, key, cluster_idx, **sized)                    # (b,h,n,m)
        else:
            compact = False
            attn = self.ops.qk(q, key, member_idx)                                       # (b,h,n,m)

        bias = self.bias_table(table)                                                     # (rows, h)
        fused = getattr(self.ops, "attn_softmax", None)
        if (fused is not None and not global_attn and not torch.is_grad_enabled()
                and not _drops(self.attn_drop) and self.ops.attn_softmax_supported(attn, attn.shape[-1])):
            # inference: bias gather, mask, blank-token logit and softmax in one kernel
            attn, blank = fused(attn, bias, pe_idx, cluster_mask, query=q, blank_key=self.blank_k)
        else:
            blank = (q * self.blank_k.reshape(1, h, 1, ch)).sum(-1, keepdim=True)        # (b,h,n,1)
            if (fused is not None and getattr(self.ops, "attn_softmax_backward", None) is not None
                    and getattr(self.ops, "bias_table_grad", None) is not None and torch.is_grad_enabled()
                    and not global_attn and attn.is_cuda
                    and not _drops(self.attn_drop)
                    and self.ops.attn_softmax_supported(attn, attn.shape[-1])):
                # training: the same glue as one kernel forward and one backward
                attn, blank = _AttnSoftmax.apply(attn, bias, pe_idx, cluster_mask, blank, self.ops)
            else:
                attn = attn + _position_bias(bias, pe_idx, self.ops)
                if cluster_mask is not None and not global_attn:
                    attn = attn + (1 - cluster_mask.reshape(b, 1, n, -1)) * (-100)
                attn = torch.softmax(torch.cat([attn, blank], dim=-1), dim=-1)
                attn = self.attn_drop(attn)
                blank, attn = attn[..., -1:], attn[..., :-1]

        if global_attn:
            out = attn @ v
        elif compact:
            out = self.ops.av_clusters(attn, v, cluster_idx, **sized)
        else:
            out = self.ops.av(attn, v, member_idx)                                       # (b,h,n,ch)
        out = out + blank * self.blank_v.reshape(1, h, 1, ch)
        return out.permute(0, 2, 1, 3).reshape(b, n, c)


class ClusterTransformerBlock(_Module):
    def __init__(self, dim, num_heads, mlp_ratio=2.0, drop=0.0, attn_drop=0.0, drop_path=0.0, layer_scale=0.0,
                 ops=None):
        super().__init__()
        self.norm1 = nn.LayerNorm(dim)
        self.attn = ClusterAttention(dim, num_heads, attn_drop=attn_drop, proj_drop=drop, ops=ops)
        self.drop_path = DropPath(drop_path) if drop_path > 0.0 else nn.Identity()
        self.norm2 = nn.LayerNorm(dim)
        self.mlp = Mlp(dim, int(dim * mlp_ratio), drop=drop, ops=ops)
        self.layer_scale = isinstance(layer_scale, (int, float)) and layer_scale > 0
        if self.layer_scale:
            self.gamma1 = nn.Parameter(layer_scale * torch.ones(dim))
            self.gamma2 = nn.Parameter(layer_scale * torch.ones(dim))

    def _fused_dtype(self, feat):
        """The type the block kernels work in, or None when the block runs layer by layer: on widths or types the kernels
        are not built for, with layer scale or an active dropout, with modules of other types or with hooks, and when the
        caller's `ops` has another implementation of a layer they stand for."""
        ops = self.attn.ops
        grad = torch.is_grad_enabled()
        if (self.layer_scale or not feat.is_cuda or getattr(ops, "block_tail", None) is None
                or (grad and getattr(ops, "block_tail_backward", None) is None) or not self.plain()):
            return None
        if _drops(self.mlp.drop) or _drops(self.attn.proj_drop) or (not grad and _drops(self.drop_path)):
            return None
        dt = torch.get_autocast_dtype("cuda") if torch.is_autocast_enabled("cuda") else torch.float32
        if (not ops.block_supported(feat, dt, self.mlp.fc1.out_features) or (grad and (_transformed() or feat.numel() == 0))
                or not all(_kernel_parameter(t, feat) for t in self.tensors())):
            return None
        return dt if all(getattr(ops, name, None) is fn for name, fn in ops.block_stands_for) else None

    def plain(self):
        """True when calling the block's modules runs the `forward` of their classes and nothing else."""
        m = self._modules
        attn, mlp = m["attn"], m["mlp"]
        a, ml = attn._modules, mlp._modules
        mods = (m["norm1"], attn, m["norm2"], mlp, a["q"], a["kv"], a["proj"], ml["fc1"], ml["fc2"], a["pos_embed"],
                a["attn_drop"], a["proj_drop"], ml["drop"])
        if tuple(map(type, mods)) != _BLOCK_TYPES or type(m["drop_path"]) not in (nn.Identity, DropPath):
            return False
        if not torch.is_grad_enabled():                    # hooks of backward passes have nothing to see
            if _module._global_forward_hooks or _module._global_forward_pre_hooks:
                return False
            for mod in mods:
                d = mod.__dict__
                if d["_forward_hooks"] or d["_forward_pre_hooks"] or "forward" in d:
                    return False
            d = m["drop_path"].__dict__
            return not (d["_forward_hooks"] or d["_forward_pre_hooks"] or "forward" in d)
        return not (any(map(_hooked, mods)) or _hooked(m["drop_path"]))

    def issued_with(self, ops, cluster_size):
        """True when an inference forward of the block may be issued from outside: nothing but its own modules' forwards runs, they
        use `ops` on clusters of that size, and nothing drops."""
        d = self.__dict__
        if d["_forward_hooks"] or d["_forward_pre_hooks"] or "forward" in d or self.layer_scale or not self.plain():
            return False
        m = d["_modules"]
        attn, mlp = m["attn"], m["mlp"]
        if attn.ops is not ops or mlp.ops is not ops or attn.cluster_size != cluster_size:
            return False
        a = attn._modules
        for mod in (a["attn_drop"], a["proj_drop"], mlp._modules["drop"], m["drop_path"]):
            if mod.training and _drops(mod):
                return False
        return True

    def tensors(self):
        """The parameters of the block in one tuple, straight from the modules' tables: the look-ups of 30 blocks are a
        visible part of a small forward's host time.  Where one is not in its table - replicas and wrappers set plain
        attributes - all come by attribute."""
        m = self._modules
        attn, mlp = m["attn"], m["mlp"]
        a, ml = attn._modules, mlp._modules
        try:
            n1, n2, ap = m["norm1"]._parameters, m["norm2"]._parameters, attn._parameters
            q, kv, proj, pe = a["q"]._parameters, a["kv"]._parameters, a["proj"]._parameters, a["pos_embed"]._parameters
            f1, f2 = ml["fc1"]._parameters, ml["fc2"]._parameters
            return (n1["weight"], n1["bias"], n2["weight"], n2["bias"], q["bias"], kv["bias"], proj["bias"], f1["bias"], f2["bias"],
                    ap["blank_k"], ap["blank_v"], q["weight"], kv["weight"], proj["weight"], f1["weight"], f2["weight"],
                    pe["weight"], pe["bias"])
        except KeyError:
            n1, n2, q, kv, proj, pe, f1, f2 = m["norm1"], m["norm2"], a["q"], a["kv"], a["proj"], a["pos_embed"], ml["fc1"], ml["fc2"]
            return (n1.weight, n1.bias, n2.weight, n2.bias, q.bias, kv.bias, proj.bias, f1.bias, f2.bias, attn.blank_k, attn.blank_v,
                    q.weight, kv.weight, proj.weight, f1.weight, f2.weight, pe.weight, pe.bias)

    def _packed(self, dt):
        """(weights of the five Linear layers as the block kernels read them, byte offset of each).  16-bit ones are kept until a
        weight changes, like the 16-bit copies of single layers.  fp32 ones are laid out anew in every forward: without
        mixed precision a forward reads the parameters as they are, also after a write that leaves no trace in the key
        (through `p.data`, or by a replayed recording)."""
        attn, mlp = self.attn, self.mlp
        weights = (attn.q.weight, attn.kv.weight, attn.proj.weight, mlp.fc1.weight, mlp.fc2.weight)
        if dt == torch.float32:
            return attn.ops.block_pack(attn.dim, dt, [(w.detach(), False) for w in weights])
        key = (dt,) + tuple((w._version, w.data_ptr()) for w in weights)

        def make():
            held = [w.detach() for w in weights]
            return attn.ops.block_pack(attn.dim, dt, [(w, False) for w in held]), held

        return _kept(self.__dict__, "_pack_cache", key, make).value

    def fits(self, c, hidden, heads, table_cols=5):
        """True when every parameter has the shape of a block of c channels with `hidden` hidden ones and `heads` heads."""
        want = 5 * [(c,)] + [(2 * c,), (c,), (hidden,)] + 3 * [(c,)] + [(c, c), (2 * c, c), (c, c), (hidden, c), (c, hidden),
                                                                     (heads, table_cols), (heads,)]
        return [tuple(t.shape) for t in self.tensors()] == want

    def _factors(self, feat, dt):
        """The images' factors of both branches under stochastic depth (fp32), or None."""
        if not _drops(self.drop_path):
            return None
        return torch.stack([self.drop_path.factors(feat.shape[0], dt, feat.device) for _ in range(2)]).float()

    def _train_whole(self, feat, dt, global_attn, table, pe_idx, cluster_idx, grid_lists):
        """(plan, pairs) when a training pass of the block is one native call - local attention of clusters of 8 by its kernel, or, as (None,
        None), global attention of a short sequence - else None."""
        attn, ops = self.attn, self.attn.ops
        if (getattr(ops, "block_train_forward", None) is None or _drops(attn.attn_drop) or table.requires_grad
                or any(getattr(ops, name, None) is not fn for name, fn in ops.block_train_stands_for)):
            return None
        plan = pairs = None
        if not global_attn:
            if cluster_idx is None or cluster_idx.shape[2] != 6 or attn.cluster_size != 8 or grid_lists is None or len(grid_lists) < 5:
                return None
            plan, pairs = grid_lists[3:5]
        if not (ops.block_train_supported(feat, dt, attn.num_heads, self.mlp.fc1.out_features, table, pe_idx, plan, pairs)
                and self.fits(feat.shape[2], self.mlp.fc1.out_features, attn.num_heads, table.shape[1])):
            return None
        return plan, pairs

    def forward(self, feat, member_idx, cluster_mask, pe_idx, global_attn, table, cluster_idx=None, grid_lists=None,
                carry=None):
        """Returns (feat, branch): the block's output is feat + branch.  The addition is left to the caller, which
        hands `branch` to the next block as `carry` so that it can ride along with that block's first norm."""
        ops = self.attn.ops
        if carry is not None and torch.is_grad_enabled():
            feat, carry = feat + carry, None
        dt = self._fused_dtype(feat)
        if dt is not None and torch.is_grad_enabled():
            # training: the same kernels, keeping what their backward reads
            attn, mlp, norm1, norm2 = self.attn, self.mlp, self.norm1, self.norm2
            whole = self._train_whole(feat, dt, global_attn, table, pe_idx, cluster_idx, grid_lists)
            if whole is not None:
                plan, pairs = whole
                return (_DenseAttentionRows if plan is None else _ClusterAttentionRows).apply(
                    feat, table, pe_idx, plan, pairs, self._factors(feat, dt), member_idx, cluster_mask, dt, attn.num_heads,
                    mlp.fc1.out_features, (norm1.eps, norm2.eps), attn.scale, ops, *self.tensors()), None
            qkv, feat = _NormLinearRows.apply(feat, norm1.weight, norm1.bias, attn.q.weight, attn.q.bias, attn.kv.weight,
                                              attn.kv.bias, norm1.eps, dt, ops)
            c = attn.dim
            a = attn.attend(qkv[..., :c], qkv[..., c:], member_idx, cluster_mask, pe_idx, global_attn, table, cluster_idx, grid_lists)
            scale = self._factors(feat, dt)
            return _BlockTail.apply(a.to(dt).contiguous(), feat, attn.proj.weight, attn.proj.bias, norm2.weight, norm2.bias,
                                    mlp.fc1.weight, mlp.fc1.bias, mlp.fc2.weight, mlp.fc2.bias, scale, norm2.eps, dt, ops), None
        if dt is not None:
            # inference: three kernels - norm and projections, attention, everything behind it
            if carry is not None:
                feat = feat + carry
            attn, mlp = self.attn, self.mlp
            packed, at = self._packed(dt)
            c = feat.shape[2]
            qkv = ops.norm_linear(feat, self.norm1.weight, self.norm1.bias, self.norm1.eps, packed, at[0], attn.q.bias,
                                  attn.kv.bias, 3 * c)
            a = attn.attend(qkv[..., :c], qkv[..., c:], member_idx, cluster_mask, pe_idx, global_attn, table, cluster_idx,
                            grid_lists)
            a = a if a.dtype == dt else a.to(dt)
            return ops.block_tail(a.contiguous(), feat, packed, at[2:], attn.proj.bias, self.norm2.weight, self.norm2.bias,
                                  self.norm2.eps, mlp.fc1.bias, mlp.fc2.bias), None
        feat, x = _add_layer_norm(self.norm1, feat, carry, ops)
        a = self.attn(x, member_idx, cluster_mask, pe_idx, global_attn, table, cluster_idx, grid_lists)
        feat, x = _add_layer_norm(self.norm2, feat, self.drop_path(self.gamma1 * a if self.layer_scale else a), ops)
        f = self.mlp(x)
        return feat, self.drop_path(self.gamma2 * f if self.layer_scale else f)


_BLOCK_TYPES = (nn.LayerNorm, ClusterAttention, nn.LayerNorm, Mlp, nn.Linear, nn.Linear, nn.Linear, nn.Linear, nn.Linear,
                nn.Linear, nn.Dropout, nn.Dropout, nn.Dropout)


def _kernel_parameter(t, feat):
    """True for a parameter the block kernels read in place."""
    return (t is not None and t.dtype == torch.float32 and t.is_contiguous() and t.device == feat.device
            and t.data_ptr() % 16 == 0)


class ClusterMerging(_Module):
    """Adaptive down-sampling: keeps ds_rate of the tokens and merges each one's neighbourhood into it."""

    INNER = 4

    def __init__(self, dim, out_dim, alpha=4.0, ds_rate=0.25, reserve_on=True, ops=None):
        super().__init__()
        self.alpha, self.ds_rate, self.reserve_on = alpha, ds_rate, reserve_on
        self.weight_net = nn.Sequential(nn.Linear(5, self.INNER), nn.LayerNorm(self.INNER), nn.GELU())
        self.norm = nn.LayerNorm(self.INNER * dim)
        self.linear = nn.Linear(self.INNER * dim, out_dim)
        self.ops = ops

    def select(self, pos, learned_prob, stride, reserve_num):
        """Indices (b, n') of the tokens kept as merge centres (aff_transformer.py:296-334)."""
        b, n, _ = pos.shape
        keep = int(n * self.ds_rate)
        one_pass = getattr(self.ops, "merge_centres", None)
        if one_pass is not None and self.ops.merge_centres_supported(pos, learned_prob):
            # scores, selection and the reserved tokens in one kernel; among equal scores at the cut the lower index
            dist = None if stride == 2 else knn(pos, pos, 2, return_dist=True)[1][:, :, 1]
            return one_pass(pos, dist, learned_prob, float(self.alpha), stride,
                            keep - reserve_num if self.reserve_on else keep, reserve_num, self.reserve_on)
        if stride == 2:                      # tokens still fill the grid: every other row and column
            prior = ((pos % stride).sum(-1) == 0).float()
        else:                                # adaptive grid: spacing from the distance to the nearest other token
            _, dist = knn(pos, pos, 2, return_dist=True)
            spacing = 2 ** (dist[:, :, 1].log2().ceil() + 1)
            prior = ((pos.long() % spacing.unsqueeze(2).long()).sum(-1) == 0).float()
        score = prior
        if learned_prob is not None:
            # widened before the addition (the values are those of the mixed-type addition; the framework's kernel
            # for mixed types has a fixed cost of some 45 us on this device, however small the tensors)
            score = score + (learned_prob.detach().view(b, n) * self.alpha).float()
        if not self.reserve_on:
            return score.topk(keep, dim=1, sorted=False)[1]
        reserved = ((pos % (stride * 2)).sum(-1) == 0)
        score = score + reserved.float() * (-100)
        sampled = score.topk(keep - reserve_num, dim=1, sorted=False)[1]
        # the reserved tokens in ascending index order; there are exactly reserve_num of them per image
        kept = reserved.to(torch.uint8).sort(dim=1, descending=True, stable=True)[1][:, :reserve_num]
        return torch.cat([sampled, kept], dim=1)

    def forward(self, pos, feat, member_idx, cluster_mask, learned_prob, stride, pe_idx, reserve_num, table):
        b, n, c = feat.shape
        m = member_idx.shape[-1]
        centre = self.select(pos, learned_prob, stride, reserve_num)                     # (b, n')
        n_out = centre.shape[1]
        assert n_out == int(n * self.ds_rate), "number of merge centres"
        rows_op = getattr(self.ops, "merge_rows", None)
        mask_rows = None
        if rows_op is not None and self.ops.merge_rows_supported(pos, member_idx, pe_idx):
            # the rows of the per-token tensors at the centres in one launch
            if cluster_mask is not None and not cluster_mask.requires_grad and self.ops.merge_rows_supported(cluster_mask):
                pos, member_idx, pe_idx, mask_rows = rows_op(centre, pos, member_idx, pe_idx, cluster_mask)
            else:
                pos, member_idx, pe_idx = rows_op(centre, pos, member_idx, pe_idx)
            rows = centre.unsqueeze(2).expand(-1, -1, m)
        else:
            pos = pos.gather(1, centre.unsqueeze(2).expand(-1, -1, pos.shape[2]))
            rows = centre.unsqueeze(2).expand(-1, -1, m)
            member_idx = member_idx.gather(1, rows)                                      # (b, n', m)
            pe_idx = pe_idx.gather(1, rows)
        if cluster_mask is not None and mask_rows is None:
            mask_rows = cluster_mask.gather(1, rows)
        table_w = _table_function(self, "_weight_table_cache", self.weight_net, table,
                                  lambda: _weight_table(self.weight_net, table, self.ops))  # (rows, 4)
        one_pass = getattr(self.ops, "merge_weights", None)
        if one_pass is not None and not torch.is_grad_enabled() and self.ops.merge_weights_supported(table_w):
            # inference: lookup, importance of each neighbour and mask in one kernel
            weights = one_pass(table_w, pe_idx, member_idx, learned_prob, mask_rows)
        elif (one_pass is not None and getattr(self.ops, "merge_weights_backward", None) is not None and torch.is_grad_enabled()
              and learned_prob is not None and table_w.is_cuda and table_w.dtype == torch.float32 and table_w.is_contiguous() and pe_idx.dtype == torch.int64
              and self.ops.merge_weights_supported(table_w) and not _transformed() and not (mask_rows is not None and mask_rows.requires_grad)
              and not torch.are_deterministic_algorithms_enabled()):           # its gradient of the scores is added up by atomics
            weights = _MergeWeights.apply(table_w, learned_prob.float().reshape(b, n), pe_idx, member_idx, mask_rows, self.ops)
        else:
            weights = _table_rows(table_w, pe_idx)                                       # (b, n', m, 4)
            if learned_prob is not None:
                weights = weights * learned_prob.gather(1, member_idx.reshape(b, -1, 1)).reshape(b, n_out, m, 1)
            if cluster_mask is not None:
                weights = weights * mask_rows.unsqueeze(3)
        merged = self.ops.wf(weights, feat, member_idx).reshape(b, n_out, -1)            # channel = ic * c + c'
        return pos, _linear(self.linear, _layer_norm(self.norm, merged, self.ops, True, self.linear), self.ops)


class BasicLayer(_Module):
    """One stage: neighbourhood lists, `depth` blocks over them, optional merging into the next stage."""

    def __init__(self, dim, out_dim, cluster_size, nbhd_size, depth, num_heads, mlp_ratio, alpha=4.0, ds_rate=0.25,
                 reserve_on=True, drop=0.0, attn_drop=0.0, drop_path=0.0, layer_scale=0.0, downsample=True,
                 ops=None):
        super().__init__()
        assert cluster_size > 0
        self.cluster_size, self.nbhd_size = cluster_size, nbhd_size
        self.ops = ops
        rates = drop_path if isinstance(drop_path, (list, tuple)) else [drop_path] * depth
        self.blocks = nn.ModuleList([
            ClusterTransformerBlock(dim, num_heads, mlp_ratio, drop, attn_drop, rates[i], layer_scale, ops=ops)
            for i in range(depth)])
        for blk in self.blocks:
            blk.attn.cluster_size = cluster_size
        if downsample:
            self.downsample = ClusterMerging(dim, out_dim, alpha, ds_rate, reserve_on, ops=ops)
            self.prob_net = nn.Linear(dim, 1)
        else:
            self.downsample = None
        self._grid_cache = {}

    def neighbourhoods(self, pos, h, w, radius, table_width):
        """(pos reordered, ranking or None, member_idx (b,n,nbhd), mask or None, pe_idx (b,n,nbhd),
        cluster numbers (b,n,nnc) int32 or None).

        aff_transformer.py:454-487.  The list of token i holds the members of its nnc nearest clusters,
        nearest cluster first; members of cluster g are tokens g*m .. g*m+m-1 of the reordered sequence.
        """
        b, n, d = pos.shape
        m = self.cluster_size
        k = int(math.ceil(n / float(m)))
        nnc = min(int(round(self.nbhd_size / float(m))), k)
        ranking = None
        if k == n:
            centres, members, mask = pos, torch.arange(n, device=pos.device).reshape(1, n, 1).expand(b, -1, -1), None
        else:
            pos, centres, members, mask, ranking = space_filling_cluster(pos, m, h, w)
        nearest = knn(pos, centres, nnc)                                                  # (b, n, nnc)
        one_pass = getattr(self.ops, "neighbour_lists", None)
        if (ranking is not None and one_pass is not None and not torch.is_grad_enabled()
                and self.ops.neighbour_lists_supported(pos, nearest)):
            # the four index tensors in one kernel
            member_idx, mask, pe_idx, cluster_idx = one_pass(pos, nearest, m, radius, table_width, mask is not None)
            return pos, ranking, member_idx, mask, pe_idx, (cluster_idx if m in (8, 24) else None)
        if ranking is not None:
            # cluster order: cluster g owns tokens g*m .. g*m+m-1, pad slots of the last one hold index 0 and mask 0
            rows = nearest.unsqueeze(3) * m + torch.arange(m, device=pos.device)
            valid = rows < n
            member_idx = torch.where(valid, rows, torch.zeros_like(rows)).reshape(b, n, nnc * m)
            if mask is not None:
                mask = valid.reshape(b, n, nnc * m).to(mask.dtype)
        else:
            pick = nearest.reshape(b, -1, 1).expand(-1, -1, m)
            member_idx = members.gather(1, pick).reshape(b, n, nnc * m)
            if mask is not None:
                mask = mask.gather(1, pick).reshape(b, n, nnc * m)
        nb_pos = pos.gather(1, member_idx.reshape(b, -1, 1).expand(-1, -1, d)).reshape(b, n, nnc * m, d)
        rel = nb_pos - (pos.unsqueeze(2) - radius)
        pe_idx = (rel[..., 1] * table_width + rel[..., 0]).long()
        # with clusters of m in cluster order, member_idx[b,i,m*r+t] = m*nearest[b,i,r]+t (0 past the last token):
        # the cluster numbers alone describe the lists (the kernels take clusters of 8 and, in part, of 24)
        cluster_idx = nearest.to(torch.int32).contiguous() if (ranking is not None and m in (8, 24)) else None
        return pos, ranking, member_idx, mask, pe_idx, cluster_idx

    def _grid(self, key, make):
        """What the lists of a full grid are made into, kept for good."""
        return _kept(self._grid_cache, key, None, lambda: (make(), ()), lasting=True).value

    def _grid_lists(self, key, pos1, h, w, radius):
        return self._grid(key, lambda: self.neighbourhoods(pos1, h, w, radius, 2 * radius + 1))

    def grid_order(self, pos1, h, w, radius):
        """The order (n,) in which this stage, as the first one, takes the tokens of the full grid (`pos1`: the
        positions of one image), or None when it leaves them as they are; fills the stage's cache of grid lists."""
        n = pos1.shape[1]
        if self.nbhd_size >= n:
            return None
        key = (n, h, w, str(pos1.device))
        ranking = self._grid_lists(key, pos1[:1], h, w, radius)[1]
        return None if ranking is None else ranking[0, :, 0]

    def _issue_blocks(self, feat, pe_idx, global_attn, table, lists):
        """The stage's blocks through one call that issues all their kernels, or None when they go one by one: with
        gradients, where a block would not take its three kernels (`_fused_dtype`), where the attention is not one kernel,
        and when the caller's `ops` has another implementation of one of the pieces."""
        ops = self.ops
        if not feat.is_cuda or torch.is_grad_enabled() or getattr(ops, "blocks_forward", None) is None or not len(self.blocks):
            return None
        if not all(type(blk) is ClusterTransformerBlock and blk.issued_with(ops, self.cluster_size) for blk in self.blocks):
            return None
        first = self.blocks[0]
        dt = first._fused_dtype(feat)
        b, n, c = feat.shape
        h = first.attn.num_heads
        if dt is None or c != 32 * h or any(getattr(ops, name, None) is not fn for name, fn in ops.blocks_stand_for) or (
                dt == torch.float32 and getattr(ops, "block_layout", None) is None):
            return None
        if global_attn:
            if n > 64:
                return None
            plan = None
        else:
            plan = lists[3] if lists is not None and len(lists) > 3 else None
            if plan is None or not (self.cluster_size == 8 or (self.cluster_size == 24 and dt != torch.float32)):
                return None
        by_heads = plan is not None or dt == torch.float32         # bias tables (heads, rows); else (rows, heads)
        tensors = [blk.tensors() for blk in self.blocks]
        hidden, scale = first.mlp.fc1.out_features, first.attn.scale
        try:
            key = (dt, table.data_ptr(), table._version, table.dtype, c, h, hidden, plan is None,
                   [[(t._version, t.data_ptr()) for t in ts] for ts in tensors],
                   [(m["norm1"].eps, m["norm2"].eps, m["attn"].scale, m["attn"].num_heads) for m in map(_modules_of, self.blocks)])
        except AttributeError:                                     # a parameter is None, say the bias of a layer without one
            return None

        def make():
            held, made = [table] + [t.detach() for ts in tensors for t in ts], []
            # the call has one width, hidden layer, number of heads and scale for all blocks
            if not all(blk.fits(c, hidden, h) and blk.attn.num_heads == h and blk.attn.scale == scale
                       and all(_kernel_parameter(t, feat) for t in ts) for blk, ts in zip(self.blocks, tensors)):
                return (None, None), held, made
            params = (ops.block_params * len(tensors))()
            for p, blk, ts in zip(params, self.blocks, tensors):
                bias = blk.attn.bias_table(table)
                bias = bias.detach().to(dt)
                bias = (bias.t() if by_heads else bias).contiguous()
                made.append(bias)
                if dt != torch.float32:
                    packed, at = blk._packed(dt)
                    made.append(packed)
                    p.w_qkv, p.w_proj, p.w1, p.w2 = (packed.data_ptr() + o for o in (at[0],) + tuple(at[2:]))
                (p.norm1_w, p.norm1_b, p.norm2_w, p.norm2_b, p.b_q, p.b_kv, p.b_proj, p.b1, p.b2, p.blank_k,
                 p.blank_v) = (t.data_ptr() for t in ts[:11])
                p.bias_table, p.eps1, p.eps2 = bias.data_ptr(), blk.norm1.eps, blk.norm2.eps
            layout = ops.block_layout([w.detach() for ts in tensors for w in ts[11:16]]) if dt == torch.float32 else None
            return (params, layout), held, made

        kept = _kept(self.__dict__, "_issue_cache", key, make)     # in this frame until the kernels are issued
        params, layout = kept.value
        if params is None:
            return None
        if layout is not None:
            # fp32: the weights as they are now (`_packed`), for this call only
            packed, at = layout.pack(c, dt)
            base = packed.data_ptr()
            params = type(params).from_buffer_copy(params)
            for i, p in enumerate(params):
                p.w_qkv, _, p.w_proj, p.w1, p.w2 = (base + o for o in at[5 * i:5 * i + 5])
        return ops.blocks_forward(params, feat, h, hidden, dt, scale, plan, pe_idx if plan is None else None,
                                  table.shape[0] if by_heads else 0)

    def forward(self, pos, feat, h, w, on_grid, stride, table, radius, feat_ordered=False):
        """`feat_ordered`: the tokens already stand in the order `grid_order` gave (first stage only)."""
        b, n, d = pos.shape
        table_width = 2 * radius + 1
        global_attn = self.nbhd_size >= n
        cluster_idx = grid_lists = None
        if global_attn:
            member_idx = mask = None
            rel = (pos[:, None, :, :] + radius) - pos[:, :, None, :]
            pe_idx = (rel[..., 1] * table_width + rel[..., 0]).long()
        else:
            if on_grid:
                # grid tokens are the same for every image: one image's lists serve the whole batch
                key = (n, h, w, str(pos.device))
                pos1, ranking, *lists = self._grid_lists(key, pos[:1], h, w, radius)
                member_idx, mask, pe_idx, cluster_idx = lists
                if cluster_idx is not None:
                    grid_lists = (cluster_idx, pe_idx, mask)           # one image's lists, for the one-kernel attention
                    planner = getattr(self.ops, "cluster_attention_plan", None)
                    if (planner is not None and not torch.is_grad_enabled() and cluster_idx.shape[2] == 6 and pe_idx.is_cuda
                            and (self.cluster_size == 8 or torch.is_autocast_enabled("cuda"))):
                        # what that kernel makes of them, kept with them
                        grid_lists = grid_lists + (self._grid((key, "plan"), lambda: planner(*grid_lists)),)
                # the batch-sized copies the operators read
                member_idx, mask, pe_idx, cluster_idx = self._grid(
                    (key, b), lambda: [None if t is None else t.expand(b, -1, -1).contiguous() for t in lists])
                pos = pos1.expand(b, -1, -1)
                if ranking is not None and not feat_ordered:
                    feat = feat[:, ranking[0, :, 0]]
            else:
                pos, ranking, member_idx, mask, pe_idx, cluster_idx = self.neighbourhoods(pos, h, w, radius, table_width)
                if ranking is not None:
                    rows_op = getattr(self.ops, "gather_rows", None)
                    if rows_op is not None and not torch.is_grad_enabled() and self.ops.gather_rows_supported(feat):
                        feat = rows_op(feat, ranking[:, :, 0])          # inference: one row-gather kernel
                    else:
                        feat = feat.gather(1, ranking.expand(-1, -1, feat.shape[2]))

        planner = getattr(self.ops, "cluster_attention_plan", None)
        if (grid_lists is None and cluster_idx is not None and planner is not None and not torch.is_grad_enabled()
                and cluster_idx.shape[2] == 6 and cluster_idx.is_cuda
                and ((feat.dtype == torch.float32 and self.cluster_size == 8) or torch.is_autocast_enabled("cuda"))):
            # the one-kernel attention of every block reads what it makes of the lists from a plan built once
            grid_lists = (cluster_idx, pe_idx, mask, planner(cluster_idx, pe_idx, mask))
        if ((grid_lists is None or len(grid_lists) == 3) and cluster_idx is not None and planner is not None
                and torch.is_grad_enabled() and getattr(self.ops, "cluster_attention_backward", None) is not None
                and not global_attn and self.cluster_size == 8 and cluster_idx.shape[2] == 6 and cluster_idx.is_cuda
                and (torch.is_autocast_enabled("cuda") or feat.dtype == torch.float32)):
            # training (fp32, or mixed precision): the plan of the one-kernel attention and the sorted pair lists of its
            # backward's scatters, built once for all blocks of the stage (a grid stage hands over one image's lists)
            # from the numbers, which the forward reads: lists of whole clusters by construction
            from_numbers = getattr(self.ops, "cluster_pairs_from_numbers", None)
            if any(getattr(self.ops, name, None) is not fn for name, fn in getattr(self.ops, "cluster_pairs_from_numbers_stands_for", ())):
                from_numbers = None
            pairs = self.ops.cluster_pairs(member_idx) if from_numbers is None else from_numbers(cluster_idx)
            if pairs is not None:
                lists = grid_lists if grid_lists is not None else (cluster_idx, pe_idx, mask)
                grid_lists = tuple(lists) + (planner(lists[0], lists[1], lists[2]), pairs)
        carry = None
        issued = self._issue_blocks(feat, pe_idx, global_attn, table, grid_lists)
        if issued is not None:
            feat = issued
        for blk in self.blocks if issued is None else ():
            feat, carry = blk(feat, member_idx, mask, pe_idx, global_attn, table, cluster_idx, grid_lists, carry)
        learned_prob = None
        scorer = getattr(self.ops, "add_row_score", None)
        if (self.downsample is not None and scorer is not None and not torch.is_grad_enabled() and feat.is_cuda
                and torch.is_autocast_enabled("cuda")):
            # inference: the last residual addition and the importance score of the tokens in one pass
            w16, b16 = _cast_params(self.prob_net, torch.get_autocast_dtype("cuda")).value
            if self.ops.add_row_score_supported(feat, carry, w16):
                feat, learned_prob = scorer(feat, carry, w16, b16)
                carry = None
        if carry is not None:
            feat = feat + carry

        if self.downsample is not None:
            if global_attn:   # merging after a dense stage: every token is every token's neighbour
                member_idx = torch.arange(n, device=feat.device).expand(b, n, n).contiguous()
            if learned_prob is None:
                learned_prob = _score(self.prob_net, feat, self.ops)
            reserve_num = math.ceil(h / (stride * 2)) * math.ceil(w / (stride * 2))
            pos, feat = self.downsample(pos, feat, member_idx, mask, learned_prob, stride, pe_idx, reserve_num, table)
        return pos, feat


class PatchEmbed(_Module):
    """Two stride-2 3x3 convolutions (BatchNorm + GELU between them): one token per 4x4 pixels."""

    def __init__(self, in_chans=3, embed_dim=32, patch_norm=True, ops=None):
        super().__init__()
        self.ops = ops
        self.proj1 = nn.Conv2d(in_chans, embed_dim // 2, kernel_size=3, stride=2, padding=1)
        self.bn = nn.BatchNorm2d(embed_dim // 2)
        self.act1 = nn.GELU()
        self.proj2 = nn.Conv2d(embed_dim // 2, embed_dim, kernel_size=3, stride=2, padding=1)
        self.norm = nn.LayerNorm(embed_dim) if patch_norm else None

    def _bn_affine(self):
        """BatchNorm in inference as y = x * scale + shift per channel, the first convolution's bias folded in; kept
        until a parameter or a running statistic changes."""
        bn, conv = self.bn, self.proj1
        parts = [t for t in (bn.weight, bn.bias, bn.running_mean, bn.running_var, conv.bias) if t is not None]
        key = tuple((t.data_ptr(), t._version) for t in parts)

        def make():
            scale = torch.rsqrt(bn.running_var.float() + bn.eps)
            if bn.weight is not None:
                scale = scale * bn.weight.float()
            shift = -bn.running_mean.float() if conv.bias is None else conv.bias.float() - bn.running_mean.float()
            shift = shift * scale
            if bn.bias is not None:
                shift = shift + bn.bias.float()
            return (scale.detach(), shift.detach()), [t.detach() for t in parts]

        return _kept(self.__dict__, "_bn_affine_cache", key, make).value

    def forward(self, x, token_order=None):
        """`token_order(pos_of_one_image, h, w)`, when given, returns the order (N,) in which the first stage wants
        the tokens (or None); the tokens then leave in that order when the final norm can take it along, and the
        fifth return value says whether they did."""
        fused = getattr(self.ops, "channel_affine_gelu", None)
        if (fused is not None and not torch.is_grad_enabled() and not self.bn.training and x.is_cuda
                and torch.is_autocast_enabled("cuda") and self.bn.track_running_stats):
            # inference: bias, BatchNorm (an affine map per channel) and GELU in one pass over the convolution's output
            y = F.conv2d(x, self.proj1.weight, None, self.proj1.stride, self.proj1.padding)
            if self.ops.channel_affine_gelu_supported(y):
                y = fused(y, *self._bn_affine())
            else:
                y = self.act1(self.bn(y if self.proj1.bias is None else y + self.proj1.bias.view(1, -1, 1, 1)))
        else:
            y = self.act1(self.bn(self.proj1(x)))
        b, _, h0, w0 = y.shape
        h, w = (h0 + 1) // 2, (w0 + 1) // 2
        ys, xs = torch.meshgrid(torch.arange(h, device=x.device), torch.arange(w, device=x.device), indexing="ij")
        pos = torch.stack([xs, ys], dim=2).reshape(1, -1, 2)
        order = None
        if self.norm is not None and token_order is not None and x.is_cuda and not torch.is_grad_enabled():
            order = token_order(pos.float(), h, w)
        if order is not None or (self.norm is not None and self.proj2.bias is not None and x.is_cuda
                                 and not torch.is_grad_enabled()):
            # the second convolution's bias and the reordering ride along with the norm
            z = F.conv2d(y, self.proj2.weight, None, self.proj2.stride, self.proj2.padding)
            z = z.flatten(2).transpose(1, 2).contiguous()
            if _one_pass_norm_available(self.ops, z):
                tokens = self.ops.layer_norm(z, self.norm.weight, self.norm.bias, self.norm.eps, None, order,
                                             self.proj2.bias)
                return pos.expand(b, -1, -1).to(tokens.dtype), tokens, h, w, order is not None
            if self.proj2.bias is not None:
                z = z + self.proj2.bias
            tokens = self.norm(z)
            return pos.expand(b, -1, -1).to(tokens.dtype), tokens, h, w, False
        tokens = self.proj2(y).flatten(2).transpose(1, 2)
        assert tokens.shape[1] == h * w
        if self.norm is not None:
            tokens = _layer_norm(self.norm, tokens, self.ops)
        return pos.expand(b, -1, -1).to(tokens.dtype), tokens, h, w, False


class AutoFocusFormer(_Module):
    """aff_transformer.py:560-670.  Defaults are the reference's; `aff_tiny()` gives configs/aff_tiny.yaml."""

    def __init__(self, in_chans=3, num_classes=1000, embed_dim=(32, 128, 256, 512), cluster_size=8,
                 nbhd_size=(48, 48, 48, 49), alpha=4.0, ds_rate=0.25, reserve_on=True, depths=(2, 2, 6, 2),
                 num_heads=(3, 6, 12, 24), mlp_ratio=2.0, drop_rate=0.0, attn_drop_rate=0.0, drop_path_rate=0.1,
                 patch_norm=True, layer_scale=0.0, img_size=224, ops=None):
        super().__init__()
        ops = ops if ops is not None else default_ops()
        self.num_classes = num_classes
        self.num_features = embed_dim[-1]
        self.ops = ops
        self.patch_embed = PatchEmbed(in_chans, embed_dim[0], patch_norm, ops=ops)
        self.pos_drop = nn.Dropout(drop_rate)
        table, self.radius = relative_position_table(img_size)
        self.register_buffer("pre_table", table, persistent=False)
        rates = [r.item() for r in torch.linspace(0, drop_path_rate, sum(depths))]
        last = len(depths) - 1
        self.layers = nn.ModuleList([
            BasicLayer(embed_dim[i], embed_dim[i + 1] if i < last else None, cluster_size, nbhd_size[i], depths[i],
                       num_heads[i], mlp_ratio, alpha, ds_rate, reserve_on, drop_rate, attn_drop_rate,
                       rates[sum(depths[:i]):sum(depths[:i + 1])], layer_scale, downsample=i < last, ops=ops)
            for i in range(len(depths))])
        self.norm = nn.LayerNorm(self.num_features)
        self.head = nn.Linear(self.num_features, num_classes) if num_classes > 0 else nn.Identity()
        self.apply(self._init_weights)

    @staticmethod
    def _init_weights(mod):
        if isinstance(mod, nn.Linear):
            nn.init.trunc_normal_(mod.weight, std=0.02)
            if mod.bias is not None:
                nn.init.zeros_(mod.bias)
        elif isinstance(mod, nn.LayerNorm):
            nn.init.zeros_(mod.bias)
            nn.init.ones_(mod.weight)

    def forward_features(self, x):
        first = self.layers[0]
        pos, x, h, w, ordered = self.patch_embed(x, lambda pos1, h, w: first.grid_order(pos1, h, w, self.radius))
        x = self.pos_drop(x)
        table = self.pre_table
        if not torch.is_grad_enabled() and table.is_cuda and torch.is_autocast_enabled("cuda"):
            # every block's position-embedding Linear would round the table to 16 bits again: one copy, kept
            dt = torch.get_autocast_dtype("cuda")
            key = (table.data_ptr(), table._version, dt)
            full = table
            table = _kept(self.__dict__, "_table_cast_cache", key, lambda: (full.to(dt), [full])).value
        for i, layer in enumerate(self.layers):
            pos, x = layer(pos, x, h, w, on_grid=(i == 0), stride=2 ** (i + 1), table=table, radius=self.radius,
                           feat_ordered=(i == 0 and ordered))
        return _layer_norm(self.norm, x, self.ops).mean(1)

    def forward(self, x):
        x = self.forward_features(x)
        return _linear(self.head, x, self.ops) if isinstance(self.head, nn.Linear) else x


def aff_tiny(**kw):
    """configs/aff_tiny.yaml: depths 3/4/18/5, dims 64/128/256/512, heads 2/4/8/16, mlp ratio 3, 48 neighbours."""
    cfg = dict(embed_dim=(64, 128, 256, 512), depths=(3, 4, 18, 5), num_heads=(2, 4, 8, 16), mlp_ratio=3.0,
               cluster_size=8, nbhd_size=(48, 48, 48, 49), alpha=4.0, ds_rate=0.25, drop_path_rate=0.2)
    cfg.update(kw)
    return AutoFocusFormer(**cfg)


class CapturedForward:
    """One inference forward of `net` at a fixed input shape, recorded into a HIP graph and replayed.

    A forward of AFF-Tiny is some 170 kernel launches of 5-100 us each; issued one by one from Python they take, for few
    images, longer on the host than on the GPU.  Replaying the recorded graph leaves one launch per forward.  The
    model's forward has no host synchronisation and every kernel of the library takes the current stream and
    allocates through the framework, so the recording is the plain forward under `torch.cuda.graph`.

    The tables made of parameters (position bias, merge weights) and, under mixed precision, the 16-bit copies of the weights and
    the folded BatchNorm are those of the time of recording, held by this object: record again after the weights change.
    Everything else is read in place by every replay; with `autocast_dtype=None`, which records without mixed precision,
    that is every weight matrix.  The same output tensor is returned every time: copy it before the next call if it
    must outlive it.
    """

    def __init__(self, net, example, autocast_dtype=torch.float16, warmup=3):
        if not example.is_cuda:
            raise RuntimeError("CapturedForward records GPU work: the example input must be a CUDA tensor")
        self.net = net
        self.autocast_dtype = autocast_dtype
        self.static_in = example.clone()
        side = torch.cuda.Stream(device=example.device)
        side.wait_stream(torch.cuda.current_stream(example.device))
        with torch.cuda.stream(side):        # library handles, kernel selection and caches settle outside the recording
            for _ in range(warmup):
                self._forward()
        torch.cuda.current_stream(example.device).wait_stream(side)
        torch.cuda.synchronize(example.device)
        self.graph = torch.cuda.CUDAGraph()
        _thread.reads = self._reads = []      # the graph has their addresses
        try:
            with torch.cuda.graph(self.graph):
                self.static_out = self._forward()
        finally:
            del _thread.reads

    def _forward(self):
        with torch.no_grad(), torch.autocast("cuda", dtype=self.autocast_dtype or torch.float16,
                                            enabled=self.autocast_dtype is not None):
            return self.net(self.static_in)

    def __call__(self, x):
        if x.shape != self.static_in.shape or x.dtype != self.static_in.dtype:
            raise RuntimeError("CapturedForward was recorded for inputs of shape %s and dtype %s"
                               % (tuple(self.static_in.shape), self.static_in.dtype))
        if x.data_ptr() != self.static_in.data_ptr():
            self.static_in.copy_(x)
        self.graph.replay()
        return self.static_out
