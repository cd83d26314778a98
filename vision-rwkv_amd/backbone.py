"""Plain-PyTorch VRWKV backbone (no mmcv / mmcls) that calls the HIP Bi-WKV through RUN_CUDA.

It exists to time the operator in situ (VRWKV-L forward, benchmark config 4) and mirrors, module
for module and parameter name for parameter name,
classification/mmcls_custom/models/backbones/vrwkv.py:82-432 (identical copy:
classification_internimage/models/vrwkv.py) with the VRWKV-L settings of
classification_internimage/configs/vrwkv_l_22kto1k_384.yaml:10-28.  PatchEmbed is
Conv2d(kernel = stride = patch) + flatten (mmcv's PatchEmbed with these arguments) and the position
embedding is resized bicubically as in detection/mmdet_custom/models/utils/embed.py:6-47.
"""
import math

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.nn.modules import module as _hooks

from . import ops
from .ops import (RUN_CUDA, divided_takes, wkv_divided, bi_wkv_forward, q_shift, q_shift_mix, q_shift_mix_autograd, stack_mixes, row_fuse, resize_table, weight_grad, weight_grad_group, linear_takes, linear_group, transposed, sigmoid_gate_backward, EPI_RELU_SQ, EPI_RELU_SQ_BWD, EPI_ROUND, block_takes, block_weights_fit, block_forward, _dense, _equal_quarters, _forward_mode, _transformed, batched_cotangent, PRE_NONE, PRE_RELU_SQ, POST_NONE,
                  POST_SIGMOID_GATE, POST_RESIDUAL)


def resize_pos_embed(pos_embed, src_shape, dst_shape, mode="bicubic", num_extra_tokens=0):
    """Position table (1, extra + Hs*Ws, C) resampled to the grid dst_shape, extra tokens passed through: the
    interpolation of detection/mmdet_custom/models/utils/embed.py:6-47 (F.interpolate, align_corners=False), which
    the backbones call with no extra tokens (vrwkv.py:411-415)."""
    if tuple(src_shape) == tuple(dst_shape):
        return pos_embed
    _, L, C = pos_embed.shape
    if L != src_shape[0] * src_shape[1] + num_extra_tokens:
        raise RuntimeError(f"pos_embed has {L} tokens, expected {src_shape[0]}*{src_shape[1]}+{num_extra_tokens}")
    extra, grid = pos_embed[:, :num_extra_tokens], pos_embed[:, num_extra_tokens:]
    w = resize_table(grid, src_shape, dst_shape) if mode == "bicubic" else None
    if w is not None:
        return torch.cat((extra, w), dim=1) if num_extra_tokens else w
    w = grid.reshape(1, src_shape[0], src_shape[1], C).permute(0, 3, 1, 2)
    w = F.interpolate(w.float(), size=dst_shape, align_corners=False, mode=mode).to(pos_embed.dtype)
    w = torch.flatten(w, 2).transpose(1, 2)
    return torch.cat((extra, w), dim=1) if num_extra_tokens else w


class _Kept(dict):
    """What eval_cached keeps on a module; a copy of the module starts without."""

    def __deepcopy__(self, memo):
        return _Kept()

    def __reduce__(self):
        return _Kept, ()


def eval_cached(module, name, params, extra, make):
    """Value derived from parameters (a dtype conversion, a stacked table), kept on the module between forward passes
    without autograd and rebuilt when a parameter was written to (its version counter), moved or cast.  The entry holds on to
    the memory it was derived from, so that no later parameter can be found at the same address.  A write through p.data
    counts as no new version: after one, the next in-place write, cast or move of the parameter brings the value up to date.
    A value made while the stream is recorded into a graph exists when the graph runs, and is not kept."""
    key = [extra]
    for p in params:
        key += (p._version, p.dtype, p.get_device(), p.data_ptr())
    kept = module.__dict__.get("_eval_cache")
    if kept is None:
        kept = module.__dict__.setdefault("_eval_cache", _Kept())
    hit = kept.get(name)
    if hit is None or hit[0] != key:
        hit = (key, make(), [p.detach() for p in params])
        if params[0].is_cuda and torch.cuda.is_current_stream_capturing():
            return hit[1]
        kept[name] = hit
    return hit[1]


def _mix(module, x, mixes, shift_pixel, gamma, patch_resolution, fused, head_dim=0, through=0):
    """[x*m + q_shift(x)*(1-m) for m in mixes], and x itself `through` times for its other uses (see _branch): one fused kernel
    (forward, and backward under autograd); tensor ops when `fused` is off or the tensors are not on the GPU."""
    if fused and x.is_cuda and not _forward_mode():
        if torch.is_grad_enabled() and (x.requires_grad or any(m.requires_grad for m in mixes)):
            return q_shift_mix_autograd(x, mixes, shift_pixel, gamma, patch_resolution, head_dim, through)
        table = eval_cached(module, "mix_table", mixes, x.device, lambda: stack_mixes(mixes, x.device))
        return q_shift_mix(x.contiguous(), mixes, shift_pixel, gamma, patch_resolution, head_dim, mix_table=table) + [x] * through
    xx = q_shift(x, shift_pixel, gamma, patch_resolution)
    return [x * m + xx * (1 - m) for m in mixes] + [x] * through


# Whose weight gradient is the framework's own kernel, by the weight's elements and the multiplications: its deep split pays until
# the library's partial products fill the chip for long, which weights beyond about 0.6 million elements do sooner.  Own / the
# library's batched partial products and their sum, in us:
#   12544 tokens   768 x 768 34 / 44     384 x 384 23 / 40   1536 x 384 34 / 43   192 x 192 18 / 33   160 x 768 22 / 39   5 of 32 x 768 24 / 45
#                  1024 x 1024 45 / 43   9408 tokens: 4096 x 256 39 / 42           25088: 1024 x 1024 73 / 65, 1024 x 768 62 / 59
#   100352 tokens  768 x 768 189 / 274   384 x 384 60 / 118  192 x 192 35 / 98    1024 x 1024 317 / 230     301056: 768 x 768 537 / 408
OWN_WEIGHT_GRAD = ((650_000, 100_000_000_000), (1 << 20, 10_000_000_000))           # elements up to, multiplications up to


def _token_product(a, b, splits):
    """a^T b over the rows (tokens) of a (M, O), b (M, I) or of stacks of them: an own kernel (fp32 sums, rounded once), or
    `splits` batched partial products of the library.  A gradient that is itself to be differentiated, batched or traced takes tensor
    ops."""
    (M, O), I = a.shape[-2:], b.shape[-1]
    if (not torch.is_grad_enabled() and any(O * I <= n and M * O * I <= work for n, work in OWN_WEIGHT_GRAD) and O % 8 == 0 and I % 8 == 0 and a.dtype == b.dtype
            and not batched_cotangent(a, b) and not _transformed()
            and M * max(a.stride(-2), b.stride(-2), O, I) < 1 << 30):
        return weight_grad(a, b)
    S = splits if M % splits == 0 else 1
    part = torch.matmul(a.reshape(a.shape[:-2] + (S, M // S, O)).transpose(-1, -2), b.reshape(b.shape[:-2] + (S, M // S, I)))
    return part.sum(-3)                   # one kernel: the sum of 16-bit values accumulates in fp32 and is rounded once


class _SplitKLinear(torch.autograd.Function):
    """x @ W^T whose weight gradient g^T x -- a contraction over all B*T tokens into a small (out, in) matrix, which the
    library's GEMM runs as one deep sum on too few workgroups -- is split over the tokens (_token_product).  Forward and input gradient are the library's plain GEMMs."""

    @staticmethod
    def forward(ctx, x, weight, splits):
        ctx.save_for_backward(x, weight)
        ctx.splits = splits
        return F.linear(x, weight)

    @staticmethod
    def backward(ctx, g):
        x, weight = ctx.saved_tensors
        S = ctx.splits
        gx = g @ weight if ctx.needs_input_grad[0] else None
        gw = None
        if ctx.needs_input_grad[1]:
            gw = (_weight_products([g], [x])[0] if weight.numel() >= 1 << 21
                  else _token_product(g.reshape(-1, g.shape[-1]), x.reshape(-1, x.shape[-1]), S))
        return gx, gw, None


class _SplitKMatmul(torch.autograd.Function):
    """x @ W for a parameter matrix W (in, out): the same split of the weight gradient x^T g over the tokens."""

    @staticmethod
    def forward(ctx, x, weight, splits):
        ctx.save_for_backward(x, weight)
        ctx.splits = splits
        return x @ weight

    @staticmethod
    def backward(ctx, g):
        x, weight = ctx.saved_tensors
        S = ctx.splits
        gx = g @ weight.t() if ctx.needs_input_grad[0] else None
        gw = None
        if ctx.needs_input_grad[1]:
            gw = _token_product(x.reshape(-1, x.shape[-1]), g.reshape(-1, g.shape[-1]), S)
        return gx, gw, None


class _SplitKBmm(torch.autograd.Function):
    """torch.bmm(x, W) for a stack of parameter matrices W (n, in, out) and x (n, M, in) with M = all B*T tokens: each
    weight gradient x_i^T g_i is split over the tokens like _SplitKMatmul's (the library runs the deep, narrow
    contraction on a handful of workgroups otherwise)."""

    @staticmethod
    def forward(ctx, x, weight, splits):
        ctx.save_for_backward(x, weight)
        ctx.splits = splits
        return torch.bmm(x, weight)

    @staticmethod
    def backward(ctx, g):
        x, weight = ctx.saved_tensors
        S = ctx.splits
        gx = torch.bmm(g, weight.transpose(1, 2).contiguous()) if ctx.needs_input_grad[0] else None
        gw = None
        if ctx.needs_input_grad[1]:
            gw = _token_product(x, g, S)
        return gx, gw, None


def _bmm(x, weight):
    """torch.bmm(x, weight) for stacked low-rank parameter matrices; split weight gradient under autograd with many
    tokens."""
    if (x.is_cuda and torch.is_grad_enabled() and weight.requires_grad and x.dtype == weight.dtype
            and x.dtype in (torch.bfloat16, torch.float16) and weight.dim() == 3 and x.dim() == 3):
        M = x.shape[1]
        if M >= 4096 and M % 8 == 0:
            return _SplitKBmm.apply(x, weight, 8)
    return torch.bmm(x, weight)


def _matmul(x, weight):
    """x @ weight for a low-rank parameter matrix; split weight gradient under autograd with many tokens."""
    if (x.is_cuda and torch.is_grad_enabled() and weight.requires_grad and x.dtype == weight.dtype
            and x.dtype in (torch.bfloat16, torch.float16) and weight.dim() == 2):
        M = x.numel() // x.shape[-1]
        if M >= 4096 and M % 8 == 0:
            return _SplitKMatmul.apply(x, weight, 8)
    return x @ weight


def _only_multiplies(*linears):
    """True for projections whose module call does nothing but multiply with their weight: no hook, no bias, no other class or forward."""
    return (not _hooks._global_forward_hooks and not _hooks._global_forward_pre_hooks and not _hooks._global_backward_hooks
            and not _hooks._global_backward_pre_hooks
            and all(_as_built(l, nn.Linear) and not l._backward_hooks and not l._backward_pre_hooks and l.bias is None for l in linears))


def _proj(linear, x):
    """linear(x) for the bias-free projections of a block; under autograd on the GPU with many tokens the weight gradient
    is split over the tokens (see _SplitKLinear)."""
    if (x.is_cuda and torch.is_grad_enabled() and x.dtype in (torch.bfloat16, torch.float16) and x.numel() >= 4096 * x.shape[-1]
            and _only_multiplies(linear) and linear.weight.requires_grad and x.dtype == linear.weight.dtype):
        w = linear.weight
        S = 4 if w.numel() >= (1 << 21) else 8
        if x.numel() // x.shape[-1] % S == 0:
            return _SplitKLinear.apply(x, w, S)
    return linear(x)


def _rows(t):
    return t.reshape(-1, t.shape[-1])


def _plain_backward(*tensors):
    """True where a backward may launch kernels: nothing records, batches or traces it."""
    return not torch.is_grad_enabled() and not batched_cotangent(*tensors) and not _transformed()


def _weight_products(gs, xs):
    """The gradients g^T x of several projections' weights (see _SplitKLinear), in one launch where kernels may be launched (12544 tokens,
    own kernel one by one / the library / together: three of 768 x 768 110 / 127 / 60 us, 3072 x 768, 768 x 3072 and 768 x 768 263 / 200 / 137);
    of single ones the large (3072 x 768 93 / 83 / 67, 4096 x 1024 156 / 115 / 102, but 768 x 768 34 / 43 / 36)."""
    gs, xs = [_rows(g) for g in gs], [_rows(x) for x in xs]
    M = gs[0].shape[0] if gs else 0
    if (gs and (len(gs) > 1 or gs[0].shape[1] * xs[0].shape[1] >= 1 << 21) and M > 0 and gs[0].dtype in (torch.bfloat16, torch.float16) and _plain_backward(*gs)
            and all(t.is_cuda and t.dtype == gs[0].dtype and t.shape[0] == M and t.shape[1] % 8 == 0 and t.shape[1] <= 65536 for t in (*gs, *xs))
            and all((M + 256) * max(t.stride(0), t.shape[1]) < 1 << 30 for t in (*gs, *xs))
            and all(g.shape[1] * x.shape[1] <= 1 << 28 for g, x in zip(gs, xs))):
        return weight_grad_group(gs, xs)
    return [_token_product(g, x, 4 if g.shape[1] * x.shape[1] >= 1 << 21 else 8) for g, x in zip(gs, xs)]


class _Projections(torch.autograd.Function):
    """[x @ W^T for x, W in zip(xs, ws)] as one launch (vrwkv_linear_group), the gradients of the inputs likewise."""

    @staticmethod
    def forward(ctx, *xw):
        ctx.save_for_backward(*xw)
        n = len(xw) // 2
        outs = linear_group([dict(a=_rows(x), w=w) for x, w in zip(xw[:n], xw[n:])])
        return tuple(o.reshape(*x.shape[:-1], -1) for o, x in zip(outs, xw))

    @staticmethod
    def backward(ctx, *gs):
        xw, n = ctx.saved_tensors, len(gs)
        xs, ws = xw[:n], xw[n:]
        gx, gw = [None] * n, [None] * n
        need = [i for i in range(n) if ctx.needs_input_grad[i]]
        if _plain_backward(*gs) and len(need) > 1:
            outs = linear_group([dict(a=_rows(gs[i]), w=wt) for i, wt in zip(need, transposed([_dense(ws[i]) for i in need]))])
            for i, o in zip(need, outs):
                gx[i] = o.reshape(xs[i].shape)
        else:
            for i in need:
                gx[i] = gs[i] @ ws[i]
        need = [i for i in range(n) if ctx.needs_input_grad[n + i]]
        for i, w in zip(need, _weight_products([gs[i] for i in need], [xs[i] for i in need])):
            gw[i] = w
        return (*gx, *gw)


class _ChannelMix(torch.autograd.Function):
    """sigmoid(xr @ Wr^T) * (relu^2(xk @ Wk^T) @ Wv^T) (vrwkv.py:250-261 without key_norm): key and receptance in one launch, and every
    element-wise step, forward and backward, in the epilogue of the product before it: the (tokens, hidden) matrices, four times as
    wide as x, are written once and not read again to be squared or masked.  The steps see the products rounded, as the
    operators one by one do: a network of 16-bit activations amplifies last bits (VRWKV6: 3e-2 of its gradients' norm)."""

    @staticmethod
    def forward(ctx, xk, xr, wk, wr, wv):
        (kk, k), r = linear_group([dict(a=_rows(xk), w=wk, epi=EPI_RELU_SQ | EPI_ROUND, raw=True), dict(a=_rows(xr), w=wr)])
        out, y = linear_group([dict(a=kk, w=wv, gate=r, epi=EPI_ROUND, raw=True)])[0]
        ctx.save_for_backward(xk, xr, wk, wr, wv, k, kk, r, y)
        return out.reshape(xk.shape)

    @staticmethod
    def backward(ctx, g):
        xk, xr, wk, wr, wv, k, kk, r, y = ctx.saved_tensors
        plain = _plain_backward(g)
        g2 = _rows(g)
        if plain:
            g2 = g2.to(y.dtype).contiguous()
            plain = g2.data_ptr() % 16 == 0
        if plain:
            wk, wr, wv, k, r, y = (_dense(t) for t in (wk, wr, wv, k, r, y))
            gy, gr = sigmoid_gate_backward(y, r, g2)
            wkt, wrt, wvt = transposed([wk, wr, wv])
            gk = linear_group([dict(a=gy, w=wvt, gate=k, epi=EPI_RELU_SQ_BWD | EPI_ROUND)])[0]
            gxk, gxr = (t.reshape(xk.shape) for t in linear_group([dict(a=gk, w=wkt), dict(a=gr, w=wrt)]))
        else:                                                # from the inputs anew, so that it can be differentiated again
            k, r = F.linear(_rows(xk), wk), F.linear(_rows(xr), wr)
            kk = torch.square(torch.relu(k))
            s = torch.sigmoid(r)
            gy, gr = g2 * s, g2 * F.linear(kk, wv) * s * (1 - s)
            gk = (gy @ wv) * (2 * torch.relu(k))
            gxk, gxr = (gk @ wk).reshape(g.shape), (gr @ wr).reshape(g.shape)
        need = ctx.needs_input_grad
        of = [(gk, xk), (gr, xr), (gy, kk)]
        which = [i for i in range(3) if need[2 + i]]
        gw = dict(zip(which, _weight_products([of[i][0] for i in which], [of[i][1] for i in which])))
        return (gxk if need[0] else None, gxr if need[1] else None, gw.get(0), gw.get(1), gw.get(2))


# Where the grouped launches take the place of the library's products.  Two or more projections of one shape on M tokens in one launch
# are ahead from 70 tiles of 128 x 128 each on; a single one without an epilogue stays with the library.  M x K x N, library / own, us:
#   three of 784 x 768 x 768 23 / 14    4096 36 / 21    8192 47 / 34    11760 63 / 52    12544 80 / 52    (one: 7.6 / 13, 12 / 15, 15 / 17, 20 / 21, 27 / 21)
#   three of 784 x 1024 x 1024 27 / 19  4096 41 / 33    9216 89 / 61    10816 80 / 80    12544 79 / 82    three of 12544 x 384 x 384 33 / 23
# A whole channel mix without key_norm takes them from 256 tiles on, where the passes they save (28 us forward, 43 back at 12544 x 3072)
# outweigh a slower product: 4096 x 3072 x 768 28 / 34, 8192 42 / 40, 12544 62 / 54; 12544 x 768 x 3072 66 / 67; 12544 x 4096 x 1024 86 / 91.
# With key_norm the products stay the library's: inside VRWKV-L, whose weights come from memory, a value product with the gate as its epilogue
# takes 93 us at 9216 x 4096 x 1024 (two stages; 66 on operands that lie in the caches), the library's and the gate's pass 67 + 10.  All of these but the
# last were taken on operands in the caches; on others the own kernel gives up more (csrc/linear_wide.hip).
# Training steps of 64 images of 224 x 224, start and both of these: VRWKV-B 16195 -> 15108 us, VRWKV6-B 25761 -> 24499, bit for bit the same.
CHANNEL_MIX_TILES = 256 * 128 * 128


def _own_weights(linears, x, widths=None):
    """The weights of projections whose module call does nothing but multiply, and which vrwkv_linear_group takes; else None.  widths: of
    the projections' inputs, where they are not x."""
    if any(type(l) is not nn.Linear or type(l._parameters.get("weight")) is not nn.Parameter for l in linears):
        return None
    ws = [l._parameters["weight"] for l in linears]
    return ws if linear_takes(x, ws, widths) and _only_multiplies(*linears) else None       # (sizes first: few tokens are the usual no)


def _projs(linears, xs):
    """[linear(x) for linear, x in zip(linears, xs)] for projections of one shape."""
    ws = _own_weights(linears, xs[0]) if type(xs[0]) is torch.Tensor and all(x.shape == xs[0].shape and x.dtype == xs[0].dtype for x in xs) else None
    if ws is None:
        return [_proj(l, x) for l, x in zip(linears, xs)]
    if torch.is_grad_enabled() and any(t.requires_grad for t in (*xs, *ws)):
        return list(_Projections.apply(*xs, *ws))
    return [o.reshape(*x.shape[:-1], -1) for o, x in zip(linear_group([dict(a=_rows(x), w=w) for x, w in zip(xs, ws)]), xs)]


def _channel_mix(ffn, xk, xr):
    """What a channel mix makes of its two mixed inputs (vrwkv.py:250-261), by the rules above."""
    kn = ffn.key_norm
    if kn is None and ops.ROW_FUSE_ENABLED and type(xk) is type(xr) is torch.Tensor and xk.shape == xr.shape and xk.dtype == xr.dtype and xk.numel() >= CHANNEL_MIX_TILES:
        C, wk = xk.shape[-1], ffn.key._parameters.get("weight")
        ws = _own_weights((ffn.key, ffn.receptance, ffn.value), xk, (C, C, wk.shape[0] if wk is not None else 0))
        if ws is not None and ws[1].shape[0] == ws[2].shape[0] == C <= 8192:       # (the gate's backward kernel takes rows of up to that)
            wk, wr, wv = ws
            if torch.is_grad_enabled() and any(t.requires_grad for t in (xk, xr, *ws)):
                return _ChannelMix.apply(xk, xr, wk, wr, wv)
            kk, r = linear_group([dict(a=_rows(xk), w=wk, epi=EPI_RELU_SQ | EPI_ROUND), dict(a=_rows(xr), w=wr)])
            return linear_group([dict(a=kk, w=wv, gate=r, epi=EPI_ROUND)])[0].reshape(xk.shape)
    # relu^2 (+ key_norm) and the sigmoid gate (vrwkv.py:256-261), one pass each; tensor ops under autograd
    k = row_fuse(_proj(ffn.key, xk), None, kn.weight if kn is not None else None, kn.bias if kn is not None else None, None,
                 PRE_RELU_SQ, POST_NONE, kn.eps if kn is not None else 1e-5)
    return row_fuse(_proj(ffn.value, k), _proj(ffn.receptance, xr), None, None, None, PRE_NONE, POST_SIGMOID_GATE)


def _layer_norm(ln, x):
    """nn.LayerNorm over the channels through the fused row kernel (forward and backward); tensor ops where it does
    not apply."""
    return row_fuse(x, None, ln.weight, ln.bias, None, PRE_NONE, POST_NONE, ln.eps)


# Whether a block runs as one native call (vrwkv_block_fwd), by M C C, the multiplications of a (C, C) projection on M tokens.
# Operator by operator the host takes 215 to 290 us a block (VRWKV6 340 to 430) and sets the pace up to some thousand tokens; the native call
# takes it 36 at most (VRWKV6 69), so called eagerly it gains until its time on the GPU reaches the host's or the library's, whichever is longer.
# Recorded into a graph only the time on the GPU counts.  There the native call saves launches and passes over the tokens, and
# its products are slower than the library's where the contraction is long: up to 17 % of a 16-bit block from about 1000 tokens of 768
# or more channels on.  Up to 512 channels it is ahead in 16 bits.  (VRWKV6, whose operators are more, is within a few % on the GPU at the
# eager line; its operators would also record the forming of their tables, which its native call does not leave behind.)  Twelve blocks
# of tokens x channels, pre-norm without key norms, operators ->
# native, eager | replayed, in us:
#   VRWKV  bf16  784 x 768   3323 -> 1185 | 1410 -> 1185      1568 x 768   2980 -> 1446 | 1449 -> 1446      392 x 1024 3328 -> 1444 | 1508 -> 1444
#                784 x 1024  3280 -> 1555 | 1645 -> 1558      3136 x 1024  2969 -> 2720 | 2317 -> 2718      6272 x 768 2588 -> 2428 | 2581 -> 2430
#                6272 x 1024 3930 -> 3804 | 3907 -> 3804      12544 x 768  4193 -> 3802 | 4174 -> 3799      196 x 192  3496 ->  430 | 1505 ->  388
#                3136 x 512  2948 -> 1355 | 1465 -> 1359      12544 x 512  2639 -> 2423 | 2615 -> 2452      12544 x 192 2925 -> 1173 | 1413 -> 1177
#   VRWKV6 bf16  6272 x 768  4041 -> 3673 | 3870 -> 3648      3136 x 1024  4575 -> 3634 | 3408 -> 3629      6272 x 1024 5511 -> 5260 | 5513 -> 5251
#                12544 x 768 6377 -> 5912 | 6440 -> 5916      12544 x 1024 8959 -> 8563 | 8932 -> 8581      196 x 192  5066 ->  833 | 2484 ->  829
# The 16-bit lines were drawn before the native call's projections of many tokens went to the wide kernel (widths in multiples of 128 as well): called
# eagerly 6272 and 12544 x 1024 are 3 and 4 % ahead natively today, and 784 x 1024 recorded 5 %, which the lines leave to the operators.
# fp32: a gap between few tokens, where launches count, and many, where the products of either are alike and the passes over the
# tokens count: there the library's products are ahead (784 x 768, 1568 x 768, 392 and 784 x 1024, 1960 and 2352 x 512).
#   VRWKV        392 x 768   3226 -> 1757 | 1893 -> 1761      784 x 768    3267 -> 2481 | 2261 -> 2484      1568 x 768 3348 -> 3875 | 3319 -> 3876
#                3136 x 768  6996 -> 6275 | 6975 -> 6277      784 x 1024   3411 -> 3842 | 3392 -> 3844      1568 x 1024 5550 -> 5390 | 5512 -> 5397
#                3136 x 384  3296 -> 2441 | 2392 -> 2433      6272 x 384   5733 -> 3964 | 5728 -> 3964      1568 x 512  3309 -> 2223 | 2336 -> 2226
#                1960 x 512  3506 -> 2441 | 2170 -> 2437      3136 x 448   3877 -> 2937 | 3822 -> 2933      43904 x 192 7934 -> 7932 | 7905 -> 7933
#   VRWKV6       784 x 768   5200 -> 3322 | 3362 -> 3324      1568 x 768   5247 -> 4912 | 4632 -> 4919      1568 x 1024 7079 -> 6769 | 7069 -> 6768
#                2352 x 512  5298 -> 3957 | 3993 -> 3951      25088 x 192  7745 -> 7315 | 7729 -> 7325      3136 x 1024 13191 -> 12315 | 13177 -> 12304
NATIVE_NARROW = 512
NATIVE_WORK = {False: (600_000_000, 3_800_000_000), True: (7_500_000_000, 7_500_000_000)}       # VRWKV6: most work recorded if wider, most work
NATIVE_FP32_GAP = {                                   # (VRWKV6, narrow): the work left to the operators, recorded and called
    (False, True): ((420_000_000, 620_000_000), (0, 0)), (False, False): ((300_000_000, 1_500_000_000), (600_000_000, 1_500_000_000)),
    (True, True): ((0, 0), (0, 0)), (True, False): ((0, 0), (0, 0))}


def _native_size(x, hidden, v6):
    """The rule above, and 32-bit byte offsets inside every token matrix of the call."""
    B, T, C = x.shape
    M, fp32 = B * T, x.dtype == torch.float32
    if M * max(C, hidden, 160) * (4 if fp32 else 2) >= 1 << 30:
        return False
    work, narrow = M * C * C, C <= NATIVE_NARROW
    if fp32:
        (lo, hi), (lo2, hi2) = NATIVE_FP32_GAP[v6, narrow]
        recorded, called = not lo < work < hi, not lo2 < work < hi2
    else:
        most, most2 = NATIVE_WORK[v6]
        recorded, called = narrow or work <= most, work <= most2
    return called and (recorded or not torch.cuda.is_current_stream_capturing())


# In 16 bits the projections of many tokens go to a kernel of 256-channel tiles (csrc/linear_wide.hip) with three stages where C and the
# hidden width are multiples of 192, and up to 768 channels such a block is ahead called eagerly at every size, recorded but for a
# stretch where a block with key norms is 8 % behind (2352 x 768; 5 % at 3136 x 768, past the stretch).  Of VRWKV6's projections
# the output and the channel mix's go there: key, value, receptance and gate share their launch with the decay's first product, whose tanh
# the wide kernel does not take, and stay on tiles of 128 x 128.  Operators -> native, eager | replayed:
#   VRWKV  bf16  1568 x 768   2980 -> 1446 | 1449 -> 1446      2352 x 768, key norms 3185 -> 1818 | 1677 -> 1811      6272 x 768 2588 -> 2428 | 2581 -> 2430
#                12544 x 768  4193 -> 3802 | 4174 -> 3799      3136 x 768, key norms 3195 -> 1957 | 1871 -> 1966      25088 x 768 7840 -> 7131 | 7850 -> 7142
#                12544 x 192  2925 -> 1173 | 1413 -> 1177
#   VRWKV6 bf16  1568 x 768   4611 -> 2115 | 2244 -> 2086      12544 x 768  6377 -> 5912 | 6440 -> 5916      12544 x 192 4546 -> 1931 | 2244 -> 1927
NATIVE_WIDE, NATIVE_WIDE_GAP = 768, (600_000_000, 1_600_000_000)


def _native_wide(x, hidden, v6):
    """The rule above, and the offsets as there."""
    B, T, C = x.shape
    if (x.dtype == torch.float32 or C > NATIVE_WIDE or C % 192 or hidden % 192 or hidden == 0 or B * T * max(C, hidden) * 2 >= 1 << 30):
        return False
    lo, hi = NATIVE_WIDE_GAP
    return v6 or C <= NATIVE_NARROW or not lo < B * T * C * C < hi or not torch.cuda.is_current_stream_capturing()


def _as_built(module, kind):
    """True when calling `module` does what `kind`'s own forward does with the module's parameters and nothing else."""
    return (type(module) is kind and not module._forward_hooks and not module._forward_pre_hooks and "forward" not in module.__dict__
            and module._compiled_call_impl is None)


def _branch(mix, kind, x, res):
    """mix(x), and x as the residual branch beside it takes it: where autograd records, what the token shift hands on, so that the shift's
    backward kernel adds the residual branch's gradient and no pass over the tokens does.  A module with hooks is called as it is."""
    if (torch.is_grad_enabled() and type(x) is torch.Tensor and x.is_cuda and x.requires_grad and _as_built(mix, kind)
            and not mix._backward_hooks and not mix._backward_pre_hooks and not _hooks._global_forward_hooks and not _hooks._global_forward_pre_hooks
            and not _hooks._global_backward_hooks and not _hooks._global_backward_pre_hooks and not _transformed()):
        return mix.with_residual(x, res)
    return mix(x, res), x


def _block_weights(block, att, ffn, x):
    """The weights of a block that one native call can run (its linear maps with the shapes and without the biases they are
    built with, the norms with both vectors) and the numbers that go with them, as fields of vrwkv_block_args; None for any
    other block, KeyError where a name is missing (pruned, normed, parametrised weights and buffers stand elsewhere)."""
    am, fm, bm, C = att._modules, ffn._modules, block._modules, x.shape[2]
    key = fm["key"]
    weight = key._parameters["weight"] if type(key) is nn.Linear else None
    hidden = weight.shape[0] if weight is not None else 0
    if not (C % 32 == 0 and hidden % 32 == 0 and 0 < hidden <= 4096 and att.fused_shift and ffn.fused_shift
            and att.shift_pixel == ffn.shift_pixel and (_native_wide(x, hidden, "gate" in am) or _native_size(x, hidden, "gate" in am))):
        return None
    w, num = {}, dict(hidden=hidden, shift_pixel=att.shift_pixel, post_norm=int(block.post_norm))
    for name, lin, shape in (("key", am["key"], (C, C)), ("value", am["value"], (C, C)), ("receptance", am["receptance"], (C, C)),
                             ("output", am["output"], (C, C)), ("ffn_key", key, (hidden, C)),
                             ("ffn_receptance", fm["receptance"], (C, C)), ("ffn_value", fm["value"], (C, hidden))):
        if not _as_built(lin, nn.Linear):
            return None
        p = lin._parameters
        if p["bias"] is not None or p["weight"] is None or p["weight"].shape != shape:
            return None
        w[name] = p["weight"]
    for name, ln, n in (("ln1", bm["ln1"], C), ("ln2", bm["ln2"], C), ("att_kn", am.get("key_norm"), C),
                        ("ffn_kn", fm.get("key_norm"), hidden)):
        if ln is None and name.endswith("kn"):
            continue
        if not _as_built(ln, nn.LayerNorm) or ln.normalized_shape != (n,):
            return None
        p = ln._parameters
        if p["weight"] is None or p["bias"] is None:
            return None
        w[name + "_w"], w[name + "_b"] = p["weight"], p["bias"]
        num[name + "_eps"] = ln.eps
    if block.layer_scale:
        for name in ("gamma1", "gamma2"):
            w[name] = block._parameters[name]
            if w[name] is None or w[name].shape != (C,):
                return None
    return w, num


def _block_may_fuse(block, att_kind, ffn_kind):
    """The checks that come before a look at the weights."""
    return (not _hooks._global_forward_hooks and not _hooks._global_forward_pre_hooks
            and _as_built(block._modules["att"], att_kind) and _as_built(block._modules["ffn"], ffn_kind))


class VRWKV_SpatialMix(nn.Module):
    def __init__(self, n_embd, n_layer, layer_id, channel_gamma=1 / 4, shift_pixel=1, key_norm=False, fused_shift=True):
        super().__init__()
        self.layer_id, self.n_layer, self.n_embd = layer_id, n_layer, n_embd
        self.shift_pixel, self.channel_gamma, self.fused_shift = shift_pixel, channel_gamma, fused_shift
        r01 = layer_id / max(n_layer - 1, 1)
        r10 = 1.0 - layer_id / n_layer
        h = torch.arange(n_embd, dtype=torch.float32)
        self.spatial_decay = nn.Parameter(-5 + 8 * (h / (n_embd - 1)) ** (0.7 + 1.3 * r01))
        zigzag = torch.tensor([(i + 1) % 3 - 1 for i in range(n_embd)], dtype=torch.float32) * 0.5
        self.spatial_first = nn.Parameter(torch.ones(n_embd) * math.log(0.3) + zigzag)
        x = (h / n_embd).reshape(1, 1, n_embd)
        self.spatial_mix_k = nn.Parameter(torch.pow(x, r10))
        self.spatial_mix_v = nn.Parameter(torch.pow(x, r10) + 0.3 * r01)
        self.spatial_mix_r = nn.Parameter(torch.pow(x, 0.5 * r10))
        self.key = nn.Linear(n_embd, n_embd, bias=False)
        self.value = nn.Linear(n_embd, n_embd, bias=False)
        self.receptance = nn.Linear(n_embd, n_embd, bias=False)
        self.key_norm = nn.LayerNorm(n_embd) if key_norm else None
        self.output = nn.Linear(n_embd, n_embd, bias=False)
        self.fused_gate = True     # inference without key_norm: sigmoid(r) * y inside the Bi-WKV kernel

    def forward(self, x, patch_resolution):
        return self.with_residual(x, patch_resolution)[0]

    def with_residual(self, x, patch_resolution):
        """forward(x), and x as the residual branch is to take it (see _branch)."""
        B, T, C = x.shape
        res = x
        if self.shift_pixel > 0:
            xk, xv, xr, res = _mix(self, x, [self.spatial_mix_k, self.spatial_mix_v, self.spatial_mix_r], self.shift_pixel,
                                   self.channel_gamma, patch_resolution, self.fused_shift, through=1)
        else:
            xk = xv = xr = x
        k, v, r = _projs((self.key, self.value, self.receptance), (xk, xv, xr))
        wd = self.spatial_decay.dtype
        if torch.is_grad_enabled() or _forward_mode() or k.dtype != (wd if wd in (torch.half, torch.bfloat16) else torch.float32):
            w, u = self.spatial_decay, self.spatial_first
            y = wkv_divided(w, u, T, k, v) if divided_takes(w, u, k, v) else RUN_CUDA(w / T, u / T, k, v)      # vrwkv.py:183
        else:
            # what WKV.forward does with these arguments, the scaled fp32 copies of w and u kept between calls
            w, u = eval_cached(self, "wu", (self.spatial_decay, self.spatial_first), T,
                               lambda: ((self.spatial_decay / T).float().contiguous(),
                                        (self.spatial_first / T).float().contiguous()))
            if self.key_norm is None and self.fused_gate and r.dtype == k.dtype:
                # the receptance gate (vrwkv.py:185-186) applied inside the operator, before y is stored
                return _proj(self.output, bi_wkv_forward(w, u, k.contiguous(), v.contiguous(), gate=r.contiguous())), res
            y = bi_wkv_forward(w, u, k.contiguous(), v.contiguous())
        y = y.to(r.dtype)
        # key_norm and the sigmoid gate (vrwkv.py:184-186) in one pass; tensor ops under autograd
        kn = self.key_norm
        y = row_fuse(y, r, kn.weight if kn is not None else None, kn.bias if kn is not None else None, None,
                     PRE_NONE, POST_SIGMOID_GATE, kn.eps if kn is not None else 1e-5)
        return _proj(self.output, y), res


class VRWKV_ChannelMix(nn.Module):
    def __init__(self, n_embd, n_layer, layer_id, channel_gamma=1 / 4, shift_pixel=1, hidden_rate=4, key_norm=False,
                 fused_shift=True):
        super().__init__()
        self.shift_pixel, self.channel_gamma, self.fused_shift = shift_pixel, channel_gamma, fused_shift
        r10 = 1.0 - layer_id / n_layer
        x = (torch.arange(n_embd, dtype=torch.float32) / n_embd).reshape(1, 1, n_embd)
        self.spatial_mix_k = nn.Parameter(torch.pow(x, r10))
        self.spatial_mix_r = nn.Parameter(torch.pow(x, r10))
        hidden = hidden_rate * n_embd
        self.key = nn.Linear(n_embd, hidden, bias=False)
        self.key_norm = nn.LayerNorm(hidden) if key_norm else None
        self.receptance = nn.Linear(n_embd, n_embd, bias=False)
        self.value = nn.Linear(hidden, n_embd, bias=False)

    def forward(self, x, patch_resolution):
        return self.with_residual(x, patch_resolution)[0]

    def with_residual(self, x, patch_resolution):
        """forward(x), and x as the residual branch is to take it (see _branch)."""
        res = x
        if self.shift_pixel > 0:
            xk, xr, res = _mix(self, x, [self.spatial_mix_k, self.spatial_mix_r], self.shift_pixel, self.channel_gamma,
                               patch_resolution, self.fused_shift, through=1)
        else:
            xk = xr = x
        return _channel_mix(self, xk, xr), res


class Block(nn.Module):
    def __init__(self, n_embd, n_layer, layer_id, channel_gamma=1 / 4, shift_pixel=1, hidden_rate=4, init_values=None,
                 post_norm=False, key_norm=False, fused_shift=True):
        super().__init__()
        self.layer_id, self.post_norm = layer_id, post_norm
        self.ln1, self.ln2 = nn.LayerNorm(n_embd), nn.LayerNorm(n_embd)
        if layer_id == 0:
            self.ln0 = nn.LayerNorm(n_embd)
        self.att = VRWKV_SpatialMix(n_embd, n_layer, layer_id, channel_gamma, shift_pixel, key_norm, fused_shift)
        self.ffn = VRWKV_ChannelMix(n_embd, n_layer, layer_id, channel_gamma, shift_pixel, hidden_rate, key_norm, fused_shift)
        self.layer_scale = init_values is not None
        if self.layer_scale:
            self.gamma1 = nn.Parameter(init_values * torch.ones(n_embd))
            self.gamma2 = nn.Parameter(init_values * torch.ones(n_embd))

    def _native(self, x, res):
        """The block in one native call (vrwkv_block_fwd) where that computes the same; None elsewhere."""
        if not block_takes(x):
            return None
        try:
            fields = self._native_fields(x, res)
        except KeyError:                                     # a parameter or module that is held otherwise than built
            return None
        return block_forward(x, fields[0], **fields[1]) if fields is not None else None

    def _native_fields(self, x, res):
        if not _block_may_fuse(self, VRWKV_SpatialMix, VRWKV_ChannelMix):
            return None
        att, ffn = self._modules["att"], self._modules["ffn"]
        T, C = x.shape[1:]
        wn = _block_weights(self, att, ffn, x)
        if (wn is None or not block_weights_fit(x, wn[0].values()) or T != res[0] * res[1] or not att.fused_gate or att.shift_pixel <= 0
                or att.channel_gamma != ffn.channel_gamma or not _equal_quarters(C, att.channel_gamma, 0)):
            return None
        w, num = wn
        ap, fp = att._parameters, ffn._parameters
        decay, first = ap["spatial_decay"], ap["spatial_first"]
        am = [ap["spatial_mix_k"], ap["spatial_mix_v"], ap["spatial_mix_r"]]
        fm = [fp["spatial_mix_k"], fp["spatial_mix_r"]]
        if (decay is None or first is None or am[0] is None or am[1] is None or am[2] is None or fm[0] is None or fm[1] is None
                or decay.dtype != x.dtype):
            return None
        # under the operators' names: what an eager native call formed, a recorded forward that takes the operators finds
        device = x.device
        wd, u = eval_cached(att, "wu", (decay, first), T, lambda: ((decay / T).float().contiguous(), (first / T).float().contiguous()))
        att_mix = eval_cached(att, "mix_table", am, device, lambda: stack_mixes(am, device))
        ffn_mix = eval_cached(ffn, "mix_table", fm, device, lambda: stack_mixes(fm, device))
        index = x.get_device()
        if (wd.numel() != C or u.numel() != C or att_mix.numel() != 3 * C or ffn_mix.numel() != 2 * C
                or wd.get_device() != index or u.get_device() != index):
            return None                                      # (the operators refuse these)
        w["w"], w["u"], w["att_mix"], w["ffn_mix"] = wd, u, att_mix, ffn_mix
        num["Hp"], num["Wp"], num["quarter"] = res[0], res[1], int(C * att.channel_gamma)
        return w, num

    def forward(self, x, patch_resolution):
        if self.layer_id == 0:
            x = _layer_norm(self.ln0, x)
        y = self._native(x, patch_resolution)
        if y is not None:
            return y
        g1 = self.gamma1 if self.layer_scale else None
        g2 = self.gamma2 if self.layer_scale else None
        # residual with layer scale (vrwkv.py:300-313): x + gamma * ln(branch(x)) or x + gamma * branch(ln(x)), the
        # scale, the add and the post-norm in one pass; tensor ops under autograd
        if self.post_norm:
            x = row_fuse(*_branch(self.att, VRWKV_SpatialMix, x, patch_resolution), self.ln1.weight, self.ln1.bias, g1, PRE_NONE, POST_RESIDUAL, self.ln1.eps)
            x = row_fuse(*_branch(self.ffn, VRWKV_ChannelMix, x, patch_resolution), self.ln2.weight, self.ln2.bias, g2, PRE_NONE, POST_RESIDUAL, self.ln2.eps)
        else:
            x = row_fuse(self.att(_layer_norm(self.ln1, x), patch_resolution), x, None, None, g1, PRE_NONE, POST_RESIDUAL)
            x = row_fuse(self.ffn(_layer_norm(self.ln2, x), patch_resolution), x, None, None, g2, PRE_NONE, POST_RESIDUAL)
        return x


class VRWKV(nn.Module):
    """vrwkv.py:322-432 without the mmcv base classes.  With `out_indices` left at None it returns the last feature map
    (B, C, Hp, Wp); with an int or a sequence of layer indices (negative ones count from the end) it returns the tuple
    of those layers' feature maps, as the reference does for the mmdet / mmseg callers (vrwkv.py:368-378, 421-432)."""

    def __init__(self, img_size=224, patch_size=16, in_channels=3, embed_dims=256, depth=12, channel_gamma=1 / 4,
                 shift_pixel=1, post_norm=False, key_norm=False, init_values=None, hidden_rate=4, final_norm=True,
                 interpolate_mode="bicubic", fused_shift=True, out_indices=None):
        super().__init__()
        if out_indices is not None:
            out_indices = [out_indices] if isinstance(out_indices, int) else list(out_indices)
            out_indices = [depth + i if i < 0 else i for i in out_indices]
            for i in out_indices:
                if not 0 <= i <= depth:
                    raise ValueError(f"Invalid out_indices {i}")
        self.out_indices = out_indices
        self.patch_size = patch_size
        self.patch_embed = nn.Conv2d(in_channels, embed_dims, kernel_size=patch_size, stride=patch_size, bias=True)
        self.patch_resolution = (img_size // patch_size, img_size // patch_size)
        self.pos_embed = nn.Parameter(torch.zeros(1, self.patch_resolution[0] * self.patch_resolution[1], embed_dims))
        self.interpolate_mode = interpolate_mode
        self.layers = nn.ModuleList([
            Block(embed_dims, depth, i, channel_gamma, shift_pixel, hidden_rate, init_values, post_norm, key_norm,
                  fused_shift) for i in range(depth)])
        self.final_norm = final_norm
        if final_norm:
            self.ln1 = nn.LayerNorm(embed_dims)

    def load_reference_state_dict(self, state_dict, strict=True):
        """Load a checkpoint written by the reference backbones (vrwkv.py:322-432, vrwkv6.py, the mmdet / mmseg /
        classification_internimage copies).  Their parameter names are the ones used here except for the patch
        embedding, which mmcv's PatchEmbed keeps as `patch_embed.projection.{weight,bias}` (vrwkv.py:351-358);
        whole-model checkpoints carry a `backbone.` prefix and other modules' entries (`head.*`, `neck.*`), which are
        dropped.  A position table trained on another grid replaces this model's table and pre-training grid (it is
        interpolated to the input's grid in forward, as vrwkv.py:411-415 does).  Returns what
        nn.Module.load_state_dict returns."""
        sd = state_dict.get("state_dict", state_dict)
        if any(k.startswith("backbone.") for k in sd):
            sd = {k[len("backbone."):]: v for k, v in sd.items() if k.startswith("backbone.")}
        own = set(self.state_dict().keys())
        out = {}
        for k, v in sd.items():
            k = k.replace("patch_embed.projection.", "patch_embed.")
            if k in own:
                out[k] = v
            elif strict and k.split(".")[0] in {"patch_embed", "pos_embed", "layers", "ln1", "cls_token"}:
                raise KeyError(f"unexpected backbone entry {k!r} in the checkpoint")
        pe = out.get("pos_embed")
        if pe is not None and pe.shape != self.pos_embed.shape:
            n = pe.shape[1]
            side = int(round(n ** 0.5))
            if pe.dim() != 3 or pe.shape[2] != self.pos_embed.shape[2] or side * side != n:
                raise RuntimeError(f"pos_embed of shape {tuple(pe.shape)} does not fit this model")
            self.pos_embed = nn.Parameter(torch.zeros_like(pe, dtype=self.pos_embed.dtype, device=self.pos_embed.device))
            self.patch_resolution = (side, side)
        return self.load_state_dict(out, strict=strict)

    def _pos_embed_for(self, res):
        """Position embedding at grid `res`; in eval mode the interpolated table is computed once per grid
        (the reference re-runs the bicubic resize in every forward, vrwkv.py:411-415)."""
        if self.training or torch.is_grad_enabled():
            return resize_pos_embed(self.pos_embed, self.patch_resolution, res, self.interpolate_mode)
        key = (tuple(res), self.pos_embed._version, self.pos_embed.device, self.pos_embed.dtype)
        if getattr(self, "_pos_cache_key", None) != key:
            self._pos_cache = resize_pos_embed(self.pos_embed.detach(), self.patch_resolution, res, self.interpolate_mode)
            self._pos_cache_key = key
        return self._pos_cache

    def embed(self, img):
        """Patch embedding: (B, 3, H, W) -> (B, Hp*Wp, C) tokens and the patch grid (Hp, Wp)."""
        # kernel = stride = patch: the convolution is one GEMM over the flattened patches
        B, Cin, Hi, Wi = img.shape
        P = self.patch_size
        res = (Hi // P, Wi // P)
        patches = img[:, :, :res[0] * P, :res[1] * P].reshape(B, Cin, res[0], P, res[1], P)
        patches = patches.permute(0, 2, 4, 1, 3, 5).reshape(B, res[0] * res[1], Cin * P * P)
        x = F.linear(patches, self.patch_embed.weight.reshape(self.patch_embed.out_channels, -1), self.patch_embed.bias)
        return x, res

    def forward(self, img):
        x, res = self.embed(img)
        x = x + self._pos_embed_for(res).to(x.dtype)
        B, _, C = x.shape
        outs = []
        last = len(self.layers) - 1
        for i, layer in enumerate(self.layers):
            x = layer(x, res)
            if i == last and self.final_norm:
                x = _layer_norm(self.ln1, x)
            if self.out_indices is not None and i in self.out_indices:
                outs.append(x.reshape(B, res[0], res[1], C).permute(0, 3, 1, 2))
        if self.out_indices is not None:
            return tuple(outs)
        return x.reshape(B, res[0], res[1], C).permute(0, 3, 1, 2)


def vrwkv_l(**kw):
    """VRWKV-L as fine-tuned at 384x384: classification_internimage/configs/vrwkv_l_22kto1k_384.yaml:10-28
    (pre-training grid 192/16 = 12x12, interpolated to 24x24; K_NORM defaults to True, config.py:82)."""
    cfg = dict(img_size=192, patch_size=16, embed_dims=1024, depth=24, post_norm=True, init_values=1e-5,
               hidden_rate=4, key_norm=True, final_norm=True)
    cfg.update(kw)
    return VRWKV(**cfg)
