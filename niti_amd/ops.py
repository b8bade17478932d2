"""Tensor-level front end of the C ABI: takes torch device tensors, allocates outputs and
workspaces with the torch allocator, launches on torch's current stream.  Nothing here
computes: every function is one (or a few) calls into libniti_gfx950.so - those that a layer makes on every
step through the native module _host (csrc/host), the others through ctypes."""
from __future__ import annotations

from typing import Optional, Tuple

import torch

from . import _lib as L


def _stream(t: torch.Tensor):
    return torch.cuda.current_stream(t.device).cuda_stream


def _chk_dev(*ts: torch.Tensor) -> None:
    for t in ts:
        if t is None:
            continue
        if not t.is_cuda:
            raise RuntimeError("niti_amd: tensor must live on the GPU")
        if not t.is_contiguous():
            raise RuntimeError("niti_amd: tensor must be contiguous")


def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


def new_scalar_u32(device) -> torch.Tensor:
    """Zeroed device scalar the kernels fold max|x| into (stored as int32 bits of a uint32)."""
    return torch.zeros(1, dtype=torch.int32, device=device)


def _flags(f32_epilogue: bool) -> int:
    return L.EPI_F32_ROUNDTRIP if f32_epilogue else 0


def conv_filter_bytes(w, N, H, W, stride=1, padding=1, dgrad=False) -> int:
    """Bytes of conv_filter_prepare's copy, 0 when the kernels read the filter as stored.  The forward copy's layout depends on
    the filter alone: one copy serves every [N,H,W] for which this is not 0."""
    K, R, S, C = w.shape
    return L.lib().niti_conv2d_i8_filter_workspace(N, H, W, C, K, R, S, stride, padding, int(dgrad))


def conv_filter_prepare(w, N, H, W, stride=1, padding=1, dgrad=False, out=None):
    """Kernel-ready copy of the [K,R,S,C] filter for a convolution over an [N,H,W,*] input (forward) or
    the data gradient of one (dgrad=True).  Returns None when the kernels read the filter as stored.  ``out``: int8 tensor of
    conv_filter_bytes bytes to write instead of a new one."""
    _chk_dev(w, out)
    K, R, S, C = w.shape
    nbytes = conv_filter_bytes(w, N, H, W, stride, padding, dgrad)
    if nbytes == 0:
        return None
    if out is not None and (out.dtype != torch.int8 or out.numel() != nbytes or out.device != w.device):
        raise RuntimeError("conv_filter_prepare: out must be an int8 tensor of %d bytes next to the filter" % nbytes)
    dst = torch.empty(nbytes, dtype=torch.int8, device=w.device) if out is None else out
    st = L.lib().niti_conv2d_i8_filter_prepare(_ptr(w), _ptr(dst), nbytes, N, H, W, C, K, R, S, stride, padding,
                                               int(dgrad), _stream(w))
    L.check(st, "niti_conv2d_i8_filter_prepare")
    return dst


def conv2d_fprop(x, w, stride=1, padding=1, f32_epilogue=False, absmax: Optional[torch.Tensor] = None,
                 prepared_filter=None):
    """x [N,H,W,C] int8, w [K,R,S,C] int8 -> [N,P,Q,K] int32.  ``prepared_filter``: the output of
    conv_filter_prepare(w, N, H, W, stride, padding), to keep the filter copy out of the call."""
    return L.host().conv_fprop(x, w, stride, padding, L.EPI_F32_ROUNDTRIP if f32_epilogue else 0, absmax, prepared_filter)


def conv2d_dgrad(err, w, stride=1, padding=1, f32_epilogue=False, absmax=None, prepared_filter=None, forward_filter=None):
    """err [N,P,Q,K] int8, w [K,R,S,C] int8 -> dx [N,H,W,C] int32 (stride 1).  ``prepared_filter``:
    the output of conv_filter_prepare(w, N, H, W, stride, padding, dgrad=True).  ``forward_filter``: the copy the
    FORWARD pass reads (conv_filter_prepare(.., dgrad=False)), for shapes where both passes run the 3x3 kernel."""
    forward = forward_filter is not None
    return L.host().conv_dgrad(err, w, stride, padding, L.EPI_F32_ROUNDTRIP if f32_epilogue else 0, absmax,
                               forward_filter if forward else prepared_filter, forward)


def conv_requant_sync_words(N, H, W, C, K, R=3, S=3, stride=1, padding=1, dgrad=False) -> int:
    """uint32 words of the sync buffer conv2d_fprop_requant / conv2d_dgrad_requant need for a convolution with
    INPUT [N,H,W,C] and filter [K,R,S,C]; 0 when only the two-pass path (conv2d_* then requant) covers the shape."""
    return int(L.lib().niti_conv2d_i8_requant_sync_words(N, H, W, C, K, R, S, stride, padding, int(dgrad)))


def conv2d_fprop_requant(x, w, stride=1, padding=1, f32_epilogue=False, target_bits=7, method="round", div_mode="floor",
                         bw_mode="int", relu=False, sync=None, shift_out=None, exp_a=None, exp_b=None, exp_out=None,
                         prepared_filter=None, shift_hint=False, pool_out=None, rand=None, any_shape=False):
    """conv2d_fprop + requant as one launch: x [N,H,W,C] int8, w [K,R,S,C] int8 -> ([N,P,Q,K] int8, device shift,
    sync).  method "sto" takes ``rand`` (int32, shaped like the output).  ``pool_out`` ([N,P/2,Q/2,K] int8): also receives the 2x2 / stride-2 maximum of the output.  sync[0] holds max|sum| afterwards, sync[1] != 0 flags a timed-out wait (invalid output).  ``sync``, if
    given, must hold conv_requant_sync_words(...) zeroed int32 words.  ``shift_hint``: ``shift_out`` holds a
    predicted shift on entry (e.g. this tensor's shift of the previous training step); a good prediction saves the
    kernel a second store pass, the results do not depend on it.  ``any_shape``: also batches that are no whole tiles of 256
    pixels (NITI_RQ_ANY_SHAPE)."""
    return L.host().conv_fprop_requant(x, w, stride, padding, f32_epilogue, target_bits, L.ROUND[method], L.DIV[div_mode], L.BW[bw_mode],
                                       relu, shift_hint, sync, shift_out, exp_a, exp_b, exp_out, prepared_filter, False, None, pool_out,
                                       None, 0, rand, any_shape)


def conv2d_fprop_requant_static(x, w, stride=1, padding=1, f32_epilogue=False, target_bits=7, method="round", div_mode="floor",
                                bw_mode="int", relu=False, y=None, shift_out=None, exp_a=None, exp_b=None, exp_out=None,
                                prepared_filter=None, range_out=None):
    """conv2d_fprop_requant through the entry point that takes no scratch memory from the caller (the library keeps its
    sync words and filter copy in a device array of its own): only the tensors given here are touched, and when ``y``,
    ``shift_out`` are passed in nothing is allocated at all.  ``range_out``: int32[2], receives max|sum| and the
    timed-out flag.  Calls on one GPU must not overlap.  Returns (y, shift_out)."""
    _chk_dev(x, w, y, shift_out, exp_a, exp_b, exp_out, prepared_filter, range_out)
    if x.dtype != torch.int8 or w.dtype != torch.int8:
        raise RuntimeError("conv2d_fprop_requant_static: int8 tensors expected")
    N, H, W, C = x.shape
    K, R, S, C2 = w.shape
    if C2 != C:
        raise RuntimeError("conv2d_fprop_requant_static: channel mismatch %d vs %d" % (C, C2))
    P = (H + 2 * padding - R) // stride + 1
    Q = (W + 2 * padding - S) // stride + 1
    if y is None:
        y = torch.empty((N, P, Q, K), dtype=torch.int8, device=x.device)
    elif y.dtype != torch.int8 or tuple(y.shape) != (N, P, Q, K) or not y.is_contiguous():
        raise RuntimeError("conv2d_fprop_requant_static: y must be a contiguous int8 [N,P,Q,K] tensor")
    if shift_out is None:
        shift_out = torch.empty(1, dtype=torch.int32, device=x.device)
    if range_out is not None and (range_out.dtype != torch.int32 or range_out.numel() < 2):
        raise RuntimeError("conv2d_fprop_requant_static: range_out must hold two int32 words")
    flags = _flags(f32_epilogue) | (L.CONV_FILTER_PREPARED if prepared_filter is not None else 0)
    st = L.lib().niti_conv2d_i8_fprop_requant_static(
        _ptr(x), _ptr(prepared_filter if prepared_filter is not None else w), _ptr(y), N, H, W, C, K, R, S, stride, padding, flags,
        target_bits, L.ROUND[method], L.DIV[div_mode], L.BW[bw_mode], L.RQ_RELU if relu else 0, _ptr(shift_out), _ptr(exp_a),
        _ptr(exp_b), _ptr(exp_out), _ptr(range_out), _stream(x))
    L.check(st, "niti_conv2d_i8_fprop_requant_static")
    return y, shift_out


def conv2d_dgrad_requant(err, w, stride=1, padding=1, f32_epilogue=False, target_bits=7, method="round", div_mode="floor",
                         bw_mode="int", sync=None, shift_out=None, exp_a=None, exp_b=None, exp_out=None,
                         prepared_filter=None, relu_mask=None, forward_filter=None, shift_hint=False, unpool=None, rand=None,
                         any_shape=False):
    """conv2d_dgrad + requant as one launch: err [N,P,Q,K] int8, w [K,R,S,C] int8 -> ([N,H,W,C] int8, shift, sync).
    method "sto" takes ``rand`` (int32, shaped like the output; not together with ``unpool``).
    ``unpool`` = (pool_in [N,2H,2W,C] int8, "first" | "all") with ``relu_mask`` = the pooled map: the backward pass of
    the 2x2 / stride-2 max-pool in front of the layer is folded in and the result has pool_in's shape.
    ``relu_mask`` (int8 [N,H,W,C]): results whose mask element is not positive are stored as zero, after range
    and rounding were taken from the unmasked sums (the backward pass of a ReLU in front of the layer).
    ``forward_filter``: the copy the forward pass reads, in place of ``prepared_filter`` (see conv2d_dgrad)."""
    forward = forward_filter is not None
    pool_in, ties = unpool if unpool is not None else (None, "first")
    return L.host().conv_dgrad_requant(err, w, stride, padding, f32_epilogue, target_bits, L.ROUND[method], L.DIV[div_mode], L.BW[bw_mode],
                                       False, shift_hint, sync, shift_out, exp_a, exp_b, exp_out,
                                       forward_filter if forward else prepared_filter, forward, relu_mask, None, pool_in, L.TIES[ties], rand,
                                       any_shape)


def _index(device) -> int:
    dev = torch.device(device)
    return torch.cuda.current_device() if dev.index is None else dev.index


def scratch(nbytes: int, device) -> torch.Tensor:
    """One grow-only int8 buffer per stream for kernel workspaces that live only inside a call.  Calls on one
    stream run in order, so they can all use the same memory - which also keeps the partial sums of
    consecutive weight-gradient launches in the same cache-resident region instead of walking through fresh
    allocations.  Under graph capture: memory of the graph.  The buffers of the sixteen streams used last are kept.  A buffer for
    each stream does not make it safe to run layers on several streams at once: see _SyncArena."""
    return L.host().scratch(nbytes, _index(device))


class _SyncArena:
    """Zeroed int32 words for the single-launch kernels of one training step: one fill per step instead of one
    per kernel.  ``reset`` starts handing out slices from the arena's beginning; ``take`` returns the next slice, zeroed: a
    chunk is filled when its first slice since the reset is taken, so a step pays for the chunks it uses and not for
    those that earlier callers made the arena grow to, and a step captured into a graph contains the fill of every
    chunk it uses.  Slices are handed out once per reset, so a kernel never sees words another kernel of the
    same step wrote.  An arena that runs out (or was never reset) grows by another chunk; ``timed_out`` covers every
    slice handed out since the last reset.  Every stream, and every stream capture, has an arena of its own
    (csrc/host/host.cpp; those of the sixteen streams used last are kept); reset and take work on the current stream's.

    Not for several streams at once: a launch that exchanges its range waits for all of its workgroups, so it must have the
    device to itself.  Two such launches that run side by side can each hold compute units that the other's workgroups wait
    for; both then give up at the wait limit (2 s) with wrong shifts, which ``timed_out`` and ``sync_timeouts`` report.
    Streams that take turns (an event or wait_stream between them) are fine."""

    def reset(self, device):
        L.host().arena_reset(_index(device))

    def take(self, words, device):
        return L.host().arena_take(words, _index(device))

    def timed_out(self, device) -> bool:
        """True if a single-launch kernel that used a slice since the last reset flagged that its grid-wide wait ran
        into the time limit (its output is then invalid).  Copies the flags to the host: for the end of a step or an
        epoch, not for the inner loop."""
        flags = L.host().arena_flags(_index(device))
        if not flags:
            return False
        return bool(torch.cat(flags).ne(0).any().item())


def sync_timeouts(device=None, clear=True) -> bool:
    """True if any grid-wide wait of the library's kernels on ``device`` gave up since the flag was last cleared
    (niti_sync_timeouts): some int8 output or weight update since then was made with a wrong shift.  Unlike
    ``sync_arena.timed_out`` this survives the arena's resets.  Waits for the device's current stream."""
    import ctypes
    dev = torch.device("cuda", torch.cuda.current_device()) if device is None else torch.device(device)
    flag = ctypes.c_uint32(0)
    with torch.cuda.device(dev):
        st = L.lib().niti_sync_timeouts(ctypes.byref(flag), int(clear), torch.cuda.current_stream(dev).cuda_stream)
    L.check(st, "niti_sync_timeouts")
    return flag.value != 0


sync_arena = _SyncArena()


def conv2d_wgrad(act, err, R, S, stride=1, padding=1, f32_epilogue=False, absmax=None, workspace=None):
    """act [N,H,W,C] int8, err [N,P,Q,K] int8 -> dw [K,R,S,C] int32 (stride 1).  ``workspace``: int8 tensor of
    at least niti_conv2d_i8_wgrad_workspace bytes (default: the stream's scratch buffer)."""
    return L.host().conv_wgrad(act, err, R, S, stride, padding, L.EPI_F32_ROUNDTRIP if f32_epilogue else 0, absmax, workspace)


def wgrad_update_sync_words(N, H, W, C, K, R=3, S=3, stride=1, padding=1) -> int:
    """uint32 words of the sync buffer conv2d_wgrad_update needs; 0 when only the two-pass path covers the shape."""
    return int(L.lib().niti_conv2d_i8_wgrad_update_sync_words(N, H, W, C, K, R, S, stride, padding))


def conv2d_wgrad_update(act, err, w, stride=1, padding=1, f32_epilogue=False, mu=5, method="psto", div_mode="floor",
                        bw_mode="int", sync=None, want_grad=False, want_dw=False, shift_out=None, exp_a=None, exp_b=None,
                        exp_out=None, workspace=None, prepared_filter=None, shift_hint=False, any_kernel=False):
    """Weight gradient + grad_calc + weight update: act [N,H,W,C] int8 (C may carry zero channel padding), err
    [N,H,W,K] int8, w [K,3,3,Cw] int8 updated in place.  Returns (g8 or None, dw int32 or None, device shift, sync).
    ``prepared_filter``: conv_filter_prepare(w padded to C channels, N, H, W) made earlier; it receives the updated
    weights too and stays valid for the next forward pass.  ``shift_hint``: ``shift_out`` holds a predicted shift
    on entry (the previous step's): the update's stores then overlap the wait for the tensor's range.  ``any_kernel``: small
    batches may run on the kernel for any shape (NITI_CONV_ANY_KERNEL)."""
    if shift_hint and shift_out is None:
        raise RuntimeError("conv2d_wgrad_update: shift_hint needs shift_out, holding the predicted shift")
    flags = (L.EPI_F32_ROUNDTRIP if f32_epilogue else 0) | (L.CONV_SHIFT_HINT if shift_hint else 0) | (L.CONV_ANY_KERNEL if any_kernel else 0)
    return L.host().conv_wgrad_update(act, err, w, stride, padding, flags, mu, L.ROUND[method], L.DIV[div_mode], L.BW[bw_mode], sync,
                                      want_grad, want_dw, shift_out, exp_a, exp_b, exp_out, workspace, prepared_filter)


def conv2d_backward(err, act, w, padding=1, f32_epilogue=False, err_bits=7, err_method="round", mu=5, grad_method="psto", div_mode="floor",
                    bw_mode="int", relu_mask=None, pool_in=None, ties="first", err_rand=None, want_grad=False, exp_err=None, exp_w=None,
                    exp_act=None, prepared_filter=None, err_shift=None, grad_shift=None):
    """TiConv2d.backward (ti_torch.py:404-437), stride 1: err [N,P,Q,K], act [N,H,W,C], w [K,R,S,C] int8, w updated in place behind the
    data gradient that reads it; both gradients in one call of the library where that is the faster way.  ``pool_in``: relu_mask is the output of
    a 2x2 / stride-2 max-pool on it, the error comes back at its size (element 2 of the result says whether it did).
    ``err_shift`` / ``grad_shift``: predicted shifts, overwritten with the actual ones.
    Returns (error, its exponent, unpooled?, int8 gradient or None, int32 gradient or None, gradient shift, gradient exponent, one call?)."""
    return L.host().conv_layer_backward(True, err, act, w, 1, padding, f32_epilogue, err_bits, L.ROUND[err_method], L.DIV[div_mode], L.BW[bw_mode],
                                        err_shift, exp_err, exp_w, prepared_filter, relu_mask, pool_in, L.TIES[ties], err_rand, mu,
                                        L.ROUND[grad_method], want_grad, False, grad_shift, exp_act, prepared_filter, None)


def gemm(a, b, trans_a=False, trans_b=False, absmax=None, out=None, f32_epilogue=False):
    """c[m,n] = op(a) @ op(b), int8 x int8 -> int32.  trans_a: a stored [k,m]; trans_b: b stored [n,k].
    f32_epilogue: every sum takes the int32 -> float32 -> int32 round trip of the reference's convolution epilogue."""
    return L.host().gemm(a, b, trans_a, trans_b, absmax, out, L.EPI_F32_ROUNDTRIP if f32_epilogue else 0)


def absmax_i32(x, absmax=None):
    return L.host().absmax_i32(x, absmax)


def requant(x, absmax, target_bits=7, method="round", div_mode="floor", bw_mode="int", rand=None, relu=False,
            shift_out=None, exp_a=None, exp_b=None, exp_out=None):
    """int32 -> int8 (act_calc / err_calc / grad_calc).  Returns (int8 tensor, device int32 shift).
    exp_out (device int32), when given, receives shift + exp_a + exp_b."""
    _chk_dev(x, absmax, rand, shift_out, exp_a, exp_b, exp_out)
    if x.dtype != torch.int32:
        raise RuntimeError("requant: int32 input expected")
    if rand is not None and (rand.dtype != torch.int32 or rand.numel() != x.numel()):
        raise RuntimeError("requant: rand must be int32 with one entry per element")
    y = torch.empty(x.shape, dtype=torch.int8, device=x.device)
    if shift_out is None:
        shift_out = torch.empty(1, dtype=torch.int32, device=x.device)
    st = L.lib().niti_requant_i32_i8(_ptr(x), _ptr(y), x.numel(), _ptr(absmax), target_bits, L.ROUND[method],
                                     L.DIV[div_mode], L.BW[bw_mode], _ptr(rand), L.RQ_RELU if relu else 0,
                                     _ptr(shift_out), _ptr(exp_a), _ptr(exp_b), _ptr(exp_out), _stream(x))
    L.check(st, "niti_requant_i32_i8")
    return y, shift_out


def grad_update(g, w, absmax, mu, method="psto", div_mode="floor", bw_mode="int", rand=None, want_grad=False,
                shift_out=None, exp_a=None, exp_b=None, exp_out=None):
    """Fused grad_calc + weight update, in place on w.  Returns (int8 grad or None, device shift)."""
    _chk_dev(g, w, absmax, rand, shift_out, exp_a, exp_b, exp_out)
    if g.dtype != torch.int32 or w.dtype != torch.int8 or g.numel() != w.numel():
        raise RuntimeError("grad_update: int32 grad and int8 weight of equal size expected")
    g8 = torch.empty(w.shape, dtype=torch.int8, device=w.device) if want_grad else None
    if shift_out is None:
        shift_out = torch.empty(1, dtype=torch.int32, device=w.device)
    st = L.lib().niti_grad_update_i8(_ptr(g), _ptr(w), g.numel(), _ptr(absmax), mu, L.ROUND[method], L.DIV[div_mode],
                                     L.BW[bw_mode], _ptr(rand), _ptr(g8), _ptr(shift_out), _ptr(exp_a), _ptr(exp_b),
                                     _ptr(exp_out), _stream(g))
    L.check(st, "niti_grad_update_i8")
    return g8, shift_out


def _chk_bytes(t, nbytes, who):
    """A launch reads ``nbytes`` of ``t``."""
    if t.numel() * t.element_size() < nbytes:
        raise RuntimeError("%s: a tensor of %d bytes expected, got %d" % (who, nbytes, t.numel() * t.element_size()))


def weight_update(w, g):
    _chk_dev(w, g)
    _chk_bytes(g, w.numel(), "weight_update")
    st = L.lib().niti_weight_update_i8(_ptr(w), _ptr(g), w.numel(), _stream(w))
    L.check(st, "niti_weight_update_i8")
    return w


def relu_fwd(x):
    _chk_dev(x)
    y = torch.empty_like(x)
    L.check(L.lib().niti_relu_i8_fwd(_ptr(x), _ptr(y), x.numel(), _stream(x)), "niti_relu_i8_fwd")
    return y


def quantize_input(x, bits=7, cpad=16, out=None, exp_out=None, target=None, target_out=None, start_step=False):
    """Float NCHW batch -> (int8 NHWC batch with the channels zero-padded to ``cpad``, exponent as a 1-element int32
    tensor): the reference's input quantiser and the layout change behind it in two launches (one for a few images).
    ``out`` / ``exp_out``: tensors to write instead of new ones; ``target`` (int64) is copied to ``target_out`` on the way."""
    return L.host().quantize_input(x, bits, cpad, out, exp_out, target, target_out, start_step)


def batch_metrics(out_val, out_exp, target, sums):
    """sums (float64 [3]) += batch size x (display loss, top-1 %, top-5 %) of int8 logits [n, classes >= 5] with exponent
    ``out_exp`` (1-element int32 device tensor), in one launch.  Targets of -100 are left out of the loss's mean and hit
    nothing; any other target outside the classes makes all three sums NaN."""
    _chk_dev(out_val, out_exp, target, sums)
    n, classes = out_val.shape
    if (out_val.dtype != torch.int8 or out_exp.dtype != torch.int32 or target.dtype != torch.int64 or target.numel() != n
            or sums.dtype != torch.float64 or sums.numel() != 3):
        raise RuntimeError("batch_metrics: int8 logits [n, classes], int32 exponent, int64 targets [n] and float64 sums [3] expected")
    L.check(L.lib().niti_batch_metrics_i8(_ptr(out_val), _ptr(out_exp), _ptr(target), n, classes, _ptr(sums), _stream(out_val)),
            "niti_batch_metrics_i8")


def mask_features(x, mask, exp_in=None, exp_add=None):
    """x [rows, F] int8 times a keep / drop byte per feature (mask [F] int8 0/1) in one launch.  With ``exp_add`` also
    returns a 1-element int32 tensor holding exp_in + exp_add."""
    _chk_dev(x, mask, exp_in)
    if x.dtype != torch.int8 or mask.dtype != torch.int8 or x.dim() != 2 or mask.numel() != x.shape[1]:
        raise RuntimeError("mask_features: int8 [rows, F] tensor and int8 [F] mask expected")
    if exp_in is not None and exp_in.numel() != 1:
        raise RuntimeError("mask_features: an exponent is one value")
    y = torch.empty_like(x)
    exp_out = torch.empty(1, dtype=torch.int32, device=x.device) if exp_add is not None else None
    L.check(L.lib().niti_mask_features_i8(_ptr(x), _ptr(mask), _ptr(y), x.shape[0], x.shape[1], _ptr(exp_in), _ptr(exp_out),
                                         int(exp_add or 0), _stream(x)), "niti_mask_features_i8")
    return (y, exp_out) if exp_add is not None else y


def relu_bwd(act, dy):
    _chk_dev(act, dy)
    _chk_bytes(act, dy.numel(), "relu_bwd")
    dx = torch.empty_like(dy)
    L.check(L.lib().niti_relu_i8_bwd(_ptr(act), _ptr(dy), _ptr(dx), dy.numel(), _stream(dy)), "niti_relu_i8_bwd")
    return dx


FC_PASS = {"forward": 0, "dgrad": 1, "wgrad": 2}


def fc_sync_words(which, M, O, F) -> int:
    """uint32 sync words the one-launch TiLinear kernels need for act [M,F], weight [O,F]; 0 when the shape is
    outside them (more than 16 output features, ...) and the GEMM entry point has to be used."""
    return int(L.lib().niti_fc_i8_sync_words(FC_PASS[which], M, O, F))


def _fc_sync(which, M, O, F, sync, device, who):
    words = fc_sync_words(which, M, O, F)
    if words == 0:
        raise L.NitiError("%s: shape not covered by the few-output-features kernels" % who)
    if sync is None:
        sync = sync_arena.take(words, device)
    elif sync.dtype != torch.int32 or sync.numel() < words:
        raise RuntimeError("%s: sync must be a zeroed int32 tensor of at least %d words" % (who, words))
    return sync


def fc_fwd_requant(act, w, target_bits=7, method="round", div_mode="floor", bw_mode="int", relu=False, sync=None,
                   shift_out=None, exp_a=None, exp_b=None, exp_out=None):
    """act_calc(act @ w^T) as one launch: act [M,F] int8, w [O,F] int8 (O <= 16) -> ([M,O] int8, shift, sync)."""
    _chk_dev(act, w, sync, shift_out, exp_a, exp_b, exp_out)
    if act.dtype != torch.int8 or w.dtype != torch.int8 or act.dim() != 2 or w.dim() != 2 or act.shape[1] != w.shape[1]:
        raise RuntimeError("fc_fwd_requant: int8 act [M,F] and w [O,F] expected")
    M, F = act.shape
    O = w.shape[0]
    sync = _fc_sync("forward", M, O, F, sync, act.device, "fc_fwd_requant")
    out = torch.empty((M, O), dtype=torch.int8, device=act.device)
    if shift_out is None:
        shift_out = torch.empty(1, dtype=torch.int32, device=act.device)
    st = L.lib().niti_fc_i8_fwd_requant(_ptr(act), _ptr(w), _ptr(out), M, O, F, target_bits, L.ROUND[method], L.DIV[div_mode],
                                        L.BW[bw_mode], L.RQ_RELU if relu else 0, _ptr(sync), sync.numel(), _ptr(shift_out),
                                        _ptr(exp_a), _ptr(exp_b), _ptr(exp_out), _stream(act))
    L.check(st, "niti_fc_i8_fwd_requant")
    return out, shift_out, sync


def fc_dgrad_requant(err, w, target_bits=7, method="round", div_mode="floor", bw_mode="int", sync=None, shift_out=None,
                     exp_a=None, exp_b=None, exp_out=None):
    """err_calc(err @ w) as one launch: err [M,O] int8, w [O,F] int8 (O <= 16) -> ([M,F] int8, shift, sync)."""
    _chk_dev(err, w, sync, shift_out, exp_a, exp_b, exp_out)
    if err.dtype != torch.int8 or w.dtype != torch.int8 or err.dim() != 2 or w.dim() != 2 or err.shape[1] != w.shape[0]:
        raise RuntimeError("fc_dgrad_requant: int8 err [M,O] and w [O,F] expected")
    M, O = err.shape
    F = w.shape[1]
    sync = _fc_sync("dgrad", M, O, F, sync, err.device, "fc_dgrad_requant")
    dx = torch.empty((M, F), dtype=torch.int8, device=err.device)
    if shift_out is None:
        shift_out = torch.empty(1, dtype=torch.int32, device=err.device)
    st = L.lib().niti_fc_i8_dgrad_requant(_ptr(err), _ptr(w), _ptr(dx), M, O, F, target_bits, L.ROUND[method], L.DIV[div_mode],
                                          L.BW[bw_mode], _ptr(sync), sync.numel(), _ptr(shift_out), _ptr(exp_a), _ptr(exp_b),
                                          _ptr(exp_out), _stream(err))
    L.check(st, "niti_fc_i8_dgrad_requant")
    return dx, shift_out, sync


def fc_wgrad_update(err, act, w, mu=5, method="psto", div_mode="floor", bw_mode="int", sync=None, want_grad=False,
                    shift_out=None, exp_a=None, exp_b=None, exp_out=None):
    """g = grad_calc(err^T @ act, mu); w = clip(w - g) in place, as one launch: err [M,O], act [M,F], w [O,F] int8
    (O <= 16, M <= 512) -> (g as int8 [O,F] if want_grad else None, shift, sync)."""
    _chk_dev(err, act, w, sync, shift_out, exp_a, exp_b, exp_out)
    if err.dtype != torch.int8 or act.dtype != torch.int8 or w.dtype != torch.int8 or err.dim() != 2 or act.dim() != 2 \
            or tuple(w.shape) != (err.shape[1], act.shape[1]) or err.shape[0] != act.shape[0]:
        raise RuntimeError("fc_wgrad_update: int8 err [M,O], act [M,F] and w [O,F] expected")
    M, O = err.shape
    F = act.shape[1]
    sync = _fc_sync("wgrad", M, O, F, sync, err.device, "fc_wgrad_update")
    g8 = torch.empty_like(w) if want_grad else None
    if shift_out is None:
        shift_out = torch.empty(1, dtype=torch.int32, device=err.device)
    st = L.lib().niti_fc_i8_wgrad_update(_ptr(err), _ptr(act), _ptr(w), M, O, F, mu, L.ROUND[method], L.DIV[div_mode],
                                         L.BW[bw_mode], _ptr(sync), sync.numel(), _ptr(g8), _ptr(shift_out), _ptr(exp_a),
                                         _ptr(exp_b), _ptr(exp_out), _stream(err))
    L.check(st, "niti_fc_i8_wgrad_update")
    return g8, shift_out, sync


def linear_sync_words(which, M, O, F) -> int:
    """uint32 words of the sync buffer the any-width TiLinear kernels need for a pass ("forward", "dgrad", "wgrad") on
    the current device; 0 when the shape is outside them (then: gemm + requant / grad_update)."""
    return int(L.lib().niti_linear_i8_sync_words({"forward": 0, "dgrad": 1, "wgrad": 2}[which], M, O, F))


def _linear_sync(which, M, O, F, sync, device, who):
    words = linear_sync_words(which, M, O, F)
    if words == 0:
        raise L.NitiError("%s: shape not covered by the any-width linear kernels" % who)
    if sync is None:
        sync = sync_arena.take(words, device)
    elif sync.dtype != torch.int32 or sync.numel() < words:
        raise RuntimeError("%s: sync must be a zeroed int32 tensor of at least %d words" % (who, words))
    return sync


def _chk_linear(rows, inner, w, who):
    """Rows [M,features] against weights [O,F] along whose dimension ``inner`` they are multiplied."""
    if rows.dim() != 2 or w.dim() != 2 or rows.shape[1] != w.shape[inner]:
        raise RuntimeError("%s: rows %s do not go with weights %s" % (who, tuple(rows.shape), tuple(w.shape)))


def _chk_rand(rand, shape, who):
    if rand is not None and (rand.dtype != torch.int32 or tuple(rand.shape) != tuple(shape) or not rand.is_contiguous()):
        raise RuntimeError("%s: rand must be a contiguous int32 tensor shaped like the output" % who)


def linear_fwd_requant(act, w, target_bits=7, method="round", div_mode="floor", bw_mode="int", relu=False, rand=None, sync=None,
                       shift_out=None, exp_a=None, exp_b=None, exp_out=None):
    """act_calc(act @ w^T) in one launch for a layer of any width: act [M,F] int8, w [O,F] int8 -> ([M,O] int8, shift,
    sync).  ``rand`` (int32 [M,O]) for method "sto"."""
    _chk_dev(act, w, rand, sync, shift_out, exp_a, exp_b, exp_out)
    _chk_linear(act, 1, w, "linear_fwd_requant")
    M, F = act.shape
    O = w.shape[0]
    _chk_rand(rand, (M, O), "linear_fwd_requant")
    sync = _linear_sync("forward", M, O, F, sync, act.device, "linear_fwd_requant")
    y = torch.empty((M, O), dtype=torch.int8, device=act.device)
    if shift_out is None:
        shift_out = torch.empty(1, dtype=torch.int32, device=act.device)
    L.check(L.lib().niti_linear_i8_fwd_requant(_ptr(act), _ptr(w), _ptr(y), M, O, F, target_bits, L.ROUND[method], L.DIV[div_mode],
                                               L.BW[bw_mode], L.RQ_RELU if relu else 0, _ptr(rand), _ptr(sync), sync.numel(),
                                               _ptr(shift_out), _ptr(exp_a), _ptr(exp_b), _ptr(exp_out), _stream(act)),
            "niti_linear_i8_fwd_requant")
    return y, shift_out, sync


def linear_dgrad_requant(err, w, target_bits=7, method="round", div_mode="floor", bw_mode="int", rand=None, sync=None,
                         shift_out=None, exp_a=None, exp_b=None, exp_out=None):
    """err_calc(err @ w) in one launch: err [M,O] int8, w [O,F] int8 -> ([M,F] int8, shift, sync)."""
    _chk_dev(err, w, rand, sync, shift_out, exp_a, exp_b, exp_out)
    _chk_linear(err, 0, w, "linear_dgrad_requant")
    M, O = err.shape
    F = w.shape[1]
    _chk_rand(rand, (M, F), "linear_dgrad_requant")
    sync = _linear_sync("dgrad", M, O, F, sync, err.device, "linear_dgrad_requant")
    y = torch.empty((M, F), dtype=torch.int8, device=err.device)
    if shift_out is None:
        shift_out = torch.empty(1, dtype=torch.int32, device=err.device)
    L.check(L.lib().niti_linear_i8_dgrad_requant(_ptr(err), _ptr(w), _ptr(y), M, O, F, target_bits, L.ROUND[method], L.DIV[div_mode],
                                                 L.BW[bw_mode], _ptr(rand), _ptr(sync), sync.numel(), _ptr(shift_out), _ptr(exp_a),
                                                 _ptr(exp_b), _ptr(exp_out), _stream(err)), "niti_linear_i8_dgrad_requant")
    return y, shift_out, sync


def linear_wgrad_update(err, act, w, mu=5, method="psto", div_mode="floor", bw_mode="int", rand=None, sync=None, want_grad=False,
                        shift_out=None, exp_a=None, exp_b=None, exp_out=None):
    """grad_calc(err^T @ act) and the weight update in one launch: err [M,O], act [M,F], w [O,F] int8 updated in place.
    Returns (int8 gradient or None, shift, sync)."""
    _chk_dev(err, act, w, rand, sync, shift_out, exp_a, exp_b, exp_out)
    _chk_linear(err, 0, w, "linear_wgrad_update")
    _chk_linear(act, 1, w, "linear_wgrad_update")
    if act.shape[0] != err.shape[0]:
        raise RuntimeError("linear_wgrad_update: %d errors for %d rows of activations" % (err.shape[0], act.shape[0]))
    M, O = err.shape
    F = act.shape[1]
    _chk_rand(rand, (O, F), "linear_wgrad_update")
    sync = _linear_sync("wgrad", M, O, F, sync, err.device, "linear_wgrad_update")
    g8 = torch.empty((O, F), dtype=torch.int8, device=w.device) if want_grad else None
    if shift_out is None:
        shift_out = torch.empty(1, dtype=torch.int32, device=w.device)
    L.check(L.lib().niti_linear_i8_wgrad_update(_ptr(err), _ptr(act), _ptr(w), M, O, F, mu, L.ROUND[method], L.DIV[div_mode],
                                                L.BW[bw_mode], _ptr(rand), _ptr(sync), sync.numel(), _ptr(g8), _ptr(shift_out),
                                                _ptr(exp_a), _ptr(exp_b), _ptr(exp_out), _stream(err)), "niti_linear_i8_wgrad_update")
    return g8, shift_out, sync


def linear_backward(err, act, w, err_bits=7, err_method="round", mu=5, grad_method="psto", div_mode="floor", bw_mode="int", err_rand=None,
                    grad_rand=None, want_grad=False, exp_err=None, exp_w=None, exp_act=None):
    """TiLinear.backward (ti_torch.py:249-266): err [M,O], act [M,F], w [O,F] int8, w updated in place behind the data gradient that
    reads it; one launch where both gradients' workgroups fit on the device together.  Returns (error [M,F] int8, its exponent,
    int8 gradient or None, int32 gradient or None, gradient shift, gradient exponent)."""
    _chk_dev(err, act, w, err_rand, grad_rand, exp_err, exp_w, exp_act)
    return L.host().linear_backward(True, err, act, w, err_bits, L.ROUND[err_method], mu, L.ROUND[grad_method], L.DIV[div_mode], L.BW[bw_mode],
                                    want_grad, False, exp_err, exp_w, exp_act, err_rand, grad_rand)


def pad_last_dim(t, multiple=16):
    """``t`` with zeros appended along its last dimension up to a multiple of ``multiple`` (``t`` itself when it
    already is one): the channel padding of conv2d_int8 (ti_torch.py:182-187) as one launch."""
    c = t.shape[-1]
    if c % multiple == 0:
        return t
    _chk_dev(t)
    if t.dtype != torch.int8:
        raise RuntimeError("pad_last_dim: int8 tensor expected")
    cp = (c + multiple - 1) // multiple * multiple
    out = torch.empty(tuple(t.shape[:-1]) + (cp,), dtype=torch.int8, device=t.device)
    L.check(L.lib().niti_pad_rows_i8(_ptr(t), _ptr(out), t.numel() // c, c, cp, _stream(t)), "niti_pad_rows_i8")
    return out


def loss_grad(out_val, out_exp, target, rand, div_mode="floor"):
    """TiLoss.forward (ti_loss.py:5-36) as one launch: int8 logits [n, classes] with exponent ``out_exp`` (1-element
    int32 device tensor), int64 targets [n], int32 random integers [n, classes] -> int8 gradient (exponent 0)."""
    _chk_dev(out_val, out_exp, target, rand)
    if out_val.dtype != torch.int8 or out_val.dim() != 2 or not out_val.is_contiguous():
        raise RuntimeError("loss_grad: contiguous int8 [n, classes] logits expected")
    if out_exp.dtype != torch.int32 or target.dtype != torch.int64 or rand.dtype != torch.int32:
        raise RuntimeError("loss_grad: int32 exponent, int64 targets and int32 random integers expected")
    n, classes = out_val.shape
    if target.numel() != n or tuple(rand.shape) != (n, classes) or not rand.is_contiguous() or not target.is_contiguous():
        raise RuntimeError("loss_grad: shape mismatch")
    grad = torch.empty_like(out_val)
    st = L.lib().niti_loss_grad_i8(_ptr(out_val), _ptr(out_exp), _ptr(target), _ptr(rand), _ptr(grad), n, classes,
                                   L.DIV[div_mode], _stream(out_val))
    L.check(st, "niti_loss_grad_i8")
    return grad


def loss_grad_rng(out_val, out_exp, target, rng, div_mode="floor"):
    """``loss_grad`` with the random integers drawn in the kernel from the generator state ``rng`` (see rng_state)."""
    _chk_dev(out_val, out_exp, target, rng)
    if out_val.dtype != torch.int8 or out_val.dim() != 2 or not out_val.is_contiguous():
        raise RuntimeError("loss_grad_rng: contiguous int8 [n, classes] logits expected")
    if out_exp.dtype != torch.int32 or target.dtype != torch.int64 or target.numel() != out_val.shape[0] or not target.is_contiguous():
        raise RuntimeError("loss_grad_rng: int32 exponent and int64 targets [n] expected")
    _check_rng(rng, "loss_grad_rng")
    n, classes = out_val.shape
    grad = torch.empty_like(out_val)
    L.check(L.lib().niti_loss_grad_i8_rng(_ptr(out_val), _ptr(out_exp), _ptr(target), _ptr(rng), _ptr(grad), n, classes,
                                          L.DIV[div_mode], _stream(out_val)), "niti_loss_grad_i8_rng")
    return grad


RNG_STREAM = {"dropout": 1, "loss": 2}
_rng_states = {}


def _check_rng(rng, who):
    if rng.dtype != torch.int32 or rng.numel() != 4 or not rng.is_contiguous() or not rng.is_cuda:
        raise RuntimeError("%s: the generator state is a contiguous int32 tensor of 4 words on the GPU" % who)


def rng_state(device=None, key=None):
    """Generator state for the kernels that draw their own random integers (dropout mask, loss gradient rounding):
    int32[4] = {key0, key1, step, 0}.  Without ``key`` returns the device's shared state, created on first use with
    a key taken from torch's default CPU generator (so ``torch.manual_seed`` fixes the sequence); with ``key`` (an
    int, 64 bits used) a fresh state at step 0.  Creating a state copies to the device: not under graph capture."""
    dev = torch.device("cuda", torch.cuda.current_device()) if device is None else torch.device(device)
    if dev.index is None:
        dev = torch.device("cuda", torch.cuda.current_device())
    if key is None:
        if str(dev) not in _rng_states:
            if torch.cuda.is_current_stream_capturing():
                raise RuntimeError("rng_state: first use under graph capture; run one step eagerly first")
            k = int(torch.empty((), dtype=torch.int64).random_().item())
            _rng_states[str(dev)] = rng_state(dev, k)
        return _rng_states[str(dev)]
    words = [key & 0xFFFFFFFF, (key >> 32) & 0xFFFFFFFF, 0, 0]
    return torch.tensor([w - (1 << 32) if w >= (1 << 31) else w for w in words], dtype=torch.int32).to(dev)


def rng_words(rng, stream, n):
    """The first ``n`` words (int32 tensor, to be read as unsigned) of stream "dropout" / "loss" that a kernel launched
    now would draw from ``rng``; the state is not advanced."""
    _check_rng(rng, "rng_words")
    out = torch.empty(n, dtype=torch.int32, device=rng.device)
    L.check(L.lib().niti_rng_words_u32(_ptr(rng), RNG_STREAM[stream] if isinstance(stream, str) else int(stream), _ptr(out), n,
                                       _stream(rng)), "niti_rng_words_u32")
    return out


def head_sync_words(which, M, O, F) -> int:
    """uint32 sync words of the classifier-head kernels ("forward" / "backward"); 0 = shape not covered."""
    return int(L.lib().niti_head_i8_sync_words(1 if which == "backward" else 0, M, O, F))


def head_forward(act, w, target_bits=7, method="round", div_mode="floor", bw_mode="int", relu=False, dropout=None,
                 drop_mask=None, rng=None, exp_bias=0, target=None, loss_rand=None, sync=None, shift_out=None, exp_a=None,
                 exp_b=None, exp_out=None):
    """Classifier forward in one launch (niti_head_i8_forward): act_calc((act * mask) @ w^T) for act [M,F], w [O,F],
    O <= 16.  ``dropout``: None, "given" (``drop_mask`` int8 [F] of 0 / 1 is read) or "draw" (the mask is drawn from
    ``rng`` and written to ``drop_mask``, allocated here when None).  With ``target`` (int64 [M]) the loss gradient
    of the logits is computed as well, rounded with ``loss_rand`` (int32 [M,O]) or with draws from ``rng``.
    Returns (out8 [M,O], drop_mask or None, loss gradient [M,O] or None, shift, sync)."""
    _chk_dev(act, w, sync, shift_out, exp_a, exp_b, exp_out, drop_mask, rng, target, loss_rand)
    if act.dtype != torch.int8 or w.dtype != torch.int8 or act.dim() != 2 or w.dim() != 2 or act.shape[1] != w.shape[1]:
        raise RuntimeError("head_forward: int8 act [M,F] and w [O,F] expected")
    if not act.is_contiguous() or not w.is_contiguous():
        raise RuntimeError("head_forward: contiguous operands expected")
    M, F = act.shape
    O = w.shape[0]
    mode = {None: 0, "given": 1, "draw": 2}[dropout]
    if mode == 2 and drop_mask is None:
        drop_mask = torch.empty(F, dtype=torch.int8, device=act.device)
    if mode != 0 and (drop_mask is None or drop_mask.dtype != torch.int8 or drop_mask.numel() != F or not drop_mask.is_contiguous()):
        raise RuntimeError("head_forward: drop_mask must be a contiguous int8 tensor of F elements")
    if rng is not None:
        _check_rng(rng, "head_forward")
    loss_grad_out = None
    if target is not None:
        if target.dtype != torch.int64 or target.numel() != M or not target.is_contiguous():
            raise RuntimeError("head_forward: int64 targets [M] expected")
        if loss_rand is not None and (loss_rand.dtype != torch.int32 or tuple(loss_rand.shape) != (M, O) or not loss_rand.is_contiguous()):
            raise RuntimeError("head_forward: loss_rand must be a contiguous int32 [M,O] tensor")
        loss_grad_out = torch.empty((M, O), dtype=torch.int8, device=act.device)
    words = head_sync_words("forward", M, O, F)
    if words == 0:
        raise L.NitiError("head_forward: shape not covered by the few-output-features kernels")
    if sync is None:
        sync = sync_arena.take(words, act.device)
    elif sync.dtype != torch.int32 or sync.numel() < words:
        raise RuntimeError("head_forward: sync must be a zeroed int32 tensor of at least %d words" % words)
    out = torch.empty((M, O), dtype=torch.int8, device=act.device)
    if shift_out is None:
        shift_out = torch.empty(1, dtype=torch.int32, device=act.device)
    st = L.lib().niti_head_i8_forward(_ptr(act), _ptr(w), _ptr(out), M, O, F, mode, _ptr(drop_mask) if mode else None, _ptr(rng),
                                      int(exp_bias), _ptr(target), _ptr(loss_rand), _ptr(loss_grad_out), target_bits,
                                      L.ROUND[method], L.DIV[div_mode], L.BW[bw_mode], L.RQ_RELU if relu else 0, _ptr(sync),
                                      sync.numel(), _ptr(shift_out), _ptr(exp_a), _ptr(exp_b), _ptr(exp_out), _stream(act))
    L.check(st, "niti_head_i8_forward")
    return out, (drop_mask if mode else None), loss_grad_out, shift_out, sync


def head_backward(err, act, w, err_bits=7, err_method="psto", grad_bits=5, grad_method="psto", div_mode="floor", bw_mode="int",
                  drop_mask=None, want_grad=False, sync=None, exp_err=None, exp_w=None, exp_act=None, exp_act_bias=0,
                  err_exp_out=None, grad_exp_out=None, unpool=None):
    """Classifier backward in one launch (niti_head_i8_backward): err [M,O], act [M,F] (in front of the dropout),
    w [O,F] (updated in place), ``drop_mask`` int8 [F] of 0 / 1 or None.  Returns (dx8 [M,F] with the mask applied,
    rounded gradient [O,F] or None, err shift, grad shift, sync).
    ``unpool`` = (pool_in [M,2P,2Q,C], ties, relu): act is the flattened output of a 2 x 2 max-pool over pool_in; the launch
    also routes dx8 through that pool's backward pass (niti_head_i8_backward_unpool) and a sixth element is returned:
    the gradient [M,2P,2Q,C]."""
    _chk_dev(err, act, w, drop_mask, sync, exp_err, exp_w, exp_act, err_exp_out, grad_exp_out)
    if (err.dtype != torch.int8 or act.dtype != torch.int8 or w.dtype != torch.int8 or err.dim() != 2 or act.dim() != 2
            or w.dim() != 2 or err.shape[0] != act.shape[0] or tuple(w.shape) != (err.shape[1], act.shape[1])):
        raise RuntimeError("head_backward: int8 err [M,O], act [M,F], w [O,F] expected")
    if not (err.is_contiguous() and act.is_contiguous() and w.is_contiguous()):
        raise RuntimeError("head_backward: contiguous operands expected")
    M, O = err.shape
    F = act.shape[1]
    if drop_mask is not None and (drop_mask.dtype != torch.int8 or drop_mask.numel() != F or not drop_mask.is_contiguous()):
        raise RuntimeError("head_backward: drop_mask must be a contiguous int8 tensor of F elements")
    words = head_sync_words("backward", M, O, F)
    if words == 0:
        raise L.NitiError("head_backward: shape not covered (M <= 256, O <= 16, F a multiple of 64)")
    if sync is None:
        sync = sync_arena.take(words, err.device)
    elif sync.dtype != torch.int32 or sync.numel() < words:
        raise RuntimeError("head_backward: sync must be a zeroed int32 tensor of at least %d words" % words)
    dx = torch.empty((M, F), dtype=torch.int8, device=err.device)
    g8 = torch.empty_like(w) if want_grad else None
    shifts = torch.empty(2, dtype=torch.int32, device=err.device)
    if unpool is not None:
        pool_in, ties, relu = unpool
        _chk_dev(pool_in)
        if pool_in.dtype != torch.int8 or pool_in.dim() != 4 or not pool_in.is_contiguous() or pool_in.shape[0] != M:
            raise RuntimeError("head_backward: unpool wants the pool's contiguous int8 input [M,2P,2Q,C]")
        H2, W2, C = pool_in.shape[1:]
        if H2 % 2 or W2 % 2 or (H2 // 2) * (W2 // 2) * C != F:
            raise RuntimeError("head_backward: the pool's input %s does not pool to %d features" % (tuple(pool_in.shape), F))
        out = torch.empty_like(pool_in)
        st = L.lib().niti_head_i8_backward_unpool(
            _ptr(err), _ptr(act), _ptr(drop_mask), _ptr(w), _ptr(dx), M, O, F, err_bits, L.ROUND[err_method], grad_bits,
            L.ROUND[grad_method], L.DIV[div_mode], L.BW[bw_mode], _ptr(sync), sync.numel(), _ptr(g8), _ptr(shifts[0:1]),
            _ptr(shifts[1:2]), _ptr(exp_err), _ptr(exp_w), _ptr(exp_act), int(exp_act_bias), _ptr(err_exp_out), _ptr(grad_exp_out),
            _ptr(pool_in), _ptr(out), H2 // 2, W2 // 2, C, L.TIES[ties] | (L.POOL_BWD_RELU if relu else 0), _stream(err))
        L.check(st, "niti_head_i8_backward_unpool")
        return dx, g8, shifts[0:1], shifts[1:2], sync, out
    st = L.lib().niti_head_i8_backward(_ptr(err), _ptr(act), _ptr(drop_mask), _ptr(w), _ptr(dx), M, O, F, err_bits,
                                       L.ROUND[err_method], grad_bits, L.ROUND[grad_method], L.DIV[div_mode], L.BW[bw_mode],
                                       _ptr(sync), sync.numel(), _ptr(g8), _ptr(shifts[0:1]), _ptr(shifts[1:2]), _ptr(exp_err),
                                       _ptr(exp_w), _ptr(exp_act), int(exp_act_bias), _ptr(err_exp_out), _ptr(grad_exp_out),
                                       _stream(err))
    L.check(st, "niti_head_i8_backward")
    return dx, g8, shifts[0:1], shifts[1:2], sync


def mfma_probe(operands, workgroups=512, iters=1200, shape="32x32x32"):
    """Times the library's register-resident int8 MFMA loop over the given operand bytes (int8 tensor, >= 128 bytes), on the
    instruction of ``shape`` ("32x32x32" or "16x16x64").
    Returns (tera-operations per second, shader clock in GHz during the loop): the matrix-unit ceiling for operands
    with these values."""
    name = {"32x32x32": "niti_mfma_probe_i8", "16x16x64": "niti_mfma_probe_i8_16x16x64"}[shape]
    _chk_dev(operands)
    if operands.dtype != torch.int8 or not operands.is_contiguous():
        raise RuntimeError("mfma_probe: contiguous int8 tensor expected")
    out = torch.empty(workgroups * 512, dtype=torch.int32, device=operands.device)
    clocks = torch.zeros(2, dtype=torch.int64, device=operands.device)
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)

    def launch():
        L.check(getattr(L.lib(), name)(_ptr(operands), operands.numel(), workgroups, iters, _ptr(out), _ptr(clocks), _stream(operands)), name)
    for _ in range(3):
        launch()
    e0.record()
    launch()
    e1.record()
    torch.cuda.synchronize()
    ms = e0.elapsed_time(e1)
    c = clocks.tolist()
    tops = workgroups * 8 * iters * 12 * 65536.0 / (ms * 1e-3) / 1e12
    return tops, (c[0] / (c[1] * 10.0) if c[1] else 0.0)


def maxpool_fwd(x, kernel_size=2, stride=2, padding=0):
    return L.host().maxpool_fwd(x, kernel_size, stride, padding)


def maxpool_bwd(y, dy, x, kernel_size=2, stride=2, padding=0, ties="first", relu=False):
    """``relu``: also zero the gradient where x <= 0 (the backward pass of a ReLU whose output x is)."""
    return L.host().maxpool_bwd(y, dy, x, kernel_size, stride, padding, L.TIES[ties] | (L.POOL_BWD_RELU if relu else 0))


def group_conv_f32(x, w, stride, padding, dilation, groups):
    _chk_dev(x, w)
    N, H, W, C = x.shape
    K, R, S, Cg = w.shape
    P = (H + 2 * padding - dilation * (R - 1) - 1) // stride + 1
    Q = (W + 2 * padding - dilation * (S - 1) - 1) // stride + 1
    y = torch.empty((N, max(P, 0), max(Q, 0), K), dtype=torch.float32, device=x.device)
    st = L.lib().niti_group_conv_i8_f32(_ptr(x), _ptr(w), _ptr(y), N, H, W, C, K, R, S, Cg, stride, padding, dilation,
                                        groups, _stream(x))
    L.check(st, "niti_group_conv_i8_f32")
    return y
