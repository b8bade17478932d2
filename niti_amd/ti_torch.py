"""Integer layer library with the reference's ``ti_torch`` API (class and function names, tuple
conventions ``(int8 tensor, exponent)``, module-level switches) on top of libniti_gfx950.so.

Differences in mechanism, not in results:
  * every requantisation is one device kernel that reads the tensor range the producing
    conv/GEMM kernel left in device memory; shifts and exponents stay on the device as 1-element
    int32 tensors, so a training step contains no host synchronisation (the reference
    synchronises twice per requantisation, ti_torch.py:369-377);
  * dgrad and wgrad are C-ABI entry points instead of flip/transpose/contiguous copies around the
    forward convolution (ti_torch.py:404-405, 430-432);
  * the weight gradient is rounded and applied to the weights in one pass (ti_torch.py:16-21).

Switches (module globals, like the reference's ti_torch.py:457-464 plus the two that main.py
injects): BITWIDTH, ACT_ROUND_METHOD, ERROR_ROUND_METHOD, GRAD_ROUND_METHOD, WEIGHT_INIT_METHOD,
GPU, GRAD_BITWIDTH, TRAINING.  Added here: DIV_MODE ("floor" = meaning of ``//`` on torch >= 1.13,
"trunc" = torch <= 1.12), BW_MODE ("int" exact ceil(log2) / "f32" the reference's float
evaluation), F32_EPILOGUE (reproduce the CUTLASS int32->fp32->int32 epilogue), POOL_TIES.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F
from torch.nn.modules import Module

from . import _lib, ops

GPU = "cuda"
BITWIDTH = 7
GRAD_BITWIDTH = 5      # main.py:72-77 sets 5 -> 4 -> 3 over the epochs
TRAINING = True        # main.py:146-149
DIV_MODE = "floor"
BW_MODE = "int"
F32_EPILOGUE = True
POOL_TIES = "first"


# ------------------------------------------------------------------------------------------
# small helpers
# ------------------------------------------------------------------------------------------
_EXP_CONSTANTS = {}


def _exp_tensor(e, device) -> torch.Tensor:
    """Exponent as a 1-element int32 device tensor (accepts int, float, 0-d or 1-element tensors).
    Host values are uploaded once and cached, so steady-state steps issue no host-to-device copies
    (which also keeps a step capturable into a HIP graph)."""
    if isinstance(e, torch.Tensor):
        if e.is_cuda:
            if e.dtype == torch.int32 and e.dim() == 1:
                return e
            return e.reshape(1) if e.dtype == torch.int32 else e.reshape(1).to(torch.int32)
        e = int(e)
    key = (int(e), device)
    t = _EXP_CONSTANTS.get(key)
    if t is None:
        t = torch.tensor([int(e)], dtype=torch.int32, device=device)
        _EXP_CONSTANTS[key] = t
    return t


def _planted_absmax(shift: int, target_bits: int, device) -> torch.Tensor:
    """A range whose bit-width is exactly target_bits + shift (so a kernel applies that shift)."""
    bits = target_bits + int(shift)
    if not 1 <= int(shift) or bits > 31:
        raise ValueError("shift %d out of range" % shift)
    key = ("absmax", bits, str(device))
    t = _EXP_CONSTANTS.get(key)
    if t is None:
        t = torch.tensor([2 ** (bits - 1) + 1], dtype=torch.int64, device=device).to(torch.int32)
        _EXP_CONSTANTS[key] = t
    return t


def _standalone(x: torch.Tensor, shift: int, method: str, rand=None) -> torch.Tensor:
    x32 = x.to(torch.int32).contiguous()
    am = _planted_absmax(shift, BITWIDTH, x32.device)
    y, _ = ops.requant(x32, am, BITWIDTH, method, DIV_MODE, "int", rand)
    return y


def RoundShift(input, shift):
    """ti_torch.py:23-31."""
    return _standalone(input, shift, "round")


def StoShift(input, shift, rand=None):
    """ti_torch.py:33-46; ``rand`` (int32, one per element, in [0, 2**shift)) replaces the device
    ``torch.randint`` when given."""
    if rand is None:
        rand = torch.randint(0, 2 ** shift, input.shape, dtype=torch.int32, device=input.device)
    return _standalone(input, shift, "sto", rand.to(torch.int32).contiguous())


def PstoShift(input, shift):
    """ti_torch.py:48-69."""
    return _standalone(input, shift, "psto")


ACT_ROUND_METHOD = RoundShift
ERROR_ROUND_METHOD = RoundShift
GRAD_ROUND_METHOD = PstoShift


_METHODS = {RoundShift: "round", StoShift: "sto", PstoShift: "psto"}
_METHOD_CODES = {fn: _lib.ROUND[name] for fn, name in _METHODS.items()}
_STO = _lib.ROUND["sto"]


def _method_name(fn) -> str:
    try:
        return _METHODS[fn]
    except KeyError:
        raise ValueError("rounding method must be RoundShift, StoShift or PstoShift") from None


def _method_code(fn) -> int:
    """The library's number of a rounding method."""
    try:
        return _METHOD_CODES[fn]
    except KeyError:
        raise ValueError("rounding method must be RoundShift, StoShift or PstoShift") from None


def _rand_bits_like(x: torch.Tensor) -> torch.Tensor:
    """31 uniform random bits per element; the kernel keeps the low `shift` ones."""
    return torch.randint(0, 2 ** 31 - 1, x.shape, dtype=torch.int32, device=x.device)


def int8_clip(input, clip_val=127):
    """ti_torch.py:71-72."""
    return torch.clamp(input, -clip_val, clip_val).type(torch.int8)


def Int8Tensor(val):
    return torch.tensor(val, dtype=torch.int8).to(GPU)


def Int8zeros(size):
    return torch.zeros(size=size, dtype=torch.int8, device=GPU)


def roundoff4(size):
    return (size + 3) // 4 * 4


# ------------------------------------------------------------------------------------------
# range estimate and requantisation (ti_torch.py:103-147, 366-377)
# ------------------------------------------------------------------------------------------
def TensorBitwidth(val):
    """ti_torch.py:366-367 (host value; synchronises)."""
    return int(_lib.lib().niti_bitwidth(int(val), _lib.BW[BW_MODE]))


def RangeEstimate(input):
    """ti_torch.py:369-377.  Returns a Python int like the reference, which costs a device->host
    copy; the layers below never call it."""
    am = ops.absmax_i32(input.to(torch.int32).contiguous())
    return TensorBitwidth(int(am.item()) & 0xFFFFFFFF)


def _requant(acc, target_bits, fn, absmax=None, rand=None, relu=False, exp_a=None, exp_b=None, want_exp=False):
    acc = acc.contiguous()
    if acc.dtype != torch.int32:
        acc = acc.to(torch.int32)        # first-layer gradients arrive as integer-valued float32
    if absmax is None:
        absmax = ops.absmax_i32(acc)
    method = _method_name(fn)
    if method == "sto" and rand is None:
        rand = _rand_bits_like(acc)
    exp_out = torch.empty(1, dtype=torch.int32, device=acc.device) if want_exp else None
    y, shift = ops.requant(acc, absmax, target_bits, method, DIV_MODE, BW_MODE, rand, relu,
                           exp_a=exp_a, exp_b=exp_b, exp_out=exp_out)
    return y, shift, exp_out


def act_calc(int32_acc, exp_in, absmax=None, rand=None):
    """ti_torch.py:103-117.  Returns (int8 tensor, exp_out) with exp_out a 1-element int32 device
    tensor equal to exp_in + shift."""
    e = _exp_tensor(exp_in, int32_acc.device)
    y, _, exp_out = _requant(int32_acc, BITWIDTH, ACT_ROUND_METHOD, absmax, rand, exp_a=e, want_exp=True)
    return y, exp_out


def err_calc(int32_acc, absmax=None, rand=None):
    """ti_torch.py:119-133.  Returns (int8 tensor, shift) with shift a 1-element int32 device tensor."""
    y, shift, _ = _requant(int32_acc, BITWIDTH, ERROR_ROUND_METHOD, absmax, rand)
    return y, shift


def grad_calc(int32_acc, mu, absmax=None, rand=None):
    """ti_torch.py:135-147."""
    y, shift, _ = _requant(int32_acc, mu, GRAD_ROUND_METHOD, absmax, rand)
    return y, shift


FUSE_CONV_REQUANT = True     # run a product + requantisation as one launch where the library covers the shape
KEEP_INT32_GRAD = False      # also store layer.grad_int32acc when the weight gradient is rounded and applied in one call


def _sto_rand(method, rand, shape, dev):
    """Random integers (int32, contiguous) for a rounding of a tensor of ``shape``: the caller's or 31 random bits each,
    of which a kernel keeps the low `shift` ones; None where the method takes none."""
    if method != _STO:
        return None
    return torch.randint(0, 2 ** 31 - 1, shape, dtype=torch.int32, device=dev) if rand is None else rand.contiguous()


# ------------------------------------------------------------------------------------------
# op wrappers (ti_torch.py:152-233)
# ------------------------------------------------------------------------------------------
def int8mm(lhs, rhs):
    """ti_torch.py:152-176: [m,k] x [k,n] -> contiguous int32 [m,n] (any m, n, k)."""
    return ops.gemm(lhs.contiguous(), rhs.contiguous())


def _pad_channels16(t):
    if t.size(3) % 16 == 0:
        return t
    if t.is_cuda and t.dtype == torch.int8:
        return ops.pad_last_dim(t.contiguous(), 16)
    return F.pad(t, (0, 16 - t.size(3) % 16), "constant", 0)


def conv2d_int8(input, weight, stride=1, padding=1, absmax=None):
    """ti_torch.py:178-192: NHWC int8 x KRSC int8 -> NPQK int32."""
    return ops.conv2d_fprop(_pad_channels16(input).contiguous(), _pad_channels16(weight).contiguous(), stride, padding,
                            f32_epilogue=F32_EPILOGUE, absmax=absmax)


def conv2d_weight_int8(input, weight_size, grad_output, stride=1, padding=0, dilation=1):
    """ti_torch.py:194-233: first-layer weight gradient, returned like the reference as an
    integer-valued float32 KRSC tensor."""
    if stride != 1 or dilation != 1:
        raise RuntimeError("conv2d_weight_int8: only stride 1, dilation 1 (as guarded in the reference, ti_torch.py:413)")
    dw = ops.conv2d_wgrad(input.contiguous(), grad_output.contiguous(), weight_size[1], weight_size[2], stride, padding)
    return dw.float()


# ------------------------------------------------------------------------------------------
# quantisers / initialisers (ti_torch.py:77-99, 334-364)
# ------------------------------------------------------------------------------------------
def _ceil_log2(r):
    """``torch.ceil(torch.log2(r))`` of ti_torch.py:336,348.  BW_MODE "int" (default): exact arithmetic on the float's
    exponent and mantissa (r = m * 2^e, 0.5 <= m < 1: e - 1 for a power of two, e otherwise), so that every device
    gives the same integer.  BW_MODE "f32": the reference's own float32 expression, whose log2 rounds
    k + log2(1 + d) back to k for the first float32 values above 2^k, k >= 4 (nextafter(16) gives 4 where the exact
    value is 5: the exponent is then one lower and the largest value saturates at 127).  0-d float tensor."""
    if BW_MODE == "f32":
        return torch.ceil(torch.log2(r.float()))
    m, e = torch.frexp(r.float())
    return torch.where(m == 0.5, e - 1, e).to(torch.float32)


def weight_quant(input):
    """ti_torch.py:334-339.  Returns (int8 weights on the GPU, exponent as a 0-d float tensor)."""
    input_range = torch.max(torch.abs(input))
    input_bitwidth = _ceil_log2(input_range)
    act_exp = input_bitwidth - 7
    round_val = torch.round(input / input_range * (2 ** 7 - 1)).type(torch.int8).to(GPU)
    return round_val, act_exp


def UniformWeights(size):
    """ti_torch.py:77-85 (Xavier-uniform drawn in KCRS, stored KRSC)."""
    if len(size) == 4:
        temp = torch.zeros(size).permute(0, 3, 1, 2).contiguous()
        torch.nn.init.xavier_uniform_(temp)
        return weight_quant(temp.permute(0, 2, 3, 1).contiguous())
    temp = torch.zeros(size)
    torch.nn.init.xavier_uniform_(temp)
    return weight_quant(temp)


def NormalWeight(size):
    """ti_torch.py:87-95."""
    if len(size) == 4:
        temp = torch.zeros(size).permute(0, 3, 1, 2).contiguous()
        torch.nn.init.xavier_normal_(temp)
        return weight_quant(temp.permute(0, 2, 3, 1).contiguous())
    temp = torch.zeros(size)
    torch.nn.init.xavier_normal_(temp)
    return weight_quant(temp)


WEIGHT_INIT_METHOD = UniformWeights


def TiFloatToInt8(input):
    """ti_torch.py:341-356: float tensor -> (int8 tensor on the GPU, exponent).  The exponent is
    returned as a 0-d float tensor like the reference; no host synchronisation.  The range is a tensor-library
    reduction, whose multi-block form clears its scratch words with a memset node: keep this call outside a captured
    HIP graph (train.StepGraph quantises eagerly and captures forward_int8 + backward)."""
    input = input.to(GPU)
    input_range = torch.max(torch.abs(input))
    input_bitwidth = _ceil_log2(input_range)
    act_exp = input_bitwidth - BITWIDTH
    norm_val = input * (2 ** (BITWIDTH - input_bitwidth))
    round_val = torch.round(norm_val)
    clamp_val = torch.clamp(round_val, -128, 127).type(torch.int8)
    return clamp_val, act_exp


def TiInt8ToFloat(input):
    """ti_torch.py:358-364."""
    act_in, exp_in = input
    if not isinstance(exp_in, torch.Tensor):
        exp_in = torch.tensor(float(exp_in), device=act_in.device)
    return act_in.float() * (2 ** (exp_in.float().reshape(())))


# ------------------------------------------------------------------------------------------
# layers
# ------------------------------------------------------------------------------------------
class UpdateWeight(Module):
    """ti_torch.py:11-21: vanilla integer SGD shared by TiConv2d and TiLinear.  grad_calc and the
    saturating subtraction run as one kernel; ``self.grad`` (the rounded int8 gradient) is kept only
    when ``keep_grad`` is set."""
    keep_grad = False

    def _init_weight(self, size):
        w, e = WEIGHT_INIT_METHOD(size)
        self.weight = w.to(GPU).contiguous()
        self.weight_exp = e if isinstance(e, torch.Tensor) else torch.tensor(float(e))

    def _wexp(self):
        """weight_exp (a host-side 0-d float tensor, as in the reference) as a cached device int32."""
        cached = getattr(self, "_wexp_cache", None)
        if cached is None or cached[0] is not self.weight_exp:
            cached = (self.weight_exp, _exp_tensor(self.weight_exp, self.weight.device))
            self._wexp_cache = cached
        return cached[1]

    def weight_update(self, absmax=None, rand=None):
        g = self.grad_int32acc
        if g.dtype != torch.int32:
            g = g.to(torch.int32)
        g = g.contiguous()
        if absmax is None:
            absmax = ops.absmax_i32(g)
        method = _method_name(GRAD_ROUND_METHOD)
        if method == "sto" and rand is None:
            rand = _rand_bits_like(g)
        self.grad_exp = torch.empty(1, dtype=torch.int32, device=g.device)
        if not self.weight.is_contiguous():
            self.weight = self.weight.contiguous()
        self.grad, self.grad_shift = ops.grad_update(
            g, self.weight, absmax, GRAD_BITWIDTH, method, DIV_MODE, BW_MODE, rand, want_grad=self.keep_grad,
            exp_a=_exp_tensor(self.err_exp, g.device), exp_b=_exp_tensor(self.act_in_exp, g.device), exp_out=self.grad_exp)
        self._weights_changed()

    def _weights_changed(self):
        """The weights have been updated by a call that kept no copy of them in step."""


class TiConv2d(UpdateWeight):
    """ti_torch.py:379-437: int8 convolution layer, NHWC activations, KRSC weights.
    ``fuse_relu`` folds the following TiReLU's forward into the activation requantisation."""

    def __init__(self, in_channels, out_channels, kernel_size=3, stride=1, padding=1, first_layer=False):
        super().__init__()
        self._init_weight(torch.Size([out_channels, kernel_size, kernel_size, in_channels]))
        self.first_layer = first_layer
        self.stride = stride
        self.padding = padding
        self.fuse_relu = False
        self.relu_below = False
        self.pool_after = None      # the 2x2 / stride-2 TiMaxpool2d behind this layer's (fused) ReLU, if its forward is folded in
        self.pool_below = None      # the 2x2 / stride-2 TiMaxpool2d in front of this layer, if its backward pass is folded in

    def forward(self, input, rand=None):
        d = self.__dict__       # plain attributes: Module.__setattr__ looks for parameters first
        act, act_exp = input
        d["act"], d["act_in_exp"] = act, act_exp
        dev = act.device
        # channel-padded copy, reused by the weight gradient
        act16 = d["act16"] = act if act.shape[3] % 16 == 0 and act.is_contiguous() else _pad_channels16(act).contiguous()
        weight = self.weight
        # With an up-to-date kernel-ready filter copy the padded weights are passed for their shape only: the first
        # layer then reuses the padded tensor the copy was made from instead of padding the weights again every step.
        key = (weight.data_ptr(), weight._version, act16.shape)
        fresh = d.get("_wprep_key") == key
        if weight.shape[3] % 16 == 0:
            w16, shape_only = (weight if weight.is_contiguous() else weight.contiguous()), False
            d["_w16_kept"] = None
        else:
            shape_only = fresh and d.get("_wprep") is not None and d.get("_w16_kept") is not None
            w16 = d["_w16_kept"] = self._w16_kept if shape_only else _pad_channels16(weight).contiguous()
        if not fresh:
            d["_wprep"] = self._filter_copy(w16, act16.shape)
            d["_wprep_key"] = key
        method = _method_code(ACT_ROUND_METHOD)
        if method == _STO:
            R, S = w16.shape[1:3]
            N, H, W, _ = act16.shape
            rand = _sto_rand(method, rand, (N, (H + 2 * self.padding - R) // self.stride + 1, (W + 2 * self.padding - S) // self.stride + 1,
                                            w16.shape[0]), dev)
        elif rand is not None:
            rand = None
        y, exp_out, pooled = _lib.host().conv_layer_forward(
            FUSE_CONV_REQUANT, act16, w16, self.stride, self.padding, F32_EPILOGUE, BITWIDTH, method, _lib.DIV[DIV_MODE], _lib.BW[BW_MODE],
            self.fuse_relu, self._shift_state("act", dev), _exp_tensor(act_exp, dev), self._wexp(), d["_wprep"],
            self.pool_after is not None, rand, not shape_only)
        if pooled is not None:      # the pooling layer finds its result ready when it sees this tensor
            self.pool_after.__dict__["preset"] = (y, pooled)
        return y, exp_out

    def backward(self, input, rand=None, grad_rand=None):
        d = self.__dict__
        err_in, err_exp = input
        if not err_in.is_contiguous():
            err_in = err_in.contiguous()
        dev = err_in.device
        host = _lib.host()
        div, bw = _lib.DIV[DIV_MODE], _lib.BW[BW_MODE]
        d["err_exp_in"] = d["err_exp"] = _exp_tensor(err_exp, dev)
        act, act16, weight = d["act"], d["act16"], self.weight
        if not weight.is_contiguous():
            weight = self.weight = weight.contiguous()
        prepared = self._synced_filter()
        if not self.first_layer:
            # data gradient with the weights as they were in the forward pass
            # relu_below: the ReLU in front of this layer (possibly with a max-pool in between) leaves its backward
            # pass to this layer, whose input is that ReLU's (pooled) output
            mask = pool_in = None
            if self.relu_below:
                mask = act if act.is_contiguous() else act.contiguous()
                pool = self.pool_below
                # the max-pool in front of this layer: its backward pass is written by this launch's epilogue
                if pool is not None and err_in.shape[1] >= 2:
                    pooled, whole = pool.__dict__.get("act_out"), pool.__dict__.get("act_in")
                    if pooled is not None and pooled.data_ptr() == mask.data_ptr() and whole.is_contiguous():
                        pool_in = whole
            method = _method_code(ERROR_ROUND_METHOD)
            if method == _STO:
                N, P, Q, _ = err_in.shape
                _, R, S, C = weight.shape
                rand = _sto_rand(method, rand, (N, P - 2 * self.padding + R - 1, Q - 2 * self.padding + S - 1, C), dev)
            elif rand is not None:
                rand = None
        g_method = _method_code(GRAD_ROUND_METHOD)
        grad_rand = _sto_rand(g_method, grad_rand, tuple(weight.shape), dev)
        if self.first_layer:
            d["grad"], d["grad_int32acc"], d["grad_shift"], d["grad_exp"], one = host.conv_layer_wgrad_update(
                FUSE_CONV_REQUANT and grad_rand is None, act16, err_in, weight, self.stride, self.padding, False, GRAD_BITWIDTH, g_method, div, bw,
                self.keep_grad, KEEP_INT32_GRAD, self._shift_state("grad", dev), d["err_exp"], _exp_tensor(d["act_in_exp"], dev), prepared,
                grad_rand)
        else:
            err_out, d["err_exp"], unpooled, d["grad"], d["grad_int32acc"], d["grad_shift"], d["grad_exp"], one = host.conv_layer_backward(
                FUSE_CONV_REQUANT, err_in, act16, weight, self.stride, self.padding, F32_EPILOGUE, BITWIDTH, method, div, bw,
                self._shift_state("err", dev), d["err_exp_in"], self._wexp(), prepared if act16.shape[3] == weight.shape[3] else None, mask,
                pool_in, _lib.TIES[POOL_TIES], rand, GRAD_BITWIDTH, g_method, self.keep_grad, KEEP_INT32_GRAD, self._shift_state("grad", dev),
                _exp_tensor(d["act_in_exp"], dev), prepared, grad_rand)
            if unpooled:
                pool.__dict__["bwd_done"] = err_out
        if not one or prepared is not d.get("_wprep_kept"):
            self._weights_changed()
        if not self.first_layer:
            return err_out, d["err_exp"]

    def _filter_copy(self, w16, shape):
        """Kernel-ready copy of the filter for activations of ``shape``, None where the kernels read it as stored.  The layer keeps
        one buffer, whatever batches and maps come along: captured steps hold its address.  It is written here when the weight
        tensor was replaced or modified through torch; the one-call update keeps it in step with its own changes, and
        _weights_changed follows every other update."""
        d, (N, H, W, _), weight = self.__dict__, shape, self.weight
        nbytes = ops.conv_filter_bytes(w16, N, H, W, self.stride, self.padding)
        if nbytes == 0:
            return None
        kept = d.get("_wprep_kept")
        if kept is None or kept.numel() != nbytes or kept.device != w16.device:
            kept = d["_wprep_kept"] = torch.empty(nbytes, dtype=torch.int8, device=w16.device)
            d["_wprep_of"] = None
        made_of = (weight.data_ptr(), weight._version)
        if d["_wprep_of"] != made_of:
            ops.conv_filter_prepare(w16, N, H, W, self.stride, self.padding, out=kept)
            # the alias keeps the weights' memory from being given to another tensor, which their address would not tell apart
            d["_wprep_of"], d["_wprep_for"], d["_wprep_weight"] = made_of, (N, H, W), weight.detach()
        return kept

    def _weights_changed(self):
        d = self.__dict__
        kept = d.get("_wprep_kept")
        if kept is None:
            return
        w16 = _pad_channels16(self.weight).contiguous()
        if w16.device != kept.device or ops.conv_filter_bytes(w16, *d["_wprep_for"], self.stride, self.padding) != kept.numel():
            d["_wprep_kept"] = d["_wprep_key"] = None      # another filter has taken the place of the one it was made for
            return
        ops.conv_filter_prepare(w16, *d["_wprep_for"], self.stride, self.padding, out=kept)
        d["_wprep_of"], d["_wprep_weight"] = (self.weight.data_ptr(), self.weight._version), self.weight.detach()

    def _shift_state(self, which, device):
        """1-element int32 device tensor that keeps the requantisation shift of this layer's activations ("act") or
        errors ("err") from one step to the next; the single-launch kernels take it as their prediction."""
        states = self.__dict__.get("_shift_states")
        if states is None:
            states = self.__dict__["_shift_states"] = {}
        key = (which, device)
        state = states.get(key)
        if state is None:
            state = states[key] = torch.zeros(1, dtype=torch.int32, device=device)
        return state

    def _synced_filter(self):
        """The forward filter copy if it matches the weights as they are now (then the update maintains it)."""
        d = self.__dict__
        key, weight = d.get("_wprep_key"), self.weight
        if key is None or key[0] != weight.data_ptr() or key[1] != weight._version:
            d["_wprep_key"] = None
            return None
        return d["_wprep"]


class TiLinear(UpdateWeight):
    """ti_torch.py:235-266: int8 fully connected layer, weight [out_features, in_features]."""

    def __init__(self, in_features, out_features, last_layer=False):
        super().__init__()
        self._init_weight(torch.Size([out_features, in_features]))
        self.last_layer = last_layer
        self.__dict__["drop_below"] = None   # the TiDropout in front of this layer whose masking this layer's kernels take over
        self.rng = None             # RngBox of the network (dropout mask / loss rounding drawn inside the kernels)
        self.next_target = None     # (targets, random integers or None): evaluate the loss gradient in the next forward
        self.loss_grad = None       # (targets, loss gradient) left by that forward
        self._dropped = None        # dropout mask the last forward applied itself

    def _rng_state(self, dev):
        return self.rng.state(dev) if self.rng is not None else ops.rng_state(dev)

    def forward(self, input, rand=None):
        d = self.__dict__
        d["act_in"] = input
        act_in, exp_in = input
        if not act_in.is_contiguous():
            act_in = act_in.contiguous()
        dev = act_in.device
        weight = self.weight if self.weight.is_contiguous() else self.weight.contiguous()
        host = _lib.host()
        method, div, bw = _method_code(ACT_ROUND_METHOD), _lib.DIV[DIV_MODE], _lib.BW[BW_MODE]
        drop = self.drop_below
        d["_dropped"] = d["loss_grad"] = None
        pending = drop is not None and drop.pending is not None and drop.pending[0] is input[0]
        want_loss, d["next_target"] = self.next_target, None
        # the classifier-head kernel: dropout and loss gradient folded in, where no rounding needs random input
        if (pending or want_loss is not None) and FUSE_CONV_REQUANT and rand is None and method != _STO:
            target, loss_rand = want_loss if want_loss is not None else (None, None)
            given = drop.pending[1] if pending else None
            draws = (pending and given is None) or (want_loss is not None and loss_rand is None)
            done = host.head_forward(act_in, weight, BITWIDTH, method, div, bw, 0 if not pending else (2 if given is None else 1), given,
                                     self._rng_state(dev) if draws else None, 1 if pending else 0, target, loss_rand,
                                     _exp_tensor(exp_in, dev), self._wexp())
            if done is not None:
                if pending:
                    drop.__dict__["drop_mask"] = d["_dropped"] = done[2]
                    drop.__dict__["pending"] = None
                if want_loss is not None:
                    d["loss_grad"] = (target, done[3])
                return done[0], done[1]
        if pending:   # the dropout left its work to this layer, which cannot take it: do it now
            act_in, exp_in = drop.apply_now(act_in, exp_in)
            d["act_in"] = (act_in, exp_in)
        rand = _sto_rand(method, rand, (act_in.shape[0], weight.shape[0]), dev)
        return host.linear_forward(FUSE_CONV_REQUANT, act_in, weight, BITWIDTH, method, div, bw, _exp_tensor(exp_in, dev), self._wexp(), rand)

    def backward(self, input, rand=None, grad_rand=None):
        d = self.__dict__
        err_in, err_exp = input
        if not err_in.is_contiguous():
            err_in = err_in.contiguous()
        dev = err_in.device
        act, d["act_in_exp"] = d["act_in"]
        if not act.is_contiguous():
            act = act.contiguous()
        weight = self.weight
        if not weight.is_contiguous():
            weight = self.weight = weight.contiguous()
        host = _lib.host()
        e_method, g_method = _method_code(ERROR_ROUND_METHOD), _method_code(GRAD_ROUND_METHOD)
        div, bw = _lib.DIV[DIV_MODE], _lib.BW[BW_MODE]
        d["err_exp_in"] = _exp_tensor(err_exp, dev)
        mask = self._dropped     # the forward pass read ``act`` through this mask: act_in is the tensor in front of the dropout
        if not KEEP_INT32_GRAD and FUSE_CONV_REQUANT and rand is None and grad_rand is None and e_method != _STO and g_method != _STO:
            # the 2x2 max-pool whose flattened output this layer read (TiNet.fuse): its backward pass in the same launch
            pool = d.get("pool_below")
            pool_in = None
            if pool is not None:
                pooled, whole = pool.__dict__.get("act_out"), pool.__dict__.get("act_in")
                if (pooled is not None and pooled.data_ptr() == act.data_ptr() and pooled.numel() == act.numel() and whole.dim() == 4
                        and whole.is_contiguous() and whole.dtype == torch.int8 and whole.shape[3] % 64 == 0):
                    pool_in = whole
            done = host.head_backward(
                err_in, act, weight, BITWIDTH, e_method, GRAD_BITWIDTH, g_method, div, bw, mask, self.keep_grad, d["err_exp_in"],
                self._wexp(), _exp_tensor(d["act_in_exp"], dev), 1 if mask is not None else 0, pool_in,
                _lib.TIES[POOL_TIES] | (_lib.POOL_BWD_RELU if pool_in is not None and pool.relu_below else 0))
            if done is not None:
                err_out, d["grad"], d["grad_shift"], d["err_exp"], d["grad_exp"], routed = done
                d["grad_int32acc"] = None
                if mask is not None:
                    self.drop_below.__dict__["bwd_done"] = err_out     # masked already
                if routed is not None:
                    pool.__dict__["bwd_routed"] = (err_out, routed)
                return err_out, d["err_exp"]
        if mask is not None:     # the separate passes want the masked activations and their exponent
            act, d["act_in_exp"] = ops.mask_features(act, mask, _exp_tensor(d["act_in_exp"], dev), 1)
        rand = _sto_rand(e_method, rand, tuple(act.shape), dev)
        grad_rand = _sto_rand(g_method, grad_rand, tuple(weight.shape), dev)
        err_out, d["err_exp"], d["grad"], d["grad_int32acc"], d["grad_shift"], d["grad_exp"] = host.linear_backward(
            FUSE_CONV_REQUANT, err_in, act, weight, BITWIDTH, e_method, GRAD_BITWIDTH, g_method, div, bw, self.keep_grad, KEEP_INT32_GRAD,
            d["err_exp_in"], self._wexp(), _exp_tensor(d["act_in_exp"], dev), rand, grad_rand)
        return err_out, d["err_exp"]


class TiReLU(Module):
    """ti_torch.py:268-290.  With ``fused`` set the preceding TiConv2d already clamped at zero and
    forward only records its input (the clamped tensor: ``act > 0`` is the same test on it)."""

    def __init__(self):
        super().__init__()
        self.fused = False
        self.bwd_folded = False

    def forward(self, input):
        self.__dict__["act_in"] = input      # a plain attribute: Module.__setattr__ looks for parameters first
        act_in, exp_in = input
        if self.fused:
            return input
        return ops.relu_fwd(act_in.contiguous()), exp_in

    def backward(self, input):
        if self.bwd_folded:      # the convolution or pooling above this layer masked its data gradient already
            return input
        err_in, err_exp = input
        act, _ = self.act_in
        return ops.relu_bwd(act.contiguous(), err_in.contiguous()), err_exp


class TiMaxpool2d(Module):
    """ti_torch.py:292-316."""

    def __init__(self, kernel_size, stride, padding=0):
        super().__init__()
        self.kernel_size = kernel_size
        self.stride = stride
        self.padding = padding
        self.relu_below = False     # the ReLU in front of this layer leaves its backward pass to this layer
        self.preset = None          # (input tensor, pooled tensor) left by the convolution that computed both
        self.bwd_done = None        # the error tensor a convolution behind this layer has already routed through it
        self.bwd_routed = None      # (error tensor, routed result) left by the classifier behind this layer

    def forward(self, input):
        d = self.__dict__       # plain attributes: Module.__setattr__ looks for parameters first
        act_in, exp_in = input
        preset, d["preset"] = d["preset"], None
        if preset is not None and preset[0] is act_in:
            d["act_in"], d["act_out"] = act_in, preset[1]
            return preset[1], exp_in
        d["act_in"] = act_in = act_in.contiguous()
        d["act_out"] = _lib.host().maxpool_fwd(act_in, self.kernel_size, self.stride, self.padding)
        return d["act_out"], exp_in

    def backward(self, input):
        err_in, err_exp = input
        d = self.__dict__
        done, d["bwd_done"] = d["bwd_done"], None
        if done is not None and done is err_in:
            return input        # the data gradient behind this layer wrote its result through this pooling already
        routed, d["bwd_routed"] = d["bwd_routed"], None
        if routed is not None and routed[0].data_ptr() == err_in.data_ptr() and routed[0].numel() == err_in.numel():
            return routed[1], err_exp     # the classifier's backward launch has run this pass
        err_out = _lib.host().maxpool_bwd(d["act_out"], err_in.contiguous(), d["act_in"], self.kernel_size, self.stride, self.padding,
                                          _lib.TIES[POOL_TIES] | (_lib.POOL_BWD_RELU if self.relu_below else 0))
        return err_out, err_exp


class TiFlat(Module):
    """ti_torch.py:318-332."""

    def forward(self, input):
        self.__dict__["act_in"] = input
        act_in, exp_in = input
        return act_in.view(-1, act_in.nelement() // act_in.size(0)), exp_in

    def backward(self, input):
        err_in, err_exp = input
        act, _ = self.act_in
        return err_in.view_as(act), err_exp


class TiDropout(Module):
    """ti_torch.py:439-455: one keep/drop decision per feature (not per sample), exponent + 1.
    ``mask`` (int8 0/1 per feature) can be supplied for reproducible runs.  With ``head`` set (TiNet.fuse: the
    TiLinear that follows) the masking is left to that layer's kernels, which also draw the mask."""

    def __init__(self):
        super().__init__()
        self.__dict__["head"] = None   # the TiLinear behind this layer that applies the mask in its own launches
        self.pending = None      # (activation tensor, given mask or None) handed to that layer
        self.bwd_done = None     # the error tensor that layer has already masked

    def forward(self, input, mask=None):
        if TRAINING:
            act_in, exp_in = input
            if mask is not None:
                mask = mask.to(act_in.device)
            if (self.head is not None and FUSE_CONV_REQUANT and act_in.is_cuda and act_in.dtype == torch.int8 and act_in.dim() == 2
                    and act_in.is_contiguous() and (mask is None or (mask.dtype == torch.int8 and mask.is_contiguous()))):
                self.__dict__["pending"] = (act_in, mask)
                return input
            return self.apply_now(act_in, exp_in, mask)
        self.__dict__["pending"] = None
        return input

    def apply_now(self, act_in, exp_in, mask=None):
        if mask is None and self.pending is not None:
            mask = self.pending[1]
        self.pending = None
        if mask is None:
            mask = torch.randint(low=0, high=2, size=(act_in.size(1),), dtype=torch.int8, device=act_in.device)
        self.drop_mask = mask.to(act_in.device)
        if self._one_launch(act_in):
            return ops.mask_features(act_in, self.drop_mask, _exp_tensor(exp_in, act_in.device), 1)
        return act_in * self.drop_mask, _exp_tensor(exp_in, act_in.device) + 1

    def _one_launch(self, t):
        m = self.drop_mask
        return (t.is_cuda and t.dtype == torch.int8 and m.dtype == torch.int8 and t.dim() == 2 and t.is_contiguous()
                and m.is_contiguous() and t.shape[1] % 16 == 0 and t.data_ptr() % 16 == 0 and m.data_ptr() % 16 == 0)

    def backward(self, input):
        err_in, err_exp = input
        done, self.__dict__["bwd_done"] = self.bwd_done, None
        if done is not None and done is err_in:
            return input        # the layer behind this one masked its data gradient already
        if self._one_launch(err_in):
            return ops.mask_features(err_in, self.drop_mask), err_exp
        return err_in * self.drop_mask, err_exp


class RngBox:
    """The generator state (ops.rng_state) of one network, created on first use with a key drawn from torch's default
    CPU generator: two networks built after the same ``torch.manual_seed`` draw the same sequence."""

    def __init__(self):
        self._state = {}

    def state(self, device):
        key = str(device)
        if key not in self._state:
            if torch.cuda.is_current_stream_capturing():
                raise RuntimeError("RngBox: first use under graph capture; run one step eagerly first")
            self._state[key] = ops.rng_state(device, int(torch.empty((), dtype=torch.int64).random_().item()))
        return self._state[key]
