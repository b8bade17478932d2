"""Stand-in for the reference's ``int8mm_cuda`` extension (pytorch/int8mm-extension/int8mm.cpp:9-18)."""
from .. import _lib as L
from .. import ops  # noqa: F401  (brings torch in before the native module)


def int8_mm(lhs, rhs):
    """int8mm_kernel.cu:8-34: [m,k] x [k,n] -> exact int32 [m,n], returned like the reference as the
    transposed view of an [n,m] buffer (callers do ``.contiguous()``, ti_torch.py:176)."""
    return L.host().int8_mm(lhs, rhs)
