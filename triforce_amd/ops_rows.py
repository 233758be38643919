"""Products of many rows in 16 bits (prefill) over the C ABI: x . W^T and x . W^T with a gated unit behind it, float16 by libtriforce_hip.so,
bfloat16 by libtriforce_tile.so (csrc/rows_gemm.h).

Same rules as ops.py: torch owns the memory and the stream.  What the kernel does not take, and what a derivative, transform or trace
follows, goes to torch.
"""
import ctypes
import functools

import torch
import torch.nn.functional as F
from torch.autograd import forward_ad

from . import hip

PLAIN, SILU_HALVES, GELU_EIGHTS = 0, 1, 2
_FORMS = {torch.float16: (PLAIN, SILU_HALVES), torch.bfloat16: (PLAIN, GELU_EIGHTS)}


def unwatched(*ts):
    """Device tensors that no derivative, transform, trace or autocast follows: a launch behind torch's back would be lost on them."""
    if torch.is_autocast_enabled() or torch.compiler.is_compiling() or torch.jit.is_tracing() or torch._C._len_torch_dispatch_stack() \
            or torch._C._functorch.peek_interpreter_stack() is not None:
        return False
    return all(t.is_cuda and type(t) in (torch.Tensor, torch.nn.Parameter) and not (t.requires_grad and torch.is_grad_enabled())
               and forward_ad.unpack_dual(t).tangent is None for t in ts)


def takes(x, w, form=PLAIN):
    """Does the kernel take x [rows, k] . w [n, k]^T as it stands?  (entry() of csrc/rows_gemm.h)"""
    if x.dim() != 2 or w.dim() != 2 or x.dtype != w.dtype or form not in _FORMS.get(x.dtype, ()):
        return False
    (rows, k), n = x.shape, w.shape[0]
    ld = x.stride(0)
    return (w.shape[1] == k and rows >= 1 and n >= 16 and n % (16 if form == PLAIN else 32) == 0 and k >= 64 and k % 64 == 0 and x.stride(1) == 1
            and ld >= k and ld % 8 == 0 and rows * ld < 1 << 31 and n * k < 1 << 31 and n < 1 << 26 and rows * n < 1 << 37 and w.is_contiguous()
            and x.device == w.device and unwatched(x, w) and x.device.index == torch.cuda.current_device() and (x.data_ptr() | w.data_ptr()) % 16 == 0)


def library_fills(rows, n):
    """Do tiles of 256 x 256 fill whole rounds of the 256 CUs?  There the library's kernel is the faster one, for a plain product of more than
    1 152 columns: 4 096 x 4 096 x 4 096 93.9 us against 98.5, 4 096 x 12 288 282 against 293, 8 000 x 4 096 x 11 008 480 against 487 (but
    4 096 x 8 192 x 512 41 against 38); where they do not, the other way round (3 100 x 12 288 x 4 096 256 against 245, 3 100 x 22 016
    547 against 425)."""
    tiles = -(-rows // 256) * -(-n // 256)
    return tiles % 256 == 0 and 100 * rows * n >= 97 * 65536 * tiles


def library_is_faster(rows, n, k):
    """Is the library's kernel the one to take for a plain product, from 33 rows on?  On the device alone the two are within 10 % of each other at most sizes
    (24 products of 256 .. 32 000 outputs and 256 .. 15 104 columns at 57 counts of rows up to 8 000, weights from memory: this kernel 0.87 of the
    library's time on average, more than 1.05 of it in one of nine).  A call of the library is 7 us of the host's time more, and some 50 where
    its sizes are new, as a prompt's mostly are: forwards of 80 and 300 tokens with the library's products wherever those were the faster
    ones 1 054 -> 1 197 and 1 430 -> 1 483 us (kemurax, four layers), of 550 and 1 700 tokens 1 244 -> 1 264 and 2 787 -> 2 812 (llama).  So it is
    taken where it gains more than that, or inside graphs (this kernel's time over the library's):
      * whole rounds of tiles of 256 x 256, see library_fills: 1.02 to 1.10 from 2 048 rows and 1 280 columns on; at 512 and 1 024 rows 0.83 to 1.02, and of
        512 columns 0.98;
      * a few tiles with parts of k that cost more than they bring: 576 x 4 096, 1 024 x 4 096 and 768 x 3 072 (the 68M draft's chunks of 64 rows, 7.1 us
        against 8.9) 0.9 to 1.25 up to 320 rows; on either side of these 512 x 2 048 and 768 x 1 536 1.0 to 1.05, 1 536 x 4 096 0.82 to 1.07, 1 280 x
        5 120 0.73 to 0.9, 640 x 8 192 0.7 to 1.06, and all of them 0.8 to 1.0 at 600 rows;
      * 97 to 192 rows of 234 MB of weights and more (logits), where tiles of 128 x 256 leave half of the CUs without one: 32 000 x 4 096 1.0 to 1.27 (62 us
        against 72), x 5 120 0.8 to 1.19, 28 672 x 4 096 1.05 to 1.21, x 8 192 1.08 to 1.13, 24 576 x 5 120 1.01 to 1.13, 16 384 x 8 192 1.13 to 1.28; but
        18 784 x 6 144 0.91 to 1.03, 40 960 x 3 072 and 49 152 x 4 096 0.94 to 1.08, 128 256 x 4 096 0.68 to 0.82 and 8 192 x 28 672 0.36 to 0.51."""
    if rows >= 2048:
        return k > 1152 and library_fills(rows, n)
    return (rows <= 320 and 512 < n <= 1024 and 2048 <= k <= 4096) or (96 < rows <= 192 and 16384 <= n <= 32768 and k <= 9600 and n * k >= 117e6)


@functools.lru_cache(maxsize=4096)
def _plan(dtype, rows, n, k):
    shape, splits = ctypes.c_int32(), ctypes.c_int32()
    f = hip.lib().tf_rows_gemm_plan if dtype == torch.float16 else hip.tile_lib().tfl_rows_gemm_plan
    floats = f(rows, n, k, ctypes.byref(shape), ctypes.byref(splits))
    if floats < 0:
        hip.check(floats, "rows_gemm_plan")
    return shape.value, splits.value, floats


@functools.lru_cache(maxsize=4096)
def _choice(dtype, rows, k, n):
    """linear's plan of the kernel, None where the library is taken.  (One look-up: at 50 rows a forward waits for the host.)"""
    return None if library_is_faster(rows, n, k) else _plan(dtype, rows, n, k)[:2]


def product(x, w, form=PLAIN, plan=None):
    """The kernel's product.  plan = (shape, splits): another than its own choice."""
    (rows, k), n = x.shape, w.shape[0]
    if plan is None:
        shape, splits, floats = _plan(x.dtype, rows, n, k)
    else:
        shape, splits = plan
        floats = splits * rows * n if splits > 1 else 0
    n_out = n if form == PLAIN else n // 2
    out = torch.empty(rows, n_out, dtype=x.dtype, device=x.device)
    ws = torch.empty(floats, dtype=torch.float32, device=x.device) if floats else None
    f, name = (hip.lib().tf_rows_gemm, "tf_rows_gemm") if x.dtype == torch.float16 else (hip.tile_lib().tfl_rows_gemm, "tfl_rows_gemm")
    hip.check(f(x.data_ptr(), x.stride(0), w.data_ptr(), out.data_ptr(), n_out, ws.data_ptr() if floats else None, floats, rows, n, k, form, shape, splits,
                torch.cuda.current_stream().cuda_stream), name)
    return out


def linear(x, w):
    """x . W^T, w [n, k] contiguous.  Up to 32 rows only large weights are the kernel's: 18 784 x 4 096 at 16 rows 67 -> 38 us, 4 096 x 11 008 29 -> 23,
    but 4 096 x 4 096 11.0 -> 11.7, 256 x 4 096 7.8 -> 10.0 (at 40 rows 12.6 -> 12.3 and 11.3 -> 9.8)."""
    if (x.shape[0] > 32 or w.numel() > 1 << 25) and takes(x, w):
        plan = _choice(x.dtype, *x.shape, w.shape[0])
        if plan is not None:
            return product(x, w, PLAIN, plan)
    return F.linear(x, w)


def glu_linear(x, w, form):
    """The gated unit ``form`` of x . W^T in one launch, None where it is not one.  (65 to 160 rows of 22 016 x 4 096 are 2 to 4 us more than the library's
    product and the unit's launch, 48 -> 51, whose calls cost the host 16 more.)"""
    return product(x, w, form) if takes(x, w, form) else None
