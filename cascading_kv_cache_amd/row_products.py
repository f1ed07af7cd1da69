"""Products of a few rows: the projections of a decoding step, each with what surrounds it in a decoder layer (norm in front; bias,
gate or residual behind) in one launch of the library, the same bits as the operations it stands for.

A product's bits hang on the order its float32 sums are added up in, and a rounding that flips in one hidden state is a percent of
the logits of a decoder of random weights further on.  So the library's kernel is used where one of the orders it knows is that of
torch's product of the same sizes (:func:`library_orders` tries them, once, when a decoder fuses its projections), and torch's product
stays everywhere else.
"""
import math

import torch
from torch import nn

from . import _abi
from .cascading_cache import on_device, raw_stream

ROW_TYPES = (torch.bfloat16, torch.float16)
_GATED_TYPES = (torch.bfloat16, torch.float16, torch.float32)
#: (parts, unit) of ``ckv_linear_rows``, or (parts, unit, runs): see :func:`_cut_orders`
ORDERS = ((1, 1), (4, 1), (4, 2), (2, 2))
MAX_ROWS = 16
# not public: where torch lacks one of them, somebody may be following
_function_modes = getattr(torch._C, "_len_torch_function_stack", lambda: 1)
_dispatch_modes = getattr(torch._C, "_len_torch_dispatch_stack", lambda: 1)
_functorch_levels = getattr(getattr(torch._C, "_functorch", None), "peek_interpreter_stack", lambda: 1)


def followed(x) -> bool:
    """May anybody follow torch's operations on ``x``: gradients of either mode, vmap, tracing, a tensor subclass, a mode?"""
    return (type(x) is not torch.Tensor or torch.is_grad_enabled() or x.requires_grad or _function_modes() != 0 or _dispatch_modes() != 0
            or getattr(torch.autograd.forward_ad, "_current_level", 0) >= 0 or _functorch_levels() is not None
            or torch.jit.is_tracing() or torch.compiler.is_compiling())


#: kind of module: (name, method) of what calling one runs
_OWN = {}


def own_methods(kind, *names):
    """Takes down the methods that calling a ``kind`` runs, ``forward`` and the named ones, for :func:`plain` to know them by."""
    def own(name):
        method, home = getattr(kind, name), next(c for c in kind.__mro__ if name in vars(c))
        # torch's classes may have been given another one before
        original = (method.__module__ == home.__module__ and method.__qualname__.startswith(home.__qualname__ + ".")
                    and not hasattr(method, "__wrapped__"))
        return name, method if original else None
    _OWN[kind] = tuple(map(own, ("__call__", "_call_impl", "forward", *names)))


own_methods(nn.Linear)


def plain(module, kind) -> bool:
    """Is calling ``module`` nothing but the methods that :func:`own_methods` has taken down for ``kind``: no subclass, no hooks, not
    compiled, no method put on the object or on its class since?"""
    every = nn.modules.module
    if not (type(module) is kind and not module._forward_hooks and not module._forward_pre_hooks
            and getattr(module, "_compiled_call_impl", None) is None
            and not getattr(every, "_global_forward_hooks", True) and not getattr(every, "_global_forward_pre_hooks", True)):
        return False
    for name, method in _OWN[kind]:
        if getattr(kind, name) is not method or name in module.__dict__:
            return False
    return True


def gated_silu(gate_up):
    """``silu(gate) * up`` of rows of ``gate | up``: one launch of the library, the same bits, where nobody follows what is done."""
    if gate_up.device.type != "cuda" or not gate_up.is_contiguous() or gate_up.dtype not in _GATED_TYPES or followed(gate_up):
        gate, up = gate_up.chunk(2, dim=-1)
        return nn.functional.silu(gate) * up
    inter = gate_up.size(-1) // 2
    out = torch.empty(gate_up.shape[:-1] + (inter,), dtype=gate_up.dtype, device=gate_up.device)
    with on_device(gate_up.device):
        _abi.check(_abi.lib().ckv_gated_silu(gate_up.data_ptr(), out.data_ptr(), gate_up.numel() // (2 * inter), inter, 2 * inter,
                                             _abi.dtype_code(gate_up.dtype), raw_stream(gate_up.device)), "ckv_gated_silu")
    return out


def _fits(rows, n, k, order, norm) -> bool:
    """Sizes that ``ckv_linear_rows`` takes: the rows, the norm's weights and a ring of stages share the LDS of a compute unit."""
    ring = {1: 4 * 4, 2: 2 * 8, 4: 4 * 4}[order[0]] * 2048
    return 0 < rows <= MAX_ROWS and n % 16 == 0 and k % 64 == 0 and ring + rows * (2 * k + 16) + 2 * k * norm + 256 <= 160 * 1024


def _crowded(rows, n, k, order, units) -> bool:
    """Is a product with the norm in front slower than torch's because one workgroup, of 16 outputs, fills a compute unit's LDS?  Each of
    them brings and normalises the rows again, which nothing covers then, round after round.  us, torch's operations and the kernel, four
    parts:  152064 x 3584, by rows  2: 226 163  3: 226 175  4: 227 323   100352 x 4096  2: 182 123  3: 182 197; with few rounds it is
    level (6144 x 4096  3: 19.5 18.1  4: 19.6 20.6), and one part has more outputs a workgroup (128256 x 4096  4: 190 161)."""
    return order[0] == 4 and n // 16 > 4 * units and 2 * (6 * 4 * 2048 + rows * (2 * k + 16) + 2 * k + 256) > 160 * 1024


def _at(t) -> int:
    return 0 if t is None else t.data_ptr()


def linear_rows(x, weight, order, bias=None, residual=None, norm=None, eps=0.0, gated=False):
    """``ckv_linear_rows`` of ``x (B, q, k)``, whose rows lie a fixed stride apart (a single row has none)."""
    n, k = weight.shape
    rows = x.size(0) * x.size(1)
    out = torch.empty(x.shape[:-1] + (n // 2 if gated else n,), dtype=x.dtype, device=x.device)
    stride = k if rows == 1 else x.stride(0) if x.size(1) == 1 else x.stride(1)
    with on_device(x.device):
        _abi.check(_abi.lib().ckv_linear_rows(x.data_ptr(), weight.data_ptr(), _at(bias), _at(residual), _at(norm), eps, out.data_ptr(),
                                              rows, n, k, stride, int(gated), order[0], order[1] + 256 * sum(order[2:]),
                                              _abi.dtype_code(x.dtype), raw_stream(x.device)), "ckv_linear_rows")
    return out


def _rows_apart(x) -> bool:
    """Are the rows of ``x (B, q, k)`` contiguous, a fixed stride of whole 16-byte pieces apart, and aligned?"""
    if x.dim() != 3 or x.stride(2) != 1 or x.data_ptr() % 16:
        return False
    b, q, k = x.shape
    sb, sq, _ = x.stride()
    return (b == 1 or (sb if q == 1 else sq * q) == sb) and (b * q == 1 or (sb if q == 1 else sq) % 8 == 0) and (q == 1 or sq >= k) and (b == 1 or sb >= k)


def _operand(t, x, *shape) -> bool:
    return (type(t) in (torch.Tensor, nn.Parameter) and t.dtype == x.dtype and t.device == x.device and t.shape == shape and t.is_contiguous()
            and t.data_ptr() % 16 == 0)


def row_linear(x, weight, orders, bias=None, norm=None, residual=None, gated=False):
    """``residual + linear(norm(x))``, or the gate of it, of ``x (B, q, k)`` (nobody follows, see :func:`followed`): one launch where
    ``orders`` (rows: order) has one for so many rows.  ``norm``: a fused RMSNorm module."""
    rows, (n, k) = x.size(0) * x.size(1), weight.shape   # three dimensions: the callers ask
    order = orders.get(rows)
    if (order is not None and x.size(2) == k and (order[0] == 1 or not gated) and _fits(rows, n, k, order, norm is not None) and _rows_apart(x)
            and _operand(weight, x, n, k) and (bias is None or _operand(bias, x, n)) and (norm is None or _operand(norm.weight, x, k))
            and (residual is None or _operand(residual, x, x.size(0), x.size(1), n))):
        return linear_rows(x, weight, order, bias, residual, None if norm is None else norm.weight, 0.0 if norm is None else norm.eps, gated)
    y = nn.functional.linear(x if norm is None else norm(x), weight, bias)
    if gated:
        y = gated_silu(y)
    return y if residual is None else residual + y


# not public: where torch lacks one of them, its public form is slower or there is no such switch
_SETTINGS = (getattr(torch._C, "_get_blas_preferred_backend", getattr(torch.backends.cuda, "preferred_blas_library", None)),
             *(getattr(torch._C, name, None) for name in ("_get_cublas_allow_bf16_reduced_precision_reduction",
                                                          "_get_cublas_allow_fp16_reduced_precision_reduction",
                                                          "_get_cublas_allow_fp16_accumulation", "_cuda_tunableop_is_enabled")))
_SETTINGS = tuple(f for f in _SETTINGS if f is not None)
_tuning = getattr(torch._C, "_cuda_tunableop_is_enabled", lambda: False)


def product_settings() -> tuple:
    """What decides, beside its sizes, which product torch runs (0.5 us)."""
    return (torch.__version__, *[f() for f in _SETTINGS])


#: what library_orders has found, by device, type, sizes and settings: facts about torch's products and norms, not about a weight
_FOUND = {}


def _chains(order, k) -> tuple:
    """The stretches of 64 elements that each chain of a sum adds up; two orders with the same chains are one."""
    parts, unit = order
    chains = (tuple(s for s in range(k // 64) if s // unit % parts == part) for part in range(parts))
    return tuple(c for c in chains if c)


def _cut_orders(n, k, units) -> list:
    """Orders of a library that lays the tiles which do not come out even on its workgroups (of 256 rows of the weight and 64 elements, or
    of 32 rows and 256 elements) end to end and cuts the line into runs of one length, whatever tiles they end in: by the number of its
    workgroups, for which it takes most of a chip of ``units`` compute units.  Of numbers that cut alike the largest."""
    found = {}
    for runs in range(units, units * 3 // 4, -1):
        for parts, height in ((1, 256), (4, 32)):
            tiles, span = -(-n // height), k // (64 * parts)
            if k % (64 * parts) == 0 and tiles > runs and tiles % runs:
                shared = tiles % runs + runs
                found.setdefault((parts, shared, -(-shared * span // runs)), (parts, 1, runs))
    return list(found.values())


_FRACTION = {torch.bfloat16: 8, torch.float16: 11}   # bits of a value, the leading one included


def _norms_like_torch(k, eps, most_rows, like) -> set:
    """Numbers of rows whose norm in front of a product has the bits of torch's, looked at through a product with the identity.  Another
    order of the sum of squares moves half the rows' factors by the last bit of a float32, which rounds one element of 65536 of bfloat16
    (8192 of float16) to another value: enough rows are tried to expect eight."""
    key = ("norm", like["device"], like["dtype"], k, eps, most_rows, product_settings())
    if key in _FOUND:
        return _FOUND[key]
    left = {rows for rows in range(1, most_rows + 1) if _fits(rows, k, k, (1, 1), True)}
    enough = math.ceil(8 * 2 ** (25 - _FRACTION[like["dtype"]]) / k)
    same, w = torch.eye(k, device=like["device"], dtype=like["dtype"]), 1 + 0.1 * torch.randn(k, **like)
    for rows in sorted(left):
        differ = torch.zeros((), dtype=torch.int64, device=like["device"])
        for x in torch.randn(math.ceil(enough / rows), rows, 1, k, **like):
            differ += (linear_rows(x, same, (1, 1), norm=w, eps=eps) != nn.functional.rms_norm(x, (k,), w, eps)).sum()
        if differ.item():
            left.remove(rows)
    _FOUND[key] = left
    return left


def library_orders(weight, bias=None, most_rows=4, norm=None, cut=False):
    """``{rows: order}`` whose bits are those of ``torch.nn.functional.linear`` for so many rows of 16 bits, with a fused RMSNorm module
    in front or none, found by trying, 20 to 60 ms a size, once.  ``cut``: of the orders of :func:`_cut_orders` too (0.2 s).

    Rows, weights and bias are drawn, so that what is found hangs on sizes and settings alone and not on a model that is all zeros or has
    a NaN.  Two orders differ in few outputs (4096 x 4096: one of 4000 to 6000), in proportion to the root of the products summed up.  A
    library whose tiles do not come out even on its workgroups cuts the last ones up, and such an order differs from the others' in an
    output or two a row (152064 x 3584).  So 64 rows are tried, which also expects eight differences of the smallest product that is
    taken, twice as many while two are left, and if two are left then there is none.

    Four rows: the norm of five costs the products behind it more than torch takes (6144 x 4096 with the norm, us, torch's operations and
    the kernel, by rows  1: 19.6 10.9  3: 19.5 18.1  4: 19.6 20.6  5: 19.5 23.0; the four products of that layer  1: 136 84  4: 131 98),
    and 4 x 14336 is all that fits."""
    if (type(weight) not in (torch.Tensor, nn.Parameter) or _dispatch_modes() != 0 or _functorch_levels() is not None
            or weight.device.type != "cuda" or weight.dtype not in ROW_TYPES or not weight.is_contiguous() or _tuning()):
        return {}
    n, k = weight.shape
    if 3.5e6 / (n * math.sqrt(k)) > 64:   # rows that eight differences take
        return {}
    key = (weight.device, weight.dtype, n, k, bias is not None, most_rows, None if norm is None else norm.eps, cut, product_settings())
    if key in _FOUND:
        return _FOUND[key]
    if torch.cuda.is_current_stream_capturing():
        return {}
    orders = {}
    like = dict(generator=torch.Generator(device=weight.device).manual_seed(n + k), device=weight.device, dtype=weight.dtype)
    with torch.no_grad(), torch.autocast("cuda", enabled=False):
        try:
            w, b = torch.randn(n, k, **like), None if bias is None else torch.randn(n, **like)
        except torch.OutOfMemoryError:   # a model that fills the device: nothing is tried, and nothing taken down
            return {}

        def agreeing(left, rows):
            tried = 0
            while left and (tried < 64 or (len(left) > 1 and tried < 128)):
                x = torch.randn(rows, 1, k, **like)
                want = nn.functional.linear(x, w, b)
                left = [o for o in left if torch.equal(linear_rows(x, w, o, b), want)]
                tried += rows
            return left

        units = torch.cuda.get_device_properties(weight.device).multi_processor_count
        for rows in range(1, most_rows + 1) if norm is None else sorted(_norms_like_torch(k, norm.eps, most_rows, like)):
            fits = [o for o in ORDERS if _fits(rows, n, k, o, norm is not None) and (norm is None or not _crowded(rows, n, k, o, units))]
            left = agreeing(list({_chains(o, k): o for o in reversed(fits)}.values()), rows)
            if cut and not left:
                left = agreeing([o for o in _cut_orders(n, k, units) if o[:2] in fits], rows)
            if len(left) == 1:
                orders[rows] = left[0]
    _FOUND[key] = orders
    return orders
