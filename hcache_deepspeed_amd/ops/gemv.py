"""bf16 linears of up to 1,100 rows: ``linear(x, w, b)`` equals ``F.linear``. One row and the shapes where its weight stream is
faster than hipBLASLt's small-M GEMM (``profiles/gemv_bench_r2.jsonl``) run the HIP GEMV, 2 to 16 rows the matrix-core skinny GEMM
(both csrc/kernels/gemv.hip), 9 and more the tiled one (csrc/kernels/linear.hip) where ``hds_linear_plan`` takes them; everything
else goes to ``F.linear``."""
import functools

import torch
import torch.nn.functional as F
from torch.utils._device import DeviceContext

from . import native

# Weight sizes (elements) that take the GEMV. At M = 1 every size does: in a real decode step (weights streamed from
# HBM, not re-read from the 256 MB MALL as in a micro-benchmark loop) the GEMV beats hipBLASLt's small-M GEMM on the
# gate_up projection and the LM head as well -- Llama-3-8B v2 decode 234.8 vs 211.0 tok/s at B = 1, same box
# (profiles/r3/v2_decode_gemv_rule_r3.jsonl). Its dot products make it VALU-bound as M grows (M = 4: qkv 1.4x,
# down 0.73x; M = 8: o 1.36x, qkv 0.98x, gate_up a loss in decode: 1124 vs 1462 tok/s at B = 8), so beyond one row
# the limit is 32M elements up to M = 4 and 16M up to M = 8 (profiles/gemv_bench_r2.jsonl).
_os = __import__("os")
MAX_GEMV_NUMEL_M1 = int(_os.environ.get("HDS_GEMV_MAX_NUMEL_M1", str(1 << 40)))
MAX_GEMV_NUMEL = int(_os.environ.get("HDS_GEMV_MAX_NUMEL", str(64 * 1024 * 1024)))


def max_numel(M):
    return MAX_GEMV_NUMEL_M1 if M == 1 else MAX_GEMV_NUMEL >> (1 if M <= 4 else 2)


def gemv_ok(x2, w, b=None):
    if not (native.use_native(x2) and x2.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and w.dim() == 2):
        return False
    M, K = x2.shape
    N = w.shape[0]
    if M > 8 or w.shape[1] != K or not w.is_contiguous() or x2.stride(1) != 1 or x2.stride(0) % 8:
        return False
    if x2.data_ptr() % 16 or w.data_ptr() % 16 or N * K > max_numel(M):
        return False
    if b is not None and (b.dtype != torch.bfloat16 or not b.is_contiguous()):
        return False
    return bool(native.kernels().hds_gemv_bf16_supported(M, N, K))


def gemv(x2, w, b=None):
    M, K = x2.shape
    N = w.shape[0]
    y = torch.empty(M, N, dtype=x2.dtype, device=x2.device)
    native.check(native.kernels().hds_gemv_bf16(x2.data_ptr(), w.data_ptr(), native.ptr(b), y.data_ptr(), M, N, K,
                                                x2.stride(0), N, native.stream()), "gemv_bf16")
    return y


# 2..16 token rows: the matrix-core skinny GEMM (csrc/kernels/gemv.hip skinny_lines_kernel) instead of the VALU GEMV /
# hipBLASLt's small-M tiles (HDS_SKINNY_GEMM=0: those)
SKINNY = _os.environ.get("HDS_SKINNY_GEMM", "1") == "1"
MAX_ROWS = 16  # of either kernel
SKINNY_MIN_M = int(_os.environ.get("HDS_SKINNY_MIN_M", "2"))  # 1: one-row linears too (instead of the VALU GEMV)


def _skinny_wanted(n, K):
    """Do the switches leave up to MAX_ROWS rows (n values of K) to the matrix-core kernels, skinny or tiled?"""
    return SKINNY and n >= SKINNY_MIN_M * K


def skinny_ok(x2, w, b=None):
    if not (SKINNY and native.use_native(x2) and x2.dtype == torch.bfloat16 and w.dtype == torch.bfloat16
            and w.dim() == 2):
        return False
    M, K = x2.shape
    if not SKINNY_MIN_M <= M <= MAX_ROWS or w.shape[1] != K or K % 128 or not w.is_contiguous() or x2.stride(1) != 1 or x2.stride(0) % 8:
        return False
    if x2.data_ptr() % 16 or w.data_ptr() % 16:
        return False
    return b is None or (b.dtype == torch.bfloat16 and b.is_contiguous())


def skinny(x2, w, b=None):
    M, K = x2.shape
    N = w.shape[0]
    y = torch.empty(M, N, dtype=x2.dtype, device=x2.device)
    native.check(native.kernels().hds_skinny_gemm_bf16(x2.data_ptr(), w.data_ptr(), native.ptr(b), y.data_ptr(), M, N,
                                                       K, x2.stride(0), N, 0, native.stream()), "skinny_gemm_bf16")
    return y


# 9 to 1,100 rows: csrc/kernels/linear.hip where hds_linear_plan takes them
_TENSORS = (torch.Tensor, torch.nn.Parameter)


@functools.lru_cache(maxsize=4096)
def _plan(M, N, K, glu=0):
    """Tile + 16 x slices of K on csrc/kernels/linear.hip, 0 for products that stay the library's."""
    return int(native.kernels().hds_linear_plan(M, N, K, glu)) if max(M, N, K) < 1 << 31 else 0


_dispatch_modes, _function_modes = torch._C._len_torch_dispatch_stack, torch._C._len_torch_function_stack


def _watched():
    """Does a function mode see or replace operations (a default device does neither)?"""
    return any(type(torch._C._get_function_stack_at(i)) is not DeviceContext for i in range(_function_modes()))


def rows_linear(x, w, b=None, glu=0, out=None):
    """``F.linear(x, w, b)`` of 9 rows and more, or with ``glu`` = 1 + activation code the gated unit of w = [gate; up],
    written to ``out`` (contiguous, x's type) where given; None where the kernel does not take the call, as where anything could want a record of it (``native.plain``, torch.compile, a
    dispatch or function mode: a trace by make_fx, a counter, fake tensors would find the allocation of the result only)."""
    if torch.compiler.is_compiling():
        return None
    # (sizes first: a call of a prompt that stays the library's pays 2 us less for having asked)
    if type(x) not in _TENSORS or not x.is_cuda or torch._C._get_tracing_state() is not None:
        return None
    shape = x.shape
    K = shape[-1] if len(shape) else 0
    if K == 0:
        return None
    rows = w.shape[0]
    M, N = x.numel() // K, rows // 2 if glu else rows
    plan = _plan(M, N, K, 1 if glu else 0)
    # (autocast to another type is the library call's to see, and so is a tensor on another device than the current one, whose
    # stream the launch would take)
    if plan == 0 or torch.is_autocast_enabled() or x.get_device() != torch.cuda.current_device():
        return None
    if not native.plain(x, w, b) or _dispatch_modes() or (_function_modes() and _watched()):
        return None
    if x.dtype != torch.bfloat16 or w.dtype != torch.bfloat16 or w.dim() != 2 or not w.is_contiguous() or K != w.shape[1] or \
            w.get_device() != x.get_device():
        return None
    x2 = x if x.dim() == 2 else x.reshape(M, K)
    ld, one = x2.stride()
    px, pw = x2.data_ptr(), w.data_ptr()
    if one != 1 or ld % 8 or not K <= ld <= 1 << 22 or (px | pw) % 16 or (glu and rows % 2):
        return None
    if b is not None and (b.dtype != torch.bfloat16 or not b.is_contiguous() or b.shape != w.shape[:1] or
                          b.get_device() != x.get_device()):
        return None
    if out is not None and (out.dtype != torch.bfloat16 or out.device != x.device or not out.is_contiguous()
                            or out.shape != (M, N) or out.data_ptr() % 8):
        return None
    y = torch.empty(M, N, dtype=torch.bfloat16, device=x.device) if out is None else out
    part = torch.empty(plan // 16, M, rows, dtype=torch.float32, device=x.device) if plan >= 32 else None
    native.check(native.kernels().hds_linear_bf16(px, ld, pw, native.ptr(b), y.data_ptr(), N, native.ptr(part), M, N, K, glu,
                                                  plan, native.stream()), "linear_bf16")
    return y if x.dim() == 2 else y.view(*x.shape[:-1], N)


# Norms between the products of 2 to 16 rows, without a launch of their own (csrc/kernels/row_norm.h)
class ScaledRows:
    """RMS-normed rows before their factor of each row: ``x`` is bf16(r * gamma) of the residual stream r, ``ssq`` holds the
    sums of r * r of every 16 columns, [columns / 16, 16], which the product behind makes the factors of."""

    __slots__ = ("x", "ssq", "eps")

    def __init__(self, x, ssq, eps):
        self.x, self.ssq, self.eps = x, ssq, eps


def scaled_rows_ok(M):
    """May steps of M rows go through ``norm_linear`` and ``scaled_linear``? Where the skinny kernel takes them and nothing could
    want a record of the separate operations."""
    return (SKINNY and max(2, SKINNY_MIN_M) <= M <= MAX_ROWS and not torch.is_grad_enabled()
            and torch._C._get_tracing_state() is None and not torch.compiler.is_compiling() and not _dispatch_modes()
            and not (_function_modes() and _watched()) and not torch.is_autocast_enabled())


def scaled_weight_ok(w, into=False):
    """Is ``w`` [out, in] one that ``scaled_linear`` takes, or (``into``) ``norm_linear``?"""
    return (torch.is_tensor(w) and w.is_cuda and w.dtype == torch.bfloat16 and w.dim() == 2 and w.is_contiguous()
            and w.data_ptr() % 16 == 0 and w.shape[1] % 128 == 0 and (not into or w.shape[0] % 16 == 0))


def norm_linear(x, w, res, gamma, eps):
    """(``ScaledRows`` of RMSNorm(x . w^T + res) * gamma, the new residual stream). x [M, K], res [M, N] contiguous bf16; the
    product and the sum are rounded as ``linear`` and the norm's kernel round them."""
    M, K = x.shape
    N = w.shape[0]
    assert x.is_contiguous() and res.is_contiguous() and res.shape == (M, N) and gamma.is_contiguous() and gamma.numel() == N
    assert x.dtype == res.dtype == gamma.dtype == torch.bfloat16 and w.shape[1] == K
    y, r = torch.empty_like(res), torch.empty_like(res)
    ssq = torch.empty(N // 16, 16, dtype=torch.float32, device=x.device)
    native.check(native.kernels().hds_skinny_norm_bf16(x.data_ptr(), w.data_ptr(), y.data_ptr(), None, 0.0, res.data_ptr(),
                                                       gamma.data_ptr(), r.data_ptr(), ssq.data_ptr(), M, N, K, 0,
                                                       native.stream()), "skinny_norm_bf16")
    return ScaledRows(y, ssq, float(eps)), r


def scaled_linear(rows, w, act=None):
    """The normed rows times w^T, or with ``act`` the gated unit of w = [gate; up]."""
    x, glu = rows.x, 0 if act is None else 1 + _GATHER_ACTS[act]
    M, K = x.shape
    N = w.shape[0] // 2 if glu else w.shape[0]
    assert w.shape[1] == K == 16 * rows.ssq.shape[0]
    y = torch.empty(M, N, dtype=x.dtype, device=x.device)
    plan = _plan(M, N, K, 1 if glu else 0) if M > 8 else 0
    lib = native.kernels()
    if 0 < plan < 32 and plan % 16 < 2:
        native.check(lib.hds_linear_scaled_bf16(x.data_ptr(), w.data_ptr(), y.data_ptr(), rows.ssq.data_ptr(), rows.eps, M, N, K,
                                                glu, plan, native.stream()), "linear_scaled_bf16")
    else:
        native.check(lib.hds_skinny_norm_bf16(x.data_ptr(), w.data_ptr(), y.data_ptr(), rows.ssq.data_ptr(), rows.eps, None,
                                              None, None, None, M, N, K, glu, native.stream()), "skinny_norm_bf16")
    return y


def _needs_grad(*tensors):
    """The kernels have no backward, and a trace would hold the allocation of their result only: with gradients wanted, or a
    trace in progress, the products are torch's."""
    return (torch.is_grad_enabled() and any(torch.is_tensor(t) and t.requires_grad for t in tensors)) or \
        torch._C._get_tracing_state() is not None


def glu_linear(x, w, b, act):
    """act(x . gate^T) * (x . up^T) for ``w`` = [gate; up] (and ``b``) in one call, for 2..16 rows of the skinny GEMM and 9..256
    of ``rows_linear``; None for anything else. The projections are rounded to bf16 first, as the separate kernels store them."""
    if act not in _GATHER_ACTS or not (x.dim() >= 1 and x.is_cuda and torch.is_tensor(w)):
        return None
    if x.numel() > 256 * x.shape[-1] or _needs_grad(x, w, b):
        return None
    n, K = x.numel(), x.shape[-1]
    if n > MAX_ROWS * K or (n > 8 * K and _skinny_wanted(n, K)):
        y = rows_linear(x, w, b, 1 + _GATHER_ACTS[act])
        if y is not None or n > MAX_ROWS * K:
            return y
    x2 = x.reshape(-1, x.shape[-1])
    if not skinny_ok(x2, w, b) or w.shape[0] % 2:
        return None
    (M, K), N = x2.shape, w.shape[0] // 2
    y = torch.empty(M, N, dtype=x2.dtype, device=x2.device)
    native.check(native.kernels().hds_skinny_gemm_bf16(x2.data_ptr(), w.data_ptr(), native.ptr(b), y.data_ptr(), M, N,
                                                       K, x2.stride(0), N, 1 + _GATHER_ACTS[act], native.stream()),
                 "skinny_gemm_bf16")
    return y.view(*x.shape[:-1], N)


def linear(x, w, b=None):
    """``F.linear(x, w, b)``; unless a gradient is wanted, bf16 inputs run the HIP GEMV (one row), the skinny matrix-core GEMM
    (2..16 rows) or, of 9 to 1,100 rows, the tiled and sliced one where it is the faster."""
    if x.dim() >= 1 and x.is_cuda:
        n, K = x.numel(), x.shape[-1]
        if n > MAX_ROWS * K:
            # (hds_linear_plan takes none beyond; asking costs 1 us, 3 % of the host's time for a prompt of that length)
            y = rows_linear(x, w, b) if n <= 320 * K or K >= 8192 else None
            if y is not None:
                return y
        elif not _needs_grad(x, w, b):
            if n > 8 * K and _skinny_wanted(n, K):
                y = rows_linear(x, w, b)
                if y is not None:
                    return y
            x2 = x.reshape(-1, K)
            if skinny_ok(x2, w, b):
                return skinny(x2, w, b).view(*x.shape[:-1], w.shape[0])
            if gemv_ok(x2, w, b):
                return gemv(x2, w, b).view(*x.shape[:-1], w.shape[0])
    return F.linear(x, w, b)


def fused_ok(h2, w, gamma=None, glu=False):
    """Can ``fused_gemv`` take these decode rows on the HIP kernel (bf16, <= 8 rows, 16-B aligned rows)?"""
    if not (native.use_native(h2) and h2.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and w.dim() == 2):
        return False
    M, K = h2.shape
    if M > 8 or w.shape[1] != K or K % 8 or not w.is_contiguous() or h2.stride(1) != 1 or h2.stride(0) != K:
        return False
    if glu and w.shape[0] % 2:
        return False
    if gamma is not None and (gamma.dtype != torch.bfloat16 or not gamma.is_contiguous() or gamma.numel() != K):
        return False
    return h2.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0 and w.numel() <= max_numel(M)


def _unfused(h2, w, res, gamma, eps, glu):
    from .activations import glu as _glu
    from .norm import rms_norm
    r, x = h2, h2
    if gamma is not None:
        if res is None:
            x = rms_norm(h2, gamma, eps)
        else:
            x, r = rms_norm(h2, gamma, eps, res)
    y = linear(x, w)
    return (_glu(y, "silu") if glu else y), r, x


def fused_gemv(h, w, res=None, gamma=None, eps=1e-5, glu=False, want_x=False, x_out=None):
    """Decode projection with the pre-norm and / or the gated activation folded in (csrc/kernels/gemv.hip
    ``hds_gemv_fused_bf16``). With ``gamma``: the rows are RMSNorm(h + res) * gamma -- the new residual ``h + res`` is
    returned too (``h`` itself without ``res``), and the normed rows when ``want_x`` (HCache hidden latents). With
    ``glu``: ``w`` is [gate; up] and the result is silu(x . gate^T) * (x . up^T). Returns (y, residual, x or None);
    rows or weights the fused kernel does not take run the unfused kernels (the same arithmetic). ``x_out``: a
    contiguous [rows, K] buffer the normed rows are written into (``want_x``; the unfused fallback returns its own)."""
    shape = h.shape
    h2 = h.reshape(-1, shape[-1])
    res2 = None if res is None else res.reshape(-1, shape[-1])
    N = w.shape[0] // 2 if glu else w.shape[0]
    ok = (fused_ok(h2, w, gamma, glu) and (gamma is not None or glu)
          and (res2 is None or (res2.dtype == h2.dtype and res2.stride() == h2.stride() and res2.data_ptr() % 16 == 0)))
    if not ok:  # the unfused kernels (GEMV or hipBLASLt by the size rules, RMSNorm, GLU): the model's other path
        y, r, x = _unfused(h2, w, res2, gamma, eps, glu)
    else:
        M, K = h2.shape
        y = torch.empty(M, N, dtype=h2.dtype, device=h2.device)
        r = h2 if res2 is None else torch.empty_like(h2)  # never in place: other workgroups still read res
        x = None
        if want_x and gamma is not None:
            ok_out = (x_out is not None and x_out.dtype == h2.dtype and x_out.is_contiguous()
                      and x_out.numel() == h2.numel() and x_out.data_ptr() % 16 == 0)
            x = x_out.view(h2.shape) if ok_out else torch.empty_like(h2)
        native.check(native.kernels().hds_gemv_fused_bf16(
            h2.data_ptr(), native.ptr(res2), native.ptr(gamma), float(eps), w.data_ptr(), y.data_ptr(),
            native.ptr(r if res2 is not None else None), native.ptr(x), int(bool(glu)), 0.0, M, N, K, K, N,
            native.stream()), "gemv_fused_bf16")
        if gamma is None:
            x = h2
    lead = shape[:-1]
    return (y.view(*lead, N), r.view(shape), None if x is None or not want_x else x.view(shape))


_GLU_GEMV_ACTS = {"silu": 0, "gelu_tanh": 1, "relu": 2, "clamped": 5}


def glu_gemv(x2, w, act, out, limit=0.0):
    """act(x . gate^T) * (x . up^T) (or the clamped unit) of decode rows into ``out`` [M, I] (strided column block) in one kernel; ``w`` is
    [gate; up]. Returns False, with nothing written, for rows or weights the kernel does not take."""
    if act not in _GLU_GEMV_ACTS or not torch.is_tensor(w) or not fused_ok(x2, w, None, True):
        return False
    M, K = x2.shape
    native.check(native.kernels().hds_gemv_fused_bf16(x2.data_ptr(), None, None, 0.0, w.data_ptr(), out.data_ptr(),
                                                      None, None, 1 + _GLU_GEMV_ACTS[act], float(limit), M,
                                                      w.shape[0] // 2, K,
                                                      x2.stride(0), out.stride(0), native.stream()), "glu_gemv")
    return True


_GATHER_ACTS = {"silu": 0, "gelu_tanh": 1, "relu": 2}


def gather_gemv(x2, w, act, table, ids):
    """act(x . w^T) * table[ids] of decode rows (at most 16) in one kernel, [M, N]; table: [vocab, N] with any row stride. None
    for rows or weights the kernel does not take."""
    if act not in _GATHER_ACTS or not torch.is_tensor(w) or x2.shape[0] > 16 or not (
            skinny_ok(x2, w) if x2.shape[0] > 1 else gemv_ok(x2, w)):
        return None
    assert table.dtype == x2.dtype and table.stride(1) == 1 and table.shape[1] == w.shape[0]
    assert ids.dtype == torch.int64 and ids.numel() == x2.shape[0]
    M, K = x2.shape
    y = torch.empty(M, w.shape[0], dtype=x2.dtype, device=x2.device)
    native.check(native.kernels().hds_gather_gemv_bf16(x2.data_ptr(), w.data_ptr(), table.data_ptr(), table.stride(0),
                                                       ids.data_ptr(), table.shape[0], _GATHER_ACTS[act], y.data_ptr(), M,
                                                       w.shape[0], K, x2.stride(0), y.stride(0), native.stream()),
                 "gather_gemv")
    return y
