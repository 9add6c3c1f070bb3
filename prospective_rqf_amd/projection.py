"""Projection GEMMs around the scans: drive ``z = W h`` and selector logits.

The reference computes these with plain ``torch.matmul`` calls:
``_SelectiveLayerScan`` (rqf_models/ops/selective_scan.py:117-118, 144-146),
``_SplitProjection`` (rqf_models/backbones/rqf/selective.py:78-97) and, through
autograd, the FBT stack's ``W_c @ h`` (rqf_models/backbones/rqf/pure.py:222-223).
Their weight gradients reduce over batch*time (~1e6 columns) into a small
(out, in) matrix.  A single GEMM of that shape has only a handful of output
tiles to spread over the 256 CUs.  On MI355X the complex64 one runs at
2.4 TFLOP/s: ``dz @ x.mH`` takes 222 ms at B=64, T=16000, H=256, against
2.8 ms for the scan's whole backward.  Here the columns are split over blocks
whose partial products are summed (csrc/wgrad.hip); tensors that kernel does not
serve go through ``splits`` batched library GEMMs, likewise summed.

The products with a weight on the left, ``W h`` and ``W^H g``, run on the kernels of
csrc/proj.hip for float32 and complex64 device tensors (``matmul``,
``matmul_adjoint``) and on torch elsewhere.  ``fused_forward`` and ``fused_dx`` stack several of them in one:
- the drive GEMM and the selector projection stacked into one real GEMM over
  the interleaved complex input, with no ``[Re; Im]`` copy;
- their input gradients likewise stacked, reading ``dz`` and the logit
  gradients where they lie.
"""

from __future__ import annotations

import ctypes

import torch
from torch import Tensor
from torch.autograd import forward_ad

# Batched GEMMs the reduction is split into, and the least columns per split.
# Measured on MI355X for (out, in, batch*time) = (256, 256, 1.02e6):
# 16 -> 14.0 ms, 32 -> 7.0, 64 -> 3.9, 128 -> 4.0, 256 -> 4.6; at (48, 48, 5.1e5):
# 64 -> 1.78 ms, 128 -> 0.17, 256 -> 0.18.
WGRAD_SPLITS = 128
WGRAD_MIN_COLUMNS = 1024


def unobserved() -> bool:
    """Whether plain tensors are all there is to a call: no open level of dual numbers,
    whose tangents a kernel would drop, and no tracer or dispatch mode, which would take
    its result for a constant."""
    return (forward_ad._current_level < 0 and not torch._C._is_tracing()
            and torch._C._len_torch_dispatch_stack() == 0 and not torch.compiler.is_compiling())


# Columns and matrix side from which the kernel beats the batched GEMMs: complex 48 x 48,
# 4000 columns 23 against 49 us; real 520 x 512, 1000 columns 35 against 21 us, 4000 42
# against 56; real 10 x 256, 512000 columns 146 against 122 us.
WGRAD_KERNEL_COLUMNS, WGRAD_KERNEL_SIDE = 2048, 16


def _wgrad_serves(g: Tensor, x: Tensor, columns: int = WGRAD_KERNEL_COLUMNS,
                  least: int = WGRAD_KERNEL_SIDE) -> bool:
    """Whether ``outer_sum`` takes these contiguous matrices, as ``_kernel_serves``."""
    side = min(t.shape[0] * (2 if t.is_complex() else 1) for t in (g, x))
    return (
        x.shape[1] >= columns and side >= least
        and max(g.shape[0], x.shape[0]) <= MAX_SIDE
        and all((t.dtype is torch.complex64 or t.dtype is torch.float32) and type(t) in _PLAIN
                and t.is_cuda and t.get_device() == torch._C._cuda_getDevice()
                and not t.is_conj() and not t.is_neg() and torch._C._has_storage(t)
                for t in (g, x))
        and not (torch.is_grad_enabled() and (g.requires_grad or x.requires_grad))
        and not torch.is_autocast_enabled("cuda")
        and unobserved()
    )


def outer_sum(a: Tensor, b: Tensor) -> Tensor:
    """The sum over the columns of contiguous ``a`` (M, N) and ``b`` (K, N), complex64 or
    float32, on the device: ``a @ b^H`` (M, K) for two complex or two real ones,
    ``a @ [Re b; Im b]^T`` (M, 2K) and ``[Re a; Im a] @ b^T`` (2M, K) for one of each."""
    from prospective_rqf_amd import _lib

    (m, n), k = a.shape, b.shape[0]
    ac, bc = a.is_complex(), b.is_complex()
    out = torch.empty(2 * m if ac and not bc else m, 2 * k if bc and not ac else k,
                      dtype=a.dtype if ac and bc else torch.float32, device=a.device)
    lib = _lib.load()
    nbytes = lib.rqf_weight_grad_workspace(m, ac, k, bc, n)
    ws = _lib.workspace(nbytes, a.device)
    _lib.check(lib.rqf_weight_grad(a.data_ptr(), m, ac, b.data_ptr(), k, bc, n, out.data_ptr(),
                                   _lib.ptr(ws), nbytes, _lib.stream_of(a)), "rqf_weight_grad")
    return out


# The kernel reads a complex operand where it lies, from the first column on, but pads a
# narrow real one to 64 rows.  Against batched products of the interleaved storage (us):
# 128 complex rows and 3, 1000 columns 14 against 18, 512000 columns 178 against 150; and
# 8, 177 against 175; 48 and 3, 131072 columns 29 against 31, 262144 46 against 45.
WGRAD_NARROW, WGRAD_NARROW_MOST = 8, 1 << 24


def real_weight_grad(a: Tensor, b: Tensor) -> Tensor:
    """``A @ B^T`` for one complex and one real operand, the complex one as its
    ``[Re; Im]`` rows.  A complex ``a`` is not copied."""
    if a.is_complex():
        if ((b.shape[0] >= WGRAD_NARROW or a.numel() < WGRAD_NARROW_MOST)
                and _wgrad_serves(a, b, 1, 1)):
            return outer_sum(a, b)
        # [Re a; Im a] b^T from the interleaved storage against b spread over it
        (m, n), k = a.shape, b.shape[0]
        spread = torch.zeros(2 * k, 2 * n, dtype=b.dtype, device=b.device)
        spread[:k, 0::2] = b
        spread[k:, 1::2] = b
        g = weight_grad(torch.view_as_real(a).reshape(m, 2 * n), spread)
        return torch.cat((g[:, :k], g[:, k:]))
    if _wgrad_serves(a, b):
        return outer_sum(a, b)
    return weight_grad(a, torch.cat((b.real, b.imag)))


def weight_grad(g: Tensor, x: Tensor, splits: int = WGRAD_SPLITS) -> Tensor:
    """``g @ x^H`` (``g @ x.T`` for real tensors) for ``g`` (M, N) and ``x`` (K, N),
    with the reduction over N split.

    The partial products are summed in a fixed order, so the result is
    deterministic.  Tensors the kernel does not serve, or any with ``splits``
    given, take at most ``splits`` batched GEMMs, and one more for the last
    ``N % splits`` columns."""
    if g.dim() != 2 or x.dim() != 2 or g.shape[1] != x.shape[1]:
        raise ValueError(f"weight_grad needs (M, N) and (K, N), got {tuple(g.shape)} and "
                         f"{tuple(x.shape)}")
    g = g.contiguous()
    x = x.contiguous()
    if splits == WGRAD_SPLITS and g.dtype is x.dtype and _wgrad_serves(g, x):
        return outer_sum(g, x)
    m, n = g.shape
    k_rows = x.shape[0]
    s = min(int(splits), n // WGRAD_MIN_COLUMNS)
    if s < 2:
        return g @ (x.mH if x.is_complex() else x.T)
    cols = n // s
    main = s * cols
    # (s, M, cols) and (s, K, cols) views: split j covers columns [j*cols, (j+1)*cols).
    a = g.as_strided((s, m, cols), (cols, n, 1))
    b = x.as_strided((s, k_rows, cols), (cols, n, 1))
    out = torch.bmm(a, b.mH if x.is_complex() else b.transpose(1, 2)).sum(0)
    if main < n:
        tail = x[:, main:]
        out = out + g[:, main:] @ (tail.mH if x.is_complex() else tail.T)
    return out


# Weight layouts (RQF_PACK_* of include/rqf_scan.h).
FORWARD, ADJOINT, REAL, REAL_T, PAIRED, PAIRED_T = range(6)
# Largest weight side and most columns sent there (one launch grid holds them), and
# the multiplications, weight size times columns, from which two launches of these
# kernels beat the library's one: complex 48 x 48 weights, 5000 columns 13.0 against
# 11.7 us, 10304 13.1 against 15.8; real 520 x 512, 2500 columns 28 against 23 us,
# 10304 47 against 78.  A block walks the inner dimension in series (40 us at 1024), so from
# 512 on real products need as many times more of them: 1032 x 1024, 1288 columns 45
# against 32 us, 2576 56 against 53, 5152 72 against 108.
MAX_SIDE, MAX_COLS = 8192, (1 << 25) - 1
MIN_WORK = {torch.complex64: 1 << 24, torch.float32: 1 << 30}
REAL_INNER = 512
_PLAIN = (Tensor, torch.nn.Parameter)


def _kernel_serves(weight: Tensor, x: Tensor) -> bool:
    """Whether a product of these runs on the kernels: plain float32 or complex64
    matrices of one dtype on the current device, enough work, the data ``x``
    contiguous, and nothing recorded, traced or in forward mode (``unobserved``), batched
    (those tensors have no storage of their own) or autocast.  Everything else stays on
    torch."""
    dt = x.dtype
    if dt not in MIN_WORK or x.dim() != 2 or weight.dim() != 2:
        return False
    work = weight.numel() * x.shape[1]
    if work < MIN_WORK[dt] or (dt is torch.float32
                               and work * REAL_INNER < MIN_WORK[dt] * x.shape[0]):
        return False
    return (
        weight.dtype is dt and weight.numel() > 0 and 0 < x.shape[1] <= MAX_COLS
        and max(weight.shape) <= MAX_SIDE
        and type(x) in _PLAIN and type(weight) in _PLAIN
        and x.is_cuda and weight.is_cuda
        and x.get_device() == weight.get_device() == torch._C._cuda_getDevice()
        and torch._C._has_storage(x) and torch._C._has_storage(weight)
        and x.is_contiguous() and not x.is_conj() and not x.is_neg()
        and not (torch.is_grad_enabled() and (x.requires_grad or weight.requires_grad))
        and not torch.is_autocast_enabled("cuda")
        and unobserved()
    )


def matmul(weight: Tensor, x: Tensor) -> Tensor:
    """``weight @ x`` for a small ``weight`` (out, in) and an ``x`` (in, columns)."""
    if not _kernel_serves(weight, x) or weight.shape[1] != x.shape[0]:
        return weight @ x
    if x.is_complex():
        return gemm(FORWARD, weight, None, x, None)[0]
    return gemm(REAL, None, weight, None, x)[1]


def matmul_adjoint(weight: Tensor, g: Tensor) -> Tensor:
    """``weight.mH @ g`` (``weight.T @ g`` for real tensors)."""
    if not _kernel_serves(weight, g) or weight.shape[0] != g.shape[0]:
        return (weight.mH if weight.is_complex() else weight.T) @ g
    if g.is_complex():
        return gemm(ADJOINT, weight, None, g, None)[0]
    return gemm(REAL_T, None, weight, None, g)[1]


class _Projection(torch.autograd.Function):
    """``W @ h`` with the split weight gradient."""

    @staticmethod
    def forward(ctx, weight, h):
        ctx.save_for_backward(weight, h)
        with torch.autocast(h.device.type, enabled=False):
            return matmul(weight, h)

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, grad):
        weight, h = ctx.saved_tensors
        dw = dh = None
        with torch.autocast(h.device.type, enabled=False):
            if ctx.needs_input_grad[0]:
                dw = weight_grad(grad, h)
            if ctx.needs_input_grad[1]:
                dh = matmul_adjoint(weight, grad.contiguous())
        return dw, dh


def project(weight: Tensor, h: Tensor) -> Tensor:
    """``weight @ h`` for a 2-D ``h`` (in, batch*time), differentiable, with the
    split weight gradient.  Drop-in for the FBT stack's ``W_c @ h``
    (pure.py:222-223)."""
    return _Projection.apply(weight, h)


class _SplitProjection(torch.autograd.Function):
    """Mirror of the reference's ``_SplitProjection`` (selective.py:78-97):
    ``(weights @ v).split(sizes)``, with the split weight gradient."""

    @staticmethod
    def forward(ctx, v, weights, sizes):
        ctx.save_for_backward(v, weights)
        ctx.sizes = sizes
        ctx.set_materialize_grads(False)
        return matmul(weights, v).split(sizes)

    @staticmethod
    def backward(ctx, *grads):
        v, weights = ctx.saved_tensors
        grad = stacked([
            g if g is not None else v.new_zeros((n, v.shape[1]))
            for g, n in zip(grads, ctx.sizes)
            if n
        ])
        with torch.autocast(v.device.type, enabled=False):
            return matmul_adjoint(weights, grad), weight_grad(grad, v), None


def split_projection(v: Tensor, weights: Tensor, sizes) -> tuple[Tensor, ...]:
    """``(weights @ v).split(sizes)`` (selective.py:217), differentiable."""
    return _SplitProjection.apply(v, weights, tuple(sizes))


# ---------------------------------------------------------------------------
# Fused projections and the k-major weights of rqf_proj_gemm (csrc/proj.hip)
# ---------------------------------------------------------------------------

_PK, _PM = 16, 128  # what the k-major weights are padded to multiples of


def _padded(a: Tensor) -> Tensor:
    """(M, K) fp32 weight rows -> the kernel's (k_pad, m_pad) k-major layout."""
    m, k = a.shape
    out = torch.zeros((k + _PK - 1) // _PK * _PK, (m + _PM - 1) // _PM * _PM,
                      dtype=torch.float32, device=a.device)
    out[:k, :m] = a.T
    return out


def pack_forward(weight: Tensor, heads: Tensor | None) -> Tensor:
    """A of ``[z; logits] = A [x_0.re, x_0.im, x_1.re, ...]``: rows 2f, 2f+1 give
    Re z_f, Im z_f of ``z = weight @ x``; then one row per selector head row j,
    ``heads[j] @ [Re x; Im x]`` (selective.py:205-217)."""
    f, d = weight.shape
    wr, wi = weight.real.float(), weight.imag.float()
    ml = 0 if heads is None else heads.shape[0]
    a = torch.empty(2 * f + ml, 2 * d, dtype=torch.float32, device=weight.device)
    a[0:2 * f:2, 0::2], a[0:2 * f:2, 1::2] = wr, -wi
    a[1:2 * f:2, 0::2], a[1:2 * f:2, 1::2] = wi, wr
    if ml:
        a[2 * f:, 0::2], a[2 * f:, 1::2] = heads[:, :d].float(), heads[:, d:].float()
    return _padded(a)


def pack_dx(weight: Tensor, heads: Tensor | None) -> Tensor:
    """A of ``dx = A [dz_0.re, dz_0.im, ..., g_0, g_1, ...]``: rows 2d, 2d+1 give
    Re, Im of ``weight.mH @ dz + complex(dv[:D], dv[D:])`` with ``dv = heads.T @ g``
    (selective_scan.py:144, selective.py:96)."""
    f, d = weight.shape
    wr, wi = weight.real.float(), weight.imag.float()
    ml = 0 if heads is None else heads.shape[0]
    a = torch.empty(2 * d, 2 * f + ml, dtype=torch.float32, device=weight.device)
    a[0::2, 0:2 * f:2], a[0::2, 1:2 * f:2] = wr.T, wi.T
    a[1::2, 0:2 * f:2], a[1::2, 1:2 * f:2] = -wi.T, wr.T
    if ml:
        a[0::2, 2 * f:], a[1::2, 2 * f:] = heads[:, :d].T.float(), heads[:, d:].T.float()
    return _padded(a)


def gemm(mode: int, weight: Tensor | None, heads: Tensor | None, b_cplx: Tensor | None,
         b_real: Tensor | None, bias: Tensor | None = None, relu: bool = False):
    """``(complex rows, real rows)`` of the product the layout ``mode`` stands for
    (``rqf_projection``): ``weight`` complex (w_rows, w_cols), ``heads`` real,
    ``b_cplx`` (complex64) and ``b_real`` (float32) contiguous (rows, n)."""
    from prospective_rqf_amd import _lib

    b = b_real if b_cplx is None else b_cplx
    n, device = b.shape[1], b.device
    w, h = weight, heads
    if w is not None and not (w.dtype is torch.complex64 and w.is_contiguous()
                              and not w.is_conj() and not w.is_neg()):
        w = w.to(torch.complex64).resolve_conj().resolve_neg().contiguous()
    if h is not None and not (h.dtype is torch.float32 and h.is_contiguous()
                              and not h.is_neg()):
        h = h.float().resolve_neg().contiguous()
    h_rows = 0 if h is None else h.shape[0]
    if w is not None:
        w_rows, w_cols = w.shape
    else:
        w_rows, w_cols = 0, h.shape[1] // 2 if mode <= ADJOINT else h.shape[1]
    cplx = (w_rows, w_cols, 0, 0, h_rows // 2, 0)[mode]
    real = (h_rows, 0, h_rows, w_cols, 0, w_cols)[mode]
    out_c = torch.empty(cplx, n, dtype=torch.complex64, device=device) if cplx else None
    out_r = torch.empty(real, n, dtype=torch.float32, device=device) if real else None
    lib = _lib.load()
    nbytes = lib.rqf_projection_workspace(mode, w_rows, w_cols, h_rows, n)
    ws = _lib.workspace(nbytes, device)
    _lib.check(lib.rqf_projection(
        mode, _lib.ptr(w), w_rows, w_cols, _lib.ptr(h), h_rows, _lib.ptr(b_cplx),
        _lib.ptr(b_real), n, _lib.ptr(out_c), _lib.ptr(out_r), _lib.ptr(bias), int(relu),
        _lib.ptr(ws), nbytes, _lib.stream_of(b)), "rqf_projection")
    return out_c, out_r


def _proj_gemm(packed: Tensor, b_cplx: Tensor | None, b_real: Tensor | None, n: int,
               out_cplx_rows: int, out_real_rows: int, device, bias: Tensor | None = None,
               relu: bool = False):
    """The product with weights in the k-major fp32 layout (``pack_forward``, ``pack_dx``)."""
    from prospective_rqf_amd import _lib

    lib = _lib.load()
    out_c = (torch.empty(out_cplx_rows, n, dtype=torch.complex64, device=device)
             if out_cplx_rows else None)
    out_r = (torch.empty(out_real_rows, n, dtype=torch.float32, device=device)
             if out_real_rows else None)
    a = _lib.ProjGemmArgs()
    a.weights, a.k_pad, a.m_pad = packed.data_ptr(), packed.shape[0], packed.shape[1]
    a.b_cplx = 0 if b_cplx is None else b_cplx.data_ptr()
    a.b_cplx_rows = 0 if b_cplx is None else b_cplx.shape[0]
    a.b_real = 0 if b_real is None else b_real.data_ptr()
    a.b_real_rows = 0 if b_real is None else b_real.shape[0]
    a.n = n
    a.out_cplx = 0 if out_c is None else out_c.data_ptr()
    a.out_cplx_rows = out_cplx_rows
    a.out_real = 0 if out_r is None else out_r.data_ptr()
    a.out_real_rows = out_real_rows
    a.out_real_bias = 0 if bias is None else bias.data_ptr()
    a.out_real_relu = int(bool(relu))
    _lib.check(lib.rqf_proj_gemm(ctypes.byref(a), _lib.stream_of(packed)), "rqf_proj_gemm")
    return out_c, out_r


def stacked(blocks: list) -> Tensor | None:
    """The row blocks as one (rows, N) tensor: their common storage when they are
    consecutive row ranges of one contiguous buffer (as ``selective_backward``
    allocates the logit gradients), else a concatenation."""
    blocks = [b for b in blocks if b is not None and b.shape[0]]
    if not blocks:
        return None
    flat = [b.reshape(b.shape[0], -1) if b.dim() != 2 else b for b in blocks]
    base = flat[0]
    storage = base.untyped_storage()
    same = all(b.is_contiguous() and b.dtype == base.dtype and b.shape[1] == base.shape[1]
               and b.untyped_storage().data_ptr() == storage.data_ptr() for b in flat)
    if same and all(flat[i + 1].data_ptr() == flat[i].data_ptr() + flat[i].numel() * flat[i].element_size()
                    for i in range(len(flat) - 1)):
        rows = sum(b.shape[0] for b in flat)
        return base.as_strided((rows, base.shape[1]), (base.shape[1], 1))
    return torch.cat(flat, 0)


def fused_forward(x: Tensor, weight: Tensor, heads: Tensor | None = None,
                  packed: Tensor | None = None):
    """``z = weight @ x`` (complex64, (F, N)) and ``heads @ [Re x; Im x]`` (fp32,
    (rows, N), or None) from one pass over ``x`` (D, N) complex64."""
    from prospective_rqf_amd import _lib

    _lib.require_device(x, weight, heads)
    if x.dtype != torch.complex64 or weight.dtype != torch.complex64:
        raise TypeError("fused_forward takes complex64 x and weight")
    x = x.resolve_conj().contiguous()
    ml = 0 if heads is None else heads.shape[0]
    if packed is None:
        return gemm(FORWARD, weight, heads, x, None)
    return _proj_gemm(packed, x, None, x.shape[1], weight.shape[0], ml, x.device)


def fused_dx(dz: Tensor, grads: list, weight: Tensor, heads: Tensor | None = None,
             packed: Tensor | None = None) -> Tensor:
    """``weight.mH @ dz + complex(dv[:D], dv[D:])``, ``dv = heads.T @ g`` with ``g``
    the fp32 row blocks ``grads`` stacked (rows summing to ``heads.shape[0]``), in
    one pass over ``dz`` (F, N) complex64 and ``g``.  Blocks that are consecutive
    row ranges of one buffer are read in place."""
    from prospective_rqf_amd import _lib

    _lib.require_device(dz, weight, heads, *grads)
    dz = dz.resolve_conj().contiguous()
    g = stacked([b.float() for b in grads])
    rows = 0 if g is None else g.shape[0]
    if heads is None and rows:
        raise ValueError("logit gradients given without selector heads")
    if heads is not None and rows != heads.shape[0]:
        raise ValueError("logit gradient rows must match the selector heads")
    if packed is None:
        return gemm(ADJOINT, weight, heads, dz, g)[0]
    out, _ = _proj_gemm(packed, dz, g, dz.shape[1], weight.shape[1], 0, dz.device)
    return out
