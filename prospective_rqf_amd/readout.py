"""Per-timestep ``[Re; Im]`` MLP readout on complex features.

Mirrors the head of the reference's ``ComplexReadoutClassifier``
(train.py:74-136).  Per time step the logits are
``W2 relu(W1 [Re f; Im f] + b1) + b2``, or ``W1 [Re f; Im f] + b1`` with no
hidden layer, and they are mean-pooled over time outside training.

It runs on the channel-outermost (F, B*T) features the FBT stack produces
(pure.py:510-536).  The reference first permutes them back to (B, T, F)
(pure.py:536) and concatenates real and imaginary parts (train.py:130); here
the first layer is one MFMA GEMM (``rqf_projection``) that reads the
interleaved complex features in place, with the bias and the ReLU fused into
its stores.  Dropout is the identity, as in evaluation; training with dropout
keeps the reference's module.
"""

from __future__ import annotations

import torch
from torch import Tensor

from prospective_rqf_amd.projection import (
    ADJOINT,
    FORWARD,
    _PLAIN,
    gemm,
    real_weight_grad,
    unobserved,
    weight_grad,
)


# Most classes that rqf_readout_grads takes.
_MAX_CLASSES = 64


def _head_grads(dlogits: Tensor, hidden: Tensor, w2: Tensor):
    """``(dh, dw2, db1, db2)`` of ``logits = w2 relu(h) + b2`` from ``hidden = relu(h)``:
    one pass over ``hidden`` where the kernel serves, torch elsewhere."""
    from prospective_rqf_amd import _lib

    w2 = w2.float().contiguous()
    (c, n), rows = dlogits.shape, w2.shape[1]
    if not (0 < c <= _MAX_CLASSES and 0 < rows <= 1 << 20 and n > 0
            and hidden.shape == (rows, n) and hidden.dtype is torch.float32
            and unobserved()
            and all(type(t) in _PLAIN and t.is_cuda and t.is_contiguous() and not t.is_neg()
                    and t.get_device() == torch._C._cuda_getDevice()
                    and torch._C._has_storage(t) for t in (dlogits, hidden, w2))):
        dh = (w2.T @ dlogits).mul_(hidden > 0)
        return dh, weight_grad(dlogits, hidden), dh.sum(1), dlogits.sum(1)
    dh = torch.empty_like(hidden)
    dw2 = torch.empty_like(w2)
    db1, db2 = hidden.new_empty(rows), hidden.new_empty(c)
    lib = _lib.load()
    nbytes = lib.rqf_readout_grads_workspace(c, rows, n)
    ws = _lib.workspace(nbytes, hidden.device)
    _lib.check(lib.rqf_readout_grads(
        dlogits.data_ptr(), hidden.data_ptr(), w2.data_ptr(), c, rows, n, dh.data_ptr(),
        dw2.data_ptr(), db1.data_ptr(), db2.data_ptr(), _lib.ptr(ws), nbytes,
        _lib.stream_of(hidden)), "rqf_readout_grads")
    return dh, dw2, db1, db2


class _ComplexReadout(torch.autograd.Function):
    @staticmethod
    def forward(ctx, feats, w1, b1, w2, b2):
        relu = w2 is not None
        _, out = gemm(FORWARD, None, w1, feats, None, bias=b1.float().contiguous(),
                      relu=relu)
        if relu:
            logits = torch.addmm(b2.float()[:, None], w2.float(), out)
        else:
            logits = out
        ctx.save_for_backward(feats, w1, w2, out if relu else None)
        return logits

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, dlogits):
        feats, w1, w2, hidden = ctx.saved_tensors
        dlogits = dlogits.float().contiguous()
        dw2 = db2 = None
        if w2 is not None:
            dh, dw2, db1, db2 = _head_grads(dlogits, hidden, w2)
        else:
            dh, db1 = dlogits, dlogits.sum(1)
        dw1 = real_weight_grad(dh, feats)
        dfeats = None
        if ctx.needs_input_grad[0]:
            dfeats, _ = gemm(ADJOINT, None, w1, None, dh)
        return dfeats, dw1, db1, dw2, db2


def complex_readout(feats: Tensor, w1: Tensor, b1: Tensor, w2: Tensor | None = None,
                    b2: Tensor | None = None, pool: bool = True) -> Tensor:
    """Logits of the per-timestep readout on FBT-layout features.

    ``feats``: (F, B, T) complex64, channel outermost.  ``w1`` (H, 2F), ``b1`` (H)
    and, with a hidden layer, ``w2`` (C, H), ``b2`` (C), as ``nn.Linear`` stores
    them.  Returns (B, C) mean-pooled logits, or (B, T, C) with ``pool=False``
    (the per-step-loss training contract, train.py:131-134).
    """
    from prospective_rqf_amd import _lib

    _lib.require_device(feats, w1, b1, w2, b2)
    if feats.dtype != torch.complex64:
        raise TypeError("complex_readout takes complex64 features")
    if (w2 is None) != (b2 is None):
        raise ValueError("w2 and b2 go together")
    f, b, t = feats.shape
    if w1.shape[1] != 2 * f:
        raise ValueError(f"w1 has {w1.shape[1]} inputs for {f} complex features")
    logits = _ComplexReadout.apply(feats.resolve_conj().contiguous().reshape(f, b * t), w1, b1,
                                   w2, b2)
    logits = logits.reshape(-1, b, t)
    return logits.mean(-1).T if pool else logits.permute(1, 2, 0)
