"""GPU parity of the (B,T,F) scans whose sequences run in chunks.

Few sequences of at least four passes are cut into chunks of whole passes, run from
the end states of the chunks before them (after them, for an adjoint).  Sizes: four
passes exactly and one step more or less, chunks of one pass and of several with a
shorter last one, a last pass of one step, filters past the 16 of a block.  The bars are
those of the other parity tests, against the fp64 oracle.
"""

import numpy as np
import pytest
import torch

from oracle import oracle
from prospective_rqf_amd import _lib
from prospective_rqf_amd.chunked_scan_kernel import (
    _chunked_prospective_forward_raw,
    _triton_chunked_scan,
    _triton_chunked_scan_prospective,
)
from prospective_rqf_amd.multi_osc_scan import (
    _forward,
    _triton_sequential_scan_multi_osc,
    _triton_sequential_scan_multi_osc_real,
)
from prospective_rqf_amd.scan import sequential_scan_abs
from tests.helpers import PARITY_RTOL, chanerr, crandn, relerr
from tests.test_gpu_multi_osc import (
    test_gradient_subsets_launch_their_own_variants as _subsets_case,
)
from tests.test_gpu_multi_osc import test_multi_osc_forward_backward as _multi_osc_case
from tests.test_gpu_timeinv import _c64, _coeffs, _dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


@pytest.mark.parametrize("prospective", [True, False])
@pytest.mark.parametrize("B,T,F", [(1, 2048, 3), (1, 1537, 16), (1, 3073, 17), (2, 4095, 5),
                                   (1, 4096, 40), (3, 4097, 16), (2, 16000, 33), (40, 5121, 40)])
def test_chunked_scans(B, T, F, prospective):
    print(f"case: time split {B} {T} {F} {prospective}", flush=True)
    rng = np.random.default_rng(B + T + F)
    c1, t0, t1 = _coeffs(rng, F)
    u, gy = _c64(crandn(rng, B, T, F)), _c64(crandn(rng, B, T, F))
    t1 = t1 if prospective else None
    y_ref = oracle.twotap_fwd(c1, t0, t1, u)
    gu_ref, gc1_ref, g0_ref, g1_ref = oracle.twotap_bwd(c1, t0, t1, u, y_ref, gy)
    C1, T0, U = _dev(c1), _dev(t0), _dev(u)
    T1 = _dev(t1) if prospective else None
    y = (_triton_chunked_scan_prospective(C1, T0, T1, U) if prospective
         else _triton_chunked_scan(C1, T0, U))
    y.backward(torch.as_tensor(gy.astype(np.complex64), device="cuda"))
    assert relerr(y, y_ref) <= PARITY_RTOL
    assert relerr(U.grad, gu_ref) <= PARITY_RTOL
    for got, want in ((C1, gc1_ref), (T0, g0_ref), (T1, g1_ref)):
        if got is not None:
            assert relerr(got.grad, want) <= PARITY_RTOL
            assert chanerr(got.grad, want) <= PARITY_RTOL


def test_forward_without_workspace_runs_whole_sequences():
    g = torch.Generator().manual_seed(1)
    B, T, F = 1, 5000, 20
    c = [torch.randn(F, dtype=torch.complex64, generator=g).cuda() * 0.5 for _ in range(3)]
    x = torch.randn(B, T, F, dtype=torch.complex64, generator=g).cuda()
    want = _chunked_prospective_forward_raw(*c, x)
    out = torch.empty_like(x)
    _lib.check(_lib.load().rqf_chunked_prospective_fwd(
        *(t.data_ptr() for t in c), x.data_ptr(), out.data_ptr(), B, T, F, None, 0,
        _lib.stream_of(x)), "rqf_chunked_prospective_fwd")
    assert relerr(out, want) <= 1e-6


@pytest.mark.parametrize("real", [False, True])
@pytest.mark.parametrize("N", [1, 2, 4, 5, 9])
@pytest.mark.parametrize("B,T,F", [(1, 2561, 3), (1, 4097, 17), (2, 8193, 5), (33, 2100, 80)])
def test_multi_osc(B, T, F, N, real):
    """Oscillators in launches of up to four share the backward's chunks; the last shape
    runs whole sequences of several passes."""
    _multi_osc_case((B, T, F), N, real)


@pytest.mark.parametrize("real", [False, True])
def test_abs_readout(real):
    rng = np.random.default_rng(3)
    B, T, F = 2, 9001, 21
    c1, c2, _ = _coeffs(rng, F)
    u = _c64(crandn(rng, B, T, F))
    u = u.real.astype(np.float32).astype(np.float64) if real else u
    y = oracle.twotap_fwd(c1, c2, None, u.astype(np.complex128))
    U = torch.as_tensor(u.astype(np.float32 if real else np.complex64), device="cuda")
    with torch.no_grad():
        C1, C2 = _dev(c1).detach(), _dev(c2).detach()
        got = sequential_scan_abs(C1, C2, U)
        raw = _forward(C1, C2, U, None, 1, real=real, absolute=False)
    assert relerr(got, np.abs(y)) <= PARITY_RTOL
    assert relerr(raw, y) <= PARITY_RTOL


@pytest.mark.parametrize("real", [False, True])
@pytest.mark.parametrize("N", [1, 2, 4])
def test_multi_osc_gradient_subsets(N, real):
    _subsets_case((1, 2600, 18), N, real)


# 64 sequences in chunks of eight passes (4096 steps): 1.25^4096 is past float64
UNSTABLE = (64, 16000, 16)


def _unstable(F):
    return (1.25 * np.exp(0.3j * np.arange(F))).astype(np.complex64).astype(np.complex128)


@pytest.mark.parametrize("prospective", [True, False])
def test_unstable_filters_stay_finite_while_their_state_is_zero(prospective):
    """Silence, then 50 steps: what whole sequences gave, from those steps alone."""
    rng = np.random.default_rng(5)
    (B, T, F), n = UNSTABLE, 50
    _, t0, t1 = _coeffs(rng, F)
    c1, t1 = _unstable(F), t1 if prospective else None
    u, gy = _c64(crandn(rng, B, n, F)), _c64(crandn(rng, B, n, F))
    leaves = [_dev(c) for c in (c1, t0) + ((t1,) if prospective else ())]
    scan = _triton_chunked_scan_prospective if prospective else _triton_chunked_scan
    x = torch.zeros(B, T, F, dtype=torch.complex64, device="cuda")
    x[:, T - n:] = torch.as_tensor(u.astype(np.complex64))
    with torch.no_grad():
        y = scan(*leaves, x)
    assert not y[:, :T - n].any()
    assert relerr(y[:, T - n:], oracle.twotap_fwd(c1, t0, t1, u)) <= PARITY_RTOL
    # the adjoint runs the other way: a cotangent of the first steps only
    x = x.flip(1).contiguous().requires_grad_(True)
    g = torch.zeros(B, T, F, dtype=torch.complex64, device="cuda")
    g[:, :n] = torch.as_tensor(gy.astype(np.complex64))
    scan(*leaves, x).backward(g)
    u = u[:, ::-1]
    gu, *gc = oracle.twotap_bwd(c1, t0, t1, u, oracle.twotap_fwd(c1, t0, t1, u), gy)
    assert not x.grad[:, n:].any()
    assert relerr(x.grad[:, :n], gu) <= PARITY_RTOL
    for got, want in zip(leaves, gc):
        assert relerr(got.grad, want) <= PARITY_RTOL


@pytest.mark.parametrize("real", [False, True])
@pytest.mark.parametrize("N", [1, 2, 4])
def test_unstable_oscillators_stay_finite_while_their_state_is_zero(N, real):
    """Each layout's whole-sequence result from the same steps (50 of them run whole)."""
    rng = np.random.default_rng(6)
    (B, T, F), n = UNSTABLE, 50
    scan = _triton_sequential_scan_multi_osc_real if real else _triton_sequential_scan_multi_osc
    c1 = _unstable(F * N)
    c2, cw = _c64(crandn(rng, F * N)), torch.randn(F * N, 2, device="cuda")
    u = torch.randn(B, n, F, dtype=torch.float32 if real else torch.complex64, device="cuda")
    g = torch.randn(B, n, F, dtype=torch.complex64, device="cuda")

    def run(x, gy):
        leaves = [_dev(c1), _dev(c2), x.requires_grad_(True), cw.clone().requires_grad_(True)]
        y = scan(*leaves, N)
        return y.detach(), torch.autograd.grad(y, leaves, gy)

    def padded(v, front):
        out = torch.zeros(B, T, F, dtype=v.dtype, device="cuda")
        (out[:, T - n:] if front else out[:, :n]).copy_(v)
        return out

    y, want = run(u.clone(), g)
    late, _ = run(padded(u, True), padded(g, False))
    assert not late[:, :T - n].any() and relerr(late[:, T - n:], y) <= PARITY_RTOL
    _, got = run(padded(u, False), padded(g, False))
    assert not got[2][:, n:].any()
    for a, b in zip((got[0], got[1], got[2][:, :n], got[3]), want):
        assert relerr(a, b) <= PARITY_RTOL
