"""GPU parity of the split-bf16 products (csrc/proj.hip) at the edges of their tiles.

A product of float32 values carries everything down to 2^-24 of it, and the sums are
float32, so a result's 2-norm error is that of a float32 sum of its length: each of
its at most K / 16 + 1 additions rounds by at most 2^-24 of a partial sum, which
gives a 2-norm error below 2^-24 sqrt(K / 16 + 1) for products of random sign.  The
bar is four times that, against float64 on the same inputs.
"""

import ctypes
import math

import pytest
import torch
from torch.autograd import forward_ad
from torch.fx.experimental.proxy_tensor import make_fx

from prospective_rqf_amd import _lib
from prospective_rqf_amd import projection as P

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def _bar(k):
    return 4 * 2.0 ** -24 * math.sqrt(k / 16 + 1)


def _err(got, want):
    d = (got.to(want.dtype) - want).abs()
    return float(torch.linalg.vector_norm(d) / torch.linalg.vector_norm(want))


def _rand(g, *shape, cplx=False):
    if cplx:
        return torch.view_as_complex(torch.randn(*shape, 2, generator=g, device="cuda"))
    return torch.randn(*shape, generator=g, device="cuda")


def _gen(*key):
    return torch.Generator(device="cuda").manual_seed(sum(key))


# out rows, in rows, columns: one of each, below and past a 16- and a 32-row block, half
# and all of a 32-k stage, 16 of a wavefront's columns and a 128-column tile, every tile
# height, odd columns.
SHAPES = [(1, 1, 1), (1, 9, 31), (15, 8, 127), (17, 7, 129), (33, 12, 257), (48, 48, 1001),
          (65, 33, 130), (97, 20, 4099), (130, 5, 70001), (145, 64, 66000), (260, 256, 66001),
          (8, 16, 16), (9, 15, 17), (20, 8, 113), (31, 24, 145), (130, 17, 3001)]


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_products_and_adjoints(m, k, n, monkeypatch):
    print(f"case: products {m} {k} {n}", flush=True)
    monkeypatch.setattr(P, "MIN_WORK", dict.fromkeys(P.MIN_WORK, 0))
    g = _gen(m, k, n)
    for cplx in (True, False):
        w, x, y = (_rand(g, *s, cplx=cplx) for s in ((m, k), (k, n), (m, n)))
        wide = torch.complex128 if cplx else torch.float64
        assert _err(P.matmul(w, x), w.to(wide) @ x.to(wide)) <= _bar(2 * k)
        assert _err(P.matmul_adjoint(w, y), w.to(wide).mH @ y.to(wide)) <= _bar(2 * m)
    s = _rand(g, 2 * m, k)  # stacked [Wr; Wi]
    x, z = _rand(g, k, n), _rand(g, m, n, cplx=True)
    got = P.gemm(P.PAIRED, None, s, None, x)[0]
    want = s.double() @ x.double()
    assert _err(got, torch.complex(want[:m], want[m:])) <= _bar(k)
    got = P.gemm(P.PAIRED_T, None, s, z, None)[1]
    z64 = z.to(torch.complex128)
    assert _err(got, s.double().T @ torch.cat((z64.real, z64.imag))) <= _bar(2 * m)


@pytest.mark.parametrize("f,d,ml,n", [(5, 7, 3, 130), (24, 8, 17, 513), (9, 40, 1, 20001)])
def test_stacked_heads_and_caller_packed_weights(f, d, ml, n):
    """Complex rows that end inside a 16-k stage, with real rows behind them; the fp32
    layout a caller may keep (``packed``) gives the same product."""
    print(f"case: stacked {f} {d} {ml} {n}", flush=True)
    g = _gen(f, d, ml, n)
    w, h = _rand(g, f, d, cplx=True), _rand(g, ml, 2 * d)
    x, dz, gl = _rand(g, d, n, cplx=True), _rand(g, f, n, cplx=True), _rand(g, ml, n)
    w64, x64, dz64 = (t.to(torch.complex128) for t in (w, x, dz))
    dv = h.double().T @ gl.double()
    for packed in (False, True):
        z, logits = P.fused_forward(x, w, h, P.pack_forward(w, h) if packed else None)
        assert _err(z, w64 @ x64) <= _bar(2 * d)
        assert _err(logits, h.double() @ torch.cat((x64.real, x64.imag))) <= _bar(2 * d)
        dx = P.fused_dx(dz, [gl], w, h, P.pack_dx(w, h) if packed else None)
        assert _err(dx, w64.mH @ dz64 + torch.complex(dv[:d], dv[d:])) <= _bar(2 * f + ml)


@pytest.mark.parametrize("cplx", [True, False])
def test_values_that_are_not_sums_of_three_parts(cplx, monkeypatch):
    """Infinities, NaN, values near the largest float and a whole tile of values near
    the smallest normal one."""
    monkeypatch.setattr(P, "MIN_WORK", dict.fromkeys(P.MIN_WORK, 0))
    g = _gen(11, cplx)
    w, x = _rand(g, 40, 24, cplx=cplx), _rand(g, 24, 300, cplx=cplx)
    wide = torch.complex128 if cplx else torch.float64
    big = x.clone()
    (torch.view_as_real(big) if cplx else big)[3, 7] = 3.0e38
    got = P.matmul(w * 1e-3, big)
    assert _err(got * 1e-30, ((w * 1e-3).to(wide) @ big.to(wide)) * 1e-30) <= _bar(48)
    tiny = x * 1.0e-37  # every product of the sums below is a float32 one or zero
    got = P.matmul(w, tiny)
    assert _err(got.to(wide) * 1e37, (w.to(wide) @ tiny.to(wide)) * 1e37) <= 1e-6
    for bad in (math.inf, -math.inf, math.nan):
        y = x.clone()
        (torch.view_as_real(y) if cplx else y)[5, 130] = bad
        got, want = P.matmul(w, y), P.matmul(w, x)
        keep = torch.arange(300, device="cuda") != 130
        col = got[:, 130]
        col = torch.view_as_real(col) if cplx else col
        if cplx:  # both parts are: inf - inf or inf + inf
            assert not torch.isfinite(col).any()
        else:
            assert torch.equal(col.nan_to_num(7.0), (w[:, 5] * bad).nan_to_num(7.0))
        assert _err(got[:, keep], want[:, keep].to(wide)) <= _bar(48)
    w[2, 3] = math.inf
    got = P.matmul(w, x)
    assert not torch.isfinite(torch.view_as_real(got[2]) if cplx else got[2]).any()
    rows = torch.arange(40, device="cuda") != 2
    assert _err(got[rows], w.to(wide)[rows] @ x.to(wide)) <= _bar(48)


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("exponent", [-100, -112, -116, -120, -125])
def test_small_weights_keep_every_bit(exponent, packed):
    """Weights whose last bits lie below bf16's smallest values, at the usual bar."""
    g = _gen(64, 50, 3000)
    w = torch.randn(50, 64, 2, generator=g, device="cuda").clamp_(-2, 2)
    w = torch.view_as_complex((w + w.sign()) * 2.0 ** exponent)  # all normal
    x = _rand(g, 64, 3000, cplx=True)
    z, _ = P.fused_forward(x, w, None, P.pack_forward(w, None) if packed else None)
    up = 2.0 ** -exponent
    assert _err(z.to(torch.complex128) * up, (w.to(torch.complex128) * up) @ x.to(torch.complex128)
                ) <= _bar(128)


@pytest.mark.parametrize("m,k,n,kernel", [(1024, 1024, 1024, False), (1024, 1024, 2047, False),
                                          (1024, 1024, 2048, True), (512, 512, 4095, False),
                                          (512, 512, 4096, True), (256, 256, 16384, True)])
def test_long_inner_dimensions_need_more_columns(m, k, n, kernel, monkeypatch):
    taken = []
    gemm = P.gemm
    monkeypatch.setattr(P, "gemm", lambda *a, **kw: taken.append(a[0]) or gemm(*a, **kw))
    g = _gen(m, k, n)
    w, x, y = _rand(g, m, k), _rand(g, k, n), _rand(g, m, n)
    got = P.matmul(w, x), P.matmul_adjoint(w, y)
    assert taken == ([P.REAL, P.REAL_T] if kernel else [])
    for a, want in zip(got, (w.double() @ x.double(), w.double().T @ y.double())):
        assert _err(a, want) <= 4 * 2.0 ** -24 * math.sqrt(k)


def test_everything_else_stays_on_torch(monkeypatch):
    """Forms the kernels do not serve: dtypes, strides, lazy conjugates, graphs of graphs,
    autocast, empty sizes, vectors."""
    monkeypatch.setattr(P, "MIN_WORK", dict.fromkeys(P.MIN_WORK, 0))
    g = _gen(12)
    w, x = _rand(g, 6, 5), _rand(g, 5, 40)
    wc, xc = _rand(g, 6, 5, cplx=True), _rand(g, 5, 40, cplx=True)
    for a, b in [(w.double(), x.double()), (w, x.T.contiguous().T), (wc, xc.conj()),
                 (w, x[:, :0]), (w[:0], x), (w, x[:, 0]), (w.half(), x.half())]:
        assert torch.equal(P.matmul(a, b), a @ b)
    assert torch.allclose(P.matmul(wc.conj(), xc), wc.conj() @ xc, rtol=0, atol=1e-5)
    a, b = w.clone().requires_grad_(), x.clone().requires_grad_()
    (y,) = P.split_projection(b, a, (6,))
    (ga,) = torch.autograd.grad(y.square().sum(), a, create_graph=True)
    (gg,) = torch.autograd.grad(ga.sum(), b)
    r, c = a.detach().clone().requires_grad_(), b.detach().clone().requires_grad_()
    (gr,) = torch.autograd.grad((r @ c).square().sum(), r, create_graph=True)
    (gw,) = torch.autograd.grad(gr.sum(), c)
    assert torch.allclose(ga, gr, rtol=1e-4, atol=1e-4) and torch.allclose(gg, gw, rtol=1e-4,
                                                                         atol=1e-4)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert P.split_projection(x, w, (6,))[0].dtype == (w @ x).dtype


# rows, rows, columns: a single product, below and past the 64- and 128-row tiles, a
# last stage of 1 to 31 columns, several splits with a ragged last one, both tile sizes on
# either side of 512 blocks.
SUMS = [(1, 1, 1), (3, 33, 31), (16, 16, 2049), (31, 40, 4097), (65, 64, 5003), (48, 48, 60001),
        (130, 20, 10304), (200, 129, 9000), (16, 16, 65535), (16, 16, 65536), (256, 256, 16383),
        (256, 256, 16384)]


@pytest.mark.parametrize("m,k,n", SUMS)
@pytest.mark.parametrize("ac,bc", [(True, True), (False, False), (False, True), (True, False)])
def test_weight_gradients(m, k, n, ac, bc):
    print(f"case: weight gradient {m} {k} {n} {ac} {bc}", flush=True)
    g = _gen(m, k, n, ac, bc)
    a, b = _rand(g, m, n, cplx=ac), _rand(g, k, n, cplx=bc)
    got = P.outer_sum(a, b)
    if ac and bc:
        want = a.to(torch.complex128) @ b.to(torch.complex128).mH
    else:
        want = torch.cat((a.real, a.imag)).double() if ac else a.double()
        want = want @ (torch.cat((b.real, b.imag)) if bc else b).double().T
    assert _err(got, want) <= _bar(2 * min(n, 2048))
    assert torch.equal(got, P.outer_sum(a, b))  # fixed order
    tiny = P.outer_sum(a * 2.0 ** -123, b)  # near the smallest normal float
    assert _err(tiny.to(want.dtype) * 2.0 ** 123, want) <= 1e-5


def test_weight_gradient_of_infinities():
    g = _gen(13)
    a, b = _rand(g, 70, 5000), _rand(g, 90, 5000)
    want = a.double() @ b.double().T
    a[66, 4999] = math.inf
    got = P.weight_grad(a, b)
    assert torch.equal(got[66], b[:, 4999] * math.inf)
    rows = torch.arange(70, device="cuda") != 66
    assert _err(got[rows], want[rows]) <= _bar(2048)


def test_batched_gradients_stay_on_torch():
    """Batched tensors have no storage; columns enough for the kernels otherwise."""
    g = _gen(7)
    w, h = _rand(g, 20, 18, cplx=True), _rand(g, 18, 50000, cplx=True)
    v = _rand(g, 2, 20, 50000, cplx=True)
    for leaf, want in ((0, torch.stack([a @ h.mH for a in v])),
                       (1, torch.stack([w.mH @ a for a in v]))):
        leaves = [w.clone(), h.clone()]
        leaves[leaf].requires_grad_(True)
        y = P.project(*leaves)
        got, = torch.autograd.grad(y, leaves[leaf], v, is_grads_batched=True)
        assert _err(got, want) <= 2 * _bar(50000)


def test_columns_past_a_descriptor():
    """More columns than a half stage's descriptor holds take 64-bit addresses."""
    n = P.MAX_COLS + 2
    x = torch.ones(1, n, device="cuda")
    x[0, 3], x[0, n - 1] = 2.5, -7.0
    y = P.gemm(P.REAL, None, torch.tensor([[3.0]], device="cuda"), None, x)[1]
    assert torch.equal(y, 3 * x)


def test_packed_columns_past_a_descriptor():
    n = P.MAX_COLS + 2
    x = torch.ones(1, n, device="cuda")
    x[0, 3], x[0, n - 1] = 2.5, -7.0
    packed = P._padded(torch.tensor([[3.0]], device="cuda"))
    assert torch.equal(P._proj_gemm(packed, None, x, n, 0, 1, x.device)[1], 3 * x)


def test_weight_gradient_of_complex_rows_against_real_ones():
    g = _gen(11)
    a, b = _rand(g, 64, 4100, cplx=True), _rand(g, 128, 4100)
    got = P.outer_sum(a, b)
    want = torch.cat((a.real, a.imag)).double() @ b.double().T
    assert _err(got, want) <= _bar(4100)


@pytest.mark.parametrize("relu", [0, 1])
@pytest.mark.parametrize("k_pad", [0, 16])
def test_packed_product_over_nothing_is_the_bias(k_pad, relu):
    weights = torch.ones(16, 128, device="cuda")
    bias = torch.tensor([1.5, -2.0, 0.5], device="cuda")
    z = torch.ones(2, 130, dtype=torch.complex64, device="cuda")
    out = torch.ones(3, 130, device="cuda")
    a = _lib.ProjGemmArgs()
    a.weights, a.k_pad, a.m_pad, a.n = weights.data_ptr(), k_pad, 128, 130
    a.out_cplx, a.out_cplx_rows = z.data_ptr(), 2
    a.out_real, a.out_real_rows = out.data_ptr(), 3
    a.out_real_bias, a.out_real_relu = bias.data_ptr(), relu
    _lib.check(_lib.load().rqf_proj_gemm(ctypes.byref(a), _lib.stream_of(out)), "rqf_proj_gemm")
    assert not z.any()
    assert torch.equal(out, (bias.relu() if relu else bias)[:, None].expand(3, 130))


# both sides of the narrow operand's limits, no column and one
@pytest.mark.parametrize("f,d,n", [(64, 3, 1 << 18), (64, 3, (1 << 18) - 1), (64, 7, 1 << 18),
                                   (64, 8, 1 << 18), (5, 3, 1), (5, 4, 300), (5, 3, 0)])
def test_narrow_layer0_weight_gradient_copies_no_gradient(f, d, n):
    g = _gen(f, d, n)
    gz, h = _rand(g, f, n, cplx=True), _rand(g, d, n)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    got = P.real_weight_grad(gz, h)
    used = torch.cuda.max_memory_allocated() - before
    if n > 1000:
        assert used < gz.numel() * 8
    want = torch.cat((gz.real, gz.imag)).double() @ h.double().T
    assert got.shape == (2 * f, d) and got.dtype is torch.float32
    assert _err(got, want) <= _bar(2 * min(n, 4096)) if n else not got.any()


@pytest.mark.parametrize("ac,bc,m,k", [(False, False, 1100, 1030), (True, False, 550, 1030),
                                       (False, True, 1100, 515), (True, True, 550, 515)])
def test_weight_gradients_in_several_passes(ac, bc, m, k):
    """74 splits of 5.3 MB run in two passes; an infinity in the second stays its own."""
    n = 150001
    print(f"case: weight gradient in passes {m} {k} {n} {ac} {bc}", flush=True)
    g = _gen(m, k, ac, bc)
    a, b = _rand(g, m, n, cplx=ac), _rand(g, k, n, cplx=bc)
    got = P.outer_sum(a, b)
    if ac and bc:
        want = a.to(torch.complex128) @ b.to(torch.complex128).mH
    else:
        want = torch.cat((a.real, a.imag)).double() if ac else a.double()
        want = want @ (torch.cat((b.real, b.imag)) if bc else b).double().T
    assert _err(got, want) <= _bar(2 * 2048)
    assert torch.equal(got, P.outer_sum(a, b))
    (torch.view_as_real(a)[3, n - 2, 0] if ac else a[3, n - 2]).fill_(math.inf)
    got = P.outer_sum(a, b)
    rows = torch.arange(got.shape[0], device="cuda") != 3
    assert not got[3].isfinite().any() and _err(got[rows], want[rows]) <= _bar(2 * 2048)


def test_forward_mode_keeps_its_tangents():
    """Dual cotangents through a backward (forward over reverse), and the products
    themselves: at these sizes the kernels serve otherwise."""
    g = _gen(15)
    v, w = _rand(g, 512, 8192).requires_grad_(), _rand(g, 520, 512).requires_grad_()
    (y,) = P.split_projection(v, w, (520,))
    gy, ty = _rand(g, 520, 8192), _rand(g, 520, 8192)
    with forward_ad.dual_level():
        dual = forward_ad.make_dual(gy, ty)
        got = [forward_ad.unpack_dual(t).tangent for t in (
            *torch.autograd.grad(y, (v, w), dual), P.weight_grad(dual, v.detach()),
            P.matmul_adjoint(w.detach(), dual))]
    dv, dw = w.detach().double().T @ ty.double(), ty.double() @ v.detach().double().T
    for t, want in zip(got, (dv, dw, dw, dv)):
        # the library may add one product at a time: N additions, not N / 16
        assert t is not None and _err(t, want) <= _bar(16 * 8192)


def test_lazily_negated_weights():
    g = _gen(16)
    w, x, h = _rand(g, 40, 24, cplx=True), _rand(g, 24, 20000, cplx=True), _rand(g, 7, 48)
    want = -w.to(torch.complex128) @ x.to(torch.complex128)
    neg = torch._neg_view(w)
    assert neg.is_neg() and _err(P.matmul(neg, x), want) <= _bar(48)
    z, logits = P.fused_forward(x, neg, torch._neg_view(h))
    assert _err(z, want) <= _bar(48)
    v = torch.cat((x.real, x.imag)).double()
    assert _err(logits, -h.double() @ v) <= _bar(48)


@pytest.mark.parametrize("tracer", ["jit", "fx"])
def test_traces_hold_the_products(tracer):
    """A trace of products that the kernels serve, run on other data."""
    g = _gen(17)
    w, x, y = (_rand(g, *s, cplx=True) for s in ((64, 64), (64, 20000), (64, 20000)))

    def products(w, x, y):
        leaf = w.detach().requires_grad_()
        out = [P.matmul(w, x), P.matmul_adjoint(w, x), P.weight_grad(x, y)]
        if tracer == "fx":
            out += torch.autograd.grad(P.project(leaf, x), leaf, y)
        return out

    trace = (make_fx(products)(w, x, y) if tracer == "fx"
             else torch.jit.trace(products, (w, x, y), check_trace=False))
    other = [_rand(g, *t.shape, cplx=True) for t in (w, x, y)]
    w64, x64, y64 = (t.to(torch.complex128) for t in other)
    wants = [w64 @ x64, w64.mH @ x64, x64 @ y64.mH, y64 @ x64.mH]
    for got, want in zip(trace(*other), wants):
        # the library may add one product at a time: N additions, not N / 16
        assert _err(got, want) <= _bar(16 * 40000)
