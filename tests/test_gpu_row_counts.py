"""GPU parity of the row kernels by how many rows there are and how long they are.

The forwards pick a block's wavefronts by the tiles of a row and by the rows against
the 256 CUs, the FBT backward its form by the rows and their length (row blocks for at
most 1024 rows of more than twice as many steps), and the selective kernels place (item, batch element) pairs for any batch size.  Every
choice is checked against the fp64 oracle, at the bars of the other parity tests.
"""

import numpy as np
import pytest
import torch

from oracle import oracle
from prospective_rqf_amd.fbt_scan_kernel import (
    fbt_layer0_real_scan,
    fbt_prospective_scan,
    fbt_recompute_scan,
)
from tests.helpers import PARITY_RTOL, chanerr, cotangent_off_relu_kink, crandn, relerr
from tests.test_gpu_dispatch_matrix import OUTPUTS, SETS
from tests.test_gpu_selective import CASE_ALL, run_case
from tests.test_gpu_timeinv import _c64, _coeffs, _dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


# one to five 512-step tiles, two super-tiles of 16 wavefronts, and 1100 rows (the
# backward with one wavefront per row; five rows per CU)
SHAPES = [(3, 1, 161), (2, 2, 511), (2, 1, 513), (3, 1, 1025), (2, 1, 2049), (3, 1, 4097),
          (2, 1, 8193), (550, 2, 301), (275, 4, 257), (300, 1, 599), (300, 1, 601),
          (1023, 1, 2047)]


@pytest.mark.parametrize("variant", ["raw", "act", "recompute", "layer0"])
@pytest.mark.parametrize("F,B,T", SHAPES)
def test_fbt_rows(variant, F, B, T):
    print(f"case: fbt rows {variant} {F} {B} {T}", flush=True)
    rng = np.random.default_rng(F + B + T)
    c1, t0, t1 = _coeffs(rng, F)
    layer0 = variant == "layer0"
    w = rng.standard_normal((2 * F, 1)).astype(np.float32)
    h = rng.standard_normal((1, B * T)).astype(np.float32)
    wz = w[:F, 0].astype(np.float64) + 1j * w[F:, 0]
    z = (_c64(wz[:, None] * h).reshape(F, B, T) if layer0 else _c64(crandn(rng, F, B, T)))
    mask = variant != "raw"
    y_ref, act_ref = oracle.twotap_fwd(c1, t0, t1, z, layout=oracle.FBT, act=True)
    gy = _c64(crandn(rng, F, B, T))
    if mask:
        gy = _c64(cotangent_off_relu_kink(y_ref, gy)[0])
    gz, *gc = oracle.twotap_bwd(c1, t0, t1, z, y_ref, gy, layout=oracle.FBT, mask_act=mask)
    C1, T0, T1 = _dev(c1), _dev(t0), _dev(t1)
    if layer0:
        x = torch.as_tensor(h, device="cuda").requires_grad_(True)
        y = fbt_layer0_real_scan(torch.as_tensor(w, device="cuda"), x, C1, T0, T1, B)
        gz = (wz.conj()[:, None] * gz.reshape(F, -1)).sum(0, keepdims=True).real
    else:
        x = _dev(z)
        y = (fbt_recompute_scan(C1, T0, T1, x) if variant == "recompute"
             else fbt_prospective_scan(C1, T0, T1, x, fuse_act=mask))
    y.backward(torch.as_tensor(gy.astype(np.complex64), device="cuda"))
    assert relerr(y, act_ref if mask else y_ref) <= PARITY_RTOL
    assert relerr(x.grad, gz) <= PARITY_RTOL
    for got, want in zip((C1.grad, T0.grad, T1.grad), gc):
        assert relerr(got, want) <= PARITY_RTOL and chanerr(got, want) <= PARITY_RTOL


@pytest.mark.parametrize("B", [1, 2, 7, 8, 9, 17])
def test_selective_batch_order(B):
    """Every batch size against the eight chunks of the block order."""
    print(f"case: selective B={B}", flush=True)
    run_case(6, B, 300, CASE_ALL, seed=B)


@pytest.mark.parametrize("outputs", [(False, True), (True, False), (True, True)])
@pytest.mark.parametrize("T", [4097, 8191, 8192, 8193, 9001])
def test_selective_sixteen_wavefronts(T, outputs):
    """Super-tiles of 8192 steps: few rows longer than 4096 steps take them."""
    print(f"case: selective few rows T={T} outputs={outputs}", flush=True)
    run_case(3, 1, T, CASE_ALL, activate=outputs[0], write_raw=outputs[1], chunk=256, seed=T)


@pytest.mark.parametrize("out", list(OUTPUTS))
@pytest.mark.parametrize("name", list(SETS))
@pytest.mark.parametrize("waves,T", [("narrow", 2051), ("narrow", 2052), ("few", 8200),
                                     ("few", 8203)])
def test_selective_block_sizes_of_every_option_set(monkeypatch, waves, T, name, out):
    print(f"case: selective {waves} {name} {out}", flush=True)
    monkeypatch.setenv("RQF_FWD_WAVES", waves)
    case, opts = SETS[name]
    activate, write_raw = OUTPUTS[out]
    run_case(3, 2, T, case, activate=activate, write_raw=write_raw, chunk=256, G=3, seed=T,
             **opts)


@pytest.mark.parametrize("out", list(OUTPUTS))
@pytest.mark.parametrize("name", list(SETS))
@pytest.mark.parametrize("waves", ["narrow", "wide", "few"])
@pytest.mark.parametrize("T", [1, 161, 511])
def test_selective_rows_below_one_tile(monkeypatch, T, waves, name, out):
    """Unaligned rows without a whole 512-step tile have kernels of their own."""
    print(f"case: selective short T={T} {waves} {name} {out}", flush=True)
    monkeypatch.setenv("RQF_FWD_WAVES", waves)
    case, opts = SETS[name]
    activate, write_raw = OUTPUTS[out]
    run_case(3, 2, T, case, activate=activate, write_raw=write_raw, chunk=64, G=3, seed=T, **opts)


@pytest.mark.parametrize("F,T,G", [(16, 100, 1), (40, 2000, 1), (40, 2001, 1), (30, 1000, 3),
                                   (30, 1001, 3)])
def test_selective_one_recording(F, T, G):
    """The backward of one short recording runs on one XCD, up to 80000 steps of all
    channels with one or two warp rows, else 30000."""
    print(f"case: selective one recording {F} {T} {G}", flush=True)
    run_case(F, 1, T, CASE_ALL, G=G, seed=T)
