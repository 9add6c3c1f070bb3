"""Products over zero terms, on the host.

A projection whose data has no rows has no weight planes either: every layout refuses
it before anything is launched, as the Python layer's empty weights always did.  The
calls pass stand-in device pointers (aligned, non-null, never dereferenced on the
host); one that got past the check would reach a HIP launch and return a HIP error
code.  Stand-in pointers must never reach a device, so the module is skipped where one
is visible.
"""

import pytest
import torch

from prospective_rqf_amd import _lib
from prospective_rqf_amd import projection as P

pytestmark = pytest.mark.skipif(torch.cuda.is_available(),
                                reason="stand-in device pointers: host-side checks only")

PTR = 0x10000  # stand-in device pointer: non-null and 16-byte aligned
ERR_ARG = -1
# (w_rows, w_cols, h_rows) without a row of data, with a row of output
EMPTY = {P.FORWARD: (5, 0, 3), P.ADJOINT: (0, 5, 0), P.REAL: (0, 0, 4), P.REAL_T: (0, 4, 0),
         P.PAIRED: (0, 0, 6), P.PAIRED_T: (0, 6, 0)}


@pytest.mark.parametrize("mode", sorted(EMPTY))
@pytest.mark.parametrize("workspace", [None, PTR])
def test_every_layout_refuses_it(mode, workspace):
    lib = _lib.load()
    w_rows, w_cols, h_rows = EMPTY[mode]
    rc = lib.rqf_projection(mode, PTR, w_rows, w_cols, PTR, h_rows, PTR, PTR, 300, PTR, PTR, None,
                            0, workspace, 0, None)
    assert rc == ERR_ARG
    # no column, or no row of output: nothing to do
    assert lib.rqf_projection(mode, PTR, w_rows, w_cols, PTR, h_rows, PTR, PTR, 0, PTR, PTR, None,
                              0, workspace, 0, None) == 0
    assert lib.rqf_projection(mode, None, 0, 0, None, 0, None, None, 300, None, None, None, 0,
                              workspace, 0, None) == 0
