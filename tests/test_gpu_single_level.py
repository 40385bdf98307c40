"""Refinement solves on one level: that level is the finest and the coarsest
at once, so its smoothing starts from a zero correction and runs in FP64
arithmetic where the level fits one workgroup."""
import numpy as np
import pytest

import mgp

from test_gpu_parity import tuned

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsmooth,coarse", [(2, 0), (3, 0), (2, 8)])
@pytest.mark.parametrize("dims,bc", [((13, 13, 9), "DDDDDD"), ((9, 11, 14), "NNDDND"), ((15, 15, 17), "DDNNDD"),
                                     ((21, 21, 21), "DDDDDD")])
def test_single_level_refinement_keeps_fp64_smoothing(dims, bc, nsmooth, coarse):
    """With and without pairs of sweeps: the zero correction's first pair must
    not replace the FP64 passes.  (21, 21, 21) does not fit in FP64: FP32 passes
    either way."""
    got = []
    for pair in (0, 1):
        with tuned(sweep__pair=pair):
            s = mgp.Solver(dims, 1, 1.0 / (dims[0] - 1), bc=bc, mode=mgp.CONSISTENT, restriction=mgp.FULL_WEIGHTING,
                           problem=2, dtype=mgp.MIXED, flags=mgp.QUIET, maxiter=4, tolerance=1e-30,
                           coarse_sweeps=coarse)
            s.to_device()
            print("case single level", dims, bc, nsmooth, coarse, pair, flush=True)
            its, rel, _ = s.solve("Vcycle", nsmooth, 1.0)
            s.to_host()
            got.append((its, rel, s.array("u").copy(), s.lo_word()))
            s.close()
    assert got[0][0] == got[1][0] and got[0][1] == got[1][1]
    np.testing.assert_array_equal(got[0][2], got[1][2])
    np.testing.assert_array_equal(got[0][3], got[1][3])
