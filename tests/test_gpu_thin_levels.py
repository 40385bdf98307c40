"""mgp_rbgs_sweeps_* on thin levels at the limit of its size: the rows and
planes padded to odd lengths take the most LDS there (FP64 408 x 2 x 2: 82000
bytes for a level that fills 64 KiB)."""
import ctypes

import numpy as np
import pytest

import mgp

from test_gpu_parity import random_level

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,shape", [("f64", (408, 2, 2)), ("f64", (2, 408, 2)), ("f64", (2, 2, 408)),
                                        ("f64", (254, 2, 4)), ("f64", (100, 4, 6)), ("f32_f64", (408, 2, 2)),
                                        ("f32", (512, 2, 2)), ("f32", (256, 4, 4))])
def test_thin_levels_at_the_limit(name, shape):
    """Three passes in one launch equal three one-pass sweeps."""
    dtype = np.float64 if name == "f64" else np.float32
    halo, u0, f, faces, F, box = random_level(shape, "NNNNNN", mgp.CONSISTENT, dtype, (name, shape))
    u, out = (mgp.DeviceArray(shape, halo, dtype=dtype).upload(u0) for _ in range(2))
    print("case thin", name, shape, flush=True)
    mgp.call("mgp_rbgs_sweeps_" + name, mgp.CONSISTENT, u.ref(), out.ref(), f.ref(), ctypes.byref(F), mgp.box(box),
             0.93, 3, None)
    # the sweeps one by one, in the arithmetic's type
    wide = np.float32 if name == "f32" else np.float64
    a, b, rhs = (mgp.DeviceArray(shape, halo, dtype=wide).upload(v) for v in (u.download(), u.download(), f.download()))
    g = {q: mgp.DeviceBuffer(faces[q].download().astype(wide)) for q in faces}
    for q in g:
        F.g[q] = g[q].ptr
    for _ in range(3):
        mgp.call("mgp_rbgs_sweep_" + a.sfx, mgp.CONSISTENT, a.ref(), b.ref(), rhs.ref(), ctypes.byref(F),
                 mgp.box(box), 0.93, None)
        a, b = b, a
    inner = tuple(slice(1, -1) for _ in shape)
    np.testing.assert_array_equal(out.download()[inner], a.download()[inner].astype(dtype))
