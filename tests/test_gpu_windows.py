"""Sweeps on levels that are windows into larger arrays (strides wider than the
shape): the same bits as on compact arrays, and nothing written outside the
window.  The planes of the wide windows lie so far apart that an array spans
more than 1 and more than 4 GiB."""
import ctypes
import zlib

import numpy as np
import pytest
import torch

import mgp

from test_gpu_parity import random_level, shape_slices

pytestmark = pytest.mark.gpu

REST = -77.0  # the larger array's values outside the window


class Window:
    """`values` (halo included) at `place` in an array of the dimensions `dims`."""

    def __init__(self, values, shape, halo, dims, place, dtype):
        self.t = torch.full(dims, REST, dtype=torch.float64 if dtype == np.float64 else torch.float32, device="cuda")
        self.part = self.t[tuple(slice(p, p + n) for p, n in zip(place, values.shape))]
        self.part.copy_(torch.from_numpy(np.ascontiguousarray(values, dtype=dtype)))
        self.desc = mgp.Array()
        self.desc.data = self.part.data_ptr()
        self.desc.shape[:], self.desc.halo[:], self.desc.stride[:] = shape, halo, self.part.stride()

    def ref(self):
        return ctypes.byref(self.desc)

    def download(self):
        torch.cuda.synchronize()
        return self.part.cpu().numpy()

    def rest_is_untouched(self):
        torch.cuda.synchronize()
        self.part.fill_(REST)
        return bool((self.t == REST).all())


KINDS = ["sweep", "sweep2", "sweep2_prolong", "sweep2_from_zero"]
WIDE = [("f64", (129, 17, 33), "DDDDDD", (1025, 1025)), ("f64", (129, 17, 33), "NDNNDN", (1025, 1025)),
        ("f64", (129, 17, 33), "NNNNDD", (2049, 2049)), ("f32", (257, 17, 33), "DNDNND", (1025, 1025)),
        ("f64", (9, 17, 33), "NNNNNN", (31, 67))]


@pytest.mark.parametrize("sfx,shape,bc,plane", WIDE, ids=["%s_%dx%d_%s" % (w[0], w[3][0], w[3][1], w[2]) for w in WIDE])
def test_sweeps_on_windows_equal_compact_levels(sfx, shape, bc, plane):
    dtype = np.float64 if sfx == "f64" else np.float32
    halo, u0, f, faces, F, box = random_level(shape, bc, mgp.CONSISTENT, dtype, (sfx, shape, bc, plane))
    cs = tuple((n - 1) // 2 + 1 for n in shape)
    rng = np.random.default_rng(zlib.crc32(repr((sfx, shape, bc)).encode()))
    c0, other = rng.standard_normal(mgp.padded_shape(cs, halo)), rng.standard_normal(u0.shape)
    dims, place = (u0.shape[0],) + plane, (0, plane[0] // 3, plane[1] // 3)
    compact = {k: mgp.DeviceArray(s, halo, dtype=dtype).upload(v)
               for k, s, v in (("ui", shape, u0), ("uo", shape, other), ("c", cs, c0))}
    compact["f"] = f
    wide = {k: Window(v, s, halo, d, place, dtype)
            for k, s, v, d in (("ui", shape, u0, dims), ("uo", shape, other, dims), ("f", shape, f.download(), dims),
                               ("c", cs, c0, (c0.shape[0] + 1,) + plane))}
    for kind in KINDS:
        got = []
        for a in (compact, wide):
            first = [] if kind == "sweep2_from_zero" else [a["ui"].ref()]
            last = [a["c"].ref()] if kind == "sweep2_prolong" else []
            print("case", kind, sfx, shape, bc, plane, flush=True)
            mgp.call("mgp_rbgs_%s_%s" % (kind, sfx), mgp.CONSISTENT, *first, a["uo"].ref(), a["f"].ref(),
                     ctypes.byref(F), mgp.box(box), 0.93, *last, None)
            got.append(a["uo"].download())
        np.testing.assert_array_equal(got[1], got[0])
        assert not np.array_equal(got[0][shape_slices(shape, halo)], other.astype(dtype)[shape_slices(shape, halo)])
    assert all(w.rest_is_untouched() for w in wide.values())


# f without the halo u has (as a caller's right-hand side is stored), or with rows
# or planes further apart: a sweep reads it by its own strides
@pytest.mark.parametrize("f_halo,more", [((0,) * 6, None), ((1, 0, 0, 2, 0, 3), None), ((0,) * 6, (40, 9)),
                                         (None, (11, 0))], ids=["none", "own", "window", "planes"])
@pytest.mark.parametrize("sfx", ["f64", "f32"])
@pytest.mark.parametrize("mode", [mgp.REFERENCE, mgp.CONSISTENT])
@pytest.mark.parametrize("shape,bc", [((3, 3, 3), "NNNNNN"), ((9, 31, 65), "NNNNNN"), ((17, 33, 127), "DNDNND"),
                                      ((6, 29, 62), "DDNNDD"), ((65, 129, 65), "NNNNDD")])
def test_sweep_reads_f_by_its_own_strides(shape, bc, mode, sfx, f_halo, more):
    dtype = np.float64 if sfx == "f64" else np.float32
    lv = random_level(shape, bc, mode, dtype, (shape, bc, mode, "f strides"))
    if lv is None:
        pytest.skip("reference colouring is not a checkerboard for this halo layout")
    halo, u0, f, faces, F, box = lv
    values = f.download()[shape_slices(shape, halo)]
    f_halo = halo if f_halo is None else f_halo
    own = np.full(mgp.padded_shape(shape, f_halo), 1e30)
    own[shape_slices(shape, f_halo)] = values
    dims = tuple(n + m for n, m in zip(own.shape, (0,) + (more or (0, 0))))
    got = []
    for rhs in (f, Window(own, shape, f_halo, dims, (0, dims[1] - own.shape[1], 0), dtype)):
        a = mgp.DeviceArray(shape, halo, dtype=dtype).upload(u0)
        b = mgp.DeviceArray(shape, halo, dtype=dtype).upload(u0)
        print("case f strides", shape, bc, mode, sfx, dims, flush=True)
        mgp.call("mgp_rbgs_sweep_" + sfx, mode, a.ref(), b.ref(), rhs.ref(), ctypes.byref(F), mgp.box(box), 0.93, None)
        got.append(b.download())
    np.testing.assert_array_equal(got[1], got[0])
