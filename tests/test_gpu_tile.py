"""The workgroup-tile passes (mgp_tile.hip), the block passes of small levels
(mgp_block.hip, mgp_descend.hip) and the Jacobi march (mgp_jacobi.hip) against
the wave marches and the per-point kernel, bit for bit: one sweep, two sweeps,
two sweeps of u + P(coarse) and of zero, at the sizes where tiles, remainders
and chunks begin and end."""
import ctypes
import zlib

import numpy as np
import pytest

import mgp

from test_gpu_parity import random_level, shape_slices, tuned

pytestmark = pytest.mark.gpu

# most blocks of a launch: none (then tiles), or every level here
PATHS = {"tile": 0, "block": 1 << 20}
# blocks are 16 planes x 12 (FP64) or 16 (FP32) rows x 64 columns.  Tiles are 32 (FP64) or 64 (FP32) rows x 128 columns, two columns per lane;
# rings of 2 (one sweep) or 4 (two sweeps) inside the box
SHAPES = [((3, 3, 3), "NNNNNN"), ((5, 33, 17), "DDDDDD"), ((9, 32, 128), "NNDDNN"), ((8, 34, 130), "DDDDDD"),
          ((11, 35, 131), "DNNDND"), ((7, 56, 129), "NDDNDN"), ((13, 57, 249), "NNNNDD"), ((6, 58, 248), "NNNNNN"),
          ((9, 90, 251), "DDNNDD"), ((21, 31, 370), "NNDDNN"), ((40, 67, 61), "NNNNND"), ((17, 121, 127), "DNDNND"),
          ((300, 9, 7), "NNNNDD"), ((65, 129, 65), "NNNNDD")]


def level(shape, bc, mode, sfx, what):
    dtype = np.float64 if sfx == "f64" else np.float32
    lv = random_level(shape, bc, mode, dtype, (shape, bc, mode, what))
    if lv is None:
        pytest.skip("reference colouring is not a checkerboard for this halo layout")
    return (dtype,) + lv


def run(name, mode, u0, halo, shape, dtype, f, F, box, extra=(), zero=False):
    """The call into a buffer that starts with other values, and its input after it."""
    a = mgp.DeviceArray(shape, halo, dtype=dtype).upload(u0)
    b = mgp.DeviceArray(shape, halo, dtype=dtype).upload(np.random.default_rng(7).standard_normal(u0.shape))
    first = [] if zero else [a.ref()]
    mgp.call(name, mode, *first, b.ref(), f.ref(), ctypes.byref(F), mgp.box(box), 0.93, *extra, None)
    return b.download(), a.download()


@pytest.mark.parametrize("path", list(PATHS))
@pytest.mark.parametrize("sfx", ["f64", "f32"])
@pytest.mark.parametrize("mode", [mgp.REFERENCE, mgp.CONSISTENT])
@pytest.mark.parametrize("shape,bc", SHAPES, ids=["%dx%dx%d_%s" % (s + (b,)) for s, b in SHAPES])
def test_tile_sweeps_equal_wave_marches(shape, bc, mode, sfx, path):
    dtype, halo, u0, f, faces, F, box = level(shape, bc, mode, sfx, "tile")
    rows = 12 if sfx == "f64" else 16
    for name, keys in (("mgp_rbgs_sweep_", {"sweep__rows": rows}), ("mgp_rbgs_sweep2_", {"sweep2__rows": 16})):
        with tuned(**keys):
            want, _ = run(name + sfx, mode, u0, halo, shape, dtype, f, F, box)
        with tuned(sweep2__blocks=PATHS[path]):
            got, after = run(name + sfx, mode, u0, halo, shape, dtype, f, F, box)
        np.testing.assert_array_equal(got, want)
        np.testing.assert_array_equal(after, u0.astype(dtype))


@pytest.mark.parametrize("path", list(PATHS))
@pytest.mark.parametrize("sfx", ["f64", "f32"])
@pytest.mark.parametrize("shape,bc", SHAPES, ids=["%dx%dx%d_%s" % (s + (b,)) for s, b in SHAPES])
def test_tile_correction_and_zero_equal_wave_marches(shape, bc, sfx, path):
    fine = tuple(v | 1 for v in shape)
    dtype, halo, u0, f, faces, F, box = level(fine, bc, mgp.CONSISTENT, sfx, "tile correction")
    cs = tuple((v - 1) // 2 + 1 for v in fine)
    rng = np.random.default_rng(zlib.crc32(repr((shape, bc)).encode()))
    coarse = mgp.DeviceArray(cs, halo, dtype=dtype)
    coarse.upload(rng.standard_normal(coarse.pshape))
    for name, extra, zero in (("mgp_rbgs_sweep2_prolong_", (coarse.ref(),), False),
                              ("mgp_rbgs_sweep2_from_zero_", (), True)):
        with tuned(sweep2__rows=16):
            want, _ = run(name + sfx, mgp.CONSISTENT, u0, halo, fine, dtype, f, F, box, extra, zero)
        with tuned(sweep2__blocks=PATHS[path]):
            got, _ = run(name + sfx, mgp.CONSISTENT, u0, halo, fine, dtype, f, F, box, extra, zero)
        inner = shape_slices(fine, halo)
        np.testing.assert_array_equal(got[inner], want[inner])


@pytest.mark.parametrize("points", [0, 1 << 24], ids=["march", "block"])
@pytest.mark.parametrize("sfx", ["f64", "f32"])
@pytest.mark.parametrize("shape,bc", SHAPES, ids=["%dx%dx%d_%s" % (s + (b,)) for s, b in SHAPES])
def test_descents_equal_wave_march(shape, bc, sfx, points):
    """mgp_residual_restrict_fw through blocks and through the march with
    running sums, r as stored outside the box."""
    dtype, halo, u0, f, faces, F, box = level(shape, bc, mgp.CONSISTENT, sfx, "descent")
    cs = tuple((v - 1) // 2 + 1 for v in shape)
    u = mgp.DeviceArray(shape, halo, dtype=dtype).upload(u0)
    r = mgp.DeviceArray(shape, halo, dtype=dtype).upload(np.random.default_rng(3).standard_normal(u0.shape))
    got = []
    for rows in (6, 0):
        c = mgp.DeviceArray(cs, halo, dtype=dtype)
        c.upload(np.random.default_rng(5).standard_normal(c.pshape))
        with tuned(residual_fw__rows=rows, residual_fw__block_points=points):
            mgp.call("mgp_residual_restrict_fw_" + sfx, mgp.CONSISTENT, u.ref(), f.ref(), r.ref(), c.ref(),
                     mgp.box(box), F.h, None)
        got.append(c.download())
    np.testing.assert_array_equal(got[1], got[0])


# a level of more points than "sweep.small_points": chunks of 6 planes at least
def test_hilo_rows_give_the_same_bits():
    shape, bc = (70, 66, 71), "NNNNDD"
    dtype, halo, u0, f, faces, F, box = level(shape, bc, mgp.CONSISTENT, "f64", "hilo")
    rng = np.random.default_rng(11)
    new = lambda dt, v: mgp.DeviceArray(shape, halo, dtype=dt).upload(v)  # noqa: E731
    hi, lo = new(np.float64, u0), new(np.float32, rng.standard_normal(u0.shape) * 1e-16)
    e, r = new(np.float32, rng.standard_normal(u0.shape) * 1e-3), new(np.float64, rng.standard_normal(u0.shape))
    got = []
    for rows in (16, 8):
        nrm = mgp.DeviceBuffer(np.zeros(1))
        un, ln, out = (new(dt, np.ones(u0.shape)) for dt in (np.float64, np.float32, np.float32))
        with tuned(update_residual__rows=rows):
            mgp.call("mgp_update_residual_hilo_f64_f32", hi.ref(), un.ref(), lo.ref(), ln.ref(), e.ref(), f.ref(),
                     r.ref(), out.ref(), ctypes.byref(F), mgp.box(box), nrm.ptr, None)
        got.append([a.download() for a in (un, ln, out, nrm)])
    for a, b in zip(*got):
        np.testing.assert_array_equal(a, b)


# tiles of 16 rows x 124 columns; the three arrays with halos of their own
@pytest.mark.parametrize("sfx", ["f64", "f32"])
@pytest.mark.parametrize("mode", [mgp.REFERENCE, mgp.CONSISTENT])
@pytest.mark.parametrize("shape,bc", SHAPES + [((4, 17, 124), "NNNNNN"), ((3, 16, 125), "NNNNNN"),
                                               ((5, 4, 250), "DDDDDD"), ((2, 20, 2), "NNNNNN")])
def test_jacobi_march_equals_per_point(shape, bc, mode, sfx):
    dtype = np.float64 if sfx == "f64" else np.float32
    rng = np.random.default_rng(zlib.crc32(repr((shape, bc, mode, sfx)).encode()))
    box = [v for d in range(3) for v in (0 if bc[2 * d] == "N" else 1, shape[d] - (bc[2 * d + 1] == "D"))]
    v, f = (mgp.DeviceArray(shape, halo, dtype=dtype) for halo in ((1,) * 6, (2, 0, 1, 3, 0, 1)))
    for a in (v, f):
        a.upload(rng.standard_normal(a.pshape))
    got = []
    for kernel in (1, 2):
        u = mgp.DeviceArray(shape, (0, 1, 0, 2, 1, 0), dtype=dtype)
        u.upload(np.random.default_rng(7).standard_normal(u.pshape))
        with tuned(jacobi__kernel=kernel):
            mgp.call("mgp_jacobi_" + sfx, mode, u.ref(), v.ref(), f.ref(), mgp.box(box), 6.0 / 7.0, 1.0 / 16, None)
        got.append(u.download())
    np.testing.assert_array_equal(got[1], got[0])


# one workgroup, points per thread and colour: 2 (FP64 and FP32) and 4 (FP32),
# odd and even box lengths
@pytest.mark.parametrize("sfx,shape,bc", [("f64", (15, 15, 14), "NNNNNN"), ("f64", (15, 15, 14), "DNNDND"),
                                          ("f32", (19, 19, 19), "DDDDDD"), ("f32", (18, 20, 19), "NDDNDN"),
                                          ("f64", (40, 2, 3), "NNDDDD"), ("f32", (16, 14, 15), "NNNNNN")])
@pytest.mark.parametrize("mode", [mgp.REFERENCE, mgp.CONSISTENT])
def test_lds_sweeps_with_several_points_per_thread(mode, sfx, shape, bc):
    dtype, halo, u0, f, faces, F, box = level(shape, bc, mode, sfx, "lds")
    a = mgp.DeviceArray(shape, halo, dtype=dtype).upload(u0)
    b = mgp.DeviceArray(shape, halo, dtype=dtype).upload(u0)
    c = mgp.DeviceArray(shape, halo, dtype=dtype).upload(u0)
    mgp.call("mgp_rbgs_sweeps_" + sfx, mode, a.ref(), c.ref(), f.ref(), ctypes.byref(F), mgp.box(box), 0.93, 3, None)
    for _ in range(3):
        mgp.call("mgp_rbgs_sweep_" + sfx, mode, a.ref(), b.ref(), f.ref(), ctypes.byref(F), mgp.box(box), 0.93, None)
        a, b = b, a
    np.testing.assert_array_equal(c.download(), a.download())


# boxes that leave planes, rows and columns outside, nothing, or everything
@pytest.mark.parametrize("sfx", ["f64", "f32"])
@pytest.mark.parametrize("shape,box", [((9, 7, 70), (1, 8, 2, 6, 3, 69)), ((6, 5, 4), (0, 6, 0, 5, 0, 4)),
                                       ((6, 5, 4), (2, 2, 1, 4, 1, 3)), ((20, 33, 65), (0, 19, 1, 33, 1, 64)),
                                       ((7, 40, 3), (3, 7, 0, 40, 1, 2)), ((5, 6, 130), (1, 4, 5, 6, 0, 130))])
def test_residual_norm_outside_the_box(shape, box, sfx):
    dtype = np.float64 if sfx == "f64" else np.float32
    rng = np.random.default_rng(zlib.crc32(repr((shape, box, sfx)).encode()))
    u, f = (mgp.DeviceArray(shape, (1,) * 6, dtype=dtype) for _ in range(2))
    for a in (u, f):
        a.upload(rng.standard_normal(a.pshape))
    r0 = rng.standard_normal(u.pshape)
    for place in [(0, 0, 0), (shape[0] - 1, shape[1] - 1, shape[2] - 1), (shape[0] // 2, 0, 1), (1, shape[1] // 2, 0)]:
        r0[1:-1, 1:-1, 1:-1][place] = 1e6 * (1 + sum(place))  # read where the box leaves it out
        r = mgp.DeviceArray(shape, (1,) * 6, dtype=dtype)
        for name in ("mgp_residual_", "mgp_residual_norm_"):
            r.upload(r0)
            nrm = mgp.DeviceBuffer(np.zeros(1))
            mgp.call(name + sfx, mgp.CONSISTENT, u.ref(), f.ref(), r.ref(), mgp.box(box), 1.0, nrm.ptr, None)
            if name == "mgp_residual_":
                want = float(np.abs(r.download()[1:-1, 1:-1, 1:-1]).max())
            assert nrm.download()[0] == want


@pytest.mark.parametrize("sfx", ["f64", "f32"])
@pytest.mark.parametrize("shape,bc", [((3, 3, 3), "NNNNNN"), ((5, 33, 17), "DDDDDD"), ((17, 9, 129), "NDDNDN"),
                                      ((33, 35, 65), "NNNNDD")])
def test_small_levels_per_point_equal_marches(shape, bc, sfx):
    """Prolongation + add and the stored residual: the route of small levels
    against the march."""
    got = []
    for points in (1 << 30, 0):
        with tuned(small__point_points=points):
            for mode in (mgp.REFERENCE, mgp.CONSISTENT):
                dtype, halo, u0, f, faces, F, box = level(shape, bc, mgp.CONSISTENT, sfx, "small")
                u, r = (mgp.DeviceArray(shape, halo, dtype=dtype).upload(u0) for _ in range(2))
                mgp.call("mgp_residual_" + sfx, mode, u.ref(), f.ref(), r.ref(), mgp.box(box), F.h, None, None)
                got.append(r.download())
            c = mgp.DeviceArray(tuple((v - 1) // 2 + 1 for v in shape), halo, dtype=dtype)
            c.upload(np.random.default_rng(9).standard_normal(c.pshape))
            mgp.call("mgp_prolong_add_" + sfx, c.ref(), u.ref(), None)
            got.append(u.download())
    for a, b in zip(got[:3], got[3:]):
        np.testing.assert_array_equal(a, b)
