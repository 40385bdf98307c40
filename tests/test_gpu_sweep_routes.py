"""Routes of the sweeps that small levels at default keys do not take, bit for
bit against another route: the packed wave marches over several x chunks, and
the workgroup tiles where a march is long, a narrow last z column is not packed
and a single sweep has Dirichlet faces only."""
import ctypes
import zlib

import numpy as np
import pytest
import torch

import mgp

from test_gpu_parity import PRO_CHUNKS, PRO_SHAPES, random_level, shape_slices, tuned

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunks", range(len(PRO_CHUNKS)), ids=["c1", "c4", "cx"])
@pytest.mark.parametrize("sfx", ["f64", "f32"])
@pytest.mark.parametrize("shape,bc", PRO_SHAPES, ids=[str(i) for i in range(len(PRO_SHAPES))])
def test_packed_wave_marches_over_chunks(shape, bc, sfx, chunks):
    """"sweep2.rows" 16 keeps the two-sweep passes on the wave march, its stages
    packed by colour: with the correction inside and from zero, against the
    default route of the separate calls."""
    dtype = np.float64 if sfx == "f64" else np.float32
    halo, u0, f, faces, F, box = random_level(shape, bc, mgp.CONSISTENT, dtype, (shape, bc, sfx, "packed march"))
    cs = tuple((n - 1) // 2 + 1 for n in shape)
    rng = np.random.default_rng(zlib.crc32(repr((shape, bc, "packed march")).encode()))
    c = mgp.DeviceArray(cs, halo, dtype=dtype)
    c.upload(rng.standard_normal(c.pshape))
    a, b, want, got = (mgp.DeviceArray(shape, halo, dtype=dtype).upload(u0) for _ in range(4))
    inner = shape_slices(shape, halo)
    print("case packed march", shape, bc, sfx, chunks, flush=True)
    tail = (f.ref(), ctypes.byref(F), mgp.box(box), 0.93)
    mgp.call("mgp_prolong_add_" + sfx, c.ref(), a.ref(), None)
    mgp.call("mgp_rbgs_sweep2_" + sfx, mgp.CONSISTENT, a.ref(), want.ref(), *tail, None)
    with tuned(sweep2__rows=16, sweep2__pack=3, **PRO_CHUNKS[chunks]):
        mgp.call("mgp_rbgs_sweep2_prolong_" + sfx, mgp.CONSISTENT, b.ref(), got.ref(), *tail, c.ref(), None)
    np.testing.assert_array_equal(got.download()[inner], want.download()[inner])
    a.upload(np.zeros(a.pshape))
    mgp.call("mgp_rbgs_sweep2_" + sfx, mgp.CONSISTENT, a.ref(), want.ref(), *tail, None)
    with tuned(sweep2__rows=16, sweep2__pack=3, **PRO_CHUNKS[chunks]):
        mgp.call("mgp_rbgs_sweep2_from_zero_" + sfx, mgp.CONSISTENT, got.ref(), *tail, None)
    np.testing.assert_array_equal(got.download()[inner], want.download()[inner])


class Field:
    """A device array of random values (or `fill`), its halo included."""

    def __init__(self, shape, halo, dtype, seed, fill=None):
        p = mgp.padded_shape(shape, halo)
        g = torch.Generator(device="cuda").manual_seed(seed)
        self.t = torch.randn(p, dtype=dtype, device="cuda", generator=g) if fill is None else \
            torch.full(p, fill, dtype=dtype, device="cuda")
        self.shape = self.t[shape_slices(shape, halo)]
        self.desc = mgp.Array()
        self.desc.data = self.t.data_ptr()
        self.desc.shape[:], self.desc.halo[:], self.desc.stride[:] = shape, halo, self.t.stride()

    def ref(self):
        return ctypes.byref(self.desc)


# 2^25 points and more: the correction's narrow last z column (9 of 128 columns)
# is not packed in FP64; 2^27 and more: neither in FP32, nor in the FP64 pair.
# 257 x 257 x 129: marches of some 24 planes, past the steps near their ends
LONG = [((257, 257, 129), "NNNNDD", "f64"), ((257, 257, 129), "DNDNND", "f32"), ((641, 65, 257), "NNNNNN", "f32"),
        ((401, 90, 249), "DDDDDD", "f64"), ((513, 513, 129), "NNNNNN", "f64"), ((513, 521, 129), "DDDDDN", "f64"),
        ((1025, 1025, 129), "NNNNNN", "f32"), ((1025, 1025, 131), "NDDNND", "f32"), ((1025, 1025, 129), "NNNNNN", "f64")]


@pytest.mark.parametrize("shape,bc,sfx", LONG, ids=["%dx%dx%d_%s_%s" % (s + (b, t)) for s, b, t in LONG])
def test_long_tile_marches_equal_wave_marches(shape, bc, sfx):
    dtype = torch.float64 if sfx == "f64" else torch.float32
    halo = [1 if ch == "N" else 0 for ch in bc]
    F = mgp.Faces()
    F.h = 1.0 / 64
    faces = []
    for q in range(6):
        n = [1 if d == (1, 1, 0, 0, 2, 2)[q] else shape[d] for d in range(3)]
        faces.append(Field(n, [0] * 6, dtype, q))
        F.type[q] = mgp.NEUMANN if bc[q] == "N" else mgp.DIRICHLET
        F.g[q] = faces[q].t.data_ptr() if bc[q] == "N" else None
    box = [int(bc[3] == "D"), shape[0] - int(bc[2] == "D"), int(bc[1] == "D"), shape[1] - int(bc[0] == "D"),
           int(bc[5] == "D"), shape[2] - int(bc[4] == "D")]
    cs = [(n - 1) // 2 + 1 for n in shape]
    u, f, c = Field(shape, halo, dtype, 10), Field(shape, halo, dtype, 11), Field(cs, halo, dtype, 12)
    kinds = ["sweep", "sweep2", "sweep2_from_zero"]
    if all(n % 2 for n in shape):  # nested 2:1
        kinds.append("sweep2_prolong")
    for kind in kinds:
        first = [] if kind == "sweep2_from_zero" else [u.ref()]
        last = [c.ref()] if kind == "sweep2_prolong" else []
        got = []
        for keys in ({"sweep__rows": 12 if sfx == "f64" else 16, "sweep2__rows": 16}, {"sweep2__blocks": 0}):
            out = Field(shape, halo, dtype, 0, fill=-77.0)
            torch.cuda.synchronize()
            print("case long", kind, shape, bc, sfx, keys, flush=True)
            with tuned(**keys):
                mgp.call("mgp_rbgs_%s_%s" % (kind, sfx), mgp.CONSISTENT, *first, out.ref(), f.ref(), ctypes.byref(F),
                         mgp.box(box), 0.93, *last, None)
            mgp.check(mgp.lib().mgp_stream_sync(None))
            got.append(out.t)
        assert torch.equal(got[1], got[0]), kind
        del got
