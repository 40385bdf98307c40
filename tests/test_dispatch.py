"""Which kernel a call takes, checked on the CPU with the launches recorded
instead of run: what a kernel's addresses cannot reach goes to one that can."""
import pytest

import launch_recorder

NO_HALO = [0] * 6


@pytest.fixture(scope="module")
def recorder(tmp_path_factory):
    return launch_recorder.build(str(tmp_path_factory.mktemp("recorder")))


def sweep_call(kind, sfx, shape, strides=None, f_strides=None, c_strides=None, bc="DDDDDD", keys=None):
    """mgp_rbgs_<kind>_<sfx> on arrays without halo (strides None: compact)."""
    arrays = {"ui": (shape, NO_HALO, strides), "uo": (shape, NO_HALO, strides),
              "f": (shape, NO_HALO, f_strides or strides),
              "c": ([(n - 1) // 2 + 1 for n in shape], NO_HALO, c_strides)}
    first = [1] + ([] if kind == "sweep2_from_zero" else ["ui"])
    last = (["c"] if kind == "sweep2_prolong" else []) + ([3] if kind == "sweeps" else [])
    box = [0 if bc[3] == "N" else 1, shape[0] - (bc[2] == "D"), 0 if bc[1] == "N" else 1, shape[1] - (bc[0] == "D"),
           0 if bc[5] == "N" else 1, shape[2] - (bc[4] == "D")]
    return {"name": "mgp_rbgs_%s_%s" % (kind, sfx), "arrays": arrays, "bc": bc, "box": box, "h": 1.0 / 16,
            "args": first + ["uo", "f", "faces", "box", 0.93] + last + ["stream"], "keys": keys or {}}


PAIRS = ["sweep2", "sweep2_prolong", "sweep2_from_zero"]


# a window of `shape` in an array of n1 x n2 points per plane: its points are few
# enough for blocks, its bytes from first to last are past what a 32-bit offset
# with an out-of-range value left over can address
@pytest.mark.parametrize("kind", PAIRS)
@pytest.mark.parametrize("sfx,shape,n1,n2", [("f64", [129, 17, 33], 1025, 1025), ("f64", [129, 17, 33], 2049, 2049),
                                             ("f32", [257, 33, 33], 1025, 1025), ("f64", [3, 9, 33], 4097, 16385)])
def test_wide_windows_do_not_run_as_blocks(recorder, kind, sfx, shape, n1, n2):
    size = 8 if sfx == "f64" else 4
    wide = [n1 * n2, n2, 1]
    span = ((shape[0] - 1) * wide[0] + (shape[1] - 1) * wide[1] + shape[2]) * size
    assert span >= 1 << 30
    # the same window with its planes just close enough, and compact
    near = [((1 << 30) // size - (shape[1] - 1) * n2 - shape[2] - 1) // (shape[0] - 1), n2, 1]
    calls = [sweep_call(kind, sfx, shape, s) for s in (wide, near, None)]
    kernels = [[k[0] for k in ks] for rc, ks in launch_recorder.record(recorder, calls) if rc == 0]
    assert ["k_rbgs_tile" in k[0] for k in kernels] == [True, False, False], kernels
    assert ["k_rbgs_block" in k[0] for k in kernels] == [False, True, True], kernels


def test_wide_coarse_planes_do_not_run_as_blocks(recorder):
    """A coarse plane past 1 GiB is refused by the blocks as by the tiles and the
    wave march: MGP_ERR_ARG, and nothing launched."""
    shape = [17, 33, 33]
    wide = [17 << 23, 1 << 23, 1]  # 16 rows on: 1 GiB in FP64
    ok = [17 << 22, 1 << 22, 1]
    r = launch_recorder.record(recorder, [sweep_call("sweep2_prolong", "f64", shape, c_strides=s) for s in (wide, ok)])
    assert r[0] == (-1, [])
    assert r[1][0] == 0 and "k_rbgs_block" in r[1][1][0][0]


# f beside a u with a halo on every face: without one, with rows or planes
# further apart
F_LAYOUTS = {"no halo": lambda n: [n[1] * n[2], n[2], 1], "rows apart": lambda n: [(n[1] + 2) * (n[2] + 9), n[2] + 9, 1],
             "planes apart": lambda n: [(n[1] + 40) * (n[2] + 2), n[2] + 2, 1]}


@pytest.mark.parametrize("layout", list(F_LAYOUTS))
@pytest.mark.parametrize("sfx", ["f64", "f32"])
@pytest.mark.parametrize("shape", [[5, 9, 33], [129, 33, 130]])
def test_f_with_its_own_strides_is_not_read_by_u_strides(recorder, shape, sfx, layout):
    """One sweep goes to the kernel that addresses f by its own strides; a pair,
    which has none, is refused (single sweeps then)."""
    calls = []
    for kind in ["sweep"] + PAIRS:
        c = sweep_call(kind, sfx, shape, bc="NNNNNN")
        for name in ("ui", "uo", "c"):
            c["arrays"][name] = (c["arrays"][name][0], [1] * 6, None)
        c["arrays"]["f"] = (shape, NO_HALO, F_LAYOUTS[layout](shape))
        calls.append(c)
    got = launch_recorder.record(recorder, calls)
    assert got[0][0] == 0 and len(got[0][1]) == 1 and "k_rbgs_march" in got[0][1][0][0], got[0]
    assert got[1:] == [(-1, [])] * 3, got[1:]


@pytest.mark.parametrize("sfx", ["f64", "f32"])
def test_planes_past_32_bit_offsets_are_refused(recorder, sfx):
    """A plane of u or f whose bytes do not fit 32-bit offsets: MGP_ERR_ARG."""
    n2 = 1 << (25 if sfx == "f64" else 26)
    wide, near, shape = [17 * n2, n2, 1], [17 * n2, n2 - 8, 1], [5, 17, 33]
    calls = [sweep_call("sweep", sfx, shape, wide), sweep_call("sweep", sfx, shape, None, wide),
             sweep_call("sweep", sfx, shape, near), sweep_call("sweep", sfx, shape, None, near)]
    got = launch_recorder.record(recorder, calls)
    assert got[:2] == [(-1, [])] * 2, got[:2]
    assert all(rc == 0 and "k_rbgs_march" in k[0][0] for rc, k in got[2:]), got[2:]


@pytest.mark.parametrize("sfx", ["f64", "f32"])
@pytest.mark.parametrize("shape", [[129, 129, 129], [257, 131, 70], [513, 513, 33]])
def test_descent_march_takes_target_zero_as_the_sweeps_target(recorder, shape, sfx):
    """"residual_fw.target_wgs" 0 means the value of "sweep.target_wgs": as many
    waves as that value set directly, not one march per tile."""
    coarse = [(n - 1) // 2 + 1 for n in shape]
    arrays = {"u": (shape, [1] * 6, None), "f": (shape, [1] * 6, None), "r": (shape, [1] * 6, None),
              "c": (coarse, NO_HALO, None)}
    calls = [{"name": "mgp_residual_restrict_fw_" + sfx, "arrays": arrays, "bc": "NNNNNN", "h": 1.0 / 16,
              "box": [0, shape[0], 0, shape[1], 0, shape[2]], "args": [1, "u", "f", "r", "c", "box", 1.0 / 16, "stream"],
              "keys": {"residual_fw.target_wgs": target, "sweep.target_wgs": 20000}} for target in (0, 20000, 1)]
    (zero, same, one) = (k for rc, k in launch_recorder.record(recorder, calls))
    assert "k_resid_fw_march" in zero[0][0]
    assert zero == same and zero[0][1] > 2 * one[0][1]


def jacobi_call(sfx, shape, keys=None):
    arrays = {n: (shape, [1] * 6, None) for n in "uvf"}
    return {"name": "mgp_jacobi_" + sfx, "arrays": arrays, "bc": "NNNNNN", "h": 1.0, "keys": keys or {},
            "box": [0, shape[0], 0, shape[1], 0, shape[2]],
            "args": [1, "u", "v", "f", "box", 0.9, 1.0, "stream"]}


# box sizes on both sides of the rule: points, and (FP32) how much of 16 rows x
# 124 columns per tile the box fills
@pytest.mark.parametrize("sfx,shape,march", [
    ("f64", [33, 33, 33], False), ("f64", [56, 332, 34], False), ("f64", [127, 128, 64], False),
    ("f64", [128, 128, 64], True), ("f64", [1025, 33, 33], False), ("f64", [2049, 33, 33], True),
    ("f64", [1025, 32, 41], False), ("f64", [1025, 32, 42], True), ("f64", [385, 353, 321], True),
    ("f32", [65, 65, 65], False), ("f32", [127, 128, 128], False), ("f32", [128, 128, 128], True),
    ("f32", [359, 125, 61], False), ("f32", [1024, 512, 61], False), ("f32", [1024, 512, 62], True),
    ("f32", [1024, 17, 248], True), ("f32", [1024, 17, 220], False), ("f32", [707, 707, 33], False)])
def test_jacobi_march_where_it_pays(recorder, sfx, shape, march):
    calls = [jacobi_call(sfx, shape), jacobi_call(sfx, shape, {"jacobi.kernel": 2}),
             jacobi_call(sfx, shape, {"jacobi.kernel": 1})]
    names = [k[0][0] for rc, k in launch_recorder.record(recorder, calls)]
    assert ["k_jacobi_march" in n for n in names] == [march, True, False], names


# levels on both sides of the rule: 3 * 2^19 points, and 5 * 2^19 lanes with the
# rows of z filled up to 64
@pytest.mark.parametrize("shape,per_point", [
    ([65, 65, 65], True), ([129, 129, 65], True), ([33, 33, 17], True), ([45, 73, 309], True), ([129, 129, 129], False),
    ([105, 381, 13], True), ([109, 381, 13], False), ([359, 279, 11], False), ([125, 733, 15], False), ([647, 257, 9], False)])
@pytest.mark.parametrize("sfx", ["f64", "f32"])
def test_small_levels_per_point_unless_narrow(recorder, sfx, shape, per_point):
    coarse = [(n - 1) // 2 + 1 for n in shape]
    box = [0, shape[0], 0, shape[1], 0, shape[2]]
    calls = []
    for keys in ({}, {"small.point_points": 0}, {"small.point_points": 1 << 30}):
        base = {"bc": "NNNNNN", "h": 1.0, "box": box, "keys": keys}
        calls.append({"name": "mgp_prolong_add_" + sfx, "args": ["c", "u", "stream"],
                      "arrays": {"c": (coarse, NO_HALO, None), "u": (shape, NO_HALO, None)}, **base})
        calls.append({"name": "mgp_residual_" + sfx, "args": [1, "u", "f", "r", "box", 1.0, None, "stream"],
                      "arrays": {n: (shape, [1] * 6, None) for n in "ufr"}, **base})
    names = [k[0][0] for rc, k in launch_recorder.record(recorder, calls)]
    marches = ["_wave" in n for n in names]
    assert marches == [not per_point] * 2 + [True] * 2 + [False] * 2, names


# levels on both sides of each line: 2^21 points, 512 blocks with at most half
# their columns, 5 * 2^24 points (the last two in FP64)
@pytest.mark.parametrize("shape,f64,f32", [
    ([65, 65, 33], "block", "block"), ([129, 129, 125], "block", "block"), ([129, 129, 129], "march", "march"),
    ([233, 303, 11], "march", "block"), ([121, 257, 31], "march", "block"), ([121, 257, 33], "block", "block"),
    ([121, 251, 31], "block", "block"), ([513, 513, 257], "march", "march"), ([483, 525, 407], "wave", "march"),
    ([511, 513, 319], "march", "march"), ([513, 513, 319], "wave", "march"), ([1025, 1025, 513], "wave", "march")])
def test_descent_kernel_by_size(recorder, shape, f64, f32):
    coarse = [(n - 1) // 2 + 1 for n in shape]
    calls = [{"name": "mgp_residual_restrict_fw_" + sfx, "bc": "NNNNNN", "h": 1.0,
              "arrays": {**{n: (shape, [1] * 6, None) for n in "ufr"}, "c": (coarse, NO_HALO, None)},
              "box": [0, shape[0], 0, shape[1], 0, shape[2]], "args": [1, "u", "f", "r", "c", "box", 1.0, "stream"]}
             for sfx in ("f64", "f32")]
    names = [k[0][0] for rc, k in launch_recorder.record(recorder, calls)]
    assert all("k_resid_fw_" + want in name for name, want in zip(names, (f64, f32))), names


# flat levels too large for blocks, on both sides of the rule: 16 rows in the box, 24
# with the correction (FP32, Dirichlet faces)
@pytest.mark.parametrize("kind,sfx,ny,bc,tile", [
    ("sweep2", "f32", 16, "DDDDDD", False), ("sweep2", "f32", 17, "DDDDDD", True),
    ("sweep2_from_zero", "f32", 16, "DDDDDD", False), ("sweep2_from_zero", "f32", 17, "DDDDDD", True),
    ("sweep2_prolong", "f32", 23, "DDDDDD", False), ("sweep2_prolong", "f32", 25, "DDDDDD", True),
    ("sweep2", "f64", 9, "DDDDDD", True), ("sweep2_prolong", "f64", 9, "DDDDDD", True),
    ("sweep2", "f32", 9, "DDNDDD", True), ("sweep2_prolong", "f32", 9, "DDDDND", True)])
def test_flat_levels_pair_by_wave_march(recorder, kind, sfx, ny, bc, tile):
    call = sweep_call(kind, sfx, [513, ny + 2, 513], bc=bc)
    ((rc, kernels),) = launch_recorder.record(recorder, [call])
    assert rc == 0 and ("k_rbgs_tile" in kernels[0][0], "_wave" in kernels[0][0]) == (tile, not tile), kernels
