"""Launch settings and what is launched, over the stand-in for the HIP runtime (host_hip.py)."""
import pytest

import host_hip


def test_sweeps_follow_the_workgroup_size():
    """... also on lattices whose single steps run tiles or runs of cells, which do not show it."""
    host_hip.run("""
for knob, value in ((_lib.TUNE_LDS, 1), (_lib.TUNE_CPL, 2), (_lib.TUNE_CPL, 4), (_lib.TUNE_LDS, 0)):
    L = cavity((64, 40, 40))
    L.set_tuning(knob, value)
    L.set_tuning(_lib.TUNE_SWEEP_KB, 2048)
    for block in (512, 1024, 256, 64, 512):
        L.set_tuning(_lib.TUNE_BLOCK, block)
        L.step(1)
        launches()
        L.step(8)
        got = launches()
        assert len(got) > 8 and {b for _, b in got} == {block}, (knob, value, block, set(got))
""")


@pytest.mark.parametrize("size,kw,lanes", [
    ((1, 1, 5), {}, 128), ((32, 32, 32), {}, 128), ((33, 32, 32), {}, 256), ((64, 32, 32), {}, 256),
    ((65, 32, 32), {}, 512), ((33, 32, 32), {"q": 27, "dtype": "f64"}, 256),
    ((65, 64, 64), {"q": 27, "dtype": "f64", "periodic": True}, 256), ((32, 32, 32), {"q": 15}, 128)])
def test_values_of_what_runs(size, kw, lanes):
    """Small lattices take the smallest workgroup that gives every CU at most one, D3Q27 in FP64 256 lanes; the
    values say so, the settings (512 and 4) until somebody chooses stand for it."""
    host_hip.run("""
L = cavity(%r, **%r)
assert L.tuning() == (512, 4)
L.step(1)
launches()
for choose in (None, 512, 1024, 64):
    if choose:
        L.set_tuning(_lib.TUNE_BLOCK, choose)
        L.set_tuning(_lib.TUNE_XCD_REMAP, 3)
    L.step(2)
    (grid, block), again = launches()
    assert again == (grid, block) and L.tuning_value(_lib.TUNE_BLOCK) == block, (choose, block)
    most = 512 if (L.q, L.host_dtype) == (27, np.float64) else 1024
    assert block == (min(choose, most) if choose else %d), (choose, block)
    assert L.tuning_value(_lib.TUNE_XCD_REMAP) == (3 if choose else max(1, grid // 8))
    if choose:
        assert L.tuning() == (min(choose, most), 3)
""" % (size, kw, lanes))


def test_values_of_tiles_and_runs_of_cells():
    host_hip.run("""
for knob, value, want in ((_lib.TUNE_LDS, 1, 256), (_lib.TUNE_LDS, 2, 128), (_lib.TUNE_CPL, 2, 128), (_lib.TUNE_CPL, 4, 128)):
    L = cavity((16, 16, 16))
    L.set_tuning(knob, value)
    L.step(2)
    launches()
    L.step(2)
    got = [b for _, b in launches()]
    assert L.tuning_value(_lib.TUNE_BLOCK) == want and want in got, (knob, value, got)
    L.set_tuning(_lib.TUNE_BLOCK, 1024)
    L.step(2)
    got = [b for _, b in launches()]
    assert L.tuning_value(_lib.TUNE_BLOCK) in got and L.tuning()[0] == L.tuning_value(_lib.TUNE_BLOCK), (knob, value, got)
""")


def test_autotune_keeps_the_small_workgroups():
    """16^3 runs fastest with the 128 lanes that no fixed candidate has: it stays automatic."""
    host_hip.run("""
for k in (TILE, RUN):
    cost(k, 100.0)
for block, ms in ((128, 1.0), (256, 1.1), (512, 1.3), (1024, 2.0)):
    cost(DIRECT, ms * block / 128, block)
L = cavity((16, 16, 16))
L.step(2)
assert L.autotune(10) == (512, 4) == L.tuning()
launches()
L.step(1)
assert launches() == [(32, 128)]
cost(DIRECT, 0.1, 1024)
assert L.autotune(10)[0] == 1024
launches()
L.step(1)
assert launches() == [(4, 1024)] and L.tuning_value(_lib.TUNE_BLOCK) == 1024
""")


def test_autotune_keeps_the_sweeps():
    """A box whose single steps are fastest with tiles and whose runs are faster in sweeps (their launches of few
    workgroups find the cache): runs still sweep, single steps still take tiles."""
    host_hip.run("""
L = cavity((256, 182, 180))
assert 19 * 4 * L.len > 560 << 20
whole = 256 * 182 * 180 // 512
cost(DIRECT, 1.1, 512)
cost(DIRECT, 1.3, 256)
cost(DIRECT, 2.6, 1024)
cost(TILE, 0.5)
for block in (256, 512, 1024):
    cost(DIRECT, 0.9 * block / 512, block, whole)
L.step(2)
L.autotune(20)
launches()
L.step(20)
got = launches()
assert len(got) > 20, got
L.step(1)
assert launches() == [(len(range(0, 182 * 182, 256)) * 256, 256)]
assert L.tuning_value(_lib.TUNE_LDS) == 1 and L.tuning_value(_lib.TUNE_SWEEP_KB) == -1
cost(TILE, 0.1)  # tiles better than any sweep: chosen for runs too
L.autotune(20)
launches()
L.step(20)
assert len(launches()) == 20
""")


def test_autotune_steps_as_often_as_before():
    """The trial steps advance the simulation: 60 candidates on a small box, 24 on a periodic lattice."""
    host_hip.run("""
for kw, n in ((dict(), 6 + 6 * 3 + 2 * 6 * 3), (dict(periodic=True), 6 * 3)):
    L = cavity((24, 20, 22), **kw)
    L.step(2)
    launches()
    L.autotune(9)
    assert len(launches()) == 10 * n
""")


def test_large_fp64_d3q27_lattices():
    """Whole-lattice launches that stream from HBM take 512 lanes, sweeps and smaller lattices 256."""
    host_hip.run("""
for n, lanes in ((180, 256), (210, 512)):
    L = cavity((n, n, n), 27, dtype="f64", periodic=True)
    L.step(2)
    launches()
    L.step(2)
    assert {b for _, b in launches()} == {lanes} and L.tuning_value(_lib.TUNE_BLOCK) == lanes
    L.step(8)
    got = launches()
    assert len(got) > 8 and {b for _, b in got} == {256}
    B = asl_amd.Batch([L])
    B.step(1)
    assert {b for _, b in launches("k_step_batch")} == {lanes}
""")
