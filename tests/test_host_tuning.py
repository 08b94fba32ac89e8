"""Launch settings and what is launched, over the stand-in for the HIP runtime (host_hip.py)."""
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
