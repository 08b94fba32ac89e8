"""The launches of a batch's steps, over the stand-in for the HIP runtime (host_hip.py)."""
import pytest

import host_hip


@pytest.mark.parametrize("sizes,kw,steps,want", [
    # every lattice streams from HBM: tiles, one launch a step
    ((160, 156), {}, 9, ["tile"] * 9), ((160, 156), {}, 2, ["tile"] * 2),
    # one does, three fill a group of the cache: a launch of its own each; few steps take all at once, streamed
    ((160, 90, 60, 24), {}, 9, ["tile"] * 9 + ["direct"] * 9),
    ((160, 90, 60, 24), {}, 2, ["tile"] * 2),
    # groups that the cache holds, one group that it holds
    ((110, 110, 90), {}, 8, ["direct"] * 16), ((110, 110, 90), {}, 7, ["tile"] * 7), ((60, 24), {}, 3, ["direct"] * 3),
    # nothing but D3Q19 in FP32 boxes
    ((160, 156), {"dtype": "f64"}, 2, ["direct"] * 2), ((160, 156), {"periodic": True}, 2, ["direct"] * 2),
    ((160, 156), {"q": 15}, 2, ["direct"] * 2)])
def test_tiles_by_group(sizes, kw, steps, want):
    host_hip.run("""
Ls = [cavity((n, n, n), **%r) for n in %r]
B = asl_amd.Batch(Ls)
B.step(1)
H.host_hip_forget()
B.step(%d)
got = ["tile" if "k_step_batch_tile" in l else "direct" for l in H.host_hip_launches().decode().splitlines()
       if "k_step" in l]
assert got == %r, got
""" % (kw, sizes, steps, want))


def test_one_group_by_choice_and_explicit_tiles():
    host_hip.run("""
Ls = [cavity((n, n, n)) for n in (110, 110, 90)]
B = asl_amd.Batch(Ls)
B.step(1)
for knob, value, want in ((_lib.TUNE_GROUP_MB, 0, [True] * 8), (_lib.TUNE_LDS, 0, [False] * 8),
                          (_lib.TUNE_GROUP_MB, 224, [False] * 16), (_lib.TUNE_LDS, 1, [True] * 16)):
    B.set_tuning(knob, value)
    H.host_hip_forget()
    B.step(8)
    got = ["k_step_batch_tile" in l for l in H.host_hip_launches().decode().splitlines()]
    assert got == want, (knob, value, got)
for bad in (-1, 2):
    try:
        B.set_tuning(_lib.TUNE_LDS, bad)
        raise SystemExit("taken")
    except asl_amd.ASLError:
        pass
""")
