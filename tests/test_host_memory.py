"""What the library does when device memory runs out: host side only, over the
stand-in for the HIP runtime (host_hip.py)."""
import host_hip


def test_a_failed_allocation_is_reported_once():
    """... by the call that needed it, not by the next launch, whose step would be taken for not done."""
    host_hip.run("""
L = cavity((8, 8, 8))
L.step(1)
for call in (lambda: asl_amd.Lattice((64, 64, 64), 19, nu=0.1), L.f, lambda: L.surface_force(np.ones(L.S, np.float32))):
    H.host_hip_limit(H.host_hip_used() + 1000)
    try:
        call()
        raise SystemExit("it fitted")
    except asl_amd.ASLError as e:
        assert "memory" in str(e), e
    launches()
    L.step(2)
    assert len(launches()) == 2
    H.host_hip_limit(0)
""")


def test_training_after_a_batch_that_did_not_fit():
    """The sums of a smaller batch get a buffer again (the kernel would write through a null pointer)."""
    host_hip.run("""
M = asl_amd.Mlp(np.zeros(_lib.CLOSURE_NPARAM, np.float32))
n = 1 << 20
M.set_data(np.zeros((n, 7), np.float32), np.zeros(n, np.float32))
M.gradient(0, 256)
held = H.host_hip_used()
for call in (lambda: M.gradient(0, n), lambda: M.train(1, n, 1e-3)):
    H.host_hip_limit(held + 100000)
    try:
        call()
        raise SystemExit("the large batch fitted")
    except asl_amd.ASLError:
        pass
    M.gradient(0, 256)
    assert H.host_hip_used() == held, (H.host_hip_used(), held)
    H.host_hip_limit(0)
M.gradient(0, n)
assert H.host_hip_used() > held + 100000
""")


def test_a_batch_keeps_its_setting_when_the_new_table_does_not_fit():
    """Launches of another workgroup size than the table's would read it past its end."""
    host_hip.run("""
Ls = [cavity((24, 24, 24)) for _ in range(3)]
B = asl_amd.Batch(Ls)
B.step(3)
before = launches("k_step_batch")
for knob, value in ((_lib.TUNE_BLOCK, 256), (_lib.TUNE_LDS, 1), (_lib.TUNE_GROUP_MB, 1)):
    H.host_hip_limit(H.host_hip_used() + 1)
    try:
        B.set_tuning(knob, value)
        raise SystemExit("it fitted")
    except asl_amd.ASLError:
        pass
    B.step(2)
    assert launches("k_step_batch") == before, value
H.host_hip_limit(0)
B.set_tuning(_lib.TUNE_BLOCK, 256)
B.step(1)
assert launches("k_step_batch")[0] == (3 * 24**3 // 256, 256)
""")
