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


def test_kept_buffers_are_bounded():
    """Views and surface buffers stay with their lattices up to 512 MiB in all and 256 MiB each."""
    host_hip.run("""
def held(L, call):
    before = H.host_hip_used()
    call(L)
    call(L)
    return H.host_hip_used() - before


view, surface = (lambda L: L.f()), (lambda L: L.surface_force(np.ones(L.S, np.float32)))
Ls = [asl_amd.Lattice((100, 100, 100), 19, nu=0.1, periodic=True) for _ in range(10)]
for L in Ls:
    L.init_equilibrium()
    L.step(1)
kept = [held(L, view) for L in Ls]  # 81 MB each
assert kept == [76 * Ls[0].len] * 6 + [0] * 4, kept
for L in Ls[:6]:
    L.write_f(np.ones((19,) + L.S, np.float32))
used = H.host_hip_used()
del L, Ls[:6]
assert held(Ls[0], view) == 76 * Ls[0].len and held(Ls[0], surface) == 16 * Ls[0].len
big = asl_amd.Lattice((260, 260, 260), 15, nu=0.1, periodic=True)
big.init_equilibrium()
big.step(1)
assert 16 * big.len > 256 << 20 and held(big, surface) == 0
""")


def test_kept_buffers_make_room():
    """A lattice that fits only without the kept buffers of others fits; they are allocated again when needed."""
    host_hip.run("""
A = cavity((100, 100, 100))
B = cavity((60, 60, 60))
f = np.ones((19,) + A.S, np.float32)
A.step(1)
B.step(1)
want = H.host_hip_used()
A.surface_force(np.ones(A.S, np.float32))
A.write_f(f)
B.f()
assert H.host_hip_used() > want + 76 * A.len
H.host_hip_limit(H.host_hip_used() + 1000)
C = cavity((80, 80, 80))
C.step(1)
H.host_hip_limit(0)
A.f()
A.write_f(f)
B.f()
del C
H.host_hip_limit(H.host_hip_used() + 1000)
M = asl_amd.Mlp(np.zeros(_lib.CLOSURE_NPARAM, np.float32))
M.set_data(np.zeros((10000, 7), np.float32), np.zeros(10000, np.float32))
M.gradient()
""")


def test_initial_fields_that_do_not_fit():
    """The first field's buffer goes back when the second has no room."""
    host_hip.run("""
L = asl_amd.Lattice((40, 40, 40), 19, nu=0.1, periodic=True)
rho, u = np.ones(L.S, np.float32), np.zeros((3,) + L.S, np.float32)
used = H.host_hip_used()
for room in (13, 5):  # bytes a cell, of 16
    H.host_hip_limit(used + room * L.len)
    for _ in range(2):
        try:
            L.init_equilibrium(rho, u)
            raise SystemExit("it fitted")
        except asl_amd.ASLError:
            assert H.host_hip_used() == used, H.host_hip_used() - used
H.host_hip_limit(used + 17 * L.len)
L.init_equilibrium(rho, u)
assert H.host_hip_used() == used
""")
