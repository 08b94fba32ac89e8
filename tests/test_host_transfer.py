"""Which way host transfers go, over the stand-in for the HIP runtime (host_hip.py)."""
import host_hip


def test_memory_the_runtime_knows_is_copied_directly():
    """Reads into pinned memory and writes from it take no detour through the ring's buffers."""
    host_hip.run("""
L = cavity((60, 60, 60))
view = L.q * L.len * 4
buf = ctypes.c_void_p()
assert H.hipHostMalloc(ctypes.byref(buf), ctypes.c_size_t(view), 0) == 0
H.host_hip_forget()
_lib.call("aslhip_read_velocity", L.h, buf)
assert copies() == [("p", "d", 12 * L.len)]
_lib.call("aslhip_read_f", L.h, buf)
assert copies() == [("p", "d", view)]
_lib.call("aslhip_write_f", L.h, buf)
assert copies() == [("d", "p", view)]
""")


def test_small_transfers():
    """To the device without the ring below 14 MiB, to the host through one buffer up to 2 MiB; all bytes arrive."""
    host_hip.run("""
MB = 1 << 20
M = asl_amd.Mlp(np.arange(_lib.CLOSURE_NPARAM, dtype=np.float32))
H.host_hip_forget()
assert np.array_equal(M.params(), np.arange(_lib.CLOSURE_NPARAM))
assert copies() == [("p", "d", 4 * _lib.CLOSURE_NPARAM)]
for n, direct in ((3, True), (14 * MB // 28 - 1, True), (14 * MB // 28 + 1, False)):
    x = np.zeros((n, 7), np.float32)
    M.set_data(x, np.zeros(n, np.float32))
    got = [c for c in copies() if c[0] == "d"]
    assert sum(c[2] for c in got) == 32 * n
    assert (got[0] == ("d", "h", 28 * n)) == direct, (n, got[:3])
""")


def test_a_lattice_of_another_device_than_the_current_one():
    """The ring's events belong to a device: transfers on another one's stream do without them."""
    host_hip.run("""
L = asl_amd.Lattice((80, 80, 80), 19, nu=0.05, periodic=True)
L.init_equilibrium()
M = asl_amd.Mlp(np.zeros(_lib.CLOSURE_NPARAM, np.float32))
f = np.ones((19,) + L.S, np.float32)
assert f.nbytes >= 14 << 20
L.velocity()
for device in (1, 0, 1):
    H.host_hip_device(device)
    L.write_f(f)
    L.velocity()
    L.rho()
""")


def test_no_memory_for_the_copy_threads():
    """The caller copies by itself, and no exception leaves the C entry."""
    host_hip.run("""
L = asl_amd.Lattice((80, 80, 80), 19, nu=0.05, periodic=True)
L.init_equilibrium()
out = np.zeros(3 * L.len, np.float32)
lib = _lib.load_library()
p = ctypes.c_void_p(out.ctypes.data)
assert lib.aslhip_read_velocity(L.h, p) == 0  # the ring is there
want = out.copy()
out[:] = 7
H.host_hip_no_new(1)
r = lib.aslhip_read_velocity(L.h, p)
H.host_hip_no_new(0)
assert r == 0 and want.tobytes() == out.tobytes()
""")


def test_small_reads_wait_for_an_event_after_many_launches():
    host_hip.run("""
L = cavity((16, 16, 16))
L.step(1)


def waits(read):
    before = H.host_hip_event_waits()
    read()
    return H.host_hip_event_waits() - before


for steps, want in ((0, 0), (3, 0), (6, 0), (7, 1), (0, 1), (1, 1)):
    L.step(steps)
    assert waits(L.rho) == want, (steps, want)
L.synchronize()
assert waits(L.velocity) == 0
""")
