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
