"""The CFL minimum of host-driven steps beside captured work of the same
method: a caller's graph of the device-side timestep may be replayed between
any two host-driven calls and leaves its own minimum behind."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

G = 3


def _ev():
    import enzoe_vlct as ev
    return ev


def _state(n, seed, mhd, speed):
    rng = np.random.default_rng(seed)
    m = (n + 2 * G,) * 3
    a = {"density": 1.0 + rng.random(m)}
    for c in "xyz":
        a["velocity_" + c] = speed * rng.standard_normal(m)
    b2 = 0.0
    if mhd:
        for ax, c in zip((2, 1, 0), "xyz"):
            shape = list(m)
            shape[ax] += 1
            a["bfieldi_" + c] = np.full(shape, 0.3)
            a["bfield_" + c] = np.full(m, 0.3)
            b2 = b2 + a["bfield_" + c] ** 2
    a["total_energy"] = 1.5 / a["density"] + 0.5 * sum(
        a["velocity_" + c] ** 2 for c in "xyz") + 0.5 * b2 / a["density"]
    return a


def _hip(ev):
    h = ev.hip()
    vp = ctypes.c_void_p
    h.hipStreamBeginCapture.argtypes = [vp, ctypes.c_int]
    h.hipStreamEndCapture.argtypes = [vp, ctypes.POINTER(vp)]
    h.hipGraphInstantiate.argtypes = [ctypes.POINTER(vp), vp, vp, ctypes.c_char_p,
                                      ctypes.c_size_t]
    h.hipGraphLaunch.argtypes = [vp, vp]
    h.hipGraphExecDestroy.argtypes = [vp]
    h.hipGraphDestroy.argtypes = [vp]
    return h


@pytest.mark.parametrize("mhd,n", [(True, 20), (False, 18), (False, 44)])
def test_host_driven_dt_is_its_own_beside_a_replayed_graph(mhd, n):
    """Eager calls, then between host-driven steps replays of a captured
    timestep over a block of fast flow: every dt equals that of a method that
    never saw a graph."""
    ev = _ev()
    h = _hip(ev)
    m, fresh = (ev.VlctMethod(mhd=mhd, riemann="hlld" if mhd else "hllc", reconstruct="plm",
                              theta=1.5, courant=0.3) for _ in range(2))
    slow, other, fast = (ev.DeviceBlock(n + 2 * G, n + 2 * G, n + 2 * G, G, (1.0 / n,) * 3,
                                        mhd=mhd) for _ in range(3))
    for b in (slow, other):
        b.upload(_state(n, 1, mhd, 0.2))
    fast.upload(_state(n, 2, mhd, 9.0))
    state = ev.DeviceBuffer(2 * 8)
    dp = ctypes.POINTER(ctypes.c_double)

    def device_dt(stream):
        base = state.ptr.value
        ev.check(ev.lib().enzoe_vlct_timestep_device(
            m.handle, m._blocks([fast]), 1, ctypes.cast(base, dp), 1e9,
            ctypes.cast(base + 8, dp), 1, stream), "enzoe_vlct_timestep_device")

    ev.to_device(state.ptr.value, np.zeros(2))
    device_dt(None)  # uploads the table
    ev.synchronize()
    stream = ctypes.c_void_p()
    graph, execu = ctypes.c_void_p(), ctypes.c_void_p()
    ev.hip_check(h.hipStreamCreate(ctypes.byref(stream)), "hipStreamCreate")
    ev.hip_check(h.hipStreamBeginCapture(stream, 2), "hipStreamBeginCapture")
    device_dt(stream)
    ev.hip_check(h.hipStreamEndCapture(stream, ctypes.byref(graph)), "hipStreamEndCapture")
    ev.hip_check(h.hipGraphInstantiate(ctypes.byref(execu), graph, None, None, 0),
                 "hipGraphInstantiate")
    dt_fast = fresh.timestep([fast])
    dt = fresh.timestep([other])
    assert dt_fast < 0.5 * dt
    for i in range(4):
        want = fresh.compute_timestep([other], 0.5 * dt)
        assert m.compute_timestep([slow], 0.5 * dt) == want
        for _ in range(i):
            ev.hip_check(h.hipGraphLaunch(execu, stream), "hipGraphLaunch")
            ev.hip_check(h.hipStreamSynchronize(stream), "hipStreamSynchronize")
            assert ev.from_device(state.ptr.value, (2,))[1] == dt_fast
        dt = want
    h.hipGraphExecDestroy(execu)
    h.hipGraphDestroy(graph)
    h.hipStreamDestroy(stream)
    a, b = slow.download(), other.download()
    for k in a:
        assert np.array_equal(a[k], b[k]), k
