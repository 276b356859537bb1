"""Reading stage times waits for the evaluation they are of, not for what a
caller enqueues behind it on a stream of its own, nor for other work of the
process.  The work behind is a strict direct evaluation of about 100 ms, or the
launchers' on the null stream; the reading has 30 ms."""
import time

import numpy as np
import pytest

import gpp_inputs
import hiprt
from test_gpu_parity import problem_of

pytestmark = pytest.mark.gpu


def read(c):
    t0 = time.perf_counter()
    t = c.last_timing()
    s = c.timing_summary(4)
    return 1e3 * (time.perf_counter() - t0), t, s


def check(t, s, n):
    total = t.pop("total")
    assert all(0 < v < 50 for v in t.values()) and abs(sum(t.values()) - total) < 1e-9, (t, total)
    assert s["evaluations"] == n and 0 < s["total"] < 50


@pytest.mark.parametrize("form", ["direct", "factored-f64", "factored-ozaki-i8"])
def test_not_for_later_work_on_the_callers_stream(gpplib, form):
    import pygpp
    a = gpp_inputs.seeded_inputs(24, 1000, 50, seed=71)
    s = hiprt.Stream()
    with pygpp.Context(0) as c, pygpp.Context(0) as behind:
        behind.generate_seeded(pygpp.Problem(512, 2, 32768, 1638, 3), 1)
        behind.sigma("direct-strict")
        c.upload(problem_of(a, 2), a)
        c.sigma(form)  # the first on its own stream
        c.set_stream(s.handle)
        behind.set_stream(s.handle)
        for acht in (False, True):
            for _ in range(3):
                c.sigma_async(form, acht_n1_loc=acht)
            behind.sigma_async("direct-strict")
            behind.sigma_async("direct-strict")
            ms, t, summary = read(c)
            t0 = time.perf_counter()
            s.synchronize()
            left = 1e3 * (time.perf_counter() - t0)
            check(t, summary, 3 if acht and form != "direct" else 4)  # the direct forms' stages are the same
            assert ms < 30 and left > 50, (ms, left)
        c.set_stream(None)  # its last evaluation ran on the other stream
        check(c.last_timing(), c.timing_summary(2), 2)
        behind.set_stream(None)
    s.close()


def test_not_for_the_null_stream(ctx, gpplib):
    a = gpp_inputs.seeded_inputs(600, 24000, 1000, seed=72)
    d = {k: hiprt.DeviceArray(v) for k, v in a.items()}
    out = [hiprt.DeviceArray(np.zeros(n)) for n in (3, 3, 1200)]
    small = gpp_inputs.seeded_inputs(24, 1000, 50, seed=73)
    ctx.upload(problem_of(small, 2), small)

    def launch():
        assert gpplib.d_noFlagOCCSolver(600, 2, 1000, 24000, d["inv_igp_index"].ptr, d["wx_array"].ptr,
                                        d["wtilde_array"].ptr, d["aqsmtemp"].ptr, d["aqsntemp"].ptr,
                                        d["I_eps_array"].ptr, d["vcoul"].ptr, out[0].ptr, out[1].ptr, out[2].ptr) == 0

    launch()
    assert hiprt.rt().hipDeviceSynchronize() == 0
    ctx.sigma("factored-f64")
    launch()
    launch()
    ms, t, s = read(ctx)
    t0 = time.perf_counter()
    assert hiprt.rt().hipDeviceSynchronize() == 0
    left = 1e3 * (time.perf_counter() - t0)
    check(t, s, s["evaluations"])
    assert ms < 10 and left > 10, (ms, left)


def test_a_capture_is_left_alone(gpplib):
    """Asked for while the caller's stream is being captured, the times are
    refused; the capture goes on, and its replays note theirs."""
    import ctypes
    import pygpp
    rt = hiprt.rt()
    vp = ctypes.c_void_p
    rt.hipStreamBeginCapture.argtypes = [vp, ctypes.c_int]
    rt.hipStreamEndCapture.argtypes = [vp, ctypes.POINTER(vp)]
    rt.hipGraphInstantiate.argtypes = [ctypes.POINTER(vp), vp, vp, vp, ctypes.c_size_t]
    rt.hipGraphLaunch.argtypes = [vp, vp]
    rt.hipGraphExecDestroy.argtypes = rt.hipGraphDestroy.argtypes = [vp]
    a = gpp_inputs.seeded_inputs(24, 1000, 50, seed=74)
    s = hiprt.Stream()
    with pygpp.Context(0) as c:
        c.upload(problem_of(a, 2), a)
        c.set_stream(s.handle)
        want = c.sigma("factored-f64")
        assert rt.hipStreamBeginCapture(s.handle, 2) == 0  # relaxed: the runtime's own calls are not refused
        c.sigma_async("factored-f64")
        with pytest.raises(pygpp.GppError):
            c.last_timing()
        graph, ex = vp(), vp()
        assert rt.hipStreamEndCapture(s.handle, ctypes.byref(graph)) == 0
        assert rt.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, 0) == 0
        for _ in range(3):
            assert rt.hipGraphLaunch(ex, s.handle) == 0
            check(c.last_timing(), c.timing_summary(1), 1)
            got = c.wait()
            for k in ("achtemp", "asxtemp", "achstemp"):
                np.testing.assert_array_equal(got[k], want[k])
        rt.hipGraphExecDestroy(ex)
        rt.hipGraphDestroy(graph)
        c.set_stream(None)
    s.close()
