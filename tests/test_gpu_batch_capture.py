"""Batch calls of more than 64 trajectories beside their staging ring: captured
into a caller's graph, which replays the captured list after the ring has been
reused, and issued faster than the device takes them."""
import ctypes

import numpy as np
import pytest

import common

pytestmark = pytest.mark.gpu


class At:
    """a device address inside a buffer"""

    def __init__(self, buf, offset):
        self.handle = ctypes.c_void_p(buf.handle.value + offset)
        self.buf = buf


class Lists:
    """A ragged list on buffers of its own, and the flat call's results for it"""

    def __init__(self, rbd, ctx, n_traj, seed):
        lengths = np.random.default_rng(seed).integers(1, 40 if n_traj < 1000 else 5, n_traj)
        self.n = int(lengths.sum())
        self.x = common.knots(self.n, seed=seed + 1)
        self.d_in = rbd.DeviceBuffer.from_array(self.x)
        self.d_out = rbd.DeviceBuffer.from_array(np.full(self.n * 105, 7.5, np.float32))
        starts = np.concatenate([[0], np.cumsum(lengths)])
        self.trajs = rbd.TrajList([(At(self.d_in, int(s) * 84), At(self.d_out, int(s) * 420), int(n))
                                   for s, n in zip(starts, lengths)])
        d_flat = rbd.DeviceBuffer(self.n * 420)
        ctx.fdgrad(self.n, self.d_in, d_flat)
        self.want = d_flat.download((self.n, 105))

    def take(self):
        """the results so far, their buffer filled anew"""
        got = self.d_out.download((self.n, 105))
        self.d_out.upload(np.full(self.n * 105, 7.5, np.float32))
        return got


def hip_ok(err, what):
    assert err == 0, f"{what}: HIP error {err}"


@pytest.mark.parametrize("n_traj", [65, 128, 129, 1000, 4097])
def test_captured_call_keeps_its_list(rbd, n_traj):
    ctx = rbd.Context(lanes_per_knot=1)                # one lane: bitwise the flat call
    b, s, H = rbd.Batch(ctx, 4097), rbd.Stream(), rbd.hip()
    mine = Lists(rbd, ctx, n_traj, 800)
    others = [Lists(rbd, ctx, k, 810 + 2 * i) for i, k in enumerate((4097, 66, 300, 65, 4096, 700))]
    print(f"captured batch of {n_traj} trajectories, {mine.n} knots", flush=True)
    for o in others[:3]:                               # slots in use when the capture begins
        b.run(o.trajs, stream=s)
    graph, execg = ctypes.c_void_p(), ctypes.c_void_p()
    hip_ok(H.hipStreamBeginCapture(s.handle, 0), "begin capture")      # 0: global mode
    try:
        b.run(mine.trajs, stream=s)
    finally:
        hip_ok(H.hipStreamEndCapture(s.handle, ctypes.byref(graph)), "end capture")
    hip_ok(H.hipGraphInstantiate(ctypes.byref(execg), graph, None, None, ctypes.c_size_t(0)), "instantiate")
    for o in others[:3]:
        s.synchronize()
        np.testing.assert_array_equal(o.take(), o.want)
    assert np.all(mine.take() == 7.5)                  # a captured call runs nothing by itself
    for turn in range(4):
        for o in others[turn:] + others[:turn]:        # more calls than the ring has slots
            b.run(o.trajs, stream=s)
        hip_ok(H.hipGraphLaunch(execg, s.handle), "launch")
        s.synchronize()
        np.testing.assert_array_equal(mine.take(), mine.want)
        for o in others:
            np.testing.assert_array_equal(o.take(), o.want)
    hip_ok(H.hipGraphExecDestroy(execg), "destroy")
    hip_ok(H.hipGraphDestroy(graph), "destroy")
    b.close()
    s.destroy()
    ctx.close()


def test_calls_ahead_of_the_device(rbd):
    """Twelve different lists issued in one go on one batch object behind a long
    call, so that the ring comes round to slots that have not been read yet;
    then the object goes while lists are pending."""
    ctx = rbd.Context(lanes_per_knot=1)
    b, s = rbd.Batch(ctx, 4097), rbd.Stream()
    lists = [Lists(rbd, ctx, (65, 4096, 200, 1000, 4097)[i % 5], 830 + 2 * i) for i in range(12)]
    n = 1 << 20
    d_in, d_out = rbd.DeviceBuffer.from_array(common.knots(n, seed=860)), rbd.DeviceBuffer(n * 420)
    print(f"twelve lists of {sum(o.n for o in lists)} knots behind {n}", flush=True)
    for turn in range(2):
        for _ in range(20):
            ctx.fdgrad(n, d_in, d_out, stream=s)
        for o in lists:
            b.run(o.trajs, stream=s)
        if turn:
            b.close()
        s.synchronize()
        for o in lists:
            np.testing.assert_array_equal(o.take(), o.want)
    s.destroy()
    ctx.close()
