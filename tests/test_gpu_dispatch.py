"""GPU tests of rules that take a call to one path or another by its size:
the mapping of entry points without kernels of their own for small lane groups
(16-lane groups up to 8 knots per SIMD, one lane above), streaming or plain
stores of structure-of-arrays rows (rows that start on a line, or not) and how
a batch's list of trajectories reaches the device (kernel arguments up to 64, one staging
kernel up to 4,096, a copy and a plan kernel above)."""
import ctypes

import numpy as np
import pytest

import common

pytestmark = pytest.mark.gpu

EDGE = 32 * 256          # 8 knots per SIMD, 4 SIMDs on each of 256 compute units


class At:
    """A place in a device buffer, as the calls take it."""

    def __init__(self, buf, offset):
        self.buf, self.handle = buf, ctypes.c_void_p(buf.ptr.value + offset)


def fext_call(rbd, ctx, x, f):
    n = len(x)
    d_in, d_f = rbd.DeviceBuffer.from_array(x), rbd.DeviceBuffer.from_array(f)
    d_out = rbd.DeviceBuffer(n * 105 * 4)
    ctx.fdgrad_fext(n, d_in, d_f, 42, d_out)
    return d_out.download((n, 105))


@pytest.mark.parametrize("n,lanes", [(EDGE, 16), (EDGE + 1, 1)])
def test_mapping_without_small_groups(rbd, n, lanes):
    x = common.knots(n, seed=720)
    f = np.random.default_rng(721).uniform(-20, 20, (n, 42)).astype(np.float32)
    got = []
    for chosen in (0, lanes):
        ctx = rbd.Context(lanes_per_knot=chosen)
        print(f"fext n={n} lanes={chosen}", flush=True)
        got.append(fext_call(rbd, ctx, x, f))
        ctx.close()
    np.testing.assert_array_equal(got[0], got[1])


@pytest.mark.parametrize("n", [1, 63, 64, 65, 511, 513, 640, 131201])
def test_soa_row_alignment(rbd, n):
    """Rows aligned or not: the array-of-structures result bit for bit, and
    nothing written between the rows."""
    x = common.knots(n, seed=740)
    ctx = rbd.Context(lanes_per_knot=1)
    d_in, d_out = rbd.DeviceBuffer.from_array(x), rbd.DeviceBuffer(n * 420)
    ctx.fdgrad(n, d_in, d_out)
    want = d_out.download((n, 105))
    whole = (n + 31) // 32 * 32
    for ld, offset in ((whole, 0), (whole, 64), (whole + 16, 0), (whole + 1, 0), (n, 4)):
        print(f"soa n={n} ld={ld} offset={offset}", flush=True)
        xt = np.zeros((21, ld), np.float32)
        xt[:, :n] = x.T
        d_x = rbd.DeviceBuffer.from_array(xt)
        d_y = rbd.DeviceBuffer.from_array(np.full(105 * ld + 32, 7.5, np.float32))
        ctx.fdgrad_soa(n, d_x, ld, At(d_y, offset), ld)
        raw = d_y.download((105 * ld + 32,))
        got = raw[offset // 4:offset // 4 + 105 * ld].reshape(105, ld)
        np.testing.assert_array_equal(got[:, :n], want.T)
        assert np.all(got[:, n:] == 7.5) and np.all(raw[:offset // 4] == 7.5) and np.all(raw[offset // 4 + 105 * ld:] == 7.5)
    ctx.close()


@pytest.mark.parametrize("lanes", [0, 1])
@pytest.mark.parametrize("n_traj", [64, 65, 127, 1025, 4095, 4096, 4097])
def test_batch_list_sizes(rbd, n_traj, lanes):
    """Ragged lists with empty trajectories at the edges of the three ways,
    each run six times (more than the staging ring's slots) on one batch object with different lengths."""
    ctx = rbd.Context(lanes_per_knot=lanes)
    b = rbd.Batch(ctx, 4097)
    for turn in range(6):
        rng = np.random.default_rng(730 + turn)
        lengths = rng.integers(0, 70 if n_traj <= 127 else 8, n_traj)
        lengths[[0, n_traj - 1]] = (0, 1) if turn % 2 else (64, 0)
        total = int(lengths.sum())
        x = common.knots(total, seed=731 + turn)
        d_in, d_out = rbd.DeviceBuffer.from_array(x), rbd.DeviceBuffer.from_array(np.full(total * 105 + 8, 7.5, np.float32))
        starts = np.concatenate([[0], np.cumsum(lengths)])
        trajs = [(At(d_in, int(s) * 84), At(d_out, int(s) * 420), int(n))
                 for s, n in zip(starts, lengths)]
        print(f"batch {n_traj} trajectories, {total} knots, lanes={lanes}", flush=True)
        b.run(trajs)
        got = d_out.download((total * 105 + 8,))
        np.testing.assert_array_equal(got[total * 105:], np.full(8, 7.5, np.float32))
        flat = rbd.Context(lanes_per_knot=b.last_lanes)
        d_flat = rbd.DeviceBuffer(total * 420)
        flat.fdgrad(total, d_in, d_flat)
        want = d_flat.download((total, 105))
        if lanes:
            np.testing.assert_array_equal(got[:total * 105].reshape(total, 105), want)
        else:
            err = common.max_block_errors(got[:total * 105].reshape(total, 105), want.astype(np.float64))
            assert max(err.values()) < 1e-5, err       # lane groups: another compilation, as in the batch tests
        flat.close()
    b.close()
    ctx.close()
