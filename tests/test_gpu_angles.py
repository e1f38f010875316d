"""GPU tests of joint angles far outside a turn: the kernels reduce angles of
up to 512 (FP32) and 65,536 (FP64) one way and larger ones by integer
arithmetic.  Against the FP64 oracle on the same FP32 angles,
in every mapping, with the angles spread over a wave so that most of its lanes
stay in range."""
import numpy as np
import pytest

import common

pytestmark = pytest.mark.gpu

ANGLES = (511.9, 512.0, 512.1, 1000.0, 65535.0, 65536.0, 65537.0, 1e5, 3e7, 1.1e9, 1e15, 3e38, np.pi * 100,
          np.pi * 1e6, 1e-7)


@pytest.mark.parametrize("lanes", [1, 4, 7, 8, 16, 32])
@pytest.mark.parametrize("precision", ["fp32", "fp64_columns", "fp64"])
def test_large_angles(rbd, oracle, precision, lanes):
    n = 150
    x = common.knots(n, seed=720)
    rng = np.random.default_rng(721)
    for i in range(0, n, 3):                       # every third knot, one or all joints, either sign
        a = np.float32(ANGLES[(i // 3) % len(ANGLES)] * rng.choice([-1.0, 1.0]))
        if i % 2:
            x[i, :7] = a
        else:
            x[i, rng.integers(0, 7)] = a
    print(f"large angles {precision} lanes={lanes}", flush=True)
    ctx = rbd.Context(precision=precision, lanes_per_knot=lanes)
    err = common.max_block_errors(ctx.run_aos(x), oracle.fdgrad(x.astype(np.float64)))
    assert max(err.values()) < common.REL_TOL, err
    ctx.close()
