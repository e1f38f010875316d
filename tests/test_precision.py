"""CPU check of how exact the kernel arithmetic is, not only that it holds the
bar: errors against the FP64 oracle in the 2-norm over many knots, per output
block, for every knot-to-lane mapping and both robots (the iiwa and the
synthetic arm, whose joint frames are dense).

The bounds are what the articulated-body recursion for Minv itself, with
-Minv dtau by a product, measures in the same build on the same knots: the
factored mass matrix has to be no less exact than the recursion it replaces."""
import ctypes
import os

import numpy as np
import pytest

import common

FP = ctypes.POINTER(ctypes.c_float)
N = 8000
# 2-norm of the error over that of the result: qdd, dqdd/dq, dqdd/dqd; Minv
RECURSION = {
    ("iiwa", "fp32"): (6.33e-8, 2.35e-7, 1.03e-6),
    ("iiwa", "fp64_pivot"): (6.13e-8, 2.29e-7, 1.03e-6),
    ("iiwa", "fp64_columns"): (6.33e-8, 2.14e-7, 2.24e-7),
    ("iiwa", "minv"): 4.11e-8,
    ("arm7", "fp32"): (1.09e-7, 5.17e-7, 7.32e-7),
    ("arm7", "fp64_pivot"): (1.04e-7, 5.63e-7, 7.53e-7),
    ("arm7", "fp64_columns"): (1.09e-7, 4.84e-7, 3.23e-7),
    ("arm7", "minv"): 9.73e-8,
}
PRECISIONS = {"fp32": 0, "fp64_pivot": 1, "fp64_columns": 2}


@pytest.fixture(scope="module", params=["iiwa", "arm7"])
def robot(request, oracle):
    """(name, host library, knots, FP64 results, FP64 Minv of the first 1,000)"""
    x = common.knots(N, seed=730)
    x64 = x.astype(np.float64)

    def results():
        minv = np.array([oracle.fd(k[:7], k[7:14], k[14:21])[1] for k in x64[:1000]])
        return oracle.fdgrad(x64, threads=8), minv
    if request.param == "iiwa":
        return ("iiwa", common.hostcheck_lib(), x) + results()
    with oracle.using_model(*common.generate_model(os.path.join(common.GOLDEN, "synthetic_arm7.urdf"), "arm7")):
        ref = results()
    return ("arm7", common.hostcheck_lib("arm7"), x) + ref


def norm_error(got, ref):
    return float(np.linalg.norm(got.astype(np.float64) - ref) / np.linalg.norm(ref))


def mappings(host, x, out, prec):
    a, o, n = x.ctypes.data_as(FP), out.ctypes.data_as(FP), ctypes.c_long(len(x))
    yield "one lane", lambda: host.host_fdgrad_f32(n, a, o, 0, prec, 0)
    yield "16 lanes", lambda: host.host_fdgrad_f32(n, a, o, 0, prec, 1)
    yield "two waves", lambda: host.host_fdgrad_two_wave_f32(n, a, o, 0, prec)
    for lanes in (4, 7, 8):
        yield f"{lanes} lanes", lambda lanes=lanes: host.host_fdgrad_group_f32(n, a, o, 0, prec, lanes)


@pytest.mark.parametrize("precision", PRECISIONS)
def test_blocks_no_less_exact_than_the_recursion(robot, precision):
    name, host, x, ref, _ = robot
    out = np.empty((N, 105), np.float32)
    for mapping, call in mappings(host, x, out, PRECISIONS[precision]):
        call()
        err = {b: norm_error(out[:, sl], ref[:, sl]) for b, sl in common.BLOCKS.items()}
        for block, bound in zip(common.BLOCKS, RECURSION[name, precision]):
            assert err[block] <= bound, (mapping, block, err)


def test_minv_no_less_exact_than_the_recursion(robot):
    name, host, x, _, ref = robot
    qdd, minv = np.empty((1000, 7), np.float32), np.empty((1000, 49), np.float32)
    host.host_fd_f32(1000, x.ctypes.data_as(FP), qdd.ctypes.data_as(FP), minv.ctypes.data_as(FP), 0)
    assert norm_error(minv.reshape(1000, 7, 7), ref) <= RECURSION[name, "minv"]
