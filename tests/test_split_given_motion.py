"""The split layout's inverse-dynamics gradient takes v, a and f as given: they
may be those of an arm on a base that moves, where link 0 has more motion than
its own joint's.  Against the FP64 oracle on the same v, a and f, in every
mapping, on the CPU build of the kernel arithmetic and on the GPU."""
import ctypes

import numpy as np
import pytest

import common

FP = ctypes.POINTER(ctypes.c_float)
S = np.array([0, 0, 1.0, 0, 0, 0])


@pytest.fixture(scope="module")
def moving_base(oracle):
    """(vol (n, 154) FP32, cdu (n, 98) FP64): base twists of +-1, base accelerations of +-3 beside gravity"""
    n, rng, model = 80, np.random.default_rng(750), common.UrdfModel()
    x = common.knots(n, seed=751).astype(np.float64)
    vol = np.zeros((n, 154))
    for i in range(n):
        q, qd, qdd = x[i, :7], x[i, 7:14], rng.uniform(-5, 5, 7)
        v, a = rng.uniform(-1, 1, 6), rng.uniform(-3, 3, 6) + np.array([0, 0, 0, 0, 0, 9.81])
        X, vs, accs, fs = [], [], [], []
        for k in range(7):
            X.append(model.transform(k, q[k]))
            v = X[k] @ v + S * qd[k]
            a = X[k] @ a + S * qdd[k] + common._crm(v) @ S * qd[k]
            inertia = model.inertia(k)
            vs.append(v)
            accs.append(a)
            fs.append(inertia @ a + common._crf(v) @ inertia @ v)
        for k in range(6, 0, -1):
            fs[k - 1] = fs[k - 1] + X[k].T @ fs[k]
        vol[i] = np.concatenate([q, qd, x[i, 14:], qdd, np.ravel(vs), np.ravel(accs), np.ravel(fs)])
    vol = vol.astype(np.float32)
    return vol, oracle.id_gradient_split(vol.astype(np.float64))


def check(got, ref):
    err = common.dqdd_block_errors(got, ref)
    assert max(float(v.max()) for v in err.values()) < 2e-5, err       # FP32: the bar of the staged variants' tests


@pytest.mark.parametrize("lanes", [0, 1])
def test_host(moving_base, lanes):
    vol, ref = moving_base
    out = np.full(ref.shape, np.nan, np.float32)
    common.hostcheck_lib().host_id_gradient_f32(len(vol), vol.ctypes.data_as(FP), out.ctypes.data_as(FP), 0, 1, lanes)
    check(out, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp32", "fp64_columns"])
@pytest.mark.parametrize("lanes", [1, 16])
def test_gpu(rbd, moving_base, precision, lanes):
    vol, ref = moving_base
    ctx = rbd.Context(precision=precision, lanes_per_knot=lanes)
    check(ctx.id_gradient_split(vol), ref)
    ctx.close()
