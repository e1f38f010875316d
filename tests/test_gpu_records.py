"""GPU tests of the one-lane kernels' record paths (outputs through LDS in
halves of 32 records, inputs of the split and finish stages as whole lines):
sizes around a half and a whole block of 64 knots, and buffers that are 16-,
8- and 4-byte aligned, which take different copy loops.

Each output must equal bit for bit the same knots in one aligned call of all
knots (a knot's arithmetic does not depend on its place), that call must hold
the bar against the FP64 oracle, and nothing may be written past the last
record."""
import ctypes

import numpy as np
import pytest

import common

pytestmark = pytest.mark.gpu

N = 191
SIZES = (1, 31, 32, 33, 63, 64, 65, 96, 128, N)
GUARD = 8          # floats after the last record that must stay as they were


class At:
    """A device buffer starting `offset` bytes into a 16-byte-aligned allocation."""

    def __init__(self, rbd, a, offset):
        raw = np.zeros(a.size + 4, dtype=np.float32)
        raw[offset // 4:offset // 4 + a.size] = a.ravel()
        self.buf = rbd.DeviceBuffer.from_array(raw)
        self.offset, self.shape = offset, a.shape
        self.handle = ctypes.c_void_p(self.buf.ptr.value + offset)

    def read(self):
        raw = self.buf.download((self.buf.nbytes // 4,))
        return raw[self.offset // 4:self.offset // 4 + int(np.prod(self.shape))].reshape(self.shape)


@pytest.fixture(scope="module")
def data(oracle):
    x = common.knots(N, seed=710, near_singular_frac=0.1)
    x64 = x.astype(np.float64)
    fext = np.random.default_rng(711).uniform(-20, 20, (N, 42)).astype(np.float32)
    ref = oracle.fdgrad(x64)
    minv = np.array([oracle.fd(k[:7], k[7:14], k[14:21])[1].T.reshape(49) for k in x64])
    vol28 = np.concatenate([x, ref[:, :7].astype(np.float32)], axis=1)
    vaf = oracle.vaf(np.concatenate([vol28.astype(np.float64), np.zeros((N, 126))], axis=1)).astype(np.float32)
    cdu = oracle.id_gradient(vol28.astype(np.float64))
    minv32, cdu32 = minv.astype(np.float32), cdu.astype(np.float32)
    vol77 = np.concatenate([vol28, minv32], axis=1)
    return {
        "aos": ((x,), (105,), (ref,)),
        "minv": ((x,), (105, 49), (ref, minv)),
        "wafr": ((x,), (7, 147), (ref[:, :7], np.concatenate([ref[:, 7:], minv], axis=1))),
        "fext": ((x, fext), (105,), (oracle.fdgrad(x64, fext=fext.astype(np.float64)),)),
        "ref": ((vol77,), (98,), (oracle.fdgrad_refmode(vol77.astype(np.float64)),)),
        "fused": ((vol28,), (98,), (cdu,)),
        "split": ((vaf,), (98,), (oracle.id_gradient_split(vaf.astype(np.float64)),)),
        "finish": ((cdu32, minv32), (98,), (oracle.finish(minv32.astype(np.float64), cdu32.astype(np.float64)),)),
    }


def call(ctx, name, n, ins, outs):
    if name == "aos":
        ctx.fdgrad(n, ins[0], outs[0])
    elif name == "minv":
        ctx.fdgrad_minv(n, ins[0], outs[0], outs[1])
    elif name == "wafr":
        ctx.fdgrad_wafr(n, ins[0], outs[0], outs[1])
    elif name == "fext":
        ctx.fdgrad_fext(n, ins[0], ins[1], 42, outs[0])
    elif name == "ref":
        ctx.dynamics_gradient_kernel(n, outs[0], ins[0])
    elif name == "fused":
        ctx.dynamics_gradient_kernel_fused(n, outs[0], ins[0])
    elif name == "split":
        ctx.dynamics_gradient_kernel_split(n, outs[0], ins[0])
    else:
        ctx.gradient_finish_dev(n, outs[0], ins[0], ins[1])


def run(rbd, ctx, name, n, inputs, widths, offset):
    ins = [At(rbd, a[:n], offset) for a in inputs]
    outs = [At(rbd, np.full(n * w + GUARD, 7.5, np.float32), offset) for w in widths]
    call(ctx, name, n, ins, outs)
    res = []
    for o, w in zip(outs, widths):
        a = o.read()
        np.testing.assert_array_equal(a[n * w:], np.full(GUARD, 7.5, np.float32))
        res.append(a[:n * w].reshape(n, w))
    return res


@pytest.mark.parametrize("precision", ["fp32", "fp64_columns"])
@pytest.mark.parametrize("name", ["aos", "minv", "wafr", "fext", "ref", "fused", "split", "finish"])
def test_records_at_block_edges(rbd, data, name, precision):
    inputs, widths, refs = data[name]
    ctx = rbd.Context(precision=precision, lanes_per_knot=1)
    print(f"records {name} {precision}", flush=True)
    whole = run(rbd, ctx, name, N, inputs, widths, 0)
    for got, ref in zip(whole, refs):
        # per knot and 49-column block (or the whole of a shorter output), the bar of all parity tests
        for a in range(0 if ref.shape[1] % 49 == 0 else ref.shape[1] % 49, ref.shape[1], 49):
            e = np.abs(got[:, a:a + 49] - ref[:, a:a + 49]).max(1) / np.maximum(np.abs(ref[:, a:a + 49]).max(1), 1e-6)
            assert e.max() < common.REL_TOL, (a, e.max())
        if ref.shape[1] % 49:
            a = ref.shape[1] % 49
            e = np.abs(got[:, :a] - ref[:, :a]).max(1) / np.maximum(np.abs(ref[:, :a]).max(1), 1e-6)
            assert e.max() < common.REL_TOL, e.max()
    for n in SIZES:
        for offset in (0, 4, 8):
            for got, ref in zip(run(rbd, ctx, name, n, inputs, widths, offset), whole):
                np.testing.assert_array_equal(got, ref[:n], err_msg=f"{name} n={n} offset={offset}")
    ctx.close()
