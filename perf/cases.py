"""Performance cases of the forward-dynamics-gradient library on one GPU.

`listed()` names the calls that are timed, `draw()` gives more of the same
ranges; `prepare()` makes what a program holds before the call (inputs on the
GPU, output buffers, a context or batch object), `run()` is one pass through
the public entry points of rbdgrad, `work()` its unavoidable bytes and
operations, and `exact()` the same outputs from a plain torch restatement of
the rigid-body equations in 64 bits, straight from the robot's URDF numbers.

A case is a dict:
  kind       "full": q, qd, u -> qdd, dqdd/dq, dqdd/dqd, device buffers
             "host": the same from and to host arrays
             "batch": the same for `trajs` trajectories of 8 to 256 knots in one launch
             "minv", "wafr": the full path plus dqdd/du = Minv, in either output layout
             "fext": the full path with one set of external link forces per knot
             "ref": qdd and Minv given (the reference's timed configuration)
             "fd": forward dynamics alone, qdd and Minv
             "split", "fused": the staged pipeline, inverse-dynamics gradient
             (with v, a, f precomputed, or not) and then -Minv times it
  n          knot points (kind "batch": decided by trajs and the seed)
  layout     "aos" or "soa" (kind "full")
  precision  a name of rbdgrad.PRECISIONS
  damping, gravity   model options
  stretched  fraction of knots at the stretched-arm pose (joints 2, 4, 6 near 0)
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fast-rbd-gradients_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import rbdgrad  # noqa: E402

NQ = 7
BLOCKS = {"qdd": (0, 7), "dqdd_dq": (7, 56), "dqdd_dqd": (56, 105)}


def _case(name=None, kind="full", n=0, trajs=0, layout="aos", precision="fp32", damping=False, gravity=True,
          stretched=0.0):
    c = {"kind": kind, "n": int(n), "trajs": int(trajs), "layout": layout, "precision": precision,
         "damping": bool(damping), "gravity": bool(gravity), "stretched": float(stretched)}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one MPC trajectory of 128 knots, the reference harness's size, from host
        # memory to host memory (its "GPU compute + I/O"): latency
        _case("host_128", kind="host", n=128),
        # a few controllers' trajectories on the device in one call: latency
        _case("call_2500", n=2500),
        # 64 solvers' trajectories of uneven length in one launch
        _case("batch_64", kind="batch", trajs=64),
        # a sampling controller's knots, an odd count below one wave per SIMD of 16-knot groups
        _case("call_12007", n=12007, damping=True),
        # an ordinary throughput call of ragged size
        _case("aos_100003", n=100003, damping=True, stretched=0.1),
        # dataset and value-function sweeps: the largest calls, both layouts
        _case("soa_1048576", n=1 << 20, layout="soa", stretched=0.1),
        _case("aos_1000003", n=1000003, stretched=0.1),
        # iLQR/DDP linearisation: A and B matrices (dqdd/du = Minv) per knot
        _case("minv_262144", kind="minv", n=1 << 18, stretched=0.1),
        # contact forces on every link
        _case("fext_150001", kind="fext", n=150001),
        # the reference's timed configuration at a throughput size
        _case("ref_300007", kind="ref", n=300007, stretched=0.1),
        # the reference's staged pipeline: setup, split inverse-dynamics gradient, finish
        _case("split_200003", kind="split", n=200003, damping=True),
        # derivative columns in FP64, for callers that need the last digits
        _case("fp64col_131072", n=1 << 17, layout="soa", precision="fp64_columns", stretched=0.1),
    ]


# largest knots drawn per kind: no more bytes than the listed 2^20-knot call moves
_MOST = {"full": 1 << 20, "host": 16384, "minv": 1 << 19, "wafr": 1 << 19, "fext": 1 << 19, "ref": 1 << 19,
         "fd": 1 << 20, "split": 1 << 18, "fused": 1 << 18}
_LEAST = {"full": 100, "host": 10, "fd": 1000, "minv": 100, "wafr": 100, "fext": 100, "ref": 100, "split": 100,
          "fused": 100}


def draw(rng):
    kind = rng.choice(["full", "full", "full", "full", "host", "batch", "minv", "wafr", "fext", "ref", "fd", "split",
                       "fused"])
    damping, gravity = rng.random() < 0.5, rng.random() < 0.8
    stretched = rng.choice([0.0, 0.1])
    if kind == "batch":
        return _case(kind=kind, trajs=rng.randint(2, 400), damping=damping, gravity=gravity, stretched=stretched)
    lo, hi = math.log(_LEAST[kind]), math.log(_MOST[kind])
    n = int(round(math.exp(rng.uniform(lo, hi))))
    precision, layout = "fp32", "aos"
    if kind == "full":
        layout = rng.choice(["aos", "soa"])
        precision = rng.choice(["fp32"] * 5 + ["fp32_hw_trig", "fp64_pivot", "fp64_columns"])
        if precision == "fp64_columns":
            n = min(n, 300000 + n % 1000)
    return _case(kind=kind, n=n, layout=layout, precision=precision, damping=damping, gravity=gravity,
                 stretched=stretched)


# Floats in and out of a pass per knot, and floating-point operations (the
# non-zero ones of the recursions, rounded): what the results cannot do without.
_FLOATS = {"full": 21 + 105, "host": 21 + 105, "batch": 21 + 105, "minv": 21 + 154, "wafr": 21 + 154,
           "fext": 21 + 42 + 105, "ref": 21 + 28 + 98, "fd": 21 + 56, "split": 28 + 28 + 126 + 98 + 98,
           "fused": 28 + 28 + 98 + 98}
_FLOPS = {"fd": 4000, "ref": 8000, "split": 8000, "fused": 8000}


def work(case):
    n = case["n"] or 132 * case["trajs"]
    return {"bytes": 4 * n * _FLOATS[case["kind"]], "flops": n * _FLOPS.get(case["kind"], 11000)}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _knots(case, n, seed):
    """n knots [q | qd | u] as (n, 21): q in +-pi, qd in +-2 rad/s, u in +-50 N m."""
    dev = _device()
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed) * 7919 + 11)
    x = torch.rand((n, 21), generator=g, device=dev, dtype=torch.float32) * 2 - 1
    x[:, 0:7] *= math.pi
    x[:, 7:14] *= 2.0
    x[:, 14:21] *= 50.0
    if case["stretched"] > 0:
        m = torch.rand((n, 1), generator=g, device=dev) < case["stretched"]
        near = (torch.rand((n, 3), generator=g, device=dev) * 2 - 1) * 1e-3
        x[:, [1, 3, 5]] = torch.where(m, near, x[:, [1, 3, 5]])
    return x, g


def _lengths(case, seed):
    rng = np.random.default_rng(int(seed) + 17)
    return rng.integers(8, 257, size=case["trajs"])


def _starts(case):
    """First row of each trajectory in one buffer with room for 256 knots each, and the rows in all."""
    return np.arange(case["trajs"]) * 256, 256 * case["trajs"]


def _inputs(case, seed):
    """What a pass reads, as plain tensors: the same for prepare() and exact()."""
    kind = case["kind"]
    if kind == "batch":
        lens = _lengths(case, seed)
        start, rows = _starts(case)
        x, _ = _knots(case, rows, seed)
        return {"x": x, "lens": lens, "start": start, "rows": rows}
    n = case["n"]
    x, g = _knots(case, n, seed)
    d = {"x": x}
    if kind == "fext":
        d["fext"] = (torch.rand((n, 42), generator=g, device=x.device) * 2 - 1) * 20.0
    if kind in ("ref", "split", "fused"):
        qdd, minv = _forward_dynamics(x.double(), case)
        d["qdd"] = qdd.float()
        d["minv"] = minv.reshape(n, 49).float()      # symmetric: column-major is row-major
    return d


class _Dev:
    """A torch tensor as the binding takes device buffers."""

    def __init__(self, t):
        assert t.is_contiguous()
        self.t = t
        self.handle = ctypes.c_void_p(t.data_ptr())


def prepare(case, seed):
    kind, n = case["kind"], case["n"]
    d = _inputs(case, seed)
    x = d["x"]
    flags = (rbdgrad.VEL_DAMPING if case["damping"] else 0) | (0 if case["gravity"] else rbdgrad.NO_GRAVITY)
    s = {"kind": kind, "n": n, "ctx": rbdgrad.Context(device=0, flags=flags, precision=case["precision"])}

    def empty(*shape):
        return _Dev(torch.zeros(shape, device=x.device, dtype=torch.float32))
    if kind == "host":
        s["x"] = x.cpu().numpy()
    elif kind == "batch":
        out = empty(d["rows"], 105)
        s["in"], s["out"] = _Dev(x), out
        s["batch"] = rbdgrad.Batch(s["ctx"], case["trajs"])
        s["trajs"] = rbdgrad.TrajList([(_Dev(x[a:a + k]), _Dev(out.t[a:a + k]), int(k))
                                       for a, k in zip(d["start"].tolist(), d["lens"].tolist())])
    elif kind == "full" and case["layout"] == "soa":
        s["soa"], s["in"], s["out"] = True, _Dev(x.t().contiguous()), empty(105, n)
    elif kind in ("full", "minv", "wafr", "fext", "fd"):
        s["in"] = _Dev(x)
        if kind == "fext":
            s["fext"] = _Dev(d["fext"])
        if kind in ("minv", "fd"):
            s["minv"] = empty(n, 49)
        if kind in ("wafr", "fd"):
            s["qdd"] = empty(n, 7)
        s["out"] = empty(n, 147 if kind == "wafr" else 105)
    elif kind == "ref":
        s["vol"] = _Dev(torch.cat([x, d["qdd"], d["minv"]], 1).contiguous())
        s["out"] = empty(n, 98)
    else:
        s["minv"], s["cdu"], s["out"] = _Dev(d["minv"]), empty(n, 98), empty(n, 98)
        if kind == "split":
            s["vol"] = empty(n, 154)
            s["vol"].t[:, :21] = x
            s["vol"].t[:, 21:28] = d["qdd"]
        else:
            s["vol"] = _Dev(torch.cat([x, d["qdd"]], 1).contiguous())
    if kind != "host":
        s["result"] = _outputs(s)
    return s


def _blocks(t, dim):
    return {k: t.narrow(dim, a, b - a) for k, (a, b) in BLOCKS.items()}


def _pair(t):
    return {"dq": t[:, 0:49], "dqd": t[:, 49:98]}


def _outputs(s):
    """The output buffers of a state as named blocks, views made once."""
    kind = s["kind"]
    o = s["out"].t if "out" in s else None
    if kind == "wafr":
        return {"qdd": s["qdd"].t, "dqdd_dq": o[:, 0:49], "dqdd_dqd": o[:, 49:98], "minv": o[:, 98:147]}
    if kind == "fd":
        return {"qdd": s["qdd"].t, "minv": s["minv"].t}
    if kind == "ref":
        return _pair(o)
    if kind in ("split", "fused"):
        r = {"dtau": _pair(s["cdu"].t), "dqdd": _pair(o)}
        if kind == "split":
            v = s["vol"].t
            r.update(v=v[:, 28:70], a=v[:, 70:112], f=v[:, 112:154])
        return r
    r = _blocks(o, 0 if "soa" in s else 1)
    if kind == "minv":
        r["minv"] = s["minv"].t
    return r


def run(s):
    kind, n, ctx = s["kind"], s["n"], s["ctx"]
    if kind == "host":
        out = ctx.fdgrad_host(s["x"])
        return {k: out[:, a:b] for k, (a, b) in BLOCKS.items()}
    if kind == "full":
        if "soa" in s:
            ctx.fdgrad_soa(n, s["in"], n, s["out"], n)
        else:
            ctx.fdgrad(n, s["in"], s["out"])
    elif kind == "batch":
        s["batch"].run(s["trajs"])
    elif kind == "minv":
        ctx.fdgrad_minv(n, s["in"], s["out"], s["minv"])
    elif kind == "wafr":
        ctx.fdgrad_wafr(n, s["in"], s["qdd"], s["out"])
    elif kind == "fext":
        ctx.fdgrad_fext(n, s["in"], s["fext"], 42, s["out"])
    elif kind == "ref":
        ctx.dynamics_gradient_kernel(n, s["out"], s["vol"])
    elif kind == "fd":
        ctx.forward_dynamics_dev(n, s["in"], s["qdd"], s["minv"])
    else:
        if kind == "split":
            ctx.gradient_setup_split_dev(n, s["vol"])
            ctx.dynamics_gradient_kernel_split(n, s["cdu"], s["vol"])
        else:
            ctx.dynamics_gradient_kernel_fused(n, s["cdu"], s["vol"])
        ctx.gradient_finish_dev(n, s["out"], s["cdu"], s["minv"])
    return s["result"]


# ---------------------------------------------------------------------------
# The same in 64 bits: recursive Newton-Euler with its derivatives by the
# product rule, the mass matrix from unit accelerations, Gauss-Jordan for its
# inverse.  Vectors are (6 or 3, columns, knots) tensors, [angular; linear].
# ---------------------------------------------------------------------------
# KUKA iiwa 14 URDF: joint origin xyz and rpy; link mass, centre of mass,
# inertia about it (ixx, ixy, ixz, iyy, iyz, izz)
_HALF = math.pi / 2
_URDF = [
    ((0, 0, 0.1575), (0, 0, 0), 5.76, (0, -0.03, 0.12), (0.121, 0, 0, 0.116, -0.021, 0.0175)),
    ((0, 0, 0.2025), (_HALF, 0, math.pi), 6.35, (0.0003, 0.059, 0.042),
     (0.0638, 0.0001, 8e-05, 0.0416, 0.0157, 0.0331)),
    ((0, 0.2045, 0), (_HALF, 0, math.pi), 3.5, (0, 0.03, 0.13), (0.0873, 0, 0, 0.083, 0.014, 0.0108)),
    ((0, 0, 0.2155), (_HALF, 0, 0), 3.5, (0, 0.067, 0.034), (0.0368, 0, 0, 0.02045, 0.008, 0.02171)),
    ((0, 0.1845, 0), (-_HALF, math.pi, 0), 3.5, (0.0001, 0.021, 0.076),
     (0.0318, 7e-06, 2.7e-05, 0.028916, 0.005586, 0.006)),
    ((0, 0, 0.2155), (_HALF, 0, 0), 1.8, (0, 0.0006, 0.0004), (0.0049, 0, 0, 0.0047, 0, 0.0036)),
    ((0, 0.081, 0), (-_HALF, math.pi, 0), 1.2, (0, 0, 0.02), (0.0055, 0, 0, 0.0055, 0, 0.005)),
]
_GRAVITY = 9.81


def _skew(v):
    return np.array([[0, -v[2], v[1]], [v[2], 0, -v[0]], [-v[1], v[0], 0]], dtype=np.float64)


def _rpy(r, p, y):
    cr, sr, cp, sp, cy, sy = math.cos(r), math.sin(r), math.cos(p), math.sin(p), math.cos(y), math.sin(y)
    return (np.array([[cy, -sy, 0], [sy, cy, 0], [0, 0, 1]]) @ np.array([[cp, 0, sp], [0, 1, 0], [-sp, 0, cp]]) @
            np.array([[1, 0, 0], [0, cr, -sr], [0, sr, cr]]))


def _inertia(k):
    _, _, m, com, (xx, xy, xz, yy, yz, zz) = _URDF[k]
    c = _skew(com)
    out = np.zeros((6, 6))
    out[:3, :3] = np.array([[xx, xy, xz], [xy, yy, yz], [xz, yz, zz]]) + m * c @ c.T
    out[:3, 3:], out[3:, :3], out[3:, 3:] = m * c, m * c.T, m * np.eye(3)
    return out


def _cross(a, b):
    return torch.stack([a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]])


def _crm(a, b):       # motion cross product a x b
    return torch.cat([_cross(a[:3], b[:3]), _cross(a[3:], b[:3]) + _cross(a[:3], b[3:])])


def _crf(a, b):       # force cross product a x* b
    return torch.cat([_cross(a[:3], b[:3]) + _cross(a[3:], b[3:]), _cross(a[:3], b[3:])])


def _const(m, x):     # a constant matrix times (rows, columns, knots)
    return torch.stack([sum((float(m[i, j]) * x[j] for j in range(m.shape[1]) if m[i, j] != 0.0),
                            torch.zeros_like(x[0])) for i in range(m.shape[0])])


def _joint(k, q):
    """Motion and force transforms of joint k at angle q (knots,): parent to child, and transposed."""
    xyz, rpy = _URDF[k][0], _URDF[k][1]
    f = np.round(_rpy(*rpy).T, 12)
    r = np.array(xyz, dtype=np.float64)
    c, s = torch.cos(q), torch.sin(q)

    def rot(x):
        y = _const(f, x)
        return torch.stack([c * y[0] + s * y[1], c * y[1] - s * y[0], y[2]])

    def rot_t(x):
        return _const(f.T, torch.stack([c * x[0] - s * x[1], s * x[0] + c * x[1], x[2]]))

    def motion(x):
        return torch.cat([rot(x[:3]), rot(x[3:] - _const(_skew(r), x[:3]))])

    def force_t(x):
        lin = rot_t(x[3:])
        return torch.cat([rot_t(x[:3]) + _const(_skew(r), lin), lin])
    return motion, force_t


def _unit(x):
    s = torch.zeros_like(x)
    s[2] = 1.0
    return s


def _rnea(q, qd, qdd, gravity, fext=None, columns=False):
    """q, qd (7, knots); qdd (7, columns, knots).  Returns per link v, a, f (after
    the backward pass) and, with columns, dtau/d(q, qd) as (7, 14, knots)."""
    m, n = qdd.shape[1], q.shape[1]
    z = torch.zeros((6, m, n), dtype=q.dtype, device=q.device)
    v, a = z, z.clone()
    a[5] = gravity
    dv = da = torch.zeros((6, 14, n), dtype=q.dtype, device=q.device)
    s1 = _unit(z[:, :1])
    joints, vs, as_, fs, dfs = [], [], [], [], []
    for k in range(NQ):
        motion, force_t = _joint(k, q[k])
        joints.append(force_t)
        inertia = _inertia(k)
        tv, ta = motion(v), motion(a)
        v = tv + s1 * qd[k]
        a = ta + s1 * qdd[k] + _crm(v, s1 * qd[k])
        iv = _const(inertia, v)
        f = _const(inertia, a) + _crf(v, iv)
        if fext is not None:
            f = f - fext[6 * k:6 * k + 6].unsqueeze(1)
        if columns:
            dv, da = motion(dv), motion(da)
            dv[:, k] -= _crm(s1, tv)[:, 0]
            dv[2, 7 + k] += 1.0
            da[:, k] -= _crm(s1, ta)[:, 0]
            da = da + _crm(dv, s1 * qd[k])
            da[:, 7 + k] += _crm(v, s1)[:, 0]
            dfs.append(_const(inertia, da) + _crf(dv, iv) + _crf(v, _const(inertia, dv)))
        vs.append(v)
        as_.append(a)
        fs.append(f)
    dtau = [None] * NQ
    for k in range(NQ - 1, -1, -1):
        if columns:
            dtau[k] = dfs[k][2]
        if k > 0:
            if columns:
                g = dfs[k].clone()
                g[:, k] += _crf(s1, fs[k])[:, 0]
                dfs[k - 1] = dfs[k - 1] + joints[k](g)
            fs[k - 1] = fs[k - 1] + joints[k](fs[k])
    return vs, as_, fs, torch.stack(dtau) if columns else None


def _invert(mm):
    """(7, 7, knots) symmetric positive definite, by Gauss-Jordan without pivoting."""
    n = mm.shape[2]
    eye = torch.eye(NQ, dtype=mm.dtype, device=mm.device).unsqueeze(2).expand(NQ, NQ, n)
    w = torch.cat([mm, eye], 1)
    for k in range(NQ):
        row = w[k] / w[k, k]
        w = w - w[:, k].unsqueeze(1) * row.unsqueeze(0)
        w[k] = row
    inv = w[:, NQ:]
    return 0.5 * (inv + inv.transpose(0, 1))


def _chunks(n):
    step = 1 << 16
    return [(a, min(n, a + step)) for a in range(0, n, step)]


def _fd_chunk(x, case, fext=None):
    """qdd (7, knots) and Minv (7, 7, knots) of x (21, knots)."""
    q, qd, u = x[0:7], x[7:14], x[14:21]
    n = x.shape[1]
    grav = _GRAVITY if case["gravity"] else 0.0
    eye = torch.eye(NQ, dtype=x.dtype, device=x.device).unsqueeze(2).expand(NQ, NQ, n)
    mass = torch.stack([f[2] for f in _rnea(q, torch.zeros_like(qd), eye, 0.0)[2]])
    bias = torch.stack([f[2, 0] for f in _rnea(q, qd, torch.zeros_like(q).unsqueeze(1), grav, fext)[2]])
    if case["damping"]:
        bias = bias + 0.5 * qd
    minv = _invert(mass)
    return (minv * (u - bias).unsqueeze(0)).sum(1), minv


def _forward_dynamics(x, case):
    """qdd (n, 7) and Minv (n, 7, 7) of x (n, 21), 64 bits."""
    parts = [_fd_chunk(x[a:b].t().contiguous(), case) for a, b in _chunks(len(x))]
    return torch.cat([p[0].t() for p in parts]), torch.cat([p[1].permute(2, 0, 1) for p in parts])


def _dtau_chunk(x, qdd, case, fext=None):
    grav = _GRAVITY if case["gravity"] else 0.0
    v, a, f, dtau = _rnea(x[0:7], x[7:14], qdd.unsqueeze(1), grav, fext, columns=True)
    if case["damping"]:
        dtau = dtau.clone()
        for k in range(NQ):
            dtau[k, 7 + k] += 0.5
    return v, a, f, dtau


def _columns(m):
    """(7, columns, knots) as (knots, 7 * columns), column-major."""
    return m.permute(2, 1, 0).reshape(m.shape[2], -1)


def _minus_times(minv, dtau):
    return -sum(minv[:, k].unsqueeze(1) * dtau[k].unsqueeze(0) for k in range(NQ))


def exact(case, seed):
    kind = case["kind"]
    d = _inputs(case, seed)
    x, parts = d["x"].double(), []
    for a, b in _chunks(len(x)):
        xc = x[a:b].t().contiguous()
        fe = d["fext"][a:b].double().t().contiguous() if kind == "fext" else None
        if kind in ("ref", "split", "fused"):
            qdd = d["qdd"][a:b].double().t()
            minv = d["minv"][a:b].double().reshape(-1, 7, 7).permute(1, 2, 0)
            minv = torch.triu(minv.permute(2, 0, 1)).permute(1, 2, 0)
            minv = minv + torch.tril(minv.permute(2, 1, 0), -1).permute(1, 2, 0)
        else:
            qdd, minv = _fd_chunk(xc, case, fe)
        r = {}
        if kind == "fd":
            r["qdd"], r["minv"] = qdd.t(), _columns(minv)
        else:
            v, acc, f, dtau = _dtau_chunk(xc, qdd, case, fe)
            g = _columns(_minus_times(minv, dtau))
            if kind in ("split", "fused"):
                t = _columns(dtau)
                r["dtau"], r["dqdd"] = _pair(t), _pair(g)
                if kind == "split":
                    r["v"], r["a"], r["f"] = (torch.cat([y[:, 0] for y in w]).t() for w in (v, acc, f))
            elif kind == "ref":
                r = _pair(g)
            else:
                r = {"qdd": qdd.t(), "dqdd_dq": g[:, 0:49], "dqdd_dqd": g[:, 49:98]}
                if kind in ("minv", "wafr"):
                    r["minv"] = _columns(minv)
        parts.append(r)

    def join(ps):
        if isinstance(ps[0], dict):
            return {k: join([p[k] for p in ps]) for k in ps[0]}
        return torch.cat(ps)
    r = join(parts)
    if kind == "batch":
        keep = torch.zeros((d["rows"], 1), dtype=torch.float64, device=x.device)
        for a, k in zip(d["start"].tolist(), d["lens"].tolist()):
            keep[a:a + k] = 1.0
        r = {k: v * keep for k, v in r.items()}
    if kind == "full" and case["layout"] == "soa":
        r = {k: v.t() for k, v in r.items()}
    return r
