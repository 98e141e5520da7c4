"""The work that programs have this framework do, as cases that can be timed and
compared: time steps of single lattices (plain and binary fluid, FP64 and
FP32-shifted storage, the fused step and the reference's call sequence, with
and without Lees-Edwards planes), replica ensembles, and the learned surrogate
(one convolution layer forward and backward, network inference, a training
step, and a jump with its correction steps).

listed() gives the named cases, draw(rng) further ones of the same ranges,
prepare(case, seed) what a program holds before the call, run(state) one pass
through the public entry points, work(case) what a pass cannot do without,
tolerance(case) how far another correct implementation may be off, and
exact(case, seed) the same outputs in 64 bits from plain torch.
"""

import ctypes
import math
import random

import numpy as np
import torch

import ludwig_amd as L
from ludwig_amd import ensemble as E
from ludwig_amd import surrogate as S
from ludwig_amd import surrogate_study

# The free energy and mobility of the binary-fluid workloads (the explicit
# Cahn-Hilliard step is stable at M = 0.25 for |phi| <= 1.1).
FE = dict(a=-0.0625, b=0.0625, kappa=0.04, mobility=0.25)
ETA = (1.0 - 0.5)/3.0                     # tau = 1
METHODS = {"stress": L.FORCE_STRESS_DIVERGENCE, "gradmu": L.FORCE_PHI_GRADMU}


# ---------------------------------------------------------------------------
# Cases


def listed():
    return [
        # The plain fluid on a small box (the 32^3, tau = 0.8 workload): a
        # launch every few microseconds, so launch latency counts.
        dict(name="single_32_f64", kind="single", nx=32, ny=32, nz=32, bits=64, tau=0.8, steps=20),
        # The regression and error-study size of the binary fluid, with the
        # 27-point gradient of the reference's own regression input.
        dict(name="binary_64_f64_27pt", kind="binary", nx=64, ny=64, nz=64, bits=64, order=1, stencil=27,
             method="stress", conserve=0, steps=20),
        # The benchmark's workload: spinodal decomposition at 128^3 in FP64.
        dict(name="binary_128_f64", kind="binary", nx=128, ny=128, nz=128, bits=64, order=1, stencil=7,
             method="stress", conserve=0, steps=10),
        # The large production lattice in both storage precisions.
        dict(name="binary_256_f64", kind="binary", nx=256, ny=256, nz=256, bits=64, order=1, stencil=7,
             method="stress", conserve=0, steps=5),
        dict(name="binary_256_f32", kind="binary", nx=256, ny=256, nz=256, bits=32, order=1, stencil=7,
             method="stress", conserve=0, steps=5),
        # A host program that makes the reference's calls one by one, on a box
        # with no power of two in it: third-order advection, phi grad mu.
        dict(name="staged_100x84x76_f64", kind="staged", nx=100, ny=84, nz=76, bits=64, order=3, stencil=7,
             method="gradmu", conserve=0, steps=5),
        # Steady shear between two Lees-Edwards planes at the benchmark's size.
        dict(name="shear_128_f64", kind="shear", nx=128, ny=128, nz=128, bits=64, order=1, stencil=7,
             planes=2, uy=0.05, steps=10),
        # Data generation: uneven replicas advanced together, with snapshots.
        dict(name="ensemble_24_f32", kind="ensemble", replicas=24, smallest=48, largest=96, mix=2026, bits=32,
             order=1, steps=10),
        # One convolution layer, forward and backward, on a ragged lattice.
        dict(name="layer_48_to_64", kind="layer", batch=3, nx=36, ny=44, nz=52, cin=48, cout=64),
        # Network inference at full size.
        dict(name="unet_8x64", kind="unet", batch=8, nx=64, ny=64, nz=64),
        # One optimiser step of the training run.
        dict(name="train_4x64", kind="train", batch=4, nx=64, ny=64, nz=64),
        # The surrogate in use: a jump of every replica, then 20 plain steps.
        dict(name="jump_16x64_f32", kind="jump", replicas=16, n=64, steps=20),
    ]


def _side(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["single", "binary", "binary", "binary", "staged", "shear", "ensemble", "layer", "layer",
                       "unet", "train", "jump"])
    if kind in ("single", "binary", "staged"):
        lo, hi = 24, {"single": 128, "binary": 224, "staged": 144}[kind]
        c = dict(kind=kind, nx=_side(rng, lo, hi), ny=_side(rng, lo, hi), nz=_side(rng, lo, hi),
                 bits=rng.choice([64, 64, 32]))
        if kind == "single":
            c.update(tau=rng.choice([0.8, 1.0]))
        else:
            c.update(order=rng.choice([1, 1, 2, 3, 4]), stencil=rng.choice([7, 7, 27]),
                     method=rng.choice(["stress", "stress", "gradmu"]), conserve=rng.choice([0, 0, 1]))
        c.update(steps=max(3, min(20, 10*128**3//(c["nx"]*c["ny"]*c["nz"]))))
        return c
    if kind == "shear":
        planes = rng.choice([1, 2, 4])
        return dict(kind=kind, nx=planes*_side(rng, 24, 128)//2*2, ny=_side(rng, 24, 144), nz=_side(rng, 24, 144),
                    bits=64, order=rng.choice([1, 2, 3]), stencil=rng.choice([7, 27]), planes=planes,
                    uy=rng.choice([0.02, 0.05]), steps=5)
    if kind == "ensemble":
        return dict(kind=kind, replicas=rng.randint(4, 40), smallest=rng.choice([32, 48]), largest=96,
                    mix=rng.randrange(1 << 20), bits=rng.choice([32, 32, 64]), order=rng.choice([1, 1, 2, 3]), steps=5)
    if kind == "layer":
        return dict(kind=kind, batch=rng.randint(1, 4), nx=_side(rng, 8, 64), ny=_side(rng, 8, 64),
                    nz=_side(rng, 8, 64), cin=16*rng.randint(1, 10), cout=16*rng.randint(1, 6))
    if kind == "jump":
        return dict(kind=kind, replicas=rng.randint(2, 20), n=rng.choice([48, 64, 80, 96]), steps=rng.choice([10, 20]))
    hi = 96 if kind == "unet" else 64
    return dict(kind=kind, batch=rng.randint(1, 6 if kind == "unet" else 4), nx=8*max(2, _side(rng, 16, hi)//8),
                ny=8*max(2, _side(rng, 16, hi)//8), nz=8*max(2, _side(rng, 16, hi)//8))


# ---------------------------------------------------------------------------
# Device memory as tensors


class _Span:
    """A span of the framework's device memory."""

    def __init__(self, ptr, shape, typestr):
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=typestr, data=(int(ptr), False), version=3)


def _view(ptr, shape, typestr, owner):
    """A tensor over the owner's device memory; the owner lives as long as
    the tensor does."""
    t = torch.as_tensor(_Span(ptr, shape, typestr), device="cuda")
    t.owner = owner
    return t


def _array(d, shape=None):
    """A DeviceArray as a tensor."""
    return _view(d.ptr, shape or (d.n,), d.dtype.str, d)


def _vp(t):
    return ctypes.c_void_p(t.data_ptr())


# ---------------------------------------------------------------------------
# Inputs


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _smooth(shape, g, scale):
    """A random field on the periodic box, unit RMS, with structure on
    `scale` sites."""
    w = torch.randn(shape, generator=g, device="cuda", dtype=torch.float64)
    k2 = sum((torch.fft.fftfreq(n, device="cuda", dtype=torch.float64)*2*math.pi).reshape(
        [-1 if b == a else 1 for b in range(3)])**2 for a, n in enumerate(shape))
    w = torch.fft.ifftn(torch.fft.fftn(w)*torch.exp(-0.5*k2*scale**2)).real
    return w/w.square().mean().sqrt()


def _noise(shape, g, amp):
    """The spinodal start: uniform noise of +-amp (values FP32 can hold)."""
    return ((torch.rand(shape, generator=g, device="cuda", dtype=torch.float64) - 0.5)*2*amp).float().double()


def _domains(shape, g, phi0=0.0):
    """phi of a phase-separated mixture: domains of phi = +-1 some ten sites
    across, and the slow smooth flow that goes with them."""
    phi = torch.tanh(2.0*_smooth(shape, g, 3.0) + 2.0*phi0)
    u = torch.stack([2.0e-3*_smooth(shape, g, 3.0) for _ in range(3)])
    return phi.float(), u.float()


def _shape(case):
    return case["nx"], case["ny"], case["nz"]


def _fluid(case, seed):
    shape, bits = _shape(case), case["bits"]
    g = _generator(seed)
    if case["kind"] == "single":
        b = L.SingleFluid(shape, tau=case["tau"], precision=bits, fatal=True)
    else:
        more = dict(le_planes=case["planes"], le_uy=case["uy"]) if case["kind"] == "shear" else {}
        b = L.BinaryFluid(shape, tau=1.0, precision=bits, order=case["order"], stencil=case["stencil"],
                          force_method=METHODS[case.get("method", "stress")], conserve=case.get("conserve", 0),
                          fatal=True, **FE, **more)
        b.set_phi(_noise(shape, g, 0.05).cpu().numpy())
    if case["kind"] == "shear":
        b.le_init_shear_profile()
    else:
        f = _distributions(b)
        if case["kind"] == "single":
            u = _noise((3,) + tuple(shape), g, 1.0e-3)
            u = u - u.mean(dim=(1, 2, 3), keepdim=True)
            f0 = _equilibrium(torch.ones(shape, device="cuda", dtype=torch.float64), u)
        else:
            f0 = _W.reshape(19, 1, 1, 1).cuda().expand((19,) + tuple(shape))
        f.copy_(f0 - (_W.reshape(19, 1, 1, 1).cuda() if bits == 32 else 0.0))
    torch.cuda.synchronize()
    return b


def _distributions(b):
    p, es, sh = ctypes.c_void_p(), ctypes.c_int(), ctypes.c_int()
    L._ck(L.lib().ldw_lb_device_f(b.lb, ctypes.byref(p), ctypes.byref(es), ctypes.byref(sh)), "ldw_lb_device_f")
    return _view(p.value, (19,) + b.shape, "<f%d" % es.value, b)


def _fields(b, binary):
    """The lattice's state where it lies in device memory."""
    lib, es = L.lib(), ctypes.c_int()
    rho, u, force, phi = (ctypes.c_void_p() for _ in range(4))
    L._ck(lib.ldw_hydro_device(b.hydro, ctypes.byref(rho), ctypes.byref(u), ctypes.byref(force), ctypes.byref(es)),
          "ldw_hydro_device")
    t = "<f%d" % es.value
    out = dict(f=_distributions(b), rho=_view(rho.value, b.shape, t, b), u=_view(u.value, (3,) + b.shape, t, b))
    if binary:
        L._ck(lib.ldw_field_device(b.phi, ctypes.byref(phi), ctypes.byref(es)), "ldw_field_device")
        out.update(phi=_view(phi.value, b.shape, t, b), force=_view(force.value, (3,) + b.shape, t, b))
    return out


def _bind():
    lib, vp, ip = L.lib(), ctypes.POINTER(ctypes.c_void_p), ctypes.POINTER(ctypes.c_int)
    lib.ldw_lb_device_f.argtypes = [ctypes.c_void_p, vp, ip, ip]
    lib.ldw_field_device.argtypes = [ctypes.c_void_p, vp, ip]
    lib.ldw_hydro_device.argtypes = [ctypes.c_void_p, vp, vp, vp, ip]


def _specs(case, seed):
    """Replicas with phi0, kappa and M drawn from the seed; the sizes belong
    to the case."""
    if case["kind"] == "jump":
        sizes = [case["n"]]*case["replicas"]
    else:
        r = random.Random(case["mix"])
        sizes = [r.choice(range(case["smallest"], case["largest"] + 1, 16)) for _ in range(case["replicas"])]
    drawn = E.draw_replicas(len(sizes), seed)
    return [E.replica(n, s.seed, phi0=s.phi0, kappa=s.kappa, mobility=s.mobility) for n, s in zip(sizes, drawn)]


def _replica_states(case, seed, specs):
    g = _generator(seed + 1)
    got = []
    for s in specs:
        shape = (s.nx, s.ny, s.nz)
        if case["kind"] == "jump":
            phi, u = _domains(shape, g, s.phi0)
        else:
            phi = (s.phi0 + _noise(shape, g, 0.05)).float()
            u = torch.stack([1.0e-4*_smooth(shape, g, 2.0) for _ in range(3)]).float()
        got.append(torch.cat([phi[None], u]).contiguous())
    return got


def _network():
    net = S.UNet(seed=0)
    norm = net.load(surrogate_study.WEIGHTS)
    return net, norm


def _samples(case, seed):
    """(state now, state one jump later, parameters) of every sample."""
    g = _generator(seed)
    rng = random.Random(seed)
    got = []
    for _ in range(case["batch"]):
        s = E.replica(_shape(case), 1, phi0=rng.uniform(-0.3, 0.3), kappa=rng.uniform(0.02, 0.08),
                      mobility=rng.uniform(0.1, 0.5))
        phi, u = _domains(_shape(case), g, s.phi0)
        now = torch.cat([phi[None], u]).contiguous()
        change = 0.1*torch.stack([_smooth(_shape(case), g, 3.0) for _ in range(4)])
        change[1:] *= 5.0e-3
        got.append((now, (now + change.float()).contiguous(), s))
    return got


def _layer_inputs(case, seed):
    g = _generator(seed)
    ci, co = case["cin"], case["cout"]
    n = case["batch"]*case["nx"]*case["ny"]*case["nz"]
    x = torch.nn.functional.silu(torch.randn((n, ci), generator=g, device="cuda")).bfloat16()
    w = (torch.randn((27, co, ci), generator=g, device="cuda")*math.sqrt(2.0/(27*ci))).bfloat16()
    bias = 0.1*torch.randn(co, generator=g, device="cuda")
    da = 1.0e-3*torch.randn((n, co), generator=g, device="cuda")
    return n, x, w, bias, da


# ---------------------------------------------------------------------------
# prepare


def prepare(case, seed):
    _bind()
    kind = case["kind"]
    s = dict(case=case)
    if kind in ("single", "binary", "staged", "shear"):
        s["b"] = _fluid(case, seed)
    elif kind in ("ensemble", "jump"):
        specs = _specs(case, seed)
        e = E.Ensemble(specs, precision=case.get("bits", 32), order=case.get("order", 1), fatal=True)
        e.tune(reps=2)
        states = _replica_states(case, seed, specs)
        torch.cuda.synchronize()
        for r, st in enumerate(states):
            e.load_device(r, st.data_ptr())
        torch.cuda.synchronize()
        snap = torch.empty(4*e.nsite, device="cuda")
        where = np.cumsum([0] + [16*int(np.prod(sh)) for sh in e.shapes])
        s.update(e=e, snap=snap, where=[snap.data_ptr() + int(o) for o in where[:-1]])
        if kind == "jump":
            net, norm = _network()
            s.update(jumper=S.Jumper(net, norm, conserve=True))
    elif kind == "unet":
        net, norm = _network()
        ns = int(np.prod(_shape(case)))
        x = L.DeviceArray(case["batch"]*ns*S.CIN, np.uint16)
        data = _samples(case, seed)
        torch.cuda.synchronize()
        for j, (now, _, spec) in enumerate(data):
            S.encode(now.data_ptr(), ns, spec, norm, x, j*ns)
        L.lib().ldw_device_synchronize()
        s.update(net=net, x=x)
    elif kind == "train":
        net, norm = _network()
        data = _samples(case, seed)
        s.update(net=net, trainer=S.Trainer(net, norm, batch=case["batch"]), data=data,
                 items=[(a.data_ptr(), b.data_ptr(), q) for a, b, q in data])
    else:
        n, x, w, bias, da = _layer_inputs(case, seed)
        ci, co = case["cin"], case["cout"]
        f32 = lambda *sh: torch.empty(sh, device="cuda")                           # noqa: E731
        b16 = lambda *sh: torch.empty(sh, device="cuda", dtype=torch.bfloat16)     # noqa: E731
        s.update(n=n, x=x, w=w, bias=bias, da=da, wd=b16(27, ci, co), z=f32(n, co), a=b16(n, co), dz=f32(n, co),
                 dzb=b16(n, co), dw=f32(27, co, ci), db=f32(co), dx=f32(n, ci))
        w32 = w.float()
        torch.cuda.synchronize()
        L._ck(L.lib().ldw_conv3d_weights_prep(_vp(w32), None, _vp(s["wd"]), ci, co), "ldw_conv3d_weights_prep")
    torch.cuda.synchronize()
    L.lib().ldw_device_synchronize()
    return s


# ---------------------------------------------------------------------------
# run


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind in ("single", "binary", "shear"):
        s["b"].step(c["steps"])
        return _fields(s["b"], kind != "single")
    if kind == "staged":
        b = s["b"]
        for _ in range(c["steps"]):
            b.f_zero()
            b.force_stage()
            b.cahn_hilliard_stage()
            b.u_zero()
            b.collide(b.fe)
            b.propagate()
        return _fields(b, True)
    if kind in ("ensemble", "jump"):
        e = s["e"]
        if kind == "jump":
            s["jumper"].jump(e)
        e.step(c["steps"])
        for r, p in enumerate(s["where"]):
            e.snapshot_device(r, p)
        return s["snap"]
    if kind == "unet":
        y = s["net"].forward(s["x"], c["batch"], _shape(c), keep=False)
        return _array(y, (y.n//S.COUT, S.COUT))
    if kind == "train":
        net = s["net"]
        loss = s["trainer"].step_arrays(s["items"], _shape(c), 1.0e-5)
        return dict(loss=loss, g=_array(net.g), w=_array(net.w), m=_array(net.m), v=_array(net.v))
    lib = L.lib()
    at = (c["batch"],) + _shape(c) + (c["cin"], c["cout"])
    L._ck(lib.ldw_conv3d_fwd_silu(_vp(s["x"]), _vp(s["w"]), _vp(s["bias"]), _vp(s["z"]), _vp(s["a"]), *at), "forward")
    L._ck(lib.ldw_nn_silu_bwd(_vp(s["z"]), _vp(s["da"]), _vp(s["dz"]), _vp(s["dzb"]), s["n"]*c["cout"]), "silu")
    L._ck(lib.ldw_conv3d_bwd_weight(_vp(s["x"]), _vp(s["dzb"]), _vp(s["dw"]), *at, 0), "weight gradient")
    L._ck(lib.ldw_nn_bias_grad(_vp(s["dz"]), _vp(s["db"]), s["n"], c["cout"], 0), "bias gradient")
    L._ck(lib.ldw_conv3d_bwd_data(_vp(s["dzb"]), _vp(s["wd"]), _vp(s["dx"]), *at, 0), "data gradient")
    return {k: s[k] for k in ("z", "a", "dz", "dzb", "dw", "db", "dx")}


# ---------------------------------------------------------------------------
# work and tolerance


def _sites(case):
    if case["kind"] in ("ensemble", "jump"):
        return sum(q.nx*q.ny*q.nz for q in _specs(case, 1))
    return case.get("batch", 1)*int(np.prod(_shape(case)))


def _network_flops(npos):
    return sum(2*27*ci*co*npos/8**S.LEVEL[name] for name, ci, co in S.LAYERS)


def work(case):
    """Bytes and operations of a pass.  A time step reads and writes the 19
    distributions, phi and u and writes rho once per site; about 250 operations
    per site collide it and 230 form the force and the fluxes."""
    kind, n = case["kind"], _sites(case)
    es = case.get("bits", 32)//8
    per = {"single": 19 + 19 + 4, "shear": 47 + 3, "staged": 47 + 6}.get(kind, 47)
    ops = 250 if kind == "single" else 480
    if kind in ("single", "binary", "staged", "shear"):
        return dict(bytes=float(es*per*n*case["steps"]), flops=float(ops*n*case["steps"]))
    if kind == "ensemble":
        return dict(bytes=float(es*per*n*case["steps"] + (4*es + 16)*n), flops=float(ops*n*case["steps"]))
    params = sum(27*ci*co + co for _, ci, co in S.LAYERS)
    if kind == "jump":
        return dict(bytes=float(es*per*n*case["steps"] + 4*(4 + 4 + 19 + 8)*n),
                    flops=float(ops*n*case["steps"]) + _network_flops(n))
    if kind == "unet":
        return dict(bytes=float(2*S.CIN*n + 4*S.COUT*n + 2*params), flops=_network_flops(n))
    if kind == "train":
        return dict(bytes=float(32*n + 28*params), flops=3*_network_flops(n))
    ci, co = case["cin"], case["cout"]
    return dict(bytes=float(n*(2*ci + 4*ci + (4 + 2 + 4 + 4 + 2)*co) + 27*ci*co*8), flops=float(3*2*27*ci*co*n))


def tolerance(case):
    kind = case["kind"]
    if kind in ("single", "binary", "staged", "shear", "ensemble"):
        # about four times what the same steps in plain torch, summed in
        # another order, are off: u is small, so the round-off of the
        # distributions weighs most in it (1e-11 and 4e-7)
        return {"rel": 5.0e-11, "max": 2.0e-9} if case["bits"] == 64 else {"rel": 2.0e-6, "max": 1.0e-4}
    # BF16 operands and activations, FP32 sums: 2e-3 a layer and for the whole
    # network's output, 5e-4 for its gradients and for a state after a jump
    return {"layer": {"rel": 7.0e-3, "max": 0.3}, "unet": {"rel": 7.0e-3, "max": 0.3},
            "train": {"rel": 3.0e-3, "max": 0.5}, "jump": {"rel": 2.0e-3, "max": 0.1}}[kind]


# ---------------------------------------------------------------------------
# The same in 64 bits

_C = torch.tensor([[0, 0, 0], [1, 1, 0], [1, 0, 1], [1, 0, 0], [1, 0, -1], [1, -1, 0], [0, 1, 1], [0, 1, 0],
                   [0, 1, -1], [0, 0, 1], [0, 0, -1], [0, -1, 1], [0, -1, 0], [0, -1, -1], [-1, 1, 0], [-1, 0, 1],
                   [-1, 0, 0], [-1, 0, -1], [-1, -1, 0]])
_W = torch.tensor([{0: 12.0, 1: 2.0, 2: 1.0}[int(c.abs().sum())] for c in _C], dtype=torch.float64)/36.0


def _equilibrium(rho, u):
    uu = (u*u).sum(0)
    out = []
    for c, w in zip(_C.tolist(), _W.tolist()):
        cu = c[0]*u[0] + c[1]*u[1] + c[2]*u[2]
        out.append(w*rho*(1.0 + 3.0*cu + 4.5*cu*cu - 1.5*uu))
    return torch.stack(out)


def _collide(f, force, eta):
    """Post-collision distributions, density and velocity."""
    r = 1.0/(0.5 + 3.0*eta)
    j = [sum(c[a]*f[p] for p, c in enumerate(_C.tolist()) if c[a]) for a in range(3)]
    rho = f.sum(0)
    u = [(j[a] + 0.5*force[a])/rho for a in range(3)]
    s, eq = {}, {}
    for a in range(3):
        for b in range(a, 3):
            s[a, b] = sum(c[a]*c[b]*f[p] for p, c in enumerate(_C.tolist()) if c[a]*c[b]) - (rho/3.0 if a == b else 0.0)
            eq[a, b] = rho*u[a]*u[b]
    ts, te = (sum(q[a, a] for a in range(3)) for q in (s, eq))
    new = {}
    for a, b in s:
        d = (ts/3.0, te/3.0) if a == b else (0.0, 0.0)
        v = s[a, b] - d[0]
        v = v - r*(v - (eq[a, b] - d[1]))
        if a == b:
            v = v + (ts - r*(ts - te))/3.0
        new[a, b] = v + (2.0 - r)*(u[a]*force[b] + force[a]*u[b])
    out = torch.empty_like(f)
    for p, (c, w) in enumerate(zip(_C.tolist(), _W.tolist())):
        v = rho + sum(3.0*c[a]*(j[a] + force[a]) for a in range(3) if c[a])
        for a, b in new:
            k = (1.0 if a == b else 2.0)*(c[a]*c[b] - (1.0/3.0 if a == b else 0.0))
            if k:
                v = v + 4.5*k*new[a, b]
        out[p] = w*v
    return out, rho, torch.stack(u)


def _at(a, axis, k):
    """a at the site k further along the axis."""
    return torch.roll(a, -k, dims=axis) if k else a


def _gradient(phi, stencil):
    if stencil == 7:
        g = [0.5*(_at(phi, a, 1) - _at(phi, a, -1)) for a in range(3)]
        return g, sum(_at(phi, a, 1) + _at(phi, a, -1) for a in range(3)) - 6.0*phi
    cube = phi
    for a in range(3):
        cube = _at(cube, a, -1) + cube + _at(cube, a, 1)
    g = []
    for a in range(3):
        d = _at(phi, a, 1) - _at(phi, a, -1)
        for b in range(3):
            if b != a:
                d = _at(d, b, -1) + d + _at(d, b, 1)
        g.append(d/18.0)
    return g, (cube - 27.0*phi)/9.0


def _face_flux(phi, uf, axis, order):
    """uf phi on the upper face of each site along the axis."""
    p0, p1 = phi, _at(phi, axis, 1)
    if order == 1:
        return uf*torch.where(uf < 0, p1, p0)
    if order == 2:
        return uf*0.5*(p0 + p1)
    pm, p2 = _at(phi, axis, -1), _at(phi, axis, 2)
    if order == 3:
        a1, a2, a3 = -0.213933, 0.927865, 0.286067
        return uf*torch.where(uf < 0, a1*p2 + a2*p1 + a3*p0, a1*pm + a2*p0 + a3*p1)
    return uf*((9.0/16.0)*(p0 + p1) - (1.0/16.0)*(pm + p2))


def _binary_steps(phi, f, rho, u, steps, fe, order, stencil, method, streamed):
    """`steps` binary-fluid steps; f is post-collision where `streamed`."""
    a, b, kappa, mobility = fe
    force = None
    for _ in range(steps):
        g, lap = _gradient(phi, stencil)
        mu = a*phi + b*phi**3 - kappa*lap
        if method == "stress":
            p0 = 0.5*a*phi**2 + 0.75*b*phi**4 - kappa*phi*lap - 0.5*kappa*sum(q*q for q in g)
            force = []
            for i in range(3):
                v = 0.0
                for k in range(3):
                    s = kappa*g[i]*g[k] + (p0 if i == k else 0.0)
                    v = v - 0.5*(_at(s, k, 1) - _at(s, k, -1))
                force.append(v)
        else:
            force = [-phi*0.5*(_at(mu, k, 1) - _at(mu, k, -1)) for k in range(3)]
        change = 0.0
        for k in range(3):
            q = -mobility*(_at(mu, k, 1) - mu)
            if u is not None:
                q = q + _face_flux(phi, 0.5*(u[k] + _at(u[k], k, 1)), k, order)
            change = change + q - _at(q, k, -1)
        phi = phi - change
        if streamed:
            f = torch.stack([torch.roll(f[p], c, dims=(0, 1, 2)) for p, c in enumerate(_C.tolist())])
        f, rho, u = _collide(f, force, ETA)
        streamed = True
    return phi, f, rho, u, None if force is None else torch.stack(force)


def _exact_fluid(case, seed):
    shape = _shape(case)
    g = _generator(seed)
    if case["kind"] == "single":
        u = _noise((3,) + shape, g, 1.0e-3)
        u = u - u.mean(dim=(1, 2, 3), keepdim=True)
        f = _equilibrium(torch.ones(shape, device="cuda", dtype=torch.float64), u)
        zero = torch.zeros((3,) + shape, device="cuda", dtype=torch.float64)
        for k in range(case["steps"]):
            if k:
                f = torch.stack([torch.roll(f[p], c, dims=(0, 1, 2)) for p, c in enumerate(_C.tolist())])
            f, rho, u = _collide(f, zero, (case["tau"] - 0.5)/3.0)
        out = dict(f=f, rho=rho, u=u)
    else:
        phi = _noise(shape, g, 0.05)
        f = _W.reshape(19, 1, 1, 1).cuda().expand((19,) + shape).clone()
        phi, f, rho, u, force = _binary_steps(phi, f, None, None, case["steps"],
                                              (FE["a"], FE["b"], FE["kappa"], FE["mobility"]), case["order"],
                                              case["stencil"], case["method"], False)
        out = dict(f=f, rho=rho, u=u, phi=phi, force=force)
    if case["bits"] == 32:
        out["f"] = out["f"] - _W.reshape(19, 1, 1, 1).cuda()
    return out


class _Conv(torch.autograd.Function):
    """The periodic 3 x 3 x 3 convolution, x [b][nx][ny][nz][ci], w [27][co][ci]."""

    @staticmethod
    def forward(ctx, x, w, bias):
        ctx.save_for_backward(x, w)
        y = bias.expand(x.shape[:-1] + (w.shape[1],)).clone().reshape(-1, w.shape[1])
        for t, o in enumerate(_TAPS):
            y += torch.roll(x, [-k for k in o], dims=(1, 2, 3)).reshape(-1, x.shape[-1]) @ w[t].t()
        return y.reshape(x.shape[:-1] + (w.shape[1],))

    @staticmethod
    def backward(ctx, dy):
        x, w = ctx.saved_tensors
        d = dy.reshape(-1, w.shape[1])
        dx, dw = torch.zeros_like(x), torch.empty_like(w)
        for t, o in enumerate(_TAPS):
            dw[t] = d.t() @ torch.roll(x, [-k for k in o], dims=(1, 2, 3)).reshape(-1, x.shape[-1])
            dx += torch.roll((d @ w[t]).reshape(x.shape), list(o), dims=(1, 2, 3))
        return dx, dw, d.sum(0)


_TAPS = [(i, j, k) for i in (-1, 0, 1) for j in (-1, 0, 1) for k in (-1, 0, 1)]


def _net_params():
    d = np.load(surrogate_study.WEIGHTS)
    norm = {k[5:]: float(d[k]) for k in d.files if k.startswith("norm_")}
    w = (d["w_bf16"].astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    bias = d["bias"].astype(np.float64)
    got, i, j = {}, 0, 0
    for name, ci, co in S.LAYERS:
        got[name] = (torch.from_numpy(w[i:i + 27*co*ci].reshape(27, co, ci)).cuda(),
                     torch.from_numpy(bias[j:j + co]).cuda())
        i, j = i + 27*co*ci, j + co
    return got, norm, int(d["step"])


def _net(x, p):
    def act(name, v):
        return torch.nn.functional.silu(_Conv.apply(v, *p[name]))

    def down(v):
        b, n0, n1, n2, c = v.shape
        return v.reshape(b, n0//2, 2, n1//2, 2, n2//2, 2, c).mean(dim=(2, 4, 6))

    def up(v):
        return v.repeat_interleave(2, 1).repeat_interleave(2, 2).repeat_interleave(2, 3)

    e0 = act("e0b", act("e0a", x))
    e1 = act("e1b", act("e1a", down(e0)))
    e2 = act("e2b", act("e2a", down(e1)))
    v = act("b1", act("b0", down(e2)))
    for name, skip in (("d2", e2), ("d1", e1), ("d0", e0)):
        v = act(name, torch.cat([up(v), skip], dim=-1))
    return _Conv.apply(v, *p["out"])


def _encoded(now, spec, norm):
    """The network's input for a state of 4 planes."""
    x = torch.zeros(tuple(now.shape[1:]) + (S.CIN,), device="cuda", dtype=torch.float64)
    x[..., 0] = (now[0] - norm["phi_shift"])*norm["phi_scale"]
    for k in range(3):
        x[..., 1 + k] = now[1 + k]*norm["u_scale"]
    for k, v in enumerate((spec.phi0/0.3, (spec.kappa - 0.05)/0.03, (spec.mobility - 0.3)/0.2)):
        x[..., 4 + k] = v
    return x


def _exact_replicas(case, seed):
    specs = _specs(case, seed)
    out = []
    p, norm, _ = _net_params() if case["kind"] == "jump" else (None, None, None)
    for s, now in zip(specs, _replica_states(case, seed, specs)):
        now = now.double()
        if p is not None:
            with torch.no_grad():
                y = _net(_encoded(now, s, norm)[None], p)[0]
            gain = (norm["jump_gain_phi"]/norm["dphi_scale"],) + (norm["jump_gain_u"]/norm["du_scale"],)*3
            new = torch.stack([(now[k] + y[..., k]*gain[k]).clamp(-m, m)
                               for k, m in enumerate((S.PHI_MAX,) + (S.U_MAX,)*3)])
            now = new + (now - new).mean(dim=(1, 2, 3), keepdim=True)
        phi, u = now[0], now[1:]
        rho = torch.ones_like(phi)
        phi, _, _, u, _ = _binary_steps(phi, _equilibrium(rho, u), rho, u, case["steps"],
                                        (s.a, s.b, s.kappa, s.mobility), case.get("order", 1), 7, "stress", True)
        out.append(torch.cat([phi.reshape(-1), u.reshape(-1)]))
    return torch.cat(out)


def exact(case, seed):
    kind = case["kind"]
    if kind == "shear":
        # the planes' interpolations, corrections and reprojections have no
        # short form in plain torch; the reference's own vectors hold them
        return None
    if kind in ("single", "binary", "staged"):
        return _exact_fluid(case, seed)
    if kind in ("ensemble", "jump"):
        return _exact_replicas(case, seed)
    if kind == "layer":
        n, x, w, bias, da = _layer_inputs(case, seed)
        x = x.double().reshape((case["batch"],) + _shape(case) + (case["cin"],)).requires_grad_()
        w, bias = w.double().requires_grad_(), bias.double().requires_grad_()
        z = _Conv.apply(x, w, bias)
        z.retain_grad()
        a = torch.nn.functional.silu(z)
        a.backward(da.double().reshape(a.shape))
        flat = lambda v: v.detach().reshape(n, -1)          # noqa: E731
        return dict(z=flat(z), a=flat(a), dz=flat(z.grad), dzb=flat(z.grad), dw=w.grad, db=bias.grad, dx=flat(x.grad))
    p, norm, step = _net_params()
    data = _samples(case, seed)
    x = torch.stack([_encoded(now.double(), q, norm) for now, _, q in data])
    if kind == "unet":
        with torch.no_grad():
            return _net(x, p).reshape(-1, S.COUT)
    for w, bias in p.values():
        w.requires_grad_()
        bias.requires_grad_()
    y = _net(x, p)[..., :4]
    scale = torch.tensor([norm["dphi_scale"]] + [norm["du_scale"]]*3, device="cuda", dtype=torch.float64)
    want = torch.stack([torch.movedim(nxt.double() - now.double(), 0, -1) for now, nxt, _ in data])*scale
    loss = (torch.tensor([1.0, 0.1, 0.1, 0.1], device="cuda", dtype=torch.float64)*(y - want)**2).mean()
    loss.backward()
    flat = lambda f: torch.cat([torch.cat([f(w).reshape(-1), f(bias)]) for w, bias in p.values()])   # noqa: E731
    g, w = flat(lambda v: v.grad), flat(lambda v: v.detach())
    h = g*min(1.0, 1.0/max(float(g.norm()), 1.0e-30))
    b1, b2, t = 0.9, 0.999, step + 1
    m, v = (1 - b1)*h, (1 - b2)*h*h
    lr = 1.0e-5*math.sqrt(1 - b2**t)/(1 - b1**t)
    return dict(loss=float(loss.detach()), g=g, w=w - lr*m/(v.sqrt() + 1.0e-8), m=m, v=v)
