"""What a program that uses this library spends its GPU time on, as measurable cases.

A case is a dict of plain values.  Every case goes through the C entry points
of the library as a program does that owns a handle and a (pinned) buffer for
the configurations it fetches: HMC trajectories, Metropolis sweeps, the
observables of one configuration, the gradient-flow table, the flow's
forward / backward pair, and the batched ensemble.

    listed()            the listed cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) inputs and handle, from the seed alone
    run(state)          one pass; the results and the updated fields
    work(case)          bytes and operations a pass cannot do without
    exact(case, seed)   what run() returns, from plain torch in 64 bits

Links that come back in the FP32 form are given in float32, which is what the
form stores (the entry points hand every field out as doubles).
"""
import ctypes as C
import math
import random

import numpy as np
import torch
import torch.utils.checkpoint

import su2_amd as S

U1, SU2 = S.U1, S.SU2
PREC = {"fp64": S.FP64, "fp32": S.FP32}


# ------------------------------------------------------------------ the cases --
def _hmc(name, group, dims, beta, prec, integrator, nsteps, ntraj, xi=1.0):
    """ntraj trajectories of device momenta, then the configuration is fetched
    (measured or saved by the caller).  dims = Lx, Ly, Lz, Lt, nd."""
    return dict(name=name, kind="hmc", group=group, Lx=dims[0], Ly=dims[1], Lz=dims[2],
                Lt=dims[3], nd=dims[4], beta=beta, xi=xi, prec=prec, integrator=integrator,
                nsteps=nsteps, ntraj=ntraj)


def listed():
    return [
        # a first look at a small lattice: 41 or fewer short launches a trajectory, latency counts
        _hmc("hmc_su2_8x4_fp64", "su2", (8, 8, 8, 8, 4), 2.3, "fp64", "leapfrog", 10, 4),
        # the benchmark workload of this repository, in both forms
        _hmc("hmc_su2_32x4_fp64", "su2", (32, 32, 32, 32, 4), 2.4, "fp64", "omf2", 20, 4),
        _hmc("hmc_su2_32x4_fp32", "su2", (32, 32, 32, 32, 4), 2.4, "fp32", "omf2", 20, 2),
        # beyond the last-level cache (the largest size of bench.py's default run)
        _hmc("hmc_su2_48x4_fp64", "su2", (48, 48, 48, 48, 4), 2.5, "fp64", "omf2", 20, 2),
        # a lattice of odd and uneven extents
        _hmc("hmc_su2_ragged_fp64", "su2", (20, 18, 15, 27, 4), 2.4, "fp64", "omf2", 10, 4),
        # an anisotropic lattice (temporal and spatial weights)
        _hmc("hmc_su2_24x3x48_xi2", "su2", (24, 24, 24, 48, 4), 2.4, "fp64", "omf2", 10, 2, xi=2.0),
        # the other gauge group
        _hmc("hmc_u1_24x4_fp64", "u1", (24, 24, 24, 24, 4), 1.0, "fp64", "leapfrog", 20, 4),
        # many small lattices of both groups in d = 2, 3, 4 advanced together (this repository's ensemble)
        dict(name="batch_224_fp32", kind="batch", n_u1=128, n_d3=64, n_d4=32, mix=13526463,
             prec="fp32", ntraj=2),
        # Metropolis updates between two measurements, at the benchmark size
        dict(name="sweep_su2_32x4_fp64", kind="sweep", group="su2", Lx=32, Ly=32, Lz=32, Lt=32,
             nd=4, beta=2.4, xi=1.0, prec="fp64", delta=0.3, nhit=10, nsweep=10),
        # what is measured on one configuration: plaquette, clover energy density and charge
        dict(name="measure_su2_32x4_fp64", kind="measure", group="su2", Lx=32, Ly=32, Lz=32,
             Lt=32, nd=4, beta=2.4, xi=1.0, prec="fp64"),
        # the gradient-flow table of one configuration
        dict(name="flow_su2_24x4_fp64", kind="flow", group="su2", Lx=24, Ly=24, Lz=24, Lt=24,
             nd=4, beta=2.4, xi=1.0, prec="fp64", eps=0.01, nrows=20),
        # the flow's forward and backward pass, at the size of bench.py
        dict(name="adjoint_su2_24x4_fp32", kind="adjoint", group="su2", Lx=24, Ly=24, Lz=24,
             Lt=24, nd=4, beta=2.4, xi=1.0, prec="fp32", eps=0.01, nsteps=100, ckpt=20),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _extents(rng, nd, lo, hi, even=False):
    """Lx, Ly, Lz, Lt, nd: equal multiples of 4 as often as uneven ones."""
    if rng.random() < 0.5:
        n = max(4, 4 * int(round(_log_int(rng, lo, hi) / 4)))
        e = [n] * nd
        if rng.random() < 0.5:
            e[0] = min(2 * n, 64)  # longer in t
    else:
        e = [_log_int(rng, lo, hi) for _ in range(nd)]
    if even:
        e = [v + v % 2 for v in e]
    t, x = e[0], e[1]
    y = e[2] if nd > 2 else 1
    z = e[3] if nd > 3 else 1
    return dict(Lx=x, Ly=y, Lz=z, Lt=t, nd=nd)


def _beta(rng, group, nd):
    lo, hi = {("su2", 4): (2.2, 2.6), ("su2", 3): (3.0, 8.0), ("su2", 2): (1.0, 8.0),
              ("u1", 4): (0.8, 1.2), ("u1", 3): (1.0, 2.5), ("u1", 2): (1.0, 6.0)}[(group, nd)]
    return round(rng.uniform(lo, hi), 3)


_RANGE = {4: (4, 40), 3: (8, 96), 2: (16, 512)}


def draw(rng):
    kind = rng.choice(["hmc", "hmc", "hmc", "batch", "sweep", "measure", "flow", "adjoint"])
    prec = rng.choice(["fp64", "fp32"])
    if kind == "batch":
        n = _log_int(rng, 8, 224)
        return dict(kind=kind, n_u1=(4 * n) // 7, n_d3=(2 * n) // 7, n_d4=max(1, n // 7),
                    mix=rng.randrange(1 << 30), prec=prec, ntraj=2)
    group = "u1" if kind != "adjoint" and rng.random() < 0.25 else "su2"
    nd = rng.choice([4, 4, 4, 3, 2]) if kind in ("hmc", "sweep", "measure") else 4
    lo, hi = _RANGE[nd]
    if kind in ("flow", "adjoint"):
        lo, hi = 6, 24
    c = dict(kind=kind, group=group, **_extents(rng, nd, lo, hi))
    c.update(beta=_beta(rng, group, nd), prec=prec,
             xi=rng.choice([1.0, 1.0, 1.0, 1.5, 2.0]) if kind == "hmc" and nd > 2 else 1.0)
    if kind == "hmc":
        c.update(integrator=rng.choice(["omf2", "leapfrog"]), nsteps=rng.randint(10, 20),
                 ntraj=2 if prec == "fp64" else 1)
    elif kind == "sweep":
        c.update(delta=round(rng.uniform(0.1, 0.5), 3), nhit=rng.randint(1, 10),
                 nsweep=rng.randint(1, 10))
    elif kind == "flow":
        c.update(eps=0.01, nrows=rng.randint(5, 20))
    elif kind == "adjoint":
        c.update(eps=0.01, nsteps=rng.randint(10, 60), ckpt=rng.choice([5, 10, 20]))
    return c


# ----------------------------------------------------------------- the inputs --
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _dims(case):
    return (case["Lt"], case["Lx"], case["Ly"], case["Lz"])


def _mul(u, v):
    """(a1, b1)(a2, b2) of [[a, b], [-b*, a*]], complex128 fields"""
    return u[0] * v[0] - u[1] * v[1].conj(), u[0] * v[1] + u[1] * v[0].conj()


def _dag(u):
    return u[0].conj(), -u[1]


def _up(u, d):
    """the field at x + d"""
    if isinstance(u, tuple):
        return tuple(torch.roll(c, -1, d) for c in u)
    return torch.roll(u, -1, d)


def _dn(u, d):
    if isinstance(u, tuple):
        return tuple(torch.roll(c, 1, d) for c in u)
    return torch.roll(u, 1, d)


def _links(group, dims, nd, beta, gen, dev):
    """Links of a chain on its way from a hot start to equilibrium (about half
    the plaquette it has there at this beta), in a random gauge: per direction
    (a, b) complex or phases.  Trajectories from there are accepted."""
    shape = tuple(dims)
    if group == "su2":
        p = max(0.05, 0.45 * (1.0 - 0.888 / beta))
        # E[cos |w|] = (1 - s^2) exp(-s^2 / 2) = p^(1/4) for w ~ N(0, s^2) in R^3
        s2, r = 0.0, p ** 0.25
        for _ in range(60):
            s2 = 1.0 - r * math.exp(s2 / 2)
        rnd = lambda k: torch.randn((k,) + shape, generator=gen, device=dev, dtype=torch.float64)  # noqa: E731
        g = rnd(4)
        g = g / g.square().sum(0).sqrt()
        g = (torch.complex(g[0], g[1]), torch.complex(g[2], g[3]))
        out = []
        for mu in range(nd):
            w = rnd(3) * math.sqrt(s2)
            n = w.square().sum(0).sqrt()
            sc = torch.sin(n) / n
            u = (torch.complex(torch.cos(n), sc * w[2]), torch.complex(sc * w[1], sc * w[0]))
            out.append(_mul(_mul(g, u), _dag(_up(g, mu))))
        return out
    p = max(0.05, 0.45 * (1.0 - 0.5 / beta))
    s = math.sqrt(-math.log(p) / 2.0)  # E[cos of four] = exp(-2 s^2)
    al = (2 * torch.rand(shape, generator=gen, device=dev, dtype=torch.float64) - 1) * math.pi
    return [al - _up(al, mu)
            + s * torch.randn(shape, generator=gen, device=dev, dtype=torch.float64)
            for mu in range(nd)]


def _to_aos(links, group):
    """device fields -> the entry points' order: (sites, nd, components)"""
    if group == "su2":
        u = torch.stack([torch.stack([a.real, a.imag, b.real, b.imag], -1) for a, b in links], -2)
        return u.reshape(-1, 4)
    return torch.stack(links, -1).reshape(-1)


def _gen(seed, dev):
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed) % (1 << 60))
    return g


def _start(group, dims, nd, beta, prec, seed, k=0):
    """the start configuration of a case (FP32 form: values an FP32 link holds)"""
    dev = _device()
    u = _links(group, dims, nd, beta, _gen(int(seed) * 4096 + k, dev), dev)
    if prec == "fp32":
        r = lambda x: x.to(torch.float32).to(torch.float64)  # noqa: E731
        if group == "su2":
            u = [tuple(torch.complex(r(c.real), r(c.imag)) for c in l) for l in u]
        else:
            u = [r(l) for l in u]
    return u


def _members(case):
    """the ensemble: U(1) d=2, L in 16..128; SU(2) d=3, L in 8..24; SU(2) d=4, L in
    {8, 12, 16}; leapfrog, tau = 1, 10..40 steps"""
    r, out = random.Random(case["mix"]), []
    for _ in range(case["n_u1"]):
        n = r.randint(16, 128)
        out.append(dict(group="u1", dims=(n, n, 1, 1), nd=2, beta=r.uniform(1, 6)))
    for _ in range(case["n_d3"]):
        n = r.randint(8, 24)
        out.append(dict(group="su2", dims=(n, n, n, 1), nd=3, beta=r.uniform(3, 8)))
    for _ in range(case["n_d4"]):
        n = r.choice([8, 12, 16])
        out.append(dict(group="su2", dims=(n, n, n, n), nd=4, beta=r.uniform(2.2, 2.6)))
    for m in out:
        m["nsteps"] = r.randint(10, 40)
    return out


def _chain_seed(seed, k=0):
    return (int(seed) % (1 << 40)) * 1024 + 7 + k


def _ck(rc):
    if rc != 0:
        raise RuntimeError(S.load_library().su2gpu_last_error().decode())


def _host(n):
    return torch.empty(n, dtype=torch.float64, pin_memory=torch.cuda.is_available())


class State:
    """a handle and the host buffers its program keeps; given back at the end"""

    def __init__(self, case):
        self.case, self.lib = case, S.load_library()
        self.h, self.batch, self.f32 = None, None, None

    def own(self, n):
        self.buf = _host(n)
        if self.case["prec"] == "fp32":
            self.f32 = torch.empty(n, dtype=torch.float32)

    def fetched(self):
        return self.buf if self.f32 is None else self.f32.copy_(self.buf)

    def numbers(self, v):
        return np.array(v, dtype=np.float64 if self.f32 is None else np.float32)

    def __del__(self):
        if self.h:
            self.lib.su2gpu_destroy(self.h)
        if self.batch:
            self.lib.su2gpu_batch_destroy(self.batch)


def prepare(case, seed):
    st = State(case)
    if case["kind"] == "batch":
        return _prepare_batch(st, case, seed)
    group, nd = case["group"], case["nd"]
    h = C.c_void_p()
    _ck(st.lib.su2gpu_create(C.byref(h), SU2 if group == "su2" else U1, case["Lx"], case["Ly"],
                             case["Lz"], case["Lt"], nd, case["beta"], case["xi"],
                             PREC[case["prec"]]))
    st.h = h
    aos = _to_aos(_start(group, _dims(case), nd, case["beta"], case["prec"], seed), group)
    n = aos.numel()
    st.own(aos.shape[0] * 3 if case["kind"] == "adjoint" else n)
    src = st.buf if st.buf.numel() == n else _host(n)
    src.view(aos.shape).copy_(aos)
    _ck(st.lib.su2gpu_set_links(h, C.c_void_p(src.data_ptr()), S.LAYOUT_PACKED))
    st.seed, st.count = _chain_seed(seed), 0
    if case["kind"] == "flow":
        st.rows = np.zeros((case["nrows"] + 2, 9))
    return st


def _prepare_batch(st, case, seed):
    st.members = _members(case)
    arr = (S.BatchMember * len(st.members))()
    for i, m in enumerate(st.members):
        t, x, y, z = m["dims"]
        arr[i] = S.BatchMember(SU2 if m["group"] == "su2" else U1, x, y, z, t, m["nd"], m["beta"],
                               S.LEAPFROG, m["nsteps"], 1.0, _chain_seed(seed, i))
    b = C.c_void_p()
    _ck(st.lib.su2gpu_batch_create(C.byref(b), arr, len(st.members), PREC[case["prec"]]))
    st.batch = b
    sizes = [math.prod(m["dims"]) * m["nd"] * (4 if m["group"] == "su2" else 1)
             for m in st.members]
    st.off = np.concatenate([[0], np.cumsum(sizes)]).tolist()
    st.own(st.off[-1])
    for i, m in enumerate(st.members):
        u = _start(m["group"], m["dims"], m["nd"], m["beta"], case["prec"], seed, i + 1)
        st.buf[st.off[i]:st.off[i + 1]].copy_(_to_aos(u, m["group"]).reshape(-1))
        _ck(st.lib.su2gpu_batch_set_links(b, i, C.cast(st.buf.data_ptr() + 8 * st.off[i],
                                                       C.POINTER(C.c_double))))
    _ck(st.lib.su2gpu_batch_use_graph(b, 1))
    st.res = (S.MDResult * len(st.members))()
    st.count = 0
    return st


# ------------------------------------------------------------------- the pass --
_FIELDS = ("kin_old", "gauge_old", "kin_new", "gauge_new")


def run(st):
    case, lib, h = st.case, st.lib, st.h
    kind = case["kind"]
    if kind == "hmc":
        energies, accept = [], []
        r = S.MDResult()
        for _ in range(case["ntraj"]):
            _ck(lib.su2gpu_md_update(h, st.seed + st.count, S.INTEGRATORS[case["integrator"]],
                                     case["nsteps"], 1.0, 0, 0, S.MOMENTA_DEVICE, C.byref(r)))
            st.count += 1
            energies.append([getattr(r, f) for f in _FIELDS])
            accept.append(r.accept)
        _ck(lib.su2gpu_get_links(h, C.c_void_p(st.buf.data_ptr()), S.LAYOUT_PACKED))
        return {"links": st.fetched(), "energies": st.numbers(energies),
                "accept": np.array(accept, dtype=np.int64)}
    if kind == "sweep":
        rates = []
        a, b = C.c_double(), C.c_double()
        for _ in range(case["nsweep"]):
            _ck(lib.su2gpu_sweep(h, st.seed, st.count, case["delta"], case["nhit"], C.byref(a),
                                 C.byref(b)))
            st.count += 1
            rates.append([a.value, b.value])
        _ck(lib.su2gpu_get_links(h, C.c_void_p(st.buf.data_ptr()), S.LAYOUT_PACKED))
        return {"links": st.fetched(), "rates": st.numbers(rates)}
    if kind == "measure":
        g, e, q = C.c_double(), C.c_double(), C.c_double()
        _ck(lib.su2gpu_gauge_energy(h, 0, C.byref(g)))
        _ck(lib.su2gpu_energy_density(h, 1, 0, C.byref(e), C.byref(q)))
        return {"observables": st.numbers([g.value / _den(case), e.value, q.value])}
    if kind == "flow":
        n = C.c_size_t()
        _ck(lib.su2gpu_gradient_flow(h, (2 * case["nrows"] - 1) * case["eps"], case["eps"], 0.0,
                                     st.rows.ctypes.data_as(C.c_void_p), st.rows.shape[0],
                                     C.byref(n)))
        return {"rows": st.numbers(st.rows[: n.value])}
    if kind == "adjoint":
        v = C.c_double()
        _ck(lib.su2gpu_flow_forward(h, case["eps"], case["nsteps"], case["ckpt"],
                                    S.OBS_CLOVER_E, C.byref(v)))
        _ck(lib.su2gpu_flow_backward(h, C.c_void_p(st.buf.data_ptr())))
        return {"value": st.numbers(v.value), "grad": st.fetched()}
    # batch: trajectories of every lattice, then their configurations
    energies, accept = [], []
    for _ in range(case["ntraj"]):
        _ck(lib.su2gpu_batch_trajectory(st.batch, S.MOMENTA_DEVICE, st.count, 1, st.res))
        st.count += 1
        energies.append([[getattr(r, f) for f in _FIELDS] for r in st.res])
        accept.append([r.accept for r in st.res])
    for i in range(len(st.members)):
        _ck(lib.su2gpu_batch_get_links(st.batch, i, C.cast(st.buf.data_ptr() + 8 * st.off[i],
                                                           C.POINTER(C.c_double))))
    return {"links": st.fetched(), "energies": st.numbers(energies),
            "accept": np.array(accept, dtype=np.int64)}


def _den(case):
    return math.prod(_dims(case)) * (2.0 if case["group"] == "su2" else 1.0)


# ------------------------------------------------------------------- the work --
def _forces(case):
    n = case["nsteps"]
    return 2 * n + 1 if case.get("integrator") == "omf2" else n + 1


def _link_bytes(group, prec):
    real = 8 if prec == "fp64" else 4
    return (4 * real, 3 * real) if group == "su2" else (real, real)


def _staple_flops(group, nd):
    """one link's force: 2 (nd - 1) staples of two products, the product with the link"""
    per = 2 * 28 + 4 if group == "su2" else 10
    return 2 * (nd - 1) * per + (28 if group == "su2" else 8)


def _traj_work(group, nd, volume, prec, forces):
    """per P-then-U step: read U and P, write U and P; the last force reads U, P and writes P"""
    u, p = _link_bytes(group, prec)
    links = volume * nd
    return (links * (forces - 1) * (2 * u + 2 * p) + links * (u + 2 * p),
            links * forces * (_staple_flops(group, nd) + (60 if group == "su2" else 4)))


def work(case):
    kind, prec = case["kind"], case["prec"]
    if kind == "batch":
        total = [0.0, 0.0]
        for m in _members(case):
            b, f = _traj_work(m["group"], m["nd"], math.prod(m["dims"]), prec, m["nsteps"] + 1)
            total[0] += case["ntraj"] * b
            total[1] += case["ntraj"] * f
        return {"bytes": total[0], "flops": total[1]}
    group, nd, volume = case["group"], case["nd"], math.prod(_dims(case))
    u, p = _link_bytes(group, prec)
    links = volume * nd
    planes = nd * (nd - 1) // 2
    product = 28 if group == "su2" else 4
    if kind == "hmc":
        b, f = _traj_work(group, nd, volume, prec, _forces(case))
        return {"bytes": case["ntraj"] * b, "flops": case["ntraj"] * f}
    if kind == "sweep":
        # each hit: one random element, one product, two traces, one exponential
        hit = 100 if group == "su2" else 40
        return {"bytes": case["nsweep"] * links * 2.0 * u,
                "flops": case["nsweep"] * links * (_staple_flops(group, nd) + case["nhit"] * hit)}
    clover = volume * planes * 4 * 3 * product
    if kind == "measure":
        return {"bytes": 2.0 * links * u, "flops": clover + volume * planes * 3 * product}
    stage = links * (2.0 * u + 2.0 * p)  # one Runge-Kutta stage: read W, Z, write W, Z
    force = links * (_staple_flops(group, nd) + 60)
    if kind == "flow":
        steps = 2 * case["nrows"]
        return {"bytes": steps * (3 * stage + 2.0 * links * u),
                "flops": steps * (3 * force + clover + volume * planes * 3 * product)}
    # forward: three stages a step; backward: the stage states, lambda_W and lambda_Z read, both written
    n = case["nsteps"]
    return {"bytes": n * 3 * (stage + links * (u + 5.0 * p)), "flops": n * 3 * 3.0 * force}


# -------------------------------------------------------- the same in 64 bits --
_M0, _M1, _W0, _W1, _LOW = 0xD2511F53, 0xCD9E8D57, 0x9E3779B9, 0xBB67AE85, 0xFFFFFFFF


def _hi(m, c):
    """upper 32 bits of the product of two 32-bit numbers, in int64"""
    return ((m >> 16) * c + (((m & 0xFFFF) * c) >> 16)) >> 16


def _philox(c, seed):
    """Philox4x32-10 (Salmon et al., SC'11), c: four int64 tensors of 32-bit words"""
    k0, k1 = seed & _LOW, (seed >> 32) & _LOW
    for _ in range(10):
        c = [_hi(_M1, c[2]) ^ c[1] ^ k0, (_M1 * c[2]) & _LOW,
             _hi(_M0, c[0]) ^ c[3] ^ k1, (_M0 * c[0]) & _LOW]
        k0, k1 = (k0 + _W0) & _LOW, (k1 + _W1) & _LOW
    return c


def _words(lid, w1, number, seed):
    full = lambda x: torch.full_like(lid, x)  # noqa: E731
    return _philox([lid, full(w1), full(number & _LOW), full((number >> 32) & _LOW)], seed)


class _Field:
    """one lattice in plain torch: links as complex pairs (SU(2)) or phases (U(1))"""

    def __init__(self, group, dims, nd, beta, links, xi=1.0):
        self.su2, self.dims, self.nd, self.beta, self.U = group == "su2", dims, nd, beta, links
        self.Nc, self.xi = (2.0 if self.su2 else 1.0), xi
        dev = (links[0][0] if self.su2 else links[0]).device
        self.site = torch.arange(math.prod(dims), device=dev, dtype=torch.int64).reshape(dims)

    def w(self, mu, nu):
        return 1.0 / self.xi if min(mu, nu) == 0 else self.xi

    def staples(self, mu, U=None):
        U = self.U if U is None else U
        K = None
        for nu in range(self.nd):
            if nu == mu:
                continue
            if self.su2:
                a = _mul(_mul(_up(U[nu], mu), _dag(_up(U[mu], nu))), _dag(U[nu]))
                b = _dn(_mul(_mul(_dag(_up(U[nu], mu)), _dag(U[mu])), U[nu]), nu)
                t = (a[0] + b[0], a[1] + b[1])
                t = (self.w(mu, nu) * t[0], self.w(mu, nu) * t[1])
                K = t if K is None else (K[0] + t[0], K[1] + t[1])
            else:
                a = _up(U[nu], mu) - _up(U[mu], nu) - U[nu]
                b = _dn(-_up(U[nu], mu) - U[mu] + U[nu], nu)
                t = self.w(mu, nu) * (torch.polar(torch.ones_like(a), a)
                                      + torch.polar(torch.ones_like(b), b))
                K = t if K is None else K + t
        return K

    def force(self, mu, U=None):
        """get_deriv(U K): the momentum components of one direction"""
        U = self.U if U is None else U
        K = self.staples(mu, U)
        if self.su2:
            m = _mul(U[mu], K)
            return torch.stack([2 * m[1].imag, 2 * m[1].real, 2 * m[0].imag])
        return (torch.polar(torch.ones_like(U[mu]), U[mu]) * K).imag[None]

    def exp_mul(self, p, u):
        if not self.su2:
            return u + p[0]
        n = p.square().sum(0).sqrt()
        sc = torch.where(n > 1e-6, torch.sin(n) / n.clamp_min(1e-300), 1 - n * n / 6)
        return _mul((torch.complex(torch.cos(n), sc * p[2]),
                     torch.complex(sc * p[1], sc * p[0])), u)

    def plaquettes(self, weighted=False, mu0=0):
        total = 0.0
        for mu in range(mu0, self.nd):
            for nu in range(mu + 1, self.nd):
                U = self.U
                if self.su2:
                    p = _mul(_mul(U[mu], _up(U[nu], mu)),
                             _dag(_mul(U[nu], _up(U[mu], nu))))[0].real * 2
                else:
                    p = torch.cos(U[mu] + _up(U[nu], mu) - _up(U[mu], nu) - U[nu])
                total = total + (self.w(mu, nu) if weighted else 1.0) * p.sum()
        return float(total)

    def normalise(self):
        if self.su2:
            for mu in range(self.nd):
                a, b = self.U[mu]
                n = (a.abs().square() + b.abs().square()).sqrt()
                self.U[mu] = (a / n, b / n)

    def momenta(self, seed, number):
        out = []
        for mu in range(self.nd):
            c = _words(self.site * self.nd + mu, 0, number, seed)
            z = []
            for h in (0, 2):
                r = torch.sqrt(-2 * torch.log((c[h].double() + 1) * 2.0 ** -32))
                ang = 2 * math.pi * (c[h + 1].double() * 2.0 ** -32)
                z += [r * torch.cos(ang), r * torch.sin(ang)]
            out.append(torch.stack(z[:3] if self.su2 else z[:1]))
        return out

    def trajectory(self, integrator, nsteps, seed, number=0):
        P = self.momenta(seed, number)
        keep = list(self.U)
        kin = lambda: 0.5 * float(sum(p.square().sum() for p in P))  # noqa: E731
        act = lambda: -self.beta / self.Nc * self.plaquettes(True)  # noqa: E731
        old = (kin(), act())
        dt = 1.0 / nsteps
        if integrator == "omf2":
            lam = 0.1938
            ops = [lam] + [0.5, 1 - 2 * lam, 0.5, 2 * lam] * nsteps
            ops[-1] = lam
        else:
            ops = [0.5] + [1.0, 1.0] * nsteps
            ops[-1] = 0.5
        for k, c in enumerate(ops):
            if k % 2 == 0:
                for mu in range(self.nd):
                    P[mu] = P[mu] - c * dt * self.beta / self.Nc * self.force(mu)
            else:
                self.U = [self.exp_mul(c * dt * P[mu], self.U[mu]) for mu in range(self.nd)]
        self.normalise()
        new = (kin(), act())
        dH = (new[0] - old[0]) + (new[1] - old[1])
        accept = 1
        if dH > 0:
            one = torch.full((1,), _LOW, dtype=torch.int64)
            c = _words(one, _LOW, number, seed)
            u = (((int(c[0]) << 32 | int(c[1])) >> 11) + 0.5) / 2.0 ** 53
            accept = int(u <= math.exp(-dH))
        if not accept:
            self.U = keep
        return [old[0], old[1], new[0], new[1]], accept

    def colours(self, mu):
        """the sub-sweeps of direction mu: site parity, or three classes where an extent is odd"""
        co = torch.meshgrid(*[torch.arange(n, device=self.site.device) for n in self.dims],
                            indexing="ij")
        if all(n % 2 == 0 for n in self.dims[: self.nd]):
            return sum(co[: self.nd]) % 2, 2
        col = 0
        for d in range(self.nd):
            if d != mu:
                col = col + co[d] + co[d].clamp_max((3 - self.dims[d] % 3) % 3)
        return col % 3, 3

    def sweep(self, seed, number, delta, nhit):
        hits, hits_t = 0, 0
        for mu in range(self.nd):
            col, ncol = self.colours(mu)
            lid = self.site * self.nd + mu
            for k in range(ncol):
                K = self.staples(mu)
                sel = col == k
                for n in range(nhit):
                    c = [(x.double() + 0.5) * 2.0 ** -32 for x in _words(lid, n, number, seed)]
                    if self.su2:
                        uu = 2 * c[1] - 1
                        r = torch.sqrt(1 - uu * uu)
                        al, th = 2 * math.pi * delta * c[0], 2 * math.pi * c[2]
                        sa = torch.sin(al)
                        R = (torch.complex(torch.cos(al), sa * uu),
                             torch.complex(sa * r * torch.sin(th), sa * r * torch.cos(th)))
                        new = _mul(self.U[mu], R)
                        dS = self.beta / 2 * 2 * (_mul(self.U[mu], K)[0].real
                                                  - _mul(new, K)[0].real)
                        nn = (new[0].abs().square() + new[1].abs().square()).sqrt()
                        new = (new[0] / nn, new[1] / nn)
                    else:
                        new = self.U[mu] + math.pi * delta * (2 * c[0] - 1)
                        e = lambda t: (torch.polar(torch.ones_like(t), t) * K).real  # noqa: E731
                        dS = self.beta * (e(self.U[mu]) - e(new))
                    ok = sel & ((dS < 0) | (c[3] < torch.exp(-dS)))
                    if self.su2:
                        self.U[mu] = tuple(torch.where(ok, x, y)
                                           for x, y in zip(new, self.U[mu]))
                    else:
                        self.U[mu] = torch.where(ok, new, self.U[mu])
                    got = int(ok.sum())
                    hits += got
                    hits_t += got if mu == 0 else 0
        V = math.prod(self.dims)
        return [hits / (nhit * V * self.nd), hits_t / (nhit * V)]

    def clover(self, mu, nu, U=None):
        """sum of the four leaves: the traceless antihermitian part as a 3-vector (U(1): sum of sines)"""
        U = self.U if U is None else U
        m, n = U[mu], U[nu]
        if self.su2:
            bottom, top, right = m, _up(m, nu), _up(n, mu)
            p = _mul(_mul(_mul(bottom, right), _dag(top)), _dag(n))             # at x
            l2 = _mul(_mul(_mul(n, _dag(_dn(top, mu))), _dag(_dn(n, mu))), _dn(m, mu))
            dd = lambda f: _dn(_dn(f, mu), nu)  # noqa: E731
            l3 = _mul(_mul(_mul(_dag(_dn(m, mu)), _dag(dd(n))), dd(m)), _dn(n, nu))
            l4 = _mul(_mul(_mul(_dag(_dn(n, nu)), _dn(m, nu)), _dn(right, nu)), _dag(m))
            a = p[0] + l2[0] + l3[0] + l4[0]
            b = p[1] + l2[1] + l3[1] + l4[1]
            return torch.stack([a.imag, b.real, b.imag])
        f = torch.sin(m + _up(n, mu) - _up(m, nu) - n)
        return (f + _dn(f, mu) + _dn(f, nu) + _dn(_dn(f, mu), nu))[None]

    def energy(self, mu0=0):
        """clover energy density and topological charge"""
        G = {(m, n): self.clover(m, n) for m in range(mu0, self.nd)
             for n in range(m + 1, self.nd)}
        V = math.prod(self.dims)
        f = 2.0 if self.su2 else 1.0
        E = f * sum(g.square().sum() for g in G.values()) / V / 16
        Q = 0.0
        if self.nd == 4 and mu0 == 0:
            q = ((G[0, 1] * G[2, 3]) - (G[0, 2] * G[1, 3]) + (G[0, 3] * G[1, 2])).sum()
            Q = 4 * 2 * f * float(q) / (32 * math.pi ** 2) / 16
        elif self.nd == 2 and not self.su2:
            Q = 4 * float(G[0, 1].sum()) / (32 * math.pi ** 2) / 16
        return float(E), Q

    def rk_stage(self, U, Z, f, eps):
        z = (-17.0 / 36.0, 8.0 / 9.0, -3.0 / 4.0)[f]
        e = (-36.0 / 4.0 / 17.0, 1.0, -1.0)[f]
        D = [2 * z * self.force(mu, U) for mu in range(self.nd)]
        Z = D if Z is None else [a + b for a, b in zip(Z, D)]
        return [self.exp_mul(-eps * e * Z[mu], U[mu]) for mu in range(self.nd)], Z

    def rk(self, eps):
        Z = None
        for f in range(3):
            self.U, Z = self.rk_stage(self.U, Z, f, eps)

    def flow_rows(self, eps, nrows):
        d, V = self.nd, math.prod(self.dims)
        ndf, ndf_ss = d * (d - 1) / 2.0, (d - 1) * (d - 2) / 2.0
        rows, t = [], 0.0
        for _ in range(nrows):
            self.rk(eps)
            t += eps
            P, Pss = self.plaquettes() / (V * self.Nc), self.plaquettes(mu0=1) / (V * self.Nc)
            (E, Q), (Ess, _) = self.energy(), self.energy(1)
            Ep, Epss = ndf - P, ndf_ss - Pss
            xi = math.sqrt(((Ep - Epss) / (d - 1)) / (Epss / ndf_ss))
            rows.append([t, xi, P, Pss, Ep, Epss, E, Ess, Q])
            self.rk(eps)
            t += eps
        return rows

    def adjoint(self, eps, nsteps):
        """t^2 E(t) and its derivative with respect to U -> exp(X) U at X = 0"""
        def one_step(*flat):
            U = [(flat[2 * m], flat[2 * m + 1]) for m in range(self.nd)]
            Z = None
            for f in range(3):
                U, Z = self.rk_stage(U, Z, f, eps)
            return tuple(c for u in U for c in u)

        X = [torch.zeros((3,) + tuple(self.dims), dtype=torch.float64, device=self.site.device,
                         requires_grad=True) for _ in range(self.nd)]
        U = [_mul((torch.complex(torch.ones_like(x[0]), x[2]), torch.complex(x[1], x[0])), u)
             for x, u in zip(X, self.U)]
        flat = tuple(c for u in U for c in u)
        for _ in range(nsteps):
            flat = torch.utils.checkpoint.checkpoint(one_step, *flat, use_reentrant=False,
                                                     preserve_rng_state=False)
        U = [(flat[2 * m], flat[2 * m + 1]) for m in range(self.nd)]
        E = 0.0
        for m in range(self.nd):
            for n in range(m + 1, self.nd):
                E = E + self.clover(m, n, U).square().sum()
        E = 2.0 * E / math.prod(self.dims) / 16 * (eps * nsteps) ** 2
        E.backward()
        return float(E), torch.stack([x.grad.movedim(0, -1) for x in X], -2).reshape(-1)

    def flat(self):
        return _to_aos(self.U, "su2" if self.su2 else "u1").reshape(-1).cpu()


def _seconds(case):
    """a rough guess of exact()'s time on a GPU, from the number of link-force evaluations"""
    if case["kind"] == "batch":
        return 1.5e-4 * case["ntraj"] * sum(m["nsteps"] * m["nd"] ** 2 for m in _members(case))
    links = math.prod(_dims(case)) * case["nd"]
    n = {"hmc": case.get("ntraj", 0) * _forces(case) if case["kind"] == "hmc" else 0,
         "sweep": case.get("nsweep", 0) * (8 + 0.5 * 2 * case.get("nhit", 0)),
         "measure": 6, "flow": 2 * 3 * case.get("nrows", 0) * 2,
         "adjoint": 3 * 4 * case.get("nsteps", 0)}[case["kind"]]
    return 8e-9 * links * n


def exact(case, seed):
    if _seconds(case) > 15:
        return None
    if case["kind"] == "batch":
        links, energies = [], []
        for i, m in enumerate(_members(case)):
            f = _Field(m["group"], m["dims"], m["nd"], m["beta"],
                       _start(m["group"], m["dims"], m["nd"], m["beta"], case["prec"], seed, i + 1))
            energies.append([f.trajectory("leapfrog", m["nsteps"], _chain_seed(seed, i), k)[0]
                             for k in range(case["ntraj"])])
            links.append(f.flat())
        return {"links": torch.cat(links), "energies": np.array(energies).swapaxes(0, 1),
                "accept": None}
    f = _Field(case["group"], _dims(case), case["nd"], case["beta"],
               _start(case["group"], _dims(case), case["nd"], case["beta"], case["prec"], seed),
               case["xi"])
    kind = case["kind"]
    if kind == "hmc":
        energies = [f.trajectory(case["integrator"], case["nsteps"], _chain_seed(seed) + k)[0]
                    for k in range(case["ntraj"])]
        return {"links": f.flat(), "energies": np.array(energies), "accept": None}
    if kind == "sweep":
        rates = [f.sweep(_chain_seed(seed), k, case["delta"], case["nhit"])
                 for k in range(case["nsweep"])]
        return {"links": f.flat(), "rates": np.array(rates)}
    if kind == "measure":
        E, Q = f.energy()
        return {"observables": np.array([f.plaquettes() / _den(case), E, Q])}
    if kind == "flow":
        return {"rows": np.array(f.flow_rows(case["eps"], case["nrows"]))}
    value, grad = f.adjoint(case["eps"], case["nsteps"])
    return {"value": np.array(value), "grad": grad.cpu()}
