"""What a program that uses this framework has it do, as cases to be timed.

Every case is one pass of a program's loop through the public entry points (DgSolver, BatchSolver, or
the kernel-level C ABI), with the mesh and the solver already built, as a program keeps them:

    loop     one step() and one downloadState() per pass: the reference's own time loop, which takes
             the state off the device after every step (small meshes, where latency counts)
    run      a whole simulation on a kept solver: uploadState, run() over many steps, downloadState
    monitor  the stretch between two field snapshots of a monitored run: on-device probes, and every
             `every` steps the diagnostics and the probe history; then the snapshot
    batch    many independent cavities of mixed size and order in one solver (parameter sweeps)
    kernels  one LSRK45 step line for line through the launchers that replace the reference's own
             (nw_launch_*), on device arrays that the caller owns

Fields of FP32 runs come off the device as float64 holding FP32 values; such a program keeps its
snapshots in float32, so the runs end with that conversion.  FP64 runs keep what downloadState wrote.

Meshes are box meshes, uniform or with their interior vertices displaced (`jitter`, as a share of the
element size), periodic or PEC per axis, in vacuum or with per-element media, and optionally with the x
faces cut and fed through the on-device halo stand-in.
"""
import math

import numpy as np
import torch

import nekwave_amd as nw
from nekwave_amd._lib import check, lib

DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64 = torch.float64

# LSRK45 (Carpenter & Kennedy 1994)
RK_A = (0.0, -567301805773.0 / 1357537059087.0, -2404267990393.0 / 2016746695238.0,
        -3550918686646.0 / 2091501179385.0, -1275806237668.0 / 842570457699.0)
RK_B = (1432997174477.0 / 9575080441755.0, 5161836677717.0 / 13612068292357.0, 1720146321549.0 / 2090206949498.0,
        3134564353537.0 / 4481467310338.0, 2277821191437.0 / 14882151754819.0)


def _case(name, kind, precision, n1, nx, ny, nz, periodic, steps, jitter=0.0, media="none", halo=False,
          pipeline="fused", **more):
    return dict({"name": name, "kind": kind, "precision": precision, "pipeline": pipeline, "n1": n1, "nx": nx, "ny": ny,
                 "nz": nz, "periodic": periodic, "jitter": jitter, "media": media, "halo": halo, "steps": steps}, **more)


def listed():
    return [
        # the reference's default mesh (3^3 box), stepped and downloaded as its Case loop does: pure latency
        _case("loop_3_n4_fp64", "loop", "fp64", 4, 3, 3, 3, "", 1),
        # the unit-cube cavity of the verification runs, 200 steps: launches and small grids
        _case("run_4_n5_fp64", "run", "fp64", 5, 4, 4, 4, "", 200),
        # a small FP32 production mesh: less than one round of workgroups over the chip
        _case("run_8_n8_fp32", "run", "fp32", 8, 8, 8, 8, "xyz", 200, jitter=0.1),
        # a monitored FP64 run: 4 probes, diagnostics every 10 steps
        _case("monitor_10_n6_fp64", "monitor", "fp64", 6, 10, 10, 10, "xy", 50, media="layers", probes=4, every=10),
        # the headline mesh: periodic 16^3, jittered, p = 7
        _case("run_16_n8_fp32", "run", "fp32", 8, 16, 16, 16, "xyz", 200, jitter=0.1),
        # the same mesh in the default precision
        _case("run_16_n8_fp64", "run", "fp64", 8, 16, 16, 16, "xyz", 80, jitter=0.1),
        # odd sizes, mixed boundaries, jitter and media together, FP64 registers under FP32 fields
        _case("run_13x9x11_n7_k64", "run", "fp32_k64", 7, 13, 9, 11, "y", 200, jitter=0.15, media="random"),
        # a large cavity filled with random media: the state is several times the Infinity Cache
        _case("run_32_n8_fp32", "run", "fp32", 8, 32, 32, 32, "", 100, media="random"),
        # one GPU's share of a partitioned domain at p = 5, cut faces through the halo stand-in
        _case("run_48_n6_fp32_halo", "run", "fp32", 6, 48, 48, 48, "x", 60, media="lognormal", halo=True),
        # a sweep of small cavities of mixed order in one solver
        _case("batch_64_fp32", "batch", "fp32", 0, 0, 0, 0, "", 100, media="uniform", count=64, kmin=2, kmax=12,
              pmin=3, pmax=8, mix=4),
        # ten points per direction (only the plain pipeline takes it)
        _case("plain_8_n10_fp64", "run", "fp64", 10, 8, 8, 8, "z", 30, jitter=0.1, media="random", pipeline="plain"),
        # the reference's step kept line for line on the replacement launchers
        _case("kernels_12_n7_fp64", "kernels", "fp64", 7, 12, 12, 12, "xyz", 1, jitter=0.1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same families: sizes spread over their logarithm, axes of their own lengths."""
    kind = rng.choice(["loop", "run", "run", "run", "run", "monitor", "batch", "plain", "kernels"])
    per = "".join(a for a in "xyz" if rng.random() < 0.5)
    jit = rng.choice([0.0, 0.05, 0.1, 0.15])
    media = rng.choice(["none", "none", "random", "layers", "lognormal"])

    def box(n1, lo, hi):  # about lo .. hi nodes in all
        nodes = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        k = (nodes / n1 ** 3) ** (1.0 / 3.0)
        return [max(2, int(round(k * rng.uniform(0.75, 1.3)))) for _ in range(3)]

    if kind == "loop":
        n1 = rng.randint(3, 8)
        return _case("", kind, rng.choice(["fp64", "fp32"]), n1, *box(n1, 1e3, 3e4), per, 1, jitter=jit, media=media)
    if kind == "run":
        n1 = rng.randint(4, 9)
        prec = rng.choice(["fp64", "fp32", "fp32", "fp32", "fp32_k64"] + (["bf16x3"] if n1 == 8 else []))
        b = box(n1, 5e3, 1.2e7 if prec != "fp64" else 6e6)
        nodes = n1 ** 3 * b[0] * b[1] * b[2]
        halo = rng.random() < 0.2
        steps = max(30, min(200, int(4e8 / nodes)))
        return _case("", kind, prec, n1, *b, per if not halo else "x" + per.replace("x", ""), steps,
                     jitter=0.0 if halo else jit, media=media, halo=halo)
    if kind == "monitor":
        n1 = rng.randint(4, 8)
        return _case("", kind, rng.choice(["fp64", "fp32"]), n1, *box(n1, 2e4, 1e6), per, 40, media=media,
                     probes=rng.randint(1, 12), every=rng.choice([5, 8, 10, 20]))
    if kind == "batch":
        p0 = rng.randint(3, 6)
        return _case("", kind, rng.choice(["fp32", "fp32", "fp64"]), 0, 0, 0, 0, "", 30, media="uniform",
                     count=_log_int(rng, 6, 64), kmin=2, kmax=rng.randint(5, 11), pmin=p0, pmax=rng.randint(p0, 8),
                     mix=rng.randint(0, 1 << 20))
    if kind == "plain":
        n1 = rng.randint(5, 10)
        return _case("", "run", "fp64", n1, *box(n1, 5e4, 6e5), per, 20, jitter=jit, media=media, pipeline="plain")
    n1 = rng.randint(4, 10)
    return _case("", kind, "fp64", n1, *box(n1, 5e4, 8e5), per, 1, jitter=jit)


# --- boxes, media and fields (made here, from the seed alone) ---------------------------------------------


def _gll(n1):
    """GLL nodes, weights and the differentiation matrix D_ij = l_j'(z_i)."""
    p = n1 - 1
    P = np.polynomial.legendre.Legendre.basis(p)
    z = np.concatenate([[-1.0], np.sort(P.deriv().roots().real), [1.0]])
    for _ in range(3):  # polish the inner nodes (Newton on P')
        z[1:-1] -= P.deriv()(z[1:-1]) / P.deriv(2)(z[1:-1])
    L = P(z)
    w = 2.0 / (p * (p + 1) * L * L)
    D = np.zeros((n1, n1))
    for i in range(n1):
        for j in range(n1):
            if i != j:
                D[i, j] = L[i] / (L[j] * (z[i] - z[j]))
    D[0, 0], D[p, p] = -p * (p + 1) / 4.0, p * (p + 1) / 4.0
    return z, w, D


_OFF = ((0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1))


def _lengths(case):
    m = max(case["nx"], case["ny"], case["nz"])
    return [case[k] / m for k in ("nx", "ny", "nz")]


def _corners(case, seed):
    """Element corners [nz, ny, nx, 8, 3], interior vertices displaced by up to jitter times the element size."""
    n = (case["nx"], case["ny"], case["nz"])
    L = _lengths(case)
    ax = [np.linspace(0.0, L[d], n[d] + 1) for d in range(3)]
    V = np.stack(np.meshgrid(ax[2], ax[1], ax[0], indexing="ij")[::-1], axis=-1)  # [z, y, x, 3]
    if case["jitter"] > 0:
        r = np.random.default_rng([seed, 1])
        h = np.array([L[d] / n[d] for d in range(3)])
        inner = V[1:-1, 1:-1, 1:-1]
        inner += case["jitter"] * h * r.uniform(-1.0, 1.0, inner.shape)
    return np.stack([V[o[2]:o[2] + n[2], o[1]:o[1] + n[1], o[0]:o[0] + n[0]] for o in _OFF], axis=3)


def _media(case, seed):
    """Per-element eps and mu, or None in vacuum."""
    n = (case["nz"], case["ny"], case["nx"])
    r = np.random.default_rng([seed, 2])
    kind = case["media"]
    if kind == "none":
        return None
    if kind == "random":
        return r.uniform(1.0, 4.0, n), np.ones(n)
    if kind == "lognormal":
        return np.exp(0.3 * r.standard_normal(n).clip(-3, 3)), np.exp(0.3 * r.standard_normal(n).clip(-3, 3))
    if kind == "layers":
        return np.broadcast_to(r.uniform(1.0, 4.0, (n[0], 1, 1)), n).copy(), np.ones(n)
    return np.full(n, r.uniform(1.0, 4.0)), np.ones(n)  # uniform


def _dt(case, media):
    """The automatic rule (CFL 0.4 * 1.75 / sqrt 3 on the smallest node distance) at the fastest wave speed."""
    z = _gll(case["n1"])[0]
    h = 1.0 / max(case["nx"], case["ny"], case["nz"]) * (1.0 - 2.0 * case["jitter"])
    speed = 1.0 if media is None else max(1.0, float(np.max(1.0 / np.sqrt(media[0] * media[1]))))
    return 0.4 * 1.75 / math.sqrt(3.0) * 0.5 * h * float(z[1] - z[0]) / speed


def _shape(n1):
    """Trilinear shape functions [8, k, j, i] at the GLL nodes and their r, s, t derivatives."""
    z = _gll(n1)[0]
    one = np.ones(n1)
    N, d = [], [[], [], []]
    for o in _OFF:
        s = [2 * c - 1 for c in o]
        f = [0.5 * (1 + s[x] * z) for x in range(3)]
        g = [0.5 * s[x] * one for x in range(3)]
        N.append(np.einsum("k,j,i->kji", f[2], f[1], f[0]))
        d[0].append(np.einsum("k,j,i->kji", f[2], f[1], g[0]))
        d[1].append(np.einsum("k,j,i->kji", f[2], g[1], f[0]))
        d[2].append(np.einsum("k,j,i->kji", g[2], f[1], f[0]))
    t = lambda a: torch.tensor(np.stack(a), dtype=F64, device=DEV)  # noqa: E731
    return t(N), [t(x) for x in d]


def _field(case, seed, corners):
    """The initial state [6, nz, ny, nx, k, j, i]: a few Gaussian pulses on smooth standing waves."""
    r = np.random.default_rng([seed, 3])
    N, _ = _shape(case["n1"])
    c = torch.tensor(corners, device=DEV)
    L = _lengths(case)
    xyz = [torch.einsum("zyxa,akji->zyxkji", c[..., d].contiguous(), N) for d in range(3)]
    u = torch.empty((6,) + tuple(xyz[0].shape), dtype=F64, device=DEV)
    cen, wid = r.uniform(0.25, 0.75, (3, 3)) * np.array(L), r.uniform(0.08, 0.16, 3)
    pulse = [torch.exp(-sum((xyz[d] - cen[q][d]) ** 2 for d in range(3)) / wid[q] ** 2) for q in range(3)]
    for f in range(6):
        a = r.uniform(-1.0, 1.0, 4)
        ph = r.uniform(0.0, 2.0 * math.pi, 3)
        m = r.integers(1, 3, 3)
        wave = a[3]
        for d in range(3):
            wave = wave * torch.cos(2.0 * math.pi * int(m[d]) / L[d] * xyz[d] + ph[d])
        u[f] = wave + a[0] * pulse[0] + a[1] * pulse[1] + a[2] * pulse[2]
    return u


def _mesh(case, corners, media):
    L = _lengths(case)
    box = nw.Mesh(case["n1"])
    box.createBoxMesh(case["nx"], case["ny"], case["nz"], 0, L[0], 0, L[1], 0, L[2], "x" in case["periodic"],
                      "y" in case["periodic"], "z" in case["periodic"])
    m = box
    if case["jitter"] > 0:
        m = nw.Mesh.fromCorners(case["n1"], corners, *box.getFaces())
    if media is not None:
        m.setMaterials(media[0].ravel(), media[1].ravel())
    if case["halo"]:
        m.selfHaloX()
    return m


def _members(case):
    """The cavities of a batch: each a PEC cube of k^3 elements of degree p, sizes from `mix`."""
    r = np.random.default_rng(case["mix"])
    ks = r.integers(case["kmin"], case["kmax"] + 1, case["count"])
    ps = r.integers(case["pmin"], case["pmax"] + 1, case["count"])
    return [dict(case, kind="run", n1=int(p) + 1, nx=int(k), ny=int(k), nz=int(k)) for k, p in zip(ks, ps)]


def _probe_points(case, seed):
    r = np.random.default_rng([seed, 4])
    return r.uniform(0.05, 0.95, (case["probes"], 3)) * np.array(_lengths(case))


def _host(u):
    return u.reshape(-1).cpu().numpy()


# --- prepare and run -------------------------------------------------------------------------------------


def prepare(case, seed):
    if case["kind"] == "batch":
        members = _members(case)
        media = [_media(c, seed + 7919 * x) for x, c in enumerate(members)]
        meshes, states = [], []
        for x, c in enumerate(members):
            cor = _corners(c, seed + 7919 * x)
            meshes.append(_mesh(c, cor, media[x]))
            states.append(_host(_field(c, seed + 7919 * x, cor)))
        s = nw.BatchSolver(precision=case["precision"])
        s.initialize(meshes, 1.0)
        return {"case": case, "solver": s, "meshes": meshes, "host": states,
                "dt": min(_dt(c, m) for c, m in zip(members, media))}
    cor, media = _corners(case, seed), _media(case, seed)
    u = _field(case, seed, cor)
    if case["kind"] == "kernels":
        return _prepare_kernels(case, cor, u)
    m = _mesh(case, cor, media)
    s = nw.DgSolver(precision=case["precision"], pipeline=case["pipeline"])
    s.initialize(m, 1.0)
    host = _host(u)
    st = {"case": case, "solver": s, "mesh": m, "host": host, "out": np.zeros_like(host), "dt": _dt(case, media)}
    if case["precision"] != "fp64":
        st["snap"] = torch.zeros(host.size, dtype=torch.float32)
    if case["kind"] in ("loop", "monitor"):
        s.uploadState(host)
    if case["kind"] == "monitor":
        s.setProbes(m, _probe_points(case, seed), capacity=case["every"] + 1)
    return st


def _kept(st):
    """The downloaded fields as the program keeps them."""
    return st["snap"].copy_(torch.from_numpy(st["out"])) if "snap" in st else st["out"]


def run(st):
    case, s = st["case"], st.get("solver")
    if case["kind"] == "kernels":
        return _run_kernels(st)
    if case["kind"] == "batch":
        for x, h in enumerate(st["host"]):
            s.uploadState(x, h)
        s.run(st["dt"], case["steps"])
        out = [s.downloadState(x) for x in range(len(st["host"]))]
        return out if case["precision"] == "fp64" else [torch.from_numpy(a).to(torch.float32) for a in out]
    if case["kind"] == "loop":
        s.step(st["dt"])
        s.downloadState(st["out"])
        return _kept(st)
    if case["kind"] == "run":
        s.uploadState(st["host"])
        s.run(st["dt"], case["steps"])
        s.downloadState(st["out"])
        return _kept(st)
    # monitor
    log, rec, left = [], [], case["steps"]
    while left > 0:
        n = min(case["every"], left)
        s.run(st["dt"], n)
        d = s.diagnostics()
        log.append((d["energy"], d["max_e"], d["max_h"]))
        rec.append(s.probeHistory())
        left -= n
    s.downloadState(st["out"])
    keep = np.float64 if case["precision"] == "fp64" else np.float32
    return {"state": _kept(st), "log": np.array(log, dtype=keep), "probes": np.concatenate(rec).astype(keep)}


def _prepare_kernels(case, cor, u):
    """The arrays the reference's DgSolver::initialize keeps on the device, on a vacuum box."""
    g = _Grid(case, cor, None)
    n1, nelt, n2 = case["n1"], case["nx"] * case["ny"] * case["nz"], case["n1"] ** 2
    npts, tfp = nelt * n1 ** 3, nelt * 6 * n2
    d = {"u": u.reshape(6, npts).contiguous(), "k": torch.zeros(6, npts, dtype=F64, device=DEV)}
    d["rhs"] = torch.zeros(6, npts, dtype=F64, device=DEV)
    d["fE"] = torch.zeros(3 * tfp, dtype=F64, device=DEV)
    d["fH"], d["fl"] = torch.zeros_like(d["fE"]), torch.zeros(6 * tfp, dtype=F64, device=DEV)
    d["D"] = g.D.t().contiguous()  # column-major
    w = torch.tensor(_gll(n1)[1], device=DEV)
    d["w3"] = torch.einsum("k,j,i->kji", w, w, w).contiguous()
    d["jac"] = g.J.contiguous()
    for x, a in enumerate("rst"):
        for y, b in enumerate("xyz"):
            d[a + b] = (g.C[x][y] / g.J).contiguous()
    # face points: element-major, faces in the reference's order, p fastest
    ids = torch.arange(npts, device=DEV).reshape(g.shape)
    vm, vp, nrm, da = [], [], [], []
    for dim, side, first in _FACES:
        at = n1 - 1 if side > 0 else 0
        vm.append(ids.select(dim, at).reshape(nelt, n2))
        plus = torch.roll(ids.select(dim, n1 - 1 - at), -side, dims=first)
        if not g.periodic[first]:
            plus = plus.clone()
            plus.select(first, g.shape[first] - 1 if side > 0 else 0).fill_(-1)
        vp.append(plus.reshape(nelt, n2))
        N = [side * g.C[5 - dim][e].select(dim, at).reshape(nelt, n2) for e in range(3)]
        ln = torch.sqrt(N[0] ** 2 + N[1] ** 2 + N[2] ** 2)
        nrm.append(torch.stack([x / ln for x in N]))
        da.append(ln * torch.einsum("q,p->qp", w, w).reshape(1, n2))
    d["vM"] = torch.stack(vm, 1).to(torch.int32).contiguous()
    d["vP"] = torch.stack(vp, 1).to(torch.int32).contiguous()
    d["bc"] = (d["vP"] < 0).to(torch.int32)
    nrm = torch.stack(nrm, 2)  # [3, nelt, 6, n2]
    d["nx"], d["ny"], d["nz"] = (nrm[e].contiguous() for e in range(3))
    d["dA"] = torch.stack(da, 1).contiguous()
    if DEV == "cuda":
        torch.cuda.synchronize()
    return {"case": case, "d": d, "p": {k: v.data_ptr() for k, v in d.items()}, "npts": npts, "tfp": tfp,
            "nelt": nelt, "dt": _dt(case, None)}


def _run_kernels(st):
    p, npts, tfp, n1, nelt = st["p"], st["npts"], st["tfp"], st["case"]["n1"], st["nelt"]
    L = lib()
    u, rhs = [p["u"] + 8 * npts * c for c in range(6)], [p["rhs"] + 8 * npts * c for c in range(6)]
    geo = [p[k] for k in ("D", "w3", "jac", "rx", "sx", "tx", "ry", "sy", "ty", "rz", "sz", "tz")]
    for s in range(5):
        check(L.nw_launch_volume_curl(u[3], u[4], u[5], rhs[0], rhs[1], rhs[2], *geo, 1.0, n1, nelt, None))
        check(L.nw_launch_volume_curl(u[0], u[1], u[2], rhs[3], rhs[4], rhs[5], *geo, -1.0, n1, nelt, None))
        check(L.nw_launch_restrict_faces(p["u"], p["fE"], p["fH"], p["vM"], tfp, npts, None))
        check(L.nw_launch_compute_flux(p["u"], p["fE"], p["fH"], p["vP"], p["bc"], p["nx"], p["ny"], p["nz"], p["fl"],
                                       1.0, tfp, npts, p["vM"], None, None, None, n1 ** 3, npts, None))
        check(L.nw_launch_add_flux(p["fl"], p["vM"], p["dA"], p["rhs"], tfp, npts, None))
        check(L.nw_launch_inv_mass(p["rhs"], p["jac"], p["w3"], nelt, n1 ** 3, npts, None, None, None))
        check(L.nw_launch_lsrk45_update(p["u"], p["k"], p["rhs"], RK_A[s], RK_B[s], st["dt"], npts, npts, None))
    check(L.nw_dev_sync())
    return {"state": st["d"]["u"], "k": st["d"]["k"]}


# --- what a pass cannot do without -----------------------------------------------------------------------


def _step_work(case):
    """Bytes and operations of one step: stage 1 reads u, writes u and k; stages 2-4 read and write u and k; stage 5
    reads u and k and writes u; plus 8 corners, eps and mu per element and stage."""
    n1, nelt = case["n1"], case["nx"] * case["ny"] * case["nz"]
    su = 8 if case["precision"] == "fp64" else 4
    sk = 4 if case["precision"] in ("fp32", "bf16x3") else 8
    nodes = nelt * n1 ** 3
    by = 6 * nodes * (10 * su + 8 * sk) + 5 * nelt * 26 * 8
    # per node and stage: 18 derivatives, their fold into the curls, update; per face point about 90
    return by, 5 * (nodes * (36 * n1 + 36 + 24 + 24) + nelt * 6 * n1 * n1 * 90)


def work(case):
    members = _members(case) if case["kind"] == "batch" else [case]
    by = fl = 0.0
    for c in members:
        b, f = _step_work(c)
        nodes = c["n1"] ** 3 * c["nx"] * c["ny"] * c["nz"]
        if case["kind"] == "kernels":  # the launchers' arrays: metrics, faces and scratch belong to the interface
            faces = 6.0 * c["n1"] ** 2 * c["nx"] * c["ny"] * c["nz"]
            b = 5 * (nodes * 8 * (12 + 20 + 6 + 12 + 1 + 24) + faces * 8 * (12 + 12 + 3 + 6 + 7) + faces * 16)
            by, fl = by + b, fl + f
            continue
        moves = {"loop": 1, "monitor": 1}.get(case["kind"], 2)  # host transfers, as float64
        by += b * case["steps"] + moves * nodes * 48
        fl += f * case["steps"]
    return {"bytes": by, "flops": fl}


# --- the same in 64 bits, without the framework ----------------------------------------------------------

# face f: axis of its points' missing index in [z, y, x, k, j, i], outward side, the grid axis of the neighbour
_FACES = ((4, -1, 1), (5, 1, 2), (4, 1, 1), (5, -1, 2), (3, -1, 0), (3, 1, 0))


class _Grid:
    """Metrics of a box of hexes at the GLL nodes: cofactors C[d][e] = J d(r_d)/d(x_e) and J."""

    def __init__(self, case, corners, media):
        _, dN = _shape(case["n1"])
        z, w, D = _gll(case["n1"])
        self.n1, self.D, self.w0 = case["n1"], torch.tensor(D, device=DEV), float(w[0])
        c = torch.tensor(corners, device=DEV)
        T = [[torch.einsum("zyxa,akji->zyxkji", c[..., e].contiguous(), dN[d]) for e in range(3)] for d in range(3)]
        cross = lambda a, b: [a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]]  # noqa: E731
        self.C = [cross(T[1], T[2]), cross(T[2], T[0]), cross(T[0], T[1])]
        self.J = sum(T[0][e] * self.C[0][e] for e in range(3))
        self.shape = tuple(self.J.shape)
        self.periodic = {0: "z" in case["periodic"], 1: "y" in case["periodic"], 2: "x" in case["periodic"]}
        lift = lambda a: torch.tensor(a, device=DEV).reshape(self.shape[:3] + (1, 1, 1))  # noqa: E731
        self.eps, self.mu = (None, None) if media is None else (lift(media[0]), lift(media[1]))

    def grad(self, f):
        n = self.n1
        lead = f.shape[:3]
        return (torch.matmul(f, self.D.t()), torch.matmul(self.D, f),
                torch.matmul(self.D, f.reshape(lead + (n, n * n))).reshape(f.shape))

    def curl(self, v):
        """J curl v."""
        o = [0.0, 0.0, 0.0]
        for e in range(3):  # component e: its derivatives enter the two other components
            g = self.grad(v[e])
            a, b = (e + 1) % 3, (e + 2) % 3
            da = sum(g[d] * self.C[d][a] for d in range(3))
            db = sum(g[d] * self.C[d][b] for d in range(3))
            o[b] = o[b] - da
            o[a] = o[a] + db
        return o

    def rhs(self, u):
        cE, cH = self.curl(u[0:3]), self.curl(u[3:6])
        r = torch.stack(cH + [-x for x in cE])
        n = self.n1
        for dim, side, first in _FACES:
            at = n - 1 if side > 0 else 0
            M = u.select(dim + 1, at)
            P = torch.roll(u.select(dim + 1, n - 1 - at), -side, dims=first + 1)
            j = P - M
            if not self.periodic[first]:
                wall = self.shape[first] - 1 if side > 0 else 0
                j[0:3].select(first + 1, wall).copy_(-2.0 * M[0:3].select(first + 1, wall))
                j[3:6].select(first + 1, wall).zero_()
            N = [side * self.C[5 - dim][e].select(dim, at) for e in range(3)]
            ln = torch.sqrt(N[0] ** 2 + N[1] ** 2 + N[2] ** 2)
            nr = [x / ln for x in N]
            cross = lambda b: [nr[1] * b[2] - nr[2] * b[1], nr[2] * b[0] - nr[0] * b[2], nr[0] * b[1] - nr[1] * b[0]]  # noqa: E731
            nE, nH = cross(j[0:3]), cross(j[3:6])
            nnE, nnH = cross(nE), cross(nH)
            if self.eps is None:
                a, b, c, d = 0.5, 0.5, 0.5, 0.5
            else:
                zm = torch.sqrt(self.mu / self.eps).reshape(self.shape[:3] + (1, 1))
                zp = torch.roll(zm, -side, dims=first)
                if not self.periodic[first]:
                    wall = self.shape[first] - 1 if side > 0 else 0
                    zp = zp.clone()
                    zp.select(first, wall).copy_(zm.select(first, wall))
                ym, yp = 1.0 / zm, 1.0 / zp
                a, b, c, d = zp / (zp + zm), 1.0 / (zp + zm), yp / (yp + ym), 1.0 / (yp + ym)
            for e in range(3):
                r[e].select(dim, at).add_(ln / self.w0 * (a * nH[e] - b * nnE[e]))
                r[3 + e].select(dim, at).add_(ln / self.w0 * (-c * nE[e] - d * nnH[e]))
        r /= self.J
        if self.eps is not None:
            r[0:3] /= self.eps
            r[3:6] /= self.mu
        return r

    def step(self, u, k, dt):
        for a, b in zip(RK_A, RK_B):
            r = self.rhs(u)
            k.mul_(a).add_(r, alpha=dt)
            u.add_(k, alpha=b)


def _exact_record(g, u, case, pts):
    z, _, _ = _gll(case["n1"])
    L, n = _lengths(case), (case["nx"], case["ny"], case["nz"])
    out = []
    for x in pts:
        el = [min(n[d] - 1, int(x[d] / L[d] * n[d])) for d in range(3)]
        xi = [2.0 * (x[d] / L[d] * n[d] - el[d]) - 1.0 for d in range(3)]
        lag = [torch.tensor([math.prod((xi[d] - z[b]) / (z[a] - z[b]) for b in range(len(z)) if b != a)
                             for a in range(len(z))], dtype=F64, device=DEV) for d in range(3)]
        out.append(torch.einsum("fkji,k,j,i->f", u[:, el[2], el[1], el[0]], lag[2], lag[1], lag[0]))
    return torch.stack(out)


def exact(case, seed):
    if case["kind"] == "batch":
        if case["count"] * case["steps"] > 2500:
            return None
        members = _members(case)
        media = [_media(c, seed + 7919 * x) for x, c in enumerate(members)]
        dt = min(_dt(c, m) for c, m in zip(members, media))
        out = []
        for x, c in enumerate(members):
            cor = _corners(c, seed + 7919 * x)
            g, u = _Grid(c, cor, media[x]), _field(c, seed + 7919 * x, cor)
            k = torch.zeros_like(u)
            for _ in range(c["steps"]):
                g.step(u, k, dt)
            out.append(u.reshape(-1))
        return out
    nodes = case["n1"] ** 3 * case["nx"] * case["ny"] * case["nz"]
    if nodes * case["steps"] > 6e8:
        return None
    cor, media = _corners(case, seed), _media(case, seed)
    g, u, dt = _Grid(case, cor, media), _field(case, seed, cor), _dt(case, media)
    k = torch.zeros_like(u)
    if case["kind"] == "kernels":
        g.step(u, k, dt)
        return {"state": u.reshape(6, nodes), "k": k.reshape(6, nodes)}
    if case["kind"] != "monitor":
        for _ in range(case["steps"]):
            g.step(u, k, dt)
        return u.reshape(-1)
    w = torch.tensor(_gll(case["n1"])[1], device=DEV)
    dv = g.J * torch.einsum("k,j,i->kji", w, w, w)
    pts, log, rec = _probe_points(case, seed), [], []
    for n in range(1, case["steps"] + 1):
        g.step(u, k, dt)
        rec.append(_exact_record(g, u, case, pts))
        if n % case["every"] == 0 or n == case["steps"]:
            e2, h2 = (u[0:3] ** 2).sum(0), (u[3:6] ** 2).sum(0)
            en = 0.5 * ((e2 if g.eps is None else g.eps * e2) + (h2 if g.mu is None else g.mu * h2)) * dv
            log.append([float(en.sum()), float(e2.max().sqrt()), float(h2.max().sqrt())])
    return {"state": u.reshape(-1), "log": torch.tensor(log, dtype=F64), "probes": torch.stack(rec)}
