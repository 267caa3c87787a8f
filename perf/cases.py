"""Performance cases: the calls a program built on this library makes in
earnest, over the sizes and options it makes them with.

Families (the "kind" of a case):

  stage      one substep of the SSPRK3 cycle on one patch: asx_substep, the
             state's boundary fill, asx_con2prim_group, the primitives'
             boundary fill -- what every time step of an evolution is made of
  batch      one SSPRK3 step of a plan over many uneven patches
             (asx_batch_step): one GPU's share of a refined grid
  scheduled  the right-hand side through the unfused scheduled functions
             (asx_fluxes, asx_source_terms, asx_rhs and the SYNC after each),
             as a host driver that keeps the reference's schedule calls them
  zones      con2prim of independent zones: ideal gas from the plain seed,
             with the learned guess, and on a table with composition
  tmunu      the stress-energy tensor at the vertices (asx_tmunu) into zeroed
             eT, once per substep of a run coupled to the spacetime
  refine     the level operators: a new patch's prolongation, or the
             coarse-fine ghost fill followed by the restriction

The data are the Fishbone-Moncrief torus on a Kerr-Schild hole, the
Balsara-1 shock tube, and the zone distributions of the con2prim workloads.
Evolution cases advance in place, as a simulation does.  Launch shapes are
the defaults: what a program gets that tunes nothing.
"""
import ctypes as C
import functools
import math

import torch

from asterx_amd import abi, batch, lib, mlp, seeds, tabeos, torus
from asterx_amd.driver import Evolution
from asterx_amd.patch import Patch

F64 = torch.float64


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest patch a refined run holds, odd extents: launches count
        dict(name="stage-small", kind="stage", flow="torus", nx=22, ny=17, nz=13,
             recon="mp5", flux="LxF"),
        # a regression-sized run on the flat metric
        dict(name="stage-tube-64", kind="stage", flow="tube", nx=64, ny=64, nz=64,
             recon="ppm", flux="HLLE"),
        # the standard production patch of the disk runs
        dict(name="stage-torus-192", kind="stage", flow="torus", nx=192, ny=192, nz=192,
             recon="wenoz", flux="HLLE"),
        # the largest patch, ragged extents, the other method and flux
        dict(name="stage-torus-ragged", kind="stage", flow="torus", nx=253, ny=231, nz=246,
             recon="mp5", flux="LxF"),
        # the disk on a tabulated equation of state
        dict(name="stage-table-128", kind="stage", flow="table", nx=128, ny=128, nz=128,
             recon="wenoz", flux="HLLE"),
        # one GPU's share of a refined grid: uneven boxes of 16 to 64 cells
        dict(name="batch-48", kind="batch", patches=48, recon="wenoz", flux="HLLE"),
        # the reference's schedule, call by call, fourth-order sources, z vector
        dict(name="scheduled-96", kind="scheduled", nx=96, ny=80, nz=101, recon="ppm",
             flux="LxF", var="z_vec", order=4),
        # con2prim of many zones from the previous step's primitives
        dict(name="zones-ideal", kind="zones", eos="ideal", zones=4000037, cold=False),
        # the same solver started by the learned guess, from a cold start
        dict(name="zones-guess", kind="zones", eos="guess", zones=16777216, cold=True),
        # con2prim with composition on the table
        dict(name="zones-table", kind="zones", eos="table", zones=1000003, cold=False),
        # the tensor a coupled spacetime reads after every substep
        dict(name="tmunu-192", kind="tmunu", nx=192, ny=192, nz=192, order=4),
        # the coarse-fine ghost fill and restriction of one level's substep
        dict(name="refine-96", kind="refine", nx=96, ny=96, nz=96, order=3, region=1),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _extents(rng, lo, hi, most):
    while True:
        n = [_log_int(rng, lo, hi) for _ in range(3)]
        if n[0] * n[1] * n[2] <= most:
            return dict(nx=n[0], ny=n[1], nz=n[2])


def draw(rng):
    kind = rng.choice(["stage", "stage", "stage", "table", "batch", "scheduled", "ideal",
                       "guess", "ztable", "tmunu", "refine"])
    recon = rng.choice(["wenoz", "wenoz", "mp5", "ppm"])
    flux = rng.choice(["HLLE", "HLLE", "LxF"])
    if kind == "stage":
        flow = rng.choice(["torus", "torus", "tube"])
        big = dict(_extents(rng, 12, 256, 10 ** 7 if flow == "torus" else 2 * 10 ** 6))
        return dict(kind="stage", flow=flow, recon=recon, flux=flux, **big)
    if kind == "table":
        return dict(kind="stage", flow="table", recon=recon, flux=flux,
                    **_extents(rng, 16, 144, 2 * 10 ** 6))
    if kind == "batch":
        return dict(kind="batch", patches=_log_int(rng, 4, 64), recon=recon, flux=flux)
    if kind == "scheduled":
        return dict(kind="scheduled", recon=rng.choice(["wenoz", "mp5", "ppm", "minmod"]),
                    flux=flux, var=rng.choice(["v_vec", "z_vec"]), order=rng.choice([2, 4]),
                    **_extents(rng, 12, 160, 2 * 10 ** 6))
    if kind == "ideal":
        return dict(kind="zones", eos="ideal", zones=_log_int(rng, 10 ** 4, 10 ** 7),
                    cold=rng.random() < 0.5)
    if kind == "guess":
        return dict(kind="zones", eos="guess", zones=_log_int(rng, 10 ** 4, 10 ** 7),
                    cold=rng.random() < 0.5)
    if kind == "ztable":
        return dict(kind="zones", eos="table", zones=_log_int(rng, 10 ** 4, 2 * 10 ** 6),
                    cold=False)
    if kind == "tmunu":
        return dict(kind="tmunu", order=rng.choice([2, 4]), **_extents(rng, 12, 256, 10 ** 7))
    n = _extents(rng, 8, 64, 2 * 10 ** 5)
    return dict(kind="refine", order=rng.choice([1, 3, 3, 5]), region=rng.choice([0, 1]),
                **{k: 2 * v for k, v in n.items()})


# ---------------------------------------------------------------------------
# Parameters, patches and initial data
# ---------------------------------------------------------------------------
NG = 3
GROUPS = {  # outputs by kind: one buffer each
    "rho": ["rho"], "vel": ["velx", "vely", "velz"], "eps": ["eps"], "press": ["press"],
    "temperature": ["temperature"], "entropy": ["entropy"], "Ye": ["Ye"],
    "Bvec": ["Bvecx", "Bvecy", "Bvecz"], "dB": abi.DB, "zvec": abi.ZS[:3], "svec": abi.ZS[3:],
    "flag": ["con2prim_flag"]}
STATE_GROUPS = {
    "dens": ["dens"], "mom": ["momx", "momy", "momz"], "tau": ["tau"], "DEnt": ["DEnt"],
    "DYe": ["DYe"], "Avec_x": ["Avec_x"], "Avec_y": ["Avec_y"], "Avec_z": ["Avec_z"],
    "Psi": ["Psi"]}
SYNC_PRIMS = batch.SYNC_PRIMS
PTR = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731


@functools.lru_cache(maxsize=1)
def _table():
    """The synthetic 234 x 180 x 50 table, read once by a program."""
    return tabeos.Table(tabeos.build(), device="cuda")


def _params(case):
    kw = {}
    if "recon" in case:
        kw = dict(reconstruction_method=case["recon"], flux_type=case["flux"],
                  recon_type=case.get("var", "v_vec"),
                  local_spatial_order=case.get("order", 2))
    if case["kind"] == "tmunu":
        kw = dict(tmunu_interp_order=case["order"])
    eos = case.get("eos")
    if eos in ("ideal", "guess"):
        return abi.params(gl_gamma=5.0 / 3.0, eps_max=1e8, rho_max=1e8, rho_abs_min=1e-12,
                          vw_lim=1e3, B_lim=1e3, c2p_tol=1e-10)
    if eos == "table" or case.get("flow") == "table":
        return _table().attach(abi.params(
            c2p_prime="Palenzuela", c2p_second="None", use_temperature=1, use_press_atmo=0,
            thermal_eos_atmo=1, rho_abs_min=1e-14, t_atmo=0.01, Ye_atmo=0.5, c2p_tol=1e-10,
            max_iter=100, vw_lim=1e3, B_lim=1e3, ye_min=0.035, ye_max=0.55,
            reconstruct_with_temperature=1, **kw))
    if case.get("flow") == "tube":
        return abi.params(gl_gamma=5.0 / 3.0, eps_max=1e8, rho_max=1e8, rho_abs_min=1e-8, **kw)
    return torus.eos_params(torus.TorusSpec(), **kw)


def _alloc(p, groups):
    """The groups' fields as views of one buffer per group; returns the buffers."""
    out = {}
    for key, names in groups.items():
        out[key] = torch.zeros((len(names),) + p.shape(names[0]), dtype=F64, device="cuda")
        for i, name in enumerate(names):
            p.arr[name] = out[key][i]
    return out


def _v2c(a):
    a = a[:-1] + a[1:]
    a = a[:, :-1] + a[:, 1:]
    return (a[..., :-1] + a[..., 1:]) / 8


def _sym(f, names=("gxx", "gxy", "gxz", "gyy", "gyz", "gzz")):
    xx, xy, xz, yy, yz, zz = (f[n] for n in names)
    return ((xx, xy, xz), (xy, yy, yz), (xz, yz, zz))


def _low(g, v):
    return [sum(g[i][j] * v[j] for j in range(3)) for i in range(3)]


def _dot(a, b):
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]


def _flow(case, seed, n, extra=()):
    """A patch of n cells with the case's initial data: primitives, metric,
    vector potential, B from A and the conserved state, ghosts included.
    Returns (patch, parameters, output buffers)."""
    par, be = _params(case), lib.backend()
    flow = case.get("flow", "torus")
    if flow == "tube":
        L, x0 = 1.0, (-0.5,) * 3
        dx = tuple(L / m for m in n)
    else:  # no vertex on the axis or at the centre
        dx = tuple(80.0 / m for m in n)
        x0 = tuple(-40.0 + 0.25 * d for d in dx)
    p = Patch(n, NG, x0, dx, device="cuda")
    outs = _alloc(p, {**GROUPS, **STATE_GROUPS})
    for name in abi.ADM + abi.SAVED + ["aster_mask_cc"] + abi.DBSTAG + list(extra):
        p.alloc(name)
    if flow == "tube":
        seeds.minkowski(p)
        seeds.balsara(p, "Balsara1", "x", gamma=par.gl_gamma, perturb=1e-3, seed=seed)
        seeds.post_initial(p, par.gl_gamma)
    else:
        spec = torus.TorusSpec(seed=seed)
        q = Patch(n, NG, x0, dx, device="cuda")
        torus.set_metric(q, spec)
        disk = torus.set_disk(q, spec)
        torus.set_avec(q, spec, 1.0)
        rho, press = q["rho"], q["press"]
        if flow == "table":
            rel = rho / rho[disk].max()
            rho = torch.clamp(1e-4 * rel, min=1e-14)
            temp = 0.02 + 10.0 * rel ** (2.0 / 3.0)
            temp = temp * (1 + 1e-3 * (press / press.max()))  # the seeded perturbation
            ye = torch.clamp(0.5 - 0.4 * torch.sqrt(rel), 0.05, 0.5)
            press, eps, ent = torus.eos_from_rho_temp(be, par, rho, temp, ye)
        else:
            rho = torch.clamp(rho, min=par.rho_abs_min)
            press = torch.clamp(press, min=par.p_atmo)
            eps = press / (rho * (par.gl_gamma - 1))
            temp = (par.gl_gamma - 1) * eps
            ent = temp * rho ** (1 - par.gl_gamma)
            ye = torch.full_like(rho, 0.5)
        for name in abi.ADM + ["velx", "vely", "velz", "Avec_x", "Avec_y", "Avec_z"]:
            p.arr[name].copy_(q[name])
        for name, v in (("rho", rho), ("press", press), ("eps", eps), ("temperature", temp),
                        ("entropy", ent), ("Ye", ye)):
            p.arr[name].copy_(v)
        del q
    ev = Evolution(be, p, par, bc="copy")

    def b_from_a():
        be.bstag_from_A(p.struct())
        ev.sync(abi.DBSTAG)
        be.dB_from_bstag(p.struct())
        ev.sync(abi.DB)
        be.B_from_dB(p.struct())
        ev.sync(["Bvecx", "Bvecy", "Bvecz"])

    b_from_a()
    if flow != "tube":
        scale = math.sqrt(torus.plasma_beta_min(p, disk) / spec.beta_min)
        for name in ("Avec_x", "Avec_y"):
            p.arr[name].mul_(scale)
        b_from_a()
    vel = [p["velx"], p["vely"], p["velz"]]
    vl = _low(_sym({m: _v2c(p[m]) for m in ("gxx", "gxy", "gxz", "gyy", "gyz", "gzz")}), vel)
    w = 1 / torch.sqrt(1 - _dot(vl, vel))
    hw2 = (p["rho"] * (1 + p["eps"]) + p["press"]) * w * w
    for i, c in enumerate("xyz"):
        p.arr["zvec_" + c].copy_(w * vel[i])
        p.arr["svec_" + c].copy_(hw2 * vel[i])
        p.arr["saved_vel" + c].copy_(vel[i])
    for c in ("rho", "eps", "Ye"):
        p.arr["saved_" + c].copy_(p[c])
    be.prim2con(p.struct())
    ev.sync(abi.CONS + abi.DB)
    return p, par, outs


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------
def _slots(names):
    return (C.c_int32 * len(names))(*[abi.SLOT[m] for m in names])


def _prepare_stage(case, seed):
    p, par, outs = _flow(case, seed, (case["nx"], case["ny"], case["nz"]))
    for name in abi.DBSTAG:  # con2prim takes dB from A
        del p.arr[name]
    L, dt = lib.lib(), 0.2 * min(p.dx)
    own = {m: p.arr[m] for m in abi.STATE}
    bufs, keys = [own], [{k: outs[k] for k in STATE_GROUPS}]
    for _ in range(2):
        q = Patch(p.n, p.ng, p.x0, p.dx, device="cuda")
        keys.append(_alloc(q, STATE_GROUPS))
        bufs.append({m: q.arr[m] for m in abi.STATE})
    structs, states = [], []
    for b in bufs:
        p.arr.update(b)
        structs.append(p.struct())
        states.append(p.state())
    p.arr.update(own)
    st, pr = _slots(abi.STATE), _slots(SYNC_PRIMS)
    kind, calls, results = abi.BC["copy"], [], []
    for s, (c0, c1, c2) in enumerate(batch.SSPRK3):
        i, o = batch.STAGE_IN[s], batch.STAGE_OUT[s]
        calls.append((
            (L.asx_substep, (C.byref(structs[i]), C.byref(states[0]), C.byref(states[o]), c0, c1,
                             c2 * dt, C.byref(par), None)),
            (L.asx_bc_fill_many, (C.byref(structs[o]), len(abi.STATE), st, kind, None)),
            (L.asx_con2prim_group, (C.byref(structs[o]), C.byref(par), None, None)),
            (L.asx_bc_fill_many, (C.byref(structs[o]), len(SYNC_PRIMS), pr, kind, None))))
        results.append(_flags_whole({**{k: outs[k] for k in GROUPS}, **keys[o]}))
    return dict(kind="stage", patch=p, par=par, keep=(bufs, structs, states), calls=calls,
                results=results, at=0, dt=dt)


def _flags_whole(res):
    """The con2prim flags (whole numbers held as doubles) as the integers of
    their bits, so that they are compared as the whole values they are."""
    res["flag"] = res["flag"].view(torch.int64)
    return res


def _run_stage(s):
    k = s["at"]
    s["at"] = (k + 1) % 3
    for f, a in s["calls"][k]:
        abi.check("asx", f(*a))
    return s["results"][k]


BATCH_SOURCE = 128


def _prepare_batch(case, seed):
    """Patches cut from the torus at random offsets, 16 to 64 cells an edge;
    every field's patches lie one after another in one buffer."""
    src, par, _ = _flow(case, seed, (BATCH_SOURCE,) * 3)
    boxes = batch.sample_boxes(src.n, case["patches"], seed=2024 + case["patches"])
    groups = {**GROUPS, **STATE_GROUPS}
    outs, at = {}, {}
    for key, names in groups.items():
        total = 0
        for n, _ in boxes:
            ex, ey, ez = abi.extents(n, NG, abi.centering(names[0]))
            total += len(names) * ex * ey * ez
        outs[key], at[key] = torch.zeros(total, dtype=F64, device="cuda"), 0
    patches = []
    for n, o in boxes:
        q = batch.cut_patch(src, n, o, names=abi.ADM + abi.SAVED + ["aster_mask_cc"])
        for key, names in groups.items():
            for name in names:
                ex, ey, ez = abi.extents(n, NG, abi.centering(name))
                v = outs[key][at[key]:at[key] + ex * ey * ez].view(ez, ey, ex)
                at[key] += ex * ey * ez
                v.copy_(src.arr[name][o[2]:o[2] + ez, o[1]:o[1] + ey, o[0]:o[0] + ex])
                q.arr[name] = v
        patches.append(q)
    dt = 0.2 * min(src.dx)
    plan = batch.Plan(lib.lib(), patches, par, dt, bc="copy")
    return dict(kind="batch", plan=plan, patches=patches, par=par, dt=dt,
                results=_flags_whole(outs))


def _run_batch(s):
    s["plan"].step(1)
    return s["results"]


RHS_GROUPS = {"hydro": ["densrhs"], "mom": ["momxrhs", "momyrhs", "momzrhs"], "tau": ["taurhs"],
              "DEnt": ["DEntrhs"], "DYe": ["DYe_rhs"], "A_x": ["Avec_x_rhs"],
              "A_y": ["Avec_y_rhs"], "A_z": ["Avec_z_rhs"], "Psi": ["Psi_rhs"]}


def _prepare_scheduled(case, seed):
    p, par, _ = _flow(case, seed, (case["nx"], case["ny"], case["nz"]),
                      extra=abi.FLUX + abi.AUX)
    outs = _alloc(p, RHS_GROUPS)
    ev = Evolution(lib.backend(), p, par, bc="linear")
    ev.sync(abi.DBSTAG)
    return dict(kind="scheduled", patch=p, par=par, ev=ev, results=outs)


def _run_scheduled(s):
    s["ev"].rhs()
    return s["results"]


def _unit(g, v):
    return v / torch.sqrt(_dot(v, torch.stack(_low(g, v))))


def _prepare_zones(case, seed):
    nz, table = case["zones"], case["eos"] == "table"
    par, L = _params(case), lib.lib()
    gen = torch.Generator(device="cuda").manual_seed(seed)
    uni = lambda a, b, *s: a + (b - a) * torch.rand(  # noqa: E731
        *s, nz, dtype=F64, device="cuda", generator=gen)
    log = lambda a, b: torch.exp(uni(math.log(a), math.log(b)))  # noqa: E731
    off = uni(-0.1 / 3, 0.1 / 3, 6)
    gm = torch.stack([1 + off[0], off[1], off[2], 1 + off[3], off[4], 1 + off[5]])
    g = ((gm[0], gm[1], gm[2]), (gm[1], gm[3], gm[4]), (gm[2], gm[4], gm[5]))
    rho = log(1e-12, 1e-4) if table else log(1e-10, 1e-2)
    w = uni(1.0, 10.0)
    nrm = lambda: torch.randn(3, nz, dtype=F64, device="cuda", generator=gen)  # noqa: E731
    vel = _unit(g, nrm()) * torch.sqrt(1 - 1 / (w * w))
    nb = _unit(g, nrm())
    vl = torch.stack(_low(g, vel))
    B = nb * torch.sqrt(rho * log(1e-4, 1e2) / (1 / (w * w) + _dot(nb, vl) ** 2))
    if table:
        temp, ye = log(0.05, 80.0), uni(0.06, 0.5)
        press, eps, _ = torus.eos_from_rho_temp(lib.backend(), par, rho, temp, ye)
    else:
        press = rho * log(1e-6, 1e2)
        eps = press / (rho * (par.gl_gamma - 1))
        temp, ye = (par.gl_gamma - 1) * eps, torch.full_like(rho, 0.5)
    sq = torch.sqrt(_det(g))
    Bl = torch.stack(_low(g, B))
    bst = w * _dot(B, vl)
    b2 = (_dot(B, Bl) + bst * bst) / (w * w)
    hw2 = w * w * (rho * (1 + eps) + press + b2)
    dens = sq * rho * w
    mom = sq * (hw2 * vl - bst * (Bl / w + bst * vl))
    tau = sq * (hw2 - (press + 0.5 * b2) - bst * bst) - dens
    cons = torch.cat([dens[None], mom, tau[None], sq * B] +
                     ([(dens * ye)[None]] if table else []))
    if case["cold"]:
        zero = torch.zeros_like(rho)
        sd = [dens / sq, tau / dens, zero, zero, zero]
    else:
        sd = [x * uni(0.99, 1.01) for x in (rho, eps, vel[0], vel[1], vel[2])]
    seed_t = torch.stack(sd + ([ye, temp] if table else [])).contiguous()
    prim = torch.empty((9 if table else 8, nz), dtype=F64, device="cuda")
    flag = torch.empty(nz, dtype=F64, device="cuda")
    iters = torch.empty(nz, dtype=torch.int32, device="cuda")
    keep = [cons.contiguous(), gm.contiguous(), seed_t, prim, flag, iters, par]
    args = [nz, PTR(keep[0]), PTR(keep[1]), PTR(seed_t)]
    tail = [PTR(prim), PTR(flag), PTR(iters)]
    res = {"rho": prim[0], "eps": prim[1], "press": prim[2], "vel": prim[3:6], "w": prim[6],
           "temperature": prim[7], "flag": flag}
    if table:
        f, res["Ye"] = L.asx_c2p_batch_ye, prim[8]
    elif case["eos"] == "guess":
        blob = torch.from_numpy(mlp.load()).cuda()
        back = torch.empty(nz, dtype=torch.int32, device="cuda")
        keep += [blob, back]
        f, args, tail = L.asx_c2p_batch_mlp, args + [PTR(blob), 8], tail + [PTR(back)]
    else:
        f = L.asx_c2p_batch
    if table:
        truth = dict(rho=rho, eps=eps, press=press, vel=vel, w=w, temperature=temp, Ye=ye)
    else:  # the solver's temperature floor
        T = temp.clamp(min=par.t_atmo)
        truth = dict(rho=rho, eps=T / (par.gl_gamma - 1), press=rho * T, vel=vel, w=w,
                     temperature=T)
    return dict(kind="zones", f=f, args=args + tail + [C.byref(par), None], keep=keep,
                results=_flags_whole(res), truth=truth)


def _run_zones(s):
    abi.check("asx_c2p_batch", s["f"](*s["args"]))
    return s["results"]


def _prepare_tmunu(case, seed):
    p, par, _ = _flow(case, seed, (case["nx"], case["ny"], case["nz"]))
    for name in abi.STATE + abi.DB + abi.DBSTAG + abi.SAVED + abi.ZS:
        if name in p:
            del p.arr[name]
    out = _alloc(p, {"eT": abi.TMUNU})["eT"]
    return dict(kind="tmunu", patch=p, par=par, struct=p.struct(), eT=out)


def _run_tmunu(s):
    s["eT"].zero_()
    abi.check("asx_tmunu", lib.lib().asx_tmunu(C.byref(s["struct"]), C.byref(s["par"]), None))
    return s["eT"]


def _prepare_refine(case, seed):
    """A coarse patch of n cells and the fine patch (n cells) over its middle half."""
    n = (case["nx"], case["ny"], case["nz"])
    c, par, couts = _flow(case, seed, n)
    lo = [m // 4 for m in n]
    f = Patch(tuple(2 * (m // 2) for m in n), NG,
              tuple(c.x0[d] + lo[d] * c.dx[d] for d in range(3)),
              tuple(d / 2 for d in c.dx), device="cuda")
    fouts = _alloc(f, STATE_GROUPS)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    for name in abi.STATE:
        big = c.arr[name].abs().max()
        f.arr[name].copy_(big * torch.rand(f.shape(name), dtype=F64, device="cuda",
                                           generator=gen))
    couts = {k: couts[k] for k in STATE_GROUPS}
    for name in list(c.arr):
        if name not in abi.STATE:
            del c.arr[name]
    return dict(kind="refine", c=c, f=f, cs=c.struct(), fs=f.struct(), order=case["order"],
                region=case["region"], slots=_slots(abi.STATE),
                results={"coarse": couts, "fine": fouts})


def _run_refine(s):
    L, m = lib.lib(), len(abi.STATE)
    abi.check("asx_prolongate", L.asx_prolongate(
        C.byref(s["cs"]), C.byref(s["fs"]), m, s["slots"], s["order"], s["region"], None))
    if s["region"] == 1:
        abi.check("asx_restrict", L.asx_restrict(
            C.byref(s["fs"]), C.byref(s["cs"]), m, s["slots"], None))
        return s["results"]
    return s["results"]["fine"]


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(state):
    return globals()["_run_" + state["kind"]](state)


# ---------------------------------------------------------------------------
# Work and tolerance
# ---------------------------------------------------------------------------
RECON_FLOPS = {"minmod": 30, "ppm": 65, "wenoz": 115, "mp5": 90}  # per cell, variable, axis


def work(case):
    """Bytes: each grid function read or written once per point; operations:
    those of the formulas, + - * / sqrt counted 1."""
    k = case["kind"]
    n = case.get("nx", 1) * case.get("ny", 1) * case.get("nz", 1)
    if k in ("stage", "batch"):
        stages = 1
        if k == "batch":
            boxes = batch.sample_boxes((BATCH_SOURCE,) * 3, case["patches"],
                                       seed=2024 + case["patches"])
            n, stages = sum(b[0] * b[1] * b[2] for b, _ in boxes), 3
        # read: 12 primitives, 11 state, 16 ADM, 6 saved, 11 previous-stage
        # fields in two stages of three; written: 11 state, 12 primitives,
        # 3 dB, 6 z and s, 6 saved, flag, mask
        fields = 12 + 11 + 16 + 6 + 11 * 2 / 3 + 11 + 12 + 3 + 6 + 6 + 2
        return dict(bytes=8 * fields * n * stages,
                    flops=(3 * (9 * RECON_FLOPS[case["recon"]] + 450) + 1200 + 900) * n * stages)
    if k == "scheduled":
        # read: 9 primitives reconstructed, eps, 3 normal fields, 16 ADM, 4 A
        # and Psi; written: 30 fluxes, 7 aux, 11 right-hand sides
        return dict(bytes=8 * (13 + 16 + 4 + 30 + 7 + 11) * n,
                    flops=(3 * (9 * RECON_FLOPS[case["recon"]] + 450) + 1200) * n)
    if k == "zones":
        rows = {"ideal": 8 + 6 + 5 + 9, "guess": 8 + 6 + 5 + 9, "table": 9 + 6 + 7 + 10}
        return dict(bytes=(8 * rows[case["eos"]] + 4) * case["zones"],
                    flops={"ideal": 1100, "guess": 830 + 9088, "table": 2500}[case["eos"]] *
                    case["zones"])
    if k == "tmunu":
        return dict(bytes=8 * (9 + 10 + 10) * n, flops=(9 * (2 * case["order"] * 21 // 4) + 250) * n)
    fields = len(abi.STATE)
    if case["region"] == 0:
        return dict(bytes=9 * fields * n, flops=2 * case["order"] * 2 * fields * n)
    ghosts = 1.0
    for d in "xyz":
        ghosts *= case["n" + d] + 2 * NG
    return dict(bytes=8 * fields * (1.125 * (ghosts - n) + n / 8 + n / 2), flops=fields * n)


def tolerance(case):
    """About four times the difference from exact() over the drawn ranges:
    rounding where the path is explicit; con2prim's stopping rule (1e-10 in
    the solver's unknown), amplified in cold or fast zones, where it solves;
    the table's coarse energy inversion near its floor.  Flags and other
    whole values may differ where a zone sits on a branch."""
    k = case["kind"]
    if k == "refine":
        return {"rel": 1e-15, "max": 4e-15}
    if k == "tmunu":
        return {"rel": 2e-15, "max": 2e-14}
    if k == "scheduled":
        return {"rel": 2e-12, "max": 1e-10}
    if k == "zones":
        rel, most = (8e-9, 4e-8) if case["eos"] == "table" else (2e-9, 2e-7)
    else:
        rel, most = (1.5e-4, 5e-2) if case.get("flow") == "table" else (2e-9, 2e-6)
    return {"rel": rel, "max": most, "differ": 1e-5}


# ---------------------------------------------------------------------------
# The same results in 64 bits with plain torch
# ---------------------------------------------------------------------------
def _det(g):
    return (g[0][0] * (g[1][1] * g[2][2] - g[1][2] ** 2) -
            g[0][1] * (g[0][1] * g[2][2] - g[1][2] * g[0][2]) +
            g[0][2] * (g[0][1] * g[1][2] - g[1][1] * g[0][2]))


def _inv(g):
    d = _det(g)
    xx = (g[1][1] * g[2][2] - g[1][2] ** 2) / d
    xy = (g[0][2] * g[1][2] - g[0][1] * g[2][2]) / d
    xz = (g[0][1] * g[1][2] - g[0][2] * g[1][1]) / d
    yy = (g[0][0] * g[2][2] - g[0][2] ** 2) / d
    yz = (g[0][1] * g[0][2] - g[0][0] * g[1][2]) / d
    zz = (g[0][0] * g[1][1] - g[0][1] ** 2) / d
    return ((xx, xy, xz), (xy, yy, yz), (xz, yz, zz))


def _ext(a, ng, kind):
    """Interior array -> full extent, ghosts by copy or linear extrapolation, x, y, z in turn."""
    for ax in (2, 1, 0):
        m = a.shape[ax]
        lo, hi = a.narrow(ax, 0, 1), a.narrow(ax, m - 1, 1)
        d = (ng - torch.arange(ng, device=a.device, dtype=a.dtype)).reshape(
            [-1 if x == ax else 1 for x in range(3)])
        if kind == "copy":
            l, r = lo.expand_as(lo * d), hi.expand_as(hi * d)
        else:
            l = lo + d * (lo - a.narrow(ax, 1, 1))
            r = hi + d.flip(ax) * (hi - a.narrow(ax, m - 2, 1))
        a = torch.cat([l, a, r], ax)
    return a


def _inner(a, ng=NG):
    return a[ng:-ng, ng:-ng, ng:-ng]


def _minmod(x, y):
    r = torch.where(x.abs() < y.abs(), x, y)
    return torch.where(torch.signbit(x) == torch.signbit(y), r, torch.zeros_like(r))


def _weno(s, eps):
    """The value on the upper side of cell s[2] (WENO-Z, fifth order)."""
    b = [13 / 12 * (s[i] - 2 * s[i + 1] + s[i + 2]) ** 2 for i in range(3)]
    b[0] = b[0] + (s[0] - 4 * s[1] + 3 * s[2]) ** 2 / 4 + eps
    b[1] = b[1] + (s[1] - s[3]) ** 2 / 4 + eps
    b[2] = b[2] + (3 * s[2] - 4 * s[3] + s[4]) ** 2 / 4 + eps
    t = (b[0] - b[2]).abs()
    a = [c * (1 + t / x) for c, x in zip((0.1, 0.6, 0.3), b)]
    q = (2 * s[0] - 7 * s[1] + 11 * s[2], -s[1] + 5 * s[2] + 2 * s[3],
         2 * s[2] + 5 * s[3] - s[4])
    return sum(x * y for x, y in zip(a, q)) / (6 * (a[0] + a[1] + a[2]))


def _mp5(s, alpha):
    ul = (2 * s[0] - 13 * s[1] + 47 * s[2] + 27 * s[3] - 3 * s[4]) / 60
    dm_ = s[2] - s[1]
    ump = s[2] + _minmod(s[3] - s[2], alpha * dm_)
    dm, d, dp = (s[i] - 2 * s[i + 1] + s[i + 2] for i in range(3))
    dmp = _minmod(_minmod(4 * d - dp, 4 * dp - d), _minmod(d, dp))
    dmm = _minmod(_minmod(4 * dm - d, 4 * d - dm), _minmod(dm, d))
    uul, umd = s[2] + alpha * dm_, (s[2] + s[3]) / 2 - dmp / 2
    ulc = s[2] + dm_ / 2 + 4 / 3 * dmm
    lo = torch.maximum(torch.minimum(s[2], torch.minimum(s[3], umd)),
                       torch.minimum(s[2], torch.minimum(uul, ulc)))
    hi = torch.minimum(torch.maximum(s[2], torch.maximum(s[3], umd)),
                       torch.maximum(s[2], torch.maximum(uul, ulc)))
    return torch.where((ul - s[2]) * (ul - ump) <= 1e-10, ul, ul + _minmod(lo - ul, hi - ul))


def _ppm(s, p, par, is_rho):
    zero = torch.zeros_like(s[2])

    def slope(i):
        a, b, c = s[i - 1], s[i], s[i + 1]
        d = 0.5 * (c - a)
        lim = torch.minimum(d.abs(), torch.minimum(2 * (b - a).abs(), 2 * (c - b).abs()))
        return torch.where((c - b) * (b - a) > 0, torch.sign(d) * lim, zero)

    dl, dc, dr = slope(1), slope(2), slope(3)
    lo = 0.5 * (s[1] + s[2]) + (dl - dc) / 6
    up = 0.5 * (s[2] + s[3]) + (dc - dr) / 6
    if is_rho and par.ppm_shock_detection:
        di, dpr = s[3] - s[1], p[3] - p[1]
        touch = (par.poly_k * par.poly_gamma * di.abs() * torch.minimum(p[1], p[3]) >=
                 dpr.abs() * torch.minimum(s[1], s[3]))
        d2m, d2p = s[2] - 2 * s[1] + s[0], s[4] - 2 * s[3] + s[2]
        big = di.abs() - par.ppm_eps_shock * torch.minimum(s[1].abs(), s[3].abs()) > 0
        eta = torch.where((d2m * d2p < 0) & big, -(d2p - d2m) / (6 * di), zero)
        eta = (par.ppm_eta1 * (eta - par.ppm_eta2)).clamp(0, 1)
        eta = torch.where(touch, eta, zero)
        lo = (1 - eta) * lo + eta * (s[1] + 0.5 * dl)
        up = (1 - eta) * up + eta * (s[3] - 0.5 * dr)
    flat = (up - s[2]) * (s[2] - lo) <= 0
    d = up - lo
    g6 = 6 * d * (s[2] - 0.5 * (lo + up))
    nlo = torch.where(g6 > d * d, 3 * s[2] - 2 * up, lo)
    nup = torch.where(g6 < -d * d, 3 * s[2] - 2 * lo, up)
    return torch.where(flat, s[2], nlo), torch.where(flat, s[2], nup)


def _sides(case, par, s, p, is_rho):
    m = case["recon"]
    if m == "wenoz":
        return _weno(s[::-1], par.weno_eps), _weno(s, par.weno_eps)
    if m == "mp5":
        return _mp5(s[::-1], par.mp5_alpha), _mp5(s, par.mp5_alpha)
    if m == "ppm":
        return _ppm(s, p, par, is_rho)
    d = _minmod(s[3] - s[2], s[2] - s[1]) / 2
    return s[2] - d, s[2] + d


class _Ideal:
    def __init__(self, par):
        self.g, self.par, self.ye = par.gl_gamma, par, (par.ye_min, par.ye_max)

    def of_recon(self, rho, th, ye):
        eps = th / (rho * (self.g - 1))
        return eps, th, (self.g - 1) * eps / (eps + 1 / self.g)

    def of_eps(self, rho, eps, ye):
        t = (self.g - 1) * eps
        return rho * t, t, t * rho ** (1 - self.g), eps

    def of_temp(self, rho, t, ye):
        return rho * t, t / (self.g - 1), t * rho ** (1 - self.g)

    def atmo(self):
        p = self.par
        rho = max(p.rho_min, p.rho_abs_min)
        t = p.p_atmo / rho if p.use_press_atmo else p.t_atmo
        return rho, t


class _Tab:
    """Trilinear interpolation in (log rho, log T, Ye); T(eps) by bisection."""

    def __init__(self, par):
        t = _table()
        self.par, self.d, self.ax, self.shift = par, t.data, t.axes, t.host["shift"]
        self.emin, self.emax = t.host["eps_min"], t.host["eps_max"]
        self.ye = t.ranges()[2]

    def _at(self, x, ax):
        h = ax[1] - ax[0]
        i = ((x - ax[0]) / h).floor().clamp(0, len(ax) - 2).long()
        return i, (x - ax[i]) / (ax[i + 1] - ax[i])

    def _mix(self, v, lr, lt, ye):
        (i, a), (j, b), (k, c) = (self._at(x, q) for x, q in zip((lr, lt, ye), self.ax))
        n0, n1 = len(self.ax[0]), len(self.ax[1])
        flat, o = self.d[..., v].reshape(-1), i + n0 * (j + n1 * k)
        out = 0
        for dk, wk in ((0, 1 - c), (n0 * n1, c)):
            for dj, wj in ((0, 1 - b), (n0, b)):
                out = out + wk * wj * ((1 - a) * flat[o + dj + dk] + a * flat[o + dj + dk + 1])
        return out

    def _logs(self, rho, t):
        c = lambda x, a: torch.log(x).clamp(float(a[0]), float(a[-1]))  # noqa: E731
        return c(rho, self.ax[0]), c(t, self.ax[1])

    def of_temp(self, rho, t, ye):
        lr, lt = self._logs(rho, t)
        return (torch.exp(self._mix(0, lr, lt, ye)),
                torch.exp(self._mix(1, lr, lt, ye)) - self.shift, self._mix(3, lr, lt, ye))

    def of_recon(self, rho, th, ye):
        lr, lt = self._logs(rho, th)
        p, eps, _ = self.of_temp(rho, th, ye)
        return eps, p, self._mix(2, lr, lt, ye)

    def of_eps(self, rho, eps, ye):
        lr = self._logs(rho, rho)[0]
        lo = torch.full_like(rho, float(self.ax[1][0]))
        hi = torch.full_like(rho, float(self.ax[1][-1]))
        want = torch.log(eps.clamp(min=self.emin) + self.shift)
        for _ in range(48):
            mid = 0.5 * (lo + hi)
            below = self._mix(1, lr, mid, ye) < want
            lo, hi = torch.where(below, mid, lo), torch.where(below, hi, mid)
        lt = 0.5 * (lo + hi)
        return (torch.exp(self._mix(0, lr, lt, ye)), torch.exp(lt), self._mix(3, lr, lt, ye),
                torch.exp(self._mix(1, lr, lt, ye)) - self.shift)

    def atmo(self):
        return max(math.exp(float(self.ax[0][0])), self.par.rho_abs_min), max(
            math.exp(float(self.ax[1][0])), self.par.t_atmo)


def _eos(case, par):
    return _Tab(par) if case.get("flow") == "table" else _Ideal(par)


def _curl(f, idx, d):
    j, k = (d + 1) % 3, (d + 2) % 3
    A = [f["Avec_x"], f["Avec_y"], f["Avec_z"]]
    return idx[j] * torch.diff(A[k], dim=2 - j) - idx[k] * torch.diff(A[j], dim=2 - k)


def _face_fluxes(case, par, eos, f, idx, d):
    """The ten fluxes through the faces normal to d (zero where no stencil fits)."""
    ax, d1, d2 = 2 - d, (d + 1) % 3, (d + 2) % 3
    N = f["rho"].shape[ax]
    st = lambda a: [a.narrow(ax, m, N - 4) for m in range(5)]  # noqa: E731
    vel = "zvec_" if case.get("var") == "z_vec" else "vel"
    names = ["rho", "entropy", "Ye", "temperature" if case.get("flow") == "table" else "press",
             "Bvec" + "xyz"[d1], "Bvec" + "xyz"[d2], vel + "x", vel + "y", vel + "z"]
    ps = st(f["press"])
    lo, up = zip(*[_sides(case, par, st(f[m]), ps, q == 0) for q, m in enumerate(names)])
    blo = sum((a <= 0).int() for a in lo[:4]) > 0
    bup = sum((a <= 0).int() for a in up[:4]) > 0
    c = [st(f[m])[2] for m in names]  # the low-order method: the cell value
    lo = [torch.where(blo, y, x) for x, y in zip(lo, c)]
    up = [torch.where(bup, y, x) for x, y in zip(up, c)]
    S = [[a.narrow(ax, 0, N - 5) for a in up], [a.narrow(ax, 1, N - 5) for a in lo]]

    def v2f(name):
        a = f[name].narrow(ax, 3, N - 5)
        for t in (2 - d1, 2 - d2):
            a = a.narrow(t, 0, a.shape[t] - 1) + a.narrow(t, 1, a.shape[t] - 1)
        return a / 4

    alp, beta = v2f("alp"), [v2f("beta" + x) for x in "xyz"]
    g = _sym({m: v2f(m) for m in ("gxx", "gxy", "gxz", "gyy", "gyz", "gzz")})
    sq = torch.sqrt(_det(g))
    u = _inv(g)[d][d]
    bn = _curl(f, idx, d).narrow(ax, 3, N - 5) / sq
    U, F, lam = [], [], []
    for rho, ent, ye, th, b1, b2, *v in S:
        eps, p, cs2 = eos.of_recon(rho, th, ye)
        if case.get("var") == "z_vec":
            w = torch.sqrt(1 + _dot(_low(g, v), v))
            v = [x / w for x in v]
        else:
            w = 1 / torch.sqrt(1 - _dot(_low(g, v), v))
        vl = _low(g, v)
        B = [None] * 3
        B[d], B[d1], B[d2] = bn, b1, b2
        vt = [alp * v[i] - beta[i] for i in range(3)]
        ab0, Bl = w * _dot(B, vl), _low(g, B)
        Bsq = _dot(B, Bl)
        bl = [Bl[i] / w + ab0 * vl[i] for i in range(3)]
        bs = (Bsq + ab0 ** 2) / w ** 2
        h, dens = 1 + eps + p / rho, sq * rho * w
        dhw, pm = dens * h * w, p + bs / 2
        mom = [(dhw + sq * (ab0 ** 2 + Bsq)) * vl[i] - sq * ab0 * bl[i] for i in range(3)]
        tau = dhw - dens + sq * (Bsq - pm)
        Bt = [sq * x for x in B]
        bw = B[d] / w
        U.append([dens, *mom, tau, dens * ye, dens * ent, *Bt])
        E = [Bt[(i + 1) % 3] * vt[(i + 2) % 3] - Bt[(i + 2) % 3] * vt[(i + 1) % 3]
             for i in range(3)]
        fb = [torch.zeros_like(rho)] * 3
        fb[d1], fb[d2] = -E[d2], E[d1]
        F.append([dens * vt[d]] +
                 [mom[i] * vt[d] + alp * sq * (pm * (i == d) - bl[i] * bw) for i in range(3)] +
                 [tau * vt[d] + alp * sq * (pm * v[d] - ab0 * bw), dens * ye * vt[d],
                  dens * ent * vt[d]] + fb)
        hr = h * rho
        a2 = bs + hr * (cs2 + w ** 2 - cs2 * w ** 2)
        a1 = 2 * beta[d] * (bs + cs2 * hr) - 2 * (cs2 - 1) * hr * (beta[d] - alp * v[d]) * w ** 2
        a0 = ((bs + cs2 * hr) * (beta[d] ** 2 - alp ** 2 * u) -
              (cs2 - 1) * hr * (beta[d] - alp * v[d]) ** 2 * w ** 2)
        r = torch.sqrt((a1 ** 2 - 4 * a2 * a0).clamp(min=0))
        lam += [(-a1 + r) / (2 * a2 * alp), (-a1 - r) / (2 * a2 * alp)]
    cmax = functools.reduce(torch.maximum, lam).clamp(min=0)
    cmin = functools.reduce(torch.minimum, lam).clamp(max=0)
    cabs = torch.maximum(cmax, -cmin)
    out = []
    for q in range(10):
        u0, u1, f0, f1 = U[0][q], U[1][q], F[0][q], F[1][q]
        if q == 7 + d:
            v = torch.zeros_like(u0)
        elif case["flux"] == "HLLE":
            v = (cmax * f0 - cmin * f1 + cmax * cmin * (u1 - u0)) / (cmax - cmin)
        else:
            v = 0.5 * (f0 + f1 - cabs * (u1 - u0))
        shape = list(v.shape)
        shape[ax] = N + 1
        full = torch.zeros(shape, dtype=F64, device=v.device)
        full.narrow(ax, 3, N - 5).copy_(v)
        out.append(full)
    return out


def _aux(f):
    """Fx, Fy, Fz, beta^i Psi and G at the vertices (zero on the outermost ones)."""
    s = (slice(1, -1),) * 3
    A = []
    for i, name in enumerate(("Avec_x", "Avec_y", "Avec_z")):
        a = f[name]
        a = (a.narrow(2 - i, 1, a.shape[2 - i] - 1) + a.narrow(2 - i, 0, a.shape[2 - i] - 1)) / 2
        A.append(a[tuple(slice(None) if x == 2 - i else slice(1, -1) for x in range(3))])
    g = _sym({m: f[m][s] for m in ("gxx", "gxy", "gxz", "gyy", "gyz", "gzz")})
    sq, up = torch.sqrt(_det(g)), _low(_inv(g), A)
    alp, psi, beta = f["alp"][s], f["Psi"][s], [f["beta" + c][s] for c in "xyz"]
    vals = [alp * sq * x for x in up] + [b * psi for b in beta] + [alp * psi / sq - _dot(beta, A)]
    return [torch.nn.functional.pad(v, (1,) * 6) for v in vals]


def _sources(case, f, n, idx, order):
    vx = lambda a: a[NG:NG + n[2] + 1, NG:NG + n[1] + 1, NG:NG + n[0] + 1]  # noqa: E731
    c = {m: _inner(f[m]) for m in ("rho", "eps", "press", "Bvecx", "Bvecy", "Bvecz")}
    avg = {m: _v2c(vx(f[m])) for m in abi.ADM}

    def grad(name, d):
        a, ax = f[name], 2 - d
        for x in range(3):
            if x != ax:
                a = a.narrow(x, NG, n[2 - x] + 1)
                a = a.narrow(x, 0, n[2 - x]) + a.narrow(x, 1, n[2 - x])
        at = lambda o: a.narrow(ax, NG + o, n[d])  # noqa: E731
        df = at(1) - at(0) if order == 2 else (at(-1) - at(2) + 27 * (at(1) - at(0))) / 24
        return df * idx[d] / 4

    alp, beta = avg["alp"], [avg["beta" + x] for x in "xyz"]
    g = _sym(avg)
    sq, ug = torch.sqrt(_det(g)), _inv(g)
    if case.get("var") == "z_vec":
        z = [_inner(f["zvec_" + x]) for x in "xyz"]
        w = torch.sqrt(1 + _dot(_low(g, z), z))
        v = [x / w for x in z]
    else:
        v = [_inner(f["vel" + x]) for x in "xyz"]
        w = 1 / torch.sqrt(1 - _dot(_low(g, v), v))
    vl = _low(g, v)
    B = [c["Bvec" + x] for x in "xyz"]
    vs = [v[i] - beta[i] / alp for i in range(3)]
    b0 = w * _dot(B, vl) / alp
    bs = [B[i] / w + alp * b0 * vs[i] for i in range(3)]
    b2 = (_dot(B, _low(g, B)) + (alp * b0) ** 2) / w ** 2
    gb, gbs = _low(g, beta), _low(g, bs)
    E = (c["rho"] * (1 + c["eps"]) + c["press"] + b2) * w * w
    P = c["press"] + b2 / 2
    t00 = (E - P) / alp ** 2 - b0 ** 2
    t0 = [E * vs[i] / alp + P * beta[i] / alp ** 2 - b0 * bs[i] for i in range(3)]
    t0l = [E * vl[i] / alp - b0 * (gb[i] * b0 + gbs[i]) for i in range(3)]
    t = lambda i, j: (E * vs[i] * vs[j] + P * (ug[i][j] - beta[i] * beta[j] / alp ** 2) -  # noqa: E731
                      bs[i] * bs[j])
    K = _sym(avg, ("kxx", "kxy", "kxz", "kyy", "kyz", "kzz"))
    da = [grad("alp", d) for d in range(3)]
    tau = -t00 * _dot(beta, da) - _dot(t0, da)
    for i in range(3):
        for j in range(3):
            tau = tau + K[i][j] * (t00 * beta[i] * beta[j] + 2 * t0[i] * beta[j] + t(i, j))
    mom = []
    for d in range(3):
        m = -t00 * alp * da[d]
        for i in range(3):
            m = m + t0l[i] * grad("beta" + "xyz"[i], d)
            for j in range(3):
                name = "g" + "".join(sorted("xyz"[i] + "xyz"[j]))
                m = m + grad(name, d) * (0.5 * (t00 * beta[i] * beta[j] + t(i, j)) + t0[i] * beta[j])
        mom.append(alp * sq * m)
    zero = torch.zeros_like(tau)
    return [zero, *mom, alp * sq * tau, zero, zero]


def _rhs(case, par, f, fl, aux, src, n, idx):
    """The eleven right-hand sides on interior points, state order."""
    div = lambda q: -sum(idx[d] * torch.diff(fl[d][q].narrow(2 - d, NG, n[d] + 1)[tuple(  # noqa: E731
        slice(None) if x == 2 - d else slice(NG, -NG) for x in range(3))], dim=2 - d)
        for d in range(3))
    out = [s + div(q) for s, q in zip(src, (0, 1, 2, 3, 4, 6, 5))]
    for i in range(3):
        j, k = (i + 1) % 3, (i + 2) % 3

        def pair(a, along):  # at an edge: the face at it and the one below along `along`
            for x in range(3):
                m = n[2 - x] + (0 if x == 2 - i else 1)
                lo = NG - 1 if x == 2 - along else NG
                a = a.narrow(x, lo, m + (1 if x == 2 - along else 0))
            x = 2 - along
            return a.narrow(x, 0, a.shape[x] - 1) + a.narrow(x, 1, a.shape[x] - 1)

        E = 0.25 * (pair(fl[k][7 + j], j) - pair(fl[j][7 + k], k))
        G = aux[6]
        for x in range(3):
            G = G.narrow(x, NG, n[2 - x] + 1)
        out.append(-E - torch.diff(G, dim=2 - i) * idx[i])
    at = lambda a, d, o: a[tuple(slice(NG + (o if x == 2 - d else 0),  # noqa: E731
                                       NG + (o if x == 2 - d else 0) + n[2 - x] + 1)
                                 for x in range(3))]
    df = 0
    for d in range(3):
        F, Fb, b = aux[d], aux[3 + d], at(f["beta" + "xyz"[d]], d, 0)
        up = -(at(Fb, d, 2) - 4 * at(Fb, d, 1) + 3 * at(Fb, d, 0))
        dn = at(Fb, d, -2) - 4 * at(Fb, d, -1) + 3 * at(Fb, d, 0)
        df = df + 0.5 * idx[d] * (at(F, d, 1) - at(F, d, -1) - torch.where(b < 0, dn, up))
    out.append(-df - par.lorenz_damp_fac * at(f["alp"], 0, 0) * at(f["Psi"], 0, 0))
    return out


def _c2p(case, par, eos, g, cons, B):
    """Primitives and conserved variables from D, S_i, tau, DYe (densitized)
    and B^i: the root of the Palenzuela residual by bisection, then the floors."""
    sq = torch.sqrt(_det(g))
    rho_a, t_a = (torch.full_like(sq, x) for x in eos.atmo())
    cut = rho_a * (1 + par.atmo_tol)
    ye_a = torch.full_like(sq, par.Ye_atmo)
    p_a, eps_a, s_a = eos.of_temp(rho_a, t_a, ye_a)
    atm = cons[0] <= sq * cut
    Bl = _low(g, B)
    Bsq = _dot(B, Bl)
    D, S, tau = cons[0] / sq, [x / sq for x in cons[1:4]], cons[4] / sq
    tau = torch.maximum(tau, Bsq / 2)
    Su = _low(_inv(g), S)
    S2 = _dot(S, Su)
    lim = (D + tau) ** 2
    k = torch.where(S2 > lim, torch.sqrt(lim / S2), torch.ones_like(S2))
    S, Su, S2 = [x * k for x in S], [x * k for x in Su], S2 * k * k
    BS, ye = _dot(S, B), cons[6] / cons[0]
    q, s, r, t = tau / D, Bsq / D, S2 / D ** 2, BS / D ** 1.5
    table = isinstance(eos, _Tab)

    def at(x):
        wm2 = (1 - (x * x * r + (2 * x + s) * t * t) / (x * x * (x + s) ** 2)).clamp(1e-10, 1)
        w = 1 / torch.sqrt(wm2)
        eps = w - 1 + (1 - w * w) * x / w + w * (q - s + t * t / (2 * x * x) + s / (2 * w * w))
        if table:
            eps = torch.minimum(torch.maximum(eps, eps_a), torch.full_like(eps, eos.emax))
        return w, D / w, eps

    lo, hi = (1 + q - s).clamp(min=1e-10), 3 + 3 * q - 1.5 * s
    for _ in range(60):
        x = 0.5 * (lo + hi)
        w, rho, eps = at(x)
        p = eos.of_eps(rho, eps, ye)[0]
        below = x - (1 + eps + p / rho) * w < 0
        lo, hi = torch.where(below, x, lo), torch.where(below, hi, x)
    x = 0.5 * (lo + hi)
    w, rho, eps = at(x)
    Z = x * rho * w
    v = [Su[i] / (Z + Bsq) + BS * B[i] / (Z * (Z + Bsq)) for i in range(3)]
    p, T, ent, eps = eos.of_eps(rho, eps, ye)
    atm = atm | (rho < cut) | (eps <= 0)  # no valid root: the atmosphere
    yl, yh = eos.ye
    out = (ye < yl) | (ye > yh)
    ye = ye.clamp(yl, yh)
    wl = math.sqrt(1 + par.vw_lim ** 2)
    speed = torch.sqrt(_dot(_low(g, v), v))
    fast = speed > par.vw_lim / wl
    again = fast | out
    rho, w = torch.where(fast, D / wl, rho), torch.where(fast, torch.full_like(w, wl), w)
    v = [torch.where(fast, a * (par.vw_lim / wl / speed), a) for a in v]
    if table:
        p2, e2, s2 = eos.of_temp(rho, T, ye)
        p, eps, ent = (torch.where(again, a, b) for a, b in ((p2, p), (e2, eps), (s2, ent)))
    else:
        e2 = p / (rho * (par.gl_gamma - 1))
        _, T2, s2, _ = eos.of_eps(rho, e2, ye)
        eps, T, ent = (torch.where(fast, a, b) for a, b in ((e2, eps), (T2, T), (s2, ent)))
    if par.use_press_atmo:
        fix = p < par.p_atmo
        p = p.clamp(min=par.p_atmo)
        e2 = p / (rho * (par.gl_gamma - 1))
        _, T2, ent2, _ = eos.of_eps(rho, e2, ye)
        eps, T, ent = (torch.where(fix, a, b) for a, b in ((e2, eps), (T2, T), (ent2, ent)))
    else:
        fix = T < t_a
        T = torch.maximum(T, t_a)
        p2, e2, s2 = eos.of_temp(rho, T, ye)
        p, eps, ent = (torch.where(fix, a, b) for a, b in ((p2, p), (e2, eps), (s2, ent)))
    pick = lambda a, b: torch.where(atm, a, b)  # noqa: E731
    zero = torch.zeros_like(w)
    rho, eps, p, T, ent = (pick(a, b) for a, b in ((rho_a, rho), (eps_a, eps), (p_a, p),
                                                   (t_a, T), (s_a, ent)))
    ye, v, w = pick(ye_a, ye), [pick(zero, a) for a in v], pick(zero + 1, w)
    vl = _low(g, v)
    bst = w * _dot(B, vl)
    b2 = (Bsq + bst ** 2) / w ** 2
    hw2 = w * w * (rho * (1 + eps) + p + b2)
    dens = sq * rho * w
    mom = [sq * (hw2 * vl[i] - bst * (Bl[i] / w + bst * vl[i])) for i in range(3)]
    tau2 = sq * (hw2 - (p + b2 / 2) - bst ** 2) - dens
    redo = fix | again | atm
    dens, tau2 = torch.where(redo, dens, cons[0]), torch.where(redo, tau2, sq * tau)
    mom = [torch.where(redo, a, sq * b) for a, b in zip(mom, S)]
    hw = (rho * (1 + eps) + p) * w * w
    return {"rho": [rho], "vel": v, "eps": [eps], "press": [p], "temperature": [T],
            "entropy": [ent], "Ye": [ye], "Bvec": B, "dB": [sq * b for b in B],
            "zvec": [w * a for a in v], "svec": [hw * a for a in v], "dens": [dens], "mom": mom,
            "tau": [tau2], "DEnt": [dens * ent], "DYe": [dens * ye]}


def _stage_ref(case, par, f, u0, n, dx, c0, c1, c2):
    """One substep of the fields f (full extents): the updated fields."""
    eos, idx = _eos(case, par), [1 / d for d in dx]
    fl = [_face_fluxes(case, par, eos, f, idx, d) for d in range(3)]
    rhs = _rhs(case, par, f, fl, _aux(f), _sources(case, f, n, idx, par.local_spatial_order), n,
               idx)
    del fl
    new = dict(f)
    for name, r in zip(abi.STATE, rhs):
        v = c1 * _inner(f[name]) + c2 * r
        new[name] = _ext(v + c0 * _inner(u0[name]) if c0 else v, NG, "copy")
    vx = lambda a: a[NG:NG + n[2] + 1, NG:NG + n[1] + 1, NG:NG + n[0] + 1]  # noqa: E731
    g = _sym({m: _v2c(vx(f[m])) for m in ("gxx", "gxy", "gxz", "gyy", "gyz", "gzz")})
    sq = torch.sqrt(_det(g))
    B = []
    for d in range(3):
        b = _curl(new, idx, d)
        b = b.narrow(2 - d, NG, n[d] + 1)[tuple(slice(None) if x == 2 - d else slice(NG, -NG)
                                                for x in range(3))]
        B.append(0.5 * (b.narrow(2 - d, 0, n[d]) + b.narrow(2 - d, 1, n[d])) / sq)
    res = _c2p(case, par, eos, g, [_inner(new[m]) for m in abi.CONS], B)
    for key, vals in res.items():
        names = {**GROUPS, **STATE_GROUPS}[key]
        for name, v in zip(names, vals):
            if name in SYNC_PRIMS:
                new[name] = _ext(v, NG, "copy")
            else:  # interior written, ghosts as they were
                new[name] = new[name].clone()
                _inner(new[name]).copy_(v)
    return new


def _gather(f, groups):
    return {k: torch.stack([f[m] for m in v]) for k, v in groups.items()}


def _exact_stage(case, seed):
    s = _prepare_stage(case, seed)
    p = s["patch"]
    c0, c1, c2 = batch.SSPRK3[0]
    new = _stage_ref(case, s["par"], dict(p.arr), p.arr, p.n, p.dx, c0, c1, c2 * s["dt"])
    return {**_gather(new, {**GROUPS, **STATE_GROUPS}), "flag": None}


def _exact_batch(case, seed):
    if case["patches"] > 50:
        return None
    s = _prepare_batch(case, seed)
    out = {k: [] for k in {**GROUPS, **STATE_GROUPS}}
    for p in s["patches"]:
        f = u0 = dict(p.arr)
        for c0, c1, c2 in batch.SSPRK3:
            f = _stage_ref(case, s["par"], f, u0, p.n, p.dx, c0, c1, c2 * s["dt"])
        for k, names in {**GROUPS, **STATE_GROUPS}.items():
            out[k] += [f[m].reshape(-1) for m in names]
    return {**{k: torch.cat(v) for k, v in out.items()}, "flag": None}


def _exact_scheduled(case, seed):
    s = _prepare_scheduled(case, seed)
    p, par = s["patch"], s["par"]
    f, n, idx = p.arr, p.n, [1 / d for d in p.dx]
    fl = [[_ext(_inner(a), NG, "linear") for a in
           _face_fluxes(case, par, _eos(case, par), f, idx, d)] for d in range(3)]
    aux = [_ext(_inner(a), NG, "linear") for a in _aux(f)]
    rhs = _rhs(case, par, f, fl, aux, _sources(case, f, n, idx, case["order"]), n, idx)
    named = dict(zip(abi.STATE_RHS, (_ext(r, NG, "linear") for r in rhs)))
    return _gather(named, RHS_GROUPS)


def _exact_zones(case, seed):
    return {**_prepare_zones(case, seed)["truth"], "flag": None}


def _exact_tmunu(case, seed):
    s = _prepare_tmunu(case, seed)
    p, n = s["patch"], s["patch"].n
    wt = (0.5, 0.5) if case["order"] == 2 else (-1 / 16, 9 / 16, 9 / 16, -1 / 16)

    def c2v(name):
        a = p[name]
        for ax in range(3):
            a = sum(w * a.narrow(ax, NG - len(wt) // 2 + i, n[2 - ax] + 1)
                    for i, w in enumerate(wt))
        return a

    rho, eps, press = c2v("rho"), c2v("eps"), c2v("press")
    B, v = ([c2v(m + x) for x in "xyz"] for m in ("Bvec", "vel"))
    m = {k: _inner(p[k]) for k in abi.ADM[:10]}
    g, beta, alp = _sym(m), [m["beta" + x] for x in "xyz"], m["alp"]
    bl, vl = _low(g, beta), _low(g, v)
    w = 1 / torch.sqrt(1 - _dot(v, vl))
    # u_mu and b_mu of the fluid and the field, the four-metric
    ul = [w * (_dot(bl, v) - alp)] + [w * x for x in vl]
    b0 = w * _dot(B, vl) / alp
    bu = [B[i] / w + alp * b0 * (v[i] - beta[i] / alp) for i in range(3)]
    g4 = [[_dot(bl, beta) - alp ** 2] + bl] + [[bl[i]] + list(g[i]) for i in range(3)]
    bd = [b0 * g4[0][0] + _dot(bl, bu)] + [b0 * bl[i] + x for i, x in enumerate(_low(g, bu))]
    b2 = b0 * bd[0] + _dot(bu, bd[1:])
    out = torch.zeros_like(s["eT"])
    q = 0
    for i in range(4):
        for j in range(i, 4):
            _inner(out[q]).copy_((rho * (1 + eps) + press + b2) * ul[i] * ul[j] +
                                 (press + b2 / 2) * g4[i][j] - bd[i] * bd[j])
            q += 1
    return out


def _exact_refine(case, seed):
    s = _prepare_refine(case, seed)
    c, f, P = s["c"], s["f"], case["order"]
    off = [2 * (m // 4) for m in c.n]
    poly = {1: (1, 1), 3: (-1, 9, 9, -1), 5: (3, -25, 150, 150, -25, 3)}[P]
    low = {1: (1,), 3: (1 / 8, 1, -1 / 8), 5: (-3 / 128, 11 / 64, 1, -11 / 64, 3 / 128)}[P]
    fine, coarse = {}, {}
    for name in abi.STATE:
        cent, a, back = abi.centering(name), c[name], f[name]
        for d in range(3):
            ax, vert = 2 - d, (cent >> d) & 1
            I = torch.arange(f.shape(name)[ax], device="cuda") - NG + off[d]
            out = 0
            half, odd = torch.div(I, 2, rounding_mode="floor") + NG, (I % 2).bool()
            shape = [-1 if x == ax else 1 for x in range(3)]
            for m in range(P + 1 if vert else P):
                at = half + m - (P - 1) // 2
                if vert:
                    wt = torch.where(odd, poly[m] / sum(poly), float(m == (P - 1) // 2))
                else:
                    wt = torch.where(odd, low[P - 1 - m], low[m])
                at = at.clamp(0, a.shape[ax] - 1)  # weight zero where it reaches past the end
                out = out + wt.to(F64).reshape(shape) * a.index_select(ax, at)
            a = out
        if case["region"] == 1:
            inner = _inner(back).clone()
            _inner(a).copy_(inner)
            new = c[name].clone()
            dst = []
            for d in range(3):
                ax, vert = 2 - d, (cent >> d) & 1
                m = inner.shape[ax]
                ev = inner.narrow(ax, 0, m).index_select(ax, torch.arange(0, m, 2, device="cuda"))
                if not vert:
                    ev = 0.5 * (ev + inner.index_select(ax, torch.arange(1, m, 2, device="cuda")))
                inner = ev
                dst.insert(0, slice(NG + off[d] // 2, NG + off[d] // 2 + ev.shape[ax]))
            new[tuple(dst)] = inner
            coarse[name] = new
        fine[name] = a
    if case["region"] == 0:
        return _gather(fine, STATE_GROUPS)
    return {"coarse": _gather(coarse, STATE_GROUPS), "fine": _gather(fine, STATE_GROUPS)}


def exact(case, seed):
    return globals()["_exact_" + case["kind"]](case, seed)
