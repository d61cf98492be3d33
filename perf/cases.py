"""Performance cases of the forward model, its Jacobian, the retrieval and
table production, through the public entry points of jurassic_amd.

A case names a path and its sizes:
  forward    Context.formod_device: device-resident rays, radiances and
             transmittances of every channel
  jacobian   Context.jacobian_device: the same with all rows of K (adjoint)
  formod     gpu.formod, the drop-in on host structs (one observation)
  kernel     gpu.kernel, kernel()'s finite differences on host structs
  retrieval  gpu.optimal_estimation, a batch of retrievals on host structs
  tblgen     gpu.tblgen_batch, the rows of one lookup table

Atmospheres are the repository's standard profile (81 levels) with seeded
Gaussian random fields (3 K and 10% vmr, 5 km correlation length).  Tables
have 40 pressures x 20 temperatures; their columns either share one grid of
200 column densities or hold the rows that table production writes (factor
1.122 between rows, emissivities from 1e-6 to 0.999999, so every column
starts elsewhere).  exact() is the same model in plain torch, FP64
throughout, with its Jacobian by automatic differentiation.
"""
import ctypes as C
import math
import os
import re
import tempfile

import numpy as np
import torch

from jurassic_amd import abi, gpu, scenes

GASES = ["CO2", "H2O", "O3", "CH4", "N2O", "CO", "HNO3", "F11"]
SCALE = {"CO2": 1e-2, "H2O": 1e-3, "O3": 5e-3}
NLEV, TP, TT, TU = 81, 40, 20, 200
RE, KB, NA, P0 = 6367.421, 1.3806504e-23, 6.02214199e23, 1013.25
C1, C2 = 1.19104259e-8, 1.43877506
RAYDS, RAYDZ = 10.0, 0.1
DEV = torch.device("cuda:0" if torch.cuda.is_available() else "cpu")
F64 = torch.float64


def _dev(path, name, view, nprof, nview, nch, ngas, **kw):
    c = dict(name=name, path=path, view=view, nprof=nprof, nview=nview, nch=nch, ngas=ngas, fp32=True, ega=True,
             ctm=True, refrac=True, bbt=False, rows=False)
    c.update(kw)
    return c


def listed():
    return [
        # one observation through the C drop-in, as an existing host program
        # calls formod(): launches, copies and the march's latency
        dict(name="formod_nadir", path="formod", view="nadir", nview=10, nch=2, ngas=1, fp32=False),
        # kernel()'s finite differences for one observation (T and CO2)
        dict(name="kernel_fd_nadir", path="kernel", view="nadir", nview=10, nch=2, ngas=1, fp32=False),
        # a limb scan of some profiles: a few wavefronts per compute unit
        _dev("forward", "forward_limb_small", "limb", 77, 5, 12, 3),
        # the limb sounder at full size
        _dev("forward", "forward_limb", "limb", 4096, 32, 12, 3),
        # the same sounder in the reference's precision
        _dev("forward", "forward_limb_f64", "limb", 512, 32, 12, 3, fp32=False),
        # a nadir imager by the Curtis-Godson approximation, on tables as
        # table production writes them
        _dev("forward", "forward_nadir_cga", "nadir", 3001, 7, 33, 3, ega=False, rows=True),
        # a hyperspectral sounder: many channels, eight emitters
        _dev("forward", "forward_wide", "nadir", 1000, 1, 256, 8, rows=True),
        # adjoint Jacobians of a nadir sounder, T and three gases
        _dev("jacobian", "jacobian_nadir", "nadir", 1024, 8, 96, 3),
        # the Jacobians of one serving round of limb scans
        _dev("jacobian", "jacobian_limb_small", "limb", 64, 32, 12, 3, bbt=True),
        # adjoint Jacobians in FP64 (ragged blocks)
        _dev("jacobian", "jacobian_nadir_f64", "nadir", 100, 5, 13, 2, fp32=False),
        # a batch of temperature retrievals, three iterations each
        dict(name="retrieval_nadir", path="retrieval", view="nadir", nret=24, nview=8, nch=12, ngas=3, fp32=True),
        # the rows of one table: 40 x 20 spectra of one channel
        dict(name="tblgen_table", path="tblgen", nspec=800, npts=4001),
    ]


def _log(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.random()
    view = rng.choice(["limb", "nadir"])
    if kind < 0.1:
        return dict(path="formod", view=view, nview=_log(rng, 1, 200), nch=_log(rng, 2, 24), ngas=rng.randint(1, 3),
                    fp32=rng.random() < 0.5)
    if kind < 0.17:
        return dict(path="retrieval", view="nadir", nret=_log(rng, 1, 40), nview=rng.randint(2, 12),
                    nch=rng.randint(6, 16), ngas=3, fp32=True)
    if kind < 0.25:
        return dict(path="tblgen", nspec=_log(rng, 4, 1500), npts=_log(rng, 501, 6001))
    opt = dict(fp32=rng.random() < 0.75, ega=rng.random() < 0.75, ctm=rng.random() < 0.85, refrac=rng.random() < 0.9,
               bbt=rng.random() < 0.3, rows=rng.random() < 0.5)
    nview, ngas = _log(rng, 1, 32), rng.choice([1, 2, 3, 3, 4, 5, 8])
    nch = _log(rng, 2, 200)
    # radiances of the pass: at most those of the full limb sounder's, less
    # for Jacobians (which cost some ten times as much), FP64 and more gases
    top = 1.2e6 if kind < 0.65 else 1.5e5
    top *= (1.0 if opt["fp32"] else 0.3) * min(1.0, 3.0 / ngas) * (1.0 if view == "limb" else 1.3)
    if not opt["ega"] and kind >= 0.65:
        top *= 0.3
    nprof = max(1, int(_log(rng, 2000, top) / (nview * nch)))
    c = _dev("forward" if kind < 0.65 else "jacobian", "", view, nprof, nview, nch, ngas, **opt)
    del c["name"]
    return c


# ----------------------------------------------------------------------
# Inputs.
# ----------------------------------------------------------------------

def _nus(case):
    n = case["nch"]
    lo, hi = (700.0, 1400.0) if case["view"] == "limb" else (650.0, 1600.0)
    return [round(float(v), 4) for v in np.linspace(lo, hi, n)] if n > 1 else [792.0]


def _grids():
    return (np.exp(np.linspace(math.log(0.01), math.log(1100.0), TP)), np.linspace(160.0, 340.0, TT),
            np.exp(np.linspace(math.log(1e15), math.log(1e27), TU)))


def _strength(nu, gases):
    """k of eps = 1 - exp(-k (u/1e20)^0.8): [channel][gas][p][T]."""
    p, t, _ = _grids()
    s = np.array([SCALE.get(g, 1e-2) for g in gases])
    f = 0.2 + 0.8 * (0.5 + 0.5 * np.sin(2 * math.pi * np.asarray(nu) / 97.0))
    pt = (p[:, None] / P0) ** 0.7 * (t[None, :] / 250.0) ** -1.5
    return torch.tensor(f, device=DEV)[:, None, None, None] * torch.tensor(s[:, None, None] * pt, device=DEV)[None]


def _tables(case, nu):
    """(u, eps) float32 [channel][gas][p][T][n] of the case's tables."""
    k = _strength(nu, GASES[:case["ngas"]])
    if case.get("rows"):
        # rows u = 1.122^j from the first emissivity of 1e-6 to 0.999999
        n = int(math.log(-math.log(1e-6) / 1e-6) / 0.8 / math.log(1.122))
        j0 = torch.ceil((math.log(1e20) + torch.log(1.0000005e-6 / k) / 0.8) / math.log(1.122))
        ln_u = (j0[..., None] + torch.arange(n, dtype=F64, device=DEV)) * math.log(1.122)
    else:
        ln_u = torch.tensor(np.log(_grids()[2]), device=DEV).expand(*k.shape, TU)
    u = torch.exp(ln_u).float()
    eps = torch.empty_like(u)
    for c in range(0, len(nu), 32):
        eps[c:c + 32] = -torch.expm1(-k[c:c + 32, ..., None] * torch.exp(0.8 * (ln_u[c:c + 32] - math.log(1e20))))
    return u.contiguous(), eps


def _filters(nu):
    """Boxcar filters of 1 cm^-1 (zero samples at both ends)."""
    off = np.arange(len(nu) + 1, dtype=np.int32) * 105
    i = np.arange(105)
    x = np.concatenate([np.round(v + (i - 52) * 0.01, 4) for v in nu])
    return off, x, np.tile(((i >= 2) & (i < 102)).astype(float), len(nu))


def _profiles(case, seed, n):
    """T [n][81] and q [n][gas][81] of n atmospheres."""
    gases = GASES[:case["ngas"]]
    z = np.arange(NLEV, dtype=float)
    cov = np.exp(-np.abs(z[:, None] - z[None, :]) / 5.0) + 1e-12 * np.eye(NLEV)
    chol = torch.tensor(np.linalg.cholesky(cov), device=DEV)
    gen = torch.Generator(device=DEV).manual_seed(int(seed) % (1 << 40))
    x = torch.randn(n, 1 + len(gases), NLEV, dtype=F64, device=DEV, generator=gen) @ chol.T
    t = torch.tensor(scenes.std_temperature(z), device=DEV) + 3.0 * x[:, 0]
    q = torch.tensor(np.array([scenes.vmr_profile(g, z) for g in gases]), device=DEV) * torch.exp(0.1 * x[:, 1:])
    return t, q


def _geometry(case):
    """[view][7]: time, observer z lon lat, view point z lon lat."""
    n = case["nview"]
    g = (scenes.limb_geometry(800.0, np.linspace(5.0, 67.0, n) if n > 1 else [20.0]) if case["view"] == "limb"
         else scenes.nadir_geometry(705.0, np.linspace(0.0, 50.0, n)))
    return np.stack([np.zeros(n)] + [g[k] for k in ("obsz", "obslon", "obslat", "vpz", "vplon", "vplat")], axis=1)


def _ctl(case, nu, tblbase="-", **kw):
    on = 1 if case.get("ctm", True) else 0
    return abi.make_ctl(GASES[:case["ngas"]], nu, tblbase=tblbase, tblfmt=2, ctm_co2=on, ctm_h2o=on, ctm_n2=on,
                        ctm_o2=on, refrac=1 if case.get("refrac", True) else 0,
                        write_bbt=1 if case.get("bbt") else 0, formod=1 if case.get("ega", True) else 0, **kw)


_CONTEXT = {}


def _context(case, nu):
    """The device context of the case's tables: a program makes it once and
    keeps it over its batches (the last one made here is kept)."""
    key = tuple(case[k] for k in ("view", "nch", "ngas", "ctm", "refrac", "bbt", "ega", "rows"))
    if key not in _CONTEXT:
        for old in _CONTEXT.values():
            old.close()
        _CONTEXT.clear()
        u, eps = _tables(case, nu)
        nd, ng, n = len(nu), case["ngas"], u.shape[-1]
        p, t, _ = _grids()
        i32 = dict(dtype=torch.int32, device=DEV)
        tabs = dict(np=torch.full((nd, ng), TP, **i32), nt=torch.full((nd, ng, TP), TT, **i32),
                    nu=torch.full((nd, ng, TP, TT), n, **i32),
                    p=torch.tensor(p, device=DEV).expand(nd, ng, TP).contiguous(),
                    t=torch.tensor(t, device=DEV).expand(nd, ng, TP, TT).contiguous(), u=u, eps=eps)
        torch.cuda.synchronize()
        ctl = _ctl(case, nu[:1])
        _CONTEXT[key] = gpu.Context.from_device_tables(ctl, nu, tabs, filters=_filters(nu))
    return _CONTEXT[key]


def _host_ctl(case, **kw):
    """ctl of the host paths: tables and filters in files, as formod reads
    them (written once)."""
    nu = _nus(case)
    root = os.path.join(tempfile.gettempdir(), "jurassic_perf_%d" % os.getuid(), "%s_%d" % (case["view"], case["nch"]))
    os.makedirs(root, exist_ok=True)
    base = os.path.join(root, "tab")
    p, t, u = _grids()
    files = [scenes.table_name(base, v, g) for v in nu for g in GASES[:case["ngas"]]]
    if not all(os.path.exists(f) for f in files):
        eps = _tables(dict(case, rows=False), nu)[1].cpu().numpy()
        for i, f in enumerate(files):
            scenes.write_table_bin(f + ".new%d" % os.getpid(), p, t, u, eps[i // case["ngas"], i % case["ngas"]])
            os.replace(f + ".new%d" % os.getpid(), f)
    off, x, w = _filters(nu)
    for i, v in enumerate(nu):
        f = "%s_%.4f.filt" % (base, v)
        if not os.path.exists(f):
            with open(f + ".new%d" % os.getpid(), "w") as out:
                for a, b in zip(x[off[i]:off[i + 1]], w[off[i]:off[i + 1]]):
                    out.write("%.4f %d\n" % (a, b))
            os.replace(f + ".new%d" % os.getpid(), f)
    return _ctl(case, nu, tblbase=base, **kw)


def _host_atm(t, q):
    z = np.arange(NLEV, dtype=float)
    return abi.make_atm(z, scenes.std_pressure(z), t.cpu().numpy(), q.cpu().numpy(), np.zeros((1, NLEV)))


def _host_obs(case):
    g = _geometry(case)
    return abi.make_obs(*[g[:, k] for k in range(1, 7)])


def _device_atms(case, seed, n):
    """n atm_t records in device memory."""
    t, q = _profiles(case, seed, n)
    z = np.arange(NLEV, dtype=float)
    words = C.sizeof(abi.atm_t) // 8
    a = torch.zeros(n, words, dtype=F64, device=DEV)
    a.view(torch.int32)[:, 0] = NLEV

    def at(field, extra=0):
        o = getattr(abi.atm_t, field).offset // 8 + extra
        return slice(o, o + NLEV)
    a[:, at("z")] = torch.tensor(z, device=DEV)
    a[:, at("p")] = torch.tensor(scenes.std_pressure(z), device=DEV)
    a[:, at("t")] = t
    for g in range(case["ngas"]):
        a[:, at("q", g * abi.NP)] = q[:, g]
    o = abi.atm_t.sfeps.offset // 8
    a[:, o:o + abi.NSF] = 1.0
    return a


def _state_windows(case):
    """State of the Jacobians: T and at most three gases, all levels."""
    n = min(case["ngas"], 3)
    return dict(rett_zmin=-100, rett_zmax=100, retq_zmin=[-100] * n, retq_zmax=[100] * n)


def prepare(case, seed):
    path = case["path"]
    if path == "tblgen":
        return _tblgen_input(case, seed)
    if path == "formod":
        t, q = _profiles(case, seed, 1)
        return dict(case=case, ctl=_host_ctl(case), atm=_host_atm(t[0], q[0]), obs=_host_obs(case))
    if path == "kernel":
        t, q = _profiles(case, seed, 1)
        ctl = _host_ctl(case, **_state_windows(case))
        return dict(case=case, ctl=ctl, atm=_host_atm(t[0], q[0]), obs=_host_obs(case),
                    m=case["nview"] * case["nch"], n=NLEV * (1 + case["ngas"]))
    if path == "retrieval":
        n = case["nret"]
        t, q = _profiles(case, seed, n)
        ctl = _host_ctl(case, rett_zmin=-100, rett_zmax=100)
        ctl.write_bbt = 1
        truth, meas = (abi.atm_t * n)(), (abi.obs_t * n)()
        noise = np.random.default_rng(seed).normal(0.0, 0.1, (n, case["nch"], case["nview"]))
        apr = []
        for i in range(n):
            truth[i] = _host_atm(t[i], q[i])
            meas[i] = _host_obs(case)
            a = abi.copy_struct(truth[i])
            abi.np_view(a.t)[:NLEV] = scenes.std_temperature(np.arange(NLEV))
            apr.append(a)
        gpu.formod_batch(ctl, truth, meas, abi.JUR_FP64)
        for i in range(n):
            for d in range(case["nch"]):
                abi.np_view(meas[i].rad[d])[:case["nview"]] += noise[i, d]
        ret = abi.ret_t()
        ret.kernel_recomp, ret.conv_itmax, ret.conv_dmin = 1, 3, 0.0
        for d in range(case["nch"]):
            ret.err_noise[d] = math.sqrt(0.1)
        ret.err_temp, ret.err_temp_cz, ret.err_temp_ch = 2.0, 5.0, 1e10
        return dict(case=case, ctl=ctl, ret=ret, meas=[abi.copy_struct(o) for o in meas], apr=apr)
    nu = _nus(case)
    ctx = _context(case, nu)
    nprof, nview, nd = case["nprof"], case["nview"], case["nch"]
    nray = nprof * nview
    # rays by view, then atmosphere: a block of 64 holds similar paths
    prof = torch.arange(nprof, dtype=torch.int32, device=DEV).repeat(nview)
    geom = torch.tensor(_geometry(case), device=DEV).repeat_interleave(nprof, dim=0).contiguous()
    s = dict(case=case, ctx=ctx, atm=_device_atms(case, seed, nprof), prof=prof, geom=geom,
             rad=torch.empty(nray, nd, dtype=F64, device=DEV), tau=torch.empty(nray, nd, dtype=F64, device=DEV))
    if path == "jacobian":
        ctl = _ctl(case, nu[:1], **_state_windows(case))
        a = abi.atm_t.from_buffer_copy(s["atm"][0].cpu().numpy().tobytes())
        s["xmap"], n = gpu.state_map(ctl, a)
        s["pmap"] = torch.zeros(nprof, dtype=torch.int32, device=DEV)
        s["k"] = torch.empty(nray, nd, n, dtype=F64, device=DEV)
    torch.cuda.synchronize()
    return s


# ----------------------------------------------------------------------
# One pass.
# ----------------------------------------------------------------------

def _padded(rows):
    """The rows (u, eps) of every spectrum as arrays [spectrum][400]."""
    u, e = np.zeros((len(rows), 400)), np.zeros((len(rows), 400))
    for k, (a, b) in enumerate(rows):
        u[k, :len(a)], e[k, :len(b)] = a, b
    return dict(u=u, eps=e)


def run(s):
    case = s["case"]
    path = case["path"]
    prec = abi.JUR_FP32 if case.get("fp32") else abi.JUR_FP64
    if path == "tblgen":
        rows = gpu.tblgen_batch(s["press"], s["temp"], s["tau"], s["nu0"], s["nu1"], s["nuf"], s["filt"])
        return _padded(rows)
    if path == "formod":
        gpu.formod(s["ctl"], s["atm"], s["obs"], prec)
        rad, tau = abi.obs_arrays(s["obs"], s["ctl"])
        return dict(rad=rad, tau=tau)
    if path == "kernel":
        return dict(k=gpu.kernel(s["ctl"], s["atm"], s["obs"], abi.JUR_JAC_FD, prec, s["m"], s["n"]))
    if path == "retrieval":
        atm, obs, hist, niter = gpu.optimal_estimation(s["ret"], s["ctl"], s["meas"], s["apr"],
                                                       abi.JUR_JAC_ADJOINT, prec)
        return dict(t=np.array([abi.np_view(a.t)[:NLEV] for a in atm]), niter=np.array(niter),
                    bt=np.array([abi.obs_arrays(o, s["ctl"])[0] for o in obs]),
                    chisq=np.array([h[-1] for h in hist]))
    nray = case["nprof"] * case["nview"]
    args = (case["nprof"], s["atm"].data_ptr(), nray, s["prof"].data_ptr(), s["geom"].data_ptr(),
            s["rad"].data_ptr(), s["tau"].data_ptr())
    if path == "forward":
        s["ctx"].formod_device(*args, precision=prec)
        return dict(rad=s["rad"], tau=s["tau"])
    s["ctx"].jacobian_device(*args, s["xmap"], s["pmap"].data_ptr(), s["k"].shape[2], s["k"].data_ptr(),
                             precision=prec)
    return dict(rad=s["rad"], tau=s["tau"], k=s["k"])


# ----------------------------------------------------------------------
# Work and tolerance.
# ----------------------------------------------------------------------

def _points(case):
    """Mean LOS points of a ray (80 km in steps of 0.1 km vertically or 10 km
    along the path)."""
    if case["view"] == "nadir":
        return 805
    h = np.linspace(5.0, 67.0, case["nview"]) if case["nview"] > 1 else np.array([20.0])
    return float(np.mean(2 * (80.0 - h) / RAYDZ)) + 8


def work(case):
    """Bytes: atmospheres and geometry read once, outputs written once, and
    the distinct table entries that the paths can touch (at most the whole
    tables).  Operations: one lookup step per (ray, point, channel, emitter)
    as four corners of two linear interpolations and the cell weights (60),
    one accumulation step per (ray, point, channel) (60), one march step per
    (ray, point) (300); twice that again for the adjoint."""
    path = case["path"]
    if path == "tblgen":
        m = case["nspec"] * case["npts"]
        return {"bytes": 8.0 * m + 16.0 * 400 * case["nspec"], "flops": 0.8 * m * 400 * 20.0}
    nd, ng, nv = case["nch"], case["ngas"], case["nview"]
    n = {"formod": 1, "kernel": 1 + NLEV * (1 + ng), "retrieval": case.get("nret", 0) * 4}.get(path) or case["nprof"]
    nray = n * nv
    pts = nray * _points(case)
    flops = pts * (nd * (60.0 * ng + 60.0) + 300.0)
    table = nd * ng * TP * TT * TU * 8.0
    size = (nray * nd * 16.0 + n * 8.0 * NLEV * (3 + ng) + nray * 56.0 +
            min(table, pts * nd * ng * 32.0))
    if path in ("jacobian", "retrieval"):
        state = NLEV * (1 + min(ng, 3)) if path == "jacobian" else NLEV
        flops *= 3.0
        size += nray * nd * state * 8.0
    if path == "kernel":
        size = nv * nd * 8.0 * n + min(table, pts * nd * ng * 32.0)
    return {"bytes": size, "flops": flops}


def tolerance(case):
    if case["path"] == "tblgen":
        return {"rel": 1e-12, "max": 1e-9}
    if case["path"] == "kernel":
        return {"rel": 1e-8, "max": 1e-6}
    if case["path"] == "retrieval":
        return {"rel": 1e-4, "max": 1e-2}
    if not case["fp32"]:
        return {"rel": 1e-10, "max": 1e-8}
    # four times the distance of the FP32 path from exact(): 1e-6 of the
    # radiances, 9e-5 of brightness temperatures (radiances near zero among
    # them), 2e-3 of limb Jacobians (entries of nearly opaque paths up to
    # their root mean square)
    if case["path"] == "jacobian":
        return {"rel": 8e-3, "max": 0.9}
    return {"rel": 4e-4, "max": 3e-3} if case.get("bbt") else {"rel": 1e-5, "max": 2e-4}


# ----------------------------------------------------------------------
# The model in FP64 by plain torch.
# ----------------------------------------------------------------------

def _continuum_tables():
    """The published continuum coefficients (plain numbers in a C header)."""
    path = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "jurassic_amd", "csrc",
                        "ctm_coeffs.h")
    with open(path) as f:
        text = f.read()
    return {m.group(1): np.array([float(v) for v in m.group(2).replace("\n", " ").split(",") if v.strip()])
            for m in re.finditer(r"double JUR_CTM_(\w+)\[\d+\] = \{([^}]*)\}", text)}


def _channel_constants(nu):
    """Per-channel continuum coefficients, [channel] each."""
    c = _continuum_tables()
    out = {k: np.zeros(len(nu)) for k in ("c296", "c260", "c230", "slf", "ratio", "frn", "n2b", "n2beta", "o2b", "o2beta")}
    out["ratio"][:] = 1.0
    for i, v in enumerate(nu):
        xw = v / 2 + 1
        if 1 <= xw < 2001:
            for k, name in (("c296", "CO2_296"), ("c260", "CO2_260"), ("c230", "CO2_230")):
                out[k][i] = np.interp(xw - 1, np.arange(2001), c[name])
        xw = v / 10 + 1
        if 1 <= xw < 2001:
            w296, w260, wfrn = (np.interp(xw - 1, np.arange(2001), c["H2O_" + k]) for k in ("296", "260", "FRN"))
            sfac = 1.0 if v <= 820 or v >= 960 else np.interp((v - 820) / 10, np.arange(15), c["H2O_XFCREV"])
            vf2 = (v - 370) ** 2
            out["slf"][i], out["ratio"][i] = sfac * w296, w260 / w296
            out["frn"][i] = wfrn * (1 - 0.25 * 36100 / (vf2 + vf2 ** 3 * 1e-8 + 36100))
        for g in ("N2", "O2"):
            x = c[g + "_NU"]
            if x[0] <= v <= x[-1]:
                out[g.lower() + "b"][i] = np.interp(v, x, c[g + "_B"])
                out[g.lower() + "beta"][i] = np.interp(v, x, c[g + "_BETA"])
    return {k: torch.tensor(v, device=DEV) for k, v in out.items()}


def _source_table(nu):
    """Filter-weighted Planck means, [channel][1200 temperatures 100..400 K]."""
    off, x, w = _filters(nu)
    st = torch.tensor(100.0 + 300.0 / 1199.0 * np.arange(1200), device=DEV)
    rows = []
    for i in range(len(nu)):
        a, b = x[off[i]:off[i + 1]], w[off[i]:off[i + 1]]
        d = np.diff(a).min()
        s = np.add.accumulate(np.concatenate([[a[0]], np.full(2 * len(a), d)]))
        s = s[s <= a[-1]]
        f = torch.tensor(np.interp(s, a, b), device=DEV)
        s = torch.tensor(s, device=DEV)
        b = C1 * s ** 3 / torch.expm1(C2 * s / st[:, None])
        rows.append((b * f).sum(1) / f.sum())
    return torch.stack(rows)


class _Model:
    """rays V x channels C; every ray has its own atmosphere (p, t, q of its
    levels) and its own channels ch [V][C]."""

    def __init__(self, case, nu, ch):
        self.case, self.ch, self.ng = case, ch, case["ngas"]
        u, e = _tables(case, nu)
        self.n = u.shape[-1]
        self.u, self.e = u.reshape(-1), e.reshape(-1)
        p, t, _ = _grids()
        self.pg, self.tg = torch.tensor(p, device=DEV), torch.tensor(t, device=DEV)
        self.sr = _source_table(nu).reshape(-1)
        k = _channel_constants(nu)
        self.k = {name: v[ch] for name, v in k.items()}
        self.nu = torch.tensor(nu, dtype=F64, device=DEV)[ch]
        self.tab = (ch[..., None] * self.ng + torch.arange(self.ng, device=DEV)) * (TP * TT)

    # -- atmosphere ------------------------------------------------------
    @staticmethod
    def _levels(z):
        i = torch.clamp(torch.floor(z.detach()).long(), 0, NLEV - 2)
        return i, z - i

    def _pt(self, z, lp, t):
        """p and T at altitudes z [V][k] (levels are 1 km apart)."""
        i, w = self._levels(z)
        l0, l1 = lp.gather(1, i), lp.gather(1, i + 1)
        t0, t1 = t.gather(1, i), t.gather(1, i + 1)
        return torch.exp(l0 + (l1 - l0) * w), t0 + (t1 - t0) * w

    def _q(self, z, q):
        i, w = self._levels(z)
        i = i[:, None, None].expand(-1, self.ng, 1)
        q0, q1 = q.gather(2, i)[..., 0], q.gather(2, i + 1)[..., 0]
        return q0 + (q1 - q0) * w[:, None]

    # -- table columns ---------------------------------------------------
    def _search(self, col, vals, x):
        """Largest i in [0, n-2] with vals[col][i] <= x (0 if none)."""
        with torch.no_grad():
            lo = torch.zeros_like(col)
            hi = torch.full_like(col, self.n - 1)
            base = col * self.n
            for _ in range(int(math.ceil(math.log2(self.n)))):
                mid = (lo + hi) >> 1
                go = vals[base + mid] <= x
                more = hi > lo + 1
                lo = torch.where(more & go, mid, lo)
                hi = torch.where(more & ~go, mid, hi)
            return base + lo, lo

    def _line(self, xs, ys, col, x):
        """y(x) on columns: linear in brackets (slopes of the float32 table
        entries formed in float32, as the tables define them), through the
        origin below the first knot; (value, above the last knot)."""
        at, i = self._search(col, xs, x.detach())
        x0, y0, x1, y1 = xs[at], ys[at], xs[at + 1], ys[at + 1]
        below = x.detach() < x0
        s = torch.where(below, y0 / x0, (y1 - y0) / (x1 - x0))
        s = torch.where(torch.isfinite(s), s, torch.zeros_like(s)).double()
        y = torch.where(below, s * x, y0.double() + s * (x - x0.double()))
        return y, x.detach() > x1

    def _decay(self, col):
        last = col * self.n + self.n - 1
        a = torch.log((1.0 - self.e[last]).double()) / self.u[last].double()
        return torch.clamp(a, min=-1e30)

    def _eps(self, col, a, u):
        y, above = self._line(self.u, self.e, col, u)
        return torch.where(above, -torch.expm1(a * torch.where(above, u, torch.zeros_like(u))), y)

    def _inv(self, col, a, e):
        y, above = self._line(self.e, self.u, col, e)
        return torch.where(above, torch.log1p(-torch.where(above, e, torch.zeros_like(e))) / a, y)

    def _cell(self, p, t):
        """Weights and the four corner columns at p, t [V][1 or C][G]."""
        pd, td = p.detach(), t.detach()
        lp = torch.log(self.pg)
        ip = torch.clamp(torch.floor((torch.log(pd) - lp[0]) / (lp[1] - lp[0])).long(), 0, TP - 2)
        it = torch.clamp(torch.floor((td - self.tg[0]) / (self.tg[1] - self.tg[0])).long(), 0, TT - 2)
        col = self.tab + ip * TT + it
        col = torch.stack([col, col + 1, col + TT, col + TT + 1], -1)
        wt = (t - self.tg[it]) / (self.tg[it + 1] - self.tg[it])
        pa, pb = self.pg[ip], self.pg[ip + 1]
        wp = (p - pa) / (pb - pa) if self.case.get("ega", True) else torch.log(p / pa) / torch.log(pb / pa)
        return col, wt, wp

    # -- one segment -----------------------------------------------------
    def _segment(self, st, z, p, t, q, ds, on):
        tp, cu, cp, ct, tau, rad = st
        u = 10 * q * (p / (KB * t) * ds)[:, None]                      # [V][G]
        us = u[:, None, :]
        on3 = on[:, None, None]
        if self.case.get("ega", True):
            col, wt, wp = self._cell(p[:, None, None], t[:, None, None])
            a = self._decay(col)
            e = self._eps(col, a, self._inv(col, a, (1 - tp)[..., None].expand(col.shape)) + us[..., None])
        else:
            cu, cp, ct = cu + us, cp + us * p[:, None, None], ct + us * t[:, None, None]
            col, wt, wp = self._cell(cp / cu, ct / cu)
            a = self._decay(col)
            e = self._eps(col, a, cu[..., None].expand(col.shape))
        e0, e1 = e[..., 0] + (e[..., 1] - e[..., 0]) * wt, e[..., 2] + (e[..., 3] - e[..., 2]) * wt
        e = torch.clamp(e0 + (e1 - e0) * wp, 0.0, 1.0)
        opaque = tp.detach() < 1e-9
        new = torch.where(opaque, torch.zeros_like(tp), 1 - e)
        trans = torch.where(opaque, torch.zeros_like(tp), new / torch.where(opaque, torch.ones_like(tp), tp))
        gas = trans.prod(-1)
        k, nu = self.k, self.nu
        pc, tc, dc = p[:, None], t[:, None], ds[:, None]
        beta = torch.zeros_like(gas)
        if self.case.get("ctm", True):
            d230, d260, d296 = tc - 230, tc - 260, tc - 296
            ctw = d260 * 5.050505e-4 * d296 * k["c230"] - d230 * 9.259259e-4 * d296 * k["c260"] + d230 * 4.208754e-4 * d260 * k["c296"]
            beta = beta + u[:, :1] / NA / 1000 * pc / P0 * ctw / dc
            if self.ng > 1:
                qh = q[:, 1:2]
                slf = k["slf"] * torch.exp((296 - tc) / 36.0 * torch.log(k["ratio"]))
                beta = beta + (nu * u[:, 1:2] * torch.tanh(0.7193876 / tc * nu) * 296 / tc *
                               (pc / P0 * (qh * slf + (1 - qh) * k["frn"]) * 1e-20)) / dc
            r = pc / P0 * 273.0 / tc
            beta = beta + (0.1 * r * r * torch.exp(k["n2beta"] * (1 / 296.0 - 1 / tc)) * 0.79 * k["n2b"] *
                           (0.79 + 0.21 * (1.294 - 0.4545 * tc / 296.0)))
            beta = beta + 0.1 * r * r * torch.exp(k["o2beta"] * (1 / 296.0 - 1 / tc)) * 0.21 * k["o2b"]
        src = self._src(tc)
        ok = on[:, None] & (gas.detach() > 0)
        s = torch.where(ok, gas * torch.exp(-beta * dc), torch.ones_like(gas))
        rad = rad + torch.where(ok, src * (1 - s) * tau, torch.zeros_like(rad))
        return torch.where(on3, new, tp), cu, cp, ct, tau * s, rad

    def _src(self, t):
        d = 300.0 / 1199.0
        i = torch.clamp(torch.floor((t.detach() - 100.0) / d).long(), 0, 1198)
        a, b = self.sr[self.ch * 1200 + i], self.sr[self.ch * 1200 + i + 1]
        return a + (b - a) * ((t - (100.0 + d * i.double())) / d)

    # -- the path --------------------------------------------------------
    def _entry(self, geom):
        def cart(z, lon, lat):
            la, lo = lat / 180 * math.pi, lon / 180 * math.pi
            return (z + RE)[:, None] * torch.stack([torch.cos(la) * torch.cos(lo), torch.cos(la) * torch.sin(lo), torch.sin(la)], 1)
        xo, xv = cart(*geom[:, 1:4].T), cart(*geom[:, 4:7].T)
        e = xv - xo
        norm = e.norm(dim=1)
        e = e / norm[:, None]
        top = float(NLEV - 1)
        dmax, dmin, x = norm.clone(), torch.zeros_like(norm), xo.clone()
        go = torch.ones_like(norm, dtype=torch.bool)
        while bool(go.any()):
            d = (dmax + dmin) / 2
            x = torch.where(go[:, None], xo + d[:, None] * e, x)
            z = x.norm(dim=1) - RE
            go = go & ~((z <= top) & (z > top - 0.001))
            near = z < top - 0.0005
            dmax, dmin = torch.where(go & near, d, dmax), torch.where(go & ~near, d, dmin)
            go = go & ((dmin - dmax).abs() > 0.001)
        return x, e

    def _steps(self, nstep, lp, t, q, x, e, prev, raw, raw2, xl, life, st):
        """nstep steps of the march and the segments behind them.  prev:
        altitude of the point before, raw and raw2: raw step lengths of the last two
        points, life: 2 marching, 1 last point pending, 0 done."""
        first = prev is None
        for _ in range(nstep):
            r = x.norm(dim=1)
            z = r - RE
            cosa = ((e * x).sum(1) / r).abs()
            ds = torch.clamp(RAYDZ / cosa, max=RAYDS)
            out = (life == 2) & ((z.detach() < 0) | (z.detach() > NLEV - 1))
            if not first:
                # the step that left the range is clipped to it, and with it
                # the raw length of the point before
                bound = torch.where(z.detach() < 0, 0.0, float(NLEV - 1))
                zp = prev["z"]
                frac = torch.where(out, bound - zp, torch.zeros_like(z)) / torch.where(out, z - zp, torch.ones_like(z))
                xc = torch.where(out[:, None], xl + frac[:, None] * (x - xl), x)
                raw = torch.where(out, ds * frac, raw)
                ends = life == 1
                dtr = 0.5 * (raw2 + torch.where(ends, torch.zeros_like(raw), raw))
                on = life > 0
                st = self._segment(st, prev["z"], prev["p"], prev["t"], prev["q"], torch.where(on, dtr, torch.ones_like(dtr)), on)
                life = torch.where(ends, torch.zeros_like(life), torch.where(out, torch.ones_like(life), life))
                raw2 = torch.where(ends, raw2, raw)
            else:
                xc, raw2 = x, torch.zeros_like(ds)
            first = False
            zc = xc.norm(dim=1) - RE
            p, tt = (v[:, 0] for v in self._pt(zc[:, None], lp, t))
            held = life == 0
            keep = (lambda a, b: torch.where(held if a.dim() == 1 else held[:, None], b, a)) if prev is not None else (lambda a, b: a)
            now = dict(z=zc, p=p, t=tt, q=self._q(zc, q))
            prev = {k: keep(now[k], (prev or now)[k]) for k in now}
            move = life == 2
            raw, xl = torch.where(move, ds, torch.zeros_like(ds)), x
            n, grad = torch.ones_like(z), torch.zeros_like(x)
            if self.case.get("refrac", True):
                low = z.detach() <= 60
                mid = x + 0.5 * ds[:, None] * e
                probes = torch.stack([mid] + [mid + 0.02 * torch.eye(3, dtype=F64, device=DEV)[i] for i in range(3)], 1)
                pq, tq = self._pt(probes.norm(dim=2) - RE, lp, t)
                ref = 7.753e-05 * pq / tq
                n = torch.where(low, 1 + 7.753e-05 * p / tt, n)
                grad = torch.where(low[:, None], (ref[:, 1:] - ref[:, :1]) / 0.02, grad)
            v = e * n[:, None] + ds[:, None] * grad
            e1 = v / v.norm(dim=1, keepdim=True)
            x1 = x + 0.5 * ds[:, None] * (e + e1)
            x, e = torch.where(move[:, None], x1, x), torch.where(move[:, None], e1, e)
        return x, e, prev, raw, raw2, xl, life, st

    def __call__(self, geom, p, t, q):
        """(rad, tau) [V][C] of rays geom [V][7] through p, t [V][81], q [V][G][81]."""
        lp = torch.log(p)
        x, e = self._entry(geom)
        v, c = self.ch.shape
        tp = torch.ones(v, c, self.ng, dtype=F64, device=DEV)
        zero = torch.zeros_like(tp)
        st = (tp, zero, zero, zero, torch.ones(v, c, dtype=F64, device=DEV), torch.zeros(v, c, dtype=F64, device=DEV))
        life = torch.full((v,), 2, device=DEV)
        s = self._steps(1, lp, t, q, x, e, None, None, None, None, life, st)
        while bool((s[6] > 0).any()):
            s = self._steps(25, lp, t, q, *s)
        prev, st = s[2], s[7]
        ground = prev["z"].detach() < 1.0
        rad = st[5] + torch.where(ground[:, None], self._src(prev["t"][:, None]) * st[4], torch.zeros_like(st[5]))
        if self.case.get("bbt"):
            rad = C2 * self.nu / torch.log1p(C1 * self.nu ** 3 / rad)
        return rad, st[4]


def _tblgen_input(case, seed):
    n, m = case["nspec"], case["npts"]
    rng = np.random.default_rng(seed)
    npr = max(1, n // 20)
    press = np.repeat(np.logspace(math.log10(1100.0), -2, npr), -(-n // npr))[:n]
    temp = np.tile(np.linspace(160.0, 320.0, -(-n // npr)), npr)[:n]
    nu0, nu1 = 700.0, 702.0
    nu = np.linspace(nu0, nu1, m)
    base = np.full(m, 1e-6)
    for c, s, w in zip(rng.uniform(nu0, nu1, 30), 10 ** rng.uniform(-3, 0, 30), rng.uniform(0.001, 0.01, 30)):
        base += s * w / np.pi / ((nu - c) ** 2 + w * w)
    tau = base[None, :] * (press / 300.0)[:, None] * (250.0 / temp)[:, None]
    nuf = np.linspace(700.2, 701.8, 33)
    return dict(case=case, press=press, temp=temp, tau=tau, nu0=nu0, nu1=nu1, nuf=nuf,
                filt=np.exp(-0.5 * ((nuf - 701.0) / 0.3) ** 2))


def _tblgen_exact(case, seed):
    s = _tblgen_input(case, seed)
    n, m = s["tau"].shape
    nu = s["nu0"] + (s["nu1"] - s["nu0"]) / (m - 1.0) * np.arange(m)
    i0 = int((s["nuf"][0] - s["nu0"]) / (s["nu1"] - s["nu0"]) * m)
    use = (np.arange(m) >= i0) & (nu >= s["nuf"][0]) & (nu <= s["nuf"][-1])
    f = torch.tensor(np.interp(nu[use], s["nuf"], s["filt"]), device=DEV)
    us = [1.0]
    while us[-1] * 1.122 <= 1e30:
        us.append(us[-1] * 1.122)
    us = torch.tensor(us, dtype=F64, device=DEV)
    uref = 1e-6 * s["press"] * 100 / (1.380658e-23 * s["temp"]) * 1000 / 1e4
    a = torch.tensor(s["tau"][:, use] / uref[:, None], device=DEV)
    rows = []
    for k in range(n):
        e = (1 - (torch.exp(-a[k] * us[:, None]) * f).sum(1) / f.sum()).cpu().numpy()
        last = int(np.argmax(e > 0.999999)) if (e > 0.999999).any() else len(e)
        old = np.concatenate([[0.0], e[:-1]])
        keep = (e >= 1e-6) & (e <= 0.999999) & (e > old) & (np.arange(len(e)) < last)
        rows.append((us.cpu().numpy()[keep], e[keep]))
    return _padded(rows)


def exact(case, seed):
    path = case["path"]
    if path == "tblgen":
        return _tblgen_exact(case, seed)
    if path == "retrieval":
        return None  # its Jacobians by automatic differentiation take minutes
    nu, nv, nd, ng = _nus(case), case["nview"], case["nch"], case["ngas"]
    nprof = case.get("nprof", 1)
    t, q = _profiles(case, seed, nprof)
    p = torch.tensor(scenes.std_pressure(np.arange(NLEV)), device=DEV).expand(nprof, NLEV)
    geom = torch.tensor(_geometry(case), device=DEV)
    if path == "kernel":
        # one-sided differences: 1 K, and 1% of a vmr
        x = torch.cat([t[0], q[0].reshape(-1)])
        h = torch.cat([torch.ones(NLEV, dtype=F64, device=DEV), torch.clamp(0.01 * q[0].reshape(-1), min=1e-15)])
        xs = torch.cat([x[None], x + torch.diag(h)])
        t, q = xs[:, :NLEV], xs[:, NLEV:].reshape(len(xs), ng, NLEV)
        p, nprof = p[:1].expand(len(xs), NLEV), len(xs)
    rays = nprof * nv
    columns = rays * nd * ng * 4
    if columns > (3e5 if path == "jacobian" else 9e6 if case["view"] == "nadir" else 6e6):
        return None
    at = torch.arange(nprof, device=DEV).repeat(nv)
    geom = geom.repeat_interleave(nprof, dim=0)
    if path != "jacobian":
        m = _Model(case, nu, torch.arange(nd, device=DEV).expand(rays, nd))
        with torch.no_grad():
            rad, tau = m(geom, p[at], t[at], q[at])
        if path == "formod":
            return dict(rad=rad.T, tau=tau.T)
        if path == "kernel":
            r = rad.reshape(nv, nprof, nd)
            return dict(k=((r[:, 1:] - r[:, :1]) / h[None, :, None]).permute(0, 2, 1).reshape(nv * nd, -1))
        return dict(rad=rad, tau=tau)
    # one row of K per (ray, channel): each with its own copy of the state,
    # so that one reverse pass over their sum gives every row
    m = _Model(case, nu, torch.arange(nd, device=DEV).repeat(rays)[:, None])
    at = at.repeat_interleave(nd)
    tl, ql = t[at].requires_grad_(True), q[at].requires_grad_(True)
    rad, tau = m(geom.repeat_interleave(nd, dim=0), p[at], tl, ql)
    rad.sum().backward()
    k = torch.cat([tl.grad, ql.grad[:, :min(ng, 3)].reshape(len(at), -1)], 1)
    return dict(rad=rad.detach().reshape(rays, nd), tau=tau.detach().reshape(rays, nd), k=k.reshape(rays, nd, -1))
