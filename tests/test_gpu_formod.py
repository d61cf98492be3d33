"""GPU parity of the forward model against the CPU FP64 oracle.

FP64 path: radiance and transmittance within 1e-10 relative of the oracle
(the oracle restates the reference formod; the GPU kernels keep its
operation order except for a few products by reciprocals and the H2O
continuum's power and tanh through exp/expm1, so only differences of a few
ulp remain).
FP32 path: brightness temperature within 0.01 K of the FP64 oracle.
All calls go through the C-ABI of libjurassic_gpu.so.
"""
import ctypes as C
import math
import os
import shutil

import numpy as np
import pytest

from jurassic_amd import abi, scenes

pytestmark = pytest.mark.gpu

RTOL64 = 1e-10
BT_TOL32 = 0.01  # K

GOLD = os.path.join(os.path.dirname(__file__), "golden")


@pytest.fixture(scope="module")
def gpu(hip_runtime):
    from jurassic_amd import gpu as G
    G.lib()
    return G


def _cmp(a, b, rtol, what, atol=0.0):
    a = np.asarray(a, dtype=float)
    b = np.asarray(b, dtype=float)
    assert a.shape == b.shape
    both_nan = np.isnan(a) & np.isnan(b)
    err = np.abs(a - b)
    lim = rtol * np.abs(b) + atol
    bad = ~both_nan & ~(err <= lim)
    if bad.any():
        i = np.argmax(np.where(bad, err / np.maximum(np.abs(b), 1e-300), 0))
        raise AssertionError("%s: %d mismatches, worst at %s: %r vs %r" %
                             (what, bad.sum(), np.unravel_index(i, a.shape), a.flat[i], b.flat[i]))


def _run_both(gpu, oracle, ctl, atm, obs, precision=abi.JUR_FP64):
    o_cpu = abi.copy_struct(obs)
    a_cpu = abi.copy_struct(atm)
    oracle.formod(ctl, a_cpu, o_cpu)
    o_gpu = abi.copy_struct(obs)
    a_gpu = abi.copy_struct(atm)
    gpu.formod(ctl, a_gpu, o_gpu, precision)
    return (a_cpu, o_cpu), (a_gpu, o_gpu)


def _assert_obs(ctl, o_gpu, o_cpu, rtol=RTOL64, row_scaled=False):
    r1, t1 = abi.obs_arrays(o_gpu, ctl)
    r0, t0 = abi.obs_arrays(o_cpu, ctl)
    if row_scaled:
        # combinations with negative weights (extrapolating interpolation):
        # the bound applies relative to the largest input of the channel
        _cmp(r1, r0, 0, "rad", atol=rtol * np.abs(r0).max(axis=1, keepdims=True))
        _cmp(t1, t0, 0, "tau", atol=rtol * np.abs(t0).max(axis=1, keepdims=True))
    else:
        _cmp(r1, r0, rtol, "rad")
        _cmp(t1, t0, rtol, "tau", atol=1e-300)
    nr = o_cpu.nr
    for f in ("tpz", "tplon", "tplat"):
        _cmp(np.ctypeslib.as_array(getattr(o_gpu, f))[:nr],
             np.ctypeslib.as_array(getattr(o_cpu, f))[:nr], 1e-11, f, atol=1e-9)


def test_nadir_co2_fp64(gpu, oracle):
    ctl, atm, obs = scenes.nadir_co2()
    (_, oc), (_, og) = _run_both(gpu, oracle, ctl, atm, obs)
    _assert_obs(ctl, og, oc)
    rad, tau = abi.obs_arrays(og, ctl)
    assert np.all(rad > 0) and np.all((tau > 0) & (tau < 1))


def test_nadir_co2_bbt_fp64(gpu, oracle):
    ctl, atm, obs = scenes.nadir_co2()
    ctl.write_bbt = 1
    (_, oc), (_, og) = _run_both(gpu, oracle, ctl, atm, obs)
    _assert_obs(ctl, og, oc)


def test_limb_3gas_fp64(gpu, oracle):
    for iprof in (0, 7):
        ctl, atm, obs = scenes.limb_3gas(iprof)
        (_, oc), (_, og) = _run_both(gpu, oracle, ctl, atm, obs)
        _assert_obs(ctl, og, oc)


def test_limb_3gas_no_continua_fp64(gpu, oracle):
    ctl, atm, obs = scenes.limb_3gas(3, ctm=False)
    (_, oc), (_, og) = _run_both(gpu, oracle, ctl, atm, obs)
    _assert_obs(ctl, og, oc)


def test_cga_fp64(gpu, oracle):
    ctl, atm, obs = scenes.limb_3gas(1, nrays=12)
    ctl.formod = 0
    (_, oc), (_, og) = _run_both(gpu, oracle, ctl, atm, obs)
    _assert_obs(ctl, og, oc)
    ctl, atm, obs = scenes.nadir_co2()
    ctl.formod = 0
    (_, oc), (_, og) = _run_both(gpu, oracle, ctl, atm, obs)
    _assert_obs(ctl, og, oc)


def test_batch_matches_oracle_and_single(gpu, oracle):
    """Packages of different atmospheres in one pass equal separate calls."""
    n = 5
    ctl = scenes.limb_3gas_ctl()
    atms = (abi.atm_t * n)()
    obss = (abi.obs_t * n)()
    for k in range(n):
        atms[k] = scenes.make_profile_atm(["CO2", "H2O", "O3"], iprof=100 + k)
        obss[k] = scenes.make_obs(scenes.limb_geometry(800.0, scenes.limb_tangent_heights()[k::3]))
    gpu.formod_batch(ctl, atms, obss)
    for k in range(n):
        o1 = scenes.make_obs(scenes.limb_geometry(800.0, scenes.limb_tangent_heights()[k::3]))
        a1 = abi.copy_struct(atms[k])
        oracle.formod(ctl, a1, o1)
        _assert_obs(ctl, obss[k], o1)
        o2 = scenes.make_obs(scenes.limb_geometry(800.0, scenes.limb_tangent_heights()[k::3]))
        gpu.formod(ctl, abi.copy_struct(atms[k]), o2)
        r1, _ = abi.obs_arrays(obss[k], ctl)
        r2, _ = abi.obs_arrays(o2, ctl)
        np.testing.assert_array_equal(r1, r2)


def _bt(rad, nu):
    c1, c2 = 1.19104259e-8, 1.43877506
    return c2 * nu / np.log1p(c1 * nu ** 3 / rad)


def test_fp32_bt_error(gpu, oracle):
    """FP32 lookups with compensated sums stay within 0.01 K of FP64."""
    worst = 0.0
    for make in (lambda: scenes.limb_3gas(0), lambda: scenes.limb_3gas(11), scenes.nadir_co2):
        ctl, atm, obs = make()
        ctl.write_bbt = 1
        (_, oc), (_, og) = _run_both(gpu, oracle, ctl, atm, obs, abi.JUR_FP32)
        r1, t1 = abi.obs_arrays(og, ctl)
        r0, t0 = abi.obs_arrays(oc, ctl)
        err = np.abs(r1 - r0)
        worst = max(worst, float(err.max()))
        assert err.max() <= BT_TOL32, err.max()
        assert np.abs(t1 - t0).max() <= 1e-4
    print("worst FP32 BT error %.2e K" % worst)


def test_fp32_cga(gpu, oracle):
    ctl, atm, obs = scenes.limb_3gas(2, nrays=16)
    ctl.formod = 0
    ctl.write_bbt = 1
    (_, oc), (_, og) = _run_both(gpu, oracle, ctl, atm, obs, abi.JUR_FP32)
    r1, _ = abi.obs_arrays(og, ctl)
    r0, _ = abi.obs_arrays(oc, ctl)
    assert np.abs(r1 - r0).max() <= BT_TOL32


def _golden_ctl(tmp_path, name):
    """The reference's limb/nadir test geometry and atmosphere with boxcar
    filters and no emissivity tables (missing tables give eps = 0, as in the
    reference), for the tangent-point columns of rad.org."""
    if name == "limb_test":
        em, nu = ["CO2", "H2O", "O3", "F11", "CCl4"], [792.0, 832.0]
    else:
        em, nu = ["CO2"], [667.782, 668.541, 669.811]
    tb = os.path.join(str(tmp_path), "g")
    for v in nu:
        scenes.write_boxcar_filter("%s_%.4f.filt" % (tb, v), v)
    ctl = abi.make_ctl(em, nu, tblbase=tb)
    atm = abi.read_atm(os.path.join(GOLD, name, "atm.tab"), ctl)
    obs = abi.read_obs(os.path.join(GOLD, name, "obs.tab"), ctl)
    ref = abi._data_rows(os.path.join(GOLD, name, "rad.org"))
    return ctl, atm, obs, ref


@pytest.mark.parametrize("name", ["limb_test", "nadir_test"])
def test_golden_tangent_points(gpu, tmp_path, name):
    ctl, atm, obs, ref = _golden_ctl(tmp_path, name)
    gpu.formod(ctl, atm, obs)
    for ir in range(obs.nr):
        got = (obs.tpz[ir], obs.tplon[ir], obs.tplat[ir])
        for j, v in enumerate(got):
            r = ref[ir][7 + j]
            if abs(r) < 1e-6:
                # rounding-noise values (e.g. a longitude of 1e-10 deg from
                # atan2 of a vanishing component, or the 1e-8 km ground-clip
                # residual): equal to far below any physical resolution
                assert abs(v - r) < 1e-9, (name, ir, j, v, r)
            else:
                assert "%g" % v == "%g" % r, (name, ir, j, v, r)
    rad, tau = abi.obs_arrays(obs, ctl)
    # without tables only the continua absorb
    assert np.all(tau > 0) and np.all(tau <= 1)


def test_surface_reflection_and_solar(gpu, oracle):
    ctl, atm, obs = scenes.nadir_co2()
    ctl.nsf = 2
    ctl.sfnu[0], ctl.sfnu[1] = 600.0, 800.0
    ctl.sftype = 3
    ctl.sfsza = 30.0
    atm.sfz = 0.0
    atm.sfp = 0.0
    atm.sft = 295.0
    atm.sfeps[0], atm.sfeps[1] = 0.8, 0.95
    (_, oc), (_, og) = _run_both(gpu, oracle, ctl, atm, obs)
    _assert_obs(ctl, og, oc)
    ctl.sfsza = -999  # solar zenith angle from time and position
    for ir in range(obs.nr):
        obs.time[ir] = 1.5e8 + 3600.0 * ir
    (_, oc), (_, og) = _run_both(gpu, oracle, ctl, atm, obs)
    _assert_obs(ctl, og, oc)


def test_clouds(gpu, oracle):
    ctl, atm, obs = scenes.limb_3gas(4, nrays=10)
    ctl.ncl = 2
    ctl.clnu[0], ctl.clnu[1] = 650.0, 1500.0
    atm.clz = 12.0
    atm.cldz = 1.5
    atm.clk[0], atm.clk[1] = 0.02, 0.05
    (_, oc), (_, og) = _run_both(gpu, oracle, ctl, atm, obs)
    _assert_obs(ctl, og, oc)


def test_extinction_window(gpu, oracle):
    ctl, atm, obs = scenes.limb_3gas(5, nrays=10)
    ctl.nw = 2
    for id_ in range(ctl.nd):
        ctl.window[id_] = id_ % 2
    for i in range(atm.np):
        atm.k[0][i] = 1e-3 * math.exp(-atm.z[i] / 10)
        atm.k[1][i] = 2e-3 * math.exp(-atm.z[i] / 5)
    (_, oc), (_, og) = _run_both(gpu, oracle, ctl, atm, obs)
    _assert_obs(ctl, og, oc)


def test_hydrostatic(gpu, oracle):
    ctl, atm, obs = scenes.limb_3gas(6, nrays=8)
    ctl.hydz = 10.0
    (ac, oc), (ag, og) = _run_both(gpu, oracle, ctl, atm, obs)
    _assert_obs(ctl, og, oc)
    _cmp(np.ctypeslib.as_array(ag.p)[:atm.np], np.ctypeslib.as_array(ac.p)[:atm.np], 1e-13, "p")


def test_fov(gpu, oracle, tmp_path):
    ctl, atm, obs = scenes.limb_3gas(8)
    fov = os.path.join(str(tmp_path), "fov.tab")
    with open(fov, "w") as f:
        for dz in np.linspace(-1.5, 1.5, 31):
            f.write("%g %g\n" % (dz, math.exp(-dz * dz)))
    ctl.fov = fov.encode()
    (_, oc), (_, og) = _run_both(gpu, oracle, ctl, atm, obs)
    _assert_obs(ctl, og, oc, row_scaled=True)


def test_mask_nan(gpu, oracle):
    ctl, atm, obs = scenes.nadir_co2()
    obs.rad[1][3] = float("nan")
    obs.rad[0][7] = float("nan")
    (_, oc), (_, og) = _run_both(gpu, oracle, ctl, atm, obs)
    _assert_obs(ctl, og, oc)
    assert math.isnan(og.rad[1][3]) and math.isnan(og.rad[0][7])
    assert not math.isnan(og.rad[0][3])


def test_ascii_tables(gpu, oracle, tmp_path):
    """TBLFMT = 1: the ASCII reader (with the monotonicity merge of saturated
    rows) on both sides."""
    nus = [667.8]
    d = str(tmp_path)
    tb = scenes.write_scene_tables(d, ["CO2"], nus, fmt=1)
    ctl = abi.make_ctl(["CO2"], nus, tblbase=tb, tblfmt=1)
    atm = scenes.make_profile_atm(["CO2"])
    obs = scenes.make_obs(scenes.nadir_geometry(705.0, [0.0, 30.0]))
    (_, oc), (_, og) = _run_both(gpu, oracle, ctl, atm, obs)
    _assert_obs(ctl, og, oc)


def test_missing_table_is_transparent(gpu, oracle, tmp_path):
    ctl, atm, obs = scenes.nadir_co2()
    d = str(tmp_path)
    for v in (667.8, 668.5):
        shutil.copy("%s_%.4f.filt" % (ctl.tblbase.decode(), v), os.path.join(d, "m_%.4f.filt" % v))
    shutil.copy("%s_%.4f_CO2.bin" % (ctl.tblbase.decode(), 667.8), os.path.join(d, "m_667.8000_CO2.bin"))
    ctl.tblbase = os.path.join(d, "m").encode()
    (_, oc), (_, og) = _run_both(gpu, oracle, ctl, atm, obs)
    _assert_obs(ctl, og, oc)


def test_error_observer_below_surface(gpu):
    ctl, atm, obs = scenes.nadir_co2()
    obs.obsz[2] = -1.0
    with pytest.raises(gpu.JurassicError) as e:
        gpu.formod(ctl, atm, obs)
    assert e.value.code == 4


def test_error_too_many_los_points(gpu):
    ctl, atm, obs = scenes.nadir_co2()
    ctl.raydz = 0.01  # 8000 points on an 80 km nadir path > NLOS
    with pytest.raises(gpu.JurassicError) as e:
        gpu.formod(ctl, atm, obs)
    assert e.value.code == 3


def test_kernel_fd_matches_oracle(gpu, oracle):
    ctl, atm, obs = scenes.nadir_co2()
    ctl.rett_zmin, ctl.rett_zmax = -100, 100
    ctl.retq_zmin[0], ctl.retq_zmax[0] = -100, 100
    m, n = oracle.sizes(ctl, atm, obs)
    k0 = oracle.kernel(ctl, abi.copy_struct(atm), abi.copy_struct(obs))
    k1 = gpu.kernel(ctl, abi.copy_struct(atm), abi.copy_struct(obs), m=m, n=n)
    # Both sides difference radiances that agree to 1e-10 relative, so each
    # entry agrees to about 2e-10 |y_i| / h_j (columns with almost no
    # sensitivity are rounding noise on both sides).
    o = abi.copy_struct(obs)
    oracle.formod(ctl, abi.copy_struct(atm), o)
    y = np.abs(np.array([o.rad[i % ctl.nd][i // ctl.nd] for i in range(m)]))
    x = np.concatenate([np.ctypeslib.as_array(atm.t)[:atm.np], np.ctypeslib.as_array(atm.q[0])[:atm.np]])
    h = np.concatenate([np.ones(atm.np), np.maximum(np.abs(0.01 * x[atm.np:]), 1e-15)])
    tol = 1e-9 * y[:, None] / h[None, :]
    assert np.all(np.abs(k1 - k0) <= tol)
    assert np.abs(k1 - k0).max() / np.abs(k0).max() < 1e-7


def test_formod_gpu_and_kernel_gpu_dropins(gpu, oracle):
    """The literal drop-ins: formod_gpu (void, ERRMSG-style errors) and
    kernel_gpu (void, finite differences in FP64) on a valid nadir case,
    against the oracle's formod and kernel()."""
    L = gpu.lib()
    L.formod_gpu.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p]
    L.formod_gpu.restype = None
    L.kernel_gpu.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p, C.POINTER(C.c_double), C.c_size_t, C.c_size_t]
    L.kernel_gpu.restype = None
    ctl, atm, obs = scenes.nadir_co2()
    ctl.write_bbt = 1
    o_gpu, a_gpu = abi.copy_struct(obs), abi.copy_struct(atm)
    L.formod_gpu(C.byref(ctl), C.byref(a_gpu), C.byref(o_gpu))
    o_cpu = abi.copy_struct(obs)
    oracle.formod(ctl, abi.copy_struct(atm), o_cpu)
    _assert_obs(ctl, o_gpu, o_cpu)
    ctl.rett_zmin, ctl.rett_zmax = -100, 100
    m, n = oracle.sizes(ctl, atm, obs)
    k0 = oracle.kernel(ctl, abi.copy_struct(atm), abi.copy_struct(obs))
    k1 = np.zeros((m, n))
    L.kernel_gpu(C.byref(ctl), C.byref(abi.copy_struct(atm)), C.byref(abi.copy_struct(obs)),
                 k1.ctypes.data_as(C.POINTER(C.c_double)), m, n)
    # BT differences over a 1 K step: entries agree to about 1e-10 BT / 1 K
    assert np.abs(k1 - k0).max() <= 2e-7
    assert np.abs(k0).max() > 0.01


def test_empty_inputs(gpu, oracle):
    """No rays: formod's ray loop (src/jurassic.c:3047) and kernel()'s rows
    are empty, and the entry points return without error. A package without
    rays in a batch leaves the others' results as they are alone, and a
    device batch without rays (null pointers) and a server request without
    rays are accepted and rejected as documented."""
    ctl, atm, obs = scenes.nadir_co2()
    empty = abi.copy_struct(obs)
    empty.nr = 0
    for prec in (abi.JUR_FP64, abi.JUR_FP32):
        o = abi.copy_struct(empty)
        gpu.formod(ctl, abi.copy_struct(atm), o, prec)
        assert o.nr == 0
    atms = (abi.atm_t * 3)()
    obss = (abi.obs_t * 3)()
    for k, src in enumerate((empty, obs, empty)):
        atms[k] = abi.copy_struct(atm)
        obss[k] = abi.copy_struct(src)
    gpu.formod_batch(ctl, atms, obss)
    alone = abi.copy_struct(obs)
    gpu.formod(ctl, abi.copy_struct(atm), alone)
    np.testing.assert_array_equal(abi.obs_arrays(obss[1], ctl)[0], abi.obs_arrays(alone, ctl)[0])
    assert obss[0].nr == 0 and obss[2].nr == 0

    ctl.rett_zmin, ctl.rett_zmax = -100, 100
    m, n = oracle.sizes(ctl, atm, empty)
    assert m == 0 and n > 0
    for method, prec in ((abi.JUR_JAC_FD, abi.JUR_FP64), (abi.JUR_JAC_ADJOINT, abi.JUR_FP32)):
        k = gpu.kernel(ctl, abi.copy_struct(atm), abi.copy_struct(empty), method, prec, m=m, n=n)
        assert k.shape == (0, n)

    ctx = gpu.Context(ctl)
    try:
        for prec in (abi.JUR_FP64, abi.JUR_FP32):
            ctx.formod_device(0, None, 0, None, None, None, None, precision=prec)
        xm, n1 = gpu.state_map(ctl, atm)
        ctx.jacobian_device(0, None, 0, None, None, None, None, xm[None, :], None, n1, None,
                            precision=abi.JUR_FP32)
    finally:
        ctx.close()

    srv = gpu.Server(ctl, _ret_for_empty(ctl.nd))
    try:
        with pytest.raises(gpu.JurassicError, match="without rays"):
            srv.submit(gpu.Server.request(abi.JUR_REQ_FORWARD, atm, empty))
    finally:
        srv.close()


def test_max_rays(gpu, oracle):
    """One observation at its capacity, obs->nr = NR (128 nadir and 128 limb
    rays of uneven LOS lengths), against the oracle; NR + 1 rays are
    rejected as the reference's raytrace/formod ERRMSG does ("Too many
    rays!")."""
    ctl, atm, _ = scenes.nadir_co2()
    half = abi.NR // 2
    g1 = scenes.nadir_geometry(705.0, np.linspace(0.0, 60.0, half))
    g2 = scenes.limb_geometry(800.0, np.linspace(4.0, 70.0, abi.NR - half))
    obs = scenes.make_obs({k: np.concatenate([g1[k], g2[k]]) for k in g1})
    assert obs.nr == abi.NR
    (_, o_cpu), (_, o_gpu) = _run_both(gpu, oracle, ctl, atm, obs)
    _assert_obs(ctl, o_gpu, o_cpu)
    (_, o_cpu), (_, o_gpu) = _run_both(gpu, oracle, ctl, atm, obs, abi.JUR_FP32)
    r1, _ = abi.obs_arrays(o_gpu, ctl)
    r0, _ = abi.obs_arrays(o_cpu, ctl)
    nu = np.asarray(ctl.nu[:ctl.nd])[:, None]
    assert np.abs(_bt(r1, nu) - _bt(r0, nu)).max() <= BT_TOL32
    bad = abi.copy_struct(obs)
    bad.nr = abi.NR + 1
    with pytest.raises(gpu.JurassicError, match="Too many rays"):
        gpu.formod(ctl, abi.copy_struct(atm), bad)


def _ret_for_empty(nd):
    ret = abi.ret_t()
    ret.kernel_recomp = 3
    ret.conv_itmax = 10
    ret.conv_dmin = 0.1
    for id in range(nd):
        ret.err_noise[id] = 0.1
    ret.err_temp = 5.0
    return ret


def test_fp32_bt_bound_limb_at_scale(gpu, oracle):
    """The 0.01 K bound over a large batch of the limb workload: 512
    atmospheres (seeded perturbed profiles) x 32 tangent heights 5..67 km x
    12 channels, CO2/H2O/O3, continua and refraction on (196,608
    radiances).  The FP64 device pass is the reference arithmetic (checked
    against the oracle to 1e-10 on the first two atmospheres), the FP32 pass
    must stay within 0.01 K of it everywhere."""
    torch = pytest.importorskip("torch")
    ctl = scenes.limb_3gas_ctl()
    zt = scenes.limb_tangent_heights()
    geom = scenes.limb_geometry(800.0, zt)
    nprof, nr = 512, len(zt)
    gases = [ctl.emitter[i].value.decode() for i in range(ctl.ng)]
    atms = (abi.atm_t * nprof)()
    for k in range(nprof):
        atms[k] = scenes.make_profile_atm(gases, iprof=k)
    nray = nprof * nr
    prof = np.tile(np.arange(nprof, dtype=np.int32), nr)
    g = np.zeros((nray, 7))
    for j in range(nr):
        for c, key in enumerate(("obsz", "obslon", "obslat", "vpz", "vplon", "vplat")):
            g[j * nprof:(j + 1) * nprof, 1 + c] = geom[key][j]
    dev = torch.device("cuda:0")
    a_d = torch.from_numpy(np.frombuffer(bytes(atms), dtype=np.uint8).copy()).to(dev)
    p_d, g_d = torch.from_numpy(prof).to(dev), torch.from_numpy(g).to(dev)
    ctx = gpu.Context(ctl)
    out = {}
    try:
        for prec in (abi.JUR_FP64, abi.JUR_FP32):
            rad = torch.zeros(nray, ctl.nd, dtype=torch.float64, device=dev)
            tau = torch.zeros_like(rad)
            ctx.formod_device(nprof, a_d.data_ptr(), nray, p_d.data_ptr(), g_d.data_ptr(), rad.data_ptr(),
                              tau.data_ptr(), precision=prec)
            torch.cuda.synchronize()
            out[prec] = rad.cpu().numpy().reshape(nr, nprof, ctl.nd)
    finally:
        ctx.close()
    for k in range(2):
        obs = scenes.make_obs(geom)
        oracle.formod(ctl, scenes.make_profile_atm(gases, iprof=k), obs)
        r0, _ = abi.obs_arrays(obs, ctl)
        _cmp(out[abi.JUR_FP64][:, k, :], r0.T, RTOL64, "FP64 device pass vs oracle, atmosphere %d" % k)
    nu = np.array([ctl.nu[i] for i in range(ctl.nd)])
    c1, c2 = 1.19104259e-8, 1.43877506

    def bt(r):
        return c2 * nu / np.log1p(c1 * nu ** 3 / r)
    err = np.abs(bt(out[abi.JUR_FP32]) - bt(out[abi.JUR_FP64]))
    assert np.isfinite(err).all()
    print("FP32 vs FP64 over %d radiances: max %.2e K, mean %.2e K" % (err.size, err.max(), err.mean()))
    assert err.max() <= BT_TOL32


def _limb_batch(torch, ctl, nprof):
    zt = scenes.limb_tangent_heights()
    geom = scenes.limb_geometry(800.0, zt)
    nr = len(zt)
    gases = [ctl.emitter[i].value.decode() for i in range(ctl.ng)]
    atms = (abi.atm_t * nprof)()
    for k in range(nprof):
        atms[k] = scenes.make_profile_atm(gases, iprof=k)
    nray = nprof * nr
    prof = np.tile(np.arange(nprof, dtype=np.int32), nr)
    g = np.zeros((nray, 7))
    for j in range(nr):
        for c, key in enumerate(("obsz", "obslon", "obslat", "vpz", "vplon", "vplat")):
            g[j * nprof:(j + 1) * nprof, 1 + c] = geom[key][j]
    dev = torch.device("cuda:0")
    a_d = torch.from_numpy(np.frombuffer(bytes(atms), dtype=np.uint8).copy()).to(dev)
    return atms, a_d, torch.from_numpy(prof).to(dev), torch.from_numpy(g).to(dev), nray, nr


def test_raytrace_lanes_per_ray_agree(gpu):
    """The ray tracer marches a ray on one lane for large batches and on four
    (one refraction probe each, exchanged by shuffles) for small ones, and
    the FP32 lookups run a chain on one lane or on four (one cell corner
    each); both with the same operations on the same values.  The FP64 and
    FP32 radiances of the same rays are equal to the last bit between a
    batch of 1100 limb atmospheres x 32 tangent heights (550 ray blocks, one
    lane per ray and chain) and one of its first 64 atmospheres (four)."""
    torch = pytest.importorskip("torch")
    ctl = scenes.limb_3gas_ctl()
    assert ctl.refrac == 1
    out = {abi.JUR_FP64: [], abi.JUR_FP32: []}
    for nprof in (1100, 64):
        atms, a_d, p_d, g_d, nray, nr = _limb_batch(torch, ctl, nprof)
        ctx = gpu.Context(ctl)
        try:
            for prec in out:
                rad = torch.zeros(nray, ctl.nd, dtype=torch.float64, device="cuda:0")
                tau = torch.zeros_like(rad)
                ctx.formod_device(nprof, a_d.data_ptr(), nray, p_d.data_ptr(), g_d.data_ptr(), rad.data_ptr(),
                                  tau.data_ptr(), precision=prec)
                torch.cuda.synchronize()
                out[prec].append(rad.cpu().numpy().reshape(nr, nprof, ctl.nd)[:, :64])
        finally:
            ctx.close()
    for prec, (big, small) in out.items():
        assert np.isfinite(big).all() and (big > 0).all()
        assert np.array_equal(big, small), prec


def test_lookup_lanes_per_chain_jacobian_agree(gpu):
    """The FP32 lookups with stored partials on four lanes per chain (small
    batches) give the Jacobian of the one-lane chains: K rows of 16 limb
    atmospheres x 32 tangent heights (T and H2O columns) agree between that
    batch alone (8 ray blocks: four lanes) and inside one of 80 atmospheres
    (40 blocks, more than the four-lane grid's 5120 wavefronts: one lane);
    both run the adjoint with one workgroup per row."""
    torch = pytest.importorskip("torch")
    ctl = scenes.limb_3gas_ctl()
    ctl.rett_zmin, ctl.rett_zmax = -100.0, 100.0
    ctl.retq_zmin[1], ctl.retq_zmax[1] = -100.0, 100.0
    out = []
    for nprof in (80, 16):
        atms, a_d, p_d, g_d, nray, nr = _limb_batch(torch, ctl, nprof)
        xm, n = gpu.state_map(ctl, atms[0])
        ctx = gpu.Context(ctl)
        try:
            rad = torch.zeros(nray, ctl.nd, dtype=torch.float64, device="cuda:0")
            tau = torch.zeros_like(rad)
            kd = torch.zeros(nray, ctl.nd, n, dtype=torch.float64, device="cuda:0")
            pmap = torch.zeros(nprof, dtype=torch.int32, device="cuda:0")
            ctx.jacobian_device(nprof, a_d.data_ptr(), nray, p_d.data_ptr(), g_d.data_ptr(), rad.data_ptr(),
                                tau.data_ptr(), xm[None, :], pmap.data_ptr(), n, kd.data_ptr(),
                                precision=abi.JUR_FP32)
            torch.cuda.synchronize()
            k = kd.view(nr, nprof, ctl.nd, n)[:, :16].cpu().numpy()
            out.append((rad.view(nr, nprof, -1)[:, :16].cpu().numpy(), k))
        finally:
            ctx.close()
    (r0, k0), (r1, k1) = out
    assert np.array_equal(r0, r1)
    assert np.isfinite(k0).all() and np.abs(k0).max() > 0
    np.testing.assert_allclose(k1, k0, rtol=1e-13, atol=1e-13 * np.abs(k0).max())


@pytest.mark.parametrize("nlev,up,refrac", [(2, True, 1), (8, False, 1), (9, True, 0), (10, True, 1), (17, False, 1)])
def test_level_grids(gpu, oracle, nlev, up, refrac):
    """Level counts around the rounds of eight of the march's altitude scan,
    ascending and descending grids, with and without refraction: the
    oracle's radiances and tangent points of limb and nadir rays.
    Transmittances to 1e-10 relative or 1e-30: that of a path of optical
    depth x carries x times the rounding of the depth, which is summed over
    about 1000 segments (up to 1e-12), so 1e-10 need not hold beyond x = 70."""
    z = np.linspace(0.0, 80.0, nlev)
    ctl, _, obs = scenes.limb_3gas(0, nrays=7)
    ctl.refrac = refrac
    atm = scenes.make_profile_atm(["CO2", "H2O", "O3"], z=z, perturb=False)
    if not up:
        rows = [atm.z, atm.p, atm.t] + [atm.q[g] for g in range(3)]
        for a in rows:
            v = abi.np_view(a)
            v[:nlev] = v[:nlev][::-1].copy()
    for o in (obs, scenes.make_obs(scenes.nadir_geometry(705.0, [0.0, 30.0, 55.0]))):
        (_, oc), (_, og) = _run_both(gpu, oracle, ctl, atm, o)
        r1, t1 = abi.obs_arrays(og, ctl)
        r0, t0 = abi.obs_arrays(oc, ctl)
        _cmp(r1, r0, RTOL64, "rad")
        _cmp(t1, t0, RTOL64, "tau", atol=1e-30)
        _cmp(abi.np_view(og.tpz)[:o.nr], abi.np_view(oc.tpz)[:o.nr], 1e-11, "tpz", atol=1e-9)


@pytest.mark.parametrize("nr", [1, 63, 65])
def test_radiance_waves_per_path_agree(gpu, nr):
    """A small batch forms a path's segments on several waves (FP32 16 or 4,
    FP64 8), a large one on one: the same bits for one package of 1, 63 or 65
    rays (a block with one lane, one short, two blocks) and for it among
    copies of itself that make 19 blocks x 12 channels (more than the 256
    workgroups of the FP32 launch with 16 waves, with the rounding to eight
    blocks) and 100 x 12 (more than the 1024 with 4 and the 512 with 8).  Limb
    paths and, every other ray, paths to a reflecting surface (emissivity
    0.8), where the down-welling sum enters the radiance: it moves there by
    more than 1e-6 with the emissivity."""
    ctl = scenes.limb_3gas_ctl()
    ctl.sftype, ctl.nsf = 2, 2
    ctl.sfnu[0], ctl.sfnu[1] = 600.0, 1600.0
    atm = scenes.make_profile_atm(["CO2", "H2O", "O3"], iprof=2)
    atm.sft = 290.0
    limb = scenes.limb_geometry(800.0, np.linspace(5.0, 60.0, nr))
    down = scenes.nadir_geometry(800.0, np.linspace(0.0, 50.0, nr))
    geom = {k: np.where(np.arange(nr) % 2 == 1, limb[k], down[k]) for k in limb}
    rads = []
    for prec in (abi.JUR_FP64, abi.JUR_FP32):
        ref = {}
        for eps in (1.0, 0.8):
            atm.sfeps[0] = atm.sfeps[1] = eps
            one = scenes.make_obs(geom)
            gpu.formod(ctl, abi.copy_struct(atm), one, prec)
            ref[eps] = abi.obs_arrays(one, ctl)
        r0, t0 = ref[0.8]
        assert np.isfinite(r0).all() and (r0 > 0).any()
        # with an emissivity below 1 the emission falls by (1 - eps) src tau
        # and the reflection adds (1 - eps) D tau: both enter if the change
        # is neither zero nor the emission's alone
        c1, c2 = 1.19104259e-8, 1.43877506
        nu = np.array([ctl.nu[i] for i in range(ctl.nd)])[:, None]
        emis = -0.2 * c1 * nu ** 3 / np.expm1(c2 * nu / 290.0) * t0
        change = r0 - ref[1.0][0]
        rads.append(r0)
        k = np.arange(0, nr, 2)
        assert (np.abs(change - emis)[:, k].max(axis=1) > 1e-6 * r0[:, k].max(axis=1)).any()
        for blocks in (19, 100):
            n = -(-64 * blocks // nr)
            atms, obss = (abi.atm_t * n)(), (abi.obs_t * n)()
            for q in range(n):
                atms[q] = atm
                obss[q] = scenes.make_obs(geom)
            gpu.formod_batch(ctl, atms, obss, prec)
            for q in (0, n // 2, n - 1):
                r1, t1 = abi.obs_arrays(obss[q], ctl)
                assert np.array_equal(r0, r1) and np.array_equal(t0, t1), (prec, blocks, q)
    # FP32 against FP64: some 1e-6 (float segments of ~1000 points)
    np.testing.assert_allclose(rads[1], rads[0], rtol=1e-5, atol=1e-7 * rads[0].max())


@pytest.mark.parametrize("nray", [3, 5600])
def test_bad_atmosphere_index(gpu, nray):
    """A device batch whose rays name atmospheres that are not there, with
    clouds and surface emissivities on (read per ray before any of its
    points): JUR_ERR_ARG from the forward model and the Jacobian, in batches
    on several waves per path and on one, and a good call afterwards.  The
    last ray is a bad one: the lanes behind it in its block follow it."""
    torch = pytest.importorskip("torch")
    ctl = scenes.limb_3gas_ctl()
    ctl.ncl, ctl.nsf, ctl.sftype = 2, 2, 2
    for i in range(2):
        ctl.clnu[i], ctl.sfnu[i] = (600.0, 1600.0)[i], (600.0, 1600.0)[i]
    ctl.rett_zmin, ctl.rett_zmax = -100, 100
    atms = (abi.atm_t * 2)()
    for k in range(2):
        atms[k] = scenes.make_profile_atm(["CO2", "H2O", "O3"], iprof=k)
        atms[k].clz, atms[k].cldz, atms[k].sft = 8.0, 1.5, 290.0
        for i in range(2):
            atms[k].clk[i], atms[k].sfeps[i] = 0.02, 0.8
    dev = torch.device("cuda:0")
    a_d = torch.from_numpy(np.frombuffer(bytes(atms), dtype=np.uint8).copy()).to(dev)
    one = scenes.nadir_geometry(705.0, [20.0])
    geom = torch.zeros(nray, 7, dtype=torch.float64)
    for c, key in enumerate(("obsz", "obslon", "obslat", "vpz", "vplon", "vplat")):
        geom[:, 1 + c] = float(one[key][0])
    geom = geom.to(dev)
    good = (torch.arange(nray, dtype=torch.int32) % 2).to(dev)
    bad = good.clone()
    bad[0], bad[nray - 1] = -1, 2
    xm, n = gpu.state_map(ctl, atms[0])
    pmap = torch.zeros(2, dtype=torch.int32, device=dev)
    rad = torch.zeros(nray, ctl.nd, dtype=torch.float64, device=dev)
    tau = torch.zeros_like(rad)
    k = torch.zeros(3, ctl.nd, n, dtype=torch.float64, device=dev)
    ctx = gpu.Context(ctl)
    try:
        for prec in (abi.JUR_FP64, abi.JUR_FP32):
            def call(prof):
                ctx.formod_device(2, a_d.data_ptr(), nray, prof.data_ptr(), geom.data_ptr(), rad.data_ptr(),
                                  tau.data_ptr(), precision=prec)

            def jac(prof):
                ctx.jacobian_device(2, a_d.data_ptr(), 3, prof.data_ptr(), geom.data_ptr(), rad.data_ptr(),
                                    tau.data_ptr(), xm[None, :], pmap.data_ptr(), n, k.data_ptr(), precision=prec)
            for f in (call, jac) if nray == 3 else (call,):
                with pytest.raises(gpu.JurassicError) as e:
                    f(bad)
                assert e.value.code == abi.JUR_ERR_ARG
            call(good)
            torch.cuda.synchronize()
            assert bool((rad > 0).all()) and bool(torch.isfinite(rad).all())
            # rays of one atmosphere and geometry agree, the last one too
            assert bool((rad[nray - 1] == rad[(nray - 1) % 2]).all())
    finally:
        ctx.close()
