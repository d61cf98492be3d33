"""jur_ctx_formod_device_noalloc, the entry point that allocates no device
memory (its work buffers are slices of the library's fixed scratch array),
against jur_ctx_formod_device on the same batches: bit-identical radiances,
transmittances and tangent points, FP64 and FP32, on two calls in a row
(the second smaller), a batch that fills the array, and a clean JUR_ERR_MEM
for a batch whose per-ray buffers exceed it, after which calls still work.
Through the C-ABI.
"""
import ctypes as C

import numpy as np
import pytest

from jurassic_amd import abi, scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu(hip_runtime):
    from jurassic_amd import gpu as G
    G.lib()
    return G


def _batch(torch, ctl, nprof, heights):
    geom = scenes.limb_geometry(800.0, heights)
    nr = len(heights)
    nray = nprof * nr
    atms = (abi.atm_t * nprof)(*[scenes.make_profile_atm(["CO2", "H2O", "O3"], iprof=k) for k in range(nprof)])
    prof = np.array([i % nprof for i in range(nray)], dtype=np.int32)
    g = np.zeros((nray, 7))
    for i in range(nray):
        j = i // nprof
        g[i] = [0.0, geom["obsz"][j], geom["obslon"][j], geom["obslat"][j], geom["vpz"][j], geom["vplon"][j],
                geom["vplat"][j]]
    dev = torch.device("cuda:0")
    a_d = torch.from_numpy(np.frombuffer(bytes(atms), dtype=np.uint8).copy()).to(dev)
    return nprof, a_d, torch.from_numpy(prof).to(dev), torch.from_numpy(g).to(dev), nray


def _run(torch, ctx, fn, b, prec):
    nprof, a_d, prof_d, geom_d, nray = b
    rad = torch.full((nray, ctx.nd), -1.0, dtype=torch.float64, device="cuda:0")
    tau = torch.full_like(rad, -1.0)
    tp = torch.full((nray, 3), -1.0, dtype=torch.float64, device="cuda:0")
    fn(nprof, a_d.data_ptr(), nray, prof_d.data_ptr(), geom_d.data_ptr(), rad.data_ptr(), tau.data_ptr(),
       tp.data_ptr(), precision=prec)
    torch.cuda.synchronize()
    return rad.cpu().numpy(), tau.cpu().numpy(), tp.cpu().numpy()


def test_noalloc_equals_formod_device(gpu):
    torch = pytest.importorskip("torch")
    ctl = scenes.limb_3gas_ctl()
    ctx = gpu.Context(ctl)
    th = scenes.limb_tangent_heights()
    try:
        # 24 x 32 rays = 12 ray blocks: more than one chunk of the scratch
        # array (about 6 blocks of limb LOS), then a smaller second call
        for prec in (abi.JUR_FP64, abi.JUR_FP32):
            for nprof, heights in ((24, th), (2, th[::4])):
                b = _batch(torch, ctl, nprof, heights)
                ref = _run(torch, ctx, ctx.formod_device, b, prec)
                got = _run(torch, ctx, ctx.formod_device_noalloc, b, prec)
                for r, g, what in zip(ref, got, ("rad", "tau", "tp")):
                    assert np.array_equal(r, g), (prec, nprof, what)
                assert np.isfinite(ref[0]).all() and (ref[0] > 0).all()
    finally:
        ctx.close()


def test_noalloc_rejects_batch_beyond_scratch(gpu):
    """About 2.1 million rays: the per-ray state alone exceeds the 256 MiB
    array, so the call returns JUR_ERR_MEM before tracing any ray; a normal
    call works afterwards."""
    torch = pytest.importorskip("torch")
    ctl = scenes.limb_3gas_ctl()
    ctx = gpu.Context(ctl)
    try:
        small = _batch(torch, ctl, 2, scenes.limb_tangent_heights()[::8])
        nprof, a_d, _, _, _ = small
        nray = 2 ** 21
        dev = torch.device("cuda:0")
        prof_d = torch.zeros(nray, dtype=torch.int32, device=dev)
        geom_d = torch.zeros(nray, 7, dtype=torch.float64, device=dev)
        rad = torch.zeros(nray, ctx.nd, dtype=torch.float64, device=dev)
        tau = torch.zeros_like(rad)
        with pytest.raises(gpu.JurassicError) as e:
            ctx.formod_device_noalloc(nprof, a_d.data_ptr(), nray, prof_d.data_ptr(), geom_d.data_ptr(),
                                      rad.data_ptr(), tau.data_ptr(), precision=abi.JUR_FP32)
        assert e.value.code == abi.JUR_ERR_MEM and "scratch" in str(e.value)
        del prof_d, geom_d, rad, tau
        ref = _run(torch, ctx, ctx.formod_device, small, abi.JUR_FP32)
        got = _run(torch, ctx, ctx.formod_device_noalloc, small, abi.JUR_FP32)
        assert all(np.array_equal(r, g) for r, g in zip(ref, got))
    finally:
        ctx.close()


def test_noalloc_full_scratch(gpu):
    """One limb ray of 211 channels and three emitters: the emissivities of
    its block's 1531 points are 211 x 3 x 1531 x 64 x 4 B = 248.1 MB, the LOS
    at its estimated capacity some 20 MB, together within 0.3 MB of the array.
    The call fits without the lookups' cell records (2.3 MB) and is taken
    without them, with the same bits (so is one of 210 channels: the rule
    counts the estimated capacity, not the points)."""
    torch = pytest.importorskip("torch")
    dev = torch.device("cuda:0")
    ng, tp, tt, tu = 3, 30, 2, 4
    p = np.exp(np.linspace(np.log(0.01), np.log(1100.0), tp))
    u = np.array([1e15, 1e20, 1e23, 1e27], dtype=np.float32)
    eps = np.array([1e-8, 1e-4, 0.1, 0.9], dtype=np.float32)
    atm = scenes.make_profile_atm(["CO2", "H2O", "O3"], iprof=0)
    a_d = torch.from_numpy(np.frombuffer(bytes(atm), dtype=np.uint8).copy()).to(dev)
    g = scenes.limb_geometry(800.0, np.array([5.0]))
    geom = np.array([[0.0] + [float(g[k][0]) for k in ("obsz", "obslon", "obslat", "vpz", "vplon", "vplat")]])
    batch = (1, a_d, torch.zeros(1, dtype=torch.int32, device=dev), torch.from_numpy(geom).to(dev), 1)
    for nd in (210, 211):
        nu = [650.0 + 5.0 * i for i in range(nd)]
        i32 = torch.int32
        tabs = dict(np=torch.full((nd, ng), tp, dtype=i32, device=dev),
                    nt=torch.full((nd, ng, tp), tt, dtype=i32, device=dev),
                    nu=torch.full((nd, ng, tp, tt), tu, dtype=i32, device=dev),
                    p=torch.tensor(p, device=dev).expand(nd, ng, tp).contiguous(),
                    t=torch.tensor([150.0, 350.0], dtype=torch.float64, device=dev).expand(nd, ng, tp, tt).contiguous(),
                    u=torch.tensor(u, device=dev).expand(nd, ng, tp, tt, tu).contiguous(),
                    eps=torch.tensor(eps, device=dev).expand(nd, ng, tp, tt, tu).contiguous())
        off = 5 * np.arange(nd + 1, dtype=np.int32)
        xs = np.concatenate([v + np.array([-0.6, -0.5, 0.0, 0.5, 0.6]) for v in nu])
        filt = (off, xs, np.tile(np.array([0.0, 1.0, 1.0, 1.0, 0.0]), nd))
        ctl = abi.make_ctl(["CO2", "H2O", "O3"], nu[:1], tblbase="-", tblfmt=2)
        ctx = gpu.Context.from_device_tables(ctl, nu, tabs, filters=filt)
        try:
            ref = _run(torch, ctx, ctx.formod_device, batch, abi.JUR_FP32)
            assert ctx.last_mean_np() == 1531
            got = _run(torch, ctx, ctx.formod_device_noalloc, batch, abi.JUR_FP32)
            assert all(np.array_equal(r, v) for r, v in zip(ref, got)), nd
        finally:
            ctx.close()
