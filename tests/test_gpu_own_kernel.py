"""The batched step against k_mdfl, the per-tracer kernel of its own.

A per-tracer MDFL-Sweby call without other outputs and with one row a wavefront
runs the batched step's pass (its tendency form), so that a comparison with such
calls would show nothing of a fault of that pass.  Here the per-tracer side runs
k_mdfl, which shares with the pass only the arithmetic of a face
(mdfl64.h): two rows a wavefront, or one with the tendency written to wrk1 too.
Every result is the same, bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KNOB = "mdfl_rows_per_wave"


def test_batched_step_equals_k_mdfl_1440x1080x50():
    """Two whole steps (T, S, diffusion, 80 barotropic subcycles) and one call's
    tendency at full size."""
    from mom5_amd.step import BatchedStep, PlainStep
    from mom5_amd.synth import make_case_device
    print("[own kernel: 1440x1080x50, T and S, two steps]", flush=True)
    case = make_case_device(1440, 1080, 50, land_frac=0.25, nts=80, n_passive=0, seed=0x4D4F4D35)
    g, d = case.info["gpu"], case.fields
    fresh = [(name, case.info["tracer"](n, np.float64)) for n, (name, _) in
             enumerate(case.tracers)]
    tend = []
    for rows in (1, 2):
        g.set_tuning(KNOB, rows)
        th = g.field3()
        g.horz_advect_tracer("mdfl_sweby", fresh[0][1], th, uhrho_et=d["uhrho_et"],
                             vhrho_nt=d["vhrho_nt"], wrho_bt=d["wrho_bt"],
                             rho_dzt_tau=d["rho_dzt"], dtime=case.dt)
        g.sync()
        tend.append(th.to_host())
    assert np.array_equal(*tend)
    plain = PlainStep(case, schemes=["mdfl_sweby"] * 2, gpu=g)        # two rows a wavefront
    batched = BatchedStep(case, gpu=g, tracers=fresh)
    plain.run(2)
    batched.run(2)
    g.sync()
    for n, name in enumerate(plain.names):
        a = plain.tracer(n).to_host()[:, 1:-1, 1:-1]
        assert np.isfinite(a).all(), name
        assert np.array_equal(a, batched.tracer(n).to_host()[:, 1:-1, 1:-1]), name
    g.close()


@pytest.mark.parametrize("cyc", [(1, 0), (0, 0), (1, 1)])
@pytest.mark.parametrize("ni,nj,nk", [(70, 18, 2), (61, 25, 4), (60, 12, 3), (125, 37, 12)])
def test_halos_as_given(cyc, ni, nj, nk):
    """Transports and rho_dzt whose halos hold no wrap, about a region's size, two
    levels up: the batched step's T(taup1) from th_tendency by k_mdfl and the
    explicit update, and the tendency call."""
    from mom5_amd import DeviceArray, OceanGPU
    from mom5_amd.synth import make_case
    print(f"[own kernel {ni}x{nj}x{nk}, cyclic x, y = {cyc}]", flush=True)
    case = make_case(ni, nj, nk, land_frac=0.2, seed=ni + nk, n_passive=1, barotropic=False,
                     cyclic_x=bool(cyc[0]),
                     **({} if cyc[0] else dict(lat_s=20.0, lat_n=50.0, lon_span=30.0)))
    g = OceanGPU(dict(case.dom, cyclic_y=cyc[1]), case.grid)
    rng, H = np.random.default_rng(nk), DeviceArray.from_host
    f = {k: np.array(case.fields[k]) for k in ("uhrho_et", "vhrho_nt", "wrho_bt", "rho_dzt")}
    for name, a in f.items():
        inner, scale = a[:, 1:-1, 1:-1].copy(), np.abs(a).max()
        a[:] = (a.mean() * (0.5 + rng.random(a.shape)) if name == "rho_dzt"
                else 0.1 * scale * rng.standard_normal(a.shape))
        a[:, 1:-1, 1:-1] = inner
    d, rhor = {k: H(v) for k, v in f.items()}, H(1.0 / f["rho_dzt"])
    Ts = [H(np.asarray(t, np.float64)) for _, t in case.tracers]
    th0 = 1e-4 * rng.standard_normal(f["rho_dzt"].shape)
    kw = dict(uhrho_et=d["uhrho_et"], vhrho_nt=d["vhrho_nt"], wrho_bt=d["wrho_bt"],
              rho_dzt_tau=d["rho_dzt"], dtime=case.dt)
    outs = [g.field3() for _ in Ts]
    g.step_tracers(Ts, outs, rho_dztr=rhor, th_tendencies=[H(th0)] + [None] * (len(Ts) - 1), **kw)
    for n, T in enumerate(Ts):
        got = []
        for rows, wrk1 in ((1, None), (2, None), (1, g.field3())):
            g.set_tuning(KNOB, rows)
            tend = H(th0 if n == 0 else np.zeros_like(th0))
            g.horz_advect_tracer("mdfl_sweby", T, tend, wrk1=wrk1, **kw)
            g.sync()
            got.append(tend.to_host())
        assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2]), n
        out = g.field3()
        g.update_tracer_explicit(T, H(got[2]), d["rho_dzt"], rhor, case.dt, out)
        g.sync()
        a = outs[n].to_host()[:, 1:-1, 1:-1]
        assert np.isfinite(a).all(), n
        assert np.array_equal(a, out.to_host()[:, 1:-1, 1:-1]), n
    g.close()
