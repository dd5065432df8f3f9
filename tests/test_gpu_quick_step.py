"""Quicker tracers in the batched step (mom_gpu_step_tracers with
scheme[n] = QUICKER): horizontal and vertical Quicker advection, the
tmask_limit flags formed inside the pass, the explicit update and the
implicit vertical diffusion, against

* the oracle's per-routine sequence (compute_tmask_limit,
  horz_advect_tracer_quicker, vert_advect_tracer_quicker, the explicit
  update, vert_diffuse_implicit; ocean_tracer.F90:2295-2350, 2432,
  2788-2892; ocean_tracer_advect.F90:2538-2653, 2981-3031), within 1e-12
  per cell (the FP64 column solver eliminates from both ends; MDFL-Sweby's
  limited fluxes are division-free);
* the plain per-tracer GPU path over two steps (which updates the tracer
  halos between steps with mom_gpu_update_domains), bit for bit.

Cases put tracer values outside their ranges so that the upwind fallbacks
run: a passive tracer above 1, salinity above 42 (flagging temperature
through tmask_limit_ts_same when temperature is the Quicker tracer).  The
halo update itself is checked against the oracle's single-PE update.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIM = {"temp": (-2.0, 32.0), "salt": (1.0, 42.0)}


def _case(kind):
    from mom5_amd.synth import make_case
    if kind == "cyclic":
        c = make_case(130, 70, 12, land_frac=0.3, nts=10, seed=61, n_passive=2, stf_scale=1e-3)
    else:
        c = make_case(41, 29, 9, land_frac=0.2, cyclic_x=False, lat_s=20.0, lat_n=50.0,
                      lon_span=30.0, nts=12, seed=62, n_passive=2, stf_scale=1e-3)
    rng = np.random.default_rng(7)
    tm = c.grid["tmask"]
    wet = np.argwhere(tm[:, 1:-1, 1:-1] > 0)
    for n, val in ((3, 1.5), (1, 42.5), (2, -0.5)):
        T = c.tracers[n][1]
        for k, j, i in wet[rng.choice(len(wet), 40, replace=False)]:
            T[k, j + 1, i + 1] = val
        if c.cyclic_x:
            T[..., 0] = T[..., -2]
            T[..., -1] = T[..., 1]
    return c


def _limits(names):
    return ([LIM.get(n, (-0.1, 1.0))[0] for n in names],
            [LIM.get(n, (-0.1, 1.0))[1] for n in names])


@pytest.mark.parametrize("kind", ["cyclic", "closed"])
@pytest.mark.parametrize("schemes,lwu", [
    (["mdfl_sweby", "mdfl_sweby", "quicker", "quicker"], False),
    (["mdfl_sweby", "mdfl_sweby", "quicker", "quicker"], True),
    (["quicker", "mdfl_sweby", "mdfl_sweby", "quicker"], False),
    (["quicker", "quicker", "quicker", "mdfl_sweby"], True)])
def test_quicker_batched_equals_oracle(oracle_lib, kind, schemes, lwu):
    from mom5_amd import DeviceArray, OceanGPU
    from _cases import assert_close_cells, oracle_tracer_step
    c = _case(kind)
    print(f"[quicker batched {kind} {schemes} limit_with_upwind={lwu}]", flush=True)
    names = [n for n, _ in c.tracers]
    mins, maxs = _limits(names)
    Ts = [np.asarray(t, np.float64) for _, t in c.tracers]
    f = c.fields
    gpu = OceanGPU(c.dom, c.grid)
    dev = {k: DeviceArray.from_host(v) for k, v in f.items() if isinstance(v, np.ndarray)}
    tin = [DeviceArray.from_host(t) for t in Ts]
    tout = [DeviceArray(t.shape, np.float64) for t in Ts]
    for a in tout:
        a.zero()
    gpu.step_tracers(tin, tout, uhrho_et=dev["uhrho_et"], vhrho_nt=dev["vhrho_nt"],
                     wrho_bt=dev["wrho_bt"], rho_dzt_tau=dev["rho_dzt"], dtime=c.dt,
                     stfs=[DeviceArray.from_host(x) for x in f["stf"][:4]],
                     btfs=[DeviceArray.from_host(x) for x in f["btf"][:4]], dzwt=dev["dzwt"],
                     diff_cbt=dev["diff_cbt"], index_salt=1, rho_dztr=dev["rho_dztr"],
                     schemes=schemes, min_limits=mins, max_limits=maxs, index_temp=0,
                     ts_same=True, limit_with_upwind=lwu)
    gpu.sync()
    got = [a.to_host() for a in tout]
    gpu.close()
    o = oracle_lib.Oracle(c)
    lims = o.tmask_limit(Ts, mins, maxs, index_temp=0, index_salt=1, ts_same=True)
    flagged = [int(l[:, 1:-1, 1:-1].sum()) for l in lims]
    assert all(x > 0 for x in flagged), flagged
    ref = oracle_tracer_step(o, Ts, f["stf"][:4], f["btf"][:4], c.dt, schemes=schemes,
                             mins=mins, maxs=maxs, index_temp=0, ts_same=True,
                             limit_with_upwind=lwu)
    for n in range(4):
        # the FP64 column solver's two-ended elimination (and MDFL-Sweby's
        # division-free limited fluxes): 1e-12 per cell
        assert_close_cells(got[n][:, 1:-1, 1:-1], ref[n][:, 1:-1, 1:-1],
                           what=f"tracer {n} ({schemes[n]})")


@pytest.mark.parametrize("kind", ["cyclic", "closed"])
def test_quicker_batched_equals_plain_over_steps(kind):
    from mom5_amd.step import BatchedStep, PlainStep
    c = _case(kind)
    print(f"[quicker batched vs plain, 2 steps, {kind}]", flush=True)
    schemes = ["mdfl_sweby", "mdfl_sweby", "quicker", "quicker"]
    plain = PlainStep(c, schemes=schemes)
    batched = BatchedStep(c, gpu=plain.gpu, schemes=schemes)
    plain.run(2)
    batched.run(2)
    plain.gpu.sync()
    for n in range(4):
        a = plain.tracer(n).to_host()[:, 1:-1, 1:-1]
        b = batched.tracer(n).to_host()[:, 1:-1, 1:-1]
        assert np.array_equal(a, b), (n, schemes[n])
    plain.gpu.close()


@pytest.mark.parametrize("cyclic", [True, False])
def test_update_domains_matches_single_pe_halo_update(oracle_lib, cyclic):
    import ctypes as C
    from mom5_amd import DeviceArray, OceanGPU
    from oracle.oracle import Dom
    from mom5_amd.synth import make_case
    kw = {} if cyclic else dict(cyclic_x=False, lat_s=20.0, lat_n=50.0, lon_span=30.0)
    c = make_case(37, 23, 5, seed=3, barotropic=False, **kw)
    rng = np.random.default_rng(1)
    a = rng.standard_normal((5, 25, 39))
    g = OceanGPU(c.dom, c.grid)
    d = DeviceArray.from_host(a)
    g.update_domains(d)
    g.sync()
    got = d.to_host()
    g.close()
    ref = a.copy()
    oracle_lib.lib().orc_halo_update(C.byref(Dom(**c.dom)), 1,
                                     ref.ctypes.data_as(C.POINTER(C.c_double)), 5, 3)
    assert np.array_equal(got, ref)
    assert cyclic == (not np.array_equal(ref, a))


# Pairs that share a pass: regions of 60 x 8 (two tracers) and 60 x 12 (one)
# cells exactly, one more and one less, two and three levels; flags OR'ed or
# not; other th_tendency terms on none, one or both of a pair.
@pytest.mark.parametrize("ni,nj,nk", [(60, 8, 2), (61, 9, 3), (59, 7, 4), (121, 25, 5)])
@pytest.mark.parametrize("schemes,ts_same,with_th", [
    (["quicker"] * 4, True, (0, 2, 3)), (["quicker"] * 4, False, ()),
    (["quicker", "mdfl_sweby", "quicker", "mdfl_sweby"], True, (0,)),
    (["mdfl_sweby", "quicker", "quicker", "quicker"], False, (1, 2))])
def test_quicker_pairs_equal_oracle(oracle_lib, ni, nj, nk, schemes, ts_same, with_th):
    from mom5_amd import DeviceArray, OceanGPU
    from mom5_amd.synth import make_case
    from _cases import assert_close_cells, oracle_tracer_step
    c = make_case(ni, nj, nk, land_frac=0.2, nts=10, seed=63, n_passive=2, stf_scale=1e-3)
    print(f"[quicker pairs {ni}x{nj}x{nk} {schemes} ts_same={ts_same} th={with_th}]", flush=True)
    rng = np.random.default_rng(9)
    tm = c.grid["tmask"]
    names = [n for n, _ in c.tracers]
    mins, maxs = _limits(names)
    Ts = [np.asarray(t, np.float64) for _, t in c.tracers]
    wet = np.argwhere(tm[:, 1:-1, 1:-1] > 0)
    for n in range(4):
        for k, j, i in wet[rng.choice(len(wet), 12, replace=False)]:
            Ts[n][k, j + 1, i + 1] = maxs[n] + 0.5
        Ts[n][..., 0], Ts[n][..., -1] = Ts[n][..., -2].copy(), Ts[n][..., 1].copy()
    ths = [1e-4 * rng.standard_normal(tm.shape) * tm if n in with_th else None for n in range(4)]
    f = c.fields
    gpu = OceanGPU(c.dom, c.grid)
    H = DeviceArray.from_host
    dev = {k: H(v) for k, v in f.items() if isinstance(v, np.ndarray)}
    tin, tout = [H(t) for t in Ts], [DeviceArray(t.shape, np.float64) for t in Ts]
    thd = [H(t) if t is not None else None for t in ths]
    for t in tout:
        t.zero()
    gpu.step_tracers(tin, tout, uhrho_et=dev["uhrho_et"], vhrho_nt=dev["vhrho_nt"],
                     wrho_bt=dev["wrho_bt"], rho_dzt_tau=dev["rho_dzt"],
                     rho_dztr=dev["rho_dztr"], dtime=c.dt, stfs=[H(s) for s in f["stf"]],
                     btfs=[H(b) for b in f["btf"]], dzwt=dev["dzwt"], diff_cbt=dev["diff_cbt"],
                     schemes=schemes, min_limits=mins, max_limits=maxs, ts_same=ts_same,
                     th_tendencies=thd)
    gpu.sync()
    want = oracle_tracer_step(oracle_lib.Oracle(c), Ts, f["stf"], f["btf"], c.dt, ths=ths,
                              schemes=schemes, mins=mins, maxs=maxs, ts_same=ts_same)
    for n in range(4):
        assert_close_cells(tout[n].to_host()[:, 1:-1, 1:-1], want[n][:, 1:-1, 1:-1],
                           what=f"{names[n]} ({schemes[n]})")
    gpu.close()
