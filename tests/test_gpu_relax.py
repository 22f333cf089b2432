"""Relaxation path on the GPU against the oracle, through the C ABI:
energy breakdown (energy.rs:80-283), the relax-mode RK23 step
(llg.rs:278-436) with FSAL and its cached field, and the relax controller
(relax.rs:334-774).

FP64 bar: energies within 1e-12 of the oracle (relative to the largest term),
RK23 states within 1e-12, eps and the next dt within 1e-9 relative; the relax
controller takes the same decisions (identical report counts) and ends in the
same state (1e-12 for a macrospin; 1e-7 for films, whose end state carries a
stability-limit mode, see test_relax_fp64_matches_oracle).  FP32: energies
within 1e-5 of FP64, relax converges to the same state.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def unit(v):
    v = np.asarray(v, dtype=np.float64)
    return v / np.linalg.norm(v, axis=-1, keepdims=True)


def rand_m(n, seed):
    return unit(np.random.default_rng(seed).standard_normal((n, 3)))


def mats(L, dmi=1.5e-3, demag=True, ku=3e5):
    kw = dict(ms=8e5, a_ex=1.3e-11, k_u=ku, easy_axis=(0.0, 0.0, 1.0), dmi=dmi, demag=demag)
    return L.Material(**kw), O.Material(**kw)


CASES = [(16, 8), (33, 17), (1, 1), (64, 1), (128, 64)]


@pytest.mark.parametrize("shape", CASES)
@pytest.mark.parametrize("geom_kind", ["none", "holes"])
def test_energy_fp64_matches_oracle(gpu_lib, shape, geom_kind):
    L = gpu_lib
    nx, ny = shape
    print(f"energy {shape} geom={geom_kind}", flush=True)
    g = (nx, ny, 4e-9, 4e-9, 3e-9)
    m = rand_m(nx * ny, nx * 7 + ny)
    geom = None
    if geom_kind == "holes":
        geom = np.ones((ny, nx), dtype=bool)
        geom[::3, ::4] = False
        geom = geom.reshape(-1)
    bx = (0.01, -0.02, 0.03)
    lm, om = mats(L)
    ctx = L.Context(L.Grid2D(*g), precision=L.F64)
    e = ctx.compute_energy_geom(m, lm, bx, geom)
    eo = O.compute_energy(O.Context(O.Grid(*g)), m, om, bx, geom=geom)
    scale = max(abs(v) for v in eo.values())
    for k in eo:
        assert abs(e[k] - eo[k]) <= 1e-12 * scale, (k, e[k], eo[k])


def test_energy_fp32_against_fp64(gpu_lib):
    L = gpu_lib
    g = L.Grid2D(256, 128, 2e-9, 2e-9, 1e-9)
    m = unit(np.tile([0.1, 0.2, 1.0], (g.n_cells(), 1)) + 0.3 * rand_m(g.n_cells(), 3))
    lm, _ = mats(L)
    e64 = L.Context(g, precision=L.F64).compute_energy(m, lm, (0.01, 0.0, 0.02))
    e32 = L.Context(g, precision=L.F32).compute_energy(m, lm, (0.01, 0.0, 0.02))
    scale = max(abs(v) for v in e64.values())
    for k in e64:
        assert abs(e32[k] - e64[k]) <= 1e-5 * scale, (k, e32[k], e64[k])


def test_rk23_steps_fp64_match_oracle(gpu_lib):
    L = gpu_lib
    g = (24, 16, 4e-9, 4e-9, 3e-9)
    lm, om = mats(L)
    m0 = rand_m(24 * 16, 21)
    ctx = L.Context(L.Grid2D(*g), precision=L.F64)
    oc, ork = O.Context(O.Grid(*g)), O.RK23(O.Grid(*g))
    mg, mo = m0.copy(), m0.copy()
    pg = L.LLGParams(alpha=0.3, dt=2e-14, b_ext=(0.01, 0.0, 0.02))
    po = O.Params(alpha=0.3, dt=2e-14, b_ext=(0.01, 0.0, 0.02))
    n_acc = n_rej = 0
    for step in range(12):
        if step == 6:
            pg.b_ext = po.b_ext = (0.0, 0.0, 0.0)        # FSAL must drop here
        rg = ctx.step_llg_rk23_recompute_field_masked_relax_adaptive(mg, pg, lm, L.FieldMask.Full,
                                                                     1e-4, 0.8, 1e-18, 1e-11)
        ro = ork.step(oc, mo, po, om, O.FULL, 1e-4, 0.8, 1e-18, 1e-11)
        assert rg[1] == ro[1] and abs(rg[2] - ro[2]) <= 1e-9 * ro[2]
        assert abs(rg[0] - ro[0]) <= 1e-9 * ro[0]
        assert abs(pg.dt - po.dt) <= 1e-9 * po.dt
        assert np.abs(mg - mo).max() <= 1e-12
        n_acc += ro[1]
        n_rej += not ro[1]
        bg, bo = ctx.rk23_last_b_eff(), ork.last_b_eff()
        assert (bg is None) == (bo is None)
        if bo is not None:
            assert np.abs(bg - bo).max() <= 1e-12 * np.abs(bo).max()
    assert n_acc >= 6
    ctx.rk23_invalidate_last_b_eff()
    assert ctx.rk23_last_b_eff() is None


def test_rk23_reject_keeps_state(gpu_lib):
    L = gpu_lib
    g = L.Grid2D(16, 16, 4e-9, 4e-9, 3e-9)
    lm, _ = mats(L, demag=False)
    m0 = rand_m(256, 5)
    m = m0.copy()
    p = L.LLGParams(alpha=0.3, dt=1e-12)
    eps, acc, dtu = L.Context(g, precision=L.F64).step_llg_rk23_recompute_field_masked_relax_adaptive(
        m, p, lm, L.FieldMask.ExchAnisDmi, 1e-12, 0.8, 1e-18, 1e-11)
    assert not acc and np.array_equal(m, m0) and p.dt < 1e-12


def near_z(n, seed, amp=0.4):
    return unit(np.tile([0.0, 0.0, 1.0], (n, 1)) + amp * rand_m(n, seed))


def relax_both(L, g, m0, lmat, omat, mask_l, mask_o, prec, **kw):
    ctx = L.Context(L.Grid2D(*g), precision=prec)
    mg = m0.copy()
    pg = L.LLGParams(alpha=0.5, dt=1e-13)
    sg = L.relax_settings(**kw)
    rg = ctx.relax_with_report(mg, pg, lmat, mask_l, sg)
    oc, ork = O.Context(O.Grid(*g)), O.RK23(O.Grid(*g))
    mo = m0.copy()
    po = O.Params(alpha=0.5, dt=1e-13)
    so = O.relax_settings(**kw)
    ro = O.relax_with_report(oc, ork, mo, po, omat, mask_o, so)
    return rg, mg, pg, sg, ro, mo, po, so


@pytest.mark.parametrize("case", ["macrospin", "film_demag", "film_mumax", "film_gate"])
def test_relax_fp64_matches_oracle(gpu_lib, case):
    L = gpu_lib
    print(f"relax {case}", flush=True)
    if case == "macrospin":
        g = (1, 1, 5e-9, 5e-9, 5e-9)
        kw = dict(ms=8e5, k_u=5e5, easy_axis=(0.0, 0.0, 1.0))
        lm, om = L.Material(**kw), O.Material(**kw)
        m0 = unit(np.array([[0.4, 0.1, 0.8]]))
        args = dict()
        masks = (L.FieldMask.ExchAnis, O.EXCH_ANIS)
    else:
        g = (16, 8, 4e-9, 4e-9, 3e-9)
        lm, om = mats(L, ku=6e5)
        m0 = near_z(128, 8)
        masks = (L.FieldMask.Full, O.FULL)
        # max_err 1e-6: at the default 1e-5 an explicit step on this exchange
        # stiffness stalls near 2e-4 T of torque, above the 1e-4 threshold
        args = dict(max_err=1e-6, max_accepted_steps=4000)
        if case == "film_mumax":
            args = dict(max_err=1e-6, max_accepted_steps=4000, torque_metric=L.TORQUE_MEANSQ,
                        torque_threshold=None, torque_plateau_checks=1, torque_plateau_min_checks=1,
                        torque_plateau_rel=0.0, rel_energy_tol=0.0)
        if case == "film_gate":
            args = dict(max_err=1e-6, max_accepted_steps=4000, final_torque_gate=1e-300,
                        gate_max_extra_accepted_steps=5, torque_metric=L.TORQUE_RMS)
    rg, mg, pg, sg, ro, mo, po, so = relax_both(L, g, m0, lm, om, masks[0], masks[1], L.F64, **args)
    for k in ("stop_reason", "last_stage_stop"):
        assert rg[k] == ro[k], (k, rg, ro)
    assert rg["final_max_err"] == ro["final_max_err"] and sg.max_err == so.max_err
    assert ro["accepted_steps"] > 0
    if case == "film_mumax":
        # MuMax's plateau stops where the float32 sum of |m x B|^2 stops falling,
        # i.e. at the rounding-noise floor of the field: the step where that
        # happens depends on rounding, so only the outcome is compared.
        assert abs(rg["accepted_steps"] - ro["accepted_steps"]) <= 0.2 * ro["accepted_steps"]
        assert np.abs(mg - mo).max() <= 1e-7
        assert abs(rg["final_torque_max"] - ro["final_torque_max"]) <= 1e-6
        return
    for k in ("accepted_steps", "rejected_steps", "torque_checks", "torque_field_rebuilds"):
        assert rg[k] == ro[k], (k, rg, ro)
    # the last step size comes from an error estimate near max_err = 1e-9, a
    # difference of nearly equal states: its rounding shows at ~1e-6 relative
    assert abs(rg["final_dt"] - ro["final_dt"]) <= 1e-3 * ro["final_dt"]
    # The films end where an explicit step sits at its stability limit on the
    # exchange stiffness (dt ~ 2 ps): the residual high-frequency mode (torque
    # ~2e-5 T of O(1 T) fields) carries the rounding of the whole run, so the
    # end states agree to ~2e-8 (measured) and the torques to ~1e-7 T, while
    # every accept / reject / stop decision above is identical.  The
    # macrospin has no such mode and is held to 1e-12.
    tol_m, tol_t = (1e-12, 1e-12) if case == "macrospin" else (1e-7, 1e-6)
    for k in ("final_torque", "final_torque_max"):
        assert (rg[k] is None) == (ro[k] is None)
        if ro[k] is not None:
            assert abs(rg[k] - ro[k]) <= tol_t, (k, rg[k], ro[k])
    assert np.abs(mg - mo).max() <= tol_m


def test_relax_fp32_converges(gpu_lib):
    L = gpu_lib
    g = (64, 32, 4e-9, 4e-9, 3e-9)
    lm, om = mats(L, ku=6e5)
    m0 = near_z(64 * 32, 12)
    ctx = L.Context(L.Grid2D(*g), precision=L.F32)
    m = m0.copy()
    p = L.LLGParams(alpha=0.5, dt=1e-13)
    s = L.relax_settings(max_err=1e-6, max_accepted_steps=20000)
    rep = ctx.relax_with_report(m, p, lm, L.FieldMask.Full, s)
    assert rep["stop_reason"] == L.STOP_TIGHTEN_FLOOR_REACHED, rep
    assert rep["final_torque"] <= 1e-4
    c64 = L.Context(L.Grid2D(*g), precision=L.F64)
    m64 = m0.copy()
    p64 = L.LLGParams(alpha=0.5, dt=1e-13)
    rep64 = c64.relax_with_report(m64, p64, lm, L.FieldMask.Full,
                                  L.relax_settings(max_err=1e-6, max_accepted_steps=20000))
    assert rep64["stop_reason"] == L.STOP_TIGHTEN_FLOOR_REACHED
    assert np.abs(m - m64).max() < 1e-3


def test_dev_relax_matches_host(gpu_lib):
    from conftest import DeviceBuffer
    L = gpu_lib
    g = L.Grid2D(16, 8, 4e-9, 4e-9, 3e-9)
    lm, _ = mats(L, ku=6e5)
    m0 = near_z(128, 8)
    ctx = L.Context(g, precision=L.F64)
    mh = m0.copy()
    ph = L.LLGParams(alpha=0.5, dt=1e-13)
    rh = ctx.relax_with_report(mh, ph, lm, L.FieldMask.Full,
                               L.relax_settings(max_err=1e-6, max_accepted_steps=3000))
    md = DeviceBuffer(3 * 128 * 8)
    ctx.dev_upload(m0, md)
    pd = L.LLGParams(alpha=0.5, dt=1e-13)
    rd = ctx.dev_relax_with_report(md, pd, lm, L.FieldMask.Full,
                                   L.relax_settings(max_err=1e-6, max_accepted_steps=3000))
    assert rd == rh
    assert np.array_equal(ctx.dev_download(md), mh)
    e_dev = ctx.dev_compute_energy_geom(md, lm, (0, 0, 0))
    e_host = ctx.compute_energy(mh, lm, (0, 0, 0))
    assert e_dev == e_host


def test_relax_argument_errors(gpu_lib):
    L = gpu_lib
    ctx = L.Context(L.Grid2D(8, 8, 4e-9, 4e-9, 3e-9), precision=L.F64)
    lm, _ = mats(L)
    m = near_z(64, 1)
    with pytest.raises(L.LlgmiError):
        ctx.relax_with_report(m, L.LLGParams(), lm, L.FieldMask.Full, L.relax_settings(torque_metric=9))
    with pytest.raises(L.LlgmiError):
        ctx.relax_with_report(m, L.LLGParams(), lm, L.FieldMask.Full,
                              L.relax_settings(dt_min=1e-10, dt_max=1e-12))


@pytest.mark.parametrize("prec,path", [("f32", "fft_fused"), ("f32", "fft_unfused"), ("f64", "fft_fused"),
                                       ("f64", "no_demag"), ("f64", "mg")])
def test_rk23_stage_epilogue_equals_stage_kernels(gpu_lib, prec, path, monkeypatch):
    """Stage states 3 and 4 formed in the field evaluation's epilogue (the
    default) against stage kernels of their own (LLGMI_RK45_FUSE=0): state, eps,
    accept, dt and the kept field bitwise equal over 8 attempts, one rejected."""
    from conftest import DeviceBuffer
    from initial_states import smoothed_random
    L = gpu_lib
    P, es = (L.F32, 4) if prec == "f32" else (L.F64, 8)
    nx, ny = 45, 21
    mat = L.Material(ms=8e5, a_ex=1.3e-11, k_u=2e4, dmi=1e-3, demag=path != "no_demag")
    if path == "mg":
        mat.demag_method = L.DemagMethod.PoissonMG
    mask = 1 if path == "no_demag" else 2
    monkeypatch.setenv("LLGMI_FFT_FUSED", "1" if path == "fft_fused" else "0")
    ctxs = [L.Context(L.Grid2D(nx, ny, 3e-9, 3e-9, 2e-9), precision=P) for _ in range(2)]
    bufs = [DeviceBuffer(3 * nx * ny * es) for _ in range(2)]
    pars = [L.LLGParams(alpha=0.3, dt=1e-13, b_ext=(0.0, 0.01, 0.02)) for _ in range(2)]
    for c, b in zip(ctxs, bufs):
        c.dev_upload(smoothed_random(nx, ny, 5).reshape(-1, 3), b)
    rejected = 0
    for step in range(8):
        if step == 4:
            pars[0].dt = pars[1].dt = 5e-11
        res = []
        for i in range(2):
            if i == 0:
                monkeypatch.delenv("LLGMI_RK45_FUSE", raising=False)
            else:
                monkeypatch.setenv("LLGMI_RK45_FUSE", "0")
            res.append(ctxs[i].dev_rk23_relax_step(bufs[i], pars[i], mat, mask, 1e-5, 0.8, 1e-18, 1e-9))
        assert res[0] == res[1] and pars[0].dt == pars[1].dt, step
        assert np.array_equal(ctxs[0].dev_download(bufs[0]), ctxs[1].dev_download(bufs[1])), step
        rejected += not res[0][1]
    assert rejected >= 1
    fields = [c.rk23_last_b_eff() for c in ctxs]
    assert (fields[0] is None) == (fields[1] is None)
    if fields[0] is not None:
        assert np.array_equal(fields[0], fields[1])
