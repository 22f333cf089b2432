"""GPU parity of the multigrid Poisson demag (demag_poisson_mg.rs) through the C ABI.

The FP64 path evaluates the reference's expressions in the reference's order,
so against the oracle it is held to 1e-12 (max |dB| / max |B|); with the
treecode or zero boundary it is bit-identical in practice.  The dipole
boundary sums its moments in a different order (1e-12 still holds).  FP32
contexts solve in FP64 from FP32 magnetisation: within 1e-5 of the oracle.
"""
import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu

OPS = {
    "rb7_inject_rd": dict(stencil=0, prolong=0, coarse_op=0, smoother=1),
    "iso27_tri_galerkin": dict(),
    "7pt_tri_rd_wj": dict(stencil=0, prolong=1, coarse_op=0),
    "iso9_inject_galerkin": dict(stencil=1, prolong=0, coarse_op=1),
}


def _rand_m(n, seed, holes=()):
    rng = np.random.default_rng(seed)
    v = rng.standard_normal((n, 3))
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    v[list(holes)] = 0.0
    return v


def _pair(L, O, **kw):
    return L.mg_config(**kw), O.mg_config(**kw)


@pytest.mark.parametrize("op", list(OPS))
@pytest.mark.parametrize("bc", [0, 1, 2])
def test_mg_fp64_matches_oracle_with_warm_start(gpu_lib, op, bc):
    from oracle import oracle as O
    L = gpu_lib
    nx, ny, cell = 20, 14, (4e-9, 4e-9, 3e-9)
    kw = dict(pad_xy=3, n_vac_z=3, tree_leaf=16, bc=bc, v_cycles_max=40, **OPS[op])
    lc, oc = _pair(L, O, **kw)
    ctx = L.Context(L.Grid2D(nx, ny, *cell), precision=L.F64)
    ctx.set_mg_config(lc)
    omg = O.MG(O.Grid(nx, ny, *cell), oc)
    mat = L.Material(ms=8e5, demag=True)
    for solve, (seed, holes) in enumerate([(1, (3, 40, 41)), (2, (3, 40, 41)), (3, (7, 8, 100))]):
        m = _rand_m(nx * ny, seed, holes)
        want = np.zeros_like(m)
        omg.add_field(m, want, 8e5)
        got = np.full_like(m, 0.125)
        ctx.add_demag_field_poisson_mg(m, got, mat)
        got -= 0.125
        st, ost = ctx.mg_last_stats(), omg.stats()
        assert st["cycles"] == ost["cycles"]
        assert st["n_charges"] == ost["n_charges"]
        assert rel_err(got, want) <= 1e-12, (solve, rel_err(got, want))
        if bc == 2:
            # the octree is reused while the charged cells stay the same
            assert st["tree_rebuilt"] == (solve != 1)


# Smoothers on the edges of their tiles, a few cycles without a tolerance, zero
# boundary: half-sweep launches with even and odd sweep counts, coarsest levels of
# nine and fewer planes and of several tiles, a flat box and one that does not
# coarsen in the plane; 640 x 600 marches in 64 x 32 boxes; 270000 rows are more
# than a launch grid's second dimension takes.  (The march's smaller boxes and its
# odd sweeps: below.)
@pytest.mark.parametrize("nx,ny,nvac,pre,post,cycles", [
    (7, 5, 3, 2, 2, 3), (26, 10, 4, 2, 1, 3), (27, 41, 8, 3, 2, 3), (50, 34, 16, 1, 4, 3), (75, 12, 16, 2, 3, 3),
    (131, 90, 5, 2, 2, 2), (640, 600, 2, 2, 2, 1), (1, 270000, 2, 2, 2, 1)])
@pytest.mark.parametrize("op", ["rb7_inject_rd", "iso27_tri_galerkin"])
def test_mg_smoother_tile_edges(gpu_lib, nx, ny, nvac, pre, post, cycles, op):
    from oracle import oracle as O
    L = gpu_lib
    cell = (4e-9, 3e-9, 2e-9)
    lc, oc = _pair(L, O, pad_xy=2, n_vac_z=nvac, bc=0, pre_smooth=pre, post_smooth=post, warm_start=0, tol_rel=None,
                   tol_abs=None, v_cycles=cycles, sor_omega=1.2, **OPS[op])
    m = _rand_m(nx * ny, nx + ny, (0, nx * ny // 2))
    want = np.zeros_like(m)
    O.MG(O.Grid(nx, ny, *cell), oc).add_field(m, want, 8e5)
    ctx = L.Context(L.Grid2D(nx, ny, *cell), precision=L.F64)
    ctx.set_mg_config(lc)
    got = ctx.compute_demag_field_poisson_mg(m, L.Material(ms=8e5, demag=True))
    assert rel_err(got, want) <= 1e-12


# Narrow boxes on the edges of the residual norm's row groups (interior widths 4 to
# 34) and planes of few and of odd cell counts, with a tolerance: fields, cycles
# and the last residual.
@pytest.mark.parametrize("nx,ny", [(1, 7), (3, 500), (5, 41), (11, 30), (13, 200), (27, 9), (29, 33), (31, 100)])
@pytest.mark.parametrize("op", list(OPS))
def test_mg_narrow_boxes(gpu_lib, nx, ny, op):
    from oracle import oracle as O
    L = gpu_lib
    cell = (4e-9, 3e-9, 2e-9)
    lc, oc = _pair(L, O, pad_xy=2, n_vac_z=3, bc=0, warm_start=0, tol_rel=1e-6, v_cycles=1, v_cycles_max=6, **OPS[op])
    m = _rand_m(nx * ny, nx + ny)
    want = np.zeros_like(m)
    omg = O.MG(O.Grid(nx, ny, *cell), oc)
    omg.add_field(m, want, 8e5)
    ctx = L.Context(L.Grid2D(nx, ny, *cell), precision=L.F64)
    ctx.set_mg_config(lc)
    got = ctx.compute_demag_field_poisson_mg(m, L.Material(ms=8e5, demag=True))
    assert rel_err(got, want) <= 1e-12
    st, ost = ctx.mg_last_stats(), omg.stats()
    assert st["cycles"] == ost["cycles"]
    assert abs(st["last_residual"] - ost["last_residual"]) <= 1e-12 * ost["rhs_max"]


# Both sides of the line between the two-sweep march and the half-sweep launches:
# wide shallow levels (290 x 202 x 8: tiles of 24 x 8 columns exactly filled, then
# with remainders) march, narrow deep ones (24 x 18 x 84) do not.
@pytest.mark.parametrize("nx,ny,nvac,pre,post,cycles", [
    (286, 198, 3, 2, 2, 2), (288, 196, 3, 4, 2, 2), (20, 14, 40, 2, 2, 3)])
def test_mg_march_or_half_sweeps(gpu_lib, nx, ny, nvac, pre, post, cycles):
    test_mg_smoother_tile_edges(gpu_lib, nx, ny, nvac, pre, post, cycles, "rb7_inject_rd")


# The finest level's odd sweep, marched on its own: tiles of 28 x 12 columns exactly
# filled and with remainders, and the large box's 60 x 28.
@pytest.mark.parametrize("nx,ny,nvac,pre,post,cycles", [
    (278, 202, 3, 1, 3, 2), (280, 200, 3, 1, 1, 2), (640, 600, 2, 1, 3, 1)])
def test_mg_odd_finest_sweep(gpu_lib, nx, ny, nvac, pre, post, cycles):
    test_mg_smoother_tile_edges(gpu_lib, nx, ny, nvac, pre, post, cycles, "rb7_inject_rd")


@pytest.mark.parametrize("op", ["rb7_inject_rd", "iso27_tri_galerkin"])
def test_mg_fp32_context_close_to_oracle(gpu_lib, op):
    from oracle import oracle as O
    L = gpu_lib
    nx, ny, cell = 24, 18, (3e-9, 3e-9, 2e-9)
    lc, oc = _pair(L, O, pad_xy=4, n_vac_z=4, tree_leaf=32, **OPS[op])
    m = _rand_m(nx * ny, 5, (0, 11))
    want = np.zeros_like(m)
    O.MG(O.Grid(nx, ny, *cell), oc).add_field(m, want, 6e5)
    ctx = L.Context(L.Grid2D(nx, ny, *cell), precision=L.F32)
    ctx.set_mg_config(lc)
    got = ctx.compute_demag_field_poisson_mg(m, L.Material(ms=6e5, demag=True))
    assert rel_err(got, want) <= 1e-5


def test_mg_hole_lattice_128_matches_oracle(gpu_lib):
    """A 128 x 128 film with a square lattice of holes (m = 0) in the
    configuration of the 512 x 512 workload (7-point, red-black SOR,
    injection, rediscretised coarse levels, treecode boundary, tol 1e-8)."""
    from oracle import oracle as O
    import initial_states as S
    L = gpu_lib
    nx = ny = 128
    cell = (3e-9, 3e-9, 3e-9)
    mask = S.hole_lattice_mask(nx, ny, cell[0], cell[1], pitch=96e-9, radius=24e-9)
    m = S.smoothed_random(nx, ny, seed=7).reshape(-1, 3)
    m[~mask.reshape(-1)] = 0.0
    kw = dict(OPS["rb7_inject_rd"], tol_rel=1e-8, v_cycles_max=200)
    lc, oc = _pair(L, O, **kw)
    want = np.zeros_like(m)
    omg = O.MG(O.Grid(nx, ny, *cell), oc)
    omg.add_field(m, want, 8.6e5)
    ctx = L.Context(L.Grid2D(nx, ny, *cell), precision=L.F64)
    ctx.set_mg_config(lc)
    got = ctx.compute_demag_field_poisson_mg(m, L.Material(ms=8.6e5, demag=True))
    st = ctx.mg_last_stats()
    assert st["cycles"] == omg.stats()["cycles"]
    assert st["last_residual"] <= st["tol_target"]
    assert rel_err(got, want) <= 1e-12
    assert (got[~mask.reshape(-1)] == 0).all()


def test_mg_512_hole_lattice_matches_oracle_cold_and_warm(gpu_lib):
    """The 512 x 512 hole-lattice workload at full size: cold and warm-started
    solves against the oracle (1e-12), convergence to tol_rel 1e-8, the padded
    box (524, 524, 36) in three levels, octree reuse on the warm solve, and the
    distance to the FFT demag of the same film (open-boundary MG with the
    7-point operator; the oracle records rel-RMSE 0.352 for this state)."""
    from oracle import oracle as O
    import initial_states as S
    L = gpu_lib
    nx = ny = 512
    cell = (3e-9, 3e-9, 3e-9)
    mask = S.hole_lattice_mask(nx, ny, cell[0], cell[1], pitch=96e-9, radius=24e-9)
    m = S.smoothed_random(nx, ny, seed=11).reshape(-1, 3)
    m[~mask.reshape(-1)] = 0.0
    kw = dict(OPS["rb7_inject_rd"], tol_rel=1e-8, v_cycles_max=300)
    lc, oc = _pair(L, O, **kw)
    omg = O.MG(O.Grid(nx, ny, *cell), oc)
    ctx = L.Context(L.Grid2D(nx, ny, *cell), precision=L.F64)
    ctx.set_mg_config(lc)
    mat = L.Material(ms=8.6e5, demag=True)
    for solve in range(2):
        want = np.zeros_like(m)
        omg.add_field(m, want, 8.6e5)
        got = ctx.compute_demag_field_poisson_mg(m, mat)
        st = ctx.mg_last_stats()
        assert st["box"] == (524, 524, 36) and st["levels"] == 3
        assert not st["diverged"] and st["last_residual"] <= st["tol_target"]
        assert st["cycles"] == omg.stats()["cycles"]
        assert st["tree_rebuilt"] == (solve == 0)
        assert rel_err(got, want) <= 1e-12, (solve, rel_err(got, want))
    fft = ctx.compute_demag_field(m, L.Material(ms=8.6e5, demag=True, demag_method=L.DemagMethod.FftUniform))
    mag = mask.reshape(-1)
    d = got[mag] - fft[mag]
    rel_rmse = np.sqrt((d ** 2).sum() / (fft[mag] ** 2).sum())
    assert 0.2 < rel_rmse < 0.5


def test_mg_dispatch_routes_and_pbc(gpu_lib, monkeypatch):
    """demag.rs:109-142: demag_method mg and dst route to the MG solver; the
    dispatcher reads LLG_DEMAG_MG_* at every call when no configuration is
    pinned; pbc > 0 falls back to the periodic FFT path."""
    L = gpu_lib
    nx, ny, cell = 16, 12, (4e-9, 4e-9, 3e-9)
    m = _rand_m(nx * ny, 9)
    for k in ("WARM_START", "PAD_XY", "NVAC_Z", "VCYCLES", "STENCIL", "PROLONG", "COARSE_OP",
              "SMOOTHER", "BC", "TOL_REL", "TOL_ABS"):
        monkeypatch.delenv("LLG_DEMAG_MG_" + k, raising=False)
    monkeypatch.delenv("LLG_DEMAG_METHOD", raising=False)
    monkeypatch.setenv("LLG_DEMAG_MG_WARM_START", "0")
    monkeypatch.setenv("LLG_DEMAG_MG_PAD_XY", "2")
    monkeypatch.setenv("LLG_DEMAG_MG_NVAC_Z", "2")
    monkeypatch.setenv("LLG_DEMAG_MG_VCYCLES", "2")
    direct = L.Context(L.Grid2D(nx, ny, *cell), precision=L.F64)
    want = direct.compute_demag_field_poisson_mg(m, L.Material(ms=8e5, demag=True))
    pinned = L.Context(L.Grid2D(nx, ny, *cell), precision=L.F64)
    pinned.set_mg_config(L.mg_config(warm_start=0, pad_xy=2, n_vac_z=2, v_cycles=2))
    np.testing.assert_array_equal(pinned.compute_demag_field_poisson_mg(m, L.Material(ms=8e5, demag=True)), want)
    for method in (L.DemagMethod.PoissonMG, L.DemagMethod.PoissonDst):
        ctx = L.Context(L.Grid2D(nx, ny, *cell), precision=L.F64)
        got = ctx.compute_demag_field(m, L.Material(ms=8e5, demag=True, demag_method=method))
        np.testing.assert_array_equal(got, want)
        b = ctx.build_h_eff(m, L.LLGParams(), L.Material(ms=8e5, demag=True, demag_method=method))
        np.testing.assert_array_equal(b, want)
        bp = np.zeros_like(m)
        ctx.add_demag_field_pbc(m, bp, L.Material(ms=8e5, demag=True, demag_method=method), 1, 0)
        bf = np.zeros_like(m)
        ctx.add_demag_field_pbc(m, bf, L.Material(ms=8e5, demag=True), 1, 0)
        np.testing.assert_array_equal(bp, bf)
    off = np.full_like(m, 0.5)
    direct.add_demag_field_poisson_mg(m, off, L.Material(ms=8e5, demag=False))
    assert (off == 0.5).all()


def test_mg_stats_and_config_errors(gpu_lib):
    L = gpu_lib
    ctx = L.Context(L.Grid2D(8, 8, 2e-9, 2e-9, 2e-9), precision=L.F64)
    with pytest.raises(L.LlgmiError):
        ctx.mg_last_stats()
    with pytest.raises(L.LlgmiError):
        ctx.set_mg_config(L.mg_config(bc=7))
    with pytest.raises(L.LlgmiError):
        ctx.set_mg_config(L.mg_config(tree_max_depth=65))
    # red-black SOR with a non-7-point operator is overridden to weighted Jacobi
    ctx.set_mg_config(L.mg_config(smoother=1, pad_xy=2, n_vac_z=2))
    m = _rand_m(64, 1)
    b = ctx.compute_demag_field_poisson_mg(m, L.Material(ms=8e5, demag=True))
    ctx.set_mg_config(L.mg_config(smoother=0, pad_xy=2, n_vac_z=2, warm_start=0))
    b2 = ctx.compute_demag_field_poisson_mg(m, L.Material(ms=8e5, demag=True))
    np.testing.assert_array_equal(b, b2)


@pytest.mark.parametrize("env", [{"LLGMI_MG_GRAPH": "0"}, {"LLGMI_MG_RB_FUSED": "0"},
                                 {"LLGMI_MG_GRAPH": "0", "LLGMI_MG_RB_FUSED": "0"}])
@pytest.mark.parametrize("op", ["rb7_inject_rd", "iso27_tri_galerkin"])
def test_mg_graph_replay_and_fused_sweeps_match_direct_launches(gpu_lib, monkeypatch, env, op):
    """The default solver replays each V-cycle from a captured HIP graph and
    runs a red-black sweep as one fused kernel; both must equal direct
    launches of the half-sweep kernels bit for bit, over several warm-started
    solves (each solve replays the graph many times, with host work between)."""
    L = gpu_lib
    nx, ny, cell = 40, 36, (3e-9, 3e-9, 3e-9)
    cfg = L.mg_config(pad_xy=4, n_vac_z=4, tol_rel=1e-9, v_cycles_max=100, **OPS[op])
    mat = L.Material(ms=8e5, demag=True)
    for k in ("LLGMI_MG_GRAPH", "LLGMI_MG_RB_FUSED"):
        monkeypatch.delenv(k, raising=False)
    fast = L.Context(L.Grid2D(nx, ny, *cell), precision=L.F64)
    fast.set_mg_config(cfg)
    ms = [_rand_m(nx * ny, s, (5, 6, 7 + s)) for s in range(3)]
    want = [fast.compute_demag_field_poisson_mg(m, mat) for m in ms]
    cycles = fast.mg_last_stats()["cycles"]
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    slow = L.Context(L.Grid2D(nx, ny, *cell), precision=L.F64)
    slow.set_mg_config(cfg)
    for m, w in zip(ms, want):
        np.testing.assert_array_equal(slow.compute_demag_field_poisson_mg(m, mat), w)
    assert slow.mg_last_stats()["cycles"] == cycles


def _xorshift_unit_vectors(n, seed):
    """init_random_unit_vectors of tests/test_demag_methods.rs:144-180."""
    import math
    mask = (1 << 64) - 1
    x = seed
    out = np.zeros((n, 3))
    for c in range(n):
        v = []
        for _ in range(3):
            x ^= (x << 13) & mask
            x ^= x >> 7
            x ^= (x << 17) & mask
            v.append(2.0 * (x / float(mask)) - 1.0)
        nrm = max(math.sqrt(v[0] ** 2 + v[1] ** 2 + v[2] ** 2), 1e-30)
        out[c] = [v[0] / nrm, v[1] / nrm, v[2] / nrm]
    return out


@pytest.mark.parametrize("case", ["unscreened_r2", "screened_r5", "holes_bscale", "galerkin_trilinear"])
def test_mg_hybrid_fp64_matches_oracle(gpu_lib, case):
    """Hybrid MG (demag_poisson_mg.rs:2512-2528, 3159-3597) against the oracle:
    the delta kernel from impulse responses, the screened solve and the local
    correction; the reference's 32 x 32 random case (tests/test_demag_methods.rs:197-267)."""
    from oracle import oracle as O
    L = gpu_lib
    print(f"hybrid {case}", flush=True)
    nx = ny = 32
    cell = (5e-9, 5e-9, 1e-9)
    m = _xorshift_unit_vectors(nx * ny, 12345)
    kw = dict(warm_start=0, pad_xy=2, n_vac_z=16, v_cycles=4)
    hyb = dict(enabled=1, radius_xy=2, delta_v_cycles=20, sigma_cells=0.0)
    if case == "screened_r5":
        hyb.update(radius_xy=5, sigma_cells=1.5)
    if case == "holes_bscale":
        mm = m.reshape(ny, nx, 3)
        mm[8:14, 10:16] = 0.0
        mm[20:25, 3:7] = 0.0
        hyb.update(radius_xy=3, sigma_cells=1.0, bscale=0.7, bmargin=2)
    if case == "galerkin_trilinear":
        kw.update(stencil=2, prolong=1, coarse_op=1, smoother=0)
        hyb.update(radius_xy=3, sigma_cells=1.2)
    oc = O.Context(O.Grid(nx, ny, *cell))
    oc.set_mg_config(O.mg_config(**kw))
    oc.set_hyb_config(O.hyb_config(**hyb))
    want = np.zeros_like(m)
    oc.add_demag(m, want, O.Material(ms=8e5, demag=True, demag_method=1))
    ctx = L.Context(L.Grid2D(nx, ny, *cell), precision=L.F64)
    ctx.set_mg_config(L.mg_config(**kw))
    ctx.set_mg_hybrid_config(L.mg_hybrid_config(**hyb))
    got = ctx.compute_demag_field_poisson_mg(m, L.Material(ms=8e5, demag=True))
    assert rel_err(got, want) <= 1e-12, rel_err(got, want)
    # a second call reuses the cached delta kernel
    again = ctx.compute_demag_field_poisson_mg(m, L.Material(ms=8e5, demag=True))
    assert rel_err(again, want) <= 1e-12
    if case in ("unscreened_r2", "screened_r5"):
        bf = ctx.compute_demag_field(m, L.Material(ms=8e5, demag=True))
        rel = np.sqrt(((got - bf) ** 2).sum() / (bf ** 2).sum())
        assert rel < 0.06, rel        # recorded "~0.32 -> ~0.04"


def test_mg_hybrid_env_and_fp32(gpu_lib, monkeypatch):
    """With no pinned hybrid configuration the context reads
    LLG_DEMAG_MG_HYBRID_* at every call; an FP32 context agrees to 1e-5."""
    L = gpu_lib
    nx, ny, cell = 24, 20, (4e-9, 4e-9, 2e-9)
    m = _rand_m(nx * ny, 31)
    kw = dict(warm_start=0, pad_xy=3, n_vac_z=4, v_cycles=3)
    pinned = L.Context(L.Grid2D(nx, ny, *cell), precision=L.F64)
    pinned.set_mg_config(L.mg_config(**kw))
    pinned.set_mg_hybrid_config(L.mg_hybrid_config(enabled=1, radius_xy=3, delta_v_cycles=10, sigma_cells=0.8))
    want = pinned.compute_demag_field_poisson_mg(m, L.Material(ms=8e5, demag=True))
    monkeypatch.setenv("LLG_DEMAG_MG_HYBRID_ENABLE", "on")
    monkeypatch.setenv("LLG_DEMAG_MG_HYBRID_RADIUS", "3")
    monkeypatch.setenv("LLG_DEMAG_MG_HYBRID_DELTA_VCYCLES", "10")
    monkeypatch.setenv("LLG_DEMAG_MG_HYBRID_SIGMA", "0.8")
    env = L.Context(L.Grid2D(nx, ny, *cell), precision=L.F64)
    env.set_mg_config(L.mg_config(**kw))
    np.testing.assert_array_equal(env.compute_demag_field_poisson_mg(m, L.Material(ms=8e5, demag=True)), want)
    monkeypatch.setenv("LLG_DEMAG_MG_HYBRID_ENABLE", "0")
    pure = env.compute_demag_field_poisson_mg(m, L.Material(ms=8e5, demag=True))
    assert rel_err(pure, want) > 1e-3
    monkeypatch.setenv("LLG_DEMAG_MG_HYBRID_ENABLE", "1")
    c32 = L.Context(L.Grid2D(nx, ny, *cell), precision=L.F32)
    c32.set_mg_config(L.mg_config(**kw))
    assert rel_err(c32.compute_demag_field_poisson_mg(m, L.Material(ms=8e5, demag=True)), want) <= 1e-5


def test_mg_hybrid_stencil_cache_file(gpu_lib, monkeypatch, tmp_path):
    """LLG_DEMAG_MG_HYBRID_CACHE=1 writes the correction stencil to the
    reference's LLGDKH8 file (demag_poisson_mg.rs:2811-3052) under
    out/demag_cache, named by DeltaKernelKey::cache_path (:2335-2374) from the
    key the file holds; a new context reads it back (bitwise the same field),
    uses what the file holds (a doubled stencil changes the field), and treats
    a truncated file as a miss (rebuilt and rewritten)."""
    import struct
    L = gpu_lib
    monkeypatch.chdir(tmp_path)
    monkeypatch.setenv("LLG_DEMAG_MG_HYBRID_CACHE", "1")
    nx, ny, cell = 24, 20, (4e-9, 4e-9, 2e-9)
    m = _rand_m(nx * ny, 31)
    mat = L.Material(ms=8e5, demag=True)

    def field():
        c = L.Context(L.Grid2D(nx, ny, *cell), precision=L.F64)
        c.set_mg_config(L.mg_config(warm_start=0, pad_xy=3, n_vac_z=4, v_cycles=3))
        c.set_mg_hybrid_config(L.mg_hybrid_config(enabled=1, radius_xy=3, delta_v_cycles=10, sigma_cells=0.8))
        return c.compute_demag_field_poisson_mg(m, mat)

    b0 = field()
    files = sorted((tmp_path / "out" / "demag_cache").glob("*"))
    assert len(files) == 1, files
    path = files[0]
    raw = path.read_bytes()
    n = 7 * 7
    assert raw[:8] == b"LLGDKH8\x00" and len(raw) == 8 + 23 * 8 + 7 * n * 8
    u = struct.unpack("<23Q", raw[8:8 + 23 * 8])
    f64 = lambda b: struct.unpack("<d", struct.pack("<Q", b))[0]
    assert u[0:2] == (nx, ny) and [f64(x) for x in u[2:5]] == list(cell)
    assert u[5:7] == (3, 4) and u[21:23] == (3, 10) and f64(u[20]) == 0.8

    def rexp(v):
        mant, e = f"{v:.3e}".split("e")
        return f"{mant}e{int(e)}"
    st = {0: "7", 1: "iso9"}.get(u[7], "iso27" if u[10] == 0 else f"iso27a{u[10]:016x}")
    op = f"{st}_{'inj' if u[8] == 0 else 'tri'}_{'rd' if u[9] == 0 else 'gal'}"
    name = (f"demag_mg_hybrid_dk_nx{u[0]}_ny{u[1]}_dx{rexp(f64(u[2]))}_dy{rexp(f64(u[3]))}_dz{rexp(f64(u[4]))}"
            f"_pad{u[5]}_nvacz{u[6]}_op{op}_bc{['dir0', 'dip', 'bh'][u[11]]}_th{rexp(f64(u[12]))}_leaf{u[13]}"
            f"_dep{u[14]}_sm{['wj', 'rb'][u[17]]}_pre{u[15]}_post{u[16]}_om{u[18]:016x}_som{u[19]:016x}"
            f"_sig{u[20]:016x}_r{u[21]}_dv{u[22]}.bin")
    assert path.name == name
    dk = np.frombuffer(raw[192:192 + 4 * n * 8], dtype="<f8").reshape(4, n)
    assert np.all(np.frombuffer(raw[192 + 4 * n * 8:], dtype="<f8") == 0.0)   # PPPM-phi stencils: none
    for c in (0, 2, 3):   # the uniform-bias fix leaves the diagonal stencils summing to zero
        assert abs(dk[c].sum()) <= 1e-12 * np.abs(dk[c]).max()

    np.testing.assert_array_equal(field(), b0)          # read back
    path.write_bytes(raw[:192] + (2.0 * dk).astype("<f8").tobytes() + raw[192 + 4 * n * 8:])
    assert np.abs(field() - b0).max() > 1e-6 * np.abs(b0).max()   # the file's stencil is the one used
    path.write_bytes(raw[:200])                          # truncated: a miss, rebuilt and rewritten
    np.testing.assert_array_equal(field(), b0)
    assert path.read_bytes() == raw

