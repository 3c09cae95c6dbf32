"""Launch tuning and ensembles: the autotuner's block shapes, the vertical segments of the
column-marching kernels, the column solvers and the graph-captured ensemble step must not change any result
(every member stays bitwise equal to its own oracle run)."""
import dataclasses

import numpy as np
import pytest

from golden_util import max_rel
from lgame.cases import dry3d_config, make_case, tiny_config
from lgame.config import PREC_FP64, PREC_MIXED
from lgame.gpu import TILE_KERNELS, Ensemble, LgameError, Step, grid_setup_device
from lgame.metrics import field_errors, worst
from pyoracle import CpuOracle

pytestmark = pytest.mark.gpu


def _oracle(cfg, g, st, n):
    o = CpuOracle(cfg, g)
    o.start(st)
    o.run(0, n)
    return o.get_state(n % 2)


def test_autotune_keeps_results():
    cfg = tiny_config(ny=9, nx=11, n_layers=7, moist=True, order=3, freeslip=True)
    g, st = make_case(cfg, cloud_frac=0.2)
    s = Step(cfg, g)
    s.start(st)
    rows = s.autotune(2)
    print(f"tiles {rows}")
    assert set(rows) == set(TILE_KERNELS) and all(r in (1, 2, 4) for r in rows.values())
    s.run(0, 5)
    got = s.get_state(1)
    s.close()
    want = _oracle(cfg, g, st, 5)
    assert all(np.array_equal(got[k], want[k]) for k in want)


def test_scalar_kernel_segments_and_rows_keep_results():
    """The scalar divergence marches down 62-cell row tiles: a domain of 3 tiles (the last one
    partial) with an odd row count, cut into 1, 2 and 4 vertical segments on 1, 2 and 4 rows per
    block, every combination bitwise equal to the oracle over 4 steps (moist, 3rd-order theta,
    free slip, terrain-following layers from level 5, where the 4-segment cut starts its second
    segment)."""
    cfg = dataclasses.replace(tiny_config(ny=7, nx=150, n_layers=16, moist=True, order=3, freeslip=True), n_oro_layers=12)
    g, st = make_case(cfg, cloud_frac=0.3)
    n = 4
    want = _oracle(cfg, g, st, n)
    for rows in (1, 2, 4):
        for seg in (1, 2, 4):
            s = Step(cfg, g)
            s.set_tiles({k: rows for k in TILE_KERNELS})
            s.segments = seg
            assert s.segments == seg
            s.start(st)
            s.run(0, n)
            got = s.get_state(n % 2)
            s.close()
            print(f"rows {rows}, segments {seg}", flush=True)
            assert all(np.array_equal(got[k], want[k]) for k in want), (rows, seg)
    s = Step(cfg, g)
    for bad in (3, 8):  # not a power of two; fewer than 4 levels per segment
        with pytest.raises(LgameError, match="segment"):
            s.segments = bad
    s.close()


def test_autotune_times_all_kernels_that_the_segments_cut():
    """161x129x47 with third-order theta in FP64: the scalar kernel alone is fastest with 2 segments (82 us,
    89 with 4), together with the theta kernel it is not (205 us, 191 with 4 and 196 with 8)."""
    cfg = dataclasses.replace(dry3d_config(n=129, n_layers=47), ny=161, theta_adv_order=3)
    g, st = make_case(cfg, grid=grid_setup_device(cfg))
    s = Step(cfg, g)
    s.start(st)
    s.autotune(16)
    print(f"segments {s.segments}", flush=True)
    assert s.segments in (4, 8)
    s.close()


VER_CASES = {
    "dry_o2": (tiny_config(ny=6, nx=70, n_layers=9), 4, 0.0),
    "moist_o3_freeslip": (tiny_config(ny=9, nx=11, n_layers=7, moist=True, order=3, freeslip=True), 5, 0.3),
    "three_layers": (tiny_config(ny=3, nx=4, n_layers=3, moist=True), 4, 0.2),
    "diff_pbl_soil_sens": (dataclasses.replace(tiny_config(moist=True, order=3).set_diffusion(True), lpbl=True,
                                               lprog_soil_temp=True, lsfc_sensible_heat_flux=True), 6, 0.3),
}


@pytest.mark.parametrize("name", list(VER_CASES))
def test_vertical_solver_passes_keep_results(name):
    """The setting of the vertical solver's passes, which columns of up to 72 layers keep and do not
    use: bitwise equal to the oracle with either; small domains default to three passes."""
    cfg, n, cf = VER_CASES[name]
    g, st = make_case(cfg, cloud_frac=cf)
    want = _oracle(cfg, g, st, n)
    for passes in (1, 3):
        s = Step(cfg, g)
        assert s.column_passes == 3  # fewer column wavefronts than SIMDs
        s.column_passes = passes
        assert s.column_passes == passes
        s.start(st)
        s.run(0, n)
        got = s.get_state(n % 2)
        s.close()
        print(f"{name}: passes {passes}", flush=True)
        assert all(np.array_equal(got[k], want[k]) for k in want), (name, passes)
    s = Step(cfg, g)
    with pytest.raises(LgameError, match="passes"):
        s.column_passes = 2
    s.close()


TALL_CASES = {
    "dry_o2": (tiny_config(ny=6, nx=70, n_layers=73), 4, 0.0),
    "dry_o3_freeslip_diff": (tiny_config(ny=5, nx=33, n_layers=80, order=3, freeslip=True).set_diffusion(True), 4, 0.0),
    # five column wavefronts (an odd one for the tracer solver's pairs), and two to a row
    "moist_o3_freeslip": (tiny_config(ny=5, nx=11, n_layers=74, moist=True, order=3, freeslip=True), 5, 0.3),
    "moist_two_wavefronts": (tiny_config(ny=3, nx=65, n_layers=73, moist=True), 4, 0.3),
    "diff_pbl_soil_sens": (dataclasses.replace(tiny_config(ny=5, nx=9, n_layers=79, moist=True, order=3).set_diffusion(True),
                                               lpbl=True, lprog_soil_temp=True, lsfc_sensible_heat_flux=True), 6, 0.3),
}


@pytest.mark.parametrize("precision", [PREC_FP64, PREC_MIXED])
@pytest.mark.parametrize("name", list(TALL_CASES))
def test_tall_column_solvers_match_oracle(name, precision):
    """Columns of more than 72 layers, which the solvers in registers do not take: the vertical solver in
    one pass per column and in three (rows, Thomas recursion, new state), the tracer solver through the
    column scratch.  Both passes give the same bits.  Against the oracle the dry FP64 form is bitwise,
    the others agree to rounding (the device's exp, log and pow); the mixed form has its own bar."""
    cfg, n, cf = TALL_CASES[name]
    g, st = make_case(cfg, cloud_frac=cf)
    want = _oracle(cfg, g, st, n)
    got = {}
    for passes in (1, 3):
        s = Step(dataclasses.replace(cfg, precision=precision), g)
        s.column_passes = passes
        s.start(st)
        s.run(0, n)
        got[passes] = s.get_state(n % 2)
        s.close()
        print(f"{name}: passes {passes}", flush=True)
    assert all(np.array_equal(got[1][k], got[3][k]) for k in want)
    if precision == PREC_MIXED:
        err = field_errors(got[1], want)
        assert worst(err, "rms_rel") < 1e-4 and worst(err, "max_rel") < 1e-4
    elif cfg.lmoist:
        assert max_rel(got[1], want) <= 1e-12
    else:
        assert all(np.array_equal(got[1][k], want[k]) for k in want)


def test_autotune_of_tall_columns_keeps_results():
    """The autotuner also times the vertical solver's passes where columns use them."""
    cfg, n, _ = TALL_CASES["dry_o2"]
    g, st = make_case(cfg)
    s = Step(cfg, g)
    s.start(st)
    s.autotune(2)
    assert s.column_passes in (1, 3)
    s.run(0, n)
    got = s.get_state(n % 2)
    s.close()
    want = _oracle(cfg, g, st, n)
    assert all(np.array_equal(got[k], want[k]) for k in want)


@pytest.mark.parametrize("nl,nx,moist", [(3, 4, False), (7, 31, False), (8, 32, True), (9, 33, False), (40, 65, False), (41, 5, True),
                                         (64, 34, False), (65, 7, False), (72, 33, True), (73, 33, False)])
def test_vertical_solver_segments_match_oracle(nl, nx, moist):
    """The vertical solver cuts columns of up to 72 layers into 8 segments (empty ones below 8 layers)
    in blocks of 32 columns: the edges of its layer ranges and of its blocks, bitwise against the
    oracle."""
    cfg = tiny_config(ny=4, nx=nx, n_layers=nl, moist=moist, freeslip=nl % 2 == 1)
    g, st = make_case(cfg, cloud_frac=0.2 if moist else 0.0)
    want = _oracle(cfg, g, st, 3)
    s = Step(cfg, g)
    s.start(st)
    s.run(0, 3)
    got = s.get_state(1)
    s.close()
    assert all(np.array_equal(got[k], want[k]) for k in want)


@pytest.mark.parametrize("layers", [(6, 44, 70), (6, 20, 73)])
def test_batched_vertical_solver_with_members_of_different_height(layers):
    cfgs = [tiny_config(ny=4 + i, nx=30 + 3 * i, n_layers=nl) for i, nl in enumerate(layers)]
    cases = [make_case(c) for c in cfgs]
    steps = []
    for c, (g, st) in zip(cfgs, cases):
        s = Step(c, g)
        s.start(st)
        steps.append(s)
    e = Ensemble(steps)
    e.run(0, 3, mode=Ensemble.BATCHED)
    e.sync()
    for c, (g, st), s in zip(cfgs, cases, steps):
        got, want = s.get_state(1), _oracle(c, g, st, 3)
        assert all(np.array_equal(got[k], want[k]) for k in want), c.n_layers
    e.close()
    for s in steps:
        s.close()


DIFF_SWITCHES = {"all": {}, "temperature": dict(lmass_diff_h=False, lmass_diff_v=False),
                 "densities": dict(ltemp_diff_h=False, ltemp_diff_v=False), "horizontal": dict(ltemp_diff_v=False, lmass_diff_v=False)}


@pytest.mark.parametrize("switches", list(DIFF_SWITCHES))
@pytest.mark.parametrize("nx,nl,oro,moist,rows,seg", [(61, 16, 12, True, 1, 4), (62, 9, 8, False, 2, 2), (63, 6, 4, True, 4, 1),
                                                      (125, 5, 1, False, 4, 1)])
def test_diffusion_columns_match_oracle(nx, nl, oro, moist, rows, seg, switches):
    """The scalar diffusion marches down 62-cell row tiles, cut into vertical segments: one partial
    tile, full ones and a third, with flat and terrain-following layers, every set
    of switches, bitwise against the oracle."""
    cfg = dataclasses.replace(tiny_config(ny=5, nx=nx, n_layers=nl, moist=moist).set_diffusion(), n_oro_layers=oro,
                              **DIFF_SWITCHES[switches])
    g, st = make_case(cfg, cloud_frac=0.3 if moist else 0.0)
    want = _oracle(cfg, g, st, 3)
    s = Step(cfg, g)
    s.set_tiles({k: rows for k in TILE_KERNELS})
    s.segments = seg
    s.start(st)
    s.run(0, 3)
    got = s.get_state(1)
    s.close()
    assert all(np.array_equal(got[k], want[k]) for k in want)


@pytest.mark.parametrize("ny,nx,nl,oro,moist,rows,seg", [(5, 61, 16, 12, True, 1, 4), (6, 62, 9, 8, False, 2, 2), (5, 63, 6, 4, True, 4, 1),
                                                         (3, 125, 5, 1, False, 4, 1)])
def test_third_order_theta_columns_match_oracle(ny, nx, nl, oro, moist, rows, seg):
    """The divergence of the theta gradient marches down 62-cell row tiles in vertical segments: one partial
    tile, full ones and a third, the fewest rows, flat and terrain-following layers, bitwise against the oracle."""
    cfg = dataclasses.replace(tiny_config(ny=ny, nx=nx, n_layers=nl, moist=moist, order=3), n_oro_layers=oro)
    g, st = make_case(cfg, cloud_frac=0.3 if moist else 0.0)
    want = _oracle(cfg, g, st, 3)
    s = Step(cfg, g)
    s.set_tiles({k: rows for k in TILE_KERNELS})
    s.segments = seg
    s.start(st)
    s.run(0, 3)
    got = s.get_state(1)
    s.close()
    assert all(np.array_equal(got[k], want[k]) for k in want)


@pytest.mark.parametrize("nl,nx", [(3, 5), (4, 63), (5, 64), (16, 65), (17, 7), (18, 7), (31, 128), (33, 129), (48, 9), (50, 9), (63, 64),
                                   (64, 70), (66, 7), (71, 64), (72, 65)])
def test_tracer_solver_levels_match_oracle(nl, nx):
    """The tracer solver keeps up to 72 levels in parts of 16, worked on in chunks of 1, 2 or 4: the
    smallest columns, the ends of chunks and parts, the tallest column that fits, bitwise against the oracle."""
    cfg = dataclasses.replace(tiny_config(ny=3, nx=nx, n_layers=nl, moist=True), n_oro_layers=max(1, nl - 4))
    g, st = make_case(cfg, cloud_frac=0.3)
    want = _oracle(cfg, g, st, 3)
    s = Step(cfg, g)
    s.start(st)
    s.run(0, 3)
    got = s.get_state(1)
    s.close()
    assert all(np.array_equal(got[k], want[k]) for k in want)


@pytest.mark.parametrize("precision,nx", [(PREC_FP64, 9), (PREC_FP64, 64), (PREC_FP64, 70), (PREC_MIXED, 70)])
def test_lowest_tall_tracer_columns_match_oracle(precision, nx):
    """65 layers, the first height of the tracer solver's tall form.  At nx 70 the FP64 form differs from the
    oracle by one unit in the last place of wind_w and cloud water in one column, where the device's exp in the
    heat capacity of ice is one unit from the host's: agreement to rounding, and the mixed form's own bar."""
    cfg = dataclasses.replace(tiny_config(ny=3, nx=nx, n_layers=65, moist=True), n_oro_layers=61)
    g, st = make_case(cfg, cloud_frac=0.3)
    want = _oracle(cfg, g, st, 3)
    s = Step(dataclasses.replace(cfg, precision=precision), g)
    s.start(st)
    s.run(0, 3)
    got = s.get_state(1)
    s.close()
    if precision == PREC_MIXED:
        err = field_errors(got, want)
        assert worst(err, "rms_rel") < 1e-4 and worst(err, "max_rel") < 1e-4
    else:
        assert max_rel(got, want) <= 1e-12


@pytest.mark.parametrize("layers", [(40, 64, 65, 72), (40, 65, 72, 73)])
def test_batched_mixed_members_of_different_height_match_single(layers):
    """The mixed form of a batched group whose members take different column solvers: every member has
    the bits it has when stepped alone."""
    cfgs = [dataclasses.replace(tiny_config(ny=4, nx=20 + 25 * i, n_layers=nl, moist=True), precision=PREC_MIXED)
            for i, nl in enumerate(layers)]
    cases = [make_case(c, cloud_frac=0.3) for c in cfgs]
    steps = []
    for c, (g, st) in zip(cfgs, cases):
        s = Step(c, g)
        s.start(st)
        steps.append(s)
    e = Ensemble(steps)
    e.run(0, 3, mode=Ensemble.BATCHED)
    e.sync()
    for c, (g, st), s in zip(cfgs, cases, steps):
        one = Step(c, g)
        one.start(st)
        one.run(0, 3)
        got, want = s.get_state(1), one.get_state(1)
        one.close()
        assert all(np.array_equal(got[k], want[k]) for k in want), c.n_layers
    e.close()
    for s in steps:
        s.close()


def test_batched_tracer_solver_with_members_of_different_height():
    cfgs = [tiny_config(ny=4 + i, nx=30 + 40 * i, n_layers=nl, moist=True) for i, nl in enumerate((66, 7, 64, 70, 73))]
    cases = [make_case(c, cloud_frac=0.3) for c in cfgs]
    steps = []
    for c, (g, st) in zip(cfgs, cases):
        s = Step(c, g)
        s.start(st)
        steps.append(s)
    e = Ensemble(steps)
    e.run(0, 3, mode=Ensemble.BATCHED)
    e.sync()
    for c, (g, st), s in zip(cfgs, cases, steps):
        got, want = s.get_state(1), _oracle(c, g, st, 3)
        assert all(np.array_equal(got[k], want[k]) for k in want), c.n_layers
    e.close()
    for s in steps:
        s.close()


def test_vertical_solver_default_passes_by_size():
    """One pass per column once the domain has as many 64-column wavefronts as the GPU has SIMDs."""
    for n, want in ((128, 3), (256, 1)):
        cfg = dry3d_config(n=n, n_layers=10)
        g, st = make_case(cfg)
        s = Step(cfg, g)
        assert s.column_passes == want, n
        s.close()


@pytest.mark.parametrize("mode", [Ensemble.GRAPH, Ensemble.SERIAL, Ensemble.BATCHED])
def test_ensemble_members_match_oracle(mode):
    cfgs = [tiny_config(ny=5, nx=7, n_layers=6, moist=True, order=3),
            tiny_config(ny=9, nx=11, n_layers=8),
            # even nx: two cells per thread in the potential vorticity of a single-domain launch,
            # one cell per thread in the batched one; nx not a multiple of 64 in the column solvers
            tiny_config(ny=6, nx=70, n_layers=7, moist=True),
            dry3d_config(n=17, n_layers=10),
            # a member with the reference's default physics: diffusion, PBL, prognostic soil
            dataclasses.replace(tiny_config(ny=7, nx=9, n_layers=8, moist=True), lpbl=True, lprog_soil_temp=True,
                                lsfc_sensible_heat_flux=True, lsfc_phase_trans=True).set_diffusion()]
    cases = [make_case(c, cloud_frac=0.1 if c.lmoist else 0.0) for c in cfgs]
    steps = []
    for c, (g, st) in zip(cfgs, cases):
        s = Step(c, g)
        s.start(st)
        if mode == Ensemble.GRAPH:
            s.set_tiles({k: (1, 2, 4)[i % 3] for i, k in enumerate(TILE_KERNELS)})
        steps.append(s)
    e = Ensemble(steps)
    n = 7
    print(f"ensemble of {len(steps)} members, mode {mode}, {n} steps", flush=True)
    e.run(0, n, mode=mode)
    e.sync()
    for c, (g, st), s in zip(cfgs, cases, steps):
        got = s.get_state(n % 2)
        want = _oracle(c, g, st, n)
        assert all(np.array_equal(got[k], want[k]) for k in want), f"member {c.ny}x{c.nx}x{c.n_layers}"
    e.close()
    for s in steps:
        s.close()


def test_batched_radiation_set_up_after_the_first_step():
    """The batched groups are made at the first batched step; a radiation set up afterwards (surface
    data, surrogate) is taken up at the first radiation update: the batched steps stay bitwise equal
    to serial ones."""
    from lgame import surrogate
    from lgame.cases import moist3d_config, radiation_surface
    from lgame.config import PREC_MIXED, RAD_SURROGATE

    mlp = surrogate.load(surrogate.DEFAULT_WEIGHTS)
    cfgs = [dataclasses.replace(moist3d_config(n=n, n_layers=60, seed=30 + n), precision=PREC_MIXED, lrad=True,
                                rad_mode=RAD_SURROGATE, dtime_rad=900.0) for n in (33, 47)]
    cases = [make_case(c, cloud_frac=0.005) for c in cfgs]
    t0 = 1576843200.0 + 3 * 3600.0
    out = {}
    for mode in (Ensemble.BATCHED, Ensemble.SERIAL):
        steps = []
        for c, (g, st) in zip(cfgs, cases):
            s = Step(c, g)
            s.start(st)
            steps.append(s)
        e = Ensemble(steps)
        e.step(0, mode=mode)
        for c, (g, st), s in zip(cfgs, cases, steps):
            s.set_rad_surface(radiation_surface(c, g, st))
            s.attach_mlp(mlp, tol_k_per_day=1.0, audit_fraction=0.05, seed=3)
        for k in range(1, 4):
            e.step(k, lrad_update=(k == 1), t_0=t0 + k * cfgs[0].dt, mode=mode)
        e.sync()
        out[mode] = [s.get_state(0) for s in steps]
        assert all(s.rad_stats()["calls"] == 1 for s in steps)
        e.close()
        for s in steps:
            s.close()
    for a, b in zip(out[Ensemble.BATCHED], out[Ensemble.SERIAL]):
        assert all(np.array_equal(a[k], b[k]) for k in a)
