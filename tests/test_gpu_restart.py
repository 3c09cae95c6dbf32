"""Fault detection and restarts through the C-ABI.

* The step's own non-finite check: after an unstable step (the Schaer case at dt 4 s, which the
  reference scheme also blows up) lgame_sync reports LGAME_ENONFINITE, as the reference's output
  check stops the run (mo_write_out.F90:63-67); a new state clears it.
* A restart from the two states plus the checkpoint of the carried fields continues the run bit
  for bit; without the checkpoint (the reference's own restart carries the state only) it does
  not.
"""
import dataclasses

import numpy as np
import pytest

from lgame import surrogate
from lgame.cases import make_case, moist3d_config, radiation_surface, schaer_config, tiny_config
from lgame.config import PREC_FP64, PREC_MIXED, RAD_SURROGATE, RAD_TEACHER
from lgame.gpu import LgameError, Step
from pyoracle import CpuOracle

pytestmark = pytest.mark.gpu
T0 = surrogate.T_EPOCH + 3 * 3600.0


def test_unstable_step_is_reported_at_sync():
    cfg = schaer_config(nx=201, n_layers=40, dtime=4.0)
    g, st = make_case(cfg)
    s = Step(cfg, g)
    s.start(st)
    s.run(0, 30)
    with pytest.raises(LgameError, match="non-finite"):
        s.sync()
    assert s.count_nonfinite(0) > 0
    # a new state clears the flag; a stable run keeps it clear
    s2 = Step(schaer_config(nx=201, n_layers=40), g)
    s2.start(st)
    s2.run(0, 30)
    s2.sync()
    s.start(st)
    s.sync()
    s.close()
    s2.close()


def _physics(cfg):
    return dataclasses.replace(cfg, lpbl=True, lprog_soil_temp=True, lsfc_sensible_heat_flux=True,
                               lsfc_phase_trans=True).set_diffusion()


def _restart_case(name):
    if name == "moist_physics_radiation":
        cfg = _physics(tiny_config(ny=9, nx=11, n_layers=8, moist=True, order=3, freeslip=True))
        cfg = dataclasses.replace(cfg, lrad=True, rad_mode=RAD_TEACHER, dtime_rad=3 * 2.0)
        g, st = make_case(cfg, cloud_frac=0.3)
        return cfg, g, st, radiation_surface(cfg, g, st), None
    if name == "mixed_surrogate":
        cfg = moist3d_config(n=33, n_layers=60, dtime=3.22, seed=21)
        cfg = dataclasses.replace(cfg, lrad=True, rad_mode=RAD_SURROGATE, dtime_rad=3 * cfg.dt, precision=PREC_MIXED)
        g, st = make_case(cfg, cloud_frac=0.01)
        return cfg, g, st, radiation_surface(cfg, g, st), surrogate.load(surrogate.DEFAULT_WEIGHTS)
    cfg = tiny_config(order=3, corio=True)
    g, st = make_case(cfg)
    return cfg, g, st, None, None


def _handle(cfg, g, sf, mlp):
    s = Step(cfg, g)
    if sf is not None:
        s.set_rad_surface(sf)
    if mlp is not None:
        s.attach_mlp(mlp, tol_k_per_day=1.0, audit_fraction=0.05, seed=3)
    return s


@pytest.mark.parametrize("name", ["dry", "moist_physics_radiation", "mixed_surrogate"])
def test_restart_from_checkpoint_is_bitwise(name):
    cfg, g, st, sf, mlp = _restart_case(name)
    k, m = 5, 6
    print(f"case {name}: {k} steps, checkpoint, {m} more", flush=True)
    a = _handle(cfg, g, sf, mlp)
    a.start(st)
    a.run(0, k, t_init=T0)
    slots = [a.get_state(0), a.get_state(1)]
    blob = a.checkpoint()
    a.run(k, m, t_init=T0)
    want = a.get_state((k + m) % 2)
    a.close()
    b = _handle(cfg, g, sf, mlp)
    b.set_state(0, slots[0])
    b.set_state(1, slots[1])
    b.restore(blob)
    b.run(k, m, t_init=T0)
    got = b.get_state((k + m) % 2)
    b.close()
    print(f"checkpoint of {len(blob) / 1e6:.2f} MB")
    assert all(np.array_equal(got[f], want[f]) for f in want)
    # the state alone (the reference's restart) does not continue the same run
    c = _handle(cfg, g, sf, mlp)
    c.set_state(0, slots[0])
    c.set_state(1, slots[1])
    c.run(k, m, t_init=T0)
    other = c.get_state((k + m) % 2)
    c.close()
    assert not all(np.array_equal(other[f], want[f]) for f in want)


def test_checkpoint_of_another_configuration_is_refused():
    cfg, g, st, _, _ = _restart_case("dry")
    a = Step(cfg, g)
    a.start(st)
    blob = a.checkpoint()
    cfg2 = dataclasses.replace(cfg, lmoist=True)
    g2, st2 = make_case(cfg2)
    b = Step(cfg2, g2)
    b.start(st2)
    with pytest.raises(LgameError, match="configuration"):
        b.restore(blob)
    with pytest.raises(LgameError, match="truncated|too short|configuration"):
        a.restore(blob[:-8])
    a.close()
    b.close()


def test_checkpoint_pressure_gradient_parts_are_summed():
    """The layout has boxes for the nonlinear and the linear pressure gradient, whose sum is what a run
    carries: a checkpoint that spreads the sum over both (halves, exact in binary) continues the
    same run."""
    cfg, g, st, _, _ = _restart_case("dry")
    a = Step(cfg, g)
    a.start(st)
    a.run(0, 5)
    slots = [a.get_state(0), a.get_state(1)]
    blob = bytearray(a.checkpoint())
    a.run(5, 4)
    want = a.get_state(1)
    a.close()
    pitch = (cfg.nx + 1 + 15) // 16 * 16
    box, head = 8 * (cfg.n_layers + 1) * (cfg.ny + 1) * pitch, 56
    part = lambda q: np.frombuffer(blob, dtype=np.float64, count=box // 8, offset=head + q * box)  # noqa: E731
    for nonlinear, linear in ((0, 3), (1, 4)):
        assert np.abs(part(nonlinear)).max() > 0.0 and np.abs(part(linear)).max() == 0.0
        half = 0.5 * part(nonlinear)
        for q in (nonlinear, linear):
            blob[head + q * box:head + (q + 1) * box] = half.tobytes()
    b = Step(cfg, g)
    b.set_state(0, slots[0])
    b.set_state(1, slots[1])
    b.restore(bytes(blob))
    b.run(5, 4)
    got = b.get_state(1)
    b.close()
    assert all(np.array_equal(got[f], want[f]) for f in want)


@pytest.mark.parametrize("precision", [PREC_FP64, PREC_MIXED])
def test_diagnosing_a_slot_keeps_the_carried_fields(precision):
    """Reading the radiation columns of either slot between steps, or the budget sums of a restored run
    before its first step, diagnoses the temperature of that slot and nothing that a run carries: the last
    step's dissipation rate (of the Klemp layer alone) and the checkpoint stay as they are."""
    cfg = dataclasses.replace(tiny_config(ny=7, nx=9, n_layers=12, moist=True), lrad=True, rad_mode=RAD_TEACHER, dtime_rad=6.0,
                              precision=precision)
    g, st = make_case(cfg, cloud_frac=0.02)
    a = Step(cfg, g)
    a.start(st)
    a.set_rad_surface(radiation_surface(cfg, g, st))
    a.run(0, 5, t_init=T0)
    rate, blob = a.diag("heating_diss"), a.checkpoint()
    assert np.abs(rate).max() > 0.0
    for slot in (0, 1):
        a.rad_columns(slot, T0)
        assert np.array_equal(a.diag("heating_diss"), rate)
    assert a.checkpoint() == blob
    b = Step(cfg, g)
    b.set_rad_surface(radiation_surface(cfg, g, st))
    for slot in (0, 1):
        b.set_state(slot, a.get_state(slot))
    b.restore(blob)
    for slot in (0, 1):
        b.integrals(slot)
    assert np.array_equal(b.diag("heating_diss"), rate)
    assert b.checkpoint() == blob
    a.close()
    b.close()


def test_restored_dissipation_rate_is_zero_below_the_klemp_layer():
    """With the Klemp layer as the only dissipation the rate is formed in its levels: a checkpoint that holds
    other values below them leaves zeros there, as soon as it is loaded, and the rate in the levels above."""
    cfg, g, st, _, _ = _restart_case("dry")
    a = Step(cfg, g)
    a.start(st)
    a.run(0, 5)
    rate, blob = a.diag("heating_diss"), bytearray(a.checkpoint())
    levels = CpuOracle(cfg, g).n_damping_levels
    assert 0 < levels < cfg.n_layers and np.abs(rate).max() > 0.0
    pitch = (cfg.nx + 1 + 15) // 16 * 16
    shape = (cfg.n_layers + 1, cfg.ny + 1, pitch)
    offset = 56 + 19 * 8 * int(np.prod(shape))  # after the header and 8 boxes of the pressure gradient, 10 of the advection and 1 of the sediment heating
    box = np.frombuffer(blob, dtype=np.float64, count=int(np.prod(shape)), offset=offset).reshape(shape).copy()
    assert np.array_equal(box[:cfg.n_layers, :cfg.ny, :cfg.nx].transpose(1, 2, 0), rate)
    box[levels:] = 1.0
    blob[offset:offset + box.nbytes] = box.tobytes()
    for _ in range(3):
        a.restore(bytes(blob))
        assert np.array_equal(a.diag("heating_diss"), rate)
    a.close()
