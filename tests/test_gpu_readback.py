"""Reading state back: the packed path (small requests, one launch) and the
field-by-field path (large ones) return the same values for every field, and
the operators' results do not depend on which one they take."""
import numpy as np
import pytest

from posidonius_amd import abi, generators as gen
from posidonius_amd.case import EnsembleSpec
from tests.oracle_runner import load_golden

pytestmark = pytest.mark.gpu

LIMIT = 2 << 20     # bytes of one request that go through the packed path


def mixed(systems):
    """Plain systems of 2 to 16 bodies, shuffled against the device order, and
    two evolving ones (left indices, pair factors, Roche radii to tell apart)."""
    spec = EnsembleSpec.concat([gen.config2(systems, seed=9, n_min=2, n_max=abi.MAX_BODIES),
                                load_golden("test_evolution-solar_like_bolmontmathis2016")[0],
                                load_golden("test_disk-enabled_disk")[0]])
    return spec


@pytest.mark.parametrize("systems", [1, 130, 1000])
def test_every_field_alone_and_together(systems):
    from posidonius_amd.ensemble import Ensemble
    spec = mixed(systems)
    with Ensemble(spec, group_size=-2) as ens:
        ens.step(3)
        whole = ens.get_state()
        size = sum(a.nbytes for a in whole.values())
        print(f"{spec.n_bodies} bodies, {size} bytes", flush=True)
        assert (size > LIMIT) == (systems == 1000)
        for k, a in whole.items():
            np.testing.assert_array_equal(ens.get_state((k,))[k], a, err_msg=k)
        again = ens.get_state()
        for k, a in whole.items():
            np.testing.assert_array_equal(again[k], a, err_msg=k)
    assert len(np.unique(whole["position"], axis=0)) == spec.n_bodies


def test_operators_on_both_sides_of_the_limit(oracle):
    """3 doubles a body: two arrays just below and just above the limit."""
    from posidonius_amd.ensemble import Ensemble
    base = mixed(200)
    bodies = LIMIT // 48
    few = EnsembleSpec.concat([base] * (bodies // base.n_bodies))
    more = EnsembleSpec.concat([base] * (bodies // base.n_bodies + 1))
    ref_e, ref_g = oracle.additional_effects(base), oracle.gravity(base)
    for spec in (few, more):
        n = spec.n_bodies // base.n_bodies
        print(f"{spec.n_bodies} bodies", flush=True)
        with Ensemble(spec) as ens:
            got = ens.additional_effects()
            grav = ens.gravity_acceleration()
        for a, b in zip(got + grav, ref_e + ref_g):
            np.testing.assert_array_equal(a, np.concatenate([b] * n))


@pytest.mark.parametrize("systems,steps,chunk_edge", [(3, 5, False), (70, 40, False), (3000, 28, True)])
def test_drained_records_in_input_order(oracle, systems, steps, chunk_edge):
    """Systems that record every step, every other one and never, in sizes
    that differ: the records come out by system, record and body, with the
    state the oracle has at that step and the constants of the input; the
    largest case takes more than one stretch of packed records (2^18)."""
    from posidonius_amd.ensemble import Ensemble
    spec = gen.config2(systems, seed=31, n_min=2, n_max=12)
    dt = spec.system["time_step"]
    every = np.arange(systems) % 3
    spec.system["historic_snapshot_period"][:] = np.where(every == 2, np.inf, (every + 0.9) * dt)
    with Ensemble(spec, group_size=-2) as ens:
        ens.enable_history(steps + 2)
        ens.step(steps)
        rec = ens.drain_history()
        assert len(ens.drain_history()) == 0
        ens.step(2)
        more = ens.drain_history()
    n = spec.n_per_system()
    print(f"{len(rec)} records", flush=True)
    assert (len(rec) > 1 << 18) == chunk_edge
    first = np.flatnonzero((rec["body"] == 0))
    assert np.all(np.diff(rec["system"]) >= 0)
    counts = np.bincount(rec["system"], minlength=systems) // n
    assert np.all(counts[every == 2] == 1) and np.all(counts[every == 0] == steps)
    want = np.concatenate([np.tile(np.arange(n[s]), counts[s]) for s in range(systems)])
    np.testing.assert_array_equal(rec["body"], want)
    body = spec.body_offset[rec["system"]] + rec["body"]
    np.testing.assert_array_equal(rec["mass"], spec.body["mass"][body])
    np.testing.assert_array_equal(rec["time_step"], dt[rec["system"]])
    np.testing.assert_array_equal(rec["scaled_dissipation_factor"],
                                  (spec.body["tides_dissipation_factor_scale"] * spec.body["tides_dissipation_factor"])[body])
    few = spec.subset(range(min(systems, 12)))
    for k in (0, 2, steps - 1):
        ref = oracle.run(few, k) if k else {"position": few.body["position"], "velocity": few.body["velocity"]}
        for s in range(0, few.n_systems, 3):       # these record at every step
            b0 = int(np.flatnonzero(rec["system"] == s)[0]) + k * n[s]
            o = slice(spec.body_offset[s], spec.body_offset[s + 1])
            np.testing.assert_array_equal(rec["position"][b0:b0 + n[s]], ref["position"][o])
            np.testing.assert_array_equal(rec["velocity"][b0:b0 + n[s]], ref["velocity"][o])
    assert len(first) == counts.sum()
    assert np.all(more["system"] % 3 != 2) and len(more) > 0


def test_draining_takes_no_device_memory():
    """The memory to pack records in comes with the record buffer, so a drain
    succeeds however full the device is by then."""
    import torch
    from posidonius_amd.ensemble import Ensemble
    torch.cuda.init()
    spec = gen.config2(3000, seed=31, n_min=7, n_max=7)
    spec.system["historic_snapshot_period"][:] = 0.9 * spec.system["time_step"]
    with Ensemble(spec) as ens:
        ens.enable_history(16)
        assert 16 * spec.n_bodies > 1 << 18        # more than one stretch of 168-byte records
        ens.step(14)
        ens.get_state(("current_time",))
        before = torch.cuda.mem_get_info()[0]
        assert len(ens.drain_history()) == 14 * spec.n_bodies
        assert before - torch.cuda.mem_get_info()[0] < 20 << 20


def test_fields_that_do_not_fit_are_read_one_by_one():
    """Four fields of three doubles fill the packed buffer up to less than the
    smallest field: every other one, per system and per body, integers and rows,
    takes the path that also serves where no pinned memory can be had."""
    from posidonius_amd.ensemble import Ensemble
    spec = gen.config2(9500, seed=12, n_min=2, n_max=3)
    spec = spec.subset(range(int(np.searchsorted(spec.body_offset, LIMIT // 96, side="right")) - 1))
    left = LIMIT - 96 * spec.n_bodies
    assert 0 <= left < 4 * spec.n_systems
    with Ensemble(spec, group_size=-2) as ens:
        ens.step(2)
        whole = ens.get_state()
        for k, a in whole.items():
            np.testing.assert_array_equal(a, ens.get_state((k,))[k], err_msg=k)
