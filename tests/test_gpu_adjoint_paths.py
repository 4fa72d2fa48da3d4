"""Every way through the adjoint, whatever an ensemble's size would choose: the
step tapes kept or the segments recomputed, and either reverse sweep, with
evolving stars, wind, every coordinate type, hosts anywhere and systems that
stop on their way."""
import os

import numpy as np
import pytest

from posidonius_amd import abi, generators as gen
from posidonius_amd.case import EnsembleSpec
from tests.test_gpu_adjoint import (BLOCKS, check_against_tangent, coordinate_workloads, directions, evolving_workload,
                                    wind_workload)
from tests.test_gpu_adjoint_sweep import RTOL, sizes

pytestmark = pytest.mark.gpu

SWEEPS = ("prepared", "kernel")
TAPES = {"kept": 0, "recomputed": -1}      # adjoint_tape_mib
STEPS, SEGMENT = 300, 70                   # five segments, the last one shorter


def handle(spec, sweep, tapes):
    from posidonius_amd.ensemble import Ensemble
    return Ensemble(spec, mapping="packed", adjoint_sweep=sweep, adjoint_tape_mib=TAPES[tapes])


def evolving_in_jacobi(n_systems, steps):
    spec = evolving_workload(n_systems, steps)
    spec.system["coordinates"][::2] = abi.COORD_JACOBI
    return spec


WORKLOADS = {"star_3planets": lambda: gen.config4(16), "wind": lambda: wind_workload(16),
             "evolution": lambda: evolving_workload(16, STEPS), "evolution_jacobi": lambda: evolving_in_jacobi(16, STEPS),
             "host_moved": lambda: coordinate_workloads()["host_moved"],
             "all_three_coordinates": lambda: coordinate_workloads()["all_three_coordinates"]}


@pytest.mark.parametrize("name", sorted(WORKLOADS))
def test_each_path_equals_tangent_linear(oracle, name):
    """Every seed block against every tangent direction to 1e-6 relative, and
    the same bits whether the tapes were kept or not."""
    spec = WORKLOADS[name]()
    d = directions(spec, np.random.default_rng(51))
    ref, tan = oracle.tangent(spec, STEPS, d, threads=max(1, min(16, os.cpu_count() or 1)))
    w = np.random.default_rng(52).standard_normal((spec.n_bodies, 3))
    for sweep in SWEEPS:
        got = {}
        for tapes in TAPES:
            print(f"{name}: {sweep} sweep, tapes {tapes}", flush=True)
            with handle(spec, sweep, tapes) as ens:
                ens.adjoint_record(STEPS, SEGMENT)
                fin = ens.get_state()
                for k in BLOCKS:
                    np.testing.assert_array_equal(fin[k], ref[k], err_msg=f"recorded forward run differs in {k}")
                check_against_tangent(ens, spec, np.random.default_rng(53), d, tan, f"{name} {sweep} {tapes}")
                got[tapes] = ens.adjoint(position=w, velocity=w, angular_momentum=w)
                for k, a in ens.get_state().items():
                    np.testing.assert_array_equal(a, fin[k], err_msg=k)
        for k, a in got["kept"].items():
            np.testing.assert_array_equal(a, got["recomputed"][k], err_msg=f"{sweep}: {k}")


def stopping(seed):
    """Sizes and coordinates mixed, hosts anywhere, wind on half of the stars;
    every fourth system stops on its way (9, 17, 25, ... steps)."""
    spec = sizes((2, 3, 5, 6, 8), seed, abi.COORD_JACOBI)
    n = spec.n_systems
    spec.system["coordinates"][:] = np.arange(n) % 3
    host = np.zeros(spec.n_bodies, dtype=bool)
    for b0, b1 in zip(spec.body_offset[:-1], spec.body_offset[1:]):
        host[b0 + np.argmax(spec.body["mass"][b0:b1])] = True
    spec.system["effects"][n // 2:] |= abi.EFFECT_WIND
    spec.body["roles"] = np.where(host, spec.body["roles"] | abi.ROLE_WIND, spec.body["roles"]).astype(spec.body["roles"].dtype)
    spec.body["wind_k_factor"] = np.where(host, 4e-12, 0.)
    spec.body["wind_rotation_saturation"] = np.full(spec.n_bodies, 1.7592918860102842)
    stop = np.where(np.arange(n) % 4 == 1, 2 * np.arange(n) + 7, 1000)
    spec.system["time_limit"][:] = (stop + 0.5) * spec.system["time_step"]
    spec.system["historic_snapshot_period"][:] = 3.3 * spec.system["time_step"]
    return spec


@pytest.mark.parametrize("sweep", SWEEPS)
def test_recomputed_segments_append_no_records(sweep):
    """Recomputing the segments of a run with snapshots and stopped systems
    gives the kept run's bits and no records of its own."""
    spec = stopping(61)
    steps, segment = 60, 9
    w = np.random.default_rng(62).standard_normal((spec.n_bodies, 3))
    got = []
    for tapes in TAPES:
        with handle(spec, sweep, tapes) as ens:
            ens.enable_history(32)
            ens.adjoint_record(steps, segment)
            rec = ens.drain_history()
            grad = [ens.adjoint(position=w, velocity=w, angular_momentum=w) for _ in range(2)]
            assert len(ens.drain_history()) == 0
            got.append((grad, rec, ens.get_state()))
    assert np.any(got[0][2]["current_iteration"] < steps) and len(got[0][1]) > 0
    with handle(spec, sweep, "kept") as ens:
        ens.enable_history(32)
        ens.step(steps)
        plain, state = ens.drain_history(), ens.get_state()
    for grad, rec, st in got:
        for k in plain.dtype.names:
            np.testing.assert_array_equal(rec[k], plain[k], err_msg=k)
        for k in state:
            np.testing.assert_array_equal(st[k], state[k], err_msg=k)
        for g in grad:
            for k, a in g.items():
                assert np.all(np.isfinite(a)), k
                np.testing.assert_array_equal(a, got[0][0][0][k], err_msg=k)


def both_sweeps(spec, steps, segment):
    w = np.random.default_rng(66).standard_normal((spec.n_bodies, 3))
    out = {}
    for sweep in SWEEPS + ("auto",):
        with handle(spec, sweep, "kept") as ens:
            ens.adjoint_record(steps, segment)
            out[sweep] = ens.adjoint(position=w, velocity=w, angular_momentum=w)
    return out


def sweeps_agree(spec, where):
    """The sweeps differ by the roundings of 24 steps (see RTOL)."""
    out = both_sweeps(spec, 24, 9)
    for k, a in out["prepared"].items():
        b = out["kernel"][k]
        assert np.all(np.isfinite(b))
        for s in range(spec.n_systems):
            i = slice(spec.body_offset[s], spec.body_offset[s + 1])
            assert np.abs(a[i] - b[i]).max() <= RTOL * np.abs(b[i]).max(), (where, k, s)


@pytest.mark.parametrize("coords", [abi.COORD_DEMOCRATIC_HELIOCENTRIC, abi.COORD_JACOBI, abi.COORD_WHDS])
@pytest.mark.parametrize("counts", [(2, 3, 4), (5, 7, 8), (2, 9, 15, 16)], ids=["4_slots", "8_slots", "16_slots"])
def test_the_two_sweeps(counts, coords):
    sweeps_agree(sizes(counts, 40, coords), f"sizes {counts} coordinates {coords}")


def test_the_two_sweeps_on_evolving_and_stopping_systems():
    sweeps_agree(EnsembleSpec.concat([evolving_in_jacobi(8, 24), sizes((2, 5, 16), 65, abi.COORD_WHDS)]), "evolving")
    sweeps_agree(stopping(61), "stopping")


@pytest.mark.parametrize("more,sweep", [(0, "prepared"), (1, "kernel")])
def test_the_sweep_by_size(more, sweep):
    """Up to one set of systems per CU the prepared sweep, beyond it the kernel."""
    from tests.test_gpu_teams import edge
    spec = gen.config2((64 // 16) * edge(1, more), seed=75, n_min=9, n_max=16)
    out = both_sweeps(spec, 6, 4)
    for k, a in out["auto"].items():
        np.testing.assert_array_equal(a, out[sweep][k], err_msg=k)
    assert any(np.any(out["prepared"][k] != out["kernel"][k]) for k in out["auto"])


@pytest.mark.parametrize("setting", ["time_limit", "snapshot_period", "roche_radius"])
@pytest.mark.parametrize("tapes", sorted(TAPES))
def test_settings_changed_after_the_recording(tapes, setting):
    """The adjoint is of the run as it was recorded: a time limit, snapshot
    period or Roche radii set afterwards stay as set but do not enter it."""
    spec = stopping(67)
    steps, segment = 60, 9
    w = np.random.default_rng(68).standard_normal((spec.n_bodies, 3))
    got = []
    for change in (False, True):
        with handle(spec, "kernel", tapes) as ens:
            ens.adjoint_record(steps, segment)
            end = ens.get_state()
            if change and setting == "time_limit":
                ens.set_time_limit(12.5 * spec.system["time_step"].min())
            if change and setting == "snapshot_period":
                ens.set_historic_snapshot_period(1.1 * spec.system["time_step"].max())
            roche = np.full_like(end["roche_radius"], 1e3) if change and setting == "roche_radius" else end["roche_radius"]
            ens.set_state({"roche_radius": roche})
            got.append(ens.adjoint(position=w, velocity=w, angular_momentum=w))
            after = ens.get_state()
        for k in end:
            np.testing.assert_array_equal(after[k], roche if k == "roche_radius" else end[k], err_msg=k)
    for k in got[0]:
        np.testing.assert_array_equal(got[1][k], got[0][k], err_msg=k)


def test_gradients_are_the_same_under_every_mapping():
    """The choice of the sweep follows from the ensemble: the same bits from
    few sets of systems and from more than one per CU, on each side of the
    autotuner."""
    from posidonius_amd.ensemble import Ensemble
    from tests.test_gpu_teams import edge
    spec = gen.config2(edge(1, 44), seed=71, n_min=2, n_max=9)
    w = np.random.default_rng(72).standard_normal((spec.n_bodies, 3))
    out = {}
    for name, options in {"pow2": dict(), "exact": dict(group_size=-1), "mixed": dict(group_size=-2),
                          "set_per_system": dict(group_size=64), "plain": dict(mapping="plain"), "tuned": dict()}.items():
        with Ensemble(spec, **{"mapping": "packed", **options}) as ens:
            if name == "tuned":
                ens.tune(16)
            ens.adjoint_record(24, 9)
            out[name] = ens.adjoint(position=w, velocity=w, angular_momentum=w)
    for name, grad in out.items():
        for k, a in grad.items():
            np.testing.assert_array_equal(a, out["pow2"][k], err_msg=f"{name}: {k}")


def test_stretches_leave_no_trace():
    """The prepared sweep walks a segment by as many steps as its workspace
    holds: the same systems alone (all steps at once) and among enough others
    to take several stretches, and segments of any length, give the same bits."""
    steps = 40
    spec = gen.config2(1024, seed=73, n_min=4, n_max=4)
    planes, half = 174 + 2 * 4, 128 << 20                   # 16 bytes a body and plane
    assert 1 < half // (16 * planes * spec.n_bodies) < steps // 2
    w = np.random.default_rng(74).standard_normal((spec.n_bodies, 3))
    few = spec.subset(range(16))

    def gradients(s, segment):
        with handle(s, "prepared", "kept") as ens:
            ens.adjoint_record(steps, segment)
            u = w[:s.n_bodies]
            return ens.adjoint(position=u, velocity=u, angular_momentum=u)

    whole = gradients(few, steps)
    for s, segment in ((spec, steps), (spec, 17), (few, 1), (few, 17)):
        for k, a in gradients(s, segment).items():
            np.testing.assert_array_equal(a[:few.n_bodies], whole[k], err_msg=f"{s.n_systems} systems, segments of {segment}: {k}")


@pytest.mark.parametrize("sweep", SWEEPS)
@pytest.mark.parametrize("coords", [abi.COORD_DEMOCRATIC_HELIOCENTRIC, abi.COORD_JACOBI, abi.COORD_WHDS])
def test_gradients_do_not_depend_on_the_systems_around(sweep, coords):
    """Each other kind of system (larger, in other coordinates, evolving) brings
    other kernels; the first systems' gradients keep their bits."""
    few = sizes((2, 3, 4), 40, coords)
    w = np.random.default_rng(76).standard_normal((few.n_bodies, 3))

    def gradients(spec):
        u = np.zeros((spec.n_bodies, 3))
        u[:few.n_bodies] = w
        with handle(spec, sweep, "kept") as ens:
            ens.adjoint_record(24, 9)
            return ens.adjoint(position=u, velocity=u, angular_momentum=u)

    alone = gradients(few)
    others = {"8_slots": sizes((6,), 41, abi.COORD_DEMOCRATIC_HELIOCENTRIC), "16_slots": sizes((16,), 42, abi.COORD_JACOBI),
              "jacobi": sizes((4,), 43, abi.COORD_JACOBI), "whds": sizes((3,), 44, abi.COORD_WHDS),
              "evolving": evolving_workload(4, 24), "wind": wind_workload(4)}
    for name, other in others.items():
        for k, a in gradients(EnsembleSpec.concat([few, other])).items():
            np.testing.assert_array_equal(a[:few.n_bodies], alone[k], err_msg=f"with {name}: {k}")
