"""The fixed-effect-set step under each team size (1, 2 or 4 wavefronts per
set of systems, chosen by how many sets a launch has): every size gives the
oracle's bits, also for systems that stop or record snapshots within a launch,
and the adjoint's gradients do not depend on it."""
import os

import numpy as np
import pytest

from posidonius_amd import abi, generators as gen
from tests.spec_tools import move_host
from tests.test_gpu_parity import THREADS, assert_same_state

pytestmark = pytest.mark.gpu

# sets of systems per CU: the last of a team size and the first of the next
EDGES = ((2, 0), (2, 1), (4, 0), (4, 1))


def edge(per_cu, more):
    import torch
    return per_cu * torch.cuda.get_device_properties(0).multi_processor_count + more


def ensemble(systems, coords, seed):
    """Systems of 2 to 16 bodies, the host anywhere in its system; some reach
    their time limit within the run, one collides in its first step."""
    spec, _ = move_host(gen.config2(systems, seed=seed, n_min=2, n_max=abi.MAX_BODIES), np.random.default_rng(seed))
    spec.system["coordinates"][:] = coords
    steps = np.where(np.arange(systems) % 5 == 3, np.arange(systems) % 17, 1000)
    spec.system["time_limit"][:] = (steps + 1.5) * spec.system["time_step"]
    hit = int(np.argmax(spec.n_per_system() >= 3))
    b0, b1 = spec.body_offset[hit:hit + 2]
    planets = [b for b in range(b0, b1) if b != b0 + np.argmax(spec.body["mass"][b0:b1])]
    for k in ("position", "velocity"):                   # inside the planets' radii
        spec.body[k][planets[1]] = spec.body[k][planets[0]] + 1e-6
    spec.system["historic_snapshot_period"][:] = 3.3 * spec.system["time_step"]
    return spec


@pytest.mark.parametrize("coords", [abi.COORD_DEMOCRATIC_HELIOCENTRIC, abi.COORD_JACOBI])
@pytest.mark.parametrize("per_cu,more", EDGES)
def test_team_sizes_against_oracle(oracle, per_cu, more, coords):
    from posidonius_amd.ensemble import Ensemble
    systems, steps = edge(per_cu, more), 40
    spec = ensemble(systems, coords, 71)
    print(f"{systems} sets of systems, coordinates {coords}", flush=True)
    ref = oracle.run(spec, steps, threads=THREADS)
    # 64 lanes per system: one set per system
    with Ensemble(spec, mapping="packed", group_size=64, steps_per_launch=16) as ens:
        ens.enable_history(16)
        ens.step(steps)
        out = ens.get_state()
        rec = ens.drain_history()
    assert_same_state(out, ref, where=f"{systems} sets")
    assert np.any(out["current_iteration"] < steps) and np.any(out["current_iteration"] == steps)
    assert np.count_nonzero(out["status"] & abi.STATUS_COLLISION)
    few = spec.subset(range(24))
    with Ensemble(few, mapping="plain") as ens:
        ens.enable_history(16)
        ens.step(steps)
        same = ens.drain_history()
    first = rec[rec["system"] < 24]
    assert len(first) == len(same)
    for k in rec.dtype.names:
        np.testing.assert_array_equal(first[k], same[k], err_msg=k)


@pytest.mark.parametrize("per_cu,more", [(2, 1), (4, 1)])
def test_adjoint_does_not_depend_on_the_team_size(per_cu, more):
    from posidonius_amd.ensemble import Ensemble
    spec = gen.config2(edge(per_cu, more), seed=5, n_min=2, n_max=4)
    spec.system["coordinates"][::3] = abi.COORD_JACOBI
    few = spec.subset(range(edge(1, 1)))      # the fewest that the same sweep serves
    w = np.random.default_rng(1).standard_normal((spec.n_bodies, 3))
    out = []
    for s in (spec, few):
        print(f"adjoint of {s.n_systems} systems", flush=True)
        with Ensemble(s, mapping="packed", group_size=64) as ens:
            ens.adjoint_record(20, 8)
            out.append((ens.get_state(("position", "velocity", "angular_momentum")),
                        ens.adjoint(position=w[:s.n_bodies], velocity=w[:s.n_bodies], angular_momentum=w[:s.n_bodies])))
    for a, b in zip(out[0], out[1]):
        for k in b:
            np.testing.assert_array_equal(a[k][:few.n_bodies], b[k], err_msg=k)


@pytest.mark.parametrize("coords,gr", [(abi.COORD_DEMOCRATIC_HELIOCENTRIC, abi.GR_KIDDER1995),
                                       (abi.COORD_WHDS, abi.GR_KIDDER1995),
                                       (abi.COORD_DEMOCRATIC_HELIOCENTRIC, abi.GR_NEWHALL1983)],
                         ids=["kidder", "whds", "newhall"])
@pytest.mark.parametrize("per_cu", [0, 2, 4])
def test_a_team_serves_set_after_set(per_cu, coords, gr):
    """With fewer workgroups than sets of systems, a team takes one set after
    another, some of systems that had stopped before the launch, in the same LDS
    and scratch memory: the bits of a workgroup per set."""
    from posidonius_amd.ensemble import Ensemble
    spec = ensemble(edge(per_cu, 20), coords, 73)
    spec.system["gr_implementation"][:] = gr
    out = []
    for grid in (0, 7):
        with Ensemble(spec, mapping="packed", group_size=64, steps_per_launch=4, persistent_grid=grid) as ens:
            ens.enable_history(16)
            ens.step(9)
            part = [ens.get_state(), ens.drain_history()]
            if gr == abi.GR_KIDDER1995:
                ens.adjoint_record(5, 2)
                w = np.ones((spec.n_bodies, 3))
                part += [ens.adjoint(position=w, velocity=w, angular_momentum=w), ens.get_state()]
            out.append(part)
    for a, b in zip(*out):
        for k in (a if isinstance(a, dict) else a.dtype.names):
            np.testing.assert_array_equal(a[k], b[k], err_msg=k)
