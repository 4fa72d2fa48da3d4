"""WHDS in the fixed-effect-set step under each team size, and the effects that
share terms among the evaluations of one implicit-midpoint solve (Anderson
1975, Newhall 1983, the disk): the oracle's bits, also where Newhall's
fixed-point test reads components (below 1e-30 AU/day^2) and where a component
is zero."""
import numpy as np
import pytest

from posidonius_amd import abi, generators as gen
from tests.spec_tools import move_host
from tests.test_gpu_parity import THREADS, assert_same_state
from tests.test_gpu_teams import EDGES, edge, ensemble

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_cu,more", EDGES)
def test_whds_team_sizes_against_oracle(oracle, per_cu, more):
    from posidonius_amd.ensemble import Ensemble
    systems, steps = edge(per_cu, more), 40
    spec = ensemble(systems, abi.COORD_WHDS, 72)
    print(f"{systems} sets of systems", flush=True)
    ref = oracle.run(spec, steps, threads=THREADS)
    with Ensemble(spec, mapping="packed", group_size=64, steps_per_launch=16) as ens:
        ens.step(steps)
        out = ens.get_state()
    assert_same_state(out, ref, where=f"WHDS {systems} sets")


@pytest.mark.parametrize("per_cu,more", [(2, 1), (4, 1)])
def test_whds_adjoint_does_not_depend_on_the_team_size(per_cu, more):
    from posidonius_amd.ensemble import Ensemble
    spec = gen.config2(edge(per_cu, more), seed=6, n_min=2, n_max=4)
    spec.system["coordinates"][:] = abi.COORD_WHDS
    few = spec.subset(range(edge(1, 1)))      # the fewest that the same sweep serves
    w = np.random.default_rng(2).standard_normal((spec.n_bodies, 3))
    out = []
    for s in (spec, few):
        print(f"WHDS adjoint of {s.n_systems} systems", flush=True)
        with Ensemble(s, mapping="packed", group_size=64) as ens:
            ens.adjoint_record(20, 8)
            out.append(ens.adjoint(position=w[:s.n_bodies], velocity=w[:s.n_bodies], angular_momentum=w[:s.n_bodies]))
    for k in out[1]:
        np.testing.assert_array_equal(out[0][k][:few.n_bodies], out[1][k], err_msg=k)


@pytest.mark.parametrize("plane", [1.0, 1e-24, 0.0], ids=["inclined", "nearly_planar", "planar"])
@pytest.mark.parametrize("coords", [abi.COORD_DEMOCRATIC_HELIOCENTRIC, abi.COORD_JACOBI, abi.COORD_WHDS])
@pytest.mark.parametrize("impl", [abi.GR_ANDERSON1975, abi.GR_NEWHALL1983])
def test_gr_solves_against_oracle(oracle, impl, coords, plane):
    """One body set of every size from 2 to 16, the host anywhere; out of the
    plane the components are as they are, tiny (Newhall's fixed point iterates)
    or zero."""
    from posidonius_amd.ensemble import Ensemble
    parts = [gen.config2(2, seed=100 + n, n_min=n, n_max=n) for n in range(2, abi.MAX_BODIES + 1)]
    spec, _ = move_host(parts[0].concat(parts), np.random.default_rng(8))
    for k in ("position", "velocity"):
        spec.body[k][:, 2] *= plane
    spec.system["coordinates"][:] = coords
    spec.system["gr_implementation"][:] = impl
    spec.system["effects"][:] &= ~np.uint32(abi.EFFECT_TIDES | abi.EFFECT_ROTATIONAL_FLATTENING)   # their torques leave the plane
    steps = 30
    print(f"GR {impl} coordinates {coords} plane {plane}", flush=True)
    ref = oracle.run(spec, steps, threads=THREADS)
    for mapping in ("packed", "plain"):
        with Ensemble(spec, mapping=mapping, steps_per_launch=16) as ens:
            ens.step(steps)
            out = ens.get_state()
        assert_same_state(out, ref, where=f"GR {impl} {coords} {plane} {mapping}")
    z = np.abs(out["position"][:, 2])
    assert np.all(np.isfinite(z))
    if plane < 1.:
        assert z.max() < 1e-20


@pytest.mark.parametrize("coords", [abi.COORD_DEMOCRATIC_HELIOCENTRIC, abi.COORD_JACOBI])
@pytest.mark.parametrize("more", [0, 1], ids=["teams", "single_wavefronts"])
def test_newhall_teams_against_oracle(oracle, more, coords):
    """As many sets of systems as the teams serve and one more: systems of 2 to
    16 bodies, some stopping on the way, one colliding in its first step, some
    launches with every system of a wavefront stopped."""
    from posidonius_amd.ensemble import Ensemble
    systems, steps = edge(1, more), 24
    spec = ensemble(systems, coords, 73)
    spec.system["gr_implementation"][:] = abi.GR_NEWHALL1983
    print(f"{systems} sets of systems, coordinates {coords}", flush=True)
    ref = oracle.run(spec, steps, threads=THREADS)
    with Ensemble(spec, mapping="packed", group_size=64, steps_per_launch=8) as ens:
        ens.step(steps)
        out = ens.get_state()
    assert_same_state(out, ref, where=f"Newhall {systems} sets")
