"""The recorded run's tapes: kept for the whole run where they fit the bound,
recomputed segment by segment from checkpoints where they do not."""
import numpy as np
import pytest

from posidonius_amd import generators as gen
from tests.test_gpu_teams import edge

pytestmark = pytest.mark.gpu

TAPE_ROW = 19 * 8                 # bytes of a body's tape row
BOUND = 1 << 30
SEGMENT = 36


def run(spec, steps, w):
    from posidonius_amd.ensemble import Ensemble
    with Ensemble(spec, mapping="packed") as ens:
        ens.adjoint_record(steps, SEGMENT)
        end = ens.get_state()
        first = ens.adjoint(position=w, velocity=w, angular_momentum=w)
        ens.step(3)               # the adjoint is of the recorded run whatever follows it
        again = ens.adjoint(position=w, velocity=w, angular_momentum=w)
        after = ens.get_state()
    for k in end:
        np.testing.assert_array_equal(end[k], after[k], err_msg=k)
    for k in first:
        np.testing.assert_array_equal(first[k], again[k], err_msg=k)
    return end, first


@pytest.mark.parametrize("prepared", [True, False])
def test_kept_and_recomputed_tapes(prepared):
    """The same systems in an ensemble whose tapes exceed the bound and in one
    whose tapes are kept, on either side of the sweeps' dispatch.  The one-kernel
    sweep gives the same bits; the prepared one starts its midpoint iterations
    afresh at each stretch, whose length depends on the ensemble: with some 100
    roundings a step, 10 N steps and orbits that amplify by less than 100 they
    agree to steps x 1e4 x 1.1e-16 of the largest component."""
    per_wave = 64 // 4
    systems = per_wave * edge(1, 0) if prepared else per_wave * edge(1, 56)
    few = systems // 8 if prepared else per_wave * edge(1, 7)
    spec = gen.config2(systems, seed=12, n_min=4, n_max=4)
    segments = BOUND // (TAPE_ROW * spec.n_bodies * (SEGMENT + 1)) + 1
    steps = segments * SEGMENT - 5
    kept = TAPE_ROW * few * 4 * (SEGMENT + 1) * segments
    assert kept <= BOUND < TAPE_ROW * spec.n_bodies * (SEGMENT + 1) * segments
    w = np.random.default_rng(4).standard_normal((spec.n_bodies, 3))
    print(f"{systems} systems, {segments} segments", flush=True)
    end, grad = run(spec, steps, w)
    sub = spec.subset(range(few))
    end1, grad1 = run(sub, steps, w[:sub.n_bodies])
    for k in ("position", "velocity", "angular_momentum"):
        np.testing.assert_array_equal(end[k][:sub.n_bodies], end1[k], err_msg=k)
    for k in grad:
        a, b = grad[k][:sub.n_bodies], grad1[k]
        assert np.all(np.isfinite(b))
        if prepared:
            assert np.abs(a - b).max() <= steps * 1e4 * 1.1e-16 * np.abs(b).max(), k
        else:
            np.testing.assert_array_equal(a, b, err_msg=k)


def test_recording_again_uses_the_new_run():
    """A second recording of the same length reuses the buffers of the first."""
    from posidonius_amd.ensemble import Ensemble
    spec = gen.config2(40, seed=3, n_min=2, n_max=6)
    w = np.random.default_rng(4).standard_normal((spec.n_bodies, 3))
    with Ensemble(spec, mapping="packed") as ens:
        ens.adjoint_record(20, 7)
        ens.adjoint(position=w)
        ens.adjoint_record(20, 7)
        second = ens.adjoint(position=w)
        ens.adjoint_record(9, 4)
        third = ens.adjoint(position=w)
    with Ensemble(spec, mapping="packed") as ens:
        ens.step(20)
        ens.adjoint_record(20, 7)
        np.testing.assert_array_equal(ens.adjoint(position=w)["position"], second["position"])
    with Ensemble(spec, mapping="packed") as ens:
        ens.step(40)
        ens.adjoint_record(9, 4)
        np.testing.assert_array_equal(ens.adjoint(position=w)["position"], third["position"])


@pytest.mark.parametrize("wind", [False, True], ids=["fixed_effect_set", "generic"])
def test_recording_takes_the_historic_snapshots_of_stepping(wind):
    """The recorded steps append the records that pos_step would; the adjoint
    appends none."""
    from posidonius_amd import abi
    from posidonius_amd.ensemble import Ensemble
    spec = gen.config2(30, seed=9, n_min=2, n_max=7)
    spec.system["historic_snapshot_period"][:] = 3.3 * spec.system["time_step"]
    if wind:
        spec.system["effects"][:] |= abi.EFFECT_WIND
    w = np.ones((spec.n_bodies, 3))
    got = []
    for record in (True, False):
        with Ensemble(spec, mapping="packed") as ens:
            ens.enable_history(16)
            if record:
                ens.adjoint_record(30, 11)
                ens.adjoint(position=w)
            else:
                ens.step(30)
            got.append((ens.drain_history(), ens.get_state()))
    assert len(got[0][0]) > 0
    for k in got[0][0].dtype.names:
        np.testing.assert_array_equal(got[0][0][k], got[1][0][k], err_msg=k)
    for k in got[0][1]:
        np.testing.assert_array_equal(got[0][1][k], got[1][1][k], err_msg=k)
