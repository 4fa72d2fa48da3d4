"""The prepared reverse sweep (at most one set of systems per CU) against the
sweep in one kernel (more sets): the same systems' gradients, alone and among
enough copies of themselves to take the other path.  Both are the same linear
products in another order.  With about 100 roundings a step on the way, 24
steps and orbits that amplify by less than 100, they agree to
24 x 100 x 100 x 1.1e-16 = 3e-11 of a system's largest component."""
import numpy as np
import pytest

from posidonius_amd import abi, generators as gen
from posidonius_amd.case import EnsembleSpec
from tests.spec_tools import move_host
from tests.test_gpu_teams import edge

pytestmark = pytest.mark.gpu

RTOL = 3e-11
STEPS, SEGMENT = 24, 9     # the last segment is shorter


def sizes(counts, seed, coords):
    parts = [gen.config2(2, seed=seed + n, n_min=n, n_max=n) for n in counts]
    spec, _ = move_host(EnsembleSpec.concat(parts), np.random.default_rng(seed))
    spec.system["coordinates"][:] = coords
    return spec


def gradients(spec, w):
    from posidonius_amd.ensemble import Ensemble
    # 64 lanes per system: one set per system
    with Ensemble(spec, mapping="packed", group_size=64) as ens:
        ens.adjoint_record(STEPS, SEGMENT)
        return ens.adjoint(position=w[0], velocity=w[1], angular_momentum=w[2])


def compare(spec, where):
    w = np.random.default_rng(3).standard_normal((3, spec.n_bodies, 3))
    copies = -(-edge(1, 1) // spec.n_systems)
    print(f"{where}: {spec.n_systems} systems, {copies} copies", flush=True)
    got = gradients(spec, w)
    many = gradients(EnsembleSpec.concat([spec] * copies), np.tile(w, (1, copies, 1)))
    for k in got:
        a, b = got[k], many[k][:spec.n_bodies]
        assert np.all(np.isfinite(b))
        for s in range(spec.n_systems):
            i = slice(spec.body_offset[s], spec.body_offset[s + 1])
            scale = np.abs(b[i]).max()
            assert np.abs(a[i] - b[i]).max() <= RTOL * scale, (where, k, s)


@pytest.mark.parametrize("coords", [abi.COORD_DEMOCRATIC_HELIOCENTRIC, abi.COORD_JACOBI, abi.COORD_WHDS])
@pytest.mark.parametrize("counts", [(2, 3, 4), (5, 7, 8), (2, 9, 15, 16)], ids=["4_slots", "8_slots", "16_slots"])
def test_prepared_sweep_against_the_other(counts, coords):
    compare(sizes(counts, 40, coords), f"sizes {counts} coordinates {coords}")


def test_prepared_sweep_of_mixed_systems():
    """Coordinates mixed, spins not integrated in some, systems that stop on
    their way (one at the first step of a segment), wind on half of the stars."""
    spec = sizes((2, 3, 5, 6, 8), 60, abi.COORD_JACOBI)
    n = spec.n_systems
    spec.system["coordinates"][:] = np.arange(n) % 3
    spec.system["effects"][n // 2:] |= abi.EFFECT_WIND
    spec.system["effects"][3] = 0
    host = np.isin(np.arange(spec.n_bodies), [spec.body_offset[i] + np.argmax(spec.body["mass"][spec.body_offset[i]:spec.body_offset[i + 1]])
                                              for i in range(n)])
    spec.body["roles"] = np.where(host, spec.body["roles"] | abi.ROLE_WIND, spec.body["roles"]).astype(spec.body["roles"].dtype)
    spec.body["wind_k_factor"] = np.where(host, 4e-12, 0.)
    spec.body["wind_rotation_saturation"] = np.full(spec.n_bodies, 1.7592918860102842)
    stop = np.where(np.arange(n) % 4 == 1, 2 * np.arange(n) + 7, 1000)   # steps 9, 17, 25, ...
    spec.system["time_limit"][:] = (stop + 0.5) * spec.system["time_step"]
    compare(spec, "mixed")
