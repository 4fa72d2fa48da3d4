"""The early end of the eccentric anomaly's Newton iteration gives the last
iterate's bits, also where iterates alternate or the count is not a multiple of
the look's."""
import pytest
import torch

from posidonius_amd.differentiable import _eccentric_anomaly


@pytest.mark.parametrize("iterations", [1, 7, 8, 9, 59, 60])
@pytest.mark.parametrize("ecc", [0.0, 0.1, 0.9, 0.99])
@pytest.mark.parametrize("n", [1, 300, 20000])
def test_early_end_is_the_last_iterate(n, ecc, iterations):
    rng = torch.Generator().manual_seed(n)
    e = ecc * torch.rand(n, dtype=torch.float64, generator=rng)
    M = 14 * torch.rand(n, dtype=torch.float64, generator=rng) - 7
    E = M.clone()
    for _ in range(iterations):
        E = E - (E - e * torch.sin(E) - M) / (1.0 - e * torch.cos(E))
    got = _eccentric_anomaly(e, M, iterations)
    assert torch.equal(got.view(torch.int64), E.view(torch.int64))
    stacked = torch.func.vmap(lambda m: _eccentric_anomaly(e, m, iterations))(torch.stack([M, M]))
    assert torch.equal(stacked[1], E)


def test_a_trace_holds_every_iteration():
    """A traced call serves other inputs than it was traced with: where the
    iteration ends for those must not be in the trace."""
    from posidonius_amd import differentiable, generators as gen
    spec = gen.config2(200, seed=3, n_min=3, n_max=9)
    a = torch.tensor(spec.elements["a"])

    def state(a, e):
        return differentiable.state_from_elements(spec, a, e)

    traced = torch.jit.trace(state, (a, torch.full_like(a, 0.01)), check_trace=False)
    e = torch.full_like(a, 0.9999)
    for got, want in zip(traced(a, e), state(a, e)):
        assert torch.equal(got, want)
