"""pqb_sample_photons, the photon loop on the GPU, against the step-by-step loop of the
strategy on the same entering photons and draws: the same samples.  Photon counts around
the step where the column-minors sweep takes over (12), mode counts around a wave and
around the size kept in LDS (1024), bunched inputs, samples of different photon counts."""

import numpy as np
import pytest

from piquassoboost_amd.sampling.simulation_strategies.GeneralizedCliffordsSimulationStrategy import (
    GeneralizedCliffordsBSimulationStrategy,
)

pytestmark = pytest.mark.gpu


def case(modes, counts, seed, bunched):
    rng = np.random.default_rng(seed)
    U = (rng.standard_normal((modes, modes)) + 1j * rng.standard_normal((modes, modes))) / np.sqrt(2 * modes)
    most = max(counts)
    pool = rng.choice(modes, size=min(modes, max(1, most // 2 if bunched else most)), replace=False)
    entering = rng.choice(pool, size=(len(counts), most))
    if not bunched and modes >= most:
        entering = np.stack([rng.permutation(pool)[:most] for _ in counts])
    return U, entering, rng.uniform(size=(len(counts), most))


@pytest.mark.parametrize("modes,counts,bunched", [
    (1, [3], True),
    (2, [1, 0, 2], True),
    (5, [2, 4, 1, 5], True),
    (24, [12, 11, 12], False),
    (64, [13, 12, 0, 14], False),
    (65, [13], True),
    (130, [17, 3, 13], False),
    (1024, [14, 12], False),
    (1025, [14, 12, 13], False),
    (40, [20] * 5, True),
])
def test_samples_of_the_step_by_step_loop(modes, counts, bunched):
    from piquassoboost_amd import _capi as C

    U, entering, draws = case(modes, counts, 900 + modes, bunched)
    got = C.sample_photons(U, counts, entering, draws)
    assert got.sum(axis=1).tolist() == list(counts)
    ref = GeneralizedCliffordsBSimulationStrategy(U, 1)._simulate_lockstep(
        modes, [entering[s][:c].tolist() for s, c in enumerate(counts)],
        [draws[s][:c].tolist() for s, c in enumerate(counts)])
    for s in range(len(counts)):
        assert np.array_equal(got[s], ref[s]), s


def test_no_weight_and_extreme_draws():
    from piquassoboost_amd import _capi as C

    U, entering, draws = case(6, [4, 4], 3, False)
    # a draw of 0 falls on the first mode, whatever its weight
    assert np.array_equal(C.sample_photons(U, [4], entering[:1], np.zeros((1, 4)))[0], [4, 0, 0, 0, 0, 0])
    # no mode has a weight, or every weight is NaN: the first mode
    for v in (0.0, np.nan):
        got = C.sample_photons(np.full_like(U, v), [4, 4], entering, draws)
        assert got.tolist() == [[4, 0, 0, 0, 0, 0]] * 2


def test_arguments():
    from piquassoboost_amd import _capi as C

    U, entering, draws = case(6, [4], 4, False)
    for bad in ([5], [-1]):
        with pytest.raises(C.EngineError):
            C.sample_photons(U, bad, entering, draws)
    with pytest.raises(C.EngineError):
        C.sample_photons(U, [4], entering + 6, draws)
    with pytest.raises(C.EngineError):
        C.sample_photons(U, [41], np.zeros((1, 41)), np.zeros((1, 41)))
    assert C.sample_photons(U, [0], entering, draws).tolist() == [[0] * 6]
