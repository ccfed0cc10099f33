"""The order that the automatic tile choice takes a plasma species to be in: in
order when loaded so and after a sort, out of order after 500 steps without one.
1.64e6 particles at 10 per cell run on 4 x 4 tiles in order, 2 x 4 out of it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CR, CZ, PPC, D = 160, 1024, 10, 5e-4
ORDERED, UNORDERED = (4, 4), (2, 4)


def _sim():
    from pdp3_amd import capi

    sim = capi.Simulation(CR + 1, CZ + 1, CR * D, CZ * D, 0.5 * D / 3e8, precision=capi.PREC_FP32)
    sim.boundary_conditions()
    idx = sim.add_species(-1, 1.0, PPC * CR * CZ)
    sim.init_uniform(idx, 3, PPC, 1e12, 0, 1.0)
    return sim


def test_adjoint_replays_do_not_age():
    """The adjoint's replayed steps are no steps of the run: 300 steps and a
    gradient over 150 leave the species 450 steps old."""
    sim = _sim()
    sim.step(300)
    sim.adjoint_run(150, 50, 10, 0.2, 0.3)
    assert sim.species_tile(0) == ORDERED
    sim.step(51)
    assert sim.species_tile(0) == UNORDERED
    sim.sort()
    assert sim.species_tile(0) == ORDERED
    sim.close()


def test_ensemble_steps_age_and_sorts_renew():
    """Steps and sorts of an ensemble count as a single run's."""
    from pdp3_amd import capi

    for interval, want in ((0, UNORDERED), (100, ORDERED)):
        sims = [_sim(), _sim()]
        ens = capi.Ensemble(sims)
        ens.set_sort_interval(interval)
        ens.step(400)
        assert [s.species_tile(0) for s in sims] == [ORDERED, ORDERED]
        ens.step(101)
        ens.close()
        assert [s.species_tile(0) for s in sims] == [want, want]
        for s in sims:
            s.close()


def test_skipped_sort_does_not_renew():
    """A periodic sort that finds more runs than its record space is skipped:
    the species stays out of order until the next one, which has the room; so
    in a run of its own and in an ensemble."""
    from pdp3_amd import capi

    rng = np.random.default_rng(5)
    src = _sim()
    st = src.download(0)
    src.close()
    p = rng.permutation(len(st["r"]))
    for ensemble in (False, True):
        sim = _sim()
        sim.step(502)
        assert sim.species_tile(0) == UNORDERED
        sim.upload(0, **{k: st[k][p] for k in ("r", "z", "vr", "vphi", "vz", "w")}, alive=np.ones(len(p), np.uint8))
        run = capi.Ensemble([sim]) if ensemble else sim
        run.set_sort_interval(2)
        # the sort before the first step (the third of an ensemble) finds a run
        # for nearly every particle
        run.step(3 if ensemble else 1)
        assert sim.species_tile(0) == UNORDERED
        run.step(2)
        assert sim.species_tile(0) == ORDERED
        if ensemble:
            run.close()
        sim.close()
