"""How particles are spread over wavefronts does not change a result.  A queue
smaller than the wavefronts the device holds at once gives each wavefront a
share of it, a larger one fills all 64 lanes; with one workgroup (grid=1, four
wavefronts) the same queue is a large one from 256 particles on.  The random
streams are keyed by history, so the dose is the same up to the order of its
FP64 sums: a region's sum of n terms carries a relative error of at most
n * 2^-53, 1e-10 for the counts here."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

omc = pytest.importorskip("ompmc_amd")
P = omc.phantoms


@pytest.fixture(scope="module")
def slab():
    ph = P.slab_phantom(32, 1.1)
    c = omc.Context(ph.media)
    yield c, c.phantom(ph)
    c.close()


@pytest.mark.parametrize("form", [omc.FORM_EVENT, omc.FORM_HISTORY], ids=["event", "history"])
@pytest.mark.parametrize("nsplit,charge", [(1, 0), (4, 0), (1, -1)], ids=["photons", "split", "electrons"])
@pytest.mark.parametrize("precision", [omc.FP32, omc.FP64], ids=["fp32", "fp64"])
def test_dose_independent_of_lane_share(slab, form, nsplit, charge, precision):
    c, ph = slab
    for nper in (1, 31, 32, 33, 128, 1025, 1500):     # two batches: queues of 2 .. 3000 primaries
        kw = dict(collimator=(-3, 3, -3, 3), charge=charge, nsplit=nsplit, precision=precision, form=form, seed=17)
        spread = c.run_dosxyz(ph, omc.Spectrum.mono(3.0), nper, 2, **kw)
        packed = c.run_dosxyz(ph, omc.Spectrum.mono(3.0), nper, 2, grid=1, **kw)
        assert spread[2].errors == 0 and packed[2].errors == 0
        for a, b in zip(spread[:2], packed[:2]):
            assert np.allclose(a, b, rtol=1e-10, atol=1e-12 * b.max()), nper


def test_vacuum_crossing_independent_of_yields():
    """An electron crosses a vacuum layer voxel by voxel; where the routine
    yields to the wave's refill does not change its track, also when the
    medium behind the layer is the one before it (the reference then goes on to
    an interaction)."""
    ph_h = P.vacuum_gap_phantom(12, 0.5)
    c = omc.Context(ph_h.media)
    ph = c.phantom(ph_h)
    kw = dict(collimator=(-1, 1, -1, 1), charge=-1, precision=omc.FP64, form=omc.FORM_EVENT, seed=23)
    ref = c.run_dosxyz(ph, omc.Spectrum.mono(6.0), 500, 2, electron_budget=1000, electron_turns=-1, **kw)[0]
    for opts in (dict(electron_budget=1), dict(electron_budget=3, electron_turns=1), dict()):
        a = c.run_dosxyz(ph, omc.Spectrum.mono(6.0), 500, 2, **opts, **kw)[0]
        assert np.allclose(a, ref, rtol=1e-10, atol=1e-12 * ref.max()), opts
    c.close()
