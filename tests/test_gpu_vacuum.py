"""Electrons in vacuum layers: the step guard counts their passes there too, and
where the routine yields to the wave's refill does not change a track, whatever
media lie before, between and behind the layers."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

omc = pytest.importorskip("ompmc_amd")
P = omc.phantoms


def _layers(nxy, width, dz, layers):
    """Layers (voxels, medium, density) of dz each, across nxy x nxy voxels."""
    med = np.concatenate([np.full(n, m, np.int32) for n, m, _ in layers])
    rho = np.concatenate([np.full(n, r) for n, _, r in layers])
    one = np.ones((len(med), nxy, nxy))
    e = np.linspace(-width / 2, width / 2, nxy + 1)
    return P.Phantom([P.WATER, P.LUNG], e, e.copy(), np.arange(len(med) + 1) * dz,
                     (one * med[:, None, None]).astype(np.int32), one * rho[:, None, None], "layers")


def test_step_guard_counts_vacuum():
    """An electron that crosses 6000 vacuum voxels takes more than 3000 passes and
    is dropped with OMC_ERR_LIMIT (4), the kernels exiting normally; the same
    bound does not trip on 10 voxels."""
    kw = dict(collimator=(-1, 1, -1, 1), charge=-1, precision=omc.FP32, form=omc.FORM_EVENT, seed=7,
              electron_budget=2, electron_turns=1, max_particle_steps=3000)
    for n, trips in ((10, False), (6000, True)):
        ph_h = _layers(1, 40.0, 0.002, [(5, 1, 1.0), (n, 0, 0.0), (5, 1, 1.0)])
        c = omc.Context(ph_h.media)
        ph = c.phantom(ph_h)
        if trips:
            with pytest.raises(omc.EngineError) as ei:
                c.run_dosxyz(ph, omc.Spectrum.mono(6.0), 50, 2, **kw)
            assert ei.value.code == 4 and "progress" in str(ei.value)
        else:
            assert c.run_dosxyz(ph, omc.Spectrum.mono(6.0), 50, 2, **kw)[2].errors == 0
        c.close()


@pytest.mark.parametrize("precision", [omc.FP32, omc.FP64], ids=["fp32", "fp64"])
def test_tracks_independent_of_yields_in_vacuum(precision):
    ph_h = _layers(9, 4.5, 0.25, [(2, 1, 1.0), (4, 0, 0.0), (2, 2, 0.26), (4, 0, 0.0), (2, 2, 0.26), (3, 0, 0.0),
                                  (4, 1, 1.0)])
    c = omc.Context(ph_h.media)
    ph = c.phantom(ph_h)
    kw = dict(collimator=(-1, 1, -1, 1), charge=-1, precision=precision, form=omc.FORM_EVENT, seed=29)
    ref = c.run_dosxyz(ph, omc.Spectrum.mono(6.0), 500, 2, electron_budget=1000, electron_turns=-1, **kw)[0]
    for opts in (dict(electron_budget=1), dict(electron_budget=1, electron_turns=1),
                 dict(electron_budget=3, electron_turns=2), dict()):
        a = c.run_dosxyz(ph, omc.Spectrum.mono(6.0), 500, 2, **opts, **kw)[0]
        assert np.allclose(a, ref, rtol=1e-10, atol=1e-12 * ref.max()), opts
    c.close()
