"""Phantoms with so many voxel planes that they do not fit in the LDS of an event
kernel beside its other tables: the dose is the one of a counting run, whose
kernels read every table from device memory, up to the order of its FP64 sums
(at most 1e-10 for the counts here), and the electron bins are staged wherever
they fit beside the planes that are."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

omc = pytest.importorskip("ompmc_amd")
P = omc.phantoms

FIVE = [P.WATER, P.LUNG, P.BONE, P.AIR, "PMMA521ICRU"]


def _thin(media, nz):
    """A column of nz thin voxels, the media in turn."""
    edge = np.array([-2.0, 2.0])
    med = (1 + np.arange(nz) * len(media) // nz).reshape(nz, 1, 1).astype(np.int32)
    rho = np.array([1.0, 0.26, 1.85, 0.0012, 1.19])[med - 1]
    return P.Phantom(media, edge, edge.copy(), np.arange(nz + 1) * (8.0 / nz), med, rho, "thin")


# planes staged and not (24 KiB), with five media beside the bins and without
# them (80 KiB)
@pytest.mark.parametrize("precision,media,nz,bins", [(omc.FP32, FIVE[:1], 5700, True), (omc.FP32, FIVE[:1], 6300, True),
                                                     (omc.FP32, FIVE, 4400, True), (omc.FP32, FIVE, 5500, False),
                                                     (omc.FP64, FIVE[:1], 2800, False),
                                                     (omc.FP64, FIVE[:1], 3200, False)])
@pytest.mark.parametrize("nsplit", [1, 4])
def test_planes_beyond_lds(precision, media, nz, bins, nsplit):
    ph_h = _thin(media, nz)
    c = omc.Context(media)
    ph = c.phantom(ph_h)
    kw = dict(collimator=(-1, 1, -1, 1), precision=precision, nsplit=nsplit, form=omc.FORM_EVENT, seed=31)
    a1, a2, sa = c.run_dosxyz(ph, omc.Spectrum.mono(3.0), 200, 4, **kw)
    b1, b2, sb = c.run_dosxyz(ph, omc.Spectrum.mono(3.0), 200, 4, count_events=1, **kw)
    c.close()
    assert sa.errors == 0 and sb.errors == 0 and b1.max() > 0
    assert np.allclose(a1, b1, rtol=1e-10, atol=1e-12 * b1.max())
    assert np.allclose(a2, b2, rtol=1e-10, atol=1e-12 * b2.max())
    assert (sa.lds_table_bytes > 0) == bins
