"""The fused batch statistics and finish of a Dij group at the batch counts where
its marks are read differently: one, several and 64 beamlets a read, a beamlet
that fills one read exactly, needs two, or leaves a remainder.  The device
matrix equals the oracle's bit for bit (the fused kernel takes the reference's
order of operations)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

omc = pytest.importorskip("ompmc_amd")
B = pytest.importorskip("oracle.bindings")
P = omc.phantoms

from tests import test_gpu_dij_assemble as base  # noqa: E402


@pytest.mark.parametrize("nbatch", [2, 3, 21, 32, 33, 63, 64, 65, 130, 255])
def test_fold_bitwise_at_batch_counts(nbatch):
    rng = np.random.default_rng(nbatch)
    nx, ny, nz = 7, 5, 9                                # 316 regions: four whole tiles and a remainder
    nbix = 9
    ctx = omc.Context([P.WATER])
    ph = base._phantom(nx, ny, nz, rng.uniform(0.03, 1.2, nx * ny * nz))
    e = base._tallies(rng, nbix, nbatch, nx * ny * nz + 1, fill=0.1)
    e[4] = 0.0                                          # a beamlet without energy
    nper = rng.integers(1, 50, nbix)
    o = B.matrad_dij(ph, e, nper, nbatch, 1e-3)
    g, st = base._run(ctx, ph, e, nper, 1e-3)
    ctx.close()
    assert st.batches_per_job == nbatch                 # the fused path
    for a, b, what in zip(g, o, ("jc", "ir", "val", "var")):
        assert a.dtype == b.dtype and np.array_equal(a, b), what
