"""Runs of different sizes share the device memory kept between them: blocks are
cut from larger ones and joined again, and no run sees another's bytes.  Every
run is repeated between runs of other sizes, and beside them in a server's
threads, and gives the dose of its first pass up to the order of its FP64 sums
(at most 1e-10 for the counts here)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

omc = pytest.importorskip("ompmc_amd")
P = omc.phantoms


def test_runs_of_different_sizes_share_memory():
    spec = omc.Spectrum.mono(4.0)
    cts = [P.synthetic_ct(nx=n, ny=n, nz=n - 8, vx=0.4, vy=0.4, vz=0.4, target_radius=1.0) for n in (24, 40, 64)]
    c = omc.Context(cts[0].media)
    gph = [c.phantom(p) for p in cts]
    bix = P.beamlets(nbeams=2, radius=1.2, hist_median=400, hist_range=(200, 800), seed=3)

    def dose(k, **kw):
        s, s2, st = c.run_dosxyz(gph[k], spec, 1500, 4, collimator=(-1, 1, -1, 1), seed=5 + k, **kw)
        assert st.errors == 0
        return [s, s2]

    def dij(k, **kw):
        (jc, ir, val), (_, _, var), _, _ = c.run_dij(gph[k], spec, bix, nbatch=4, want_var=True, seed=9 + k, **kw)
        return [jc, ir, val, var]

    runs = [lambda: dose(0), lambda: dij(2, hbm_budget=6 << 30), lambda: dose(2, event_target=1 << 19),
            lambda: dij(1, group=7, streams=3), lambda: dose(1, precision=omc.FP64), lambda: dij(0, precision=omc.FP64)]
    ref = [r() for r in runs]
    order = [3, 0, 1, 5, 2, 4, 1, 3, 2, 0, 4, 5, 5, 0]

    def check(i, got):
        for a, b in zip(got, ref[i]):
            if a.dtype.kind == "i":
                assert np.array_equal(a, b), i
            else:
                assert np.allclose(a, b, rtol=1e-10, atol=1e-12 * np.abs(b).max()), i

    for i in order:
        check(i, runs[i]())
    srv = omc.Server(c, max_inflight=4)
    ids = [(k, srv.submit_dose(cts[k], spec, 1500, 4, collimator=(-1, 1, -1, 1), seed=5 + k)) for k in (0, 2, 2, 0)]
    for i in (1, 4, 3):                    # on the context's stream, beside the server's
        check(i, runs[i]())
    for k, i in ids:
        r = srv.wait(i)
        assert r["error"] == 0
        check(0 if k == 0 else 2, [r["sum"], r["sum2"]])
    srv.close()
    c.close()
