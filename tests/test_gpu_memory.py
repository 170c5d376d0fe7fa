"""Dose runs and phantoms where little device memory is free.  A run alone on its stream keeps
more particles in flight, in pools of 12.9 GB (FP32) or 17.2 GB (FP64), where
the memory holds them beside its batch tallies; where it does not, the run goes
through with smaller pools, and gives the same dose up to the order of its FP64
sums (at most 1e-10 for the counts here)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

omc = pytest.importorskip("ompmc_amd")
torch = pytest.importorskip("torch")
P = omc.phantoms


def _leave(nbytes):
    """Takes all device memory that can be allocated but `nbytes` of it (the
    runtime can have some GB more than it reports as free)."""
    gap = torch.empty(nbytes, dtype=torch.uint8, device="cuda:0")
    fill, n = [torch.empty(torch.cuda.mem_get_info()[0] - (4 << 30), dtype=torch.uint8, device="cuda:0")], 1 << 30
    while n >= 32 << 20:
        try:
            fill.append(torch.empty(n, dtype=torch.uint8, device="cuda:0"))
        except torch.OutOfMemoryError:
            n //= 2
    del gap
    torch.cuda.empty_cache()
    return fill


@pytest.mark.parametrize("precision,entry,beside", [(omc.FP32, 96, 300 << 20), (omc.FP64, 128, 300 << 20),
                                                    (omc.FP32, 96, -(1 << 30))],
                         ids=["pools_fit_alone_fp32", "pools_fit_alone_fp64", "pools_do_not_fit"])
def test_dose_run_with_little_free_memory(precision, entry, beside):
    ph = P.water_cube(200, 0.1)                          # 64 MB a tally array, twelve of them
    c = omc.Context(ph.media)
    gph = c.phantom(ph)
    target = torch.cuda.get_device_properties(0).multi_processor_count * 4096

    def run(**kw):
        s, s2, st = c.run_dosxyz(gph, omc.Spectrum.mono(4.0), 110_000, 10, collimator=(-1, 1, -1, 1), seed=3,
                                 precision=precision, **kw)
        assert st.errors == 0 and st.batches_per_job == 10
        return s, s2

    ref = run(event_target=target)
    omc.Context(ph.media).close()                        # gives the memory kept between runs back
    pools = 4 * 8 * 4 * target * entry                   # of four times the particles in flight
    fill = _leave(pools + beside)
    try:
        got = run()
        again = run()
    finally:
        del fill
        torch.cuda.empty_cache()
        c.close()
    for x in (got, again):
        for a, b in zip(x, ref):
            assert np.allclose(a, b, rtol=1e-10, atol=1e-12 * b.max())


def test_phantom_where_the_rest_is_kept_for_runs():
    """A phantom goes into memory that the library only keeps for later runs."""
    ph = P.water_cube(220, 0.1)                          # 310 MB on the device
    c = omc.Context(ph.media)
    small = c.phantom(P.water_cube(20, 0.5))
    c.run_dosxyz(small, omc.Spectrum.mono(2.0), 110_000, 10, collimator=(-1, 1, -1, 1),
                 event_target=torch.cuda.get_device_properties(0).multi_processor_count * 4096)
    fill = _leave(200 << 20)                             # 3.2 GB are kept
    try:
        c.phantom(ph).release()
    finally:
        del fill
        torch.cuda.empty_cache()
        c.close()
