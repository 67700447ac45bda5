"""Derived maps of few samples, a thread per row of samples below 16 (means), 8
(orientations, Bingham maps) and 4 (Watson maps), 16 lanes from there on: both
sides of each line at the edges of the blocks against the oracle, and means and
maps of a large volume within a few times a copy of what they read."""
import numpy as np
import pytest

from oracle import finish_ref as fr
from tests.helpers import dev, host
from tests.test_post_rows import _samples

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [1, 2, 3, 4, 7, 8, 15, 16])
@pytest.mark.parametrize("n", [1, 37, 255, 256, 257, 515])
def test_few_samples_match_oracle(n, S):
    import torch
    from cudimot_amd import capi
    x = _samples(n, S, 100 + 10 * S + n)
    d = dev(x)
    new = lambda *s: torch.full(s, -9.0, device="cuda")  # noqa: E731
    mean, fibre, disp, fan, maps, od = new(n, 7), new(n, 3), new(n), new(n, 3), new(n, 5), new(n, 1)
    capi.sample_mean(d, mean)
    capi.dyads(d, 4, 5, fibre, disp)
    capi.dyads(d, 4, 5, fan, None, psi=6)
    capi.noddi_maps(d, 2, maps, beta=3)
    capi.noddi_maps(d, 2, od)
    capi.sync()
    np.testing.assert_allclose(host(mean), fr.sample_mean(x), rtol=1e-6, atol=1e-7)
    for got, psi in ((fibre, None), (fan, 6)):
        want, wdisp = fr.dyads(x, 4, 5, psi)
        np.testing.assert_allclose(np.abs(np.sum(host(got) * want, axis=1)), 1.0, atol=2e-5)
        if psi is None:
            np.testing.assert_allclose(host(disp), wdisp, atol=2e-6)
    np.testing.assert_allclose(host(maps), fr.noddi_maps(x, 2, 3), rtol=2e-6, atol=1e-7)
    np.testing.assert_allclose(host(od)[:, 0], np.arctan(1.0 / x[:, 2].astype(np.float64).mean(1)) * 2 / np.pi, rtol=2e-6)


@pytest.mark.parametrize("S", [1, 4])
def test_few_samples_of_a_large_volume_take_a_few_copies(S):
    import torch
    from cudimot_amd import capi
    n = 1000000
    x = torch.rand((n, 7, S), device="cuda") + 0.5
    y, mean, maps = torch.empty_like(x), torch.empty((n, 7), device="cuda"), torch.empty((n, 5), device="cuda")
    s = torch.cuda.current_stream()

    def us(f):
        best = float("inf")
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            f()
            b.record()
            torch.cuda.synchronize()
            best = min(best, 1000 * a.elapsed_time(b))
        return best

    copy = us(lambda: y.copy_(x))
    assert us(lambda: capi.sample_mean(x, mean, stream=s)) < 3 * copy + 30
    assert us(lambda: capi.noddi_maps(x, 2, maps, beta=3, stream=s)) < 3 * copy + 30
