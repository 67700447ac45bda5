"""The single-precision intra-axonal signal of NODDI_Bingham against the saddle-point
formula in extended precision."""
import numpy as np
import pytest

from tests.helpers import dev, host
from tests.test_oracle_math import _hyp_saddle_ld

pytestmark = pytest.mark.gpu

DPAR = 1.7e-3


@pytest.mark.parametrize("kappa", [0.02, 1.0, 8.0, 63.0])
@pytest.mark.parametrize("share", [0.0, 0.4, 0.999])
def test_intra_axonal_signal_of_a_fan(kappa, share):
    """Angles, gradients and the local frame are single precision: their error
    (a few 1e-7 of a unit vector) moves the exponent by up to twice b Dpar times
    that, which the tolerance allows for; the saddle point itself is double."""
    import torch
    from cudimot_amd import capi
    rng = np.random.default_rng(int(1000 * share + kappa))
    b = np.repeat([5.0, 700.0, 3000.0], 12)
    g = rng.normal(size=(36, 3))
    g[::12], g[1::12], g[2::12] = [1, 0, 0], [0, 1, 0], [0, 0, 1]
    g /= np.linalg.norm(g, axis=1)[:, None]
    cfp = np.column_stack([g, b]).astype(np.float32)
    n = 6
    angles = rng.uniform([0.05, -3, -1.5], [3.0, 3, 1.5], size=(n, 3))
    p = np.column_stack([np.zeros(n), np.ones(n), np.full((n, 2), [kappa, share * kappa]), angles]).astype(np.float32)
    sig = torch.empty((n, 36), device="cuda")
    capi.Model("NODDI_Bingham").predicted_signal(dev(p.reshape(n, -1, 1)), dev(cfp), torch.ones((n, 1), device="cuda"), sig)
    capi.sync()
    q, c = p.astype(np.float64), cfp.astype(np.float64)
    for v in range(n):
        (st, sp, ss), (ct, cp, cs) = np.sin(q[v, 4:]), np.cos(q[v, 4:])
        mu = np.array([st * cp, st * sp, ct])
        fan = np.array([-cs * sp - ct * cp * ss, cp * cs - ct * sp * ss, st * ss])
        M = q[v, 3] * np.outer(fan, fan) + q[v, 2] * np.outer(mu, mu)
        F0 = _hyp_saddle_ld(-np.linalg.eigvalsh(M))
        want = [float(_hyp_saddle_ld(-np.linalg.eigvalsh(M - m[3] * DPAR * np.outer(m[:3], m[:3]))) / F0) for m in c]
        np.testing.assert_allclose(host(sig)[v], want, rtol=1e-5, atol=1e-7)
