"""What the adjoint's tape holds of a segment: d depth / d opacity with all its bits, and a
depth that was raised to the smallest one (min_opacity times the length) known as such."""
import math

import numpy as np
import pytest

from magritte_amd import models

pytestmark = pytest.mark.gpu


def test_depth_derivative_keeps_every_bit():
    """Two points at rest, one line without emission, one bin at its centre, one segment whose
    depth (opposite opacities) does not depend on the profile: each point's opacity gradient
    is 0.5 a b rounded once, a = dz iw / sqrt(pi) and b the adjoint of the depth, which a
    width with a power of two as a gives."""
    import torch

    from magritte_amd import solver

    dz = 2.0**43
    m = models.model_line_1d(npoints=2, nquads=1, length=dz, vmax=0.0)
    m.dshift_max[:] = -1.0  # line-integrated at equal shifts
    m.emissivity[:] = 0.0
    m.opacity[:] = np.array([[1.0e-14], [-1.0e-14]])
    op = m.options()
    op.min_opacity = 2.0**-44  # a depth of one half
    op.max_interpolation_diff = 1.0e30
    assert m.nu[0, 0] == m.line[0]
    Jb = torch.zeros((2, 1), dtype=torch.float64)
    Jb[0, 0] = 1.0

    def gradient(iw):
        m.inverse_width[:] = iw
        return solver.feautrier_adjoint(solver.DeviceModel(m), op, Jb)[1].cpu().numpy().ravel()

    inv_sqrt_pi = 1.0 / math.sqrt(math.pi)
    power = 2.0 ** math.floor(math.log2(m.inverse_width[0, 0]))
    c = power / inv_sqrt_pi
    iw0 = [x for x in (math.nextafter(c, 0.0), c, math.nextafter(c, 1.0)) if x * inv_sqrt_pi == power][0]
    print("[tape] bits of the depth's derivative", flush=True)
    g0 = gradient(iw0)
    assert g0[0] == g0[1] != 0.0
    b = g0[0] / (0.5 * dz * power)  # exact
    for iw in c * np.random.default_rng(9).uniform(0.5, 2.0, 40):
        want = 0.5 * (dz * (float(iw) * inv_sqrt_pi)) * b
        assert (gradient(float(iw)) == want).all()


@pytest.mark.parametrize("nlines", [1, 3])
def test_gradient_of_clamped_depths(nlines):
    """inverted points between others: segments whose line-integrated depth lies below the
    smallest one, beside some above it; one line and three in a window, against the oracle
    (1e-9 relative, 1e-10 of the largest where signs cancel, as the other gradient tests)"""
    import torch

    from magritte_amd import solver
    from oracle import oracle

    print(f"[tape] clamped depths, {nlines} lines", flush=True)
    m = models.model_line_1d(npoints=60, nquads=7)
    if nlines > 1:
        ld = models.linedata_blended(115.0e9, [1.5e-6 * (k + 1) for k in range(nlines - 1)], A=1.0e-7)
        m.set_lines([ld], 7)
    m.params["max_width_fraction"] = 1.0e-3
    m.finalize()
    rng = np.random.default_rng(10)
    m.opacity *= rng.uniform(0.5, 1.5, m.opacity.shape)
    inverted = rng.random(m.npoints) < 0.4
    m.opacity[inverted] *= -0.2
    op = m.options()
    op.max_interpolation_diff = 1.0e30
    # as large as the depth of a weak segment at the line's centre
    op.min_opacity = 0.5 * float(np.median(np.abs(m.opacity) * m.inverse_width))
    Jb = rng.standard_normal((m.npoints, m.nfreqs))
    got = solver.feautrier_adjoint(solver.DeviceModel(m), op, torch.from_numpy(Jb))
    for name, a, b in zip(("d_eps", "d_kap"), got, oracle.J_adjoint(m, op, Jb)):
        a, b = a.cpu().numpy(), np.asarray(b)
        assert np.all(np.isfinite(b)) and np.abs(b).max() > 0
        bad = np.abs(a - b) > 1e-9 * np.abs(b) + 1e-10 * np.abs(b).max()
        assert not bad.any(), (name, float(np.max(np.abs(a - b)) / np.abs(b).max()))
