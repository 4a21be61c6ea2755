"""The statistical-equilibrium update at the edges of its register rows (8, 16, 32, 48 and 64
levels, one before and one after), against the oracle's long-double update from the same J
and Lambda: populations within 1e-10 relative plus 1e-14 of the species total, the oracle's
own accuracy on the badly scaled rate matrices of a rotor."""
import numpy as np
import pytest

from magritte_amd import _abi, models

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nlev", [2, 7, 8, 9, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64])
def test_update_at_row_edges(nlev):
    from magritte_amd import solver
    from oracle import oracle

    print(f"[stateq] {nlev} levels", flush=True)
    rng = np.random.Generator(np.random.PCG64(nlev))
    m = models.model_line_1d(npoints=7, nquads=3)
    ld = models.linedata_linear_rotor(57.6e9, 0.11, nlev)
    ld["colpar"] = [models.colpar_constant(ld, 0, 1.0e-16)]
    m.set_lines([ld], 3)
    m.finalize()
    m.temperature[:] = rng.uniform(10.0, 60.0, m.npoints)
    m.finalize()
    prm = _abi.default_nlte_params()
    dm = solver.DeviceModel(m)
    lp = solver.LevelPopulations(dm, prm)
    lp.set_lte()
    nl = oracle.NLTE(m, prm)
    nl.set_lte()
    nu = m.nu.reshape(m.npoints, m.nfreqs)
    J = 2.0 * models.HH * nu**3 / models.CC_SQUARED / np.expm1(models.HH * nu / (models.KB * 15.0))
    lam = np.zeros((m.npoints, m.nlines))
    import torch

    lp.stateq(torch.from_numpy(J).cuda(), torch.from_numpy(lam).cuda())
    nl.set_Jeff((J.reshape(m.npoints, m.nlines, 3) * m.quad_weights[0]).sum(axis=2), lam)
    nl.stateq(lam)
    pop, tot = lp.populations()
    got, ref = pop.cpu().numpy(), nl.populations()["population"]
    ptot = np.repeat(tot.cpu().numpy()[0], nlev)
    assert np.all(np.isfinite(got))
    assert np.all(np.abs(got - ref) <= 1e-10 * np.abs(ref) + 1e-14 * ptot), float(
        np.max(np.abs(got - ref) / (np.abs(ref) + 1e-4 * ptot)))


@pytest.mark.parametrize("nlev", [2, 5])
def test_pivots_whose_reciprocal_overflows(nlev):
    """Rates multiplied by one power of two have the same populations.  With some 1e-312 a
    pivot's quotients are numbers where its reciprocal is not; such a rate has about 37 bits
    (6e-12), a few of which are added up (1e-9).  The oracle's decomposition, as the
    reference's, takes a row that small for a dependent one, so the other rates' update is
    what it is compared with."""
    import torch

    from magritte_amd import solver

    print(f"[stateq] {nlev} levels, rates of 1e-312", flush=True)
    pops = []
    for scale in (1.0, 2.0**-1013):
        m = models.model_line_1d(npoints=7, nquads=3)
        ld = models.linedata_linear_rotor(57.6e9, 0.11, nlev)
        ld["colpar"] = [models.colpar_constant(ld, 0, 0.0)]
        for k in ("A", "Bs", "Ba"):
            ld[k] = ld[k] * scale
        m.set_lines([ld], 3)
        m.finalize()
        lp = solver.LevelPopulations(solver.DeviceModel(m))
        lp.set_lte()
        nu = m.nu.reshape(m.npoints, m.nfreqs)
        J = 2.0 * models.HH * nu**3 / models.CC_SQUARED / np.expm1(models.HH * nu / (models.KB * 15.0))
        lp.stateq(torch.from_numpy(J).cuda(), torch.zeros((m.npoints, m.nlines), dtype=torch.float64).cuda())
        pops.append(lp.populations()[0].cpu().numpy())
    assert np.all(pops[0] > 0)
    np.testing.assert_allclose(pops[1], pops[0], rtol=1e-9)
