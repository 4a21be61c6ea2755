"""Gradients where a line's emissivity, or emissivity and opacity, is zero, against the
oracle (pinned there by finite differences, test_oracle_adjoint.py): within 1e-9 relative, or
1e-10 of the largest gradient where contributions of both signs cancel, as the other gradient
tests.  A source is an emissivity divided by an opacity, so no interpolated entries here:
a power of zero has no derivative."""
import numpy as np
import pytest

from magritte_amd import _abi, models

pytestmark = pytest.mark.gpu


def _options(m, **kw):
    op = m.options(**kw)
    op.max_interpolation_diff = 1.0e30
    return op


def _close(got, ref, what):
    got, ref = got.cpu().numpy(), np.asarray(ref)
    assert np.all(np.isfinite(got)), what
    assert np.abs(ref).max() > 0, what
    bad = np.abs(got - ref) > 1e-9 * np.abs(ref) + 1e-10 * np.abs(ref).max()
    assert not bad.any(), (what, float(np.max(np.abs(got - ref)) / np.abs(ref).max()))


def _model(kind):
    m = models.model_wind(n_edge=6, nrays=12, nquads=7, nlev=3)
    if kind == "blended":
        m = models.model_wind(n_edge=6, nrays=12, nquads=7, v_out=1.5e3)
        m.set_lines([models.linedata_blended(115.0e9, [1.5e-6, 3.0e-6], A=1.0e-7)], 7)
        m.finalize()
    if kind == "trapezoid":
        # bins within the lines' cores at every point: in a wing an opacity's gradient beside an
        # empty point is rounding, as between two of them
        m = models.model_wind(n_edge=6, nrays=12, nquads=3, nlev=3, v_out=50.0)
        m.params["max_width_fraction"] = 1.0e6
        m.finalize()
    return m


def _darken(m, what):
    """no two of the points are neighbours: between two empty ones a segment has next to no
    depth, and the opacity's gradient there is rounding (it goes like eps / depth^2)"""
    some, taken = [], set()
    for p in np.random.default_rng(5).permutation(m.npoints)[:60]:
        if p not in taken:
            some.append(p)
            n0 = m.cum_n_neighbors[p]
            taken.update(m.neighbors[n0:n0 + m.n_neighbors[p]])
    if what == "dark everywhere":
        m.emissivity[:] = 0.0
    else:
        m.emissivity[some] = 0.0
    if what == "empty points":
        m.opacity[some] = 0.0


CASES = [("wind", "dark points"), ("wind", "dark everywhere"), ("blended", "dark points"),
         ("blended", "dark everywhere"), ("trapezoid", "dark everywhere"), ("trapezoid", "empty points")]


@pytest.mark.parametrize("approx", [_abi.APPROX_CLOSE_LINES, _abi.APPROX_NONE, _abi.APPROX_ONE_LINE])
@pytest.mark.parametrize("kind,what", CASES)
def test_J_gradient(kind, what, approx):
    import torch

    from magritte_amd import solver
    from oracle import oracle

    print(f"[zeros] J {kind} {what} approx {approx}", flush=True)
    m = _model(kind)
    _darken(m, what)
    op = _options(m, approx=approx)
    Jb = np.random.default_rng(6).standard_normal((m.npoints, m.nfreqs))
    got = solver.feautrier_adjoint(solver.DeviceModel(m), op, torch.from_numpy(Jb), want_iw=True)
    for name, a, b in zip(("d_eps", "d_kap"), got, oracle.J_adjoint(m, op, Jb)):
        _close(a, b, name)
    assert np.all(np.isfinite(got[2].cpu().numpy()))


@pytest.mark.parametrize("kind,what", CASES)
def test_image_gradient(kind, what):
    import torch

    from magritte_amd import solver
    from oracle import oracle

    print(f"[zeros] image {kind} {what}", flush=True)
    m = _model(kind)
    _darken(m, what)
    op = _options(m)
    fr = m.image_frequencies(m.line[0] * (1 - 2e-5), m.line[0] * (1 + 2e-5), 31)
    rd = np.array([0.3, -0.5, 0.81])
    Ib = np.random.default_rng(7).standard_normal((12 * 11, 31))
    got = solver.image_adjoint(solver.DeviceModel(m), op, rd, 12, 11, fr, torch.from_numpy(Ib))
    for name, a, b in zip(("d_eps", "d_kap"), got, oracle.image_adjoint(m, op, rd, 12, 11, Ib, fr)):
        _close(a, b, name)
