"""The staged sweeps of the formal solves at their edges, against the oracle: rays whose
entries end on, one before and one after a chunk of staged entries, quadratures around a
half-wave's 32 lanes, an odd and an even number of lines, windows with more lines than a
group takes side by side, interpolated entries across chunks, and ray pairs split over
waves or not.  FP64 mode differs from the oracle by a few roundings per row (1e-10
relative, as the other parity tests)."""
import numpy as np
import pytest

from magritte_amd import _abi, models

pytestmark = pytest.mark.gpu


def _check(m, op):
    from magritte_amd import solver
    from oracle import oracle

    out = solver.feautrier_forward(solver.DeviceModel(m), op)
    u, J, lam = (out[k].cpu().numpy() for k in ("u", "J", "lambda_diag"))
    for name, a, b in zip(("u", "J", "lambda"), (u, J, lam), oracle.solve(m, op)):
        assert np.all(np.isfinite(a)), name
        err = float(np.max(np.abs(a - b) / np.maximum(np.abs(b), 1e-300)))
        assert err < 1e-10, f"{name}: {err:.2e}"


@pytest.mark.parametrize("npoints", [2, 3, 31, 32, 33, 34, 63, 64, 95])
@pytest.mark.parametrize("nquads", [1, 31, 32, 33, 65])
def test_chunk_and_half_wave_edges(npoints, nquads):
    print(f"[staged] line {npoints} points {nquads} bins", flush=True)
    m = models.model_line_1d(npoints=npoints, nquads=nquads)
    _check(m, m.options())


@pytest.mark.parametrize("approx", [_abi.APPROX_NONE, _abi.APPROX_ONE_LINE, _abi.APPROX_CLOSE_LINES])
@pytest.mark.parametrize("nlines", [1, 2, 5, 17])
def test_blended_windows(approx, nlines):
    """lines a width or two apart: more than 16 of them go through two rounds of a window"""
    print(f"[staged] {nlines} blended lines approx {approx}", flush=True)
    clumps = np.exp(0.5 * np.random.Generator(np.random.PCG64(5)).standard_normal(5**3))
    m = models.model_wind(n_edge=5, nrays=12, nquads=7, clumps=clumps, v_out=1.5e3)
    ld = models.linedata_blended(115.0e9, [1.5e-6 * (k + 1) for k in range(nlines - 1)], A=1.0e-7)
    m.set_lines([ld], 7)
    m.finalize()
    _check(m, m.options(approx=approx))


def test_interpolated_entries_across_chunks():
    """a clumpy wind with many interpolated entries: several chunks per half ray"""
    clumps = np.exp(2.0 * np.random.Generator(np.random.PCG64(6)).standard_normal(7**3))
    m = models.model_wind(n_edge=7, nrays=12, nquads=9, nlev=4, clumps=clumps)
    m.params["max_interpolation_diff"] = 1.02
    print("[staged] interpolated chunks", flush=True)
    _check(m, m.options())


@pytest.mark.parametrize("nrays", [12, 48])
def test_ray_pair_parts_and_their_workspace(nrays):
    """J from the ray pairs' parts and from the stored u, and once more after the kept
    buffers were given back: the same bits"""
    from magritte_amd import solver

    print(f"[staged] parts of {nrays} rays", flush=True)
    m = models.model_wind(n_edge=6, nrays=nrays, nquads=7)
    d, op = solver.DeviceModel(m), m.options()
    want = solver.feautrier_forward(d, op)
    parts = solver.feautrier_forward(d, op, with_u=False)
    _abi.lib().mgx_release_workspace()
    again = solver.feautrier_forward(d, op, with_u=False)
    for got in (parts, again):
        for k in ("J", "lambda_diag"):
            assert (got[k] == want[k]).all(), k


@pytest.mark.parametrize("n_edge,nrays", [(3, 12), (15, 48), (26, 12)])
def test_adjoint_ray_pair_items(n_edge, nrays):
    """the J adjoint takes one ray pair per item, five with a remainder of four, or an
    origin's six; the sums' order differs: 1e-9 relative, as the other gradient tests, and
    1e-10 of the largest where contributions of both signs cancel"""
    import torch

    from magritte_amd import solver
    from oracle import oracle

    print(f"[staged] adjoint items {n_edge}^3 {nrays} rays", flush=True)
    m = models.model_wind(n_edge=n_edge, nrays=nrays, nquads=7, nlev=2)
    op = m.options()
    J_bar = np.random.Generator(np.random.PCG64(7)).standard_normal((m.npoints, m.nfreqs))
    got = solver.feautrier_adjoint(solver.DeviceModel(m), op, torch.from_numpy(J_bar))
    for name, a, b in zip(("d_eps", "d_kap"), got, oracle.J_adjoint(m, op, J_bar)):
        a, b = np.asarray(a.cpu()), np.asarray(b)
        assert np.all(np.abs(a - b) <= 1e-9 * np.abs(b) + 1e-10 * np.abs(b).max()), name
