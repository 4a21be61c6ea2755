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


@pytest.mark.parametrize("n_edge,nrays", [(3, 12), (12, 12), (15, 48), (26, 12)])
def test_adjoint_ray_pair_items(n_edge, nrays):
    """the J adjoint takes one ray pair per item, half an origin's of one line, five with a
    remainder of four, or an origin's six; the sums' order differs: 1e-9 relative, as the other gradient tests, and
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


@pytest.mark.parametrize("nlines,separation", [(63, 1.5e-6), (64, 1.5e-6), (65, 1.5e-6), (130, 1.0e-5),
                                               (130, 1.0e-4)])
def test_windows_in_long_lists(nlines, separation):
    """lists around the length from which the windows' first line is searched for, windows
    with many, a few and one of their lines"""
    print(f"[staged] {nlines} lines {separation} apart", flush=True)
    m = models.model_wind(n_edge=4, nrays=12, nquads=3, v_out=1.5e3)
    m.set_lines([models.linedata_blended(115.0e9, [separation * (k + 1) for k in range(nlines - 1)], A=1.0e-7)], 3)
    m.finalize()
    _check(m, m.options())


def _two_species(n_edge=5):
    """blended lines of two species, the second one's below the first's: the lines are not in
    ascending order"""
    m = models.model_wind(n_edge=n_edge, nrays=12, nquads=5, v_out=1.5e3)
    a = models.linedata_blended(115.0e9, [2.0e-6, 5.0e-6], A=1.0e-7, num=1)
    b = models.linedata_blended(115.0e9 * (1 - 8.0e-6), [1.0e-6, 9.0e-6], A=1.0e-7, num=1)
    m.set_lines([a, b], 5)
    m.finalize()
    assert np.any(np.diff(m.line) < 0)
    return m


@pytest.mark.parametrize("approx", [_abi.APPROX_NONE, _abi.APPROX_ONE_LINE, _abi.APPROX_CLOSE_LINES])
def test_lines_out_of_order(approx):
    import torch

    from magritte_amd import solver
    from oracle import oracle

    print(f"[staged] two species, approx {approx}", flush=True)
    m = _two_species()
    op = m.options(approx=approx)
    _check(m, op)
    J_bar = np.random.Generator(np.random.PCG64(8)).standard_normal((m.npoints, m.nfreqs))
    got = solver.feautrier_adjoint(solver.DeviceModel(m), op, torch.from_numpy(J_bar))
    for name, a, b in zip(("d_eps", "d_kap"), got, oracle.J_adjoint(m, op, J_bar)):
        a, b = np.asarray(a.cpu()), np.asarray(b)
        assert np.all(np.abs(a - b) <= 1e-9 * np.abs(b) + 1e-10 * np.abs(b).max()), name


@pytest.mark.parametrize("kind", ["apart", "close", "two species"])
@pytest.mark.parametrize("nfreqs", [3, 31, 70])
@pytest.mark.parametrize("approx", [_abi.APPROX_NONE, _abi.APPROX_CLOSE_LINES])
def test_images_with_many_lines(kind, nfreqs, approx):
    """image bins whose windows lie apart (each takes its own lines) or close together (they
    share the group's): intensities, optical depths (1e-10) and gradients, the inverse
    widths' too (bars of their tests)"""
    import torch

    from magritte_amd import solver
    from oracle import oracle

    print(f"[staged] image {kind} {nfreqs} bins approx {approx}", flush=True)
    if kind == "two species":
        m = _two_species(6)
    else:
        m = models.model_wind(n_edge=6, nrays=12, nquads=3, v_out=1.5e3)
        m.set_lines([models.linedata_blended(115.0e9, [2.0e-6 * (k + 1) for k in range(79)], A=1.0e-7)], 3)
        m.finalize()
    half = 2.0e-6 if kind == "close" else 1.0e-4
    fr = m.image_frequencies(m.line[0] * (1 + 8.0e-5 - half), m.line[0] * (1 + 8.0e-5 + half), nfreqs)
    if kind == "two species":
        fr = m.image_frequencies(m.line[0] * (1 - 1.0e-4), m.line[0] * (1 + 1.0e-4), nfreqs)
    rd, op, d = np.array([0.3, -0.5, 0.81]), m.options(approx=approx), solver.DeviceModel(m)
    for f_d, f_o in ((solver.image_new, oracle.image_new),
                     (solver.image_optical_depth_new, oracle.image_optical_depth_new)):
        got, want = f_d(d, op, rd, 9, 7, fr)[0].cpu().numpy(), f_o(m, op, rd, 9, 7, fr)[0]
        assert np.max(np.abs(got - want) / np.maximum(np.abs(want), 1e-300)) < 1e-10
    I_bar = np.random.Generator(np.random.PCG64(9)).standard_normal((63, nfreqs))
    got = solver.image_adjoint(d, op, rd, 9, 7, fr, torch.from_numpy(I_bar), want_iw=True)
    want = oracle.image_adjoint(m, op, rd, 9, 7, I_bar, fr, want_iw=True)
    for name, a, b, rel in zip(("d_eps", "d_kap", "d_iw"), got, want, (1e-9, 1e-9, 1e-6)):
        a, b = np.asarray(a.cpu()), np.asarray(b)
        assert np.all(np.abs(a - b) <= rel * np.abs(b) + 0.1 * rel * np.abs(b).max()), name


def test_workspace_is_given_back():
    """200 MB of parts are kept after a solve and given back on request"""
    import torch

    from magritte_amd import solver

    print("[staged] release", flush=True)
    m = models.model_wind(n_edge=16, nrays=48, nquads=31)
    d, op = solver.DeviceModel(m), m.options(precision=_abi.PREC_MIXED)
    solver.release_workspace()
    before = torch.cuda.mem_get_info()[0]
    J = torch.empty((m.npoints, m.nfreqs), dtype=torch.float64, device="cuda")
    out = {"u": None, "J": J, "lambda_diag": None}
    solver.feautrier_forward(d, op, out=out)
    parts = 8 * m.npoints * m.hnrays * m.nfreqs
    assert before - torch.cuda.mem_get_info()[0] >= parts
    solver.release_workspace()
    assert before - torch.cuda.mem_get_info()[0] < parts / 4
    want = J.clone()
    solver.feautrier_forward(d, op, out=out)
    assert (J == want).all()
