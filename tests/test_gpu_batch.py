"""Batched solves against the per-instance path on the same parameters and
against dense diagonalization.  Bars: E0 1e-10 relative; G(z) 1e-8 on a
Matsubara grid, both spin blocks.  An instance's own continued fractions run
through the batch kernels too, so the reference instances are solved with
lanczos_block 0: the host-driven recurrence, one fraction at a time, on the
sector's own product."""
import dataclasses
import math

import numpy as np
import pytest

from pyqcm_amd import qcm, workloads as W, _lib
from tests.dense_ref import dense_hamiltonian

pytestmark = pytest.mark.gpu

_label = [5000]
_models = set()


def _new_label():
    _label[0] += 1
    return _label[0]


@pytest.fixture(scope="module", autouse=True)
def _device():
    _lib.require_device()
    qcm.set_global_parameterC("Hamiltonian_format", "G")
    yield
    qcm.set_global_parameterC("GF_method", "L")


def _model(wl):
    name = "batch_" + wl.name
    if name not in _models:
        qcm.new_model(name, wl.n_sites, wl.n_bath)
        for op, (typ, el) in wl.operators.items():
            qcm.new_operator(name, op, typ, [(r + 1, c + 1, v) for (r, c, v) in el])
        _models.add(name)
    return name


def _dense_E0(wl, values):
    w = dataclasses.replace(wl, values=values)
    e0 = np.inf
    for sec in wl.sector.split("/"):
        N, S = qcm.sector_parse(sec)[:2]
        Nup, Ndw = (N + S) // 2, (N - S) // 2
        e0 = min(e0, np.linalg.eigvalsh(dense_hamiltonian(w.L, w.terms(), Nup, Ndw))[0])
    return e0


def _compare(wl, points, gf_method, z, dense=True):
    qcm.set_global_parameterC("GF_method", gf_method)
    name = _model(wl)
    single, batch = [], []
    for vals in points:
        la, lb = _new_label(), _new_label()
        qcm.new_model_instanceC(name, vals, wl.sector, la)
        qcm.new_model_instanceC(name, vals, wl.sector, lb)
        single.append(la)
        batch.append(lb)
    try:
        qcm.set_global_parameterC("lanczos_block", 0 if gf_method == "F" else 12)
        for la in single:
            qcm.ground_state_solve(la)
            qcm.Green_function_solveC(la)
    finally:
        qcm.set_global_parameterC("lanczos_block", 12)
    qcm.solve_batch(batch, green_function=True)
    for vals, la, lb in zip(points, single, batch):
        Ea, sa = qcm.ground_state_solve(la)
        Eb, sb = qcm.ground_state_solve(lb)
        assert abs(Ea - Eb) <= 1e-10 * abs(Ea), (vals, Ea, Eb)
        assert sa.split(":")[:3] == sb.split(":")[:3]
        if dense:
            Ed = _dense_E0(wl, vals)
            assert abs(Eb - Ed) <= 1e-10 * abs(Ed), (vals, Eb, Ed)
        for spin in (0, 1):
            Ga = qcm.Green_function_grid(z, spin_down=spin, label=la)
            Gb = qcm.Green_function_grid(z, spin_down=spin, label=lb)
            assert np.abs(Ga - Gb).max() < 1e-8, (vals, spin, np.abs(Ga - Gb).max())
    # all batched instances evaluated together equal their one-by-one evaluation
    for spin in (0, 1):
        Gs = qcm.Green_function_batch(z, batch, spin_down=spin)
        for lb, G in zip(batch, Gs):
            assert np.abs(G - qcm.Green_function_grid(z, spin_down=spin, label=lb)).max() < 1e-12
    for la, lb in zip(single, batch):
        qcm.erase_model_instance(la)
        qcm.erase_model_instance(lb)


def test_batch_2x2_neel_points_continued_fractions():
    _compare(W.vca_cluster(2, 2), W.vca_points(12, seed=4), "F", W.matsubara(32, 20.0))


def test_batch_2x3_neel_points_continued_fractions():
    _compare(W.vca_cluster(2, 3), W.vca_points(4, seed=5), "F", W.matsubara(32, 20.0))


def test_batch_ground_states_with_band_lanczos_green_functions():
    """GF_method 'L': batched ground states, band-Lanczos Green functions per instance."""
    _compare(W.vca_cluster(2, 2), W.vca_points(3, seed=6), "L", W.matsubara(32, 20.0))


@pytest.mark.parametrize("L,N,S,dim", [(2, 1, 1, 2), (4, 1, 1, 4), (5, 1, 1, 5), (3, 2, 0, 9), (5, 2, 2, 10),
                                       (4, 4, 0, 36), (5, 4, 0, 100), (6, 4, 0, 225)])
def test_ground_states_whose_krylov_space_ends_between_checks(L, N, S, dim):
    """Ritz pairs are found at each step in the one-wave workgroup, in the
    four-wave one every fourth and wherever the Krylov space may end: as many
    states as one, between one and two checks, and more."""
    wl = dataclasses.replace(W.hubbard_chain(L, U=4.0, mu=1.3), sector="R0:N%d:S%d" % (N, S))
    assert math.comb(L, (N + S) // 2) * math.comb(L, (N - S) // 2) == dim
    _compare(wl, [{"t": 1.0, "U": 4.0, "mu": 1.3}, {"t": 1.0, "U": 7.0, "mu": 2.2}], "F", W.matsubara(16, 20.0))


def test_lockstep_ground_states_beyond_the_steps_that_fit_in_lds():
    """3 100 Lanczos steps of a 4 900-state sector that may not converge (a stop
    bar below zero): the tridiagonal outgrows LDS at step 3 072 and the run ends
    as not converged at its own limit, with the batch usable afterwards."""
    wl = W.hubbard_chain(8, U=4.0, mu=2.0)
    name = _model(wl)
    label = _new_label()
    qcm.new_model_instanceC(name, wl.values, wl.sector, label)
    try:
        qcm.set_global_parameterC("max_iter_lanczos", 3100)
        qcm.set_global_parameterC("accur_lanczos", -1.0)
        with pytest.raises(_lib.EDError, match="exceeded 3100 iterations"):
            qcm.solve_batch([label], green_function=False)
    finally:
        qcm.set_global_parameterC("max_iter_lanczos", 1000)
        qcm.set_global_parameterC("accur_lanczos", 1e-12)
    qcm.solve_batch([label], green_function=False)
    E0 = qcm.ground_state_solve(label)[0]
    qcm.erase_model_instance(label)
    label = _new_label()
    qcm.new_model_instanceC(name, wl.values, wl.sector, label)
    assert abs(E0 - qcm.ground_state_solve(label)[0]) <= 1e-10 * abs(E0)
    qcm.erase_model_instance(label)


@pytest.mark.parametrize("steps", [1350, 5000])
def test_many_allowed_steps_change_nothing_in_small_sectors(steps):
    """Ground states of small sectors with more Lanczos steps allowed than their
    tridiagonal arrays fit beside them in LDS (1 350: in some sectors only): the
    energies and ground states are those of the default, to the last bit."""
    wl = W.vca_cluster(2, 2)
    wl6 = dataclasses.replace(W.hubbard_chain(6, U=4.0, mu=1.3), sector="R0:N6:S0/R0:N5:S1/R0:N2:S0/R0:N1:S1")
    out = []
    try:
        for n in (1000, steps):
            qcm.set_global_parameterC("max_iter_lanczos", n)
            got = []
            for w, pts in ((wl, W.vca_points(6, seed=9)), (wl6, [{"t": 1.0, "U": u, "mu": 1.0} for u in (2.0, 8.0)])):
                labels = [_new_label() for _ in pts]
                for lab, vals in zip(labels, pts):
                    qcm.new_model_instanceC(_model(w), vals, w.sector, lab)
                qcm.set_global_parameterC("GF_method", "F")
                qcm.solve_batch(labels, green_function=True)
                got += [qcm.ground_state_solve(lab)[0] for lab in labels]
                got += [qcm.Green_function_grid(W.matsubara(8, 20.0), label=lab) for lab in labels]
                for lab in labels:
                    qcm.erase_model_instance(lab)
            out.append(got)
    finally:
        qcm.set_global_parameterC("max_iter_lanczos", 1000)
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_batch_large_sector_four_wave_kernel():
    """A 10-site chain at half filling (dim 63 504; N +- 1 sectors 52 920): all
    items advance in lockstep, four rows of 252 to 210 states a thread."""
    wl = W.hubbard_chain(10, U=4.0, mu=2.0)
    _compare(wl, [{"t": 1.0, "U": 4.0, "mu": 2.0}, {"t": 1.0, "U": 6.0, "mu": 3.1}], "F", W.matsubara(16, 20.0),
             dense=False)


def test_batch_48400_state_sector_global_memory(oracle):
    """The 2x3 cluster with 6 bath orbitals at N = 6 (220 x 220 = 48 400
    states; the fractions run in the N +- 1 sectors of 14 520 and 108 900
    states): every item advances in lockstep with its vectors in memory.  E0
    against the oracle's Lanczos, E0 and G against the per-instance path."""
    wl = W.vca_cluster_bath(2, 3, 6)
    pts = [{**wl.values, **v} for v in W.vca_points(2, seed=4)]   # bath values kept
    _compare(wl, pts, "F", W.matsubara(16, 20.0), dense=False)
    for vals in pts:
        w = dataclasses.replace(wl, values=vals)
        M = oracle.Model(w.L, w.terms())
        x = np.random.default_rng(0).normal(size=M.dim(3, 3))
        E0r = M.lanczos_gs(3, 3, x)[0]
        lab = _new_label()
        qcm.new_model_instanceC(_model(wl), vals, wl.sector, lab)
        qcm.solve_batch([lab])
        E0 = qcm.ground_state_solve(lab)[0]
        assert abs(E0 - E0r) <= 1e-10 * abs(E0r), (vals, E0, E0r)
        qcm.erase_model_instance(lab)


def test_batch_mixed_formats_and_empty():
    """An empty batch is a no-op; instances built with the CSR format ('S')
    are solved one by one inside the same call, next to batched 'G' ones, and
    all agree with their own solves."""
    qcm.solve_batch([])
    qcm.set_global_parameterC("GF_method", "F")
    wl = W.vca_cluster(2, 2)
    name = _model(wl)
    pts = W.vca_points(4, seed=9)
    z = W.matsubara(16, 20.0)
    labs, refs = [], []
    for k, vals in enumerate(pts):
        qcm.set_global_parameterC("Hamiltonian_format", "S" if k % 2 else "G")
        la, lb = _new_label(), _new_label()
        qcm.new_model_instanceC(name, vals, wl.sector, la)
        qcm.new_model_instanceC(name, vals, wl.sector, lb)
        labs.append(la)
        refs.append(lb)
    qcm.set_global_parameterC("Hamiltonian_format", "G")
    qcm.solve_batch(labs)
    for la, lb in zip(labs, refs):
        Ea, _ = qcm.ground_state_solve(la)
        Eb, _ = qcm.ground_state_solve(lb)
        assert abs(Ea - Eb) <= 1e-10 * abs(Eb)
        for spin in (0, 1):
            Ga = qcm.Green_function_grid(z, spin_down=spin, label=la)
            Gb = qcm.Green_function_grid(z, spin_down=spin, label=lb)
            assert np.abs(Ga - Gb).max() < 1e-8
        qcm.erase_model_instance(la)
        qcm.erase_model_instance(lb)


@pytest.mark.parametrize("nx,ny,nb,N,S,npts", [(2, 2, 4, 8, 0, 1), (2, 2, 4, 7, -1, 5), (2, 2, 5, 8, 0, 2),
                                               (2, 3, 4, 6, 0, 2), (2, 2, 8, 4, 0, 3), (2, 2, 8, 6, 0, 1),
                                               (2, 1, 12, 7, 5, 1), (2, 1, 12, 7, -5, 2), (2, 1, 14, 7, 5, 1),
                                               (2, 1, 14, 7, -5, 1), (2, 1, 16, 8, 8, 1), (2, 1, 16, 8, -8, 1)])
def test_items_beyond_lds_match_single_solves(nx, ny, nb, N, S, npts):
    """Sectors too large for LDS advance in lockstep: shapes with several rows
    side by side (larger half basis up to 128 states), with four, two and one
    rows a thread (up to 2 048, 4 096 and 18 432 states) and with rows beyond
    LDS (43 758), each with either spin the larger half; one item and several
    per shape, ragged row counts, sectors on both sides of the 131 072 states
    from which items are spread over the XCDs.  Against the instance's own
    solve with lanczos_block 0 (the host-driven recurrence on the row product):
    E0 to 1e-11 relative, G on the Matsubara axis to 1e-8 (the fractions are 400
    steps without reorthogonalization, which drift apart on the real axis
    only)."""
    wl = W.vca_cluster_bath(nx, ny, nb, N=N)
    sector = "R0:N%d:S%d" % (N, S)
    name = "wide_%d%d%d_%d" % (nx, ny, nb, N)
    qcm.new_model(name, wl.n_sites, wl.n_bath)
    for op, (typ, el) in wl.operators.items():
        qcm.new_operator(name, op, typ, [(r + 1, c + 1, v) for (r, c, v) in el])
    z = W.matsubara(24, 12.0)
    qcm.set_global_parameterC("GF_method", "F")
    qcm.set_global_parameterC("hv_variant", 1)  # the single solves' product: the row kernel, for every shape
    try:
        pts = [{**wl.values, **v} for v in W.vca_points(npts, seed=11)]
        labs = list(range(30100, 30100 + npts))
        for lab, v in zip(labs, pts):
            qcm.new_model_instanceC(name, v, sector, lab)
        qcm.solve_batch(labs)
        for lab, v in zip(labs, pts):
            E = qcm.ground_state_solve(lab)[0]
            G = [qcm.Green_function_grid(z, s, lab) for s in (0, 1)]
            qcm.new_model_instanceC(name, v, sector, lab + 500)
            qcm.set_global_parameterC("lanczos_block", 0)
            E1 = qcm.ground_state_solve(lab + 500)[0]
            qcm.Green_function_solveC(lab + 500)
            qcm.set_global_parameterC("lanczos_block", 12)
            assert abs(E - E1) < 1e-11 * abs(E1)
            for s in (0, 1):
                assert np.abs(G[s] - qcm.Green_function_grid(z, s, lab + 500)).max() < 1e-8
            qcm.erase_model_instance(lab)
            qcm.erase_model_instance(lab + 500)
    finally:
        qcm.set_global_parameterC("lanczos_block", 12)
        qcm.set_global_parameterC("GF_method", "L")
        qcm.set_global_parameterC("hv_variant", 0)


@pytest.mark.parametrize("nb", [1, 13, 14, 15, 28])
def test_register_tiles_at_their_edges(nb):
    """Fractions whose halves have 3, 15, 16, 17 and 30 states (one up electron,
    so that adding a down one leads to an L x L sector): partial, full and
    two-tile register kernels against the host-driven recurrence
    (lanczos_block 0), which runs the row product; also the sectors around
    them (1 state, L, and L (L - 1) / 2 x 1).  Matsubara axis, 1e-9: the
    recurrences differ by rounding only."""
    wl = W.vca_cluster_bath(2, 1, nb, N=1)
    name = "tile_%d" % nb
    qcm.new_model(name, wl.n_sites, wl.n_bath)
    for op, (typ, el) in wl.operators.items():
        qcm.new_operator(name, op, typ, [(r + 1, c + 1, v) for (r, c, v) in el])
    z = W.matsubara(16, 8.0)
    vals = {**wl.values, "U": 5.0, "M": 0.3, "mu": 1.0}
    qcm.set_global_parameterC("GF_method", "F")
    qcm.set_global_parameterC("hv_variant", 1)
    try:
        for lab, block in ((30900, 12), (30901, 0)):
            qcm.set_global_parameterC("lanczos_block", block)
            qcm.new_model_instanceC(name, vals, "R0:N1:S1", lab)
            qcm.ground_state_solve(lab)
            qcm.Green_function_solveC(lab)
        for s in (0, 1):
            a, b = (qcm.Green_function_grid(z, s, lab) for lab in (30900, 30901))
            assert np.abs(a - b).max() < 1e-9
    finally:
        qcm.set_global_parameterC("lanczos_block", 12)
        qcm.set_global_parameterC("GF_method", "L")
        qcm.set_global_parameterC("hv_variant", 0)
        for lab in (30900, 30901):
            qcm.erase_model_instance(lab)


def test_tiles_at_once_and_shape_by_shape():
    """2x1 with 5 bath orbitals, halves of 1 to 21 states: a few points' register
    tiles go as one launch of the largest shape, many points' shape by shape and
    side by side.  A point's energy and Green function are the same to the last
    bit either way."""
    wl = W.vca_cluster_bath(2, 1, 5)
    name = _model(wl)
    pts = [{**wl.values, **v} for v in W.vca_points(400, seed=12)]
    z = W.real_axis(24)
    qcm.set_global_parameterC("GF_method", "F")
    out = []
    for which in (range(400), (0, 399)):
        labels = {k: _new_label() for k in which}
        for k, lab in labels.items():
            qcm.new_model_instanceC(name, pts[k], wl.sector, lab)
        qcm.solve_batch(list(labels.values()))
        out.append([(qcm.ground_state_solve(labels[k])[0],
                     *(qcm.Green_function_grid(z, spin_down=s, label=labels[k]) for s in (0, 1))) for k in (0, 399)])
        for lab in labels.values():
            qcm.erase_model_instance(lab)
    for a, b in zip(*out):
        for x, y in zip(a, b):
            assert np.array_equal(x, y)
