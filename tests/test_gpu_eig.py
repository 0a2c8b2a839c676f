"""The chi-truncation's one-sided Jacobi at the edges of its sizes and ranks.

Column counts n = 2 chi around 8 (one wave), 64 and 128 (the one-block limits)
and up to 800 (spread over the chip), with Gram matrices of full rank, of fewer
rows than columns, and with clusters of equal eigenvalues.
"""

import numpy as np
import pytest
import torch

from oracle import qmprs_oracle as O

pytestmark = pytest.mark.gpu


def _engine():
    from qmprs_amd import engine
    return engine


@pytest.mark.parametrize("n,chi", [(6, 1), (7, 2), (8, 3), (8, 4), (9, 5), (11, 31), (11, 32), (12, 33), (13, 63),
                                   (14, 64)])
@pytest.mark.parametrize("kind", ["uniform", "mps"])
def test_truncation_edges(gpu, n, chi, kind):
    """Targets to 1e-10 and spectra to 1e-12 of the largest eigenvalue (the
    suite's bars for the truncation): a batch of three states, of which the
    oracle truncates each by itself."""
    eng = _engine()
    svs = [O.random_uniform_state(n, s) if kind == "uniform" else O.random_mps_state(n, max(2, chi + chi // 2), s)
           for s in (1, 2, 3)]
    _, target, spec = eng.chi_truncate(eng.as_device_states(np.stack(svs)), chi, spectra=True)
    _, plain, _ = eng.chi_truncate(eng.as_device_states(np.stack(svs)), chi)
    for k, sv in enumerate(svs):
        ref, ref_spec = O.chi_truncate(O.ket(sv), n, chi)
        for got in (target, plain):
            err = np.linalg.norm(got[k].cpu().numpy() - ref) / np.linalg.norm(ref)
            print(f"n={n} chi={chi} {kind} state {k} rel.err {err:.2e}")
            assert err < 1e-10
        for i, lam in enumerate(ref_spec):
            if lam is not None:
                kk = min(len(lam), chi)
                assert np.max(np.abs(spec[k, i, :kk].cpu().numpy() - lam[:kk])) < 1e-12 * lam[0]


@pytest.mark.parametrize("pairs,chi", [(4, 16), (5, 32), (6, 64)])
def test_equal_eigenvalues(gpu, pairs, chi):
    """Bell pairs across the centre plus noise below the cutoff: 2^pairs equal
    eigenvalues at the middle bond, all kept, so the truncation returns the
    state (the cutoff of 1e-10 drops at most that weight at each of the bonds;
    the noise has 1e-16)."""
    eng = _engine()
    n = 2 * pairs
    psi = np.zeros((2 ** pairs, 2 ** pairs), dtype=np.complex128)
    psi[np.arange(2 ** pairs), np.arange(2 ** pairs)] = 2.0 ** (-pairs / 2)
    rng = np.random.default_rng(pairs)
    noise = rng.standard_normal(psi.shape) + 1j * rng.standard_normal(psi.shape)
    psi = O.ket((psi + 1e-8 * noise / np.linalg.norm(noise)).reshape(-1))
    wide = np.kron(psi, np.array([1.0, 1.0]) / np.sqrt(2.0))   # one more site: bonds above chi columns
    for sv, m in ((psi, n), (wide, n + 1)):
        _, target, _ = eng.chi_truncate(eng.as_device_states(sv), chi)
        assert np.linalg.norm(target[0].cpu().numpy() - sv) < 1e-7, m


@pytest.mark.parametrize("n,chi,kind", [(14, 65, "uniform"), (14, 65, "mps"), (15, 100, "mps"), (16, 128, "uniform"),
                                        (16, 129, "uniform"), (17, 200, "mps"), (17, 256, "uniform"),
                                        (17, 257, "mps"), (19, 400, "uniform")])
def test_truncation_above_128_columns(gpu, n, chi, kind):
    """130 to 800 columns, one to four rows per lane, Gram matrices of full
    rank and of fewer rows than columns; same bars as above."""
    eng = _engine()
    seeds = (1, 2) if n < 17 else (1,)
    svs = [O.random_uniform_state(n, s) if kind == "uniform" else O.random_mps_state(n, chi + chi // 2, s)
           for s in seeds]
    _, target, spec = eng.chi_truncate(eng.as_device_states(np.stack(svs)), chi, spectra=True)
    _, plain, _ = eng.chi_truncate(eng.as_device_states(np.stack(svs)), chi)
    for k, sv in enumerate(svs):
        ref, ref_spec = O.chi_truncate(O.ket(sv), n, chi)
        for got in (target, plain):
            err = np.linalg.norm(got[k].cpu().numpy() - ref) / np.linalg.norm(ref)
            print(f"n={n} chi={chi} {kind} state {k} rel.err {err:.2e}")
            assert err < (1e-10 if kind == "uniform" else 1e-9)
        for i, lam in enumerate(ref_spec):
            if lam is not None:
                kk = min(len(lam), chi)
                assert np.max(np.abs(spec[k, i, :kk].cpu().numpy() - lam[:kk])) < 1e-12 * lam[0]


def test_wide_batch_with_a_state_that_is_not_a_number(gpu):
    eng = _engine()
    sv = np.stack([O.random_uniform_state(14, s) for s in (4, 5, 6)])
    _, ref, _ = eng.chi_truncate(eng.as_device_states(sv), 70)
    bad = sv.copy()
    bad[1, 3] = np.nan
    _, got, _ = eng.chi_truncate(eng.as_device_states(bad), 70)
    assert torch.equal(got[0], ref[0]) and torch.equal(got[2], ref[2])
    assert not bool(torch.isfinite(torch.view_as_real(got[1])).all())


def test_state_that_is_not_a_number_stays_alone(gpu):
    eng = _engine()
    sv = np.stack([O.random_uniform_state(9, s) for s in (4, 5, 6)])
    _, ref, _ = eng.chi_truncate(eng.as_device_states(sv), 8)
    bad = sv.copy()
    bad[1, 3] = np.nan
    _, got, _ = eng.chi_truncate(eng.as_device_states(bad), 8)
    assert torch.equal(got[0], ref[0]) and torch.equal(got[2], ref[2])
    assert not bool(torch.isfinite(torch.view_as_real(got[1])).all())


def test_two_sided_option(gpu):
    """QMX_OPT_TWO_SIDED_JACOBI changes the truncation by rounding only (1e-10,
    the suite's bar); MPS truncates with it and leaves the option as it was."""
    from qmprs_amd import _lib
    from qmprs_amd.primitives import MPS
    eng = _engine()
    sv = O.random_mps_state(13, 48, 9)
    dev = eng.as_device_states(sv)
    _, one, _ = eng.chi_truncate(dev, 32)
    with _lib.two_sided_jacobi():
        _, two, _ = eng.chi_truncate(dev, 32)
    mps = MPS(sv, bond_dimension=32)
    assert torch.equal(mps.state, two)
    _, again, _ = eng.chi_truncate(dev, 32)
    assert torch.equal(one, again)
    assert float(torch.linalg.vector_norm(one - two) / torch.linalg.vector_norm(two)) < 1e-10
    with pytest.raises(ValueError):
        _lib.set_option(_lib.QMX_OPT_TWO_SIDED_JACOBI, 2)


@pytest.mark.parametrize("kind", ["bond2", "product", "ghz", "near_product", "real"])
@pytest.mark.parametrize("n", [2, 3, 5, 9, 13])
def test_layer_eigensolvers_agree(gpu, n, kind):
    """The layers' 4 x 4 eigenproblems on one wave and in one lane: the same
    bonds and widths, and gates that agree.  Both find the kept subspace to
    eps over its gap; the kept and dropped eigenvalues differ by 1e-4 of the
    trace or more (bond-2 states drop nothing but zeros; the near-product ones
    keep 1e-4 and drop 1e-8), so to 1e-11 a step, amplified by the gates that
    follow: 1e-8."""
    eng = _engine()
    from qmprs_amd import _lib
    rng = np.random.default_rng(n)
    if kind == "ghz":
        sv = np.zeros(2 ** n, dtype=np.complex128)
        sv[0] = sv[-1] = 2 ** -0.5
    elif kind in ("product", "near_product"):
        sv = np.ones(1, dtype=np.complex128)
        for _ in range(n):
            sv = np.kron(sv, rng.standard_normal(2) + 1j * rng.standard_normal(2))
        sv /= np.linalg.norm(sv)
        if kind == "near_product":
            sv = sv + 0.01 * O.ket(O.random_mps_state(n, 2, 5))
    else:
        sv = O.random_mps_state(n, 2, 5)
        sv = sv.real.astype(np.complex128) if kind == "real" else sv
    psi = O.ket(sv)
    out = []
    for serial in (False, True):
        work = eng.as_device_states(psi).clone()
        if serial:
            with _lib.two_sided_jacobi():
                g, w, b = eng.generate_layer(work)
        else:
            g, w, b = eng.generate_layer(work)
        out.append((g.cpu().numpy(), w.cpu().numpy(), b.cpu().numpy()))
    (g0, w0, b0), (g1, w1, b1) = out
    assert np.array_equal(w0, w1) and np.array_equal(b0, b1)
    if kind != "real":       # (a real part of a bond-2 state has bond 4 and drops what it may)
        assert np.abs(g0 - g1).max() < 1e-8
    for gate, width in zip(g0[0].reshape(-1, 4, 4), w0[0].reshape(-1)):
        d = 4 if width == 2 else 2
        assert np.abs(gate[:d, :d] @ gate[:d, :d].conj().T - np.eye(d)).max() < 1e-12


def test_layer_of_a_state_that_is_not_a_number_is_refused(gpu):
    """With the same error from both eigensolvers."""
    eng = _engine()
    from qmprs_amd import _lib
    sv = O.random_mps_state(6, 4, 1)
    sv[5] = np.nan
    with pytest.raises((ValueError, RuntimeError)) as wave:
        eng.extract_layers(torch.from_numpy(sv).to(gpu).unsqueeze(0).contiguous(), 1)
    with _lib.two_sided_jacobi(), pytest.raises((ValueError, RuntimeError)) as lane:
        eng.extract_layers(torch.from_numpy(sv).to(gpu).unsqueeze(0).contiguous(), 1)
    assert wave.type is lane.type and str(wave.value) == str(lane.value)
