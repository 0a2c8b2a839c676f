"""The chi-truncation of states whose Schmidt spectra run out below rounding:
what the eigensolver's factor leaves out must not be missing from the state."""

import numpy as np
import pytest
import torch

from oracle import qmprs_oracle as O

pytestmark = pytest.mark.gpu


def _smooth(n, kind):
    x = np.linspace(-1, 1, 2 ** n)
    if kind == "gauss":
        v = np.exp(-x * x / 0.0288) * np.exp(1j * (7 * x + 11 * x ** 3))
    else:
        v = np.exp(3j * x * x) / (1 + 30 * (x - 0.3) ** 2)
    return O.ket(v)


def _low_rank(n, seed):
    """Eight equal Schmidt coefficients at the middle bond and sixteen of 1e-9 to 1e-8."""
    rng = np.random.default_rng(seed)
    m = 2 ** (n // 2)
    q = [np.linalg.qr(rng.standard_normal((d, m)) + 1j * rng.standard_normal((d, m)))[0] for d in (m, 2 ** n // m)]
    s = np.zeros(m)
    s[:8] = 1
    s[8:24] = 10.0 ** (-8 - rng.random(16))
    return O.ket(((q[0] * s) @ q[1].T).reshape(-1))


def _state(n, kind):
    return _low_rank(n, n) if kind == "low" else _smooth(n, kind)


EPS = np.finfo(float).eps
SIZES = pytest.mark.parametrize("n,chi", [(12, 16), (12, 32), (14, 64), (15, 100)])
KINDS = pytest.mark.parametrize("kind", ["gauss", "lorentz", "low"])


@KINDS
@SIZES
def test_spectra_leave_the_target_as_it_is(gpu, n, chi, kind):
    """The same target with and without spectra, bit for bit (its route does not
    depend on them), at the default cutoff and at 0.  The default's against the
    oracle: the Gram matrix of 2 chi columns is off by 2 chi eps of its trace,
    which turns a kept vector of weight above the cutoff by that over its
    weight and so moves the state by 2 chi eps / sqrt(cutoff)."""
    from qmprs_amd import engine
    sv = _state(n, kind)
    dev = engine.as_device_states(sv)
    for cutoff in (1e-10, 0.0):
        _, plain, _ = engine.chi_truncate(dev, chi, cutoff=cutoff)
        _, target, _ = engine.chi_truncate(dev, chi, cutoff=cutoff, spectra=True)
        diff = float(torch.linalg.vector_norm(plain - target))
        print(f"{kind} n={n} chi={chi} cutoff={cutoff:g} spectra against none {diff:.1e}")
        assert torch.equal(plain, target)
        if cutoff > 0:
            ref, _ = O.chi_truncate(sv, n, chi, cutoff)
            assert np.linalg.norm(target[0].cpu().numpy() - ref) < max(1e-10, 2 * chi * EPS / np.sqrt(cutoff))


@KINDS
@SIZES
@pytest.mark.parametrize("cutoff", [0.0, 1e-16, 1e-14])
def test_cutoffs_below_rounding(gpu, n, chi, kind, cutoff):
    """A cutoff below 2 chi eps asks for directions that the one-sided solver has
    no vectors for: the route is the two-sided solver's, bit for bit, and the
    state keeps all but a weight of cutoff + eps a bond (the bonds of every kind
    end at 1e-8 or below, and chi holds all of them but 8 of 'low')."""
    from qmprs_amd import _lib, engine
    sv = _state(n, kind)
    dev = engine.as_device_states(sv)
    _, got, _ = engine.chi_truncate(dev, chi, cutoff=cutoff)
    with _lib.two_sided_jacobi():
        _, two, _ = engine.chi_truncate(dev, chi, cutoff=cutoff)
    diff, err = float(torch.linalg.vector_norm(got - two)), float(np.linalg.norm(got[0].cpu().numpy() - sv))
    print(f"{kind} n={n} chi={chi} cutoff={cutoff:g} against two-sided {diff:.1e}, against the state {err:.1e}")
    assert torch.equal(got, two)
    assert err < np.sqrt(n * (cutoff + EPS)) + 2e-8
