"""The two-sided eigensolvers of the chi-truncation (QMX_OPT_TWO_SIDED_JACOBI, the
drop-in calls and cutoffs below rounding): in one launch up to 48 columns, in LDS
up to 128, in one block on global memory up to 512 and by blocks above."""

import numpy as np
import pytest
import torch

from oracle import qmprs_oracle as O

pytestmark = pytest.mark.gpu

SIZES = [(8, 4), (10, 16), (11, 24), (11, 25), (12, 48), (13, 64), (14, 64), (11, 65), (11, 150), (16, 256), (18, 300)]


@pytest.mark.parametrize("kind", ["uniform", "mps"])
@pytest.mark.parametrize("n,chi", SIZES, ids=lambda v: str(v))
def test_truncation(gpu, n, chi, kind):
    """Targets to 1e-10 and spectra to 1e-9 of themselves and 1e-13 of the largest:
    the bars of test_chi_truncate_matches_oracle (targets 1e-9 for MPS above 128
    columns, whose kept vectors reach down to the cutoff); full-rank Gram matrices
    and rank-deficient ones, two states a call."""
    from qmprs_amd import _lib, engine
    svs = [O.random_uniform_state(n, s) if kind == "uniform" else O.random_mps_state(n, chi + chi // 2, s)
           for s in (21, 22)]
    with _lib.two_sided_jacobi():
        _, target, spec = engine.chi_truncate(engine.as_device_states(np.stack(svs)), chi, spectra=True)
    for k, sv in enumerate(svs):
        ref, ref_spec = O.chi_truncate(O.ket(sv), n, chi)
        err = np.linalg.norm(target[k].cpu().numpy() - ref) / np.linalg.norm(ref)
        print(f"n={n} chi={chi} {kind} rel.err {err:.1e}")
        assert err < (1e-9 if kind == "mps" and chi > 64 else 1e-10)
        for i, lam in enumerate(ref_spec):
            if lam is not None:
                kk = min(len(lam), chi)
                np.testing.assert_allclose(spec[k, i, :kk].cpu().numpy(), lam[:kk], rtol=1e-9, atol=1e-13 * lam[0])


@pytest.mark.parametrize("n,chi", [(10, 16), (11, 25), (13, 64), (11, 150), (18, 300)], ids=lambda v: str(v))
def test_sweep_cap_raises(gpu, n, chi):
    """Stopped after one sweep every one of them says so, and the next call works."""
    from qmprs_amd import _lib, engine
    dev = engine.as_device_states(O.random_uniform_state(n, 21))
    with _lib.two_sided_jacobi():
        _lib.set_option(_lib.QMX_OPT_JACOBI_SWEEP_CAP, 1)
        try:
            with pytest.raises(RuntimeError, match="converge"):
                engine.chi_truncate(dev, chi)
        finally:
            _lib.set_option(_lib.QMX_OPT_JACOBI_SWEEP_CAP, 0)
        _, target, _ = engine.chi_truncate(dev, chi)
    assert torch.isfinite(torch.view_as_real(target)).all()


def test_drop_in_call_above_64(gpu):
    """A drop-in call that truncates to 150 (300 columns, the one-block solver)."""
    from qmprs_amd import _lib, engine
    from qmprs_amd.primitives import MPS
    sv = O.random_uniform_state(11, 3)
    with _lib.two_sided_jacobi():
        _, two, _ = engine.chi_truncate(engine.as_device_states(sv), 150)
    mps = MPS(sv, bond_dimension=150)
    assert torch.equal(mps.state, two)
    ref, _ = O.chi_truncate(O.ket(sv), 11, 150)
    assert np.linalg.norm(mps.state[0].cpu().numpy() - ref) < 1e-10
