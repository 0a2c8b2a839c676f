"""Sweeps of small states in one block (the automatic mode) and windowed sweeps
whose passes leave out what the first circuit layer's gates no longer touch,
against the gate-by-gate sweep."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _states(n, b, gpu, dtype, seed):
    rng = np.random.default_rng(seed)
    psi = rng.standard_normal((b, 2 ** n)) + 1j * rng.standard_normal((b, 2 ** n))
    psi /= np.linalg.norm(psi, axis=1, keepdims=True)
    return torch.from_numpy(psi).to(gpu, dtype)


def _random_layers(n, b, layers, gpu, seed):
    """Random unitaries, two-qubit but for the last site's one-qubit gate (and
    one more one-qubit gate inside)."""
    rng = np.random.default_rng(seed)
    gates = np.zeros((b, layers, n, 4, 4), dtype=np.complex128)
    widths = np.full((b, layers, n), 2, dtype=np.int32)
    widths[:, :, n - 1] = 1
    if n > 4:
        widths[:, 0, n // 2] = 1
    for i in np.ndindex(b, layers, n):
        d = 4 if widths[i] == 2 else 2
        gates[i][:d, :d] = np.linalg.qr(rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d)))[0]
    return torch.from_numpy(gates).to(gpu), torch.from_numpy(widths).to(gpu)


@pytest.mark.parametrize("dtype", [torch.complex128, torch.complex64])
@pytest.mark.parametrize("n,layers,used", [(2, 1, [1]), (2, 3, [3, 0, 2]), (3, 2, [2, 1]), (4, 2, [2]),
                                           (5, 3, [3, 1, 0]), (6, 2, [2, 2]), (7, 1, [1]), (9, 2, [2]),
                                           (11, 2, [1, 2]), (12, 1, [1]), (12, 3, [3]), (13, 2, [2])])
def test_one_block_sweep(gpu, dtype, n, layers, used):
    _against_steps(gpu, "auto", dtype, n, layers, used)


@pytest.mark.parametrize("dtype", [torch.complex128, torch.complex64])
@pytest.mark.parametrize("n,layers,used", [(10, 1, [1, 0]), (11, 2, [2, 1]), (12, 3, [3, 1, 2]), (13, 1, [1]),
                                           (14, 2, [2]), (15, 3, [1, 3, 0]), (16, 1, [1]), (17, 2, [2, 2]),
                                           (18, 1, [1])])
def test_windowed_sweep(gpu, dtype, n, layers, used):
    _against_steps(gpu, "window", dtype, n, layers, used)


def _against_steps(gpu, sweep_mode, dtype, n, layers, used):
    """Random targets under random circuits: fidelities, overlaps, circuit
    states, gates, snapshots and the goal's stop.  The environments are generic
    but in the first circuit layer, whose gates act on |0> and are determined
    where the state is; so gates are compared above it, states everywhere.
    Sweeping twice: each of the at most 78 updates of the state is off by the
    rounding of the other mode, ~30 eps of the compute type (complex64 states
    are kept in 32 bits), over the smallest singular value, for random
    environments of a unit state >~ 1e-3: 1e-15 * 30 * 80 / 1e-3 ~ 3e-9 and
    6e-8 * 30 * 80 / 1e-3, where the latter only says that the overlap and the
    fidelity, stationary in each gate, agree to the state's own rounding,
    6e-8 * sqrt(80) * 30 ~ 2e-5."""
    from qmprs_amd import _lib, engine
    b = len(used)
    target = _states(n, b, gpu, dtype, 7 * n)
    ref = target.to(torch.complex128).contiguous()
    gates0, widths = _random_layers(n, b, layers, gpu, 11 * n + layers)
    lu = torch.tensor(used, dtype=torch.int32, device=gpu)
    out = {}
    for mode in (sweep_mode, "step"):
        try:
            _lib.set_sweep_mode(mode)
            gates = gates0.clone()
            snaps = torch.zeros((2,) + tuple(gates.shape), dtype=gates.dtype, device=gpu)
            res = engine.sweep(target, gates, widths, lu, 2, psi_ref=ref, circuit_out=True, snapshots=(0, snaps))
            torch.cuda.synchronize()
            out[mode] = (gates, snaps, res)
        finally:
            _lib.set_sweep_mode("auto")
    (ga, sa, ra), (gs, ss, rs) = out[sweep_mode], out["step"]
    tol = 3e-9 if dtype == torch.complex128 else 2e-5
    assert torch.equal(sa[0], gates0)
    for i, k in enumerate(used):
        assert torch.equal(ga[i, k:], gates0[i, k:])          # unused layers stay
        assert torch.equal(sa[:, i, k:], gates0[None, i, k:].expand_as(sa[:, i, k:]))
    assert torch.isfinite(torch.view_as_real(ga)).all()
    for m in range(b):
        for l, s in np.ndindex(used[m], n):
            d = 4 if widths[m, l, s] == 2 else 2
            u = ga[m, l, s, :d, :d]
            eye = torch.eye(d, dtype=u.dtype, device=gpu)
            assert (u @ u.conj().T - eye).abs().max() < 1e-12
    if dtype == torch.complex128 and n > 2:
        for i, k in enumerate(used):
            if k > 1:
                assert (sa[1, i, 1:k] - ss[1, i, 1:k]).abs().max() < tol
    assert (ra.fidelity - rs.fidelity).abs().max() < tol
    live = [i for i, k in enumerate(used) if k > 0]
    assert (ra.overlap[live] - rs.overlap[live]).abs().max() < tol
    assert (ra.circuit - rs.circuit).abs().max() < (tol if dtype == torch.complex128 else 2e-3)
    try:
        _lib.set_sweep_mode(sweep_mode)
        # a goal: met from the start, met after one sweep, out of reach
        f = ra.fidelity.abs().real
        for goal, want in ((f[:, 0] - 1e-3, 0), ((f[:, 0] + f[:, 1]) / 2, 1), (f[:, 0] * 0 + 2.0, 2)):
            gates = gates0.clone()
            r = engine.sweep(target, gates, widths, lu, 2, psi_ref=ref, goal=goal.contiguous(), circuit_out=True)
            done = r.sweeps_done.cpu().tolist()
            for i in live:
                if want != 1 or f[i, 1] > f[i, 0] + 1e-3:
                    assert done[i] == want
                after = [gates0, sa[1], ga][done[i]][i]
                assert (gates[i] - after).abs().max() < 1e-14
    finally:
        _lib.set_sweep_mode("auto")


@pytest.mark.parametrize("n,sweeps", [(4, 0), (10, 1), (14, 0), (14, 1)])
def test_final_state_into_awkward_places(gpu, n, sweeps):
    """The final circuit state over the fidelity reference and at an address
    that is aligned to one amplitude only: as in a buffer of its own."""
    from qmprs_amd import engine
    b, layers = 2, 2
    gates0, widths = _random_layers(n, b, layers, gpu, 5)
    lu = torch.full((b,), layers, dtype=torch.int32, device=gpu)
    for dtype, awkward in ((torch.complex128, "reference"), (torch.complex64, "address")):
        target = _states(n, b, gpu, dtype, 6)
        ref = target.to(torch.complex128).clone()
        got = []
        for place in ("own", awkward):
            psi_ref = ref.clone()
            if place == "reference":
                out = psi_ref
            elif place == "address":
                out = torch.empty(b * 2 ** n + 1, dtype=dtype, device=gpu)[1:].view(b, 2 ** n)
            else:
                out = torch.empty_like(target)
            fid = torch.zeros((b, sweeps + 1), dtype=torch.complex128, device=gpu)
            ov = torch.zeros((b, max(sweeps, 1)), dtype=torch.float64, device=gpu)
            gates = gates0.clone()
            engine.sweep_noalloc(target, gates, widths, lu, sweeps, fid, ov if sweeps else None, psi_ref,
                                 circuit_out=out)
            torch.cuda.synchronize()
            got.append((out.clone(), fid, gates))
        for x, y in zip(*got):
            assert torch.equal(x, y)
