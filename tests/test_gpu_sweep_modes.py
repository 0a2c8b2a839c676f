"""Sweep options in every mode: small states run in one block by default, so the
gate-by-gate and the windowed kernels are asked for by name."""

import numpy as np
import pytest
import torch

from oracle import qmprs_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture
def mode():
    """Sets the sweep mode; automatic again afterwards."""
    from qmprs_amd import _lib
    yield _lib.set_sweep_mode
    _lib.set_sweep_mode("auto")


def _on_gpu(gpu, target, gates, widths, b=1):
    rep = lambda a: torch.from_numpy(np.broadcast_to(a, (b,) + a.shape).copy()).to(gpu)
    used = torch.full((b,), gates.shape[0], dtype=torch.int32, device=gpu)
    return rep(target), rep(gates), rep(widths), used


@pytest.mark.parametrize("name", ["auto", "step", "window"])
@pytest.mark.parametrize("omega", [1.0, 1.3, 1.9])
@pytest.mark.parametrize("n,layers,sweeps", [(3, 2, 2), (6, 3, 3), (10, 3, 2), (12, 2, 2)])
def test_relaxed_sweep_in_every_mode(gpu, mode, name, omega, n, layers, sweeps):
    """The gate update with and without over-relaxation against the oracle's, in
    complex128; the bars are those of the suite's relaxed sweeps."""
    from qmprs_amd import _lib, engine
    sv = O.ket(O.random_uniform_state(n, 10 * n + layers))
    target, _ = O.chi_truncate(sv, n, 2 ** n)
    extracted = O.get_unitary_layers(target, n, layers)
    trace = []
    gl = O.optimize_gate_list(target, n, O.layer_gate_list(extracted), sweeps, trace, polar="jacobi", omega=omega)
    g, w = engine.layers_to_arrays(extracted, n)
    t, gates, widths, used = _on_gpu(gpu, target, g, w)
    psi = torch.from_numpy(sv).to(gpu).unsqueeze(0)
    mode(name)
    _lib.set_sweep_relaxation(omega)
    try:
        res = engine.sweep(t, gates, widths, used, sweeps, psi_ref=psi, circuit_out=True)
        torch.cuda.synchronize()
    finally:
        _lib.set_sweep_relaxation(1.0)
    state = O.circuit_state(n, gl)
    err = np.linalg.norm(res.circuit[0].cpu().numpy() - state)
    print(f"{name} omega={omega} n={n} state err {err:.1e}")
    assert err < 1e-9
    assert abs(abs(res.fidelity[0, -1].item()) - abs(np.vdot(sv, state))) < 1e-10
    np.testing.assert_allclose(res.overlap[0].cpu().numpy(), np.abs(trace), rtol=1e-10)


@pytest.mark.parametrize("n", [11, 14])
@pytest.mark.parametrize("batch", [2, 5])
def test_split_windows_equal_single_stream(gpu, mode, n, batch):
    """Two interleaved half-batches of windowed sweeps give the single stream's
    results, up to the order of the blocks' partial sums (the suite's bars for
    that: gates 1e-10, fidelities 1e-12)."""
    from qmprs_amd import _lib, engine
    svs = np.stack([O.random_mps_state(n, 24, 60 + s) for s in range(batch)])
    mode("window")
    out = []
    for split in (False, True):
        _lib.set_split_sweeps(split)
        try:
            out.append(engine.encode(svs, 16, 3, 3, sweep_dtype=torch.complex128))
            torch.cuda.synchronize()
        finally:
            _lib.set_split_sweeps(True)
    one, two = out
    assert torch.equal(one.layers_used, two.layers_used)
    assert (one.gates - two.gates).abs().max().item() < 1e-10
    assert (one.fidelity - two.fidelity).abs().max().item() < 1e-12


@pytest.mark.parametrize("name", ["step", "window"])
def test_noalloc_scratch_is_reused(gpu, mode, name):
    """A large problem without a goal, then a small one that stops at its goal, on
    the library's own scratch: the second finds the first's values in every flag
    and counter it uses, and gives what a workspace of its own gives, bit for bit."""
    from qmprs_amd import _lib, engine
    mode(name)
    _lib.set_split_sweeps(False)
    try:
        for n, batch, dtype, sweeps, stop in ((18, 2, torch.complex128, 1, False), (12, 3, torch.complex64, 4, True)):
            svs = np.stack([O.random_mps_state(n, 16, 11 + s) for s in range(batch)])
            p = engine.encode_prepare(svs, 8, 3, sweep_dtype=dtype)
            assert _lib.load().qmx_sweep_workspace(n, batch, 1 if dtype == torch.complex128 else 0) \
                <= _lib.NOALLOC_SCRATCH_BYTES
            goal = None
            if stop:
                first = engine.sweep(p.target, p.gates.clone(), p.widths, p.layers_used, 1, psi_ref=p.psi)
                goal = first.fidelity[:, -1].abs().contiguous()
                goal[1] = 2.0       # never met: the others stop around it
            want = p.gates.clone()
            r = engine.sweep(p.target, want, p.widths, p.layers_used, sweeps, psi_ref=p.psi, goal=goal,
                             circuit_out=True)
            got = p.gates.clone()
            fid, ov, done = torch.zeros_like(r.fidelity), torch.zeros_like(r.overlap).contiguous(), \
                torch.zeros_like(r.sweeps_done)
            out = torch.empty_like(p.target)
            engine.sweep_noalloc(p.target, got, p.widths, p.layers_used, sweeps, fidelity=fid, overlap=ov,
                                 psi_ref=p.psi, goal=goal, sweeps_done=done, circuit_out=out)
            torch.cuda.synchronize()
            if stop:
                assert done.tolist() == [1, sweeps, 1]
            for x, y in ((got, want), (fid, r.fidelity), (ov, r.overlap), (done, r.sweeps_done), (out, r.circuit)):
                assert torch.equal(x, y)
    finally:
        _lib.set_split_sweeps(True)


def _env(kind, rng):
    g = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
    if kind == "zero":
        return np.zeros((4, 4), dtype=np.complex128)
    if kind.startswith("rank"):
        r = int(kind[-1])
        return g(4, r) @ g(r, 4)
    if kind.endswith("columns out"):
        e = g(4, 4)
        e[:, rng.permutation(4)[:int(kind[0])]] = 0
        return e
    u, v = np.linalg.qr(g(4, 4))[0], np.linalg.qr(g(4, 4))[0]
    s = np.array([1.0, 0.5, 0.3, float(kind.split()[1])])
    return (u * s) @ v


@pytest.mark.parametrize("name", ["auto", "step"])
@pytest.mark.parametrize("kind", ["smallest 1", "smallest 1e-3", "smallest 1e-5", "smallest 1e-6", "smallest 1e-8",
                                  "smallest 1e-10", "rank 3", "rank 2", "rank 1", "1 columns out", "2 columns out",
                                  "3 columns out", "zero"])
def test_every_branch_of_the_gate_update(gpu, mode, name, kind):
    """Environments for each path of the polar factor: the iteration, matrices it
    leaves to the Jacobi path (ill-conditioned, rank 3, zero), and the closed forms
    of rank 2 and of one and two columns.  Four sites in sum |a b b a> / 2, whose
    last two-site gate has half the target as its environment (times the
    unitary gate before it).  Against the oracle with the same completion rule: a factor
    is determined to eps over the smallest singular value that counts, 10 eps / s
    over these sums; s is at least 1e-3 where a matrix is random."""
    from qmprs_amd import engine
    rng = np.random.default_rng(len(kind) + ord(kind[-1]))
    h = np.array([[1.0, 1.0], [1.0, -1.0]])
    cnot, swap = np.eye(4)[[0, 1, 3, 2]], np.eye(4)[[0, 2, 1, 3]]
    g = np.zeros((2, 4, 4, 4), dtype=np.complex128)
    g[1, 0], g[1, 1], g[1, 2] = np.kron(h, h) / 2, cnot, swap
    g[0, 0], g[0, 1], g[0, 2] = swap, cnot, np.eye(4)
    g[:, 3, :2, :2] = np.eye(2)
    w = np.full((2, 4), 2, dtype=np.int32)
    w[:, 3] = 1
    gl = [(s, int(w[l, s]), g[l, s][:2 * w[l, s], :2 * w[l, s]]) for l in (1, 0) for s in range(4)]
    small = float(kind.split()[1]) if kind.startswith("smallest") else 1e-3
    mode(name)
    for _ in range(8):
        e = _env(kind, rng)
        target = 2 * np.conj(e).reshape(2, 2, 2, 2).transpose(3, 2, 0, 1).reshape(16)
        with np.errstate(all="ignore"):     # of gates further on, not compared
            want = O.sweep_once(target, 4, gl, polar="jacobi")[0]
        t, gates, widths, used = _on_gpu(gpu, target, g, w)
        engine.sweep(t, gates, widths, used, 1)
        got = gates[0, 0, 2].cpu().numpy()
        assert np.abs(got @ got.conj().T - np.eye(4)).max() < 1e-14
        diff = np.abs(got - want[6][2]).max()
        print(f"{name} {kind} {diff:.1e}")
        assert diff < 10 * np.finfo(float).eps / min(small, 1e-3)
