"""Rounding of the gate update's polar factor, apart from everything before it.

Four sites and two layers of gates with entries 0, 1 and 1/2, after which the
environment of the first two-site gate of the sweep is the conjugate of the
target over two, a 4 x 4 matrix, without rounding.  The one-site gate before it
has the partial trace of that matrix as its environment; targets lie on a grid
of 2^-20 and have a partial trace of one, so that this gate stays the identity."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

N, LAYERS = 4, 2
COUNT = 3000


def _circuit():
    """sum_ab |a b b a> / 2, and identities on the last two sites."""
    gates = np.zeros((LAYERS, N, 4, 4), dtype=np.complex128)
    h = np.array([[1.0, 1.0], [1.0, -1.0]])
    cnot = np.eye(4)[[0, 1, 3, 2]]
    swap = np.eye(4)[[0, 2, 1, 3]]
    gates[1, 0], gates[1, 1], gates[1, 2] = np.kron(h, h) / 2, cnot, swap      # acts first
    gates[0, 0], gates[0, 1], gates[0, 2] = swap, cnot, np.eye(4)
    gates[:, 3, :2, :2] = np.eye(2)
    widths = np.full((LAYERS, N), 2, dtype=np.int32)
    widths[:, 3] = 1
    return gates, widths


def _environments(kind):
    """(COUNT, 4, 4): entry (o, i) over sites 2, 3, partial trace over site 2 one."""
    rng = np.random.default_rng(5)
    g = lambda: rng.standard_normal((COUNT, 4, 4)) + 1j * rng.standard_normal((COUNT, 4, 4))
    bits = 20
    if kind == "gauss":
        e = g()
    elif kind == "rank 3":      # but for the grid
        e, bits = g()[:, :, :3] @ g()[:, :3], 32
    else:
        u, v = np.linalg.qr(g())[0], np.linalg.qr(g())[0]
        e = (u * (1 / kind) ** rng.random((COUNT, 1, 4))) @ v
    t = np.trace(e.reshape(COUNT, 2, 2, 2, 2), axis1=1, axis2=3)
    # a factor on the right that makes the partial trace the identity, near enough
    # for the grid's correction to be small
    e = e @ np.kron(np.eye(2), np.linalg.inv(t))
    e = np.round(e * 2.0 ** bits) / 2.0 ** bits
    t = np.trace(e.reshape(COUNT, 2, 2, 2, 2), axis1=1, axis2=3)
    e[:, 2:, 2:] += np.eye(2) - t
    return e


def _polar_long(e):
    """The unitary polar factors in extended precision (Newton's iteration)."""
    x = e.astype(np.clongdouble)
    for it in range(40):
        a = np.concatenate([x, np.broadcast_to(np.eye(4, dtype=np.clongdouble), x.shape)], axis=2).copy()
        rows = np.arange(len(x))
        for k in range(4):
            p = np.argmax(np.abs(a[:, k:, k]), axis=1) + k
            a[rows, k], a[rows, p] = a[rows, p].copy(), a[rows, k].copy()
            a[:, k] /= a[:, k, k][:, None]
            for i in range(4):
                if i != k:
                    a[:, i] -= a[:, i, k][:, None] * a[:, k]
        inv = np.conj(np.swapaxes(a[:, :, 4:], 1, 2))
        z = np.sqrt(np.sqrt((np.abs(inv) ** 2).sum((1, 2)) / (np.abs(x) ** 2).sum((1, 2)))) if it < 20 else np.ones(len(x))
        x = (z[:, None, None] * x + inv / z[:, None, None]) / 2
    return x


# Root mean square of |G' - conj(polar(E))|_F that a scaled Newton iteration with
# pivoted inverses has on these matrices (measured), the rounding to keep to.
NEWTON = {"gauss": 6.9e-16, 1.0: 4.4e-16, 10.0: 5.6e-16, 100.0: 2.33e-15, 1000.0: 6.1e-15}


def _updated(gpu, mode, gates, widths, target):
    """The gates after one sweep of every target from the same circuit."""
    from qmprs_amd import _lib, engine
    b = len(target)
    out = torch.from_numpy(np.broadcast_to(gates, (b,) + gates.shape).copy()).to(gpu)
    w = torch.from_numpy(np.broadcast_to(widths, (b,) + widths.shape).copy()).to(gpu)
    used = torch.full((b,), len(gates), dtype=torch.int32, device=gpu)
    _lib.set_sweep_mode(mode)
    try:
        engine.sweep(torch.from_numpy(np.ascontiguousarray(target)).to(gpu), out, w, used, 1)
    finally:
        _lib.set_sweep_mode("auto")
    out = out.cpu().numpy()
    assert (out[:, 0, -1, :2, :2] == np.eye(2)).all()     # the one-site gate before
    return out[:, 0, -2]


def _target(e):
    # amplitude of |s0 s1 s2 s3>: E[(s2 s3), (s1 s0)] = conj(T) / 2
    return 2 * np.conj(e).reshape(-1, 2, 2, 2, 2).transpose(0, 4, 3, 1, 2).reshape(-1, 16)


def _rms(a):
    return float(np.sqrt((np.abs(a) ** 2).sum((1, 2)).mean()))


@pytest.mark.parametrize("mode", ["auto", "step"])
@pytest.mark.parametrize("kind", NEWTON)
def test_polar_factor_rounding(gpu, kind, mode):
    e = _environments(kind)
    e = e[np.linalg.cond(e) < 1e5]      # beyond it another path decides
    rms = _rms(_updated(gpu, mode, *_circuit(), _target(e)) - np.conj(_polar_long(e)))
    print(f"{kind}: rms {rms:.2e}, Newton {NEWTON[kind]:.2e}")
    assert rms <= NEWTON[kind]


def _column_case(kind):
    """(gates, widths, targets, environments, their zero columns) of one layer
    whose sites are still in |0>: the two-site gate of two sites, whose environment
    has one column, and the second one of three sites, whose environment has two."""
    rng = np.random.default_rng(6)
    n = 2 if kind == "one column" else 3
    gates = np.zeros((1, n, 4, 4), dtype=np.complex128)
    gates[0, n - 2] = np.eye(4)
    gates[0, n - 1, :2, :2] = np.eye(2)
    h = np.ones((1, 1))                                   # the circuit: sum h[r][a] |r a 0>
    if n == 3:
        hadamard = np.array([[1.0, 1.0], [1.0, -1.0]])
        gates[0, 0] = np.diag([1, 1, 1, -1]) @ np.kron(hadamard, hadamard) / 2
        h = hadamard / 2
    widths = np.full((1, n), 2, dtype=np.int32)
    widths[0, n - 1] = 1
    t = rng.standard_normal((COUNT, len(h), 2, 2)) + 1j * rng.standard_normal((COUNT, len(h), 2, 2))
    t = np.round(t * 2.0 ** 20) / 2.0 ** 20
    # the last site's environment is one column: (1, 0), so that its gate stays
    t[:, 0, 0] += (np.array([1.0, 0.0]) - np.einsum("brac,ra->bc", t[:, :, :h.shape[1]], h)) / h[0, 0]
    e = np.zeros((COUNT, 4, 4), dtype=np.complex128)
    e[:, :, :2 * h.shape[1]:2] = np.einsum("brac,ri->baci", np.conj(t), h).reshape(COUNT, 4, h.shape[1])
    return gates, widths, t.reshape(COUNT, -1), e, [1, 2, 3] if n == 2 else [1, 3]


def _completed_long(e, zero):
    """Polar factors whose zero columns are completed by the first unit vectors
    with a residual above 1/2 against the columns so far, in extended precision."""
    m, q = e.astype(np.clongdouble), []

    def residual(v):
        for _ in range(2):
            for b in q:
                v = v - b * (np.conj(b) * v).sum(1)[:, None]
        return v, np.sqrt((np.abs(v) ** 2).sum(1))

    for c in range(4):
        if c not in zero:
            v, size = residual(m[:, :, c])
            q.append(v / size[:, None])
    start = np.zeros(len(e), dtype=int)
    for c in zero:
        done = np.zeros(len(e), dtype=bool)
        for k in range(4):
            v, size = residual(np.tile(np.eye(4, dtype=np.clongdouble)[k], (len(e), 1)))
            take = ~done & (k >= start) & (size > 0.5)
            m[take, :, c] = v[take] / size[take, None]
            start[take] = k + 1
            done |= take
        q.append(m[:, :, c].copy())
    return _polar_long(m)


# the same for the one-sided Jacobi with two passes of Gram-Schmidt for the completion
TWO_PASSES = {"one column": 1.62e-16, "two columns": 2.82e-16}


@pytest.mark.parametrize("mode", ["auto", "step"])
@pytest.mark.parametrize("kind", TWO_PASSES)
def test_completed_factor_rounding(gpu, kind, mode):
    g, w, target, e, zero = _column_case(kind)
    rms = _rms(_updated(gpu, mode, g, w, target) - np.conj(_completed_long(e, zero)))
    print(f"{kind}: rms {rms:.2e}, two passes {TWO_PASSES[kind]:.2e}")
    assert rms <= TWO_PASSES[kind]


ONE_LANE = 3.45e-16


@pytest.mark.parametrize("mode", ["auto", "step"])
def test_jacobi_factor_rounding(gpu, mode):
    """A smallest singular value near 1e-10, which the Jacobi path decides: what
    U^H E lacks of being Hermitian, in units of E's norm, against that path in one
    lane's registers (measured)."""
    e = _environments("rank 3")
    u = np.conj(_updated(gpu, mode, *_circuit(), _target(e))).astype(np.clongdouble)
    h = np.conj(np.swapaxes(u, 1, 2)) @ e.astype(np.clongdouble)
    rms = _rms((h - np.conj(np.swapaxes(h, 1, 2))) / np.linalg.norm(e, axis=(1, 2))[:, None, None])
    print(f"rms {rms:.2e}")
    assert rms <= ONE_LANE
