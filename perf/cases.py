"""Performance cases of the encoder: what a user has it do, over the sizes it is used at.

``listed()`` names the cases, ``draw`` gives more of the same ranges,
``prepare`` makes a case's inputs from a seed, ``run`` is one pass through
the public entry points, ``work`` the bytes and operations that pass cannot do
without and ``exact`` its outputs in plain 64-bit torch / numpy.

States are random matrix-product states (the benchmark's workload) or, for the
drop-in calls, uniform random statevectors as in the tests.  Sweeps start from
a circuit that already fits the target in part, as the layer extraction
leaves it.  All of it comes from the seed.
"""

from __future__ import annotations

import math

import numpy as np
import torch

from qmprs_amd import engine, learned
from qmprs_amd.circuit import GateCircuit
from qmprs_amd.synthesis.mps_encoding import Sequential

C64, C128 = torch.complex64, torch.complex128


# ------------------------------------------------------------------ cases ---

def listed() -> list[dict]:
    return [
        # The smallest drop-in call: one 6-qubit statevector from host memory to
        # a circuit object (the size of the tests' scenarios).
        dict(name="prepare_n6", kind="prepare", n=6, chi=8, layers=4, sweeps=10, snake=False, compress=0.0),
        # The usage example's size: 10 qubits, bond dimension 512 (no
        # truncation), 50 sweeps.
        dict(name="prepare_n10", kind="prepare", n=10, chi=512, layers=6, sweeps=50, snake=False, compress=0.0),
        # One odd-sized state with the input options in use: snake indexing and
        # compression, truncated bonds, layers and sweeps.
        dict(name="prepare_n17_snake", kind="prepare", n=17, chi=64, layers=5, sweeps=4, snake=True, compress=2.0),
        # A service's mixed bag: states of different sizes and bond dimensions in one call.
        dict(name="ragged_n9_15", kind="ragged", n=9, n_hi=15, count=14, layers=3, sweeps=3),
        # The benchmark's truncation phase: complex64 inputs, N=20, bond 64.
        dict(name="chi_n20_b32", kind="chi", n=20, batch=32, chi=64, dtype="c64"),
        # A large bond dimension on one state (the block eigensolver).
        dict(name="chi_n18_chi300", kind="chi", n=18, batch=1, chi=300, dtype="c128"),
        # Layer extraction of a batch at the benchmark's size.
        dict(name="layers_n20_b32", kind="layers", n=20, batch=32, layers=3),
        # One sweep of the benchmark's circuits in the parity mode (complex128).
        dict(name="sweep_n20_b32", kind="sweep", n=20, batch=32, layers=10, sweeps=1, dtype="c128"),
        # A stretch of sweeps over a batch of small states.
        dict(name="sweep_n12_b64", kind="sweep", n=12, batch=64, layers=8, sweeps=4, dtype="c128"),
        # The throughput mode (complex64 states), a stretch of sweeps of shallow circuits.
        dict(name="sweep64_n20_b64", kind="sweep", n=20, batch=64, layers=2, sweeps=4, dtype="c64"),
        # Read-back of a batch of circuits with their fidelities, complex64.
        dict(name="circuit_n20_b64", kind="circuit", n=20, batch=64, layers=10, dtype="c64"),
        # One minibatch of the learned warm start's training: forward, loss, backward, Adam.
        dict(name="train_r512", kind="train", rows=512, width=512),
    ]


def draw(rng) -> dict:
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["prepare", "prepare", "ragged", "chi", "layers", "sweep", "sweep", "sweep64", "circuit", "train"])
    if kind == "prepare":
        n = rng.randint(4, 16)
        return dict(kind=kind, n=n, chi=rng.choice([4, 8, 16, 24, 32, 48, 64]), layers=rng.randint(1, 5),
                    sweeps=rng.randint(0, 20) if n < 13 else rng.randint(0, 5), snake=rng.random() < 0.3,
                    compress=rng.choice([0.0, 0.0, 1.0, 5.0]))
    if kind == "ragged":
        lo = rng.randint(6, 12)
        return dict(kind=kind, n=lo, n_hi=lo + rng.randint(1, 5), count=rng.randint(3, 20),
                    layers=rng.randint(1, 4), sweeps=rng.randint(1, 4))
    if kind == "chi":
        n = rng.randint(9, 20)
        return dict(kind=kind, n=n, batch=logint(1, max(1, min(64, 32 << (20 - n)))),
                    chi=rng.choice([8, 13, 16, 32, 50, 64]), dtype=rng.choice(["c64", "c128"]))
    if kind == "layers":
        n = rng.randint(8, 20)
        return dict(kind=kind, n=n, batch=logint(1, max(1, min(128, 32 << (20 - n)))), layers=rng.randint(1, 4))
    if kind == "sweep":
        n = rng.randint(6, 20)
        batch = logint(1, max(1, min(96, 24 << (20 - n))))
        return dict(kind=kind, n=n, batch=batch, layers=rng.randint(1, 9),
                    sweeps=1 if n > 15 else rng.randint(1, 4), dtype="c128")
    if kind == "sweep64":
        n = rng.randint(6, 20)
        return dict(kind="sweep", n=n, batch=logint(1, max(1, min(96, 48 << (20 - n)))), layers=rng.randint(1, 2),
                    sweeps=rng.randint(1, 4), dtype="c64")
    if kind == "circuit":
        n = rng.randint(6, 20)
        return dict(kind=kind, n=n, batch=logint(1, max(1, min(128, 40 << (20 - n)))), layers=rng.randint(1, 10),
                    dtype=rng.choice(["c64", "c128"]))
    return dict(kind=kind, rows=logint(200, 4096), width=rng.choice([128, 256, 512]))


def _sizes(case) -> list[tuple[int, int]]:
    """(N, bond dimension) of a ragged batch's states."""
    span = case["n_hi"] - case["n"] + 1
    return [(case["n"] + (7 * k) % span, (16, 32, 64)[k % 3]) for k in range(case["count"])]


# ----------------------------------------------------------------- inputs ---

def _gen(seed: int, stream: int) -> np.random.Generator:
    return np.random.default_rng([int(seed) & 0x7FFFFFFF, stream])


def _gauss(rng, *shape) -> np.ndarray:
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


def _mps_states(n: int, bond: int, batch: int, seed: int) -> torch.Tensor:
    """(batch, 2^n) complex128 on the GPU: normalised random MPS with complex Gaussian site tensors."""
    rng = _gen(seed, 1)
    dims = [1] + [min(bond, 2 ** i, 2 ** (n - i)) for i in range(1, n)] + [1]
    psi = torch.ones((batch, 1, 1), dtype=C128, device="cuda")
    for i in range(n):
        a = torch.from_numpy(_gauss(rng, batch, dims[i], 2 * dims[i + 1])).cuda()
        psi = torch.matmul(psi, a).reshape(batch, -1, dims[i + 1])
    psi = psi.reshape(batch, -1)
    return psi / torch.linalg.vector_norm(psi, dim=1, keepdim=True)


def _unitaries(rng, batch: int, layers: int, n: int, angle: float) -> np.ndarray:
    """(batch, layers, n, 4, 4) unitaries near the identity; the last site's act on one qubit (2 x 2 block)."""
    h = _gauss(rng, batch, layers, n, 4, 4)
    h[:, :, n - 1, 2:, :] = 0
    h[:, :, n - 1, :, 2:] = 0
    h = (h + np.conj(np.swapaxes(h, -1, -2))) / 2
    lam, v = np.linalg.eigh(h)
    u = (v * np.exp(1j * angle * lam)[..., None, :]) @ np.conj(np.swapaxes(v, -1, -2))
    u[:, :, n - 1, 2:, :] = 0
    u[:, :, n - 1, :, 2:] = 0
    return np.ascontiguousarray(u)


def _widths(batch: int, layers: int, n: int) -> torch.Tensor:
    w = torch.full((batch, layers, n), 2, dtype=torch.int32)
    w[:, :, n - 1] = 1
    return w.cuda()


def _fit(case, seed: int):
    """A target, the input state it came from and a circuit that fits both in part."""
    n, b, nl = case["n"], case["batch"], case["layers"]
    rng = _gen(seed, 2)
    g0 = _unitaries(rng, b, nl, n, 0.5)
    gates = torch.from_numpy(np.ascontiguousarray(g0 @ _unit_block(_unitaries(rng, b, nl, n, 0.15)))).cuda()
    other = _mps_states(n, 16, b, seed)
    psi = _circuit(torch.from_numpy(g0).cuda(), n) + 0.8 * other
    psi = psi / torch.linalg.vector_norm(psi, dim=1, keepdim=True)
    target = psi * 0.999     # a truncated state's norm is a little below one
    return psi.contiguous(), target.contiguous(), gates


def _unit_block(u: np.ndarray) -> np.ndarray:
    u = u.copy()
    n = u.shape[2]
    u[:, :, n - 1, 2, 2] = u[:, :, n - 1, 3, 3] = 1
    return u


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    st = {"case": case}
    if kind == "prepare":
        n = case["n"]
        v = _gauss(_gen(seed, 3), 2 ** n)
        st["statevector"] = v / np.linalg.norm(v)
        st["encoder"] = Sequential(GateCircuit)
    elif kind == "ragged":
        sizes = _sizes(case)
        st["states"] = [_mps_states(n, 48, 1, seed + 1000 * k)[0] for k, (n, _) in enumerate(sizes)]
        st["chis"] = [chi for _, chi in sizes]
    elif kind == "chi":
        st["states"] = _mps_states(case["n"], max(2 * case["chi"] * 3 // 4, 2), case["batch"], seed)
        if case["dtype"] == "c64":
            st["states"] = st["states"].to(C64)
    elif kind == "layers":
        st["psi"] = _mps_states(case["n"], 64, case["batch"], seed).contiguous()
    elif kind == "sweep":
        psi, target, gates = _fit(case, seed)
        st.update(psi=psi, target=target.to(C64) if case["dtype"] == "c64" else target, gates=gates)
        st["widths"] = _widths(case["batch"], case["layers"], case["n"])
        st["used"] = torch.full((case["batch"],), case["layers"], dtype=torch.int32, device="cuda")
    elif kind == "circuit":
        n, b, nl = case["n"], case["batch"], case["layers"]
        st["gates"] = torch.from_numpy(_unitaries(_gen(seed, 2), b, nl, n, 0.5)).cuda()
        st["psi"] = _mps_states(n, 16, b, seed).contiguous()
        st["widths"] = _widths(b, nl, n)
        st["used"] = torch.full((b,), nl, dtype=torch.int32, device="cuda")
    else:
        rng = _gen(seed, 4)
        net = learned.WarmStartMLP(case["width"], seed=int(seed) & 0xFFFF)
        x = rng.standard_normal((case["rows"], learned.IN_DIM)).astype(np.float32)
        st["net"] = net
        st["x"] = torch.from_numpy(x).cuda().to(torch.bfloat16).view(torch.int16).contiguous()
        st["t"] = torch.from_numpy(rng.standard_normal((case["rows"], learned.OUT_DIM)).astype(np.float32)).cuda()
    return st


# -------------------------------------------------------------------- run ---

def run(st: dict):
    case = st["case"]
    kind = case["kind"]
    if kind == "prepare":
        enc = st["encoder"]
        circuit = enc.prepare_state(st["statevector"], case["chi"], compression_percentage=case["compress"],
                                    index_type="snake" if case["snake"] else "row",
                                    num_layers=case["layers"], num_sweeps=case["sweeps"])
        return {"gates": np.concatenate([m.reshape(-1) for m, _ in circuit.gates]),
                "qubits": np.array([q for _, qs in circuit.gates for q in qs]),
                "fidelity": enc.last_info["fidelity"]}
    if kind == "ragged":
        res = engine.encode_ragged(st["states"], st["chis"], case["layers"], case["sweeps"], sweep_dtype=C128)
        return {"gates": torch.cat([r.gates.reshape(-1) for r in res]),
                "widths": torch.cat([r.widths.reshape(-1) for r in res]),
                "layers_used": np.array([r.layers_used for r in res]),
                "fidelity": torch.cat([r.fidelity for r in res])}
    if kind == "chi":
        psi, target, _ = engine.chi_truncate(st["states"], case["chi"])
        return {"psi": psi, "target": target}
    if kind == "layers":
        work = st["psi"].clone()
        gates, widths, used, amp0, _ = engine.extract_layers(work, case["layers"])
        return {"gates": gates, "widths": widths, "used": used, "amp0": amp0, "residual": work}
    if kind == "sweep":
        gates = st["gates"].clone()
        r = engine.sweep(st["target"], gates, st["widths"], st["used"], case["sweeps"], psi_ref=st["psi"],
                         circuit_out=True)
        if case["dtype"] == "c64":
            # Single-precision sweeps determine the circuit's state and its
            # overlaps to single precision.  The gates are not determined by
            # them: a gate that acts on a site still in |0> has an environment
            # of rank 2, whose null space is rounding noise at 1e-7.
            return {"circuit": r.circuit, "fidelity": r.fidelity.to(C64), "overlap": r.overlap.float()}
        return {"circuit": r.circuit, "fidelity": r.fidelity, "overlap": r.overlap, "gates": gates}
    if kind == "circuit":
        dt = C64 if case["dtype"] == "c64" else C128
        state, fid = engine.circuit_state(st["gates"], st["widths"], st["used"], dtype=dt, psi_ref=st["psi"])
        return {"state": state, "fidelity": fid.to(dt)}
    net = st["net"]
    y = net.forward(st["x"])
    loss, dy = learned.mse_loss(y, st["t"], None, learned.TRAJ_OUT)
    grads = net.backward(st["x"], dy)
    net.adam(grads, 1e-3)
    return {"y": y, "loss": loss, "grads": grads, "params": net.params.clone()}


# ------------------------------------------------------------------- work ---

def _chi_work(n: int, chi: int) -> float:
    """FP64 operations of the truncation chain of one state: Gram matrices, products, eigenproblems."""
    f, r = 0.0, 1
    for i in range(n - 1, 0, -1):
        cols = 2 * r
        r = min(cols, 2 ** i, chi)
        if 2 ** (n - i) > chi:
            f += 8.0 * 2 ** i * cols * (cols / 2 + 2 * r) + 8.0 * 9 * cols ** 3
    return f


def _layer_work(n: int) -> float:
    """One Ran layer: bond-2 chain (4 columns, 2 kept) and the inverse layer's gates."""
    return 8.0 * 2 ** n * (10 + 8) + 32.0 * 2 ** n * n


def _sweep_work(n: int, layers: int, sweeps: int) -> float:
    """Per gate: phi and T' by a 4 x 4 matrix and the 16 entries of E; the circuit before each sweep and after."""
    gates = layers * n
    return 2.0 ** n * 32.0 * gates * (3.0 * sweeps + (sweeps + 1))


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "prepare":
        n, nl = case["n"], case["layers"]
        return {"bytes": 16.0 * 2 ** n + 256.0 * nl * n,
                "flops": _chi_work(n, case["chi"]) + nl * _layer_work(n) + _sweep_work(n, nl, case["sweeps"])}
    if kind == "ragged":
        b = f = 0.0
        for n, chi in _sizes(case):
            b += 16.0 * 2 ** n + 260.0 * case["layers"] * n
            f += _chi_work(n, chi) + case["layers"] * _layer_work(n) + _sweep_work(n, case["layers"], case["sweeps"])
        return {"bytes": b, "flops": f}
    if kind == "train":
        w, r = case["width"], case["rows"]
        count = learned.IN_DIM * w + w * w + w * learned.OUT_DIM + 2 * w + learned.OUT_DIM
        macs = r * (learned.IN_DIM * w + w * w + w * learned.OUT_DIM)
        return {"bytes": 4.0 * count * 7 + 2.0 * count + r * (2.0 * learned.IN_DIM + 12.0 * learned.OUT_DIM),
                "flops": 6.0 * macs - 2.0 * r * learned.IN_DIM * w}
    n, b = case["n"], case["batch"]
    amps = float(b) * 2 ** n
    if kind == "chi":
        return {"bytes": amps * ((8 if case["dtype"] == "c64" else 16) + 32.0), "flops": b * _chi_work(n, case["chi"])}
    if kind == "layers":
        return {"bytes": amps * 32.0, "flops": b * case["layers"] * _layer_work(n)}
    size = 8.0 if case["dtype"] == "c64" else 16.0
    if kind == "sweep":
        return {"bytes": amps * (2 * size + 16.0), "flops": b * _sweep_work(n, case["layers"], case["sweeps"])}
    return {"bytes": amps * (size + 16.0), "flops": amps * 32.0 * case["layers"] * n}


# ------------------------------------------------------------------ exact ---

def _gate(psi: torch.Tensor, g: torch.Tensor, n: int, site: int, width: int) -> torch.Tensor:
    """psi (B, 2^n) with g (B, 4, 4; its 2 x 2 block for width 1) applied at site (site 0: top bit)."""
    d = 2 * width
    x = psi.reshape(psi.shape[0], 2 ** site, d, -1)
    y = torch.empty_like(x)
    for o in range(d):
        acc = g[:, o, 0, None, None] * x[:, :, 0]
        for i in range(1, d):
            acc += g[:, o, i, None, None] * x[:, :, i]
        y[:, :, o] = acc
    return y.reshape(psi.shape)


def _width(n: int, site: int) -> int:
    return 2 if site < n - 1 else 1


def _circuit(gates: torch.Tensor, n: int) -> torch.Tensor:
    """C|0..0>: the last layer acts first, each from site 0 on."""
    b, nl = gates.shape[:2]
    psi = torch.zeros((b, 2 ** n), dtype=C128, device=gates.device)
    psi[:, 0] = 1
    for layer in reversed(range(nl)):
        for s in range(n):
            psi = _gate(psi, gates[:, layer, s], n, s, _width(n, s))
    return psi


def _dot(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    return (a.conj() * b).sum(dim=1)


def _adj(g: torch.Tensor) -> torch.Tensor:
    return g.conj().transpose(-1, -2)


def _sweeps(target: torch.Tensor, gates: torch.Tensor, psi: torch.Tensor, n: int, sweeps: int):
    """Environment sweeps gate by gate in reverse circuit order; gates updated in place."""
    b, nl = gates.shape[:2]
    fid, over = [], []
    for _ in range(sweeps):
        phi = _circuit(gates, n)
        fid.append(_dot(psi, phi))
        t = target
        for layer in range(nl):
            for s in reversed(range(n)):
                w = _width(n, s)
                d = 2 * w
                phi = _gate(phi, _adj(gates[:, layer, s]), n, s, w)
                x = t.reshape(b, 2 ** s, d, -1).transpose(1, 2).reshape(b, d, -1)
                y = phi.reshape(b, 2 ** s, d, -1).transpose(1, 2).reshape(b, d, -1)
                u, sv, vh = np.linalg.svd(torch.matmul(x.conj(), y.transpose(1, 2).contiguous()).cpu().numpy())
                new = torch.zeros((b, 4, 4), dtype=C128)
                new[:, :d, :d] = torch.from_numpy(np.conj(u @ vh))
                gates[:, layer, s] = new.to(gates.device)
                t = _gate(t, _adj(gates[:, layer, s]), n, s, w)
        over.append(torch.from_numpy(sv.sum(axis=1)))
    phi = _circuit(gates, n)
    fid.append(_dot(psi, phi))
    return phi, torch.stack(fid, dim=1), torch.stack(over, dim=1) if over else None


def _keep(lam: np.ndarray, most: int, cutoff: float = 1e-10) -> int:
    lam = np.maximum(lam, 0)
    k = len(lam)
    tail = 0.0
    for j in range(len(lam) - 1, 0, -1):
        tail += lam[j]
        if tail > cutoff * lam.sum():
            break
        k = j
    return max(1, min(k, most))


def _truncate(psi: np.ndarray, n: int, chi: int) -> np.ndarray:
    """The chi-truncated state of one normalised statevector: right-to-left SVD chain."""
    x, ws = psi.reshape(-1, 1), []
    for i in range(n - 1, 0, -1):
        y = x.reshape(2 ** i, -1)
        if y.shape[1] <= chi:      # nothing to truncate
            ws.append(None)
            x = y
            continue
        r = np.linalg.qr(y, mode="r") if y.shape[0] > y.shape[1] else y
        _, s, vh = np.linalg.svd(r, full_matrices=False)
        w = np.conj(vh[:_keep(s * s, chi)].T)
        ws.append(w)
        x = y @ w
    for i, w in enumerate(reversed(ws), start=1):
        x = (x if w is None else x @ np.conj(w.T)).reshape(2 ** (i + 1), -1)
    return x.reshape(-1)


def _basis(v: np.ndarray) -> np.ndarray:
    """Orthonormal basis of span(v): Gram-Schmidt over the projector's columns in index order."""
    p, out = v @ np.conj(v.T), []
    for j in range(p.shape[1]):
        if len(out) == v.shape[1]:
            break
        c = p[:, j].copy()
        for _ in range(2):
            for q in out:
                c -= q * np.vdot(q, c)
        if np.linalg.norm(c) > 1e-7:
            out.append(c / np.linalg.norm(c))
    return np.stack(out, axis=1)


def _null(rows: np.ndarray) -> np.ndarray:
    """Householder null space: the trailing columns of the full QR factor of rows^T."""
    return np.linalg.qr(rows.T, mode="complete")[0][:, rows.shape[0]:]


def _layer(psi: np.ndarray, n: int):
    """Ran's layer of one normalised state with bonds of 2 at every cut: (n, 4, 4) gates."""
    x, w = psi.reshape(-1, 1), [None] * n
    for i in range(n - 1, 0, -1):
        y = x.reshape(2 ** i, -1)
        lam, v = np.linalg.eigh(np.conj(y.T) @ y)
        k = _keep(lam[::-1], 2)
        if k != 2:
            raise ValueError("a bond of one: a state of this kind has none")
        w[i] = _basis(v[:, ::-1][:, :k])
        x = y @ w[i]
    gates = np.zeros((n, 4, 4), dtype=np.complex128)
    a = x.reshape(-1) / np.linalg.norm(x)
    nu = _null(a[None])
    gates[0] = np.stack([a, nu[:, 1], nu[:, 0], nu[:, 2]], axis=1)
    for s in range(1, n - 1):
        t = np.conj(w[s].T)
        nu = _null(t)
        for c in range(2):
            if abs(nu[0, c]) > 1e-12:
                nu[:, c] *= np.conj(nu[0, c]) / abs(nu[0, c])
        gates[s] = np.stack([t[0], nu[:, 0], t[1], nu[:, 1]], axis=1)
    gates[n - 1, :2, :2] = np.conj(w[n - 1])
    return gates


def _extract(work: torch.Tensor, n: int, layers: int):
    """The layer loop: (gates, conj <0..0|state> after each layer, residual states)."""
    b = work.shape[0]
    gates = torch.zeros((b, layers, n, 4, 4), dtype=C128, device=work.device)
    amp0 = []
    for layer in range(layers):
        host = work.cpu().numpy()
        gates[:, layer] = torch.from_numpy(np.stack([_layer(h, n) for h in host])).to(work.device)
        for s in reversed(range(n)):
            work = _gate(work, _adj(gates[:, layer, s]), n, s, _width(n, s))
        amp0.append(work[:, 0].conj())
        if bool(((amp0[-1] - 1).abs() <= 1.1e-5).any()):
            raise ValueError("an early exit: a state of this kind has none")
    return gates, torch.stack(amp0, dim=1), work


def _encode(v: np.ndarray, n: int, chi: int, layers: int, sweeps: int):
    """prepare_state of one statevector: (gates, <psi|C|0> before each sweep and at the end)."""
    psi = v / np.linalg.norm(v)
    target = torch.from_numpy(_truncate(psi, n, chi))[None]
    gates, _, _ = _extract(target / torch.linalg.vector_norm(target), n, layers)
    _, fid, _ = _sweeps(target, gates, torch.from_numpy(psi)[None], n, sweeps)
    return gates[0], fid[0]


def _after(sweeps: int, gates):
    """Gates after sweeps have no one value: the null space of a gate's rank-deficient
    environment (a neighbour still in |0>) is free.  What the circuit does has one."""
    return None if sweeps else gates


def exact(case: dict, seed: int):
    """What ``run`` returns in 64 bits; None where it takes too long."""
    kind = case["kind"]
    if kind == "prepare":
        n = case["n"]
        if n < 3 or n * case["layers"] * (case["sweeps"] + 1) * 2 ** max(n - 14, 0) > 4000:
            return None
        v = _gauss(_gen(seed, 3), 2 ** n)
        v = v / np.linalg.norm(v)
        if case["snake"]:
            v = np.concatenate([v[:2 ** (n - 1)], v[2 ** (n - 1):][::-1]])
        drop = int(case["compress"] / 100 * 2 ** n)
        if drop:
            v = v.copy()
            v[np.argsort(np.abs(v), kind="stable")[:drop]] = 0
        try:
            gates, fid = _encode(v, n, case["chi"], case["layers"], case["sweeps"])
        except ValueError:
            return None
        flat, qubits = [], []
        for layer in reversed(range(case["layers"])):
            for s in range(n):
                d = 2 * _width(n, s)
                flat.append(gates[layer, s, :d, :d].reshape(-1).numpy())
                qubits += [n - 1 - s] if d == 2 else [n - 2 - s, n - 1 - s]
        return {"gates": _after(case["sweeps"], np.concatenate(flat)), "qubits": np.array(qubits),
                "fidelity": float(fid[-1].abs())}
    if kind == "ragged":
        gates, widths, fid = [], [], []
        try:
            for k, (n, chi) in enumerate(_sizes(case)):
                v = _mps_states(n, 48, 1, seed + 1000 * k)[0].cpu().numpy()
                g, f = _encode(v, n, chi, case["layers"], case["sweeps"])
                gates.append(g.reshape(-1))
                fid.append(f)
                widths.append(_widths(1, case["layers"], n).reshape(-1))
        except ValueError:
            return None
        return {"gates": _after(case["sweeps"], torch.cat(gates)), "widths": torch.cat(widths),
                "layers_used": np.full(case["count"], case["layers"]), "fidelity": torch.cat(fid)}
    if kind == "chi":
        n = case["n"]
        if case["batch"] * 2.0 ** n * case["chi"] > 2.0 ** 27:
            return None
        v = prepare(case, seed)["states"].to(C128).cpu().numpy()
        v = v / np.linalg.norm(v, axis=1, keepdims=True)
        return {"psi": v, "target": np.stack([_truncate(x, n, case["chi"]) for x in v])}
    if kind == "layers":
        if case["batch"] * case["layers"] * 2.0 ** case["n"] > 2.0 ** 25:
            return None
        try:
            gates, amp0, rest = _extract(prepare(case, seed)["psi"].cpu(), case["n"], case["layers"])
        except ValueError:
            return None
        b, nl, n = case["batch"], case["layers"], case["n"]
        return {"gates": gates, "widths": _widths(b, nl, n), "used": torch.full((b,), nl, dtype=torch.int32),
                "amp0": amp0, "residual": rest}
    if kind == "sweep":
        psi, target, gates = _fit(case, seed)
        if case["dtype"] == "c64":
            target = target.to(C64).to(C128)
        if case["batch"] * case["sweeps"] * case["layers"] * case["n"] * 2.0 ** case["n"] > 2.0 ** 34:
            return None
        circuit, fid, over = _sweeps(target, gates, psi, case["n"], case["sweeps"])
        out = {"circuit": circuit, "fidelity": fid, "overlap": over}
        if case["dtype"] == "c128":
            out["gates"] = _after(case["sweeps"], gates)
        return out
    if kind == "circuit":
        st = prepare(case, seed)
        state = _circuit(st["gates"], case["n"])
        return {"state": state, "fidelity": _dot(st["psi"], state)}
    st = prepare(case, seed)
    return {"y": _mlp(st), "loss": None, "grads": None, "params": None}


def _mlp(st: dict) -> torch.Tensor:
    """The forward pass with its BF16 rounding points and 64-bit sums."""
    net, x = st["net"], st["x"].view(torch.bfloat16).double()
    i, w, o = net.in_dim, net.width, net.out_dim
    p, pb = net.params.double(), net.params.to(torch.bfloat16).double()
    at = 0
    for k, (a, b) in enumerate(((i, w), (w, w), (w, o))):
        x = x @ pb[at:at + a * b].reshape(a, b) + p[at + a * b:at + a * b + b]
        at += a * b + b
        if k < 2:
            x = x.relu().to(torch.bfloat16).double()
    return x
