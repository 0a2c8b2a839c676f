"""The gate update's polar factor on environments that are hard for it.

States close to a product state give environments whose singular values fall
like (1, e^2, e^2, e^4): the matrix iteration takes most of them, the Jacobi path
those that it leaves, and the layer next to |0..0> gives the rank-2 and rank-1
ones, which have closed forms.
"""

import numpy as np
import pytest
import torch

from oracle import qmprs_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 6, 10, 13])
@pytest.mark.parametrize("eps", [0.3, 0.03, 0.003])
def test_sweep_near_product_states(gpu, n, eps):
    """One and two complex128 sweeps against the oracle.  A gate is determined
    to eps_machine / sigma in a direction of singular value sigma, and the
    state has weight of order sqrt(sigma) there, so the circuit's state is
    determined to eps_machine / sqrt(sigma) ~ 1e-16 / e^2 = 1e-11 per gate;
    1e-9 leaves room for the at most 52 updates."""
    from qmprs_amd import engine
    rng = np.random.default_rng(100 * n + int(1000 * eps))
    prod = np.ones(1, dtype=np.complex128)
    for _ in range(n):
        v = rng.standard_normal(2) + 1j * rng.standard_normal(2)
        prod = np.kron(prod, v / np.linalg.norm(v))
    noise = rng.standard_normal(2 ** n) + 1j * rng.standard_normal(2 ** n)
    psi = O.ket(prod + eps * noise / np.linalg.norm(noise))
    layers = O.get_unitary_layers(psi, n, 2)
    g, w = engine.layers_to_arrays(layers, n)
    gl = O.layer_gate_list(layers)
    for sweeps in (1, 2):
        trace = []
        ref = O.circuit_state(n, O.optimize_gate_list(psi, n, gl, sweeps, trace))
        gates = torch.from_numpy(g).to(gpu).unsqueeze(0).contiguous()
        widths = torch.from_numpy(w).to(gpu).unsqueeze(0).contiguous()
        used = torch.tensor([g.shape[0]], dtype=torch.int32, device=gpu)
        target = torch.from_numpy(psi).to(gpu).unsqueeze(0).contiguous()
        res = engine.sweep(target, gates, widths, used, sweeps, circuit_out=True)
        got, ws = gates[0].cpu().numpy(), widths[0].cpu().numpy()
        for layer in range(g.shape[0]):
            for s in range(n):
                d = 4 if ws[layer, s] == 2 else 2
                u = got[layer, s, :d, :d]
                assert np.abs(u @ u.conj().T - np.eye(d)).max() < 1e-12
        np.testing.assert_allclose(res.overlap[0].cpu().numpy(), np.abs(trace), rtol=1e-10)
        err = np.linalg.norm(res.circuit[0].cpu().numpy() - ref)
        print(f"n={n} eps={eps} sweeps={sweeps} state err {err:.2e}")
        assert err < 1e-9
