"""A sweep's final states written over its inputs: results as with a buffer of
their own, whatever order the states finish in."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(n, used, layers, dtype, gpu):
    rng = np.random.default_rng(n)
    b = len(used)
    psi = rng.standard_normal((b, 2 ** n)) + 1j * rng.standard_normal((b, 2 ** n))
    psi /= np.linalg.norm(psi, axis=1, keepdims=True)
    gates = np.zeros((b, layers, n, 4, 4), dtype=np.complex128)
    widths = np.full((b, layers, n), 2, dtype=np.int32)
    widths[:, :, n - 1] = 1
    for i in np.ndindex(b, layers, n):
        d = 2 * widths[i]
        gates[i][:d, :d] = np.linalg.qr(rng.standard_normal((d, d)) + 1j * rng.standard_normal((d, d)))[0]
    to = lambda a: torch.from_numpy(a).to(gpu)
    return to(psi).to(dtype), to(gates), to(widths), torch.tensor(used, dtype=torch.int32, device=gpu)


@pytest.mark.parametrize("goal", [False, True])
@pytest.mark.parametrize("place", ["reference", "reference+1", "target", "target+1"])
@pytest.mark.parametrize("dtype", [torch.complex64, torch.complex128])
@pytest.mark.parametrize("n", [4, 6, 11, 14])
def test_output_over_the_inputs(gpu, n, dtype, place, goal):
    """Twelve states with 0 to 3 of 3 layers (those with fewer finish first; one
    block each up to N = 11, two half-batches in windows at 14), the output at
    the address of the fidelity reference or the target, or one state behind:
    then a state's output lies over inputs of others."""
    used = [3, 0, 2, 0, 1, 0, 3, 0, 1, 2, 0, 3]
    b, layers, sweeps = len(used), 3, 3
    psi, gates0, widths, lu = _inputs(n, used, layers, dtype, gpu)
    ref = psi.to(torch.complex128)
    limit, got = None, []
    for where in (["own"] if goal else []) + ["own", place]:
        target = torch.zeros((b + 1, 2 ** n), dtype=dtype, device=gpu)
        psi_ref = torch.zeros((b + 1, 2 ** n), dtype=torch.complex128, device=gpu)
        target[:b], psi_ref[:b] = psi, ref
        shift = 1 if where.endswith("+1") else 0
        if where == "own":
            out = torch.zeros((b, 2 ** n), dtype=dtype, device=gpu)
        elif where.startswith("target"):
            out = target[shift:b + shift]
        else:
            out = psi_ref.view(-1).view(dtype)[shift * 2 ** n:(b + shift) * 2 ** n].view(b, 2 ** n)
        fid = torch.zeros((b, sweeps + 1), dtype=torch.complex128, device=gpu)
        ov = torch.zeros((b, sweeps), dtype=torch.float64, device=gpu)
        done = torch.zeros(b, dtype=torch.int32, device=gpu)
        gates = gates0.clone()
        _sweep(n, b, layers, lu, sweeps, target, gates, widths, psi_ref, fid, ov, limit, done, out)
        if goal and limit is None:      # a run without a goal: one that the first, third, ... state meets early
            f = fid.abs()
            limit = ((f[:, 0] + f[:, 1]) / 2).contiguous()
            limit[1::2] = 2.0
        else:
            got.append((out.clone(), fid, ov, done, gates))
    for x, y in zip(*got):
        assert torch.equal(x, y)


def _sweep(n, b, layers, lu, sweeps, target, gates, widths, psi_ref, fid, ov, goal, done, out):
    """qmx_sweep with every buffer given (two streams in windows, as by default)."""
    from qmprs_amd import _lib
    lib, h = _lib.load(), _lib.handle()
    dt = _lib.QMX_C64 if target.dtype == torch.complex64 else _lib.QMX_C128
    ws = _lib.workspace(lib.qmx_sweep_workspace(n, b, dt), target.device)
    p = _lib.ptr
    st = lib.qmx_sweep(h, n, b, layers, p(lu), sweeps, p(target), dt, p(gates), p(widths), p(psi_ref), p(fid), p(ov),
                       p(goal), p(done), p(out), p(ws), ws.numel(), _lib.stream_ptr())
    _lib.check(st, h)
    torch.cuda.synchronize()
