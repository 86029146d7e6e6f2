"""Edge sizes of kernels that split their work by chunk, tile or batch, against the FP64 oracle or the
plain arithmetic they stand for.  Each tolerance is stated with its derivation."""
import numpy as np
import pytest

import fosolvers_amd as fa
from oracle import oracle as O
from tests import meshes as M

pytestmark = pytest.mark.gpu


def _dev(a, dtype=None):
    import torch
    return torch.tensor(np.asarray(a), dtype=dtype or torch.float64, device="cuda")


@pytest.mark.parametrize("dims", [(1, 1, 1), (11, 2, 2), (8, 5, 5)], ids=["6", "264", "1200"])
@pytest.mark.parametrize("kind", ["mixed", "wall"])
def test_fp32_residual_gathers_faces_by_slot(cuda, dims, kind):
    """The FP32 residual of the tetrahedral layout: one partial chunk, a chunk and 8 cells, several.
    Within 2e-5 relative of the FP64 oracle (the bound of every FP32 residual test: 1e-7 per flux,
    amplified by the cancellation of a cell's fluxes), and bitwise the same from run to run."""
    import torch
    print(f"[case] fp32 residual dims={dims} kind={kind}", flush=True)
    _pg, fv, og, bc, ctab = M.setup(*dims, kind=kind)
    x = M.perturbed_state(og.p[:og.nC], mach=0.6, amp=0.3, seed=5)
    ref = O.rhs(og, bc, x)
    eu = fa.Euler(fv, ctab, r=M.R, gamma=M.GAMMA)
    assert eu.layout == 1
    y = _dev(x, torch.float32)
    out = [torch.zeros_like(y) for _ in range(3)]
    for o in out:
        eu.rhs_f32(y, o)
    err = M.rel(out[0].double().cpu().numpy(), ref)
    print(f"  relative error {err:.2e}")
    assert err <= 2e-5
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])
