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


def _centroid_split(pg):
    """Every tetrahedron split into four around its centroid: the four neighbour each other, so their
    elimination updates off-diagonal blocks as well (no box mesh has two neighbours of a cell adjacent)."""
    tet = np.flatnonzero(pg.sE == fa.TET)
    rest = np.flatnonzero(pg.sE != fa.TET)
    nd = pg.iNE[tet][:, :4]
    centre = len(pg.pN) + np.arange(len(tet))
    kids = np.repeat(nd[:, None, :], 4, 1)
    for v in range(4):
        kids[:, v, v] = centre
    iNE = -np.ones((4 * len(tet) + len(rest), pg.iNE.shape[1]), np.int32)
    iNE[:4 * len(tet), :4] = kids.reshape(-1, 4)
    iNE[4 * len(tet):] = pg.iNE[rest]
    n4 = 4 * len(tet)
    return fa.PolyGrid(np.concatenate([pg.pN, pg.pN[nd].mean(1)]),
                       np.concatenate([np.full(n4, fa.TET), pg.sE[rest]]),
                       np.concatenate([np.full(n4, 4), pg.nNE[rest]]), iNE,
                       np.concatenate([np.zeros(n4, int), pg.gid[rest]]))


@pytest.mark.parametrize("flags,tol", [(0, 1e-10), (fa.PREC_FP32, 1e-5)])
@pytest.mark.parametrize("dims,split", [((1, 1, 1), True), ((3, 2, 2), True), ((6, 4, 4), True), ((13, 3, 3), False)])
def test_block_ilu_factorisation_matches_oracle(cuda, dims, split, flags, tol):
    """The level kernel's rows (five lanes each, 48 to a workgroup) on levels of a few rows, with and
    without updates of other blocks of the row, at a gamma where the off-diagonal blocks matter.  The
    tolerances are the ILU tests' own: FP64 1e-10, FP32 factors 1e-5 (100 roundings of 6e-8 to 1e-7)."""
    print(f"[case] block ilu factorisation dims={dims} split={split} flags={flags}", flush=True)
    pg = M.box(*dims, 1.0, 0.5, 0.5, jitter=0.2, seed=3)
    if split:
        pg = _centroid_split(pg)
        pg.renumber(fa.RENUMBER_CHUNKS)
    fv = pg.up()
    og = O.Grid(pg.pN, pg.sE, pg.nNE, pg.iNE, pg.gid)
    cg, ct, cp = M.conds("mixed")
    bc = O.BC(og, cg, ct, cp, r=M.R, gamm=M.GAMMA)
    nC = og.nC
    nb = np.where((og.neib >= 0) & (og.neib < nC), og.neib, -1)
    triangles = sum(k >= 0 and len(set(nb[k]) & set(nb[c]) - {-1}) > 0 for c in range(nC) for k in nb[c])
    assert (triangles > 0) == split
    x = M.perturbed_state(og.p[:nC], mach=0.6, seed=8)
    jac = O.find_euler_jac(og, *O.element_state(og, bc, x), M.GAMMA)
    eu = fa.Euler(fv, fa.CondTab(cg, ct, cp), r=M.R, gamma=M.GAMMA, flags=flags)
    y, r = _dev(x), np.random.default_rng(3).standard_normal(5 * nC)
    z = y.clone()
    order = eu.ilu_order()
    for jok, gamma in ((0, 0.1 * np.cbrt(og.v.mean())), (1, 0.02 * np.cbrt(og.v.mean()))):
        assert eu.psetup(y, y, gamma, jok=jok) == 1 - jok
        eu.psolve(_dev(r), z, gamma)
        err = M.rel(z.cpu().numpy(), O.Bilu(og, jac, gamma, order=order).solve(r))
        print(f"  gamma {gamma:.2e}: relative error {err:.2e}")
        assert err <= tol


@pytest.mark.parametrize("flags", [0, fa.PREC_FP32], ids=["fp64", "mixed"])
@pytest.mark.parametrize("dims", [(1, 1, 1), (11, 2, 2), (40, 10, 10), (32, 27, 20), (45, 45, 44)],
                         ids=["6", "264", "24000", "103680", "534600"])
def test_block_ilu_solve_in_one_launch_equals_colour_launches(cuda, dims, flags, monkeypatch):
    """The single-launch solve (a partial chunk; fewer and more items than resident workgroups) and, past
    its size limit, the recorded colour launches, against colour launches one by one: bitwise, over
    repeated applies (the two copies of the exchange alternate), in place, and after a non-finite
    right-hand side, which is reported and leaves nothing behind."""
    import torch
    print(f"[case] block ilu one launch dims={dims} flags={flags}", flush=True)
    pg = M.box(*dims, 1.0, 0.5, 0.5, jitter=0.2, seed=3, renumber=fa.RENUMBER_CHUNKS)
    fv = pg.up()
    ctab = fa.CondTab(*M.conds("mixed"))
    nC = fv.nC
    y = _dev(M.perturbed_state(fv.p[:nC], mach=0.6, seed=8))
    gamma = 0.1 * np.cbrt(fv.v.mean())
    monkeypatch.setenv("FOS_ILU_EAGER", "1")
    eager = fa.Euler(fv, ctab, r=M.R, gamma=M.GAMMA, flags=flags)
    assert eager.psetup(y, y, gamma) == 1
    monkeypatch.delenv("FOS_ILU_EAGER")
    eu = fa.Euler(fv, ctab, r=M.R, gamma=M.GAMMA, flags=flags)
    assert eu.psetup(y, y, gamma) == 1
    rng = np.random.default_rng(11)
    for k in range(5):
        r = _dev(rng.standard_normal(5 * nC))
        ze, z = torch.zeros_like(r), torch.zeros_like(r)
        eager.psolve(r, ze, gamma)
        eu.psolve(r, z, gamma)
        assert torch.equal(ze, z), (k, float((ze - z).abs().max()))
        assert float(z.norm()) > 0
        eu.psolve(r, r, gamma)
        assert torch.equal(ze, r)
        if k == 2:
            bad = _dev(rng.standard_normal(5 * nC))
            bad[nC // 2] = float("nan")
            with pytest.raises(RuntimeError, match="non-finite"):
                eu.psolve(bad, z, gamma)


@pytest.mark.parametrize("start,size", [(0, 1), (7, 33), (256, 517), (3, 1200), (0, 1536)])
def test_learned_gradient_of_a_batch_matches_oracle(cuda, start, size):
    """The backward pass on batches that are no multiple of its tiles (16 rows), staged steps (32) or
    slices (512), from an odd first cell, per parameter block against the FP64 oracle on the batch's
    sub-mesh.  Tolerance 5e-2: eight BF16 roundings of 2^-9 lie between the inputs and a gradient
    (1.6e-2 if they all agree in sign), times three for blocks whose cells cancel."""
    print(f"[case] learned gradient start={start} size={size}", flush=True)
    from tests.test_gpu_learned import BLOCKS, _random_params, bf16
    _pg, fv, og, _bc, ctab = M.setup(16, 4, 4, kind="mixed")
    nC = og.nC
    assert nC == 1536
    y = _dev(M.perturbed_state(og.p[:nC], mach=0.7, seed=6, width=0.2))
    eu = fa.Euler(fv, ctab, r=M.R, gamma=M.GAMMA)
    p = _random_params(eu, 5)
    gamma = 0.02
    X, S = eu.learned_inputs(y, gamma)
    rng = np.random.default_rng(1)
    r = rng.standard_normal(5 * nC) * np.repeat(S, nC)
    delta = 0.5 * r + 0.1 * rng.standard_normal(5 * nC) * np.repeat(S, nC)
    cells = slice(start, start + size)
    nb = np.asarray(og.neib[cells])
    nb = np.where((nb >= start) & (nb < start + size), nb - start, -1).astype(np.int32)

    def part(v):
        return np.ascontiguousarray(v.reshape(5, nC)[:, cells]).ravel()
    loss_o, g_o = O.mlp_loss_grad(np.ascontiguousarray(X[cells]), np.ascontiguousarray(nb), bf16(p), S, part(r),
                                  part(delta), np.ones(size, np.int32))
    loss, g = eu.learned_loss_grad(y, _dev(r), _dev(delta), gamma, start, size)
    assert abs(loss - loss_o) <= 2e-2 * loss_o
    worst = {k: M.rel(g[a:a + n].astype(np.float64), g_o[a:a + n]) for k, (a, n) in BLOCKS.items()}
    print("  " + " ".join(f"{k} {e:.1e}" for k, e in worst.items()))
    assert max(worst.values()) <= 5e-2
    loss2, g2 = eu.learned_loss_grad(y, _dev(r), _dev(delta), gamma, start, size)
    assert loss2 == loss and np.array_equal(g, g2)


def _torch_learned_gradient(X, nbr, par, S, r, delta, device):
    """Loss and gradient of the learned preconditioner in plain FP64 torch (oracle/learned.c's definition,
    for batches that the oracle's single thread takes too long for).  nbr: cells of the batch or -1."""
    import torch
    from tests.test_gpu_learned import BLOCKS, NH, NI, NO
    n = len(X)
    P = torch.tensor(np.asarray(par, np.float64), device=device, requires_grad=True)
    shape = {"W0": (NI, NH), "W1": (2 * NH, NH), "W2": (2 * NH, NH), "W3": (NH, NO)}
    W = {k: P[a:a + m].view(shape.get(k, (m,))) for k, (a, m) in BLOCKS.items()}
    nb = torch.tensor(np.where(nbr < 0, n, nbr).astype(np.int64), device=device)
    cnt = (nb < n).sum(1, keepdim=True).clamp(min=1)

    def at(h, j):
        return torch.cat([h, h.new_zeros(1, h.shape[1])]).index_select(0, nb[:, j])

    def hidden(h, k):
        m = (at(h, 0) + at(h, 1) + at(h, 2) + at(h, 3)) / cnt
        return torch.nn.functional.silu(torch.cat([h, m], 1) @ W["W" + k] + W["b" + k])
    x = torch.tensor(np.asarray(X, np.float64), device=device)
    h = torch.nn.functional.silu(x @ W["W0"] + W["b0"])
    kappa = (x[:, 18] * (1.0 + x[:, 19])).clamp(max=1.0)
    o = (hidden(hidden(h, "1"), "2") @ W["W3"] + W["b3"]) * kappa[:, None]
    sc = torch.tensor(np.asarray(S, np.float64), device=device)
    rh, dh = r.view(5, n).T / sc, delta.view(5, n).T / sc
    t = rh + (o[:, :25].reshape(n, 5, 5) * rh[:, None, :]).sum(2)
    z = (1.0 + o[:, 29:30]) * t + sum(o[:, 25 + j:26 + j] * at(t, j) for j in range(4))
    loss = ((z - dh) ** 2).sum() / n
    loss.backward()
    return float(loss.detach()), P.grad.cpu().numpy()


def test_learned_gradient_after_a_larger_batch(cuda):
    """Batches past 131,072 rows, where a slice is more than 512 rows (140,001 rows: 244 slices), then on the
    same context a smaller batch with more slices (130,001 rows: 254): against the plain arithmetic with
    the batch tests' tolerance (5e-2, derived there), and the second bitwise a fresh context's."""
    import torch
    from tests.test_gpu_learned import BLOCKS, _random_params, bf16
    pg = M.box(30, 28, 28, 1.0, 0.5, 0.5, jitter=0.2, seed=3, renumber=fa.RENUMBER_CHUNKS)
    fv = pg.up()
    ctab = fa.CondTab(*M.conds("mixed"))
    nC = fv.nC
    assert nC == 141120
    y = _dev(M.perturbed_state(fv.p[:nC], mach=0.7, seed=6, width=0.2))
    gamma, start = 0.02, 7
    nb0 = np.asarray(fv.neib)

    def context():
        eu = fa.Euler(fv, ctab, r=M.R, gamma=M.GAMMA)
        return eu, _random_params(eu, 5)
    eu, p = context()
    X, S = eu.learned_inputs(y, gamma)
    rng = np.random.default_rng(1)
    r = rng.standard_normal(5 * nC) * np.repeat(S, nC)
    delta = 0.5 * r + 0.1 * rng.standard_normal(5 * nC) * np.repeat(S, nC)
    r, delta = _dev(r), _dev(delta)
    for size in (140_001, 130_001):
        print(f"[case] learned gradient start={start} size={size}", flush=True)
        cells = slice(start, start + size)
        nb = np.where((nb0[cells] >= start) & (nb0[cells] < start + size), nb0[cells] - start, -1)
        loss_t, g_t = _torch_learned_gradient(X[cells], nb, bf16(p), S, r.view(5, nC)[:, cells].reshape(-1),
                                              delta.view(5, nC)[:, cells].reshape(-1), y.device)
        loss, g = eu.learned_loss_grad(y, r, delta, gamma, start, size)
        assert abs(loss - loss_t) <= 2e-2 * loss_t
        worst = {k: M.rel(g[a:a + n].astype(np.float64), g_t[a:a + n]) for k, (a, n) in BLOCKS.items()}
        print("  " + " ".join(f"{k} {e:.1e}" for k, e in worst.items()))
        assert max(worst.values()) <= 5e-2
    fresh, _p = context()
    loss_f, g_f = fresh.learned_loss_grad(y, r, delta, gamma, start, size)
    assert loss == loss_f and np.array_equal(g, g_f)


@pytest.mark.parametrize("dims", [(1, 1, 1), (11, 1, 1), (13, 3, 3), (40, 10, 10)], ids=["6", "66", "702", "24000"])
def test_learned_apply_matches_oracle_at_tile_edges(cuda, dims):
    """Inference (features, fused layers, apply) where the last 64-row group or 16-row tile is partial and
    where a wave walks one tile or several; the learned tests' own BF16 tolerance of 3e-2."""
    import torch
    print(f"[case] learned apply dims={dims}", flush=True)
    from tests.test_gpu_learned import _cells_nbr, _random_params, bf16
    _pg, fv, og, _bc, ctab = M.setup(*dims, kind="mixed")
    nC = og.nC
    y = _dev(M.perturbed_state(og.p[:nC], mach=0.7, seed=4, width=0.2))
    eu = fa.Euler(fv, ctab, r=M.R, gamma=M.GAMMA)
    p = _random_params(eu, 3)
    gamma = 0.02
    X, S = eu.learned_inputs(y, gamma)
    r = np.random.default_rng(0).standard_normal(5 * nC) * np.repeat(S, nC)
    nbr = _cells_nbr(og)
    zref = O.mlp_apply(O.mlp_forward(X, nbr, bf16(p)), nbr, S, r)
    z = torch.zeros_like(y)
    for _ in range(2):
        eu.psetup_learned(y, gamma)
        eu.psolve_learned(_dev(r), z)
        err = M.rel(z.cpu().numpy(), zref)
        print(f"  relative error {err:.2e}")
        assert err <= 3e-2
        eu.learned_loss_grad(y, _dev(r), _dev(r), gamma, 0, min(nC, 100))  # training overwrites the rows


@pytest.mark.parametrize("precond", ["ilu", None])
def test_integrator_reports_a_nonfinite_product_like_the_callback(cuda, precond):
    """A state whose squares overflow FP32 but not FP64: the Newton residual is finite, the mixed-precision
    product inside GMRES is not.  With the fused product (checked at GMRES's next wait) and without (checked
    by the callback itself) the step fails as recoverable, with the state and the counters of iterations
    unchanged and nothing left behind: the next good step is the one a fresh context takes."""
    import torch
    from fosolvers_amd import _capi
    print(f"[case] non-finite product in GMRES precond={precond}", flush=True)
    pg = M.box(8, 4, 4, jitter=0.2, seed=3, renumber=fa.RENUMBER_CHUNKS)
    fv = pg.up()
    ctab = fa.CondTab(*M.conds("wall"))
    good = _dev(M.perturbed_state(fv.p[:fv.nC], mach=0.3, seed=5))
    scale = torch.ones(5, fv.nC, dtype=torch.float64, device="cuda")
    scale[0], scale[1:4], scale[4] = 1e-30, 1e-5, 1e20  # u ~ 1e25: finite in FP32 until it is squared
    huge = (good.view(5, -1) * scale).reshape(-1).contiguous()
    outs, fails = [], []
    for fused in (True, False, None):
        eu = fa.Euler(fv, ctab, r=M.R, gamma=M.GAMMA, flags=fa.PREC_FP32)
        b = fa.BDFNewtonKrylov.for_euler(eu, maxl=20, precond=precond, jtimes="analytic", fused=bool(fused))
        b.set_newton(tol=1e-8, max_iter=20, lin_tol=1e-3, max_restarts=10)
        y = torch.zeros_like(good)
        if fused is not None:
            b.set_dt(1e-28)
            b.set_iv(0.0, huge)
            rc, _t = b.step(0.0, y)
            assert rc == 1 and "non-finite" in _capi.last_error(), (rc, _capi.last_error())
            fails.append(b.stats()["nli"])
            assert not eu.nonfinite()
        b.set_dt(1e-3)
        b.set_iv(0.0, good)
        assert b.step(0.0, y)[0] == 0
        outs.append(y.clone())
    assert fails[0] == fails[1]
    assert M.rel(outs[0].cpu().numpy(), outs[2].cpu().numpy()) <= 1e-13
    assert M.rel(outs[1].cpu().numpy(), outs[2].cpu().numpy()) <= 1e-13


@pytest.mark.parametrize("precond", ["ilu", "bjac", None])
def test_integrator_names_the_nonfinite_callback(cuda, precond):
    """A product that overflows is named, also where a preconditioner solve of its result was launched before
    GMRES's wait, and no counter counts that solve: the integrator's and the context's counters are those
    of the callbacks that check for themselves.  State and step: the factors' largest entries (2e35) fit
    FP32, the enthalpy (2e40) that the product forms does not."""
    from fosolvers_amd import _capi
    import torch
    print(f"[case] name of a non-finite callback precond={precond}", flush=True)
    pg = M.box(8, 4, 4, jitter=0.2, seed=3, renumber=fa.RENUMBER_CHUNKS)
    fv = pg.up()
    ctab = fa.CondTab(*M.conds("wall"))
    good = _dev(M.perturbed_state(fv.p[:fv.nC], mach=0.3, seed=5))
    scale = torch.ones(5, fv.nC, dtype=torch.float64, device="cuda")
    scale[0], scale[4] = 1e-20, 1e20
    huge = (good.view(5, -1) * scale).reshape(-1).contiguous()
    counts = []
    for fused, name in ((True, "newton_matvec_analytic"), (False, "jtimes_analytic")):
        eu = fa.Euler(fv, ctab, r=M.R, gamma=M.GAMMA, flags=fa.PREC_FP32)
        b = fa.BDFNewtonKrylov.for_euler(eu, maxl=20, precond=precond, jtimes="analytic", fused=fused)
        b.set_newton(tol=1e-8, max_iter=20, lin_tol=1e-3, max_restarts=10)
        b.set_dt(1e-26)
        b.set_iv(0.0, huge)
        assert b.step(0.0, torch.zeros_like(good))[0] == 1
        assert _capi.last_error() == f"{name}: non-finite value in the result"
        st = b.stats()
        counts.append(({k: st[k] for k in ("nfe", "nli", "npe", "nps", "njv")}, list(eu.counters())))
    print(f"  {counts[0]}")
    assert counts[0] == counts[1] and counts[0][0]["njv"] == 1


def test_integrator_names_the_nonfinite_solve(cuda):
    """A preconditioner whose output overflows FP32 on a good state: the solve is named and counted, and no
    product was formed."""
    from fosolvers_amd import _capi
    from tests.test_gpu_learned import BLOCKS, _random_params
    import torch
    print("[case] name of a non-finite solve", flush=True)
    pg = M.box(8, 4, 4, jitter=0.2, seed=3, renumber=fa.RENUMBER_CHUNKS)
    fv = pg.up()
    eu = fa.Euler(fv, fa.CondTab(*M.conds("wall")), r=M.R, gamma=M.GAMMA)
    p = _random_params(eu, 5)
    a, n = BLOCKS["b3"]
    p[a:a + n] = 3e38  # an output of this size times itself overflows
    eu.learned_set_params(p)
    b = fa.BDFNewtonKrylov.for_euler(eu, maxl=20, precond="learned", jtimes="analytic")
    b.set_newton(tol=1e-8, max_iter=20, lin_tol=1e-3, max_restarts=10)
    b.set_dt(1e-3)
    good = _dev(M.perturbed_state(fv.p[:fv.nC], mach=0.3, seed=5))
    b.set_iv(0.0, good)
    assert b.step(0.0, torch.zeros_like(good))[0] == 1
    assert _capi.last_error() == "psolve_learned: non-finite value in the result"
    st = b.stats()
    assert (st["nps"], st["njv"], st["nli"]) == (1, 0, 0) and not eu.nonfinite()


@pytest.mark.parametrize("kind", ["mixed", "wall"])
@pytest.mark.parametrize("dims", [(1, 1, 1), (43, 2, 3), (31, 27, 26), (33, 27, 26)],
                         ids=["6", "1548", "130572", "138996"])
def test_residual_on_either_side_of_the_small_mesh_rule(cuda, dims, kind):
    """The tetrahedral FP64 residual and difference quotient with the ghost states formed in the face pass
    (up to 512 chunks) and by their own launch (beyond), against the generic layout, which forms both
    from other geometry data: 1e-12 relative, the bound of the residual tests; the quotient amplifies the
    residual's rounding (1e-16) by 1 / sigma (~1e6 with these vectors), so 1e-9."""
    import torch
    print(f"[case] small-mesh rule dims={dims} kind={kind}", flush=True)
    pg = M.box(*dims, 1.0, 0.5, 0.5, jitter=0.2, seed=3, renumber=fa.RENUMBER_CHUNKS)
    fv = pg.up()
    ctab = fa.CondTab(*M.conds(kind))
    y = _dev(M.perturbed_state(fv.p[:fv.nC], mach=0.6, amp=0.3, seed=5))
    v = _dev(np.random.default_rng(2).standard_normal(5 * fv.nC)) * (y.abs() + 0.1) * 1e-3
    out = []
    for flags in (0, fa.LAYOUT_GENERIC):
        eu = fa.Euler(fv, ctab, r=M.R, gamma=M.GAMMA, flags=flags)
        assert eu.layout == (0 if flags else 1)
        f, jv = torch.zeros_like(y), torch.zeros_like(y)
        eu.rhs(y, f)
        eu.jtimes(v, jv, y, f)
        out.append((f.cpu().numpy(), jv.cpu().numpy()))
    ef, ej = M.rel(out[0][0], out[1][0]), M.rel(out[0][1], out[1][1])
    print(f"  residual {ef:.1e}, quotient {ej:.1e}")
    assert ef <= 1e-12 and ej <= 1e-9
