"""GPU: differentiable unrolled PDHG (cuOptAmdUnrolled* through cuopt_amd.autograd)
against the CPU restatement oracle/unrolled.py, central finite differences of the
FP64 GPU map (h = 1e-6) and the envelope identities at convergence.

Tolerances: FP64 forward / VJP vs oracle 1e-9 relative (summation order is the
same, sequential per row); FP32 forward / VJP vs the FP64 oracle 2e-3 relative
(FP32 iterates over K steps); FD vs FP64 VJP 1e-6 relative."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from cuopt_amd import generators as G  # noqa: E402
from cuopt_amd.autograd import UnrolledPDHG  # noqa: E402
from oracle import unrolled as U  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = "cuda"


def problem(seed=0, m=200, n=500):
    lp = G.random_lp(m=m, n=n, seed=seed)
    return lp, lp.to_scipy()


def relerr(a, b):
    return float(np.max(np.abs(a - b)) / (1.0 + np.max(np.abs(b))))


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-9), ("fp32_mixed", 2e-3)])
def test_forward_and_vjp_match_oracle(precision, tol):
    lp, A = problem(0)
    B, K, every, lam = 8, 100, 7, 1e-3
    op = UnrolledPDHG(lp, ridge=lam, steps=K, checkpoint_every=every, precision=precision)
    eta = op.step_size
    assert abs(eta - U.step_sizes(A)) <= 1e-6 * eta
    rng = np.random.default_rng(0)
    c = lp.c[None, :] + 0.1 * rng.normal(size=(B, lp.n))
    b = lp.con_lb.copy()
    ct = torch.tensor(c, device=DEV, requires_grad=True)
    bt = torch.tensor(b, device=DEV, requires_grad=True)
    x, y = op(ct, bt)
    xo, yo, xs, ys = U.forward(A, c.T.copy(), b, b, lp.var_lb, lp.var_ub, lam, eta, K, keep=True)
    assert relerr(x.detach().cpu().numpy().T, xo) < tol
    assert relerr(y.detach().cpu().numpy().T, yo) < tol
    target = rng.uniform(0, 1, size=(B, lp.n))
    loss = ((x - torch.tensor(target, device=DEV)) ** 2).sum() + (y ** 2).sum()
    loss.backward()
    gc, glc, guc = U.backward(A, b, b, lp.var_lb, lp.var_ub, lam, eta, xs, ys, 2 * (xo - target.T), 2 * yo)
    assert relerr(ct.grad.cpu().numpy().T, gc) < tol
    assert relerr(bt.grad.cpu().numpy(), (glc + guc).sum(axis=1)) < tol


def test_ranged_rows_vjp_matches_oracle():
    lp, A = problem(1, m=120, n=300)
    B, K, every, lam = 4, 60, 9, 1e-3
    rng = np.random.default_rng(1)
    lc = np.tile(lp.con_lb - rng.uniform(0, 0.5, size=lp.m), (B, 1))
    uc = np.tile(lp.con_ub + rng.uniform(0, 0.5, size=lp.m), (B, 1))
    op = UnrolledPDHG(lp, ridge=lam, steps=K, checkpoint_every=every, precision="fp64")
    eta = op.step_size
    c = lp.c[None, :] + 0.1 * rng.normal(size=(B, lp.n))
    ct = torch.tensor(c, device=DEV, requires_grad=True)
    lt = torch.tensor(lc, device=DEV, requires_grad=True)
    ut = torch.tensor(uc, device=DEV, requires_grad=True)
    x, _ = op(ct, lt, ut)
    gx = rng.normal(size=(B, lp.n))
    (x * torch.tensor(gx, device=DEV)).sum().backward()
    xo, yo, xs, ys = U.forward(A, c.T.copy(), lc.T.copy(), uc.T.copy(), lp.var_lb, lp.var_ub, lam, eta, K, keep=True)
    gc, glc, guc = U.backward(A, lc.T.copy(), uc.T.copy(), lp.var_lb, lp.var_ub, lam, eta, xs, ys, gx.T.copy())
    assert relerr(ct.grad.cpu().numpy().T, gc) < 1e-9
    assert relerr(lt.grad.cpu().numpy().T, glc) < 1e-9
    assert relerr(ut.grad.cpu().numpy().T, guc) < 1e-9


def ragged_lp(seed=3, m=150, n=400):
    """Equality LP whose rows and columns have uneven lengths: empty rows and columns,
    rows of 1-3 nonzeros, and rows and columns far longer than a wavefront's 64-entry
    index load (so the SpMM kernels' row runs cross load and gather-group boundaries)."""
    import scipy.sparse as sp
    rng = np.random.default_rng(seed)
    rows, cols = [], []
    for i in range(m):
        k = 0 if i % 17 == 5 else (int(rng.integers(90, 140)) if i % 23 == 7 else int(rng.integers(1, 4)))
        live = np.flatnonzero(np.arange(n) % 31 != 11)  # every 31st column stays empty
        rows += [i] * k
        cols += list(rng.choice(live, size=k, replace=False))
    heavy = 3  # one column that many rows share
    for i in range(0, m, 2):
        if i % 17 != 5:
            rows.append(i)
            cols.append(heavy)
    A = sp.csr_matrix((rng.normal(size=len(rows)), (rows, cols)), shape=(m, n))
    A.sum_duplicates()
    A.sort_indices()
    x0 = rng.uniform(0, 1, size=n)
    b = A @ x0
    lp = G.LP(m=m, n=n, row_offsets=A.indptr.astype(np.int32), col_indices=A.indices.astype(np.int32),
              values=A.data.astype(np.float64), c=rng.normal(size=n), con_lb=b.copy(), con_ub=b.copy(),
              var_lb=np.zeros(n), var_ub=np.full(n, 10.0))
    return lp, A


@pytest.mark.parametrize("rows_per_wave", [1, 2, 4])
@pytest.mark.parametrize("B", [5, 70])
def test_rows_per_wavefront_forms_match_oracle(monkeypatch, rows_per_wave, B):
    # The SpMM kernels give each wavefront 1, 2 or 4 consecutive rows (chosen from the
    # matrix's shape; forced here).  Every form adds each row's products in increasing
    # order, so FP64 forward and VJP match the oracle to 1e-9 on a ragged matrix, with
    # batch sizes below and above one wavefront.
    monkeypatch.setenv("CUOPT_AMD_UNR_RPW_A", str(rows_per_wave))
    monkeypatch.setenv("CUOPT_AMD_UNR_RPW_T", str(rows_per_wave))
    lp, A = ragged_lp()
    assert np.diff(lp.row_offsets).max() > 64 and np.diff(A.tocsc().indptr).max() > 64
    assert (np.diff(lp.row_offsets) == 0).any() and (np.diff(A.tocsc().indptr) == 0).any()
    K, every, lam = 40, 7, 1e-3
    op = UnrolledPDHG(lp, ridge=lam, steps=K, checkpoint_every=every, precision="fp64")
    eta = op.step_size
    rng = np.random.default_rng(rows_per_wave * 100 + B)
    c = lp.c[None, :] + 0.1 * rng.normal(size=(B, lp.n))
    b = lp.con_lb.copy()
    print(f"ragged unrolled R={rows_per_wave} B={B}", flush=True)
    ct = torch.tensor(c, device=DEV, requires_grad=True)
    bt = torch.tensor(b, device=DEV, requires_grad=True)
    x, y = op(ct, bt)
    xo, yo, xs, ys = U.forward(A, c.T.copy(), b, b, lp.var_lb, lp.var_ub, lam, eta, K, keep=True)
    assert relerr(x.detach().cpu().numpy().T, xo) < 1e-9
    assert relerr(y.detach().cpu().numpy().T, yo) < 1e-9
    target = rng.uniform(0, 1, size=(B, lp.n))
    loss = ((x - torch.tensor(target, device=DEV)) ** 2).sum() + (y ** 2).sum()
    loss.backward()
    gc, glc, guc = U.backward(A, b, b, lp.var_lb, lp.var_ub, lam, eta, xs, ys, 2 * (xo - target.T), 2 * yo)
    assert relerr(ct.grad.cpu().numpy().T, gc) < 1e-9
    assert relerr(bt.grad.cpu().numpy(), (glc + guc).sum(axis=1)) < 1e-9


def test_vjp_matches_central_differences_fp64():
    # Sized so that no clamp of the K steps switches within +-h along the test
    # directions (the map is piecewise linear; at 300 x 750 x 200 steps some do,
    # and only h -> 0 recovers the derivative).
    lp, A = problem(2, m=100, n=250)
    B, K, lam, h = 2, 100, 1e-3, 1e-6
    op = UnrolledPDHG(lp, ridge=lam, steps=K, checkpoint_every=14, precision="fp64")
    rng = np.random.default_rng(2)
    c = torch.tensor(lp.c[None, :] + 0.1 * rng.normal(size=(B, lp.n)), device=DEV, requires_grad=True)
    b = torch.tensor(lp.con_lb, device=DEV, requires_grad=True)
    target = torch.tensor(rng.uniform(0, 1, size=(B, lp.n)), device=DEV)

    def loss(cc, bb):
        x, _ = op(cc, bb)
        return ((x - target) ** 2).sum()

    loss(c, b).backward()
    gc, gb = c.grad.clone(), b.grad.clone()
    with torch.no_grad():
        for _ in range(3):
            vc = torch.tensor(rng.normal(size=(B, lp.n)), device=DEV)
            fd = (loss(c + h * vc, b) - loss(c - h * vc, b)).item() / (2 * h)
            assert abs(fd - (gc * vc).sum().item()) <= 1e-6 * (1 + abs(fd))
            vb = torch.tensor(rng.normal(size=lp.m), device=DEV)
            fd = (loss(c, b + h * vb) - loss(c, b - h * vb)).item() / (2 * h)
            assert abs(fd - (gb * vb).sum().item()) <= 1e-6 * (1 + abs(fd))


def test_envelope_gradients_at_convergence():
    lp, A = problem(3, m=100, n=250)
    lam, K = 1e-2, 20000
    op = UnrolledPDHG(lp, ridge=lam, steps=K, checkpoint_every=141, precision="fp64")
    c = torch.tensor(lp.c[None, :], device=DEV, requires_grad=True)
    b = torch.tensor(lp.con_lb, device=DEV, requires_grad=True)
    x, y = op(c, b)
    obj = (c * x).sum() + 0.5 * lam * (x * x).sum()
    obj.backward()
    assert torch.allclose(c.grad, x.detach(), atol=1e-8)  # d obj / d c = x*
    assert torch.allclose(b.grad, y.detach()[0], atol=1e-8 * (1 + y.abs().max().item()))  # d obj / d b = y*


@pytest.mark.parametrize("precision", ["fp64", "fp32_mixed"])
def test_optimal_batch_size_on_device(precision):
    # The device-timed search returns a size the search can visit; one member is
    # always one, and the forward pass still matches the oracle at that size.
    lp, A = problem(1, m=1000, n=2500)
    op = UnrolledPDHG(lp, ridge=1e-3, steps=20, checkpoint_every=5, precision=precision)
    assert op.optimal_batch_size(1) == 1
    b = op.optimal_batch_size(512)
    visited = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64, 96, 128, 192, 256, 384, 512}
    assert b in visited, b
    c = np.tile(lp.c, (b, 1))
    x, _ = op(torch.tensor(c, device=DEV), torch.tensor(lp.con_lb, device=DEV), torch.tensor(lp.con_ub, device=DEV))
    xo, _ = U.forward(A, c.T, lp.con_lb, lp.con_ub, lp.var_lb, lp.var_ub, 1e-3, op.step_size, 20)
    assert relerr(x.cpu().numpy(), xo.T) < (1e-9 if precision == "fp64" else 2e-3)


def test_full_size_fp32_map_and_vjp_track_fp64():
    # The differentiable workload at its full size (m = 20 000, n = 50 000, K = 2 000,
    # B = 64, checkpoints every 45 steps): the FP32 forward and its VJP (FP64
    # accumulated) against the FP64 map.  x_K and the loss agree to 1e-4 (measured
    # 8e-6); the gradients agree in relative 2-norm to 1e-2 (measured 3e-3 for c,
    # 1e-3 for b).  Entry-wise they cannot be held tighter: the map is piecewise
    # linear, and a few entries of x (13 of 3.2 M measured) end on the other side of
    # a clamp in FP32, which changes the Jacobian there.  The exact gradient itself
    # is pinned by the oracle and finite-difference tests above.
    lp = G.random_lp(m=20000, n=50000, seed=0)
    B, K, lam = 64, 2000, 1e-3
    rng = np.random.default_rng(0)
    c0 = lp.c[None, :] + 0.1 * rng.normal(size=(B, lp.n))
    target = torch.tensor(rng.uniform(0, 1, size=(B, lp.n)), device=DEV)
    out = {}
    for prec in ("fp32_mixed", "fp64"):
        op = UnrolledPDHG(lp, ridge=lam, steps=K, checkpoint_every=45, precision=prec)
        c = torch.tensor(c0, device=DEV, requires_grad=True)
        b = torch.tensor(lp.con_lb, device=DEV, requires_grad=True)
        x, _ = op(c, b)
        loss = ((x - target) ** 2).sum()
        loss.backward()
        out[prec] = (x.detach().cpu().numpy(), loss.item(), c.grad.cpu().numpy(), b.grad.cpu().numpy())
    x32, l32, gc32, gb32 = out["fp32_mixed"]
    x64, l64, gc64, gb64 = out["fp64"]
    assert relerr(x32, x64) < 1e-4
    assert abs(l32 - l64) <= 1e-4 * abs(l64)
    assert np.linalg.norm(gc32 - gc64) <= 1e-2 * np.linalg.norm(gc64)
    assert np.linalg.norm(gb32 - gb64) <= 1e-2 * np.linalg.norm(gb64)


def test_segment_graph_replays_match_direct_launches(monkeypatch):
    # Full checkpoint segments replay captured graphs (forward: one per starting
    # buffer; backward: one middle segment).  Three forward/backward calls with
    # different objectives, torch work and synchronisations between them, give
    # bitwise the results of launching the same kernels directly.
    lp, A = problem(2, m=300, n=750)
    B, K, every = 16, 200, 9  # 22 full segments of odd length and a 2-step tail
    op = UnrolledPDHG(lp, ridge=1e-3, steps=K, checkpoint_every=every, precision="fp32_mixed")
    out = {}
    for flag in ("0", "1"):
        monkeypatch.setenv("CUOPT_AMD_GRAPHS", flag)
        runs = []
        for rep in range(3):
            print(f"unrolled graphs={flag} call {rep}", flush=True)
            rng = np.random.default_rng(10 + rep)
            ct = torch.tensor(lp.c[None, :] + 0.1 * rng.normal(size=(B, lp.n)), device=DEV, requires_grad=True)
            bt = torch.tensor(lp.con_lb, device=DEV, requires_grad=True)
            x, y = op(ct, bt)
            w = torch.tensor(rng.normal(size=(B, lp.n)), device=DEV)
            ((x * w).sum() + (y ** 2).sum()).backward()
            junk = torch.ones(4096, device=DEV).cumsum(0)  # eager work between calls
            torch.cuda.synchronize()
            assert float(junk[-1]) == 4096.0
            runs.append((x.detach().cpu().numpy(), y.detach().cpu().numpy(), ct.grad.cpu().numpy(),
                         bt.grad.cpu().numpy()))
        out[flag] = runs
    for a, b in zip(out["0"], out["1"]):
        for u, v in zip(a, b):
            assert np.array_equal(u, v)


def test_full_size_fp64_vjp_matches_central_differences():
    # The differentiable workload's shape (m = 20 000, n = 50 000, K = 2 000 steps,
    # checkpoints every 45) with 4 objectives in FP64: the VJP along random directions
    # of c and b against central differences of the FP64 map.  The map is piecewise
    # linear, and at this size some of its 4e8 clamp decisions change inside +-h: at
    # h = 1e-6 the difference quotient is off by about 1e-3 relative, and the error
    # falls in proportion to h, as it must when the VJP is the derivative of the
    # linear piece, down to about 1e-5 where FP64 rounding of the two losses takes over.
    lp = G.random_lp(m=20000, n=50000, seed=0)
    B, K, lam = 4, 2000, 1e-3
    op = UnrolledPDHG(lp, ridge=lam, steps=K, checkpoint_every=45, precision="fp64")
    rng = np.random.default_rng(4)
    c = torch.tensor(lp.c[None, :] + 0.1 * rng.normal(size=(B, lp.n)), device=DEV, requires_grad=True)
    b = torch.tensor(lp.con_lb, device=DEV, requires_grad=True)
    target = torch.tensor(rng.uniform(0, 1, size=(B, lp.n)), device=DEV)

    def loss(cc, bb):
        x, _ = op(cc, bb)
        return ((x - target) ** 2).sum()

    loss(c, b).backward()
    gc, gb = c.grad.clone(), b.grad.clone()
    vc = torch.tensor(rng.normal(size=(B, lp.n)), device=DEV)
    vb = torch.tensor(rng.normal(size=lp.m), device=DEV)
    with torch.no_grad():
        for name, g, v, plus, minus in (
                ("c", gc, vc, lambda h: loss(c + h * vc, b), lambda h: loss(c - h * vc, b)),
                ("b", gb, vb, lambda h: loss(c, b + h * vb), lambda h: loss(c, b - h * vb))):
            an = (g * v).sum().item()
            errs = {}
            for h in (1e-6, 1e-7, 1e-8, 1e-9):
                fd = (plus(h) - minus(h)).item() / (2 * h)
                errs[h] = abs(fd - an) / (1 + abs(an))
                print(f"direction {name}: h {h:g} fd {fd:.12e} vjp {an:.12e} rel err {errs[h]:.3e}", flush=True)
            # measured (c): 1.7e-3, 1.4e-4, 6.7e-6 at h = 1e-6, 1e-7, 1e-8; rounding takes over at 1e-9
            assert min(errs.values()) <= 2e-5, errs
            assert errs[1e-8] < errs[1e-7] < errs[1e-6], errs


@pytest.mark.parametrize("per_member_bounds", [False, True])
@pytest.mark.parametrize("prec", ["fp64", "fp32_mixed"])
def test_member_result_does_not_depend_on_the_slab_shape(monkeypatch, prec, per_member_bounds):
    # Batch sizes around the slab widths (4, 8, 16, 32) in every shape of the SpMM kernels
    # (10 x lanes per row + members per lane), on a ragged matrix: a member's point and
    # gradients are those it has in a batch of its own, bit for bit (each is the sum of
    # the same terms in the same order whatever the shape).
    lp, _ = ragged_lp(seed=4, m=1100, n=1500)
    op = UnrolledPDHG(lp, ridge=1e-3, steps=24, checkpoint_every=7, precision=prec)
    rng = np.random.default_rng(9)
    top = 33
    c = lp.c[None, :] + 0.1 * rng.normal(size=(top, lp.n))
    slack = rng.uniform(0.1, 0.5, size=(top, lp.m))
    gx, gy = rng.normal(size=(top, lp.n)), rng.normal(size=(top, lp.m))

    def run(members):
        lc = lp.con_lb - slack[members] if per_member_bounds else lp.con_lb
        uc = lp.con_ub + slack[members] if per_member_bounds else lp.con_ub
        ct, lt, ut = (torch.tensor(v, device=DEV, requires_grad=True) for v in (c[members], lc, uc))
        x, y = op(ct, lt, ut)
        torch.autograd.backward([x, y], [torch.tensor(gx[members], device=DEV), torch.tensor(gy[members], device=DEV)])
        grads = [ct.grad] + ([lt.grad, ut.grad] if per_member_bounds else [])
        return [v.detach().cpu().numpy() for v in (x, y, *grads)]

    alone = [run([i]) for i in range(top)]
    for shape in (None, 41, 81, 82, 84, 161):
        if shape:
            monkeypatch.setenv("CUOPT_AMD_UNR_SHAPE", str(shape))
        for B in (2, 4, 5, 8, 9, 16, 17, 33):
            for k, v in enumerate(run(list(range(B)))):
                for i in range(B):
                    assert np.array_equal(v[i], alone[i][k][0]), (shape, B, k, i)


@pytest.mark.parametrize("prec", ["fp64", "fp32_mixed"])
def test_one_handle_runs_other_numbers_of_steps(prec):
    # A handle whose calls take 100, 60, 100, 23 and 172 steps of the same batch and checkpoint
    # interval: its segment graphs and its working storage follow the call, so every
    # point and gradient is that of a handle made for the call, bit for bit.
    lp, _ = problem(6, m=200, n=500)
    B, every = 8, 9
    rng = np.random.default_rng(6)
    c0 = lp.c[None, :] + 0.1 * rng.normal(size=(B, lp.n))
    gx, gy = (torch.tensor(rng.normal(size=(B, k)), device=DEV) for k in (lp.n, lp.m))

    def run(op):
        c, b = (torch.tensor(v, device=DEV, requires_grad=True) for v in (c0, lp.con_lb))
        x, y = op(c, b)
        torch.autograd.backward([x, y], [gx, gy])
        return [v.detach().cpu().numpy() for v in (x, y, c.grad, b.grad)]

    kept = UnrolledPDHG(lp, ridge=1e-3, steps=100, checkpoint_every=every, precision=prec)
    for steps in (100, 60, 100, 23, 172, 60):
        kept.steps = steps
        fresh = UnrolledPDHG(lp, ridge=1e-3, steps=steps, checkpoint_every=every, precision=prec)
        for name, u, v in zip(("x", "y", "gc", "gb"), run(kept), run(fresh)):
            assert np.array_equal(u, v), (steps, name)


@pytest.mark.parametrize("prec", ["fp64", "fp32_mixed"])
def test_backward_after_a_forward_that_did_not_fit(prec):
    # A forward whose working storage cannot be allocated fails, and so does the backward
    # of any forward before it, through autograd and through the C entry point: the
    # checkpoints are gone.  The handle works on.
    import ctypes

    from cuopt_amd import autograd, c_api

    lp, _ = problem(7, m=60, n=150)
    B = 3
    rng = np.random.default_rng(7)
    c0 = lp.c[None, :] + 0.1 * rng.normal(size=(B, lp.n))
    op = UnrolledPDHG(lp, ridge=1e-3, steps=20, checkpoint_every=6, precision=prec)

    def forward():
        c, b = (torch.tensor(v, device=DEV, requires_grad=True) for v in (c0, lp.con_lb))
        return c, (op(c, b)[0] ** 2).sum()

    def native_backward():
        gx, gc = (torch.ones(lp.n, B, dtype=torch.float64, device=DEV) for _ in range(2))
        glc, guc = (torch.ones(lp.m, B, dtype=torch.float64, device=DEV) for _ in range(2))
        args = [ctypes.c_void_p(t.data_ptr() if t is not None else None) for t in (gx, None, gc, glc, guc)]
        rc = autograd._lib().cuOptAmdUnrolledBackward(op.handle, *args, None)
        torch.cuda.synchronize()
        return rc

    c, loss = forward()
    loss.backward(retain_graph=True)
    first = c.grad.clone()
    assert native_backward() == c_api.CUOPT_SUCCESS
    op.every = 10 ** 9  # segment states for so many steps: terabytes
    with pytest.raises(c_api.CuOptError):
        forward()
    op.every = 6
    with pytest.raises(RuntimeError):
        loss.backward()
    assert native_backward() != c_api.CUOPT_SUCCESS
    c, loss = forward()
    loss.backward()
    assert torch.equal(c.grad, first)


def test_more_workgroups_than_one_grid_dimension_counts():
    # One row, one column and 2^28 + 64 members: more than 2^24 workgroups of 256 lanes.  One
    # step from x = 0, y = 0 has a closed form.
    B, lam = (1 << 28) + 64, 1e-3
    if torch.cuda.mem_get_info()[0] < (150 << 30):
        pytest.skip("needs 150 GB of device memory")
    lp = G.LP(m=1, n=1, row_offsets=np.array([0, 1], np.int32), col_indices=np.zeros(1, np.int32), values=np.ones(1),
              c=np.ones(1), con_lb=np.ones(1), con_ub=np.ones(1), var_lb=np.zeros(1), var_ub=np.full(1, 5.0))
    op = UnrolledPDHG(lp, ridge=lam, steps=1, checkpoint_every=1, precision="fp64")
    eta = op.step_size
    c = torch.linspace(-6.0, 1.0, B, dtype=torch.float64, device=DEV)[:, None].requires_grad_(True)
    b = torch.ones(1, dtype=torch.float64, device=DEV)
    x, y = op(c, b)
    x.sum().backward()
    with torch.no_grad():
        moved = -eta * c / (1.0 + eta * lam)
        want = moved.clamp(0.0, 5.0)
        assert torch.all((x - want).abs() <= 1e-12)
        assert torch.all((y - eta * (1.0 - 2.0 * want)).abs() <= 1e-12)
        inside = (moved > 0.0) & (moved < 5.0)
        assert torch.all((c.grad + inside.double() * (eta / (1.0 + eta * lam))).abs() <= 1e-12)
    del op, c, x, y, moved, want, inside
    torch.cuda.empty_cache()


def test_working_storage_needs_no_more_than_the_batch(monkeypatch):
    # Slabs hold more members than a batch that their width does not divide.  Where only
    # the batch itself fits the memory that is left, the call still runs, with the same
    # result: the segment states of `every` steps are most of the storage here, 6 GB of
    # 7 GB left free, which whole slabs of this many members would pass.
    lp, _ = ragged_lp(seed=8, m=300, n=700)
    rng = np.random.default_rng(8)

    def run(prec, B, shape, every):
        print(f"working storage {prec} B={B} shape={shape} every={every}", flush=True)
        if shape:
            monkeypatch.setenv("CUOPT_AMD_UNR_SHAPE", str(shape))
        else:
            monkeypatch.delenv("CUOPT_AMD_UNR_SHAPE", raising=False)
        op = UnrolledPDHG(lp, ridge=1e-3, steps=12, checkpoint_every=every, precision=prec)
        c, b = (torch.tensor(v, device=DEV, requires_grad=True) for v in (c0[:B], lp.con_lb))
        x, y = op(c, b)
        torch.autograd.backward([x, y], [gx[:B], torch.ones_like(y)])
        return [v.detach().cpu().numpy() for v in (x, y, c.grad, b.grad)]

    cases = [("fp64", 1, None), ("fp64", 5, None), ("fp64", 9, 82), ("fp32_mixed", 3, None), ("fp32_mixed", 9, None),
             ("fp32_mixed", 37, 84)]
    c0 = lp.c[None, :] + 0.1 * rng.normal(size=(37, lp.n))
    gx = torch.tensor(rng.normal(size=(37, lp.n)), device=DEV)
    want = [run(*case, 12) for case in cases]
    torch.cuda.empty_cache()
    hog = torch.empty(torch.cuda.mem_get_info()[0] - (7 << 30), dtype=torch.uint8, device=DEV)
    try:
        got = [run(*case, (6 << 30) // ((8 if case[0] == "fp64" else 4) * case[1] * (lp.m + lp.n))) for case in cases]
    finally:
        del hog
        torch.cuda.empty_cache()
    for case, a, b in zip(cases, want, got):
        for name, u, v in zip(("x", "y", "gc", "gb"), a, b):
            assert np.array_equal(u, v), (case, name)


@pytest.mark.parametrize("prec", ["fp64", "fp32_mixed"])
def test_more_columns_than_24_bits_number(monkeypatch, prec):
    # Gathers take a 64-bit offset from 2^24 rows or columns up.  Columns without nonzeros
    # change nothing for the others, so a matrix whose few nonzeros lie among 2^24 + 40 columns
    # gives, bit for bit, what the matrix of its nonzero columns does, in every shape.
    import scipy.sparse as sp

    rng = np.random.default_rng(12)
    m, n, B = 70, (1 << 24) + 40, 7
    used = np.unique(np.concatenate([rng.choice(n, size=900, replace=False), np.arange(n - 45, n), np.arange(3)]))
    small = sp.random(m, used.size, density=0.03, random_state=12, format="csc", data_rvs=rng.standard_normal)
    small = (small + sp.csc_matrix((np.ones(used.size), (np.arange(used.size) % m, np.arange(used.size))),
                                   shape=(m, used.size))).tocsr()
    small.sort_indices()
    b = small @ rng.random(used.size)

    def lp_of(cols, width):
        return G.LP(m=m, n=width, row_offsets=small.indptr.astype(np.int32), col_indices=cols.astype(np.int32),
                    values=small.data, c=np.zeros(width), con_lb=b, con_ub=b.copy(), var_lb=np.zeros(width),
                    var_ub=np.full(width, 10.0))

    kw = dict(ridge=1e-3, steps=3, checkpoint_every=2, precision=prec)
    few = UnrolledPDHG(lp_of(small.indices, used.size), **kw)
    many = UnrolledPDHG(lp_of(used[small.indices], n), **kw)
    assert few.step_size == many.step_size
    at = torch.tensor(used, device=DEV)
    c0 = torch.tensor(rng.normal(size=(B, used.size)), device=DEV)
    gx = torch.tensor(rng.normal(size=(B, used.size)), device=DEV)

    def run(op, wide):
        c = c0
        if wide:
            c = torch.zeros(B, n, dtype=torch.float64, device=DEV)
            c[:, at] = c0
        c = c.clone().requires_grad_(True)
        bt = torch.tensor(b, device=DEV, requires_grad=True)
        x, y = op(c, bt)
        ((x[:, at] if wide else x) * gx).sum().backward()
        gc = c.grad[:, at] if wide else c.grad
        return [v.detach().cpu().numpy() for v in (x[:, at] if wide else x, y, gc, bt.grad)]

    want = run(few, False)
    for shape in (41, 81, 161, 82) + ((84,) if prec == "fp32_mixed" else ()):
        print(f"2^24 columns {prec} shape {shape}", flush=True)
        monkeypatch.setenv("CUOPT_AMD_UNR_SHAPE", str(shape))
        for name, u, v in zip(("x", "y", "gc", "gb"), want, run(many, True)):
            assert np.array_equal(u, v), (shape, name)
    del many
    torch.cuda.empty_cache()


@pytest.mark.parametrize("shape,prec,tol", [(s, "fp64", 1e-9) for s in (41, 81, 161, 82)] +
                         [(s, "fp32_mixed", 2e-3) for s in (41, 81, 161, 82, 84)])
def test_slab_shapes_match_oracle(monkeypatch, shape, prec, tol):
    # Every shape of the SpMM kernels (10 x lanes per row + members per lane; 84 is FP32 only)
    # against the oracle on a ragged matrix, with batches whose last slab is whole, holds
    # one member and holds some.
    monkeypatch.setenv("CUOPT_AMD_UNR_SHAPE", str(shape))
    lp, A = ragged_lp()
    K, every, lam = 40, 7, 1e-3
    op = UnrolledPDHG(lp, ridge=lam, steps=K, checkpoint_every=every, precision=prec)
    b, eta = lp.con_lb.copy(), op.step_size
    for B in (32, 33, 39):
        print(f"slab shape {shape} {prec} B={B}", flush=True)
        rng = np.random.default_rng(shape + B)
        c = lp.c[None, :] + 0.1 * rng.normal(size=(B, lp.n))
        ct, bt = (torch.tensor(v, device=DEV, requires_grad=True) for v in (c, b))
        x, y = op(ct, bt)
        xo, yo, xs, ys = U.forward(A, c.T.copy(), b, b, lp.var_lb, lp.var_ub, lam, eta, K, keep=True)
        assert relerr(x.detach().cpu().numpy().T, xo) < tol
        assert relerr(y.detach().cpu().numpy().T, yo) < tol
        gx, gy = rng.normal(size=(B, lp.n)), rng.normal(size=(B, lp.m))
        torch.autograd.backward([x, y], [torch.tensor(v, device=DEV) for v in (gx, gy)])
        if prec == "fp64":  # (in FP32 a clamp that ends on its other side changes the derivative there)
            gc, glc, guc = U.backward(A, b, b, lp.var_lb, lp.var_ub, lam, eta, xs, ys, gx.T.copy(), gy.T.copy())
            assert relerr(ct.grad.cpu().numpy().T, gc) < tol
            assert relerr(bt.grad.cpu().numpy(), (glc + guc).sum(axis=1)) < tol


@pytest.mark.parametrize("most,prec,tol", [(2, "fp64", 1e-9), (4, "fp64", 1e-9), (4, "fp32_mixed", 2e-3)])
def test_short_rows_match_oracle(monkeypatch, most, prec, tol):
    # Matrices whose rows (and for the transposed LP columns) have at most two or four nonzeros
    # take kernels of their own: 0 to `most` nonzeros in a row, every slab shape.
    import scipy.sparse as sp

    rng = np.random.default_rng(13)
    rows, cols = 170, 230
    per = rng.integers(0, most + 1, size=rows)
    per[:3] = 0, most, 1
    idx = [np.sort(rng.choice(cols, size=k, replace=False)) for k in per]
    M = sp.csr_matrix((rng.normal(size=per.sum()), np.concatenate(idx), np.concatenate([[0], np.cumsum(per)])),
                      shape=(rows, cols))
    K, every, lam = 30, 7, 1e-3
    for A in (M, M.T.tocsr()):
        A.sort_indices()
        m, n = A.shape
        b = A @ rng.random(n)
        lp = G.LP(m=m, n=n, row_offsets=A.indptr.astype(np.int32), col_indices=A.indices.astype(np.int32),
                  values=A.data, c=rng.normal(size=n), con_lb=b, con_ub=b.copy(), var_lb=np.zeros(n),
                  var_ub=np.full(n, 10.0))
        op = UnrolledPDHG(lp, ridge=lam, steps=K, checkpoint_every=every, precision=prec)
        eta = op.step_size
        for shape, B in ((0, 1), (0, 3), (0, 40), (41, 6), (81, 11), (161, 21), (82, 19), (84, 37)):
            print(f"short rows {most} {prec} {m}x{n} shape {shape} B={B}", flush=True)
            monkeypatch.setenv("CUOPT_AMD_UNR_SHAPE", str(shape))
            c = lp.c[None, :] + 0.1 * rng.normal(size=(B, n))
            ct, bt = (torch.tensor(v, device=DEV, requires_grad=True) for v in (c, b))
            x, y = op(ct, bt)
            xo, yo, xs, ys = U.forward(A, c.T.copy(), b, b, lp.var_lb, lp.var_ub, lam, eta, K, keep=True)
            assert relerr(x.detach().cpu().numpy().T, xo) < tol
            assert relerr(y.detach().cpu().numpy().T, yo) < tol
            gx = rng.normal(size=(B, n))
            (x * torch.tensor(gx, device=DEV)).sum().backward()
            if prec == "fp64":
                gc, glc, guc = U.backward(A, b, b, lp.var_lb, lp.var_ub, lam, eta, xs, ys, gx.T.copy())
                assert relerr(ct.grad.cpu().numpy().T, gc) < tol
                assert relerr(bt.grad.cpu().numpy(), (glc + guc).sum(axis=1)) < tol
