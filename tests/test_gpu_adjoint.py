"""Adjoint of the monodomain step (BuenoOrovio, Euler ddt, FP64), explicit and implicit:
the adjoint's forward run equals cg_tissue_step, and its gradients with respect to a
per-cell conductivity scale and tau_fi / tau_si equal central finite differences of the
loss computed by the CPU oracle's independent tissue run."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIG0 = np.array([0.17, 0.019, 0.019])
BOX = {"stimulusLocationMin": [0.0, 0.0, 0.0], "stimulusLocationMax": [6e-4, 6e-4, 6e-4],
       "stimulusDuration": 2e-3, "stimulusIntensity": 5e4, "stimulusStartTime": 0.0}
DT = 1e-5


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _dom(gpu, shape, h, algorithm="explicit", tol=1e-8, box_max=None):
    mesh = gpu.HexMesh(*shape, h)
    box = dict(BOX) if box_max is None else dict(BOX, stimulusLocationMax=list(box_max))
    coeffs = {"ionicModel": "BuenoOrovio", "tissue": "epicardialCells", "chi": 1.4e5,
              "cm": 0.01, "solutionAlgorithm": algorithm,
              "conductivity": [SIG0[0], 0, 0, 0, SIG0[1], 0, 0, 0, SIG0[2]],
              "externalStimulus": box}
    return mesh, gpu.Monodomain(mesh, coeffs, dt=DT, tol=tol)


def test_adjoint_forward_equals_tissue_step(gpu, orc):
    import torch
    _say("adjoint forward vs tissue step")
    shape, h, steps = (20, 12, 8), 2e-4, 400
    mesh, dom = _dom(gpu, shape, h)
    n = mesh.n
    cells = np.random.default_rng(1).choice(n, 16, replace=False)
    adj = gpu.TissueAdjoint(dom, cells, checkpoint_every=64)
    kappa = torch.ones(n, dtype=torch.float64, device="cuda")
    tr = gpu.probe_traces(adj, kappa, None, steps).cpu().numpy()
    ref = np.empty((steps, len(cells)))
    for s in range(steps):
        dom.step(1)
        ref[s] = dom.Vm[cells]
    err = np.max(np.abs(tr - ref)) / np.max(np.abs(ref))
    _say("  trace rel err %.3e" % err)
    assert err < 1e-12


def _oracle_loss(orc, shape, h, kappa, theta, steps, cells, target, implicit=0):
    nx, ny, nz = shape
    sig = np.zeros((kappa.size, 9))
    sig[:, 0], sig[:, 4], sig[:, 8] = kappa * SIG0[0], kappa * SIG0[1], kappa * SIG0[2]
    T = orc.OracleTissue(nx, ny, nz, h, sig, orc.BO, orc.EPI, DT, 1.4e5, 0.01, integrator=0,
                         ddt=0, implicit=implicit, pcg_tol=1e-14, nthreads=8)
    T.set_const(orc.const_index(orc.BO, "tauFi"), theta[0])
    T.set_const(orc.const_index(orc.BO, "tauSi"), theta[1])
    bx = orc.make_boxes(BOX["stimulusLocationMin"], BOX["stimulusLocationMax"], [0.0], [2e-3],
                        [5e4])
    loss = 0.0
    for s in range(steps):
        T.step(bx)
        loss += float(np.sum((T.V[cells] - target[s]) ** 2))
    return loss


def test_adjoint_gradient_vs_oracle_finite_differences(gpu, orc):
    """dL/dkappa (three random directions) and dL/dtau_fi, dL/dtau_si against central
    differences of the oracle's loss; 300 steps with checkpoints every 64 (partial last
    segment), L = sum over steps and probes of (Vm - target)^2."""
    import torch
    _say("adjoint gradient vs oracle FD")
    shape, h, steps = (12, 10, 6), 2e-4, 300
    mesh, dom = _dom(gpu, shape, h)
    n = mesh.n
    rng = np.random.default_rng(7)
    cells = rng.choice(n, 24, replace=False)
    theta0 = np.array([0.11, 1.8875])                   # epicardial tau_fi, tau_si
    kappa0 = rng.uniform(0.8, 1.25, n)
    target = -0.084 + 0.1 * rng.random((steps, cells.size))
    adj = gpu.TissueAdjoint(dom, cells, checkpoint_every=64)
    kappa = torch.tensor(kappa0, dtype=torch.float64, device="cuda", requires_grad=True)
    theta = torch.tensor(theta0, dtype=torch.float64, requires_grad=True)
    tr = gpu.probe_traces(adj, kappa, theta, steps)
    loss = ((tr - torch.tensor(target, device="cuda")) ** 2).sum()
    loss.backward()
    gk = kappa.grad.cpu().numpy()
    gt = theta.grad.numpy()
    l_or = _oracle_loss(orc, shape, h, kappa0, theta0, steps, cells, target)
    _say("  loss gpu %.12e oracle %.12e" % (loss.item(), l_or))
    assert abs(loss.item() - l_or) <= 1e-10 * abs(l_or)
    eps = 1e-6
    for k in range(3):
        d = rng.standard_normal(n)
        fp = _oracle_loss(orc, shape, h, kappa0 + eps * d, theta0, steps, cells, target)
        fm = _oracle_loss(orc, shape, h, kappa0 - eps * d, theta0, steps, cells, target)
        fd, ad = (fp - fm) / (2 * eps), float(gk @ d)
        _say("  kappa direction %d: adjoint %.9e fd %.9e" % (k, ad, fd))
        assert abs(ad - fd) <= 1e-5 * abs(fd)
    for i in range(2):
        e = np.zeros(2)
        e[i] = eps * theta0[i]
        fp = _oracle_loss(orc, shape, h, kappa0, theta0 + e, steps, cells, target)
        fm = _oracle_loss(orc, shape, h, kappa0, theta0 - e, steps, cells, target)
        fd = (fp - fm) / (2 * e[i])
        _say("  theta %d: adjoint %.9e fd %.9e" % (i, gt[i], fd))
        assert abs(gt[i] - fd) <= 1e-5 * abs(fd)


def test_adjoint_store_all_equals_checkpointing(gpu, orc):
    """Keeping every step (interval >= steps) and re-running checkpointed segments give the
    same gradient."""
    import torch
    _say("adjoint store-all vs checkpoints")
    shape, h, steps = (16, 10, 6), 2e-4, 250
    res = []
    for K in (32, 1000):
        mesh, dom = _dom(gpu, shape, h)
        cells = np.random.default_rng(3).choice(mesh.n, 12, replace=False)
        adj = gpu.TissueAdjoint(dom, cells, checkpoint_every=K)
        kappa = torch.ones(mesh.n, dtype=torch.float64, device="cuda", requires_grad=True)
        theta = torch.tensor([0.11, 1.8875], dtype=torch.float64, requires_grad=True)
        tr = gpu.probe_traces(adj, kappa, theta, steps)
        (tr ** 2).sum().backward()
        res.append((kappa.grad.cpu().numpy(), theta.grad.numpy()))
    np.testing.assert_allclose(res[0][0], res[1][0], rtol=1e-13, atol=1e-300)
    np.testing.assert_allclose(res[0][1], res[1][1], rtol=1e-13)


def test_adjoint_backward_of_a_replaced_forward_raises(gpu, orc):
    """Two forward runs on one handle before backward: the first run's backward raises
    (its checkpoints were replaced) instead of returning the second run's gradient; the
    C-ABI refuses a stale generation or a different step count; the latest run still
    differentiates."""
    import torch
    from cardiacfoam_amd import _capi
    _say("adjoint stale backward")
    shape, h = (10, 8, 6), 2e-4
    mesh, dom = _dom(gpu, shape, h)
    cells = np.arange(0, mesh.n, 37)
    adj = gpu.TissueAdjoint(dom, cells, checkpoint_every=16)
    k1 = torch.ones(mesh.n, dtype=torch.float64, device="cuda", requires_grad=True)
    k2 = torch.ones(mesh.n, dtype=torch.float64, device="cuda", requires_grad=True)
    t1 = gpu.probe_traces(adj, k1, None, 40)
    t2 = gpu.probe_traces(adj, k2, None, 25)
    with pytest.raises(RuntimeError, match="replaced"):
        (t1 ** 2).sum().backward()
    g = torch.zeros(25, cells.size, dtype=torch.float64, device="cuda")
    dk = torch.empty(mesh.n, dtype=torch.float64, device="cuda")
    dth = np.zeros(2)
    L = _capi.lib()
    import ctypes as C
    for gen, n in ((adj.generation - 1, 25), (adj.generation, 40)):
        rc = L.cg_adjoint_backward(adj.a, gen, n, C.c_void_p(g.data_ptr()),
                                   C.c_void_p(dk.data_ptr()), dth.ctypes.data_as(C.c_void_p))
        assert rc == 9, (gen, n, rc)          # CG_ERR_STATE
    (t2 ** 2).sum().backward()
    assert torch.isfinite(k2.grad).all()


def test_implicit_adjoint_forward_equals_tissue_step(gpu, orc):
    """Implicit (backward-Euler) tissue: the adjoint's forward run (PCG to 1e-14) equals
    cg_tissue_step (PCG to 1e-13).  Each step's two solves stop at different points within
    their tolerances, so the traces agree to about steps x 1e-13 of Vm's range, not to
    rounding as in the explicit case."""
    import torch
    _say("implicit adjoint forward vs tissue step")
    shape, h, steps = (20, 12, 8), 2e-4, 300
    mesh, dom = _dom(gpu, shape, h, "implicit", tol=1e-13)
    n = mesh.n
    cells = np.random.default_rng(1).choice(n, 16, replace=False)
    adj = gpu.TissueAdjoint(dom, cells, checkpoint_every=64)
    kappa = torch.ones(n, dtype=torch.float64, device="cuda")
    tr = gpu.probe_traces(adj, kappa, None, steps).cpu().numpy()
    ref = np.empty((steps, len(cells)))
    for s in range(steps):
        dom.step(1)
        ref[s] = dom.Vm[cells]
    err = np.max(np.abs(tr - ref)) / np.max(np.abs(ref))
    _say("  trace rel err %.3e" % err)
    assert err < steps * 2e-13


def _tangent_check(gpu, orc, shape, h, steps, n_probes, box_max, n_kdirs, seed, ckpt):
    """The adjoint's loss and gradient against the oracle's tangent-linear run over the
    whole horizon: the loss, n_kdirs random kappa directions and tau_fi, tau_si.  Returns
    the worst relative differences (loss, directions)."""
    import torch
    rng = np.random.default_rng(seed)
    n = int(np.prod(shape))
    mesh, dom = _dom(gpu, shape, h, box_max=box_max)
    cells = rng.choice(n, n_probes, replace=False)
    adj = gpu.TissueAdjoint(dom, cells, checkpoint_every=ckpt)
    theta0 = np.array([0.11, 1.8875])
    # target: the device's own run at a smooth conductivity perturbation
    x = (np.arange(n) % shape[0]) / shape[0]
    kt = torch.tensor(1.0 + 0.2 * np.sin(2 * np.pi * x), device="cuda")
    with torch.no_grad():
        target = gpu.probe_traces(adj, kt, torch.tensor(theta0), steps).clone()
    kappa = torch.ones(n, dtype=torch.float64, device="cuda", requires_grad=True)
    theta = torch.tensor(theta0, dtype=torch.float64, requires_grad=True)
    loss = ((gpu.probe_traces(adj, kappa, theta, steps) - target) ** 2).sum()
    loss.backward()
    gk, gt = kappa.grad.cpu().numpy(), theta.grad.numpy()
    dk = np.zeros((n_kdirs + 2, n))
    dk[:n_kdirs] = rng.standard_normal((n_kdirs, n))
    dth = np.zeros((n_kdirs + 2, 2))
    dth[n_kdirs, 0], dth[n_kdirs + 1, 1] = 1.0, 1.0
    _say("  tangent-linear oracle run: %d cells, %d steps, %d directions" %
         (n, steps, n_kdirs + 2))
    L, d, _ = orc.bo_tangent(shape, h, SIG0, orc.EPI, DT, 1.4e5, 0.01,
                             orc.make_boxes(BOX["stimulusLocationMin"],
                                            BOX["stimulusLocationMax"] if box_max is None
                                            else box_max, [0.0], [2e-3], [5e4]),
                             np.ones(n), theta0, dk, dth, steps, cells,
                             target.cpu().numpy(), nthreads=16)
    adj_d = np.concatenate([dk[:n_kdirs] @ gk, gt])
    rel = np.abs(adj_d - d) / np.maximum(np.abs(d), 1e-300)
    _say("  loss device %.12e oracle %.12e" % (loss.item(), L))
    for k in range(n_kdirs + 2):
        _say("  direction %d: adjoint %.12e tangent %.12e rel %.2e" % (k, adj_d[k], d[k], rel[k]))
    return abs(loss.item() - L) / abs(L), float(np.max(rel))


def test_adjoint_full_horizon_vs_tangent_linear(gpu, orc):
    """5000 steps (50 ms: stimulus, the wave across the block, the plateau and the start of
    repolarisation), where central differences fail (a perturbation moves threshold
    crossings by whole steps): the gradient against the oracle's tangent-linear run of the
    same discrete map, which differentiates the branch each step takes as the adjoint
    does.  Six kappa directions, tau_fi and tau_si."""
    _say("adjoint full horizon vs tangent-linear oracle")
    lrel, drel = _tangent_check(gpu, orc, (16, 12, 6), 2e-4, 5000, 32, None, 6, 11, 250)
    assert lrel <= 1e-10
    assert drel <= 1e-7


def test_handles_destroyed_in_any_order(gpu):
    """Python's cyclic collector calls finalizers in no fixed order (a failed test's
    traceback makes its locals such garbage), so the C-ABI lets handles go in any order:
    here each owner goes before what depends on it -- ionic, mesh, tissue, then the
    adjoint made from them."""
    import torch
    from cardiacfoam_amd import _capi
    _say("handles destroyed owner first")
    mesh, dom = _dom(gpu, (8, 6, 4), 2e-4, "implicit", tol=1e-10)
    dom.step(3)
    adj = gpu.TissueAdjoint(dom, [0, 5, 17], checkpoint_every=4)
    kappa = torch.ones(mesh.n, dtype=torch.float64, device="cuda")
    tr = gpu.probe_traces(adj, kappa, None, 10).cpu().numpy()
    assert np.all(np.isfinite(tr))
    L = _capi.lib()
    for obj, attr, destroy in ((dom.ionic, "h", L.cg_ionic_destroy),
                               (mesh, "m", L.cg_mesh_destroy),
                               (dom, "t", L.cg_tissue_destroy),
                               (adj, "a", L.cg_adjoint_destroy)):
        h = getattr(obj, attr)
        setattr(obj, attr, None)
        assert destroy(h) == 0


def test_implicit_adjoint_gradient_vs_oracle_finite_differences(gpu, orc):
    """The implicit tissue's gradient (three random kappa directions, tau_fi, tau_si)
    against central differences of the oracle's implicit loss (PCG to 1e-14); 240 steps with
    checkpoints every 50 (partial last segment)."""
    import torch
    _say("implicit adjoint gradient vs oracle FD")
    shape, h, steps = (12, 10, 6), 2e-4, 240
    mesh, dom = _dom(gpu, shape, h, "implicit", tol=1e-13)
    n = mesh.n
    rng = np.random.default_rng(8)
    cells = rng.choice(n, 24, replace=False)
    theta0 = np.array([0.11, 1.8875])
    kappa0 = rng.uniform(0.8, 1.25, n)
    target = -0.084 + 0.1 * rng.random((steps, cells.size))
    adj = gpu.TissueAdjoint(dom, cells, checkpoint_every=50)
    kappa = torch.tensor(kappa0, dtype=torch.float64, device="cuda", requires_grad=True)
    theta = torch.tensor(theta0, dtype=torch.float64, requires_grad=True)
    tr = gpu.probe_traces(adj, kappa, theta, steps)
    loss = ((tr - torch.tensor(target, device="cuda")) ** 2).sum()
    loss.backward()
    gk = kappa.grad.cpu().numpy()
    gt = theta.grad.numpy()
    l_or = _oracle_loss(orc, shape, h, kappa0, theta0, steps, cells, target, implicit=1)
    _say("  loss gpu %.12e oracle %.12e" % (loss.item(), l_or))
    assert abs(loss.item() - l_or) <= 1e-10 * abs(l_or)
    eps = 1e-6
    for k in range(3):
        d = rng.standard_normal(n)
        fp = _oracle_loss(orc, shape, h, kappa0 + eps * d, theta0, steps, cells, target, 1)
        fm = _oracle_loss(orc, shape, h, kappa0 - eps * d, theta0, steps, cells, target, 1)
        fd, ad = (fp - fm) / (2 * eps), float(gk @ d)
        _say("  kappa direction %d: adjoint %.9e fd %.9e" % (k, ad, fd))
        assert abs(ad - fd) <= 1e-5 * abs(fd)
    for i in range(2):
        e = np.zeros(2)
        e[i] = eps * theta0[i]
        fp = _oracle_loss(orc, shape, h, kappa0, theta0 + e, steps, cells, target, 1)
        fm = _oracle_loss(orc, shape, h, kappa0, theta0 - e, steps, cells, target, 1)
        fd = (fp - fm) / (2 * e[i])
        _say("  theta %d: adjoint %.9e fd %.9e" % (i, gt[i], fd))
        assert abs(gt[i] - fd) <= 1e-5 * abs(fd)


@pytest.mark.parametrize("shape,h", [((12, 10, 6), 2e-4), ((9, 1, 1), 2e-4), ((7, 5, 1), 4e-5),
                                     ((12, 10, 6), 4e-5), ((12, 10, 6), 2e-5)])
def test_implicit_adjoint_solver_branches(gpu, orc, shape, h):
    """The fixed-length Chebyshev solves (rho 0.07 at h = 0.2 mm and 0.65 a, 0.04 mm: the
    PCG above 0.6) against the run's own central difference in a random kappa direction.
    The potentials stay below the switches' first threshold, so the loss is smooth: the
    difference carries eps^2 truncation (1e-6 relative at eps 1e-3) and the loss's 1e-15
    rounding over eps."""
    import torch
    _say("implicit adjoint branches", shape, h)
    mesh, dom = _dom(gpu, shape, h, "implicit", tol=1e-13, box_max=[-1.0, -1.0, -1.0])
    n, steps = mesh.n, 12
    rng = np.random.default_rng(3)
    dom.set_field(0, -0.084 + 4e-4 * rng.random(n))
    cells = rng.choice(n, min(5, n), replace=False)
    adj = gpu.TissueAdjoint(dom, cells, checkpoint_every=5)
    target = torch.tensor(-0.084 + 4e-4 * rng.random((steps, cells.size)), device="cuda")
    kappa0, d = rng.uniform(0.8, 1.25, n), rng.standard_normal(n)
    theta = torch.tensor([0.11, 1.8875], dtype=torch.float64)

    def loss(k):
        return ((gpu.probe_traces(adj, k, theta, steps) - target) ** 2).sum() * 1e6

    kappa = torch.tensor(kappa0, dtype=torch.float64, device="cuda", requires_grad=True)
    loss(kappa).backward()
    ad = float(kappa.grad.cpu().numpy() @ d)
    eps = 1e-3
    lp, lm = (float(loss(torch.tensor(kappa0 + s * eps * d, device="cuda"))) for s in (1, -1))
    fd = (lp - lm) / (2 * eps)
    _say("  adjoint %.9e fd %.9e" % (ad, fd))
    assert abs(ad - fd) <= 1e-4 * abs(fd)


def test_implicit_adjoint_after_a_missed_solve(gpu, orc):
    """A run whose currents are not finite misses the fixed-length solves and is repeated
    with the conjugate gradients, forward and backward; the runs after it take the fixed-length
    solves again: traces and gradients bit for bit those of a handle that never missed (the
    conjugate gradients' differ in the last digits)."""
    import torch
    _say("implicit adjoint after a miss")
    mesh, dom = _dom(gpu, (12, 10, 6), 2e-4, "implicit", tol=1e-13)
    n, steps = mesh.n, 8
    rng = np.random.default_rng(5)
    dom.set_field(0, -0.084 + 6e-2 * rng.random(n))
    cells = rng.choice(n, 5, replace=False)
    target = torch.tensor(-0.08 + 1e-2 * rng.random((steps, cells.size)), device="cuda")
    kappa0 = torch.tensor(rng.uniform(0.8, 1.25, n), device="cuda")

    def run(adj, tfi):
        kappa = kappa0.clone().requires_grad_()
        theta = torch.tensor([tfi, 1.8875], dtype=torch.float64, requires_grad=True)
        tr = gpu.probe_traces(adj, kappa, theta, steps)
        ((tr - target) ** 2).sum().backward()
        return [x.detach().cpu().numpy() for x in (tr, kappa.grad, theta.grad)]

    fresh = run(gpu.TissueAdjoint(dom, cells, checkpoint_every=3), 0.11)
    adj = gpu.TissueAdjoint(dom, cells, checkpoint_every=3)
    run(adj, float("nan"))      # every step's right-hand side holds NaN: every solve misses
    for got, want in zip(run(adj, 0.11), fresh):
        assert np.isfinite(want).all()
        np.testing.assert_array_equal(got, want)
