"""Hand-written backward of the fused distance -> kernel -> log-sum op against a float64
torch.autograd reference of the same formula and against central finite differences."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ref_loss(img, C, w, eps):
    """float64 torch reference: images -> rfft2 -> weighted half-spectrum distances -> L_e."""
    import torch
    X = torch.fft.rfft2(img)
    n = X.shape[0]
    A = (X.abs() ** 2 * w).reshape(n, -1)
    B = (C ** 2).reshape(n, -1)
    Y = (C * X * w.sqrt()).reshape(n, -1)
    P = A @ B.T
    D = P + P.T - 2 * (Y @ Y.conj().T.contiguous()).real
    # D_ii = sum_k |C_i X_ik - C_i X_ik|^2 is exactly 0 (and so is its gradient); the expanded
    # form leaves ~1e-15 relative rounding noise of either sign there, which alone would make
    # dL/d eps at eps ~ 2^-20 median (where every off-diagonal K underflows) -- so the
    # reference uses the op's definition, an exact zero diagonal.
    D = D.masked_fill(torch.eye(n, dtype=torch.bool), 0.0)
    K = torch.exp(-D[None] / (2 * eps[:, None, None]))
    return torch.log(K.sum(2)).sum(1), D


@pytest.mark.parametrize("n,N", [(48, 32), (160, 64)])
def test_backward_matches_float64_autograd_and_fd(cuda, n, N):
    import torch
    from manifoldem_python_amd import _native as nat, autograd, synth
    s = synth.make_pd(synth.seeds(7)[2], n, N)
    rng = np.random.default_rng(0)
    img64 = torch.as_tensor(rng.normal(size=(n, N, N)), dtype=torch.float64)
    df = torch.as_tensor(s.df, device=cuda)
    ctf = nat.ctf_params(synth.PIX, synth.CS, synth.EKV, synth.AMPC, np.inf)
    # median distance sets the eps scale: 2^-20 .. 2^20 x median (41 values)
    img = img64.to(torch.float32).to(cuda).requires_grad_(True)
    fy = torch.fft.rfft2(img)
    with torch.no_grad():
        L0 = autograd.kernel_logsum(fy, df, torch.ones(1, dtype=torch.float64, device=cuda), ctf)
    k = synth.ctf_grid_k(N, synth.PIX)[:, :N // 2 + 1]
    C64 = torch.as_tensor(synth.ctf_values(k[None], s.df[:, None, None]))
    w = torch.full((N // 2 + 1,), 2.0, dtype=torch.float64)
    w[0] = 1.0
    w[-1] = 1.0
    _, Dref = _ref_loss(img64, C64, w, torch.ones(1, dtype=torch.float64))
    med = float(torch.median(Dref[~torch.eye(n, dtype=torch.bool)]))
    eps = torch.as_tensor(med * 2.0 ** np.linspace(-20, 20, 41), device=cuda).requires_grad_(True)
    g = torch.as_tensor(rng.normal(size=41), device=cuda)
    L = autograd.kernel_logsum(fy, df, eps, ctf)
    (L * g).sum().backward()
    # float64 autograd reference
    x = img64.clone().requires_grad_(True)
    e = eps.detach().cpu().clone().requires_grad_(True)
    Lr, _ = _ref_loss(x, C64, w, e)
    (Lr * g.cpu()).sum().backward()
    np.testing.assert_allclose(L.detach().cpu().numpy(), Lr.detach().numpy(), rtol=1e-5,
                               atol=1e-5)
    ge = eps.grad.cpu().numpy()
    ger = e.grad.numpy()
    err_e = np.max(np.abs(ge - ger) / (np.abs(ger) + 1e-30 + 1e-6 * np.max(np.abs(ger))))
    gx = img.grad.cpu().numpy().astype(np.float64)
    gxr = x.grad.numpy()
    rel = np.linalg.norm(gx - gxr) / np.linalg.norm(gxr)
    err_x = np.max(np.abs(gx - gxr)) / np.max(np.abs(gxr))
    print(f"[autograd n={n} N={N}] dL/deps max rel {err_e:.3e}; dL/dX norm rel {rel:.3e}, "
          f"max/max {err_x:.3e}")
    # measured on the MI355X: 1.2e-6 / 1.4e-6 (eps), 2.1e-7 / 2.6e-7 (X, norm), 2.5e-7 /
    # 3.3e-7 (X, max) at n = 48 / 160: float32 rounding of the images and spectra
    assert err_e < 1e-5, err_e
    assert rel < 2e-6, rel
    assert err_x < 3e-6, err_x
    # the float64 reference itself against central differences (step 1e-3 relative)
    for e_idx in (10, 20, 30):
        h = 1e-3 * float(e.detach()[e_idx])
        ep, em = e.detach().clone(), e.detach().clone()
        ep[e_idx] += h
        em[e_idx] -= h
        fd = float(((_ref_loss(img64, C64, w, ep)[0] - _ref_loss(img64, C64, w, em)[0])
                    * g.cpu()).sum()) / (2 * h)
        assert abs(fd - ger[e_idx]) <= 1e-5 * max(1.0, abs(ger[e_idx]))
    for (i, a, b) in ((0, 3, 5), (7, 10, 20)):
        h = 1e-3 * float(img64.abs().mean())
        xp, xm = img64.clone(), img64.clone()
        xp[i, a, b] += h
        xm[i, a, b] -= h
        fd = float(((_ref_loss(xp, C64, w, e.detach())[0] - _ref_loss(xm, C64, w, e.detach())[0])
                    * g.cpu()).sum()) / (2 * h)
        assert abs(fd - gxr[i, a, b]) <= 1e-4 * max(1.0, np.max(np.abs(gxr)))


@pytest.mark.parametrize("n,ne", [(1, 1), (31, 16), (32, 17), (33, 41), (65, 3), (100, 32)])
@pytest.mark.parametrize("symmetric", [True, False])
def test_kernel_grad_weights_tiles(cuda, n, ne, symmetric):
    """memi_kernel_grad_weights at tile edges and eps counts around a round, for a symmetric D (one
    exponential for both entries) and any other, against float64: to float32 rounding."""
    import torch
    from manifoldem_python_amd import _native as nat
    rng = np.random.default_rng(n + ne)
    D = rng.uniform(0, 4, (n, n)).astype(np.float32)
    if symmetric:
        D = np.triu(D, 1) + np.triu(D, 1).T
    eps, S = rng.uniform(0.5, 2, ne), rng.uniform(1, 2, (ne, n))
    g = rng.standard_normal(ne)
    d = lambda a: torch.as_tensor(a, device=cuda)
    Wt = torch.empty((n, n), dtype=torch.float32, device=cuda)
    nat.kernel_grad_weights(d(D), d(eps), d(S), d(g), Wt)
    c = 1 / (2 * eps)[:, None, None]
    t = -g[:, None, None] * c * np.exp(-D.astype(np.float64) * c) * (1 / S[:, :, None] + 1 / S[:, None, :])
    want = t.sum(0)
    np.fill_diagonal(want, 0)
    assert np.max(np.abs(Wt.cpu().numpy() - want)) <= 2 ** -23 * max(np.max(np.abs(want)), 1e-30)


@pytest.mark.parametrize("n,N", [(1, 8), (3, 9), (5, 45), (2, 64)])
def test_gradient_operand_and_combination(cuda, n, N):
    """memi_grad_operand to the bit and memi_grad_combine to float32 rounding against numpy, at odd
    and even sides (the half-spectrum weights of the first and last column)."""
    import torch
    from manifoldem_python_amd import _native as nat
    rng = np.random.default_rng(n * N)
    Nh = N // 2 + 1
    X = (rng.standard_normal((n, N, Nh)) + 1j * rng.standard_normal((n, N, Nh))).astype(np.complex64)
    C = rng.uniform(-1, 1, (n, N, Nh)).astype(np.float32)
    WM = rng.standard_normal((n, 3, N, Nh)).astype(np.float32)
    d = lambda a: torch.as_tensor(a, device=cuda)
    M = torch.empty((n, 3, N, Nh), dtype=torch.float32, device=cuda)
    nat.grad_operand(d(X), d(C), N, M)
    np.testing.assert_array_equal(M.cpu().numpy(), np.stack([C * C, C * X.real, C * X.imag], 1))
    out = torch.empty((n, N, Nh), dtype=torch.complex64, device=cuda)
    nat.grad_combine(d(X), d(C), d(WM), N, out)
    w = np.full(Nh, 2.0)
    w[0] = 1.0
    if N % 2 == 0:
        w[-1] = 1.0
    W = WM.astype(np.float64)
    want = 2 * w * (X.astype(np.complex128) * W[:, 0] - C * (W[:, 1] + 1j * W[:, 2]))
    assert np.max(np.abs(out.cpu().numpy() - want)) < 4 * 2 ** -24 * np.max(np.abs(want))


def test_logsum_gradient_of_a_conjugate_view(cuda):
    """Images given as a lazily conjugated view: the same gradient as for the copy."""
    import torch
    from manifoldem_python_amd import _native as nat, autograd, synth
    rng = np.random.default_rng(3)
    base = torch.fft.rfft2(torch.as_tensor(rng.standard_normal((20, 16, 16)).astype(np.float32),
                                           device=cuda))
    df = torch.as_tensor(rng.uniform(5e3, 3e4, 20), device=cuda)
    ctf = nat.ctf_params(synth.PIX, synth.CS, synth.EKV, synth.AMPC, np.inf)
    eps = torch.tensor([2e3, 8e3], dtype=torch.float64, device=cuda)
    grads = []
    for lazy in (True, False):
        x = base.clone().requires_grad_(True)
        y = x.conj() if lazy else x.conj().resolve_conj()
        autograd.kernel_logsum(y, df, eps, ctf).sum().backward()
        grads.append(x.grad.resolve_conj().cpu().numpy())
    np.testing.assert_array_equal(grads[0], grads[1])
