"""GPU optical flow (CC stage) against the oracle: diffusion, block averages, Gaussian filter,
derivatives, Horn-Schunck iterations, the movie flow and the drop-in modules
(CC/hornschunck_simple.py, CC/OpticalFlowMovie.py)."""
import numpy as np
import pytest
import torch

from oracle import optflow as of

pytestmark = pytest.mark.gpu


def _smooth_movie(nmov, F, dim, seed):
    """Movies of drifting Gaussian blobs (amplitude ~100, so the diffusion's kappa = 50 acts
    non-linearly) plus noise: (nmov, F, dim*dim) float32."""
    rng = np.random.default_rng(seed)
    y, x = np.mgrid[0:dim, 0:dim].astype(np.float64)
    out = np.zeros((nmov, F, dim, dim))
    for m in range(nmov):
        for b in range(3):
            cy, cx = rng.uniform(0.3, 0.7, 2) * dim
            vy, vx = rng.uniform(-0.3, 0.3, 2)
            a = rng.uniform(50, 150)
            s = rng.uniform(0.08, 0.15) * dim
            for f in range(F):
                out[m, f] += a * np.exp(-((y - cy - vy * f) ** 2 + (x - cx - vx * f) ** 2)
                                        / (2 * s * s))
    out += 2.0 * rng.normal(size=out.shape)
    return out.reshape(nmov, F, dim * dim).astype(np.float32)


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda")


@pytest.mark.parametrize("option", [1, 2])
def test_anisodiff_matches_oracle(cuda, option):
    from manifoldem_python_amd import optflow
    mov = _smooth_movie(3, 12, 20, 0).reshape(3, 12, 20, 20)
    mov[:, :, :, :3] *= 3.0
    got = optflow.anisodiff3(_dev(mov), 5, 50, 0.1, (5., 3., 3.), option).cpu().numpy()
    for m in range(3):
        ref = of.anisodiff3(mov[m], niter=5, kappa=50, gamma=0.1, step=(5., 3., 3.),
                            option=option)
        np.testing.assert_allclose(got[m], ref, rtol=2e-6, atol=2e-6 * np.abs(ref).max())
    one = optflow.anisodiff3(_dev(mov), 1).cpu().numpy()
    np.testing.assert_array_equal(one, mov)


@pytest.mark.parametrize("shape", [(2, 7, 33, 31), (1, 1, 5, 4), (1, 3, 2, 1100), (3, 2, 40, 1),
                                   (1, 40, 32, 32), (40, 3, 64, 33)])
@pytest.mark.parametrize("option", [1, 2])
def test_anisodiff_blocks_and_frame_pieces(cuda, shape, option):
    """Pixels across the diffusion's blocks (rows that end inside one, a row longer than one) and
    frames in one or several pieces, against the float32 update with the float64 exp rounded.
    Every operation but the exp is the same float32 operation; an exp off by one float32 ulp
    moves a voxel by at most gamma 2^-24 |flux| per face and step, 6 faces and 4 steps: below
    2e-7 of the movie's scale."""
    from manifoldem_python_amd import optflow
    rng = np.random.default_rng(sum(shape))
    mov = (60 * rng.normal(size=shape)).astype(np.float32)
    got = optflow.anisodiff3(_dev(mov), 5, 50, 0.1, (5., 3., 3.), option).cpu().numpy()
    f32 = np.float32
    for m in range(shape[0]):
        out = mov[m].copy()
        for _ in range(4):
            div = []
            for ax, h in ((0, 5.0), (1, 3.0), (2, 3.0)):
                d = np.zeros_like(out)
                lo = [slice(None)] * 3
                hi = [slice(None)] * 3
                lo[ax], hi[ax] = slice(None, -1), slice(1, None)
                d[tuple(lo)] = np.diff(out, axis=ax)
                q = d / f32(50)
                g = (np.exp(-(q * q).astype(np.float64)).astype(f32) if option == 1 else
                     f32(1) / (f32(1) + q * q)) / f32(h)
                fl = g * d
                v = fl.copy()
                v[tuple(hi)] -= fl[tuple(lo)]
                div.append(v)
            out = out + f32(0.1) * ((div[0] + div[1]) + div[2])
        np.testing.assert_allclose(got[m], out, rtol=0, atol=2e-7 * np.abs(mov).max())


def test_block_average_exact(cuda):
    from manifoldem_python_amd import _native as nat
    mov = _smooth_movie(2, 12, 9, 1).reshape(2, 12, 9, 9)
    out = torch.empty((2, 3, 9, 9), dtype=torch.float64, device="cuda")
    nat.flow_block_average(_dev(mov), 5, out)
    for m in range(2):
        np.testing.assert_array_equal(out[m].cpu().numpy(), of.block_average(mov[m], 5))


@pytest.mark.parametrize("shape,sig", [((3, 33, 40), 1.5), ((2, 17, 17), 2.0),
                                       ((1, 5, 4), 2.0)])
def test_gaussian_matches_scipy(cuda, shape, sig):
    from manifoldem_python_amd import optflow
    rng = np.random.default_rng(2)
    im = rng.normal(size=shape) * 40
    g64 = optflow.gaussian(_dev(im), sig, torch.float64).cpu().numpy()
    g32 = optflow.gaussian(_dev(im), sig, torch.float32).cpu().numpy()
    g32b = optflow.gaussian(_dev(im.astype(np.float32)), sig, torch.float32).cpu().numpy()
    for i in range(shape[0]):
        r64 = of.lowpassfilt(im[i], sig)
        r32 = of.lowpassfilt(im[i].astype(np.float32), sig)
        np.testing.assert_allclose(g64[i], r64, rtol=1e-13, atol=1e-13 * np.abs(r64).max())
        # float32 outputs of the same float64 sums: equal up to the last bit
        np.testing.assert_allclose(g32[i], r32, rtol=2.5e-7, atol=1e-7 * np.abs(r32).max())
        np.testing.assert_array_equal(g32b[i], g32[i])


def test_derivatives_exact(cuda):
    from manifoldem_python_amd import optflow
    rng = np.random.default_rng(3)
    frames = (rng.normal(size=(4, 19, 23)) * 10).astype(np.float32)
    pairs = np.array([[0, 1], [1, 2], [3, 3], [2, 0]], np.int32)
    fx, fy, ft = optflow.derivatives(_dev(frames), _dev(pairs))
    for p, (a, b) in enumerate(pairs):
        rx, ry, rt = of.compute_derivatives(frames[a], frames[b])
        np.testing.assert_array_equal(fx[p].cpu().numpy(), rx)
        np.testing.assert_array_equal(fy[p].cpu().numpy(), ry)
        np.testing.assert_array_equal(ft[p].cpu().numpy(), rt)


@pytest.mark.parametrize("H,W,niter", [(40, 56, 200), (33, 31, 7), (8, 70, 1), (20, 20, 0)])
def test_hs_op_matches_oracle(cuda, H, W, niter):
    """The drop-in op (Gaussian, derivatives, temporally blocked iterations over partial tiles)
    against the oracle, float64 flow."""
    from manifoldem_python_amd import hornschunck_simple as hs
    mov = _smooth_movie(1, 2, max(H, W), 4)[0].reshape(2, max(H, W), max(H, W))[:, :H, :W]
    U, V = hs.op(mov[0], mov[1], np.zeros(1), np.zeros(1), 2.0, 2.0, niter)
    Ur, Vr = of.hornschunck(mov[0], mov[1], np.zeros(1), np.zeros(1), 2.0, 2.0, niter)
    assert U.dtype == np.float64 and U.shape == (H, W)
    scale = max(np.abs(Ur).max(), np.abs(Vr).max(), 1e-30)
    np.testing.assert_allclose(U, Ur, rtol=0, atol=1e-9 * scale)
    np.testing.assert_allclose(V, Vr, rtol=0, atol=1e-9 * scale)


@pytest.mark.parametrize("H,W", [(1, 1), (2, 63), (65, 64), (63, 65), (64, 128), (129, 127),
                                 (40, 129), (41, 192), (70, 193), (130, 130), (200, 260)])
def test_hs_strips_match_direct_iteration(cuda, H, W):
    """The float64 iterations on register strips at the edges of their tiles (sides below, at and
    above 64, 128 and 192 columns, 40, 64 and 128 rows, several tiles each way), with large
    gradients, against the plain iteration.  uAvg is a weighted mean and the update contracts, so
    rounding (about 20 operations a step) adds up at most linearly: 37 x 20 x 1.1e-16 < 1e-13 of
    the flow's scale."""
    from scipy.ndimage import convolve
    from manifoldem_python_amd import optflow
    rng = np.random.default_rng(H * 1000 + W)
    nP, niter = 3, 37
    fx, fy, ft = (rng.normal(size=(3, nP, H, W)) * 3).astype(np.float32)
    U0, V0 = rng.normal(size=(2, nP, H, W))
    U, V = optflow.hs_iterate(_dev(fx), _dev(fy), _dev(ft), 2.0, niter, _dev(U0), _dev(V0))
    for p in range(nP):
        u, v = U0[p], V0[p]
        den = (np.float32(4.0) + fx[p] ** 2) + fy[p] ** 2
        top = max(np.abs(u).max(), np.abs(v).max())
        for _ in range(niter):
            ua, va = convolve(u, of.HSKERN), convolve(v, of.HSKERN)
            d = (fx[p] * ua + fy[p] * va + ft[p]) / den
            u, v = ua - fx[p] * d, va - fy[p] * d
            top = max(top, np.abs(u).max(), np.abs(v).max())
        np.testing.assert_allclose(U[p].cpu().numpy(), u, rtol=0, atol=1e-13 * top)
        np.testing.assert_allclose(V[p].cpu().numpy(), v, rtol=0, atol=1e-13 * top)


def test_hs_float32_start(cuda):
    """A float32 initial flow keeps the iteration in float32, as numpy does."""
    from manifoldem_python_amd import hornschunck_simple as hs
    mov = _smooth_movie(1, 2, 36, 5)[0].reshape(2, 36, 36)
    rng = np.random.default_rng(6)
    u0 = rng.normal(size=(36, 36)).astype(np.float32) * 0.1
    v0 = rng.normal(size=(36, 36)).astype(np.float32) * 0.1
    U, V = hs.op(mov[0], mov[1], u0, v0, 1.5, 2.0, 50)
    Ur, Vr = of.hornschunck(mov[0], mov[1], u0, v0, 1.5, 2.0, 50)
    assert U.dtype == np.float32 and Ur.dtype == np.float32
    scale = max(np.abs(Ur).max(), np.abs(Vr).max())
    np.testing.assert_allclose(U, Ur, rtol=0, atol=2e-6 * scale)
    np.testing.assert_allclose(V, Vr, rtol=0, atol=2e-6 * scale)


def _check_flow(res, m, Vx, Vy, tol):
    scale = max(np.abs(Vx).max(), np.abs(Vy).max())
    gx = res["Vx"][m].cpu().numpy()
    gy = res["Vy"][m].cpu().numpy()
    np.testing.assert_allclose(gx, Vx, rtol=0, atol=tol * scale)
    np.testing.assert_allclose(gy, Vy, rtol=0, atol=tol * scale)
    o, mag = of.get_orient_mag(Vx, Vy)
    np.testing.assert_allclose(res["Mag"][m].cpu().numpy(), mag, rtol=0, atol=tol * scale)
    big = mag > 1e-3 * scale  # the orientation is defined away from zero flow
    d = np.abs(res["Orient"][m].cpu().numpy() - o)[big]
    d = np.minimum(d, 2 * np.pi - d)  # (atan2 % 2) * pi wraps at 2 pi
    # a flow error e turns the angle by at most ~e / |flow|, scaled by pi in (atan2 % 2) * pi
    assert np.all(d <= np.pi * 2 * tol * scale / mag[big] + 1e-12)


# The diffusion's float32 exp is the float64 exp rounded, numpy's is its own SIMD float32 exp:
# they differ by up to an ulp, so the diffused frames agree to ~1e-6 relative, and the flow
# (driven by frame differences) to a few 1e-6 of its maximum.  The steps after the diffusion
# are checked at 1e-9 from the same diffused movie.
WHOLE_CHAIN_TOL = 2e-5


def _diffused(movs):
    from manifoldem_python_amd import optflow
    nmov, F, hw = movs.shape
    dim = int(np.sqrt(hw))
    d = optflow.anisodiff3(_dev(movs.reshape(nmov, F, dim, dim)), **optflow.ANISO)
    return d.cpu().numpy().reshape(nmov, F, hw)


def test_movie_flow_hs_matches_oracle(cuda):
    from manifoldem_python_amd import optflow
    movs = _smooth_movie(2, 23, 36, 7)
    res = optflow.movie_flows(movs, 5, "HS")
    dif = _diffused(movs)
    for m in range(2):
        Vx, Vy = of.movie_flow(dif[m], 5, "HS", diffuse=False)
        _check_flow(res, m, Vx, Vy, 1e-9)
        Vx2, Vy2 = of.movie_flow(movs[m], 5, "HS")
        _check_flow(res, m, Vx2, Vy2, WHOLE_CHAIN_TOL)
        o_rev, mag = of.get_orient_mag(-Vx, -Vy)
        scale = max(np.abs(Vx).max(), np.abs(Vy).max())
        big = mag > 1e-3 * scale
        d = np.abs(res["Orient_rev"][m].cpu().numpy() - o_rev)[big]
        d = np.minimum(d, 2 * np.pi - d)
        assert np.all(d <= np.pi * 2e-9 * scale / mag[big] + 1e-12)


def test_movie_flow_gf_hs_with_initial_flows(cuda):
    """'GF-HS' with given (float32) initial flows: pre-filtered frames, sigma 1.5, float32
    iterations."""
    from manifoldem_python_amd import optflow
    movs = _smooth_movie(1, 10, 32, 8)
    rng = np.random.default_rng(9)
    A = 2
    u0 = (0.2 * rng.normal(size=(1, A, 32, 32))).astype(np.float32)
    v0 = (0.2 * rng.normal(size=(1, A, 32, 32))).astype(np.float32)
    res = optflow.movie_flows(movs, 5, "GF-HS", (u0, v0))
    init = [(u0[0, a], v0[0, a]) for a in range(A)]
    Vx, Vy = of.movie_flow(_diffused(movs)[0], 5, "GF-HS", init, diffuse=False)
    _check_flow(res, 0, Vx, Vy, 1e-5)  # float32 iterations
    Vx2, Vy2 = of.movie_flow(movs[0], 5, "GF-HS", init)
    _check_flow(res, 0, Vx2, Vy2, WHOLE_CHAIN_TOL)


def test_movie_flow_full_size(cuda):
    """One 50-frame movie of 160 x 160 frames (the NLSA movie shape) against the oracle, and a
    static movie of that size has exactly zero flow."""
    from manifoldem_python_amd import optflow
    mov = _smooth_movie(1, 50, 160, 10)
    res = optflow.movie_flows(mov, 5, "HS")
    Vx, Vy = of.movie_flow(_diffused(mov)[0], 5, "HS", diffuse=False)
    _check_flow(res, 0, Vx, Vy, 1e-9)
    Vx2, Vy2 = of.movie_flow(mov[0], 5, "HS")
    _check_flow(res, 0, Vx2, Vy2, WHOLE_CHAIN_TOL)
    static = np.repeat(mov[:, :1], 50, axis=1)
    z = optflow.movie_flows(static, 5, "HS")
    assert float(z["Vx"].abs().max()) == 0.0 and float(z["Vy"].abs().max()) == 0.0


def test_dropin_movie_op(cuda):
    from manifoldem_python_amd import OpticalFlowMovie as ofm
    mov = _smooth_movie(1, 20, 28, 11)[0]
    with pytest.raises(NotImplementedError):
        ofm.op(mov, [0, 0], 5, "FWD", [0, 0])
    old = ofm.OF_Type
    ofm.OF_Type = "HS"
    try:
        fwd = ofm.op(mov, [0, 0], 5, "FWD", [0, 0])
        rev = ofm.op(mov, [0, 0], 5, "REV", [0, 0], fwd)
    finally:
        ofm.OF_Type = old
    Vx, Vy = of.movie_flow(_diffused(mov[None])[0], 5, "HS", diffuse=False)
    scale = np.abs(Vx).max()
    np.testing.assert_allclose(fwd["Vx"], Vx, rtol=0, atol=1e-9 * scale)
    np.testing.assert_allclose(rev["Vx"], -Vx, rtol=0, atol=1e-9 * scale)
    np.testing.assert_allclose(rev["Vy"], -Vy, rtol=0, atol=1e-9 * scale)
    o, mag = of.get_orient_mag(-Vx, -Vy)
    np.testing.assert_allclose(rev["Mag"], mag, rtol=0, atol=1e-9 * scale)
    big = mag > 1e-3 * scale
    d = np.abs(rev["Orient"] - o)[big]
    d = np.minimum(d, 2 * np.pi - d)
    assert np.all(d <= np.pi * 2e-9 * scale / mag[big] + 1e-12)
    # getOrientMag on given arrays keeps signed zeros: atan2(-0., -1) = -pi
    o2, m2 = ofm.getOrientMag(np.array([-1.0, 3.0]), np.array([-0.0, 4.0]))
    ro, rm = of.get_orient_mag(np.array([-1.0, 3.0]), np.array([-0.0, 4.0]))
    np.testing.assert_allclose(o2, ro, rtol=1e-15)
    np.testing.assert_allclose(m2, rm, rtol=1e-15)


def test_dropin_lowpass_and_aniso(cuda):
    from manifoldem_python_amd import OpticalFlowMovie as ofm
    from manifoldem_python_amd import hornschunck_simple as hs
    rng = np.random.default_rng(12)
    im = rng.normal(size=(21, 18))
    np.testing.assert_allclose(hs.lowpassfilt(im, 1.5), of.lowpassfilt(im, 1.5), rtol=1e-13,
                               atol=1e-14)
    st = (60 * rng.normal(size=(5, 9, 11))).astype(np.float32)
    ref = of.anisodiff3(st, 5, 50, 0.1, (5., 3., 3.), 1)
    np.testing.assert_allclose(ofm.anisodiff3(st, 5, 50, 0.1, (5., 3., 3.), 1), ref, rtol=2e-6,
                               atol=2e-6 * np.abs(ref).max())
    a, b = (rng.normal(size=(2, 12, 13)) * 5).astype(np.float32)
    for x, y in zip(hs.computeDerivatives(a, b), of.compute_derivatives(a, b)):
        np.testing.assert_array_equal(x, y)
