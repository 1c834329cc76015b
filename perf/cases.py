"""The calls this package is timed on: what a program that embeds cryo-EM projection directions
(PDs) has it do, over the sizes it meets.

A case is a dict of plain values.  ``prepare`` makes on the GPU what such a program holds before
the call (images, angles, plans, buffers), ``run`` is one pass through the public entry points,
``work`` is what the pass cannot do without, and ``exact`` gives the same outputs in float64 from
plain torch / numpy, without this package's code.

Kinds of case:

* ``distances``  ``batch.distances``: raw images of one or many PDs to their distance matrices;
* ``particles``  the per-PD stage-1 outputs: ``pipeline.prepare_images`` under a volume mask,
  ``pipeline.averages`` and ``pipeline.ctf_distances`` (images, spectra, CTFs, averages, D);
* ``embed``      ``pipeline.dm_embed``: distance matrices to diffusion-map coordinates;
* ``nlsa``       NLSA along one diffusion coordinate between its two embeddings: delay-embedded
                 distances, Wiener-filtered supervectors, reconstructed frames and their distances;
* ``flow``       ``optflow.movie_flows``: Horn-Schunck optical flow of a batch of movies;
* ``logsum``     ``autograd.kernel_logsum``, forward and backward.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from manifoldem_python_amd import _native as nat
from manifoldem_python_amd import autograd, batch as B, optflow, synth
from manifoldem_python_amd import pipeline as pl

FILTER = dict(type="Butter", Qc=0.5, N=8)
DF_UM = (0.5, 3.0)


def listed():
    return [
        # one small PD of a low-resolution stack: launches and latency count
        dict(name="distances_small", kind="distances", n=200, npd=1, N=70, prec="split"),
        # one large PD at the default precision
        dict(name="distances_large", kind="distances", n=2000, npd=1, N=128, prec="split"),
        # an odd box side, a ragged particle count, conjugate particles, float32 arithmetic
        dict(name="distances_odd_fp32", kind="distances", n=777, npd=1, N=105, prec="fp32",
             conj=0.25),
        # a batch of PDs of uneven (lognormal) occupancy, the throughput path
        dict(name="distances_batch", kind="distances", n=400, npd=64, N=96, prec="split"),
        # the stage-1 drop-in's outputs of one PD at a larger box under a volume mask
        dict(name="particles_masked", kind="particles", n=500, N=180, prec="split"),
        # a small PD with the full kernel and a coarse bandwidth grid
        dict(name="embed_small", kind="embed", n=200, npd=1, k=0, eps=101, eigs=8),
        # the drivers' setting: every neighbour kept, 15 eigenpairs, the 1501-point grid
        dict(name="embed_full", kind="embed", n=1273, npd=1, k=0, eps=1501, eigs=15),
        # one large PD with 200 neighbours kept
        dict(name="embed_knn", kind="embed", n=2000, npd=1, k=200, eps=1501, eigs=10),
        # a batch of PDs of uneven occupancy with 150 neighbours kept
        dict(name="embed_batch", kind="embed", n=400, npd=64, k=150, eps=1501, eigs=8),
        # NLSA of one coordinate of a PD of 1500 images
        dict(name="nlsa_frames", kind="nlsa", n=1500, N=160, con=50, trunc=8),
        # optical flow of the movies of many PDs
        dict(name="flow_movies", kind="flow", movies=64, frames=50, N=128),
        # gradient of the kernel log-sum with respect to images and bandwidths
        dict(name="logsum_grad", kind="logsum", n=1000, N=128, eps=41, prec="fp32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _side(rng, lo, hi):
    """A box side: mostly products of small primes (as boxes are cropped to), odd ones among
    them, now and then any other."""
    smooth = []
    for s in range(lo, hi + 1):
        r = s
        for q in (2, 3, 5, 7):
            while r % q == 0:
                r //= q
        if r == 1:
            smooth.append(s)
    return rng.randint(lo, hi) if rng.random() < 0.1 else rng.choice(smooth)


def draw(rng):
    kind = rng.choice(["distances", "distances", "distances", "particles", "embed", "embed",
                       "embed", "nlsa", "flow", "logsum"])
    prec = rng.choice(["split", "split", "fp32"])
    if kind == "distances":
        npd = rng.choice([1, 1, _log_int(rng, 2, 64)])
        n = _log_int(rng, 64, 2000 if npd == 1 else 400)
        return dict(kind=kind, n=n, npd=npd, N=_side(rng, 48, 128 if npd == 1 else 96),
                    prec=prec, conj=rng.choice([0.0, 0.25]))
    if kind == "particles":
        return dict(kind=kind, n=_log_int(rng, 64, 500), N=_side(rng, 64, 180), prec=prec)
    if kind == "embed":
        npd = rng.choice([1, 1, _log_int(rng, 2, 64)])
        n = _log_int(rng, 64, 2000 if npd == 1 else 400)
        return dict(kind=kind, n=n, npd=npd, k=rng.choice([0, 0, rng.randint(20, 200)]),
                    eps=rng.choice([101, 301, 1501]), eigs=rng.randint(4, 15))
    if kind == "nlsa":
        return dict(kind=kind, n=_log_int(rng, 300, 1500), N=_side(rng, 64, 160),
                    con=rng.randint(20, 50), trunc=rng.choice([8, 8, rng.randint(3, 8)]))
    if kind == "flow":
        return dict(kind=kind, movies=_log_int(rng, 1, 64), frames=rng.randint(20, 50),
                    N=_side(rng, 48, 128))
    return dict(kind=kind, n=_log_int(rng, 100, 1000), N=_side(rng, 48, 128),
                eps=rng.randint(8, 41), prec=prec)


# ---------------------------------------------------------------- inputs ------------------
def _sizes(case):
    """Particles per PD: one PD of n, or a lognormal batch with median n."""
    if case.get("npd", 1) == 1:
        return [int(case["n"])]
    n = int(case["n"])
    return [int(v) for v in synth.lognormal_sizes(5, case["npd"], median=n, sigma=0.6,
                                                  lo=max(32, n // 4), hi=6 * n)]


def _prec(case):
    return nat.PREC_FP32 if case["prec"] == "fp32" else nat.PREC_SPLIT_BF16


def _pds(case, seed):
    """Synthetic PDs: noisy CTF-affected projections of a moving blob volume."""
    dev = torch.device("cuda")
    out = []
    for p, n in enumerate(_sizes(case)):
        rng = np.random.default_rng([int(seed), p])
        out.append(synth.make_pd(rng.integers(1 << 62), n, case["N"], df_range_um=DF_UM,
                                 axis=synth.random_axis(rng), device=dev, as_torch=True,
                                 conj_frac=case.get("conj", 0.0)))
    return out


def _ctf_params():
    return nat.ctf_params(synth.PIX, synth.CS, synth.EKV, synth.AMPC, np.inf)


def _batch(case, seed):
    ss = _pds(case, seed)
    pds, off = [], 0
    for s in ss:
        conj = s.ind >= s.nStot // 2
        src = np.where(conj, s.ind - s.nStot // 2, s.ind) + off
        n = len(s.ind)
        pds.append(dict(src=src, conj=conj.astype(np.int32), q=s.q, df=s.df,
                        k=min(case.get("k") or n, n)))
        off += n
    stack = torch.cat([s.raw for s in ss]).contiguous()
    b = B.make_batch(stack, pds, case["N"], _ctf_params(), FILTER, stack.device)
    return b, ss


def _distance_like(n, seed, t=None):
    """A distance matrix as stage 1 gives one: squared distances of points on a curved
    one-parameter manifold, with the pedestal and spread that image noise adds (many independent
    directions of falling variance).  t: the points' places on it.  Symmetric float32, zero
    diagonal."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(int(seed))
    t = (torch.rand(n, 1, generator=g, dtype=torch.float64, device=dev) if t is None else
         torch.as_tensor(t, device=dev).view(n, 1))
    j = torch.arange(1, 7, dtype=torch.float64, device=dev)
    signal = torch.cos(math.pi * t * j) / j
    d = torch.arange(96, dtype=torch.float64, device=dev)
    noise = torch.randn(n, 96, generator=g, dtype=torch.float64, device=dev) * 0.25 * 0.96 ** d
    x = 60.0 * torch.cat([signal, noise], 1)
    s = (x * x).sum(1)
    G = s[:, None] + s[None, :] - 2.0 * (x @ x.t())
    G = torch.triu(G.clamp(min=1.0), 1)
    return (G + G.t()).float().contiguous()


def _eps_grid(m):
    return pl.LOG_EPS if m == len(pl.LOG_EPS) else np.linspace(-150.0, 150.0, m)


def _starts(seed, npd):
    rng = np.random.default_rng([int(seed), 7])
    return [rng.random((4, 1)) - 0.5 for _ in range(npd)]


def _rand(seed):
    rng = np.random.default_rng([int(seed), 8])
    return lambda *shape: rng.random(shape)


def prepare(case, seed):
    dev = torch.device("cuda")
    kind = case["kind"]
    st = dict(case=dict(case), seed=int(seed), kind=kind)
    if kind == "distances":
        st["batch"], _ = _batch(case, seed)
        st["wsp"] = B.Workspace(st["batch"], _prec(case))
    elif kind == "particles":
        s = _pds(dict(case, npd=1), seed)[0]
        n, N = case["n"], case["N"]
        geo = pl.pd_geometry(s.q)
        st.update(stack=s.raw, src=torch.arange(n, device=dev),
                  conj=torch.zeros(n, dtype=torch.int32, device=dev),
                  rot1=torch.as_tensor(-(180 / math.pi) * geo["Psi"], device=dev),
                  rot2=torch.full((n,), -geo["psi_p"], dtype=torch.float64, device=dev),
                  df=torch.as_tensor(s.df, device=dev), msk=_mask(N, dev), ctf=_ctf_params(),
                  op=pl.Operand(n, N, _prec(case), dev),
                  plan=nat.Plan([0], [n], [n], chunks=pl.CHUNKS[_prec(case)], device=dev))
    elif kind == "embed":
        ns = _sizes(case)
        rows0 = np.concatenate([[0], np.cumsum(ns)[:-1]]).astype(np.int64)
        ks = [min(case["k"] or n, n) for n in ns]
        st["plan"] = nat.Plan(rows0, ns, ks, device=dev)
        D = torch.zeros(max(st["plan"].info.d_elems, 1), dtype=torch.float32, device=dev)
        for p, n in enumerate(ns):
            st["plan"].block(D, p).copy_(_distance_like(n, 1000 * seed + p).view_as(
                st["plan"].block(D, p)))
        st.update(D=D, logEps=_eps_grid(case["eps"]), a0s=_starts(seed, len(ns)))
    elif kind == "nlsa":
        n, N, con, tr = case["n"], case["N"], case["con"], case["trunc"]
        m, rec = n - con, n - 2 * con
        s = _pds(dict(case, npd=1), seed)[0]
        order = np.argsort(s.t)
        C = synth.ctf_values(synth.ctf_grid_k(N, synth.PIX)[None, :, :N // 2 + 1],
                             s.df[order][:, None, None])
        # the measure and coordinates of the first embedding: cosines along the manifold
        t = (np.arange(m) + 0.5) / m
        mu = np.random.default_rng([int(seed), 9]).uniform(0.5, 1.5, m)
        psi = np.cos(math.pi * t[:, None] * np.arange(tr)) * math.sqrt(2.0)
        psi[:, 0] = 1.0
        g = torch.Generator(device=dev).manual_seed(int(seed))
        # the two leading topos of every delay, and their chronos as a Hankel matrix
        U = torch.randn(N * N, 2 * con, generator=g, dtype=torch.float64, device=dev) / N
        z = np.stack([math.sqrt(m) * psi[:, 0] + 0.3 * psi[:, 1], 0.8 * psi[:, 1] + psi[:, 2]])
        H = z[:, np.arange(con)[:, None] + np.arange(rec)[None, :]].reshape(2 * con, rec)
        st.update(D=_distance_like(n, seed, s.t), ord=torch.as_tensor(order, device=dev),
                  img=0.1 * s.raw.transpose(1, 2)[torch.as_tensor(order, device=dev)],
                  ctf=torch.as_tensor(C.reshape(n, -1).astype(np.float32), device=dev),
                  mu_psi=torch.as_tensor(mu[:, None] / mu.sum() * psi, device=dev), U=U,
                  H=torch.as_tensor(H, device=dev).contiguous())
    elif kind == "flow":
        st["movies"] = _movies(case, seed)
    else:
        n, N = case["n"], case["N"]
        s = _pds(dict(case, npd=1), seed)[0]
        img = s.raw.transpose(1, 2)
        st.update(fy=torch.fft.rfft2(img / img.std()).contiguous().requires_grad_(True),
                  df=torch.as_tensor(s.df, device=dev), ctf=_ctf_params())
        lo = math.log(0.02 * N ** 4)
        st["eps"] = torch.exp(torch.linspace(lo, lo + 6.0, case["eps"], dtype=torch.float64,
                                             device=dev)).float().requires_grad_(True)
    return st


def _mask(N, dev):
    """The projection of a roughly spherical volume mask (1 inside, 0 outside)."""
    g = torch.arange(N, dtype=torch.float32, device=dev) - N / 2
    return ((g[:, None] ** 2 + 1.3 * g[None, :] ** 2) < (0.4 * N) ** 2).float().contiguous()


def _movies(case, seed):
    """Blobs that drift, with noise: (movies, frames, N, N) float32."""
    dev = torch.device("cuda")
    m, F, N = case["movies"], case["frames"], case["N"]
    g = torch.Generator(device=dev).manual_seed(int(seed))
    r = lambda *s: torch.rand(*s, generator=g, device=dev)
    c0 = N * (0.25 + 0.5 * r(m, 6, 2))
    v = 0.08 * N * (r(m, 6, 2) - 0.5)
    sig = N * (0.05 + 0.08 * r(m, 6))
    amp = 20 + 60 * r(m, 6)
    t = torch.linspace(0, 1, F, device=dev)
    c = c0[:, None] + v[:, None] * t[None, :, None, None]              # (m, F, 6, 2)
    x = torch.arange(N, device=dev, dtype=torch.float32)
    e = lambda a: torch.exp(-(x - c[..., a, None]) ** 2 / (2 * sig[:, None, :, None] ** 2))
    mov = torch.matmul((e(0) * amp[:, None, :, None]).transpose(2, 3).contiguous(), e(1))
    return (mov + torch.randn(mov.shape, generator=g, device=dev)).contiguous()


# ---------------------------------------------------------------- one pass ----------------
def _oriented(psis):
    """Coordinates of the PDs, row after row, each with the sign that makes its PD's first
    particle positive (an eigenvector's own sign is free)."""
    sign = np.repeat([np.where(p[0] < 0, -1.0, 1.0) for p in psis], [len(p) for p in psis],
                     axis=0)
    return np.concatenate(psis) * sign


def _embedding(res):
    """Eigenvalues, coordinates, measures, bandwidths and log sums of the PDs, packed."""
    return dict(lamb=np.concatenate([r.lamb for r in res]),
                psi=_oriented([r.psi for r in res]),
                mu=np.concatenate([r.mu for r in res]),
                sigma=np.array([r.sigma for r in res]),
                logSumWij=np.stack([r.logSumWij for r in res]))


def _nlsa_frames(st):
    n, N, con, tr = (st["case"][k] for k in ("n", "N", "con", "trunc"))
    dev = st["D"].device
    m, rec = n - con, n - 2 * con
    f64 = lambda *shape: torch.empty(shape, dtype=torch.float64, device=dev)
    ConD = f64(m, m)
    nat.nlsa_condist(st["D"].reshape(-1), st["ord"], n, con, ConD)
    spec = torch.fft.rfft2(st["img"]).contiguous()
    sv = torch.empty((con, tr, N, N // 2 + 1), dtype=torch.complex64, device=dev)
    nat.nlsa_supervectors(spec, st["ctf"], n, N, con, st["mu_psi"], 5.0, sv)
    A = torch.fft.irfft2(sv, s=(N, N))
    U, Gq, inv_sd, ws = st["U"].clone(), f64(2 * con, 2 * con), f64(rec), f64((2 * con + 1) * rec)
    nat.center_gram(U, Gq)
    D2 = torch.empty((rec, rec), dtype=torch.float32, device=dev)
    nat.nlsa_recon_dist(Gq, st["H"], N * N, inv_sd, D2, ws)
    IMGT = f64(N * N, rec)
    nat.nlsa_imgt(U, st["H"], inv_sd, IMGT)
    return dict(ConD=ConD, A=A, D2=D2, inv_sd=inv_sd, IMGT=IMGT)


def run(st):
    kind, case = st["kind"], st["case"]
    if kind == "distances":
        return B.distances(st["batch"], st["wsp"]).D
    if kind == "particles":
        N = case["N"]
        out = pl.prepare_images(st["stack"], st["src"], st["conj"], st["rot1"], st["rot2"],
                                st["df"], N, FILTER, st["ctf"], operand=st["op"],
                                msk2=st["msk"])
        avg = pl.averages(out["imgAll"], out["fy"], out["ctf"], N, msk2=st["msk"])
        D = pl.ctf_distances(st["plan"], st["op"], out["fy"], out["ctf"], N).D
        return dict(out, **avg, D=D)
    if kind == "embed":
        return _embedding(pl.dm_embed(st["plan"], st["D"], 3, case["eigs"], st["logEps"],
                                      rand=_rand(st["seed"]), a0s=st["a0s"]))
    if kind == "nlsa":
        return _nlsa_frames(st)
    if kind == "flow":
        return optflow.movie_flows(st["movies"])
    L = autograd.kernel_logsum(st["fy"], st["df"], st["eps"], st["ctf"], _prec(case))
    g_fy, g_eps = torch.autograd.grad(L.sum(), (st["fy"], st["eps"]))
    return dict(L=L.detach().float(), g_fy=g_fy, g_eps=g_eps)


# ---------------------------------------------------------------- necessary work ----------
def _prep_work(n, N):
    """Raw images in; three real 2-D FFTs, two 16-tap spline rotations with their prefilters and
    the CTF per pixel; the packed row (four float32 segments of the half spectrum) out."""
    kh = N * (N // 2 + 1)
    return dict(bytes=4.0 * n * N * N, flops=n * (3 * 2.5 * N * N * math.log2(N * N) +
                                                 2 * 60.0 * N * N + 30.0 * kh))


def _gram_work(n, N):
    kh = N * (N // 2 + 1)
    return dict(bytes=4.0 * n * n, flops=8.0 * kh * n * (n - 1) / 2)


def _embed_work(n, k, eps, eigs):
    """D in, coordinates out; the kernel's row sums and normalisation over its entries, one
    product with the kernel for every two eigenpairs and eight more."""
    nnz = float(n) * min(2 * k, n)
    return dict(bytes=4.0 * n * n + 8.0 * n * (eigs + 2) + 8.0 * eps,
                flops=20.0 * nnz + 2.0 * nnz * (2 * eigs + 8))


def work(case):
    kind = case["kind"]
    parts = []
    if kind == "distances":
        for n in _sizes(case):
            parts += [_prep_work(n, case["N"]), _gram_work(n, case["N"])]
    elif kind == "embed":
        for n in _sizes(case):
            parts.append(_embed_work(n, case["k"] or n, case["eps"], case["eigs"]))
    elif kind == "particles":
        n, N = case["n"], case["N"]
        kh = N * (N // 2 + 1)
        parts += [_prep_work(n, N), _gram_work(n, N),
                  dict(bytes=n * (8.0 * N * N + 12.0 * kh), flops=n * 5.0 * N * N * 14)]
    elif kind == "nlsa":
        n, N, con, tr = case["n"], case["N"], case["con"], case["trunc"]
        m, rec, kh = n - con, n - 2 * con, N * (N // 2 + 1)
        parts += [dict(bytes=4.0 * n * n + 8.0 * m * m, flops=2.0 * m * m),
                  dict(bytes=4.0 * n * N * N + 4.0 * n * kh + 4.0 * con * tr * N * N,
                       flops=4.0 * kh * con * tr * m + 2.5 * N * N * math.log2(N * N) *
                       (n + con * tr)),
                  dict(bytes=8.0 * N * N * (rec + 2 * con) + 8.0 * 2 * con * rec,
                       flops=2.0 * N * N * 2 * con * (rec + con)),
                  dict(bytes=4.0 * rec * rec, flops=2.0 * rec * rec / 2 * 2 * con)]
    elif kind == "flow":
        m, F, N = case["movies"], case["frames"], case["N"]
        px = float(N * N)
        parts.append(dict(bytes=m * px * (4.0 * F + 5 * 8.0),
                          flops=m * px * (F * 4 * 40.0 + -(-F // 5) * 200 * 34.0)))
    else:
        n, N, e = case["n"], case["N"], case["eps"]
        kh = N * (N // 2 + 1)
        parts += [_gram_work(n, N), dict(bytes=n * 16.0 * kh,
                                         flops=2.0 * n * n * 3 * kh + 2.0 * n * n * e * 4)]
    return dict(bytes=sum(p["bytes"] for p in parts), flops=sum(p["flops"] for p in parts))


# ---------------------------------------------------------------- float64 answers ---------
def _disk(N, dev):
    xx = torch.arange(N, dtype=torch.float64, device=dev)[:, None] - N / 2 + 1
    yy = torch.arange(N, dtype=torch.float64, device=dev)[None, :] - N / 2
    return ((xx * xx + yy * yy) < (N / 2.0) ** 2).double()


def _radius(N, dev):
    a = (np.arange(-(N - 1) / 2, (N - 1) / 2 + 1) if N % 2 else np.arange(-N / 2, N / 2))
    X, Y = np.meshgrid(a, a)
    return torch.as_tensor(np.fft.ifftshift((1.0 / (N / 2.0)) * np.sqrt(X ** 2 + Y ** 2)),
                           device=dev)


def _rotate(img, deg):
    """Order-3 spline rotation of each periodically continued image about its tile's centre."""
    n, N, _ = img.shape
    dev = img.device
    sym = (4.0 + 2.0 * torch.cos(2 * math.pi * torch.fft.fftfreq(N, dtype=torch.float64,
                                                                 device=dev))) / 6.0
    coef = torch.fft.ifft2(torch.fft.fft2(img) / (sym[:, None] * sym[None, :])).real
    a = deg.double() * (math.pi / 180)
    c, s = torch.cos(a)[:, None, None], torch.sin(a)[:, None, None]
    ctr = (3 * N - 1) / 2.0
    r = (torch.arange(N, dtype=torch.float64, device=dev) + N - ctr)[None, :, None]
    q = (torch.arange(N, dtype=torch.float64, device=dev) + N - ctr)[None, None, :]
    y, x = c * r + s * q + ctr, -s * r + c * q + ctr
    fy, fx = torch.floor(y), torch.floor(x)

    def weights(t):
        u = 1.0 - t
        return (u ** 3 / 6, (4 - 6 * t ** 2 + 3 * t ** 3) / 6,
                (4 - 6 * u ** 2 + 3 * u ** 3) / 6, t ** 3 / 6)

    wy, wx = weights(y - fy), weights(x - fx)
    iy, ix = fy.long() - 1, fx.long() - 1
    flat = coef.reshape(n, N * N)
    out = torch.zeros_like(img)
    for i in range(4):
        row = torch.remainder(iy + i, N) * N
        for j in range(4):
            at = (row + torch.remainder(ix + j, N)).reshape(n, N * N)
            out += wy[i] * wx[j] * torch.gather(flat, 1, at).view(n, N, N)
    return out


def _geometry(q):
    PDs = 2 * np.vstack((q[1] * q[3] - q[0] * q[2], q[0] * q[1] + q[2] * q[3],
                         q[0] ** 2 + q[3] ** 2 - 0.5))
    PD = PDs.sum(1)
    PD = PD / np.linalg.norm(PD)
    s = -(1 + PD[2]) * q[3] - PD[0] * q[1] - PD[1] * q[2]
    c = (1 + PD[2]) * q[0] + PD[1] * q[1] - PD[0] * q[2]
    with np.errstate(divide="ignore", invalid="ignore"):
        psi = 2 * np.arctan(s / c)
    return np.where(np.isnan(psi), 0.0, psi)


def _exact_images(raw, conj, rot1, rot2, df, N):
    """Aligned images, their spectra and CTFs of one PD in float64."""
    dev = raw.device
    disk, Q = _disk(N, dev), _radius(N, dev)
    y = raw.double().transpose(1, 2)
    y = torch.where(conj.bool()[:, None, None], torch.flip(y, dims=[1]), y)
    bg = y * (1 - disk)
    mean = bg.mean(dim=(1, 2), keepdim=True)
    y = (y - mean) / torch.sqrt(((bg - mean) ** 2).mean(dim=(1, 2), keepdim=True))
    G = torch.sqrt(1.0 / (1 + (Q / FILTER["Qc"]) ** (2 * FILTER["N"])))
    y = torch.fft.ifft2(torch.fft.fft2(y) * G).real * disk
    y = _rotate(_rotate(y, rot1), rot2)
    C = torch.as_tensor(_exact_ctf(Q.cpu().numpy() / (2 * synth.PIX), df.cpu().numpy()),
                        device=dev)
    return y, C


def _exact_ctf(k, df):
    """CTF(k) of each defocus: sin(w) - A cos(w), w = (pi Cs lam^3 k^2 / 2 - pi lam df) k^2."""
    lam = 12.3986 / math.sqrt((2 * 511.0 + synth.EKV) * synth.EKV)
    k2 = (k * k)[None]
    w = (0.5 * math.pi * synth.CS * 1e7 * lam ** 3 * k2 - math.pi * lam * df[:, None, None]) * k2
    return np.sin(w) - synth.AMPC * np.cos(w)


def _exact_gram(f, C):
    n = f.shape[0]
    f, C = f.reshape(n, -1), C.reshape(n, -1)
    M = (C * C) @ (f.real ** 2 + f.imag ** 2).t()
    Y = C * f
    D = M + M.t() - 2 * (Y.real @ Y.real.t() + Y.imag @ Y.imag.t())
    D.fill_diagonal_(0.0)
    return D


def _exact_distances(case, seed):
    b, ss = _batch(case, seed)
    out, off = [], 0
    for s in ss:
        n, N = len(s.ind), case["N"]
        sl = slice(off, off + n)
        img, C = _exact_images(s.raw, b.conj[sl], b.rot1[sl], b.rot2[sl], b.df[sl], N)
        out.append(_exact_gram(torch.fft.fft2(img), C).reshape(-1))
        off += n
    return torch.cat(out)


def _exact_particles(case, seed):
    st = prepare(case, seed)
    N = case["N"]
    h = N // 2 + 1
    img, C = _exact_images(st["stack"], st["conj"], st["rot1"], st["rot2"], st["df"], N)
    m, n = st["msk"].double(), img.shape[0]
    f = torch.fft.fft2(img * m)
    wien = -((C * C).sum(0) + 1.0 / 5)
    avg = torch.fft.ifft2(torch.fft.fft2(img) * (C / wien)).real.sum(0) * m / n
    # the phase-flipped images turn on the sign of the CTF at its zeros: no value there
    return dict(imgAll=img, fy=f[:, :, :h].contiguous(), ctf=C[:, :, :h].reshape(n, -1),
                imgAvg=avg, imgAllFlip=None, imgAvgFlip=None, imgAllIntensity=None,
                D=_exact_gram(f, C).reshape(-1))


def _tanh_fit(x, y):
    """Least squares fit of d + c tanh(a x + b) by Levenberg-Marquardt (numpy)."""
    lo, hi = y.min(), y.max()
    mid = x[np.argmin(np.abs(y - 0.5 * (lo + hi)))]
    slope = np.max(np.gradient(y, x)) / max(0.5 * (hi - lo), 1e-12)
    p = np.array([slope, -slope * mid, 0.5 * (hi - lo), 0.5 * (hi + lo)])
    lam, f = 1e-3, np.inf
    for _ in range(500):
        t = np.tanh(p[0] * x + p[1])
        r = y - (p[3] + p[2] * t)
        J = np.stack([p[2] * (1 - t * t) * x, p[2] * (1 - t * t), t, np.ones_like(x)], 1)
        A, g, f = J.T @ J, J.T @ r, r @ r
        while lam < 1e12:
            step = np.linalg.solve(A + lam * np.diag(np.diag(A)), g)
            q = p + step
            r2 = y - (q[3] + q[2] * np.tanh(q[0] * x + q[1]))
            if r2 @ r2 <= f:
                break
            lam *= 4
        if lam >= 1e12 or np.max(np.abs(step) / (np.abs(q) + 1e-12)) < 1e-13:
            break
        p, lam = q, max(lam / 8, 1e-12)
    return p


def _exact_embed_one(D, k, eigs, logEps):
    """Eigenvalues, coordinates, measure, bandwidth and log sums of one PD."""
    n = D.shape[0]
    D = D.double()
    key = D.clone()
    key.fill_diagonal_(-1.0)
    keep = torch.zeros(n, n, dtype=torch.bool, device=D.device)
    if k >= n:
        keep[:] = True
    else:
        keep.scatter_(1, torch.argsort(key, dim=1, stable=True)[:, :k], True)
    keep = keep | keep.t()
    vals = D[keep]
    le = np.asarray(logEps)
    dmax = vals / (2.0 * math.exp(le.max()))
    thr = max(float(-torch.log(0.01 * torch.exp(-dmax).sum() / vals.numel())), 10.0)
    S = []
    for e in le:
        d = vals / (2.0 * math.exp(e))
        S.append(torch.where(d < thr, torch.exp(-d), torch.zeros_like(d)).sum())
    logS = torch.log(torch.stack(S)).cpu().numpy()
    p = _tanh_fit(le, logS)
    sigma = 3 * math.sqrt(2 * math.exp(-p[1] / p[0]))
    W = torch.where(keep, torch.exp(-D / sigma ** 2), torch.zeros_like(D))
    d = W.sum(0)
    W = W / (d[:, None] * d[None, :])
    d = torch.sqrt(W.sum(0))
    W = W / (d[:, None] * d[None, :])
    lam, V = torch.linalg.eigh(0.5 * (W + W.t()))
    sel = torch.argsort(-lam.abs(), stable=True)[:min(eigs, n - 3) + 1]
    sel = sel[torch.argsort(lam[sel], descending=True, stable=True)]
    V = V[:, sel].cpu().numpy()
    return lam[sel].cpu().numpy(), V[:, 1:] / V[:, :1], V[:, 0] ** 2, sigma, logS


def _exact_embed(case, Ds, ks):
    logEps = _eps_grid(case["eps"])
    r = [_exact_embed_one(D, k, case["eigs"], logEps) for D, k in zip(Ds, ks)]
    return dict(lamb=np.concatenate([x[0] for x in r]), psi=_oriented([x[1] for x in r]),
                mu=np.concatenate([x[2] for x in r]), sigma=np.array([x[3] for x in r]),
                logSumWij=np.stack([x[4] for x in r]))


def _exact_nlsa(st):
    n, N, con, tr = (st["case"][k] for k in ("n", "N", "con", "trunc"))
    m = n - con
    DD = st["D"].double()[st["ord"]][:, st["ord"]]
    ConD = sum(DD[c:c + m, c:c + m] for c in range(con))
    C = st["ctf"].double()
    S = torch.cumsum(C * C, 0)
    W = S[con:n] - S[:m] + 1.0 / 5                       # sum of C_t^2, t = i + 1 .. i + con
    G = torch.fft.rfft2(st["img"].double()).reshape(n, -1) * C
    mu = st["mu_psi"]
    A = torch.empty((con, tr, N, N), dtype=torch.float64, device=C.device)
    for ii in range(con):
        g = G[con - 1 - ii:con - 1 - ii + m] / W
        f = torch.complex(mu.t().contiguous() @ g.real.contiguous(),
                          mu.t().contiguous() @ g.imag.contiguous())
        A[ii] = torch.fft.irfft2(f.view(tr, N, N // 2 + 1), s=(N, N))
    F = (st["U"] - st["U"].mean(0)) @ st["H"]
    inv_sd = 1.0 / torch.sqrt((F * F).mean(0))
    F = F * inv_sd
    q = (F * F).sum(0)
    D2 = q[:, None] + q[None, :] - 2 * (F.t().contiguous() @ F)
    return dict(ConD=ConD, A=A, D2=torch.where(D2 < 1e-8, torch.zeros_like(D2), D2),
                inv_sd=inv_sd, IMGT=F)


def _exact_flow(st):
    mov = st["movies"].double()
    m, F, N = st["case"]["movies"], st["case"]["frames"], st["case"]["N"]
    out = mov.clone()
    for _ in range(4):
        acc = torch.zeros_like(out)
        for ax, h in ((1, 5.0), (2, 3.0), (3, 3.0)):
            d = torch.diff(out, dim=ax)
            f = torch.exp(-(d / 50.0) ** 2) / h * d
            acc.narrow(ax, 0, d.shape[ax]).add_(f)
            acc.narrow(ax, 1, d.shape[ax]).sub_(f)
        out = out + 0.1 * acc
    A = -(-F // 5)
    fr = torch.stack([out[:, 5 * b:min(5 * b + 5, F)].mean(1) for b in range(A)], 1)
    w = torch.exp(-0.5 * (torch.arange(-8, 9, dtype=torch.float64, device=mov.device) / 2) ** 2)
    w = w / w.sum()
    idx = torch.arange(-8, N + 8, device=mov.device)
    idx = torch.remainder(idx, 2 * N)
    idx = torch.where(idx >= N, 2 * N - 1 - idx, idx)
    g = fr
    for ax in (2, 3):
        p = g.index_select(ax, idx)
        g = sum(w[k] * p.narrow(ax, k, N) for k in range(17))
    prev = torch.cat([g[:, :1], g[:, :-1]], 1)

    def pad(z):                      # half-sample reflection by one
        z = torch.cat([z[..., :1, :], z, z[..., -1:, :]], -2)
        return torch.cat([z[..., :1], z, z[..., -1:]], -1)

    def four(z):                     # the 2 x 2 block below and right of each pixel
        z = pad(z)[..., 1:, 1:]
        return z[..., :-1, :-1], z[..., :-1, 1:], z[..., 1:, :-1], z[..., 1:, 1:]

    a, b = four(prev), four(g)
    fx = 0.25 * sum(z[0] + z[2] - z[1] - z[3] for z in (a, b))
    fy = 0.25 * sum(z[0] + z[1] - z[2] - z[3] for z in (a, b))
    ft = 0.25 * (sum(a) - sum(b))
    den = 2.0 ** 2 + fx * fx + fy * fy

    def around(z):
        p = pad(z)
        return ((p[..., :-2, 1:-1] + p[..., 2:, 1:-1] + p[..., 1:-1, :-2] + p[..., 1:-1, 2:]) / 6
                + (p[..., :-2, :-2] + p[..., :-2, 2:] + p[..., 2:, :-2] + p[..., 2:, 2:]) / 12)

    U, V = torch.zeros_like(fx), torch.zeros_like(fx)
    for _ in range(200):
        ua, va = around(U), around(V)
        der = (fx * ua + fy * va + ft) / den
        U, V = ua - fx * der, va - fy * der
    Vx, Vy = U.sum(1), V.sum(1)
    # the orientations jump where the angle passes a multiple of 2: no value there
    return dict(Vx=Vx, Vy=Vy, Mag=torch.sqrt(Vx * Vx + Vy * Vy), Orient=None, Orient_rev=None)


def _exact_logsum(st):
    case = st["case"]
    n, N = case["n"], case["N"]
    h = N // 2 + 1
    X = st["fy"].detach().to(torch.complex128)
    C = torch.as_tensor(_exact_ctf(_radius(N, X.device).cpu().numpy()[:, :h] / (2 * synth.PIX),
                                  st["df"].cpu().numpy()), device=X.device)
    w = torch.full((h,), 2.0, dtype=torch.float64, device=X.device)
    w[0] = 1.0
    if N % 2 == 0:
        w[-1] = 1.0
    sw = torch.sqrt(w)
    Bm = (C * C).reshape(n, -1)
    Am = ((X.real ** 2 + X.imag ** 2) * w).reshape(n, -1)
    Y = C * X
    Yr, Yi = (Y.real * sw).reshape(n, -1), (Y.imag * sw).reshape(n, -1)
    M = Am @ Bm.t()
    D = M + M.t() - 2 * (Yr @ Yr.t() + Yi @ Yi.t())
    D.fill_diagonal_(0.0)
    eps = st["eps"].detach().double()
    L, g_eps = torch.zeros_like(eps), torch.zeros_like(eps)
    Wt = torch.zeros_like(D)
    for e in range(eps.numel()):
        K = torch.exp(-D / (2 * eps[e]))
        S = K.sum(1)
        L[e] = torch.log(S).sum()
        g_eps[e] = ((K * D).sum(1) / (2 * eps[e] ** 2 * S)).sum()
        Wt += -1.0 / (2 * eps[e]) * K * (1.0 / S[:, None] + 1.0 / S[None, :])
    WB = (Wt @ Bm).view_as(C)
    full = lambda z: (Wt @ z.reshape(n, -1)).view_as(C)
    gr = w * (X.real * WB - C * full(Y.real.contiguous()))
    gi = w * (X.imag * WB - C * full(Y.imag.contiguous()))
    return dict(L=L, g_fy=2.0 * torch.complex(gr, gi), g_eps=g_eps)


def exact(case, seed):
    kind = case["kind"]
    if kind == "distances":
        return _exact_distances(case, seed)
    if kind == "particles":
        return _exact_particles(case, seed)
    if kind == "embed":
        st = prepare(case, seed)
        Ds = [st["plan"].block(st["D"], p).view(int(n), int(n))
              for p, n in enumerate(st["plan"].ns)]
        return _exact_embed(case, Ds, [int(k) for k in st["plan"].ks])
    if kind == "nlsa":
        return _exact_nlsa(prepare(case, seed))
    if kind == "flow":
        return _exact_flow(prepare(case, seed))
    if kind == "logsum":
        return _exact_logsum(prepare(case, seed))
    return None
