"""The workloads whose speed is measured, through the package's entry points.

    listed()             the cases, plain dicts
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  the model on the GPU, run parameters, k-points
    run(state)           one pass; returns the outputs
    work(case)           bytes and flops one pass cannot do without
    exact(case, seed)    the outputs in 64 bits by plain numpy / torch

Kinds of case:
    interp   ``Engine.interp`` (get_wann_interp): eigenvalues, and with
             ``velo`` the velocities (and, with a position operator, the
             connection and curvature) of a k list, back on the host
    mesh     ``Engine.run_mesh``: the k-loop over a Monkhorst-Pack mesh
    list     ``Engine.run_kpts``: the k-loop over a weighted k list
    batch    ``run_batch``: several models' meshes in one call
    network  the learned part of an adaptive refinement: train the network
             on the coarse mesh, score every cell

Models are seeded random Wannier models (complex hoppings decaying with |R|,
Hermitian), energies of a few eV; ``pos`` adds the position operator r(R),
``tb`` the Wannier centres (tight-binding convention).  ``jobs`` names the
band sums: ahc (Hall and optical conductivity from velocities), kubo and mep
(magneto-electric polarisability, Kubo and Niu), opt (optical tensors and
second-order photoconductivity, with r(R)), gyro (gyrotropic tensors).
"""
from __future__ import annotations

import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

from mepinterp_amd import capi, models, refine

AU_TO_EV = 27.211385
KB_HARTREE = 8.6173303e-5 / AU_TO_EV
KUBO_TOL = 1e-5
TWO_PI = 2.0 * math.pi
JOB_SUMS = {"ahc": ("ahc", "ahc_velo", "ohc"), "kubo": ("kubo_ic", "kubo_lc", "kubo_cs"),
            "mep": ("niu_ic", "niu_lc", "niu_cs"), "opt": ("opt_s", "opt_a", "photo"),
            "gyro": ("gyro_C", "gyro_D", "gyro_Dw")}
JOB_BITS = {"ahc": capi.MEP_JOB_AHC, "kubo": capi.MEP_JOB_KUBO, "mep": capi.MEP_JOB_MEP,
            "opt": capi.MEP_JOB_OPT, "gyro": capi.MEP_JOB_GYRO}


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def _mesh(name, n, L, grid, jobs, pos=False, tb=False, n_eF=1, n_hw=1, T=300.0, eta_eV=0.05):
    return dict(name=name, kind="mesh", n=n, L=L, n1=grid[0], n2=grid[1], n3=grid[2], jobs=jobs,
                pos=pos, tb=tb, n_eF=n_eF, n_hw=n_hw, T=T, eta_eV=eta_eV)


def listed():
    return [
        # one k-point through get_wann_interp, as the per-k procedures of the
        # reference's hosts call it: latency
        dict(name="point", kind="interp", n=8, L=1, nk=1, pos=True, tb=False, velo=True),
        # a band-structure path: eigenvalues of a few hundred k-points
        dict(name="bands", kind="interp", n=24, L=2, nk=401, pos=False, tb=True, velo=False),
        # sigma_xy of a small model with a position operator
        _mesh("hall_pos", 8, 1, (32, 32, 32), "ahc", pos=True, eta_eV=1e-3),
        # every response tensor of a mid-size model read from a _tb.dat file
        _mesh("mep_pos", 24, 1, (16, 16, 16), "ahc+kubo+mep", pos=True, tb=True, n_eF=3),
        # optical and gyrotropic spectra with the position operator
        _mesh("optics", 14, 1, (15, 14, 13), "ahc+opt+gyro", pos=True, n_eF=2, n_hw=8),
        # the benchmark's workload: AHC, Kubo and Niu MEP of a 32-band magnet
        _mesh("mep", 32, 3, (64, 64, 64), "ahc+kubo+mep", eta_eV=1e-3),
        # Fermi-level and frequency scan, tight-binding convention, ragged mesh
        _mesh("scan", 20, 2, (31, 29, 27), "ahc+kubo+mep", tb=True, n_eF=5, n_hw=16),
        # weighted k list of an adaptive refinement, T = 0
        dict(name="refined", kind="list", n=24, L=3, nk=60000, jobs="ahc", pos=False, tb=False,
             n_eF=1, n_hw=1, T=0.0, eta_eV=0.0),
        # a wide model (above 32 bands), no multiple of a matrix tile
        _mesh("wide", 44, 2, (21, 21, 21), "ahc+kubo+mep", eta_eV=1e-3),
        # a large supercell's optical conductivity on 256 frequencies and MEP
        _mesh("spectrum", 96, 2, (14, 14, 14), "ahc+kubo+mep", n_hw=256),
        # several models of a screening set in one call
        dict(name="batch", kind="batch", sizes="8,20,36,52", L=1, q=14, jobs="ahc+kubo+mep",
             pos=False, tb=False, n_eF=1, n_hw=1, T=300.0, eta_eV=1e-3),
        # network of an adaptive refinement on a 16^3 mesh (one batch an epoch)
        dict(name="network", kind="network", n1=16, n2=16, n3=16, n_freq=4, hidden=128, epochs=30),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, nk):
    """Three mesh divisions with about nk points, seldom a cube."""
    q = nk ** (1.0 / 3.0)
    a = max(1, int(round(q * rng.uniform(0.8, 1.25))))
    b = max(1, int(round(q * rng.uniform(0.8, 1.25))))
    return a, b, max(1, nk // (a * b))


def draw(rng):
    kind = rng.choice(["interp", "mesh", "mesh", "mesh_pos", "mesh_pos", "list", "batch",
                       "network"])
    if kind == "interp":
        pos = rng.random() < 0.4
        n = _log_int(rng, 4, 24) if pos else _log_int(rng, 4, 64)
        velo = pos or rng.random() < 0.5
        cap = min(2000.0, 4e6 / (n * n)) if velo else 2000.0
        return dict(kind="interp", n=n, L=rng.choice([1, 2]), nk=_log_int(rng, 1, cap), pos=pos,
                    tb=rng.random() < 0.5, velo=velo)
    T = rng.choice([0.0, 100.0, 300.0])
    eta = rng.choice([1e-3, 0.01, 0.05])
    if kind == "mesh":
        n = _log_int(rng, 4, 96)
        jobs = rng.choice(["ahc", "ahc+kubo+mep", "ahc+kubo+mep", "kubo", "ahc+gyro"])
        n_eF, n_hw = rng.choice([(1, 1), (1, 1), (1, 64), (5, 1), (3, 8), (1, 256)])
        if n_hw > 64 and n <= 32:
            n_hw = 64
        L = rng.choice([1, 2, 3]) if n <= 40 else rng.choice([1, 2])
        cap = min(110592.0, 1.0e9 / n ** 3, 2.5e9 / (n * n * n_eF * n_hw))
        g = _grid(rng, _log_int(rng, 64, max(64.0, cap)))
        c = _mesh("", n, L, g, jobs, tb=rng.random() < 0.4, n_eF=n_eF, n_hw=n_hw, T=T, eta_eV=eta)
        del c["name"]
        return c
    if kind == "mesh_pos":
        n = _log_int(rng, 4, 40)
        jobs = rng.choice(["ahc", "ahc+kubo+mep", "ahc+opt+gyro", "ahc+opt"])
        n_eF, n_hw = rng.choice([(1, 1), (1, 1), (3, 1), (2, 8)])
        cap = min(32768.0, 2.5e7 / n ** 3)
        g = _grid(rng, _log_int(rng, 64, max(64.0, cap)))
        c = _mesh("", n, 1, g, jobs, pos=True, tb=rng.random() < 0.5, n_eF=n_eF, n_hw=n_hw,
                  T=T, eta_eV=eta)
        del c["name"]
        return c
    if kind == "list":
        n = _log_int(rng, 6, 48)
        cap = min(60000.0, 5e8 / n ** 3)
        return dict(kind="list", n=n, L=rng.choice([1, 2, 3]), nk=_log_int(rng, 100, cap),
                    jobs=rng.choice(["ahc", "ahc+kubo+mep"]), pos=False, tb=rng.random() < 0.4,
                    n_eF=1, n_hw=1, T=T, eta_eV=eta)
    if kind == "batch":
        sizes = ",".join(str(_log_int(rng, 6, 60)) for _ in range(rng.randint(2, 4)))
        return dict(kind="batch", sizes=sizes, L=rng.choice([1, 2]), q=rng.randint(4, 13),
                    jobs="ahc+kubo+mep", pos=False, tb=rng.random() < 0.4, n_eF=1, n_hw=1, T=T,
                    eta_eV=eta)
    n1, n2, n3 = _grid(rng, _log_int(rng, 200, 4000))
    return dict(kind="network", n1=n1, n2=n2, n3=n3, n_freq=rng.choice([3, 4]),
                hidden=rng.choice([64, 128]), epochs=rng.randint(5, 30))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _model(case, seed, n):
    m = models.make_random(seed=1000003 * n + seed, n=n, L=case["L"], decay=1.0 + 0.25 * case["L"],
                           with_r=case["pos"], tb=case["tb"])
    return m


def _fermi(case):
    """Fermi levels around the middle of the spectrum, frequencies up to 5 eV
    (opt divides by the frequency: from 0.1 eV there)."""
    lo = 0.1 if "opt" in case["jobs"] else 0.0
    return dict(n_eF=case["n_eF"], eF_min=-0.01 if case["n_eF"] > 1 else 0.0,
                eF_max=0.01 if case["n_eF"] > 1 else 0.0, n_hw=case["n_hw"],
                hw_min=lo / AU_TO_EV, hw_max=(5.0 if case["n_hw"] > 1 else lo) / AU_TO_EV,
                T_kelvin=case["T"], eta=case["eta_eV"] / AU_TO_EV)


def _params(case, n):
    bits = 0
    for j in case["jobs"].split("+"):
        bits |= JOB_BITS[j]
    return capi.Engine.params(jobs=bits, valence_bands=max(1, n // 2), **_fermi(case))


def _mesh_points(mp):
    """The Monkhorst-Pack points (2 q - N - 1) / (2 N), x fastest, (3, N)."""
    ax = [(2.0 * np.arange(1, m + 1) - m - 1) / (2.0 * m) for m in mp]
    z, y, x = np.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    return np.asfortranarray(np.stack([x.ravel(), y.ravel(), z.ravel()]))


def _kpath(seed, nk):
    """A path through random special points, evenly spaced on each leg."""
    r = np.random.default_rng(seed + 77)
    legs = max(1, nk // 100)
    pts = r.integers(-4, 5, size=(3, legs + 1)) / 8.0 + r.uniform(-0.01, 0.01, size=(3, legs + 1))
    t = np.linspace(0.0, legs, nk) if nk > 1 else np.array([0.37])
    i = np.minimum(t.astype(int), legs - 1)
    f = t - i
    return np.asfortranarray(pts[:, i] * (1.0 - f) + pts[:, i + 1] * f)


def _klist(seed, nk):
    r = np.random.default_rng(seed + 99)
    k = np.asfortranarray(r.uniform(-0.5, 0.5, size=(3, nk)))
    w = np.where(r.random(nk) < 0.4, 1.0, r.uniform(0.0, 1.0 / 64.0, size=nk))
    return k, w


def _target(seed, k):
    """log curvature of a few planted hot spots over a smooth background."""
    r = np.random.default_rng(seed + 55)
    c = r.uniform(-0.5, 0.5, size=(3, 6))
    t = np.zeros(k.shape[1])
    for i in range(6):
        d2 = np.sum(np.sin(math.pi * (k - c[:, i:i + 1])) ** 2, axis=0)
        t += r.uniform(0.5, 2.0) / (d2 + 0.02)
    return np.log(t + 1e-3).astype(np.float32)


def _net_start(case, seed):
    """Starting weights in the network's flat layout (padding stays zero)."""
    r = np.random.default_rng(seed + 33)
    nf, h = case["n_freq"], case["hidden"]
    fp = ((6 * nf + 15) // 16) * 16
    w1 = np.zeros((fp, h))
    w1[:6 * nf] = r.uniform(-1, 1, size=(6 * nf, h)) * math.sqrt(6.0 / (6 * nf + h))
    w2, w3 = (r.uniform(-1, 1, size=(h, h)) * math.sqrt(3.0 / h) for _ in range(2))
    w4 = np.zeros((h, 16))
    w4[:, 0] = r.uniform(-1, 1, size=h) * math.sqrt(6.0 / (h + 1))
    z = np.zeros(h)
    return np.concatenate([x.ravel() for x in (w1, z, w2, z, w3, z, w4, np.zeros(16))]).astype(
        np.float32)


def _engine(m):
    return capi.Engine(m["R_frac"], m["H"], r=m["r"], wf_centers=m["wf_centers"],
                       a_latt=m["a_latt"], kubo_tol=KUBO_TOL)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "network":
        mp = (case["n1"], case["n2"], case["n3"])
        k = _mesh_points(mp)
        return dict(kind=kind, mp=mp, k=k, t=_target(seed, k), p0=_net_start(case, seed),
                    n_freq=case["n_freq"], hidden=case["hidden"], epochs=case["epochs"])
    if kind == "batch":
        sizes = [int(x) for x in case["sizes"].split(",")]
        eng = [_engine(_model(case, seed + i, n)) for i, n in enumerate(sizes)]
        for e in eng:
            e.set_workspace_limit(16e9)
        grids = [(case["q"], case["q"] + i, case["q"] + 1) for i in range(len(sizes))]
        return dict(kind=kind, eng=eng, grids=grids, jobs=case["jobs"],
                    p=[_params(case, n) for n in sizes])
    eng = _engine(_model(case, seed, case["n"]))
    if kind == "interp":
        return dict(kind=kind, eng=eng, k=_kpath(seed, case["nk"]), velo=case["velo"])
    p = _params(case, case["n"])
    if kind == "list":
        k, w = _klist(seed, case["nk"])
        return dict(kind=kind, eng=eng, k=k, w=w, jobs=case["jobs"], p=p)
    return dict(kind=kind, eng=eng, grid=(case["n1"], case["n2"], case["n3"]),
                jobs=case["jobs"], p=p)


def _asked(sums, jobs):
    """The sums of the jobs asked for (run_mesh leaves the others zero)."""
    return {key: sums[key] for j in jobs.split("+") for key in JOB_SUMS[j]} | {
        "Ne": sums["Ne"], "n_k": sums["n_k"]}


def run(state):
    kind = state["kind"]
    if kind == "interp":
        return state["eng"].interp(state["k"], velo=state["velo"])
    if kind == "mesh":
        return _asked(state["eng"].run_mesh(state["grid"], state["p"]), state["jobs"])
    if kind == "list":
        return _asked(state["eng"].run_kpts(state["k"], state["p"], weights=state["w"]),
                      state["jobs"])
    if kind == "batch":
        return [_asked(o, state["jobs"])
                for o in capi.run_batch(state["eng"], state["grids"], state["p"])]
    # as refine.refine_sigma does, from weights the caller has
    with capi.MLP(n_freq=state["n_freq"], hidden=state["hidden"]) as net:
        net.params = state["p0"]
        loss = net.train(state["k"], state["t"], epochs=state["epochs"], batch=4096, lr=2e-3)
        score = refine.cell_scores(net, state["k"], state["mp"])
        return dict(loss=loss, params=net.params, score=score)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _job_flops(case, n):
    jobs = case["jobs"].split("+")
    f = 48.0 * n ** 3                              # U^H dH U, three components
    if "kubo" in jobs or "mep" in jobs:
        f += 48.0 * n ** 3                         # itinerant terms: six products
    if "ahc" in jobs:
        f += 24.0 * n * (n - 1) * case["n_hw"] * case["n_eF"]
    if "opt" in jobs:                              # nine products, frequency sums
        f += 72.0 * n ** 3 + 8.0 * 45.0 * n * n * case["n_hw"] * case["n_eF"]
    return f


def _pipeline(case, n, nk, mesh, jobs=True, velo=True):
    """(bytes, flops) of nk k-points of an n-band model."""
    nr = (2 * case["L"] + 1) ** 3
    nmat = (10 if case["pos"] else 4) if velo else 1
    el = nmat * (n * n if case["pos"] else n * (n + 1) // 2)
    model = 16.0 * n * n * nr * (4 if case["pos"] else 1)
    ft = 8.0 * (2 * case["L"] + 1) * el if mesh else 4.0 * nr * el
    fl = ft + (16.0 / 3.0 + (8.0 if velo else 0.0)) * n ** 3
    if velo and case["pos"]:
        fl += 8.0 * n ** 3 * (3 * 2 + 3 * 2 + 3 * 6)  # A, Omega rotations, commutators
    if jobs:
        fl += _job_flops(case, n)
    elif velo:
        fl += 48.0 * n ** 3
    return model + (0.0 if mesh else 32.0 * nk), fl * nk


def work(case):
    kind = case["kind"]
    if kind == "network":
        nk, h, fp = case["n1"] * case["n2"] * case["n3"], case["hidden"], 6 * case["n_freq"]
        par = fp * h + 2 * h * h + 4 * h + 1
        mm = 2.0 * (fp * h + 2 * h * h + h)
        return dict(bytes=32.0 * nk * 10 + 8.0 * par, flops=nk * mm * (3.0 * case["epochs"] + 9.0))
    if kind == "batch":
        b = f = 0.0
        for i, n in enumerate(int(x) for x in case["sizes"].split(",")):
            bi, fi = _pipeline(case, n, case["q"] * (case["q"] + i) * (case["q"] + 1), True)
            b, f = b + bi, f + fi
        return dict(bytes=b, flops=f)
    n = case["n"]
    if kind == "interp":
        b, f = _pipeline(case, n, case["nk"], False, jobs=False, velo=case["velo"])
        out = 8.0 * n + (16.0 * n * n * (15 if case["pos"] else 3) if case["velo"] else 0.0)
        return dict(bytes=b + out * case["nk"], flops=f)
    nk = case["nk"] if kind == "list" else case["n1"] * case["n2"] * case["n3"]
    b, f = _pipeline(case, n, nk, kind == "mesh")
    return dict(bytes=b, flops=f)


# ---------------------------------------------------------------------------
# the same outputs in 64 bits, by plain numpy / torch
# ---------------------------------------------------------------------------
DEV = "cuda" if torch.cuda.is_available() else "cpu"
LEVI = [(0, 1, 2, 1.0), (1, 2, 0, 1.0), (2, 0, 1, 1.0), (0, 2, 1, -1.0), (2, 1, 0, -1.0),
        (1, 0, 2, -1.0)]


def _eigh(H):
    """Eigenvalues and eigenvectors of a stack of Hermitian matrices; each
    vector's largest-modulus component is real and positive."""
    H = H.cpu().numpy()
    part = [H[i:i + 512] for i in range(0, H.shape[0], 512)]
    with ThreadPoolExecutor(16) as ex:
        res = list(ex.map(lambda h: np.linalg.eigh(h, UPLO="U"), part))
    e = torch.from_numpy(np.concatenate([r[0] for r in res])).to(DEV)
    U = torch.from_numpy(np.concatenate([r[1] for r in res])).to(DEV)
    im = (U.real ** 2 + U.imag ** 2).argmax(dim=1, keepdim=True)
    top = torch.gather(U, 1, im)
    return e, U * (top.conj() / top.abs())


def _interp64(m, k, velo=True):
    """e (k,n), V (k,3,n,n), A (k,3,n,n), Om (k,3,3,n,n) of k-points (3,nk),
    in the reference's order of operations with a position operator."""
    n = m["H"].shape[0]
    R = torch.from_numpy(np.ascontiguousarray(m["R_frac"].T)).to(DEV)   # (nR, 3)
    kk = torch.from_numpy(np.ascontiguousarray(np.asarray(k).T)).to(DEV)
    ph = torch.polar(torch.ones((), dtype=torch.float64, device=DEV), TWO_PI * (kk @ R.T))

    def ft(X):  # X (nR, n, n)
        return (ph @ X.reshape(X.shape[0], n * n)).reshape(-1, n, n)

    X = torch.from_numpy(np.ascontiguousarray(np.moveaxis(m["H"], 2, 0))).to(DEV)
    c = [(TWO_PI * R[:, a])[:, None, None] for a in range(3)]
    H = ft(X)
    dH = [1j * ft(c[a] * X) for a in range(3)] if velo else []
    pos = velo and m["r"] is not None
    if pos:
        r = [torch.from_numpy(np.ascontiguousarray(np.moveaxis(m["r"][a], 2, 0))).to(DEV)
             for a in range(3)]
        A = [ft(r[a]) for a in range(3)]
        B = {(a, b): ft(c[a] * r[b]) for a in range(3) for b in range(3)}
    if m["wf_centers"] is not None:
        tau = torch.from_numpy(np.ascontiguousarray(m["wf_centers"])).to(DEV)
        d = tau[:, None, :] - tau[:, :, None]           # d[a, n, m] = tau_m - tau_n
        g = torch.einsum("ka,anm->knm", kk, d)
        tbp = torch.polar(torch.ones_like(g), TWO_PI * g)
        dH = [tbp * (dH[a] + 1j * TWO_PI * d[a] * H) for a in range(3)] if velo else []
        H = tbp * H
        if pos:
            B = {(a, b): tbp * (B[a, b] + TWO_PI * d[a] * A[b]) for a in range(3) for b in range(3)}
            A = [tbp * A[a] for a in range(3)]
    e, U = _eigh(H)
    if not velo:
        return e, None, None, None
    Ud = U.conj().transpose(1, 2).contiguous()
    T = [dH[a] @ U for a in range(3)]
    V = [Ud @ T[a] for a in range(3)]
    if not pos:
        return e, torch.stack(V, 1), None, None
    dE = e[:, None, :] - e[:, :, None]                  # dE[n, m] = e_m - e_n
    inv = torch.where(dE.abs() > KUBO_TOL, 1.0 / dE, torch.zeros_like(dE))
    inv.diagonal(dim1=1, dim2=2).zero_()
    D = [V[a] * inv for a in range(3)]
    AH = [V[a] @ U + 1j * D[a] for a in range(3)]       # A^(H) from the stale product

    def com(x, y):
        return x @ y - y @ x

    Om = []
    for a in range(3):
        row = []
        for b in range(3):
            w = Ud @ (1j * (B[a, b] - B[b, a])) @ U
            row.append(w - com(D[a], AH[b]) + com(D[b], AH[a]) - 1j * com(D[a], D[b]))
        Om.append(torch.stack(row, 1))
    # V_nm = Hbar_nm - i (e_m - e_n) A_nm, Hbar_nn on the diagonal (dE_nn = 0)
    VH = [V[a] - 1j * dE * AH[a] for a in range(3)]
    return e, torch.stack(VH, 1), torch.stack(AH, 1), torch.stack(Om, 1)


def _occ(e, case):
    p = _fermi(case)
    ef = np.linspace(p["eF_min"], p["eF_max"], p["n_eF"])
    x = e[:, :, None] - torch.from_numpy(ef).to(DEV)
    if p["T_kelvin"] > 1e-2:
        return 1.0 / (1.0 + torch.exp(x / (KB_HARTREE * p["T_kelvin"])))
    return (x < 0).double()


def _sums64(case, n, e, V, A, Om, w):
    """The band sums of the k-points, weighted by w, as run_mesh lays them
    out: the last axes of every tensor are (n_hw,) n_eF or the bands."""
    p = _fermi(case)
    jobs = case["jobs"].split("+")
    eta, nef, nhw, nv = p["eta"], p["n_eF"], p["n_hw"], max(1, n // 2)
    hw = np.linspace(p["hw_min"], p["hw_max"], nhw)
    f = _occ(e, case)                                     # (k, n, ef)
    eye = torch.eye(n, device=DEV).bool()
    dE = e[:, None, :] - e[:, :, None]                    # e_m - e_n at [n, m]
    dE1 = dE.masked_fill(eye, 1.0)
    inv = (1.0 / dE1).masked_fill(eye, 0.0)
    wf = w[:, None, None] * f
    cz = torch.complex128
    o = {"Ne": wf.sum((0, 1))}
    Vt = V.transpose(2, 3)
    P = V[:, :, None] * Vt[:, None]                       # V_i[n,m] V_j[m,n]
    if "ahc" in jobs:
        cv = 2.0 * (P.imag * (inv ** 2)[:, None, None]).sum(-1)
        o["ahc"] = torch.einsum("kijn,kne->ije", cv, wf)
        va = torch.zeros(3, 3, nhw, nef, dtype=cz, device=DEV)
        oh = torch.zeros_like(va)
        Pm = P.reshape(P.shape[0], 9, n * n).transpose(0, 1).reshape(9, -1)
        for s in range(nef):
            df = ((f[:, :, None, s] - f[:, None, :, s]) * w[:, None, None]).masked_fill(eye, 0.0)
            for h in range(nhw):
                z = hw[h] + 1j * eta
                g1 = (df / (dE1 ** 2 - z * z)).reshape(-1)
                g2 = (-1j * df / (dE1 * (dE1 - z))).reshape(-1)
                va[:, :, h, s] = (Pm.imag.to(cz) @ g1).reshape(3, 3)
                oh[:, :, h, s] = (Pm @ g2).reshape(3, 3)
        o["ahc_velo"], o["ohc"] = va, oh
    if "kubo" in jobs or "mep" in jobs:
        B = V * (-inv).transpose(1, 2)[:, None]           # V_l[m,n0] / (e_n0 - e_m)
        A2 = V * (inv ** 2)[:, None]                      # V_i[n0,n] / (e_n0 - e_n)^2
        A3 = A2 * (-inv)[:, None]
        vd = V.diagonal(dim1=2, dim2=3)                   # V_l[n0,n0]

        def contract(Cs, X, Y, keep):
            """ic[k,i,j,n0], lc[k,i,j,n0]; Cs[a,b][k,n,n0] = sum_m V_a B_b"""
            ic = torch.zeros(V.shape[0], 3, 3, n, dtype=torch.float64, device=DEV)
            lc = torch.zeros_like(ic)
            for j, a, b, sg in LEVI:
                for i in range(3):
                    ic[:, i, j] -= sg * (X[:, i] * Cs[a, b].transpose(1, 2)).sum(-1).real
                    lc[:, i, j] += sg * ((Y[:, i] * keep * Vt[:, a]).sum(-1) * vd[:, b]).real
            return ic, lc
        if "kubo" in jobs:
            Cs = {(a, b): V[:, a] @ B[:, b] for _, a, b, _ in LEVI}
            ic, lc = contract(Cs, A2, A3, torch.ones_like(inv))
            o["kubo_ic"] = torch.einsum("kijn,kne->ije", ic, wf)
            o["kubo_lc"] = torch.einsum("kijn,kne->ije", lc, wf)
        if "mep" in jobs:
            d = -dE                                       # d[n0, n] = e_n0 - e_n
            Cs = {(a, b): torch.zeros_like(V[:, 0]) for _, a, b, _ in LEVI}
            for n0 in range(nv):
                ok = ((d[:, n0, :, None] ** 2 * d[:, n0, None, :]).abs() > KUBO_TOL)
                for a, b in Cs:
                    Cs[a, b][:, :, n0] = ((V[:, a] * ok) @ B[:, b, :, n0, None])[..., 0]
            keep = ((d * d * d).abs() > KUBO_TOL).double()
            ic, lc = contract(Cs, A2, A3, keep)
            o["niu_ic"] = torch.einsum("kijn,k->ijn", ic[..., :nv], w)
            o["niu_lc"] = torch.einsum("kijn,k->ijn", lc[..., :nv], w)
        if A is not None:
            cs = torch.zeros(V.shape[0], n, dtype=torch.float64, device=DEV)
            for c, a, b, sg in LEVI:
                cs += 0.5 * sg * (A[:, c].diagonal(dim1=1, dim2=2).conj() *
                                  Om[:, a, b].diagonal(dim1=1, dim2=2)).real
            one = torch.eye(3, dtype=torch.float64, device=DEV)[:, :, None]
            if "kubo" in jobs:
                o["kubo_cs"] = one * torch.einsum("kn,kne->e", cs, wf)
            if "mep" in jobs:
                o["niu_cs"] = one * torch.einsum("kn,k->n", cs[:, :nv], w)
    if "opt" in jobs:
        ph = torch.zeros(3, 3, 3, nhw, nef, dtype=cz, device=DEV)
        os_ = torch.zeros(3, 3, nhw, nef, dtype=cz, device=DEV)
        oa = torch.zeros_like(os_)
        den = -dE - 1j * eta                              # [n, m]: e_n - e_m - i eta
        Q = {(b, c): V[:, b] @ (V[:, c] / den.transpose(1, 2)) for b in range(3) for c in range(3)}
        G = torch.stack([V[:, a] * Q[b, c].transpose(1, 2) for a in range(3) for b in range(3)
                         for c in range(3)], 0).reshape(27, -1)
        PA = None
        if A is not None:
            PA = (dE[:, None, None] * A[:, :, None] * A.transpose(2, 3)[:, None])
            PA = PA.reshape(PA.shape[0], 9, n * n).transpose(0, 1).reshape(9, -1)
        for s in range(nef):
            df = ((f[:, None, :, s] - f[:, :, None, s]) * w[:, None, None]).masked_fill(eye, 0.0)
            for h in range(nhw):
                g = sum(1.0 / (den + sg * hw[h] - 1j * eta) for sg in (-1.0, 1.0))
                ph[..., h, s] = (G @ (g * df / hw[h] ** 2).reshape(-1)).reshape(3, 3, 3)
                if PA is not None:
                    db = (1.0 / (math.pi * (dE - 1j * eta) - math.pi * hw[h])).imag
                    he = -(PA @ (math.pi * db * df).reshape(-1).to(cz)).reshape(3, 3)
                    ah = 1j * (PA @ (df / (dE - hw[h])).reshape(-1).to(cz)).reshape(3, 3)
                    os_[..., h, s] = torch.complex(he.real, ah.imag)
                    oa[..., h, s] = torch.complex(ah.real, he.imag)
        o["photo"], o["opt_s"], o["opt_a"] = ph, os_, oa
    if "gyro" in jobs:
        fdd = w[:, None, None] / (2.0 + 2.0 * torch.cosh(f))
        vd = V.diagonal(dim1=2, dim2=3)
        o["gyro_C"] = torch.einsum("kabn,kne->abe", vd[:, :, None] * vd[:, None], fdd.to(cz))
        if Om is not None:
            cur = Om.diagonal(dim1=3, dim2=4)
        else:
            big = (dE ** 2 >= KUBO_TOL).double() * inv ** 2
            cur = (-2.0 * (P.imag * big[:, None, None]).sum(-1)).to(cz)
        om = torch.zeros(V.shape[0], 3, n, dtype=cz, device=DEV)
        for c, a, b, sg in LEVI:
            om[:, c] += sg * cur[:, a, b]
        o["gyro_D"] = -torch.einsum("kabn,kne->abe", vd[:, :, None] * om[:, None], fdd.to(cz))
        dw = torch.zeros(3, 3, nhw, nef, dtype=cz, device=DEV)
        if A is not None:
            ww = dE ** 2
            At = A.transpose(2, 3)
            for h in range(nhw):
                g = (ww / (ww - hw[h])).masked_fill(eye, 0.0)
                for c, a, b in ((0, 1, 2), (1, 2, 0), (2, 0, 1)):
                    t = -((A[:, a] * At[:, b] - A[:, b] * At[:, a]).imag * g).sum(-1)
                    dw[:, c, h] = -torch.einsum("kan,kne->ae", vd * t[:, None], fdd.to(cz))
        o["gyro_Dw"] = dw
    return o


def _run64(case, seed, n, k, w):
    m = _model(case, seed, n)
    nef, nhw, nv = case["n_eF"], case["n_hw"], max(1, n // 2)
    z = {key: np.zeros(shape, np.complex128 if cx else np.float64) for key, shape, cx in (
        ("Ne", (nef,), 0), ("ahc", (3, 3, nef), 0), ("ahc_velo", (3, 3, nhw, nef), 1),
        ("ohc", (3, 3, nhw, nef), 1), ("kubo_ic", (3, 3, nef), 0), ("kubo_lc", (3, 3, nef), 0),
        ("kubo_cs", (3, 3, nef), 0), ("niu_ic", (3, 3, nv), 0), ("niu_lc", (3, 3, nv), 0),
        ("niu_cs", (3, 3, nv), 0), ("opt_s", (3, 3, nhw, nef), 1), ("opt_a", (3, 3, nhw, nef), 1),
        ("photo", (3, 3, 3, nhw, nef), 1), ("gyro_C", (3, 3, nef), 1), ("gyro_D", (3, 3, nef), 1),
        ("gyro_Dw", (3, 3, nhw, nef), 1))}
    step = max(64, min(16384, int(2.0e7 / (n * n))))
    for i in range(0, k.shape[1], step):
        e, V, A, Om = _interp64(m, k[:, i:i + step])
        wi = torch.from_numpy(np.ascontiguousarray(w[i:i + step])).to(DEV)
        for key, val in _sums64(case, n, e, V, A, Om, wi).items():
            z[key] += val.cpu().numpy()
    z["n_k"] = k.shape[1]
    return _asked(z, case["jobs"])


def _network64(case, seed):
    mp = (case["n1"], case["n2"], case["n3"])
    k = _mesh_points(mp)
    nf, h = case["n_freq"], case["hidden"]
    fp = ((6 * nf + 15) // 16) * 16
    shapes = [(fp, h), (h,), (h, h), (h,), (h, h), (h,), (h, 16), (16,)]
    p, o = [], 0
    flat = torch.from_numpy(_net_start(case, seed)).double().to(DEV)
    for s in shapes:
        c = math.prod(s)
        p.append(flat[o:o + c].reshape(s).clone())
        o += c

    def feat(kk):
        kk = torch.from_numpy(np.ascontiguousarray(kk)).to(DEV)
        x = torch.zeros(kk.shape[1], fp, dtype=torch.float64, device=DEV)
        for a in range(3):
            for q in range(nf):
                x[:, a * 2 * nf + 2 * q] = torch.sin(TWO_PI * (q + 1) * kk[a])
                x[:, a * 2 * nf + 2 * q + 1] = torch.cos(TWO_PI * (q + 1) * kk[a])
        return x

    def fwd(x):
        hs = [x]
        for q in range(3):
            hs.append(torch.tanh(hs[-1] @ p[2 * q] + p[2 * q + 1]))
        return hs, hs[-1] @ p[6] + p[7]

    x, t = feat(k), torch.from_numpy(_target(seed, k)).double().to(DEV)
    mom = [torch.zeros_like(q) for q in p]
    var = [torch.zeros_like(q) for q in p]
    lr = float(np.float32(2e-3))
    b1, b2, eps = float(np.float32(0.9)), float(np.float32(0.999)), float(np.float32(1e-8))
    loss = 0.0
    for ep in range(1, case["epochs"] + 1):
        hs, y = fwd(x)
        err = y[:, 0] - t
        loss = float((err * err).mean())
        dz = torch.zeros_like(y)
        dz[:, 0] = 2.0 * err / t.numel()
        g = [None] * 8
        for q in (3, 2, 1, 0):
            g[2 * q], g[2 * q + 1] = hs[q].T @ dz, dz.sum(0)
            if q:
                dz = (dz @ p[2 * q].T) * (1.0 - hs[q] ** 2)
        for q in range(8):
            mom[q] = b1 * mom[q] + (1.0 - b1) * g[q]
            var[q] = b2 * var[q] + (1.0 - b2) * g[q] ** 2
            p[q] = p[q] - lr * (mom[q] / (1.0 - b1 ** ep)) / (
                torch.sqrt(var[q] / (1.0 - b2 ** ep)) + eps)
    off = np.array(np.meshgrid([-1, 1], [-1, 1], [-1, 1])).reshape(3, -1).T
    hh = np.asarray(mp, dtype=np.float64).reshape(3, 1)
    pts = [k] + [k + s.reshape(3, 1) / (4.0 * hh) for s in off]
    score = torch.stack([fwd(feat(q))[1][:, 0] for q in pts]).max(0).values
    return dict(loss=loss, params=torch.cat([q.reshape(-1) for q in p]).cpu().numpy(),
                score=score.cpu().numpy())


def exact(case, seed):
    kind = case["kind"]
    if kind == "network":
        return _network64(case, seed)
    if kind == "batch":
        out = []
        for i, n in enumerate(int(x) for x in case["sizes"].split(",")):
            k = _mesh_points((case["q"], case["q"] + i, case["q"] + 1))
            out.append(_run64(case, seed + i, n, k, np.ones(k.shape[1])))
        return out
    n = case["n"]
    if kind == "interp":
        m, k = _model(case, seed, n), _kpath(seed, case["nk"])
        e, V, A, Om = _interp64(m, k, case["velo"])

        def back(x, perm):
            return None if x is None else np.asfortranarray(x.permute(perm).cpu().numpy())
        return (back(e, (1, 0)), back(V, (1, 2, 3, 0)), back(A, (1, 2, 3, 0)),
                back(Om, (1, 2, 3, 4, 0)))
    if kind == "list":
        k, w = _klist(seed, case["nk"])
    else:
        k = _mesh_points((case["n1"], case["n2"], case["n3"]))
        w = np.ones(k.shape[1])
    return _run64(case, seed, n, k, w)
