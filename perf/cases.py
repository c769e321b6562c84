"""The calls whose speed counts, as a user's AFQMC program makes them.

A case is one pass through the public entry points of safire_amd on inputs of stated sizes:
whole blocks of walker steps (a NOMSD or a PHMSD trial, FP64 or mixed precision), local-energy
evaluations, one back-propagated measurement, and the single operations that a program builds a
step from (vHS, vbias, Propagate, MixedDensityMatrix, orthogonalize).  The hamiltonians follow
the synthetic recipe of safire_amd.synthetic (h1 = sym N(0, 0.1) + diag(linspace(-2, 1)),
Cholesky vectors sym N(0, 1) * 0.1 * exp(-m / 20)), drawn on the GPU from the seed; the walkers
are the trial with a complex perturbation, as they are after some steps.

Sizes: N orbitals, n (up) and nd (down, 0: closed shell) electrons, M Cholesky vectors, W walkers.
"""
import math

import numpy as np
import torch

from safire_amd import afq, driver
from safire_amd.phmsd import PHMSD, build_ph_struct
from safire_amd.synthetic import make_phmsd_problem

DT = 0.005          # time step of every workload
ORDER = 6           # Taylor terms of the propagator
BLOCK = 5           # steps between two orthogonalizations
AMPLITUDE = 0.1     # Cholesky amplitude
NOISE = 0.2         # perturbation of the walkers
FIELD_SEED, FIELD_STREAM = 4242, 1


def listed():
    return [
        # the smallest production run: a minimal-basis molecule, every launch is latency
        dict(name="step_fp64_N24", kind="step", N=24, n=5, nd=0, M=96, W=64, mixed=False),
        # FP64 production run of a mid-size molecule
        dict(name="step_fp64_N108", kind="step", N=108, n=24, nd=0, M=600, W=512, mixed=False),
        # the headline run: mixed precision, large basis, one GPU full of walkers
        dict(name="step_mixed_N200", kind="step", N=200, n=40, nd=0, M=1600, W=1024, mixed=True),
        # the same run on one GPU of eight: an eighth of the walkers
        dict(name="step_mixed_N200_W128", kind="step", N=200, n=40, nd=0, M=1600, W=128,
             mixed=True),
        # a job of the serving loop, of sizes that fit no tile
        dict(name="step_mixed_N97", kind="step", N=97, n=23, nd=0, M=487, W=301, mixed=True),
        # multi-determinant run: 2000 particle-hole determinants, two spin blocks
        dict(name="step_phmsd_N64", kind="phmsd_step", N=64, n=10, M=320, W=256, ndet=2000),
        # the energy estimator's evaluation in the headline run and in the two others
        dict(name="energy_mixed_N200", kind="energy", N=200, n=40, nd=0, M=1600, W=1024,
             mixed=True),
        dict(name="energy_fp64_N108", kind="energy", N=108, n=24, nd=0, M=600, W=512,
             mixed=False),
        dict(name="energy_phmsd_N64", kind="phmsd_energy", N=64, n=10, M=320, W=256, ndet=2000),
        # one back-propagated density-matrix measurement of a small molecule (the sizes of the
        # BH inputs under tests/golden), 100-step window
        dict(name="backprop_N19", kind="backprop", N=19, n=3, M=78, W=1536, window=100),
        # single operations of a program with its own step: the largest serving job's force bias
        # in mixed precision, and the FP64 propagation of a full GPU of walkers
        dict(name="vbias_mixed_N160", kind="vbias", N=160, n=40, nd=0, M=800, W=512, mixed=True),
        dict(name="propagate_fp64_N200", kind="propagate", N=200, n=40, W=512, mixed=False),
    ]


KINDS = ("step", "step", "step", "energy", "energy", "vhs", "vbias", "propagate", "density", "qr",
         "phmsd_step", "phmsd_energy", "backprop")


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(KINDS)
    if kind in ("phmsd_step", "phmsd_energy"):
        n = rng.randint(6, 12)  # the active space holds n electrons in n + 5 orbitals
        N = _log_uniform(rng, 2 * n + 5, 64)
        return dict(kind=kind, N=N, n=n, M=int(N * rng.uniform(3.0, 5.0)),
                    W=_log_uniform(rng, 64, 256), ndet=_log_uniform(rng, 50, 2000))
    if kind == "backprop":
        N = rng.randint(12, 40)
        return dict(kind=kind, N=N, n=max(2, int(N * rng.uniform(0.1, 0.25))),
                    M=int(N * rng.uniform(3.0, 5.0)), W=_log_uniform(rng, 64, 1536),
                    window=rng.randint(20, 100))
    N = _log_uniform(rng, 16, 200)
    n = max(2, min(40, int(N * rng.uniform(0.1, 0.25))))
    case = dict(kind=kind, N=N, n=n, W=_log_uniform(rng, 64, 1024),
                mixed=kind not in ("density", "qr") and rng.random() < 0.5)
    if kind in ("step", "energy", "vhs", "vbias"):
        case["M"] = int(N * rng.uniform(3.0, 8.0))
    if kind in ("step", "energy", "vbias"):  # an open-shell (COLLINEAR) run now and then
        case["nd"] = max(1, n - rng.randint(0, 2)) if rng.random() < 0.3 else 0
    top = work(listed()[2])["flops"]  # the headline block is the largest
    while work(case)["flops"] * (1 if case["mixed"] else 2) > top:
        case["W"] = max(64, case["W"] // 2)
    return case


# ---------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------

def _ops(N, M, W, ns, mixed):
    """FLOP of the parts of a step over the spin blocks `ns` (a real trial, Cholesky tensor and
    one-body propagator: 4 FLOP a complex x real MAC, 8 a complex one)."""
    s1, s2, s3 = sum(ns), sum(n * n for n in ns), sum(n ** 3 for n in ns)
    return dict(density=16 * s2 * N + 16 * s3, overlap=8 * s2 * N + 8 * s3 / 3, qr=16 * s2 * N,
                vbias=4 * M * s1 * N, vhs=2 * N * (N + 1) * M,
                propagate=8 * ORDER * N * N * s1 + 8 * N * N * s1,
                energy=4 * s2 * N * M + 4 * s2 * M)


def work(case):
    k, N, W = case["kind"], case["N"], case["W"]
    M, mixed = case.get("M", 0), case.get("mixed", False)
    n = case["n"]
    if k.startswith("phmsd"):
        ns = (n, n)
    else:
        ns = (n, case["nd"]) if case.get("nd") else (n,)
    f = _ops(N, M, W, ns, mixed)
    r = 4 if mixed else 8           # bytes of a real number of the contractions
    s1 = sum(ns)
    phi, half, chol = 16 * W * N * s1, r * M * s1 * N, r * N * (N + 1) // 2 * M
    if k in ("step", "phmsd_step"):
        one = f["density"] + f["vbias"] + f["vhs"] + f["propagate"] + f["overlap"]
        return {"flops": W * (BLOCK * one + f["qr"]), "bytes": BLOCK * (2 * phi + half + chol)}
    if k in ("energy", "phmsd_energy"):
        return {"flops": W * (f["density"] + f["energy"]), "bytes": phi + half}
    if k == "vhs":
        return {"flops": W * f["vhs"], "bytes": chol + 2 * r * W * (M + N * N)}
    if k == "vbias":
        return {"flops": W * f["vbias"], "bytes": phi + half + 16 * W * M}
    if k == "propagate":
        return {"flops": W * 8 * (ORDER + 2) * N * N * n, "bytes": 2 * phi + 2 * r * W * N * N}
    if k == "density":
        return {"flops": W * f["density"], "bytes": 2 * phi}
    if k == "qr":
        return {"flops": W * f["qr"], "bytes": 2 * phi}
    if k == "backprop":
        one = f["vhs"] + 8 * (ORDER + 2) * N * N * n
        return {"flops": W * (case["window"] * one + f["density"] + 8 * N * N * n),
                "bytes": 16 * W * case["window"] * M + phi}
    raise ValueError(k)


# ---------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, dtype=torch.float64, device="cuda")


def _complex(g, *shape):
    return torch.complex(_normal(g, *shape), _normal(g, *shape))


def _system(case, seed, cholesky=True):
    """h1 [N][N], Likn [N][N][M] (GPU), PsiT [nel][N] (host) and the walkers of each spin block."""
    N, W = case["N"], case["W"]
    g = _generator(seed)
    up = torch.ones(N, N, dtype=torch.bool, device="cuda").triu()
    h = 0.1 * _normal(g, N, N)
    h1 = torch.where(up, h, h.T) + torch.diag(torch.linspace(-2.0, 1.0, N, dtype=torch.float64,
                                                             device="cuda"))
    L = None
    if cholesky:
        M = case["M"]
        L = _normal(g, N, N, M)
        L = torch.where(up[:, :, None], L, L.transpose(0, 1))
        L *= AMPLITUDE * torch.exp(-torch.arange(M, dtype=torch.float64, device="cuda") / 20.0)
    h1 = h1.cpu().numpy()
    orbitals = np.linalg.eigh(h1)[1]
    ns = [case["n"]] + ([case["nd"]] if case.get("nd") else [])
    PsiT = np.ascontiguousarray(np.concatenate([orbitals[:, :n].T for n in ns])
                                .astype(np.complex128))
    walkers = []
    for n in ns:
        trial = torch.from_numpy(np.ascontiguousarray(orbitals[:, :n])).to("cuda")
        walkers.append((trial + (NOISE / math.sqrt(N)) * _complex(g, W, N, n)).contiguous())
    return h1, L, PsiT, walkers


def _hamiltonian(case, seed):
    h1, L, PsiT, walkers = _system(case, seed)
    ctx = afq.Context(0)
    ham = afq.HamiltonianOperations(
        ctx, h1, L.cpu().numpy(), PsiT, case["n"], case.get("nd", 0),
        afq.AFQ_COLLINEAR if case.get("nd") else afq.AFQ_CLOSED,
        precision=afq.AFQ_MIXED if case.get("mixed") else afq.AFQ_FP64)
    return ctx, ham, PsiT, walkers


def _walker_set(walkers):
    return afq.WalkerSet(*[w.cpu().numpy() for w in walkers])


def _propagate_inputs(case, seed):
    """P1 = exp(-h1 dt / 2), a complex symmetric V of a step's size, the walkers."""
    N, W = case["N"], case["W"]
    h1, _, _, walkers = _system(case, seed, cholesky=False)
    P1 = torch.linalg.matrix_exp(torch.from_numpy(-0.5 * DT * h1)).to(torch.complex128).to("cuda")
    g = _generator(seed + 1)
    V = torch.empty(W, N, N, dtype=torch.complex64 if case["mixed"] else torch.complex128,
                    device="cuda")
    for w0 in range(0, W, 64):
        v = (0.3 / math.sqrt(N)) * _complex(g, min(64, W - w0), N, N)
        V[w0:w0 + 64] = 0.5 * (v + v.transpose(1, 2))
    return P1, V, walkers[0]


def prepare(case, seed):
    k, W, N = case["kind"], case["W"], case["N"]
    state = {"kind": k}
    if k in ("phmsd_step", "phmsd_energy"):
        p = make_phmsd_problem(N, case["n"], case["M"], case["ndet"], ncore=case["n"] - 5,
                               nactive=10, seed=int(seed) & 0x7FFFFFFF, lscale=AMPLITUDE)
        ctx = afq.Context(0)
        ham = afq.HamiltonianOperations(ctx, p.h1, p.Likn, p.PsiT, p.nact, p.nact,
                                        afq.AFQ_COLLINEAR)
        trial = PHMSD(ham, build_ph_struct(p.occa, p.occb, p.ci))
        ws = afq.WalkerSet(*p.walkers(W, seed=int(seed) & 0x7FFFFFFF, noise=NOISE))
        prop = afq.Propagator(ham, W, dt=DT, order=ORDER, seed=FIELD_SEED, stream=FIELD_STREAM,
                              trial=trial)
    elif k in ("step", "energy", "backprop"):
        ctx, ham, PsiT, walkers = _hamiltonian(case, seed)
        ws = _walker_set(walkers)
        prop = afq.Propagator(ham, W, dt=DT, order=ORDER, seed=FIELD_SEED, stream=FIELD_STREAM)
    if k in ("step", "phmsd_step"):
        state.update(ws=ws, prop=prop, Eshift=driver.initialize(prop, ws),
                     e_out=afq.empty(1, torch.float64))
    elif k in ("energy", "phmsd_energy"):
        state.update(ws=ws, prop=prop, E=afq.empty((W, 3), torch.complex128),
                     ovlp=afq.empty(W, torch.complex128),
                     precision=afq.AFQ_MIXED if case.get("mixed") else afq.AFQ_FP64)
    elif k == "backprop":
        Eshift, e_out = driver.initialize(prop, ws), afq.empty(1, torch.float64)
        prop.enable_backprop(case["window"])
        prop.bp_anchor(ws)
        for i in range(case["window"]):
            prop.step_graph(ws, Eshift, ortho=(i % BLOCK == 0), energy_out=e_out)
        state.update(ws=ws, prop=prop, window=case["window"])
    elif k in ("vhs", "vbias"):
        ctx, ham, PsiT, walkers = _hamiltonian(case, seed)
        g = _generator(seed + 1)
        state["ham"] = ham
        if k == "vhs":
            out = torch.complex64 if case["mixed"] else torch.complex128
            # fields: a normal draw and a force bias of a few tenths
            X = _normal(g, W, case["M"]) + 0.3 * _complex(g, W, case["M"])
            state.update(X=X.to(out).contiguous(), V=afq.empty((W, N, N), out))
        else:
            state.update(G=_density(PsiT, walkers),
                         v=afq.empty((W, case["M"]), torch.complex128))
    elif k == "propagate":
        ctx = afq.Context(0)
        P1, V, phi = _propagate_inputs(case, seed)
        state.update(ctx=ctx, P1=P1, V=V, Phi0=phi, Phi=torch.empty_like(phi),
                     precision=afq.AFQ_MIXED if case["mixed"] else afq.AFQ_FP64)
    elif k in ("density", "qr"):
        ctx = afq.Context(0)
        _, _, PsiT, walkers = _system(case, seed, cholesky=False)
        n = case["n"]
        state.update(ctx=ctx, PsiT=afq.device_tensor(PsiT), Phi0=walkers[0],
                     Phi=walkers[0].clone(), G=afq.empty((W, n, N), torch.complex128),
                     ld=afq.zeros(W, torch.complex128))
    torch.cuda.synchronize()
    return state


def _density(PsiT, walkers):
    """Compact density matrices [W][nel][N] of the walkers, with torch: what feeds vbias."""
    rows = torch.from_numpy(PsiT).split([w.shape[2] for w in walkers])
    return torch.cat([torch.linalg.inv(r @ w.cpu()).transpose(1, 2) @ w.cpu().transpose(1, 2)
                      for r, w in zip(rows, walkers)], dim=1).contiguous().to("cuda")


def run(state):
    k = state["kind"]
    if k in ("step", "phmsd_step"):
        ws, prop = state["ws"], state["prop"]
        for i in range(BLOCK):
            prop.step_graph(ws, state["Eshift"], ortho=(i == BLOCK - 1),
                            energy_out=state["e_out"])
        out = {"Phi": ws.Phi, "weight": ws.weight, "phase": ws.phase, "eloc": ws.eloc,
               "ovlp": ws.ovlp, "theta": ws.theta}
        if ws.Phi_b is not None:
            out["Phi_b"] = ws.Phi_b
        return out
    if k in ("energy", "phmsd_energy"):
        state["prop"].Energy(state["ws"], state["E"], state["ovlp"], state["precision"])
        return {"E": state["E"], "ovlp": state["ovlp"]}
    if k == "backprop":
        one, two = state["prop"].bp_measure(state["ws"], state["window"], ortho=10, restore=1)
        return {"onerdm": one, "diag2rdm": two}
    if k == "vhs":
        state["ham"].vHS(state["X"], state["V"], DT)
        return state["V"]
    if k == "vbias":
        state["ham"].vbias(state["G"], state["v"], DT)
        return state["v"]
    if k == "propagate":
        state["Phi"].copy_(state["Phi0"])  # the proposal leaves the walkers of the last step
        afq.det_ops.Propagate(state["ctx"], state["P1"], state["V"], state["Phi"], ORDER, "N",
                              state["precision"])
        return state["Phi"]
    if k == "density":
        state["ld"].zero_()
        afq.det_ops.MixedDensityMatrix(state["ctx"], state["PsiT"], state["Phi"], state["G"],
                                       state["ld"])
        return {"G": state["G"], "ovlp": state["ld"]}
    state["Phi"].copy_(state["Phi0"])
    state["ld"].zero_()
    afq.det_ops.orthogonalize(state["ctx"], state["Phi"], state["ld"])
    return {"Phi": state["Phi"], "ldet": state["ld"]}


# ---------------------------------------------------------------------------------------------
# the same results in 64 bits with torch and numpy
# ---------------------------------------------------------------------------------------------

def _wrap(x):
    return torch.remainder(x + math.pi, 2 * math.pi) - math.pi


def _log_det(T):
    sign, logabs = torch.linalg.slogdet(T.cpu())
    return torch.complex(logabs, torch.angle(sign)).to("cuda")


class _Exact:
    """The single-determinant walker step of a hamiltonian (CLOSED or COLLINEAR) in 64 bits."""

    def __init__(self, h1, L, PsiT, ns, closed):
        self.N, self.M = L.shape[0], L.shape[2]
        self.h1, self.L = torch.from_numpy(h1).to("cuda"), L
        rows = torch.from_numpy(np.ascontiguousarray(PsiT.real)).to("cuda").split(ns)
        self.rows, self.closed, self.c = rows, closed, 2.0 if closed else 1.0
        # half-rotated vectors [M][n][N] and one-body rows
        self.Lh = [torch.einsum("ai,ikm->mak", r, L).contiguous() for r in rows]
        self.hh = [r @ self.h1 for r in rows]

    def overlap(self, Phi):
        logs = [_log_det(r.to(torch.complex128) @ P) for r, P in zip(self.rows, Phi)]
        if self.closed:
            return 2.0 * torch.complex(logs[0].real, _wrap(logs[0].imag))
        t = torch.zeros_like(logs[0])
        for x in logs:
            t = torch.complex(t.real + x.real, _wrap(t.imag + x.imag))
        return t

    def density(self, Phi):
        return [torch.linalg.inv((r.to(torch.complex128) @ P).cpu()).to("cuda").transpose(1, 2)
                @ P.transpose(1, 2) for r, P in zip(self.rows, Phi)]

    def vbias(self, G):
        v = 0
        for g, l in zip(G, self.Lh):
            B = l.reshape(self.M, -1).T.contiguous()
            g = g.reshape(g.shape[0], -1)
            v = v + torch.complex(g.real.contiguous() @ B, g.imag.contiguous() @ B)
        return math.sqrt(DT) * self.c * v

    def vhs(self, X):
        B = self.L.reshape(-1, self.M).T
        V = torch.complex(X.real.contiguous() @ B, X.imag.contiguous() @ B)
        return math.sqrt(DT) * V.reshape(X.shape[0], self.N, self.N)

    def energy(self, Phi):
        G = self.density(Phi)
        W = G[0].shape[0]
        E = torch.zeros(W, 3, dtype=torch.complex128, device="cuda")
        K = torch.zeros(W, self.M, dtype=torch.complex128, device="cuda")
        for g, l, h in zip(G, self.Lh, self.hh):
            n = g.shape[1]
            E[:, 0] += self.c * (g * h).sum((1, 2))
            gr, gi = g.real.reshape(-1, self.N), g.imag.reshape(-1, self.N)
            step = max(1, (1 << 27) // (W * n * n))
            for m in range(0, self.M, step):
                b = l[m:m + step].reshape(-1, self.N).T
                T = torch.complex(gr @ b, gi @ b).reshape(W, n, -1, n)
                E[:, 1] -= 0.5 * self.c * (T * T.permute(0, 3, 2, 1)).sum((1, 2, 3))
                K[:, m:m + step] += torch.diagonal(T, dim1=1, dim2=3).sum(-1)
        E[:, 2] = 0.5 * self.c ** 2 * (K * K).sum(1)
        return E

    def mean_field(self):
        trial = [r.T.to(torch.complex128)[None].contiguous() for r in self.rows]
        vmf = self.vbias(self.density(trial))[0].real
        flat = self.L.reshape(self.N, -1)
        H = DT * (self.h1 - 0.5 * flat @ flat.T) + self.vhs(vmf.to(torch.complex128)[None])[0].real
        H = -0.25 * (H + H.T)
        w, U = torch.linalg.eigh(H.cpu())
        P1 = ((U * torch.exp(w)) @ U.T).to("cuda")
        return vmf, torch.where(P1.abs() > 1e-8, P1, torch.zeros_like(P1))


def _philox_uniforms(seed, stream, step, W, M):
    """Uniforms u[w][m] of Philox4x32-10 (Salmon et al., SC'11), counter (m / 2, w, step, stream),
    two draws of 53 bits a counter."""
    lo = np.uint64(0xFFFFFFFF)
    half = (M + 1) // 2
    c = [np.broadcast_to(np.arange(half, dtype=np.uint64)[None], (W, half)).copy(),
         np.broadcast_to(np.arange(W, dtype=np.uint64)[:, None], (W, half)).copy(),
         np.full((W, half), step, np.uint64), np.full((W, half), stream, np.uint64)]
    k0, k1 = seed & 0xFFFFFFFF, seed >> 32
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & lo,
             (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1), p0 & lo]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    bits = np.stack([(c[0] << np.uint64(32)) | c[1], (c[2] << np.uint64(32)) | c[3]], axis=-1)
    u = ((bits >> np.uint64(11)).astype(np.float64) + 0.5) / 9007199254740992.0
    return torch.from_numpy(np.ascontiguousarray(u.reshape(W, -1)[:, :M])).to("cuda")


def _clamp(x, bound=50.0):
    a = x.abs()
    return torch.where(a > bound, x * (bound / a), x)


def _exact_block(case, seed):
    h1, L, PsiT, Phi = _system(case, seed)
    W, M = case["W"], case["M"]
    ns = [p.shape[2] for p in Phi]
    x = _Exact(h1, L, PsiT, ns, not case.get("nd"))
    vmf, P1 = x.mean_field()
    P1 = P1.to(torch.complex128)
    Eshift = x.energy(Phi).sum(1).real.mean()
    old = x.overlap(Phi)
    weight = torch.ones(W, dtype=torch.complex128, device="cuda")
    phase = weight.clone()
    hi, lo = Eshift + 10.0 * math.sqrt(2 / DT), Eshift - math.sqrt(2 / DT)
    for step in range(BLOCK):
        vb = _clamp(x.vbias(x.density(Phi)))
        vd = 1j * (vb - _clamp(vmf.to(torch.complex128)))
        u = _philox_uniforms(FIELD_SEED, FIELD_STREAM, step, W, M)
        X = torch.special.ndtri(u) + vd
        HW = -(vd * (X - 0.5 * vd)).sum(1)
        mf = 1j * (X * vmf).sum(1) - 0.5 * (vmf * vmf).sum()
        V = x.vhs(X)
        for s, P in enumerate(Phi):
            T = P1 @ P
            S = T.clone()
            for k in range(1, ORDER + 1):
                T = (1j / k) * (V @ T)
                S += T
            Phi[s] = P1 @ S
        new = x.overlap(Phi)
        theta = new.imag - old.imag - mf.imag
        e = (mf - HW - torch.complex(new.real - old.real, new.imag - old.imag)) / DT
        e = torch.complex(e.real.clamp(lo, hi), e.imag)
        f = torch.exp(-DT * (e - Eshift))
        weight = weight * torch.cos(theta).clamp(min=0.0) * f.abs()
        phase = phase * f / f.abs()
        big = max(100.0, 0.1 * W)
        weight = torch.where(weight.abs() > big, weight * (big / weight.abs()), weight)
        old = new
    for s, P in enumerate(Phi):
        Q, R = torch.linalg.qr(P.cpu())
        d = torch.diagonal(R, dim1=1, dim2=2)
        Phi[s] = (Q * (d / d.abs())[:, None, :]).to("cuda")
    out = {"Phi": Phi[0], "weight": weight, "phase": phase, "eloc": e, "ovlp": x.overlap(Phi),
           "theta": theta.to(torch.complex128)}
    if len(Phi) > 1:
        out["Phi_b"] = Phi[1]
    return out


def exact(case, seed):
    k = case["kind"]
    if k in ("phmsd_step", "phmsd_energy", "backprop"):
        return None  # FP64 throughout; a sum over 2000 determinants or a window of 100 steps
    if k == "step":
        return _exact_block(case, seed)
    if k == "propagate":
        P1, V, T = _propagate_inputs(case, seed)
        T = P1 @ T
        S = T.clone()
        for i in range(1, ORDER + 1):
            T = (1j / i) * torch.cat([V[w:w + 64].to(torch.complex128) @ T[w:w + 64]
                                      for w in range(0, T.shape[0], 64)])
            S += T
        return P1 @ S
    if k in ("density", "qr"):
        _, _, PsiT, (Phi,) = _system(case, seed, cholesky=False)
        if k == "qr":
            Q, R = torch.linalg.qr(Phi.cpu())
            d = torch.diagonal(R, dim1=1, dim2=2)
            return {"Phi": Q * (d / d.abs())[:, None, :],
                    "ldet": torch.log(d.abs()).sum(1).to(torch.complex128)}
        T = torch.from_numpy(PsiT) @ Phi.cpu()
        sign, logabs = torch.linalg.slogdet(T)
        return {"G": torch.linalg.inv(T).transpose(1, 2) @ Phi.cpu().transpose(1, 2),
                "ovlp": torch.complex(logabs, torch.angle(sign))}
    h1, L, PsiT, Phi = _system(case, seed)
    x = _Exact(h1, L, PsiT, [p.shape[2] for p in Phi], not case.get("nd"))
    if k == "energy":
        return {"E": x.energy(Phi), "ovlp": x.overlap(Phi)}
    if k == "vbias":
        G = _density(PsiT, Phi)
        return x.vbias(list(G.split([p.shape[2] for p in Phi], dim=1)))
    g = _generator(seed + 1)
    X = _normal(g, case["W"], case["M"]) + 0.3 * _complex(g, case["W"], case["M"])
    return x.vhs(X.to(torch.complex64).to(torch.complex128) if case["mixed"] else X)
