"""Performance cases of the engine: what a user has it do, through the Python entry points.

Each family below is one kind of call, over the sizes that people run it at (a molecule's occupied /
virtual / fitting-function counts): the smallest calls, where latency and launches count, ordinary
ones, and the largest.  Inputs are seeded and made on the GPU, with the structure that molecular DF
tensors have (as fermihip.synth.molecular_like: symmetric, a decaying auxiliary spectrum, Coulomb-like
positive self-densities, MP2 energy of about -0.05 Eh per occupied orbital).

``exact`` restates every family in plain torch / numpy FP64.
"""
import gc
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "fermi.jl_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "fermi.jl_amd"))

import fermihip  # noqa: E402
from fermihip import basis as fbasis  # noqa: E402

F64 = torch.float64


def dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the correlation energy of one small molecule inside a scan: launches and latency
        {"name": "df_mp2 o5 v19", "kind": "mp2", "o": 5, "v": 19, "naux": 84},
        # the same call at the benchmark molecule's size
        {"name": "df_mp2 o40 v190", "kind": "mp2", "o": 40, "v": 190, "naux": 840},
        # one amplitude update of a small molecule, FP64, host arrays in and out
        {"name": "ccsd_update o5 v19", "kind": "update", "o": 5, "v": 19, "naux": 84},
        # RCCSD of a medium molecule to the default criteria, FP64, amplitudes returned
        {"name": "rccsd fp64 o16 v76", "kind": "rccsd", "o": 16, "v": 76, "naux": 336},
        # DF tensors -> RCCSD(T) energy with split-BF16x3 contractions and two FP64 polish iterations
        {"name": "rccsd(t) bf16x3 o28 v133", "kind": "ccsdpt", "o": 28, "v": 133, "naux": 588},
        # (T) on device-resident amplitudes: FP64, the default of RCCSDpT
        {"name": "triples fp64 o16 v76", "kind": "triples", "o": 16, "v": 76, "naux": 336, "prec": 0},
        # split-BF16x3 (T) where v is no multiple of a tile
        {"name": "triples bf16x3 o27 v131", "kind": "triples", "o": 27, "v": 131, "naux": 500, "prec": 2},
        # split-BF16x3 (T) of the benchmark molecule
        {"name": "triples bf16x3 o40 v190", "kind": "triples", "o": 40, "v": 190, "naux": 840, "prec": 2},
        # three-centre integrals of a cluster in cc-pVDZ with its RI fitting set (the DF front end)
        {"name": "eri_3c (h2o)4", "kind": "eri3c", "waters": 4, "basis": "cc-pvdz"},
        # four-centre integrals of a small molecule (the conventional chain)
        {"name": "eri_4c (h2o)2", "kind": "eri4c", "waters": 2, "basis": "cc-pvdz"},
        # DF-RHF of a medium molecule
        {"name": "df_rhf nbf96", "kind": "rhf", "nbf": 96, "naux": 464, "ndocc": 20},
        # forward + backward of the guess network on one minibatch
        {"name": "mlp_loss_grad n8192", "kind": "mlp", "n": 8192, "hidden": 128},
    ]


def _logu(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _space(rng, vmax, omax):
    v = _logu(rng, 12, vmax)
    o = max(2, min(omax, int(round(v * rng.uniform(0.15, 0.4)))))
    naux = int(round((o + v) * rng.uniform(3.2, 4.2)))
    return {"o": o, "v": v, "naux": naux}


def draw(rng):
    kind = rng.choice(["mp2", "update", "rccsd", "ccsdpt", "triples", "triples", "triples", "eri3c", "eri4c", "rhf",
                       "mlp"])
    c = {"kind": kind}
    if kind == "mp2":
        c.update(_space(rng, 190, 40))
    elif kind == "update":
        c.update(_space(rng, 110, 30))
    elif kind == "rccsd":
        c.update(_space(rng, 100, 24))
    elif kind == "ccsdpt":
        c.update(_space(rng, 140, 28))
    elif kind == "triples":
        c["prec"] = rng.choice([0, 1, 2, 2])
        c.update(_space(rng, 190 if c["prec"] == 2 else 110, 40 if c["prec"] == 2 else 24))
    elif kind == "eri3c":
        c.update(waters=rng.randint(1, 5), basis=rng.choice(["cc-pvdz", "6-31g"]))
    elif kind == "eri4c":
        c["basis"] = rng.choice(["sto-3g", "6-31g", "cc-pvdz"])
        c["waters"] = rng.randint(1, 2 if c["basis"] == "cc-pvdz" else 4)
    elif kind == "rhf":
        n = _logu(rng, 12, 140)
        c.update(nbf=n, naux=int(n * rng.uniform(3.2, 4.8)), ndocc=max(1, n // 5))
    else:
        c.update(n=_logu(rng, 100, 60000), hidden=rng.choice([32, 64, 128]))
    if kind in ("eri3c", "eri4c"):
        c["jitter"] = round(rng.uniform(0.0, 0.2), 3)  # displacement of the cluster's atoms, bohr
    return c


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=dev()).manual_seed(int(seed) * 7919 + 17)


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=dev(), dtype=F64)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=dev(), dtype=F64)


def _df(case, seed):
    """(eps_o, eps_v, Boo, Bov, Bvv) as torch FP64 tensors B[Q, p, q]."""
    o, v, Q = case["o"], case["v"], case["naux"]
    g, n = _gen(seed), o + v
    eo = torch.sort(-1.5 + 1.2 * _rand(g, o)).values
    ev = torch.sort(0.1 + 2.9 * _rand(g, v)).values
    decay = torch.exp(-torch.arange(Q, device=dev(), dtype=F64) / (Q / 3.0))
    G = _randn(g, Q, n, n)
    G = (G + G.transpose(1, 2)) * (decay / math.sqrt(2.0))[:, None, None]
    dens = _randn(g, Q, n).abs() * decay[:, None]
    X = _ovov(G[:, :o, o:])
    e1 = torch.sum(X * (2 * X - X.transpose(1, 3)) / _d2(eo, ev).permute(0, 2, 1, 3)).item()
    e2 = -o * (0.045 + 0.01 * _rand(g, 1).item())  # the MP2 correlation energy of these tensors
    B = G * (e2 / e1) ** 0.25
    idx = torch.arange(n, device=dev())
    B[:, idx, idx] += 0.15 * dens / math.sqrt(max(Q, 84) / 84.0)
    return eo, ev, B[:, :o, :o], B[:, :o, o:], B[:, o:, o:]


def _ovov(Bov):
    Q, o, v = Bov.shape
    m = Bov.reshape(Q, o * v)
    return (m.T @ m).reshape(o, v, o, v)


def _d2(eo, ev):
    return eo[:, None, None, None] + eo[None, :, None, None] - ev[None, None, :, None] - ev[None, None, None, :]


def _host(t):
    """Column-major numpy copy (the library's array order) of a torch tensor."""
    return t.permute(*reversed(range(t.dim()))).contiguous().cpu().numpy().T


def _amplitudes(case, seed, eo, ev, Bov):
    """Amplitudes on their way to convergence: MP2 doubles scaled, and singles of their usual size."""
    g = _gen(seed + 1)
    t2 = _ovov(Bov).permute(0, 2, 1, 3) / _d2(eo, ev)
    return 0.01 * _randn(g, case["o"], case["v"]), t2 * (1.0 - 0.1 * _rand(g, 1).item())


def _atoms(case, seed):
    rng = np.random.default_rng(seed)
    atoms = fbasis.water_cluster(case["waters"], seed)
    return [(s, z, np.asarray(r) + rng.normal(0.0, case.get("jitter", 0.0) + 0.01, 3)) for s, z, r in atoms]


def _scf(case, seed):
    g, n, Q = _gen(seed), case["nbf"], case["naux"]
    A = _randn(g, n, n)
    S = torch.eye(n, device=dev(), dtype=F64) + 0.15 / math.sqrt(n) * (A + A.T)
    lo = torch.linalg.eigvalsh(S.cpu()).min().item()
    if lo < 0.3:
        S = S + (abs(lo) + 0.3) * torch.eye(n, device=dev(), dtype=F64)
    d = torch.sqrt(torch.diag(S))
    S = S / d[:, None] / d[None, :]
    B = _randn(g, n, n)
    diag = torch.linspace(-5.0, 2.0, n, device=dev(), dtype=F64)
    diag[case["ndocc"]:] += 1.5  # a closed-shell molecule's gap
    H = torch.diag(diag) + 0.5 / math.sqrt(n) * (B + B.T)
    G = _randn(g, Q, n, n)
    return S, H, 0.06 * math.sqrt(420.0 / (n * Q)) * (G + G.transpose(1, 2))


def _batch(case, seed):
    g = _gen(seed)
    f = torch.float32
    X = torch.randn(case["n"], 6, generator=g, device=dev(), dtype=f)
    T = 0.5 * torch.tanh(X[:, 0] * X[:, 5]) + 0.1 * torch.randn(case["n"], generator=g, device=dev(), dtype=f)
    return X.cpu().numpy(), T.cpu().numpy()


# ------------------------------------------------------------------ prepare and run
# solver options of the energy call: the schedule of bench.py's default step
CCSDPT_OPTS = dict(precision="bf16x3", polish_iters=2, bf3_e_switch=1e-6, bf3_rms_switch=1e-7)


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": dict(case)}
    if kind in ("mp2", "update", "rccsd", "ccsdpt", "triples"):
        eo, ev, Boo, Bov, Bvv = _df(case, seed)
        ctx = st["ctx"] = fermihip.Context(0)
        host = [_host(eo), _host(ev)] + ([None, _host(Bov), None] if kind == "mp2"
                                         else [_host(Boo), _host(Bov), _host(Bvv)])
        if kind == "ccsdpt":
            st["df"] = host
        elif kind != "rccsd":
            ctx.set_df(*host)
        if kind == "update":
            st["T1"], st["T2"] = (_host(t) for t in _amplitudes(case, seed, eo, ev, Bov))
            ctx.prepare()
        elif kind == "rccsd":
            st["moints"] = fermihip.MOIntegrals(host[2], host[3], host[4], host[0], host[1], context=ctx)
            ctx.set_df(*host)
            ctx.prepare()
        elif kind == "triples":
            ctx.guess(2, copy_out=False)
    elif kind in ("eri3c", "eri4c"):
        atoms = _atoms(case, seed)
        st["ctx"] = fermihip.Context(0)
        st["bs"] = fermihip.Basis(fbasis.shells_for(atoms, case["basis"]))
        if kind == "eri3c":
            st["aux"] = fermihip.Basis(fbasis.even_tempered_aux(atoms, "ri", case["basis"]))
    elif kind == "rhf":
        st["ctx"] = fermihip.Context(0)
        st["in"] = [_host(t) for t in _scf(case, seed)]
    else:
        st["net"] = fermihip.Mlp(hidden=case["hidden"], seed=seed)
        st["X"], st["T"] = _batch(case, seed)
    if dev().type == "cuda":
        torch.cuda.empty_cache()  # the library has its own pool
    gc.collect()
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "mp2":
        return st["ctx"].mp2_energy()
    if kind == "update":
        return st["ctx"].update_amp(st["T1"], st["T2"])
    if kind == "rccsd":
        r = fermihip.RCCSD(st["moints"])
        return {"correlation": r.correlation, "T1": r.T1, "T2": r.T2}
    if kind == "ccsdpt":
        ctx = st["ctx"]
        ctx.set_df(*st["df"])
        ctx.guess(2, copy_out=False)
        r, _, _ = ctx.solve(fermihip.Options(**CCSDPT_OPTS), copy_out=False)
        return {"ccsd": r.correlation, "triples": ctx.triples(prec_mode=2)}
    if kind == "triples":
        return st["ctx"].triples(prec_mode=case["prec"])
    if kind == "eri3c":
        return st["ctx"].eri_2e3c(st["bs"], st["aux"])
    if kind == "eri4c":
        return st["ctx"].eri_2e4c(st["bs"])
    if kind == "rhf":
        r, eps, C = st["ctx"].rhf(*st["in"], case["ndocc"])
        return {"energy": r["energy"], "eps": eps, "C": C}
    loss, grad = st["net"].loss_grad(st["X"], st["T"])
    return {"loss": loss, "grad": grad}


# ------------------------------------------------------------------ work
def _ccsd_flops(o, v):
    # one amplitude update: the particle-particle ladder over unordered pairs, four ring-type o^3 v^3
    # products, the hole-hole ladder and its intermediate, and the two one-index dressings
    return o * o * v ** 4 + 8.0 * o ** 3 * v ** 3 + 4.0 * o ** 4 * v * v + 2.0 * o * o * v ** 3


def _triples_flops(o, v):
    # six permutations, each 2 v^3 (v + o), for every i >= j >= k that is not i = j = k
    return (o * (o + 1) * (o + 2) / 6 - o) * 12.0 * v ** 3 * (v + o)


def work(case):
    kind = case["kind"]
    if kind in ("mp2", "update", "rccsd", "ccsdpt", "triples"):
        o, v, Q = case["o"], case["v"], case["naux"]
        ov, t2 = o * v, o * o * v * v
        df = 8.0 * Q * (ov + o * o + v * v)
        if kind == "mp2":
            return {"bytes": 8.0 * Q * ov, "flops": 1.0 * Q * ov * (ov + 1)}
        if kind == "update":
            return {"bytes": 16.0 * t2 + df, "flops": _ccsd_flops(o, v)}
        if kind == "rccsd":
            return {"bytes": 8.0 * t2 + df, "flops": 12 * _ccsd_flops(o, v)}
        if kind == "ccsdpt":
            return {"bytes": df, "flops": 10 * _ccsd_flops(o, v) + _triples_flops(o, v)}
        return {"bytes": 8.0 * (t2 + o * v ** 3), "flops": _triples_flops(o, v)}
    if kind in ("eri3c", "eri4c"):
        atoms = _atoms(case, 0)
        sh = fbasis.shells_for(atoms, case["basis"])
        n, pr = fbasis.nbf(sh), sum(len(s["exps"]) * (2 * s["l"] + 1) for s in sh)
        if kind == "eri4c":
            return {"bytes": 8.0 * n ** 4, "flops": 20.0 * pr ** 4 / 8}
        q = fbasis.nbf(fbasis.even_tempered_aux(atoms, "ri", case["basis"]))
        return {"bytes": 8.0 * n * n * q, "flops": 20.0 * pr * pr * q / 2}
    if kind == "rhf":
        n, Q, no = case["nbf"], case["naux"], case["ndocc"]
        return {"bytes": 8.0 * (Q * n * n + 4 * n * n), "flops": 10.0 * (4.0 * Q * n * n * (1 + no) / 2 + 12.0 * n ** 3)}
    h = case["hidden"]
    return {"bytes": 28.0 * case["n"] + 8.0 * (2 * h * h + 10 * h), "flops": 6.0 * case["n"] * (2 * h * h + 7 * h)}


# ------------------------------------------------------------------ exact: plain FP64 restatements
def exact(case, seed):
    kind = case["kind"]
    if kind in ("mp2", "update", "rccsd", "ccsdpt", "triples"):
        eo, ev, Boo, Bov, Bvv = _df(case, seed)
        if kind == "mp2":
            X = _ovov(Bov)
            return torch.sum(X * (2 * X - X.transpose(1, 3)) / _d2(eo, ev).permute(0, 2, 1, 3)).item()
        m = _blocks(Boo, Bov, Bvv)
        if kind == "update":
            return tuple(_update(m, eo, ev, *_amplitudes(case, seed, eo, ev, Bov)))
        t2 = m["ovov"].permute(0, 2, 1, 3) / _d2(eo, ev)
        if kind == "triples":
            t1 = _residual(m, torch.zeros_like(Bov[0]), t2, only_t1=True) / (eo[:, None] - ev[None, :])
            return _triples(m, eo, ev, t1, t2)
        t1, t2 = _solve(m, eo, ev, t2)
        e = _energy(m, t1, t2)
        if kind == "rccsd":
            return {"correlation": e, "T1": t1, "T2": t2}
        return {"ccsd": e, "triples": _triples(m, eo, ev, t1, t2)}
    if kind == "rhf":
        e, eps = _scf_exact(case, *(t.cpu().numpy() for t in _scf(case, seed)))
        return {"energy": e, "eps": eps, "C": None}  # orbitals are defined up to their signs
    if kind in ("eri3c", "eri4c"):
        atoms = _atoms(case, seed)
        sh = fbasis.shells_for(atoms, case["basis"])
        if kind == "eri3c":
            return _eri(sh, fbasis.even_tempered_aux(atoms, "ri", case["basis"]), True)
        return _eri(sh, sh, False)
    return _mlp_exact(case, seed)


def _blocks(Boo, Bov, Bvv):
    Q, o, v = Bov.shape
    a, b, c = Boo.reshape(Q, -1), Bov.reshape(Q, -1), Bvv.reshape(Q, -1)
    return {"oooo": (a.T @ a).reshape(o, o, o, o), "ooov": (a.T @ b).reshape(o, o, o, v),
            "oovv": (a.T @ c).reshape(o, o, v, v), "ovov": (b.T @ b).reshape(o, v, o, v),
            "ovvv": (b.T @ c).reshape(o, v, v, v), "Bvv": Bvv}


def _residual(m, t1, t2, only_t1=False):
    """Numerators of the closed-shell CCSD update without the diagonal Fock terms."""
    e = torch.einsum
    ovov, ovvv, ooov, oovv, oooo = m["ovov"], m["ovvv"], m["ooov"], m["oovv"], m["oooo"]
    L = 2 * ovov - ovov.transpose(1, 3)
    u = 2 * t2 - t2.transpose(2, 3)
    tau = t2 + e("ia,jb->ijab", t1, t1)
    Fov = e("kcld,ld->kc", L, t1)
    Foo = e("kcld,ilcd->ki", L, t2) + e("kc,ic->ki", Fov, t1)
    Fvv = -e("kcld,klad->ac", L, t2) - e("ka,kc->ac", t1, Fov)
    Loo = Foo + 2 * e("kilc,lc->ki", ooov, t1) - e("likc,lc->ki", ooov, t1)
    Lvv = Fvv + 2 * e("kdac,kd->ac", ovvv, t1) - e("kcad,kd->ac", ovvv, t1)
    r1 = e("ac,ic->ia", Lvv, t1) - e("ki,ka->ia", Loo, t1) + e("kc,kica->ia", Fov, u)
    r1 = r1 + e("ic,kc,ka->ia", t1, Fov, t1) + 2 * e("kcia,kc->ia", ovov, t1) - e("kiac,kc->ia", oovv, t1)
    r1 = r1 + e("kdac,ikcd->ia", ovvv, u) - e("kilc,klac->ia", ooov, u)
    if only_t1:
        return r1
    P = 0.5 * ovov.permute(0, 2, 1, 3) + e("iacb,jc->ijab", ovvv, t1)
    P = P - e("kibj,ka->ijab", e("kibc,jc->kibj", oovv, t1), t1)
    P = P - e("kija,kb->ijab", e("kcia,jc->kija", ovov, t1) + ooov.permute(1, 2, 0, 3), t1)
    W = oooo.permute(0, 2, 1, 3) + e("kilc,jc->klij", ooov, t1) + e("ljkc,ic->klij", ooov, t1)
    W = W + e("kcld,ijcd->klij", ovov, tau)
    P = P + 0.5 * e("klij,klab->ijab", W, tau)
    # particle-particle ladder, one virtual a at a time: (ca|db) from the DF tensor, and its T1 dressing
    B = m["Bvv"]
    Q, v, _ = B.shape
    Bm = B.reshape(Q, v * v)
    for a in range(v):
        w = (B[:, :, a].T @ Bm).reshape(v, v, v)  # [c, d, b]
        P[:, :, a, :] += 0.5 * e("ijcd,cdb->ijb", tau, w)
        P[:, :, a, :] -= e("ijk,kb->ijb", e("ijcd,kdc->ijk", tau, ovvv[:, :, a, :]), t1)
    P = P + e("ac,ijcb->ijab", Lvv, t2) - e("ki,kjab->ijab", Loo, t2)
    Wa = ovov.permute(3, 0, 2, 1) + e("kcad,id->akic", ovvv, t1) - e("likc,la->akic", ooov, t1)
    Wa = Wa - e("lkci,la->akic", e("ldkc,id->lkci", ovov, t1), t1) + 0.5 * e("ldkc,ilad->akic", ovov, u)
    Wa = Wa - 0.5 * e("lckd,ilad->akic", ovov, t2)
    Wb = oovv.permute(2, 0, 3, 1) + e("kdac,id->akci", ovvv, t1) - e("kilc,la->akci", ooov, t1)
    Wb = Wb - e("lcki,la->akci", e("lckd,id->lcki", ovov, t1), t1) - 0.5 * e("lckd,ilda->akci", ovov, t2)
    P = P + e("akic,kjcb->ijab", Wa, u) - e("akci,kjcb->ijab", Wb, t2) - e("bkci,kjac->ijab", Wb, t2)
    return r1, P + P.permute(1, 0, 3, 2)


def _update(m, eo, ev, t1, t2):
    r1, r2 = _residual(m, t1, t2)
    return r1 / (eo[:, None] - ev[None, :]), r2 / _d2(eo, ev)


def _energy(m, t1, t2):
    L = 2 * m["ovov"] - m["ovov"].transpose(1, 3)
    return (torch.sum(L.permute(0, 2, 1, 3) * t2) + torch.einsum("kcld,kc,ld->", L, t1, t1)).item()


def _solve(m, eo, ev, t2):
    """Amplitudes converged well past the engine's criteria (DIIS over six vectors)."""
    t1 = torch.zeros_like(eo[:, None] * ev[None, :])
    xs, es = [], []
    for _ in range(80):
        n1, n2 = _update(m, eo, ev, t1, t2)
        x = torch.cat([n1.reshape(-1), n2.reshape(-1)])
        err = x - torch.cat([t1.reshape(-1), t2.reshape(-1)])
        rms = math.sqrt(torch.dot(err, err).item() / err.numel())
        xs, es = (xs + [x])[-6:], (es + [err])[-6:]
        if len(xs) > 1 and rms > 1e-14:
            k = len(xs)
            B = np.ones((k + 1, k + 1))
            B[k, k] = 0.0
            s = rms * rms * err.numel()
            for a in range(k):
                for b in range(k):
                    B[a, b] = torch.dot(es[a], es[b]).item() / s
            c = np.linalg.lstsq(B, np.eye(k + 1)[k], rcond=None)[0][:k]
            x = sum(float(ci) * xi for ci, xi in zip(c, xs))
        t1, t2 = x[:t1.numel()].reshape(t1.shape), x[t1.numel():].reshape(t2.shape)
        if rms < 1e-13:
            break
    return t1, t2


def _triples(m, eo, ev, t1, t2):
    """(T) energy, one triple i >= j >= k at a time (None where that takes too long)."""
    o, v = t1.shape
    if o ** 3 * v ** 4 > 1.1e14:
        return None
    vv = m["ovvv"].permute(0, 2, 1, 3).contiguous()      # vv[n][x, y, d] = (n y | x d)
    vt = vv.transpose(1, 2).contiguous()                 # vt[n][y, x, d]
    tp = t2.permute(1, 0, 3, 2).contiguous()             # tp[p, q][d, z] = t2[q, p, z, d]
    oo = m["ooov"].permute(1, 2, 0, 3).contiguous()      # oo[p, q][l, z] = (l p | q z)
    tn = t2.permute(0, 3, 2, 1).contiguous()             # tn[n][x, y, l] = t2[n, l, y, x]
    ts = tn.transpose(1, 2).contiguous()
    A = torch.cat([vv, -tn], 3).reshape(o, v * v, v + o)   # rows (x, y)
    As = torch.cat([vt, -ts], 3).reshape(o, v * v, v + o)  # rows (y, x)
    Bc = torch.cat([tp, oo], 2)                            # [p, q, v + o, z]
    del vv, vt, tp, oo, tn, ts
    ij = m["ovov"].permute(0, 2, 1, 3).contiguous()      # ij[i, j][a, b] = (ia|jb)
    De = ev[:, None, None] + ev[None, :, None] + ev[None, None, :]
    E = torch.zeros((), device=t1.device, dtype=F64)
    r = lambda x: x.reshape(v, v, v)  # noqa: E731
    for i in range(o):
        for j in range(i + 1):
            for k in range(j + 1):
                if i == j == k:
                    continue
                W = r(A[j] @ Bc[i, k]) + r(As[i] @ Bc[j, k])
                W += (r(As[i] @ Bc[k, j]) + r(A[k] @ Bc[i, j])).permute(0, 2, 1)
                W += (r(As[j] @ Bc[k, i]) + r(A[k] @ Bc[j, i])).permute(2, 0, 1)
                V = W + t1[i][:, None, None] * ij[j, k][None] + ij[i, k][:, None, :] * t1[j][None, :, None]
                V += ij[i, j][:, :, None] * t1[k][None, None, :]
                Z = 4 * V + V.permute(1, 2, 0) + V.permute(2, 0, 1)
                Z -= 2 * (V.permute(0, 2, 1) + V.permute(1, 0, 2) + V.permute(2, 1, 0))
                E += (2 - (i == j) - (j == k)) * torch.sum(W * Z / (eo[i] + eo[j] + eo[k] - De))
    return E.item()


def _scf_exact(case, S, H, b):
    n, no, Q = case["nbf"], case["ndocc"], case["naux"]
    w, U = np.linalg.eigh(S)
    X = (U / np.sqrt(w)) @ U.T
    hd = np.diag(H)
    F = 0.875 * S * (hd[:, None] + hd[None, :])
    np.fill_diagonal(F, hd)
    bm, fs, es, E = b.reshape(Q, n * n), [], [], 0.0
    for it in range(300):
        eps, C = np.linalg.eigh(X @ F @ X)
        Co = (X @ C)[:, :no]
        D = Co @ Co.T
        Z = (b.reshape(Q * n, n) @ Co).reshape(Q, n, no)
        F = H + 2 * ((bm @ D.reshape(-1)) @ bm).reshape(n, n) - np.tensordot(Z, Z, axes=([0, 2], [0, 2]))
        E = float(np.sum(D * (H + F)))
        err = X @ (F @ D @ S - S @ D @ F) @ X
        rms = float(np.sqrt(np.mean(err * err)))
        if rms < 1e-13:
            break
        fs, es = (fs + [F])[-8:], (es + [err])[-8:]
        if it > 3:
            k = len(fs)
            B = np.ones((k + 1, k + 1))
            B[k, k] = 0.0
            for x in range(k):
                for y in range(k):
                    B[x, y] = np.sum(es[x] * es[y]) / np.sum(err * err)
            c = np.linalg.lstsq(B, np.eye(k + 1)[k], rcond=None)[0][:k]
            F = sum(ci * fi for ci, fi in zip(c, fs))
    return E, np.linalg.eigvalsh(X @ F @ X)


def _mlp_exact(case, seed):
    h = case["hidden"]
    net = fermihip.Mlp(hidden=h, seed=seed)  # the initial weights are the handle's
    p = torch.tensor(net.get_params(), dtype=F64, requires_grad=True)
    net.close()
    X, T = (torch.tensor(x, dtype=F64) for x in _batch(case, seed))
    at = 0

    def take(*shape):
        nonlocal at
        k = int(np.prod(shape))
        at += k
        return p[at - k:at]

    W1 = take(h, 6).reshape(6, h)
    b1 = take(h)
    W2 = take(h, h).reshape(h, h)
    b2 = take(h)
    W3 = take(h, h).reshape(h, h)
    b3 = take(h)
    w4 = take(h)
    b4 = take(1)
    a = torch.tanh(X @ W1 + b1)
    a = torch.tanh(a @ W2 + b2)
    a = torch.tanh(a @ W3 + b3)
    loss = 0.5 * torch.mean((a @ w4 + b4 - T) ** 2)
    loss.backward()
    return {"loss": loss.item(), "grad": p.grad}


# ------------------------------------------------------------------ exact: Gaussian integrals
# Coulomb integrals by Hermite Gaussians (McMurchie and Davidson, 1978), vectorised over primitives.
def _carts(l):
    return [(x, y, l - x - y) for x in range(l, -1, -1) for y in range(l - x, -1, -1)]


def _odd(n):
    return math.prod(range(n, 0, -2)) if n > 0 else 1


def _solid(l):
    """Normalised real solid harmonics m = -l .. l over the Cartesian components, rows normalised
    relative to x^l."""
    terms = {0: [{(0, 0, 0): 1}],
             1: [{(1, 0, 0): 1}, {(0, 1, 0): 1}, {(0, 0, 1): 1}],
             2: [{(1, 1, 0): 1}, {(0, 1, 1): 1}, {(0, 0, 2): 2, (2, 0, 0): -1, (0, 2, 0): -1}, {(1, 0, 1): 1},
                 {(2, 0, 0): 1, (0, 2, 0): -1}],
             3: [{(2, 1, 0): 3, (0, 3, 0): -1}, {(1, 1, 1): 1}, {(0, 1, 2): 4, (2, 1, 0): -1, (0, 3, 0): -1},
                 {(0, 0, 3): 2, (2, 0, 1): -3, (0, 2, 1): -3}, {(1, 0, 2): 4, (3, 0, 0): -1, (1, 2, 0): -1},
                 {(2, 0, 1): 1, (0, 2, 1): -1}, {(3, 0, 0): 1, (1, 2, 0): -3}]}[l]
    cs = _carts(l)
    M = np.zeros((len(terms), len(cs)))
    for r, t in enumerate(terms):
        for k, c in t.items():
            M[r, cs.index(k)] = c
    ovl = np.array([[math.prod(_odd(x + y - 1) if (x + y) % 2 == 0 else 0 for x, y in zip(a, b)) for b in cs]
                    for a in cs]) / _odd(2 * l - 1)
    return M / np.sqrt(np.einsum("rc,cd,rd->r", M, ovl, M))[:, None]


def _contraction(s):
    """Coefficients over unnormalised x^l primitives that normalise the contracted function."""
    a, l = np.array(s["exps"], float), s["l"]
    c = np.array(s["coefs"], float) * (2 * a / math.pi) ** 0.75 * (4 * a) ** (l / 2) / math.sqrt(_odd(2 * l - 1))
    p = a[:, None] + a[None, :]
    return c / math.sqrt(np.sum(np.outer(c, c) * (math.pi / p) ** 1.5 * _odd(2 * l - 1) / (2 * p) ** l))


def _hermite(la, lb, a, b, A, B):
    p = a + b
    X = A - B
    E = {(0, 0, 0): torch.exp(-a * b / p * X * X)}
    z = torch.zeros_like(p)
    g = lambda i, j, t: E.get((i, j, t), z)  # noqa: E731
    for i in range(la + 1):
        for j in range(lb + 1):
            if i or j:
                for t in range(i + j + 1):
                    if i:
                        E[i, j, t] = 0.5 / p * g(i - 1, j, t - 1) - b / p * X * g(i - 1, j, t) + (t + 1) * g(i - 1, j, t + 1)
                    else:
                        E[i, j, t] = 0.5 / p * g(i, j - 1, t - 1) + a / p * X * g(i, j - 1, t) + (t + 1) * g(i, j - 1, t + 1)
    return E


def _tuv(L):
    return [(t, u, v) for t in range(L + 1) for u in range(L + 1 - t) for v in range(L + 1 - t - u)]


def _densities(shells, pairs):
    """Charge distributions of shell pairs (second shell None: the unit function), grouped by angular
    momenta: exponent, centre, Hermite coefficients [primitive pair, component pair, tuv], pair index."""
    out = {}
    for n, (i, j) in enumerate(pairs):
        out.setdefault((shells[i]["l"], shells[j]["l"] if j is not None else 0, j is None), []).append((n, i, j))
    groups = []
    for (la, lb, unit), members in out.items():
        rows = []
        for n, i, j in members:
            s, t = shells[i], shells[j] if j is not None else None
            for x, cx in zip(s["exps"], _contraction(s)):
                for y, cy in zip([0.0] if unit else t["exps"], [1.0] if unit else _contraction(t)):
                    rows.append([n, x, y, cx * cy, *s["center"], *(s["center"] if unit else t["center"])])
        R = torch.tensor(np.array(rows, float), device=dev())
        a, b = R[:, 1], R[:, 2]
        E = [_hermite(la, lb, a, b, R[:, 4 + d], R[:, 7 + d]) for d in range(3)]
        z = torch.zeros_like(a)
        H = torch.stack([torch.stack([torch.stack([
            E[0].get((ca[0], cb[0], t), z) * E[1].get((ca[1], cb[1], u), z) * E[2].get((ca[2], cb[2], v), z)
            for t, u, v in _tuv(la + lb)], -1) for cb in _carts(lb)], 1) for ca in _carts(la)], 1)
        Ma, Mb = (torch.tensor(_solid(l), device=dev()) for l in (la, lb))
        H = torch.einsum("nabh,xa,yb->nxyh", H, Ma, Mb) * R[:, 3, None, None, None]
        p = a + b
        C = (a[:, None] * R[:, 4:7] + b[:, None] * R[:, 7:10]) / p[:, None]
        groups.append({"l": la + lb, "p": p, "C": C, "H": H.reshape(len(rows), -1, H.shape[-1]),
                       "pair": R[:, 0].long(), "nc": (2 * la + 1, 2 * lb + 1)})
    return groups


def _boys(L, T):
    x = T.clamp(max=36.0)
    term = torch.full_like(x, 1.0 / (2 * L + 1))
    s = term.clone()
    for k in range(1, 160):
        term = term * (2 * x / (2 * L + 2 * k + 1))
        s = s + term
    F = [None] * (L + 1)
    ex = torch.exp(-x)
    F[L] = ex * s
    for n in range(L, 0, -1):
        F[n - 1] = (2 * x * F[n] + ex) / (2 * n - 1)
    big = T > 36.0
    if bool(big.any()):
        y = T.clamp(min=36.0)
        f = 0.5 * torch.sqrt(math.pi / y) * torch.erf(torch.sqrt(y))
        for n in range(L + 1):
            F[n] = torch.where(big, f, F[n])
            f = ((2 * n + 1) * f - torch.exp(-y)) / (2 * y)
    return F


def _coulomb(g, h):
    """[component pair of g, component pair of h] integrals of all primitive pairs, summed into contracted
    pairs: returns (pairs of g, pairs of h, block)."""
    L, tb, tk = g["l"] + h["l"], _tuv(g["l"]), _tuv(h["l"])
    ug, ig = torch.unique(g["pair"], return_inverse=True)
    uh, ih = torch.unique(h["pair"], return_inverse=True)
    out = torch.zeros(len(ug), len(uh), g["H"].shape[1], h["H"].shape[1], device=dev(), dtype=F64)
    sign = torch.tensor([(-1.0) ** sum(q) for q in tk], device=dev(), dtype=F64)
    step = max(1, int(2e7 / (len(h["p"]) * max(len(tb) * len(tk), 40))))
    for s in range(0, len(g["p"]), step):
        p, q = g["p"][s:s + step, None], h["p"][None, :]
        X, Y, Z = (g["C"][s:s + step, None, d] - h["C"][None, :, d] for d in range(3))
        al = p * q / (p + q)
        F = _boys(L, al * (X * X + Y * Y + Z * Z))
        lev = {}
        for n in range(L, -1, -1):
            new = {(0, 0, 0): (-2 * al) ** n * F[n]}
            for t, u, v in sorted(_tuv(L - n), key=sum)[1:]:
                if t:
                    r = X * lev[t - 1, u, v] + ((t - 1) * lev[t - 2, u, v] if t > 1 else 0.0)
                elif u:
                    r = Y * lev[t, u - 1, v] + ((u - 1) * lev[t, u - 2, v] if u > 1 else 0.0)
                else:
                    r = Z * lev[t, u, v - 1] + ((v - 1) * lev[t, u, v - 2] if v > 1 else 0.0)
                new[t, u, v] = r
            lev = new
        pre = 2 * math.pi ** 2.5 / (p * q * torch.sqrt(p + q))
        R = torch.stack([torch.stack([lev[tuple(x + y for x, y in zip(a, b))] for b in tk], -1) for a in tb], -2)
        K = torch.einsum("mnab,nkb->mnak", R * (pre[:, :, None, None] * sign), h["H"])
        acc = torch.zeros(K.shape[0], len(uh), *K.shape[2:], device=dev(), dtype=F64).index_add_(1, ih, K)
        out.index_add_(0, ig[s:s + step], torch.einsum("mja,mnak->mnjk", g["H"][s:s + step], acc))
    return ug, uh, out


def _eri(shells, others, three):
    off = np.concatenate([[0], np.cumsum([2 * s["l"] + 1 for s in shells])])
    n = int(off[-1])
    pairs = [(i, j) for i in range(len(shells)) for j in range(i + 1)]
    bra = _densities(shells, pairs)
    if three:
        aoff = np.concatenate([[0], np.cumsum([2 * s["l"] + 1 for s in others])])
        ket, kpairs, full = _densities(others, [(k, None) for k in range(len(others))]), None, (n, n, int(aoff[-1]))
    else:
        ket, kpairs, full = bra, pairs, (n, n, n, n)
    out = torch.zeros(*full, device=dev(), dtype=F64)

    def where(u, nc, plist, offs):
        """Function indices [pair, component pair] of the first and second function."""
        if plist is None:
            f = torch.tensor(offs[u.cpu().numpy()], device=dev())[:, None] + torch.arange(nc[0], device=dev())[None]
            return f, None
        ij = np.array([plist[k] for k in u.cpu().numpy()])
        a = torch.tensor(offs[ij[:, 0]], device=dev())[:, None, None] + torch.arange(nc[0], device=dev())[None, :, None]
        b = torch.tensor(offs[ij[:, 1]], device=dev())[:, None, None] + torch.arange(nc[1], device=dev())[None, None, :]
        shape = (len(ij), nc[0], nc[1])
        return a.expand(shape).reshape(len(ij), -1), b.expand(shape).reshape(len(ij), -1)

    for g in bra:
        for h in ket:
            ug, uh, blk = _coulomb(g, h)
            m, s = (x[:, None, :, None] for x in where(ug, g["nc"], pairs, off))
            c, d = where(uh, h["nc"], kpairs, aoff if three else off)
            c = c[None, :, None, :]
            if three:
                out[m, s, c] = blk
                out[s, m, c] = blk
            else:
                d = d[None, :, None, :]
                out[m, s, c, d] = blk
                out[s, m, c, d] = blk
                out[m, s, d, c] = blk
                out[s, m, d, c] = blk
    return out
