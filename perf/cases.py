"""Performance cases of the THC GW/RPA loop, through the public entry points of coqui_amd.

Every case is a dict of plain values.  `kind` selects what one pass runs:

  iteration  ThcGW.gw_iteration (chi0 -> W -> Sigma with the RPA energy), one system
  batch      ThcBatch.gw_iteration, several systems of uneven size in one captured graph
  chi0       ThcGW.pi: G(tau, k) -> chi0(tau, q)
  screen     ThcGW.tau_to_w, dyson_w (with the energy terms) and w_to_tau: chi0(tau) -> W(tau)
  sigma      ThcGW.sigma: G and W(tau) -> Sigma(tau, k)
  green      ThcGW.update_mu and dyson_g: Sigma -> chemical potential, G and density matrix
  fock       ThcGW.hf: density matrix -> THC Hartree-Fock potential
  qp         ThcGW.solve_qp: G0W0 quasiparticle energies of every state

and `form` the options the program has set on its context (FORMS).  Sizes follow the
benchmark's and the tests' systems: N_mu = 8 N_orb or so, k-grids of 2^3 to 4^3 points, IR
tables of 40, 60 and 80 tau points.
"""
import math

import numpy as np
import torch

from coqui_amd import IAFT, ThcBatch, ThcGW

BETA = 1000.0
TABLES = {40: "1e2.1e-15", 60: "1e3.1e-12", 80: "1e3.5e-18"}
#: form -> (flag 6 Dyson algorithm, flag 7 precision, flag 10 Hermitian G, flag 12 three-product mask)
FORMS = {
    "plain": (0, 0, 0, 0),             # the library's defaults: FP64, LU with partial pivoting
    "resolvent": (2, 0, 1, 0),         # FP64, (V^-1 - Pi)^-1 by Cholesky
    "mixed_resolvent": (2, 1, 1, 13),  # the benchmark's headline form: FP32 projections and k-grid transforms
    "mixed_batch": (2, 1, 1, 1),       # the benchmark's batched form
}


def listed():
    return [
        # A first run on a toy system, as in the smoke test: calls of a few dozen points, where
        # launches and host work count.
        {"name": "iteration-mu24", "kind": "iteration", "k1": 2, "k2": 2, "k3": 1, "no": 6, "nmu": 24, "nt": 40,
         "form": "plain"},
        # The smallest production-like system of the benchmark (2x2x2, N_mu = 200), default options.
        {"name": "iteration-mu200", "kind": "iteration", "k1": 2, "k2": 2, "k3": 2, "no": 26, "nmu": 200, "nt": 40,
         "form": "plain"},
        # A middle-sized system with an odd number of orbitals, in FP64 with the faster Dyson form.
        {"name": "iteration-mu328", "kind": "iteration", "k1": 3, "k2": 3, "k3": 3, "no": 41, "nmu": 328, "nt": 60,
         "form": "resolvent"},
        # The headline form on a 4x4x4 grid with the 80-point table: a whole iteration.
        {"name": "iteration-mu480", "kind": "iteration", "k1": 4, "k2": 4, "k3": 4, "no": 60, "nmu": 480, "nt": 80,
         "form": "mixed_resolvent"},
        # Many small materials at once: the batched graph, uneven sizes.
        {"name": "batch-6", "kind": "batch", "n": 6, "no_lo": 16, "no_hi": 40, "k_hi": 3, "nt": 60,
         "form": "mixed_batch"},
        # chi0 of a 4x4x4 system in FP64, ragged N_mu.
        {"name": "chi0-mu405", "kind": "chi0", "k1": 4, "k2": 4, "k3": 4, "no": 52, "nmu": 405, "nt": 60,
         "form": "plain"},
        # W with the default pivoted LU at N_mu = 800, as the plain form of the benchmark has it.
        {"name": "screen-mu800", "kind": "screen", "k1": 2, "k2": 2, "k3": 1, "no": 52, "nmu": 800, "nt": 80,
         "form": "plain"},
        # W at the benchmark's N_mu = 1600 with its fastest FP64 Dyson form: the largest matrices.
        {"name": "screen-mu1600", "kind": "screen", "k1": 2, "k2": 2, "k3": 1, "no": 104, "nmu": 1600, "nt": 80,
         "form": "mixed_resolvent"},
        # Sigma of a 4x4x4 system in FP64 with Hermitian G.
        {"name": "sigma-mu405", "kind": "sigma", "k1": 4, "k2": 4, "k3": 4, "no": 52, "nmu": 405, "nt": 60,
         "form": "resolvent"},
        # The G side of a self-consistent iteration: chemical potential search and Dyson for G.
        {"name": "green-no78", "kind": "green", "k1": 4, "k2": 4, "k3": 4, "no": 78, "nmu": 16, "nt": 80,
         "form": "plain"},
        # The Hartree-Fock part of a self-consistent iteration.
        {"name": "fock-mu800", "kind": "fock", "k1": 4, "k2": 4, "k3": 4, "no": 52, "nmu": 800, "nt": 40,
         "form": "plain"},
        # Quasiparticle energies of every state after a G0W0 iteration.
        {"name": "qp-no104", "kind": "qp", "k1": 4, "k2": 4, "k3": 4, "no": 104, "nmu": 16, "nt": 80,
         "form": "plain"},
    ]


def draw(rng):
    """One more case of the listed ranges: any kind, odd sizes, sizes spread over their logarithm."""
    kind = rng.choice(["iteration", "iteration", "iteration", "batch", "chi0", "screen", "screen", "sigma", "green",
                       "fock", "qp"])

    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    nt = rng.choice([40, 60, 80])
    if kind == "batch":
        lo = rng.randint(12, 24)
        return {"kind": kind, "n": rng.randint(2, 6), "no_lo": lo, "no_hi": lo + rng.randint(2, 16),
                "k_hi": rng.choice([2, 3]), "nt": 60, "form": "mixed_batch"}
    grids = [(2, 2, 1), (2, 2, 2), (3, 3, 1), (3, 3, 3), (4, 4, 4)]
    top = {"iteration": {4: 640, 8: 600, 9: 560, 27: 440, 64: 400}, "chi0": {4: 800, 8: 800, 9: 800, 27: 560, 64: 405},
           "sigma": {4: 800, 8: 800, 9: 800, 27: 560, 64: 405}, "screen": {2: 1600, 4: 1400, 8: 900}}
    if kind == "screen":
        grids = [(2, 1, 1), (2, 2, 1), (2, 2, 2)]
    k = rng.choice(grids)
    nk = k[0] * k[1] * k[2]
    c = {"kind": kind, "k1": k[0], "k2": k[1], "k3": k[2]}
    if kind in top:
        nmu = log_int(24 if kind == "iteration" else 150, top[kind][nk])
        form = rng.choice(["plain", "resolvent", "mixed_resolvent"])
        if kind == "screen" and form == "plain":
            nmu = min(nmu, 900)
        c.update(no=max(4, nmu // 8 + rng.randint(-2, 3)), nmu=nmu, nt=nt, form=form)
    elif kind == "fock":
        nmu = log_int(100, 800)
        c.update(no=max(8, nmu // 16 + rng.randint(0, 9)), nmu=nmu, nt=40, form="plain")
    else:  # green, qp: no auxiliary basis in the call
        c.update(no=log_int(16, 78 if kind == "green" else 104), nmu=16, nt=nt, form="plain")
    return c


# ---------------------------------------------------------------- inputs
def _gauss(g, *shape):
    a = torch.randn(shape + (2,), generator=g, device="cuda", dtype=torch.float64)
    return torch.view_as_complex(a) / math.sqrt(2.0)


def _basis(g, nk, no):
    """Random unitary C(k) and sorted energies E(k) in [-1, 1] Ha; H(k) = C E C^H."""
    q, _ = torch.linalg.qr(_gauss(g, nk, no, no))
    e = torch.rand((nk, no), generator=g, device="cuda", dtype=torch.float64) * 2.0 - 1.0
    return q.contiguous(), torch.sort(e, dim=1).values.contiguous()


def _iaft(c):
    return IAFT.from_table(BETA, TABLES[c["nt"]])


def _system(kgrid, no, nmu, ia, seed, with_v=True):
    """Context-free inputs of one system: C, E, X, V on the GPU (coqui_amd.system's distributions)."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) & 0x7FFFFFFFFFFF)
    nk = kgrid[0] * kgrid[1] * kgrid[2]
    C, E = _basis(g, nk, no)
    X = _gauss(g, nk, nmu, no)
    X = X / torch.linalg.vector_norm(X, dim=2, keepdim=True)
    V = None
    if with_v:
        V = torch.empty((nk, nmu, nmu), dtype=torch.complex128, device="cuda")
        for k in range(nk):  # V = Z Z^H / N_mu
            Z = _gauss(g, nmu, nmu)
            V[k] = Z @ Z.conj().T / nmu
    return g, C, E, X.contiguous(), V


def _self_energy(g, ctx, nk, no):
    """A causal Hermitian Sigma(tau, k): the Green's function of other levels, scaled to 0.05 Ha."""
    C2, E2 = _basis(g, nk, no)
    return 0.05 * ctx.update_G(C2, 1.5 * E2, 0.0)


def _matrix(C, E):
    return ((C * E[:, None, :]) @ C.conj().transpose(1, 2)).contiguous()


def _set_form(ctx, form):
    algo, prec, herm, _ = FORMS[form]
    ctx.set_flag(6, algo)
    ctx.set_flag(7, prec)
    ctx.set_flag(10, herm)


def _batch_specs(c, seed):
    """Systems of a batch: N_orb, N_mu = 8 N_orb and the k-grid follow from the case alone."""
    r = np.random.default_rng([c["n"], c["no_lo"], c["no_hi"], c["k_hi"]])
    out = []
    for _ in range(c["n"]):
        no, k = int(r.integers(c["no_lo"], c["no_hi"] + 1)), int(r.integers(2, c["k_hi"] + 1))
        out.append(((k, k, k), no, 8 * no))
    return out


def prepare(case, seed):
    c = dict(case)
    ia = _iaft(c)
    kind = c["kind"]
    st = {"kind": kind, "mask": FORMS[c["form"]][3]}
    if kind == "batch":
        st.update(ctxs=[], G=[], X=[], V=[], S=[], W=[])
        for i, (kg, no, nmu) in enumerate(_batch_specs(c, seed)):
            _, C, E, X, V = _system(kg, no, nmu, ia, seed * 64 + i)
            ctx = ThcGW(kg, no, nmu, ia)
            _set_form(ctx, c["form"])
            st["ctxs"].append(ctx)
            st["G"].append(ctx.update_G(C, E, 0.0))
            st["X"].append(X)
            st["V"].append(V)
            st["S"].append(torch.empty(ctx._g(), dtype=torch.complex128, device="cuda"))
            st["W"].append(torch.empty(ctx._wqt(), dtype=torch.complex128, device="cuda"))
        st["batch"] = ThcBatch(st["ctxs"], lanes=4)
        return st
    kg, no, nmu = (c["k1"], c["k2"], c["k3"]), c["no"], c["nmu"]
    nk = kg[0] * kg[1] * kg[2]
    ctx = ThcGW(kg, no, nmu, ia)
    _set_form(ctx, c["form"])
    g, C, E, X, V = _system(kg, no, nmu, ia, seed, with_v=kind not in ("chi0", "green", "qp"))
    st.update(ctx=ctx, C=C, E=E, X=X, V=V)
    new = lambda shape: torch.empty(shape, dtype=torch.complex128, device="cuda")  # noqa: E731
    if kind in ("iteration", "chi0", "screen", "sigma"):
        st["G"] = ctx.update_G(C, E, 0.0)
    if kind == "iteration":
        st.update(S=new(ctx._g()), W=new(ctx._wqt()))
    elif kind == "chi0":
        st["P"] = new(ctx._pit())
    elif kind == "screen":  # chi0 of the system itself, in the array that W(tau) goes to afterwards
        st["P"] = _chi0(st["G"], X, kg, ia)
        st.update(Pw=new(ctx._piw()), W=new(ctx._wqt()))
    elif kind == "sigma":  # a Hermitian W(q, tau) that decays from tau = 0 to beta / 2
        st["W"] = new(ctx._wqt())
        tau = torch.from_numpy(ia.tau[: ia.nt_half].copy()).cuda()
        for q in range(nk):
            B = _gauss(g, nmu, nmu)
            B = -(B @ B.conj().T) / nmu
            for t in range(ia.nt_half):
                st["W"][q, t] = B * torch.exp(-tau[t] / (40.0 + q)) / (1.0 + t)
        st["S"] = new(ctx._g())
    elif kind == "green":
        st["F"] = _matrix(C, E)[None].contiguous()
        st["Sigma"] = _self_energy(g, ctx, nk, no)
        st["target"] = 0.52 * 2.0 * no
        st["G"] = new(ctx._g())
    elif kind == "fock":
        f = 1.0 / (torch.exp(BETA / 20.0 * E) + 1.0)
        st["Dm"] = _matrix(C, f)[None].contiguous()
        st["F"] = new(ctx._kij())
    elif kind == "qp":
        st["Sigma"] = _self_energy(g, ctx, nk, no)
        st["H"] = _matrix(C, E)
        st["E0"] = E.cpu().numpy()
    return st


def run(st):
    kind = st["kind"]
    ctx = st["ctxs"][0] if kind == "batch" else st["ctx"]
    ctx.set_flag(12, st["mask"])  # an option of the process, not of the context
    if kind == "batch":
        ec = st["batch"].gw_iteration(st["G"], st["X"], st["V"], st["S"], st["W"])
        return {"Sigma": st["S"], "W": st["W"], "Ec": np.array(ec)}
    if kind == "iteration":
        S, W, ec = ctx.gw_iteration(st["G"], st["X"], st["V"], Sigma=st["S"], W_qt=st["W"])
        return {"Sigma": S, "W": W, "Ec": ec}
    if kind == "chi0":
        return ctx.pi(st["G"], st["X"], out=st["P"])
    if kind == "screen":
        Pw = ctx.tau_to_w(st["P"], out=st["Pw"])
        tr, ld = ctx.dyson_w(Pw, st["V"], with_terms=True)
        return {"W": ctx.w_to_tau(Pw, out=st["W"]), "trace": tr, "logdet": ld}
    if kind == "sigma":
        return ctx.sigma(st["G"], st["W"], st["X"], out=st["S"])
    if kind == "green":
        mu, nel = ctx.update_mu(st["F"], st["Sigma"], st["target"], 0.0)
        G, Dm = ctx.dyson_g(st["F"], st["Sigma"], mu, out=st["G"])
        return {"mu": mu, "nelec": nel, "G": G, "Dm": Dm}
    if kind == "fock":
        return ctx.hf(st["Dm"], st["X"], st["V"], out=st["F"])
    return ctx.solve_qp(st["Sigma"], st["C"], st["H"], st["E0"])


# ---------------------------------------------------------------- the work of one pass
def work(case):
    """Bytes: every input read once and every output written once.  Flops: projections (two
    products), separable k-grid transforms, tau <-> iW products, Dyson at the selected form's
    count (LU with two solves 56/3 n^3, resolvent 4 n^3 real flops) and the back-projection."""
    c = dict(case)
    ia = _iaft(c)
    nt, nth, nwh, nwf = ia.nt, ia.nt_half, ia.nw_half, ia.nw_f
    if c["kind"] == "batch":
        parts = [work(dict(kind="iteration", k1=k[0], k2=k[1], k3=k[2], no=no, nmu=nmu, nt=c["nt"], form=c["form"]))
                 for k, no, nmu in _batch_specs(c, 0)]
        return {m: float(sum(p[m] for p in parts)) for m in ("bytes", "flops")}
    k1, k2, k3, no, n = c["k1"], c["k2"], c["k3"], c["no"], c["nmu"]
    nk, M, kind = k1 * k2 * k3, float(n) * n, c["kind"]
    herm = FORMS[c["form"]][2]
    G, X, V, W = nt * nk * no * no, nk * n * no, nk * M, nk * nth * M
    # a Hermitian G needs half of the second product of X G X^H and of the first of X^H S X
    proj = 8.0 * nk * (n * no * no + M * no * (0.5 if herm else 1.0))
    back = 8.0 * nk * (n * no * no + M * no * (0.5 if herm else 1.0))
    fft = 8.0 * nk * M * (k1 + k2 + k3)
    chi0 = nt * proj + nth * (3 * fft + 8 * nk * M)
    ft = 4.0 * nwh * nth * nk * M  # the folded tables are real
    dyson = nwh * nk * M * n * (56.0 / 3.0 if FORMS[c["form"]][0] == 0 else 4.0)
    sigma = nt * (proj + back) + nth * (5 * fft + 16 * nk * M)
    if kind == "iteration":
        return {"bytes": 16.0 * (G + X + V + G + W), "flops": chi0 + 2 * ft + dyson + sigma}
    if kind == "chi0":
        return {"bytes": 16.0 * (G + X + W), "flops": chi0}
    if kind == "screen":
        return {"bytes": 16.0 * (2 * W + V), "flops": 2 * ft + dyson}
    if kind == "sigma":
        return {"bytes": 16.0 * (2 * G + X + W), "flops": sigma}
    if kind == "fock":
        return {"bytes": 16.0 * (2 * nk * no * no + X + V), "flops": proj + back + 3 * fft + 8 * nk * M}
    if kind == "green":  # one inverse per (n, k) for G and one per trial of mu (about 30 halvings)
        inv = 8.0 * nwf * nk * float(no) ** 3
        return {"bytes": 16.0 * (2 * G + 2 * nk * no * no), "flops": 31 * inv + 16.0 * nwf * nt * nk * no * no}
    # qp: MO diagonals of Sigma(tau) and Vhf, Sigma to the nfit = 18 frequencies; the roots come on top
    return {"bytes": 16.0 * (G + 2 * nk * no * no) + 16.0 * nk * no,
            "flops": 8.0 * (nt + 1) * nk * float(no) ** 3 + 8.0 * 18 * nt * nk * no}


# ---------------------------------------------------------------- 64-bit values by plain torch
def _dft(kgrid):
    """f_Rk = exp(-i k.R) / N_k and f_kR = exp(i k.R) on the C-order grid."""
    F = torch.ones((1, 1), dtype=torch.complex128, device="cuda")
    for n in kgrid:
        i = torch.arange(n, device="cuda", dtype=torch.float64)
        f = torch.polar(torch.ones((n, n), device="cuda", dtype=torch.float64), -2.0 * math.pi * i[:, None] * i / n)
        F = torch.kron(F, f)
    return F / F.shape[0], F.conj().contiguous()


def _project(X, G):
    return (X @ G) @ X.conj().transpose(1, 2).contiguous()


def _tables(ia):
    """T+ (iW_n <- tau_i) and T- (tau_i <- iW_n), particle-hole folded, and the raw bosonic tau <- iW."""
    s2 = math.sqrt(2.0)
    T, Ti = ia.Twt_bb * (ia.beta / s2), ia.Ttw_bb * (s2 / ia.beta)
    nwb, nt, nth, nwh = ia.nw_b, ia.nt, ia.nt_half, ia.nw_half
    Tp = np.array([[T[nwb // 2 + n, i] + (T[nwb // 2 + n, nt - 1 - i] if nt - 1 - i != i else 0) for i in range(nth)]
                   for n in range(nwh)])
    Tm = np.array([[Ti[i, nwb // 2 + n] + (Ti[i, nwb // 2 - n] if n else 0) for n in range(nwh)] for i in range(nth)])
    return torch.from_numpy(Tp).cuda(), torch.from_numpy(Tm).cuda(), Ti


def _chi0(G, X, kgrid, ia):
    nk, n = X.shape[0], X.shape[1]
    fRk, fkR = _dft(kgrid)
    P = torch.empty((ia.nt_half, nk, n, n), dtype=torch.complex128, device="cuda")
    for i in range(ia.nt_half):
        Gp = fRk @ _project(X, G[i, 0]).reshape(nk, -1)
        Gn = fRk @ _project(X, G[ia.nt - 1 - i, 0]).reshape(nk, -1)
        P[i] = (fkR @ (-2.0 * Gp * Gn.conj())).reshape(nk, n, n)
    return P


def _screen(P, V, ia):
    """W - V on tau in the (q, tau) order, Tr(V Pi) and ln|Re det(I - V Pi)| per (n, q)."""
    Tp, Tm, _ = _tables(ia)
    nth, nk, n, _ = P.shape
    Pw = (Tp @ P.reshape(nth, -1)).reshape(ia.nw_half, nk, n, n)
    eye = torch.eye(n, dtype=torch.complex128, device="cuda")
    tr = torch.empty((ia.nw_half, nk), dtype=torch.complex128, device="cuda")
    ld = torch.empty((ia.nw_half, nk), dtype=torch.float64, device="cuda")
    for w in range(ia.nw_half):
        B = V @ Pw[w]
        tr[w] = torch.diagonal(B, dim1=1, dim2=2).sum(1)
        LU, piv = torch.linalg.lu_factor(eye - B)
        d = torch.diagonal(LU, dim1=1, dim2=2)
        ld[w] = d.abs().log().sum(1) + (d / d.abs()).prod(1).real.abs().log()
        Pw[w] = torch.linalg.lu_solve(LU, piv, V) - V
    W = torch.empty((nk, nth, n, n), dtype=torch.complex128, device="cuda")
    for q in range(nk):
        W[q] = (Tm @ Pw[:, q].reshape(ia.nw_half, -1)).reshape(nth, n, n)
    return W, tr, ld


def _ec(tr, ld, ia):
    Ti = _tables(ia)[2]
    v = (tr + ld).sum(1).cpu().numpy()
    ew = np.zeros(ia.nw_b, complex)
    for n in range(ia.nw_half):
        ew[ia.nw_b // 2 + n] = v[n]
        ew[ia.nw_b // 2 - n] = v[n]
    return float((ia.T_beta_t_ff @ (Ti @ ew)).real / (2.0 * tr.shape[1]))


def _conv(A, B, kgrid):
    """-(1/N_k) sum_q A(k - q) o B(q) for (nk, n, n) matrices."""
    fRk, fkR = _dft(kgrid)
    nk = A.shape[0]
    return (fkR @ (-(fRk @ A.reshape(nk, -1)) * (fRk @ B.reshape(nk, -1)))).reshape(A.shape)


def _back(X, S):
    return X.conj().transpose(1, 2).contiguous() @ (S @ X)


def _sigma(G, W, X, kgrid, ia):
    S = torch.empty_like(G)
    for i in range(ia.nt_half):
        for t in {i, ia.nt - 1 - i}:
            A = _back(X, _conv(_project(X, G[t, 0]), W[:, i], kgrid))
            S[t, 0] = 0.5 * (A + A.conj().transpose(1, 2))
    return S


def _iteration_exact(G, X, V, kgrid, ia):
    W, tr, ld = _screen(_chi0(G, X, kgrid, ia), V, ia)
    return _sigma(G, W, X, kgrid, ia), W, _ec(tr, ld, ia)


def _inverse(A):
    """Inverses of many small matrices: Gauss-Jordan with partial pivoting on [A | I], all at once
    (torch.linalg.inv takes seconds for a few thousand of them)."""
    b, n, _ = A.shape
    eye = torch.eye(n, dtype=A.dtype, device=A.device)
    M = torch.cat([A, eye.expand(b, n, n)], 2)
    at = torch.arange(b, device=A.device)
    for j in range(n):
        p = j + M[:, j:, j].abs().argmax(1)
        row = M[at, p]
        M[at, p] = M[:, j]
        row = row / row[:, j, None]
        M[:, j] = row
        col = M[:, :, j].clone()
        col[:, j] = 0.0
        M -= col[:, :, None] * row[:, None, :]
    return M[:, :, n:].contiguous()


def _green_exact(st, ia):
    """mu by the search the entry point documents (a bracket in steps of 0.2 Ha, then halving until
    N is within 1e-9; in a gap of the spectrum no other mu is the same one), then G and Dm."""
    s2 = math.sqrt(2.0)
    Twt = torch.from_numpy(ia.Twt_ff * (ia.beta / s2)).cuda()
    Ttw = torch.from_numpy(ia.Ttw_ff * (s2 / ia.beta)).cuda()
    Tb = torch.from_numpy(ia.T_beta_t_ff).cuda()
    F, Sig = st["F"][0], st["Sigma"]
    nt, nk, no = ia.nt, F.shape[0], F.shape[1]
    Sw = (Twt @ Sig.reshape(nt, -1)).reshape(ia.nw_f, nk, no, no)
    wn = torch.from_numpy(ia.wn_mesh_f * math.pi / ia.beta).cuda()
    eye = torch.eye(no, dtype=torch.complex128, device="cuda")

    def inverse(mu):
        return _inverse(((mu + 1j * wn)[:, None, None, None] * eye - F - Sw).reshape(-1, no, no)).reshape(Sw.shape)

    def nelec(mu):
        t = torch.diagonal(inverse(mu), dim1=2, dim2=3).sum((1, 2)) / nk
        return float(-2.0 * (Tb @ (Ttw @ t)).real)

    target, mu = st["target"], 0.0
    n = nelec(mu)
    if abs(n - target) >= 1e-9:
        step = -0.2 if n >= target else 0.2
        far = mu + step
        while (nelec(far) > target) if step < 0 else (nelec(far) < target):
            far += step
        lo, hi = min(mu, far), max(mu, far)
        for _ in range(200):
            mu = 0.5 * (lo + hi)
            n = nelec(mu)
            if abs(n - target) < 1e-9:
                break
            lo, hi = (lo, mu) if n >= target else (mu, hi)
    G = (Ttw @ inverse(mu).reshape(ia.nw_f, -1)).reshape(nt, 1, nk, no, no)
    Dm = -(Tb @ G.reshape(nt, -1)).reshape(1, nk, no, no)
    return {"mu": mu, "nelec": n, "G": G, "Dm": Dm}


def exact(case, seed):
    c = dict(case)
    if c["kind"] == "qp":  # continued fractions and bisection in extended precision: no plain 64-bit value
        return None
    if c["kind"] not in ("batch", "green", "fock"):
        # batched factorisations of plain torch take seconds per 1e12 of n^3 matrices
        nk = c["k1"] * c["k2"] * c["k3"]
        if c["kind"] in ("iteration", "screen") and nk * c["nt"] * float(c["nmu"]) ** 3 > 2.0e11:
            return None
    ia = _iaft(c)
    st = prepare(case, seed)
    if c["kind"] == "batch":
        got = [_iteration_exact(st["G"][i], st["X"][i], st["V"][i], k, ia)
               for i, (k, _, _) in enumerate(_batch_specs(c, seed))]
        return {"Sigma": [x[0] for x in got], "W": [x[1] for x in got], "Ec": np.array([x[2] for x in got])}
    kg = (c["k1"], c["k2"], c["k3"])
    if c["kind"] == "iteration":
        S, W, ec = _iteration_exact(st["G"], st["X"], st["V"], kg, ia)
        return {"Sigma": S, "W": W, "Ec": ec}
    if c["kind"] == "chi0":
        return _chi0(st["G"], st["X"], kg, ia)
    if c["kind"] == "screen":
        W, tr, ld = _screen(st["P"], st["V"], ia)
        return {"W": W, "trace": tr.reshape(-1).cpu().numpy(), "logdet": ld.reshape(-1).cpu().numpy()}
    if c["kind"] == "sigma":
        return _sigma(st["G"], st["W"], st["X"], kg, ia)
    if c["kind"] == "green":
        return _green_exact(st, ia)
    X, V, Dm = st["X"], st["V"], st["Dm"][0]
    D = _project(X, Dm)
    S = _conv(D, V, kg)
    d = 2.0 * torch.diagonal(D, dim1=1, dim2=2).mean(0)
    S = S + torch.diag_embed(V[0] @ d)
    return _back(X, S)[None]
