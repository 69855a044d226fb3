"""Timing cases of the OVERLAP fermion hot path: what programs have this library do, from the
smallest calls to the largest workload.

A program that uses the library either evolves mode functions that stay on the device (leapfrog
steps of one lattice or of an ensemble, read back between measurements), applies one operator to
all of them, calls the reference's single-mode operators with host arrays, or evolves and measures
the gauge field.  Lattices, mode counts, link and E-field widths, degrees and flux quanta are those
of overlap_amd/configs.py, the tests and bench.py, and odd ones between them.

Kinds (`kind` of a case):
  leapfrog  ovl_fermion_update of a resident context, then every mode function of both fields and the
            links are read back
  observed  ovl_fermion_update_observed: leapfrog steps with the currents and dN_CS/dt after each
  apply     one overlap operator on every mode, read back
  ensemble  ovl_fermion_update of many uneven lattices in one context, modes read back
  dropin_wilson, dropin_overlap   WilsonEvoOperator::Compute / OverlapOperator::Compute with host arrays
  gauge     link and E-field evolution with the observables after every step
  obs       ovl_observables_noalloc on device tensors, queued on torch's stream
"""
from __future__ import annotations

import math

import numpy as np
import torch

from overlap_amd import ovl

DEV = "cuda"
OVERLAP_SIGMA = {2: 0.3, 3: 0.25}  # link widths of the SU(2) and SU(3) configurations
E_SIGMA = 0.1


def listed():
    return [
        # a gauge monitor inside a device program: seven observables of a small SU(2) lattice
        dict(name="obs_su2_8", kind="obs", nc=2, n0=8, n1=8, n2=8),
        # the smallest evolution: SU(2) Wilson fermions, 16 modes on 8^3, 100 steps with moving links
        dict(name="wilson_su2_8", kind="leapfrog", fermion="wilson", nc=2, n0=8, n1=8, n2=8, modes=16, prec="fp64",
             steps=100, dt=0.05, gauge="links", nb=0),
        # SU(3) Wilson fermions on a ragged lattice with flux, FP32 spinors, E and links both moving
        dict(name="wilson_su3_ragged_fp32", kind="leapfrog", fermion="wilson", nc=3, n0=15, n1=12, n2=10, modes=24,
             prec="fp32", steps=200, dt=0.05, gauge="full", nb=4),
        # a bandwidth-bound Wilson evolution in FP64 between two measurements
        dict(name="wilson_su3_24_fp64", kind="leapfrog", fermion="wilson", nc=3, n0=24, n1=24, n2=24, modes=64,
             prec="fp64", steps=200, dt=0.05, gauge="links", nb=4),
        # SU(2) overlap fermions, the 16^3 configuration with its 64 modes in the mixed form
        dict(name="overlap_su2_16_mixed", kind="leapfrog", fermion="overlap", nc=2, n0=16, n1=16, n2=16, modes=64,
             prec="mixed", steps=4, dt=0.02, gauge="links", nb=0, degree=256),
        # one plain FP64 overlap operator on a ragged SU(3) lattice with a partly filled mode block
        dict(name="overlap_su3_ragged_fp64", kind="apply", nc=3, n0=11, n1=14, n2=9, modes=40, prec="fp64", nb=2,
             degree=128),
        # the largest: SU(3) overlap fermions on 24^3 in a magnetic field, 256 modes, degree 384,
        # currents and dN_CS/dt after every step
        dict(name="overlap_su3_24_observed", kind="observed", nc=3, n0=24, n1=24, n2=24, modes=256, prec="mixed",
             relax=2, steps=2, dt=0.02, nb=8, degree=384),
        # uneven SU(2) overlap systems evolved together
        dict(name="ensemble_su2_mixed", kind="ensemble", nc=2, sizes="16 12 8 12 20 10", modes=32, prec="mixed", steps=2,
             dt=0.02, degree=256),
        # the reference's Wilson operator on one host mode
        dict(name="dropin_wilson_su3_24", kind="dropin_wilson", nc=3, n0=24, n1=24, n2=24),
        # the reference's overlap operator (25-pole Zolotarev, multi-shift CG) on one host mode
        dict(name="dropin_overlap_su2_12", kind="dropin_overlap", nc=2, n0=12, n1=12, n2=12),
        # the reference's own overlap step: Zolotarev sign with Ritz bounds before each half step
        dict(name="reference_step_su2_8", kind="leapfrog", fermion="overlap", nc=2, n0=8, n1=8, n2=8, modes=16,
             prec="zolotarev", steps=1, dt=0.02, gauge="links", nb=0),
        # Yang-Mills evolution of an SU(3) configuration, measured after every step
        dict(name="gauge_su3_24", kind="gauge", nc=3, n0=24, n1=24, n2=24, steps=5, dt=0.05),
    ]


def draw(rng):
    kind = rng.choice(["obs", "wilson", "wilson", "overlap", "apply", "observed", "ensemble", "dropin_wilson",
                       "dropin_overlap", "reference", "gauge"])
    nc = rng.choice([2, 3])

    def lattice(lo, hi):
        return {f"n{k}": rng.randint(lo, hi) for k in range(3)}

    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    if kind == "obs":
        return dict(kind="obs", nc=nc, **lattice(6, 32))
    if kind == "wilson":
        return dict(kind="leapfrog", fermion="wilson", nc=nc, **lattice(6, 20), modes=log_int(4, 64),
                    prec=rng.choice(["fp64", "fp32"]), steps=rng.randint(20, 200), dt=0.05,
                    gauge=rng.choice(["frozen", "links", "full"]), nb=rng.randint(0, 4))
    if kind == "overlap":
        return dict(kind="leapfrog", fermion="overlap", nc=nc, **lattice(6, 16), modes=log_int(4, 64),
                    prec=rng.choice(["mixed", "mixed", "fp64"]), steps=rng.randint(1, 3), dt=0.02,
                    gauge=rng.choice(["frozen", "links"]), nb=rng.randint(0, 6), degree=rng.choice([128, 256, 384]))
    if kind == "apply":
        return dict(kind="apply", nc=nc, **lattice(6, 18), modes=log_int(4, 128),
                    prec=rng.choice(["mixed", "fp64", "fp32"]), nb=rng.randint(0, 8), degree=rng.choice([128, 256]))
    if kind == "observed":
        return dict(kind="observed", nc=nc, **lattice(8, 24), modes=log_int(16, 160), prec="mixed",
                    relax=rng.choice([0, 2]), steps=1, dt=0.02, nb=rng.randint(0, 8), degree=rng.choice([256, 384]))
    if kind == "ensemble":
        return dict(kind="ensemble", nc=nc, sizes=" ".join(str(rng.randint(6, 14)) for _ in range(rng.randint(2, 6))),
                    modes=log_int(8, 48), prec=rng.choice(["mixed", "fp64"]), steps=1, dt=0.02,
                    degree=rng.choice([128, 256]))
    if kind == "dropin_wilson":
        return dict(kind="dropin_wilson", nc=nc, **lattice(8, 32))
    if kind == "dropin_overlap":
        return dict(kind="dropin_overlap", nc=nc, **lattice(6, 14))
    if kind == "reference":
        return dict(kind="leapfrog", fermion="overlap", nc=nc, **lattice(6, 9), modes=log_int(2, 16), prec="zolotarev",
                    steps=1, dt=0.02, gauge="links", nb=0)
    return dict(kind="gauge", nc=nc, **lattice(8, 28), steps=rng.randint(1, 8), dt=0.05)


# ---------------------------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------------------------
def _volume(n):
    return n[0] * n[1] * n[2]


def _dims(case):
    return (case["n0"], case["n1"], case["n2"])


def _link_inputs(nc, n, g):
    """SU(2): 4 reals per link; SU(3): 9 complex per link, column-major, exp(i eps n.lambda/2)."""
    V = _volume(n)
    eps = g.normal(0.0, OVERLAP_SIGMA[nc], size=(V, 3))
    v = g.normal(size=(V, 3, nc * nc - 1))
    v /= np.linalg.norm(v, axis=-1, keepdims=True)
    if nc == 2:
        u = np.empty((V, 3, 4))
        u[..., :3] = np.sin(eps / 2)[..., None] * v
        u[..., 3] = np.cos(eps / 2)
        return u.reshape(-1)
    a = 0.5 * eps[..., None] * v
    h = np.zeros((V, 3, 3, 3), complex)
    h[..., 0, 1] = a[..., 0] - 1j * a[..., 1]
    h[..., 0, 2] = a[..., 3] - 1j * a[..., 4]
    h[..., 1, 2] = a[..., 5] - 1j * a[..., 6]
    h += np.conj(np.swapaxes(h, -1, -2))
    r3 = a[..., 7] / math.sqrt(3.0)
    h[..., 0, 0], h[..., 1, 1], h[..., 2, 2] = a[..., 2] + r3, -a[..., 2] + r3, -2 * r3
    w, q = np.linalg.eigh(h)
    m = np.einsum("...ij,...j,...kj->...ki", q, np.exp(1j * w), q.conj())  # transposed: column-major
    return np.ascontiguousarray(m).reshape(-1).view(np.float64)


def _efield_inputs(nc, n, g):
    return g.normal(0.0, E_SIGMA, size=_volume(n) * 3 * (nc * nc - 1))


def _modes_inputs(nc, n, modes, seed):
    """Unit-norm complex Gaussian mode functions (modes, V nc 4), drawn on the GPU."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    z = torch.randn((modes, _volume(n) * nc * 4, 2), generator=g, device=DEV, dtype=torch.float64)
    z /= z.reshape(modes, -1).norm(dim=1)[:, None, None]
    return torch.view_as_complex(z)


def _gauge_inputs(case, seed):
    g = np.random.Generator(np.random.Philox(seed))
    n = _dims(case)
    return _link_inputs(case["nc"], n, g), _efield_inputs(case["nc"], n, g)


def _masses(case):
    """(m_fermion, m_dw) of the case's fermions."""
    if case.get("fermion") == "wilson":
        return (0.1 if case["nc"] == 2 else 0.0), 0.0
    if case["kind"] == "dropin_wilson":
        return 0.0, 1.2
    return 0.0, (1.0 if case["nc"] == 2 else 1.2)


ZOLO_INTERVAL = (0.06, 28.0)  # of h_W^2, around the spectra of these links


def _flux(n, nb):
    """Phases of the U(1) field with nb quanta through the xy plane, (3, n2, n1, n0) complex."""
    n0, n1, n2 = n
    ph = np.ones((3, n2, n1, n0), complex)
    x, y = np.arange(n0), np.arange(n1)
    ph[1] = np.exp(-2j * np.pi * nb * x / (n0 * n1))[None, None, :]
    ph[0, :, :, n0 - 1] = np.exp(2j * np.pi * nb * y * n0 / (n0 * n1))[None, :]
    return ph


def _matrices(nc, n, links):
    """Reference link format -> (3, n2, n1, n0, nc, nc) row-major complex."""
    n0, n1, n2 = n
    if nc == 2:
        u = links.reshape(-1, 3, 4)
        m = np.empty(u.shape[:2] + (2, 2), complex)
        m[..., 0, 0] = u[..., 3] + 1j * u[..., 2]
        m[..., 0, 1] = u[..., 1] + 1j * u[..., 0]
        m[..., 1, 0] = -u[..., 1] + 1j * u[..., 0]
        m[..., 1, 1] = u[..., 3] - 1j * u[..., 2]
    else:
        m = np.swapaxes(links.view(complex).reshape(-1, 3, 3, 3), -1, -2)
    return np.ascontiguousarray(np.moveaxis(m, 1, 0)).reshape(3, n2, n1, n0, nc, nc)


def _ucc(nc, n, links):
    """The drop-ins' u_cc array, [mu V + site][i][j]."""
    return _matrices(nc, n, links).reshape(-1)


# ---------------------------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------------------------
PRECS = {"fp64": ovl.PREC_FP64, "fp32": ovl.PREC_FP32, "mixed": ovl.PREC_MIXED}
GAUGES = {"frozen": ovl.GAUGE_FROZEN, "links": ovl.GAUGE_LINKS, "full": ovl.GAUGE_FULL}


def _sign(case):
    if case.get("prec") == "zolotarev":
        return ovl.sign_opts(method=ovl.SIGN_ZOLOTAREV, lmin=0.0, lmax=0.0)
    return ovl.sign_opts(degree=case.get("degree", 256), cut=0.05, precision=PRECS[case.get("prec", "fp64")],
                         relax=case.get("relax", 0))


def _step(case):
    graph = case["kind"] != "observed" and case["prec"] != "zolotarev"
    return ovl.StepOpts(kind=ovl.WILSON if case.get("fermion") == "wilson" else ovl.OVERLAP, dt=case["dt"],
                        gauge=GAUGES[case.get("gauge", "links")], sign=_sign(case), use_graph=int(graph))


def prepare(case, seed):
    kind, nc = case["kind"], case["nc"]
    m, mdw = _masses(case)
    if kind == "ensemble":
        sizes = [int(s) for s in case["sizes"].split()]
        ctx = ovl.Ensemble(nc, [(s, s, s) for s in sizes], case["modes"], m_fermion=m, m_dw=mdw)
        for k, s in enumerate(sizes):
            g = np.random.Generator(np.random.Philox([seed, k]))
            ctx.set_system_links(k, _link_inputs(nc, (s, s, s), g))
            ctx.set_system_efield(k, _efield_inputs(nc, (s, s, s), g))
            ctx.set_system_u1_flux(k, k % 7)
            psi = _modes_inputs(nc, (s, s, s), case["modes"], seed * 64 + k).cpu().numpy()
            ctx.set_system_modes(k, ovl.PSI, psi)
            ctx.set_system_modes(k, ovl.PSIMID, psi)
        return dict(kind=kind, case=case, ctx=ctx, step=_step(case))
    n = _dims(case)
    links, e = _gauge_inputs(case, seed)
    if kind == "obs":
        return dict(kind=kind, case=case, n=n, links=torch.from_numpy(links).to(DEV), e=torch.from_numpy(e).to(DEV),
                    out=torch.zeros(len(ovl.OBS_NAMES), dtype=torch.float64, device=DEV))
    ctx = ovl.Context(nc, n, case.get("modes", 1), m_fermion=m, m_dw=mdw)
    if kind in ("dropin_wilson", "dropin_overlap"):
        return dict(kind=kind, case=case, ctx=ctx, ucc=_ucc(nc, n, links),
                    phi=_modes_inputs(nc, n, 1, seed).cpu().numpy()[0])
    ctx.set_links(links)
    ctx.set_efield(e)
    if kind == "gauge":
        return dict(kind=kind, case=case, ctx=ctx)
    if case["nb"]:
        ctx.set_u1_flux(case["nb"], 1.0)
    psi = _modes_inputs(nc, n, case["modes"], seed).cpu().numpy()
    ctx.set_modes(ovl.PSI, psi)
    if kind != "apply":
        ctx.set_modes(ovl.PSIMID, psi)
    if kind == "observed":
        ctx.autotune()  # a long run tunes its context once
    return dict(kind=kind, case=case, ctx=ctx, step=_step(case) if kind != "apply" else None, sign=_sign(case))


def run(state):
    kind, case = state["kind"], state["case"]
    if kind == "obs":
        ovl.observables_noalloc(case["nc"], state["n"], state["links"].data_ptr(), state["e"].data_ptr(),
                                state["out"].data_ptr(), torch.cuda.current_stream().cuda_stream)
        return state["out"]
    ctx = state["ctx"]
    if kind == "leapfrog":
        ctx.fermion_update(state["step"], case["steps"])
        return dict(psi=ctx.get_modes(ovl.PSI), mid=ctx.get_modes(ovl.PSIMID), links=ctx.get_links())
    if kind == "observed":
        q5, ncs, jv, ja = ctx.fermion_update_observed(state["step"], case["steps"], 1)
        return dict(axial_charge=q5, ncs_dot=ncs, jv=jv, ja=ja)
    if kind == "apply":
        ctx.apply_overlap(ovl.PSI, ovl.PSIMID, state["sign"])
        return ctx.get_modes(ovl.PSIMID)
    if kind == "ensemble":
        ctx.fermion_update(state["step"], case["steps"])
        return [ctx.get_system_modes(k, f) for k in range(ctx.n_systems) for f in (ovl.PSI, ovl.PSIMID)]
    if kind == "dropin_wilson":
        return ctx.wilson_evo_compute(state["ucc"], state["phi"])
    if kind == "dropin_overlap":
        return ctx.overlap_operator_compute(state["ucc"], state["phi"], *ZOLO_INTERVAL)
    obs = []
    for _ in range(case["steps"]):
        ctx.update_efield(case["dt"])
        ctx.update_links(case["dt"])
        obs.append(list(ctx.system_observables(0).values()))
    return dict(links=ctx.get_links(), efield=ctx.get_efield(), obs=np.array(obs))


# ---------------------------------------------------------------------------------------------
# the work of one pass
# ---------------------------------------------------------------------------------------------
def work(case):
    kind, nc = case["kind"], case["nc"]
    ng, lr = nc * nc - 1, (4 if nc == 2 else 18)
    S = 4 * nc * 16.0  # one FP64 spinor
    hop = 4 * nc * 18 + 6 * 2 * (8 * nc * nc - 2 * nc)  # flops of one site and mode of h_W
    dims = [(int(s),) * 3 for s in case["sizes"].split()] if kind == "ensemble" else [_dims(case)]
    V = sum(_volume(d) for d in dims)
    gauge = V * 3 * (lr + ng) * 8.0
    if kind == "obs":
        return dict(bytes=gauge + 56, flops=V * (3 * 60 * (8 * nc ** 3)))
    if kind == "gauge":
        return dict(bytes=case["steps"] * 4 * gauge, flops=case["steps"] * V * (3 * 80 * (8 * nc ** 3)))
    if kind == "dropin_wilson":
        return dict(bytes=V * (2 * S + 3 * nc * nc * 16), flops=V * hop)
    if kind == "dropin_overlap":  # about 100 iterations of two operators and 25 shifts
        return dict(bytes=V * (2 * S + 3 * nc * nc * 16), flops=100 * V * (2 * hop + 25 * 16 * nc * 4))
    sm = float(V) * case["modes"]
    out = 2 * sm * S  # both fields read back
    if kind == "leapfrog" and case["fermion"] == "wilson":
        s = S / 2 if case["prec"] == "fp32" else S
        return dict(bytes=case["steps"] * (sm * 6 * s + 2 * gauge) + out, flops=case["steps"] * 2 * sm * (hop + 16 * nc))
    if case["prec"] == "zolotarev":
        it = 2 * 100
        return dict(bytes=it * sm * 52 * S + 2 * 2 * 2000 * V * 2 * S + out,
                    flops=it * sm * (2 * hop + 25 * 64 * nc) + 2 * 2 * 2000 * V * 2 * hop)
    # Chebyshev: four vectors per degree in the storage precision of the step
    o, deg = _sign(case), case["degree"]
    h48, h32, h16 = ovl.sign_plan(o) if case["prec"] == "mixed" else ((deg + 1,) * 3 if case["prec"] == "fp64" else
                                                                        (0, 0, deg + 1))
    per = S * (h48 + 0.75 * (h32 - h48) + 0.5 * (h16 - h32) + 0.25 * (deg + 1 - h16))
    applies = 1 if kind == "apply" else 2 * case["steps"]
    w = dict(bytes=applies * sm * 4 * per, flops=applies * sm * 2 * (deg + 1) * (hop + 32 * nc))
    if kind in ("leapfrog", "ensemble"):
        w["bytes"] += out
    return w


# ---------------------------------------------------------------------------------------------
# the same in plain torch, 64 bits
# ---------------------------------------------------------------------------------------------
_DIM = (3, 2, 1)  # torch dimension of x, y, z in a (modes, n2, n1, n0, nc, spin) field


def _isigma(k, a, b):
    """i sigma_k applied to the two-component spinor (a, b)."""
    return ((1j * b, 1j * a), (b, -a), (1j * a, -1j * b))[k]


def _colour(u, v):
    """sum_j u[..., i, j] v[..., j] for links u (n2, n1, n0, nc, nc) and a field v (modes, ..., nc)."""
    nc = u.shape[-1]
    return torch.stack([sum(u[..., i, j] * v[..., j] for j in range(nc)) for i in range(nc)], -1)


def _h_w(psi, U, A):
    """h_W = (1/2) gamma0 [A - sum_k (1 + i g_k) U_k(x) psi(x+k) + (1 - i g_k) U_k^+(x-k) psi(x-k)]."""
    out = A * psi
    for k in range(3):
        for sg in (1, -1):
            if sg > 0:
                q, u = torch.roll(psi, -1, _DIM[k]), U[k]
            else:
                q = torch.roll(psi, 1, _DIM[k])
                u = torch.roll(U[k], 1, _DIM[k] - 1).conj().transpose(-1, -2)
            s = _isigma(k, q[..., 2], q[..., 3])
            a, b = _colour(u, q[..., 0] + sg * s[0]), _colour(u, q[..., 1] + sg * s[1])
            t = _isigma(k, a, b)
            out[..., 0] -= a
            out[..., 1] -= b
            out[..., 2] += sg * t[0]
            out[..., 3] += sg * t[1]
    out *= 0.5
    out[..., 2:] *= -1
    return out


def _cheb(degree, cut):
    N = 8 * (degree + 1) + 64
    th = np.pi * (np.arange(N) + 0.5) / N
    d2 = cut * cut
    f = 1 / np.sqrt(0.5 * ((1 - d2) * np.cos(th) + 1 + d2))
    c = np.array([2 * np.sum(f * np.cos(k * th)) / N for k in range(degree + 1)])
    c[0] /= 2
    return c


def _overlap(psi, U, A, m, M, degree, cut):
    """-i h_ov psi with the Chebyshev sign."""
    lam = abs(3 + m - M) + 3
    d2 = cut * cut
    al, be = 2 / (lam * lam * (1 - d2)), -(1 + d2) / (1 - d2)
    c = _cheb(degree, cut)
    b1, b2 = torch.zeros_like(psi), torch.zeros_like(psi)
    for k in range(degree, -1, -1):
        f = 1.0 if k == 0 else 2.0
        t = _h_w(_h_w(b1, U, A), U, A)
        b1, b2 = c[k] * psi + f * (al * t + be * b1) - b2, b1
    eps = _h_w(b1, U, A) / lam
    g = psi.clone()
    g[..., 2:] *= -1
    return -1j * M * ((1 + m / 2) * g + (1 - m / 2) * eps)


def _generators(nc):
    t = np.zeros((nc * nc - 1, nc, nc), complex)
    pairs = [((0, 1), 0)] if nc == 2 else [((0, 1), 0), ((0, 2), 3), ((1, 2), 5)]
    for (i, j), a in pairs:
        t[a, i, j] = t[a, j, i] = 0.5
        t[a + 1, i, j], t[a + 1, j, i] = -0.5j, 0.5j
    t[2, 0, 0], t[2, 1, 1] = 0.5, -0.5
    if nc == 3:
        t[7] = np.diag([1, 1, -2]) / (2 * math.sqrt(3.0))
    return t


def _shift(u, k, by):
    return np.roll(u, -by, axis=2 - k)  # u: (n2, n1, n0, ...), value at x + by k


def _move_links(U, E, dt):
    """U <- exp(-i dt E) U; U (3, n2, n1, n0, nc, nc), E (3, n2, n1, n0, ng)."""
    h = np.einsum("...a,aij->...ij", E, _generators(U.shape[-1]))
    w, q = np.linalg.eigh(h)
    return np.einsum("...ij,...j,...kj->...ik", q, np.exp(-1j * dt * w), q.conj()) @ U


def _move_efield(U, E, dt):
    """E_mu += -2 dt sum_{nu != mu} Re tr(i t^a (U_{mu nu} + U_{mu -nu}))."""
    t = _generators(U.shape[-1])
    dag = lambda x: np.conj(np.swapaxes(x, -1, -2))  # noqa: E731
    out = E.copy()
    for mu in range(3):
        p = 0
        for nu in range(3):
            if nu == mu:
                continue
            unu = U[nu]
            p = p + U[mu] @ _shift(unu, mu, 1) @ dag(_shift(U[mu], nu, 1)) @ dag(unu)
            back = _shift(unu, nu, -1)
            p = p + U[mu] @ dag(_shift(back, mu, 1)) @ dag(_shift(U[mu], nu, -1)) @ back
        out[mu] += -2 * dt * np.real(1j * np.einsum("aij,...ji->...a", t, p))
    return out


def _links_out(U):
    """(3, n2, n1, n0, nc, nc) matrices -> the reference's link format."""
    nc = U.shape[-1]
    m = np.moveaxis(U.reshape(3, -1, nc, nc), 0, 1)
    if nc == 2:
        return np.stack([m[..., 0, 1].imag, m[..., 0, 1].real, m[..., 0, 0].imag, m[..., 0, 0].real], -1).reshape(-1)
    return np.ascontiguousarray(np.swapaxes(m, -1, -2)).reshape(-1).view(np.float64)


def _efield_in(nc, n, e):
    return np.ascontiguousarray(np.moveaxis(e.reshape(-1, 3, nc * nc - 1), 1, 0)).reshape(3, n[2], n[1], n[0], -1)


def _operator(case, n, m, M, nb):
    """psi, U -> -i h psi for the case's fermions, and the links with their phases on the GPU."""
    nc = case["nc"]
    A = 6 + 2 * m - 2 * M
    ph = _flux(n, nb)[..., None, None]

    def links(U):
        return torch.from_numpy(U * ph).to(DEV)

    if case.get("fermion") == "wilson" or case["kind"] == "dropin_wilson":
        return links, lambda psi, U: -1j * _h_w(psi, U, A)
    zolo = case["kind"] == "dropin_overlap" or case["prec"] == "zolotarev"
    degree, cut = (400, 0.04) if zolo else (case["degree"], 0.05)
    return links, lambda psi, U: _overlap(psi, U, A, m, M, degree, cut)


def _leapfrog(case, n, links, e, psi, nb):
    m, M = _masses(case)
    setup, op = _operator(case, n, m, M, nb)
    nc, dt, gauge = case["nc"], case["dt"], case.get("gauge", "links")
    U, E = _matrices(nc, n, links), _efield_in(nc, n, e)
    psi = psi.reshape(-1, n[2], n[1], n[0], nc, 4)
    a, b = psi.clone(), psi.clone()
    u = setup(U)
    for _ in range(case["steps"]):
        for which in (0, 1):
            if which == 0:
                a += dt * op(b, u)
            else:
                b += dt * op(a, u)
            if gauge != "frozen":
                if gauge == "full":
                    E = _move_efield(U, E, 0.5 * dt)
                U = _move_links(U, E, 0.5 * dt)
                u = setup(U)
    flat = lambda t: t.reshape(t.shape[0], -1).cpu().numpy()  # noqa: E731
    return flat(a), flat(b), _links_out(U)


def exact(case, seed):
    kind, nc = case["kind"], case["nc"]
    if kind in ("observed", "obs"):
        return None
    m, M = _masses(case)
    if kind == "ensemble":
        if nc == 3 or case["degree"] * case["steps"] > 600:
            return None
        out = []
        for k, s in enumerate(int(s) for s in case["sizes"].split()):
            n = (s, s, s)
            g = np.random.Generator(np.random.Philox([seed, k]))
            links, e = _link_inputs(nc, n, g), _efield_inputs(nc, n, g)
            a, b, _ = _leapfrog(case, n, links, e, _modes_inputs(nc, n, case["modes"], seed * 64 + k), k % 7)
            out += [a, b]
        return out
    n = _dims(case)
    links, e = _gauge_inputs(case, seed)
    if kind == "gauge":
        U, E = _matrices(nc, n, links), _efield_in(nc, n, e)
        for _ in range(case["steps"]):
            E = _move_efield(U, E, case["dt"])
            U = _move_links(U, E, case["dt"])
        back = np.ascontiguousarray(np.moveaxis(E.reshape(3, -1, nc * nc - 1), 0, 1)).reshape(-1)
        return dict(links=_links_out(U), efield=back, obs=None)
    psi = _modes_inputs(nc, n, case.get("modes", 1), seed)
    if kind == "leapfrog":
        applies = 2 * case["steps"] * (1 if case["fermion"] == "wilson" else 2 * case.get("degree", 400))
        if applies * _volume(n) * case["modes"] * nc * nc > 5e9:
            return None
        if case["gauge"] != "frozen" and case["steps"] * _volume(n) > 500000:
            return None
        a, b, u = _leapfrog(case, n, links, e, psi, case["nb"])
        return dict(psi=a, mid=b, links=u)
    setup, op = _operator(case, n, m, M, case.get("nb", 0))
    r = op(psi.reshape(-1, n[2], n[1], n[0], nc, 4), setup(_matrices(nc, n, links)))
    r = r.reshape(r.shape[0], -1).cpu().numpy()
    return r if kind == "apply" else r[0]
