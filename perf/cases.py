"""Timed cases of the particle-interaction step, through the calls a FLOWUnsteady
program makes: the UJ hooks (`UJ_gpu`, `UJ_fmm_gpu`), the time step (`nextstep`),
probe velocities (`Vvpm_on_Xs`) and the batched sweep (`UJ_gpu_batch`,
`nextstep_batch`).  All of them take the host particle matrix, as the driver
holds it, so a pass is the whole call: the field to the GPU, the evaluation and
the results back in the matrix.

  listed()            the cases, from an early wake of a few hundred particles to
                      the 1,048,576-particle cube of the benchmark
  draw(rng)           another case of the same ranges
  prepare(case, seed) the particle fields (and probes) of a case
  run(state)          one pass; returns what it wrote
  work(case)          bytes and operations a pass cannot do without
  exact(case, seed)   the same outputs from all-pairs sums in 64 bits (torch)
"""
import math

import numpy as np
import torch

from flowunsteady_amd import vpm, workloads

# Settings a case may leave out.
DEFAULTS = {"kernel": "gaussianerf", "precision": "fp64", "fmm": False, "p": 4, "ncrit": 50,
            "theta": 0.4, "core_aware": False, "sfs": "none", "viscous": "none", "relax": False,
            "static": 0.0, "m": 0, "nfields": 0}


def listed():
    return [
        # An early wake or a wing's first steps: latency of one call.
        {"name": "uj_wake_601", "op": "uj", "field": "rotor", "n": 601},
        # The vortex-ring validation run: FP64 RK3 with Pedrizzetti relaxation.
        {"name": "step_ring_8000", "op": "step", "field": "ring", "n": 8000, "relax": True},
        # A small rotor with the constant-coefficient SFS model on the direct
        # scheme, 5 % of the particles static (the bound vorticity).
        {"name": "step_sfs_direct_20011", "op": "step", "field": "rotor", "n": 20011,
         "sfs": "constant", "static": 0.05, "relax": True},
        # A mid-low-fidelity rotor wake (70 k particles), direct sums in FP64.
        {"name": "uj_direct_fp64_70001", "op": "uj", "field": "rotor", "n": 70001},
        # Probe velocities on lifting-surface control points, every time step.
        {"name": "probes_4099", "op": "probes", "field": "rotor", "n": 200003, "m": 4099,
         "precision": "mixed"},
        # The benchmark's cube: direct mixed-precision sums, the largest case.
        {"name": "uj_cube_mixed_1048576", "op": "uj", "field": "cube", "n": 1048576,
         "precision": "mixed"},
        # The algebraic kernel, which has no far-field form.
        {"name": "uj_winckelmans_131071", "op": "uj", "field": "cube", "n": 131071,
         "kernel": "winckelmans", "precision": "mixed"},
        # A mid-high-fidelity rotor wake (200 k particles) with FLOWUnsteady's
        # default FMM (p = 4, ncrit = 50, theta = 0.4, geometric acceptance),
        # core spreading and relaxation, FP64.
        {"name": "step_rotor_fmm_200003", "op": "step", "field": "rotor", "n": 200003, "fmm": True,
         "viscous": "corespreading", "static": 0.02, "relax": True},
        # High fidelity in FP64: dynamic SFS model on the default FMM.
        {"name": "step_dynamic_fp64_100003", "op": "step", "field": "rotor", "n": 100003,
         "fmm": True, "sfs": "dynamic", "relax": True},
        # A large wake at a tight tolerance: p = 8, core-aware acceptance, mixed
        # near field.
        {"name": "uj_fmm_mixed_p8_1000003", "op": "uj", "field": "rotor", "n": 1000003, "fmm": True,
         "p": 8, "core_aware": True, "precision": "mixed"},
        # High fidelity at a million particles: a volumetric wake, p = 8, dynamic
        # SFS, relaxation, RK3, mixed near field.
        {"name": "step_dynamic_mixed_786433", "op": "step", "field": "blob", "n": 786433,
         "fmm": True, "p": 8, "sfs": "dynamic", "relax": True, "precision": "mixed"},
        # A sweep of independent cases of uneven size in one launch.
        {"name": "batch_24_fields", "op": "batch_uj", "field": "rings", "n": 25000, "nfields": 24,
         "precision": "mixed"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a call, a field, a size (log-uniform over the range its
    scheme is used at) and settings."""
    kind = rng.choice(("uj_direct", "step_direct", "probes", "uj_fmm", "step_fmm", "batch"))
    if kind == "uj_direct":
        precision = rng.choice(("fp64", "mixed"))
        return {"op": "uj", "field": rng.choice(("rotor", "cube", "ring", "blob")),
                "n": _log_int(rng, 300, 150000 if precision == "fp64" else 400000),
                "kernel": rng.choice(("gaussianerf", "gaussianerf", "winckelmans", "gaussian")),
                "precision": precision}
    if kind == "step_direct":
        return {"op": "step", "field": rng.choice(("rotor", "ring")), "n": _log_int(rng, 500, 60000),
                "precision": rng.choice(("fp64", "mixed")),
                "sfs": rng.choice(("none", "constant", "dynamic")),
                "static": rng.choice((0.0, 0.05)), "relax": rng.random() < 0.7}
    if kind == "probes":
        return {"op": "probes", "field": "rotor", "n": _log_int(rng, 5000, 300000),
                "m": _log_int(rng, 100, 20000), "precision": rng.choice(("fp64", "mixed"))}
    if kind == "uj_fmm":
        return {"op": "uj", "field": rng.choice(("rotor", "blob")), "n": _log_int(rng, 20000, 1000000),
                "fmm": True, "p": rng.choice((3, 4, 6, 8, 10)), "ncrit": rng.choice((30, 50, 100)),
                "core_aware": rng.random() < 0.3, "precision": rng.choice(("fp64", "mixed"))}
    if kind == "step_fmm":
        sfs = rng.choice(("none", "dynamic"))
        return {"op": "step", "field": "rotor", "n": _log_int(rng, 20000, 250000), "fmm": True,
                "p": rng.choice((4, 4, 6, 8)), "sfs": sfs, "static": rng.choice((0.0, 0.05)),
                "relax": rng.random() < 0.7, "precision": rng.choice(("fp64", "mixed"))}
    return {"op": rng.choice(("batch_uj", "batch_step")), "field": "rings",
            "n": _log_int(rng, 1000, 15000), "nfields": rng.randint(2, 32),
            "precision": rng.choice(("fp64", "mixed"))}


# ---- fields -------------------------------------------------------------------------
def _rotor(n, seed):
    """Two blades' helical wake sheets over six revolutions: particles on a mesh
    of spacing h along the span and the helix, jittered, cores of 2.125 h, the
    circulation trailed near tip and root."""
    rng = np.random.default_rng(seed)
    h = math.sqrt(2 * 6 * 2 * math.pi * 0.9 / n)
    ns = max(1, int(round(0.9 / h)))
    nt = -(-n // (2 * ns))
    i = np.arange(2 * ns * nt)
    blade, span, age = i % 2, (i // 2) % ns, i // (2 * ns)
    r = 0.1 + 0.9 * (span + 0.5) / ns
    th = 12 * math.pi * (age + 0.5) / nt
    phi = th + math.pi * blade + rng.normal(0.0, 0.002)
    z = 0.15 * th / (2 * math.pi) * (1 + 0.3 * (1 - r))
    X = np.stack([r * np.cos(phi), r * np.sin(phi), z], axis=1)[:n]
    T = np.stack([-np.sin(phi), np.cos(phi), np.full_like(phi, 0.024)], axis=1)[:n]
    g = 0.1 * h / ns * (8 * np.exp(-((r - 0.95) / 0.06) ** 2) - 4 * np.exp(-((r - 0.15) / 0.08) ** 2)
                        + 0.5)[:n]
    X = X + rng.normal(0.0, 0.15 * h, X.shape)
    G = g[:, None] * T + rng.normal(0.0, 0.05 * 0.1 * h / ns, X.shape)
    s = 2.125 * h * (1 + 0.1 * rng.uniform(-1, 1, n))
    return X, G, s, s ** 3


def _field(kind, n, seed):
    if kind == "rotor":
        return _rotor(n, seed)
    if kind == "ring":   # the vortex ring at n particles: 5 x as many round the core as along it
        st = max(8, int(round(math.sqrt(n / 5))))
        X, G, s, v = workloads.vortex_ring(n_stations=st, n_cross=-(-n // st), seed=seed)
        return X[:n], G[:n], s[:n], v[:n]
    if kind == "cube":
        return workloads.uniform_cube(n=n, seed=seed)
    # the volumetric wake, strengths for velocities of order 1
    X, G, s, v = workloads.gaussian_blob(n=n, seed=seed)
    return X, G * (1200.0 / n), s, v


def _field_sizes(case, seed):
    """Sizes of a sweep's fields, log-uniform around case["n"] (a fifth to five times it)."""
    rng = np.random.default_rng([case["n"], case["nfields"]])   # the same sizes for every seed
    return [max(200, int(case["n"] * math.exp(u)))
            for u in rng.uniform(math.log(0.2), math.log(5.0), case["nfields"])]


def _full(case):
    return {**DEFAULTS, **case}


def _arrays(case, seed):
    """[(X, Gamma, sigma, vol, static), ...] of a case's fields."""
    c = _full(case)
    out = []
    if c["nfields"]:
        for k, n in enumerate(_field_sizes(c, seed)):
            out.append((*_field("ring" if k % 2 == 0 else "rotor", n, 1000 * seed + k), None))
        return out
    X, G, s, v = _field(c["field"], c["n"], seed)
    static = None
    if c["static"] > 0:
        static = np.zeros(c["n"])
        static[-max(1, int(c["static"] * c["n"])):] = 1.0
    return [(X, G, s, v, static)]


def _probes(case, seed):
    """Points of lifting surfaces in the wake's plane of rotation."""
    rng = np.random.default_rng(seed + 77)
    r = np.sqrt(rng.uniform(0.01, 1.2, case["m"]))
    t = rng.uniform(0, 2 * np.pi, case["m"])
    return np.stack([r * np.cos(t), r * np.sin(t), rng.normal(0.0, 0.05, case["m"])], axis=1)


# Time step: particles move by well under a per cent of a core.
DT = 2e-5
NU = 1.5e-5


def prepare(case, seed):
    c = _full(case)
    sfs = {"none": vpm.noSFS, "constant": vpm.SFS_Cs_nobackscatter(),
           "dynamic": vpm.DynamicSFS()}[c["sfs"]]
    fields = []
    for X, G, s, v, static in _arrays(c, seed):
        n = len(X)
        visc = (vpm.CoreSpreading(NU, float(np.median(s)), vpm.zeta_fmm, beta=100.0, itmax=20,
                                  tol=1e-1) if c["viscous"] == "corespreading" else vpm.Inviscid())
        pf = vpm.ParticleField(n, kernel=getattr(vpm, c["kernel"]), SFS=sfs,
                               UJ=vpm.UJ_fmm_gpu if c["fmm"] else vpm.UJ_gpu,
                               fmm=vpm.FMM(p=c["p"], ncrit=c["ncrit"], theta=c["theta"],
                                           nonzero_sigma=c["core_aware"]),
                               relaxation=vpm.pedrizzetti, precision=c["precision"], viscous=visc)
        vpm.add_particles(pf, X, G, s, vol=v, static=static)
        fields.append(pf)
    return {"case": c, "fields": fields, "Xs": _probes(c, seed) if c["m"] else None}


def _uj_out(pf):
    return {"U": vpm.get_U(pf), "J": vpm.get_J(pf)}


def _step_out(pf):
    out = {"X": vpm.get_X(pf), "Gamma": vpm.get_Gamma(pf), "sigma": vpm.get_sigma(pf),
           **_uj_out(pf)}
    if pf.SFS.kind:
        out["SFS"] = vpm.get_SFS(pf)
        out["C"] = vpm.get_C(pf)
    return out


def run(state):
    c, fields = state["case"], state["fields"]
    pf = fields[0]
    if c["op"] == "uj":
        pf.UJ(pf)
        return _uj_out(pf)
    if c["op"] == "step":
        vpm.nextstep(pf, DT, relax=c["relax"])
        return _step_out(pf)
    if c["op"] == "probes":
        return {"U": vpm.Vvpm_on_Xs(pf, state["Xs"])}
    if c["op"] == "batch_uj":
        vpm.UJ_gpu_batch(fields)
        return {"U": [vpm.get_U(f) for f in fields], "J": [vpm.get_J(f) for f in fields]}
    vpm.nextstep_batch(fields, DT, relax=c["relax"])
    return {"X": [vpm.get_X(f) for f in fields], "U": [vpm.get_U(f) for f in fields]}


def work(case):
    """Bytes: position, circulation and core in, U and J out (a step: X, Gamma,
    sigma and, with an SFS model, Estr and C as well), once per particle.
    Operations: 77 (gaussian-erf) or 81 (Winckelmans) per pair and evaluation on
    the direct scheme.  FMM: the pairs of a leaf of ncrit / 2 particles with
    itself and its 26 neighbours, and for every leaf (and its share 8/7 of the
    tree) 189 M2L translations of the (p + 1)^2 harmonic components (three
    columns, the triangle of total degree <= p: half the square)."""
    c = _full(case)
    sizes = _field_sizes(c, 0) if c["nfields"] else [c["n"]]
    steps = "step" in c["op"]
    evals = (3 + (1 if c["relax"] else 0)) if steps else 1
    n = sum(sizes)
    per = 77 if c["kernel"] != "winckelmans" else 81
    if c["op"] == "probes":
        return {"bytes": 8 * (7 * n + 15 * c["m"]), "flops": per * n * c["m"]}
    if c["fmm"]:
        half = c["ncrit"] / 2
        pairs = n * 27 * half
        m2l = (8 / 7) * (n / half) * 189 * 3 * (c["p"] + 1) ** 4
        flops = evals * (per * pairs + m2l)
    else:
        pairs = sum(k * k for k in sizes)
        flops = evals * per * pairs
    if c["sfs"] != "none":   # Estr: 42 per pair, with its derivatives about as many again
        flops += 3 * pairs * (42 if c["sfs"] == "constant" else 160)
    words = 7 + 12 + (7 if steps else 0) + (10 if steps and c["sfs"] != "none" else 0)
    return {"bytes": 8 * words * n, "flops": flops}


# ---- the same in 64 bits ------------------------------------------------------------------
def _radial(kernel, r, s):
    """g / r^3, g'/(sigma r^4) - 3 g / r^5 and their core-size derivatives, zeta / s^3 and
    zD / s^3 of the kernel (all finite at r = 0; close pairs by the series in rho)."""
    q = r / s
    q2 = q * q
    if kernel == "gaussianerf":
        e = torch.exp(-0.5 * q2)
        c = math.sqrt(2 / math.pi)
        g = torch.erf(q * math.sqrt(0.5)) - c * q * e
        dg = c * q2 * e
        z = (2 * math.pi) ** -1.5 * e
        zp_q = -z                                    # zeta' / rho
        sa, sb = torch.zeros_like(q), torch.zeros_like(q)
        for k in range(14, -1, -1):                  # g / rho^3 and (g'/rho^2 - 3 g/rho^3) / rho^2
            t = c * (-1) ** k / (2.0 ** k * math.factorial(k) * (2 * k + 3))
            sa = sa * q2 + t
            if k >= 1:
                sb = sb * q2 + 2 * k * t
        small = q < 0.8
    elif kernel == "gaussian":
        q3 = q2 * q
        e = torch.exp(-q3)
        g, dg = -torch.expm1(-q3), 3 * q2 * e
        z = 3 / (4 * math.pi) * e
        zp_q = -3 * q * z
        sa, sb = torch.zeros_like(q), torch.zeros_like(q)
        for k in range(14, -1, -1):
            sa = sa * q3 + (-1) ** k / math.factorial(k + 1)
            if k >= 1:
                sb = sb * q3 + 3 * k * (-1) ** k / math.factorial(k + 1)
        sb = sb * q
        small = q3 < 0.5
    else:   # winckelmans
        w = 1 + q2
        z = 15 / (8 * math.pi) * w ** -3.5
        zp_q = -7 * z / w
        a, b = (q2 + 2.5) * w ** -2.5, -3 * (q2 + 3.5) * w ** -3.5
        return a / s ** 3, b / s ** 5, z, zp_q
    qq = torch.where(small, torch.ones_like(q), q)
    a = torch.where(small, sa, g / qq ** 3)
    b = torch.where(small, sb, dg / qq ** 4 - 3 * g / qq ** 5)
    return a / s ** 3, b / s ** 5, z, zp_q


def _pair_sums(kernel, Xt, X, G, s, what, Jt=None, Js=None, DJt=None, DJs=None):
    """All-pairs sums at targets Xt, by blocks: ("uj") U, J; ("dsig") D[U], D[J];
    ("estr") E, and with DJ also D[E].  Sums over sources are products of the
    radial weights with source columns, taken about each block's centre."""
    outs = []
    n = len(X)
    step = max(1, 100_000_000 // n)
    for t0 in range(0, len(Xt), step):
        x = Xt[t0:t0 + step]
        ctr = x.mean(0)
        x, y = x - ctr, X - ctr
        r2 = (x[:, :1] - y[:, 0]).square_()
        for l in (1, 2):
            d = x[:, l:l + 1] - y[:, l]
            r2.addcmul_(d, d)
        r = r2.sqrt_()
        A, B, z, zp_q = _radial(kernel, r, s)
        if what == "estr":
            zs = z / s ** 3
            JG = torch.einsum("nlk,nl->nk", Js, G)           # transposed scheme: S_k = J_lk G_l
            sums = zs @ torch.cat([G, JG], 1)
            E = torch.einsum("tlk,tl->tk", Jt[t0:t0 + step], sums[:, :3]) - sums[:, 3:]
            if DJt is None:
                outs.append((E,))
                continue
            zD = -(3 * z + (r / s) ** 2 * zp_q) / s ** 3
            DJG = torch.einsum("nlk,nl->nk", DJs, G)
            s2 = zD @ torch.cat([G, JG], 1)
            s3 = zs @ DJG
            DE = (torch.einsum("tlk,tl->tk", Jt[t0:t0 + step], s2[:, :3]) - s2[:, 3:]
                  + torch.einsum("tlk,tl->tk", DJt[t0:t0 + step], sums[:, :3]) - s3)
            outs.append((E, DE))
            continue
        if what == "dsig":
            A, B = -4 * math.pi * z / s ** 3, -4 * math.pi * zp_q / s ** 5
        live = (r > 0).to(A.dtype)
        A, B = A * live, B * live
        yG = torch.cross(y, G, dim=1)                        # c = x x G - y x G
        a = A @ torch.cat([G, yG], 1)
        U = torch.cross(x, a[:, :3], dim=1) - a[:, 3:]
        cols = [G, yG] + [G * y[:, l:l + 1] for l in range(3)] + [yG * y[:, l:l + 1] for l in range(3)]
        b = B @ torch.cat(cols, 1)
        J = torch.empty(len(x), 3, 3, dtype=A.dtype, device=A.device)   # J[k, l]
        c0 = torch.cross(x, b[:, :3], dim=1) - b[:, 3:6]
        for l in range(3):
            c1 = torch.cross(x, b[:, 6 + 3 * l:9 + 3 * l], dim=1) - b[:, 15 + 3 * l:18 + 3 * l]
            J[:, :, l] = c0 * x[:, l:l + 1] - c1
        W = a[:, :3]                                         # + A eps_klm G_m
        J[:, 0, 1] += W[:, 2]; J[:, 1, 0] -= W[:, 2]
        J[:, 1, 2] += W[:, 0]; J[:, 2, 1] -= W[:, 0]
        J[:, 2, 0] += W[:, 1]; J[:, 0, 2] -= W[:, 1]
        k = -1 / (4 * math.pi)
        # d c_k / d x_l = eps_klm G_m with c = dX x G
        outs.append((k * U, k * J))
    return [torch.cat(v) for v in zip(*outs)]


ZETA0 = {"gaussianerf": (2 * math.pi) ** -1.5, "gaussian": 3 / (4 * math.pi),
         "winckelmans": 15 / (8 * math.pi)}


def _rk3(c, X, G, s, static):
    """One low-storage RK3 step of the rVPM equations and the relaxation, as nextstep."""
    kern, free = c["kernel"], (static == 0)
    A, Bc = (0.0, -5 / 9, -153 / 128), (1 / 3, 15 / 16, 8 / 15)
    qx, qg, qs = torch.zeros_like(X), torch.zeros_like(G), torch.zeros_like(s)
    E = torch.zeros_like(X)
    C = torch.zeros(len(X), 3, dtype=X.dtype, device=X.device)   # coefficient, averages
    f1 = free[:, None]
    for st in range(3):
        U, J = _pair_sums(kern, X, X, G, s, "uj")
        S = torch.einsum("nlk,nl->nk", J, G)
        sf = torch.zeros_like(s)
        if c["sfs"] == "constant":
            (E,) = _pair_sums(kern, X, X, G, s, "estr", J, J)
            ge = (G * E).sum(1)
            C[:, 0] = torch.where(0.15 * ge < 0, 0.0, 0.15)
        elif c["sfs"] == "dynamic":
            _, DJ = _pair_sums(kern, X, X, G, s, "dsig")
            E, DE = _pair_sums(kern, X, X, G, s, "estr", J, J, DJ, DJ)
            num = (3 * 0.999 - 2) / s * torch.einsum("nk,nkl,nl->n", G, DJ, G)
            den = s * s / ZETA0[kern] * (G * DE).sum(1)
            w = 0.005 if st else 1.0
            num, den = w * num + (1 - w) * C[:, 1], w * den + (1 - w) * C[:, 2]
            cc = torch.where(den != 0, num / den, torch.zeros_like(den)).clamp(0.0, 1.0)
            cc = torch.where(cc * (G * E).sum(1) < 0, torch.zeros_like(cc), cc)
            C = torch.where(f1, torch.stack([cc, num, den], 1), C)
        sf = C[:, 0] * s ** 3 / ZETA0[kern]
        g2 = (G * G).sum(1)
        Z = torch.where(g2 > 0, 0.2 * (S * G).sum(1) / torch.where(g2 > 0, g2, 1.0), 0.0)
        Fs = -s * Z + (NU / s if c["viscous"] == "corespreading" else 0.0)
        qx = A[st] * qx + DT * U
        qg = A[st] * qg + DT * (S - 3 * Z[:, None] * G - sf[:, None] * E)
        qs = A[st] * qs + DT * Fs
        X = torch.where(f1, X + Bc[st] * qx, X)
        G = torch.where(f1, G + Bc[st] * qg, G)
        s = torch.where(free, s + Bc[st] * qs, s)
    if c["relax"]:
        U, J = _pair_sums(kern, X, X, G, s, "uj")
        w = torch.stack([J[:, 2, 1] - J[:, 1, 2], J[:, 0, 2] - J[:, 2, 0], J[:, 1, 0] - J[:, 0, 1]], 1)
        nw, ng = w.norm(dim=1, keepdim=True), G.norm(dim=1, keepdim=True)
        G = torch.where(f1 & (nw > 0), 0.7 * G + 0.3 * ng * w / nw, G)
    out = {"X": X, "Gamma": G, "sigma": s, "U": U, "J": J}
    if c["sfs"] != "none":
        out["SFS"], out["C"] = E, C[:, 0]
    return out


def exact(case, seed):
    c = _full(case)
    evals = 1 if "step" not in c["op"] else {"none": 4, "constant": 7, "dynamic": 10}[c["sfs"]]
    arrays = _arrays(c, seed)
    Xs = _probes(c, seed) if c["m"] else None
    pairs = evals * sum(len(a[0]) * (c["m"] or len(a[0])) for a in arrays)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if pairs > (5e10 if dev == "cuda" else 2e9):   # over about 20 seconds
        return None

    def t(v):
        return torch.as_tensor(np.ascontiguousarray(v), dtype=torch.float64, device=dev)

    def flat(J):   # J[n, k + 3 l]
        return J.transpose(1, 2).reshape(-1, 9)

    outs = []
    for X, G, s, _, static in arrays:
        X, G, s = t(X), t(G), t(s)
        if Xs is not None:
            return {"U": _pair_sums(c["kernel"], t(Xs), X, G, s, "uj")[0].cpu()}
        if "step" in c["op"]:
            o = _rk3(c, X, G, s, t(static) if static is not None else torch.zeros_like(s))
        else:
            U, J = _pair_sums(c["kernel"], X, X, G, s, "uj")
            o = {"U": U, "J": J}
        o["J"] = flat(o["J"])
        outs.append({k: v.cpu() for k, v in o.items()})
    if not c["nfields"]:
        return outs[0]
    keys = ("U", "J") if c["op"] == "batch_uj" else ("X", "U")
    return {k: [o[k] for o in outs] for k in keys}
