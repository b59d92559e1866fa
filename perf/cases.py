"""Performance cases of the XC path: what a Kohn-Sham program has this library do.

Every case is one pass through the public entry points (`chinium_amd`), over the range of sizes, forms
and options that such a program meets: one XC build per SCF iteration (plain FP64 and mixed form, host or
device matrices, closed and open shell, LDA / GGA / meta-GGA, from one water to 128), the first build at a
new geometry (grid, AO tables and all), many molecules in one pack, the nuclear gradient, the second
derivatives with the response matrices, and the training of the learned functional.

Geometries are droplets of water, all-trans alkanes and carbon rings in the basis sets and grids of
`chinium_amd/data`. The density matrix is D = 2 C C^T of seeded orbitals that decay with the distance from
their centre and are orthonormal in the analytic overlap, so that it is positive, holds the right number of
electrons and falls off as the density matrix of a molecule with a gap does.

`exact` restates the path in plain torch and numpy (64 bits): basis and grid files, AO values, Becke
weights, functionals (by automatic differentiation) and contractions.
"""
import functools
import math
import os

import numpy as np
import torch

DATA = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "chinium_amd", "data")
BOHR = 1.8897259886  # bohr per angstrom, as the library converts
F64 = torch.float64
SYMBOL = {1: "H", 6: "C", 8: "O"}
CODES = {"SVWN5": 0, "PBE": 1, "B3LYP": 1, "R2SCAN": 2}  # functional -> family (0 LDA, 1 GGA, 2 meta-GGA)


# ---- cases --------------------------------------------------------------------------------------
def listed():
    return [
        # an SCF iteration of the smallest molecule, the reference's by-value calls: launches and latency
        dict(name="build_fp64_h2o", kind="build", mol="water", n=1, basis="cc-pvdz", grid="SG-1", func="PBE",
             form="fp64", io="host", spin=1),
        # an ordinary FP64 iteration, hybrid GGA
        dict(name="build_fp64_h2o16", kind="build", mol="water", n=16, basis="def2-svp", grid="SG-2", func="B3LYP",
             form="fp64", io="host", spin=1),
        # FP64 meta-GGA with f functions on the finest grid (cyclo[18]carbon)
        dict(name="build_fp64_c18_r2scan", kind="build", mol="ring", n=18, basis="def2-tzvp", grid="SG-3",
             func="R2SCAN", form="fp64", io="device", spin=1),
        # unrestricted: a radical cation of odd size
        dict(name="build_fp64_uks_c7", kind="build", mol="alkane", n=7, basis="def2-svp", grid="SG-1", func="PBE",
             form="fp64", io="host", spin=2),
        # the mixed form with D and V kept on the GPU: ordinary, meta-GGA, the largest basis
        dict(name="build_mixed_h2o16", kind="build", mol="water", n=16, basis="def2-svp", grid="SG-2", func="B3LYP",
             form="mixed", io="device", spin=1),
        dict(name="build_mixed_h2o48_r2scan", kind="build", mol="water", n=48, basis="def2-svp", grid="SG-2",
             func="R2SCAN", form="mixed", io="device", spin=1),
        dict(name="build_mixed_h2o128", kind="build", mol="water", n=128, basis="def2-svp", grid="SG-2", func="B3LYP",
             form="mixed", io="device", spin=1),
        # a geometry step: grid, Becke weights, screening, AO tables, then the first build on them
        dict(name="geometry_mixed_h2o24", kind="geometry", mol="water", n=24, basis="def2-svp", grid="SG-1", func="PBE",
             form="mixed", io="host", spin=1),
        # many small molecules in one pass
        dict(name="pack_mixed_alkanes24", kind="pack", mol="alkane", n=24, count=24, basis="def2-svp", grid="SG-1",
             func="PBE", form="mixed", io="device", spin=1),
        # nuclear gradient of the XC energy after an iteration
        dict(name="gradient_fp64_h2o8", kind="gradient", mol="water", n=8, basis="def2-svp", grid="SG-2", func="PBE",
             form="fp64", io="host", spin=1),
        # a frequency calculation's XC part: f_xc, skeleton terms, response matrices of a coupled-perturbed step
        dict(name="hessian_fp64_h2o2", kind="hessian", mol="water", n=2, basis="def2-svp", grid="SG-1", func="PBE",
             form="fp64", io="host", spin=1),
        # one pass of the learned functional's training (forward, backward, Adam) over its samples
        dict(name="train_surrogate_128k", kind="train", samples=131072, batch=16384),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["build"] * 6 + ["geometry", "pack", "gradient", "hessian", "train"])
    if kind == "train":
        batch = log_int(2000, 32768)
        return dict(kind=kind, samples=min(262144, int(batch * rng.uniform(1.0, 9.0))), batch=batch)
    form = "fp64" if kind in ("gradient", "hessian") else "mixed" if kind == "pack" else rng.choice(["fp64", "mixed"])
    func = rng.choice(["SVWN5", "PBE", "B3LYP", "R2SCAN", "R2SCAN"] if kind in ("build", "geometry") else ["PBE", "B3LYP"])
    mol = "alkane" if kind == "pack" else rng.choice(["water", "water", "alkane", "ring"])
    basis = rng.choice((["sto-3g"] if mol == "water" else []) + ["cc-pvdz", "def2-svp", "def2-svp", "def2-tzvp"])
    grid = rng.choice(["SG-1", "SG-2", "SG-3"]) if kind == "build" else "SG-1"
    spin = 1
    if kind == "build" and func in ("PBE", "R2SCAN") and rng.random() < 0.3:
        spin, func = 2, "PBE"
    big = {"water": 128, "alkane": 40, "ring": 18}[mol]
    if kind == "hessian":
        big = {"water": 2, "alkane": 2, "ring": 6}[mol]
    elif kind == "gradient":
        big = {"water": 12, "alkane": 10, "ring": 18}[mol]
    elif kind == "geometry":
        big = {"water": 32, "alkane": 24, "ring": 18}[mol]
    elif form == "fp64":
        big = {"water": 16, "alkane": 16, "ring": 18}[mol]
    elif func == "R2SCAN":
        big = {"water": 48, "alkane": 40, "ring": 18}[mol]
    if basis == "def2-tzvp" or grid == "SG-3":
        big = max(1 if mol != "ring" else 6, big if mol == "ring" else big // 3)
    elif spin == 2:
        big = max(1, big // 2)
    n = log_int(6 if mol == "ring" else 1, big)
    if mol == "ring":
        n = max(6, n - n % 2)
    case = dict(kind=kind, mol=mol, n=n, basis=basis, grid=grid, func=func, form=form,
                io=rng.choice(["host", "device"]) if kind == "build" else "host", spin=spin)
    if kind == "pack":
        case.update(n=min(n, 24), count=rng.randint(3, 24), basis="def2-svp", io="device")
    return case


# ---- geometries (angstrom) ------------------------------------------------------------------------
def _water(n, rng):
    """A droplet: the n cells of a jittered 3.1 A lattice nearest to its centre, each molecule turned at random."""
    m = math.ceil(n ** (1 / 3)) + 1
    cells = np.stack(np.meshgrid(*[np.arange(m) - 0.5 * (m - 1)] * 3, indexing="ij"), -1).reshape(-1, 3) * 3.1
    cells = cells[np.argsort((cells ** 2).sum(1), kind="stable")[:n]]
    half, r = math.radians(104.52) / 2, 0.9572
    mono = np.array([[0, 0, 0], [r * math.sin(half), 0, r * math.cos(half)], [-r * math.sin(half), 0, r * math.cos(half)]])
    xyz = []
    for c in cells:
        q, _ = np.linalg.qr(rng.standard_normal((3, 3)))
        xyz.append(mono @ q.T + c + rng.uniform(-0.1, 0.1, 3))
    return [8, 1, 1] * n, np.concatenate(xyz), 5 * n


def _alkane(n, rng):
    """All-trans C_nH_2n+2 with bond lengths jittered by 0.02 A."""
    half = math.radians(109.4712206) / 2
    up = lambda i: np.array([math.sin(half), math.cos(half) * (1 if i % 2 == 0 else -1), 0.0])  # noqa: E731
    jit = lambda: rng.uniform(-0.02, 0.02)  # noqa: E731
    C = [np.zeros(3)]
    for i in range(n - 1):
        C.append(C[-1] + (1.53 + jit()) * up(i))
    Z, xyz = [6] * n, list(C)
    for i in range(n):
        back, ahead = -up(i - 1), up(i)
        b = -(back + ahead) / np.linalg.norm(back + ahead)
        p = np.cross(back, ahead)
        p /= np.linalg.norm(p)
        dirs = [b * math.cos(half) + p * math.sin(half), b * math.cos(half) - p * math.sin(half)]
        dirs += ([back] if i == 0 else []) + ([ahead] if i == n - 1 else [])
        for d in dirs:
            Z.append(1)
            xyz.append(C[i] + (1.09 + jit()) * d)
    return Z, np.array(xyz), 4 * n + 1


def _ring(n, rng):
    """Carbon ring with bonds near 1.29 A."""
    R = 1.29 / (2 * math.sin(math.pi / n))
    a = 2 * math.pi * np.arange(n) / n + rng.uniform(-0.02, 0.02, n) * 2 * math.pi / n
    return [6] * n, np.stack([R * np.cos(a), R * np.sin(a), 0.01 * rng.standard_normal(n)], 1), 3 * n


def _molecule(mol, n, rng):
    Z, xyz, nocc = {"water": _water, "alkane": _alkane, "ring": _ring}[mol](n, rng)
    return np.array(Z, np.int32), xyz * BOHR, nocc


def _lengths(case):
    """Carbon counts of a pack's molecules: spread over 1..n."""
    return [1 + (7 * k) % case["n"] for k in range(case["count"])]


# ---- basis sets -------------------------------------------------------------------------------------
_R3, _R6, _R10, _R15 = math.sqrt(3), math.sqrt(6), math.sqrt(10), math.sqrt(15)
# component polynomials by angular momentum: lists of (coefficient, i, j, k) for x^i y^j z^k
POLY = {
    0: [[(1, 0, 0, 0)]],
    1: [[(1, 1, 0, 0)], [(1, 0, 1, 0)], [(1, 0, 0, 1)]],
    2: [[(_R3, 1, 1, 0)], [(_R3, 0, 1, 1)], [(1, 0, 0, 2), (-0.5, 2, 0, 0), (-0.5, 0, 2, 0)], [(_R3, 1, 0, 1)],
        [(0.5 * _R3, 2, 0, 0), (-0.5 * _R3, 0, 2, 0)]],
    3: [[(0.75 * _R10, 2, 1, 0), (-0.25 * _R10, 0, 3, 0)], [(_R15, 1, 1, 1)],
        [(_R6, 0, 1, 2), (-0.25 * _R6, 2, 1, 0), (-0.25 * _R6, 0, 3, 0)],
        [(1, 0, 0, 3), (-1.5, 2, 0, 1), (-1.5, 0, 2, 1)],
        [(_R6, 1, 0, 2), (-0.25 * _R6, 3, 0, 0), (-0.25 * _R6, 1, 2, 0)],
        [(0.5 * _R15, 2, 0, 1), (-0.5 * _R15, 0, 2, 1)], [(0.25 * _R10, 3, 0, 0), (-0.75 * _R10, 1, 2, 0)]],
}


@functools.lru_cache(None)
def _basis(name):
    """{Z: [(l, exponents, normalised coefficients)]} of a Gaussian-94 file."""
    lib, cur, z = {}, [], 0
    lines = iter(open(os.path.join(DATA, "BasisSets", name + ".gbs")))
    num = lambda t: float(t.upper().replace("D", "E"))  # noqa: E731
    for line in lines:
        w = line.split()
        if not w or w[0].startswith("!"):
            continue
        if w[0].startswith("-"):
            z, cur = {v.upper(): k for k, v in SYMBOL.items()}.get(w[0][1:].upper(), 0), []
        elif w[0] == "****":
            if z:
                lib[z] = cur
            z = 0
        else:
            rows = [[num(t) for t in next(lines).split()] for _ in range(int(w[1]))]
            for k, l in enumerate([0, 1] if w[0] == "SP" else ["SPDF".index(w[0])]):
                e, c = np.array([r[0] for r in rows]), np.array([r[1 + k] for r in rows])
                df, pi32 = math.prod(range(2 * l - 1, 0, -2)), math.pi ** 1.5
                c = c * np.sqrt(2.0 ** l * (2 * e) ** (l + 1.5) / (pi32 * df))
                s = (np.outer(c, c) * df * pi32 / (2.0 ** l * np.add.outer(e, e) ** (l + 1.5))).sum()
                cur.append((l, e, c / math.sqrt(s)))
    return lib


def _kinds(Z, basis):
    """The shells by kind: [(l, exponents, coefficients, atoms, AO columns (atoms x components))], and the AO count."""
    lib, off, by = _basis(basis), 0, {}
    for a, z in enumerate(Z):
        for k, (l, e, c) in enumerate(lib[int(z)]):
            m = 2 * l + 1
            by.setdefault((int(z), k), (l, e, c, [], []))[3].append(a)
            by[(int(z), k)][4].append(list(range(off, off + m)))
            off += m
    return [(l, torch.tensor(e, dtype=F64), torch.tensor(c, dtype=F64), at, torch.tensor(col)) for l, e, c, at, col in by.values()], off


def _overlap(kinds, n, xyz, dev):
    """Analytic overlap: Gauss-Hermite quadrature per direction (exact at these degrees)."""
    q, wq = (torch.tensor(v, dtype=F64, device=dev) for v in np.polynomial.hermite.hermgauss(4))
    S = torch.zeros(n, n, dtype=F64, device=dev)
    X = torch.as_tensor(xyz, dtype=F64, device=dev)
    for la, ea, ca, ata, cola in kinds:
        for lb, eb, cb, atb, colb in kinds:
            A, B = X[ata][:, None, :], X[atb][None, :, :]
            block = torch.zeros(len(ata), 2 * la + 1, len(atb), 2 * lb + 1, dtype=F64, device=dev)
            for i in range(len(ea)):
                for j in range(len(eb)):
                    a, b = float(ea[i]), float(eb[j])
                    p = a + b
                    P = (a * A + b * B) / p
                    x = q / math.sqrt(p) + P[..., None]  # [A, B, 3, q]
                    g = torch.exp(-a * b / p * (A - B) ** 2) / math.sqrt(p)
                    da, db = x - A[..., None], x - B[..., None]
                    one = {(u, v): g * (wq * da ** u * db ** v).sum(-1) for u in range(la + 1) for v in range(lb + 1)}
                    f = float(ca[i]) * float(cb[j])
                    for u, pu in enumerate(POLY[la]):
                        for v, pv in enumerate(POLY[lb]):
                            for (c1, i1, j1, k1) in pu:
                                for (c2, i2, j2, k2) in pv:
                                    block[:, u, :, v] += (f * c1 * c2) * one[i1, i2][..., 0] * one[j1, j2][..., 1] * one[k1, k2][..., 2]
            S[cola.reshape(-1, 1).to(dev), colb.reshape(1, -1).to(dev)] = block.reshape(cola.numel(), colb.numel())
    return S


def _density(Z, xyz, basis, nocc, rng, spin, dev):
    """D (or D_alpha, D_beta) of seeded localised orbitals, orthonormal in the overlap."""
    kinds, n = _kinds(Z, basis)
    nocc = min(nocc, n)
    S = _overlap(kinds, n, xyz, dev)
    weight, where = torch.zeros(n, dtype=F64), torch.zeros(n, 3, dtype=F64)
    X = torch.as_tensor(xyz, dtype=F64)
    for l, _, _, at, col in kinds:
        weight[col.reshape(-1)] = (1.0, 1.0, 0.15, 0.05)[l]
        where[col.reshape(-1)] = X[at].repeat_interleave(2 * l + 1, 0)
    centre = X[torch.arange(nocc) % len(Z)]
    fall = torch.exp(-torch.cdist(where, centre) / 2.5)
    C0 = torch.as_tensor(rng.standard_normal((n, nocc)))

    def d(C, f):
        C = (C * fall[:, :C.shape[1]] * weight[:, None]).to(dev)
        L = torch.linalg.cholesky(C.T @ S @ C)
        C = torch.linalg.solve_triangular(L, C.T, upper=False)
        return f * (C.T @ C)

    if spin == 1:
        return [d(C0, 2.0)]
    C1 = C0 + 0.2 * torch.as_tensor(rng.standard_normal((n, nocc)))
    return [d(C0, 1.0), d(C1[:, :max(1, nocc - 1)], 1.0)]


def _inputs(case, seed, k=0):
    """(Z, xyz in bohr, density matrices) of the case's molecule (a pack's k-th) for a seed."""
    rng = np.random.default_rng([int(seed), k])
    n = _lengths(case)[k] if case["kind"] == "pack" else case["n"]
    Z, xyz, nocc = _molecule(case["mol"], n, rng)
    return Z, xyz, _density(Z, xyz, case["basis"], nocc, rng, case["spin"], "cuda")


def _perturbations(D, seed):
    """Symmetric perturbed densities of a coupled-perturbed step (six of them)."""
    g = torch.Generator().manual_seed(int(seed) + 77)
    out = []
    for _ in range(6):
        K = 0.05 * torch.randn(D.shape, generator=g, dtype=F64).to(D.device)
        out.append(D @ K + K.T @ D)
    return out


def _samples(case, seed):
    """The learned functional's training set: descriptors in the box, smooth targets, energy-like weights."""
    rng = np.random.default_rng([int(seed), 5])
    U = rng.uniform(-1, 1, (case["samples"], 3)).astype(np.float32)
    T = (0.8 * np.tanh(1.5 * U[:, 0]) + 0.3 * np.sin(2.0 * U[:, 1] * U[:, 2]) + 0.1 * U[:, 2]).astype(np.float32)
    W = (0.5 + rng.exponential(0.5, case["samples"])).astype(np.float32)
    P = np.zeros(8641, np.float32)  # W1[64][3] b1 W2[64][64] b2 W3[64][64] b3 w4[64] b4
    for off, no, ni in ((0, 64, 3), (256, 64, 64), (4416, 64, 64), (8576, 1, 64)):
        P[off:off + no * ni] = rng.uniform(-1, 1, no * ni) * math.sqrt(6.0 / (no + ni))
    return U, T, W, P


# ---- the calls ----------------------------------------------------------------------------------------
def _grid(mol, case):
    import chinium_amd as ca

    g = ca.Grid(mol, case["grid"], 1, 0)
    g.setPrecision(ca.CHX_PREC_MIXED if case["form"] == "mixed" else ca.CHX_PREC_FP64)
    g.setType(CODES[case["func"]])
    g.getAO(0, 0)
    return g


def _host(Ds):
    return [np.asfortranarray(D.cpu().numpy()) for D in Ds]


def prepare(case, seed):
    import chinium_amd as ca

    if case["kind"] == "train":
        U, T, W, P = _samples(case, seed)
        m = ca.Surrogate(1)
        m.set_data(U, T, W)
        return dict(case=case, net=m, P=P)
    xc = ca.ExchangeCorrelation()
    xc.Spin = case["spin"]
    xc.Read(case["func"])
    s = dict(case=case, xc=xc)
    if case["kind"] == "pack":
        s.update(mols=[], grids=[], D=[], V=[])
        for k in range(case["count"]):
            Z, xyz, Ds = _inputs(case, seed, k)
            s["mols"].append(ca.Molecule(Z, xyz, case["basis"]))
            s["grids"].append(_grid(s["mols"][-1], case))
            s["D"].append(Ds[0].contiguous())
            s["V"].append(torch.empty_like(s["D"][-1]))
        s["pack"] = ca.Pack(s["grids"])
        s["Dp"], s["Vp"] = [D.data_ptr() for D in s["D"]], [V.data_ptr() for V in s["V"]]
        return s
    Z, xyz, Ds = _inputs(case, seed)
    mol = ca.Molecule(Z, xyz, case["basis"])
    s["mol"] = mol
    if case["kind"] == "geometry":
        s["D"] = _host(Ds)
        return s
    g = s["grid"] = _grid(mol, case)
    if case["kind"] == "build" and case["io"] == "device":
        s["D"] = torch.stack(Ds).contiguous()  # symmetric: column-major and row-major agree
        s["V"] = torch.empty_like(s["D"])
        return s
    s["D"] = _host(Ds)
    if case["kind"] in ("gradient", "hessian"):  # the converged iteration that these follow
        g.getDensity(s["D"])
        xc.Evaluate("ev", g)
    if case["kind"] == "hessian":
        s["Du"] = _host(_perturbations(Ds[0], seed))
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "train":
        s["net"].params = s["P"]
        loss = s["net"].train(1, case["batch"])
        return dict(params=s["net"].params, loss=loss)
    xc = s["xc"]
    if kind == "pack":
        E, N = s["pack"].xc(xc, s["Dp"], s["Vp"])
        return dict(E=E, N=N, V=s["V"])
    if kind == "gradient":
        g = s["grid"]
        g.getAO(1)
        g.getDensitySkeleton(s["D"])
        return dict(grad=g.getEnergyGrad())
    if kind == "hessian":
        g = s["grid"]
        g.getAO(2)
        xc.Evaluate("f", g)
        g.getDensitySkeleton2(s["D"])
        out = dict(hess=g.getEnergyHess(), skeleton=np.stack(g.getFockSkeleton()[0]), response=np.stack(g.getFockU(1, "s")[0]))
        g.getDensityU([s["Du"]])
        out["perturbed"] = np.stack(g.getFockU(1)[0])
        return out
    g = _grid(s["mol"], case) if kind == "geometry" else s["grid"]
    if case["io"] == "device":
        n = g.nbasis
        g.getDensityDevice(s["D"].data_ptr(), case["spin"], n)
        xc.Evaluate("ev", g)
        E = g.getEnergy()
        g.getFockDevice(s["V"].data_ptr(), case["spin"], n)
        return dict(E=np.array(E), N=np.array(g.getNumElectrons()), V=s["V"])
    g.getDensity(s["D"])
    xc.Evaluate("ev", g)
    E = g.getEnergy()
    return dict(E=np.array(E), N=np.array(g.getNumElectrons()), V=np.stack(g.getFock()))


# ---- what a pass cannot do without ----------------------------------------------------------------------
@functools.lru_cache(None)
def _points_per_atom(grid, z):
    rows = [line.split() for line in open(os.path.join(DATA, "Grids", grid, SYMBOL[z] + ".grid"))]
    return sum(int(r[0]) * int(r[1]) for r in rows[2:] if len(r) >= 2)


def _reach(case, n):
    """(points, AOs, sum over points of the AOs above 1e-14 there, squared): AOs counted at the points' own atom."""
    Z, xyz, _ = _molecule(case["mol"], n, np.random.default_rng(0))
    lib = _basis(case["basis"])
    R = np.sqrt(((xyz[:, None] - xyz[None]) ** 2).sum(-1))
    alive = np.zeros(len(Z))
    nao = 0
    for a, z in enumerate(Z):
        for l, e, _ in lib[int(z)]:
            alive += (2 * l + 1) * (R[a] < math.sqrt(math.log(1e14) / e.min()))
            nao += 2 * l + 1
    pts = np.array([_points_per_atom(case["grid"], int(z)) for z in Z])
    return float(pts.sum()), nao, float((pts * alive ** 2).sum()), len(Z)


def work(case):
    if case["kind"] == "train":
        n = case["samples"]
        return {"bytes": 20.0 * n + 8.0 * 8641, "flops": 6.0 * 8448 * n}
    b = f = 0.0
    for n in (_lengths(case) if case["kind"] == "pack" else [case["n"]]):
        pts, nao, a2, nat = _reach(case, n)
        # density and potential: one product each way; tau adds three symmetric ones (half each)
        build = {0: 2.0, 1: 4.0, 2: 10.0}[CODES[case["func"]]] * a2 * case["spin"]
        mat = 8.0 * nao * nao
        if case["kind"] == "gradient":
            f, b = f + 2.0 * a2, b + mat + 24.0 * nat + 32.0 * pts
        elif case["kind"] == "hessian":
            # D phi and D d_r phi, the six products of the Fock skeleton, the Hessian's six, one potential per
            # nuclear coordinate, one density and one potential per perturbed matrix
            f += (4 + 6 + 6 + 3 * nat + 2 * 6) * 2.0 * a2
            b += mat * (1 + 2 * 3 * nat + 2 * 6) + 72.0 * nat * nat + 32.0 * pts
        else:
            f, b = f + build, b + 2.0 * mat * case["spin"] + 32.0 * pts
    return {"bytes": b, "flops": f}


def tolerance(case):
    if case["kind"] == "train":
        return {"rel": 5e-6}  # FP32 sums (1.1e-6 off in the loss, 1e-7 in the weights)
    if case["form"] == "mixed":
        # products of 16 + 16 significant bits summed in FP32: V 1e-6 off, 8e-6 for a single methane
        return {"rel": 3e-5, "max": 3e-4}
    # 64-bit sums in another order: V 1e-13 off, the Hessian (whose terms cancel) 5e-13
    return {"rel": 2e-12, "max": 2e-11}


# ---- the path in 64 bits ----------------------------------------------------------------------------------
def _lebedev():
    rules, cur = {}, None
    for line in open(os.path.join(DATA, "lebedev_orbits.txt")):
        w = line.split()
        if not w or w[0] == "#":
            continue
        if w[0] == "rule":
            cur = rules.setdefault(int(w[1]), [])
            continue
        t, a, b, v = int(w[0]), float(w[1]), float(w[2]), float(w[3])
        g = {1: (1, 0, 0), 2: (0, math.sqrt(0.5), math.sqrt(0.5)), 3: (math.sqrt(1 / 3),) * 3,
             4: (a, a, math.sqrt(max(0.0, 1 - 2 * a * a))), 5: (a, math.sqrt(max(0.0, 1 - a * a)), 0),
             6: (a, b, math.sqrt(max(0.0, 1 - a * a - b * b)))}[t]
        seen = set()
        for p in ((0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0)):
            for s in range(8):
                q = tuple((-1 if s >> k & 1 else 1) * g[p[k]] + 0.0 for k in range(3))
                if q not in seen:
                    seen.add(q)
                    cur.append(q + (v,))
    return {k: np.array(v) for k, v in rules.items()}


def _quadrature(Z, xyz, grid, dev):
    """Points (G x 3) and Becke weights (G)."""
    rules, P, W, own = _lebedev(), [], [], []
    for a, z in enumerate(Z):
        rows = [line.split() for line in open(os.path.join(DATA, "Grids", grid, SYMBOL[int(z)] + ".grid"))]
        n = int(rows[0][1])
        i = np.arange(n)
        if rows[1][0] == "de2":
            al, x0, x1 = map(float, rows[1][1:4])
            h = (x1 - x0) / (n - 1)
            x = h * i + x0
            r, w = np.exp(al * x - np.exp(-x)), np.exp(3 * al * x - 3 * np.exp(-x)) * (al + np.exp(-x)) * h
        else:
            Rm, k = float(rows[1][1]), i + 1.0
            r, w = Rm * (k / (n + 1 - k)) ** 2, 2 * Rm ** 3 * (n + 1) * k ** 5 / (n + 1 - k) ** 7
        ang = [int(q[0]) for q in rows[2:] if len(q) >= 2 for _ in range(int(q[1]))]
        for s in range(n):
            L = rules[ang[s]]
            P.append(L[:, :3] * r[s] + xyz[a])
            W.append(4 * math.pi * w[s] * L[:, 3])
            own += [a] * len(L)
    P, W, own = torch.tensor(np.concatenate(P), device=dev), torch.tensor(np.concatenate(W), device=dev), torch.tensor(own, device=dev)
    X = torch.as_tensor(xyz, dtype=F64, device=dev)
    nat = len(Z)
    if nat > 1:
        Rab = torch.cdist(X, X, compute_mode="donot_use_mm_for_euclid_dist")
        for lo in range(0, len(W), 16384):
            p = P[lo:lo + 16384]
            d = torch.cdist(p, X, compute_mode="donot_use_mm_for_euclid_dist")
            cell = torch.empty_like(d)
            for b in range(nat):
                m = (d[:, b:b + 1] - d) / Rab[b]
                m[:, b] = 0
                for _ in range(3):
                    m = 1.5 * m - 0.5 * m ** 3
                m = 0.5 * (1 - m)
                m[:, b] = 1
                cell[:, b] = m.prod(1)
            W[lo:lo + 16384] *= cell.gather(1, own[lo:lo + 16384, None])[:, 0] / cell.sum(1)
    keep = W != 0
    return P[keep].contiguous(), W[keep].contiguous()


def _ao(kinds, n, X, P):
    """phi and its gradient at the points: [4, G, n]; X may carry a tangent or a gradient."""
    parts, cols = [], []
    for l, e, c, at, col in kinds:
        d = P[:, None, :] - X[at][None]
        r2 = (d * d).sum(-1)
        ex = c.to(P.device) * torch.exp(-r2[..., None] * e.to(P.device))
        R, R1 = ex.sum(-1), (-2.0 * ex * e.to(P.device)).sum(-1)  # grad R = R1 r
        pw = [[torch.ones_like(r2)] for _ in range(3)]
        for k in range(3):
            for _ in range(l):
                pw[k].append(pw[k][-1] * d[..., k])
        comp = []
        for poly in POLY[l]:
            q, g = 0.0, [0.0, 0.0, 0.0]
            for (f, *ijk) in poly:
                q = q + f * pw[0][ijk[0]] * pw[1][ijk[1]] * pw[2][ijk[2]]
                for k in range(3):
                    if ijk[k]:
                        u = list(ijk)
                        u[k] -= 1
                        g[k] = g[k] + f * ijk[k] * pw[0][u[0]] * pw[1][u[1]] * pw[2][u[2]]
            comp.append(torch.stack([R * q] + [R1 * d[..., k] * q + R * g[k] for k in range(3)]))
        parts.append(torch.stack(comp, -1).reshape(4, len(P), -1))
        cols.append(col.reshape(-1))
    order = torch.argsort(torch.cat(cols)).to(P.device)
    return torch.cat(parts, -1)[..., order]


_PI = math.pi
_PW = ((0.0310907, 0.21370, 7.5957, 3.5876, 1.6382, 0.49294), (0.01554535, 0.20548, 14.1189, 6.1977, 3.3662, 0.62517),
       (0.0168869, 0.11125, 10.357, 3.6231, 0.88026, 0.49671))


def _pw(rs, q, slope=False):
    s = rs.sqrt()
    Q = 2 * q[0] * (q[2] * s + q[3] * rs + q[4] * rs * s + q[5] * rs * rs)
    L = torch.log1p(1 / Q)
    if not slope:
        return -2 * q[0] * (1 + q[1] * rs) * L
    dQ = 2 * q[0] * (0.5 * q[2] / s + q[3] + 1.5 * q[4] * s + 2 * q[5] * rs)
    return -2 * q[0] * q[1] * L + 2 * q[0] * (1 + q[1] * rs) * dQ / (Q * Q + Q)


def _slater(r):
    return -0.75 * (3 / _PI) ** (1 / 3) * r ** (4 / 3)


def _vwn(rs, A, b, c, x0):
    x = rs.sqrt()
    X, Q, X0 = rs + b * x + c, math.sqrt(4 * c - b * b), x0 * x0 + b * x0 + c
    at = torch.atan(Q / (2 * x + b))
    return A * (torch.log(rs / X) + 2 * b / Q * at - b * x0 / X0 * (torch.log((x - x0) ** 2 / X) + 2 * (b + 2 * x0) / Q * at))


def _pbe_x(r, s):
    s2 = s / (4 * (3 * _PI ** 2) ** (2 / 3) * r ** (8 / 3))
    return _slater(r) * (1.804 - 0.804 / (1 + 0.219510 * s2 / 0.804))


def _pbe_c(r, z, s):
    g, beta = (1 - math.log(2)) / _PI ** 2, 0.06672632268006
    rs = (3 / (4 * _PI) / r) ** (1 / 3)
    ec, phi = _pw(rs, _PW[0]), 1.0
    if z is not None:
        up, dn = (1 + z).clamp_min(1e-15), (1 - z).clamp_min(1e-15)
        f = (up ** (4 / 3) + dn ** (4 / 3) - 2) / (2 ** (4 / 3) - 2)
        z4 = z ** 4
        ec = ec - _pw(rs, _PW[2]) * f * (1 - z4) * 9 * (2 ** (1 / 3) - 1) / 4 + (_pw(rs, _PW[1]) - ec) * f * z4
        phi = 0.5 * (up ** (2 / 3) + dn ** (2 / 3))
    t2 = s / (16 * phi ** 2 * (3 * _PI ** 2 * r) ** (1 / 3) / _PI * r * r)
    g3 = g * phi ** 3
    A = beta / g / torch.expm1(-ec / g3) * t2
    return r * (ec + g3 * torch.log1p(beta / g * t2 * (1 + A) / (1 + A + A * A)))


def _r2scan(r, s, t):
    eta, dp = 0.001, 0.361 ** 4
    cx = (1.0, -0.667, -0.4445555, -0.663086601049, 1.451297044490, -0.887998041597, 0.234528941479, -0.023185843322)
    cc = (1.0, -0.64, -0.4352, -1.535685604549, 3.061560252175, -1.915710236206, 0.516884468372, -0.051848879792)
    slope = lambda c: sum(i * v for i, v in enumerate(c))  # noqa: E731
    k2 = (3 * _PI ** 2) ** (2 / 3)
    p = s / (4 * k2 * r ** (8 / 3))
    tw = s / (8 * r)
    a = (t - tw) / (0.3 * k2 * r ** (5 / 3) + eta * tw)

    def switch(c, c1, c2, d):
        lo, mid, hi = a.clamp(max=0.0), a.clamp(0.0, 2.5), a.clamp(min=2.5)
        poly = sum(v * mid ** i for i, v in enumerate(c))
        return torch.where(a <= 0, torch.exp(-c1 * lo / (1 - lo)), torch.where(a <= 2.5, poly, -d * torch.exp(c2 / (1 - hi))))

    damp = torch.exp(-p * p / dp)
    x = ((20 / 27 + eta * 5 / 3) * -slope(cx) * (1 - 1.174) * damp + 10 / 81) * p
    h1 = 1.065 - 0.065 / (1 + x / 0.065)
    ex = _slater(r) * (h1 + switch(cx, 0.667, 0.8, 1.24) * (1.174 - h1)) * (1 - torch.exp(-4.9479 / p ** 0.25))
    g, b1, b2, b3 = (1 - math.log(2)) / _PI ** 2, 0.0285764, 0.0889, 0.125541
    rs = (3 / (4 * _PI) / r) ** (1 / 3)
    e1, d1 = _pw(rs, _PW[0]), _pw(rs, _PW[0], True)
    den = 1 + b2 * rs.sqrt() + b3 * rs
    e0, d0 = -b1 / den, b1 * (0.5 * b2 / rs.sqrt() + b3) / den ** 2
    w1 = torch.expm1(-e1 / g)
    y = 0.066725 * (1 + 0.1 * rs) / (1 + 0.1778 * rs) * (3 * _PI ** 2 / 16) ** (2 / 3) * p / rs / (g * w1)
    dy = slope(cc) / (27 * g * w1) * (20 * rs * (d0 - d1) - 45 * eta * (e0 - e1)) * p * damp
    c1 = e1 + g * torch.log1p(w1 * (1 - (1 + 4 * (y - dy)) ** -0.25))
    c0 = e0 + b1 * torch.log1p(torch.expm1(-e0 / b1) * (1 - (1 + 4 * 0.128026 * p) ** -0.25))
    return ex + r * (c1 + switch(cc, 0.64, 1.5, 0.7) * (c0 - c1))


def _energy(func, r, s, t):
    """Energy density of a closed shell."""
    rs = (3 / (4 * _PI) / r) ** (1 / 3)
    if func == "SVWN5":
        return _slater(r) + r * _vwn(rs, 0.0310907, 3.72744, 12.9352, -0.10498)
    if func == "PBE":
        return _pbe_x(r, s) + _pbe_c(r, None, s)
    if func == "R2SCAN":
        return _r2scan(r, s, t)
    h = (0.5 * r) ** (4 / 3)
    x = 0.5 * s.sqrt() / h
    b88 = -2 * h * (1.5 * (3 / (4 * _PI)) ** (1 / 3) + 0.0042 * x * x / (1 + 6 * 0.0042 * x * torch.asinh(x)))
    a, b, c, d, q = 0.04918, 0.132, 0.2533, 0.349, r ** (-1 / 3)
    dl = c * q + d * q / (1 + d * q)
    lyp = -a * r / (1 + d * q) - a * b * torch.exp(-c * q) / (1 + d * q) * (
        0.3 * (3 * _PI ** 2) ** (2 / 3) * r - r ** (-5 / 3) * s * (1 / 24 + 7 * dl / 72))
    return 0.08 * _slater(r) + 0.72 * b88 + 0.19 * r * _vwn(rs, 0.0310907, 13.0720, 42.7198, -0.409286) + 0.81 * lyp


def _live(r):
    return r >= 1e-15


def _potential(func, r, s, t):
    """e, v_rho, v_sigma, v_tau; points below the density threshold give nothing; sigma as libxc bounds it."""
    ok = _live(r)
    R = torch.where(ok, r, torch.ones_like(r)).detach().requires_grad_()
    T = torch.where(ok, t.clamp_min(1e-20), torch.ones_like(r))
    S = s.clamp_min(1e-40)
    if CODES[func] == 2:
        S = torch.minimum(S, 8 * R.detach() * T)
    S, T = S.detach().requires_grad_(), T.detach().requires_grad_()
    e = _energy(func, R, S, T)
    v = torch.autograd.grad(e.sum(), (R, S, T), allow_unused=True)
    return [torch.where(ok, x if x is not None else torch.zeros_like(r), torch.zeros_like(r)).detach() for x in (e, *v)]


def _contract(A, B):
    M = A.T @ B
    return M + M.T


def _build_exact(case, Z, xyz, Ds):
    """E, N and V per spin."""
    dev, func = Ds[0].device, case["func"]
    family = CODES[func]
    kinds, n = _kinds(Z, case["basis"])
    X = torch.as_tensor(xyz, dtype=F64, device=dev)
    P, W = _quadrature(Z, xyz, case["grid"], dev)
    E = N = 0.0
    V = [torch.zeros_like(D) for D in Ds]
    step = max(1024, int(2e8 / n))
    for lo in range(0, len(W), step):
        w = W[lo:lo + step]
        ao = _ao(kinds, n, X, P[lo:lo + step])
        rho, grad, tau = [], [], []
        for D in Ds:
            Y = ao[0] @ D
            rho.append((Y * ao[0]).sum(1))
            grad.append(torch.stack([2 * (Y * ao[k]).sum(1) for k in (1, 2, 3)]))
            tau.append(0.5 * sum(((ao[k] @ D) * ao[k]).sum(1) for k in (1, 2, 3)) if family == 2 else torch.zeros_like(w))
        if len(Ds) == 1:
            s = (grad[0] ** 2).sum(0)
            e, vr, vs, vt = _potential(func, rho[0], s, tau[0])
            fs = [(vr, 2 * vs * grad[0], vt)]
        else:
            e, fs = _pbe_pol(rho, grad)
        E, N = E + (w * e).sum(), N + (w * sum(rho)).sum()
        for k, (vr, c, vt) in enumerate(fs):
            B = (0.5 * w * vr)[:, None] * ao[0]
            if family >= 1:
                B = B + sum((w * c[j])[:, None] * ao[j + 1] for j in range(3))
            V[k] += _contract(ao[0], B)
            if family == 2:
                for j in (1, 2, 3):
                    V[k] += _contract(ao[j], (0.25 * w * vt)[:, None] * ao[j])
    return float(E), float(N), V


def _pbe_pol(rho, grad):
    """Spin-polarised PBE: e, and per spin (v_rho, the vector that multiplies grad phi, 0)."""
    ok = _live(rho[0] + rho[1])
    one = torch.ones_like(rho[0])
    sg = [(grad[0] ** 2).sum(0), (grad[0] * grad[1]).sum(0), (grad[1] ** 2).sum(0)]
    r = [torch.where(ok, x.clamp_min(1e-15), one).requires_grad_() for x in rho]
    s = [torch.where(ok, x if k == 1 else x.clamp_min(1e-40), one).requires_grad_() for k, x in enumerate(sg)]
    tot = r[0] + r[1]
    e = 0.5 * (_pbe_x(2 * r[0], 4 * s[0]) + _pbe_x(2 * r[1], 4 * s[2])) + _pbe_c(tot, (r[0] - r[1]) / tot, s[0] + 2 * s[1] + s[2])
    v = [torch.where(ok, x, torch.zeros_like(x)) for x in torch.autograd.grad(e.sum(), r + s)]
    return torch.where(ok, e, torch.zeros_like(e)).detach(), [
        (v[0], 2 * v[2] * grad[0] + v[3] * grad[1], None), (v[1], 2 * v[4] * grad[1] + v[3] * grad[0], None)]


def _fields(kinds, n, X, P, D):
    """rho and grad rho of a fixed D with the basis at X."""
    ao = _ao(kinds, n, X, P)
    Y = ao[0] @ D
    Yt = ao[0] @ D.T
    return (Y * ao[0]).sum(1), torch.stack([((Y + Yt) * ao[k]).sum(1) for k in (1, 2, 3)])


def _integrand(func, r, g):
    """v_rho and 2 v_sigma grad rho, differentiable."""
    e = lambda a, b: _energy(func, a, b, b).sum()  # noqa: E731
    s = (g ** 2).sum(0)
    vr, vs = torch.func.grad(e, (0, 1))(r, s)
    return vr, 2 * vs * g


def _derivatives_exact(case, seed, Z, xyz, D):
    """The gradient, or the Hessian case's four outputs: the basis moves, points and D stay."""
    dev, func = D.device, case["func"]
    kinds, n = _kinds(Z, case["basis"])
    X = torch.as_tensor(xyz, dtype=F64, device=dev)
    P, W = _quadrature(Z, xyz, case["grid"], dev)
    np3 = X.numel()
    hess = case["kind"] == "hessian"
    G = torch.zeros(np3, dtype=F64, device=dev)
    H = torch.zeros(np3, np3, dtype=F64, device=dev)
    FS, FR = (torch.zeros(np3, n, n, dtype=F64, device=dev) for _ in range(2))
    Du = _perturbations(D, seed) if hess else []
    FU = torch.zeros(len(Du), n, n, dtype=F64, device=dev)
    step = 8192 if hess else max(2048, int(2e7 / n))

    def matrix(ao, w, a, c):
        return _contract(ao[0], (0.5 * w * a)[:, None] * ao[0] + sum((w * c[j])[:, None] * ao[j + 1] for j in range(3)))

    for lo in range(0, len(W), step):
        p, w = P[lo:lo + step], W[lo:lo + step]
        rho, grad = _fields(kinds, n, X, p, D)
        live = _live(rho) & ((grad ** 2).sum(0) > 1e-40)
        p, w, rho, grad = p[live], w[live], rho[live], grad[:, live]
        fields = lambda x: _fields(kinds, n, x, p, D)  # noqa: E731
        if not hess:
            Xg = X.clone().requires_grad_()
            r, g = fields(Xg)
            (w * _energy(func, r, (g ** 2).sum(0), r)).sum().backward()
            G += Xg.grad.reshape(-1)
            continue
        a, c = _integrand(func, rho, grad)
        ao = _ao(kinds, n, X, p)
        energy = lambda x: (lambda f: (w * _energy(func, f[0], (f[1] ** 2).sum(0), f[0])).sum())(fields(x))  # noqa: E731
        for i in range(np3):
            T = torch.zeros(np3, dtype=F64, device=dev)
            T[i] = 1
            T = T.reshape(X.shape)
            H[i] += torch.func.jvp(torch.func.grad(energy), (X,), (T,))[1].reshape(-1)
            FS[i] += torch.func.jvp(lambda x: matrix(_ao(kinds, n, x, p), w, a, c), (X,), (T,))[1]
            dr, dg = torch.func.jvp(fields, (X,), (T,))[1]
            da, dc = torch.func.jvp(lambda u, v: _integrand(func, u, v), (rho, grad), (dr, dg))[1]
            FR[i] += matrix(ao, w, da, dc)
        for i, d in enumerate(Du):
            dr, dg = _fields(kinds, n, X, p, d)
            da, dc = torch.func.jvp(lambda u, v: _integrand(func, u, v), (rho, grad), (dr, dg))[1]
            FU[i] += matrix(ao, w, da, dc)
    if not hess:
        return dict(grad=G.reshape(-1, 3))
    return dict(hess=H, skeleton=FS, response=FR, perturbed=FU)


def _train_exact(case, seed):
    """Adam over the minibatches in order, in 64 bits: learning rate cosine-decayed from 3e-3 to 3e-5."""
    U, T, W, P = (torch.tensor(v, dtype=F64, device="cuda") for v in _samples(case, seed))
    P.requires_grad_()
    m, v = torch.zeros_like(P), torch.zeros_like(P)
    n, batch = case["samples"], case["batch"]
    steps, losses = math.ceil(n / batch), []
    for k in range(steps):
        sl = slice(k * batch, min(n, (k + 1) * batch))
        h = torch.tanh(U[sl] @ P[:192].reshape(64, 3).T + P[192:256])
        h = torch.tanh(h @ P[256:4352].reshape(64, 64).T + P[4352:4416])
        h = torch.tanh(h @ P[4416:8512].reshape(64, 64).T + P[8512:8576])
        loss = (W[sl] * (h @ P[8576:8640] + P[8640] - T[sl]) ** 2).sum() / W[sl].sum()
        g, = torch.autograd.grad(loss, P)
        losses.append(float(loss.detach()))
        lr = 3e-5 + 0.5 * (3e-3 - 3e-5) * (1 + math.cos(math.pi * k / max(1, steps)))
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        with torch.no_grad():
            P -= lr * (m / (1 - 0.9 ** (k + 1))) / ((v / (1 - 0.999 ** (k + 1))).sqrt() + 1e-8)
    return dict(params=P.detach(), loss=np.array([np.mean(losses)]))


def exact(case, seed):
    if case["kind"] == "train":
        return _train_exact(case, seed)
    if case["kind"] == "pack":
        got = [_build_exact(case, *_inputs(case, seed, k)) for k in range(case["count"])]
        return dict(E=np.array([g[0] for g in got]), N=np.array([g[1] for g in got]), V=[g[2][0] for g in got])
    if case["mol"] == "water" and case["n"] > 60:
        return None  # the Becke partition alone takes over 20 seconds in plain torch
    Z, xyz, Ds = _inputs(case, seed)
    if case["kind"] in ("gradient", "hessian"):
        return _derivatives_exact(case, seed, Z, xyz, Ds[0])
    E, N, V = _build_exact(case, Z, xyz, Ds)
    return dict(E=np.array(E), N=np.array(N), V=torch.stack(V))
