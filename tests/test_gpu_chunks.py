"""AO lists of batch chunks (shell-level screening, dense blocks gathered from D, M scattered back)
at the sizes where the packing can go wrong: one AO, less than a tile, one tile exactly, shells that
straddle tiles, many chunks whose lists differ, and every Vxc run length."""
import numpy as np
import pytest

import chinium_amd as ca
import oracle_lib as ol
from chinium_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _system(name):
    if name == "H":  # one s function; two electrons' worth of density in it
        Z, X, basis, nocc = [1], [[0.0, 0.0, 0.0]], "sto-3g", 1
    elif name == "water sto-3g":  # 7 AOs
        Z, X = wl.water_monomer_angstrom()
        basis, nocc = "sto-3g", 5
    elif name == "far hydrogens":  # 64 s functions, one or two alive in most batches
        Z, X, basis, nocc = [1] * 64, [[6.0 * (k % 8), 6.0 * (k // 8), 0.0] for k in range(64)], "sto-3g", 32
    else:  # C12 chain, 298 AOs: lists from 60 to 298 AOs, d shells across tile borders
        Z, X = wl.alkane_angstrom(12, 3)
        basis, nocc = "def2-svp", 49
    mol = ca.Molecule(np.array(Z), np.array(X, float) * ca.ANGSTROM_TO_BOHR, basis)
    D, _ = wl.workload_density(mol, nocc, 11)
    return mol, basis, D


def _grid(mol, family, form, cache=-1, thr=None, run=0):
    g = ca.Grid(mol, "SG-1", 1, 0)
    g.setPrecision(form)
    g.setAOCache(cache)
    if thr is not None:
        g.setScreening(thr)
    g.setType(family)
    g.setVxcChunk(run)
    g.getAO(0, 0)
    return g


@pytest.mark.parametrize("func", ["PBE", "R2SCAN"])
@pytest.mark.parametrize("name", ["H", "water sto-3g", "far hydrogens", "C12"])
def test_chunk_lists(name, func):
    print("chunk lists: %s %s" % (name, func), flush=True)
    mol, basis, D = _system(name)
    xc = ca.ExchangeCorrelation()
    xc.Read(func)
    fam = xc.family
    E, V = ca.xc_build(_grid(mol, fam, ca.CHX_PREC_FP64), xc, D)
    orc = ol.OracleSystem(mol.Z, mol.xyz, "SG-1", basis)
    orc.set_functional(func)
    orc.get_ao()
    Eo, _, Vo = orc.xc(D)
    assert abs(E - Eo) <= 1e-10 and np.abs(V - Vo).max() <= 1e-9
    scale = max(1.0, np.abs(V).max())
    # every list held in full: what the default threshold drops is below it in every factor
    for form, cache in ((ca.CHX_PREC_FP64, 1), (ca.CHX_PREC_FP64, 0)):
        E0, V0 = ca.xc_build(_grid(mol, fam, form, cache, thr=0.0), xc, D)
        assert abs(E0 - E) <= 1e-11 and np.abs(V0 - V).max() <= 1e-11 * scale
    # other run lengths sum in another order only
    for run in (1, 5, 128):
        E1, V1 = ca.xc_build(_grid(mol, fam, ca.CHX_PREC_FP64, 1, run=run), xc, D)
        assert abs(E1 - E) <= 1e-11 and np.abs(V1 - V).max() <= 1e-12 * scale
    # mixed form, both block shapes: 16 significant bits per operand
    for shape in (0, 1):
        g = _grid(mol, fam, ca.CHX_PREC_MIXED)
        g.setVxcShape(shape)
        Em, Vm = ca.xc_build(g, xc, D)
        assert abs(Em - E) <= 1e-5 * len(mol.Z) and np.abs(Vm - V).max() <= 5e-5 * scale


def test_coarse_threshold_moves_little():
    """A shell below 1e-6 adds less than 1e-6 times the integral of |v| over the points it leaves."""
    mol, _, D = _system("C12")
    xc = ca.ExchangeCorrelation()
    xc.Read("PBE")
    E, V = ca.xc_build(_grid(mol, 1, ca.CHX_PREC_FP64), xc, D)
    g = _grid(mol, 1, ca.CHX_PREC_FP64, thr=1e-6)
    full = _grid(mol, 1, ca.CHX_PREC_FP64, thr=0.0)
    assert g.stats()["mean_tiles"] < full.stats()["mean_tiles"]
    E6, V6 = ca.xc_build(g, xc, D)
    assert abs(E6 - E) <= 1e-4 and np.abs(V6 - V).max() <= 1e-4


@pytest.mark.parametrize("form", [ca.CHX_PREC_FP64, ca.CHX_PREC_MIXED])
@pytest.mark.parametrize("name", ["H", "water sto-3g", "C12"])
def test_tau_of_a_nonsymmetric_matrix(name, form):
    """rho and tau are quadratic forms: an antisymmetric part of D adds nothing. A symmetric D takes half of
    tau's products, one with an antisymmetric part all of them; one with rounding-level asymmetry (products
    like C C^T formed elsewhere) gives the same by either. Bounds: the forms' own rounding, 2^-16 of
    sum |D| |d phi| |d phi| (mixed), of which tau is about 1/10 at these densities."""
    mol, _, D = _system(name)
    n = len(D)
    S = np.random.default_rng(5).standard_normal((n, n)) * np.abs(D).max() * 0.05
    g = _grid(mol, 2, form)
    out = []
    for M in (D, D + (S - S.T), D + 1e-16 * np.abs(D).max() * S):
        g.getDensity([M])
        rho, _, tau, w = g.pointDensity()
        out.append((rho[w != 0], tau[w != 0]))
    tol = 1e-12 if form == ca.CHX_PREC_FP64 else 2e-4
    for k in (1, 2):
        for a, b in zip(out[0], out[k]):
            assert np.abs(a - b).max() <= tol * np.abs(a).max()


@pytest.mark.parametrize("form,cache", [(ca.CHX_PREC_FP64, 1), (ca.CHX_PREC_FP64, 0), (ca.CHX_PREC_MIXED, -1)])
def test_no_shell_alive(form, cache):
    """A threshold above every value leaves empty lists: no electrons, no potential, zero derivatives."""
    mol, _, D = _system("water sto-3g")
    xc = ca.ExchangeCorrelation()
    xc.Read("PBE")
    g = _grid(mol, 1, form, cache, thr=1e6)
    E, V = ca.xc_build(g, xc, D)
    assert g.stats()["mean_tiles"] == 0 and E == 0 and not V.any() and g.getNumElectrons() == 0
    if form == ca.CHX_PREC_FP64 and cache:
        xc.Evaluate("f", g)
        g.getDensitySkeleton([D])
        assert not g.getEnergyGrad().any()
        assert not any(F.any() for F in g.getFockSkeleton()[0])
        assert not g.getEnergyHess().any()


def _constants(nsh, type_=0):
    """One hydrogen with nsh shells of exponent 0: every s function is 1 everywhere, every Cartesian p shell x, y, z."""
    mol = ca.Molecule([1], [[0.0, 0.0, 0.0]])
    for _ in range(nsh):
        mol.add_shell(0, type_, [0.0], [1.0])
    return mol


@pytest.mark.parametrize("shape", [0, 1])
def test_products_of_a_run_are_added_in_fp64(shape):
    """Phi_I^T B_J and B_I^T Phi_J of one run, each a sum of integers below 2^24 and so exact in FP32, add up exactly
    (in one FP32 accumulator they would pass 2^24 and lose their odd part)."""
    mol = _constants(200)  # 7 tiles: two groups
    g = _grid(mol, 0, ca.CHX_PREC_MIXED, run=7)
    g.setVxcShape(shape)
    w = g.points()[:, 3]
    a = np.random.default_rng(8).integers(0, 30000, len(w)) * 2 + 1  # 16 bits: hi + lo holds them
    assert 7 * 64 * 60000 * 1.05 > 2 ** 24 > 7 * 64 * 30000 * 1.05
    g.setVrho(2 * a / w)  # the integrand's factor is w v_rho / 2
    V = g.getFock(1)[0]
    assert np.array_equal(V, np.full(V.shape, 2.0 * a.sum()))


@pytest.mark.parametrize("form", [ca.CHX_PREC_FP64, ca.CHX_PREC_MIXED])
def test_directions_of_tau_are_added_in_fp64(form):
    """Of the functions x, y, z each has one constant derivative: tau is half the trace of D, and an entry of 2^26 next to
    ones of 1 (each exact in FP32) shows a sum over the directions in FP32."""
    mol = _constants(1, 1)
    g = _grid(mol, 2, form)
    a = 65535.0 * 2 ** 10
    g.getDensity([np.diag([a, 1.0, 1.0])])
    _, _, tau, w = g.pointDensity()
    assert np.array_equal(tau[w != 0], np.full((w != 0).sum(), 0.5 * (a + 2.0)))


@pytest.mark.parametrize("form", [ca.CHX_PREC_FP64, ca.CHX_PREC_MIXED])
def test_autotuner_has_the_default_among_its_lengths(form):
    """The default rule's run length (1 to 4 batches in FP64 and in small systems) is one of those timed."""
    from chinium_amd import hip
    mol, _, D = _system("water sto-3g")
    xc = ca.ExchangeCorrelation()
    xc.Read("PBE")
    g = _grid(mol, 1, form)
    E, V = ca.xc_build(g, xc, D)
    n = len(D)
    dD, dV = hip.DeviceArray(n * n), hip.DeviceArray(n * n)
    dD.upload(np.asfortranarray(D).ravel(order="F"))
    chunk, ms = g.autotune(xc, dD.ptr, dV.ptr, reps=1)
    assert 0 in ms and ms[chunk] == min(ms.values())
    g.setVxcChunk(0)
    E0, V0 = ca.xc_build(g, xc, D)
    assert np.array_equal(V, V0)


@pytest.mark.parametrize("n", [505, 512, 513, 8200])
def test_assembly_by_basis_size(n):
    """V's assembly from the runs' blocks: a copy of the sums per wave up to 512 AOs (64 KB of LDS there, and no more
    than that left over), one for all above, two column ranges from 8193 on; against the form that adds to M. All
    terms of a density of positive orbitals have one sign: 16 bits per operand give 3 x 2^-17 of V's largest."""
    print("assembly: %d AOs" % n, flush=True)
    rng = np.random.default_rng(n)
    mol = ca.Molecule([1], [[0.0, 0.0, 0.0]])
    for e in rng.uniform(0.1, 20.0, n):
        mol.add_shell(0, 0, [e], [(2 * e / np.pi) ** 0.75])
    C = rng.uniform(0.1, 1.0, (n, 2)) / n
    D = C @ C.T
    xc = ca.ExchangeCorrelation()
    xc.Read("PBE")
    E0, V0 = ca.xc_build(_grid(mol, 1, ca.CHX_PREC_FP64, 0), xc, D)
    E, V = ca.xc_build(_grid(mol, 1, ca.CHX_PREC_FP64, 1), xc, D)
    scale = np.abs(V0).max()
    assert abs(E - E0) <= 1e-12 * abs(E0) and np.abs(V - V0).max() <= 1e-12 * scale
    assert np.array_equal(V, V.T)
    Em, Vm = ca.xc_build(_grid(mol, 1, ca.CHX_PREC_MIXED), xc, D)
    assert abs(Em - E0) <= 5e-5 * abs(E0) and np.abs(Vm - V0).max() <= 5e-5 * scale
