"""Density-fitted J/K on the GPU (mjk_df_*) against the oracle and the
reference's golden values.

* The raw integrals (a build with lindep < 0 keeps (ij|P)) and (P|Q) equal
  the oracle's to 1e-12 relative (same Rys formulation, different code).
* The fitted tensor and J/K of random densities equal the oracle's fit to
  the FP64 contract (1e-10), for H2O cc-pVDZ / weigend (g auxiliary
  functions), a cc-pVDZ chain with generally contracted s shells /
  cc-pVDZ-JKFIT, and a def2-TZVP chain (f orbital shells) /
  def2-universal-JKFIT (g).
* Golden values of pyscf/df/test/test_df_jk.py: lib.fp(vj), lib.fp(vk) of
  the seed-1 densities (9 places) and the DF-RHF energy (8 places).
* K from occupied orbitals (the SCF path) equals K of their density.
* The matrix-core exchange products on odd and even AO counts against the
  oracle, and at the edges of their tiles against numpy; the Cholesky factor at
  the edges of its blocks, and the eigenvector fit where it fails.
"""
import numpy
import pytest

from pyscf_amd import df, gto, lib, workloads
from pyscf_amd.scf import _vhf, rhf

pytestmark = pytest.mark.gpu
H2O = 'O 0 0 0; H 0 -0.757 0.587; H 0 0.757 0.587'
TOL = 1e-10

CASES = {
    'h2o_weigend': (lambda: gto.M(atom=H2O, basis='cc-pvdz'), 'weigend'),
    'chain_vdz_jkfit': (lambda: gto.M(atom=workloads.random_chain([8, 1], nmin=3, nmax=3), basis='cc-pvdz'),
                        None),
    'chain_tzvp_jkfit': (lambda: gto.M(atom=workloads.random_chain([8, 2], nmin=2, nmax=2), basis='def2-tzvp'),
                         None),
}


def dens(nao, seed, n=2, sym=False):
    d = numpy.random.default_rng(seed).standard_normal((n, nao, nao)) / nao
    return d + d.transpose(0, 2, 1) if sym else d


@pytest.mark.parametrize('name', sorted(CASES))
def test_raw_integrals(oracle, name):
    mk, auxbasis = CASES[name]
    mol = mk()
    d = df.DF(mol, auxbasis)
    d.lindep = -1.0      # keep the raw (ij|P)
    d.build()
    aux = d.auxmol
    raw = d.cderi()      # (naux, nao, nao) = (ij|P) transposed
    j3 = oracle.int3c2e(mol, aux)
    ref = j3.transpose(2, 0, 1)
    scale = abs(ref).max()
    print(name, mol.nao_nr(), aux.nao_nr(), 'max|d3c|=%.2e (max %.2e)' % (abs(raw - ref).max(), scale), flush=True)
    assert abs(raw - ref).max() <= 1e-12 * scale
    j2 = numpy.empty((aux.nao_nr(), aux.nao_nr()))
    d.engine.check(d.engine.lib.mjk_df_fetch(d.engine.handle, d.handle, 0, j2.ctypes.data_as(lib.ctypes.c_void_p)),
                   'mjk_df_fetch')
    j2o = oracle.int2c2e(mol, aux)
    assert abs(j2 - j2o).max() <= 1e-12 * abs(j2o).max()


@pytest.mark.parametrize('name', sorted(CASES))
def test_fit_and_jk_vs_oracle(oracle, name):
    mk, auxbasis = CASES[name]
    mol = mk()
    nao = mol.nao_nr()
    d = df.DF(mol, auxbasis).build()
    cd = oracle.cholesky_eri(mol, d.auxmol)
    b = d.cderi()
    assert b.shape == cd.shape
    print(name, 'max|dB|=%.2e' % abs(b - cd).max(), flush=True)
    assert abs(b - cd).max() <= TOL
    for hermi, sym in ((0, False), (1, True)):
        dms = dens(nao, 7 + hermi, sym=sym)
        vj, vk = df.get_jk(d, dms, hermi)
        j0, k0 = oracle.df_get_jk(cd, dms, hermi)
        print('  hermi=%d max|dJ|=%.2e max|dK|=%.2e' % (hermi, abs(vj - j0).max(), abs(vk - k0).max()), flush=True)
        assert abs(vj - j0).max() <= TOL and abs(vk - k0).max() <= TOL


def test_exchange_odd_and_even_aos(oracle):
    """The exchange products on the matrix cores, whose columns of an odd number of
    AOs or fitting functions start at 8-byte addresses: NH3 cc-pVDZ (29 AOs) and
    H2O cc-pVDZ (24 AOs), general and occupied-orbital paths, against the
    oracle's fit."""
    nh3 = 'N 0 0 0.11; H 0 0.94 -0.26; H 0.81 -0.47 -0.26; H -0.81 -0.47 -0.26'
    for atom in (nh3, H2O):
        mol = gto.M(atom=atom, basis='cc-pvdz')
        nao = mol.nao_nr()
        d = df.DF(mol, 'weigend').build()
        cd = oracle.cholesky_eri(mol, d.auxmol)
        for hermi, sym in ((0, False), (1, True)):
            dms = dens(nao, 11 + hermi, sym=sym)
            vj, vk = df.get_jk(d, dms, hermi)
            j0, k0 = oracle.df_get_jk(cd, dms, hermi)
            print(nao, 'hermi=%d max|dJ|=%.2e max|dK|=%.2e'
                  % (hermi, abs(vj - j0).max(), abs(vk - k0).max()), flush=True)
            assert abs(vj - j0).max() <= TOL and abs(vk - k0).max() <= TOL
        rng = numpy.random.default_rng(3)
        c = rng.standard_normal((nao, nao)) / nao
        occ = numpy.zeros(nao)
        occ[:5] = 2.0
        dm = 2.0 * c[:, :5] @ c[:, :5].T
        vj, vk = df.get_jk(d, lib.tag_array(dm, mo_coeff=c, mo_occ=occ), 1)
        j0, k0 = oracle.df_get_jk(cd, dm[None], 1)
        print(nao, 'orbitals max|dK|=%.2e' % abs(vk - k0[0]).max(), flush=True)
        assert abs(vj - j0[0]).max() <= TOL and abs(vk - k0[0]).max() <= TOL


def test_golden_fingerprints():
    mol = gto.M(atom=H2O, basis='cc-pvdz')
    d = df.DF(mol, 'weigend')
    dms = numpy.random.RandomState(1).random_sample((2, 24, 24))
    vj, vk = df.get_jk(d, dms, hermi=0)
    print('fp(vj)=%.12f fp(vk)=%.12f' % (lib.fp(vj), lib.fp(vk)), flush=True)
    assert abs(lib.fp(vj) - -194.15910890730066) < 1e-9
    assert abs(lib.fp(vk) - -46.365071587653517) < 1e-9


def test_df_rhf_golden_and_orbital_path():
    mol = gto.M(atom=H2O, basis='cc-pvdz')
    mf = rhf.RHF(mol).density_fit(auxbasis='weigend')
    mf.conv_tol = 1e-11
    e = mf.kernel()
    print('DF-RHF E=%.12f (%d cycles)' % (e, mf.cycles), flush=True)
    assert mf.converged and abs(e - -76.025936299702536) < 1e-8
    # K from the occupied orbitals equals K of their density
    dm = mf.make_rdm1(mf.mo_coeff, mf.mo_occ)
    vj1, vk1 = df.get_jk(mf.with_df, dm, 1)
    vj2, vk2 = df.get_jk(mf.with_df, numpy.asarray(dm).copy(), 1)
    assert abs(vj1 - vj2).max() <= 1e-12 and abs(vk1 - vk2).max() <= 1e-11


def test_cderi_packed_layout():
    mol = gto.M(atom=H2O, basis='cc-pvdz')
    d = df.DF(mol, 'weigend').build()
    b = d.cderi()
    packed = d._cderi
    i, j = numpy.tril_indices(24)
    assert packed.shape == (d.get_naoaux(), 24 * 25 // 2)
    assert abs(packed - b[:, i, j]).max() == 0 and abs(b - b.transpose(0, 2, 1)).max() <= 1e-13 * abs(b).max()


def test_device_resident_df_rhf():
    """The density-fitted RHF with the whole loop on the device (mjk_rhf_set_df)
    against the host-driven density-fitted RHF and the reference's golden
    energy."""
    mol = gto.M(atom=H2O, basis='cc-pvdz')
    dev = rhf.DeviceRHF(mol).density_fit(auxbasis='weigend')
    dev.conv_tol = 1e-11
    e = dev.kernel()
    print('device DF-RHF E=%.12f (%d cycles)' % (e, dev.cycles), flush=True)
    assert dev.converged and abs(e - -76.025936299702536) < 1e-8
    mol = CASES['chain_vdz_jkfit'][0]()
    host = rhf.RHF(mol).density_fit()
    host.conv_tol = 1e-11
    eh = host.kernel()
    dev = rhf.DeviceRHF(mol).density_fit()
    dev.conv_tol = 1e-11
    ed = dev.kernel()
    print('chain DF-RHF host %.12f device %.12f' % (eh, ed), flush=True)
    assert host.converged and dev.converged and abs(eh - ed) < 1e-9


@pytest.mark.parametrize('size', [1, 2, 4])
def test_exchange_matrix_core_tiles(size):
    """The exchange products of random orbitals (1 to 7 column groups: both
    sides of a sixteen, of a panel of six groups and of an odd inner length)
    and of a general density against numpy on the fitted tensor; water
    clusters of 24, 48 and 96 AOs lie on both sides of a 64-wide tile.  Sums of up to
    1e5 products of size ~1 / 100 in 64 bits: 1e-12 of the largest element."""
    mol = gto.M(atom=workloads.water_cluster(size, shape=(4, 1, 1)), basis='cc-pvdz')
    d = df.DF(mol, 'weigend').build()
    b = d.cderi()
    nao = b.shape[1]
    rng = numpy.random.default_rng(size)
    for nocc in (1, 5, 16, 17, 96, 97):
        c = rng.standard_normal((nao, nocc)) / 10
        dm = c @ c.T
        vj, vk = df.get_jk(d, lib.tag_array(dm, mo_coeff=c, mo_occ=numpy.ones(nocc)), 1)
        y = numpy.einsum('pij,jo->pio', b, c, optimize=True)
        k0 = numpy.einsum('pio,pjo->ij', y, y, optimize=True)
        j0 = numpy.tensordot(numpy.tensordot(b, dm, 2), b, (0, 0))
        assert abs(vk - k0).max() <= 1e-12 * abs(k0).max(), (nao, nocc)
        assert abs(vj - j0).max() <= 1e-12 * abs(j0).max(), (nao, nocc)
        assert (vk == vk.T).all()
    dm = rng.standard_normal((nao, nao)) / 10
    vj, vk = df.get_jk(d, dm, 0)
    k0 = numpy.einsum('pij,jk,pkl->il', b, dm, b, optimize=True)
    assert abs(vk - k0).max() <= 1e-12 * abs(k0).max()


@pytest.mark.parametrize('n', [1, 31, 32, 33, 97, 161])
def test_fit_factor_block_edges(n):
    """The blocked Cholesky factor of (P|Q) at the edges of its 32-column blocks
    and 64-row tiles, and the auxiliary transform at the ends of its row groups:
    n atoms with one s function each.  Both fits are backward stable, so they
    differ by less than 8 n eps cond(L) of the largest element."""
    import scipy.linalg
    g = numpy.array([(i % 6, i // 6 % 6, i // 36) for i in range(n)]) * 3.0
    g += numpy.random.default_rng(n).uniform(-0.4, 0.4, g.shape)
    mol = gto.M(atom=[('H', tuple(x)) for x in g], unit='bohr', basis={'H': [[0, (0.5, 1.0)]]}, spin=n % 2)
    aux = {'H': [[0, (0.8, 1.0)]]}
    d = df.DF(mol, aux)
    d.lindep = -1.0
    raw = d.build().cderi().reshape(n, -1)
    j2 = numpy.empty((n, n))
    d.engine.check(d.engine.lib.mjk_df_fetch(d.engine.handle, d.handle, 0, j2.ctypes.data_as(lib.ctypes.c_void_p)),
                   'mjk_df_fetch')
    L = numpy.linalg.cholesky(j2)
    ref = scipy.linalg.solve_triangular(L, raw, lower=True)
    fit = df.DF(mol, aux).build().cderi().reshape(n, -1)
    assert abs(fit - ref).max() <= 8 * n * 2.3e-16 * numpy.linalg.cond(L) * abs(ref).max()


@pytest.mark.parametrize('size', [1, 4])
def test_exchange_scratch_within_the_fit_workspace(size):
    """A J/K call takes no device memory for its exchange products beyond the
    half-transformed tensor: a budget of the fitted tensor, that and the call's
    densities, J, K and fitting coefficients is enough."""
    mol = gto.M(atom=workloads.water_cluster(size, shape=(4, 1, 1)), basis='cc-pvdz')
    nao = mol.nao_nr()
    dm = numpy.random.default_rng(size).standard_normal((nao, nao))
    d = df.DF(mol, 'weigend', engine=_vhf.Engine()).build()
    need = d.engine.hbm_used() + 8 * (d.get_naoaux() * (nao * nao + 1) + 3 * nao * nao)
    ref = df.get_jk(d, dm, 0)
    d2 = df.DF(mol, 'weigend', engine=_vhf.Engine(hbm_budget=need)).build()
    out = df.get_jk(d2, dm, 0)
    assert d2.engine.hbm_used() == need
    for x, r in zip(out, ref):
        assert abs(x - r).max() <= 1e-12 * abs(r).max()


def test_dependent_fitting_set_takes_the_eigenvector_fit():
    """Forty nearly equal s functions on one centre: (P|Q) is singular to FP64
    rounding (numpy's factorisation fails too), so the fit is over its
    eigenvalues above lindep.  J and K against numpy's eigenvector fit of the
    same integrals, which rounding of (P|Q) changes by up to
    n eps w_max / w_min of the kept eigenvalues."""
    mol = gto.M(atom=H2O, basis='cc-pvdz')
    aux = {'O': [[0, (0.3 * 1.03 ** k, 1.0)] for k in range(40)], 'H': [[0, (0.8, 1.0)]]}
    d = df.DF(mol, aux)
    d.lindep = -1.0
    raw = d.build().cderi()
    n = raw.shape[0]
    j2 = numpy.empty((n, n))
    d.engine.check(d.engine.lib.mjk_df_fetch(d.engine.handle, d.handle, 0, j2.ctypes.data_as(lib.ctypes.c_void_p)),
                   'mjk_df_fetch')
    with pytest.raises(numpy.linalg.LinAlgError):
        numpy.linalg.cholesky(j2)
    w, v = numpy.linalg.eigh(j2)
    keep = w > 1e-7
    fit = df.DF(mol, aux).build()
    assert fit.get_naoaux() == keep.sum() < n
    b = numpy.einsum('pk,pij->kij', v[:, keep] / numpy.sqrt(w[keep]), raw)
    dm = dens(mol.nao_nr(), 23)[0]
    vj, vk = df.get_jk(fit, dm, 0)
    j0 = numpy.einsum('pij,pkl,lk->ij', b, b, dm, optimize=True)
    k0 = numpy.einsum('pij,jk,pkl->il', b, dm, b, optimize=True)
    tol = n * 2.3e-16 * w[-1] / w[keep][0]
    assert abs(vj - j0).max() <= tol * abs(j0).max() and abs(vk - k0).max() <= tol * abs(k0).max()


def test_exchange_layout_by_column():
    """The half-transformed tensor is laid out by column from 2 MB a row on:
    orbital counts on both sides of that line (923 fitting functions, so 284 of
    them) and a general density (312 columns) against numpy on the fitted tensor,
    1e-12 of the largest element as for the small ones."""
    mol = gto.M(atom=workloads.water_cluster(13, shape=(4, 4, 1)), basis='cc-pvdz')
    d = df.DF(mol, 'weigend').build()
    b = d.cderi()
    naux, nao = b.shape[:2]
    assert (naux, nao) == (923, 312)
    rng = numpy.random.default_rng(13)
    for nocc in (284, 285, 0):
        if nocc:
            c = rng.standard_normal((nao, nocc)) / 10
            vk = df.get_jk(d, lib.tag_array(c @ c.T, mo_coeff=c, mo_occ=numpy.ones(nocc)), 1, with_j=False)[1]
            y = (b.reshape(-1, nao) @ c).reshape(naux, nao, nocc)
            k0 = sum(yp @ yp.T for yp in y)
            assert (vk == vk.T).all()
        else:
            dm = rng.standard_normal((nao, nao)) / 10
            vk = df.get_jk(d, dm, 0, with_j=False)[1]
            y = (b.reshape(-1, nao) @ dm).reshape(naux, nao, nao)
            k0 = sum(yp @ bp for yp, bp in zip(y, b))
        assert abs(vk - k0).max() <= 1e-12 * abs(k0).max(), nocc


@pytest.mark.parametrize('n', [1, 2, 3, 4, 5])
def test_exchange_few_fitting_functions(n):
    """Fewer fitting functions than a lane loads at once, and just as many."""
    mol = gto.M(atom=[('H', (0, 0, 1.1 * i)) for i in range(n)], basis='cc-pvdz', spin=n % 2)
    d = df.DF(mol, {'H': [[0, (0.8, 1.0)]]}).build()
    b = d.cderi()
    nao = b.shape[1]
    rng = numpy.random.default_rng(n)
    c = rng.standard_normal((nao, 3))
    vk = df.get_jk(d, lib.tag_array(c @ c.T, mo_coeff=c, mo_occ=numpy.ones(3)), 1)[1]
    y = numpy.einsum('pij,jo->pio', b, c)
    assert b.shape[0] == n and abs(vk - numpy.einsum('pio,pjo->ij', y, y)).max() <= 1e-12 * abs(vk).max()
    dm = rng.standard_normal((nao, nao))
    vk = df.get_jk(d, dm, 0)[1]
    assert abs(vk - numpy.einsum('pij,jk,pkl->il', b, dm, b)).max() <= 1e-12 * abs(vk).max()
