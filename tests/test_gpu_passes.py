"""The FFT passes' radix schedules and the P(k) bin edges at the sizes where they change:
one radix (8-16), a radix 12 first or reversed (12-192), no LDS stage, odd bin counts."""
import numpy as np
import pytest

import mgpicola as M
import oracle as O
from helpers import lattice_particles, rel_err

pytestmark = pytest.mark.gpu
BOX, OM = 64.0, 0.3


@pytest.mark.parametrize("model", ["lcdm", "fofr", "dgp"])
@pytest.mark.parametrize("n", [8, 12, 16, 24, 64, 96, 192])
@pytest.mark.parametrize("tcols", [8, 16])
def test_x_pass_pairs_and_screening_row(model, n, tcols):
    """GetDisplacements' paired x passes and screening rows against the oracle.  The force
    meshes hold FP32 rounding of 3 log2(n)-stage transforms: 3e-5 of the field maximum, the
    bound of the oracle comparisons of the separate passes."""
    ns = n // 2
    pos = lattice_particles(ns, BOX, amp=1.5, seed=n)
    kw, okw, mg, omg = {}, {}, None, None
    if model != "lcdm":
        d = dict(a=0.7, coupling=1 / 3 if model == "fofr" else 0.12, mass2=2e4, phi_crit=3e-8, dgp_fac=0.05,
                 rsmooth=2.0, geff=1.0)
        okw = dict(model=O.FOFR if model == "fofr" else O.DGP, mg_active=1, include_screening=1,
                   filter=O.FILTER_GAUSSIAN if model == "dgp" else O.FILTER_NONE)
        kw, mg, omg = dict(okw), M.MG(**d), O.MG(**d)
    print("model, n, tcols =", model, n, tcols, flush=True)
    g = M.MGPU(n, ns, BOX, OM, pofk_nbins=n // 2 + 1, pofk_subtract_shotnoise=0, **kw)
    g.set_fft_tile(0, tcols)
    g.set_particles(pos)
    g.get_displacements(mg=mg, pofk=True)  # records the mode counts
    _, (pk, _, nm) = g.get_displacements(mg=mg, pofk=True)
    c = O.cfg(n, ns, BOX, OM, **okw)
    dk = O.deposit(c, pos)
    dx = dk.copy()
    O.fft_r2c_3d(n, dk)
    rp, _, rn = O.pofk(c, dk, n // 2 + 1, 0, 0.0, float(n), 0)
    f = O.forces(c, dk, O.fifth_force(c, omg, dk, dx) if omg is not None else None)
    for a, mid in enumerate((M.MESH_FORCE_X, M.MESH_FORCE_Y, M.MESH_FORCE_Z)):
        assert rel_err(g.get_mesh(mid), O.real_view(f[a], n)) < 3e-5
    assert np.array_equal(nm, rn)
    ok = (rn > 0) & (np.arange(rn.size) > 0)
    np.testing.assert_allclose(pk[ok], rp[ok], rtol=1e-3)
    g.close()


@pytest.mark.parametrize("nbins,bintype,kmin,kmax", [(1, 0, 0.0, 48.0), (7, 0, 3.0, 11.5), (48, 1, 1.0, 48.0),
                                                     (333, 0, 0.0, 48.0), (500, 1, 2.5, 30.0)])
def test_pofk_bins_by_edges(nbins, bintype, kmin, kmax):
    """Every mode in the bin of the FP64 formula: mode counts equal the oracle's, for bins
    wider and finer than a mode, with modes below the first bin and past the last, in
    k_pofk (first call), the density x pass (second call) and the fused pair."""
    n, ns = 48, 24
    pos = lattice_particles(ns, BOX, amp=1.5, seed=5)
    g = M.MGPU(n, ns, BOX, OM, pofk_nbins=nbins, pofk_bintype=bintype, pofk_kmin=kmin, pofk_kmax=kmax,
               pofk_subtract_shotnoise=0)
    g.set_particles(pos)
    got = [g.pm_density(pofk=True), g.pm_density(pofk=True), g.get_displacements(pofk=True)[1]]
    c = O.cfg(n, ns, BOX, OM)
    dk = O.deposit(c, pos)
    O.fft_r2c_3d(n, dk)
    rp, rk, rn = O.pofk(c, dk, nbins, bintype, kmin, kmax, 0)
    ok = (rn > 0) & (rk > 0)
    for pk, kk, nm in got:
        assert np.array_equal(nm, rn)
        np.testing.assert_allclose(kk[ok], rk[ok], rtol=1e-12)
        # one lost or misplaced mode changes a sparse bin by its share of the power
        np.testing.assert_allclose(pk[ok], rp[ok], rtol=1e-3)
    g.close()


@pytest.mark.parametrize("ns,n", [(1, 8), (7, 16), (64, 96), (65, 96), (81, 96), (102, 128), (40, 384)])
def test_means_and_bins_over_particle_counts(ns, n):
    """The means for every number of particles per thread (up to 1024 blocks: 64^3, 65^3,
    81^3 and 102^3 take 1, 2, 4 and 8) against the particles' own FP64 means, and two
    deposits in a row, with a redshift-space one between, to the bit: the bin scan (one
    launch up to the 256 mesh, two beyond) leaves its counters cleared."""
    pos = lattice_particles(ns, BOX, amp=1.5, seed=ns, clustered=ns > 4)
    rng = np.random.default_rng(ns)
    vel = rng.normal(size=pos.shape).astype(np.float32)
    g = M.MGPU(n, ns, BOX, OM)
    g.set_particles(pos, vel)
    g.pm_deposit()
    first = g.get_mesh(M.MESH_DENSITY_X)
    g.rsd_power_spectrum(2, 0.1)
    g.pm_deposit()
    assert np.array_equal(first, g.get_mesh(M.MESH_DENSITY_X))
    sum_d, _ = g.get_displacements()
    d = g.get_disp().astype(np.float64)
    scale = np.abs(d).max() + 1e-30
    # FP64 sums of np FP32 values in another order
    assert np.abs(sum_d - d.mean(1)).max() < 1e-12 * scale
    sum_v = g.kick(0.3, 0.7, 0.1, 0.2, sum_d)
    v = g.get_particles()[1].astype(np.float64)
    assert np.abs(sum_v - v.mean(1)).max() < 1e-12 * np.abs(v).max()
    g.close()


@pytest.mark.parametrize("n,ns", [(8, 8), (16, 8), (32, 32), (48, 24), (96, 48), (96, 32), (128, 32), (128, 128)])
def test_two_slot_fold_with_constant_growth(n, ns):
    """Both LPT slots by the ln k slices against the per-|n|^2 tables, one slot at a time,
    with a growth that does not depend on k (so the slices are exact): the fold's lanes per
    row from 16 up, m = 1, 2, 3 and 4.  The slices form 1/den with a 1-ulp reciprocal and
    the sums of up to 2 m^3 aliases round in another order: 4e-6 of the field maximum."""
    import ctypes as C

    g = M.MGPU(n, ns, BOX, OM, scale_dependent=1)
    pk = 100.0 / (1.0 + np.arange(M.n2_table_len(n), dtype=np.float64))
    g.ic_displacement_fields(11, pk)
    nk, keep = 50, []

    def kslice(value, den, norm):
        a = [np.full(nk, value), np.zeros(nk), np.full(nk, den), np.zeros(nk)]
        keep.append(a)
        return M.KSlice(-6.0, 0.25, nk, *[x.ctypes.data_as(C.POINTER(C.c_double)) for x in a], norm)

    norm2 = -3.0 / 7.0 / n ** 3
    grow = [(0.8, 0.5), (0.3, 0.2)]
    M.lpt_fields_slices2(g, *[(kslice(2 * a, 2.0, 1.0), kslice(4 * b, 4.0, norm2)) for a, b in grow])
    got = [g.get_lpt(s) for s in (0, 1)]
    ones = np.ones(M.n2_table_len(n))
    for s, (a, b) in enumerate(grow):
        g.lpt_fields(s, a * ones, norm2 * b * ones)
        assert rel_err(got[s], g.get_lpt(s)) < 4e-6
    g.close()


@pytest.mark.parametrize("n", [8, 12, 16, 24, 48, 64, 96, 128])
def test_seed_table_by_chunks(n):
    """The jumped-ahead chunks of the RANLUX stream give the oracle's serial seed table: with
    fixed amplitudes every mode's phase is its column stream's draw, so one wrong seed moves
    a whole column of delta(k).  Sizes with one chunk (8-24), a part-filled last one (48, 96)
    and several waves' worth; FP32 storage of the same FP64 products: 1e-6."""
    pk = 100.0 / (1.0 + np.arange(M.n2_table_len(n), dtype=np.float64))
    for seed in (1, 5001, 2147483647):
        g = M.MGPU(n, n // 2, BOX, OM, scale_dependent=1)
        g.ic_displacement_fields(seed, pk, amplitude_fixed=1)
        want = O.complex_view(O.ic_delta(O.cfg(n, n // 2, BOX, OM), seed, pk, 0, 1, 0), n)
        assert rel_err(g.get_mesh(M.MESH_CDELTA1), want) < 1e-6
        g.close()


@pytest.mark.parametrize("tcols", [8, 16])
@pytest.mark.parametrize("n,ns", [(8, 4), (8, 8), (16, 8), (24, 8), (32, 8), (48, 20), (64, 16), (96, 16), (96, 24),
                                  (96, 48), (128, 128), (192, 64)])
def test_lpt_passes_and_fold(n, ns, tcols):
    """Lattice displacements from the fused spectrum, source and read-out against the oracle:
    fold factors 2, 3 and 4, none (Nmesh = Nsample, or 6), and lattices that do not divide the mesh
    or have no transform of their own (4, 20).  FP32 rounding of 3 log2(n)-stage transforms:
    the bounds of the oracle comparisons of the separate passes, 1e-5 and, through the
    products of the source, 2e-5 of the field maximum."""
    pk = 1000.0 / (1.0 + np.arange(M.n2_table_len(n), dtype=np.float64)) ** 1.5
    pk[0] = 0.0
    print("n, ns, tcols =", n, ns, tcols, flush=True)
    g = M.MGPU(n, ns, BOX, OM)
    g.set_fft_tile(0, tcols)
    g.ic_displacement_fields(4001, pk)
    c = O.cfg(n, ns, BOX, OM)
    za, lp = O.ic_displacements(c, O.ic_delta(c, 4001, pk), 0)
    assert rel_err(g.get_lpt(0), za) < 1e-5
    assert rel_err(g.get_lpt(1), lp) < 2e-5
    g.close()


@pytest.mark.parametrize("ns,n", [(16, 32), (32, 32), (32, 96), (40, 64), (64, 48), (64, 128), (96, 192)])
def test_bins_do_not_depend_on_particle_order(ns, n):
    """delta and the gathered Disp of lattice-ordered particles, of the same ones shuffled and
    of 32 to a point: the deposit's sums are integers, so the density is equal to the bit in
    any order, and within the oracle's FP32 rounding (1e-6 of 1 + delta) of its serial
    deposit.  Lattices with (32, 64, 96) and without (16, 40) blocks of 32 particles."""
    rng = np.random.default_rng(ns)
    pos = lattice_particles(ns, BOX, amp=1.5, seed=3)
    piles = pos.copy()
    piles[:] = np.repeat(pos[:, ::32], 32, axis=1)
    perm = rng.permutation(ns**3)
    c = O.cfg(n, ns, BOX, OM)
    g = M.MGPU(n, ns, BOX, OM)
    print("ns, n =", ns, n, flush=True)
    for p in (pos, piles):
        out = []
        for q in (p, np.ascontiguousarray(p[:, perm])):
            g.set_particles(q)
            g.pm_deposit()
            out.append(g.get_mesh(M.MESH_DENSITY_X))
        np.testing.assert_array_equal(out[0], out[1])
        ref = O.real_view(O.deposit(c, p), n)
        assert (np.abs(out[0] - ref) / np.maximum(1.0, np.abs(1.0 + ref))).max() < 1e-6
    g.set_particles(pos)
    g.get_displacements()
    d = g.get_disp()
    g.set_particles(np.ascontiguousarray(pos[:, perm]))
    g.get_displacements()
    np.testing.assert_array_equal(g.get_disp(), d[:, perm])
    g.close()


@pytest.mark.parametrize("model", ["lcdm", "dgp"])
@pytest.mark.parametrize("n", [192, 384])
def test_tile_widths_and_stores_give_the_same_forces(model, n):
    """8- and 16-column tiles (from 384 on with stores past the caches in the passes of more
    than one mesh) change no column's arithmetic: the force meshes are equal to the bit."""
    pos = lattice_particles(32, BOX, amp=1.5, seed=n)
    kw = dict(model=M.DGP, mg_active=1, include_screening=1, filter=O.FILTER_GAUSSIAN) if model == "dgp" else {}
    mg = M.MG(a=0.7, coupling=0.12, dgp_fac=0.05, rsmooth=2.0, geff=1.0) if model == "dgp" else None
    print("model, n =", model, n, flush=True)
    out = []
    for tcols in (8, 16):
        g = M.MGPU(n, 32, BOX, OM, **kw)
        g.set_fft_tile(0, tcols)
        g.set_particles(pos)
        g.get_displacements(mg=mg)
        out.append([g.get_mesh(m) for m in (M.MESH_FORCE_X, M.MESH_FORCE_Y, M.MESH_FORCE_Z)])
        g.close()
    for a, b in zip(*out):
        assert np.abs(a).max() > 0
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("after", ["deposit", "density", "fifth"])
@pytest.mark.parametrize("model,n", [("fofr", 48), ("dgp", 48), ("dgp", 384)])
def test_autotune_leaves_the_meshes_in_use(model, n, after):
    """The autotuner between the calls of a force computation: the delta(x) of slot 1 and the
    phi(k) of slot 2 stay what they were (up to 256 and beyond the y passes of the force are
    one launch and two), so the displacements are equal to the bit; force meshes, which it
    uses, are refused afterwards."""
    pos = lattice_particles(24, BOX, amp=1.5, seed=n)
    kw = dict(model=M.FOFR if model == "fofr" else M.DGP, mg_active=1, include_screening=1,
              filter=O.FILTER_NONE if model == "fofr" else O.FILTER_GAUSSIAN)
    mg = M.MG(a=0.7, coupling=1 / 3 if model == "fofr" else 0.12, mass2=2e4, phi_crit=3e-8, dgp_fac=0.05, rsmooth=2.0,
              geff=1.0)
    print("model, n, after =", model, n, after, flush=True)
    out = []
    for tune in (False, True):
        g = M.MGPU(n, 24, BOX, OM, **kw)
        g.set_particles(pos)
        for name, call in (("deposit", g.pm_deposit), ("density", g.pm_transform), ("fifth", lambda: g.fifth_force(mg)),
                           ("forces", g.forces)):
            call()
            if tune and name == after:
                g.autotune_fft()
        g.mesh_to_particles()
        out.append(g.get_disp())
    assert np.abs(out[0]).max() > 0
    np.testing.assert_array_equal(out[0], out[1])
    g.autotune_fft()
    with pytest.raises(M.MGPUError, match="no force meshes"):
        g.mesh_to_particles()
    g.close()


@pytest.mark.parametrize("tcols", [8, 16])
@pytest.mark.parametrize("n", [8, 12, 16, 24, 48, 64, 96, 128])
@pytest.mark.parametrize("bins", ["most", "more", "many", "falling"])
def test_pofk_bins_by_table(n, tcols, bins, monkeypatch):
    """The x passes with the bins' table, on both sides of its line (a third of columns times
    points by the edges, one more by the table), far beyond it (16 n + 1) and for bins that
    fall with |n|^2 (last bin below the first).
    Mode counts equal the oracle's formula; the sizes with one transform stage (8, 12, 16)
    have no other barrier between the cleared sums and the first of them added."""
    ns = n // 2
    nbins = {"most": n * tcols // 3, "more": n * tcols // 3 + 1, "many": 16 * n + 1, "falling": n // 2}[bins]
    kmin, kmax = (n / 2.0, 1.0) if bins == "falling" else (0.0, float(n))
    plain = M.make_params

    def with_range(*a):  # the binding itself asks for no last bin below the first
        p = plain(*a)
        p.pofk_kmin, p.pofk_kmax = kmin, kmax
        return p

    monkeypatch.setattr(M, "make_params", with_range)
    pos = lattice_particles(ns, BOX, amp=1.5, seed=n, clustered=ns > 4)
    print("n, tcols, bins =", n, tcols, bins, flush=True)
    mg = dict(a=0.7, coupling=1 / 3, mass2=2e4, phi_crit=3e-8, dgp_fac=0.0, rsmooth=2.0, geff=1.0)
    c = O.cfg(n, ns, BOX, OM)
    dk = O.deposit(c, pos)
    O.fft_r2c_3d(n, dk)
    rp, rk, rn = O.pofk(c, dk, nbins, 0, kmin, kmax, 0)
    ok = (rn > 0) & (rk > 0)
    assert ok.any()
    for mkw in ({}, dict(model=M.FOFR, mg_active=1, include_screening=1)):
        g = M.MGPU(n, ns, BOX, OM, pofk_nbins=nbins, pofk_subtract_shotnoise=0, **mkw)
        g.set_fft_tile(0, tcols)
        g.set_particles(pos)
        g.pm_density(pofk=True)
        for pk, kk, nm in (g.pm_density(pofk=True), g.get_displacements(mg=M.MG(**mg) if mkw else None, pofk=True)[1]):
            assert np.array_equal(nm, rn)
            np.testing.assert_allclose(kk[ok], rk[ok], rtol=1e-12)
            np.testing.assert_allclose(pk[ok], rp[ok], rtol=1e-3)
        g.close()


@pytest.mark.parametrize("n,ns", [(256, 128), (384, 192)])
def test_lpt_passes_against_the_oracle_at_larger_meshes(n, ns):
    """As test_lpt_passes_and_fold, at the 16 and 12 elements per thread of 256 and 384."""
    pk = 1000.0 / (1.0 + np.arange(M.n2_table_len(n), dtype=np.float64)) ** 1.5
    pk[0] = 0.0
    print("n, ns =", n, ns, flush=True)
    g = M.MGPU(n, ns, BOX, OM)
    g.ic_displacement_fields(4001, pk)
    c = O.cfg(n, ns, BOX, OM)
    za, lp = O.ic_displacements(c, O.ic_delta(c, 4001, pk), 0)
    assert rel_err(g.get_lpt(0), za) < 1e-5
    assert rel_err(g.get_lpt(1), lp) < 2e-5
    g.close()


@pytest.mark.parametrize("n,ns,tcols", [(256, 8, 8), (512, 8, 8), (512, 256, 16), (768, 8, 8), (768, 384, 16), (1024, 8, 8),
                                        (1024, 512, 16), (1536, 8, 8), (1536, 512, 8), (2048, 8, 8)])
def test_initial_conditions_of_a_few_modes(n, ns, tcols):
    """Power in |n|^2 <= 3 alone: the displacements have |n_a| <= 1 and, through the products of
    the source, <= 2, so every lattice of 8 points a side holds them exactly.  From the first
    order field's modes (one delta(k) for all three components) the second order follows in
    FP64, with numpy.  Read out of the mesh (ns = 8) or folded; the bounds are those of the
    oracle comparisons, 1e-5 and 2e-5 of the field maximum."""
    pk = np.zeros(M.n2_table_len(n))
    pk[1:4] = 1000.0
    print("n, ns, tcols =", n, ns, tcols, flush=True)
    g = M.MGPU(n, ns, BOX, OM)
    g.set_fft_tile(0, tcols)
    g.ic_displacement_fields(4001, pk)
    step = ns // 8
    first, second = (np.ascontiguousarray(g.get_lpt(s).reshape(3, ns, ns, ns)[:, ::step, ::step, ::step]).astype(np.float64)
                     for s in (0, 1))
    g.close()
    k1 = np.fft.fftfreq(8, 1 / 8.0) * 2 * np.pi / BOX
    k = np.array(np.meshgrid(k1, k1, k1, indexing="ij"))
    k2 = (k * k).sum(0)
    k2[0, 0, 0] = 1.0
    psi = np.fft.fftn(first, axes=(1, 2, 3))
    delta = -1j * (k * psi).sum(0)
    delta[np.round(k2 * (BOX / 2 / np.pi) ** 2) > 3] = 0
    assert np.abs(delta).max() > 0
    real = lambda x: np.fft.ifftn(x).real
    want = np.array([real(1j * k[a] / k2 * delta) for a in range(3)])
    assert rel_err(first, want) < 1e-5
    phi = {(a, b): real(-k[a] * k[b] / k2 * delta) for a in range(3) for b in range(a, 3)}
    source = np.fft.fftn(sum(phi[a, a] * phi[b, b] - phi[a, b] ** 2 for a, b in ((0, 1), (0, 2), (1, 2))))
    want = np.array([real(3.0 / 7.0 * 1j * k[a] / k2 * source) for a in range(3)])
    assert np.abs(want).max() > 0
    assert rel_err(second, want) < 2e-5


def test_seed_table_of_long_chunks():
    """768: chunks of 27 advances (16 up to 512), with fixed amplitudes against the oracle's
    delta(k); see test_seed_table_by_chunks."""
    n = 768
    pk = 100.0 / (1.0 + np.arange(M.n2_table_len(n), dtype=np.float64))
    g = M.MGPU(n, n // 2, BOX, OM, scale_dependent=1)
    g.ic_displacement_fields(5001, pk, amplitude_fixed=1)
    got = g.get_mesh(M.MESH_CDELTA1)
    g.close()
    want = O.complex_view(O.ic_delta(O.cfg(n, n // 2, BOX, OM), 5001, pk, 0, 1, 0), n)
    top = np.abs(want).max()
    assert top > 0 and max(np.abs(got[i] - want[i]).max() for i in range(n)) < 1e-6 * top
