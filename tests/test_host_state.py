"""The host side of libmgpu.so on a stand-in runtime (fake_hip.cpp): which kernels a call
launches, and what a context believes after a launch, a capture or a copy has failed.  Each
case runs in a process of its own, so that the stand-in is there before libmgpu.so.  No GPU."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PRELUDE = """
import ctypes as C, sys
import numpy as np
F = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
sys.path[:0] = sys.argv[2:]
import mgpicola as M

ran = lambda kernel: F.fake_ran(kernel.encode())

def fails(what, call, *args, **kw):
    F.fake_fail(what.encode())
    try:
        call(*args, **kw)
    except M.MGPUError:
        return
    raise AssertionError(what + " did not fail the call")

def context(n=32, ns=16, **kw):
    g = M.MGPU(n, ns, 64.0, 0.3, **kw)
    g.set_particles(np.zeros((3, ns**3), np.float32), np.zeros((3, ns**3), np.float32))
    return g

def forces_at_hand(g):
    for m in (M.MESH_FORCE_X, M.MESH_FORCE_Y, M.MESH_FORCE_Z):
        g.set_mesh(m, np.zeros((g.n,) * 3))
"""


@pytest.fixture(scope="session")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-o", so, os.path.join(HERE, "fake_hip.cpp")], check=True)

    def run(code):
        p = subprocess.run([sys.executable, "-c", PRELUDE + code, so, os.path.join(HERE, "..", "mg-picola-public_amd")],
                           stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
        assert p.returncode == 0, p.stdout

    return run


@pytest.mark.parametrize("call", ["k_gather_tile", "hipStreamEndCapture", "hipGraphInstantiate", "hipGraphLaunch"])
@pytest.mark.parametrize("members", [1, 3])
def test_bins_after_a_step_graph_that_never_ran(fake, call, members):
    """A deposit fails half-way (its counters hold counts), then the graph of the next step,
    which would have cleared them, fails before it runs: the step after that clears them, and
    a gather in between does not take the records that the graph would have sorted."""
    fake(f"""
members, call = {members}, "{call}"
ms = M.MGPU.batch(members, 32, 16, 64.0, 0.3) if members > 1 else [M.MGPU(32, 16, 64.0, 0.3)]
for g in ms:
    g.set_particles(np.zeros((3, 16**3), np.float32), np.zeros((3, 16**3), np.float32))
    g.kick(0.1, 1.0, 0.0, 0.0, g.get_displacements()[0])
a = (0.1, 1.0, 0.0, 0.0, 0.1, 0.0, 0.0)
step = lambda: M.MGPU.batch_step(ms, *a, graph=True) if members > 1 else ms[0].step(*a, graph=True)
F.fake_reset()
step()
assert ran("k_dep_bin") == 1 and ran("k_zero_u32") == 0
fails("k_dep_bin", ms[-1].pm_deposit)
F.fake_reset()
fails(call, step)
assert ran("k_dep_bin") == 0
forces_at_hand(ms[0])
ms[0].mesh_to_particles()
assert ran("k_gather_tile") == 0 and ran("k_gather") == 1
F.fake_reset()
step()
assert ran("k_dep_bin") == 1 and ran("k_zero_u32") == 1
""")


@pytest.mark.parametrize("kernel", ["k_dep_bin", "k_scan_one", "k_dep_scatter", "k_dep_tiles"])
def test_no_gather_by_the_records_of_a_failed_deposit(fake, kernel):
    """A context's first deposit fails before its records and bin offsets are written: the
    gather takes the particles one by one and not by what the memory holds."""
    fake(f"""
g = context()
fails("{kernel}", g.pm_deposit)
forces_at_hand(g)
F.fake_reset()
g.mesh_to_particles()
assert ran("k_gather_tile") == 0 and ran("k_gather") == 1
""")


@pytest.mark.parametrize("kernel", ["k_seed_table", "k_ic_delta", "k_lpt_x", "k_lpt_source"])
@pytest.mark.parametrize("sd", [0, 1])
def test_initial_conditions_that_fail_wait_for_their_uploads(fake, kernel, sd):
    """No copy from the call's own states or the caller's table is in flight on return."""
    fake(f"""
pk = np.ones(M.n2_table_len(32))
g = M.MGPU(32, 16, 64.0, 0.3, scale_dependent={sd})
fails("{kernel}", g.ic_displacement_fields, 1, pk)
assert F.fake_pending() == 0
g.ic_displacement_fields(1, pk)
assert F.fake_pending() == 0 and ran("k_seed_table") >= 1
if not {sd}:
    ms = M.MGPU.batch(2, 32, 16, 64.0, 0.3)
    fails("{kernel}", M.MGPU.batch_ic, ms, [1, 2], pk)
    assert F.fake_pending() == 0
""")


@pytest.mark.parametrize("n,tcols,nbins", [(1024, 16, 512), (1024, 16, 1876), (1024, 16, 3800), (1024, 8, 12000), (2048, 8, 3500),
                                           (128, 16, 18000), (64, 8, 19800)])
def test_pofk_stays_in_the_x_pass(fake, n, tcols, nbins):
    """Every number of bins whose sums fit the LDS beside the tile of columns is binned by the x
    pass, alone and in the fused step of every model (unscreened LCDM's takes 8 columns)."""
    fake(f"""
n, tcols, nbins = {n}, {tcols}, {nbins}
mg = M.MG(a=0.7, coupling=0.3, mass2=2e4, phi_crit=3e-8, dgp_fac=0.05, rsmooth=2.0, geff=1.0)
plain = M.make_params
def falling(*a):  # the last bin below the first, which the binding itself does not ask for
    p = plain(*a)
    p.pofk_kmin, p.pofk_kmax = float(n), 1.0
    return p
for kw, params in ((dict(), plain), (dict(model=M.FOFR, mg_active=1, include_screening=1), plain), (dict(), falling)):
    M.make_params = params
    g = context(n, 16, pofk_nbins=nbins, **kw)
    assert (g.p.pofk_kmax < g.p.pofk_kmin) == (params is falling)
    g.set_fft_tile(0, tcols)
    m = mg if kw.get("mg_active") else None
    g.pm_density(pofk=True)
    assert ran("k_pofk") >= 1
    for call in (lambda: g.pm_density(pofk=True), lambda: g.get_displacements(mg=m, pofk=True)):
        F.fake_reset()
        call()
        assert ran("k_pofk") == 0, (kw, nbins)
    assert ran("k_col_fused") == (2 if m else 1)
    g.close()
""")


def test_pofk_of_more_bins_than_the_x_pass_holds(fake):
    """Beyond that, and without the table (more than 32767 bins), by a pass of its own."""
    fake("""
for n, nbins in ((1024, 13000), (32, 33000)):
    g = context(n, 16, pofk_nbins=nbins)
    g.pm_density(pofk=True)
    for call in (lambda: g.pm_density(pofk=True), lambda: g.get_displacements(pofk=True)):
        F.fake_reset()
        call()
        assert ran("k_pofk") >= 1 and ran("k_col_pofk") + ran("k_col_fused") == 0
    g.close()
""")


@pytest.mark.parametrize("nbins", [16, 500, 5000])
def test_pofk_comes_back_without_a_copy(fake, nbins):
    """The bin sums of P(k) and of the multipoles are stored to the host by a kernel, which
    adds the x pass's sets first: no copy that grows with the sets."""
    fake(f"""
g = context(64, 32, pofk_nbins={nbins})
for call in (lambda: g.pm_density(pofk=True), lambda: g.pm_density(pofk=True), lambda: g.get_displacements(pofk=True),
             g.power_spectrum, lambda: g.rsd_power_spectrum(2, 0.1)):
    F.fake_reset()
    call()
    assert F.fake_to_host() == 0 and ran("k_bins_to_host") == 1
""")
