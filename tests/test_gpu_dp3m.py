"""Dipolar P3M on the device against the dipolar oracle (oracle/dp3m.py,
pinned in test_oracle_dp3m.py against the reference's 1000-dipole fixture
and energy derivatives), and against that fixture itself.

Tolerances: k-space forces, torques rel-rms <= 1e-10 and energy <= 1e-10
relative (FP64 on both sides, same CA weights); real-space pair terms
<= 1e-12; the fixture at the reference test's vector errors (2e-3) and
energy error (1e-3).
"""
import os

import numpy as np
import pytest

from tests import p3m_systems as S

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def _system(n, L, seed, zero_frac=0.1):
    rng = np.random.default_rng(seed)
    pos = rng.uniform(0., L, (n, 3))
    dip = rng.normal(size=(n, 3))
    dip[rng.random(n) < zero_frac] = 0.
    pos[:3, 0] += L       # outside the box (folded by the solver)
    return pos, dip


# (8, 7): the per-bucket LDS tile (11 points per edge) wraps around the mesh;
# (10, 5) and (12, 3): meshes that the buckets of 8 cells do not divide;
# (80, 3): above 64 the transforms run one pass per axis (no plane kernel)
@pytest.mark.parametrize("M,cao,epsilon", [(16, 3, 0.), (24, 5, 0.), (32, 7, 2.), (20, 4, 0.),
                                           (8, 7, 0.), (10, 5, 0.), (12, 3, 2.), (80, 3, 0.)])
def test_kspace_matches_oracle(M, cao, epsilon):
    from espresso_amd.magnetostatics import DipolarP3M
    from oracle import dp3m as D
    L = 10.
    pos, dip = _system(600, L, 10 + cao)
    alpha, r_cut = 0.9, 3.2
    dp = DipolarP3M(prefactor=1.3, accuracy=1e-4, mesh=M, cao=cao, alpha=alpha, r_cut=r_cut,
                    epsilon=epsilon, tune=False)
    dp.activate(pos, dip, box_l=L)
    f, t = np.zeros((600, 3)), np.zeros((600, 3))
    dp.add_long_range_forces(pos, dip, f, t)
    e = dp.long_range_energy(pos, dip)
    ora = D.OracleDP3M(L, M, cao, alpha, r_cut, 1.3, epsilon=epsilon)
    fr, tr, er = ora.solve(pos - L * np.floor(pos / L), dip)
    ef, et = S.rel_rms(f, fr), S.rel_rms(t, tr)
    print(f"M {M} cao {cao} eps {epsilon}: forces {ef:.2e} torques {et:.2e} "
          f"energy {e:.10f} vs {er:.10f}")
    assert ef <= 1e-10 and et <= 1e-10
    assert abs(e - er) <= 1e-10 * abs(er)


def test_kspace_clustered_and_partial_outputs():
    """Most dipoles in one corner (a few buckets holding far more particles
    than a block has threads), a spread across the periodic boundary, and
    torque-only / force-only calls equal to the combined call."""
    from espresso_amd.magnetostatics import DipolarP3M
    from oracle import dp3m as D
    L, M, cao, n = 12., 24, 5, 2500
    rng = np.random.default_rng(31)
    pos = np.concatenate([rng.uniform(-1., 1.5, (2000, 3)), rng.uniform(0., L, (n - 2000, 3))])
    dip = rng.normal(size=(n, 3))
    dp = DipolarP3M(prefactor=0.7, accuracy=1e-4, mesh=M, cao=cao, alpha=0.8, r_cut=3.,
                    tune=False)
    dp.activate(pos, dip, box_l=L)
    f, t = np.zeros((n, 3)), np.zeros((n, 3))
    dp.add_long_range_forces(pos, dip, f, t)
    ora = D.OracleDP3M(L, M, cao, 0.8, 3., 0.7)
    fr, tr, _ = ora.solve(pos - L * np.floor(pos / L), dip)
    assert S.rel_rms(f, fr) <= 1e-10 and S.rel_rms(t, tr) <= 1e-10
    t_only, f_only = np.zeros((n, 3)), np.zeros((n, 3))
    dp.add_long_range_forces(pos, dip, None, t_only)
    dp.add_long_range_forces(pos, dip, f_only, None)
    assert S.rel_rms(t_only, t) <= 1e-13 and S.rel_rms(f_only, f) <= 1e-13


@pytest.mark.parametrize("subdiv", [0, 1, 2])
def test_short_range_cell_lists_match_oracle(subdiv):
    """Every number of cells per cutoff in a box wide enough for all of them
    (the column search) against the oracle's all-pairs sum."""
    from espresso_amd.magnetostatics import DipolarP3M
    from oracle import dp3m as D
    L = 20.
    pos, dip = _system(3000, L, 8)
    dp = DipolarP3M(prefactor=1.3, accuracy=1e-4, mesh=16, cao=4, alpha=0.9, r_cut=3.5,
                    tune=False)
    dp.activate(pos, dip, box_l=L)
    dp.set_short_range_subdivision(subdiv)
    f, t = np.zeros((3000, 3)), np.zeros((3000, 3))
    e = dp.add_short_range_forces(pos, dip, f, t, energy=True)
    fr, tr, er = D.pair_terms(pos - L * np.floor(pos / L), dip, L, 1.3, 0.9, 3.5, 1e-4)
    assert S.rel_rms(f, fr) <= 1e-12 and S.rel_rms(t, tr) <= 1e-12
    assert abs(e - er) <= 1e-12 * abs(er)
    with pytest.raises(ValueError, match="subdivision must be 0, 1 or 2"):
        dp.set_short_range_subdivision(3)


def test_particle_count_beyond_int32_rejected():
    """The device sort indexes particles with 32-bit integers: a count of
    2^31 is rejected before any array is read."""
    import ctypes as C
    import torch
    from espresso_amd import _lib
    from espresso_amd.magnetostatics import DipolarP3M
    pos, dip = _system(50, 10., 3)
    dp = DipolarP3M(prefactor=1., accuracy=1e-4, mesh=8, cao=3, alpha=0.9, r_cut=3.,
                    tune=False)
    dp.activate(pos, dip, box_l=10.)
    t = torch.zeros((4, 3), dtype=torch.float64, device="cuda")
    e = C.c_double(0.)
    L = _lib.load()
    for fn in (L.p3m_dipolar_solve, L.p3m_dipolar_short_range):
        rc = fn(dp._ctx, 2 ** 31, t.data_ptr(), t.data_ptr(), None, None,
                _lib.P3M_ENERGY | _lib.P3M_DEVICE_POINTERS, C.byref(e))
        with pytest.raises(ValueError, match="2\\^31"):
            _lib.raise_for(rc, dipolar=dp._ctx)


@pytest.mark.parametrize("box", [5.6, 5.4])
def test_narrow_boxes_match_oracle(box):
    """Boxes of 2.5 to 3 cutoffs go by columns with two cells per cutoff and by
    all pairs with one, narrower ones by all pairs."""
    from espresso_amd.magnetostatics import DipolarP3M
    from oracle import dp3m as D
    n, r_cut = 700, 2.2
    pos, dip = _system(n, box, 15)
    fr, tr, er = D.pair_terms(pos - box * np.floor(pos / box), dip, box, 1.3, 0.9, r_cut, 1e-4)
    dp = DipolarP3M(prefactor=1.3, accuracy=1e-4, mesh=16, cao=4, alpha=0.9, r_cut=r_cut,
                    tune=False)
    dp.activate(pos, dip, box_l=box)
    for subdiv in (0, 1, 2):
        dp.set_short_range_subdivision(subdiv)
        f, t = np.zeros((n, 3)), np.zeros((n, 3))
        e = dp.add_short_range_forces(pos, dip, f, t, energy=True)
        assert S.rel_rms(f, fr) <= 1e-12 and S.rel_rms(t, tr) <= 1e-12
        assert abs(e - er) <= 1e-12 * abs(er)


# r_cut 3.5: columns with z bins of r_cut/2 (16 dipoles per r_cut^3 on average);
# r_cut 6.5: three columns along x and y, z bins of r_cut/4
@pytest.mark.parametrize("subdiv,r_cut", [(1, 3.5), (2, 3.5), (1, 6.5)])
def test_short_range_dense_cluster_matches_oracle(subdiv, r_cut):
    """400 dipoles packed into one place among 3000 sparse ones: several full
    home groups in one z bin, and lists that fill and drain many times."""
    from espresso_amd.magnetostatics import DipolarP3M
    from oracle import dp3m as D
    L = 20.
    pos, dip = _system(3000, L, 12)
    rng = np.random.default_rng(13)
    pos = np.concatenate([pos, 7.3 + rng.uniform(0., 1., (400, 3))])
    dip = np.concatenate([dip, rng.normal(size=(400, 3))])
    n = len(pos)
    dp = DipolarP3M(prefactor=1.1, accuracy=1e-4, mesh=16, cao=4, alpha=0.9, r_cut=r_cut,
                    tune=False)
    dp.activate(pos, dip, box_l=L)
    dp.set_short_range_subdivision(subdiv)
    f, t = np.zeros((n, 3)), np.zeros((n, 3))
    e = dp.add_short_range_forces(pos, dip, f, t, energy=True)
    fr, tr, er = D.pair_terms(pos - L * np.floor(pos / L), dip, L, 1.1, 0.9, r_cut, 1e-4)
    assert S.rel_rms(f, fr) <= 1e-12 and S.rel_rms(t, tr) <= 1e-12
    assert abs(e - er) <= 1e-12 * abs(er)


@pytest.mark.parametrize("mesh,cao,n", [
    (2, 1, 3), (8, 7, 40), (14, 6, 900),  # tiles that wrap around the mesh
    (24, 5, 1), (24, 5, 6000),            # buckets of 8 and of 3 cells
    (50, 6, 6000),                        # buckets that do not divide the mesh
    (96, 3, 500), (98, 3, 500),           # last mesh transformed by planes, first by lines
])
def test_kspace_transform_and_bucket_edges_match_oracle(mesh, cao, n):
    """Half-spectrum transforms and particle buckets at the edges of their
    rules; forces and torques, then each alone, and the energy.  Tolerance of
    the k-space tests (FP64 rounding of the FFTs and sums)."""
    from espresso_amd.magnetostatics import DipolarP3M
    from oracle import dp3m as D
    L = 10.
    pos, dip = _system(n, L, n + mesh)
    dp = DipolarP3M(prefactor=1.3, accuracy=1e-4, mesh=mesh, cao=cao, alpha=0.6, r_cut=3.,
                    tune=False)
    dp.activate(pos, dip, box_l=L)
    f, t, f1, t1 = (np.zeros((n, 3)) for _ in range(4))
    dp.add_long_range_forces(pos, dip, f, t)
    e = dp.long_range_energy(pos, dip)
    dp.add_long_range_forces(pos, dip, None, t1)
    dp.add_long_range_forces(pos, dip, f1, None)
    fr, tr, er = D.OracleDP3M(L, mesh, cao, 0.6, 3., 1.3).solve(pos - L * np.floor(pos / L), dip)
    for got, ref in ((f, fr), (t, tr), (f1, fr), (t1, tr)):
        scale = max(np.sqrt(np.mean(ref ** 2)), 1e-6)
        assert np.sqrt(np.mean((got - ref) ** 2)) <= 1e-10 * scale
    assert abs(e - er) <= 1e-10 * max(abs(er), 1e-6)


@pytest.mark.parametrize("accuracy", [1e-4, 1e-7])
@pytest.mark.parametrize("L,r_cut,n,spread", [
    (9., 2.2, 1, 1.),            # no pair at all
    (9., 2.2, 2, 0.1),
    (9., 2.2, 700, 0.25),        # crowded columns: full groups of 64 and a remainder
    (5.8, 2.2, 64 * 14 + 1, 1.), # five columns of r_cut/2 along x and y
    (130., 2., 4000, 0.05),      # 65 columns along x, one block per group
])
def test_dipolar_column_pairs_match_oracle(L, r_cut, n, spread, accuracy):
    """Forces, torques and energy of the column kernel at the edges of its
    home groups, reaches and block shares, some dipoles zero; then torques and
    forces alone.  Tolerance as in the other real-space tests: FP64 sums of
    the same terms."""
    import torch
    from espresso_amd.magnetostatics import DipolarP3M
    from oracle import dp3m as D
    rng = np.random.default_rng(n)
    pos = (rng.uniform(-0.5, 0.5, (n, 3)) * spread * L) % L
    dip = rng.normal(size=(n, 3)) * (np.arange(n) % 7 != 3)[:, None]
    dp = DipolarP3M(prefactor=1.3, accuracy=accuracy, mesh=16, cao=4, alpha=1.1, r_cut=r_cut,
                    tune=False)
    dp.activate(pos, dip, box_l=L)
    tp, td = torch.tensor(pos, device="cuda"), torch.tensor(dip, device="cuda")
    tf, tt, f1, t1 = (torch.zeros_like(tp) for _ in range(4))
    e = dp.add_short_range_forces(tp, td, tf, tt, energy=True)
    dp.add_short_range_forces(tp, td, None, t1)
    dp.add_short_range_forces(tp, td, f1, None)
    fr, tr, er = D.pair_terms(pos, dip, L, 1.3, 1.1, r_cut, accuracy)
    for got, ref in ((tf, fr), (tt, tr), (f1, fr), (t1, tr)):
        scale = max(np.sqrt(np.mean(ref ** 2)), 1e-300)
        assert np.sqrt(np.mean((got.cpu().numpy() - ref) ** 2)) <= 1e-12 * scale
    assert abs(e - er) <= 1e-12 * abs(er)


@pytest.mark.parametrize("accuracy", [1e-4, 1e-7])
def test_short_range_matches_oracle(accuracy):
    """A&S erfc for accuracy > 5e-6, libm erfc below (dp3m.hpp:176-178)."""
    import torch
    from espresso_amd.magnetostatics import DipolarP3M
    from oracle import dp3m as D
    L = 9.
    pos, dip = _system(700, L, 5)
    dp = DipolarP3M(prefactor=1.3, accuracy=accuracy, mesh=16, cao=4, alpha=1.1, r_cut=3.5,
                    tune=False)
    dp.activate(pos, dip, box_l=L)
    f, t = np.zeros((700, 3)), np.zeros((700, 3))
    e = dp.add_short_range_forces(pos, dip, f, t, energy=True)
    fr, tr, er = D.pair_terms(pos - L * np.floor(pos / L), dip, L, 1.3, 1.1, 3.5, accuracy)
    assert S.rel_rms(f, fr) <= 1e-12 and S.rel_rms(t, tr) <= 1e-12
    assert abs(e - er) <= 1e-12 * abs(er)
    # device tensors, asynchronous
    tp, td = torch.tensor(pos, device="cuda"), torch.tensor(dip, device="cuda")
    tf, tt = torch.zeros_like(tp), torch.zeros_like(tp)
    dp.add_short_range_forces(tp, td, tf, tt, sync=False)
    dp.add_long_range_forces(tp, td, tf, tt, sync=False)
    dp.synchronize()
    f2, t2 = np.zeros((700, 3)), np.zeros((700, 3))
    dp.add_long_range_forces(pos, dip, f2, t2)
    assert S.rel_rms(tf.cpu().numpy(), f + f2) <= 1e-12
    assert S.rel_rms(tt.cpu().numpy(), t + t2) <= 1e-12


def test_reference_fixture_total():
    """The reference's dipolar P3M test (dipolar_mdlc_p3m_scafacos_p2nfft.py:
    115-153): 1000 dipoles, DipolarP3M(mesh=32, accuracy=1e-6, metallic),
    tuned here; total forces, torques and energy against the expected data
    at vector errors 2e-3 and energy 1e-3."""
    from espresso_amd.magnetostatics import DipolarP3M
    d = np.load(os.path.join(GOLDEN, "p3m_magnetostatics.npz"))
    L = float(d["box_l"])
    pos, dip = d["pos"], d["dip"]
    pref = 1.1
    dp = DipolarP3M(prefactor=pref, mesh=32, accuracy=1e-6, epsilon="metallic", verbose=False)
    dp.activate(pos, dip, box_l=L)
    prm = dp.get_params()
    f, t = np.zeros((1000, 3)), np.zeros((1000, 3))
    dp.add_long_range_forces(pos, dip, f, t)
    e = dp.long_range_energy(pos, dip)
    e += dp.add_short_range_forces(pos, dip, f, t, energy=True)

    def verr(a, b):
        return np.sum(np.linalg.norm(a - b, axis=1)) / np.sqrt(a.shape[0])
    ef, et = verr(f, d["force"] * pref), verr(t, d["torque"] * pref)
    ee = e - float(d["energy"]) * pref
    print(f"tuned mesh {prm['mesh'][0]} cao {prm['cao']} r_cut {prm['r_cut']:.3f} "
          f"alpha {prm['alpha']:.4f}: force {ef:.2e} torque {et:.2e} energy {ee:.2e}")
    assert ef <= 2e-3 and et <= 2e-3 and abs(ee) <= 1e-3
