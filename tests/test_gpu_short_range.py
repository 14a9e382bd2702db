"""Device real-space pair forces (cell lists) against the FP64 oracle's
brute-force pair loop (oracle.real_space: all pairs, minimum image, the
reference's pair_force/pair_energy with the A&S erfc, p3m.hpp:146-180).

Forces rel-rms <= 1e-12, energy and virial <= 1e-12 relative: both sides
evaluate the same FP64 pair terms and differ only in summation order.  The
cases cover the column search, the all-pairs path of narrow boxes and where
the cells per cutoff draw the line between them, non-cubic boxes, uncharged
particles and positions outside the box; the cell search of ELC images is
covered with ELC.
The total device force (k-space + short range) is checked against exact
Ewald on the C3 fixture subset.
"""
import os

import numpy as np
import pytest

from tests import p3m_systems as S

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def _actor(box, r_cut, alpha, prefactor=1.3, mesh=16, cao=5):
    from espresso_amd.electrostatics import P3M
    p3m = P3M(prefactor=prefactor, accuracy=1e-3, mesh=mesh, cao=cao, r_cut=r_cut,
              alpha=alpha, tune=False)
    pos = np.random.default_rng(0).uniform(0., 1., (20, 3)) * np.asarray(box)
    p3m.activate(pos, np.where(np.arange(20) % 2 == 0, 1., -1.), box_l=list(box))
    return p3m


def _system(n, box, seed, zero_frac=0.1):
    rng = np.random.default_rng(seed)
    pos = rng.uniform(0., 1., (n, 3)) * np.asarray(box)
    q = np.where(np.arange(n) % 2 == 0, 1., -1.) * rng.uniform(0.5, 1.5, n)
    q[rng.random(n) < zero_frac] = 0.
    # a few positions outside the primary box (folded by the solver)
    pos[:5, 0] -= box[0] * 1.3
    pos[5:10, 1] += box[1] * 2.2
    return pos, q


@pytest.mark.parametrize("box,r_cut,subdiv,cells", [
    ((12., 12., 12.), 2.0, 2, (12, 12, 12)),
    ((12., 12., 12.), 2.0, 1, (6, 6, 6)),
    ((10., 12., 14.), 2.4, 0, (8, 10, 11)),
    ((4.5, 4.5, 4.5), 2.0, 0, (1, 1, 1)),       # narrower than 3 cells: all pairs
    ((7.0, 4.6, 9.0), 2.2, 0, (1, 1, 1)),       # one narrow dimension: all pairs
])
def test_short_range_matches_oracle(box, r_cut, subdiv, cells):
    import torch
    from oracle import oracle as O
    n = 3000 if box[0] > 5 else 300
    pos, q = _system(n, box, 11)
    alpha = 1.1
    p3m = _actor(box, r_cut, alpha)
    p3m.set_short_range_subdivision(subdiv)
    tp = torch.tensor(pos, device="cuda")
    tq = torch.tensor(q, device="cuda")
    f0 = np.random.default_rng(5).normal(size=(n, 3))
    tf = torch.tensor(f0, device="cuda")
    e, vir = p3m.add_short_range_forces(tp, tq, tf, energy=True, pressure=True)
    assert tuple(p3m.short_range_cells()) == cells
    e_ref, f_ref, v_ref = O.real_space(pos, q, box, 1.3, alpha, r_cut, virial=True)
    f = tf.cpu().numpy() - f0
    assert S.rel_rms(f, f_ref) <= 1e-12
    assert abs(e - e_ref) <= 1e-12 * abs(e_ref)
    assert np.max(np.abs(vir - v_ref)) <= 1e-12 * np.max(np.abs(v_ref))
    # forces only, asynchronous enqueue on device tensors
    tf2 = torch.zeros_like(tp)
    p3m.add_short_range_forces(tp, tq, tf2, sync=False)
    p3m.synchronize()
    assert S.rel_rms(tf2.cpu().numpy(), f_ref) <= 1e-12


@pytest.mark.parametrize("box,cells", [
    ((5.6, 5.7, 5.8), (5, 5, 5)),    # 2.5 to 3 cutoffs along every axis
    ((9., 5.6, 12.), (8, 5, 10)),    # along one
    ((5.4, 9., 9.), None),           # too narrow for either
])
def test_cells_per_cutoff_decide_when_all_pairs_are_taken(box, cells):
    """A box of 2.5 to 3 cutoffs is searched by columns with two cells per
    cutoff and takes all pairs with one; the same sums either way, at any
    density (500 charges, and 5000: more than 128 per cubed cutoff in the
    smallest box)."""
    import torch
    from oracle import oracle as O
    r_cut = 2.2
    p3m = _actor(box, r_cut, 1.1)
    for n in (500, 5000):
        pos, q = _system(n, box, n)
        e_ref, f_ref = O.real_space(pos, q, box, 1.3, 1.1, r_cut)
        for subdiv in (0, 1, 2):
            p3m.set_short_range_subdivision(subdiv)
            tf = torch.zeros((n, 3), dtype=torch.float64, device="cuda")
            e = p3m.add_short_range_forces(torch.tensor(pos, device="cuda"),
                                           torch.tensor(q, device="cuda"), tf, energy=True)
            pairs = subdiv == 1 or cells is None
            assert tuple(p3m.short_range_cells()) == ((1, 1, 1) if pairs else cells)
            assert S.rel_rms(tf.cpu().numpy(), f_ref) <= 1e-12
            assert abs(e - e_ref) <= 1e-12 * abs(e_ref)


def test_cells_per_cutoff_do_not_depend_on_the_density():
    """Cells of r_cut/2 by default, from sparse to 128 charges per r_cut^3 and
    more."""
    import torch
    p3m = _actor((9., 9., 9.), 2.2, 1.1)
    for n in (300, 8700, 9000):
        pos, q = _system(n, (9., 9., 9.), n)
        f = torch.zeros((n, 3), dtype=torch.float64, device="cuda")
        p3m.add_short_range_forces(torch.tensor(pos, device="cuda"),
                                   torch.tensor(q, device="cuda"), f)
        assert tuple(p3m.short_range_cells()) == (8, 8, 8)


def test_short_range_host_arrays_and_errors():
    from oracle import oracle as O
    box = (9., 9., 9.)
    pos, q = _system(800, box, 21)
    p3m = _actor(box, 3.0, 0.9)
    f = np.ones((800, 3))
    e = p3m.add_short_range_forces(pos, q, f, energy=True)
    e_ref, f_ref = O.real_space(pos, q, box, 1.3, 0.9, 3.0)
    assert S.rel_rms(f - 1., f_ref) <= 1e-12
    assert abs(e - e_ref) <= 1e-12 * abs(e_ref)
    with pytest.raises(ValueError, match="sync=False needs device"):
        p3m.add_short_range_forces(pos, q, f, sync=False)
    with pytest.raises(ValueError, match="subdivision"):
        p3m.set_short_range_subdivision(3)
    wide = _actor((5., 5., 5.), 2.6, 1.0)
    with pytest.raises(ValueError, match="half the box"):
        wide.add_short_range_forces(pos, q, f)


def test_c3_total_device_force_against_ewald():
    """k-space + short range, both on the device, for the whole 250k system;
    rms error on the exact-Ewald fixture subset within 1.5x the target."""
    import torch
    from espresso_amd.electrostatics import P3M
    from oracle import oracle as O
    pos, q, box = S.config_c3()
    L = box[0]
    fx = np.load(os.path.join(GOLDEN, "ewald_c3_subset.npz"))
    acc = 1e-4
    t = O.tune_r_cut(1.0, [64] * 3, 5, len(q), float(np.sum(q * q)), acc, [L] * 3)
    r_cut, alpha = t[0] * L, t[1] / L
    p3m = P3M(prefactor=1.0, accuracy=acc, mesh=64, cao=5, r_cut=r_cut, alpha=alpha,
              tune=False)
    p3m.activate(pos[:1000], np.where(np.arange(1000) % 2 == 0, 1., -1.), box_l=[L] * 3)
    tp = torch.tensor(pos, device="cuda")
    tq = torch.tensor(q, device="cuda")
    f = torch.zeros_like(tp)
    p3m.add_long_range_forces(tp, tq, f)
    p3m.add_short_range_forces(tp, tq, f)
    d = f.cpu().numpy()[fx["idx"]] - fx["force"]
    err = float(np.sqrt(np.mean(np.sum(d * d, axis=1))))
    print(f"C3 mesh 64 cao 5: device total-force rms error {err:.3e} (estimate {t[2]:.3e})")
    assert err <= 1.5 * acc


def test_tuning_with_device_real_space():
    """Timed tuning that charges each trial (r_cut, alpha) with the device
    pair loop: the tuned parameters meet the accuracy target, and the total
    device force on the C3 system meets it against exact Ewald."""
    import torch
    from espresso_amd.electrostatics import P3M
    pos, q, box = S.config_c3()
    L = box[0]
    fx = np.load(os.path.join(GOLDEN, "ewald_c3_subset.npz"))
    acc = 1e-4
    tuned = {}
    for mode in ("model", "device"):
        p3m = P3M(prefactor=1.0, accuracy=acc, timings=3, verbose=False)
        p3m.set_tuning_real_space(mode)
        tp = torch.tensor(pos, device="cuda")
        tq = torch.tensor(q, device="cuda")
        p3m.activate(tp, tq, box_l=[L] * 3)
        prm = p3m.get_params()
        tuned[mode] = prm
        f = torch.zeros_like(tp)
        p3m.add_long_range_forces(tp, tq, f)
        p3m.add_short_range_forces(tp, tq, f)
        d = f.cpu().numpy()[fx["idx"]] - fx["force"]
        err = float(np.sqrt(np.mean(np.sum(d * d, axis=1))))
        print(f"tuning real space {mode}: mesh {prm['mesh']} cao {prm['cao']} "
              f"r_cut {prm['r_cut']:.3f} alpha {prm['alpha']:.4f}; rms error {err:.3e}")
        assert err <= 1.5 * acc
    with pytest.raises(ValueError, match="tuning real space"):
        P3M(prefactor=1.0, accuracy=acc).set_tuning_real_space("host")


@pytest.mark.parametrize("box,r_cut,n,spread", [
    ((9., 9., 9.), 2.2, 1, 1.),          # no pair at all
    ((9., 9., 9.), 2.2, 2, 0.1),
    ((9., 9., 9.), 2.2, 700, 0.25),      # crowded columns: full groups of 64 and a remainder
    ((9., 9., 9.), 2.2, 2000, 1.),
    ((5.6, 9., 9.), 2.2, 900, 1.),       # five columns of r_cut/2 along x, three wider axes
    ((5.6, 5.7, 5.8), 2.2, 900, 1.),     # the same along x and y; z runs longer than the box
    ((30., 8., 7.), 2.2, 64 * 20 + 1, 1.),
    ((140., 140., 8.), 2.0, 4000, 1.),   # 64 x 64 columns: one block per group
    ((140., 140., 8.), 2.0, 4000, 0.05),
])
def test_column_pairs_match_oracle(box, r_cut, n, spread):
    """Pair forces, energy and virial of the column kernel at the edges of
    its home groups (1 to 64 particles of a column), reaches and block
    shares; `spread` packs the particles into a part of the box across the
    periodic corner.  Tolerance as above: FP64 sums of the same terms."""
    import torch
    from oracle import oracle as O
    rng = np.random.default_rng(n)
    b = np.asarray(box)
    pos = (rng.uniform(-0.5, 0.5, (n, 3)) * spread * b) % b
    q = np.where(np.arange(n) % 2 == 0, 1., -1.) * rng.uniform(0.5, 1.5, n)
    p3m = _actor(box, r_cut, 1.1)
    tp, tq = torch.tensor(pos, device="cuda"), torch.tensor(q, device="cuda")
    tf = torch.zeros_like(tp)
    e, vir = p3m.add_short_range_forces(tp, tq, tf, energy=True, pressure=True)
    e_ref, f_ref, v_ref = O.real_space(pos, q, box, 1.3, 1.1, r_cut, virial=True)
    scale = max(np.sqrt(np.mean(f_ref ** 2)), 1e-300)
    for _ in range(2):  # with energy, then forces alone
        assert np.sqrt(np.mean((tf.cpu().numpy() - f_ref) ** 2)) <= 1e-12 * scale
        tf.zero_()
        p3m.add_short_range_forces(tp, tq, tf)
    assert abs(e - e_ref) <= 1e-12 * np.sum(np.abs(e_ref))
    assert np.max(np.abs(vir - v_ref)) <= 1e-12 * max(np.max(np.abs(v_ref)), 1e-300)
