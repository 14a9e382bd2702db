"""Stage times of synchronous solves (device wall-clock stamps), and the order
of a solve after the stream that made its arrays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mesh,flags", [(16, "force"), (32, "force"), (32, "energy"),
                                        (104, "both")])
def test_stage_times_add_up(mesh, flags):
    import torch
    from espresso_amd.electrostatics import P3M
    n, L = 3000, 12.
    rng = np.random.default_rng(mesh)
    pos = torch.tensor(rng.uniform(0., L, (n, 3)), device="cuda")
    q = torch.tensor(np.where(np.arange(n) % 2 == 0, 1., -1.), device="cuda")
    p = P3M(prefactor=1., accuracy=1e-3, mesh=mesh, cao=5, r_cut=3., alpha=0.9, tune=False)
    p.activate(pos, q, box_l=[L] * 3)
    f = torch.zeros_like(pos)
    if flags == "energy":
        p.long_range_energy(pos, q)
    else:
        p.solve(pos, q, f, energy=flags == "both")
    t = p.last_timings()
    stages = [t[k] for k in ("bin", "spread", "fft_fwd", "convolve", "fft_bwd", "gather")]
    assert all(s >= 0. for s in stages) and 0. < t["total"] < 100.
    assert abs(sum(stages) - t["total"]) <= 1e-5 + 1e-5 * t["total"]  # float32 sums
    ran = stages if flags != "energy" else stages[:4]
    assert all(s > 0. for s in ran)


def test_solve_waits_for_the_producing_stream():
    """Positions written by a long queue of work on a side stream of torch are
    complete before the solve reads them."""
    import torch
    from espresso_amd.electrostatics import P3M
    n, L = 2000, 10.
    rng = np.random.default_rng(3)
    pos = torch.tensor(rng.uniform(0., L, (n, 3)), device="cuda")
    q = torch.tensor(np.where(np.arange(n) % 2 == 0, 1., -1.), device="cuda")
    p = P3M(prefactor=1., accuracy=1e-3, mesh=16, cao=5, r_cut=3., alpha=0.9, tune=False)
    p.activate(pos, q, box_l=[L] * 3)
    ref = torch.zeros_like(pos)
    p.add_long_range_forces(pos, q, ref)
    late, busy = torch.zeros_like(pos), torch.zeros(1 << 24, device="cuda")
    f = torch.zeros_like(pos)
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream()):
        for _ in range(50):
            busy += 1.
        late.copy_(pos)
        p.add_long_range_forces(late, q, f)
    assert torch.equal(f, ref)
