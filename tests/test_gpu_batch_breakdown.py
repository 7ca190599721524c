"""A batch in which one case's BiCGstab breaks down while others run on.  A case at
rest has a zero right-hand side and a zero residual: its iteration asks for a new
reference vector and then stops on <rh, Ap> = 0, in a launch whose workgroups see
the flag of the case cleared while they start (the larger grid has more of them
than the device holds at once).  Every case ends as alone.  Tolerance: none."""
import numpy as np
import pytest

import impact_hip as ih

pytestmark = pytest.mark.gpu

W6, PZ = (1,) * 6, (1, 1, 1, 1, -1, -1)


# the batched x update takes one group of planes a tile or four, by the tiles of the batch
@pytest.mark.parametrize("rest", [(33, 17, 17), (257, 97, 97), (249, 97, 97)], ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("sweeps", [0, 1, 4])
def test_a_case_at_rest_beside_running_ones(rest, sweeps):
    spec = [((65, 33, 33), W6), (rest, W6), ((40, 33, 34), PZ)]
    p = ih.StepParams(Re=100.0, dtime=1e-3, jor_sweeps=4, jor_omega=0.8, bicg_rel_tol=1e-9, bicg_max_it=40,
                      level_pressure=1, jor_fp32=int(sweeps > 0), precond_sweeps=sweeps)
    sets = [[ih.Case(N, bc, (2.0, 1.0, 1.0)) for N, bc in spec] for _ in range(2)]
    for cs in sets:
        rng = np.random.default_rng(12)
        for q in (0, 2):
            for f in (ih.VEL1, ih.VEL2, ih.VEL3):
                cs[q].upload(f, 0.01 * rng.standard_normal(cs[q].shape))
    bt = ih.Batch(sets[0])
    for step in range(2):
        sb = bt.timestep(p, step * 1e-3)
        for q, (a, c) in enumerate(zip(*sets)):
            ss = c.timestep(p, step * 1e-3)
            assert list(sb[q].bicg_iterations) == list(ss.bicg_iterations), (step, q)
            assert list(sb[q].bicg_final) == list(ss.bicg_final), (step, q)
            for f in (ih.PRE, ih.VEL1, ih.VEL2, ih.VEL3):
                got, want = a.download(f), c.download(f)
                assert np.array_equal(got, want), f"step {step}, case {q}, field {f}: {int((got != want).sum())} differ"
        assert all(n > 0 for n in sb[1].bicg_iterations), "the case at rest never entered its iteration"
        assert not sets[0][1].download(ih.PRE).any()
    bt.close()
    for c in sets[0] + sets[1]:
        c.close()
