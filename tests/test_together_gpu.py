"""Small periodic boxes, whose x, y and z derivatives share a launch, against the
same boxes stacked until they launch each direction by itself: the arithmetic
and the order of the divergence's sum are the same, so members and standalone
solvers agree bit for bit.  36 and 60 points leave a partial last workgroup of
lines; the stacks are the smallest beyond 2560 waves a direction."""
import numpy as np
import pytest

from mpi_3dcompact_amd import hit

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("n,members,les", [(36, 11, None), (48, 6, "VREMAN"), (56, 7, None), (60, 4, None), (64, 3, "VREMAN")])
@pytest.mark.parametrize("fd", ["PADE6", "PENTA10"])
def test_shared_launch_equals_separate_launches(n, members, les, fd):
    from mpi_3dcompact_amd.ensemble import Ensemble
    from mpi_3dcompact_amd.solver import Solver
    case = dict(fd=fd, filt="COMPACT10", alpha_f=0.49, rk="RK4", cfl=0.5)
    if les:
        case.update(les=les, les_avg="NONE")
    mu = [1e-3 / (1 + m) for m in range(members)]
    start = [hit.hit_initial_condition(n, k0=4.0, Mt=0.3, seed=m) for m in range(members)]
    e = Ensemble(hit.options_text(n, **case), [(n,) * 3] * members, mu)
    assert e.info()["buckets"][0]["shared"] == [False, False]
    for m in range(members):
        e.set_metrics(m, hit.identity_metrics(n))
        e.set_initial(m, start[m])
    e.step(2)
    for m in (0, members - 1):
        g = Solver(hit.options_text(n, mu_ref=mu[m], **case), (n,) * 3)
        g.set_metrics(hit.identity_metrics(n))
        g.set_initial(start[m])
        g.timing(True)
        g.step(2)
        assert "lineop_together" in str(g.timing_report()), g.timing_report()
        for f in ("rho", "rhoU", "rhoV", "rhoW", "rhoE", "p"):
            assert np.array_equal(e.field(m, f), g.field(f)), (m, f)
