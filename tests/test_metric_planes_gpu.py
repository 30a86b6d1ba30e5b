"""The pointwise kernels over meshes that repeat their first z-plane: the same
bits as with every point's own metric terms, and no plane is taken for repeated
that is not."""
import numpy as np
import pytest

from mpi_3dcompact_amd import hit

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def streamed(s, n):
    """Metric fields that k_flux reads point by point: 10, or 0 where it reads one plane."""
    s.timing(True)
    s.step(1)
    (k,) = [r for r in s.timing_report() if r["kernel"] == "k_flux"]
    return round(k["bytes"] / (8 * n * k["count"])) - 38  # 22 other fields and mu_sgs read, 15 written


def run(dims, metrics, own, again=None, steps=2, fields=None):
    """Conserved and k2 fields after some steps; own: every point streams its own
    metric terms (a metric field's address was handed out); again: metrics set
    after the first step; fields: how many metric fields must stream then."""
    from mpi_3dcompact_amd.solver import Solver
    shape = dims[::-1]
    s = Solver(hit.options_text(dims[0], fd="PADE6", filt="COMPACT8", rk="KENRK4", les="VREMAN", les_avg="NONE",
                                mu_ref=1e-3, dims=dims), shape)
    s.set_metrics(metrics)
    r = np.random.default_rng(5)
    s.set_initial(dict(rho=1.0 + 0.1 * r.random(shape), p=1.0 / 1.4 + 0.1 * r.random(shape),
                       **{k: 0.2 * r.standard_normal(shape) for k in "UVW"}))
    if own:
        s.device_ptr("J11")
    s.step(1)
    if again is not None:
        s.set_metrics(again)
    s.step(steps - 1)
    out = {n: s.field(n) for n in ("rho", "rhoU", "rhoV", "rhoW", "rhoE", "rhok2", "rhoUk2", "rhoEk2", "sos", "mu_sgs")}
    if fields is not None:
        assert streamed(s, dims[0] * dims[1] * dims[2]) == fields
    return out


def extruded(dims):
    """Non-diagonal metrics that depend on (x, y) alone."""
    nx, ny, nz = dims
    r = np.random.default_rng(2)
    base = hit.identity_metrics(8)
    return [np.broadcast_to(b[0, 0, 0] * (1.0 + 0.05 * r.random((ny, nx))) + 0.001 * r.random((ny, nx)),
                            (nz, ny, nx)).copy() for b in base]


@pytest.mark.parametrize("dims", [(32, 32, 32), (13, 12, 36), (64, 20, 16), (17, 17, 40)])
def test_repeated_planes_give_the_same_bits(dims):
    m = extruded(dims)
    a, b = run(dims, m, False, fields=0), run(dims, m, True, fields=10)
    for k in a:
        assert np.all(np.isfinite(a[k])) and np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("field", [0, 2, 9])
def test_one_point_of_the_last_plane(field):
    """A single value off by one bit in the last plane makes the planes differ, and
    one off by a hundredth shows in the results."""
    dims = (32, 16, 16)
    m = extruded(dims)
    m[field][-1, -1, -1] = np.nextafter(m[field][-1, -1, -1], 10.0)
    a, b = run(dims, m, False, fields=10), run(dims, m, True)
    m[field][-1, -1, -1] *= 1.01
    c, d = run(dims, m, False, fields=10), run(dims, m, True)
    for k in a:
        assert np.array_equal(a[k], b[k]) and np.array_equal(c[k], d[k]), k
    assert not np.array_equal(c["rhoE"], run(dims, extruded(dims), False)["rhoE"])


def test_metrics_set_again():
    """New metrics between steps are looked at again, in both directions."""
    dims = (32, 16, 16)
    m, v = extruded(dims), extruded(dims)
    v[5][3:] *= 1.02
    for first, second in ((m, v), (v, m)):
        a, b = run(dims, first, False, again=second, fields=10 if second is v else 0), run(dims, first, True, again=second, fields=10)
        for k in a:
            assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("order", [(0, 1, 2), (2, 1, 0), (1, 0, 2, 0), (0, 1, 2, 1)])
def test_stacked_members(order):
    """Members set in any order, some again: a member whose planes differ from the
    first member's (a plane of its own, or another first plane) is found whenever
    it is set, and one that repeats it after all is not left marked.  Bit for bit
    the members' standalone runs."""
    from mpi_3dcompact_amd.ensemble import Ensemble
    from mpi_3dcompact_amd.solver import Solver
    dims = (32, 16, 16)
    shape = dims[::-1]
    text = hit.options_text(dims[0], fd="PADE6", filt="COMPACT8", rk="KENRK4", les="VREMAN", les_avg="NONE",
                            mu_ref=1e-3, dims=dims)
    same, last, other = extruded(dims), extruded(dims), [1.25 * f for f in extruded(dims)]
    last[4][-1] *= 1.02
    r = np.random.default_rng(5)
    ic = [dict(rho=1.0 + 0.1 * r.random(shape), p=1.0 / 1.4 + 0.1 * r.random(shape),
               **{k: 0.2 * r.standard_normal(shape) for k in "UVW"}) for _ in range(3)]
    for first in ((same, same, same), (same, last, same), (last, same, same), (same, other, same), (other, same, same)):
        given = list(first)
        e = Ensemble(text, [dims] * 3)
        seen = set()
        for m in order:
            if m in seen:  # set again: the member's metrics change
                given[m] = last if given[m] is same else same
            e.set_metrics(m, given[m])
            seen.add(m)
        for m in range(3):
            e.set_initial(m, ic[m])
        e.step(2)
        for m in range(3):
            g = Solver(text, shape)
            g.set_metrics(given[m])
            g.set_initial(ic[m])
            g.step(2)
            for f in ("rho", "rhoU", "rhoE", "p"):
                assert np.array_equal(e.field(m, f), g.field(f)), (order, m, f)
