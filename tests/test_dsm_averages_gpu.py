"""DSM averages read per line or per field: each averaging on boxes of uneven
sizes and in every pencil layout, against a dense restatement of mu_sgs."""
import numpy as np
import pytest

from mpi_3dcompact_amd import hit
from test_oracle_dsm_dense import filter_matrix

pytestmark = pytest.mark.gpu


def dense_mu(g, rho, m, avg, mats):
    """mu_sgs = rho |S| <L:M> / <M:M> on [z, y, x] fields with the test filters as matrices along x, y, z."""
    def F(f):
        f = np.einsum("ij,zyj->zyi", mats[0], f)
        f = np.einsum("ij,zjx->zix", mats[1], f)
        return np.einsum("ij,jyx->iyx", mats[2], f)

    def A(f):
        if avg == "GLOBAL":
            return np.full_like(f, f.mean())
        if avg == "LOCAL":
            return F(f)
        if avg == "NONE":
            return f
        return np.broadcast_to(f.mean(axis={"XI1_AVG": 2, "XI2_AVG": 1, "XI3_AVG": 0}[avg], keepdims=True), f.shape)

    R = range(3)
    S = [[0.5 * (g[i][j] + g[j][i]) for j in R] for i in R]
    smag = np.sqrt(2.0 * sum(S[i][j] ** 2 for i in R for j in R))
    dev = lambda X: [[X[i][j] - ((X[0][0] + X[1][1] + X[2][2]) / 3.0 if i == j else 0.0) for j in R] for i in R]
    Sd, Shd = dev(S), dev([[F(S[i][j]) for j in R] for i in R])
    rh, sh, mh = F(rho), F(smag), [F(v) for v in m]
    M = [[F(2 * rho * smag * Sd[i][j]) - 8.0 * rh * sh * Shd[i][j] for j in R] for i in R]
    Ld = dev([[F(m[i] * m[j] / rho) - mh[i] * mh[j] / rh for j in R] for i in R])
    LM = sum(Ld[i][j] * M[i][j] for i in R for j in R)
    MM = sum(M[i][j] ** 2 for i in R for j in R)
    return rho * smag * A(LM) / A(MM)


@pytest.mark.parametrize("avg", ["NONE", "LOCAL", "GLOBAL", "XI1_AVG", "XI2_AVG", "XI3_AVG"])
@pytest.mark.parametrize("layout", [0, 1, 2])
def test_mu_sgs(avg, layout):
    import torch
    from mpi_3dcompact_amd.sgs import Sgs
    dims = (24, 16, 33) if layout != 2 else (17, 32, 24)
    r = np.random.default_rng(8)
    shape = dims[::-1]
    g = [[r.standard_normal(shape) for _ in range(3)] for _ in range(3)]
    rho = 1.0 + 0.3 * r.random(shape)
    m = [r.standard_normal(shape) for _ in range(3)]
    # [z, y, x] to the layout's order (slowest first): x pencil z y x, y pencil x z y, z pencil y x z
    order = {0: (0, 1, 2), 1: (2, 0, 1), 2: (1, 2, 0)}[layout]
    put = lambda f: torch.from_numpy(np.ascontiguousarray(np.transpose(f, order))).cuda()
    rhoT, mT = put(rho), [put(v) for v in m]
    gT = [put(g[i][j]) for i in range(3) for j in range(3)]
    deck = hit.options_text(dims[0], les="DSM", les_avg=avg, dims=dims, use_taukk=True)
    s = Sgs(deck, torch.ones_like(rhoT), layout=layout)
    mu, tau = torch.empty_like(rhoT), torch.empty_like(rhoT)
    s.dsm_mu_taukk(gT, rhoT, *mT, mu, tau)
    want = dense_mu(g, rho, m, avg, [filter_matrix(1, n) for n in dims])
    got = np.transpose(mu.cpu().numpy(), np.argsort(order))
    # the ratio of the (averaged) contractions carries their relative errors: near-zero denominators (NONE, LOCAL) lose most
    err = np.abs(got - want) / np.maximum(np.abs(want), np.sqrt(np.mean(want ** 2)))
    assert np.quantile(err, 0.99) <= 1e-10 and err.max() <= (1e-6 if avg in ("NONE", "LOCAL") else 1e-10)
