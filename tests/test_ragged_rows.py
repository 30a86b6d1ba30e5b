"""Ragged lines in 20- and 28-row chunks: lengths whose remainder over 16 or 32
rows is too short for the interface blocks (65, 129, 193, 257, ... points), and
y/z-lines of 257 to 320 points; and the chunk rows of evenly chunked y/z-lines."""
import numpy as np
import pytest

import test_plan_cpu as plan
from oracle import pyoracle as P

OPS = [(0, P.PADE6, 0.0), (0, P.PENTA10, 0.0), (1, P.COMPACT8, 0.49), (1, P.COMPACT10, 0.49), (1, P.COMMN5PADE, 0.0)]


@pytest.mark.parametrize("mm", [20, 28])
@pytest.mark.parametrize("n", [49, 65, 66, 97, 129, 131, 193, 225, 257, 289, 310])
def test_plan_replay(monkeypatch, n, mm):
    """The fast kernels' arithmetic over these chunks, replayed on the CPU
    against the oracle for every banded operator and boundary (bound: the
    operators' 1e-12)."""
    def ragged(t):
        return (t["N"] != t["P"] * t["MM"] and t["P"] >= 3 and t["clen"][1] < t["MM"]
                and all(c == t["MM"] for i, c in enumerate(t["clen"]) if i != 1))

    monkeypatch.setattr(plan, "ragged", ragged)
    chunks = -(-n // mm)
    for cls, kind, af in OPS:
        W = 2 if (cls, kind) in ((0, P.PENTA10), (1, P.COMMN5PADE)) else 1
        if n % mm == 0 or chunks < 3 or n - (chunks - 1) * mm < 2 * W:
            continue
        for bc in (P.PERIODIC, P.DIRICHLET):
            dd = 1.0 / n if bc == P.PERIODIC else 1.0 / (n - 1)
            t = plan.tables(cls, kind, bc, n, dd, af, mm)
            assert t["MM"] == mm and plan.fast_eligible(t)
            plan._check(t, (lambda f: P.deriv_line(kind, bc, f, dd)) if cls == 0
                        else (lambda f: P.filter_line(kind, bc, f, af)), n)


@pytest.mark.parametrize("others", [(8, 9), (32, 24)])
def test_every_length_has_a_kernel(others):
    """Every operator is accepted on every length from 11 to 4096 points, whatever
    remainder 16- and 32-row chunks leave, and a singular operator is refused as
    one at every length."""
    from mpi_3dcompact_amd._lib import Mc3dError
    from mpi_3dcompact_amd.ops import plan_kernel
    short = (211, 226, 227, 241, 242, 243, 257, 258, 259, 289, 321, 322, 323, 353, 481, 609, 641, 737, 865, 961,
             993, 994, 995, 1025, 1026, 1057)
    for n in [*range(11, 260, 3), *short]:
        for d in range(3):
            dims = list(others)
            dims.insert(d, n)
            for cls, kind, af in OPS:
                for bc in (P.PERIODIC, P.DIRICHLET):
                    bc3 = [0, 0, 0]
                    bc3[d] = bc
                    assert plan_kernel(cls, kind, d, bc3, dims, 0.1, af).startswith("lineop_")
    for n in (2049, 4033):
        assert plan_kernel(0, P.PADE6, 1, (1, 1, 1), (32, n, 24)).startswith("lineop_kernel<")
    for n in (64, 257):
        with pytest.raises(Mc3dError, match="zero pivot"):
            plan_kernel(1, P.COMPACT8, 1, (0, 0, 0), (32, n, 24), 1.0, 1.0)


def test_short_remainders_take_fast_kernels():
    """512 lines or more of 32 k + 1 points (W = 2: + 2, + 3 too) in 20- or 28-row chunks."""
    from mpi_3dcompact_amd.ops import plan_kernel
    for n, mm in ((81, 28), (129, 20), (161, 28), (241, 28), (257, 20), (258, 20), (289, 20), (321, 28), (353, 28)):
        for d in range(3):
            dims = [32, 24]
            dims.insert(d, n)
            k = plan_kernel(0, P.PENTA10, d, (1, 1, 1), dims)
            assert f", {mm}, false, ragged>" in k, (n, d, k)


@pytest.mark.parametrize("cus", [32, 256, 304])
def test_rules_follow_the_device(cus):
    """Four chunks of y/z-lines, and x-lines in groups, by workgroups (64 lines) a CU."""
    from mpi_3dcompact_amd.ops import plan_kernel
    def rows(d, dims):
        return plan_kernel(0, P.PENTA10, d, (1, 1, 1), dims, cus=cus)
    for n, four in ((64, 16), (96, 24)):
        assert f", {four}, " in rows(2, (48 * cus, 1, n)) and ", 32, " in rows(2, (48 * cus + 1, 1, n))
    for n, lines in ((112, 3 * 64 * cus), (150, 16 * cus), (160, 64 * cus + 1), (256, 64 * cus + 1)):
        assert "_groups<" in rows(0, (n, lines, 1)) and "_groups<" not in rows(0, (n, lines - 1, 1)), n


@pytest.mark.gpu
@pytest.mark.parametrize("n", [993, 1026])
@pytest.mark.parametrize("d", [0, 1, 2])
def test_long_short_remainders(n, d):
    """Lines above 992 points whose remainder over 32 rows is too short, in more
    chunks of fewer rows, against the oracle at the operators' 1e-12."""
    import torch
    from mpi_3dcompact_amd.ops import LineOp
    dims = [11, 12]
    dims.insert(d, n)
    dims = tuple(dims)
    f = np.random.default_rng(n + d).normal(size=dims[::-1])
    fin = torch.from_numpy(f).cuda()
    out = torch.empty_like(fin)
    for cls, kind, af in OPS:
        for bc in (P.PERIODIC, P.DIRICHLET):
            dd = 1.0 / n if bc == P.PERIODIC else 1.0 / (n - 1)
            bc3 = [0, 0, 0]
            bc3[d] = bc
            op = LineOp.deriv(kind, d, bc, dims, dd) if cls == 0 else LineOp.filter(kind, af, d, bc3, dims)
            print(f"n={n} dir={d} cls={cls} kind={kind} bc={bc} {op.kernel()}", flush=True)
            want = P.deriv_field(kind, d, bc, f, dd) if cls == 0 else P.filter_field(kind, af, d, bc3, f)
            op.apply([fin], [out])
            assert np.max(np.abs(out.cpu().numpy() - want)) <= 1e-12 * np.max(np.abs(want)), (cls, kind, bc)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [241, 257])
@pytest.mark.parametrize("d", [0, 1, 2])
def test_few_lines_of_short_remainders(n, d):
    """Fewer than 512 lines, which take 32-row chunks, and the transformed-periodic
    twin of the 20- and 28-row plans, which takes 32-row chunks as well."""
    import torch
    from mpi_3dcompact_amd.ops import LineOp
    rng = np.random.default_rng(n + d)
    for others in ([12, 11], [25, 24]):
        dims = list(others)
        dims.insert(d, n)
        f = rng.normal(size=dims[::-1])
        fin = torch.from_numpy(f).cuda()
        out = torch.empty_like(fin)
        for kind in (P.PADE6, P.PENTA10):
            for bc in (P.PERIODIC, P.DIRICHLET):
                op = LineOp.deriv(kind, d, bc, tuple(dims), 1.0 / n)
                print(f"n={n} dir={d} kind={kind} bc={bc} {op.kernel()}", flush=True)
                op.apply([fin], [out])
                want = P.deriv_field(kind, d, bc, f, 1.0 / n)
                assert np.max(np.abs(out.cpu().numpy() - want)) <= 1e-12 * np.max(np.abs(want)), (kind, bc)
            op = LineOp.deriv(kind, d, P.PERIODIC, tuple(dims), 1.0 / n)
            wraps = [rng.normal(size=others[0] * others[1]) for _ in range(6)]
            op.apply_tpb(fin, out, [torch.from_numpy(w).cuda() for w in wraps])
            want = P.deriv_field_tpb(kind, d, f, 1.0 / n, wraps)
            assert np.max(np.abs(out.cpu().numpy() - want)) <= 1e-12 * np.max(np.abs(want)), kind


@pytest.mark.gpu
@pytest.mark.parametrize("n", [49, 65, 81, 97, 129, 131, 161, 193, 225, 241, 257, 289, 305, 310, 321])
@pytest.mark.parametrize("d", [0, 1, 2])
def test_lines_against_oracle(n, d):
    """Every banded operator on lines of n points among 24 x 24 others, both
    boundaries, out of place and (filters) in place, at the operators' 1e-12."""
    import torch
    from mpi_3dcompact_amd.ops import LineOp
    dims = [25, 24, 24]
    dims[d] = n
    if d:
        dims[0] = 26  # a last workgroup that is not full
    dims = tuple(dims)
    f = np.random.default_rng(n + d).normal(size=dims[::-1])
    fin = torch.from_numpy(f).cuda()
    for cls, kind, af in OPS:
        for bc in (P.PERIODIC, P.DIRICHLET):
            dd = 1.0 / n if bc == P.PERIODIC else 1.0 / (n - 1)
            bc3 = [0, 0, 0]
            bc3[d] = bc
            op = LineOp.deriv(kind, d, bc, dims, dd) if cls == 0 else LineOp.filter(kind, af, d, bc3, dims)
            print(f"n={n} dir={d} cls={cls} kind={kind} bc={bc} {op.kernel()}", flush=True)
            assert not op.kernel().startswith("lineop_kernel<"), op.kernel()
            want = P.deriv_field(kind, d, bc, f, dd) if cls == 0 else P.filter_field(kind, af, d, bc3, f)
            out = torch.empty_like(fin)
            op.apply([fin], [out])
            if cls == 1:
                same = fin.clone()
                op.apply([same], [same])
                assert torch.equal(same, out)
            assert np.max(np.abs(out.cpu().numpy() - want)) <= 1e-12 * np.max(np.abs(want)), (cls, kind, bc)


@pytest.mark.gpu
@pytest.mark.parametrize("n,mm", [(64, 16), (96, 24), (144, 24), (160, 20), (224, 28), (240, 20), (336, 28), (448, 28),
                                  (112, 16), (128, 32), (256, 32)])
@pytest.mark.parametrize("d", [1, 2])
def test_even_rows(n, mm, d):
    """The rows per chunk that evenly chunked y/z-lines take, and every banded
    operator over them against the oracle at 1e-12."""
    import torch
    from mpi_3dcompact_amd.ops import LineOp
    dims = [70, 12, 12]
    dims[d] = n
    dims = tuple(dims)
    f = np.random.default_rng(n + d).normal(size=dims[::-1])
    fin = torch.from_numpy(f).cuda()
    for cls, kind, af in OPS:
        for bc in (P.PERIODIC, P.DIRICHLET):
            dd = 1.0 / n if bc == P.PERIODIC else 1.0 / (n - 1)
            bc3 = [0, 0, 0]
            bc3[d] = bc
            op = LineOp.deriv(kind, d, bc, dims, dd) if cls == 0 else LineOp.filter(kind, af, d, bc3, dims)
            assert f", {mm}, " in op.kernel() and op.kernel().startswith("lineop_strided<"), op.kernel()
            want = P.deriv_field(kind, d, bc, f, dd) if cls == 0 else P.filter_field(kind, af, d, bc3, f)
            out = torch.empty_like(fin)
            op.apply([fin], [out])
            assert np.max(np.abs(out.cpu().numpy() - want)) <= 1e-12 * np.max(np.abs(want)), (cls, kind, bc)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [96, 97, 105, 112, 131, 144, 150, 160, 165, 170, 192, 193, 200, 224, 230, 250, 256])
def test_grouped_x_lines(n):
    """x-lines of four or eight chunks staged in groups of 32 or 16 lines (17424
    or 49632 of them: a last workgroup of 16 or 32), Dirichlet and ragged periodic,
    with pass-through lines and in place, the first and last eight z-planes
    against the oracle at 1e-12."""
    import torch
    from mpi_3dcompact_amd.ops import LineOp
    dims = (n, 33, 528 if n > 112 else 1504)
    f = np.random.default_rng(n).normal(size=dims[::-1])
    fin = torch.from_numpy(f).cuda()
    ends = np.r_[0:8, dims[2] - 8:dims[2]]
    for cls, kind, af in OPS:
        for bc3 in ((0, 0, 0), (1, 0, 0), (1, 1, 1), (0, 1, 1)):
            bc = bc3[0]
            if cls == 0 and sum(bc3[1:]):
                continue
            dd = 1.0 / n if bc == P.PERIODIC else 1.0 / (n - 1)
            op = LineOp.deriv(kind, 0, bc, dims, dd) if cls == 0 else LineOp.filter(kind, af, 0, bc3, dims)
            print(f"n={n} cls={cls} kind={kind} bc3={bc3} {op.kernel()}", flush=True)
            # periodic lines that split evenly (by 16 rows, 200 by 20) keep the 16-line tiles
            if bc == P.DIRICHLET or (n % 16 and n != 200):
                assert op.kernel().startswith("lineop_contig_groups<"), op.kernel()
            sub = np.ascontiguousarray(f[ends])
            want = P.deriv_field(kind, 0, bc, sub, dd) if cls == 0 else P.filter_field(kind, af, 0, list(bc3), sub)
            out = torch.empty_like(fin)
            op.apply([fin, fin], [out, torch.empty_like(fin)])
            if cls == 1:
                same = fin.clone()
                op.apply([same], [same])
                assert torch.equal(same, out)
            assert np.max(np.abs(out.cpu().numpy()[ends] - want)) <= 1e-12 * np.max(np.abs(want)), (cls, kind, bc3)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [97, 131, 160, 193, 230, 256])
@pytest.mark.parametrize("bc", [P.PERIODIC, P.DIRICHLET])
def test_grouped_x_lines_accumulate(n, bc):
    """out += derivative, which the library's internal entry asks for (no public one
    does along x), to the bit the sum of the plain result and what was there."""
    import ctypes
    import torch
    from mpi_3dcompact_amd import lib
    from mpi_3dcompact_amd.ops import LineOp
    add = getattr(lib(), "_ZN4mc3d24lineop_launch_accumulateEPK11mc3d_lineopPKPKdPKPdiiPv")
    add.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_void_p]
    dims = (n, 33, 528 if n > 112 else 1504)
    for kind in (P.PADE6, P.PENTA10):
        op = LineOp.deriv(kind, 0, bc, dims, 1.0 / n)
        if bc == P.DIRICHLET or n % 16:
            assert op.kernel().startswith("lineop_contig_groups<"), op.kernel()
        f = torch.rand(dims[::-1], dtype=torch.float64, device="cuda")
        plain, out = torch.empty_like(f), torch.rand_like(f)
        want = out.clone()
        op.apply([f], [plain])
        pi, po = (ctypes.c_void_p * 1)(f.data_ptr()), (ctypes.c_void_p * 1)(out.data_ptr())
        assert add(op._h, pi, po, 1, 1, torch.cuda.current_stream().cuda_stream) == 0
        assert torch.equal(out, want + plain), (n, kind)


@pytest.mark.gpu
@pytest.mark.parametrize("n,few,many", [(160, 16384, 16385), (256, 16384, 16385), (112, 49151, 49152), (150, 4095, 4096)])
def test_grouped_line_counts(n, few, many):
    """Too few x-lines for two workgroups a CU keep the whole tile."""
    from mpi_3dcompact_amd.ops import LineOp
    assert LineOp.deriv(P.PENTA10, 0, P.DIRICHLET, (n, few, 1), 1.0).kernel().startswith("lineop_contig<")
    assert LineOp.deriv(P.PENTA10, 0, P.DIRICHLET, (n, many, 1), 1.0).kernel().startswith("lineop_contig_groups<")


@pytest.mark.gpu
@pytest.mark.parametrize("n,rows", [(64, 16), (96, 24)])
def test_four_chunk_line_counts(n, rows):
    """Four chunks of y/z-lines up to 12288 lines only."""
    from mpi_3dcompact_amd.ops import LineOp
    assert f", {rows}, " in LineOp.deriv(P.PENTA10, 2, P.PERIODIC, (128, 96, n), 1.0).kernel()
    assert ", 32, " in LineOp.deriv(P.PENTA10, 2, P.PERIODIC, (128, 97, n), 1.0).kernel()
