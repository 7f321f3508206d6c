"""GPU parity of the device CSR of K_side + K_side^T (pattern + values) and of the FP64
Jacobi-PCG, against scipy applied to the oracle's COO exactly as the reference's callers do
(overlay/iga_model.py:391-395: coo_matrix(...).tocsc(); K + K.T).

Bar: CSR indptr/indices identical to scipy's canonical CSR of (K + K^T) (the cases here have no
exact-zero entries, so scipy's zero dropping does not change the pattern); values within
1e-12 * max|A|; SpMV within 1e-12 relative; PCG solution against the reference's direct solve
of the same system within 1e-8 relative (the conditioning of the 10:1 cantilever bounds what any
FP64 solver can reach; the test prints the measured error)."""
import os

import numpy as np
import pytest
import scipy.sparse as sp

from oracle import oracle as O
from tests.helpers import concat_patches
from yeti_amd.geometry import make_box_patch

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def scipy_csr(K, r, c, ndof):
    A = sp.coo_matrix((K, (r, c)), shape=(ndof, ndof)).tocsc()
    A = (A + A.T).tocsr()
    A.sort_indices()
    return A


def _check_case(args_dict, tag):
    import torch
    from yeti_amd.assembly import Assembler
    from yeti_amd.solver import StiffnessCSR
    print("[case]", tag, flush=True)
    asm = Assembler(args_dict)
    K, r, c, F = asm.run_coo()
    csr = StiffnessCSR(asm)
    vals = csr.values(K)
    A = csr.to_scipy(vals)
    K0, r0, c0, F0 = O.oracle_sys_linmat((), kwargs=args_dict)
    ndof = int(args_dict["nb_dof_tot"])
    B = scipy_csr(K0, r0, c0, ndof)
    assert (B.data == 0).sum() == 0, "reference matrix has exact zeros: pattern comparison ill-posed"
    assert np.array_equal(A.indptr, B.indptr), "indptr differs"
    assert np.array_equal(A.indices, B.indices), "indices differ"
    assert np.abs(A.data - B.data).max() <= 1e-12 * np.abs(B.data).max()
    x = torch.from_numpy(np.random.default_rng(1).standard_normal(ndof)).cuda()
    y = csr.spmv(vals, x)
    y0 = B @ x.cpu().numpy()
    assert np.abs(y.cpu().numpy() - y0).max() <= 1e-12 * np.abs(y0).max()
    return asm, csr, K, vals, F


@pytest.mark.parametrize("nel,p", [((16, 4, 4), 2), ((4, 3, 2), 3), ((2, 2, 2), 4), ((3, 2, 2), 1)])
def test_csr_matches_scipy(gpu, nel, p):
    bp = make_box_patch(nel=nel, p=p, seed=3 + p)
    _check_case(bp.args, "csr box %s p=%d" % (nel, p))


def _relabelled(a, seed):
    """The model with its control points numbered at random."""
    ncp = int(a["nb_cp"])
    new = np.random.default_rng(seed).permutation(ncp)          # old id -> new id, 0-based
    X = np.empty_like(a["COORDS3D"])
    X[:, new] = a["COORDS3D"]
    a["COORDS3D"] = np.asfortranarray(X)
    a["IEN"] = (new[a["IEN"] - 1] + 1).astype(np.int32)
    a["bc_target"] = (new[a["bc_target"] - 1] + 1).astype(np.int32)
    free = a["ind_dof_free"][:a["nb_dof_free"]].astype(np.int64) - 1
    ind = np.zeros_like(a["ind_dof_free"])
    ind[:free.size] = np.sort(3 * new[free // 3] + free % 3) + 1
    a["ind_dof_free"] = ind
    return a


ROWS, SHORT, LIST, EVERY = 0, 1, 2, 3


@pytest.mark.parametrize("nel,p,relabel,kinds", [
    ((9, 8, 7), 1, False, (ROWS, SHORT, LIST, EVERY)), ((9, 8, 7), 1, True, (LIST, EVERY)),
    ((6, 5, 5), 2, False, (ROWS, LIST, EVERY)), ((6, 5, 5), 2, True, (LIST, EVERY)),
    ((3, 2, 1), 2, True, (LIST, EVERY)), ((3, 4, 3), 3, True, (LIST, EVERY)),
    ((3, 4, 3), 3, False, (ROWS, LIST, EVERY)), ((3, 2, 2), 4, False, (ROWS, LIST, EVERY))])
def test_csr_values_by_rows_and_by_blocks(gpu, nel, p, relabel, kinds):
    """The ways the values are gathered: whole element rows (elements numbered against their
    control points, one slot per lane, two at p = 4), 16 lanes per short row, the listed blocks
    J >= I with their transposes, and every block by itself, with inactive elements and control
    points in order or numbered at random. Against scipy in the way the model takes by itself; the
    others have its bits, and the ways the model does not allow are refused."""
    import torch
    from yeti_amd._lib import YetiError
    from yeti_amd.solver import StiffnessCSR
    a = dict(make_box_patch(nel=nel, p=p, seed=4 + p).args)
    a["activeElement"] = a["activeElement"].copy()
    a["activeElement"][[0, -1]] = 0
    if relabel:
        a = _relabelled(a, p)
    asm, csr, K, vals, _ = _check_case(a, "csr %s p=%d relabel=%s" % (nel, p, relabel))
    for kind in (ROWS, SHORT, LIST, EVERY):
        if kind not in kinds and not (kind == SHORT and relabel and p == 1):
            with pytest.raises(YetiError):
                StiffnessCSR(asm, kind=kind)
        elif kind in kinds:
            other = StiffnessCSR(asm, kind=kind)
            assert other.kind == kind and torch.equal(other.values(K), vals), kind


@pytest.mark.parametrize("nel,p,relabel,kind", [
    ((9, 8, 7), 1, False, SHORT), ((9, 8, 7), 1, True, EVERY), ((8, 8, 8), 2, False, LIST), ((16, 15, 16), 2, False, ROWS),
    ((16, 15, 16), 2, True, LIST), ((12, 12, 11), 3, False, ROWS), ((8, 8, 8), 4, False, LIST), ((18, 18, 17), 4, False, ROWS),
    (((40, 8, 8), (2, 2, 2)), (1, 4), False, LIST)])
def test_csr_way_taken(gpu, nel, p, relabel, kind):
    """Which way a model takes: element rows from enough rows on (more at p = 4), 16 lanes per row
    at p = 1 unless a patch of higher degree has longer rows, every block where short rows are
    numbered at random, the list of blocks J >= I otherwise."""
    from yeti_amd.assembly import Assembler
    from yeti_amd.solver import StiffnessCSR
    if isinstance(p, tuple):
        a = concat_patches(make_box_patch(nel=nel[0], p=p[0]), make_box_patch(nel=nel[1], p=p[1]))
    else:
        a = dict(make_box_patch(nel=nel, p=p).args)
    if relabel:
        a = _relabelled(a, 7)
    assert StiffnessCSR(Assembler(a)).kind == kind


def test_csr_multipatch(gpu):
    m = concat_patches(make_box_patch(nel=(3, 2, 2), p=2, seed=1), make_box_patch(nel=(2, 2, 2), p=3, seed=2))
    _check_case(m, "csr two patches")


def test_pcg_cantilever_against_direct_solve(gpu):
    import torch
    from yeti_amd.solver import free_mask_from_args
    d = np.load(os.path.join(GOLD, "cantilever_16x4x4_p2.npz"))
    bp = make_box_patch(nel=(16, 4, 4), p=2)
    asm, csr, K, vals, F = _check_case(bp.args, "pcg cantilever")
    mask = free_mask_from_args(bp.args)
    x, it, rel = csr.pcg(vals, F, mask, rtol=1e-13, maxit=200000)
    x2, it2, rel2 = csr.pcg(vals, F, mask, rtol=1e-13, maxit=200000)
    torch.cuda.synchronize()
    assert torch.equal(x, x2) and it == it2, "PCG is not bit-reproducible"
    u = x.cpu().numpy()[d["free0"]]
    err = np.linalg.norm(u - d["u"]) / np.linalg.norm(d["u"])
    print("[pcg] iterations %d, relative residual %.2e, error vs reference direct solve %.2e" % (it, rel, err))
    assert rel <= 1e-13
    assert err <= 1e-8
    # fixed dofs stay exactly zero
    fixed = np.setdiff1d(np.arange(bp.nb_dof_tot), d["free0"])
    assert np.all(x.cpu().numpy()[fixed] == 0.0)


def test_pcg_reports_non_convergence(gpu):
    from yeti_amd._lib import YetiError
    from yeti_amd.solver import free_mask_from_args
    bp = make_box_patch(nel=(4, 2, 2), p=2)
    asm, csr, K, vals, F = _check_case(bp.args, "pcg iteration cap")
    with pytest.raises(YetiError) as ei:
        csr.pcg(vals, F, free_mask_from_args(bp.args), rtol=1e-14, maxit=3)
    assert ei.value.code == 6


def test_canonical_drops_exact_zeros_like_scipy(gpu):
    """The canonical form (scipy's K_side + K_side^T drops entries that sum to exactly 0): with
    exact zeros planted in the device values, the compacted CSR equals scipy's eliminate_zeros of
    the same matrix (indptr, indices and values bit-exact, row order kept)."""
    import torch
    from yeti_amd.assembly import Assembler
    from yeti_amd.solver import StiffnessCSR
    print("[case] canonical with planted zeros", flush=True)
    bp = make_box_patch(nel=(4, 3, 2), p=2, seed=11)
    asm = Assembler(bp.args)
    K, r, c, F = asm.run_coo()
    csr = StiffnessCSR(asm)
    vals = csr.values(K)
    rng = np.random.default_rng(5)
    kill = torch.from_numpy(rng.choice(csr.nnz, csr.nnz // 7, replace=False)).cuda()
    vals[kill] = 0.0
    rp, ci, v = (t.cpu().numpy() for t in csr.canonical(vals))
    rp0, ci0 = csr.pattern_host()
    B = sp.csr_matrix((vals[: csr.nnz].cpu().numpy(), ci0, rp0), shape=(csr.nrows, csr.nrows))
    B.eliminate_zeros()
    assert np.array_equal(rp, B.indptr) and np.array_equal(ci, B.indices) and np.array_equal(v, B.data)
    assert v.size == csr.nnz - kill.numel()


@pytest.mark.parametrize("nel,p", [((16, 4, 4), 2), ((3, 2, 2), 3)])
def test_build_stiffness_matrix_dropin(gpu, nel, p):
    """yeti_amd.solver.build_stiffness_matrix against the reference's own steps on the oracle COO:
    (coo_matrix(...).tocsc() + transpose) (overlay/iga_model.py:389-395): same type (CSC), same
    canonical pattern, values within 1e-12 of max |A|, same rhs."""
    from yeti_amd.solver import build_stiffness_matrix
    print("[case] build_stiffness_matrix %s p=%d" % (nel, p), flush=True)
    bp = make_box_patch(nel=nel, p=p, seed=2 + p)
    A, rhs = build_stiffness_matrix(bp.args)
    K0, r0, c0, F0 = O.oracle_sys_linmat((), kwargs=bp.args)
    n = int(bp.args["nb_dof_tot"])
    S = sp.coo_matrix((K0, (r0, c0)), shape=(n, n), dtype="float64").tocsc()
    B = S + S.transpose()
    assert A.format == B.format == "csc"
    B.sort_indices()
    assert np.array_equal(A.indptr, B.indptr) and np.array_equal(A.indices, B.indices)
    assert np.abs(A.data - B.data).max() <= 1e-12 * np.abs(B.data).max()
    assert np.abs(rhs - F0).max() <= 1e-12 * max(np.abs(F0).max(), 1e-300)


@pytest.mark.parametrize("solver", ["csr", "matrix-free"])
def test_max_norm_stopping_rule(gpu, solver):
    """norm "inf" stops as iga_mf_cg_3d does, on max|r| / max|b| over the free dofs
    (mf_iga_solver.f90:779,935): the reported ratio is <= rtol, the true residual of the returned
    iterate meets it too (to rounding), and the |A||x| product bounds |Ax| entrywise."""
    import torch
    from yeti_amd.assembly import Assembler
    from yeti_amd.matfree import F64, MatrixFree
    from yeti_amd.solver import StiffnessCSR, free_mask_from_args
    print("[case] max-norm stop:", solver, flush=True)
    bp = make_box_patch(nel=(12, 4, 4), p=2, seed=4)
    asm = Assembler(bp.args)
    K, r, c, F = asm.run_coo()
    csr = StiffnessCSR(asm)
    vals = csr.values(K)
    mask = free_mask_from_args(bp.args)
    rtol = 1e-8
    if solver == "csr":
        u, it, rel = csr.pcg(vals, F, mask, rtol=rtol, norm="inf", check_every=1)
        u2, it2, rel2 = csr.pcg(vals, F, mask, rtol=rtol, norm="2", check_every=1)
    else:
        mf = MatrixFree(bp.args, precisions=F64)
        u, it, rel = mf.pcg_f64(F, mask, rtol=rtol, norm="inf", check_every=1)
        u2, it2, rel2 = mf.pcg_f64(F, mask, rtol=rtol, norm="2", check_every=1)
    m = mask.bool()
    res = (F - csr.spmv(vals, u))[m]
    true_inf = float(res.abs().max() / F[m].abs().max())
    print("  inf-norm stop: %d iterations, reported %.3e, true %.3e; 2-norm stop: %d iterations"
          % (it, rel, true_inf, it2), flush=True)
    assert rel <= rtol and true_inf <= 1.01 * rtol and rel2 <= rtol
    ya = csr.spmv_abs(vals, u)
    assert bool(((csr.spmv(vals, u)).abs() <= ya * (1 + 1e-12)).all())
