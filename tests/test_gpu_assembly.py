"""GPU parity of the assembly drop-in against the oracle (C restatement) and, where it was
built, the compiled YETI reference (oracle/_ref).

Bar: COO row/col indices bit-exact; values |dK| <= 1e-12 * max|K| entry-wise and a relative
Frobenius error <= 1e-12 (per-entry relative error is ill-posed for near-cancelling entries
because the GPU sums Gauss points in a different order); F within 1e-12 * max|F|.
"""
import numpy as np
import pytest

from oracle import oracle as O
from tests.helpers import all_face_loads, concat_patches, set_loads, with_inactive
from yeti_amd.geometry import make_box_patch

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _cmp(got, exp, tag=""):
    K, r, c, F = got
    K0, r0, c0, F0 = exp
    print("[case]", tag, "nb_data", K0.size, flush=True)
    assert K.shape == K0.shape
    assert np.array_equal(r, r0), "row ids differ"
    assert np.array_equal(c, c0), "col ids differ"
    scale = np.abs(K0).max()
    err = np.abs(K - K0).max()
    assert err <= TOL * scale, "max |dK| = %g (scale %g)" % (err, scale)
    fro = np.linalg.norm(K - K0) / np.linalg.norm(K0)
    assert fro <= TOL, "relative Frobenius %g" % fro
    fs = max(np.abs(F0).max(), 1e-300)
    assert np.abs(F - F0).max() <= TOL * fs, "max |dF| = %g (scale %g)" % (np.abs(F - F0).max(), fs)


def _dropin(args):
    from yeti_amd.stiffmtrx_elemstorage import sys_linmat_lindef_static
    return sys_linmat_lindef_static(*args)


@pytest.mark.parametrize("nel,p", [((16, 4, 4), 2), ((3, 2, 2), 1), ((4, 3, 2), 3), ((2, 2, 3), 4)])
def test_assembly_matches_oracle(gpu, nel, p):
    bp = make_box_patch(nel=nel, p=p, seed=11 + p)
    args = bp.f2py_args()
    _cmp(_dropin(args), O.oracle_sys_linmat(args), "box %s p=%d" % (nel, p))


def test_cantilever_matches_compiled_reference(gpu):
    if not O.ref_available():
        pytest.skip("oracle/_ref not built (YETI sources absent where this tree was built)")
    bp = make_box_patch(nel=(16, 4, 4), p=2)
    args = bp.f2py_args()
    _cmp(_dropin(args), O.ref_sys_linmat_serial(args), "16x4x4 p=2 vs compiled reference")


@pytest.mark.parametrize("p", [2, 3])
def test_all_load_types_match_oracle(gpu, p):
    bp = make_box_patch(nel=(3, 2, 2), p=p, seed=5)
    a = all_face_loads(bp)
    from yeti_amd.stiffmtrx_elemstorage import sys_linmat_lindef_static
    got = sys_linmat_lindef_static(**a)
    exp = O.oracle_sys_linmat((), kwargs=a)
    _cmp(got, exp, "all loads p=%d" % p)


def test_multipatch_and_inactive_packed(gpu):
    m = concat_patches(make_box_patch(nel=(3, 2, 2), p=2, seed=1), make_box_patch(nel=(2, 2, 2), p=3, seed=2))
    m = with_inactive(m)
    n2, n3 = 27, 64
    act = m["activeElement"]
    ne1 = 12
    m["nb_data"] = float(act[:ne1].sum() * (3 * n2) * (3 * n2 + 1) // 2 + act[ne1:].sum() * (3 * n3) * (3 * n3 + 1) // 2)
    from yeti_amd.stiffmtrx_elemstorage import sys_linmat_lindef_static
    _cmp(sys_linmat_lindef_static(**m), O.oracle_sys_linmat((), kwargs=m), "two patches, inactive, packed")


def test_slotted_layout_matches_omp_reference(gpu):
    bp = make_box_patch(nel=(4, 2, 2), p=2, seed=9)
    a = with_inactive(bp.args)
    n = 27
    a["nb_data"] = float(bp.nb_elem * (3 * n) * (3 * n + 1) // 2)   # slotted: every element owns a slot
    from yeti_amd.stiffmtrx_elemstorage_omp import sys_linmat_lindef_static_omp
    kw = {k.lower(): v for k, v in a.items()}
    got = sys_linmat_lindef_static_omp(**kw, num_threads=4)
    exp = O.oracle_sys_linmat((), kwargs=a, layout=1)
    _cmp(got, exp, "slotted")
    if O.ref_available():
        ref = O.ref_sys_linmat_omp((), kwargs=a, num_threads=2)
        _cmp(got, ref, "slotted vs compiled OMP reference")


def test_device_handle_values_only_and_rhs(gpu):
    import torch
    from yeti_amd.assembly import Assembler
    bp = make_box_patch(nel=(6, 3, 3), p=3, seed=4)
    asm = Assembler(bp.f2py_args())
    K, r, c, F = asm.run_coo()
    K2 = torch.full_like(K, float("nan"))
    asm.run_values(K2)
    F2 = asm.run_rhs()
    torch.cuda.synchronize()
    assert torch.equal(K, K2), "values-only run differs from the full run"
    assert torch.equal(F, F2)
    # determinism: a second run is bit-identical
    K3, r3, c3, F3 = asm.run_coo()
    torch.cuda.synchronize()
    assert torch.equal(K, K3) and torch.equal(r, r3) and torch.equal(c, c3) and torch.equal(F, F3)
    exp = O.oracle_sys_linmat(bp.f2py_args())
    _cmp((K.cpu().numpy(), r.cpu().numpy(), c.cpu().numpy(), F.cpu().numpy()), exp, "device handle")


def test_errors_are_raised(gpu):
    from yeti_amd._lib import YetiError
    from yeti_amd.stiffmtrx_elemstorage import sys_linmat_lindef_static
    bp = make_box_patch(nel=(2, 2, 2), p=2)
    a = dict(bp.args)
    a["ELT_TYPE"] = "U3"
    with pytest.raises(YetiError) as ei:
        sys_linmat_lindef_static(**a)
    assert ei.value.code == 2
    a = dict(make_box_patch(nel=(2, 2, 2), p=4).args)
    a["NBINT"] = np.array([216], np.int32)    # p=4 with 6 points: 125 nodes, beyond the general path
    with pytest.raises(YetiError) as ei:
        sys_linmat_lindef_static(**a)
    assert ei.value.code == 3
    a = dict(bp.args)
    a["nb_data"] = 10.0
    with pytest.raises(YetiError) as ei:
        sys_linmat_lindef_static(**a)
    assert ei.value.code == 4


@pytest.mark.parametrize("p,nel", [(4, (16, 16, 2)), (3, (16, 16, 3)), (2, (16, 16, 4)), (1, (16, 16, 6))])
def test_several_elements_per_workgroup(gpu, p, nel):
    """Patches with more elements than workgroups (the element kernel is persistent, one
    workgroup per CU): elements that are the first, second and last of their workgroup, with
    indices (run_matrix) and values only (run_values), against the oracle run on those elements
    alone. Indices bit-exact, values within 1e-12 of the largest magnitude."""
    import torch
    from yeti_amd.assembly import Assembler
    print("[case] several elements per workgroup", p, nel, flush=True)
    bp = make_box_patch(nel=nel, p=p, seed=31 + p)
    args = dict(bp.args)
    n = (p + 1) ** 3
    nde = 9 * n * (n - 1) // 2 + 6 * n
    ne = bp.nb_elem
    sel = np.array(sorted({0, 1, 255, 256, 257, 300, ne // 2, ne - 1}))
    act = np.zeros(ne, np.int32)
    act[sel] = 1
    sub = dict(args)
    sub["activeElement"] = act
    sub["nb_data"] = float(sel.size * nde)
    Ko, ro, co, _ = O.oracle_sys_linmat((), kwargs=sub)
    asm = Assembler(args)
    K, r, c = asm.alloc_coo(True)
    asm.run_matrix(K, r, c)
    Kv = torch.full((asm.nb_data,), float("nan"), dtype=torch.float64, device="cuda")
    asm.run_values(Kv)
    idx = torch.as_tensor((sel[:, None] * nde + np.arange(nde)[None, :]).ravel(), device="cuda")
    scale = np.abs(Ko).max()
    assert np.array_equal(r[idx].cpu().numpy(), ro) and np.array_equal(c[idx].cpu().numpy(), co)
    assert np.abs(K[idx].cpu().numpy() - Ko).max() <= 1e-12 * scale
    assert np.abs(Kv[idx].cpu().numpy() - Ko).max() <= 1e-12 * scale
    asm.close()


@pytest.mark.parametrize("p,ng", [(1, 2), (1, 9), (3, 5), (4, 5)])
def test_load_point_chunks_match_oracle(gpu, p, ng):
    """Every load type with 4 to 729 points per load and 8 to 125 nodes: each split of a load's
    points over the lanes (16, 8 and 4 lanes per point), points past one 64-point chunk and node
    counts on both sides of the splits of the node sums (F within 1e-12 of its maximum: sums of
    at most 729 products of O(1) factors in 64 bits)."""
    print("[case] loads p=%d ng=%d" % (p, ng), flush=True)
    bp = make_box_patch(nel=(2, 2, 1), p=p, seed=6, ngauss=ng)
    a = all_face_loads(bp)
    from yeti_amd.stiffmtrx_elemstorage import sys_linmat_lindef_static
    F = sys_linmat_lindef_static(**a)[3]
    F0 = O.oracle_sys_linmat((), kwargs=a)[3]
    assert np.abs(F - F0).max() <= 1e-12 * np.abs(F0).max()


@pytest.mark.parametrize("face", [5, 6, 7, 8, 9])
def test_face_codes_above_six_load_face_six(gpu, face):
    """The face digit of a load code is 1..9 and every digit above 6 means face 6, as in the oracle:
    normal loads (types 0 and 4) keep face 6's sign on odd digits too, in F (within 1e-12 of its
    maximum) and in 2 u^T dF/dX (central differences of u^T F, step 1e-6: rounding 1e-16 / 1e-6 of
    F and a second-order term, within 1e-6 of the maximum)."""
    import torch
    from yeti_amd.assembly import Assembler
    print("[case] face digit", face, flush=True)
    bp = make_box_patch(nel=(2, 2, 2), p=2, seed=8)
    rng = np.random.default_rng(face)
    nd = np.asfortranarray(rng.uniform(-1, 1, size=(2, bp.nb_cp)))
    u = rng.standard_normal(3 * bp.nb_cp)
    target = np.arange(1, bp.nb_elem + 1, dtype=np.int32)
    for typ in (0, 1, 2, 3, 4):
        a = set_loads(bp.args, [(10 * face + typ, 1.3, target, [2.0] if typ == 4 else [])], nodal_dist=nd)
        F0 = O.oracle_sys_linmat((), kwargs=a)[3]
        asm = Assembler(a)
        try:
            F = asm.run_rhs().cpu().numpy()
            assert np.abs(F - F0).max() <= 1e-12 * np.abs(F0).max(), typ
            g = asm.load_shape_grad(torch.from_numpy(u).cuda()).cpu().numpy()
            X = np.ascontiguousarray(np.asarray(a["COORDS3D"]).T).reshape(-1)
            for i in rng.choice(X.size, 6, replace=False):
                f = []
                for h in (1e-6, -1e-6):
                    Y = X.copy()
                    Y[i] += h
                    asm.update_coords(torch.from_numpy(Y).cuda())
                    f.append(2.0 * float(u @ asm.run_rhs().cpu().numpy()))
                assert abs((f[0] - f[1]) / 2e-6 - g[i]) <= 1e-6 * np.abs(g).max(), (typ, i)
        finally:
            asm.close()


@pytest.mark.parametrize("nel", [(1, 1, 1), (3, 2, 1), (13, 11, 16)])
def test_p3_kernel_runs_and_offsets(gpu, nel):
    """The p = 3 kernel with one element, with fewer elements than the 8 runs they are dealt in, and
    with runs of unequal length and several elements per workgroup; inactive elements; outputs at
    an even and an odd address: indices bit-exact, values within 1e-12 of their maximum of the
    oracle, values only the same bits."""
    import torch
    from yeti_amd.assembly import Assembler
    print("[case] p=3 kernel", nel, flush=True)
    a = dict(make_box_patch(nel=nel, p=3, seed=12).args)
    if a["nb_elem"] > 2:
        a["activeElement"] = a["activeElement"].copy()
        a["activeElement"][[1, -1]] = 0
    Ko, ro, co, _ = O.oracle_sys_linmat((), kwargs=a)
    asm = Assembler(a)
    n = asm.nb_data
    for off in (0, 1):
        K = torch.zeros(n + 2, dtype=torch.float64, device="cuda")[off:]
        r, c = (torch.zeros(n + 4, dtype=torch.int32, device="cuda")[k + off:] for k in (0, 1))
        asm.run_matrix(K, r, c)
        assert np.array_equal(r[:n].cpu().numpy(), ro[:n]) and np.array_equal(c[:n].cpu().numpy(), co[:n])
        assert np.abs(K[:n].cpu().numpy() - Ko[:n]).max() <= 1e-12 * np.abs(Ko).max()
        V = torch.zeros(n + 1, dtype=torch.float64, device="cuda")
        asm.run_values(V)
        assert torch.equal(V[:n], K[:n]) and float(K[n:].abs().max()) == 0.0


def test_right_hand_side_beyond_one_launch(gpu):
    """2^24 + 5 elements of degree 1 with a body load, 5 more than the 256-thread workgroups of 2^32
    threads (a launch takes fewer and drops the rest without an error): element e has the control
    points of group e mod 4096, so F is the one-element model's times the group's element count
    (added one by one: 4097 roundings, 1e-12 of the maximum)."""
    import torch
    from yeti_amd.assembly import Assembler
    ne, ng = (1 << 24) + 5, 4096
    print("[case] right-hand side beyond one launch", flush=True)
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 80e9:
        pytest.skip("needs 80 GB of free device memory")
    bp = make_box_patch(nel=(1, 1, 1), p=1, seed=9)
    one = set_loads(bp.args, [(102, -1.5, [1], [0.2, -0.7, 0.4])])
    F1 = O.oracle_sys_linmat((), kwargs=one)[3]
    group = np.arange(ne, dtype=np.int32) % ng
    every = np.arange(1, ne + 1, dtype=np.int32)
    a = set_loads(bp.args, [(102, -1.5, every, [0.2, -0.7, 0.4])], nodal_dist=np.zeros((1, 8 * ng), order="F"))
    a.update(IEN=(8 * group[:, None] + one["IEN"][None, :]).ravel(), weight=np.tile(one["weight"], ne),
             activeElement=np.ones(ne, np.int32), Nijk=np.asfortranarray(np.broadcast_to(one["Nijk"], (3, ne))),
             nb_elem_patch=np.array([ne], np.int32), nb_elem=ne, nb_data=300.0 * ne, nb_cp=8 * ng, nb_dof_tot=24 * ng,
             COORDS3D=np.asfortranarray(np.tile(one["COORDS3D"], ng)), ind_dof_free=np.arange(1, 24 * ng + 1, dtype=np.int32),
             nb_dof_free=24 * ng)
    asm = Assembler(a)
    del a, every, group
    try:
        F = asm.run_rhs().cpu().numpy().reshape(ng, 24)
    finally:
        asm.close()
    count = np.full(ng, ne // ng)
    count[:ne % ng] += 1
    assert np.abs(F - count[:, None] * F1[None, :]).max() <= 1e-12 * np.abs(F).max()
