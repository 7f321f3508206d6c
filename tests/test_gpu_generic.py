"""The general element kernel (elem_general.hip; p = 3 with 4 points has a stiffness kernel of its own,
p = 3 and 4 with p + 1 points a mass kernel) on degree triples and Gauss orders that only it takes -- unequal
degrees per direction, NBINT other than (p + 1)^3 -- against the oracle (COO indices bit-exact,
values and F within 1e-12 of their maximum), in the serial (packed) and OpenMP (slotted) layouts of
the drop-ins, and the consistent mass matrix, the shape gradients (factorised at max(p) + 1 points,
the run-time-order kernel at others), the VTU vertex fields and the displacement at parametric
points on the same cases.
"""
import os

import numpy as np
import pytest

from oracle import oracle as O
from yeti_amd.geometry import make_box_patch
from yeti_amd.model import IGAparametrization

MODELS = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "models")


def box(p, ng):
    return make_box_patch(nel=(3, 2, 2), p=p, seed=40 + 10 * p + ng, ngauss=ng).f2py_args()


def refined(name, deg, ref):
    m = IGAparametrization(filename=os.path.join(MODELS, name))
    m.refine(np.array(ref), np.array(deg))
    return m.get_inputs4system_elemStorage()


CASES = {
    "box p=2 ng=4": lambda: box(2, 4),
    "box p=1 ng=3": lambda: box(1, 3),
    "box p=3 ng=3": lambda: box(3, 3),
    "beam degrees (2,3,1)": lambda: refined("beam-dist", (1, 2, 0), (1, 1, 2)),
    "beam degrees (1,1,2)": lambda: refined("load_combination/beam-centrif-dloadF2-dloadF4", (0, 0, 1), (0, 0, 0)),
    "beam degrees (3,2,2)": lambda: refined("volume_force_3D", (2, 1, 1), (1, 1, 1)),
}


def test_cases_take_the_general_path():
    """No case here has the equal degrees and p + 1 points that other kernels are built for."""
    for name, make in CASES.items():
        a = make()
        from yeti_amd._abi import args_to_dict
        d = args_to_dict(a)
        p = np.asarray(d["Jpqr"]).reshape(-1)[:3]
        nbint = int(np.asarray(d["NBINT"]).reshape(-1)[0])
        ng = int(round(nbint ** (1.0 / 3.0)))
        assert not (p[0] == p[1] == p[2] and ng == p[0] + 1), name
        assert np.prod(p + 1) <= 64, name


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(CASES))
def test_gpu_general_degrees_match_oracle(name):
    from yeti_amd.stiffmtrx_elemstorage import sys_linmat_lindef_static
    from yeti_amd.stiffmtrx_elemstorage_omp import sys_linmat_lindef_static_omp
    from yeti_amd._abi import args_to_dict
    from oracle.oracle import YETI_LAYOUT_SLOTTED
    print("[case] general degrees: %s" % name, flush=True)
    args = CASES[name]()
    K, r, c, F = sys_linmat_lindef_static(*args)
    Ko, ro, co, Fo = O.oracle_sys_linmat(args)
    assert np.array_equal(r, ro) and np.array_equal(c, co)
    assert np.abs(K - Ko).max() <= 1e-12 * np.abs(Ko).max()
    assert np.abs(F - Fo).max() <= 1e-12 * max(np.abs(Fo).max(), 1e-300)
    kw = {k.lower(): v for k, v in args_to_dict(args).items()}
    K2, r2, c2, F2 = sys_linmat_lindef_static_omp(**kw)
    Ks, rs, cs, _ = O.oracle_sys_linmat([], layout=YETI_LAYOUT_SLOTTED, kwargs=kw)
    assert np.array_equal(r2, rs) and np.array_equal(c2, cs)
    assert np.abs(K2 - Ks).max() <= 1e-12 * np.abs(Ks).max()


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(CASES))
def test_gpu_general_degrees_mass_match_oracle(name):
    from yeti_amd._abi import args_to_dict
    from yeti_amd.assembly import Assembler
    print("[case] general degrees mass: %s" % name, flush=True)
    d = args_to_dict(CASES[name]())
    d["RHO"] = np.full(int(np.asarray(d["nb_elem_patch"]).size), 7.8)
    asm = Assembler(d)
    try:
        M, r, c = asm.run_mass()
        Mo, ro, co = O.oracle_mass_coo(d)
        n = Mo.size
        assert np.array_equal(r[:n].cpu().numpy(), ro) and np.array_equal(c[:n].cpu().numpy(), co)
        assert np.abs(M[:n].cpu().numpy() - Mo).max() <= 1e-12 * np.abs(Mo).max()
    finally:
        asm.close()


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(CASES))
def test_gpu_general_degrees_vib_grad_match_oracle(name):
    from yeti_amd._abi import args_to_dict
    from yeti_amd.assembly import Assembler
    print("[case] general degrees vibration gradient: %s" % name, flush=True)
    d = args_to_dict(CASES[name]())
    d["RHO"] = np.full(int(np.asarray(d["nb_elem_patch"]).size), 7.8e-9)
    ncp = int(np.asarray(d["COORDS3D"]).shape[1])
    V = np.random.default_rng(5).standard_normal((5, 3, ncp))
    L = np.linspace(1e6, 4e7, 5)
    asm = Assembler(d)
    try:
        g = asm.run_vib_grad(V, L).cpu().numpy()
    finally:
        asm.close()
    go = O.oracle_grad_vibration(d, V, L)
    assert np.abs(g - go).max() <= 1e-11 * np.abs(go).max()


def _energy(d, u):
    """u^T K u from the oracle's packed COO (upper blocks, diagonal halved: K = C + C^T)."""
    K, r, c, _ = O.oracle_sys_linmat([], kwargs={k.lower(): v for k, v in d.items()})
    return 2.0 * float(np.sum(K * u[r] * u[c]))


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(CASES))
def test_gpu_general_degrees_strain_energy_grad(name):
    """-d(u^T K u)/dX of Assembler.strain_energy_grad against (1) the oracle's natural-frequency
    gradient with eigenvalue 0 times the mode mass u^T M u (that gradient divides by it), within
    1e-11 of the maximum, and (2) central differences of the oracle's u^T K(X) u along random
    directions (step 1e-5 of the model size, within 1e-6 of |g| |d|)."""
    import torch
    from yeti_amd._abi import args_to_dict
    from yeti_amd.assembly import Assembler
    print("[case] general degrees strain energy gradient: %s" % name, flush=True)
    d = args_to_dict(CASES[name]())
    d["RHO"] = np.full(int(np.asarray(d["nb_elem_patch"]).size), 7.8)
    X = np.asarray(d["COORDS3D"], dtype=np.float64)
    ncp = X.shape[1]
    V = np.random.default_rng(6).standard_normal((1, 3, ncp))
    u = np.ascontiguousarray(V[0].T.reshape(-1))
    asm = Assembler(d)
    try:
        g = asm.strain_energy_grad(torch.from_numpy(u).cuda()).cpu().numpy()
    finally:
        asm.close()
    M, rm, cm = O.oracle_mass_coo(d)
    mass = 2.0 * float(np.sum(M * u[rm] * u[cm]))
    go = -O.oracle_grad_vibration(d, V, np.zeros(1))[0].T.reshape(-1) * mass
    assert np.abs(g - go).max() <= 1e-11 * np.abs(go).max()
    size = float(np.ptp(X, axis=1).max())
    rng = np.random.default_rng(7)
    for k in range(2):
        dX = rng.standard_normal(X.shape)
        h = 1e-5 * size
        dp, dm = dict(d), dict(d)
        dp["COORDS3D"] = np.asfortranarray(X + h * dX)
        dm["COORDS3D"] = np.asfortranarray(X - h * dX)
        fd = -(_energy(dp, u) - _energy(dm, u)) / (2 * h)
        an = float(g @ dX.T.reshape(-1))
        assert abs(fd - an) <= 1e-6 * np.linalg.norm(g) * np.linalg.norm(dX), (fd, an)


@pytest.mark.gpu
@pytest.mark.parametrize("name,make", [("p=3, 4 points", lambda: box(3, 4)), ("p=4, 5 points", lambda: box(4, 5)),
                                       ("degrees (2,3,1)", CASES["beam degrees (2,3,1)"]),
                                       ("p=3, 3 points", lambda: box(3, 3)), ("p=1, 3 points", lambda: box(1, 3))])
def test_gpu_work_gradients_of_different_fields(name, make):
    """grad_lin_elast_work for a state and 5 adjoints that differ from it (more than one launch
    takes), factorised and with run-time orders: -a^T (dK/dX) u by polarisation,
    (E(u - a) - E(u + a)) / 4 with E(v) = v^T (dK/dX) v from the oracle's natural-frequency gradient
    at eigenvalue 0 times v^T M v, within 1e-11 of the maximum."""
    import torch
    from yeti_amd._abi import args_to_dict
    from yeti_amd.assembly import Assembler
    print("[case] work gradients of different fields: %s" % name, flush=True)
    d = args_to_dict(make())
    d["RHO"] = np.full(int(np.asarray(d["nb_elem_patch"]).size), 7.8)
    ncp = int(np.asarray(d["COORDS3D"]).shape[1])
    rng = np.random.default_rng(8)
    u, adj = rng.standard_normal(3 * ncp), rng.standard_normal((5, 3 * ncp))
    asm = Assembler(d)
    try:
        g = asm.grad_lin_elast_work(torch.from_numpy(u).cuda(), torch.from_numpy(adj).cuda())[0].cpu().numpy()
    finally:
        asm.close()
    v = np.concatenate([u - adj, u + adj])
    M, rm, cm = O.oracle_mass_coo(d)
    mass = 2.0 * (v[:, rm] * v[:, cm]) @ M
    E = O.oracle_grad_vibration(d, v.reshape(10, ncp, 3).transpose(0, 2, 1), np.zeros(10))
    E = E.transpose(0, 2, 1).reshape(10, 3 * ncp) * mass[:, None]
    go = (E[:5] - E[5:]) / 4
    for k in range(5):
        assert np.abs(g[k] - go[k]).max() <= 1e-11 * np.abs(go[k]).max(), k


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(CASES))
def test_gpu_general_degrees_postprocessing_match_oracle(name):
    from yeti_amd._abi import args_to_dict
    from yeti_amd.postproc import evaldisp_points, svars_solid
    print("[case] general degrees post-processing: %s" % name, flush=True)
    d = args_to_dict(CASES[name]())
    ncp = int(np.asarray(d["COORDS3D"]).shape[1])
    sol = np.random.default_rng(6).standard_normal((ncp, 3)) * 1e-3
    kw = dict(IEN=d["IEN"], elementsByPatch=d["nb_elem_patch"], Nkv=d["Nkv"], Ukv=d["Ukv"], Nijk=d["Nijk"],
              weight=d["weight"], Jpqr=d["Jpqr"], NNODE=d["NNODE"])
    sv = svars_solid(1, (2, 2, 2), (True, True, True), sol.T, d["COORDS3D"], MATERIAL_PROPERTIES=d["MATERIAL_PROPERTIES"],
                     **kw)
    so = O.oracle_svars_solid(d, 0, sol, (2, 2, 2), (True, True, True))
    assert sv.shape == so.shape
    assert np.abs(sv[:, :, :6] - so[:, :, :6]).max() <= 1e-13 * np.abs(so[:, :, :6]).max()
    assert np.abs(sv[:, :, 6:] - so[:, :, 6:]).max() <= 1e-11 * np.abs(so[:, :, 6:]).max()
    xi = np.random.default_rng(7).uniform(0.0, 1.0, (256, 3))
    u = evaldisp_points(1, xi, sol.T, **kw)
    uo = O.oracle_evaldisp(1, xi, sol.T, **kw)
    assert np.abs(u - uo).max() <= 1e-13 * np.abs(uo).max()


@pytest.mark.gpu
@pytest.mark.parametrize("deg,nel,ng", [((1, 1, 1), (3, 3, 1), 2), ((2, 2, 2), (5, 1, 2), 3), ((4, 2, 1), (2, 2, 2), 5),
                                        ((3, 3, 2), (2, 1, 2), 4), ((3, 4, 2), (1, 2, 1), 5), ((3, 3, 3), (1, 1, 2), 9),
                                        ((4, 4, 4), (3, 2, 2), 5)])
def test_gpu_general_kernel_tiles_and_offsets(deg, nel, ng):
    """elem_general at 8 to 64 nodes and at 125 (one to four or eight node tiles, full and partly
    filled; above 32 nodes the entries leave in several rounds), 8 to 729 points (whole and partial
    chunks), elements whose COO range starts at odd entries and at every inactive-element offset, and
    outputs at an odd address: stiffness and mass against the oracle, indices bit-exact, values
    within 1e-12 of their maximum."""
    import torch
    from perf.cases import _model
    from yeti_amd.assembly import Assembler
    print("[case] general kernel degrees %s ng=%d" % (deg, ng), flush=True)
    case = dict(n0=nel[0], n1=nel[1], n2=nel[2], p0=deg[0], p1=deg[1], p2=deg[2], ng=ng)
    d = _model(case, 3)
    d["activeElement"] = d["activeElement"].copy()
    d["activeElement"][1] = 0
    Ko, ro, co, _ = O.oracle_sys_linmat([], kwargs={k.lower(): v for k, v in d.items()})
    Mo = O.oracle_mass_coo(d)[0]
    asm = Assembler(d)
    try:
        n = asm.nb_data
        for off in (0, 1):
            K = torch.zeros(n + 2, dtype=torch.float64, device="cuda")[off:]
            r, c = (torch.zeros(n + 4, dtype=torch.int32, device="cuda")[k + off:] for k in (0, 1))
            asm.run_matrix(K, r, c)
            assert np.array_equal(r[:n].cpu().numpy(), ro[:n]) and np.array_equal(c[:n].cpu().numpy(), co[:n])
            assert np.abs(K[:n].cpu().numpy() - Ko[:n]).max() <= 1e-12 * np.abs(Ko).max()
            assert float(K[n:].abs().max()) == 0.0
            V = torch.zeros(n + 1, dtype=torch.float64, device="cuda")
            asm.run_values(V)
            assert torch.equal(V[:n], K[:n])
            r.zero_()
            M = asm.run_mass(K, r, c)[0]
            assert np.array_equal(r[:n].cpu().numpy(), ro[:n]) and np.array_equal(c[:n].cpu().numpy(), co[:n])
            assert np.abs(M[:n].cpu().numpy() - Mo[:n]).max() <= 1e-12 * np.abs(Mo).max()
    finally:
        asm.close()


@pytest.mark.gpu
def test_gpu_general_kernel_beyond_one_launch():
    """67,109,864 elements of degree 1, 1000 more than the 64-thread workgroups of 2^32 threads
    (a launch takes fewer and drops the rest without an error): 161 GB of values, every element the same (one set of control points), so
    each must have the bits of the first one, and the first one the values of a one-element model
    (1e-12 of their maximum)."""
    import torch
    from yeti_amd.assembly import Assembler
    print("[case] general kernel beyond one launch", flush=True)
    ne = (1 << 26) + 1000
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 200e9:
        pytest.skip("needs 200 GB of free device memory")
    bp = make_box_patch(nel=(1, 1, 1), p=1, seed=9)
    a = dict(bp.args)
    one = O.oracle_sys_linmat((), kwargs=a)[0]
    a.update(IEN=np.tile(a["IEN"], ne), weight=np.tile(a["weight"], ne), activeElement=np.ones(ne, np.int32),
             Nijk=np.asfortranarray(np.broadcast_to(a["Nijk"], (3, ne))), nb_elem_patch=np.array([ne], np.int32),
             nb_elem=ne, nb_data=300.0 * ne)
    asm = Assembler(a)
    del a
    try:
        K = torch.empty(asm.nb_data, dtype=torch.float64, device="cuda")
        K.fill_(float("nan"))
        asm.run_values(K)
        rows = K.view(ne, 300)
        assert np.abs(rows[0].cpu().numpy() - one).max() <= 1e-12 * np.abs(one).max()
        first = rows[0].clone()
        for i0 in range(0, ne, 1 << 21):
            assert bool((rows[i0:i0 + (1 << 21)] == first).all()), i0
    finally:
        asm.close()
        del K, rows
        torch.cuda.empty_cache()
