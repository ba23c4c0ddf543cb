"""FP64 GMRES: the cycles on the split operator with each degree of the Neumann polynomial, the
plain cycles where the split operator is not available, the iteration limit inside both, and
the conjugate gradients of the deposition system."""
import numpy as np
import pytest

from chm_amd import abi, meshgen
from tests.conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("points,layers,restart", [
    (13, 2, 1), (13, 5, 3), (300, 5, 3), (300, 16, 4), (300, 17, 4), (2500, 10, 6), (2501, 7, 31),
    (300, 20, 30), (6000, 9, 30), (6000, 9, 4),  # 100,000 rows and more: degree 4
    (106000, 10, 30)])  # a basis vector of more than 16 MB: degree 10
def test_restarted_gmres_solves_the_same_system(points, layers, restart):
    """Both solve to 1e-12, so their fields differ by the forward error of that tolerance alone."""
    from chm_amd import pbsm3d as pb

    print(f"[case] gmres cycles points={points} L={layers} restart={restart}", flush=True)
    mesh = meshgen.synthetic_mesh(points, seed=5)
    g = pb.face_geometry(mesh)
    fo = meshgen.forcing_c2(mesh.n_faces, seed=9)
    ref = pb.Context(g, pb.default_config(nLayer=layers, tol=1e-12, krylov=abi.KRYLOV_BICGSTAB, max_iters=4000))
    ro, rst = ref.step(fo, want_fields=True)
    ctx = pb.Context(g, pb.default_config(nLayer=layers, tol=1e-12, restart=restart, max_iters=4000))
    for _ in range(2):  # the second step reuses the work vectors
        ctx.set_state(np.zeros(mesh.n_faces), np.zeros(mesh.n_faces))
        o, st = ctx.step(fo, want_fields=True)
        assert rst["susp_resid"] <= 1e-12 and st["susp_resid"] <= 1e-12
        for k in ("conc", "Qsusp", "Qsubl", "qdep"):
            assert rel_err(o[k], ro[k]) < 1e-8, (k, rel_err(o[k], ro[k]))
    ctx.close()
    ref.close()


@pytest.mark.parametrize("points,layers", [(2500, 10), (6000, 9), (300, 17)])
def test_iteration_limit_inside_a_cycle(points, layers):
    from chm_amd import pbsm3d as pb

    print(f"[case] gmres iteration limit points={points} L={layers}", flush=True)
    mesh = meshgen.synthetic_mesh(points, seed=0)
    g = pb.face_geometry(mesh)
    fo = meshgen.forcing_c2(mesh.n_faces, seed=9)
    for limit in (1, 3, 4, 5, 7):  # less than, exactly and more than one step of degree 4
        ctx = pb.Context(g, pb.default_config(nLayer=layers, restart=2, max_iters=limit))
        with pytest.raises(pb.Pbsm3dError) as e:
            ctx.step(fo)
        assert e.value.code == abi.PBSM3D_ENOCONV
        ctx.close()


def test_second_orthogonalisation_pass():
    """ortho_passes = 2 adds the conditional pass; the solution is the same."""
    from chm_amd import pbsm3d as pb

    print("[case] gmres two passes", flush=True)
    mesh = meshgen.synthetic_mesh(1201, seed=6)
    g = pb.face_geometry(mesh)
    fo = meshgen.forcing_c2(mesh.n_faces, seed=3)
    out = []
    for passes in (1, 2):
        ctx = pb.Context(g, pb.default_config(nLayer=6, tol=1e-12, ortho_passes=passes, max_iters=4000))
        o, st = ctx.step(fo, want_fields=True)
        assert st["susp_resid"] <= 1e-12 and st["dep_resid"] <= 1e-12
        out.append(o)
        ctx.close()
    for k in ("conc", "qdep"):
        assert rel_err(out[0][k], out[1][k]) < 1e-8


@pytest.mark.parametrize("points,layers", [(12, 2), (40, 3), (300, 5), (2501, 5), (20011, 5)])
@pytest.mark.parametrize("smooth", [0.0, 820.0, -2.0e3])
def test_deposition_cg_and_its_fallback(points, layers, smooth):
    """The deposition system by conjugate gradients against GMRES with the Jacobi preconditioner, both to
    1e-12: the default smoothing, none (a diagonal system), and a negative coefficient, whose
    indefinite system either goes to GMRES or is refused by both."""
    from chm_amd import pbsm3d as pb

    print(f"[case] deposition cg points={points} smooth={smooth}", flush=True)
    mesh = meshgen.synthetic_mesh(points, seed=8, extent=1.0e3 if smooth < 0 else 1.0e4)
    g = pb.face_geometry(mesh)
    fo = meshgen.forcing_c2(mesh.n_faces, seed=4)
    res = []
    for pc in (abi.PC_MCILU0, abi.PC_JACOBI):
        ctx = pb.Context(g, pb.default_config(nLayer=layers, tol=1e-12, dep_precond=pc, smooth_coeff=smooth,
                                              max_iters=600))
        try:
            o, st = ctx.step(fo, want_fields=True)
            assert st["dep_resid"] <= 1e-12
            res.append(o["qdep"])
        except pb.Pbsm3dError as e:
            assert smooth < 0 and e.code == abi.PBSM3D_ENOCONV
        ctx.close()
    assert len(res) == 2 or smooth < 0
    if len(res) == 2 and smooth >= 0:
        assert rel_err(res[0], res[1]) < 1e-8


def _residual(ctx, conc):
    """||b - A x|| / ||b|| of the exported suspension system, on the host."""
    import scipy.sparse as sp

    rp, col, val, b = ctx.system(0)
    A = sp.csr_matrix((val, col, rp), shape=(b.size, b.size))
    return np.linalg.norm(b - A @ conc) / np.linalg.norm(b)


def test_limit_that_plain_cycles_meet(oracle):
    """max_iters bounds GMRES's own iterations: a limit that GMRES(30) with the same preconditioner
    meets is met, also where the polynomial's applications would exceed it."""
    from chm_amd import pbsm3d as pb

    print("[case] gmres limit of plain cycles", flush=True)
    mesh = meshgen.synthetic_mesh(6000, seed=5)
    g = pb.face_geometry(mesh)
    fo = meshgen.forcing_c2(mesh.n_faces, seed=9)
    orc = oracle.Oracle(g, oracle.oracle_config(nLayer=9, precond=abi.PC_MCILU0))
    _, ost = orc.step(fo)
    for limit in (ost["susp_iters"] + 1, ost["susp_iters"] + 3):
        ctx = pb.Context(g, pb.default_config(nLayer=9, max_iters=limit))
        o, st = ctx.step(fo, want_fields=True)
        assert st["susp_iters"] <= limit and st["susp_resid"] <= 1e-8
        assert _residual(ctx, o["conc"]) <= 1.01e-8
        ctx.close()


def test_spectrum_that_the_polynomial_does_not_suit():
    """A small negative diffusion constant leaves a system that GMRES(30) solves in 40 iterations and
    the polynomial's cycles (degree 10 at this size) do not solve in 1000 applications."""
    from chm_amd import pbsm3d as pb

    print("[case] gmres negative diffusion", flush=True)
    mesh = meshgen.synthetic_mesh(106000, seed=5)
    g = pb.face_geometry(mesh)
    fo = meshgen.forcing_c2(mesh.n_faces, seed=9)
    ctx = pb.Context(g, pb.default_config(nLayer=10, snow_diffusion_const=-0.024))
    o, st = ctx.step(fo, want_fields=True)
    assert st["susp_iters"] < 100 and st["susp_resid"] <= 1e-8
    assert _residual(ctx, o["conc"]) <= 1.01e-8
    ctx.close()


def test_rejected_cycle_leaves_the_start_as_it_was():
    """A polynomial cycle after which the residual is larger than before: plain cycles go on from the x
    before it, so the whole solve takes that cycle's 30 steps of degree 10 and what plain cycles
    take from the start (which a limit below 300 shows)."""
    from chm_amd import pbsm3d as pb

    print("[case] gmres rejected cycle", flush=True)
    mesh = meshgen.synthetic_mesh(106000, seed=5)
    g = pb.face_geometry(mesh)
    fo = meshgen.forcing_c2(mesh.n_faces, seed=9)
    iters = {}
    for limit in (200, 1000):
        ctx = pb.Context(g, pb.default_config(nLayer=10, snow_diffusion_const=-0.028, max_iters=limit))
        o, st = ctx.step(fo, want_fields=True)
        assert _residual(ctx, o["conc"]) <= 1.01e-8
        iters[limit] = st["susp_iters"]
        ctx.close()
    assert iters[1000] == 300 + iters[200], iters


@pytest.mark.parametrize("points,smooth,krylov", [
    (18, -820.0, abi.KRYLOV_GMRES), (18, -820.0, abi.KRYLOV_BICGSTAB_SPLIT), (18, -1.0e4, abi.KRYLOV_GMRES),
    (18, -1.0e4, abi.KRYLOV_BICGSTAB), (18, -1.0e4, abi.KRYLOV_BICGSTAB_SPLIT), (60, -300.0, abi.KRYLOV_GMRES),
    (60, -820.0, abi.KRYLOV_BICGSTAB_SPLIT), (60, -2.0e3, abi.KRYLOV_BICGSTAB_SPLIT)])
def test_indefinite_deposition_system(points, smooth, krylov):
    """A negative smoothing coefficient that leaves an indefinite system, on which conjugate gradients
    break down: the configuration's own method solves it, in the first step and in the next one (which
    does not try them again), to the solution of the dense system."""
    from chm_amd import pbsm3d as pb

    print(f"[case] indefinite deposition points={points} smooth={smooth} krylov={krylov}", flush=True)
    mesh = meshgen.synthetic_mesh(points, seed=8, extent=1.0e3)
    g = pb.face_geometry(mesh)
    fo = meshgen.forcing_c2(mesh.n_faces, seed=4)
    iters = set()
    ctx = pb.Context(g, pb.default_config(nLayer=5, tol=1e-12, smooth_coeff=smooth, krylov=krylov, max_iters=600))
    for _ in range(2):
        ctx.set_state(np.zeros(mesh.n_faces), np.zeros(mesh.n_faces))
        o, st = ctx.step(fo, want_fields=True)
        rp, col, val, b = ctx.system(1)
        A = np.zeros((b.size, b.size))
        A[np.repeat(np.arange(b.size), np.diff(rp)), col] = val
        assert np.linalg.eigvalsh(A).min() < 0 < np.linalg.eigvalsh(A).max()
        want = np.linalg.solve(A, b)
        # relative residual 1e-12: the error is at most cond(A) times that
        assert st["dep_resid"] <= 1e-12
        assert np.linalg.norm(o["qdep"] - want) <= 1e-12 * np.linalg.cond(A) * np.linalg.norm(want)
        iters.add(st["dep_iters"])
    ctx.close()
    assert len(iters) == 1, iters


def test_deposition_limit_that_the_configured_method_meets(oracle):
    """max_iters bounds the deposition solve by the configuration's own method: a limit that GMRES(30), or
    split BiCGStab (which a batch runs), meets and conjugate gradients do not is met, and no more
    iterations than it are reported."""
    from chm_amd import pbsm3d as pb

    print("[case] deposition limit", flush=True)
    mesh = meshgen.synthetic_mesh(2500, seed=8)
    g = pb.face_geometry(mesh)
    fo = meshgen.forcing_c2(mesh.n_faces, seed=4)
    kw = dict(nLayer=5, settling_scale=30.0, smooth_coeff=1.0e5)  # few suspension, many deposition iterations
    orc = oracle.Oracle(g, oracle.oracle_config(precond=abi.PC_MCILU0, dep_precond=abi.PC_MCILU0, **kw))
    _, ost = orc.step(fo)
    batch = pb.Batch([g], [pb.default_config(krylov=abi.KRYLOV_BICGSTAB_SPLIT, **kw)])
    _, bst = batch.step([fo])
    batch.close()
    for krylov, limit in ((abi.KRYLOV_GMRES, ost["dep_iters"] + 1), (abi.KRYLOV_BICGSTAB_SPLIT, bst[0]["dep_iters"] + 1)):
        free = pb.Context(g, pb.default_config(krylov=krylov, **kw))
        fout, fst = free.step(fo, want_fields=True)
        assert fst["dep_iters"] > limit  # conjugate gradients need more
        ctx = pb.Context(g, pb.default_config(krylov=krylov, max_iters=limit, **kw))
        o, st = ctx.step(fo, want_fields=True)
        assert st["dep_iters"] <= limit and st["dep_resid"] <= 1e-8, st
        assert rel_err(o["qdep"], fout["qdep"]) < 1e-6
        ctx.close()
        free.close()


def test_sweep_mode_of_the_split_cycles():
    """pbsm3d_precond_select(0, ..) fixes the workgroup mapping of the split sweeps that FP64 GMRES runs,
    pbsm3d_precond_tuning(0) reports the tuner's choice of it and the times of both; the fields are
    the same bit for bit, and the split BiCGStab's other modes stay refused."""
    from chm_amd import pbsm3d as pb

    print("[case] gmres sweep mode", flush=True)
    mesh = meshgen.synthetic_mesh(6000, seed=5)
    g = pb.face_geometry(mesh)
    fo = meshgen.forcing_c2(mesh.n_faces, seed=9)
    ctx = pb.Context(g, pb.default_config(nLayer=9))
    outs = []
    for mode in (None, 0, 1, -1):
        if mode is not None:
            ctx.precond_select(0, mode)
        ctx.set_state(np.zeros(mesh.n_faces), np.zeros(mesh.n_faces))
        o, st = ctx.step(fo, want_fields=True)
        outs.append((st["susp_iters"], o))
        tun = ctx.precond_tuning(0)
        assert tun["mode"] == mode if mode in (0, 1) else tun["mode"] in (0, 1), (mode, tun)
        assert all(ms > 0 for ms in tun["ms"][:2]) and all(ms == 0 for ms in tun["ms"][2:]), tun
    for it, o in outs[1:]:
        assert it == outs[0][0]
        for k in ("conc", "qdep"):
            np.testing.assert_array_equal(o[k], outs[0][1][k])
    for mode in (2, 3):
        with pytest.raises(pb.Pbsm3dError):
            ctx.precond_select(0, mode)
    ctx.close()


def test_error_left_at_the_production_size():
    """999,968 faces x 10 layers at the production tolerance, the forcing of eighteen draws that leaves most of
    its error in slow modes: the error against a solve to 1e-12 is no larger than the largest that
    plain GMRES(30) cycles left over those draws (8.2e-7 in the concentration's 2-norm)."""
    import torch

    from chm_amd import pbsm3d as pb

    print("[case] gmres error at the production size", flush=True)
    mesh = meshgen.synthetic_mesh(500000, seed=0)
    g = pb.face_geometry(mesh)
    F = mesh.n_faces
    fo = {k: torch.as_tensor(v, dtype=torch.float64, device="cuda:0") for k, v in
          meshgen.forcing_c2(F, seed=6).items()}
    conc = []
    for kw in (dict(tol=1e-12, krylov=abi.KRYLOV_BICGSTAB_SPLIT, max_iters=4000), {}):
        ctx = pb.Context(g, pb.default_config(nLayer=10, **kw))
        o = {"conc": torch.zeros(10 * F, dtype=torch.float64, device="cuda:0")}
        ctx.step(fo, outs=o, on_device=True)
        conc.append(o["conc"])
        ctx.close()
    err = float((conc[1] - conc[0]).norm() / conc[0].norm())
    print(f"[gmres] error {err:.2e}", flush=True)
    assert err <= 8.2e-7, err
