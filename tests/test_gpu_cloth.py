"""GPU parity of the cloth terms (Baraff-Witkin membrane, discrete-shell
bending; femEnergy.cu:2215-2300, 2431-2630) against the oracle: element
assembly, energies, Newton iterations and a drape trajectory over a fixed
box."""
import numpy as np
import pytest

from helpers import rel

pytestmark = pytest.mark.gpu


def _scene(**kw):
    from sgipc import scene as S
    import sgipc
    sc = S.cloth_scene(n=10, size=0.2, **kw)
    sc.mas_precision = sgipc.SGIPC_MAS_FP64
    return sc


def _dense(nv, rowptr, cols, vals):
    A = np.zeros((3 * nv, 3 * nv))
    for i in range(nv):
        for k in range(rowptr[i], rowptr[i + 1]):
            A[3 * i:3 * i + 3, 3 * cols[k]:3 * cols[k] + 3] += vals[k]
    return A


@pytest.mark.parametrize("amp", [3e-3, 2e-2])
def test_cloth_assembly_and_energy(oracle, amp):
    """deformed sheet (stretched, compressed, sheared and bent triangles;
    projected bending Hessians): gradient and Hessian within 1e-10 relative,
    the cloth energy within 1e-12"""
    import sgipc
    sc = _scene(height=0.13)
    sc.kappa = 1e5
    rng = np.random.default_rng(7)
    x = sc.x.copy()
    cloth = np.zeros(sc.n_verts, bool)
    cloth[np.unique(sc.tris)] = True
    x[cloth] += amp * rng.normal(size=(cloth.sum(), 3))
    sim = sgipc.Simulation(sc)
    sim.set_positions(x)
    w = oracle.World(sc)
    w.set_positions(x)
    g, rp, cl, vl = sim.assemble()
    go, Ao = w.assemble()
    Ag = _dense(sc.n_verts, rp, cl, vl)
    print(f"[cloth-assemble] amp={amp} nnzb gpu={cl.size} oracle={Ao.nnzb} "
          f"g={rel(g, go):.2e} H={rel(Ag, Ao.dense()):.2e}", flush=True)
    assert rel(g, go) < 1e-10
    assert rel(Ag, Ao.dense()) < 1e-10
    e, eo = sim.energy(), w.energy()
    print(f"[cloth-energy] gpu={e[6]:.12e} oracle={eo[6]:.12e}", flush=True)
    assert eo[6] > 0
    assert e[6] == pytest.approx(eo[6], rel=1e-12)
    assert rel(e[:7], eo[:7]) < 1e-12


def test_cloth_newton_iterations_match(oracle):
    """sheet within contact range of the box: per Newton iteration equal PCG
    iteration counts; step sizes and positions identical to rounding before
    contact.  Once the CCD bound limits the step, additive CCD's stopping
    test on directions that differ by PCG rounding moves alpha by a few 1e-6
    relative and the mid-step iterate by up to ~1e-7 (the two sides sum
    element and contact terms in different orders, so their bank matrices
    differ in the last bits, and the cloth's ill-conditioned banks amplify
    that in the inverses), so mid-step iterates are held to 1e-5 in alpha and
    1e-6 in positions"""
    import sgipc
    sc = _scene(height=0.1022)
    sim = sgipc.Simulation(sc)
    w = oracle.World(sc)
    sim.kappa = 1e4
    w.kappa = 1e4
    for it in range(4):
        st = sim.newton_iteration()
        so = w.newton_iteration()
        xg, xo = sim.positions(), w.positions()
        err = np.abs(xg - xo).max() / np.abs(xo).max()
        print(f"[cloth-newton] it={it} pcg={st['pcg_iterations']}/{so['pcg_iterations']} "
              f"alpha={st['alpha']:.6g}/{so['alpha']:.6g} err={err:.2e}", flush=True)
        assert st["converged"] == so["converged"]
        if st["converged"]:
            break
        assert st["pcg_iterations"] == so["pcg_iterations"]
        assert st["alpha"] == pytest.approx(so["alpha"], rel=1e-5)
        assert err < 1e-6


def _bumped_sheet(height):
    """sheet with a flat rest shape, started with a two-bump out-of-plane
    displacement (bent and slightly stretched), over the ground only"""
    sc = _scene(height=height, n_boxes=0)
    sc.x_rest = sc.x.copy()
    u = (sc.x[:, 0] + 0.1) / 0.2
    v = (sc.x[:, 2] + 0.1) / 0.2
    sc.x = sc.x.copy()
    sc.x[:, 1] += 0.004 * np.sin(2 * np.pi * u) * np.sin(np.pi * v)
    return sc


# Cloth steps need many Newton iterations (the projected membrane and bending
# Hessians make Newton converge linearly) of 50-150 PCG iterations each.  When
# a PCG residual lands near the stopping threshold at a check, rounding
# differences (summation order on the GPU, where run-to-run results also
# differ) change the iteration count by one check period, and the step
# then differs by up to the Newton stopping tolerance (1e-2 dt = 1e-4 m).
# Trajectories are therefore held to that scale once the paths split.
_NEWTON_SCALE = 1e-3


def test_cloth_ground_trajectory(oracle):
    """bent sheet relaxing (membrane and bending forces) while it falls onto
    the ground: 10 time steps within the Newton-tolerance scale of the oracle,
    no vertex below the ground"""
    import sgipc
    sc = _bumped_sheet(0.006)
    sim = sgipc.Simulation(sc)
    w = oracle.World(sc)
    touched = False
    for step in range(10):
        sg = sim.time_step()
        so = w.time_step()
        xg, xo = sim.positions(), w.positions()
        err = np.abs(xg - xo).max() / np.abs(xo).max()
        touched |= xg[:, 1].min() < 1e-3
        print(f"[cloth-ground] step={step} newton={sg['newton_iterations']}/"
              f"{so['newton_iterations']} pcg={sg['pcg_iterations']}/{so['pcg_iterations']} "
              f"err={err:.2e} ymin={xg[:, 1].min():.6f} bend={sim.energy()[6]:.4e}", flush=True)
        assert err < _NEWTON_SCALE
        assert xg[:, 1].min() > 0.0
    assert touched


def test_cloth_drape_over_box(oracle):
    """sheet dropped onto a fixed box.  Free fall and first contact (Newton
    paths identical) agree to 1e-8 as one trajectory.  The drape over the box
    corners takes ~25 Newton iterations per step, and GPU runs (atomic
    summation order) can take another Newton path that ends elsewhere within
    the Newton tolerance; over several steps those differences compound like
    any chaotic contact trajectory.  From the third step on, the oracle is
    therefore started from the GPU's state each step and the single step is
    held to the Newton-tolerance scale, plus the contact invariant: no cloth
    vertex inside the box"""
    import sgipc
    sc = _scene(height=0.105)
    sim = sgipc.Simulation(sc)
    w = oracle.World(sc)
    cloth = np.unique(sc.tris)
    box = np.setdiff1d(np.arange(sc.n_verts), cloth)
    lo, hi = sc.x[box].min(0), sc.x[box].max(0)
    for step in range(5):
        if step >= 2:
            w.set_state(sim.positions(), sim.velocities(), sim.xtilde(), sim.kappa)
        sg = sim.time_step()
        so = w.time_step()
        xg, xo = sim.positions(), w.positions()
        err = np.abs(xg - xo).max() / np.abs(xo).max()
        print(f"[cloth-drape] step={step} newton={sg['newton_iterations']}/"
              f"{so['newton_iterations']} pcg={sg['pcg_iterations']}/{so['pcg_iterations']} "
              f"err={err:.2e} ymin={xg[cloth, 1].min():.5f}", flush=True)
        assert err < (1e-8 if step < 2 else 5 * _NEWTON_SCALE)
        inside = np.all((xg[cloth] > lo) & (xg[cloth] < hi), axis=1)
        assert not inside.any()


def _cloth_over_abd(prec):
    """reduced cloth-over-affine-boxes configuration: a 12 x 12 sheet (0.24 m,
    membrane E 1e6, bending 1e-4, thickness 1e-3) dropped onto three free
    affine boxes (kappa 1e11) on the ground; PCG stops on the FP64 true
    residual 1e-6 and Newton on |dx|_inf < 1e-8, so each step's end point is
    the incremental potential's minimiser to well below 1e-6"""
    import sgipc
    from sgipc import scene as S
    sc = S.cloth_scene(n=12, size=0.24, height=0.075, n_boxes=3, box_size=0.06, box_cells=2,
                       abd_boxes=True, abd_kappa=1e11, seed=1)
    sc.mas_precision = sgipc.SGIPC_MAS_FP64
    sc.solver_precision = prec
    sc.pcg_rel_tol = 1e-6
    sc.pcg_use_preconditioned_norm = 0
    sc.abs_xdelta_tol = 1e-8
    return sc


def test_cloth_over_affine_boxes_mixed_tracks_fp64(oracle):
    """sheet over three affine boxes, 6 time steps (free fall, first contact,
    draping over the box edges with up to ~170 Newton iterations per step):
    the FP64 GPU solve against the oracle, and the mixed-precision solve (FP32
    inner PCG with FP64 residual refinement) against the FP64 GPU solve, both
    within 1e-8 of the scene scale per step (the Newton stop |dx|_inf < 1e-8
    bounds how far either end point is from the step's minimiser); the boxes
    stay rigid and the sheet lands on them"""
    import sgipc
    sims = {}
    for prec in (sgipc.SGIPC_SOLVE_FP64, sgipc.SGIPC_SOLVE_MIXED):
        sims[prec] = sgipc.Simulation(_cloth_over_abd(prec))
    sc = _cloth_over_abd(sgipc.SGIPC_SOLVE_FP64)
    w = oracle.World(sc)
    abd = sc.abd_body
    cloth = np.unique(sc.tris)
    x0 = sc.x.copy()
    box_top = x0[abd >= 0, 1].max()
    fell = False
    for step in range(6):
        s64 = sims[sgipc.SGIPC_SOLVE_FP64].time_step()
        s32 = sims[sgipc.SGIPC_SOLVE_MIXED].time_step()
        so = w.time_step()
        x64 = sims[sgipc.SGIPC_SOLVE_FP64].positions()
        x32 = sims[sgipc.SGIPC_SOLVE_MIXED].positions()
        xo = w.positions()
        scale = np.abs(xo).max()
        e_or = np.abs(x64 - xo).max() / scale
        e_mx = np.abs(x32 - x64).max() / scale
        print(f"[cloth-abd] step={step} newton={s64['newton_iterations']}/"
              f"{s32['newton_iterations']}/{so['newton_iterations']} "
              f"pcg={s64['pcg_iterations']}/{s32['pcg_iterations']}/{so['pcg_iterations']} "
              f"err_oracle={e_or:.2e} err_mixed={e_mx:.2e} "
              f"ymin={x64[cloth, 1].min():.5f}", flush=True)
        assert s64["capped"] == 0 and s32["capped"] == 0
        assert e_or < 1e-8
        assert e_mx < 1e-8
        fell |= x64[cloth, 1].min() < box_top
    assert fell
    for x in (x64, x32):
        for b in range(int(abd.max()) + 1):
            d0 = np.linalg.norm(x0[abd == b][:, None] - x0[abd == b][None], axis=2)
            d = np.linalg.norm(x[abd == b][:, None] - x[abd == b][None], axis=2)
            assert np.abs(d - d0).max() < 1e-6


@pytest.mark.parametrize("n,one", [(20, 1), (40, 0)])
def test_newton_iteration_with_long_contact_rows(oracle, n, one):
    """A sheet lying flat on the top face of a fixed box: the box's few
    vertices carry the contact blocks of the whole sheet, more than a
    workgroup of the one-launch solve takes in one round; with too many
    rounds a launch per operation is faster and taken.  One Newton
    iteration against the oracle (the scale of the iterates above)."""
    import sgipc
    from sgipc import scene as S
    sc = S.cloth_scene(n=n, size=0.095, height=0.1013, n_boxes=1)
    sc.mas_precision = sgipc.SGIPC_MAS_FP64
    sim = sgipc.Simulation(sc)
    w = oracle.World(sc)
    sim.kappa = 1e4
    w.kappa = 1e4
    _, rowptr, cols, _ = sim.assemble()
    box = np.setdiff1d(np.arange(sc.n_verts), sc.tris)
    far = sum(int(np.isin(cols[rowptr[v]:rowptr[v + 1]], box, invert=True).sum()) for v in box)
    sim.profile(1)
    st = sim.newton_iteration()
    launches = {k: sim.profile_query(k)[0] for k in ("pcg", "spmv")}
    so = w.newton_iteration()
    err = np.abs(sim.positions() - w.positions()).max() / np.abs(w.positions()).max()
    print(f"[cloth-rows] n={n} {launches} box contact blocks={far} coo={sim.sizes()['coo_blocks']} "
          f"pcg={st['pcg_iterations']}/{so['pcg_iterations']} err={err:.2e}", flush=True)
    assert far > 512 and launches["pcg"] == one and (launches["spmv"] == 0) == (one == 1)
    assert abs(st["pcg_iterations"] - so["pcg_iterations"]) <= 10
    assert err < 1e-6


@pytest.mark.parametrize("name", ["sheet", "stack", "affine"])
def test_contact_solve_ways_agree(name):
    """From one state in contact, a Newton iteration whose solve runs as one
    launch and as a launch per operation: three PCG iterations with FP64
    inverses end at the same positions up to rounding (contact blocks are summed
    by atomics, in an order that varies too)."""
    import sgipc
    from sgipc import scene as S
    sc = {"sheet": lambda: S.cloth_scene(n=20, size=0.095, height=0.1013, n_boxes=1),
          "stack": lambda: S.stack_scene(n=3, cells=4, friction_mu=0.2),
          "affine": lambda: S.abd_scene(n_abd=3, cells=3)}[name]()
    sc.mas_precision = sgipc.SGIPC_MAS_FP64
    sim = sgipc.Simulation(sc)
    sim.kappa = 1e4
    sim.set_pcg(rel_tol=0.0, max_iter=4)
    state = (sim.positions(), sim.velocities(), sim.xtilde(), sim.kappa)
    x = {}
    for polls in (-1, 0):
        sim.one_launch(polls)
        sim.set_state(*state)
        sim.profile(1)
        st = sim.newton_iteration()
        assert sim.profile_query("pcg")[0] == (1 if polls else 0)
        x[polls] = sim.positions() - state[0]
    err = np.abs(x[-1] - x[0]).max() / np.abs(x[0]).max()
    print(f"[ways-contact] {name} coo={sim.sizes()['coo_blocks']} pairs={st['n_pairs']} "
          f"ground={st['n_ground']} step={np.abs(x[0]).max():.2e} diff={err:.2e}", flush=True)
    assert st["n_pairs"] > 0 and np.abs(x[0]).max() > 0.0
    # positions of about 0.1 round at 1e-17, steps are larger than 1e-6
    assert err < 1e-10
