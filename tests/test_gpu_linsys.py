"""GPU parity of the linear-system path (BSR SpMV, MAS, PCG) against the
oracle on assembled Stiff-GIPC systems."""
import numpy as np
import pytest

from helpers import assembled_system, rel

pytestmark = pytest.mark.gpu


def _scenes():
    from sgipc import scene as S
    return {
        "bar": S.bar_scene(),
        "cubes8": S.cubes_scene(n_side=2, cells=4, size=0.2, spacing=0.35, seed=3),
    }


@pytest.fixture(scope="module")
def systems(oracle):
    out = {}
    for name, sc in _scenes().items():
        w, g, A = assembled_system(sc, perturb=0.004, seed=1)
        out[name] = (sc, g, A)
    return out


@pytest.mark.parametrize("name", ["bar", "cubes8"])
def test_spmv_matches_oracle(systems, name):
    import sgipc
    sc, g, A = systems[name]
    ls = sgipc.LinearSystem(A.rowptr, A.cols, A.vals, sc.part_id, sgipc.SGIPC_PRECOND_DIAG)
    rng = np.random.default_rng(7)
    x = rng.normal(size=3 * A.nb)
    y = ls.spmv(x)
    print(f"[spmv] {name} nb={A.nb} nnzb={A.nnzb}", flush=True)
    assert rel(y, A.spmv(x)) < 1e-13


@pytest.mark.parametrize("name", ["bar", "cubes8"])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_mas_hierarchy_and_apply(systems, oracle, name, prec):
    import sgipc
    sc, g, A = systems[name]
    fp32 = prec == "fp32"
    ls = sgipc.LinearSystem(A.rowptr, A.cols, A.vals, sc.part_id, sgipc.SGIPC_PRECOND_MAS,
                            sgipc.SGIPC_MAS_FP32 if fp32 else sgipc.SGIPC_MAS_FP64)
    m = oracle.Mas(A, sc.part_id, fp32=fp32)
    L, sizes, tc = ls.mas_info()
    print(f"[mas] {name} {prec} levels={L} sizes={sizes.tolist()} total={tc}", flush=True)
    assert L == m.levels
    assert tc == m.total_clusters()
    np.testing.assert_array_equal(sizes, m.level_sizes())
    np.testing.assert_array_equal(ls.mas_chain(), m.chain())
    rng = np.random.default_rng(11)
    r = rng.normal(size=3 * A.nb)
    z = ls.precond(r)
    zo = m.apply(r)
    assert rel(z, zo) < (2e-5 if fp32 else 1e-10)


@pytest.mark.parametrize("name", ["bar", "cubes8"])
@pytest.mark.parametrize("pc", ["mas", "diag"])
def test_pcg_matches_oracle(systems, oracle, name, pc):
    import sgipc
    sc, g, A = systems[name]
    pcid = sgipc.SGIPC_PRECOND_MAS if pc == "mas" else sgipc.SGIPC_PRECOND_DIAG
    ls = sgipc.LinearSystem(A.rowptr, A.cols, A.vals, sc.part_id, pcid, sgipc.SGIPC_MAS_FP64)
    x, st = ls.pcg(g, rel_tol=1e-4)
    m = oracle.Mas(A, sc.part_id, fp32=False) if pc == "mas" else None
    xo, ito, rz0, rz = oracle.pcg(A, g, m, 1 if pc == "mas" else 0, rel_tol=1e-4)
    print(f"[pcg] {name} {pc} it={st.iterations} oracle_it={ito} relres={st.rel_residual:.3e}",
          flush=True)
    assert st.iterations == ito
    assert rel(x, xo) < 1e-8
    D = A.dense()
    assert np.linalg.norm(D @ x - g) / np.linalg.norm(g) == pytest.approx(st.rel_residual, rel=1e-6)


@pytest.fixture(scope="module")
def deep(oracle):
    from helpers import deep_hierarchy_system
    return deep_hierarchy_system()


@pytest.fixture(scope="module")
def deep_wide(oracle):
    from helpers import deep_hierarchy_system
    return deep_hierarchy_system(nblob=8192)


def _first_tail_level(sizes, item):
    """the first level from which on R, its members, and 256 vertices' nodes and
    products on every level fit 64 KB"""
    L = sizes.shape[0] - 1
    for l in range(1, L):
        span = (sizes[L - 1].sum() - sizes[l, 1] + 15) // 16 * 16
        if 3 * (span + 256 * (L - l)) * item + 4 * (256 * (L - l) + span) <= 64 * 1024:
            return l
    return L


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_mas_deep_hierarchy(deep, deep_wide, oracle, prec):
    """Two large coarse levels (own launches) then a tail that every workgroup
    of the last launch restricts in its LDS: hierarchy equal, apply equal to the
    oracle."""
    import sgipc
    fp32 = prec == "fp32"
    A, part, b = deep_wide if fp32 else deep
    ls = sgipc.LinearSystem(A.rowptr, A.cols, A.vals, part, sgipc.SGIPC_PRECOND_MAS,
                            sgipc.SGIPC_MAS_FP32 if fp32 else sgipc.SGIPC_MAS_FP64)
    m = oracle.Mas(A, part, fp32=fp32)
    L, sizes, tc = ls.mas_info()
    print(f"[mas-deep] {prec} levels={L} sizes={sizes.tolist()}", flush=True)
    np.testing.assert_array_equal(sizes, m.level_sizes())
    assert _first_tail_level(sizes, 4 if fp32 else 8) == 3 < L
    r = np.random.default_rng(5).normal(size=3 * A.nb)
    assert rel(ls.precond(r), m.apply(r)) < (2e-5 if fp32 else 1e-10)


def test_pcg_deep_hierarchy(deep, oracle):
    import sgipc
    A, part, b = deep
    ls = sgipc.LinearSystem(A.rowptr, A.cols, A.vals, part, sgipc.SGIPC_PRECOND_MAS,
                            sgipc.SGIPC_MAS_FP64)
    x, st = ls.pcg(b, rel_tol=1e-6)
    m = oracle.Mas(A, part, fp32=False)
    xo, ito, _, _ = oracle.pcg(A, b, m, 1, rel_tol=1e-6)
    print(f"[pcg-deep] it={st.iterations} oracle_it={ito} relres={st.rel_residual:.3e}",
          flush=True)
    assert st.iterations == ito
    assert rel(x, xo) < 1e-8
    ls = sgipc.LinearSystem(A.rowptr, A.cols, A.vals, part, sgipc.SGIPC_PRECOND_MAS,
                            sgipc.SGIPC_MAS_FP32)
    _same_first_iterates(oracle, ls, A, part, b)


@pytest.mark.parametrize("name", ["bar", "cubes8"])
@pytest.mark.parametrize("pc", ["mas", "diag"])
def test_mixed_precision_refinement(systems, oracle, name, pc):
    """FP32 matrix/vectors/MAS PCG with its periodic residual recomputation in
    FP64 (reliable updates) reaches the FP64 true relative residual asked for,
    in about the FP64 solve's iteration count, and its solution agrees with the
    dense FP64 solve (condition number permitting)."""
    import sgipc
    sc, g, A = systems[name]
    pcid = sgipc.SGIPC_PRECOND_MAS if pc == "mas" else sgipc.SGIPC_PRECOND_DIAG
    ls = sgipc.LinearSystem(A.rowptr, A.cols, A.vals, sc.part_id, pcid, sgipc.SGIPC_MAS_FP32)
    x, st = ls.pcg(g, rel_tol=1e-6, use_rz=False, solver_precision=sgipc.SGIPC_SOLVE_MIXED)
    D = A.dense()
    res = np.linalg.norm(D @ x - g) / np.linalg.norm(g)
    x64, st64 = ls.pcg(g, rel_tol=1e-6, use_rz=False)
    print(f"[mixed] {name} {pc} inner_it={st.iterations} outer={st.outer_iterations} "
          f"relres={st.rel_residual:.3e} (dense {res:.3e}); fp64 it={st64.iterations} "
          f"relres={st64.rel_residual:.3e}", flush=True)
    assert st.converged
    assert st.rel_residual <= 1e-6
    assert st.iterations <= 2 * st64.iterations + 20
    assert res == pytest.approx(st.rel_residual, rel=1e-3, abs=1e-12)
    xd = np.linalg.solve(D, g)
    assert rel(x, xd) < 1e-3


def test_mixed_precision_deep_hierarchy(deep, oracle):
    import sgipc
    A, part, b = deep
    ls = sgipc.LinearSystem(A.rowptr, A.cols, A.vals, part, sgipc.SGIPC_PRECOND_MAS,
                            sgipc.SGIPC_MAS_FP32)
    x, st = ls.pcg(b, rel_tol=1e-8, use_rz=False, solver_precision=sgipc.SGIPC_SOLVE_MIXED)
    print(f"[mixed-deep] it={st.iterations} outer={st.outer_iterations} "
          f"relres={st.rel_residual:.3e}", flush=True)
    assert st.converged and st.rel_residual <= 1e-8
    assert rel(A.spmv(x), b) <= 1.01e-8


def test_mixed_precision_stiff_contrast(systems, oracle):
    """A system with a 1e8 stiffness contrast (one cube's rows and columns
    scaled by 1e4, i.e. D A D): the FP32 iteration may stall or diverge; the
    mixed solve must still reach the FP64 true residual asked for (FP64
    continuation from its iterate), within the FP32 plus FP64 iteration
    budget, and agree with the dense solve"""
    import sgipc
    sc, g, A = systems["cubes8"]
    nb = A.nb
    scale = np.where(sc.body_id == 0, 1e4, 1.0)
    rows = np.repeat(np.arange(nb), np.diff(A.rowptr))
    vals = A.vals.reshape(-1, 3, 3) * (scale[rows] * scale[A.cols])[:, None, None]
    ls = sgipc.LinearSystem(A.rowptr, A.cols, vals.reshape(A.vals.shape), sc.part_id,
                            sgipc.SGIPC_PRECOND_MAS, sgipc.SGIPC_MAS_FP32)
    b = g * np.repeat(scale, 3)
    x, st = ls.pcg(b, rel_tol=1e-10, use_rz=False, solver_precision=sgipc.SGIPC_SOLVE_MIXED)
    x64, st64 = ls.pcg(b, rel_tol=1e-10, use_rz=False)
    print(f"[mixed-stiff] it={st.iterations} outer={st.outer_iterations} "
          f"relres={st.rel_residual:.3e}; fp64 it={st64.iterations} "
          f"relres={st64.rel_residual:.3e}", flush=True)
    assert st.rel_residual <= 1e-10
    assert st64.rel_residual <= 1e-10
    assert st.iterations <= 4 * st64.iterations + 400
    assert rel(x, x64) < 1e-5


@pytest.mark.parametrize("name", ["bar", "cubes8"])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_mas_bank_inverse_bit_exact(systems, oracle, name, prec):
    """Every bank inverse of every level equals the oracle's unpivoted
    Gauss-Jordan (the reference's operation order) of the GPU's own bank
    matrix bit for bit (FP64), or its FP32 rounding; the bank matrices equal
    the oracle's Galerkin banks to 1e-12."""
    import sgipc
    sc, g, A = systems[name]
    fp32 = prec == "fp32"
    ls = sgipc.LinearSystem(A.rowptr, A.cols, A.vals, sc.part_id, sgipc.SGIPC_PRECOND_MAS,
                            sgipc.SGIPC_MAS_FP32 if fp32 else sgipc.SGIPC_MAS_FP64)
    L, sizes, tc = ls.mas_info()
    nbank = tc // 16
    print(f"[bank inverse] {name} {prec} banks={nbank}", flush=True)
    checked = 0
    for b in range(nbank):
        m, inv = ls.mas_bank(b)
        M = m.copy()
        d = np.arange(48)
        zero = M[d, d] == 0.0
        M[d[zero], d[zero]] = 1.0
        Mi = oracle.inverse_gj(M)
        up = np.triu(Mi)
        sym = up + np.triu(Mi, 1).T
        expect = sym.astype(np.float32).astype(np.float64) if fp32 else sym
        assert np.array_equal(inv.view(np.uint64), expect.view(np.uint64)), f"bank {b}"
        checked += 1
    assert checked == nbank > 0


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("kind", ["chain", "diagonal"])
@pytest.mark.parametrize("nb", [1, 17, 255, 257, 1000])
def test_mas_apply_workgroup_edges(oracle, nb, kind, prec):
    """Systems that end inside, at and after a 256-vertex workgroup of the
    apply's last launch.  A chain has one tail node per bank; without
    couplings every vertex is its own node on every level, so a workgroup
    multiplies more rows than it has threads."""
    import sgipc
    rng = np.random.default_rng(nb)
    n = np.arange(nb)
    S = rng.normal(size=(nb, 3, 3))
    vals = 4.0 * np.eye(3) + 0.3 * (S + S.transpose(0, 2, 1))
    rows, cols = n, n
    if kind == "chain" and nb > 1:
        off = 0.4 * rng.normal(size=(nb - 1, 3, 3))
        vals = np.concatenate([vals + 2.0 * np.eye(3), off])
        rows, cols = np.concatenate([n, n[:-1]]), np.concatenate([n, n[1:]])
    A = oracle.bsr_from_upper_triplets(nb, rows, cols, vals.reshape(-1, 9))
    part = (n // 16).astype(np.int32)
    fp32 = prec == "fp32"
    ls = sgipc.LinearSystem(A.rowptr, A.cols, A.vals, part, sgipc.SGIPC_PRECOND_MAS,
                            sgipc.SGIPC_MAS_FP32 if fp32 else sgipc.SGIPC_MAS_FP64)
    m = oracle.Mas(A, part, fp32=fp32)
    np.testing.assert_array_equal(ls.mas_info()[1], m.level_sizes())
    r = rng.normal(size=3 * nb)
    # FP32: inverses and sums of 48 products per level round at 6e-8 each
    assert rel(ls.precond(r), m.apply(r)) < (2e-5 if fp32 else 1e-10)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("nb", [2000, 3000, 5000, 20000])
def test_mas_nothing_clusters(oracle, nb, prec):
    """Blocks without couplings: every level has as many nodes as there are
    vertices, the most that the hierarchy's arrays have to hold.  The apply is
    the inverse block once per level."""
    import sgipc
    rng = np.random.default_rng(nb)
    S = rng.normal(size=(nb, 3, 3))
    D = 2.0 * np.eye(3) + 0.1 * S @ S.transpose(0, 2, 1)
    fp32 = prec == "fp32"
    part = (np.arange(nb) // 16).astype(np.int32)
    ls = sgipc.LinearSystem(np.arange(nb + 1), np.arange(nb), D, part, sgipc.SGIPC_PRECOND_MAS,
                            sgipc.SGIPC_MAS_FP32 if fp32 else sgipc.SGIPC_MAS_FP64)
    L, sizes, total = ls.mas_info()
    print(f"[mas-uncoupled] nb={nb} {prec} levels={L} sizes={sizes.tolist()}", flush=True)
    pad = (nb + 15) // 16 * 16
    assert sizes[1:, 0].tolist() == [nb] * L and total == L * pad
    np.testing.assert_array_equal(ls.mas_chain().reshape(nb, L - 1),
                                  np.arange(nb)[:, None] + pad * np.arange(1, L))
    r = rng.normal(size=3 * nb)
    x = np.linalg.solve(D, r.reshape(-1, 3, 1)).ravel()
    # the blocks' condition is a few; L terms rounded at the inverses' precision
    bound = 1e-6 if fp32 else 1e-14
    assert rel(ls.precond(r), L * x) < bound
    # so the first iteration of a solve (max_iter is one more) ends at the solution
    assert rel(ls.pcg(r, rel_tol=0.0, max_iter=2)[0], x) < bound


def _spd_system(oracle, nb, seed, reach=40):
    """A diagonally dominant block system with couplings to the next rows and
    to random far ones (rows of 3 to about 20 blocks), 16-row parts."""
    rng = np.random.default_rng(seed)
    i = np.arange(nb)
    pairs = [np.stack([i[:-d], i[d:]], 1) for d in (1, 3, 17, reach) if nb > d]
    if nb > 4:
        far = np.sort(rng.integers(0, nb, size=(2 * nb, 2)), axis=1)
        pairs.append(far[far[:, 0] != far[:, 1]])
    e = np.unique(np.concatenate(pairs), axis=0) if pairs else np.zeros((0, 2), np.int64)
    off = 0.1 * rng.normal(size=(e.shape[0], 3, 3))
    load = np.zeros(nb)
    np.add.at(load, e.ravel(), np.abs(off).sum(axis=2).max(axis=1).repeat(2))
    S = 0.1 * rng.normal(size=(nb, 3, 3))
    diag = (1.2 * load + 0.5)[:, None, None] * np.eye(3) + S + S.transpose(0, 2, 1)
    A = oracle.bsr_from_upper_triplets(nb, np.concatenate([i, e[:, 0]]),
                                       np.concatenate([i, e[:, 1]]),
                                       np.concatenate([diag, off]).reshape(-1, 9))
    return A, (i // 16).astype(np.int32), rng.normal(size=3 * nb)


def _same_first_iterates(oracle, ls, A, part, b):
    """The first iterates of a one-launch solve with FP32 inverses against the
    oracle's with FP32 inverses, while the error is still large and the iterate
    depends on every term of the preconditioner."""
    m = oracle.Mas(A, part, fp32=True)
    for cap in (2, 4):
        x, st = ls.pcg(b, rel_tol=0.0, max_iter=cap)
        xo, _, _, _ = oracle.pcg(A, b, m, 1, rel_tol=0.0, max_iter=cap)
        print(f"[first iterates] nb={A.nb} cap={cap} diff={rel(x, xo):.2e} "
              f"relres={st.rel_residual:.2e}", flush=True)
        assert st.one_launch == 1
        # sums of 48 products per level, rounded at 6e-8 each in another order
        assert rel(x, xo) < 1e-6


@pytest.mark.parametrize("pc,prec", [("mas", "fp32"), ("mas", "fp64"), ("diag", "fp64")])
@pytest.mark.parametrize("nb", [40, 63, 129, 700, 8200, 33000])
def test_pcg_one_launch_sizes(oracle, nb, pc, prec):
    """The one-launch solve at one workgroup, at the edges of its row ranges,
    with one and two passes per row range and rows longer than it keeps in
    registers: the solution of the system and the oracle's iterate after a
    fixed number of iterations (max_iter is one more, as in the reference's
    loop), with a stop test between."""
    import sgipc
    A, part, b = _spd_system(oracle, nb, nb)
    ls = sgipc.LinearSystem(A.rowptr, A.cols, A.vals, part,
                            sgipc.SGIPC_PRECOND_MAS if pc == "mas" else sgipc.SGIPC_PRECOND_DIAG,
                            sgipc.SGIPC_MAS_FP32 if prec == "fp32" else sgipc.SGIPC_MAS_FP64)
    for use_rz in (True, False):
        x, st = ls.pcg(b, rel_tol=1e-12, use_rz=use_rz)
        print(f"[one-launch] nb={nb} {pc} {prec} rz={use_rz} it={st.iterations} "
              f"relres={st.rel_residual:.2e}", flush=True)
        assert st.converged and st.iterations % 10 == 0 and st.one_launch == 1
        # the residual norm follows the tested norm up to the conditioning
        # (about 10) of the preconditioned system
        assert np.linalg.norm(A.spmv(x) - b) <= 1e-10 * np.linalg.norm(b)
    if prec == "fp32":
        _same_first_iterates(oracle, ls, A, part, b)
    else:
        m = oracle.Mas(A, part, fp32=False) if pc == "mas" else None
        for cap in (1, 2, 8, 13):
            x, st = ls.pcg(b, rel_tol=0.0, max_iter=cap)
            xo, ito, _, _ = oracle.pcg(A, b, m, 1 if pc == "mas" else 0, rel_tol=0.0,
                                       max_iter=cap)
            assert st.iterations == ito == cap and not st.converged and st.one_launch == 1
            # FP64 sums in another order, amplified by at most cap steps
            assert np.linalg.norm(x - xo) <= 1e-11 * np.linalg.norm(xo)


@pytest.mark.parametrize("nb,low", [(500, 1), (6000, 1), (43000, 3)])
def test_pcg_one_launch_uneven_parts(oracle, nb, low):
    """Parts of low .. 16 rows: workgroups with unequal numbers of banks, whose
    inverses stay in LDS whole, stay there packed, or come in again each
    iteration."""
    import sgipc
    A, _, b = _spd_system(oracle, nb, nb)
    size = np.random.default_rng(1).integers(low, 17, size=nb)
    part = np.repeat(np.arange(nb), size)[:nb].astype(np.int32)
    for prec in (sgipc.SGIPC_MAS_FP64, sgipc.SGIPC_MAS_FP32):
        ls = sgipc.LinearSystem(A.rowptr, A.cols, A.vals, part, sgipc.SGIPC_PRECOND_MAS, prec)
        x, st = ls.pcg(b, rel_tol=1e-12)
        assert st.converged and st.one_launch == 1
        assert np.linalg.norm(A.spmv(x) - b) <= 1e-10 * np.linalg.norm(b)
        if prec == sgipc.SGIPC_MAS_FP32:
            _same_first_iterates(oracle, ls, A, part, b)
        else:
            x, st = ls.pcg(b, rel_tol=0.0, max_iter=13)
            xo, _, _, _ = oracle.pcg(A, b, oracle.Mas(A, part, fp32=False), 1, rel_tol=0.0,
                                     max_iter=13)
            # FP64 sums in another order, amplified by at most 13 steps
            assert np.linalg.norm(x - xo) <= 1e-11 * np.linalg.norm(xo)


@pytest.mark.parametrize("pc", ["mas", "diag"])
def test_pcg_beyond_one_launch(oracle, pc):
    """More rows than the one-launch solve takes (256 per workgroup): a
    launch per operation."""
    import sgipc
    A, part, b = _spd_system(oracle, 65700, 3)
    ls = sgipc.LinearSystem(A.rowptr, A.cols, A.vals, part,
                            sgipc.SGIPC_PRECOND_MAS if pc == "mas" else sgipc.SGIPC_PRECOND_DIAG,
                            sgipc.SGIPC_MAS_FP64)
    x, st = ls.pcg(b, rel_tol=1e-12)
    assert st.converged and st.one_launch == 0
    assert np.linalg.norm(A.spmv(x) - b) <= 1e-10 * np.linalg.norm(b)
    m = oracle.Mas(A, part, fp32=False) if pc == "mas" else None
    x, st = ls.pcg(b, rel_tol=0.0, max_iter=13)
    xo, _, _, _ = oracle.pcg(A, b, m, 1 if pc == "mas" else 0, rel_tol=0.0, max_iter=13)
    assert np.linalg.norm(x - xo) <= 1e-11 * np.linalg.norm(xo)


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("pc,prec", [("mas", "fp32"), ("mas", "fp64"), ("diag", "fp64")])
@pytest.mark.parametrize("nb", [40, 700, 8200])
def test_pcg_ways_agree(oracle, nb, pc, prec, noalloc):
    """A solve as one launch and as a launch per operation, chosen by the
    caller: the stats say which way it ran, the counts are equal, and after
    three iterations, well before convergence hides the preconditioner, the
    iterates differ by rounding."""
    import sgipc
    A, part, b = _spd_system(oracle, nb, nb)
    ls = sgipc.LinearSystem(A.rowptr, A.cols, A.vals, part,
                            sgipc.SGIPC_PRECOND_MAS if pc == "mas" else sgipc.SGIPC_PRECOND_DIAG,
                            sgipc.SGIPC_MAS_FP32 if prec == "fp32" else sgipc.SGIPC_MAS_FP64)
    pcg = ls.pcg_noalloc if noalloc else ls.pcg
    runs = []
    for polls in (-1, 0, -1):
        ls.one_launch(polls)
        x, st = pcg(b, rel_tol=0.0, max_iter=4)
        it = [pcg(b, rel_tol=1e-8, use_rz=rz)[1].iterations for rz in (True, False)]
        runs.append((x, st, it))
    print(f"[ways] nb={nb} {pc} {prec} it={[r[2] for r in runs]} "
          f"diff={rel(runs[0][0], runs[1][0]):.2e}", flush=True)
    assert [r[1].one_launch for r in runs] == [1, 0, 1]
    assert runs[0][2] == runs[1][2] == runs[2][2]
    assert np.array_equal(runs[0][0], runs[2][0])
    # sums in another order: at the precision of the vectors, and with FP32
    # inverses of the preconditioner's products, amplified by three steps
    assert rel(runs[0][0], runs[1][0]) < (1e-6 if prec == "fp32" else 1e-13)
    with pytest.raises(sgipc.SgipcError):
        ls.one_launch(-2)


@pytest.mark.parametrize("noalloc", [False, True])
@pytest.mark.parametrize("pc", ["mas", "diag"])
def test_pcg_wait_runs_out(oracle, pc, noalloc):
    """One poll is too few for over a hundred workgroups to meet: they leave,
    and the solve is done with a launch per operation, the following ones
    without trying; a new bound tries again."""
    import sgipc
    A, part, b = _spd_system(oracle, 8200, 1)
    ls = sgipc.LinearSystem(A.rowptr, A.cols, A.vals, part,
                            sgipc.SGIPC_PRECOND_MAS if pc == "mas" else sgipc.SGIPC_PRECOND_DIAG)
    pcg = ls.pcg_noalloc if noalloc else ls.pcg
    ls.one_launch(0)
    x0, s0 = pcg(b, rel_tol=1e-8)
    ls.one_launch(1)
    for _ in range(2):
        x1, s1 = pcg(b, rel_tol=1e-8)
        assert s1.converged and s1.one_launch == 0 and s1.iterations == s0.iterations
        assert np.array_equal(x0, x1)
    ls.one_launch()
    x2, s2 = pcg(b, rel_tol=1e-8)
    assert s2.one_launch == 1 and s2.iterations == s0.iterations
    # sums in another order, up to where the solves stop
    assert rel(x2, x0) < 1e-9


def test_pcg_threads_one_launch_each(oracle):
    """Solves of eight threads, together more workgroups than the device holds
    at once: every one runs as one launch and ends where it does alone."""
    import threading
    import sgipc
    rows = [300, 700, 2100, 4000, 8200, 8200, 17000, 33000]
    sys_ = []
    for k, nb in enumerate(rows):
        A, part, b = _spd_system(oracle, nb, 10 + k)
        pc = sgipc.SGIPC_PRECOND_DIAG if k == 4 else sgipc.SGIPC_PRECOND_MAS
        ls = sgipc.LinearSystem(A.rowptr, A.cols, A.vals, part, pc)
        sys_.append((ls, b, ls.pcg(b, rel_tol=1e-8)))
    bad = []

    def work(ls, b, alone):
        try:
            for _ in range(12):
                x, st = ls.pcg(b, rel_tol=1e-8)
                if st.one_launch != 1 or not np.array_equal(x, alone[0]):
                    bad.append((ls.nb, st.one_launch, rel(x, alone[0])))
        except Exception as e:  # reported by the main thread
            bad.append(repr(e))
    th = [threading.Thread(target=work, args=s) for s in sys_]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad[:4]


def test_pcg_small_solves_of_threads_overlap(oracle):
    """Four threads with a small system each (a few workgroups) take less than
    the solves would one after the other; best of five."""
    import threading
    import time
    import sgipc
    A, part, b = _spd_system(oracle, 425, 3)
    own = [sgipc.LinearSystem(A.rowptr, A.cols, A.vals, part) for _ in range(4)]

    def run(ls):
        for _ in range(20):
            assert ls.pcg(b, rel_tol=0.0, max_iter=201)[1].one_launch == 1

    def timed(systems):
        th = [threading.Thread(target=run, args=(ls,)) for ls in systems]
        t0 = time.perf_counter()
        for t in th:
            t.start()
        for t in th:
            t.join()
        return time.perf_counter() - t0
    for ls in own:
        run(ls)
    ratio = min(timed(own) / timed(own[:1]) for _ in range(5))
    print(f"[threads] four threads / one = {ratio:.2f}", flush=True)
    assert ratio < 2.5
