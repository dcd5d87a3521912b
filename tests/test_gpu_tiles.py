"""Tiled sweeps against the CPU oracle's PCG at the sizes where the tiling can
go wrong: fewer rows than a wavefront, chunks of exactly 64 rows and one more
or less, one tile and many, tiles of a single chunk, rows without entries on
one side, two- and three-dimensional patterns, both precisions. The merged
sweeps (ASTG_TILES=0) are the reference for the octree and uniform forms.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def box(shape, rng, diagonals=False):
    """SPD matrix of a box (x fastest): 7-point, or 27-point with diagonals."""
    nz, ny, nx = shape
    idx = np.arange(nz * ny * nx).reshape(shape)
    off = [(0, 0, 1), (0, 1, 0), (1, 0, 0)]
    if diagonals:
        off += [(0, 1, 1), (0, 1, -1), (1, 0, 1), (1, 0, -1), (1, 1, 0), (1, -1, 0)]
    n = idx.size
    rows, cols, vals = [np.arange(n)], [np.arange(n)], [np.zeros(n)]
    diag = np.full(n, 0.05)
    for d in off:
        a = idx[tuple(slice(max(0, -v), s - max(0, v)) for v, s in zip(d, shape))].ravel()
        b = idx[tuple(slice(max(0, v), s - max(0, -v)) for v, s in zip(d, shape))].ravel()
        w = rng.uniform(0.2, 1.0, a.size)
        rows += [a, b]
        cols += [b, a]
        vals += [-w, -w]
        np.add.at(diag, a, w)
        np.add.at(diag, b, w)
    r, c, v = np.concatenate(rows), np.concatenate(cols), np.concatenate(vals)
    v[:n] = diag
    o = np.lexsort((c, r))
    rs = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]).astype(np.int32)
    return rs, c[o].astype(np.int32), v[o]


CASES = [
    ((1, 1, 1), 1), ((1, 1, 63), 1), ((1, 1, 64), 1), ((1, 1, 65), 2), ((1, 5, 13), 3), ((3, 5, 7), 4),
    ((4, 4, 4), 64), ((8, 8, 8), 1), ((8, 8, 8), 8), ((9, 11, 13), 5), ((16, 16, 16), 31), ((5, 40, 41), 64),
    ((21, 22, 23), 7), ((1, 120, 121), 16), ((40, 41, 42), 256),
]


@pytest.mark.parametrize("diagonals", [False, True], ids=["7pt", "19pt"])
@pytest.mark.parametrize("shape,tiles", CASES)
def test_csr_matches_oracle(shape, tiles, diagonals, monkeypatch):
    import astg
    from oracle import oracle as orc
    rng = np.random.default_rng(shape[0] * 7 + tiles)
    rs, col, val = box(shape, rng, diagonals)
    n = len(rs) - 1
    b = rng.standard_normal(n)
    tol = 1e-12
    monkeypatch.setenv("ASTG_TILES", str(tiles))
    c = astg.Context(0)
    x, r = c.pcg_solve_csr(rs, col, val, b, astg.default_params(tol=tol, max_iterations=3000))
    xm, rm = c.pcg_solve_csr(rs, col, val, b, astg.default_params(tol=tol, max_iterations=3000,
                                                                  precision=astg.PREC_MIXED))
    c.close()
    want, _, iters, ok = orc.pcg(rs, col, val, b, tol=tol)
    assert ok
    # The diagonal exceeds the row's off-diagonal sum by 0.05, so the smallest
    # eigenvalue is at least 0.05, and ||x - x'||inf <= ||r||inf / 0.05 for a
    # diagonally dominant matrix: 2 tol ||b|| / 0.05 for two solves.
    bound = 2 * tol * np.abs(b).max() / 0.05
    assert r.converged == 1 and abs(r.iterations - iters) <= 1
    assert np.abs(x - want).max() <= bound
    assert rm.converged == 1 and np.abs(xm - want).max() <= bound


@pytest.mark.parametrize("precision,ordering", [("fp64", 1), ("fp64", 2), ("mixed", 1), ("mixed", 2)])
@pytest.mark.parametrize("tiles,used", [(1, 1), (5, 4), (27, 27), (200, 180)])
def test_octree_matches_merged_sweeps(tiles, used, precision, ordering, monkeypatch, capfd):
    """The same preconditioner through tiles and through merged sweeps: the
    iterates agree up to rounding, so the iteration counts do. Boxes near cubes:
    4 of 5 and 180 of 200 asked for."""
    import astg
    from astg import scenes
    monkeypatch.setenv("ASTG_TIMING", "1")
    out = []
    for t in (0, tiles):
        monkeypatch.setenv("ASTG_TILES", str(t))
        ctx, info = scenes.smoke_64(device=0)
        scenes.fill_velocity(ctx, info["levels"], 3)
        prm = astg.default_params(tol=1e-10, max_iterations=3000, ordering=ordering,
                                  precision=astg.PREC_MIXED if precision == "mixed" else astg.PREC_FP64)
        res = ctx.project(info["dt"], info["rho"], prm)
        out.append((res.iterations, ctx.system(res.n, res.nnz)[4]))
        ctx.close()
    err = capfd.readouterr().err
    assert err.count("tiles: n") == 1 and " K %d (" % used in err
    (i0, p0), (i1, p1) = out
    assert abs(i0 - i1) <= (1 if precision == "fp64" else 4)
    # both residuals are 1e-10 of b; the systems' condition is below 1e4 here
    assert np.linalg.norm(p1 - p0) <= 2e-6 * np.linalg.norm(p0)


@pytest.mark.parametrize("res", [(34, 21), (19, 18, 17)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_uniform_matches_merged_sweeps(res, precision, monkeypatch):
    import astg
    from astg import uniform
    rng = np.random.default_rng(5)
    d = len(res)
    open_ = (rng.random(int(np.prod([r + 1 for r in res]))) < 0.3).astype(np.uint8)
    mac = [rng.standard_normal(int(np.prod([r + (i == a) for i, r in enumerate(res)]))) for a in range(d)]
    tilt = rng.standard_normal((open_.size, 4 if d == 2 else 8))
    out = []
    for t in (0, 1, 7):
        monkeypatch.setenv("ASTG_TILES", str(t))
        s = uniform.ASTSolver(d, res, 1.0 / res[0])
        s.set_layout(open_)
        s.set_velocity(mac, tilt)
        prm = uniform.default_params(precision=astg.PREC_MIXED if precision == "mixed" else astg.PREC_FP64,
                                     tol=1e-9)
        r = s.project(0.025, 2.0, prm)
        out.append((r.iterations, np.concatenate([u.ravel() for u in s.velocity()[0]])))
    for it, u in out[1:]:
        assert abs(it - out[0][0]) <= (1 if precision == "fp64" else 4)
        assert np.abs(u - out[0][1]).max() <= 1e-7 * np.abs(u).max()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("tiles", [1, 3, 16])
def test_batch_matches_merged_sweeps(tiles, precision, monkeypatch):
    """Stacked systems through tiles that cut them anywhere, and a system of a
    single row among them."""
    import astg
    rng = np.random.default_rng(11)
    systems = []
    for shape in ((1, 1, 1), (9, 8, 7), (1, 20, 31), (16, 17, 18), (3, 3, 3)):
        rs, col, val = box(shape, rng)
        systems.append((rs, col, val, rng.standard_normal(len(rs) - 1)))
    prm = astg.default_params(tol=1e-11, max_iterations=3000,
                              precision=astg.PREC_MIXED if precision == "mixed" else astg.PREC_FP64)
    out = []
    for t in (0, tiles):
        monkeypatch.setenv("ASTG_TILES", str(t))
        c = astg.Context(0)
        out.append(c.pcg_solve_batch(systems, prm))
        c.close()
    (x0, r0), (x1, r1) = out
    for s, a, b, p, q in zip(systems, x0, x1, r0, r1):
        assert p.converged and q.converged and abs(p.iterations - q.iterations) <= 2
        # both within tol ||b|| / 0.05 of the solution (test_csr_matches_oracle)
        assert np.abs(a - b).max() <= 2 * 1e-11 * np.abs(s[3]).max() / 0.05


def test_fp64_solve_on_tiles_that_hold_fp32_only(monkeypatch):
    """A block-colour pattern whose tiles fit the LDS in FP32 only: its first
    FP64 solve rebuilds it with merged sweeps and gives what those give, and
    the mixed form works before and after."""
    import astg
    from astg import scenes
    fp64 = astg.default_params(tol=1e-10, max_iterations=3000, ordering=astg.ORDER_BLOCK_COLOUR)
    mixed = astg.default_params(tol=1e-10, max_iterations=3000, precision=astg.PREC_MIXED)
    out = []
    for tiled in (False, True):
        monkeypatch.setenv("ASTG_TILES", "0")
        ctx, info = scenes.smoke_64(device=0, R=96)
        scenes.fill_velocity(ctx, info["levels"], 3)
        if tiled:
            n = ctx.numbering(0)[2]
            # 20 k to 40 k rows a tile: above 160 KB in FP64, below in FP32
            monkeypatch.setenv("ASTG_TILES", str(max(1, round(n / 28000))))
        ctx.snapshot(False)
        m0 = ctx.project(info["dt"], info["rho"], mixed)
        ctx.snapshot(True)
        r = ctx.project(info["dt"], info["rho"], fp64)
        p = ctx.system(r.n, r.nnz)[4]
        ctx.snapshot(True)
        m1 = ctx.project(info["dt"], info["rho"], mixed)
        pm = ctx.system(r.n, r.nnz)[4]
        assert m0.converged and r.converged and m1.converged
        assert np.linalg.norm(pm - p) <= 2e-6 * np.linalg.norm(p)
        out.append((r.n, r.iterations, p))
        ctx.close()
    (n, i0, p0), (_, i1, p1) = out
    print("n %d" % n)
    assert i0 == i1 and np.array_equal(p0, p1)


@pytest.mark.parametrize("tiles", ["256", "0"], ids=["tiled", "merged"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_stopping_launch_ends_in_every_block(precision, tiles, monkeypatch, capfd):
    """The launch that finds the solve finished stores that while its other
    blocks start: each of them leaves as a whole or takes the decision itself.
    Solves that end on many different launches, by convergence, by the
    iteration limit and on a zero right-hand side: no block waits for one that
    left (which would be reported and retried), and every repetition gives the
    same solution."""
    import astg
    rng = np.random.default_rng(2)
    rs, col, val = box((24, 25, 26), rng)
    b = rng.standard_normal(len(rs) - 1)
    prec = astg.PREC_MIXED if precision == "mixed" else astg.PREC_FP64
    monkeypatch.setenv("ASTG_TILES", tiles)
    c = astg.Context(0)
    first = {}
    for rep in range(6):
        for tol, limit in [(10.0 ** -k, 3000) for k in range(1, 9)] + [(1e-9, k) for k in range(1, 9)]:
            x, r = c.pcg_solve_csr(rs, col, val, b, astg.default_params(tol=tol, max_iterations=limit, precision=prec),
                                   allow_unconverged=True)
            key = tol, limit
            if key not in first:
                first[key] = x, r.iterations
            assert r.iterations == first[key][1] and np.array_equal(x, first[key][0])
        x, r = c.pcg_solve_csr(rs, col, val, 0 * b, astg.default_params(precision=prec))
        assert r.iterations == 0 and not x.any()
    c.close()
    assert "retrying" not in capfd.readouterr().err


@pytest.mark.parametrize("tiles", [2, 5, 16])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_finished_systems_of_a_batch_take_no_part(precision, tiles, monkeypatch):
    """The deepest system of the batch, a chain of 20000 rows whose factor is
    exact, finishes first: the iterations after that do not run its chain. One
    sweep over it takes at least 2 x 20000 dependent steps of over 0.1 us, so
    the solve stays below half of iterations x 4 ms only without it. The
    others' solutions are those they have without it in the batch."""
    import astg
    rng = np.random.default_rng(4)
    others = []
    for shape in ((20, 20, 20), (9, 8, 7), (1, 20, 31)):
        rs, col, val = box(shape, rng)
        others.append((rs, col, val, rng.standard_normal(len(rs) - 1)))
    rs, col, val = box((1, 1, 20000), rng)
    deep = (rs, col, val, rng.standard_normal(20000))
    tol = 1e-11
    prm = astg.default_params(tol=tol, max_iterations=3000,
                              precision=astg.PREC_MIXED if precision == "mixed" else astg.PREC_FP64)
    monkeypatch.setenv("ASTG_TILES", str(tiles))
    c = astg.Context(0)
    alone, ra = c.pcg_solve_batch(others, prm)
    c.pcg_solve_batch([deep] + others, prm)  # plans and first launches
    x, r = c.pcg_solve_batch([deep] + others, prm)
    c.close()
    most = max(q.iterations for q in r)
    print("iterations %s, %.2f ms" % ([q.iterations for q in r], r[0].ms_solve))
    assert r[0].iterations < most / 4
    assert r[0].ms_solve < 0.5 * 4.0 * most
    for s, u, v, p, q in zip(others, alone, x[1:], ra, r[1:]):
        assert p.converged and q.converged and abs(p.iterations - q.iterations) <= 2
        # both within tol ||b|| / 0.05 of the solution (test_csr_matches_oracle)
        assert np.abs(u - v).max() <= 2 * tol * np.abs(s[3]).max() / 0.05
    d = deep[2] * x[0][col]
    assert np.abs(np.add.reduceat(d, rs[:-1]) - deep[3]).max() <= 2 * tol * np.abs(deep[3]).max()


def ordered(rs, col, val, key):
    """The matrix with its rows sorted by key."""
    n = len(rs) - 1
    new = np.empty(n, np.int64)
    new[np.argsort(key, kind="stable")] = np.arange(n)
    r, c = new[np.repeat(np.arange(n), np.diff(rs))], new[col]
    o = np.lexsort((c, r))
    return np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]).astype(np.int32), c[o].astype(np.int32), val[o]


def colours(shape, blocks):
    """0: none; 1: two colours; b: blocks of b cells in 8 colours."""
    Z, Y, X = [a.ravel() for a in np.meshgrid(*[np.arange(s) for s in shape], indexing="ij")]
    if blocks < 2:
        return blocks * (X + Y + Z) % 2
    x, y, z = X // blocks, Y // blocks, Z // blocks
    return ((x & 1) + 2 * (y & 1) + 4 * (z & 1)) * 10 ** 6 + x + 100 * (y + 100 * z)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("shape,count,blocks,tiled", [
    ((20, 20, 20), 1, 1, False), ((20, 20, 20), 1, 4, True), ((28, 28, 28), 1, 4, False), ((28, 28, 28), 1, 8, True),
    ((28, 28, 28), 1, 0, True), ((20, 20, 20), 24, 1, False), ((30, 30, 30), 2, 4, False), ((30, 30, 30), 2, 0, True),
])
def test_orders_of_few_wide_levels_sweep_merged(shape, count, blocks, tiled, precision, monkeypatch):
    """Index-range tiles are for long dependency chains; a colouring keeps the
    merged sweeps. Which form a solve took shows in its solution's last bits."""
    import astg
    rng = np.random.default_rng(6)
    systems = []
    for _ in range(count):
        rs, col, val = ordered(*box(shape, rng), colours(shape, blocks))
        systems.append((rs, col, val, rng.standard_normal(len(rs) - 1)))
    prm = astg.default_params(tol=1e-9, max_iterations=3000,
                              precision=astg.PREC_MIXED if precision == "mixed" else astg.PREC_FP64)

    def solve():
        c = astg.Context(0)
        x = c.pcg_solve_batch(systems, prm)[0] if count > 1 else [c.pcg_solve_csr(*systems[0], prm)[0]]
        c.close()
        return np.concatenate(x)

    x = solve()
    monkeypatch.setenv("ASTG_TILES", "0")
    merged = solve()
    assert np.array_equal(x, merged) == (not tiled)
    assert np.abs(x - merged).max() <= 2 * 1e-9 * max(np.abs(s[3]).max() for s in systems) / 0.05


@pytest.mark.parametrize("tiles,done", [(1, False), (2, True)])
def test_no_tiles_are_set_up_for_rows_that_do_not_fit(tiles, done, monkeypatch, capfd):
    """24000 rows in one tile exceed the LDS by their values alone: the set-up
    (sorts, counts) is not begun. In two tiles they fit."""
    import astg
    rng = np.random.default_rng(8)
    rs, col, val = box((20, 30, 40), rng)
    b = rng.standard_normal(len(rs) - 1)
    monkeypatch.setenv("ASTG_TILES", str(tiles))
    monkeypatch.setenv("ASTG_TIMING", "1")
    c = astg.Context(0)
    x, r = c.pcg_solve_csr(rs, col, val, b, astg.default_params(tol=1e-8, max_iterations=3000))
    c.close()
    assert r.converged == 1
    assert ("tiles: n 24000 " in capfd.readouterr().err) == done


@pytest.fixture
def narrow(monkeypatch):
    """A projection in block colours whose tiles hold 20 k to 40 k rows: more
    than 160 KB in FP64, less in FP32."""
    from astg import scenes
    ctx, info = scenes.smoke_64(device=0, R=96)
    scenes.fill_velocity(ctx, info["levels"], 3)
    monkeypatch.setenv("ASTG_TILES", str(max(1, round(ctx.numbering(0)[2] / 28000))))
    ctx.snapshot(False)

    def project(precision, tol=1e-10):
        import astg
        prm = astg.default_params(tol=tol, max_iterations=3000, ordering=astg.ORDER_BLOCK_COLOUR,
                                  precision=astg.PREC_MIXED if precision == "mixed" else astg.PREC_FP64)
        ctx.snapshot(True)
        r = ctx.project(info["dt"], info["rho"], prm)
        return r, ctx.system(r.n, r.nnz)[4]

    yield ctx, project
    ctx.close()


def test_each_precision_keeps_its_sweeps(narrow, monkeypatch, capfd):
    """Mixed and FP64 solves in turn on one pattern: the mixed one stays in
    tiles, the FP64 one merged, whatever came before, and neither is set up a
    second time. Which form a solve took shows in its solution's last bits."""
    monkeypatch.setenv("ASTG_TIMING", "1")
    ctx, project = narrow
    m0, f0 = project("mixed"), project("fp64")
    capfd.readouterr()
    m1, f1, f2, m2 = project("mixed"), project("fp64"), project("fp64"), project("mixed")
    assert "timing] sweeps/" not in capfd.readouterr().err
    for a, b in ((m0, m1), (m0, m2), (f0, f1), (f0, f2)):
        assert a[0].iterations == b[0].iterations and np.array_equal(a[1], b[1])


def test_fp64_projections_set_no_fp32_tiles_up(narrow, monkeypatch, capfd):
    monkeypatch.setenv("ASTG_TIMING", "1")
    ctx, project = narrow
    capfd.readouterr()
    f0 = project("fp64")
    err = capfd.readouterr().err
    assert "tiles: n" not in err and err.count("timing] sweeps/merged order") == 1
    project("mixed")
    assert "tiles: n" in capfd.readouterr().err
    assert np.array_equal(project("fp64")[1], f0[1])


@pytest.mark.parametrize("which", ["FWD64", "BWD64"])
def test_fp64_sweeps_can_be_timed_after_a_mixed_solve(narrow, which):
    import astg
    ctx, project = narrow
    m0 = project("mixed")
    ms, by = ctx.kernel_time(getattr(astg, "K_" + which), 2)
    assert ms > 0 and by > 0
    t, lev = ctx.sweep_timeline(getattr(astg, "K_" + which), m0[0].n)
    assert (t[:, 2] > 0).all() and lev.min() == 0
    assert np.array_equal(project("mixed")[1], m0[1])


def test_a_mixed_projection_sets_one_systems_sweeps_up(monkeypatch, capfd):
    """The block-colour copy's: the reference numbering is not swept."""
    import astg
    from astg import scenes
    monkeypatch.setenv("ASTG_TIMING", "1")
    ctx, info = scenes.smoke_64(device=0)
    scenes.fill_velocity(ctx, info["levels"], 3)
    ctx.project(info["dt"], info["rho"], astg.default_params(tol=1e-6, precision=astg.PREC_MIXED))
    ctx.close()
    assert capfd.readouterr().err.count("timing] sweeps/permuted pattern") == 1


@pytest.mark.parametrize("tiles,patterns", [(3, 2), (0, 4)])
def test_tuner_times_what_differs(tiles, patterns, monkeypatch, capfd):
    """In tiles the levels per group are nothing to choose: one pattern is
    timed (and the chosen one set up), and another value of it takes no new
    pattern. Merged sweeps are timed with each value."""
    import astg
    rng = np.random.default_rng(12)
    systems = []
    for shape in ((9, 8, 7), (16, 17, 18)):
        rs, col, val = box(shape, rng)
        systems.append((rs, col, val, rng.standard_normal(len(rs) - 1)))
    monkeypatch.setenv("ASTG_TILES", str(tiles))
    monkeypatch.setenv("ASTG_TIMING", "1")
    prm = astg.default_params(tol=1e-8, max_iterations=3000)
    c = astg.Context(0)
    best = c.tune_batch(systems, prm, iterations=3)
    assert capfd.readouterr().err.count("timing] setPattern/factorisation plan") == patterns
    assert best.merge_levels == 2 or not tiles
    x, r = c.pcg_solve_batch(systems, prm)
    c.set_batch_tuning(5, best.stream_blocks_per_cu, best.lanes_per_row)
    y, q = c.pcg_solve_batch(systems, prm)
    assert capfd.readouterr().err.count("timing] setPattern/factorisation plan") == (0 if tiles else 1)
    c.close()
    for u, v in zip(x, y):
        assert np.array_equal(u, v) if tiles else np.abs(u - v).max() <= 1e-6 * np.abs(u).max()


def test_reported_times_hold_no_set_up():
    """The times in a solve's result are those of its work, also where the sweeps
    had to be set up first (sorts, device allocations: several times as long as
    the two iterations here)."""
    import astg
    rng = np.random.default_rng(13)
    rs, col, val = box((48, 48, 48), rng)
    b = rng.standard_normal(len(rs) - 1)
    prm = astg.default_params(tol=1e-12, max_iterations=2)
    for _ in range(2):  # the first context loads the kernels
        c = astg.Context(0)
        csr = [c.pcg_solve_csr(rs, col, val, b, prm, allow_unconverged=True)[1].ms_solve for _ in range(4)]
        batch = [c.pcg_solve_batch([(rs, col, val, b)] * 2, prm, allow_unconverged=True)[1][0].ms_solve
                 for _ in range(4)]
        c.close()
    print(csr, batch)
    for t in (csr, batch):
        assert t[0] <= 2 * max(t[1:])
