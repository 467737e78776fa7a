"""The structured-grid SpMV (LDS-window line sweep, option spmv_grid_enable) against the
row-parallel kernel: the same products in the same order, so results are bit-identical;
and full solves with the grid path on against the oracle (the dot partials are summed in
another order, so the solver bar applies)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture
def grid_on(gpu):
    gpu.set_option("spmv_grid_enable", 1)
    yield gpu
    gpu.set_option("spmv_grid_enable", 2)  # the default: by row length


def _mats(X):
    row, col, val = X.cube(13, 11, 9)
    yield "cube13x11x9", row, col, val
    r, c, v, _ = X.q1fem27(10, 9, 7)
    yield "q1fem27_10x9x7", r, c, v
    r, c, v, _ = X.varcoef7(17, 6, 5, sigma=1.0)
    yield "varcoef7_17x6x5", r, c, v


@pytest.mark.parametrize("prec", [0, 1])
def test_grid_spmv_bit_identical(grid_on, prec):
    X = grid_on
    for name, row, col, val in _mats(X):
        n = len(row) - 1
        A = X.Matrix(row, col, val, prec=prec)
        assert A.grid() is not None, name
        dt = np.float64 if prec == 0 else np.float32
        for nv in (1, 2, 4, 8, 16, 32, 64):
            print(f"case {name} prec {prec} nv {nv}", flush=True)
            x = X.DeviceArray.from_host(np.random.default_rng(nv).standard_normal(n * nv).astype(dt))
            out = []
            for ge in (0, 1):
                X.set_option("spmv_grid_enable", ge)
                y = X.DeviceArray(n * nv, dt)
                A.spmv(nv, x, y)
                y2 = X.DeviceArray.from_host(np.linspace(-1, 1, n * nv).astype(dt))
                A.spmv(nv, x, y2, accumulate=True)
                out.append((y.to_host(), y2.to_host()))
            X.set_option("spmv_grid_enable", 1)
            assert np.array_equal(out[0][0], out[1][0]), (name, nv)
            assert np.array_equal(out[0][1], out[1][1]), (name, nv)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("dims", [(10, 9, 7), (33, 5, 4)])
def test_grid_codes_bit_identical(gpu, prec, dims):
    # the row-parallel kernel on 1-byte neighbour codes against its column indices: products
    # of a random x, and a V-cycle with Chebyshev smoothing (from zero and non-zero x)
    X = gpu
    row, col, val = X.q1fem27(*dims)[:3]
    n = len(row) - 1
    A = X.Matrix(row, col, val, prec=prec)
    assert A.grid() == dims
    dt = np.float64 if prec == 0 else np.float32
    levels = X.Amg(row, col, val, coarse_size=40).export()
    prm = X.default_params(smoother="Chebyshev", poly_order=4, mg_prec=2 * prec)
    try:
        X.set_option("spmv_codes_min_bytes", 0)  # at this size for every RHS count
        for nv in (1, 2, 4, 8, 16, 32, 64):
            x = X.DeviceArray.from_host(np.random.default_rng(nv).standard_normal(n * nv).astype(dt))
            S = X.Solver(X.Hier(levels), prm, nv)
            db = X.DeviceArray.from_host(X.rhs_uniform(nv, n, nv))
            out = []
            for ge in (0, 2):
                X.set_option("spmv_grid_enable", ge)
                y, dx = X.DeviceArray(n * nv, dt), X.DeviceArray(n * nv)
                y2 = X.DeviceArray.from_host(np.linspace(-1, 1, n * nv).astype(dt))
                A.spmv(nv, x, y)
                A.spmv(nv, x, y2, accumulate=True)
                S.precond_apply(db, dx)
                out.append((y.to_host(), y2.to_host(), dx.to_host()))
            for a, b in zip(*out):
                assert np.array_equal(a, b), nv
    finally:
        X.set_option("spmv_grid_enable", 2)
        X.set_option("spmv_codes_min_bytes", 200000000)


@pytest.mark.parametrize("mg_prec,nv,reached,want", [
    (0, 1, False, True), (0, 4, False, True), (0, 8, False, False), (0, 8, True, True),
    (0, 64, False, False), (0, 64, True, True), (2, 2, True, False), (2, 4, False, True),
    (2, 8, True, False), (2, 16, False, False), (2, 16, True, True)])
def test_codes_by_rhs_and_bytes(gpu, mg_prec, nv, reached, want):
    # which launches of a 27-point operator read neighbour codes: a smoother's residual by
    # precision, RHS count and the bytes of matrix, x and y on both sides of the line; a
    # launch with dots (fp64) up to 8 RHS
    X = gpu
    row, col, val = X.q1fem27(20, 20, 20)[:3]
    n, prec = len(row) - 1, int(mg_prec == 2)
    sv, si = (4 if prec else 8), X.Matrix(row, col, val, prec=prec).info()["index_bits"] // 8
    nbytes = len(col) * (sv + si) + 2 * n * nv * sv
    levels = X.Amg(row, col, val, coarse_size=300).export()
    prm = X.default_params(method="MergedPBiCGStab", smoother="Jacobi", sweeps=2, mg_prec=mg_prec)
    S = X.Solver(X.Hier(levels), prm, nv)
    db, dx = X.DeviceArray.from_host(X.rhs_uniform(1, n, nv)), X.DeviceArray(n * nv)
    dx.zero()
    try:
        X.set_option("spmv_codes_min_bytes", nbytes + (0 if reached else 1))
        X.set_option("spmv_wave_enable", 0)
        names = {(k["kernel"], k["level"]) for k in S.profile(db, dx, 1)}
    finally:
        X.set_option("spmv_codes_min_bytes", 200000000)
        X.set_option("spmv_wave_enable", 2)
    t = "float" if prec else "double"
    assert ((f"k_spmv<{t},grid,{nv},OP_RESID>", 0) in names) == want, names
    assert any(k == f"k_spmv<double,grid,{nv},OP_DOT1>" for k, _ in names) == (nv <= 8), names


def test_grid_path_by_row_length(gpu):
    # the default reads neighbour codes for the 27-point operator (27 entries per interior
    # row; at this size its launches with dots) and columns for the 7-point cube: the
    # launches of a solve show it, none of them a line sweep
    X = gpu
    X.set_option("spmv_grid_enable", 2)
    nv = 8
    for name, (row, col, val), want in (("q1fem27", X.q1fem27(12, 12, 12)[:3], True),
                                        ("cube", X.cube(12), False)):
        levels = X.Amg(row, col, val).export()
        prm = X.default_params(method="MergedPBiCGStab", smoother="Chebyshev", poly_order=2)
        S = X.Solver(X.Hier(levels), prm, nv)
        n = len(row) - 1
        db = X.DeviceArray.from_host(X.rhs_uniform(3, n, nv))
        dx = X.DeviceArray(n * nv)
        names = {k["kernel"] for k in S.profile(db, dx, 1)}
        assert any(k.startswith("k_spmv<double,grid,") for k in names) == want, (name, names)
        assert not any(k.startswith("k_spmv_sweep<") for k in names), (name, names)


@pytest.mark.parametrize("dims,nv,want", [
    ((64, 40, 44), 32, True),    # 110 tiles of 16 lines x 16 segments: 1760 of 2048
    ((64, 40, 36), 32, False),   # 1440 work items
    ((64, 60, 36), 32, False),   # 2160: two for some workgroups
    ((64, 60, 60), 16, True),    # 120 tiles of 32 lines x 16
    ((64, 40, 44), 16, False),
    ((64, 40, 44), 8, False),
    ((64, 40, 44), 64, False),
])
def test_sweep_by_filled_workgroups(gpu, dims, nv, want):
    # in the default mode the SpMMs with dots run the line sweep where its work items fill the
    # chip (here with segments of 4 rows, so that small grids can); the solution does not
    # depend on it beyond the order of the dot partials
    X = gpu
    row, col, val = X.q1fem27(*dims)[:3]
    n = len(row) - 1
    H = X.Hier(X.Amg(row, col, val, max_levels=1).export())
    S = X.Solver(H, X.default_params(method="PBiCGStab", precond="Chebyshev", poly_order=8,
                                     max_iters=400, rel_tol=1e-10), nv)
    b = X.rhs_uniform(5, n, nv)
    db, dx = X.DeviceArray.from_host(b), X.DeviceArray(n * nv)
    try:
        X.set_option("spmv_grid_min_seg", 4)
        dx.zero()
        names = {k["kernel"] for k in S.profile(db, dx, 2)}
        x = S.solve(b)
        X.set_option("spmv_grid_enable", 0)
        x0 = S.solve(b)
    finally:
        X.set_option("spmv_grid_enable", 2)
        X.set_option("spmv_grid_min_seg", 32)
    for op in ("OP_DOT1", "OP_DOT3", "OP_RESID0"):
        assert (f"k_spmv_sweep<double,{nv},{op}>" in names) == want, names
    assert (np.abs(x - x0).reshape(n, nv).max(0) / np.abs(x0).reshape(n, nv).max(0)).max() <= 1e-6


@pytest.mark.parametrize("mg_prec,nv,dims,want", [
    (0, 32, (64, 48, 40), True),   # 1920 of 2048 workgroups
    (0, 32, (64, 40, 44), False),  # 1760
    (0, 32, (64, 44, 48), False),  # 2112: two for some
    (2, 64, (64, 40, 44), True), (2, 64, (64, 40, 36), False),
    (0, 64, (64, 48, 40), False), (0, 16, (64, 48, 40), False), (2, 32, (64, 48, 40), False)])
def test_sweep_residuals_by_filled_workgroups(gpu, mg_prec, nv, dims, want):
    # residuals of a V-cycle in the default mode (segments of 4 rows, as above): the sweep for
    # 16 lanes per row where its work items fill the chip, with the bits of the row kernel
    X = gpu
    row, col, val = X.q1fem27(*dims)[:3]
    n = len(row) - 1
    levels = X.Amg(row, col, val, agg_num_levels=2, num_paths=2, coarse_size=500).export()
    prm = X.default_params(method="MergedPBiCGStab", smoother="Jacobi", sweeps=2, mg_prec=mg_prec)
    S = X.Solver(X.Hier(levels), prm, nv)
    db, dx = X.DeviceArray.from_host(X.rhs_uniform(5, n, nv)), X.DeviceArray(n * nv)
    out = []
    try:
        X.set_option("spmv_grid_min_seg", 4)
        dx.zero()
        names = {k["kernel"] for k in S.profile(db, dx, 1) if k["level"] == 0}
        for ge in (2, 0):
            X.set_option("spmv_grid_enable", ge)
            S.precond_apply(db, dx)
            out.append(dx.to_host())
    finally:
        X.set_option("spmv_grid_enable", 2)
        X.set_option("spmv_grid_min_seg", 32)
    t = "float" if mg_prec else "double"
    assert (f"k_spmv_sweep<{t},{nv},OP_RESID>" in names) == want, names
    assert np.array_equal(*out)


def test_no_grid_view_for_partial_grids(gpu):
    X = gpu
    row, col, val = X.cube(8, 6, 5)
    n = len(row) - 1
    r2, c2, v2 = [0], [], []
    for i in range(n):
        cs, vs = list(col[row[i]:row[i + 1]]), list(val[row[i]:row[i + 1]])
        if i % 7 == 0:
            cs.append((i + n // 2) % n)
            vs.append(0.25)
        c2 += cs
        v2 += vs
        r2.append(len(c2))
    A = X.Matrix(np.array(r2, np.uint32), np.array(c2, np.uint32), np.array(v2))
    assert A.grid() is None
    assert X.Matrix(row, col, val).grid() == (8, 6, 5)


@pytest.mark.parametrize("method,smoother,nv", [("MergedPBiCGStab", "Chebyshev", 32),
                                                ("PBiCGStab", "HSGS", 8),
                                                ("RBiCGStab", "Jacobi", 4),
                                                ("PCG", "Chebyshev", 16)])
def test_solver_with_grid_path_matches_oracle(grid_on, O, method, smoother, nv):
    X = grid_on
    N = 20
    row, col, val = X.cube(N)
    levels = X.Amg(row, col, val).export()
    prm = X.default_params(method=method, smoother=smoother, poly_order=3,
                           sweeps=1 if smoother != "Jacobi" else 2)
    b = X.rhs_uniform(1, N ** 3, nv)
    S = X.Solver(X.Hier(levels), prm, nv)
    x = S.solve(b)
    it, conv, _, _ = S.stats()
    ref = O.solve(O.Hier(levels), O.params_from(prm), nv, b)
    assert conv.all() and ref["conv"].all() and abs(it - ref["iters"]) <= 1
    a, r = x.reshape(-1, nv), ref["x"].reshape(-1, nv)
    assert (np.abs(a - r).max(0) / np.abs(r).max(0)).max() <= 1e-6
