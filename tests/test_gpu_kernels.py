"""GPU kernel parity through the C ABI: SpMM and dense matvec bit-exact against the oracle
(same summation order, no FMA contraction on either side)."""
import numpy as np
import pytest
from conftest import random_csr

pytestmark = pytest.mark.gpu

NVS = [1, 2, 4, 8, 16, 32, 64]


@pytest.mark.parametrize("nv", NVS)
@pytest.mark.parametrize("index_mode", [1, 2])
def test_spmv_cube_bit_exact(gpu, O, nv, index_mode):
    X = gpu
    row, col, val = X.cube(24, 20, 18)
    n = len(row) - 1
    rng = np.random.default_rng(nv)
    vals = rng.standard_normal(len(val))
    A = X.Matrix(row, col, vals, prec=0, index_mode=index_mode)
    assert A.info()["index_bits"] == (32 if index_mode == 1 else 16)
    x = rng.standard_normal(n * nv)
    dx, dy = X.DeviceArray.from_host(x), X.DeviceArray(n * nv)
    A.spmv(nv, dx, dy)
    assert np.array_equal(dy.to_host(), O.spmv(row, col, vals, x, nv))
    y0 = rng.standard_normal(n * nv)
    dy.upload(y0)
    A.spmv(nv, dx, dy, accumulate=True)
    assert np.array_equal(dy.to_host(), O.spmv(row, col, vals, x, nv, y=y0))


@pytest.mark.parametrize("nv", NVS)
def test_spmv_fp32_bit_exact(gpu, O, nv):
    # rows up to 40 nonzeros: several chunks and batches for every lane-group width
    X = gpu
    rng = np.random.default_rng(11)
    row, col, val = random_csr(rng, 700, 700, 0.02, max_row=40)
    A = X.Matrix(row, col, val, prec=1, index_mode=1)
    x = rng.standard_normal(700 * nv).astype(np.float32)
    dx, dy = X.DeviceArray.from_host(x), X.DeviceArray(700 * nv, np.float32)
    A.spmv(nv, dx, dy)
    assert np.array_equal(dy.to_host(), O.spmv(row, col, val, x, nv, f32=True))


@pytest.mark.parametrize("nv", NVS)
def test_spmv_irregular_rows_bit_exact(gpu, O, nv):
    # empty rows, long rows (> 16 nonzeros: several cooperative chunks), rectangular
    X = gpu
    rng = np.random.default_rng(nv + 3)
    n, m = 1500, 900
    row, col, val = random_csr(rng, n, m, 0.03, diag=False)
    row = row.copy()
    lens = np.diff(row).astype(np.int64)
    lens[::7] = 0  # empty rows
    keep = np.concatenate([np.arange(row[i], row[i] + lens[i]) for i in range(n)]).astype(np.int64)
    col, val = col[keep], val[keep]
    row = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    assert lens.max() > 16
    A = X.Matrix(row, col, val, prec=0, index_mode=1, ncols=m)
    x = rng.standard_normal(m * nv)
    dx, dy = X.DeviceArray.from_host(x), X.DeviceArray(n * nv)
    A.spmv(nv, dx, dy)
    assert np.array_equal(dy.to_host(), O.spmv(row, col, val, x, nv, ncols=m))


@pytest.mark.parametrize("nv", [8, 32])
@pytest.mark.parametrize("prec", [0, 1])
def test_spmv_wide_batches_bit_exact(gpu, O, nv, prec):
    # few rows of many entries (the coarse levels of an aggressively coarsened hierarchy)
    # take the 16-wide batches (with the long-row kernel off, which is faster on fewer rows):
    # the same sums in the same order as the 8-wide kernel and, in fp64, as the oracle;
    # y = A x and y += A x, u16 and u32 columns, empty rows
    X = gpu
    rng = np.random.default_rng(nv * 7 + prec)
    n = 2000
    row, col, val = random_csr(rng, n, n, 0.04)
    lens = np.diff(row).astype(np.int64)
    lens[::11] = 0
    keep = np.concatenate([np.arange(row[i], row[i] + lens[i]) for i in range(n)]).astype(np.int64)
    col, val = col[keep], val[keep]
    row = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    assert len(col) >= 32 * n
    dt = np.float64 if prec == 0 else np.float32
    x = rng.standard_normal(n * nv)
    y0 = np.linspace(-1, 1, n * nv)
    try:
        X.set_option("spmv_wave_enable", 0)
        for index_mode in (1, 2):
            A = X.Matrix(row, col, val, prec=prec, index_mode=index_mode)
            out = []
            for wide in (0, 1):
                X.set_option("spmv_wide_batches", wide)
                dx = X.DeviceArray.from_host(x.astype(dt))
                dy = X.DeviceArray(n * nv, dt)
                A.spmv(nv, dx, dy)
                dz = X.DeviceArray.from_host(y0.astype(dt))
                A.spmv(nv, dx, dz, accumulate=True)
                out.append((dy.to_host(), dz.to_host()))
            assert np.array_equal(out[0][0], out[1][0]), index_mode
            assert np.array_equal(out[0][1], out[1][1]), index_mode
            if prec == 0:
                assert np.array_equal(out[1][0], O.spmv(row, col, val, x, nv))
    finally:
        X.set_option("spmv_wide_batches", 1)
        X.set_option("spmv_wave_enable", 2)


def test_wide_batches_in_the_coarse_levels(gpu):
    # the coarse levels of the aggressively coarsened 64^3 cube (levels 2 and 3: 2295 and
    # 587 rows of 34 and 45 entries) take the 16-wide SpMVs with the long-row kernel off; the
    # preconditioner is bit-identical with them off
    X = gpu
    row, col, val = X.cube(64)
    levels = X.Amg(row, col, val, agg_num_levels=2, num_paths=2, coarse_size=500).export()
    n = len(row) - 1
    prm = X.default_params(method="MergedPBiCGStab", smoother="Chebyshev", poly_order=4)
    try:
        X.set_option("spmv_wave_enable", 0)
        for nv in (8, 32):
            b = X.rhs_uniform(nv, n, nv)
            out, names = [], []
            for wide in (0, 1):
                X.set_option("spmv_wide_batches", wide)
                S = X.Solver(X.Hier(levels), prm, nv)
                db, dx = X.DeviceArray.from_host(b), X.DeviceArray(n * nv)
                S.precond_apply(db, dx)
                out.append(dx.to_host())
                dx.zero()
                names.append({(k["kernel"], k["level"]) for k in S.profile(db, dx, 1)})
            assert np.array_equal(out[0], out[1]), nv
            wide = [{lv for k, lv in q if k.startswith("k_spmv<") and k.endswith(",16>")}
                    for q in names]
            assert not wide[0]
            assert max(wide[1]) >= 2 and 0 not in wide[1], names[1]
            assert not any(k.startswith("k_spmv_wave<") for q in names for k, _ in q)
    finally:
        X.set_option("spmv_wide_batches", 1)
        X.set_option("spmv_wave_enable", 2)


@pytest.mark.parametrize("nv", [8, 32])
def test_long_row_kernel_in_the_coarse_levels(gpu, nv):
    # by default the same levels take the long-row kernel: at nv = 8 both, at nv = 32 (a cap of
    # 1536 rows) the 587 rows, the 2295 rows the 16-wide SpMVs
    X = gpu
    row, col, val = X.cube(64)
    levels = X.Amg(row, col, val, agg_num_levels=2, num_paths=2, coarse_size=500).export()
    prm = X.default_params(method="MergedPBiCGStab", smoother="Chebyshev", poly_order=4)
    S = X.Solver(X.Hier(levels), prm, nv)
    n = len(row) - 1
    db, dx = X.DeviceArray.from_host(X.rhs_uniform(nv, n, nv)), X.DeviceArray(n * nv)
    dx.zero()
    names = {(k["kernel"], k["level"]) for k in S.profile(db, dx, 1) if "OP_CHEB" in k["kernel"]}
    for lv, wave in ((2, nv == 8), (3, True)):
        if not any(q == lv for _, q in names):
            continue  # the coarsest level is solved directly
        want = "k_spmv_wave<" if wave else "k_spmv<"
        assert all(k.startswith(want) and k.endswith(",16>") for k, q in names if q == lv), names
    assert any(q == 2 for _, q in names)


def test_spmv_order_sensitive_row(gpu):
    # a row whose value depends on the summation order: (2^53 + 1) - 2^53 = 0 in the
    # reference's stored order
    X = gpu
    big = float(2 ** 53)
    row = np.array([0, 3], np.uint32)
    col = np.array([0, 1, 2], np.uint32)
    A = X.Matrix(row, col, np.array([big, 1.0, -big]), index_mode=1, ncols=3)
    dx, dy = X.DeviceArray.from_host(np.ones(3 * 4)), X.DeviceArray(4)
    A.spmv(4, dx, dy)
    assert np.array_equal(dy.to_host(), np.zeros(4))


def test_dense_matvec_bit_exact(gpu, O):
    import ctypes as C

    X = gpu
    rng = np.random.default_rng(5)
    n, nv = 97, 8
    D = rng.standard_normal((n, n))
    x = rng.standard_normal(n * nv)
    dD, dx, dy = X.DeviceArray.from_host(D.ravel()), X.DeviceArray.from_host(x), X.DeviceArray(n * nv)
    X.check(X.hip().xh_dense_matvec(n, nv, 0, dD.ptr, dx.ptr, dy.ptr), "xh_dense_matvec")
    y = np.zeros(n * nv)
    O.lib().xo_dense_matvec_d(n, n, D.ctypes.data_as(C.c_void_p), nv, x.ctypes.data_as(C.c_void_p),
                              y.ctypes.data_as(C.c_void_p))
    assert np.array_equal(dy.to_host(), y)


@pytest.mark.parametrize("n,nv", [(1, 1), (33, 1), (63, 2), (64, 4), (65, 8), (129, 16),
                                  (200, 32), (7, 64), (191, 64),
                                  (1100, 32), (530, 64), (700, 1),
                                  # called on its own: the last sizes without tiles and the
                                  # first with, by nv
                                  (95, 1), (96, 1), (96, 2), (127, 4), (128, 8), (193, 32),
                                  (179, 8), (180, 8), (192, 2), (449, 32), (450, 32), (1099, 64),
                                  (2799, 16), (2800, 16),
                                  # four waves per workgroup
                                  (1100, 64), (1153, 64), (2049, 32), (4097, 16)])
@pytest.mark.parametrize("prec", [0, 1])
def test_dense_matvec_tile_edges_bit_exact(gpu, n, nv, prec):
    # sums in column order with separate multiply and add, at the edges of the row blocks
    # (1 to 32 rows), of the 64-column tiles (one, even and odd tile counts), of the direct
    # and the tiled kernel, and of the two-wave and four-wave variants
    X = gpu
    rng = np.random.default_rng(n + nv)
    dt = np.float64 if prec == 0 else np.float32
    D, x = rng.standard_normal((n, n)).astype(dt), rng.standard_normal((n, nv)).astype(dt)
    y = np.zeros((n, nv), dt)
    for j in range(n):
        y = y + D[:, j:j + 1] * x[j]
    dD, dx, dy = (X.DeviceArray.from_host(a.ravel()) for a in (D, x, np.zeros((n, nv), dt)))
    X.check(X.hip().xh_dense_matvec(n, nv, prec, dD.ptr, dx.ptr, dy.ptr), "xh_dense_matvec")
    assert np.array_equal(dy.to_host(), y.ravel())


@pytest.mark.parametrize("nv", NVS)
@pytest.mark.parametrize("prec", [0, 1])
def test_spmv_long_row_kernel_bit_exact(gpu, O, nv, prec):
    # the kernel that loads a whole row at once, at row lengths around its batches of 8, its
    # passes of 32 and 64 entries and an empty row, u32 and u16 columns, set and add
    X = gpu
    rng = np.random.default_rng(nv)
    lens = [0, 1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 129, 200, 0, 5]
    n, m = len(lens), 700
    row = np.concatenate(([0], np.cumsum(lens))).astype(np.uint32)
    col = np.concatenate([rng.choice(m, k, replace=False) for k in lens]).astype(np.uint32)
    val = rng.standard_normal(len(col))
    dt = np.float64 if prec == 0 else np.float32
    x, y0 = rng.standard_normal(m * nv).astype(dt), rng.standard_normal(n * nv).astype(dt)
    dx = X.DeviceArray.from_host(x)
    X.set_option("spmv_wave_enable", 1)
    try:
        for index_mode in (1, 2):
            A = X.Matrix(row, col, val, prec=prec, index_mode=index_mode, ncols=m)
            for add in (False, True):
                dy = X.DeviceArray.from_host(y0)
                A.spmv(nv, dx, dy, accumulate=add)
                ref = O.spmv(row, col, val, x, nv, y=y0 if add else None, ncols=m, f32=prec == 1)
                assert np.array_equal(dy.to_host(), ref), (index_mode, add)
    finally:
        X.set_option("spmv_wave_enable", 2)


@pytest.mark.parametrize("nv,prec", [(1, 0), (1, 1), (2, 0), (4, 1)])
def test_spmv_many_long_rows_few_rhs_bit_exact(gpu, O, nv, prec):
    # more than 65536 rows: 4 lanes per row
    X = gpu
    row, col, val = X.q1fem27(41, 41, 41)[:3]
    n = len(row) - 1
    dt = np.float64 if prec == 0 else np.float32
    x = np.random.default_rng(nv).standard_normal(n * nv).astype(dt)
    A = X.Matrix(row, col, val, prec=prec)
    dx, dy = X.DeviceArray.from_host(x), X.DeviceArray(n * nv, dt)
    X.set_option("spmv_wave_enable", 1)
    try:
        A.spmv(nv, dx, dy)
    finally:
        X.set_option("spmv_wave_enable", 2)
    assert np.array_equal(dy.to_host(), O.spmv(row, col, val, x, nv, f32=prec == 1))


@pytest.mark.parametrize("nv,mg_prec,dims,want", [
    (1, 0, (40, 40, 40), True), (2, 0, (40, 40, 40), False), (2, 0, (52, 51, 51), True),
    (2, 2, (40, 40, 40), True), (2, 0, (30, 30, 30), True), (4, 0, (30, 30, 30), False)])
def test_long_row_kernel_by_size_on_codes(gpu, nv, mg_prec, dims, want):
    # 27-point operators in the default mode: fp64 with two RHS reads codes between the cap of
    # 32768 rows and 2^17 rows; one RHS, and two in fp32, take the long-row kernel there
    X = gpu
    row, col, val = X.q1fem27(*dims)[:3]
    n = len(row) - 1
    levels = X.Amg(row, col, val, agg_num_levels=1, coarse_size=500).export()
    prm = X.default_params(method="MergedPBiCGStab", smoother="Jacobi", sweeps=2, mg_prec=mg_prec)
    S = X.Solver(X.Hier(levels), prm, nv)
    db, dx = X.DeviceArray.from_host(X.rhs_uniform(1, n, nv)), X.DeviceArray(n * nv)
    dx.zero()
    names = {k["kernel"] for k in S.profile(db, dx, 1) if k["level"] == 0}
    took = [k for k in names if k.startswith("k_spmv_wave<") and "OP_RESID" in k]
    assert bool(took) == want, names


@pytest.mark.parametrize("N,nv,want", [(28, 1, True), (32, 1, False), (28, 2, True),
                                       (32, 2, False), (12, 4, False)])
def test_long_row_kernel_by_size_on_short_rows(gpu, N, nv, want):
    # 7-point operators (4 to 12 entries per row) in the default mode: the long-row kernel up
    # to 24576 rows with one lane per entry, with more lanes none of a matrix with a grid view
    X = gpu
    row, col, val = X.varcoef7(N, sigma=1.0, seed=3)[:3]
    levels = X.Amg(row, col, val, agg_num_levels=1, coarse_size=60).export()
    prm = X.default_params(method="MergedPBiCGStab", smoother="Jacobi", sweeps=2)
    S = X.Solver(X.Hier(levels), prm, nv)
    db, dx = X.DeviceArray.from_host(X.rhs_uniform(1, N ** 3, nv)), X.DeviceArray(N ** 3 * nv)
    dx.zero()
    names = {k["kernel"] for k in S.profile(db, dx, 1)
             if k["level"] == 0 and "OP_RESID" in k["kernel"] and "RESID0" not in k["kernel"]}
    assert any(k.startswith("k_spmv_wave<") for k in names) == want, names


@pytest.mark.parametrize("smoother,nv,mg_prec", [("Chebyshev", 1, 0), ("Chebyshev", 8, 2),
                                                 ("Chebyshev", 32, 1), ("Jacobi", 4, 0),
                                                 ("HSGS", 2, 2), ("Chebyshev", 64, 0)])
def test_long_row_kernel_in_a_vcycle_is_identical(gpu, smoother, nv, mg_prec):
    # every V-cycle operation that can take it (residuals stored in fp32, Chebyshev steps
    # from zero and non-zero x, prolongation), against the row-parallel kernel
    X = gpu
    N = 20
    row, col, val = X.cube(N)
    levels = X.Amg(row, col, val, agg_num_levels=1, num_paths=2, coarse_size=60).export()
    prm = X.default_params(smoother=smoother, poly_order=4, mg_prec=mg_prec)
    S = X.Solver(X.Hier(levels), prm, nv)
    db = X.DeviceArray.from_host(X.rhs_uniform(3, N ** 3, nv))
    out = {}
    try:
        for on in (0, 1, 2):
            X.set_option("spmv_wave_enable", on)
            dx = X.DeviceArray(N ** 3 * nv)
            S.precond_apply(db, dx)
            out[on] = dx.to_host()
    finally:
        X.set_option("spmv_wave_enable", 2)
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])


@pytest.mark.parametrize("N,coarse_size,nv,mg_prec", [
    (10, 70, 8, 0), (10, 70, 32, 2), (10, 70, 64, 0), (10, 70, 64, 1), (16, 60, 64, 2),
    (16, 600, 16, 1), (16, 600, 64, 0), (16, 600, 1, 2)])
def test_dense_kernel_of_the_coarse_solve(gpu, O, N, coarse_size, nv, mg_prec):
    # coarse solves run in tiles, but for 64 RHS on less than 40 unknowns (33 here, then 45 and
    # 512); the fp64 solve of an fp32 hierarchy reads its vectors as they are
    X = gpu
    row, col, val = X.cube(N)
    levels = X.Amg(row, col, val, agg_num_levels=1, num_paths=2, coarse_size=coarse_size).export()
    nc, n = levels[-1]["A"][0], len(row) - 1
    assert nc == {70: 33, 60: 45, 600: 512}[coarse_size]
    prm = X.default_params(method="MergedPBiCGStab", mg_prec=mg_prec)
    S = X.Solver(X.Hier(levels), prm, nv)
    b = X.rhs_uniform(2, n, nv)
    db, dx = X.DeviceArray.from_host(b), X.DeviceArray(n * nv)
    S.precond_apply(db, dx)
    assert np.array_equal(dx.to_host(), O.mg_apply(O.Hier(levels), O.params_from(prm), nv, b))
    dx.zero()
    names = {k["kernel"] for k in S.profile(db, dx, 1)}
    types = {0: "double,double", 1: "float,float", 2: "double,float"}[mg_prec]
    assert f"k_dense{'_direct' if nv == 64 and nc < 40 else ''}<{types}>" in names, (nc, names)


def test_spmv_full_size_cube_128(gpu, O):
    # the benchmark operator at full size: 2,097,152 rows, u16 panel columns, nv = 32
    X = gpu
    row, col, val = X.cube(128)
    n, nv = len(row) - 1, 32
    A = X.Matrix(row, col, val, prec=0, index_mode=0)
    info = A.info()
    assert info["index_bits"] == 16 and info["panel_rows"] == 32768
    x = X.rhs_uniform(3, n, nv)
    dx, dy = X.DeviceArray.from_host(x), X.DeviceArray(n * nv)
    A.spmv(nv, dx, dy)
    assert np.array_equal(dy.to_host(), O.spmv(row, col, val, x, nv))


def test_bad_arguments_are_rejected(gpu):
    X = gpu
    row, col, val = X.cube(4)
    A = X.Matrix(row, col, val)
    d = X.DeviceArray(64 * 3)
    assert X.hip().xh_spmv(A.m, 3, d.ptr, d.ptr, 0) < 0  # nv = 3 unsupported
    bad = col.copy()
    bad[0] = 10 ** 6
    with pytest.raises(X.XamgError):
        X.Matrix(row, bad, val)
    with pytest.raises(X.XamgError):  # a row spanning more than 65536 columns
        X.Matrix(np.array([0, 2], np.uint32), np.array([0, 100000], np.uint32), np.ones(2),
                 index_mode=2, ncols=100001)
