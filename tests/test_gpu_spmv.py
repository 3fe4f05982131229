"""GPU parity: SELL-C-sigma sparse matrix times block vector and its fused
variants, through the C ABI, against the oracle (the builtin restatement
pinned in test_oracle.py).

Bars: index work (CRS order, SELL layout) bit-exact; FP64 results within
1e-12 relative to the oracle (normwise per column); FP32 results within
1e-5 relative to the FP64 oracle.  The reference's own golden vectors
(A2_precalc_result) are checked to sqrt(eps) as in its test.
"""
import ctypes
import json
import os

import numpy as np
import pytest

import oracle_lib as ol

pytestmark = pytest.mark.gpu

MATS = ["Dsprandn25", "Dsprandn388", "Dsprandn_nodiag25", "Dsprandsym163", "DsymmMat20", "DjadaTestMat512",
        "Dspshift25", "Dspzero25", "Dspeye25"]
RTOL = {np.float64: 1e-12, np.float32: 1e-5}


def colwise_rel(got, ref):
    """max over columns of ||got-ref|| / max(||ref||, tiny)"""
    num = np.linalg.norm(got - ref, axis=0)
    den = np.maximum(np.linalg.norm(ref, axis=0), 1e-300)
    return float(np.max(num / den)) if got.size else 0.0


def mm(name):
    return os.path.join(ol.MATRICES, name + ".mm")


@pytest.mark.parametrize("mat", MATS)
def test_crs_index_bitexact(be64, mat):
    A = be64.read_mm(mm(mat))
    ref = ol.crs_from_mm(mm(mat))
    ro, ci, va = A.crs()
    assert np.array_equal(ro, ref.row_offset)
    assert np.array_equal(ci, ref.col_idx)
    assert np.array_equal(va, ref.val)
    A.delete()


@pytest.mark.parametrize("mat", MATS)
def test_sell_invariants(be64, mat):
    A = be64.read_mm(mm(mat))
    ref = ol.crs_from_mm(mm(mat))
    s = A.sell()
    C, nch = s["C"], s["nchunks"]
    perm = s["perm"]
    n = ref.nrows
    # bijection on the real rows, padding rows marked -1
    assert sorted(perm[perm >= 0].tolist()) == list(range(n))
    assert np.all(perm[n:] == -1)
    lens = np.diff(ref.row_offset)
    # descending length inside sigma windows (stable)
    sig = s["sigma"]
    for w0 in range(0, n, max(sig, 1)):
        win = perm[w0:min(n, w0 + max(sig, 1))]
        l = lens[win]
        assert np.all(l[:-1] >= l[1:]) or sig == 1
    # chunk widths and slots reproduce every row in CRS order, padding is zero
    for c in range(nch):
        w = s["chunk_w"][c]
        assert s["chunk_ptr"][c + 1] - s["chunk_ptr"][c] == w * C
        for r in range(C):
            row = perm[c * C + r]
            slots = s["chunk_ptr"][c] + np.arange(w) * C + r
            if row < 0:
                assert np.all(s["val"][slots] == 0)
                continue
            a, b = ref.row_offset[row] - 1, ref.row_offset[row + 1] - 1
            L = b - a
            assert w >= L
            assert np.array_equal(s["col"][slots[:L]], ref.col_idx[a:b] - 1)
            assert np.array_equal(s["val"][slots[:L]], ref.val[a:b])
            assert np.all(s["val"][slots[L:]] == 0)
    A.delete()


@pytest.mark.parametrize("nvec", [1, 4])
def test_reference_golden_vectors(be64, nvec):
    with open(os.path.join(ol.GOLDEN, "a2_precalc_sprandn25.json")) as f:
        g = json.load(f)
    A = be64.read_mm(mm("Dsprandn25"))
    m = be64.map(25)
    x = be64.mvec(m, nvec, np.array([[i + j * 25 for j in range(nvec)] for i in range(25)], float))
    y = be64.mvec(m, nvec)
    be64.spmv(1.0, A, x, 0.0, y)
    ref = np.array(g[f"nvec{nvec}"]).reshape(25, nvec)
    assert np.max(np.abs(y.get() - ref)) <= np.sqrt(np.finfo(float).eps)
    for o in (x, y, A):
        o.delete()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("mat", MATS)
@pytest.mark.parametrize("nvec", [1, 2, 3, 4, 7, 8, 12, 16, 32])
@pytest.mark.parametrize("alpha,beta,shifted", [(1.0, 0.0, False), (0.7, -0.3, False), (-1.3, 0.5, True)])
def test_spmv_vs_oracle(be64, be32, dtype, mat, nvec, alpha, beta, shifted):
    be = be64 if dtype == np.float64 else be32
    A = be.read_mm(mm(mat))
    ref = ol.crs_from_mm(mm(mat))
    rng = np.random.default_rng(nvec * 31 + len(mat))
    X = rng.uniform(-1, 1, (ref.ncols, nvec)).astype(dtype)
    Y0 = rng.uniform(-1, 1, (ref.nrows, nvec)).astype(dtype)
    sh = rng.uniform(-1, 1, nvec).astype(dtype)
    m = be.map(ref.nrows)
    x = be.mvec(m, nvec, X)
    y = be.mvec(m, nvec, Y0)
    if shifted:
        be.spmv_shifted(alpha, A, sh, x, beta, y)
    else:
        be.spmv(alpha, A, x, beta, y)
    want = ol.spmv(ref, alpha, X.astype(float), beta, Y0.astype(float), shifts=sh.astype(float) if shifted else None)
    assert colwise_rel(y.get().astype(float), want) <= RTOL[dtype]
    for o in (x, y, A):
        o.delete()
    m.delete()


@pytest.mark.parametrize("nvec,jmin,jmax", [(8, 2, 5), (12, 4, 11), (5, 1, 1), (16, 0, 7)])
def test_spmv_on_column_views(be64, nvec, jmin, jmax):
    """strided views (lda > nvec): x and y are column blocks of wider mvecs"""
    A = be64.read_mm(mm("Dsprandn388"))
    ref = ol.crs_from_mm(mm("Dsprandn388"))
    rng = np.random.default_rng(1)
    X = rng.uniform(-1, 1, (388, nvec))
    Y = rng.uniform(-1, 1, (388, nvec))
    m = be64.map(388)
    x = be64.mvec(m, nvec, X)
    y = be64.mvec(m, nvec, Y)
    xv = x.view(jmin, jmax)
    yv = y.view(jmin, jmax)
    be64.spmv(0.9, A, xv, 0.4, yv)
    want = Y.copy()
    want[:, jmin:jmax + 1] = ol.spmv(ref, 0.9, X[:, jmin:jmax + 1], 0.4, Y[:, jmin:jmax + 1])
    got = y.get()
    assert colwise_rel(got, want) <= 1e-12
    # columns outside the view are untouched (bit-exact)
    mask = np.ones(nvec, bool)
    mask[jmin:jmax + 1] = False
    assert np.array_equal(got[:, mask], Y[:, mask])
    for o in (xv, yv, x, y, A):
        o.delete()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nvec", [1, 4, 8, 16])
@pytest.mark.parametrize("beta", [0.0, 0.25])
@pytest.mark.parametrize("which", ["both", "ww", "vw", "none"])
def test_fused_spmv_mvdot(be64, be32, dtype, nvec, beta, which):
    be = be64 if dtype == np.float64 else be32
    A = be.read_mm(mm("Dsprandsym163"))
    ref = ol.crs_from_mm(mm("Dsprandsym163"))
    rng = np.random.default_rng(nvec)
    V = rng.uniform(-1, 1, (163, nvec)).astype(dtype)
    W0 = rng.uniform(-1, 1, (163, nvec)).astype(dtype)
    m = be.map(163)
    v = be.mvec(m, nvec, V)
    w = be.mvec(m, nvec, W0)
    ww, vw = be.fused_spmv_mvdot(1.1, A, v, beta, w, want_ww=which in ("both", "ww"), want_vw=which in ("both", "vw"))
    Wref = ol.spmv(ref, 1.1, V.astype(float), beta, W0.astype(float))
    tol = RTOL[dtype]
    assert colwise_rel(w.get().astype(float), Wref) <= tol
    if ww is not None:
        assert np.allclose(ww, ol.dot(Wref, Wref), rtol=10 * tol, atol=0)
    if vw is not None:
        scale = ol.dot(np.abs(V.astype(float)), np.abs(Wref))
        assert np.all(np.abs(vw - ol.dot(V.astype(float), Wref)) <= 10 * tol * scale)
    for o in (v, w, A):
        o.delete()


def test_fused_spmv_mvdot_mvadd(be64):
    A = be64.read_mm(mm("Dsprandn388"))
    ref = ol.crs_from_mm(mm("Dsprandn388"))
    rng = np.random.default_rng(5)
    V, W0, U0 = (rng.uniform(-1, 1, (388, 4)) for _ in range(3))
    m = be64.map(388)
    v, w, u = be64.mvec(m, 4, V), be64.mvec(m, 4, W0), be64.mvec(m, 4, U0)
    import ctypes
    ww = np.zeros(4)
    vw = np.zeros(4)
    be64.call("fused_spmv_mvdot_mvadd", be64.s(0.5), A.h, v.h, be64.s(2.0), w.h, be64.s(-1.5), be64.s(0.75), u.h,
              ww.ctypes.data_as(ctypes.c_void_p), vw.ctypes.data_as(ctypes.c_void_p))
    Wref = ol.spmv(ref, 0.5, V, 2.0, W0)
    Uref = -1.5 * Wref + 0.75 * U0
    assert colwise_rel(w.get(), Wref) <= 1e-12
    assert colwise_rel(u.get(), Uref) <= 1e-12
    assert np.allclose(ww, ol.dot(Wref, Wref), rtol=1e-12)
    assert np.allclose(vw, ol.dot(V, Wref), rtol=1e-11, atol=1e-12)
    for o in (v, w, u, A):
        o.delete()


def test_spmv_alpha_zero_only_scales(be64):
    A = be64.read_mm(mm("Dsprandn25"))
    m = be64.map(25)
    Y = np.random.default_rng(0).uniform(-1, 1, (25, 3))
    x = be64.mvec(m, 3, np.full((25, 3), np.nan))
    y = be64.mvec(m, 3, Y)
    be64.spmv(0.0, A, x, 0.5, y)
    assert np.array_equal(y.get(), 0.5 * Y)
    for o in (x, y, A):
        o.delete()


def test_empty_rows_and_zero_matrix(be64):
    # Dspzero25 holds explicit zeros; a fully empty matrix only scales y
    import ctypes
    import phist_amd
    rows = ol.crs_from_rows(6, 6, [([], []), ([0, 5], [1.0, 2.0]), ([], []), ([3], [4.0]), ([], []), ([], [])])

    @phist_amd.ROWFUNC
    def rf(i, nnz, cols, vals, arg):
        a, b = rows.row_offset[i] - 1, rows.row_offset[i + 1] - 1
        nnz[0] = b - a
        dv = ctypes.cast(vals, ctypes.POINTER(ctypes.c_double))
        for k in range(a, b):
            cols[k - a] = rows.col_idx[k] - 1
            dv[k - a] = rows.val[k]
        return 0

    A = be64.from_rowfunc(6, 2, rf, None)
    m = be64.map(6)
    X = np.arange(12.0).reshape(6, 2)
    x = be64.mvec(m, 2, X)
    y = be64.mvec(m, 2, np.full((6, 2), 3.0))
    be64.spmv(2.0, A, x, 0.0, y)
    assert np.array_equal(y.get(), ol.spmv(rows, 2.0, X, 0.0, np.zeros((6, 2))))
    ro, ci, va = A.crs()
    assert np.array_equal(ro, rows.row_offset) and np.array_equal(ci, rows.col_idx)
    for o in (x, y, A):
        o.delete()


@pytest.mark.parametrize("C,sigma", [(1, 1), (4, 1), (8, 16), (32, 256), (64, 64)])
def test_sell_parameters(be64, C, sigma):
    """any power-of-two C and any sigma give the same product"""
    import ctypes
    iflag = ctypes.c_int(0)
    be64.L.phist_amd_sparseMat_set_format(C, sigma, ctypes.byref(iflag))
    try:
        A = be64.read_mm(mm("DjadaTestMat512"))
    finally:
        be64.L.phist_amd_sparseMat_set_format(0, 0, ctypes.byref(iflag))
    ref = ol.crs_from_mm(mm("DjadaTestMat512"))
    s = A.sell()
    assert s["C"] == C
    X = np.random.default_rng(C).uniform(-1, 1, (512, 8))
    m = be64.map(512)
    x = be64.mvec(m, 8, X)
    y = be64.mvec(m, 8)
    be64.spmv(1.0, A, x, 0.0, y)
    assert colwise_rel(y.get(), ol.spmv(ref, 1.0, X, 0.0, np.zeros((512, 8)))) <= 1e-12
    for o in (x, y, A):
        o.delete()


@pytest.mark.parametrize("n,nnz,hb", [(20000, 32, 500), (4096, 9, 100)])
def test_banded_generator_rows_and_product(be64, n, nnz, hb):
    """the bench's generator through create_fromRowFuncWithConstructor:
    distinct columns inside the band, diagonal 40, product vs the oracle"""
    A = be64.banded_random(n, nnz, hb, 40.0, 1234)
    ro, ci, va = A.crs()
    ref = ol.Crs(n, n, ro, ci, va)
    lens = np.diff(ro)
    assert np.all(lens == nnz)
    for i in range(0, n, 997):
        cols = ci[ro[i] - 1:ro[i + 1] - 1] - 1
        assert len(set(cols)) == len(cols) and np.all(np.diff(cols) > 0)
        assert np.all(np.abs(cols - i) <= hb)
        d = va[ro[i] - 1:ro[i + 1] - 1][cols == i]
        assert d.tolist() == [40.0]
    X = np.random.default_rng(2).uniform(-1, 1, (n, 8))
    m = be64.map(n)
    x = be64.mvec(m, 8, X)
    y = be64.mvec(m, 8)
    ww, vw = be64.fused_spmv_mvdot(1.0, A, x, 0.0, y)
    Yref = ol.spmv(ref, 1.0, X, 0.0, np.zeros((n, 8)))
    assert colwise_rel(y.get(), Yref) <= 1e-12
    assert np.allclose(ww, ol.dot(Yref, Yref), rtol=1e-12)
    for o in (x, y, A):
        o.delete()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nvec", [12, 16, 24])
def test_spmv_column_blocks_large(be64, be32, dtype, nvec):
    """300000 rows of 9 nonzeros and 12-24 columns (a persistent grid of
    many tiles per workgroup): shifts, beta and both dot products"""
    be = be64 if dtype == np.float64 else be32
    n = 300000
    A = be.banded_random(n, 9, 100, 40.0, 77)
    ro, ci, va = A.crs()
    ref = ol.Crs(n, n, ro, ci, va.astype(float))
    rng = np.random.default_rng(nvec)
    X = rng.uniform(-1, 1, (n, nvec)).astype(dtype)
    Y0 = rng.uniform(-1, 1, (n, nvec)).astype(dtype)
    shifts = rng.uniform(-2, 2, nvec).astype(dtype)
    m = be.map(n)
    x, y = be.mvec(m, nvec, X), be.mvec(m, nvec, Y0)
    be.spmv_shifted(0.7, A, shifts, x, 0.3, y)
    Xf = X.astype(float)
    want = ol.spmv(ref, 0.7, Xf, 0.3, Y0.astype(float), shifts=shifts.astype(float))
    tol = RTOL[dtype]
    assert colwise_rel(y.get().astype(float), want) <= tol
    w = be.mvec(m, nvec, Y0)
    ww, vw = be.fused_spmv_mvdot(1.1, A, x, 0.5, w)
    Wref = ol.spmv(ref, 1.1, Xf, 0.5, Y0.astype(float))
    assert colwise_rel(w.get().astype(float), Wref) <= tol
    assert np.allclose(ww, ol.dot(Wref, Wref), rtol=10 * tol, atol=0)
    scale = ol.dot(np.abs(Xf), np.abs(Wref))
    assert np.all(np.abs(vw - ol.dot(Xf, Wref)) <= 10 * tol * scale)
    for o in (x, y, w, A):
        o.delete()


def _p(a):
    import ctypes
    return a.ctypes.data_as(ctypes.c_void_p)


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nvec", [1, 4, 8])
def test_spmv_add_mvec_scalar_shift(be64, be32, dtype, nvec):
    """sparseMat_times_mvec_add_mvec: y = alpha*(A + shift I)x + beta*y with one scalar shift
    (kernels_common_impl_def.h:55-64)"""
    be = be64 if dtype == np.float64 else be32
    A = be.read_mm(mm("Dsprandn388"))
    ref = ol.crs_from_mm(mm("Dsprandn388"))
    rng = np.random.default_rng(nvec + 40)
    X = rng.uniform(-1, 1, (388, nvec)).astype(dtype)
    Y0 = rng.uniform(-1, 1, (388, nvec)).astype(dtype)
    m = be.map(388)
    x, y = be.mvec(m, nvec, X), be.mvec(m, nvec, Y0)
    be.call("sparseMat_times_mvec_add_mvec", be.s(0.6), A.h, be.s(-1.7), x.h, be.s(0.4), y.h)
    want = ol.spmv(ref, 0.6, X.astype(float), 0.4, Y0.astype(float), shifts=np.full(nvec, -1.7))
    assert colwise_rel(y.get().astype(float), want) <= RTOL[dtype]
    for o in (x, y, A):
        o.delete()


def _gram_bound(tol, a, b):
    return 8 * tol * (np.abs(a).T @ np.abs(b))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nvec", [1, 3, 4, 8, 16, 17, 24, 32, 40])
@pytest.mark.parametrize("case", ["W", "W_beta", "W_null", "ww_only", "vw_only", "W_no_gram"])
def test_fused_spmv_mvTmv(be64, be32, dtype, nvec, case):
    """fused_spmv_mvTmv (phist_kernels_fused_decl.h:68, kernels_no_fused_spmv_mvTmv.cpp:9-57):
    W = alpha*A*V + beta*W, WtW = W'W, VtW = V'W; W = NULL means alpha = 1, beta = 0 and W is not
    returned; WtW / VtW may be NULL.  Up to 32 columns this is one pass (Gram epilogue on the matrix
    cores), 40 columns take the three-pass path."""
    be = be64 if dtype == np.float64 else be32
    A = be.read_mm(mm("DjadaTestMat512"))
    ref = ol.crs_from_mm(mm("DjadaTestMat512"))
    n = ref.nrows
    rng = np.random.default_rng(nvec * 7 + len(case))
    V = rng.uniform(-1, 1, (n, nvec)).astype(dtype)
    W0 = rng.uniform(-1, 1, (n, nvec)).astype(dtype)
    alpha, beta = 0.9, (0.35 if case == "W_beta" else 0.0)
    m = be.map(n)
    v = be.mvec(m, nvec, V)
    w = None if case == "W_null" else be.mvec(m, nvec, W0)
    C0 = rng.uniform(-1, 1, (nvec, nvec))
    wtw = None if case in ("vw_only", "W_no_gram") else be.sdmat(nvec, nvec, C0)
    vtw = None if case in ("ww_only", "W_no_gram") else be.sdmat(nvec, nvec, C0)
    be.call("fused_spmv_mvTmv", be.s(alpha), A.h, v.h, be.s(beta), w.h if w else None, wtw.h if wtw else None,
            vtw.h if vtw else None)
    Vf = V.astype(float)
    a_eff, b_eff = (1.0, 0.0) if w is None else (alpha, beta)
    Wref = ol.spmv(ref, a_eff, Vf, b_eff, W0.astype(float))
    tol = RTOL[dtype]
    if w is not None:
        Wgot = w.get().astype(float)
        assert colwise_rel(Wgot, Wref) <= tol
        if case == "W_no_gram":
            assert np.array_equal(Wgot, Wref) or colwise_rel(Wgot, Wref) <= tol
    if wtw is not None:
        G = wtw.get().astype(float)
        assert np.all(np.abs(G - ol.gram(1.0, Wref, Wref, 0.0, np.zeros((nvec, nvec)))) <=
                      _gram_bound(tol, Wref, Wref))
        assert np.array_equal(G, G.T)  # the mirrored tiles are exact copies
    if vtw is not None:
        G = vtw.get().astype(float)
        assert np.all(np.abs(G - ol.gram(1.0, Vf, Wref, 0.0, np.zeros((nvec, nvec)))) <= _gram_bound(tol, Vf, Wref))
    for o in (v, w, wtw, vtw, A):
        if o is not None:
            o.delete()


@pytest.mark.parametrize("nvec", [8, 32])
def test_fused_spmv_mvTmv_large(be64, nvec):
    """one-pass Gram epilogue over a persistent grid (300000 rows): both Grams against the oracle"""
    n = 300000
    A = be64.banded_random(n, 9, 100, 40.0, 31)
    ro, ci, va = A.crs()
    ref = ol.Crs(n, n, ro, ci, va)
    rng = np.random.default_rng(nvec)
    V = rng.uniform(-1, 1, (n, nvec))
    m = be64.map(n)
    v, w = be64.mvec(m, nvec, V), be64.mvec(m, nvec)
    wtw, vtw = be64.sdmat(nvec, nvec), be64.sdmat(nvec, nvec)
    be64.call("fused_spmv_mvTmv", be64.s(1.3), A.h, v.h, be64.s(0.0), w.h, wtw.h, vtw.h)
    Wref = ol.spmv(ref, 1.3, V, 0.0, np.zeros((n, nvec)))
    assert colwise_rel(w.get(), Wref) <= 1e-12
    assert np.all(np.abs(wtw.get() - ol.gram(1.0, Wref, Wref, 0.0, np.zeros((nvec, nvec)))) <=
                  _gram_bound(1e-12, Wref, Wref))
    assert np.all(np.abs(vtw.get() - ol.gram(1.0, V, Wref, 0.0, np.zeros((nvec, nvec)))) <=
                  _gram_bound(1e-12, V, Wref))
    for o in (v, w, wtw, vtw, A):
        o.delete()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nvec", [1, 4])
def test_fused_spmv_pair(be64, be32, dtype, nvec):
    """fused_spmv_pair: Y = alpha*(shifts1[j]*A1 + shifts2[j]*A2) X_j + beta*Y
    (phist_kernels_fused_decl.h:45, kernels_no_fused_spmv_pair.cpp:9-49)"""
    be = be64 if dtype == np.float64 else be32
    A1, A2 = be.read_mm(mm("Dsprandn25")), be.read_mm(mm("Dspshift25"))
    r1, r2 = ol.crs_from_mm(mm("Dsprandn25")), ol.crs_from_mm(mm("Dspshift25"))
    rng = np.random.default_rng(nvec + 3)
    X = rng.uniform(-1, 1, (25, nvec)).astype(dtype)
    Y0 = rng.uniform(-1, 1, (25, nvec)).astype(dtype)
    s1 = rng.uniform(-2, 2, nvec).astype(dtype)
    s2 = rng.uniform(-2, 2, nvec).astype(dtype)
    m = be.map(25)
    x, y = be.mvec(m, nvec, X), be.mvec(m, nvec, Y0)
    be.call("fused_spmv_pair", be.s(0.7), _p(s1), A1.h, _p(s2), A2.h, x.h, be.s(-0.5), y.h)
    Xf = X.astype(float)
    t1 = ol.spmv(r1, 0.7, Xf, 0.0, np.zeros((25, nvec)))
    t2 = ol.spmv(r2, 0.7, Xf, 0.0, np.zeros((25, nvec)))
    want = s1.astype(float) * t1 + s2.astype(float) * t2 - 0.5 * Y0.astype(float)
    assert colwise_rel(y.get().astype(float), want) <= RTOL[dtype]
    for o in (x, y, A1, A2):
        o.delete()


def test_mvec_QR_not_implemented(be64):
    """builtin's mvec_QR returns -99 so that callers fall back to CholQR (kernels_def.hpp:939-947)"""
    m = be64.map(100)
    v = be64.mvec(m, 4, np.random.default_rng(0).uniform(-1, 1, (100, 4)))
    r = be64.sdmat(4, 4)
    assert be64.call("mvec_QR", v.h, r.h, allow=(0, -99)) == -99
    for o in (v, r):
        o.delete()
    m.delete()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nvec", [8, 16, 32])
def test_spmv_lane_widths_bitexact(be64, be32, dtype, nvec):
    """every gather width per lane (one scalar, one to four 16-byte vectors)
    gives the default's SpMV result bit for bit, shifts and beta included (a
    row's sum is formed by the lane owning its columns, in entry order), and
    the default agrees with the oracle.  The column dots are reduced over the
    rows of a wave, whose number changes with the lane width, so they agree
    to rounding only."""
    import ctypes
    be = be64 if dtype == np.float64 else be32
    n = 40000
    A = be.banded_random(n, 17, 3000, 40.0, 99)
    ro, ci, va = A.crs()
    ref = ol.Crs(n, n, ro, ci, va.astype(float))
    rng = np.random.default_rng(nvec + 5)
    X = rng.uniform(-1, 1, (n, nvec)).astype(dtype)
    Y0 = rng.uniform(-1, 1, (n, nvec)).astype(dtype)
    shifts = rng.uniform(-2, 2, nvec).astype(dtype)
    m = be.map(n)
    x = be.mvec(m, nvec, X)
    fl = ctypes.c_int(0)
    out = {}
    try:
        for lb in (0, np.dtype(dtype).itemsize, 16, 32, 64):
            be.L.phist_amd_set_spmv_lane_bytes(lb, ctypes.byref(fl))
            assert fl.value == 0
            y = be.mvec(m, nvec, Y0)
            be.spmv_shifted(0.7, A, shifts, x, 0.3, y)
            w = be.mvec(m, nvec, Y0)
            ww, vw = be.fused_spmv_mvdot(1.1, A, x, 0.5, w)
            out[lb] = (y.get(), w.get(), ww, vw)
            y.delete()
            w.delete()
    finally:
        be.L.phist_amd_set_spmv_lane_bytes(0, ctypes.byref(fl))
    want = ol.spmv(ref, 0.7, X.astype(float), 0.3, Y0.astype(float), shifts=shifts.astype(float))
    assert colwise_rel(out[0][0].astype(float), want) <= RTOL[dtype]
    dtol = 1e-13 if dtype == np.float64 else 1e-5
    for lb, got in out.items():
        for g, d in zip(got[:2], out[0][:2]):
            assert np.array_equal(g, d), f"lane width {lb} bytes: SpMV result differs from the default"
        for g, d in zip(got[2:], out[0][2:]):
            assert np.max(np.abs(g - d) / np.abs(d)) <= dtol, f"lane width {lb} bytes: dots differ"
    for o in (x, A):
        o.delete()
    m.delete()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["sheet", "stencil", "band12", "band20", "band30"])
def test_spmv_widths_by_column(be64, be32, kind, dtype):
    """every block width runs each column's own sum: the columns of a block
    product equal the one-column products bit for bit, whole vectors and
    ragged widths, rows of at most 4, of 7, 12, 20 and 30 entries, plain and
    shifted with beta, on whole blocks and on a column view that starts and
    ends unaligned; the columns next to the view stay as they were; the dots
    agree with the columns"""
    be = be64 if dtype == np.float64 else be32
    A = {"sheet": lambda: be.honeycomb(37, 23, 0, 0, 0, 1.0, 7), "stencil": lambda: be.laplace3d(13, 7, 9),
         "band12": lambda: be.banded_random(1001, 12, 60, 40.0, 5),
         "band20": lambda: be.banded_random(999, 20, 90, 40.0, 9),
         "band30": lambda: be.banded_random(997, 30, 400, 40.0, 6)}[kind]()
    n, widest = A.nrows, 133
    rng = np.random.default_rng(17)
    X, Y0 = (rng.uniform(-1, 1, (n, widest)).astype(dtype) for _ in range(2))
    sh = rng.uniform(-2, 2, widest).astype(dtype)
    m = be.map(n)
    one, shifted = np.empty_like(X), np.empty_like(X)
    x, y = be.mvec(m, 1), be.mvec(m, 1)
    for c in range(widest):
        x.set(X[:, c:c + 1])
        be.spmv(0.75, A, x, 0.0, y)
        one[:, c:c + 1] = y.get()
        y.set(Y0[:, c:c + 1])
        be.spmv_shifted(0.75, A, sh[c:c + 1], x, -0.3, y)
        shifted[:, c:c + 1] = y.get()
    x.delete()
    y.delete()
    tol = 1e-12 if dtype == np.float64 else 1e-4  # sums of at most 1001 terms, products of like sign summed
    for k in (2, 3, 4, 5, 6, 7, 8, 9, 12, 15, 16, 17, 31, 32, 33, 63, 65, 129, 133):
        x, y = be.mvec(m, k, X[:, :k]), be.mvec(m, k, Y0[:, :k])
        be.spmv(0.75, A, x, 0.0, y)
        assert np.array_equal(y.get(), one[:, :k]), k
        y.set(Y0[:, :k])
        be.spmv_shifted(0.75, A, sh[:k], x, -0.3, y)
        assert np.array_equal(y.get(), shifted[:, :k]), k
        if k <= 64:
            ww, vw = be.fused_spmv_mvdot(0.75, A, x, 0.0, y)
            assert np.array_equal(y.get(), one[:, :k]), k
            w, v = one[:, :k].astype(float), X[:, :k].astype(float)
            assert np.all(np.abs(ww - (w * w).sum(0)) <= tol * (w * w).sum(0)), k
            assert np.all(np.abs(vw - (v * w).sum(0)) <= tol * np.abs(v * w).sum(0)), k
        x.delete()
        y.delete()
        big = np.full((n, k + 2), 3.0, dtype)
        big[:, 1:k + 1] = X[:, :k]
        X2, Y2 = be.mvec(m, k + 2, big), be.mvec(m, k + 2, np.full((n, k + 2), 5.0, dtype))
        x, y = X2.view(1, k), Y2.view(1, k)
        be.spmv(0.75, A, x, 0.0, y)
        got = Y2.get()
        assert np.array_equal(got[:, 1:k + 1], one[:, :k]), k
        assert np.all(got[:, [0, k + 1]] == 5.0), k
        for o in (x, y, X2, Y2):
            o.delete()
    A.delete()
    m.delete()


@pytest.mark.parametrize("k", [1, 3, 4])
def test_spmv_block_over_4_gib(be64, k):
    """x rows beyond 4 GiB of their block (a view of a wide block, 64-bit
    offsets): the product of the compact block, bit for bit"""
    A = be64.laplace3d(108, 107, 106)
    n, ld = A.nrows, 448
    assert n * ld * 8 > 2**32
    m = be64.map(n)
    X = np.random.default_rng(3).uniform(-1, 1, (n, k))
    x, y = be64.mvec(m, k, X), be64.mvec(m, k)
    be64.spmv(1.0, A, x, 0.0, y)
    want = y.get()
    wide = be64.mvec(m, ld)
    xv = wide.view(ld - k, ld - 1)
    be64.call("mvec_add_mvec", be64.s(1.0), x.h, be64.s(0.0), xv.h)
    be64.spmv(1.0, A, xv, 0.0, y)
    assert np.array_equal(y.get(), want)
    for o in (xv, wide, x, y, A):
        o.delete()
    m.delete()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["sheet", "stencil", "band12", "band30"])
def test_spmv_blocks_past_one_launch(be64, be32, kind, dtype):
    """blocks wider than the 256 columns of a launch, at every lane width: the
    columns equal those of products of at most 100 columns bit for bit, plain
    and with a shift per column, and the dots agree with the columns"""
    be = be64 if dtype == np.float64 else be32
    A = {"sheet": lambda: be.honeycomb(19, 23, 0, 0, 0, 1.0, 7), "stencil": lambda: be.laplace3d(9, 7, 8),
         "band12": lambda: be.banded_random(501, 12, 60, 40.0, 5),
         "band30": lambda: be.banded_random(497, 30, 100, 40.0, 6)}[kind]()
    n, widest = A.nrows, 1048
    rng = np.random.default_rng(23)
    X, Y0 = (rng.uniform(-1, 1, (n, widest)).astype(dtype) for _ in range(2))
    sh = rng.uniform(-2, 2, widest).astype(dtype)
    m = be.map(n)
    one, shifted = np.empty_like(X), np.empty_like(X)
    for c in range(0, widest, 100):
        s = slice(c, min(widest, c + 100))
        x, y = be.mvec(m, s.stop - c, X[:, s]), be.mvec(m, s.stop - c)
        be.spmv(0.75, A, x, 0.0, y)
        one[:, s] = y.get()
        y.set(Y0[:, s])
        be.spmv_shifted(0.75, A, sh[s], x, -0.3, y)
        shifted[:, s] = y.get()
        x.delete()
        y.delete()
    tol = 1e-12 if dtype == np.float64 else 1e-4  # sums of at most 504 products
    fl = ctypes.c_int(0)
    try:
        for lane_bytes in (0, np.dtype(dtype).itemsize, 32, 64):
            be.L.phist_amd_set_spmv_lane_bytes(lane_bytes, ctypes.byref(fl))
            assert fl.value == 0
            for k in (255, 256, 257, 264, 272, 511, 512, 520, 1024, 1048):
                x, y = be.mvec(m, k, X[:, :k]), be.mvec(m, k, Y0[:, :k])
                be.spmv_shifted(0.75, A, sh[:k], x, -0.3, y)
                assert np.array_equal(y.get(), shifted[:, :k]), (lane_bytes, k)
                be.spmv(0.75, A, x, 0.0, y)
                assert np.array_equal(y.get(), one[:, :k]), (lane_bytes, k)
                ww, vw = be.fused_spmv_mvdot(0.75, A, x, 0.0, y)
                assert np.array_equal(y.get(), one[:, :k]), (lane_bytes, k)
                w, v = one[:, :k].astype(float), X[:, :k].astype(float)
                assert np.all(np.abs(ww - (w * w).sum(0)) <= tol * (w * w).sum(0)), (lane_bytes, k)
                assert np.all(np.abs(vw - (v * w).sum(0)) <= tol * np.abs(v * w).sum(0)), (lane_bytes, k)
                x.delete()
                y.delete()
    finally:
        be.L.phist_amd_set_spmv_lane_bytes(0, ctypes.byref(fl))
    A.delete()
    m.delete()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind,widths", [("stencil", (4, 5, 8)), ("chain", (4, 7, 8)), ("band12", (4, 5, 8, 16)),
                                         ("band30", (4, 5, 8, 33)), ("far30", (1, 33, 65)), ("short30", (4, 16, 33))])
def test_spmv_launch_rules(be64, be32, kind, widths, dtype):
    """the launches chosen by rows in flight, by how near and how far apart
    the gathered x rows lie and by the size of the block: each gives the
    columns of the one-column products bit for bit, plain and shifted with
    beta, and dots that agree with them"""
    be = be64 if dtype == np.float64 else be32
    A = {"stencil": lambda: be.laplace3d(53, 52, 51), "chain": lambda: be.spinchain_sz(19, 9),
         "band12": lambda: be.banded_random(70001, 12, 3000, 40.0, 5),
         "band30": lambda: be.banded_random(40001, 30, 3000, 40.0, 6),
         "far30": lambda: be.banded_random(140001, 30, 35000, 40.0, 7),
         "short30": lambda: be.banded_random(5001, 30, 1200, 40.0, 8)}[kind]()
    n, widest = A.nrows, max(widths)
    rng = np.random.default_rng(29)
    X, Y0 = (rng.uniform(-1, 1, (n, widest)).astype(dtype) for _ in range(2))
    sh = rng.uniform(-2, 2, widest).astype(dtype)
    m = be.map(n)
    one, shifted = np.empty_like(X), np.empty_like(X)
    x, y = be.mvec(m, 1), be.mvec(m, 1)
    for c in range(widest):
        x.set(X[:, c:c + 1])
        be.spmv(0.75, A, x, 0.0, y)
        one[:, c:c + 1] = y.get()
        y.set(Y0[:, c:c + 1])
        be.spmv_shifted(0.75, A, sh[c:c + 1], x, -0.3, y)
        shifted[:, c:c + 1] = y.get()
    x.delete()
    y.delete()
    eps = np.finfo(dtype).eps
    for k in widths:
        x, y = be.mvec(m, k, X[:, :k]), be.mvec(m, k, Y0[:, :k])
        be.spmv_shifted(0.75, A, sh[:k], x, -0.3, y)
        assert np.array_equal(y.get(), shifted[:, :k]), k
        be.spmv(0.75, A, x, 0.0, y)
        assert np.array_equal(y.get(), one[:, :k]), k
        ww, vw = be.fused_spmv_mvdot(0.75, A, x, 0.0, y)
        assert np.array_equal(y.get(), one[:, :k]), k
        w, v = one[:, :k].astype(float), X[:, :k].astype(float)
        assert np.all(np.abs(ww - (w * w).sum(0)) <= (n + 2) * eps * (w * w).sum(0)), k
        assert np.all(np.abs(vw - (v * w).sum(0)) <= (n + 2) * eps * np.abs(v * w).sum(0)), k
        x.delete()
        y.delete()
    A.delete()
    m.delete()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("kind", ["sheet", "stencil", "band20", "band30"])
def test_spmv_views_of_a_wide_block(be64, be32, kind, dtype):
    """columns of a block of 40 and 41, each row on cache lines of its own,
    have launches of their own: the compact block's product bit for bit,
    plain and shifted with beta, dots that agree with it, and the columns
    beside the view as they were"""
    be = be64 if dtype == np.float64 else be32
    A = {"sheet": lambda: be.honeycomb(301, 299, 0, 0, 0, 1.0, 7), "stencil": lambda: be.laplace3d(53, 52, 51),
         "band20": lambda: be.banded_random(30001, 20, 7000, 40.0, 5),
         "band30": lambda: be.banded_random(40001, 30, 3000, 40.0, 6)}[kind]()
    n = A.nrows
    rng = np.random.default_rng(31)
    m = be.map(n)
    eps = np.finfo(dtype).eps
    for k, ld, ofs in ((1, 41, 0), (1, 40, 1), (2, 40, 0), (2, 41, 39), (4, 40, 4), (4, 41, 1), (5, 40, 0), (8, 40, 3),
                       (33, 41, 2)):
        X, Y = (rng.uniform(-1, 1, (n, ld)).astype(dtype) for _ in range(2))
        sh = rng.uniform(-2, 2, k).astype(dtype)
        cols = slice(ofs, ofs + k)
        x, y = be.mvec(m, k, X[:, cols]), be.mvec(m, k, Y[:, cols])
        be.spmv_shifted(0.75, A, sh, x, -0.3, y)
        shifted = y.get()
        be.spmv(0.75, A, x, 0.0, y)
        plain = y.get()
        XB, YB = be.mvec(m, ld, X), be.mvec(m, ld, Y)
        xv, yv = XB.view(ofs, ofs + k - 1), YB.view(ofs, ofs + k - 1)
        be.spmv_shifted(0.75, A, sh, xv, -0.3, yv)
        got, want = YB.get(), Y.copy()
        want[:, cols] = shifted
        assert np.array_equal(got, want), (k, ld, ofs)
        be.spmv(0.75, A, xv, 0.0, yv)
        want[:, cols] = plain
        assert np.array_equal(YB.get(), want), (k, ld, ofs)
        ww, vw = be.fused_spmv_mvdot(0.75, A, xv, 0.0, yv)
        assert np.array_equal(YB.get(), want), (k, ld, ofs)
        w, v = plain.astype(float), X[:, cols].astype(float)
        assert np.all(np.abs(ww - (w * w).sum(0)) <= (n + 2) * eps * (w * w).sum(0)), (k, ld, ofs)
        assert np.all(np.abs(vw - (v * w).sum(0)) <= (n + 2) * eps * np.abs(v * w).sum(0)), (k, ld, ofs)
        for o in (xv, yv, XB, YB, x, y):
            o.delete()
    A.delete()
    m.delete()
