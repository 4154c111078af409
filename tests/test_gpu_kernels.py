"""GPU tests of the dense linear-algebra kernels through the C ABI."""
import ctypes

import numpy as np
import pytest
import scipy.linalg as sla
import torch

pytestmark = pytest.mark.gpu


def _lib():
    from updes_amd import _lib as L
    L.require_gpu()
    return L


@pytest.mark.parametrize("trans", [0, 1])
@pytest.mark.parametrize("m,n,lda,alpha,beta", [(1, 1, 1, 1.0, 0.0), (5, 40006, 40006, -1.0, 1.0),
                                                (7, 301, 301, 2.0, 0.5), (1000, 257, 264, 1.0, 0.0),
                                                (3001, 3001, 3008, -1.0, 1.0), (2049, 130, 131, 1.0, 0.0),
                                                (64, 129, 130, 1.0, -1.0)])
def test_gemv_matches_numpy(trans, m, n, lda, alpha, beta):
    """rbfx_gemv_f64, both orientations: the row-per-wave product and the
    transposed product over row chunks (paired 16-byte columns where lda is
    even, single columns otherwise, odd column counts, row counts that are
    not multiples of the four waves), against NumPy in FP64."""
    L = _lib()
    rng = np.random.default_rng(m + 3 * n + lda)
    A = rng.standard_normal((m, lda))
    x = rng.standard_normal(m if trans else n)
    y0 = rng.standard_normal(n if trans else m)
    dA = torch.as_tensor(A).cuda()
    dx = torch.as_tensor(x).cuda()
    dy = torch.as_tensor(y0).cuda()
    ws = L.workspace(L.lib().rbfx_gemv_workspace(trans, m, n), "cuda")
    L.check(L.lib().rbfx_gemv_f64(trans, m, n, alpha, L.ptr(dA), lda, L.ptr(dx), beta, L.ptr(dy), L.ptr(ws),
                                  ws.numel(), L.stream()))
    Am = A[:, :n]
    ref = alpha * ((Am.T @ x) if trans else (Am @ x)) + beta * y0
    got = dy.cpu().numpy()
    scale = np.abs(Am).sum(axis=0 if trans else 1).max() * np.abs(x).max() * abs(alpha) + np.abs(y0).max()
    assert np.abs(got - ref).max() <= 1e-14 * scale * max(1, (m if trans else n) ** 0.5)


@pytest.mark.parametrize("n", [1, 255, 257, 2048, 2049, 4095, 4096, 8192, 8193, 20001])
@pytest.mark.parametrize("m,beta", [(1, 0.0), (3, -0.5), (2047, 1.0)])
def test_gemv_few_long_rows(m, n, beta):
    """Product with a workgroup per row (256 threads, 1,024 from 4,096 columns,
    batches of eight and their remainders) against NumPy in FP64."""
    L = _lib()
    rng = np.random.default_rng(m + 3 * n)
    A, x, y0 = rng.standard_normal((m, n)), rng.standard_normal(n), rng.standard_normal(m)
    dA, dx = torch.as_tensor(A).cuda(), torch.as_tensor(x).cuda()
    dy = torch.as_tensor(y0 if beta else np.full(m, np.nan)).cuda()
    L.check(L.lib().rbfx_gemv_f64(0, m, n, 2.0, L.ptr(dA), n, L.ptr(dx), beta, L.ptr(dy), None, 0, L.stream()))
    ref = 2.0 * (A @ x) + (beta * y0 if beta else 0.0)
    # at most n / 256 + 16 sums in sequence on the device, NumPy's pairwise or
    # blocked ones no more than that: each within eps / 2 of the terms' magnitudes
    bound = (n / 256 + 32) * np.finfo(float).eps * (2.0 * np.abs(A) @ np.abs(x) + np.abs(beta * y0))
    assert (np.abs(dy.cpu().numpy() - ref) <= bound).all()


@pytest.mark.parametrize("m", [1, 3, 4, 31, 32, 33, 63, 64, 65])
@pytest.mark.parametrize("n,lda,beta", [(1, 1, 0.0), (63, 64, 1.0), (65, 65, 0.0), (4097, 4100, -0.5)])
def test_gemv_transposed_few_rows(m, n, lda, beta):
    """Transposed product of at most 64 rows (one kernel, a wave per fourth
    row) and of 65: against NumPy in FP64; y is not read when beta is 0, and an
    infinite last row stays infinite."""
    L = _lib()
    rng = np.random.default_rng(m + 3 * n)
    A, x, y0 = rng.standard_normal((m, lda)), rng.standard_normal(m), rng.standard_normal(n)
    A[-1, 0], x[-1] = np.inf, 1.0
    dA, dx = torch.as_tensor(A).cuda(), torch.as_tensor(x).cuda()
    dy = torch.as_tensor(y0 if beta else np.full(n, np.nan)).cuda()
    ws = L.workspace(L.lib().rbfx_gemv_workspace(1, m, n), "cuda")
    L.check(L.lib().rbfx_gemv_f64(1, m, n, -1.0, L.ptr(dA), lda, L.ptr(dx), beta, L.ptr(dy), L.ptr(ws), ws.numel(),
                                  L.stream()))
    got = dy.cpu().numpy()
    assert got[0] == -np.inf
    ref = -(A[:, 1:n].T @ x) + (beta * y0[1:] if beta else 0.0)
    # m products and m + 1 sums, each within eps / 2 of the terms' magnitudes, on both sides
    bound = (m + 2) * np.finfo(float).eps * (np.abs(A[:, 1:n]).T @ np.abs(x) + np.abs(beta * y0[1:]))
    assert (np.abs(got[1:] - ref) <= bound).all()


@pytest.mark.parametrize("m,n,lda,nrs", [(1, 1, 1, 1), (300, 257, 264, 200), (5000, 301, 301, 5000), (64, 64, 64, 0)])
def test_frobenius_norms_match_numpy(m, n, lda, nrs):
    """rbfx_frobenius_f64 (rows i < n_scaled scaled) and the one-pass pair
    (scaled, unscaled) against NumPy."""
    L = _lib()
    from updes_amd import engine as E
    rng = np.random.default_rng(m + n)
    A = rng.standard_normal((m, lda))
    rs = rng.uniform(0.5, 2.0, nrs)
    dA = torch.as_tensor(A).cuda()
    drs = torch.as_tensor(rs).cuda()
    scale = np.ones(m)
    scale[:nrs] = rs
    ref_s = np.linalg.norm(A[:, :n] * scale[:, None])
    ref = np.linalg.norm(A[:, :n])
    got_s, got = E.frobenius_pair(dA, m, n, drs)
    assert abs(got_s - ref_s) <= 1e-13 * ref_s and abs(got - ref) <= 1e-13 * ref
    assert E.frobenius(dA, m, n, drs) == got_s and E.frobenius(dA, m, n) == got


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("m,n,k,beta", [(1, 1, 1, 1.0), (130, 70, 17, 1.0), (300, 257, 64, 1.0),
                                         (512, 384, 256, 1.0), (300, 258, 64, 1.0), (130, 72, 16, 0.0),
                                         (1000, 520, 512, 1.0), (257, 8, 8, 0.0), (129, 136, 32, 1.0),
                                         (2944, 2952, 64, 1.0)])
def test_gemm_matches_torch(dtype, m, n, k, beta):
    """All GEMM paths: LDS-DMA with 128 x 128 tiles (products with at least
    2 x CU-count such tiles, the last shape) or 64 x 64 tiles (smaller FP64
    products), both needing k a multiple of the k-tile and n of 16 bytes, and
    register-staged (the rest), with partial tiles on every edge."""
    L = _lib()
    g = torch.Generator().manual_seed(m * 7 + n + k)
    A = torch.randn(m, k, generator=g, dtype=torch.float64)
    B = torch.randn(k, n, generator=g, dtype=torch.float64)
    C = torch.randn(m, n, generator=g, dtype=torch.float64)
    ref = beta * C - A @ B
    dA, dB, dC = (t.to(dtype).cuda().contiguous() for t in (A, B, C))
    fn = L.lib().rbfx_gemm_f64 if dtype == torch.float64 else L.lib().rbfx_gemm_f32
    L.check(fn(m, n, k, -1.0, L.ptr(dA), k, L.ptr(dB), n, beta, L.ptr(dC), n, L.stream()))
    torch.cuda.synchronize()
    tol = 1e-12 if dtype == torch.float64 else 2e-4
    err = (dC.double().cpu() - ref).abs().max().item() / max(1.0, ref.abs().max().item())
    assert err < tol, err


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("m,n,k", [(1, 1, 16), (65, 3, 16), (130, 63, 32), (64, 65, 64), (300, 129, 64),
                                   (2945, 2951, 32)])
def test_gemm_ragged_columns_in_padded_rows(dtype, m, n, k):
    """A column count that is not a whole number of 16-byte chunks, in rows
    that hold the last chunk: same product, and the padding behind C's rows
    stays as it was (B's padding is NaN and must not reach a result)."""
    L = _lib()
    ld = -(-n // 64) * 64
    g = torch.Generator().manual_seed(m + n + k)
    A = torch.randn(m, k, generator=g, dtype=torch.float64)
    B = torch.full((k, ld), float("nan"), dtype=torch.float64)
    B[:, :n] = torch.randn(k, n, generator=g, dtype=torch.float64)
    C = torch.randn(m, ld, generator=g, dtype=torch.float64)
    dA, dB, dC = (t.to(dtype).cuda().contiguous() for t in (A, B, C))
    pad = dC[:, n:].clone()
    ref = C[:, :n] - A @ B[:, :n]
    fn = L.lib().rbfx_gemm_f64 if dtype == torch.float64 else L.lib().rbfx_gemm_f32
    L.check(fn(m, n, k, -1.0, L.ptr(dA), k, L.ptr(dB), ld, 1.0, L.ptr(dC), ld, L.stream()))
    torch.cuda.synchronize()
    tol = 1e-12 if dtype == torch.float64 else 2e-4
    assert (dC[:, :n].double().cpu() - ref).abs().max().item() < tol * max(1.0, ref.abs().max().item())
    assert torch.equal(dC[:, n:], pad)


@pytest.mark.parametrize("alpha", [0.5, 1.0])
def test_gemm_alpha(alpha):
    """alpha = +-1 takes the LDS-DMA kernel, other values the register-staged one."""
    L = _lib()
    m, n, k = 260, 136, 64
    g = torch.Generator().manual_seed(5)
    A, B, C = (torch.randn(*sh, generator=g, dtype=torch.float64) for sh in ((m, k), (k, n), (m, n)))
    ref = C + alpha * (A @ B)
    dA, dB, dC = (t.cuda().contiguous() for t in (A, B, C))
    L.check(L.lib().rbfx_gemm_f64(m, n, k, alpha, L.ptr(dA), k, L.ptr(dB), n, 1.0, L.ptr(dC), n, L.stream()))
    torch.cuda.synchronize()
    assert (dC.cpu() - ref).abs().max().item() < 1e-12 * ref.abs().max().item()


def _random_well(n, seed):
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((n, n))
    return a


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n", [1, 7, 64, 200, 600, 1301])
def test_getrf_getrs(dtype, n):
    from updes_amd import engine as E
    _lib()
    a = _random_well(n, n)
    ld = E._ld(n)
    m = torch.zeros((n, ld), dtype=dtype)
    m[:, :n] = torch.as_tensor(a).to(dtype)
    m = m.cuda()
    lu = E.LU(m, n)
    assert lu.singular == 0
    ipiv = lu.ipiv.cpu().numpy()
    LU = lu.a[:, :n].double().cpu().numpy()
    Lm = np.tril(LU, -1) + np.eye(n)
    Um = np.triu(LU)
    pa = a.astype(np.float64 if dtype == torch.float64 else np.float32).astype(np.float64).copy()
    for i in range(n):
        p = ipiv[i]
        assert i <= p < n
        pa[[i, p]] = pa[[p, i]]
    rel = np.abs(Lm @ Um - pa).max() / np.abs(a).max()
    tol = 1e-13 * n if dtype == torch.float64 else 1e-6 * n
    assert rel < tol, rel
    assert np.abs(np.tril(LU, -1)).max() <= 1.0 + 1e-12   # partial pivoting bound
    b = np.random.default_rng(1).standard_normal(n)
    for trans in (False, True):
        x = lu.solve(torch.as_tensor(b).cuda(), trans=trans).cpu().numpy()
        aa = a if dtype == torch.float64 else a.astype(np.float32).astype(np.float64)
        res = (aa.T if trans else aa) @ x - b
        bound = (1e-11 if dtype == torch.float64 else 1e-3) * np.linalg.norm(aa, 1) * np.linalg.norm(x, 1) * max(1, n / 100)
        assert np.abs(res).max() < bound + 1e-12, (trans, np.abs(res).max(), bound)


@pytest.mark.parametrize("n", [65, 511, 513, 700, 1100, 1536])
def test_getrs_substitutes_in_ill_conditioned_blocks(n):
    """FP64 diagonal blocks whose condition estimate exceeds 1e7 are solved by
    substitution over their 64-row sub-blocks: here every block that holds one
    of the columns (one per 200) scaled by 1e-9 (the solution is compared in
    the unscaled unknowns).  Same result as SciPy's substitution with the same factors."""
    import scipy.linalg as sl
    from updes_amd import engine as E
    _lib()
    scale = np.ones(n)
    scale[::200] = 1e-9
    a = (_random_well(n, 5 * n) + 2.0 * np.sqrt(n) * np.eye(n)) * scale[None, :]
    m = torch.zeros((n, E._ld(n)), dtype=torch.float64)
    m[:, :n] = torch.as_tensor(a)
    lu = E.LU(m.cuda(), n)
    n64, n512 = -(-n // 64), -(-n // 512)
    cond = lu.dinv.cpu().numpy()[n64 * 2 * 64 ** 2 + n512 * 2 * 512 ** 2:][:2 * n512].reshape(n512, 2)
    assert cond[0, 1] > 1e7
    LU, piv = lu.a[:, :n].cpu().numpy(), lu.ipiv.cpu().numpy()
    b = np.random.default_rng(n).standard_normal(n)
    for trans in (False, True):
        rhs = b * scale if trans else b
        x = lu.solve(torch.as_tensor(rhs).cuda(), trans=trans).cpu().numpy()
        ref = sl.lu_solve((LU, piv), rhs, trans=1 if trans else 0)
        if not trans:
            x, ref = x * scale, ref * scale
        rel = np.linalg.norm(x - ref) / np.linalg.norm(ref)
        assert rel < 1e-11, (trans, rel)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n", [1, 63, 65, 511, 513, 1100])
def test_getrs_prepare_inverts_diagonal_blocks(dtype, n):
    """The 64 x 64 and 512 x 512 inverses of the diagonal blocks of L and U
    (identity past n) and their condition estimates, from the stored factors
    of a diagonally dominant matrix (blocks of condition below 10)."""
    from updes_amd import engine as E
    _lib()
    a = _random_well(n, n) + 4.0 * n * np.eye(n)
    m = torch.zeros((n, E._ld(n)), dtype=dtype)
    m[:, :n] = torch.as_tensor(a).to(dtype)
    lu = E.LU(m.cuda(), n)
    LU = lu.a[:, :n].double().cpu().numpy()
    d = lu.dinv.cpu().numpy()
    n64, n512 = -(-n // 64), -(-n // 512)
    cond = d[n64 * 2 * 64 ** 2 + n512 * 2 * 512 ** 2:][:2 * n512].reshape(n512, 2)
    off = 0
    for size, count in ((64, n64), (512, n512)):
        X = d[off:off + count * 2 * size ** 2].reshape(count, 2, size, size)
        off += count * 2 * size ** 2
        for b in range(count):
            s = slice(b * size, min(n, (b + 1) * size))
            w = s.stop - s.start
            for which, T in ((0, np.tril(LU[s, s], -1) + np.eye(w)), (1, np.triu(LU[s, s]))):
                full = np.eye(size)
                full[:w, :w] = T
                # each entry sums at most 512 products of a well-conditioned block
                assert np.abs(X[b, which] @ full - np.eye(size)).max() <= 512 * 4 * np.finfo(float).eps * 10
                if size == 512:
                    Xw = X[b, which][:w, :w]
                    ref = max(np.linalg.norm(T, p) * np.linalg.norm(Xw, p) for p in (1, np.inf))
                    assert abs(cond[b, which] - ref) <= 1e-12 * ref


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n", [511, 1301, 2100, 4099])
def test_getrs_applies_stored_factors(dtype, n):
    """The superblock sweeps apply the stored factors (FP32 ones included) in
    FP64: x matches an FP64 substitution with the same factors (SciPy) to
    near machine precision, for ragged last superblocks and empty chunks."""
    import scipy.linalg as sl
    from updes_amd import engine as E
    _lib()
    a = _random_well(n, 7 * n)
    m = torch.zeros((n, E._ld(n)), dtype=dtype)
    m[:, :n] = torch.as_tensor(a).to(dtype)
    lu = E.LU(m.cuda(), n)
    LU = lu.a[:, :n].double().cpu().numpy()
    piv = lu.ipiv.cpu().numpy()
    b = np.random.default_rng(n).standard_normal(n)
    for trans in (False, True):
        x = lu.solve(torch.as_tensor(b).cuda(), trans=trans).cpu().numpy()
        ref = sl.lu_solve((LU, piv), b, trans=1 if trans else 0)
        rel = np.linalg.norm(x - ref) / np.linalg.norm(ref)
        assert rel < 1e-11, (trans, rel)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n,groups,narrow", [(500, 1, 0), (700, 1, 0), (1301, 2, 0), (1301, 3, 0),
                                             (1301, 0, 1), (700, 1, 1), (1301, 3, 600)])
def test_getrf_multirow_leaves(dtype, n, groups, narrow):
    """Leaves with two or three rows per thread (panel launches capped to few
    workgroups) and 16-wide leaves (narrow: panels of at least that many rows;
    0 = default, none at these sizes): same pivots as LAPACK and a small
    P A - L U residual."""
    from updes_amd import engine as E
    L = _lib()
    a = _random_well(n, 11)
    ld = E._ld(n)
    m = torch.zeros((n, ld), dtype=dtype)
    m[:, :n] = torch.as_tensor(a).to(dtype)
    L.check(L.lib().rbfx_set_panel_groups(groups))
    L.check(L.lib().rbfx_set_narrow_leaf_rows(narrow))
    try:
        lu = E.LU(m.cuda(), n)
        torch.cuda.synchronize()
    finally:
        L.check(L.lib().rbfx_set_panel_groups(0))
        L.check(L.lib().rbfx_set_narrow_leaf_rows(0))
    assert lu.singular == 0
    ipiv = lu.ipiv.cpu().numpy()
    if dtype == torch.float64:
        _, piv_ref = sla.lu_factor(a)
        assert np.array_equal(ipiv, piv_ref)
    LU = lu.a[:, :n].double().cpu().numpy()
    pa = a.astype(np.float64 if dtype == torch.float64 else np.float32).astype(np.float64).copy()
    for i in range(n):
        pa[[i, ipiv[i]]] = pa[[ipiv[i], i]]
    rel = np.abs((np.tril(LU, -1) + np.eye(n)) @ np.triu(LU) - pa).max() / np.abs(a).max()
    assert rel < (1e-13 if dtype == torch.float64 else 1e-6) * n, rel


def test_getrf_f32_leaf_geometry_does_not_change_the_factors():
    """The FP32 leaves run on at most a quarter of the CUs by default (two or
    three rows per thread on tall panels); the factors and pivots are the
    same, bit for bit, as with one row per thread on up to 256 workgroups:
    every row's arithmetic is the same whichever workgroup holds it."""
    from updes_amd import engine as E
    L = _lib()
    n = 17000  # the first panels have more than 16,384 rows: two rows per thread
    g = torch.Generator().manual_seed(17)
    a = torch.randn(n, n, generator=g, dtype=torch.float32) + 4.0 * torch.eye(n, dtype=torch.float32)
    m = torch.zeros((n, E._ld(n)), dtype=torch.float32)
    m[:, :n] = a
    default = E.LU(m.cuda(), n)
    torch.cuda.synchronize()
    L.check(L.lib().rbfx_set_panel_groups(256))
    try:
        wide = E.LU(m.cuda(), n)
        torch.cuda.synchronize()
    finally:
        L.check(L.lib().rbfx_set_panel_groups(0))
    assert default.singular == 0 and wide.singular == 0
    assert torch.equal(default.ipiv, wide.ipiv)
    assert torch.equal(default.a[:, :n], wide.a[:, :n])


@pytest.mark.parametrize("n", [4096, 4097, 4161, 4608])
def test_getrf_f64_panels_at_the_recursion_limit(n):
    """FP64 panels are recursive up to n = 4096 and factored leaf by leaf
    above; last panels of 1, 65 and 512 columns.  Same pivots as LAPACK and the
    P A - L U residual of a partial-pivoting LU."""
    from updes_amd import engine as E
    _lib()
    a = _random_well(n, n)
    m = torch.zeros((n, E._ld(n)), dtype=torch.float64)
    m[:, :n] = torch.as_tensor(a)
    lu = E.LU(m.cuda(), n)
    assert lu.singular == 0
    assert np.array_equal(lu.ipiv.cpu().numpy(), sla.lu_factor(a)[1])
    LU = lu.a[:, :n]
    PA = torch.as_tensor(a).cuda()[lu.perm]
    R = (torch.tril(LU, -1) + torch.eye(n, dtype=torch.float64, device="cuda")) @ torch.triu(LU) - PA
    assert R.abs().max().item() < 1e-13 * n * np.abs(a).max()


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n", [63, 65, 256, 257, 512, 513, 768, 769, 1024, 1025])
def test_getrf_lone_leaves_match_exchanging_leaves(dtype, n):
    """Leaves of at most 768 (FP64) or 1024 (FP32) rows run in one workgroup
    that exchanges nothing.  A cap on the workgroups keeps the exchanging
    leaves: same factors and pivots, bit for bit, and LAPACK's info for an
    exactly zero column."""
    from updes_amd import engine as E
    L = _lib()
    a = _random_well(n, 3 * n)
    zero = n // 2
    for col in (None, zero):
        if col is not None:
            a[:, col] = 0.0
        m = torch.zeros((n, E._ld(n)), dtype=dtype)
        m[:, :n] = torch.as_tensor(a).to(dtype)
        lone = E.LU(m.cuda(), n)
        L.check(L.lib().rbfx_set_panel_groups(4))
        try:
            shared = E.LU(m.cuda(), n)
            torch.cuda.synchronize()
        finally:
            L.check(L.lib().rbfx_set_panel_groups(0))
        assert torch.equal(lone.ipiv, shared.ipiv)
        assert torch.equal(lone.a[:, :n], shared.a[:, :n])
        assert lone.singular == shared.singular == (0 if col is None else col + 1)
    if dtype == torch.float64:
        a = _random_well(n, 3 * n)
        m[:, :n] = torch.as_tensor(a)
        assert np.array_equal(E.LU(m.cuda(), n).ipiv.cpu().numpy(), sla.lu_factor(a)[1])


def test_getrf_matches_lapack_pivots():
    """Same pivot sequence as LAPACK getrf on a matrix without ties."""
    from updes_amd import engine as E
    _lib()
    n = 300
    a = _random_well(n, 5)
    ld = E._ld(n)
    m = torch.zeros((n, ld), dtype=torch.float64)
    m[:, :n] = torch.as_tensor(a)
    lu = E.LU(m.cuda(), n)
    lu_ref, piv_ref = sla.lu_factor(a)
    assert np.array_equal(lu.ipiv.cpu().numpy(), piv_ref)
    assert np.abs(lu.a[:, :n].cpu().numpy() - lu_ref).max() < 1e-10


def test_getrf_pivot_ties_take_the_lowest_row():
    """The pivot rule in its documented form: partial pivoting on |value|
    with the 20 low mantissa bits of FP64 values cleared, ties to the lowest
    row.  An exact tie and a near-tie (relative difference 2^-40, which
    LAPACK resolves to the larger value) both go to the lower row; the
    factorisation stays backward stable."""
    from updes_amd import engine as E
    _lib()
    n = 300
    for near in (False, True):
        a = _random_well(n, 17)
        a[:, 0] *= 0.4 / np.abs(a[:, 0]).max()
        a[3, 0] = 1.0
        a[5, 0] = 1.0 + (2.0 ** -40 if near else 0.0)
        m = torch.zeros((n, E._ld(n)), dtype=torch.float64)
        m[:, :n] = torch.as_tensor(a)
        lu = E.LU(m.cuda(), n)
        ipiv = lu.ipiv.cpu().numpy()
        assert ipiv[0] == 3, (near, ipiv[0])
        assert sla.lu_factor(a)[1][0] == (5 if near else 3)
        LU = lu.a[:, :n].cpu().numpy()
        Lm = np.tril(LU, -1) + np.eye(n)
        pa = a.copy()
        for i in range(n):
            pa[[i, ipiv[i]]] = pa[[ipiv[i], i]]
        assert np.abs(Lm @ np.triu(LU) - pa).max() < 1e-13 * n * np.abs(a).max()


def test_expired_sweep_wait_fails_fast_and_the_next_solve_recovers():
    """Failure handling of the triangular sweeps, forced from the host: with a
    wait bound of 0 the waits that are not satisfied at once expire, the
    solve's kernels exit, NaN is written, and LU.solve raises RbfxError
    (RBFX_ERR_TIMEOUT) within seconds.  With the default bound restored the
    same factors solve normally (each solve clears its status word)."""
    import time
    from updes_amd import engine as E
    L = _lib()
    lib = L.lib()
    n = 20000
    a = _random_well(n, 11)
    m = torch.zeros((n, E._ld(n)), dtype=torch.float32)
    m[:, :n] = torch.as_tensor(a, dtype=torch.float32)
    lu = E.LU(m.cuda(), n)
    b = torch.as_tensor(np.random.default_rng(3).standard_normal(n), device="cuda")
    L.check(lib.rbfx_set_wait_seconds(0.0))
    try:
        t0 = time.perf_counter()
        with pytest.raises(L.RbfxError) as ei:
            lu.solve(b)
        assert ei.value.status == L.RBFX_ERR_TIMEOUT
        assert time.perf_counter() - t0 < 10.0
    finally:
        L.check(lib.rbfx_set_wait_seconds(-1.0))
    x = lu.solve(b).cpu().numpy()
    aa = a.astype(np.float32).astype(np.float64)
    res = aa @ x - b.cpu().numpy()
    assert np.isfinite(x).all()
    assert np.abs(res).max() < 1e-3 * np.linalg.norm(aa, 1) * np.linalg.norm(x, 1) * n / 100


def _guarded_getrf(a, dtype, wait=None):
    """info, pivots and whether the memory around the matrix is untouched, of
    a factorisation inside a larger allocation, with garbage in the workspace
    and in the pivots before the call."""
    from updes_amd import engine as E
    L = _lib()
    n = a.shape[0]
    ld = E._ld(n)
    pad = 640 * ld                        # more rows than a panel's interchanges could reach
    flat = torch.full((pad + n * ld + pad,), 12345.0, dtype=dtype, device="cuda")
    m = flat[pad:pad + n * ld].view(n, ld)
    m[:, :n] = torch.as_tensor(a).to(dtype).cuda()
    ipiv = torch.full((n,), 1 << 40, dtype=torch.int64, device="cuda")
    info = torch.full((1,), 77, dtype=torch.int32, device="cuda")
    nbytes = 8 if dtype == torch.float64 else 4
    ws = L.workspace(L.lib().rbfx_getrf_workspace(n, nbytes), "cuda").fill_(0x7f)
    fn = L.lib().rbfx_getrf_f64 if nbytes == 8 else L.lib().rbfx_getrf_f32
    if wait is not None:
        L.check(L.lib().rbfx_set_wait_seconds(wait))
    try:
        L.check(fn(n, L.ptr(m), ld, L.ptr(ipiv), L.ptr(ws), ws.numel(), L.ptr(info), L.stream()))
        torch.cuda.synchronize()
    finally:
        if wait is not None:
            L.check(L.lib().rbfx_set_wait_seconds(-1.0))
    around = bool((flat[:pad] == 12345.0).all()) and bool((flat[pad + n * ld:] == 12345.0).all())
    return int(info.item()), ipiv.cpu().numpy(), around


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("n", [65, 300, 603, 1100, 4200])
@pytest.mark.parametrize("where", ["row", "first column", "late column"])
def test_getrf_of_a_non_finite_matrix_stays_inside_it(dtype, n, where):
    """A leaf without a finite candidate stops early: the factorisation reports
    info = -1 (RbfxError in Python), its interchanges stay inside the matrix
    (memory around it unchanged) and the pivots are well formed.  A NaN row
    loses every pivot until the last column; one panel and several, recursive
    and leaf-by-leaf panels, leaves of one workgroup and of many."""
    from updes_amd import engine as E
    L = _lib()
    a = _random_well(n, 3 * n)
    if where == "row":
        a[n // 3] = np.nan
    else:
        a[:, 0 if where == "first column" else n - n // 4] = np.nan
    info, ipiv, around = _guarded_getrf(a, dtype)
    assert info == -1
    assert around
    assert (ipiv >= np.arange(n)).all() and (ipiv < n).all()
    m = torch.zeros((n, E._ld(n)), dtype=dtype)
    m[:, :n] = torch.as_tensor(a).to(dtype)
    with pytest.raises(L.RbfxError):
        E.LU(m.cuda(), n)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_getrf_whose_waits_expire_stays_inside_the_matrix(dtype):
    """With a wait bound of 0 a leaf of several workgroups gives up wherever a
    record is not there at once: every kernel still ends, the memory around the matrix
    is unchanged, and info and the pivots are well formed."""
    n = 2100
    info, ipiv, around = _guarded_getrf(_random_well(n, 1), dtype, wait=0.0)
    assert info in (0, -1)
    assert around
    assert (ipiv >= np.arange(n)).all() and (ipiv < n).all()


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("groups", [0, 6])
def test_getrf_panel_solves_round_once(dtype, groups):
    """The inverse X of a panel's unit-lower block L11 and the solves with its
    64 x 64 diagonal blocks are formed in FP64 and rounded once.  L11 itself
    stands in the matrix (unit diagonal, smaller entries below: no row moves
    and the elimination is exact), beside identity columns, where U then shows
    X (a product with the identity is exact) or, inside the panel, the solve."""
    from updes_amd import engine as E
    L = _lib()
    n, half = 1100, 2.0 ** (-53 if dtype == torch.float64 else -24)
    rng = np.random.default_rng(5)
    low = np.tril(rng.uniform(-0.25, 0.25, (512, 512)).astype(np.float32).astype(np.float64), -1) + np.eye(512)
    for inside in (False, True):
        a = np.eye(n)
        if inside:
            a[:64, :64] = low[:64, :64]
            a[:64, 64:128] = np.eye(64)
        else:
            a[:512, :512] = low
            a[:512, 512:1024] = np.eye(512)
        m = torch.zeros((n, E._ld(n)), dtype=dtype)
        m[:, :n] = torch.as_tensor(a).to(dtype)
        L.check(L.lib().rbfx_set_panel_groups(groups))
        try:
            lu = E.LU(m.cuda(), n)
        finally:
            L.check(L.lib().rbfx_set_panel_groups(0))
        assert np.array_equal(lu.ipiv.cpu().numpy(), np.arange(n))
        got = lu.a[:, :n].double().cpu().numpy()
        T = low[:64, :64] if inside else low
        w = len(T)
        assert np.array_equal(np.tril(got[:w, :w], -1) + np.eye(w), T)
        got = got[:w, 64:128] if inside else got[:w, 512:1024]
        X = sla.solve_triangular(T, np.eye(w), lower=True, unit_diagonal=True)
        # FP64 arithmetic: at most 512 terms per entry, forward error through |X| |L| |X|
        noise = 512 * 2.0 ** -53 * (np.abs(X) @ np.abs(T) @ np.abs(X))
        bound = half * np.abs(X) + noise
        for b in range(0, w, 64):          # rows below use the rounded rows above
            r = slice(b, b + 64)
            D = sla.solve_triangular(T[r, r], np.eye(64), lower=True, unit_diagonal=True)
            bound[r, :b] += np.abs(D) @ (np.abs(T[r, :b]) @ bound[:b, :b])
        assert (np.abs(got - X) <= bound).all(), (inside, np.max(np.abs(got - X) / np.maximum(bound, 1e-300)))


@pytest.mark.parametrize("m", [1, 5, 64])
@pytest.mark.parametrize("n", [131071, 131072, 131073, 300001])
def test_gemv_transposed_few_long_rows(m, n):
    """Transposed product of few rows on both sides of 131,072 columns (one
    kernel; chunks and their sum) against NumPy in FP64."""
    L = _lib()
    rng = np.random.default_rng(m + n)
    A, x, y0 = rng.standard_normal((m, n)), rng.standard_normal(m), rng.standard_normal(n)
    dA, dx, dy = (torch.as_tensor(v).cuda() for v in (A, x, y0))
    ws = L.workspace(L.lib().rbfx_gemv_workspace(1, m, n), "cuda")
    L.check(L.lib().rbfx_gemv_f64(1, m, n, -1.0, L.ptr(dA), n, L.ptr(dx), 0.5, L.ptr(dy), L.ptr(ws), ws.numel(),
                                  L.stream()))
    ref = -(A.T @ x) + 0.5 * y0
    # m products and m + 1 sums, each within eps / 2 of the terms' magnitudes, on both sides
    bound = (m + 2) * np.finfo(float).eps * (np.abs(A).T @ np.abs(x) + np.abs(0.5 * y0))
    assert (np.abs(dy.cpu().numpy() - ref) <= bound).all()


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("at,value", [(0, -1), (99, 98), (299, 300)])
def test_getrs_prepare_refuses_pivots_before_any_work(dtype, at, value):
    """An invalid pivot is refused with nothing queued: the inverses' buffer
    and the permutation stay as they were."""
    from updes_amd import engine as E
    L = _lib()
    n = 300
    m = torch.eye(n, E._ld(n), dtype=dtype, device="cuda")
    ipiv = torch.arange(n, device="cuda")
    ipiv[at] = value
    perm = torch.full((n,), -7, dtype=torch.int64, device="cuda")
    dinv = torch.full((L.lib().rbfx_getrs_dinv_elems(n),), 3.5, dtype=torch.float64, device="cuda")
    fn = L.lib().rbfx_getrs_prepare_f64 if dtype == torch.float64 else L.lib().rbfx_getrs_prepare_f32
    st = fn(n, L.ptr(m), E._ld(n), L.ptr(ipiv), L.ptr(perm), L.ptr(dinv), None, 0, L.stream())
    assert st != 0 and b"invalid pivot" in L.lib().rbfx_last_error()
    torch.cuda.synchronize()
    assert bool((dinv == 3.5).all()) and bool((perm == -7).all())
