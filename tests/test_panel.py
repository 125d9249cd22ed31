"""Register-resident LU panel (bfa_panel.hip) at the sizes where its workgroup
shape changes: one row, the edges of a 256-column panel, the first size of each
rows-a-workgroup variant, and the largest matrix that takes it whole (4,096 rows
in complex128, 6,144 in complex64: every workgroup full)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")


def _load():
    import __graft_entry__ as ge
    return ge._load_pkg()


def _factor(bfa, A, f64):
    """LU of the matrix whose column-major storage is A (A[c, r] = M(r, c))."""
    n = len(A)
    piv = torch.zeros(n, dtype=torch.int32, device="cuda")
    info = (bfa.lu_factor if f64 else bfa.lu_factor_c)(A, n, piv)
    return info, piv.cpu().numpy()


@pytest.mark.gpu
@pytest.mark.parametrize("f64", [True, False])
@pytest.mark.parametrize("n", [1, 2, 65, 255, 257, 600, 1025, 2049, 3073, 4097])
def test_panel_backward_error_and_pivots(n, f64):
    bfa = _load()
    rng = np.random.default_rng(n)
    dt = np.complex128 if f64 else np.complex64
    M = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))).astype(dt)
    A = torch.from_numpy(np.ascontiguousarray(M.T)).cuda()
    info, piv = _factor(bfa, A, f64)
    assert info == 0
    LU = A.T.to(torch.complex128)
    L = torch.tril(LU, -1) + torch.eye(n, dtype=LU.dtype, device="cuda")
    U = torch.triu(LU)
    perm = np.arange(n)
    for i, p in enumerate(piv):
        assert i <= p < n
        perm[[i, p]] = perm[[p, i]]
    PA = torch.from_numpy(M[perm].astype(np.complex128)).cuda()
    # |PA - LU| <= gamma_n |L||U| entry by entry, gamma_n = n sqrt(8) u for complex arithmetic; in norms
    u = np.finfo(np.float64 if f64 else np.float32).eps / 2
    bound = n * np.sqrt(8.0) * u * torch.linalg.norm(L.abs() @ U.abs())
    assert torch.linalg.norm(PA - L @ U) <= bound
    # partial pivoting: no multiplier is larger than its pivot in |re| + |im| (izamax's norm): |l| <= sqrt(2),
    # and the float rounding of the compared magnitudes
    assert L.abs().max() <= np.sqrt(2.0) * (1 + 1e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [40, 300])
def test_panel_equals_lapack_pivots_and_ties(n):
    """The first of equal magnitudes wins, as izamax chooses it; a permuted identity needs every interchange."""
    bfa = _load()
    import scipy.linalg as sl
    rng = np.random.default_rng(3)
    P = np.eye(n)[rng.permutation(n)].astype(np.complex128)
    S = rng.choice([1.0, -1.0, 1j, -1j], (n, n)) + 4.0 * P      # many equal magnitudes
    for M in (P, S):
        A = torch.from_numpy(np.ascontiguousarray(M.T)).cuda()
        info, piv = _factor(bfa, A, True)
        assert info == 0
        ref = sl.lu_factor(M)[1]
        same = piv == ref
        # rounding decides ties after the first steps in S; the permutation has none
        assert same.all() if M is P else same[0]


@pytest.mark.gpu
def test_panel_zero_column_reports_info():
    bfa = _load()
    n = 300
    rng = np.random.default_rng(5)
    M = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
    M[:, 270] = 0.0
    A = torch.from_numpy(np.ascontiguousarray(M.T)).cuda()
    info, piv = _factor(bfa, A, True)
    assert info == 271
    assert bool(torch.isfinite(torch.view_as_real(A)).all())


@pytest.mark.gpu
@pytest.mark.parametrize("f64,n", [(True, 256), (True, 320), (False, 256), (False, 320), (False, 700), (False, 1100)])
def test_panel_factor_error_without_interchanges(n, f64):
    """Diagonally dominant: |PA - LU| stays a few units of |A| however many
    columns a panel has, because products are summed before they are
    subtracted.  The norm is the diagonal's: its entries are rounded once per
    XP_FOLD = 32 columns of their panel (8 at most), three times on the way out
    and once per panel before, each by u / 2 to u; in quadrature under 3 u for
    n up to 1,100 (1.3 measured).  One rounding a column instead gives
    sqrt(256 / 3) u = 9 u (6.5 to 7 measured)."""
    bfa = _load()
    rng = np.random.default_rng(n)
    M = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n)) + 4 * n * np.eye(n)
    M = M.astype(np.complex128 if f64 else np.complex64)
    A = torch.from_numpy(np.ascontiguousarray(M.T)).cuda()
    info, piv = _factor(bfa, A, f64)
    assert info == 0 and (piv == np.arange(n)).all()
    if f64:     # the product in extended precision
        LU = A.T.cpu().numpy().astype(np.clongdouble)
        E = M.astype(np.clongdouble) - (np.tril(LU, -1) + np.eye(n)) @ np.triu(LU)
        err = float(np.sqrt((np.abs(E) ** 2).sum()) / np.sqrt((np.abs(M) ** 2).sum()))
    else:
        LU = A.T.to(torch.complex128)
        L = torch.tril(LU, -1) + torch.eye(n, dtype=LU.dtype, device="cuda")
        MM = torch.from_numpy(M.astype(np.complex128)).cuda()
        err = (torch.linalg.norm(MM - L @ torch.triu(LU)) / torch.linalg.norm(MM)).item()
    u = np.finfo(np.float64 if f64 else np.float32).eps / 2
    assert err <= 3 * u


@pytest.mark.gpu
def test_panel_factor_error_with_interchanges():
    """Random matrices, where sums and entries are of one size: |PA - LU| as in
    plain elimination that rounds each complex product before it subtracts it
    (ratio 1.04; 1.17 with both roundings of a product at the sum's size)."""
    bfa = _load()
    n, got, ref = 200, [], []

    def error(M, LU, perm):
        LU = LU.astype(np.clongdouble)
        E = M[perm].astype(np.clongdouble) - (np.tril(LU, -1) + np.eye(n)) @ np.triu(LU)
        return float(np.sqrt((np.abs(E) ** 2).sum())) / np.linalg.norm(M)

    for seed in range(3):
        rng = np.random.default_rng(100 * n + seed)
        M = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
        A = torch.from_numpy(np.ascontiguousarray(M.T)).cuda()
        info, piv = _factor(bfa, A, True)
        assert info == 0
        perm, LU, rows = np.arange(n), M.copy(), np.arange(n)
        for j, p in enumerate(piv):
            perm[[j, p]] = perm[[p, j]]
            q = j + np.argmax(np.abs(LU[j:, j].real) + np.abs(LU[j:, j].imag))
            LU[[j, q]], rows[[j, q]] = LU[[q, j]], rows[[q, j]]
            LU[j + 1:, j] /= LU[j, j]
            LU[j + 1:, j + 1:] -= np.outer(LU[j + 1:, j], LU[j, j + 1:])
        got.append(error(M, A.T.cpu().numpy(), perm))
        ref.append(error(M, LU, rows))
    # the mean of three knows the ratio to 1 %
    assert np.mean(got) <= 1.1 * np.mean(ref)


@pytest.mark.gpu
def test_panel_multiplier_is_as_exact_as_division():
    """l = a / p by the pivot's inverse: against the same formula in float with
    IEEE divisions, |p|^2 without and the product with fused multiply-adds
    (which of them the compiler fuses is its choice)."""
    bfa = _load()
    rng = np.random.default_rng(1)
    f = np.float32
    got, ref = [], []
    for _ in range(600):
        M = (rng.standard_normal((2, 2)) + 1j * rng.standard_normal((2, 2))) * np.exp(rng.uniform(-3, 3))
        M[0] *= 3
        M = M.astype(np.complex64)
        A = torch.from_numpy(np.ascontiguousarray(M.T)).cuda()
        info, piv = _factor(bfa, A, False)
        assert info == 0
        a, p = (M[1, 0], M[0, 0]) if piv[0] == 0 else (M[0, 0], M[1, 0])
        # float products are exact in double: one rounding each
        d = f(f(p.real * p.real) + f(p.imag * p.imag))
        v = [np.float64(f(p.real / d)), np.float64(f(-p.imag / d))]
        ar, ai = np.float64(a.real), np.float64(a.imag)
        want = complex(f(ar * v[0] - f(ai * v[1])), f(ar * v[1] + f(ai * v[0])))
        exact = complex(a) / complex(p)
        got.append(abs(complex(A.cpu().numpy()[0, 1]) - exact) / abs(exact))
        ref.append(abs(want - exact) / abs(exact))
    rms = lambda e: np.sqrt(np.mean(np.square(e)))
    # 0.84 u against 0.87 u on the same samples; 0.94 u with products by an inverse rounded once more
    assert rms(got) <= rms(ref)


@pytest.mark.parametrize("f64", [0, 1])
def test_panel_workgroups_run_at_once(f64):
    """The variant of a panel: fewest rows whose workgroups, which wait for each
    other, all fit -- 128 of them, and what the CUs hold."""
    import ctypes
    lib = _load().lib()
    variants = [8, 16, 24, 32] if f64 else [8, 16, 32, 48]
    for cus in (1, 4, 16, 32, 64, 128, 256):
        for per in ([4, 2, 1, 1], [7, 4, 2, 1], [1, 1, 1, 1], [1, 1, 0, 0], [0, 0, 0, 0]):
            arr = (ctypes.c_int * 4)(*per)
            for m in (1, 8, 9, 255, 256, 270, 1024, 1025, 2048, 2049, 3072, 3073, 4096, 4097, 6144, 6145):
                rows = lib.bfa_xpanel_rows(f64, m, cus, arr)
                fits = [r for r, p in zip(variants, per) if -(-m // r) <= min(128, p * cus)]
                assert rows == (fits[0] if fits else 0)


def _masked_stream(hip):
    import ctypes
    h = ctypes.c_void_p()
    mask = (ctypes.c_uint32 * 8)(0xFFFFFFFF)
    assert hip.hipExtStreamCreateWithCUMask(ctypes.byref(h), 8, mask) == 0
    return h, torch.cuda.ExternalStream(h.value)


@pytest.mark.gpu
@pytest.mark.parametrize("f64", [True, False])
def test_panel_on_a_stream_with_part_of_the_cus(f64):
    """A caller's stream that owns 32 CUs: 1,350 rows would take 85 workgroups."""
    import ctypes
    bfa = _load()
    torch.zeros(1, device="cuda")
    hip = ctypes.CDLL("libamdhip64.so")
    h, st = _masked_stream(hip)
    n = 1350
    rng = np.random.default_rng(2)
    M = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))).astype(np.complex128 if f64 else np.complex64)
    A = torch.from_numpy(np.ascontiguousarray(M.T)).cuda()
    piv = torch.zeros(n, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    assert (bfa.lu_factor if f64 else bfa.lu_factor_c)(A, n, piv, stream=st) == 0
    torch.cuda.synchronize()
    _check_factors(M, A, piv.cpu().numpy(), f64)
    assert hip.hipStreamDestroy(h) == 0


def _check_factors(M, A, piv, f64):
    n = len(M)
    LU = A.T.to(torch.complex128)
    L = torch.tril(LU, -1) + torch.eye(n, dtype=LU.dtype, device="cuda")
    U = torch.triu(LU)
    perm = np.arange(n)
    for i, p in enumerate(piv):
        assert i <= p < n
        perm[[i, p]] = perm[[p, i]]
    PA = torch.from_numpy(M[perm].astype(np.complex128)).cuda()
    # |PA - LU| <= gamma_n |L||U| entry by entry, gamma_n = n sqrt(8) u for complex arithmetic; in norms
    u = np.finfo(np.float64 if f64 else np.float32).eps / 2
    bound = n * np.sqrt(8.0) * u * torch.linalg.norm(L.abs() @ U.abs())
    assert torch.linalg.norm(PA - L @ U) <= bound
    # partial pivoting: no multiplier is larger than its pivot in |re| + |im| (izamax's norm): |l| <= sqrt(2),
    # and the float rounding of the compared magnitudes
    assert L.abs().max() <= np.sqrt(2.0) * (1 + 1e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("n,f64", [(4096, True), (6144, False)])
def test_panel_every_workgroup_full(n, f64):
    bfa = _load()
    rng = np.random.default_rng(n)
    M = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))).astype(np.complex128 if f64 else np.complex64)
    A = torch.from_numpy(np.ascontiguousarray(M.T)).cuda()
    info, piv = _factor(bfa, A, f64)
    assert info == 0
    _check_factors(M, A, piv, f64)


@pytest.mark.gpu
@pytest.mark.parametrize("f64", [True, False])
@pytest.mark.parametrize("n,lda", [(300, 301), (513, 1000)])
def test_panel_leading_dimension(n, lda, f64):
    """Columns further apart than their length: nothing between them is touched."""
    bfa = _load()
    rng = np.random.default_rng(lda)
    M = (rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))).astype(np.complex128 if f64 else np.complex64)
    A = torch.full((n, lda), 7 - 3j, dtype=torch.complex128 if f64 else torch.complex64, device="cuda")
    A[:, :n] = torch.from_numpy(np.ascontiguousarray(M.T)).cuda()
    piv = torch.zeros(n, dtype=torch.int32, device="cuda")
    assert (bfa.lu_factor if f64 else bfa.lu_factor_c)(A, n, piv, lda=lda) == 0
    _check_factors(M, A[:, :n], piv.cpu().numpy(), f64)
    assert (A[:, n:] == 7 - 3j).all()


@pytest.mark.gpu
def test_panel_sequence_numbers_restart():
    """The exchange's 24-bit sequence numbers run out within a factorisation:
    they begin again at 1, and words of the first use of these numbers are gone."""
    import ctypes
    bfa = _load()
    lib = bfa.lib()
    lib.bfa_xpanel_seq.restype = ctypes.c_uint
    for k, n in enumerate((600, 520, 700, 600)):
        rng = np.random.default_rng(k)
        M = rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n))
        A = torch.from_numpy(np.ascontiguousarray(M.T)).cuda()
        if k == 1:
            lib.bfa_xpanel_seq((1 << 24) - 300)
        info, piv = _factor(bfa, A, True)
        assert info == 0
        _check_factors(M, A, piv, True)
        if k == 1:
            assert 1 < lib.bfa_xpanel_seq(0) < 1000


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["nan", "inf", "column", "underflow"])
@pytest.mark.parametrize("path", ["registers", "lds", "tall", "local"])
def test_lu_of_values_that_are_not_numbers(path, kind):
    """NaN in a matrix (a permittivity of exactly 1 puts it there), infinities,
    and entries whose squares underflow in complex64: every panel still chooses
    rows of its own, the factors carry the NaN on, and the solve ends."""
    import ctypes
    bfa = _load()
    n = 6400 if path == "tall" else 300
    g = torch.Generator(device="cuda").manual_seed(n)
    M = torch.complex(*[torch.randn(n, n, generator=g, device="cuda") for _ in range(2)])
    if kind == "nan":
        M.fill_(complex("nan"))
    elif kind == "inf":
        M[3, 5] = float("inf")
    elif kind == "column":
        M[17] = complex("nan")
    else:
        M *= 1e-30
    piv = torch.full((n,), -7, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    factor = bfa.lu_factor_c_local if path == "local" else bfa.lu_factor_c
    if path == "lds":
        hip = ctypes.CDLL("libamdhip64.so")
        h, st = _masked_stream(hip)
        factor(M, n, piv, stream=st)
        torch.cuda.synchronize()
        assert hip.hipStreamDestroy(h) == 0
    else:
        factor(M, n, piv)
    p = piv.cpu().numpy()
    assert ((p >= np.arange(n)) & (p < n)).all()
    assert not bool(torch.isfinite(torch.view_as_real(M)).all())
    B = torch.ones((2, n), dtype=torch.complex64, device="cuda")
    bfa.lu_solve_c(M, n, piv, B, 2)
    torch.cuda.synchronize()
    assert not bool(torch.isfinite(torch.view_as_real(B)).all())
