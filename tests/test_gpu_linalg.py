"""GPU kernels against textbook references: the gather-GEMM behind every
tensordot (numpy tensordot/einsum in float64), transposes, and the SVD
(numpy's LAPACK SVD; reconstruction and orthogonality)."""
import numpy as np
import pytest

import tenes_amd as ta

pytestmark = pytest.mark.gpu

RTOL = 1e-12


def _rel(a, b):
    return np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300)


@pytest.mark.parametrize("M,N,K", [(16, 16, 4), (1, 1, 1), (5, 7, 3), (64, 64, 64), (100, 37, 250),
                                   (300, 260, 129), (1024, 1024, 64), (3, 5, 5000), (250000 // 100, 50, 25)])
def test_matmul_shapes(gpu_ctx, M, N, K):
    rng = np.random.default_rng(M * 1000 + N * 10 + K)
    A = rng.standard_normal((M, K))
    B = rng.standard_normal((K, N))
    C = ta.tensordot(gpu_ctx.tensor(A), gpu_ctx.tensor(B), [1], [0]).numpy()
    assert C.shape == (M, N)
    assert _rel(C, A @ B) < RTOL


@pytest.mark.parametrize("M,N,K", [(2500, 2500, 2500), (3500, 3500, 2000), (2100, 2100, 1024),
                                   (2000, 2300, 1500), (2500, 2500, 1100)])
def test_matmul_stream_k(gpu_ctx, M, N, K):
    """tenes_ctx_set_stream_k: row-major FP64 products whose 128 x 128 tile
    grid leaves a partial round (2500^2: 400 tiles on 512 workgroup slots)
    run stream-K: K
    iterations split evenly over 512 workgroups, split tiles summed by
    their last contributor.  Checked against numpy (1e-12 of max|C|), over
    three launches in a row (the arrival counters must come back to zero),
    bit-identical between launches (the shares are summed in rank order),
    and the launch must be the stream-K one (kernel report); (3500, 3500,
    2000) has a data-parallel round (512 tiles) before the split ones."""
    rng = np.random.default_rng(M + N + K)
    A = rng.standard_normal((M, K))
    B = rng.standard_normal((K, N))
    ref = A @ B
    ta_, tb_ = gpu_ctx.tensor(A), gpu_ctx.tensor(B)
    gpu_ctx.set_profiling(True)
    gpu_ctx.set_stream_k(True)
    try:
        first = None
        for _ in range(3):
            C = ta.tensordot(ta_, tb_, [1], [0]).numpy()
            assert _rel(C, ref) < RTOL
            if first is None:
                first = C
            else:
                assert np.array_equal(C, first)
        names = [k for k in gpu_ctx.kernel_report() if f"[{M}x{N}x{K}]" in k]
    finally:
        gpu_ctx.set_profiling(False)
        gpu_ctx.set_stream_k(False)
    assert names and all("+sk" in k for k in names), names
    # and off (the default) the same product takes the data-parallel grid
    C = ta.tensordot(ta_, tb_, [1], [0]).numpy()
    assert _rel(C, ref) < RTOL


@pytest.mark.parametrize("case", [
    # (shapeA, shapeB, axA, axB, perm)
    ((4, 5, 6), (6, 5, 3), [1, 2], [1, 0], None),
    ((7, 3, 4, 2), (2, 4, 9), [2, 3], [1, 0], [2, 0, 1]),
    ((10, 10, 5, 5), (10, 5, 5, 11), [1, 2], [0, 1], [3, 1, 0, 2]),
    ((3, 4), (5, 6), [], [], None),
    ((20, 20, 4, 4), (20, 4, 4, 20), [0, 2, 3], [0, 1, 2], [1, 0]),
    ((2, 3, 2, 3, 2), (2, 3, 2, 3, 2), [0, 1, 4], [0, 1, 4], [1, 3, 0, 2]),
])
def test_tensordot_permuted(gpu_ctx, case):
    sa, sb, axa, axb, perm = case
    rng = np.random.default_rng(len(sa) * 7 + len(sb))
    A = rng.standard_normal(sa)
    B = rng.standard_normal(sb)
    ref = np.tensordot(A, B, axes=(axa, axb))
    if perm is not None:
        ref = ref.transpose(perm)
    got = ta.tensordot(gpu_ctx.tensor(A), gpu_ctx.tensor(B), axa, axb, perm).numpy()
    assert got.shape == ref.shape
    assert _rel(got, ref) < RTOL


@pytest.mark.parametrize("M,N,K", [(16, 16, 4), (5, 7, 3), (300, 260, 129), (2500, 2500, 64), (64, 64, 5000)])
def test_matmul_fp32_compute(gpu_ctx, M, N, K):
    """The FP32-compute GEMM: inputs rounded to FP32, FP32 accumulation.
    Against the FP64 product the error is that of FP32 sums of K terms
    (bound: K * 2^-23 * sum|a||b|); its output layout is checked by the
    small shapes (a wrong row order would be an O(1) error)."""
    rng = np.random.default_rng(M + N + K)
    A = rng.standard_normal((M, K))
    B = rng.standard_normal((K, N))
    gpu_ctx.set_fp32_contractions(True)
    try:
        C = ta.tensordot(gpu_ctx.tensor(A), gpu_ctx.tensor(B), [1], [0]).numpy()
    finally:
        gpu_ctx.set_fp32_contractions(False)
    ref = A @ B
    bound = K * 2.0 ** -23 * (np.abs(A) @ np.abs(B))
    assert np.all(np.abs(C - ref) <= bound), float(np.max(np.abs(C - ref) / bound))
    A32, B32 = A.astype(np.float32).astype(np.float64), B.astype(np.float32).astype(np.float64)
    assert _rel(C, A32 @ B32) < 1e-5
    # and the FP64 path is unaffected afterwards
    C64 = ta.tensordot(gpu_ctx.tensor(A), gpu_ctx.tensor(B), [1], [0]).numpy()
    assert _rel(C64, ref) < RTOL


def _bf16(x32):
    """float32 -> nearest-even bfloat16 value, as float32 (finite inputs)."""
    b = x32.view(np.uint32).astype(np.uint64)
    r = ((b + 0x7FFF + ((b >> 16) & 1)) >> 16) << 16
    return r.astype(np.uint32).view(np.float32)


def _split_bf16(x):
    x32 = x.astype(np.float32)
    hi = _bf16(x32)
    lo = _bf16((x32 - hi).astype(np.float32))
    return hi.astype(np.float64), lo.astype(np.float64)


@pytest.mark.parametrize("M,N,K,case", [(16, 16, 32, "nn"), (5, 7, 3, "nn"), (300, 260, 129, "nn"),
                                        (300, 260, 129, "tn"), (2500, 128, 2500, "tn"),
                                        (2500, 2500, 64, "nn"), (64, 64, 5000, "tt")])
def test_matmul_split_bf16(gpu_ctx, M, N, K, case):
    """The split-precision GEMM (contraction mode 2): both operands split
    into bf16 halves x = x_hi + x_lo (x_lo = bf16(x - x_hi), from the FP32
    value), three products A_hi B_hi + A_hi B_lo + A_lo B_hi on the bf16 MFMA
    with FP32 accumulation.  Against the same three products formed in FP64
    from the same halves (numpy) the difference is FP32 accumulation only
    (K * 2^-23 * sum|a||b|); against the FP64 product the split itself adds
    ~2^-16 per product.  Operand layouts "n"/"t" (row- or column-contiguous
    contracted index) exercise both loaders; a wrong MFMA lane layout would be
    an O(1) error at every shape."""
    rng = np.random.default_rng(M + 3 * N + 7 * K)
    A = rng.standard_normal((M, K))
    B = rng.standard_normal((K, N))
    At = gpu_ctx.tensor(A.T.copy()) if case[0] == "t" else gpu_ctx.tensor(A)
    Bt = gpu_ctx.tensor(B.T.copy()) if case[1] == "t" else gpu_ctx.tensor(B)
    axa = [0] if case[0] == "t" else [1]
    axb = [1] if case[1] == "t" else [0]
    gpu_ctx.set_contraction_mode(2)
    try:
        C = ta.tensordot(At, Bt, axa, axb).numpy()
    finally:
        gpu_ctx.set_contraction_mode(0)
    Ah, Al = _split_bf16(A)
    Bh, Bl = _split_bf16(B)
    emu = Ah @ Bh + Ah @ Bl + Al @ Bh
    mag = np.abs(A) @ np.abs(B)
    assert np.all(np.abs(C - emu) <= (K + 2) * 2.0 ** -23 * mag), float(np.max(np.abs(C - emu) / mag))
    ref = A @ B
    err = np.max(np.abs(C - ref) / mag)
    assert err < 2.0 ** -14 + K * 2.0 ** -23, err
    # the FP64 path is unaffected afterwards
    C64 = ta.tensordot(At, Bt, axa, axb).numpy()
    assert _rel(C64, ref) < RTOL


def test_transpose(gpu_ctx):
    rng = np.random.default_rng(3)
    A = rng.standard_normal((3, 4, 5, 6, 2))
    for axes in [(4, 3, 2, 1, 0), (2, 3, 0, 1, 4), (1, 2, 3, 0, 4), (3, 0, 1, 2, 4)]:
        got = ta.transpose(gpu_ctx.tensor(A), axes).numpy()
        assert np.array_equal(got, A.transpose(axes))


def _check_svd(A, U, s, V, k, srel):
    s_ref = np.linalg.svd(A, compute_uv=False)[:k]
    assert np.max(np.abs(s - s_ref)) / s_ref[0] < srel
    # orthonormal columns and A V = U S on the kept triplets
    assert np.max(np.abs(U.T @ U - np.eye(k))) < 1e-10
    assert np.max(np.abs(V.T @ V - np.eye(k))) < 1e-10
    assert np.max(np.abs(A @ V - U * s)) / s[0] < 1e-10


@pytest.mark.parametrize("m,n", [(7, 7), (40, 40), (128, 128), (100, 60), (60, 100), (1, 5)])
def test_svd_direct_jacobi(gpu_ctx, m, n):
    rng = np.random.default_rng(m + 3 * n)
    A = rng.standard_normal((m, n))
    k = min(m, n)
    U, s, V = ta.svd_top(gpu_ctx.tensor(A), k)
    _check_svd(A, U.numpy(), s, V.numpy(), k, 1e-13)


@pytest.mark.parametrize("m,n", [(1000, 80), (80, 1000)])
def test_svd_qr_reduction(gpu_ctx, m, n):
    rng = np.random.default_rng(11)
    # graded columns: singular values spanning 12 decades
    Q1, _ = np.linalg.qr(rng.standard_normal((max(m, n), min(m, n))))
    Q2, _ = np.linalg.qr(rng.standard_normal((min(m, n), min(m, n))))
    sv = np.logspace(0, -12, min(m, n))
    A = (Q1 * sv) @ Q2.T
    if m < n:
        A = A.T
    k = 60
    U, s, V = ta.svd_top(gpu_ctx.tensor(A), k)
    _check_svd(A, U.numpy(), s, V.numpy(), k, 1e-13)


def test_svd_randomized_decaying(gpu_ctx):
    rng = np.random.default_rng(5)
    n = 1500
    Q1, _ = np.linalg.qr(rng.standard_normal((n, 400)))
    Q2, _ = np.linalg.qr(rng.standard_normal((n, 400)))
    sv = np.exp(-np.arange(400) / 12.0)
    A = (Q1 * sv) @ Q2.T
    k = 100
    U, s, V = ta.svd_top(gpu_ctx.tensor(A), k, power_iters=4)
    _check_svd(A, U.numpy(), s, V.numpy(), k, 1e-12)


def test_svd_rank_deficient(gpu_ctx):
    rng = np.random.default_rng(9)
    n = 600
    X = rng.standard_normal((n, 5))
    A = X @ rng.standard_normal((5, n))
    U, s, V = ta.svd_top(gpu_ctx.tensor(A), 20)
    s_ref = np.linalg.svd(A, compute_uv=False)[:20]
    assert np.max(np.abs(s[:5] - s_ref[:5])) / s_ref[0] < 1e-12
    assert np.all(s[5:] < 1e-12 * s[0])


def test_gemm_autotune():
    """tenes_ctx_set_autotune: the first contraction of a plan times every
    candidate launch shape and keeps the fastest; the tuning call and the
    tuned calls give the product to FP64 rounding (1e-12 relative), for a
    square GEMM, a long-K one (split-K candidates) and a permuted one."""
    import tenes_amd as ta

    ctx = ta.Context(0, seed=5)
    ctx.set_autotune(True)
    rng = np.random.default_rng(9)
    cases = [((600, 520), (520, 610), [1], [0]),
             ((96, 4000), (4000, 80), [1], [0]),
             ((40, 30, 50), (50, 30, 70), [1, 2], [1, 0])]
    for sa, sb, axa, axb in cases:
        A = rng.standard_normal(sa)
        B = rng.standard_normal(sb)
        ref = np.tensordot(A, B, (axa, axb))
        ta_, tb_ = ctx.tensor(A), ctx.tensor(B)
        for _ in range(3):
            C = ta.tensordot(ta_, tb_, axa, axb).numpy()
            assert np.max(np.abs(C - ref)) < 1e-12 * np.max(np.abs(ref)), (sa, sb)
    ctx.close()


def test_gemm_autotune_each_mode():
    """One plan tuned in FP64, FP32 and split bf16 in turn (1000 x 400 x 400:
    32 x 32 tiles in FP64, split K in the others): every mode keeps its own
    launch shape, and its results stay within its own bound: 1e-12, the FP32
    summation bound, and three times the 2^-16 of a dropped low x low product
    beside it."""
    ctx = ta.Context(0, seed=5)
    ctx.set_autotune(True)
    rng = np.random.default_rng(10)
    A, B = rng.standard_normal((1000, 400)), rng.standard_normal((400, 400))
    ref, mag = A @ B, np.abs(A) @ np.abs(B)
    a, b = ctx.tensor(A), ctx.tensor(B)
    fp32 = 402 * 2.0 ** -24 * mag
    for mode in (0, 1, 2, 0, 2, 1):
        ctx.set_contraction_mode(mode)
        C = ta.tensordot(a, b, [1], [0]).numpy()
        bound = (1e-12 * np.max(np.abs(ref)), fp32, fp32 + 3 * 2.0 ** -16 * mag)[mode]
        assert np.all(np.abs(C - ref) <= bound), mode
    ctx.close()


def test_autotuned_ctm_matches_oracle():
    """A CTM run with autotuning on (fresh context): energy and Sz against the
    oracle to 1e-10, as without it."""
    import tenes_amd as ta
    from oracle import ctm as O, itps, models
    from oracle.lattice import SquareLattice
    from ctm_cases import su_tensors

    Tn, ham = su_tensors("heisenberg", 3, 60)
    Tn = list(Tn)
    lat = SquareLattice(2, 2)
    p = O.PEPSParameters(CHI=20, Max_CTM_Iteration=4, CTM_Convergence_Epsilon=0.0)
    env, _, _ = O.Calc_CTM_Environment(Tn, p, lat)
    ctx = ta.Context(0, seed=6)
    ctx.set_autotune(True)
    genv = ta.Environment(ctx, 2, 2)
    genv.set_site_tensors(Tn)
    genv.calc_ctm_environment(ta.peps_parameters(CHI=20, Max_CTM_Iteration=4, CTM_Convergence_Epsilon=0.0))
    E = 0.0
    gE = 0.0
    for s, leg in models.square_bonds(lat):
        dx, dy = (1, 0) if leg == 2 else (0, 1)
        gE += genv.contract_two_sites_op12(s, dx, dy, ham) / genv.contract_cluster(s, dx, dy)
    two = [{"name": "b", "group": 0, "source": s, "dx": 1 if leg == 2 else 0, "dy": 0 if leg == 2 else 1,
            "op": ham} for s, leg in models.square_bonds(lat)]
    w, _ = itps.measure_twosite(env, Tn, lat, two, [])
    E = np.real(sum(w[0].values()))
    assert abs(gE - E) < 1e-10 * abs(E), (gE, E)
    del genv
    ctx.close()


@pytest.mark.parametrize("p", [1, 2, 15, 16, 17, 31, 48, 100, 112, 113, 127, 128])
@pytest.mark.parametrize("deficient", [False, True])
def test_tall_svd_block_edges(gpu_ctx, p, deficient):
    """CholeskyQR of a tall block at the 16-wide block edges of its
    factorisation: singular values, left basis and reconstruction against
    LAPACK; with a zero and a dependent column the range is kept and the
    dropped directions carry no weight.  Columns of lengths over six decades.
    Tolerance: three passes leave ||Q^T Q - 1|| at a few p eps = 128 * 2.2e-16,
    times ten for the products around them: 3e-13 of the largest value."""
    rng = np.random.default_rng(100 + p)
    A = rng.standard_normal((300, p)) * np.logspace(0, -6, p)
    if deficient and p >= 3:
        A[:, p // 2] = 0.0
        A[:, p - 1] = 2.0 * A[:, 0]
    U, s, V = ta.svd_top(gpu_ctx.tensor(A), p)
    U, V = U.numpy(), V.numpy()
    ref = np.linalg.svd(A, compute_uv=False)
    assert np.max(np.abs(s - ref)) < 3e-13 * ref[0]
    assert np.max(np.abs((U * s) @ V.T - A)) < 3e-13 * ref[0]
    r = p - 2 if deficient and p >= 3 else p
    assert np.max(np.abs(U[:, :r].T @ U[:, :r] - np.eye(r))) < 3e-13


@pytest.mark.parametrize("m,p", [(1, 1), (1, 5), (5, 1), (3, 2), (8, 8), (16, 16), (17, 16), (16, 17), (32, 33),
                                 (33, 32), (40, 40), (64, 64), (65, 63), (63, 65), (100, 128), (128, 100),
                                 (127, 127), (128, 128)])
@pytest.mark.parametrize("scale", [1.0, 1e-90, 1e90])
def test_jacobi_svd_slot_edges(gpu_ctx, m, p, scale):
    """The one-workgroup Jacobi SVD at the edges of its column slots (16, 32,
    64, 128) and rows per lane, with a graded spectrum, a repeated singular
    value and (from 8 columns on) a rank-deficient block, also far from
    unit scale.  Tolerance: orthogonality is iterated to sqrt(m) eps per
    pair and the factors accumulate about ten sweeps of rotations: 128 eps
    times ten, 3e-13."""
    rng = np.random.default_rng(1000 * m + p)
    k = min(m, p)
    q1, _ = np.linalg.qr(rng.standard_normal((m, k)))
    q2, _ = np.linalg.qr(rng.standard_normal((p, k)))
    s0 = np.logspace(0, -10, k)
    if k >= 3:
        s0[1] = s0[0]
    if k >= 8:
        s0[-2:] = 0.0
    A = (q1 * s0) @ q2.T * scale
    U, s, V = ta.svd_top(gpu_ctx.tensor(A), k)
    U, V = U.numpy(), V.numpy()
    ref = np.linalg.svd(A, compute_uv=False)[:k]
    assert s.shape == (k,)
    assert np.max(np.abs(s - ref)) < 3e-13 * ref[0]
    assert np.max(np.abs((U * s) @ V.T - A)) < 3e-13 * ref[0]
    assert np.max(np.abs(V.T @ V - np.eye(k))) < 3e-13
    r = k - 2 if k >= 8 else k
    assert np.max(np.abs(U[:, :r].T @ U[:, :r] - np.eye(r))) < 3e-13


@pytest.mark.parametrize("m,n,at", [(1, 1, (0, 0)), (1, 9, (0, 8)), (9, 1, (0, 0)), (9, 1, (8, 0)), (5, 7, (0, 0)),
                                    (3, 40, (2, 39)), (40, 40, (0, 3)), (128, 128, (127, 127)), (128, 70, (64, 0))])
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_exact_svd_reports_non_finite_input(gpu_ctx, m, n, at, bad):
    """One NaN or infinite entry in a matrix of the exact path, in the first
    row (the first pivot of its QR), in a row that is never a pivot and in a
    column past min(m, n): every singular value of the SVD is NaN, and a corner's
    normalised spectrum has NaN; the next matrix is not affected."""
    rng = np.random.default_rng(m + n)
    A = rng.standard_normal((m, n))
    k = min(m, n)
    good = np.linalg.svd(A, compute_uv=False)
    B = A.copy()
    B[at] = bad
    U, s, V = ta.svd_top(gpu_ctx.tensor(B), k)
    assert s.shape == (k,) and np.all(np.isnan(s))
    assert np.all(np.isnan(V.numpy()))
    env = ta.Environment(gpu_ctx, 1, 1)
    env.set("C1", 0, B)
    assert np.any(np.isnan(env.corner_spectrum("C1", 0)))
    env.set("C1", 0, A)
    assert np.max(np.abs(env.corner_spectrum("C1", 0) - good / np.linalg.norm(good))) < 3e-13


_I = np.arange(400)
_SPECTRA = {
    "exponential": np.exp(-0.2 * _I),
    "flat_exponential": np.exp(-0.1 * _I),
    "algebraic": (1.0 + _I) ** -6.0,
    "step_1e-9": np.where(_I < 10, 1.0, 1e-9) * np.exp(-0.1 * _I),
    "step_1e-5": np.where(_I < 60, 1.0, 1e-5) * np.exp(-0.1 * _I),
    "two_steps": np.where(_I < 20, 1.0, np.where(_I < 60, 1e-6, 1e-11)) * np.exp(-0.1 * _I),
    "degenerate": np.exp(-0.2 * (_I // 8 * 8)),
    "flat_rank_100": np.where(_I < 100, 1.0, 0.0),
    "rank_30": np.where(_I < 30, np.exp(-0.3 * _I), 0.0),
}


@pytest.mark.parametrize("name", sorted(_SPECTRA))
@pytest.mark.parametrize("q", [1, 2, 8])
def test_range_finder_spectra(gpu_ctx, name, q):
    """The 128-wide range finder from a Gaussian block (two shifted
    orthonormalisations in the first iteration, plain ones after) on 400 x 400
    matrices of nine kinds of spectra, against LAPACK: values, residuals of the
    triplets and orthogonality of the directions above the plain passes'
    pivot floor.  Tolerance, of the largest value: the subspace error
    (s_129 / s_k)^(2q+1) times s_k (k = 60; measured against the spectrum
    itself, times 100 for the Gaussian block's constant) and 3e-13 for the
    arithmetic (128 eps times ten)."""
    rng = np.random.default_rng(len(name) + q)
    sv, k = _SPECTRA[name], 60
    q1, _ = np.linalg.qr(rng.standard_normal((400, 400)))
    q2, _ = np.linalg.qr(rng.standard_normal((400, 400)))
    A = (q1 * sv) @ q2.T
    U, s, V = ta.svd_top(gpu_ctx.tensor(A), k, power_iters=q)
    U, V = U.numpy(), V.numpy()
    err = 100.0 * sv[k - 1] * (sv[128] / sv[k - 1]) ** (2 * q + 1) if sv[k - 1] > 0.0 else 0.0
    tol = 3e-13 + err / sv[0]
    assert np.max(np.abs(s - sv[:k])) < tol * sv[0]
    r = int(np.sum(s > 1e-12 * s[0]))
    assert r == int(np.sum(sv[:k] > 1e-12))
    assert np.max(np.abs(A @ V[:, :r] - U[:, :r] * s[:r])) < tol * sv[0]
    # exact for U in the range found: only the arithmetic
    assert np.max(np.abs(A.T @ U[:, :r] - V[:, :r] * s[:r])) < 3e-13 * sv[0]
    for X in (U, V):
        assert np.max(np.abs(X[:, :r].T @ X[:, :r] - np.eye(r))) < 3e-13


def _graded(rng, m, n, scale, decades=10):
    """m x n with singular values over `decades` decades below `scale`."""
    k = min(m, n)
    q1, _ = np.linalg.qr(rng.standard_normal((m, k)))
    q2, _ = np.linalg.qr(rng.standard_normal((n, k)))
    return (q1 * np.logspace(0, -decades, k)) @ q2.T * scale


@pytest.mark.parametrize("m,n", [(1, 1), (5, 3), (3, 5), (40, 40), (33, 64), (64, 33), (128, 128)])
@pytest.mark.parametrize("scale", [1e-290, 1e-200, 1e200, 1e290])
def test_exact_svd_scale(gpu_ctx, m, n, scale):
    """Entries whose squares overflow or vanish: the exact path is scaled by
    powers of two, so the errors relative to the largest value are those of
    test_jacobi_svd_slot_edges (3e-13)."""
    A = _graded(np.random.default_rng(m + 2 * n), m, n, scale)
    k = min(m, n)
    U, s, V = ta.svd_top(gpu_ctx.tensor(A), k)
    U, V = U.numpy(), V.numpy()
    ref = np.linalg.svd(A / scale, compute_uv=False)
    assert np.max(np.abs(s / scale - ref)) < 3e-13
    assert np.max(np.abs((U * (s / scale)) @ V.T - A / scale)) < 3e-13
    assert np.max(np.abs(V.T @ V - np.eye(k))) < 3e-13
    assert np.max(np.abs(U.T @ U - np.eye(k))) < 3e-13


@pytest.mark.parametrize("m,n", [(129, 129), (160, 130), (130, 160), (256, 256), (20, 200)])
@pytest.mark.parametrize("power", [-460, -300, -101, -99, 99, 101, 300, 460])
def test_large_corner_spectrum_scale(gpu_ctx, m, n, power):
    """Spectra of corners above 128 (the Jacobi in global memory), far from
    unit scale and on both sides of its scaling limit of 2^100.  A power of
    two changes no rounding while nothing overflows or vanishes, so the
    normalised spectrum has the bits of the unscaled matrix's.  (The host's
    normalisation squares the values: a corner stays within 2^500.)"""
    A = _graded(np.random.default_rng(m + 2 * n), m, n, 1.0)
    env = ta.Environment(gpu_ctx, 1, 1)
    env.set("C1", 0, A)
    ref = env.corner_spectrum("C1", 0)
    env.set("C1", 0, np.ldexp(A, power))
    assert np.array_equal(env.corner_spectrum("C1", 0), ref)


@pytest.mark.parametrize("m,n", [(2, 2), (5, 5), (4, 9), (9, 4), (64, 64)])
@pytest.mark.parametrize("tiny", [1e-130, 1e-145, 1e-155, 1e-157, 1e-162, 1e-200, 0.0])
def test_exact_svd_decoupled_small_entry(gpu_ctx, m, n, tiny):
    """A remainder of the QR whose squared norm is denormal or zero beside an
    entry of 1 (a decoupled index): nothing overflows in 1 / (squared norm),
    the factors stay finite and orthonormal, and 1e-130 keeps its value."""
    A = np.zeros((m, n))
    A[0, 0], A[-1, -1] = 1.0, tiny
    U, s, V = ta.svd_top(gpu_ctx.tensor(A), 2)
    U, V = U.numpy(), V.numpy()
    assert s[0] == 1.0 and 0.0 <= s[1] <= 1.001 * tiny
    if tiny == 1e-130:
        assert abs(s[1] - tiny) < 1e-12 * tiny
    assert np.all(np.isfinite(U)) and np.max(np.abs(V.T @ V - np.eye(2))) < 1e-15
    assert abs(abs(U[0, 0]) - 1.0) < 1e-15 and abs(abs(V[0, 0]) - 1.0) < 1e-15


@pytest.mark.parametrize("M,N,K", [(1, 1, 400), (31, 33, 15), (32, 32, 16), (33, 31, 17), (32, 700, 400),
                                   (700, 32, 401), (33, 33, 400), (1024, 2048, 31), (1025, 2047, 33),
                                   (2500, 128, 128), (128, 128, 400), (32, 32, 8191), (32, 32, 8192),
                                   (9, 18, 18225), (33, 32, 8200), (64, 64, 131072), (200, 130, 9000)])
@pytest.mark.parametrize("ta_, tb_", [(False, False), (True, False), (False, True), (True, True)])
def test_matmul_dispatch_edges(gpu_ctx, M, N, K, ta_, tb_):
    """Both sides of the lines between 32, 64 and 128 tiles, the unsplit, the
    split and the many-split launch, for the four operand orders, with the
    mixed-precision modes' own tile choice beside (FP32: its summation bound).
    FP64 tolerance: 1e-12 of max|C|, as the other products."""
    rng = np.random.default_rng(M * 7 + N * 3 + K)
    A = rng.standard_normal((K, M) if ta_ else (M, K))
    B = rng.standard_normal((N, K) if tb_ else (K, N))
    ref = (A.T if ta_ else A) @ (B.T if tb_ else B)
    a, b = gpu_ctx.tensor(A), gpu_ctx.tensor(B)
    axes = ([0 if ta_ else 1], [1 if tb_ else 0])
    C = ta.tensordot(a, b, *axes).numpy()
    assert _rel(C, ref) < RTOL
    C2 = ta.tensordot(a, b, *axes, [1, 0]).numpy()
    assert np.array_equal(C2, C.T)
    gpu_ctx.set_contraction_mode(1)
    try:
        F = ta.tensordot(a, b, *axes).numpy()
    finally:
        gpu_ctx.set_contraction_mode(0)
    bound = (K + 2) * 2.0 ** -24 * (np.abs(A.T if ta_ else A) @ np.abs(B.T if tb_ else B))
    assert np.all(np.abs(F - ref) <= bound + 1e-12)
