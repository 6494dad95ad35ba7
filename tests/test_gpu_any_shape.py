"""MTTKRP of unaligned shapes, ranks above 64 and float64 on the matrix cores,
at the edges of its tiles: 16 rows, 64 / 32 columns, 32 / 16 contiguous
values, rank tiles of 16 and slabs of 64.  Reference: FP64 torch on the same
inputs.

Tolerances (relative, Frobenius): each term is a product of up to five
rounded values, and the partial sums of q terms of random sign are about
sqrt(q) terms large, so their roundings add up to about sqrt(q) eps of the
result in one chain.  The chains here have at most 4,900 terms: 70 eps, halved
because the partial sums grow to that size only at the end: 32 eps, 2e-6 for
float32 and 4e-15 for float64."""
import warnings

import pytest
import torch

import any_shape_cases

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 2e-6, torch.float64: 4e-15}


def reference(X, w, F, mode):
    k = None
    for i, f in enumerate(F):
        if i != mode:
            f = f.double()
            k = f if k is None else (k[:, None, :] * f[None, :, :]).reshape(-1, f.shape[1])
    if w is not None and len(F) > 2:  # khatri_rao of one matrix ignores the weights
        k = k * w.double()
    return torch.movedim(X.double(), mode, 0).reshape(X.shape[mode], -1) @ k


def problem(cuda, shape, rank, dtype, seed):
    g = torch.Generator(device=cuda).manual_seed(seed)
    X = torch.randn(shape, generator=g, device=cuda, dtype=dtype)
    F = [torch.randn((s, rank), generator=g, device=cuda, dtype=dtype) for s in shape]
    w = torch.rand(rank, generator=g, device=cuda, dtype=dtype) + 0.5
    return X, F, w


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("rank", [1, 16, 17, 33, 64, 65, 130])
@pytest.mark.parametrize("shape", [(7, 9), (33, 4), (17, 3), (15, 16, 17), (16, 5, 33), (300, 7, 9), (65, 66, 67),
                                   (3, 2, 130), (130, 3, 4), (5, 6, 7, 8), (12, 10, 8, 31), (4, 3, 2, 3, 5)])
def test_mttkrp_any_shape(cuda, shape, rank, dtype):
    import tensorly_amd as tla
    X, F, w = problem(cuda, shape, rank, dtype, sum(shape) + rank)
    for mode in range(len(shape)):
        for weights in (None, w):
            out = tla.unfolding_dot_khatri_rao(X, (weights, F), mode)
            ref = reference(X, weights, F, mode)
            assert out.dtype == dtype and out.shape == ref.shape
            err = float(torch.linalg.vector_norm(out.double() - ref) / torch.linalg.vector_norm(ref))
            assert err < TOL[dtype], (mode, err)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("shape", [(19, 21, 35), (6, 5, 11, 37)])
def test_mttkrp_any_shape_infinities_stay_in_their_rows(cuda, shape, dtype):
    """Padded rows, columns and rank columns must not carry an infinity or a
    NaN into an output that does not depend on it."""
    import tensorly_amd as tla
    X, F, w = problem(cuda, shape, 5, dtype, 3)
    F = [f.abs() + 0.1 for f in F]
    for where, value in ((tuple(s - 1 for s in shape), float("inf")), (tuple(0 for _ in shape), float("nan")),
                         (tuple(s // 2 for s in shape), float("-inf"))):
        Y = X.clone()
        Y[where] = value
        for mode in range(len(shape)):
            out = tla.unfolding_dot_khatri_rao(Y, (w, F), mode)
            hit = torch.zeros(shape[mode], dtype=torch.bool, device=cuda)
            hit[where[mode]] = True
            assert bool(torch.isfinite(out[~hit]).all()), (where, mode)
            bad = out[hit]
            assert bool(torch.isnan(bad).all() if value != value else (bad == value).all()), (where, mode)


def test_mttkrp_any_shape_without_scratch(cuda):
    """A caller that brings no scratch gets the same result (to rounding)."""
    from tensorly_amd import _lib
    X, F, w = problem(cuda, (37, 41, 43), 9, torch.float32, 11)
    sh, _k = _lib.shape_array(X.shape)
    pp, _kf = _lib.ptr_array(F)
    for mode in range(3):
        out = torch.empty((X.shape[mode], 9), device=cuda)
        _lib.check(_lib.lib().tla_mttkrp(_lib.F32, _lib.ptr(X), 3, sh, pp, _lib.ptr(w), 9, mode, _lib.PREC_FP32,
                                         _lib.ptr(out), None, 0, _lib.stream(cuda)))
        ref = reference(X, w, F, mode)
        assert float(torch.linalg.vector_norm(out.double() - ref) / torch.linalg.vector_norm(ref)) < TOL[torch.float32]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("J", [1, 16, 17, 64, 65, 200])
@pytest.mark.parametrize("shape", [(9,), (33, 4), (17, 19, 23), (3, 2, 130), (65, 66, 67), (300, 5, 9), (4, 3, 2),
                                   (2, 70, 129), (4, 3, 2, 5)])
def test_mode_dot_any_shape(cuda, shape, J, dtype):
    """The tiles of the n-mode product: 16 or 64 rows, 64 / 32 columns, 16 rows
    of the matrix per tile and 64 per block; sums of at most 300 terms, so the
    tolerance above holds with room."""
    import tensorly_amd as tla
    g = torch.Generator(device=cuda).manual_seed(sum(shape) + J)
    X = torch.randn(shape, generator=g, device=cuda, dtype=dtype)
    for mode in range(len(shape)):
        for transpose in (False, True):
            U = torch.randn((shape[mode], J) if transpose else (J, shape[mode]), generator=g, device=cuda, dtype=dtype)
            out = tla.mode_dot(X, U, mode, transpose=transpose)
            A = (U.T if transpose else U).double()
            ref = torch.movedim(torch.tensordot(A, X.double(), dims=([1], [mode])), 0, mode)
            assert out.dtype == dtype and out.shape == ref.shape
            err = float(torch.linalg.vector_norm(out.double() - ref) / torch.linalg.vector_norm(ref))
            assert err < TOL[dtype], (mode, transpose, err)


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_mode_dot_any_shape_infinities_stay_in_their_fibres(cuda, mode):
    import tensorly_amd as tla
    g = torch.Generator(device=cuda).manual_seed(5)
    shape = (19, 21, 35)
    X = torch.randn(shape, generator=g, device=cuda)
    where = tuple(s - 1 for s in shape)
    X[where] = float("inf")
    U = torch.rand((shape[mode], 18), generator=g, device=cuda) + 0.1
    out = torch.movedim(tla.mode_dot(X, U, mode, transpose=True), mode, -1)
    hit = torch.zeros(out.shape[:2], dtype=torch.bool, device=cuda)
    hit[tuple(s - 1 for s in out.shape[:2])] = True
    assert bool(torch.isfinite(out[~hit]).all()) and bool((out[hit] == float("inf")).all())


@pytest.mark.parametrize("rows,rank,n_iter", [(37, 1, 100), (16, 4, 127), (17, 5, 128), (33, 8, 129), (50, 20, 300),
                                              (9, 1, 300)])
def test_hals_chunks_and_stopping_rule(cuda, rows, rank, n_iter):
    """The chunk lengths (128 iterations), workgroups of 16 rows, and the rule:
    at rank 1 the second iteration changes nothing, so it fires there.  FP64
    against the oracle: 300 iterations of a convergent descent, rounding
    about 1e-13 relative to the largest entry."""
    import numpy as np
    from oracle import tensorly_np as T
    from tensorly_amd import _lib
    from tensorly_amd.cp_tensor import grams64
    g = torch.Generator(device=cuda).manual_seed(rows + rank)
    F = [torch.rand((s, rank), generator=g, device=cuda, dtype=torch.float64) for s in (rows, 12, 10)]
    M = torch.randn((rows, rank), generator=g, device=cuda, dtype=torch.float64) * 3 + 1
    A0, L = F[0].cpu().numpy(), _lib.lib()
    grams = grams64(F)
    gp, _k = _lib.ptr_array(grams)
    iters = torch.zeros(1, dtype=torch.int32, device=cuda)
    nb = L.tla_hals_nnls_workspace_size(rows, rank)
    ws = _lib.workspace(nb, F[0].device)
    _lib.check(L.tla_hals_nnls(_lib.F64, _lib.ptr(F[0]), _lib.ptr(M), rows, rank, gp, 3, 0, None, _lib.F64, 0.0, 0,
                               n_iter, 1e-8, _lib.ptr(iters), _lib.ptr(ws), nb, _lib.stream(F[0].device)), "hals")
    Fn = [f.cpu().numpy() for f in F]
    utu = (Fn[1].T @ Fn[1]) * (Fn[2].T @ Fn[2])
    ref = T.hals_nnls(M.cpu().numpy().T, utu, A0.T, n_iter_max=n_iter, tol=1e-8).T
    np.testing.assert_allclose(Fn[0], ref, rtol=1e-9, atol=1e-12 * np.abs(ref).max())
    assert int(iters) == (2 if rank == 1 else n_iter)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("rank", [1, 4, 5, 16, 33, 64])
@pytest.mark.parametrize("shape,nnz", [((3, 40), 700), ((1, 9, 7), 257), ((40, 3, 5), 64), ((6, 5, 4, 3), 1000),
                                       ((2, 3, 4, 5, 6), 300), ((70, 2, 2), 1)])
def test_mttkrp_coo_tiles(cuda, shape, nnz, rank, dtype):
    """Lane groups of the padded rank, pieces of 256 nonzeros and their ends,
    rows without nonzeros.  Sums of at most 1,000 terms: tolerance as above."""
    from tensorly_amd.tenalg import unfolding_dot_khatri_rao_coo
    g = torch.Generator(device=cuda).manual_seed(nnz + rank)
    coords = torch.stack([torch.randint(0, s, (nnz,), generator=g, device=cuda) for s in shape])
    values = torch.randn(nnz, generator=g, device=cuda, dtype=dtype)
    F = [torch.randn((s, rank), generator=g, device=cuda, dtype=dtype) for s in shape]
    w = torch.rand(rank, generator=g, device=cuda, dtype=dtype) + 0.5
    for mode in range(len(shape)):
        out = unfolding_dot_khatri_rao_coo(coords, values, shape, (w, F), mode)
        t = values.double()[:, None].expand(nnz, rank)
        for m in range(len(shape)):
            if m != mode:
                t = t * F[m].double()[coords[m]]
        ref = torch.zeros((shape[mode], rank), dtype=torch.float64, device=cuda).index_add_(0, coords[mode], t)
        if len(shape) > 2:
            ref = ref * w.double()
        assert out.dtype == dtype and out.shape == ref.shape
        err = float(torch.linalg.vector_norm(out.double() - ref) / torch.linalg.vector_norm(ref))
        assert err < TOL[dtype], (mode, err)
    assert torch.equal(unfolding_dot_khatri_rao_coo(coords, values, shape, (w, F), 0),
                       unfolding_dot_khatri_rao_coo(coords, values, shape, (w, F), 0))


def _spd(kind, n, rng):
    import numpy as np
    q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    lam = {"spread": 10.0 ** -np.linspace(0, 6, n), "noise": np.sort(rng.random(n))[::-1] + 1.0,
           "clusters": np.repeat(np.arange(n // 4 + 1, 0, -1.0), 4)[:n],
           "low rank": np.where(np.arange(n) < max(1, n // 3), n - np.arange(n), 0.0),
           "identity": np.ones(n)}[kind]
    a = (q * lam) @ q.T
    return (a + a.T) / 2, np.sort(lam)[::-1]


@pytest.mark.parametrize("kind", ["spread", "noise", "clusters", "low rank", "identity"])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 16, 17, 48, 63, 64, 65, 90, 127, 128])
def test_sym_eig_small(cuda, kind, n):
    """The direct solver (separated eigenvalues) and the Jacobi sweeps it
    leaves clusters to: eigenvalues, residuals and orthonormality to 1e-13 n
    of the norm (backward stable steps of n rotations or reflections each)."""
    import numpy as np
    from tensorly_amd.svd import gram_eigh
    a, lam = _spd(kind, n, np.random.default_rng(n))
    G = torch.tensor(a, device=cuda)
    for k in sorted({1, max(1, n // 3), n}):
        w, v = (t.cpu().numpy() for t in gram_eigh(G, k))
        tol = 1e-13 * max(n, 4) * lam[0]
        assert np.max(np.abs(w - lam[:k])) < tol
        assert np.max(np.abs(a @ v - v * w)) < tol
        assert np.max(np.abs(v.T @ v - np.eye(k))) < 1e-13 * max(n, 4)


@pytest.mark.parametrize("a", [[[0.0, 0.0], [0.0, 0.0]], [[2.0, 0.0, 0.0], [0.0, 3.0, 0.0], [0.0, 0.0, 1.0]],
                               [[1e-30, 1e-31], [1e-31, 3e-30]], [[1e30, 1e29], [1e29, 3e30]]])
def test_sym_eig_scales_and_diagonals(cuda, a):
    import numpy as np
    from tensorly_amd.svd import gram_eigh
    a = np.array(a)
    w, v = (t.cpu().numpy() for t in gram_eigh(torch.tensor(a, device=cuda), len(a)))
    ref = np.linalg.eigvalsh(a)[::-1]
    np.testing.assert_allclose(w, ref, rtol=1e-13, atol=0)
    np.testing.assert_allclose(v.T @ v, np.eye(len(a)), atol=1e-13)


@pytest.mark.parametrize("n,rank,k", [(144, 28, 28), (181, 28, 4), (200, 12, 30), (150, 1, 2), (130, 40, 44),
                                      (256, 3, 60), (300, 90, 100), (160, 0, 5)])
@pytest.mark.parametrize("warm", [False, True])
def test_sym_eig_rank_below_the_block(cuda, n, rank, k, warm):
    """Fewer independent directions than the block iteration keeps (48, 64 or
    128), and than it is asked for: eigenvalues, residuals and orthonormality
    as for a matrix of full rank.  2e-11: the solver stops at residuals of
    1e-11 of the largest eigenvalue."""
    import numpy as np
    from tensorly_amd.svd import gram_eigh
    x = np.random.default_rng(n).random((n, rank))
    a = x @ x.T
    q0 = torch.tensor(np.linalg.eigh(a)[1][:, ::-1][:, :k].copy(), device=cuda) if warm else None
    w, v = (t.cpu().numpy() for t in gram_eigh(torch.tensor(a, device=cuda), k, q0))
    lam = np.linalg.eigvalsh(a)[::-1]
    tol = 2e-11 * lam[0]
    assert np.max(np.abs(w - lam[:k])) <= tol
    assert np.max(np.abs(a @ v - v * w)) <= tol
    assert np.max(np.abs(v.T @ v - np.eye(k))) < 1e-12 * n


@pytest.mark.parametrize("n", [40, 100, 150, 300])
def test_sym_eig_nan(cuda, n):
    """NaN in, NaN out, and the next solve is right."""
    from tensorly_amd.svd import gram_eigh
    w, v = gram_eigh(torch.full((n, n), float("nan"), device=cuda, dtype=torch.float64), 5)
    assert torch.isnan(w).all()
    w, v = gram_eigh(torch.eye(n, device=cuda, dtype=torch.float64), 5)
    assert (w - 1).abs().max() < 1e-12


@pytest.mark.parametrize("n,k", [(130, 1), (200, 5), (256, 24), (256, 32), (300, 47), (256, 48)])
@pytest.mark.parametrize("move", [1e-3, 1e-5, 1e-7, 1e-9, 1e-12])
def test_sym_eig_warm_block_of_a_moved_matrix(cuda, n, k, move):
    """Ritz problems from far to almost diagonal, over both sides of the
    perturbation branch's limits, with a tail too flat to converge.  Residuals:
    the solver's 1e-11, doubled; columns orthonormal to 1e-11 (third-order
    terms: k^2 products of three ratios of at most 1e-5, ~1e-12)."""
    import numpy as np
    from tensorly_amd.svd import gram_left_singular
    rng = np.random.default_rng(n + k)
    lam = np.concatenate([np.linspace(10.0, 2.0, k), rng.uniform(0.3, 0.5, n - k)])
    q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    a = (q * lam) @ q.T
    d = rng.standard_normal((n, n))
    b = a + move * (d + d.T) / np.sqrt(n)
    _, _, blk = gram_left_singular(torch.tensor((a + a.T) / 2, device=cuda), k, torch.float64, want_block=True)
    for _ in range(2):
        u, s, blk = gram_left_singular(torch.tensor(b, device=cuda), k, torch.float64, warm=blk, want_block=True)
        u, w = u.cpu().numpy(), s.cpu().numpy() ** 2
        assert np.max(np.abs(w - np.linalg.eigvalsh(b)[::-1][:k])) < 2e-10
        assert np.max(np.abs(b @ u - u * w)) < 2e-10
        assert np.max(np.abs(u.T @ u - np.eye(k))) < 1e-11


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("shape", [(1, 1), (2, 1), (1, 40), (33, 16), (32, 13), (32, 14), (31, 17), (65, 1, 64), (5, 33, 16),
                                   (3, 70, 19), (2, 1, 16), (130, 40, 2), (7, 64, 8, 2), (257, 1030), (40, 3, 37)])
def test_mode_gram_any_shape(cuda, shape, dtype):
    """Every mode, over the edges of tiles (32 rows) and pieces (16 columns),
    against the same product in float64: sums of n products of float64."""
    from tensorly_amd.svd import mode_gram
    x = torch.randn(shape, dtype=dtype, generator=torch.Generator().manual_seed(len(shape))).to(cuda)
    for m in range(len(shape)):
        u = torch.movedim(x, m, 0).reshape(shape[m], -1).double().cpu()
        bound = 2.3e-16 * u.shape[1] * (u.abs() @ u.abs().T)
        assert bool(((mode_gram(x, m).cpu() - u @ u.T).abs() <= bound).all()), m


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n", [1, 1023, 4096, 8192 * 3 + 5, 1024 * 4096 + 4097])
def test_sqnorm_any_size_and_alignment(cuda, n, dtype):
    """From an odd element on: n products summed in float64."""
    from tensorly_amd.decomposition._tucker import _sqnorm64
    x = torch.randn(n + 1, dtype=dtype, generator=torch.Generator().manual_seed(n))[1:].to(cuda)
    ref = float((x.double().cpu() ** 2).sum())
    assert abs(float(_sqnorm64(x)) - ref) <= 2.3e-16 * n * ref


@pytest.mark.parametrize("shape,rank", [((149, 40, 300), 6), ((5, 70, 131), 9), ((260, 3), 3), ((2, 3, 2, 2, 2, 2, 2, 3), 2)])
def test_svd_init_batch_equals_single_modes(cuda, shape, rank):
    """All modes' solves in one call against one by one: the same solver on
    the same Grams, up to eight at a time."""
    from tensorly_amd.svd import leading_left_singular_vectors, leading_left_singular_vectors_batch
    x = torch.rand(shape, dtype=torch.float64, generator=torch.Generator().manual_seed(rank)).to(cuda)
    n = len(shape)
    for m, (U, S, blk) in enumerate(leading_left_singular_vectors_batch(x, list(range(n)), [rank] * n)):
        U1, S1, blk1 = leading_left_singular_vectors(x, m, rank, return_warm=True)
        assert torch.equal(U, U1) and torch.equal(S, S1)
        assert (blk is None) == (blk1 is None) and (blk is None or torch.equal(blk, blk1))


@pytest.mark.parametrize("shape,rank", [((2, 3, 2, 2, 2, 2, 2, 2, 3), 2), ((4, 100), 100), ((3, 4), 6), ((1, 1), 1)])
def test_svd_init_of_any_order_and_rank(cuda, shape, rank):
    """Orders above the kernels' eight, and ranks above a mode's size (random
    columns after U's) or above both sizes (a warning): U and S of numpy's
    SVD, to the rounding of the squared spectrum (1e-7 of the largest)."""
    import numpy as np
    from tensorly_amd.decomposition._cp import initialize_cp
    x = torch.rand(shape, dtype=torch.float64, generator=torch.Generator().manual_seed(3)).to(cuda)
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        factors = initialize_cp(x, rank, init="svd", random_state=0)[1]
    for m, f in enumerate(factors):
        assert tuple(f.shape) == (shape[m], rank)
        u, s, _ = np.linalg.svd(torch.movedim(x, m, 0).reshape(shape[m], -1).cpu().numpy(), full_matrices=False)
        k = min(rank, len(s))
        got = f[:, :k].cpu().numpy()
        want = u[:, :k] * (s[:k] if m == 0 else 1.0)
        assert np.max(np.abs(np.abs(got) - np.abs(want))) < 1e-7 * max(1.0, s[0])


@pytest.mark.parametrize("shape,rank,precision", [((256, 256, 256), 16, "fp32"), ((512, 512, 64), 16, "fp32"),
                                                  ((64, 128, 2048), 33, "fp32"), ((256, 256, 260), 5, "fp32"),
                                                  ((256, 256, 256), 24, "bf16x3"), ((256, 256, 256), 4, "valu")])
def test_cp_lstsq_grad_shared_contraction(cuda, shape, rank, precision):
    """Sizes on both sides of the shared contraction's rule (2^24 entries,
    shape[2] >= 4 rank, a matrix-core kernel), with weights, against float64.
    The MTTKRP's tolerance above on the larger of the two terms."""
    import tensorly_amd as tla
    gen = torch.Generator(device=cuda).manual_seed(rank)
    x = torch.randn(shape, device=cuda, generator=gen)
    w = torch.rand(rank, device=cuda, generator=gen) + 0.5
    F = [torch.randn(s, rank, device=cuda, generator=gen) for s in shape]
    with tla.tenalg.precision(precision):
        grads = tla.cp_lstsq_grad((w, F), x).factors
    D, wd, xd = [f.double() for f in F], w.double(), x.double()
    G = [d.T @ d for d in D]
    for m in range(3):
        i, j = (k for k in range(3) if k != m)
        acc = G[i] * G[j] * (wd[:, None] * wd[None, :])
        model = D[m] @ acc
        mt = reference(xd, wd, D, m)
        err = (grads[m].double() - (model - mt)).norm()
        assert float(err / max(model.norm(), mt.norm())) < (2e-6 if precision != "bf16x3" else 2e-5)


@pytest.mark.parametrize("rows,rank", [(1, 1), (63, 16), (64, 17), (65, 33), (577, 64), (1500, 10)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_gram64_edges(cuda, rows, rank, dtype):
    """Row blocks of 64, rank tiles of 16, eight partials at a time: sums of
    `rows` float64 products."""
    from tensorly_amd.cp_tensor import grams64
    a = torch.randn(rows, rank, dtype=dtype, generator=torch.Generator().manual_seed(rows)).to(cuda)
    g, d = grams64([a])[0].cpu(), a.double().cpu()
    assert bool(((g - d.T @ d).abs() <= 2.3e-16 * (rows + 8) * (d.abs().T @ d.abs())).all())


@pytest.mark.parametrize("rank", [1, 10, 17, 40, 64])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_parafac_any_shape_sweeps(cuda, rank, dtype):
    """Two sweeps from given factors, the next solve's inverse formed beside
    the sum of partials, against the normal equations in float64: cond(V) is
    below 1e3 for such factors, times 100 eps for the sums."""
    import tensorly_amd as tla
    shape = (131, 145, 270)
    x, F, _ = problem(cuda, shape, rank, dtype, rank)
    got = tla.parafac(x, rank, n_iter_max=2, tol=0, init=(None, [f.clone() for f in F])).factors
    D, xd = [f.double() for f in F], x.double()
    for _ in range(2):
        for m in range(3):
            i, j = (k for k in range(3) if k != m)
            D[m] = torch.linalg.solve((D[i].T @ D[i]) * (D[j].T @ D[j]), reference(xd, None, D, m).T).T
    tol = 1e5 * torch.finfo(dtype).eps
    for a, b in zip(got, D):
        assert float((a.double() - b).norm() / b.norm()) < tol


@pytest.mark.parametrize("n,k", [(200, 5), (256, 24), (256, 32), (300, 40)])
@pytest.mark.parametrize("move", [1e-2, 8e-4, 5e-4, 1e-4])
@pytest.mark.parametrize("max_iter", [2, 3])
def test_sym_eig_iteration_limit_returns_orthonormal_vectors(cuda, n, k, move, max_iter):
    """A warm solve that the iteration limit ends: whatever step was the last,
    its vectors are orthonormal (to 1e-11, as above) and its values are their
    Ritz values.  The moves of 8e-4 and 5e-4 leave a Ritz matrix that second-order
    perturbation would diagonalise to 1e-10 only."""
    import numpy as np
    from tensorly_amd.svd import gram_left_singular
    rng = np.random.default_rng(n + k)
    lam = np.concatenate([np.linspace(10.0, 2.0, k), rng.uniform(3e-3, 5e-3, n - k)])
    q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    a = (q * lam) @ q.T
    d = rng.standard_normal((n, n))
    b = a + move * (d + d.T) / np.sqrt(n)
    _, _, blk = gram_left_singular(torch.tensor((a + a.T) / 2, device=cuda), k, torch.float64, want_block=True)
    u, s, _ = gram_left_singular(torch.tensor(b, device=cuda), k, torch.float64, warm=blk, max_iter=max_iter)
    u, w = u.cpu().numpy(), s.cpu().numpy() ** 2
    assert np.max(np.abs(u.T @ u - np.eye(k))) < 1e-11
    assert np.max(np.abs(np.einsum("ij,ik,kj->j", u, b, u) - w)) < 2e-10


@pytest.mark.parametrize("half", [1, 2, 5, 16, 40])
def test_svd_init_signs_of_tied_entries(cuda, half):
    """Left singular vectors [u, u] and [u, -u], whose largest entries tie but
    for the rounding of the solve: the sign rule looks at the vectors in the
    tensor's type, where the first of equal entries decides, in the init as in
    the SVD of one unfolding."""
    from tensorly_amd.decomposition._cp import initialize_cp
    from tensorly_amd.svd import svd_interface
    g = torch.Generator().manual_seed(half)
    a, b = (torch.randint(-8, 9, (half, 60), generator=g).float() for _ in range(2))
    # rows i and half + i have the Gram of the pair swapped
    x = torch.cat([torch.cat([a, b], 1), torch.cat([b, a], 1)], 0).reshape(2 * half, 12, 10).to(cuda)
    rank = min(2 * half, 10)
    U = initialize_cp(x, rank, init="svd")[1][0]
    V, S, _ = svd_interface(x.reshape(2 * half, -1), n_eigenvecs=rank)
    V = V[:, :rank] * S[:rank]
    for r in range(rank):  # (columns of equal values may turn)
        if all(abs(float(S[r] - S[q])) > 1e-3 * float(S[0]) for q in range(rank) if q != r):
            assert float((U[:, r] - V[:, r]).norm()) < 1e-5 * float(S[0]), r
            assert float(U[U[:, r].abs().argmax(), r]) > 0


@pytest.mark.parametrize("shape", [(70_000_000, 2, 4), (67_108_864, 4, 4)])
def test_mode_dot_past_the_tiles_of_a_launch(cuda, shape):
    """More short runs than one launch has tiles for (2.2 and 4.3 GB): sums of
    two and four products."""
    import tensorly_amd as tla
    X = torch.arange(shape[0], device=cuda, dtype=torch.float32).remainder_(1024)[:, None, None].expand(shape).contiguous()
    U = torch.tensor([[1.0, 2.0, 4.0, 8.0][: shape[1]], [3.0, 5.0, 7.0, 9.0][: shape[1]]], device=cuda)
    for J in (1, 2):
        out = tla.mode_dot(X, U[:J], 1)
        for j in range(J):
            assert bool((out[:, j] == X[:, 0] * U[j].sum()).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("shape,rank,mode", [((3, 1200, 1001, 8), 64, 0), ((5, 1100, 1301, 6), 50, 0), ((1100, 1001, 3, 3), 64, 2),
                                             ((1100, 1009, 2, 5), 64, 3), ((1100, 2003, 3, 5), 100, 3),
                                             ((2, 3001, 3, 166, 4), 70, 0), ((3, 1_100_003, 5), 64, 0),
                                             ((1500, 4, 901, 3), 64, 1)])
def test_mttkrp_any_shape_scale_rows_in_slices(cuda, shape, rank, mode, dtype):
    """Output and contiguous mode both short: a table of the other modes'
    scale rows would be larger than the tensor, and is made 256 MiB at a time.
    Sums of up to 9.6 million terms in chains of at most a hundredth of them:
    sqrt(q / 100) eps.  The reference's own float64 sums are taken 4,096 terms
    at a time and those added up pairwise."""
    import tensorly_amd as tla
    from tensorly_amd import _lib
    X, F, w = problem(cuda, shape, rank, dtype, rank)
    n, size = X.numel(), X.element_size()
    sh, _k = _lib.shape_array(shape)
    ws = _lib.lib().tla_mttkrp_workspace_size(_lib.dtype_code(X), len(shape), sh, rank, mode, _lib.PREC_FP32)
    assert ws <= (256 << 20) + (32 << 20) + 512
    for weights in (None, w):
        out = tla.unfolding_dot_khatri_rao(X, (weights, F), mode)
        k = w.double()[None, :] if weights is not None else torch.ones((1, rank), dtype=torch.float64, device=cuda)
        for m, f in enumerate(F):
            if m != mode:
                k = (k[:, None, :] * f.double()[None, :, :]).reshape(-1, rank)
        u = torch.movedim(X.double(), mode, 0).reshape(shape[mode], -1)
        ref = torch.stack([u[:, q : q + 4096] @ k[q : q + 4096] for q in range(0, u.shape[1], 4096)], -1).sum(-1)
        err = float(torch.linalg.vector_norm(out.double() - ref) / torch.linalg.vector_norm(ref))
        assert err < max(1.0, 0.05 * (n / shape[mode]) ** 0.5 / 16) * TOL[dtype], err


@pytest.mark.parametrize("order", [2, 3])
def test_mttkrp_coo_mode_of_more_than_32_bits(cuda, order):
    """A contracted mode of more than 2^32 entries (a factor of 17 GB, zero but
    where the nonzeros look), alone and beside another."""
    from tensorly_amd.tenalg import unfolding_dot_khatri_rao_coo
    n = 2 ** 32 + 1000
    at = torch.tensor([0, 1000, 2 ** 31, 2 ** 32 - 1, 2 ** 32, 2 ** 32 + 7, n - 1], device=cuda)
    big = torch.zeros((n, 1), device=cuda)
    big[at, 0] = torch.arange(1.0, 8.0, device=cuda)
    F = [torch.tensor([[2.0], [3.0]], device=cuda), big]
    coords = torch.stack([torch.arange(7, device=cuda) % 2, at])
    values = torch.arange(10.0, 17.0, device=cuda)
    if order == 2:
        out = unfolding_dot_khatri_rao_coo(coords, values, (2, n), (None, F), 0)
        t = values * big[at, 0]
        assert out[:, 0].tolist() == [float(t[0::2].sum()), float(t[1::2].sum())]
    else:
        F3, c3 = [F[0], big, torch.ones((3, 1), device=cuda)], torch.cat([coords, coords[:1]], 0)
        out = unfolding_dot_khatri_rao_coo(c3, values, (2, n, 3), (None, F3), 2)
        t = values * big[at, 0] * F[0][coords[0], 0]
        assert out[:, 0].tolist() == [float(t[0::2].sum()), float(t[1::2].sum()), 0.0]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("rank", [1, 5, 16, 33, 64])
@pytest.mark.parametrize("rows,heavy", [(8192, 0), (8193, 0), (20001, 1), (100003, 5)])
def test_mttkrp_coo_many_rows(cuda, rows, heavy, rank, dtype):
    """Four rows per workgroup, rows of more than 64 segments (16,384 nonzeros)
    by the whole of it, most rows empty or of one nonzero.  Sums of up to
    20,000 terms in chains of 256 and fewer: tolerance as above."""
    from tensorly_amd.tenalg import unfolding_dot_khatri_rao_coo
    g = torch.Generator(device=cuda).manual_seed(rows + rank)
    idx = [torch.randint(0, rows, (30_000,), generator=g, device=cuda)]
    for h in range(heavy):
        idx.append(torch.full((16_300 + 60 * h,), (rows - 1) * (h + 1) // heavy, device=cuda))
    idx = torch.cat(idx)
    nnz, shape = idx.shape[0], (rows, 7, 9)
    coords = torch.stack([idx] + [torch.randint(0, s, (nnz,), generator=g, device=cuda) for s in shape[1:]])
    values = torch.randn(nnz, generator=g, device=cuda, dtype=dtype)
    F = [torch.randn((s, rank), generator=g, device=cuda, dtype=dtype) for s in shape]
    w = torch.rand(rank, generator=g, device=cuda, dtype=dtype) + 0.5
    out = unfolding_dot_khatri_rao_coo(coords, values, shape, (w, F), 0)
    t = values.double()[:, None] * F[1].double()[coords[1]] * F[2].double()[coords[2]] * w.double()
    ref = torch.zeros((rows, rank), dtype=torch.float64, device=cuda).index_add_(0, idx, t)
    for h in range(heavy):  # (one after another, so many would round more than the kernel)
        ref[(rows - 1) * (h + 1) // heavy] = t[idx == (rows - 1) * (h + 1) // heavy].sum(0)
    assert float(torch.linalg.vector_norm(out.double() - ref) / torch.linalg.vector_norm(ref)) < TOL[dtype]
    assert bool((out[torch.bincount(idx, minlength=rows) == 0] == 0).all())


def _hals(F, M, n_iter, tol, dtype):
    """tla_hals_nnls on F[0] in place; the iterations run."""
    from tensorly_amd import _lib
    from tensorly_amd.cp_tensor import grams64
    L, (rows, rank) = _lib.lib(), F[0].shape
    grams = grams64(F[1:])
    gp, _k = _lib.ptr_array([grams[0]] + grams)
    iters = torch.zeros(1, dtype=torch.int32, device=F[0].device)
    nb = L.tla_hals_nnls_workspace_size(rows, rank)
    ws = _lib.workspace(nb, F[0].device)
    _lib.check(L.tla_hals_nnls(_lib.dtype_code(F[0]), _lib.ptr(F[0]), _lib.ptr(M), rows, rank, gp, len(F), 0, None,
                               _lib.F64, 0.0, 0, n_iter, tol, _lib.ptr(iters), _lib.ptr(ws), nb,
                               _lib.stream(F[0].device)), "hals")
    return int(iters)


@pytest.mark.parametrize("rows,rank,n_iter,tol", [(40, 64, 100, 0.6), (40, 64, 2, 0.0), (40, 33, 3, 0.0), (40, 16, 5, 0.0),
                                                  (40, 5, 7, 0.0)])
def test_hals_from_a_start_far_above_the_solution(cuda, rows, rank, n_iter, tol):
    """The gradient falls by orders of magnitude in the first iteration: its
    rounding must not stay at the first size.  Against the oracle in FP64;
    tolerance as above."""
    import numpy as np
    from oracle import tensorly_np as T
    g = torch.Generator(device=cuda).manual_seed(rows + rank)
    F = [torch.rand((s, rank), generator=g, device=cuda, dtype=torch.float64) for s in (rows, 130, 110)]
    M = torch.rand((rows, rank), generator=g, device=cuda, dtype=torch.float64) * 3 + 1
    Fn = [f.cpu().numpy() for f in F]
    utu = (Fn[1].T @ Fn[1]) * (Fn[2].T @ Fn[2])
    ref = T.hals_nnls(M.cpu().numpy().T, utu, Fn[0].T.copy(), n_iter_max=n_iter, tol=tol).T
    _hals(F, M, n_iter, tol, torch.float64)
    np.testing.assert_allclose(F[0].cpu().numpy(), ref, rtol=1e-9, atol=1e-12 * np.abs(ref).max())


@pytest.mark.parametrize("rows,rank,n_iter,tol", [(40, 64, 300, 1e-8), (40, 48, 100, 0.9), (40, 64, 100, 0.6), (17, 64, 9, 0.0),
                                                  (110_000, 16, 30, 1e-8), (1_100_003, 3, 20, 1e-8), (1_100_003, 3, 100, 0.5),
                                                  (33, 7, 1, 1e-8), (1_050_000, 1, 1, 0.5)])
def test_hals_growing_chunks_and_many_rows(cuda, rows, rank, n_iter, tol):
    """A first chunk of 16 iterations (long ones, and many rows), rules
    that fire in a chunk, more rows than workgroups, and single
    iterations, against the oracle in FP64; tolerance as above."""
    import numpy as np
    from oracle import tensorly_np as T
    g = torch.Generator(device=cuda).manual_seed(rows + rank)
    F = [torch.rand((s, rank), generator=g, device=cuda, dtype=torch.float64) for s in (rows, 130, 110)]
    M = torch.rand((rows, rank), generator=g, device=cuda, dtype=torch.float64) * 3 + 1
    Fn = [f.cpu().numpy() for f in F]
    utu = (Fn[1].T @ Fn[1]) * (Fn[2].T @ Fn[2])
    ref = T.hals_nnls(M.cpu().numpy().T, utu, Fn[0].T.copy(), n_iter_max=n_iter, tol=tol).T
    _hals(F, M, n_iter, tol, torch.float64)
    np.testing.assert_allclose(F[0].cpu().numpy(), ref, rtol=1e-9, atol=1e-12 * np.abs(ref).max())


def test_hals_rows_past_a_launch(cuda):
    """2^30 rows: more than one launch has workgroups of 16 rows for.  At rank
    1 every iteration gives max(m / u, 0)."""
    rows = 2 ** 30 + 5
    F = [torch.ones((rows, 1), device=cuda), torch.full((2, 1), 2.0, device=cuda), torch.full((2, 1), 0.5, device=cuda)]
    M = torch.arange(rows, device=cuda, dtype=torch.float32).remainder_(64).sub_(16)[:, None]
    iters = _hals(F, M, 2, 0.0, torch.float32)
    wrong = int((F[0] != M.clamp_(min=0) / 4).sum())
    assert iters == 2 and wrong == 0


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("shape", [(33, 16), (33, 17), (33, 21), (33, 22), (33, 24), (33, 25), (7, 34, 20), (7, 34, 23),
                                   (2, 65, 37), (2049, 5801), (2049, 5802), (3, 600, 515)])
def test_mode_gram_rules(cuda, shape, dtype):
    """Both sides of the rules on the length of the runs and on float64 rows
    off the 16-byte grid: sums of n products of float64, and as much for the
    reference's own."""
    from tensorly_amd.svd import mode_gram
    x = torch.randn(shape, dtype=dtype, generator=torch.Generator().manual_seed(len(shape))).to(cuda)
    m = len(shape) - 2
    u = torch.movedim(x, m, 0).reshape(shape[m], -1).double()
    bound = 2 * 2.3e-16 * u.shape[1] * (u.abs() @ u.abs().T)
    worst = float(((mode_gram(x, m) - u @ u.T).abs() - bound).max())
    assert worst <= 0


def _sym_eig(a, k, cuda):
    """(values, vectors, iterations) of tla_sym_eig."""
    from tensorly_amd import _lib
    L, n = _lib.lib(), a.shape[0]
    G = torch.tensor(a, device=cuda)
    w, v = torch.empty(k, device=cuda, dtype=torch.float64), torch.empty((n, k), device=cuda, dtype=torch.float64)
    it = torch.zeros(1, dtype=torch.int32, device=cuda)
    nb = L.tla_sym_eig_workspace_size(n)
    ws = _lib.workspace(nb, G.device)
    _lib.check(L.tla_sym_eig(_lib.ptr(G), n, k, None, 0, _lib.ptr(w), _lib.ptr(v), 1e-11, 300, _lib.ptr(it), _lib.ptr(ws),
                             nb, _lib.stream(G.device)))
    return w.cpu().numpy(), v.cpu().numpy(), int(it)


@pytest.mark.parametrize("kind", ["clusters", "low rank", "blocks", "projector", "wilkinson"])
@pytest.mark.parametrize("n", [4, 8, 17, 33, 48, 63, 64, 65, 90, 127, 128])
def test_sym_eig_clusters(cuda, kind, n):
    """Clusters, where the vectors of the twisted factorisations cannot be told
    apart.  Eigenvalues, residuals and orthonormality as above."""
    import numpy as np
    rng = np.random.default_rng(n)
    if kind in ("clusters", "low rank"):
        a = _spd(kind, n, rng)[0]
    elif kind == "blocks":  # a tridiagonal form that falls apart
        b = rng.standard_normal((n // 2, n // 2))
        a = np.kron(np.eye(2), b @ b.T) if n % 2 == 0 else np.pad(np.kron(np.eye(2), b @ b.T), (0, 1))
    elif kind == "projector":
        q = np.linalg.qr(rng.standard_normal((n, n)))[0][:, : (n + 1) // 2]
        a = q @ q.T
    else:  # pairs of eigenvalues that agree to all digits
        a = np.diag(np.abs(np.arange(n) - (n - 1) / 2.0)) + np.diag(np.ones(n - 1), 1) + np.diag(np.ones(n - 1), -1)
    a = (a + a.T) / 2
    lam = np.linalg.eigvalsh(a)[::-1]
    for k in sorted({n // 2, n}):
        w, v, _ = _sym_eig(a, k, cuda)
        tol = 1e-13 * n * np.abs(lam).max()
        assert np.max(np.abs(w - lam[:k])) < tol
        assert np.max(np.abs(a @ v - v * w)) < tol
        assert np.max(np.abs(v.T @ v - np.eye(k))) < 1e-13 * n


@pytest.mark.parametrize("n", [1, 2, 5, 48, 64, 65, 128])
def test_sym_eig_of_a_diagonal_matrix_is_exact(cuda, n):
    """Diagonal already: no rotations, no reflections."""
    import numpy as np
    d = np.random.default_rng(n).permutation(n) + 0.3
    w, v, it = _sym_eig(np.diag(d), n, cuda)
    assert it == 0 and np.array_equal(w, np.sort(d)[::-1])
    assert np.array_equal(v, np.eye(n)[:, np.argsort(-d)])


def reference_in_blocks(X, w, F, mode):
    """The reference with its sums taken 256 terms at a time and those added
    up pairwise, so that its own rounding stays below the float64 kernels'."""
    k = w.double()[None, :] if w is not None and len(F) > 2 else None
    for m, f in enumerate(F):
        if m != mode:
            k = f.double() if k is None else (k[:, None, :] * f.double()[None, :, :]).reshape(-1, f.shape[1])
    u = torch.movedim(X.double(), mode, 0).reshape(X.shape[mode], -1)
    return torch.stack([u[:, q : q + 256] @ k[q : q + 256] for q in range(0, u.shape[1], 256)], -1).sum(-1)


@pytest.mark.parametrize("case", any_shape_cases.MTTKRP, ids=lambda c: "%s-%s-%d-%d" % (("f32", "f64")[c[0]],
                         "x".join(map(str, c[1])), c[2], c[3]))
def test_mttkrp_any_shape_tiles_per_wave(cuda, case):
    """Two and more tiles per wave, with their remainders of rows, columns,
    rank columns and chunks.  Up to 32,000 terms, in chains of at most a
    hundredth of them and then of the partial sums': tolerance as above."""
    import tensorly_amd as tla
    f64, shape, rank, mode, weights, _ = case
    dtype = torch.float64 if f64 else torch.float32
    X, F, w = problem(cuda, shape, rank, dtype, rank + mode)
    w = w if weights else None
    out = tla.unfolding_dot_khatri_rao(X, (w, F), mode)
    ref = reference_in_blocks(X, w, F, mode)
    err = torch.linalg.vector_norm(out.double() - ref, dim=1) / torch.linalg.vector_norm(ref, dim=1)
    assert float(torch.linalg.vector_norm(out.double() - ref) / torch.linalg.vector_norm(ref)) < TOL[dtype]
    assert float(err.max()) < 10 * TOL[dtype]  # (and no row far off: the edges of tiles)


@pytest.mark.parametrize("case", any_shape_cases.MODE_DOT, ids=lambda c: "%s-%s-%d" % (("f32", "f64")[c[0]],
                         "x".join(map(str, c[1])), c[3]))
def test_mode_dot_any_shape_tiles_per_wave(cuda, case):
    """Wide tiles of columns and rows, alone and shared by a block's waves.
    Sums of at most 37 terms: tolerance as above."""
    import tensorly_amd as tla
    f64, shape, mode, J, _, _ = case
    dtype = torch.float64 if f64 else torch.float32
    g = torch.Generator(device=cuda).manual_seed(J)
    X = torch.randn(shape, generator=g, device=cuda, dtype=dtype)
    U = torch.randn((J, shape[mode]), generator=g, device=cuda, dtype=dtype)
    out = tla.mode_dot(X, U, mode)
    ref = torch.movedim(torch.movedim(X.double(), mode, -1) @ U.double().T.contiguous(), -1, mode)
    err = (out.double() - ref).abs()
    assert float(torch.linalg.vector_norm(err) / torch.linalg.vector_norm(ref)) < TOL[dtype]
    scale = torch.movedim(torch.movedim(X.double().abs(), mode, -1) @ U.double().abs().T.contiguous(), -1, mode)
    assert float((err / scale).max()) < TOL[dtype]  # (every element: the edges of tiles)
