"""GPU parity of the sparse primitives and of jacobian(), restating
ceviche tests/test_primitives.py:14-121 (np.random.seed(2), N = 8, M = 44,
random complex COO with duplicate indices, objective |sum(out)|, reverse and
forward jacobians against grad_num to 3 decimals) plus exact comparisons with
the oracle."""
import numpy as np
import pytest
import torch

from oracle import primitives_ref as P
from oracle.numdiff import grad_num

pytestmark = pytest.mark.gpu
DECIMAL = 3


def _setup():
    np.random.seed(2)
    N = 8
    M = N ** 2 - 20
    d = dict(N=N, M=M, ind=P.make_rand_indices(N, M), ent=P.make_rand_complex(M),
             ind2=P.make_rand_indices(N, M - 2), ent2=P.make_rand_complex(M - 2),
             x=P.make_rand_complex(N), b=P.make_rand_complex(N))
    return d


def out_fn(o):
    return abs(o.sum())


def _check(fn, arg):
    import ceviche_amd as cv
    grad_rev = cv.jacobian(fn, mode='reverse')(arg)[0]
    grad_for = cv.jacobian(fn, mode='forward')(arg)[0]
    grad_true = grad_num(fn, arg)
    np.testing.assert_almost_equal(grad_rev, grad_true, decimal=DECIMAL)
    np.testing.assert_almost_equal(grad_for, grad_true, decimal=DECIMAL)


def test_values_match_oracle():
    from ceviche_amd import primitives as cp
    d = _setup()
    y = cp.sp_mult(d['ent'], d['ind'], d['x'])
    assert isinstance(y, np.ndarray) and y.dtype == np.complex128
    assert np.allclose(y, P.sp_mult(d['ent'], d['ind'], d['x']), rtol=1e-14, atol=1e-14)
    xs = cp.sp_solve(d['ent'], d['ind'], d['b'])
    ref = P.sp_solve(d['ent'], d['ind'], d['b'])
    assert np.linalg.norm(xs - ref) <= 1e-10 * np.linalg.norm(ref)
    eb, ib = cp.spsp_mult(d['ent'], d['ind'], d['ent2'], d['ind2'], d['N'])
    rb = P.make_sparse(*P.spsp_mult(d['ent'], d['ind'], d['ent2'], d['ind2'], d['N']), (d['N'], d['N']))
    assert np.allclose(P.make_sparse(eb, ib, (d['N'], d['N'])).toarray(), rb.toarray(), rtol=1e-14, atol=1e-14)


def test_index_sets_modified_in_place_are_reanalysed():
    """The symbolic grouping is cached per index set: an index array (numpy
    or torch) changed in place must give the new matrix's product."""
    from ceviche_amd import primitives as cp
    d = _setup()
    ind = d['ind'].copy()
    for as_torch in (False, True):
        idx = torch.from_numpy(ind.copy()).cuda() if as_torch else ind.copy()
        ent = d['ent']
        x = d['x']
        y0 = cp.sp_mult(ent, idx, x)
        idx[1, :5] = (idx[1, :5] + 3) % d['N']          # in place
        y1 = cp.sp_mult(ent, idx, x)
        host = idx.cpu().numpy() if as_torch else idx
        assert np.allclose(y0, P.sp_mult(ent, ind, x), rtol=1e-14, atol=1e-14)
        assert np.allclose(y1, P.sp_mult(ent, host, x), rtol=1e-14, atol=1e-14)
        eb, ib = cp.spsp_mult(ent, idx, ent, idx, d['N'])
        ib = ib.cpu().numpy() if isinstance(ib, torch.Tensor) else ib
        rb = P.make_sparse(*P.spsp_mult(ent, host, ent, host, d['N']), (d['N'], d['N']))
        eb = eb.cpu().numpy() if isinstance(eb, torch.Tensor) else eb
        assert np.allclose(P.make_sparse(eb, ib, (d['N'], d['N'])).toarray(), rb.toarray(), rtol=1e-14, atol=1e-14)


def test_mult_entries():
    from ceviche_amd.primitives import sp_mult
    d = _setup()
    entries = P.make_rand_complex(d['M'])
    _check(lambda e: out_fn(sp_mult(e, d['ind'], d['x'])), entries)


def test_mult_x():
    from ceviche_amd.primitives import sp_mult
    d = _setup()
    x = P.make_rand_complex(d['N'])
    _check(lambda xx: out_fn(sp_mult(d['ent'], d['ind'], xx)), x)


def test_solve_entries():
    from ceviche_amd.primitives import sp_solve
    d = _setup()
    entries = P.make_rand_complex(d['M'])
    _check(lambda e: out_fn(sp_solve(e, d['ind'], d['b'])), entries)


def test_solve_b():
    from ceviche_amd.primitives import sp_solve
    d = _setup()
    b = P.make_rand_complex(d['N'])
    _check(lambda bb: out_fn(sp_solve(d['ent'], d['ind'], bb)), b)


def test_spsp_chain():
    """spsp_mult(spsp_mult(A(e), X), ...) then sp_solve, as test_spmut_entries."""
    from ceviche_amd.primitives import sp_solve, spsp_mult
    d = _setup()
    N = d['N']

    def fn(entries):
        ec, ic = spsp_mult(entries, d['ind'], d['ent2'], d['ind2'], N=N)
        ed, idd = spsp_mult(d['ent'], d['ind'], ec, ic, N=N)
        return out_fn(sp_solve(ed, idd, d['b']))

    entries = P.make_rand_complex(d['M'])
    _check(fn, entries)


def test_vjp_rules_match_oracle_formulas():
    """torch-convention gradients are the conjugates of the reference's VJPs."""
    from ceviche_amd import primitives as cp
    d = _setup()
    e = torch.tensor(d['ent'], requires_grad=True)
    b = torch.tensor(d['b'], requires_grad=True)
    x = cp.sp_solve(e, d['ind'], b)
    v = np.random.default_rng(1).standard_normal(d['N']) + 0j
    (torch.from_numpy(v).cuda() * x).real.sum().backward()
    # reference VJP with cotangent v (real, so both conventions agree on v)
    ge_ref = P.sp_solve_vjp_entries(v, d['ent'], d['ind'], d['b'])
    gb_ref = P.sp_solve_vjp_b(v, d['ent'], d['ind'], d['b'])
    assert np.allclose(e.grad.numpy(), np.conj(ge_ref), rtol=1e-9, atol=1e-12)
    assert np.allclose(b.grad.numpy(), np.conj(gb_ref), rtol=1e-9, atol=1e-12)


def test_larger_solve_and_singular_matrix():
    from ceviche_amd import primitives as cp
    rng = np.random.default_rng(3)
    N = 300
    rows = np.concatenate([np.arange(N), rng.integers(0, N, 4 * N)])
    cols = np.concatenate([np.arange(N), rng.integers(0, N, 4 * N)])
    ent = rng.standard_normal(rows.size) + 1j * rng.standard_normal(rows.size)
    ent[:N] += 20.0
    ind = np.vstack((rows, cols))
    b = rng.standard_normal(N) + 1j * rng.standard_normal(N)
    x = cp.sp_solve(ent, ind, b)
    assert np.linalg.norm(P.sp_mult(ent, ind, x) - b) <= 1e-11 * np.linalg.norm(b)
    sing = np.vstack((np.array([0, 1]), np.array([0, 1])))
    with pytest.warns(RuntimeWarning):
        xs = cp.sp_solve(np.array([1.0 + 0j, 0.0]), sing, np.ones(2))
    assert np.all(np.isnan(xs))


def test_jacobian_shapes_and_modes():
    import ceviche_amd as cv
    A = np.random.default_rng(0).standard_normal((3, 2))

    def fn(x):
        return torch.as_tensor(A) @ x

    x0 = np.array([0.3, -1.2])
    for mode in ('reverse', 'forward', 'numerical'):
        J = cv.jacobian(fn, mode=mode)(x0)
        assert J.shape == (3, 2)
        assert np.allclose(J, A, atol=1e-5)
    with pytest.raises(ValueError):
        cv.jacobian(fn, mode='sideways')


@pytest.mark.parametrize('n', [1, 2, 7, 16, 17, 63, 64, 65, 130, 1023, 1025, 1041, 2056, 3074])
def test_dense_lu_blocks_and_solves(n):
    """The blocked dense LU and its triangular solves around the edges of
    their panels (8 and 16 columns), row capacities (1024, 2048, 3072) and
    64-row blocks, for A, A^T and A^H and two right-hand sides, on matrices
    whose pivots come from far below the diagonal; backward error within
    50 n^(1/2) roundings (growth of partial pivoting on random matrices is
    about n^(1/2) at most)."""
    from ceviche_amd._lib import lib, ptr, stream_ptr, check
    print('dense lu', n, flush=True)
    g = torch.Generator().manual_seed(n)
    A = torch.randn(n, n, generator=g, dtype=torch.complex128)
    A[torch.arange(n), torch.arange(n)] *= 1e-3
    B = torch.randn(n, 2, generator=g, dtype=torch.complex128)
    dev = A.t().contiguous().cuda()                       # column-major
    piv = torch.empty(n, dtype=torch.int32, device='cuda')
    info = torch.full((1,), 7, dtype=torch.int32, device='cuda')
    check(lib().cv_dense_lu(n, ptr(dev), ptr(piv), ptr(info), stream_ptr()), 'lu')
    assert int(info.item()) == 0
    LU = dev.t()
    assert float(torch.tril(LU, -1).abs().max()) <= 1.5 if n > 1 else True   # multipliers of |re| + |im| pivoting
    for trans, M in ((0, A), (1, A.t()), (2, A.conj().t())):
        x = B.t().contiguous().cuda()
        check(lib().cv_dense_lu_solve(n, ptr(dev), ptr(piv), ptr(x), 2, trans, stream_ptr()), 'solve')
        X = x.t().cpu()
        r = (M.resolve_conj() @ X - B).norm()
        assert float(r) <= 50 * n ** 0.5 * 2.2e-16 * float(M.norm() * X.norm()), (trans, float(r))


def test_dense_lu_reports_the_first_zero_pivot():
    from ceviche_amd._lib import lib, ptr, stream_ptr, check
    A = torch.eye(40, dtype=torch.complex128)
    A[19] = A[18]                                          # rows 18 and 19 equal: column 19 has no pivot
    dev = A.t().contiguous().cuda()
    piv = torch.empty(40, dtype=torch.int32, device='cuda')
    info = torch.zeros(1, dtype=torch.int32, device='cuda')
    check(lib().cv_dense_lu(40, ptr(dev), ptr(piv), ptr(info), stream_ptr()), 'lu')
    assert int(info.item()) == 20


@pytest.mark.parametrize('lengths', [[1], [0, 3, 4, 5], [8, 0, 0, 9, 1, 2], [4] * 300, None])
def test_segsum_batches_and_unit_segments(lengths):
    """Segments shorter and longer than the batch of entries in flight, empty
    ones, and (None) the form without a segment pointer; storage-order sums
    agree to a few roundings."""
    from ceviche_amd.primitives import segsum
    g = torch.Generator().manual_seed(5)
    n_seg = 515 if lengths is None else len(lengths)
    m = n_seg if lengths is None else sum(lengths)
    p = torch.arange(n_seg + 1) if lengths is None else torch.tensor([0] + list(np.cumsum(lengths)))
    u, v = (torch.randn(37, generator=g, dtype=torch.complex128) for _ in range(2))
    iu, iv = (torch.randint(0, 37, (max(m, 1),), generator=g) for _ in range(2))
    out = torch.zeros(n_seg, dtype=torch.complex128, device='cuda')
    segsum(n_seg, None if lengths is None else p.cuda(), iu.cuda(), iv.cuda(), u.cuda(), v.cuda(), out, conj_v=True,
           alpha=2.0 - 1.0j)
    want = torch.stack([(2.0 - 1.0j) * (u[iu[p[s]:p[s + 1]]] * v[iv[p[s]:p[s + 1]]].conj()).sum() for s in range(n_seg)])
    assert float((out.cpu() - want).abs().max()) <= 1e-14 * max(1, max(lengths or [1]))


@pytest.mark.parametrize('n', [3, 70])
def test_dense_lu_solves_more_right_hand_sides_than_a_grid_has_rows(n):
    """65600 right-hand sides, beyond the 65535 workgroups of a launch's second
    and third dimension: backward error of the worst of them, 50 n^(1/2)
    roundings as above."""
    from ceviche_amd._lib import lib, ptr, stream_ptr, check
    g = torch.Generator().manual_seed(n)
    A = torch.randn(n, n, generator=g, dtype=torch.complex128)
    B = torch.randn(65600, n, generator=g, dtype=torch.complex128)
    dev, x = A.t().contiguous().cuda(), B.cuda()
    piv = torch.empty(n, dtype=torch.int32, device='cuda')
    info = torch.zeros(1, dtype=torch.int32, device='cuda')
    check(lib().cv_dense_lu(n, ptr(dev), ptr(piv), ptr(info), stream_ptr()), 'lu')
    check(lib().cv_dense_lu_solve(n, ptr(dev), ptr(piv), ptr(x), B.shape[0], 0, stream_ptr()), 'solve')
    X = x.cpu()
    r = (X @ A.t() - B).norm(dim=1)
    assert float((r / X.norm(dim=1)).max()) <= 50 * n ** 0.5 * 2.2e-16 * float(A.norm())
