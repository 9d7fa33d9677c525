"""The float32 products at tile, stage and split edges, in every operand layout, against
float64; and with values that do not split into bf16 parts."""
import pytest
import torch

from neuralangelo_amd import functional as Fn
from neuralangelo_amd._lib import NA_ACT_RELU, NA_ACT_SOFTPLUS, NA_EPI_ATOMIC, NA_EPI_STORE

pytestmark = pytest.mark.gpu


def operand(rows, k, trans, g, scale=1.0):
    """[rows, k] values and their storage ([rows, ld] or, transposed, [k, ld]; ld % 4 == 0)."""
    v = (torch.randn(rows, k, generator=g) * scale).cuda()
    m = v.t() if trans else v
    ld = (m.shape[1] + 3) // 4 * 4
    s = torch.full((m.shape[0], ld), 7.0, device="cuda")  # the padding is never part of a product
    s[:, :m.shape[1]] = m
    return v, s, ld


def bound(A, B, k):
    """One rounding per product and one per addition, in any order."""
    return (k + 16) * 2.0 ** -24 * (A.double().abs() @ B.double().abs().t()) + 1e-37


@pytest.mark.parametrize("ta, tb", [(0, 0), (1, 1), (1, 0), (0, 1)])
@pytest.mark.parametrize("M, N, K", [(1, 8, 4), (127, 256, 68), (128, 136, 136), (131, 280, 256),
                                     (70, 3, 20), (257, 160, 100), (4100, 96, 36), (64, 84, 3204)])
def test_layouts_and_edges(M, N, K, ta, tb):
    g = torch.Generator().manual_seed(M + N + K)
    A, a, lda = operand(M, K, ta, g)
    B, b, ldb = operand(N, K, tb, g)
    ref = A.double() @ B.double().t()
    C = torch.full((M, N), 3.0, device="cuda")
    Fn.gemm(a, lda, ta, b, ldb, tb, M, N, K, C, N)
    assert ((C.double() - ref).abs() <= bound(A, B, K)).all()
    C.fill_(0.5)
    Fn.gemm(a, lda, ta, b, ldb, tb, M, N, K, C, N, epilogue=NA_EPI_ATOMIC, split_k=3)
    # each part's sum is rounded once more as it is added
    parts = -(-K // 32)
    slack = (parts + 2) * 2.0 ** -24 * (ref.abs() + 0.5 + (A.double().abs() @ B.double().abs().t()))
    assert ((C.double() - ref - 0.5).abs() <= bound(A, B, K) + slack).all()


@pytest.mark.parametrize("M, N, K", [(5, 8, 16), (129, 256, 68), (640, 272, 256)])
def test_epilogue_terms(M, N, K):
    g = torch.Generator().manual_seed(M)
    A, a, lda = operand(M, K, 0, g, 0.1)
    B, b, ldb = operand(N, K, 0, g, 0.1)
    bias = torch.randn(N, generator=g).cuda()
    z = A.double() @ B.double().t() + bias.double()
    err = bound(A, B, K) + 2.0 ** -23 * z.abs()
    for act, ref in ((NA_ACT_RELU, z.relu()), (NA_ACT_SOFTPLUS, torch.nn.functional.softplus(z, beta=100))):
        C = torch.empty(M, N, device="cuda")
        Fn.gemm(a, lda, 0, b, ldb, 0, M, N, K, C, N, bias=bias, act=act)
        # both have slopes of at most 1; softplus adds a few ulps of 1 / beta
        assert ((C.double() - ref).abs() <= err + 1e-8 + 2.0 ** -22 * ref.abs()).all()
    y = torch.rand(M, N, generator=g).cuda() - 0.3
    r1a, r1b = torch.randn(M, generator=g).cuda(), torch.randn(N, generator=g).cuda()
    C, cs = torch.empty(M, N, device="cuda"), torch.ones(N, device="cuda")
    Fn.gemm(a, lda, 0, b, ldb, 0, M, N, K, C, N, dact=NA_ACT_RELU, dact_y=y, ld_dact=N, r1_a=r1a,
            r1_b=r1b, colsum=cs)
    v = (z - bias.double() + r1a.double()[:, None] * r1b.double()) * (y > 0)
    e = err + 2.0 ** -22 * (r1a.double()[:, None] * r1b.double()).abs()
    assert ((C.double() - v).abs() <= e).all()
    assert ((cs.double() - 1 - v.sum(0)).abs() <= e.sum(0) + M * 2.0 ** -23 * (1 + v.abs().sum(0))).all()


@pytest.mark.parametrize("ta, tb, N", [(0, 0, 264), (1, 1, 64), (0, 0, 5)])
def test_values_that_do_not_split(ta, tb, N):
    M, K = 300, 64
    g = torch.Generator().manual_seed(N)
    A, a, lda = operand(M, K, ta, g)
    B, b, ldb = operand(N, K, tb, g, 1e-3)
    sa, sb = (a.t() if ta else a), (b.t() if tb else b)
    for m, k, v in ((3, 5, float("inf")), (40, 0, float("nan")), (200, 63, 3.4e38), (299, 7, -float("inf"))):
        A[m, k] = sa[m, k] = v
    B[2, 9] = sb[2, 9] = -3.4e38
    B[4, 11] = sb[4, 11] = 0.0
    ref = A.double() @ B.double().t()
    C = torch.zeros(M, N, device="cuda")
    epi = NA_EPI_ATOMIC if ta else NA_EPI_STORE
    Fn.gemm(a, lda, ta, b, ldb, tb, M, N, K, C, N, epilogue=epi)
    ref[ref.abs() > 3.4028235e38] *= float("inf")  # past the float32 range
    assert torch.equal(C.isnan(), ref.isnan()) and torch.equal(C.isinf(), ref.isinf())
    fin = ref.isfinite()
    assert torch.equal(C[C.isinf()].sign().double(), ref[ref.isinf()].sign())
    assert ((C.double() - ref).abs()[fin] <= bound(A, B, K)[fin]).all()


@pytest.mark.parametrize("ta, tb", [(1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("M, N, K", [(129, 256, 68), (300, 40, 100), (70, 70, 36)])
def test_epilogue_terms_of_transposed_operands(M, N, K, ta, tb):
    """Tiles of 64 and 128 columns, and widths that only the staged epilogue takes."""
    g = torch.Generator().manual_seed(M)
    A, a, lda = operand(M, K, ta, g, 0.1)
    B, b, ldb = operand(N, K, tb, g, 0.1)
    bias = torch.randn(N, generator=g).cuda()
    z = A.double() @ B.double().t()
    err = bound(A, B, K) + 2.0 ** -23 * (z + bias.double()).abs()
    C = torch.empty(M, N, device="cuda")
    Fn.gemm(a, lda, ta, b, ldb, tb, M, N, K, C, N, bias=bias, act=NA_ACT_SOFTPLUS)
    ref = torch.nn.functional.softplus(z + bias.double(), beta=100)
    assert ((C.double() - ref).abs() <= err + 1e-8 + 2.0 ** -22 * ref.abs()).all()
    y = torch.rand(M, N, generator=g).cuda() - 0.3
    r1a, r1b = torch.randn(M, generator=g).cuda(), torch.randn(N, generator=g).cuda()
    r1 = r1a.double()[:, None] * r1b.double()
    cs = torch.ones(N, device="cuda")
    Fn.gemm(a, lda, ta, b, ldb, tb, M, N, K, C, N, dact=NA_ACT_RELU, dact_y=y, ld_dact=N, r1_a=r1a,
            r1_b=r1b, colsum=cs)
    v = (z + r1) * (y > 0)
    e = err + 2.0 ** -22 * r1.abs() + 2.0 ** -23 * z.abs()
    assert ((C.double() - v).abs() <= e).all()
    assert ((cs.double() - 1 - v.sum(0)).abs() <= e.sum(0) + M * 2.0 ** -23 * (1 + v.abs().sum(0))).all()


@pytest.mark.parametrize("rows, N, K", [(500, 64, 36), (3200, 256, 84), (20001 * 4, 90, 131)])
def test_weight_gradients_repeat(rows, N, K):
    """With the workspace the parts of the sum add up in order: the same bits on every call."""
    g = torch.Generator().manual_seed(rows)
    D, dpre, ldd = operand(N, rows, 1, g)
    X, x, ldx = operand(K, rows, 1, g)
    out = []
    for _ in range(4):
        dW = torch.full((N, K), 0.25, device="cuda")
        Fn.gemm(dpre, ldd, 1, x, ldx, 1, N, K, rows, dW, K, epilogue=NA_EPI_ATOMIC)
        out.append(dW)
    assert all(torch.equal(o, out[0]) for o in out[1:])
    ref = D.double() @ X.double().t()
    slack = 600 * 2.0 ** -24 * (ref.abs() + 0.25 + (D.double().abs() @ X.double().abs().t()))
    assert ((out[0].double() - 0.25 - ref).abs() <= bound(D, X, rows) + slack).all()


def test_split_k_of_one_is_one_addition():
    """Without a workspace the caller's split_k holds: one part adds once to each output."""
    rows, N, K = 3200, 256, 84
    g = torch.Generator().manual_seed(1)
    D, dpre, ldd = operand(N, rows, 1, g)
    X, x, ldx = operand(K, rows, 1, g)
    out = []
    for _ in range(4):
        dW = torch.zeros(N, K, device="cuda")
        Fn.gemm(dpre, ldd, 1, x, ldx, 1, N, K, rows, dW, K, epilogue=NA_EPI_ATOMIC,
                wgrad_partials=False)
        out.append(dW)
    assert all(torch.equal(o, out[0]) for o in out[1:])
    assert ((out[0].double() - D.double() @ X.double().t()).abs() <= bound(D, X, rows)).all()


@pytest.mark.parametrize("rows, N, K, parts", [(3204, 64, 84, 3), (500, 130, 257, 40), (36, 8, 20, 7)])
def test_split_k_parts_without_a_workspace(rows, N, K, parts):
    """The caller's parts add atomically, also where some of them hold no rows."""
    g = torch.Generator().manual_seed(parts)
    D, dpre, ldd = operand(N, rows, 1, g)
    X, x, ldx = operand(K, rows, 1, g)
    dW = torch.full((N, K), 0.5, device="cuda")
    Fn.gemm(dpre, ldd, 1, x, ldx, 1, N, K, rows, dW, K, epilogue=NA_EPI_ATOMIC, split_k=parts,
            wgrad_partials=False)
    ref, size = D.double() @ X.double().t(), D.double().abs() @ X.double().abs().t()
    slack = (parts + 2) * 2.0 ** -24 * (0.5 + size)
    assert ((dW.double() - 0.5 - ref).abs() <= bound(D, X, rows) + slack).all()
