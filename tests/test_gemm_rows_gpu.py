"""bf16 products whose rows do not fill 128-row tiles: the rows past the end stay out of
the outputs, the column sums and the head, and nothing past the last row is written."""
import pytest
import torch

from neuralangelo_amd import functional as Fn
from neuralangelo_amd._lib import NA_ACT_RELU, NA_ACT_SOFTPLUS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [128, 256])
@pytest.mark.parametrize("K", [144, 256, 280])
@pytest.mark.parametrize("M", [1, 31, 33, 127, 129, 1000, 33001])
def test_ragged_rows(M, N, K):
    g = torch.Generator().manual_seed(M + N + K)
    A = (torch.randn(M, K, generator=g) * 0.2).bfloat16().cuda()
    B = (torch.randn(N, K, generator=g) * 0.2).bfloat16().cuda()
    bias, hw = torch.randn(N, generator=g).cuda(), torch.randn(N, generator=g).cuda()
    z = A.double() @ B.double().t()
    # float32 accumulation: one rounding per product and per addition
    e = (K + 8) * 2.0 ** -23 * (A.double().abs() @ B.double().abs().t())
    out = torch.full((M + 2, N), 9.0, device="cuda")

    def run(**kw):
        out.fill_(9.0)
        Fn.gemm(A, K, 0, B, K, 0, M, N, K, out, N, **kw)
        assert (out[M:] == 9.0).all()
        return out[:M].double()
    assert ((run() - z).abs() <= e).all()
    zb = z + bias.double()
    eb = e + 2.0 ** -22 * zb.abs()
    assert ((run(bias=bias, act=NA_ACT_RELU) - zb.relu()).abs() <= eb).all()
    Z = torch.full((M + 1, N), 9.0, device="cuda")
    parts = torch.full((Fn.head_parts(N) * M + 5,), 9.0, device="cuda")
    sp = torch.nn.functional.softplus(zb, beta=100)
    es = eb + 1e-7 + 2.0 ** -21 * sp
    assert ((run(bias=bias, act=NA_ACT_SOFTPLUS, z_out=Z, head_w=hw, head_out=parts) - sp).abs() <= es).all()
    assert ((Z[:M].double() - zb).abs() <= eb).all() and (Z[M:] == 9.0).all() and (parts[-5:] == 9.0).all()
    head = parts[:-5].view(-1, M)[:N // 32].double().sum(0)
    assert ((head - sp @ hw.double()).abs() <= (es + 64 * 2.0 ** -23 * sp) @ hw.double().abs()).all()
    y = (torch.rand(M, N, generator=g) - 0.3).bfloat16().cuda()
    r1a, r1b = torch.randn(M, generator=g).cuda(), torch.randn(N, generator=g).cuda()
    cs = torch.zeros(N, device="cuda")
    got = run(dact=NA_ACT_RELU, dact_y=y, ld_dact=N, r1_a=r1a, r1_b=r1b, colsum=cs)
    rank1 = r1a.double()[:, None] * r1b.double()
    ref, er = (z + rank1) * (y > 0), e + 2.0 ** -22 * rank1.abs()
    assert ((got - ref).abs() <= er).all()
    assert ((cs.double() - ref.sum(0)).abs() <= er.sum(0) + (M + 8) * 2.0 ** -23 * ref.abs().sum(0)).all()
