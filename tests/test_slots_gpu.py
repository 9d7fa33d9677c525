"""Column sums in several copies (the _slots calls): every copy receives its workgroups'
share and nothing else, for row counts around the workgroup ranges."""
import ctypes

import pytest
import torch

from neuralangelo_amd import _lib
from neuralangelo_amd import functional as Fn
from neuralangelo_amd._lib import NA_ACT_RELU

pytestmark = pytest.mark.gpu


def close(got, terms):
    """got against the float64 sum of `terms` over rows: one rounding per addition."""
    ref, size = terms.double().sum(0), terms.double().abs().sum(0)
    return ((got.double() - ref).abs() <= (terms.shape[0] + 4) * 2.0 ** -24 * size + 1e-30).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 2047, 2048, 5000, 70001])
def test_slot_copies_add_up(rows, dtype):
    N, S, pad = 256, 3, 64
    g = torch.Generator().manual_seed(rows)
    dy = torch.randn(rows, N, generator=g).to(dtype).cuda()
    y = (torch.rand(rows, N, generator=g) - 0.3).to(dtype).cuda()
    buf = torch.zeros(S, N + pad, device="cuda")
    out = Fn.act_grad(dy, y, NA_ACT_RELU, torch.float32, colsum=buf[0], n_cols=N, slots=(S, N + pad))
    terms = dy.float() * (y.float() > 0)
    assert torch.equal(out, terms)
    assert close(buf[:, :N].sum(0), terms) and (buf[:, N:] == 0).all()

    # the narrow layer: dW, db and the input gradient's column sums share the copies
    W, d = torch.randn(1, N, generator=g).cuda(), torch.randn(rows, 1, generator=g).cuda()
    buf = torch.zeros(S, 2 * N + 64, device="cuda")
    dW, cs, db = buf[0, :N], buf[0, N:2 * N], buf[0, 2 * N:]
    dX = torch.empty(rows, N, device="cuda")
    _lib.call("na_linear_narrow_bwd_slots", _lib.ptr(y), N, _lib.dtype_code(dtype), rows, N,
              _lib.ptr(W), 1, _lib.ptr(d), _lib.ptr(dW), _lib.ptr(db), _lib.ptr(dX), N, _lib.NA_F32,
              0, _lib.ptr(y), N, _lib.dtype_code(dtype), NA_ACT_RELU, 1.0, _lib.ptr(cs), S,
              buf.shape[1], _lib.stream_of(y))
    total = buf.sum(0)
    assert close(total[:N], d * y.float()) and close(total[N:2 * N], dX) and close(total[2 * N:2 * N + 1], d)

    # a product's column sums, on the path its type takes
    B = torch.randn(N, N, generator=g).to(dtype).cuda()
    C = torch.empty(rows, N, device="cuda")
    buf = torch.zeros(S, N + pad, device="cuda")
    Fn.gemm(dy, N, 0, B, N, 0, rows, N, N, C, N, dact=NA_ACT_RELU, dact_y=y, ld_dact=N,
            colsum=buf[0], slots=(S, N + pad))
    assert close(buf[:, :N].sum(0), C) and (buf[:, N:] == 0).all()


def test_bad_slots_are_refused():
    a = _lib.GemmArgs()
    assert _lib.load().na_gemm_slots(ctypes.byref(a), 0, 0, None) == _lib.NA_ERR_ARGUMENT
