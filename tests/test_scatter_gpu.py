"""The table-gradient scatter at the sizes where its batches, runs and row loads end,
against a float64 sum over the encoder's own corner indices and weights."""
import ctypes

import pytest
import torch

from neuralangelo_amd import _lib
from neuralangelo_amd.encoding import Encoding, growth_rate

pytestmark = pytest.mark.gpu


def ray_points(n, seed):
    """Samples along a few rays (runs of points that share cells or corners), some of
    them past the unit cube's faces."""
    g = torch.Generator().manual_seed(seed)
    o, v = torch.rand(8, 3, generator=g) * 1.1 - 0.05, torch.randn(8, 3, generator=g) * 0.004
    k = torch.arange(n)
    return (o[k // 40 % 8] + v[k // 40 % 8] * (k % 40)[:, None].float()).contiguous()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("F", [1, 2, 4, 8])
@pytest.mark.parametrize("n, pad", [(1, 0), (63, 1), (64, 0), (65, 3), (1000, 8), (40013, 0)])
def test_scatter_sizes_and_row_alignment(F, dtype, n, pad):
    L, active = 16, 13
    enc = Encoding(3, dict(n_levels=L, n_features_per_level=F, log2_hashmap_size=14,
                           base_resolution=8, per_level_scale=growth_rate(3, 9, L))).cuda()
    x = ray_points(n, n).cuda()
    g = torch.Generator().manual_seed(n + F)
    rows = torch.randn(n, L * F + pad, generator=g).to(dtype).cuda()
    rows[::5] = 0  # samples without a gradient
    dy = rows[:, pad:]  # pad 1, 3: rows without the vector loads' alignment
    grad = torch.zeros(enc.n_params, device="cuda")
    _lib.call("na_sdf_input_bwd", ctypes.byref(enc.desc), _lib.ptr(x), n, 0.0, 1.0,
              _lib.ptr(dy), _lib.dtype_code(dtype), L * F + pad, _lib.ptr(grad), active,
              _lib.stream_of(x))
    idx, w = enc.corners(x)
    add = w.double()[..., None] * dy.double().view(n, L, 1, F)
    add[:, active:] = 0
    rows64 = [torch.zeros(enc.n_params // F, k, dtype=torch.float64, device="cuda") for k in (F, F, 1)]
    at = idx.long().reshape(-1)
    for r, v in zip(rows64, (add, add.abs(), torch.ones_like(add[..., :1]))):
        r.index_add_(0, at, v.reshape(at.numel(), -1))
    ref, size, count = rows64
    # one rounding per contribution and one per addition, in any order
    bound = (count + 2) * 2.0 ** -23 * size
    assert ((grad.view(-1, F).double() - ref).abs() <= bound).all()
    assert (grad.view(-1, F)[enc.offsets[active]:] == 0).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("F", [1, 2, 4, 8])
@pytest.mark.parametrize("n, eps", [(1, 1e-3), (15, 1e-3), (17, 2e-3), (1003, 0.0), (1003, 1e-3), (1003, 0.02)])
def test_tap_scatter_pairs(F, dtype, n, eps):
    """The centre-and-taps scatter, whose lanes own the even or the odd x of a box: every
    start parity, runs cut by the end, cells wider apart than the box (eps 0.02)."""
    from neuralangelo_amd import functional as Fn
    L, active = 16, 14
    enc = Encoding(3, dict(n_levels=L, n_features_per_level=F, log2_hashmap_size=14,
                           base_resolution=8, per_level_scale=growth_rate(3, 9, L))).cuda()
    x = ray_points(n, n).cuda()
    g = torch.Generator().manual_seed(n + F)
    dyc = torch.randn(n, L * F, generator=g).to(dtype).cuda()
    dyt = torch.randn(4 * n, L * F, generator=g).to(dtype).cuda()
    dyc[::5] = 0
    dyt[3::7] = 0
    grad = torch.zeros(enc.n_params, device="cuda")
    _lib.call("na_sdf_taps_bwd", ctypes.byref(enc.desc), _lib.ptr(x), n, 0.0, 1.0, float(eps),
              _lib.ptr(dyc), _lib.ptr(dyt), None, _lib.dtype_code(dtype), L * F, _lib.ptr(grad),
              active, 0, _lib.stream_of(x))
    idx, w = enc.corners(torch.cat([x, Fn.taps_points(x, eps).view(-1, 3)]))
    add = w.double()[..., None] * torch.cat([dyc, dyt]).double().view(5 * n, L, 1, F)
    add[:, active:] = 0
    rows64 = [torch.zeros(enc.n_params // F, k, dtype=torch.float64, device="cuda") for k in (F, F, 1)]
    at = idx.long().reshape(-1)
    for r, v in zip(rows64, (add, add.abs(), torch.ones_like(add[..., :1]))):
        r.index_add_(0, at, v.reshape(at.numel(), -1))
    ref, size, count = rows64
    # three roundings of the weight, one of its product with the gradient, one per addition
    bound = (count + 6) * 2.0 ** -23 * size
    assert ((grad.view(-1, F).double() - ref).abs() <= bound).all()
    assert (grad.view(-1, F)[enc.offsets[active]:] == 0).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("F", [1, 2, 4, 8])
@pytest.mark.parametrize("n, shared", [(1, True), (17, False), (1003, True)])
def test_tap_scatter_increments(F, dtype, n, shared):
    """Point-major tap rows with and without the row that the four taps share: the two lanes of
    a feature load half of a point's rows each and exchange them."""
    from neuralangelo_amd import functional as Fn
    L, active, eps = 16, 14, 1e-3
    enc = Encoding(3, dict(n_levels=L, n_features_per_level=F, log2_hashmap_size=14,
                           base_resolution=8, per_level_scale=growth_rate(3, 9, L))).cuda()
    x = ray_points(n, n).cuda()
    g = torch.Generator().manual_seed(n + F)
    dyc = torch.randn(n, L * F, generator=g).to(dtype).cuda()
    dyt = torch.randn(n, 4, L * F, generator=g).to(dtype).cuda()
    dyq = torch.randn(n, L * F, generator=g).to(dtype).cuda() if shared else None
    for t in (dyc, dyt) + ((dyq,) if shared else ()):
        t[::5] = 0
    grad = torch.zeros(enc.n_params, device="cuda")
    _lib.call("na_sdf_taps_bwd", ctypes.byref(enc.desc), _lib.ptr(x), n, 0.0, 1.0, float(eps),
              _lib.ptr(dyc), _lib.ptr(dyt), _lib.ptr(dyq), _lib.dtype_code(dtype), L * F,
              _lib.ptr(grad), active, 1, _lib.stream_of(x))
    gt = dyt.float() + (dyq.float()[:, None] if shared else 0.0)
    gc = dyc.float() - ((gt[:, 0] + gt[:, 1]) + (gt[:, 2] + gt[:, 3]))
    idx, w = enc.corners(torch.cat([x, Fn.taps_points(x, eps).view(-1, 3)]))
    rows = torch.cat([gc, gt.transpose(0, 1).reshape(4 * n, -1)]).double()
    add = w.double()[..., None] * rows.view(5 * n, L, 1, F)
    add[:, active:] = 0
    rows64 = [torch.zeros(enc.n_params // F, k, dtype=torch.float64, device="cuda") for k in (F, F, 1)]
    at = idx.long().reshape(-1)
    for r, v in zip(rows64, (add, add.abs(), torch.ones_like(add[..., :1]))):
        r.index_add_(0, at, v.reshape(at.numel(), -1))
    ref, size, count = rows64
    # three roundings of the weight, one of its product with the gradient, one per addition
    assert ((grad.view(-1, F).double() - ref).abs() <= (count + 6) * 2.0 ** -23 * size).all()
