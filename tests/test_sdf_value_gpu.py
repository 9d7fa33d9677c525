"""SDF values in one kernel (encoding, first layer, softplus, head) against float64 over the
same encoding: tiles of 64 points and their remainders, each grid and hidden width that the
kernel covers, inactive levels, and values that no bf16 split holds."""
import ctypes

import pytest
import torch

from neuralangelo_amd import _lib
from neuralangelo_amd import functional as Fn
from neuralangelo_amd.encoding import Encoding, growth_rate

pytestmark = pytest.mark.gpu


def _setup(F, hidden, cdt, active, seed=0):
    g = torch.Generator().manual_seed(seed)
    enc = Encoding(3, dict(n_levels=16, n_features_per_level=F, log2_hashmap_size=14,
                           base_resolution=8, per_level_scale=growth_rate(3, 9, 16)), dtype=cdt).cuda()
    enc.vol_range, enc.active_levels = (-1.0, 1.0), active
    with torch.no_grad():
        enc.params.copy_(torch.randn(enc.params.shape, generator=g) * 0.3)
    n = 16 * F
    W0 = (torch.randn(hidden, 3 + n, generator=g) * 0.1).cuda()
    b0, bs = torch.randn(hidden, generator=g).cuda() * 0.1, torch.randn(1, generator=g).cuda()
    ws = torch.randn(1, hidden, generator=g).cuda()
    return enc, Fn.SDFWeights(W0, b0, None, None, ws, bs, n, cdt), g


def _covered(enc, w):
    table = enc.table_for_forward()
    return table.dtype == w.cdt and _lib.call("na_sdf_value_supported", ctypes.byref(enc.desc),
                                              Fn._code(table), w.hidden)


def _reference(enc, w, x):
    """float64 products over the kernels' own encoding, and the sum of the magnitudes."""
    X = Fn.sdf_input(enc, x, w.cdt, w.k0p).double()[:, :w.n_enc]
    W = w.W0p.double()
    n = w.n_enc
    Wx = W[:, n:n + 3] + (W[:, n + 6:n + 9] if w.split else 0.0)
    z = X @ W[:, :n].t() + x.double() @ Wx.t() + w.b0.double()
    az = X.abs() @ W[:, :n].abs().t() + x.double().abs() @ Wx.abs().t() + w.b0.double().abs()
    h = torch.nn.functional.softplus(z, beta=100)
    ref = h @ w.ws.double().t() + w.bs.double()
    # one float32 rounding per addition, in each layer (and the softplus, 1e-7 absolute, 2^-21)
    eh = (w.k0p + 8) * 2.0 ** -23 * az + 1e-7 + 2.0 ** -21 * h
    e = (eh + (w.hidden + 8) * 2.0 ** -23 * h) @ w.ws.double().abs().t() + 2.0 ** -22 * ref.abs()
    return ref, e


@pytest.mark.parametrize("cdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("F,hidden,active", [(8, 256, 16), (8, 128, 16), (4, 256, 16), (4, 128, 16),
                                             (8, 256, 4), (4, 256, 3), (8, 128, 1), (8, 256, 0)])
def test_sdf_value(F, hidden, active, cdt):
    enc, w, g = _setup(F, hidden, cdt, active)
    assert _covered(enc, w)
    for P in (1, 63, 64, 65, 1000, 20001):
        x = (torch.rand(P, 3, generator=g) * 2.2 - 1.1).cuda()
        with torch.no_grad():
            got = Fn.sdf_forward_nograd(enc, w, x).double()
            ref, e = _reference(enc, w, x)
        assert got.shape == (P, 1) and ((got - ref).abs() <= e).all()


def test_sdf_value_no_points():
    enc, w, _ = _setup(8, 256, torch.float32, 16)
    with torch.no_grad():
        assert Fn.sdf_forward_nograd(enc, w, torch.zeros(0, 3, device="cuda")).shape == (0, 1)


@pytest.mark.parametrize("value", [float("inf"), -float("inf"), float("nan"), 3.4e38, 1e-30])
def test_sdf_value_unsplittable(value):
    """float32 weights that are not finite, or whose bf16 parts would overflow."""
    enc, w, g = _setup(4, 256, torch.float32, 16)
    w.W0p[5, 7] = value
    x = (torch.rand(130, 3, generator=g) * 2 - 1).cuda()
    with torch.no_grad():
        X = Fn.sdf_input(enc, x, w.cdt, w.k0p).double()
        z = X @ w.W0p.double().t() + w.b0.double()
        ref = torch.nn.functional.softplus(z, beta=100) @ w.ws.double().t() + w.bs.double()
        got = Fn.sdf_forward_nograd(enc, w, x).double()
    if abs(value) > 1e37 or value != value:
        nan, small = ref.isnan(), ref.abs() < 1e30
        assert (got.isnan() == nan).all()
        assert (got[small] - ref[small]).abs().max() <= 1e-3 if small.any() else True
        big = ~nan & ~small
        assert (torch.sign(got[big]) == torch.sign(ref[big])).all() and (got[big].abs() > 1e29).all()
    else:
        assert (got - ref).abs().max() <= 1e-3


@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3.4e38])
@pytest.mark.parametrize("F,hidden", [(8, 256), (8, 128), (4, 256), (4, 128)])
def test_sdf_value_recomputed_tile(F, hidden, value):
    """One bad entry of a float32 table: its tile is formed again in float32, the points that
    read the entry follow it, and the tile's other points keep their accuracy."""
    enc, w, g = _setup(F, hidden, torch.float32, 16)
    x = (torch.rand(200, 3, generator=g) * 2 - 1).cuda()
    with torch.no_grad():
        idx, wt = enc.corners((x + 1.0) / 2.0)
        entry = int(idx[70, 15, 3])  # a corner of point 70 at the finest level
        enc.params.view(-1, F)[entry, F - 1] = value
        hit = (idx == entry).flatten(1).any(1)
        assert hit[70] and hit[64:128].sum() < 8
        got = Fn.sdf_forward_nograd(enc, w, x).double()
        ref, e = _reference(enc, w, x)
    assert ((got - ref).abs() <= e)[~hit].all()
    if abs(value) != 3.4e38:
        assert not got[hit].isfinite().any() and not ref[hit].isfinite().any()
