"""noise_head_ce: the head with the vocabulary of a token tile shared out over several workgroups, at row counts on
and off the tiles (the last tile ragged) and with every kernel that serves it. The sums of 128
vocabulary rows are added in order whoever forms them, so a split loss has the unsplit one's bits."""
import ctypes
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device('cuda', 0)


def _loss64(logits, targets):
    z = 15 * torch.tanh(logits / 15)
    ce = torch.logsumexp(z, -1) - z.gather(-1, targets.clamp(0, 4095)[..., None])[..., 0]
    ce = torch.where(targets == -1, torch.zeros_like(ce), ce)
    return torch.where((targets < -1) | (targets >= 4096), torch.full_like(ce, float('nan')), ce)


def _targets(rows, g):
    y = torch.randint(0, 4096, (rows,), device=DEV, generator=g)
    y[0] = 4095
    if rows > 3:
        y[1], y[2], y[rows - 1] = -1, 0, 4096
    return y


@pytest.mark.parametrize('rows', [1, 15, 16, 127, 128, 129, 300, 3000, 33000])
def test_fp32_rows_against_64_bits(rows):
    """The head_loss drop-in: fp32 rows split in the kernel, normed in the logits. bf16 rounds by at most 2^-8 of a value, so a
    term h w of a logit loses at most 3 x 2^-16 of itself (lo lo, and the rounding of both lo halves); the 512 terms' losses
    have either sign, and a quarter of the sum of their bounds is allowed. The loss takes at most two logits' errors, and
    the fp32 sums and the exponentials add 1e-5."""
    from noise_amd.dust import head_loss
    print(rows, flush=True)
    g = torch.Generator(DEV).manual_seed(rows)
    x, w = torch.randn(rows, 512, device=DEV, generator=g) * 3, torch.randn(4096, 512, device=DEV, generator=g) * 0.1
    y = _targets(rows, g)
    got = head_loss(x, w, y, 4096).double()
    xd = x.double()
    h = xd * torch.rsqrt(xd.square().mean(-1, keepdim=True) + 1.1920928955078125e-07)
    ref = _loss64(h @ w.double().t(), y)
    bound = 2 * 3 * 2.0 ** -18 * (h.abs() @ w.double().abs().t()).amax(-1) + 1e-5
    assert torch.equal(got.isnan(), ref.isnan())
    assert ((got - ref).nan_to_num().abs() <= bound).all()
    odd = torch.empty(rows * 512 + 1, device=DEV)[1:].view(rows, 512).copy_(x)   # off the 16 B alignment
    assert torch.equal(head_loss(odd, w, y, 4096).nan_to_num(), got.float().nan_to_num())


@pytest.mark.parametrize('K', [512, 1536])
@pytest.mark.parametrize('m,T,pert,eager', [(1, 256, False, False), (3, 256, True, False), (2, 768, False, True),
                                            (5, 131, True, False), (300, 256, True, False)])
def test_split_equals_unsplit(K, m, T, pert, eager):
    from noise_amd import _lib
    if eager and K == 1536:
        pytest.skip('eager rounding is for the bf16 head')
    print(K, m, T, pert, eager, flush=True)
    g = torch.Generator(DEV).manual_seed(m * T)
    x = torch.randn(m, T, K, device=DEV, generator=g).bfloat16()
    w = (torch.randn(4096, K, device=DEV, generator=g) * 0.2).bfloat16()
    y = _targets(T, g)
    sign = torch.randn(m, device=DEV, generator=g) * 0.1
    dots = torch.randn(m * T, device=DEV, generator=g)
    a = torch.randn(-(-m // 2), 4096, device=DEV, generator=g)
    r1 = _lib.Rank1(a.data_ptr(), a.data_ptr(), 4096, 4096) if pert else _lib.Rank1(None, None, 0, 0)
    pop = _lib.Population(m, T, sign.data_ptr(), 2, _lib.ROUNDING_EAGER if eager else _lib.ROUNDING_FUSED)
    ws, need = _lib.head_workspace(m, T, K, 4096, DEV)
    out = []
    for work in (ws, None):
        loss = torch.full((m, T), -7.0, device=DEV)
        _lib.call('noise_head_ce', ctypes.byref(pop), _lib.View(x.data_ptr(), T * K, K), 0, w.data_ptr(), K, 4096,
                  ctypes.byref(r1), dots.data_ptr(), y.data_ptr(), 0, loss.data_ptr(), _lib.ptr(work), need if work is not None else 0,
                  _lib.stream_ptr(DEV))
        out.append(loss)
    assert (m * T > 100000) == (need == 0) or need > 0
    assert torch.equal(out[0].isnan(), out[1].isnan())
    assert torch.equal(out[0].nan_to_num(), out[1].nan_to_num())


@pytest.mark.parametrize('rows', [40, 33000])
def test_rows_whose_squares_overflow(rows):
    """Finite rows whose sum of squares passes fp32 norm to zeros (x rsqrt(inf), utils/model.py:46-47 in fp32), whatever
    their products with the weights come to; an infinity or a NaN among the values makes the loss NaN."""
    from noise_amd.dust import head_loss
    g = torch.Generator(DEV).manual_seed(rows)
    x, w = torch.randn(rows, 512, device=DEV, generator=g), torch.randn(4096, 512, device=DEV, generator=g)
    y = torch.randint(0, 4096, (rows,), device=DEV, generator=g)
    plain = head_loss(x, w, y, 4096)
    big = torch.finfo(torch.float32).max
    x[3], x[7], x[17], x[21] = big, 1e30 * x[7], -big * torch.rand(512, device=DEV, generator=g), 3e19 * x[21]
    x[5, 9], x[6, 1] = float('inf'), float('nan')
    x[8, 500] = big
    got = head_loss(x, w, y, 4096)
    zeros, bad = [3, 7, 17, 21, 8], [5, 6]
    assert ((got[zeros] - math.log(4096)).abs() <= 1e-5).all()
    assert got[bad].isnan().all()
    keep = torch.ones(rows, dtype=torch.bool, device=DEV)
    keep[zeros + bad] = False
    assert torch.equal(got[keep], plain[keep])
