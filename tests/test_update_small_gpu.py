"""The update's small parameters past the direction count where their slices are drawn once per chunk of directions,
against a float64 contraction of the same device slices: fp32 sums of n terms w a b, each partial sum rounded, stay
within sqrt(n) 2^-24 of the terms' root sum of squares times a small factor; 32 allowed here."""
import pytest
import torch

pytestmark = pytest.mark.gpu


class _Params(torch.nn.Module):
    def __init__(self):
        super().__init__()
        for name, shape in dict(big=(256, 256), gate=(8, 32), lam=(8,), one=(1,), odd=(3, 341), wide=(512,),
                                entries=(32, 32)).items():
            setattr(self, name, torch.nn.Parameter(torch.zeros(*shape)))


@pytest.mark.parametrize('pairs', [4095, 4096, 4097, 8209, 20000])
def test_small_parameters(pairs):
    from noise_amd.eggroll import Eggroll
    print(pairs, flush=True)
    es = Eggroll(_Params().cuda(), pairs)
    offsets = es.offsets(1)
    losses = torch.randn(2 * pairs, device='cuda', generator=torch.Generator('cuda').manual_seed(pairs))
    grads = es.update(losses, offsets)
    f = (losses[1::2] - losses[0::2]).double()
    w = f / (f.std() + 1e-8)
    for name, n in es.noise(offsets, torch.arange(pairs, device='cuda')).items():
        if isinstance(n, tuple):
            a, b = n[0].double(), n[1].double()
            ref, rss = (w[:, None] * a).t() @ b, ((w[:, None] * a).square().t() @ b.square()).sqrt()
        else:
            ref, rss = w @ n.double(), (w.square() @ n.double().square()).sqrt()
        tol = 2e-4 if name == 'big' else 32 * 2.0 ** -24 * pairs ** 0.5
        assert ((grads[name].double() + ref / pairs).abs() <= tol * rss / pairs).all(), name
    again = es.update(losses, offsets)
    assert all(torch.equal(grads[n], again[n]) for n in grads)
