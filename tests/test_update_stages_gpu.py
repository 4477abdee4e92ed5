"""The update's matrix GEMM over chunks longer and shorter than the 512 directions (32 stages of 16) whose addresses
it forms at once: one direction, the ends of a stage and of a block of 32 stages, and a second and third block.

Tolerance: bf16 has 8 significant bits and rounds by at most 2^-8 of a value, so lo is at most 2^-8 of it and hi + lo
misses it by at most 2^-16; both factors' misses and the dropped lo * lo make 3 * 2^-16 of a product. 3 n fp32 additions
round by 2^-24 each of at most the sum of the products' magnitudes, and the fp32 weights by 2^-21."""
import pytest
import torch

pytestmark = pytest.mark.gpu


class _Params(torch.nn.Module):
    def __init__(self):
        super().__init__()
        self.q = torch.nn.Parameter(torch.zeros(512, 512))
        self.fc = torch.nn.Parameter(torch.zeros(1024, 256))


@pytest.mark.parametrize('pairs', [2, 15, 16, 17, 511, 512, 513, 561, 1041])
def test_long_chunks(pairs):
    from noise_amd.eggroll import Eggroll
    print(pairs, flush=True)
    es = Eggroll(_Params().cuda(), pairs, noise_numel=1 << 22)
    offsets = es.offsets(7)
    losses = torch.randn(2 * pairs, device='cuda', generator=torch.Generator('cuda').manual_seed(pairs))
    g_regen = es.update(losses, offsets, chunk=2048, materialise=False)
    g_buf = es.update(losses, offsets, chunk=2048, materialise=True)
    score = (losses[1::2] - losses[0::2]).double()
    w = (score / (score.std() + 1e-8)) / pairs
    for n, (a, b) in es.noise(offsets, torch.arange(pairs, device='cuda')).items():
        a, b = a.double().reshape(pairs, -1), b.double().reshape(pairs, -1)
        ref = -(a * w[:, None]).T.contiguous() @ b
        mag = (a * w[:, None]).abs().T.contiguous() @ b.abs()
        assert torch.equal(g_regen[n], g_buf[n]), n
        bound = (3 * 2.0 ** -16 + 3 * pairs * 2.0 ** -24 + 2.0 ** -21) * mag
        assert ((g_buf[n].double() - ref).abs() <= bound).all(), n
    # a slice leaving the draw in the last stage, and in the first stage of the last block of 32
    for k, o in ((pairs - 1, es.noise_numel - 700), (pairs // 512 * 512 % pairs, -40)):
        offsets['q'][k] = o
    g_regen = es.update(losses, offsets, chunk=2048, materialise=False)
    g_buf = es.update(losses, offsets, chunk=2048, materialise=True)
    nan = torch.isnan(g_buf['q'])
    assert torch.equal(nan, torch.isnan(g_regen['q']))
    assert torch.equal(torch.nan_to_num(g_buf['q'], nan=0.0), torch.nan_to_num(g_regen['q'], nan=0.0))
    assert nan[:40].all() and not nan[40:, :188].any()


def test_a_slab_of_more_than_2_to_the_30_elements():
    """The last direction of a chunk whose regenerated slices pass 4 GiB, alone in its stage: its copies' byte offsets
    do not fit 32 bits. Its weight outweighs the others', so that another direction's slice in its place shows."""
    from noise_amd.eggroll import Eggroll
    pairs, rows, cols = 16385, 65280, 256
    assert (pairs - 1) * (rows + cols) == 2 ** 30 and pairs % 16 == 1
    p = torch.nn.Module()
    p.wide = torch.nn.Parameter(torch.zeros(rows, cols))
    es = Eggroll(p.cuda(), pairs)
    offsets = es.offsets(3)
    losses = torch.randn(2 * pairs, device='cuda', generator=torch.Generator('cuda').manual_seed(1))
    losses[-1] += 1e4
    one = es.update(losses, offsets, chunk=pairs, materialise=False)['wide']
    three = es.update(losses, offsets, chunk=8192, materialise=False)['wide']
    score = (losses[1::2] - losses[0::2]).double()
    w = (score / (score.std() + 1e-8)) / pairs
    pick = torch.tensor([0, 1, 255, 256, 40000, rows - 1], device='cuda')
    d = torch.arange(pairs, device='cuda')
    a = torch.cat([es.buffer.gather(offsets['wide'] + r, 1, rows=d) for r in pick.tolist()], 1).double()
    b = es.buffer.gather(offsets['wide'] + rows, cols, rows=d).double()
    ref = -(a * w[:, None]).T.contiguous() @ b
    mag = (a * w[:, None]).abs().T.contiguous() @ b.abs()
    bound = (3 * 2.0 ** -16 + 3 * pairs * 2.0 ** -24 + 2.0 ** -21) * mag
    for g in (one, three):
        assert ((g[pick].double() - ref).abs() <= bound).all()
