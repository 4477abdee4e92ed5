"""The one-launch preparations of an update, bit for bit: Weights (noise_weights_prepare) against torch's casts and
the block layout's formula, DeviceGenerator.randint_many against torch.randint on a device generator, and
Eggroll.noise_tables against Eggroll.noise for every parameter."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = torch.device('cuda', 0)


def _block_order(w):
    r, c = w.shape
    g = w.view(r, c // 32, 8, 4)
    return g[:, :, [0, 4, 1, 5, 2, 6, 3, 7]].reshape(r, c)


@pytest.mark.parametrize('fp32_embeddings', [True, False])
def test_weights_are_the_parameters(fp32_embeddings):
    from noise_amd.eggroll import Weights
    from noise_amd.model import make_model
    model = make_model(DEV, 3, fp32_embeddings=fp32_embeddings)
    for q in model.parameters():
        if q.dim() == 1 or q.shape[0] == 8:
            q.copy_(torch.randn(q.shape, device=DEV))
    p = dict(model.named_parameters())
    p['transformer.h.2.attn.c_q.weight'] = p['transformer.h.2.attn.c_q.weight'].t().contiguous().t()  # not contiguous
    odd = torch.empty(512 * 512 + 1, device=DEV)[1:].view(512, 512).copy_(p['transformer.h.3.attn.c_k.weight'])
    p['transformer.h.3.attn.c_k.weight'] = odd  # off the 16 B alignment
    p['transformer.h.4.attn.c_v.weight'] = p['transformer.h.4.attn.c_v.weight'].double()
    W = Weights(p)
    keys = dict(q='attn.c_q', k='attn.c_k', v='attn.c_v', o='attn.c_proj', fc='mlp.c_fc', mp='mlp.c_proj')
    for i, blk in enumerate(W.blocks):
        for k, name in keys.items():
            ref = p[f'transformer.h.{i}.{name}.weight'].bfloat16()
            assert torch.equal(blk[k], ref), (i, k)
            if k + '_blk' in blk:
                assert torch.equal(blk[k + '_blk'], _block_order(ref)), (i, k)
        assert ('q_blk' in blk) == (i > 0) and 'fc_blk' in blk and 'mp_blk' in blk
        if 'gate' in blk:
            assert torch.equal(blk['gate'], p[f'transformer.h.{i}.attn.ve_gate.weight'].bfloat16().float())
            assert torch.equal(blk['ve'], p[f'value_embeds.{i}.weight'].float())
    assert torch.equal(W.wte, p['transformer.wte.weight'].float()) and torch.equal(W.lm_head, p['lm_head.weight'].bfloat16())
    assert torch.equal(W.resid_lambdas, p['resid_lambdas']) and torch.equal(W.x0_lambdas, p['x0_lambdas'])
    p['x0_lambdas'].add_(1)
    assert not torch.equal(W.x0_lambdas, p['x0_lambdas'])  # a snapshot


@pytest.mark.parametrize('numel', [1, 7, 8, 2047, 2049])
@pytest.mark.parametrize('kind', [0, 1, 2])
def test_entry_tails(numel, kind):
    from noise_amd import _lib
    src = torch.randn(numel, device=DEV)
    dst = torch.full((numel + 8,), 5.0, device=DEV, dtype=torch.bfloat16 if kind == 0 else torch.float32)
    table = (_lib.Weight * 1)(_lib.Weight(src.data_ptr(), dst.data_ptr(), None, numel, 0, kind))
    _lib.call('noise_weights_prepare', table, 1, _lib.stream_ptr(DEV))
    ref = [src.bfloat16(), src, src.bfloat16().float()][kind]
    assert torch.equal(dst[:numel], ref) and (dst[numel:] == 5).all()


@pytest.mark.parametrize('n,count', [(1, 1), (5, 64), (300, 65), (70000, 3), (2 ** 21 + 3, 2)])
def test_randint_many_is_torch(n, count):
    from noise_amd.noise import DeviceGenerator
    highs = [2 ** 28 - 1 - 977 * k for k in range(count)]
    g, t = DeviceGenerator(11, DEV), torch.Generator(DEV).manual_seed(11)
    got = g.randint_many(highs, n)
    for k, h in enumerate(highs):
        assert torch.equal(got[k], torch.randint(0, h, (n,), device=DEV, generator=t)), k
    assert torch.equal(g.randint(0, 1000, 9), torch.randint(0, 1000, (9,), device=DEV, generator=t))


def test_noise_tables_are_the_noise():
    from noise_amd.eggroll import Eggroll
    from noise_amd.model import make_model
    es = Eggroll(make_model('cpu', 0).to(DEV), 7)
    offsets = es.offsets(2)
    directions = torch.tensor([6, 0, 3], device=DEV)
    tables, ref = es.noise_tables(offsets, directions), es.noise(offsets, directions)
    assert set(tables) == set(ref)
    for n, v in ref.items():
        for a, b in zip(v if isinstance(v, tuple) else (v,), tables[n] if isinstance(v, tuple) else (tables[n],)):
            assert torch.equal(a, b), n


def test_rotary_tables_are_complete_when_cached():
    """The rotary tables are shared by every stream: nothing that fills them is left on the first caller's stream."""
    from noise_amd.eggroll import _rope_tables
    from noise_amd.model import rotary_tables
    stream = torch.cuda.Stream(DEV)
    with torch.cuda.stream(stream):
        torch.cuda._sleep(2_000_000)
        cos, sin = _rope_tables(1003, DEV)   # (no other test's length)
        assert stream.query()
    for got, ref in zip((cos, sin), rotary_tables(1003)):
        assert got.dtype == torch.bfloat16 and got.is_contiguous() and torch.equal(got.cpu(), ref.bfloat16())


def test_small_parameters_of_any_number_of_directions():
    """Parameters whose slices are no whole 256s are gathered for more directions than one launch of the table serves."""
    from noise_amd.eggroll import Eggroll
    pairs = 65536 + 70
    p = torch.nn.Module()
    p.lam, p.gate, p.mat = (torch.nn.Parameter(torch.zeros(*s)) for s in ((8,), (8, 32), (256, 256)))
    es = Eggroll(p.to(DEV), pairs)
    offsets = es.offsets(1)
    directions = torch.arange(pairs, device=DEV).flip(0)
    small = {n: offsets[n] for n in ('lam', 'gate')}
    tables, ref = es.noise_tables(small, directions), es.noise(offsets, directions)
    assert torch.equal(tables['lam'], ref['lam']) and all(torch.equal(a, b) for a, b in zip(tables['gate'], ref['gate']))
    with pytest.raises(ValueError, match='65535'):
        es.noise_tables(offsets, directions)


def test_parameters_that_are_neither_vectors_nor_matrices():
    """Their slice is one row per direction (eggroll.py:127-128), and the parameters after them keep their columns."""
    from noise_amd.eggroll import Eggroll
    p = torch.nn.Module()
    p.cube, p.lam, p.mat = (torch.nn.Parameter(torch.zeros(*s)) for s in ((2, 3, 4), (8,), (8, 32)))
    es = Eggroll(p.to(DEV), 5)
    offsets, directions = es.offsets(0), torch.arange(5, device=DEV)
    tables, ref = es.noise_tables(offsets, directions), es.noise(offsets, directions)
    assert torch.equal(tables['cube'], ref['cube']) and torch.equal(tables['lam'], ref['lam'])
    assert all(torch.equal(a, b) for a, b in zip(tables['mat'], ref['mat']))
