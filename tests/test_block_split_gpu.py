"""The block's split launches (noise_pop_block_split, noise_pop_block_qkv_split, and noise_pop_qkv's shared heads)
against the one-launch block kernel: the same products in the same order and the same reductions, so every output is
equal bit for bit, at every number of parts (by the number of token tiles), with and without noise, value embeddings,
mixing, the split head rows and DUST's jitter."""
import ctypes

import pytest
import torch

from tests.test_block_qkv_gpu import DEV, _case, _common, _rank1

pytestmark = pytest.mark.gpu


def _bits(t):
    return t.view(torch.int16 if t.dtype == torch.bfloat16 else torch.int32)


def _workspace(m, T):
    return torch.full((m * T * (2048 + 4096),), 0xFF, dtype=torch.uint8, device=DEV)


@pytest.mark.parametrize('m,T,noise,ve,ve_noise,rows', [
    (1, 128, None, False, False, False), (3, 256, 'all', True, True, True), (8, 256, 'all', True, True, False),
    (6, 512, 'k', True, False, False), (11, 384, 'all', False, False, False), (9, 1024, 'all', True, True, True),
    (8, 2048, 'all', True, True, False)])
def test_block_qkv(m, T, noise, ve, ve_noise, rows):
    from noise_amd import _lib
    print(m, T, noise, ve, flush=True)
    c = _case(m, T, m * T, noise, ve, ve_noise, rows, block_noise=noise is not None)
    got = []
    # (_common's layout copies of the weights are freed on its return: everything else is allocated before it)
    work, wq = _workspace(m, T), [torch.empty_like(w) for w in c['wq']]
    for w, o in zip(c['wq'], wq):
        _lib.call('noise_block_weight_layout', w.data_ptr(), o.data_ptr(), 512, 512, _lib.stream_ptr(DEV))
    for split in (False, True):
        pop, stream, V, head, xout, outs, r_q, cos, sin, idx_sm = _common(c)
        gate, vn = _rank1(c['rgate']), _rank1(c['rve'])
        ws = (ctypes.c_void_p * 3)(*[w.data_ptr() for w in wq])
        out = (ctypes.c_void_p * 3)(*[o.data_ptr() for o in outs])
        args = (*head, ws, r_q, cos.data_ptr(), sin.data_ptr(), _lib.ptr(c['ve']), 0 if c['ve'] is None else c['ve'].shape[0],
                c['idx'].data_ptr(), idx_sm, _lib.ptr(c['gate_w']), ctypes.byref(gate), ctypes.byref(vn), out)
        if split:
            _lib.call('noise_pop_block_qkv_split', *args, None, work.data_ptr(), work.numel(), stream)
        else:
            _lib.call('noise_pop_block_qkv', *args, stream)
        got.append([xout, *outs])
    for name, a, b in zip(('x', 'q', 'k', 'v'), *got):
        assert torch.equal(_bits(a), _bits(b)), (name, (a.float() - b.float()).abs().max().item())


@pytest.mark.parametrize('m,T,noise,split3', [(2, 128, True, 0), (8, 256, True, 1), (5, 640, False, 0), (4, 2048, True, 1)])
def test_last_block(m, T, noise, split3):
    from noise_amd import _lib
    print(m, T, noise, split3, flush=True)
    c = _case(m, T, m + T, None, False, False, False, block_noise=noise)
    nb = torch.randn(-(-m // 2), 512, device=DEV)
    got = []
    work = _workspace(m, T)
    for split in (False, True):
        h = torch.full((m, T, 512 * (3 if split3 else 1)), 7.0, dtype=torch.bfloat16, device=DEV)
        dots = torch.full((m * T,), 7.0, device=DEV)
        pop, stream, V, head, xout, *_ = _common(c)
        head = head[:11] + (xout.data_ptr(), 0, None, None, None, None, 0, _lib.View(None, 0, 0))
        nxt = (_lib.Rank1 * 1)(_lib.Rank1(None, nb.data_ptr(), 0, 512))
        args = (*head, h.data_ptr(), split3, nxt if noise else None, int(noise), dots.data_ptr() if noise else None)
        if split:
            _lib.call('noise_pop_block_split', *args, None, work.data_ptr(), work.numel(), stream)
        else:
            _lib.call('noise_pop_block', *args, stream)
        got.append((h, dots, xout))
    for a, b in zip(*got):
        assert torch.equal(_bits(a), _bits(b))


@pytest.mark.parametrize('fc,mlp', [(True, False), (False, True), (True, True)])
def test_jitter(fc, mlp):
    from noise_amd import _lib
    m, T = 5, 256
    c = _case(m, T, 77, None, True, False, True, block_noise=False)
    jf = (torch.randn(m, T, 2048, device=DEV) * 0.1).bfloat16() if fc else None
    jm = (torch.randn(m, T, 512, device=DEV) * 0.1).bfloat16() if mlp else None
    zero = torch.zeros(512, dtype=torch.bfloat16, device=DEV)
    js = _lib.BlockJitter(_lib.ptr(jf), _lib.ptr(jm), zero.data_ptr())
    none = _lib.Rank1(None, None, 0, 0)
    got, work = [], _workspace(m, T)
    for split in (False, True):
        pop, stream, V, head, xout, outs, r_q, cos, sin, idx_sm = _common(c)
        ws = (ctypes.c_void_p * 3)(*[w.data_ptr() for w in c['wq']])
        out = (ctypes.c_void_p * 3)(*[o.data_ptr() for o in outs])
        ve = (c['ve'].data_ptr(), c['ve'].shape[0], c['idx'].data_ptr(), idx_sm, c['gate_w'].data_ptr())
        if split:
            _lib.call('noise_pop_block_qkv_split', *head, ws, r_q, cos.data_ptr(), sin.data_ptr(), *ve, ctypes.byref(none),
                      ctypes.byref(none), out, ctypes.byref(js), work.data_ptr(), work.numel(), stream)
        else:
            _lib.call('noise_pop_block_qkv_jit', head[0], head[1], head[2], head[6], head[7], head[9], head[11], head[13],
                      head[14], head[18], ws, cos.data_ptr(), sin.data_ptr(), *ve, out, ctypes.byref(js), stream)
        got.append([xout, *outs])
    for name, a, b in zip(('x', 'q', 'k', 'v'), *got):
        assert torch.equal(_bits(a), _bits(b)), name


def test_the_same_members_alone_and_among_many():
    """Eggroll's losses do not depend on how many members share a launch: 4 members (split launches, shared heads)
    against the same members of 160 x 256 (one workgroup per tile)."""
    from noise_amd.eggroll import Eggroll, Weights, _pair_signs, population_forward
    from noise_amd.model import make_model
    model = make_model('cpu', 0).to(DEV)
    model.lm_head.weight.mul_(30)
    es = Eggroll(model, 80)
    offsets = es.offsets(0)
    g = torch.Generator(DEV).manual_seed(0)
    tokens = torch.randint(0, 4096, (257,), device=DEV, generator=g)
    for fp32_head in (False, True):
        W = Weights(es.params, fp32_head=fp32_head)
        whole = population_forward(W, es.noise_tables(offsets, torch.arange(80, device=DEV)), _pair_signs(80, 0.02, DEV),
                                   tokens[:-1], tokens[1:], dir_div=2)
        part = population_forward(W, es.noise_tables(offsets, torch.tensor([3, 70], device=DEV)), _pair_signs(2, 0.02, DEV),
                                  tokens[:-1], tokens[1:], dir_div=2)
        assert torch.equal(part, whole[[6, 7, 140, 141]])


def test_workspace_is_checked():
    from noise_amd import _lib
    lib = _lib.lib()
    assert lib.noise_block_split_workspace_bytes(8, 256) == 8 * 256 * 6144
    assert lib.noise_block_split_workspace_bytes(512, 2048) == 0 and lib.noise_block_split_workspace_bytes(0, 256) == -1
    c = _case(2, 128, 1, None, False, False, False, block_noise=False)
    pop, stream, V, head, xout, *_ = _common(c)
    h, work = torch.empty(2, 128, 512, dtype=torch.bfloat16, device=DEV), _workspace(2, 128)
    with pytest.raises(RuntimeError, match='workspace'):
        _lib.call('noise_pop_block_split', *head, h.data_ptr(), 0, None, 0, None, None, work.data_ptr(), 100, stream)


@pytest.mark.parametrize('B,T,layer,site', [(1, 256, 1, 'fc'), (1, 512, 0, None), (3, 256, 3, 'attn'), (5, 512, 2, 'mlp'),
                                            (49, 256, 1, 'o'), (49, 256, 1, 'fc'), (56, 256, 5, 'mlp'), (65, 512, 7, 'attn'),
                                            (100, 256, 4, None)])
def test_block_forward_against_the_tiled_kernels(B, T, layer, site):
    """block_forward at few and at many sequences (split launches, one workgroup per tile) against noise_dust_block. Both
    round to bf16 at the same six places (h, q/k/v, weights, y, h, hidden) with sums in other orders: an increment differs by
    less than sqrt(6) 2^-9 = 4.8e-3 of itself."""
    from noise_amd.dust import block_forward, block_forward_tiled
    from noise_amd.model import rotary_tables, window_sizes
    g = torch.Generator(DEV).manual_seed(B + T)
    r = lambda *s: torch.randn(*s, device=DEV, generator=g)
    w = dict(q=r(512, 512) * .044, k=r(512, 512) * .044, v=r(512, 512) * .044, proj=r(512, 512) * .044,
             fc=r(2048, 512) * .044, out=r(512, 2048) * .022, gate=r(8, 32) * .3 if layer % 2 else None)
    ve = r(B, T, 512) if layer % 2 else None
    jit = {site: r(B, T, 2048 if site == 'fc' else 512) * .1} if site else {}
    x = r(B * T * 512 + 1)[1:].view(B, T, 512)  # off the 16 B alignment
    cos, sin = (t.to(DEV) for t in rotary_tables(T))
    got = block_forward(x, w, ve, cos, sin, window_sizes()[layer], **jit)
    ref = block_forward_tiled(x.clone(), w, ve, cos, sin, window_sizes()[layer], **jit)
    rel = float((got - ref).norm() / (ref - x).norm())
    print(B, T, layer, site, rel, flush=True)
    assert rel <= 4.8e-3


def _block_inputs(B, T, seed):
    g = torch.Generator(DEV).manual_seed(seed)
    r = lambda *s: torch.randn(*s, device=DEV, generator=g)
    w = dict(q=r(512, 512) * .044, k=r(512, 512) * .044, v=r(512, 512) * .044, proj=r(512, 512) * .044,
             fc=r(2048, 512) * .044, out=r(512, 2048) * .022, gate=None)
    return r(B, T, 512), w, (r(B, T, 2048) * .1).bfloat16()


@pytest.mark.parametrize('B,T', [(1, 256), (49, 256)])
def test_c_fc_jitter_alone_is_the_one_with_zero_rows(B, T):
    """Without mlp.c_proj jitter the block adds zeros of its own, in the split and in the one-launch form: the bits of
    jitter rows that hold zeros, +0 and -0 products included."""
    from noise_amd.dust import block_forward
    from noise_amd.model import rotary_tables
    x, w, fc = _block_inputs(B, T, B)
    w['out'][::2] = 0
    x[..., ::3] = -0.0
    cos, sin = (t.to(DEV) for t in rotary_tables(T))
    got = block_forward(x, w, None, cos, sin, 128, fc=fc)
    ref = block_forward(x, w, None, cos, sin, 128, fc=fc, mlp=torch.zeros(B, T, 512, dtype=torch.bfloat16, device=DEV))
    assert torch.equal(_bits(got), _bits(ref))


def test_jitter_on_two_streams():
    """A call whose stream is far behind holds nothing that a call on another stream reads: results are the same bits."""
    from noise_amd.dust import block_forward
    from noise_amd.model import rotary_tables
    x, w, fc = _block_inputs(50, 256, 3)
    cos, sin = (t.to(DEV) for t in rotary_tables(256))
    behind, ahead = torch.cuda.Stream(DEV), torch.cuda.Stream(DEV)
    torch.full((1 << 22,), float('nan'), device=DEV)   # blocks freed here and taken again hold no zeros
    torch.cuda.synchronize()
    outs = []
    for stream in (behind, ahead):
        with torch.cuda.stream(stream):
            torch.full((1 << 16,), float('nan'), device=DEV)
            if stream is behind:
                torch.cuda._sleep(20_000_000)
            outs.append(block_forward(x, w, None, cos, sin, 128, fc=fc))
    torch.cuda.synchronize()
    ref = block_forward(x, w, None, cos, sin, 128, fc=fc)
    for out in outs:
        assert torch.equal(_bits(out), _bits(ref))


@pytest.mark.parametrize('fuse_qkv', [True, False])
def test_one_perturbed_matrix_of_q_k_and_v(fuse_qkv):
    """The dot slots of unperturbed matrices beside a perturbed one hold dots with zeros of the call's own: losses are those
    of rank-1 terms that are zero, on any stream."""
    from noise_amd.eggroll import Eggroll, Weights, _pair_signs, population_forward
    from noise_amd.model import make_model
    model = make_model('cpu', 0).to(DEV)
    model.lm_head.weight.mul_(30)
    es = Eggroll(model, 3)
    tokens = torch.randint(0, 4096, (257,), device=DEV, generator=torch.Generator(DEV).manual_seed(0))
    W, sign = Weights(es.params), _pair_signs(3, 0.02, DEV)
    names = [f'transformer.h.{i}.attn.c_{x}.weight' for i in (0, 5) for x in 'kqv']
    offsets = es.offsets(0)
    noise = es.noise_tables({n: offsets[n] for n in names}, torch.arange(3, device=DEV))
    forward = lambda n: population_forward(W, n, sign, tokens[:-1], tokens[1:], dir_div=2, fuse_qkv=fuse_qkv)
    ref = forward({n: v if '.c_k.' in n else (torch.zeros_like(v[0]), v[1]) for n, v in noise.items()})
    alone = {n: v for n, v in noise.items() if '.c_k.' in n}
    assert torch.equal(forward(alone), ref)
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.Stream(DEV)):
        other = forward(alone)
    torch.cuda.synchronize()
    assert torch.equal(other, ref)
