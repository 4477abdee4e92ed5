"""The work that users of noise_amd have it do, as cases that a timing program can run.

Six kinds of call, each through the entry point a program uses:

  attention    noise_amd.model.attention: the drop-in of every attention layer (prefill; any length, both windows)
  lowrank      noise_amd.eggroll.lowrank: a perturbed linear layer of a population
  block        noise_amd.dust.block_forward: one transformer block with jitter at a site
  head         noise_amd.dust.head_loss: the fp32 head with its per-token cross-entropy
  population   Eggroll.population: one update's population losses (weights laid out, noise drawn, forward)
  update       Eggroll.update: the gradients from one update's losses

Widths are those of the fixed model (512, heads of 64, 2048 hidden, 4096 tokens); lengths, members, pairs and batch
sizes run over what the entry points take.
"""
import math

import torch

from noise_amd.dust import block_forward, head_loss
from noise_amd.eggroll import BLOCK_MATRIX_SUFFIXES, SEED, SIGMA, Eggroll, lowrank
from noise_amd.model import attention, has_ve, make_model, rotary_tables, window_sizes

DEV = 'cuda'
F64 = torch.float64
H, D, E, VOCAB, LAYERS = 8, 64, 512, 4096, 8
NOISE = 2 ** 28
DTYPES = {'bf16': torch.bfloat16, 'fp32': torch.float32}
# (in, out) of the model's matrices: attention projections, c_fc, mlp.c_proj, the head, the value-embedding gate
LINEARS = [(512, 512), (512, 2048), (2048, 512), (512, 4096), (32, 8)]


def listed():
    return [
        # a short prompt through one attention layer: the call itself is what counts
        dict(name='attention-least', kind='attention', batch=1, length=100, window=64, dtype='bf16', packed=False),
        # the model's long-window layer on a batch of training sequences
        dict(name='attention-prefill', kind='attention', batch=16, length=2048, window=2048, dtype='bf16',
             packed=False),
        # documents of an odd length, q, k and v in fp32 as autocast leaves them after the norm
        dict(name='attention-ragged', kind='attention', batch=5, length=1111, window=500, dtype='fp32', packed=False),
        # the value-embedding gate of a small population: h[..., :32] through its [8, 32] weight
        dict(name='lowrank-gate', kind='lowrank', members=16, tokens=256, n_in=32, n_out=8, shared=False, div=1,
             dtype='fp32'),
        # mlp.c_fc of a small population on sequences of an odd length
        dict(name='lowrank-ragged', kind='lowrank', members=24, tokens=1000, n_in=512, n_out=2048, shared=False,
             div=1, dtype='fp32'),
        # the antithetic perturbed linear layer on one shared input, 512 members
        dict(name='lowrank-shared', kind='lowrank', members=512, tokens=2048, n_in=512, n_out=2048, shared=True,
             div=2, dtype='bf16'),
        # one block of DUST's rerun on a batch of 8 sequences, jittered at its c_fc
        dict(name='block-batch', kind='block', batch=8, length=2048, layer=1, site='fc'),
        # the fp32 head on three sequences of an odd length
        dict(name='head-ragged', kind='head', batch=3, length=1000),
        # the smallest population, every parameter perturbed, as Eggroll.step does
        dict(name='population-least', kind='population', pairs=4, length=256, perturbed='all', fp32_head=False),
        # one chunk of a full population: 512 members on 2048 tokens, the block matrices perturbed
        dict(name='population-chunk', kind='population', pairs=256, length=2048, perturbed='blocks',
             fp32_head=False),
        # gradients of a 512-pair population, every parameter
        dict(name='update-ordinary', kind='update', pairs=512),
        # gradients at the record run's population
        dict(name='update-largest', kind='update', pairs=131072),
    ]


def _log(rng, low, high):
    """A whole number from low .. high, spread over the logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(['attention', 'attention', 'lowrank', 'lowrank', 'block', 'head', 'population', 'update'])
    if kind == 'attention':
        length = _log(rng, 16, 2048)
        return dict(kind=kind, batch=_log(rng, 1, 24), length=length, window=_log(rng, 16, 2048),
                    dtype=rng.choice(['bf16', 'fp32']), packed=rng.random() < 0.3)
    if kind == 'lowrank':
        n_in, n_out = rng.choice(LINEARS)
        members, tokens, shared = _log(rng, 1, 512), _log(rng, 16, 2048), rng.random() < 0.3
        if rng.random() < 0.4:
            tokens = max(256, tokens - tokens % 256)
        if shared and tokens % 256 == 0 and n_in == 512:
            members = min(members, 2 ** 31 // (tokens * n_out))    # the members' outputs bound it
        else:
            members = min(members, 24_000 * 2048 * 512 // (tokens * n_in * n_out))
        return dict(kind=kind, members=max(1, members), tokens=tokens, n_in=n_in, n_out=n_out, shared=shared,
                    div=rng.choice([1, 2]), dtype=rng.choice(['bf16', 'fp32']))
    if kind == 'block':
        return dict(kind=kind, batch=_log(rng, 1, 32), length=256 * rng.randint(1, 8), layer=rng.randint(0, 7),
                    site=rng.choice(['none', 'o', 'attn', 'fc', 'mlp']))
    if kind == 'head':
        return dict(kind=kind, batch=_log(rng, 1, 16), length=_log(rng, 16, 2048))
    if kind == 'population':
        return dict(kind=kind, pairs=_log(rng, 1, 96), length=256 * rng.randint(1, 8),
                    perturbed=rng.choice(['all', 'blocks']), fp32_head=rng.random() < 0.3)
    return dict(kind=kind, pairs=_log(rng, 2, 131072))


# --- inputs ---


def _perturbed(case, model):
    """Names of the perturbed parameters (None: all of them, as Eggroll.step)."""
    if case['perturbed'] == 'all':
        return None
    return [n for n, _ in model.named_parameters()
            if n.startswith('transformer.h.') and n.endswith(BLOCK_MATRIX_SUFFIXES)]


def _model(seed):
    """A model whose head has grown, as training grows it (at initialisation the loss does not depend on the
    blocks)."""
    model = make_model(DEV, seed)
    with torch.no_grad():
        model.lm_head.weight.mul_(30)
    return model


def prepare(case, seed):
    g = torch.Generator(DEV).manual_seed(seed)
    randn = lambda *s, dtype=torch.float32: torch.randn(*s, device=DEV, generator=g).to(dtype)
    kind = case['kind']
    s = dict(case=dict(case), kind=kind)
    if kind == 'attention':
        shape = (case['batch'], case['length'], H, D)
        dt = DTYPES[case['dtype']]
        unit = lambda t: torch.nn.functional.rms_norm(t, (D,))   # q and k come out of the head norm
        q, k, v = unit(randn(*shape)), unit(randn(*shape)), randn(*shape)
        if case['packed']:
            q, k, v = torch.stack([q, k, v], 2).to(dt).unbind(2)
        s.update(q=q.to(dt), k=k.to(dt), v=v.to(dt), window=case['window'])
    elif kind == 'lowrank':
        m, T, n_in, n_out, dt = case['members'], case['tokens'], case['n_in'], case['n_out'], DTYPES[case['dtype']]
        rows = 1 if case['shared'] else m
        if n_in == 32:
            x = randn(rows, T, E, dtype=dt)[..., :32]   # the gate reads the first columns of the block input
        else:
            x = randn(rows, T, n_in, dtype=dt)
        dirs = -(-m // case['div'])
        sign = torch.full((m,), SIGMA, device=DEV)
        sign[1::2] = -SIGMA
        s.update(x=x.expand(m, T, n_in) if case['shared'] else x, sign=sign, div=case['div'],
                 weight=randn(n_out, n_in) * n_in ** -0.5, a=randn(dirs, n_out), b=randn(dirs, n_in))
    elif kind == 'block':
        B, T, layer = case['batch'], case['length'], case['layer']
        w = dict(q=randn(E, E) * 0.044, k=randn(E, E) * 0.044, v=randn(E, E) * 0.044, gate=None,
                 proj=randn(E, E) * 0.044, fc=randn(4 * E, E) * 0.044, out=randn(E, 4 * E) * 0.022)
        ve = None
        if has_ve(layer):
            w['gate'] = randn(8, 32) * 0.3
            ve = randn(B, T, E, dtype=torch.bfloat16)
        jitter = {}
        if case['site'] != 'none':
            width = 4 * E if case['site'] == 'fc' else E
            draws = torch.randint(0, 2, (B, T, width), device=DEV, generator=g) * 2 - 1
            jitter[case['site']] = (0.1 * draws).bfloat16()
        cos, sin = (t.bfloat16().to(DEV) for t in rotary_tables(T))
        s.update(x=randn(B, T, E), w=w, ve=ve, cos=cos, sin=sin, window=window_sizes()[layer], jitter=jitter)
    elif kind == 'head':
        shape = (case['batch'], case['length'])
        y = torch.randint(0, VOCAB, shape, device=DEV, generator=g)
        y[:, 0] = -1
        s.update(x=randn(*shape, E) * 2, weight=randn(VOCAB, E) * 0.03, y=y)
    elif kind == 'population':
        model = _model(seed)
        tokens = torch.randint(0, VOCAB, (1, case['length'] + 1), device=DEV, generator=g)
        s.update(es=Eggroll(model, case['pairs']), step=seed % 4096, x=tokens[:, :-1], y=tokens[:, 1:],
                 names=_perturbed(case, model), fp32_head=case['fp32_head'])
    else:
        model = _model(seed)
        base = 8.3 + 0.02 * randn(case['pairs']).repeat_interleave(2)
        s.update(es=Eggroll(model, case['pairs']), step=seed % 4096, losses=base + 1e-3 * randn(2 * case['pairs']))
    return s


def run(s):
    kind = s['kind']
    if kind == 'attention':
        return attention(s['q'], s['k'], s['v'], s['window'])
    if kind == 'lowrank':
        return lowrank(s['x'], s['weight'], s['a'], s['b'], s['sign'], dir_div=s['div'])
    if kind == 'block':
        return block_forward(s['x'], s['w'], s['ve'], s['cos'], s['sin'], s['window'], **s['jitter'])
    if kind == 'head':
        return head_loss(s['x'], s['weight'], s['y'], VOCAB)
    if kind == 'population':
        return s['es'].population(s['step'], s['x'], s['y'], names=s['names'], fp32_head=s['fp32_head'])
    return s['es'].update(s['losses'], s['es'].offsets(s['step']))


# --- what a pass cannot do without ---


def _pairs(T, window):
    """Visible (query, key) pairs of one head: query s sees keys s - window .. s."""
    full = min(T, window + 1)
    return full * (full + 1) // 2 + (T - full) * (window + 1)


MODEL_PARAMS = LAYERS * 12 * E * E + 6 * VOCAB * E + 4 * 8 * 32 + 2 * LAYERS


def work(case):
    kind = case['kind']
    if kind == 'attention':
        size = 2 if case['dtype'] == 'bf16' else 4
        n = case['batch'] * case['length'] * E
        return dict(bytes=4 * size * n, flops=4 * D * H * case['batch'] * _pairs(case['length'], case['window']))
    if kind == 'lowrank':
        m, T, i, o = case['members'], case['tokens'], case['n_in'], case['n_out']
        dirs = -(-m // case['div'])
        rows = 1 if case['shared'] else m
        size = 2 if case['dtype'] == 'bf16' else 4
        dots = dirs if case['shared'] else m
        return dict(bytes=size * rows * T * i + 4 * (o * i + dirs * (i + o) + m) + 4 * m * T * o,
                    flops=2 * rows * T * i * o + 2 * dots * T * i + 2 * m * T * o)
    if kind == 'block':
        B, T = case['batch'], case['length']
        ve = has_ve(case['layer'])
        width = {'none': 0, 'fc': 4 * E}.get(case['site'], E)
        return dict(bytes=B * T * (8 * E + (2 * E if ve else 0) + 2 * width) + 4 * 12 * E * E,
                    flops=2 * B * T * 12 * E * E + 4 * D * H * B * _pairs(T, window_sizes()[case['layer']]))
    if kind == 'head':
        n = case['batch'] * case['length']
        return dict(bytes=n * (4 * E + 8 + 4) + 4 * VOCAB * E, flops=2 * n * E * VOCAB)
    if kind == 'population':
        m, T = 2 * case['pairs'], case['length']
        attn = sum(4 * D * H * _pairs(T, w) for w in window_sizes())
        return dict(bytes=4 * MODEL_PARAMS + 16 * T + 4 * m,
                    flops=m * (T * (2 * LAYERS * 12 * E * E + 2 * E * VOCAB) + attn))
    return dict(bytes=4 * MODEL_PARAMS + 8 * case['pairs'], flops=2 * case['pairs'] * MODEL_PARAMS)


def tolerance(case):
    """About four times the distance from the 64-bit results: bf16 operands and outputs for the layers (2e-3 to
    3.4e-3), the head and the gradients as products split over bf16 pairs (4e-7 and 4.6e-6), and member means of a
    bf16 forward (3e-5)."""
    return {
        'attention': {'rel': 1.2e-2},
        'lowrank': {'rel': 1.2e-2},
        'block': {'rel': 1.2e-2},
        'head': {'rel': 4e-6},
        'population': {'rel': 1.2e-4},
        'update': {'rel': 2e-5},
    }[case['kind']]


# --- the same results in 64 bits ---


def _norm64(x):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + torch.finfo(torch.float32).eps)


def _attention64(q, k, v, window):
    """[B, T, H, D] in 64 bits, one sequence at a time."""
    B, T = q.shape[:2]
    i = torch.arange(T, device=q.device)
    hidden = (i[:, None] < i[None, :]) | (i[:, None] - i[None, :] > window)
    out = torch.empty(q.shape, dtype=F64, device=q.device)
    for n in range(B):
        qh, vh = (t[n].double().transpose(0, 1).contiguous() for t in (q, v))
        kt = k[n].double().permute(1, 2, 0).contiguous()
        p = torch.softmax((torch.bmm(qh, kt) / math.sqrt(D)).masked_fill_(hidden, -math.inf), -1)
        out[n] = torch.bmm(p, vh).transpose(0, 1)
    return out


def _rotary64(x, cos, sin):
    a, b = x[..., :D // 2], x[..., D // 2:]
    c, s = cos.double()[None, :, None, :], sin.double()[None, :, None, :]
    return torch.cat([a * c + b * s, b * c - a * s], -1)


def _block64(x, w, ve, cos, sin, window, o=None, attn=None, fc=None, mlp=None):
    """run.py:102-117 in 64 bits."""
    B, T, _ = x.shape
    plus = lambda t, j: t if j is None else t + j.double()
    w = {n: None if t is None else t.double() for n, t in w.items()}
    h = _norm64(x)
    q, k, v = ((h @ w[n].t()).view(B, T, H, D) for n in 'qkv')
    if ve is not None:
        gate = 2 * torch.sigmoid(h[..., :32] @ w['gate'].t())
        v = v + gate[..., None] * ve.double().view(B, T, H, D)
    q, k = _norm64(_rotary64(q, cos, sin)), _norm64(_rotary64(k, cos, sin))
    y = plus(_attention64(q, k, v, window).reshape(B, T, E), o)
    x = x + plus(y @ w['proj'].t(), attn)
    hidden = plus(_norm64(x) @ w['fc'].t(), fc)
    return x + plus(torch.relu(hidden).square() @ w['out'].t(), mlp)


def _head64(x, weight, y):
    logits = 15 * torch.tanh(_norm64(x.double()) @ weight.double().t() / 15)
    loss = torch.logsumexp(logits, -1) - logits.gather(-1, y.clamp(min=0)[..., None])[..., 0]
    return torch.where(y < 0, torch.zeros_like(loss), loss)


def _slices64(buffer, offsets, width):
    """[n, width] of the noise buffer at the directions' offsets, in 64 bits."""
    return buffer[offsets[:, None] + torch.arange(width, device=DEV)].double()


def _offsets(params, step, pairs):
    g = torch.Generator(DEV).manual_seed(1_000_003 * SEED + step)
    return {n: torch.randint(0, NOISE - sum(p.shape), (pairs,), device=DEV, generator=g) for n, p in params.items()}


def _population64(s, case):
    params = dict(s['es'].params)
    names = set(params if s['names'] is None else s['names'])
    buffer = torch.randn(NOISE, device=DEV, generator=torch.Generator(DEV).manual_seed(SEED))
    offsets = _offsets(params, s['step'], case['pairs'])
    x, y, T = s['x'][0], s['y'][0], case['length']
    cos, sin = (t.to(DEV) for t in rotary_tables(T))
    out = []
    for m in range(2 * case['pairs']):
        sigma = SIGMA if m % 2 == 0 else -SIGMA

        def p(name):
            w = params[name].double()
            if name not in names:
                return w
            noise = _slices64(buffer, offsets[name][m // 2:m // 2 + 1], sum(w.shape))[0]
            return w + sigma * (torch.outer(noise[:w.shape[0]], noise[w.shape[0]:]) if w.dim() == 2 else noise)

        x0 = _norm64(p('transformer.wte.weight')[x][None])
        h, lam_r, lam_x = x0, p('resid_lambdas'), p('x0_lambdas')
        for i in range(LAYERS):
            pre = f'transformer.h.{i}.'
            w = dict(q=p(pre + 'attn.c_q.weight'), k=p(pre + 'attn.c_k.weight'), v=p(pre + 'attn.c_v.weight'),
                     gate=p(pre + 'attn.ve_gate.weight') if has_ve(i) else None, proj=p(pre + 'attn.c_proj.weight'),
                     fc=p(pre + 'mlp.c_fc.weight'), out=p(pre + 'mlp.c_proj.weight'))
            ve = p(f'value_embeds.{i}.weight')[x][None] if has_ve(i) else None
            h = _block64(lam_r[i] * h + lam_x[i] * x0, w, ve, cos, sin, window_sizes()[i])
        out.append(_head64(h[0], p('lm_head.weight'), y).mean())
    return torch.stack(out)


def _update64(s, case):
    params, pairs = s['es'].params, case['pairs']
    buffer = torch.randn(NOISE, device=DEV, generator=torch.Generator(DEV).manual_seed(SEED))
    offsets = _offsets(params, s['step'], pairs)
    losses = s['losses'].double()
    fitness = losses[1::2] - losses[0::2]
    fitness = fitness / (fitness.std() + 1e-8)
    out = {}
    for name, p in params.items():
        g = torch.zeros(p.shape, dtype=F64, device=DEV)
        for d in range(0, pairs, 16384):
            rows = _slices64(buffer, offsets[name][d:d + 16384], sum(p.shape))
            f = fitness[d:d + 16384]
            if p.dim() == 2:
                g -= (f[:, None] * rows[:, :p.shape[0]]).t() @ rows[:, p.shape[0]:]
            else:
                g -= f @ rows
        out[name] = g / pairs
    return out


def exact(case, seed):
    s = prepare(case, seed)
    kind = case['kind']
    if kind == 'attention':
        return _attention64(s['q'], s['k'], s['v'], s['window'])
    if kind == 'lowrank':
        m, T = case['members'], case['tokens']
        w = s['weight'].double().t()
        y = torch.empty(m, T, case['n_out'], dtype=F64, device=DEV)
        for n in range(m):
            x = s['x'][n].double()
            a, b = s['a'][n // s['div']].double(), s['b'][n // s['div']].double()
            y[n] = x @ w + s['sign'][n].double() * (x @ b)[:, None] * a
        return y
    if kind == 'block':
        return _block64(s['x'].double(), s['w'], s['ve'], s['cos'], s['sin'], s['window'], **s['jitter'])
    if kind == 'head':
        return _head64(s['x'], s['weight'], s['y']).reshape(-1)
    if kind == 'population':
        return _population64(s, case)
    return _update64(s, case)
