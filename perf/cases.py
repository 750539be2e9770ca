"""Performance cases: the calls that a training or scoring program on this library makes, over the sizes it makes them.

    forward      GPT.forward on a batch of token rows: the logits of a short prompt, the per-token losses of a validation
                 batch (ragged lengths, padded inside)
    population   one chunk of an EGGROLL step: antithetic members of the fixed GPT, each with its own noise row, through
                 run_forward; per-member and per-token losses
    update       the second half of an EGGROLL step: fitness, the directions' noise rows, every parameter's outer-product
                 gradient and AdamW, over the whole model (the C entry points and classes that Eggroll.step calls)
    credit       the cross-token credit readout: value_credit (both passes), or the key-context pass
    attention    the windowed causal attention as the module-by-module forward calls it
    lowrank      the perturbed linear, every member with its own x or all with one, the outputs stored
    sumsq        the perturbed linear with x shared by all members, only each member's sum of squares kept
    head_error   Dust's head-slab estimator of the lm_head outputs' errors
    reassemble   Dust's map from a site's output error to its weight error, for the linears and the embeddings

Each kind has its listed cases and a range that draw() samples. prepare() makes what the program holds before the call;
run() is the call; exact() restates it in float64 with plain torch.
"""
import ctypes
import math

import torch

from noise_amd import _lib, credit, dust, model as nm, population
from noise_amd.optim import AdamW

V, D, F, H, L = 4096, 512, 2048, 8, 8  # the fixed model: vocabulary, width, MLP width, heads, blocks
WINDOWS = [1024, 1024, 1024, 2048, 1024, 1024, 1024, 2048]
SIGMA = 0.002
EPS = 1.1920928955078125e-07
# the largest sizes of a drawn case
MAX_ROWS = 512 * 2048


def listed():
    return [
        # the smallest call: one short prompt's logits, where launches and latency count
        dict(name='forward 1x64', kind='forward', batch=1, T=64, logits=True),
        # a few ragged rows scored per token (evaluate's rows, Dust's losses)
        dict(name='score 3x1000', kind='forward', batch=3, T=1000, logits=False),
        # a small population on short rows: 8 antithetic pairs
        dict(name='population 16x256', kind='population', members=16, seqs=2, T=256),
        # the headline step: 256 members x 2 sequences x 2048 tokens
        dict(name='population 512x2048', kind='population', members=512, seqs=2, T=2048),
        # one chunk of directions of the update, the whole model's gradients and AdamW
        dict(name='update 1024', kind='update', pairs=1024),
        # the full credit readout of a 16-sequence batch, bounded logits, the source's high part
        dict(name='credit 128x2048', kind='credit', op='value', rows=128, T=2048, window=2048, hi_lo=False, bounded=True),
        # one sequence's heads at a short length, general logits, high and low parts
        dict(name='credit 8x640', kind='credit', op='value', rows=8, T=640, window=512, hi_lo=True, bounded=False),
        # the module-by-module forward's attention, a ragged length
        dict(name='attention 3x1500', kind='attention', batch=3, T=1500, window=1024, fp32=False),
        # a linear of a few members, each with its own rows
        dict(name='lowrank 24x640', kind='lowrank', members=24, T=640, n_in=512, n_out=2048, shared=False),
        # one linear shared by 64 members, only the sums of squares kept
        dict(name='sumsq 64x32768', kind='sumsq', members=64, T=32768, n_in=512, n_out=2048, mode='expansion'),
        # the head's error estimate over part of a batch
        dict(name='head_error 8x512', kind='head_error', b=8, t=512, vocab=4096, padded=4096, draws=2048),
        # an 8 x 2048 batch's errors of the MLP's input linear
        dict(name='reassemble 16384', kind='reassemble', tokens=16384, n_out=2048, n_in=512, bf16=False, table=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(['forward', 'forward', 'population', 'population', 'update', 'credit', 'attention', 'lowrank',
                       'sumsq', 'head_error', 'reassemble', 'reassemble'])
    if kind == 'forward':
        return dict(kind=kind, batch=_log(rng, 1, 32), T=_log(rng, 32, 2048), logits=rng.random() < 0.5)
    if kind == 'population':
        T = 128 * rng.randint(1, 16)
        return dict(kind=kind, members=_log(rng, 4, min(512, MAX_ROWS // T)), seqs=rng.choice([1, 2, 4]), T=T)
    if kind == 'update':
        return dict(kind=kind, pairs=_log(rng, 48, 1024))
    if kind == 'credit':
        T = 128 * rng.randint(1, 16)
        op = rng.choice(['value', 'value', 'context'])
        return dict(kind=kind, op=op, rows=_log(rng, 4, 128), T=T, window=rng.randint(T // 4, T),
                    hi_lo=op == 'value' and rng.random() < 0.5, bounded=op == 'value' and rng.random() < 0.5)
    if kind == 'attention':
        T = _log(rng, 48, 2048)
        return dict(kind=kind, batch=_log(rng, 1, 32), T=T, window=rng.choice([1024, 2048, rng.randint(32, T)]),
                    fp32=rng.random() < 0.5)
    if kind == 'lowrank':
        n_in, n_out = rng.choice([(512, 512), (512, 2048), (2048, 512), (512, 4096)])
        shared = rng.random() < 0.3
        return dict(kind=kind, members=_log(rng, 2, 48), T=(256 if shared else 128) * rng.randint(1, 4), n_in=n_in,
                    n_out=n_out, shared=shared)
    if kind == 'sumsq':
        n_in, n_out = rng.choice([(512, 512), (512, 2048), (2048, 512), (544, 768)])
        return dict(kind=kind, members=_log(rng, 4, 96), T=256 * _log(rng, 2, 128), n_in=n_in, n_out=n_out,
                    mode=rng.choice(['expansion', 'direct']))
    if kind == 'head_error':
        vocab = 256 * rng.randint(2, 16)
        n = rng.choice([16, 12])
        return dict(kind=kind, b=rng.randint(1, 8), t=_log(rng, 40, 512), vocab=vocab,
                    padded=vocab + rng.choice([0, 256]), draws=n * (vocab // 256) * rng.randint(1, 8))
    if rng.random() < 0.3:
        return dict(kind=kind, tokens=_log(rng, 200, 16384), n_out=V, n_in=D, bf16=False, table=True)
    n_out, n_in, bf16 = rng.choice([(512, 512, True), (512, 512, False), (2048, 512, False), (512, 2048, True),
                                    (4096, 512, False), (8, 32, False)])
    return dict(kind=kind, tokens=_log(rng, 200, 16384), n_out=n_out, n_in=n_in, bf16=bf16, table=False)


# ---- inputs ---------------------------------------------------------------------------------------------------------

DEV = torch.device('cuda', 0)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, device=DEV, generator=g)


def _uniform(g, bound, *shape):
    return (torch.rand(*shape, device=DEV, generator=g) * 2 - 1) * bound


def _has_ve(i):
    return i % 2 == (L - 1) % 2


def _weights(g):
    """The fixed model's parameters in named_parameters() order: the training run's initial distributions, with a head
    and gates of a model that has trained for a while."""
    s = math.sqrt(3 / D)
    w = {'resid_lambdas': 1 + 0.05 * _randn(g, L), 'x0_lambdas': 0.1 + 0.05 * _randn(g, L),
         'transformer.wte.weight': _randn(g, V, D)}
    for i in range(L):
        pre = f'transformer.h.{i}.'
        for name in ('c_q', 'c_k', 'c_v'):
            w[pre + f'attn.{name}.weight'] = _uniform(g, s, D, D)
        w[pre + 'attn.c_proj.weight'] = _uniform(g, 1.5 * s, D, D)
        if _has_ve(i):
            w[pre + 'attn.ve_gate.weight'] = 0.05 * _randn(g, H, 32)
        w[pre + 'mlp.c_fc.weight'] = _uniform(g, s, F, D)
        w[pre + 'mlp.c_proj.weight'] = _uniform(g, 1.5 * math.sqrt(3 / F), D, F)
    w['lm_head.weight'] = 0.02 * _randn(g, V, D)
    for i in range(L):
        if _has_ve(i):
            w[f'value_embeds.{i}.weight'] = _uniform(g, s, V, D)
    return w


def _model(w):
    with torch.device('meta'):
        m = nm.GPT(nm.GPTConfig())
    m.to_empty(device=DEV)
    m.init_weights()
    m.transformer.wte.float()
    for e in m.value_embeds.values():
        e.float()
    m.load_state_dict(w, strict=True)
    return m.requires_grad_(False)


def _tokens(g, *shape):
    """Zipf(1.1) token ids."""
    p = 1.0 / torch.arange(1, V + 1, device=DEV, dtype=torch.float64) ** 1.1
    return torch.multinomial(p.float(), math.prod(shape), replacement=True, generator=g).view(*shape)


def _text(g, rows, T):
    t = _tokens(g, rows, T + 1)
    return t[:, :-1].contiguous(), t[:, 1:].contiguous()


def _stride(w):
    return sum(sum(t.shape) for t in w.values())


def _rms(x):
    return torch.nn.functional.rms_norm(x, (x.shape[-1],))


def _inputs(c, seed):
    """The case's plain inputs, from the seed alone (prepare and exact share them)."""
    g, kind = _gen(seed), c['kind']
    if kind == 'forward':
        return dict(w=_weights(g), text=_text(g, c['batch'], c['T']))
    if kind == 'population':
        w = _weights(g)
        m, n = c['members'], c['seqs']
        i = torch.arange(m, device=DEV)
        pair = i // (2 * n)
        return dict(w=w, text=_text(g, n, c['T']), rows=_randn(g, int(pair.max()) + 1, _stride(w)),
                    seq=(i % n).int(), row=pair.int(), sign=torch.where(i // n % 2 == 0, SIGMA, -SIGMA).float())
    if kind == 'update':
        w = _weights(g)
        n = sum(t.numel() for t in w.values())
        return dict(w=w, losses=8.3 + 0.05 * _randn(g, 2 * c['pairs']), m=1e-3 * _randn(g, n),
                    v=1e-6 * _randn(g, n).square(), step=seed % 1000)
    if kind == 'credit':
        r, T = c['rows'], c['T']
        q, k = (_rms(_randn(g, r, T, 64)).bfloat16() for _ in range(2))
        return dict(q=q, k=k, hub=_randn(g, r, T, 64), values=_randn(g, r, T, 64).bfloat16())
    if kind == 'attention':
        dt = torch.float32 if c['fp32'] else torch.bfloat16
        q, k = (_rms(_randn(g, c['batch'], c['T'], H, 64)).to(dt) for _ in range(2))
        return dict(q=q, k=k, v=_randn(g, c['batch'], c['T'], H, 64).to(dt))
    if kind in ('lowrank', 'sumsq'):
        m, T, n_in, n_out = c['members'], c['T'], c['n_in'], c['n_out']
        x = _rms(_randn(g, *((T, n_in) if kind == 'sumsq' or c['shared'] else (m, T, n_in)))).bfloat16()
        sign = torch.where(torch.arange(m, device=DEV) % 2 == 0, SIGMA, -SIGMA).float()
        return dict(x=x, w=(0.02 * _randn(g, n_out, n_in)).bfloat16(), a=_randn(g, m, n_out), b=_randn(g, m, n_in),
                    sign=sign)
    if kind == 'head_error':
        b, t, vocab = c['b'], c['t'], c['vocab']
        raw = (3.0 * _randn(g, b, t, c['padded'])).bfloat16()
        y = torch.randint(0, vocab, (b, t), device=DEV, generator=g)
        z = 15 * torch.tanh(raw[..., :vocab].double() / 15)
        ce = (torch.logsumexp(z, -1) - z.gather(-1, y.unsqueeze(-1)).squeeze(-1)).float()
        y[torch.rand(b, t, device=DEV, generator=g) < 0.03] = -1
        return dict(raw=raw, y=y, clean=ce, seed=seed)
    x = _tokens(g, c['tokens']) if c['table'] else _rms(_randn(g, c['tokens'], c['n_in']))
    x = x.bfloat16() if c['bf16'] else x
    return dict(x=x, error=0.01 * _randn(g, c['tokens'], D if c['table'] else c['n_out']))


def prepare(case, seed):
    st = dict(_inputs(case, seed), case=case)
    kind = case['kind']
    if kind in ('forward', 'population'):
        st['model'] = _model(st.pop('w'))
        st['layout'] = population.NoiseLayout(st['model'])
        st['model'].packed()  # the weights laid out once, as after a program's first call
    elif kind == 'update':
        _prepare_update(st)
    elif kind == 'sumsq':
        st['rows'] = torch.cat([st.pop('a'), st.pop('b')], 1).contiguous()
    return st


def _prepare_update(st):
    """The model, its optimizer in mid-run and the update's plan; parameters, gradients and moments as views of flat
    buffers."""
    mdl = _model(st.pop('w'))
    pairs = st['case']['pairs']
    es = population.Eggroll(mdl, pairs)
    named = list(mdl.named_parameters())
    flat = torch.cat([p.detach().reshape(-1) for _, p in named])
    grad = torch.empty_like(flat)
    opt = AdamW(mdl.parameters(), lr=1e-3, betas=(0.5, 0.95), eps=1e-8, weight_decay=0.0)
    at, mats, vecs = 0, [], []
    for (name, p), c0 in zip(named, es.layout.col0):
        sl = slice(at, at + p.numel())
        p.data = flat[sl].view(p.shape)
        p.grad = grad[sl].view(p.shape)
        opt.state[p] = dict(step=10, exp_avg=st['m'][sl].view(p.shape), exp_avg_sq=st['v'][sl].view(p.shape))
        (mats if p.dim() == 2 else vecs).append((c0, p.shape, p.grad))
        at += p.numel()
    arr = lambda vals, t: (t * len(vals))(*vals)
    plan = (arr([c0 for c0, _, _ in mats], ctypes.c_int64), arr([c0 + s[0] for c0, s, _ in mats], ctypes.c_int64),
            arr([s[0] for _, s, _ in mats], ctypes.c_int64), arr([s[1] for _, s, _ in mats], ctypes.c_int64),
            arr([t.data_ptr() for _, _, t in mats], ctypes.c_void_p))
    st.update(model=mdl, es=es, opt=opt, flat=flat, grad=grad, vecs=vecs, n_mats=len(mats), plan=plan,
              directions=torch.arange(pairs, device=DEV))


def run(st):
    c = st['case']
    return {'forward': _run_forward, 'population': _run_population, 'update': _run_update, 'credit': _run_credit,
            'attention': _run_attention, 'lowrank': _run_lowrank, 'sumsq': _run_sumsq, 'head_error': _run_head,
            'reassemble': _run_reassemble}[c['kind']](st, c)


def _run_forward(st, c):
    x, y = st['text']
    return st['model'](x) if c['logits'] else st['model'](x, y, loss_reduction='none')


def _run_population(st, c):
    x, y = st['text']
    out = population.run_forward(st['model'], x, y, st['seq'], noise=st['rows'], member_row=st['row'],
                                 member_sign=st['sign'], layout=st['layout'], want_tokens=True, check_tables=False)
    return out['loss_sum'], out['token_loss']


def _run_update(st, c):
    es, pairs, losses = st['es'], c['pairs'], st['losses']
    stream = _lib.stream(DEV)
    fitness, weight = torch.empty(pairs, device=DEV), torch.empty(pairs, device=DEV)
    _lib.call('noise_fitness', _lib.ptr(losses), 2 * pairs, pairs, _lib.ptr(fitness), _lib.ptr(weight), stream)
    rows = es.rows(es.offset_table(st['step']), st['directions'])
    for c0, shape, grad in st['vecs']:
        _lib.call('noise_outer_grad', _lib.ptr(rows), es.layout.stride, c0, -1, _lib.ptr(weight), pairs, 1, shape[0],
                  -1.0 / pairs, 0, _lib.ptr(grad), stream)
    _lib.call('noise_outer_grad_batch', _lib.ptr(rows), es.layout.stride, _lib.ptr(weight), pairs, st['n_mats'],
              *st['plan'], -1.0 / pairs, 0, stream)
    st['opt'].step()
    return fitness, st['grad'], st['flat'], st['m'], st['v']


def _run_credit(st, c):
    if c['op'] == 'context':
        return credit.key_context(st['q'], st['k'], st['values'], st['hub'], c['window'])
    return credit.value_credit(st['q'], st['k'], st['hub'], c['window'], hi_lo=c['hi_lo'], bounded=c['bounded'])


def _run_attention(st, c):
    return nm.attention(st['q'], st['k'], st['v'], c['window'])


def _run_lowrank(st, c):
    return population.lowrank(st['x'], st['w'], st['a'], st['b'], st['sign'])


def _run_sumsq(st, c):
    return population.lowrank_sumsq(st['x'], st['w'], st['rows'], 0, c['n_out'], st['sign'], mode=c['mode'])


def _run_head(st, c):
    return dust.head_error(st['raw'], st['y'], st['clean'], c['draws'], sigma=0.1, nrep=16, seed=st['seed'],
                           vocab=c['vocab'])


def _run_reassemble(st, c):
    x, error = st['x'], st['error']
    if c['table']:
        out = torch.empty(V, D, device=DEV)
        _lib.call('noise_reassemble_embedding', _lib.ptr(error), D, _lib.ptr(x), c['tokens'], V, D, _lib.ptr(out),
                  _lib.stream(DEV))
        return out
    out = torch.empty(c['n_out'], c['n_in'], device=DEV)
    _lib.call('noise_reassemble', _lib.ptr(error), c['n_out'], _lib.ptr(x), int(c['bf16']), c['n_in'], c['tokens'],
              c['n_out'], c['n_in'], 1.0, _lib.ptr(out), _lib.stream(DEV))
    return out


# ---- what a pass cannot do without ----------------------------------------------------------------------------------

GEMM_WEIGHTS = L * (4 * D * D + 2 * D * F) + V * D
PARAMS = GEMM_WEIGHTS + V * D + sum(V * D + 8 * 32 for i in range(L) if _has_ve(i)) + 2 * L


def _pairs(T, window):
    """In-window causal pairs of one row of T tokens."""
    w = min(window, T - 1)
    return (w + 1) * (w + 2) // 2 + (T - w - 1) * (w + 1)


def _forward_flops(rows, T):
    return rows * (2.0 * GEMM_WEIGHTS * T + 4.0 * D * sum(_pairs(T, w) for w in WINDOWS))


def work(case):
    c, kind = case, case['kind']
    if kind == 'forward':
        M = c['batch'] * c['T']
        out = M * 4 * (V if c['logits'] else 1)
        # the weights as bf16, the embedding rows of the tokens in the token and value tables, the tokens, the result
        return dict(bytes=2 * GEMM_WEIGHTS + min(M, V) * 5 * D * 4 + 16 * M + out, flops=_forward_flops(c['batch'], c['T']))
    if kind == 'population':
        M = c['members'] * c['T']
        rows = -(-c['members'] // (2 * c['seqs']))
        return dict(bytes=2 * GEMM_WEIGHTS + 5 * V * D * 4 + rows * 101552 * 4 + 4 * M,
                    flops=_forward_flops(c['members'], c['T']))
    if kind == 'update':  # the gradient written; parameters and moments read and written
        return dict(bytes=28 * PARAMS, flops=2.0 * c['pairs'] * PARAMS)
    if kind == 'credit':
        r, T = c['rows'], c['T']
        per = 6 + 2 * c['hi_lo'] if c['op'] == 'value' else 4
        io = (2 + 2 + 4 + 4) * 64 if c['op'] == 'value' else 4 * 2 * 64 + 8
        return dict(bytes=r * T * io, flops=per * 64.0 * r * _pairs(T, c['window']))
    if kind == 'attention':
        n = c['batch'] * H
        return dict(bytes=n * c['T'] * 64 * 4 * (4 if c['fp32'] else 2), flops=4 * 64.0 * n * _pairs(c['T'], c['window']))
    if kind in ('lowrank', 'sumsq'):
        m, T, n_in, n_out = c['members'], c['T'], c['n_in'], c['n_out']
        one = kind == 'sumsq' or c['shared']
        io = 2 * (1 if one else m) * T * n_in + 2 * n_in * n_out + 4 * m * (n_in + n_out)
        y = 4 * m if kind == 'sumsq' else 4 * m * T * n_out
        per = 2 * n_out if kind == 'sumsq' else 2 * n_out  # a member's own term of every output
        return dict(bytes=io + y, flops=2.0 * (1 if one else m) * T * n_in * n_out + m * T * (2.0 * n_in + per))
    if kind == 'head_error':
        rows = c['b'] * c['t']
        # per jittered logit: a Gaussian, a soft cap, an exponential and a weighted sum, about 40 operations
        return dict(bytes=rows * c['padded'] * 6 + 12 * rows, flops=40.0 * c['draws'] * rows * 256)
    if c['table']:
        return dict(bytes=c['tokens'] * (8 + D * 4) + V * D * 4, flops=1.0 * c['tokens'] * D)
    return dict(bytes=c['tokens'] * (4 * c['n_out'] + (2 if c['bf16'] else 4) * c['n_in']) + 4 * c['n_out'] * c['n_in'],
                flops=2.0 * c['tokens'] * c['n_out'] * c['n_in'])


def tolerance(case):
    """About four times the error against float64 that a correct pass shows over the ranges."""
    return dict(rel={
        'forward': 0.03 if case.get('logits') else 2e-3,  # bf16 operands through 8 blocks; losses near 8.3 move less
        'population': 2e-3,
        'update': 1e-5,  # fp32 sums of up to 1,024 products, noise values to about 1e-7
        'credit': 0.01 if case.get('op') == 'value' else 1e-4,  # bf16 probabilities; the key context's are fp32
        'attention': 8e-3,
        'lowrank': 7e-3,
        'sumsq': 3e-5,
        'head_error': 2e-4,  # rewards are differences of fp32 losses
        'reassemble': 1e-5,
    }[case['kind']])


# ---- the same in float64 --------------------------------------------------------------------------------------------

def _rms64(x):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)


def _attend64(q, k, v, window):
    """q, k, v [n, T, 64] -> [n, T, 64]."""
    T = q.shape[1]
    lag = torch.arange(T, device=DEV)[:, None] - torch.arange(T, device=DEV)[None, :]
    z = torch.bmm(q, k.transpose(1, 2).contiguous()) / 8
    return torch.bmm(z.masked_fill_((lag < 0) | (lag > window), -math.inf).softmax(-1), v)


def _rotary64(x):
    """x [n, T, H, 64]; the model's bf16 tables."""
    f = 1.0 / 10000 ** (torch.arange(0, 64, 2, dtype=torch.float32, device=DEV) / 64)
    t = torch.outer(torch.arange(x.shape[1], dtype=torch.float32, device=DEV), f)
    c, s = (u.bfloat16().double()[None, :, None, :] for u in (t.cos(), t.sin()))
    a, b = x[..., :32], x[..., 32:]
    return torch.cat([a * c + b * s, b * c - a * s], -1)


def _gpt64(w, idx, rows=None, sign=None):
    """Capped logits [n, T, V] of token rows idx [n, T], each with its noise row (or none) scaled by sign [n]."""
    n, T = idx.shape
    w = {k: t.double() for k, t in w.items()}
    at, col = {}, 0
    for k, t in w.items():
        at[k] = col
        col += sum(t.shape)

    def ab(k):
        o, i = w[k].shape
        return rows[:, at[k]:at[k] + o], rows[:, at[k] + o:at[k] + o + i]

    def linear(k, x):
        y = x @ w[k].t()
        if rows is not None:
            a, b = ab(k)
            y = y + sign[:, None, None] * torch.bmm(x, b.unsqueeze(-1)) * a[:, None, :]
        return y

    def embed(k):
        y = w[k][idx]
        if rows is not None:
            a, b = ab(k)
            y = y + sign[:, None, None] * a.gather(1, idx).unsqueeze(-1) * b[:, None, :]
        return y

    def scalar(k, i):
        s = w[k][i].expand(n)
        return (s if rows is None else s + sign * rows[:, at[k] + i])[:, None, None]

    heads = lambda t: t.transpose(1, 2).reshape(n * H, T, 64).contiguous()
    x = x0 = _rms64(embed('transformer.wte.weight'))
    for i in range(L):
        pre = f'transformer.h.{i}.'
        x = scalar('resid_lambdas', i) * x + scalar('x0_lambdas', i) * x0
        h = _rms64(x)
        q, k, v = (linear(pre + f'attn.{c}.weight', h).view(n, T, H, 64) for c in ('c_q', 'c_k', 'c_v'))
        if _has_ve(i):
            gate = 2 * torch.sigmoid(linear(pre + 'attn.ve_gate.weight', h[..., :32].contiguous()))
            v = v + gate.unsqueeze(-1) * embed(f'value_embeds.{i}.weight').view(n, T, H, 64)
        q, k = _rms64(_rotary64(q)), _rms64(_rotary64(k))
        y = _attend64(heads(q), heads(k), heads(v), WINDOWS[i])
        y = y.view(n, H, T, 64).transpose(1, 2).reshape(n, T, D)
        x = x + linear(pre + 'attn.c_proj.weight', y)
        x = x + linear(pre + 'mlp.c_proj.weight', torch.relu(linear(pre + 'mlp.c_fc.weight', _rms64(x))).square())
    return 15 * torch.tanh(linear('lm_head.weight', _rms64(x)) / 15)


def _ce64(z, y):
    return torch.logsumexp(z, -1) - z.gather(-1, y.unsqueeze(-1)).squeeze(-1)


def _philox(c0, c1, c2, c3, key):
    """Philox4x32-10 (Salmon et al., SC'11) on int64 tensors holding 32-bit words."""
    M = 0xFFFFFFFF
    k0, k1 = key & M, key >> 32 & M
    for _ in range(10):
        p0, p1 = c0 * 0xD2511F53, c2 * 0xCD9E8D57
        c0, c1, c2, c3 = (p1 >> 32 & M) ^ c1 ^ k0, p1 & M, (p0 >> 32 & M) ^ c3 ^ k1, p0 & M
        k0, k1 = k0 + 0x9E3779B9 & M, k1 + 0xBB67AE85 & M
    return c0, c1, c2, c3


def _gauss(words):
    """Box-Muller on the words' top 24 bits: four Gaussians per counter, last axis."""
    out = []
    for x, y in (words[:2], words[2:]):
        r = torch.sqrt(-2 * torch.log(((x >> 8) + 1).double() * 2.0 ** -24))
        t = 2 * math.pi * (y >> 8).double() * 2.0 ** -24
        out += [r * torch.cos(t), r * torch.sin(t)]
    return torch.stack(out, -1)


def _exact_update(c, i):
    pairs, w = c['pairs'], i['w']
    L2 = i['losses'].double()
    f = L2[1::2] - L2[0::2]
    f = f / (f.std() + 1e-8)
    d = torch.arange(pairs, device=DEV)
    zero = torch.zeros_like(d)
    grads = []
    for p, (name, t) in enumerate(w.items()):
        width = sum(t.shape)
        span = 2 ** 28 - width
        off = _philox(d, zero + p, zero, zero + 0x4F464653, i['step'])[0] * span >> 32  # seed 0: the key is the step
        quad = (off >> 2)[:, None] + torch.arange(width // 4 + 1, device=DEV)
        z = torch.zeros_like(quad)
        val = _gauss(_philox(quad, z, z, z + 0x4E4F4953, 0)).view(pairs, -1)
        rows = val.gather(1, (off & 3)[:, None] + torch.arange(width, device=DEV))
        if t.dim() == 2:
            grads.append((-((f[:, None] * rows[:, :t.shape[0]]).t().contiguous() @ rows[:, t.shape[0]:]) / pairs).reshape(-1))
        else:
            grads.append(-(f @ rows) / pairs)
    g = torch.cat(grads)
    m, v = i['m'].double(), i['v'].double()
    m = m + 0.5 * (g - m)
    v = 0.95 * v + 0.05 * g * g
    p = torch.cat([t.reshape(-1) for t in w.values()]).double()
    p = p - 1e-3 / (1 - 0.5 ** 11) * m / (v.sqrt() / math.sqrt(1 - 0.95 ** 11) + 1e-8)
    return f, g, p, m, v


def _exact_credit(c, i):
    r, T, W = c['rows'], c['T'], c['window']
    lag = torch.arange(T, device=DEV)[:, None] - torch.arange(T, device=DEV)[None, :]
    outs = []
    for a in range(0, r, 8):
        q, k, hub, val = (i[n][a:a + 8].double() for n in ('q', 'k', 'hub', 'values'))
        z = torch.bmm(q, k.transpose(1, 2).contiguous()) / 8
        z = z.masked_fill_((lag < 0) | (lag > W), -math.inf)
        p = z.softmax(-1)
        if c['op'] == 'value':
            outs.append((torch.bmm(p.transpose(1, 2).contiguous(), hub),))
        else:
            s = torch.bmm(i['hub'][a:a + 8].bfloat16().double(), val.transpose(1, 2).contiguous())
            outs.append((torch.logsumexp(z, -1), (p * s).sum(-1)))
    outs = [torch.cat(t) for t in zip(*outs)]
    return outs[0] if c['op'] == 'value' else tuple(outs)


def _exact_head(c, i):
    b, t, vocab, draws = c['b'], c['t'], c['vocab'], c['draws']
    rows, slabs = b * t, vocab // 256
    n = next(k for k in range(min(16, draws), 0, -1) if draws % k == 0)
    raw, y, clean = i['raw'].view(rows, -1).double(), i['y'].view(rows), i['clean'].view(rows).double()
    z = 15 * torch.tanh(raw[:, :vocab] / 15)
    ez = z.exp()
    total, tgt = ez.sum(-1), y.clamp(min=0)
    tz = z.gather(1, tgt[:, None])[:, 0]
    err = torch.zeros(rows, c['padded'], dtype=torch.float64, device=DEV)
    ctr = (torch.arange(rows, device=DEV)[:, None] * 64 + torch.arange(64, device=DEV))
    zero = torch.zeros_like(ctr)
    for g in range(draws):
        lo = g // n % slabs * 256
        a = _gauss(_philox(ctr, zero + g, zero, zero + 0x44414548, i['seed'])).view(rows, 256)
        zj = 15 * torch.tanh((raw[:, lo:lo + 256] + 0.1 * a) / 15)
        hit = (tgt >= lo) & (tgt < lo + 256)
        tj = torch.where(hit, zj.gather(1, (tgt - lo).clamp(0, 255)[:, None])[:, 0], tz)
        ce = torch.log(total - ez[:, lo:lo + 256].sum(-1) + zj.exp().sum(-1)) - tj
        rw = torch.where(y != -1, clean - ce, torch.zeros_like(ce))
        if b > 1:
            rw = (rw.view(b, t) - rw.view(b, t).mean(0)).view(rows)
        err[:, lo:lo + 256] -= (rw / 0.1)[:, None] * a
    return (err / (draws // slabs)).view(b, t, -1)


def exact(case, seed):
    c, kind = case, case['kind']
    if kind in ('forward', 'population') and c.get('batch', c.get('members')) * c['T'] > 65536:
        return None  # the float64 model over this many rows takes too long
    if kind == 'head_error' and c['draws'] * c['b'] * c['t'] > 1 << 24:
        return None
    i = _inputs(c, seed)
    if kind == 'forward':
        x, y = i['text']
        z = torch.cat([_gpt64(i['w'], x[a:a + 1]) for a in range(c['batch'])])
        return z if c['logits'] else _ce64(z, y).reshape(-1)
    if kind == 'population':
        x, y = i['text']
        ce = []
        for a in range(c['members']):
            q = int(i['seq'][a])
            row = i['rows'][int(i['row'][a])][None].double()
            ce.append(_ce64(_gpt64(i['w'], x[q:q + 1], row, i['sign'][a:a + 1].double()), y[q:q + 1]))
        ce = torch.cat(ce)
        return ce.sum(-1), ce.reshape(-1)
    if kind == 'update':
        return _exact_update(c, i)
    if kind == 'credit':
        return _exact_credit(c, i)
    if kind == 'attention':
        n, T = c['batch'], c['T']
        q, k, v = (i[s].double().transpose(1, 2).reshape(n * H, T, 64).contiguous() for s in 'qkv')
        y = torch.cat([_attend64(q[a:a + 8], k[a:a + 8], v[a:a + 8], c['window']) for a in range(0, n * H, 8)])
        return y.view(n, H, T, 64).transpose(1, 2).contiguous()
    if kind in ('lowrank', 'sumsq'):
        x, w, a, b, s = (i[k].double() for k in ('x', 'w', 'a', 'b', 'sign'))
        if kind == 'sumsq':  # the expanded square of x W^T + s (x . b) a^T
            y = x @ w.t()
            u = x @ b.t()
            return y.square().sum() + 2 * s * ((u.t() @ y) * a).sum(1) + s * s * u.square().sum(0) * a.square().sum(1)
        u = x @ b.t() if c['shared'] else torch.bmm(x, b.unsqueeze(-1))[..., 0].t()  # [T, m]
        return x @ w.t() + (s[:, None] * u.t()).unsqueeze(-1) * a[:, None, :]
    if kind == 'head_error':
        return _exact_head(c, i)
    e = i['error'].double()
    if c['table']:
        return torch.zeros(V, D, dtype=torch.float64, device=DEV).index_add_(0, i['x'], e)
    return e.t().contiguous() @ i['x'].double()
