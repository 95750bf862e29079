"""Performance cases of the population forward and of the work around it, one per kind of call that a program makes.

Every case goes through a public entry point: the torch wrappers (`noise_amd.ops`, `noise_amd.population`,
`noise_amd.eggroll`, `noise_amd.optim`, `noise_amd.credit`, `noise_amd.probes`) or, where a program calls the C ABI with
device buffers of its own (attention, the head, the update), the ctypes binding. Sizes are those of this repository's
configurations, tests and benchmark: the fixed model (8 layers, 512 wide, 8 heads of 64, hidden 2048, vocabulary 4096),
sequences of 128 .. 2048 tokens, populations of one to several hundred members. Inputs come from the seed alone and live
on the GPU.
"""
import math

import torch

from noise_amd import _lib, credit, ops, probes
from noise_amd.eggroll import Eggroll
from noise_amd.eval import load_model
from noise_amd.optim import Adam
from noise_amd.population import Weights, autocast_forward, population_loss

DEV = 'cuda'
D, F, V, LAYERS, HEADS, HD, VE_CH = 512, 2048, 4096, 8, 8, 64, 32
EPS = 2.0 ** -23
SIGMA = 1e-3
f64 = torch.float64


def listed():
    return [
        # one rank-1 perturbed linear on a ragged batch: rows that fill no whole tile of any kernel
        {'name': 'linear ragged', 'kind': 'linear', 'members': 6, 'tokens': 200, 'd_in': 512, 'd_out': 1536,
         'shared': False, 'pair': True, 'out': 'f32'},
        # the MLP sublayer of a small population (8 members x 256 tokens): launches and few workgroups
        {'name': 'mlp small', 'kind': 'mlp', 'members': 8, 'tokens': 256, 'hidden': F, 'shared': False, 'out': 'f32'},
        # the MLP microbenchmark of bench.py: 256 members reading one shared sequence
        {'name': 'mlp population', 'kind': 'mlp', 'members': 256, 'tokens': 2048, 'hidden': F, 'shared': True,
         'out': 'bf16'},
        # attention on separate q, k, v heads (the credit path's baseline): one full-length sequence, short window
        {'name': 'attention one sequence', 'kind': 'heads', 'batch': 1, 'tokens': 2048, 'window': 1024,
         'qk_norm': True},
        # attention of a population with the c_proj dots and the per-head moments, operands as the forward writes them
        {'name': 'attention population', 'kind': 'attention', 'members': 64, 'tokens': 2048, 'window': 2048,
         'format': 'f16_log2', 'moments': True},
        # final norm, fp32 head and soft-capped cross-entropy of a population
        {'name': 'head population', 'kind': 'head', 'members': 128, 'tokens': 2048, 'vocab': V, 'head': 'fp32',
         'input': 'bf16', 'gain': True, 'reduction': 'none'},
        # the whole population forward at its smallest: 8 members, 256 tokens, through the drop-in call
        {'name': 'population small', 'kind': 'population', 'members': 8, 'tokens': 256},
        # the scorer's batch: 16 rows of 2048 tokens at the autocast rounding, per-token losses
        {'name': 'score batch', 'kind': 'score', 'batch': 16, 'tokens': 2048},
        # one training step: 512 members on 8 sequences, fitness, update and Adam
        {'name': 'step', 'kind': 'step', 'pairs': 256, 'chunk_pairs': 32, 'sequences': 8, 'tokens': 2048},
        # the update of a large population alone: fitness, every weight's outer-product sum, Adam
        {'name': 'update', 'kind': 'update', 'pairs': 1536, 'fitness': 'rank'},
        # one chunk of key credit: moved keys, 64 attention reruns, scores through the matched filter, the estimate
        {'name': 'credit keys', 'kind': 'credit', 'which': 'k', 'draws': 64, 'batch': 1, 'tokens': 2048,
         'window': 1024, 'sigma': 0.5},
        # readout probes of 1024 tokens along a cycle of 512 directions
        {'name': 'probes cycle', 'kind': 'probes', 'tokens': 1024, 'directions': 512, 'vocab': V, 'rows': 0},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _tokens128(rng, hi=2048):
    return 128 * _log_int(rng, 1, hi // 128)


def draw(rng):
    kind = rng.choice(('linear', 'linear', 'mlp', 'mlp', 'heads', 'attention', 'attention', 'head', 'head', 'population',
                       'score', 'step', 'update', 'credit', 'probes'))
    if kind == 'linear':
        while True:
            c = {'kind': kind, 'members': _log_int(rng, 1, 64), 'tokens': _log_int(rng, 8, 2048),
                 'd_in': rng.choice((512, 2048, 64 * _log_int(rng, 1, 32))),
                 'd_out': rng.choice((512, 2048, 128 * _log_int(rng, 1, 32))), 'shared': rng.random() < 0.3,
                 'pair': rng.random() < 0.5, 'out': rng.choice(('f32', 'bf16', 'accumulate'))}
            if c['members'] * c['tokens'] * c['d_in'] * c['d_out'] <= 1.5e11:
                return c
    if kind == 'mlp':
        while True:
            c = {'kind': kind, 'members': _log_int(rng, 1, 256), 'tokens': 32 * _log_int(rng, 1, 64),
                 'hidden': rng.choice((F, F, 256 * _log_int(rng, 1, 8))), 'shared': rng.random() < 0.3,
                 'out': rng.choice(('f32', 'bf16', 'accumulate'))}
            if c['members'] * c['tokens'] <= 256 * 2048:
                return c
    if kind == 'heads':
        T = _tokens128(rng)
        return {'kind': kind, 'batch': _log_int(rng, 1, 32), 'tokens': T,
                'window': rng.choice((1024, 2048, _log_int(rng, 32, T))), 'qk_norm': rng.random() < 0.6}
    if kind == 'attention':
        T = _tokens128(rng)
        return {'kind': kind, 'members': _log_int(rng, 1, 128), 'tokens': T,
                'window': rng.choice((1024, 2048, _log_int(rng, 32, T))),
                'format': rng.choice(('f16_log2', 'f16_log2', 'bf16', 'bf16_v')), 'moments': rng.random() < 0.5}
    if kind == 'head':
        while True:
            c = {'kind': kind, 'members': _log_int(rng, 1, 128), 'tokens': _log_int(rng, 16, 2048),
                 'vocab': rng.choice((V, V, V, 256 * _log_int(rng, 2, 32))),
                 'head': rng.choice(('fp32', 'fp32', 'bf16', 'fp32_split')), 'input': rng.choice(('bf16', 'f32')),
                 'gain': rng.random() < 0.5, 'reduction': rng.choice(('member', 'none'))}
            if c['members'] * c['tokens'] * c['vocab'] <= 128 * 2048 * V:
                return c
    if kind == 'population':
        while True:
            c = {'kind': kind, 'members': _log_int(rng, 1, 64), 'tokens': _tokens128(rng)}
            if c['members'] * c['tokens'] <= 32768:
                return c
    if kind == 'score':
        return {'kind': kind, 'batch': _log_int(rng, 1, 16), 'tokens': _tokens128(rng)}
    if kind == 'step':
        while True:
            c = {'kind': kind, 'chunk_pairs': rng.choice((8, 16, 32, 64, 128)), 'sequences': _log_int(rng, 1, 8),
                 'tokens': _tokens128(rng)}
            c['pairs'] = c['chunk_pairs'] * rng.randint(1, 8)
            if 2 * c['pairs'] * c['tokens'] <= 512 * 2048 and c['sequences'] <= 2 * c['pairs']:
                return c
    if kind == 'update':
        return {'kind': kind, 'pairs': _log_int(rng, 16, 2048), 'fitness': rng.choice(('rank', 'zscore'))}
    if kind == 'credit':
        T = _tokens128(rng)
        return {'kind': kind, 'which': rng.choice('qk'), 'draws': _log_int(rng, 4, 64), 'batch': rng.choice((1, 1, 2)),
                'tokens': T, 'window': rng.choice((1024, 2048, _log_int(rng, 32, T))), 'sigma': 0.5}
    return {'kind': 'probes', 'tokens': _log_int(rng, 16, 1024), 'directions': _log_int(rng, 16, 512),
            'vocab': rng.choice((V, V, 256 * _log_int(rng, 2, 16))), 'rows': rng.choice((0, 0, _log_int(rng, 1, 64)))}


# ---------------------------------------------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(DEV).manual_seed(seed)


def _randn(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, device=DEV, generator=g).to(dtype)


def _signs(members, sigma=SIGMA):
    """[+sigma, -sigma, ...]: antithetic members."""
    return torch.tensor([sigma, -sigma], device=DEV).repeat((members + 1) // 2)[:members].contiguous()


def _zipf(g, *shape):
    """Token ids with p(id = r - 1) ~ r^-1.1, as bench.py's sequences."""
    p = torch.arange(1, V + 1, device=DEV, dtype=torch.float32).pow(-1.1)
    n = math.prod(shape)
    return torch.multinomial(p, n, replacement=True, generator=g).view(*shape)


def _shapes():
    """name -> shape of the fixed model's parameters, in the model's order."""
    out = {'resid_lambdas': (LAYERS,), 'x0_lambdas': (LAYERS,), 'transformer.wte.weight': (V, D)}
    for i in range(LAYERS):
        pre = f'transformer.h.{i}.'
        for n in ('c_q', 'c_k', 'c_v', 'c_proj'):
            out[pre + f'attn.{n}.weight'] = (D, D)
        if i % 2:
            out[pre + 'attn.ve_gate.weight'] = (HEADS, VE_CH)
        out[pre + 'mlp.c_fc.weight'] = (F, D)
        out[pre + 'mlp.c_proj.weight'] = (D, F)
    out['lm_head.weight'] = (V, D)
    for i in range(1, LAYERS, 2):
        out[f'value_embeds.{i}.weight'] = (V, D)
    return out


def _state_dict(g):
    """Weights of trained-model scale, the embeddings holding bf16 values as a GPU stores them."""
    out = {}
    for name, shape in _shapes().items():
        if name == 'resid_lambdas':
            w = 1 + 0.1 * _randn(g, *shape)
        elif name == 'x0_lambdas':
            w = 0.1 + 0.05 * _randn(g, *shape)
        elif name == 'transformer.wte.weight':
            w = _randn(g, *shape).bfloat16().float()
        elif name == 'lm_head.weight':
            w = _randn(g, *shape) * (2 * D ** -0.5)
        elif name.endswith('ve_gate.weight'):
            w = _randn(g, *shape) * 0.2
        else:
            scale = (1.5 * (3 / shape[1]) ** 0.5) if 'c_proj' in name else (3 / D) ** 0.5
            w = (2 * torch.rand(*shape, device=DEV, generator=g) - 1) * scale
            if name.startswith('value_embeds'):
                w = w.bfloat16().float()
        out[name] = w
    return out


def _noise(g, rows):
    """One direction per row for every parameter: (a, b) of a matrix, eps of the mixing scalars."""
    return {n: (_randn(g, rows, s[0]), _randn(g, rows, s[1])) if len(s) == 2 else _randn(g, rows, s[0])
            for n, s in _shapes().items()}


def _rotary(T):
    inv = 1.0 / 10000 ** (torch.arange(0, HD, 2, device=DEV, dtype=torch.float32) / HD)
    f = torch.outer(torch.arange(T, device=DEV, dtype=torch.float32), inv)
    return f.cos().bfloat16(), f.sin().bfloat16()


def _unit_heads(x):
    """Rows of 64 scaled to unit mean square (QK norm)."""
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)


def _make_linear(c, g):
    m, T, i, o = c['members'], c['tokens'], c['d_in'], c['d_out']
    dirs = (m + 1) // 2 if c['pair'] else m
    s = {'x': _randn(g, *((T, i) if c['shared'] else (m, T, i)), dtype=torch.bfloat16),
         'w': (_randn(g, o, i) * i ** -0.5).bfloat16(), 'a': _randn(g, dirs, o), 'b': _randn(g, dirs, i),
         'sign': _signs(m, 1e-2), 'T': T, 'shift': int(c['pair']), 'out': None, 'accumulate': c['out'] == 'accumulate',
         'dtype': torch.bfloat16 if c['out'] == 'bf16' else torch.float32}
    if s['accumulate']:
        s['out'] = _randn(g, m, T, o)
    return s


def _make_mlp(c, g):
    m, T, f = c['members'], c['tokens'], c['hidden']
    dirs = (m + 1) // 2
    s = {'x': _randn(g, *((T, D) if c['shared'] else (m, T, D)), dtype=torch.bfloat16),
         'w1': (_randn(g, f, D) * D ** -0.5).bfloat16(), 'w2': (_randn(g, D, f) * f ** -0.5).bfloat16(),
         'v': (_randn(g, dirs, f), _randn(g, dirs, D), _randn(g, dirs, D), _randn(g, dirs, f)), 'sign': _signs(m),
         'T': T, 'accumulate': c['out'] == 'accumulate',
         'out': (_randn(g, m, T, D) if c['out'] == 'accumulate' else
                 torch.empty(m, T, D, device=DEV, dtype=torch.bfloat16 if c['out'] == 'bf16' else torch.float32)),
         'ws': torch.empty(ops.mlp_workspace_bytes(m, T, D, f), device=DEV, dtype=torch.uint8)}
    return s


def _make_heads(c, g):
    q, k, v = (_randn(g, c['batch'], c['tokens'], HEADS, HD) for _ in range(3))
    if c['qk_norm']:
        q, k = _unit_heads(q), _unit_heads(k)
    return {'q': q.bfloat16(), 'k': k.bfloat16(), 'v': v.bfloat16(), 'window': c['window'], 'qk_norm': c['qk_norm']}


FORMATS = {'f16_log2': _lib.QK_F16_Q_LOG2, 'bf16': _lib.QK_BF16, 'bf16_v': _lib.QK_BF16_V_BF16}
LOG2E = 1.4426950408889634


def _make_attention(c, g):
    m, T = c['members'], c['tokens']
    x = _randn(g, m * T, 3, HEADS, HD)
    norm = c['format'] != 'bf16'
    if norm:
        x[:, :2] = _unit_heads(x[:, :2])
    if c['format'] == 'f16_log2':
        x[:, 0] *= LOG2E / 8
        rows = x.half().view(torch.bfloat16)
    else:
        rows = x.bfloat16()
        if c['format'] == 'bf16':
            rows[:, 2] = rows[:, 2].half().view(torch.bfloat16)
    del x
    ws = _lib.size_query('noise_attention_workspace_size', m, T)
    return {'m': m, 'T': T, 'window': c['window'], 'norm': int(norm), 'format': FORMATS[c['format']], 'qkv': rows,
            'b': _randn(g, m, D), 'y': torch.empty(m * T, D, device=DEV, dtype=torch.bfloat16),
            'u': torch.empty(m * T, HEADS, device=DEV),
            'mom': torch.empty(m, HEADS, 2, HD, device=DEV) if c['moments'] else None,
            'ws': torch.empty(ws, device=DEV, dtype=torch.uint8) if c['moments'] else None}


HEAD_CODE = {'fp32': _lib.HEAD_FP32, 'fp32_split': _lib.HEAD_FP32_SPLIT, 'bf16': _lib.HEAD_BF16}


def _make_head(c, g):
    m, T, vocab = c['members'], c['tokens'], c['vocab']
    w = _randn(g, vocab, D) * D ** -0.5
    code = HEAD_CODE[c['head']]
    gain = 0.9 + 0.2 * torch.rand(D, device=DEV, generator=g) if c['gain'] else None
    op = w
    if c['head'] != 'fp32':
        # the formats' operands as a program lays them out once per step (the split one holds hi | lo | hi rows)
        op = torch.empty(vocab, (3 if c['head'] == 'fp32_split' else 1) * D, device=DEV, dtype=torch.bfloat16)
        _lib.call('noise_cast_bf16', w.data_ptr(), op.data_ptr(), w.numel(), D if c['head'] == 'fp32_split' else 0,
                  torch.cuda.current_stream().cuda_stream)
    n = m if c['reduction'] == 'member' else m * T
    ws = _lib.size_query('noise_head_ce_workspace_size', m, T, vocab, code)
    return {'m': m, 'T': T, 'vocab': vocab, 'code': code, 'w32': w, 'w': op, 'gain': gain,
            'x': _randn(g, m * T, D, dtype=torch.bfloat16 if c['input'] == 'bf16' else torch.float32),
            'a': _randn(g, (m + 1) // 2, vocab), 'b': _randn(g, (m + 1) // 2, D), 'sign': _signs(m),
            'targets': _zipf(g, T) % vocab, 'loss': torch.empty(n, device=DEV),
            'red': _lib.CE_MEMBER_MEAN if c['reduction'] == 'member' else _lib.CE_NONE,
            'ws': torch.empty(ws, device=DEV, dtype=torch.uint8)}


def _make_population(c, g):
    m = c['members']
    model = load_model(_state_dict(g), DEV)
    pairs = _noise(g, (m + 1) // 2)

    def per_member(t):
        return t.repeat_interleave(2, 0)[:m].contiguous()
    noise = {n: tuple(per_member(t) for t in v) if isinstance(v, tuple) else per_member(v) for n, v in pairs.items()}
    seq = _zipf(g, c['tokens'] + 1)
    return {'model': model, 'p': dict(model.named_parameters()), 'noise': noise, 'sign': _signs(m),
            'idx': seq[:-1].contiguous(), 'targets': seq[1:].contiguous()}


def _make_score(c, g):
    model = load_model(_state_dict(g), DEV)
    seq = _zipf(g, c['batch'], c['tokens'] + 1)
    return {'model': model, 'weights': Weights(dict(model.named_parameters()), model.config, 'bf16'),
            'x': seq[:, :-1].contiguous(), 'y': seq[:, 1:].contiguous()}


def _make_step(c, g):
    model = load_model(_state_dict(g), DEV)
    seq = _zipf(g, c['sequences'], c['tokens'] + 1)
    return {'es': Eggroll(model, c['pairs'], chunk_pairs=c['chunk_pairs']),
            'opt': Adam(model.parameters(), lr=1e-3, betas=(0.5, 0.95), eps=1e-8), 'step': 0,
            'x': seq[:, :-1].contiguous(), 'y': seq[:, 1:].contiguous()}


def _make_update(c, g):
    """A population's losses and noise rows, and the model's weights and gradients as views of two flat buffers."""
    n = c['pairs']
    shapes = _shapes()
    total = sum(math.prod(s) for s in shapes.values())
    flat, grad = torch.cat([w.flatten() for w in _state_dict(g).values()]), torch.zeros(total, device=DEV)
    noise, params, mats, at = _noise(g, n), [], [], 0
    for name, s in shapes.items():
        k = math.prod(s)
        p = torch.nn.Parameter(flat[at:at + k].view(s), requires_grad=False)
        p.grad = grad[at:at + k].view(s)
        params.append(p)
        if len(s) == 2:
            a, b = noise[name]
            mats.append((a.data_ptr(), s[0], b.data_ptr(), s[1], s[0], s[1], p.grad.data_ptr()))
        else:
            mats.append((0, 0, noise[name].data_ptr(), s[0], 1, s[0], p.grad.data_ptr()))
        at += k
    return {'pairs': n, 'losses': 8.3 + 4e-3 * _randn(g, 2 * n), 'noise': noise, 'flat': flat, 'grad': grad,
            'mode': _lib.FITNESS_RANK if c['fitness'] == 'rank' else _lib.FITNESS_ZSCORE, 'mats': mats,
            'fit': torch.empty(n, device=DEV), 'weight': torch.empty(n, device=DEV),
            'opt': Adam(params, lr=1e-3, betas=(0.5, 0.95), eps=1e-8)}


def _mask(T, window):
    pos = torch.arange(T, device=DEV)
    lag = pos[:, None] - pos[None, :]
    return (lag >= 0) & (lag <= window)


def _rotate(x, cos, sin):
    x1, x2 = x[..., :32], x[..., 32:]
    c, s = cos[:, None, :].to(x.dtype), sin[:, None, :].to(x.dtype)
    return torch.cat([x1 * c + x2 * s, x2 * c - x1 * s], -1)


def _dense_attention(q, k, v, window, dtype, keep=None):
    """softmax(q k^T / 8) v on [b, t, h, 64], one batch row at a time; keep receives each row's probabilities."""
    out, hide = [], ~_mask(q.shape[1], window)
    for i in range(q.shape[0]):
        qh, kh, vh = (t[i].transpose(0, 1).to(dtype).contiguous() for t in (q, k, v))
        p = torch.matmul(qh, kh.transpose(1, 2).contiguous()).mul_(0.125).masked_fill_(hide, float('-inf')).softmax(-1)
        if keep is not None:
            keep.append(p)
        out.append(torch.matmul(p, vh).transpose(0, 1))
    return torch.stack(out)


def _make_credit(c, g):
    n, b, T, window = c['draws'], c['batch'], c['tokens'], c['window']
    cos, sin = (t.float() for t in _rotary(T))
    raw, other = _randn(g, b, T, HEADS, HD), _unit_heads(_rotate(_randn(g, b, T, HEADS, HD), cos, sin)).bfloat16()
    values = _randn(g, b, T, HEADS, HD, dtype=torch.bfloat16)
    moved = _unit_heads(_rotate(raw, cos, sin)).bfloat16()
    q, k = (moved, other) if c['which'] == 'q' else (other, moved)
    maps = []
    base = _dense_attention(q, k, values, window, torch.float32, maps)
    filt = None
    if c['which'] == 'k':
        # the matched filter: the clean attention map, each query's row over its largest weight, transposed
        filt = torch.stack([(p / p.amax(-1, keepdim=True)).transpose(1, 2) for p in maps]).bfloat16().contiguous()
    return {'which': c['which'], 'raw': raw, 'a': _randn(g, n, b, T, HEADS, HD, dtype=torch.bfloat16),
            'sigma': c['sigma'], 'cos': cos, 'sin': sin, 'fixed': other, 'values': values, 'window': window,
            'base': base.bfloat16(), 'target': _randn(g, b, T, HEADS, HD), 'filter': filt}


def _make_probes(c, g):
    n, P, vocab, K = c['tokens'], c['directions'], c['vocab'], c['rows']
    x = _randn(g, n, D) * 1.5
    w = _randn(g, vocab, D) * (2 * D ** -0.5)
    dirs = _randn(g, D, P) * D ** -0.5
    y = _zipf(g, n) % vocab
    y[::17] = -1
    dots, dir_sq, rows = x @ dirs, dirs.square().sum(0), None
    if K:
        rows = torch.randint(0, P, (n, K), device=DEV, generator=g)
        dots, dir_sq = dots.gather(1, rows), dir_sq[rows]
    return {'base': x @ w.t(), 'C': (w @ dirs).t().contiguous(), 'rows': rows, 'y': y,
            'steps': 0.1 * x.square().mean(-1, keepdim=True).sqrt(), 'sq': x.square().sum(-1, keepdim=True),
            'dots': dots.contiguous(), 'dir_sq': dir_sq.contiguous()}


MAKE = {'linear': _make_linear, 'mlp': _make_mlp, 'heads': _make_heads, 'attention': _make_attention,
        'head': _make_head, 'population': _make_population, 'score': _make_score, 'step': _make_step,
        'update': _make_update, 'credit': _make_credit, 'probes': _make_probes}


@torch.no_grad()
def prepare(case, seed):
    return {'kind': case['kind'], **MAKE[case['kind']](case, _gen(seed))}


# ---------------------------------------------------------------------------------------------------- one pass

def _run_attention(s):
    mom, ws = s['mom'], s['ws']
    _lib.call('noise_attention', s['qkv'].data_ptr(), s['m'], s['T'], s['window'], s['norm'], s['format'],
              s['b'].data_ptr(), 0, s['y'].data_ptr(), s['u'].data_ptr(), None if mom is None else mom.data_ptr(),
              None if mom is None else ws.data_ptr(), 0 if mom is None else ws.numel(),
              torch.cuda.current_stream().cuda_stream)
    return {'y': s['y'], 'u': s['u']} if mom is None else {'y': s['y'], 'u': s['u'], 'mom': mom}


def _run_head(s):
    _lib.call('noise_head_ce', s['x'].data_ptr(), int(s['x'].dtype == torch.bfloat16),
              None if s['gain'] is None else s['gain'].data_ptr(), s['w'].data_ptr(), s['vocab'], s['code'],
              s['a'].data_ptr(), s['b'].data_ptr(), s['sign'].data_ptr(), s['targets'].data_ptr(), 0, s['m'], s['T'], 1,
              s['red'], s['loss'].data_ptr(), None, s['ws'].data_ptr(), s['ws'].numel(), None, 0,
              torch.cuda.current_stream().cuda_stream)
    return s['loss']


def _run_step(s):
    s['step'] += 1
    mean = s['es'].step(s['x'], s['y'], s['opt'], s['step'])
    return {'mean': mean, 'losses': s['es'].last_losses, 'params': list(s['es'].params.values())}


def _run_update(s):
    stream = torch.cuda.current_stream().cuda_stream
    n = s['pairs']
    _lib.call('noise_fitness', s['losses'].data_ptr(), 2 * n, n, s['mode'], s['fit'].data_ptr(), s['weight'].data_ptr(),
              stream)
    ptr, count, _keep = _lib.outer_mats(s['mats'])
    _lib.call('noise_outer_update_batch', ptr, count, s['weight'].data_ptr(), n, -1.0 / n, stream)
    s['opt'].step()
    return {'weight': s['weight'], 'grad': s['grad'], 'params': s['flat']}


@torch.no_grad()
def run(state):
    s, kind = state, state['kind']
    if kind == 'linear':
        return ops.lowrank_linear(s['x'], s['w'], s['a'], s['b'], s['sign'], T=s['T'], pair_shift=s['shift'],
                                  out=s['out'], accumulate=s['accumulate'], out_dtype=s['dtype'])
    if kind == 'mlp':
        return ops.lowrank_mlp(s['x'], s['w1'], s['w2'], *s['v'], s['sign'], T=s['T'], pair_shift=1, out=s['out'],
                               accumulate=s['accumulate'], workspace=s['ws'])
    if kind == 'heads':
        return credit.attention(s['q'], s['k'], s['v'], s['window'], s['qk_norm'])
    if kind == 'attention':
        return _run_attention(s)
    if kind == 'head':
        return _run_head(s)
    if kind == 'population':
        return population_loss(s['model'], s['p'], s['noise'], s['sign'], s['idx'], s['targets'])
    if kind == 'score':
        return autocast_forward(s['model'], s['x'], s['y'], 'none', weights=s['weights'])
    if kind == 'step':
        return _run_step(s)
    if kind == 'update':
        return _run_update(s)
    if kind == 'credit':
        return credit.credit_chunk(s['which'], s['raw'], s['a'], s['sigma'], s['cos'], s['sin'], s['fixed'],
                                   s['values'], s['window'], s['base'], s['target'], s['filter'])
    if s['rows'] is None:
        return probes.cycle_derivatives(s['base'], s['C'], s['y'], s['steps'], s['sq'], s['dots'], s['dir_sq'])
    return probes.row_derivatives(s['base'], s['C'], s['rows'], s['y'], s['steps'], s['sq'], s['dots'], s['dir_sq'])


# ---------------------------------------------------------------------------------------------------- work

def _visible(T, window):
    """(query, key) pairs of one head."""
    return sum(min(q, window) + 1 for q in range(T))


PARAMS = sum(math.prod(s) for s in _shapes().values())
NOISE_ROW = sum(sum(s) for s in _shapes().values())


def _forward_flops(T):
    """Of one sequence: the matrices (rank-1 terms are negligible beside them) and the visible attention pairs."""
    mats = LAYERS * 2 * (4 * D * D + 2 * D * F) + (LAYERS // 2) * 2 * VE_CH * HEADS + 2 * D * V
    windows = [1024, 1024, 1024, 2048] * (LAYERS // 4)
    return mats * T + sum(4 * HD * HEADS * _visible(T, w) for w in windows)


def work(case):
    c, kind = case, case['kind']
    if kind == 'linear':
        M, i, o = c['members'] * c['tokens'], c['d_in'], c['d_out']
        dirs = (c['members'] + 1) // 2 if c['pair'] else c['members']
        size = {'f32': 4, 'bf16': 2, 'accumulate': 8}[c['out']]
        rows = c['tokens'] if c['shared'] else M
        return {'bytes': 2 * rows * i + 2 * i * o + 4 * dirs * (i + o) + size * M * o, 'flops': 2 * M * i * o}
    if kind == 'mlp':
        M, f = c['members'] * c['tokens'], c['hidden']
        size = {'f32': 4, 'bf16': 2, 'accumulate': 8}[c['out']]
        rows = c['tokens'] if c['shared'] else M
        return {'bytes': 2 * rows * D + 4 * D * f + 8 * ((c['members'] + 1) // 2) * (D + f) + size * M * D,
                'flops': 4 * M * D * f}
    if kind == 'heads':
        M = c['batch'] * c['tokens']
        return {'bytes': 4 * 2 * M * D, 'flops': 4 * HD * HEADS * c['batch'] * _visible(c['tokens'], c['window'])}
    if kind == 'attention':
        m, M = c['members'], c['members'] * c['tokens']
        return {'bytes': 4 * 2 * M * D + 4 * m * D + 4 * M * HEADS + 4 * m * HEADS * 2 * HD * c['moments'],
                'flops': 4 * HD * HEADS * m * _visible(c['tokens'], c['window'])}
    if kind == 'head':
        M, vocab = c['members'] * c['tokens'], c['vocab']
        size = 2 if c['input'] == 'bf16' else 4
        return {'bytes': size * M * D + 4 * vocab * D + 4 * ((c['members'] + 1) // 2) * (vocab + D) +
                4 * (c['members'] if c['reduction'] == 'member' else M), 'flops': 2 * M * D * vocab}
    if kind == 'population':
        m, T = c['members'], c['tokens']
        return {'bytes': 4 * PARAMS + 4 * m * NOISE_ROW + 16 * T + 4 * m, 'flops': m * _forward_flops(T)}
    if kind == 'score':
        B, T = c['batch'], c['tokens']
        # the linear weights and the head in bf16, the embedding rows that the tokens name in fp32
        emb = 5 * V * D
        return {'bytes': 2 * (PARAMS - emb) + 4 * min(B * T, V) * 5 * D + 20 * B * T, 'flops': B * _forward_flops(T)}
    if kind == 'step':
        n, T = c['pairs'], c['tokens']
        # weights, gradients and both moments move through the update; every direction's noise row is read once
        return {'bytes': 4 * 7 * PARAMS + 4 * n * NOISE_ROW, 'flops': 2 * n * _forward_flops(T) + 2 * n * PARAMS}
    if kind == 'update':
        n = c['pairs']
        return {'bytes': 4 * n * NOISE_ROW + 4 * 8 * PARAMS + 16 * n, 'flops': 2 * n * PARAMS}
    if kind == 'credit':
        n, b, T = c['draws'], c['batch'], c['tokens']
        M = b * T
        flops = 4 * HD * HEADS * n * b * _visible(T, c['window'])
        size = 2 * n * M * D + 4 * M * D + 2 * 3 * M * D + 4 * 2 * M * D
        if c['which'] == 'k':
            size += 2 * b * HEADS * T * T
            flops += 2 * b * HEADS * T * T * n
        return {'bytes': size, 'flops': flops}
    n, P, vocab = c['tokens'], c['directions'], c['vocab']
    K = c['rows'] or P
    return {'bytes': 4 * (n * vocab + P * vocab + 2 * n * K + P), 'flops': 10 * n * K * vocab}


# ---------------------------------------------------------------------------------------------------- 64 bits

def _norm(x):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)


def _lowrank64(x, w, a, b, s):
    """x [m, T, in] through w + s a b^T of each member."""
    return x @ w.t() + s * (x @ b.unsqueeze(-1)) * a.unsqueeze(1)


def _forward64(p, noise, sign, idx, targets, step=8, none=False):
    """Losses of perturbed members, `step` at a time: mean per member, or per token. idx [m, T]; noise rows per member."""
    T = idx.shape[1]
    cos, sin = _rotary(T)
    step = max(1, min(step, 16384 // T))
    p = {n: w.to(f64) for n, w in p.items()}
    out = []
    for lo in range(0, idx.shape[0], step):
        sl = slice(lo, lo + step)
        nz = {n: tuple(t[sl].to(f64) for t in v) if isinstance(v, tuple) else v[sl].to(f64) for n, v in noise.items()}
        s, ids = sign[sl].to(f64)[:, None, None], idx[sl]
        m = ids.shape[0]

        def embed(name):
            a, b = nz[name]
            return p[name][ids] + s * a.gather(1, ids).unsqueeze(-1) * b.unsqueeze(1)

        def lin(name, x):
            return _lowrank64(x, p[name], *nz[name], s)
        x = x0 = _norm(embed('transformer.wte.weight'))
        for i in range(LAYERS):
            pre = f'transformer.h.{i}.'
            x = ((p['resid_lambdas'][i] + s * nz['resid_lambdas'][:, i, None, None]) * x +
                 (p['x0_lambdas'][i] + s * nz['x0_lambdas'][:, i, None, None]) * x0)
            h = _norm(x)
            q, k, v = (lin(pre + f'attn.c_{n}.weight', h).view(m, T, HEADS, HD) for n in 'qkv')
            if i % 2:
                gate = 2 * torch.sigmoid(lin(pre + 'attn.ve_gate.weight', h[..., :VE_CH]))
                v = v + gate.unsqueeze(-1) * embed(f'value_embeds.{i}.weight').view(m, T, HEADS, HD)
            q, k = _norm(_rotate(q, cos, sin)), _norm(_rotate(k, cos, sin))
            y = _dense_attention(q, k, v, 2048 if i % 4 == 3 else 1024, f64).reshape(m, T, D)
            x = x + lin(pre + 'attn.c_proj.weight', y)
            x = x + lin(pre + 'mlp.c_proj.weight', lin(pre + 'mlp.c_fc.weight', _norm(x)).relu().square())
        z = 15 * torch.tanh(lin('lm_head.weight', _norm(x)) / 15)
        ce = torch.logsumexp(z, -1) - z.gather(-1, targets[sl].unsqueeze(-1)).squeeze(-1)
        out.append(ce.flatten() if none else ce.mean(-1))
    return torch.cat(out)


def _by_member(members, rows, f, lim=1 << 17):
    """f over slices of members whose rows stay under lim, concatenated."""
    step = max(1, lim // rows)
    return torch.cat([f(slice(lo, min(members, lo + step))) for lo in range(0, members, step)])


def _exact_linear(c, s):
    x, w = s['x'], s['w'].to(f64)
    pick = torch.arange(c['members'], device=DEV) >> s['shift']
    a, b = s['a'][pick].to(f64), s['b'][pick].to(f64)

    def some(sl):
        xs = (x.unsqueeze(0) if c['shared'] else x[sl]).to(f64)
        y = _lowrank64(xs, w, a[sl], b[sl], s['sign'][sl].to(f64)[:, None, None])
        return s['out'][sl].to(f64) + y if s['accumulate'] else y
    return _by_member(c['members'], c['tokens'], some)


def _exact_mlp(c, s):
    x, w1, w2 = s['x'], s['w1'].to(f64), s['w2'].to(f64)
    pick = torch.arange(c['members'], device=DEV) >> 1
    a1, b1, a2, b2 = (t[pick].to(f64) for t in s['v'])

    def some(sl):
        sg = s['sign'][sl].to(f64)[:, None, None]
        xs = (x.unsqueeze(0) if c['shared'] else x[sl]).to(f64)
        y = _lowrank64(_lowrank64(xs, w1, a1[sl], b1[sl], sg).relu().square(), w2, a2[sl], b2[sl], sg)
        return s['out'][sl].to(f64) + y if s['accumulate'] else y
    return _by_member(c['members'], c['tokens'], some, 1 << 16)


def _exact_attention(c, s):
    m, T = c['members'], c['tokens']
    rows = s['qkv'].view(m, T, 3, HEADS, HD)
    half = c['format'] == 'f16_log2'
    y, u, mom = [], [], []
    for i in range(m):
        q, k, v = (rows[i, :, j].view(torch.float16) if half or (j == 2 and c['format'] == 'bf16') else rows[i, :, j]
                   for j in range(3))
        q = q.to(f64) * (8 / LOG2E if half else 1)
        o = _dense_attention(q.unsqueeze(0), k.unsqueeze(0), v.unsqueeze(0), c['window'], f64)[0]
        y.append(o.reshape(T, D))
        u.append((o * s['b'][i].to(f64).view(HEADS, HD)).sum(-1))
        mom.append(torch.stack([o.mean(0), o.square().mean(0)], 1))
    out = {'y': torch.cat(y), 'u': torch.cat(u)}
    if c['moments']:
        out['mom'] = torch.stack(mom)
    return out


def _exact_head(c, s):
    m, T = c['members'], c['tokens']
    x, w = s['x'].view(m, T, D), s['w32'].to(f64)

    def some(sl):
        pick = torch.arange(sl.start, sl.stop, device=DEV) >> 1
        h = _norm(x[sl].to(f64))
        if s['gain'] is not None:
            h = h * s['gain'].to(f64)
        z = _lowrank64(h, w, s['a'][pick].to(f64), s['b'][pick].to(f64), s['sign'][sl].to(f64)[:, None, None])
        z = 15 * torch.tanh(z / 15)
        ce = torch.logsumexp(z, -1) - z[..., torch.arange(T, device=DEV), s['targets']]
        return ce.mean(-1) if c['reduction'] == 'member' else ce.flatten()
    return _by_member(m, T, some, 1 << 14)


def _exact_step(c, s):
    """The member losses (fp32 N(0, 1) slices of the fixed noise buffer, antithetic members, one sequence per chunk).
    The first Adam step moves a weight by lr times its gradient's sign, and rounding decides the sign of a gradient
    near zero: the weights have no value of their own here."""
    n, cp = c['pairs'], c['chunk_pairs']
    params = {name: w.clone() for name, w in s['es'].params.items()}
    buf = torch.randn(2 ** 28, device=DEV, generator=_gen(0))
    g = _gen(1)
    noise = {}
    members = max(2 * n, 2 * c['sequences'])
    pick = torch.arange(members, device=DEV) // 2 % n
    for name, w in params.items():
        off = torch.randint(0, 2 ** 28 - sum(w.shape), (n,), device=DEV, generator=g)
        rows = buf[off[:, None] + torch.arange(sum(w.shape), device=DEV)][pick]
        noise[name] = rows.split(list(w.shape), 1) if w.dim() == 2 else rows
    per_seq = members // c['sequences']
    seq = torch.arange(members, device=DEV) // (2 * cp) * (2 * cp) // per_seq
    losses = _forward64(params, noise, _signs(members, 0.002), s['x'][seq], s['y'][seq])
    return {'mean': losses.mean(), 'losses': losses, 'params': [None] * len(params)}


def _exact_update(c, s):
    n = c['pairs']
    f = s['losses'].to(f64).view(n, 2)
    f = f[:, 1] - f[:, 0]
    if c['fitness'] == 'rank':
        f32 = s['losses'].view(n, 2)
        order = torch.sort(f32[:, 1] - f32[:, 0], stable=True).indices
        weight = torch.empty(n, device=DEV, dtype=f64)
        weight[order] = torch.arange(n, device=DEV, dtype=f64) / (n - 1) - 0.5
    else:
        weight = f / (f.std() + 1e-8)
    grads = []
    for name, v in s['noise'].items():
        if isinstance(v, tuple):
            a, b = (t.to(f64) for t in v)
            grads.append((a * weight[:, None]).t().contiguous() @ b)
        else:
            grads.append(weight @ v.to(f64))
    grad = torch.cat([x.flatten() for x in grads]) * (-1.0 / n)
    return {'weight': weight, 'grad': grad, 'params': s['flat'].to(f64) - 1e-3 * grad / (grad.abs() + 1e-8)}


def _exact_credit(c, s):
    n, b, T = c['draws'], c['batch'], c['tokens']
    cos, sin = s['cos'].to(f64), s['sin'].to(f64)
    score = torch.empty(b, HEADS, T, n, device=DEV, dtype=f64)
    for j in range(n):
        moved = _norm(_rotate(s['raw'].to(f64) + c['sigma'] * s['a'][j].to(f64), cos, sin))
        q, k = (moved, s['fixed']) if c['which'] == 'q' else (s['fixed'], moved)
        o = _dense_attention(q, k, s['values'], c['window'], f64)
        score[..., j] = ((o - s['base'].to(f64)) * s['target'].to(f64)).sum(-1).transpose(1, 2)
    if c['which'] == 'k':
        score = torch.stack([s['filter'][i].to(f64) @ score[i] for i in range(b)])
    est = torch.zeros(b, T, HEADS, HD, device=DEV, dtype=f64)
    for j in range(n):
        est += score[..., j].transpose(1, 2).unsqueeze(-1) * s['a'][j].to(f64)
    return est


def _exact_probes(c, s):
    base, C, y = s['base'].to(f64), s['C'].to(f64), s['y']
    steps, sq, dots, dir_sq = (s[k].to(f64) for k in ('steps', 'sq', 'dots', 'dir_sq'))
    tgt = y.clamp(min=0)

    def loss(z, t):
        z = 15 * torch.tanh(z / 15)
        return torch.logsumexp(z, -1) - z.gather(-1, t.unsqueeze(-1)).squeeze(-1)
    out = []
    for i in range(c['tokens']):
        mine = C if s['rows'] is None else C[s['rows'][i]]
        clean = loss(base[i] * torch.rsqrt(sq[i] / D + EPS), tgt[i])
        dsq = dir_sq if s['rows'] is None else dir_sq[i]
        inv = torch.rsqrt((sq[i] + 2 * steps[i] * dots[i] + steps[i] ** 2 * dsq) / D + EPS)
        z = (base[i] + steps[i] * mine) * inv[:, None]
        out.append((loss(z, tgt[i].expand(z.shape[0])) - clean) / steps[i] * (y[i] >= 0))
    return torch.stack(out)


@torch.no_grad()
def exact(case, seed):
    c = case
    s = prepare(case, seed)
    kind = c['kind']
    if kind == 'heads':
        return _dense_attention(s['q'], s['k'], s['v'], c['window'], f64)
    if kind == 'population':
        one = torch.zeros(c['members'], 1, device=DEV, dtype=torch.int64)
        return _forward64(s['p'], s['noise'], s['sign'], s['idx'] + one, s['targets'] + one)
    if kind == 'score':
        zero = {n: tuple(torch.zeros(c['batch'], k, device=DEV) for k in w.shape) if w.dim() == 2 else
                torch.zeros(c['batch'], w.shape[0], device=DEV) for n, w in s['model'].named_parameters()}
        return _forward64(dict(s['model'].named_parameters()), zero, torch.zeros(c['batch'], device=DEV), s['x'], s['y'],
                          none=True)
    return {'linear': _exact_linear, 'mlp': _exact_mlp, 'attention': _exact_attention, 'head': _exact_head,
            'step': _exact_step, 'update': _exact_update, 'credit': _exact_credit, 'probes': _exact_probes}[kind](c, s)


def tolerance(case):
    """About four times the error against 64 bits (or, for a whole step, against the step with the other fp32 head)."""
    kind = case['kind']
    if kind == 'linear':
        return {'rel': 8e-3}  # bf16 products: 2.3e-3
    if kind == 'mlp':
        return {'rel': 1.6e-2}  # bf16 hidden rounded twice: 4.4e-3
    if kind in ('heads', 'attention'):
        return {'rel': 1e-2}  # fp16 or bf16 probabilities, bf16 output and its dots: 2.7e-3
    if kind == 'head':
        # per token 2.3e-5 (fp16 h), 3.2e-4 (bf16), 5e-7 (bf16 pairs); means over a member average their rounding
        per_token = {'fp32': 1e-4, 'bf16': 1.2e-3, 'fp32_split': 2e-6}[case['head']]
        return {'rel': per_token if case['reduction'] == 'none' else per_token / 4}
    if kind == 'population':
        return {'rel': 5e-4}  # 1.5e-4
    if kind == 'score':
        return {'rel': 1e-2}  # 2.9e-3: a bf16 residual stream through 8 layers
    if kind == 'step':
        # losses 2e-4; the weights (2e-3) differ where rounding turns the sign of a gradient near zero, each by 2 lr
        return {'rel': 8e-3, 'max': 0.5}
    if kind == 'update':
        return {'rel': 3e-6, 'max': 1e-2}  # 8e-7; a weight near zero moves by lr times a sign that rounding may turn
    if kind == 'credit':
        return {'rel': 2.4e-2, 'max': 0.5}  # 5.9e-3: the change of bf16 attention outputs, 0.11 where it is smallest
    return {'rel': 6e-4}  # probes: 1.5e-4, a difference of fp32 losses over the step
