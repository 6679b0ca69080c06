"""The work that users of this package have it do, as cases that can be timed and checked.

A training case is what a training program does between two reports: it resumes from
weights and optimizer state it holds, takes a few compiled steps (forward, backward and
optimizer in one call each), and reads the losses and the updated weights back. Batches
come either from host arrays, as `step` takes them, or from slots staged on the device, as
a program that prefetches keeps them. An inference case is one `run` of a compiled forward.

Weights are of the size that a model in the middle of a training has them (N(0, 1/fan_in),
biases and norms that are not at their initial values), and Adam's second moments are warm,
so that an update is a smooth function of its gradient, as it is after the first few
hundred steps of a training.
"""
import math

import numpy as np
import torch

import tensorgrad_amd.ops as O
from tensorgrad_amd import configs, nn
from tensorgrad_amd.backend import NativeRuntime
from tensorgrad_amd.compile import compile_forward, trace, trace_forward
from tensorgrad_amd.module import Module

RESUMED_AT = 1000          # optimizer steps (and PRNG seeds) taken before a training case begins
SLOTS = 4                  # batches that a staged case keeps on the device
TAPS = [(2.0 ** k) * math.pi for k in range(configs.N_FREQS)]


# ---- models that only these cases need ------------------------------------------------------

class Images(Module):
    """Two 3x3 convolutions, a 2x2 pool and two linear layers over [B, 1, S, S] images."""

    def __init__(self, size, c1, c2, hidden):
        self.conv1 = nn.Conv2d(1, c1, 3)
        self.conv2 = nn.Conv2d(c1, c2, 3)
        self.fc1 = nn.Linear(c2 * ((size - 4) // 2) ** 2, hidden)
        self.fc2 = nn.Linear(hidden, 10)


class Downsample(Module):
    """A padded convolution and a strided one that halves the image."""

    def __init__(self, c1, c2):
        self.same = nn.Conv2d(c1, c2, 3, padding=1)
        self.half = nn.Conv2d(c2, c2, 3, stride=2, padding=1)


class AttentionBlock(Module):
    def __init__(self, d):
        self.ln1 = nn.LayerNorm(d)
        self.attn = configs.Attention(d)


class FeedForward(Module):
    def __init__(self, d, hidden):
        self.ln2 = nn.LayerNorm(d)
        self.mlp = configs.MLP(d, hidden)


class Head(Module):
    """Token embedding, norm and output head: what a language model does per vocabulary entry."""

    def __init__(self, vocab, d):
        self.emb = nn.Embedding(vocab, d)
        self.lnf = nn.LayerNorm(d)
        self.head = nn.Linear(d, vocab)


def _squares(y, target):
    return O.mean(O.square(O.sub(y, target)))


def _downsample_loss(p, inp):
    return _squares(p.half.fwd(O.relu(p.same.fwd(inp['x']))), inp['target'])


def _attention_loss(heads, drop):
    def loss(p, inp):
        x = inp['x']
        return _squares(O.add(x, configs._attention(p.attn, p.ln1.fwd(x), heads, drop)), inp['target'])
    return loss


def _feed_forward_loss(drop):
    def loss(p, inp):
        x = inp['x']
        y = p.mlp.down.fwd(O.gelu(p.mlp.up.fwd(p.ln2.fwd(x))))
        return _squares(O.add(x, O.dropout(y, drop)), inp['target'])
    return loss


def _head_loss(p, inp):
    return nn.cross_entropy(p.head.fwd(p.lnf.fwd(p.emb.fwd(inp['tokens']))), inp['targets'])


def _nerf_colors(m, inp):
    pe = configs.nerf_pos_enc(inp['x'], inp['freqs'])
    h = pe
    for i, layer in enumerate(m.layers):
        h = O.relu(layer.fwd(O.concat([h, pe], 1) if i == m.skip else h))
    return m.head.fwd(h)


# ---- the kinds of work ------------------------------------------------------------------------

ADAM = {'kind': 'adam', 'lr': 1e-3}
ADAMW = {'kind': 'adamw', 'lr': 3e-4, 'weightDecay': 0.01}
SGD = {'kind': 'sgd', 'lr': 0.01, 'momentum': 0.9}


def _i32(*shape):
    return {'shape': list(shape), 'dtype': 'i32'}


def _program(c):
    """(model, loss or forward, inputs, optimizer) of a case, as a user writes them."""
    k = c['kind']
    if k == 'sin_mlp':
        return (configs.SinMLP(c['hidden']), configs.sin_mlp_loss,
                {'x': [c['batch'], 1], 'y': [c['batch'], 1]}, ADAM)
    if k == 'char_mlp':
        return (configs.CharMLP(c['vocab'], c['context'], c['emb'], c['hidden']), configs.char_mlp_loss,
                {'tokens': _i32(c['batch'], c['context']), 'targets': _i32(c['batch'])}, dict(ADAMW, lr=1e-3))
    if k == 'cnn':
        return (Images(c['size'], c['c1'], c['c2'], c['hidden']), configs.cnn_loss,
                {'x': [c['batch'], 1, c['size'], c['size']], 'y': _i32(c['batch'])}, dict(SGD, lr=1e-4))
    if k == 'conv':
        s, half = c['size'], (c['size'] + 1) // 2
        return (Downsample(c['c1'], c['c2']), _downsample_loss,
                {'x': [c['batch'], c['c1'], s, s], 'target': [c['batch'], c['c2'], half, half]}, dict(SGD, lr=1e-3))
    if k in ('nerf', 'render'):
        model = configs.NeRF(c['width'], c['depth'], c['depth'] // 2)
        if k == 'render':
            return model, _nerf_colors, {'x': [None, 3], 'freqs': [configs.N_FREQS]}, None
        return (model, configs.nerf_loss, {'x': [c['points'], 3], 'freqs': [configs.N_FREQS], 'target': [c['points'], 4]},
                dict(ADAM, lr=5e-4))
    if k in ('transformer', 'logits'):
        model = configs.Transformer(c['vocab'], c['seq'], c['dim'], c['layers'], c['heads'], 4 * c['dim'],
                                    c['drop'] if k == 'transformer' else 0.0)
        if k == 'logits':
            return model, lambda p, inp: configs.transformer_logits(p, inp['tokens']), {'tokens': _i32(c['batch'], c['seq'])}, None
        opt = dict(ADAMW, clipGradNorm=c['clip']) if c['clip'] else ADAMW
        return (model, configs.transformer_loss,
                {'tokens': _i32(c['batch'], c['seq']), 'targets': _i32(c['batch'], c['seq'])}, opt)
    if k == 'attention':
        shape = [c['batch'], c['seq'], c['dim']]
        return AttentionBlock(c['dim']), _attention_loss(c['heads'], c['drop']), {'x': shape, 'target': shape}, SGD
    if k == 'feed_forward':
        shape = [c['rows'], c['dim']]
        return FeedForward(c['dim'], c['hidden']), _feed_forward_loss(c['drop']), {'x': shape, 'target': shape}, SGD
    if k == 'head':
        return (Head(c['vocab'], c['dim']), _head_loss, {'tokens': _i32(c['rows']), 'targets': _i32(c['rows'])}, ADAMW)
    raise KeyError(k)


def _batch(c, rng):
    """One batch of a case's inputs, with the distributions that its data has."""
    k = c['kind']
    f32 = lambda a: np.asarray(a, np.float32)  # noqa: E731
    ids = lambda n, *shape: rng.integers(0, n, shape, dtype=np.int32)  # noqa: E731
    if k == 'sin_mlp':
        x = f32(rng.uniform(-math.pi, math.pi, (c['batch'], 1)))
        return {'x': x, 'y': f32(np.sin(x.astype(np.float64)))}
    if k == 'char_mlp':
        return {'tokens': ids(c['vocab'], c['batch'], c['context']), 'targets': ids(c['vocab'], c['batch'])}
    if k == 'cnn':
        return {'x': rng.random((c['batch'], 1, c['size'], c['size']), dtype=np.float32), 'y': ids(10, c['batch'])}
    if k == 'conv':
        s, half = c['size'], (c['size'] + 1) // 2
        return {'x': rng.standard_normal((c['batch'], c['c1'], s, s), dtype=np.float32),
                'target': rng.standard_normal((c['batch'], c['c2'], half, half), dtype=np.float32)}
    if k in ('nerf', 'render'):
        got = {'x': f32(rng.uniform(-1, 1, (c['points'], 3))), 'freqs': f32(TAPS)}
        return dict(got, target=rng.random((c['points'], 4), dtype=np.float32)) if k == 'nerf' else got
    if k == 'transformer':
        return {'tokens': ids(c['vocab'], c['batch'], c['seq']), 'targets': ids(c['vocab'], c['batch'], c['seq'])}
    if k == 'logits':
        return {'tokens': ids(c['vocab'], c['batch'], c['seq'])}
    if k == 'head':
        return {'tokens': ids(c['vocab'], c['rows']), 'targets': ids(c['vocab'], c['rows'])}
    shape = (c['batch'], c['seq'], c['dim']) if k == 'attention' else (c['rows'], c['dim'])
    return {'x': rng.standard_normal(shape, dtype=np.float32), 'target': rng.standard_normal(shape, dtype=np.float32)}


def _weights(c, shapes, rng):
    """Weights and Adam second moments of a training under way: {name: f32 array} each."""
    relu = c['kind'] in ('sin_mlp', 'cnn', 'conv', 'nerf', 'render')
    p, v = {}, {}
    for name, shape in shapes.items():
        last = name.rsplit('.', 1)[-1]
        w = rng.standard_normal(int(np.prod(shape)), dtype=np.float32)
        if last == 'g':
            w = 1 + w / 10
        elif last == 'b':
            w = w / 10
        elif 'emb' in name:
            w = w / 2
        else:
            fan = shape[0] if len(shape) == 2 else int(np.prod(shape[1:]))
            w = w * math.sqrt((2 if relu else 1) / fan)
        p[name] = np.asarray(w, np.float32)
        v[name] = np.asarray(GRADIENT.get(c['kind'], 1.0) ** 2 * rng.uniform(0.5, 1.5, w.size), np.float32)
    return p, v


# size of the gradients that Adam's second moments have seen
GRADIENT = {'sin_mlp': 1.0, 'char_mlp': 1e-2, 'nerf': 3e-2, 'transformer': 1e-2, 'head': 1e-3}
BATCHES = 4                # host batches that a training program cycles through


def _given(c, seed):
    """(program, traced graph's parameter shapes, batches, weights, second moments) from the seed alone."""
    rng = np.random.default_rng([int(seed), len(c['kind'])])
    model, fn, inputs, opt = _program(c)
    if opt is None:
        known = {n: ({'shape': [c['points'] if d is None else d for d in s], 'dtype': 'f32'} if isinstance(s, list) else s)
                 for n, s in inputs.items()}
        ir = trace_forward(model, fn, known)
        batches = [_batch(c, rng)]
    else:
        ir = trace(model, fn, inputs, opt)
        batches = [_batch(c, rng) for _ in range(min(BATCHES, c['steps']))]
    p, v = _weights(c, ir.param_shapes(), rng)
    return (model, fn, inputs, opt), ir, batches, p, v


class _Program:
    """What a program holds: the compiled graph, its batches; freed with the last reference."""

    def __init__(self, case, handle, batches):
        self.case, self.handle, self.batches = case, handle, batches

    def __del__(self):
        self.handle.destroy()


# ---- the interface ------------------------------------------------------------------------------

def listed():
    return [
        # regression of a curve by a tiny MLP: launches and latency are all there is
        {'name': 'sin_mlp', 'kind': 'sin_mlp', 'batch': 256, 'hidden': 64, 'steps': 64, 'feed': 'host'},
        # a character model over a window of tokens: embedding, tanh layer, small head
        {'name': 'char_mlp', 'kind': 'char_mlp', 'batch': 1024, 'vocab': 27, 'context': 8, 'emb': 24, 'hidden': 512,
         'steps': 32, 'feed': 'host'},
        # an image classifier
        {'name': 'cnn', 'kind': 'cnn', 'batch': 128, 'size': 28, 'c1': 32, 'c2': 64, 'hidden': 128, 'steps': 32,
         'feed': 'host'},
        # a coordinate network over the rays of a large batch: long GEMMs of width 256, the largest case
        {'name': 'nerf', 'kind': 'nerf', 'points': 65536, 'width': 256, 'depth': 8, 'steps': 6, 'feed': 'staged'},
        # a language model's training step with dropout
        {'name': 'transformer', 'kind': 'transformer', 'batch': 32, 'seq': 128, 'dim': 256, 'layers': 4, 'heads': 4,
         'vocab': 65, 'drop': 0.1, 'clip': 0.0, 'steps': 24, 'feed': 'host'},
        # a sample-sized transformer with clipped gradients: many small launches
        {'name': 'transformer_small', 'kind': 'transformer', 'batch': 64, 'seq': 16, 'dim': 64, 'layers': 2, 'heads': 4,
         'vocab': 13, 'drop': 0.0, 'clip': 1.0, 'steps': 24, 'feed': 'host'},
        # one attention layer of a wider model at a ragged sequence length
        {'name': 'attention', 'kind': 'attention', 'batch': 8, 'seq': 200, 'dim': 512, 'heads': 8, 'drop': 0.1,
         'steps': 16, 'feed': 'staged'},
        # one MLP layer of a wider model
        {'name': 'feed_forward', 'kind': 'feed_forward', 'rows': 4000, 'dim': 512, 'hidden': 2048, 'drop': 0.1,
         'steps': 16, 'feed': 'staged'},
        # embedding and head of a larger, odd vocabulary
        {'name': 'head', 'kind': 'head', 'rows': 2048, 'dim': 256, 'vocab': 5003, 'steps': 16, 'feed': 'staged'},
        # a convolution stage inside a network
        {'name': 'conv', 'kind': 'conv', 'batch': 32, 'size': 33, 'c1': 32, 'c2': 64, 'steps': 16, 'feed': 'staged'},
        # inference: colours of a frame's worth of points, from host array to host array
        {'name': 'render', 'kind': 'render', 'points': 50000, 'width': 256, 'depth': 8},
        # inference: the logits of one request
        {'name': 'logits', 'kind': 'logits', 'batch': 1, 'seq': 128, 'dim': 256, 'layers': 4, 'heads': 4, 'vocab': 65},
    ]


LARGEST = 1.1e12           # operations of the largest listed case (nerf): no drawn case costs more


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    k = rng.choice(['sin_mlp', 'char_mlp', 'cnn', 'nerf', 'transformer', 'attention', 'feed_forward', 'head', 'conv',
                    'render', 'logits'])
    c = {'kind': k}
    if k == 'sin_mlp':
        c.update(batch=_log(rng, 16, 16384), hidden=_log(rng, 8, 128), steps=32, feed='host')
    elif k == 'char_mlp':
        c.update(batch=_log(rng, 64, 8192), vocab=rng.randint(20, 128), context=rng.randint(3, 16), emb=rng.randint(8, 64),
                 hidden=_log(rng, 64, 1024), steps=16, feed='host')
    elif k == 'cnn':
        c.update(batch=_log(rng, 8, 256), size=rng.randint(12, 40), c1=rng.choice([8, 12, 16, 32, 48]),
                 c2=rng.choice([16, 24, 32, 64, 80]), hidden=_log(rng, 32, 256), steps=16, feed='host')
    elif k == 'nerf':
        c.update(points=_log(rng, 256, 65536), width=rng.choice([32, 64, 100, 128, 192, 256]), depth=rng.randint(4, 8),
                 steps=6, feed='staged')
    elif k == 'transformer':
        heads = rng.choice([2, 4, 6])
        c.update(batch=_log(rng, 2, 48), seq=_log(rng, 8, 256), dim=heads * rng.choice([8, 16, 32, 48, 64]),
                 layers=rng.randint(1, 4), heads=heads, vocab=rng.randint(13, 200), drop=rng.choice([0.0, 0.1]),
                 clip=rng.choice([0.0, 1.0]), steps=12, feed='host')
    elif k == 'attention':
        heads = rng.randint(1, 8)
        c.update(batch=_log(rng, 1, 32), seq=_log(rng, 16, 512), dim=heads * rng.choice([16, 32, 40, 64, 96]), heads=heads,
                 drop=rng.choice([0.0, 0.1]), steps=12, feed='staged')
    elif k == 'feed_forward':
        d = rng.randint(32, 768)
        c.update(rows=_log(rng, 64, 8192), dim=d, hidden=rng.choice([2, 4]) * d, drop=rng.choice([0.0, 0.1]), steps=12,
                 feed='staged')
    elif k == 'head':
        c.update(rows=_log(rng, 64, 4096), dim=rng.randint(32, 512), vocab=_log(rng, 50, 8000), steps=12, feed='staged')
    elif k == 'conv':
        c.update(batch=_log(rng, 2, 64), size=rng.randint(9, 48), c1=rng.choice([3, 8, 16, 32, 48, 64]),
                 c2=rng.choice([8, 16, 32, 48, 64, 96]), steps=12, feed='staged')
    elif k == 'render':
        c.update(points=_log(rng, 64, 65536), width=rng.choice([32, 64, 100, 128, 192, 256]), depth=rng.randint(4, 8))
    else:
        heads = rng.choice([2, 4, 6])
        c.update(batch=_log(rng, 1, 32), seq=_log(rng, 8, 256), dim=heads * rng.choice([16, 32, 64]),
                 layers=rng.randint(1, 4), heads=heads, vocab=rng.randint(13, 200))
    count = next(n for n in ('batch', 'rows', 'points') if n in c)
    while work(c)['flops'] > LARGEST:
        c[count] = c[count] * 3 // 4
    return c


def prepare(case, seed):
    (model, fn, inputs, opt), ir, batches, p, v = _given(case, seed)
    if opt is None:
        forward = compile_forward(model, fn, inputs, seed=0)
        forward.upload_params(p)
        forward.run(batches[0])            # compiles the graph of this shape
        return _Program(case, forward, batches)
    rt = NativeRuntime(ir.wire_json())
    rt.upload_params(p)
    state = {}
    for name in rt.state_names():
        of = name.split('_', 2)[2]
        state[name] = v[of] if name.startswith('adam_v_') else np.zeros(p[of].size, np.float32)
    rt.upload_state(state, RESUMED_AT, RESUMED_AT)
    if case['feed'] == 'staged':
        for slot, b in enumerate(batches):
            rt.stage_batch(slot, b)
    return _Program(case, rt, batches)


def run(state):
    c, at, n = state.case, state.handle, len(state.batches)
    if 'steps' not in c:
        r = at.run(state.batches[0])
        if r.error is not None:
            raise r.error
        return r.output
    if c['feed'] == 'staged':
        losses = [at.step_staged(i % n) for i in range(c['steps'])]
    else:
        losses = [at.step(state.batches[i % n]) for i in range(c['steps'])]
    return {'losses': np.array(losses, np.float32), 'weights': at.download_params()}


# ---- work and tolerance --------------------------------------------------------------------------

def _flops(c):
    """Floating point operations of one forward's matrix products and convolutions, and of its first
    layer's (whose input takes no gradient)."""
    k = c['kind']
    if k == 'sin_mlp':
        return 2 * c['batch'] * (2 * c['hidden'] + c['hidden'] ** 2), 2 * c['batch'] * c['hidden']
    if k == 'char_mlp':
        return 2 * c['batch'] * c['hidden'] * (c['context'] * c['emb'] + c['vocab']), 0
    if k == 'cnn':
        s, b = c['size'], c['batch']
        first = 2 * b * (s - 2) ** 2 * c['c1'] * 9
        return (first + 2 * b * (s - 4) ** 2 * c['c1'] * c['c2'] * 9
                + 2 * b * c['hidden'] * (c['c2'] * ((s - 4) // 2) ** 2 + 10)), first
    if k == 'conv':
        s, half = c['size'], (c['size'] + 1) // 2
        first = 2 * c['batch'] * s * s * c['c1'] * c['c2'] * 9
        return first + 2 * c['batch'] * half * half * c['c2'] ** 2 * 9, first
    if k in ('nerf', 'render'):
        e, w = 3 + 6 * configs.N_FREQS, c['width']
        return 2 * c['points'] * (2 * e * w + (c['depth'] - 1) * w * w + 4 * w), 2 * c['points'] * e * w
    if k in ('transformer', 'logits', 'attention'):
        rows, d = c['batch'] * c['seq'], c['dim']
        layer = 2 * rows * 4 * d * d + 2 * rows * (c['seq'] + 1) * d      # causal half of QK^T and PV
        if k == 'attention':
            return layer, 0
        return c['layers'] * (layer + 2 * rows * 8 * d * d) + 2 * rows * d * c['vocab'], 0
    if k == 'feed_forward':
        return 4 * c['rows'] * c['dim'] * c['hidden'], 0
    return 2 * c['rows'] * c['dim'] * c['vocab'], 0


def work(case):
    model, fn, inputs, opt = _program(case)
    given = sum(4 * int(np.prod([case['points'] if d is None else d for d in (s['shape'] if isinstance(s, dict) else s)]))
                for s in inputs.values())
    sizes = []

    def of(m):
        for x in (vars(m).values() if isinstance(m, Module) else m if isinstance(m, list) else ()):
            if isinstance(x, (Module, list)):
                of(x)
            elif hasattr(x, 'init_fn'):
                sizes.append(int(np.prod(x.shape)))
    of(model)
    flops, first = _flops(case)
    if opt is None:
        out = case['points'] * 4 if case['kind'] == 'render' else case['batch'] * case['seq'] * case['vocab']
        return {'bytes': given + 4 * sum(sizes) + 4 * out, 'flops': flops}
    # weights and optimizer state read and written by each update, and the weights read back once
    each = (16 if opt['kind'] == 'sgd' else 24) * sum(sizes)
    return {'bytes': case['steps'] * (given + each) + 4 * sum(sizes), 'flops': case['steps'] * (3 * flops - first)}


def tolerance(case):
    # Every value is held and summed in 32 bits: against 64 bits most cases are 1e-7 to 5e-7 off. With ReLU an input
    # within rounding of zero can fall on either side of it and move one position's whole gradient, which the weights
    # of a later step carry on (up to 1e-6 off, single weights 4e-5).
    if case['kind'] in ('cnn', 'conv', 'nerf', 'sin_mlp'):
        return {'rel': 4e-6, 'max': 2e-4}
    return {'rel': 2e-6, 'max': 2e-5}


# ---- the same in 64 bits ------------------------------------------------------------------------

def _erf(x):
    """The IR defines erf by formula 7.1.26 of Abramowitz and Stegun."""
    t = 1 / (1 + 0.3275911 * x.abs())
    poly = ((((1.061405429 * t - 1.453152027) * t + 1.421413741) * t - 0.284496736) * t + 0.254829592) * t
    return torch.sign(x) * (1 - poly * torch.exp(-x * x))


class _Erf(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        ctx.save_for_backward(x)
        return _erf(x)

    @staticmethod
    def backward(ctx, g):
        x, = ctx.saved_tensors
        return g * 2 / math.sqrt(math.pi) * torch.exp(-x * x)


def _drop(x, p, seed, salt):
    """The IR's dropout mask: a PCG hash of the seed, the op's salt and the flat index, its products rounded to
    double before they wrap."""
    if not p:
        return x
    wrap = 0xFFFFFFFF
    h = torch.arange(x.numel(), device=x.device, dtype=torch.int64) ^ (seed ^ ((salt * 0x9E3779B1) & wrap))
    h = (h.double() * 747796405.0 + 2891336453.0).long() & wrap
    h = ((h ^ (h >> ((h >> 28) + 4))).double() * 277803737.0).long() & wrap
    h = h ^ (h >> 22)
    return x * ((h.double() / 2.0 ** 32 >= p).double() / (1 - p)).reshape(x.shape)


def _linear(w, name, x):
    y = x @ w[name + '.W']
    return y + w[name + '.b'] if name + '.b' in w else y


def _norm(w, name, x):
    c = x - x.mean(-1, keepdim=True)
    return c / torch.sqrt((c * c).mean(-1, keepdim=True) + 1e-5) * w[name + '.g'] + w[name + '.b']


def _conv(w, name, x, stride=1, pad=0):
    k = w[name + '.W']
    b, s = x.shape[0], (x.shape[2] + 2 * pad - 3) // stride + 1
    cols = torch.nn.functional.unfold(x, 3, padding=pad, stride=stride)
    y = (k.reshape(1, k.shape[0], -1).expand(b, -1, -1).contiguous() @ cols.contiguous()).reshape(b, -1, s, s)
    return y + w[name + '.b'].reshape(1, -1, 1, 1)


def _attend(w, name, x, heads, p, seed, salt):
    b, t, d = x.shape
    q, k, v = (_linear(w, name + '.' + n, x).reshape(b, t, heads, d // heads).transpose(1, 2).contiguous() for n in 'qkv')
    s = q @ k.transpose(-1, -2).contiguous() / math.sqrt(d // heads)
    ahead = torch.ones(t, t, dtype=torch.bool, device=x.device).triu(1)
    a = _drop(torch.softmax(s.masked_fill(ahead, -math.inf), -1), p, seed, salt)
    return _drop(_linear(w, name + '.o', (a @ v).transpose(1, 2).reshape(b, t, d)), p, seed, salt + 1)


def _mlp(w, name, x):
    h = _linear(w, name + '.up', x)
    return _linear(w, name + '.down', 0.5 * h * (1 + _Erf.apply(h / math.sqrt(2))))


def _forward64(c, w, inp, seed):
    """The loss (or, for inference, the output) of a case for weights `w` and one batch."""
    k, relu = c['kind'], torch.relu
    entropy = torch.nn.functional.cross_entropy
    if k == 'sin_mlp':
        y = _linear(w, 'l3', relu(_linear(w, 'l2', relu(_linear(w, 'l1', inp['x'])))))
        return ((y - inp['y']) ** 2).mean()
    if k == 'char_mlp':
        h = torch.tanh(_linear(w, 'l1', w['emb.W'][inp['tokens']].reshape(c['batch'], -1)))
        return entropy(_linear(w, 'l2', h), inp['targets'])
    if k == 'cnn':
        h = relu(_conv(w, 'conv2', relu(_conv(w, 'conv1', inp['x']))))
        h = torch.nn.functional.max_pool2d(h, 2).reshape(c['batch'], -1)
        return entropy(_linear(w, 'fc2', relu(_linear(w, 'fc1', h))), inp['y'])
    if k == 'conv':
        return ((_conv(w, 'half', relu(_conv(w, 'same', inp['x'], 1, 1)), 2, 1) - inp['target']) ** 2).mean()
    if k in ('nerf', 'render'):
        x = inp['x']
        at = (x.unsqueeze(-1) * inp['freqs'].reshape(1, 1, -1)).float().double()     # the angle is held in 32 bits
        pe = torch.cat([x, torch.sin(at).reshape(len(x), -1), torch.cos(at).reshape(len(x), -1)], 1)
        h = pe
        for i in range(c['depth']):
            h = relu(_linear(w, 'layers.%d' % i, torch.cat([h, pe], 1) if i == c['depth'] // 2 else h))
        y = _linear(w, 'head', h)
        return y if k == 'render' else ((y - inp['target']) ** 2).mean()
    if k in ('transformer', 'logits'):
        p = c.get('drop', 0.0)
        x = w['tok_emb'][inp['tokens']] + w['pos_emb']
        for i in range(c['layers']):
            n = 'layers.%d.' % i
            x = x + _attend(w, n + 'attn', _norm(w, n + 'ln1', x), c['heads'], p, seed, 3 * i)
            x = x + _drop(_mlp(w, n + 'mlp', _norm(w, n + 'ln2', x)), p, seed, 3 * i + 2)
        y = _linear(w, 'head', _norm(w, 'lnf', x))
        return y if k == 'logits' else entropy(y.reshape(-1, c['vocab']), inp['targets'].reshape(-1))
    x = inp.get('x')
    if k == 'attention':
        y = _attend(w, 'attn', _norm(w, 'ln1', x), c['heads'], c['drop'], seed, 0)
        return ((x + y - inp['target']) ** 2).mean()
    if k == 'feed_forward':
        y = _drop(_mlp(w, 'mlp', _norm(w, 'ln2', x)), c['drop'], seed, 0)
        return ((x + y - inp['target']) ** 2).mean()
    return entropy(_linear(w, 'head', _norm(w, 'lnf', w['emb.W'][inp['tokens']])), inp['targets'])


def exact(case, seed):
    (_, _, _, opt), ir, batches, p, v = _given(case, seed)
    dev = 'cuda' if torch.cuda.is_available() else 'cpu'
    up = lambda a: torch.from_numpy(a).to(dev)  # noqa: E731
    shapes = ir.param_shapes()
    w = {n: up(a).double().reshape(shapes[n]) for n, a in p.items()}
    batches = [{n: up(a).double() if a.dtype == np.float32 else up(a).long() for n, a in b.items()} for b in batches]
    if opt is None:
        with torch.no_grad():
            return _forward64(case, w, batches[0], 0).cpu().numpy()
    m = {n: torch.zeros_like(a) for n, a in w.items()}
    v = {n: up(a).double().reshape(shapes[n]) for n, a in v.items()}
    losses = []
    for i in range(case['steps']):
        t = RESUMED_AT + 1 + i
        for a in w.values():
            a.requires_grad_(True)
        loss = _forward64(case, w, batches[i % len(batches)], t)
        g = dict(zip(w, torch.autograd.grad(loss, list(w.values()))))
        losses.append(float(loss.detach()))
        with torch.no_grad():
            if opt.get('clipGradNorm'):
                norm = torch.sqrt(sum((a * a).sum() for a in g.values()))
                scale = min(1.0, opt['clipGradNorm'] / (float(norm) + 1e-6))
                g = {n: a * scale for n, a in g.items()}
            for n in w:
                if opt['kind'] == 'sgd':
                    m[n] = opt['momentum'] * m[n] + g[n]
                    w[n] = w[n].detach() - opt['lr'] * m[n]
                    continue
                m[n] = 0.9 * m[n] + 0.1 * g[n]
                v[n] = 0.999 * v[n] + 0.001 * g[n] * g[n]
                # weights decay, biases and norms (whose initial values are constants) do not
                keep = 1 - opt['lr'] * opt.get('weightDecay', 0.0) * (n.rsplit('.', 1)[-1] not in ('b', 'g'))
                rate = opt['lr'] * math.sqrt(1 - 0.999 ** t) / (1 - 0.9 ** t)
                w[n] = keep * w[n].detach() - rate * m[n] / (torch.sqrt(v[n]) + 1e-8)
    return {'losses': np.array(losses), 'weights': {n: a.detach().reshape(-1).cpu().numpy() for n, a in w.items()}}
