"""What a user of this package has it do, as measurable cases.

Serving: a mixture-of-experts layer of compressed experts called with one token
(generation), a few (a small batch), a token for every expert (a full batch) and
thousands (encoding whole sequences), with and without the router and the module
around it, prepared or straight from the packed buffers; and single compressed
matrices called with one token and with whole sequences.  Storing and loading:
compressing a matrix, expanding it again, and preparing a layer from the tensors
of its experts.

Sizes are the three Switch shapes of qmoe_amd.synthetic.SHAPES (wi is
[d_ff, d_model], wo [d_model, d_ff]) and odd ones between them; weights are
ternary with 80 to 95 % zeros (0.9 is usual), or with a share that differs from
row to row.

A case: `kind` names the path (one function below each for what it needs and what
it does), the other entries its sizes and options.
"""
import math

import torch
from torch import nn

from qmoe_amd import sub1, sub1_hip, synthetic

DEVICE = 'cuda:0'


def _layer(kind, name, shape, experts, tokens, route, zeros=0.9, **options):
    d_model, d_ff = synthetic.SHAPES[shape]
    return dict(name=name, kind=kind, d_model=d_model, d_ff=d_ff, experts=experts, tokens=tokens,
                route=route, zeros=zeros, **options)


def _matrix(kind, name, height, width, zeros=0.9, **options):
    return dict(name=name, kind=kind, height=height, width=width, zeros=zeros, **options)


def listed():
    return [
        # generation, batch 1: one token through one expert of a layer
        _layer('experts', 'one_token_c2048', 'c2048', 64, 1, 'router'),
        # a small, odd batch of requests that generate together
        _layer('experts', 'few_tokens_large', 'large', 128, 13, 'router'),
        # a Switch block's sparse MLP as a model calls it: router, experts, scaling, on
        # one short sequence
        _layer('block', 'switch_block_base', 'base', 128, 64, 'router', dtype='bf16'),
        # a full batch: every expert of a slice of the largest layer gets a token, so
        # that 1.2 GB of weights pass through once
        _layer('experts', 'full_batch_c2048', 'c2048', 512, 512, 'each'),
        # encoding eight sequences of 512 tokens: 32 tokens an expert on average
        _layer('experts', 'encode_base', 'base', 128, 4096, 'router'),
        # a layer served from the packed buffers, no prepared copy in memory; weights as
        # uneven as a quantiser leaves them
        _layer('packed', 'packed_large', 'large', 64, 61, 'router', zeros='rows'),
        # the operator itself: one product with one matrix
        _matrix('matvec', 'matvec_c2048_wo', 2080, 6144),
        # one compressed layer on a sequence of the length the projections are timed with
        _matrix('linear', 'linear_sequence_large_wi', 4096, 1024, tokens=568),
        # and on a long one, the largest matrix
        _matrix('linear', 'linear_long_c2048_wi', 6144, 2080, tokens=2272),
        # compressing a ternarised matrix
        _matrix('compress', 'compress_c2048_wi', 6144, 2080),
        # expanding a compressed matrix to symbols and weights; a ragged one
        _matrix('expand', 'expand_ragged', 3001, 1023, zeros=0.88),
        # loading: a layer taken from its experts' tensors, up to its first batch
        _layer('load', 'load_base', 'base', 128, 256, 'router'),
    ]


def draw(rng):
    def log(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    kind = rng.choice(['experts', 'experts', 'experts', 'block', 'packed', 'matvec', 'linear', 'linear',
                       'compress', 'expand', 'load'])
    zeros = rng.choice([0.8, 0.85, 0.88, 0.9, 0.9, 0.95, 'rows'])
    if rng.random() < 0.5:
        d_model, d_ff = synthetic.SHAPES[rng.choice(sorted(synthetic.SHAPES))]
    else:
        d_model, d_ff = rng.randint(500, 2080), rng.randint(2000, 6144)
    if kind in ('matvec', 'linear', 'compress', 'expand'):
        height, width = rng.choice([(d_ff, d_model), (d_model, d_ff)])
        case = dict(kind=kind, height=height, width=width, zeros=zeros)
        if kind == 'linear':
            case['tokens'] = log(2, 2272)
        return case
    # a slice of a layer: at most the weights of 128 large experts in memory, and at most
    # the work of 4096 tokens through base experts (a quarter of it from packed buffers)
    weights = 2 * d_model * d_ff
    experts = rng.randint(8, max(8, min(128, 2 ** 30 // weights)))
    most = 4096 * 2 * 768 * 3072 // weights
    tokens = log(1, {'experts': most, 'block': min(most, 1024), 'packed': most // 16, 'load': 256}[kind])
    case = dict(kind=kind, d_model=d_model, d_ff=d_ff, experts=experts, tokens=tokens,
                route=rng.choice(['router', 'router', 'each']), zeros=zeros)
    if kind == 'block':
        case['route'] = 'router'
        case['dtype'] = rng.choice(['bf16', 'fp32'])
    return case


# ------------------------------------------------------------- preparing ---

class Top1Router(nn.Module):
    """A Switch router as models have it: fp32 softmax over a linear classifier,
    the best expert of each token, at most `capacity` tokens of a sequence to an
    expert.  Returns (mask, probabilities, logits)."""

    def __init__(self, d_model, experts, capacity, generator):
        super().__init__()
        weight = torch.randn((experts, d_model), generator=generator, device=DEVICE)
        self.classifier = nn.Parameter(weight / d_model ** 0.5, requires_grad=False)
        self.capacity = capacity

    def forward(self, hidden):
        logits = nn.functional.linear(hidden.float(), self.classifier)
        probs, index = torch.softmax(logits, dim=-1).max(dim=-1, keepdim=True)
        mask = torch.zeros(logits.shape, dtype=torch.int64, device=logits.device)
        mask.scatter_(-1, index, 1)
        mask = mask * (torch.cumsum(mask, dim=-2) <= self.capacity)
        return mask, probs.to(hidden.dtype), logits


class Expert(nn.Module):
    def __init__(self, wi, wo):
        super().__init__()
        self.wi, self.wo = wi, wo


class SparseMLP(nn.Module):
    def __init__(self, router, experts):
        super().__init__()
        self.router = router
        self.experts = nn.ModuleDict({'expert_%d' % i: e for i, e in enumerate(experts)})


def _zeros(case):
    return synthetic.ROWS if case['zeros'] == 'rows' else case['zeros']


def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _linear(w_comp, row_off, ter_minmax):
    """A Sub1Linear holding these buffers, as a checkpoint is loaded into one."""
    linear = sub1.Sub1Linear(row_off.numel() - 1, w_comp.numel())
    linear.w_comp, linear.row_off, linear.ter_minmax = w_comp, row_off, ter_minmax
    return linear


def _stack(case, seed):
    return synthetic.build_stack(case['experts'], case['d_model'], case['d_ff'], _zeros(case), seed)


def _layers(case, seed):
    """(wi, wo) as lists of one Sub1Linear per expert."""
    stack = _stack(case, seed)
    pairs = [[_linear(*t) for t in synthetic.expert_layers(stack, e)] for e in range(case['experts'])]
    return [p[0] for p in pairs], [p[1] for p in pairs]


def _tokens(case, seed):
    x = synthetic.activations(case['tokens'], case['d_model'], seed)
    if case['route'] == 'each':
        route = torch.arange(case['tokens'], dtype=torch.int32, device=DEVICE) % case['experts']
    else:
        route = synthetic.softmax_router(case['tokens'], case['experts'], seed + 1)
    return x, route


def _dense(case, seed):
    """bf16 [height, width] with ternary rows."""
    g = _generator(seed)
    symbols = synthetic.draw_symbols(case['height'], case['width'], _zeros(case), g, DEVICE)
    values = synthetic.draw_minmax(case['height'], g, DEVICE).view(-1, 2)
    values = torch.cat((torch.zeros_like(values[:, :1]), values), dim=1)       # 0, min, max
    return torch.gather(values, 1, symbols.to(torch.int64))


def prepare(case, seed):
    kind = case['kind']
    seed = 1000 * seed
    if kind == 'experts':
        layer = sub1.Sub1Experts(*_layers(case, seed))
        x, route = _tokens(case, seed + 1)
        layer(x[:1], route[:1])             # the stream is made on first use: a server does that at start
        return dict(layer=layer, x=x, route=route)
    if kind == 'block':
        wi, wo = _layers(case, seed)
        router = Top1Router(case['d_model'], case['experts'],
                            capacity=max(2, 2 * case['tokens'] // case['experts']), generator=_generator(seed + 1))
        block = sub1.FasterMLP(SparseMLP(router, [Expert(*p) for p in zip(wi, wo)]))
        hidden = synthetic.activations(case['tokens'], case['d_model'], seed + 2)[None]
        hidden = hidden.to(torch.float32 if case['dtype'] == 'fp32' else torch.bfloat16)
        block(hidden[:, :1])
        return dict(block=block, hidden=hidden)
    if kind == 'packed':
        x, route = _tokens(case, seed + 1)
        return dict(stack=_stack(case, seed), x=x, route=route)
    if kind == 'load':
        wi, wo = _layers(case, seed)
        x, route = _tokens(case, seed + 1)
        return dict(wi=wi, wo=wo, x=x, route=route)
    w = _dense(case, seed)
    if kind == 'compress':
        # where a compressor collects the codes of its matrices: as many as they can be
        store = torch.zeros(case['height'] * ((case['width'] + 1) // 2), dtype=torch.int16, device=DEVICE)
        return dict(w=w, store=store)
    linear = sub1.Sub1Linear.make(w)
    if kind == 'matvec':
        return dict(linear=linear, x=synthetic.activations(1, case['width'], seed + 1)[0])
    if kind == 'linear':
        x = synthetic.activations(case['tokens'], case['width'], seed + 1)
        linear(x)                           # its own form of the weights is made on first use
        return dict(linear=linear, x=x)
    return dict(linear=linear, width=case['width'])     # expand


# --------------------------------------------------------------- running ---

def run(state):
    with torch.no_grad():
        if 'layer' in state:
            return state['layer'](state['x'], state['route'])
        if 'block' in state:
            hidden, (logits, index) = state['block'](state['hidden'])
            return hidden, logits, index
        if 'stack' in state:
            return state['stack'].forward(state['x'], state['route'])
        if 'wi' in state:
            return sub1.Sub1Experts(state['wi'], state['wo'])(state['x'], state['route'])
        if 'w' in state:
            linear = sub1.Sub1Linear.make(state['w'])
            state['store'][:linear.w_comp.numel()] = linear.w_comp
            return state['store'], linear.row_off, linear.ter_minmax
        linear = state['linear']
        buffers = (sub1.DEC[0], linear.w_comp, linear.row_off, linear.ter_minmax)
        if 'width' in state:
            return sub1_hip.sub1decode(*buffers, state['width'])
        if state['x'].dim() == 2:
            return linear(state['x'])
        y = torch.zeros(linear.row_off.numel() - 1, dtype=torch.bfloat16, device=DEVICE)
        sub1_hip.sub1matvec(*buffers, state['x'], y)
        return y


# --------------------------------------------- what it needs, and accuracy ---

def _code_bytes(weights, zeros):
    """Bytes of the dictionary codes of that many weights: 1.2 times their entropy
    (measured 0.69 bit a weight at 90 % zeros)."""
    p = 0.865 if zeros == 'rows' else zeros
    entropy = -p * math.log2(p) - (1 - p) * math.log2((1 - p) / 2)
    return 1.2 * entropy * weights / 8


def _stored(height, width, zeros):
    """Bytes of one compressed matrix: codes, row offsets, (min, max) pairs."""
    return _code_bytes(height * width, zeros) + 4 * (height + 1) + 4 * height


def work(case):
    kind, zeros = case['kind'], case['zeros']
    if kind in ('experts', 'block', 'packed', 'load'):
        d_model, d_ff, experts, tokens = case['d_model'], case['d_ff'], case['experts'], case['tokens']
        expert = _stored(d_ff, d_model, zeros) + _stored(d_model, d_ff, zeros)
        # the experts that some token goes to, on average, are read once each
        hit = min(tokens, experts) if case['route'] == 'each' else experts * (1 - (1 - 1 / experts) ** tokens)
        read = experts if kind == 'load' else hit
        amount = dict(bytes=expert * read + tokens * (4 * d_model + 4), flops=4 * tokens * d_model * d_ff)
        if kind == 'load':                  # the prepared form is written and read once more
            amount['bytes'] += 2 * expert * experts
        if kind == 'block':
            amount['bytes'] += 4 * experts * d_model + tokens * (4 * experts + 8)
            amount['flops'] += 2 * tokens * experts * d_model
        return amount
    height, width = case['height'], case['width']
    stored = _stored(height, width, zeros)
    if kind == 'compress':
        return dict(bytes=2 * height * width + stored, flops=0)
    if kind == 'expand':
        return dict(bytes=stored + 3 * height * width, flops=0)
    tokens = case.get('tokens', 1)
    return dict(bytes=stored + 2 * tokens * (width + height), flops=2 * tokens * height * width)


def tolerance(case):
    # codes, offsets, symbols and weights are whole numbers or copies: no freedom
    if case['kind'] in ('compress', 'expand'):
        return 'exact'
    # bf16 results of fp32 sums in some order (and of h, rounded to bf16 between wi and
    # wo): an element off by a place of bf16 here and there.  Measured between the
    # orders of the packed and the prepared kernels: up to 4.5e-5, one place at most
    # (2^-7); against sums in float64, rounded the same way, up to 2.1e-5
    return {'rel': 2e-4, 'max': 0.03, 'differ': 0.0}
