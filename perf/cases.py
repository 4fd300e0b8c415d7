"""Workloads whose speed this library answers for, each through the entry
points a serving program calls.

Four kinds of call cover a model step of a G256 checkpoint:

* ``layer``  - the whole MoE layer (router, top-8, routed experts, shared
  expert) through ``native.moe_layer``, N32 banks.
* ``routed`` - the routed experts alone, given top-8 weights and ids, through
  the ``ornith_g256::routed_out`` op: checkpoint (N16) banks, 8-bit
  activations up to 64 tokens and 4-bit ones above, as a server that sets
  ``routed_prefill_activation_bits`` runs them.
* ``dense``  - G256 linears through ``ornith_g256::dense_out``: the exact
  8-bit path up to ``a8_max_rows`` rows, the bf16 GEMM above.
* ``w8_head`` / ``g256_head`` - the LM heads with the greedy hand-off.

Steps of at most 2048 rows are captured once and replayed, as a serving loop
replays its captured decode steps and full prefill chunks; longer prefills are
launched eagerly.  Small steps run through several layers with weights of
their own, as a model does, so the memory-side cache cannot serve repeats.
Weights, router biases and activations follow the distributions of bench.py.
"""
import functools
import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / 'ornith-ciru-halo-agent_amd'))
from ornith_g256 import native, synthetic, tables  # noqa: E402

E, TOP, H, I, G = 256, 8, 2048, 512, 256
EXPERT_BYTES = 3 * H * I // 2 + 4 * 3 * H * I // G
CAPACITY = 8192                  # max_num_batched_tokens of the served configuration
CAPTURED_ROWS = 2048
G256_VOCAB = 151936
DENSE_SHAPES = ((6144, 2048), (12288, 2048), (2048, 4096), (1024, 2048), (2048, 512))
SETTINGS = {'routed_prefill_activation_bits': 4}


def listed():
    return [
        # one user decoding: every layer streams nine experts for one token
        dict(name='layer_1', kind='layer', rows=1, zipf=0.0, layers=40),
        # eight requests with four draft positions each
        dict(name='layer_32', kind='layer', rows=32, zipf=0.0, layers=40),
        # a ragged mixed batch: short prompts beside decode rows
        dict(name='layer_131', kind='layer', rows=131, zipf=0.0, layers=1),
        # the usual prefill chunk, and the largest batch a server admits, with skewed experts
        dict(name='layer_1120', kind='layer', rows=1120, zipf=1.1, layers=1),
        dict(name='layer_8192', kind='layer', rows=8192, zipf=1.3, layers=1),
        # a long prefill chunk with 4-bit activations on the checkpoint's own banks
        dict(name='routed_a4_4480', kind='routed', rows=4480, zipf=1.1, layers=1),
        # attention / linear-attention projections of a decode step, one user and a full batch
        dict(name='dense_1', kind='dense', rows=1, n=6144, k=2048, a8_max_rows=32, layers=40),
        dict(name='dense_32', kind='dense', rows=32, n=6144, k=2048, a8_max_rows=32, layers=40),
        # the same projections of a prefill chunk
        dict(name='dense_1120', kind='dense', rows=1120, n=6144, k=2048, a8_max_rows=32, layers=8),
        # next-token logits: one user, a full batch, and the 4-bit head
        dict(name='w8_head_1', kind='w8_head', rows=1),
        dict(name='w8_head_32', kind='w8_head', rows=32),
        dict(name='g256_head_32', kind='g256_head', rows=32),
    ]


def _spread(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(('layer', 'layer', 'layer', 'layer', 'layer', 'routed', 'dense', 'dense', 'dense', 'w8_head',
                       'w8_head', 'g256_head'))
    if kind in ('layer', 'routed'):
        rows = _spread(rng, 1, 8192)
        zipf = round(rng.uniform(0.8, 1.4), 2) if rows > 64 and rng.random() < 0.7 else 0.0
        return dict(kind=kind, rows=rows, zipf=zipf, layers=_decode_layers(rows))
    if kind == 'dense':
        rows = _spread(rng, 1, 8192)
        n, k = rng.choice(DENSE_SHAPES)
        return dict(kind=kind, rows=rows, n=n, k=k, a8_max_rows=rng.choice((32, 64)),
                    layers=40 if rows <= 8 else 16 if rows <= 64 else 8 if rows <= CAPTURED_ROWS else 1)
    return dict(kind=kind, rows=_spread(rng, 1, 64))


def _decode_layers(rows):
    return 40 if rows <= 4 else 10 if rows <= 64 else 1


# ---------------------------------------------------------------------------
# Inputs and weights
# ---------------------------------------------------------------------------
def _device():
    return torch.device('cuda', torch.cuda.current_device())


def _rows(case, seed, dev, k=H):
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed * 1000 + 1)
    return torch.randn((case['rows'], k), generator=gen, device=dev).to(torch.bfloat16)


def _moe_weights(case, seed, dev, layer):
    bias = synthetic.zipf_bias(case['zipf'], seed * 1000 + 7 + layer, dev) if case['zipf'] else None
    return synthetic.moe_layer(seed * 1000 + 100 + layer, dev, bias)


def _n16_weights(case, seed, dev, layer):
    """Routed banks as a checkpoint holds them, with the routing of the rows."""
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed * 1000 + 100 + layer)
    banks = []
    for n, k in ((2 * I, H), (H, I)):
        codes, meta = synthetic.bank(gen, n, k, dev, E)
        banks += [codes.view(E, n // 16, k // G, 32, 16), meta.view(E, n // 16, k // G, 16)]
    logits = torch.randn((case['rows'], E), generator=gen, device=dev) * (0.02 * math.sqrt(H))
    if case['zipf']:
        logits += synthetic.zipf_bias(case['zipf'], seed * 1000 + 7 + layer, dev)
    top = torch.softmax(logits, 1).topk(TOP, 1)
    weights = (top.values / top.values.sum(1, keepdim=True)).contiguous()
    return dict(banks=banks, weights=weights, ids=top.indices.to(torch.int32).contiguous())


def _dense_bank(case, seed, dev, layer):
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed * 1000 + 100 + layer)
    n, k = case['n'], case['k']
    codes, meta = synthetic.bank(gen, n, k, dev)
    return codes.view(n // 16, k // G, 32, 16), meta.view(n // 16, k // G, 16)


def _w8_bank(seed, dev):
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed * 1000 + 100)
    n = native.HEAD_VOCAB
    codes = torch.randint(-127, 128, (n // 16, H // 16, 4, 16, 4), generator=gen, device=dev, dtype=torch.int8)
    scales = torch.empty((n, 16), device=dev).uniform_(2e-4, 1e-3, generator=gen).half()
    return codes.view(torch.int32).view(n // 16, H // 16, 4, 16), scales


def _g256_bank(seed, dev):
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed * 1000 + 100)
    return synthetic.bank(gen, G256_VOCAB, H, dev)


@functools.lru_cache(maxsize=None)
def _shared_tables(dev):
    return tables.load(dev)          # constants of the library, loaded once per process


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def prepare(case, seed):
    dev = _device()
    state = dict(kind=case['kind'], rows=case['rows'], graph=None,
                 flags=torch.zeros(1, dtype=torch.int32, device=dev))
    {'layer': _prepare_layer, 'routed': _prepare_routed, 'dense': _prepare_dense, 'w8_head': _prepare_w8,
     'g256_head': _prepare_g256}[case['kind']](case, seed, dev, state)
    if case['rows'] <= CAPTURED_ROWS:
        side = torch.cuda.Stream(device=dev)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            state['step']()              # the first call outside the capture
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            state['step']()
        state['graph'] = graph
    return state


def run(state):
    if state['graph'] is not None:
        state['graph'].replay()
    else:
        state['step']()
    return dict(state['outputs'], flags=state['flags'])


def _prepare_layer(case, seed, dev, state):
    T, L = case['rows'], case['layers']
    x = _rows(case, seed, dev)
    layers = [_moe_weights(case, seed, dev, i) for i in range(L)]
    silu, sigmoid = _shared_tables(dev)
    workspace = torch.zeros(native.routed_layout(CAPACITY, 'layer').workspace_bytes, dtype=torch.uint8, device=dev)
    out = torch.empty((L, T, H), dtype=torch.bfloat16, device=dev)
    weights = torch.empty((L, T, TOP), dtype=torch.float32, device=dev)
    ids = torch.empty((L, T, TOP), dtype=torch.int32, device=dev)
    gate_logit = torch.empty((L, T), dtype=torch.bfloat16, device=dev)

    def step():
        for i, w in enumerate(layers):
            native.moe_layer(x, w['router'], w['bias'], w['gate'], *w['w13'], *w['w2'], *w['s13'], *w['s2'], silu,
                             sigmoid, workspace, weights[i], ids[i], gate_logit[i], out[i], state['flags'], CAPACITY)
    state.update(step=step, outputs=dict(out=out, weights=weights, ids=ids))


def _prepare_routed(case, seed, dev, state):
    T, L = case['rows'], case['layers']
    x = _rows(case, seed, dev)
    layers = [_n16_weights(case, seed, dev, i) for i in range(L)]
    workspace = torch.empty(native.configure(SETTINGS, CAPACITY, DENSE_SHAPES), dtype=torch.uint8, device=dev)
    out = torch.empty((L, T, H), dtype=torch.bfloat16, device=dev)

    def step():
        for i, w in enumerate(layers):
            native.routed_out(x, w['weights'], w['ids'], *w['banks'], workspace, out[i], state['flags'], CAPACITY)
    state.update(step=step, outputs=dict(out=out))


def _prepare_dense(case, seed, dev, state):
    M, L, n, k = case['rows'], case['layers'], case['n'], case['k']
    x = _rows(case, seed, dev, k)
    banks = [_dense_bank(case, seed, dev, i) for i in range(L)]
    workspace = torch.empty(native.configure(SETTINGS, CAPACITY, DENSE_SHAPES), dtype=torch.uint8, device=dev)
    out = torch.empty((L, M, n), dtype=torch.bfloat16, device=dev)

    def step():
        for i, (codes, meta) in enumerate(banks):
            native.dense_out(x, codes, meta, workspace, out[i], state['flags'], CAPACITY, n, k, 2,
                             case['a8_max_rows'])
    state.update(step=step, outputs=dict(out=out))


def _prepare_w8(case, seed, dev, state):
    M = case['rows']
    x = _rows(case, seed, dev)
    codes, scales = _w8_bank(seed, dev)
    workspace = torch.empty(native.configure(SETTINGS, CAPACITY, DENSE_SHAPES), dtype=torch.uint8, device=dev)
    logits = torch.empty((M, native.HEAD_VOCAB), dtype=torch.bfloat16, device=dev)
    tokens = torch.empty((M,), dtype=torch.int64, device=dev)

    def step():
        native.head_out(x, codes, scales, workspace, logits, state['flags'], 2)
        native.logits_argmax(logits, tokens)
    state.update(step=step, outputs=dict(logits=logits, tokens=tokens))


def _prepare_g256(case, seed, dev, state):
    M = case['rows']
    x = _rows(case, seed, dev)
    codes, meta = _g256_bank(seed, dev)
    workspace = torch.empty(native.lib().ornith_dense_g256_head_workspace_bytes(64, G256_VOCAB), dtype=torch.uint8,
                            device=dev)
    logits = torch.empty((M, G256_VOCAB), dtype=torch.float32, device=dev)
    tokens = torch.empty((M,), dtype=torch.int64, device=dev)

    def step():
        native.dense_head(x, codes, meta, workspace, logits, None, tokens, state['flags'], 64)
    state.update(step=step, outputs=dict(logits=logits, tokens=tokens))


# ---------------------------------------------------------------------------
# Compulsory work
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _experts_touched(rows, zipf):
    """Distinct experts of `rows` tokens whose logits are normal with the
    router's spread plus the popularity bias (one seeded sample)."""
    gen = torch.Generator()
    gen.manual_seed(5)
    logits = torch.randn((rows, E), generator=gen) * (0.02 * math.sqrt(H))
    logits -= zipf * torch.log(torch.arange(1, E + 1, dtype=torch.float32))
    return int(logits.topk(TOP, 1).indices.unique().numel())


def work(case):
    M, L = case['rows'], case.get('layers', 1)
    if case['kind'] in ('layer', 'routed'):
        banks = _experts_touched(M, case['zipf'])
        nbytes = banks * EXPERT_BYTES + M * (4 * H + 8 * TOP)       # rows in and out, routing in or out
        flops = 2 * M * TOP * 3 * H * I
        if case['kind'] == 'layer':                                 # the shared expert, the router and its gate row
            nbytes += EXPERT_BYTES + (E + 1) * H * 2
            flops += 2 * M * (3 * H * I + (E + 1) * H)
        return dict(bytes=L * nbytes, flops=L * flops)
    if case['kind'] == 'dense':
        n, k = case['n'], case['k']
        return dict(bytes=L * (n * k // 2 + 4 * n * k // G + 2 * M * (n + k)), flops=L * 2 * M * n * k)
    if case['kind'] == 'w8_head':
        n = native.HEAD_VOCAB
        return dict(bytes=n * (H + 32) + M * (2 * H + 2 * n + 8), flops=2 * M * n * H)
    n = G256_VOCAB
    return dict(bytes=n * (H // 2 + 4 * H // G) + M * (2 * H + 4 * n + 8), flops=2 * M * n * H)


def tolerance(case):
    """Outputs are bf16 except the 4-bit head's fp32 logits.  A sum in another
    order moves single activations to the neighbouring code (8-bit: 1/127 of a
    group's largest value, 4-bit: 1/7), single bf16 results to the neighbour,
    and near-equal router logits or logit maxima to the other choice."""
    kind = case['kind']
    if kind == 'layer':
        return dict(rel=0.01, max=0.5, differ=0.002)
    if kind == 'routed':
        return dict(rel=0.01, max=0.5)
    if kind == 'dense':
        return dict(rel=0.007, max=0.1)
    if kind == 'w8_head':
        return dict(rel=0.007, max=0.1, differ=0.01)
    return dict(rel=0.0005, max=0.02, differ=0.01)


# ---------------------------------------------------------------------------
# The same calls in 64 bits
# ---------------------------------------------------------------------------
def _h128(x):
    """Orthonormal 128-point Hadamard transform of each 128 columns."""
    h = torch.ones((1, 1), dtype=torch.float64, device=x.device)
    while h.shape[0] < 128:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return (x.reshape(-1, 128) @ (h / math.sqrt(128.0))).reshape(x.shape)


def _quantised(x, qmax=127, group=G):
    """x on the activation grid of the format: per group, an fp16 step of
    absmax / qmax and whole multiples of it."""
    v = x.reshape(x.shape[0], -1, group)
    absmax = v.abs().amax(2, keepdim=True)
    step = (absmax / qmax).clamp_min(2.0 ** -14).half().double()
    q = torch.round(v / step).clamp(-qmax, qmax)
    return torch.where(absmax == 0, 0.0, q * step).reshape(x.shape)


def _weights64(codes, meta):
    """[N/t, K/256, 32, t] code words and [N/t, K/256, t] metadata -> [N, K]."""
    nt, groups, _, tile = codes.shape
    shifts = torch.arange(0, 32, 4, device=codes.device, dtype=torch.int32)
    c = (codes.permute(0, 3, 1, 2)[..., None] >> shifts) & 15                   # [nt, tile, groups, 32, 8]
    c = c.reshape(nt * tile, groups, G).double()
    half = meta.contiguous().view(torch.float16).view(nt, groups, tile, 2).permute(0, 2, 1, 3).double()
    half = half.reshape(nt * tile, groups, 2)
    return (c * half[..., :1] + half[..., 1:]).reshape(nt * tile, groups * G)


def _expert64(xq, w13, w2, qmax=127):
    y = xq @ _weights64(*w13).T
    middle = torch.nn.functional.silu(y[:, :I]) * y[:, I:]
    return _quantised(_h128(middle), qmax) @ _weights64(*w2).T


def _routed64(xq, weights, ids, w13, w2, qmax=127):
    out = torch.zeros((xq.shape[0], H), dtype=torch.float64, device=xq.device)
    order = ids.flatten().argsort(stable=True)
    counts = torch.bincount(ids.flatten(), minlength=E).cpu().tolist()
    start = 0
    for e, n in enumerate(counts):
        if n:
            routes = order[start:start + n]
            rows = routes // TOP
            y = _expert64(xq[rows], (w13[0][e], w13[1][e]), (w2[0][e], w2[1][e]), qmax)
            out.index_add_(0, rows, y * weights.flatten()[routes][:, None])
            start += n
    return out


def exact(case, seed):
    """The outputs of `run` in 64 bits: the format's own grids (4-bit codes,
    quantised activations) are kept, every other rounding is left out."""
    dev = _device()
    x = _rows(case, seed, dev, case.get('k', H)).double()
    if case['kind'] == 'layer':
        xq, outs, weights = _quantised(_h128(x)), [], []
        for i in range(case['layers']):
            w = _moe_weights(case, seed, dev, i)
            logits = x @ w['router'].double().T
            if w['bias'] is not None:
                logits = logits + w['bias'].double()
            top = torch.softmax(logits, 1).topk(TOP, 1)
            rw = top.values / top.values.sum(1, keepdim=True)
            shared = _expert64(xq, w['s13'], w['s2'])
            gate = torch.sigmoid(x @ w['gate'].double())
            outs.append(_routed64(xq, rw, top.indices, w['w13'], w['w2']) + gate[:, None] * shared)
            weights.append(rw)
        return dict(out=torch.stack(outs), weights=torch.stack(weights), ids=None, flags=None)
    if case['kind'] == 'routed':
        qmax, outs = 7 if case['rows'] > 64 else 127, []
        xq = _quantised(_h128(x), qmax)
        for i in range(case['layers']):
            w = _n16_weights(case, seed, dev, i)
            outs.append(_routed64(xq, w['weights'].double(), w['ids'].long(), w['banks'][:2], w['banks'][2:], qmax))
        return dict(out=torch.stack(outs), flags=None)
    if case['kind'] == 'dense':
        xt = _h128(x)
        if case['rows'] <= case['a8_max_rows']:
            xt = _quantised(xt)
        outs = [xt @ _weights64(*_dense_bank(case, seed, dev, i)).T for i in range(case['layers'])]
        return dict(out=torch.stack(outs), flags=None)
    if case['kind'] == 'w8_head':
        codes, scales = _w8_bank(seed, dev)
        xq = _quantised(_h128(x), group=128)
        parts = []
        for c, s in zip(codes.split(1552), scales.split(1552 * 16)):
            q = c.view(torch.int8).view(-1, H // 16, 4, 16, 4).permute(0, 3, 1, 2, 4).reshape(-1, 16, 128)
            parts.append(xq @ (q.double() * s.double()[..., None]).reshape(-1, H).T)
        return dict(logits=torch.cat(parts, 1), tokens=None, flags=None)
    codes, meta = _g256_bank(seed, dev)
    xq = _quantised(_h128(x))
    parts = [xq @ _weights64(c, m).T for c, m in zip(codes.split(256), meta.split(256))]
    return dict(logits=torch.cat(parts, 1), tokens=None, flags=None)
