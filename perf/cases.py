"""The work that users of this engine have it do, as cases that can be timed.

Each case is one use of the public API (`Model`, `step_batch_greedy` and the
operator entries of `include/qwen_gpu.h`) on a seeded random-init Qwen3-0.6B
pack. `listed()` gives the fixed cases, `draw(rng)` further ones of the same
ranges. The seed of `prepare(case, seed)` chooses every token and value; the
weights are the same for all of them, as in a program that serves one model.

Tokens after the prompt are given, not chosen from the logits: the work of a
decode step does not depend on its token, and a tie between two logits cannot
send two correct runs down different texts.
"""
import importlib.util
import math
import sys
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parents[1]
PACK_DIR = Path('/tmp/qwen_gpu_packs/seed0')  # where tests and bench.py keep the same pack

LAYERS, HIDDEN, FFN, VOCAB = 28, 1024, 3072, 151936
HEADS, KV_HEADS, HEAD_DIM = 16, 8, 128
QKV_ROWS = (HEADS + 2 * KV_HEADS) * HEAD_DIM
CONTEXT = 4096
LAYER_BYTES = 2 * (QKV_ROWS * HIDDEN + HIDDEN * HEADS * HEAD_DIM + 3 * FFN * HIDDEN)
HEAD_BYTES = 2 * VOCAB * HIDDEN
KV_BYTES = LAYERS * 2 * KV_HEADS * HEAD_DIM * 2  # one position, all layers
STATIC_ELEMENTS = 1 << 20  # rows x columns limit of qwen_gpu_op_gemm_static

_loaded = {}


def _package():
    if 'package' not in _loaded:
        directory = ROOT / 'fpga-qwen_amd'
        spec = importlib.util.spec_from_file_location('fpga_qwen_amd', directory / '__init__.py',
                                                      submodule_search_locations=[str(directory)])
        module = importlib.util.module_from_spec(spec)
        sys.modules['fpga_qwen_amd'] = module
        spec.loader.exec_module(module)
        _loaded['package'] = module
        _loaded['library'] = module.load_library()
    return _loaded['package']


def _library():
    _package()
    return _loaded['library']


def _pack():
    return _package().ensure_random_pack(PACK_DIR, seed=0)


def _model():
    """A sequence of its own on the one weight upload of this process."""
    if 'owner' not in _loaded:
        _loaded['owner'] = _package().Model(_pack(), context=16)
    return _loaded['owner'].share(context=CONTEXT)


# ---- the cases ----

def listed():
    return [
        # Greedy decoding at batch 1, the engine's first purpose: right after
        # a short chat prompt, and near the end of the context.
        {'name': 'decode-85', 'kind': 'decode', 'position': 85, 'steps': 16},
        {'name': 'decode-3968', 'kind': 'decode', 'position': 3968, 'steps': 16},
        # Speculative decoding: one drafted token verified with the next one.
        {'name': 'verify-300', 'kind': 'verify', 'position': 300, 'pairs': 8},
        # Several sequences on one GPU, with a common system prompt and without.
        {'name': 'batch-8x2048', 'kind': 'batch', 'sequences': 8, 'prefix': 512, 'position': 2048, 'steps': 16},
        {'name': 'batch-3x300', 'kind': 'batch', 'sequences': 3, 'prefix': 0, 'position': 300, 'steps': 16},
        # Time to first token: the next turn of a chat, then prompts of the
        # lengths the reference benchmark publishes.
        {'name': 'turn-17-at-612', 'kind': 'prefill', 'position': 612, 'rows': 17},
        {'name': 'prefill-85', 'kind': 'prefill', 'position': 0, 'rows': 85},
        {'name': 'prefill-452', 'kind': 'prefill', 'position': 0, 'rows': 452},
        {'name': 'prefill-1024', 'kind': 'prefill', 'position': 0, 'rows': 1024},
        {'name': 'prefill-3968', 'kind': 'prefill', 'position': 0, 'rows': 3968},
        # The blocks of one layer that can be called alone: attention of a
        # long suffix behind a reused 512-token prefix, and a projection of a
        # ragged number of rows (the down projection's shape).
        {'name': 'attention-1531-at-512', 'kind': 'attention', 'position': 512, 'rows': 1531},
        {'name': 'linear-341x1024x3072', 'kind': 'linear', 'rows': 341, 'outputs': 1024, 'inputs': 3072},
    ]


def _spread(rng, low, high):
    """A whole number between low and high, even over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(['decode', 'verify', 'batch', 'prefill', 'prefill', 'prefill', 'attention', 'linear'])
    if kind == 'decode':
        steps = rng.randint(4, 24)
        return {'kind': kind, 'position': _spread(rng, 2, CONTEXT - steps), 'steps': steps}
    if kind == 'verify':
        pairs = rng.randint(2, 12)
        return {'kind': kind, 'position': _spread(rng, 2, CONTEXT - 2 * pairs), 'pairs': pairs}
    if kind == 'batch':
        sequences, steps = rng.randint(1, 8), rng.randint(4, 16)
        position = _spread(rng, 16, 2048)
        prefix = rng.choice([0, 64 * rng.randint(0, position // 64)])
        return {'kind': kind, 'sequences': sequences, 'prefix': prefix, 'position': position, 'steps': steps}
    if kind == 'prefill':
        rows = _spread(rng, 2, 3968)
        position = rng.choice([0, rng.randint(0, 3968 - rows)])
        return {'kind': kind, 'position': position, 'rows': rows}
    if kind == 'attention':
        rows = _spread(rng, 2, 3968)
        return {'kind': kind, 'position': rng.choice([0, rng.randint(0, 3968 - rows)]), 'rows': rows}
    outputs, inputs = rng.choice([(4096, 1024), (1024, 2048), (6144, 1024), (1024, 3072)])
    return {'kind': 'linear', 'rows': _spread(rng, 1, STATIC_ELEMENTS // inputs), 'outputs': outputs, 'inputs': inputs}


# ---- one case: what the caller holds, and one pass ----

def _tokens(seed, count):
    return np.random.default_rng([seed, 17]).integers(0, VOCAB, count).astype(np.int32)


def _after_prompt(case):
    """Tokens a pass consumes behind the prompt, per sequence."""
    return {'decode': case.get('steps'), 'verify': 2 * case.get('pairs', 0), 'prefill': case.get('rows'),
            'batch': case.get('steps')}[case['kind']]


def _sequence_tokens(case, seed):
    """Prompt and pass tokens of every sequence: [sequences, position + pass]."""
    count, prefix = case.get('sequences', 1), case.get('prefix', 0)
    tokens = _tokens(seed, count * (case['position'] + _after_prompt(case))).reshape(count, -1)
    tokens[:, :prefix] = tokens[0, :prefix]
    return tokens


def _attention_inputs(case, seed):
    """Queries and keys of unit RMS (they leave a QK-norm), values as a
    projection of a normalized row gives them."""
    g = torch.Generator(device='cuda').manual_seed(int(seed))
    rows, context = case['rows'], case['position'] + case['rows']
    qkv = torch.randn(rows, QKV_ROWS, device='cuda', generator=g)
    keys = torch.randn(KV_HEADS, context, HEAD_DIM, device='cuda', generator=g).half()
    values = (0.64 * torch.randn(KV_HEADS, context, HEAD_DIM, device='cuda', generator=g)).half()
    return qkv, keys, values


def _linear_inputs(case, seed):
    g = torch.Generator(device='cuda').manual_seed(int(seed))
    a = torch.randn(case['rows'], case['inputs'], device='cuda', generator=g)
    w = (0.02 * torch.randn(case['outputs'], case['inputs'], device='cuda', generator=g)).half()
    return a, w


def prepare(case, seed):
    kind = case['kind']
    if kind == 'attention':
        qkv, keys, values = _attention_inputs(case, seed)
        out = torch.empty(2, case['rows'], HEADS * HEAD_DIM, dtype=torch.float16, device='cuda')
        return {'case': case, 'qkv': qkv, 'keys': keys, 'values': values, 'out': out, 'library': _library()}
    if kind == 'linear':
        a, w = _linear_inputs(case, seed)
        out = torch.empty(case['rows'], case['outputs'], device='cuda')
        return {'case': case, 'a': a, 'w': w, 'out': out, 'library': _library()}
    tokens, position = _sequence_tokens(case, seed), case['position']
    models = [_model() for _ in tokens]
    first = case.get('prefix', 0)
    for i, (model, ids) in enumerate(zip(models, tokens)):
        done = 0
        if i and first:
            model.copy_prefix(models[0], first)
            done = first
        elif first:
            model.prefill(ids[:first])
            done = first
        if position > done:
            model.prefill(ids[done:position])
    given = tokens[:, position:]
    state = {'case': case, 'models': models, 'given': given if kind == 'prefill' else given.T.tolist(),
             'position': position, 'package': _package()}
    return state


def run(state):
    kind = state['case']['kind']
    if kind == 'attention':
        qkv, keys, values, out = state['qkv'], state['keys'], state['values'], state['out']
        stream = torch.cuda.current_stream().cuda_stream
        if state['library'].qwen_gpu_op_attention_prefill(qkv.data_ptr(), keys.data_ptr(), values.data_ptr(),
                                                          out[0].data_ptr(), out[1].data_ptr(), qkv.shape[0],
                                                          state['case']['position'], keys.shape[1], stream):
            raise RuntimeError(state['library'].qwen_gpu_last_error().decode())
        return torch.add(out[0].float(), out[1])  # the result is the sum of the two planes
    if kind == 'linear':
        a, w, out = state['a'], state['w'], state['out']
        stream = torch.cuda.current_stream().cuda_stream
        if state['library'].qwen_gpu_op_gemm_static(a.data_ptr(), w.data_ptr(), out.data_ptr(), a.shape[0],
                                                    w.shape[0], w.shape[1], 0, stream):
            raise RuntimeError(state['library'].qwen_gpu_last_error().decode())
        return out
    models, given = state['models'], state['given']
    for model in models:
        model.truncate(state['position'])
    if kind == 'prefill':
        models[0].prefill(given[0])
        return models[0].logits()
    if kind == 'decode':
        for (token,) in given:
            models[0].step(token)
        return models[0].logits()
    if kind == 'verify':
        for i in range(0, len(given), 2):
            models[0].verify_two_greedy(given[i][0], given[i + 1][0])
            models[0].commit_verified(2)
        return models[0].logits()
    for tokens in given:
        state['package'].step_batch_greedy(models, tokens)
    return [model.logits() for model in models]


# ---- what a pass cannot do without ----

def _scores(position, rows):
    """Query-key pairs of rows queries behind position cached positions."""
    return rows * position + rows * (rows + 1) // 2


def _pass_work(groups):
    """Bytes and FLOPs of passes over the layers that read the weights once
    each: (weight passes, new rows, cached positions read, query-key pairs,
    rows through the head)."""
    passes, rows, cached, pairs, heads, head_passes = groups
    return {'bytes': passes * LAYERS * LAYER_BYTES + head_passes * HEAD_BYTES + (cached + rows) * KV_BYTES
            + rows * 2 * HIDDEN + heads * 4 * VOCAB,
            'flops': rows * LAYERS * LAYER_BYTES + heads * HEAD_BYTES + LAYERS * 4 * HEADS * HEAD_DIM * pairs}


def work(case):
    kind, position = case['kind'], case.get('position', 0)
    if kind == 'attention':
        rows = case['rows']
        return {'bytes': 8 * rows * HEADS * HEAD_DIM + 4 * KV_HEADS * HEAD_DIM * (position + rows),
                'flops': 4 * HEADS * HEAD_DIM * _scores(position, rows)}
    if kind == 'linear':
        m, n, k = case['rows'], case['outputs'], case['inputs']
        return {'bytes': 4 * m * k + 2 * n * k + 4 * m * n, 'flops': 2 * m * n * k}
    if kind == 'prefill':
        rows = case['rows']
        return _pass_work((1, rows, position, _scores(position, rows), 1, 1))
    if kind == 'decode':
        n = case['steps']
        return _pass_work((n, n, _scores(position, n) - n, _scores(position, n), n, n))
    if kind == 'verify':
        n = case['pairs']
        cached = sum(position + 2 * i for i in range(n))
        return _pass_work((n, 2 * n, cached, _scores(position, 2 * n), 2 * n, n))
    n, count, prefix = case['steps'], case['sequences'], case['prefix']
    own = _scores(position, n) - n
    cached = count * own - (count - 1) * n * prefix
    return _pass_work((n, n * count, cached, count * _scores(position, n), n * count, n))


def tolerance(case):
    if case['kind'] == 'attention':
        return {'rel': 4e-6, 'max': 1e-4}  # 6.4e-7 off 64 bits, twice for two sides, times about four
    if case['kind'] == 'linear':
        return {'rel': 3e-6, 'max': 1e-4}  # 5e-7 off 64 bits
    # Cached keys and values are rounded to 16 bits: a sum taken in another
    # order moves some of them by one unit there, and the layers that follow
    # carry that on. Measured 0.6e-4 (long contexts) to 1.5e-4 (short ones)
    # off 64 bits.
    return {'rel': 1e-3, 'max': 1e-2}


# ---- the same results in 64 bits, in plain torch ----

def _weights64():
    """The pack's tensors (64-byte header; '.index': name, type, rows,
    columns, offset, length) in double on the GPU."""
    path = str(_pack())
    blob = np.memmap(path, dtype=np.uint8, mode='r')
    tensors = {}
    for line in Path(path + '.index').read_text().splitlines()[1:]:
        fields = line.split()
        if len(fields) != 6:
            continue
        name, kind, rows, cols, offset, length = fields
        raw = np.array(blob[int(offset):int(offset) + int(length)])
        value = torch.from_numpy(raw.view('<f2' if kind == 'F16' else '<f4')).cuda()
        tensors[name] = value.reshape((int(rows), int(cols)) if kind == 'F16' else (int(rows),))
    return tensors


def _causal64(q, k, v, position):
    """q [rows, heads, 128] behind `position` cached positions, k and v
    [positions, KV heads, 128], all in double."""
    rows = q.shape[0]
    out = torch.empty(rows, HEADS, HEAD_DIM, dtype=torch.float64, device=q.device)
    for head in range(HEADS):
        kh, vh = k[:, head // 2].contiguous(), v[:, head // 2].contiguous()
        for b in range(0, rows, 1024):
            part = q[b:b + 1024, head]
            last = position + torch.arange(b, b + part.shape[0], device=q.device)
            s = part @ kh.T.contiguous() / math.sqrt(HEAD_DIM)
            s.masked_fill_(torch.arange(kh.shape[0], device=q.device)[None] > last[:, None], -math.inf)
            out[b:b + 1024, head] = torch.softmax(s, 1) @ vh
    return out


def _forward64(weights, tokens):
    """Logits of the last position. Cached keys and values are rounded to 16
    bits, as the model's cache holds them."""
    def norm(x, w):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * w.double()

    ids = torch.from_numpy(np.asarray(tokens, np.int64)).cuda()
    n = ids.numel()
    angle = torch.arange(n, device='cuda', dtype=torch.float64)[:, None] / \
        1000000.0 ** (torch.arange(64, device='cuda', dtype=torch.float64) * 2 / HEAD_DIM)
    cos, sin = torch.cos(angle)[:, None], torch.sin(angle)[:, None]

    def rope(x):
        a, b = x[..., :64], x[..., 64:]
        return torch.cat((a * cos - b * sin, b * cos + a * sin), -1)

    embed = weights['model.embed_tokens.weight']
    x = embed[ids].double()
    for layer in range(LAYERS):
        def w(suffix):
            return weights['model.layers.%d.%s.weight' % (layer, suffix)]

        def project(h, suffix):
            return h @ w(suffix).double().T.contiguous()

        h = norm(x, w('input_layernorm'))
        q = rope(norm(project(h, 'self_attn.q_proj').view(n, HEADS, HEAD_DIM), w('self_attn.q_norm')))
        k = rope(norm(project(h, 'self_attn.k_proj').view(n, KV_HEADS, HEAD_DIM), w('self_attn.k_norm')))
        v = project(h, 'self_attn.v_proj').view(n, KV_HEADS, HEAD_DIM)
        a = _causal64(q, k.float().half().double(), v.float().half().double(), 0)
        x = x + project(a.reshape(n, -1), 'self_attn.o_proj')
        h = norm(x, w('post_attention_layernorm'))
        gate = project(h, 'mlp.gate_proj')
        x = x + project(gate * torch.sigmoid(gate) * project(h, 'mlp.up_proj'), 'mlp.down_proj')
    return embed.double() @ norm(x[-1], weights['model.norm.weight'])


def exact(case, seed):
    kind = case['kind']
    if kind == 'attention':
        qkv, keys, values = _attention_inputs(case, seed)
        q = qkv[:, :HEADS * HEAD_DIM].double().view(-1, HEADS, HEAD_DIM)
        out = _causal64(q, keys.double().transpose(0, 1), values.double().transpose(0, 1), case['position'])
        return out.reshape(-1, HEADS * HEAD_DIM)
    if kind == 'linear':
        a, w = _linear_inputs(case, seed)
        return a.double() @ w.double().T.contiguous()
    if 'weights' not in _loaded:
        _loaded['weights'] = _weights64()
    logits = [_forward64(_loaded['weights'], ids) for ids in _sequence_tokens(case, seed)]
    return [x for x in logits] if kind == 'batch' else logits[0]
