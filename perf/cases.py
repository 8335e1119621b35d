'''The calls that stand for how a program uses this framework, for timing and comparison.

Each case is one call (or one request) through a public entry point:

  gdn_chunk      chunk_gated_delta_rule, inference (a program with its own layer around the op)
  gdn_train      the same op forward and backward (a training step's share of one layer)
  gdn_prefill    GatedDeltaAttention over a prompt, with or without a carried cache
  gdn_decode     GatedDeltaAttention, one token per sequence
  chord_prefill  apply_chord_attention over a prompt or a later piece of one
  chord_train    the same op forward and backward
  chord_decode   apply_chord_attention, one or two new tokens over a cached context
  model_prefill  the 172M model over prompts, logits of every position
  model_serve    one request batch of the 172M model: prefill into a fixed-capacity cache,
                 then decode steps through DecodeGraph

Sizes: 12 heads, 3 kv heads, GatedDelta head sizes 64 / 128 and width 768 are the 172M
model's; 4 heads of 64 / 64 over 256 tokens, 2048 and 4096 tokens and 64 decode rows are
the benchmark's configurations; the rest are generic.
'''
import math
import os
import sys

import torch
import torch.nn.functional as F

# the package of the tree that the program runs in
sys.path.insert(0, os.path.join(os.getcwd(), 'codon-motif_amd'))

from motif.block.attention import GatedDeltaAttention  # noqa: E402
from motif.model.cache import GatedDeltaAttentionLayerCache, ModelCache  # noqa: E402
from motif.model.decode_graph import DecodeGraph  # noqa: E402
from motif.model.motif import MotifChordModel  # noqa: E402
from motif.model.presets import config_172m  # noqa: E402
from motif.ops import apply_chord_attention, chunk_gated_delta_rule  # noqa: E402

DEV = 'cuda'
DTYPES = {'bf16': torch.bfloat16, 'fp16': torch.float16, 'fp32': torch.float32}
WIDTH, HEADS, KV_HEADS, DK, DV, CONV, INNER, VOCAB = 768, 12, 3, 64, 128, 4, 2048, 32000
EPS = 1e-6      # norm epsilon of the layers
GGD_EPS = 1e-5  # epsilon of the distance bias


def listed():
    return [
        # the op at its smallest configuration, in the accuracy mode: short prompts, few chunks
        dict(name='gdn_chunk_fp32_t256', kind='gdn_chunk', dtype='fp32', B=1, H=4, T=256, dk=64, dv=64, state=False),
        # the op over a long prompt at the model's heads
        dict(name='gdn_chunk_bf16_t8192', kind='gdn_chunk', dtype='bf16', B=1, H=12, T=8192, dk=64, dv=128, state=True),
        # one layer's op in a training step
        dict(name='gdn_train_bf16_t4096', kind='gdn_train', dtype='bf16', B=1, H=12, T=4096, dk=64, dv=128),
        # a layer over two ragged prompts that continue earlier ones
        dict(name='gdn_prefill_b2_t1000', kind='gdn_prefill', B=2, T=1000, cached=True),
        # interactive decoding: one sequence, where launches and the host count
        dict(name='gdn_decode_b1', kind='gdn_decode', B=1),
        # batched decoding: the recurrent states stream through memory
        dict(name='gdn_decode_b64', kind='gdn_decode', B=64),
        # the attention op of a 4096-token prefill at the model's grouped heads
        dict(name='chord_prefill_bf16_t4096', kind='chord_prefill', dtype='bf16', B=1, H=12, Hkv=3, D=64, L=4096,
             S=4096),
        # the same op in the accuracy mode, an odd length
        dict(name='chord_prefill_fp32_t1023', kind='chord_prefill', dtype='fp32', B=1, H=12, Hkv=3, D=64, L=1023,
             S=1023),
        # the attention op of a training step, two sequences, as many kv heads as heads
        dict(name='chord_train_b2_t2048', kind='chord_train', B=2, H=12, Hkv=12, L=2048),
        # batched decoding over long contexts: the KV cache streams through memory
        dict(name='chord_decode_b64_s4097', kind='chord_decode', B=64, H=12, Hkv=3, L=1, S=4097),
        # scoring / prompt ingestion with the whole model
        dict(name='model_prefill_b4_t2048', kind='model_prefill', B=4, T=2048),
        # serving: a batch of requests, ragged prompt length, then token by token
        dict(name='model_serve_b8_t300', kind='model_serve', B=8, T=300, steps=16),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(['gdn_chunk', 'gdn_train', 'gdn_prefill', 'gdn_decode', 'chord_prefill', 'chord_prefill',
                       'chord_train', 'chord_decode', 'model_prefill', 'model_serve'])
    if kind in ('gdn_chunk', 'gdn_train'):
        train = kind == 'gdn_train'
        B, H = rng.choice([1, 1, 2, 3]), rng.choice([4, 8, 12])
        dk, dv = rng.choice([(64, 128), (64, 64)] if train else [(64, 128), (64, 64), (32, 64)])
        c = dict(kind=kind, dtype=rng.choice(['bf16', 'bf16', 'fp32']), B=B, H=H,
                 T=_log_int(rng, 17, (4096 if train else 8192) * 12 // (B * H * 2)), dk=dk, dv=dv)
        if not train:
            c['state'] = rng.random() < 0.5
        return c
    if kind == 'gdn_prefill':
        B = rng.choice([1, 1, 2, 4])
        return dict(kind=kind, B=B, T=_log_int(rng, 2, 8192 // B), cached=rng.random() < 0.5)
    if kind == 'gdn_decode':
        return dict(kind=kind, B=_log_int(rng, 1, 64))
    if kind == 'chord_prefill':
        dtype = rng.choice(['bf16', 'bf16', 'bf16', 'fp16', 'fp32'])
        B, (H, Hkv) = rng.choice([1, 1, 2]), rng.choice([(12, 3), (12, 12), (8, 2)])
        D = rng.choice([64, 64, 64, 32, 128])
        S = _log_int(rng, 33, 4096 if dtype == 'bf16' and D == 64 else 1024)
        return dict(kind=kind, dtype=dtype, B=B, H=H, Hkv=Hkv, D=D,
                    L=S if rng.random() < 0.7 else rng.randint(17, S), S=S)
    if kind == 'chord_train':
        B, (H, Hkv) = rng.choice([1, 2]), rng.choice([(12, 3), (12, 12), (8, 2)])
        return dict(kind=kind, B=B, H=H, Hkv=Hkv, L=_log_int(rng, 33, 2048))
    if kind == 'chord_decode':
        H, Hkv = rng.choice([(12, 3), (12, 12), (8, 2)])
        B = _log_int(rng, 1, 64 * 3 // Hkv)
        return dict(kind=kind, B=B, H=H, Hkv=Hkv, L=rng.choice([1, 1, 1, 2]), S=_log_int(rng, 65, 4097))
    if kind == 'model_prefill':
        B = rng.choice([1, 2, 4])
        return dict(kind=kind, B=B, T=_log_int(rng, 65, 8192 // B))
    return dict(kind=kind, B=_log_int(rng, 1, 16), T=_log_int(rng, 17, 512), steps=rng.randint(4, 16))


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _gdn_inputs(case, seed):
    '''What a GatedDelta layer hands the op: L2-normalised q (scaled) and k, SiLU values,
    beta in (0, 1), log decays -A softplus(a + dt_bias) of the layer's initial range.'''
    g = _gen(seed)
    B, H, T, dk, dv = case['B'], case['H'], case['T'], case['dk'], case['dv']
    dt = DTYPES[case['dtype']]
    q = F.normalize(_randn(g, B, H, T, dk), dim=-1) * dk ** -0.5
    k = F.normalize(F.silu(_randn(g, B, H, T, dk)), dim=-1)
    v = F.silu(_randn(g, B, H, T, dv))
    beta = torch.sigmoid(_randn(g, B, H, T))
    A = torch.rand(H, generator=g, device=DEV) * 15 + 1
    d = torch.exp(torch.rand(H, generator=g, device=DEV) * math.log(100.0) + math.log(0.001))
    bias = d + torch.log(-torch.expm1(-d))
    gate = -A[:, None] * F.softplus(0.5 * _randn(g, B, H, T) + bias[:, None])
    # the op's tensors as a layer has them: [B, T, H, D] storage, transposed views
    q, k, v, beta, gate = (t.transpose(1, 2).to(dt).contiguous().transpose(1, 2) for t in (q, k, v, beta, gate))
    S = 0.1 * _randn(g, B, H, dk, dv) if case.get('state') else None
    do = _randn(g, B, T, H, dv).to(dt).transpose(1, 2)
    return q, k, v, beta, gate, S, do


def _chord_inputs(case, seed):
    '''What a Chord layer hands the op: RMS-normalised q and k, positive alpha, small beta
    and mu, ssmax near 1, log_n = ln(position + 1).'''
    g = _gen(seed)
    B, H, Hkv, L = case['B'], case['H'], case['Hkv'], case['L']
    S, D = case.get('S', L), case.get('D', 64)
    dt = DTYPES[case.get('dtype', 'bf16')]

    def rms(t):
        return t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + EPS)
    q = rms(_randn(g, B, H, L, D)).to(dt)
    k = rms(_randn(g, B, Hkv, S, D)).to(dt)
    v = (0.5 * _randn(g, B, Hkv, S, D)).to(dt)
    par = [torch.exp(0.3 * _randn(g, H)), 0.2 * _randn(g, H), 2 * torch.sinh(0.1 * _randn(g, H)),
           1 + 0.1 * _randn(g, H)]
    log_n = torch.log(torch.arange(S - L + 1, S + 1, dtype=torch.float32, device=DEV))[None].expand(B, L).contiguous()
    do = _randn(g, B, L, H, D).to(dt).transpose(1, 2)
    return q, k, v, par, log_n, do


@torch.no_grad()
def _fill(module, g):
    '''Random weights of a trained model's kind: short convs that mostly pass the current
    token, q / k norms below 1.  (Fresh weights with neither make the 16 layers a chaotic
    map: a rounding in the first moves the logits by their own size.)'''
    for name, p in module.named_parameters():
        last = name.rsplit('.', 1)[-1]
        if last == 'A_log':
            p.copy_(torch.log(torch.rand(p.shape, generator=g, device=DEV) * 15 + 1))
        elif last == 'dt_bias':
            d = torch.exp(torch.rand(p.shape, generator=g, device=DEV) * math.log(100.0) + math.log(0.001))
            p.copy_(d + torch.log(-torch.expm1(-d)))
        elif last == 'theta_alpha':
            p.copy_(0.3 * _randn(g, *p.shape))
        elif last == 'theta_beta':
            p.copy_(0.2 * _randn(g, *p.shape))
        elif last == 'theta_mu':
            p.copy_(0.1 * _randn(g, *p.shape))
        elif last == 'ssmax_s' or 'norm' in name:
            p.copy_((1 + 0.1 * _randn(g, *p.shape)) * (0.3 if 'q_norm' in name or 'k_norm' in name else 1.0))
        elif 'pseudo_queries' in name:
            p.copy_(0.005 * _randn(g, *p.shape))
        elif '_conv.' in name:
            p.copy_(0.06 * _randn(g, *p.shape))
            p[:, :, -1] += 1
        else:
            p.copy_(0.06 * _randn(g, *p.shape))
    return module.to(torch.bfloat16).eval()


def _layer(seed):
    with torch.device(DEV):
        layer = GatedDeltaAttention(hidden_size=WIDTH, num_heads=HEADS, head_k_dim=DK, expand_v=2.0)
    return _fill(layer, _gen(seed + 1))


def _model(seed):
    with torch.device(DEV):
        model = MotifChordModel(config_172m(VOCAB))
    return _fill(model, _gen(seed + 1))


def _layer_cache(B, g):
    '''What a layer's cache holds after earlier tokens: fp32 state, conv tails.'''
    state = 0.1 * _randn(g, B, HEADS, DK, DV)
    tails = tuple(_randn(g, B, HEADS * d, CONV - 1).to(torch.bfloat16) for d in (DK, DK, DV))
    return state, tails


def prepare(case, seed):
    kind = case['kind']
    g = _gen(seed + 2)
    st = dict(kind=kind)
    if kind in ('gdn_chunk', 'gdn_train'):
        st['args'] = _gdn_inputs(case, seed)
        if kind == 'gdn_train':
            for t in st['args'][:5]:
                t.requires_grad_()
    elif kind in ('chord_prefill', 'chord_train', 'chord_decode'):
        st['args'] = _chord_inputs(case, seed)
        if kind == 'chord_train':
            q, k, v, par, _, _ = st['args']
            for t in (q, k, v, par[0], par[1], par[3]):
                t.requires_grad_()
    elif kind in ('gdn_prefill', 'gdn_decode'):
        st['layer'] = _layer(seed)
        st['x'] = _randn(g, case['B'], case.get('T', 1), WIDTH).to(torch.bfloat16)
        st['carried'] = _layer_cache(case['B'], g) if kind == 'gdn_decode' or case['cached'] else None
    else:
        st['model'] = _model(seed)
        st['ids'] = torch.randint(0, VOCAB, (case['B'], case['T']), generator=g, device=DEV)
        if kind == 'model_serve':
            st['steps'] = torch.randint(0, VOCAB, (case['B'], case['steps']), generator=g, device=DEV)
            cache = ModelCache.for_decode(st['model'], case['B'], case['T'] + case['steps'], DEV, torch.bfloat16)
            st['cache'] = cache
            st['graph'] = DecodeGraph(st['model'], cache, case['B'])
    return st


# ------------------------------------------------------------------ one pass
def run(state):
    kind = state['kind']
    if kind == 'gdn_train':
        q, k, v, beta, gate, _, do = state['args']
        o, _ = chunk_gated_delta_rule(q, k, v, beta, gate)
        return [o.detach(), *torch.autograd.grad(o, (q, k, v, beta, gate), do)]
    if kind == 'chord_train':
        q, k, v, par, log_n, do = state['args']
        o = apply_chord_attention(q, k, v, *par, log_n)
        return [o.detach(), *torch.autograd.grad(o, (q, k, v, par[0], par[1], par[3]), do)]
    with torch.no_grad():
        if kind == 'gdn_chunk':
            q, k, v, beta, gate, S, _ = state['args']
            return list(chunk_gated_delta_rule(q, k, v, beta, gate, S))
        if kind in ('chord_prefill', 'chord_decode'):
            q, k, v, par, log_n, _ = state['args']
            return apply_chord_attention(q, k, v, *par, log_n)
        if kind in ('gdn_prefill', 'gdn_decode'):
            cache = GatedDeltaAttentionLayerCache()
            if state['carried'] is not None:
                cache.update(*state['carried'])
            y = state['layer'](state['x'], past_key_value=cache).output
            return [y, cache.state, *cache.conv_state]
        if kind == 'model_prefill':
            return state['model'](state['ids']).logits
        # a new request batch in the program's decode cache: prompts, then given tokens
        cache, graph, steps = state['cache'], state['graph'], state['steps']
        for lc in cache.layer_caches():
            lc.reset()
        for block in cache:
            block.attn_res.reset()
        first = state['model'](state['ids'], cache=cache).last_logits
        rest = [graph.step(steps[:, i:i + 1]).clone() for i in range(steps.shape[1])]
        return [first, torch.cat(rest, 1)]


# ------------------------------------------------------------------ what a pass cannot do without
def _gdn_flops(B, H, T, dk, dv):
    C = 64
    return B * H * T * (2 * C * (3 * dk + 2 * dv) + 6 * dk * dv + C * C / 3)


def _pairs(L, S):
    '''Visible (query, key) pairs of L queries that end at position S.'''
    return L * (S - L) + L * (L + 1) // 2


def _weights_params(layers_gdn, layers_chord, vocab=0):
    gdn = WIDTH * (2 * HEADS * DK + 2 * HEADS * DV + 2 * HEADS) + HEADS * DV * WIDTH
    chord = 3 * WIDTH * WIDTH + 2 * WIDTH * KV_HEADS * 64
    mlp = 3 * WIDTH * INNER
    return layers_gdn * (gdn + (mlp if vocab else 0)) + layers_chord * (chord + mlp) + vocab * WIDTH


def work(case):
    kind, B = case['kind'], case['B']
    if kind in ('gdn_chunk', 'gdn_train'):
        H, T, dk, dv = case['H'], case['T'], case['dk'], case['dv']
        e = DTYPES[case['dtype']].itemsize
        io = B * H * T * e * (2 * dk + 2 * dv + 2)
        if kind == 'gdn_train':  # forward, then inputs and dO again and a gradient per input
            return dict(bytes=io + 2 * B * H * T * e * (2 * dk + dv + 2) + B * H * T * e * dv,
                        flops=3 * _gdn_flops(B, H, T, dk, dv))
        return dict(bytes=io + 4 * B * H * dk * dv * (2 if case['state'] else 1), flops=_gdn_flops(B, H, T, dk, dv))
    if kind in ('chord_prefill', 'chord_train', 'chord_decode'):
        H, Hkv, L = case['H'], case['Hkv'], case['L']
        S, D = case.get('S', L), case.get('D', 64)
        e = DTYPES[case.get('dtype', 'bf16')].itemsize
        pairs = B * H * _pairs(L, S)
        nq, nkv = B * H * L * D, B * Hkv * S * D
        if kind == 'chord_train':
            return dict(bytes=e * (2 * nq + 2 * nkv + 4 * nq + 4 * nkv), flops=14 * D * pairs)
        return dict(bytes=e * (2 * nq + 2 * nkv), flops=4 * D * pairs)
    if kind in ('gdn_prefill', 'gdn_decode'):
        T = case.get('T', 1)
        n = _weights_params(1, 0)
        state = 4 * B * HEADS * DK * DV * (2 if kind == 'gdn_decode' or case['cached'] else 1)
        delta = _gdn_flops(B, HEADS, T, DK, DV) if T > 1 else 6.0 * B * HEADS * DK * DV
        return dict(bytes=2 * n + 4 * B * T * WIDTH + state, flops=2 * n * B * T + delta)
    T, steps = case['T'], case.get('steps', 0)
    n = _weights_params(12, 4)
    body = B * T * 2 * n + 12 * _gdn_flops(B, HEADS, T, DK, DV) + 4 * B * HEADS * 256 * _pairs(T, T)
    if kind == 'model_prefill':
        return dict(bytes=2 * (n + VOCAB * WIDTH) + 2 * B * T * VOCAB, flops=body + 2 * B * T * VOCAB * WIDTH)
    # the prompt's logits at its last position, then per step the weights, states and KV
    kv = 4 * 2 * 2 * KV_HEADS * 64 * B
    per = 2 * (n + VOCAB * WIDTH) + 12 * 2 * 4 * B * HEADS * DK * DV
    return dict(bytes=2 * n + sum(per + kv * (T + i) for i in range(steps)) + 2 * B * VOCAB * (steps + 1),
                flops=body + 2 * B * (steps + 1) * VOCAB * WIDTH + 2 * B * steps * n)


def tolerance(case):
    '''About four times the distance from the 64-bit result that was measured over the
    ranges above (the relative 2-norm and the largest error, over every output).'''
    kind, dtype = case['kind'], case.get('dtype', 'bf16')
    if kind in ('model_prefill', 'model_serve'):  # 16 layers of bf16 roundings: 7e-2 measured
        return {'rel': 0.25}
    if kind == 'chord_train':  # the sums over all pairs for alpha and ssmax cancel: up to 4e-2
        return {'rel': 0.15}
    if kind in ('gdn_prefill', 'gdn_decode'):
        return {'rel': 3e-2, 'max': 0.35}
    if dtype == 'fp32':
        return {'rel': 4e-6, 'max': 1e-4}
    if dtype == 'fp16':
        return {'rel': 1e-3, 'max': 5e-3}
    return {'rel': 1e-2, 'max': 0.15} if kind in ('gdn_chunk', 'gdn_train') else {'rel': 7e-3, 'max': 4e-2}


# ------------------------------------------------------------------ the same in 64 bits
def _gdn64(q, k, v, beta, g, S=None, C=64):
    '''The gated delta rule in its chunked form, differentiable.'''
    B, H, L, dk = q.shape
    dv = v.shape[-1]
    pad = (C - L % C) % C
    if pad:
        q, k, v = (F.pad(t, (0, 0, 0, pad)) for t in (q, k, v))
        beta, g = F.pad(beta, (0, pad)), F.pad(g, (0, pad))
    N = (L + pad) // C
    q, k, v = (t.reshape(B, H, N, C, -1) for t in (q, k, v))
    beta, g = beta.reshape(B, H, N, C), g.reshape(B, H, N, C)
    gam = g.cumsum(-1)
    low = torch.ones(C, C, dtype=torch.bool, device=q.device).tril()
    D = torch.exp((gam[..., :, None] - gam[..., None, :]).masked_fill(~low, float('-inf')))
    kb = k * beta[..., None]
    A = ((kb @ k.transpose(-1, -2)) * D).tril(-1)
    rhs = torch.cat([kb * gam.exp()[..., None], v * beta[..., None]], -1)
    eye = torch.eye(16, dtype=q.dtype, device=q.device)
    WU = rhs[..., :0, :]
    for r in range(0, C, 16):  # (I + A) WU = rhs by 16-row blocks; A's diagonal blocks are nilpotent
        a = A[..., r:r + 16, r:r + 16]
        inv, pw = eye - a, a @ a
        for _ in range(3):
            inv, pw = inv + inv @ pw, pw @ pw
        WU = torch.cat([WU, inv @ (rhs[..., r:r + 16, :] - A[..., r:r + 16, :r] @ WU)], -2)
    W, U = WU[..., :dk], WU[..., dk:]
    attn = (q @ k.transpose(-1, -2)) * D
    kd = (k * torch.exp(gam[..., -1:] - gam)[..., None]).transpose(-1, -2)
    qe = q * gam.exp()[..., None]
    last = gam[..., -1].exp()[..., None, None]
    S = torch.zeros(B, H, dk, dv, dtype=q.dtype, device=q.device) if S is None else S
    outs = []
    for n in range(N):
        X = U[:, :, n] - W[:, :, n] @ S
        outs.append(qe[:, :, n] @ S + attn[:, :, n] @ X)
        S = last[:, :, n] * S + kd[:, :, n] @ X
    return torch.cat(outs, 2)[:, :, :L], S


def _chord64(q, k, v, alpha, beta, mu, ssmax, log_n):
    B, H, L, D = q.shape
    S = k.shape[2]
    k, v = (t.repeat_interleave(H // t.shape[1], 1) for t in (k, v))
    d = torch.arange(S, device=q.device)[None] - (torch.arange(L, device=q.device)[:, None] + S - L)
    col = lambda t: t.view(H, 1, 1)  # noqa: E731
    outs = []
    for i in range(0, L, 1024):
        di = d[i:i + 1024]
        bias = -col(alpha) * ((di - col(mu)).abs() + GGD_EPS) ** col(beta)
        z = (q[:, :, i:i + 1024] @ k.transpose(-1, -2)) * D ** -0.5 + bias
        z = z * (col(ssmax) * log_n[:, None, i:i + 1024, None])
        outs.append(torch.softmax(z.masked_fill(di > 0, float('-inf')), -1) @ v)
    return torch.cat(outs, 2)


def _rms64(x, w):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w


def _gdn_layer64(x, p, state=None, tails=None):
    B, L, _ = x.shape
    heads, new_tails = [], []
    for i, n in enumerate('qkv'):
        xt = (x @ p[n + '_proj.weight'].t()).transpose(1, 2)
        w = p[n + '_conv.weight']
        t = xt.new_zeros(B, xt.shape[1], CONV - 1) if tails is None else tails[i]
        xc = torch.cat([t, xt], -1)
        new_tails.append(xc[..., -(CONV - 1):])
        y = sum(xc[..., j:j + L] * w[:, 0, j, None] for j in range(CONV))
        heads.append(F.silu(y).transpose(1, 2).reshape(B, L, HEADS, -1).transpose(1, 2))
    q, k, v = heads
    q, k = F.normalize(q, dim=-1) * DK ** -0.5, F.normalize(k, dim=-1)
    beta = torch.sigmoid(x @ p['b_proj.weight'].t()).transpose(1, 2)
    g = (-p['A_log'].exp() * F.softplus(x @ p['a_proj.weight'].t() + p['dt_bias'])).transpose(1, 2)
    o, S = _gdn64(q, k, v, beta, g, state)
    gate = (x @ p['g_proj.weight'].t()).view(B, L, HEADS, DV)
    y = _rms64(o.transpose(1, 2), p['o_norm.weight']) * F.silu(gate)
    return y.reshape(B, L, -1) @ p['o_proj.weight'].t(), S, new_tails


def _chord_layer64(x, p):
    B, L, _ = x.shape
    q, k, v = ((x @ p[n + '_proj.weight'].t()).view(B, L, -1, 64).transpose(1, 2) for n in 'qkv')
    q, k = _rms64(q, p['q_norm.weight']), _rms64(k, p['k_norm.weight'])
    mu = p['theta_mu'].exp() - (-p['theta_mu']).exp()
    log_n = torch.log(torch.arange(1, L + 1, dtype=x.dtype, device=x.device))[None].expand(B, L)
    o = torch.cat([_chord64(q[b:b + 1], k[b:b + 1], v[b:b + 1], p['theta_alpha'].exp(), p['theta_beta'], mu,
                            p['ssmax_s'], log_n[b:b + 1]) for b in range(B)])
    o = o.transpose(1, 2).reshape(B, L, -1) @ p['o_proj.weight'].t()
    return o * torch.sigmoid(x @ p['g_proj.weight'].t())


def _model64(p, ids, rows=None):
    '''Logits of every position, or of the last `rows` only.'''
    x = p['embed.weight' if 'embed.weight' in p else 'lm_head.weight'][ids]
    for b in range(4):
        pre = f'blocks.{b}.'
        sources, total = [x], None
        for i in range(4):
            if i == 0:
                h = x
            else:
                V = torch.stack(sources)
                K = _rms64(V, p[f'{pre}attn_res_norms.{i}.weight'])
                h = ((K @ p[f'{pre}pseudo_queries.{i}']).softmax(0)[..., None] * V).sum(0)
            f = f'{pre}features.{i}.'
            lp = {n[len(f) + 5:]: t for n, t in p.items() if n.startswith(f + 'attn.')}
            a = _rms64(h, p[f + 'attn_norm.weight'])
            a = _chord_layer64(a, lp) if i == 3 else _gdn_layer64(a, lp)[0]
            u, gt = (_rms64(h, p[f + 'mlp_norm.weight']) @ p[f + 'mlp.gate_up_proj.weight'].t()).chunk(2, -1)
            inc = a + (u * F.silu(gt)) @ p[f + 'mlp.down_proj.weight'].t()
            sources.append(inc)
            total = inc if total is None else total + inc
        x = total
    x = x if rows is None else x[:, -rows:]
    return _rms64(x, p['norm.weight']) @ p['lm_head.weight'].t()


def exact(case, seed):
    kind = case['kind']
    if kind == 'gdn_train':
        q, k, v, beta, gate, _, do = _gdn_inputs(case, seed)
        xs = [t.double().requires_grad_() for t in (q, k, v, beta, gate)]
        o = _gdn64(*xs)[0]
        return [o.detach(), *torch.autograd.grad(o, xs, do.double())]
    if kind == 'chord_train':
        q, k, v, par, log_n, do = _chord_inputs(case, seed)
        xs = [t.double().requires_grad_() for t in (q, k, v, *par)]
        o = _chord64(*xs, log_n.double())
        g = torch.autograd.grad(o, xs, do.double())
        return [o.detach(), *g[:5], g[6]]
    with torch.no_grad():
        if kind == 'gdn_chunk':
            q, k, v, beta, gate, S, _ = _gdn_inputs(case, seed)
            return list(_gdn64(*(t.double() for t in (q, k, v, beta, gate)), None if S is None else S.double()))
        if kind in ('chord_prefill', 'chord_decode'):
            q, k, v, par, log_n, _ = _chord_inputs(case, seed)
            return _chord64(*(t.double() for t in (q, k, v, *par, log_n)))
        st = prepare(case, seed)
        if kind in ('gdn_prefill', 'gdn_decode'):
            p = {n: t.double() for n, t in st['layer'].named_parameters()}
            S, tails = st['carried'] if st['carried'] is not None else (None, None)
            y, S, tails = _gdn_layer64(st['x'].double(), p, None if S is None else S.double(),
                                       None if tails is None else [t.double() for t in tails])
            return [y, S, *tails]
        p = {n: t.double() for n, t in st['model'].named_parameters()}
        p.setdefault('lm_head.weight', p.get('embed.weight'))
        if kind == 'model_prefill':
            return _model64(p, st['ids'])
        ids = torch.cat([st['ids'], st['steps']], 1)
        logits = _model64(p, ids, case['steps'] + 1)
        return [logits[:, 0], logits[:, 1:]]
