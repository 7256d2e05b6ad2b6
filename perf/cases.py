"""The work a user of this framework has it do, as cases that can be timed and checked one by one.

The path is batch-1 speech recognition at the dimensions of whisper-large-v3-turbo (1280 channels, 20 heads,
32 encoder and 4 decoder layers, 30 s windows of 1500 encoder frames). Each case calls public entry points as
``CustomModel`` does: ``load_ext()`` ops on tensors that the caller keeps, chains of launches inside a graph where
the model captures one, and ``CustomModel.transcribe`` for the whole call. Lengths are those of 1 to 30 s of audio
(50 encoder frames a second), the decoder positions those of its 448-token cache.

Kinds:
  mel        the log-mel front end of one clip (per-clip half, filterbank prepared once)
  stem       the two convolutions of the encoder's stem
  attention  the first half of an encoder layer: LayerNorm, q/k/v projection, self attention
  mlp        its second half: output projection + residual, LayerNorm, fc1 + GELU, split fc2, residual + next LayerNorm
  cross_kv   the cross K/V of every decoder layer from the encoder output
  encoder    stem, layers, final LayerNorm and cross K/V as one captured graph
  prompt     the 4 prompt positions as one launch
  steps      n decoder steps as one launch
  lane       one decoder step as separate launches in a graph (what concurrent lanes run)
  attend     one decode_attention call (self attention into the cache, or cross attention)
  transcribe waveform on the host to token ids
"""

import math

import numpy as np
import torch

from flash_whisper_amd._lib import (ACT_GELU, EPI_BIAS_GELU, EPI_BIAS_GELU_POS, EPI_BIAS_RESID, EPI_BIAS_RESID_CLAMP)
from flash_whisper_amd.audio import mel_filters, synthetic_clip
from flash_whisper_amd.ext import load_ext
from flash_whisper_amd.model import CustomModel

D, HEADS, FFN, VOCAB, MELS, MAX_POS, ENC = 1280, 20, 5120, 51866, 128, 448, 1500
DEC_LAYERS, EPS, SELF_SPLIT, CROSS_SPLIT = 4, 1e-5, 64, 256
HALF, DEV = torch.float16, 'cuda'


def listed():
    return [
        # the reference's drop-in attention op: one query over 224 cached positions, the smallest call
        {'name': 'attend_self', 'kind': 'attend', 'length': 224, 'max_len': MAX_POS, 'own': True},
        # the front end of every clip: a full window
        {'name': 'mel_30s', 'kind': 'mel', 'samples': 480000},
        # the stem of every clip
        {'name': 'stem_30s', 'kind': 'stem', 'frames': 1500},
        # the two halves of each of the 32 encoder layers of a full window
        {'name': 'attention_30s', 'kind': 'attention', 'frames': 1500},
        {'name': 'mlp_30s', 'kind': 'mlp', 'frames': 1500},
        # once per clip, the largest single product
        {'name': 'cross_kv_30s', 'kind': 'cross_kv', 'frames': 1500, 'layers': 4},
        # an encoder over a short clip's own frames (5 s, an odd count): few tiles, launches count
        {'name': 'encoder_5s', 'kind': 'encoder', 'frames': 251, 'layers': 4},
        # the whole encoder of a full window, as the model replays it
        {'name': 'encoder_30s', 'kind': 'encoder', 'frames': 1500, 'layers': 32},
        # time to first token: the prompt pass after the encoder
        {'name': 'prompt', 'kind': 'prompt', 'position': 0},
        # a chunk of 8 tokens in the middle of a transcript
        {'name': 'steps_8', 'kind': 'steps', 'position': 116, 'steps': 8},
        # one token of one of several concurrent lanes
        {'name': 'lane_step', 'kind': 'lane', 'position': 116},
        # the whole call: 30 s of audio, 224 tokens
        {'name': 'transcribe_30s', 'kind': 'transcribe', 'samples': 480000, 'tokens': 224},
    ]


def _spread(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(['mel', 'stem', 'attention', 'mlp', 'cross_kv', 'encoder', 'prompt', 'steps', 'lane', 'attend'])
    if kind == 'mel':
        return {'kind': kind, 'samples': _spread(rng, 8000, 480000)}
    if kind == 'cross_kv':
        return {'kind': kind, 'frames': _spread(rng, 50, 1500), 'layers': rng.randint(1, 4)}
    if kind == 'encoder':
        return {'kind': kind, 'frames': _spread(rng, 50, 1500), 'layers': rng.randint(2, 6)}
    if kind == 'prompt':
        return {'kind': kind, 'position': rng.randint(0, MAX_POS - 4)}
    if kind == 'steps':
        return {'kind': kind, 'position': rng.randint(4, MAX_POS - 9), 'steps': rng.randint(1, 8)}
    if kind == 'lane':
        return {'kind': kind, 'position': rng.randint(4, MAX_POS - 1)}
    if kind == 'attend':
        if rng.random() < 0.3:
            n = _spread(rng, 50, 1500)
            return {'kind': kind, 'length': n, 'max_len': n, 'own': False}
        return {'kind': kind, 'length': rng.randint(1, MAX_POS), 'max_len': MAX_POS, 'own': True}
    return {'kind': kind, 'frames': _spread(rng, 50, 1500)}


# ---- inputs -----------------------------------------------------------------------------------
class _Make:
    """Seeded tensors on the GPU. Weights are N(0, 0.02) as the framework's own seeded checkpoint has them;
    q and k rows of the attention are wider, so that the softmax has rows with a clear maximum as a trained
    model's does."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(int(seed))

    def normal(self, *shape, std=1.0, mean=0.0, dtype=HALF):
        return (torch.randn(*shape, generator=self.g, device=DEV) * std + mean).to(dtype)

    def linear(self, n, k, std=0.02):
        return self.normal(n, k, std=std), self.normal(n, std=0.02)

    def ln(self):
        return self.normal(D, std=0.05, mean=1.0), self.normal(D, std=0.05), EPS

    def qkv(self):
        w, b = self.linear(3 * D, D)
        w[:2 * D] *= 2.0
        b[D:2 * D] = 0
        return w, b


def _stem_weights(m):
    return {'w1': m.normal(D, 3 * MELS, std=0.02), 'b1': m.normal(D, std=0.02), 'w2': m.normal(D, 3 * D, std=0.02),
            'b2': m.normal(D, std=0.02)}


def _mel_input(m, frames):
    """Log-mel features lie in about [-1, 1.5] with neighbouring bins alike."""
    return (m.normal(2 * frames, MELS, std=0.4) + m.normal(2 * frames, 1, std=0.3)).clamp(-1, 1.5).contiguous()


def _enc_layer(m):
    qkv_w, qkv_b = m.qkv()
    out_w, out_b = m.linear(D, D)
    fc1_w, fc1_b = m.linear(FFN, D)
    fc2_w, fc2_b = m.linear(D, FFN)
    return {'ln1': m.ln(), 'qkv_w': qkv_w, 'qkv_b': qkv_b, 'out_w': out_w, 'out_b': out_b, 'ln2': m.ln(),
            'fc1_w': fc1_w, 'fc1_b': fc1_b, 'fc2_w': fc2_w, 'fc2_b': fc2_b}


def _cross_weights(m, layers):
    w, b = m.linear(layers * 2 * D, D)
    b.view(layers, 2, D)[:, 0] = 0
    return w, b


def _dec_layer(m):
    qkv_w, qkv_b = m.qkv()
    lay = {'qkv_w': qkv_w, 'qkv_b': qkv_b}
    for j in (1, 2, 3):
        lay[f'ln{j}_gamma'], lay[f'ln{j}_beta'], lay[f'ln{j}_eps'] = m.ln()
    for name, n, k in (('out', D, D), ('cross_q', D, D), ('cross_out', D, D), ('fc1', FFN, D), ('fc2', D, FFN)):
        lay[f'{name}_w'], lay[f'{name}_b'] = m.linear(n, k)
    return lay


def _decoder(m, position):
    """A decoder in the middle of a transcript: weights, a cache filled up to `position`, the cross K/V of a full
    window, a token to feed."""
    dec = {'layers': [_dec_layer(m) for _ in range(DEC_LAYERS)], 'embed': m.normal(VOCAB, D, std=0.02),
           'pos_embed': m.normal(MAX_POS, D, std=0.02), 'ln': m.ln(),
           'self_kv': m.normal(DEC_LAYERS, 2, HEADS, MAX_POS, 64), 'cross_kv': m.normal(DEC_LAYERS, 2, HEADS, ENC, 64)}
    dec['suppress'] = torch.zeros(VOCAB, dtype=torch.bool, device=DEV)
    dec['suppress'][torch.randint(0, VOCAB, (30,), generator=m.g, device=DEV)] = True
    dec['start'] = torch.tensor([position, 0], device=DEV)
    dec['fed'] = torch.randint(0, VOCAB, (4,), generator=m.g, device=DEV)
    return dec


def _decoder_state(dec):
    """The buffers and handles a program keeps beside the weights."""
    ext = load_ext()
    for i, lay in enumerate(dec['layers']):
        lay['self_k'], lay['self_v'] = dec['self_kv'][i, 0], dec['self_kv'][i, 1]
        lay['cross_k'], lay['cross_v'] = dec['cross_kv'][i, 0], dec['cross_kv'][i, 1]
    dec['wq'], dec['meta'] = ext.lm_head_q8_table(dec['embed'])
    dec['cur'] = torch.zeros(1, dtype=torch.long, device=DEV)
    dec['state'] = torch.zeros(2, dtype=torch.long, device=DEV)
    dec['tokens'] = torch.zeros(MAX_POS, dtype=torch.long, device=DEV)
    return ext


def _split_workspace(splits):
    return (torch.empty(HEADS * splits, device=DEV), torch.empty(HEADS * splits, device=DEV),
            torch.empty(HEADS * splits * 64, device=DEV))


def _captured(fn):
    """fn's launches as a graph, warmed up on a side stream, as the model captures its own."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        fn()
    return graph


# ---- the launches of each kind ----------------------------------------------------------------
def _stem(ext, s, out):
    ext.conv1d(s['mel'], 1, s['w1'], s['b1'], s['x1'], EPI_BIAS_GELU)
    ext.conv1d(s['x1'], 2, s['w2'], s['b2'], out, EPI_BIAS_GELU_POS, res=s['pos'])


def _attention_half(ext, s, lay):
    ext.encoder_qkv(s['y'], lay['qkv_w'], lay['qkv_b'], s['qkv'], s['vt'], HEADS)
    ext.encoder_attention(s['qkv'], s['vt'], s['attn'], HEADS)


def _mlp_half(ext, s, lay, res, ln_next, out):
    ext.gemm(s['attn'], lay['out_w'], lay['out_b'], s['h'], EPI_BIAS_RESID, res=res)
    ext.layernorm_rows(s['h'], *lay['ln2'][:2], s['y'], EPS)
    ext.gemm(s['y'], lay['fc1_w'], lay['fc1_b'], s['ffn'], EPI_BIAS_GELU)
    ext.gemm_splitk(s['ffn'], lay['fc2_w'], s['part'])
    ext.layernorm_rows_residual(s['part'], lay['fc2_b'], s['h'], *ln_next[:2], out, EPS, EPI_BIAS_RESID_CLAMP)


def _encoder(ext, s):
    _stem(ext, s, s['h'])
    ext.layernorm_rows(s['h'], *s['layers'][0]['ln1'][:2], s['y'], EPS)
    for i, lay in enumerate(s['layers']):
        last = i + 1 == len(s['layers'])
        _attention_half(ext, s, lay)
        _mlp_half(ext, s, lay, s['h'], s['ln'] if last else s['layers'][i + 1]['ln1'], s['enc_out'] if last else s['y'])
    ext.cross_kv(s['enc_out'], s['cross_w'], s['cross_b'], s['cross_kv'])


def _lane_step(ext, s):
    """One token in separate launches, as a lane of several in flight runs it."""
    ws, h = s['ws'], s['hb']
    q, k_new, v_new = s['qkv'][:D], s['qkv'][D:2 * D], s['qkv'][2 * D:]
    a, b = 0, 1
    for i, lay in enumerate(s['layers']):
        embed = (s['cur'], s['state'], s['embed'], s['pos_embed']) if i == 0 else None
        ext.ln_gemv(None if i == 0 else h[b], None if i == 0 else s['pending'], h[a], lay['ln1_gamma'], lay['ln1_beta'],
                    EPS, lay['qkv_w'], lay['qkv_b'], s['qkv'], embed=embed)
        ext.attention_split(q, lay['self_k'], lay['self_v'], s['state'], k_new, v_new, *ws, 0.125, SELF_SPLIT)
        ext.attn_out_gemv(*ws, s['state'], HEADS, MAX_POS, lay['out_w'], lay['out_b'], s['xo'], SELF_SPLIT)
        ext.ln_gemv(h[a], s['xo'], h[b], lay['ln2_gamma'], lay['ln2_beta'], EPS, lay['cross_q_w'], lay['cross_q_b'],
                    s['q'])
        ext.attention_split(s['q'], lay['cross_k'], lay['cross_v'], None, None, None, *ws, 0.125, CROSS_SPLIT)
        ext.attn_out_gemv(*ws, None, HEADS, ENC, lay['cross_out_w'], lay['cross_out_b'], s['xo'], CROSS_SPLIT)
        ext.ln_gemv(h[b], s['xo'], h[a], lay['ln3_gamma'], lay['ln3_beta'], EPS, lay['fc1_w'], lay['fc1_b'], s['ffn'],
                    act=ACT_GELU)
        ext.gemv(s['ffn'], lay['fc2_w'], lay['fc2_b'], s['pending'])
        a, b = b, a
    s['last'] = b
    ext.lm_head_argmax_q8(h[b], s['pending'], *s['ln'], s['embed'], s['wq'], s['meta'], s['suppress'], s['best'],
                          s['tokens'], s['state'], s['cur'], MAX_POS)


# ---- prepare / run ----------------------------------------------------------------------------
def _inputs(case, seed):
    """The inputs of a case, made from the seed alone: what exact() and prepare() both start from."""
    m, kind = _Make(seed), case['kind']
    if kind == 'mel':
        clip = synthetic_clip(seed, case['samples'])
        return {'wave': torch.from_numpy(clip).to(DEV), 'filters': torch.from_numpy(mel_filters()).to(DEV)}
    if kind == 'stem':
        t = case['frames']
        return {'mel': _mel_input(m, t), 'pos': m.normal(t, D, std=0.7), **_stem_weights(m)}
    if kind == 'attention':
        return {'x': m.normal(case['frames'], D), 'layer': _enc_layer(m)}
    if kind == 'mlp':
        t = case['frames']
        return {'x': m.normal(t, D), 'attn': m.normal(t, D, std=0.5), 'layer': _enc_layer(m), 'next': m.ln()}
    if kind == 'cross_kv':
        w, b = _cross_weights(m, case['layers'])
        return {'enc_out': m.normal(case['frames'], D), 'cross_w': w, 'cross_b': b}
    if kind == 'encoder':
        t = case['frames']
        w, b = _cross_weights(m, DEC_LAYERS)
        return {'mel': _mel_input(m, t), 'pos': m.normal(t, D, std=0.7), **_stem_weights(m), 'ln': m.ln(),
                'layers': [_enc_layer(m) for _ in range(case['layers'])], 'cross_w': w, 'cross_b': b}
    if kind in ('prompt', 'steps', 'lane'):
        return _decoder(m, case['position'])
    if kind == 'attend':
        s = {'q': m.normal(HEADS * 64, std=2.0), 'k': m.normal(HEADS, case['max_len'], 64),
             'v': m.normal(HEADS, case['max_len'], 64)}
        if case['own']:
            s.update(k_new=m.normal(HEADS * 64), v_new=m.normal(HEADS * 64),
                     state=torch.tensor([case['length'] - 1, 0], device=DEV))
        return s
    return {'audio': synthetic_clip(seed, case['samples'])}


def prepare(case, seed):
    ext, kind, s = load_ext(), case['kind'], _inputs(case, seed)
    s['case'], s['ext'] = case, ext

    def half(*shape):
        return torch.zeros(*shape, dtype=HALF, device=DEV)

    if kind == 'mel':
        n = case['samples'] // 160
        s['out'], s['out16'] = torch.empty(MELS, n, device=DEV), half(n, MELS)
        s['ws'] = ext.log_mel_workspace(case['samples'])
        ext.log_mel_prepare(s['filters'], s['ws'])
    elif kind == 'stem':
        s['x1'], s['out'] = half(2 * case['frames'], D), half(case['frames'], D)
    elif kind in ('attention', 'mlp', 'encoder'):
        t = case['frames']
        for name, cols in (('y', D), ('h', D), ('enc_out', D), ('ffn', FFN)):
            s[name] = half(t, cols)
        s['part'] = torch.empty(2, t, D, device=DEV)
        if kind != 'mlp':
            s['qkv'], s['attn'], s['vt'] = half(t, 3 * D), half(t, D), ext.encoder_vt_workspace(t, HEADS)
        if kind == 'encoder':
            s['x1'], s['cross_kv'] = half(2 * t, D), half(DEC_LAYERS, 2, HEADS, t, 64)
            s['graph'] = _captured(lambda: _encoder(ext, s))
    elif kind == 'cross_kv':
        s['cross_kv'] = half(case['layers'], 2, HEADS, case['frames'], 64)
    elif kind in ('prompt', 'steps'):
        _decoder_state(s)
        s['y'] = half(D)
        s['step_ws'] = ext.decoder_step_workspace(DEC_LAYERS)
        s['table'] = ext.decoder_layer_table(s['layers'])
        s['head'] = ext.decoder_head(*s['ln'], s['embed'], s['wq'], s['meta'], s['suppress'], s['tokens'], s['y'])
    elif kind == 'lane':
        _decoder_state(s)
        s['hb'], s['qkv'], s['q'], s['xo'], s['ffn'] = half(2, D), half(3 * D), half(D), half(D), half(FFN)
        s['pending'], s['best'] = half(D), torch.zeros(1, dtype=torch.long, device=DEV)
        s['ws'] = _split_workspace(-(-ENC // SELF_SPLIT))
        s['state'].copy_(s['start'])  # the warm-up writes the cache row that every pass writes
        s['graph'] = _captured(lambda: _lane_step(ext, s))
    elif kind == 'attend':
        s['out'], s['ws'] = half(HEADS * 64), _split_workspace(-(-case['max_len'] // SELF_SPLIT))
    else:
        s['model'] = CustomModel(seed=seed, selftest=False)
    return s


def run(s):
    ext, case = s['ext'], s['case']
    kind = case['kind']
    if kind == 'mel':
        ext.log_mel_run(s['wave'], s['filters'], s['out'], s['out16'], s['ws'])
        return {'mel': s['out'], 'mel16': s['out16']}
    if kind == 'stem':
        _stem(ext, s, s['out'])
        return {'x1': s['x1'], 'x': s['out']}
    if kind == 'attention':
        ext.layernorm_rows(s['x'], *s['layer']['ln1'][:2], s['y'], EPS)
        _attention_half(ext, s, s['layer'])
        return {'y': s['y'], 'attn': s['attn']}
    if kind == 'mlp':
        _mlp_half(ext, s, s['layer'], s['x'], s['next'], s['enc_out'])
        return {'h': s['h'], 'y': s['enc_out']}
    if kind == 'cross_kv':
        ext.cross_kv(s['enc_out'], s['cross_w'], s['cross_b'], s['cross_kv'])
        return s['cross_kv']
    if kind == 'encoder':
        s['graph'].replay()
        return {'enc_out': s['enc_out'], 'cross_kv': s['cross_kv']}
    if kind == 'prompt':
        s['state'].copy_(s['start'])
        ext.decoder_prompt(s['table'], s['head'], s['fed'], s['cur'], s['state'], s['embed'], s['pos_embed'], MAX_POS,
                           ENC, 0.125, s['step_ws'], VOCAB)
        return {'y': s['y'], 'self_kv': s['self_kv'], 'cur': s['cur'], 'state': s['state']}
    if kind == 'steps':
        s['state'].copy_(s['start'])
        s['cur'].copy_(s['fed'][:1])
        ext.decoder_step(s['table'], s['head'], s['cur'], s['state'], s['embed'], s['pos_embed'], MAX_POS, ENC, 0.125,
                         s['step_ws'], VOCAB, n_steps=case['steps'])
        return {'y': s['y'], 'self_kv': s['self_kv'], 'tokens': s['tokens'], 'state': s['state']}
    if kind == 'lane':
        s['state'].copy_(s['start'])
        s['cur'].copy_(s['fed'][:1])
        s['graph'].replay()
        return {'h': s['hb'][s['last']], 'x': s['pending'], 'self_kv': s['self_kv'], 'cur': s['cur'],
                'state': s['state']}
    if kind == 'attend':
        ext.decode_attention(s['q'], s['k'], s['v'], s['out'], s.get('state'), s.get('k_new'), s.get('v_new'), *s['ws'],
                             0.125)
        return {'out': s['out'], 'k': s['k'], 'v': s['v']} if case['own'] else {'out': s['out']}
    model = s['model']
    ids = model.transcribe(s['audio'], max_new_tokens=case['tokens'], stop_at_eos=False)['token_ids']
    return {'ids': np.array(ids, dtype=np.int64), 'mel': model.mel32, 'enc_out': model.enc_out,
            'cross_kv': model.cross_kv}


# ---- what a pass cannot do without --------------------------------------------------------------
def _gemm(m, n, k):
    return 2.0 * m * n * k


def _encoder_layer_work(t):
    weights = 2.0 * (4 * D * D + 2 * D * FFN)
    return weights, _gemm(t, 4 * D + 2 * FFN, D) + 4.0 * t * t * D


def _step_bytes(position, vectors=1):
    """Weights of the layers, the caches that are read, the int8 LM head (its row scales and flags too)."""
    layer = 2.0 * (6 * D * D + 2 * D * FFN) + 2.0 * 2 * ENC * D + 2.0 * 2 * (position + vectors) * D
    return DEC_LAYERS * layer + VOCAB * (D + 9.0)


def work(case):
    kind = case['kind']
    if kind == 'mel':
        n = case['samples'] // 160
        return {'bytes': 4.0 * case['samples'] + 6.0 * MELS * n, 'flops': n * (2.5 * 400 * math.log2(400) + 4 * 400)}
    t = case.get('frames', ENC)
    stem = {'bytes': 2.0 * (2 * t * MELS + 3 * MELS * D + 3 * D * D + 2 * t * D + 2 * t * D),
            'flops': _gemm(2 * t, D, 3 * MELS) + _gemm(t, D, 3 * D)}
    if kind == 'stem':
        return stem
    if kind == 'attention':
        return {'bytes': 2.0 * (3 * D * D + 2 * t * D), 'flops': _gemm(t, 3 * D, D) + 4.0 * t * t * D}
    if kind == 'mlp':
        return {'bytes': 2.0 * (D * D + 2 * D * FFN + 4 * t * D), 'flops': _gemm(t, D + 2 * FFN, D)}
    cross = case.get('layers', 0) if kind == 'cross_kv' else DEC_LAYERS
    kv = {'bytes': 2.0 * (2 * cross * D * D + t * D + 2 * cross * t * D), 'flops': _gemm(t, 2 * cross * D, D)}
    if kind == 'cross_kv':
        return kv
    if kind in ('encoder', 'transcribe'):
        weights, flops = _encoder_layer_work(t)
        layers = case.get('layers', 32)
        w = {'bytes': stem['bytes'] + layers * weights + kv['bytes'], 'flops': stem['flops'] + layers * flops + kv['flops']}
        if kind == 'transcribe':
            w['bytes'] += 4.0 * case['samples'] + case['tokens'] * _step_bytes(4 + case['tokens'] / 2)
            w['flops'] += case['tokens'] * 2 * (DEC_LAYERS * (6 * D * D + 2 * D * FFN) + VOCAB * D)
        return w
    if kind in ('prompt', 'steps', 'lane'):
        n = 4 if kind == 'prompt' else case.get('steps', 1)
        b = _step_bytes(case['position'], 4) if kind == 'prompt' else n * _step_bytes(case['position'] + (n - 1) / 2)
        return {'bytes': b, 'flops': n * 2.0 * (DEC_LAYERS * (6 * D * D + 2 * D * FFN) + VOCAB * D)}
    return {'bytes': 2.0 * (2 * case['length'] * D + 2 * D), 'flops': 4.0 * case['length'] * D}


def tolerance(case):
    """fp16 activations, 32-bit sums. Measured: each kind's distance from the 64-bit result, which another
    correct order of the sums moves by less; about four times that is stated."""
    return {
        'mel': {'rel': 9e-4},
        'stem': {'rel': 1.2e-3},
        'attention': {'rel': 3e-3},
        'mlp': {'rel': 1.8e-3},
        'cross_kv': {'rel': 8e-4},
        'encoder': {'rel': 7e-3},
        'prompt': {'rel': 6e-3, 'differ': 0.01},
        'steps': {'rel': 6e-3, 'differ': 0.01},
        'lane': {'rel': 6e-3, 'differ': 0.01},
        'attend': {'rel': 8e-4},
        'transcribe': {'rel': 7e-3, 'differ': 0.01},
    }[case['kind']]


# ---- the same in 64 bits ------------------------------------------------------------------------
def _f(x):
    return x.double()


def _lin(x, w, b):
    return x @ _f(w).T + _f(b)


def _norm(x, ln):
    return torch.nn.functional.layer_norm(x, (D,), _f(ln[0]), _f(ln[1]), EPS)


def _gelu(x):
    return torch.nn.functional.gelu(x)


def _conv(x, w, b, stride):
    """Kernel 3, padding 1; columns of w are tap-major."""
    p = torch.nn.functional.pad(x, (0, 0, 1, 1))
    n = (x.size(0) - 1) // stride + 1
    taps = [p[i:i + (n - 1) * stride + 1:stride] for i in range(3)]
    return _lin(torch.cat(taps, 1), w, b)


def _attend(q, k, v, scale):
    """q [n, D], k and v [keys, D], head by head."""
    outs = []
    for h in range(HEADS):
        c = slice(64 * h, 64 * h + 64)
        outs.append(torch.softmax(q[:, c] @ k[:, c].T * scale, -1) @ v[:, c])
    return torch.cat(outs, 1)


def _exact_stem(s):
    x1 = _gelu(_conv(_f(s['mel']), s['w1'], s['b1'], 1))
    return x1, _gelu(_conv(x1, s['w2'], s['b2'], 2)) + _f(s['pos'])


def _exact_attention(y, lay):
    qkv = _lin(y, lay['qkv_w'], lay['qkv_b'])
    return _attend(qkv[:, :D], qkv[:, D:2 * D], qkv[:, 2 * D:], 0.125)


def _exact_mlp(x, attn, lay):
    h = x + _lin(attn, lay['out_w'], lay['out_b'])
    return h + _lin(_gelu(_lin(_norm(h, lay['ln2']), lay['fc1_w'], lay['fc1_b'])), lay['fc2_w'], lay['fc2_b'])


def _exact_cross(enc, w, b, layers):
    return _lin(enc, w, b).view(enc.size(0), layers, 2, HEADS, 64).permute(1, 2, 3, 0, 4)


def _exact_mel(wave, filters):
    x = _f(wave)
    spec = torch.stft(x, 400, 160, window=torch.hann_window(400, device=DEV, dtype=torch.float64), return_complex=True)
    mel = torch.clamp(_f(filters).T @ spec[..., :wave.numel() // 160].abs().square(), min=1e-10).log10()
    return (torch.maximum(mel, mel.max() - 8.0) + 4.0) / 4.0


def _exact_decoder(s, ids, position):
    """The rows of `ids` from `position` on: (residual before the last fc2, its output, final LayerNorm, caches)."""
    n = len(ids)
    kv, x = _f(s['self_kv']).clone(), _f(s['embed'][ids]) + _f(s['pos_embed'][position:position + n])
    add = None
    for i, lay in enumerate(s['layers']):
        ln = [(lay[f'ln{j}_gamma'], lay[f'ln{j}_beta']) for j in (1, 2, 3)]
        x = x if add is None else x + add
        qkv = _lin(_norm(x, ln[0]), lay['qkv_w'], lay['qkv_b'])
        kv[i, :, :, position:position + n] = qkv[:, D:].view(n, 2, HEADS, 64).permute(1, 2, 0, 3)
        rows = []
        for z in range(n):
            k, v = (kv[i, j, :, :position + z + 1].permute(1, 0, 2).reshape(-1, D) for j in (0, 1))
            rows.append(_attend(qkv[z:z + 1, :D], k, v, 0.125))
        x = x + _lin(torch.cat(rows), lay['out_w'], lay['out_b'])
        k, v = (_f(s['cross_kv'][i, j]).permute(1, 0, 2).reshape(-1, D) for j in (0, 1))
        q = _lin(_norm(x, ln[1]), lay['cross_q_w'], lay['cross_q_b'])
        x = x + _lin(_attend(q, k, v, 0.125), lay['cross_out_w'], lay['cross_out_b'])
        add = _lin(_gelu(_lin(_norm(x, ln[2]), lay['fc1_w'], lay['fc1_b'])), lay['fc2_w'], lay['fc2_b'])
    return x[-1], add[-1], _norm(x + add, s['ln'])[-1], kv


def exact(case, seed):
    kind = case['kind']
    if kind == 'transcribe':  # its stages are the cases 'encoder' and 'steps'; here the front end
        wave = torch.from_numpy(synthetic_clip(seed, case['samples'])).to(DEV)
        return {'ids': None, 'mel': _exact_mel(wave, torch.from_numpy(mel_filters()).to(DEV)), 'enc_out': None,
                'cross_kv': None}
    if kind == 'steps' and case['steps'] > 1:  # a tie that rounds the other way feeds another token
        return None
    s = _inputs(case, seed)
    if kind == 'mel':
        mel = _exact_mel(s['wave'], s['filters'])
        return {'mel': mel, 'mel16': mel.T.contiguous()}
    if kind == 'stem':
        x1, x = _exact_stem(s)
        return {'x1': x1, 'x': x}
    if kind == 'attention':
        y = _norm(_f(s['x']), s['layer']['ln1'])
        return {'y': y, 'attn': _exact_attention(y, s['layer'])}
    if kind == 'mlp':
        h = _exact_mlp(_f(s['x']), _f(s['attn']), s['layer'])
        return {'h': h, 'y': _norm(h, s['next'])}
    if kind == 'cross_kv':
        return _exact_cross(_f(s['enc_out']), s['cross_w'], s['cross_b'], case['layers'])
    if kind == 'encoder':
        x = _exact_stem(s)[1]
        for lay in s['layers']:
            x = _exact_mlp(x, _exact_attention(_norm(x, lay['ln1']), lay), lay)
        enc = _norm(x, s['ln'])
        return {'enc_out': enc, 'cross_kv': _exact_cross(enc, s['cross_w'], s['cross_b'], DEC_LAYERS)}
    if kind in ('prompt', 'steps', 'lane'):
        ids = s['fed'] if kind == 'prompt' else s['fed'][:1]
        h, x, y, kv = _exact_decoder(s, ids, case['position'])
        if kind == 'lane':
            return {'h': h, 'x': x, 'self_kv': kv, 'cur': None, 'state': None}
        whole = {'cur': None} if kind == 'prompt' else {'tokens': None}
        return {'y': y, 'self_kv': kv, **whole, 'state': None}
    k, v, n = _f(s['k']), _f(s['v']), case['length']
    if case['own']:
        k[:, n - 1], v[:, n - 1] = _f(s['k_new']).view(HEADS, 64), _f(s['v_new']).view(HEADS, 64)
    out = _attend(_f(s['q']).view(1, D), k[:, :n].permute(1, 0, 2).reshape(-1, D), v[:, :n].permute(1, 0, 2).reshape(-1, D),
                  0.125)[0]
    return {'out': out, 'k': k, 'v': v} if case['own'] else {'out': out}
