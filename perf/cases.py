"""The performance cases of this library: what its users have it do, through its public classes.

Eight kinds of work, one function per kind and step below:

  act      per-token fake quantization of activations (RTN.a_qdq), from one decode batch to a prefill of 8192 tokens
  rtn      round-to-nearest of one weight matrix: fake and / or real quantization, every row type
  vllm     real-quantized containers in the compressed-tensors layout (VllmRealQuantLinear.new): quantize, pack
  awq_pack real-quantized containers in the AutoAWQ layout (AutoawqRealQuantLinear.new)
  blockfp8 block-wise float8 weights to bf16 and back (float8 checkpoints)
  gptq     GPTQ of one subset list: Hessians from calibration batches, Cholesky chains, column loops
  awq      AWQ 20-point scale search on a SwiGLU MLP (the forward passes are library GEMMs)
  clip     AWQ weight-clip search and the clamp of every Linear of an MLP block

Weights are Gaussian with a few large outliers, activations Gaussian with a lognormal scale per channel: the outlier
channels are what the algorithms exist for.
"""
import math

import torch

from lightcompress_amd import IntegerQuantizer
from lightcompress_amd.auto_clip import AutoClipper
from lightcompress_amd.awq import Awq
from lightcompress_amd.gptq import GPTQ
from lightcompress_amd.kernel import weight_cast_to_bf16, weight_cast_to_fp8
from lightcompress_amd.module_utils import AutoawqRealQuantLinear, VllmRealQuantLinear
from lightcompress_amd.rtn import RTN

DTYPES = {'bf16': torch.bfloat16, 'fp16': torch.float16, 'fp32': torch.float32}
SIZE = {'bf16': 2, 'fp16': 2, 'fp32': 4}


def listed():
    return [
        # activations of a decode step: 16 sequences, one token each, in front of a w8a8 Linear; called once per Linear
        # and token, so the call itself is what counts
        dict(name='act_decode_int8', kind='act', tokens=16, cols=4096, dtype='bf16', quant='int8'),
        # activations of a long prefill, float8 per token (the largest activation tensor of the benchmark)
        dict(name='act_prefill_fp8', kind='act', tokens=8192, cols=7168, dtype='bf16', quant='e4m3'),
        # a half-precision checkpoint with a ragged number of tokens, int8 per token
        dict(name='act_fp16_ragged', kind='act', tokens=2049, cols=5120, dtype='fp16', quant='int8'),
        # round-to-nearest of a full-precision weight, int4 asymmetric groups of 128: evaluation and codes
        dict(name='rtn_int4_fp32', kind='rtn', rows=4096, cols=4096, dtype='fp32', bit=4, sym=False, group=128, mode='both'),
        # round-to-nearest with the 80-step mean-squared-error range search (calib_algo mse)
        dict(name='rtn_mse_bf16', kind='rtn', rows=4096, cols=4096, dtype='bf16', bit=4, sym=False, group=128, mode='mse'),
        # deployment of eight experts' gate / up / down matrices for vLLM: int4 groups of 128, packed
        dict(name='vllm_int4_experts', kind='vllm', linears=24, rows=2048, cols=7168, dtype='bf16', bit=4, group=128),
        # deployment of one MLP matrix for AutoAWQ
        dict(name='awq_pack_mlp', kind='awq_pack', rows=11008, cols=4096, dtype='bf16', group=128),
        # a block-wise float8 checkpoint matrix to bf16 and back, last blocks partly filled
        dict(name='blockfp8_ragged', kind='blockfp8', rows=2112, cols=7168),
        # GPTQ of a small Linear on few tokens: symmetric, no act-order, ragged batches; the serial parts dominate
        dict(name='gptq_small', kind='gptq', layer='one', rows=1000, cols=1024, batches=32, tokens=501, dtype='bf16', sym=True,
             actorder=False, group=128),
        # GPTQ of a whole decoder layer, 128 x 2048 tokens per activation stream: the headline workload
        dict(name='gptq_layer', kind='gptq', layer='decoder', rows=4096, cols=14336, batches=128, tokens=2048, dtype='bf16',
             sym=False, actorder=True, group=128),
        # AWQ scale search of an MLP's gate and up projections, 128 x 512 tokens
        dict(name='awq_search_mlp', kind='awq', hidden=4096, inter=11008, batches=128, tokens=512, group=128),
        # weight clipping of the same MLP's three Linears, 512 sampled tokens
        dict(name='clip_mlp', kind='clip', hidden=4096, inter=11008, tokens=512, sym=False, group=128),
    ]


def _log(rng, lo, hi, step=1):
    """A size between lo and hi, spread over its logarithm, a multiple of `step`."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(step, int(round(v / step)) * step)


def draw(rng):
    kind = rng.choice(['act', 'act', 'rtn', 'rtn', 'vllm', 'awq_pack', 'blockfp8', 'gptq', 'gptq', 'awq', 'clip'])
    if kind == 'act':
        return dict(kind=kind, tokens=_log(rng, 1, 8192), cols=_log(rng, 1024, 14336, rng.choice([1, 8, 64, 128])),
                    dtype=rng.choice(['bf16', 'bf16', 'fp16']), quant=rng.choice(['int8', 'e4m3']))
    if kind == 'rtn':
        group = rng.choice([0, 32, 64, 128, 128])            # 0: one range per output channel
        return dict(kind=kind, rows=_log(rng, 64, 14336), cols=_log(rng, 512, 14336, group or rng.choice([1, 8, 128])),
                    dtype=rng.choice(['bf16', 'bf16', 'fp16', 'fp32']), bit=rng.choice([4, 8]), sym=rng.choice([True, False]),
                    group=group, mode=rng.choice(['fake', 'real', 'both', 'mse'] if group else ['fake', 'real', 'both']))
    if kind == 'vllm':
        return dict(kind=kind, linears=rng.randint(1, 24), rows=_log(rng, 256, 7168, 8), cols=_log(rng, 512, 7168, 128),
                    dtype='bf16', bit=rng.choice([4, 8]), group=rng.choice([32, 128]))
    if kind == 'awq_pack':
        return dict(kind=kind, rows=_log(rng, 256, 14336, 32), cols=_log(rng, 512, 14336, 128),
                    dtype=rng.choice(['bf16', 'fp16']), group=rng.choice([64, 128]))
    if kind == 'blockfp8':
        return dict(kind=kind, rows=_log(rng, 128, 14336), cols=_log(rng, 512, 14336, rng.choice([8, 128])))
    if kind == 'gptq':
        return dict(kind=kind, layer='one', rows=_log(rng, 128, 14336), cols=_log(rng, 512, 11008, 128),
                    batches=_log(rng, 16, 128), tokens=_log(rng, 256, 2048), dtype=rng.choice(['bf16', 'bf16', 'fp16']),
                    sym=rng.choice([True, False]), actorder=rng.choice([True, False]), group=rng.choice([64, 128]))
    if kind == 'awq':
        return dict(kind=kind, hidden=_log(rng, 1024, 4096, 128), inter=_log(rng, 2048, 11008, 128), batches=_log(rng, 4, 64),
                    tokens=512, group=rng.choice([64, 128]))
    return dict(kind='clip', hidden=_log(rng, 1024, 4096, 256), inter=_log(rng, 2048, 11008, 256), tokens=_log(rng, 128, 512),
                sym=rng.choice([True, False]), group=rng.choice([64, 128]))


# -- inputs ------------------------------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device='cuda').manual_seed(seed)


def _weight(g, rows, cols, dtype, scale=0.02):
    w = torch.randn(rows, cols, generator=g, device='cuda', dtype=torch.float32).mul_(scale)
    n = max(1, rows * cols // 1000)
    at = torch.randint(0, rows * cols, (n,), generator=g, device='cuda')
    w.view(-1)[at] *= 10.0
    return w.to(dtype)


def _acts(g, shape, dtype):
    sigma = torch.exp(torch.randn(shape[-1], generator=g, device='cuda'))
    if dtype == torch.float16:
        sigma = sigma.clamp(max=64.0)
    x = torch.randn(*shape, generator=g, device='cuda', dtype=dtype)
    return x.mul_(sigma.to(dtype))


def _linear(w):
    fc = torch.nn.utils.skip_init(torch.nn.Linear, w.shape[1], w.shape[0], bias=False, device='cuda', dtype=w.dtype)
    fc.weight = torch.nn.Parameter(w, requires_grad=False)
    return fc


class _MLP(torch.nn.Module):
    def __init__(self, gate, up, down):
        super().__init__()
        self.gate_proj, self.up_proj, self.down_proj = _linear(gate), _linear(up), _linear(down)

    def forward(self, x):
        return self.down_proj(torch.nn.functional.silu(self.gate_proj(x)) * self.up_proj(x))


# out_features, in_features and activation stream of a decoder layer's Linears; subsets in the order they are calibrated
def _decoder(case):
    h, i = case['rows'], case['cols']
    kv = h // 4
    return [[('q_proj', h, h), ('k_proj', kv, h), ('v_proj', kv, h)], [('o_proj', h, h)],
            [('gate_proj', i, h), ('up_proj', i, h)], [('down_proj', h, i)]]


def _gptq_subsets(case):
    return _decoder(case) if case['layer'] == 'decoder' else [[('fc', case['rows'], case['cols'])]]


def prepare(case, seed):
    g = _gen(seed)
    k = case['kind']
    s = {'case': case}
    if k == 'act':
        if case['quant'] == 'int8':
            act = dict(bit=8, symmetric=True, granularity='per_token')
        else:
            act = dict(quant_type='float-quant', bit='e4m3', symmetric=True, granularity='per_token', use_qtorch=True)
        s['rtn'] = RTN({'weight': dict(bit=8, symmetric=True, granularity='per_channel'), 'act': act})
        s['x'] = _acts(g, (1, case['tokens'], case['cols']), DTYPES[case['dtype']])
    elif k == 'rtn':
        kw = dict(granularity='per_group', group_size=case['group']) if case['group'] else dict(granularity='per_channel')
        if case['mode'] == 'mse':
            kw['calib_algo'] = 'mse'
        s['q'] = IntegerQuantizer(case['bit'], case['sym'], **kw)
        s['w'] = _weight(g, case['rows'], case['cols'], DTYPES[case['dtype']])
    elif k == 'vllm':
        s['rtn'] = RTN({'weight': dict(bit=case['bit'], symmetric=True, granularity='per_group', group_size=case['group'],
                                       need_pack=True)})
        s['layers'] = [_linear(_weight(g, case['rows'], case['cols'], DTYPES[case['dtype']], 0.006))
                       for _ in range(case['linears'])]
    elif k == 'awq_pack':
        s['rtn'] = RTN({'weight': dict(bit=4, symmetric=False, granularity='per_group', group_size=case['group'],
                                       pack_version='gemm_pack')})
        s['layer'] = _linear(_weight(g, case['rows'], case['cols'], DTYPES[case['dtype']]))
    elif k == 'blockfp8':
        w = _weight(g, case['rows'], case['cols'], torch.bfloat16)
        s['w8'], s['s8'] = weight_cast_to_fp8(w)
    elif k == 'gptq':
        dt = DTYPES[case['dtype']]
        s['gptq'] = GPTQ({'weight': dict(bit=4, symmetric=case['sym'], granularity='per_group', group_size=case['group']),
                          'special': dict(actorder=case['actorder'], static_groups=False, percdamp=0.01, blocksize=128,
                                          true_sequential=True)}, dt)
        s['subsets'] = []
        for linears in _gptq_subsets(case):
            weights = {n: _weight(g, r, c, dt) for n, r, c in linears}
            x = _acts(g, (case['batches'], case['tokens'], linears[0][2]), dt)
            s['subsets'].append(({n: _linear(w) for n, w in weights.items()}, weights, x))
    elif k == 'awq':
        h, i = case['hidden'], case['inter']
        s['mlp'] = _MLP(_weight(g, i, h, torch.bfloat16), _weight(g, i, h, torch.bfloat16), _weight(g, h, i, torch.bfloat16))
        s['awq'] = Awq({'weight': dict(bit=4, symmetric=False, granularity='per_group', group_size=case['group']), 'special': {}})
        s['x'] = _acts(g, (case['batches'], case['tokens'], h), torch.bfloat16)
    elif k == 'clip':
        h, i = case['hidden'], case['inter']
        s['weights'] = {'gate_proj': _weight(g, i, h, torch.bfloat16), 'up_proj': _weight(g, i, h, torch.bfloat16),
                        'down_proj': _weight(g, h, i, torch.bfloat16)}
        s['mlp'] = _MLP(**{n.split('_')[0]: w for n, w in s['weights'].items()})
        q = IntegerQuantizer(4, case['sym'], 'per_group', group_size=case['group'])
        s['clipper'] = AutoClipper(w_only=True, wquantizer=q, aquantizer=None, clip_version='v1', clip_sym=case['sym'],
                                   save_clip=False, padding_mask=None)
        x, mid = _acts(g, (1, case['tokens'], h), torch.bfloat16), _acts(g, (1, case['tokens'], i), torch.bfloat16)
        s['feats'] = {'gate_proj': [x], 'up_proj': [x], 'down_proj': [mid]}
    else:
        raise ValueError(k)
    return s


# -- one pass ----------------------------------------------------------------------------------------------------

def run(state):
    case = state['case']
    k = case['kind']
    if k == 'act':
        return state['rtn'].a_qdq(state['x'], None, state['rtn'].aquantizer)
    if k == 'rtn':
        out = {}
        if case['mode'] != 'real':
            out['fake'] = state['q'].fake_quant_weight_dynamic(state['w'])
        if case['mode'] in ('real', 'both'):
            out['codes'], out['scales'], out['zeros'] = state['q'].real_quant_weight_dynamic(state['w'])
        return out
    if k == 'vllm':
        made = [VllmRealQuantLinear.new(fc, **state['rtn'].get_replacement_params('vllm_quant')) for fc in state['layers']]
        return [(m.weight_packed, m.weight_scale) for m in made]
    if k == 'awq_pack':
        m = AutoawqRealQuantLinear.new(state['layer'], **state['rtn'].get_replacement_params('autoawq_quant'))
        return m.qweight, m.scales, m.qzeros
    if k == 'blockfp8':
        w = weight_cast_to_bf16(state['w8'], state['s8']).to(torch.bfloat16)
        return w, weight_cast_to_fp8(w)
    if k == 'gptq':
        gp, out = state['gptq'], {}
        for layers, weights, x in state['subsets']:
            for n, fc in layers.items():
                fc.weight.data = weights[n]                  # the pass before left its result here
            subset = {'layers': layers}
            gp.subset_init(subset)
            for b in range(x.shape[0]):
                for n, fc in layers.items():                 # every Linear's forward hook fires on every batch
                    gp.add_batch(fc, n, x[b:b + 1], None)
            gp.subset_transform(subset)
            for n, fc in layers.items():
                out[n] = (fc.weight.data, fc.buf_scales, None if case['sym'] else fc.buf_zeros, gp.last_errors[n])
        return out
    if k == 'awq':
        awq, mlp = state['awq'], state['mlp']
        best = awq.search_scale_subset(None, {'gate_proj': mlp.gate_proj, 'up_proj': mlp.up_proj}, [state['x']], mlp, False, {})
        return best, awq.search_losses
    mlp = state['mlp']
    for n, w in state['weights'].items():
        getattr(mlp, n).weight.data = w                      # the pass before left the clamped weight here
    state['clipper'].run(mlp, 0, {n: list(f) for n, f in state['feats'].items()}, n_sample_token=case['tokens'])
    return mlp.gate_proj.weight.data, mlp.up_proj.weight.data, mlp.down_proj.weight.data


# -- what a pass cannot do without ---------------------------------------------------------------------------------

def work(case):
    k = case['kind']
    if k == 'act':
        n = case['tokens'] * case['cols']
        return {'bytes': 2 * n * SIZE[case['dtype']], 'flops': 6 * n}
    if k == 'rtn':
        n, b = case['rows'] * case['cols'], SIZE[case['dtype']]
        qp = n // (case['group'] or case['cols']) * 2 * b
        code = 1 if case['bit'] == 8 else 4
        moved = n * b + (n * b if case['mode'] != 'real' else 0) + (n * code + qp if case['mode'] in ('real', 'both') else 0)
        return {'bytes': moved, 'flops': 80 * 10 * n if case['mode'] == 'mse' else 6 * n}
    if k == 'vllm':
        n = case['linears'] * case['rows'] * case['cols']
        return {'bytes': n * SIZE[case['dtype']] + n * case['bit'] // 8 + n // case['group'] * 2, 'flops': 6 * n}
    if k == 'awq_pack':
        n = case['rows'] * case['cols']
        return {'bytes': n * SIZE[case['dtype']] + n // 2 + n // case['group'] * 5 // 2, 'flops': 6 * n}
    if k == 'blockfp8':
        n = case['rows'] * case['cols']
        return {'bytes': n * (1 + 2 + 1), 'flops': 4 * n}
    if k == 'gptq':
        moved = flops = 0
        for linears in _gptq_subsets(case):
            c, t = linears[0][2], case['batches'] * case['tokens']
            moved += t * c * SIZE[case['dtype']] + 4 * c * c
            flops += t * c * c + c ** 3 // 3                 # the symmetric half of X^T X; one Cholesky factor
            for _, r, _ in linears:
                moved += r * c * (SIZE[case['dtype']] + 4)
                flops += r * c * c                           # every column's error meets the columns behind it
        return {'bytes': moved, 'flops': flops}
    if k == 'awq':
        h, i, t = case['hidden'], case['inter'], case['batches'] * case['tokens']
        return {'bytes': 20 * (2 * 2 * h * i * 2 + 3 * t * h * 2), 'flops': 21 * 2 * t * 3 * h * i}
    h, i, t = case['hidden'], case['inter'], case['tokens']
    return {'bytes': 2 * 3 * h * i * 2 + t * (2 * h + i) * 2, 'flops': 11 * 2 * t * 3 * h * i}


def tolerance(case):
    """Quantizer outputs are exact: every operation is rounded as torch rounds it.  The searches and GPTQ compare or
    round fp32 sums, so a sum in another order turns a decision that was a tie up to its last bits: measured with the
    path against itself (other factorization, other accumulators, sums in fp64), times about four."""
    k = case['kind']
    if k == 'rtn' and case['mode'] == 'mse':
        return {'rel': 4e-3, 'max': 0.9}                     # 8.7e-4 / 0.27: one group in 16000 takes another range
    if k == 'gptq':
        return {'rel': 4e-3, 'max': 0.5}                     # 5.5e-4 / 0.13: one zero point in 60000 rounds the other way
    if k == 'awq':
        return {'rel': 1e-3, 'max': 1e-2}                    # 1e-4 in a loss, one bf16 step in a scale
    if k == 'clip':
        return {'rel': 1e-3, 'max': 0.3}                     # a tie moves a group's range by a twentieth
    return 'exact'
