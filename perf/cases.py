"""Performance cases: the work that DETR-style models have this package do, through its public entry points.

A case is a dict of plain values:

  kind     'op'     ma_deform_attn (value projection + deformable attention, mode 'auto'), `layers` times as a decoder
                    runs it: one memory, each layer with weights, locations and attention of its own
           'layer'  MSDeformAttnLayer: the whole deformable cross-attention of a decoder layer
           'points' ma_deform_sample_v2: the D-FINE core, per-level point counts on values projected elsewhere
           'train'  ma_deform_attn_train, forward and backward, gradients for all five differentiable inputs
  dtype    'float32', 'float16' or 'bfloat16'
  B, Q, H, D, C   batch, queries, heads, head width, memory channels
  levels   the feature maps, 'HxW,HxW,...'; P: points per level ('points': points per level, 'a,b,...')
  where    'decoder': each query samples around a centre of its own; 'encoder': every token is a query (Q is unused)
           and samples around its own pixel on every level
  mask     whether images carry a padding mask
  graph    whether the program keeps the pass as a captured HIP graph, as serving loops and the benchmark do, or calls
           the entry points eagerly
"""

import torch
import torch.nn.functional as F

import marearts_tinydeform_amd as td

RTDETR = '80x80,40x40,20x20'                  # a 640 x 640 image at strides 8, 16, 32
DINO = '100x167,50x84,25x42,13x21'            # an 800 x 1333 image at strides 8 to 64
LIMIT = '128x128,64x64,32x32,16x16'           # the limit shape's maps: C = 1024, 64 samples a query and head


def _case(name, kind, dtype, B, Q, H, D, C, levels, P, where='decoder', mask=False, graph=False, layers=1):
    return {'name': name, 'kind': kind, 'dtype': dtype, 'B': B, 'Q': Q, 'H': H, 'D': D, 'C': C, 'levels': levels,
            'P': P, 'where': where, 'mask': mask, 'graph': graph, 'layers': layers}


def listed():
    return [
        # one eager call on one frame with few queries: what a call costs before there is any work to speak of
        _case('call-fp16-b1-q50', 'op', 'float16', 1, 50, 8, 32, 256, RTDETR, 4),
        # a detector's decoder on one frame, six layers replayed as one graph: single-stream serving
        _case('decoder-fp16-b1-q300', 'op', 'float16', 1, 300, 8, 32, 256, RTDETR, 4, graph=True, layers=6),
        # a large float32 batch: the reference sweep's largest size in PyTorch's default type
        _case('op-fp32-b8-q900', 'op', 'float32', 8, 900, 8, 32, 256, RTDETR, 4, graph=True),
        # the decoder-layer module as it is dropped into a model, called eagerly on an odd batch of odd-sized images
        _case('layer-bf16-b7-q300', 'layer', 'bfloat16', 7, 300, 8, 32, 256, '75x93,38x47,19x24', 4),
        # the decoder layer at four levels and 900 queries, padded batch, captured
        _case('layer-fp16-b4-q900-mask', 'layer', 'float16', 4, 900, 8, 32, 256, DINO, 4, mask=True, graph=True),
        # D-FINE's core: per-level points, values projected by the caller, eager
        _case('points-fp16-b4-q300', 'points', 'float16', 4, 300, 8, 32, 256, RTDETR, '3,6,3'),
        # an encoder layer's self-attention: every token a query
        _case('encoder-fp16-b2', 'op', 'float16', 2, 0, 8, 32, 256, DINO, 4, where='encoder', graph=True),
        # the widest shape: 1024 channels, 64 samples per query and head, compute-bound projection
        _case('op-bf16-c1024-b2-q900', 'op', 'bfloat16', 2, 900, 16, 64, 1024, LIMIT, 16, graph=True),
        # fine-tuning steps: one image in half precision, captured
        _case('train-fp16-b1-q300', 'train', 'float16', 1, 300, 8, 32, 256, RTDETR, 4, graph=True),
        # the same model in float32, PyTorch's default, on a batch, called eagerly
        _case('train-fp32-b8-q300', 'train', 'float32', 8, 300, 8, 32, 256, RTDETR, 4),
        # twelve heads of 32 and ragged five-level maps in bfloat16
        _case('train-bf16-c384-b5-q250', 'train', 'bfloat16', 5, 250, 12, 32, 384,
              '97x131,49x66,25x33,13x17,7x9', 4, graph=True),
        # an encoder layer's training step
        _case('train-encoder-fp16-b2', 'train', 'float16', 2, 0, 8, 32, 256, DINO, 4, where='encoder'),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _maps(rng, count, tokens):
    """`count` maps of a ragged image, each half the one before, about `tokens` tokens in all."""
    aspect = 0.6 + rng.random()
    h = max(3, int((tokens * 0.75 / aspect) ** 0.5))
    w = max(3, int(h * aspect))
    out = []
    for _ in range(count):
        out.append('%dx%d' % (h, w))
        h, w = (h + 1) // 2, (w + 1) // 2
    return ','.join(out)


def draw(rng):
    while True:
        kind = rng.choice(['op', 'op', 'layer', 'points', 'train', 'train'])
        where = 'encoder' if kind in ('op', 'train') and rng.random() < 0.25 else 'decoder'
        dtype = rng.choice(['float32', 'float16', 'bfloat16'])
        H, D = rng.choice([(8, 32), (8, 32), (8, 32), (4, 32), (12, 32), (16, 32), (20, 32), (8, 64), (12, 64),
                           (16, 64), (4, 16)])
        C = H * D
        B = _log_int(rng, 1, 8)
        Q = _log_int(rng, 50, 900)
        count = rng.randint(1, 5)
        levels = _maps(rng, count, _log_int(rng, 600, 22000))
        if kind == 'points':
            P = ','.join(str(rng.choice([2, 3, 4, 6])) for _ in range(count))
        else:
            P = rng.choice([4, 4, 4, 8] if count > 1 else [4, 8, 16])
        case = _case('', kind, dtype, B, 0 if where == 'encoder' else Q, H, D, C, levels, P, where,
                     mask=rng.random() < 0.3, graph=rng.random() < 0.6,
                     layers=6 if kind == 'op' and where == 'decoder' and rng.random() < 0.2 else 1)
        del case['name']
        if _cost(case) <= _LARGEST:
            return case


def _levels(case):
    return [tuple(int(n) for n in m.split('x')) for m in case['levels'].split(',')]


def _sizes(case):
    levels = _levels(case)
    N = sum(h * w for h, w in levels)
    return levels, N, N if case['where'] == 'encoder' else case['Q']


def _samples(case):
    """Samples per query and head."""
    if case['kind'] == 'points':
        return sum(int(n) for n in case['P'].split(','))
    return case['P'] * len(_levels(case))


def work(case):
    levels, N, Q = _sizes(case)
    B, H, D, C, S = case['B'], case['H'], case['D'], case['C'], _samples(case)
    s = 4 if case['dtype'] == 'float32' else 2
    HD, mask = H * D, case['B'] * N if case['mask'] else 0
    gather = 2 * 4 * B * Q * H * S * D              # four corners a sample, a multiply and an add per channel
    sampled = B * Q * H * S * 3 * s                 # locations and weights
    if case['kind'] == 'points':
        return {'bytes': B * N * HD * s + sampled + B * Q * HD * s + mask, 'flops': gather}
    proj = 2 * B * N * C * HD
    weights = (HD * C + HD) * s
    if case['kind'] == 'layer':
        heads = 3 * H * S
        moved = (B * N * C + 2 * B * Q * C + B * Q * 4 + heads * (C + 1) + HD * C + C) * s + weights + mask
        return {'bytes': moved + (B * Q * C + B * Q * H * S) * s,
                'flops': proj + gather + 2 * B * Q * C * (heads + HD)}
    if case['kind'] == 'op':
        n = case['layers']
        # projecting the sampled sums is the cheaper order where queries are few
        flops = min(proj + gather, 2 * 4 * B * Q * H * S * C + 2 * B * Q * C * HD)
        return {'bytes': B * N * C * s + n * (weights + sampled + B * Q * HD * s) + mask, 'flops': n * flops}
    # read memory, weights, samples and grad_out; write out, and a gradient the size of each input
    return {'bytes': 2 * (B * N * C * s + weights + sampled) + 2 * B * Q * HD * s + mask,
            'flops': 3 * proj + 4 * gather}


def _cost(case):
    """Work of a pass in one figure, bytes; the corner rows it gathers counted each time."""
    levels, N, Q = _sizes(case)
    w = work(case)
    s = 4 if case['dtype'] == 'float32' else 2
    rows = 4 * case['B'] * Q * case['H'] * _samples(case) * case['D'] * s * case['layers']
    return w['bytes'] + w['flops'] / 100 + rows * (3 if case['kind'] == 'train' else 1)


_LARGEST = max(_cost(c) for c in listed())

# About four times the distance from exact() that was measured, in the largest of a pass's outputs: float32 sums (which
# differ by their order only) 4e-7, float16 3.5e-4 and bfloat16 2.8e-3, where the results, and between the kernels the
# projected values and their gradients, are rounded to the type. float32 is given more for the longest sums drawn.
_TOLERANCE = {'float32': {'rel': 4e-6}, 'float16': {'rel': 1.4e-3}, 'bfloat16': {'rel': 1.2e-2}}


def tolerance(case):
    return dict(_TOLERANCE[case['dtype']])


def _generator(seed):
    return torch.Generator(device='cuda').manual_seed(seed)


def _locations(case, g):
    """Normalised sampling locations [B, Q, H, S, 2], float32, level by level, on a grid of 2^-14: a location times a
    map's width is then exact in every type it fits, and a sample's pixel does not hang on how the product rounds."""
    levels, N, Q = _sizes(case)
    B, H = case['B'], case['H']
    if case['kind'] == 'points':
        counts = [int(n) for n in case['P'].split(',')]
    else:
        counts = [case['P']] * len(levels)
    S = sum(counts)
    offset = torch.randn(B, Q, H, S, 2, generator=g, device='cuda')
    if case['where'] == 'encoder':
        centre, scale, at = [], [], 0
        for h, w in levels:
            y, x = torch.meshgrid((torch.arange(h, device='cuda') + 0.5) / h, (torch.arange(w, device='cuda') + 0.5) / w,
                                  indexing='ij')
            centre.append(torch.stack([x.flatten(), y.flatten()], -1))
        for (h, w), n in zip(levels, counts):
            scale += [[2.0 / w, 2.0 / h]] * n       # offsets of about two pixels of the level
        loc = torch.cat(centre)[None, :, None, None] + offset * torch.tensor(scale, device='cuda')
    else:
        loc = torch.rand(B, Q, 1, 1, 2, generator=g, device='cuda') + 0.05 * offset
    return (loc * 16384).round() / 16384


def _inputs(case, seed):
    """Tensors of the case by name, in its dtype, made from the seed alone."""
    levels, N, Q = _sizes(case)
    B, H, D, C, S = case['B'], case['H'], case['D'], case['C'], _samples(case)
    L, HD, g = len(levels), case['H'] * case['D'], _generator(seed)
    dtype = getattr(torch, case['dtype'])

    def randn(*shape, scale=1.0):
        return (torch.randn(*shape, generator=g, device='cuda') * scale).to(dtype)

    shapes = torch.tensor(levels, dtype=torch.long, device='cuda')
    sizes = shapes[:, 0] * shapes[:, 1]
    t = {'shapes': shapes, 'starts': torch.cat([sizes.new_zeros(1), sizes.cumsum(0)[:-1]]), 'mask': None}
    if case['mask']:                                # images padded at the right and the bottom, as batches are
        keep = 0.6 + 0.4 * torch.rand(B, 2, generator=g, device='cuda')
        keep[0] = 1.0
        parts = []
        for h, w in levels:
            y = torch.arange(h, device='cuda')[None, :, None] >= (keep[:, 0] * h).ceil()[:, None, None]
            x = torch.arange(w, device='cuda')[None, None, :] >= (keep[:, 1] * w).ceil()[:, None, None]
            parts.append((y | x).flatten(1))
        t['mask'] = torch.cat(parts, 1)
    t['memory'] = randn(B, N, C if case['kind'] != 'points' else HD)
    if case['kind'] == 'layer':
        t['hidden'], t['position'] = randn(B, Q, C), randn(B, Q, C, scale=0.5)
        box = torch.rand(B, Q, 1, 4, generator=g, device='cuda')
        t['boxes'] = torch.cat([box[..., :2], box[..., 2:] * 0.3 + 0.02], -1).to(dtype)
        t['w'] = {'sampling_offsets.weight': randn(H * S * 2, C, scale=C ** -0.5), 'sampling_offsets.bias': randn(H * S * 2),
                  'attention_weights.weight': randn(H * S, C, scale=C ** -0.5), 'attention_weights.bias': randn(H * S, scale=0.3),
                  'value_proj.weight': randn(HD, C, scale=C ** -0.5), 'value_proj.bias': randn(HD, scale=0.1),
                  'output_proj.weight': randn(C, HD, scale=HD ** -0.5), 'output_proj.bias': randn(C, scale=0.1)}
        return t
    shape = (B, Q, H, S) if case['kind'] == 'points' else (B, Q, H, L, case['P'])
    t['layers'] = []
    for _ in range(case['layers']):
        loc = _locations(case, g).to(dtype).view(*shape, 2)
        attn = torch.randn(B, Q, H, S, generator=g, device='cuda').softmax(-1).to(dtype).view(shape)
        t['layers'].append((randn(HD, C, scale=C ** -0.5), randn(HD, scale=0.1), loc, attn))
    if case['kind'] == 'train':
        t['grad'] = randn(B, Q, HD)
    return t


def _call(case, t):
    """The pass as a function of no arguments."""
    shapes, starts, mask, memory = t['shapes'], t['starts'], t['mask'], t['memory']
    if case['kind'] == 'op':
        def call():
            with torch.inference_mode():
                return [td.ma_deform_attn(memory, w, b, shapes, starts, loc, attn, padding_mask=mask)
                        for w, b, loc, attn in t['layers']]
    elif case['kind'] == 'points':
        points = [int(n) for n in case['P'].split(',')]
        _, _, loc, attn = t['layers'][0]

        def call():
            with torch.inference_mode():
                return td.ma_deform_sample_v2(memory, shapes, starts, loc, attn, points, padding_mask=mask)
    elif case['kind'] == 'layer':
        module = td.MSDeformAttnLayer(case['C'], len(_levels(case)), case['H'], case['P'])
        module.load_state_dict(t['w'])
        module = module.to('cuda', getattr(torch, case['dtype'])).eval()
        valid = None if mask is None else ~mask

        def call():
            with torch.inference_mode():
                return module(t['hidden'], valid, memory, position_embeddings=t['position'],
                              reference_points=t['boxes'], spatial_shapes=shapes, level_start_index=starts)
    else:
        w, b, loc, attn = t['layers'][0]
        inputs = [x.requires_grad_() for x in (memory, w, b, loc, attn)]

        def call():
            out = td.ma_deform_attn_train(*inputs[:3], shapes, starts, *inputs[3:], padding_mask=mask)
            return [out.detach(), *torch.autograd.grad(out, inputs, t['grad'])]
    return call


def prepare(case, seed):
    t = _inputs(case, seed)
    state = {'call': _call(case, t), 'graph': None}
    if case['graph']:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            state['call']()
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            state['out'] = state['call']()
        state['graph'] = graph
    return state


def run(state):
    if state['graph'] is not None:
        state['graph'].replay()
        return state['out']
    return state['call']()


def _sampled(value, levels, counts, loc, attn):
    """Bilinear sampling with zero padding in plain torch: value [B, N, H, D], loc [B, Q, H, S, 2], attn [B, Q, H, S]."""
    B, N, H, D = value.shape
    Q = loc.shape[1]
    maps, out, at, s = value.permute(0, 2, 3, 1).reshape(B * H, D, N), 0, 0, 0
    grid = (loc * 2 - 1).permute(0, 2, 1, 3, 4).flatten(0, 1)
    weight = attn.permute(0, 2, 1, 3).flatten(0, 1)[:, None]
    for (h, w), n in zip(levels, counts):
        part = F.grid_sample(maps[:, :, at:at + h * w].view(B * H, D, h, w), grid[:, :, s:s + n], mode='bilinear',
                             padding_mode='zeros', align_corners=False)
        out = out + (part * weight[..., s:s + n]).sum(-1)
        at, s = at + h * w, s + n
    return out.view(B, H, D, Q).permute(0, 3, 1, 2).reshape(B, Q, H * D)


def exact(case, seed):
    t = _inputs(case, seed)
    levels, N, Q = _sizes(case)
    B, H, D, S = case['B'], case['H'], case['D'], _samples(case)
    points = case['kind'] == 'points'
    counts = [int(n) for n in case['P'].split(',')] if points else [case['P']] * len(levels)

    def sampled(memory, w, b, loc, attn):
        value = memory if w is None else F.linear(memory, w, b)
        if t['mask'] is not None:
            value = value.masked_fill(t['mask'][..., None], 0)
        return _sampled(value.view(B, N, H, D), levels, counts, loc.reshape(B, Q, H, S, 2), attn.reshape(B, Q, H, S))

    memory = t['memory'].double()
    if case['kind'] == 'layer':
        w = {k: v.double() for k, v in t['w'].items()}
        x, box = t['hidden'].double() + t['position'].double(), t['boxes'].double()[:, :, None, :, None, :]
        off = F.linear(x, w['sampling_offsets.weight'], w['sampling_offsets.bias']).view(B, Q, H, len(levels), -1, 2)
        attn = F.linear(x, w['attention_weights.weight'], w['attention_weights.bias']).view(B, Q, H, S).softmax(-1)
        loc = box[..., :2] + off / case['P'] * box[..., 2:] * 0.5
        core = sampled(memory, w['value_proj.weight'], w['value_proj.bias'], loc, attn)
        return (F.linear(core, w['output_proj.weight'], w['output_proj.bias']),
                attn.view(B, Q, H, len(levels), -1))
    if points:
        _, _, loc, attn = t['layers'][0]
        return sampled(memory, None, None, loc.double(), attn.double())
    if case['kind'] == 'op':
        return [sampled(memory, *(x.double() for x in layer)) for layer in t['layers']]
    inputs = [x.requires_grad_() for x in (memory, *(x.double() for x in t['layers'][0]))]
    out = sampled(*inputs)
    return [out.detach(), *torch.autograd.grad(out, inputs, t['grad'].double())]
