"""Gradients where the levels do not tile the tokens: level_start_index is an argument, and tokens that lie in no level,
tokens that two levels share and levels that reach past the tokens are all forms the forward takes."""

import pytest
import torch

from inputs import workload
from oracle import gridsample
from test_gpu_backward import NAMES, check, gpu_grads, grad_out_for

pytestmark = pytest.mark.gpu


def placed(kind, levels):
    """Where the levels lie: (first token of each, tokens in all)."""
    size = [h * w for h, w in levels]
    starts = [sum(size[:l]) for l in range(len(size))]
    total = sum(size)
    if kind == 'tiled':
        return starts, total
    if kind == 'gaps':          # tokens before, between and after the levels that belong to none
        return [s + 3 + 5 * l for l, s in enumerate(starts)], total + 5 * len(size) + 4
    if kind == 'after':         # as a model with a few extra tokens at the end
        return starts, total + 4
    if kind == 'reversed':      # all tokens covered, in another order
        return [total - s - n for s, n in zip(starts, size)], total
    if kind == 'shared':        # every level begins in the one before it
        return [s - 7 * l for l, s in enumerate(starts)], total - 7 * (len(size) - 1)
    if kind == 'same':          # all levels on the first one's tokens, and tokens after it
        return [0] * len(size), size[0] + 11
    assert kind == 'outside'    # the first level begins before the tokens, the last ends after them
    return [s - 9 for s in starts], total - 9 - 13


KINDS = ('gaps', 'after', 'reversed', 'shared', 'same', 'outside')


def compare(kind, B, Q, H, D, levels, P, dtype, where, masked=False):
    """The gradients against the oracle's; Q None: as many queries as tokens. The oracle slices whole levels, so it
    gets the tokens with padded ones before and after."""
    starts, N = placed(kind, levels)
    before = max(0, -min(starts))
    after = max(0, max(s + h * w for s, (h, w) in zip(starts, levels)) - N)
    Q = N if Q is None else Q
    args = workload(B, Q, H, D, 32, levels, P, dtype, loc_dist=where, seed=6)
    gen = torch.Generator().manual_seed(8)
    args[0] = torch.randn(B, N, 32, generator=gen).to(dtype)
    args[4] = torch.tensor(starts)
    args[5] = (args[5].float() * 1024).round().div(1024).to(dtype)     # pixels that do not hang on how a product rounds
    mask = torch.rand(B, N, generator=gen) < 0.2 if masked else None
    go = grad_out_for(args)
    torch.use_deterministic_algorithms(True)    # with it, torch.empty fills what it gives with NaN
    try:
        grads, _ = gpu_grads(args, go, dtype, mask=mask)
    finally:
        torch.use_deterministic_algorithms(False)
    padded = [torch.nn.functional.pad(args[0], (0, 0, before, after))] + args[1:]
    padded[4] = args[4] + before
    keep = torch.zeros(B, N, dtype=torch.bool) if mask is None else mask
    ref = gridsample.deform_attn_grads(*padded, go.to(dtype),
                                       padding_mask=torch.nn.functional.pad(keep, (before, after), value=True))
    ref['memory'] = ref['memory'][:, before:before + N]
    for n in NAMES:
        check(f'{kind} {B}x{Q}x{H}x{D} {dtype} d{n}', grads[n], ref[n], dtype)
    lonely = torch.ones(N, dtype=torch.bool)
    for s, (h, w) in zip(starts, levels):
        lonely[max(s, 0):s + h * w] = False
    assert not grads['memory'][:, lonely.cuda()].any()      # exactly zero where no level lies


@pytest.mark.parametrize('kind', KINDS)
@pytest.mark.parametrize('dtype', [torch.float32, torch.float16, torch.bfloat16])
def test_decoder_gradients(kind, dtype):
    # 2^18 corners and more: the binned value gradient. A hot spot makes split bins
    compare(kind, 2, 350, 8, 32, [(40, 60), (20, 30), (10, 15)], 4, dtype, 'uniform')
    compare(kind, 2, 350, 8, 16, [(40, 60), (20, 30), (10, 15)], 4, dtype, 'clustered', masked=True)
    compare(kind, 3, 300, 8, 8, [(60, 80), (30, 40), (15, 20)], 4, dtype, 'clustered')


@pytest.mark.parametrize('kind', KINDS)
@pytest.mark.parametrize('dtype', [torch.float32, torch.float16])
def test_self_attention_gradients(kind, dtype):
    # as many queries as tokens: a query counts once whether its token lies in no level, one or two. 32768 rows and more,
    # then under them
    compare(kind, 6, None, 4, 64, [(33, 49), (21, 35)], 4, dtype, 'encoder')
    compare(kind, 7, None, 5, 32, [(29, 40), (24, 31)], 4, dtype, 'encoder', masked=True)
    compare(kind, 2, None, 8, 32, [(29, 40), (12, 16)], 4, dtype, 'encoder')


def test_self_attention_gradients_large_tiles():
    # the 16-bit form from 131072 rows
    for kind in ('gaps', 'shared', 'same'):
        compare(kind, 4, None, 8, 32, [(55, 85), (28, 36), (14, 15)], 4, torch.bfloat16, 'encoder', masked=kind == 'gaps')


@pytest.mark.parametrize('kind', (*KINDS, 'tiled'))
def test_self_attention_gradients_of_narrow_heads(kind):
    # four channels a head: 8 x 4-pixel tiles of the bucketed scatter; windows that fit and that do not
    for where in ('encoder', 'uniform'):
        compare(kind, 2, None, 3, 4, [(33, 49), (21, 35), (3, 5)], 4, torch.float32, where, masked=where == 'uniform')
    compare(kind, 1, None, 2, 4, [(6, 9)], 8, torch.float32, 'encoder')
