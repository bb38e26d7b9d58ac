"""The self-attention value-gradient scatter by query tiles (csrc/td_backward.hip, scatter_tile_kernel)."""

import pytest
import torch

from inputs import workload
from marearts_tinydeform_amd import _native
from oracle import gridsample
from test_gpu_backward import NAMES, check, gpu_grads, grad_out_for

pytestmark = pytest.mark.gpu

# B, H, D, P, levels: 16 x 16 tiles (131072 rows and more, 1024 threads) with maps that end inside a tile; 16 x 8, and
# by P or D 8 x 8 and 8 x 4; five levels (the samples of four are loaded together); one map smaller than a tile
SHAPES = [
    (4, 8, 32, 4, [(55, 57), (28, 29), (14, 15)]),
    (2, 8, 64, 8, [(65, 67), (61, 66)]),
    (4, 4, 32, 4, [(33, 49), (17, 25), (9, 13), (5, 7), (3, 4)]),
    (8, 3, 64, 4, [(31, 47), (16, 24)]),
    (6, 6, 16, 16, [(24, 39)]),
    (8, 8, 8, 2, [(25, 15), (40, 5)]),
    (1, 2, 32, 4, [(31, 47), (16, 24)]),    # consecutive queries
    (2, 8, 32, 4, [(31, 37), (16, 19)]),    # from 16000 rows (20000 under 32 channels) to 32768: 8 x 4 tiles
    (2, 8, 8, 8, [(31, 37), (16, 19)]),
]


@pytest.mark.parametrize('shape', SHAPES)
@pytest.mark.parametrize('dtype', [torch.float16, torch.bfloat16])
def test_tile_scatter(shape, dtype):
    B, H, D, P, levels = shape
    N = sum(h * w for h, w in levels)
    args = workload(B, N, H, D, 64, levels, P, dtype, loc_dist='encoder', seed=5)
    loc = args[5]
    loc[:, ::7, :, :, 0] = 0.5              # many corners in one pixel, far from most of their tiles
    loc[:, 3::11, :, :, -1] += 3.0          # outside the map
    loc[:, 5::13, :, :, -1] = float('nan')
    go = grad_out_for(args)
    grads, _ = gpu_grads(args, go, dtype)
    loc64 = loc.clone()
    loc64[loc64.isnan()] = -9.0             # nothing, as a location outside
    args[5] = loc64
    ref = gridsample.deform_attn_grads(*args, go.to(dtype))
    for n in NAMES:
        check(f'tiles {shape} {dtype} d{n}', grads[n], ref[n], dtype)


# 16 x 16, 16 x 8 and 8 x 4 tiles and consecutive queries: in float32 (which has no 16 x 16), with padded tokens in and
# outside the windows, and with locations all over the map, whose corners are mostly added directly
@pytest.mark.parametrize('shape', [SHAPES[0], SHAPES[2], SHAPES[4], SHAPES[7], SHAPES[6]])
@pytest.mark.parametrize('dtype', [torch.float32, torch.float16])
@pytest.mark.parametrize('masked', [False, True])
def test_tile_scatter_masked_and_far(shape, dtype, masked):
    B, H, D, P, levels = shape
    N = sum(h * w for h, w in levels)
    mask = torch.rand(B, N, generator=torch.Generator().manual_seed(3)) < 0.25 if masked else None
    for where in ('encoder', 'uniform'):
        args = workload(B, N, H, D, 64, levels, P, dtype, loc_dist=where, seed=7)
        args[5] = (args[5].float() * 1024).round().div(1024).to(dtype)     # pixels that do not hang on rounding
        go = grad_out_for(args)
        grads, _ = gpu_grads(args, go, dtype, mask=mask)
        ref = gridsample.deform_attn_grads(*args, go.to(dtype), padding_mask=mask)
        for n in NAMES:
            check(f'tiles {shape} {dtype} {where} masked={masked} d{n}', grads[n], ref[n], dtype)


def test_tile_scatter_keeps_infinities_where_they_belong():
    # an infinite grad_out row reaches the pixels it samples and no other, in float16 too
    levels = [(80, 100), (40, 50)]
    N = sum(h * w for h, w in levels)
    args = workload(1, N, 4, 32, 128, levels, 4, torch.float16, loc_dist='encoder', seed=2)
    # corners of non-zero weight only (0 times infinity is NaN, here as anywhere)
    args[5][0, 100] = torch.linspace(0.2131, 0.4377, 4 * 2 * 4 * 2).view(4, 2, 4, 2).half()
    for l, (h, w) in enumerate(levels):
        pix = args[5][0, 100, :, l].float() * torch.tensor([w, h]) - 0.5
        args[5][0, 100, :, l] += (pix == pix.floor()).half() * 0.001    # off the pixel centres
        pix = args[5][0, 100, :, l].float() * torch.tensor([w, h]) - 0.5
        assert (pix != pix.floor()).all()
    value = torch.randn(1, N, 128, generator=torch.Generator().manual_seed(1)).half()
    go = torch.ones(1, N, 128).half()
    go[0, 100, :32] = float('inf')          # head 0 of query 100
    dev = [t.cuda() for t in (value, args[3], args[4], args[5], args[6])]
    gv, _, _ = _native.sample_backward(dev[0], 4, dev[1], dev[2], dev[3], dev[4], go.cuda())
    bad = (~gv.isfinite()).any(-1)[0].cpu()
    assert torch.isfinite(gv[0, :, 32:]).all()
    go[0, 100, :32] = 0
    go[0, :100] = 0
    go[0, 101:] = 0
    go[0, 100, :32] = 1
    alone, _, _ = _native.sample_backward(dev[0], 4, dev[1], dev[2], dev[3], dev[4], go.cuda())
    hit = (alone[0, :, :32] != 0).any(-1).cpu()
    assert hit.any() and bool((bad == hit).all())


@pytest.mark.parametrize('D', [8, 16, 32, 64])
@pytest.mark.parametrize('masked', [False, True])
def test_binned_float32_value_gradient(D, masked):
    # the decoders' binned value gradient in float32 (2^18 corners and more), hot spots and uniform locations in turn;
    # and with the accumulator kept, which holds the gradient as it always did
    levels, B, Q, H, P = [(40, 60), (20, 30), (10, 15)], 2, 350, 8, 4
    N = sum(h * w for h, w in levels)
    for where in ('clustered', 'uniform'):
        args = workload(B, Q, H, D, 64, levels, P, torch.float32, loc_dist=where, seed=4)
        args[5] = (args[5] * 4096).round() / 4096     # pixels that do not hang on how a product rounds
        mask = torch.rand(B, N, generator=torch.Generator().manual_seed(4)) < 0.3 if masked else None
        go = grad_out_for(args)
        grads, _ = gpu_grads(args, go, torch.float32, mask=mask)
        ref = gridsample.deform_attn_grads(*args, go, padding_mask=mask)
        for n in NAMES:
            check(f'binned float32 D={D} {where} d{n}', grads[n], ref[n], torch.float32)
    value = torch.randn(B, N, H * D).cuda()
    shapes, starts, loc, attn, go = (t.cuda() for t in (args[3], args[4], args[5], args[6], go))
    gv, gl, ga = _native.sample_backward(value, H, shapes, starts, loc, attn, go)
    acc, out = torch.empty_like(value), torch.empty_like(value)
    gl2, ga2 = torch.empty_like(loc), torch.empty_like(attn)
    rc = _native.lib.td_sample_backward(0, value.data_ptr(), shapes.data_ptr(), starts.data_ptr(), loc.data_ptr(),
                                        attn.data_ptr(), None, go.data_ptr(), acc.data_ptr(), out.data_ptr(),
                                        gl2.data_ptr(), ga2.data_ptr(), B, Q, N, H, D, len(levels), P,
                                        torch.cuda.current_stream().cuda_stream)
    assert rc == 0 and torch.equal(acc, out)
    assert torch.allclose(gv, acc, rtol=1e-4, atol=1e-4) and torch.allclose(ga, ga2, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize('D,binned', [(32, True), (24, False), (128, False)])
def test_float32_decoders_second_buffer(D, binned):
    # a float32 value gradient takes a second buffer of its size only where its sums are binned
    levels, B, Q, H, P = [(40, 60), (20, 30), (10, 15)], 2, 350, 8, 4
    N = sum(h * w for h, w in levels)
    args = [t.cuda() for t in workload(B, Q, H, D, 8, levels, P, torch.float32)[3:7]]
    value, go = torch.randn(B, N, H * D, device='cuda'), torch.randn(B, Q, H * D, device='cuda')
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    grads = _native.sample_backward(value, H, *args, go)
    size = value.numel() * 4
    extra = torch.cuda.max_memory_allocated() - before - sum(t.numel() * 4 for t in grads)
    assert (extra >= size) if binned else extra < size // 2
