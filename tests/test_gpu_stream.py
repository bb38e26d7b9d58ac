"""The streaming 16-bit projection at 384 channels (csrc/td_gemm_stream.hip) against the float64 oracle."""

import pytest
import torch

from marearts_tinydeform_amd import _native
from oracle import bruteforce
from test_gpu_parity import GEMM_EPS, assert_close, heads_of

pytestmark = pytest.mark.gpu


# shares of 42 or 43 tokens (a second step of 10 or 11), one past, whole steps, many steps off the step size
@pytest.mark.parametrize('M', [10881, 11009, 16384, 36001, 70003])
@pytest.mark.parametrize('bias', [True, False])
@pytest.mark.parametrize('dtype', [torch.float16, torch.bfloat16])
def test_streaming_384(M, bias, dtype):
    g = torch.Generator().manual_seed(M)
    x = torch.randn(1, M, 384, generator=g).to(dtype)
    w = (torch.randn(384, 384, generator=g) / 384 ** 0.5).to(dtype)
    b = (torch.randn(384, generator=g) * 0.1).to(dtype) if bias else None
    assert _native.value_proj_plan(dtype, M, 384, 384, bias=bias) == 22
    got = _native.value_proj(x.cuda(), w.cuda(), None if b is None else b.cuda()).cpu()
    assert_close(f'stream 384 {dtype} {M}', got, bruteforce.project(x, w, b), GEMM_EPS[dtype], GEMM_EPS[dtype])


@pytest.mark.parametrize('dtype', [torch.float16, torch.bfloat16])
def test_streaming_384_heads_and_input_gradient(dtype):
    g = torch.Generator().manual_seed(1)
    x = torch.randn(3, 5003, 384, generator=g).to(dtype)
    w = (torch.randn(384, 384, generator=g) / 384 ** 0.5).to(dtype)
    b = (torch.randn(384, generator=g) * 0.1).to(dtype)
    assert _native.value_proj_plan(dtype, 3 * 5003, 384, 384, heads=12, N=5003) == 22
    got = _native.value_proj_heads(x.cuda(), w.cuda(), b.cuda(), 12).cpu()
    assert_close(f'heads 384 {dtype}', got, heads_of(bruteforce.project(x, w, b), 12), GEMM_EPS[dtype], GEMM_EPS[dtype])
    # W as stored, from the combined entry, and through the transposed copy: the same bits
    gm, _, _ = _native.input_weight_grad(x.cuda(), w.cuda(), x.cuda())
    assert torch.equal(gm, _native.input_grad(x.cuda(), w.cuda()))


def test_streaming_384_needs_aligned_operands():
    for k in ('memory', 'weight', 'value', 'bias'):
        assert _native.value_proj_plan(torch.float16, 20000, 384, 384, offsets={k: 8}) != 22
