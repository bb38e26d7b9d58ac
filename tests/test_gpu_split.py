"""Float32 projections on split operands (csrc/td_gemm_split.hip) against the float64 oracle."""

import pytest
import torch

from marearts_tinydeform_amd import _native
from oracle import bruteforce
from test_gpu_parity import shifted

pytestmark = pytest.mark.gpu

# Rounding of float32 sums of K terms, each product within 2^-22 of itself: |error| <= (K + 4) 2^-24 sum |x w|; the
# largest seen is a few times smaller, as roundings cancel.
EPS = 2.0 ** -24


def problem(M, K, NO, seed=0):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(1, M, K, generator=g)
    w = torch.randn(NO, K, generator=g) / K ** 0.5
    return x, w, torch.randn(NO, generator=g)


# one row past 4500 (one step of 18 tokens a workgroup), shares that end 1 and 16 and 17 tokens into a step, many steps
@pytest.mark.parametrize('M', [4501, 8193, 12288, 12545, 33600, 67201])
@pytest.mark.parametrize('K', [128, 256])
@pytest.mark.parametrize('bias', [True, False])
def test_split_projection(M, K, bias):
    x, w, b = problem(M, K, 256)
    x[0, -1] *= 2.0 ** 40    # tokens of other scales beside the rest: the split is exact for each
    x[0, 0] *= 2.0 ** -60
    got = _native.value_proj(x.cuda(), w.cuda(), b.cuda() if bias else None).cpu().double()
    ref = torch.from_numpy(bruteforce.project(x, w, b if bias else None))
    bound = (K + 4) * EPS * (x.double().abs() @ w.double().abs().T + b.double().abs() * bias)
    assert ((got - ref).abs() <= bound).all()


@pytest.mark.parametrize('K', [128, 256])
def test_split_projection_beyond_the_split(K):
    # infinities, NaN and values whose bfloat16 rounds to infinity: what float32 arithmetic gives, and only there
    x, w, _ = problem(9001, K, 256)
    x[0, 40, 3], x[0, 41, 5], x[0, 8999, 0], x[0, 77, 1] = float('inf'), float('nan'), -float('inf'), 3.4e38
    w[7, 1] = 0.0
    got = _native.value_proj(x.cuda(), w.cuda(), None).cpu()
    ref = x @ w.T
    rows = [40, 41, 8999]
    assert torch.equal(got[0, rows].isnan(), ref[0, rows].isnan())
    assert torch.equal(got[0, rows].nan_to_num(0, 1, -1), ref[0, rows].nan_to_num(0, 1, -1))
    assert torch.allclose(got[0, 77], ref[0, 77], rtol=1e-5, atol=0) and got[0, 77, 7].abs() < 100
    keep = torch.ones(9001, dtype=torch.bool)
    keep[rows + [77]] = False
    assert torch.allclose(got[0, keep], ref[0, keep], rtol=0, atol=2e-5)
    # a weight beyond the split reaches every token
    w[9, 4] = float('inf')
    got = _native.value_proj(x.cuda(), w.cuda(), None).cpu()
    ref = x @ w.T
    assert torch.equal(got.isfinite(), ref.isfinite()) and torch.equal(got.isnan(), ref.isnan())


def test_split_input_gradient():
    # grad_memory = G . W with W as stored, from the combined entry and through the transposed copy: the same bits
    g, w, _ = problem(9001, 256, 256, 3)
    m = torch.randn(1, 9001, 256)
    gm, _, _ = _native.input_weight_grad(g.cuda(), w.cuda(), m.cuda())
    assert torch.equal(gm, _native.input_grad(g.cuda(), w.cuda()))
    bound = 260 * EPS * (g.double().abs() @ w.double().abs())
    assert ((gm.cpu().double() - g.double() @ w.double()).abs() <= bound).all()


def test_split_projection_of_unaligned_rows():
    # operands off a 16-byte boundary keep the kernels that take them
    x, w, b = problem(5000, 256, 256)
    got = _native.value_proj(shifted(x.cuda(), 4), w.cuda(), b.cuda()).cpu().double()
    ref = torch.from_numpy(bruteforce.project(x, w, b))
    assert (got - ref).abs().max() < 1e-4
