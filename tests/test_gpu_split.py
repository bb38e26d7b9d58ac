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


# one step a workgroup, shares that end 1, 16 and 17 tokens into a step, many steps
@pytest.mark.parametrize('M,K', [(6401, 256), (8193, 256), (12288, 256), (12545, 256), (67201, 256), (12801, 128),
                                 (16385, 128), (33600, 128), (45057, 128)])
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
    M = 2304001 // K  # 9000 rows of 256
    x, w, _ = problem(M, K, 256)
    x[0, 40, 3], x[0, 41, 5], x[0, 8999, 0], x[0, 77, 1] = float('inf'), float('nan'), -float('inf'), 3.4e38
    w[7, 1] = 0.0
    got = _native.value_proj(x.cuda(), w.cuda(), None).cpu()
    ref = x @ w.T
    rows = [40, 41, 8999]
    assert torch.equal(got[0, rows].isnan(), ref[0, rows].isnan())
    assert torch.equal(got[0, rows].nan_to_num(0, 1, -1), ref[0, rows].nan_to_num(0, 1, -1))
    assert torch.allclose(got[0, 77], ref[0, 77], rtol=1e-5, atol=0) and got[0, 77, 7].abs() < 100
    keep = torch.ones(M, dtype=torch.bool)
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
    x, w, b = problem(7000, 256, 256)
    got = _native.value_proj(shifted(x.cuda(), 4), w.cuda(), b.cuda()).cpu().double()
    ref = torch.from_numpy(bruteforce.project(x, w, b))
    assert (got - ref).abs().max() < 1e-4


# tiles cut on both sides, one partial split, many; bias in the last, partial, tile of columns; up to 128 columns on
# both sides of the line that those have for themselves
@pytest.mark.parametrize('M,NO,K', [(6401, 256, 256), (20011, 256, 128), (4801, 384, 384), (9001, 100, 260),
                                    (16003, 132, 200), (2048, 64, 1024), (20003, 100, 260), (5003, 64, 1024),
                                    (12800, 128, 256)])
def test_split_weight_gradient(M, NO, K):
    gen = torch.Generator().manual_seed(1)
    G, X = torch.randn(1, M, NO, generator=gen), torch.randn(1, M, K, generator=gen)
    gw, gb = _native.weight_grad(G.cuda(), X.cuda())
    G64, X64 = G[0].double(), X[0].double()
    # sums over M tokens in splits: the largest sum's roundings, as above
    assert ((gw.cpu().double() - G64.T @ X64).abs() <= M ** 0.5 * 8 * EPS * (G64.abs().T @ X64.abs()) / M ** 0.5).all()
    assert ((gb.cpu().double() - G64.sum(0)).abs() <= 64 * EPS * G64.abs().sum(0)).all()


def test_split_weight_gradient_beyond_the_split():
    G, X = torch.randn(1, 8192, 256), torch.randn(1, 8192, 256)
    G[0, 5, 7], X[0, 900, 3], G[0, 3000, 9] = float('inf'), float('nan'), 3.3e38
    gw, _ = _native.weight_grad(G.cuda(), X.cuda())
    gw = gw.cpu()
    ref = G[0].double().T @ X[0].double()
    assert gw[:, 3].isnan().all() and not gw[:7, [0, 1, 2]].isnan().any()
    rest = [c for c in range(256) if c != 3]
    assert torch.equal(gw[7, rest], torch.full((255,), float('inf')) * X[0, 5, rest].sign())
    over = ref[9, rest].abs() > 3.4e38
    assert torch.equal(gw[9, rest].isinf(), over) or ((gw[9, rest].isinf() == over) | (ref[9, rest].abs() > 3.39e38)).all()
    assert torch.allclose(gw[10:, rest].double(), ref[10:, rest], rtol=0, atol=2e-3)


# operands whose third and second parts fall under bfloat16's smallest subnormal: every bit of them still counts
@pytest.mark.parametrize('scale', [-100, -112, -120, -126])
@pytest.mark.parametrize('K', [128, 256])
def test_split_projection_of_small_values(scale, K):
    M = 2304001 // K
    x, w, _ = problem(M, K, 256)
    small = torch.zeros(M, dtype=torch.bool)
    small[[0, 70, M - 1]] = small[4000:4100] = True
    x[0, small] = (1 + x[0, small].abs()) * 2.0 ** scale
    w *= 2.0 ** 40
    got = _native.value_proj(x.cuda(), w.cuda(), None).cpu().double()
    ref = x.double() @ w.double().T
    assert ((got - ref).abs() <= (K + 4) * EPS * (x.double().abs() @ w.double().abs().T)).all()
    # small weights, and the input gradient, which reads them as stored
    x, w, _ = problem(M, K, 256, seed=1)
    x, w = x * 2.0 ** 40, (1 + w.abs()) * 2.0 ** scale
    got = _native.value_proj(x.cuda(), w.cuda(), None).cpu().double()
    ref = x.double() @ w.double().T
    assert ((got - ref).abs() <= (K + 4) * EPS * (x.double().abs() @ w.double().abs().T)).all()
    if K == 256:
        gm, _, _ = _native.input_weight_grad(x.cuda(), w.cuda(), x.cuda())
        ref = x.double() @ w.double()
        assert ((gm.cpu().double() - ref).abs() <= (K + 4) * EPS * (x.double().abs() @ w.double().abs())).all()


@pytest.mark.parametrize('scale', [-100, -112, -120, -126])
def test_split_weight_gradient_of_small_values(scale):
    M = 8193
    gen = torch.Generator().manual_seed(2)
    G, X = torch.randn(1, M, 256, generator=gen), torch.randn(1, M, 200, generator=gen) * 2.0 ** 40
    G[0] = (1 + G[0].abs()) * 2.0 ** scale
    gw, gb = _native.weight_grad(G.cuda(), X.cuda())
    G64, X64 = G[0].double(), X[0].double()
    assert ((gw.cpu().double() - G64.T @ X64).abs() <= 8 * EPS * (G64.abs().T @ X64.abs())).all()
    G = torch.randn(1, M, 256, generator=gen) * 2.0 ** 40
    X = (1 + torch.randn(1, M, 200, generator=gen).abs()) * 2.0 ** scale
    gw, _ = _native.weight_grad(G.cuda(), X.cuda())
    G64, X64 = G[0].double(), X[0].double()
    assert ((gw.cpu().double() - G64.T @ X64).abs() <= 8 * EPS * (G64.abs().T @ X64.abs())).all()
