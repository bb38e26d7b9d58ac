"""The decoder layer's query prologue on both sides of its size rule (csrc/td_layer.hip, launch_prologue)."""

import pytest
import torch

from inputs import make_layer
from marearts_tinydeform_amd import _native
from marearts_tinydeform_amd.reference import layer_locations_reference

pytestmark = pytest.mark.gpu


# below 1.2e8 multiply-adds (one kernel); above, finalized by the projections (16 samples), ragged rows, no position
# embeddings; with 12 samples, finalized apart, on both sides of 2e8; above with channels the two projections' launch does
# not take
@pytest.mark.parametrize('B,Q,C,H,L,P,pos', [(1, 900, 256, 8, 4, 4, True), (3, 417, 256, 8, 4, 4, True),
                                             (3, 567, 256, 8, 3, 4, True), (3, 967, 256, 8, 3, 4, True),
                                             (2, 331, 384, 12, 4, 4, False), (3, 500, 264, 8, 4, 4, True)])
@pytest.mark.parametrize('dtype', [torch.float16, torch.bfloat16])
def test_prologue_matches_float64(B, Q, C, H, L, P, pos, dtype):
    levels = [(40 >> l, 56 >> l) for l in range(L)]
    a = make_layer(B, Q, H, 32, C, levels, P, dtype=dtype, pos=pos, seed=3)
    hidden, memory, ref, shapes, starts, ow, ob, aw, ab = a[:9]
    position = a[-1]
    dev = [None if t is None else t.cuda() for t in (hidden, position, ref, ow, ob, aw, ab, shapes)]
    loc, attn = _native.layer_prologue(*dev, H, P)
    want_loc, want_attn = layer_locations_reference(
        hidden.double(), ref.double(), shapes, ow.double(), ob.double(), aw.double(), ab.double(), H, P,
        None if position is None else position.double())
    # float32 sums of C products of order 1 / sqrt(C), twice with position embeddings, and expf
    assert (loc.cpu().double() - want_loc).abs().max() < 2e-5
    assert (attn.cpu().double() - want_attn).abs().max() < 1e-5
