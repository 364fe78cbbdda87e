"""The shared expert's hidden state made in one launch (gate and up rows taken
in turn by one wave) where no other launch makes it: chunks under 8 tokens,
against the oracle's moe_chunk. One and two row pairs per wave, up to four
16-byte chunks per lane (the real K3 shape covers eight), both widths of weights.

Bar: 1e-4 of max|ref|, the exact mode's; the sums are fp32 over at most 2304
inputs.
"""
import numpy as np
import pytest

import container as ct
from gpu_util import BALANCED, open_ctx, rel_err
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits,group,hidden,inter,n_shared", [
    (8, 32, 256, 64, 1), (8, 32, 2304, 96, 1), (4, 128, 256, 128, 3), (8, 64, 128, 1088, 4), (4, 32, 128, 1056, 4),
    (8, 32, 160, 96, 1), (4, 32, 2304, 64, 1)])
def test_shared_hidden_state(bits, group, hidden, inter, n_shared):
    import warp_amd
    spec = ct.Spec(hidden=hidden, inter=inter, experts=4, top_k=2, layers=1, fmt="VQ2R", seed=bits * hidden + inter,
                   shared_bits=bits, shared_group=group, n_shared=n_shared, subnormals=False, keep_codes=False,
                   act="situ" if group == 64 else "silu", **BALANCED)
    model = ct.build(spec)
    X = np.random.default_rng(43).normal(size=(7, hidden)).astype(np.float32)
    ctx = open_ctx(model, max_tokens=7)
    try:
        warp_amd.load_container_model(ctx, model)
        for T in (1, 3, 7):
            out, route, _ = ctx.moe_chunk_host(0, X[:T])
            ro, rr, _ = po.LayerView(model, 0).moe_chunk(X[:T])
            assert np.array_equal(route, rr)
            assert rel_err(out, ro) <= 1e-4, (T, rel_err(out, ro))
    finally:
        ctx.close()
