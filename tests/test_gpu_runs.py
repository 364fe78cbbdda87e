"""Prefill by runs at the edges of its jobs and loops, against the oracle's
moe_chunk through the C ABI: three experts and top-2, so that an expert's
tokens fill one job, one job and a bit, a run of two jobs (exact products), a
run of four (reduced precision) and more; positions that are fewer than a
loop's loads in flight, or leave every remainder of them; whole and partial
64-row blocks; a unit or two for the whole launch.

Bars: 1e-4 of max|ref| for exact products (x carries 22 bits, sums are fp32
over at most 352 inputs: about 1e-6) and 2e-3 for reduced precision (2^-11
per rounded value).
"""
import numpy as np
import pytest

import container as ct
from gpu_util import BALANCED, open_ctx, rel_err
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp16", [False, True])
@pytest.mark.parametrize("fmt", ["VQ3R", "VQ2R", "VQ12"])
@pytest.mark.parametrize("hidden,inter", [(352, 224), (128, 64), (64, 320)])
def test_runs_at_job_edges(fmt, hidden, inter, fp16):
    import warp_amd
    spec = ct.Spec(hidden=hidden, inter=inter, experts=3, top_k=2, layers=1, fmt=fmt, seed=hidden + inter,
                   subnormals=False, keep_codes=False, **{**BALANCED, "shared_bits": 0})
    model = ct.build(spec)
    X = np.random.default_rng(41).normal(size=(97, hidden)).astype(np.float32)
    ctx = open_ctx(model, max_tokens=len(X), prefill_fp16=fp16)
    try:
        warp_amd.load_container_model(ctx, model)
        seen = set()
        for T in (1, 2, 12, 13, 25, 50, 97):
            out, route, _ = ctx.moe_chunk_host(0, X[:T])
            ro, rr, _ = po.LayerView(model, 0).moe_chunk(X[:T])
            assert np.array_equal(route, rr)
            e = rel_err(out, ro)
            assert e <= (2e-3 if fp16 else 1e-4), (T, e)
            seen.update((np.bincount(route.ravel(), minlength=3) + 7) // 8)
        assert {1, 2, 3} <= seen and max(seen) > 4, seen
    finally:
        ctx.close()
