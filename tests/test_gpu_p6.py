"""The VQ4P int8-table kernels where their tiles end: widths that leave a
partial group of 4 positions, a partial block of 32 and a partial row block,
tables of several LDS passes, jobs of 1 to 8 tokens, and launches with one
and with four row blocks per block. A matvec is bit for bit the oracle's
(integer sums and a fixed order of fp32 folds); layers meet the 1e-4 bar.
"""
import ctypes

import numpy as np
import pytest

import container as ct
from gpu_util import BALANCED, dev, empty, host, open_ctx, rel_err
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def model_of(hidden, inter, experts=6, top_k=3):
    return ct.build(ct.Spec(hidden=hidden, inter=inter, experts=experts, top_k=top_k, layers=1, fmt="VQ4P",
                            shared_bits=0, seed=hidden + inter, keep_codes=False, **BALANCED))


@pytest.mark.parametrize("hidden,inter", [(8, 8), (264, 72), (328, 200), (2080, 136), (4104, 64)])
def test_matvec_bits(hidden, inter):
    import warp_amd
    model = model_of(hidden, inter)
    ctx = open_ctx(model)
    try:
        warp_amd.load_container_model(ctx, model)
        bT = po.books_T(model.books_raw)
        rng = np.random.default_rng(hidden)
        for e in (0, 5):
            raw = model.layers[0].records[e]
            r, hdr = np.frombuffer(raw, np.uint8), np.frombuffer(raw[:48], np.uint32)
            for kind in range(3):
                M, N = (inter, hidden) if kind < 2 else (hidden, inter)
                x, y = rng.normal(size=N).astype(np.float32), empty(M)
                ctx.vq_matvec(0, kind, ctx.resident(0, e), dev(x), y)
                at = int(hdr[8]) + 2 * (0, inter, 2 * inter)[kind]
                scale = r[at:at + 2 * M].view(np.uint16).copy()
                ref = po.vq_matvec("VQ4P", r[int(hdr[5 + kind]):].copy(), scale, x, bT, kind * 4, M, N)
                assert np.array_equal(host(y), ref), (e, kind)
    finally:
        ctx.close()


@pytest.mark.parametrize("shift", [1, 2, 3])
def test_matvec_index_blocks_at_any_byte(shift):
    """A record's header may put its index blocks at any byte; the code words
    are read four bytes at a time."""
    import warp_amd
    hidden, inter = 328, 200
    model = model_of(hidden, inter)
    ctx = open_ctx(model)
    try:
        warp_amd.load_container_model(ctx, model)
        bT = po.books_T(model.books_raw)
        raw = model.layers[0].records[5]
        r, hdr = np.frombuffer(raw, np.uint8), np.frombuffer(raw[:48], np.uint32)
        off = [int(v) for v in hdr[5:9]]
        rows = 2 * (2 * inter + hidden)
        moved, at = np.zeros_like(r), []
        for k, (a, e) in enumerate(zip(off, off[1:] + [off[3] + rows])):
            at.append(a + (4 * k + 4 + shift if k < 3 else 16))
            moved[at[k]:at[k] + e - a] = r[a:e]
        moved[:48] = r[:48]
        moved[20:36] = np.array(at, np.uint32).view(np.uint8)
        rec = dev(moved)
        rng = np.random.default_rng(shift)
        for kind in range(3):
            M, N = (inter, hidden) if kind < 2 else (hidden, inter)
            x, y = rng.normal(size=N).astype(np.float32), empty(M)
            ctx.vq_matvec(0, kind, rec, dev(x), y)
            s0 = off[3] + 2 * (0, inter, 2 * inter)[kind]
            ref = po.vq_matvec("VQ4P", r[off[kind]:].copy(), r[s0:s0 + 2 * M].view(np.uint16).copy(), x, bT, kind * 4,
                               M, N)
            assert np.array_equal(host(y), ref), kind
    finally:
        ctx.close()


@pytest.mark.parametrize("hidden,inter,experts,T", [(328, 200, 6, 1), (328, 200, 6, 5), (328, 200, 6, 23),
                                                    (264, 520, 40, 150), (2080, 136, 6, 37)])
def test_chunk_jobs(hidden, inter, experts, T):
    """Launches with one row block per block (few jobs, or few row blocks)."""
    import warp_amd
    model = model_of(hidden, inter, experts)
    ctx = open_ctx(model, max_tokens=T)
    try:
        warp_amd.load_container_model(ctx, model)
        X = np.random.default_rng(T).normal(size=(T, hidden)).astype(np.float32)
        out = empty((T, hidden))
        ctx.moe_chunk(0, dev(X), out, T)
        ctx.sync()
        ref = po.LayerView(model, 0).moe_chunk(X)[0]
        assert rel_err(host(out), ref) <= 1e-4
    finally:
        ctx.close()


@pytest.mark.parametrize("hidden,inter,T", [(264, 712, 150), (264, 840, 150), (1416, 728, 151)])
def test_chunk_four_row_blocks(hidden, inter, T):
    """Launches with four row blocks per block: gate and up of 12 and of 14
    row blocks (the last group partial), and at 1416 the down rows' 23 too.
    The jobs hold 1, 2, 3 to 4 and 5 to 8 tokens, a kernel loop each."""
    import warp_amd
    from warp_amd.device import rt
    experts, top_k = 40, 3
    n = ctypes.c_int()
    assert rt().hipDeviceGetAttribute(ctypes.byref(n), 63, 0) == 0 and n.value > 0     # multiprocessor count
    n_cu = n.value
    jobs = min(T * top_k, T * top_k // 8 + experts + 1)     # the most that a list holds
    blocks = lambda M: (M + 63) // 64
    assert jobs * 2 * blocks(inter) >= 8 * n_cu and (hidden < 1416 or jobs * blocks(hidden) >= 8 * n_cu)
    model = model_of(hidden, inter, experts, top_k)
    ctx = open_ctx(model, max_tokens=T)
    try:
        warp_amd.load_container_model(ctx, model)
        X = np.random.default_rng(T).normal(size=(T, hidden)).astype(np.float32)
        out, route, _ = ctx.moe_chunk_host(0, X)
        counts = np.bincount(route.ravel(), minlength=experts)
        sizes = set(int(n) for c in counts for n in [8] * (c // 8) + [c % 8])
        assert {1, 2, 8} <= sizes and sizes & {3, 4}, sizes
        ref = po.LayerView(model, 0).moe_chunk(X)[0]
        assert rel_err(out, ref) <= 1e-4
    finally:
        ctx.close()
