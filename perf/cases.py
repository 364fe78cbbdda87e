"""The workloads whose speed this library is measured by.

Each case is a dict of plain values; prepare() builds what a program holds
before the call (an opened context with its weights and resident expert
records, device inputs and outputs, a captured graph where a program replays
one), run() makes one pass through the public entry points, exact() says in
64 bits, with plain torch, what the pass returns.

Kinds:
  decode   one token through a stack of MoE layers (h <- h + moe(h)), the
           step captured as a HIP graph and replayed: a token of generation
  host     one token through one layer from host buffers and back
           (moe_decode_host): the call an engine on the CPU makes
  chunk    a batch of tokens through one layer: prompt prefill, or one token
           each of several sequences; captured and replayed
  experts  single experts' FFNs of one token, no routing, for callers that
           route themselves
  kda      T steps of the delta-attention recurrence, its state on the device
  encode   the converter's residual-VQ encoder

Records are byte for byte the container's: a 48-byte header, the gate, up and
down index blocks ([64-row block][position of 8 weights][row][slot bytes]),
one fp16 scale per row. Codes are uniform, codebooks N(0, 0.3), row scales
U(0.01, 0.05), so that a layer's experts and its shared expert both show in
its output. Routers are N(0, 0.02); where only some experts of a wide layer
are held resident, a bias lifts those. A prefill's tokens lean on their
experts with Zipf(1.1) popularity, as real prompts do.
"""
import math
import struct

import numpy as np
import torch

from warp_amd import hip
from warp_amd.device import Graph

STAGES = {"VQ3R": 3, "VQ2R": 2, "VQ4P": 4, "VQ12": 2}
ENTRIES = {"VQ3R": 256, "VQ2R": 256, "VQ4P": 64, "VQ12": 4096}
SLOT = {"VQ3R": 3, "VQ2R": 2, "VQ4P": 3, "VQ12": 3}
HDR = 48
ROUTED_SCALE = 2.0
EPS = 1e-5
BETA, LBETA = 4.0, 2.0                   # SiTU's two betas
GROUP = {8: 32, 4: 128}                  # shared expert's scale groups
LATENT_GROUP = 128


def _layer(name, kind, fmt, hidden, inter, experts, top_k, **kw):
    c = dict(name=name, kind=kind, fmt=fmt, hidden=hidden, inter=inter, experts=experts, top_k=top_k, layers=1,
             resident=experts, shared=8, inter_shared=inter, latent=0, act="silu", router="sigmoid", tokens=1,
             fp16=False, zipf=0.0)
    c.update(kw)
    return c


def listed():
    return [
        # one expert at a time at the smallest serving shape, where a call is mostly its launches
        dict(name="experts-vq12", kind="experts", fmt="VQ12", hidden=2304, inter=1024, calls=64),
        # an engine on the CPU handing over one layer call: copies in and out, one wait
        _layer("host-vq2r", "host", "VQ2R", 2304, 1024, 256, 8),
        # token generation, a 48B-class model: every record resident, softmax top-8, a shared expert
        _layer("decode-vq12", "decode", "VQ12", 2304, 1024, 256, 8, layers=4, router="softmax"),
        # the same class in the int8-table format
        _layer("decode-vq4p", "decode", "VQ4P", 2304, 1024, 256, 8, layers=2),
        # token generation at the largest layer: 384 experts, top-16, 64 of them resident
        _layer("decode-vq12-wide", "decode", "VQ12", 7168, 2048, 384, 16, layers=4, resident=64, shared=0),
        # a latent MoE: experts on a 3584-wide projection, two shared experts, 896 to choose from
        _layer("decode-vq3r-latent", "decode", "VQ3R", 7168, 3072, 896, 16, layers=2, resident=48, latent=3584,
               inter_shared=6144),
        # a short prompt in the int8-table format
        _layer("chunk-vq4p", "chunk", "VQ4P", 2304, 1024, 256, 8, tokens=24),
        # an odd-sized prompt, exact products, the byte-code format, 4-bit shared expert
        _layer("chunk-vq3r", "chunk", "VQ3R", 2304, 1024, 256, 8, tokens=201, shared=4, zipf=1.1),
        # a prefill chunk in the reduced-precision mode
        _layer("chunk-vq12-fp16", "chunk", "VQ12", 2304, 1024, 256, 8, tokens=512, router="softmax", fp16=True,
               zipf=1.1),
        # 32 sequences' tokens of one step through the largest layer, everything resident
        _layer("chunk-vq12-wide", "chunk", "VQ12", 7168, 2048, 384, 16, tokens=32, shared=0),
        # a prompt's delta-attention layer: 32 heads of 128 x 128
        dict(name="kda", kind="kda", heads=32, key=128, value=128, steps=256),
        # conversion of one 2048 x 7168 matrix to 3 x 256 byte codes
        dict(name="encode", kind="encode", vectors=1835008, stages=3, entries=256),
    ]


def _log(rng, lo, hi, step=1):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step) * step))


def draw(rng):
    kind = rng.choice(["decode"] * 4 + ["chunk"] * 4 + ["host", "experts", "kda", "encode"])
    if kind == "kda":
        return dict(kind=kind, heads=_log(rng, 4, 64), key=rng.choice([64, 72, 96, 128]),
                    value=rng.choice([64, 96, 128, 200]), steps=_log(rng, 1, 256))
    if kind == "encode":
        wide = rng.random() < 0.3
        return dict(kind=kind, vectors=_log(rng, 20001, 180001 if wide else 1835008),
                    stages=2 if wide else rng.choice([1, 2, 3]), entries=4096 if wide else rng.choice([64, 255, 256]))
    fmt = rng.choice(sorted(STAGES))
    hidden, inter = _log(rng, 512, 7168, 32), _log(rng, 256, 3072, 32)
    if kind == "experts":
        return dict(kind=kind, fmt=fmt, hidden=hidden, inter=inter, calls=_log(rng, 8, 64))
    latent = hidden // 64 * 32 if rng.random() < 0.2 else 0
    experts = _log(rng, 16, 896)
    top_k = min(experts // 2, rng.choice([2, 4, 6, 8, 8, 16]))
    case = _layer("", kind, fmt, hidden, inter, experts, top_k, latent=latent, shared=rng.choice([0, 8, 8, 4]),
                  act=rng.choice(["silu", "silu", "situ"]), router=rng.choice(["sigmoid", "sigmoid", "softmax"]))
    del case["name"]
    if case["shared"]:
        # a shared expert's rows are whole groups
        case["hidden"] = hidden = max(512, hidden // GROUP[case["shared"]] * GROUP[case["shared"]])
        case["inter_shared"] = max(256, inter // 128 * 128)
        case["latent"] = hidden // 64 * 32 if latent else 0
    if kind == "chunk":
        # no larger than the listed chunks: in records held, and in products
        case["experts"] = min(experts, 384, int(384 * 7168 * 2048 / (hidden * inter)))
        most = 512 * 8 * 2304 * 1024 // (top_k * hidden * inter)
        most = max(2, min(512, most // 8 if fmt == "VQ4P" else most))
        case["tokens"] = _log(rng, 2, most)
        case["fp16"] = fmt != "VQ4P" and rng.random() < 0.4
        case["zipf"] = rng.choice([0.0, 1.1])
    else:
        case["layers"] = rng.choice([1, 2, 4]) if kind == "decode" else 1
    case["resident"] = case["experts"] if kind == "chunk" else min(experts, 48)
    case["top_k"] = min(top_k, case["resident"] // 2)
    return case


# ---- inputs, from the seed alone -------------------------------------------------------------------


def _gen(seed, *tag):
    g = torch.Generator(device="cuda")
    g.manual_seed(hash((int(seed),) + tag) & 0x7FFFFFFFFFFFFFFF)
    return g


def _normal(seed, tag, shape, std=1.0):
    return torch.randn(shape, generator=_gen(seed, *tag), device="cuda") * std


def _uniform(seed, tag, shape, lo, hi):
    return torch.rand(shape, generator=_gen(seed, *tag), device="cuda") * (hi - lo) + lo


def _bytes(seed, tag, n):
    out = torch.empty((n + 7) // 8, dtype=torch.int64, device="cuda")
    out.random_(-2 ** 63, None, generator=_gen(seed, *tag))
    return out.view(torch.uint8)


def _width(case):
    return case.get("latent") or case["hidden"]


def _index_bytes(fmt, M, N):
    return (M + 63) // 64 * (N // 8) * 64 * SLOT[fmt]


def _rec(case):
    """(offsets of gate, up, down and scales, scales, record stride)"""
    H, I = _width(case), case["inter"]
    gate, down = _index_bytes(case["fmt"], I, H), _index_bytes(case["fmt"], H, I)
    off = [HDR, HDR + gate, HDR + 2 * gate, HDR + 2 * gate + down]
    return off, 2 * I + H, (off[3] + 2 * (2 * I + H) + 4095) // 4096 * 4096


def _ids(case, seed, layer):
    n, r = case["experts"], case["resident"]
    return sorted(np.random.default_rng((seed, layer, 7)).permutation(n)[:r].tolist())


def _record(case, seed, layer, expert):
    """One expert's record, its header last (it names the layer's first codebook)."""
    off, rows, stride = _rec(case)
    rec = _bytes(seed, (1, layer, expert), stride)
    rec[off[3] + 2 * rows:] = 0
    rec[off[3]:off[3] + 2 * rows] = _uniform(seed, (2, layer, expert), rows, 0.01, 0.05).half().view(torch.uint8)
    code = {"VQ3R": 4, "VQ2R": 5, "VQ4P": 8, "VQ12": 9}[case["fmt"]]
    hdr = struct.pack("<IHHBBHHHIIIIIIII", 0x50584557, layer, expert, code, 0, layer * 3 * STAGES[case["fmt"]], 0, 0,
                      stride // 4096, off[0], off[1], off[2], off[3], 0, 0, 0)
    rec[:HDR] = torch.frombuffer(bytearray(hdr), dtype=torch.uint8).cuda()
    return rec


def _books(case, seed, layer):
    """[gate, up, down][stages][entries][8] fp16"""
    S, E = STAGES[case["fmt"]], ENTRIES[case["fmt"]]
    return _normal(seed, (3, layer), (3, S, E, 8), 0.3).half()


def _router(case, seed, layer):
    W = _normal(seed, (4, layer), (case["experts"], case["hidden"]), 0.02)
    bias = torch.zeros(case["experts"], device="cuda")
    if case["resident"] < case["experts"]:
        bias[_ids(case, seed, layer)] = 1.0
    return W, bias


def _quant(seed, tag, M, N, bits, group, lo, hi):
    """Q8G / Q4G rows (whole groups) and their fp16 group scales."""
    q = _bytes(seed, tag, M * N * bits // 8)[:M * N * bits // 8].view(M, -1)
    if bits == 8:
        q[q == 128] = 0                  # -128 does not occur
    return q, _uniform(seed, tag + (1,), (M, N // group), lo, hi).half()


def _dequant(q, s, bits):
    if bits == 8:
        w = q.view(torch.int8).double()
    else:
        w = torch.stack([q & 15, q >> 4], -1).reshape(q.shape[0], -1).double() - 8
    return (w.view(q.shape[0], s.shape[1], -1) * s.double()[:, :, None]).view(q.shape[0], -1)


def _shared(case, seed, layer):
    H, I, b = case["hidden"], case["inter_shared"], case["shared"]
    lo, hi = (1e-4, 3e-4) if b == 8 else (1.5e-3, 4.5e-3)
    return [_quant(seed, (5, layer, k), M, N, b, GROUP[b], lo, hi)
            for k, (M, N) in enumerate([(I, H), (I, H), (H, I)])]


def _latent(case, seed, layer):
    H, L = case["hidden"], case["latent"]
    s = [1.0 / (73.0 * math.sqrt(n)) for n in (H, L)]
    g = [LATENT_GROUP if H % LATENT_GROUP == 0 and L % LATENT_GROUP == 0 else 32] * 2
    return [_quant(seed, (6, layer, k), M, N, 8, g[k], 0.7 * s[k], 1.3 * s[k])
            for k, (M, N) in enumerate([(L, H), (H, L)])] + [_uniform(seed, (6, layer, 2), L, 0.5, 1.5)]


def _tokens(case, seed):
    """The inputs [T][hidden]; with zipf, each leans on top_k experts drawn by popularity."""
    X = _normal(seed, (8,), (case["tokens"], case["hidden"]))
    if case["zipf"]:
        W, _ = _router(case, seed, 0)
        pop = -case["zipf"] * torch.log(1.0 + torch.randperm(case["experts"], generator=_gen(seed, 9), device="cuda"))
        u = _uniform(seed, (10,), (case["tokens"], case["experts"]), 1e-9, 1.0)
        pick = (pop - torch.log(-torch.log(u))).topk(case["top_k"], 1).indices
        X += 6.0 * (W / W.square().sum(1, keepdim=True))[pick].sum(1)
    return X


# ---- the calls -------------------------------------------------------------------------------------


def _open(case):
    _, _, stride = _rec(case)
    n = case.get("layers", 1)
    return hip.Context(hidden=case["hidden"], inter=case["inter"], n_experts=case["experts"], top_k=case["top_k"],
                       n_layers=n, fmt=case["fmt"], renorm=True, routed_scale=ROUTED_SCALE,
                       router_act=hip.ROUTE_SOFTMAX if case["router"] == "softmax" else hip.ROUTE_SIGMOID,
                       act_situ=case["act"] == "situ", situ_beta=BETA, situ_linear_beta=LBETA,
                       max_tokens=case["tokens"], rec_bytes=stride, cache_bytes=n * case["resident"] * stride,
                       latent=case["latent"], latent_norm=True, norm_eps=EPS, prefill_fp16=case["fp16"])


def _load(ctx, case, seed):
    for L in range(case["layers"]):
        books = _books(case, seed, L).view(torch.int16).cpu().numpy()
        ctx.set_codebooks(L, L * 3 * STAGES[case["fmt"]], books)
        W, bias = _router(case, seed, L)
        ctx.set_router(L, W.cpu().numpy(), bias.cpu().numpy())
        if case["latent"]:
            d, u, norm = _latent(case, seed, L)
            ctx.set_latent(L, 8, case["hidden"] // d[1].shape[1], *[
                (q.cpu().numpy(), s.view(torch.int16).cpu().numpy(), q.shape[1]) for q, s in (d, u)],
                norm.cpu().numpy())
        if case["shared"]:
            sh = _shared(case, seed, L)
            ctx.set_shared(L, case["shared"], case["hidden"] // sh[0][1].shape[1], case["inter_shared"],
                           [q.cpu().numpy() for q, _ in sh], [s.view(torch.int16).cpu().numpy() for _, s in sh],
                           [q.shape[1] for q, _ in sh])
        for e in _ids(case, seed, L):
            rec = _record(case, seed, L, e)
            torch.cuda.current_stream().synchronize()
            ctx.put_expert_dev(L, e, rec)
    ctx.sync()


def _replay(ctx, step):
    """`step` warmed up once, then captured; replayed on the program's own stream."""
    step()
    ctx.sync()
    g = Graph(ctx.stream, step)
    g.stream = torch.cuda.current_stream().cuda_stream
    return g


def prepare(case, seed):
    kind = case["kind"]
    if kind == "kda":
        T, H, K, V = case["steps"], case["heads"], case["key"], case["value"]
        return dict(kind=kind, dims=(T, H, K, V), q=_normal(seed, (1,), (T, H, K)), k=_normal(seed, (2,), (T, H, K)),
                    v=_normal(seed, (3,), (T, H, V)), g=-0.1 * _normal(seed, (4,), (T, H, K)).abs(),
                    beta=_uniform(seed, (5,), (T, H), 0.1, 0.9), S=_normal(seed, (6,), (H, K, V), 0.1),
                    o=torch.empty((T, H, V), device="cuda"))
    if kind == "encode":
        n, S, E = case["vectors"], case["stages"], case["entries"]
        books = torch.stack([_normal(seed, (2, s), (E, 8), 0.6 ** s) for s in range(S)])
        return dict(kind=kind, n=n, X=_normal(seed, (1,), (n, 8)), books=books, resid=torch.empty((n, 8), device="cuda"),
                    codes=torch.empty((n, S), dtype=torch.int16, device="cuda"))
    if kind == "experts":
        n = case["calls"]
        full = _layer("", kind, case["fmt"], case["hidden"], case["inter"], n, 1, shared=0)
        ctx = _open(full)
        ctx.set_codebooks(0, 0, _books(full, seed, 0).view(torch.int16).cpu().numpy())
        for e in range(n):
            rec = _record(full, seed, 0, e)
            torch.cuda.current_stream().synchronize()
            ctx.put_expert_dev(0, e, rec)
        x, out = _normal(seed, (8,), case["hidden"]), torch.empty((n, case["hidden"]), device="cuda")
        torch.cuda.synchronize()

        def step():
            for e in range(n):
                ctx.expert_ffn(0, e, x, out[e])
        return dict(kind=kind, ctx=ctx, x=x, out=out, graph=_replay(ctx, step))
    ctx = _open(case)
    _load(ctx, case, seed)
    X = _tokens(case, seed)
    torch.cuda.synchronize()
    if kind == "host":
        return dict(kind=kind, ctx=ctx, x=X[0].cpu().numpy())
    out = torch.empty((case["layers"],) + tuple(X.shape), device="cuda")
    if kind == "decode":
        def step():
            h = X[0]
            for L in range(case["layers"]):
                ctx.moe_decode(L, h, out[L], resid_dev=h)
                h = out[L]
    else:
        def step():
            ctx.moe_chunk(0, X, out, case["tokens"])
    return dict(kind=kind, ctx=ctx, X=X, out=out, graph=_replay(ctx, step))


def run(state):
    kind = state["kind"]
    if kind == "kda":
        # the state carries on, as a sequence's next chunk finds it
        rc = hip.lib().warp_hip_kda_forward(*state["dims"], *(state[k].data_ptr() for k in "qkvg"),
                                            state["beta"].data_ptr(), state["S"].data_ptr(), state["o"].data_ptr(),
                                            torch.cuda.current_stream().cuda_stream)
        if rc:
            raise hip.WarpHipError(rc, "kda_forward")
        return state["o"], state["S"]
    if kind == "encode":
        b = state["books"]
        rc = hip.lib().warp_hip_vq_encode_dev(state["X"].data_ptr(), state["n"], b.data_ptr(), b.shape[0], b.shape[1],
                                              state["resid"].data_ptr(), state["codes"].data_ptr(),
                                              torch.cuda.current_stream().cuda_stream)
        if rc:
            raise hip.WarpHipError(rc, "vq_encode_dev")
        return state["codes"]
    if kind == "host":
        return state["ctx"].moe_decode_host(0, state["x"])
    state["graph"].launch()
    return state["out"]


# ---- what a pass cannot do without -----------------------------------------------------------------


def _distinct(case):
    """Experts that a batch touches, in the mean: each token's top_k of the resident ones, by popularity."""
    n, K, T = case["resident"], case["top_k"], case["tokens"]
    w = (1.0 + np.arange(n)) ** -case["zipf"]
    lo, hi = 0.0, 1e6
    for _ in range(80):
        mid = (lo + hi) / 2
        lo, hi = (mid, hi) if (1 - np.exp(-mid * w)).sum() < K else (lo, mid)
    return float((1 - np.exp(-lo * w) ** T).sum())


def work(case):
    kind = case["kind"]
    if kind == "kda":
        T, H, K, V = case["steps"], case["heads"], case["key"], case["value"]
        return {"bytes": 4 * (T * H * (3 * K + 2 * V + 1) + 2 * H * K * V), "flops": 7 * T * H * K * V}
    if kind == "encode":
        n, S, E = case["vectors"], case["stages"], case["entries"]
        return {"bytes": n * (32 + 2 * S) + S * E * 32, "flops": 16 * n * S * E}
    H, I, He = case["hidden"], case["inter"], _width(case)
    off, rows, _ = _rec(case)
    pair = off[3] - HDR + 2 * rows
    books = 3 * STAGES[case["fmt"]] * ENTRIES[case["fmt"]] * 16
    if kind == "experts":
        n = case["calls"]
        return {"bytes": n * (pair + 4 * H) + books + 4 * H, "flops": n * 6 * H * I}
    T, K, E = case["tokens"], case["top_k"], case["experts"]
    b = _distinct(case) * pair + books + 4 * E * (H + 1) + 8 * T * H
    f = T * K * 6 * He * I + 2 * T * E * H
    if case["shared"]:
        w = 3 * H * case["inter_shared"]
        b += w * case["shared"] / 8 + 2 * w / GROUP[case["shared"]]
        f += 2 * T * w
    if case["latent"]:
        b += 2 * H * He * (1 + 2 / LATENT_GROUP)
        f += 4 * T * H * He
    return {"bytes": case["layers"] * b, "flops": case["layers"] * f}


def tolerance(case):
    if case["kind"] == "encode":
        return "exact"
    if case["kind"] == "kda":
        return {"rel": 1e-5}
    if case.get("fp16"):
        return {"rel": 2e-3}             # 16-bit products, which the caller asked for
    if case["fmt"] == "VQ4P":
        return {"rel": 4e-3}             # tables rounded to int8: a last bit of h moves some entries by one
    return {"rel": 1e-5}


# ---- the same in 64 bits ---------------------------------------------------------------------------


def _codes(case, rec, kind):
    """The stages' codes of one matrix of a record: [M][N / 8][stages]"""
    H, I, fmt = _width(case), case["inter"], case["fmt"]
    off, _, _ = _rec(case)
    M, N = (H, I) if kind == 2 else (I, H)
    raw = rec[off[kind]:off[kind] + _index_bytes(fmt, M, N)]
    b = raw.view(-1, N // 8, 64, SLOT[fmt]).permute(0, 2, 1, 3).reshape(-1, N // 8, SLOT[fmt])[:M].long()
    if fmt in ("VQ3R", "VQ2R"):
        return b
    w = b[..., 0] | b[..., 1] << 8 | b[..., 2] << 16
    bits, S = (6, 4) if fmt == "VQ4P" else (12, 2)
    return torch.stack([w >> bits * s & (1 << bits) - 1 for s in range(S)], -1)


def _matvec(case, rec, books, kind, X):
    """X [T][N] times one matrix of a record, its codebooks [stages][entries][8]."""
    off, _, _ = _rec(case)
    I = case["inter"]
    codes = _codes(case, rec, kind)
    M, nv, S = codes.shape
    at = off[3] + 2 * (0, I, 2 * I)[kind]
    scale = rec[at:at + 2 * M].view(torch.float16).double()
    if case["fmt"] != "VQ4P":
        W = sum(books[s][codes[..., s]] for s in range(S)).view(M, nv * 8)
        return X @ W.T * scale
    # the int8-table format: each position's products with every entry, rounded to 8 bits by 32 positions
    out = []
    at = codes + 64 * torch.arange(4, device="cuda") + 256 * torch.arange(nv, device="cuda")[:, None]
    for x in X:
        T = torch.einsum("vd,scd->vsc", x.view(nv, 8), books)
        m = torch.stack([b.abs().max() for b in T.split(32)]).repeat_interleave(32)[:nv, None, None]
        q = (T * (127 / m)).round().clamp(-127, 127) * (m / 127)
        out.append(q.view(-1)[at].sum((1, 2)) * scale)
    return torch.stack(out)


def _act(case, g, u):
    if case.get("act") == "situ":
        return BETA * torch.tanh(g / BETA) * torch.sigmoid(g) * LBETA * torch.tanh(u / LBETA)
    return g * torch.sigmoid(g) * u


def _ffn(case, seed, layer, expert, books, X):
    rec = _record(case, seed, layer, expert)
    h = _act(case, *(_matvec(case, rec, books[k], k, X) for k in (0, 1)))
    return _matvec(case, rec, books[2], 2, h)


def _flushed(books):
    return torch.where(books.abs() < 2.0 ** -14, torch.zeros_like(books), books).double()


def _moe(case, seed, layer, X):
    W, bias = _router(case, seed, layer)
    logits = X @ W.double().T
    score = logits.softmax(1) if case["router"] == "softmax" else logits.sigmoid()
    pick = (score + bias.double()).topk(case["top_k"], 1).indices
    w = score.gather(1, pick)
    w = ROUTED_SCALE * w / w.sum(1, keepdim=True)
    books = _flushed(_books(case, seed, layer))
    Xe, norm = X, None
    if case["latent"]:
        d, u, norm = _latent(case, seed, layer)
        Xe = X @ _dequant(*d, 8).T
    y = torch.zeros((X.shape[0], _width(case)), dtype=torch.float64, device="cuda")
    for e in pick.unique().tolist():
        t, k = (pick == e).nonzero(as_tuple=True)
        y[t] += w[t, k, None] * _ffn(case, seed, layer, e, books, Xe[t])
    if case["latent"]:
        y = y * norm.double() / (y.square().mean(1, keepdim=True) + EPS).sqrt()
        y = y @ _dequant(*u, 8).T
    if case["shared"]:
        g, u, d = (_dequant(q, s, case["shared"]) for q, s in _shared(case, seed, layer))
        y = y + _act(case, X @ g.T, X @ u.T) @ d.T
    return y


def exact(case, seed):
    kind = case["kind"]
    if kind == "encode":
        return None                      # whole numbers
    if kind == "kda":
        s = prepare(case, seed)
        T, H, K, V = s["dims"]
        q, k, v, g, beta, S = (s[n].double() for n in ("q", "k", "v", "g", "beta", "S"))
        k = k / (k.square().sum(-1, keepdim=True) + 1e-12).sqrt()
        q = q / (q.square().sum(-1, keepdim=True) + 1e-12).sqrt() / math.sqrt(K)
        out = []
        for t in range(T):
            S = S * g[t].exp()[:, :, None]
            d = beta[t][:, None] * (v[t] - (S * k[t][:, :, None]).sum(1))
            S = S + k[t][:, :, None] * d[:, None, :]
            out.append((S * q[t][:, :, None]).sum(1))
        return torch.stack(out), S
    if kind == "experts":
        full = _layer("", kind, case["fmt"], case["hidden"], case["inter"], case["calls"], 1, shared=0)
        books, x = _flushed(_books(full, seed, 0)), _normal(seed, (8,), case["hidden"]).double()[None]
        return torch.cat([_ffn(full, seed, 0, e, books, x) for e in range(case["calls"])])
    X = _tokens(case, seed).double()
    if kind == "host":
        return _moe(case, seed, 0, X)[0].cpu().numpy(), None
    out = []
    for L in range(case["layers"]):
        y = _moe(case, seed, L, X)
        X = X + y if kind == "decode" else y
        out.append(X)
    return torch.stack(out)
