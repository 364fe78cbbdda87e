"""The encoder on the device against the reference's own (src/vq.c).

warp_hip_vq_encode must give the codes of waste_vq_encode bit for bit:
per stage the first minimum of the squared distance summed in dimension
order with unfused fp32 arithmetic, the exact residual feeding the next
stage. Checked against the compiled reference (oracle/_ref) on random
vectors, a duplicated codebook entry (the first copy wins) and vectors equal
to codebook entries; the 4096-entry variant (16-bit codes, beyond the
reference's 8-bit output) against the oracle's restatement. One
warp_hip_vq_lloyd iteration must give the reference's centroids bit for bit
(means summed in double in index order) and its count of non-empty
clusters, with clusters left empty.
"""
import ctypes
import os

import numpy as np
import pytest

from gpu_util import dev, empty, log
from oracle import pyoracle as po

pytestmark = pytest.mark.gpu


def ref_lib():
    if not os.path.exists(po.REF_LIB):
        pytest.skip("compiled reference not built")
    L = ctypes.CDLL(po.REF_LIB)
    L.waste_vq_encode.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_int, ctypes.c_int,
                                  ctypes.c_int, ctypes.c_void_p, ctypes.c_int]
    L.waste_vq_encode.restype = None
    L.waste_vq_lloyd.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_int, ctypes.c_int,
                                 ctypes.c_int]
    L.waste_vq_lloyd.restype = ctypes.c_int
    return L


def test_encode_matches_reference():
    import warp_amd.hip as wh
    L = ref_lib()
    rng = np.random.default_rng(61)
    S, E, n = 3, 256, 20000
    books = rng.normal(0.0, 1.0, size=(S, E, 8)).astype(np.float32)
    books[0, 40] = books[0, 7]                        # a duplicate: entry 7 must win
    X = rng.normal(0.0, 1.0, size=(n, 8)).astype(np.float32)
    X[:50] = books[0, 7]                              # exactly on the duplicated entry
    X[50:100] = books[0, rng.integers(0, E, 50)]      # exactly on entries
    got = wh.vq_encode(X, books)
    ref = np.empty((n, S), np.uint8)
    L.waste_vq_encode(X.ctypes.data, n, books.ctypes.data, S, E, 8, ref.ctypes.data, 4)
    assert np.array_equal(got, ref), int(np.count_nonzero(got != ref))
    assert (got[:50, 0] == 7).all()
    log(f"vq_encode: {n} vectors x {S} stages of {E} bit-identical to waste_vq_encode")


def test_encode16_matches_oracle():
    import warp_amd.hip as wh
    rng = np.random.default_rng(62)
    S, E, n = 2, 4096, 6000
    books = rng.normal(0.0, 0.5, size=(S, E, 8)).astype(np.float32)
    books[1, 4000] = books[1, 12]
    X = rng.normal(0.0, 1.0, size=(n, 8)).astype(np.float32)
    got = wh.vq_encode(X, books)
    ref = np.empty((n, S), np.uint16)
    po.lib().or_vq_encode(X.ctypes.data, n, books.ctypes.data, S, E, 8, ref.ctypes.data)
    assert got.dtype == np.uint16 and np.array_equal(got, ref), int(np.count_nonzero(got != ref))
    log(f"vq_encode16: {n} vectors x {S} stages of {E} bit-identical to the oracle")


def test_lloyd_matches_reference():
    import warp_amd.hip as wh
    L = ref_lib()
    rng = np.random.default_rng(63)
    n, E = 30000, 256
    X = rng.normal(0.0, 1.0, size=(n, 8)).astype(np.float32)
    C0 = X[rng.permutation(n)[:E]].copy()
    C0[200:] = 1.0e6                                  # far away: these clusters stay empty
    for it in range(3):
        got, ref = C0.copy(), C0.copy()
        live = wh.vq_lloyd(X, got)
        live_ref = L.waste_vq_lloyd(X.ctypes.data, n, ref.ctypes.data, E, 8, 4)
        assert live == live_ref == 200, (live, live_ref)
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), it
        C0 = ref
    log(f"vq_lloyd: 3 iterations over {n} vectors, {E} clusters (56 empty) bit-identical to waste_vq_lloyd")


@pytest.mark.parametrize("S,E,n", [
    (1, 1, 1), (2, 15, 63), (3, 16, 65), (3, 17, 1000), (17, 16, 130), (3, 255, 20001), (3, 256, 131072 + 1),
    (4, 257, 3000), (3, 512, 3000), (2, 1024, 3000), (2, 1025, 3000), (1, 2000, 131072 - 63), (2, 4095, 3000)])
def test_encode_scores_never_decide(S, E, n):
    """The winner the matrix cores propose is confirmed or the vector scanned:
    codes equal the oracle's at the edges of tiles (16 entries), of their
    numbering (256), of LDS pieces (1024), of launches (96 tiles, 16 stages)
    and of blocks, for duplicated entries in one group of 4 and across groups,
    vectors on entries and on zero, vectors and codebooks out of the scores'
    range, infinities and NaN."""
    import warp_amd.hip as wh
    rng = np.random.default_rng(1000 * S + E)
    books = (rng.normal(0.0, 1.0, size=(S, E, 8)) * 0.6 ** np.arange(S)[:, None, None]).astype(np.float32)
    X = rng.normal(0.0, 1.0, size=(n, 8)).astype(np.float32)
    for i in range(1, 40):                            # duplicates, near and far
        books[rng.integers(S), rng.integers(E)] = books[rng.integers(S), rng.integers(E)]
    books[0, E // 2] = 0.0
    m = min(n, 40)
    X[:m] = books[0, rng.integers(0, E, m)]
    X[m // 2:m] = 0.0
    for i, v in enumerate([np.nan, np.inf, -np.inf, 3e38, 1e25, 1e10, 1e-30, 1e-42, 100.0]):
        X[(7 + 61 * i) % n, i % 8] = v                # one component
        with np.errstate(over="ignore", invalid="ignore"):
            X[(11 + 67 * i) % n] *= np.float32(v)
    kinds = {"": books}
    if n <= 3000:
        with np.errstate(over="ignore"):
            kinds.update(offset=books + np.float32(300.0), tiny=books * np.float32(1e-25), huge=books * np.float32(1e25),
                         zero=books * 0.0)
        kinds["bad"] = books.copy()
        kinds["bad"][0, E // 3, 3], kinds["bad"][S - 1, E // 4, 0] = np.nan, np.inf
    for kind, b in kinds.items():
        b = np.ascontiguousarray(b, dtype=np.float32)
        got, ref = wh.vq_encode(X, b), np.empty((n, S), np.uint16)
        po.lib().or_vq_encode(X.ctypes.data, n, b.ctypes.data, S, E, 8, ref.ctypes.data)
        assert np.array_equal(got, ref), (kind, int(np.count_nonzero(got != ref)))


def spread_books(kind, rng, S, E):
    """Codebooks whose entries differ in length, offset or not at all."""
    b = rng.normal(0.0, 1.0, size=(S, E, 8)).astype(np.float32)
    if kind == "one x100":
        b[:, E // 2] *= np.float32(100.0)
    elif kind == "three far":
        b[:, E // 4] *= np.float32(1e4)
        b[:, E // 2] *= np.float32(1e20)
        b[:, E - 1, 3] = np.inf
    elif kind == "heavy":
        b /= np.sqrt(rng.chisquare(2, size=b.shape) / 2).astype(np.float32)
    elif kind == "offset":
        b[0] += np.float32(64.0)
    elif kind == "copies":
        b[:, E // 2:] = b[:, :E - E // 2]
    elif kind == "near copies":
        b[:, E // 2:] = b[:, :E - E // 2] * np.float32(1.0 + 2.0 ** -22)
    elif kind == "zeros":
        b[:, ::2] *= np.float32(0.0)                  # 0 and -0
    return b


SPREADS = ["one x100", "three far", "heavy", "offset", "copies", "near copies", "zeros"]


@pytest.mark.parametrize("S,E,n", [(3, 256, 5000), (3, 32, 5000), (2, 33, 4999), (17, 33, 130), (2, 1500, 3000)])
def test_encode_spread_codebooks(S, E, n):
    """Codes of codebooks with a few long entries, heavy tails, an offset,
    entries twice and almost twice, zeros of both signs: the oracle's. The
    vectors are of the entries' kind, some of them entries."""
    import warp_amd.hip as wh
    for kind in SPREADS:
        rng = np.random.default_rng(S * E + n)
        b = spread_books(kind, rng, S, E)
        X = spread_books(kind, rng, 1, n)[0]
        X[::7] = b[0, rng.integers(0, E, len(X[::7]))]
        X[~np.isfinite(X)] = 0.0
        got, ref = wh.vq_encode(X, b), np.empty((n, S), np.uint16)
        po.lib().or_vq_encode(X.ctypes.data, n, b.ctypes.data, S, E, 8, ref.ctypes.data)
        assert np.array_equal(got, ref), (kind, int(np.count_nonzero(got != ref)))


def test_encode_several_tiles_per_wave():
    """Enough vectors that a wave takes several 64-vector tiles, the last ones
    ragged: codes equal the oracle's, also where a tile's scan has the wave
    scan the next ones too."""
    import warp_amd.hip as wh
    S, E, n = 2, 34, 2 * 262144 + 65
    for kind in ("heavy", "near copies"):
        rng = np.random.default_rng(5)
        b = spread_books(kind, rng, S, E)
        X = rng.normal(0.0, 1.0, size=(n, 8)).astype(np.float32)
        got, ref = wh.vq_encode(X, b), np.empty((n, S), np.uint16)
        po.lib().or_vq_encode(X.ctypes.data, n, b.ctypes.data, S, E, 8, ref.ctypes.data)
        assert np.array_equal(got, ref), (kind, int(np.count_nonzero(got != ref)))


def encode_ms(X, books, reps=20):
    """The device's time of one warp_hip_vq_encode_dev of X [n][8]."""
    import warp_amd.hip as wh
    from warp_amd.device import Event
    n, (S, E, _) = X.shape[0], books.shape
    x, b, r, codes = dev(X), dev(books), empty((n, 8)), empty((n, S), np.uint16)

    def go():
        assert wh.lib().warp_hip_vq_encode_dev(x.ptr, n, b.ptr, S, E, r.ptr, codes.ptr, None) == 0
    go()
    best = np.inf
    for _ in range(3):
        e0, e1 = Event(), Event()
        e0.record(None)
        for _ in range(reps):
            go()
        e1.record(None)
        e1.synchronize()
        best = min(best, e0.elapsed_ms(e1) / reps)
    return best


def test_encode_time_hardly_depends_on_the_entries():
    """A codebook with a long entry, heavy tails, an offset or copies takes no
    more than 3 times the time of one without (measured: 2 at most, with
    copies). Scanning every vector takes 4 times, one by one 8 times."""
    rng = np.random.default_rng(9)
    S, E, n = 3, 256, 400000
    plain = encode_ms(rng.normal(size=(n, 8)).astype(np.float32), spread_books("", rng, S, E))
    for kind in ("one x100", "heavy", "offset", "copies", "zeros"):
        ms = encode_ms(spread_books(kind, rng, 1, n)[0], spread_books(kind, rng, S, E))
        log(f"vq_encode {kind}: {ms * 1e3:.1f} us, {ms / plain:.2f} times the plain codebook's")
        assert ms <= 3.0 * plain, (kind, ms, plain)


def test_encode_small_codebooks_are_scanned():
    """16 entries cost well below 64 (measured: 0.42 of the time; 0.85 with
    scores), and no more for a launch that fills the device less."""
    rng = np.random.default_rng(10)
    for n in (20001, 219432):
        X = rng.normal(size=(n, 8)).astype(np.float32)
        small, large = (encode_ms(X, spread_books("", rng, 1, E), 200) for E in (16, 64))
        log(f"vq_encode {n}: 16 entries {small * 1e3:.2f} us, 64 entries {large * 1e3:.2f} us")
        assert small <= 0.7 * large, (n, small, large)
